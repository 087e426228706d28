"""Large update batches around the sizes where the tiles of the heads, plan and
offsets passes change (512 and 2,048 entries; 131,071 triples between them) and
at remainders of both, against the oracle: runs of one coordinate that cross
tiles, deletions, untouched and new rows.  Structure and update values bit for
bit; a triple outside the matrix rejects the batch."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import assert_same_structure, check_healthy, check_layout, to_host_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [7_169, 10_241, 12_799, 12_800, 12_801, 65_536, 131_070, 131_071, 131_072, 133_120, 300_001])
def test_tiles(n):
    check(40_003, n)


@pytest.mark.parametrize("R,n", [(52_428, 131_072), (52_430, 131_072), (300_007, 140_001)])
def test_coordinates_per_row(R, n):
    """Both probes on both sides of five coordinates per two rows."""
    check(R, n)


def check(R, n):
    import dcsr_amd
    C = 30_000
    rng = np.random.default_rng(n)
    key = np.unique(rng.integers(0, R, 400_000) * np.int64(C) + rng.integers(0, C, 400_000))
    r, c = (key // C).astype(np.int32), (key % C).astype(np.int32)
    v = rng.integers(1, 5, key.size).astype(np.float32)
    m = dcsr_amd.DcsrMatrix(R, C, pool_factor=6.0)
    m.LoadMatrix(r, c, v)
    A = O.coo_to_csr(R, C, r, c, v)
    for flags in (0, dcsr_amd.UPDATE_NOSYNC):
        br, bc = rng.integers(0, R, n), rng.integers(0, C, n)
        bv = rng.uniform(-1, 1, n).astype(np.float32)
        at = rng.permutation(n)
        rows = np.repeat(np.arange(R), np.diff(A.off))
        pick = rng.integers(0, A.nnz, n // 4)
        i = at[: n // 4]  # deletions
        br[i], bc[i], bv[i] = rows[pick], A.col[pick], -A.val[pick]
        i = at[n // 4: n // 4 + 3_000]  # three long runs of one coordinate
        br[i], bc[i] = R // 3 * (np.arange(i.size) % 3), 7
        i = at[n // 4 + 3_000: n // 4 + 5_000]  # a long row
        br[i] = R - 1
        bt = br.astype(np.int32), bc.astype(np.int32), bv
        m.UpdateMatrix(*bt, flags=flags)
        A = O.update(A, *bt)
        assert_same_structure(to_host_csr(m), A)
    bad = bt[0].copy()
    bad[n // 2] = R
    with pytest.raises(dcsr_amd.DcsrError):
        m.UpdateMatrix(bad, bt[1], bt[2])
    assert_same_structure(to_host_csr(m), A)
    assert check_layout(m)["nnz"] == A.nnz
    check_healthy(m)
    m.close()
