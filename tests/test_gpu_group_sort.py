"""The row-group sort of an update batch (7,169 to 2^21 triples) against the
oracle: groups whose keys spread, a long row (its buckets are split), one
coordinate hundreds of times (digit passes in LDS; in the longest case local keys
of 53 bits, which leave no room for a position), a group past 3,072 pairs.
Structure and update values bit for bit: the sums see arrival order."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import assert_same_structure, check_healthy, to_host_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [7_169, 20_000, 300_000])
@pytest.mark.parametrize("mode", ["spread", "row", "same", "both", "crowd"])
@pytest.mark.parametrize("R,C", [(900, 50_000), (300_000, 5_000), (200_003, 2**31 - 1)])
def test_groups(R, C, mode, n):
    run(R, C, mode, n)


def test_long_keys():
    run(2**25 + 1, 2**31 - 1, "both", 7_500)


def run(R, C, mode, n):
    import dcsr_amd
    rng = np.random.default_rng(n + len(mode) + R)
    k = 4_000
    r, c = rng.integers(0, R, k).astype(np.int32), rng.integers(0, C, k).astype(np.int32)
    v = rng.integers(1, 5, k).astype(np.float32)
    m = dcsr_amd.DcsrMatrix(R, C, pool_factor=3.0 + 4.0 * n / k)
    m.LoadMatrix(r, c, v)
    A = O.coo_to_csr(R, C, r, c, v)
    br, bc = rng.integers(0, R, n), rng.integers(0, C, n)
    bv = rng.uniform(-1, 1, n).astype(np.float32)
    p = rng.permutation(n)
    if mode in ("row", "both"):  # a long row and a shorter one
        br[p[:2_400]] = R // 2
        br[p[2_400:2_700]] = R // 2 + 1
    if mode in ("same", "both"):  # runs of one coordinate, of 65 and of 700
        br[p[3_000:3_700]], bc[p[3_000:3_700]] = R // 3, C // 3
        br[p[3_700:3_765]], bc[p[3_700:3_765]] = R - 1, C - 1
    if mode == "crowd":  # more than a group holds in LDS
        br[p[:5_000]] = R // 2
        bc[p[:2_500]] = bc[p[:2_500]] % 40
    bt = br.astype(np.int32), bc.astype(np.int32), bv
    m.UpdateMatrix(*bt)
    assert_same_structure(to_host_csr(m), O.update(A, *bt))
    check_healthy(m)
    m.close()
