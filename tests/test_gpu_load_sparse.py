"""CSR loads of matrices whose rows are mostly empty: entries of one wave's share
(512) next to each other, just within and just past the rows that it walks, and
millions of rows apart; rows in and out of column order.  No arithmetic: compared
bit for bit."""
import numpy as np
import pytest

from tests.helpers import check_healthy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,rows", [
    (3_000_000, [0, 0, 2_999_999]), (3_000_000, [1, 1_500_000]), (700, [0, 699]), (1, [0] * 700),
    (1_025, list(range(512)) + [1_023]), (1_026, list(range(511)) + [1_024]), (2_000, list(range(511)) + [1_025, 1_999]),
    (1_000_000, "hundredth"), (200_000, "clumps"), (40_000, "tail"), (40_000, "head"),
])
@pytest.mark.parametrize("order", ["ascending", "descending"])
def test_empty_rows(R, rows, order):
    import dcsr_amd
    rng = np.random.default_rng(R)
    if rows == "hundredth":
        rows = np.arange(0, R, 100)
    elif rows == "clumps":  # full waves of one row between long gaps
        rows = np.sort(np.repeat(rng.permutation(R)[:9], [1, 511, 512, 513, 1, 2_000, 64, 3, 300]))
    elif rows == "tail":
        rows = R - 1 - np.arange(3_000)[::-1] // 3
    elif rows == "head":
        rows = np.arange(3_000) // 3
    rows = np.asarray(rows)
    off = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=R))]).astype(np.int32)
    C = 5_000
    k = np.arange(rows.size) - off[rows]  # place in the row
    c = k if order == "ascending" else off[rows + 1] - off[rows] - 1 - k
    v = rng.integers(1, 100, rows.size).astype(np.float32)
    m = dcsr_amd.DcsrMatrix(R, C)
    m.load_csr(off, c.astype(np.int32), v)
    o = np.lexsort((c, rows))
    got = [t.cpu().numpy() for t in m.to_csr()]
    np.testing.assert_array_equal(got[0], off)
    np.testing.assert_array_equal(got[1], c[o])
    np.testing.assert_array_equal(got[2], v[o])
    bad = c.astype(np.int32)
    bad[-1] = C
    with pytest.raises(dcsr_amd.DcsrError) as e:
        m.load_csr(off, bad, v)
    assert e.value.code == 2  # DCSR_ERR_BAD_INDEX
    check_healthy(m)
    m.close()
