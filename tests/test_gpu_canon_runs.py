"""Runs of equal columns in the canonical export: lengths around the entries that
are summed at a time (8), starting anywhere in a 64-entry word, the same column
again at the start of the next row, the last run at the matrix's end.  Sums run
in stored order: compared bit for bit."""
import numpy as np
import pytest

from tests.helpers import check_healthy

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens", [[1, 2, 7, 8, 9], [10, 15, 16, 17, 1], [63, 64, 65], [3_000, 1, 5], [12_345]])
@pytest.mark.parametrize("lead", [0, 1, 57])
def test_runs(lens, lead):
    import dcsr_amd
    rng = np.random.default_rng(len(lens) + lead)
    reps, R = 40, 40 * len(lens) + 1
    runs = np.array(lens * reps)
    r = np.repeat(np.arange(1, R), runs)
    c = np.full(r.size, 9)  # every row starts with the column that the last one ended with
    r, c = np.concatenate([np.zeros(lead, int), r]), np.concatenate([np.arange(lead), c])
    v = rng.uniform(-1, 1, r.size).astype(np.float32)
    m = dcsr_amd.DcsrMatrix(R, 64)
    m.LoadMatrix(r.astype(np.int32), c.astype(np.int32), v)
    want_v, want_r, i = [], [], 0
    while i < r.size:
        j, s = i, np.float32(0)
        while j < r.size and r[j] == r[i] and c[j] == c[i]:
            s = np.float32(s + v[j])
            j += 1
        if s != 0:
            want_v.append(s)
            want_r.append(r[i])
        i = j
    off, col, val = (t.cpu().numpy() for t in m.to_csr(canonical=True))
    np.testing.assert_array_equal(off, np.concatenate([[0], np.cumsum(np.bincount(want_r, minlength=R))]))
    np.testing.assert_array_equal(val.view(np.int32), np.array(want_v, np.float32).view(np.int32))
    np.testing.assert_array_equal(col, np.concatenate([np.arange(lead), np.full(col.size - lead, 9)]))
    check_healthy(m)
    m.close()
