"""Batches whose coordinates crowd into few rows, on every path that places them
by bisection: runs of one row that start and end on, before and past the edges
of 64 coordinates, with inserts, deletions to zero, adds and cancelled sums among
them.  Structure and values are compared with the oracle's bit for bit."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import assert_same_structure, check_healthy, check_layout, to_host_csr

pytestmark = pytest.mark.gpu
R = 60_000


@pytest.mark.parametrize("n", [2_049, 7_168, 8_000, 131_071, 140_000])
@pytest.mark.parametrize("runs", [[1_000_000], [64], [63, 65, 1], [1, 127, 640, 5]])
def test_runs_of_one_row(n, runs):
    import dcsr_amd
    rng = np.random.default_rng(n + len(runs))
    lens, at = [], 0
    while at < n:
        lens.append(min(runs[len(lens) % len(runs)], n - at, R))
        at += lens[-1]
    rows = np.sort(rng.permutation(R)[:len(lens)])
    br = np.repeat(rows, lens)
    bc = np.concatenate([np.sort(rng.permutation(R)[:k]) for k in lens])
    old = rng.random(n) < 0.5  # already stored
    r, c = br[old].astype(np.int32), bc[old].astype(np.int32)
    v = rng.integers(1, 4, r.size).astype(np.float32)
    bv = rng.integers(-1, 3, n).astype(np.float32)  # zeros insert nothing
    bv[old] = np.where(rng.random(r.size) < 0.5, -v, bv[old])
    p = rng.permutation(n)
    b = br[p].astype(np.int32), bc[p].astype(np.int32), bv[p]
    m = dcsr_amd.DcsrMatrix(R, R, pool_factor=8.0)
    m.LoadMatrix(r, c, v)
    A = O.coo_to_csr(R, R, r, c, v)
    for flags in (0, dcsr_amd.UPDATE_NOSYNC):
        m.UpdateMatrix(*b, flags=flags)
        A = O.update(A, *b)
        assert_same_structure(to_host_csr(m), A)
        check_layout(m)
    check_healthy(m)
    m.close()
