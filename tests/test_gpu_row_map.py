"""Flat offsets and row map on both sides of the line past which the map is filled
by a launch of its own (32 entries per row, tiles of 4,096 rows): every product,
export and compaction finds its rows through them.  Small integers: sums are
exact."""
import numpy as np
import pytest

from tests.helpers import check_healthy, check_layout

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [1, 300, 4_095, 4_096, 4_097, 9_000])
@pytest.mark.parametrize("L", [31, 32, 33, 400])
@pytest.mark.parametrize("ragged", [False, True])
def test_rows_through_the_map(R, L, ragged):
    import torch
    import dcsr_amd
    rng = np.random.default_rng(R + L)
    lens = np.full(R, L)
    if ragged:  # empty rows, one long one, the same total
        lens = np.bincount(rng.integers(0, max(R // 2, 1), R * L), minlength=R)
        if R > 2:
            lens[1] += lens[0]
            lens[0] = 0
    C = int(lens.max()) + 40
    r = np.repeat(np.arange(R), lens)
    k = np.arange(r.size) - np.concatenate([[0], np.cumsum(lens)])[r]
    c = k + rng.integers(0, 40, R)[r]  # ascending, unique
    v = rng.integers(1, 4, r.size).astype(np.float32)
    x = rng.integers(-3, 4, C).astype(np.float32)
    want = np.bincount(r, weights=v * x[c], minlength=R).astype(np.float32)
    off = np.concatenate([[0], np.cumsum(lens)])
    m = dcsr_amd.DcsrMatrix(R, C)
    dx = torch.from_numpy(x).cuda()

    def check():
        np.testing.assert_array_equal(m.spmv(dx).cpu().numpy(), want)
        for got, w in zip(m.to_csr(), (off, c, v)):
            np.testing.assert_array_equal(got.cpu().numpy(), w)

    m.load_csr(off.astype(np.int32), c.astype(np.int32), v)
    check()
    m.SortMatrixRow()
    check()
    m.BinRows()
    check()
    p = rng.permutation(r.size)
    m.LoadMatrix(r[p].astype(np.int32), c[p].astype(np.int32), v[p])
    check()
    check_layout(m)
    check_healthy(m)
    m.close()
