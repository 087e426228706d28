"""Load and export at the edges of their tiles: triples in and out of order,
CSR rows with and without ascending columns, duplicates and explicit zeros in
the canonical export, long runs of empty rows, output buffers one entry too
small.  Loads and raw exports do no arithmetic and the canonical export sums
in stored order, so everything is compared bit for bit."""
import ctypes

import numpy as np
import pytest

from tests.helpers import check_healthy

pytestmark = pytest.mark.gpu


def stored(R, r, c, v):
    """Stable by (row, column): what the rows hold after a load."""
    o = np.lexsort((np.arange(r.size), c, r))
    return np.concatenate([[0], np.cumsum(np.bincount(r, minlength=R))]), c[o], v[o], r[o]


def canonical(R, r, c, v):
    _, c, v, r = stored(R, r, c, v)
    rows, cols, vals = [], [], []
    i = 0
    while i < r.size:
        j, s = i, np.float32(0)
        while j < r.size and r[j] == r[i] and c[j] == c[i]:
            s = np.float32(s + v[j])
            j += 1
        if s != 0:
            rows.append(r[i])
            cols.append(c[i])
            vals.append(s)
        i = j
    rows = np.array(rows, np.int64)
    return np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=R))]), np.array(cols, np.int32), \
        np.array(vals, np.float32)


def same(got, want):
    for g, w in zip(got, want):
        g = g.cpu().numpy()
        assert g.shape == w.shape
        np.testing.assert_array_equal(g.view(np.int32), np.ascontiguousarray(w.astype(g.dtype)).view(np.int32))


@pytest.mark.parametrize("n", [0, 1, 63, 64, 65, 1023, 1024, 1025, 2047, 2048, 2049, 30_000])
@pytest.mark.parametrize("order", ["random", "sorted", "hot"])
def test_load_and_export(n, order):
    import torch
    import dcsr_amd
    R, C = (3, 5) if order == "hot" else (5_000, 700)
    rng = np.random.default_rng(n + len(order))
    r = rng.integers(0, R, n).astype(np.int32)
    if order == "random" and n > 1:
        r[: n // 2] = rng.integers(R - 3, R, n // 2)  # most rows empty, a long gap before the last ones
    c = rng.integers(0, C, n).astype(np.int32)
    v = rng.integers(-2, 3, n).astype(np.float32)  # zeros, and runs that cancel
    if order == "sorted":
        o = np.lexsort((c, r))
        r, c, v = r[o], c[o], v[o]
    m = dcsr_amd.DcsrMatrix(R, C)
    m.LoadMatrix(r, c, v)
    want = stored(R, r, c, v)[:3]
    same(m.to_csr(), want)
    want_c = canonical(R, r, c, v)
    same(m.to_csr(canonical=True), want_c)
    # one entry too small: an error, and the buffers as they were
    for canon, size in ((0, n), (1, want_c[1].size)):
        if size == 0 or (canon and size == n):
            continue
        off = torch.full((R + 1,), 7, dtype=torch.int32, device="cuda")
        col = torch.full((size,), 7, dtype=torch.int32, device="cuda")
        val = torch.full((size,), 7.0, device="cuda")
        k = ctypes.c_int64(0)
        code = dcsr_amd.lib().dcsr_export_csr(m.handle, off.data_ptr(), col.data_ptr(), val.data_ptr(), size - 1,
                                              ctypes.byref(k), canon, torch.cuda.current_stream().cuda_stream)
        assert code == 7  # DCSR_ERR_CAPACITY
        assert (off == 7).all() and (col == 7).all() and (val == 7.0).all()
    # CSR in, rows as stored and with their columns reversed
    off, c2, v2 = want
    for flip in (False, True):
        cc, vv = c2.copy(), v2.copy()
        if flip:
            for i in range(R):
                cc[off[i]:off[i + 1]] = cc[off[i]:off[i + 1]][::-1]
                vv[off[i]:off[i + 1]] = vv[off[i]:off[i + 1]][::-1]
        m.load_csr(off.astype(np.int32), cc, vv)
        rr = np.repeat(np.arange(R), np.diff(off)).astype(np.int32)
        same(m.to_csr(), stored(R, rr, cc, vv)[:3])
    check_healthy(m)
    m.close()


def test_export_after_nosync_updates_checks_the_capacity():
    """The count is read back after the copy: a buffer that holds the old
    entries but not the new ones stays untouched."""
    import torch
    import dcsr_amd
    R = 3_000
    rng = np.random.default_rng(3)
    r, c = rng.integers(0, R, 9_000).astype(np.int32), rng.integers(0, R, 9_000).astype(np.int32)
    key = np.unique(r.astype(np.int64) * R + c)
    r, c = (key // R).astype(np.int32), (key % R).astype(np.int32)
    m = dcsr_amd.DcsrMatrix(R, R, pool_factor=8.0)
    m.LoadMatrix(r, c, np.ones(r.size, np.float32))
    br, bc = rng.integers(0, R, 500).astype(np.int32), rng.integers(0, R, 500).astype(np.int32)
    bkey = np.unique(br.astype(np.int64) * R + bc)
    size = np.union1d(key, bkey).size
    m.UpdateMatrix(bkey // R, bkey % R, np.ones(bkey.size, np.float32), flags=dcsr_amd.UPDATE_NOSYNC)
    k = ctypes.c_int64(0)
    off = torch.full((R + 1,), 7, dtype=torch.int32, device="cuda")
    col = torch.full((size,), 7, dtype=torch.int32, device="cuda")
    val = torch.full((size,), 7.0, device="cuda")
    args = (off.data_ptr(), col.data_ptr(), val.data_ptr())
    s = torch.cuda.current_stream().cuda_stream
    assert dcsr_amd.lib().dcsr_export_csr(m.handle, *args, size - 1, ctypes.byref(k), 0, s) == 7
    assert (off == 7).all() and (col == 7).all() and (val == 7.0).all()
    assert dcsr_amd.lib().dcsr_export_csr(m.handle, *args, size, ctypes.byref(k), 0, s) == 0
    got = np.repeat(np.arange(R), np.diff(off.cpu().numpy())).astype(np.int64) * R + col.cpu().numpy()
    np.testing.assert_array_equal(got, np.union1d(key, bkey))
    m.close()


@pytest.mark.parametrize("n", [255, 256, 257, 2**20 - 1, 2**20, 2**20 + 1, 1_300_003])
def test_export_on_both_sides_of_the_copy_span(n):
    import dcsr_amd
    R, C = 150_000, 40_000
    rng = np.random.default_rng(n)
    r = rng.integers(0, R, n).astype(np.int32)
    r[: n // 8] = R // 2  # a long row
    c, v = rng.integers(0, C, n).astype(np.int32), rng.random(n, np.float32)
    m = dcsr_amd.DcsrMatrix(R, C, pool_factor=1.2)
    m.LoadMatrix(r, c, v)
    m.SortMatrixRow()  # the same copy, into the pool
    same(m.to_csr(), stored(R, r, c, v)[:3])
    check_healthy(m)
    m.close()
