"""SpMV where the rows meet the waves' 256-entry ranges: rows that start and end
on, before and past the edges, single entries, runs of empty rows, one row over
many ranges, a whole range of one-entry rows, and the remainders of the last
range; as loaded (rows side by side), after an update (rows anywhere in the
pool) and over the paneled copy.  Small integers: every order of summation is
exact, so results are compared for equality with the integer product."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PATTERNS = {
    "one_row": [1000],
    "edges": [256, 256, 255, 1, 257, 255, 64, 192, 0, 0, 256],
    "ones": [1] * 700,
    "gaps": ([0] * 200 + [1] + [0] * 70 + [3]) * 6 + [0] * 300,
    "mixed": [5, 0, 300, 1, 1, 1, 40, 0, 700, 2] * 5,
    "fours": [4] * 200 + [3, 1] * 100,
    "short_last": [256, 256, 1],
    "tail_empty": [100, 0, 0, 0],
    "sixties": [63, 64, 65, 66, 1, 62] * 8,
}


@pytest.mark.parametrize("name", sorted(PATTERNS))
@pytest.mark.parametrize("paneled", [False, True])
def test_rows_and_ranges(name, paneled, monkeypatch):
    import torch
    import dcsr_amd
    C = 2000
    if paneled:
        monkeypatch.setenv("DCSR_SPMV_PANEL_COLS", "300")
        monkeypatch.setenv("DCSR_SPMV_PANEL_MIN_NNZ", "0")
    rng = np.random.default_rng(len(name))
    lens = np.array(PATTERNS[name])
    R = lens.size
    r = np.repeat(np.arange(R), lens).astype(np.int32)
    c = np.concatenate([np.sort(rng.permutation(C)[:k]) for k in lens]).astype(np.int32)
    v = rng.integers(1, 4, r.size).astype(np.float32)
    m = dcsr_amd.DcsrMatrix(R, C, pool_factor=4.0)
    m.LoadMatrix(r, c, v)
    x = rng.integers(-4, 5, C).astype(np.float32)
    dx = torch.from_numpy(x).cuda()
    D = np.zeros((R, C))
    D[r, c] = v
    X2 = torch.from_numpy(np.stack([x, -x, 2 * x], 1)).cuda()

    def check():
        for _ in range(3):
            np.testing.assert_array_equal(m.spmv(dx).cpu().numpy(), (D @ x).astype(np.float32))
        y0 = rng.integers(-5, 6, R).astype(np.float32)
        y = torch.from_numpy(y0.copy()).cuda()
        m.spmv(dx, y, alpha=2.0, beta=-3.0)
        np.testing.assert_array_equal(y.cpu().numpy(), (2 * (D @ x) - 3 * y0).astype(np.float32))
        np.testing.assert_array_equal(m.spmm(X2).cpu().numpy(), (D @ X2.cpu().numpy()).astype(np.float32))

    check()
    assert m.info()["spmv_paneled"] == int(paneled)
    br, bc = rng.integers(0, R, 50).astype(np.int32), rng.integers(0, C, 50).astype(np.int32)
    key = np.unique(br.astype(np.int64) * C + bc)
    br, bc = key // C, key % C
    m.UpdateMatrix(br, bc, np.full(key.size, 7.0, np.float32))
    D[br, bc] += 7
    check()
    m.close()


@pytest.mark.parametrize("narrow", [False, True])
def test_captured_product_follows_updates(narrow, monkeypatch):
    """A product captured after the copy exists replays the rows as they are."""
    import torch
    import dcsr_amd
    monkeypatch.setenv("DCSR_SPMV_PANEL_COLS", "1000" if narrow else "1500")
    monkeypatch.setenv("DCSR_SPMV_PANEL_MIN_NNZ", "1500" if narrow else "0")
    R, C, n = 400, 2000 + 500 * narrow, 2000
    rng = np.random.default_rng(3)
    key = rng.permutation(R * C)[:n]
    r, c = (key // C).astype(np.int32), (key % C).astype(np.int32)
    v = rng.integers(1, 9, n).astype(np.float32)
    m = dcsr_amd.DcsrMatrix(R, C, pool_factor=4.0)
    m.LoadMatrix(r, c, v)
    xh = rng.integers(-4, 5, C).astype(np.float32)
    x, y = torch.from_numpy(xh).cuda(), torch.empty(R, device="cuda")
    for _ in range(5):  # the copy is built on the way
        m.spmv(x, y)
    torch.cuda.synchronize()
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        m.spmv(x, y)  # eager, on the capture's stream
        s.synchronize()
        with torch.cuda.graph(g, stream=s):
            m.spmv(x, y)
    want = np.zeros(R)
    np.add.at(want, r, v * xh[c])
    for k in range(3):
        y.fill_(7.0)
        g.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(y.cpu().numpy(), want.astype(np.float32))
        m.UpdateMatrix(r, c, np.full(n, k + 1.0, np.float32))  # in place: the rows stay where they are
        np.add.at(want, r, (k + 1.0) * xh[c])
    m.close()
