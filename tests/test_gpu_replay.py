"""Updates replayed from a captured graph: the rows change without a call, so
every later call on the matrix (products, squares, exports, compaction, further
updates) has to find them out for itself.  Before each replay the counters are
queried, so that the host holds figures which the replay then outdates, and each
replay brings other triples in the same buffers.  Small integers: every order of
summation is exact, so results are compared for equality with the oracle's."""
import ctypes

import numpy as np
import pytest

import oracle as O
from tests.helpers import assert_same_structure, check_healthy, check_layout, to_host_csr

pytestmark = pytest.mark.gpu
R = 400


def batch(rng, n):
    return (rng.integers(0, R, n).astype(np.int32), rng.integers(0, R, n).astype(np.int32),
            rng.integers(-2, 4, n).astype(np.float32))


class Replayed:
    """A matrix, its oracle, and a graph that holds one update of n triples (and
    a product when y is given)."""

    def __init__(self, entry, n, product=False):
        import torch
        import dcsr_amd
        self.torch, self.D = torch, dcsr_amd
        self.rng = np.random.default_rng(n)
        r, c, v = batch(self.rng, 500)
        self.A = O.update(O.coo_to_csr(R, R, r[:0], c[:0], v[:0]), r, c, v)
        self.m = dcsr_amd.DcsrMatrix(R, R, min_pool=3_000_000)
        self.m.load_csr(self.A.canonical().off, self.A.canonical().col, self.A.canonical().val)
        self.buf = [torch.zeros(n, dtype=t, device="cuda") for t in (torch.int32, torch.int32, torch.float32)]
        self.x = torch.from_numpy(self.rng.integers(-3, 4, R).astype(np.float32)).cuda()
        self.y = torch.empty(R, device="cuda")
        self.entry, self.n = entry, n
        s, self.g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            self.update()  # zeros: changes nothing, sizes what a capture cannot allocate
            self.m.spmv(self.x, self.y)
            s.synchronize()
            with torch.cuda.graph(self.g, stream=s):
                self.update()
                if product:
                    self.m.spmv(self.x, self.y)
        torch.cuda.synchronize()

    def update(self):
        if self.entry == "update":
            self.m.UpdateMatrix(*self.buf, flags=self.D.UPDATE_NOSYNC)
        else:
            code = self.D.lib().dcsr_update_noalloc(self.m.handle, *(t.data_ptr() for t in self.buf), self.n,
                                                    self.D.UPDATE_NOSYNC, self.torch.cuda.current_stream().cuda_stream)
            assert code == 0

    def replay(self):
        assert self.m.info()["nnz"] == self.A.nnz
        b = batch(self.rng, self.n)
        for t, a in zip(self.buf, b):
            t.copy_(self.torch.from_numpy(a))
        self.g.replay()
        self.torch.cuda.synchronize()
        self.A = O.update(self.A, *b)

    def product(self):
        return (self.A.to_scipy(np.float64) @ self.x.cpu().numpy()).astype(np.float32)


@pytest.mark.parametrize("entry", ["noalloc", "update"])
@pytest.mark.parametrize("n", [1_000, 9_000])
def test_calls_after_a_replay(entry, n):
    t = Replayed(entry, n)
    torch, D, m = t.torch, t.D, t.m
    other = D.DcsrMatrix(R, R)
    r, c, v = batch(t.rng, 900)
    B = O.update(O.coo_to_csr(R, R, r[:0], c[:0], v[:0]), r, c, v).canonical()
    other.load_csr(B.off, B.col, B.val)
    C = [D.DcsrMatrix(R, R) for _ in range(3)]

    def exported():
        off = torch.empty(R + 1, dtype=torch.int32, device="cuda")
        col, val = torch.empty(R * R, dtype=torch.int32, device="cuda"), torch.empty(R * R, device="cuda")
        k = ctypes.c_int64(0)
        D.check(D.lib().dcsr_export_csr(m.handle, off.data_ptr(), col.data_ptr(), val.data_ptr(), R * R,
                                        ctypes.byref(k), 0, torch.cuda.current_stream().cuda_stream))
        return O.Csr(R, R, off.cpu().numpy(), col[:k.value].cpu().numpy(), val[:k.value].cpu().numpy())

    def square(i, A, B, a, b):
        return lambda: assert_same_structure(to_host_csr(D.spgemm(a, b, C[i])), O.spgemm(A().canonical(), B().canonical()))

    def updated(flags):
        def go():
            b = batch(t.rng, 700)
            m.UpdateMatrix(*b, flags=flags)
            t.A = O.update(t.A, *b)
            assert_same_structure(exported(), t.A)
        return go

    def compacted():
        m.SortMatrixRow()
        check_layout(m)
        assert_same_structure(exported(), t.A)

    X = torch.stack([t.x, -t.x, 2 * t.x], 1)
    checks = [
        lambda: np.testing.assert_array_equal(m.spmv(t.x).cpu().numpy(), t.product()),
        square(0, lambda: t.A, lambda: t.A, m, m),
        square(1, lambda: t.A, lambda: B, m, other),
        square(2, lambda: B, lambda: t.A, other, m),
        lambda: assert_same_structure(exported(), t.A),
        lambda: np.testing.assert_array_equal(m.spmm(X).cpu().numpy()[:, 2], 2 * t.product()),
        updated(0),
        updated(D.UPDATE_NOSYNC),
        square(0, lambda: t.A, lambda: t.A, m, m),
        compacted,  # last: it moves the pool away from the graph
    ]
    for k, check in enumerate(checks):
        print(f"[gpu-replay] {entry} n={n} check {k}", flush=True)
        t.replay()
        check()
    check_healthy(m)
    for h in [m, other] + C:
        h.close()


@pytest.mark.parametrize("entry", ["noalloc", "update"])
def test_a_product_in_the_graph_follows_the_rows(entry):
    t = Replayed(entry, 5_000, product=True)
    for _ in range(4):
        t.replay()
        np.testing.assert_array_equal(t.y.cpu().numpy(), t.product())
        t.y.fill_(7.0)
    check_healthy(t.m)
    t.m.close()


def test_a_captured_product_of_a_paneled_matrix_follows_updates(monkeypatch):
    """Many panels and many entries per panel: the copy that an eager product
    takes is not what a capture records."""
    import torch
    import dcsr_amd
    monkeypatch.setenv("DCSR_SPMV_PANEL_COLS", "300")
    monkeypatch.setenv("DCSR_SPMV_PANEL_MIN_NNZ", "500")
    C, n = 3_000, 4_000
    rng = np.random.default_rng(7)
    key = np.sort(rng.permutation(R * C)[:n])
    r, c = (key // C).astype(np.int32), (key % C).astype(np.int32)
    v = rng.integers(1, 9, n).astype(np.float32)
    m = dcsr_amd.DcsrMatrix(R, C, pool_factor=8.0)
    m.LoadMatrix(r, c, v)
    xh = rng.integers(-4, 5, C).astype(np.float32)
    x, y = torch.from_numpy(xh).cuda(), torch.empty(R, device="cuda")
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        for _ in range(5):
            m.spmv(x, y)
        assert m.info()["spmv_paneled"] == 1
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
