"""A request may write what an earlier one reads: queries that wait together are
answered from their operands as they were when the earlier ones were submitted,
whichever of them are packed.  Small integers: sums are exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("packed", [1, 3])
def test_a_later_query_overwrites_an_earlier_operand(packed):
    import torch
    import dcsr_amd
    R, n = 60_000, 1_500_000
    rng = np.random.default_rng(packed)
    r, c = rng.integers(0, R, n).astype(np.int32), rng.integers(0, R, n).astype(np.int32)
    m = dcsr_amd.DcsrMatrix(R, R)
    m.LoadMatrix(r, c, rng.integers(1, 3, n).astype(np.float32))
    m.UpdateMatrix(r[:1], c[:1], np.ones(1, np.float32))
    srv = dcsr_amd.DcsrServer(m, max_cols=64)
    wide = torch.randint(-2, 3, (R, 64), device="cuda").float()
    sink = torch.empty_like(wide)
    Z = torch.randint(-2, 3, (R, 32), device="cuda").float()
    B = torch.empty((R, 32), device="cuda")
    ys = [torch.empty(R, device="cuda") for _ in range(packed)]
    want_Y = m.spmm(Z)
    for k in range(10):
        B.copy_(torch.randint(-2, 3, (R, 32), device="cuda"))
        xs = [B.view(-1)[q * R:(q + 1) * R] for q in range(packed)]
        want = [m.spmv(x) for x in xs]
        torch.cuda.synchronize()
        for _ in range(4):  # what the others wait behind, so that they form one group
            srv.spmm(wide, sink)
        for x, y in zip(xs, ys):
            srv.spmv(x, y)
        srv.spmm(Z, B)  # whole lines: multiplied in place
        srv.drain()
        torch.cuda.synchronize()
        for y, w in zip(ys, want):
            assert torch.equal(y, w), k
        assert torch.equal(B, want_Y)
    srv.close()
    m.close()
