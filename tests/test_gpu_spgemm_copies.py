"""SpGEMM with and without its copies of the operands: every row class both ways
bit for bit against the oracle, and products that find no room for the copies, or
for their own output beside them."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import assert_same_structure, to_host_csr
from tests.test_gpu_spgemm_rows import case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("copies", [False, True])
@pytest.mark.parametrize("cols,pattern", [(5_000, "crowded"), (300_000, "spread"), (5_000_000, "repeated"),
                                          (1 << 26, "spread")])
def test_row_classes_both_ways(copies, cols, pattern, monkeypatch):
    import dcsr_amd
    monkeypatch.setenv("DCSR_SPGEMM_PAIR_MIN", "0" if copies else str(1 << 60))
    A, B = case(cols, pattern, cols % 89)
    mA, mB = dcsr_amd.DcsrMatrix(A.rows, A.cols, pool_factor=4.0), dcsr_amd.DcsrMatrix(B.rows, B.cols)
    mA.load_csr(A.off, A.col, A.val)
    mB.load_csr(B.off, B.col, B.val)
    mC = dcsr_amd.DcsrMatrix(A.rows, B.cols)
    rng = np.random.default_rng(cols)
    for _ in range(2):  # as loaded, then with rows anywhere in the pool
        dcsr_amd.spgemm(mA, mB, mC)
        assert_same_structure(to_host_csr(mC), O.spgemm(A.canonical(), B.canonical()))
        b = (rng.integers(0, A.rows, 200).astype(np.int32), rng.integers(0, A.cols, 200).astype(np.int32),
             rng.standard_normal(200).astype(np.float32))
        mA.UpdateMatrix(*b)
        A = O.update(A, *b)
    for m in (mA, mB, mC):
        m.close()


@pytest.mark.parametrize("short_of", ["copies", "output"])
def test_no_room_for_the_copies(short_of):
    """20M entries of A: their records take 200 MB, the output little or 120 MB."""
    import torch
    import dcsr_amd
    R, L, n = 200_000, 100, 1_000_000
    g = torch.Generator(device="cuda").manual_seed(5)
    col = (torch.randint(0, n // L, (R * L,), generator=g, device="cuda") +
           torch.arange(L, device="cuda").repeat(R) * (n // L)).int()
    mA = dcsr_amd.DcsrMatrix(R, n, pool_factor=1.0)
    mA.load_csr(torch.arange(R + 1, device="cuda") * L, col, torch.ones(R * L, device="cuda"))
    # one entry in some rows of B: every A entry there is a partial
    step = 1_000 if short_of == "copies" else 4
    rows = torch.arange(0, n, step, device="cuda")
    mB = dcsr_amd.DcsrMatrix(n, 50, pool_factor=1.0)
    mB.LoadMatrix(rows.int(), (rows // step % 50).int(), torch.ones(rows.numel(), device="cuda"))
    hit = (col % step == 0)
    want = torch.zeros(R * 50, device="cuda")
    want.index_add_(0, (torch.arange(R, device="cuda").repeat_interleave(L) * 50 + (col // step % 50).long())[hit],
                    torch.ones(int(hit.sum()), device="cuda"))
    mC = dcsr_amd.DcsrMatrix(R, 50, pool_factor=1.0)
    torch.cuda.empty_cache()
    torch.cuda.synchronize()
    leave, ballast = (120 if short_of == "copies" else 260) << 20, []
    while torch.cuda.mem_get_info()[0] > leave + (16 << 20):  # the first allocation can leave more than was asked
        ballast.append(torch.empty(torch.cuda.mem_get_info()[0] - leave, dtype=torch.uint8, device="cuda"))
    dcsr_amd.spgemm(mA, mB, mC)
    del ballast
    off, c, v = mC.to_csr()
    got = torch.zeros(R * 50, device="cuda")
    got[torch.repeat_interleave(torch.arange(R, device="cuda"), (off[1:] - off[:-1]).long()) * 50 + c.long()] = v
    assert torch.equal(got, want)
    for m in (mA, mB, mC):
        m.close()
