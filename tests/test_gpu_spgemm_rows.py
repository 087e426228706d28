"""SpGEMM rows at the edges of the row classes (partial products at and just
past each class's largest count), with columns spread over the row's range, all
crowded at one end of it but for one (the bucket sort gives up and the row is
sorted without buckets), and the same few columns again and again; column
counts on both sides of the 32-bit sort keys of each class.  Sums follow the
host path's order, so values are compared bit for bit."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import assert_same_structure

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 15, 16, 17, 31, 32, 33, 64, 65, 96, 97, 128, 129, 255, 256, 257, 512, 513, 1023, 1024, 1025, 2048, 4095,
         4096, 4097, 8191, 8192, 8193, 16383, 16384, 16385]


def case(cols, pattern, seed):
    rng = np.random.default_rng(seed)
    nb = 2200  # rows of B with 8 entries; then one row each of 1..7 entries
    lens = np.concatenate([np.full(nb, 8), np.arange(1, 8)])
    br = np.repeat(np.arange(lens.size), lens)
    bc = []
    for n in lens:
        if pattern == "spread":
            c = np.unique(rng.integers(0, cols, 4 * n + 8))
            c = np.sort(rng.permutation(c)[:n])
        elif pattern == "crowded":
            c = np.concatenate([np.sort(rng.permutation(40)[: n - 1]), [cols - 1]])
        else:
            c = np.arange(n) * 3
        bc.append(c)
    bc = np.concatenate(bc)
    bv = rng.standard_normal(br.size).astype(np.float32)
    B = O.coo_to_csr(lens.size, cols, br.astype(np.int32), bc.astype(np.int32), bv)
    ar, ac = [], []
    for i, p in enumerate(EDGES):
        ids = np.sort(rng.permutation(nb)[: p // 8])
        if p % 8:
            ids = np.concatenate([ids, [nb + p % 8 - 1]])
        ar.append(np.full(ids.size, i))
        ac.append(ids)
    ar, ac = np.concatenate(ar), np.concatenate(ac)
    A = O.coo_to_csr(len(EDGES), lens.size, ar.astype(np.int32), ac.astype(np.int32),
                     rng.standard_normal(ar.size).astype(np.float32))
    return A, B


@pytest.mark.parametrize("pattern", ["spread", "crowded", "repeated"])
@pytest.mark.parametrize("cols", [5_000, 300_000, 3_000_000, 5_000_000, 1 << 26])
def test_row_class_edges(cols, pattern):
    import dcsr_amd
    from tests.helpers import to_host_csr
    A, B = case(cols, pattern, cols % 97)
    mA, mB = dcsr_amd.DcsrMatrix(A.rows, A.cols), dcsr_amd.DcsrMatrix(B.rows, B.cols)
    mA.load_csr(A.off, A.col, A.val)
    mB.load_csr(B.off, B.col, B.val)
    mC = dcsr_amd.spgemm(mA, mB)
    assert_same_structure(to_host_csr(mC), O.spgemm(A.canonical(), B.canonical()), values="exact")
    for m in (mA, mB, mC):
        m.close()
