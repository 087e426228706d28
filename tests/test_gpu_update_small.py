"""Small update batches (one workgroup sorts, probes and plans them; 2,048
triples on both sides of the one-launch form, 10,240 of the whole path) against
the oracle after every update, synchronous and asynchronous: keys spread over
the matrix, crowded into one row or one column, one coordinate again and again,
deletions, rows of every length.  Structure and update values bit for bit."""
import numpy as np
import pytest

import oracle as O
from tests.helpers import assert_same_structure, check_healthy, check_layout, fp64_spmv_check, to_host_csr

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 63, 64, 65, 1023, 1024, 1025, 2047, 2048, 2049, 5119, 5120, 5121, 7168, 7169, 10239, 10240, 10241]


def base(rng, R, C, n):
    key = np.unique(rng.integers(0, R, n) * np.int64(C) + (rng.random(n) ** 3 * C).astype(np.int64))
    hub = np.unique(R // 2 * np.int64(C) + rng.integers(0, C, 3000))  # a long row
    key = np.union1d(key, hub)
    return (key // C).astype(np.int32), (key % C).astype(np.int32), rng.integers(1, 5, key.size).astype(np.float32)


def batch(rng, A, n, mode):
    rows = np.repeat(np.arange(A.rows), np.diff(A.off))
    br, bc = rng.integers(0, A.rows, n), rng.integers(0, A.cols, n)
    bv = rng.integers(-3, 4, n).astype(np.float32)
    if mode == "hub":  # every triple in the long row and its neighbour
        br = A.rows // 2 + rng.integers(0, 2, n)
    elif mode == "same":  # a handful of coordinates
        br, bc = br[rng.integers(0, min(n, 5), n)], bc[rng.integers(0, min(n, 5), n)]
        bv = rng.uniform(-1, 1, n).astype(np.float32)
    elif mode == "ends":  # the first and last coordinates, and one in between
        br = np.where(rng.random(n) < 0.5, 0, A.rows - 1)
        bc = np.where(rng.random(n) < 0.5, 0, A.cols - 1)
    elif n > 3:
        pick = rng.integers(0, A.nnz, n // 2)
        br[: pick.size], bc[: pick.size] = rows[pick], A.col[pick]
        bv[: pick.size // 2] = -A.val[pick[: pick.size // 2]]
        p = rng.permutation(n)
        br, bc, bv = br[p], bc[p], bv[p]
    return br.astype(np.int32), bc.astype(np.int32), bv


@pytest.mark.parametrize("mode", ["mixed", "hub", "same", "ends"])
@pytest.mark.parametrize("shape", [(300, 5000, 4000), (200_000, 70_000, 300_000)])
def test_sizes(shape, mode):
    import torch
    import dcsr_amd
    R, C, nnz = shape
    rng = np.random.default_rng(R + len(mode))
    r, c, v = base(rng, R, C, nnz)
    for flags in (0, dcsr_amd.UPDATE_NOSYNC):
        m = dcsr_amd.DcsrMatrix(R, C, pool_factor=1.5 if flags == 0 else 3.0)
        m.LoadMatrix(r, c, v)
        A = O.coo_to_csr(R, C, r, c, v)
        for n in SIZES:
            bt = batch(rng, A, n, mode)
            m.UpdateMatrix(*bt, flags=flags)
            A = O.update(A, *bt)
            assert_same_structure(to_host_csr(m), A)
        x = rng.uniform(-1, 1, C).astype(np.float32)
        y = m.spmv(torch.from_numpy(x).cuda())
        torch.cuda.synchronize()
        fp64_spmv_check(A, x, y.cpu().numpy())
        assert check_layout(m)["nnz"] == A.nnz
        check_healthy(m)
        m.close()


@pytest.mark.parametrize("n", [1, 1024, 2048, 2049, 10240])
def test_bad_index_rejects_the_batch(n):
    import dcsr_amd
    rng = np.random.default_rng(n)
    r, c, v = base(rng, 500, 6000, 4000)
    m = dcsr_amd.DcsrMatrix(500, 6000, pool_factor=4.0)
    m.LoadMatrix(r, c, v)
    want = to_host_csr(m)
    for where, row, col in ((0, 500, 0), (n - 1, 0, 6000), (n // 2, -1, 0), (n // 3, 0, -1)):
        br, bc = rng.integers(0, 500, n).astype(np.int32), rng.integers(0, 6000, n).astype(np.int32)
        br[where], bc[where] = row, col
        with pytest.raises(dcsr_amd.DcsrError) as e:
            m.UpdateMatrix(br, bc, np.ones(n, np.float32))
        assert e.value.code == 2
        m.UpdateMatrix(br, bc, np.ones(n, np.float32), flags=dcsr_amd.UPDATE_NOSYNC)
        assert m.status() == 2 and m.status() == 0
    assert_same_structure(to_host_csr(m), want)
    m.UpdateMatrix(r[:n], c[:n], v[:n])
    assert_same_structure(to_host_csr(m), O.update(O.coo_to_csr(500, 6000, r, c, v), r[:n], c[:n], v[:n]))
    m.close()
