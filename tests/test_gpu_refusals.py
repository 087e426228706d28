"""Refused calls leave nothing behind: a canonical export into a negative
capacity writes nothing, and a batch refused for a bad index does not count
against the next one."""
import ctypes

import numpy as np
import pytest

import oracle as O
from tests.helpers import assert_same_structure, check_healthy, to_host_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("canon", [0, 1])
@pytest.mark.parametrize("cap", [-1, -2**40])
def test_export_into_a_negative_capacity(canon, cap):
    import torch
    import dcsr_amd
    R = 50
    rng = np.random.default_rng(1)
    r, c = rng.integers(0, R, 600).astype(np.int32), rng.integers(0, 8, 600).astype(np.int32)  # duplicates
    m = dcsr_amd.DcsrMatrix(R, R)
    m.LoadMatrix(r, c, np.ones(r.size, np.float32))
    off = torch.full((R + 1,), 7, dtype=torch.int32, device="cuda")
    col = torch.full((r.size,), 7, dtype=torch.int32, device="cuda")
    val = torch.full((r.size,), 7.0, device="cuda")
    n = ctypes.c_int64(0)
    code = dcsr_amd.lib().dcsr_export_csr(m.handle, off.data_ptr(), col.data_ptr(), val.data_ptr(), cap,
                                          ctypes.byref(n), canon, torch.cuda.current_stream().cuda_stream)
    assert code == 7  # DCSR_ERR_CAPACITY
    assert (off == 7).all() and (col == 7).all() and (val == 7.0).all()
    m.close()


@pytest.mark.parametrize("n", [500, 5_000, 8_000])
@pytest.mark.parametrize("nosync", [False, True])
@pytest.mark.parametrize("clean", ["load", "product"])
def test_a_refused_batch_does_not_refuse_the_next(n, nosync, clean):
    import dcsr_amd
    R = 300
    rng = np.random.default_rng(n)

    def batch(k):
        return (rng.integers(0, R, k).astype(np.int32), rng.integers(0, R, k).astype(np.int32),
                rng.integers(1, 4, k).astype(np.float32))

    m = dcsr_amd.DcsrMatrix(R, R, pool_factor=8.0, min_pool=1 << 20)
    r, c, v = batch(900)
    m.LoadMatrix(np.concatenate([r, r[:50]]), np.concatenate([c, c[:50]]), np.concatenate([v, v[:50]]))  # duplicates
    bad = batch(n)
    bad[0][n // 2] = R
    with pytest.raises(dcsr_amd.DcsrError) as e:
        m.UpdateMatrix(*bad)
    assert e.value.code == 2  # DCSR_ERR_BAD_INDEX
    key = np.unique(r.astype(np.int64) * R + c)
    A = O.coo_to_csr(R, R, (key // R).astype(np.int32), (key % R).astype(np.int32), np.ones(key.size, np.float32))
    if clean == "load":
        m.load_csr(A.off, A.col, A.val)
    else:
        a = dcsr_amd.DcsrMatrix(R, R)
        a.load_csr(A.off, A.col, A.val)
        dcsr_amd.spgemm(a, a, m)
        A = O.spgemm(A.canonical(), A.canonical())
        a.close()
    good = batch(n)
    m.UpdateMatrix(*good, flags=dcsr_amd.UPDATE_NOSYNC if nosync else 0)
    check_healthy(m)
    assert_same_structure(to_host_csr(m), O.update(A, *good))
    m.close()
