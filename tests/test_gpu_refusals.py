"""Refused calls leave nothing behind: a canonical export into a negative
capacity writes nothing."""
import ctypes

import numpy as np
import pytest

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
