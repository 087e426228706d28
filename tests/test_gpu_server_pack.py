"""Query groups of the serving loop with every kind of column split: widths
around the 32-column blocks, padded leading dimensions, outputs that start off
a line, row counts around the packing tiles.  All values are positive, so each
answer is compared with FP64 within 1e-5 of the sum of its terms."""
import numpy as np
import pytest

import oracle as O
from dcsr_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [1, 63, 64, 65, 1000, 20_001])
@pytest.mark.parametrize("max_cols", [3, 32, 64, 100])
def test_mixed_widths(R, max_cols):
    import torch
    import dcsr_amd
    rng = np.random.default_rng(R + max_cols)
    n = 12 * R
    key = np.unique(rng.integers(0, R, n) * np.int64(R) + rng.integers(0, R, n))
    r, c = (key // R).astype(np.int32), (key % R).astype(np.int32)
    v = (1 - rng.random(r.size)).astype(np.float32)
    S = O.coo_to_csr(R, R, r, c, v).to_scipy(np.float64)
    m = dcsr_amd.DcsrMatrix(R, R)
    m.LoadMatrix(r, c, v)
    srv = dcsr_amd.DcsrServer(m, max_cols=max_cols)
    widths = [k for k in (1, 2, 1, 3, 1, 32, 5, 1, 31, 16, 33, 64, 1, 8, 32, 96, 7) if k <= max_cols]
    inputs = []
    for i in range(48):
        k = widths[i % len(widths)]
        X = (1 - rng.random((R, k + (i % 3) * 3))).astype(np.float32)
        inputs.append((k, torch.from_numpy(X).cuda(), torch.full((R, k + (i % 2) * 4), -7.0, device="cuda")))
    torch.cuda.synchronize()
    tickets = []
    for k, X, Y in inputs:
        if k == 1 and X.shape[1] == 1 and Y.shape[1] == 1:
            tickets.append(srv.spmv(X[:, 0], Y[:, 0])[0])
        else:
            tickets.append(srv.spmm(X[:, :k] if X.shape[1] == k else X[:, :k].contiguous(), Y[:, :k])[0])
    for t in tickets:
        srv.wait(t)
    torch.cuda.synchronize()
    for k, X, Y in inputs:
        want = S @ X[:, :k].cpu().numpy().astype(np.float64)
        got = Y.cpu().numpy().astype(np.float64)
        assert (np.abs(got[:, :k] - want) <= 1e-5 * want + 1e-30).all()
        assert (got[:, k:] == -7.0).all()
    srv.close()
    m.close()
