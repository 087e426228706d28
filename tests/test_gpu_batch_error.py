"""Products of rewritten rows of the batched step against 64 bits.  A row's product
is summed in double whatever its length, so for positive values two roundings are
left: that of each product and that of the result, 2^-24 of y each at most.  The
first averages out over a row of hundreds of entries, so the rms over many rows is
the second's alone: at most 2^-24 / sqrt(3) = 3.44e-8."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [200, 500, 1_024, 2_000])
def test_rewritten_rows(L):
    import torch
    import dcsr_amd
    rng = np.random.default_rng(L)
    count, size, R = 100, 4_096, 8
    sizes = np.full(count, size, np.int32)
    b = dcsr_amd.DcsrBatch(sizes, sizes, pool_factor=4.0)
    col = np.concatenate([np.sort(rng.permutation(size)[:L]) for _ in range(count * R)]).astype(np.int32)
    row = np.tile(np.repeat(np.arange(R), L), count).astype(np.int32)
    val = (1 - rng.random(col.size)).astype(np.float32)
    b.load_coo(np.arange(count + 1, dtype=np.int64) * (R * L), row, col, val)
    x = (1 - rng.random(b.total_cols)).astype(np.float32)
    br = np.tile(np.arange(R), count).astype(np.int32)  # one entry into every row
    bc = np.array([next(c for c in rng.permutation(size) if c not in set(col[i * L:(i + 1) * L]))
                   for i in range(count * R)], np.int32)
    bv = (1 - rng.random(br.size)).astype(np.float32)
    y = b.step(np.arange(count + 1, dtype=np.int64) * R, br, bc, bv, x=torch.from_numpy(x).cuda())
    y = y.cpu().numpy().astype(np.float64).reshape(count, size)[:, :R].ravel()
    mat = np.repeat(np.arange(count), R)
    want = (val.astype(np.float64).reshape(-1, L) * x[mat[:, None] * size + col.reshape(-1, L)].astype(np.float64)).sum(1)
    want += bv.astype(np.float64) * x[mat * size + bc].astype(np.float64)
    err = np.abs(y - want) / want
    assert err.max() <= 2.0**-23 * (1 + 2.0**-20)
    assert np.sqrt((err**2).mean()) <= 3.5e-8
    b.close()
