"""Products of long rows against 64 bits: a row over many waves' ranges, as loaded
and over the paneled copy.  A wave's sum of positive values is off by a few 2^-24
of itself, which averages out over the row's waves; their sums are added in
double and rounded once, so the rms over many rows is that rounding's, at most
2^-24 / sqrt(3) = 3.44e-8, and a little for the waves'."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [3_000, 20_000, 120_000])
@pytest.mark.parametrize("paneled", [False, True])
def test_rows_over_many_waves(L, paneled, monkeypatch):
    import torch
    import dcsr_amd
    if paneled:
        monkeypatch.setenv("DCSR_SPMV_PANEL_COLS", "30000")
        monkeypatch.setenv("DCSR_SPMV_PANEL_MIN_NNZ", "0")
    R, C = min(1_000, 9_000_000 // L), 120_000
    g = torch.Generator(device="cuda").manual_seed(L)
    c = torch.stack([torch.randperm(C, generator=g, device="cuda")[:L].sort()[0] for _ in range(R)]).flatten()
    r = torch.arange(R, device="cuda").repeat_interleave(L)
    v = 1 - torch.rand(R * L, generator=g, device="cuda")
    x = 1 - torch.rand(C, generator=g, device="cuda")
    m = dcsr_amd.DcsrMatrix(R, C, pool_factor=1.0)
    m.LoadMatrix(r.int(), c.int(), v)
    for _ in range(4):
        y = m.spmv(x)
    assert m.info()["spmv_paneled"] == int(paneled)
    want = (v.double() * x[c].double()).view(R, L).sum(1)
    err = ((y.double() - want) / want).abs()
    rms = float((err**2).mean().sqrt())
    print(f"[gpu-error] L={L} paneled={paneled}: rms {rms:.3e} max {float(err.max()):.3e}", flush=True)
    assert rms <= 3.6e-8
    m.close()
