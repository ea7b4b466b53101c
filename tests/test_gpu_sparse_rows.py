"""Sparse 3D type 2: the FFT's last pass writes only the rows that the points
read.  The values must equal the same plan's without that (the same gather
from the whole grid) bit for bit: a few points, points at the interval's ends
(supports that wrap on every axis), several vectors, and a grid that a call
before filled with infinities, of which no written cell may keep one.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,eps,n_modes", [("f32", 1e-6, [104, 97, 110]),
                                              ("f64", 1e-6, [75, 80, 99]),
                                              ("f64", 1e-12, [90, 64, 101])])
@pytest.mark.parametrize("M", [1, 40, 700])
def test_sparse_rows_leave_the_values(prec, eps, n_modes, M):
    import torch
    import wgpunufft_amd as W
    f64 = prec == "f64"
    real, cplx = (torch.float64, torch.complex128) if f64 else (torch.float32, torch.complex64)
    B = 2
    gen = torch.Generator(device="cuda").manual_seed(M)
    x = ((2 * torch.rand(M, 3, generator=gen, device="cuda", dtype=torch.float64) - 1)
         * 3.1415925).to(real)
    x[0] = torch.tensor([-3.1415925, 3.1415925, 3.1415925])
    # enough points in one tile that the same values come from the whole grid
    dense = x[torch.arange(40000, device="cuda") % M].contiguous()
    N = int(np.prod(n_modes))
    f = torch.randn(B * N, generator=gen, device="cuda", dtype=cplx)
    cfg = W.NufftConfig(n_modes, eps).with_batch(B)
    if f64:
        cfg = cfg.with_precision(W.F64)
    plan = W.NufftPlan.type2_gpu(cfg)
    fine = plan.info()["fine"]
    assert np.prod(fine) * (16 if f64 else 8) >= 64e6
    w = plan.info()["width"]
    assert 40000 * w * w * (w + 15) >= 0.5 * np.prod(fine)  # `dense` takes the whole grid
    plan.encode_gpu(x, torch.full_like(f, float("inf")))
    sparse = plan.encode_gpu(x, f).view(B, M).clone()
    whole = plan.encode_gpu(dense, f).view(B, -1)[:, :M]
    assert torch.equal(torch.view_as_real(sparse), torch.view_as_real(whole))
    again = plan.execute_gpu(f).view(B, -1)[:, :M]
    assert torch.equal(torch.view_as_real(again), torch.view_as_real(whole))
