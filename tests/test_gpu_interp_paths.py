"""Type-2 interpolation picks its kernel by rank, width and point count: few
points in their own order, gathered in bin order, or from LDS tiles.  Every
point's value may depend on that choice in rounding only, so a large set's
values are compared with those of its first points alone (another path), for
each rank and precision, several vectors, points at the ends of the interval
(supports that wrap) and one point.  Bounds: sums of at most 13^3 products
of one precision in another order (2e-6 FP32, 1e-13 FP64).
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,eps", [("f32", 1e-2), ("f32", 1e-6), ("f64", 1e-6), ("f64", 1e-12)])
@pytest.mark.parametrize("n_modes,M", [([500], 70000), ([2_200_000], 60000), ([61, 40], 250000),
                                       ([17, 33, 20], 200000), ([60, 61, 50], 30000)])
def test_interpolation_paths_agree(n_modes, M, prec, eps):
    import torch
    import wgpunufft_amd as W
    f64 = prec == "f64"
    if len(n_modes) == 1 and n_modes[0] > 1000 and not f64:
        pytest.skip("FP32 rounding of that many modes")
    real, cplx = (torch.float64, torch.complex128) if f64 else (torch.float32, torch.complex64)
    B = 3
    gen = torch.Generator(device="cuda").manual_seed(7)
    x = (2 * torch.rand(M, len(n_modes), generator=gen, device="cuda", dtype=torch.float64) - 1)
    x = (x * 3.14159265).clamp(-3.1415925, 3.1415925).to(real)
    x[0], x[1], x[2] = -3.1415925, 3.1415925, 0.0
    N = int(np.prod(n_modes))
    f = torch.randn(B * N, generator=gen, device="cuda", dtype=cplx)
    cfg = W.NufftConfig(n_modes, eps).with_batch(B)
    if f64:
        cfg = cfg.with_precision(W.F64)
    plan = W.NufftPlan.type2_gpu(cfg)
    full = plan.encode_gpu(x, f).view(B, M)
    for m in (1, 500, 9000):
        part = plan.encode_gpu(x[:m].contiguous(), f).view(B, m)
        d = rel_l2(part.cpu().numpy(), full[:, :m].cpu().numpy())
        assert d <= (1e-13 if f64 else 2e-6), (m, d)
