"""The line FFT's radix plans (2 to 16, one to four passes, composite and prime
radices, one-pass axes) against rocFFT on the same plan: type-1 and type-2
transforms of both signs over fine lengths of every shape the plans take.
Bounds: two FFT engines of one precision over at most 2^22 cells (a few ulp
times log n; 1e-6 FP32, 2e-15 FP64 with a factor of four).
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

# modes whose fine lengths (twice them, rounded up to 2,3,5,7,11,13-smooth)
# run from 14 cells to four passes, with every prime radix among them
MODES = [1, 7, 9, 11, 13, 15, 18, 33, 65, 75, 77, 121, 128, 169, 243, 256, 343, 450, 512, 625,
         1001, 1183]


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("kind,isign", [(1, -1), (2, 1)])
def test_line_fft_radices_match_rocfft(kind, isign, prec):
    import torch
    import wgpunufft_amd as W
    f64 = prec == "f64"
    real, cplx = (torch.float64, torch.complex128) if f64 else (torch.float32, torch.complex64)
    gen = torch.Generator(device="cuda").manual_seed(3)
    x = ((2 * torch.rand(500, 2, generator=gen, device="cuda", dtype=torch.float64) - 1)
         * 3.14159).to(real)
    seen = set()
    for i, n in enumerate(MODES):
        modes = [n, 24] if i % 2 else [24, n]  # as the contiguous and the strided axis
        cfg = W.NufftConfig(modes, 1e-5).with_isign(isign)
        if f64:
            cfg = cfg.with_precision(W.F64)
        v = torch.randn(500 if kind == 1 else modes[0] * modes[1], generator=gen, device="cuda",
                        dtype=cplx)
        out = []
        for engine in ("lines", "rocfft"):
            plan = W.NufftPlan(kind, cfg).set_fft_engine(engine)
            if engine == "lines" and plan.fft_engine() != "lines":
                break  # the length does not fit the LDS lines
            out.append(plan.encode_gpu(x, v).cpu().numpy())
            seen.add(plan.info()["fine"][0 if i % 2 else 1])
        if len(out) == 2:
            d = rel_l2(out[0], out[1])
            assert d <= (2e-15 if f64 else 1e-6), (modes, d)
    assert len(seen) >= 18
