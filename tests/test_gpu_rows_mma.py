"""The plain row tiles' matrix-instruction sum (four records per
v_mfma_{f32,f64}_16x16x4, weights from panel polynomials) at the sizes where
it can go wrong: one record to a few past a staged chunk of 64 (groups of
four and eight with missing records), supports that touch one row or column
block of a tile, every kernel width, against the output-stationary blocks,
which evaluate every weight by sqrt and exp (src/gpu_nd_spread.rs:1583-1667).

Bounds: both sides sum a few hundred products at most.  FP64: the blocks'
weight exp(beta (sqrt(q) - 1)) carries up to beta 2^-54 (2e-15 at beta 37) on
each axis, the panel polynomials less, sums and the FFT a few 1e-16: 1e-14.
FP32: beta 2^-25 (about 5e-7 at beta 18), the sums and the FFT a few 1e-7.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

COUNTS = [1, 2, 3, 4, 5, 7, 8, 9, 63, 64, 65, 67, 131]


def _both(prec, eps, n_modes, x, c):
    import torch
    import wgpunufft_amd as W
    cfg = W.NufftConfig(n_modes, eps)
    if prec == "f64":
        cfg = cfg.with_precision(W.F64)
    xt, ct = torch.from_numpy(x).cuda(), torch.from_numpy(c).cuda()
    out = []
    for rows in (True, False):
        plan = W.NufftPlan.type1_gpu(cfg).set_bin_tuning(0, rows)
        out.append(plan.encode_gpu(xt, ct).cpu().numpy())
        if rows:
            assert plan.tuning()["plain_rows"]
    return out


def _points(M, fine, dim, dtype, rng):
    """Points within one tile and its reach, so that supports end inside it."""
    cell = rng.uniform(-14.0, 18.0, (M, dim))
    x = np.mod(cell * 2 * np.pi / np.asarray(fine) + np.pi, 2 * np.pi) - np.pi
    return np.clip(x, -3.1415925, 3.1415925).astype(dtype)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("prec,eps", [("f32", 10.0 ** -e) for e in range(1, 8)] +
                         [("f64", 10.0 ** -e) for e in range(1, 16)])
def test_rows_sum_few_records(dim, prec, eps):
    w = max(2, int(np.ceil(-np.log10(eps) - 1e-9)) + 1)
    real, cplx = (np.float64, np.complex128) if prec == "f64" else (np.float32, np.complex64)
    n_modes = [20, 18, 17][:dim]
    rng = np.random.default_rng(100 * w + dim)
    bound = 2e-6 if prec == "f32" else 1e-14
    for M in COUNTS:
        x = _points(M, [2 * n for n in n_modes], dim, real, rng)
        c = (rng.standard_normal(M) + 1j * rng.standard_normal(M)).astype(cplx)
        rows, blocks = _both(prec, eps, n_modes, x, c)
        d = rel_l2(rows, blocks)
        assert d <= bound, f"dim {dim} {prec} w {w} M {M}: {d:.3e}"


@pytest.mark.parametrize("sigma", [2.0, 1.25])
@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("eps", [10.0 ** -e for e in range(1, 8)])
def test_fp32_rows_are_as_exact_as_the_blocks(eps, dim, sigma):
    """FP32 rows and blocks against the same kernel's FP64 transform: the
    rows' weights carry no more rounding than sqrtf and expf, at the narrow
    widths of end cells alone too (one record at a time, so that no error
    averages out; a tenth for the spread of 400 records)."""
    import torch
    import wgpunufft_amd as W
    n_modes = [20, 18, 17][:dim]
    rng = np.random.default_rng(dim)
    cfg = W.NufftConfig(n_modes, eps).with_sigma(sigma)
    exact = W.NufftPlan.type1_gpu(cfg.with_precision(W.F64))
    info = exact.info()
    if info["width"] > 8:
        pytest.skip("beyond the FP32 row tiles")
    err = {}
    x = _points(400, [2 * n for n in n_modes], dim, np.float32, rng)
    for rows in (True, False):
        plan = W.NufftPlan.type1_gpu(cfg).set_bin_tuning(0, rows)
        assert plan.info()["width"] == info["width"]
        one = torch.ones(1, dtype=torch.complex64, device="cuda")
        got, ref = [], []
        for p in x:
            xt = torch.from_numpy(p[None]).cuda()
            got.append(plan.encode_gpu(xt, one).clone())
            ref.append(exact.encode_gpu(xt.double(), one.to(torch.complex128)).clone())
        err[rows] = rel_l2(torch.stack(got).cpu().numpy(), torch.stack(ref).cpu().numpy())
    assert err[True] <= 1.1 * err[False]
