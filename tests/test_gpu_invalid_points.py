"""Points that the fold cannot reach (NaN, infinities, |x| > 4 pi) weigh zero
in every kernel (tests/gpu_invalid_points.rs:20-44): a type-1 transform with
such points, whatever their strengths, is that of the other points, and a
type-2 transform gives them zero and every other point its own value.

Type 1 compares with the same set whose bad points lie at the origin with
strength zero: equal up to the order of sums of a few thousand terms (2e-6
FP32, 1e-13 FP64; the matrix cores by their operands' rounding, 2^-11 to
2^-21).
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

BAD = [np.nan, np.inf, -np.inf, 1e30, -1e30, 5 * np.pi, -5 * np.pi, 13.0]


def _points(M, dim, real, seed):
    """Uniform points, and the same with the first ones bad on one axis."""
    rng = np.random.default_rng(seed)
    x = np.clip(rng.uniform(-np.pi, np.pi, (M, dim)), -3.1415925, 3.1415925).astype(real)
    bad = x.copy()
    for i, v in enumerate(BAD):
        bad[i, i % dim] = v
    return x, bad, rng


def _types(prec):
    return (np.float64, np.complex128) if prec == "f64" else (np.float32, np.complex64)


def _cfg(W, n_modes, eps, prec):
    cfg = W.NufftConfig(n_modes, eps)
    return cfg.with_precision(W.F64) if prec == "f64" else cfg


METHODS = {"mfma_f16": 4e-3, "mfma_bf16x3": 2e-4, "mfma_f16x3": 8e-6}


@pytest.mark.parametrize("dim,prec,eps,spread", [
    (1, "f32", 1e-2, "plain"), (1, "f32", 1e-6, "plain"), (1, "f64", 1e-9, "plain"),
    (2, "f32", 1e-2, "plain"), (2, "f32", 1e-6, "plain"), (2, "f64", 1e-7, "plain"),
    (2, "f64", 1e-12, "plain"), (3, "f32", 1e-3, "plain"), (3, "f32", 1e-6, "plain"),
    (3, "f64", 1e-5, "plain"), (3, "f64", 1e-9, "plain"), (2, "f32", 1e-6, "blocks"),
    (3, "f32", 1e-6, "blocks"), (3, "f64", 1e-9, "blocks"),
    (3, "f32", 1e-6, "mfma_f16x3"), (3, "f32", 1e-6, "mfma_bf16x3"), (3, "f32", 1e-3, "mfma_f16")])
def test_type1_bad_points_add_nothing(dim, prec, eps, spread):
    import torch
    import wgpunufft_amd as W
    real, cplx = _types(prec)
    n_modes = [60] if dim == 1 else [20, 18, 17][:dim]
    for M in (len(BAD), 3000):
        x, bad, rng = _points(M, dim, real, 10 * dim + M)
        c = (rng.standard_normal((2, M)) + 1j * rng.standard_normal((2, M))).astype(cplx)
        ref_x, ref_c = x.copy(), c.copy()
        ref_x[: len(BAD)] = 0
        ref_c[:, : len(BAD)] = 0
        plan = W.NufftPlan.type1_gpu(_cfg(W, n_modes, eps, prec).with_batch(2))
        if spread == "blocks":
            plan.set_bin_tuning(0, False)
        elif spread != "plain":
            plan.set_spread_method(spread)
        out = [plan.encode_gpu(torch.from_numpy(a).cuda(), torch.from_numpy(v).cuda().reshape(-1))
               .cpu().numpy() for a, v in ((bad, c), (bad, ref_c), (ref_x, ref_c))]
        bound = METHODS.get(spread, 2e-6 if prec == "f32" else 1e-13)
        for got in out[:2]:
            if M == len(BAD):
                assert not got.any()
            else:
                assert rel_l2(got, out[2]) <= bound


@pytest.mark.parametrize("n_modes,M,prec,eps", [
    ([60], 500, "f32", 1e-6), ([60], 500, "f64", 1e-9),          # gathered, unsorted
    ([31, 18], 1500, "f32", 1e-6), ([31, 18], 1500, "f64", 1e-12),   # 2D, the points' own order
    ([31, 18], 160_000, "f32", 1e-6), ([31, 18], 160_000, "f64", 1e-7),  # 2D tiles
    ([31, 18], 40_000, "f64", 1e-12),
    ([20, 18, 17], 2000, "f32", 1e-6), ([60, 61, 50], 30_000, "f32", 1e-6),  # 3D gathers
    ([20, 18, 17], 40_000, "f32", 1e-6), ([20, 18, 17], 300_000, "f32", 1e-2),  # 3D tiles
    ([20, 18, 17], 40_000, "f64", 1e-6), ([20, 18, 17], 40_000, "f64", 1e-9),
    ([20, 18, 17], 40_000, "f64", 1e-14)])
def test_type2_bad_points_are_zero(n_modes, M, prec, eps):
    import torch
    import wgpunufft_amd as W
    real, cplx = _types(prec)
    x, bad, rng = _points(M, len(n_modes), real, M)
    N = int(np.prod(n_modes))
    f = torch.from_numpy((rng.standard_normal(N) + 1j * rng.standard_normal(N)).astype(cplx)).cuda()
    plan = W.NufftPlan.type2_gpu(_cfg(W, n_modes, eps, prec))
    good = plan.encode_gpu(torch.from_numpy(x).cuda(), f).cpu().numpy()
    got = plan.encode_gpu(torch.from_numpy(bad).cuda(), f).cpu().numpy()
    assert not got[: len(BAD)].any()
    assert np.array_equal(got[len(BAD):], good[len(BAD):])


@pytest.mark.parametrize("n_modes", [[31, 18], [20, 18, 17]])
def test_batches_of_bad_points(n_modes):
    import torch
    import wgpunufft_amd as W
    dim, N = len(n_modes), int(np.prod(n_modes))
    cfg = W.NufftConfig(n_modes, 1e-6)
    xs, vs, ms = [], [], []
    for M in (3000, 40_000):
        _, bad, rng = _points(M, dim, np.float32, M)
        xs.append(torch.from_numpy(bad).cuda())
        for n, to in ((M, vs), (N, ms)):
            v = rng.standard_normal(n) + 1j * rng.standard_normal(n)
            to.append(torch.from_numpy(v.astype(np.complex64)).cuda())
    for many, kind, values in ((W.encode_type1_many, 1, vs), (W.encode_type2_many, 2, ms)):
        plans = [W.NufftPlan(kind, cfg) for _ in xs]
        for plan, x, v, out in zip(plans, xs, values, [o.clone() for o in many(plans, xs, values)]):
            alone = plan.encode_gpu(x, v)
            assert torch.equal(torch.view_as_real(out), torch.view_as_real(alone))
            assert torch.isfinite(torch.view_as_real(out)).all()
            if kind == 2:
                assert not out[: len(BAD)].any()
