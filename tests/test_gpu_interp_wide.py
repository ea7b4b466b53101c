"""Type-2 interpolation of wide FP64 kernels (widths 9 to 16) from LDS tiles:
3D with four lanes per point, 2D on 8 x 8 tiles, on the smallest grids that
qualify and ragged ones (halos that wrap, bins cut by the grid's end, dense
tiles of more than one work item).  The reference gathers every point from
the grid (src/gpu_3d.rs:1238-1359); so does the engine for sparse point sets,
which the tiled values match to FP64 rounding (weights good to a few 1e-15,
sums of up to 4096 products of mixed sign).  FP64 direct sums bound the
transform itself (40 eps, as the other F64 cases).
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


def _run(W, torch, n_modes, eps, x, f):
    plan = W.NufftPlan.type2_gpu(W.NufftConfig(n_modes, eps).with_precision(W.F64))
    out = plan.encode_gpu(torch.from_numpy(x).cuda(), torch.from_numpy(f).cuda())
    return out.cpu().numpy(), plan.info()


@pytest.mark.parametrize("n_modes,shape", [([16, 16, 16], "smallest"), ([19, 25, 16], "ragged")])
@pytest.mark.parametrize("width", range(9, 17))
def test_wide_3d_tiles_match_gather_and_direct_sums(width, n_modes, shape):
    import torch
    import wgpunufft_amd as W
    from oracle import oracle as O
    eps = 10.0 ** -(width - 1)
    rng = np.random.default_rng(width)
    probe = W.NufftPlan.type2_gpu(W.NufftConfig(n_modes, eps).with_precision(W.F64)).info()
    assert probe["width"] == width
    M = 8 * probe["nbins"] + 3000
    x = rng.uniform(-np.pi, np.pi, (M, 3))
    x[:2500] = x[0] + rng.uniform(0, 1e-3, (2500, 3))  # one tile of several work items
    x = np.clip(x, -np.pi, np.nextafter(np.pi, 0))
    f = rng.standard_normal(int(np.prod(n_modes))) + 1j * rng.standard_normal(
        int(np.prod(n_modes)))
    tiled, _ = _run(W, torch, n_modes, eps, x, f)
    pick = rng.permutation(M)[:400]
    gathered, _ = _run(W, torch, n_modes, eps, np.ascontiguousarray(x[pick]), f)
    assert rel_l2(tiled[pick], gathered) <= 1e-13
    ref = O.direct_type2(np.ascontiguousarray(x[pick]), f, n_modes)
    assert rel_l2(tiled[pick], ref) <= max(40 * eps, 1e-13)


@pytest.mark.parametrize("n_modes", [[16, 16], [31, 18]])
@pytest.mark.parametrize("width", range(9, 17))
def test_wide_2d_tiles_match_direct_sums(width, n_modes):
    import torch
    import wgpunufft_amd as W
    from oracle import oracle as O
    eps = 10.0 ** -(width - 1)
    rng = np.random.default_rng(50 + width)
    x = rng.uniform(-np.pi, np.pi, (1500, 2))
    f = rng.standard_normal(int(np.prod(n_modes))) + 1j * rng.standard_normal(
        int(np.prod(n_modes)))
    got, info = _run(W, torch, n_modes, eps, x, f)
    assert info["width"] == width
    assert rel_l2(got, O.direct_type2(x, f, n_modes)) <= max(40 * eps, 1e-13)
