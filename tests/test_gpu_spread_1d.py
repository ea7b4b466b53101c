"""1D type-1 spread, where a lane walks the records of its own cells: grids
of one block and of a few cells, ragged ones whose last block is cut and
whose reach wraps, dense sets split into parts, every kernel width, against
FP64 direct sums (src/direct.rs:9-62; the reference's 1D bound of 20 eps,
tests/gpu_nufft_1d.rs) and for bitwise repeat.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_modes,M", [(1, 1), (3, 7), (16, 300), (127, 65), (128, 5000),
                                       (200, 40000), (1001, 20000)])
@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_1d_spread_matches_direct_sums(n_modes, M, prec):
    import torch
    import wgpunufft_amd as W
    from oracle import oracle as O
    f64 = prec == "f64"
    rng = np.random.default_rng(n_modes + M)
    x = rng.uniform(-np.pi, np.pi, (M, 1))
    x[: M // 3] = 0.4 + 0.01 * rng.standard_normal((M // 3, 1))
    x[-1] = np.pi - 1e-6  # its support wraps
    x = np.clip(x, -3.1415925, 3.1415925).astype(np.float64 if f64 else np.float32)
    c = (rng.standard_normal(M) + 1j * rng.standard_normal(M)).astype(
        np.complex128 if f64 else np.complex64)
    ref = O.direct_type1(x.astype(np.float64), c.astype(np.complex128), [n_modes])
    for e in range(1, 16 if f64 else 7):
        eps = 10.0 ** -e
        cfg = W.NufftConfig([n_modes], eps)
        if f64:
            cfg = cfg.with_precision(W.F64)
        plan = W.NufftPlan.type1_gpu(cfg)
        xt, ct = torch.from_numpy(x).cuda(), torch.from_numpy(c).cuda()
        a = plan.encode_gpu(xt, ct).clone()
        b = plan.execute_gpu(ct)
        assert torch.equal(torch.view_as_real(a), torch.view_as_real(b))
        got = rel_l2(a.cpu().numpy(), ref)
        assert got <= max(20 * eps, 1e-13 if f64 else 2e-6), (eps, got)
