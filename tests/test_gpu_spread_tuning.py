"""The work-plan knobs of the type-1 spread: a plan whose knobs are set to the
defaults sums as a default plan does, bit for bit, and other knobs change the
order of the sums only (a few ulp of FP32 sums of a few hundred terms)."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_modes,M", [([128, 128], 100_000), ([20, 18, 17], 60_000),
                                       ([3000], 200_000)])
def test_knobs_at_their_defaults_are_the_default(n_modes, M):
    import torch
    import wgpunufft_amd as W
    gen = torch.Generator(device="cuda").manual_seed(M)
    x = (2 * torch.rand(M, len(n_modes), generator=gen, device="cuda") - 1) * 3.14159
    c = torch.randn(M, generator=gen, device="cuda", dtype=torch.complex64)

    def run(*knobs):
        plan = W.NufftPlan.type1_gpu(W.NufftConfig(n_modes, 1e-6))
        for k in knobs:
            plan.set_spread_tuning(*k)
        t = plan.tuning()
        return torch.view_as_real(plan.encode_gpu(x, c)).cpu().numpy(), t["light_limit"], t["min_part"]

    default, light, part = run()
    for knobs in ([(light, part)], [(light, 0)], [(0, part)], [(300, 64), (light, part)]):
        assert np.array_equal(run(*knobs)[0], default), knobs
    other, l2, p2 = run((1 << 20, 0))
    assert (l2, p2) == (1 << 20, part)
    assert not np.array_equal(other, default)
    assert rel_l2(other.view(np.float32), default.view(np.float32)) <= 2e-6
