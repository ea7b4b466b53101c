"""Scratch of a type-1 plan: the row tiles read no record starts (16 bytes a
point) and their plans hold none until a spread that reads them is chosen.
Device memory in use before and after, with the pools' granularity of a few
MiB as margin."""
import pytest

pytestmark = pytest.mark.gpu


def _used(torch):
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info()
    return total - free


def test_row_tile_plans_hold_no_starts():
    import torch
    import wgpunufft_amd as W
    M, margin = 8_000_000, 16 << 20
    x = (2 * torch.rand(M, 2, device="cuda") - 1) * 3.14159
    plan = W.NufftPlan.type1_gpu(W.NufftConfig([128, 128], 1e-6))
    plan.set_points_gpu(x)
    rows = _used(torch)
    plan.set_points_gpu(x)
    assert _used(torch) <= rows + margin
    plan.set_bin_tuning(0, False)  # the output-stationary blocks read them
    plan.set_points_gpu(x)
    assert _used(torch) - rows >= 16 * M - margin
