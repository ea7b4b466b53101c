"""Points kept for many executes are sorted where an encode of the same points
is not (one execute does not pay for the sort).  The sort may not change a
value: executes over kept points, encodes and vectors one by one give the same
bits, on either side of the 8 points a tile from which kept 2D sets are sorted.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,eps", [("f32", 1e-6), ("f64", 1e-6), ("f64", 1e-11)])
@pytest.mark.parametrize("n_modes,M,batch,kept_sorted,encode_sorted", [
    ([500], 20_000, 1, False, False),
    ([40, 40], 799, 1, False, False), ([40, 40], 800, 1, True, False),   # 10 x 10 tiles of 8 x 8
    ([40, 40], 20_000, 8, True, False),
    ([40, 40], 20_000, 96, True, True),   # an encode of over 1e9 bytes of gathers
    ([32, 36, 35], 3000, 1, False, False), ([32, 36, 35], 3000, 4, True, False),
    ([16, 18, 17], 3000, 4, False, False),
    ([104, 97, 110], 300, 4, True, False)])   # the last FFT pass on marked rows
def test_kept_points_give_the_bits_of_encodes(n_modes, M, batch, kept_sorted, encode_sorted, prec,
                                              eps):
    import torch
    import wgpunufft_amd as W
    f64 = prec == "f64"
    real, cplx = (torch.float64, torch.complex128) if f64 else (torch.float32, torch.complex64)
    gen = torch.Generator(device="cuda").manual_seed(M + batch)
    x = ((2 * torch.rand(M, len(n_modes), generator=gen, device="cuda", dtype=torch.float64) - 1)
         * 3.1415925).to(real)
    N = int(np.prod(n_modes))
    f = torch.randn(batch * N, generator=gen, device="cuda", dtype=cplx)
    cfg = W.NufftConfig(n_modes, eps).with_batch(batch)
    plan = W.NufftPlan.type2_gpu(cfg.with_precision(W.F64) if f64 else cfg)
    encoded = plan.encode_gpu(x, f).clone()
    torch.cuda.synchronize()
    # an encode's timing covers its execute; the sort stage ran or did not
    plan.timing_history(True)
    plan.encode_gpu(x, f)
    assert (plan.stage_times()["sort"] is not None) == encode_sorted
    again = plan.execute_gpu(f)  # an encode's points executed again are kept ones
    assert (plan.stage_times()["sort"] is not None) == (kept_sorted and not encode_sorted)
    assert torch.equal(torch.view_as_real(again), torch.view_as_real(encoded))
    plan.execute_gpu(f)
    assert plan.stage_times()["sort"] is None
    plan.set_points_gpu(x)
    assert (plan.stage_times()["sort"] is not None) == kept_sorted
    plan.timing_history(False)
    for _ in range(2):
        kept = plan.execute_gpu(f)
        assert torch.equal(torch.view_as_real(kept), torch.view_as_real(encoded))
    if batch > 1:
        one = plan.encode_gpu(x, f[N:2 * N].contiguous(), active_batch=1)
        assert torch.equal(torch.view_as_real(one), torch.view_as_real(encoded[M:2 * M]))


def test_encode_errors_keep_the_points():
    """An encode refused for its values has set the points, as set_points_gpu
    and execute_gpu one after the other do."""
    import torch
    import wgpunufft_amd as W
    plan = W.NufftPlan.type2_gpu(W.NufftConfig([16, 16], 1e-6))
    x = torch.rand(300, 2, device="cuda")
    f = torch.randn(256, dtype=torch.complex64, device="cuda")
    for bad in (f[:100], f.to(torch.complex128)):
        with pytest.raises(ValueError):
            plan.encode_gpu(x, bad)
        got = plan.execute_gpu(f)
        assert torch.equal(torch.view_as_real(got), torch.view_as_real(plan.encode_gpu(x, f)))
    with pytest.raises(W.NufftError):
        plan.encode_gpu(x, f.repeat(2), active_batch=2)
    assert plan.execute_gpu(f).numel() == 300
