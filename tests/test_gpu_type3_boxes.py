"""Targets grouped by box through workgroup counters: one target to a few past
a workgroup's 2048, targets that all fall into one box, and more boxes than the
counters hold (1024; the rest are counted in global memory).  Each target is
computed once, to the direct sums (src/type3.rs) at the plan's tolerance with
the margin of 100 that the type-3 tests use.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("boxes,count,spread", [
    ([3], 1, 1.0), ([3], 255, 1.0), ([5], 2048, 1.0), ([5], 2049, 1.0), ([4], 6000, 0.1),
    ([2, 3], 4100, 1.0), ([36, 30], 3000, 1.0)])
def test_type3_targets_by_box(boxes, count, spread):
    import torch
    import wgpunufft_amd as W
    from oracle import oracle as O
    dim, eps = len(boxes), 1e-6
    rng = np.random.default_rng(count + dim)
    x = rng.uniform(-2.0, 2.0, (200, dim))
    s = spread * rng.uniform(-20.0, 20.0, (count, dim))
    c = rng.standard_normal(200) + 1j * rng.standard_normal(200)
    plan = W.NufftType3Plan(dim, [(-2, 2)] * dim, [(-20, 20)] * dim, eps=eps, precision=W.F64)
    assert plan.boxes(boxes) == boxes
    out = plan.encode_gpu(*(torch.from_numpy(a).cuda() for a in (x, c, s))).cpu().numpy()
    assert rel_l2(out.reshape(-1), O.direct_type3(x, c, s)) <= 100 * eps
