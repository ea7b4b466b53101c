"""Vectors summed two at a time on the 3D matrix-core tiles, an odd last one
by itself (tests/gpu_nufft_batch.rs:96-133, batch == loop): each vector's
sums, with its own strength scale, are bit for bit those of the vector alone,
for every operand form, the smallest and the largest kernel width, counts
about a staged chunk of 64 and tiles that are split into parts.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [2, 3, 5])
@pytest.mark.parametrize("method", ["mfma_f16", "mfma_f16x3", "mfma_bf16x3"])
@pytest.mark.parametrize("eps", [1e-1, 1e-7])
def test_mfma_vectors_in_pairs_equal_single(method, eps, batch):
    import torch
    import wgpunufft_amd as W
    n_modes = [20, 18, 17]
    rng = np.random.default_rng(10 * batch + len(method))
    plan = W.NufftPlan.type1_gpu(W.NufftConfig(n_modes, eps).with_batch(batch))
    plan.set_spread_method(method)
    for M in (1, 63, 65, 6000):
        x = rng.uniform(-3.14159, 3.14159, (M, 3)).astype(np.float32)
        if M == 6000:  # most of them in one tile: parts and partial sums
            x[:5000] *= 0.05
        xt = torch.from_numpy(x).cuda()
        c = rng.standard_normal((batch, M)) + 1j * rng.standard_normal((batch, M))
        c *= 10.0 ** rng.uniform(-6, 6, (batch, 1))
        ct = torch.from_numpy(c.astype(np.complex64)).cuda()
        together = plan.encode_gpu(xt, ct.reshape(-1)).cpu().numpy().reshape(batch, -1)
        for v in range(batch):
            alone = plan.encode_gpu(xt, ct[v].contiguous(), active_batch=1).cpu().numpy()
            assert np.array_equal(alone.reshape(-1).view(np.uint32),
                                  together[v].view(np.uint32)), (M, v)
        ref = W.NufftPlan.type1_gpu(W.NufftConfig(n_modes, eps)).encode_gpu(
            xt, ct[batch - 1].contiguous()).cpu().numpy().reshape(-1)
        # operands rounded to 2^-11 (f16), 2^-16 (bf16 pairs) or 2^-21 (f16 pairs)
        bound = {"mfma_f16": 2e-3, "mfma_bf16x3": 1e-4, "mfma_f16x3": 4e-6}[method]
        assert np.linalg.norm(together[-1] - ref) <= bound * np.linalg.norm(ref)
