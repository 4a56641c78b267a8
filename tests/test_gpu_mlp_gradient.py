"""The predictor's gradient at the edges of its tiles (16 samples), blocks (4
wavefronts) and grid (256 blocks: from 16,385 samples on a wavefront takes a
second tile), against the CPU mirror with the same BF16 roundings.

Bars: per parameter block 1e-2 of its 2-norm -- two BF16 roundings (2^-9 each)
of a derivative may fall the other way where FP32 sums differ in order, and at
one sample a block is a handful of products; the loss, FP32 per sample, 1e-4
relative.  Two calls give the same bits.
"""
import numpy as np
import pytest

import intpointsfem_amd as ipf
from oracle import mlp as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65, 1000, 16384, 16385, 40001])
def test_gradient(gpu, n):
    import torch
    rng = np.random.default_rng(n)
    feat = np.zeros((n, 8), dtype=np.float32)
    feat[:, :3] = np.sort(rng.normal(0, 3, (n, 3)), axis=1)[:, ::-1]
    feat[:, 3] = rng.uniform(0, 3, n)
    feat[:, 4:6] = rng.uniform(0.35, 0.7, (n, 2))
    feat[:, 6] = rng.exponential(1.0, n)
    label = rng.integers(0, 5, n).astype(np.int32)
    target = rng.normal(0, 1, n).astype(np.float32)
    mlp = ipf.MLP(device=0, seed=3)
    args = tuple(torch.as_tensor(a, device=gpu) for a in (feat, label, target))
    loss, grad = mlp.gradient(*args)
    loss2, grad2 = mlp.gradient(*args)
    assert loss == loss2 and np.array_equal(grad, grad2)
    ref_loss, ref = M.gradient(mlp.params(), feat, label, target)
    assert abs(loss - ref_loss) <= 1e-4 * abs(ref_loss)
    ends = [M.OFF_W1, M.OFF_B1, M.OFF_W2, M.OFF_B2, M.OFF_W3, M.OFF_B3, M.NPAR]
    for a, b in zip(ends[:-1], ends[1:]):
        assert np.linalg.norm(grad[a:b] - ref[a:b]) <= 1e-2 * np.linalg.norm(ref[a:b]), (a, b)
