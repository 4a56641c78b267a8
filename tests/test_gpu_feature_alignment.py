"""The predictor's features at any float address: extraction, gradient and
inference on a feature array 1 to 3 floats behind a 16-byte boundary give the
bits of an aligned one."""
import numpy as np
import pytest

import intpointsfem_amd as ipf
from intpointsfem_amd import wellbore as wb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [1, 2, 3])
def test_shifted_features(gpu, shift):
    import torch
    m = wb.make_mesh((7, 6, 2, 1.1))
    ctx = ipf.StructMatrix(m, device=0)
    sm, ctx = ctx, ctx.context()
    n = sm.sizes()["npts"]
    u = torch.as_tensor(wb.lame_displacement(m.nodes(), wb.normal_stress(10), scale=6.0), dtype=torch.float64, device=gpu)
    mlp = ipf.MLP(device=0, seed=2)
    out = []
    for s in (0, shift):
        buf = torch.full((8 * n + 4,), float("nan"), dtype=torch.float32, device=gpu)
        feat = buf[s:s + 8 * n]
        br = torch.zeros(n, dtype=torch.int32, device=gpu)
        tg = torch.zeros(n, dtype=torch.float32, device=gpu)
        pr, po = torch.zeros_like(br), torch.zeros((n, 6), dtype=torch.float32, device=gpu)
        torch.cuda.synchronize()
        ctx.point_features(u, feat, br, tg)
        ctx.synchronize()
        assert torch.isnan(buf[:s]).all() and torch.isnan(buf[s + 8 * n:]).all()
        loss, grad = mlp.gradient(feat, br, tg, n=n)
        mlp.predict(feat, pr, po, n=n)
        torch.cuda.synchronize()
        out.append([a.cpu().numpy() for a in (feat, br, tg, pr, po)] + [loss, grad])
    for a, b in zip(*out):
        assert np.array_equal(a, b)
