"""The stable counting sort of branch ids (ipf_branch_order and its
allocation-free form) against numpy's stable argsort: from 4 points to more
than one round of 1,024 keys per block (1,048,576 points), ids below, inside
and above the range (out-of-range ids sort last), and a single id throughout.
Integers: equality.
"""
import numpy as np
import pytest

import intpointsfem_amd as ipf
from intpointsfem_amd import wellbore as wb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh", [(1, 1, 1), (3, 3, 2), (16, 4, 3), (16, 16, 1), (11, 11, 2), (16, 16, 3), (137, 50, 2),
                                  (512, 512, 1), (350, 347, 2)], ids=str)
def test_stable_order(gpu, mesh):
    import torch
    m = wb.make_mesh((*mesh, 1.0))
    sm = ipf.StructMatrix(m, device=0)
    ctx = sm.context()
    n = ctx.info()["npts"]
    rng = np.random.default_rng(n)
    for keys in (rng.integers(-2, 8, n), np.full(n, 2), np.full(n, -3), np.sort(rng.integers(0, 5, n))[::-1],
                 np.where(rng.random(n) < 0.999, 0, 3)):
        k = torch.as_tensor(keys.astype(np.int32).copy(), device=gpu)
        ref = np.argsort(np.where((keys < 0) | (keys > 4), 4, keys), kind="stable")
        for call in (ctx.branch_order, ctx.branch_order_noalloc):
            o = torch.full((n,), -1, dtype=torch.int32, device=gpu)
            call(k, o)
            ctx.synchronize()
            assert np.array_equal(o.cpu().numpy(), ref)
