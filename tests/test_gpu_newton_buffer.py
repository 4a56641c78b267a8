"""ipf_newton beside calls that are still pending on another stream.

Calls that take the element / node launches share one buffer of element
forces, lent to one stream at a time; the step graph of ipf_newton sums its
residual through the solver's own.  -B^T (w sigma) of a fixed vector (no state
is read) is left pending many times over on a first stream while a Newton solve
runs on a second: both are bit for bit what each gives alone (every sum has a
fixed order).
"""
import numpy as np
import pytest

import intpointsfem_amd as ipf
from intpointsfem_amd import wellbore as wb

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh", [(24, 20, 2, 1.1), (9, 11, 3, 1.2)], ids=str)
def test_newton_leaves_pending_calls_of_another_stream_alone(gpu, mesh):
    import torch
    m = wb.make_mesh(mesh)
    m.set_normal_stress(wb.normal_stress(4), 0.0)
    sm = ipf.StructMatrix(m, device=0)
    ctx = sm.context()
    ctx.set_dirichlet_mask(m.dirichlet_mask())
    state = ctx.get_state()
    neq, npts = m.info()["neq"], sm.sizes()["npts"]
    ws = torch.as_tensor(np.random.default_rng(7).standard_normal(3 * npts), device=gpu)
    first, second = torch.cuda.Stream(), torch.cuda.Stream()

    def solve(x):
        ctx.set_stream(second.cuda_stream)
        return ctx.newton(x, rtol=1e-12, maxit=3, cg_rtol=1e-10, cg_maxit=400)

    def outputs(n):
        out = [torch.full((neq,), float("nan"), dtype=torch.float64, device=gpu) for _ in range(n)]
        torch.cuda.synchronize()
        return out

    ctx.set_stream(first.cuda_stream)
    (want,) = outputs(1)
    ctx.multiply_transpose(ws, want)
    ctx.synchronize()
    x_want = torch.zeros(neq, dtype=torch.float64, device=gpu)
    torch.cuda.synchronize()
    s_want = solve(x_want)
    assert s_want["iterations"] == 3
    for spin in (0, 200_000):
        outs = outputs(300)
        x = torch.zeros(neq, dtype=torch.float64, device=gpu)
        torch.cuda.synchronize()
        ctx.set_state(state[0], state[1])  # the solve before committed its state
        ctx.set_stream(first.cuda_stream)
        with torch.cuda.stream(first):
            torch.cuda._sleep(spin)  # clock cycles: the pending calls start while the solve runs
        for out in outs:
            ctx.multiply_transpose(ws, out)
        s = solve(x)
        torch.cuda.synchronize()
        ctx.set_stream(first.cuda_stream)
        ctx.synchronize()
        assert torch.equal(x, x_want) and s == s_want
        assert all(torch.equal(out, want) for out in outs)
    ctx.set_stream(None)
