"""Strains of displacements and forces of stresses that hold infinite or NaN
values: the oracle's products, in which a block's zero times such a value is
NaN -- from the corners, from stored blocks, and by the launches per color (a
second stream).  Strains bit for bit; forces NaN and infinite in the same
places, the others within 1e-12 of the largest (order of the colors)."""
import numpy as np
import pytest

import intpointsfem_amd as ipf
from intpointsfem_amd import wellbore as wb
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("mesh", [(9, 7, 1, 1.1), (9, 7, 2, 1.1), (7, 5, 3, 1.1)], ids=str)
def test_strains_and_forces(gpu, mesh, value):
    import torch
    m = wb.make_mesh(mesh)
    sm = ipf.StructMatrix(m, device=0)
    b, ix, s = sm.export_blocks(), sm.export_indexes(), sm.sizes()
    stored = ipf.DeviceContext(device=0)
    stored.transfer_data(b["row_sizes"], b["col_sizes"], b["matrix_position"], b["row_first"], b["col_first"],
                         b["storage"], ix["dof_indexes"], ix["color_indexes"], s["ncolor"], s["neq"], ix["weight"])
    B = O.Blocks(b["row_sizes"], b["col_sizes"], b["matrix_position"], b["row_first"], b["col_first"], b["storage"])
    rng = np.random.default_rng(4)
    neq, npts = s["neq"], s["npts"]
    for part in range(3):  # x (xx), y (yy), both (xx and yy of opposite sign)
        u = rng.standard_normal(neq) * 1e-3
        nodes = rng.choice(neq // 2, max(1, neq // 60), replace=False)
        ws = rng.standard_normal((npts, 3))
        points = rng.choice(npts, max(1, npts // 60), replace=False)
        if part != 1:
            u[2 * nodes], ws[points, 0] = value, value
        if part != 0:
            u[2 * nodes + 1], ws[points, 2] = -value, -value
        with np.errstate(all="ignore"):
            e_o = O.multiply(B, ix["dof_indexes"], u)
            f_o = O.multiply_transpose(B, ix["color_indexes"], s["ncolor"], neq, ws.reshape(-1))
        du, dw = (torch.as_tensor(a.reshape(-1), dtype=torch.float64, device=gpu) for a in (u, ws))
        for ctx in (sm.context(), stored):
            for stream in (None, torch.cuda.Stream()):
                ctx.set_stream(None if stream is None else stream.cuda_stream)
                e = torch.zeros(3 * npts, dtype=torch.float64, device=gpu)
                f = torch.zeros(neq, dtype=torch.float64, device=gpu)
                torch.cuda.synchronize()
                ctx.multiply(du, e)
                ctx.multiply_transpose(dw, f)
                torch.cuda.synchronize()
                assert np.array_equal(e.cpu().numpy(), e_o, equal_nan=True)
                f, fin = f.cpu().numpy(), np.isfinite(f_o)
                assert np.array_equal(f[~fin], f_o[~fin], equal_nan=True)
                assert np.abs(f[fin] - f_o[fin]).max() <= 1e-12 * np.abs(f_o[fin]).max()
            ctx.synchronize()
            ctx.set_stream(None)
            ctx.synchronize()
