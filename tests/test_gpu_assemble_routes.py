"""The routes of the CSR assembly against each other and the oracle's element
matrices: B from the corners, B from stored blocks with the 2D elasticity
pattern, and general stored blocks (the pattern broken by one entry); a
pattern every entry of which has an element (no clear of Kg) and one with
entries of no element.

Bars: geometric and stored pattern blocks bit-identical to each other and to
the oracle's element matrices summed color by color; general blocks
bit-identical to the oracle's of the same blocks; entries of no element
exactly 0; Kg NaN-filled before every call.
"""
import numpy as np
import pytest

import intpointsfem_amd as ipf
from intpointsfem_amd import wellbore as wb
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def assemble(gpu, ctx, u, nnz):
    import torch
    kg = torch.full((nnz,), float("nan"), dtype=torch.float64, device=gpu)
    du = torch.as_tensor(u, dtype=torch.float64, device=gpu)
    ctx.assemble_tangent(du, torch.zeros_like(du), kg)
    ctx.synchronize()
    return kg.cpu().numpy()


def context(m, sm, b, ix, pat, nnz):
    s, d = sm.sizes(), m.material()
    ctx = ipf.DeviceContext(device=0)
    ctx.transfer_data(b["row_sizes"], b["col_sizes"], b["matrix_position"], b["row_first"], b["col_first"],
                      b["storage"], ix["dof_indexes"], ix["color_indexes"], s["ncolor"], s["neq"], ix["weight"])
    ctx.set_material(d["lambda"], d["mu"], d["phi"], d["psi"], d["cohesion"])
    ctx.set_rhs_linear(ix["rhs_linear"])
    ctx.set_tangent_pattern(ix["el_color_index"], pat["color_l_sequence"], nnz)
    return ctx


def oracle_kg(m, b, ix, pat, u, nnz):
    B = O.Blocks(b["row_sizes"], b["col_sizes"], b["matrix_position"], b["row_first"], b["col_first"], b["storage"])
    d = m.material()
    wd = O.compute_sigma(O.multiply(B, ix["dof_indexes"], u), ix["weight"], d["lambda"], d["mu"], d["phi"], d["psi"],
                         d["cohesion"], dep=True)[1]
    kc = O.element_tangents(B, wd, ix["el_color_index"])
    kg, fl, cl = np.zeros(nnz), pat["first_color_l_index"], pat["color_l_sequence"]
    for c in range(len(fl) - 1):
        idx = cl[fl[c]:fl[c + 1]]
        kg[idx] = kg[idx] + kc[fl[c]:fl[c + 1]]
    return kg


@pytest.mark.parametrize("mesh", [(1, 1, 1, 1.0), (5, 7, 1, 1.2), (13, 3, 1, 1.1), (1, 2, 2, 1.1), (9, 8, 2, 1.1),
                                  (1, 1, 3, 1.0), (5, 4, 3, 1.3)], ids=str)
def test_routes(gpu, mesh):
    m = wb.make_mesh(mesh)
    sm = ipf.StructMatrix(m, device=0)
    b, ix, pat = sm.export_blocks(), sm.export_indexes(), sm.tangent_pattern()
    nnz, extra = len(pat["ja"]), 5
    u = wb.lame_displacement(m.nodes(), wb.normal_stress(10), scale=6.0)
    ref = oracle_kg(m, b, ix, pat, u, nnz)
    geo = sm.context()
    assert geo.build_tangent_pattern() == nnz
    np.testing.assert_array_equal(assemble(gpu, geo, u, nnz), ref)
    np.testing.assert_array_equal(assemble(gpu, context(m, sm, b, ix, pat, nnz), u, nnz), ref)
    kg = assemble(gpu, context(m, sm, b, ix, pat, nnz + extra), u, nnz + extra)
    np.testing.assert_array_equal(kg[:nnz], ref)
    assert (kg[nnz:] == 0.0).all()
    g = dict(b, storage=b["storage"].copy())
    g["storage"][1] = 1e-3 * np.abs(g["storage"]).max()  # row xx, a y column: 0 in the pattern
    np.testing.assert_array_equal(assemble(gpu, context(m, sm, g, ix, pat, nnz), u, nnz),
                                  oracle_kg(m, g, ix, pat, u, nnz))
