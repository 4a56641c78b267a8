"""The element / node launches against the launch per color.

Bars: residual, residual with tangent and tangent product bit-identical (the
node launch sums in color order), on meshes from one element up, every order, uneven batches with
several materials and triangles next to quadrilaterals; a CG solution's own
residual ||b - K x|| <= 10 rtol ||b|| (the recurrence's residual is <= rtol
||b||; the true one may drift from it by rounding).  A second stream keeps the
launch per color until the first one has been waited for: that is how the
tests reach it.
"""
import os

import numpy as np
import pytest

import intpointsfem_amd as ipf
from intpointsfem_amd import batch as ipf_batch
from intpointsfem_amd import wellbore as wb

pytestmark = pytest.mark.gpu
MIXED = os.path.join(os.path.dirname(__file__), "golden", "gmsh", "wellbore_mix.msh")


def both_ways(gpu, ctx, neq, call):
    """call(out) on the context's first stream, then on a second one."""
    import torch
    outs = []
    for stream in (None, torch.cuda.Stream()):
        ctx.set_stream(None if stream is None else stream.cuda_stream)
        out = torch.full((neq,), float("nan"), dtype=torch.float64, device=gpu)
        torch.cuda.synchronize()
        call(out)
        torch.cuda.synchronize()
        outs.append(out.cpu().numpy())
    ctx.synchronize()
    ctx.set_stream(None)
    ctx.synchronize()
    return outs


def compare(gpu, ctx, u, v):
    import torch
    neq = len(u)
    du = torch.as_tensor(u, dtype=torch.float64, device=gpu)
    dv = torch.as_tensor(v, dtype=torch.float64, device=gpu)
    for mode in ("exact", "certified-elastic"):
        ctx.set_residual_mode(mode)
        a, b = both_ways(gpu, ctx, neq, lambda out: ctx.residual(du, out))
        assert np.isfinite(a).all() and np.array_equal(a, b), mode
    kv = []

    def tangent(out):
        y = torch.zeros_like(out)
        ctx.residual_tangent(du, out)
        ctx.tangent_apply(dv, y)
        kv.append(y)
    r, s = both_ways(gpu, ctx, neq, tangent)
    assert np.array_equal(r, s) and torch.equal(kv[0], kv[1])
    # committing, the residual with tangent leaves the state the residual leaves
    before, states = ctx.get_state(), []
    for call in (ctx.residual, ctx.residual_tangent):
        ctx.set_state(before[0], before[1])
        ctx.set_update_mem(True)
        call(du, torch.zeros_like(du))
        ctx.set_update_mem(False)
        states.append(ctx.get_state())
    assert all(np.array_equal(x, y) for x, y in zip(*states))
    ctx.set_state(before[0], before[1])
    for fmt in ("geometry-fp64", "geometry-fp32"):
        ctx.set_b_format("geometry-fp64", fmt)
        a, b = both_ways(gpu, ctx, neq, lambda out: ctx.tangent_apply(dv, out))
        assert np.isfinite(a).all() and np.array_equal(a, b), fmt


@pytest.mark.parametrize("mesh", [(1, 1, 1, 1.0), (1, 1, 3, 1.0), (2, 1, 2, 1.1), (7, 3, 2, 1.2), (16, 16, 1, 1.1),
                                  (15, 14, 2, 1.1), (5, 9, 3, 1.2)], ids=str)
def test_same_bits_as_the_launch_per_color(gpu, mesh):
    m = wb.make_mesh(mesh)
    sm = ipf.StructMatrix(m, device=0)
    u = wb.lame_displacement(m.nodes(), wb.normal_stress(10), scale=3.0)
    compare(gpu, sm.context(), u, np.random.default_rng(1).standard_normal(len(u)))


def test_same_bits_on_a_batch(gpu):
    rows = [dict(N=n, p=p, phi_deg=30.0, cohesion=c, E=5000.0, nu=0.2, pw_final=-19.5)
            for n, p, c in ((5, 1, 10.0), (9, 2, 3.0), (4, 3, 7.0), (6, 2, 10.0), (3, 1, 2.0))]
    meshes = [ipf_batch.instance_mesh(r) for r in rows]
    B = ipf_batch.Batch(meshes, device=0)
    u = np.concatenate([wb.lame_displacement(m.nodes(), wb.normal_stress(10), scale=2.0) for m in meshes])
    compare(gpu, B.ctx, u, np.random.default_rng(2).standard_normal(len(u)))


@pytest.mark.parametrize("p", [1, 2, 3])
def test_same_bits_on_triangles_and_quadrilaterals(gpu, p):
    m = ipf.CompMesh.from_gmsh(MIXED, p)
    m.set_material(wb.E, wb.NU, wb.COHESION, wb.PHI, wb.PSI)
    m.set_normal_stress(wb.normal_stress(10), 0.0)
    sm = ipf.StructMatrix(m, device=0)
    xy = m.nodes()
    u = wb.lame_displacement(xy, wb.normal_stress(10), scale=2.0, r_out=float(np.hypot(*xy.T).max()))
    compare(gpu, sm.context(), u, np.random.default_rng(3).standard_normal(len(u)))


@pytest.mark.parametrize("mesh", [(1, 1, 1, 1.0), (2, 3, 1, 1.1), (20, 13, 2, 1.1), (40, 40, 2, 1.1), (9, 11, 3, 1.2),
                                  (120, 100, 1, 1.02)], ids=str)
def test_cg_solution(gpu, mesh):
    import torch
    m = wb.make_mesh(mesh)
    sm = ipf.StructMatrix(m, device=0)
    ctx = sm.context()
    mask = m.dirichlet_mask()
    ctx.set_dirichlet_mask(mask)
    u = torch.as_tensor(wb.lame_displacement(m.nodes(), wb.normal_stress(10)), dtype=torch.float64, device=gpu)
    r, x, y = torch.zeros_like(u), torch.zeros_like(u), torch.zeros_like(u)
    ctx.residual_tangent(u, r)
    b = np.where(mask, 0.0, np.random.default_rng(4).standard_normal(len(mask)))
    db = torch.as_tensor(b, dtype=torch.float64, device=gpu)
    rtol = 1e-10
    it, rel = ctx.cg_solve(db, x, rtol=rtol, maxit=20000)
    assert rel <= rtol and it < 20000
    ctx.tangent_apply(x, y)
    ctx.synchronize()
    res = np.where(mask, 0.0, b - y.cpu().numpy())
    assert np.linalg.norm(res) <= 10 * rtol * np.linalg.norm(b)


@pytest.mark.parametrize("mesh", [(1, 1, 1, 1.0), (7, 9, 1, 1.2), (1, 1, 2, 1.0), (5, 6, 2, 1.2), (4, 3, 3, 1.3)],
                         ids=str)
def test_stored_blocks_and_corners_agree(gpu, mesh):
    """Every element launch from the stored compact values and from the
    corners (bit-identical values, so bit-identical results), and the strains
    and forces against numpy's dense blocks (1e-14 of the terms' sum per
    column, a few columns)."""
    import torch
    m = wb.make_mesh(mesh)
    sm = ipf.StructMatrix(m, device=0)
    b, ix, s, d = sm.export_blocks(), sm.export_indexes(), sm.sizes(), m.material()
    stored = ipf.DeviceContext(device=0)
    stored.transfer_data(b["row_sizes"], b["col_sizes"], b["matrix_position"], b["row_first"], b["col_first"],
                         b["storage"], ix["dof_indexes"], ix["color_indexes"], s["ncolor"], s["neq"], ix["weight"])
    stored.set_material(d["lambda"], d["mu"], d["phi"], d["psi"], d["cohesion"])
    stored.set_rhs_linear(ix["rhs_linear"])
    u = wb.lame_displacement(m.nodes(), wb.normal_stress(10), scale=4.0)
    du = torch.as_tensor(u, dtype=torch.float64, device=gpu)
    n, neq = s["npts"], s["neq"]

    def zeros(k, t=torch.float64):
        return torch.full((k,), 7, dtype=t, device=gpu)
    out = []
    for ctx in (sm.context(), stored):
        r, rt, y, f = (zeros(neq) for _ in range(4))
        e, w, wd, w2 = zeros(3 * n), zeros(3 * n), zeros(9 * n), zeros(3 * n)
        feat, br, tg = zeros(8 * n, torch.float32), zeros(n, torch.int32), zeros(n, torch.float32)
        torch.cuda.synchronize()
        ctx.residual(du, r)
        ctx.residual_tangent(du, rt)
        ctx.tangent_apply(du, y)
        ctx.multiply(du, e)
        ctx.compute_sigma(e, w)
        ctx.compute_sigma_dep(e, w2, wd)
        ctx.multiply_transpose(w, f)
        ctx.point_features(du, feat, br, tg)
        ctx.synchronize()
        out.append([t.cpu().numpy() for t in (r, rt, y, e, w, w2, wd, f, feat, br, tg)])
    for x, z in zip(*out):
        assert np.isfinite(x).all() and np.array_equal(x, z)
    r, rt, y, e, w, w2, wd, f, *_ = out[0]
    assert np.array_equal(r, rt) and np.array_equal(w, w2)
    nb, C = s["nblocks"], int(b["col_sizes"][0])
    B = b["storage"].reshape(nb, -1, C)
    dof = np.asarray(ix["dof_indexes"]).reshape(nb, C)
    bound = 1e-14 * C
    ref, size = (B * u[dof][:, None, :]).sum(-1), (np.abs(B) * np.abs(u[dof])[:, None, :]).sum(-1)
    assert (np.abs(e.reshape(ref.shape) - ref) <= bound * size).all()
    t = B * w.reshape(nb, -1)[:, :, None]
    ref, size = np.zeros(neq), np.zeros(neq)
    np.add.at(ref, dof, -t.sum(1))
    np.add.at(size, dof, np.abs(t).sum(1))
    assert (np.abs(f - ref) <= 1e-14 * B.shape[1] * size).all()
