"""Which launches a call takes (ipf_launch_routes), on meshes of 5 and 8 colors
of triangles next to quadrilaterals -- the elements of the first colors of
gmsh/wellbore_mix.msh, which has 9; the rest of its nodes then belong to no
element -- set up from the corners and from stored blocks.

Bars: a call on the context's first stream takes the element / node launches,
the same call on a second one (the first not waited for by ipf_synchronize) the
launches per color, and both give the same bits; strains and stresses are the
oracle's bit for bit; a CG solution's own residual ||b - K x|| <= 10 rtol ||b||.
ipf_autotune times the launches that the calls take.
"""
import os

import numpy as np
import pytest

import intpointsfem_amd as ipf
from intpointsfem_amd import wellbore as wb
from oracle import oracle as O

pytestmark = pytest.mark.gpu
MIXED = os.path.join(os.path.dirname(__file__), "golden", "gmsh", "wellbore_mix.msh")


class Part:
    """The elements of the first ncolor colors of the mixed mesh at order p."""

    def __init__(self, p, ncolor):
        m = ipf.CompMesh.from_gmsh(MIXED, p)
        m.set_material(wb.E, wb.NU, wb.COHESION, wb.PHI, wb.PSI)
        m.set_normal_stress(wb.normal_stress(10), 0.0)
        sm = ipf.StructMatrix(m, device=-1)
        b, ix = sm.export_blocks(), sm.export_indexes()
        self.mesh, self.neq, self.ncolor = m, m.info()["neq"], ncolor
        first = b["col_first"][:-1]
        color = ix["color_indexes"][first] // self.neq
        assert color.max() >= ncolor
        keep = np.flatnonzero(color < ncolor)
        self.rows, self.cols = b["row_sizes"][keep], b["col_sizes"][keep]

        def take(a, start, count):
            return np.concatenate([a[start[e]:start[e] + n] for e, n in zip(keep, count)])

        def offsets(n, t):
            return np.concatenate([[0], np.cumsum(n)]).astype(t)
        self.storage = take(b["storage"], b["matrix_position"], self.rows.astype(np.int64) * self.cols)
        self.dof = take(ix["dof_indexes"], b["col_first"], self.cols)
        self.colors = take(ix["color_indexes"], b["col_first"], self.cols)
        self.weight = take(ix["weight"], b["row_first"] // 3, self.rows // 3)
        self.position = offsets(self.rows.astype(np.int64) * self.cols, np.int64)
        self.row_first, self.col_first = offsets(self.rows, np.int32), offsets(self.cols, np.int32)
        self.rhs = ix["rhs_linear"]
        self.types, self.corners = m.element_types()[keep].astype(np.int32), m.corners()[keep]
        assert set(self.types) == {0, 1}
        self.blocks = O.Blocks(self.rows, self.cols, self.position, self.row_first, self.col_first, self.storage)
        # no element on a DoF: fixed, like the mesh's symmetry DoFs and, so that
        # no part of what is left can move freely, half of the others
        fixed = m.dirichlet_mask() | (np.random.default_rng(9).random(self.neq) < 0.5)
        fixed[np.setdiff1d(np.arange(self.neq), self.dof)] = True
        self.fixed = fixed

    def context(self, source):
        ctx = ipf.DeviceContext(device=0)
        if source == "corners":
            sizes, tabs = zip(*(self.mesh.shape_table(t) for t in (0, 1)))
            ctx.transfer_geometry(sizes, np.concatenate(tabs), self.types, self.corners, self.dof, self.colors,
                                  self.ncolor, self.neq)
        else:
            ctx.transfer_data(self.rows, self.cols, self.position, self.row_first, self.col_first, self.storage,
                              self.dof, self.colors, self.ncolor, self.neq, self.weight)
        d = self.mesh.material()
        ctx.set_material(d["lambda"], d["mu"], d["phi"], d["psi"], d["cohesion"])
        ctx.set_rhs_linear(self.rhs)
        ctx.set_dirichlet_mask(self.fixed)
        return ctx


def both_ways(gpu, ctx, neq, call, calls=1):
    """call(out) on the context's first stream, then on a second one, each by
    its own launches."""
    import torch
    outs = []
    for k, stream in enumerate((None, torch.cuda.Stream())):
        ctx.set_stream(None if stream is None else stream.cuda_stream)
        out = torch.full((neq,), float("nan"), dtype=torch.float64, device=gpu)
        torch.cuda.synchronize()
        before = ctx.launch_routes()
        call(out)
        after = ctx.launch_routes()
        torch.cuda.synchronize()
        taken = (after[0] - before[0], after[1] - before[1])
        assert taken == ((calls, 0) if k == 0 else (0, calls)), taken
        outs.append(out.cpu().numpy())
    ctx.synchronize()
    ctx.set_stream(None)
    ctx.synchronize()
    return outs


@pytest.mark.parametrize("source", ["corners", "stored"])
@pytest.mark.parametrize("p,ncolor", [(1, 5), (1, 8), (2, 5), (2, 8), (3, 5), (3, 8)])
def test_triangles_and_quadrilaterals(gpu, p, ncolor, source):
    import torch
    part = Part(p, ncolor)
    ctx, neq, n3 = part.context(source), part.neq, int(part.rows.sum())
    xy = part.mesh.nodes()
    u = wb.lame_displacement(xy, wb.normal_stress(10), scale=2.0, r_out=float(np.hypot(*xy.T).max()))
    rng = np.random.default_rng(3)

    def dev(a):
        return torch.as_tensor(a, dtype=torch.float64, device=gpu)

    def new(n):
        return torch.full((n,), float("nan"), dtype=torch.float64, device=gpu)
    du, dv, dw = dev(u), dev(rng.standard_normal(neq)), dev(rng.standard_normal(n3))
    for mode in ("exact", "certified-elastic"):
        ctx.set_residual_mode(mode)
        a, b = both_ways(gpu, ctx, neq, lambda out: ctx.residual(du, out))
        assert np.isfinite(a).all() and np.array_equal(a, b), mode
    kv = []

    def tangent(out):
        y = new(neq)
        torch.cuda.synchronize()
        ctx.residual_tangent(du, out)
        ctx.tangent_apply(dv, y)
        kv.append(y)
    r, s = both_ways(gpu, ctx, neq, tangent, calls=2)
    assert np.isfinite(r).all() and np.array_equal(r, s) and torch.equal(kv[0], kv[1])
    a, b = both_ways(gpu, ctx, neq, lambda out: ctx.multiply_transpose(dw, out))
    assert np.isfinite(a).all() and np.array_equal(a, b)
    if source == "corners":
        ctx.set_b_format("geometry-fp32", "geometry-fp32")
        for call in (lambda out: ctx.residual(du, out), lambda out: ctx.tangent_apply(dv, out)):
            a, b = both_ways(gpu, ctx, neq, call)
            assert np.isfinite(a).all() and np.array_equal(a, b)
        ctx.set_b_format("geometry-fp64", "geometry-fp64")
    # strains, stresses and tangents: the oracle's bits
    d = part.mesh.material()
    eps_o = O.multiply(part.blocks, part.dof, u)
    ws_o, wd_o, *_ = O.compute_sigma(eps_o, part.weight, d["lambda"], d["mu"], d["phi"], d["psi"], d["cohesion"],
                                     dep=True)
    e, ws, wd = new(n3), new(n3), new(3 * n3)
    torch.cuda.synchronize()
    ctx.multiply(du, e)
    ctx.compute_sigma_dep(e, ws, wd)
    ctx.synchronize()
    for got, want in ((e, eps_o), (ws, ws_o), (wd, wd_o)):
        assert np.array_equal(got.cpu().numpy(), want)
    # CG, with the elastic tangent (that of u may be singular)
    b = np.where(part.fixed, 0.0, rng.standard_normal(neq))
    x, y, db, rtol = dev(np.zeros(neq)), new(neq), dev(b), 1e-10
    du.mul_(0.05)
    torch.cuda.synchronize()
    ctx.residual_tangent(du, y)
    it, rel = ctx.cg_solve(db, x, rtol=rtol, maxit=20000)
    assert rel <= rtol and 0 < it < 20000
    ctx.tangent_apply(x, y)
    ctx.synchronize()
    res = np.where(part.fixed, 0.0, b - y.cpu().numpy())
    assert np.linalg.norm(res) <= 10 * rtol * np.linalg.norm(b)


@pytest.mark.parametrize("mesh", [(12, 10, 2, 1.1), (7, 5, 3, 1.1)], ids=str)
def test_autotune_times_the_launches_of_the_calls(gpu, mesh):
    import torch
    m = wb.make_mesh(mesh)
    sm = ipf.StructMatrix(m, device=0)
    ctx = sm.context()
    u = torch.as_tensor(wb.lame_displacement(m.nodes(), wb.normal_stress(10)), dtype=torch.float64, device=gpu)
    r = torch.zeros_like(u)
    torch.cuda.synchronize()
    ctx.residual_tangent(u, r)
    reps = 10
    before = ctx.launch_routes()
    t = ctx.autotune(u, reps=reps, allow_fp32=True)
    after = ctx.launch_routes()
    # element / node launches: compact and geometric FP64 (and FP32 geometric
    # for the product); the other forms have launches per color only
    split = sum(f in ("compact-fp64", "geometry-fp64") for f in t["residual"])
    split += sum(f in ("compact-fp64", "geometry-fp64", "geometry-fp32") for f in t["tangent"])
    per_color = len(t["residual"]) + len(t["tangent"]) - split
    assert split == 5 and per_color == 4
    assert (after[0] - before[0], after[1] - before[1]) == (split * (reps + 2), per_color * (reps + 2))
    # two launches against four: the choice stays with the forms that have them
    assert t["selected"][0] in ("compact-fp64", "geometry-fp64")
