"""The work a user of intpointsfem_amd has it do, one timed case each.

The sizes are the framework's own configurations (40x40 and 800x800 wellbore
meshes, orders 1 to 3, batches of uneven instances, the branch predictor's
minibatch) and generic ones between them.  A case's inputs come from a seed:
the wellbore's linear-elastic displacement at a drawn load level with a
smooth perturbation (what a Newton iterate looks like), a committed plastic
state, and a wall load.  ``exact`` evaluates the same problem in 64 bits with
torch alone: closed-form Mohr-Coulomb return, Lagrange quadrilaterals on the
structured quarter annulus.

Kinds:
  residual  r = f - sum B^T w sigma(B u), the call of every Newton residual,
            time step check and line search
  batch     the same over many uneven instances in one context
  tangent   residual with consistent tangent, then one product K v (the head
            of a Krylov solve)
  assemble  residual and the tangent's CSR values (for a direct solver)
  apply     one product K v with a tangent at hand (each Krylov iteration)
  cg        one linear solve
  newton    one load step from the virgin state, state read back
  steps     strain, stress and force as the three separate calls
  train     gradient of the branch predictor on one batch of pairs
  infer     features, predicted branch and visiting order of every point
"""
import math

import numpy as np
import torch

import intpointsfem_amd as ipf
from intpointsfem_amd import batch as ipf_batch
from intpointsfem_amd import wellbore as wb

MAX_POINTS = 10_240_000  # 800 x 800 cells of order 3


def listed():
    return [
        # the reference's own verification mesh: 1,600 elements, every call a few launches of a few waves
        {"name": "residual-40x40-q2", "kind": "residual", "nr": 40, "nt": 40, "p": 2, "mode": "exact"},
        # the headline workload: 5.76 M points in a plastic state
        {"name": "residual-800x800-q2", "kind": "residual", "nr": 800, "nt": 800, "p": 2, "mode": "exact"},
        # the largest mesh configuration: 10.24 M points
        {"name": "residual-800x800-q3", "kind": "residual", "nr": 800, "nt": 800, "p": 3, "mode": "exact"},
        # a parameter study: uneven meshes, orders and materials in one context, the certified fast path
        {"name": "batch-16-certified", "kind": "batch", "n": 16, "lo": 50, "hi": 200, "table": 0,
         "mode": "certified-elastic"},
        # residual and tangent of one Newton iterate, and the first Krylov product
        {"name": "tangent-400x400-q2", "kind": "tangent", "nr": 400, "nt": 400, "p": 2},
        # the CSR stiffness a direct solver factorises
        {"name": "assemble-201x150-q2", "kind": "assemble", "nr": 201, "nt": 150, "p": 2},
        # the Krylov product of the headline mesh, thousands of them per load step
        {"name": "apply-800x800-q2", "kind": "apply", "nr": 800, "nt": 800, "p": 2, "format": "geometry-fp64"},
        # one linear solve of an ordinary mesh
        {"name": "cg-100x100-q2", "kind": "cg", "nr": 100, "nt": 100, "p": 2},
        # one whole load step of the verification mesh
        {"name": "newton-40x40-q2", "kind": "newton", "nr": 40, "nt": 40, "p": 2},
        # a caller of the reference's three separate steps, odd sizes
        {"name": "steps-317x251-q2", "kind": "steps", "nr": 317, "nt": 251, "p": 2},
        # one minibatch of the branch predictor's training
        {"name": "train-4096", "kind": "train", "n": 4096},
        # the predictor over an ordinary mesh, end to end
        {"name": "infer-400x400-q2", "kind": "infer", "nr": 400, "nt": 400, "p": 2},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["residual", "residual", "batch", "tangent", "assemble", "apply", "cg", "newton", "steps",
                       "train", "infer"])
    if kind == "train":
        return {"kind": kind, "n": _log(rng, 1000, 500_000)}
    if kind == "batch":
        lo = _log(rng, 20, 120)
        return {"kind": kind, "n": rng.randint(2, 24), "lo": lo, "hi": lo + _log(rng, 10, 100),
                "table": rng.randint(0, 10 ** 6), "mode": rng.choice(["exact", "certified-elastic"])}
    p = rng.choice([1, 2, 2, 3])
    # the longest side of each kind's range; whole solves stay within a second or so
    top = {"residual": 800, "apply": 800, "tangent": 500, "steps": 400, "infer": 500, "assemble": 250, "cg": 120,
           "newton": 60}[kind]
    c = {"kind": kind, "nr": _log(rng, 20, top), "nt": _log(rng, 20, top), "p": p}
    if kind == "residual":
        c["mode"] = rng.choice(["exact", "exact", "certified-elastic"])
    if kind == "apply":
        c["format"] = rng.choice(["geometry-fp64", "geometry-fp64", "geometry-fp32"])
    return c


# ------------------------------------------------------------------ sizes


def _instances(case):
    """[(nr, nt, p, E, nu, c, phi, load)] of a case: one wellbore mesh, or the batch's table."""
    if case["kind"] != "batch":
        return [(case["nr"], case["nt"], case["p"], wb.E, wb.NU, wb.COHESION, wb.PHI, wb.normal_stress(wb.NSTEPS))]
    g = np.random.Generator(np.random.PCG64(case["table"]))
    n = case["n"]
    N = g.integers(case["lo"], case["hi"], size=n, endpoint=True)
    p = g.integers(1, 3, size=n, endpoint=True)
    phi = np.radians(g.uniform(20.0, 40.0, size=n))
    c = np.exp(g.uniform(math.log(2.0), math.log(20.0), size=n))
    E = g.uniform(2000.0, 20000.0, size=n)
    nu = g.uniform(0.15, 0.3, size=n)
    load = -(g.uniform(-30.0, -15.0, size=n) - wb.SIGMA0)
    return [(int(N[i]), int(N[i]), int(p[i]), float(E[i]), float(nu[i]), float(c[i]), float(phi[i]), float(load[i]))
            for i in range(n)]


def _neq(nr, nt, p):
    return 2 * (p * nr + 1) * (p * nt + 1)


def work(case):
    """Bytes read and written once (u, f, r; 32 of plastic strain per point, 64 of corners and 4 per node index
    per element) and the operations of the formulas."""
    k = case["kind"]
    if k == "train":  # forward, and twice that backward
        return {"bytes": 40 * case["n"], "flops": 6 * (7 * 64 + 64 * 64 + 64 * 6) * case["n"]}
    by = fl = 0.0
    for nr, nt, p, *_ in _instances(case):
        ne, nsh = nr * nt, (p + 1) ** 2
        npt, neq = ne * nsh, _neq(nr, nt, p)
        geo = ne * (64 + 4 * nsh)
        prod = npt * (30 + 6 * nsh)          # the map, its inverse, the gradients
        side = npt * 8 * nsh                 # B u, or B^T s
        if k in ("residual", "batch"):
            by += 24 * neq + 32 * npt + geo
            fl += prod + 2 * side + 300 * npt
        elif k == "tangent":                 # w D written and read once more
            by += 24 * neq + 32 * npt + 2 * geo + 144 * npt + 16 * neq
            fl += 2 * prod + 4 * side + 1000 * npt
        elif k == "assemble":
            nt_e = nsh * (2 * nsh + 1)       # packed upper triangle, and its positions
            by += 24 * neq + 32 * npt + geo + 4 * ne * nt_e + 8 * _nnz(nr, nt, p)
            fl += prod + 2 * side + 1000 * npt + npt * (15 * 2 * nsh + 6 * nt_e)
        elif k == "apply":
            by += 16 * neq + (72 if case["format"] == "geometry-fp64" else 36) * npt + geo
            fl += prod + 2 * side + 15 * npt
        elif k in ("cg", "newton"):
            its = _iterations(nr, nt, p) * (1 if k == "cg" else 5)
            by += its * (96 * neq + 72 * npt + geo)
            fl += its * (prod + 2 * side + 15 * npt + 20 * neq)
        elif k == "steps":                   # strain and stress written and read
            by += 16 * neq + 32 * npt + 2 * geo + 96 * npt
            fl += 2 * prod + 2 * side + 300 * npt
        elif k == "infer":                   # features, labels, logits, branch, order
            by += 8 * neq + 40 * npt + geo + (32 + 8) * npt + 32 * npt + 28 * npt + 8 * npt
            fl += prod + side + 300 * npt + 2 * (7 * 64 + 64 * 64 + 64 * 6) * npt
    return {"bytes": by, "flops": fl}


def _nnz(nr, nt, p):
    """Upper-triangle entries of the element graph of an nr x nt grid of order p."""
    def pairs(n):  # node pairs along one direction that share a cell
        return sum(((2 * p + 1) if i % p == 0 and 0 < i < p * n else (p + 1)) for i in range(p * n + 1))
    node_pairs = pairs(nr) * pairs(nt)
    nodes = (p * nr + 1) * (p * nt + 1)
    return (4 * node_pairs + 2 * nodes) // 2


def _iterations(nr, nt, p):
    """Roughly what a conjugate gradient needs on such a mesh."""
    return 6 * p * max(nr, nt)


# ------------------------------------------------------------------ inputs


class _Grid:
    """The structured quarter annulus of nr x nt cells of order p: corners, nodes and connectivity."""

    def __init__(self, nr, nt, p):
        q = 1.1 ** (40.0 / nr)
        L = wb.R_OUT - wb.R_IN
        h0 = L / nr if q == 1.0 else L * (q - 1.0) / (q ** nr - 1.0)
        R = wb.R_IN + np.concatenate([[0.0], np.cumsum(h0 * q ** np.arange(nr))])
        R[-1] = wb.R_OUT
        th = (math.pi / 2) * np.arange(nt + 1) / nt
        c, s = np.cos(th), np.sin(th)
        c[-1], s[0] = 0.0, 0.0
        self.nr, self.nt, self.p, self.q = nr, nt, p, q
        self.grid = np.stack([np.outer(c, R), np.outer(s, R)], axis=-1)  # [nt + 1, nr + 1, 2]

    def corners(self):
        g = self.grid
        return np.stack([g[:-1, :-1], g[:-1, 1:], g[1:, 1:], g[1:, :-1]], axis=2).reshape(-1, 4, 2)

    def local(self):
        """(a, b) grid position of each local node: vertices, edge interiors, interior."""
        p = self.p
        n = [(0, 0), (p, 0), (p, p), (0, p)]
        n += [(a, 0) for a in range(1, p)] + [(p, b) for b in range(1, p)]
        n += [(a, p) for a in range(p - 1, 0, -1)] + [(0, b) for b in range(p - 1, 0, -1)]
        return n + [(a, b) for b in range(1, p) for a in range(1, p)]

    def connectivity(self):
        p, w = self.p, self.p * self.nr + 1
        j, i = np.divmod(np.arange(self.nr * self.nt), self.nr)
        return np.stack([(p * j + b) * w + p * i + a for a, b in self.local()], axis=1)

    def nodes(self):
        p, g = self.p, self.grid
        t = np.arange(p * self.nr + 1)
        i = np.minimum(t // p, self.nr - 1)
        f = ((t - p * i) / p)[None, :, None]
        e = g[:, i] * (1 - f) + g[:, i + 1] * f                # along r at every corner angle
        t = np.arange(p * self.nt + 1)
        j = np.minimum(t // p, self.nt - 1)
        f = ((t - p * j) / p)[:, None, None]
        return (e[j] * (1 - f) + e[j + 1] * f).reshape(-1, 2)

    def load(self, sigma):
        """Consistent nodal forces of the radial stress sigma on the inner arc."""
        p, f = self.p, np.zeros((self.p * self.nt + 1, 2))
        A, B = self.grid[:-1, 0], self.grid[1:, 0]             # one straight edge per cell
        t = np.stack([-(B[:, 1] - A[:, 1]), B[:, 0] - A[:, 0]], axis=1) * sigma  # stress times length times normal
        share = {1: [1 / 2, 1 / 2], 2: [1 / 6, 4 / 6, 1 / 6], 3: [1 / 8, 3 / 8, 3 / 8, 1 / 8]}[p]
        for b, s in enumerate(share):
            np.add.at(f, p * np.arange(self.nt) + b, s * t)
        out = np.zeros((p * self.nt + 1, p * self.nr + 1, 2))
        out[:, 0] = f
        return out.reshape(-1)

    def fixed(self):
        m = np.zeros((self.p * self.nt + 1, self.p * self.nr + 1, 2), dtype=bool)
        m[0, :, 1] = True
        m[-1, :, 0] = True
        return m.reshape(-1)


def _smooth(rng, xy, load, E, nu, level):
    """The thick cylinder's displacement at `level` times the load, with a smooth perturbation of a few percent."""
    u = wb.lame_displacement(xy, load, scale=level, E_=E, nu=nu)
    r = np.hypot(xy[:, 0], xy[:, 1])
    th = np.arctan2(xy[:, 1], xy[:, 0])
    f = np.ones(len(xy))
    for _ in range(3):
        f += rng.uniform(0.005, 0.02) * np.cos(rng.integers(1, 4) * 2 * th + rng.uniform(0, 6.28)) * \
            np.cos(rng.uniform(1, 6) * np.log(r / wb.R_IN) + rng.uniform(0, 6.28))
    return u * np.repeat(f, 2)


def _inputs(case, seed):
    """Grids, committed-state and trial displacements, a direction, the loads and the materials of a case."""
    rng = np.random.Generator(np.random.PCG64([seed, 7]))
    # load levels: a plastic state below a further-loaded iterate; linear solves and load steps start elastic
    commit = rng.uniform(1.8, 2.2)
    level = rng.uniform(0.9, 1.1) if case["kind"] == "cg" else rng.uniform(2.8, 3.2)
    if case["kind"] in ("cg", "newton"):
        commit = 0.0
    out = []
    for nr, nt, p, E, nu, c, phi, load in _instances(case):
        g = _Grid(nr, nt, p)
        xy = g.nodes()
        lam, mu = E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))
        out.append(dict(grid=g, u0=_smooth(rng, xy, load, E, nu, commit) if commit else None,
                        u=_smooth(rng, xy, load, E, nu, level), v=rng.standard_normal(len(xy) * 2),
                        f=g.load(load * (rng.uniform(0.4, 0.6) if case["kind"] == "newton" else 1.0)),
                        mat=(lam, mu, phi, phi, c), E=E, nu=nu, load=load))
    return out


def _pairs(n, seed):
    """n training pairs as the exact return map emits them: features, branch, increment."""
    rng = np.random.Generator(np.random.PCG64([seed, 11]))
    c = np.exp(rng.uniform(math.log(1.0), math.log(20.0), size=n))
    phi = np.radians(rng.uniform(20.0, 40.0, size=n))
    s = -np.sort(-(rng.standard_normal((n, 3)) * 2.0 - 1.0), axis=1)
    plane = s[:, 0] - s[:, 2] + (s[:, 0] + s[:, 2]) * np.sin(phi) - 2 * np.cos(phi)
    edge = (1 - np.sin(phi)) * s[:, 0] - 2 * s[:, 1] + (1 + np.sin(phi)) * s[:, 2]
    far = plane > 4.0
    br = np.where(plane <= 0, 0, np.where(far & (s.sum(1) > 4), 4, np.where(far, np.where(edge > 0, 2, 3), 1)))
    f = np.stack([s[:, 0], s[:, 1], s[:, 2], np.log(c), phi, phi, rng.exponential(0.2, n), np.zeros(n)], axis=1)
    return f.astype(np.float32), br.astype(np.int32), (0.3 * np.maximum(plane, 0)).astype(np.float32)


_LAYERS = [(7, 16, 64, 64), (64, 64, 64, 64), (64, 64, 6, 16)]  # inputs, stored inputs, outputs, stored outputs


def _weights(seed):
    """The predictor's weights: matrices and biases, and the vector set_params takes (padded rows and columns zero)."""
    rng = np.random.Generator(np.random.PCG64([seed, 13]))
    net, flat = [], []
    for i, ip, o, op in _LAYERS:
        W = np.zeros((ip, op), dtype=np.float32)
        b = np.zeros(op, dtype=np.float32)
        W[:i, :o] = rng.uniform(-1, 1, (i, o)) * math.sqrt(6.0 / (i + o))
        b[:o] = rng.uniform(-0.1, 0.1, o)
        net.append((W, b))
        flat += [W.reshape(-1), b]
    return net, np.concatenate(flat)


def _f64(a):
    return torch.as_tensor(a, dtype=torch.float64, device="cuda")


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case, k = case, case["kind"]
    if k in ("train", "infer"):
        s.mlp = ipf.MLP(device=0, seed=0)
        s.mlp.set_params(_weights(seed)[1])
    if k == "train":
        f, b, t = _pairs(case["n"], seed)
        s.feat, s.branch, s.target = (torch.as_tensor(x, device="cuda") for x in (f, b, t))
        return s
    parts = _inputs(case, seed)
    meshes = []
    for d in parts:
        g = d["grid"]
        m = ipf.CompMesh(g.nr, g.nt, g.p, wb.R_IN, wb.R_OUT, g.q)
        lam, mu, phi, psi, c = d["mat"]
        m.set_material(d["E"], d["nu"], c, phi, psi)
        m.set_normal_stress(d["load"], 0.0)
        meshes.append(m)
    if k == "batch":
        s.own = ipf_batch.Batch(meshes, device=0)
        s.ctx = s.own.ctx
    else:
        s.own = ipf.StructMatrix(meshes[0], device=0)
        s.ctx = s.own.context()
    ctx = s.ctx
    ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    s.f = np.concatenate([d["f"] for d in parts])
    ctx.set_rhs_linear(s.f)
    s.u = _f64(np.concatenate([d["u"] for d in parts]))
    s.r = torch.zeros_like(s.u)
    if parts[0]["u0"] is not None:  # the committed plastic state
        u0 = _f64(np.concatenate([d["u0"] for d in parts]))
        ctx.set_update_mem(True)
        ctx.residual(u0, s.r)
        ctx.set_update_mem(False)
        ctx.synchronize()
    npts = ctx.info()["npts"]
    if k in ("residual", "batch"):
        ctx.set_residual_mode(case["mode"])
    if k in ("tangent", "apply"):
        s.v = _f64(np.concatenate([d["v"] for d in parts]))
        s.y = torch.zeros_like(s.u)
    if k == "apply":
        ctx.set_b_format("geometry-fp64", case["format"])
        ctx.residual_tangent(s.u, s.r)
    if k == "assemble":
        s.kg = torch.zeros(ctx.build_tangent_pattern(), dtype=torch.float64, device="cuda")
    if k in ("cg", "newton"):
        ctx.set_dirichlet_mask(parts[0]["grid"].fixed())
    if k == "cg":
        ctx.residual_tangent(s.u, s.r)
        s.x = torch.zeros_like(s.u)
    if k == "newton":
        s.virgin = np.zeros(6 * npts)
    if k == "steps":
        s.strain = torch.zeros(3 * npts, dtype=torch.float64, device="cuda")
        s.wsigma = torch.zeros_like(s.strain)
    if k == "infer":
        s.mlp.set_stream(ctx.stream())  # one stream: the predictor reads what the context writes
        s.feat = torch.zeros((npts, 8), dtype=torch.float32, device="cuda")
        s.label = torch.zeros(npts, dtype=torch.int32, device="cuda")
        s.target = torch.zeros(npts, dtype=torch.float32, device="cuda")
        s.out = torch.zeros((npts, 6), dtype=torch.float32, device="cuda")
        s.branch, s.order = torch.zeros_like(s.label), torch.zeros_like(s.label)
    ctx.synchronize()
    return s


def run(s):
    k = s.case["kind"]
    if k in ("residual", "batch"):
        s.ctx.residual(s.u, s.r)
        return [s.r]
    if k == "tangent":
        s.ctx.residual_tangent(s.u, s.r)
        s.ctx.tangent_apply(s.v, s.y)
        return [s.r, s.y]
    if k == "assemble":
        s.ctx.assemble_tangent(s.u, s.r, s.kg)
        return [s.r, s.kg]
    if k == "apply":
        s.ctx.tangent_apply(s.v, s.y)
        return [s.y]
    if k == "cg":
        s.ctx.cg_solve(s.r, s.x, rtol=1e-10, maxit=20000)
        return [s.x]
    if k == "newton":
        s.ctx.set_state(s.virgin)
        s.u.zero_()
        s.ctx.newton(s.u)
        ep, alpha, *_ = s.ctx.get_state()
        return [s.u, ep, alpha]
    if k == "steps":
        s.ctx.multiply(s.u, s.strain)
        s.ctx.compute_sigma(s.strain, s.wsigma)
        s.ctx.multiply_transpose(s.wsigma, s.r)
        return [s.strain, s.wsigma, s.r]
    if k == "train":
        loss, grad = s.mlp.gradient(s.feat, s.branch, s.target)
        return [loss, grad]
    s.ctx.point_features(s.u, s.feat, s.label, s.target)
    s.mlp.predict(s.feat, branch=s.branch, out=s.out)
    s.ctx.branch_order(s.branch, s.order)
    return [s.feat, s.label, s.target, s.out, s.branch, s.order]


# ------------------------------------------------------------------ 64-bit values


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


class _Exact:
    """One mesh in 64 bits: strains, forces, stiffness."""

    def __init__(self, g, mat):
        dev = _dev()
        p, self.mat = g.p, mat
        gx, gw = np.polynomial.legendre.leggauss(p + 1)
        z = np.linspace(-1.0, 1.0, p + 1)
        basis = [np.polynomial.Polynomial.fromroots(np.delete(z, k)) / np.prod(z[k] - np.delete(z, k))
                 for k in range(p + 1)]
        L = np.array([[b(x) for b in basis] for x in gx])
        dL = np.array([[b.deriv()(x) for b in basis] for x in gx])
        loc = g.local()
        dN, xi, eta, wq = [], [], [], []
        for qi in range(p + 1):  # second direction fastest
            for qj in range(p + 1):
                dN.append([(dL[qi, a] * L[qj, b], L[qi, a] * dL[qj, b]) for a, b in loc])
                xi.append(gx[qi])
                eta.append(gx[qj])
                wq.append(gw[qi] * gw[qj])
        xi, eta = np.array(xi), np.array(eta)
        M = np.stack([np.stack([-(1 - eta), (1 - eta), 1 + eta, -(1 + eta)], 1) / 4,
                      np.stack([-(1 - xi), -(1 + xi), 1 + xi, 1 - xi], 1) / 4], axis=-1)  # [q, 4, 2]
        self.t = lambda a: torch.as_tensor(a, dtype=torch.float64, device=dev)
        self.dN, self.M, self.wq = self.t(np.array(dN)), self.t(M), self.t(wq)
        self.X = self.t(g.corners())
        self.conn = torch.as_tensor(g.connectivity(), device=dev)
        self.ne, self.nsh, self.nip = self.conn.shape[0], self.conn.shape[1], len(wq)
        self.neq = 2 * (p * g.nr + 1) * (p * g.nt + 1)
        step = max(1, 4_000_000 // (self.nip * self.nsh))
        self.cuts = [slice(a, min(a + step, self.ne)) for a in range(0, self.ne, step)]

    def geo(self, c):
        """Gradients [e, q, a, 2] and weights [e, q] of the elements of a slice."""
        J = torch.einsum("eci,qcj->eqij", self.X[c], self.M)  # dx_i / dxi_j
        det = J[..., 0, 0] * J[..., 1, 1] - J[..., 0, 1] * J[..., 1, 0]
        a, b = J[..., 1, 1] / det, -J[..., 1, 0] / det
        cc, d = -J[..., 0, 1] / det, J[..., 0, 0] / det
        dx = a[..., None] * self.dN[..., 0] + b[..., None] * self.dN[..., 1]
        dy = cc[..., None] * self.dN[..., 0] + d[..., None] * self.dN[..., 1]
        return dx, dy, self.wq * det.abs()

    def strain(self, c, u, dx, dy):
        ux, uy = u[2 * self.conn[c]], u[2 * self.conn[c] + 1]
        s = lambda d, w: (d * w[:, None, :]).sum(-1)  # noqa: E731
        return torch.stack([s(dx, ux), s(dy, ux) + s(dx, uy), s(dy, uy)], dim=-1)

    def push(self, c, s, dx, dy, y):
        """y += B^T s, s [e, q, 3]."""
        fx = (dx * s[..., 0:1] + dy * s[..., 1:2]).sum(1)
        fy = (dx * s[..., 1:2] + dy * s[..., 2:3]).sum(1)
        y.index_add_(0, (2 * self.conn[c]).reshape(-1), fx.reshape(-1))
        y.index_add_(0, (2 * self.conn[c] + 1).reshape(-1), fy.reshape(-1))

    def commit(self, u):
        """Plastic strain [ne, nip, 4] (xx, xy, yy, zz) and hardening variable after committing at u."""
        z = torch.zeros(self.ne, self.nip, 4, dtype=torch.float64, device=self.X.device)
        if u is None:
            return z, z[..., 0].clone()
        u, al = self.t(u), z[..., 0].clone()
        for c in self.cuts:
            dx, dy, _ = self.geo(c)
            e = self.strain(c, u, dx, dy)
            m = _return_map(e, z[c], self.mat)
            z[c], al[c] = m["ep"], m["dalpha"]
        return z, al

    def forces(self, u, ep, f, dep=None, keep=None):
        """r = f - sum B^T w sigma; dep (a list) collects w D, keep strain and w sigma."""
        r = self.t(f).clone()
        u = u if torch.is_tensor(u) else self.t(u)
        for c in self.cuts:
            dx, dy, w = self.geo(c)
            e = self.strain(c, u, dx, dy)
            m = _return_map(e, ep[c], self.mat, dep is not None)
            s = m["sig"] * w[..., None]
            self.push(c, -s, dx, dy, r)
            if dep is not None:
                dep.append(m["dep"] * w[..., None, None])
            if keep is not None:
                keep.append((e, s))
        return r

    def product(self, dep, v):
        y = torch.zeros(self.neq, dtype=torch.float64, device=self.X.device)
        for c, D in zip(self.cuts, dep):
            dx, dy, _ = self.geo(c)
            e = self.strain(c, v, dx, dy)
            self.push(c, (D * e[..., None, :]).sum(-1), dx, dy, y)
        return y

    def stiffness(self, dep):
        """Element matrices [ne, 2 nsh, 2 nsh]."""
        out = []
        for c, D in zip(self.cuts, dep):
            dx, dy, _ = self.geo(c)
            z = torch.zeros_like(dx)
            B = torch.stack([torch.stack([dx, z], -1).flatten(-2), torch.stack([dy, dx], -1).flatten(-2),
                             torch.stack([z, dy], -1).flatten(-2)], dim=2)  # [e, q, 3, 2 nsh]
            K = 0
            for q in range(self.nip):
                DB = D[:, q].contiguous() @ B[:, q].contiguous()
                K = K + B[:, q].transpose(1, 2).contiguous() @ DB
            out.append(K)
        return torch.cat(out)

    def solve(self, dep, b, free):
        """K x = b on the free DoFs: Jacobi-preconditioned conjugate gradient to rounding."""
        K = self.stiffness(dep)
        dof = torch.stack([2 * self.conn, 2 * self.conn + 1], -1).flatten(1)
        diag = torch.zeros_like(b).index_add_(0, dof.reshape(-1), torch.diagonal(K, dim1=1, dim2=2).reshape(-1))
        m = free / diag

        def mul(p):
            q = (K * p[dof][:, None, :]).sum(-1)
            return torch.zeros_like(p).index_add_(0, dof.reshape(-1), q.reshape(-1)) * free
        x = torch.zeros_like(b)
        for _ in range(2):  # a second solve on the residual takes out what the recurrence lost
            r = b * free - mul(x)
            z = m * r
            p, rz, d = z, r @ z, torch.zeros_like(b)
            stop = 1e-14 * (b * free).norm()
            for it in range(6000):
                q = mul(p)
                a = rz / (p @ q)
                d = d + a * p
                r = r - a * q
                if it % 20 == 0 and float(r.norm()) <= float(stop):
                    break
                z = m * r
                rz, old = r @ z, rz
                p = z + (rz / old) * p
            x = x + d
        return x


def _return_map(e, ep, mat, want_dep=False):
    """Plane-strain Mohr-Coulomb (perfect plasticity) in closed form: e [..., 3], ep [..., 4]."""
    lam, mu, phi, psi, c = mat
    K = lam + 2 * mu / 3
    sf, cf, sp = math.sin(phi), math.cos(phi), math.sin(psi)
    ex, g, ey, ez = e[..., 0] - ep[..., 0], e[..., 1] - ep[..., 1], e[..., 2] - ep[..., 2], -ep[..., 3]
    tr = lam * (ex + ey + ez)
    sx, sy, sz, sxy = tr + 2 * mu * ex, tr + 2 * mu * ey, tr + 2 * mu * ez, mu * g
    m, d = 0.5 * (sx + sy), 0.5 * (sx - sy)
    R = torch.hypot(d, sxy)
    co, si = torch.where(R > 0, d / R, torch.ones_like(R)), torch.where(R > 0, sxy / R, torch.zeros_like(R))
    ev = torch.stack([m + R, m - R, sz], -1)
    zero = torch.zeros_like(R)
    # in-plane projections (xx, xy, yy) and the zz share of each principal direction
    N = torch.stack([torch.stack([0.5 * (1 + co), 0.5 * si, 0.5 * (1 - co), zero], -1),
                     torch.stack([0.5 * (1 - co), -0.5 * si, 0.5 * (1 + co), zero], -1),
                     torch.stack([zero, zero, zero, zero + 1], -1)], dim=-2)
    ev, order = ev.sort(dim=-1, descending=True)
    N = N.gather(-2, order[..., None].expand(N.shape))
    s1, s2, s3 = ev.unbind(-1)
    f = s1 - s3 + (s1 + s3) * sf - 2 * c * cf
    up = lambda *t: torch.tensor(t, dtype=torch.float64, device=e.device)  # noqa: E731
    n13, n12, n23 = up(1 + sf, 0, sf - 1), up(1 + sf, sf - 1, 0), up(0, 1 + sf, sf - 1)
    dirs = [up(1 + sp, 0, sp - 1), up(1 + sp, sp - 1, 0), up(0, 1 + sp, sp - 1)]
    C = up(*([0.0] * 9)).reshape(3, 3) + (K - 2 * mu / 3) + 2 * mu * torch.eye(3, dtype=torch.float64, device=e.device)

    def planes(ns, fl):
        """Projection onto the planes n . s = 2 c cos(phi): stress, sum of multipliers, gradient."""
        n, fd = torch.stack(ns), torch.stack([C @ q for q in fl])
        A = torch.linalg.inv(n @ fd.T)
        gam = (ev @ n.T - 2 * c * cf) @ A.T
        return ev - gam @ fd, gam.sum(-1), torch.eye(3, dtype=torch.float64, device=e.device) - fd.T @ A @ n
    one, g1, t1 = planes([n13], dirs[:1])
    rig, g2, t2 = planes([n13, n12], dirs[:2])
    lef, g3, t3 = planes([n13, n23], [dirs[0], dirs[2]])
    inside = lambda s: ((s[..., 0] >= s[..., 1] - 1e-12) & (s[..., 1] >= s[..., 2] - 1e-12))[..., None]  # noqa: E731
    right = ((1 - sp) * s1 - 2 * s2 + (1 + sp) * s3 > 0)[..., None]
    top = c / math.tan(phi)
    apex = torch.full_like(ev, top)
    dv = (ev.mean(-1, keepdim=True) - top) / K
    el, ok1 = (f < 1e-12)[..., None], inside(one)
    ok2 = torch.where(right, inside(rig), inside(lef))

    def pick(e_, a, b, c_, d_):
        return torch.where(el, e_, torch.where(ok1, a, torch.where(ok2, torch.where(right, b, c_), d_)))
    s = pick(ev, one, rig, lef, apex)
    da = pick(zero[..., None], 2 * cf * g1[..., None], 2 * cf * g2[..., None], 2 * cf * g3[..., None],
              cf / sp * dv)[..., 0]
    sig = (s[..., None] * N).sum(-2)  # xx, xy, yy, zz
    t = sig[..., 0] + sig[..., 2] + sig[..., 3]
    iso = lam / (2 * mu * (3 * lam + 2 * mu)) * t
    es = sig / (2 * mu)
    tot = torch.stack([e[..., 0], e[..., 1], e[..., 2], zero], -1)
    new = tot - torch.stack([es[..., 0] - iso, 2 * es[..., 1], es[..., 2] - iso, es[..., 3] - iso], -1)
    out = {"sig": sig[..., :3], "ep": new, "dalpha": da, "ev": ev,
           "branch": pick(0 * zero[..., None], 1 + 0 * zero[..., None], 2 + 0 * zero[..., None],
                          3 + 0 * zero[..., None], 4 + 0 * zero[..., None])[..., 0]}
    if want_dep:
        eye = torch.eye(3, dtype=torch.float64, device=e.device)
        w = lambda T: T.expand(*ev.shape, 3)  # noqa: E731
        el4, k1, k2, rg = el[..., None], ok1[..., None], ok2[..., None], right[..., None]
        G = torch.where(el4, w(eye), torch.where(k1, w(t1), torch.where(k2, torch.where(rg, w(t2), w(t3)),
                                                                       w(0 * eye))))
        P = N[..., :3]                                              # rows: sigma components of each direction
        Q = 2 * mu * P + lam * up(1.0, 0.0, 1.0)                    # trial principal stress per strain component
        # the shear part rotates the principal axes at the elastic modulus (the framework's trial-stress rule)
        S = torch.stack([-si, co, si], -1)
        out["dep"] = P.transpose(-1, -2) @ G @ Q + mu * S[..., :, None] * S[..., None, :]
    return out


def _mlp64(net, feat):
    h = feat[:, :7]
    for i, (W, b) in enumerate(net):
        h = h @ W + b
        if i < 2:
            h = torch.relu(h)
    return h


def exact(case, seed):
    k = case["kind"]
    t = lambda a: torch.as_tensor(a, dtype=torch.float64, device=_dev())  # noqa: E731
    if k in ("train", "infer"):
        net = [(t(W[:i, :o]).requires_grad_(k == "train"), t(b[:o]).requires_grad_(k == "train"))
               for (W, b), (i, _, o, _) in zip(_weights(seed)[0], _LAYERS)]
    if k == "train":
        f, b, g = _pairs(case["n"], seed)
        z = _mlp64(net, t(f))
        loss = torch.nn.functional.cross_entropy(z[:, :5], torch.as_tensor(b, device=_dev()).long()) + \
            0.1 * ((z[:, 5] - t(g)) ** 2).mean()
        loss.backward()
        flat = []
        for (W, bb), (i, ip, o, op) in zip(net, _LAYERS):
            P, q = torch.zeros(ip, op, dtype=torch.float64), torch.zeros(op, dtype=torch.float64)
            P[:i, :o], q[:o] = W.grad.cpu(), bb.grad.cpu()
            flat += [P.reshape(-1), q]
        return [float(loss.detach()), torch.cat(flat)]
    parts = _inputs(case, seed)
    if k == "newton":
        return _exact_newton(parts[0])
    if k == "batch" or k == "residual":
        r = []
        for d in parts:
            x = _Exact(d["grid"], d["mat"])
            r.append(x.forces(d["u"], x.commit(d["u0"])[0], d["f"]))
        return [torch.cat(r)]
    d = parts[0]
    x = _Exact(d["grid"], d["mat"])
    ep, al = x.commit(d["u0"])
    if k == "steps":
        keep = []
        r = x.forces(d["u"], ep, np.zeros(x.neq), keep=keep)
        return [torch.cat([a.reshape(-1) for a, _ in keep]), torch.cat([b.reshape(-1) for _, b in keep]), r]
    if k == "infer":
        lam, mu, phi, psi, c = d["mat"]
        feat, tg = [], []
        u = t(d["u"])
        for s in x.cuts:
            dx, dy, _ = x.geo(s)
            m = _return_map(x.strain(s, u, dx, dy), ep[s], d["mat"])
            one = torch.ones_like(al[s])[..., None]
            feat.append(torch.cat([m["ev"] / c, one * math.log(c), one * phi, one * psi, 1e3 * al[s][..., None],
                                   0 * one], -1).reshape(-1, 8))
            tg.append(1e3 * m["dalpha"].reshape(-1))
        feat = torch.cat(feat)
        return [feat, None, torch.cat(tg), _mlp64(net, feat), None, None]
    dep = []
    r = x.forces(d["u"], ep, d["f"], dep=dep)
    if k == "tangent":
        return [r, x.product(dep, t(d["v"]))]
    if k == "apply":
        return [x.product(dep, t(d["v"]))]
    if k == "cg":
        return [x.solve(dep, r, t(~d["grid"].fixed()))]
    K = x.stiffness(dep)  # assemble: the upper triangle's values, row by row, columns ascending
    dof = torch.stack([2 * x.conn, 2 * x.conn + 1], -1).flatten(1)
    i, j = dof[:, :, None].expand(K.shape), dof[:, None, :].expand(K.shape)
    up = i <= j
    key, inv = torch.unique((i * x.neq + j)[up], return_inverse=True)
    return [r, torch.zeros(len(key), dtype=torch.float64, device=K.device).index_add_(0, inv, K[up])]


def _exact_newton(d):
    """One load step from the virgin state, to rounding."""
    x = _Exact(d["grid"], d["mat"])
    ep, _ = x.commit(None)
    free = x.t(~d["grid"].fixed())
    u = torch.zeros(x.neq, dtype=torch.float64, device=x.X.device)
    first = None
    for _ in range(25):
        dep = []
        r = x.forces(u, ep, d["f"], dep=dep)
        n = float((r * free).norm())
        first = first or n
        if n <= 1e-13 * first:
            break
        u = u + x.solve(dep, r, free)
    ep, al = x.commit(u)
    z = torch.zeros_like(al)
    state = torch.stack([ep[..., 0], ep[..., 1], z, ep[..., 2], z, ep[..., 3]], -1)
    return [u, state.reshape(-1), al.reshape(-1)]
