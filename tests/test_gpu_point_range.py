"""The return map over the whole range of its operands, against the oracle.

The GPU kernels take quotients and roots by their own correctly rounded
sequences inside a stated range and by the operators outside it; the results
are the oracle's bit for bit either way (NaN in the same places): stresses,
tangents, committed in-plane plastic strain, alpha, mtype and branch.
"""
import numpy as np
import pytest

import intpointsfem_amd as ipf
from intpointsfem_amd import wellbore as wb
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _point_map(gpu, mesh):
    import torch
    m = wb.make_mesh(mesh)
    sm = ipf.StructMatrix(m, device=0)
    ctx, d, w = sm.context(), m.material(), sm.export_indexes()["weight"]
    n = sm.sizes()["npts"]
    mat = (d["lambda"], d["mu"], d["phi"], d["psi"], d["cohesion"])

    def compare(eps):
        eps = np.ascontiguousarray(eps, dtype=np.float64).reshape(-1)
        with np.errstate(all="ignore"):
            want = O.compute_sigma(eps, w, *mat, update_mem=True, dep=True, nthreads=8)
        ctx.set_state(np.zeros(6 * n), np.zeros(n))
        e = torch.as_tensor(eps, device=gpu)
        ws = torch.zeros(3 * n, dtype=torch.float64, device=gpu)
        wd = torch.zeros(9 * n, dtype=torch.float64, device=gpu)
        torch.cuda.synchronize()
        ctx.set_update_mem(True)
        ctx.compute_sigma_dep(e, ws, wd)
        ctx.set_update_mem(False)
        ctx.synchronize()
        ep, al, mt, br = ctx.get_state()
        inplane = [0, 1, 3, 5]  # XZ and YZ are not stored
        got = (ws.cpu().numpy(), wd.cpu().numpy(), ep.reshape(n, 6)[:, inplane], al, mt, br)
        want = (want[0], want[1], want[2].reshape(n, 6)[:, inplane], *want[3:])
        for name, a, b in zip(("w sigma", "w Dep", "plastic strain", "alpha", "mtype", "branch"), got, want):
            assert np.array_equal(a, b, equal_nan=a.dtype.kind == "f"), name
    return n, compare


def test_scales(gpu):
    n, compare = _point_map(gpu, (20, 20, 2, 1.1))
    base = np.random.default_rng(5).standard_normal((n, 3))
    for k in (-322, -320, -316, -313, -312, -311, -310, -308, -300, -160, -158, -156, -155, -154, -152, -148, -146, -145,
              -144, -100, -20, -3, -1, 0, 10, 100, 139, 140, 141, 142, 145, 150, 152, 155, 200, 303, 305):
        with np.errstate(all="ignore"):
            eps = base * np.float64(f"1e{k}")
        try:
            compare(eps)
        except AssertionError as e:
            raise AssertionError(f"strains of 1e{k}") from e


@pytest.mark.parametrize("lo,hi", [(-320, 0), (-320, -280), (-160, 0), (-150, -138), (-150, 150), (-300, 300), (0, 300)])
def test_mixed_magnitudes(gpu, lo, hi):
    n, compare = _point_map(gpu, (40, 40, 2, 1.1))
    rng = np.random.default_rng(6)
    with np.errstate(all="ignore"):
        compare(rng.standard_normal((n, 3)) * 10.0 ** rng.uniform(lo, hi, (n, 3)))


@pytest.mark.parametrize("case", ["zero", "no shear", "uniaxial", "isotropic", "shear 1e-313", "shear 1e-303",
                                  "deviatoric, shear 1e-312", "infinite and NaN"])
def test_special_states(gpu, case):
    n, compare = _point_map(gpu, (40, 40, 2, 1.1))
    e = np.random.default_rng(7).standard_normal((n, 3)) * 1e-3
    if case == "zero":
        e[:] = 0
    elif case == "no shear":
        e[:, 1] = 0
    elif case == "uniaxial":
        e[:, :2] = 0
    elif case == "isotropic":
        e[:, 1], e[:, 2] = 0, e[:, 0]
    elif case == "shear 1e-313":
        e[:, 1] *= 1e-310
    elif case == "shear 1e-303":
        e[:, 1] *= 1e-300
    elif case == "deviatoric, shear 1e-312":
        e[:, 2] = -e[:, 0]
        e[:, 1] *= 1e-309
    else:
        e[::3, 0], e[1::5, 1], e[2::7, 2], e[::4, 2] = np.inf, -np.inf, np.nan, np.inf
    compare(e)


def test_a_million_points(gpu):
    n, compare = _point_map(gpu, (334, 333, 2, 1.01))
    assert n > 1_000_000
    rng = np.random.default_rng(8)
    compare(rng.standard_normal((n, 3)) * 10.0 ** rng.uniform(-8, -1, (n, 1)))
    compare(rng.standard_normal((n, 3)) * 10.0 ** rng.uniform(-12, 0, (n, 3)))
