"""A collider that lies on a periodic seam with more cells on one side of it than on the other: the
seam's face 0 and its duplicate, face n, are then constrained in places by the solid beyond one of them
only (operators.cu:466-497), and the reverse of the constraint has to carry the duplicate's adjoint to
face 0 also where face 0 itself is constrained. Against the oracle, whose reverse agrees with its
tangent and with finite differences there.
"""
import numpy as np
import pytest

from ds_smoke import abi, scenes
from helpers import collider, random_fields, rel

pytestmark = pytest.mark.gpu

RES = (14, 12, 13)
H = 1.0 / 16.0


def _scene(axis, centre):
    sc = scenes.Scene(resolution=RES, cell_size=H, time_step=0.5 * H, name="seam-solid")
    sc.velocity_modes = tuple(m for a in range(3) for m in ((3, 3) if a == axis else (0, 2)))
    sc.pressure_modes = sc.density_modes = sc.temperature_modes = tuple(m for a in range(3) for m in ((2, 2) if a == axis else (1, 1)))
    c = [0.5 * n * H for n in RES]
    c[axis] = centre * H
    sc.colliders = [collider(abi.SHAPE_ELLIPSOID, tuple(c), (2.6 * H, 2.6 * H, 2.6 * H), velocity=(0.1, 0.0, 0.05))]
    sc.params = (0.1, -0.1, 1.0, 0.0)
    return sc


@pytest.mark.parametrize("side", ["low", "high"])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_reverse_at_the_seam(axis, side):
    import oracle as O
    from ds_smoke.solver import Context

    print(f"solid on the seam of axis {axis}, {side}", flush=True)
    sc = _scene(axis, 1.0 if side == "low" else RES[axis] - 1.0)
    ctx = Context(sc.config(tolerance=1e-8), abi.MODE_DIFFERENTIABLE)
    orc = O.Oracle(sc, tolerance=1e-11)
    f = random_fields(sc, seed=3, vel_scale=0.4)
    # the constraint alone: a copy or a sum of two per face
    ua = ctx.zeros_faces()
    ctx.constrain_vjp(tuple(ctx.to_device(v) for v in f["face_adj"]), ua)
    ref_ua = orc.zeros_faces()
    orc.constrain_vjp(f["face_adj"], ref_ua)
    for a in range(3):
        assert rel(ctx.to_host(ua[a]), ref_ua[a]) < 1e-7, (a, rel(ctx.to_host(ua[a]), ref_ua[a]))
    # and in a step
    s = {"density": f["rho"], "temperature": f["T"], "velocity": f["vel"]}
    k = {"density_source": f["s_rho"], "temperature_source": f["s_T"], "external_acceleration": f["e"]}
    params = ctx.allocate_parameters(sc.params)
    st, kt = ctx.state_from_host(s), ctx.control_from_host(k)
    nxt, cache, _ = ctx.forward_step(st, kt, params)
    ref, ref_cache, _ = orc.forward_step(s, k, sc.params)
    adj = {"density": f["cell_adj"], "temperature": f["cell_adj2"], "velocity": f["face_adj"]}
    prev, _ = ctx.vjp_step(st, kt, params, nxt, cache, ctx.state_from_host(adj))
    ref_prev, _ = orc.vjp_step(ref, ref_cache, sc.params, adj)
    g = ctx.to_host(prev)
    for key in ("density", "temperature"):
        assert rel(g[key], ref_prev[key]) < 1e-5, (key, rel(g[key], ref_prev[key]))
    # 1e-6 of rounding, and a trace whose midpoint lies within FP32 rounding of a cell boundary takes the
    # other cell's derivative: one in these six scenes, 5.5e-4 at the four faces of its start stencil,
    # 4.0e-5 of the norm (without the seam's share the error is 0.1 to 0.2)
    for a in range(3):
        assert rel(g["velocity"][a], ref_prev["velocity"][a]) < 1e-4, (a, rel(g["velocity"][a], ref_prev["velocity"][a]))
