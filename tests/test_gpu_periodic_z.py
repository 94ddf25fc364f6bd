"""Domains that are periodic in z (alone, with y, and in every direction): the wrapped planes of the
multigrid kernels over every box and over grids of one to three cells along an axis, the wrapped halos
of the red-black boxes along y and z, and the seams of the traces in a step, its reverse and its
tangent. Grids of the boxes' sizes with remainders, a collider on the seam.
"""
import numpy as np
import pytest

from ds_smoke import abi, scenes
from helpers import collider, pressure_residual, random_fields, rel

pytestmark = pytest.mark.gpu

AXES = [(False, False, True), (False, True, True), (True, True, True)]


def _scene(res, periodic, h=None):
    h = h or 1.0 / max(res)
    sc = scenes.Scene(resolution=res, cell_size=h, time_step=0.5 * h, name="periodic_z")
    sc.velocity_modes = tuple(m for p in periodic for m in ((3, 3) if p else (0, 2)))
    sc.pressure_modes = sc.density_modes = sc.temperature_modes = tuple(m for p in periodic for m in ((2, 2) if p else (1, 1)))
    if min(res) > 4:
        sc.colliders = [collider(abi.SHAPE_ELLIPSOID, (0.4 * res[0] * h, 0.5 * res[1] * h, h), (0.2 * res[0] * h, 0.2 * res[1] * h, 2.6 * h),
                                 velocity=(0.1, 0.0, 0.05), density=0.3, temperature=0.2)]
    return sc


# small, medium and large boxes of level 0, both of the coarser levels, one to three cells along an axis
@pytest.mark.parametrize("periodic", AXES)
@pytest.mark.parametrize("res", [(20, 18, 22), (17, 13, 9), (49, 40, 37), (96, 80, 75), (130, 96, 91), (40, 33, 1), (40, 33, 2), (21, 34, 3),
                                 (2, 33, 40), (33, 1, 40), (1, 33, 37), (3, 3, 80), (1, 1, 700)])
def test_multigrid(res, periodic):
    from ds_smoke.solver import Context

    print(f"multigrid {res} periodic {periodic}", flush=True)
    ctx = Context(_scene(res, periodic).config(tolerance=1e-6), abi.MODE_FORWARD)
    _, code = ctx.masks()
    b = np.where(code > 0, np.random.default_rng(41).standard_normal(code.shape), 0.0).astype(np.float32)
    x, info, st = ctx.pcg_solve(ctx.to_device(b))
    print(f"  {info.iterations} iterations", flush=True)
    assert st == abi.DS_OK and info.converged and info.iterations <= 30
    x = ctx.to_host(x)
    # x is rounded to FP32 on return: an error of 2^-24 |x|, through rows of at most 6 + 6
    bound = 1e-6 * np.linalg.norm(b) + 12.0 * 2.0 ** -24 * np.linalg.norm(x)
    assert np.linalg.norm(pressure_residual(code, x, b, periodic)) <= bound


# flat boxes, and the deep ones of more than 256 flat boxes
@pytest.mark.parametrize("iterations", [1, 4])
@pytest.mark.parametrize("res,periodic", [((34, 18, 8), AXES[0]), ((33, 18, 6), AXES[1]), ((34, 18, 8), AXES[2]), ((8, 6, 2), AXES[2]),
                                          ((97, 83, 44), AXES[0]), ((97, 84, 46), AXES[1]), ((96, 82, 46), AXES[2])])
def test_red_black_boxes(res, periodic, iterations):
    import oracle as O
    from ds_smoke.solver import Context

    print(f"red-black {res} periodic {periodic} iterations {iterations}", flush=True)
    sc = _scene(res, periodic)
    ctx = Context(sc.config(solver=abi.PROJECTION_RBGS, rbgs_iterations=iterations), abi.MODE_FORWARD)
    orc = O.Oracle(sc, solver=abi.PROJECTION_RBGS, rbgs_iterations=iterations)
    f = random_fields(sc, seed=71, vel_scale=0.5)
    out, p, _, _ = ctx.projection_forward(tuple(ctx.to_device(v) for v in f["vel"]))
    ref, ref_p, _, _ = orc.projection_forward(f["vel"])
    # FP32 sums of seven terms and a division, contracted by the sweeps: 1e-6 per iteration at most
    assert rel(ctx.to_host(p), ref_p) < 1e-6 * iterations, rel(ctx.to_host(p), ref_p)
    got = ctx.to_host(out)
    for a in range(3):
        assert rel(got[a], ref[a]) < 1e-5, (a, rel(got[a], ref[a]))


# deep boxes with remainders, an odd extent along x, solids and a fixed-value face
@pytest.mark.parametrize("res", [(97, 83, 45), (98, 81, 47)])
def test_red_black_deep_boxes_with_solids(res):
    import oracle as O
    from ds_smoke.solver import Context
    from helpers import scene_solids

    print(f"red-black deep, solids {res}", flush=True)
    sc = scene_solids(res)
    ctx = Context(sc.config(solver=abi.PROJECTION_RBGS, rbgs_iterations=5), abi.MODE_FORWARD)
    orc = O.Oracle(sc, solver=abi.PROJECTION_RBGS, rbgs_iterations=5)
    f = random_fields(sc, seed=73, vel_scale=0.5)
    _, p, _, _ = ctx.projection_forward(tuple(ctx.to_device(v) for v in f["vel"]))
    _, ref_p, _, _ = orc.projection_forward(f["vel"])
    assert rel(ctx.to_host(p), ref_p) < 5e-6, rel(ctx.to_host(p), ref_p)


# a cell size that is a power of two and one that is not; h = 1 / 16 as a last axis of one cell too
@pytest.mark.parametrize("res,h", [((16, 12, 14), 1.0 / 16.0), ((15, 13, 11), 1.0 / 15.0), ((18, 11, 1), 1.0 / 16.0)])
@pytest.mark.parametrize("periodic", AXES)
def test_step_reverse_and_tangent(res, h, periodic):
    import oracle as O
    from ds_smoke.solver import Context

    print(f"step {res} periodic {periodic}", flush=True)
    sc = _scene(res, periodic, h)
    sc.params = (0.1, -0.1, 1.0, 0.0)
    ctx = Context(sc.config(tolerance=1e-8), abi.MODE_DIFFERENTIABLE)
    orc = O.Oracle(sc, tolerance=1e-11)
    f = random_fields(sc, seed=79, vel_scale=0.4)
    s = {"density": f["rho"], "temperature": f["T"], "velocity": f["vel"]}
    k = {"density_source": f["s_rho"], "temperature_source": f["s_T"], "external_acceleration": f["e"]}
    params = ctx.allocate_parameters(sc.params)
    st, kt = ctx.state_from_host(s), ctx.control_from_host(k)
    nxt, cache, info = ctx.forward_step(st, kt, params)
    ref, ref_cache, _ = orc.forward_step(s, k, sc.params)
    got = ctx.to_host(nxt)
    for key in ("density", "temperature"):
        assert rel(got[key], ref[key]) < 1e-5, (key, rel(got[key], ref[key]))
    for a in range(3):
        assert rel(got["velocity"][a], ref["velocity"][a]) < 1e-5, (a, rel(got["velocity"][a], ref["velocity"][a]))

    adj = {"density": f["cell_adj"], "temperature": f["cell_adj2"], "velocity": f["face_adj"]}
    prev, _ = ctx.vjp_step(st, kt, params, nxt, cache, ctx.state_from_host(adj))
    ref_prev, _ = orc.vjp_step(ref, ref_cache, sc.params, adj)
    g = ctx.to_host(prev)
    for key in ("density", "temperature"):
        assert rel(g[key], ref_prev[key]) < 1e-4, (key, rel(g[key], ref_prev[key]))
    for a in range(3):
        assert rel(g["velocity"][a], ref_prev["velocity"][a]) < 1e-4, (a, rel(g["velocity"][a], ref_prev["velocity"][a]))

    # the tangent along (adj, zero control) against the reverse of the same step: <J t, v> = <t, J^T v>
    t = random_fields(sc, seed=83, vel_scale=1.0)
    st_t = {"density": t["cell_adj"], "temperature": t["cell_adj2"], "velocity": t["face_adj"]}
    zero = ctx.allocate_control()
    out, _ = ctx.jvp_step(st, kt, params, nxt, cache, ctx.state_from_host(st_t), zero, ctx.allocate_parameters())
    o = ctx.to_host(out)
    pairs = [(o["density"], adj["density"]), (o["temperature"], adj["temperature"])] + list(zip(o["velocity"], adj["velocity"]))
    back = [(st_t["density"], g["density"]), (st_t["temperature"], g["temperature"])] + list(zip(st_t["velocity"], g["velocity"]))
    dot = lambda ps: sum(float(np.sum(a.astype(np.float64) * b.astype(np.float64))) for a, b in ps)
    size = sum(float(np.linalg.norm(a.astype(np.float64)) * np.linalg.norm(b.astype(np.float64))) for a, b in pairs)
    assert abs(dot(pairs) - dot(back)) <= 1e-4 * size, (dot(pairs), dot(back), size)
