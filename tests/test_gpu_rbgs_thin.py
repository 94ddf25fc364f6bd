"""The red-black sweeps on grids that are thin along one axis (csrc/rbgs.hip, rbgs_solve_kind: more than
256 flat boxes, along x more than 256 deep ones, and less than two thirds of the deep boxes' points), with
remainders, a collider, a fixed-value face and a periodic axis along and across the thin one. Against the
oracle's FP64 sweeps: FP32 sums of seven terms and a division, contracted by the sweeps, 1e-6 per
iteration at most. And the cost of the sweeps, which with the deep box followed the box and not the cells.
"""
import numpy as np
import pytest

from ds_smoke import abi, scenes
from helpers import collider, random_fields, rel

pytestmark = pytest.mark.gpu

SIZES = [(1, 300, 250), (2, 181, 200), (5, 130, 266), (4, 261, 150), (8, 100, 90), (129, 1, 140), (131, 2, 130), (700, 301, 1), (702, 300, 2)]


def _scene(res, periodic_axis=None):
    h = 1.0 / max(res)
    sc = scenes.Scene(resolution=res, cell_size=h, time_step=0.5 * h, name="thin")
    sc.colliders = [collider(abi.SHAPE_BOX, tuple(0.4 * v * h for v in res), tuple(0.1 * v * h if v > 8 else 0.5 * h for v in res))]
    sc.pressure_modes = (1, 1, 1, 1, 1, 0)
    sc.pressure_values = (0.0, 0.0, 0.0, 0.0, 0.0, 0.1)
    if periodic_axis is not None:
        sc.velocity_modes, sc.pressure_modes, sc.density_modes, sc.temperature_modes = (
            tuple(p if f // 2 == periodic_axis else m for f, m in enumerate(modes))
            for modes, p in ((sc.velocity_modes, 3), (sc.pressure_modes, 2), (sc.density_modes, 2), (sc.temperature_modes, 2)))
    return sc


@pytest.mark.parametrize("periodic_axis", [None, 0, 1, 2])
@pytest.mark.parametrize("res", SIZES)
def test_sweeps_on_thin_grids(res, periodic_axis):
    import oracle as O
    from ds_smoke.solver import Context

    if periodic_axis is not None and res[periodic_axis] % 2:
        pytest.skip("a periodic axis of odd extent is swept by one launch a colour")
    print(f"RBGS thin {res} periodic {periodic_axis}", flush=True)
    iterations = 3
    sc = _scene(res, periodic_axis)
    ctx = Context(sc.config(solver=abi.PROJECTION_RBGS, rbgs_iterations=iterations), abi.MODE_FORWARD)
    orc = O.Oracle(sc, solver=abi.PROJECTION_RBGS, rbgs_iterations=iterations)
    f = random_fields(sc, seed=67, vel_scale=0.5)
    out, p, _, info = ctx.projection_forward(tuple(ctx.to_device(v) for v in f["vel"]))
    assert info.iterations == iterations
    ref, ref_p, _, _ = orc.projection_forward(f["vel"])
    assert rel(ctx.to_host(p), ref_p) < 1e-6 * iterations, rel(ctx.to_host(p), ref_p)
    got = ctx.to_host(out)
    for a in range(3):
        assert rel(got[a], ref[a]) < 1e-5, (a, rel(got[a], ref[a]))


def test_a_sweep_costs_what_its_cells_do():
    import torch
    from ds_smoke.solver import Context

    def ms(res):
        h = 1.0 / max(res)
        sc = scenes.Scene(resolution=res, cell_size=h, time_step=0.5 * h, name="thin")
        ctx = Context(sc.config(solver=abi.PROJECTION_RBGS, rbgs_iterations=80), abi.MODE_FORWARD)
        u = tuple(ctx.to_device(v) for v in random_fields(sc, seed=67)["vel"])
        times = []
        for _ in range(5):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record(ctx.stream)
            ctx.projection_forward(u)
            b.record(ctx.stream)
            b.synchronize()
            times.append(a.elapsed_time(b))
        print(f"{res}: {1e3 * np.median(times):.0f} us", flush=True)
        ctx.close()
        return float(np.median(times))

    cube = ms((128, 128, 64))
    for res in [(1024, 1024, 1), (1024, 1, 1024), (1, 1024, 1024), (2, 1024, 512)]:
        assert ms(res) <= 3.0 * cube, res
