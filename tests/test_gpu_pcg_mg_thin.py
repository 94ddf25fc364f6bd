"""The multigrid-preconditioned PCG on large grids that are thin along one axis (csrc/pcg_mg.hip,
choose_box; 2^19 cells and more, 2^17 of a coarser level): every thin box with remainders, a periodic
axis across and along the thin one, a collider. The residual of the returned solution in FP64 against
the tolerance, and the cost of an iteration, which with the cubic box followed the planes of a box and
not the cells (1 x 1024 x 1024: 9 times that of 128 x 128 x 64).
"""
import numpy as np
import pytest

from ds_smoke import abi, scenes
from helpers import collider, pressure_residual

pytestmark = pytest.mark.gpu

SIZES = [(1, 1023, 517), (3, 500, 370), (1021, 1, 600), (2, 701, 390), (900, 590, 1), (601, 450, 2)]


@pytest.mark.parametrize("periodic", [(False, False, False), (True, False, True), (False, True, True)])
@pytest.mark.parametrize("res", SIZES)
def test_thin_grids(res, periodic):
    from ds_smoke.solver import Context

    print(f"thin grid {res}, periodic {periodic}", flush=True)
    h = 1.0 / max(res)
    sc = scenes.Scene(resolution=res, cell_size=h, time_step=0.5 * h, name="thin")
    sc.velocity_modes = tuple(m for p in periodic for m in ((3, 3) if p else (0, 0)))
    sc.pressure_modes = sc.density_modes = sc.temperature_modes = tuple(m for p in periodic for m in ((2, 2) if p else (1, 1)))
    sc.colliders = [collider(abi.SHAPE_BOX, tuple(0.4 * v * h for v in res), tuple(0.1 * v * h if v > 8 else h for v in res))]
    ctx = Context(sc.config(tolerance=1e-6), abi.MODE_FORWARD)
    _, code = ctx.masks()
    b = np.where(code > 0, np.random.default_rng(31).standard_normal(code.shape), 0.0).astype(np.float32)
    x, info, st = ctx.pcg_solve(ctx.to_device(b))
    print(f"  {info.iterations} iterations", flush=True)
    assert st == abi.DS_OK and info.converged and info.iterations <= 30
    x = ctx.to_host(x)
    # x is rounded to FP32 on return: an error of 2^-24 |x|, through rows of at most 6 + 6
    bound = 1e-6 * np.linalg.norm(b) + 12.0 * 2.0 ** -24 * np.linalg.norm(x)
    assert np.linalg.norm(pressure_residual(code, x, b, periodic)) <= bound


def test_an_iteration_costs_what_its_cells_do():
    from ds_smoke.solver import Context

    def iteration_ms(res):
        h = 1.0 / max(res)
        ctx = Context(scenes.Scene(resolution=res, cell_size=h, time_step=0.5 * h, name="thin").config(tolerance=1e-6), abi.MODE_FORWARD)
        b = ctx.to_device(np.random.default_rng(31).standard_normal(res[::-1]))
        ctx.pcg_solve(b)
        ctx.profile_enable(1)
        for _ in range(3):
            ctx.pcg_solve(b)
        launches, samples, ms = ctx.profile_read()["pcg_mg_iteration"]
        print(f"{res}: {samples} iterations, {1e3 * ms:.1f} us each", flush=True)
        ctx.close()
        return ms

    cube = iteration_ms((128, 128, 64))
    for res in [(1024, 1024, 1), (1024, 1, 1024), (1, 1024, 1024), (2, 1024, 512)]:
        assert iteration_ms(res) <= 2.5 * cube, res
