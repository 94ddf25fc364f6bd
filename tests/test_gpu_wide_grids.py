"""Grids with more than 512 tiles of 64 x 8 cells in a plane (1024 x 264 and wider; resolutions up to
1024 per axis are accepted): the plane-marching tiling of the Jacobi PCG forms has no block count for
them, and context creation used to look for one without end. The multigrid form, which does not use
the tiling, solves on them; the Jacobi forms are refused; the red-black projection runs whatever
cg_variant says.
"""
import numpy as np
import pytest

from ds_smoke import abi, scenes
from helpers import pressure_residual, random_fields

pytestmark = pytest.mark.gpu

RES = (1024, 272, 2)   # 16 x 34 = 544 tiles


def _scene():
    return scenes.Scene(resolution=RES, cell_size=1.0 / 1024.0, time_step=0.5 / 1024.0, name="wide")


def test_multigrid_solves_on_a_wide_grid():
    from ds_smoke.solver import Context

    print(f"wide grid {RES}, multigrid", flush=True)
    ctx = Context(_scene().config(tolerance=1e-6), abi.MODE_FORWARD)
    _, code = ctx.masks()
    b = np.where(code > 0, np.random.default_rng(5).standard_normal(code.shape), 0.0).astype(np.float32)
    x, info, st = ctx.pcg_solve(ctx.to_device(b))
    print(f"  {info.iterations} iterations", flush=True)
    assert st == abi.DS_OK and info.converged and info.iterations <= 30
    x = ctx.to_host(x)
    # x is rounded to FP32 on return: an error of 2^-24 |x|, through rows of at most 6 + 6
    bound = 1e-6 * np.linalg.norm(b) + 12.0 * 2.0 ** -24 * np.linalg.norm(x)
    assert np.linalg.norm(pressure_residual(code, x, b)) <= bound


@pytest.mark.parametrize("variant", [abi.CG_SINGLE_REDUCTION, abi.CG_TWO_REDUCTION, abi.CG_SINGLE_REDUCTION_RESIDENT, abi.CG_S_STEP])
def test_jacobi_forms_are_refused_on_a_wide_grid(variant):
    from ds_smoke.solver import Context, SolverError

    print(f"wide grid {RES}, form {variant}", flush=True)
    with pytest.raises(SolverError) as e:
        Context(_scene().config(cg_variant=variant), abi.MODE_FORWARD)
    assert e.value.status == abi.DS_ERROR_UNSUPPORTED and "PCG tiling" in str(e.value)


def test_red_black_projection_runs_on_a_wide_grid():
    from ds_smoke.solver import Context, SolverError

    print(f"wide grid {RES}, red-black", flush=True)
    sc = _scene()
    f = random_fields(sc, seed=3, vel_scale=0.2)

    def project(variant):
        ctx = Context(sc.config(solver=abi.PROJECTION_RBGS, rbgs_iterations=3, cg_variant=variant), abi.MODE_FORWARD)
        out, p, _, info = ctx.projection_forward(tuple(ctx.to_device(v) for v in f["vel"]))
        assert info.iterations == 3
        return ctx, ctx.to_host(p)

    ctx, p = project(abi.CG_SINGLE_REDUCTION)
    _, q = project(abi.CG_MULTIGRID)
    assert np.array_equal(p, q) and p.any()
    with pytest.raises(SolverError) as e:
        ctx.pcg_solve(ctx.zeros_cell())
    assert e.value.status == abi.DS_ERROR_UNSUPPORTED
