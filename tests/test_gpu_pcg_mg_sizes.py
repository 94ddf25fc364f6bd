"""The multigrid-preconditioned PCG on both sides of the cell counts at which its kernels change:
512 cells (solved directly up to there), 2^16 and 2^19 cells (boxes of the level-0 kernels), 2^17
cells of a coarser level (boxes of the coarse kernels), with odd extents, a periodic axis and a
collider. Against the two-reduction Jacobi form on the same matrix and right-hand side: two solves to
1e-6 ||b|| differ by twice the error of one (5e-5 against the oracle on the smaller hierarchies).
"""
import numpy as np
import pytest

from helpers import collider, rel

pytestmark = pytest.mark.gpu

SIZES = [(8, 8, 8), (9, 8, 8), (40, 40, 40), (41, 40, 40), (80, 80, 81), (81, 81, 80), (100, 100, 100), (102, 101, 102)]


def _scene(res, periodic):
    from ds_smoke import abi, scenes

    h = 1.0 / res[0]
    sc = scenes.Scene(resolution=res, cell_size=h, time_step=0.5 * h, name="mg-sizes")
    if periodic:
        sc.velocity_modes = (3, 3, 0, 0, 0, 0)
        sc.pressure_modes = sc.density_modes = sc.temperature_modes = (2, 2, 1, 1, 1, 1)
        sc.colliders = [collider(abi.SHAPE_ELLIPSOID, (0.5, 0.45 * res[1] * h, 0.5 * res[2] * h), (0.2, 0.15, 0.18))]
    return sc


@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("res", SIZES)
def test_both_sides_of_each_size(res, periodic):
    from ds_smoke import abi
    from ds_smoke.solver import Context

    print(f"multigrid sizes {res} periodic {periodic}", flush=True)
    sc = _scene(res, periodic)
    ctx = Context(sc.config(tolerance=1e-6, cg_variant=abi.CG_MULTIGRID), abi.MODE_FORWARD)
    _, code = ctx.masks()
    b = np.where(code > 0, np.random.default_rng(29).standard_normal(code.shape), 0.0).astype(np.float32)
    x, info, st = ctx.pcg_solve(ctx.to_device(b))
    print(f"  {info.iterations} iterations, residual {info.final_residual / info.rhs_norm:.2e}", flush=True)
    assert st == 0 and info.converged and info.iterations <= 30
    assert info.final_residual <= 1e-6 * info.rhs_norm * (1 + 1e-9)
    other = Context(sc.config(tolerance=1e-6, cg_variant=abi.CG_TWO_REDUCTION), abi.MODE_FORWARD)
    y, _, st = other.pcg_solve(other.to_device(b))
    assert st == 0
    assert rel(ctx.to_host(x), other.to_host(y)) < 1e-4, rel(ctx.to_host(x), other.to_host(y))
