"""The reverse of the red-black sweeps where a periodic axis is one cell long: a cell is then its own
neighbour twice, each sweep reads its old value, and the reverse keeps that share of the adjoint.
Against the oracle's unrolled reverse, and against the tangent: <J t, w> = <t, J^T w>.
"""
import numpy as np
import pytest

from ds_smoke import abi, scenes
from helpers import collider, random_fields, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res,axes", [((12, 15, 1), (2,)), ((1, 8, 9), (0,)), ((9, 1, 14), (1,)), ((1, 1, 16), (0, 1)), ((20, 16, 1), (0, 2))])
def test_reverse(res, axes):
    import oracle as O
    from ds_smoke.solver import Context

    print(f"red-black reverse {res}, periodic {axes}", flush=True)
    h = 1.0 / 16.0
    per = [a in axes for a in range(3)]
    sc = scenes.Scene(resolution=res, cell_size=h, time_step=0.5 * h, name="one-cell")
    sc.velocity_modes = tuple(m for p in per for m in ((3, 3) if p else (0, 2)))
    sc.pressure_modes = sc.density_modes = sc.temperature_modes = tuple(m for p in per for m in ((2, 2) if p else (1, 1)))
    if min(res[0], res[1]) > 4:
        sc.colliders = [collider(abi.SHAPE_BOX, (0.3 * res[0] * h, 0.6 * res[1] * h, 0.5 * h), (1.2 * h, 1.2 * h, h))]
    config = dict(solver=abi.PROJECTION_RBGS, rbgs_iterations=4)
    ctx = Context(sc.config(**config), abi.MODE_DIFFERENTIABLE)
    orc = O.Oracle(sc, **config)
    f, t = random_fields(sc, seed=89), random_fields(sc, seed=97)
    ua, _ = ctx.projection_vjp(tuple(ctx.to_device(v) for v in f["face_adj"]))
    ref = orc.projection_vjp(f["face_adj"])
    ref = ref[0] if isinstance(ref[0], (tuple, list)) else ref
    back = ctx.to_host(ua)
    for a in range(3):
        # FP32 sums of seven terms, contracted by 8 sweeps
        assert rel(back[a], ref[a]) < 5e-6, (a, rel(back[a], ref[a]))
    out, _ = ctx.projection_jvp(tuple(ctx.to_device(v) for v in t["vel"]))
    dot = lambda p, q: sum(float(np.sum(x.astype(np.float64) * y.astype(np.float64))) for x, y in zip(p, q))
    size = sum(float(np.linalg.norm(x) * np.linalg.norm(y)) for x, y in zip(ctx.to_host(out), f["face_adj"]))
    assert abs(dot(ctx.to_host(out), f["face_adj"]) - dot(t["vel"], back)) <= 1e-5 * size
