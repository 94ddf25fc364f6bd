"""Buffers that a context keeps between trajectory calls: calls of other lengths and other kinds in a
row on one context (each takes what the ones before it left, with their contents) give what a fresh
context gives, and closing the context frees them.
"""
import pytest

from helpers import rel

pytestmark = pytest.mark.gpu

CALLS = [(6, 2), (3, 1), (7, 3), (6, 2)]


@pytest.mark.parametrize("warm", ["none", "extrapolate"])
def test_calls_of_other_lengths_in_a_row(warm):
    import torch
    from ds_smoke import abi, scenes
    from ds_smoke.solver import Context

    sc = scenes.plume(16)
    kind = {"none": abi.WARM_START_NONE, "extrapolate": abi.WARM_START_EXTRAPOLATE}[warm]

    def make():
        ctx = Context(sc.config(tolerance=1e-6, warm_start=kind), abi.MODE_DIFFERENTIABLE)
        return ctx, (ctx.state_from_host(scenes.initial_state(sc)), ctx.control_from_host(scenes.control(sc)),
                     ctx.allocate_parameters(sc.params))

    def call(ctx, x, steps, interval):
        loss, grad, _ = ctx.loss_gradient(*x, steps, interval, ctx.to_device(sc.target))
        final, _ = ctx.simulate(*x, steps)
        return loss, ctx.to_host(grad), ctx.to_host(final)

    kept, x = make()
    for steps, interval in CALLS:
        got = call(kept, x, steps, interval)
        fresh, y = make()
        ref = call(fresh, y, steps, interval)
        fresh.close()
        # the reverse adds in no fixed order (FP64 sums rounded to FP32, an ulp or two)
        assert abs(got[0] - ref[0]) <= 1e-6 * ref[0], (steps, interval)
        for a, b in zip(got[1:], ref[1:]):
            for f in ("density", "temperature"):
                assert rel(a[f], b[f]) < 2e-6 or not b[f].any(), (steps, interval, f)
            for i in range(3):
                assert rel(a["velocity"][i], b["velocity"][i]) < 2e-6, (steps, interval, i)
    kept.close()
    torch.cuda.synchronize()


def test_closing_the_context_frees_them():
    import torch
    from ds_smoke import abi, scenes
    from ds_smoke.solver import Context

    sc = scenes.plume(64)

    def once():
        ctx = Context(sc.config(tolerance=1e-6), abi.MODE_DIFFERENTIABLE)
        ctx.loss_gradient(ctx.state_from_host(scenes.initial_state(sc)), ctx.control_from_host(scenes.control(sc)),
                          ctx.allocate_parameters(sc.params), 32, 1, ctx.to_device(sc.target))
        ctx.close()
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        return torch.cuda.mem_get_info()[0]

    first = once()   # 32 checkpoints of 5 MiB and more
    assert abs(once() - first) < 64 << 20
