"""The device buffers that contexts keep between trajectory calls do not stand in the way of other
allocations: a public call gives them back, an allocation of the library or of its Python layer that
fails is tried again without them, another thread may release them at any time, and what is kept stays
within 1/16 of the card and is nothing when a call ends with less than a quarter of it free.
"""
import ctypes as C
import threading

import numpy as np
import pytest

from ds_smoke import abi, scenes

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def _free():
    import torch

    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    return torch.cuda.mem_get_info()[0]


class Problem:
    def __init__(self, n):
        from ds_smoke.solver import Context

        sc = scenes.plume(n)
        self.ctx = Context(sc.config(tolerance=1e-4), abi.MODE_DIFFERENTIABLE)
        self.x = (self.ctx.state_from_host(scenes.initial_state(sc)), self.ctx.control_from_host(scenes.control(sc)),
                  self.ctx.allocate_parameters(sc.params))
        self.target = self.ctx.to_device(sc.target)
        self.adj = self.ctx.allocate_state_adjoint()

    def gradient(self, steps):
        return self.ctx.loss_gradient(*self.x, steps, 1, self.target, initial_adj=self.adj)[0]


def test_the_release_call_returns_them():
    from ds_smoke.solver import release_buffers

    print("release call", flush=True)
    a, b = Problem(64), Problem(64)
    loss = a.gradient(32)
    b.gradient(32)
    full = _free()
    a.ctx.release_buffers()   # 33 states of 5 MiB and 32 tapes of 2
    one = _free()
    assert one - full > 128 * MIB
    release_buffers()
    assert _free() - one > 128 * MIB
    assert abs(a.gradient(32) - loss) <= 1e-6 * abs(loss)


@pytest.mark.parametrize("kind", ["ds_allocate", "context", "torch"])
def test_an_allocation_that_fails_takes_them(kind):
    import torch
    from ds_smoke.solver import Context

    print(f"allocation by {kind} on a full card", flush=True)
    a = Problem(128)
    a.gradient(32)   # 33 states of 40 MiB and 32 tapes of 16
    hog = torch.empty(_free() - 1024 * MIB, dtype=torch.uint8, device="cuda")
    assert torch.cuda.mem_get_info()[0] < 1800 * MIB
    try:
        if kind == "ds_allocate":
            p = C.c_void_p()
            st = a.ctx.lib.ds_allocate(a.ctx.h, C.c_size_t(2048 * MIB), C.byref(p))
            assert st == abi.DS_OK, a.ctx.lib.ds_last_error().decode()
            assert a.ctx.lib.ds_release(a.ctx.h, p) == abi.DS_OK
            a.ctx.synchronize()
        elif kind == "context":
            Context(scenes.plume(240).config(), abi.MODE_DIFFERENTIABLE).close()   # about 2.2 GiB
        else:
            assert a.ctx._zeros((512 * MIB,)).numel() == 512 * MIB
    finally:
        del hog
        a.ctx.close()
        torch.cuda.empty_cache()


def test_released_by_another_thread():
    from ds_smoke.solver import release_buffers

    print("released by another thread", flush=True)
    a = Problem(32)
    ref = a.gradient(8)
    stop = threading.Event()

    def release():
        while not stop.is_set():
            release_buffers()

    t = threading.Thread(target=release)
    t.start()
    try:
        losses = [a.gradient(8) for _ in range(30)]
    finally:
        stop.set()
        t.join()
    assert np.all(np.abs(np.array(losses) - ref) <= 1e-6 * abs(ref))


def test_what_is_kept_is_bounded():
    import torch

    print("bounds", flush=True)
    total = torch.cuda.mem_get_info()[1]
    a = Problem(192)
    a.gradient(2)
    a.ctx.release_buffers()
    before = _free()
    a.gradient(int(1.3 * total / 16 / (7 * 4 * 192 ** 3)))   # a state and a tape a step: more than 1/16 of the card
    kept = before - _free()
    print(f"  kept {kept / 2 ** 30:.1f} of {total / 2 ** 30:.0f} GiB", flush=True)
    assert total / 32 < kept <= total / 16 + 512 * MIB
    hog = torch.empty(int(_free() - 0.2 * total), dtype=torch.uint8, device="cuda")
    before = torch.cuda.mem_get_info()[0]
    a.gradient(2)
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] - before > 0.9 * kept   # all of it given back
    del hog
    a.ctx.close()
    torch.cuda.empty_cache()
