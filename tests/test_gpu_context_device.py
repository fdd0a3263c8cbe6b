"""The per-block entries refuse a context that belongs to another device, and
launch nothing."""
import ctypes

import pytest

from alpaca_amd import gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [2, 3])
def test_context_of_another_device_is_refused(dim):
    import torch

    print(f"[context device] dim={dim}", flush=True)
    lib = gpu.load_library()
    ctx = ctypes.c_void_p()
    gpu.check(lib.alpaca_context_create(gpu._stream_ptr(), ctypes.byref(ctx)), "context_create")
    # The context's device, its first member: as if created on the next device.
    device = ctypes.c_int.from_address(ctx.value)
    assert device.value == torch.cuda.current_device()
    desc = ctypes.byref(gpu.make_desc(dim, [1, 1, 1], [0, 0, 0], cell_size=1.0 / 64))
    shape = (dim + 2, 24, 24, 24 if dim == 3 else 1)
    avg = torch.ones(shape, dtype=torch.float64, device="cuda")
    rhs = torch.full_like(avg, 7.0)
    jump = torch.full((6, dim + 2, 16, 16 if dim == 3 else 1), 5.0, dtype=torch.float64, device="cuda")
    flux = torch.full((3, dim + 2, 17, 17, 17 if dim == 3 else 2), 3.0, dtype=torch.float64,
                      device="cuda")
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    calls = [lambda: lib.alpaca_ctx_right_hand_side(ctx, desc, 1, P(avg), P(rhs)),
             lambda: lib.alpaca_ctx_right_hand_side_jump_fluxes(ctx, desc, 1, P(avg), P(rhs), P(jump)),
             lambda: lib.alpaca_ctx_convective_fluxes(ctx, desc, 1, P(avg), P(flux))]
    device.value += 1
    assert [c() for c in calls] == [1, 1, 1]  # ALPACA_ERR_INVALID
    torch.cuda.synchronize()
    assert (rhs == 7.0).all() and (jump == 5.0).all() and (flux == 3.0).all()
    device.value -= 1
    assert [c() for c in calls] == [0, 0, 0]
    gpu.check(lib.alpaca_context_destroy(ctx), "context_destroy")
