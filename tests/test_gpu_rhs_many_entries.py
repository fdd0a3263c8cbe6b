"""A right-hand side over a list of more entries than workgroups of 512 threads
could be launched for: all but a few lie outside the pool and are skipped."""
import ctypes

import numpy as np
import pytest

from alpaca_amd import cases, gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1 << 20) - 1, 1 << 20, (1 << 21) - 1])
@pytest.mark.parametrize("prec", [gpu.FP64_FMA, gpu.MIXED])
def test_long_lists(prec, n):
    import torch

    print(f"[many entries] prec={prec} n={n}", flush=True)
    lib, ctx = gpu.load_library(), ctypes.c_void_p()
    gpu.check(lib.alpaca_context_create(gpu._stream_ptr(), ctypes.byref(ctx)), "context_create")
    desc = ctypes.byref(gpu.make_desc(3, [1, 1, 1], [0, 0, 0], precision=prec, cell_size=1.0 / 64))
    avg = torch.as_tensor(np.stack([cases.random_block(3, s) for s in range(3)]), device="cuda")
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    out = []
    for entries, at in ((3, [0, 1, 2]), (n, [5, n // 2, n - 1])):
        index = torch.full((entries,), -1, dtype=torch.int32, device="cuda")
        index[torch.tensor(at, device="cuda")] = torch.arange(3, dtype=torch.int32, device="cuda")
        rhs, jump = torch.zeros_like(avg), torch.zeros((3, 6, 5, 16, 16), dtype=torch.float64,
                                                       device="cuda")
        gpu.check(lib.alpaca_ctx_right_hand_side_jump_fluxes_list(
            ctx, desc, 3, P(index), entries, P(avg), P(rhs), P(jump)), "rhs")
        out.append((rhs, jump))
    assert out[0][0].abs().max() > 0
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
    gpu.check(lib.alpaca_context_destroy(ctx), "context_destroy")
