"""The boundary-flux save of the 2D right-hand side in every tile shape: a block's
surfaces do not depend on how many blocks a call holds, and the Top and Bottom
surfaces, which have no faces in 2D, receive 0.0 once."""
import ctypes

import numpy as np
import pytest

from alpaca_amd import cases, gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [gpu.FP64, gpu.FP64_FMA, gpu.MIXED])
@pytest.mark.parametrize("flux", [gpu.FLUX_HLLC, gpu.FLUX_ROE])
def test_surfaces_are_the_same_in_every_shape(flux, prec):
    import torch

    lib = gpu.load_library()
    desc = gpu.make_desc(2, [1, 1], [0, 0], flux=flux, precision=prec, cell_size=1.0 / 64)
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    base = torch.as_tensor(np.stack([cases.random_block(2, 21 + s) for s in range(3)]), device="cuda")
    start = torch.as_tensor(np.random.default_rng(4).uniform(-1.0, 1.0, (3, 6, 4, 16)), device="cuda")
    start[:, 4:, :, ::3] = -0.0

    def surfaces(n):
        which = torch.arange(n, device="cuda") % 3
        blocks, jump = base[which].contiguous(), start[which].contiguous()
        rhs = torch.empty_like(blocks)
        gpu.check(lib.alpaca_right_hand_side_jump_fluxes(ctypes.byref(desc), n, P(blocks), P(rhs),
                                                         P(jump), gpu._stream_ptr()), "rhs")
        return jump

    want = surfaces(3)
    assert torch.equal(want[:, 4:], start[:, 4:] + 0.0)
    assert not torch.signbit(want[:, 4:][want[:, 4:] == 0.0]).any()
    assert not torch.equal(want[:, :4], start[:, :4])
    for n in (160, 161, 256, 257, 320, 321, 1151, 1152):
        print(f"[jump 2d] flux={flux} prec={prec} n={n}", flush=True)
        got = surfaces(n)
        assert torch.equal(got, want[torch.arange(n, device="cuda") % 3]), n
        assert not torch.signbit(got[:, 4:][got[:, 4:] == 0.0]).any()
