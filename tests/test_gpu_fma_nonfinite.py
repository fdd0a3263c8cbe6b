"""FP64 with FMA beside a density that is not positive: the face has no
eigensystem, and its flux is zero only if every value of its stencil is finite.
An infinity or a NaN elsewhere in the stencil makes it NaN, so the right-hand
side is finite in the cells where the oracle's is."""
import ctypes

import numpy as np
import pytest

from alpaca_amd import cases, gpu
import oracle_py

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flux", [gpu.FLUX_HLLC, gpu.FLUX_ROE])
@pytest.mark.parametrize("density,value", [(-1.0, np.nan), (-1.0, np.inf), (0.0, np.nan),
                                           (0.0, -np.inf)])
@pytest.mark.parametrize("dim", [2, 3])
def test_rhs_beside_a_nonpositive_density(dim, flux, density, value):
    import torch

    print(f"[fma nonfinite] dim={dim} flux={flux} rho={density} value={value}", flush=True)
    blocks = []
    for axis in range(dim):
        for field in range(dim + 2):
            for offset in (-4, -2, -1, 1, 3, 5):
                blk = cases.random_block(dim, 5 + field, smooth=True)
                at = [11, 9, 10 if dim == 3 else 0]
                blk[(0, *at)] = density
                at[axis] += offset
                blk[(field, *at)] = value
                blocks.append(blk)
    blocks.append(cases.random_block(dim, 3, smooth=True))
    blocks[-1][0, 11, 9, 10 if dim == 3 else 0] = density  # and nothing else
    dev = torch.as_tensor(np.stack(blocks), device="cuda").contiguous()
    rhs = torch.zeros_like(dev)
    desc = gpu.make_desc(dim, [1, 1, 1], [0, 0, 0], flux=flux, precision=gpu.FP64_FMA,
                         cell_size=1.0 / 64)
    gpu.check(gpu.load_library().alpaca_right_hand_side(
        ctypes.byref(desc), len(blocks), ctypes.c_void_p(dev.data_ptr()),
        ctypes.c_void_p(rhs.data_ptr()), gpu._stream_ptr()), "rhs")
    for i, blk in enumerate(blocks):
        got = gpu.from_blocks(rhs[i:i + 1], dim, [1, 1, 1]).cpu().numpy()
        want = oracle_py.block_rhs(dim, flux, 1.4, 0.0, blk, 1.0 / 64).reshape(got.shape)
        assert np.array_equal(np.isfinite(got), np.isfinite(want)), i
