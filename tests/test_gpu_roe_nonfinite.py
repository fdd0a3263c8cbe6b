"""Exact flux splitting where a stencil holds infinities or NaN: the products of
the eigenvectors' zero entries, which the kernel otherwise leaves out, make
the oracle's NaN."""
import ctypes

import numpy as np
import pytest

from alpaca_amd import cases, gpu
import oracle_py

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 1e300])
@pytest.mark.parametrize("dim,field", [(d, e) for d in (2, 3) for e in range(d + 2)])
def test_roe_rhs_of_nonfinite_stencils(dim, field, value):
    import torch

    print(f"[roe nonfinite] dim={dim} field={field} value={value}", flush=True)
    blk = cases.random_block(dim, 17 + field, smooth=True)
    # one cell inside, and one in a face halo
    blk[(field, 11, 9, 10 if dim == 3 else 0)] = value
    blk[(field, 2, 14, 12 if dim == 3 else 0)] = value
    dev = torch.as_tensor(blk[None], device="cuda").contiguous()
    rhs = torch.zeros_like(dev)
    desc = gpu.make_desc(dim, [1, 1, 1], [0, 0, 0], flux=gpu.FLUX_ROE, cell_size=1.0 / 64)
    gpu.check(gpu.load_library().alpaca_right_hand_side(
        ctypes.byref(desc), 1, ctypes.c_void_p(dev.data_ptr()), ctypes.c_void_p(rhs.data_ptr()),
        gpu._stream_ptr()), "rhs")
    got = gpu.from_blocks(rhs, dim, [1, 1, 1]).cpu().numpy()
    want = oracle_py.block_rhs(dim, 1, 1.4, 0.0, blk, 1.0 / 64).reshape(got.shape)
    assert np.array_equal(got, want, equal_nan=True)
