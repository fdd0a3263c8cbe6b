"""Block counts on both sides of every line at which the fused kernels change
their tile shape: the exact stage kernels give the oracle's bits, and the
right-hand side of a block does not depend on how many blocks a call holds."""
import ctypes

import numpy as np
import pytest

from alpaca_amd import cases, gpu
import oracle_py

pytestmark = pytest.mark.gpu

# Blocks per launch, for 256 compute units: (2D) 8x8 tiles up to 160 blocks,
# 16x16 with 640 threads up to 256, 8x8 up to 320, 16x8 up to 1535, then 16x16
# with 128; (3D) lines at 4, 8, 16, 32 and 48 blocks.
COUNTS = {2: [(1, 1), (10, 16), (7, 23), (16, 16), (257, 1), (20, 16), (3, 107), (5, 307), (12, 128)],
          3: [(1, 1, 1), (2, 2, 1), (5, 1, 1), (2, 2, 2), (3, 3, 1), (4, 2, 2), (17, 1, 1), (4, 4, 2),
              (3, 11, 1), (4, 4, 3), (7, 7, 1)]}


@pytest.fixture(scope="module")
def torch():
    import torch as _t
    assert _t.cuda.is_available()
    gpu.load_library()
    return _t


def _state(dim, nb, seed):
    rng = np.random.default_rng(seed)
    n = [16 * m for m in nb]
    x = np.meshgrid(*[np.arange(m) / max(n) for m in n], indexing="ij")
    wave = sum(np.sin(2 * np.pi * (a + 1) * x[a] + rng.uniform(0, 6)) for a in range(dim))
    rho = 1.0 + 0.2 * wave / dim + 0.4 * (x[0] > 0.5 * n[0] / max(n))
    p = 1.0 + 0.3 * (x[-1] > 0.5 * n[-1] / max(n)) + 0.05 * rng.random(n)
    vel = [0.3 * np.cos(2 * np.pi * x[a] + rng.uniform(0, 6)) for a in range(dim)]
    c = cases.primes_to_conservatives(dim, 1.4, 0.0, rho, vel, p)
    return np.ascontiguousarray(c[..., None] if dim == 2 else c)


@pytest.mark.parametrize("flux", [gpu.FLUX_HLLC, gpu.FLUX_ROE])
@pytest.mark.parametrize("dim,nb", [(d, nb) for d in (2, 3) for nb in COUNTS[d]])
def test_stage_matches_oracle_at_every_shape(torch, dim, nb, flux):
    print(f"[shapes stage] dim={dim} nb={nb} flux={flux}", flush=True)
    st0 = _state(dim, nb, 7 + sum(nb))
    bc = [gpu.BC_PERIODIC, gpu.BC_SYMMETRY, gpu.BC_ZERO_GRADIENT][:dim]
    case = gpu.GpuCase(gpu.make_desc(dim, list(nb), bc, flux=flux), st0, cfl=0.5)
    case.advance(2)  # the first step's dt from the signal kernel, the second's from the last stage
    want, dts, t = oracle_py.run(dim, list(nb), bc, flux, 0.5, 1e300, 2, st0)
    rec = case.record()
    assert rec.steps == 2 and rec.flags == 0 and rec.time == dts[0] + dts[1]
    assert np.array_equal(case.download(), want.reshape(case.download().shape))


@pytest.mark.parametrize("flux", [gpu.FLUX_HLLC, gpu.FLUX_ROE])
@pytest.mark.parametrize("prec", [gpu.FP64, gpu.FP64_FMA, gpu.MIXED])
@pytest.mark.parametrize("dim", [2, 3])
def test_rhs_of_a_block_is_the_same_in_every_shape(torch, dim, prec, flux):
    lib = gpu.load_library()
    desc = gpu.make_desc(dim, [1, 1, 1], [0, 0, 0], flux=flux, precision=prec, cell_size=1.0 / 64)
    P = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    base = torch.as_tensor(np.stack([cases.random_block(dim, 11 + s, smooth=s == 1)
                                     for s in range(3)]), device="cuda")
    counts = [int(np.prod(nb)) for nb in COUNTS[dim]]
    want = None
    for n in sorted(counts):
        print(f"[shapes rhs] dim={dim} prec={prec} flux={flux} n={n}", flush=True)
        blocks = base[torch.arange(n, device="cuda") % 3].contiguous()
        rhs = torch.full_like(blocks, np.nan)
        gpu.check(lib.alpaca_right_hand_side(ctypes.byref(desc), n, P(blocks), P(rhs),
                                             gpu._stream_ptr()), "rhs")
        if want is None:  # one block: the others from calls of one block each
            want = torch.full_like(base, np.nan)
            for s in range(3):
                gpu.check(lib.alpaca_right_hand_side(ctypes.byref(desc), 1, P(base[s]), P(want[s]),
                                                     gpu._stream_ptr()), "rhs")
        assert torch.equal(rhs, want[torch.arange(n, device="cuda") % 3]), f"n={n}"
