"""3D cases on both sides of the block counts at which a case marches plane by plane (on
256 compute units: exact 256 and 353 to 384 blocks but not 257 to 352 nor 385, flux
splitting with FMA from 353, HLLC with FMA from 2048), with every kind of side and on uneven grids, one block thick among them: the
exact forms give the oracle's bits, the others stay near them."""
import numpy as np
import pytest

from alpaca_amd import gpu
import oracle_py
from test_gpu_launch_shapes import _state

pytestmark = pytest.mark.gpu

SIDES = {"psz": [gpu.BC_PERIODIC, gpu.BC_SYMMETRY, gpu.BC_ZERO_GRADIENT],
         "zps": [gpu.BC_ZERO_GRADIENT, gpu.BC_PERIODIC, gpu.BC_SYMMETRY],
         "szz": [gpu.BC_SYMMETRY, gpu.BC_ZERO_GRADIENT, gpu.BC_ZERO_GRADIENT]}


def _advance(nb, bc, flux, prec, st0):
    case = gpu.GpuCase(gpu.make_desc(3, list(nb), SIDES[bc], flux=flux, precision=prec), st0, cfl=0.5)
    case.advance(2)
    rec = case.record()
    assert rec.steps == 2 and rec.flags == 0
    return case, rec


# 100 blocks on tiles, 256, 355 and 360 marching (355: 710 slabs, not a multiple of the
# 8 XCDs), 385 on tiles again.
@pytest.mark.parametrize("flux", [gpu.FLUX_HLLC, gpu.FLUX_ROE])
@pytest.mark.parametrize("nb,bc", [((5, 5, 4), "psz"), ((8, 4, 8), "zps"), ((5, 71, 1), "szz"),
                                   ((1, 5, 71), "psz"), ((9, 1, 40), "zps"), ((7, 5, 11), "szz")])
def test_exact_forms_match_oracle(nb, bc, flux):
    print(f"[march] nb={nb} bc={bc} flux={flux}", flush=True)
    st0 = _state(3, nb, 5 + sum(nb))
    case, rec = _advance(nb, bc, flux, gpu.FP64, st0)
    want, dts, _ = oracle_py.run(3, list(nb), SIDES[bc], flux, 0.5, 1e300, 2, st0)
    assert rec.time == dts[0] + dts[1]
    assert np.array_equal(case.download(), want.reshape(case.download().shape))


@pytest.mark.parametrize("nb,bc,flux", [((8, 4, 8), "psz", gpu.FLUX_ROE), ((5, 71, 1), "szz", gpu.FLUX_ROE),
                                        ((8, 6, 8), "zps", gpu.FLUX_ROE),
                                        ((16, 8, 16), "psz", gpu.FLUX_HLLC),
                                        ((13, 158, 1), "zps", gpu.FLUX_HLLC),
                                        ((1, 23, 91), "szz", gpu.FLUX_HLLC)])
def test_fma_forms_near_the_exact_form(nb, bc, flux):
    print(f"[march fma] nb={nb} bc={bc} flux={flux}", flush=True)
    st0 = _state(3, nb, 9 + sum(nb))
    exact, _ = _advance(nb, bc, flux, gpu.FP64, st0)
    fma, _ = _advance(nb, bc, flux, gpu.FP64_FMA, st0)
    # FP64 rounding over two steps, as for the other shapes.
    assert (fma.u - exact.u).abs().max() <= 1e-12 * exact.u.abs().max()


@pytest.mark.parametrize("nb,flux", [((36, 47), gpu.FLUX_ROE), ((41, 61), gpu.FLUX_ROE)])
def test_pairs_with_fma_near_the_exact_form(nb, flux):
    print(f"[pairs fma] nb={nb} flux={flux}", flush=True)
    st0 = _state(2, nb, 2 + sum(nb))
    bc = [gpu.BC_SYMMETRY, gpu.BC_PERIODIC]
    out = []
    for prec in (gpu.FP64, gpu.FP64_FMA):
        case = gpu.GpuCase(gpu.make_desc(2, list(nb), bc, flux=flux, precision=prec), st0, cfl=0.5)
        case.advance(2)
        assert case.record().steps == 2 and case.record().flags == 0
        out.append(case.u)
    assert (out[0] - out[1]).abs().max() <= 1e-12 * out[0].abs().max()
    # the even and odd block counts of the pairs in the exact form
    want, _, _ = oracle_py.run(2, list(nb), bc, flux, 0.5, 1e300, 2, st0)
    got = gpu.from_blocks(out[0], 2, list(nb) + [1]).cpu().numpy()
    assert np.array_equal(got.reshape(want.shape), want)


# 2D blocks beside the line between 16x8 and 16x16 tiles.
@pytest.mark.parametrize("flux", [gpu.FLUX_HLLC, gpu.FLUX_ROE])
@pytest.mark.parametrize("nb", [(1151, 1), (32, 36)])
def test_2d_tiles_match_oracle(nb, flux):
    print(f"[2d tiles] nb={nb} flux={flux}", flush=True)
    st0 = _state(2, nb, 3 + sum(nb))
    bc = [gpu.BC_PERIODIC, gpu.BC_ZERO_GRADIENT]
    case = gpu.GpuCase(gpu.make_desc(2, list(nb), bc, flux=flux), st0, cfl=0.5)
    case.advance(2)
    want, _, _ = oracle_py.run(2, list(nb), bc, flux, 0.5, 1e300, 2, st0)
    assert np.array_equal(case.download().reshape(want.shape), want)
