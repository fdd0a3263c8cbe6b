"""2D cases of many blocks, where a workgroup takes two blocks at a time: even
and odd block counts give the oracle's bits in the exact form, and the other
forms stay within their bounds of it."""
import numpy as np
import pytest

from alpaca_amd import gpu
import oracle_py
from test_gpu_launch_shapes import _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb,flux,prec", [
    ((32, 48), gpu.FLUX_HLLC, gpu.FP64), ((41, 39), gpu.FLUX_HLLC, gpu.FP64),
    ((41, 39), gpu.FLUX_ROE, gpu.FP64), ((1, 1537), gpu.FLUX_HLLC, gpu.FP64),
    ((91, 91), gpu.FLUX_HLLC, gpu.FP64_FMA), ((91, 91), gpu.FLUX_HLLC, gpu.MIXED),
    ((64, 128), gpu.FLUX_ROE, gpu.MIXED)])
def test_pairs_match_oracle(nb, flux, prec):
    print(f"[pairs] nb={nb} flux={flux} prec={prec}", flush=True)
    st0 = _state(2, nb, 3 + sum(nb))
    bc = [gpu.BC_SYMMETRY, gpu.BC_PERIODIC]
    case = gpu.GpuCase(gpu.make_desc(2, list(nb), bc, flux=flux, precision=prec), st0, cfl=0.5)
    case.advance(2)
    want, dts, _ = oracle_py.run(2, list(nb), bc, flux, 0.5, 1e300, 2, st0)
    rec = case.record()
    got = case.download().reshape(want.shape)
    assert rec.steps == 2 and rec.flags == 0
    if prec == gpu.FP64:
        assert rec.time == dts[0] + dts[1] and np.array_equal(got, want)
    else:  # FP32 faces: 24 bits over two steps of CFL 0.5; FMA: FP64 rounding
        bound = 1e-5 if prec == gpu.MIXED else 1e-12
        assert np.max(np.abs(got - want)) <= bound * np.max(np.abs(want))
