"""Tile shapes and workgroups per CU changed between steps, of one class and of two,
with fewer and more blocks than the workgroups that a tuning asks for: every case's
steps equal those it makes alone."""
import pytest

from alpaca_amd import cases, gpu
from alpaca_amd.ensemble import Ensemble

pytestmark = pytest.mark.gpu

TUNINGS = [(0, 0), (0, 12), (2, 16), (0, 12), (1, 2), (0, 3)]


@pytest.mark.parametrize("precs", [[gpu.FP64], [gpu.FP64, gpu.MIXED]])
@pytest.mark.parametrize("sizes", [[(3, 2), (1, 5)], [(30, 20), (13, 47)], [(40, 28), (1, 9)]])
def test_tuning_changed_between_steps(precs, sizes):
    import torch

    print(f"[ensemble tuning] precs={precs} sizes={sizes}", flush=True)
    ens = Ensemble(2, sum(a * b for a, b in sizes), len(sizes), [(gpu.FLUX_HLLC, p) for p in precs])
    specs = [(gpu.make_desc(2, list(nb), [gpu.BC_ZERO_GRADIENT] * 2, precision=precs[i % len(precs)]),
              cases.four_quadrant_2d(nb[0], nb[1], seed=i)) for i, nb in enumerate(sizes)]
    ids = [ens.add_case(d, u, 1e300, 0.4) for d, u in specs]
    ens.step(2)
    for tuning in TUNINGS:
        ens.set_tuning(*tuning)
        ens.step(2)
    records = ens.states()
    for cid, (desc, u) in zip(ids, specs):
        case = gpu.GpuCase(desc, u, cfl=0.4)
        case.advance(2 + 2 * len(TUNINGS))
        assert records[cid].steps == 2 + 2 * len(TUNINGS)
        h = slice(4, 20)
        got = ens.case_blocks(cid).reshape(case.u.shape)
        assert torch.equal(got[:, :, h, h], case.u[:, :, h, h])
    ens.close()
