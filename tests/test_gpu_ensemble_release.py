"""Cases released and replaced between steps without a wait: the newcomer takes
over the slot and the blocks, and every case's steps equal those it makes
alone, in one class and in two side by side."""
import numpy as np
import pytest

from alpaca_amd import cases, gpu
from alpaca_amd.ensemble import Ensemble

pytestmark = pytest.mark.gpu

SIZES = [(4, 4), (2, 5), (3, 3), (5, 2)]


def _desc(nb, prec):
    return gpu.make_desc(2, list(nb), [gpu.BC_ZERO_GRADIENT] * 2, precision=prec)


def _alone(nb, prec, seed, steps):
    case = gpu.GpuCase(_desc(nb, prec), cases.four_quadrant_2d(nb[0], nb[1], seed=seed), cfl=0.5)
    case.advance(steps)
    return case.u


@pytest.mark.parametrize("precs", [[gpu.FP64], [gpu.FP64, gpu.MIXED]])
def test_released_slots_are_taken_over_in_order(precs):
    import torch

    print(f"[ensemble release] precs={precs}", flush=True)
    blocks = sum(a * b for a, b in SIZES)
    ens = Ensemble(2, blocks, len(SIZES), [(gpu.FLUX_HLLC, p) for p in precs])
    for turn in range(3):
        ids = []
        for i, nb in enumerate(SIZES):
            prec = precs[(i + turn) % len(precs)]
            seed = 10 * turn + i
            ids.append((ens.add_case(_desc(nb, prec), cases.four_quadrant_2d(nb[0], nb[1], seed=seed),
                                     1e300, 0.5), nb, prec, seed))
        ens.step(3)
        ens.step(1)
        # half of the cases are replaced while the steps are queued
        for cid, nb, prec, seed in ids[:2]:
            ens.remove_case(cid)
        late = []
        for k, (_, nb, prec, _) in enumerate(ids[:2]):
            seed = 100 + 10 * turn + k
            late.append((ens.add_case(_desc(nb, prec),
                                      cases.four_quadrant_2d(nb[0], nb[1], seed=seed), 1e300, 0.5),
                         nb, prec, seed))
        ens.step(2)
        records = ens.states()
        for group, steps in ((ids[2:], 6), (late, 2)):
            for cid, nb, prec, seed in group:
                assert records[cid].steps == steps
                got = ens.case_blocks(cid)
                want = _alone(nb, prec, seed, steps)
                h = slice(4, 20)
                assert torch.equal(got.reshape(want.shape)[:, :, h, h], want[:, :, h, h]), (turn, nb)
        for cid, *_ in ids[2:] + late:
            ens.remove_case(cid)
    ens.close()
