"""Calls of several host threads on one ensemble take effect one after the other:
records read and cancellations made while another thread steps fall between its
calls, so a cancelled case's record counts exactly the steps its blocks took."""
import threading
import time

import pytest

from alpaca_amd import cases, gpu
from alpaca_amd.ensemble import CASE_CANCELLED, Ensemble

pytestmark = pytest.mark.gpu

SIZES = [(2, 3), (3, 2), (1, 4), (2, 2)]
CALLS, PER_CALL = 12, 25


def _desc(nb, prec):
    return gpu.make_desc(2, list(nb), [gpu.BC_PERIODIC] * 2, precision=prec)


@pytest.mark.parametrize("precs", [[gpu.FP64], [gpu.FP64, gpu.MIXED]])
def test_records_and_cancellations_fall_between_steps(precs):
    import torch

    print(f"[ensemble threads] precs={precs}", flush=True)
    ens = Ensemble(2, sum(a * b for a, b in SIZES), len(SIZES), [(gpu.FLUX_HLLC, p) for p in precs])
    specs = [(nb, precs[i % len(precs)], cases.four_quadrant_2d(nb[0], nb[1], seed=i))
             for i, nb in enumerate(SIZES)]
    ids = [ens.add_case(_desc(nb, prec), u, 1e300, 0.4) for nb, prec, u in specs]
    ens.step(1)  # captured
    failed = []

    def stepper():
        try:
            for _ in range(CALLS):
                ens.step(PER_CALL)
        except Exception as err:  # reported by the main thread
            failed.append(err)

    thread = threading.Thread(target=stepper)
    thread.start()
    seen = []
    for cid in ids[1:]:
        time.sleep(0.002)
        ens.cancel_case(cid)
        seen.append([r.steps for r in ens.states()])
    thread.join()
    records = ens.states()
    assert not failed
    for counts in seen:
        assert all((counts[c] - 1) % PER_CALL == 0 for c in ids), counts
    assert records[ids[0]].steps == 1 + CALLS * PER_CALL
    for cid, (nb, prec, u) in zip(ids, specs):
        rec = records[cid]
        assert (rec.steps - 1) % PER_CALL == 0
        assert bool(rec.flags & CASE_CANCELLED) == (cid != ids[0])
        case = gpu.GpuCase(_desc(nb, prec), u, cfl=0.4)
        case.advance(rec.steps)
        want = case.u
        got = ens.case_blocks(cid)
        h = slice(4, 20)
        assert torch.equal(got.reshape(want.shape)[:, :, h, h], want[:, :, h, h])
        assert case.record().time == rec.time
    ens.close()
