"""The largest link counts that the multiresolution operators accept: more threads
than one launch can count.  All links but a few are invalid and skipped; the
few, spread over the whole list, give what they give alone."""
import numpy as np
import pytest

from alpaca_amd import multiresolution as mr
import mr_states

pytestmark = pytest.mark.gpu

N = 1 << 24
WHERE = [0, 1917396, 3355443, 9586980, 13421772, N - 1]  # beside the counts of one launch


def _setup(dim):
    import torch

    pairs = [mr_states.pair(dim, "smooth", i % (1 << dim)) for i in range(len(WHERE))]
    pool = torch.as_tensor(np.stack([b for p, c in pairs for b in (p, c)]), device="cuda").contiguous()
    few = torch.as_tensor(mr.make_links([(2 * i + 1, 2 * i, i % (1 << dim), 1)
                                         for i in range(len(WHERE))]), device="cuda")
    many = torch.full((N, 4), -1, dtype=torch.int32, device="cuda")
    at = torch.tensor(WHERE, device="cuda")
    many[at] = few
    return torch, pool, few, many, at


@pytest.mark.parametrize("dim", [2, 3])
def test_prediction_and_jump_halos(dim):
    torch, pool, few, many, at = _setup(dim)
    for rng in ((4, 16) * dim, (0, 24) * dim, (0, 4) * dim, (2, 20) * dim):
        print(f"[many links] dim={dim} prediction {rng}", flush=True)
        want, got = pool.clone(), pool.clone()
        mr.Multiresolution.prediction(want, dim, few, rng)
        mr.Multiresolution.prediction(got, dim, many, rng)
        assert not torch.equal(want, pool)
        assert torch.equal(got, want)
    print(f"[many links] dim={dim} jump halos", flush=True)
    want, got = pool.clone(), pool.clone()
    where = torch.zeros(N, dtype=torch.int32, device="cuda")
    mr.Multiresolution.jump_halo_update(want, dim, few, where[:len(WHERE)].contiguous())
    mr.Multiresolution.jump_halo_update(got, dim, many, where)
    assert not torch.equal(want, pool)
    assert torch.equal(got, want)


@pytest.mark.parametrize("norm", [mr.LINF, mr.L1, mr.L2])
@pytest.mark.parametrize("dim", [2, 3])
def test_details(dim, norm):
    torch, pool, few, many, at = _setup(dim)
    print(f"[many links] dim={dim} details norm={norm}", flush=True)
    op = mr.Multiresolution(mr.ThresholdComputer(dim, 2, 2, 1e-2), norm=norm)
    want, want_decisions = op.child_needs_remeshing(pool, dim, few)
    details, decisions = op.child_needs_remeshing(pool, dim, many)
    assert torch.equal(details[at], want) and torch.equal(decisions[at], want_decisions)
    assert int(torch.isnan(details).sum()) == N - len(WHERE)
    assert int((decisions == -1).sum()) == N - len(WHERE)
