"""3D refinement on both sides of the link count from which a child row's edges are
read before it is written: a link's child does not depend on the links beside it,
and nothing but its internal cells changes."""
import pytest

from alpaca_amd import multiresolution as mr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1092, 1093, 1208])
def test_refinement_of_many_links(n):
    import torch

    print(f"[mr edges] n={n}", flush=True)
    parents = (n + 7) // 8
    gen = torch.Generator(device="cuda").manual_seed(n)
    pool = torch.rand((parents + n, 5, 24, 24, 24), dtype=torch.float64, device="cuda", generator=gen)
    pool[parents::3] = float("nan")  # what a child held does not matter
    links = torch.as_tensor(mr.make_links([(parents + i, i // 8, i % 8, 1) for i in range(n)]),
                            device="cuda")
    want, got = pool.clone(), pool.clone()
    rng = (4, 16) * 3
    for part in links.split(500):
        mr.Multiresolution.prediction(want, 3, part.contiguous(), rng)
    mr.Multiresolution.prediction(got, 3, links, rng)
    inner = (slice(None), slice(None)) + (slice(4, 20),) * 3
    assert torch.isfinite(got[inner]).all()
    assert torch.equal(got[inner], want[inner])
    got[inner], pool[inner] = 0.0, 0.0
    assert torch.equal(got.nan_to_num(7.0), pool.nan_to_num(7.0))
    assert torch.equal(want[:parents, 0, 0], pool[:parents, 0, 0])
