"""3D prediction over ranges whose pairs of parent cells along z do not come
out even, in both window layouts, and over ranges as large as the internal
cells at other places: the oracle's bits."""
import numpy as np
import pytest

from alpaca_amd import multiresolution as mr
import mr_states
import oracle_py as O

pytestmark = pytest.mark.gpu

# (x, y, z) starts and counts: 1, 3, 7, 9 and 11 predicted cells along z, windows
# of at most 12 and of up to 16 cells, and 8 per axis beside the internal cells.
RANGES = [(0, 2, 0, 2, 0, 2), (2, 4, 4, 10, 6, 6), (0, 16, 8, 16, 10, 14), (4, 6, 4, 2, 6, 18),
          (0, 24, 0, 24, 2, 22), (2, 22, 0, 18, 0, 24), (0, 16, 0, 16, 0, 16), (8, 16, 6, 16, 2, 16),
          (4, 16, 4, 16, 4, 16), (0, 24, 0, 24, 0, 24)]


@pytest.mark.parametrize("rng", RANGES)
def test_prediction_3d_of_uneven_ranges(rng):
    import torch

    print(f"[mr shapes] range={rng}", flush=True)
    pairs = [(pos, *mr_states.pair(3, kind, pos)) for pos, kind in
             ((0, "smooth"), (3, "random"), (5, "nonfinite"), (7, "zeros"))]
    host = np.stack([b for _, p, c in pairs for b in (p, c)])
    dev = torch.as_tensor(host, device="cuda").contiguous()
    links = torch.as_tensor(mr.make_links([(2 * i + 1, 2 * i, pos, 1)
                                           for i, (pos, _, _) in enumerate(pairs)]), device="cuda")
    mr.Multiresolution.prediction(dev, 3, links, rng)
    got = dev.cpu().numpy()
    for i, (pos, p, c) in enumerate(pairs):
        want = np.stack([O.mr_prediction(3, p[e], c[e], pos, rng) for e in range(5)])
        assert np.array_equal(got[2 * i + 1], want, equal_nan=True), (rng, pos)
        assert np.array_equal(got[2 * i], p, equal_nan=True)
