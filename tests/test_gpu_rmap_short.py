"""Region sums of many short regions (a wave per region and 64 columns): equal
to the oracle's bit for bit for regions of none, one and around 32 vertices,
every column class, more than one block of columns, and a base that is not
16-byte aligned."""

import numpy as np
import pytest

import oracle as O
from tvb_hpc.hip import RegionMap

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('nvar,P', [(1, 1), (2, 1), (6, 2), (1, 63), (1, 64),
                                    (5, 13), (2, 64), (3, 65)])
def test_region_sums_of_short_regions(ctx, nvar, P):
    torch = pytest.importorskip('torch')
    print('columns', nvar, P, flush=True)
    rng = np.random.default_rng(nvar * P)
    size = np.resize([0, 1, 2, 31, 32, 33, 64, 65, 5, 0, 7], 400)
    rmap = rng.permutation(np.repeat(np.arange(400), size)).astype(np.int32)
    node = rng.standard_normal((rmap.size, nvar, P)).astype(np.float32)
    m = RegionMap(rmap, 400)
    ref = O.rmap_to_avg(rmap, node, 400)
    flat = torch.zeros(node.size + 1, device='cuda')
    off = flat[1:].view(node.shape)
    off.copy_(torch.from_numpy(node))
    for t in (torch.from_numpy(node).cuda(), off):
        assert np.array_equal(m.to_avg(t).cpu().numpy(), ref)
