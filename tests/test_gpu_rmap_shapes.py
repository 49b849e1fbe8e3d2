"""Region sums and their spreading over the shapes where the kernels' tiles
end: every column count class and its neighbours, more than one block of 64
columns, regions empty, of one vertex, around a tile's length and many tiles
long, and arrays whose base is not 16-byte aligned.  The sums add in
ascending vertex order, so they equal the oracle's bit for bit."""

import numpy as np
import pytest

import oracle as O
from tvb_hpc.hip import RegionMap

pytestmark = pytest.mark.gpu

# vertices per tile are 4096 / (columns rounded up to a power of two, <= 64)
COLS = [(1, 1), (2, 1), (1, 3), (1, 4), (5, 1), (3, 3), (1, 16), (1, 17),
        (3, 11), (1, 63), (2, 32), (5, 13), (1, 128), (3, 65)]


@pytest.mark.parametrize('nvar,P', COLS)
def test_region_sums_at_tile_edges(ctx, nvar, P):
    torch = pytest.importorskip('torch')
    print('columns', nvar, P, flush=True)
    C = nvar * P
    tile = 4096 // min(64, 1 << (C - 1).bit_length())
    size = [0, 1, 2, 3, tile - 1, tile, tile + 1, 2 * tile, 3 * tile - 1, 0,
            3 * tile + 1, 6 * tile + 5, 31, 32, 33, 0]
    rng = np.random.default_rng(C)
    rmap = rng.permutation(np.repeat(np.arange(len(size)), size)
                           ).astype(np.int32)
    node = rng.standard_normal((rmap.size, nvar, P)).astype(np.float32)
    m = RegionMap(rmap, len(size))
    # one float past an aligned base: rows of 4 k columns misaligned too
    flat = torch.zeros(node.size + 1, device='cuda')
    off = flat[1:].view(node.shape)
    off.copy_(torch.from_numpy(node))
    ref = O.rmap_to_avg(rmap, node, len(size))
    for t in (torch.from_numpy(node).cuda(), off):
        assert np.array_equal(m.to_avg(t).cpu().numpy(), ref)
    spread = O.rmap_from_avg(rmap, ref)
    roi = torch.from_numpy(ref).cuda()
    assert np.array_equal(m.from_avg(roi).cpu().numpy(), spread)
    out = torch.full((node.size + 1,), 7.0, device='cuda')
    m.from_avg(roi, out[1:].view(node.shape))
    assert np.array_equal(out[1:].view(node.shape).cpu().numpy(), spread)
    assert float(out[0]) == 7.0
