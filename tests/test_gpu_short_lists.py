"""Binning of lists short enough for the forms with fewer launches: one count
block storing the offsets itself (at most 4096 items), and sort tiles of 4096
records (up to 128 of them, and 65536 digit counts) whose histograms the
scatter adds up itself; and the sort's 9-bit passes.  Whole numbers: every
list equals the oracle's."""

import numpy as np
import pytest
import torch

from helpers import assert_equal, np32
from oracle import binning

pytestmark = pytest.mark.gpu

from r2splat.cuda import _ops  # noqa: E402

DEV = "cuda:0"


def _compare(lists, tpg, ids, flat, offsets):
    assert_equal(np32(lists.tiles_per_gauss), tpg, "tiles_per_gauss")
    assert_equal(np32(lists.isect_ids), ids, "isect_ids")
    assert_equal(np32(lists.flatten_ids), flat, "flatten_ids")
    assert_equal(np32(lists.tile_offsets), offsets, "tile_offsets")
    emit, src = (np32(t) for t in lists.emission)
    assert_equal(emit, np.repeat(np.arange(tpg.size), tpg.reshape(-1)), "emit_ids")
    assert_equal(emit[src], flat, "emit_ids[isect_src]")
    # Stable: within a key the emission order is kept.
    assert np.all((np.diff(src) > 0) | (np.diff(ids) > 0))


# 64 tiles that every Gaussian overlaps, 64 N records: 4096 and 4097 Gaussians
# stand on either side of the items' limit, 8192 and 8193 (128 and 129 sort
# tiles) of the tiles' limit; the capacity guessed by the second call is an
# eighth and 4096 records above the count.  (32, 32): 1024 digits and 59 sort
# tiles, 67 at the guess, the words' limit between.  (45, 46): 2070 keys, two
# sort passes.
@pytest.mark.parametrize("tiles,n", [((8, 8), 1), ((8, 8), 4096), ((8, 8), 4097), ((8, 8), 7300),
                                     ((8, 8), 8192), ((8, 8), 8193), ((32, 32), 12000),
                                     ((45, 46), 4096), ((1, 1), 700)])
def test_tiles(tiles, n):
    _ops._COUNT_HISTORY.clear()
    tw, th = tiles
    g = torch.Generator().manual_seed(n)
    m2 = (torch.rand(1, n, 2, generator=g) * torch.tensor([16.0 * tw, 16.0 * th])).float()
    full = tw * th == 64
    r = (torch.full((1, n, 2), 200) if full else torch.randint(0, 60, (1, n, 2), generator=g)).int()
    tpg, ids, flat = binning.isect_tiles(m2.numpy(), r.numpy(), 16, tw, th)
    assert not full or ids.size == 64 * n
    offsets = binning.isect_offset_encode(ids, 1, tw, th)
    for _ in range(2):  # the exact capacity, then a guessed one
        for keep in (True, False):
            lists = _ops.bin_tiles_2d(m2.to(DEV), r.to(DEV), 16, tw, th, keep_ids=keep)
            _compare(lists, tpg, ids, flat, offsets)


@pytest.mark.parametrize("bricks,n", [((4, 4, 4), 4096), ((4, 4, 4), 4097), ((13, 13, 13), 4096)])
def test_bricks(bricks, n):
    _ops._COUNT_HISTORY.clear()
    n2, n1, n0 = bricks
    g = torch.Generator().manual_seed(n)
    m3 = (torch.rand(n, 3, generator=g) * torch.tensor([8.0 * n2, 8.0 * n1, 8.0 * n0])).float()
    full = n2 * n1 * n0 == 64
    r = (torch.full((n, 3), 100) if full else torch.randint(0, 20, (n, 3), generator=g)).int()
    tpg, ids, flat = binning.isect_tiles_3d(m3.numpy(), r.numpy(), 8, n2, n1, n0)
    offsets = binning.isect_offset_encode_3d(ids, n2, n1, n0)
    for _ in range(2):
        lists = _ops.bin_tiles_3d(m3.to(DEV), r.to(DEV), 8, n2, n1, n0)
        _compare(lists, tpg, ids, flat, offsets)


# 18-bit keys (two passes of 9 bits) and 25-bit keys (three passes of 9, 9 and
# 7 bits): the 512-digit form of the first, a middle and the last pass.
@pytest.mark.parametrize("bricks", [(64, 64, 40), (512, 256, 160)])
def test_nine_bit_passes(bricks):
    n2, n1, n0 = bricks
    n = 3000
    g = torch.Generator().manual_seed(n0)
    m3 = (torch.rand(n, 3, generator=g) * torch.tensor([8.0 * n2, 8.0 * n1, 8.0 * n0])).float()
    r = torch.randint(0, 20, (n, 3), generator=g).int()
    tpg, ids, flat = binning.isect_tiles_3d(m3.numpy(), r.numpy(), 8, n2, n1, n0)
    offsets = binning.isect_offset_encode_3d(ids, n2, n1, n0)
    for keep in (True, False):
        lists = _ops.bin_tiles_3d(m3.to(DEV), r.to(DEV), 8, n2, n1, n0, keep_ids=keep)
        _compare(lists, tpg, ids, flat, offsets)
