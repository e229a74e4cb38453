"""The backward blocks that stage their tiles' upstream gradient in LDS, beside
those whose records span too many tiles for it, on ragged and whole images:
against the oracle at the usual bar (tests/helpers.py)."""

from __future__ import annotations

import pytest
import torch

from helpers import check_raster, np32, raster_references
from r2splat.cuda import _wrapper as W
from test_gpu_ops import DEV, _raster_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,shape,views,staged", [
    (4000, (70, 45), 1, True),      # ragged, several blocks per tile
    (4000, (64, 48), 2, True),      # whole, blocks across a view's end
    (60, (333, 217), 2, False),     # ragged rows that no 16-byte load fits, sparse tiles
    (60, (336, 208), 1, False),     # whole, sparse tiles
    (7, (17, 15), 1, True),         # one partial wave, partial tiles
])
def test_raster_backward_blocks(dtype, n, shape, views, staged):
    W_img, H_img = shape
    d, m2, con, mu, op, ids, fl, off = _raster_case(n, 3, W_img, H_img, 16, views, dtype,
                                                    log_mu=-3.6 if staged else -3.0)
    # Tiles per block of 256 consecutive records.
    blocks = [int(b.max() - b.min()) + 1 for b in ids.split(256)]
    assert (max(blocks) <= 4) if n == 7 else (min(blocks) <= 4) == staged, blocks
    v = torch.randn((views, H_img, W_img), generator=d["gen"], dtype=dtype)
    refs = raster_references(np32(m2), np32(con), np32(op), np32(mu), np32(off), np32(fl), W_img,
                             H_img, 16, v_image=v.numpy())
    got = W.rasterize_to_pixels_bwd_per_gaussian(m2, con, op, mu, off, ids, fl, v.to(DEV), W_img,
                                                 H_img, 16, True)
    for name, r in check_raster(refs, grads=[np32(t) for t in got]).items():
        print(name, r)
