"""The backward blocks that stage their tiles' (bricks') upstream gradient in
LDS, beside those whose records span too many tiles for it, on ragged and
whole images (volumes), and the voxel forward that walks every row of large
footprints: against the oracle at the usual bar (tests/helpers.py)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import (assert_close, check_raster, check_voxel, np32, raster_references,
                     voxel_references)
from oracle import ops
from r2splat.cuda import _ops
from r2splat.cuda import _wrapper as W
from test_gpu_ops import DEV, _prepared, _raster_case, _voxel_case

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


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("two_pass", [True, False])
@pytest.mark.parametrize("ts", [8, 16])
@pytest.mark.parametrize("n,shape,views", [(40, (64, 44), 1), (40, (64, 44), 2),
                                           (60, (336, 204), 1), (60, (336, 204), 2)])
def test_raster_backward_ragged_bottom(n, shape, views, ts, two_pass, dtype):
    """Rows that a 16-byte load fits, no ragged column, a ragged last tile row, and lists too
    sparse to stage: waves of whole and ragged tiles side by side, with footprints that cross
    the image's bottom edge."""
    W_img, H_img = shape
    d, m2, con, mu, op, ids, fl, off = _raster_case(n, 5, W_img, H_img, ts, views, dtype,
                                                    log_mu=-2.6 if W_img == 64 else -3.0)
    tw, th = W_img // ts, -(-H_img // ts)
    assert W_img % ts == 0 and H_img % ts != 0
    bottom = ids % (tw * th) // tw == th - 1
    assert any(b.any() and not b.all() for b in bottom.split(64))
    assert int(ids[:256].max() - ids[:256].min()) >= 4
    if not two_pass:
        fl = fl.clone()
    assert (_ops.emission_order(fl, off.numel()) is not None) == two_pass
    v = torch.randn((views, H_img, W_img), generator=d["gen"], dtype=dtype)
    for absgrad in (True, False):
        refs = raster_references(np32(m2), np32(con), np32(op), np32(mu), np32(off), np32(fl),
                                 W_img, H_img, ts, v_image=v.numpy(), absgrad=absgrad)
        got = W.rasterize_to_pixels_bwd_per_gaussian(m2, con, op, mu, off, ids, fl, v.to(DEV),
                                                     W_img, H_img, ts, absgrad)
        for name, r in check_raster(refs, grads=[None if t is None else np32(t)
                                                 for t in got]).items():
            print(absgrad, name, r)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,dims,log_mu,staged", [
    (2500, (30, 20, 26), -3.2, True),   # ragged
    (2500, (29, 21, 9), -1.6, True),    # ragged, waves that walk every row
    (60, (90, 61, 77), -3.4, False),    # ragged, sparse bricks
    (60, (96, 64, 80), -3.4, False),    # whole, sparse bricks
    (5, (7, 3, 5), -3.2, True),         # one partial brick
])
def test_voxel_backward_blocks(dtype, n, dims, log_mu, staged):
    d, m3, con, ids, fl, off = _voxel_case(n, 4, dims, 8, dtype, log_mu=log_mu)
    blocks = [int(b.max() - b.min()) + 1 for b in ids.split(256)]
    assert (min(blocks) <= 6) == staged, blocks
    op = d["opac"]
    vol = W.voxelize_to_voxels_fwd(m3, con, op, off, fl, *dims, 8)
    v = torch.randn(vol.shape, generator=d["gen"], dtype=dtype)
    refs = voxel_references(np32(m3), np32(con), np32(op), np32(off), np32(fl), *dims, 8,
                            v_volume=v.numpy())
    print("volume", check_voxel(refs, volume=np32(vol)))
    vol_r, reach = _ops.voxelize_with_reach(m3, con, op, off, fl, *dims)
    assert torch.equal(vol, vol_r)
    plain = W.voxelize_to_voxels_bwd_per_gaussian(m3, con, op, off, ids, fl, v.to(DEV), *dims, 8)
    for name, r in check_voxel(refs, grads=[np32(t) for t in plain]).items():
        print(name, r)
    n2, n1, n0 = (-(-x // 8) for x in dims)
    lists = _ops.TileLists(None, ids, fl, *_ops.emission_order(fl, n2 * n1 * n0), off)
    given = _ops.voxel_backward(m3, con, op, off, lists, v.to(DEV), *dims, 8, reach=reach)
    for a, b in zip(plain, given):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n,dims,dtype", [
    (n, dims, dtype) for dims in ((90, 61, 77), (92, 61, 77), (96, 61, 80), (96, 64, 80))
    for n, dtype in ((0, torch.float32), (0, torch.float64),
                     (66_000 if dims == (96, 64, 80) else 42_000,
                      torch.float64 if dims == (92, 61, 77) else torch.float32))])
def test_voxel_backward_full_chunk_lists(n, dims, dtype):
    """A few Gaussians that cover the whole volume: records that reach every row, in blocks over
    too many bricks to stage, of bricks that cannot be read whole (ragged, or rows that no
    16-byte load fits) and of whole ones.  n: small Gaussians that crowd a corner beside them,
    whose records make the list one that stages where it can; the rest takes the same kernel's
    longest chunk lists."""
    n2, n1, n0 = (-(-x // 8) for x in dims)
    d = _prepared(5 + n, 8, dtype, log_mu=-0.7)
    small = ops.parameter_transform_fwd(
        d["raw"].quats.double().numpy(), np.full((5 + n, 3), -7.0), 5e-4, 1.0)[0]
    d["covars"][5:] = torch.as_tensor(small, dtype=dtype, device=DEV)[5:]
    d["means"][5:] = 0.01 * d["means"][5:] - 0.94
    ranges, centers = (torch.full((3,), x, dtype=dtype, device=DEV) for x in (2.0, 0.0))
    m3, con, r3 = W.world_to_volume_mapping_fwd(d["means"], d["covars"], d["opac"], ranges,
                                                centers, *dims, 1e-8, 3.0)
    _, ids, fl = W.isect_tiles_3d(m3, r3, 8, n2, n1, n0)
    off = W.isect_offset_encode_3d(ids, n2, n1, n0)
    whole = all(x % 8 == 0 for x in dims)
    assert (ids.numel() >= (65536 if whole else 256 * off.numel() / 6)) == (n > 0)
    spans = np.array([int(b.max() - b.min()) + 1 for b in ids.split(256)[:-1]])
    assert spans.max() > 6 and (spans.min() <= 6) == (n > 0)
    op = d["opac"]
    _, reach = _ops.voxelize_with_reach(m3, con, op, off, fl, *dims)
    rows = np.array([bin(int(x)).count("1") for x in reach.cpu().numpy().view(np.uint64)])
    chunks = np.add.reduceat(-(-rows // 8), np.arange(0, rows.size, 64))
    assert chunks[np.repeat(spans > 6, 4)[:chunks.size].nonzero()].max() > 448, chunks
    v = torch.randn((dims[2], dims[1], dims[0]), generator=d["gen"], dtype=dtype)
    refs = voxel_references(np32(m3), np32(con), np32(op), np32(off), np32(fl), *dims, 8,
                            v_volume=v.numpy())
    plain = W.voxelize_to_voxels_bwd_per_gaussian(m3, con, op, off, ids, fl, v.to(DEV), *dims, 8)
    for name, r in check_voxel(refs, grads=[np32(t) for t in plain]).items():
        print(name, r)
    lists = _ops.TileLists(None, ids, fl, *_ops.emission_order(fl, off.numel()), off)
    given = _ops.voxel_backward(m3, con, op, off, lists, v.to(DEV), *dims, 8, reach=reach)
    for a, b in zip(plain, given):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dims,dtype", [((80, 72, 72), torch.float32),
                                        ((69, 64, 70), torch.float32),
                                        ((69, 64, 70), torch.float64)])
def test_voxel_backward_of_records_that_reach_nothing(dims, dtype):
    """Lists that name mostly Gaussians of other bricks, as long thin Gaussians' boxes do: blocks
    in which no record reaches a row, and blocks over too many bricks to stage whose reaching
    records lie in few; with and without the forward's reach masks."""
    n2, n1, n0 = (-(-x // 8) for x in dims)
    keys = n0 * n1 * n2
    d = _prepared(400, 8, dtype, log_mu=-4.5)
    d["means"][:, 0] = 0.5 * d["means"][:, 0] - 0.5  # in one half of the volume
    ranges, centers = (torch.full((3,), x, dtype=dtype, device=DEV) for x in (2.0, 0.0))
    m3, con, r3 = W.world_to_volume_mapping_fwd(d["means"], d["covars"], d["opac"], ranges,
                                                centers, *dims, 1e-8, 3.0)
    rng = np.random.default_rng(3)
    count = np.where(np.arange(keys) % 12 < 10, 25, 400)
    fl = np.concatenate([np.sort(rng.choice(400, c, replace=False)) for c in count])
    ids = torch.as_tensor(np.repeat(np.arange(keys), count), device=DEV)
    off = torch.as_tensor((np.cumsum(count) - count).astype(np.int32), device=DEV)
    off = off.reshape(n0, n1, n2)
    order = np.argsort(fl, kind="stable")  # Gaussian by Gaussian, as the records are emitted
    src = np.empty(fl.size, np.int32)
    src[order] = np.arange(fl.size)
    emit, src, fl = (torch.as_tensor(a.astype(np.int32), device=DEV) for a in (fl[order], src, fl))
    op = d["opac"]
    _, reach = _ops.voxelize_with_reach(m3, con, op, off, fl, *dims)
    hit = reach.cpu().numpy() != 0
    span = {True: 0, False: 0}
    empty = 0
    for h, k in zip(np.split(hit, range(256, hit.size, 256)),
                    np.split(ids.cpu().numpy(), range(256, hit.size, 256))):
        empty += not h.any()
        if h.any():
            span[np.ptp(k) >= 6 and np.ptp(k[h]) < 6] += 1
    assert empty > 5 and span[True] > 5 and span[False] > 5, (empty, span)
    whole = all(x % 8 == 0 for x in dims)
    assert hit.size >= (max(65536, 64 * keys) if whole else 256 * keys / 6)  # lists that stage
    v = torch.randn((dims[2], dims[1], dims[0]), generator=d["gen"], dtype=dtype)
    refs = voxel_references(np32(m3), np32(con), np32(op), np32(off), np32(fl), *dims, 8,
                            v_volume=v.numpy())
    lists = _ops.TileLists(None, ids, fl, emit, src, off)
    plain, given = (_ops.voxel_backward(m3, con, op, off, lists, v.to(DEV), *dims, 8, **k)
                    for k in ({}, {"reach": reach}))
    for name, r in check_voxel(refs, grads=[np32(t) for t in plain]).items():
        print(name, r)
    for a, b in zip(plain, given):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("dims", [(64, 64, 64), (40, 37, 33), (20, 17, 18)])
@pytest.mark.parametrize("order", ["large first", "small first", "mixed"])
def test_voxel_forward_over_batches_of_both_kinds(order, dims, dtype):
    """Large Gaussians and small ones in one list: waves that walk every row of one batch and
    each row's own set of the next, with one, two and four waves a brick.  The volume is the
    oracle's, and the same bit for bit where every batch's masks are formed."""
    n = 1500
    d = _prepared(2 * n, 13, dtype, log_mu=-1.0)
    small = ops.parameter_transform_fwd(d["raw"].quats.double().numpy(),
                                        np.full((2 * n, 3), -3.5), 5e-4, 1.0)[0]
    at = torch.arange(2 * n, device=DEV)
    large = {"large first": at < 300, "small first": at >= 2 * n - 300,
             "mixed": at // 100 % 10 == 0}[order]
    covars = torch.where(large[:, None], d["covars"], torch.as_tensor(small, dtype=dtype).to(DEV))
    ranges, centers = (torch.full((3,), x, dtype=dtype, device=DEV) for x in (2.0, 0.0))
    m3, con, r3 = W.world_to_volume_mapping_fwd(d["means"], covars, d["opac"], ranges, centers,
                                                *dims, 1e-8, 3.0)
    grid = [-(-x // 8) for x in dims]
    _, ids, fl = W.isect_tiles_3d(m3, r3, 8, *grid)
    off = W.isect_offset_encode_3d(ids, *grid)
    vol = W.voxelize_to_voxels_fwd(m3, con, d["opac"], off, fl, *dims, 8)
    vol_r, reach = _ops.voxelize_with_reach(m3, con, d["opac"], off, fl, *dims)
    assert torch.equal(vol, vol_r)
    rows = np.array([bin(int(x)).count("1") for x in reach.cpu().numpy().view(np.uint64)])
    dense = np.add.reduceat(rows, np.arange(0, rows.size, 64)) >= 48 * 64
    assert dense.any() and not dense.all()
    refs = voxel_references(np32(m3), np32(con), np32(d["opac"]), np32(off), np32(fl), *dims, 8)
    print(fl.numel() // off.numel(), dense.mean(), check_voxel(refs, volume=np32(vol)))


@pytest.mark.parametrize("first", [1, 100, 700])
def test_offsets_that_start_after_the_first_record(first):
    """Records before a caller's first tile (brick) offset have no key to be found: they count
    to key 0, as when the keys are given."""
    d, m2, con, mu, op, ids, fl, off = _raster_case(4000, 9, 160, 144, 16)
    assert off.numel() > 64 and fl.numel() > 1000
    off, ids = off.clamp(min=first), torch.where(torch.arange(ids.numel(), device=DEV) < first, 0,
                                                 ids)
    v = torch.randn((1, 144, 160), generator=d["gen"]).to(DEV)
    for absgrad in (True, False):
        got = W.rasterize_to_pixels_bwd(m2, con, op, mu, off, fl, v, 160, 144, 16, absgrad)
        want = W.rasterize_to_pixels_bwd_per_gaussian(m2, con, op, mu, off, ids, fl, v, 160, 144,
                                                      16, absgrad)
        for a, b in zip(got[not absgrad:], want[not absgrad:]):
            assert torch.equal(a, b)
    dims = (40, 36, 32)
    d, m3, con, ids, fl, off = _voxel_case(3000, 10, dims, 8)
    assert off.numel() > 64 and fl.numel() > 1000
    off, ids = off.clamp(min=first), torch.where(torch.arange(ids.numel(), device=DEV) < first, 0,
                                                 ids)
    v = torch.randn(dims[::-1], generator=d["gen"]).to(DEV)
    got = W.voxelize_to_voxels_bwd(m3, con, d["opac"], off, fl, v, *dims, 8)
    want = W.voxelize_to_voxels_bwd_per_gaussian(m3, con, d["opac"], off, ids, fl, v, *dims, 8)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("ts", [4, 8, 10])
def test_brick_grid_larger_than_the_volume(ts):
    """Bricks of a caller's grid that lie beyond the volume hold no voxel: the volume and the
    gradients are those of the exact grid."""
    dims = (30, 20, 26)
    n2, n1, n0 = (-(-x // ts) for x in dims)
    d, m3, con, _, _, _ = _voxel_case(1500, 12, dims, ts)
    v = torch.randn(dims[::-1], generator=d["gen"]).to(DEV)
    # Radii that take in every brick.
    r3 = torch.full((m3.shape[0], 3), 200, dtype=torch.int32, device=DEV)
    outs = []
    for e2, e1, e0 in ((0, 0, 0), (2, 1, 2)):
        grid = (n2 + e2, n1 + e1, n0 + e0)
        _, ids, fl = W.isect_tiles_3d(m3, r3, ts, *grid)
        off = W.isect_offset_encode_3d(ids, *grid)
        assert off[-1, -1, -1] < fl.numel()
        outs.append([W.voxelize_to_voxels_fwd(m3, con, d["opac"], off, fl, *dims, ts),
                     *W.voxelize_to_voxels_bwd_per_gaussian(m3, con, d["opac"], off, ids, fl, v,
                                                            *dims, ts)])
    want, got = outs
    # Sums of the same terms: in other waves and orders, 1e-5 of the largest is their rounding.
    for name, a, b in zip(("volume", "v_means3d", "v_conics", "v_opacities"), got, want):
        assert_close(np32(a), np32(b), name, rtol=1e-5, atol=1e-5 * float(b.abs().max()))


@pytest.mark.parametrize("dims", [(30, 20, 26), (32, 24, 32)])
def test_non_finite_record_in_a_ragged_brick(dims):
    """A record with a non-finite conic passes the alpha test wherever its sigma is NaN or
    infinite: its own gradients are those of the one-pass kernel (NaN where they are), and
    no other Gaussian's change."""
    d, m3, con, ids, fl, off = _voxel_case(400, 6, dims, 8)
    op, bad = d["opac"], int(fl[fl.numel() // 2])
    v = torch.randn((dims[2], dims[1], dims[0]), generator=d["gen"]).to(DEV)
    clean = W.voxelize_to_voxels_bwd_per_gaussian(m3, con, op, off, ids, fl, v, *dims, 8)
    con2 = con.clone()
    con2[bad, 3] = float("inf")
    got = W.voxelize_to_voxels_bwd_per_gaussian(m3, con2, op, off, ids, fl, v, *dims, 8)
    one_pass = W.voxelize_to_voxels_bwd_per_gaussian(m3, con2, op, off, ids, fl.clone(), v, *dims,
                                                     8)
    others = torch.arange(m3.shape[0], device=DEV) != bad
    for a, b, c in zip(got, clean, one_pass):
        assert torch.equal(a[others], b[others])
        assert torch.equal(torch.isnan(a[bad]), torch.isnan(c[bad]))


@pytest.mark.parametrize("absgrad", [True, False])
@pytest.mark.parametrize("beside", [True, False])
def test_raster_backward_sums_lose_nothing_to_the_split_row(beside, absgrad):
    """The half rows of a tile are summed apart and then added: the rounding error of the sums
    over a tile is no larger than row by row.  The conics are powers of two so flat that every
    weight is the upstream gradient itself, so float64 gives the sums exactly and what is left is
    the order's rounding (of 40960 records).  Measured: halves apart 0.82-0.89 of row by row,
    halves in one chain 1.01-1.05 already in the signed sums.  beside: means beside the tile,
    where the absolute sums take the signed form."""
    f, per, tw = np.float32, 40, 32
    rng = np.random.default_rng(5)
    n, flat = per * tw * tw, 2.0 ** -44
    tile = np.arange(n) // per
    lo, hi = (-40, -2) if beside else (2, 14)
    rel = rng.uniform(lo, hi, (n, 2)).astype(f)  # from the tile's corner
    corner = np.stack([tile % tw, tile // tw], 1) * 16
    m2 = (corner + rel).astype(f)
    v = rng.standard_normal((16 * tw, 16 * tw)).astype(f)
    to = lambda a: torch.as_tensor(a).to(DEV)  # noqa: E731
    con = to(np.tile(np.array([flat, 0, flat], f), (1, n, 1)))
    one, ar = torch.ones(1, n, device=DEV), torch.arange(n, device=DEV, dtype=torch.int32)
    off = torch.arange(0, n, per, device=DEV, dtype=torch.int32).reshape(1, tw, tw)
    lists = _ops.TileLists(None, to(tile.astype(np.int64)), ar, ar, ar, off)
    v_abs, v_xy = _ops.raster_backward(to(m2)[None], con, one, one, off, lists, to(v)[None],
                                       16 * tw, 16 * tw, 16, absgrad)[:2]
    w = v.reshape(tw, 16, tw, 16).transpose(0, 2, 1, 3).reshape(-1, 16, 16)[tile]
    centre = corner[:, :, None] + np.arange(16) + 0.5
    d = (centre - m2[:, :, None].astype(np.float64))
    d32 = centre.astype(f) - m2[:, :, None]

    def by_rows(x):  # float32, column after column, row after row
        return np.add.accumulate(np.add.accumulate(x, axis=2)[:, :, -1], axis=1)[:, -1]

    def rms(x):
        return np.sqrt(np.mean(np.square(x, dtype=np.float64)))

    want = (w.astype(np.float64).sum(2) * d[:, 1]).sum(1)
    rows = np.add.accumulate(np.add.accumulate(w, axis=2)[:, :, -1] * d32[:, 1], axis=1)[:, -1]
    got = v_xy[0, :, 1].double().cpu().numpy() / flat
    print("signed", rms(got - want) / rms(rows - want))
    assert rms(got - want) <= rms(rows - want)
    if absgrad:
        want = (np.abs(w).astype(np.float64).sum(1) * np.abs(d[:, 0])).sum(1)
        rows = by_rows(np.abs(w) * np.abs(d32[:, 0])[:, None, :])
        got = v_abs[0, :, 0].double().cpu().numpy() / flat
        print("absolute", rms(got - want) / rms(rows - want))
        assert rms(got - want) <= rms(rows - want)
