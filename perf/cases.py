"""Workloads of the r2splat Gaussian backend, for timing and for checking.

Each case is one call that a program built on this framework makes through
its public entry points, on inputs made from a seed:

* ``project``  a training projection: activate the parameters, rasterize one
  or more cone-beam views, map an image gradient back to the parameters;
* ``render``   forward-only projections of a prepared scene (evaluation);
* ``step``     a whole training step: projection, a regularised (sub-)volume,
  the trainer's loss, the explicit backward and the Adam step;
* ``voxels``   voxelization forward and backward through the operators;
* ``volume``   forward-only voxelization of a prepared scene (export);
* ``loss``     the projection and total-variation losses and their gradients;
* ``refine``   a densify split and a prune of the whole model table.

``exact`` restates all of them in plain float64 torch.
"""

from __future__ import annotations

import math
import os
import sys
from types import SimpleNamespace

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "bt-3dgs_amd"))

from r2splat import geometry, optim, scenes  # noqa: E402
from r2splat.cuda import _wrapper as W  # noqa: E402
from r2splat.ops import densify, direct, explicit, loss  # noqa: E402

DEV = "cuda"
SMIN, SMAX = scenes.SCALE_MIN, scenes.SCALE_MAX
# The operating point of every configuration: tile 16, brick 8, blur 1e-8,
# three sigmas, absolute gradients on.
TILE, BRICK, EPS, CLIP = 16, 8, 1e-8, 3.0
THR_2D, THR_3D = 1e-5, 1e-6
LRS = {"means": 6.0e-4, "scales": 4.0e-3, "quats": 3.0e-4, "opacities": 1.0e-2}
LOSS_WEIGHTS = (1.0, 0.25, 1.0, 0.05, 0.05)  # l1, ssim, edge, tv, hierarchy
KEYS = ("means", "scales", "quats", "opacities")
# Sums of more (pixel | voxel, record) pairs than this have no float64 value here.
MAX_EXACT_PAIRS = 1.5e10


# ------------------------------------------------------------------ cases --


def listed():
    return [
        # A first fit or a unit test: few Gaussians, a small detector. The call is launches.
        {"name": "project_4k_64", "kind": "project", "scene": "random", "n": 4096,
         "width": 64, "height": 64, "views": 1},
        # One view of a mid-sized scan, the ordinary training projection.
        {"name": "project_50k_256", "kind": "project", "scene": "random", "n": 50_000,
         "width": 256, "height": 256, "views": 1},
        # A grown tree on a full detector: the projection late in training.
        {"name": "project_tree_500k_512", "kind": "project", "scene": "tree", "n": 500_000,
         "width": 512, "height": 512, "views": 1},
        # The largest projection: two million small Gaussians on a large detector.
        {"name": "project_dense_2m_1024", "kind": "project", "scene": "dense",
         "n": 2_000_000, "width": 1024, "height": 1024, "views": 1},
        # Evaluation: several views in one call, a detector that no tile divides.
        {"name": "render_50k_9x333x217", "kind": "render", "scene": "random", "n": 50_000,
         "width": 333, "height": 217, "views": 9},
        # Early training: a young tree of large leaves, a sampled 32^3 sub-volume for TV.
        {"name": "step_tree_2k_512_tv32", "kind": "step", "scene": "tree", "n": 2048,
         "width": 512, "height": 512, "dim": 32, "extent": 0.25},
        # Late training: the whole step of the 500k tree with a 128^3 volume.
        {"name": "step_tree_500k_512_tv128", "kind": "step", "scene": "tree", "n": 500_000,
         "width": 512, "height": 512, "dim": 128, "extent": 2.0},
        # Volume fitting through the operators, forward and backward.
        {"name": "voxels_200k_256", "kind": "voxels", "scene": "fine", "n": 200_000,
         "d2": 256, "d1": 256, "d0": 256},
        # The largest volume, of the same two million.
        {"name": "voxels_dense_2m_512", "kind": "voxels", "scene": "dense",
         "n": 2_000_000, "d2": 512, "d1": 512, "d0": 512},
        # Export of a trained tree onto a ragged grid.
        {"name": "volume_tree_300k_odd", "kind": "volume", "scene": "tree", "n": 300_000,
         "d2": 250, "d1": 201, "d0": 173},
        # The trainer's losses alone, forward and backward.
        {"name": "loss_512_tv64", "kind": "loss", "width": 512, "height": 512, "dim": 64},
        # Densify and prune one per cent of a 500k table, moments and archive included.
        {"name": "refine_500k", "kind": "refine", "scene": "tree", "n": 500_000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["project", "project", "render", "step", "voxels", "volume", "loss",
                       "refine"])
    if kind in ("project", "render"):
        views = 1 if kind == "project" else rng.randint(1, 12)
        return {"kind": kind, "scene": rng.choice(["random", "tree"]),
                "n": _log_int(rng, 2000, 500_000 // views), "width": _log_int(rng, 60, 700),
                "height": _log_int(rng, 60, 700), "views": views}
    if kind == "step":
        dim, extent = rng.choice([(32, 0.25), (48, 0.5), (96, 2.0), (128, 2.0)])
        return {"kind": kind, "scene": "tree", "n": _log_int(rng, 1500, 400_000),
                "width": _log_int(rng, 100, 600), "height": _log_int(rng, 100, 600),
                "dim": dim, "extent": extent}
    if kind == "voxels":
        return {"kind": kind, "scene": rng.choice(["fine", "random"]),
                "n": _log_int(rng, 4000, 200_000),
                "d2": _log_int(rng, 40, 260), "d1": _log_int(rng, 40, 260),
                "d0": _log_int(rng, 40, 260)}
    if kind == "volume":
        return {"kind": kind, "scene": rng.choice(["fine", "tree"]),
                "n": _log_int(rng, 4000, 300_000),
                "d2": _log_int(rng, 40, 260), "d1": _log_int(rng, 40, 260),
                "d0": _log_int(rng, 40, 260)}
    if kind == "loss":
        return {"kind": kind, "width": _log_int(rng, 60, 1024), "height": _log_int(rng, 60, 1024),
                "dim": _log_int(rng, 16, 160)}
    return {"kind": kind, "scene": "tree", "n": _log_int(rng, 5000, 500_000)}


# ----------------------------------------------------------------- inputs --


_TREES = {}


def _scene(kind, n, g):
    """Raw parameters (means, quats, raw_scales, raw_opacities) on the host."""
    if kind == "tree":
        # A trained tree is no exact lattice: the grown one, with every leaf moved,
        # stretched and turned a little. The lattice itself does not depend on the seed.
        if n not in _TREES:
            _TREES[n] = scenes.binary_tree_gaussians(n)
        raw = _TREES[n]
        scale = scenes.activate_scale(raw.raw_scales)
        means = raw.means + 0.3 * scale * torch.randn(n, 3, generator=g)
        quats = F.normalize(raw.quats + 0.1 * torch.randn(n, 4, generator=g), dim=-1)
        scales = scenes.inverse_activate_scale(
            scale * torch.exp(0.1 * torch.randn(n, 3, generator=g)))
        opac = scenes.inverse_softplus(torch.rand(n, generator=g))
        return means, quats, scales, opac
    # Needle-like scenes are left out: their float32 gradients keep no digit in any order
    # of summation, so they could not be compared.
    mu, sigma = {"random": (-4.0, 0.5), "fine": (-4.5, 0.6), "dense": (-5.0, 0.5)}[kind]
    raw = scenes.random_gaussians(n, g, mu, sigma)
    return raw.means, raw.quats, raw.raw_scales, raw.raw_opacities


def _inputs(case, seed):
    """Every input of a case as device tensors, from the seed alone."""
    g = torch.Generator().manual_seed(seed)
    s = SimpleNamespace(kind=case["kind"])
    n = case.get("n")
    if n is not None:
        s.means, s.quats, s.scales, s.opacities = (t.to(DEV).contiguous() for t in
                                                   _scene(case["scene"], n, g))
    if "width" in case:
        s.width, s.height = case["width"], case["height"]
    if s.kind in ("project", "render", "step"):
        views = case.get("views", 1)
        first = float(torch.rand(1, generator=g)) * 2 * math.pi
        vms, Ks = zip(*(_view(first + 2 * math.pi * v / views, s.width, s.height)
                        for v in range(views)))
        s.viewmats, s.Ks = torch.stack(vms).to(DEV), torch.stack(Ks).to(DEV)
    if s.kind == "project":
        # A mean loss's image gradient: of the size of one over the pixel count.
        s.v_image = torch.randn(views, s.height, s.width, generator=g).to(DEV) \
            / (s.width * s.height)
    if s.kind in ("voxels", "volume"):
        s.dims = (case["d2"], case["d1"], case["d0"])  # x, y, z
        s.ranges = torch.full((3,), 2.0, device=DEV)
        s.centers = torch.zeros(3, device=DEV)
    if s.kind == "voxels":
        d2, d1, d0 = s.dims
        s.v_volume = torch.randn(d0, d1, d2, generator=g).to(DEV)
    if s.kind == "step":
        d, ext = case["dim"], case["extent"]
        s.dims = (d, d, d)
        s.ranges = torch.full((3,), ext, device=DEV)
        s.centers = ((torch.rand(3, generator=g) - 0.5) * (2.0 - ext)).to(DEV)
        # The last split's archive: leaf i's parent is entry i // 2, a little larger.
        h = max(1, n // 2)
        s.parent = torch.clamp(torch.arange(n) // 2, max=h - 1).to(torch.int32).to(DEV)
        s.history_means = s.means[:h * 2:2][:h].clone()
        s.history_scales = (s.scales[:h * 2:2][:h] + 0.5).clone()
        s.history_quats = s.quats[:h * 2:2][:h].clone()
        s.moments = {}
        for key in KEYS:
            shape = getattr(s, key).shape
            s.moments[key] = ((1e-6 * torch.randn(shape, generator=g)).to(DEV),
                              torch.full(shape, 1e-10, device=DEV))
    if s.kind in ("step", "loss"):
        h, w = s.height, s.width
        s.targets = torch.rand(1, h, w, 1, generator=g).to(DEV)
        s.edge_mask = (torch.rand(1, h, w, 1, generator=g) < 0.1).float().to(DEV)
    if s.kind == "loss":
        s.renders = (s.targets + 0.2 * torch.randn(1, h, w, 1, generator=g).to(DEV)).clamp_min(0)
        s.volume = torch.rand((case["dim"],) * 3, generator=g).to(DEV)
    if s.kind == "refine":
        s.state = {k: torch.rand(n, generator=g).to(DEV) for k in ("grad2d", "count", "radii")}
        s.state["scene_scale"] = 1.0
        s.moments = {k: tuple(torch.randn(getattr(s, k).shape, generator=g).to(DEV)
                              for _ in range(2)) for k in KEYS}
        # One row in a hundred grows, and as many of the grown table are pruned.
        k = n // 100
        s.grow = _mask(n, k, g)
        s.prune = _mask(n + k, k, g)
        s.parent = torch.randint(0, n, (n,), generator=g, dtype=torch.int32).to(DEV)
        s.level = torch.randint(0, 20, (n,), generator=g, dtype=torch.int32).to(DEV)
    return s


def _mask(n, k, g):
    mask = torch.zeros(n, dtype=torch.bool)
    mask[torch.randperm(n, generator=g)[:k]] = True
    return mask.to(DEV)


def _view(angle, width, height):
    """View matrix and intrinsics of a 3 x 3 detector of width x height pixels."""
    K = geometry.cone_beam_K((height, width), (3.0, 3.0), 1.5)
    pose = geometry.cone_beam_camtoworld(angle, 1.0)
    return geometry.invert_rigid_transform(pose), K


class _Tree(torch.nn.Module):
    """The attributes of a binary-tree Gaussian model that densification touches."""

    def __init__(self):
        super().__init__()
        self._use_sigmoid_scale = True
        self._scale_min, self._scale_max = torch.tensor(SMIN), torch.tensor(SMAX)
        self._scale_eps = scenes.SCALE_EPS


def _fill_table(s):
    """The table as it stood before a refinement (which replaces arrays and
    writes to none), so that every pass refines the same one."""
    m = s.model
    for key in KEYS:
        p = s.params[key]
        setattr(m, key, p)
        if key in s.opts:
            s.opts[key].param_groups[0]["params"] = [p]
            s.opts[key].state.clear()
            s.opts[key].state[p] = {"step": s.step, "exp_avg": s.moments[key][0],
                                    "exp_avg_sq": s.moments[key][1]}
    m.parent, m.level = s.parent, s.level
    for key, t in s.history.items():
        setattr(m, "history_" + key, t)
    s.stats = dict(s.state)


def _optimizers(model, moments):
    opts = {}
    for key in KEYS:
        p = getattr(model, key)
        opts[key] = optim.Adam([{"params": p, "name": key}], lr=LRS[key], eps=1e-15)
        m, v = moments[key]
        opts[key].state[p] = {"step": torch.tensor(100.0), "exp_avg": m.clone(),
                              "exp_avg_sq": v.clone()}
    return opts


def prepare(case, seed):
    s = _inputs(case, seed)
    if s.kind in ("project", "step"):
        for key in KEYS:
            setattr(s, key, torch.nn.Parameter(getattr(s, key)))
    if s.kind == "step":
        s.opts = _optimizers(s, s.moments)
        w_l1, w_ssim, w_edge, w_tv, w_hier = LOSS_WEIGHTS
        s.loss = loss.BinaryTreeLossComputer(w_l1=w_l1, w_ssim=w_ssim, w_tv=w_tv, w_edge=w_edge,
                                             w_hierarchy=w_hier, ssim_window=11)
    if s.kind in ("render", "volume"):
        s.prepared = direct.prepare_inference_gaussians(s.quats, s.scales, s.opacities,
                                                        scale_min=SMIN, scale_max=SMAX)
    if s.kind == "voxels":
        s.covars, s.max_scales, s.weights = W.prepare_gaussians(s.quats, s.scales, s.opacities,
                                                                SMIN, SMAX)
    if s.kind == "loss":
        s.renders.requires_grad_(True)
        s.volume.requires_grad_(True)
        w_l1, w_ssim, _, w_tv, _ = LOSS_WEIGHTS
        s.loss = loss.LossComputer(w_l1=w_l1, w_ssim=w_ssim, w_tv=w_tv, ssim_window=11)
    if s.kind == "refine":
        h = s.means.shape[0] // 2
        s.history = {k: getattr(s, k)[:h].clone() for k in KEYS + ("parent", "level")}
        s.params = {k: torch.nn.Parameter(getattr(s, k)) for k in KEYS}
        s.step = torch.tensor(100.0)
        s.model, s.opts = _Tree(), {}
        _fill_table(s)
        s.opts = _optimizers(s.model, s.moments)
    return s


# -------------------------------------------------------------------- run --


def run(s):
    return _RUN[s.kind](s)


def _rasterize(s, state):
    return explicit.explicit_rasterize(state, s.means, s.viewmats, s.Ks, img_w=s.width,
                                       img_h=s.height, tile_size=TILE, eps2d=EPS,
                                       radius_clip=CLIP, absgrad=True)


def _run_project(s):
    for key in KEYS:
        getattr(s, key).grad = None
    state = explicit.prepare_explicit_gaussians(s.quats, s.scales, s.opacities, scale_min=SMIN,
                                                scale_max=SMAX)
    res = _rasterize(s, state)
    res.image.grad = s.v_image
    explicit.explicit_backward(state, s.means, s.quats, s.scales, s.opacities)
    return {"image": res.image.detach(), "radii": res.radii, "means2d": res.means2d.detach(),
            "v_means": s.means.grad, "v_quats": s.quats.grad, "v_scales": s.scales.grad,
            "v_opacities": s.opacities.grad, "v_means2d": res.means2d.grad,
            "v_means2d_abs": res.means2d.absgrad}


def _run_render(s):
    res = direct.inference_rasterize(s.prepared, s.means, s.viewmats, s.Ks, img_w=s.width,
                                     img_h=s.height, tile_size=TILE, eps2d=EPS, radius_clip=CLIP)
    return {"image": res.image, "radii": res.radii, "means2d": res.means2d}


def _run_step(s):
    for key in KEYS:
        getattr(s, key).grad = None
    state = explicit.prepare_explicit_gaussians(s.quats, s.scales, s.opacities, scale_min=SMIN,
                                                scale_max=SMAX)
    res = _rasterize(s, state)
    d2, d1, d0 = s.dims
    vox = explicit.explicit_voxelize(state, s.means, s.ranges, s.centers, dim2=d2, dim1=d1,
                                     dim0=d0, tile_size=BRICK, eps3d=EPS, radius_clip=CLIP)
    hier = loss.compute_hierarchy_loss(s.means, s.parent, s.history_means, s.history_scales,
                                       s.history_quats, scenes.activate_scale, 1.0)
    out = s.loss(res.image.unsqueeze(-1), s.targets, s.edge_mask, vox.volume,
                 hierarchy_loss=hier)
    out["total"].backward()
    explicit.explicit_backward(state, s.means, s.quats, s.scales, s.opacities)
    optim.step_all(s.opts)
    return {"image": res.image.detach(), "volume": vox.volume.detach(),
            "total": out["total"].detach(),
            "v_means": s.means.grad, "v_quats": s.quats.grad, "v_scales": s.scales.grad,
            "v_opacities": s.opacities.grad, "v_means2d_abs": res.means2d.absgrad,
            "means": s.means.detach(), "quats": s.quats.detach(), "scales": s.scales.detach(),
            "opacities": s.opacities.detach()}


def _run_voxels(s):
    d2, d1, d0 = s.dims
    n2, n1, n0 = (-(-d // BRICK) for d in s.dims)
    m3, con, r3 = W.world_to_volume_mapping_fwd(s.means, s.covars, s.max_scales, s.ranges,
                                                s.centers, d2, d1, d0, EPS, CLIP)
    _, ids, flat = W.isect_tiles_3d(m3, r3, BRICK, n2, n1, n0)
    off = W.isect_offset_encode_3d(ids, n2, n1, n0)
    vol = W.voxelize_to_voxels_fwd(m3, con, s.weights, off, flat, d2, d1, d0, BRICK)
    vm3, vcon, vw = W.voxelize_to_voxels_bwd_per_gaussian(m3, con, s.weights, off, ids, flat,
                                                          s.v_volume, d2, d1, d0, BRICK)
    vm, vcov = W.world_to_volume_mapping_bwd(s.means, s.covars, s.ranges, s.centers, d2, d1, d0,
                                             EPS, vm3, vcon)
    return {"volume": vol, "radii": r3, "v_means": vm, "v_covars": vcov, "v_weights": vw}


def _run_volume(s):
    d2, d1, d0 = s.dims
    res = direct.inference_voxelize(s.prepared, s.means, s.ranges, s.centers, dim2=d2, dim1=d1,
                                    dim0=d0, tile_size=BRICK, eps3d=EPS, radius_clip=CLIP)
    return {"volume": res.volume, "radii": res.radii}


def _run_loss(s):
    s.renders.grad = s.volume.grad = None
    out = s.loss(s.renders, s.targets, s.volume)
    out["total"].backward()
    return {"l1": out["proj_l1"].detach(), "ssim": out["proj_ssim"].detach(),
            "tv": out["vol_tv"].detach(), "total": out["total"].detach(),
            "v_renders": s.renders.grad, "v_volume": s.volume.grad}


def _run_refine(s):
    m = s.model
    _fill_table(s)
    densify.split(m, s.opts, s.stats, s.grow, list(KEYS))
    densify.remove(m, s.opts, s.stats, s.prune, list(KEYS))
    out = {k: getattr(m, k).detach() for k in KEYS}
    out.update(parent=m.parent, level=m.level, history_means=m.history_means,
               history_scales=m.history_scales, history_quats=m.history_quats,
               history_opacities=m.history_opacities, history_parent=m.history_parent,
               history_level=m.history_level, grad2d=s.stats["grad2d"], count=s.stats["count"],
               radii=s.stats["radii"])
    for k in KEYS:
        st = s.opts[k].state[getattr(m, k)]
        out["m_" + k], out["v_" + k] = st["exp_avg"], st["exp_avg_sq"]
    return out


_RUN = {"project": _run_project, "render": _run_render, "step": _run_step,
        "voxels": _run_voxels, "volume": _run_volume, "loss": _run_loss, "refine": _run_refine}


# ------------------------------------------------------- work, tolerances --


def work(case):
    """Bytes of the inputs and outputs, and the arithmetic of the pairs that a
    footprint of one tile (brick) per Gaussian costs at least: the real record
    count depends on the scene and is not known here."""
    kind, n = case["kind"], case.get("n", 0)
    pix = case.get("width", 0) * case.get("height", 0) * case.get("views", 1)
    if kind == "project":
        per = 44 + 44 + case["views"] * 32  # parameters, their gradients, per-view results
        return {"bytes": n * per + 8 * pix, "flops": n * case["views"] * 256 * (15 + 51)}
    if kind == "render":
        return {"bytes": n * (40 + case["views"] * 16) + 4 * pix,
                "flops": n * case["views"] * 256 * 15}
    if kind == "step":
        vox = case["dim"] ** 3
        inside = n * min(1.0, case["extent"] / 2.0) ** 3
        # Parameters and moments read and written, gradients written; the
        # archive read; images and the volume.
        return {"bytes": n * (44 * 7 + 16) + n // 2 * 40 + 16 * pix + 4 * vox,
                "flops": n * 256 * (15 + 51) + inside * 512 * (24 + 77)}
    if kind in ("voxels", "volume"):
        vox = case["d2"] * case["d1"] * case["d0"]
        if kind == "volume":
            return {"bytes": n * (44 + 24) + 4 * vox, "flops": n * 512 * 24}
        return {"bytes": n * (44 + 12 + 40) + 8 * vox, "flops": n * 512 * (24 + 77)}
    if kind == "loss":
        vox = case["dim"] ** 3
        return {"bytes": 12 * pix + 8 * vox, "flops": pix * 11 * 2 * 8 * 2 + 12 * vox}
    rows = n + n // 100
    return {"bytes": 4 * (44 - 6) * (2 * n + 2 * rows) + 4 * 13 * 2 * (n // 2 + n // 100),
            "flops": n}


def tolerance(case):
    """About four times the largest relative error against float64 seen over the
    listed and drawn cases: v_quats of trees 1.1e-4 and of the other scenes 5.1e-5 in a
    projection, means2d 2.1e-6 in a render, v_quats and the absolute gradients 1.8e-5 in
    a step, v_covars 3.0e-5 of the voxels, 1.0e-5 of a volume, 4.7e-7 of the losses and
    1.3e-8 of the refined rows."""
    kind = case["kind"]
    if kind == "project":
        return {"rel": 5e-4 if case["scene"] == "tree" else 2e-4}
    return {"rel": {"render": 1e-5, "step": 8e-5, "voxels": 1.2e-4, "volume": 4e-5,
                    "loss": 2e-6, "refine": 5e-8}[kind]}


# --------------------------------------------------------- float64 values --


def _d(t):
    return t.detach().to(torch.float64)


def _rotation(q):
    w, x, y, z = F.normalize(q, dim=-1, eps=1e-12).unbind(-1)
    return torch.stack([1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y),
                        2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x),
                        2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y)],
                       -1).reshape(-1, 3, 3)


def _activate(quats, scales, opac):
    """Covariances [N,3,3], opacities [N]."""
    s = SMIN + (SMAX - SMIN) * torch.sigmoid(scales)
    m = _rotation(quats) * s[:, None, :]
    return m @ m.transpose(1, 2), F.softplus(opac)


def _project(means, cov, viewmat, K, width, height):
    """Detector means [N,2], conics [N,3], mus [N] and radii [N,2] of one view."""
    R, t = viewmat[:3, :3], viewmat[:3, 3]
    fx, fy, cx, cy = K[0, 0], K[1, 1], K[0, 2], K[1, 2]
    x, y, z = (means @ R.T + t).unbind(-1)
    front = z > 0.01
    z = torch.where(front, z, torch.ones_like(z))
    u, v = fx * x / z + cx, fy * y / z + cy
    mx, my = 0.3 * 0.5 * width / fx, 0.3 * 0.5 * height / fy
    tx = z * torch.minimum(torch.maximum(x / z, -(cx / fx + mx)), (width - cx) / fx + mx)
    ty = z * torch.minimum(torch.maximum(y / z, -(cy / fy + my)), (height - cy) / fy + my)
    l = torch.sqrt(tx * tx + ty * ty + z * z)
    o = torch.zeros_like(z)
    J = torch.stack([torch.stack([fx / z, o, -fx * tx / z ** 2], -1),
                     torch.stack([o, fy / z, -fy * ty / z ** 2], -1),
                     torch.stack([tx / l, ty / l, z / l], -1)], -2)
    M = J @ R
    C = M @ cov @ M.transpose(1, 2)
    a, b, c, d, e, f = (C[:, 0, 0] + EPS, C[:, 0, 1], C[:, 0, 2], C[:, 1, 1] + EPS, C[:, 1, 2],
                        C[:, 2, 2] + EPS)
    det2 = a * d - b * b
    det3 = a * d * f - a * e * e - b * b * f + 2 * b * c * e - c * c * d
    ok2 = front & (det2 > 1e-9)
    safe = torch.where(ok2, det2, torch.ones_like(det2))
    conics = torch.where(ok2[:, None], torch.stack([d, -b, a], -1) / safe[:, None], 0.0)
    pos = ok2 & (det3 / safe > 0)
    ratio = torch.where(pos, det3 / safe, torch.ones_like(det3))
    mus = torch.where(pos, torch.sqrt(2 * math.pi * ratio), 0.0)
    mus = torch.where(det3 > 1e-9, mus, mus.detach())  # no gradient through a flat footprint
    with torch.no_grad():
        r = torch.ceil(CLIP * torch.stack([a, d], -1).clamp_min(0).sqrt())
        m = torch.stack([u, v], -1)
        size = torch.tensor([width, height], dtype=r.dtype, device=r.device)
        on = front & (det2 > 0) & (r > 0).all(-1) & torch.isfinite(r).all(-1)
        on &= ((m + r > 0) & (m - r < size)).all(-1)
        radii = torch.where(on[:, None], r, 0.0)
    return torch.where(front[:, None], torch.stack([u, v], -1), 0.0), conics, mus, radii


def _map(means, cov, ranges, centers, dims):
    """Voxel-space means [N,3] (x, y, z), conics [N,3,3] and radii [N,3]."""
    size = torch.tensor(dims, dtype=means.dtype, device=means.device)
    r = size / ranges
    m = (means - centers) * r + size * 0.5
    S = cov * r[:, None] * r + EPS * torch.eye(3, dtype=means.dtype, device=means.device)
    det = torch.linalg.det(S)
    ok = det.abs() >= 1e-12
    P = torch.linalg.inv(torch.where(ok[:, None, None], S, torch.eye(3, dtype=S.dtype,
                                                                     device=S.device)))
    with torch.no_grad():
        rad = torch.ceil(CLIP * torch.diagonal(S, dim1=1, dim2=2).clamp_min(0).sqrt())
        good = ok & torch.isfinite(rad).all(-1) & (rad > 0).all(-1)
    return m, torch.where(ok[:, None, None], P, 0.0), torch.where(good[:, None], rad, 0.0)


def _pairs(m, radii, dims, tile):
    """(ids [I], first pixel of each record's tile [I, D]), one record per tile
    that a Gaussian's box of +-radii covers."""
    cells = [-(-d // tile) for d in dims]
    lim = torch.tensor(cells, dtype=m.dtype, device=m.device)
    lo = torch.floor((m - radii) / tile).clamp_min(0).minimum(lim).long()
    hi = torch.ceil((m + radii) / tile).clamp_min(0).minimum(lim).long()
    ext = torch.where((radii > 0).all(-1)[:, None], (hi - lo).clamp_min(0), 0)
    count = ext.prod(-1)
    total = int(count.sum())
    if total * tile ** len(dims) > MAX_EXACT_PAIRS:
        return None
    ids = torch.repeat_interleave(count)
    local = torch.arange(total, device=m.device) - (count.cumsum(0) - count)[ids]
    at = []
    for a in range(len(dims)):
        e = ext[ids, a]
        at.append((lo[ids, a] + local % e) * tile)
        local = local // e
    return ids, torch.stack(at, -1)


def _splat(m, P, w, pairs, dims, tile, thr, v=None):
    """The sum over records of w exp(-sigma) on a grid of ``dims`` (x first),
    and, for an upstream gradient v of that grid, the gradients of the means
    (and of their absolute per-cell terms), of P and of w."""
    D = len(dims)
    ids, first = pairs
    out = torch.zeros(dims[::-1], dtype=m.dtype, device=m.device)
    grads = None
    if v is not None:
        grads = [torch.zeros_like(m), torch.zeros_like(m), torch.zeros_like(P),
                 torch.zeros_like(w)]
    cell = torch.stack(torch.meshgrid(*[torch.arange(tile, device=m.device)] * D, indexing="ij"),
                       -1).reshape(-1, D)
    size = torch.tensor(dims, device=m.device)
    stride = torch.tensor([math.prod(dims[:a]) for a in range(D)], device=m.device)
    chunk = (1 << 25) // tile ** D
    for b in range(0, ids.numel(), chunk):
        i = ids[b:b + chunk]
        px = first[b:b + chunk, None, :] + cell  # [I, cells, D]
        inside = (px < size).all(-1)
        at = torch.where(inside, (px * stride).sum(-1), 0)
        d = px.to(m.dtype) + 0.5 - m[i][:, None, :]
        t = d @ P[i]
        sigma = 0.5 * (t * d).sum(-1)
        e = torch.exp(-sigma)
        alpha = w[i][:, None] * e
        on = inside & (sigma >= 0) & (alpha.abs() >= thr)
        e, alpha = e * on, torch.where(on, alpha, 0.0)
        out.view(-1).index_add_(0, at.reshape(-1), alpha.reshape(-1))
        if v is not None:
            up = v.reshape(-1)[at]
            k = (up * alpha)[..., None] * t
            grads[0].index_add_(0, i, k.sum(1))
            grads[1].index_add_(0, i, k.abs().sum(1))
            outer = -0.5 * (d * (up * alpha)[..., None]).transpose(1, 2) @ d
            grads[2].index_add_(0, i, outer)
            grads[3].index_add_(0, i, (up * e).sum(1))
    return out, grads


def _sym2(con):
    a, b, c = con.unbind(-1)
    return torch.stack([torch.stack([a, b], -1), torch.stack([b, c], -1)], -2)


def _raster(means, cov, op, s, v_image=None):
    """All views' images; with v_image also the graph outputs and their gradients."""
    images, outs, ups, m2s, v2s, vabs = [], [], [], [], [], []
    for c in range(s.viewmats.shape[0]):
        m, con, mu, radii = _project(means, cov, _d(s.viewmats[c]), _d(s.Ks[c]), s.width,
                                     s.height)
        P = _sym2(con)
        dims = (s.width, s.height)
        pairs = _pairs(m.detach(), radii, dims, TILE)
        if pairs is None:
            return None
        v = None if v_image is None else v_image[c]
        image, g = _splat(m.detach(), P.detach(), (op * mu).detach(), pairs, dims, TILE, THR_2D,
                          v)
        images.append(image)
        m2s.append(m.detach())
        if g is not None:
            outs += [m, P, op * mu]
            ups += [g[0], g[2], g[3]]
            v2s.append(g[0])
            vabs.append(g[1])
    stack = lambda x: torch.stack(x) if x else None  # noqa: E731
    return stack(images), outs, ups, stack(m2s), stack(v2s), stack(vabs)


def _leaves(s):
    return {k: _d(getattr(s, k)).requires_grad_(True) for k in KEYS}


def _exact_project(s):
    p = _leaves(s)
    cov, op = _activate(p["quats"], p["scales"], p["opacities"])
    r = _raster(p["means"], cov, op, s, _d(s.v_image))
    if r is None:
        return None
    image, outs, ups, m2, v2, vabs = r
    torch.autograd.backward(outs, ups)
    return {"image": image, "radii": None, "means2d": m2, "v_means": p["means"].grad,
            "v_quats": p["quats"].grad, "v_scales": p["scales"].grad,
            "v_opacities": p["opacities"].grad, "v_means2d": v2, "v_means2d_abs": vabs}


def _exact_render(s):
    with torch.no_grad():
        cov, op = _activate(_d(s.quats), _d(s.scales), _d(s.opacities))
        r = _raster(_d(s.means), cov, op, s)
    return None if r is None else {"image": r[0], "radii": None, "means2d": r[3]}


def _packed(P):
    return torch.stack([P[:, 0, 0], P[:, 0, 1] + P[:, 1, 0], P[:, 0, 2] + P[:, 2, 0], P[:, 1, 1],
                        P[:, 1, 2] + P[:, 2, 1], P[:, 2, 2]], -1)


def _exact_voxels(s):
    means = _d(s.means).requires_grad_(True)
    cov, op = _activate(_d(s.quats), _d(s.scales), _d(s.opacities))
    cov.requires_grad_(True)
    m, P, radii = _map(means, cov, _d(s.ranges), _d(s.centers), s.dims)
    pairs = _pairs(m.detach(), radii, s.dims, BRICK)
    if pairs is None:
        return None
    volume, g = _splat(m.detach(), P.detach(), op, pairs, s.dims, BRICK, THR_3D, _d(s.v_volume))
    torch.autograd.backward([m, P], [g[0], g[2]])
    return {"volume": volume, "radii": None, "v_means": means.grad, "v_covars": _packed(cov.grad),
            "v_weights": g[3]}


def _exact_volume(s):
    with torch.no_grad():
        cov, op = _activate(_d(s.quats), _d(s.scales), _d(s.opacities))
        m, P, radii = _map(_d(s.means), cov, _d(s.ranges), _d(s.centers), s.dims)
        pairs = _pairs(m, radii, s.dims, BRICK)
        if pairs is None:
            return None
        return {"volume": _splat(m, P, op, pairs, s.dims, BRICK, THR_3D)[0], "radii": None}


def _ssim(x, y):
    """Mean SSIM of [H, W] images with the 11 x 11 window of sigma 1.5."""
    e = torch.tensor([math.exp(-((k - 5) ** 2) / 4.5) for k in range(11)])
    taps = (e / e.sum())[:, None]
    win = (taps @ taps.T).double().to(x.device)

    def f(t):
        pad = F.pad(t, (5, 5, 5, 5))
        return sum(win[i, j] * pad[i:i + t.shape[0], j:j + t.shape[1]]
                   for i in range(11) for j in range(11))

    c1, c2 = 0.01 ** 2, 0.03 ** 2
    mx, my = f(x), f(y)
    xx, yy, xy = f(x * x) - mx * mx, f(y * y) - my * my, f(x * y) - mx * my
    return (((2 * mx * my + c1) * (2 * xy + c2)) /
            ((mx * mx + my * my + c1) * (xx + yy + c2))).mean()


def _tv(v):
    parts = [(v.diff(dim=a)).abs() for a in range(3)]
    return sum(p.sum() for p in parts) / sum(p.numel() for p in parts)


def _exact_loss(s):
    x, v = _d(s.renders).requires_grad_(True), _d(s.volume).requires_grad_(True)
    y = _d(s.targets)
    l1, ssim, tv = (x - y).abs().mean(), 1 - _ssim(x[0, :, :, 0], y[0, :, :, 0]), _tv(v)
    w_l1, w_ssim, _, w_tv, _ = LOSS_WEIGHTS
    total = w_l1 * l1 + w_ssim * ssim + w_tv * tv
    total.backward()
    return {"l1": l1.detach(), "ssim": ssim.detach(), "tv": tv.detach(), "total": total.detach(),
            "v_renders": x.grad, "v_volume": v.grad}


def _hierarchy(means, s):
    ids = s.parent.long()
    R = _rotation(_d(s.history_quats))[ids]
    scale = (SMIN + (SMAX - SMIN) * torch.sigmoid(_d(s.history_scales))).clamp_min(1e-6)[ids]
    u = (R.transpose(1, 2) @ (means - _d(s.history_means)[ids])[..., None])[..., 0] / scale
    r = (u.square().sum(-1) + 1e-300).sqrt()
    return (r - 1.0).clamp_min(0).square().mean()


def _exact_step(s):
    p = _leaves(s)
    cov, op = _activate(p["quats"], p["scales"], p["opacities"])
    r = _raster(p["means"], cov, op, s)
    m, P, radii = _map(p["means"], cov, _d(s.ranges), _d(s.centers), s.dims)
    pairs = _pairs(m.detach(), radii, s.dims, BRICK)
    if r is None or pairs is None:
        return None
    image = r[0].requires_grad_(True)
    volume = _splat(m.detach(), P.detach(), op.detach(), pairs, s.dims, BRICK, THR_3D)[0]
    volume.requires_grad_(True)
    y, mask = _d(s.targets)[0, :, :, 0], _d(s.edge_mask)[0, :, :, 0]
    diff = (image[0] - y).abs()
    w_l1, w_ssim, w_edge, w_tv, w_hier = LOSS_WEIGHTS
    total = (w_l1 * diff.mean() + w_ssim * (1 - _ssim(image[0], y)) + w_edge *
             (mask * diff).mean() + w_tv * _tv(volume) + w_hier * _hierarchy(p["means"], s))
    total.backward()
    _, outs, ups, _, _, vabs = _raster(p["means"], cov, op, s, image.grad)
    _, g = _splat(m.detach(), P.detach(), op.detach(), pairs, s.dims, BRICK, THR_3D, volume.grad)
    torch.autograd.backward(outs + [m, P, op], ups + [g[0], g[2], g[3]])
    out = {"image": image.detach(), "volume": volume.detach(), "total": total.detach(),
           "v_means2d_abs": vabs}
    for key in KEYS:
        grad = p[key].grad
        m1, m2 = (_d(t) for t in s.moments[key])
        m1 = m1 + 0.1 * (grad - m1)
        m2 = 0.999 * m2 + 0.001 * grad * grad
        step = LRS[key] / (1 - 0.9 ** 101)
        out["v_" + key] = grad
        out[key] = p[key].detach() - step * m1 / (m2.sqrt() / math.sqrt(1 - 0.999 ** 101) + 1e-15)
    return out


def _exact_refine(s):
    n = s.means.shape[0]
    sel, rest = torch.where(s.grow)[0], torch.where(~s.grow)[0]
    keep = torch.where(~s.prune)[0]
    h = n // 2
    scale = SMIN + (SMAX - SMIN) * torch.sigmoid(_d(s.scales)[sel])
    axis = F.one_hot(scale.argmax(-1), 3).to(scale.dtype)
    offset = (_rotation(_d(s.quats)[sel]) @ (scale * axis)[..., None])[..., 0]
    child = (scale / (1 + 0.6 * axis)).clamp(SMIN + scenes.SCALE_EPS, SMAX - scenes.SCALE_EPS)
    child = ((child - SMIN) / (SMAX - SMIN)).clamp(1e-6, 1 - 1e-6)
    new = {"means": torch.cat([_d(s.means)[sel] + offset, _d(s.means)[sel] - offset]),
           "scales": torch.logit(child).repeat(2, 1)}
    take = lambda t, tail: torch.cat([t[rest], tail])[keep]  # noqa: E731
    twice = lambda t: t[torch.cat([sel, sel])]  # noqa: E731
    out = {}
    for key in KEYS:
        t = _d(getattr(s, key))
        out[key] = take(t, new.get(key, twice(t)))
        for name, mom in zip("mv", s.moments[key]):
            out[f"{name}_{key}"] = take(_d(mom), torch.zeros_like(twice(_d(mom))))
    for key in ("grad2d", "count", "radii"):
        out[key] = take(_d(s.state[key]), twice(_d(s.state[key])))
    for key in KEYS:
        t = _d(getattr(s, key))
        out["history_" + key] = torch.cat([t[:h], t[sel]])
    out.update(parent=None, level=None, history_parent=None, history_level=None)
    return out


_EXACT = {"project": _exact_project, "render": _exact_render, "step": _exact_step,
          "voxels": _exact_voxels, "volume": _exact_volume, "loss": _exact_loss,
          "refine": _exact_refine}


def exact(case, seed):
    return _EXACT[case["kind"]](_inputs(case, seed))
