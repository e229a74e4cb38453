"""The loss computers' one reduction launch and the scales formed inside the
backward kernels, against the separate projection and TV operators (which are
checked against the oracle): the terms and gradients are the same bits, and
the total, summed in double, is the correctly rounded weighted sum."""

import pytest
import torch

from r2splat.cuda import _wrapper as W
from r2splat.ops import loss as LO

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("shape,vol_shape,edge", [
    ((1, 1, 1, 1), None, False),
    ((1, 1, 1, 1), (1, 1, 1), True),
    ((1, 33, 31, 1), (1, 1, 5), False),
    ((2, 64, 48, 2), (40, 33, 17), True),
    ((3, 300, 217, 1), (64, 64, 64), True),     # more block sums than threads
    ((1, 40, 70, 1), (0, 4, 4), False),
])
@pytest.mark.parametrize("hier", [None, torch.float32, torch.float64])
def test_total_of_a_step(shape, vol_shape, edge, hier):
    g = torch.Generator().manual_seed(sum(shape))
    rnd = lambda *s: torch.rand(*s, generator=g).to(DEV)  # noqa: E731
    r, t = rnd(*shape).requires_grad_(True), rnd(*shape)
    e, m = (rnd(*shape), rnd(*shape)) if edge else (None, None)
    v = None if vol_shape is None else rnd(*vol_shape).requires_grad_(True)
    weights = (0.8, 0.2, 0.3, 0.05, 0.7)
    h = None if hier is None else torch.tensor(0.37, dtype=hier, device=DEV, requires_grad=True)
    comp = LO.BinaryTreeLossComputer(w_l1=weights[0], w_ssim=weights[1], w_edge=weights[2],
                                     w_tv=weights[3], w_hierarchy=weights[4])
    out = comp(r, t, m, v, hierarchy_loss=h, edge_targets=e)
    planes = [None if x is None else LO._planes(x.detach()) for x in (r, t, e, m)]
    losses, ws = W.projection_loss_fwd(*planes)
    squeezed = None if v is None else v.detach().squeeze()
    has_tv = squeezed is not None and squeezed.dim() == 3
    tv = W.tv_fwd(squeezed) if has_tv else torch.zeros((), device=DEV)
    for name, want in (("proj_l1", losses[0]), ("proj_ssim", losses[1]), ("edge", losses[2]),
                       ("vol_tv", tv)):
        assert torch.equal(out[name].detach(), want), name
    w = torch.tensor(weights, device=DEV)
    terms = torch.stack([*losses, tv, torch.zeros((), device=DEV) if h is None
                         else h.detach().float()])
    assert torch.equal(out["total"].detach(), (w.double() * terms.double()).sum().float())
    up = torch.tensor(1.7, device=DEV)
    out["total"].backward(up)
    scales = w * up
    assert torch.equal(LO._planes(r.grad), W.projection_loss_bwd(*planes, scales[:3], ws))
    if has_tv:
        assert torch.equal(v.grad.squeeze(), W.tv_bwd(squeezed, scales[3:4]))
    if h is not None:
        assert torch.equal(h.grad, scales[4].to(hier))
