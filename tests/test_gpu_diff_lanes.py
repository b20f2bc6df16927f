"""The differentiable forward at each number of lanes per ray (16, 4, 1) and the scatter with a
view's rays split or not: the same view rendered alone and among others is the same, bit for bit;
gradients of a small launch equal those summed from its views' own launches to rounding."""
import numpy as np
import pytest

from hydrant_amd import workloads as W
from hydrant_amd.diff import DiffRenderer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_steps,ckpt", [(512, 64), (98, 64), (5, 2), (64, 7)])
@pytest.mark.parametrize("W_,H_,n_views", [(33, 29, 3), (61, 47, 30), (133, 110, 12)])
def test_views_alone_and_together(gpu_ctx, W_, H_, n_views, n_steps, ckpt):
    """n_views together run fewer lanes per ray than one view alone (957 rays: 16 lanes; 86,010: 4;
    175,560: 1)."""
    import torch

    wl = W.differentiable(n=20, n_views=n_views, W=W_, H=H_, n_steps=n_steps, ckpt_every=ckpt, sigma=40.0)
    vol, tf = torch.from_numpy(wl.hidden_volume).cuda(), torch.from_numpy(wl.hidden_tf).cuda()
    views = wl.views()
    grad = torch.from_numpy(np.random.default_rng(1).normal(size=(n_views, H_, W_, 4)).astype(np.float32)).cuda()
    r = DiffRenderer(gpu_ctx, views, W_, H_, (wl.n,) * 3, n_steps, ckpt, wl.sigma)
    rgba, ck, cnt = r.forward_raw(vol, tf, count=True)
    gv, gt = r.backward_raw(vol, tf, ck, grad)
    sv, st, total = torch.zeros_like(gv).double(), torch.zeros_like(gt).double(), 0
    for i in range(n_views):
        one = DiffRenderer(gpu_ctx, views[i:i + 1], W_, H_, (wl.n,) * 3, n_steps, ckpt, wl.sigma)
        a, c, m = one.forward_raw(vol, tf, count=True)
        assert torch.equal(a[0], rgba[i]) and torch.equal(c[0], ck[i])
        total += int(m.item())
        g = one.backward_raw(vol, tf, c, grad[i:i + 1].contiguous())
        sv += g[0].double()
        st += g[1].double()
    assert total == int(cnt.item()) > 0
    # FP32 sums of up to 30 views' blocks (and one fixed-point scale per launch):
    # 2^-24 a term, 64 terms
    assert float((gv - sv).abs().max()) <= 64 * 2 ** -24 * float(sv.abs().max())
    assert float((gt - st).abs().max()) <= 64 * 2 ** -24 * float(st.abs().max())
