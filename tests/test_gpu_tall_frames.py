"""Slivers taller than one launch holds rows of two: they run one lane per ray, eight rows a
workgroup, whatever their work."""
import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import dataset as D
from hydrant_amd import workloads as W
from tests.helpers import oracle_view, oracle_volume

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("schedule", [L.SCHED_REFERENCE, L.SCHED_LATTICE])
@pytest.mark.parametrize("H_", [131070, 131071, 140003])
def test_one_pixel_wide(gpu_ctx, schedule, H_):
    import torch

    n = 16
    vol = D.gen_blobs(n, 6, 31, sig=(4.0, 10.0), sigma_scale=n / 32.0, amp=(0.4, 1.0))
    b = D.make_bricked(vol, 8, 1, L.FMT_U8, None, resident=1.0, seed=5)
    sc = W.Scene("tall", b, D.README_TF.copy(), 1, H_, (33.0, 21.0, 2.2), 60.0, D.geometry((n, n, n), 8, 0.5),
                 density=0.2, schedule=schedule)
    ctx, p, view = gpu_ctx, sc.volume_params(), sc.view()
    ctx.load(b, sc.tf)
    out = ctx.render_volume(p, view, 1, H_, film=False, count=True)
    r = oracle_volume(sc).render(oracle_view(sc), 32, film=False)
    assert int(out["samples"].item()) == r["samples"] > 0
    assert np.max(np.abs(out["rgba"].cpu().numpy() - r["rgba"])) <= 1e-4
    if schedule == L.SCHED_LATTICE:
        t = torch.from_numpy(b.pool).cuda()
        sset = ctx.segment_set([(L.FMT_U8, b.pad, t, b.vaddr, b.page_k, b.page_b)])
        rgba, cnt = ctx.render_sort_last_set(p, view, 1, H_, sset, count=True)
        assert int(cnt.item()) == r["samples"]
        assert float((rgba - out["rgba"]).abs().max()) <= 1e-5
        sset.close()


@pytest.mark.parametrize("H_", [131070, 131071, 131072])
def test_differentiable_one_pixel_wide(gpu_ctx, H_):
    """A view alone (four lanes per ray while its rows fit) and twice in a launch (one lane)."""
    import torch

    from hydrant_amd.diff import DiffRenderer

    wl = W.differentiable(n=12, n_views=1, W=1, H=H_, n_steps=16, ckpt_every=8, sigma=40.0)
    vol, tf = torch.from_numpy(wl.hidden_volume).cuda(), torch.from_numpy(wl.hidden_tf).cuda()
    out = []
    for views in (wl.views(), wl.views() * 2):
        r = DiffRenderer(gpu_ctx, views, 1, H_, (wl.n,) * 3, 16, 8, wl.sigma)
        rgba, ck, cnt = r.forward_raw(vol, tf, count=True)
        out.append((rgba[0].clone(), ck[0].clone(), int(cnt.item())))
    assert 2 * out[0][2] == out[1][2] > 0
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
