"""Sort-last segments over bricks without an apron, whose taps clamp at the brick's faces: the
sampler chosen per group must give the clamping sampler's values, at every number of lanes per
ray and for runs that end one, two or three samples into a group."""
import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import dataset as D
from hydrant_amd import workloads as W

pytestmark = pytest.mark.gpu

# opacities for values up to 0.6; the last entry is out of their reach
TF = np.stack([np.linspace(0.1, 1, 16), np.linspace(1, 0.2, 16), np.tile([0.3, 0.9], 8), np.linspace(0.01, 0.2, 16)],
              1).astype(np.float32)


def _scene(fmt, n, bs, arm, W_, H_):
    vol = np.random.default_rng(n).integers(0, 141, (n, n, n)).astype(np.uint8)   # noise: every tap matters
    if fmt != L.FMT_U8:
        vol = vol.astype(np.float32) / np.float32(255)
        vol = vol.astype(np.float16).view(np.uint16) if fmt == L.FMT_F16 else vol
    b = D.make_bricked(vol, bs or n, 0, fmt, None, resident=1.0, seed=5)
    return W.Scene("noise", b, TF, W_, H_, arm, 60.0, D.geometry((n, n, n), bs or n, 0.5), density=0.3,
                   schedule=L.SCHED_LATTICE)


@pytest.mark.parametrize("W_,H_", [(37, 29), (163, 157), (1001, 997)])
@pytest.mark.parametrize("n,bs", [(16, 0), (21, 5)])
@pytest.mark.parametrize("fmt", [L.FMT_U8, L.FMT_F16, L.FMT_F32])
def test_segments_without_an_apron(gpu_ctx, fmt, n, bs, W_, H_):
    """One pass per batch and sets, 16, 4 and 1 lanes per ray.  A table with an entry that is not
    finite (beyond the volume's values) keeps every sample on the clamping sampler: same image and
    count; and the single lattice march agrees to its rounding."""
    import torch

    for arm in ((33.0, 21.0, 2.2), (0.0, 0.0, 2.0), (200.0, -40.0, 1.3)):
        sc = _scene(fmt, n, bs, arm, W_, H_)
        b, p, view = sc.bricked, sc.volume_params(), sc.view()
        batches = []
        for ids in (b.order[0::2], b.order[1::2]):
            if len(ids) == 0:
                continue
            pool = b.pool[b.vaddr.reshape(-1)[ids]]
            va = np.full(b.vaddr.shape, -1, np.int32)
            va.reshape(-1)[ids] = np.arange(len(ids), dtype=np.int32)
            t = torch.from_numpy(pool.view(np.int16) if pool.dtype == np.uint16 else pool).cuda()
            batches.append((fmt, b.pad, t, va, b.page_k[:1].repeat(len(ids)), np.repeat(b.page_b[:1], len(ids), axis=0)))
        clamped = TF.copy()
        clamped[-1, :3] = np.inf
        out = []
        for tf in (clamped, TF):
            gpu_ctx.load(b, tf)
            sset = gpu_ctx.segment_set(batches)
            for render, arg in ((gpu_ctx.render_sort_last_set, (sset,)),
                                (gpu_ctx.render_sort_last_resident, (batches, b.grid))):
                rgba, n_samples = render(p, view, W_, H_, *arg, count=True)
                out.append((rgba.clone(), int(n_samples.item())))
            sset.close()
        for rgba, n_samples in out[1:]:
            assert n_samples == out[0][1] > 0
            assert torch.equal(rgba, out[0][0])
        gpu_ctx.load(b, TF)
        one = gpu_ctx.render_volume(p, view, W_, H_, film=False, count=True)
        assert int(one["samples"].item()) == out[0][1]
        assert float((one["rgba"] - out[0][0]).abs().max()) <= 1e-5
