"""Four lanes a ray and macrocells in the batched renderer: the image and the sample count are
those of one lane a ray, and of the march that samples everything, bit for bit; the macrocells follow
a new transfer function and rewritten pages, eagerly and in a replayed graph."""
import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import workloads as W
from hydrant_amd.hip import Context, batch_config

pytestmark = pytest.mark.gpu

QUAD, ONE = batch_config(8, 4, 8), batch_config(16, 2, 8)


def _tf(clear):
    tf = np.random.default_rng(clear).uniform(0.1, 1.0, (16, 4)).astype(np.float32)
    tf[:clear, 3] = 0.0
    return tf


def _setup(wl, sampled):
    """A context; sampled: a second set of volumes names the same pages under another scale,
    so that no page has classes."""
    ctx = Context(0)
    ctx.upload_pool(wl.fmt, wl.bs + 2 * wl.apron, wl.pool)
    descs = wl.volume_descs()
    ctx.set_volumes(descs + [dict(d, value_scale=2.0 * d["value_scale"]) for d in descs] if sampled else descs)
    return ctx


@pytest.mark.parametrize("fmt", [L.FMT_U8, L.FMT_F16, L.FMT_F32])
@pytest.mark.parametrize("switch", [None, "HYD_BATCH_NO_QUADS"])
@pytest.mark.parametrize("ert,bs", [(0.0, 32), (0.9, 16)])
def test_lanes_and_macrocells_render_the_same(monkeypatch, fmt, switch, ert, bs):
    import torch

    if switch:
        monkeypatch.setenv(switch, "1")
    wl = W.batched(sizes=(40, 96), n_views=5, res_choices=(33, 64, 97), fmt=fmt, bs=bs, apron=1, seed=11)
    ctxs = [_setup(wl, False), _setup(wl, True)]
    pool = np.ascontiguousarray(wl.pool).copy()
    for clear in (3, 9):
        got = []
        for ctx in ctxs:
            ctx.set_tf(_tf(clear))
            b = ctx.batch(wl.hip_views())
            for cfg in (QUAD, ONE):
                out, cnt = b.render(cfg, wl.density, ert, count=True)
                got.append((out.clone(), int(cnt.item())))
            b.close()
        for out, cnt in got[1:]:
            assert cnt == got[0][1], clear
            assert torch.equal(out, got[0][0]), clear
        for ctx in ctxs:   # the second table finds other pages
            pool[1:3] = pool[1:3][::-1].copy() if ctx is ctxs[0] else pool[1:3]
            ctx.write_pool_pages(1, pool[1:3])
    for ctx in ctxs:
        ctx.close()


def test_replays_follow_rewritten_pages():
    import torch

    wl = W.batched(sizes=(64, 64), n_views=4, res_choices=(48, 64), fmt=L.FMT_U8, bs=16, apron=1, seed=3)
    ctxs = [_setup(wl, False), _setup(wl, True)]
    for ctx in ctxs:
        ctx.set_tf(_tf(6))
    b, ref = [ctx.batch(wl.hip_views()) for ctx in ctxs]
    out = b.new_output()
    b.capture(QUAD, wl.density, wl.ert, out)
    pool = np.ascontiguousarray(wl.pool)
    n = pool.shape[0]
    for rep in range(4):
        new = np.ascontiguousarray(np.roll(pool, rep, axis=0))   # empty pages become full and back
        for ctx in ctxs:
            ctx.write_pool_pages(0, new[: n // 2])
        out.fill_(-1.0)
        b.replay()
        want = ref.render(ONE, wl.density, wl.ert)[0]
        torch.cuda.synchronize()
        assert torch.equal(out, want), rep
    for x in (b, ref, *ctxs):
        x.close()
