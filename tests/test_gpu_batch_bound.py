"""Batches over a bound pool: where the renderer holds no copies of the pool's layouts it reads the
pool itself, and so follows contents changed in place."""
import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import workloads as W
from hydrant_amd.hip import Context, batch_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [L.FMT_U8, L.FMT_F16, L.FMT_F32])
def test_single_layout_follows_the_pool(monkeypatch, fmt):
    import torch

    monkeypatch.setenv("HYD_BATCH_SINGLE_LAYOUT", "1")
    wl = W.batched(sizes=(96,), n_views=3, res_choices=(64, 97), fmt=fmt, bs=32, apron=1, seed=11)
    pools = [np.ascontiguousarray(wl.pool), np.ascontiguousarray(wl.pool[::-1])]
    as_t = lambda p: torch.from_numpy(p.view(np.int16) if p.dtype == np.uint16 else p).cuda()
    pad = wl.bs + 2 * wl.apron
    bound, t = Context(0), as_t(pools[0])
    bound.bind_pool_device(fmt, pad, len(pools[0]), t.data_ptr())
    bound.set_volumes(wl.volume_descs())
    bound.set_tf(wl.tf)
    b = bound.batch(wl.hip_views())
    cfg = batch_config(8, 4, 8, 1)
    for pool in pools:
        t.copy_(as_t(pool))
        got = b.render(cfg, wl.density, 0.0)[0].clone()
        ref = Context(0)
        ref.upload_pool(fmt, pad, pool)
        ref.set_volumes(wl.volume_descs())
        ref.set_tf(wl.tf)
        rb = ref.batch(wl.hip_views())
        assert torch.equal(got, rb.render(cfg, wl.density, 0.0)[0]) and bool((got > 0).any())
        torch.cuda.synchronize()
        rb.close()
        ref.close()
    b.close()
    bound.close()
