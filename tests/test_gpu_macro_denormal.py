"""Macrocells of volumes whose values are denormal: half the least denormal rounds to zero, so that
samples lie on zero where every voxel is above or below it."""
import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import dataset as D
from hydrant_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sign", [-1.0, 1.0])
@pytest.mark.parametrize("W_,H_", [(61, 43), (163, 157), (641, 621)])
def test_least_denormals(gpu_ctx, W_, H_, sign):
    import torch

    n = 70
    vol = (np.float32(sign) * np.random.default_rng(3).choice(np.float32([1.4e-45, 2.8e-45]), (n, n, n))).astype(np.float32)
    b = D.make_bricked(vol, n, 0, L.FMT_F32, None, resident=1.0, seed=5)
    tf = np.array([[1, 0.5, 0.2, 0.3]] + [[0, 0, 0, 0]] * 7, np.float32)   # a colour at zero alone
    sc = W.Scene("denormal", b, tf, W_, H_, (33.0, 21.0, 2.2), 60.0, D.geometry((n, n, n), n, 0.5), density=0.1,
                 extra={"isovalue": 0.0, "corrected": 1, "bisect_steps": 8})
    t = torch.from_numpy(b.pool).cuda()
    out = []
    for owned in (True, False):
        gpu_ctx.load(b, tf)
        if not owned:
            gpu_ctx.bind_pool_device(b.fmt, b.pad, b.n_pages, t.data_ptr())
        r = gpu_ctx.render_volume(sc.volume_params(), sc.view(), W_, H_, film=False, count=True)
        i = gpu_ctx.render_iso(W.iso_params(sc), sc.view(), W_, H_, count=True)
        out.append((r["rgba"].clone(), i["px"].view(torch.int32).clone(), int(r["samples"].item()),
                    int(i["samples"].item())))
    assert out[0][2] == out[1][2] > 0 and out[0][3] == out[1][3] > 0
    assert torch.equal(out[0][0], out[1][0]) and bool((out[1][0] > 0).any())
    assert torch.equal(out[0][1], out[1][1])
