"""Segment sets whose pools lie far apart: the offsets reach them, the launch is chosen by what the
pools hold, and the image is that of the same pools side by side."""
import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import dataset as D
from hydrant_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [L.FMT_U8, L.FMT_F16, L.FMT_F32])
@pytest.mark.parametrize("W_,H_", [(37, 29), (163, 157), (1001, 997)])
def test_pools_six_gib_apart(gpu_ctx, fmt, W_, H_):
    import torch

    n = 40
    vol = D.gen_blobs(n, 6, 31, sig=(4.0, 10.0), sigma_scale=n / 32.0, amp=(0.4, 1.0))
    if fmt != L.FMT_U8:
        vol = vol.astype(np.float32) / np.float32(255)
        vol = vol.astype(np.float16).view(np.uint16) if fmt == L.FMT_F16 else vol
    b = D.make_bricked(vol, 8, 1, fmt, None, resident=1.0, seed=5)
    sc = W.Scene("far", b, D.README_TF.copy(), W_, H_, (33.0, 21.0, 2.2), 60.0, D.geometry((n, n, n), 8, 0.5),
                 density=0.2, schedule=L.SCHED_LATTICE)
    big = torch.empty((6 << 30) + (64 << 20), dtype=torch.uint8, device="cuda")
    gpu_ctx.load(b, sc.tf)
    out = []
    for gap in (0, 6 << 30):
        batches = []
        for j in range(2):
            ids = b.order[j::2]
            pool = b.pool[b.vaddr.reshape(-1)[ids]]
            va = np.full(b.vaddr.shape, -1, np.int32)
            va.reshape(-1)[ids] = np.arange(len(ids), dtype=np.int32)
            t = torch.from_numpy(pool.view(np.int16) if pool.dtype == np.uint16 else pool).cuda()
            if gap:
                size = t.numel() * t.element_size()
                far = big[j * gap:j * gap + size].view(t.dtype).view(t.shape)
                far.copy_(t)
                t = far
            batches.append((fmt, b.pad, t, va, b.page_k[:1].repeat(len(ids)), np.repeat(b.page_b[:1], len(ids), axis=0)))
        sset = gpu_ctx.segment_set(batches)
        rgba, cnt = gpu_ctx.render_sort_last_set(sc.volume_params(), sc.view(), W_, H_, sset, count=True)
        out.append((rgba.clone(), int(cnt.item())))
        sset.close()
    assert out[0][1] == out[1][1] > 0
    assert torch.equal(out[0][0], out[1][0])
