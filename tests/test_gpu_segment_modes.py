"""Segment sets in the modes that recolour samples: Paging colours a sample by its page's id in the
batch that holds it, so a set renders what one pass per batch does."""
import ctypes as C

import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import dataset as D
from hydrant_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", [L.MODE_PAGING, L.MODE_PARTITION])
@pytest.mark.parametrize("overlap", [False, True])
@pytest.mark.parametrize("W_,H_", [(37, 29), (163, 157), (1001, 997)])
def test_set_colours_as_its_passes(gpu_ctx, W_, H_, overlap, mode):
    import torch

    n, lowest = 40, 20
    vol = D.gen_blobs(n, 6, 31, sig=(4.0, 10.0), sigma_scale=n / 32.0, amp=(0.4, 1.0))
    b = D.make_bricked(vol, 8, 1, L.FMT_U8, None, resident=1.0, seed=5)
    sc = W.Scene("modes", b, D.README_TF.copy(), W_, H_, (33.0, 21.0, 2.2), 60.0, D.geometry((n, n, n), 8, 0.5),
                 density=0.2, schedule=L.SCHED_LATTICE, mode=mode, rank=0.25)
    order = b.order
    parts = [order[0::3], order[1::3], order[2::3]]   # 42, 42 and 41 pages: ids on both sides of `lowest` in each
    if overlap:
        parts[1] = np.concatenate([parts[1], parts[0][:2]])
    ctx, p, view = gpu_ctx, sc.volume_params(), sc.view()
    slots_n = int(sum(b.grid))
    batches = []
    for ids in parts:
        va = np.full(b.vaddr.shape, -1, np.int32)
        va.reshape(-1)[ids] = np.arange(len(ids), dtype=np.int32)
        batches.append((L.FMT_U8, b.pad, torch.from_numpy(b.pool[b.vaddr.reshape(-1)[ids]]).cuda(), va,
                        b.page_k[:1].repeat(len(ids)), np.repeat(b.page_b[:1], len(ids), axis=0)))
    b.lowest_blkcnt = lowest
    ctx.load(b, sc.tf)
    sset = ctx.segment_set(batches)
    ctx.sync_stream()
    res = []
    for one_launch in (True, False):
        slots = torch.empty((slots_n, H_, W_, 4), device="cuda")
        nslots = torch.zeros((H_, W_), dtype=torch.int32, device="cuda")
        L.call("hyd_segments_begin", ctx.h, W_, H_, slots_n, C.c_void_p(slots.data_ptr()))
        out = (W_, H_, slots_n, C.c_void_p(slots.data_ptr()), C.c_void_p(nslots.data_ptr()), C.c_void_p(0))
        if one_launch:
            L.call("hyd_segments_pass_set", ctx.h, sset.h, C.byref(p), C.byref(view), *out)
        else:
            for fmt, pad, t, va, k, pb in batches:
                ctx.bind_pool_device(fmt, pad, t.shape[0], t.data_ptr())
                ctx.set_page_table(va, k, pb, lowest)
                L.call("hyd_segments_pass", ctx.h, C.byref(p), C.byref(view), *out)
        ctx.synchronize()
        res.append((slots, nslots))
    sset.close()
    assert torch.equal(res[0][1], res[1][1])
    assert torch.equal(res[0][0], res[1][0])
    # the mode's colours are there: an image of one colour would not tell the ids apart
    filled = res[0][0][res[0][0][..., 3] > 0]
    if mode == L.MODE_PAGING:
        assert bool((filled[:, 0] > 0).any()) and bool((filled[:, 1] > 0).any())
