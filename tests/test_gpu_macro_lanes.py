"""Macrocells passed over at 16, 4 and 1 lanes per ray (and in the handover of a wave's last rays):
volumes mostly empty, so that the lookups are on, in pages large enough for them; films, images and
counts of an owned pool are those of the bound one, bit for bit, in one pass and resumed."""
import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import dataset as D
from hydrant_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("schedule,ert", [(L.SCHED_REFERENCE, 0.0), (L.SCHED_LATTICE, 0.0), (L.SCHED_LATTICE, 0.5)])
@pytest.mark.parametrize("W_,H_", [(61, 43), (163, 157), (641, 621), (1201, 990)])
@pytest.mark.parametrize("fmt,bs", [(L.FMT_U8, 48), (L.FMT_F16, 0), (L.FMT_F32, 48)])
def test_sparse_volumes(gpu_ctx, fmt, bs, W_, H_, schedule, ert):
    import torch

    n = 96
    vol = D.gen_blobs(n, 3, 17, sig=(3.0, 6.0), sigma_scale=1.5, amp=(0.4, 1.0))
    if fmt != L.FMT_U8:
        vol = vol.astype(np.float32) / np.float32(255)
        vol = vol.astype(np.float16).view(np.uint16) if fmt == L.FMT_F16 else vol
    b = D.make_bricked(vol, bs or n, 1 if bs else 0, fmt, None, resident=1.0, seed=5)
    tf = D.README_TF.copy()
    tf[: len(tf) // 4, 3] = 0.0
    sc = W.Scene("sparse", b, tf, W_, H_, (40.0, 15.0, 1.9), 60.0, D.geometry((n,) * 3, bs or n, 0.5), density=0.3,
                 schedule=schedule, ert=ert)
    ctx, p, view = gpu_ctx, sc.volume_params(), sc.view()
    t = torch.from_numpy(b.pool.view(np.int16) if b.pool.dtype == np.uint16 else b.pool).cuda()
    part = b.vaddr.copy()
    part[np.random.default_rng(5).random(part.shape) < 0.5] = -1
    out = []
    for owned in (True, False):
        ctx.load(b, tf)
        if not owned:
            ctx.bind_pool_device(b.fmt, b.pad, b.n_pages, t.data_ptr())
        whole = ctx.render_volume(p, view, W_, H_, film=True, count=True)
        image = ctx.render_volume(p, view, W_, H_, film=False)["rgba"]
        ctx.set_page_table(part, b.page_k, b.page_b)
        film = ctx.render_volume(p, view, W_, H_, film=True)["film"]
        ctx.set_page_table(b.vaddr, b.page_k, b.page_b)
        film = ctx.resume_volume(p, film)["film"]
        out.append([x.view(torch.int32).clone() for x in (whole["film"], whole["samples"], image, film)])
    for x, y in zip(*out):
        assert torch.equal(x, y)
    assert bool((out[0][2] != 0).any())
