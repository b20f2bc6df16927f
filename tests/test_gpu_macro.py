"""Marches over empty macrocells: a pool the context owns (whose macrocells it keeps) renders the
film, image and sample count of the same pool bound from outside (sampled throughout), bit for
bit, over formats, brick sizes, schedules, modes and cameras; the macrocells follow a new
transfer function and rewritten pages."""
import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import dataset as D
from hydrant_amd import workloads as W

pytestmark = pytest.mark.gpu


def _scene(n, fmt, bs, schedule, seed, density=1e-2, ert=0.0, mode=L.MODE_DEFAULT):
    rng = np.random.default_rng(seed)
    vol = D.gen_blobs(n, 3, seed, sig=(3.0, 6.0), sigma_scale=n / 32.0, amp=(0.4, 1.0))
    b = D.make_bricked(vol, bs or n, 1 if bs else 0, fmt, None, resident=1.0, seed=5)
    arm = (float(rng.uniform(0, 360)), float(rng.uniform(-80, 80)), float(rng.uniform(0.4, 2.6)))
    sc = W.Scene("macro", b, D.README_TF.copy(), 61, 43, arm, 60.0, D.geometry((n, n, n), bs or n, 0.5),
                 density=density, schedule=schedule, ert=ert, mode=mode, rank=0.25)
    b.lowest_blkcnt = b.n_pages // 2
    return sc


def _render(ctx, sc):
    import torch

    out = ctx.render_volume(sc.volume_params(), sc.view(), sc.W, sc.H, film=True, count=True)
    img = ctx.render_volume(sc.volume_params(), sc.view(), sc.W, sc.H, film=False)["rgba"]
    ctx.synchronize()
    return out["film"].view(torch.int32).clone(), out["rgba"].clone(), img.clone(), int(out["samples"].item())


def _bound(ctx, sc, tf=None):
    import torch

    b = sc.bricked
    t = torch.from_numpy(b.pool.view(np.int16) if b.pool.dtype == np.uint16 else b.pool).cuda()
    ctx.load(b, sc.tf if tf is None else tf)
    ctx.bind_pool_device(b.fmt, b.pad, b.n_pages, t.data_ptr())
    r = _render(ctx, sc)
    return r


def _equal(a, b):
    import torch

    assert a[3] == b[3] > 0
    for x, y in zip(a[:3], b[:3]):
        assert torch.equal(x, y)


@pytest.mark.parametrize("schedule,ert", [(L.SCHED_REFERENCE, 0.0), (L.SCHED_LATTICE, 0.0), (L.SCHED_LATTICE, 0.5)])
@pytest.mark.parametrize("fmt", [L.FMT_U8, L.FMT_F16, L.FMT_F32])
@pytest.mark.parametrize("n,bs", [(8, 0), (33, 0), (64, 0), (50, 7), (70, 16), (96, 32)])
def test_owned_equals_bound(gpu_ctx, fmt, n, bs, schedule, ert):
    for seed, density in ((n + bs, 1e-2), (n + bs + 1, 0.4)):
        sc = _scene(n, fmt, bs, schedule, seed, density, ert)
        ref = _bound(gpu_ctx, sc)
        gpu_ctx.load(sc.bricked, sc.tf)
        _equal(_render(gpu_ctx, sc), ref)


@pytest.mark.parametrize("mode", [L.MODE_PARTITION, L.MODE_PAGING])
def test_recoloured_modes(gpu_ctx, mode):
    sc = _scene(70, L.FMT_U8, 16, L.SCHED_REFERENCE, 9, 0.2, mode=mode)
    ref = _bound(gpu_ctx, sc)
    gpu_ctx.load(sc.bricked, sc.tf)
    _equal(_render(gpu_ctx, sc), ref)


def test_new_transfer_function_and_pages(gpu_ctx):
    """The same context through a table that empties another range, then rewritten pages, then a
    page table whose mappings differ (no macrocells apply)."""
    sc = _scene(70, L.FMT_F16, 16, L.SCHED_REFERENCE, 21, 0.1)
    b = sc.bricked
    tf2 = D.README_TF[::-1].copy()
    tf2[3:6, 3] = 0.0
    ref = _bound(gpu_ctx, sc, tf2)
    gpu_ctx.load(b, sc.tf)
    _render(gpu_ctx, sc)
    gpu_ctx.set_tf(tf2)
    _equal(_render(gpu_ctx, sc), ref)
    other = D.make_bricked(D.gen_blobs(70, 4, 77, sig=(3.0, 6.0), sigma_scale=2.0, amp=(0.4, 1.0)), 16, 1, L.FMT_F16,
                           None, resident=1.0, seed=5)
    first, n = 3, b.n_pages // 2
    gpu_ctx.write_pool_pages(first, other.pool[first:first + n])
    b.pool[first:first + n] = other.pool[first:first + n]
    got = _render(gpu_ctx, sc)
    _equal(got, _bound(gpu_ctx, sc, tf2))
    b.page_k[::2] *= np.float32(0.5)
    ref = _bound(gpu_ctx, sc, tf2)
    gpu_ctx.load(b, tf2)
    _equal(_render(gpu_ctx, sc), ref)


@pytest.mark.parametrize("corrected", [0, 1])
@pytest.mark.parametrize("fmt", [L.FMT_U8, L.FMT_F16, L.FMT_F32])
@pytest.mark.parametrize("n,bs", [(12, 8), (50, 7), (70, 16), (96, 32)])
def test_isosurface_owned_equals_bound(gpu_ctx, fmt, n, bs, corrected):
    import torch

    rng = np.random.default_rng(n + bs)
    if fmt == L.FMT_U8:
        vol, iso = D.gen_blobs(n, 3, n, sig=(3.0, 6.0), sigma_scale=n / 32.0, amp=(0.4, 1.0)), 0.3
    else:
        vol, iso = D.gen_sdf_spheres(n, 9, (2.0, n / 5.0), 2.0, n), 0.25
        if fmt == L.FMT_F32:
            vol = vol.view(np.float16).astype(np.float32)
            vol.reshape(-1)[rng.choice(vol.size, 20, replace=False)] = np.resize([np.nan, np.inf, -np.inf], 20)
    b = D.make_bricked(vol, bs, 1, fmt, None, resident=1.0, seed=5)
    arm = (float(rng.uniform(0, 360)), float(rng.uniform(-80, 80)), 2.2)
    sc = W.Scene("iso", b, np.zeros((1, 4), np.float32), 61, 43, arm, 60.0, D.geometry((n, n, n), bs, 1.0),
                 extra={"isovalue": iso, "corrected": corrected, "bisect_steps": 8})
    p = W.iso_params(sc)
    t = torch.from_numpy(b.pool.view(np.int16) if b.pool.dtype == np.uint16 else b.pool).cuda()
    res = []
    for owned in (False, True):
        gpu_ctx.load(b)
        if not owned:
            gpu_ctx.bind_pool_device(b.fmt, b.pad, b.n_pages, t.data_ptr())
        r = gpu_ctx.render_iso(p, sc.view(), sc.W, sc.H, count=True)
        gpu_ctx.synchronize()
        res.append((r["px"].view(torch.int32).clone(), int(r["samples"].item())))
    assert res[0][1] == res[1][1] > 0
    assert torch.equal(res[0][0], res[1][0])
