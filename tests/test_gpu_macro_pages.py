"""Pools of very many pages: the macrocells of every page are made, whatever the number."""
import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import dataset as D
from hydrant_amd import hip
from hydrant_amd.hip import Context

pytestmark = pytest.mark.gpu


def test_pool_of_16_million_pages():
    """2^24 + 5 pages of 2^3 voxels (256 threads a page pass 2^32): taken, and its last pages render
    as in a bound pool, which is sampled throughout."""
    import torch

    n, g, W_, H_ = (1 << 24) + 5, 8, 61, 43
    rng = np.random.default_rng(3)
    pool = np.zeros((n, 2, 2, 2), np.uint8)
    used = g ** 3
    pool[-used:] = rng.integers(0, 256, (used, 1, 1, 1)) * (rng.random((used, 1, 1, 1)) < 0.5)
    vaddr = (n - used + np.arange(used, dtype=np.int32)).reshape(g, g, g)
    k, b = np.ones(n, np.float32), np.zeros((n, 3), np.float32)
    tf = np.array([[0, 0, 0, 0], [0.2, 0.5, 1, 0], [1, 1, 1, 0.5], [1, 0.2, 0.1, 0.2]], np.float32)
    geom = D.geometry((2 * g,) * 3, 2, 0.5)
    view = hip.make_view(hip.orbit_camera((33.0, 21.0, 2.2)), geom.center, geom.f_dim)
    p = hip.volume_params((0.0, 0.0, 0.0), geom.f_dim, geom.step, geom.du, density=0.3)
    ctx, images = Context(0), []
    bound = torch.from_numpy(pool).cuda()
    for owned in (True, False):
        if owned:
            ctx.upload_pool(L.FMT_U8, 2, pool)
        else:
            ctx.bind_pool_device(L.FMT_U8, 2, n, bound.data_ptr())
        ctx.set_page_table(vaddr, k, b)
        ctx.set_empty_grid(np.zeros((g, g, g), np.int32))
        ctx.set_tf(tf)
        out = ctx.render_volume(p, view, W_, H_, film=False, count=True)
        images.append((out["rgba"].clone(), int(out["samples"].item())))
    ctx.close()
    assert images[0][1] == images[1][1] > 0
    assert torch.equal(images[0][0], images[1][0]) and bool((images[0][0] > 0).any())


@pytest.mark.parametrize("fmt", [L.FMT_U8, L.FMT_F16, L.FMT_F32])
@pytest.mark.parametrize("n", [2, 3, 4, 5, 9, 17, 67, 131, 257])
def test_ranges_at_odd_page_edges(gpu_ctx, fmt, n):
    """One page of every kind of edge (below and above the four-voxel loads and the macrocell's
    eight), with single contributing voxels that a lost column or row would drop."""
    import torch

    rng = np.random.default_rng(n)
    vol = np.zeros((n, n, n), np.uint8)
    for _ in range(12):   # faces and corners among them
        vol[tuple(int(rng.choice([0, n - 1, int(rng.integers(0, n))])) for _ in range(3))] = 255
    if fmt != L.FMT_U8:
        vol = vol.astype(np.float32) / np.float32(255)
        vol = vol.astype(np.float16).view(np.uint16) if fmt == L.FMT_F16 else vol
    b = D.single_brick(vol, fmt)
    tf = np.array([[0, 0, 0, 0]] * 2 + [[1, 0.5, 0.2, 0.4]] * 6, np.float32)
    geom = D.geometry((n,) * 3, n, 0.5)
    p = hip.volume_params((0.0, 0.0, 0.0), geom.f_dim, geom.step, geom.du, density=0.5)
    t = torch.from_numpy(b.pool.view(np.int16) if b.pool.dtype == np.uint16 else b.pool).cuda()
    for arm, size in (((33.0, 21.0, 2.2), (61, 43)), ((200.0, -50.0, 1.2), (163, 157)), ((0.0, 0.0, 2.0), (641, 621))):
        view = hip.make_view(hip.orbit_camera(arm), geom.center, geom.f_dim)
        images = []
        for owned in (True, False):
            gpu_ctx.load(b, tf)
            if not owned:
                gpu_ctx.bind_pool_device(b.fmt, b.pad, b.n_pages, t.data_ptr())
            out = gpu_ctx.render_volume(p, view, *size, film=False, count=True)
            images.append((out["rgba"].clone(), int(out["samples"].item())))
        assert images[0][1] == images[1][1] > 0
        assert torch.equal(images[0][0], images[1][0])
