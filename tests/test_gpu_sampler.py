"""The march's samplers at their edges, bit for bit against the oracle: tap weights of exactly
zero (rays along an axis through voxel centres), voxels and transfer-function entries that are
not finite, page faces, and the register form of the u8 normalisation."""
import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import dataset as D
from hydrant_amd import workloads as W
from tests.helpers import film_fields, oracle_film_fields, oracle_view, oracle_volume

pytestmark = pytest.mark.gpu


def _scene(n, fmt, bs, arm, density=1e-2, tf=None, poke=None, W_=37, H_=29):
    vol = D.gen_blobs(n, 6, 31, sig=(4.0, 10.0), sigma_scale=n / 32.0, amp=(0.4, 1.0))
    if fmt == L.FMT_F32:
        vol = vol.astype(np.float32) / np.float32(255)
    elif fmt == L.FMT_F16:
        vol = (vol.astype(np.float32) / np.float32(255)).astype(np.float16).view(np.uint16)
    if poke is not None:
        flat = vol.reshape(-1)
        v = flat if fmt == L.FMT_F32 else flat.view(np.float16)
        at = np.random.default_rng(3).choice(flat.size, flat.size // 50, replace=False)
        v[at] = np.resize(np.array(poke, v.dtype), at.size)
    b = D.make_bricked(vol, bs or n, 1 if bs else 0, fmt, None, resident=1.0, seed=5)
    geom = D.geometry((n, n, n), bs or n, 0.5)
    return W.Scene("sampler", b, D.README_TF.copy() if tf is None else tf, W_, H_, arm, 60.0, geom, density=density)


def _same(a, b):
    a, b = np.asarray(a, np.float32), np.asarray(b, np.float32)
    return np.array_equal(a, b, equal_nan=True)


def _check(ctx, sc):
    ctx.load(sc.bricked, sc.tf)
    out = ctx.render_volume(sc.volume_params(), sc.view(), sc.W, sc.H, film=True, count=True)
    img = ctx.render_volume(sc.volume_params(), sc.view(), sc.W, sc.H, film=False)["rgba"].cpu().numpy()
    g = film_fields(out["film"].cpu().numpy())
    with np.errstate(all="ignore"):
        r = oracle_volume(sc).render(oracle_view(sc), 32, film=True)
        o = oracle_film_fields(r["film"])
    assert int(out["samples"].item()) == r["samples"] > 0
    assert _same(img, r["rgba"])
    for k in ("v", "theta", "phi", "o"):
        assert _same(g[k], o[k]), k
    assert np.array_equal(g["nsteps"], o["nsteps"]) and np.array_equal(g["step_size"], o["step_size"])


AXIS = [(0.0, 0.0, 2.2), (90.0, 0.0, 2.2), (33.0, 21.0, 2.2)]


@pytest.mark.parametrize("arm", AXIS)
@pytest.mark.parametrize("fmt,n,bs", [(L.FMT_F32, 25, 0), (L.FMT_F32, 33, 16), (L.FMT_F16, 25, 0), (L.FMT_F16, 48, 16),
                                      (L.FMT_U8, 25, 0), (L.FMT_U8, 33, 16), (L.FMT_U8, 5, 0)])
def test_zero_weights_and_faces(gpu_ctx, fmt, n, bs, arm):
    _check(gpu_ctx, _scene(n, fmt, bs, arm))


@pytest.mark.parametrize("arm", AXIS)
@pytest.mark.parametrize("fmt,bs", [(L.FMT_F32, 0), (L.FMT_F32, 8), (L.FMT_F16, 0), (L.FMT_F16, 8)])
def test_voxels_that_are_not_finite(gpu_ctx, fmt, bs, arm):
    _check(gpu_ctx, _scene(25, fmt, bs, arm, poke=[np.nan, np.inf, -np.inf, -1.0, 3.0]))


@pytest.mark.parametrize("fmt,bs", [(L.FMT_F32, 0), (L.FMT_U8, 16)])
@pytest.mark.parametrize("bad", [(3, 1, np.inf), (4, 2, np.nan), (5, 3, -0.5), (2, 3, 40.0)])
def test_transfer_functions_outside_the_unit_range(gpu_ctx, fmt, bs, bad):
    tf = D.README_TF.copy()
    tf[bad[0], bad[1]] = bad[2]
    _check(gpu_ctx, _scene(25, fmt, bs, AXIS[2], density=1.0, tf=tf))


def test_u8_normalisation_of_every_count(gpu_ctx):
    """A volume holding every count, read at voxel centres: the alpha of a linear table."""
    vol = np.arange(256, dtype=np.uint8).repeat(108)[: 30 ** 3 - 30 ** 3 % 27].tolist()
    vol = np.resize(np.array(vol, np.uint8), (30, 30, 30))
    b = D.single_brick(vol, L.FMT_U8)
    tf = np.stack([np.linspace(0, 1, 256)] * 3 + [np.linspace(0, 0.5, 256)], 1).astype(np.float32)
    sc = W.Scene("u8", b, tf, 33, 31, AXIS[2], 60.0, D.geometry((30, 30, 30), 30, 0.5), density=0.1)
    _check(gpu_ctx, sc)


@pytest.mark.parametrize("fmt", [L.FMT_F32, L.FMT_F16, L.FMT_U8])
@pytest.mark.parametrize("W_,H_", [(1, 1), (5, 3), (3, 8191), (163, 157), (641, 621)])
def test_lanes_per_ray(gpu_ctx, fmt, W_, H_):
    """Frames of few, some and many rays (16, 4 and 1 lanes per ray), with partial tiles, at a
    density where steps escalate inside groups."""
    sc = _scene(24, fmt, 8, AXIS[2], density=0.5, W_=W_, H_=H_)
    if (W_, H_) != (3, 8191):
        return _check(gpu_ctx, sc)
    ctx = gpu_ctx          # a sliver: the oracle's image alone
    ctx.load(sc.bricked, sc.tf)
    img = ctx.render_volume(sc.volume_params(), sc.view(), sc.W, sc.H, film=False)["rgba"].cpu().numpy()
    assert _same(img, oracle_volume(sc).render(oracle_view(sc), 32, film=False)["rgba"])


@pytest.mark.parametrize("fmt", [L.FMT_F32, L.FMT_U8])
@pytest.mark.parametrize("W_,H_", [(37, 29), (163, 157), (641, 621)])
def test_lattice_lanes_per_ray(gpu_ctx, fmt, W_, H_):
    """The lattice march at each number of lanes per ray: samples and counts of the oracle's (1e-4
    for its rounding, as the lattice tests)."""
    sc = _scene(24, fmt, 8, AXIS[2], density=0.2, W_=W_, H_=H_)
    sc.schedule, sc.ert = L.SCHED_LATTICE, 0.9
    gpu_ctx.load(sc.bricked, sc.tf)
    out = gpu_ctx.render_volume(sc.volume_params(), sc.view(), sc.W, sc.H, film=True, count=True)
    r = oracle_volume(sc).render(oracle_view(sc), 32, film=False)
    assert int(out["samples"].item()) == r["samples"] > 0
    assert np.max(np.abs(out["rgba"].cpu().numpy() - r["rgba"])) <= 1e-4


@pytest.mark.parametrize("fmt", [L.FMT_U8, L.FMT_F16, L.FMT_F32])
@pytest.mark.parametrize("W_,H_,overlap", [(37, 29, False), (163, 157, False), (163, 157, True), (1201, 621, False)])
def test_segment_sets_at_every_lane_count(gpu_ctx, fmt, W_, H_, overlap):
    """A segment set (one walk for all batches; one pass each when two batches hold a brick) fills
    the slots of one pass per batch, at 16, 4 and 1 lanes per ray: image and counts bit for bit."""
    import torch

    sc = _scene(40, fmt, 8, AXIS[2], density=0.2, W_=W_, H_=H_)
    sc.schedule = L.SCHED_LATTICE
    b = sc.bricked
    order = b.order
    parts = [order[0::3], order[1::3], order[2::3]]
    if overlap:
        parts[1] = np.concatenate([parts[1], parts[0][:2]])
    batches = []
    for ids in parts:
        pool = b.pool[b.vaddr.reshape(-1)[ids]]
        va = np.full(b.vaddr.shape, -1, np.int32)
        va.reshape(-1)[ids] = np.arange(len(ids), dtype=np.int32)
        t = torch.from_numpy(pool.view(np.int16) if pool.dtype == np.uint16 else pool).cuda()
        batches.append((fmt, b.pad, t, va, b.page_k[:1].repeat(len(ids)), np.repeat(b.page_b[:1], len(ids), axis=0)))
    gpu_ctx.load(b, sc.tf)
    p, view = sc.volume_params(), sc.view()
    ref, rc = gpu_ctx.render_sort_last_resident(p, view, W_, H_, batches, b.grid, count=True)
    gpu_ctx.load(b, sc.tf)
    sset = gpu_ctx.segment_set(batches)
    got, gc = gpu_ctx.render_sort_last_set(p, view, W_, H_, sset, count=True)
    gpu_ctx.synchronize()
    assert int(rc.item()) == int(gc.item()) > 0
    assert torch.equal(ref, got)
    if not overlap:
        one = gpu_ctx.render_volume(p, view, W_, H_, film=False, count=True)
        assert int(one["samples"].item()) == int(gc.item())
        assert float((one["rgba"] - got).abs().max()) <= 1e-5
    sset.close()
