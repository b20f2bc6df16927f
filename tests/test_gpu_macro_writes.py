"""Pages written between renders: frames, lattice frames, isosurfaces and batches follow, whatever the
order and number of the writes and of the state changes between them, and equal those of a bound
pool (sampled throughout)."""
import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import dataset as D
from hydrant_amd import workloads as W
from hydrant_amd.hip import Context, batch_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [L.FMT_U8, L.FMT_F16, L.FMT_F32])
@pytest.mark.parametrize("seed", range(4))
def test_writes_between_renders(gpu_ctx, fmt, seed):
    import torch

    rng = np.random.default_rng(seed)
    n, bs, W_, H_ = 40, 4, 61, 43   # 1000 pages: more scattered writes than one launch lists
    vols = []
    for k in (0, 1):
        vol = D.gen_blobs(n, 3, 9 + k, sig=(3.0, 6.0), sigma_scale=n / 32.0, amp=(0.4, 1.0))
        if fmt != L.FMT_U8:
            vol = vol.astype(np.float32) / np.float32(255)
            vol = vol.astype(np.float16).view(np.uint16) if fmt == L.FMT_F16 else vol
        vols.append(D.make_bricked(vol, bs, 1, fmt, None, resident=1.0, seed=5))
    b, other = vols
    blank = np.zeros_like(b.pool)
    tfs = [D.README_TF.copy(), D.README_TF[::-1].copy()]
    tfs[1][3:6, 3] = 0.0
    geom = D.geometry((n,) * 3, bs, 0.5)
    scenes = [W.Scene("w", b, tfs[0], W_, H_, (40.0, 15.0, 2.2), 60.0, geom, density=0.1, schedule=s,
                      extra={"isovalue": 0.3, "corrected": 1, "bisect_steps": 8})
              for s in (L.SCHED_REFERENCE, L.SCHED_LATTICE)]
    view = scenes[0].view()
    desc = {"grid": b.grid, "bs": bs, "apron": 1, "bbox_max": geom.f_dim, "step": geom.step,
            "value_scale": 1 / 255.0 if fmt == L.FMT_U8 else 1.0, "vaddr": b.vaddr, "cheb": b.cheb}

    def renders(ctx, batch, what):
        if what == "batch":
            return batch.render(batch_config(8, 4, 8, 1), 0.1, 0.0)[0].view(torch.int32).clone()
        if what == "iso":
            return ctx.render_iso(W.iso_params(scenes[0]), view, W_, H_)["px"].view(torch.int32).clone()
        p = scenes[what == "lattice"].volume_params()
        out = ctx.render_volume(p, view, W_, H_, film=True, count=True)
        return torch.cat([out["film"].view(torch.int32).reshape(-1), out["samples"].view(torch.int32)])

    owned, pool, tf = Context(0), blank.copy(), 0
    owned.load(b, tfs[0])
    owned.upload_pool(fmt, b.pad, pool)
    owned.set_volumes([desc])
    batch = owned.batch([(view, W_, H_, 0)])
    for step in range(14):
        op = rng.choice(["run", "scatter", "overlap", "tf", "upload", "none"])
        src = [b.pool, other.pool, blank][int(rng.integers(0, 3))]
        if op == "run":
            f, k = int(rng.integers(0, 900)), int(rng.integers(1, 100))
            writes = [(f, k)]
        elif op == "scatter":
            writes = [(int(f), 1) for f in rng.permutation(1000)[:int(rng.integers(1, 200))]]
        elif op == "overlap":
            f = int(rng.integers(0, 900))
            writes = [(f, 20), (f + 10, 30), (f + 5, 3), (max(f - 4, 0), 60)]
        else:
            writes = []
        for f, k in writes:
            k = min(k, 1000 - f)
            pool[f:f + k] = src[f:f + k]
            owned.write_pool_pages(f, pool[f:f + k])
        if op == "tf":
            tf = 1 - tf
            owned.set_tf(tfs[tf])
        if op == "upload":
            pool[:] = src
            owned.upload_pool(fmt, b.pad, pool)
        bound = Context(0)
        t = torch.from_numpy(pool.view(np.int16) if pool.dtype == np.uint16 else pool).cuda()
        bound.load(b, tfs[tf])
        bound.bind_pool_device(fmt, b.pad, b.n_pages, t.data_ptr())
        bound.set_volumes([desc, dict(desc, value_scale=2 * desc["value_scale"])])   # no classes
        ref = bound.batch([(view, W_, H_, 0)])
        for what in rng.permutation(["frame", "lattice", "iso", "batch"])[:int(rng.integers(1, 5))]:
            assert torch.equal(renders(owned, batch, what), renders(bound, ref, what)), (step, op, what)
        torch.cuda.synchronize()
        ref.close()
        bound.close()
    batch.close()
    owned.close()
