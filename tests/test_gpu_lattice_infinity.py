"""Opacities that are not finite in the lattice march and the segments: without a termination alpha
no alpha ends a ray or a segment, so samples are the oracle's and infinities turn to NaN where its
do."""
import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import dataset as D
from hydrant_amd import workloads as W
from tests.helpers import oracle_view, oracle_volume

pytestmark = pytest.mark.gpu


def _kinds(a):
    a = np.asarray(a, np.float32)
    return np.where(np.isnan(a), 3, np.where(np.isposinf(a), 2, np.where(np.isneginf(a), 1, 0)))


@pytest.mark.parametrize("W_,H_", [(37, 29), (163, 157), (1001, 997)])
@pytest.mark.parametrize("ert", [0.0, 0.9, np.inf])
def test_infinite_opacity(gpu_ctx, ert, W_, H_):
    import torch

    n = 24
    vol = D.gen_blobs(n, 6, 31, sig=(4.0, 10.0), sigma_scale=n / 32.0, amp=(0.4, 1.0))
    b = D.make_bricked(vol, 8, 1, L.FMT_U8, None, resident=1.0, seed=5)
    tf = D.README_TF.copy()
    tf[-3, 3] = np.inf
    sc = W.Scene("inf", b, tf, W_, H_, (33.0, 21.0, 2.2), 60.0, D.geometry((n, n, n), 8, 0.5), density=0.2,
                 schedule=L.SCHED_LATTICE, ert=ert)
    ctx = gpu_ctx
    ctx.load(b, tf)
    out = ctx.render_volume(sc.volume_params(), sc.view(), W_, H_, film=True, count=True)
    with np.errstate(all="ignore"):
        r = oracle_volume(sc).render(oracle_view(sc), 32, film=False)
    got = out["rgba"].cpu().numpy()
    assert int(out["samples"].item()) == r["samples"] > 0
    kinds = _kinds(r["rgba"])
    assert (kinds == 3).any() or ert == np.float32(0.9)
    assert np.array_equal(_kinds(got), kinds)
    finite = kinds == 0
    assert np.max(np.abs(got[finite] - r["rgba"][finite])) <= 1e-4
    if ert == 0.0:   # segments have no termination
        t = torch.from_numpy(b.pool).cuda()
        batch = [(L.FMT_U8, b.pad, t, b.vaddr, b.page_k, b.page_b)]
        sset = ctx.segment_set(batch)
        _, ns = ctx.render_sort_last_set(sc.volume_params(), sc.view(), W_, H_, sset, count=True)
        _, nr = ctx.render_sort_last_resident(sc.volume_params(), sc.view(), W_, H_, batch, b.grid, count=True)
        assert int(ns.item()) == int(nr.item()) == r["samples"]
        sset.close()
