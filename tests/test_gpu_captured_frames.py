"""Frames, resumes, isosurfaces and segment passes captured in a caller's HIP graph: a replay renders
with the page table as it is then (hyd_set_page_table rewrites it in place), also when its mappings
differ from those at the capture."""
import ctypes as C

import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import dataset as D
from hydrant_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mapping", ["half", "whole"])   # "whole": taps that clamp at the page's faces
@pytest.mark.parametrize("what", ["frame", "lattice", "resume", "iso", "segments"])
@pytest.mark.parametrize("W_,H_", [(61, 43), (641, 621)])
def test_replay_follows_the_page_table(gpu_ctx, what, mapping, W_, H_):
    import torch

    n, bs = 70, 16
    vol = D.gen_blobs(n, 3, 9, sig=(3.0, 6.0), sigma_scale=n / 32.0, amp=(0.4, 1.0))
    b = D.make_bricked(vol, bs, 1, L.FMT_U8, None, resident=1.0, seed=5)
    sc = W.Scene("graph", b, D.README_TF.copy(), W_, H_, (40.0, 15.0, 2.2), 60.0, D.geometry((n, n, n), bs, 0.5),
                 density=0.1, schedule=L.SCHED_LATTICE if what in ("lattice", "segments") else L.SCHED_REFERENCE,
                 extra={"isovalue": 0.3, "corrected": 1, "bisect_steps": 8})
    k2, b2 = b.page_k.copy(), b.page_b.copy()
    if mapping == "half":
        k2[::2] *= np.float32(0.5)
    else:
        k2[::2], b2[::2] = np.float32(1.0), np.float32(0.0)
    ctx, p, view = gpu_ctx, sc.volume_params(), sc.view()
    ctx.load(b, sc.tf)
    film0 = None
    if what == "resume":
        ctx.set_page_table(np.full_like(b.vaddr, -1), b.page_k, b.page_b)
        film0 = ctx.render_volume(p, view, W_, H_, film=True)["film"]
        ctx.set_page_table(b.vaddr, b.page_k, b.page_b)
    slots_n = int(sum(b.grid))

    def run(film, slots, nslots):
        if what in ("frame", "lattice"):
            return ctx.render_volume(p, view, W_, H_, film=False)["rgba"]
        if what == "resume":
            film.copy_(film0)
            return ctx.resume_volume(p, film)["rgba"]
        if what == "iso":
            return ctx.render_iso(W.iso_params(sc), view, W_, H_)["px"]
        ctx.sync_stream()
        L.call("hyd_segments_begin", ctx.h, W_, H_, slots_n, C.c_void_p(slots.data_ptr()))
        L.call("hyd_segments_pass", ctx.h, C.byref(p), C.byref(view), W_, H_, slots_n, C.c_void_p(slots.data_ptr()),
               C.c_void_p(nslots.data_ptr()), C.c_void_p(0))
        return slots

    def buffers():
        return (torch.empty((H_, W_, 16), device="cuda"),
                torch.empty((slots_n if what == "segments" else 1, H_, W_, 4), device="cuda"),
                torch.empty((H_, W_), dtype=torch.int32, device="cuda"))

    keep = buffers()
    run(*keep)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = run(*keep)
    ctx.sync_stream()
    for k, pb in ((b.page_k, b.page_b), (k2, b2), (b.page_k, b.page_b), (k2, b2)):
        ctx.set_page_table(b.vaddr, k, pb)
        graph.replay()
        torch.cuda.synchronize()
        got = out.view(torch.int32).clone()
        ref = run(*buffers()).view(torch.int32).clone()
        torch.cuda.synchronize()
        assert bool((ref != 0).any())
        assert torch.equal(got, ref)
