"""Performance cases of the render path: the work a user of the library has it do.

Kinds:
  frame      one Volume-mode frame (reference or lattice schedule) of a resident volume
  stream     a paged frame in two passes: film emitted over a partial residency, the rest of
             the bricks made resident, the film resumed, RGB8 written
  sortlast   a volume held as residency batches, one segment launch, in-GPU composite
  iso        one isosurface frame
  batch      many views of several volumes in one persistent launch
  diff       one training step's render: differentiable forward and adjoint
  composite  sort-last composite of partial images gathered from other ranks

Volumes, transfer function, cameras and sizes follow hydrant_amd/workloads.py, bench.py and
the tests.  ``exact`` restates each model in 64-bit torch.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

DEV = "cuda"
DENSITY = 1e-2
# 9-point README transfer function (alpha 0 at both ends)
TF = np.array([[0, 0, 0, 0], [1, 0, 0, 1], [1, .5, 0, 1], [1, 1, 0, 1], [0, 1, 0, 1], [0, 1, 1, 1], [0, 0, 1, 1],
               [1, 0, 1, 1], [0, 0, 0, 0]], np.float32)
FMT = {"u8": 0, "f16": 1, "f32": 2}
TORCH_FMT = {"u8": torch.uint8, "f16": torch.float16, "f32": torch.float32}


# ------------------------------------------------------------------- cases ----
def listed():
    return [
        # smallest call: a thumbnail of a small volume (latency and launch cost)
        dict(name="frame_f32_thumb", kind="frame", n=32, bs=0, fmt="f32", data="blobs", w=48, h=40,
             schedule="reference", resident=1.0),
        # the plain view: a 256^3 FP32 volume as one brick, 512^2
        dict(name="frame_f32_512", kind="frame", n=256, bs=0, fmt="f32", data="blobs", w=512, h=512,
             schedule="reference", resident=1.0),
        # a large paged volume, 40% of the bricks resident, rays stop at page faults
        dict(name="frame_u8_paged", kind="frame", n=1024, bs=64, fmt="u8", data="fbm", w=512, h=512,
             schedule="reference", resident=0.4),
        # an interactive window of ragged size over a bricked FP16 volume, order-independent schedule
        dict(name="frame_f16_lattice", kind="frame", n=500, bs=64, fmt="f16", data="blobs", w=765, h=431,
             schedule="lattice", resident=1.0),
        # paging: emit over half the bricks, page in the rest, resume the film
        dict(name="stream_u8", kind="stream", n=256, bs=32, fmt="u8", data="fbm", w=384, h=300),
        # a volume larger than one pool: three residency batches, one launch, composite
        dict(name="sortlast_u8", kind="sortlast", n=1024, bs=64, fmt="u8", data="fbm", w=512, h=512, batches=3),
        # isosurface of an FP16 signed distance field
        dict(name="iso_f16_1024", kind="iso", n=512, bs=64, fmt="f16", data="sdf", w=1024, h=1024, iso=0.0),
        # offline throughput: 96 views of three volumes, replayed from a graph
        dict(name="batch_f16_96", kind="batch", n0=256, n1=512, n2=768, bs=64, fmt="f16", views=96, res0=256,
             res1=1024, graph=True),
        # serving: a few small views of one volume per request
        dict(name="batch_u8_8", kind="batch", n0=200, n1=0, n2=0, bs=64, fmt="u8", views=8, res0=96, res1=320,
             graph=False),
        # training step at full size: 32 views at 256^2 of a 128^3 volume, 512 samples a ray
        dict(name="diff_32x256", kind="diff", n=128, w=256, h=256, views=32, steps=512, ckpt=64),
        # training step of a small fit
        dict(name="diff_6x64", kind="diff", n=48, w=64, h=64, views=6, steps=512, ckpt=64),
        # compositing the partial images of eight ranks
        dict(name="composite_8", kind="composite", parts=8, w=1024, h=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame", "frame", "frame", "stream", "sortlast", "iso", "iso", "batch", "batch", "diff", "diff",
                       "composite"])
    w, h = _log(rng, 48, 1000), _log(rng, 40, 1000)
    if kind == "frame":
        bs = rng.choice([0, 32, 64])
        fmt = rng.choice(["u8", "f16", "f32"])
        n = _log(rng, 32, 320 if bs == 0 else 640)
        return dict(kind=kind, n=n, bs=bs, fmt=fmt, data=rng.choice(["blobs", "fbm"]), w=w, h=h,
                    schedule=rng.choice(["reference", "reference", "lattice"]),
                    resident=1.0 if bs == 0 else rng.choice([0.4, 1.0]))
    if kind == "stream":
        return dict(kind=kind, n=_log(rng, 64, 400), bs=rng.choice([32, 64]), fmt=rng.choice(["u8", "f16"]),
                    data=rng.choice(["blobs", "fbm"]), w=w, h=h)
    if kind == "sortlast":
        return dict(kind=kind, n=_log(rng, 128, 640), bs=rng.choice([32, 64]), fmt=rng.choice(["u8", "f16"]),
                    data=rng.choice(["blobs", "fbm"]), w=min(w, 640), h=min(h, 640), batches=rng.choice([2, 3, 4]))
    if kind == "iso":
        fmt, data, iso = rng.choice([("f16", "sdf", 0.0), ("f32", "sdf", 0.0), ("u8", "blobs", 0.35)])
        return dict(kind=kind, n=_log(rng, 64, 512), bs=rng.choice([32, 64]), fmt=fmt, data=data, w=w, h=h, iso=iso)
    if kind == "batch":
        n = sorted(_log(rng, 64, 400) for _ in range(rng.choice([1, 2, 3])))
        n += [0] * (3 - len(n))
        return dict(kind=kind, n0=n[0], n1=n[1], n2=n[2], bs=rng.choice([32, 64, 64]),
                    fmt=rng.choice(["u8", "f16", "f16", "f32"]), views=_log(rng, 1, 48), res0=_log(rng, 48, 200),
                    res1=_log(rng, 200, 600), graph=rng.choice([True, False]))
    if kind == "diff":
        return dict(kind=kind, n=_log(rng, 16, 120), w=_log(rng, 24, 200), h=_log(rng, 24, 200),
                    views=_log(rng, 1, 24), steps=rng.choice([96, 200, 256, 512]), ckpt=rng.choice([32, 64]))
    return dict(kind=kind, parts=rng.choice([2, 3, 5, 8, 16]), w=w, h=h)


# ------------------------------------------------------------------ inputs ----
def _gen(seed):
    return np.random.default_rng(int(seed))


def _blobs(n, rng, count=16, sig=(8.0, 40.0), ref=256.0):
    """Sum of Gaussian blobs as 8-bit counts, (z, y, x)."""
    c, s = rng.uniform(0, n, (count, 3)), rng.uniform(*sig, count) * n / ref
    amp = rng.uniform(0.3, 1.0, count)
    x = np.arange(n) + 0.5
    g = [torch.tensor(np.exp(-(x[None] - c[:, a, None]) ** 2 / (2 * s[:, None] ** 2)), dtype=torch.float32, device=DEV)
         for a in range(3)]
    g[2] = g[2] * torch.tensor(amp[:, None], dtype=torch.float32, device=DEV)
    zy = (g[2][:, :, None] * g[1][:, None, :]).reshape(count, -1)
    v = (zy.t() @ g[0]).reshape(n, n, n)
    return v.mul_(255.0).add_(0.5).floor_().clamp_(0, 255).to(torch.uint8)


def _fbm(n, rng, octaves=5):
    """Value-noise fBm (base period n/8 voxels, persistence 0.5) saturating at both ends, 8-bit counts."""
    v = torch.zeros((n, n, n), dtype=torch.float32, device=DEV)
    amp, var = 1.0, 0.0
    for o in range(octaves):
        m = 8 * 2 ** o
        x = (np.arange(n) + 0.5) * m / n
        i, t = np.floor(x).astype(int), x - np.floor(x)
        t = t * t * t * (t * (t * 6 - 15) + 10)
        wt = np.zeros((n, m + 2), np.float32)
        wt[np.arange(n), i], wt[np.arange(n), i + 1] = 1 - t, t
        wt = torch.from_numpy(wt).to(DEV)
        lat = torch.from_numpy(rng.uniform(-1, 1, (m + 2,) * 3).astype(np.float32)).to(DEV)
        a = torch.matmul(lat.reshape(-1, m + 2), wt.t()).reshape(m + 2, m + 2, n)
        a = torch.matmul(wt, a)                                    # (z lattice, y, x)
        v.reshape(n, -1).addmm_(wt, a.reshape(m + 2, -1), alpha=amp)
        amp, var = amp * 0.5, var + amp * amp
    return v.mul_(255 * 0.95 / math.sqrt(var)).add_(128.0).floor_().clamp_(0, 255).to(torch.uint8)


def _sdf(n, rng, count=64):
    """Smooth union of spheres (radius 10-60 voxels at 512^3) in voxels, FP32."""
    s = n / 512.0
    c, r, k = rng.uniform(0, n, (count, 3)), rng.uniform(10 * s, 60 * s, count), 8.0 * s
    x = torch.arange(n, dtype=torch.float32, device=DEV) + 0.5
    v = None
    for j in range(count):
        q = [(x - float(c[j, a])) ** 2 for a in range(3)]
        d = (q[2][:, None, None] + q[1][None, :, None] + q[0][None, None, :]).sqrt_().sub_(float(r[j]))
        if v is None:
            v = d
        else:
            h = (v - d).abs_().neg_().add_(k).clamp_(min=0).div_(k)
            v = torch.minimum(v, d).sub_(h.square_().mul_(k * 0.25))
    return v


def _volume(data, n, rng):
    return {"blobs": _blobs, "fbm": _fbm, "sdf": _sdf}[data](n, rng)


def _stored(vol, fmt, counts=False):
    """Voxels in the pool's format: 8-bit counts, or their value / 255 (counts: kept as counts)."""
    if vol.dtype == torch.uint8 and fmt != "u8":
        v = vol.float()
        return (v if counts else v / 255.0).to(TORCH_FMT[fmt])
    return vol.to(TORCH_FMT[fmt])


def _values(stored, counts=False):
    """Renderer's value of a stored voxel as a factor on the raw number."""
    return 1.0 / 255.0 if stored.dtype == torch.uint8 or counts else 1.0


class Bricks:
    """A volume cut into padded bricks: brick grid, emptiness, page order (bs 0: one brick, no apron)."""

    def __init__(self, stored, bs, empty_fn, rng, counts=False):
        from hydrant_amd import dataset as D

        n = stored.shape[0]
        self.n, self.bs, self.apron = n, bs or n, 1 if bs else 0
        self.pad = self.bs + 2 * self.apron
        g = self.g = -(-n // self.bs)
        v = stored
        if bs:
            idx = torch.arange(-1, g * self.bs + 1, device=DEV).clamp_(0, n - 1)
            v = v[idx][:, idx][:, :, idx]
        win = v.unfold(0, self.pad, self.bs).unfold(1, self.pad, self.bs).unfold(2, self.pad, self.bs)
        scale = _values(stored, counts)
        lo = torch.stack([w.amin((2, 3, 4)).float() for w in win]).cpu().numpy() * scale
        hi = torch.stack([w.amax((2, 3, 4)).float() for w in win]).cpu().numpy() * scale
        self.empty = np.zeros((g, g, g), bool) if empty_fn is None or not bs else np.asarray(empty_fn(lo, hi), bool)
        self.cheb = D.chebyshev(self.empty.astype(np.uint8))
        full = np.flatnonzero(~self.empty.reshape(-1))
        self.order = rng.permutation(full).astype(np.int64) if bs else full
        self.win = win
        k, b = D.mapping(self.bs, self.apron)
        self.k, self.b = k, b

    def pages(self, ids):
        t = torch.as_tensor(np.asarray(ids), device=DEV)
        g = self.g
        return self.win[t // (g * g), (t // g) % g, t % g].contiguous()

    def table(self, ids):
        va = np.full((self.g,) * 3, -1, np.int32)
        va.reshape(-1)[ids] = np.arange(len(ids), dtype=np.int32)
        return va, np.full(max(len(ids), 1), self.k, np.float32), np.full((max(len(ids), 1), 3), self.b, np.float32)


def _host(t):
    t = t.cpu()
    return t.view(torch.int16).numpy().view(np.uint16) if t.dtype == torch.float16 else t.numpy()


def _tf_empty():
    from hydrant_amd import dataset as D

    return D.volume_empty_fn(TF)


def _arm(rng):
    return float(rng.uniform(0, 360)), float(rng.uniform(-70, 70)), 2.2


def _geom(n, bs, rate):
    bs = bs or n
    f = np.full(3, np.float32(n) / np.float32(bs), np.float32)
    return f, np.float32(1) / np.float32(bs) / np.float32(4) / np.float32(rate)


def _inputs(case, seed):
    """What both prepare() and exact() start from: the volume, its bricks and the camera arm."""
    rng = _gen(seed)
    arm = _arm(rng)
    vol = _stored(_volume(case["data"], case["n"], rng), case["fmt"])
    iso = case.get("iso")
    fn = _tf_empty() if iso is None else (lambda lo, hi: (lo > iso) | (hi < iso))
    return vol, Bricks(vol, case["bs"], fn, rng), arm


def _view(arm, f_dim):
    from hydrant_amd import hip

    return hip.make_view(hip.orbit_camera(arm), f_dim / 2, f_dim)


def _params(case, lattice, ert=0.0):
    from hydrant_amd import hip

    f, step = _geom(case["n"], case["bs"], 0.5)
    return hip.volume_params(np.zeros(3), f, step, 1.0 / (case["bs"] or case["n"]), density=DENSITY,
                             schedule=1 if lattice else 0, ert=ert)


def prepare(case, seed):
    from hydrant_amd import hip

    kind = case["kind"]
    st = {"case": case}
    if kind == "composite":
        g = torch.Generator(device=DEV).manual_seed(int(seed))
        shape = (case["parts"], case["h"], case["w"])
        a = torch.rand(shape + (1,), generator=g, device=DEV) * 0.4
        rgb = torch.rand(shape + (3,), generator=g, device=DEV) * a
        st["parts"] = torch.cat([rgb, 1 - a, rgb, a], -1).contiguous()
        st["z"] = _gen(seed).permutation(case["parts"]).astype(np.int32)
        st["ctx"] = hip.Context(0)
        return st
    if kind == "diff":
        from hydrant_amd.diff import DiffRenderer

        vol, tf, grad, arms = _diff_inputs(case, seed)
        one = np.ones(3, np.float32)
        ctx = hip.Context(0)
        st["r"] = DiffRenderer(ctx, [_view(a, one) for a in arms], case["w"], case["h"], (case["n"],) * 3,
                               case["steps"], case["ckpt"], 8.0)
        st.update(vol=vol, tf=tf, grad=grad, ctx=ctx)
        return st
    if kind == "batch":
        vols, views = _batch_inputs(case, seed)
        ctx = hip.Context(0)
        pools, descs, base = [], [], 0
        for stored, b in vols:
            pools.append(b.pages(b.order))
            va, _, _ = b.table(b.order)
            va[va >= 0] += base
            base += len(b.order)
            f, step = _geom(b.n, b.bs, 0.5)
            descs.append(dict(grid=(b.g,) * 3, bs=b.bs, apron=b.apron, bbox_max=f, step=step,
                              value_scale=1.0 / 255.0, vaddr=va, cheb=b.cheb))
        ctx.upload_pool(FMT[case["fmt"]], vols[0][1].pad, _host(torch.cat(pools)))
        ctx.set_tf(TF)
        ctx.set_volumes(descs)
        hv = [(_view(arm, descs[i]["bbox_max"]), w, h, i) for i, w, h, arm in views]
        st["ctx"], st["batch"] = ctx, ctx.batch(hv)
        st["cfg"] = hip.batch_config(tile_w=8, unroll=4, waves_per_cu=16)
        if case["graph"]:
            st["out"] = st["batch"].new_output()
            st["batch"].capture(st["cfg"], DENSITY, 0.9999, st["out"])
        return st
    vol, b, arm = _inputs(case, seed)
    f, _ = _geom(case["n"], case["bs"], 0.5)
    ctx = st["ctx"] = hip.Context(0)
    st["view"] = _view(arm, f)
    ctx.set_empty_grid(b.cheb)
    fmt = FMT[case["fmt"]]
    if kind == "sortlast":
        ctx.set_tf(TF)
        st["p"] = _params(case, True)
        parts = []
        for ids in np.array_split(b.order, case["batches"]):
            va, k, o = b.table(ids)
            parts.append((fmt, b.pad, b.pages(ids if len(ids) else [0]), va, k, o))
        st["set"] = ctx.segment_set(parts)
        return st
    keep = b.order[: max(1, int(round(case["resident"] * b.g ** 3)))] if kind == "frame" else b.order
    ctx.upload_pool(fmt, b.pad, _host(b.pages(keep if len(keep) else [0])))
    st["table"] = b.table(keep)
    ctx.set_page_table(*st["table"])
    if kind == "iso":
        st["p"] = _iso_params(case, arm)
        return st
    ctx.set_tf(TF)
    lattice = case.get("schedule") == "lattice"
    st["p"] = _params(case, lattice, 0.9999 if lattice else 0.0)
    if kind == "stream":
        half = st["table"][0].copy()
        half[half >= (len(keep) + 1) // 2] = -1
        st["half"] = (half,) + st["table"][1:]
    return st


def run(st):
    case, ctx = st["case"], st["ctx"]
    kind = case["kind"]
    if kind == "frame":
        return ctx.render_volume(st["p"], st["view"], case["w"], case["h"], film=False)["rgba"]
    if kind == "stream":
        ctx.set_page_table(*st["half"])
        film = ctx.render_volume(st["p"], st["view"], case["w"], case["h"], film=True)["film"]
        ctx.set_page_table(*st["table"])
        out = ctx.resume_volume(st["p"], film)
        rgb = ctx.pixel_pass(out["rgba"])
        return {"rgba": out["rgba"], "rgb": rgb, "ray": film[..., :6], "steps": film.view(torch.int32)[..., 6:8],
                "theta": film[..., 12:]}
    if kind == "sortlast":
        return ctx.render_sort_last_set(st["p"], st["view"], case["w"], case["h"], st["set"])[0]
    if kind == "iso":
        px = ctx.render_iso(st["p"], st["view"], case["w"], case["h"])["px"]
        return {"rgba": px[..., :4], "depth": px[..., 4], "hit": px.view(torch.int32)[..., 5]}
    if kind == "batch":
        if case["graph"]:
            st["batch"].replay()
            return st["out"]
        return st["batch"].render(st["cfg"], DENSITY, 0.9999)[0]
    if kind == "diff":
        rgba, ck, _ = st["r"].forward_raw(st["vol"], st["tf"])
        gv, gt = st["r"].backward_raw(st["vol"], st["tf"], ck, st["grad"])
        return {"rgba": rgba, "grad_volume": gv, "grad_tf": gt}
    rgba, rgb = ctx.composite(st["parts"], st["z"])
    return {"rgba": rgba, "rgb": rgb}


def work(case):
    """Bytes: the voxels and images once.  Operations: 45 a sample (21 trilinear, 12 transfer
    function, 12 compositing) over the rays that meet the volume (about 0.45 of the pixels, mean
    chord 0.7 of the edge); 150 a sample for a forward and adjoint step."""
    kind = case["kind"]
    if kind == "composite":
        px = case["w"] * case["h"]
        return {"bytes": px * (32.0 * case["parts"] + 19), "flops": px * 14.0 * case["parts"]}
    if kind == "diff":
        rays = case["views"] * case["w"] * case["h"]
        return {"bytes": 2 * 4.0 * case["n"] ** 3 + rays * 32.0, "flops": 0.45 * rays * case["steps"] * 150.0}
    size = {"u8": 1, "f16": 2, "f32": 4}[case["fmt"]]
    if kind == "batch":
        ns = [n for n in (case["n0"], case["n1"], case["n2"]) if n]
        px = case["views"] * (0.5 * (case["res0"] + case["res1"])) ** 2
        return {"bytes": size * sum(float(n) ** 3 for n in ns) + 16 * px,
                "flops": px * 0.45 * 0.7 * 2 * (sum(ns) / len(ns)) * 45}
    px = case["w"] * case["h"]
    rate = 4 if kind == "iso" else 2
    res = case.get("resident", 1.0)
    out = {"iso": 24, "stream": 16 + 64 + 3}.get(kind, 16)
    return {"bytes": res * size * float(case["n"]) ** 3 + out * px,
            "flops": px * 0.45 * 0.7 * rate * case["n"] * res * (25 if kind == "iso" else 45)}


# ------------------------------------------------------- inputs of the rest ----
def _batch_inputs(case, seed):
    rng = _gen(seed)
    vols = []
    for n in (case["n0"], case["n1"], case["n2"]):
        if n:
            stored = _stored(_blobs(n, rng), case["fmt"], counts=True)
            vols.append((stored, Bricks(stored, case["bs"], _tf_empty(), rng, counts=True)))
    # resolutions: five sizes from res0 to res1, as a set of thumbnails, previews and full frames has
    sizes = [int(round(case["res0"] * (case["res1"] / case["res0"]) ** (i / 4))) for i in range(5)]
    views = []
    for v in range(case["views"]):
        w, h = sizes[v % 5], sizes[v % 5] if v % 3 else sizes[(v + 1) % 5]
        views.append((v % len(vols), w, h, _arm(rng)))
    return vols, views


def _diff_inputs(case, seed):
    """A fit in progress: a blob volume, a transfer function of smooth bumps, image residuals."""
    rng = _gen(seed)
    vol = _blobs(case["n"], rng, 8, (6.0, 20.0), 128.0).float() / 255.0
    s = (np.arange(256) + 0.5) / 256
    tf = np.zeros((256, 4))
    for _ in range(4):
        bump = np.exp(-0.5 * ((s - rng.uniform(0.15, 0.95)) / rng.uniform(0.04, 0.15)) ** 2)
        tf[:, :3] += bump[:, None] * rng.uniform(0.2, 1.0, 3)
        tf[:, 3] += rng.uniform(0.3, 1.0) * bump
    tf = torch.from_numpy(np.clip(tf, 0, 1).astype(np.float32)).to(DEV)
    arms = [(float(rng.uniform(0, 360)), float(rng.uniform(-60, 60)), 2.2) for _ in range(case["views"])]
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    grad = torch.randn((case["views"], case["h"], case["w"], 4), generator=g, device=DEV)
    return vol, tf, grad, arms


def _light(arm):
    """Light of the isosurface renderer: position + target + up + cross(target, up)."""
    pos = _camera64(arm)[0]
    return pos + np.array([0.0, 1.0, 0.0])


def _iso_params(case, arm):
    from hydrant_amd import _lib as L
    from hydrant_amd import hip

    f, step = _geom(case["n"], case["bs"], 1.0)
    cam = hip.orbit_camera(arm)
    c, s = (f / 2).astype(np.float32), f
    iet, inv = np.zeros(16, np.float32), np.zeros(16, np.float32)
    L.call("hyd_exhibit_iet", L.ptr(c, C.c_float), L.ptr(s, C.c_float), L.ptr(iet, C.c_float))
    L.call("hyd_mat4_inverse", L.ptr(iet, C.c_float), L.ptr(inv, C.c_float))
    p = L.IsoParams()
    p.bbox_min, p.bbox_max = L.f3(0, 0, 0), L.f3(*[float(x) for x in f])
    p.step, p.du, p.max_steps, p.mode = float(step), 1.0 / case["bs"], 4_000_000, 0
    p.to_world = L.f16(*[float(x) for x in inv])
    p.eye_pos, p.light_pos = L.f3(*cam.position[:]), L.f3(*[float(x) for x in _light(arm)])
    p.surface_color = L.f3(1.0, 1.0, 1.0)
    p.isovalue, p.corrected, p.bisect_steps = float(case["iso"]), 1, 8
    return p


# ------------------------------------------------------------ 64-bit models ----
def _camera64(arm):
    a, e, dist = math.radians(arm[0]), math.radians(arm[1]), arm[2]
    x, y = dist * math.cos(e), dist * math.sin(e)
    pos = np.array([x * math.cos(a), y, -x * math.sin(a)])
    f = -pos / np.linalg.norm(pos)
    s = np.cross(f, [0.0, 1.0, 0.0])
    s /= np.linalg.norm(s)
    return pos, s, np.cross(s, f), f


def _rays64(arm, f_dim, w, h):
    """Origin and unit directions (rays, 3) in block units, integer pixel corners."""
    pos, s, u, f = _camera64(arm)
    f_dim = np.asarray(f_dim, np.float64)
    scale = float(np.max(np.abs(f_dim / 2)))
    y, x = torch.meshgrid(torch.arange(h, dtype=torch.float64, device=DEV),
                          torch.arange(w, dtype=torch.float64, device=DEV), indexing="ij")
    ux, uy = (x - w / 2) * 2 / h, -(y - h / 2) * 2 / h
    ctg = 1.0 / math.tan(math.radians(30.0))
    t = lambda a: torch.tensor(a, dtype=torch.float64, device=DEV)  # noqa: E731
    d = ux[..., None] * t(s) + uy[..., None] * t(u) + ctg * t(f)
    d = d.reshape(-1, 3)
    return t(pos * scale + f_dim / 2), d / d.norm(dim=1, keepdim=True)


def _clip64(o, d, hi):
    hi = torch.as_tensor(np.asarray(hi, np.float64), device=DEV)
    t0, t1 = -o / d, (hi - o) / d
    near, far = torch.minimum(t0, t1).amax(1), torch.maximum(t0, t1).amin(1)
    return near.clamp(min=0), far.clamp(min=0), far > near


class Sampler64:
    """Trilinear value at points p (block units) of brick ip, taps clamped to the padded brick."""

    def __init__(self, stored, b, scale):
        self.v, self.b, self.scale = stored.reshape(-1), b, scale
        self.empty = torch.from_numpy(b.empty.reshape(-1)).to(DEV)
        self.cheb = torch.from_numpy(b.cheb.reshape(-1)).to(DEV)

    def skip(self, p, ip, cell, d, step):
        """Steps over an empty brick's neighbourhood, as the reference schedule counts them."""
        far = torch.maximum((ip - p) / d, (ip + 1 - p) / d).amin(1)
        return ((far + (self.cheb[cell] - 1) / d.abs().amax(1)) / step).ceil() + 1

    def brick(self, p):
        ip = p.floor()
        c = ip.long().clamp_(0, self.b.g - 1)
        return ip, (c[:, 2] * self.b.g + c[:, 1]) * self.b.g + c[:, 0]

    def __call__(self, p, ip):
        b = self.b
        f = (p - ip) * b.bs + (b.apron - 0.5)
        fl = f.floor()
        w = f - fl
        first = ip.long() * b.bs - b.apron
        at = [(first + x.long().clamp(0, b.pad - 1)).clamp(0, b.n - 1) for x in (fl, f.ceil())]
        out = 0
        for c in range(8):
            s = [(c >> a) & 1 for a in range(3)]
            wt = 1.0
            for a in range(3):
                wt = wt * (w[:, a] if s[a] else 1 - w[:, a])
            out = out + wt * self.v[(at[s[2]][:, 2] * b.n + at[s[1]][:, 1]) * b.n + at[s[0]][:, 0]].double()
        return out * self.scale


def _tf64(tf, s):
    n = tf.shape[0]
    f = n * s
    ok = (f >= 0) & (f <= n)
    f = torch.where(ok, f, torch.zeros_like(f)) - 0.5
    fl = f.floor()
    t = (f - fl)[:, None]
    i, j = fl.long().clamp(0, n - 1), f.ceil().long().clamp(0, n - 1)
    return torch.where(ok[:, None], tf[i] * (1 - t) + tf[j] * t, torch.zeros((), dtype=torch.float64, device=DEV))


def _march64(samp, o, d, f_dim, step, lattice, resident=None, ert=0.0, chunk=48):
    """RGBA of the Volume march over rays d from o."""
    tf = torch.from_numpy(TF).double().to(DEV)
    step = float(step)
    near, far, hit = _clip64(o, d, f_dim)
    out = torch.zeros((d.shape[0], 4), dtype=torch.float64, device=DEV)
    idx = hit.nonzero()[:, 0]
    d, near, far = d[idx], near[idx], far[idx]
    o0 = o + d * near[:, None]
    span = (far - near) / step
    v = torch.zeros((len(idx), 4), dtype=torch.float64, device=DEV)
    if lattice:
        left, k = span, torch.zeros_like(span)
    else:
        left, k = span.floor(), torch.zeros_like(span)      # k: steps taken, in units of the first step
    ss = torch.ones_like(span)
    while len(idx):
        for _ in range(chunk):
            on = k < left
            if lattice:
                w = (left - k).clamp(max=1.0)
                p = o0 + d * ((k + 0.5 * w) * step)[:, None]
            else:
                w = 1.0
                p = o0 + d * (k * step)[:, None]
            ip, cell = samp.brick(p)
            full = ~samp.empty[cell]
            if resident is not None:
                stop = on & full & ~resident[cell]
                left = torch.where(stop, torch.zeros_like(left), left)
                on = on & ~stop
            c = _tf64(tf, samp(p, ip))
            a = torch.where(on & full, c[:, 3] * DENSITY * w, torch.zeros_like(k))
            v = v + torch.cat([c[:, :3] * a[:, None], a[:, None]], 1) * (1 - v[:, 3:])
            if lattice:
                k = k + 1
                if ert > 0:
                    left = torch.where(v[:, 3] > ert, torch.zeros_like(left), left)
            else:
                up = torch.where(v[:, 3] > 0.93, 16.0, torch.where(v[:, 3] > 0.85, 4.0, 1.0)).double()
                ss = torch.where(on & full, up, ss)
                hop = torch.where(full, ss, ss * samp.skip(p, ip, cell, d, step * ss))
                k = torch.where(on, k + hop, k)
        done = k >= left
        out[idx[done]] = v[done]
        go = ~done
        idx, d, o0, left, k, ss, v = (x[go] for x in (idx, d, o0, left, k, ss, v))
    return out


def _diff64(case, seed):
    vol, tf, grad, arms = _diff_inputs(case, seed)
    n, K = case["n"], case["steps"]
    gv = torch.zeros(n ** 3, dtype=torch.float64, device=DEV)
    gt = torch.zeros((256, 4), dtype=torch.float64, device=DEV)
    rep, imgs = 512, []
    ks = torch.arange(K, dtype=torch.float64, device=DEV) + 0.5
    for view, arm in enumerate(arms):
        o, d = _rays64(arm, np.ones(3), case["w"], case["h"])
        near, far, hit = _clip64(o, d, np.ones(3))
        img = torch.zeros((d.shape[0], 4), dtype=torch.float64, device=DEV)
        for idx in hit.nonzero()[:, 0].split(16384):
            dt = (far[idx] - near[idx]) / K
            p = o + d[idx][:, None, :] * (near[idx][:, None] + ks * dt[:, None])[..., None]
            f = (n * p - 0.5).reshape(-1, 3)
            fl = f.floor()
            w = f - fl
            at = [(fl.long() + a).clamp_(0, n - 1) for a in (0, 1)]
            # a replica of the volume and of the table per group of rays keeps the 64-bit sums apart
            v = vol.reshape(-1).double().requires_grad_(True)
            t = tf.double().repeat(rep, 1).requires_grad_(True)
            s = 0
            for c in range(8):
                b = [(c >> a) & 1 for a in range(3)]
                wt = (w[:, 0] if b[0] else 1 - w[:, 0]) * (w[:, 1] if b[1] else 1 - w[:, 1]) * \
                    (w[:, 2] if b[2] else 1 - w[:, 2])
                s = s + wt * v.index_select(0, (at[b[2]][:, 2] * n + at[b[1]][:, 1]) * n + at[b[0]][:, 0])
            fx = 256 * s - 0.5
            lo = fx.detach().floor()
            u = (fx - lo)[:, None]
            own = torch.arange(s.shape[0], device=DEV) % rep * 256
            c = t.index_select(0, lo.long().clamp(0, 255) + own) * (1 - u) + \
                t.index_select(0, (lo.long() + 1).clamp(0, 255) + own) * u
            c = c.reshape(len(idx), K, 4)
            tau = 8.0 * c[..., 3].clamp(min=0) * dt[:, None]
            before = torch.exp(-(tau.cumsum(1) - tau))
            a = before * -torch.expm1(-tau)
            rgba = torch.cat([(a[..., None] * c[..., :3]).sum(1), (1 - torch.exp(-tau.sum(1)))[:, None]], 1)
            g = grad[view].reshape(-1, 4)[idx].double()
            dv, dtf = torch.autograd.grad(rgba, (v, t), g)
            gv += dv
            gt += dtf.reshape(rep, 256, 4).sum(0)
            img[idx] = rgba.detach()
        imgs.append(img.reshape(case["h"], case["w"], 4))
    return {"rgba": torch.stack(imgs), "grad_volume": gv.reshape(n, n, n), "grad_tf": gt}


def exact(case, seed):
    kind = case["kind"]
    if kind == "composite":
        g = torch.Generator(device=DEV).manual_seed(int(seed))
        shape = (case["parts"], case["h"], case["w"])
        a = torch.rand(shape + (1,), generator=g, device=DEV) * 0.4
        rgb = torch.rand(shape + (3,), generator=g, device=DEV) * a
        p = torch.cat([rgb, 1 - a, rgb, a], -1).double()
        z = _gen(seed).permutation(case["parts"])
        f = p[int(z[0])][..., 4:]
        for k in z[1:]:
            b = p[int(k)]
            f = torch.cat([f[..., :3] + b[..., 4:7] - f[..., 3:] * b[..., :3], b[..., 3:4] * f[..., 3:] + b[..., 7:]], -1)
        return {"rgba": f, "rgb": None}
    if kind == "diff":
        return _diff64(case, seed) if case["views"] * case["w"] * case["h"] * case["steps"] < 2.4e8 else None
    if kind == "batch":
        steps = sum(2 * max(case["n0"], case["n1"], case["n2"]) for _ in range(case["views"]))
        if steps * (0.5 * (case["res0"] + case["res1"])) ** 2 > 3e9:
            return None
        vols, views = _batch_inputs(case, seed)
        out = []
        for i, w, h, arm in views:
            stored, b = vols[i]
            f, step = _geom(b.n, b.bs, 0.5)
            o, d = _rays64(arm, f, w, h)
            out.append(_march64(Sampler64(stored, b, 1.0 / 255.0), o, d, f, step, True, ert=0.9999))
        return torch.cat(out)
    if kind == "iso":
        # a ray that enters at the upper faces takes its first value from either end of the last
        # brick, by the rounding of its entry point: a 64-bit march hits elsewhere on such rays
        return None
    vol, b, arm = _inputs(case, seed)
    samp = Sampler64(vol, b, _values(vol))
    f, step = _geom(case["n"], case["bs"], 0.5)
    o, d = _rays64(arm, f, case["w"], case["h"])
    lattice = kind == "sortlast" or case.get("schedule") == "lattice"
    res = None
    if kind == "frame" and case["resident"] < 1:
        va = b.table(b.order[: max(1, int(round(case["resident"] * b.g ** 3)))])[0]
        res = torch.from_numpy(va.reshape(-1) >= 0).to(DEV)
    v = _march64(samp, o, d, f, step, lattice, res, 0.9999 if lattice and kind == "frame" else 0.0)
    v = v.reshape(case["h"], case["w"], 4)
    return v if kind != "stream" else {"rgba": v, "rgb": None, "ray": None, "steps": None, "theta": None}
