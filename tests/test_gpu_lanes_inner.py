"""Frames over bricks without an apron at 16, 4 and 1 lanes per ray, against the oracle: groups whose
taps clamp at the brick's faces next to groups that need no clamps."""
import numpy as np
import pytest

from hydrant_amd import _lib as L
from hydrant_amd import dataset as D
from hydrant_amd import workloads as W
from tests.helpers import oracle_view, oracle_volume

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("schedule", [L.SCHED_REFERENCE, L.SCHED_LATTICE])
@pytest.mark.parametrize("W_,H_", [(37, 29), (163, 157), (641, 621)])
@pytest.mark.parametrize("n,bs", [(16, 0), (21, 5)])
@pytest.mark.parametrize("fmt", [L.FMT_U8, L.FMT_F16, L.FMT_F32])
def test_frames_without_an_apron(gpu_ctx, fmt, n, bs, W_, H_, schedule):
    vol = np.random.default_rng(n).integers(0, 256, (n, n, n)).astype(np.uint8)   # noise: every tap matters
    if fmt != L.FMT_U8:
        vol = vol.astype(np.float32) / np.float32(255)
        vol = vol.astype(np.float16).view(np.uint16) if fmt == L.FMT_F16 else vol
    b = D.make_bricked(vol, bs or n, 0, fmt, None, resident=1.0, seed=5)
    sc = W.Scene("noise", b, D.README_TF.copy(), W_, H_, (33.0, 21.0, 2.2), 60.0, D.geometry((n, n, n), bs or n, 0.5),
                 density=0.3, schedule=schedule)
    gpu_ctx.load(b, sc.tf)
    out = gpu_ctx.render_volume(sc.volume_params(), sc.view(), W_, H_, film=False, count=True)
    r = oracle_volume(sc).render(oracle_view(sc), 32, film=False)
    assert int(out["samples"].item()) == r["samples"] > 0
    got = out["rgba"].cpu().numpy()
    if schedule == L.SCHED_REFERENCE:
        assert np.array_equal(got, r["rgba"].astype(np.float32))
    else:
        assert np.max(np.abs(got - r["rgba"])) <= 1e-4
