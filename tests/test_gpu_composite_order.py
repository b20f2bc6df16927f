"""Composites whose z order fits the launch's arguments (64 images) and whose does not (65):
the oracle's image and bytes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 5, 64, 65])
def test_composite_orders(gpu_ctx, n):
    import torch
    from oracle import oracle as O

    rng = np.random.default_rng(n)
    a = rng.random((n, 9, 31, 1)).astype(np.float32) * 0.5
    rgb = rng.random((n, 9, 31, 3)).astype(np.float32) * a
    parts = np.concatenate([rgb, 1 - a, rgb, a], axis=3).astype(np.float32)
    z = rng.permutation(n).tolist()
    rgba, bytes_ = gpu_ctx.composite(torch.from_numpy(parts).cuda(), z)
    want, want_bytes = O.composite(parts, z)
    assert np.array_equal(rgba.cpu().numpy(), want)
    assert np.array_equal(bytes_.cpu().numpy(), want_bytes)


@pytest.mark.parametrize("n", [1, 64, 65])
def test_iso_composite_orders(gpu_ctx, n):
    import torch
    from oracle import oracle as O

    rng = np.random.default_rng(n)
    val = rng.integers(0, 256, (n, 9, 31, 3), dtype=np.uint8)
    depth = rng.random((n, 9, 31)).astype(np.float32)
    z = rng.permutation(n).tolist()
    parts = np.zeros((n, 9, 31, 8), np.uint8)   # val, padding, depth
    parts[..., 0:3] = val
    parts[..., 4:8] = depth[..., None].view(np.uint8)
    rgb, d = gpu_ctx.composite_iso(torch.from_numpy(parts).cuda(), z)
    want_rgb, want_d = O.composite_iso(val, depth, z)
    assert np.array_equal(d.cpu().numpy(), want_d)
    assert np.array_equal(rgb.cpu().numpy(), want_rgb)
