"""The raycast's eight-samples-at-a-time march against the oracle, bit for bit,
where it can go wrong: images of one pixel, of parts of a wave's tile and of an
XCD's patch; volumes down to one cell; runs of free and unseen space (+-32767,
+-32766, -32768) broken by thin surfaces, so that the coarse steps' shortcut
and every kind of event fall on each of a group's lanes; rays along a surface,
whose fine steps go on for most of the volume."""
import numpy as np
import pytest

import test_raycast_oracle as RO
from test_raycast_gpu import check, noisy_volume

pytestmark = pytest.mark.gpu


def layered_volume(shape, seed):
    """Slabs of saturated space with ramps of a few voxels between them."""
    rng = np.random.default_rng(seed)
    Z, Y, X = shape
    z, y, x = np.meshgrid(np.arange(Z), np.arange(Y), np.arange(X), indexing="ij")
    k = rng.normal(size=3)
    d = (k[0] * x + k[1] * y + k[2] * z) / np.linalg.norm(k)
    f = np.sin(d / 7.0 + rng.uniform(0, 6)) * 8.0
    s = np.clip(np.rint(f * 12000), -32768, 32767).astype(np.int16)
    hi = rng.random(shape) < 0.3
    s[(s == 32767) & hi] = 32766
    s[(s == -32768) & hi] = -32766
    s[(s == -32768) & (rng.random(shape) < 0.5)] = -32767
    return s.view(np.uint16).astype(np.uint32) | (1 << 16)


@pytest.mark.parametrize("W,H", [(1, 1), (2, 4), (3, 5), (16, 16), (17, 33)])
@pytest.mark.parametrize("shape", [(2, 2, 2), (2, 40, 9), (33, 5, 64), (60, 61, 62)])
def test_edges_bit_exact(dev, shape, W, H):
    print(f"[case] raycast lanes {shape} {W}x{H}", flush=True)
    Z, Y, X = shape
    h = 0.01
    size = np.array([X, Y, Z], np.float64)
    for k, vol in enumerate((layered_volume(shape, 3), noisy_volume(shape, 4))):
        for n, (ax, ay, az) in enumerate([(0.0, 0.0, 0.0), (0.3, 2.6, 0.1), (1.5, 0.4, 0.7)]):
            R = RO.rot(ax, ay, az)
            eye = size * (0.5, 0.31, 0.74)[n] - (0.0, 0.9, 0.2)[n] * size.max() * R[:, 2]
            pose = np.concatenate([R.reshape(-1), eye * h]).astype(np.float32)
            intr = np.array([1.1 * max(W, 4), 1.1 * max(W, 4), W / 2 - 0.5, H / 2 - 0.5],
                            np.float32)
            check(vol, h, intr, pose, W, H, 0.5 * (k & 1), dev)


def test_rays_along_a_surface_bit_exact(dev):
    print("[case] raycast along a plane, 200 voxels", flush=True)
    Z, Y, X = 200, 24, 40
    z, y, x = np.meshgrid(np.arange(Z), np.arange(Y), np.arange(X), indexing="ij")
    f = (y - 9.3 + 0.002 * z) / 6.0  # the camera looks along z, one voxel above the plane
    s = np.clip(np.rint(f * 32766), -32767, 32767).astype(np.int16)
    vol = s.view(np.uint16).astype(np.uint32) | (1 << 16)
    pose = np.array([1, 0, 0, 0, 1, 0, 0, 0, 1, 0.2, 0.105, -0.02], np.float32)
    d, _ = check(vol, 0.01, np.array([400, 400, 15.5, 11.5], np.float32), pose, 32, 24, 0.0, dev)
    assert (d > 1.0).any() and (d == 0).any()
