"""The raycast where its lanes a ray change (2^18 rays with volumes up to 160
voxels and longer, 7 * 2^17 rays): images just below and above, whose last tiles
and patches are partial, through volumes from one cell to longer than the limit,
against the oracle, bit for bit."""
import numpy as np
import pytest

import test_raycast_oracle as RO
from test_raycast_gpu import check, noisy_volume
from test_raycast_lanes_gpu import layered_volume

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(511, 513), (512, 512), (619, 433), (1217, 753), (1213, 757)])
@pytest.mark.parametrize("shape", [(2, 2, 2), (33, 5, 64), (20, 162, 9)])
def test_images_bit_exact(dev, shape, W, H):
    print(f"[case] raycast {shape} {W}x{H}", flush=True)
    Z, Y, X = shape
    h = 0.01
    size = np.array([X, Y, Z], np.float64)
    for k, vol in enumerate((layered_volume(shape, 3), noisy_volume(shape, 4))):
        R = RO.rot(*((0.3, 2.6, 0.1), (1.5, 0.4, 0.7))[k])
        eye = size * (0.5, 0.31)[k] - (0.9, 0.0)[k] * size.max() * R[:, 2]
        pose = np.concatenate([R.reshape(-1), eye * h]).astype(np.float32)
        intr = np.array([1.1 * W, 1.1 * W, W / 2 - 0.5, H / 2 - 0.5], np.float32)
        check(vol, h, intr, pose, W, H, 0.5 * (k & 1), dev)


@pytest.mark.parametrize("W,H", [(520, 506), (960, 960)])
def test_rays_along_a_surface_bit_exact(dev, W, H):
    print(f"[case] raycast along a plane, 150 voxels, {W}x{H}", flush=True)
    Z, Y, X = 150, 24, 40
    z, y, x = np.meshgrid(np.arange(Z), np.arange(Y), np.arange(X), indexing="ij")
    f = (y - 9.3 + 0.002 * z) / 6.0  # the camera looks along z, one voxel above the plane
    s = np.clip(np.rint(f * 32766), -32767, 32767).astype(np.int16)
    vol = s.view(np.uint16).astype(np.uint32) | (1 << 16)
    pose = np.array([1, 0, 0, 0, 1, 0, 0, 0, 1, 0.2, 0.105, -0.02], np.float32)
    intr = np.array([12.5 * W, 12.5 * W, W / 2 - 0.5, H / 2 - 0.5], np.float32)
    d, _ = check(vol, 0.01, intr, pose, W, H, 0.0, dev)
    assert (d > 1.0).any()
