"""Integration with pose matrices that are no rotations (scaled, mirrored) at
the edge of what a frame updates: every frame measures one pixel, the one that
a voxel is seen at, at a distance that puts its sdf within a few ulps of
-trunc, and the voxel is alone in its brick, so the test of the brick has
nothing but its margin.  Byte-compared with the oracle."""
import ctypes

import numpy as np
import pytest
import torch

from marching_cube_amd import _capi
from marching_cube_amd.mesh import _ptr, _stream_handle
from oracle import oracle as O

pytestmark = pytest.mark.gpu

F = np.float32
H0 = F(0.005)  # voxel size
K, W, H = 512, 64, 48
INTR = np.array([60.0, 60.0, 31.5, 23.5], F)


def fma(a, b, c):
    return (np.float64(a) * np.float64(b) + np.float64(c)).astype(F)


def rotations(rng, n):
    q = rng.normal(size=(n, 4))
    w, x, y, z = (q / np.linalg.norm(q, axis=1, keepdims=True)).T
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w),
                     2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w),
                     2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)],
                    1).reshape(n, 3, 3)


def frames_at_the_edge(rng, voxel, scale, mirror, trunc):
    """(poses, depth): q = R^T (p - t) with R a rotation times scale (one
    column negated: mirrored)."""
    R = rotations(rng, K)
    if mirror:
        R[:, :, rng.integers(0, 3)] *= -1
    p = ((voxel + F(0.5)) * H0).astype(F)
    q = np.stack([rng.uniform(-0.3, 0.3, K), rng.uniform(-0.3, 0.3, K), np.ones(K)], 1)
    q *= rng.uniform(0.5, 4, K)[:, None]
    t = (p - np.einsum("nij,nj->ni", R, q)).astype(F)
    R = (R * scale).astype(F)
    d = p - t
    qv = [fma(R[:, 2, c], d[:, 2], fma(R[:, 1, c], d[:, 1], R[:, 0, c] * d[:, 0]))
          for c in range(3)]
    u = np.rint(fma(INTR[0], qv[0] / qv[2], INTR[2])).astype(int)
    v = np.rint(fma(INTR[1], qv[1] / qv[2], INTR[3])).astype(int)
    assert ((u >= 0) & (u < W - 2) & (v >= 0) & (v < H - 2)).all()
    ax, ay = (F(1) * u - INTR[2]) / INTR[0], (F(1) * v - INTR[3]) / INTR[1]
    rf = np.sqrt(fma(ay, ay, (ax * ax).astype(F)) + F(1)).astype(F)
    qn = np.sqrt(fma(qv[2], qv[2], fma(qv[1], qv[1], qv[0] * qv[0])))
    z = ((qn - trunc) / rf).astype(F)
    z = (z + rng.integers(-3, 4, K) * np.spacing(z)).astype(F)
    depth = np.zeros((K, H, W), F)
    depth[np.arange(K), v, u] = z
    return np.concatenate([R.reshape(K, 9), t], 1).astype(F), depth


@pytest.mark.parametrize("mirror", [False, True])
@pytest.mark.parametrize("scale", [0.001, 1.0, 1000.0])
@pytest.mark.parametrize("dims", [(1, 1, 1), (9, 9, 5), (65, 65, 65)])
def test_updates_at_minus_trunc(dev, dims, scale, mirror):
    print(f"[case] {dims}, matrices of scale {scale}, mirrored {mirror}", flush=True)
    X, Y, Z = dims
    rng = np.random.default_rng(X + int(1000 * scale) + mirror)
    trunc = F(0.02 * scale)
    poses, depth = frames_at_the_edge(rng, np.array(dims, F) - 1, scale, mirror, trunc)
    ref = np.zeros((Z, Y, X), np.uint32)
    O.integrate_ex(ref, H0, trunc, trunc, 60000, INTR, poses, depth, 1.0)
    seen = int(ref[-1, -1, -1] >> 16)
    assert 100 < seen < K  # some at or above -trunc, some below
    lib, it = _capi.load(), (ctypes.c_float * 4)(*INTR)
    vol = torch.zeros((Z, Y, X), dtype=torch.int32, device=dev)
    d_poses, d_depth = torch.from_numpy(poses).to(dev), torch.from_numpy(depth).to(dev)
    ws = torch.empty(lib.mcx_integrate_workspace_size(W, H), dtype=torch.uint8, device=dev)
    _capi.check(lib.mcx_integrate_ex(
        _ptr(vol), X, Y, Z, H0, trunc, trunc, 60000, it, _ptr(d_poses), _ptr(d_depth),
        _capi.DEPTH_F32, 1.0, W, H, K, _ptr(ws), ws.numel(),
        _stream_handle(dev)), "mcx_integrate_ex")
    got = vol.cpu().numpy().view(np.uint32)
    assert int(got[-1, -1, -1] >> 16) == seen
    assert got.tobytes() == ref.tobytes()
