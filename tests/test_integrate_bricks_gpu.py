"""GPU parity of the integration's bricks and frame tests at the sizes where
they can go wrong: volumes ending inside a brick or one voxel past it, frames
whose tiles end inside the image, cameras outside, inside and facing away,
depth values that are no measurement (0, negative, infinite, NaN, denormal),
and workspaces that hold some or none of the frames' tile tables.  Every
result is byte-compared with the oracle, voxel by voxel and frame by frame."""
import ctypes

import numpy as np
import pytest
import torch

from marching_cube_amd import _capi, fusion, synth
from marching_cube_amd.mesh import _ptr, _stream_handle
from oracle import oracle as O

pytestmark = pytest.mark.gpu

H0 = 0.02  # voxel size


def random_poses(rng, K, dims):
    """Cameras around, inside and beside a volume, most of them looking at it."""
    c = 0.5 * H0 * np.array(dims)
    out = np.zeros((K, 12), np.float32)
    for k in range(K):
        eye = c + rng.normal(size=3) * (1.0 if k % 3 else 0.05)
        fwd = c - eye + rng.normal(size=3) * 0.1
        if k % 7 == 6:
            fwd = -fwd
        fwd /= np.linalg.norm(fwd)
        right = np.cross(fwd, rng.normal(size=3))
        right /= np.linalg.norm(right)
        out[k, :9] = np.stack([right, np.cross(fwd, right), fwd], axis=1).reshape(-1)
        out[k, 9:] = eye
    return out


def random_depth(rng, K, H, W, f32):
    """Walls at several distances, holes, speckle; float frames hold odd values."""
    d = np.zeros((K, H, W))
    for k in range(K):
        d[k] = rng.uniform(0.3, 3.0)
        for _ in range(4):
            y, x = rng.integers(0, H), rng.integers(0, W)
            d[k, y:y + H // 2, x:x + W // 3] = rng.choice([0.0, rng.uniform(0.1, 2.0)])
    d *= rng.random(d.shape) > 0.02
    if not f32:
        return (d * 1000).astype(np.uint16)
    d = (d * 1000).astype(np.float32)
    odd = np.array([np.nan, np.inf, -np.inf, -1.0, 1e-39, 1e-30, 3e38], np.float32)
    at = rng.integers(0, d.size, 40)
    d.reshape(-1)[at] = odd[np.arange(40) % len(odd)]
    return d


@pytest.mark.parametrize("dims,K,W,H,f32", [
    ((33, 9, 5), 9, 96, 72, False), ((31, 8, 4), 1, 97, 71, True), ((64, 17, 37), 1, 40, 33, False),
    ((8, 40, 33), 17, 41, 24, True), ((1, 1, 9), 8, 96, 72, False), ((70, 7, 3), 2, 3, 3, True),
    ((95, 41, 66), 24, 160, 120, False), ((40, 33, 12), 7, 16, 200, True),
    ((20, 17, 9), 70, 64, 48, False), ((9, 20, 12), 64, 33, 40, True)])
def test_integrate_brick_edges(dev, dims, K, W, H, f32):
    print(f"[case] bricks {dims} K={K} {W}x{H} f32={f32}", flush=True)
    rng = np.random.default_rng(sum(dims) + K)
    X, Y, Z = dims
    poses, depth = random_poses(rng, K, dims), random_depth(rng, K, H, W, f32)
    intr = [0.9 * W, 0.8 * W, 0.5 * W - 0.5, 0.45 * H]
    start = synth.noise_volume((Z, Y, X), seed=K, p_zero_w=0.3, max_w=9)
    ref = start.copy()
    O.integrate_ex(ref, H0, 0.07, 0.05, 8, np.array(intr, np.float32), poses, depth)
    lib, it = _capi.load(), (ctypes.c_float * 4)(*intr)
    d_depth = torch.from_numpy(depth.view(np.int16) if not f32 else depth).to(dev)
    d_poses = torch.from_numpy(poses).to(dev)
    full = lib.mcx_integrate_workspace_size(W, H)
    tile = 8 * ((W + 7) // 8) * ((H + 7) // 8)
    sizes = {full, 4 * W * H, (4 * W * H + 255) // 256 * 256 + 256 + (K // 2) * tile}
    for nbytes in sorted(sizes):
        vol = torch.from_numpy(start.view(np.int32)).to(dev)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
        _capi.check(lib.mcx_integrate_ex(
            _ptr(vol), X, Y, Z, H0, 0.07, 0.05, 8, it, _ptr(d_poses), _ptr(d_depth),
            _capi.DEPTH_F32 if f32 else _capi.DEPTH_U16, 0.001, W, H, K, _ptr(ws), nbytes,
            _stream_handle(dev)), "mcx_integrate_ex")
        assert vol.cpu().numpy().view(np.uint32).tobytes() == ref.tobytes(), nbytes
    if f32:
        f0 = np.random.default_rng(1).uniform(-1, 1, (Z, Y, X)).astype(np.float32)
        rf, rw = f0.copy(), np.full((Z, Y, X), 2, np.int32)
        O.integrate_tsdf(rf, rw, H0, 0.05, 8, np.array(intr, np.float32), poses, depth, 0.001)
        for nbytes in sorted(sizes):
            tf = torch.from_numpy(f0).to(dev)
            tw = torch.full((Z, Y, X), 2, dtype=torch.int32, device=dev)
            ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
            _capi.check(lib.mcx_integrate_tsdf(
                _ptr(tf), _ptr(tw), X, Y, Z, H0, 0.05, 8, it, _ptr(d_poses), _ptr(d_depth), 0.001,
                W, H, K, _ptr(ws), nbytes, _stream_handle(dev)), "mcx_integrate_tsdf")
            assert tf.cpu().numpy().tobytes() == rf.tobytes(), nbytes
            assert tw.cpu().numpy().tobytes() == rw.tobytes(), nbytes


def test_workspace_that_is_too_small_is_refused(dev):
    print("[case] workspace below the ray factors", flush=True)
    vox = fusion.voxel_new((8, 8, 8), 0.05, H0, device=dev)
    depth = torch.ones((1, 9, 11), dtype=torch.int16, device=dev)
    poses = torch.zeros((1, 12), device=dev)
    ws = torch.empty(4096, dtype=torch.uint8, device=dev)
    st = _capi.load().mcx_integrate_ex(
        _ptr(vox.data), 8, 8, 8, H0, 0.05, 0.05, 8, (ctypes.c_float * 4)(9, 9, 5, 4), _ptr(poses),
        _ptr(depth), _capi.DEPTH_U16, 0.001, 11, 9, 1, _ptr(ws), 4 * 11 * 9 - 1,
        _stream_handle(dev))
    assert st == _capi.ERR_WORKSPACE
