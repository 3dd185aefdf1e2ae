"""Integration where the planes of a brick and the use of tile tables change:
volumes just below and above 2^17, 2^18 and 2^20 voxels, numbers and sizes of
frames on both sides of their limits, volumes that end inside a brick, and
workspaces with room for some or none of the tables; single volumes and batches,
byte-compared with the oracle."""
import ctypes

import numpy as np
import pytest
import torch

from marching_cube_amd import _capi, batch, synth
from marching_cube_amd.mesh import _ptr, _stream_handle
from oracle import oracle as O
from test_integrate_bricks_gpu import H0, random_depth, random_poses

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,K,W,H,f32", [
    ((64, 64, 32), 3, 96, 72, False), ((64, 64, 33), 32, 200, 170, True),
    ((64, 64, 33), 33, 200, 170, False), ((64, 64, 33), 40, 200, 160, True),
    ((64, 64, 64), 4, 97, 71, False), ((65, 64, 64), 7, 96, 72, True),
    ((65, 64, 64), 8, 96, 72, True), ((65, 64, 64), 9, 640, 480, False),
    ((70, 67, 61), 9, 40, 33, True), ((257, 33, 37), 70, 96, 72, False),
    ((33, 129, 70), 16, 33, 200, True), ((129, 127, 65), 1, 97, 71, False),
    ((129, 127, 65), 3, 96, 72, True), ((129, 127, 63), 1, 96, 72, True)])
def test_single(dev, dims, K, W, H, f32):
    print(f"[case] planes {dims} K={K} {W}x{H} f32={f32}", flush=True)
    rng = np.random.default_rng(sum(dims) + K)
    X, Y, Z = dims
    poses, depth = random_poses(rng, K, dims), random_depth(rng, K, H, W, f32)
    intr = [0.9 * W, 0.8 * W, 0.5 * W - 0.5, 0.45 * H]
    start = synth.noise_volume((Z, Y, X), seed=K, p_zero_w=0.3, max_w=9)
    ref = start.copy()
    O.integrate_ex(ref, H0, 0.07, 0.05, 8, np.array(intr, np.float32), poses, depth)
    assert ref.tobytes() != start.tobytes()
    lib, it, s = _capi.load(), (ctypes.c_float * 4)(*intr), _stream_handle(dev)
    d_depth = torch.from_numpy(depth if f32 else depth.view(np.int16)).to(dev)
    d_poses = torch.from_numpy(poses).to(dev)
    sizes = [4 * W * H, lib.mcx_integrate_workspace_size_frames(W, H, K // 2),
             lib.mcx_integrate_workspace_size_frames(W, H, K)]
    for nbytes in sizes:
        vol = torch.from_numpy(start.view(np.int32)).to(dev)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
        _capi.check(lib.mcx_integrate_ex(
            _ptr(vol), X, Y, Z, H0, 0.07, 0.05, 8, it, _ptr(d_poses), _ptr(d_depth),
            _capi.DEPTH_F32 if f32 else _capi.DEPTH_U16, 0.001, W, H, K, _ptr(ws), nbytes, s),
            "mcx_integrate_ex")
        assert vol.cpu().numpy().view(np.uint32).tobytes() == ref.tobytes(), nbytes
    if not f32:
        return
    f0 = np.random.default_rng(1).uniform(-1, 1, (Z, Y, X)).astype(np.float32)
    rf, rw = f0.copy(), np.full((Z, Y, X), 2, np.int32)
    O.integrate_tsdf(rf, rw, H0, 0.05, 8, np.array(intr, np.float32), poses, depth, 0.001)
    for nbytes in sizes:
        tf = torch.from_numpy(f0).to(dev)
        tw = torch.full((Z, Y, X), 2, dtype=torch.int32, device=dev)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
        _capi.check(lib.mcx_integrate_tsdf(_ptr(tf), _ptr(tw), X, Y, Z, H0, 0.05, 8, it,
                                           _ptr(d_poses), _ptr(d_depth), 0.001, W, H, K, _ptr(ws),
                                           nbytes, s), "mcx_integrate_tsdf")
        assert tf.cpu().numpy().tobytes() == rf.tobytes(), nbytes
        assert tw.cpu().numpy().tobytes() == rw.tobytes(), nbytes


@pytest.mark.parametrize("copies,K,W,H", [(1, 3, 40, 33), (3, 9, 40, 33), (3, 9, 300, 200),
                                          (12, 4, 40, 33)])
def test_batched(dev, copies, K, W, H):
    """Batches of 57 thousand to 700 thousand voxels: the fused volumes against the
    oracle, and a sparse gradient's backward against the single volumes'."""
    print(f"[case] planes, {copies} times two volumes, K={K} {W}x{H}", flush=True)
    shapes = [(31, 40, 33), (13, 20, 65)] * copies
    rng = np.random.default_rng(copies + K)
    poses = [random_poses(rng, K, s[::-1]) for s in shapes]
    depth = [random_depth(rng, K, H, W, True) for _ in shapes]
    intr = np.array([0.9 * W, 0.8 * W, 0.5 * W - 0.5, 0.45 * H], np.float32)
    at = np.cumsum([0] + [int(np.prod(s)) for s in shapes])
    t = torch.empty(int(at[-1]), device=dev)
    w = torch.empty(int(at[-1]), dtype=torch.int32, device=dev)
    plan = batch.BatchPlan([t[at[k]:at[k + 1]].view(s) for k, s in enumerate(shapes)],
                           [H0] * len(shapes))
    lib, it, s = _capi.load(), (ctypes.c_float * 4)(*intr), _stream_handle(dev)
    d_depth = torch.from_numpy(np.stack(depth)).to(dev)
    d_poses = torch.from_numpy(np.stack(poses)).to(dev)
    ws = torch.empty(lib.mcx_integrate_workspace_size_frames(W, H, len(shapes) * K),
                     dtype=torch.uint8, device=dev)
    _capi.check(lib.mcx_integrate_tsdf_batched(
        plan.handle, _ptr(t), _ptr(w), 1, -1.0, 0.05, 8, it, _ptr(d_poses), _ptr(d_depth), 0.001,
        W, H, K, _ptr(ws), ws.numel(), s), "mcx_integrate_tsdf_batched")
    for k, shape in enumerate(shapes):
        rf, rw = np.full(shape, -1.0, np.float32), np.zeros(shape, np.int32)
        O.integrate_tsdf(rf, rw, H0, 0.05, 8, intr, poses[k], depth[k], 0.001)
        assert t[at[k]:at[k + 1]].cpu().numpy().tobytes() == rf.tobytes(), k
        assert w[at[k]:at[k + 1]].cpu().numpy().tobytes() == rw.tobytes(), k
    from marching_cube_amd import fusion_diff
    g = torch.zeros_like(t)
    g[::3] = torch.from_numpy(rng.choice(np.array([-1, 1], np.float32), len(g[::3]))).to(dev)
    gd = torch.empty_like(d_depth)
    wb = torch.empty(lib.mcx_integrate_tsdf_backward_batched_workspace_size(plan.handle, W, H, K),
                     dtype=torch.uint8, device=dev)
    _capi.check(lib.mcx_integrate_tsdf_backward_batched(
        plan.handle, _ptr(g), None, None, 0.05, 8, it, _ptr(d_poses), _ptr(d_depth), 0.001, W, H,
        K, _ptr(gd), _ptr(wb), wb.numel(), s), "mcx_integrate_tsdf_backward_batched")
    assert gd.abs().max() > 0
    for k in (0, 1, len(shapes) - 2, len(shapes) - 1):  # the same largest |gradient|: same scale
        ig = fusion_diff._Integrator(shapes[k], W, H, K, H0, 0.05, 8, intr, dev)
        one = torch.empty_like(d_depth[k])
        ig.backward(g[at[k]:at[k + 1]].view(shapes[k]), torch.zeros(shapes[k], dtype=torch.int32,
                                                                   device=dev),
                    d_poses[k], d_depth[k], one, 0.001)
        assert torch.equal(gd[k], one), k
