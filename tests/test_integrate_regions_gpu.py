"""Integration of volumes whose regions are not whole rounds of the XCDs: the
grid's last workgroups lie past the last region (with blocks of extent 0 where
the region rows are a multiple of 8 and the last slab is partial).  Packed
volume, fp32 volume and its backward against the oracle and a taller
volume's launches."""
import ctypes

import numpy as np
import pytest
import torch

from marching_cube_amd import _capi, fusion_diff, synth
from marching_cube_amd.mesh import _ptr, _stream_handle
from oracle import oracle as O
from test_integrate_bricks_gpu import H0, random_depth, random_poses

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,K", [((96, 64, 684), 2), ((96, 64, 684), 1), ((33, 128, 390), 9),
                                    ((70, 64, 13), 40)])
def test_regions_past_the_last(dev, dims, K):
    print(f"[case] regions {dims} K={K}", flush=True)
    X, Y, Z = dims
    W, H, trunc = 96, 72, 0.05
    rng = np.random.default_rng(sum(dims) + K)
    poses, depth = random_poses(rng, K, dims), random_depth(rng, K, H, W, True)
    intr = np.array([0.9 * W, 0.8 * W, 0.5 * W - 0.5, 0.45 * H], np.float32)
    start = synth.noise_volume((Z, Y, X), seed=K, p_zero_w=0.3, max_w=9)
    ref = start.copy()
    O.integrate_ex(ref, H0, trunc, trunc, 8, intr, poses, depth)
    lib, it, s = _capi.load(), (ctypes.c_float * 4)(*intr), _stream_handle(dev)
    d_depth, d_poses = torch.from_numpy(depth).to(dev), torch.from_numpy(poses).to(dev)
    vol = torch.from_numpy(start.view(np.int32)).to(dev)
    ws = torch.empty(lib.mcx_integrate_workspace_size(W, H), dtype=torch.uint8, device=dev)
    _capi.check(lib.mcx_integrate_ex(_ptr(vol), X, Y, Z, H0, trunc, trunc, 8, it, _ptr(d_poses),
                                     _ptr(d_depth), _capi.DEPTH_F32, 0.001, W, H, K, _ptr(ws),
                                     ws.numel(), s), "mcx_integrate_ex")
    assert vol.cpu().numpy().view(np.uint32).tobytes() == ref.tobytes()
    rf = np.full((Z, Y, X), 0.5, np.float32)
    rw = np.full((Z, Y, X), 2, np.int32)
    O.integrate_tsdf(rf, rw, H0, trunc, 8, intr, poses, depth, 0.001)
    tf, tw = torch.full((Z, Y, X), 0.5, device=dev), torch.full((Z, Y, X), 2, dtype=torch.int32,
                                                                 device=dev)
    ig = fusion_diff._Integrator((Z, Y, X), W, H, K, H0, trunc, 8, intr, dev)
    ig.forward(tf, tw, d_poses, d_depth, 0.001)
    assert tf.cpu().numpy().tobytes() == rf.tobytes()
    assert tw.cpu().numpy().tobytes() == rw.tobytes()
    # backward: of a gradient in the far half along z alone, as that of a taller
    # volume with whole rounds and the same gradient
    g = torch.zeros((Z, Y, X), device=dev)
    g[Z // 2:] = torch.from_numpy(rng.standard_normal((Z - Z // 2, Y, X)).astype(np.float32)).to(dev)
    w0 = torch.full((Z, Y, X), 2, dtype=torch.int32, device=dev)
    gd, gd2 = torch.empty_like(d_depth), torch.empty_like(d_depth)
    ig.backward(g, w0, d_poses, d_depth, gd, 0.001)
    Z2 = (Z + 255) // 256 * 256
    pad = torch.zeros((Z2 - Z, Y, X), device=dev)
    ig2 = fusion_diff._Integrator((Z2, Y, X), W, H, K, H0, trunc, 8, intr, dev)
    ig2.backward(torch.cat([g, pad]), torch.cat([w0, pad.to(torch.int32)]), d_poses, d_depth, gd2,
                 0.001)
    assert gd.nan_to_num().abs().max() > 0 and gd.cpu().numpy().tobytes() == gd2.cpu().numpy().tobytes()
