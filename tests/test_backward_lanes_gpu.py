"""The integration backward with a gradient on some lanes of a brick only: the
gradients of a set of voxels and of all others add up to that of all voxels (the
accumulators are exact sums at one scale, since all have the same largest
|gradient|; each result is rounded once to fp32), for bricks of one plane and of
four, inside and across the edges of frames and volumes."""
import numpy as np
import pytest
import torch

from marching_cube_amd import fusion_diff
from test_integrate_bricks_gpu import H0, random_depth, random_poses

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("every", [2, 37, 1000])
@pytest.mark.parametrize("dims,K", [((33, 9, 5), 9), ((70, 67, 61), 3), ((70, 67, 61), 16),
                                    ((260, 260, 130), 8)])
def test_sets_of_voxels_add_up(dev, dims, K, every):
    print(f"[case] backward {dims} K={K}, one voxel in {every}", flush=True)
    X, Y, Z = dims
    W, H = 96, 72
    rng = np.random.default_rng(X + K)
    poses = torch.from_numpy(random_poses(rng, K, dims)).to(dev)
    depth = torch.from_numpy(random_depth(rng, K, H, W, True)).to(dev)
    intr = np.array([0.9 * W, 0.8 * W, 0.5 * W - 0.5, 0.45 * H], np.float32)
    ig = fusion_diff._Integrator((Z, Y, X), W, H, K, H0, 0.05, 8, intr, dev)
    w0 = torch.full((Z, Y, X), 2, dtype=torch.int32, device=dev)
    g = torch.from_numpy(rng.choice(np.array([-1, 1], np.float32), (Z, Y, X))).to(dev)
    some = torch.zeros(Z * Y * X, dtype=torch.bool, device=dev)
    some[rng.integers(0, every)::every] = True
    some = some.view(Z, Y, X)
    out = []
    for part in (g, g * some, g * ~some):
        gd = torch.empty_like(depth)
        ig.backward(part, w0, poses, depth, gd, 0.001)
        out.append(gd.double())
    most = float(out[0].abs().max())
    assert most > 0
    if int(some.sum()) > 50:  # (a voxel or two may be seen by no frame)
        assert float(out[1].abs().max()) > 0
    assert float((out[1] + out[2] - out[0]).abs().max()) <= 3 * 2.0 ** -24 * most
