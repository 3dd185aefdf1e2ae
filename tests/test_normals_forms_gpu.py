"""The normals' exact short forms and paired corner loads against the oracle,
bit for bit: spacings and positions inside and outside the forms' range (zeros
of both signs, denormals, 2^-61), positions on voxels, on the last cell and
outside, flat and saturated cells, widths that leave pairs at odd words."""
import numpy as np
import pytest
import torch

from marching_cube_amd import mesh
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h", [0.02, 1.0 / 3.0, 2.0 ** -60, 2.0 ** -61, 2.0 ** 61])
@pytest.mark.parametrize("shape", [(2, 2, 2), (5, 9, 7), (12, 6, 33)])
def test_normals_bit_exact(dev, shape, h):
    print(f"[case] normals forms {shape} h={h}", flush=True)
    rng = np.random.default_rng(sum(shape))
    Z, Y, X = shape
    t = rng.integers(-32767, 32768, shape)
    t[rng.random(shape) < 0.5] = 1200  # flat cells: a zero norm
    t[rng.random(shape) < 0.1] = 1201
    t[rng.random(shape) < 0.03] = 32766
    vol = t.astype(np.int16).view(np.uint16).astype(np.uint32) | np.uint32(1 << 16)
    n = 4000
    p = rng.uniform(-0.2, 1.05, (n, 3)) * np.array([X, Y, Z])
    whole = rng.random((n, 3)) < 0.2
    p[whole] = np.rint(p[whole])
    p = (p * h).astype(np.float32)
    for v in (0.0, -0.0, 1e-42, 2.0 ** -61, -1e-30):
        p[rng.random((n, 3)) < 0.03] = np.float32(v)
    ref = O.normals(vol, h, p)
    got = mesh.normals(torch.from_numpy(vol.view(np.int32)).to(dev), h,
                       torch.from_numpy(p).to(dev)).cpu().numpy()
    assert got.tobytes() == ref.tobytes()
    assert (np.abs(ref).max(axis=1) > 0).any() or h != 0.02
