"""The ver_voxel map, cleared by workgroups beside the scan: maps full of other
values, of sizes that end anywhere in 16 bytes, aligned and not (cleared before
the count then), of more bytes than one pass of the clearing workgroups, and
volumes without a cube, against the oracle; the words around the map untouched."""
import numpy as np
import pytest
import torch

from marching_cube_amd import mesh, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1, 8])
@pytest.mark.parametrize("shape", [(2, 2, 2), (3, 5, 7), (1, 6, 5), (9, 10, 11), (40, 33, 65),
                                   (300, 240, 250)])
def test_map_is_cleared(dev, shape, offset):
    print(f"[case] ver_voxel clear {shape} +{offset}", flush=True)
    vol, h = synth.noise_volume(shape, seed=3), 0.1
    n = int(np.prod(shape))
    buf = torch.full((n + 32,), -7, dtype=torch.int16, device=dev)
    ver = buf[8 + offset:8 + offset + n].view(shape)
    v = torch.from_numpy(vol.view(np.int32)).to(dev)
    count = mesh.extract_into(v, h, ver_voxel=ver, cap=1 << 40)
    ref = O.extract(vol, h, want=("ver_voxel",))
    assert count == ref["n"]
    got = buf.cpu().numpy()
    assert got[8 + offset:8 + offset + n].tobytes() == ref["ver_voxel"].tobytes()
    assert (got[:8 + offset] == -7).all() and (got[8 + offset + n:] == -7).all()
