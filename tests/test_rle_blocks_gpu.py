"""The codec's blocks against the oracle: slices that end just before, at and
just after a block of 4096 voxels, of one voxel, of many blocks; runs that cross
blocks and are cut at 0x3fff voxels (literal and saturated), one start per
block; more blocks than a scan group holds, and more groups than one."""
import ctypes

import numpy as np
import pytest
import torch

import test_rle_oracle as RO
from marching_cube_amd import _capi, mesh, volio
from oracle import oracle as O
from test_volio_gpu import dev_vol, random_volume

pytestmark = pytest.mark.gpu


def sparse_volume(shape, seed, every):
    """A start about every `every` voxels; saturated and literal runs."""
    rng = np.random.default_rng(seed)
    n = int(np.prod(shape))
    starts = np.sort(rng.choice(n, max(1, n // every), replace=False))
    vals = rng.choice([RO.vox(32766, 0), RO.vox(-32766, 0), RO.vox(32766, 3), RO.vox(5, 9),
                       RO.vox(-32767, 1), RO.vox(0, 0)], len(starts) + 1).astype(np.uint32)
    return vals[np.searchsorted(starts, np.arange(n), side="right")].reshape(shape)


SHAPES = [(3, 1, 1), (5, 63, 65), (4, 64, 64), (4, 241, 17), (3, 33, 31), (2, 150, 333),
          (2000, 3, 7), (3, 4096, 33)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("every", [1, 40, 3000, 40000])
def test_blocks_bit_exact(dev, shape, every):
    print(f"[case] rle blocks {shape}, a start in {every}", flush=True)
    Z, Y, X = shape
    v = random_volume(shape, 7) if every == 1 else sparse_volume(shape, every + Z, every)
    ref = O.rle_encode_dump(v)
    got = volio.encode(dev_vol(v, dev))
    assert got == ref
    back = volio.decode(got, X, Y, volio.slice_offsets(got, Z), dev)
    assert back.cpu().numpy().tobytes() == O.rle_decode_dump(ref, X, Y, 0, Z).tobytes()


@pytest.mark.parametrize("X,nz", [(1, 65535), (69632, 65535)])
def test_many_blocks(dev, X, nz):
    """65,535 slices of 1 and of 17 blocks: two and three levels of the scan."""
    print(f"[case] rle {nz} slices of {X}", flush=True)
    v = torch.full((nz, 1, X), 32766, dtype=torch.int32, device=dev)
    k = (X + 0x3fff - 1) // 0x3fff
    lens = [min(0x3fff, X - r * 0x3fff) for r in range(k)]
    one = np.array([2 * k, 0] + [n | 1 << 14 for n in lens], np.uint16)
    lib = _capi.load()
    out = torch.zeros(nz * (4 + 2 * k), dtype=torch.uint8, device=dev)
    ws = torch.empty(lib.mcx_rle_encode_workspace_size(X, 1, nz), dtype=torch.uint8, device=dev)
    total = ctypes.c_int64(0)
    _capi.check(lib.mcx_rle_encode(mesh._ptr(v), X, 1, nz, 0, nz, mesh._ptr(out), out.numel(),
                                   None, ctypes.byref(total), mesh._ptr(ws), ws.numel(),
                                   mesh._stream_handle(dev)), "mcx_rle_encode")
    assert total.value == out.numel()
    assert out.cpu().numpy().tobytes() == one.tobytes() * nz


@pytest.mark.parametrize("n", [volio.STAGE_BYTES + d for d in (-1, 0, 1)] +
                         [3 * volio.STAGE_BYTES - 1, 3 * volio.STAGE_BYTES + 5])
def test_staged_copies(dev, n):
    print(f"[case] staged copies of {n} bytes", flush=True)
    data = np.random.default_rng(n).integers(0, 256, n, dtype=np.uint8).tobytes()
    d = volio._to_device(data, dev)
    assert d.cpu().numpy().tobytes() == data
    assert volio._to_bytes(d) == data


def test_slabs_when_the_dump_is_large(dev):
    """All slices at once would need more than the slab's buffer."""
    print("[case] rle slabs", flush=True)
    v = np.arange(9 * 70 * 80, dtype=np.uint32).reshape(9, 70, 80) % 1000 | np.uint32(7 << 16)
    for slices in (1, 2, 4, 9):
        assert volio.encode(dev_vol(v, dev), slab_voxels=slices * 5600) == O.rle_encode_dump(v)
