"""The weld's blocks of 1024 vertices and its table of indices against numpy's
first occurrences: sizes at the edges of a block and past the block sums of one
scan pass (4096 blocks), keys that all fall in one group of the table, that
come in falling order (later workgroups hold the first occurrence of none), that
differ in the high half only, and that are all distinct; strides of 3 and 7."""
import ctypes

import numpy as np
import pytest
import torch

from marching_cube_amd import _capi, mesh
from test_weld_gpu import ref_weld

pytestmark = pytest.mark.gpu


def make_keys(pattern, V):
    i = np.arange(V, dtype=np.int64)
    if pattern == "falling":
        return (V - i) // 5 * 32
    if pattern == "high":
        return (i % 997) << 32
    if pattern == "distinct":
        return i * 32
    if pattern == "group":
        return i % 32
    return np.random.default_rng(V).integers(0, V // 6 + 1, V) * 3 + 2


@pytest.mark.parametrize("pattern,V,stride", [
    ("distinct", 1, 3), ("distinct", 512, 7), ("distinct", 1023, 3), ("falling", 1024, 3),
    ("group", 1025, 7), ("high", 2049, 3), ("falling", 70001, 7), ("distinct", 262144, 3),
    ("random", 4096 * 1024 + 1, 3)])
def test_blocks(dev, pattern, V, stride):
    print(f"[case] weld blocks {pattern} V={V}", flush=True)
    keys = make_keys(pattern, V)
    pos = np.random.default_rng(1).standard_normal((V, stride)).astype(np.float32)
    lib = _capi.load()
    k, p = torch.from_numpy(keys).to(dev), torch.from_numpy(pos).to(dev)
    upos = torch.empty((V, 3), dtype=torch.float32, device=dev)
    idx = torch.empty(V, dtype=torch.int32, device=dev)
    d_nu = torch.zeros(1, dtype=torch.int64, device=dev)
    ws = torch.empty(lib.mcx_weld_workspace_size(V), dtype=torch.uint8, device=dev)
    nu = ctypes.c_int64(0)
    _capi.check(lib.mcx_weld(mesh._ptr(k), mesh._ptr(p), stride, V, mesh._ptr(upos),
                             mesh._ptr(idx), mesh._ptr(d_nu), ctypes.byref(nu), mesh._ptr(ws),
                             ws.numel(), mesh._stream_handle(dev)), "mcx_weld")
    rupos, ridx = ref_weld(keys, pos[:, :3])
    assert nu.value == int(d_nu) == len(rupos)
    assert upos[:nu.value].cpu().numpy().tobytes() == np.ascontiguousarray(rupos).tobytes()
    assert idx.cpu().numpy().tobytes() == ridx.tobytes()
