"""The weld's table where groups of keys meet: dense runs of distinct keys that
half fill it, in order, shuffled and repeated, and keys whose whole sequences of
slots are the same, so that they go through every line of the sequence and on to
the slots after it; against numpy's first occurrences."""
import ctypes

import numpy as np
import pytest
import torch

from marching_cube_amd import _capi
from marching_cube_amd.mesh import _ptr, _stream_handle
from test_weld_gpu import ref_weld

pytestmark = pytest.mark.gpu


def mix64(k):
    k = k ^ (k >> np.uint64(33))
    k = k * np.uint64(0xff51afd7ed558ccd)
    k = k ^ (k >> np.uint64(33))
    k = k * np.uint64(0xc4ceb9fe1a85ec53)
    return k ^ (k >> np.uint64(33))


def meeting_keys(count):
    """Keys with the same first slot and step in a table of 1024 slots (32 lines)."""
    keys = np.random.default_rng(5).integers(0, 1 << 62, 1 << 23).astype(np.uint64)
    m = mix64(keys >> np.uint64(5))
    line, place = m & np.uint64(31), (keys ^ (m >> np.uint64(59))) & np.uint64(31)
    step = (m >> np.uint64(32)) & np.uint64(15)
    same = keys[(line == 3) & (place == 7) & (step == 2)]
    assert len(same) >= count
    return same[:count].astype(np.int64)


def run(dev, keys):
    V = len(keys)
    pos = np.random.default_rng(1).standard_normal((V, 3)).astype(np.float32)
    lib = _capi.load()
    k, p = torch.from_numpy(keys).to(dev), torch.from_numpy(pos).to(dev)
    upos = torch.empty((V, 3), dtype=torch.float32, device=dev)
    idx = torch.empty(V, dtype=torch.int32, device=dev)
    ws = torch.empty(lib.mcx_weld_workspace_size(V), dtype=torch.uint8, device=dev)
    nu = ctypes.c_int64(0)
    _capi.check(lib.mcx_weld(_ptr(k), _ptr(p), 3, V, _ptr(upos), _ptr(idx), None, ctypes.byref(nu),
                             _ptr(ws), ws.numel(), _stream_handle(dev)), "mcx_weld")
    rupos, ridx = ref_weld(keys, pos)
    assert nu.value == len(rupos)
    assert upos[:nu.value].cpu().numpy().tobytes() == np.ascontiguousarray(rupos).tobytes()
    assert idx.cpu().numpy().tobytes() == ridx.tobytes()


@pytest.mark.parametrize("V", [31, 512, 513, 70000, 524288])
@pytest.mark.parametrize("pattern", ["order", "shuffled", "falling", "four times"])
def test_dense_keys(dev, pattern, V):
    print(f"[case] weld, dense keys {pattern}, V={V}", flush=True)
    i = np.arange(V, dtype=np.int64)
    run(dev, {"order": i, "shuffled": np.random.default_rng(V).permutation(i), "falling": V - i,
              "four times": i % (V // 4 + 1)}[pattern])


@pytest.mark.parametrize("V", [16, 17, 33, 300])
def test_keys_with_one_sequence_of_slots(dev, V):
    print(f"[case] weld, {V} keys that meet everywhere", flush=True)
    run(dev, meeting_keys(V))
    run(dev, np.repeat(meeting_keys(V // 2), 3)[:V])
