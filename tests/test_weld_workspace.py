"""The weld's workspace is what its arrays take: one 4-byte table of at least two
slots a vertex, two 4-byte words a vertex, a word per 1024 vertices; a call
stays inside it and is refused with less."""
import ctypes

import numpy as np
import pytest

from marching_cube_amd import _capi


@pytest.mark.parametrize("V", [1, 511, 512, 513, 1024, 1025, 2_450_000, (1 << 31) - 1])
def test_size(V):
    slots = 1024
    while slots < 2 * V:
        slots *= 2
    arrays = 4 * slots + 2 * 4 * V + 4 * ((V + 1023) // 1024 + 1)
    got = _capi.load().mcx_weld_workspace_size(V)
    assert arrays <= got <= arrays + 4 * 256  # each array starts at 256 bytes


def test_size_of_nothing():
    assert _capi.load().mcx_weld_workspace_size(-1) == 0
    assert _capi.load().mcx_weld_workspace_size(0) > 0


@pytest.mark.gpu
@pytest.mark.parametrize("V", [1, 513, 1024, 70001])
def test_stays_inside(dev, V):
    import torch

    from marching_cube_amd.mesh import _ptr, _stream_handle
    from test_weld_gpu import ref_weld
    print(f"[case] weld in exactly its workspace, V={V}", flush=True)
    lib = _capi.load()
    keys = np.random.default_rng(V).integers(0, V // 3 + 1, V)
    pos = np.random.default_rng(1).standard_normal((V, 3)).astype(np.float32)
    k, p = torch.from_numpy(keys).to(dev), torch.from_numpy(pos).to(dev)
    upos = torch.empty((V, 3), dtype=torch.float32, device=dev)
    idx = torch.empty(V, dtype=torch.int32, device=dev)
    nu = ctypes.c_int64(0)
    n = lib.mcx_weld_workspace_size(V)
    ws = torch.full((n + 4096,), 0x5a, dtype=torch.uint8, device=dev)
    args = (_ptr(k), _ptr(p), 3, V, _ptr(upos), _ptr(idx), None, ctypes.byref(nu), _ptr(ws))
    assert lib.mcx_weld(*args, n - 1, _stream_handle(dev)) == _capi.ERR_WORKSPACE
    _capi.check(lib.mcx_weld(*args, n, _stream_handle(dev)), "mcx_weld")
    rupos, ridx = ref_weld(keys, pos)
    assert upos[:nu.value].cpu().numpy().tobytes() == np.ascontiguousarray(rupos).tobytes()
    assert idx.cpu().numpy().tobytes() == ridx.tobytes()
    assert (ws[n:] == 0x5a).all()
