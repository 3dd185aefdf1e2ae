"""The backward's gather where the number of waves that share a window of 512
voxels changes: volumes just below and above the limits, planes that end inside a
window's half, quarter and 64, and batches of them; against the oracle's FP64
gradient, and the batch bit for bit against single volumes (which other splits
serve)."""
import ctypes

import numpy as np
import pytest
import torch

from marching_cube_amd import _capi, batch, diff
from marching_cube_amd.mesh import _ptr, _stream_handle
from oracle import oracle as O

pytestmark = pytest.mark.gpu

H = 0.01


def field(shape, seed):
    """Mostly outside, with inside voxels strewn in: long runs without a cube."""
    rng = np.random.default_rng(seed)
    f = rng.uniform(0.25, 1.0, shape).astype(np.float32)
    at = rng.integers(0, f.size, max(8, f.size // 2000))
    f.reshape(-1)[at] *= -1
    return f


@pytest.mark.parametrize("shape", [(2, 3, 21), (5, 8, 17), (9, 13, 20), (7, 33, 31),
                                   (128, 128, 128), (129, 127, 129), (131, 251, 255),
                                   (127, 257, 257)])
def test_single(dev, shape):
    print(f"[case] gather {shape}", flush=True)
    f = field(shape, sum(shape))
    ex = diff.DiffExtractor(shape, dev)
    v = torch.from_numpy(f).to(dev)
    n = len(ex.forward(v, H))
    g = np.random.default_rng(1).standard_normal((n, 3)).astype(np.float32)
    got = ex.backward(v, torch.from_numpy(g).to(dev), out=torch.full_like(v, 7.0)).cpu().numpy()
    want = O.extract_backward_f64(f, H, g.astype(np.float64))
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
    assert (got[want == 0] == 0).all()


@pytest.mark.parametrize("copies", [1, 40, 150])
def test_batched(dev, copies):
    print(f"[case] gather, a batch of {copies} times three shapes", flush=True)
    lib, shapes = _capi.load(), [(9, 13, 20), (31, 40, 33), (5, 8, 17)]
    fs = [field(s, k) for k, s in enumerate(shapes)]
    flat = torch.from_numpy(np.concatenate([f.reshape(-1) for f in fs] * copies)).to(dev)
    at = np.cumsum([0] + [f.size for f in fs] * copies)
    plan = batch.BatchPlan([flat[at[k]:at[k + 1]].view(shapes[k % 3]) for k in range(3 * copies)],
                           [H] * (3 * copies))
    ws = torch.zeros(lib.mcx_batch_workspace_size(plan.handle, len(flat)), dtype=torch.uint8,
                     device=dev)
    scratch = torch.empty(lib.mcx_batch_backward_scratch_size(plan.handle, ws.numel()),
                          dtype=torch.uint8, device=dev)
    vbase = torch.empty(3 * copies + 1, dtype=torch.int64, device=dev)
    count, s = ctypes.c_int64(0), _stream_handle(dev)
    assert lib.mcx_extract_diff_batched(plan.handle, None, 0, _ptr(vbase), None,
                                        ctypes.byref(count), _ptr(ws), ws.numel(),
                                        s) == _capi.ERR_CAPACITY
    vb = vbase.cpu().numpy()
    g = torch.from_numpy(np.random.default_rng(1).standard_normal((count.value, 3)).astype(
        np.float32)).to(dev)
    gv, most = torch.full_like(flat, 7.0), torch.zeros(1, dtype=torch.float32, device=dev)
    _capi.check(lib.mcx_extract_backward_batched(plan.handle, _ptr(g), _ptr(gv), _ptr(most),
                                                 _ptr(ws), ws.numel(), _ptr(scratch),
                                                 scratch.numel(), s))
    assert float(most) == float(gv.abs().max()) > 0
    for k in [0, 1, 2, 3 * copies - 2, 3 * copies - 1]:
        ex = diff.DiffExtractor(shapes[k % 3], dev)
        v = torch.from_numpy(fs[k % 3]).to(dev)
        assert len(ex.forward(v, H)) == vb[k + 1] - vb[k]
        one = ex.backward(v, g[vb[k]:vb[k + 1]])
        assert torch.equal(gv[at[k]:at[k + 1]].view(shapes[k % 3]), one), k
