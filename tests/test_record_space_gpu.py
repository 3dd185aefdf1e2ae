"""The differentiable forms without h_count when the record scratch is too
small: the mesh is whole, and the gradient is NaN throughout (no contribution
exists for the tiles that found no room, and none is read), for scratches that
hold no tile, some tiles and all but the last of them, single, recomputed and
batched; the same for a batch whose vertices' gradient has too few rows;
FusionGraph.check() reports both."""
import ctypes

import numpy as np
import pytest
import torch

from marching_cube_amd import _capi, batch, fusion_diff
from marching_cube_amd.mesh import _ptr, _stream_handle
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def noisy(shape, seed):
    rng = np.random.default_rng(seed)
    return (rng.uniform(0.25, 1.0, shape) * np.where(rng.random(shape) < 0.2, -1, 1)).astype(
        np.float32)


def workspace(nbytes, dev):
    ws = torch.empty(max(4096, nbytes), dtype=torch.uint8, device=dev)
    _capi.check(_capi.load().mcx_workspace_init(_ptr(ws), ws.numel(), _stream_handle(dev)))
    return ws


def staged_tiles(ws, dev):
    n = ctypes.c_int64(-1)
    _capi.check(_capi.load().mcx_workspace_staged_tiles(_ptr(ws), ws.numel(), ctypes.byref(n),
                                                        _stream_handle(dev)))
    return n.value


@pytest.mark.parametrize("recompute", [False, True])
@pytest.mark.parametrize("shape,share", [((9, 64, 66), 0.0), ((9, 64, 66), 0.5),
                                         ((70, 8, 64), 0.9), ((4, 73, 7), 0.5)])
def test_single(dev, shape, share, recompute):
    print(f"[case] {shape}, room for {share} of the records, recompute {recompute}", flush=True)
    lib, h = _capi.load(), 0.01
    Z, Y, X = shape
    f = noisy(shape, sum(shape))
    ref = O.extract(f, h, want=("pos",))["pos"]
    neg = (f < 0).astype(np.int32)
    corners = sum(neg[dz:Z - 1 + dz, dy:Y - 1 + dy, dx:X - 1 + dx]
                  for dz in (0, 1) for dy in (0, 1) for dx in (0, 1))
    records = int(share * ((corners > 0) & (corners < 8)).sum())
    ws = workspace(lib.mcx_extract_workspace_size_ex(X, Y, Z, records), dev)
    scratch = torch.zeros(max(16, lib.mcx_backward_scratch_size(X, Y, Z, ws.numel())),
                          dtype=torch.uint8, device=dev)
    v = torch.from_numpy(f).to(dev)
    pos = torch.empty(ref.shape, dtype=torch.float32, device=dev)
    g, gv = torch.ones_like(pos), torch.zeros_like(v)
    s = _stream_handle(dev)
    _capi.check(lib.mcx_extract_diff(_ptr(v), X, Y, Z, h, _ptr(pos), len(ref), None, None,
                                     _ptr(ws), ws.numel(), s))
    assert staged_tiles(ws, dev) > 0
    assert pos.cpu().numpy().tobytes() == ref.tobytes()
    back = lib.mcx_extract_backward_recompute if recompute else lib.mcx_extract_backward
    _capi.check(back(_ptr(v), X, Y, Z, h, _ptr(g), _ptr(gv), _ptr(ws), ws.numel(), _ptr(scratch),
                     scratch.numel(), s))
    assert torch.isnan(gv).all()


def test_planes_of_the_32_bit_count(dev):
    print("[case] 2 x 10000 x 11000, no room", flush=True)
    lib, (Z, Y, X), h = _capi.load(), (2, 10000, 11000), 0.01
    v = torch.ones((Z, Y, X), dtype=torch.float32, device=dev)
    v[0, 5::1000, 7::1000] = -1
    ws = workspace(lib.mcx_extract_workspace_size_ex(X, Y, Z, 16), dev)
    scratch = torch.zeros(max(16, lib.mcx_backward_scratch_size(X, Y, Z, ws.numel())),
                          dtype=torch.uint8, device=dev)
    g, gv = torch.ones((8192, 3), dtype=torch.float32, device=dev), torch.zeros_like(v)
    s = _stream_handle(dev)
    _capi.check(lib.mcx_extract_diff(_ptr(v), X, Y, Z, h, None, 0, None, None, _ptr(ws),
                                     ws.numel(), s))
    assert staged_tiles(ws, dev) > 0
    _capi.check(lib.mcx_extract_backward(_ptr(v), X, Y, Z, h, _ptr(g), _ptr(gv), _ptr(ws),
                                         ws.numel(), _ptr(scratch), scratch.numel(), s))
    assert torch.isnan(gv).all()


@pytest.mark.parametrize("records", [0, 3000])
def test_batched(dev, records):
    print(f"[case] batched, room for {records} records", flush=True)
    lib, h = _capi.load(), 0.01
    fs = [noisy(s, k) for k, s in enumerate([(9, 64, 66), (5, 16, 32), (19, 23, 29)])]
    flat = torch.from_numpy(np.concatenate([f.reshape(-1) for f in fs])).to(dev)
    at = np.cumsum([0] + [f.size for f in fs])
    plan = batch.BatchPlan([flat[at[k]:at[k + 1]].view(f.shape) for k, f in enumerate(fs)],
                           [h] * len(fs))
    refs = [O.extract(f, h, want=("pos",))["pos"] for f in fs]
    n = sum(len(r) for r in refs)
    ws = workspace(lib.mcx_batch_workspace_size(plan.handle, records), dev)
    scratch = torch.zeros(max(16, lib.mcx_batch_backward_scratch_size(plan.handle, ws.numel())),
                          dtype=torch.uint8, device=dev)
    vbase = torch.empty(len(fs) + 1, dtype=torch.int64, device=dev)
    pos = torch.empty((n, 3), dtype=torch.float32, device=dev)
    g, gv = torch.ones_like(pos), torch.zeros_like(flat)
    most = torch.zeros(1, dtype=torch.float32, device=dev)
    s = _stream_handle(dev)
    _capi.check(lib.mcx_extract_diff_batched(plan.handle, _ptr(pos), n, _ptr(vbase), None, None,
                                             _ptr(ws), ws.numel(), s))
    assert staged_tiles(ws, dev) > 0
    assert pos.cpu().numpy().tobytes() == np.concatenate(refs).tobytes()
    _capi.check(lib.mcx_extract_backward_batched(plan.handle, _ptr(g), _ptr(gv), _ptr(most),
                                                 _ptr(ws), ws.numel(), _ptr(scratch),
                                                 scratch.numel(), s))
    assert torch.isnan(gv).all() and torch.isnan(most).all()


def test_fusion_graph_reports_it(dev):
    print("[case] FusionGraph with a workspace that became too small", flush=True)
    K, W, H = 2, 64, 48
    depth = [torch.full((K, H, W), 1.0, device=dev)]
    poses = [torch.tensor([[1, 0, 0, 0, 1, 0, 0, 0, 1, 0.5, 0.5, -0.5]] * K,
                          dtype=torch.float32, device=dev)]
    targets = [torch.full((4, 3), 0.5, device=dev)]
    g = fusion_diff.FusionGraph([(24, 24, 24)], [1 / 24], depth, poses, targets,
                                [60.0, 60.0, 31.5, 23.5], trunc=0.1)
    g.step()
    g.check()
    assert int(g.total.item()) > 0 and torch.isfinite(g.gtsdf_all).all()
    g.ws = workspace(_capi.load().mcx_batch_workspace_size(g.plan.handle, 0), dev)
    g.step()
    with pytest.raises(_capi.McxError) as e:
        g.check()
    assert e.value.status == _capi.ERR_WORKSPACE
    assert torch.isnan(g.gtsdf_all).all()


@pytest.mark.parametrize("missing", [-1, 0, 1, 10**6])
def test_batched_rows(dev, missing):
    """The gradient's rows as many as the vertices, one more, one fewer, none."""
    print(f"[case] batched backward, {missing} rows short", flush=True)
    lib, h = _capi.load(), 0.01
    fs = [noisy(s, k) for k, s in enumerate([(9, 20, 21), (5, 16, 32)])]
    flat = torch.from_numpy(np.concatenate([f.reshape(-1) for f in fs])).to(dev)
    at = np.cumsum([0] + [f.size for f in fs])
    plan = batch.BatchPlan([flat[at[k]:at[k + 1]].view(f.shape) for k, f in enumerate(fs)],
                           [h] * len(fs))
    n = sum(O.extract(f, h, want=("pos",))["n"] for f in fs)
    rows = max(0, n - missing)
    ws = workspace(lib.mcx_batch_workspace_size(plan.handle, 65536), dev)
    scratch = torch.zeros(lib.mcx_batch_backward_scratch_size(plan.handle, ws.numel()),
                          dtype=torch.uint8, device=dev)
    vbase = torch.empty(len(fs) + 1, dtype=torch.int64, device=dev)
    g = torch.from_numpy(np.random.default_rng(2).standard_normal((n + 1, 3)).astype(
        np.float32)).to(dev)
    gv, plain = torch.zeros_like(flat), torch.zeros_like(flat)
    s = _stream_handle(dev)
    _capi.check(lib.mcx_extract_diff_batched(plan.handle, None, 0, _ptr(vbase), None, None,
                                             _ptr(ws), ws.numel(), s))
    assert staged_tiles(ws, dev) == 0 and int(vbase[-1].item()) == n
    _capi.check(lib.mcx_extract_backward_batched_rows(plan.handle, _ptr(g), rows, _ptr(gv), None,
                                                      _ptr(ws), ws.numel(), _ptr(scratch),
                                                      scratch.numel(), s))
    _capi.check(lib.mcx_extract_backward_batched(plan.handle, _ptr(g), _ptr(plain), None, _ptr(ws),
                                                 ws.numel(), _ptr(scratch), scratch.numel(), s))
    assert plain.abs().max() > 0 and torch.isfinite(plain).all()
    if rows < n:
        assert torch.isnan(gv).all()
    else:
        assert torch.equal(gv, plain)


def test_fusion_graph_past_its_capacity(dev):
    print("[case] FusionGraph with more vertices than its cap", flush=True)
    K, W, H = 2, 64, 48
    depth = [torch.full((K, H, W), 1.0, device=dev)]
    poses = [torch.tensor([[1, 0, 0, 0, 1, 0, 0, 0, 1, 0.5, 0.5, -0.5]] * K,
                          dtype=torch.float32, device=dev)]
    g = fusion_diff.FusionGraph([(24, 24, 24)], [1 / 24], depth, poses,
                                [torch.full((4, 3), 0.5, device=dev)],
                                [60.0, 60.0, 31.5, 23.5], trunc=0.1, cap=30)
    g.step()
    with pytest.raises(_capi.McxError) as e:
        g.check()
    assert e.value.status == _capi.ERR_CAPACITY
    assert torch.isnan(g.gtsdf_all).all()


@pytest.mark.parametrize("share", [0.0, 0.25, 0.5, 0.9, 1.3, 8.0])
@pytest.mark.parametrize("kind", ["short2", "f32"])
def test_plain_extraction(dev, kind, share):
    """No room, a pool that runs out on the way, room for all: the same mesh."""
    print(f"[case] plain extraction {kind}, records for {share} of the cubes", flush=True)
    from marching_cube_amd import synth
    lib, h, (Z, Y, X) = _capi.load(), 0.01, (40, 61, 67)
    if kind == "short2":
        f = synth.noise_volume((Z, Y, X), seed=3, p_zero_w=0.02)
        ref = O.extract(f, h, want=("vv",))
        want = ref["vv"].view(np.int32).reshape(-1, 7)
        v, elem = torch.from_numpy(f.view(np.int32)).to(dev), _capi.ELEM_SHORT2
    else:
        f = noisy((Z, Y, X), 3)
        ref = O.extract(f, h, want=("pos",))
        want = ref["pos"]
        v, elem = torch.from_numpy(f).to(dev), _capi.ELEM_F32
    tiles = (Z - 1) * ((X * Y + 511) // 512)
    records = int(share * (Z - 1) * (Y - 1) * (X - 1))
    ws = workspace(lib.mcx_extract_workspace_size_ex(X, Y, Z, records), dev)
    n = ctypes.c_int64(0)
    out = torch.empty(want.shape, dtype=torch.int32 if kind == "short2" else torch.float32,
                      device=dev)
    for _ in range(2):
        out.zero_()
        _capi.check(lib.mcx_extract(_ptr(v), elem, X, Y, Z, h,
                                    _ptr(out) if kind == "short2" else None,
                                    None if kind == "short2" else _ptr(out), None, None, len(want),
                                    None, ctypes.byref(n), _ptr(ws), ws.numel(),
                                    _stream_handle(dev)), "mcx_extract")
        assert n.value == len(want) and out.cpu().numpy().tobytes() == want.tobytes()
        staged = staged_tiles(ws, dev)
        assert staged <= tiles
        if share in (0.0, 0.25, 0.5):  # (at 0.9 the active cubes may all fit)
            assert staged > 0
        if share == 8.0:
            assert staged == 0
