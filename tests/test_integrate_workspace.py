"""The integration's workspace is sized by the frames of a call: the size
function's values (no GPU needed), and what a live differentiable fusion
holds."""
import pytest

from marching_cube_amd import _capi


def table(W, H):
    """Bytes of a frame's tiles: 8 x 8 and 32 x 32 pixels, two floats each."""
    return 8 * (((W + 7) // 8) * ((H + 7) // 8) + ((W + 31) // 32) * ((H + 31) // 32))


@pytest.mark.parametrize("W,H", [(3, 3), (97, 71), (640, 480), (1920, 1080), (8192, 8192)])
def test_sizes(W, H):
    size = _capi.load().mcx_integrate_workspace_size_frames
    base = (4 * W * H + 255) // 256 * 256 + 256
    most = max(1, (32 << 20) // table(W, H))  # tables are kept for no more frames
    for frames in (0, 1, 2, most, most + 1, 1 << 40):
        assert size(W, H, frames) == base + min(frames, most) * table(W, H)
    assert _capi.load().mcx_integrate_workspace_size(W, H) == size(W, H, most)


def test_sizes_of_nothing():
    size = _capi.load().mcx_integrate_workspace_size_frames
    assert size(0, 5, 1) == size(5, 0, 1) == size(-1, 5, 1) == size(5, 5, -1) == 0
    assert _capi.load().mcx_integrate_workspace_size(0, 5) == 0


@pytest.mark.gpu
def test_live_fusions_hold_no_forward_workspace(dev):
    import torch

    from marching_cube_amd import fusion_diff
    print("[case] eight live fusions of 16^3, one 64x48 frame each", flush=True)
    f0, w0 = fusion_diff.tsdf_init((16, 16, 16), dev, -1.0)
    poses = torch.tensor([[1, 0, 0, 0, 1, 0, 0, 0, 1, 0.5, 0.5, -0.5]], device=dev)
    depth = torch.full((1, 48, 64), 1.0, device=dev, requires_grad=True)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated(dev)
    live = [fusion_diff.integrate_tsdf(depth, f0, w0, poses, 1 / 16, 0.1, 8,
                                       [60.0, 60.0, 31.5, 23.5])[0] for _ in range(8)]
    # a result (16 KB), its weights, and the backward's workspace (37 KB)
    assert torch.cuda.memory_allocated(dev) - before <= 8 * (128 << 10)
    sum(t.sum() for t in live).backward()
    assert torch.isfinite(depth.grad).all()


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [0, 4, 8, 16])
@pytest.mark.parametrize("W", [64, 72, 70])
def test_unaligned_workspace(dev, W, offset):
    """Ray factors are written 16 bytes at a time only where rows and workspace
    allow it."""
    import ctypes

    import numpy as np
    import torch

    from marching_cube_amd.mesh import _ptr, _stream_handle
    from oracle import oracle as O
    from test_integrate_bricks_gpu import H0, random_depth, random_poses
    print(f"[case] workspace at {offset} bytes, frames {W} wide", flush=True)
    rng = np.random.default_rng(W + offset)
    dims, K, H = (70, 67, 61), 9, 40
    X, Y, Z = dims
    poses, depth = random_poses(rng, K, dims), random_depth(rng, K, H, W, True)
    intr = np.array([0.9 * W, 0.8 * W, 0.5 * W - 0.5, 0.45 * H], np.float32)
    ref = np.zeros((Z, Y, X), np.uint32)
    O.integrate_ex(ref, H0, 0.07, 0.05, 8, intr, poses, depth)
    lib = _capi.load()
    n = lib.mcx_integrate_workspace_size_frames(W, H, K)
    ws = torch.full((n + 4096,), 0x5a, dtype=torch.uint8, device=dev)
    vol = torch.zeros((Z, Y, X), dtype=torch.int32, device=dev)
    d_depth, d_poses = torch.from_numpy(depth).to(dev), torch.from_numpy(poses).to(dev)
    _capi.check(lib.mcx_integrate_ex(
        _ptr(vol), X, Y, Z, H0, 0.07, 0.05, 8, (ctypes.c_float * 4)(*intr), _ptr(d_poses),
        _ptr(d_depth), _capi.DEPTH_F32, 0.001, W, H, K, ctypes.c_void_p(ws.data_ptr() + offset), n,
        _stream_handle(dev)), "mcx_integrate_ex")
    assert vol.cpu().numpy().view(np.uint32).tobytes() == ref.tobytes()
    assert (ws[:offset] == 0x5a).all() and (ws[offset + n:] == 0x5a).all()
