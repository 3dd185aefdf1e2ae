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
