"""Rows of the chamfer loss without a vertex cost their zeros, whatever the
number of targets: 2 M rows, none or few of them vertices, with 1,024 targets
against one (the work is equal where none is; a target loop over idle rows
takes 25 times as long), and their gradients are zero."""
import pytest
import torch

from marching_cube_amd import _capi
from marching_cube_amd.mesh import _ptr, _stream_handle

pytestmark = pytest.mark.gpu


def time_us(f):
    best = float("inf")
    for _ in range(5):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        for _ in range(20):
            f()
        b.record()
        b.synchronize()
        best = min(best, a.elapsed_time(b) * 50)
    return best


@pytest.mark.parametrize("live", [0, 1, 700])
def test_idle_rows(dev, live):
    print(f"[case] chamfer, {live} of 2 M rows", flush=True)
    lib, cap = _capi.load(), 2_000_000
    pos = torch.rand((cap, 3), device=dev)
    vbase = torch.tensor([0, live // 2, live], device=dev)
    loss, g = torch.empty(2, device=dev), torch.ones((cap, 3), device=dev)
    ws = torch.empty(lib.mcx_chamfer_workspace_size(cap), dtype=torch.uint8, device=dev)
    us = {}
    for M in (1, 1024):
        t = torch.rand((2, M, 3), device=dev)

        def run():
            _capi.check(lib.mcx_chamfer_batched(_ptr(pos), _ptr(vbase), 2, _ptr(t), M, cap,
                                                _ptr(loss), _ptr(g), _ptr(ws), ws.numel(),
                                                _stream_handle(dev)), "mcx_chamfer_batched")
        run()
        assert (g[live:] == 0).all() and (g[:live] != 0).any(dim=1).all()
        if live == 0:
            us[M] = time_us(run)
    if live == 0:
        assert us[1024] <= 5 * us[1], us
