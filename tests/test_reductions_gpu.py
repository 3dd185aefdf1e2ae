"""The chamfer loss's rows and sums against plain torch where they can go wrong:
workgroups (512 rows) that span volumes, empty volumes, rows past the total and
past the capacity, one to 1,024 targets, ties; bit-exact (the sum's order is
restated)."""
import numpy as np
import pytest
import torch

from marching_cube_amd import _capi, mesh

pytestmark = pytest.mark.gpu


def fma(a, b, c):  # products of fp32 are exact in fp64; the sum rounds there, then to fp32
    return (a.astype(np.float64) * b + c.astype(np.float64)).astype(np.float32)


@pytest.mark.parametrize("counts,M,pad", [((1,), 1, 0), ((511, 0, 1, 700), 3, 5),
                                          ((512, 512), 64, 0), ((0, 5000, 3, 0), 1024, 300),
                                          ((40, 2100), 7, -600)])
def test_chamfer_rows_and_sums(dev, counts, M, pad):
    print(f"[case] chamfer {counts} x {M} targets", flush=True)
    rng = np.random.default_rng(M)
    total, nvol = sum(counts), len(counts)
    cap = total + pad
    vbase = np.concatenate([[0], np.cumsum(counts)]).astype(np.int64)
    # a coarse lattice: many ties, and sums of squares that are exact
    p = rng.integers(-8, 9, (max(total, cap), 3)).astype(np.float32) / 8
    t = rng.integers(-8, 9, (nvol, M, 3)).astype(np.float32) / 8
    d = {k: torch.from_numpy(v).to(dev) for k, v in (("p", p), ("t", t), ("vb", vbase))}
    loss = torch.full((nvol,), -1.0, device=dev)
    g = torch.full((cap, 3), np.nan, device=dev)
    lib = _capi.load()
    ws = torch.empty(lib.mcx_chamfer_workspace_size(cap), dtype=torch.uint8, device=dev)
    _capi.check(lib.mcx_chamfer_batched(mesh._ptr(d["p"]), mesh._ptr(d["vb"]), nvol,
                                        mesh._ptr(d["t"]), M, cap, mesh._ptr(loss), mesh._ptr(g),
                                        mesh._ptr(ws), ws.numel(), mesh._stream_handle(dev)),
                "mcx_chamfer_batched")
    want = np.zeros((cap, 3), np.float32)
    for b in range(nvol):
        lo, hi = vbase[b], min(vbase[b + 1], cap)
        q = p[lo:hi]
        e = q[:, None, :] - t[b][None]
        d2 = fma(e[..., 2], e[..., 2], fma(e[..., 1], e[..., 1], e[..., 0] * e[..., 0]))
        j = d2.argmin(1) if len(q) else np.zeros(0, int)
        want[lo:hi] = 2 * (q - t[b][j])
        part = np.zeros(256, np.float32)  # thread k: rows k, k + 256, ... in order
        for i, x in enumerate(d2.min(1) if len(q) else ()):
            part[i % 256] += x
        w = 128
        while w:
            part[:w] += part[w:2 * w]
            w //= 2
        assert loss[b].item() == part[0]
    assert g.cpu().numpy().tobytes() == want.tobytes()
