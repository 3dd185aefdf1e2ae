"""The fp32 volumes' 128-bit count against the oracle, where it can go wrong:
planes that end at, just past and just before a tile of 512 voxels, widths that
are no multiple of a lane's four voxels, rows longer than a tile, the smallest
volumes; signed zeros, denormals, infinities and NaN (only f < 0 is inside);
with the active-cube masks that the backward's gather reads in runs of 512 voxels,
and batched."""
import numpy as np
import pytest
import torch

from marching_cube_amd import batch, diff, mesh
from oracle import oracle as O

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (3, 17, 31), (5, 16, 32), (4, 27, 19), (4, 73, 7), (6, 5, 1030),
          (19, 23, 29), (9, 64, 66), (70, 8, 64)]


def noisy(shape, seed, specials=()):
    rng = np.random.default_rng(seed)
    f = (rng.uniform(0.25, 1.0, shape) * np.where(rng.random(shape) < 0.2, -1, 1))
    f = f.astype(np.float32)
    f[rng.random(shape) < 0.05] = -0.0
    f[rng.random(shape) < 0.05] = 0.0
    for v in specials:
        f[rng.random(shape) < 0.04] = np.float32(v)
    return f


@pytest.mark.parametrize("shape", SHAPES)
def test_positions_and_gradient(dev, shape):
    print(f"[case] fp32 count {shape}", flush=True)
    f, h = noisy(shape, sum(shape)), 0.01
    ref = O.extract(f, h, want=("pos",))
    v = torch.from_numpy(f).to(dev)
    assert mesh.extract(v, h, want=("pos",)).pos.cpu().numpy().tobytes() == ref["pos"].tobytes()
    if not ref["n"]:
        return
    v.requires_grad_(True)
    p = diff.extract_positions(v, h)
    assert p.detach().cpu().numpy().tobytes() == ref["pos"].tobytes()
    g = np.random.default_rng(1).standard_normal(ref["pos"].shape)
    p.backward(torch.from_numpy(g.astype(np.float32)).to(dev))
    want = O.extract_backward_f64(f, h, g.astype(np.float32).astype(np.float64))
    got = v.grad.cpu().numpy().astype(np.float64)
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
    assert (got[want == 0] == 0).all()


@pytest.mark.parametrize("specials", [(1e-40, -1e-40), (np.inf, -np.inf), (np.nan, -1e-45)])
def test_special_values(dev, specials):
    print(f"[case] fp32 count with {specials}", flush=True)
    f, h = noisy((6, 21, 27), 5, specials), 0.01
    with np.errstate(all="ignore"):
        ref = O.extract(f, h, want=("pos",))
    r = mesh.extract(torch.from_numpy(f).to(dev), h, want=("pos",))
    assert r.count == ref["n"] > 0
    # a fraction of inf / inf or NaN: the oracle makes all three coordinates NaN,
    # the emit kernel only the one along the edge
    ok = ~np.isnan(ref["pos"])
    assert np.array_equal(r.pos.cpu().numpy()[ok], ref["pos"][ok])


def test_batched(dev):
    print("[case] fp32 count, a batch of all shapes", flush=True)
    fs = [noisy(s, 7 + k) for k, s in enumerate(SHAPES)]
    plan = batch.BatchPlan([torch.from_numpy(f).to(dev) for f in fs], [0.01] * len(fs))
    n, vbase, out = plan.extract(want=("pos",))
    vb, pos = vbase.cpu().numpy(), out["pos"].cpu().numpy()
    for k, f in enumerate(fs):
        ref = O.extract(f, 0.01, want=("pos",))["pos"]
        assert pos[vb[k]:vb[k + 1]].tobytes() == ref.tobytes(), SHAPES[k]


@pytest.mark.parametrize("recompute", [False, True])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 16, 65])
def test_units_of_the_backward(dev, n, recompute):
    """n voxels inside, apart from one another: 8 n records, units of 64."""
    print(f"[case] backward units, {8 * n} records, recompute {recompute}", flush=True)
    f = np.full((14, 41, 50), 0.5, np.float32)
    rng = np.random.default_rng(n)
    spots = np.stack(np.meshgrid(range(1, 13, 3), range(1, 40, 3), range(1, 49, 3),
                                 indexing="ij"), -1).reshape(-1, 3)
    for z, y, x in spots[np.sort(rng.choice(len(spots), n, replace=False))]:
        f[z, y, x] = -rng.uniform(0.25, 1.0)
    h = 0.02
    ref = O.extract(f, h, want=("pos",))
    v = torch.from_numpy(f).to(dev).requires_grad_(True)
    ex = diff.DiffExtractor(f.shape, dev, recompute=recompute)
    p = diff.extract_positions(v, h, extractor=ex)
    assert p.detach().cpu().numpy().tobytes() == ref["pos"].tobytes()
    g = np.random.default_rng(1).standard_normal(ref["pos"].shape).astype(np.float32)
    p.backward(torch.from_numpy(g).to(dev))
    want = O.extract_backward_f64(f, h, g.astype(np.float64))
    got = v.grad.cpu().numpy().astype(np.float64)
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
    assert (got[want == 0] == 0).all()
