"""The workloads that this package is timed on, each one pass through its public entry points.

A case is a dict of plain values; ``prepare`` makes what a program has in hand before the call
(volumes, frames, plans, output buffers), ``run`` is the call, ``work`` says what the call cannot do
without and ``exact`` what it should return, in 64 bits, from plain torch.

Scenes are those of the benchmark: spheres and boxes seen by an orbiting 640x480 depth camera with
noise and dropout, fused into a packed volume over a 3 m cube; an fp32 field of Gaussian bumps; and
batches of small volumes holding one shape each.
"""
import json
import math
import os

import numpy as np
import torch

from marching_cube_amd import batch, diff, fusion, fusion_diff, mesh, synth, volio

DEVICE = "cuda"
EXTENT = 3.0  # metres covered by the largest side of a fused volume
TRUNC = 0.03
VGA = (640, 480, (525.0, 525.0, 319.5, 239.5))
QVGA = (320, 240, (262.5, 262.5, 159.5, 119.5))


def listed():
    return [
        # a preview mesh of a small volume, redone on every change: latency of one synchronous call
        dict(name="mesh_64", kind="mesh", X=64, Y=64, Z=64, frames=24),
        # the reference's export: every output of its run() and the normals, of a cropped volume
        dict(name="mesh_normals_ragged", kind="mesh", X=387, Y=250, Z=301, frames=100, normals=True),
        # the headline: vertex records of a volume already in memory, calls queued back to back
        dict(name="extract_512", kind="extract", X=512, Y=512, Z=512, frames=300),
        # thousands of uneven volumes (one object each) in one launch sequence
        dict(name="batch_3000", kind="batch", count=3000, lo=16, hi=128),
        # an indexed mesh for a viewer or a file
        dict(name="indexed_400", kind="indexed", X=400, Y=400, Z=400, frames=100),
        # mesh of an fp32 field and its gradient: one step of optimising the field
        dict(name="field_256", kind="field", X=256, Y=256, Z=256, bumps=64),
        # a scanner's loop: one frame into a full volume
        dict(name="frame_512", kind="frame", X=512, Y=512, Z=512, frames=8, depth="u16"),
        # a recording fused at once
        dict(name="fuse_512", kind="fuse", X=512, Y=512, Z=512, frames=300, depth="u16"),
        # the map a scanner aligns its next frame with
        dict(name="raycast_512", kind="raycast", X=512, Y=512, Z=512, frames=100),
        # one small differentiable fusion, forward and backward to every depth pixel
        dict(name="fuse_grad_96", kind="fuse_grad", X=96, Y=88, Z=104, frames=8),
        # a batch of differentiable fusions as one captured graph
        dict(name="fusion_graph_64", kind="graph", count=64, lo=64, hi=192, frames=16),
        # a volume written to its run-length form and read back, through host bytes
        dict(name="vol_512", kind="vol", X=512, Y=512, Z=512, frames=100),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mesh", "extract", "batch", "indexed", "field", "frame", "fuse", "raycast",
                       "fuse_grad", "graph", "vol"])
    c = dict(kind=kind)
    if kind == "batch":
        c.update(count=_log(rng, 8, 3000), lo=rng.randint(9, 24), hi=rng.randint(64, 128))
        return c
    if kind == "graph":
        c.update(count=_log(rng, 2, 64), lo=rng.randint(40, 90), hi=rng.randint(96, 192),
                 frames=rng.randint(2, 16))
        return c
    hi = {"field": 256, "fuse_grad": 160, "indexed": 400}.get(kind, 512)
    lo = 33 if kind in ("field", "fuse_grad") else 48
    c.update(X=_log(rng, lo, hi), Y=_log(rng, lo, hi), Z=_log(rng, lo, hi))
    if kind == "field":
        c.update(bumps=rng.randint(4, 64))
    elif kind == "fuse":
        c.update(frames=_log(rng, 2, 300), depth=rng.choice(["u16", "f32"]),
                 split=rng.random() < 0.3)
    elif kind == "frame":
        c.update(frames=8, depth=rng.choice(["u16", "f32"]), split=rng.random() < 0.3)
    elif kind == "fuse_grad":
        c.update(frames=rng.randint(1, 12))
    else:
        c.update(frames=rng.randint(20, 100))
    if kind == "mesh":
        c.update(normals=rng.random() < 0.5)
    return c


# ---- inputs ---------------------------------------------------------------------------------

def _orbit(case, n, seed):
    """Poses of a camera circling the middle of the case's volume."""
    poses = synth.orbit_poses(n, EXTENT, seed=seed)
    poses[:, 9:] += 0.5 * (_sides(case) - EXTENT)
    return poses.astype(np.float32)


def _sides(case):
    dims = np.array([case["X"], case["Y"], case["Z"]], np.float64)
    return EXTENT * dims / dims.max()


def _frames(case, seed, n):
    """(poses, uint16 frames) of n views of the benchmark's scene made from `seed`, its objects
    spread over the case's volume."""
    W, H, intr = VGA
    objs = synth.kinfu_scene(40, EXTENT, seed)
    objs[:, 1:4] *= (_sides(case) / EXTENT).astype(np.float32)
    poses = _orbit(case, n, seed)
    depth = fusion.synth_depth(intr, poses, objs, W, H, sigma=0.0015, dropout=0.02,
                               seed=seed & 0x7FFFFFFF, device=DEVICE)
    return torch.from_numpy(poses).to(DEVICE), depth


def _empty(case, split=False):
    dims = (case["X"], case["Y"], case["Z"])
    return fusion.voxel_new(dims, TRUNC, EXTENT / max(dims), device=DEVICE,
                            max_t=1.5 * TRUNC if split else None)


def _fused(case, seed):
    vox = _empty(case)
    poses, depth = _frames(case, seed, case["frames"])
    return fusion.integrate(vox, VGA[2], poses, depth, max_w=128)


def _field(case, seed):
    """fp32 field of Gaussian bumps and a little low-frequency noise (synth.bumps_volume, on the
    device and with three sides)."""
    rng = np.random.default_rng(seed)
    X, Y, Z, n = case["X"], case["Y"], case["Z"], max(case["X"], case["Y"], case["Z"])
    ax = [(torch.arange(m, device=DEVICE, dtype=torch.float32) + 0.5) / n for m in (Z, Y, X)]
    ext = np.array([Z, Y, X]) / n
    f = torch.full((Z, Y, X), 0.5, device=DEVICE)
    for _ in range(case["bumps"]):
        c, s, a = rng.uniform(0.2, 0.8, 3) * ext, rng.uniform(0.05, 0.12), rng.uniform(0.4, 1.0)
        g = [torch.exp(-(x - float(m)) ** 2 / float(2 * s * s)) for x, m in zip(ax, c)]
        f -= float(a) * g[0][:, None, None] * g[1][None, :, None] * g[2][None, None, :]
    for _ in range(4):
        k, ph = rng.integers(1, 6, 3), rng.uniform(0, 2 * math.pi)
        g = [torch.cos(2 * math.pi * int(m) * x) for x, m in zip(ax, k)]
        f += (0.02 / n) * torch.cos(2 * math.pi * int(k[0]) * ax[0] + float(ph))[:, None, None] \
            * g[1][None, :, None] * g[2][None, None, :]
    return f.contiguous(), 1.0 / n


def _small_fusion(n, K, seed):
    """Frames of three objects before a far wall, in float metres, with an orbiting camera."""
    W, H, intr = QVGA
    wall = np.array([[1, 0.5, 0.5, 0.5, 20.0, 20.0, 20.0, 0]], np.float32)
    objs = np.concatenate([synth.kinfu_scene(3, extent=1.0, seed=seed), wall])
    poses = synth.orbit_poses(K, extent=1.0, radius=1.6, seed=seed)
    d = fusion.synth_depth(intr, poses, objs, W, H, sigma=0.0015, dropout=0.02,
                           seed=seed & 0x7FFFFFFF, device=DEVICE)
    return torch.from_numpy(poses).to(DEVICE), (d.to(torch.float32) * 0.001).contiguous()


def _sphere_targets(M=64):
    i = np.arange(M) + 0.5
    phi, th = np.arccos(1 - 2 * i / M), np.pi * (1 + 5 ** 0.5) * i
    p = np.stack([np.cos(th) * np.sin(phi), np.sin(th) * np.sin(phi), np.cos(phi)], -1)
    return torch.from_numpy((0.5 + 0.25 * p).astype(np.float32)).to(DEVICE)


def _graph_inputs(case, seed):
    rng = np.random.default_rng(seed)
    shapes, hs, poses, depth = [], [], [], []
    for b in range(case["count"]):
        s = tuple(int(a) for a in rng.integers(case["lo"], case["hi"] + 1, 3))
        p, d = _small_fusion(max(s), case["frames"], int(rng.integers(1 << 30)))
        shapes.append(s)
        hs.append(1.0 / max(s))
        poses.append(p)
        depth.append(d)
    return shapes, hs, poses, depth


# ---- what a program has in hand before the call --------------------------------------------

def _capacity(case):
    """Vertices that a program makes room for: more than any scene of these sizes has."""
    if case["kind"] == "batch":
        dims = synth.batch_dims(case["count"], case["lo"], case["hi"], seed=1)
        return 4096 + int(case["count"] * 16 * np.mean(np.prod(dims, axis=1) ** (2 / 3)) * 2.5)
    return 4096 + int(64 * (case["X"] * case["Y"] * case["Z"]) ** (2 / 3))


def _rows(n, width, dtype=torch.int32):
    """A caller's buffer; rows that a call does not fill stay 0."""
    return torch.zeros((n, width), dtype=dtype, device=DEVICE)


def prepare(case, seed):
    kind, s = case["kind"], dict(case)
    if kind in ("mesh", "extract", "indexed", "raycast", "vol"):
        s["vox"] = vox = _fused(case, seed)
        X, Y, Z = vox.size
        n = _capacity(case)
        if kind in ("mesh", "extract"):
            s["vv"] = _rows(n, mesh.VV_WORDS)
        if kind == "mesh":
            s["mc"] = mesh.MarchingCubes(DEVICE)
            s["map"] = _rows(n, 3)
            s["ver_voxel"] = torch.empty((Z, Y, X), dtype=torch.int16, device=DEVICE)
            s["n"] = _rows(n, 3, torch.float32) if case.get("normals") else None
        elif kind == "indexed":
            s["vertices"], s["faces"] = _rows(n // 3, 3, torch.float32), _rows(n // 3, 3)
        elif kind == "vol":
            s["file"] = np.zeros(min(6 * X * Y * Z, int(400 * (X * Y * Z) ** (2 / 3))) + 4 * Z, np.uint8)
        elif kind == "extract":
            s["ws"] = mesh.Workspace(DEVICE)
            s["n"] = torch.zeros(1, dtype=torch.int64, device=DEVICE)
        elif kind == "raycast":
            W, H, _ = VGA
            s["pose"] = _orbit(case, 5, seed + 1)[seed % 5]
            s["depth"] = torch.empty((H, W), dtype=torch.float32, device=DEVICE)
            s["normals"] = torch.empty((H, W, 3), dtype=torch.float32, device=DEVICE)
    elif kind == "batch":
        vols, hs = synth.batch_shapes(case["count"], case["lo"], case["hi"], seed=seed,
                                      device=DEVICE)
        s["plan"] = plan = batch.BatchPlan(vols, hs)
        plan.workspace()
        s["vv"] = _rows(_capacity(case), mesh.VV_WORDS)
        s["vbase"] = torch.empty(len(vols) + 1, dtype=torch.int64, device=DEVICE)
    elif kind == "field":
        f, s["h"] = _field(case, seed)
        s["field"] = f.requires_grad_()
        s["extractor"] = diff.DiffExtractor(f.shape, f.device, cap=_capacity(case))
        s["extractor"].pos.zero_()
    elif kind in ("frame", "fuse"):
        s["vox"] = _empty(case, case.get("split", False))
        s["poses"], d = _frames(case, seed, case["frames"])
        s["frames"] = d if case["depth"] == "u16" else d.to(torch.float32)
        s["next"] = 0
        if kind == "frame":  # the volume already holds the frames once
            fusion.integrate(s["vox"], VGA[2], s["poses"], s["frames"])
    elif kind == "fuse_grad":
        shape = (case["Z"], case["Y"], case["X"])
        s["h"] = 1.0 / max(shape)
        s["poses"], d = _small_fusion(max(shape), case["frames"], seed)
        s["depth"] = d.requires_grad_()
        s["pos"] = _rows(_capacity(case), 3, torch.float32)
        s["tsdf0"], s["w0"] = fusion_diff.tsdf_init(shape, DEVICE, -1.0)
    elif kind == "graph":
        shapes, hs, poses, depth = _graph_inputs(case, seed)
        g = fusion_diff.FusionGraph(shapes, hs, depth, poses, [_sphere_targets()] * len(shapes),
                                    QVGA[2], trunc=TRUNC)
        g.capture()
        s["graph"] = g
    return s


def run(s):
    kind = s["kind"]
    if kind == "mesh":
        vox = s["vox"]
        tri, buf, vmap, ver = s["mc"].run(vox, s["vv"], s["map"], s["ver_voxel"])
        out = {"triangles": buf, "map": vmap, "ver_voxel": ver}
        if s.get("normals"):
            s["n"][:len(tri)] = mesh.normals(vox.data, vox.grid_s, tri)
            out["normals"] = s["n"]
        return out
    if kind == "extract":
        vox = s["vox"]
        mesh.extract_into(vox.data, vox.grid_s, vv=s["vv"], d_count=s["n"], workspace=s["ws"],
                          sync=False)
        return {"triangles": s["vv"], "count": s["n"]}
    if kind == "batch":
        s["plan"].extract_into(vv=s["vv"], vbase=s["vbase"], sync=False)
        return {"triangles": s["vv"], "ranges": s["vbase"]}
    if kind == "indexed":
        vertices, faces = mesh.indexed_mesh(s["vox"].data, s["vox"].grid_s)
        s["vertices"][:len(vertices)] = vertices  # into the viewer's buffers
        s["faces"][:len(faces)] = faces
        return {"vertices": s["vertices"], "faces": s["faces"]}
    if kind == "field":
        pos = diff.extract_positions(s["field"], s["h"], s["extractor"])
        (grad,) = torch.autograd.grad(pos, s["field"], pos.detach() - 0.5)
        return {"pos": s["extractor"].pos, "grad": grad}
    if kind == "frame":
        i, s["next"] = s["next"], (s["next"] + 1) % s["frames"].shape[0]
        return fusion.integrate(s["vox"], VGA[2], s["poses"][i:i + 1], s["frames"][i:i + 1]).data
    if kind == "fuse":
        fusion.voxel_init(s["vox"].data)
        return fusion.integrate(s["vox"], VGA[2], s["poses"], s["frames"]).data
    if kind == "raycast":
        W, H, intr = VGA
        d, n = fusion.raycast(s["vox"], intr, s["pose"], W, H, depth=s["depth"],
                              normals=s["normals"])
        return {"depth": d, "normals": n}
    if kind == "fuse_grad":
        tsdf, w = fusion_diff.integrate_tsdf(s["depth"], s["tsdf0"], s["w0"], s["poses"], s["h"],
                                             TRUNC, 128, QVGA[2])
        pos = diff.extract_positions(tsdf, s["h"])
        (grad,) = torch.autograd.grad(pos, s["depth"], pos.detach() - 0.5)
        s["pos"][:len(pos)] = pos.detach()
        return {"tsdf": tsdf.detach(), "weight": w, "pos": s["pos"], "grad": grad}
    if kind == "graph":
        g = s["graph"]
        g.replay()
        return {"loss": g.loss, "ranges": g.vbase, "grad": g.grad_depth_all}
    X, Y, Z = s["vox"].size  # vol
    dump = volio.encode(s["vox"].data)
    back = volio.decode(dump, X, Y, volio.slice_offsets(dump, Z), DEVICE)
    s["file"][:len(dump)] = np.frombuffer(dump, np.uint8)
    return {"dump": s["file"], "bytes": len(dump), "volume": back}


# ---- what a pass cannot do without ---------------------------------------------------------

def work(case):
    """Inputs read once and outputs written once; vertex counts are those these scenes typically
    have (they grow with the area of the sides).  An observation of a voxel by a frame is taken
    as 40 operations, an interpolated vertex as 20."""
    kind = case["kind"]
    if kind == "batch":
        lo, hi = case["lo"], case["hi"]
        vox = case["count"] * ((hi - lo) / math.log(hi / lo)) ** 3
        V = 0.07 * vox
        return dict(bytes=4 * vox + 28 * V, flops=20 * V)
    if kind == "graph":
        B, K, pix = case["count"], case["frames"], 320 * 240
        vox = B * ((case["lo"] + case["hi"]) / 2) ** 3
        V = 0.1 * vox
        # depth read and its gradient written; the volume is an intermediate result
        return dict(bytes=8 * B * K * pix, flops=80 * vox * K + (20 + 8 * 64) * V)
    X, Y, Z = case["X"], case["Y"], case["Z"]
    vox, area, K = X * Y * Z, (X * Y * Z) ** (2 / 3), case.get("frames", 0)
    V = 16 * area
    if kind == "mesh":
        b = 4 * vox + (28 + 12) * V + 2 * vox + (12 * V if case.get("normals") else 0)
        return dict(bytes=b, flops=20 * V * (4 if case.get("normals") else 1))
    if kind == "extract":
        return dict(bytes=4 * vox + 28 * V, flops=20 * V)
    if kind == "indexed":
        return dict(bytes=4 * vox + 4 * V + 12 * V / 6, flops=20 * V)
    if kind == "field":
        V = 20 * area
        return dict(bytes=8 * vox + 24 * V, flops=60 * V)
    pixel = 2 if case.get("depth") == "u16" else 4
    if kind == "frame":
        return dict(bytes=8 * vox * 0.5 + 640 * 480 * pixel, flops=40 * vox)
    if kind == "fuse":
        return dict(bytes=4 * vox + K * 640 * 480 * pixel, flops=40 * vox * K)
    if kind == "raycast":
        return dict(bytes=16 * 640 * 480 + 4 * 16 * area, flops=640 * 480 * 60 * area ** 0.5)
    if kind == "fuse_grad":
        return dict(bytes=8 * K * 320 * 240 + 16 * vox + 12 * V, flops=80 * vox * K)
    return dict(bytes=2 * (4 * vox + 8 * 16 * area), flops=8 * vox)  # vol


# ---- the same in 64 bits -------------------------------------------------------------------

_CORNER = np.array([[0, 0, 0], [1, 0, 0], [1, 1, 0], [0, 1, 0],
                    [0, 0, 1], [1, 0, 1], [1, 1, 1], [0, 1, 1]])  # x, y, z
_EDGE = np.array([[0, 1], [1, 2], [2, 3], [3, 0], [4, 5], [5, 6], [6, 7], [7, 4],
                  [0, 4], [1, 5], [2, 6], [3, 7]])


def _tables():
    """Triangle table with each triangle's vertices in output order (reversed), -1 padded."""
    with open(os.path.join("tests", "golden", "mc_tables.json")) as f:
        t = np.array(json.load(f)["triTable"])[:, :15].reshape(256, 5, 3)[:, :, ::-1]
    return torch.from_numpy(t.reshape(256, 15).copy()).to(DEVICE)


def _march(f, h, solid=None):
    """(positions, lower corner * 3 + axis of each vertex's edge) of the iso-0 surface of a
    float64 field, differentiable; cubes with a corner outside `solid` have no triangles."""
    Z, Y, X = f.shape
    ci = torch.zeros((Z - 1, Y - 1, X - 1), dtype=torch.int64, device=f.device)
    ok = torch.ones_like(ci, dtype=torch.bool)
    for k, (x, y, z) in enumerate(_CORNER):
        cut = (slice(z, z + Z - 1), slice(y, y + Y - 1), slice(x, x + X - 1))
        ci += (f.detach()[cut] < 0).to(torch.int64) << k
        if solid is not None:
            ok &= solid[cut]
    tri = _tables()
    cubes = torch.nonzero(ok & (ci > 0) & (ci < 255))
    rows = tri[ci[cubes[:, 0], cubes[:, 1], cubes[:, 2]]]
    at, slot = torch.nonzero(rows >= 0, as_tuple=True)
    ends = torch.from_numpy(_EDGE).to(f.device)[rows[at, slot]]
    corner = torch.from_numpy(_CORNER).to(f.device)
    base = cubes[at].flip(1)  # x, y, z
    a, b = base + corner[ends[:, 0]], base + corner[ends[:, 1]]
    flat = f.reshape(-1)
    ia, ib = ((p[:, 2] * Y + p[:, 1]) * X + p[:, 0] for p in (a, b))
    fa, fb = flat[ia], flat[ib]
    t = (-fa / (fb - fa + 1e-15)).unsqueeze(1)
    pa, pb = (a.double() + 0.5) * h, (b.double() + 0.5) * h
    return pa + t * (pb - pa), torch.minimum(ia, ib) * 3 + (a != b).to(torch.int64).argmax(1)


def _unpacked(vol):
    """(tsdf / 32766, weight > 0) of a packed volume."""
    t = ((vol & 0xFFFF) ^ 0x8000) - 0x8000
    return t.double() / 32766.0, (vol >> 16) != 0, t.abs() == 32766


def _cell(v, X, Y):
    return (v[:, 2] * Y + v[:, 1]) * X + v[:, 0]


def _gradient(f, flat_bad, c, t):
    """Differences of bilinear interpolations over opposite faces of the cells at c, at t."""
    Z, Y, X = f.shape
    base, flat = _cell(c, X, Y), f.reshape(-1)
    v = torch.stack([torch.stack([torch.stack([flat[base + (z * Y + y) * X + x] for x in (0, 1)])
                                  for y in (0, 1)]) for z in (0, 1)])  # z, y, x
    bad = sum(flat_bad[base + (z * Y + y) * X + x].int() for z in (0, 1) for y in (0, 1)
              for x in (0, 1)) > 0
    wx, wy, wz = ((1 - t[:, d], t[:, d]) for d in range(3))
    g = []
    for d in range(3):
        s = 0
        for z in (0, 1):
            for y in (0, 1):
                for x in (0, 1):
                    w = [wx[x], wy[y], wz[z]]
                    w[d] = (-1.0, 1.0)[(x, y, z)[d]]
                    s = s + v[z, y, x] * w[0] * w[1] * w[2]
        g.append(s)
    n = torch.stack(g, 1)
    norm = n.norm(dim=1, keepdim=True)
    n = torch.where(norm > np.finfo(np.float32).eps, n / norm, n)
    return torch.where(bad.unsqueeze(1), torch.zeros_like(n), n)


def _exact_normals(vol, h):
    f, solid, flat = _unpacked(vol)
    pos, _ = _march(f, h, solid)
    p = pos / h
    c = p.floor().to(torch.int64)
    size = torch.tensor(f.shape[::-1], device=f.device)
    inside = ((c >= 0) & (c + 1 < size)).all(1)
    c = torch.where(inside.unsqueeze(1), c, torch.zeros_like(c))
    n = _gradient(f, flat.reshape(-1), c, p - c)
    return torch.where(inside.unsqueeze(1), n, torch.zeros_like(n))


def _exact_indexed(vol, h):
    f, solid, _ = _unpacked(vol)
    pos, key = _march(f, h, solid)
    k, order = torch.sort(key, stable=True)
    first = torch.ones_like(k, dtype=torch.bool)
    first[1:] = k[1:] != k[:-1]
    return pos[torch.sort(order[first]).values]


def _pixels(axes, pose, camera, h):
    """Nearest pixels (u, v) of the voxel centres and whether they lie in the window, decided in 32
    bits with fused multiply-adds (a product is exact in 64)."""
    W, H, intr = camera
    fx, fy, cx, cy = (torch.tensor(a, dtype=torch.float32, device=pose.device) for a in intr)

    def fma(a, b, c):
        return (a.double() * b.double() + c.double()).float()

    z, y, x = torch.meshgrid(*((a.float() + 0.5) * np.float32(h) for a in axes), indexing="ij")
    d = [x - pose[9], y - pose[10], z - pose[11]]
    q = [fma(pose[6 + i], d[2], fma(pose[3 + i], d[1], pose[i] * d[0])) for i in range(3)]
    seen = q[2] > 1e-30
    qz = torch.where(seen, q[2], torch.ones_like(q[2]))
    u, v = torch.round(fma(fx, q[0] / qz, cx)), torch.round(fma(fy, q[1] / qz, cy))
    seen &= (u >= 0) & (v >= 0) & (u < W - 2) & (v < H - 2)
    zero = torch.zeros_like(u)
    return torch.where(seen, u, zero).double(), torch.where(seen, v, zero).double(), seen


def _observed(tsdf, w, poses, depth, h, trunc, max_w, camera):
    """Running average of the truncated ray-distance observations, in float64."""
    W, H, (fx, fy, cx, cy) = camera
    Z, Y, X = tsdf.shape
    axes = [torch.arange(m, device=tsdf.device, dtype=torch.float64) for m in (Z, Y, X)]
    pz, py, px = torch.meshgrid(*((a + 0.5) * h for a in axes), indexing="ij")
    f, w = tsdf.double(), w.double()
    for k in range(poses.shape[0]):
        P = [float(a) for a in poses[k].double()]
        d = [px - P[9], py - P[10], pz - P[11]]
        q = [P[i] * d[0] + P[3 + i] * d[1] + P[6 + i] * d[2] for i in range(3)]
        u, v, seen = _pixels(axes, poses[k], camera, h)
        fac = (((u - cx) / fx) ** 2 + ((v - cy) / fy) ** 2 + 1).sqrt()
        z = depth[k].reshape(-1)[(v * W + u).to(torch.int64)] * fac
        sdf = z - (q[0] ** 2 + q[1] ** 2 + q[2] ** 2).sqrt()
        seen = seen & (z > 0) & (sdf >= -trunc)
        f = torch.where(seen, (f * w + (sdf / trunc).clamp(-1, 1)) / (w + 1), f)
        w = torch.where(seen, (w + 1).clamp(max=max_w), w)
    return f


def _exact_raycast(vol, h, intr, pose, W, H, origin=0.5):
    f, _, sat = _unpacked(vol)
    Z, Y, X = f.shape
    flat, sat = f.reshape(-1), sat.reshape(-1)
    P = torch.tensor(np.asarray(pose, np.float64), device=f.device)
    R, c = P[:9].view(3, 3), P[9:] / h - origin
    v, u = torch.meshgrid(*(torch.arange(m, device=f.device, dtype=torch.float64)
                            for m in (H, W)), indexing="ij")
    ray = torch.stack([(u - intr[2]) / intr[0], (v - intr[3]) / intr[1], torch.ones_like(u)], -1)
    ray = ray.view(-1, 3)
    scale = ray.norm(dim=1)
    r = (ray / scale.unsqueeze(1)) @ R.T
    hi = torch.tensor([X - 1.0, Y - 1.0, Z - 1.0], device=f.device, dtype=torch.float64)
    t0 = torch.full_like(scale, math.inf)
    t1 = torch.zeros_like(scale)
    for a in range(3):
        o = [i for i in range(3) if i != a]
        for side in (1.0, float(hi[a])):
            t = (side - c[a]) / r[:, a]
            p = r * t.unsqueeze(1) + c
            ok = (t > 0) & ((p[:, o] > 1) & (p[:, o] < hi[o])).all(1)
            t0, t1 = torch.where(ok & (t < t0), t, t0), torch.where(ok & (t > t1), t, t1)
    t0 = torch.where(t0 == t1, torch.ones_like(t0), t0)
    depth, normal = torch.zeros_like(scale), torch.zeros_like(r)
    ids = torch.nonzero(t0 < t1).view(-1)
    t, end = t0[ids], t1[ids]
    dt, last, last_sdf = torch.ones_like(t), torch.zeros_like(t), torch.ones_like(t)
    fine = torch.zeros_like(t, dtype=torch.bool)
    while ids.numel():
        rr = r[ids]
        p = rr * t.unsqueeze(1) + c
        inside = ((p >= 0) & (p < hi)).all(1)
        cell = torch.where(inside.unsqueeze(1), p, torch.zeros_like(p)).floor().to(torch.int64)
        w, base = p - cell, _cell(cell, X, Y)
        sdf, stop = torch.zeros_like(t), torch.zeros_like(t)
        for x, y, z in ((0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (0, 1, 1),
                        (1, 1, 0), (1, 1, 1)):
            at = base + (z * Y + y) * X + x
            val = flat[at]
            stop = torch.where((stop == 0) & sat[at], val, stop)
            sdf += val * (w[:, 0] if x else 1 - w[:, 0]) * (w[:, 1] if y else 1 - w[:, 1]) \
                * (w[:, 2] if z else 1 - w[:, 2])
        sdf = torch.where(stop != 0, stop, sdf)
        hit = inside & (sdf < 0) & (sdf > -1) & (last_sdf >= 0) & (last_sdf < 1)
        back = inside & ~hit & (last_sdf <= 0) & (last_sdf > -1) & (sdf >= 0) & (sdf < 1)
        if hit.any():
            at = last[hit] - dt[hit] * last_sdf[hit] / (sdf[hit] - last_sdf[hit])
            depth[ids[hit]] = at.abs() / scale[ids[hit]] * h
            q = rr[hit] * at.unsqueeze(1) + c
            k = torch.minimum(q.floor().clamp(min=0), hi - 1).to(torch.int64)
            normal[ids[hit]] = _gradient(f, sat, k, q - k) @ R
        band = inside & (sdf > -1) & (sdf < 1)
        enter = band & ~fine
        keep = inside & ~enter
        leave = inside & ~band & fine
        last, last_sdf = torch.where(keep, t, last), torch.where(keep, sdf, last_sdf)
        t = torch.where(enter, t - dt, t)
        fine = (fine | enter) & ~leave
        dt = torch.where(enter, 0.25, torch.where(leave, 1.0, dt))
        t = t + dt
        go = ~hit & ~back & (t < end)
        ids, t, end, dt, last, last_sdf, fine = (a[go] for a in
                                                 (ids, t, end, dt, last, last_sdf, fine))
    return depth.view(H, W), normal.view(H, W, 3)


def _filled(rows, n):
    out = torch.zeros((n, 3), dtype=torch.float64, device=rows.device)
    out[:len(rows)] = rows.detach()
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "mesh" and case.get("normals"):
        vox = _fused(case, seed)
        return {"triangles": None, "map": None, "ver_voxel": None,
                "normals": _filled(_exact_normals(vox.data, float(np.float32(vox.grid_s))),
                                   _capacity(case))}
    if kind == "indexed":
        vox = _fused(case, seed)
        return {"vertices": _filled(_exact_indexed(vox.data, float(np.float32(vox.grid_s))),
                                    _capacity(case) // 3), "faces": None}
    if kind == "raycast":
        s = prepare(case, seed)
        W, H, intr = VGA
        d, n = _exact_raycast(s["vox"].data, float(np.float32(s["vox"].grid_s)), intr, s["pose"],
                              W, H)
        return {"depth": d, "normals": n}
    if kind == "field":
        f, h = _field(case, seed)
        f = f.double().requires_grad_()
        pos, _ = _march(f, float(np.float32(h)))
        (grad,) = torch.autograd.grad(pos, f, pos.detach() - 0.5)
        return {"pos": _filled(pos, _capacity(case)), "grad": grad}
    if kind == "fuse_grad":
        s = prepare(case, seed)
        d = s["depth"].detach().double().requires_grad_()
        h = float(np.float32(s["h"]))
        f = _observed(s["tsdf0"], s["w0"], s["poses"], d, h, TRUNC, 128, QVGA)
        pos, _ = _march(f, h)
        (grad,) = torch.autograd.grad(pos, d, pos.detach() - 0.5)
        return {"tsdf": f.detach(), "weight": None, "pos": _filled(pos, _capacity(case)),
                "grad": grad}
    if kind == "graph":
        shapes, hs, poses, depth = _graph_inputs(case, seed)
        targets, loss, grad = _sphere_targets().double(), [], []
        for shape, h, p, d in zip(shapes, hs, poses, depth):
            d, h = d.double().requires_grad_(), float(np.float32(h))
            t0 = torch.full(shape, -1.0, device=DEVICE)
            pos, _ = _march(_observed(t0, torch.zeros_like(t0), p, d, h, TRUNC, 128, QVGA), h)
            x = pos.detach()
            j = torch.cat([torch.cdist(y, targets).argmin(1) for y in x.split(65536)])
            e = pos - targets[j]
            each = e.square().sum()
            (g,) = torch.autograd.grad(each, d)
            loss.append(each.detach())
            grad.append(g)
        return {"loss": torch.stack(loss), "ranges": None, "grad": torch.stack(grad)}
    return None
