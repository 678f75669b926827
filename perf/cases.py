"""Timed cases of cubvh_amd: what its users call, from a few queries to full grids.

Eight families, each over a range of sizes (``listed`` holds its usual points, ``draw``
takes others):

  udf       cuBVH.unsigned_distance: a handful of probe points, a surface sample, a grid
  train     cubvh_amd.udf forward and backward: gradients of a distance loss to the query
            points and to the mesh's vertices
  sdf       cuBVH.signed_distance, watertight (grids for a network's targets) or raystab
            (meshes with holes)
  rays      cuBVH.ray_trace: scattered probe rays, or pinhole cameras in pixel order
  forest    cubvh_amd.udf_batched: a minibatch of meshes, forward and backward
  flood     floodfill of a voxelized shell (inside / outside labels)
  voxels    cuHashTable: a sparse voxel set built and searched
  cells     sparse_marching_cubes over the cut cells of a lattice

Meshes are subdivided icospheres (20 * 4^level faces) with a smooth radial perturbation,
or jittered vertices, or a smooth sphere with holes and loose triangles (a soup).
"""
from __future__ import annotations

import math

import numpy as np
import torch

import cubvh_amd

DEVICE = "cuda"
_UNIT: dict = {}


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # an interactive tool probing one small mesh with a few points: latency
        {"name": "udf_few", "family": "udf", "mesh": "smooth", "level": 4, "points": "normal", "n": 777, "uvw": True},
        # a surface-near sample for one evaluation step
        {"name": "udf_sample", "family": "udf", "mesh": "jitter", "level": 6, "points": "normal", "n": 50_003,
         "uvw": False},
        # a dense distance field for one large mesh
        {"name": "udf_grid256", "family": "udf", "mesh": "smooth", "level": 8, "points": "grid", "n": 256 ** 3,
         "uvw": False},
        # one optimization step on points and vertices
        {"name": "train_points", "family": "train", "mesh": "jitter", "level": 6, "n": 1 << 20},
        # signed targets on a grid
        {"name": "sdf_grid128", "family": "sdf", "mode": "watertight", "mesh": "smooth", "level": 7, "points": "grid",
         "n": 128 ** 3},
        # signs for a mesh that is not closed
        {"name": "sdf_soup", "family": "sdf", "mode": "raystab", "mesh": "soup", "level": 7, "points": "uniform",
         "n": 600_011},
        # picking: a few scattered rays
        {"name": "rays_few", "family": "rays", "mesh": "jitter", "level": 6, "kind": "scatter", "n": 1_501},
        # four rendered views
        {"name": "rays_camera", "family": "rays", "mesh": "soup", "level": 8, "kind": "camera", "width": 1920,
         "height": 1080, "views": 4},
        # a minibatch of meshes of mixed size, distances with gradients to all vertices
        {"name": "forest_train", "family": "forest", "meshes": 48, "min_level": 3, "max_level": 6, "min_n": 4_096,
         "max_n": 65_536},
        # inside / outside labels of a voxelized surface
        {"name": "flood_256", "family": "flood", "batch": 1, "h": 256, "w": 256, "d": 256, "noise": 0.0},
        # sparse voxels: build the table, then a search of random order, half of it absent
        {"name": "voxels_random", "family": "voxels", "res": 1024, "samples": 1 << 22, "pattern": "random",
         "m": 1 << 23},
        # surface extraction from the cut cells of a lattice
        {"name": "cells_512", "family": "cells", "res": 512, "average": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["udf", "udf", "train", "sdf", "rays", "forest", "flood", "voxels", "cells"])
    if family == "udf":
        return {"family": family, "mesh": rng.choice(["smooth", "jitter"]), "level": rng.randint(4, 8),
                "points": rng.choice(["normal", "uniform"]), "n": _log(rng, 300, 2_000_000), "uvw": rng.random() < 0.5}
    if family == "train":
        return {"family": family, "mesh": "jitter", "level": rng.randint(4, 6), "n": _log(rng, 2_000, 1 << 20)}
    if family == "sdf":
        if rng.random() < 0.5:
            return {"family": family, "mode": "watertight", "mesh": "smooth", "level": rng.randint(5, 8),
                    "points": "uniform", "n": _log(rng, 2_000, 128 ** 3)}
        return {"family": family, "mode": "raystab", "mesh": "soup", "level": rng.randint(5, 7), "points": "uniform",
                "n": _log(rng, 500, 600_000)}
    if family == "rays":
        if rng.random() < 0.5:
            return {"family": family, "mesh": rng.choice(["smooth", "jitter"]), "level": rng.randint(4, 8),
                    "kind": "scatter", "n": _log(rng, 300, 1_000_000)}
        return {"family": family, "mesh": rng.choice(["smooth", "soup"]), "level": rng.randint(6, 8), "kind": "camera",
                "width": rng.randint(200, 1920), "height": rng.randint(200, 1080), "views": rng.randint(1, 4)}
    if family == "forest":
        return {"family": family, "meshes": _log(rng, 4, 48), "min_level": 3, "max_level": rng.randint(4, 6),
                "min_n": 1_000, "max_n": _log(rng, 4_000, 65_536)}
    if family == "flood":
        return {"family": family, "batch": rng.randint(1, 2), "h": _log(rng, 24, 200), "w": _log(rng, 24, 200),
                "d": _log(rng, 24, 200), "noise": rng.choice([0.0, 0.0, 0.3])}
    if family == "voxels":
        return {"family": family, "res": rng.choice([256, 512, 1024]), "samples": _log(rng, 1 << 14, 1 << 22),
                "pattern": rng.choice(["random", "neighbours"]), "m": _log(rng, 1 << 14, 1 << 23)}
    return {"family": family, "res": rng.randint(40, 512), "average": rng.random() < 0.4}


# ------------------------------------------------------------------ inputs
def _unit_sphere(level):
    """Unit icosphere of 20 * 4^level faces: vertices float64 [V, 3], faces int64 [F, 3]."""
    if level in _UNIT:
        return _UNIT[level]
    if level == 0:
        t = (1.0 + math.sqrt(5.0)) / 2.0
        v = np.array([(s * a, u * b, 0.0) for a, b in ((1.0, t),) for s in (-1, 1) for u in (-1, 1)])
        v = np.concatenate([v, v[:, [2, 0, 1]], v[:, [1, 2, 0]]])
        # faces: triples of vertices at the edge length 2 from one another, wound outward
        near = np.abs(np.linalg.norm(v[:, None] - v[None], axis=2) - 2.0) < 1e-6
        f = []
        for i in range(12):
            for j in range(i + 1, 12):
                for k in range(j + 1, 12):
                    if near[i, j] and near[j, k] and near[i, k]:
                        out = np.dot(np.cross(v[j] - v[i], v[k] - v[i]), v[i]) > 0.0
                        f.append((i, j, k) if out else (i, k, j))
        _UNIT[0] = v / np.linalg.norm(v, axis=1, keepdims=True), np.array(f, dtype=np.int64)
        return _UNIT[0]
    v, f = _unit_sphere(level - 1)
    n = len(v)
    pairs = np.concatenate([f[:, [0, 1]], f[:, [1, 2]], f[:, [2, 0]]])
    lo, hi = pairs.min(axis=1), pairs.max(axis=1)
    edges, which = np.unique(lo * n + hi, return_inverse=True)
    mid = v[edges // n] + v[edges % n]
    mid /= np.linalg.norm(mid, axis=1, keepdims=True)
    m0, m1, m2 = which.reshape(3, -1) + n
    f = np.concatenate([np.stack(t, axis=1) for t in
                        ((f[:, 0], m0, m2), (f[:, 1], m1, m0), (f[:, 2], m2, m1), (m0, m1, m2))])
    _UNIT[level] = np.concatenate([v, mid]), f
    return _UNIT[level]


def _mesh(kind, level, seed, scale=1.0):
    rng = np.random.default_rng(seed)
    v, f = _unit_sphere(level)
    if kind == "jitter":
        return (0.5 * scale * v + rng.normal(0.0, 0.32 / 2 ** level, v.shape)).astype(np.float32), f.astype(np.int32)
    a, b = rng.integers(1, 5, 8), rng.integers(1, 5, 8)
    shift = rng.uniform(0.0, 2.0 * np.pi, 8)
    theta, phi = np.arccos(np.clip(v[:, 2], -1.0, 1.0)), np.arctan2(v[:, 1], v[:, 0])
    r = np.full(len(v), 0.5)
    for k in range(8):
        r += 0.05 * np.sin(a[k] * theta + b[k] * phi + shift[k])
    v = v * (scale * r)[:, None]
    if kind == "soup":  # a fifth of the faces gone, and loose triangles in and around the surface
        f = f[rng.random(len(f)) < 0.8]
        loose = len(f) // 6
        c = rng.uniform(-0.6, 0.6, (loose, 1, 3))
        size = 1.3 / 2 ** (level - 1)
        v = np.concatenate([v, (c + rng.normal(0.0, 0.5 * size, (loose, 3, 3))).reshape(-1, 3)])
        f = np.concatenate([f, len(v) - 3 * loose + np.arange(3 * loose).reshape(-1, 3)])
    return v.astype(np.float32), f.astype(np.int32)


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _points(kind, n, seed):
    gen = _generator(seed + 1)
    if kind == "grid":  # a cubic lattice over [-1, 1]^3, shifted within one step
        side = round(n ** (1.0 / 3.0))
        assert side ** 3 == n
        x = torch.linspace(-1.0, 1.0, side, device=DEVICE)
        g = torch.stack(torch.meshgrid(x, x, x, indexing="ij"), dim=-1).reshape(-1, 3)
        return (g + torch.rand(3, device=DEVICE, generator=gen) / side).contiguous()
    if kind == "uniform":
        return torch.rand(n, 3, device=DEVICE, generator=gen) * 2.0 - 1.0
    return torch.randn(n, 3, device=DEVICE, generator=gen) * 0.4


def _rays(case, seed):
    gen = _generator(seed + 2)
    if case["kind"] == "scatter":  # from a sphere around the mesh towards points in it
        o = torch.randn(case["n"], 3, device=DEVICE, generator=gen)
        o = 2.0 * o / o.norm(dim=1, keepdim=True)
        d = torch.rand(case["n"], 3, device=DEVICE, generator=gen) - 0.5 - o
        return o.contiguous(), (d / d.norm(dim=1, keepdim=True)).contiguous()
    w, h = case["width"], case["height"]
    tan = math.tan(math.radians(50.0) / 2.0)
    x = ((torch.arange(w, device=DEVICE) + 0.5) / w * 2.0 - 1.0) * tan * w / h
    y = (1.0 - (torch.arange(h, device=DEVICE) + 0.5) / h * 2.0) * tan
    origins, directions = [], []
    for _ in range(case["views"]):
        c = torch.randn(3, device=DEVICE, generator=gen)
        c = 2.0 * c / c.norm()
        fwd = -c / c.norm()
        right = torch.linalg.cross(fwd, torch.tensor([0.0, 0.0, 1.0], device=DEVICE))
        right = right / right.norm()
        up = torch.linalg.cross(right, fwd)
        d = fwd + x[None, :, None] * right + y[:, None, None] * up
        directions.append(d / d.norm(dim=-1, keepdim=True))
        origins.append(c.expand(h, w, 3))
    return torch.stack(origins).contiguous(), torch.stack(directions).contiguous()


def _forest_spec(case):
    """(level, points, scale) of every mesh of the batch."""
    rng = np.random.default_rng(case["meshes"])
    levels = rng.integers(case["min_level"], case["max_level"] + 1, case["meshes"])
    counts = np.exp(rng.uniform(math.log(case["min_n"]), math.log(case["max_n"]), case["meshes"])).astype(np.int64)
    scales = rng.uniform(0.3, 0.9, case["meshes"])
    return [(int(l), int(c), float(s)) for l, c, s in zip(levels, counts, scales)]


def _bumpy(x, y, z, seed):
    """A closed star-shaped surface as the zero set of a smooth function on [0, 1]^3."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(0.0, 2.0 * np.pi, 3)
    q = [8.0 * (t - 0.5) for t in (x, y, z)]
    bump = 0.03 * (torch.sin(q[0] * 2.0 + c[0]) + torch.sin(q[1] * 2.5 + c[1]) + torch.sin(q[2] * 3.0 + c[2]))
    return torch.sqrt((x - 0.5) ** 2 + (y - 0.5) ** 2 + (z - 0.5) ** 2) - 0.35 - bump


def _axes(*sizes):
    return torch.meshgrid(*[torch.linspace(0.0, 1.0, s, device=DEVICE) for s in sizes], indexing="ij")


def _voxels(case, seed):
    gen = _generator(seed + 3)
    res = case["res"]
    g = torch.randn(case["samples"], 3, device=DEVICE, generator=gen)
    v = ((g / g.norm(dim=1, keepdim=True) * 0.45 + 0.5) * res).floor().to(torch.int64).clamp_(0, res - 1)
    key = torch.unique((v[:, 0] * res + v[:, 1]) * res + v[:, 2])
    if case["pattern"] == "random":
        key = key[torch.randperm(key.numel(), device=DEVICE, generator=gen)]
    coords = torch.stack([key // (res * res), key // res % res, key % res], dim=1).to(torch.int32).contiguous()
    m = case["m"]
    if case["pattern"] == "neighbours":  # a sparse stencil: every voxel's neighbours in turn
        step = torch.randint(-1, 2, (m // coords.shape[0] + 1, 1, 3), device=DEVICE, generator=gen, dtype=torch.int32)
        return coords, (coords[None] + step).reshape(-1, 3)[:m].contiguous()
    stored = coords[torch.randint(0, coords.shape[0], (m - m // 2,), device=DEVICE, generator=gen)]
    other = torch.randint(0, res, (m // 2, 3), device=DEVICE, generator=gen, dtype=torch.int32)
    q = torch.cat([stored, other])
    return coords, q[torch.randperm(m, device=DEVICE, generator=gen)].contiguous()


_CORNERS = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]


def _cells(case, seed):
    n, gen = case["res"], _generator(seed + 4)
    # the cut cells are the shape's, the values at their corners the seed's
    f = _bumpy(*_axes(n, n, n), n) * (0.7 + 0.6 * torch.rand(n, n, n, device=DEVICE, generator=gen))
    neg = f < 0.0
    views = [neg[a:n - 1 + a, b:n - 1 + b, c:n - 1 + c] for a, b, c in _CORNERS]
    some, every = views[0].clone(), views[0].clone()
    for view in views[1:]:
        some |= view
        every &= view
    idx = torch.nonzero(some & ~every)
    corners = torch.stack([f[idx[:, 0] + a, idx[:, 1] + b, idx[:, 2] + c] for a, b, c in _CORNERS], dim=1)
    if case["average"]:  # every cell's own estimate of its corners, to be made consistent
        corners = corners * (0.9 + 0.2 * torch.rand(corners.shape, device=DEVICE, generator=gen))
    return idx.to(torch.int32).contiguous(), corners.contiguous()


def prepare(case, seed):
    family = case["family"]
    s = {"case": case}
    if family in ("udf", "sdf", "train", "rays"):
        v, f = _mesh(case["mesh"], case["level"], seed)
        s["bvh"] = cubvh_amd.cuBVH(v, f)
        if family == "rays":
            s["o"], s["d"] = _rays(case, seed)
        elif family == "train":
            s["p"] = _points("normal", case["n"], seed).requires_grad_()
            s["v"] = torch.from_numpy(v).to(DEVICE).requires_grad_()
        else:
            s["p"] = _points(case["points"], case["n"], seed)
    elif family == "forest":
        spec = _forest_spec(case)
        meshes = [_mesh("smooth", level, seed * 1000 + k, scale) for k, (level, _, scale) in enumerate(spec)]
        s["forest"] = cubvh_amd.cuBVHForest([cubvh_amd.cuBVH(*m) for m in meshes])
        s["v"] = s["forest"].concatenated_mesh(DEVICE)[0].requires_grad_()
        counts = [c for _, c, _ in spec]
        s["off"] = torch.tensor(np.concatenate([[0], np.cumsum(counts)]))  # on the host, as a collate makes it
        s["p"] = _points("uniform", sum(counts), seed).requires_grad_()
    elif family == "flood":
        dims = (case["h"], case["w"], case["d"])
        f = torch.stack([_bumpy(*_axes(*dims), seed + 17 * b) for b in range(case["batch"])])
        s["grid"] = f.abs() < 1.7 / min(dims)
        if case["noise"]:  # a noisy scan: stray occupied voxels
            s["grid"] |= torch.rand(f.shape, device=DEVICE, generator=_generator(seed + 5)) < case["noise"]
    elif family == "voxels":
        s["coords"], s["queries"] = _voxels(case, seed)
        s["table"] = cubvh_amd.cuHashTable()
    else:
        s["coords"], s["corners"] = _cells(case, seed)
    return s


def run(s):
    case = s["case"]
    family = case["family"]
    if family == "udf":
        d, face, uvw = s["bvh"].unsigned_distance(s["p"], return_uvw=case["uvw"])
        return (d, face, uvw) if case["uvw"] else (d, face)
    if family == "sdf":
        return s["bvh"].signed_distance(s["p"], mode=case["mode"])[:2]
    if family == "rays":
        return s["bvh"].ray_trace(s["o"], s["d"])
    if family == "train":
        d, face, uvw = cubvh_amd.udf(s["bvh"], s["p"], s["v"])
        return (d.detach(), *torch.autograd.grad((d * d).mean(), (s["p"], s["v"])))
    if family == "forest":
        d, face, uvw = cubvh_amd.udf_batched(s["forest"], s["p"], s["off"], s["v"])
        return (d.detach(), *torch.autograd.grad((d * d).mean(), (s["p"], s["v"])))
    if family == "flood":
        return cubvh_amd.floodfill(s["grid"])
    if family == "voxels":
        s["table"].build(s["coords"])
        return s["table"].search(s["queries"])
    return cubvh_amd.sparse_marching_cubes(s["coords"], s["corners"], 0.0, case["average"])


def work(case):
    """Bytes: the mesh's faces (9 floats each), every input and every output once.  Flops:
    the one face (or face and sign) a query's answer comes from."""
    family = case["family"]

    def faces(kind, level):
        return 20 * 4 ** level * (14 if kind == "soup" else 15) // 15

    if family in ("udf", "sdf"):
        out = 12 + (12 if case.get("uvw") else 0)
        return {"bytes": 36 * faces(case["mesh"], case["level"]) + (12 + out) * case["n"], "flops": 100 * case["n"]}
    if family == "train":
        f = faces(case["mesh"], case["level"])
        # points, distance, face and barycentrics; the gradients to points and vertices
        return {"bytes": 36 * f + (12 + 24 + 12 + 4) * case["n"] + 12 * (f // 2 + 2), "flops": 150 * case["n"]}
    if family == "rays":
        n = case["n"] if case["kind"] == "scatter" else case["width"] * case["height"] * case["views"]
        return {"bytes": 36 * faces(case["mesh"], case["level"]) + (24 + 24) * n, "flops": 60 * n}
    if family == "forest":
        mean_n = (case["max_n"] - case["min_n"]) / math.log(case["max_n"] / case["min_n"])
        levels = range(case["min_level"], case["max_level"] + 1)
        f = case["meshes"] * sum(20 * 4 ** l for l in levels) / len(levels)
        n = case["meshes"] * mean_n
        return {"bytes": int(36 * f + 52 * n + 6 * f), "flops": int(150 * n)}
    if family == "flood":
        n = case["batch"] * case["h"] * case["w"] * case["d"]
        return {"bytes": 5 * n, "flops": n}
    if family == "voxels":
        # distinct voxels of a sphere shell: about 1.5 per unit of its area
        n = min(case["samples"], int(1.5 * 4.0 * math.pi * (0.45 * case["res"]) ** 2))
        return {"bytes": 12 * n + 16 * case["m"], "flops": 10 * (n + case["m"])}
    # cut cells: about 1.9 per unit of the surface's area; a vertex and two triangles each
    n = int(1.9 * 4.0 * math.pi * (0.35 * case["res"]) ** 2)
    return {"bytes": 44 * n + 36 * n, "flops": 30 * n}


# ------------------------------------------------------------------ 64-bit answers
def _closest64(v, f, p):
    """Nearest point of the mesh for every p, over all faces: (distance, point, face)."""
    tri = v[f]  # [F, 3, 3]
    n, chunk = p.shape[0], max(1, (1 << 24) // f.shape[0])
    dist, face = p.new_empty(n), torch.empty(n, dtype=torch.int64, device=p.device)
    nor = torch.linalg.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0])
    nn = (nor * nor).sum(-1)

    def dot(a, b):
        return a[..., 0] * b[..., 0] + a[..., 1] * b[..., 1] + a[..., 2] * b[..., 2]

    def squared(pt, t, normal, n2):
        best, inside = None, None
        for k in range(3):
            a, e = t[..., k, :], t[..., (k + 1) % 3, :] - t[..., k, :]
            w, ee = pt - a, dot(e, e)
            s = (dot(w, e) / ee).clamp(0.0, 1.0)
            r = w - s[..., None] * e
            q = dot(r, r)
            best = q if best is None else torch.minimum(best, q)
            side = dot(torch.linalg.cross(normal.expand_as(e), e), w) >= 0.0
            inside = side if inside is None else inside & side
        h = dot(pt - t[..., 0, :], normal)
        return torch.where(inside, h * h / n2, best)

    for i in range(0, n, chunk):
        q = squared(p[i:i + chunk, None], tri[None], nor[None], nn[None])
        m = q.min(dim=1)
        dist[i:i + chunk], face[i:i + chunk] = m.values.sqrt(), m.indices
    return dist, face


def _foot64(tri, p):
    """Barycentric weights of the point of each triangle [n, 3, 3] closest to p [n, 3]."""
    a, b, c = tri.unbind(1)
    ab, ac, ap = b - a, c - a, p - a
    d00, d01, d11 = (ab * ab).sum(-1), (ab * ac).sum(-1), (ac * ac).sum(-1)
    d20, d21 = (ap * ab).sum(-1), (ap * ac).sum(-1)
    den = d00 * d11 - d01 * d01
    v, w = (d11 * d20 - d01 * d21) / den, (d00 * d21 - d01 * d20) / den
    bary = torch.stack([1.0 - v - w, v, w], dim=1)
    best = torch.full_like(v, math.inf)
    edge = torch.zeros_like(bary)
    for k in range(3):
        j = (k + 1) % 3
        e = tri[:, j] - tri[:, k]
        s = (((p - tri[:, k]) * e).sum(-1) / (e * e).sum(-1)).clamp(0.0, 1.0)
        q = ((p - tri[:, k] - s[:, None] * e) ** 2).sum(-1)
        take = q < best
        best = torch.where(take, q, best)
        on = torch.zeros_like(bary)
        on[:, k], on[:, j] = 1.0 - s, s
        edge = torch.where(take[:, None], on, edge)
    return torch.where((bary >= 0.0).all(dim=1)[:, None], bary, edge)


def _train64(v, f, p):
    """The distances and the gradients of their mean square to p and v."""
    dist, face = _closest64(v, f, p)
    idx = f[face]
    w = _foot64(v[idx], p)
    g = 2.0 * (p - (w[..., None] * v[idx]).sum(1)) / p.shape[0]
    gv = torch.zeros_like(v)
    gv.index_add_(0, idx.reshape(-1), (-w[..., None] * g[:, None]).reshape(-1, 3))
    return dist, g, gv


def _rays64(v, f, o, d):
    tri = v[f]
    e1, e2 = tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    chunk = max(1, (1 << 24) // f.shape[0])
    depth = []
    for i in range(0, o.shape[0], chunk):
        oo, dd = o[i:i + chunk, None], d[i:i + chunk, None]
        h = torch.linalg.cross(dd.expand(-1, e2.shape[0], -1), e2[None].expand(dd.shape[0], -1, -1))
        inv = 1.0 / (e1 * h).sum(-1)
        s = oo - tri[None, :, 0]
        u = (s * h).sum(-1) * inv
        q = torch.linalg.cross(s, e1[None].expand_as(s))
        w = (dd * q).sum(-1) * inv
        t = (e2 * q).sum(-1) * inv
        t = torch.where((u >= 0) & (w >= 0) & (u + w <= 1) & (t >= 0), t, torch.full_like(t, 1000.0))
        depth.append(t.min(dim=1).values.clamp(max=1000.0))
    return torch.cat(depth)


def _cells64(coords, corners):
    """Vertices of the zero level in order of (lowest lattice point, axis), each from the
    first cell that holds its edge."""
    c, val = coords.to(torch.int64), corners.double()
    off = torch.tensor(_CORNERS, device=c.device)
    span = int(c.max()) + 2
    keys, cell, vert = [], [], []
    for a in range(8):
        for b in range(a + 1, 8):
            step = (off[b] - off[a]).abs()
            if int(step.sum()) != 1:
                continue
            cut = torch.nonzero((val[:, a] < 0.0) != (val[:, b] < 0.0)).squeeze(1)
            low = c[cut] + torch.minimum(off[a], off[b])
            keys.append(((low[:, 0] * span + low[:, 1]) * span + low[:, 2]) * 3 + int(step.argmax()))
            t = (-val[cut, a] / (val[cut, b] - val[cut, a]))[:, None]
            vert.append((c[cut] + off[a]).double() + t * (off[b] - off[a]).double())
            cell.append(cut)
    keys, cell, vert = torch.cat(keys), torch.cat(cell), torch.cat(vert)
    by_cell = torch.argsort(cell, stable=True)
    order = by_cell[torch.argsort(keys[by_cell], stable=True)]
    k = keys[order]
    first = torch.cat([k.new_ones(1, dtype=torch.bool), k[1:] != k[:-1]])
    return vert[order][first]


def exact(case, seed):
    family = case["family"]
    if family in ("flood", "voxels", "forest") or family == "sdf":
        return None
    if family == "cells":
        if case["average"]:
            return None
        return _cells64(*_cells(case, seed)), None
    v, f = _mesh(case["mesh"], case["level"], seed)
    n = case["n"] if "n" in case else case["width"] * case["height"] * case["views"]
    if n * len(f) > 1 << 32:
        return None
    v, f = torch.from_numpy(v).to(DEVICE).double(), torch.from_numpy(f).to(DEVICE).long()
    if family == "rays":
        o, d = (t.double() for t in _rays(case, seed))
        t = _rays64(v, f, o.reshape(-1, 3), d.reshape(-1, 3)).reshape(o.shape[:-1])
        return o + t[..., None] * d, None, t
    if family == "train":
        return _train64(v, f, _points("normal", n, seed).double())
    dist, _ = _closest64(v, f, _points(case["points"], n, seed).double())
    return (dist, None, None) if case["uvw"] else (dist, None)
