"""One wave per query (small calls) against packets of queries and the oracle.

Calls below 2^18 queries walk one wave per query, larger ones as packets of 64 in Morton
order; distance_ordered always walks packets.  Both have to give the oracle's bits, so
each is held to the other bit for bit on inputs that the oracle tests also cover.
"""
import numpy as np
import pytest
import torch

import cubvh_amd
from cubvh_amd import synthetic as S

pytestmark = pytest.mark.gpu

WAVE_MAX = 1 << 18


def _same(a, b):
    """Equal bits, NaN included (+0 and -0 differ)."""
    for x, y in zip(a, b):
        assert x.dtype == y.dtype
        if x.dtype == torch.float32:
            x, y = x.view(torch.int32), y.view(torch.int32)
        assert torch.equal(x, y)


def _mesh(kind):
    if kind == "copies":  # one face many times, all tied: more pending nodes than any real mesh
        t = np.array([[0.1, 0.0, 0.0], [0.0, 0.1, 0.0], [0.0, 0.0, 0.1]], dtype=np.float32)
        return np.tile(t, (3000, 1)), np.arange(9000, dtype=np.int32).reshape(-1, 3)
    if kind == "flat":  # zero-area faces among the others
        v, f = S.icosphere(4, 0.5)
        f = f.copy()
        f[::7, 1] = f[::7, 0]
        return v, f
    if kind == "nine":
        v, f = S.icosphere(0, 0.5)
        return v, f[:9]
    return S.soup(5, seed=3, n_random=4000)


def _points(n):
    p = S.uniform_points(n, seed=n)
    p[: n // 4] *= 0.05  # near the middle, where thousands of faces are about as far
    special = np.array([[np.nan, 0, 0], [0, np.inf, 0], [np.nan] * 3, [2000, 0, 0], [0, 0, 0]], dtype=np.float32)
    p[: min(n, 5)] = special[: min(n, 5)]
    return torch.from_numpy(p).cuda()


@pytest.mark.parametrize("n", [1, 63, 65, 2047, 30011])
@pytest.mark.parametrize("kind", ["nine", "soup", "copies", "flat"])
def test_wave_distance_equals_packets(gpu, kind, n):
    v, f = _mesh(kind)
    bvh = cubvh_amd.cuBVH(v, f)
    p = _points(n)
    order = torch.arange(n, dtype=torch.int32, device=gpu)
    _same(bvh.unsigned_distance(p, return_uvw=True), bvh.distance_ordered(p, order, return_uvw=True))
    _same(bvh.signed_distance(p)[:2], bvh.distance_ordered(p, order, signed=True)[:2])


@pytest.mark.parametrize("kind", ["nine", "soup", "copies"])
def test_wave_results_at_the_size_limit(gpu, kind):
    """The same queries in one call at the limit (packets) and in two below it (waves)."""
    v, f = _mesh(kind)
    bvh = cubvh_amd.cuBVH(v, f)
    n = WAVE_MAX if kind == "nine" else WAVE_MAX + 77
    m = 30011 if kind == "copies" else n // 2
    p = _points(n)
    whole = bvh.unsigned_distance(p, return_uvw=True)
    for part in (slice(0, m), slice(n - m, n)):
        _same([t[part] for t in whole], bvh.unsigned_distance(p[part], return_uvw=True))
    o, d = (torch.from_numpy(t).cuda() for t in S.sphere_rays(n, seed=5))
    d[:3] = torch.tensor([[0.0, 0.0, 0.0], [float("nan"), 1.0, 0.0], [0.0, 0.0, 1.0]])
    o[3:9] = torch.from_numpy(v[f[:6]].mean(axis=1)).cuda()  # origins on faces: hits at 0 and -0
    hits = bvh.ray_trace(o, d)
    for part in (slice(0, m), slice(n - m, n)):
        _same([t[part] for t in hits], bvh.ray_trace(o[part], d[part]))


@pytest.mark.parametrize("scale", [1.0, 1e-3, 1e9])
@pytest.mark.parametrize("kind", ["nine", "soup", "copies", "flat"])
def test_ray_packets_equal_waves(gpu, kind, scale):
    """Parallel and pinhole rays (packets) from outside, from a face and along a face's plane
    against the same rays in calls small enough for a wave each.  A ray in a face's plane
    can meet it at a rounded t before the mesh's own box; which of several copies of the face
    it then reports is the order of the walk's, so such hits' face ids are not compared."""
    v, f = _mesh(kind)
    bvh = cubvh_amd.cuBVH(v, f)
    x = torch.linspace(-0.6, 0.6, 181, device=gpu)
    g = torch.stack(torch.meshgrid(x, x, indexing="ij"), dim=-1).reshape(-1, 2)
    t = torch.from_numpy(v[f[1]]).to(gpu)
    edge = t[1] - t[0]
    z = torch.ones_like(g[:, :1])
    eye = torch.tensor([0.3, -0.2, 1.7], device=gpu)
    o = [torch.cat([g, 3.0 * z], 1), eye.expand(len(g), 3), (t[0] - 2.0 * edge).expand(len(g), 3) + 1e-7 * torch.cat([g, z], 1),
         t.mean(0).expand(len(g), 3)]
    d = [torch.tensor([0.0, 0.0, -1.0], device=gpu).expand(len(g), 3), torch.cat([0.4 * g, -1.7 * z], 1),
         edge / edge.norm() + 1e-4 * torch.cat([g, z], 1), torch.cat([0.1 * g, z], 1)]
    rep = WAVE_MAX // (4 * len(g)) + 1
    o, d = torch.cat(o).repeat(rep, 1).contiguous(), (torch.cat(d) * scale).repeat(rep, 1).contiguous()
    assert len(o) >= WAVE_MAX
    whole = bvh.ray_trace(o, d)
    lo, hi = (torch.from_numpy(e).to(gpu) for e in (v[f].min(axis=(0, 1)) - 1e-3, v[f].max(axis=(0, 1)) + 1e-3))
    off = (whole[1] >= 0) & ~((whole[0] >= lo) & (whole[0] <= hi)).all(dim=1)
    assert int(off.sum()) < len(o) // 1000
    m = 4 * len(g)
    for at in range(0, len(o), m):
        part = slice(at, at + m)
        small = bvh.ray_trace(o[part], d[part])
        _same([whole[0][part], whole[2][part]], [small[0], small[2]])
        _same([whole[1][part][~off[part]]], [small[1][~off[part]]])


@pytest.mark.parametrize("kind", ["nine", "soup", "copies", "closed"])
def test_raystab_sizes_agree(gpu, oracle, kind):
    """Raystab signs with lines by waves (small calls), by lanes and waves (from 2^18) and by
    lanes (from 2^20) on the same leading queries (a query's directions depend on its index),
    and against the oracle."""
    v, f = S.icosphere(3, 0.5) if kind == "closed" else _mesh(kind)
    bvh = cubvh_amd.cuBVH(v, f)
    p = _points((1 << 20) + 77 if kind != "copies" else WAVE_MAX + 77)
    p[5:400] *= 0.3
    big = bvh.signed_distance(p, mode="raystab")[:2]
    for n in (1, 65, 2049, WAVE_MAX - 1, WAVE_MAX + 1):
        _same(bvh.signed_distance(p[:n], mode="raystab")[:2], [t[:n] for t in big])
    od, of, _ = oracle.sdf_brute(v, f, p[5:500].cpu().numpy(), 1, return_uvw=False)
    np.testing.assert_array_equal(big[0][5:500].cpu().numpy(), od)
    np.testing.assert_array_equal(big[1][5:500].cpu().numpy(), of)
