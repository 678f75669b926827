"""Packet walks (64 queries or rays a wave) where they can go wrong, held to the wave walks
and to the oracle."""
import contextlib
import ctypes
import inspect
import math

import numpy as np
import pytest
import torch

import cubvh_amd
from cubvh_amd import synthetic as S
import test_gpu_queries
from test_ray_line_host import check, rim_rays, thin_faces  # noqa: F401 (a fixture)

pytestmark = pytest.mark.gpu

COPIES = 64  # of every ray: a packet's tile of equal rays


def same_bits(a, b):
    """Equal bits, NaN included (+0 and -0 differ)."""
    for x, y in zip(a, b):
        assert x.dtype == y.dtype and x.shape == y.shape
        if x.dtype == torch.float32:
            x, y = x.view(torch.int32), y.view(torch.int32)
        assert torch.equal(x, y)


@pytest.mark.parametrize("aspect", [1e-2, 1e-5, 3e-7, 1e-7, 3e-8])
@pytest.mark.parametrize("builder", ["host", "gpu", "gpu_sah"])
def test_thin_faces_ray_packets_equal_waves(gpu, check, builder, aspect):  # noqa: F811
    """One leaf of 16 faces down to thinner than their rounding, rays around their ends that
    the intersector says hit them: the line test of the packets drops none."""
    rng = np.random.default_rng(int(1e9 * aspect))
    tris, u, nrm = thin_faces(rng, 16, aspect, 1.0)
    pick = rng.integers(0, 16, 400_000)
    o, d = rim_rays(rng, tris[pick], u[pick], nrm[pick], 1.0)
    hit = np.flatnonzero(check(tris[pick], o, d) & 1)
    hit = hit[np.argsort(-np.abs((d[hit] * nrm[pick[hit]]).sum(axis=1)), kind="stable")][:8192]
    o, d = (torch.from_numpy(np.resize(x[hit], (8192, 3)).astype(np.float32)).to(gpu) for x in (o, d))
    bvh = cubvh_amd.cuBVH(tris.reshape(-1, 3), np.arange(48, dtype=np.int32).reshape(-1, 3), build=builder)
    small = bvh.ray_trace(o, d)
    large = bvh.ray_trace(o.repeat_interleave(COPIES, 0), d.repeat_interleave(COPIES, 0))
    same_bits([x[::COPIES] for x in large], small)
    assert (small[1] >= 0).any()


@pytest.mark.parametrize("builder", ["host", "gpu", "gpu_lbvh"])
@pytest.mark.parametrize("n_faces", [12, 90, 700])
def test_watertight_sign_is_the_exact_normal_sums(gpu, n_faces, builder):
    """Sheets back to back whose normals cancel, with small ones left over: the sign is the
    exact sum's, whatever the order of the faces, by waves and by packets."""
    rng = np.random.default_rng(n_faces)
    up = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0]], np.float32)
    small = [1e-9, 1e-12, 3e-17, 1e-20, 1e-25, 2.5e-30, 1e-36]
    for trial in range(24):
        pairs = n_faces // 3
        # normals (-1, 0, -x) of faces that go down from the edge shared by all
        left = rng.choice(small[trial % 4:], n_faces - 2 * pairs) * rng.choice([-1.0, 1.0], n_faces - 2 * pairs)
        left[1::2] = -left[:-1:2][: len(left[1::2])]  # in turn cancelled, but for the last
        left = np.append(left[:-1], rng.choice(small[3:]) * rng.choice([-1.0, 1.0])).astype(np.float32)
        faces = [up, up[[0, 2, 1]]] * pairs + [np.array([[0, 0, 0], [0, 1, 0], [x, 0, -1]], np.float32) for x in left]
        faces = np.stack([faces[i] for i in rng.permutation(n_faces)])
        inside = -math.fsum(left.tolist()) < 0.0
        bvh = cubvh_amd.cuBVH(faces.reshape(-1, 3), np.arange(3 * n_faces, dtype=np.int32).reshape(-1, 3), build=builder)
        p = torch.zeros(100, 3, device=gpu)
        p[:, 1] = torch.linspace(0.1, 0.9, 100, device=gpu)
        p[:, 2] = torch.linspace(0.01, 0.5, 100, device=gpu)
        waves = bvh.signed_distance(p)
        packets = bvh.distance_ordered(p, torch.arange(100, dtype=torch.int32, device=gpu), signed=True)
        same_bits(waves[:2], packets[:2])
        assert bool((torch.signbit(waves[0]) == inside).all())


def test_ordered_calls_leave_skipped_queries_alone(gpu):
    """Order entries past the end: the queries they leave out keep their outputs, whatever is
    in them, and the others get theirs, small normals among the sheets or not."""
    faces = np.array([[[0, 0, 0], [1, 0, 0], [0, 1, 0]], [[0, 0, 0], [0, 1, 0], [1, 0, 0]], [[0, 0, 0], [0, 1, 0], [-1e-20, 0, -1]]],
                     np.float32)[[0, 1, 2] * 4]
    bvh = cubvh_amd.cuBVH(faces.reshape(-1, 3), np.arange(36, dtype=np.int32).reshape(-1, 3))
    n = 5000
    p = torch.rand(n, 3, device=gpu)
    p[:, 0] = 0.0
    order = torch.randperm(n, device=gpu).to(torch.int32)
    skipped = order[::3].long()
    order[::3] = n + 7
    d = torch.full((n,), 3.0, device=gpu)
    f = torch.full((n,), -12345, dtype=torch.int64, device=gpu)
    lib = cubvh_amd._lib.load()
    stream = ctypes.c_void_p(torch.cuda.current_stream(gpu).cuda_stream)
    cubvh_amd._lib.check(lib.cubvh_distance_ordered(bvh._h, gpu.index, n, 1, p.data_ptr(), order.data_ptr(), d.data_ptr(),
                                                    f.data_ptr(), None, stream))
    ref = bvh.signed_distance(p)
    kept = torch.ones(n, dtype=torch.bool, device=gpu)
    kept[skipped] = False
    assert bool((d[skipped] == 3.0).all()) and bool((f[skipped] == -12345).all())
    same_bits([d[kept], f[kept]], [ref[0][kept], ref[1][kept]])


@contextlib.contextmanager
def walks(handle, route=0, cap=-1, first=0, factor=-1):
    """The tree's (or forest's) queries walk as told; yields a function that says how many
    queries the last call handed over."""
    lib = cubvh_amd._lib.load()
    fn = lib.cubvh_forest_walk_control if isinstance(handle, cubvh_amd.cuBVHForest) else lib.cubvh_bvh_walk_control

    def control(*values):
        cubvh_amd._lib.check(fn(handle._h, (ctypes.c_int32 * 4)(*values), None))

    def handed():
        count = ctypes.c_uint32(0)
        cubvh_amd._lib.check(fn(handle._h, None, ctypes.byref(count)))
        return count.value

    control(route, cap, first, factor)
    try:
        yield handed
    finally:
        control(0, -1, 0, -1)


@pytest.mark.parametrize("level", [0, 2, 4, 6])
def test_routes_agree_around_their_limits(gpu, level):
    """Calls just below and above the sizes where the route changes: the same bits from the
    route taken and from the other one."""
    v, f = S.icosphere(level, 0.5)
    bvh = cubvh_amd.cuBVH(v, f)
    for n in (98_303, 98_304, 131_072, 147_456, 196_607, 196_608, 262_144):
        p = torch.from_numpy(S.uniform_points(n, seed=n)).to(gpu)
        o, d = (torch.from_numpy(x).to(gpu) for x in S.sphere_rays(n, seed=n))
        calls = [lambda: bvh.unsigned_distance(p, return_uvw=True), lambda: bvh.signed_distance(p)[:2],
                 lambda: bvh.ray_trace(o, d)]
        if n in (131_072, 196_607):
            calls.append(lambda: bvh.signed_distance(p, mode="raystab")[:2])
        for call in calls:
            out = call()
            for route in (1, 2):
                with walks(bvh, route):
                    same_bits(out, call())


# route, places of the list, steps before a walk may end, sixteenths of the average
CONTROLS = {"packets": (2, -1, 0, -1), "handed over": (2, 1 << 19, 8, 0), "list full": (2, 37, 8, 0), "no list": (2, 0, 8, 0)}


@pytest.mark.parametrize("control", CONTROLS)
@pytest.mark.parametrize("name", [
    "test_udf_leading_dims_and_far_points", "test_udf_perturbed_level6_bit_exact", "test_rays_bit_exact_and_vs_fp64",
    "test_sdf_watertight_bit_exact", "test_sdf_raystab_threshold_sizes_and_empty_lists", "test_duplicate_faces_tie_to_lowest_index",
    "test_camera_rays_packet_path_bit_exact", "test_nan_and_inf_queries", "test_degenerate_faces_bit_exact",
    "test_ray_edge_cases_bit_exact", "test_points_on_the_surface_bit_exact", "test_random_soups_bit_exact"])
def test_oracle_by_packets(gpu, request, monkeypatch, name, control):
    """The oracle tests of the query calls, whose sizes the library gives to waves, with every
    query in packets, whose walks all end where told or may hand over after a few steps."""
    init = cubvh_amd.cuBVH.__init__

    def controlled(self, *args, **kwargs):
        init(self, *args, **kwargs)
        walks(self, *CONTROLS[control]).__enter__()

    monkeypatch.setattr(cubvh_amd.cuBVH, "__init__", controlled)
    test = getattr(test_gpu_queries, name)
    given = {"seed": 103} if name == "test_random_soups_bit_exact" else {}
    for arg in inspect.signature(test).parameters:
        if arg not in given:
            given[arg] = request.getfixturevalue(arg)
    test(**given)


def _cells_of(case, gpu):
    """Mesh and calls of a hand-over case: name -> call, the same queries at their own order."""
    rng = np.random.default_rng(11)
    v, f = S.soup(5, seed=3, n_random=4000)
    n = 60_011
    p = S.uniform_points(n, seed=12)
    p[: n // 3] = (v[f[rng.integers(0, len(f), n // 3)]].mean(axis=1) + rng.normal(0, 0.01, (n // 3, 3))).astype(np.float32)
    p[:5] = [[np.nan, 0, 0], [0, np.inf, 0], [np.nan] * 3, [2000, 0, 0], [0, 0, 0]]
    P = torch.from_numpy(p[rng.permutation(n)]).to(gpu)
    if case == "lanes":
        rays = S.sphere_rays(n, seed=13)
    else:
        rays = S.camera_rays(width=320, height=96, n_poses=2, seed=3)
    O, D = (torch.from_numpy(x).to(gpu) for x in rays)
    bvh = cubvh_amd.cuBVH(v, f)
    return bvh, {"unsigned": lambda: bvh.unsigned_distance(P, return_uvw=True), "watertight": lambda: bvh.signed_distance(P, return_uvw=True),
                 "lanes": lambda: bvh.ray_trace(O, D), "camera": lambda: bvh.ray_trace(O, D)}[case]


@pytest.mark.parametrize("case", ["unsigned", "watertight", "lanes", "camera"])
def test_handed_over_walks_equal_waves(gpu, case):
    """Lists that hold every walk that ends early, some of them (places in the middle of a
    wave's run stay empty), and none: the same bits, and the list was used, or too short."""
    bvh, call = _cells_of(case, gpu)
    with walks(bvh, 1):
        ref = call()
    for cap in (1 << 19, 5000, 100, 1, 0):
        for factor in (0, 24):
            with walks(bvh, 2, cap, 8, factor) as handed:
                same_bits(ref, call())
                assert handed() > (cap if cap <= 100 or (cap == 5000 and factor == 0) else 0)


@pytest.mark.parametrize("tuning", [(4, 0, 8, 1), (4, 0, 8, 8), (4, 1, 4, 2), (0, 1, 16, 4)])
def test_handed_over_forest_walks_equal_single_meshes(gpu, tuning):
    meshes = [S.soup(4, seed=s, n_random=500) for s in range(5)] + [S.icosphere(1, 0.4)]
    bvhs = [cubvh_amd.cuBVH(*m) for m in meshes]
    counts = [9000, 0, 12_345, 70, 8000, 3000]
    off = torch.from_numpy(np.concatenate([[0], np.cumsum(counts)]))
    P = torch.from_numpy(S.uniform_points(sum(counts), seed=5)).to(gpu)
    forest = cubvh_amd.cuBVHForest(bvhs)
    ref = [torch.cat(x) for x in zip(*[b.unsigned_distance(P[a:e], return_uvw=True) for b, a, e in zip(bvhs, off, off[1:]) if e > a])]
    for cap in (1 << 19, 1000, 100, 0):
        with walks(forest, 0, cap, 8, 0) as handed:
            same_bits(ref, forest.unsigned_distance(P, off, return_uvw=True, tuning=tuning))
            assert handed() > (0 if cap == 1 << 19 else cap)
