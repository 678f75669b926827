"""The rays' test of a line against a face's bounding sphere drops only misses (CPU).

csrc/ray_line.hpp and the intersector are compiled for the host, with the host builder's
face disks, and run over rays aimed at the rim of faces from fat to thinner than their own
rounding, along the face's length, where the intersector's rounding moves a hit the most.
"""
import ctypes
import subprocess
from pathlib import Path

import numpy as np
import pytest

ROOT = Path(__file__).resolve().parents[1]


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    so = tmp_path_factory.mktemp("ray_line") / "ray_line.so"
    csrc = ROOT / "cubvh_amd" / "csrc"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", f"-I{csrc}", str(ROOT / "tests" / "host_ray_line.cpp"), str(csrc / "build.cpp"),
                    "-pthread", "-o", str(so)], check=True)
    lib = ctypes.CDLL(str(so))

    def run(tris, o, d):
        out = np.zeros(len(tris), np.uint8)
        arrays = [np.ascontiguousarray(x, np.float32) for x in (tris, o, d)]
        lib.ray_line_check(ctypes.c_int64(len(tris)), *[ctypes.c_void_p(x.ctypes.data) for x in arrays],
                           ctypes.c_void_p(out.ctypes.data))
        return out

    return run


def thin_faces(rng, n, aspect, length):
    """Faces [n, 9] of the given length and altitude/length about the origin, the vertex
    order turned at random, with their length direction [n, 3] and unit normal."""
    u, w = rng.normal(size=(2, n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    w -= (w * u).sum(1, keepdims=True) * u
    w /= np.linalg.norm(w, axis=1, keepdims=True)
    c = rng.uniform(-0.5, 0.5, (n, 3))
    x = rng.uniform(-0.5, 0.5, (n, 1))
    v = np.stack([c - 0.5 * length * u, c + 0.5 * length * u, c + length * (x * u + aspect * w)], axis=1)
    turn = (rng.integers(0, 3, n)[:, None] + np.arange(3)) % 3
    return np.take_along_axis(v, turn[:, :, None], axis=1).reshape(n, 9).astype(np.float32), u, np.cross(u, w)


def rim_rays(rng, tris, u, nrm, length):
    """Rays in the plane of the face's length and its normal, at every angle to the face:
    three in four towards its length line around its bounding sphere's rim, one into it."""
    n = len(tris)
    v = tris.reshape(n, 3, 3).astype(np.float64)
    inside = rng.random((n, 1)) < 0.25
    mean = np.where(inside, (v * rng.dirichlet(np.ones(3), n)[:, :, None]).sum(axis=1), v.mean(axis=1))
    out = np.where(inside, 0.0, rng.choice([-1.0, 1.0], (n, 1)) * length * rng.uniform(0.4, 0.75, (n, 1)))
    angle = np.exp(rng.uniform(np.log(0.02), np.log(1.5), (n, 1))) * rng.choice([-1.0, 1.0], (n, 1))
    d = np.cos(angle) * u + np.sin(angle) * nrm
    o = mean + out * u - rng.uniform(0.5, 4.0, (n, 1)) * d
    return o, d * np.exp(rng.uniform(-3.0, 3.0, (n, 1)))


@pytest.mark.parametrize("aspect", [0.5, 0.1, 0.0626, 0.03, 1e-2, 1e-3, 1e-4, 1e-5, 3e-6, 1e-6, 3e-7, 1e-7])
@pytest.mark.parametrize("length", [1.0, 0.1, 0.01])
def test_rejected_lines_are_misses(check, aspect, length):
    rng = np.random.default_rng(int(1e7 * aspect) + int(1000 * length))
    n = 100_000
    tris, u, nrm = thin_faces(rng, n, aspect, length)
    out = check(tris, *rim_rays(rng, tris, u, nrm, length))
    hit, rejected, exempt = (out & 1) != 0, (out & 2) != 0, (out & 4) != 0
    assert hit.any()
    assert not (hit & rejected).any()
    if aspect == 0.5:  # the test does its work on ordinary faces
        assert rejected.any() and not exempt.any()


def test_degenerate_faces_are_never_rejected(check):
    """Zero-area faces, faces whose products under- or overflow, NaN and infinite corners."""
    rng = np.random.default_rng(1)
    base = rng.normal(size=(64, 9))
    faces = [base * s for s in (1e-15, 1e13, 0.0)]
    flat = base.copy()
    flat[:, 3:6] = flat[:, :3]
    bad = base.copy()
    bad[::2, 4], bad[1::2, 7] = np.nan, np.inf
    faces = np.concatenate([*faces, flat, bad]).astype(np.float32)
    o, d = rng.normal(size=(2, len(faces), 3))
    assert (check(faces, 5.0 * o, d) & 6 == 4).all()
