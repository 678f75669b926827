"""Packet walks (64 queries or rays a wave) where they can go wrong, held to the wave walks
and to the oracle."""
import numpy as np
import pytest
import torch

import cubvh_amd
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
