"""GPU floodfill (union-find kernels) against the oracle's BFS and scipy: bit-exact."""
import numpy as np
import pytest
import torch

import cubvh_amd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 16, 16, 16), (3, 9, 9, 9), (2, 5, 7, 11), (1, 1, 1, 64), (4, 32, 8, 2)])
def test_floodfill_random_grids(gpu, oracle, shape):
    rng = np.random.default_rng(sum(shape))
    for p in (0.1, 0.3, 0.5, 0.8):
        g = rng.random(shape) < p
        lab = cubvh_amd.floodfill(torch.from_numpy(g).to(gpu))
        assert lab.dtype == torch.int32 and tuple(lab.shape) == shape
        np.testing.assert_array_equal(lab.cpu().numpy(), oracle.floodfill_bfs(g))


def test_floodfill_cubic_equals_reference_loop(gpu, oracle):
    rng = np.random.default_rng(1)
    g = rng.random((2, 24, 24, 24)) < 0.45
    lab = cubvh_amd.floodfill(torch.from_numpy(g).to(gpu)).cpu().numpy()
    ref, it = oracle.floodfill_ref(g)
    assert it > 0
    np.testing.assert_array_equal(lab, ref)


def test_floodfill_3d_input_and_edge_cases(gpu, oracle):
    g = torch.zeros(8, 8, 8, dtype=torch.bool)
    lab = cubvh_amd.floodfill(g)  # 3-D CPU input: moved, unsqueezed, squeezed back
    assert lab.shape == (8, 8, 8) and lab.is_cuda
    assert (lab == 0).all()
    lab = cubvh_amd.floodfill(torch.ones(2, 4, 4, 4, dtype=torch.bool, device=gpu))
    assert (lab == -1).all()
    g = torch.zeros(1, 10, 10, 10, dtype=torch.bool)
    g[0, 5] = True
    lab = cubvh_amd.floodfill(g.to(gpu)).cpu()
    assert set(lab[0, :5].unique().tolist()) == {0} and set(lab[0, 6:].unique().tolist()) == {600}


def test_floodfill_occupancy_of_distance_field(gpu, oracle):
    """Occupancy udf < 2/res of a perturbed sphere at 96^3: inside and outside are two
    components; the labels equal the BFS."""
    from cubvh_amd import synthetic as S

    res = 96
    v, f, _ = S.perturbed_sphere(5, seed=0)
    bvh = cubvh_amd.cuBVH(v, f)
    pts = torch.from_numpy(S.grid_points(res)).to(gpu)
    d, _, _ = bvh.unsigned_distance(pts)
    occ = (d < 2.0 / res).reshape(1, res, res, res)
    lab = cubvh_amd.floodfill(occ).cpu().numpy()
    ref = oracle.floodfill_bfs(occ.cpu().numpy())
    np.testing.assert_array_equal(lab, ref)
    assert len(np.unique(lab[lab >= 0])) >= 2


@pytest.mark.parametrize("shape", [(1, 8, 8, 64), (1, 9, 17, 65), (2, 33, 3, 130), (1, 17, 40, 63), (1, 64, 64, 128)])
@pytest.mark.parametrize("kind", ["noise", "open", "maze"])
def test_floodfill_across_tiles(gpu, oracle, shape, kind):
    """Sizes around the labelling tiles (64 x 8 x 8): random grids, one open component, and
    one long winding corridor (walls with a gap at alternating ends)."""
    rng = np.random.default_rng(sum(shape))
    if kind == "noise":
        g = rng.random(shape) < 0.55
    elif kind == "open":
        g = np.zeros(shape, dtype=bool)
        g[..., shape[-1] // 2] = rng.random(shape[:-1]) < 0.9
    else:
        g = np.zeros(shape, dtype=bool)
        g[:, 1::2] = True
        g[:, 1::4, -1, -1] = False
        g[:, 3::4, 0, 0] = False
        g[:, ::2, 1::2] = True
        g[:, ::2, 1::4, -1] = False
        g[:, ::2, 3::4, 0] = False
    lab = cubvh_amd.floodfill(torch.from_numpy(g).to(gpu)).cpu().numpy()
    np.testing.assert_array_equal(lab, oracle.floodfill_bfs(g))


@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (5, 1, 1, 1), (1, 1, 1, 70), (1, 1, 70, 1), (3, 70, 1, 1), (2, 33, 50, 1), (1, 1, 17, 9),
                                   (1, 40, 1, 12), (1, 16, 16, 16), (2, 17, 33, 2), (1, 50, 35, 16), (1, 50, 35, 17),
                                   (3, 9, 70, 7), (1, 100, 90, 1), (70, 4, 4, 4), (1023, 5, 6, 3), (1024, 5, 6, 3), (256, 16, 16, 16),
                                   (130, 17, 19, 2), (1, 257, 249, 16), (1, 250, 265, 9), (3, 129, 300, 5), (300, 15, 9, 13)])
@pytest.mark.parametrize("free", [0.4, 0.65, 0.9, 1.0])
def test_floodfill_short_axes(gpu, oracle, shape, free):
    """A short last axis (tiles of 16 x 16 x 16 from 1,024 tiles of 64 x 8 x 8 on), around their
    sizes, and axes of one voxel."""
    g = np.random.default_rng(sum(shape)).random(shape) >= free
    lab = cubvh_amd.floodfill(torch.from_numpy(g).to(gpu)).cpu().numpy()
    np.testing.assert_array_equal(lab, oracle.floodfill_bfs(g))


def test_floodfill_flat_grid_of_more_than_2_30_voxels(gpu):
    """2^15 x (2^15 + 8) x 1: more tiles than one launch takes if tiles are laid along the last
    axis.  Two occupied rows leave three components, each labelled by its first voxel."""
    h, w = 1 << 15, (1 << 15) + 8
    g = torch.zeros((1, h, w, 1), dtype=torch.bool, device=gpu)
    g[0, 1000] = True
    g[0, 20_001] = True
    lab = cubvh_amd.floodfill(g)[0, :, :, 0]
    for first, last, value in ((0, 1000, 0), (1000, 1001, -1), (1001, 20_001, 1001 * w), (20_001, 20_002, -1), (20_002, h, 20_002 * w)):
        assert bool((lab[first:last] == value).all())
