"""The octree sweeps' cell lists and launch order on the GPU, bit for bit against the CPU oracle: leaves
that step one level at a time (lists of two levels share launches), and coarse leaves against fine cells
(cells with more neighbour entries than the head holds)."""
import numpy as np
import pytest

import zq_oracle as O
from test_gpu_octree import assert_same, exterior_masks, run_sim, scene
from util import faces

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,thresh,iters", [((72, 64, 64), (4, 8, 24), 13), ((72, 64, 64), (4, 8, 24), 1),
                                               ((64, 72, 80), (8, 16, 20), 6)])
def test_leaves_stepping_one_level_at_a_time(dims, thresh, iters):
    W, H, D = dims
    print("octree", dims, thresh, iters, flush=True)
    rng = np.random.default_rng(31)
    u, v, w = faces(rng, W, H, D)
    occ = scene(W, H, D, 31, [(0.0, 0.0, 8.0)])
    gu, gv, gw, _ = run_sim(W, H, D, u, v, w, occ, iters, thresh)
    leaves, _ = O.octree_projection(u, v, w, occ, iters, thresh, False)
    assert all(a.any() for a in leaves)
    for g, r, m, n in zip((gu, gv, gw), (u, v, w), exterior_masks(leaves), "uvw"):
        assert_same(g, r, n, m)


@pytest.mark.parametrize("closed", [False, True], ids=["open", "closed"])
@pytest.mark.parametrize("levels", [(3, 0), (3, 1), (3, 2), (2, 0), (3, 2, 1, 0)], ids=str)
def test_blocks_of_any_two_levels_side_by_side(levels, closed):
    """8^3 blocks of given levels in a checkerboard, some solid cells among the fine ones: up to 384
    entries a cell."""
    import zq_smokesimulation_amd as z
    W, H, D = 40, 32, 24
    print("octree blocks", levels, closed, flush=True)
    rng = np.random.default_rng(32)
    u, v, w = faces(rng, W, H, D)
    zz, yy, xx = np.mgrid[:D // 8, :H // 8, :W // 8]
    pick = np.array(levels)[(xx + yy + zz) % len(levels)]
    leaves = []
    for L in range(4):
        m = (pick == L).astype(np.uint8)
        for ax in range(3):
            m = np.repeat(m, 8 >> L, ax)
        leaves.append(m)
    leaves[0] &= (rng.random(leaves[0].shape) > 0.05).astype(np.uint8)
    mean = 0.01 if closed else 0.0
    ps = O.octree_solve(leaves, O.octree_divergence(u, v, w), 9, closed, mean)
    ru, rv, rw = u.copy(), v.copy(), w.copy()
    O.octree_adjust(leaves, ps, ru, rv, rw)
    assert z.stages.solve_octree(u, v, w, leaves, 9, div_per_volume=mean if closed else None) >= 0
    for g, r, n in zip((u, v, w), (ru, rv, rw), "uvw"):
        assert_same(g, r, n)
