"""GPU: the quad-layout sweeps (several red-black iterations per launch, planes or boxes in registers) against the
oracle's SOR bit for bit, at the sizes where tiles, row groups, lanes and chunks end."""
import numpy as np
import pytest

import zq_oracle as O

pytestmark = pytest.mark.gpu


def project(W, H, D, shapes, iters, mask, closed, seed=3):
    import zq_smokesimulation_amd as z
    from util import faces, occupancy
    rng = np.random.default_rng(seed)
    u, v, w = faces(rng, W, H, D)
    occ = occupancy(rng, W, H, D, 0.1, shell=closed)
    sim = z.SmokeSim3D(W, H, D, sor_open_mask=mask, sor_closed_mean=0, sor_omega=1.7, sor_iters=iters)
    ref = [a.copy() for a in (u, v, w)]
    O.project(*ref, occ, mask, 0.0, 1.7, iters)
    for shape in shapes:
        sim.set_sor_shape(*shape)
        if shape[0]:
            assert sim.sor_kernel() == ("k_sor_block" if shape[0] <= -100000 else "k_sor_quad")
        sim.set_state(u=u, v=v, w=w, occ=occ)
        sim.project()
        g = sim.get_state()
        for name, a in zip("uvw", ref):
            assert np.array_equal(g[name].view(np.uint32), a.view(np.uint32)), (W, H, D, shape, iters, name)
    sim.close()


# W: 2 and 3 cells; 4-cell padding 0..3; one full wave of lanes (128 and 256 cells) and one cell more (two
# tiles with halo lanes); H and D around a tile's rows and a chunk's planes
@pytest.mark.parametrize("dims", [(2, 3, 2), (3, 2, 5), (16, 9, 7), (17, 20, 9), (18, 33, 8), (19, 12, 31),
                                  (64, 17, 13),
                                  (127, 18, 10), (128, 11, 9), (129, 16, 12), (256, 19, 6), (257, 9, 9), (300, 25, 7),
                                  (521, 7, 5)])
@pytest.mark.parametrize("iters", [0, 1, 2, 5])
def test_default_shape_at_tile_edges(dims, iters):
    project(*dims, [(0, 0), (-1216, 4), (-1408, 8)], iters, O.OPEN_YHI | O.OPEN_XLO, False)


# (code, grid): few and many waves, both lane widths, each on a grid that it cuts along several axes (at 140
# columns fewer than 5 waves would own no row beside their halo)
@pytest.mark.parametrize("code,dims", [(-1202, (20, 61, 21)), (-1204, (48, 61, 21)), (-1208, (140, 41, 21)),
                                       (-1212, (140, 41, 21)), (-1216, (140, 71, 21)), (-1402, (40, 61, 21)),
                                       (-1405, (140, 41, 21)), (-1408, (270, 41, 21))])
def test_every_width_and_wave_count(code, dims):
    shapes = [(code, zc) for zc in (2, 4, 16)]
    project(*dims, shapes, 7, 0, True)
    project(*dims, shapes, 4, O.ALL_FACES, False)


# boxes of lx x ty x tz threads (code: log2 lx, ty, tz), one box and several along each axis, odd sizes, a
# last box of a few cells, iteration counts that the launches do not divide
@pytest.mark.parametrize("code,ks,dims", [((3, 8, 4), (1, 2, 3), (20, 24, 16)), ((3, 8, 4), (2,), (33, 17, 19)),
                                          ((4, 12, 4), (1,), (20, 24, 16)), ((4, 12, 4), (1,), (3, 2, 2)),
                                          ((2, 5, 3), (1,), (29, 23, 26)), ((6, 4, 4), (1,), (128, 9, 21)),
                                          ((6, 6, 2), (1,), (131, 13, 13)), ((5, 6, 5), (1, 2), (65, 40, 37)),
                                          ((1, 5, 5), (1,), (4, 21, 30)), ((4, 10, 6), (2, 3), (70, 31, 40))])
def test_boxes_held_in_registers(code, ks, dims):
    ty = -(100000 + 10000 * code[0] + 100 * code[1] + code[2])
    shapes = [(ty, k) for k in ks]
    project(*dims, shapes, 7, 0, True)
    project(*dims, shapes, 4, O.ALL_FACES, False)
    project(*dims, shapes, 1, O.OPEN_ZHI, False)


def test_shapes_outside_the_range_are_refused():
    import zq_smokesimulation_amd as z
    sim = z.SmokeSim3D(40, 40, 40)
    for s in ((-1200, 4), (-1217, 4), (-1409, 4), (-1308, 4), (-1208, 3), (-1208, 0), (-1208, 66), (-1201, 4),
              (-130804, 0), (-130804, 9), (-130800, 2), (-100804, 2), (-170804, 1), (-161610, 1), (-120404, 2)):
        with pytest.raises(z._lib.ZQ3DError):
            sim.set_sor_shape(*s)
    sim.close()
