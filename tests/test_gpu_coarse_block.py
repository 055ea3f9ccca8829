"""The coarse sweeps on boxes held in registers, against the oracle's sweep order (faces on coarse planes bit
for bit): one box and several along each axis, odd sizes, solids, open and closed sides."""
import numpy as np
import pytest

import zq_oracle as O
from test_gpu_coarse import assert_same, scene
from util import faces

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,zcs", [((40, 24, 36), [(1, -30804), (2, -30804), (1, -20803), (3, -40804), (1, -20402)]),
                                      ((12, 8, 20), [(1, -30804), (1, -20402), (2, -40402)]),
                                      ((132, 44, 36), [(2, -30804), (1, -30508), (1, -50404), (2, -50503)])])
@pytest.mark.parametrize("mask,iters", [(O.ALL_FACES, 23), (O.OPEN_YHI, 4), (O.ALL_FACES, 1), (O.ALL_FACES, 0)])
def test_boxes_give_the_oracles_bits(dims, zcs, mask, iters):
    from zq_smokesimulation_amd.sim import SmokeSim3D
    import zq_smokesimulation_amd._lib as L
    rng = np.random.default_rng(17)
    (W, H, D), s = dims, 4
    u, v, w = faces(rng, W, H, D)
    occ = scene(rng, W, H, D, 0.02)
    ru, rv, rw = u.copy(), v.copy(), w.copy()
    O.coarse_projection(ru, rv, rw, occ, s, iters, 1.4, mask)
    sim = SmokeSim3D(W, H, D, sub_size=s, sor_iters=iters, sor_omega=1.4, sor_open_mask=mask)
    try:
        for k, zc in zcs:
            print("boxes", dims, k, zc, iters, flush=True)
            sim.set_coarse_sweep(k, zc)
            assert sim.coarse_sweep() == (k, zc)
            sim.set_state(u=u, v=v, w=w, occ=occ)
            sim.project()
            got = [sim.download(f) for f in (L.FIELD_U, L.FIELD_V, L.FIELD_W)]
            assert_same(got[0][:, :, ::s], ru[:, :, ::s], "u coarse planes %d %d" % (k, zc))
            assert_same(got[1][:, ::s, :], rv[:, ::s, :], "v coarse planes %d %d" % (k, zc))
            assert_same(got[2][::s], rw[::s], "w coarse planes %d %d" % (k, zc))
        for k, zc in ((2, -5), (1, -808), (9, -30804), (2, -70804), (1, -41604 - 12), (-1, -30804)):
            with pytest.raises(L.ZQ3DError):
                sim.set_coarse_sweep(k, zc)
    finally:
        sim.close()
