"""The ensemble's two-iterations-a-launch sweeps at their edges: members of no, one and an odd number of
iterations beside even ones, rows of several tiles, a few cells an axis, every shape; each member steps
bit for bit as its SmokeSim3D."""
import numpy as np
import pytest

from test_gpu_ensemble import SPHERE, initial, member_args

pytestmark = pytest.mark.gpu

MEMBERS = [((3, 2, 2), False, 2), ((300, 11, 9), True, 7), ((24, 90, 20), False, 0), ((40, 9, 70), True, 1),
           ((67, 35, 33), True, 12)]
SHAPES = [(2, 8, 8), (2, 16, 8), (2, 16, 16), (4, 8, 8), (4, 8, 16), (4, 8, 32)]


@pytest.mark.parametrize("which", [[0, 1, 2, 3, 4], [2], [0, 4]], ids=str)
def test_members_of_any_iteration_count_and_size(which):
    import zq_smokesimulation_amd as z
    from zq_smokesimulation_amd.ensemble import SmokeEnsemble, member_config
    cfgs, sims, states = [], [], []
    for n in which:
        (W, H, D), closed, iters = MEMBERS[n]
        args = member_args(closed, 0.03, 0.8, iters, W)
        cfgs.append(member_config(W, H, D, **args))
        sim = z.SmokeSim3D(W, H, D, **args)
        st = initial(W, H, D, closed, n == 4, 40 + n)
        sim.set_state(**st)
        sim.set_sphere_sources(SPHERE)
        sims.append(sim)
        states.append(st)
    ens = SmokeEnsemble(cfgs)
    for m, st in enumerate(states):
        ens.set_state(m, **st)
        ens.set_sources(m, spheres=SPHERE)
    try:
        # the shapes every ensemble has, and those chosen for this one's members
        own = [(c["tbx"], c["tby"], c["blocks"]) for c in ens.autotune(2)["candidates"] if c["kind"] != "half_sweeps"]
        for shape in [None] + sorted(set(SHAPES + own)):
            print("ensemble", which, shape, flush=True)
            if shape:
                ens.set_sweep(1, *shape)
                assert ens.sweep() == ("split_one_launch",) + shape
            ens.step(1, graph=shape != (4, 8, 16))
            ens.synchronize()
            for m, sim in enumerate(sims):
                sim.step()
                want, got = sim.get_state(), ens.get_state(m)
                for k in ("u", "v", "w", "T", "rho"):
                    a, b = np.asarray(got[k]).view(np.uint32), np.asarray(want[k]).view(np.uint32)
                    assert np.array_equal(a, b), "member %d %s shape %s: %d differ" % (m, k, shape, (a != b).sum())
        with pytest.raises(z.ZQ3DError):
            ens.set_sweep(1, 3, 8, 8)
    finally:
        for sim in sims:
            sim.close()
        ens.close()


def test_the_sweep_that_runs_is_reported():
    """A saved shape of the sweeps on 64 slots selects the nearest one and is reported as that; a refused shape
    changes nothing."""
    import zq_smokesimulation_amd as z
    from zq_smokesimulation_amd.ensemble import SmokeEnsemble, member_config
    ens = SmokeEnsemble([member_config(24, 20, 18, **member_args(True, 0.0, 0.5, 3, 24))])
    try:
        for rows, planes, want in ((8, 8, (2, 8, 8)), (8, 16, (2, 8, 16)), (16, 8, (2, 16, 8)), (16, 32, (2, 16, 16)),
                                   (32, 8, (2, 16, 8)), (32, 16, (2, 16, 16))):
            print("saved shape", rows, planes, flush=True)
            ens.set_sweep("split_one_launch", 64, rows, planes)
            assert ens.sweep() == ("split_one_launch",) + want
        for bad in ((1, 64, 16, 12), (1, 2, 8, 7), (0, 64, 5, 0), (0, 64, 4, -1), (2, 64, 4, 0)):
            with pytest.raises(z.ZQ3DError):
                ens.set_sweep(*bad)
            assert ens.sweep() == ("split_one_launch", 2, 16, 16)
        ens.set_sweep("half_sweeps", 32, 8, 256)
        assert ens.sweep() == ("half_sweeps", 32, 8, 256)
    finally:
        ens.close()
