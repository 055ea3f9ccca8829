"""The coarse sweeps' schedule is chosen by a rule (csrc/zq3d_block_cut.h: block_cost_weighted), compiled with g++:
on the CPU every grid of 1 to 129 cells an axis gets boxes that cover it and fit a workgroup of 512 threads, and
none is predicted faster; on the GPU a simulation takes exactly the rule's schedule, each time it is created."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include "zq3d_block_cut.h"
#include <cstdio>
#include <cstdlib>
using namespace zq3d;
static BlockCut rule(int W, int H, int D, double* us) {
    return block_best_cut(W, H, D, 40, 512, us, block_cost_weighted);
}
int main(int argc, char** argv) {
    double us = 0.0;
    if (argc == 4) {
        const BlockCut c = rule(atoi(argv[1]), atoi(argv[2]), atoi(argv[3]), &us);
        int lg = 0;
        while ((1 << lg) < c.lx) lg++;
        return std::printf("%d %d\n", c.K, -(10000 * lg + 100 * c.ty + c.tz)), 0;
    }
    for (int W : {1, 2, 5, 16, 33, 64, 129})
        for (int H : {1, 3, 8, 24, 65, 129})
            for (int D : {1, 2, 9, 32, 100, 129}) {
                const BlockCut c = rule(W, H, D, &us);
                if (!c.nx || c.K < 1 || c.K > 4 || block_threads(c) > 512 || block_lds_bytes(c) > 64 * 1024)
                    return std::printf("%d %d %d: no cut\n", W, H, D), 1;
                for (int lx = 2; lx <= 64; lx *= 2)
                    for (int ty : {4, 7, 10, 16, 32})
                        for (int tz = 1; tz <= 8; tz++)
                            for (int K = 1; K <= 4; K++) {
                                const BlockCut o = block_cut(W, H, D, lx, ty, tz, K);
                                if (!o.nx || block_threads(o) > 512 || (!o.halo && K > 1)) continue;
                                const int k = o.halo ? K : 40;
                                if (block_cost_weighted(o, k) / k < us)
                                    return std::printf("%d %d %d: %d %d %d %d\n", W, H, D, lx, ty, tz, K), 1;
                            }
            }
    std::printf("ok\n");
    return 0;
}
"""


@pytest.fixture
def rule(tmp_path):
    src = tmp_path / "rule.cpp"
    src.write_text(SRC)
    exe = str(tmp_path / "rule")
    inc = os.path.join(ROOT, "zq_smokesimulation_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", inc, str(src), "-o", exe], check=True)
    return lambda *dims: subprocess.run([exe, *map(str, dims)], capture_output=True, text=True).stdout.strip()


def test_every_grid_gets_its_cheapest_boxes(rule):
    assert rule() == "ok"


@pytest.mark.gpu
@pytest.mark.parametrize("dims,sub", [((64, 64, 64), 2), ((80, 80, 80), 1), ((24, 40, 12), 1), ((96, 80, 64), 8)],
                         ids=str)
def test_a_simulation_takes_the_rules_schedule(rule, dims, sub):
    from zq_smokesimulation_amd.sim import SmokeSim3D
    want = tuple(map(int, rule(*[n // sub for n in dims]).split()))
    for _ in range(2):
        print("coarse schedule", dims, sub, want, flush=True)
        sim = SmokeSim3D(*dims, sub_size=sub)
        try:
            assert sim.coarse_sweep() == want
        finally:
            sim.close()
