"""Tile numbers of the register sweeps on grids that are millions of cells long: the division by the number of
tiles along an axis (csrc/zq3d_quad_cut.h), compiled with g++, is exact beyond 2^16 tiles, so every tile of a
launch is somebody's; on the GPU, boxes of four lanes and marching tiles of one wave on long thin grids
give the oracle's bits."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include "zq3d_block_cut.h"
#include <cstdio>
#include <random>
using namespace zq3d;
int main() {
    std::mt19937 rng(3);
    const int edge[] = {1, 2, 3, 60, 65535, 65536, 65537, 74777, 107143, 178572, (1 << 30) - 1, 1 << 30, 0x7fffffff};
    for (int k = 0; k < 4000000; k++) {
        const int n = k % 3 ? 1 + (int)(rng() % (1u << (1 + rng() % 31))) % 0x7fffffff : edge[rng() % 13];
        int i = k % 2 ? (int)(rng() >> 1) : (int)((rng() >> 1) / n * (long long)n % 0x7fffffff);
        if (k % 5 == 0 && i) i--;
        if (quad_div(i, quad_magic(n), n) != i / n) return std::printf("%d / %d\n", i, n), 1;
    }
    // every tile of the cuts that long grids get
    for (int W : {299111, 892887, 8388607, 12000000, 20000000, 60000000}) {
        const QuadCut q = quad_best_cut(W, 2, 2, 2, 2, 16);
        const BlockCut small = block_cut(W, 2, 2, 4, 1, 1, 1), best = block_best_cut(W, 2, 2, 40, BLOCK_THREADS);
        const int n[3][3] = {{q.nx, q.ny, q.nz}, {small.nx, small.ny, small.nz}, {best.nx, best.ny, best.nz}};
        const unsigned m[3][2] = {{q.mnx, q.mny}, {small.mnx, small.mny}, {best.mnx, best.mny}};
        for (int c = 0; c < 3; c++)
            for (int t = 0; t < n[c][0] * n[c][1] * n[c][2]; t++) {
                const int r = quad_div(t, m[c][0], n[c][0]), z = quad_div(r, m[c][1], n[c][1]);
                if (r != t / n[c][0] || z != r / n[c][1]) return std::printf("W %d cut %d tile %d\n", W, c, t), 1;
            }
    }
    std::printf("ok\n");
    return 0;
}
"""


def test_the_division_is_exact(tmp_path):
    src = tmp_path / "div.cpp"
    src.write_text(SRC)
    exe = str(tmp_path / "div")
    inc = os.path.join(ROOT, "zq_smokesimulation_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", "-I", inc, str(src), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("dims,shapes", [((410444, 2, 3), [(-120101, 1), (0, 0)]), ((23, 2, 4), [(-120101, 1)]),
                                         ((8700025, 2, 2), [(-1202, 2)])], ids=str)
def test_long_grids_keep_every_tile(dims, shapes):
    import zq_oracle as O
    import zq_smokesimulation_amd as z
    from util import faces, occupancy
    W, H, D = dims
    print("long grid", dims, flush=True)
    rng = np.random.default_rng(2)
    u, v, w = faces(rng, W, H, D)
    occ = occupancy(rng, W, H, D, 0.1, shell=False)
    ref = [a.copy() for a in (u, v, w)]
    O.project(*ref, occ, O.ALL_FACES, 0.0, 1.7, 3)
    sim = z.SmokeSim3D(W, H, D, sor_open_mask=O.ALL_FACES, sor_closed_mean=0, sor_omega=1.7, sor_iters=3)
    try:
        for shape in shapes:
            sim.set_sor_shape(*shape)
            sim.set_state(u=u, v=v, w=w, occ=occ)
            sim.project()
            g = sim.get_state()
            for name, a in zip("uvw", ref):
                assert np.array_equal(g[name].view(np.uint32), a.view(np.uint32)), (shape, name)
    finally:
        sim.close()
