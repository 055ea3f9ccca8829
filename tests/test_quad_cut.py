"""How the quad-layout sweeps cut a grid into tiles (csrc/zq3d_quad_cut.h), compiled with g++ and checked
on the CPU: over shapes, waves and planes, every cell has exactly one owner, every tile covers its own
cells plus the 2K cells of halo on each side that borders another tile, chunk walks begin on even planes,
the multiply-shift divisions are exact, and the LDS of the chosen cuts fits a workgroup."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include "zq3d_quad_cut.h"
#include <cstdio>
#include <cstdlib>
#include <vector>
using namespace zq3d;
static int fail(const char* what, int W, int H, int D, int K, int cx, int nw, int zc) {
    std::printf("%s: %dx%dx%d K %d cx %d nw %d zc %d\n", what, W, H, D, K, cx, nw, zc);
    return 1;
}
static int check(int W, int H, int D, int K, int cx, const QuadCut& c) {
    const int S = quad_stride(W), J = 2 * K, hl = quad_halo_lanes(K, cx), nw = c.nw, zc = c.zc;
    if (S % 4 || S < W || S - W > 3) return fail("stride", W, H, D, K, cx, nw, zc);
    if (c.rows != c.nw * c.g * QUAD_R || c.g * c.lx > 64 || zc % 2) return fail("shape", W, H, D, K, cx, nw, zc);
    if (c.g > 1 && !c.mask && S == W) return fail("unmasked group edge", W, H, D, K, cx, nw, zc);
    // the LDS of a tile: row groups plus one zero group on either side
    if ((c.nw * c.g + 2) * c.lx * (cx / 2) > quad_edge_floats(cx, 64 * c.nw))
        return fail("lds", W, H, D, K, cx, nw, zc);
    for (int b = 0; b < c.nx; b++) {
        const int o0 = quad_x_begin(c, K, cx, b, S), o1 = quad_x_begin(c, K, cx, b + 1, S);
        const int x0 = o0 - (b ? cx * hl : 0), x1 = x0 + cx * c.lx;
        if (o0 % cx || o1 <= o0 || x0 < 0 || (b && o0 - x0 < J)) return fail("x low side", W, H, D, K, cx, nw, zc);
        if (b + 1 < c.nx ? x1 - o1 < J : x1 < S) return fail("x high side", W, H, D, K, cx, nw, zc);
    }
    for (int b = 0; b < c.ny; b++) {
        const int o0 = quad_y_begin(c, K, b, H), o1 = quad_y_begin(c, K, b + 1, H);
        const int y0 = o0 - (b ? J : 0), y1 = y0 + c.rows;
        if (y0 % 2 || o1 <= o0 || y0 < 0) return fail("y low side", W, H, D, K, cx, nw, zc);
        if (b + 1 < c.ny ? y1 - o1 < J : y1 < H) return fail("y high side", W, H, D, K, cx, nw, zc);
    }
    for (int b = 0; b < c.nz; b++) {
        const int z0 = quad_z_begin(c, K, b, D), z1 = quad_z_begin(c, K, b + 1, D);
        const int t = b ? z0 - J + 1 : 0;
        if (z1 <= z0 || t < 0 || t % 2) return fail("z", W, H, D, K, cx, nw, zc);
    }
    if (quad_z_begin(c, K, 0, D) != 0 || quad_z_begin(c, K, c.nz, D) != D || quad_x_begin(c, K, cx, c.nx, S) != S ||
        quad_y_begin(c, K, c.ny, H) != H) return fail("cover", W, H, D, K, cx, nw, zc);
    for (int l = 0; l < 64; l++)
        if (quad_div(l, c.mlx) != l / c.lx) return fail("lane division", W, H, D, K, cx, nw, zc);
    const long long tiles = (long long)c.nx * c.ny * c.nz;
    for (long long t = 0; t < tiles; t += 1 + tiles / 997)
        if (quad_div((int)t, c.mnx) != t / c.nx || quad_div((int)(t / c.nx), c.mny) != t / c.nx / c.ny)
            return fail("tile division", W, H, D, K, cx, nw, zc);
    return 0;
}
int main() {
    unsigned r = 7;
    auto rnd = [&](int n) { r = r * 1664525u + 1013904223u; return (int)((r >> 8) % (unsigned)n); };
    int bad = 0, seen = 0;
    for (int i = 0; i < 20000 && !bad; i++) {
        const int top = i % 3 == 0 ? 12 : i % 3 == 1 ? 80 : 700;
        const int W = 2 + rnd(top), H = 2 + rnd(top), D = 2 + rnd(top), K = 1 + rnd(2), cx = K == 2 && rnd(2) ? 4 : 2;
        const int nw = 1 + rnd(cx == 4 ? 8 : 16), zc = 2 + 2 * rnd(32);
        const QuadCut c = quad_cut(W, H, D, K, cx, nw, zc);
        if (c.ny == 0) continue;
        seen++;
        bad += check(W, H, D, K, cx, c);
        if (i % 10 == 0) {
            const QuadCut b = quad_best_cut(W, H, D, K, cx, cx == 4 ? 8 : 16);
            if (b.nw < 1 || b.ny < 1) bad += fail("no cut", W, H, D, K, cx, nw, zc);
            else bad += check(W, H, D, K, cx, b);
        }
    }
    // extreme grids: a long row, a long column, a flat one
    const int ext[][3] = {{100000, 2, 2}, {2, 100000, 2}, {2, 2, 100000}, {20000, 20000, 2}, {1000, 1000, 1000}};
    for (auto& e : ext)
        for (int cx = 2; cx <= 4; cx += 2) {
            const QuadCut b = quad_best_cut(e[0], e[1], e[2], 2, cx, cx == 4 ? 8 : 16);
            if (b.nw < 1 || b.ny < 1) bad += fail("no cut", e[0], e[1], e[2], 2, cx, 0, 0);
            else bad += check(e[0], e[1], e[2], 2, cx, b);
        }
    if (4 * quad_lds_floats(2, 2, 1024) > 160 * 1024 || 4 * quad_lds_floats(2, 4, 512) > 160 * 1024) bad++;
    std::printf("%d cuts checked, %d bad\n", seen, bad);
    return bad || seen < 5000;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("quad")
    src = d / "cut.cpp"
    src.write_text(SRC)
    exe = d / "cut"
    subprocess.check_call(["g++", "-O1", "-std=c++17", "-Wall", "-I",
                           os.path.join(ROOT, "zq_smokesimulation_amd", "csrc"), "-o", str(exe), str(src)])
    return str(exe)


def test_every_cut_covers_the_grid_once_with_its_halos(program):
    r = subprocess.run([program], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
