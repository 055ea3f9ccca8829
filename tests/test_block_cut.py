"""How the block sweeps cut a grid into boxes (csrc/zq3d_block_cut.h), compiled with g++ and checked on the
CPU: every cell has exactly one owner, a box covers its own cells plus 2K cells beside every other box,
boxes begin at even cells, and the threads and LDS of a chosen cut fit a workgroup."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include "zq3d_block_cut.h"
#include <cstdio>
using namespace zq3d;
static int axis(const BlockCut& c, int N, int n, int R) {
    int at = 0;
    for (int i = 0; i < n; i++) {
        const int b = block_begin(i, n, N, R, c.halo), e = block_begin(i + 1, n, N, R, c.halo);
        const int lo = b - (i ? c.halo : 0), hi = lo + R;
        if (b != at || e <= b || lo < 0 || lo % 2) return 1;
        if (i && b - lo < 2 * c.K) return 2;
        if (i + 1 < n ? hi - e < 2 * c.K : hi < N) return 3;
        at = e;
    }
    return at == N ? 0 : 4;
}
static int check(int W, int H, int D, const BlockCut& c) {
    if (!c.nx) return 0;
    const int a = axis(c, quad_stride(W), c.nx, BLOCK_X * c.lx), b = axis(c, H, c.ny, BLOCK_Y * c.ty),
              e = axis(c, D, c.nz, BLOCK_Z * c.tz);
    const bool fits = block_threads(c) <= BLOCK_THREADS && block_lds_bytes(c) <= 160 * 1024 && 64 % c.lx == 0;
    bool div = true;
    for (int i = 0; i < 1024; i++) div = div && quad_div(i, c.mty) == i / c.ty;
    for (int i = 0; i < c.nx * c.ny * c.nz; i++) {
        const int r = quad_div(i, c.mnx);
        div = div && r == i / c.nx && quad_div(r, c.mny) == r / c.ny;
    }
    if (a || b || e || !fits || !div)
        return std::printf("%dx%dx%d lx %d ty %d tz %d K %d: %d %d %d %d %d\n", W, H, D, c.lx, c.ty, c.tz, c.K, a, b, e,
                           fits, div), 1;
    return 0;
}
int main() {
    const int ds[] = {1, 2, 3, 5, 8, 15, 16, 17, 24, 33, 64, 100, 129};
    for (int W : ds)
        for (int H : ds)
            for (int D : ds) {
                for (int lx = 2; lx <= 64; lx *= 2)
                    for (int ty : {1, 3, 4, 8, 12, 32})
                        for (int tz : {1, 2, 3, 4, 8})
                            for (int K = 1; K <= 4; K++)
                                if (check(W, H, D, block_cut(W, H, D, lx, ty, tz, K))) return 1;
                const BlockCut best = block_best_cut(W, H, D, 40, BLOCK_THREADS);
                if (!best.nx || check(W, H, D, best)) return std::printf("best %d %d %d\n", W, H, D), 1;
            }
    std::printf("ok\n");
    return 0;
}
"""


def test_every_cell_has_one_owner_and_its_halo(tmp_path):
    src = tmp_path / "cut.cpp"
    src.write_text(SRC)
    exe = str(tmp_path / "cut")
    inc = os.path.join(ROOT, "zq_smokesimulation_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", inc, str(src), "-o", exe], check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "ok", out.stdout
