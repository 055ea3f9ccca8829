// zq3d_block_cut.h -- how the block sweeps (zq3d_sor_block.h) cut a grid into boxes: plain C++ that the
// kernels, their launchers and a host test share.
#pragma once

#include "zq3d_quad_cut.h"

namespace zq3d {

// Cells a thread holds along x, y and z.
constexpr int BLOCK_X = 2, BLOCK_Y = 2, BLOCK_Z = 4;
constexpr int BLOCK_THREADS = 1024;
constexpr int BLOCK_MOST = 2000;  // iterations a launch of a grid that is one box

struct BlockCut {
    int lx, ty, tz;  // threads along x (a power of two up to 64), y and z
    int K;           // iterations a launch
    int halo;        // cells recomputed beside another box: 2K, 0 for a single box
    int nx, ny, nz;  // boxes; 0: no such cut
    unsigned mty, mnx, mny;  // quad_magic of ty, nx, ny
};

ZQ_HD inline int block_threads(const BlockCut& c) { return c.lx * c.ty * c.tz; }
// two buffers of a thread's values of one colour (row 0, row 1) and their end planes, and a slot of zeros
inline int block_lds_bytes(const BlockCut& c) { return 32 + 2 * (block_threads(c) + 1) * 48; }

// boxes of R cells with halo h that cover N cells; the first cell box i owns (the end for i == n)
ZQ_HD inline int block_axis(int N, int R, int h) {
    if (N <= R) return 1;
    if (R <= 2 * h) return 0;
    const int left = N - 2 * (R - h), mid = R - 2 * h;
    return 2 + (left > 0 ? (left + mid - 1) / mid : 0);
}
ZQ_HD inline int block_begin(int i, int n, int N, int R, int h) {
    return i == 0 ? 0 : i >= n ? N : R - h + (i - 1) * (R - 2 * h);
}

// The cut of a W x H x D grid into boxes of lx x ty x tz threads, K iterations a launch.
inline BlockCut block_cut(int W, int H, int D, int lx, int ty, int tz, int K) {
    BlockCut c{};
    c.lx = lx, c.ty = ty, c.tz = tz, c.K = K;
    const int S = quad_stride(W);
    const bool one = S <= BLOCK_X * lx && H <= BLOCK_Y * ty && D <= BLOCK_Z * tz;
    c.halo = one ? 0 : 2 * K;
    c.nx = block_axis(S, BLOCK_X * lx, c.halo);
    c.ny = block_axis(H, BLOCK_Y * ty, c.halo);
    c.nz = block_axis(D, BLOCK_Z * tz, c.halo);
    if (!c.nx || !c.ny || !c.nz || block_threads(c) > BLOCK_THREADS) c.nx = c.ny = c.nz = 0;
    c.mty = quad_magic(ty), c.mnx = quad_magic(c.nx), c.mny = quad_magic(c.ny);
    return c;
}

// Predicted microseconds of a launch of k iterations: boundary, loads and store, then 2k single-colour
// sweeps that cost their issue time per wave a SIMD runs.  A CU holds 16 waves of these kernels; boxes
// beyond what the CUs hold at once run in further rounds.  (Fitted to 2800 launches on 8 grids from
// 32^3 to 128^3.  On the 24 grids of profiles/sweep_shapes.txt where boxes are chosen, they are within 5.2 %
// of the fastest cut.)
inline double block_cost(const BlockCut& c, int k) {
    const int waves = (block_threads(c) + 63) / 64, boxes = c.nx * c.ny * c.nz;
    const int per = (boxes + 255) / 256, holds = std::max(1, 16 / waves);
    const int rounds = (per + holds - 1) / holds;
    const double simd = std::max(1.0, waves * std::min(per, holds) / 4.0);
    return 3.65 + rounds * (0.96 + 0.35 * simd + 2.0 * k * 0.26 * simd);
}

// The same of the weighted operator (the coarse grid's sweeps), whose weights fill the registers: a CU holds 8
// waves, and all boxes' loads (six arrays of short rows) count, 0.67 ps a cell and 8.7 a row of the box.
// (Fitted to 3700 launches on 17 grids from 8^3 to 256^3, profiles/coarse_box_shapes.txt.)
inline double block_cost_weighted(const BlockCut& c, int k) {
    const int waves = (block_threads(c) + 63) / 64, boxes = c.nx * c.ny * c.nz;
    const int per = (boxes + 255) / 256, holds = std::max(1, 8 / waves);
    const int rounds = (per + holds - 1) / holds;
    const double simd = std::max(1.0, waves * std::min(per, holds) / 4.0);
    const double rows = (double)boxes * (BLOCK_Y * c.ty) * (BLOCK_Z * c.tz);
    return 2.0 + rounds * (2.2 + 0.55 * simd + 2.0 * k * (0.26 + 0.2 * simd)) +
           1e-6 * rows * (0.67 * BLOCK_X * c.lx + 8.7);
}

// The cheapest cut per iteration of at most `most` threads (iters: of a pass; a single box runs all of
// them in one launch).
inline BlockCut block_best_cut(int W, int H, int D, int iters, int most, double* cost = nullptr,
                               double (*price)(const BlockCut&, int) = block_cost) {
    static const int tys[] = {4, 5, 6, 7, 8, 9, 10, 12, 14, 16, 20, 24, 32};
    static const int tzs[] = {1, 2, 3, 4, 5, 6, 7, 8};
    BlockCut best{};
    double least = 0.0;
    for (int lx = 2; lx <= 64; lx *= 2)
        for (int ty : tys)
            for (int tz : tzs)
                for (int K = 1; K <= 4; K++) {
                    const BlockCut c = block_cut(W, H, D, lx, ty, tz, K);
                    if (!c.nx || (c.halo == 0 && K > 1) || block_threads(c) > most) continue;
                    const int k = c.halo ? K : std::max(iters, 1);
                    const double t = price(c, k) / k;
                    if (best.nx == 0 || t < least) {
                        best = c;
                        least = t;
                    }
                }
    if (cost) *cost = least;
    return best;
}

}  // namespace zq3d
