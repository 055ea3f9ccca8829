// zq3d_quad_cut.h -- how the quad-layout sweeps (zq3d_sor_quad.h) cut a grid into tiles: plain C++ that
// the kernels, their launchers and a host test share.
#pragma once

#include <algorithm>
#include <cstdint>

#if defined(__HIPCC__)
#define ZQ_HD __host__ __device__
#else
#define ZQ_HD
#endif

namespace zq3d {

// Rows of the quad layout: W rounded up to 4 cells, so that a row starts on 16 bytes.
ZQ_HD inline int quad_stride(int W) { return (W + 3) & ~3; }

constexpr int QUAD_R = 2;  // rows a thread holds

struct QuadCut {
    int lx, g, mask;  // lanes per row; row groups per wave; 1: a group's edge lanes need their outer neighbour masked
    int nw;           // waves per workgroup
    int rows;         // rows of a tile (halo included)
    int nx, ny, nz;   // tiles
    int zc;           // planes of a chunk after the first (even; the first has zc + 2K - 1)
    unsigned mlx, mnx, mny;  // quad_magic of lx, nx, ny
};

// i / n = floor(i * ceil(2^32 / n) / 2^32) while i * n < 2^32 (a tile's prologue is on the critical path
// of small grids, and the compiler's division sequence is long); 0 stands for n = 1
ZQ_HD inline unsigned quad_magic(int n) { return n > 1 ? (unsigned)(((1ull << 32) + n - 1) / n) : 0u; }
ZQ_HD inline int quad_div(int i, unsigned magic) { return magic ? (int)(((uint64_t)(unsigned)i * magic) >> 32) : i; }
// the same for any 0 <= i, n < 2^31 (tile numbers: a grid of millions of cells along one axis has more than
// 2^16 tiles there): the estimate is at most one too large
ZQ_HD inline int quad_div(int i, unsigned magic, int n) {
    const int q = quad_div(i, magic);
    return q - ((unsigned)q * (unsigned)n > (unsigned)i ? 1 : 0);
}

// whether the cut has tiles whose numbers quad_div needs the divisor for
ZQ_HD inline bool quad_far(const QuadCut& c) {
    return (long long)c.nx * c.ny * c.nz * (c.nx > c.ny ? c.nx : c.ny) >= 1ll << 32;
}

// LDS floats of a tile of at most nt threads: the table of reciprocals, then two buffers x 2K arrays x
// first / last row of every row group (and a zero group on either side, 128 lanes at most), cx/2
// values a thread.  A block's stride is fixed by nt, so that the accesses have constant offsets.
ZQ_HD constexpr int quad_edge_floats(int cx, int nt) { return (nt + 128) * (cx / 2); }
ZQ_HD constexpr int quad_lds_floats(int K, int cx, int nt) { return 8 + 2 * (2 * K) * 2 * quad_edge_floats(cx, nt); }

// lanes of halo beside another tile along x: 2K cells, one per single-colour sweep
ZQ_HD constexpr int quad_halo_lanes(int K, int cx) { return (2 * K + cx - 1) / cx; }

// first owned cell of tile column bx (padding included in the last), first owned row of tile row by,
// first owned plane of chunk bz; a tile owns up to the next one's first
ZQ_HD inline int quad_x_begin(const QuadCut& c, int K, int cx, int bx, int S) {
    const int hl = quad_halo_lanes(K, cx);
    return bx == 0 ? 0 : bx == c.nx ? S : cx * (c.lx - hl + (bx - 1) * (c.lx - 2 * hl));
}
ZQ_HD inline int quad_y_begin(const QuadCut& c, int K, int by, int H) {
    return by == 0 ? 0 : by == c.ny ? H : c.rows - 2 * K + (by - 1) * (c.rows - 4 * K);
}
ZQ_HD inline int quad_z_begin(const QuadCut& c, int K, int bz, int D) {
    const int z = bz == 0 ? 0 : c.zc + 2 * K - 1 + (bz - 1) * c.zc;
    return bz == c.nz || z > D ? D : z;
}

// chunks of zc planes that D planes make (the first holds 2K - 1 more)
ZQ_HD inline int quad_chunks(int D, int K, int zc) {
    const int first = zc + 2 * K - 1;
    return 1 + (D > first ? (D - first + zc - 1) / zc : 0);
}

// The cut of a W x H x D grid for K iterations a pass, cx cells a lane, nw waves and zc planes (even).
// ny == 0: a tile of these waves would own no row.
inline QuadCut quad_cut(int W, int H, int D, int K, int cx, int nw, int zc) {
    QuadCut c{};
    const int J = 2 * K, lanes = quad_stride(W) / cx, hl = quad_halo_lanes(K, cx);
    if (lanes <= 64) {
        c.lx = lanes;
        c.g = 64 / lanes;
        c.nx = 1;
        // with several groups a wave, a group's outer neighbours are another row's cells; padding cells
        // (zero) separate them unless the rows have none
        c.mask = c.g > 1 && W % 4 == 0;
    } else {
        c.lx = 64;
        c.g = 1;
        const int left = lanes - 2 * (64 - hl), mid = 64 - 2 * hl;
        c.nx = 2 + (left > 0 ? (left + mid - 1) / mid : 0);
    }
    const int per = c.g * QUAD_R;
    c.nw = std::min(nw, (H + per - 1) / per);
    c.rows = c.nw * per;
    if (c.rows >= H) c.ny = 1;
    else if (c.rows <= 2 * J) c.ny = 0;
    else {
        const int left = H - 2 * (c.rows - J), mid = c.rows - 2 * J;
        c.ny = 2 + (left > 0 ? (left + mid - 1) / mid : 0);
    }
    c.zc = zc;
    c.nz = quad_chunks(D, K, zc);
    c.mlx = quad_magic(c.lx);
    c.mnx = quad_magic(c.nx);
    c.mny = quad_magic(std::max(c.ny, 1));
    return c;
}

// Predicted microseconds of a plane step: a latency and the issue time per wave a SIMD runs.
inline double quad_step_us(int K, int cx, int nw) {
    const double issue = (cx / 2) * (K == 2 ? 0.21 : 0.12);
    return 0.24 + issue * std::max(1.0, nw / 4.0);
}

// Predicted microseconds of one launch: a fixed cost, then every workgroup's steps (CUs beyond one round of
// workgroups share them).
inline double quad_cost(const QuadCut& c, int K, int cx) {
    const double tiles = (double)c.nx * c.ny * c.nz, steps = c.zc + 4 * K - 2;
    const double rounds = std::max(1.0, tiles / 256.0);
    // beyond one round the last one may be nearly empty
    const double full = tiles <= 256.0 ? 1.0 : 0.5 * (rounds + (double)((int)((tiles + 255.0) / 256.0)));
    return 4.0 + steps * quad_step_us(K, cx, c.nw) * full;
}

// The cheapest cut of up to `most` waves by quad_cost.
inline QuadCut quad_best_cut(int W, int H, int D, int K, int cx, int most, double* cost = nullptr) {
    static const int nws[] = {2, 4, 5, 6, 8, 10, 12, 14, 16};
    static const int zcs[] = {2, 4, 6, 8, 10, 12, 14, 16, 20, 24, 28, 32, 40, 48, 64};
    QuadCut best{};
    double least = 0.0;
    for (int nw : nws) {
        if (nw > most) break;
        for (int zc : zcs) {
            const QuadCut c = quad_cut(W, H, D, K, cx, nw, zc);
            if (c.ny == 0) break;
            const double t = quad_cost(c, K, cx);
            if (best.nw == 0 || t < least) {
                best = c;
                least = t;
            }
            if (c.nz == 1) break;
        }
    }
    if (cost) *cost = least;
    return best;
}

}  // namespace zq3d
