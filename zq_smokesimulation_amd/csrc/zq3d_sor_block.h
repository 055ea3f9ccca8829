// zq3d_sor_block.h -- K red-black SOR iterations of one box of cells, the whole box in registers; for
// grids so small that a launch is all latency, and for the face-weighted operator of the coarse grid.
//
// Storage: the quad layout (zq3d_sor_quad.h): cell (x, y, z) at (z*H + y)*S + x, no ghosts; cells W..S-1
// have a diagonal of 0 and p = 0.  A thread holds 2 x 2 x 4 cells (x pair, two rows, four planes) with
// their right-hand sides and diagonals, so in a row of the pair one cell is of each colour and which one
// is fixed at compile time (boxes begin at even cells).  x neighbours come from the next lane (DPP), y
// and z neighbours of other threads through LDS: after a single-colour sweep every thread publishes the
// eight values it has written, into one of two buffers, so one barrier a sweep suffices.  A cell's sum,
// order and rounding are those of a single-colour sweep: the result is the same bits.
//
// A box carries 2K cells of halo on each side that borders another box; they are recomputed and
// dropped.  A grid that fits one box has no halo, and all iterations run in one launch.
//
// What bounds it: nothing but latency: the launch boundary (1.5 us on the device), one round trip for all
// loads at once, then 2K sweeps of 8 updates a thread (0.2 us of issue at one wave a SIMD, as much again
// for LDS and the barrier).  The marching tiles (zq3d_sor_quad.h) pay a step for each of their planes
// and 4K - 2 more for their pipeline; they win where a box's halo costs more than that.  Measured
// figures stand at quad_plan (kernels_project.hip) and at the coarse sweeps (kernels_coarse.hip).
#pragma once

#include "zq3d_block_cut.h"
#include "zq3d_device.h"
#include "zq3d_sor_split.h"
#include "zq3d_stencils.h"

namespace zq3d {

// Weights of the low x, y, z faces of every cell (quad layout), 1/diagonal (0: not updated).
struct BlockWeights {
    const float *x, *y, *z, *inv;
};

// WT: the weighted operator (sum over the sides of face weight * p), else the plain one with n = 4 * count.
template <bool WT>
struct BlockTile {
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    static constexpr int NY = BLOCK_Y, NZ = BLOCK_Z;

    float P[NY][NZ][2], B[NY][NZ][2], C[NY][NZ][2];  // pressure, right-hand side, 1/diagonal
    // face weights: low sides, and the high side of the last cell along each axis
    float wx[WT ? NY : 1][NZ][3], wy[WT ? NY + 1 : 1][NZ][2], wz[WT ? NY : 1][NZ + 1][2];
    bool lo, hi;       // first / last lane of a row
    float omega, omw;
    f4* rows;          // [buffer][row][slots]: the threads' published values
    f2* ends;          // [buffer][first, last plane][slots]
    int slots, me, up, dn, be, ab;  // this thread's slot and its neighbours' (rows above / below, planes below / above)

    static __device__ __forceinline__ float shr1(float x) {  // the left lane's value (0 for lane 0)
        return __builtin_bit_cast(
            float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x138, 0xf, 0xf, true));
    }
    static __device__ __forceinline__ float shl1(float x) {  // the right lane's value (0 for lane 63)
        return __builtin_bit_cast(
            float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x130, 0xf, 0xf, true));
    }

    // publish colour c's values into buffer buf
    template <int c>
    __device__ __forceinline__ void share(int buf) {
        float v[NY][NZ];
#pragma unroll
        for (int r = 0; r < NY; r++)
#pragma unroll
            for (int z = 0; z < NZ; z++) v[r][z] = P[r][z][(r + z + c) & 1];
        f4* q = rows + 2 * buf * slots + me;
        q[0] = f4{v[0][0], v[0][1], v[0][2], v[0][3]};
        q[slots] = f4{v[1][0], v[1][1], v[1][2], v[1][3]};
        f2* e = ends + 2 * buf * slots + me;
        e[0] = f2{v[0][0], v[1][0]};
        e[slots] = f2{v[0][NZ - 1], v[1][NZ - 1]};
    }

    // the sweep of colour c, its neighbours' values in buffer buf
    template <int c>
    __device__ __forceinline__ void sweep(int buf) {
        const f4 u = rows[(2 * buf + 1) * slots + up], d = rows[2 * buf * slots + dn];
        const f2 b = ends[(2 * buf + 1) * slots + be], a = ends[2 * buf * slots + ab];
#pragma unroll
        for (int r = 0; r < NY; r++)
#pragma unroll
            for (int z = 0; z < NZ; z++) {
                const int e = (r + z + c) & 1;
                // (every lane moves its value: a lane masked off would have none to give)
                const float next = e ? shl1(P[r][z][0]) : shr1(P[r][z][1]);
                const float side = (e ? hi : lo) ? 0.0f : next;
                const float xm = e ? P[r][z][0] : side, xp = e ? side : P[r][z][1];
                const float ym = r ? P[0][z][e] : u[z], yp = r ? d[z] : P[1][z][e];
                const float zm = z ? P[r][z ? z - 1 : 0][e] : b[r];
                const float zp = z + 1 < NZ ? P[r][z + 1 < NZ ? z + 1 : z][e] : a[r];
                float s;
                if constexpr (WT)
                    s = wx[r][z][e] * xm + wx[r][z][e + 1] * xp + wy[r][z][e] * ym + wy[r + 1][z][e] * yp +
                        wz[r][z][e] * zm + wz[r][z + 1][e] * zp;
                else
                    s = xm + xp + ym + yp + zm + zp;
                const float own = P[r][z][e], pg = (s - B[r][z][e]) * C[r][z][e];
                const float upd = omw * own + omega * pg;
                P[r][z][e] = C[r][z][e] != 0.0f ? upd : own;
            }
    }
};

// Box (bx, by, bz) of the cut, `iters` iterations (c.K of them unless the grid is one box); src ==
// nullptr: the source is all zeros.  b: right-hand side, m: the mean subtracted from it.  n: counts of
// the plain operator; w: of the weighted one.  lds: block_lds_bytes(c) bytes.
template <bool WT>
__device__ __forceinline__ void sor_block_tile(const uint8_t* n, const BlockWeights& w, const float* b, float m,
                                               const float* src, float* dst, const Dims& d, const BlockCut& c, int bx,
                                               int by, int bz, int iters, float omega, float omw, float* lds) {
    using T = BlockTile<WT>;
    typedef typename T::f2 f2;
    T q;
    const int S = quad_stride(d.W), tid = threadIdx.x;
    const int ix = tid & (c.lx - 1), row = tid / c.lx;  // (lx is a power of two)
    const int iz = quad_div(row, c.mty), iy = row - iz * c.ty;
    const bool on = iz < c.tz;
    const int rx = BLOCK_X * c.lx, ry = BLOCK_Y * c.ty, rz = BLOCK_Z * c.tz;  // cells of a box
    const int xo0 = block_begin(bx, c.nx, S, rx, c.halo), xo1 = block_begin(bx + 1, c.nx, S, rx, c.halo);
    const int yo0 = block_begin(by, c.ny, d.H, ry, c.halo), yo1 = block_begin(by + 1, c.ny, d.H, ry, c.halo);
    const int zo0 = block_begin(bz, c.nz, d.D, rz, c.halo), zo1 = block_begin(bz + 1, c.nz, d.D, rz, c.halo);
    const int x = xo0 - (bx ? c.halo : 0) + BLOCK_X * ix;
    const int y0 = yo0 - (by ? c.halo : 0) + BLOCK_Y * iy;
    const int z0 = zo0 - (bz ? c.halo : 0) + BLOCK_Z * iz;
    const uint32_t plane = (uint32_t)S * (uint32_t)d.H, cells = plane * (uint32_t)d.D;
    const bool xin = on && x < S;  // (x >= 0: a box that is not the first begins at least its halo in)
    const uint32_t o0 = (uint32_t)z0 * plane + (uint32_t)y0 * (uint32_t)S + (uint32_t)x;
    // cell index of the pair (r, z), SPLIT_NONE/4 or more where there is none
    auto at = [&](int r, int z) -> uint32_t {
        return xin && y0 + r < d.H && z0 + z < d.D ? o0 + (uint32_t)z * plane + (uint32_t)(r * S) : SPLIT_NONE >> 2;
    };
    auto pair = [&](__amdgpu_buffer_rsrc_t rs, uint32_t o, float (&v)[2]) {
        const f2 t = __builtin_bit_cast(f2, __builtin_amdgcn_raw_buffer_load_b64(rs, (int)(4u * o), 0, 0));
        v[0] = t.x, v[1] = t.y;
    };
    const __amdgpu_buffer_rsrc_t rp = split_buf(src, src ? 4u * cells : 0u), rb = split_buf(b, 4u * cells);
    unsigned nn[T::NY][T::NZ];
    const __amdgpu_buffer_rsrc_t rn = split_buf(WT ? (const void*)w.inv : (const void*)n, WT ? 4u * cells : cells);
#pragma unroll
    for (int r = 0; r < T::NY; r++)
#pragma unroll
        for (int z = 0; z < T::NZ; z++) {
            const uint32_t o = at(r, z);
            if constexpr (WT) pair(rn, o, q.C[r][z]);
            else nn[r][z] = (unsigned)__builtin_amdgcn_raw_buffer_load_b16(rn, (int)o, 0, 0);
            pair(rp, o, q.P[r][z]);
            pair(rb, o, q.B[r][z]);
        }
    if constexpr (WT) {
        const __amdgpu_buffer_rsrc_t bwx = split_buf(w.x, 4u * cells), bwy = split_buf(w.y, 4u * cells),
                                     bwz = split_buf(w.z, 4u * cells);
#pragma unroll
        for (int r = 0; r <= T::NY; r++)
#pragma unroll
            for (int z = 0; z <= T::NZ; z++) {
                const uint32_t o = at(r, z);
                if (r < T::NY && z < T::NZ) {
                    float t[2];
                    pair(bwx, o, t);
                    q.wx[r][z][0] = t[0], q.wx[r][z][1] = t[1];
                }
                if (z < T::NZ) pair(bwy, o, q.wy[r][z]);
                if (r < T::NY) pair(bwz, o, q.wz[r][z]);
            }
    }
    q.lo = ix == 0;
    q.hi = ix == c.lx - 1;
    q.omega = omega, q.omw = omw;
    // LDS: 8 reciprocals, then the two buffers; a slot past the threads' holds zeros
    const int threads = c.lx * c.ty * c.tz;
    q.slots = threads + 1;
    q.rows = (typename T::f4*)(lds + 8);
    q.ends = (f2*)(lds + 8 + 16 * q.slots);
    const int zero = threads;
    q.me = on ? tid : zero;  // an idle thread's values are zeros
    q.up = on && iy > 0 ? tid - c.lx : zero;
    q.dn = on && iy + 1 < c.ty ? tid + c.lx : zero;
    q.be = on && iz > 0 ? tid - c.lx * c.ty : zero;
    q.ab = on && iz + 1 < c.tz ? tid + c.lx * c.ty : zero;
    if (tid < 8) lds[tid] = tid >= 1 && tid <= 6 ? rcp_count(tid) : 0.0f;
    if (tid < 4) {
        q.rows[tid * q.slots + zero] = typename T::f4{0.0f, 0.0f, 0.0f, 0.0f};
        q.ends[tid * q.slots + zero] = f2{0.0f, 0.0f};
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < T::NY; r++)
#pragma unroll
        for (int z = 0; z < T::NZ; z++) {
#pragma unroll
            for (int e = 0; e < 2; e++) {
                if constexpr (!WT) q.C[r][z][e] = *(const float*)((const char*)lds + ((nn[r][z] >> (8 * e)) & 0xffu));
                q.B[r][z][e] = q.B[r][z][e] - m;
            }
            if constexpr (WT) {
                const float next = T::shl1(q.wx[r][z][0]);
                q.wx[r][z][2] = q.hi ? 0.0f : next;
            }
        }
    q.template share<1>(0);
    __syncthreads();
    for (int it = 0; it < iters; it++) {
        q.template sweep<0>(0);
        q.template share<0>(1);
        __syncthreads();
        q.template sweep<1>(1);
        q.template share<1>(0);
        __syncthreads();
    }
    const __amdgpu_buffer_rsrc_t rd = split_buf(dst, 4u * cells);
    const bool xown = xin && x >= xo0 && x < xo1;
#pragma unroll
    for (int r = 0; r < T::NY; r++)
#pragma unroll
        for (int z = 0; z < T::NZ; z++) {
            const bool own = xown && y0 + r >= yo0 && y0 + r < yo1 && z0 + z >= zo0 && z0 + z < zo1;
            const uint32_t o = own ? 4u * at(r, z) : SPLIT_NONE;
            const f2 t{q.P[r][z][0], q.P[r][z][1]};
            __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(typename T::u2, t), rd, (int)o, 0, 0);
        }
}

}  // namespace zq3d
