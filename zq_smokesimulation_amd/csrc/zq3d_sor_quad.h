// zq3d_sor_quad.h -- K red-black SOR iterations of one tile in one pass over memory, with the tile's
// planes in registers; shared by the single-grid kernel (kernels_project.hip) and the ensemble
// kernel (kernels_ensemble.hip).
//
// Storage ("quad" layout): interleaved rows of S = quad_stride(W) values, no ghosts: cell (x, y, z) at
// (z*H + y)*S + x.  b holds the right-hand side, n the byte offset 4*count of 1/count in the tile's
// table (0: not updated); cells W..S-1 have n = 0 and, in every pressure a sweep writes, p = 0.
//
// A thread owns CX neighbouring cells (both colours) of R rows and marches z.  With V_0 the old black
// values and V_s the values after single-colour sweep s = 1..2K (odd red, even black), step t
// computes V_1 on plane t, V_2 on plane t-1, ..., V_2K on plane t-2K+1: sweep s at plane z needs
// V_(s-1) on planes z-1, z, z+1, the newest of which the same thread has just computed, so the z
// neighbours and the older values never leave registers.  x neighbours come from the next lane
// (DPP), y neighbours across threads through LDS.  Those are on the plane computed in the step
// before, so one barrier a step suffices however many sweeps the step runs.  A cell's sum, order and
// rounding are those of a single-colour sweep (st_sor_half): the result is the same bits.
//
// The tile's rows and planes shrink by one per sweep where it borders another tile: such a tile
// carries 2K extra rows, planes and cells on that side, whose values are recomputed and dropped.
// Rows and planes outside the grid read as n = 0, p = 0, the solver's ghost, and need no halo.
//
// What bounds it: at one sweep pair per pass (the colour-split tile of zq3d_sor_split.h) a step's
// instructions are mostly indexing, LDS and selects (47 VALU a cell update); here an update takes
// about 14, so K = 2 pays although it updates the halos twice.  Measured figures stand at
// quad_plan (kernels_project.hip).
#pragma once

#include "zq3d_device.h"
#include "zq3d_quad_cut.h"
#include "zq3d_sor_split.h"
#include "zq3d_stencils.h"

namespace zq3d {

template <int K, int CX, int R, bool MASK, int NT>
struct QuadTile {
    static_assert(CX == 2 || CX == 4, "");
    static_assert(R % 2 == 0, "a row's parity must not depend on the thread");
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    static constexpr int M = CX / 2;  // cells of one colour in a row
    static constexpr int J = 2 * K;   // sweeps a step
    // ring slots: planes modulo RS, an even number (a slot's parity is its plane's) that holds the planes of B
    // in use, t-J+1 .. t+1
    static constexpr int RS = 6;
    static_assert(J + 1 <= RS, "");

    float P[RS][R][CX];        // pressures as loaded
    float B[RS][R][CX];        // right-hand sides minus the mean
    unsigned N[RS][R];         // CX count bytes
    float V[J][RS][R][M];      // V[j]: values after sweep j (j >= 1)
    // fixed per thread
    // byte offset of the row's cells in a plane of floats; the same where stored, else SPLIT_NONE
    uint32_t off[R], soff[R];
    bool lo, hi;               // first / last lane of a row group
    // plane t + 2 of the source, t + 1 of b and n, t - J + 1 of the destination, and a plane's bytes
    const char *src, *b, *n;
    char* dst;
    uint32_t sbytes, bytes, nbytes;
    int D;
    float m, omega, omw;
    float* lds;
    int me, ab, be;  // this thread's values in an LDS block, the row group's above and below

    static constexpr int EDGE = quad_edge_floats(CX, NT);
    __device__ __forceinline__ float up(int j, int buf, int mm) const {  // last row of the group above
        return lds[8 + ((buf * J + j) * 2 + 1) * EDGE + ab + mm];
    }
    __device__ __forceinline__ float dn(int j, int buf, int mm) const {  // first row of the group below
        return lds[8 + ((buf * J + j) * 2 + 0) * EDGE + be + mm];
    }

    static __device__ __forceinline__ float shr1(float x) {  // the left lane's value (0 for lane 0)
        return __builtin_bit_cast(
            float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x138, 0xf, 0xf, true));
    }
    static __device__ __forceinline__ float shl1(float x) {  // the right lane's value (0 for lane 63)
        return __builtin_bit_cast(
            float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x130, 0xf, 0xf, true));
    }
    __device__ __forceinline__ float left(float x) const {
        const float y = shr1(x);
        return MASK && lo ? 0.0f : y;
    }
    __device__ __forceinline__ float right(float x) const {
        const float y = shl1(x);
        return MASK && hi ? 0.0f : y;
    }

    // a plane outside the grid is a buffer of no bytes: every lane reads 0
    __device__ __forceinline__ __amdgpu_buffer_rsrc_t plane_buf(const char* p, int z, uint32_t len) const {
        return split_buf(p, (unsigned)z < (unsigned)D ? len : 0u);
    }
    template <int SLOT>
    __device__ __forceinline__ void load_p(int z) {
        const __amdgpu_buffer_rsrc_t rs = plane_buf(src, z, sbytes);
        src += bytes;
#pragma unroll
        for (int r = 0; r < R; r++) load_row(rs, off[r], P[SLOT][r]);
    }
    static __device__ __forceinline__ void load_row(__amdgpu_buffer_rsrc_t rs, uint32_t o, float (&v)[CX]) {
        // (the vector is cast whole: a bit cast of one element of it reads element 0)
        if constexpr (CX == 4) {
            const f4 q = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)o, 0, 0));
            v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
        } else {
            const f2 q = __builtin_bit_cast(f2, __builtin_amdgcn_raw_buffer_load_b64(rs, (int)o, 0, 0));
            v[0] = q.x, v[1] = q.y;
        }
    }
    template <int SLOT>
    __device__ __forceinline__ void load_bn(int z) {
        const __amdgpu_buffer_rsrc_t rb = plane_buf(b, z, bytes), rn = plane_buf(n, z, nbytes);
        b += bytes;
        n += nbytes;
#pragma unroll
        for (int r = 0; r < R; r++) {
            load_row(rb, off[r], B[SLOT][r]);
            // a lane with nothing to load has off = SPLIT_NONE; a quarter of it is still past the end
            const int o = (int)(off[r] >> 2);
            if constexpr (CX == 4) N[SLOT][r] = (unsigned)__builtin_amdgcn_raw_buffer_load_b32(rn, o, 0, 0);
            else N[SLOT][r] = (unsigned)__builtin_amdgcn_raw_buffer_load_b16(rn, o, 0, 0);
        }
    }

    // value of sweep j (0: old black) in ring slot s, row r, cell m; e: parity of that colour's cells there
    template <int j>
    __device__ __forceinline__ float val(int s, int r, int mm, int e) const {
        if constexpr (j == 0) return P[s][r][2 * mm + e];
        else return V[j][s][r][mm];
    }

    // LDS rows of sweep j's values in ring slot s into buffer buf; e0: parity of row 0's cells there
    template <int j>
    __device__ __forceinline__ void share(int s, int buf, int e0) {
#pragma unroll
        for (int mm = 0; mm < M; mm++) {
            lds[8 + ((buf * J + j) * 2 + 0) * EDGE + me + mm] = val<j>(s, 0, mm, e0);
            lds[8 + ((buf * J + j) * 2 + 1) * EDGE + me + mm] = val<j>(s, R - 1, mm, (e0 + R - 1) & 1);
        }
    }

    // sweep j+1 of the step with t = PH (mod RS): plane t-j from V_j; up / down: the rows beside the thread's
    template <int PH, int j>
    __device__ __forceinline__ void sweep(const float (&u)[M], const float (&d)[M], float (&out)[R][M]) {
        constexpr int sz = (PH - j + 2 * RS) % RS, sm = (PH - j + 2 * RS - 1) % RS, sp = (PH - j + 2 * RS + 1) % RS;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int e = (r + PH) & 1;  // parity of the updated cells; the other colour's in this row is 1 - e
            float c[M];
#pragma unroll
            for (int mm = 0; mm < M; mm++) c[mm] = val<j>(sz, r, mm, 1 - e);
#pragma unroll
            for (int mm = 0; mm < M; mm++) {
                const float xm = e ? c[mm] : (mm ? c[mm - 1] : left(c[M - 1]));
                const float xp = e ? (mm + 1 < M ? c[mm + 1] : right(c[0])) : c[mm];
                const float ym = r ? val<j>(sz, r - 1, mm, e) : u[mm];
                const float yp = r + 1 < R ? val<j>(sz, r + 1, mm, e) : d[mm];
                const float s = xm + xp + ym + yp + val<j>(sm, r, mm, e) + val<j>(sp, r, mm, e);
                float own;
                if constexpr (j < 2) own = P[sz][r][2 * mm + e];
                else own = V[j - 1][sz][r][mm];
                const unsigned nb = (N[sz][r] >> (8 * (2 * mm + e))) & 0xffu;
                const float rc = *(const float*)((const char*)lds + nb);
                const float pg = (s - B[sz][r][2 * mm + e]) * rc;
                const float upd = omw * own + omega * pg;
                out[r][mm] = rc != 0.0f ? upd : own;
            }
        }
    }

    template <int PH, int j>
    __device__ __forceinline__ void sweeps(const float (&u)[J][M], const float (&d)[J][M], float (&last)[R][M]) {
        if constexpr (j + 1 < J) {
            sweep<PH, j>(u[j], d[j], V[j + 1][(PH - j + 2 * RS) % RS]);
            sweeps<PH, j + 1>(u, d, last);
        } else {
            sweep<PH, j>(u[j], d[j], last);
        }
    }
    template <int PH, int j>
    __device__ __forceinline__ void share_all() {
        // V_j's newest plane t-j+1 is the next step's centre plane; the parity of row 0's cells of V_j's
        // colour there is that of sweep j's output in this step (j >= 1), black at plane t+1 for j = 0
        share<j>((PH - j + 2 * RS + 1) % RS, (PH + 1) & 1, PH & 1);
        if constexpr (j + 1 < J) share_all<PH, j + 1>();
    }

    template <int PH>
    __device__ __forceinline__ void step(int t, int z0) {
        float u[J][M], d[J][M];
#pragma unroll
        for (int j = 0; j < J; j++)
#pragma unroll
            for (int mm = 0; mm < M; mm++) {
                u[j][mm] = up(j, PH & 1, mm);
                d[j][mm] = dn(j, PH & 1, mm);
            }
        load_p<(PH + 2) % RS>(t + 2);
        load_bn<(PH + 1) % RS>(t + 1);
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int c = 0; c < CX; c++) B[PH][r][c] = B[PH][r][c] - m;
        float last[R][M];
        sweeps<PH, 0>(u, d, last);
        share_all<PH, 0>();
        const int zo = t - J + 1;
        if (zo >= z0) {  // (zo < z1 in every step)
            const __amdgpu_buffer_rsrc_t rd = split_buf(dst, bytes);
            dst += bytes;
            constexpr int so = (PH - J + 1 + 2 * RS) % RS;
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int e = (r + PH) & 1;
                float o[CX];
#pragma unroll
                for (int mm = 0; mm < M; mm++) {
                    o[2 * mm + e] = last[r][mm];
                    o[2 * mm + 1 - e] = val<J - 1>(so, r, mm, 1 - e);
                }
                if constexpr (CX == 4)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, f4{o[0], o[1], o[2], o[3]}), rd,
                                                           (int)soff[r], 0, 0);
                else
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, f2{o[0], o[1]}), rd, (int)soff[r], 0,
                                                          0);
            }
        }
        __syncthreads();
    }
};

// One tile: workgroup of c.nw waves, tile (bx, by, bz) of the cut.  src == nullptr: the source is all
// zeros.  m: the mean subtracted from b.  lds: quad_lds_floats(K, CX, NT) floats, NT >= 64 c.nw.
template <int K, int CX, int R, bool MASK, int NT>
__device__ __forceinline__ void sor_quad_tile(const uint8_t* n, const float* b, float m, const float* src, float* dst,
                                              const Dims& d, const QuadCut& c, int bx, int by, int bz, float omega,
                                              float omw, float* lds) {
    using T = QuadTile<K, CX, R, MASK, NT>;
    constexpr int J = 2 * K;
    T q;
    const int S = quad_stride(d.W);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int g = quad_div(lane, c.mlx), ix = lane - g * c.lx;
    const int rg = wave * c.g + g;
    const bool on = g < c.g;
    // the tile's halo: lanes and rows beside another tile, planes below (the planes above are marched over)
    const int xo0 = quad_x_begin(c, K, CX, bx, S), xo1 = quad_x_begin(c, K, CX, bx + 1, S);
    const int x = xo0 - (bx ? CX * quad_halo_lanes(K, CX) : 0) + CX * ix;
    const int yo0 = quad_y_begin(c, K, by, d.H), yo1 = quad_y_begin(c, K, by + 1, d.H);
    const int y0 = yo0 - (by ? J : 0) + rg * R;
    const int z0 = quad_z_begin(c, K, bz, d.D), z1 = quad_z_begin(c, K, bz + 1, d.D);
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int y = y0 + r;
        const bool in = on && x >= 0 && x < S && y < d.H;
        const uint32_t o = 4u * (uint32_t)(y * S + x);
        q.off[r] = in ? o : SPLIT_NONE;
        q.soff[r] = in && x >= xo0 && x < xo1 && y >= yo0 && y < yo1 ? o : SPLIT_NONE;
    }
    q.lo = ix == 0;
    q.hi = ix == c.lx - 1;
    const int tb = bz ? z0 - J + 1 : 0;  // the first step's plane: even, as chunks begin at odd planes
    const long long plane = (long long)S * d.H;
    q.bytes = 4u * (uint32_t)plane;
    q.nbytes = (uint32_t)plane;
    q.sbytes = src ? q.bytes : 0u;
    q.src = (const char*)src + 4 * plane * (tb - 1);
    q.b = (const char*)b + 4 * plane * tb;
    q.n = (const char*)n + plane * tb;
    q.dst = (char*)dst + 4 * plane * z0;
    q.D = d.D;
    q.m = m, q.omega = omega, q.omw = omw;
    const int groups = c.nw * c.g;
    // idle lanes write zeros (n = 0, p = 0) to the last zero group
    q.me = ((on ? rg + 1 : groups + 1) * c.lx + ix) * T::M;
    q.ab = q.me - c.lx * T::M;
    q.be = on ? q.me + c.lx * T::M : q.me;
    q.lds = lds;
    // the groups above the first and below the last row group stay zero (the rest is written before it
    // is read, or read only for values outside the tile's valid range, which are dropped)
    for (int e = wave; e < 2 * J * 2 * 2; e += c.nw)
        for (int k = lane; k < c.lx * T::M; k += 64)
            lds[8 + (e >> 1) * T::EDGE + (e & 1 ? (groups + 1) * c.lx * T::M : 0) + k] = 0.0f;
    if (threadIdx.x < 8) lds[threadIdx.x] = threadIdx.x >= 1 && threadIdx.x <= 6 ? rcp_count(threadIdx.x) : 0.0f;
#pragma unroll
    for (int s = 0; s < T::RS; s++)
#pragma unroll
        for (int r = 0; r < R; r++) {
            q.N[s][r] = 0;
#pragma unroll
            for (int k = 0; k < CX; k++) q.P[s][r][k] = q.B[s][r][k] = 0.0f;
#pragma unroll
            for (int j = 0; j < J; j++)
#pragma unroll
                for (int mm = 0; mm < T::M; mm++) q.V[j][s][r][mm] = 0.0f;
        }
    int t = tb;
    const int te = z1 + J - 2;
    q.template load_p<T::RS - 1>(t - 1);
    q.template load_p<0>(t);
    q.template load_p<1>(t + 1);
    q.template load_bn<0>(t);
    __syncthreads();  // the zeros above before the rows below
    q.template share<0>(0, 0, 1);  // black at plane t: odd cells of row 0
    __syncthreads();
    for (;;) {
        q.template step<0>(t, z0);
        if (++t > te) break;
        q.template step<1>(t, z0);
        if (++t > te) break;
        q.template step<2>(t, z0);
        if (++t > te) break;
        q.template step<3>(t, z0);
        if (++t > te) break;
        q.template step<4>(t, z0);
        if (++t > te) break;
        q.template step<5>(t, z0);
        if (++t > te) break;
    }
}

}  // namespace zq3d
