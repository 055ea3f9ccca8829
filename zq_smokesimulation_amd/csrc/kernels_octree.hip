// kernels_octree.hip -- gfx950 kernels of the octree projection with the red-black solver
// (OPEN_OCTREE_POISSON_SOR / CLOSED_OCTREE_POISSON_SOR, ZQ_SmokeOctreeGrid3D.cpp).
//
// Build.  The reference fills a distance field breadth-first from the solid cells
// (_seedFilling, :5034-5167); that is the taxicab distance, computed here exactly by three
// separable line passes (each a forward and a backward min-plus scan).  Block minima per level and
// one pass over the fine cells then give the leaves (_buildOctreeInfo, :5377-5534) as one byte per
// fine cell: the level of the leaf holding it.
//
// Solve.  The reference precomputes per-leaf neighbour lists on the host
// (_selectInfos_for_CUDAOpenPoissonRedBlack3, :6330-9305) and hands them to the red-black kernels.
// Here each leaf walks its six faces over the level map instead: the fine cells behind a face,
// visited in the order of their interleaved (slower axis high) coordinates, meet the leaves behind
// the face in exactly the order the reference's lists hold them (same level or coarser first,
// else the finer leaves square by square), and a level-m leaf's cells form one aligned run of 4^m
// positions, skipped at once.  The sums coeff += w, sigma += w * p run in that order, so the
// result is the lists' bit for bit.  The walks run once per projection: they fill compact
// per-level, per-colour cell lists with their neighbour entries and diagonals, so that each sweep
// launch is a gather over short lists (a scene far from its obstacles is mostly 8^3 leaves, and the
// launches touch only those).
#include <vector>

#include "zq3d_coarse.h"
#include "zq3d_kernels.h"
#include "zq3d_octree.h"

namespace zq3d {
namespace {

constexpr int OCT_INF = 1 << 29;

struct OG {
    int W, H, D;
};

__device__ __forceinline__ int ow(const OG& g, int L) { return g.W >> L; }
__device__ __forceinline__ int oh(const OG& g, int L) { return g.H >> L; }
__device__ __forceinline__ int od(const OG& g, int L) { return g.D >> L; }
__device__ __forceinline__ size_t oat(const OG& g, int L, int x, int y, int z) {
    return ((size_t)z * (g.H >> L) + y) * (size_t)(g.W >> L) + x;
}

// weight[L][M] = 4^min(L,M) / (len_L + len_M), len = 0.5 * 2^L (the reference's weight tables,
// CPU_PoissonSolver3D_OpenOctreePoisson.cpp:408,452,496,540)
struct OctW {
    float w[4][4];
};

OctW make_weights() {
    OctW t{};
    for (int L = 0; L < 4; L++)
        for (int M = 0; M < 4; M++) {
            const int m = L < M ? L : M;
            const float area = (float)(1 << (2 * m));
            const float a = 0.5f * (float)(1 << L), b = 0.5f * (float)(1 << M);
            t.w[L][M] = area / (a + b);
        }
    return t;
}

struct LevelPtrs {
    const float* p[4];
};

// ---------------------------------------------------------------------------- distance field
// x lines: one wave per (y, z) row, 64 cells at a time; a ballot of the solid cells gives every lane the
// nearest one at or below it (forward pass) and above it (backward pass), with the last one met carried
// from chunk to chunk.  (One thread a row walked the row with a load a step: 345 us at 256^3.)
__global__ __launch_bounds__(256) void k_oct_dist_x(OG g, const uint8_t* __restrict__ occ, int32_t* __restrict__ dist) {
    const size_t line = (size_t)blockIdx.x * 4 + threadIdx.x / 64;
    if (line >= (size_t)g.H * g.D) return;
    const int lane = threadIdx.x & 63;
    const size_t base = line * g.W;
    const unsigned long long below = ~0ull >> (63 - lane), above = ~0ull << lane;
    int last = -1;  // the nearest solid cell before the chunk
    for (int x0 = 0; x0 < g.W; x0 += 64) {
        const int i = x0 + lane;
        const unsigned long long solid = __ballot(i < g.W && occ[base + i] != 0), m = solid & below;
        const int at = m ? x0 + 63 - __clzll((long long)m) : last;
        if (i < g.W) dist[base + i] = at >= 0 ? i - at : OCT_INF;
        if (solid) last = x0 + 63 - __clzll((long long)solid);
    }
    int next = -1;
    for (int x0 = (g.W - 1) / 64 * 64; x0 >= 0; x0 -= 64) {
        const int i = x0 + lane;
        const unsigned long long solid = __ballot(i < g.W && occ[base + i] != 0), m = solid & above;
        const int at = m ? x0 + __ffsll(m) - 1 : next;
        if (i < g.W && at >= 0) dist[base + i] = min(dist[base + i], at - i);
        if (solid) next = x0 + __ffsll(solid) - 1;
    }
}

// lines along y (axis 1) or z (axis 2): one thread per (x, other) pair, x fastest across lanes; the
// values of OCT_AHEAD steps are in flight together (a load a step left each of the few waves waiting
// out the memory's latency 2 n times)
constexpr int OCT_AHEAD = 16;
__global__ __launch_bounds__(64) void k_oct_dist_yz(OG g, int axis, int32_t* __restrict__ dist, int finish) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int n = axis == 1 ? g.H : g.D;
    const int other = axis == 1 ? g.D : g.H;
    if (t >= (size_t)g.W * other) return;
    const int x = (int)(t % g.W), o = (int)(t / g.W);
    const size_t stride = axis == 1 ? (size_t)g.W : (size_t)g.W * g.H;
    int32_t* const p = dist + (axis == 1 ? (size_t)o * g.H * g.W + x : (size_t)o * g.W + x);
    int d = OCT_INF;
    for (int i0 = 0; i0 < n; i0 += OCT_AHEAD) {
        int v[OCT_AHEAD];
#pragma unroll
        for (int q = 0; q < OCT_AHEAD; q++) v[q] = i0 + q < n ? p[(i0 + q) * stride] : OCT_INF;
#pragma unroll
        for (int q = 0; q < OCT_AHEAD; q++) {
            d = min(v[q], min(d + 1, OCT_INF));
            if (i0 + q < n) p[(i0 + q) * stride] = d;
        }
    }
    d = OCT_INF;
    for (int i0 = (n - 1) / OCT_AHEAD * OCT_AHEAD; i0 >= 0; i0 -= OCT_AHEAD) {
        int v[OCT_AHEAD];
#pragma unroll
        for (int q = 0; q < OCT_AHEAD; q++) v[q] = i0 + q < n ? p[(i0 + q) * stride] : OCT_INF;
#pragma unroll
        for (int q = OCT_AHEAD - 1; q >= 0; q--) {
            d = min(v[q], min(d + 1, OCT_INF));
            // no solid cell anywhere: every distance is W + H + D (_buildOctreeInfo, :5365-5373)
            if (i0 + q < n) p[(i0 + q) * stride] = (finish && d >= OCT_INF) ? g.W + g.H + g.D : d;
        }
    }
}

// smallest distance in each level-L block from the level below
__global__ __launch_bounds__(256) void k_oct_min(OG g, int L, const int32_t* __restrict__ src, int32_t* __restrict__ dst) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int wl = ow(g, L), hl = oh(g, L);
    if (t >= (size_t)wl * hl * od(g, L)) return;
    const int x = (int)(t % wl), y = (int)((t / wl) % hl), z = (int)(t / ((size_t)wl * hl));
    int m = OCT_INF;
    for (int k = 0; k < 2; k++)
        for (int j = 0; j < 2; j++)
            for (int i = 0; i < 2; i++) m = min(m, src[oat(g, L - 1, 2 * x + i, 2 * y + j, 2 * z + k)]);
    dst[t] = m;
}

// level map and leaf flags: a level-3 block is a leaf when its smallest distance exceeds t3, a
// level-2 block outside level-3 leaves when its smallest distance exceeds t2, a level-1 block
// outside coarser leaves likewise with t1; a fine cell in no coarser leaf is a level-0 leaf unless
// solid
__global__ __launch_bounds__(256) void k_oct_levels(OG g, int t1, int t2, int t3, const uint8_t* __restrict__ occ,
                                                    const int32_t* __restrict__ m1, const int32_t* __restrict__ m2,
                                                    const int32_t* __restrict__ m3, uint8_t* __restrict__ lev,
                                                    uint8_t* __restrict__ l1, uint8_t* __restrict__ l2,
                                                    uint8_t* __restrict__ l3) {
    const int x = blockIdx.x * 64 + threadIdx.x, y = blockIdx.y * 4 + threadIdx.y, z = blockIdx.z;
    if (x >= g.W || y >= g.H) return;
    const bool a3 = m3[oat(g, 3, x >> 3, y >> 3, z >> 3)] > t3;
    const bool a2 = !a3 && m2[oat(g, 2, x >> 2, y >> 2, z >> 2)] > t2;
    const bool a1 = !a3 && !a2 && m1[oat(g, 1, x >> 1, y >> 1, z >> 1)] > t1;
    const size_t c = oat(g, 0, x, y, z);
    lev[c] = a3 ? 3 : a2 ? 2 : a1 ? 1 : (occ[c] ? OCT_SOLID : 0);
    if (((x | y | z) & 1) == 0) l1[oat(g, 1, x >> 1, y >> 1, z >> 1)] = a1;
    if (((x | y | z) & 3) == 0) l2[oat(g, 2, x >> 2, y >> 2, z >> 2)] = a2;
    if (((x | y | z) & 7) == 0) l3[oat(g, 3, x >> 3, y >> 3, z >> 3)] = a3;
}

// level map from caller-given leaf flags (the first level whose flag covers the cell; none: solid)
__global__ __launch_bounds__(256) void k_oct_levels_given(OG g, const uint8_t* __restrict__ a0,
                                                          const uint8_t* __restrict__ a1,
                                                          const uint8_t* __restrict__ a2,
                                                          const uint8_t* __restrict__ a3, uint8_t* __restrict__ lev,
                                                          uint8_t* __restrict__ l1, uint8_t* __restrict__ l2,
                                                          uint8_t* __restrict__ l3) {
    const int x = blockIdx.x * 64 + threadIdx.x, y = blockIdx.y * 4 + threadIdx.y, z = blockIdx.z;
    if (x >= g.W || y >= g.H) return;
    const size_t c = oat(g, 0, x, y, z);
    const bool b1 = a1[oat(g, 1, x >> 1, y >> 1, z >> 1)] != 0, b2 = a2[oat(g, 2, x >> 2, y >> 2, z >> 2)] != 0;
    const bool b3 = a3[oat(g, 3, x >> 3, y >> 3, z >> 3)] != 0;
    lev[c] = a0[c] ? 0 : b1 ? 1 : b2 ? 2 : b3 ? 3 : OCT_SOLID;
    if (((x | y | z) & 1) == 0) l1[oat(g, 1, x >> 1, y >> 1, z >> 1)] = b1;
    if (((x | y | z) & 3) == 0) l2[oat(g, 2, x >> 2, y >> 2, z >> 2)] = b2;
    if (((x | y | z) & 7) == 0) l3[oat(g, 3, x >> 3, y >> 3, z >> 3)] = b3;
}

// ---------------------------------------------------------------------------- divergence
// fine cells: u(i+1) - u(i) + v(j+1) - v(j) + w(k+1) - w(k), left to right; p0 = 0
__global__ __launch_bounds__(256) void k_oct_div0(OG g, const float* __restrict__ u, const float* __restrict__ v,
                                                  const float* __restrict__ w, float* __restrict__ d0,
                                                  float* __restrict__ p0) {
    const int x = blockIdx.x * 64 + threadIdx.x, y = blockIdx.y * 4 + threadIdx.y, z = blockIdx.z;
    if (x >= g.W || y >= g.H) return;
    const size_t cu = ((size_t)z * g.H + y) * (g.W + 1) + x, cv = ((size_t)z * (g.H + 1) + y) * g.W + x;
    const size_t cw = ((size_t)z * g.H + y) * g.W + x;
    d0[cw] = u[cu + 1] - u[cu] + v[cv + g.W] - v[cv] + w[cw + (size_t)g.W * g.H] - w[cw];
    p0[cw] = 0.0f;
}

// level L: the sum of the eight children in x-fastest order, left to right; p_L = 0
__global__ __launch_bounds__(256) void k_oct_restrict(OG g, int L, const float* __restrict__ src,
                                                      float* __restrict__ dst, float* __restrict__ pl) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int wl = ow(g, L), hl = oh(g, L);
    if (t >= (size_t)wl * hl * od(g, L)) return;
    const int x = (int)(t % wl), y = (int)((t / wl) % hl), z = (int)(t / ((size_t)wl * hl));
    const int M = L - 1, X = 2 * x, Y = 2 * y, Z = 2 * z;
    dst[t] = src[oat(g, M, X, Y, Z)] + src[oat(g, M, X + 1, Y, Z)] + src[oat(g, M, X, Y + 1, Z)] +
             src[oat(g, M, X + 1, Y + 1, Z)] + src[oat(g, M, X, Y, Z + 1)] + src[oat(g, M, X + 1, Y, Z + 1)] +
             src[oat(g, M, X, Y + 1, Z + 1)] + src[oat(g, M, X + 1, Y + 1, Z + 1)];
    pl[t] = 0.0f;
}

// ---------------------------------------------------------------------------- Gauss-Seidel
// The cells each sweep updates, per level and colour (red: even x + y + z at the level): every
// level-0..2 leaf, and every level-3 leaf whose column's block at z = 0 is a leaf (the reference's
// level-3 list test, ZQ_SmokeOctreeGrid3D.cpp:8416; the blocks that test takes that are no leaf are
// never read, so they are left out).  Within a list the order is free: cells of one colour and level
// never neighbour each other.
// A workgroup counts its cells per list in LDS, takes its places with one atomic a list and writes (an
// atomic a wave and list had all of the fine grid's waves queue at eight addresses: 170 us at 256^3).
constexpr int OCT_LIST_CELLS = 8;  // cells a thread
__global__ __launch_bounds__(256) void k_oct_lists(OG g, const uint8_t* __restrict__ lev, uint32_t* l00, uint32_t* l01,
                                                   uint32_t* l10, uint32_t* l11, uint32_t* l20, uint32_t* l21,
                                                   uint32_t* l30, uint32_t* l31, uint32_t* count) {
    __shared__ uint32_t n[OCT_LISTS], base[OCT_LISTS];
    if (threadIdx.x < OCT_LISTS) n[threadIdx.x] = 0u;
    __syncthreads();
    const size_t N = (size_t)g.W * g.H * g.D;
    int list[OCT_LIST_CELLS];  // -1: in none
    uint32_t idx[OCT_LIST_CELLS], pos[OCT_LIST_CELLS];
#pragma unroll
    for (int q = 0; q < OCT_LIST_CELLS; q++) {
        const size_t c = ((size_t)blockIdx.x * OCT_LIST_CELLS + q) * 256 + threadIdx.x;
        list[q] = -1;
        if (c >= N) continue;
        const int L = lev[c];
        if (L == OCT_SOLID) continue;
        const int x = (int)(c % g.W), y = (int)((c / g.W) % g.H), z = (int)(c / ((size_t)g.W * g.H));
        if ((x | y | z) & ((1 << L) - 1)) continue;
        if (L == 3 && lev[oat(g, 0, x, y, 0)] != 3) continue;
        list[q] = 2 * L + (((x >> L) + (y >> L) + (z >> L)) & 1);
        idx[q] = (uint32_t)oat(g, L, x >> L, y >> L, z >> L);
        pos[q] = atomicAdd(&n[list[q]], 1u);
    }
    __syncthreads();
    if (threadIdx.x < OCT_LISTS && n[threadIdx.x]) base[threadIdx.x] = atomicAdd(count + threadIdx.x, n[threadIdx.x]);
    __syncthreads();
    uint32_t* const lists[OCT_LISTS] = {l00, l01, l10, l11, l20, l21, l30, l31};
#pragma unroll
    for (int q = 0; q < OCT_LIST_CELLS; q++)
#pragma unroll
        for (int k = 0; k < OCT_LISTS; k++)
            if (list[q] == k) lists[k][base[k] + pos[q]] = idx[q];
}

__global__ void k_oct_zero(uint32_t* count) {
    if (threadIdx.x < 4 * OCT_LISTS) count[threadIdx.x] = 0u;
}

// A neighbour entry: level in bits 30-31, the linear index at that level below.  An open domain face
// is OCT_OPEN in a walk; it weighs in the diagonal only, so the stored entries leave it out.  OCT_NONE
// fills a cell's unused entries.
constexpr uint32_t OCT_OPEN = 0xFFFFFFFFu;
constexpr uint32_t OCT_NONE = 0xFFFFFFFFu;

__device__ __forceinline__ uint32_t oct_entry(const OG& g, int m, int x, int y, int z) {
    return ((uint32_t)m << 30) | (uint32_t)oat(g, m, x >> m, y >> m, z >> m);
}

// The neighbour entries of the level-L cell (x, y, z), in the reference's order, handed to put(e).
// Per face: an open domain face; else the leaf behind the face's first fine
// cell when it is as large as this one (at level 0: the fine neighbour unless solid); else the face's
// fine cells in interleaved order (slower axis high), one entry per leaf met (its run of 4^m
// positions skipped), solid cells skipped.
template <class Put>
__device__ __forceinline__ void oct_walk(const OG& g, const uint8_t* __restrict__ lev, int L, int x, int y, int z,
                                         Put put) {
    const int S = 1 << L;
    const int cl[3] = {x, y, z}, dims[3] = {ow(g, L), oh(g, L), od(g, L)}, base[3] = {x * S, y * S, z * S};
#pragma unroll
    for (int f = 0; f < 6; f++) {
        const int ax = f >> 1, sd = (f & 1) ? 1 : -1;
        if ((sd < 0 && cl[ax] == 0) || (sd > 0 && cl[ax] == dims[ax] - 1)) {
            put(OCT_OPEN);
            continue;
        }
        const int slow = ax == 2 ? 1 : 2, fast = ax == 0 ? 1 : 0;
        int q0[3] = {base[0], base[1], base[2]};
        q0[ax] = sd < 0 ? base[ax] - 1 : base[ax] + S;
        const int m0 = lev[oat(g, 0, q0[0], q0[1], q0[2])];
        if (m0 != OCT_SOLID && m0 >= L) {  // one leaf as large as this one covers the face
            put(oct_entry(g, m0, q0[0], q0[1], q0[2]));
            continue;
        }
        for (int t = 0; t < S * S;) {
            int a = 0, b = 0;
            for (int j = 0; j < L; j++) {
                b |= ((t >> (2 * j)) & 1) << j;
                a |= ((t >> (2 * j + 1)) & 1) << j;
            }
            int q[3] = {q0[0], q0[1], q0[2]};
            q[slow] += a;
            q[fast] += b;
            const int m = lev[oat(g, 0, q[0], q[1], q[2])];
            if (m == OCT_SOLID) {
                t += 1;
                continue;
            }
            put(oct_entry(g, m, q[0], q[1], q[2]));
            t += 1 << (2 * m);  // m < L here: the rest of that leaf's run on this face
        }
    }
}

__device__ __forceinline__ void oct_cell(const OG& g, int L, uint32_t c, int& x, int& y, int& z) {
    const uint32_t wl = (uint32_t)ow(g, L), hl = (uint32_t)oh(g, L);
    x = (int)(c % wl);
    y = (int)((c / wl) % hl);
    z = (int)(c / (wl * hl));
}

// The lists one launch takes, one after the other over its blocks of OCT_BLOCK cells.  The set-up
// launches take all eight, a sweep launch at most one per level.
constexpr int OCT_BLOCK = 64;

struct OctSeg {
    const uint32_t* list;
    uint32_t* head;  // entry j of cell i at j * n + i
    uint32_t* ovo;   // a cell's first entry in ovf, and its entries there
    uint32_t* ovn;
    uint32_t* ovf;
    float* coeff;
    float* rhs;
    uint32_t n, first;  // cells; the launch's first block of this list
    int k, width;       // list number 2 L + colour; entries per cell kept in the head
    int over;           // some cell of the list has entries in ovf
    float w0, w1, w2, w3;  // the level's weights towards a leaf of level 0..3 (open domain face: 3)
};

__device__ __forceinline__ float oct_weight(const OctSeg& q, uint32_t m) {
    const float lo = m & 1 ? q.w1 : q.w0, hi = m & 1 ? q.w3 : q.w2;
    return m & 2 ? hi : lo;
}

template <int N>
struct OctSegs {
    OctSeg s[N];
    int count;
};

// the list of this block (every block has one: the grid is the sum of the lists' blocks)
template <int N>
__device__ __forceinline__ OctSeg oct_seg(const OctSegs<N>& t, uint32_t& i) {
    OctSeg r = t.s[0];
#pragma unroll
    for (int j = 1; j < N; j++)
        if (j < t.count && blockIdx.x >= t.s[j].first) r = t.s[j];
    i = (blockIdx.x - r.first) * OCT_BLOCK + threadIdx.x;
    return r;
}

// Per listed cell the entries beyond OCT_WIDE (ovn) and their place in ovf (ovo: order free, an
// atomic hands out the runs); per list their sum, the largest number of entries of a cell and the
// levels the entries name (count + 8, + 16, + 24).
__global__ __launch_bounds__(OCT_BLOCK) void k_oct_count(OG g, const uint8_t* __restrict__ lev, OctSegs<OCT_LISTS> t,
                                                         uint32_t* __restrict__ count) {
    uint32_t i;
    const OctSeg q = oct_seg(t, i);
    uint32_t k = 0, seen = 0;
    if (i < q.n) {
        int x, y, z;
        oct_cell(g, q.k >> 1, q.list[i], x, y, z);
        oct_walk(g, lev, q.k >> 1, x, y, z, [&](uint32_t e) {
            if (e == OCT_OPEN) return;
            k++;
            seen |= 1u << (e >> 30);
        });
        const uint32_t o = k > OCT_WIDE ? k - OCT_WIDE : 0u;
        q.ovn[i] = o;
        q.ovo[i] = o ? atomicAdd(count + OCT_LISTS + q.k, o) : 0u;
    }
    for (int d = 32; d; d >>= 1) {
        k = max(k, (uint32_t)__shfl_xor((int)k, d, 64));
        seen |= (uint32_t)__shfl_xor((int)seen, d, 64);
    }
    if (threadIdx.x == 0) {
        // an older value read here costs at most an atomic that changes nothing
        uint32_t *most = count + 2 * OCT_LISTS + q.k, *levels = count + 3 * OCT_LISTS + q.k;
        if (k > __hip_atomic_load(most, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(most, k);
        if (seen & ~__hip_atomic_load(levels, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicOr(levels, seen);
    }
}

// The entries, their weights' sum in walk order (open faces included) and the rest of the head row
// filled with OCT_NONE.  A wave's stores of one entry number are contiguous.
__global__ __launch_bounds__(OCT_BLOCK) void k_oct_fill(OG g, const uint8_t* __restrict__ lev, OctSegs<OCT_LISTS> t) {
    uint32_t i;
    const OctSeg q = oct_seg(t, i);
    if (i >= q.n) return;
    int x, y, z;
    const int L = q.k >> 1;
    oct_cell(g, L, q.list[i], x, y, z);
    uint32_t* ov = q.ovf + q.ovo[i];
    float coeff = 0.0f;
    int k = 0;
    oct_walk(g, lev, L, x, y, z, [&](uint32_t e) {
        const uint32_t m = e >> 30;  // OCT_OPEN: the level-3 weight
        coeff += oct_weight(q, m);
        if (e == OCT_OPEN) return;
        if (k < q.width) q.head[(size_t)k * q.n + i] = e;
        else ov[k - q.width] = e;
        k++;
    });
    for (; k < q.width; k++) q.head[(size_t)k * q.n + i] = OCT_NONE;
    q.coeff[i] = coeff;
}

// right-hand side per listed cell in list order: the level's divergence, with `mean` the closed form
// div - mean * 8^L
__global__ __launch_bounds__(OCT_BLOCK) void k_oct_rhs(LevelPtrs dl, OctSegs<OCT_LISTS> t,
                                                       const float* __restrict__ mean) {
    uint32_t i;
    const OctSeg q = oct_seg(t, i);
    if (i >= q.n) return;
    const int L = q.k >> 1;
    const float* d = L == 0 ? dl.p[0] : L == 1 ? dl.p[1] : L == 2 ? dl.p[2] : dl.p[3];
    const float dd = d[q.list[i]];
    q.rhs[i] = mean ? dd - *mean * (float)(1 << (3 * L)) : dd;
}

// The pressures of all four levels sit in one allocation: level m starts off[m] floats after p.
struct OctP {
    float* p;
    uint32_t off[4];
};

__device__ __forceinline__ uint32_t oct_level_off(const OctP& P, uint32_t m) {
    const uint32_t lo = m & 1 ? P.off[1] : P.off[0], hi = m & 1 ? P.off[3] : P.off[2];
    return m & 2 ? hi : lo;
}

// NE entries at once: every pressure they name is in flight before the first sum.  An unused entry
// reads cell 0 of level 0 and adds 0 (the sum is never -0, so it stays as it is).
template <int NE>
__device__ __forceinline__ float oct_sum(const OctP& P, const OctSeg& q, const uint32_t (&e)[NE], float sigma) {
    float pv[NE];
#pragma unroll
    for (int j = 0; j < NE; j++) {
        const uint32_t m = e[j] >> 30;
        const uint32_t at = e[j] == OCT_NONE ? 0u : oct_level_off(P, m) + (e[j] & 0x3FFFFFFFu);
        pv[j] = P.p[at];
    }
#pragma unroll
    for (int j = 0; j < NE; j++) {
        const uint32_t m = e[j] >> 30;
        const float wg = oct_weight(q, m);
        sigma += wg * (e[j] == OCT_NONE ? 0.0f : pv[j]);
    }
    return sigma;
}

template <int NE>
__device__ __forceinline__ void oct_gs_cell(const OctP& P, const OctSeg& q, uint32_t i) {
    const uint32_t c = q.list[i];
    const float r = q.rhs[i], coeff = q.coeff[i];
    uint32_t ev[NE], no = 0, o0 = 0;
    if (q.over) {
        no = q.ovn[i];
        o0 = q.ovo[i];
    }
#pragma unroll
    for (int j = 0; j < NE; j++) ev[j] = q.head[(size_t)j * q.n + i];
    float sigma = oct_sum<NE>(P, q, ev, 0.0f);
    for (uint32_t k0 = 0; k0 < no; k0 += 8) {
        uint32_t e8[8];
#pragma unroll
        for (int j = 0; j < 8; j++) e8[j] = k0 + j < no ? q.ovf[o0 + k0 + j] : OCT_NONE;
        sigma = oct_sum<8>(P, q, e8, sigma);
    }
    sigma -= r;
    P.p[oct_level_off(P, (uint32_t)q.k >> 1) + c] = sigma / coeff;
}

// One update p = (sigma - rhs) / coeff, sigma += w * p over a cell's entries in order
// (CPU_PoissonSolver3D_OpenOctreePoisson.cpp:404-425), for every cell of the launch's lists; no two
// of them neighbour each other.  A launch is a few microseconds of latency: every list but that of a
// finest region is a few waves per CU at most.  So the chain of dependent loads is kept at two (the
// list, the right-hand side, the diagonal and all head entries; then all pressures), waves spread
// over the CUs one to a block, and a launch takes every list that may run beside the others.  256^3
// around one sphere, thresholds 4, 8, 24 (levels step one at a time), 600 passes: 4800 launches of 7.9
// us before, 2404 now, the frame 42.5 -> 13.9 ms.
__global__ __launch_bounds__(OCT_BLOCK) void k_oct_gs(OctP P, OctSegs<4> t) {
    uint32_t i;
    const OctSeg q = oct_seg(t, i);
    if (i >= q.n) return;
    if (q.width <= 6) oct_gs_cell<6>(P, q, i);
    else if (q.width <= 12) oct_gs_cell<12>(P, q, i);
    else oct_gs_cell<OCT_WIDE>(P, q, i);
}

// ---------------------------------------------------------------------------- face correction
// half the size of the level-m leaf holding fine cell (x, y, z), and its pressure
__device__ __forceinline__ float oct_half(int m) { return 0.5f * (float)(1 << m); }
__device__ __forceinline__ float oct_pressure(const OG& g, const LevelPtrs& P, int m, int x, int y, int z) {
    const float* p = m & 2 ? (m & 1 ? P.p[3] : P.p[2]) : (m & 1 ? P.p[1] : P.p[0]);
    return p[oat(g, m, x >> m, y >> m, z >> m)];
}

// face -= (p2 - p1) / (len1 + len2) between two leaves (no face inside a leaf or beside a solid cell);
// domain faces against a ghost 4 cells out
// (Adjust_MAC_{u,v,w}_OpenOctreePoisson_Kernel, CPU_PoissonSolver3D_OpenOctreePoisson.cpp:6-373).
// A thread does its cell's low faces, beside the last cell of an axis also the domain's high face: the
// cell's level and pressure serve all of them.  (A thread a face: 240 us at 256^3; now 115.)
__global__ __launch_bounds__(256) void k_oct_adjust(OG g, LevelPtrs P, const uint8_t* __restrict__ lev,
                                                    float* __restrict__ u, float* __restrict__ v,
                                                    float* __restrict__ w) {
    const int x = blockIdx.x * 64 + threadIdx.x, y = blockIdx.y * 4 + threadIdx.y, z = blockIdx.z;
    if (x >= g.W || y >= g.H) return;
    const size_t c = oat(g, 0, x, y, z), plane = (size_t)g.W * g.H;
    const int m = lev[c];
    if (m == OCT_SOLID) return;
    const int mx = x ? lev[c - 1] : 0, my = y ? lev[c - g.W] : 0, mz = z ? lev[c - plane] : 0;
    const int low = (1 << m) - 1;
    const float len = oct_half(m);
    const size_t cu = ((size_t)z * g.H + y) * (g.W + 1) + x, cv = ((size_t)z * (g.H + 1) + y) * g.W + x, cw = c;
    // this leaf's side of the low faces, and whether the neighbour's block also ends there
    const bool fx = (x & low) == 0, fy = (y & low) == 0, fz = (z & low) == 0;
    const bool hx = x == g.W - 1, hy = y == g.H - 1, hz = z == g.D - 1;
    if (!(fx || fy || fz || hx || hy || hz)) return;
    const float pc = oct_pressure(g, P, m, x, y, z);
    auto between = [&](float* face, int n, int f, float pn) {
        if (f & ((1 << n) - 1)) return;
        *face = *face - (pc - pn) / (oct_half(n) + len);
    };
    if (fx) {
        if (x == 0) u[cu] = u[cu] - (pc - 0.0f) / (4.0f + len);
        else if (mx != OCT_SOLID) between(u + cu, mx, x, oct_pressure(g, P, mx, x - 1, y, z));
    }
    if (fy) {
        if (y == 0) v[cv] = v[cv] - (pc - 0.0f) / (4.0f + len);
        else if (my != OCT_SOLID) between(v + cv, my, y, oct_pressure(g, P, my, x, y - 1, z));
    }
    if (fz) {
        if (z == 0) w[cw] = w[cw] - (pc - 0.0f) / (4.0f + len);
        else if (mz != OCT_SOLID) between(w + cw, mz, z, oct_pressure(g, P, mz, x, y, z - 1));
    }
    // (the dimensions are multiples of 8: a leaf always ends at the domain's high side)
    if (hx) u[cu + 1] = u[cu + 1] - (0.0f - pc) / (4.0f + len);
    if (hy) v[cv + g.W] = v[cv + g.W] - (0.0f - pc) / (4.0f + len);
    if (hz) w[cw + plane] = w[cw + plane] - (0.0f - pc) / (4.0f + len);
}

unsigned blocks_of(size_t n, int b) { return (unsigned)((n + b - 1) / b); }
dim3 fine_grid(const Dims& g) { return dim3((unsigned)((g.W + 63) / 64), (unsigned)((g.H + 3) / 4), (unsigned)g.D); }
size_t level_cells(const Dims& g, int L) { return (size_t)(g.W >> L) * (g.H >> L) * (g.D >> L); }
size_t up256(size_t b) { return (b + 255) & ~(size_t)255; }

hipError_t grow(void** p, size_t* cap, size_t need) {
    if (need <= *cap && *p) return hipSuccess;
    if (*p) (void)hipFree(*p);
    *p = nullptr;
    *cap = 0;
    const size_t c = need + need / 2 + 4096;
    hipError_t e = hipMalloc(p, c);
    if (e == hipSuccess) *cap = c;
    return e;
}

}  // namespace

size_t octree_bytes(const Dims& g) {
    size_t b = up256(level_cells(g, 0)) + up256(4 * level_cells(g, 0));  // lev, dist
    for (int L = 1; L <= 3; L++) b += up256(level_cells(g, L)) + up256(4 * level_cells(g, L));  // leaf, mn
    for (int L = 0; L <= 3; L++) b += 2 * up256(4 * level_cells(g, L));  // p, d
    for (int L = 0; L <= 3; L++) b += 2 * up256(4 * (level_cells(g, L) / 2 + 1));  // lists
    return b + 256;  // counts
}

void octree_layout(const Dims& g, char* mem, OctreeBufs* B) {
    size_t o = 0;
    auto take = [&](size_t bytes) {
        char* p = mem + o;
        o += up256(bytes);
        return p;
    };
    B->lev = (uint8_t*)take(level_cells(g, 0));
    B->dist = (int32_t*)take(4 * level_cells(g, 0));
    B->leaf[0] = nullptr;
    B->mn[0] = B->dist;
    for (int L = 1; L <= 3; L++) {
        B->leaf[L] = (uint8_t*)take(level_cells(g, L));
        B->mn[L] = (int32_t*)take(4 * level_cells(g, L));
    }
    for (int L = 0; L <= 3; L++) {
        B->p[L] = (float*)take(4 * level_cells(g, L));
        B->d[L] = (float*)take(4 * level_cells(g, L));
    }
    for (int L = 0; L <= 3; L++)
        for (int c = 0; c < 2; c++) B->list[L][c] = (uint32_t*)take(4 * (level_cells(g, L) / 2 + 1));
    B->count = (uint32_t*)take(4 * 4 * OCT_LISTS);
}

void launch_octree_build(const Dims& d, const uint8_t* occ, int t1, int t2, int t3, const OctreeBufs& B,
                         hipStream_t s) {
    const OG g{d.W, d.H, d.D};
    hipLaunchKernelGGL(k_oct_dist_x, dim3(blocks_of((size_t)d.H * d.D, 4)), dim3(256), 0, s, g, occ, B.dist);
    hipLaunchKernelGGL(k_oct_dist_yz, dim3(blocks_of((size_t)d.W * d.D, 64)), dim3(64), 0, s, g, 1, B.dist, 0);
    hipLaunchKernelGGL(k_oct_dist_yz, dim3(blocks_of((size_t)d.W * d.H, 64)), dim3(64), 0, s, g, 2, B.dist, 1);
    for (int L = 1; L <= 3; L++)
        hipLaunchKernelGGL(k_oct_min, dim3(blocks_of(level_cells(d, L), 256)), dim3(256), 0, s, g, L,
                           (const int32_t*)B.mn[L - 1], B.mn[L]);
    hipLaunchKernelGGL(k_oct_levels, fine_grid(d), dim3(64, 4), 0, s, g, t1, t2, t3, occ, (const int32_t*)B.mn[1],
                       (const int32_t*)B.mn[2], (const int32_t*)B.mn[3], B.lev, B.leaf[1], B.leaf[2], B.leaf[3]);
}

void launch_octree_from_leaves(const Dims& d, const uint8_t* l0, const uint8_t* l1, const uint8_t* l2,
                               const uint8_t* l3, const OctreeBufs& B, hipStream_t s) {
    const OG g{d.W, d.H, d.D};
    hipLaunchKernelGGL(k_oct_levels_given, fine_grid(d), dim3(64, 4), 0, s, g, l0, l1, l2, l3, B.lev, B.leaf[1],
                       B.leaf[2], B.leaf[3]);
}

void launch_octree_prepare(const Dims& d, const float* u, const float* v, const float* w, const OctreeBufs& B,
                           hipStream_t s) {
    const OG g{d.W, d.H, d.D};
    hipLaunchKernelGGL(k_oct_div0, fine_grid(d), dim3(64, 4), 0, s, g, u, v, w, B.d[0], B.p[0]);
    for (int L = 1; L <= 3; L++)
        hipLaunchKernelGGL(k_oct_restrict, dim3(blocks_of(level_cells(d, L), 256)), dim3(256), 0, s, g, L,
                           (const float*)B.d[L - 1], B.d[L], B.p[L]);
}

namespace {

// the launch table of the lists in `mask` (bit k: list k), and its blocks
template <int N>
uint32_t oct_segs(const OctreeBufs& B, const OctreeLists& Ls, uint32_t mask, OctSegs<N>* t) {
    const OctW wt = make_weights();
    uint32_t blocks = 0;
    t->count = 0;
    for (int k = 0; k < OCT_LISTS; k++) {
        const uint32_t n = Ls.counts[k];
        if (!(mask >> k & 1) || !n) continue;
        t->s[t->count++] = OctSeg{B.list[k / 2][k % 2], Ls.head[k], Ls.ovo[k], Ls.ovn[k], Ls.ovf[k], Ls.coeff[k],
                                  Ls.rhs[k], n, blocks, k, Ls.width[k], Ls.over[k],
                                  wt.w[k / 2][0], wt.w[k / 2][1], wt.w[k / 2][2], wt.w[k / 2][3]};
        blocks += blocks_of(n, OCT_BLOCK);
    }
    return blocks;
}

}  // namespace

hipError_t octree_build_lists(const Dims& d, const OctreeBufs& B, OctreeLists* Ls, hipStream_t s) {
    const OG g{d.W, d.H, d.D};
    hipLaunchKernelGGL(k_oct_zero, dim3(1), dim3(64), 0, s, B.count);
    hipLaunchKernelGGL(k_oct_lists, dim3(blocks_of(level_cells(d, 0), 256 * OCT_LIST_CELLS)), dim3(256), 0, s, g,
                       (const uint8_t*)B.lev, B.list[0][0], B.list[0][1], B.list[1][0], B.list[1][1], B.list[2][0],
                       B.list[2][1], B.list[3][0], B.list[3][1], B.count);
    uint32_t got[4 * OCT_LISTS];
    hipError_t e = hipMemcpyAsync(got, B.count, 4 * OCT_LISTS, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return e;
    size_t bytes = 0;
    for (int k = 0; k < OCT_LISTS; k++) {
        Ls->counts[k] = got[k];
        bytes += 4 * up256(4 * (size_t)got[k]);
    }
    if ((e = grow(&Ls->dyn, &Ls->dyn_cap, bytes)) != hipSuccess) return e;
    char* p = (char*)Ls->dyn;
    for (int k = 0; k < OCT_LISTS; k++) {
        const size_t one = up256(4 * (size_t)Ls->counts[k]);
        Ls->ovo[k] = (uint32_t*)p;
        Ls->ovn[k] = (uint32_t*)(p + one);
        Ls->coeff[k] = (float*)(p + 2 * one);
        Ls->rhs[k] = (float*)(p + 3 * one);
        Ls->head[k] = Ls->ovf[k] = nullptr;
        Ls->width[k] = Ls->over[k] = 0;
        p += 4 * one;
    }
    OctSegs<OCT_LISTS> t{};
    const uint32_t blocks = oct_segs(B, *Ls, 0xFF, &t);
    if (!blocks) return hipGetLastError();
    hipLaunchKernelGGL(k_oct_count, dim3(blocks), dim3(OCT_BLOCK), 0, s, g, (const uint8_t*)B.lev, t, B.count);
    e = hipMemcpyAsync(got, B.count, sizeof got, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) return e;
    const uint32_t *over = got + OCT_LISTS, *most = got + 2 * OCT_LISTS, *seen = got + 3 * OCT_LISTS;
    bytes = 0;
    for (int L = 0; L < 4; L++) Ls->beside[L] = 0;
    for (int k = 0; k < OCT_LISTS; k++) {
        Ls->width[k] = most[k] <= 6 ? 6 : most[k] <= 12 ? 12 : (int)OCT_WIDE;
        Ls->over[k] = over[k] != 0;
        bytes += up256(4 * (size_t)Ls->width[k] * Ls->counts[k]) + up256(4 * (size_t)over[k]);
        for (int m = 0; m < 4; m++)
            if (seen[k] >> m & 1) {
                Ls->beside[k / 2] |= 1u << m;
                Ls->beside[m] |= 1u << (k / 2);
            }
    }
    if ((e = grow(&Ls->ent, &Ls->ent_cap, bytes)) != hipSuccess) return e;
    p = (char*)Ls->ent;
    for (int k = 0; k < OCT_LISTS; k++) {
        Ls->head[k] = (uint32_t*)p;
        p += up256(4 * (size_t)Ls->width[k] * Ls->counts[k]);
        Ls->ovf[k] = (uint32_t*)p;
        p += up256(4 * (size_t)over[k]);
    }
    oct_segs(B, *Ls, 0xFF, &t);
    hipLaunchKernelGGL(k_oct_fill, dim3(blocks), dim3(OCT_BLOCK), 0, s, g, (const uint8_t*)B.lev, t);
    return hipGetLastError();
}

void octree_free_lists(OctreeLists* Ls) {
    if (!Ls) return;
    for (void** p : {&Ls->dyn, &Ls->ent})
        if (*p) (void)hipFree(*p);
    Ls->dyn = Ls->ent = nullptr;
    Ls->dyn_cap = Ls->ent_cap = 0;
}

int launch_octree_sweeps(const Dims& d, const OctreeBufs& B, const OctreeLists& Ls, int iters, const float* mean,
                         hipStream_t s) {
    OctSegs<OCT_LISTS> all{};
    const uint32_t blocks = oct_segs(B, Ls, 0xFF, &all);
    if (!blocks) return 0;
    const LevelPtrs dl{{B.d[0], B.d[1], B.d[2], B.d[3]}};
    hipLaunchKernelGGL(k_oct_rhs, dim3(blocks), dim3(OCT_BLOCK), 0, s, dl, all, mean);
    if (iters <= 0) return 0;
    OctP P{B.p[0], {}};
    for (int L = 0; L < 4; L++) P.off[L] = (uint32_t)(B.p[L] - B.p[0]);
    const std::vector<uint8_t> plan = oct_schedule(Ls.counts, Ls.beside, iters);
    for (uint8_t mask : plan) {
        OctSegs<4> t{};
        const uint32_t nb = oct_segs(B, Ls, mask, &t);
        hipLaunchKernelGGL(k_oct_gs, dim3(nb), dim3(OCT_BLOCK), 0, s, P, t);
    }
    return (int)plan.size();
}

void launch_octree_adjust(const Dims& d, const OctreeBufs& B, float* u, float* v, float* w, hipStream_t s) {
    const OG g{d.W, d.H, d.D};
    const LevelPtrs P{{B.p[0], B.p[1], B.p[2], B.p[3]}};
    hipLaunchKernelGGL(k_oct_adjust, fine_grid(d), dim3(64, 4), 0, s, g, P, (const uint8_t*)B.lev, u, v, w);
}

void launch_octree_sub_project(const Dims& d, const OctreeBufs& B, float* u, float* v, float* w, hipStream_t s) {
    // level 1 keeps the reference's w write-back (ZQ_SmokeOctreeGrid3D.cpp:1125-1135)
    launch_sub_regular_mask(d, 2, B.leaf[1], u, v, w, 1, s);
    launch_sub_regular_mask(d, 4, B.leaf[2], u, v, w, 0, s);
    launch_sub_regular_mask(d, 8, B.leaf[3], u, v, w, 0, s);
}

}  // namespace zq3d
