// kernels_ensemble.hip -- one launch per stage for a whole ensemble of independent smoke grids.
//
// No reference counterpart.  The members have their own sizes and parameters.  Every stage is a launch
// over a list of tiles, member after member: a record names the member and the cells, and the workgroup
// runs the same per-cell functions (zq3d_stencils.h) that the single-grid kernels run for those cells.
// Each member therefore steps bit for bit as a zq3d_sim of the same configuration (plain FP32
// projection).  A tile of the cell stages is 256 consecutive cells of a plane through a few planes, so
// no lane idles beside a row of odd length, and a face stage does a cell's three faces at once; only
// the projection set-up keeps the single-grid blocks of 64 x 4 cells, whose partial sums it has to
// reproduce.  The red-black sweeps take their tile shape from the ensemble autotuner.
//
// 64 members of 32 to 96 cells an axis (17.5 M cells), us a launch before (64 x 4 blocks found by a
// binary search, one launch a face axis) and now: cell advection 1302, 938; scalar advection 1295, 923;
// MAC to cells 292, 94; set-up 417, 300; cell force 274, 191; vorticity 197, 165; force faces 460, 247;
// face apply 446, 189; correction 468, 152.  All bound by memory or, the advections, by their gathers.
#include "zq3d_ensemble.h"
#include "zq3d_lds.h"
#include "zq3d_sor_quad.h"
#include "zq3d_stencils.h"

namespace zq3d {

namespace {

constexpr int NT = 256;

// the tiles of a table, one a thread; the member by binary search over the members' first tiles
__global__ __launch_bounds__(NT) void ke_tiles(const EnsMember* __restrict__ M, int count,
                                               const int* __restrict__ first, int total, EnsTiling t,
                                               EnsTile* __restrict__ out) {
    const int tile = blockIdx.x * NT + threadIdx.x;
    if (tile >= total) return;
    int lo = 0, hi = count - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first[mid] <= tile) lo = mid;
        else hi = mid - 1;
    }
    const Dims d = M[lo].d;
    const int local = tile - first[lo], per = ens_plane_tiles(d, t), z = local / per, b = local - z * per;
    out[tile] = t.tbx ? EnsTile{lo, b, local, z}
                      : EnsTile{lo, 256 * b, z * kEnsPlanes, min((z + 1) * kEnsPlanes, d.D)};
}

// Runs f(member, i, j, k) over the tiles of table T: cells first .. first + 255 of the plane, planes
// k0 .. k1 - 1.
template <class F>
__device__ __forceinline__ void for_cells(const EnsTable& T, const EnsMember* __restrict__ M, F&& f) {
    for (int tile = blockIdx.x; tile < T.total; tile += gridDim.x) {
        const EnsTile t = T.tiles[tile];
        const EnsMember& m = M[t.member];
        const unsigned at = (unsigned)t.first + threadIdx.x, W = (unsigned)m.d.W;
        const int j = (int)(at / W), i = (int)(at - j * W);
        if (j >= m.d.H) continue;  // past the plane
        for (int k = t.k0; k < t.k1; k++) f(m, i, j, k);
    }
}

// A cell's low u, v and w faces; beside the last column, row and plane also the domain's high face.
template <class F0, class F1, class F2>
__device__ __forceinline__ void cell_faces(const Dims& d, int i, int j, int k, F0&& fu, F1&& fv, F2&& fw) {
    fu(i, j, k);
    if (i == d.W - 1) fu(i + 1, j, k);
    fv(i, j, k);
    if (j == d.H - 1) fv(i, j + 1, k);
    fw(i, j, k);
    if (k == d.D - 1) fw(i, j, k + 1);
}

// Runs f(m, local tile, i, j, k) over a block table of TBX x TBY threads (HALF: half rows).
template <int TBX, int TBY, bool HALF, class F>
__device__ __forceinline__ void for_blocks(const EnsTable& T, const EnsMember* __restrict__ M, F&& f) {
    const int tx = threadIdx.x % TBX, ty = threadIdx.x / TBX;
    for (int tile = blockIdx.x; tile < T.total; tile += gridDim.x) {
        const EnsTile t = T.tiles[tile];
        const EnsMember& m = M[t.member];
        const int gx = ((HALF ? (m.d.W + 1) / 2 : m.d.W) + TBX - 1) / TBX;
        const int by = t.first / gx, bx = t.first - by * gx;
        f(m, t.k0, bx * TBX + tx, by * TBY + ty, t.k1);
    }
}

__global__ __launch_bounds__(NT) void ke_vorticity(const EnsMember* __restrict__ M, EnsTable T) {
    for_cells(T, M, [&](const EnsMember& m, int i, int j, int k) {
        // four planes of the member's N values in its vel4 slot (the advection fills it again)
        st_vorticity_to<float>(m.u, m.v, m.w, VortPlanesOut<float>{(float*)m.vel4, m.d.W * m.d.H * m.d.D}, m.d,
                               m.two_h, i, j, k);
    });
}

__global__ __launch_bounds__(NT) void ke_force_cells(const EnsMember* __restrict__ M, EnsTable T) {
    for_cells(T, M, [&](const EnsMember& m, int i, int j, int k) {
        st_force_cell_from<float, true>(VortPlanesIn<float>{(const float*)m.vel4, m.d.W * m.d.H * m.d.D}, m.T, m.R,
                                        (const float*)nullptr, m.scratch, m.d, m.ch, m.beta, m.alpha, m.Tamb, m.aT,
                                        m.aR, i, j, k);
    });
}

__global__ __launch_bounds__(NT) void ke_force_faces(const EnsMember* __restrict__ M, EnsTable T) {
    for_cells(T, M, [&](const EnsMember& m, int i, int j, int k) {
        cell_faces(
            m.d, i, j, k,
            [&](int x, int y, int z) {
                st_force_face<float, 0, true>(m.u, m.occ, m.scratch, m.d, m.dt, m.dth, m.aV, x, y, z);
            },
            [&](int x, int y, int z) {
                st_force_face<float, 1, true>(m.v, m.occ, m.scratch, m.d, m.dt, m.dth, m.aV, x, y, z);
            },
            [&](int x, int y, int z) {
                st_force_face<float, 2, true>(m.w, m.occ, m.scratch, m.d, m.dt, m.dth, m.aV, x, y, z);
            });
    });
}

// MAC -> cell velocity of the current faces
__global__ __launch_bounds__(NT) void ke_mac_to_cell4(const EnsMember* __restrict__ M, EnsTable T) {
    for_cells(T, M, [&](const EnsMember& m, int i, int j, int k) {
        st_mac_to_cell4<float>(m.u, m.v, m.w, m.vel4, m.d, i, j, k, m.occ);
    });
}

__global__ __launch_bounds__(NT) void ke_advect_cells(const EnsMember* __restrict__ M, EnsTable T) {
    for_cells(T, M, [&](const EnsMember& m, int i, int j, int k) {
        st_advect_cell<float>(m.vel4, m.occ, m.scratch, m.d, StepScale<float>{m.h, m.inv_h}, m.steps, m.dtt, i, j, k);
    });
}

// (the reference's stage always advects with is_open = true, ZQ_SmokeSimulationUtils3D.cpp:2163)
__global__ __launch_bounds__(NT) void ke_cells_to_faces(const EnsMember* __restrict__ M, EnsTable T) {
    for_cells(T, M, [&](const EnsMember& m, int i, int j, int k) {
        cell_faces(
            m.d, i, j, k,
            [&](int x, int y, int z) { st_cells_to_face<float, 0>(m.scratch, m.occ, m.u, m.d, 1, x, y, z); },
            [&](int x, int y, int z) { st_cells_to_face<float, 1>(m.scratch, m.occ, m.v, m.d, 1, x, y, z); },
            [&](int x, int y, int z) { st_cells_to_face<float, 2>(m.scratch, m.occ, m.w, m.d, 1, x, y, z); });
    });
}

__global__ __launch_bounds__(NT) void ke_advect_scalar(const EnsMember* __restrict__ M, EnsTable T) {
    for_cells(T, M, [&](const EnsMember& m, int i, int j, int k) {
        const RegularVelCached<float> V{m.vel4, m.d, {}};
        st_advect_scalar<float, RegularVelCached<float>>(V, m.occ, m.T, m.R, m.T2, m.R2, m.d,
                                                         StepScale<float>{m.h, m.inv_h}, m.steps, m.dtt, i, j, k);
    });
}

// the advected scalars back into place, then the sources
__global__ __launch_bounds__(NT) void ke_reinject(const EnsMember* __restrict__ M, EnsTable T) {
    for_cells(T, M, [&](const EnsMember& m, int i, int j, int k) {
        const int o = cidx(m.d, i, j, k);
        m.T[o] = m.T2[o];
        m.R[o] = m.R2[o];
        for (int q = 0; q < m.n_box; q++) {
            const float* b = m.box[q];
            st_reinject_box<float>(m.T, m.R, m.d, b[0], b[1], b[2], b[3], b[4], b[5], b[6], b[7], i, j, k);
        }
        for (int q = 0; q < m.n_sph; q++) {
            const float* b = m.sph[q];
            st_reinject_sphere<float>(m.T, m.R, m.d, b[0], b[1], b[2], b[3], b[4], b[5], i, j, k);
        }
    });
}

// set-up of the plain projection; the per-tile (sum, count) of the divergence goes to the member's
// partials at the tile's index, as the single-grid set-up writes them per block
__global__ __launch_bounds__(NT) void ke_proj_setup(const EnsMember* __restrict__ M, EnsTable T, int quad) {
    __shared__ double red[4];
    for_blocks<64, 4, false>(T, M, [&](const EnsMember& m, int local, int i, int j, int k) {
        double dsum = 0.0, dcnt = 0.0;
        st_proj_setup_plain(m.u, m.v, m.w, m.occ, m.open_mask, m.nc, quad ? m.qb : m.b, m.p, m.d, i, j, k, dsum, dcnt,
                            quad ? m.qn : nullptr);
        const double sm = block_reduce<false>(dsum, red);
        __syncthreads();
        const double ct = block_reduce<false>(dcnt, red);
        if (threadIdx.x == 0) {
            m.part[2 * local] = sm;
            m.part[2 * local + 1] = ct;
        }
        __syncthreads();
    });
}

// one workgroup of 1024 threads per member
__global__ __launch_bounds__(1024) void ke_finish_mean(const EnsMember* __restrict__ M) {
    __shared__ double ss[1024], sc[1024];
    const int s = blockIdx.x;
    const EnsMember& m = M[s];
    st_fold_mean(m.part, m.tiles, m.mean32, nullptr, m.closed_mean, ss, sc);
}

// one colour of iteration `it` of the red-black SOR; members whose own iteration count is reached
// are left alone
template <int TBX, int TBY>
__global__ __launch_bounds__(NT) void ke_sor_half(const EnsMember* __restrict__ M, EnsTable T, int colour,
                                                 int it) {
    for_blocks<TBX, TBY, true>(T, M, [&](const EnsMember& m, int, int t, int j, int k) {
        if (it >= m.iters) return;
        st_sor_half(m.nc, m.b, m.mean32, m.p, m.d, m.omega, m.omw, colour, t, j, k);
    });
}

// K iterations of every member's SOR in one launch (sor_quad_tile, each member cut by itself).  Members
// with an odd count run one iteration first (K == 1, which takes only those, from zero); launch `at` of
// the pairs then takes every member that still has two to do.
template <int K, int CX, int NTH>
__global__ __launch_bounds__(NTH) void ke_sor_quad(const EnsMember* __restrict__ M, EnsQuadTable T, int at) {
    extern __shared__ float quad_lds[];
    const EnsQuadTile t = T.tiles[blockIdx.x];
    const EnsMember& m = M[t.member];
    const int odd = m.iters & 1;
    if (K == 1 ? !odd : 2 * at + 2 > m.iters - odd) return;
    const QuadCut c = T.cuts[t.member];
    if ((int)threadIdx.x >= 64 * c.nw) return;  // a wave that this member's tiles do not need
    const int from = K == 1 ? 0 : (odd + at) & 1;
    const float* src = K == 1 || (at == 0 && !odd) ? nullptr : m.qp[from];
    sor_quad_tile<K, CX, QUAD_R, true, NTH>(m.qn, m.qb, *m.mean32, src, m.qp[1 - from], m.d, c, t.bx, t.by, t.bz,
                                              m.omega, m.omw, quad_lds);
}

template <class P>
__device__ __forceinline__ void correct_faces(const EnsMember& m, const P& p, int i, int j, int k) {
    cell_faces(
        m.d, i, j, k, [&](int x, int y, int z) { st_correct<0>(m.occ, m.open_mask, p, m.u, m.d, x, y, z); },
        [&](int x, int y, int z) { st_correct<1>(m.occ, m.open_mask, p, m.v, m.d, x, y, z); },
        [&](int x, int y, int z) { st_correct<2>(m.occ, m.open_mask, p, m.w, m.d, x, y, z); });
}

__global__ __launch_bounds__(NT) void ke_correct(const EnsMember* __restrict__ M, EnsTable T, int quad) {
    for_cells(T, M, [&](const EnsMember& m, int i, int j, int k) {
        if (quad) correct_faces(m, QuadPressure{m.qres}, i, j, k);
        else correct_faces(m, PadPressure<float>{m.p}, i, j, k);
    });
}

__global__ __launch_bounds__(NT) void ke_zero(float* __restrict__ dst, size_t n) {
    const size_t stride = (size_t)gridDim.x * NT;
    for (size_t x = (size_t)blockIdx.x * NT + threadIdx.x; x < n; x += stride) dst[x] = 0.0f;
}

inline unsigned grid_of(const EnsTable& T, int blocks) {
    return (unsigned)(blocks > 0 && blocks < T.total ? blocks : (T.total > 0 ? T.total : 1));
}

}  // namespace

// tile layouts of the sweep kernel (TBX x TBY) the autotuner may pick
const int kEnsSweepShapes[kEnsSweepShapeCount][2] = {{64, 4}, {32, 8}, {16, 16}};

hipError_t ens_launch_tiles(const EnsMember* members, int count, const int* first, int total, EnsTiling t, EnsTile* out,
                            hipStream_t s) {
    hipLaunchKernelGGL(ke_tiles, dim3((unsigned)((total + NT - 1) / NT)), dim3(NT), 0, s, members, count, first, total,
                       t, out);
    return hipGetLastError();
}

hipError_t ens_launch_step(const EnsLaunch& L, hipStream_t s) {
    const dim3 nt(NT), gc(grid_of(L.cells, L.blocks));
    const EnsMember* M = L.members;
    // force + attenuation
    hipLaunchKernelGGL(ke_vorticity, gc, nt, 0, s, M, L.cells);
    hipLaunchKernelGGL(ke_force_cells, gc, nt, 0, s, M, L.cells);
    hipLaunchKernelGGL(ke_force_faces, gc, nt, 0, s, M, L.cells);
    // velocity advection (inRegular_outRegular)
    hipLaunchKernelGGL(ke_mac_to_cell4, gc, nt, 0, s, M, L.cells);
    hipLaunchKernelGGL(ke_advect_cells, gc, nt, 0, s, M, L.cells);
    hipLaunchKernelGGL(ke_cells_to_faces, gc, nt, 0, s, M, L.cells);
    // plain projection
    ens_launch_setup(L, s);
    const hipError_t e = ens_launch_sweeps(L, L.max_iters, s);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(ke_correct, gc, nt, 0, s, M, L.cells, L.sweep_quad);
    // scalar advection through the projected velocity, then the sources
    hipLaunchKernelGGL(ke_mac_to_cell4, gc, nt, 0, s, M, L.cells);
    hipLaunchKernelGGL(ke_advect_scalar, gc, nt, 0, s, M, L.cells);
    hipLaunchKernelGGL(ke_reinject, gc, nt, 0, s, M, L.cells);
    return hipGetLastError();
}

void ens_launch_setup(const EnsLaunch& L, hipStream_t s) {
    if (!L.sweep_quad) hipLaunchKernelGGL(ke_zero, dim3(2048), dim3(NT), 0, s, L.p_pool, L.p_pool_size);
    hipLaunchKernelGGL(ke_proj_setup, dim3(grid_of(L.setup, L.blocks)), dim3(NT), 0, s, L.members, L.setup,
                       L.sweep_quad);
    hipLaunchKernelGGL(ke_finish_mean, dim3(L.count), dim3(1024), 0, s, L.members);
}

void ens_launch_probe(const EnsLaunch& L, hipStream_t s) {
    const unsigned gc = grid_of(L.cells, L.blocks);
    hipLaunchKernelGGL(ke_mac_to_cell4, dim3(gc), dim3(NT), 0, s, L.members, L.cells);
    hipLaunchKernelGGL(ke_advect_cells, dim3(gc), dim3(NT), 0, s, L.members, L.cells);
}

namespace {

template <int K, int CX, int NTH>
hipError_t launch_quad(const EnsLaunch& L, const EnsQuadTable& T, int at, hipStream_t s) {
    constexpr int lds = 4 * quad_lds_floats(K, CX, NTH);
    if constexpr (lds > 64 * 1024) {
        static LdsLimit limit;
        const hipError_t e = limit.raise((const void*)ke_sor_quad<K, CX, NTH>, lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((ke_sor_quad<K, CX, NTH>), dim3((unsigned)T.total), dim3(NTH), lds, s, L.members, T, at);
    return hipGetLastError();
}

}  // namespace

hipError_t ens_launch_sweeps(const EnsLaunch& L, int iters, hipStream_t s) {
    const dim3 nt(NT);
    if (L.sweep_quad) {
        const int r = L.sweep_quad - 1;
        const EnsQuadTable& T = L.quad[r];
        hipError_t e = hipSuccess;
        if (L.any_odd && iters > 0) e = launch_quad<1, 2, 512>(L, L.quad_one, 0, s);
        for (int at = 0; 2 * at + 2 <= iters && e == hipSuccess; at++) {
            if (L.quad_shape[r][0] == 4) e = launch_quad<2, 4, 512>(L, T, at, s);
            else if (L.quad_shape[r][1] <= 8) e = launch_quad<2, 2, 512>(L, T, at, s);
            else e = launch_quad<2, 2, 1024>(L, T, at, s);
        }
        return e;
    }
    const EnsTable& H = L.half[L.sweep_shape];
    const unsigned gh = grid_of(H, L.sweep_blocks);
    for (int it = 0; it < iters; it++)
        for (int c = 0; c < 2; c++) {
            switch (L.sweep_shape) {
            case 1: hipLaunchKernelGGL((ke_sor_half<32, 8>), dim3(gh), nt, 0, s, L.members, H, c, it); break;
            case 2: hipLaunchKernelGGL((ke_sor_half<16, 16>), dim3(gh), nt, 0, s, L.members, H, c, it); break;
            default: hipLaunchKernelGGL((ke_sor_half<64, 4>), dim3(gh), nt, 0, s, L.members, H, c, it); break;
            }
        }
    return hipGetLastError();
}

}  // namespace zq3d
