// zq3d_ensemble.h -- device-side description of an ensemble of smoke grids and the launchers of
// kernels_ensemble.hip.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "zq3d_device.h"
#include "zq3d_quad_cut.h"

namespace zq3d {

constexpr int kEnsMaxSources = 4;

// One member: device pointers into the ensemble's pools and its step parameters, precomputed on
// the host exactly as the single-grid launchers compute them.
struct EnsMember {
    Dims d;
    float *u, *v, *w, *T, *R, *T2, *R2;
    uint8_t *occ, *nc;
    float4* vel4;    // cell velocity; also the vorticity scratch of the force stage
    float* scratch;  // 3N: cell force, then advected cell velocity
    float *b, *p;    // divergence, padded pressure
    // quad-layout SOR storage (zq3d_sor_quad.h): counts, right-hand side, the two pressures the sweeps
    // ping-pong between and the one that ends up with the result
    uint8_t* qn;
    float *qb, *qp[2], *qres;
    double* part;    // (sum, count) per set-up tile
    int tiles;       // set-up tiles
    float* mean32;
    float h, dt, dth, two_h, ch, dtt;
    float inv_h;     // 1/h when h is a power of two (backtrace steps multiply), else 0 (they divide)
    int steps;
    float beta, alpha, Tamb, aV, aT, aR;
    int open_mask, closed_mean, iters;
    float omega, omw;
    int n_box, n_sph;
    float box[kEnsMaxSources][8];  // cx, cy, cz, hx, hy, hz (cells), rho, T
    float sph[kEnsMaxSources][6];  // x0, y0, z0 (cells), r^2 (cells^2), rho, T
};

// One tile of a cell table: cells first .. first + 255 (x fastest) of a plane, planes k0 .. k1 - 1.
// Of a block table (TBX x TBY cells of one plane): first = the block's number in the plane, k0 = in the
// member, k1 = the plane.
struct EnsTile {
    int member, first, k0, k1;
};
constexpr int kEnsPlanes = 4;  // planes of a cell tile

// How a stage cuts a plane: blocks of tbx x tby cells (half: of half rows), or, with tbx == 0, the cell tiles.
struct EnsTiling {
    int tbx, tby;
    bool half;
};
__host__ __device__ inline int ens_plane_tiles(const Dims& d, EnsTiling t) {
    if (!t.tbx) return (d.W * d.H + 255) / 256;
    return ((t.half ? (d.W + 1) / 2 : d.W) + t.tbx - 1) / t.tbx * ((d.H + t.tby - 1) / t.tby);
}
__host__ __device__ inline int ens_tiles_of(const Dims& d, EnsTiling t) {
    return ens_plane_tiles(d, t) * (t.tbx ? d.D : (d.D + kEnsPlanes - 1) / kEnsPlanes);
}

// Every member's tiles, member after member.
struct EnsTable {
    const EnsTile* tiles;
    int total;
};

constexpr int kEnsSweepShapeCount = 3;
extern const int kEnsSweepShapes[kEnsSweepShapeCount][2];  // TBX x TBY of the sweep kernel
// cells a lane x waves x planes of the sweeps that run two red-black iterations a launch.  With thousands
// of tiles it is issue that counts, and four cells a lane share the row's neighbours best; then how
// evenly the tiles fill the CUs (one tile of four cells a lane a CU), which depends on the members.  64
// members of 32 to 96 cells an axis (17.5 M cells), us per iteration: 34.5 to 45.6 with two cells a lane;
// with four 37.2 at 8 planes, 28.9 at 16, 24.5 at 32 (the one-iteration launches on colour-split storage
// that these replace took 83.9, the half sweeps at best 175).
constexpr int kEnsQuadShapeCount = 12;
constexpr int kEnsQuadFixed = 7;  // shapes every ensemble has; the rest are the depths of four cells a lane
                                  // that are predicted fastest for its members
constexpr int kEnsQuadShapes[kEnsQuadFixed][3] = {{2, 8, 8}, {2, 8, 16}, {2, 16, 8}, {2, 16, 16},
                                                  {4, 8, 8}, {4, 8, 16}, {4, 8, 32}};
constexpr int kEnsQuadOne[3] = {2, 8, 8};  // the shape of the launch of one iteration

struct EnsQuadTile {
    int member, bx, by, bz;
};

// Every member's tiles, the longest first (workgroups start in this order, so the short ones fill the
// end), and how each member is cut.
struct EnsQuadTable {
    const EnsQuadTile* tiles;
    const QuadCut* cuts;
    int total;
};

struct EnsLaunch {
    const EnsMember* members;  // device array
    int count;
    EnsTable cells, setup;               // cell tiles; 64 x 4 blocks of the projection set-up
    EnsTable half[kEnsSweepShapeCount];  // half-row grids of the sweep, one per tile shape (made on need)
    int sweep_shape;                     // index into kEnsSweepShapes
    EnsQuadTable quad[kEnsQuadShapeCount], quad_one;  // (made on need)
    int quad_shape[kEnsQuadShapeCount][3];
    int sweep_quad;                      // 0: half sweeps of sweep_shape; r > 0: quad_shape[r - 1]
    int any_odd;                         // some member's iteration count is odd
    int blocks;                          // workgroups of the persistent launches (<= 0: one per tile)
    int sweep_blocks;
    int max_iters;
    float* p_pool;
    size_t p_pool_size;
};

// fills a table of `total` tiles of the tiling: member s begins at tile first[s]
hipError_t ens_launch_tiles(const EnsMember* members, int count, const int* first, int total, EnsTiling t, EnsTile* out,
                            hipStream_t s);
// all stages of one step of every member
hipError_t ens_launch_step(const EnsLaunch& L, hipStream_t s);
// projection set-up of every member: counts, divergence and mean, for the selected sweep
void ens_launch_setup(const EnsLaunch& L, hipStream_t s);
// mac -> cell velocity and cell advection of every member: writes only scratch, so it can be
// repeated to time launch shapes
void ens_launch_probe(const EnsLaunch& L, hipStream_t s);
// `iters` red-black iterations of every member's SOR, no more than the member's own count
hipError_t ens_launch_sweeps(const EnsLaunch& L, int iters, hipStream_t s);

}  // namespace zq3d
