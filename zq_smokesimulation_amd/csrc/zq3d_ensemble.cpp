// zq3d_ensemble.cpp -- Part 6 of the C ABI: an ensemble of independent smoke grids of uneven sizes
// stepped together, one persistent launch per stage (kernels_ensemble.hip), the whole step
// captured once in a hipGraph and replayed.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "zq3d_ens_plan.h"
#include "zq3d_ensemble.h"
#include "zq3d_internal.h"
#include "zq3d_kernels.h"
#include "zq_smoke3d.h"

using namespace zq3d;
using namespace zq3d::detail;

struct zq3d_ens {
    int count = 0;
    std::vector<zq3d_config> cfg;
    std::vector<Dims> dims;
    std::vector<EnsMember> host;  // descriptors as uploaded
    EnsMember* dev_members = nullptr;
    std::vector<void*> allocs;
    hipStream_t stream = nullptr;
    EnsLaunch L{};
    // pool offsets per member (elements)
    std::vector<size_t> off_u, off_v, off_w, off_c, off_p, off_part, off_q;
    float *u = nullptr, *v = nullptr, *w = nullptr, *T = nullptr, *R = nullptr, *T2 = nullptr, *R2 = nullptr;
    uint8_t *occ = nullptr, *nc = nullptr;
    float4* vel4 = nullptr;
    float *scratch = nullptr, *b = nullptr, *p = nullptr, *mean32 = nullptr;
    double* part = nullptr;
    uint8_t* quad_n = nullptr;  // quad-layout counts, right-hand sides, pressures (two)
    float *quad_b = nullptr, *quad_p[2] = {nullptr, nullptr};
    size_t Nu = 0, Nv = 0, Nw = 0, Nc = 0, Np = 0, Nparts = 0, Nq = 0;
    long long cells = 0;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    bool graph_stale = true;
};

namespace {

int cdiv(int a, int b) { return (a + b - 1) / b; }

void drop_graph(zq3d_ens* e) {
    if (e->exec) (void)hipGraphExecDestroy(e->exec);
    if (e->graph) (void)hipGraphDestroy(e->graph);
    e->exec = nullptr;
    e->graph = nullptr;
    e->graph_stale = true;
}

int check_member(const zq3d_config& c, const char* where) {
    if (c.struct_size != (int)sizeof(zq3d_config)) { set_err(where, "zq3d_config.struct_size mismatch"); return ZQ3D_ERR_ARG; }
    if (int rc = check_dims(c.width, c.height, c.depth, where)) return rc;
    if (int rc = check_sor_opts(c.sor, where)) return rc;
    if (c.steps < 1 || !(c.voxel_size > 0.0f)) { set_err(where, "steps >= 1 and voxel_size > 0 required"); return ZQ3D_ERR_ARG; }
    if (c.adv_vel_type != 0 || c.adv_sca_type != 2) {
        set_err(where, "ensemble members use ADV_VEL_INREG_OUTREG and ADV_SCA_REG");
        return ZQ3D_ERR_ARG;
    }
    if (c.sor.mixed_precision) {
        set_err(where, "ensemble members use the plain FP32 projection (a fixed sweep count, so a step can be captured)");
        return ZQ3D_ERR_ARG;
    }
    return ZQ3D_OK;
}

template <class T>
int ens_alloc(zq3d_ens* e, T** p, size_t bytes) {
    void* q = nullptr;
    if (hipMalloc(&q, bytes ? bytes : 1) != hipSuccess) return 1;
    e->allocs.push_back(q);
    *p = (T*)q;
    return 0;
}

// Columns of tiles of the same waves and planes.
struct QuadColumns {
    int nw, D;
    long long n;
};

// The members' tile columns under shapes of cx cells a lane and nw waves.
std::vector<QuadColumns> quad_columns(const zq3d_ens* e, int cx, int nw) {
    std::vector<QuadColumns> all;
    for (int s = 0; s < e->count; s++) {
        const Dims& d = e->dims[s];
        const Dims* last = s ? &e->dims[s - 1] : nullptr;
        if (last && last->W == d.W && last->H == d.H && last->D == d.D) {
            all.push_back(all.back());
            continue;
        }
        const QuadCut c = quad_cut(d.W, d.H, d.D, 2, cx, nw, 2);
        all.push_back(QuadColumns{c.nw, d.D, (long long)c.nx * c.ny});
    }
    std::sort(all.begin(), all.end(),
              [](const QuadColumns& x, const QuadColumns& y) { return x.nw != y.nw ? x.nw < y.nw : x.D < y.D; });
    size_t n = 0;
    for (const QuadColumns& c : all)
        if (n && all[n - 1].nw == c.nw && all[n - 1].D == c.D) all[n - 1].n += c.n;
        else all[n++] = c;
    all.resize(n);
    return all;
}

// Microseconds that a launch of two iterations with chunks of zc planes is predicted to take.
double quad_us(const std::vector<QuadColumns>& columns, int cx, int zc) {
    // tiles by their steps and waves, which set their time
    constexpr int MOST = 17;
    std::vector<long long> tiles((size_t)(zc + 8) * MOST, 0);
    for (const QuadColumns& q : columns) {
        QuadCut c{};
        c.zc = zc;
        c.nz = quad_chunks(q.D, 2, zc);
        // (all chunks but the last take the same steps)
        tiles[(size_t)ens_chunk_steps(c, 2, 0, q.D) * MOST + q.nw] += q.n * (c.nz - 1);
        tiles[(size_t)ens_chunk_steps(c, 2, c.nz - 1, q.D) * MOST + q.nw] += q.n;
    }
    std::vector<EnsRun> runs;
    for (size_t k = 0; k < tiles.size(); k++)
        if (tiles[k]) runs.push_back(EnsRun{ens_tile_us((int)(k / MOST), 2, cx, (int)(k % MOST)), tiles[k]});
    std::sort(runs.begin(), runs.end(), [](const EnsRun& x, const EnsRun& y) { return x.us > y.us; });
    return ens_fill_us(runs);
}

// The shapes of an ensemble: the fixed ones, then the depths of four cells a lane predicted fastest;
// returns the shape predicted fastest of all.
int quad_shapes(const zq3d_ens* e, int (*shapes)[3]) {
    struct Depth {
        double us;
        int zc;
    };
    std::vector<Depth> depths;
    double best_us = 0.0;
    int n = 0, best = 0;
    auto add = [&](int cx, int nw, int zc, double us) {
        shapes[n][0] = cx, shapes[n][1] = nw, shapes[n][2] = zc;
        if (n == 0 || us < best_us) {
            best_us = us;
            best = n;
        }
        n++;
    };
    std::vector<QuadColumns> columns;
    for (int k = 0; k < kEnsQuadFixed; k++) {
        const auto& f = kEnsQuadShapes[k];
        if (!k || f[0] != kEnsQuadShapes[k - 1][0] || f[1] != kEnsQuadShapes[k - 1][1])
            columns = quad_columns(e, f[0], f[1]);
        add(f[0], f[1], f[2], quad_us(columns, f[0], f[2]));
    }
    columns = quad_columns(e, 4, 8);
    for (int zc = 2; zc <= 64; zc += 2) {
        bool had = false;
        for (const auto& f : kEnsQuadShapes) had = had || (f[0] == 4 && f[2] == zc);
        if (!had) depths.push_back(Depth{quad_us(columns, 4, zc), zc});
    }
    std::stable_sort(depths.begin(), depths.end(), [](const Depth& a, const Depth& b) { return a.us < b.us; });
    for (int i = 0; n < kEnsQuadShapeCount; i++) add(4, 8, depths[i].zc, depths[i].us);
    return best;
}

// The table of a shape: every member's cut, and the tiles, the longest first.  Made when the shape is first
// selected (most ensembles run one).
int make_quad_table(zq3d_ens* e, int K, const int shape[3], EnsQuadTable* table, const char* where) {
    if (table->total) return ZQ3D_OK;
    struct Chunk {
        double us;
        int s, z, nx, ny;
    };
    std::vector<Chunk> chunks;
    std::vector<QuadCut> cuts;
    size_t total = 0;
    for (int s = 0; s < e->count; s++) {
        const Dims& d = e->dims[s];
        const QuadCut c = quad_cut(d.W, d.H, d.D, K, shape[0], shape[1], shape[2]);
        cuts.push_back(c);
        for (int z = 0; z < c.nz; z++)
            chunks.push_back(Chunk{ens_tile_us(ens_chunk_steps(c, K, z, d.D), K, shape[0], c.nw), s, z, c.nx, c.ny});
        total += (size_t)c.nx * c.ny * c.nz;
    }
    std::stable_sort(chunks.begin(), chunks.end(), [](const Chunk& a, const Chunk& b) { return a.us > b.us; });
    std::vector<EnsQuadTile> tiles;
    tiles.reserve(total);
    for (const Chunk& c : chunks)
        for (int y = 0; y < c.ny; y++)
            for (int x = 0; x < c.nx; x++) tiles.push_back(EnsQuadTile{c.s, x, y, c.z});
    EnsQuadTile* dt = nullptr;
    QuadCut* dc = nullptr;
    if (ens_alloc(e, &dt, tiles.size() * sizeof(EnsQuadTile)) || ens_alloc(e, &dc, cuts.size() * sizeof(QuadCut))) {
        set_err(where, "device allocation failed");
        return ZQ3D_ERR_HIP;
    }
    ZQ_HIP(hipMemcpy(dt, tiles.data(), tiles.size() * sizeof(EnsQuadTile), hipMemcpyHostToDevice), where);
    ZQ_HIP(hipMemcpy(dc, cuts.data(), cuts.size() * sizeof(QuadCut), hipMemcpyHostToDevice), where);
    *table = EnsQuadTable{dt, dc, (int)tiles.size()};
    return ZQ3D_OK;
}

// The table of a cell or block stage, written on the device from the members' first tiles.
int make_table(zq3d_ens* e, EnsTiling t, EnsTable* table, const char* where) {
    if (table->total) return ZQ3D_OK;
    std::vector<int> first(1, 0);
    for (const Dims& d : e->dims) first.push_back(first.back() + ens_tiles_of(d, t));
    EnsTile* tiles = nullptr;
    int* dev = nullptr;
    if (ens_alloc(e, &tiles, (size_t)first.back() * sizeof(EnsTile)) ||
        ens_alloc(e, &dev, first.size() * sizeof(int))) {
        set_err(where, "device allocation failed");
        return ZQ3D_ERR_HIP;
    }
    ZQ_HIP(hipMemcpyAsync(dev, first.data(), first.size() * sizeof(int), hipMemcpyHostToDevice, e->stream), where);
    ZQ_HIP(ens_launch_tiles(e->dev_members, e->count, dev, first.back(), t, tiles, e->stream), where);
    ZQ_HIP(hipStreamSynchronize(e->stream), where);
    *table = EnsTable{tiles, first.back()};
    return ZQ3D_OK;
}

// The tables of the sweeps that L selects.
int make_sweep_tables(zq3d_ens* e, EnsLaunch* L, const char* where) {
    if (!L->sweep_quad) {
        const int* shape = kEnsSweepShapes[L->sweep_shape];
        return make_table(e, EnsTiling{shape[0], shape[1], true}, &L->half[L->sweep_shape], where);
    }
    if (L->any_odd)
        if (int rc = make_quad_table(e, 1, kEnsQuadOne, &L->quad_one, where)) return rc;
    return make_quad_table(e, 2, L->quad_shape[L->sweep_quad - 1], &L->quad[L->sweep_quad - 1], where);
}

int field_span(zq3d_ens* e, int s, int field, void** p, size_t* bytes) {
    const Sizes z(e->dims[s]);
    switch (field) {
    case ZQ3D_FIELD_U: *p = e->u + e->off_u[s]; *bytes = z.Nu * 4; return 0;
    case ZQ3D_FIELD_V: *p = e->v + e->off_v[s]; *bytes = z.Nv * 4; return 0;
    case ZQ3D_FIELD_W: *p = e->w + e->off_w[s]; *bytes = z.Nw * 4; return 0;
    case ZQ3D_FIELD_T: *p = e->T + e->off_c[s]; *bytes = z.N * 4; return 0;
    case ZQ3D_FIELD_RHO: *p = e->R + e->off_c[s]; *bytes = z.N * 4; return 0;
    case ZQ3D_FIELD_OCC: *p = e->occ + e->off_c[s]; *bytes = z.N; return 0;
    default: return 1;
    }
}

int upload_members(zq3d_ens* e, const char* where) {
    ZQ_HIP(hipMemcpyAsync(e->dev_members, e->host.data(), sizeof(EnsMember) * e->count, hipMemcpyHostToDevice,
                          e->stream),
           where);
    ZQ_HIP(hipStreamSynchronize(e->stream), where);
    return ZQ3D_OK;
}

}  // namespace

extern "C" int zq3d_ens_create(int count, const zq3d_config* cfgs, zq3d_ens** out) {
    const char* where = "zq3d_ens_create";
    if (!out || !cfgs || count < 1) { set_err(where, "bad argument"); return ZQ3D_ERR_ARG; }
    *out = nullptr;
    for (int s = 0; s < count; s++)
        if (int rc = check_member(cfgs[s], where)) return rc;
    zq3d_ens* e = new zq3d_ens();
    e->count = count;
    e->cfg.assign(cfgs, cfgs + count);
    for (int s = 0; s < count; s++) {
        const Dims d{cfgs[s].width, cfgs[s].height, cfgs[s].depth};
        const Sizes z(d);
        e->dims.push_back(d);
        e->off_u.push_back(e->Nu);
        e->off_v.push_back(e->Nv);
        e->off_w.push_back(e->Nw);
        e->off_c.push_back(e->Nc);
        e->off_p.push_back(e->Np);
        e->off_part.push_back(e->Nparts);
        e->off_q.push_back(e->Nq);
        e->Nq += quad_cells(d);
        e->Nu += z.Nu;
        e->Nv += z.Nv;
        e->Nw += z.Nw;
        e->Nc += z.N;
        e->Np += z.Np;
        e->Nparts += 2 * (size_t)cdiv(d.W, 64) * cdiv(d.H, 4) * d.D;
        e->cells += (long long)z.N;
    }
    int bad = 0;
    bad |= ens_alloc(e, &e->u, e->Nu * 4) | ens_alloc(e, &e->v, e->Nv * 4) | ens_alloc(e, &e->w, e->Nw * 4);
    bad |= ens_alloc(e, &e->T, e->Nc * 4) | ens_alloc(e, &e->R, e->Nc * 4) | ens_alloc(e, &e->T2, e->Nc * 4) |
           ens_alloc(e, &e->R2, e->Nc * 4);
    bad |= ens_alloc(e, &e->occ, e->Nc) | ens_alloc(e, &e->nc, e->Nc) | ens_alloc(e, &e->vel4, e->Nc * 16);
    bad |= ens_alloc(e, &e->scratch, (e->Nu + e->Nv + e->Nw) * 4) | ens_alloc(e, &e->b, e->Nc * 4) |
           ens_alloc(e, &e->p, e->Np * 4);
    bad |= ens_alloc(e, &e->part, e->Nparts * 8) | ens_alloc(e, &e->mean32, (size_t)count * 4);
    bad |= ens_alloc(e, &e->quad_n, e->Nq) | ens_alloc(e, &e->quad_b, e->Nq * 4) |
           ens_alloc(e, &e->quad_p[0], e->Nq * 4) | ens_alloc(e, &e->quad_p[1], e->Nq * 4);
    bad |= ens_alloc(e, &e->dev_members, sizeof(EnsMember) * count);
    if (bad || hipStreamCreate(&e->stream) != hipSuccess) {
        set_err(where, "device allocation failed");
        zq3d_ens_destroy(e);
        return ZQ3D_ERR_HIP;
    }
    size_t off_scr = 0;
    for (int s = 0; s < count; s++) {
        const zq3d_config& c = cfgs[s];
        const Dims d = e->dims[s];
        const Sizes z(d);
        EnsMember m;
        std::memset(&m, 0, sizeof(m));
        m.d = d;
        m.u = e->u + e->off_u[s];
        m.v = e->v + e->off_v[s];
        m.w = e->w + e->off_w[s];
        m.T = e->T + e->off_c[s];
        m.R = e->R + e->off_c[s];
        m.T2 = e->T2 + e->off_c[s];
        m.R2 = e->R2 + e->off_c[s];
        m.occ = e->occ + e->off_c[s];
        m.nc = e->nc + e->off_c[s];
        m.vel4 = e->vel4 + e->off_c[s];
        m.scratch = e->scratch + off_scr;
        off_scr += z.Nu + z.Nv + z.Nw;
        m.b = e->b + e->off_c[s];
        m.p = e->p + e->off_p[s];
        m.part = e->part + e->off_part[s];
        m.tiles = cdiv(d.W, 64) * cdiv(d.H, 4) * d.D;
        m.mean32 = e->mean32 + s;
        m.qn = e->quad_n + e->off_q[s];
        m.qb = e->quad_b + e->off_q[s];
        for (int q = 0; q < 2; q++) m.qp[q] = e->quad_p[q] + e->off_q[s];
        // launches that write this member's pressure: the odd iteration and the pairs
        m.qres = m.qp[(c.sor.iters + 1) / 2 & 1];
        // the single-grid launchers' host arithmetic (launch_force_atten, launch_advect_*, launch_sor)
        m.h = c.voxel_size;
        m.inv_h = step_scale<float>(c.voxel_size).inv;
        m.dt = c.step_time;
        m.dth = c.step_time * 0.5f;
        m.two_h = 2.0f * c.voxel_size;
        m.ch = c.confine * c.voxel_size;
        m.dtt = c.step_time / c.steps;
        m.steps = c.steps;
        m.beta = c.buoyancy;
        m.alpha = c.gravity;
        m.Tamb = c.Tamb;
        m.aV = c.vel_atten;
        m.aT = c.temp_atten;
        m.aR = c.dens_atten;
        m.open_mask = c.sor.open_mask;
        m.closed_mean = c.sor.closed_mean ? 1 : 0;
        m.iters = c.sor.iters;
        m.omega = c.sor.omega;
        m.omw = 1.0f - c.sor.omega;
        e->host.push_back(m);
        e->L.max_iters = std::max(e->L.max_iters, c.sor.iters);
        e->L.any_odd |= c.sor.iters & 1;
    }
    Errs E;
    E(hipMemsetAsync(e->u, 0, e->Nu * 4, e->stream));
    E(hipMemsetAsync(e->v, 0, e->Nv * 4, e->stream));
    E(hipMemsetAsync(e->w, 0, e->Nw * 4, e->stream));
    E(hipMemsetAsync(e->T, 0, e->Nc * 4, e->stream));
    E(hipMemsetAsync(e->R, 0, e->Nc * 4, e->stream));
    E(hipMemsetAsync(e->occ, 0, e->Nc, e->stream));
    E(hipMemsetAsync(e->p, 0, e->Np * 4, e->stream));
    E(hipMemsetAsync(e->nc, 0, e->Nc, e->stream));
    E(hipMemsetAsync(e->b, 0, e->Nc * 4, e->stream));
    // a member of no iterations keeps this pressure
    E(hipMemsetAsync(e->quad_p[0], 0, e->Nq * 4, e->stream));
    if (E.e != hipSuccess) {
        set_err(where, hipGetErrorString(E.e));
        zq3d_ens_destroy(e);
        return ZQ3D_ERR_HIP;
    }
    EnsLaunch& L = e->L;
    L.members = e->dev_members;
    L.count = count;
    L.sweep_shape = 0;
    L.sweep_quad = quad_shapes(e, L.quad_shape) + 1;
    L.blocks = 0;
    L.sweep_blocks = 0;
    L.p_pool = e->p;
    L.p_pool_size = e->Np;
    int rc = upload_members(e, where);
    if (!rc) rc = make_table(e, EnsTiling{0, 0, false}, &L.cells, where);
    if (!rc) rc = make_table(e, EnsTiling{64, 4, false}, &L.setup, where);
    if (!rc) rc = make_sweep_tables(e, &L, where);
    if (rc) {
        zq3d_ens_destroy(e);
        return rc;
    }
    *out = e;
    return ZQ3D_OK;
}

extern "C" void zq3d_ens_destroy(zq3d_ens* e) {
    if (!e) return;
    if (e->stream) (void)hipStreamSynchronize(e->stream);
    drop_graph(e);
    for (void* p : e->allocs) (void)hipFree(p);
    if (e->stream) (void)hipStreamDestroy(e->stream);
    delete e;
}

extern "C" int zq3d_ens_set_sources(zq3d_ens* e, int member, int n_box, const float* boxes8, int n_sphere,
                                    const float* spheres6) {
    const char* where = "zq3d_ens_set_sources";
    if (!e || member < 0 || member >= e->count || n_box < 0 || n_sphere < 0 || n_box > kEnsMaxSources ||
        n_sphere > kEnsMaxSources || (n_box && !boxes8) || (n_sphere && !spheres6)) {
        set_err(where, "bad argument (at most 4 box and 4 sphere sources per member)");
        return ZQ3D_ERR_ARG;
    }
    EnsMember& m = e->host[member];
    const Dims d = e->dims[member];
    m.n_box = n_box;
    m.n_sph = n_sphere;
    for (int q = 0; q < n_box; q++) {
        const float* b = boxes8 + 8 * q;
        // launch_reinject_box: centre and half extents scaled by the grid on the host
        const float v[8] = {b[0] * d.W, b[1] * d.H, b[2] * d.D, b[3] * d.W, b[4] * d.H, b[5] * d.D, b[6], b[7]};
        std::memcpy(m.box[q], v, sizeof(v));
    }
    for (int q = 0; q < n_sphere; q++) {
        const float* sp = spheres6 + 6 * q;
        const float rr = sp[3] * d.W;  // launch_reinject_sphere
        const float v[6] = {sp[0] * d.W, sp[1] * d.H, sp[2] * d.D, rr * rr, sp[4], sp[5]};
        std::memcpy(m.sph[q], v, sizeof(v));
    }
    return upload_members(e, where);
}

extern "C" int zq3d_ens_upload(zq3d_ens* e, int member, int field, const void* host, size_t bytes) {
    const char* where = "zq3d_ens_upload";
    if (!e || !host || member < 0 || member >= e->count) { set_err(where, "bad argument"); return ZQ3D_ERR_ARG; }
    void* p;
    size_t n;
    if (field_span(e, member, field, &p, &n)) { set_err(where, "unknown field"); return ZQ3D_ERR_ARG; }
    if (n != bytes) { set_err(where, "size mismatch"); return ZQ3D_ERR_ARG; }
    ZQ_HIP(hipMemcpyAsync(p, host, n, hipMemcpyHostToDevice, e->stream), where);
    ZQ_HIP(hipStreamSynchronize(e->stream), where);
    return ZQ3D_OK;
}

extern "C" int zq3d_ens_download(zq3d_ens* e, int member, int field, void* host, size_t bytes) {
    const char* where = "zq3d_ens_download";
    if (!e || !host || member < 0 || member >= e->count) { set_err(where, "bad argument"); return ZQ3D_ERR_ARG; }
    void* p;
    size_t n;
    if (field_span(e, member, field, &p, &n)) { set_err(where, "unknown field"); return ZQ3D_ERR_ARG; }
    if (n != bytes) { set_err(where, "size mismatch"); return ZQ3D_ERR_ARG; }
    ZQ_HIP(hipMemcpyAsync(host, p, n, hipMemcpyDeviceToHost, e->stream), where);
    ZQ_HIP(hipStreamSynchronize(e->stream), where);
    return ZQ3D_OK;
}

extern "C" int zq3d_ens_step(zq3d_ens* e, int steps, int use_graph) {
    const char* where = "zq3d_ens_step";
    if (!e || steps < 0) { set_err(where, "bad argument"); return ZQ3D_ERR_ARG; }
    if (!use_graph) {
        for (int n = 0; n < steps; n++) ZQ_HIP(ens_launch_step(e->L, e->stream), where);
        return ZQ3D_OK;
    }
    if (e->graph_stale) {
        drop_graph(e);
        ZQ_HIP(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal), where);
        const hipError_t cap = ens_launch_step(e->L, e->stream);
        const hipError_t end = hipStreamEndCapture(e->stream, &e->graph);
        ZQ_HIP(cap, where);
        ZQ_HIP(end, where);
        ZQ_HIP(hipGraphInstantiate(&e->exec, e->graph, nullptr, nullptr, 0), where);
        e->graph_stale = false;
    }
    for (int n = 0; n < steps; n++) ZQ_HIP(hipGraphLaunch(e->exec, e->stream), where);
    return ZQ3D_OK;
}

extern "C" int zq3d_ens_synchronize(zq3d_ens* e) {
    if (!e) { set_err("zq3d_ens_synchronize", "null ensemble"); return ZQ3D_ERR_ARG; }
    ZQ_HIP(hipStreamSynchronize(e->stream), "zq3d_ens_synchronize");
    return ZQ3D_OK;
}

extern "C" long long zq3d_ens_cells(zq3d_ens* e) { return e ? e->cells : 0; }

extern "C" int zq3d_ens_stream(zq3d_ens* e, void** stream) {
    if (!e || !stream) { set_err("zq3d_ens_stream", "bad argument"); return ZQ3D_ERR_ARG; }
    *stream = e->stream;
    return ZQ3D_OK;
}

extern "C" int zq3d_ens_set_sweep(zq3d_ens* e, int kind, int tbx, int tby, int blocks) {
    const char* where = "zq3d_ens_set_sweep";
    if (!e) { set_err(where, "null ensemble"); return ZQ3D_ERR_ARG; }
    EnsLaunch L = e->L;
    bool ok = false;
    if (kind == 0) {
        for (int sh = 0; sh < kEnsSweepShapeCount; sh++)
            if (kEnsSweepShapes[sh][0] == tbx && kEnsSweepShapes[sh][1] == tby && blocks >= 0) {
                L.sweep_quad = 0;
                L.sweep_shape = sh;
                L.sweep_blocks = blocks;
                ok = true;
            }
    } else if (kind == 1) {
        // saved shapes of the sweeps on 64 slots that these replaced: the nearest one here (same bits)
        static const int old[][2] = {{8, 8}, {8, 16}, {16, 8}, {16, 16}, {16, 32}, {32, 8}, {32, 16}};
        if (tbx == 64)
            for (const auto& o : old)
                if (o[0] == tby && o[1] == blocks) {
                    tbx = 2;
                    tby = tby == 8 ? 8 : 16;
                    blocks = blocks == 8 ? 8 : 16;
                    break;
                }
        for (int r = 0; r < kEnsQuadShapeCount; r++)
            if (L.quad_shape[r][0] == tbx && L.quad_shape[r][1] == tby && L.quad_shape[r][2] == blocks) {
                L.sweep_quad = r + 1;
                ok = true;
            }
    }
    if (!ok) { set_err(where, "not a sweep candidate (see zq3d_ens_autotune)"); return ZQ3D_ERR_ARG; }
    if (int rc = make_sweep_tables(e, &L, where)) return rc;
    e->L = L;
    e->graph_stale = true;
    return ZQ3D_OK;
}

extern "C" int zq3d_ens_get_sweep(zq3d_ens* e, int* kind, int* tbx, int* tby, int* blocks) {
    if (!e || !kind || !tbx || !tby || !blocks) { set_err("zq3d_ens_get_sweep", "null argument"); return ZQ3D_ERR_ARG; }
    const EnsLaunch& L = e->L;
    const int* quad = L.sweep_quad ? L.quad_shape[L.sweep_quad - 1] : nullptr;
    *kind = quad ? 1 : 0;
    *tbx = quad ? quad[0] : kEnsSweepShapes[L.sweep_shape][0];
    *tby = quad ? quad[1] : kEnsSweepShapes[L.sweep_shape][1];
    *blocks = quad ? quad[2] : L.sweep_blocks;
    return ZQ3D_OK;
}

// Times the sweep kernel for every tile shape and persistent-launch size, and the cell kernels for
// every launch size, on the ensemble's own grids; keeps the fastest of each.  The fields are left
// as they were (only projection and advection scratch is written).
extern "C" int zq3d_ens_autotune(zq3d_ens* e, int iters, zq3d_ens_tune* rep) {
    const char* where = "zq3d_ens_autotune";
    if (!e || iters < 1) { set_err(where, "bad argument"); return ZQ3D_ERR_ARG; }
    static const int blocks[] = {0, 256, 1024, 4096};
    const int nb = (int)(sizeof(blocks) / sizeof(blocks[0]));
    // (kept also where tuning fails later on)
    for (int sh = 0; sh < kEnsSweepShapeCount; sh++) {
        const EnsTiling t{kEnsSweepShapes[sh][0], kEnsSweepShapes[sh][1], true};
        if (int rc = make_table(e, t, &e->L.half[sh], where)) return rc;
    }
    for (int r = 0; r < kEnsQuadShapeCount; r++)
        if (int rc = make_quad_table(e, 2, e->L.quad_shape[r], &e->L.quad[r], where)) return rc;
    if (e->L.any_odd)
        if (int rc = make_quad_table(e, 1, kEnsQuadOne, &e->L.quad_one, where)) return rc;
    hipEvent_t a = nullptr, b = nullptr;
    ZQ_HIP(hipEventCreate(&a), where);
    ZQ_HIP(hipEventCreate(&b), where);
    if (rep) std::memset(rep, 0, sizeof(*rep));
    EnsLaunch L = e->L;
    Errs E;
    auto time_it = [&](auto&& launch) {
        launch();  // warm
        E(hipEventRecord(a, e->stream));
        launch();
        E(hipEventRecord(b, e->stream));
        E(hipEventSynchronize(b));
        float ms = 0.0f;
        E(hipEventElapsedTime(&ms, a, b));
        return ms;
    };
    // the sweeps run on the live counts and right-hand sides (interleaved and quad layout)
    for (int q = 0; q < 2; q++) {
        L.sweep_quad = q;
        ens_launch_setup(L, e->stream);
    }
    int best_sh = 0, best_sb = 0, best_quad = 0;
    float best = -1.0f;
    int n = 0;
    auto consider = [&](int tbx, int tby, int blk, float us, int sh, int sb, int quad) {
        if (rep && n < ZQ3D_ENS_TUNE_MAX) {
            rep->kind[n] = quad ? 1 : 0;
            rep->tbx[n] = tbx;
            rep->tby[n] = tby;
            rep->blocks[n] = blk;
            rep->us_per_iter[n] = us;
            n++;
        }
        if (best < 0.0f || us < best) {
            best = us;
            best_sh = sh;
            best_sb = sb;
            best_quad = quad;
        }
    };
    L.sweep_quad = 0;
    for (int sh = 0; sh < kEnsSweepShapeCount; sh++)
        for (int bi = 0; bi < nb; bi++) {
            L.sweep_shape = sh;
            L.sweep_blocks = blocks[bi];
            const float ms = time_it([&] { E(ens_launch_sweeps(L, iters, e->stream)); });
            consider(kEnsSweepShapes[sh][0], kEnsSweepShapes[sh][1], blocks[bi], 1e3f * ms / iters, sh, blocks[bi], 0);
        }
    const int even = (iters + 1) & ~1;  // two iterations a launch
    for (int r = 0; r < kEnsQuadShapeCount; r++) {
        L.sweep_quad = r + 1;
        const float ms = time_it([&] { E(ens_launch_sweeps(L, even, e->stream)); });
        consider(L.quad_shape[r][0], L.quad_shape[r][1], L.quad_shape[r][2], 1e3f * ms / even, 0, 0, r + 1);
    }
    L.sweep_shape = best_sh;
    L.sweep_blocks = best_sb;
    L.sweep_quad = best_quad;
    int best_b = 0;
    float best_cell = -1.0f;
    for (int bi = 0; bi < nb; bi++) {
        L.blocks = blocks[bi];
        const float ms = time_it([&] { ens_launch_probe(L, e->stream); });
        if (best_cell < 0.0f || ms < best_cell) {
            best_cell = ms;
            best_b = blocks[bi];
        }
    }
    L.blocks = best_b;
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    if (E.e != hipSuccess) { set_err(where, hipGetErrorString(E.e)); return ZQ3D_ERR_HIP; }
    e->L = L;
    e->graph_stale = true;
    if (rep) {
        rep->count = n;
        rep->best_kind = best_quad ? 1 : 0;
        rep->best_tbx = best_quad ? L.quad_shape[best_quad - 1][0] : kEnsSweepShapes[best_sh][0];
        rep->best_tby = best_quad ? L.quad_shape[best_quad - 1][1] : kEnsSweepShapes[best_sh][1];
        rep->best_sweep_blocks = best_quad ? L.quad_shape[best_quad - 1][2] : best_sb;
        rep->best_us_per_iter = best;
        rep->best_blocks = best_b;
        rep->probe_ms = best_cell;
    }
    return ZQ3D_OK;
}
