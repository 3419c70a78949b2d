// Host driver of the warp-field solver: capacity allocation, the once-per-solve
// index build and the Gauss-Newton loop over a batch of solves, behind the
// C-ABI of include/sh/warp_solver.h.
//
// Mirrors WarpSolver (examples/mono_star/opt/WarpSolver.cu:50-389) without its
// host synchronisation inside the GN loop: the reference synchronises four
// streams and downloads residuals every iteration (DenseImageDebug.cu:5-27,
// NodeGraphHandler.cu:111-139, WarpSolverPCG.cu:19-31); here the index build
// reads back two counts (valid pixels, unique node pairs) and the GN loop runs
// without any host round trip.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "sh_common.hpp"
#include "sh_engine.hpp"
#include "sh_kernels.hpp"

namespace sh
{
namespace
{
inline uint32_t div_up(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

#define SH_HIP(call)                                                                                                   \
    do                                                                                                                 \
    {                                                                                                                  \
        const hipError_t e_ = (call);                                                                                  \
        if (e_ != hipSuccess)                                                                                          \
        {                                                                                                              \
            last_hip_error = e_;                                                                                       \
            return SH_E_HIP;                                                                                           \
        }                                                                                                              \
    } while (0)
} // namespace

hipError_t last_hip_error = hipSuccess;

Engine::~Engine() { release(); }

void Engine::release()
{
    for (void *p : allocs_)
        (void)hipFree(p);
    allocs_.clear();
    for (Slot &sl : slots_)
    {
        if (sl.part_buf)
            (void)hipFree(sl.part_buf);
        sl.part_buf = nullptr;
        sl.part_bytes = 0;
        if (sl.tile_buf)
            (void)hipFree(sl.tile_buf);
        sl.tile_buf = nullptr;
        sl.tile_bytes = 0;
    }
    for (char *&h : gws_.h_tab)
    {
        if (h)
            (void)hipHostFree(h);
        h = nullptr;
    }
    if (gws_.h_out)
        (void)hipHostFree(gws_.h_out);
    gws_ = GroupWs{};
    if (h_meta_)
        (void)hipHostFree(h_meta_);
    h_meta_ = nullptr;
    if (h_flag_)
        (void)hipHostFree(h_flag_);
    h_flag_ = nullptr;
    if (h_stage_)
        (void)hipHostFree(h_stage_);
    h_stage_ = nullptr;
    if (graph_exec_)
        (void)hipGraphExecDestroy(graph_exec_);
    graph_exec_ = nullptr;
    if (cap_stream_)
        (void)hipStreamDestroy(cap_stream_);
    cap_stream_ = nullptr;
    for (Mark &m : marks_)
        (void)hipEventDestroy(m.ev);
    marks_.clear();
    if (sync_ev_)
        (void)hipEventDestroy(sync_ev_);
    sync_ev_ = nullptr;
    if (index_ev_)
        (void)hipEventDestroy(index_ev_);
    index_ev_ = nullptr;
    n_marks_ = 0;
}

int Engine::alloc(void **p, size_t bytes)
{
    *p = nullptr;
    if (bytes == 0)
        bytes = 16;
    bytes = (bytes + 255) & ~size_t(255);
    const hipError_t e = hipMalloc(p, bytes);
    if (e != hipSuccess)
    {
        last_hip_error = e;
        *p = nullptr;
        return SH_E_NOMEM;
    }
    allocs_.push_back(*p);
    bytes_ += bytes;
    return SH_OK;
}

int Engine::init(const sh_solver_config &c, uint32_t max_slots)
{
    if (c.knn != 4 && c.knn != 8)
        return SH_E_ARG;
    if (c.max_nodes < c.knn || c.max_nodes > kPairBase || c.max_width == 0 || c.max_height == 0 || max_slots == 0)
        return SH_E_ARG;
    if (c.pcg_iterations == 0 || c.pcg_iterations > 1000 || c.gn_iterations > 1000)
        return SH_E_ARG;
    if (c.stream_precision > SH_STREAM_FP16 || c.spmv_mode > SH_SPMV_AUTO || (c.flags & ~2047u) ||
        ((c.flags & SH_FLAG_TILE_PIX_64) && (c.flags & SH_FLAG_TILE_PIX_256)))
        return SH_E_ARG;
    cfg_ = c;
    if (cfg_.flags & SH_FLAG_PAIR_MAJOR)
        cfg_.flags |= SH_FLAG_REFERENCE_INDEX;
    K_ = int(c.knn);
    fp16_ = (c.stream_precision == SH_STREAM_FP16);
    const uint32_t np = uint32_t(K_ * (K_ - 1) / 2);
    pcap_ = c.max_width * c.max_height;
    if (uint64_t(pcap_) >= (1ull << 25))
        return SH_E_ARG; // dense pair entries carry the pixel index in 25 bits
    tcap_ = tile_order_size(c.max_width, c.max_height);
    ncap_ = c.max_nodes;
    ecap_ = ncap_ * uint32_t(K_);
    ucap_ = std::min<uint64_t>(uint64_t(ncap_) * (ncap_ - 1) / 2, uint64_t(ncap_) * 96u);
    n2t_cap_ = pcap_ * uint32_t(K_) + 2 * ecap_ + ncap_;
    pair_cap_ = std::max<uint64_t>(uint64_t(pcap_) * np + ecap_, 2ull * ucap_);
    if (pair_cap_ >= (1ull << 31))
        return SH_E_ARG;

    slots_.resize(max_slots);
    int st;
    for (uint32_t s = 0; s < max_slots; ++s)
    {
        Slot &sl = slots_[s];
        SolveDesc &d = sl.d;
        std::memset(&d, 0, sizeof(d));
        d.K = K_;
        d.pcg_iters = int(c.pcg_iterations);
        d.blk_cap = uint32_t(ncap_ + 2 * ucap_);
#define A(ptr, bytes)                                                                                                  \
    if ((st = alloc(reinterpret_cast<void **>(&(ptr)), (bytes))) != SH_OK)                                            \
        return st;
        A(d.pix, size_t(pcap_) * 8);
        A(d.pknn, size_t(pcap_) * K_ * 2);
        A(d.pw, size_t(pcap_) * K_ * 4);
        A(sl.tpix, size_t(pcap_) * 8);
        A(sl.tpknn, size_t(pcap_) * K_ * 2);
        A(sl.tpw, size_t(pcap_) * K_ * 4);
        d.gpix = d.pix;
        d.gpknn = d.pknn;
        d.gpw = d.pw;
        A(d.n2t_off, size_t(ncap_ + 1) * 4);
        A(d.n2t_terms, size_t(n2t_cap_) * 4);
        if (cfg_.flags & SH_FLAG_REFERENCE_INDEX) // normalised: PAIR_MAJOR implies it
        {
            // the reference's node-pair index, only built on request
            A(d.half_keys, size_t(ucap_) * 4);
            A(d.half_off, size_t(ucap_ + 1) * 4);
            A(d.pair_entries, size_t(pcap_) * np * 4 + size_t(ecap_) * 4);
            A(d.upper_pos, size_t(ucap_) * 4);
            A(d.lower_pos, size_t(ucap_) * 4);
        }
        A(d.row_ptr, size_t(ncap_ + 1) * 4);
        A(d.blk_col, (size_t(ncap_) + 2 * size_t(ucap_)) * 4);
        A(d.dq[0], size_t(ncap_) * 32);
        A(d.dq[1], size_t(ncap_) * 32);
        A(d.dense_cnt, size_t(ncap_) * 4);
        A(d.seg_ptr, size_t(ncap_ + 1) * 4);
        A(d.tile_cbase, size_t(div_up(pcap_, kTilePixMin) + 1) * 4);
        A(d.tile_sbase, size_t(div_up(pcap_, kTilePixMin) + 1) * 4);
        A(d.list_off, (size_t(ncap_) + 2 * size_t(ucap_) + 1) * 4);
        A(d.blk_transpose, (size_t(ncap_) + 2 * size_t(ucap_)) * 4);
        A(d.jr, size_t(pcap_) * kHG * (fp16_ ? 2 : 4));
        A(d.reg, size_t(ecap_) * kReg * 4);
        A(d.ttrans, size_t(ncap_) * 16);
        A(d.blk, (size_t(ncap_) + 2 * size_t(ucap_)) * 36 * 4);
        A(d.dinv, size_t(ncap_) * 36 * 8);
        A(d.rhs, size_t(ncap_) * 6 * 4);
        A(d.x, size_t(ncap_) * 6 * 4);
        A(d.r, size_t(ncap_) * 6 * 4);
        A(d.s, size_t(ncap_) * 6 * 4);
        A(d.q, size_t(ncap_) * 6 * 4);
        A(d.dv[0], size_t(ncap_) * 6 * 4);
        A(d.dv[1], size_t(ncap_) * 6 * 4);
        A(d.mv[0], size_t(ncap_) * 6 * 8);
        A(d.mv[1], size_t(ncap_) * 6 * 8);
        A(d.delta, size_t(c.pcg_iterations + 1) * 8);
        A(d.cost, size_t(c.gn_iterations + 2) * 8);
        A(d.cost_part, (size_t(div_up(pcap_, 64)) + div_up(ecap_ + ncap_, 256) + 1) * 8);
        A(d.rot_cut, size_t(std::max(1u, c.gn_iterations)) * ncap_);
        A(d.twist_l1, size_t(std::max(1u, c.gn_iterations)) * ncap_ * 4);
    }
    tiles_cap_ = div_up(pcap_, kTilePixMin); // the most tiles: the smallest tile size
    // index-build workspace: groups of up to eight solves of the largest frame
    // (or more, smaller ones); the reference index builds one solve at a time
    {
        constexpr uint32_t kGroupUnits = 8;
        group_units_ = (cfg_.flags & SH_FLAG_REFERENCE_INDEX) ? 1u : std::min(max_slots, kGroupUnits);
        if (int rc = alloc_group_ws(group_units_, max_slots); rc != SH_OK)
            return rc;
    }
    // batch-wide launch state
    // the launch's descriptors followed by its work maps: one upload per launch
    A(d_descs_, size_t(max_slots) * sizeof(SolveDesc) + size_t(kNumMaps) * (max_slots + 1) * 4);
    d_wmaps_ = static_cast<char *>(d_descs_) + size_t(max_slots) * sizeof(SolveDesc);
    const size_t pcg_wg = size_t(max_slots) * div_up(ncap_, kPcgNodesPerWg);
    A(d_part_rs_, pcg_wg * 8);
    A(d_part_dq_, pcg_wg * kPcgSpmvPer * 8);
    A(d_slots_, size_t(max_slots) * kPcgMaxGroups * sizeof(PcgSlot));
    A(d_slots2_, size_t(max_slots) * kPcgMaxGroups * sizeof(PcgSlot2));
    A(d_flags_, 64);
    // How long the resident PCG's groups wait for each other depends on the page
    // that their slots lie in (solve_barrier_sum), and the allocations before
    // them decide that: arrays that the exchange does not use lie behind them.
    for (Slot &sl : slots_)
    {
        SolveDesc &d = sl.d;
        A(d.tile_nodes, size_t(tiles_cap_) * 4);
        A(d.tile_group, size_t(tiles_cap_) * (kTileGroups + 1) * 2);
        A(d.gprank, size_t(pcap_) * K_);
    }
    SH_HIP(hipMemset(d_slots_, 0, size_t(max_slots) * kPcgMaxGroups * sizeof(PcgSlot)));
    SH_HIP(hipMemset(d_slots2_, 0, size_t(max_slots) * kPcgMaxGroups * sizeof(PcgSlot2)));
    SH_HIP(hipMemset(d_flags_, 0, 64));
#undef A
    SH_HIP(hipHostMalloc(reinterpret_cast<void **>(&h_meta_), 64, hipHostMallocDefault));
    SH_HIP(hipHostMalloc(reinterpret_cast<void **>(&h_flag_), 64, hipHostMallocDefault));
    SH_HIP(hipEventCreateWithFlags(&sync_ev_, hipEventDisableTiming));
    SH_HIP(hipEventCreateWithFlags(&index_ev_, hipEventDisableTiming));
    stage_bytes_ = size_t(max_slots) * sizeof(SolveDesc) + size_t(kNumMaps) * (max_slots + 1) * 4;
    SH_HIP(hipHostMalloc(&h_stage_, stage_bytes_, hipHostMallocDefault));
    // the result view holds max_nodes identity transforms until the first solve
    // (the reference's constructor, SolverIterationData.cu:78-88 -> :234-247)
    {
        std::vector<float> ident(size_t(ncap_) * 8, 0.f);
        for (uint32_t n = 0; n < ncap_; ++n)
            ident[size_t(n) * 8 + 3] = 1.f; // q0 = (0, 0, 0, 1), q1 = 0
        for (Slot &sl : slots_)
        {
            SH_HIP(hipMemcpy(sl.d.dq[cfg_.gn_iterations & 1u], ident.data(), ident.size() * 4, hipMemcpyHostToDevice));
            sl.result_n = ncap_;
        }
    }
    return SH_OK;
}

int Engine::set_inputs(uint32_t slot, const sh_camera *cam, const sh_measure_maps *meas, const sh_render_maps *rend,
                       const sh_geometry *geo, const sh_node_graph *ng, const sh_node_flow *nf, const sh_flow_map *flow,
                       const sh_keypoints *kp, const float cam2world[16])
{
    (void)kp;
    if (slot >= slots_.size() || !cam || !meas || !rend || !geo || !ng || !cam2world)
        return SH_E_ARG;
    if (!meas->vertex_confid || !meas->normal_radius || !rend->reference_vertex || !rend->reference_normal ||
        !rend->index_map || !geo->surfel_knn || !geo->surfel_knn_spatial_weight || !geo->surfel_knn_connect_weight ||
        !ng->reference_node_coords || !ng->node_graph || !ng->node_knn_connect_weight)
        return SH_E_ARG;
    if (cam->width == 0 || cam->height == 0 || ng->num_nodes == 0)
        return SH_E_ARG;
    if (cam->width > cfg_.max_width || cam->height > cfg_.max_height || ng->num_nodes > ncap_ ||
        ng->num_edges > ecap_ || cam->width > 65535 || cam->height > 65535)
        return SH_E_CAPACITY;
    Slot &sl = slots_[slot];
    SolveDesc &d = sl.d;
    d.W = int(cam->width);
    d.H = int(cam->height);
    d.fx = cam->fx;
    d.fy = cam->fy;
    d.cx = cam->cx;
    d.cy = cam->cy;
    // world2camera = inverse(camera2world) for a rigid transform (WarpSolver.cu:151-154)
    double R[3][3], t[3];
    for (int a = 0; a < 3; ++a)
    {
        for (int b = 0; b < 3; ++b)
            R[a][b] = cam2world[4 * a + b];
        t[a] = cam2world[4 * a + 3];
    }
    for (int a = 0; a < 3; ++a)
    {
        for (int b = 0; b < 3; ++b)
            d.w2c_r[3 * a + b] = float(R[b][a]);
        d.w2c_t[a] = float(-(R[0][a] * t[0] + R[1][a] * t[1] + R[2][a] * t[2]));
    }
    d.lam2_depth = cfg_.lambda_depth * cfg_.lambda_depth;
    d.lam2_flow = cfg_.lambda_flow * cfg_.lambda_flow;
    d.lam2_reg = cfg_.lambda_reg * cfg_.lambda_reg;
    d.lam2_nt = cfg_.lambda_node_translation * cfg_.lambda_node_translation;
    d.damping = cfg_.damping;
    d.node_radius_square = ng->node_radius_square;
    d.N = int(ng->num_nodes);
    d.E = int(ng->num_edges);
    d.S = geo->num_surfels;
    d.meas_v = reinterpret_cast<const float4 *>(meas->vertex_confid);
    d.meas_n = reinterpret_cast<const float4 *>(meas->normal_radius);
    d.ref_v = reinterpret_cast<const float4 *>(rend->reference_vertex);
    d.ref_n = reinterpret_cast<const float4 *>(rend->reference_normal);
    d.index_map = rend->index_map;
    d.flow = (flow && flow->flow) ? reinterpret_cast<const float2 *>(flow->flow) : nullptr;
    d.surfel_knn = geo->surfel_knn;
    d.surfel_spatial = geo->surfel_knn_spatial_weight;
    d.surfel_connect = geo->surfel_knn_connect_weight;
    d.node_coords = reinterpret_cast<const float4 *>(ng->reference_node_coords);
    d.edges = ng->node_graph;
    d.node_connect = ng->node_knn_connect_weight;
    d.node_pred = (nf && nf->node_motion_pred) ? reinterpret_cast<const float4 *>(nf->node_motion_pred) : nullptr;
    d.P = 0;
    d.U = 0;
    d.n_pair_entries = 0;
    sl.has_inputs = true;
    sl.indexed = false;
    sl.solved = false;
    return SH_OK;
}

// The tile path reads the pixel streams in tile order; the row-segment and
// pair-major paths read the records by Node2Term term id, the raster index.
bool Engine::tile_order() const
{
    return !(cfg_.flags & (SH_FLAG_ROW_SEGMENTS | SH_FLAG_PAIR_MAJOR));
}

// Index-build workspace for groups of up to `units` solves of the largest
// frame with every pixel valid (and at most max_items solves).
static constexpr uint32_t kFlagUnits = 4;
int Engine::alloc_group_ws(uint32_t units, uint32_t max_items)
{
    GroupWs &g = gws_;
    const uint64_t kp = uint64_t(K_ * (K_ + 1) / 2);
    const uint64_t kv_unit = std::max<uint64_t>(n2t_cap_, pair_cap_);
    const uint64_t tent_unit = (uint64_t(pcap_) + kTilePixMax) * kp;
    // every position of the concatenated arrays stays below 2^31
    const uint64_t lim = (1ull << 31) - 1;
    units = uint32_t(std::max<uint64_t>(
        1, std::min<uint64_t>({units, lim / kv_unit, lim / tent_unit, lim / (pcap_ * uint64_t(kFlagUnits)),
                               lim / (tcap_ * uint64_t(kFlagUnits))})));
    group_units_ = units;
    // the flag stage takes kFlagUnits frames per unit (16 bytes per map
    // pixel), and the node arrays kFlagUnits node sets per unit (a batch's
    // solves have far fewer nodes than the largest); the row and tile stages'
    // groups are then formed by the valid pixels, a fraction of the frame
    g.cap_m = uint64_t(units) * kFlagUnits * pcap_;
    g.cap_h = uint64_t(units) * kFlagUnits * tcap_; // the tuning may switch the tile order on later
    g.cap_kv = uint64_t(units) * kv_unit;
    g.cap_nodes = uint64_t(units) * kFlagUnits * (uint64_t(ncap_) + 1); // about 1.6 KB a node
    g.cap_tcnt = uint64_t(units) * (uint64_t(tiles_cap_) + 2);
    g.cap_tent = uint64_t(units) * tent_unit;
    g.cap_items = max_items;
    void *p = nullptr;
    int rc;
#define A(field, type, count)                                                                                         \
    if ((rc = alloc(&p, size_t(count) * sizeof(type))) != SH_OK)                                                      \
        return rc;                                                                                                    \
    field = static_cast<type *>(p);
    A(g.ws.flags, uint32_t, g.cap_m);
    A(g.ws.pos, uint32_t, g.cap_m);
    A(g.ws.tflags, uint32_t, g.cap_h);
    A(g.ws.tpos, uint32_t, g.cap_h);
    A(g.ws.errs, uint32_t, max_items);
    A(g.ws.meta, uint32_t, size_t(max_items) * 16);
    A(g.ws.bitmap, uint32_t, g.cap_nodes * kBitmapWords);
    A(g.ws.bitpre, uint2, g.cap_nodes * kBitmapWords);
    A(g.ws.rowlen, uint32_t, g.cap_nodes);
    A(g.ws.segcnt, uint32_t, g.cap_nodes);
    A(g.ws.tcontrib, uint16_t, g.cap_tent);
    A(g.ws.tslot_block, uint32_t, g.cap_tent);
    A(g.ws.tslot_first, uint16_t, g.cap_tent);
    A(g.ws.tnslot, uint32_t, g.cap_tcnt);
    A(g.ws.tncontrib, uint32_t, g.cap_tcnt);
    A(g.ka, uint32_t, g.cap_kv);
    A(g.kb, uint32_t, g.cap_kv);
    A(g.va, uint32_t, g.cap_kv);
    A(g.vb, uint32_t, g.cap_kv);
    if (cfg_.flags & SH_FLAG_REFERENCE_INDEX)
    {
        A(g.head, uint32_t, pair_cap_);
        A(g.hpos, uint32_t, pair_cap_);
    }
    SH_HIP(hipMemset(g.ws.errs, 0, size_t(max_items) * 4)); // then cleared by each build's count kernel
    {
        size_t b0 = 0, b1 = 0;
        SH_HIP(sort_pairs_u32_u32(nullptr, b0, nullptr, nullptr, nullptr, nullptr, uint32_t(g.cap_kv), 32, nullptr));
        SH_HIP(exclusive_scan_u32(nullptr, b1, nullptr, nullptr,
                                  uint32_t(std::max(std::max(g.cap_m, g.cap_h), uint64_t(pair_cap_))), nullptr));
        g.sort_temp_bytes = std::max(b0, b1);
        if ((rc = alloc(&g.sort_temp, g.sort_temp_bytes)) != SH_OK)
            return rc;
    }
    // device tables: descriptors | items | work maps | scan jobs (row scans, tile scans)
    auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
    const size_t C = max_items;
    g.off_items = up(C * sizeof(SolveDesc));
    g.off_maps = g.off_items + C * sizeof(IndexItem);
    g.off_jobs = up(g.off_maps + size_t(kNumGroupMaps) * (C + 1) * 4);
    g.tab_bytes = g.off_jobs + 2 * (2 * C) * sizeof(ScanJob);
    A(g.d_tab, char, g.tab_bytes);
#undef A
    for (char *&h : g.h_tab)
        SH_HIP(hipHostMalloc(reinterpret_cast<void **>(&h), g.tab_bytes, hipHostMallocDefault));
    SH_HIP(hipHostMalloc(reinterpret_cast<void **>(&g.h_out), C * 8 * 4, hipHostMallocDefault));
    g_maps_.assign(size_t(kNumGroupMaps) * (C + 1), 0u);
    return SH_OK;
}

IndexGroup Engine::group_view() const
{
    IndexGroup v;
    v.sds = reinterpret_cast<const SolveDesc *>(gws_.d_tab);
    v.items = reinterpret_cast<const IndexItem *>(gws_.d_tab + gws_.off_items);
    v.n = int(g_items_.size());
    return v;
}

const uint32_t *Engine::group_map(int m) const
{
    return reinterpret_cast<const uint32_t *>(gws_.d_tab + gws_.off_maps) + size_t(m) * (gws_.cap_items + 1);
}

// One copy of the group's tables (the current descriptors of its slots, the
// items, work maps and scan jobs) through the stage's own pinned buffer: a
// stage's buffer is rewritten only after the host has waited for that
// stage's copy in the previous build.
int Engine::upload_group(int stage, hipStream_t st)
{
    GroupWs &g = gws_;
    char *h = g.h_tab[stage];
    const size_t n = g_items_.size(), C = g.cap_items;
    for (size_t i = 0; i < n; ++i)
        std::memcpy(h + i * sizeof(SolveDesc), &slots_[g_slots_[i]].d, sizeof(SolveDesc));
    std::memcpy(h + g.off_items, g_items_.data(), n * sizeof(IndexItem));
    std::memcpy(h + g.off_maps, g_maps_.data(), g_maps_.size() * 4);
    std::memcpy(h + g.off_jobs, g_jobs_[0].data(), g_jobs_[0].size() * sizeof(ScanJob));
    std::memcpy(h + g.off_jobs + 2 * C * sizeof(ScanJob), g_jobs_[1].data(), g_jobs_[1].size() * sizeof(ScanJob));
    SH_HIP(hipMemcpyAsync(g.d_tab, h, g.tab_bytes, hipMemcpyHostToDevice, st));
    return SH_OK;
}

// The index builds of several slots, in groups: a group takes slots while
// their frames fit the flag stage's workspace (the row and tile stages then
// run over sub-groups sized by the valid pixels); one solve of the largest
// frame always fits.  With rcs, a slot whose inputs are rejected (SH_E_ARG /
// SH_E_CAPACITY / SH_E_NOMEM) records its status there and the others go on;
// without, the first failure ends the build.
int Engine::build_indexes(const uint32_t *list, uint32_t n, hipStream_t st, int *rcs)
{
    if (rcs)
        for (uint32_t i = 0; i < n; ++i)
            rcs[i] = SH_OK;
    const GroupWs &g = gws_;
    const bool tiled = tile_order(), ref = (cfg_.flags & SH_FLAG_REFERENCE_INDEX) != 0;
    uint32_t i = 0;
    while (i < n)
    {
        uint64_t m = 0, h = 0;
        uint32_t j = i;
        while (j < n && j - i < g.cap_items && !(ref && j > i))
        {
            const SolveDesc &d = slots_[list[j]].d;
            const uint64_t m1 = m + uint64_t(d.W) * uint64_t(d.H);
            const uint64_t h1 = h + (tiled ? tile_order_size(uint32_t(d.W), uint32_t(d.H)) : 0u);
            if (j > i && (m1 > g.cap_m || h1 > g.cap_h))
                break;
            m = m1, h = h1;
            ++j;
        }
        if (int rc = build_group(list + i, j - i, st, rcs ? rcs + i : nullptr); rc != SH_OK)
            return rc;
        i = j;
    }
    return SH_OK;
}

// Once-per-solve index build (WarpSolver::buildSolverIndexStreamed, WarpSolver.cu:194-223).
int Engine::build_index(uint32_t slot, hipStream_t st) { return build_indexes(&slot, 1, st, nullptr); }

// Smallest bit count that holds every key below n_keys.
static int key_bits(uint64_t n_keys)
{
    int b = 1;
    while (b < 32 && (1ull << b) < n_keys)
        ++b;
    return b;
}

// The index build of one group, in three stages with one host readback
// between them (stages 2 and 3 once per sub-group of the slots that pass
// stage 1, sized by their valid pixels):
//  1. valid-pixel flags (raster and tile order) with the id range checks,
//     their group-wide scans; the pixel counts and check flags to the host;
//  2. compaction into each slot's pixel streams and the Node2Term pairs, one
//     stable node sort over the group (keys node0 + node), each slot's
//     n2t lists, row bitmaps and dense-term counts, the row and segment scans,
//     the block columns (the reference index: its pair index instead), the
//     per-tile contribution sort and the tile count scans; the row, pair and
//     slot totals to the host;
//  3. compaction of the tiles' contributions and slots, one stable block sort
//     over the group (keys blk0 + block), each slot's block lists and the
//     block transpose map.
// A slot that fails a check leaves the group (rcs) or ends the build.
int Engine::build_group(const uint32_t *list, uint32_t n, hipStream_t st, int *rcs)
{
    GroupWs &g = gws_;
    const bool tiled = tile_order(), ref = (cfg_.flags & SH_FLAG_REFERENCE_INDEX) != 0;
    const uint32_t TP = tile_pix(), C = g.cap_items;
    if (n == 0)
        return SH_OK;
    if (n > C || (ref && n > 1))
        return SH_E_STATE;
    std::vector<uint32_t> where(n); // each item's position in list (for rcs)
    auto keep = [&](uint32_t i, int rc) {
        // false: the build ends with rc
        if (rcs && rc != SH_E_HIP)
        {
            rcs[where[i]] = rc;
            return true;
        }
        return false;
    };
    auto set_map = [&](int m, auto wg_of) {
        uint32_t *w = g_maps_.data() + size_t(m) * (C + 1);
        uint32_t t = 0;
        for (size_t i = 0; i < g_items_.size(); ++i)
        {
            w[i] = t;
            t += wg_of(i);
        }
        w[g_items_.size()] = t;
        return t;
    };
    auto desc_of = [&](size_t i) -> SolveDesc & { return slots_[g_slots_[i]].d; };
    // drops the items whose rc is set (or ends the build), renumbering the rest
    auto compact_items = [&](const std::vector<int> &rc_of) -> int {
        size_t k = 0;
        for (size_t i = 0; i < g_items_.size(); ++i)
        {
            if (rc_of[i] != SH_OK)
            {
                if (!keep(uint32_t(i), rc_of[i]))
                    return rc_of[i];
                continue;
            }
            g_slots_[k] = g_slots_[i];
            g_items_[k] = g_items_[i];
            g_items_[k].slot = uint32_t(k);
            where[k] = where[i];
            ++k;
        }
        g_slots_.resize(k);
        g_items_.resize(k);
        return SH_OK;
    };
    g_jobs_[0].clear();
    g_jobs_[1].clear();

    // ---- stage 1
    g_slots_.assign(list, list + n);
    g_items_.assign(n, IndexItem{});
    uint64_t m0 = 0, h0 = 0;
    for (uint32_t i = 0; i < n; ++i)
    {
        where[i] = i;
        Slot &sl = slots_[list[i]];
        SolveDesc &d = sl.d;
        // the GN phase's pixel order: tile order on the tile path, raster on the others
        d.gpix = tiled ? sl.tpix : d.pix;
        d.gpknn = tiled ? sl.tpknn : d.pknn;
        d.gpw = tiled ? sl.tpw : d.pw;
        d.tile_pix = int(TP);
        d.P = 0;
        d.n_tiles = 0;
        sl.indexed = false;
        IndexItem &it = g_items_[i];
        it.slot = i;
        it.m0 = uint32_t(m0);
        it.h0 = uint32_t(h0);
        m0 += uint64_t(d.W) * uint64_t(d.H);
        h0 += tiled ? tile_order_size(uint32_t(d.W), uint32_t(d.H)) : 0u;
    }
    if (m0 > g.cap_m || h0 > g.cap_h)
        return SH_E_STATE; // never: build_indexes sized the group
    uint32_t wg = set_map(kGmFlags, [&](size_t i) {
        const SolveDesc &d = desc_of(i);
        const uint32_t px = uint32_t(d.W) * uint32_t(d.H);
        const uint32_t nh = tiled ? tile_order_size(uint32_t(d.W), uint32_t(d.H)) : 0u;
        return div_up(std::max(std::max(px, nh), uint32_t(d.E)), 256u * kPixPer);
    });
    int rc;
    if ((rc = upload_group(0, st)) != SH_OK)
        return rc;
    IndexGroup gv = group_view();
    SH_HIP(launch_pixel_flags(gv, group_map(kGmFlags), wg, tiled, g.ws, st));
    size_t tb = g.sort_temp_bytes;
    SH_HIP(exclusive_scan_u32(g.sort_temp, tb, g.ws.flags, g.ws.pos, uint32_t(m0), st));
    if (tiled && h0 > 0)
    {
        tb = g.sort_temp_bytes;
        SH_HIP(exclusive_scan_u32(g.sort_temp, tb, g.ws.tflags, g.ws.tpos, uint32_t(h0), st));
    }
    SH_HIP(launch_index_counts(gv, 1, g.ws, g.h_out, st));
    if ((rc = wait_stream(st, index_ev_)) != SH_OK)
        return rc;
    {
        std::vector<int> rc_of(n, SH_OK);
        for (uint32_t i = 0; i < n; ++i)
        {
            const uint32_t *o = g.h_out + size_t(i) * 8;
            if (o[1] != 0)
                rc_of[i] = SH_E_ARG; // a surfel or node id out of range
            else if (o[0] > pcap_)
                rc_of[i] = SH_E_CAPACITY;
            else
                desc_of(i).P = int(o[0]);
        }
        if ((rc = compact_items(rc_of)) != SH_OK)
            return rc;
    }
    if (g_items_.empty())
        return SH_OK;

    // stages 2 and 3 over sub-groups whose valid pixels fit the row and
    // tile workspace
    auto rows_tiles = [&]() -> int {
        g_jobs_[0].clear();
        g_jobs_[1].clear();
        // ---- stage 2
        uint64_t kv0 = 0, node0 = 0, t0 = 0, tc0 = 0;
        for (size_t i = 0; i < g_items_.size(); ++i)
        {
            SolveDesc &d = desc_of(i);
            IndexItem &it = g_items_[i];
            const uint32_t P = uint32_t(d.P), N = uint32_t(d.N);
            d.n_tiles = int(div_up(P, TP));
            d.n_pair_entries = 0;
            it.kv0 = uint32_t(kv0);
            it.node0 = uint32_t(node0);
            it.t0 = uint32_t(t0);
            it.tc0 = uint32_t(tc0);
            kv0 += uint64_t(P) * uint64_t(K_) + 2 * uint64_t(d.E) + N;
            node0 += uint64_t(N) + 1;
            t0 += uint64_t(d.n_tiles);
            tc0 += uint64_t(d.n_tiles) + 2;
            g_jobs_[0].push_back(ScanJob{g.ws.segcnt + it.node0, d.seg_ptr, N + 1, 0});
            if (!ref)
                g_jobs_[0].push_back(ScanJob{g.ws.rowlen + it.node0, d.row_ptr, N + 1, 0});
            const uint32_t nt = uint32_t(d.n_tiles);
            g_jobs_[1].push_back(ScanJob{g.ws.tnslot + it.tc0, d.tile_sbase, nt + 1, 0});
            g_jobs_[1].push_back(ScanJob{g.ws.tncontrib + it.tc0, d.tile_cbase, nt + 1, 0});
        }
        if (kv0 > g.cap_kv || node0 > g.cap_nodes || tc0 > g.cap_tcnt || t0 * TP * uint64_t(K_ * (K_ + 1) / 2) > g.cap_tent)
            return SH_E_STATE; // never: build_indexes sized the group
        const uint32_t wg_compact = set_map(kGmCompact, [&](size_t i) {
            const SolveDesc &d = desc_of(i);
            // the pixel work-groups walk the tile-order index space when tiled
            const uint32_t walk = tiled ? tile_order_size(uint32_t(d.W), uint32_t(d.H)) : uint32_t(d.W) * uint32_t(d.H);
            return std::max(1u, div_up(walk, 256u)) + div_up(uint32_t(d.E + d.N), 256u);
        });
        const uint32_t wg_split = set_map(kGmSplit, [&](size_t i) {
            const SolveDesc &d = desc_of(i);
            // kSplitPer sorted pairs a thread (every node has its translation term)
            return div_up(uint32_t(d.P) * uint32_t(K_) + 2u * uint32_t(d.E) + uint32_t(d.N), 256u * kSplitPer);
        });
        const uint32_t wg_node = set_map(kGmNode, [&](size_t i) { return div_up(uint32_t(desc_of(i).N), kRowNodes); });
        // a wave per node once that launch fills the device (256 CUs x eight
        // 256-thread work-groups x four nodes = 8,192 nodes); a work-group per
        // node below that (a single solve of a thousand nodes)
        const uint32_t row_npw = node0 >= 4u * 256u * 8u ? kRowNodes : 1u;
        const uint32_t wg_rowbits =
            set_map(kGmRowBits, [&](size_t i) { return div_up(uint32_t(desc_of(i).N), row_npw); });
        const uint32_t wg_tile = set_map(kGmTile, [&](size_t i) { return uint32_t(desc_of(i).n_tiles); });
        if ((rc = upload_group(1, st)) != SH_OK)
            return rc;
        gv = group_view();
        const ScanJob *jobs = reinterpret_cast<const ScanJob *>(g.d_tab + g.off_jobs);
        SH_HIP(launch_compact_pixels(K_, gv, group_map(kGmCompact), wg_compact, tiled, g.ws, g.ka, g.va, st));
        // Node2TermsIndex::BuildIndex (Node2TermsIndex.cu:191-199,312-360): one
        // stable sort of the group's (node key, term) pairs
        if (kv0 > 0)
        {
            tb = g.sort_temp_bytes;
            SH_HIP(sort_pairs_u32_u32(g.sort_temp, tb, g.ka, g.kb, g.va, g.vb, uint32_t(kv0), key_bits(node0), st));
        }
        SH_HIP(launch_n2t_split(gv, group_map(kGmSplit), wg_split, g.kb, g.vb, st));
        SH_HIP(launch_row_bitmap(K_, row_npw, gv, group_map(kGmRowBits), wg_rowbits, g.ws, st));
        SH_HIP(launch_scan_jobs(jobs, uint32_t(g_jobs_[0].size()), st));
        // the word prefix counts of the row bitmaps, and the block columns (the
        // reference index builds them from its pair index)
        SH_HIP(launch_row_cols(gv, group_map(kGmNode), wg_node, g.ws, !ref, st));
        if (ref && (rc = reference_pair_index(slots_[g_slots_[0]], st)) != SH_OK)
            return keep(0, rc) ? SH_OK : rc;
        // the row structure is complete here (blk_col bounded by blk_cap)
        SH_HIP(launch_tile_build(K_, TP, gv, group_map(kGmTile), wg_tile, g.ws, st));
        SH_HIP(launch_scan_jobs(jobs + 2 * C, uint32_t(g_jobs_[1].size()), st));
        SH_HIP(launch_index_counts(gv, 2, g.ws, g.h_out, st));
        if ((rc = wait_stream(st, index_ev_)) != SH_OK)
            return rc;
        std::vector<uint32_t> n_slots(g_items_.size());
        {
            std::vector<int> rc_of(g_items_.size(), SH_OK);
            for (size_t i = 0; i < g_items_.size(); ++i)
            {
                const uint32_t *o = g.h_out + i * 8;
                Slot &sl = slots_[g_slots_[i]];
                SolveDesc &d = sl.d;
                int r = SH_OK;
                if (o[2] > ucap_)
                    r = SH_E_CAPACITY;
                else
                {
                    d.U = int(o[2]);
                    if (!ref)
                    {
                        sl.max_row_len = o[1];
                        d.n_seg = int(o[0]);
                        r = size_partials(sl);
                    }
                }
                if (r == SH_OK && uint64_t(o[3]) > pair_cap_)
                    r = SH_E_CAPACITY;
                if (r == SH_OK)
                {
                    sl.tile_slot_max = d.n_tiles > 0 ? o[5] : 0u;
                    sl.tiles_listed = d.n_tiles > 0 ? o[6] : 0u;
                    r = size_tiles(sl, o[3], o[4]);
                }
                n_slots[i] = o[3];
                rc_of[i] = r;
            }
            // n_slots follows the items
            size_t k = 0;
            for (size_t i = 0; i < rc_of.size(); ++i)
                if (rc_of[i] == SH_OK)
                    n_slots[k++] = n_slots[i];
            if ((rc = compact_items(rc_of)) != SH_OK)
                return rc;
        }
        if (g_items_.empty())
            return SH_OK;

        // ---- stage 3
        uint64_t sb0 = 0, blk0 = 0;
        for (size_t i = 0; i < g_items_.size(); ++i)
        {
            const SolveDesc &d = desc_of(i);
            g_items_[i].sb0 = uint32_t(sb0);
            g_items_[i].blk0 = uint32_t(blk0);
            sb0 += n_slots[i];
            blk0 += uint64_t(d.N) + 2 * uint64_t(d.U) + 1;
        }
        if (sb0 > g.cap_kv)
            return SH_E_STATE; // never: each solve's slots are at most its upper bound
        const uint32_t wg_tile3 = set_map(kGmTile, [&](size_t i) { return uint32_t(desc_of(i).n_tiles); });
        const uint32_t wg_lists = set_map(kGmLists, [&](size_t i) {
            const SolveDesc &d = desc_of(i);
            return div_up(std::max(n_slots[i], uint32_t(d.N) + 2u * uint32_t(d.U) + 1u), 256u);
        });
        const uint32_t wg_node3 = set_map(kGmNode, [&](size_t i) { return div_up(uint32_t(desc_of(i).N), kRowNodes); });
        if ((rc = upload_group(2, st)) != SH_OK)
            return rc;
        gv = group_view();
        SH_HIP(launch_tile_compact(K_, TP, gv, group_map(kGmTile), wg_tile3, g.ws, g.ka, g.va, st));
        if (sb0 > 0)
        {
            // the slots of every block in tile order (stable)
            tb = g.sort_temp_bytes;
            SH_HIP(sort_pairs_u32_u32(g.sort_temp, tb, g.ka, g.kb, g.va, g.vb, uint32_t(sb0), key_bits(blk0), st));
        }
        SH_HIP(launch_slot_lists(gv, group_map(kGmLists), wg_lists, g.kb, g.vb, st));
        SH_HIP(launch_block_transpose(gv, group_map(kGmNode), wg_node3, g.ws, st));
        for (uint32_t s : g_slots_)
            slots_[s].indexed = true;
        return SH_OK;
    };
    const std::vector<uint32_t> s1_slots = g_slots_;
    const std::vector<IndexItem> s1_items = g_items_;
    const std::vector<uint32_t> s1_where(where.begin(), where.begin() + s1_items.size());
    const uint64_t kp = uint64_t(K_ * (K_ + 1) / 2);
    for (size_t a = 0; a < s1_items.size();)
    {
        uint64_t kv = 0, nodes = 0, tcnt = 0, tent = 0, sub = 0;
        size_t b = a;
        for (; b < s1_items.size(); ++b)
        {
            const SolveDesc &d = slots_[s1_slots[b]].d;
            const uint64_t nt = div_up(uint32_t(d.P), TP);
            const uint64_t kv1 = kv + uint64_t(d.P) * uint64_t(K_) + 2 * uint64_t(d.E) + uint64_t(d.N);
            const uint64_t n1 = nodes + uint64_t(d.N) + 1, tc1 = tcnt + nt + 2, te1 = tent + nt * TP * kp;
            const uint64_t s1 = sub + std::min<uint64_t>(nt * TP * kp, pair_cap_);
            if (b > a && (kv1 > g.cap_kv || n1 > g.cap_nodes || tc1 > g.cap_tcnt || te1 > g.cap_tent || s1 > g.cap_kv))
                break;
            kv = kv1, nodes = n1, tcnt = tc1, tent = te1, sub = s1;
        }
        g_slots_.assign(s1_slots.begin() + a, s1_slots.begin() + b);
        g_items_.assign(s1_items.begin() + a, s1_items.begin() + b);
        for (size_t i = 0; i < g_items_.size(); ++i)
            g_items_[i].slot = uint32_t(i);
        where.assign(s1_where.begin() + a, s1_where.begin() + b);
        if ((rc = rows_tiles()) != SH_OK)
            return rc;
        a = b;
    }
    return SH_OK;
}

// The reference's node-pair index and symmetric row blocks for the group's
// one solve (NodePair2TermsIndex::BuildHalfIndex, :294-298,591-654, and
// BuildSymmetricAndRowBlocksIndex, :300-312), after its node lists, row
// bitmaps and segment scan: half keys and offsets, pair entries, row_ptr and
// blk_col; sizes the segment partials.
int Engine::reference_pair_index(Slot &sl, hipStream_t st)
{
    SolveDesc &d = sl.d;
    GroupWs &g = gws_;
    if (!d.pair_entries || !d.half_keys || !d.half_off || !d.upper_pos || !d.lower_pos || !g.head)
        return SH_E_STATE; // never launch on unallocated pair arrays
    const uint32_t np = uint32_t(K_ * (K_ - 1) / 2);
    const uint32_t n_pkv = uint32_t(d.P) * np + uint32_t(d.E);
    uint32_t *meta = g.ws.meta; // the group's only item
    SH_HIP(hipMemcpyAsync(h_meta_ + 6, d.seg_ptr + d.N, 4, hipMemcpyDeviceToHost, st));
    SH_HIP(launch_pair_kv(d, g.ka, g.va, st));
    size_t tb = g.sort_temp_bytes;
    SH_HIP(sort_pairs_u32_u32(g.sort_temp, tb, g.ka, g.kb, g.va, g.vb, n_pkv, 24, st));
    SH_HIP(launch_pair_heads(g.kb, n_pkv, g.head, meta + 8, st));
    tb = g.sort_temp_bytes;
    SH_HIP(exclusive_scan_u32(g.sort_temp, tb, g.head, g.hpos, n_pkv, st));
    // the half arrays go to the workspace first: U is checked against the capacity below
    SH_HIP(launch_pair_compact(g.kb, g.head, g.hpos, n_pkv, meta + 8, g.ka, g.va, meta + 2, st));
    SH_HIP(hipMemcpyAsync(h_meta_, meta, 16, hipMemcpyDeviceToHost, st));
    if (int rc = wait_stream(st, index_ev_); rc != SH_OK)
        return rc;
    const uint32_t U = h_meta_[2];
    if (U > ucap_)
        return SH_E_CAPACITY;
    d.U = int(U);
    d.n_pair_entries = int(h_meta_[3]);
    sl.max_row_len = h_meta_[0];
    d.n_seg = int(h_meta_[6]);
    if (int rc = size_partials(sl); rc != SH_OK)
        return rc;
    SH_HIP(hipMemcpyAsync(d.half_keys, g.ka, size_t(U) * 4, hipMemcpyDeviceToDevice, st));
    SH_HIP(hipMemcpyAsync(d.half_off, g.va, size_t(U + 1) * 4, hipMemcpyDeviceToDevice, st));
    SH_HIP(launch_pair_entries(d, g.vb, st));
    SH_HIP(launch_sym_kv(d, g.ka, g.va, st));
    tb = g.sort_temp_bytes;
    if (U > 0)
        SH_HIP(sort_pairs_u32_u32(g.sort_temp, tb, g.ka, g.kb, g.va, g.vb, 2 * U, 24, st));
    SH_HIP(launch_sym_scatter(d, g.kb, g.vb, st));
    SH_HIP(launch_row_ptr(d, g.kb, st));
    return SH_OK;
}

// Replaces a slot's grown buffer with one of `bytes`, with the growth hook's
// consent; on failure the slot holds no buffer.
int Engine::grow_buffer(void **buf, size_t *held, size_t bytes)
{
    if (grow_fn_ && !grow_fn_(grow_ctx_, int64_t(bytes) - int64_t(*held)))
        return SH_E_CAPACITY;
    hipError_t e = hipSuccess;
    if (*buf)
        e = hipFree(*buf);
    *buf = nullptr;
    if (e == hipSuccess)
        e = hipMalloc(buf, bytes);
    if (e != hipSuccess)
    {
        last_hip_error = e;
        *buf = nullptr;
        *held = 0;
        if (grow_fn_)
            grow_fn_(grow_ctx_, -int64_t(bytes));
        return SH_E_NOMEM;
    }
    *held = bytes;
    return SH_OK;
}

// One grown device buffer per slot, cut into the tile arrays.
int Engine::size_tiles(Slot &sl, uint32_t n_slots, uint32_t n_contrib)
{
    SolveDesc &d = sl.d;
    auto up = [](size_t b) { return (b + 255) & ~size_t(255); };
    const size_t b_contrib = up(size_t(n_contrib) * 2 + 2);
    const size_t b_first = up((size_t(n_slots) + 1) * 4);
    const size_t b_items = up(size_t(n_slots) * 4 + 4);
    const size_t b_part = up(size_t(n_slots) * kPartStride * 4 + 16); // 128-byte partials, 256-aligned base
    const size_t b_pair = up(size_t(n_slots) * 2 + 2);
    const size_t need = b_contrib + b_first + 2 * b_items + b_part + b_pair;
    if (need > sl.tile_bytes)
        if (int rc = grow_buffer(&sl.tile_buf, &sl.tile_bytes, need + need / 4); rc != SH_OK)
            return rc;
    char *b = static_cast<char *>(sl.tile_buf);
    d.tc_contrib = reinterpret_cast<uint16_t *>(b);
    d.tc_slot_first = reinterpret_cast<uint32_t *>(b + b_contrib);
    d.list_items = reinterpret_cast<uint32_t *>(b + b_contrib + b_first);
    d.tpart = reinterpret_cast<float *>(b + b_contrib + b_first + b_items);
    d.slot_pos = reinterpret_cast<uint32_t *>(b + b_contrib + b_first + b_items + b_part);
    d.slot_pair = reinterpret_cast<uint16_t *>(b + b_contrib + b_first + 2 * b_items + b_part);
    return SH_OK;
}

// Segment partials: 8 floats of rhs + 21 per block of the longest row, per
// segment.  Grown (never shrunk) outside the GN loop.
int Engine::size_partials(Slot &sl)
{
    SolveDesc &d = sl.d;
    d.part_stride = (sl.max_row_len + 1) * 21 + 8;
    const size_t need = std::max<size_t>(size_t(d.n_seg) * d.part_stride * sizeof(float), 256);
    if (need > sl.part_bytes)
        if (int rc = grow_buffer(&sl.part_buf, &sl.part_bytes, need + need / 4); rc != SH_OK)
            return rc;
    d.part = static_cast<float *>(sl.part_buf);
    return SH_OK;
}

// Rows of a launch from which the tile combine runs one wave per row.
constexpr uint32_t kCombineWaveRows = 8192;

// Groups of the register-resident PCG for one solve: rows split evenly, at
// most `max_rows` (<= kPcgResRows) rows and kPcgResBlocks blocks (rows x
// longest row) each; 0 when that takes more than kPcgMaxGroups groups.
static uint32_t resident_groups(int n, uint32_t max_row_len, uint32_t max_rows)
{
    const uint32_t rows = std::min(std::min(max_rows, kPcgResRows), kPcgResBlocks / (max_row_len + 1));
    if (rows == 0 || n <= 0)
        return n <= 0 && rows > 0 ? 1u : 0u;
    const uint32_t g = div_up(uint32_t(n), rows);
    return g <= kPcgMaxGroups ? g : 0u;
}

void Engine::build_maps(uint32_t ns)
{
    maps_.assign(size_t(kNumMaps) * (ns + 1), 0u);
    coop_resident_ = !(cfg_.flags & SH_FLAG_STREAMING_PCG);
    for (uint32_t s = 0; s < ns; ++s)
        if (resident_groups(slots_[batch_[s]].d.N, slots_[batch_[s]].max_row_len, res_rows_) == 0)
            coop_resident_ = false;
    for (int m = 0; m < kNumMaps; ++m)
    {
        uint32_t acc = 0;
        for (uint32_t s = 0; s < ns; ++s)
        {
            const SolveDesc &d = slots_[batch_[s]].d;
            uint32_t wg = 0;
            switch (m)
            {
            case kMapPixel:
                wg = div_up(uint32_t(d.P), kThreads);
                break;
            case kMapReg:
                wg = div_up(uint32_t(d.E + d.N), kThreads);
                break;
            case kMapNodeWave:
                wg = div_up(uint32_t(d.N), kWavesPerWg);
                break;
            case kMapPairWave:
                wg = div_up(uint32_t(d.U), kWavesPerWg);
                break;
            case kMapPcg:
                wg = div_up(uint32_t(d.N), kPcgNodesPerWg);
                break;
            case kMapNode:
                wg = div_up(uint32_t(d.N), kThreads);
                break;
            case kMapRow:
                wg = uint32_t(d.N);
                break;
            case kMapCoop:
                wg = coop_resident_ ? resident_groups(d.N, slots_[batch_[s]].max_row_len, res_rows_)
                                    : std::min(kPcgMaxGroups, std::max(1u, div_up(uint32_t(d.N) + 2u * uint32_t(d.U),
                                                                                  kPcgBlocksPerGroup)));
                break;
            case kMapSeg:
                wg = uint32_t(d.n_seg);
                break;
            case kMapTile:
                wg = uint32_t(d.n_tiles);
                break;
            }
            maps_[size_t(m) * (ns + 1) + s] = acc;
            acc += wg;
        }
        maps_[size_t(m) * (ns + 1) + ns] = acc;
        map_total_[m] = acc;
    }
}

int Engine::upload(uint32_t ns, hipStream_t st)
{
    char *h = static_cast<char *>(h_stage_);
    for (uint32_t s = 0; s < ns; ++s)
        std::memcpy(h + size_t(s) * sizeof(SolveDesc), &slots_[batch_[s]].d, sizeof(SolveDesc));
    const size_t mb = maps_.size() * 4;
    std::memcpy(h + size_t(ns) * sizeof(SolveDesc), maps_.data(), mb);
    // the maps follow the ns descriptors directly (u32 entries, 8-byte aligned)
    d_wmaps_ = static_cast<char *>(d_descs_) + size_t(ns) * sizeof(SolveDesc);
    SH_HIP(hipMemcpyAsync(d_descs_, h, size_t(ns) * sizeof(SolveDesc) + mb, hipMemcpyHostToDevice, st));
    return SH_OK;
}

const uint32_t *Engine::map(int m, uint32_t ns) const
{
    return static_cast<const uint32_t *>(d_wmaps_) + size_t(m) * (ns + 1);
}

// The Gauss-Newton loop (WarpSolver::SolveStreamed :260-337) for the slots of
// batch_: `iters` iterations, the first starting at each solve's gn_iter, from
// the identity warp field when `identity` is set.
int Engine::enqueue_gn(uint32_t ns, hipStream_t st, uint32_t iters, bool identity)
{
    const SolveDesc *sds = static_cast<const SolveDesc *>(d_descs_);
    const int n = int(ns);
    const bool fp16 = fp16_;
    if (identity)
        SH_HIP(launch_identity(sds, map(kMapNode, ns), n, map_total_[kMapNode], st));
    uint32_t max_n = 0, max_l = 0, tile = 1, slot_cap = 1, n_listed = 0;
    const uint32_t *coop_begin = maps_.data() + size_t(kMapCoop) * (ns + 1);
    for (uint32_t s = 0; s < ns; ++s)
    {
        const SolveDesc &d = slots_[batch_[s]].d;
        max_n = std::max(max_n, uint32_t(d.N));
        max_l = std::max(max_l, slots_[batch_[s]].max_row_len);
        slot_cap = std::max(slot_cap, slots_[batch_[s]].tile_slot_max);
        n_listed += slots_[batch_[s]].tiles_listed;
        // blocks of one persistent-PCG group: its share plus one whole row
        const uint32_t G = coop_begin[s + 1] - coop_begin[s];
        const uint32_t nb = uint32_t(d.N) + 2u * uint32_t(d.U);
        tile = std::max(tile, div_up(nb, G) + slots_[batch_[s]].max_row_len + 2u);
    }
    const size_t coop_lds = size_t(tile) * 6 * sizeof(float);
    if (coop_lds != coop_lds_)
    {
        coop_lds_ = coop_lds;
        coop_max_groups_ = coop_lds <= 160u * 1024u ? pcg_coop_max_groups(coop_lds) : 0;
    }
    if (res_max_groups_ < 0)
        res_max_groups_ = pcg_resident_max_groups();
    if (pipe_max_groups_ < 0)
        pipe_max_groups_ = pcg_pipe_max_groups();
    const bool pipelined = (cfg_.flags & SH_FLAG_PIPELINED_PCG) != 0;
    // more groups than can be co-resident: the pipelined PCG runs in rounds
    // of consecutive solves whose groups fit together
    bool pipe_rounds = coop_resident_ && pipelined && pipe_max_groups_ > 0 &&
                       map_total_[kMapCoop] > uint32_t(pipe_max_groups_);
    for (uint32_t s = 0; pipe_rounds && s < ns; ++s)
        if (coop_begin[s + 1] - coop_begin[s] > uint32_t(pipe_max_groups_))
            pipe_rounds = false;
    const bool resident =
        coop_resident_ &&
        (map_total_[kMapCoop] <= uint32_t(pipelined ? pipe_max_groups_ : res_max_groups_) || pipe_rounds);
    // the matrix-free operator reads the tile index: not with the other materialisations
    const bool matrix_free = cfg_.spmv_mode == SH_SPMV_MATRIX_FREE;
    if (matrix_free && (cfg_.flags & (SH_FLAG_PAIR_MAJOR | SH_FLAG_ROW_SEGMENTS)))
        return SH_E_ARG;
    const bool use_coop = !matrix_free && !(cfg_.flags & SH_FLAG_NO_PERSISTENT_PCG) &&
                          (resident || (!coop_resident_ && coop_max_groups_ > 0 &&
                                        map_total_[kMapCoop] <= uint32_t(coop_max_groups_)));
    uint32_t *flags = static_cast<uint32_t *>(d_flags_);
    const RowsPlan plan = rows_plan(max_n, max_l);
    // every solve of the launch was indexed with the tile size in use (a tuning
    // change takes effect at the next index build)
    for (uint32_t s = 0; s < ns; ++s)
        if (slots_[batch_[s]].d.tile_pix != int(tile_pix()))
            return SH_E_STATE;
    // the tile combine: one wave per row when the launch has enough rows to
    // fill the CUs several times over (batches, server steps); one work-group
    // per row otherwise, where a single solve's rows finish sooner (and for
    // rows too long for the wave form's registers).  Both give the same bits.
    const bool comb_wave = map_total_[kMapRow] >= kCombineWaveRows && max_l + 1 <= kWaveCombineMaxBlocks;
    const size_t tiles_lds = tiles_combine_lds(max_n, max_l, comb_wave);
    if ((cfg_.flags & SH_FLAG_ROW_SEGMENTS) && std::max(plan.lds, plan.lds_combine) > 160u * 1024u)
        return SH_E_CAPACITY;
    if (!(cfg_.flags & (SH_FLAG_ROW_SEGMENTS | SH_FLAG_PAIR_MAJOR)) && tiles_lds > 160u * 1024u)
        return SH_E_CAPACITY;
    const bool tiles_path = !(cfg_.flags & (SH_FLAG_ROW_SEGMENTS | SH_FLAG_PAIR_MAJOR));
    // the tile kernel builds the FP32 per-pixel records itself, so they never
    // go through HBM; FP16 records are streamed (that is their point), and the
    // matrix-free operator reads the stored records every PCG iteration
    const bool fused = tiles_path && !fp16 && !matrix_free;
    for (uint32_t s = 0; s < ns; ++s)
        slots_[batch_[s]].records_fused = fused;
    const uint32_t pipe_slots = use_coop && resident && pipelined ? map_total_[kMapCoop] : 0u;
    for (uint32_t it = 0; it < iters; ++it)
    {
        const int parity = int(it); // iteration offset: DQ buffer (gn_iter + it) & 1, cost slot gn_iter + it
        SH_HIP(mark(kPhDense, st));
        SH_HIP(launch_terms(K_, fp16, sds, map(kMapPixel, ns), fused ? 0u : map_total_[kMapPixel], map(kMapReg, ns),
                            map_total_[kMapReg], n, parity, st));
        if (cfg_.flags & SH_FLAG_PAIR_MAJOR)
        {
            SH_HIP(mark(kPhDiagRhs, st));
            SH_HIP(launch_diag_rhs(K_, fp16, sds, map(kMapNodeWave, ns), n, map_total_[kMapNodeWave], st));
            SH_HIP(mark(kPhOffdiag, st));
            SH_HIP(launch_offdiag(K_, fp16, sds, map(kMapPairWave, ns), n, map_total_[kMapPairWave], st));
        }
        else if (cfg_.flags & SH_FLAG_ROW_SEGMENTS)
        {
            SH_HIP(mark(kPhRowsSeg, st));
            SH_HIP(launch_rows_seg(K_, fp16, sds, map(kMapSeg, ns), n, map_total_[kMapSeg], plan, st));
            SH_HIP(mark(kPhRowsCombine, st));
            SH_HIP(launch_rows_combine(sds, map(kMapRow, ns), n, map_total_[kMapRow], plan, st));
        }
        else
        {
            SH_HIP(mark(kPhTiles, st));
            SH_HIP(launch_tiles(K_, fp16, tile_pix(), fused, parity, sds, map(kMapTile, ns), n, map_total_[kMapTile],
                                slot_cap, n_listed, st));
            SH_HIP(mark(kPhTilesCombine, st));
            SH_HIP(launch_tiles_combine(sds, map(kMapRow, ns), n, map_total_[kMapRow], tiles_lds, comb_wave,
                                        static_cast<PcgSlot2 *>(d_slots2_), pipe_slots, st));
        }
        if (!tiles_path) // the tile combine inverts the diagonal blocks itself
        {
            SH_HIP(mark(kPhDinv, st));
            SH_HIP(launch_dinv(sds, map(kMapNode, ns), n, map_total_[kMapNode], static_cast<PcgSlot2 *>(d_slots2_),
                               pipe_slots, st));
        }
        SH_HIP(mark(kPhPcg, st));
        if (use_coop)
        {
            if (resident && pipelined)
                for (uint32_t s0 = 0; s0 < ns;)
                {
                    uint32_t s1 = s0 + 1;
                    while (s1 < ns && coop_begin[s1 + 1] - coop_begin[s0] <= uint32_t(pipe_max_groups_))
                        ++s1;
                    SH_HIP(launch_pcg_pipe(sds + s0, map(kMapCoop, ns) + s0, int(s1 - s0),
                                           coop_begin[s1] - coop_begin[s0], int(cfg_.pcg_iterations),
                                           static_cast<PcgSlot2 *>(d_slots2_), flags + 0, flags + 1, wait_limit_,
                                           parity, st));
                    s0 = s1;
                }
            else if (resident)
                SH_HIP(launch_pcg_resident(sds, map(kMapCoop, ns), n, map_total_[kMapCoop],
                                           int(cfg_.pcg_iterations), static_cast<PcgSlot *>(d_slots_), flags + 0,
                                           flags + 1, wait_limit_, st));
            else
                SH_HIP(launch_pcg_coop(sds, map(kMapCoop, ns), n, map_total_[kMapCoop], int(cfg_.pcg_iterations),
                                       static_cast<PcgSlot *>(d_slots_), flags + 0, flags + 1, wait_limit_, tile, st));
        }
        else if (cfg_.flags & SH_FLAG_NO_GRAPH)
            SH_HIP(enqueue_pcg_launches(ns, matrix_free, st));
        else
        {
            // the PCG loop as one hipGraph, captured once per launch shape and
            // replayed for every GN iteration and every solve of that shape
            SH_HIP(pcg_graph(ns, matrix_free, st));
            SH_HIP(hipGraphLaunch(graph_exec_, st));
        }
        if (!pipe_slots) // the pipelined PCG applies the update itself
        {
            SH_HIP(mark(kPhUpdate, st));
            SH_HIP(launch_update(sds, map(kMapNode, ns), n, map_total_[kMapNode], parity, st));
        }
    }
    SH_HIP(mark(kNumPhases, st));
    return SH_OK;
}

// The per-iteration PCG launches (split or matrix-free) of the current batch.
hipError_t Engine::enqueue_pcg_launches(uint32_t ns, bool matrix_free, hipStream_t st)
{
    const SolveDesc *sds = static_cast<const SolveDesc *>(d_descs_);
    const int n = int(ns);
    double *prs = static_cast<double *>(d_part_rs_), *pdq = static_cast<double *>(d_part_dq_);
    hipError_t e;
#define SH_TRY(x)                                                                                                      \
    if ((e = (x)) != hipSuccess)                                                                                       \
        return e;
    SH_TRY(launch_pcg_init(sds, map(kMapPcg, ns), n, map_total_[kMapPcg], prs, st));
    for (uint32_t k = 0; k < cfg_.pcg_iterations; ++k)
    {
        if (matrix_free)
        {
            // ApplyJtJ without the blocks: d_k, then q = J^T W J d_k from the
            // per-pixel records, then the dot and the update
            SH_TRY(launch_pcg_dir(sds, map(kMapPcg, ns), n, map_total_[kMapPcg], int(k), prs, st));
            SH_TRY(launch_mf_tiles(K_, fp16_, tile_pix(), sds, map(kMapTile, ns), n, map_total_[kMapTile], int(k),
                                   nullptr, st));
            SH_TRY(launch_mf_rows(sds, map(kMapRow, ns), n, map_total_[kMapRow], int(k), nullptr, nullptr, st));
            SH_TRY(launch_pcg_dot(sds, map(kMapPcg, ns), n, map_total_[kMapPcg], int(k), pdq, st));
        }
        else
            SH_TRY(launch_pcg_spmv(sds, map(kMapPcg, ns), n, map_total_[kMapPcg], int(k), prs, pdq, st));
        SH_TRY(launch_pcg_update(sds, map(kMapPcg, ns), n, map_total_[kMapPcg], int(k), matrix_free ? 1u : kPcgSpmvPer,
                                 pdq, prs, st));
    }
#undef SH_TRY
    return hipSuccess;
}

// Captures the PCG launches into graph_exec_ unless the graph of this launch
// shape (solve count, work-group totals, mode) is already there.  Kernel
// arguments are device pointers to the uploaded descriptors and maps, which
// keep their addresses, so a replay reads the current solves.
hipError_t Engine::pcg_graph(uint32_t ns, bool matrix_free, hipStream_t st)
{
    const uint64_t key[5] = {ns, map_total_[kMapPcg], map_total_[kMapTile], map_total_[kMapRow],
                             uint64_t(matrix_free) | (uint64_t(K_) << 1) | (uint64_t(fp16_) << 8)};
    if (graph_exec_ && std::equal(key, key + 5, graph_key_))
        return hipSuccess;
    if (graph_exec_)
    {
        (void)hipGraphExecDestroy(graph_exec_);
        graph_exec_ = nullptr;
    }
    // capture on an engine-owned stream: the caller's may be the legacy NULL
    // stream, which cannot be captured; the graph is then launched on st
    (void)st;
    hipError_t e = hipSuccess;
    if (!cap_stream_ && (e = hipStreamCreateWithFlags(&cap_stream_, hipStreamNonBlocking)) != hipSuccess)
        return e;
    if ((e = hipStreamBeginCapture(cap_stream_, hipStreamCaptureModeThreadLocal)) != hipSuccess)
        return e;
    const hipError_t le = enqueue_pcg_launches(ns, matrix_free, cap_stream_);
    hipGraph_t g = nullptr;
    e = hipStreamEndCapture(cap_stream_, &g);
    if (le != hipSuccess || e != hipSuccess)
    {
        if (g)
            (void)hipGraphDestroy(g);
        return le != hipSuccess ? le : e;
    }
    e = hipGraphInstantiate(&graph_exec_, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e != hipSuccess)
    {
        graph_exec_ = nullptr;
        return e;
    }
    std::copy(key, key + 5, graph_key_);
    return hipSuccess;
}

// Phase timing (SH_FLAG_PHASE_TIMING): an event before each GN-phase launch;
// the span from one mark to the next is charged to the earlier mark's phase.
hipError_t Engine::mark(int phase, hipStream_t st)
{
    if (!(cfg_.flags & SH_FLAG_PHASE_TIMING))
        return hipSuccess;
    if (n_marks_ == marks_.size())
    {
        // no system-scope fence: the marks order device work only, and a fence
        // per mark would add an L2 write-back to every phase it times
        hipEvent_t e;
        if (hipError_t r = hipEventCreateWithFlags(&e, hipEventDisableSystemFence); r != hipSuccess)
            return r;
        marks_.push_back({e, 0});
    }
    marks_[n_marks_].phase = phase;
    return hipEventRecord(marks_[n_marks_++].ev, st);
}

void Engine::collect_marks()
{
    std::lock_guard<std::mutex> lock(phase_mu_);
    for (size_t m = 0; m + 1 < n_marks_; ++m)
    {
        float ms = 0.f;
        if (marks_[m].phase < kNumPhases && hipEventElapsedTime(&ms, marks_[m].ev, marks_[m + 1].ev) == hipSuccess)
        {
            phase_ms_[marks_[m].phase] += double(ms);
            phase_calls_[marks_[m].phase] += 1;
        }
    }
    n_marks_ = 0;
}

int Engine::phase_times(double *ms, uint32_t *calls, uint32_t n, bool reset)
{
    std::lock_guard<std::mutex> lock(phase_mu_);
    for (uint32_t p = 0; p < n && p < uint32_t(kNumPhases); ++p)
    {
        if (ms)
            ms[p] = phase_ms_[p];
        if (calls)
            calls[p] = phase_calls_[p];
    }
    if (reset)
        for (int p = 0; p < kNumPhases; ++p)
        {
            phase_ms_[p] = 0.0;
            phase_calls_[p] = 0;
        }
    return SH_OK;
}

const char *Engine::phase_name(uint32_t p)
{
    static const char *names[kNumPhases] = {"dense_terms", "reg_terms", "rows_seg", "rows_combine",
                                            "diag_rhs",    "offdiag",   "dinv",     "pcg",
                                            "update",      "tiles",     "tiles_combine"};
    return p < uint32_t(kNumPhases) ? names[p] : nullptr;
}

int Engine::solve(uint32_t ns, hipStream_t st)
{
    n_marks_ = 0;
    if (ns == 0 || ns > slots_.size())
        return SH_E_ARG;
    for (uint32_t s = 0; s < ns; ++s)
        if (!slots_[s].has_inputs)
            return SH_E_STATE;
    int rc;
    {
        std::vector<uint32_t> all(ns);
        for (uint32_t s = 0; s < ns; ++s)
            all[s] = s;
        if ((rc = build_indexes(all.data(), ns, st)) != SH_OK)
            return rc;
    }
    batch_.resize(ns);
    for (uint32_t s = 0; s < ns; ++s)
    {
        batch_[s] = s;
        slots_[s].d.gn_iter = 0;
    }
    build_maps(ns);
    if ((rc = upload(ns, st)) != SH_OK)
        return rc;
    auto run = [&]() -> int {
        int r;
        if ((r = enqueue_gn(ns, st, cfg_.gn_iterations, true)) != SH_OK)
            return r;
        if (cfg_.flags & SH_FLAG_COST_HISTORY)
        {
            // cost at the final warp field: the terms once more, then the reduction
            const SolveDesc *sds = static_cast<const SolveDesc *>(d_descs_);
            const int it = int(cfg_.gn_iterations);
            SH_HIP(launch_terms(K_, fp16_, sds, map(kMapPixel, ns), map_total_[kMapPixel], map(kMapReg, ns),
                                map_total_[kMapReg], int(ns), it, st, 0));
            SH_HIP(launch_cost_final(sds, int(ns), it, st));
        }
        return finish(st);
    };
    rc = run();
    if (rc == SH_E_HIP && barrier_timeout_)
    {
        // the whole solve again, from the identity, with the split PCG
        if ((rc = fall_back_to_split_pcg(st)) != SH_OK)
            return rc;
        n_marks_ = 0;
        rc = run();
    }
    if (rc != SH_OK)
        return rc;
    for (uint32_t s = 0; s < ns; ++s)
    {
        slots_[s].d.gn_iter = int(cfg_.gn_iterations);
        slots_[s].solved = true;
        slots_[s].result_n = uint32_t(slots_[s].d.N);
    }
    return SH_OK;
}

// y = J^T W J x (+ damping) with the system of the slot's last GN iteration:
// over the materialised blocks, or matrix-free from the per-pixel records.
int Engine::apply_jtj(uint32_t slot, const float *x, float *y, bool matrix_free, hipStream_t st)
{
    if (slot >= slots_.size() || !slots_[slot].solved || !x || !y)
        return !x || !y ? SH_E_ARG : SH_E_STATE;
    if (matrix_free && (cfg_.flags & (SH_FLAG_PAIR_MAJOR | SH_FLAG_ROW_SEGMENTS)))
        return SH_E_ARG; // the tile index is not built for those paths
    batch_.assign(1, slot);
    build_maps(1);
    int rc;
    if ((rc = upload(1, st)) != SH_OK)
        return rc;
    const SolveDesc *sds = static_cast<const SolveDesc *>(d_descs_);
    if (matrix_free)
    {
        if (slots_[slot].records_fused)
        {
            // the records of the last GN iteration were built inside the tile
            // kernel and never stored: store them from the warp field that
            // iteration started from (the other buffer of the pair)
            SH_HIP(launch_terms(K_, fp16_, sds, map(kMapPixel, 1), map_total_[kMapPixel], map(kMapReg, 1), 0, 1, -1,
                                st));
            slots_[slot].records_fused = false;
        }
        SH_HIP(launch_mf_tiles(K_, fp16_, uint32_t(slots_[slot].d.tile_pix), sds, map(kMapTile, 1), 1,
                               map_total_[kMapTile], 0, x, st));
        SH_HIP(launch_mf_rows(sds, map(kMapRow, 1), 1, map_total_[kMapRow], 0, x, y, st));
    }
    else
        SH_HIP(launch_spmv_rows(sds, map(kMapRow, 1), 1, map_total_[kMapRow], x, y, st));
    SH_HIP(hipStreamSynchronize(st));
    return SH_OK;
}

// Tuning that can change between solves without reallocating: the
// materialisation path, the PCG variant and the resident PCG's rows per group.
static constexpr uint32_t kTunableFlags = SH_FLAG_ROW_SEGMENTS | SH_FLAG_STREAMING_PCG | SH_FLAG_NO_PERSISTENT_PCG |
                                          SH_FLAG_PIPELINED_PCG | SH_FLAG_TILE_PIX_64 | SH_FLAG_TILE_PIX_256;

int Engine::set_tuning(const sh_tuning &t)
{
    if ((t.flags & ~kTunableFlags) || t.spmv_mode > SH_SPMV_AUTO || t.pcg_rows_per_group > kPcgResRows ||
        ((t.flags & SH_FLAG_TILE_PIX_64) && (t.flags & SH_FLAG_TILE_PIX_256)) ||
        (cfg_.flags & (SH_FLAG_PAIR_MAJOR)) ||
        (t.spmv_mode == SH_SPMV_MATRIX_FREE && (t.flags & SH_FLAG_ROW_SEGMENTS)))
        return SH_E_ARG;
    cfg_.flags = (cfg_.flags & ~kTunableFlags) | t.flags;
    cfg_.spmv_mode = t.spmv_mode;
    res_rows_ = t.pcg_rows_per_group ? t.pcg_rows_per_group : kPcgResRows;
    return SH_OK;
}

sh_tuning Engine::tuning() const
{
    sh_tuning t{};
    t.flags = cfg_.flags & kTunableFlags;
    t.spmv_mode = cfg_.spmv_mode;
    t.pcg_rows_per_group = res_rows_;
    return t;
}

// Times every candidate tuning on the slots' current inputs (median of
// `repeats` solves each, HIP events on `st`) and keeps the fastest.
// Median solve time of tuning c (after one warm-up solve) into *ms; 0 when a
// persistent PCG's barrier wait ran out during it (it then ran as the split PCG).
int Engine::time_candidate(const sh_tuning &c, uint32_t ns, hipStream_t st, uint32_t repeats, hipEvent_t e0,
                           hipEvent_t e1, double *ms_out)
{
    int rc;
    if ((rc = set_tuning(c)) != SH_OK)
        return rc;
    const uint32_t fallbacks = pcg_fallbacks_;
    std::vector<double> t;
    for (uint32_t r = 0; r < repeats + 1; ++r)
    {
        float ms = 0.f;
        if (hipEventRecord(e0, st) != hipSuccess)
            return SH_E_HIP;
        if ((rc = solve(ns, st)) != SH_OK)
            return rc;
        if (hipEventRecord(e1, st) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
            hipEventElapsedTime(&ms, e0, e1) != hipSuccess)
            return SH_E_HIP;
        if (r > 0) // the first run warms up
            t.push_back(ms);
    }
    std::sort(t.begin(), t.end());
    *ms_out = pcg_fallbacks_ != fallbacks ? 0.0 : t[t.size() / 2];
    return SH_OK;
}

int Engine::autotune(uint32_t ns, hipStream_t st, uint32_t repeats, sh_tuning *best_out)
{
    if (cfg_.flags & SH_FLAG_PAIR_MAJOR)
        return SH_E_ARG;
    std::vector<sh_tuning> cands;
    for (uint32_t rows : {85u, 64u, 48u, 32u})
        cands.push_back({0u, SH_SPMV_MATERIALIZED, rows, 0.0});
    // smallest first: a later candidate must win by 2% (below), and 16 rows
    // beat 24 by less than that on a 1,024-node frame
    for (uint32_t rows : {16u, 24u, 32u, 48u, 64u, 85u})
        cands.push_back({SH_FLAG_PIPELINED_PCG, SH_SPMV_MATERIALIZED, rows, 0.0});
    cands.push_back({SH_FLAG_STREAMING_PCG, SH_SPMV_MATERIALIZED, kPcgResRows, 0.0});
    cands.push_back({SH_FLAG_NO_PERSISTENT_PCG, SH_SPMV_MATERIALIZED, kPcgResRows, 0.0});
    cands.push_back({SH_FLAG_ROW_SEGMENTS, SH_SPMV_MATERIALIZED, kPcgResRows, 0.0});
    cands.push_back({0u, SH_SPMV_MATRIX_FREE, kPcgResRows, 0.0});
    hipEvent_t e0, e1;
    SH_HIP(hipEventCreate(&e0));
    SH_HIP(hipEventCreate(&e1));
    const sh_tuning keep = tuning();
    sh_tuning best{};
    best.ms = 1e30;
    int rc = SH_OK;
    for (sh_tuning &c : cands)
    {
        double ms = 0.0;
        if ((rc = time_candidate(c, ns, st, repeats, e0, e1, &ms)) != SH_OK)
            break;
        if (ms <= 0.0)
            continue; // its barrier waits ran out: timed as the split PCG, and not chosen
        c.ms = ms;
        // a later candidate must be 2% faster to replace an earlier one, so that
        // near-ties resolve to the same (earlier, default-first) choice run to run
        if (c.ms < best.ms * (best.ms < 1e30 ? 0.98 : 1.0))
            best = c;
    }
    // then the tile size, for a winner on the tile path: 64 and 256 pixels
    // against the default 128 (the same 2% margin)
    if (rc == SH_OK && best.ms < 1e30 && !(best.flags & SH_FLAG_ROW_SEGMENTS))
    {
        const sh_tuning base = best;
        for (uint32_t tf : {uint32_t(SH_FLAG_TILE_PIX_64), uint32_t(SH_FLAG_TILE_PIX_256)})
        {
            sh_tuning c = base;
            c.flags = (c.flags & ~uint32_t(SH_FLAG_TILE_PIX_64 | SH_FLAG_TILE_PIX_256)) | tf;
            double ms = 0.0;
            if ((rc = time_candidate(c, ns, st, repeats, e0, e1, &ms)) != SH_OK)
                break;
            c.ms = ms;
            if (ms > 0.0 && ms < best.ms * 0.98)
                best = c;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc != SH_OK)
    {
        (void)set_tuning(keep);
        return rc;
    }
    if ((rc = set_tuning(best)) != SH_OK)
        return rc;
    if (best_out)
        *best_out = best;
    return SH_OK;
}

// FP64 cost history of a solved slot (host copy).
int Engine::cost_history(uint32_t slot, double *out, uint32_t capacity, uint32_t *count) const
{
    if (slot >= slots_.size() || !slots_[slot].solved)
        return SH_E_STATE;
    const uint32_t n = cfg_.gn_iterations + ((cfg_.flags & SH_FLAG_COST_HISTORY) ? 1u : 0u);
    if (count)
        *count = n;
    if (!out)
        return SH_OK;
    if (capacity < n)
        return SH_E_CAPACITY;
    SH_HIP(hipMemcpy(out, slots_[slot].d.cost, size_t(n) * sizeof(double), hipMemcpyDeviceToHost));
    return SH_OK;
}

// Waits for the work on st by polling ev (one event per thread that waits):
// the host sees the readbacks of an index build and the end of a solve within
// microseconds, where a blocking synchronisation measured 22-38 us late on
// this device.
int Engine::wait_stream(hipStream_t st, hipEvent_t ev)
{
    SH_HIP(hipEventRecord(ev, st));
    hipError_t q;
    while ((q = hipEventQuery(ev)) == hipErrorNotReady)
        __builtin_ia32_pause();
    if (q != hipSuccess)
    {
        last_hip_error = q;
        return SH_E_HIP;
    }
    return SH_OK;
}

// Synchronise the launch stream and check the PCG barrier flag.
int Engine::finish(hipStream_t st)
{
    barrier_timeout_ = false;
    SH_HIP(hipMemcpyAsync(h_flag_, static_cast<uint32_t *>(d_flags_) + 1, 4, hipMemcpyDeviceToHost, st));
    if (int rc = wait_stream(st, sync_ev_); rc != SH_OK)
        return rc;
    collect_marks();
    if (*h_flag_ != 0)
    {
        barrier_timeout_ = true;
        last_hip_error = hipErrorLaunchTimeOut; // a persistent-PCG barrier wait ran out
        return SH_E_HIP;
    }
    return SH_OK;
}

// A persistent PCG needs every group of a solve resident at once.  Kernels
// that the caller runs on other streams can hold CUs long enough for a
// barrier wait to run out; the launch then drained with meaningless sums and
// may have left the slots' epochs out of step with the epoch base.  Clear the
// barrier state and switch this engine to the split PCG, which has no
// inter-group waits; the caller re-runs the GN iterations from the warp field
// they started from (the failed updates only wrote the other DQ buffer or,
// for a whole solve, start again from the identity).
int Engine::fall_back_to_split_pcg(hipStream_t st)
{
    const size_t groups = slots_.size() * size_t(kPcgMaxGroups);
    SH_HIP(hipMemsetAsync(d_slots_, 0, groups * sizeof(PcgSlot), st));
    SH_HIP(hipMemsetAsync(d_slots2_, 0, groups * sizeof(PcgSlot2), st));
    SH_HIP(hipMemsetAsync(d_flags_, 0, 2 * sizeof(uint32_t), st)); // epoch base and barrier error
    SH_HIP(hipStreamSynchronize(st));
    cfg_.flags = (cfg_.flags & ~uint32_t(SH_FLAG_STREAMING_PCG | SH_FLAG_PIPELINED_PCG)) | SH_FLAG_NO_PERSISTENT_PCG;
    barrier_timeout_ = false;
    ++pcg_fallbacks_;
    return SH_OK;
}

// Index build for one slot and its identity start: the admission half of
// continuous batching (uses the index workspace only).
int Engine::admit(uint32_t slot, hipStream_t st)
{
    if (slot >= slots_.size() || !slots_[slot].has_inputs)
        return SH_E_STATE;
    Slot &sl = slots_[slot];
    sl.solved = false;
    if (int rc = build_index(slot, st); rc != SH_OK)
        return rc;
    SH_HIP(launch_identity_dq(sl.d.dq[0], uint32_t(sl.d.N), st));
    sl.d.gn_iter = 0;
    return wait_stream(st, index_ev_);
}

int Engine::admit_many(const uint32_t *list, uint32_t n, hipStream_t st, int *rcs)
{
    for (uint32_t i = 0; i < n; ++i)
    {
        if (list[i] >= slots_.size() || !slots_[list[i]].has_inputs)
            return SH_E_STATE;
        slots_[list[i]].solved = false;
    }
    if (int rc = build_indexes(list, n, st, rcs); rc != SH_OK)
        return rc;
    for (uint32_t i = 0; i < n; ++i)
        if (rcs[i] == SH_OK)
        {
            Slot &sl = slots_[list[i]];
            SH_HIP(launch_identity_dq(sl.d.dq[0], uint32_t(sl.d.N), st));
            sl.d.gn_iter = 0;
        }
    return wait_stream(st, index_ev_);
}

// One GN iteration for an arbitrary set of admitted slots, each at its own
// iteration: the step half of continuous batching (uses the launch state only).
int Engine::step(const uint32_t *list, uint32_t n, hipStream_t st)
{
    n_marks_ = 0;
    if (n == 0)
        return SH_OK;
    batch_.assign(list, list + n);
    for (uint32_t s = 0; s < n; ++s)
        if (batch_[s] >= slots_.size() || !slots_[batch_[s]].indexed ||
            slots_[batch_[s]].d.gn_iter >= int(cfg_.gn_iterations))
            return SH_E_STATE;
    build_maps(n);
    int rc;
    if ((rc = upload(n, st)) != SH_OK)
        return rc;
    if ((rc = enqueue_gn(n, st, 1, false)) != SH_OK)
        return rc;
    rc = finish(st);
    if (rc == SH_E_HIP && barrier_timeout_)
    {
        // the iteration again from the same DQ buffer (the failed update only
        // wrote the other one), with the split PCG
        if ((rc = fall_back_to_split_pcg(st)) != SH_OK)
            return rc;
        n_marks_ = 0;
        if ((rc = enqueue_gn(n, st, 1, false)) != SH_OK)
            return rc;
        rc = finish(st);
    }
    if (rc != SH_OK)
        return rc;
    for (uint32_t s = 0; s < n; ++s)
    {
        Slot &sl = slots_[batch_[s]];
        sl.d.gn_iter += 1;
        sl.solved = sl.d.gn_iter == int(cfg_.gn_iterations);
        if (sl.solved)
            sl.result_n = uint32_t(sl.d.N);
    }
    return SH_OK;
}

const dq8 *Engine::result(uint32_t slot) const
{
    return slots_[slot].d.dq[cfg_.gn_iterations & 1u];
}

int Engine::debug_view(uint32_t slot, const char *name, const void **ptr, size_t *count) const
{
    if (slot >= slots_.size() || !name || !ptr || !count)
        return SH_E_ARG;
    const SolveDesc &d = slots_[slot].d;
    const std::string n(name);
    const size_t P = size_t(d.P), N = size_t(d.N), U = size_t(d.U), E = size_t(d.E), K = size_t(K_);
    struct V
    {
        const char *name;
        const void *p;
        size_t c;
    };
    const V views[] = {
        {"pix", d.pix, P * 4},
        {"gpix", d.gpix, P * 4},
        {"pknn", d.pknn, P * K},
        {"pw", d.pw, P * K},
        {"n2t_off", d.n2t_off, N + 1},
        {"n2t_terms", d.n2t_terms, P * K + 2 * E + N},
        {"half_keys", d.half_keys, U},
        {"half_off", d.half_off, U + 1},
        {"pair_entries", d.pair_entries, size_t(d.n_pair_entries)},
        {"upper_pos", d.upper_pos, U},
        {"lower_pos", d.lower_pos, U},
        {"row_ptr", d.row_ptr, N + 1},
        {"blk_col", d.blk_col, N + 2 * U},
        {"hg", d.jr, P * kHG},
        {"dense_cnt", d.dense_cnt, N},
        {"seg_ptr", d.seg_ptr, N + 1},
        {"tile_cbase", d.tile_cbase, size_t(d.n_tiles) + 1},
        {"tile_sbase", d.tile_sbase, size_t(d.n_tiles) + 1},
        {"tile_nodes", d.tile_nodes, size_t(d.n_tiles)},
        {"list_off", d.list_off, N + 2 * U + 1},
        {"blk_transpose", d.blk_transpose, N + 2 * U},
        {"reg", d.reg, E * kReg},
        {"blk", d.blk, (N + 2 * U) * 36},
        {"dinv", d.dinv, N * 36},
        {"rhs", d.rhs, N * 6},
        {"x", d.x, N * 6},
        {"dq0", d.dq[0], N * 8},
        {"dq1", d.dq[1], N * 8},
        {"delta", d.delta, size_t(cfg_.pcg_iterations) + 1},
        {"rot_cut", d.rot_cut, size_t(cfg_.gn_iterations) * N},
        {"twist_l1", d.twist_l1, size_t(cfg_.gn_iterations) * N},
    };
    for (const V &v : views)
        if (n == v.name)
        {
            *ptr = v.p;
            *count = v.c;
            return SH_OK;
        }
    return SH_E_ARG;
}

} // namespace sh

// ======================================================================= C-ABI
struct sh_solver
{
    sh::Engine eng;
    struct JtjOp
    {
        sh_solver *solver;
        bool matrix_free;
    } jtj_op[2] = {{this, false}, {this, true}};
};
struct sh_batch
{
    sh::Engine eng;
};

extern "C"
{
    const char *sh_version(void) { return "starhub_amd 0.1.0 gfx950"; }

    const char *sh_last_hip_error(void) { return hipGetErrorString(sh::last_hip_error); }

    const char *sh_status_string(int s)
    {
        switch (s)
        {
        case SH_OK:
            return "ok";
        case SH_E_ARG:
            return "invalid argument";
        case SH_E_CAPACITY:
            return "capacity exceeded";
        case SH_E_HIP:
            return "HIP runtime error";
        case SH_E_NAN:
            return "non-finite system";
        case SH_E_STATE:
            return "call out of order";
        case SH_E_NOMEM:
            return "device allocation failed";
        default:
            return "unknown status";
        }
    }

    int sh_solver_create(const sh_solver_config *config, sh_solver **out)
    {
        if (!config || !out)
            return SH_E_ARG;
        *out = nullptr;
        sh_solver *s = new sh_solver();
        const int rc = s->eng.init(*config, 1);
        if (rc != SH_OK)
        {
            delete s;
            return rc;
        }
        *out = s;
        return SH_OK;
    }

    int sh_solver_destroy(sh_solver *solver)
    {
        delete solver;
        return SH_OK;
    }

    int sh_solver_set_inputs(sh_solver *solver, const sh_camera *camera, const sh_measure_maps *measure,
                             const sh_render_maps *render, const sh_geometry *geometry,
                             const sh_node_graph *node_graph, const sh_node_flow *node_flow, const sh_flow_map *flow,
                             const sh_keypoints *keypoints, const float cam2world[16])
    {
        if (!solver)
            return SH_E_ARG;
        return solver->eng.set_inputs(0, camera, measure, render, geometry, node_graph, node_flow, flow, keypoints,
                                      cam2world);
    }

    int sh_solver_solve(sh_solver *solver, sh_stream_t stream)
    {
        if (!solver)
            return SH_E_ARG;
        return solver->eng.solve(1, reinterpret_cast<hipStream_t>(stream));
    }

    int sh_solver_node_se3(const sh_solver *solver, const sh_dual_quat **view, uint32_t *num_nodes)
    {
        if (!solver || !view || !num_nodes)
            return SH_E_ARG;
        *view = reinterpret_cast<const sh_dual_quat *>(solver->eng.result(0));
        *num_nodes = solver->eng.result_nodes(0);
        return SH_OK;
    }

    int sh_solver_sizes(const sh_solver *solver, uint32_t *num_pixels, uint32_t *num_pairs, uint32_t *num_node_terms)
    {
        if (!solver)
            return SH_E_ARG;
        const sh::SolveDesc &d = solver->eng.desc(0);
        if (num_pixels)
            *num_pixels = uint32_t(d.P);
        if (num_pairs)
            *num_pairs = uint32_t(d.U);
        if (num_node_terms)
            *num_node_terms = uint32_t(d.P * d.K + 2 * d.E + d.N);
        return SH_OK;
    }

    int sh_solver_debug_view(const sh_solver *solver, const char *name, const void **device_ptr, size_t *count)
    {
        if (!solver)
            return SH_E_ARG;
        return solver->eng.debug_view(0, name, device_ptr, count);
    }

    int sh_solver_cost_history(const sh_solver *solver, double *out, uint32_t capacity, uint32_t *count)
    {
        if (!solver)
            return SH_E_ARG;
        return solver->eng.cost_history(0, out, capacity, count);
    }

    int sh_solver_autotune(sh_solver *solver, sh_stream_t stream, uint32_t repeats, sh_tuning *best)
    {
        if (!solver || repeats == 0)
            return SH_E_ARG;
        return solver->eng.autotune(1, reinterpret_cast<hipStream_t>(stream), repeats, best);
    }

    int sh_solver_set_tuning(sh_solver *solver, const sh_tuning *tuning)
    {
        if (!solver || !tuning)
            return SH_E_ARG;
        return solver->eng.set_tuning(*tuning);
    }

    int sh_solver_get_tuning(const sh_solver *solver, sh_tuning *tuning)
    {
        if (!solver || !tuning)
            return SH_E_ARG;
        *tuning = solver->eng.tuning();
        return SH_OK;
    }

    int sh_solver_set_wait_limit(sh_solver *solver, uint32_t polls)
    {
        if (!solver)
            return SH_E_ARG;
        solver->eng.set_wait_limit(polls);
        return SH_OK;
    }

    int sh_solver_pcg_fallbacks(const sh_solver *solver, uint32_t *count)
    {
        if (!solver || !count)
            return SH_E_ARG;
        *count = solver->eng.pcg_fallbacks();
        return SH_OK;
    }

    int sh_batch_set_tuning(sh_batch *batch, const sh_tuning *tuning)
    {
        if (!batch || !tuning)
            return SH_E_ARG;
        return batch->eng.set_tuning(*tuning);
    }

    int sh_batch_autotune(sh_batch *batch, uint32_t num_solves, sh_stream_t stream, uint32_t repeats,
                          sh_tuning *best)
    {
        if (!batch || repeats == 0 || num_solves == 0 || num_solves > batch->eng.num_slots())
            return SH_E_ARG;
        return batch->eng.autotune(num_solves, reinterpret_cast<hipStream_t>(stream), repeats, best);
    }

    int sh_solver_apply_jtj(sh_solver *solver, const float *x, float *y, uint32_t matrix_free, sh_stream_t stream)
    {
        if (!solver)
            return SH_E_ARG;
        return solver->eng.apply_jtj(0, x, y, matrix_free != 0, reinterpret_cast<hipStream_t>(stream));
    }

    static int solver_jtj_cb(void *user, const float *x, float *y, sh_stream_t stream)
    {
        const sh_solver::JtjOp *op = static_cast<const sh_solver::JtjOp *>(user);
        return op->solver->eng.apply_jtj(0, x, y, op->matrix_free, reinterpret_cast<hipStream_t>(stream));
    }

    int sh_solver_spmv_ops(sh_solver *solver, uint32_t matrix_free, sh_spmv_ops *ops)
    {
        if (!solver || !ops)
            return SH_E_ARG;
        if (!solver->eng.solved(0))
            return SH_E_STATE;
        ops->user = &solver->jtj_op[matrix_free ? 1 : 0];
        ops->matrix_size = 6u * uint32_t(solver->eng.desc(0).N);
        ops->apply_spmv = solver_jtj_cb;
        ops->init_residual = nullptr;
        return SH_OK;
    }

    int sh_skin_surfels(const float *surfel_vertex4, uint32_t num_surfels, const float *node_coords4,
                        uint32_t num_nodes, uint32_t knn, float node_radius_square, uint16_t *surfel_knn,
                        float *spatial_weight, float *connect_weight, sh_stream_t stream)
    {
        if ((knn != 4 && knn != 8) || num_nodes < knn || num_nodes > 65535 || !surfel_vertex4 || !node_coords4 ||
            !surfel_knn || !spatial_weight || !connect_weight)
            return SH_E_ARG;
        const hipError_t e = sh::launch_skin(knn, reinterpret_cast<const float4 *>(surfel_vertex4), num_surfels,
                                             reinterpret_cast<const float4 *>(node_coords4), num_nodes,
                                             node_radius_square, surfel_knn, spatial_weight, connect_weight,
                                             reinterpret_cast<hipStream_t>(stream));
        if (e != hipSuccess)
        {
            sh::last_hip_error = e;
            return SH_E_HIP;
        }
        return SH_OK;
    }

    static int hip_rc(hipError_t e)
    {
        if (e != hipSuccess)
        {
            sh::last_hip_error = e;
            return SH_E_HIP;
        }
        return SH_OK;
    }

    static bool depth_camera_ok(const sh_depth_camera *c)
    {
        return c && c->width > 0 && c->height > 0 && c->width <= 16384 && c->height <= 16384 && c->fx != 0.f &&
               c->fy != 0.f && c->downsample_scale > 0.f && c->downsample_scale <= 1.f;
    }

    int sh_filter_depth(const uint16_t *depth_mm, const sh_depth_camera *c, float *filtered, sh_stream_t stream)
    {
        if (!depth_camera_ok(c) || !depth_mm || !filtered)
            return SH_E_ARG;
        return hip_rc(sh::launch_filter_depth(depth_mm, int(c->width), int(c->height), c->fx, c->fy, c->cx, c->cy,
                                              c->clip_near, c->clip_far, filtered,
                                              reinterpret_cast<hipStream_t>(stream)));
    }

    int sh_measure_maps_from_depth(const float *filtered, const sh_depth_camera *c, float *vertex_confid,
                                   float *normal_radius, sh_stream_t stream)
    {
        if (!depth_camera_ok(c) || !filtered || !vertex_confid || !normal_radius)
            return SH_E_ARG;
        // filterAndScaleVertex's size: the float product, truncated (SurfelMapInitializer.cu:319-320)
        const int w = int(unsigned(float(c->width) * c->downsample_scale));
        const int h = int(unsigned(float(c->height) * c->downsample_scale));
        const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
        int rc = hip_rc(sh::launch_scaled_vertex(filtered, int(c->width), int(c->height), w, h, c->downsample_scale,
                                                 c->fx, c->fy, c->cx, c->cy, c->clip_near, c->clip_far,
                                                 vertex_confid, st));
        if (rc == SH_OK)
            rc = hip_rc(sh::launch_normal_radius(vertex_confid, w, h, c->surfel_radius_scale, normal_radius, st));
        return rc;
    }

    int sh_normal_radius_map(const float *vertex_confid, uint32_t width, uint32_t height, float radius_scale,
                             float *normal_radius, sh_stream_t stream)
    {
        if (!vertex_confid || !normal_radius || width > 16384 || height > 16384)
            return SH_E_ARG;
        return hip_rc(sh::launch_normal_radius(vertex_confid, int(width), int(height), radius_scale, normal_radius,
                                               reinterpret_cast<hipStream_t>(stream)));
    }

    int sh_vertex_confid_map(const uint16_t *depth_mm, uint32_t width, uint32_t height, float fx, float fy, float cx,
                             float cy, float *vertex_confid, sh_stream_t stream)
    {
        if (!depth_mm || !vertex_confid || width > 16384 || height > 16384 || fx == 0.f || fy == 0.f)
            return SH_E_ARG;
        return hip_rc(sh::launch_vertex_confid(depth_mm, int(width), int(height), fx, fy, cx, cy, vertex_confid,
                                               reinterpret_cast<hipStream_t>(stream)));
    }

    int sh_flow_map_from_of16(const uint16_t *of16, uint32_t raw_width, uint32_t raw_height, float scale,
                              float *flow_map2, sh_stream_t stream)
    {
        if (!of16 || !flow_map2 || raw_width == 0 || raw_height == 0 || raw_width > 16384 || raw_height > 16384 ||
            !(scale > 0.f) || scale > 1.f)
            return SH_E_ARG;
        return hip_rc(sh::launch_flow_from_of16(of16, int(raw_width), int(raw_height), scale, flow_map2,
                                                reinterpret_cast<hipStream_t>(stream)));
    }

    int sh_node_motion_from_flow(const float *rgbd_prev4, const float *rgbd4, const float *flow_map2,
                                 const uint32_t *index_map_prev, uint32_t width, uint32_t height,
                                 const uint16_t *surfel_knn, const float *surfel_spatial, uint32_t num_surfels,
                                 uint32_t knn, const float cam2world[16], float fx, float fy, float cx, float cy,
                                 uint32_t num_nodes, void *workspace, float *out4, sh_stream_t stream)
    {
        if ((knn != 4 && knn != 8) || !cam2world || !workspace || !out4 || width > 16384 || height > 16384 ||
            fx == 0.f || fy == 0.f ||
            (width && height && (!rgbd_prev4 || !rgbd4 || !flow_map2 || !index_map_prev || !surfel_knn ||
                                 !surfel_spatial)))
            return SH_E_ARG;
        return hip_rc(sh::launch_node_motion(rgbd_prev4, rgbd4, flow_map2, index_map_prev, int(width), int(height),
                                             surfel_knn, surfel_spatial, num_surfels, int(knn), cam2world, fx, fy, cx,
                                             cy, num_nodes, static_cast<unsigned long long *>(workspace), out4,
                                             reinterpret_cast<hipStream_t>(stream)));
    }

    int sh_node_motion_from_flow_noalloc(const float *rgbd_prev4, const float *rgbd4, const float *flow_map2,
                                         const uint32_t *index_map_prev, uint32_t width, uint32_t height,
                                         const uint16_t *surfel_knn, const float *surfel_spatial,
                                         uint32_t num_surfels, uint32_t knn, const float cam2world[16], float fx,
                                         float fy, float cx, float cy, uint32_t num_nodes, float *out4,
                                         sh_stream_t stream)
    {
        if ((knn != 4 && knn != 8) || !cam2world || !out4 || width > 16384 || height > 16384 || fx == 0.f ||
            fy == 0.f ||
            (width && height && (!rgbd_prev4 || !rgbd4 || !flow_map2 || !index_map_prev || !surfel_knn ||
                                 !surfel_spatial)))
            return SH_E_ARG;
        if (num_nodes > sh::kNoAllocMaxNodes)
            return SH_E_CAPACITY;
        unsigned long long *sums = nullptr;
        if (const hipError_t e = sh::noalloc_sums(&sums); e != hipSuccess)
            return hip_rc(e);
        return hip_rc(sh::launch_node_motion(rgbd_prev4, rgbd4, flow_map2, index_map_prev, int(width), int(height),
                                             surfel_knn, surfel_spatial, num_surfels, int(knn), cam2world, fx, fy, cx,
                                             cy, num_nodes, sums, out4, reinterpret_cast<hipStream_t>(stream)));
    }

    int sh_render_solver_maps(const float *vertex4, const float *normal4, const float *color_time4,
                              uint32_t num_surfels, const float world2camera[16], const sh_camera *cam,
                              float max_depth, float current_time, int with_recent_observation, void *zbuffer,
                              float *out_vertex4, float *out_normal4, uint32_t *out_index, sh_stream_t stream)
    {
        if (!world2camera || !cam || !zbuffer || !out_vertex4 || !out_normal4 || !out_index ||
            (num_surfels && (!vertex4 || !normal4)) || cam->width == 0 || cam->height == 0 || cam->width > 16384 ||
            cam->height > 16384 || !(max_depth > 0.f))
            return SH_E_ARG;
        return hip_rc(sh::launch_render_solver_maps(
            vertex4, normal4, color_time4, num_surfels, world2camera, int(cam->width), int(cam->height), cam->fx,
            cam->fy, cam->cx, cam->cy, max_depth, current_time, with_recent_observation != 0,
            static_cast<unsigned long long *>(zbuffer), out_vertex4, out_normal4, out_index,
            reinterpret_cast<hipStream_t>(stream)));
    }

    int sh_forward_warp(const sh_dual_quat *warp_field, uint32_t num_nodes, uint32_t knn, const float *ref_v4,
                        const float *ref_n4, const uint16_t *s_knn, const float *s_spatial, const float *s_connect,
                        uint32_t num_surfels, const float *ref_node4, const uint16_t *n_knn, const float *n_spatial,
                        const float *n_connect, float *live_v4, float *live_n4, float *live_node4, sh_stream_t stream)
    {
        if ((knn != 4 && knn != 8) || !warp_field || num_nodes == 0)
            return SH_E_ARG;
        if (num_surfels && (!ref_v4 || !ref_n4 || !s_knn || !s_spatial || !s_connect || !live_v4 || !live_n4))
            return SH_E_ARG;
        const bool nodes = ref_node4 != nullptr;
        if (nodes && (!n_knn || !n_spatial || !n_connect || !live_node4))
            return SH_E_ARG;
        const hipError_t e = sh::launch_forward_warp(
            knn, reinterpret_cast<const float4 *>(warp_field), reinterpret_cast<const float4 *>(ref_v4),
            reinterpret_cast<const float4 *>(ref_n4), s_knn, s_spatial, s_connect, num_surfels,
            reinterpret_cast<const float4 *>(ref_node4), n_knn, n_spatial, n_connect, nodes ? num_nodes : 0,
            reinterpret_cast<float4 *>(live_v4), reinterpret_cast<float4 *>(live_n4),
            reinterpret_cast<float4 *>(live_node4), reinterpret_cast<hipStream_t>(stream));
        if (e != hipSuccess)
        {
            sh::last_hip_error = e;
            return SH_E_HIP;
        }
        return SH_OK;
    }

    int sh_build_node_graph(const float *node_coords4, uint32_t num_nodes, uint32_t knn, float node_radius_square,
                            uint16_t *node_knn, float *node_spatial_weight, uint16_t *node_graph,
                            float *node_connect_weight, sh_stream_t stream)
    {
        if ((knn != 4 && knn != 8) || num_nodes < knn || num_nodes > 65535 || !node_coords4 || !node_knn ||
            !node_spatial_weight || !node_graph || !node_connect_weight)
            return SH_E_ARG;
        const hipError_t e = sh::launch_node_graph(knn, reinterpret_cast<const float4 *>(node_coords4), num_nodes,
                                                   node_radius_square, node_knn, node_spatial_weight, node_graph,
                                                   node_connect_weight, reinterpret_cast<hipStream_t>(stream));
        if (e != hipSuccess)
        {
            sh::last_hip_error = e;
            return SH_E_HIP;
        }
        return SH_OK;
    }

    int sh_batch_create(const sh_solver_config *config, uint32_t max_solves, sh_batch **out)
    {
        if (!config || !out || max_solves == 0)
            return SH_E_ARG;
        *out = nullptr;
        sh_batch *b = new sh_batch();
        const int rc = b->eng.init(*config, max_solves);
        if (rc != SH_OK)
        {
            delete b;
            return rc;
        }
        *out = b;
        return SH_OK;
    }

    int sh_batch_destroy(sh_batch *batch)
    {
        delete batch;
        return SH_OK;
    }

    int sh_batch_set_inputs(sh_batch *batch, uint32_t slot, const sh_camera *camera, const sh_measure_maps *measure,
                            const sh_render_maps *render, const sh_geometry *geometry,
                            const sh_node_graph *node_graph, const sh_node_flow *node_flow, const sh_flow_map *flow,
                            const sh_keypoints *keypoints, const float cam2world[16])
    {
        if (!batch)
            return SH_E_ARG;
        return batch->eng.set_inputs(slot, camera, measure, render, geometry, node_graph, node_flow, flow, keypoints,
                                     cam2world);
    }

    int sh_batch_solve(sh_batch *batch, uint32_t num_solves, sh_stream_t stream)
    {
        if (!batch)
            return SH_E_ARG;
        return batch->eng.solve(num_solves, reinterpret_cast<hipStream_t>(stream));
    }

    int sh_batch_node_se3(const sh_batch *batch, uint32_t slot, const sh_dual_quat **view, uint32_t *num_nodes)
    {
        if (!batch || !view || !num_nodes)
            return SH_E_ARG;
        if (slot >= batch->eng.num_slots() || !batch->eng.solved(slot))
            return SH_E_STATE;
        *view = reinterpret_cast<const sh_dual_quat *>(batch->eng.result(slot));
        *num_nodes = uint32_t(batch->eng.desc(slot).N);
        return SH_OK;
    }

    const char *sh_phase_name(uint32_t phase) { return sh::Engine::phase_name(phase); }

    int sh_solver_phase_times(sh_solver *solver, double *ms, uint32_t *calls, uint32_t num_phases, uint32_t reset)
    {
        if (!solver)
            return SH_E_ARG;
        return solver->eng.phase_times(ms, calls, num_phases, reset != 0);
    }

    int sh_batch_phase_times(sh_batch *batch, double *ms, uint32_t *calls, uint32_t num_phases, uint32_t reset)
    {
        if (!batch)
            return SH_E_ARG;
        return batch->eng.phase_times(ms, calls, num_phases, reset != 0);
    }
}
