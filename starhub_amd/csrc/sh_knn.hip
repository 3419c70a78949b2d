// The input producers: surfel skinning and the node graph, both a K nearest
// neighbour search over the nodes (SkinnerKernel, libs/star/geometry/
// node_graph/Skinner.cu:10-94; NodeGraph::BuildNodeGraphFromScratch,
// NodeGraph.cu:10-145,339-365).
//
// The reference scans the nodes in index order into a list of K that replaces
// its largest entry, and sorts the list with a Lomuto quicksort
// (brute_force_knn.cuh:52-135).  Without equal distances the result is simply
// the K nearest in ascending order, however they are found; among equal
// distances the scan decides which node is kept and in which order.  So:
//   k_skin_grid   finds each surfel's K nearest through a uniform grid over
//                 the nodes, and rescans the nodes in index order for the
//                 surfels that meet an equal distance among them;
//   k_skin        the scan alone, for few nodes and for more than the grid's
//                 LDS holds;
//   k_node_graph  the scan (16-bit distances are equal often), one wave per
//                 node, 64 candidates a step.
#include "sh_common.hpp"
#include "sh_kernels.hpp"

namespace sh
{
namespace
{
// fma(dz,dz,fma(dy,dy,dx*dx)) with no further contraction (NodeGraph.cu:32-34);
// the same bits for a - b and b - a
__device__ __forceinline__ float sqdist(float4 a, float4 b)
{
    const float dx = __fsub_rn(a.x, b.x), dy = __fsub_rn(a.y, b.y), dz = __fsub_rn(a.z, b.z);
    return __fmaf_rn(dz, dz, __fmaf_rn(dy, dy, __fmul_rn(dx, dx)));
}

// Entry i of a register array by selects: indexed at run time the array would
// live in scratch memory, and so it does when the compiler sees through the
// selects (the empty asm makes each entry opaque).
template <int K, class T>
__device__ __forceinline__ T pick(const T (&a)[K], int i)
{
    T v = a[0];
    asm("" : "+v"(v));
#pragma unroll
    for (int k = 1; k < K; ++k)
    {
        T e = a[k];
        asm("" : "+v"(e));
        v = i == k ? e : v;
    }
    return v;
}

template <int K, class T>
__device__ __forceinline__ void put(T (&a)[K], int i, T v)
{
#pragma unroll
    for (int k = 0; k < K; ++k)
    {
        T e = a[k];
        asm("" : "+v"(e));
        a[k] = i == k ? v : e;
    }
}

// Ascending Lomuto quicksort, last element the pivot; the partitions are
// disjoint, so the order in which they are sorted does not matter.
template <int K>
__device__ __forceinline__ void lomuto_sort(float (&dist)[K], uint32_t (&idx)[K])
{
    static_assert(K <= 8, "(lo, hi) fit a byte, the pending partitions of two or more entries eight bytes");
    unsigned long long stack = K - 1; // bytes (lo << 4 | hi)
    int top = 1;
    while (top > 0)
    {
        const int lo = int((stack >> 4) & 15u), hi = int(stack & 15u);
        stack >>= 8;
        --top;
        const float pivot = pick(dist, hi);
        auto swap = [&](int a, int b) {
            const float da = pick(dist, a), db = pick(dist, b);
            const uint32_t ia = pick(idx, a), ib = pick(idx, b);
            put(dist, a, db);
            put(dist, b, da);
            put(idx, a, ib);
            put(idx, b, ia);
        };
        int i = lo - 1;
        for (int j = lo; j < hi; ++j)
            if (pick(dist, j) < pivot)
                swap(++i, j);
        swap(++i, hi);
        if (i + 1 < hi)
        {
            stack = (stack << 8) | uint32_t((i + 1) << 4 | hi);
            ++top;
        }
        if (lo < i - 1)
        {
            stack = (stack << 8) | uint32_t(lo << 4 | (i - 1));
            ++top;
        }
    }
}

// The scan's list of K, one per thread: a candidate below the largest entry
// replaces the first such entry.
template <int K>
struct ThreadScan
{
    float dist[K];
    uint32_t idx[K];
    int max_id;
    float max_d;
    __device__ __forceinline__ void init(float d0)
    {
#pragma unroll
        for (int k = 0; k < K; ++k)
        {
            dist[k] = d0;
            idx[k] = 0;
        }
        refresh();
    }
    __device__ __forceinline__ void refresh()
    {
        max_id = 0;
        max_d = dist[0];
#pragma unroll
        for (int k = 1; k < K; ++k)
            if (dist[k] > max_d)
            {
                max_d = dist[k];
                max_id = k;
            }
    }
    __device__ __forceinline__ void update(uint32_t id, float d)
    {
        if (d < max_d)
        {
            put(dist, max_id, d);
            put(idx, max_id, id);
            refresh();
        }
    }
    // Candidates base .. base + n - 1, in order, four at a time: one test of
    // the smallest passes over all four when none is below the largest entry
    // (NaN distances never are).
    __device__ __forceinline__ void scan(uint32_t base, float4 v, const float4 *__restrict__ p, uint32_t n)
    {
        uint32_t i = 0;
        for (; i + 4 <= n; i += 4)
        {
            float d[4];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j)
                d[j] = sqdist(v, p[i + j]);
            if (fminf(fminf(d[0], d[1]), fminf(d[2], d[3])) < max_d)
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j)
                    update(base + i + j, d[j]);
        }
        for (; i < n; ++i)
            update(base + i, sqdist(v, p[i]));
    }
};

// The same list kept by a whole wave for one position: entry k in lane k < K,
// the other lanes hold -1 (below every distance).  64 candidates a step, one
// per lane; those below the largest entry are taken in lane order, each
// against the list as the ones before it left it: the scan's own sequence.
template <int K>
struct WaveScan
{
    static_assert(K <= 8, "the maximum is taken over eight lanes");
    float dist;
    uint32_t idx;
    float max_d; // uniform
    template <int kCtrl>
    static __device__ __forceinline__ float dpp_max(float v)
    {
        const int o = __builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xf, 0xf, true);
        return fmaxf(v, __int_as_float(o));
    }
    __device__ __forceinline__ void refresh()
    {
        float m = dpp_max<0xB1>(dist); // lane ^ 1
        m = dpp_max<0x4E>(m);          // lane ^ 2
        m = dpp_max<0x141>(m);         // the other four of the eight (row_half_mirror)
        max_d = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(m), 0));
    }
    uint32_t lane;
    __device__ __forceinline__ void init(float d0, uint32_t ln)
    {
        lane = ln;
        dist = lane < uint32_t(K) ? d0 : -1.f;
        idx = 0;
        max_d = d0;
    }
    // d: this lane's candidate, node base + lane (not below any entry where there is none)
    __device__ __forceinline__ void step(uint32_t base, float d)
    {
        unsigned long long m = __ballot(d < max_d);
        while (m)
        {
            const int l = __ffsll(m) - 1;
            const float v = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(d), l));
            const uint32_t slot = uint32_t(__ffsll((unsigned long long)__ballot(dist == max_d)) - 1);
            if (lane == slot)
            {
                dist = v;
                idx = base + uint32_t(l);
            }
            refresh();
            m &= __ballot(d < max_d) & (~1ull << l);
        }
    }
    __device__ __forceinline__ void entries(float (&d)[K], uint32_t (&i)[K]) const
    {
#pragma unroll
        for (int k = 0; k < K; ++k)
        {
            d[k] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dist), k));
            i[k] = uint32_t(__builtin_amdgcn_readlane(int(idx), k));
        }
    }
};

// Normalised Gaussian weights of sorted squared distances.
template <int K>
__device__ __forceinline__ void gauss_weights(const float (&dist)[K], float r2, float (&w)[K])
{
    float wsum = 0.f;
#pragma unroll
    for (int k = 0; k < K; ++k)
    {
        w[k] = __expf(-dist[k] / (2.f * r2));
        wsum += w[k];
    }
    const float inv = 1.f / wsum;
#pragma unroll
    for (int k = 0; k < K; ++k)
        w[k] *= inv;
}

// A surfel's K ids and weights; the distances are taken from the nodes again,
// as an entry the scan never filled names node 0.
template <int K>
__device__ __forceinline__ void store_scanned(const float4 *__restrict__ nodes, float4 v, const uint32_t (&idx)[K],
                                              float r2, uint32_t s, uint16_t *__restrict__ knn,
                                              float *__restrict__ spatial, float *__restrict__ connect)
{
    float dist[K], w[K];
#pragma unroll
    for (int k = 0; k < K; ++k)
        dist[k] = sqdist(v, nodes[idx[k]]);
    gauss_weights<K>(dist, r2, w);
#pragma unroll
    for (int k = 0; k < K; ++k)
    {
        knn[size_t(s) * K + k] = uint16_t(idx[k]);
        spatial[size_t(s) * K + k] = w[k];
        connect[size_t(s) * K + k] = 1.f;
    }
}

// Surfel s at v (the same in all lanes) scanned by the wave over the nodes in LDS
template <int K>
__device__ __forceinline__ void scan_by_wave(const float4 *__restrict__ nodes, uint32_t N, float4 v, float r2, uint32_t s,
                                             uint16_t *__restrict__ knn, float *__restrict__ spatial,
                                             float *__restrict__ connect)
{
    const uint32_t lane = __lane_id();
    WaveScan<K> h;
    h.init(1e6f, lane);
    for (uint32_t base = 0; base < N; base += 64)
        h.step(base, base + lane < N ? sqdist(v, nodes[base + lane]) : INFINITY);
    float dist[K];
    uint32_t idx[K];
    h.entries(dist, idx);
    lomuto_sort<K>(dist, idx);
    if (lane == 0)
        store_scanned<K>(nodes, v, idx, r2, s, knn, spatial, connect);
}

// A surfel a lane, of those that are on; the others take nothing
template <int K>
__device__ __forceinline__ void scan_by_lane(const float4 *__restrict__ nodes, uint32_t N, float4 v, uint32_t s, bool on,
                                             float r2, uint16_t *__restrict__ knn, float *__restrict__ spatial,
                                             float *__restrict__ connect)
{
    ThreadScan<K> h;
    h.init(on ? 1e6f : -1.f);
    h.scan(0, v, nodes, N);
    lomuto_sort<K>(h.dist, h.idx);
    if (on)
        store_scanned<K>(nodes, v, h.idx, r2, s, knn, spatial, connect);
}

constexpr uint32_t kSkinTile = 256;

// SkinnerKernel (Skinner.cu:10-94): nodes staged through LDS in tiles.
template <int K>
__global__ __launch_bounds__(kSkinTile) void k_skin(const float4 *__restrict__ surfels, uint32_t S,
                                                    const float4 *__restrict__ nodes, uint32_t N, float r2,
                                                    uint16_t *__restrict__ knn, float *__restrict__ spatial,
                                                    float *__restrict__ connect)
{
    __shared__ float4 tile[kSkinTile];
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    const bool live = s < S;
    const float4 v = live ? surfels[s] : make_float4(0.f, 0.f, 0.f, 0.f);
    ThreadScan<K> h;
    h.init(1e6f);
    for (uint32_t base = 0; base < N; base += kSkinTile)
    {
        __syncthreads();
        if (base + threadIdx.x < N)
            tile[threadIdx.x] = nodes[base + threadIdx.x];
        __syncthreads();
        h.scan(base, v, tile, min(kSkinTile, N - base));
    }
    if (!live)
        return;
    lomuto_sort<K>(h.dist, h.idx);
    store_scanned<K>(nodes, v, h.idx, r2, s, knn, spatial, connect);
}

// ------------------------------------------------------------ skinning through a grid
// Every work-group sorts the nodes into a uniform grid in its own LDS (node
// and id in cell order, cell ends as 16-bit counts) and then takes surfels
// until there are none.  A surfel searches the 3x3x3 cells around its own,
// then one shell of cells more at a time, until its K-th distance lies
// below the distance to every cell not searched.  A cell is about two node
// spacings wide for nodes on a surface, so the first 27 cells, some 40 nodes,
// mostly suffice, against N distances for the scan.  Surfels that need the
// scan (equal distances, far from all nodes) are marked in the output; when
// a work-group has any, it puts the nodes in index order in the grid's place
// and scans them: each wave its own, a surfel a lane, or, when they are few,
// all waves from one list, a surfel a wave (64 candidates a step, but its sort
// and its list's updates serve one surfel).  K = 8, 2% of the nodes there
// twice, so a sixth of the surfels marked: 512 nodes with 20k, 100k and 300k
// surfels 90, 140 and 220 us (each wave its own, a surfel a wave up to 24 of
// them, 236, 277 and 397; a thread per surfel scanning all nodes, one
// candidate after another, 164, 168 and 253).  With every distance equal to
// some other the search comes on top of the scan (512 nodes, 300k surfels: 336
// us, that scan 234).
// The grid takes no memory of the caller's and none is kept between calls:
// building it costs a work-group a few microseconds (N reads from L2), so the
// launch is at most two 1024-thread work-groups a CU.
// K = 8: 1.2M surfels, 4096 nodes 197 us; 300k, 1024 72 us (a thread per surfel
// scanning all nodes, one candidate after another, 2335 and 370 us).
// Few nodes (N K <= 512) are scanned by k_skin, equal distances or not, for
// most need not be tied for the search to cost more; nodes spread evenly, 80
// and 290 surfels a node, scan and grid in us: K = 4, 64 nodes 13 13 and 20 24,
// 128 nodes 22 19 and 24 29, 192 nodes 28 26 and 26 31; K = 8, 64 nodes 22 22
// and 25 29, 96 nodes 29 27 and 30 34, 128 nodes 36 32 and 30 36.
// More than kGridNodes nodes take k_skin too: 64 KB of nodes and 12 KB of cells
// leave room for two work-groups a CU, and a graph of the solver has no more.
constexpr uint32_t kScanEntries = 512;
constexpr uint32_t kGridNodes = 4096;
constexpr uint32_t kGridCells = 6144; // at most, and 3/2 N (a small set's grid is cheap to build)
constexpr uint32_t kGridThreads = 1024;
constexpr uint32_t kGridGroups = 512; // two for each of the 256 CUs
constexpr uint16_t kToScan = 0xffffu; // first id of a surfel that the grid leaves to the scan (no id: N <= 4096)
constexpr uint32_t kFewShare = 16; // N / 16 + 16 marked surfels of a work-group are few: shared by its waves
static_assert((kGridNodes / kFewShare + kFewShare) * 8 <= kGridCells, "their list lies in the cells' words");
constexpr float kFarCells = 2.f;
constexpr int kMaxShells = 6; // at most 13^3 cells, about a third of a full grid's

struct GridShape
{
    float lo[3], h, inv_h;
    int n[3];
};

__device__ __forceinline__ int cell_coord(float u, float inv_h, int n)
{
    // fmaxf(NaN, 0) = 0
    return int(fminf(fmaxf(u * inv_h, 0.f), float(n - 1)));
}

__device__ __forceinline__ int cell_of(const GridShape &g, float4 p)
{
    const int x = cell_coord(p.x - g.lo[0], g.inv_h, g.n[0]), y = cell_coord(p.y - g.lo[1], g.inv_h, g.n[1]),
              z = cell_coord(p.z - g.lo[2], g.inv_h, g.n[2]);
    return (z * g.n[1] + y) * g.n[0] + x;
}

// The grid of a bounding box: cells of about two spacings of N points spread
// over a surface of the box's extent, fewer when that makes more than
// kGridCells, a single cell for a box without a usable extent.
__device__ __forceinline__ GridShape grid_shape(const float (&lo)[3], const float (&hi)[3], uint32_t N, uint32_t max_cells)
{
    GridShape g;
    const float ex = hi[0] - lo[0], ey = hi[1] - lo[1], ez = hi[2] - lo[2];
    const float area = ex * ey + ey * ez + ez * ex, ext = fmaxf(ex, fmaxf(ey, ez));
    float h = fmaxf(2.f * sqrtf(area / float(N)), ext * (1.f / 256.f));
    const bool usable = ext > 0.f && ext < 1e15f && h > 0.f && h < 1e15f && 1.f / h < 1e30f;
    float n[3] = {1.f, 1.f, 1.f};
    if (usable)
        for (;;)
        {
            n[0] = floorf(ex / h) + 1.f;
            n[1] = floorf(ey / h) + 1.f;
            n[2] = floorf(ez / h) + 1.f;
            if (n[0] * n[1] * n[2] <= float(max_cells))
                break;
            h *= 1.05f; // the counts fall to 1 each
        }
    g.h = usable ? h : 1.f;
    g.inv_h = usable ? 1.f / h : 0.f;
#pragma unroll
    for (int c = 0; c < 3; ++c)
    {
        g.lo[c] = lo[c];
        g.n[c] = int(n[c]);
    }
    return g;
}

template <int K>
__global__ __launch_bounds__(kGridThreads, 8) void k_skin_grid(const float4 *__restrict__ surfels, uint32_t S,
                                                  const float4 *__restrict__ nodes, uint32_t N, float r2,
                                                  uint16_t *__restrict__ knn, float *__restrict__ spatial,
                                                  float *__restrict__ connect, int aligned)
{
    constexpr uint32_t NT = kGridThreads;
    extern __shared__ float4 gnode[]; // N nodes in cell order, w = the id's bits
    __shared__ __align__(16) uint32_t cend[kGridCells / 2]; // the ends of the cells, two 16-bit counts a word
    __shared__ float red[NT / 64][6];
    __shared__ uint32_t wsum[NT / 64];
    __shared__ uint32_t n_scan; // surfels left to the scan
    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));

    // ---- bounding box (NaN coordinates leave it as it is)
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t i = tid; i < N; i += NT)
    {
        const float4 p = nodes[i];
        const float c[3] = {p.x, p.y, p.z};
#pragma unroll
        for (int a = 0; a < 3; ++a)
        {
            lo[a] = fminf(lo[a], c[a]);
            hi[a] = fmaxf(hi[a], c[a]);
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
#pragma unroll
        for (int a = 0; a < 3; ++a)
        {
            lo[a] = fminf(lo[a], __shfl_xor(lo[a], o, 64));
            hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], o, 64));
        }
    if (lane == 0)
#pragma unroll
        for (int a = 0; a < 3; ++a)
        {
            red[wave][a] = lo[a];
            red[wave][3 + a] = hi[a];
        }
    const uint32_t max_cells = min(kGridCells, max(64u, (N + N / 2u) & ~1u)), words = max_cells / 2;
    for (uint32_t w = tid; w < words; w += NT)
        cend[w] = 0u;
    if (tid == 0)
        n_scan = 0u;
    __syncthreads();
#pragma unroll
    for (uint32_t w = 0; w < NT / 64; ++w)
#pragma unroll
        for (int a = 0; a < 3; ++a)
        {
            lo[a] = fminf(lo[a], red[w][a]);
            hi[a] = fmaxf(hi[a], red[w][3 + a]);
        }
    // the same in every lane: kept in scalar registers
    GridShape g = grid_shape(lo, hi, N, max_cells);
    auto uniform = [](float v) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v))); };
    g.h = uniform(g.h);
    g.inv_h = uniform(g.inv_h);
#pragma unroll
    for (int a = 0; a < 3; ++a)
    {
        g.lo[a] = uniform(g.lo[a]);
        g.n[a] = __builtin_amdgcn_readfirstlane(g.n[a]);
    }

    // ---- counting sort of the nodes by cell
    for (uint32_t i = tid; i < N; i += NT)
    {
        const int c = cell_of(g, nodes[i]);
        atomicAdd(&cend[c >> 1], 1u << (16 * (c & 1)));
    }
    __syncthreads();
    {
        // exclusive prefix over the cells: a run of words per thread (N <= 4096: no carry into the upper half)
        const uint32_t per = (words + NT - 1) / NT;
        const uint32_t w0 = min(words, tid * per), w1 = min(words, w0 + per);
        uint32_t own = 0;
        for (uint32_t w = w0; w < w1; ++w)
            own += (cend[w] & 0xffffu) + (cend[w] >> 16);
        uint32_t x = own;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1)
        {
            const uint32_t u = __shfl_up(x, o, 64);
            if (int(lane) >= o)
                x += u;
        }
        if (lane == 63)
            wsum[wave] = x;
        __syncthreads();
        uint32_t run = x - own;
#pragma unroll
        for (uint32_t w = 0; w < NT / 64; ++w)
            run += w < wave ? wsum[w] : 0u;
        for (uint32_t w = w0; w < w1; ++w)
        {
            const uint32_t v = cend[w], c0 = v & 0xffffu;
            cend[w] = run | ((run + c0) << 16);
            run += c0 + (v >> 16);
        }
    }
    __syncthreads();
    for (uint32_t i = tid; i < N; i += NT)
    {
        const float4 p = nodes[i];
        const int c = cell_of(g, p);
        const uint32_t at = (atomicAdd(&cend[c >> 1], 1u << (16 * (c & 1))) >> (16 * (c & 1))) & 0xffffu;
        gnode[at] = make_float4(p.x, p.y, p.z, __uint_as_float(i));
    }
    __syncthreads();
    // the cursors now stand at the cells' ends: cell c holds [end(c - 1), end(c))
    auto end_of = [&](int c) -> uint32_t {
        return c < 0 ? 0u : uint32_t(reinterpret_cast<const uint16_t *>(cend)[c]);
    };

    // ---- the surfels, 64 a wave, dealt to the work-groups first and then to
    // their waves, so that what does not fill a round spreads over the CUs;
    // each four waves take their turns rotated by work-group, so that it
    // spreads over a CU's SIMDs too (wave w runs on SIMD w mod 4) and still
    // falls to the first waves, which run ahead
    const uint32_t turn = (wave & ~3u) | ((wave + blockIdx.x + 2u * (blockIdx.x / (kGridGroups / 2))) & 3u);
    const uint32_t chunk0 = turn * gridDim.x + blockIdx.x;
    for (uint32_t chunk = chunk0; chunk < (S + 63u) / 64u; chunk += (NT / 64) * gridDim.x)
    {
        const uint32_t s = chunk * 64u + lane;
        const bool live = s < S;
        const float4 v = surfels[live ? s : S - 1];
        // ascending; `out`: the smallest distance met that is not in the list
        float dist[K];
        uint32_t idx[K];
#pragma unroll
        for (int k = 0; k < K; ++k)
        {
            dist[k] = 1e6f;
            idx[k] = 0;
        }
        float out = INFINITY;
        auto visit = [&](int row, int x0, int x1) {
            const uint32_t e = end_of(row + x1);
            for (uint32_t j = end_of(row + x0 - 1); j < e; ++j)
            {
                const float4 p = gnode[j];
                const float d = sqdist(v, p);
                if (!(d < dist[K - 1]))
                {
                    out = fminf(out, d);
                    continue;
                }
                const uint32_t id = __float_as_uint(p.w);
                out = fminf(out, dist[K - 1]);
                // insertion: entry k takes entry k - 1, d, or stays
#pragma unroll
                for (int k = K - 1; k > 0; --k)
                {
                    const bool below = d < dist[k], under = d < dist[k - 1];
                    idx[k] = under ? idx[k - 1] : (below ? id : idx[k]);
                    dist[k] = under ? dist[k - 1] : (below ? d : dist[k]);
                }
                const bool first = d < dist[0];
                idx[0] = first ? id : idx[0];
                dist[0] = first ? d : dist[0];
            }
        };
        const float u[3] = {v.x - g.lo[0], v.y - g.lo[1], v.z - g.lo[2]};
        // a surfel far from the nodes, by its place or by the shells it would
        // take, is left to the scan, which costs the same anywhere
        int c[3];
        bool far = false;
#pragma unroll
        for (int a = 0; a < 3; ++a)
        {
            c[a] = cell_coord(u[a], g.inv_h, g.n[a]);
            far = far || !(u[a] > -kFarCells * g.h && u[a] < (float(g.n[a]) + kFarCells) * g.h);
        }
        for (int r = 1; !far; ++r)
        {
            const int x0 = max(c[0] - r, 0), x1 = min(c[0] + r, g.n[0] - 1);
            const int y0 = max(c[1] - r, 0), y1 = min(c[1] + r, g.n[1] - 1);
            const int z0 = max(c[2] - r, 0), z1 = min(c[2] + r, g.n[2] - 1);
            for (int z = z0; z <= z1; ++z)
                for (int y = y0; y <= y1; ++y)
                {
                    const int row = (z * g.n[1] + y) * g.n[0];
                    // the first step takes the whole block, a later one its shell
                    if (r == 1 || abs(z - c[2]) == r || abs(y - c[1]) == r)
                        visit(row, x0, x1);
                    else
                    {
                        if (c[0] - r >= 0)
                            visit(row, x0, x0);
                        if (c[0] + r < g.n[0])
                            visit(row, x1, x1);
                    }
                }
            // the distance to the nearest cell not searched, less what the
            // rounding of cell borders and distances can make up
            float bound = INFINITY;
#pragma unroll
            for (int a = 0; a < 3; ++a)
            {
                if (c[a] - r > 0)
                    bound = fminf(bound, u[a] - float(c[a] - r) * g.h);
                if (c[a] + r < g.n[a] - 1)
                    bound = fminf(bound, float(c[a] + r + 1) * g.h - u[a]);
            }
            if (bound == INFINITY)
                break; // every cell is searched
            bound -= 1e-3f * g.h;
            if (bound > 0.f && bound * bound * (1.f - 1e-5f) > dist[K - 1])
                break;
            far = r >= kMaxShells;
        }
        // equal distances in the list or at its end (or a list not full): the scan decides
        bool equal = far || !(out > dist[K - 1]) || !(dist[K - 1] < 1e6f);
#pragma unroll
        for (int k = 1; k < K; ++k)
            equal = equal || dist[k] == dist[k - 1];
        if (live && !equal)
        {
            float w[K];
            gauss_weights<K>(dist, r2, w);
            if (aligned)
            {
                uint32_t pk[K / 2];
#pragma unroll
                for (int k = 0; k < K / 2; ++k)
                    pk[k] = idx[2 * k] | (idx[2 * k + 1] << 16);
                if constexpr (K == 8)
                    reinterpret_cast<uint4 *>(knn)[s] = make_uint4(pk[0], pk[1], pk[2], pk[3]);
                else
                    reinterpret_cast<uint2 *>(knn)[s] = make_uint2(pk[0], pk[1]);
#pragma unroll
                for (int k = 0; k < K / 4; ++k)
                {
                    reinterpret_cast<float4 *>(spatial)[size_t(s) * (K / 4) + k] =
                        make_float4(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
                    reinterpret_cast<float4 *>(connect)[size_t(s) * (K / 4) + k] = make_float4(1.f, 1.f, 1.f, 1.f);
                }
            }
            else
#pragma unroll
                for (int k = 0; k < K; ++k)
                {
                    knn[size_t(s) * K + k] = uint16_t(idx[k]);
                    spatial[size_t(s) * K + k] = w[k];
                    connect[size_t(s) * K + k] = 1.f;
                }
        }
        if (live && equal)
            knn[size_t(s) * K] = kToScan;
        const uint32_t n = uint32_t(__popcll(__ballot(live && equal)));
        if (n && lane == 0)
            atomicAdd(&n_scan, n);
    }
    __syncthreads();
    if (n_scan == 0)
        return;

    // ---- the marked surfels: the nodes in index order in the grid's place
    // (the lane is asked for again, so that no register keeps it till here)
    const uint32_t ln = __lane_id();
    for (uint32_t i = wave * 64u + ln; i < N; i += NT)
        gnode[i] = nodes[i];
    if (wave == 0u && ln == 0u)
        wsum[0] = 0u;
    __syncthreads();
    const uint32_t n = n_scan;
    const bool few = n <= N / kFewShare + kFewShare;
    float4 *__restrict__ list = reinterpret_cast<float4 *>(cend);
    for (uint32_t chunk = chunk0; chunk < (S + 63u) / 64u; chunk += (NT / 64) * gridDim.x)
    {
        const uint32_t s = chunk * 64u + ln;
        const bool to_do = s < S && knn[size_t(s) * K] == kToScan;
        const float4 v = surfels[min(s, S - 1u)];
        if (few)
        {
            if (to_do) // listed in the cells' place
                list[atomicAdd(&wsum[0], 1u)] = make_float4(v.x, v.y, v.z, __uint_as_float(s));
        }
        else if (__any(to_do))
            scan_by_lane<K>(gnode, N, v, s, to_do, r2, knn, spatial, connect);
    }
    if (!few)
        return;
    __syncthreads();
    for (uint32_t i = wave; i < n; i += NT / 64)
        scan_by_wave<K>(gnode, N, list[i], r2, __float_as_uint(list[i].w), knn, spatial, connect);
}

// ------------------------------------------------------------ node graph
constexpr int kGraphThreads = 512; // eight nodes a work-group
constexpr uint32_t kGraphTile = 2048;

// UpdateNodeDistanceKernel + BuildNodeGraphKernel + BuildNodeGraphPairKernel
// + ResetNodeConnectionKernel (NodeGraph.cu:10-145): the FP16 distance of each
// pair is recomputed on the fly instead of being stored as an N x N matrix.
// The compiler makes a distance's last multiply-add and its conversion one
// instruction, which rounds once, straight to 16 bits: where the 32-bit value
// would lie midway between two 16-bit ones, the result may be the other one.
// One wave per node, so that few nodes fill the chip too and a step looks at
// 64 candidates; bound by the step's chain of ballots and list updates (K = 8:
// 4096 nodes 35 us, 256 nodes 15 us; with a thread per node 818 and 112 us).
template <int K>
__global__ __launch_bounds__(kGraphThreads) void k_node_graph(const float4 *__restrict__ nodes, uint32_t N, float r2,
                                                              uint16_t *__restrict__ node_knn,
                                                              float *__restrict__ node_spatial,
                                                              uint16_t *__restrict__ edges,
                                                              float *__restrict__ node_connect)
{
    __shared__ float4 tile[kGraphTile];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t i = blockIdx.x * (kGraphThreads / 64) + (threadIdx.x >> 6);
    const float4 vi = nodes[min(i, N - 1)];
    WaveScan<K> h;
    h.init(1e3f, lane);
    for (uint32_t base = 0; base < N; base += kGraphTile)
    {
        const uint32_t cnt = min(kGraphTile, N - base);
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < cnt; j += kGraphThreads)
            tile[j] = nodes[base + j];
        __syncthreads();
        for (uint32_t j = 0; j < cnt; j += 64)
            h.step(base + j, j + lane < cnt ? __half2float(__float2half_rn(sqdist(vi, tile[j + lane]))) : INFINITY);
    }
    if (i >= N)
        return;
    float dist[K], w[K];
    uint32_t idx[K];
    h.entries(dist, idx);
    lomuto_sort<K>(dist, idx);
    gauss_weights<K>(dist, r2, w);
    if (lane < uint32_t(K))
    {
        const uint32_t id = pick(idx, int(lane));
        const size_t e = size_t(i) * K + lane;
        node_knn[e] = uint16_t(id);
        node_spatial[e] = pick(w, int(lane));
        node_connect[e] = 1.f;
        edges[3 * e] = uint16_t(i);
        edges[3 * e + 1] = uint16_t(id);
        edges[3 * e + 2] = uint16_t(lane);
    }
}

template <int K>
hipError_t start_skin(const float4 *surfels, uint32_t S, const float4 *nodes, uint32_t N, float r2, uint16_t *knn,
                      float *spatial, float *connect, hipStream_t st)
{
    if (N * K <= kScanEntries || N > kGridNodes)
    {
        hipLaunchKernelGGL(k_skin<K>, dim3((S + kSkinTile - 1) / kSkinTile), dim3(kSkinTile), 0, st, surfels, S,
                           nodes, N, r2, knn, spatial, connect);
        return hipGetLastError();
    }
    const size_t lds = size_t(N) * sizeof(float4);
    if (lds > 32768) // with the kernel's own LDS past the default limit of 64 KB
    {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_skin_grid<K>),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 int(kGridNodes * sizeof(float4)));
        if (e != hipSuccess)
            return e;
    }
    const int aligned = ((reinterpret_cast<uintptr_t>(knn) | reinterpret_cast<uintptr_t>(spatial) |
                          reinterpret_cast<uintptr_t>(connect)) &
                         15u) == 0;
    hipLaunchKernelGGL(k_skin_grid<K>, dim3(min(kGridGroups, (S + 63u) / 64u)), dim3(kGridThreads), lds, st, surfels,
                       S, nodes, N, r2, knn, spatial, connect, aligned);
    return hipGetLastError();
}
} // namespace

hipError_t launch_skin(uint32_t K, const float4 *surfels, uint32_t S, const float4 *nodes, uint32_t N, float r2,
                       uint16_t *knn, float *spatial, float *connect, hipStream_t st)
{
    if (S == 0)
        return hipSuccess;
    return K == 8 ? start_skin<8>(surfels, S, nodes, N, r2, knn, spatial, connect, st)
                  : start_skin<4>(surfels, S, nodes, N, r2, knn, spatial, connect, st);
}

hipError_t launch_node_graph(uint32_t K, const float4 *nodes, uint32_t N, float r2, uint16_t *node_knn,
                             float *node_spatial, uint16_t *edges, float *node_connect, hipStream_t st)
{
    const uint32_t per = kGraphThreads / 64;
    if (K == 8)
        hipLaunchKernelGGL(k_node_graph<8>, dim3((N + per - 1) / per), dim3(kGraphThreads), 0, st, nodes, N, r2,
                           node_knn, node_spatial, edges, node_connect);
    else
        hipLaunchKernelGGL(k_node_graph<4>, dim3((N + per - 1) / per), dim3(kGraphThreads), 0, st, nodes, N, r2,
                           node_knn, node_spatial, edges, node_connect);
    return hipGetLastError();
}
} // namespace sh
