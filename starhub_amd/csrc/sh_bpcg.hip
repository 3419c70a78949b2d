// The reference's linear-solver plug-in: BlockPCG<6> over an abstract
// ApplySpMVBase<6> operator (libs/star/pcg_solver/BlockPCG.h:14-115,
// BlockPCG.cuh:16-483, ApplySpMVBase.h:9-47), for callers that bring their
// own system.  The warp solver itself runs its PCG inside the persistent
// kernels of sh_pcg.hip; this is the standalone form with the reference's
// call sequence: SetSolverInput(inv_diag, spmv, b, x) and
// Solve(iterations, zero_init).
//
// With the built-in block-CSR product an iteration is two kernels:
//   k_bp_spmv    delta = t.s of the last update; beta = delta / delta_old;
//                d = s + beta d where a row gathers it; q = A d; partials of d.q
//   k_bp_update  alpha = delta / (d.q); x += alpha d; t = r - alpha q;
//                s = M^-1 t; partial sums of t.s
// With an operator of the caller's (a host callback that enqueues on the
// solve's stream) the product needs d in memory, and it is four: the callback,
// k_bp_dot (partials of d.q), k_bp_update, k_bp_dir (d).  To the same bits up
// to 8192 rows; of more, where the two forms of the product differ, the
// partials of d.q may be of other rows.
// Bound by launches and by the latency of each kernel's dependent loads, not
// by bandwidth: one lane per scalar row of a block, so that loads are
// contiguous over six lanes, five lanes to a scalar row's blocks in the
// product, and all of a lane's loads in flight before partials are summed.
// Work-groups take turns so that there are at most 1024 partials.  256 rows and 10 iterations take 107 us,
// 4096 rows and 20 iterations 214 us (whole calls); with one thread per 6-row
// block and a row's blocks one after another in four kernels 174 and 363 us.
// Every work-group reduces the same partials in the same order, so alpha and
// beta are the same bits everywhere; vectors are FP32 as in the reference,
// the product's row sums, dot products, alpha and beta FP64 (cuBLAS Sdot in the reference,
// BlockPCG.cuh:418-471).  A zero system gives alpha = beta = 0 instead of 0/0.
#include <algorithm>
#include <cmath>
#include <utility>

#include "../../include/sh/warp_solver.h"
#include "sh_common.hpp"
#include "sh_engine.hpp"

#pragma clang fp contract(off)

namespace sh
{
namespace
{
constexpr int kBpThreads = 256;
constexpr int kBpWaveRows = 10;                               // 6-row blocks of a wave: 60 lanes, one scalar row each
constexpr int kBpGroupRows = kBpWaveRows * (kBpThreads / 64); // and of a work-group
// The product: two rows a wave, five blocks of each at a time (a lane holds
// one scalar row of a block), kBpAhead of these in flight.  20 iterations with
// 16 blocks a row, 256 / 4096 / 20000 rows: 211 / 226 / 419 us with two in
// flight, 207 / 233 / 462 with three, 212 / 237 / 504 with four (136
// registers, fewer waves); one lane per scalar row of the system with its
// blocks one after another 240 / 282 us at 256 and 4096 rows; with work-groups
// of 512 and 1024 threads 256 rows take a fifth and two fifths longer.
constexpr int kBpRowBlocks = 5;
constexpr int kBpRowLanes = 6 * kBpRowBlocks;
constexpr int kBpAhead = 2;
constexpr int kBpSpmvThreads = 256;
constexpr int kBpSpmvRows = 2 * (kBpSpmvThreads / 64); // rows of a work-group in one turn
constexpr uint32_t kBpSpmvGroups = 1024;           // more rows than these take turns
// Larger systems: at kBpSharedRows the work-group begins to sum the partials
// together (each wave for itself, a wave's loads are too many), and the row
// kernels take turns past kBpRowGroups (1024 and not 2048: 60000 rows 303 and
// 316 us).  With at most kBpLongBlocks blocks a row the product takes one lane
// per scalar row there, as the row kernels do: the rows fill the chip by
// themselves, and five lanes to one would mostly idle.  From kBpApartBlocks on
// the product is a kernel of its own for the built-in operator too: it gathers
// d alone then, not s and d, and is long against a launch.  Ten iterations, us:
//   rows x blocks   pairs of rows  lane a row  apart
//   10000 x 11      146            134         155
//   16384 x 25      222            260         231
//   32768 x 11      265            222         251
//   60000 x 5       293            196         217
//   60000 x 11      309            299         312
//   60000 x 25      546            586         486
//   150000 x 11     1027           782         660
constexpr uint32_t kBpSharedRows = kBpSpmvRows * kBpSpmvGroups + 1;
constexpr uint32_t kBpRowGroups = 1024;
constexpr uint32_t kBpLongBlocks = 16;
constexpr uint32_t kBpApartBlocks = 1u << 20;

// A lane's scalar row: row 6 * row + a of the system, in the wave's lane 6 * (row of the wave) + a
struct BpLane
{
    uint32_t row, a, i; // clamped to the last row where off
    int first;          // the lane of the block's first row
    bool on;
};

__device__ inline BpLane bp_lane(uint32_t row0, uint32_t nblk)
{
    const uint32_t lane = threadIdx.x % 64u, wave = threadIdx.x / 64u;
    BpLane l;
    l.a = lane % 6u;
    l.first = int(lane - l.a);
    const uint32_t row = row0 + wave * kBpWaveRows + lane / 6u;
    l.on = lane < 6u * kBpWaveRows && row < nblk;
    l.row = min(row, nblk - 1u);
    l.i = 6u * l.row + l.a;
    return l;
}

// f(row0) for each turn of a row kernel's work-group: one where there are no turns
template <bool TURNS, class F>
__device__ inline void bp_turns(uint32_t nblk, F f)
{
    if constexpr (TURNS)
        for (uint32_t row0 = blockIdx.x * kBpGroupRows; row0 < nblk; row0 += gridDim.x * kBpGroupRows)
            f(row0);
    else
        f(blockIdx.x * kBpGroupRows);
}

// This lane's part of the sum of `n` FP64 partials: lane j of a wave takes j,
// j + 64, ...; SHARED: thread j of the work-group takes j, j + 256, ....  Eight
// loads in flight, past the end the last partial again.
template <bool SHARED>
__device__ inline double lane_partials(const double *__restrict__ part, uint32_t n)
{
    constexpr uint32_t kStep = SHARED ? kBpThreads : 64u;
    double v = 0.0;
    for (uint32_t i = threadIdx.x % kStep; i < n; i += 8 * kStep)
    {
        double p[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u)
            p[u] = part[min(i + kStep * u, n - 1u)];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u)
            v = i + kStep * u < n ? v + p[u] : v;
    }
    return v;
}

// The partials' sum from the lanes' parts, in a fixed order: a shuffle tree,
// by every wave for itself, or (SHARED) over the work-group, whose waves' sums
// are added in wave order; the same bits in every wave.  SHARED: all threads
// call it, once a kernel.
template <bool SHARED>
__device__ inline double sum_partials(double lane_sum)
{
    double v = wave_sum(lane_sum);
    if constexpr (SHARED)
    {
        __shared__ double ws[kBpThreads / 64];
        if (threadIdx.x % 64u == 0)
            ws[threadIdx.x / 64u] = v;
        __syncthreads();
        v = ws[0];
#pragma unroll
        for (int w = 1; w < kBpThreads / 64; ++w)
            v += ws[w];
    }
    return v;
}

// Work-group sum of one value per thread, in a fixed order: wave sums, then
// the waves' sums in wave order.  Written by thread 0 to out.
template <int THREADS = kBpThreads>
__device__ inline void block_sum_store(double v, double *__restrict__ out)
{
    __shared__ double ws[THREADS / 64];
    v = wave_sum(v);
    if (threadIdx.x % 64u == 0)
        ws[threadIdx.x / 64u] = v;
    __syncthreads();
    if (threadIdx.x == 0)
    {
        double s = 0.0;
        for (int w = 0; w < THREADS / 64; ++w)
            s += ws[w];
        *out = s;
    }
}

// this lane's row of M^-1 (36 FP32 per block, row-major) and its product with
// v, FP64 accumulation; v: the lane's own entry, the block's others from its lanes
struct BpInvRow
{
    float m[6];
};

__device__ inline BpInvRow load_inv(const float *__restrict__ minv, const BpLane &l)
{
    BpInvRow mi;
#pragma unroll
    for (int j = 0; j < 6; ++j)
        mi.m[j] = minv[6 * size_t(l.i) + j];
    return mi;
}

__device__ inline float precond6(const BpInvRow &mi, float v, const BpLane &l)
{
    double acc = 0.0;
#pragma unroll
    for (int j = 0; j < 6; ++j)
        acc += double(mi.m[j]) * double(__shfl(v, l.first + j, 64));
    return float(acc);
}

// r = b, x = 0 (zero_init) or r given (InitResidual already ran); s = M^-1 r;
// partials of r.s  (blockPCGZeroInitKernel / Initialize, BlockPCG.cuh:395-440)
template <bool SHARED>
__global__ void k_bp_init(const float *__restrict__ b, const float *__restrict__ minv, float *__restrict__ r,
                          float *__restrict__ s, float *__restrict__ x, uint32_t nblk, int zero_init,
                          double *__restrict__ part)
{
    double rs = 0.0;
    bp_turns<SHARED>(nblk, [&](uint32_t row0) __attribute__((always_inline)) {
        const BpLane l = bp_lane(row0, nblk);
        const float rv = zero_init ? b[l.i] : r[l.i];
        const float y = precond6(load_inv(minv, l), rv, l);
        if (l.on)
        {
            if (zero_init)
            {
                r[l.i] = rv;
                x[l.i] = 0.f;
            }
            s[l.i] = y;
        }
        rs += l.on ? double(y) * double(rv) : 0.0;
    });
    block_sum_store(rs, part + blockIdx.x);
}

// delta[it] = sum of the partials (one wave; SHARED: one work-group)
template <bool SHARED>
__global__ void k_bp_delta(const double *__restrict__ part, uint32_t n, double *__restrict__ delta, uint32_t it)
{
    const double s = sum_partials<SHARED>(lane_partials<SHARED>(part, n));
    if (threadIdx.x == 0)
        delta[it] = s;
}

// r = b - y  (InitResidual through ApplySpMV when the operator has no InitResidual)
__global__ void k_bp_sub(const float *__restrict__ b, const float *__restrict__ y, float *__restrict__ r, uint32_t n)
{
    const uint32_t i = blockIdx.x * kBpThreads + threadIdx.x;
    if (i < n)
        r[i] = b[i] - y[i];
}

// A lane's place in the product: row r of the wave's two, blocks j, j + 5, ...
// of it, scalar row a; lead: a lane that holds a scalar row's sum
struct BpRowLane
{
    uint32_t r, j, a;
    bool lead;
};

__device__ inline BpRowLane bp_row_lane()
{
    const uint32_t lane = threadIdx.x % 64u;
    BpRowLane l;
    l.r = min(lane / uint32_t(kBpRowLanes), 1u); // the last four lanes repeat row 1 and sum nothing
    const uint32_t e = lane - l.r * kBpRowLanes;
    l.j = e / 6u;
    l.a = e % 6u;
    l.lead = l.j == 0u;
    return l;
}

// the dot product d.q over the lanes and turns of k_bp_spmv
template <bool LONG>
__global__ void k_bp_dot(const float *__restrict__ d, const float *__restrict__ q, uint32_t nblk,
                         double *__restrict__ part)
{
    constexpr uint32_t kRows = LONG ? kBpGroupRows : kBpSpmvRows;
    double v = 0.0;
    for (uint32_t row0 = blockIdx.x * kRows; row0 < nblk; row0 += gridDim.x * kRows)
    {
        if constexpr (LONG)
        {
            const BpLane l = bp_lane(row0, nblk);
            if (l.on)
                v += double(d[l.i]) * double(q[l.i]);
        }
        else
        {
            const BpRowLane l = bp_row_lane();
            const uint32_t row = row0 + (threadIdx.x / 64u) * 2u + l.r;
            if (l.lead && row < nblk)
                v += double(d[6 * size_t(row) + l.a]) * double(q[6 * size_t(row) + l.a]);
        }
    }
    block_sum_store<kBpSpmvThreads>(v, part + blockIdx.x);
}

// the second kernel of the reference's iteration (BlockPCG.cuh:442-472)
template <bool SHARED>
__global__ void k_bp_update(float *__restrict__ x, const float *__restrict__ r, const float *__restrict__ d,
                            const float *__restrict__ q, const float *__restrict__ minv, float *__restrict__ t,
                            float *__restrict__ s, uint32_t nblk, const double *__restrict__ part_dq,
                            uint32_t n_dq, const double *__restrict__ delta, uint32_t it,
                            double *__restrict__ part_ts)
{
    double ts = 0.0;
    float a = 0.f;
    bool first = true;
    bp_turns<SHARED>(nblk, [&](uint32_t row0) __attribute__((always_inline)) {
        const BpLane l = bp_lane(row0, nblk);
        // everything is loaded before the partials are summed
        const double delta_it = delta[it];
        const float xv = x[l.i], rv = r[l.i], dv = d[l.i], qv = q[l.i];
        const BpInvRow mi = load_inv(minv, l);
        if (first)
        {
            const double dq = sum_partials<SHARED>(lane_partials<SHARED>(part_dq, n_dq));
            a = float(dq != 0.0 ? delta_it / dq : 0.0);
            first = false;
        }
        const float tv = rv - a * qv;
        const float y = precond6(mi, tv, l);
        if (l.on)
        {
            x[l.i] = xv + a * dv;
            t[l.i] = tv;
            s[l.i] = y;
        }
        ts += l.on ? double(y) * double(tv) : 0.0;
    });
    block_sum_store(ts, part_ts + blockIdx.x);
}

// delta' = t.s and beta = delta' / delta of iteration it, from the lanes' sums;
// the first work-group keeps delta' for the update and the history
template <bool SHARED>
__device__ inline float bp_beta(double lane_sum, double *__restrict__ delta, uint32_t it)
{
    const double dold = it ? delta[it - 1] : 0.0;
    const double dn = sum_partials<SHARED>(lane_sum);
    if (blockIdx.x == 0 && threadIdx.x == 0)
        delta[it] = dn;
    return float(dold != 0.0 ? dn / dold : 0.0);
}

// the third kernel (BlockPCG.cuh:474-483): d = s + beta d; delta[it] = t.s (iteration 0: d = s)
template <bool SHARED>
__global__ void k_bp_dir(const float *__restrict__ s, float *__restrict__ d, uint32_t nblk,
                         const double *__restrict__ part_ts, uint32_t n_ts, double *__restrict__ delta, uint32_t it)
{
    float beta = 0.f;
    bool first = true;
    bp_turns<SHARED>(nblk, [&](uint32_t row0) __attribute__((always_inline)) {
        const BpLane l = bp_lane(row0, nblk);
        const float sv = s[l.i], dv = it ? d[l.i] : 0.f;
        if (first)
            beta = bp_beta<SHARED>(lane_partials<SHARED>(part_ts, n_ts), delta, it);
        first = false;
        if (l.on)
            d[l.i] = it ? sv + beta * dv : sv;
    });
}

struct BpVector // a vector in memory
{
    struct Entries
    {
        float x[6];
    };
    const float *__restrict__ x;
    __device__ void load(uint32_t col, Entries &e) const
    {
#pragma unroll
        for (int c = 0; c < 6; ++c)
            e.x[c] = x[6 * size_t(col) + c];
    }
    __device__ float value(const Entries &e, int c) const { return e.x[c]; }
};

struct BpDirection // d = s + beta d_old (iteration 0: s)
{
    struct Entries
    {
        float s[6], d[6];
    };
    const float *__restrict__ s, *__restrict__ d;
    bool old;
    float beta;
    __device__ void load(uint32_t col, Entries &e) const
    {
#pragma unroll
        for (int c = 0; c < 6; ++c)
            e.s[c] = s[6 * size_t(col) + c];
#pragma unroll
        for (int c = 0; c < 6; ++c)
            e.d[c] = d[6 * size_t(col) + c];
    }
    __device__ float value(const Entries &e, int c) const { return old ? e.s[c] + beta * e.d[c] : e.s[c]; }
};

// Scalar row 6 * row + a of A v over a 6x6 block-CSR (row-major blocks;
// performSparseMVKernel, ApplySpMVBinBlockCSR.cuh:13-60), in FP64, rounded
// once; valid in the row's lead lanes.  Five lanes share a scalar row, each
// with kBpAhead blocks in flight, so that a row of up to ten blocks costs one
// trip to memory after its columns; past the row's end the last block is
// loaded again and not summed.  ready() runs in the whole wave when the first
// blocks are in flight.
template <class V, class F>
__device__ inline float bcsr_row(const uint32_t *__restrict__ row_ptr, const uint32_t *__restrict__ col,
                                 const float *__restrict__ blocks, uint32_t row, const BpRowLane &l, V &v, F ready)
{
    const uint32_t k0 = row_ptr[row], k1 = row_ptr[row + 1];
    const uint32_t last = k1 > k0 ? k1 - 1u : 0u; // an empty row loads block 0 (there is one) and sums nothing
    float m[kBpAhead][6];
    typename V::Entries e[kBpAhead];
    auto load = [&](uint32_t k) __attribute__((always_inline)) {
        uint32_t cols[kBpAhead];
#pragma unroll
        for (int u = 0; u < kBpAhead; ++u)
            cols[u] = col[min(k + u * kBpRowBlocks, last)];
#pragma unroll
        for (int u = 0; u < kBpAhead; ++u)
        {
            const float *blk = blocks + 36 * size_t(min(k + u * kBpRowBlocks, last)) + 6 * l.a;
#pragma unroll
            for (int c = 0; c < 6; ++c)
                m[u][c] = blk[c];
        }
#pragma unroll
        for (int u = 0; u < kBpAhead; ++u)
            v.load(cols[u], e[u]);
    };
    double acc = 0.0;
    auto sum = [&](uint32_t k) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kBpAhead; ++u)
        {
            double with = acc;
#pragma unroll
            for (int c = 0; c < 6; ++c)
                with = fma(double(m[u][c]), double(v.value(e[u], c)), with);
            acc = k + u * kBpRowBlocks < k1 ? with : acc;
        }
    };
    uint32_t k = k0 + l.j;
    load(k);
    ready();
    sum(k);
#pragma unroll 1
    for (k += kBpAhead * kBpRowBlocks; k < k1; k += kBpAhead * kBpRowBlocks)
    {
        load(k);
        sum(k);
    }
    // the row's five sums, in the lanes of the first
    const int lane = int(threadIdx.x % 64u);
    const double pair = acc + __shfl(acc, lane + 12, 64);
    const double fifth = __shfl(acc, lane + 24, 64);
    return float(pair + __shfl(pair, lane + 6, 64) + fifth);
}

// The same by one lane, a block after another: for long systems, whose rows
// fill the chip by themselves.  Bound by the blocks' bytes; unrolled, four
// blocks' loads at a time (150000 rows of 11 blocks 43 us, a pair of rows a
// wave 48, one block ahead without the unrolling 46).  The row of m is copied
// before the vector is asked for: otherwise the loads stay one by one (the
// fused product at 32768 rows 279 and not 222 us in ten iterations).
template <class V, class F>
__device__ inline float bcsr_long_row(const uint32_t *__restrict__ row_ptr, const uint32_t *__restrict__ col,
                                      const float *__restrict__ blocks, const BpLane &l, V &v, F ready)
{
    const uint32_t k0 = row_ptr[l.row], k1 = row_ptr[l.row + 1];
    ready();
    double acc = 0.0;
#pragma unroll 4
    for (uint32_t k = k0; k < k1; ++k)
    {
        const float *blk = blocks + 36 * size_t(k) + 6 * l.a;
        float m[6];
#pragma unroll
        for (int c = 0; c < 6; ++c)
            m[c] = blk[c];
        typename V::Entries e;
        v.load(col[k], e);
#pragma unroll
        for (int c = 0; c < 6; ++c)
            acc = fma(double(m[c]), double(v.value(e, c)), acc);
    }
    return float(acc);
}

// y = A x, or y = b - A x (b: InitResidual's r = b - A x)
template <bool LONG>
__global__ __launch_bounds__(kBpSpmvThreads) void k_bcsr_spmv(const uint32_t *__restrict__ row_ptr,
                                                          const uint32_t *__restrict__ col,
                                                          const float *__restrict__ blocks, const float *__restrict__ x,
                                                          const float *__restrict__ b, float *__restrict__ y,
                                                          uint32_t nrows)
{
    const BpVector v{x};
    if constexpr (LONG)
    {
        const BpLane l = bp_lane(blockIdx.x * kBpGroupRows, nrows);
        const float acc = bcsr_long_row(row_ptr, col, blocks, l, v, [] {});
        if (l.on)
            y[l.i] = b ? b[l.i] - acc : acc;
    }
    else
    {
        const BpRowLane l = bp_row_lane();
        const uint32_t row = blockIdx.x * kBpSpmvRows + (threadIdx.x / 64u) * 2u + l.r;
        const size_t i = 6 * size_t(row) + l.a;
        const float acc = bcsr_row(row_ptr, col, blocks, min(row, nrows - 1u), l, v, [] {});
        if (l.lead && row < nrows)
            y[i] = b ? b[i] - acc : acc;
    }
}

// k_bp_dir, k_bcsr_spmv and k_bp_dot in one: the direction is formed where it
// is gathered, from s and the old direction, and each row stores its own part
// of the new one (another buffer: other rows still read the old)
template <bool SHARED, bool LONG>
__global__ __launch_bounds__(kBpSpmvThreads) void k_bp_spmv(const uint32_t *__restrict__ row_ptr,
                                                        const uint32_t *__restrict__ col,
                                                        const float *__restrict__ blocks, const float *__restrict__ s,
                                                        const float *__restrict__ d_old, float *__restrict__ d,
                                                        float *__restrict__ q, uint32_t nblk,
                                                        const double *__restrict__ part_ts, uint32_t n_ts,
                                                        double *__restrict__ delta, uint32_t it,
                                                        double *__restrict__ part_dq)
{
    const double ts = lane_partials<SHARED>(part_ts, n_ts);
    BpDirection v{s, it ? d_old : s, it != 0u, 0.f};
    bool first = true;
    auto ready = [&] {
        if (first)
            v.beta = bp_beta<SHARED>(ts, delta, it);
        first = false;
    };
    double dq = 0.0;
    constexpr uint32_t kRows = LONG ? kBpGroupRows : kBpSpmvRows;
    for (uint32_t row0 = blockIdx.x * kRows; row0 < nblk; row0 += gridDim.x * kRows)
    {
        bool own;
        size_t i;
        float sv, ov, acc;
        if constexpr (LONG)
        {
            const BpLane l = bp_lane(row0, nblk);
            own = l.on;
            i = l.i;
            sv = s[i], ov = v.d[i];
            acc = bcsr_long_row(row_ptr, col, blocks, l, v, ready);
        }
        else
        {
            const BpRowLane l = bp_row_lane();
            const uint32_t row = row0 + (threadIdx.x / 64u) * 2u + l.r;
            own = l.lead && row < nblk;
            i = 6 * size_t(min(row, nblk - 1u)) + l.a;
            sv = s[i], ov = v.d[i];
            acc = bcsr_row(row_ptr, col, blocks, min(row, nblk - 1u), l, v, ready);
        }
        if (own)
        {
            const float dv = it ? sv + v.beta * ov : sv;
            d[i] = dv;
            q[i] = acc;
            dq += double(dv) * double(acc);
        }
    }
    block_sum_store<kBpSpmvThreads>(dq, part_dq + blockIdx.x);
}

__global__ void k_bcsr_check(const uint32_t *__restrict__ row_ptr, const uint32_t *__restrict__ col, uint32_t nrows,
                             uint32_t nnz, uint32_t *__restrict__ bad)
{
    const uint32_t row = blockIdx.x * kBpThreads + threadIdx.x;
    if (row >= nrows)
        return;
    const uint32_t b0 = row_ptr[row], b1 = row_ptr[row + 1];
    if (b0 > b1 || b1 > nnz || (row == nrows - 1 && b1 != nnz) || (row == 0 && b0 != 0))
    {
        *bad = 1u;
        return;
    }
    for (uint32_t k = b0; k < b1; ++k)
        if (col[k] >= nrows)
            *bad = 1u;
}

inline uint32_t grid_of(uint32_t n) { return (n + kBpThreads - 1) / kBpThreads; }
inline uint32_t row_groups(uint32_t nblk) { return (nblk + kBpGroupRows - 1) / kBpGroupRows; }
inline uint32_t row_grid(uint32_t nblk) { return std::min(row_groups(nblk), kBpRowGroups); }
inline uint32_t pair_groups(uint32_t nblk) { return (nblk + kBpSpmvRows - 1) / kBpSpmvRows; } // two rows a wave
inline uint32_t pair_grid(uint32_t nblk) { return std::min(pair_groups(nblk), kBpSpmvGroups); }
inline bool long_rows(uint32_t nblk, uint32_t nnz)
{
    return nblk >= kBpSharedRows && nnz / kBpLongBlocks <= nblk;
}

// y = A x or b - A x
void start_bcsr_spmv(const uint32_t *row_ptr, const uint32_t *col, const float *blocks, const float *x, const float *b,
                     float *y, uint32_t rows, uint32_t nnz, hipStream_t st)
{
    if (long_rows(rows, nnz))
        hipLaunchKernelGGL(k_bcsr_spmv<true>, dim3(row_groups(rows)), dim3(kBpSpmvThreads), 0, st, row_ptr, col, blocks,
                           x, b, y, rows);
    else
        hipLaunchKernelGGL(k_bcsr_spmv<false>, dim3(pair_groups(rows)), dim3(kBpSpmvThreads), 0, st, row_ptr, col, blocks, x, b, y, rows);
}

int status_of(hipError_t e)
{
    if (e == hipSuccess)
        return SH_OK;
    last_hip_error = e;
    return SH_E_HIP;
}
} // namespace
} // namespace sh

struct sh_spmv
{
    uint32_t rows = 0, nnz = 0;
    const uint32_t *row_ptr = nullptr, *col = nullptr;
    const float *blocks = nullptr;
};

struct sh_block_pcg
{
    uint32_t cap = 0; // max_matrix_size
    void *block = nullptr; // one allocation for the vectors and partials
    float *r = nullptr, *t = nullptr, *d = nullptr, *d_old = nullptr, *q = nullptr, *s = nullptr;
    double *part_a = nullptr, *part_b = nullptr, *delta = nullptr;
    uint32_t max_iters = 0;  // delta holds max_iters + 1 entries
    uint32_t last_iters = 0; // iterations the last solve ran
    // SetSolverInput
    const float *inv_diag = nullptr, *b = nullptr;
    float *x = nullptr;
    uint32_t n = 0;
    sh_spmv_ops ops{};
    bool has_input = false;
};

namespace
{
void bpcg_free(sh_block_pcg *p)
{
    if (p->block)
        (void)hipFree(p->block);
    if (p->delta)
        (void)hipFree(p->delta);
    delete p;
}

int ensure_delta(sh_block_pcg *p, uint32_t iters)
{
    if (iters <= p->max_iters && p->delta)
        return SH_OK;
    double *nd = nullptr;
    if (hipMalloc(&nd, size_t(iters + 1) * 8) != hipSuccess)
        return SH_E_NOMEM;
    if (p->delta)
        (void)hipFree(p->delta);
    p->delta = nd;
    p->max_iters = iters;
    return SH_OK;
}
} // namespace

extern "C"
{
    int sh_spmv_create_block_csr(uint32_t num_block_rows, uint32_t num_blocks, const uint32_t *row_ptr,
                                 const uint32_t *block_col, const float *blocks, sh_spmv **out)
    {
        if (!out || num_block_rows == 0 || num_blocks == 0 || !row_ptr || !block_col || !blocks)
            return SH_E_ARG;
        if (uint64_t(num_block_rows) * 6u > 0xffffffffull)
            return SH_E_ARG;
        *out = new sh_spmv{num_block_rows, num_blocks, row_ptr, block_col, blocks};
        return SH_OK;
    }

    int sh_spmv_destroy(sh_spmv *spmv)
    {
        delete spmv;
        return SH_OK;
    }

    int sh_spmv_check(const sh_spmv *spmv, sh_stream_t stream)
    {
        if (!spmv)
            return SH_E_ARG;
        uint32_t *bad = nullptr;
        if (hipMalloc(&bad, 4) != hipSuccess)
            return SH_E_NOMEM;
        const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
        uint32_t h = 0;
        int rc = sh::status_of(hipMemsetAsync(bad, 0, 4, st));
        if (rc == SH_OK)
        {
            hipLaunchKernelGGL(sh::k_bcsr_check, dim3(sh::grid_of(spmv->rows)), dim3(sh::kBpThreads), 0, st,
                               spmv->row_ptr, spmv->col, spmv->rows, spmv->nnz, bad);
            rc = sh::status_of(hipGetLastError());
        }
        if (rc == SH_OK)
            rc = sh::status_of(hipMemcpyAsync(&h, bad, 4, hipMemcpyDeviceToHost, st));
        if (rc == SH_OK)
            rc = sh::status_of(hipStreamSynchronize(st));
        (void)hipFree(bad);
        if (rc != SH_OK)
            return rc;
        return h ? SH_E_ARG : SH_OK;
    }

    int sh_spmv_matrix_size(const sh_spmv *spmv, uint32_t *size)
    {
        if (!spmv || !size)
            return SH_E_ARG;
        *size = 6u * spmv->rows;
        return SH_OK;
    }

    int sh_spmv_apply(sh_spmv *spmv, const float *x, float *y, sh_stream_t stream)
    {
        if (!spmv || !x || !y)
            return SH_E_ARG;
        sh::start_bcsr_spmv(spmv->row_ptr, spmv->col, spmv->blocks, x, nullptr, y, spmv->rows, spmv->nnz,
                            reinterpret_cast<hipStream_t>(stream));
        return sh::status_of(hipGetLastError());
    }

    int sh_spmv_init_residual(sh_spmv *spmv, const float *x_init, const float *b, float *residual,
                              sh_stream_t stream)
    {
        if (!spmv || !x_init || !b || !residual)
            return SH_E_ARG;
        sh::start_bcsr_spmv(spmv->row_ptr, spmv->col, spmv->blocks, x_init, b, residual, spmv->rows, spmv->nnz,
                            reinterpret_cast<hipStream_t>(stream));
        return sh::status_of(hipGetLastError());
    }

    static int bcsr_apply_cb(void *user, const float *x, float *y, sh_stream_t stream)
    {
        return sh_spmv_apply(static_cast<sh_spmv *>(user), x, y, stream);
    }

    static int bcsr_init_cb(void *user, const float *x, const float *b, float *r, sh_stream_t stream)
    {
        return sh_spmv_init_residual(static_cast<sh_spmv *>(user), x, b, r, stream);
    }

    int sh_spmv_ops_of(sh_spmv *spmv, sh_spmv_ops *ops)
    {
        if (!spmv || !ops)
            return SH_E_ARG;
        ops->user = spmv;
        ops->matrix_size = 6u * spmv->rows;
        ops->apply_spmv = bcsr_apply_cb;
        ops->init_residual = bcsr_init_cb;
        return SH_OK;
    }

    int sh_block_pcg_create(uint32_t max_matrix_size, sh_block_pcg **out)
    {
        if (!out || max_matrix_size == 0 || max_matrix_size % 6u != 0)
            return SH_E_ARG;
        sh_block_pcg *p = new sh_block_pcg();
        p->cap = max_matrix_size;
        const size_t vb = (size_t(max_matrix_size) * 4 + 255) / 256 * 256; // a vector's stride
        const size_t na = std::max(sh::pair_grid(max_matrix_size / 6u), sh::row_grid(max_matrix_size / 6u)), nb = sh::row_grid(max_matrix_size / 6u);
        const bool ok = hipMalloc(&p->block, 6 * vb + (na + nb) * 8) == hipSuccess && ensure_delta(p, 16) == SH_OK;
        float **const vec[6] = {&p->r, &p->t, &p->d, &p->d_old, &p->q, &p->s};
        for (int i = 0; ok && i < 6; ++i)
            *vec[i] = reinterpret_cast<float *>(static_cast<char *>(p->block) + i * vb);
        p->part_a = ok ? reinterpret_cast<double *>(static_cast<char *>(p->block) + 6 * vb) : nullptr;
        p->part_b = ok ? p->part_a + na : nullptr;
        if (!ok)
        {
            bpcg_free(p);
            return SH_E_NOMEM;
        }
        *out = p;
        return SH_OK;
    }

    int sh_block_pcg_destroy(sh_block_pcg *pcg)
    {
        if (pcg)
            bpcg_free(pcg);
        return SH_OK;
    }

    int sh_block_pcg_set_input(sh_block_pcg *pcg, const float *inv_diag_blocks, const sh_spmv_ops *spmv,
                               const float *b, float *x, uint32_t actual_size)
    {
        if (!pcg || !inv_diag_blocks || !spmv || !spmv->apply_spmv || !b || !x)
            return SH_E_ARG;
        const uint32_t n = actual_size ? actual_size : spmv->matrix_size;
        if (n == 0 || n % 6u != 0 || spmv->matrix_size != n)
            return SH_E_ARG;
        if (n > pcg->cap)
            return SH_E_CAPACITY;
        pcg->inv_diag = inv_diag_blocks;
        pcg->ops = *spmv;
        pcg->b = b;
        pcg->x = x;
        pcg->n = n;
        pcg->has_input = true;
        return SH_OK;
    }

    // Solve / SolveNoConvergeCheck and SolveConvergeChecked (BlockPCG.cuh:325-393):
    // epsilon > 0 stops after the first iteration with
    // |delta| < epsilon^2 |delta_0| (one host readback per iteration, as there)
    static int bpcg_run(sh_block_pcg *pcg, uint32_t max_iterations, int zero_init, float epsilon,
                        sh_stream_t stream, uint32_t *iterations)
    {
        if (!pcg)
            return SH_E_ARG;
        if (!pcg->has_input)
            return SH_E_STATE;
        int rc = ensure_delta(pcg, max_iterations);
        if (rc != SH_OK)
            return rc;
        const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
        const uint32_t nblk = pcg->n / 6u, g = sh::row_grid(nblk);
        pcg->last_iters = 0;
        if (!zero_init)
        {
            // r = b - A x_init (ApplySpMVBase::InitResidual), or through ApplySpMV
            if (pcg->ops.init_residual)
                rc = pcg->ops.init_residual(pcg->ops.user, pcg->x, pcg->b, pcg->r, stream);
            else if ((rc = pcg->ops.apply_spmv(pcg->ops.user, pcg->x, pcg->q, stream)) == SH_OK)
            {
                hipLaunchKernelGGL(sh::k_bp_sub, dim3(sh::grid_of(pcg->n)), dim3(sh::kBpThreads), 0, st, pcg->b,
                                   pcg->q, pcg->r, pcg->n);
                rc = sh::status_of(hipGetLastError());
            }
            if (rc != SH_OK)
                return rc;
        }
        // s = M^-1 r and the partials of r.s; each iteration begins with their sum
        const bool shared = nblk >= sh::kBpSharedRows;
        hipLaunchKernelGGL(shared ? sh::k_bp_init<true> : sh::k_bp_init<false>, dim3(g), dim3(sh::kBpThreads), 0, st,
                           pcg->b, pcg->inv_diag, pcg->r, pcg->s, pcg->x, nblk, zero_init ? 1 : 0, pcg->part_b);
        // the sum by itself, where the host or the history needs it and no iteration follows
        auto store_delta = [&](uint32_t it) {
            hipLaunchKernelGGL(shared ? sh::k_bp_delta<true> : sh::k_bp_delta<false>, dim3(1),
                               dim3(shared ? sh::kBpThreads : 64), 0, st, pcg->part_b, g, pcg->delta, it);
        };
        if (epsilon > 0.f || max_iterations == 0)
            store_delta(0);
        if ((rc = sh::status_of(hipGetLastError())) != SH_OK)
            return rc;
        double delta0 = 0.0;
        if (epsilon > 0.f &&
            (rc = sh::status_of(hipMemcpyAsync(&delta0, pcg->delta, 8, hipMemcpyDeviceToHost, st))) != SH_OK)
            return rc;
        // the built-in product takes the direction and the dot product into its
        // kernel; any other operator needs the direction in memory
        const sh_spmv *own = pcg->ops.apply_spmv == bcsr_apply_cb ? static_cast<const sh_spmv *>(pcg->ops.user) : nullptr;
        if (own && (own->rows != nblk || own->nnz >= sh::kBpApartBlocks))
            own = nullptr;
        const bool by_lane = own ? sh::long_rows(nblk, own->nnz) : shared; // the lanes that hold d.q's terms
        const uint32_t gq = by_lane ? g : sh::pair_grid(nblk);
        float *r = pcg->r, *t = pcg->t, *d = pcg->d, *d_old = pcg->d_old;
        for (uint32_t it = 0; it < max_iterations; ++it)
        {
            if (own)
            {
                auto spmv = [&](auto kernel) {
                    hipLaunchKernelGGL(kernel, dim3(gq), dim3(sh::kBpSpmvThreads), 0, st, own->row_ptr, own->col,
                                       own->blocks, pcg->s, d_old, d, pcg->q, nblk, pcg->part_b, g, pcg->delta, it,
                                       pcg->part_a);
                };
                if (by_lane)
                    spmv(sh::k_bp_spmv<true, true>);
                else if (shared)
                    spmv(sh::k_bp_spmv<true, false>);
                else
                    spmv(sh::k_bp_spmv<false, false>);
            }
            else
            {
                hipLaunchKernelGGL(shared ? sh::k_bp_dir<true> : sh::k_bp_dir<false>, dim3(g), dim3(sh::kBpThreads), 0,
                                   st, pcg->s, d, nblk, pcg->part_b, g, pcg->delta, it);
                if ((rc = sh::status_of(hipGetLastError())) != SH_OK ||
                    (rc = pcg->ops.apply_spmv(pcg->ops.user, d, pcg->q, stream)) != SH_OK)
                    return rc;
                hipLaunchKernelGGL(by_lane ? sh::k_bp_dot<true> : sh::k_bp_dot<false>, dim3(gq),
                                   dim3(sh::kBpSpmvThreads), 0, st, d, pcg->q, nblk, pcg->part_a);
            }
            hipLaunchKernelGGL(shared ? sh::k_bp_update<true> : sh::k_bp_update<false>, dim3(g), dim3(sh::kBpThreads), 0,
                               st, pcg->x, r, d, pcg->q, pcg->inv_diag, t, pcg->s, nblk, pcg->part_a, gq, pcg->delta,
                               it, pcg->part_b);
            if (epsilon > 0.f || it + 1 == max_iterations)
                store_delta(it + 1);
            if ((rc = sh::status_of(hipGetLastError())) != SH_OK)
                return rc;
            std::swap(r, t);
            if (own)
                std::swap(d, d_old);
            pcg->last_iters = it + 1;
            if (epsilon > 0.f)
            {
                double delta = 0.0;
                if ((rc = sh::status_of(hipMemcpyAsync(&delta, pcg->delta + it + 1, 8, hipMemcpyDeviceToHost, st))) !=
                        SH_OK ||
                    (rc = sh::status_of(hipStreamSynchronize(st))) != SH_OK)
                    return rc;
                if (std::fabs(delta) < double(epsilon) * double(epsilon) * std::fabs(delta0))
                    break;
            }
        }
        if (iterations)
            *iterations = pcg->last_iters;
        return sh::status_of(hipStreamSynchronize(st));
    }

    int sh_block_pcg_solve(sh_block_pcg *pcg, uint32_t max_iterations, int zero_init, sh_stream_t stream)
    {
        return bpcg_run(pcg, max_iterations, zero_init, 0.f, stream, nullptr);
    }

    int sh_block_pcg_solve_converge_checked(sh_block_pcg *pcg, uint32_t max_iterations, int zero_init,
                                            float epsilon, sh_stream_t stream, uint32_t *iterations)
    {
        if (!(epsilon > 0.f))
            return SH_E_ARG;
        return bpcg_run(pcg, max_iterations, zero_init, epsilon, stream, iterations);
    }

    int sh_block_pcg_delta_history(const sh_block_pcg *pcg, double *out, uint32_t capacity, uint32_t *count)
    {
        if (!pcg || !count)
            return SH_E_ARG;
        if (!pcg->has_input)
            return SH_E_STATE;
        *count = pcg->last_iters + 1;
        if (!out)
            return SH_OK;
        const uint32_t n = std::min(capacity, pcg->last_iters + 1);
        return sh::status_of(hipMemcpy(out, pcg->delta, size_t(n) * 8, hipMemcpyDeviceToHost));
    }
}
