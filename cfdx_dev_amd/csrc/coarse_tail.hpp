// The coarse end of an FP64 V-cycle in one launch.
//
// Below a few thousand rows a V-cycle is a chain of launches that each take
// 4 to 5 us whatever they do: the launch itself and the dependent loads of row
// offsets, entries and x. One workgroup runs every level from the first small
// one down to the coarsest and back up instead. The vectors of those levels
// live in LDS, the matrix in hand in registers over all sweeps of a smoothing
// pass, and a phase (a sweep, a residual, a transfer) costs one barrier. On a
// 12^3 box (1727 + 406 + 57 + 14 rows, 6 + 6 sweeps) the cycle takes 76 us
// (under the kernel trace) against 45 launches of 4.5 us.
//
// Matrix layout: a row of at most 64 entries belongs to one lane and takes
// batches of eight slots there; a lane holds at most 8 batches in registers
// (8 waves of 256 VGPRs). Rows go to the lanes longest first, so the lanes of
// a wavefront have like counts. Longer rows (the coarse levels of filtered
// aggregation have a few rows that span the level) are streamed in groups, a
// wavefront each: their products go through LDS, then a lane a row adds them
// in order. That chain of additions bounds a sweep on such a level (about
// 5 ns an entry whether LDS, lane reads or DPP feed it; 2.4 ns from registers).
//
// Forms that lost (12^3 box): every product staged in LDS as the CSR-stream
// kernel does, 163 us; the matrix streamed from L2 in every phase, 144 us (one
// CU draws about 60 GB/s); one code path for all phases so that it stays in
// the instruction cache, 325 us (the held matrix spills). FP32 cycles smooth
// these levels once, so nothing is held, and the launches are as fast.
//
// The arithmetic is that of the per-launch kernels: rows are summed in storage
// order by one lane, the epilogues evaluate the same expressions. A padding
// slot multiplies -0.0 with a cell of the vector that holds 1.0, and adding
// -0.0 changes no sum.
#pragma once

#include "device_amg.hpp"
#include "kernels.hpp"

namespace cfdxhip {

constexpr int kTailThreads = kTailWaves * 64;
constexpr uint32_t kTailBatches = 8;
constexpr uint32_t kTailMaxLevels = 12;
constexpr uint32_t kTailLaneRow = 8 * kTailBatches;  // longest row one lane holds
constexpr uint32_t kTailChunk = 1024;                // products of longer rows a wavefront stages at a time
constexpr uint32_t kTailMaxRows = 8191;              // columns are 16-bit

// Control word of a lane's batch: the row, whether it starts and ends here.
constexpr uint32_t kTailStart = 1u << 16, kTailEnd = 1u << 17;

struct TailLu {
    uint32_t n;  // order of the coarsest factors, 0: the last level is smoothed
    const uint32_t* piv;
    const double* factor;
    const double* upper;
};

template <bool kCheb>
__global__ __launch_bounds__(kTailThreads) void coarse_tail_kernel(const TailLevel* __restrict__ lv, uint32_t nl,
                                                                   uint32_t cells, uint32_t stage, double omega,
                                                                   uint32_t pre, uint32_t post, uint32_t last_sweeps,
                                                                   TailLu lu, const double* __restrict__ b_in,
                                                                   double* __restrict__ x_out) {
#pragma clang fp contract(off)
    constexpr int kB = kTailBatches;
    // Per level x and b at lv[l].x and lv[l].b; behind them, each of the
    // first level's size: y, the other x of a sweep; the inverse diagonal;
    // the Chebyshev direction. Then the wavefronts' staging for long rows.
    extern __shared__ __align__(16) double lds[];
    const uint32_t n0 = lv[0].A.n + 1;
    double* const y = lds + cells;
    double* const inv = y + n0;
    double* const dir = inv + n0;
    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63u;
    double* const staged = lds + stage + wave * kTailChunk;

    // The matrix in hand.
    uint32_t ctl[kB];
    uint4 ec[kB];
    double ev[kB][8];
    uint32_t nb = 0;
    auto take = [&](const TailMat& M) __attribute__((always_inline)) {
        nb = __builtin_amdgcn_readfirstlane(M.count[wave]);
        const size_t at = size_t(__builtin_amdgcn_readfirstlane(M.first[wave])) * 64 + lane;
        const double2* vq = reinterpret_cast<const double2*>(M.vals) + (at - lane) * 4 + lane;
#pragma unroll
        for (int k = 0; k < kB; ++k)
            if (uint32_t(k) < nb) {
                ctl[k] = M.ctl[at + size_t(k) * 64];
                ec[k] = M.cols[at + size_t(k) * 64];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const double2 v = vq[size_t(k) * 256 + q * 64];
                    ev[k][2 * q] = v.x;
                    ev[k][2 * q + 1] = v.y;
                }
            }
    };
    // done(row, init(row) + (M v)[row]) for every row; M is in hand.
    auto apply = [&](const TailMat& M, const double* v, auto init, auto done) __attribute__((always_inline)) {
        for (uint32_t i = wave; i < M.ngroups; i += kTailWaves) {
            const uint4 m = M.groups[i];
            const uint32_t off = __builtin_amdgcn_readfirstlane(m.x), len = __builtin_amdgcn_readfirstlane(m.y),
                           rows = __builtin_amdgcn_readfirstlane(m.w);
            const uint4 mine = M.lrows[__builtin_amdgcn_readfirstlane(m.z) + min(lane, rows - 1)];
            double s = init(mine.x);
            for (uint32_t base = 0; base < len; base += kTailChunk) {
                const uint32_t here = min(len - base, kTailChunk);
                constexpr uint32_t kU = 8;
                for (uint32_t k0 = 0; k0 < here; k0 += kU * 64) {
                    uint32_t c[kU];
                    double w[kU];
#pragma unroll
                    for (uint32_t u = 0; u < kU; ++u) {
                        const uint32_t k = min(k0 + u * 64 + lane, here - 1);
                        c[u] = M.lcols[off + base + k];
                        w[u] = M.lvals[off + base + k];
                    }
#pragma unroll
                    for (uint32_t u = 0; u < kU; ++u) {
                        const uint32_t k = k0 + u * 64 + lane;
                        const double p = w[u] * v[c[u]];
                        if (k < here) staged[k] = p;
                    }
                }
                wave_fence();
                // A group of several rows is one chunk; a row alone may take more.
                // (Groups of 16 operands in flight would spill the matrix.)
                if (rows > 1) {
                    if (lane < rows) s = ordered_sum<false>(staged, mine.y, mine.z, s);
                } else if (lane == 0) {
                    s = ordered_sum<false>(staged, 0u, here, s);
                }
                wave_fence();
            }
            if (lane < rows) done(mine.x, s);
        }
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < kB; ++k)
            if (uint32_t(k) < nb) {
                const uint32_t row = ctl[k] & 0xffffu;
                const uint32_t cw[4] = {ec[k].x, ec[k].y, ec[k].z, ec[k].w};
                double xv[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) xv[j] = v[j & 1 ? cw[j / 2] >> 16 : cw[j / 2] & 0xffffu];
                if (ctl[k] & kTailStart) s = init(row);
#pragma unroll
                for (int j = 0; j < 8; ++j) s += ev[k][j] * xv[j];
                if (ctl[k] & kTailEnd) done(row, s);
            }
        __syncthreads();
    };
    auto zero = [](uint32_t) { return 0.0; };
    // Sweeps first..last-1 of a smoothing pass from the vector x; returns the
    // one that holds the result (x or the other one, o).
    auto sweeps = [&](const TailLevel& L, bool ch, uint32_t first, uint32_t last, double* x, double* o)
        __attribute__((always_inline)) {
        const double* b = lds + L.b;
        for (uint32_t k = first; k < last; ++k) {
            const double c1 = ch && k > 0 ? L.c1[k] : 0.0, c2 = ch ? L.c2[k] : omega;
            apply(L.A, x, zero, [&](uint32_t row, double s) {
                const double delta = inv[row] * (b[row] - s);
                if (ch) {
                    const double dn = k == 0 ? c2 * delta : c1 * dir[row] + c2 * delta;
                    dir[row] = dn;
                    o[row] = x[row] + dn;
                } else {
                    o[row] = x[row] + c2 * delta;
                }
            });
            double* t = x;
            x = o;
            o = t;
        }
        return x;
    };
    // Smoothing from x = 0 (the first sweep is a scaling), the result in x.
    auto from_zero = [&](const TailLevel& L, bool ch, uint32_t count) __attribute__((always_inline)) {
        const uint32_t n = L.A.n;
        double* x = lds + L.x;
        double* z = count && (count - 1) % 2 ? y : x;
        const double c = ch ? L.c2[0] : omega;
        for (uint32_t i = tid; i < n; i += kTailThreads) {
            const double iv = L.inv[i];
            inv[i] = iv;
            const double v = count ? c * (iv * lds[L.b + i]) : 0.0;
            z[i] = v;
            if (kCheb) dir[i] = v;
        }
        if (tid == 0) x[n] = y[n] = 1.0;
        __syncthreads();
        sweeps(L, ch, 1, count, z, z == x ? y : x);
    };

    // Each thread reads back in from_zero the b cells it writes here.
    for (uint32_t i = tid; i < n0 - 1; i += kTailThreads) lds[lv[0].b + i] = b_in[i];
    for (uint32_t l = 0; l + 1 < nl; ++l) {
        const TailLevel& L = lv[l];
        take(L.A);
        from_zero(L, kCheb, kCheb ? L.degree : pre);
        const double* b = lds + L.b;
        apply(L.A, lds + L.x, zero, [&](uint32_t row, double s) { y[row] = b[row] - s; });
        take(L.R);
        double* bc = lds + lv[l + 1].b;
        apply(L.R, y, zero, [&](uint32_t row, double s) { bc[row] = s; });
    }
    {
        const TailLevel& L = lv[nl - 1];
        if (lu.n) {
            if (tid < 64)
                coarse_lu_solve<double>(lu.n, L.A.n, lu.piv, lu.factor, lu.upper, lds + L.b, lds + L.x, lds + stage);
            if (tid == 0) lds[L.x + L.A.n] = 1.0;
            __syncthreads();
        } else {
            take(L.A);
            from_zero(L, false, last_sweeps);
        }
    }
    double* x = lds + lv[nl - 1].x;
    for (uint32_t l = nl - 1; l-- > 0;) {
        const TailLevel& L = lv[l];
        const uint32_t n = L.A.n;
        double* xl = lds + L.x;
        take(L.P);
        for (uint32_t i = tid; i < n; i += kTailThreads) inv[i] = L.inv[i];
        if (tid == 0) y[n] = 1.0;
        apply(L.P, lds + lv[l + 1].x, [&](uint32_t row) { return xl[row]; },
              [&](uint32_t row, double s) { xl[row] = s; });
        take(L.A);
        x = sweeps(L, kCheb, 0, kCheb ? L.degree : post, xl, y);
        if (l > 0 && x != xl) {
            for (uint32_t i = tid; i < n; i += kTailThreads) xl[i] = x[i];
            __syncthreads();
        }
    }
    for (uint32_t i = tid; i < n0 - 1; i += kTailThreads) x_out[i] = x[i];
}

// vals[i] = src[i] of a matrix's stored values (kTailPad: a padding slot).
constexpr uint32_t kTailPad = 0xFFFFFFFFu;
static __global__ __launch_bounds__(kBlock) void tail_values_kernel(uint32_t n, const uint32_t* __restrict__ src,
                                                                    const double* __restrict__ v,
                                                                    double* __restrict__ out) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) out[i] = src[i] == kTailPad ? -0.0 : v[src[i]];
}

}  // namespace cfdxhip
