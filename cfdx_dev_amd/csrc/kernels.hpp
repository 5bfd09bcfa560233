// Device kernels for the sparse solve (included by .hip translation units).
//
// CSR-stream SpMV: one 256-thread workgroup per row block. Phase 1 streams
// the block's values and column indices with unit stride (coalesced) and
// stages val * x[col] in LDS; phase 2 gives each row to one thread, which sums
// its products sequentially in storage order. The per-row order matches the
// reference's scalar CSR loop (sparse_matrix.h:182-197), so FP64 results are
// bit-identical to it. Epilogue functors fuse the Jacobi update, residual,
// prolongation and dot-product partials into the same pass.
//
// Workgroups are dispatched round-robin over the 8 XCDs; xcd_block() gives
// every XCD one contiguous range of row blocks so each XCD's L2 sees a
// contiguous window of x.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace cfdxhip {

constexpr int kBlock = 256;
// Products a CSR-stream row block stages in LDS: FP64 blocks hold twice as
// many entries (32 KiB), so a block of ~28-entry coarse rows keeps about 150
// of its 256 threads summing a row (measured: the FP64 sweep on the first
// coarse level of the 16.8M-cell box 495 -> 383 us); FP32 keeps 2048, which
// leaves the small coarse levels more workgroups.
template <class T>
struct StreamNnz {
    static constexpr int value = 4096;
};
template <>
struct StreamNnz<float> {
    static constexpr int value = 2048;
};
constexpr int kMaxRowsPerBlock = 1024;
constexpr int kXcds = 8;

__device__ __forceinline__ uint32_t xcd_block(uint32_t bid, uint32_t nb) {
    const uint32_t xcd = bid % kXcds, local = bid / kXcds;
    const uint32_t per = nb / kXcds, extra = nb % kXcds;
    return xcd * per + (xcd < extra ? xcd : extra) + local;
}

// ---------------------------------------------------------------- reduce --

// Deterministic wavefront sum (fixed butterfly order).
template <class T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Orders a wavefront's LDS accesses (no barrier with other wavefronts).
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Lane `src`'s value (src uniform).
__device__ __forceinline__ double lane_value(double v, int src) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), src),
                            __builtin_amdgcn_readlane(__double2loint(v), src));
}

// Block sum for 256 threads: wave sums, then a fixed-order sum of 4 waves.
template <class T>
__device__ __forceinline__ T block_sum(T v, T* smem4) {
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) smem4[wid] = v;
    __syncthreads();
    T r = T(0);
    if (threadIdx.x == 0) r = ((smem4[0] + smem4[1]) + smem4[2]) + smem4[3];
    __syncthreads();
    return r;
}

// Sums `count` partial arrays (each of length n, stride `stride`) into
// out[j], one workgroup an array (of up to 63 in a Gram-Schmidt step, where one
// workgroup for all took 7.9 us on average), in a fixed order: deterministic.
// mirror: pinned host memory that receives the sums as well, so that a host
// that waits for them needs no copy.
// The write to the host costs a launch about 1.5 us, so only sums that are
// waited for ask for it.
__device__ __forceinline__ double sum_partials(const double* __restrict__ p, uint32_t n, double* sm /* 16 */) {
    double v = 0.0;
    for (uint32_t i = threadIdx.x; i < n; i += 1024) v += p[i];
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) sm[wid] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < 16; ++w) s += sm[w];
    return s;
}

static __global__ __launch_bounds__(1024) void reduce_partials_kernel(const double* __restrict__ partials,
                                                               uint32_t n, uint32_t stride,
                                                               double* __restrict__ out,
                                                               double* __restrict__ mirror) {
    __shared__ double sm[16];
    const uint32_t j = blockIdx.x;
    const double s = sum_partials(partials + size_t(j) * stride, n, sm);
    if (threadIdx.x != 0) return;
    out[j] = s;
    if (mirror) mirror[j] = s;
}

// Tells a host that polls `done` (pinned) that this workgroup's writes to pinned
// memory, all made by the calling thread, have arrived.
__device__ __forceinline__ void signal_host(unsigned long long* done, unsigned long long ticket) {
    __threadfence_system();
    __hip_atomic_store(done, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// The sums that end a PCG iteration, of three arrays of their own lengths, in one
// launch: out[j] = sum of p[j]; mirror receives them and, in front of them, the
// scalar that precedes out. done[j]: see signal_host.
struct PartialList {
    const double* p[3];
    uint32_t n[3];
};
static __global__ __launch_bounds__(1024) void reduce_list_kernel(PartialList list, double* __restrict__ out,
                                                                 double* __restrict__ mirror,
                                                                 unsigned long long* __restrict__ done,
                                                                 unsigned long long ticket) {
    __shared__ double sm[16];
    const uint32_t j = blockIdx.x;
    const double s = sum_partials(list.p[j], list.n[j], sm);
    if (threadIdx.x != 0) return;
    out[j] = mirror[j] = s;
    if (j == 0) mirror[-1] = out[-1];
    signal_host(done + j, ticket);
}

// The sum that ends a Gram-Schmidt step, with the step's `count` products (src)
// for the host as well: mirror[0..count) and *sum_mirror.
static __global__ __launch_bounds__(1024) void reduce_step_kernel(const double* __restrict__ partials, uint32_t n,
                                                                 double* __restrict__ out,
                                                                 double* __restrict__ sum_mirror, uint32_t count,
                                                                 const double* __restrict__ src,
                                                                 double* __restrict__ mirror,
                                                                 unsigned long long* __restrict__ done,
                                                                 unsigned long long ticket) {
    __shared__ double sm[16];
    for (uint32_t k = threadIdx.x; k < count; k += 1024) mirror[k] = src[k];
    __threadfence_system();
    const double s = sum_partials(partials, n, sm);  // a barrier between the copies and the signal
    if (threadIdx.x != 0) return;
    *out = *sum_mirror = s;
    signal_host(done, ticket);
}

// ------------------------------------------------------------------ SpMV --

// s + p[b] + p[b+1] + ... + p[e-1], added strictly left to right. The sum of
// a long row is a chain of dependent additions, so kG LDS reads are always in
// flight ahead of the additions that use the previous ones. One wavefront
// draws FP64 operands from LDS at 13.6 clocks an addition with groups of 8,
// 11.6 with groups of 16 (5.8 from registers).
template <int kG, class T>
__device__ __forceinline__ T chain_sum(const T* p, uint32_t& k, uint32_t e, T s) {
#pragma clang fp contract(off)
    T v[kG], w[kG];
#pragma unroll
    for (int j = 0; j < kG; ++j) v[j] = p[k + j];
    k += kG;
    for (; k + 2 * kG <= e; k += 2 * kG) {
#pragma unroll
        for (int j = 0; j < kG; ++j) w[j] = p[k + j];
#pragma unroll
        for (int j = 0; j < kG; ++j) s += v[j];
#pragma unroll
        for (int j = 0; j < kG; ++j) v[j] = p[k + kG + j];
#pragma unroll
        for (int j = 0; j < kG; ++j) s += w[j];
    }
#pragma unroll
    for (int j = 0; j < kG; ++j) s += v[j];
    return s;
}
template <bool kWide = true, class T>
__device__ __forceinline__ T ordered_sum(const T* p, uint32_t b, uint32_t e, T s) {
#pragma clang fp contract(off)
    uint32_t k = b;
    if (kWide && sizeof(T) == 8 && k + 128 <= e) s = chain_sum<16>(p, k, e, s);
    if (k + 8 <= e) s = chain_sum<8>(p, k, e, s);
    for (; k + 4 <= e; k += 4) {
        T v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = p[k + j];
#pragma unroll
        for (int j = 0; j < 4; ++j) s += v[j];
    }
    for (; k < e; ++k) s += p[k];
    return s;
}

// FP64 sums keep the reference's per-row order (bit-exact results); FP32
// sums of long rows are split across lanes.
template <class T>
struct OrderedSum {
    static constexpr bool value = true;
};
template <>
struct OrderedSum<float> {
    static constexpr bool value = false;
};
#ifndef CFDX_GROUP_LANES
#define CFDX_GROUP_LANES 16
#endif
constexpr uint32_t kGroupRowNnz = 12;                // FP32: lanes per row above this mean row length
constexpr uint32_t kGroupLanes = CFDX_GROUP_LANES;   // power of two, at most 64

// FP32 rows of a block that one lane (16 lanes in a block of long rows) would
// sum for longer than the whole wavefront: the coarse levels mix rows of a few
// entries with rows that span the level, and such a row summed by one lane
// kept a launch of seven workgroups waiting 12 us (4.5 us so).
constexpr uint32_t kWaveRowNnz = 24;
constexpr uint32_t kGroupRowMax = 128;

// Sums of the rows [b, e) of the lanes with `mine`, one row after the other
// by the whole wavefront (strided partial sums, fixed butterfly): each such
// lane receives its row's sum. Collective over the wavefront.
template <class T>
__device__ __forceinline__ T wave_row_sums(const T* p, uint32_t b, uint32_t e, bool mine) {
    const uint32_t lane = threadIdx.x & 63u;
    T out = T(0);
    for (uint64_t m = __ballot(mine); m; m &= m - 1) {
        const int src = __builtin_ctzll(m);
        const uint32_t rb = __shfl(b, src, 64), re = __shfl(e, src, 64);
        T s = T(0);
        for (uint32_t k = rb + lane; k < re; k += 64) s += p[k];
        s = wave_sum(s);
        if (int(lane) == src) out = s;
    }
    return out;
}

// The rows of one row block [lo, hi) (row, first entry), summed by the
// workgroup and handed to the epilogue; returns this thread's partial.
template <class T, class Init, class Epi, int kStreamNnz = StreamNnz<T>::value>
__device__ __forceinline__ double stream_rows(uint2 lo, uint2 hi, const uint32_t* __restrict__ rowp,
                                              const uint32_t* __restrict__ cols, const T* __restrict__ vals,
                                              const T* __restrict__ x, const Init& init, const Epi& epi) {
#pragma clang fp contract(off)
    constexpr bool kOrdered = OrderedSum<T>::value;
    __shared__ T prod[kStreamNnz];
    const uint32_t r0 = lo.x, r1 = hi.x, k0 = lo.y, k1 = hi.y;
    double part = 0.0;
    if (k1 - k0 <= uint32_t(kStreamNnz)) {
        // The epilogue inputs of this thread's first row (its offsets, the
        // initial value and the epilogue's vectors) are loaded before the
        // matrix stream, so their latency hides behind it.
        const uint32_t row1 = r0 + threadIdx.x;
        typename Epi::Pre pre{};
        T ini = T(0);
        uint32_t rb = 0, re = 0;
        if (row1 < r1) {
            rb = rowp[row1];
            re = rowp[row1 + 1];
            pre = epi.load(row1);
            ini = init(row1);
        }
        // All of this thread's matrix loads are issued before the dependent
        // gathers of x; values and columns are read once, so they bypass the
        // caches (non-temporal) and leave L2/MALL to x.
        // The gathers are unconditional (out-of-range slots read x[0]) so
        // that all of them are in flight together; a predicated gather
        // would wait for each load before issuing the next.
        constexpr int kPer = kStreamNnz / kBlock;
        uint32_t ci[kPer];
        T vi[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const uint32_t k = k0 + threadIdx.x + uint32_t(j) * kBlock;
            ci[j] = 0;
            vi[j] = T(0);
            if (k < k1) {
                ci[j] = __builtin_nontemporal_load(cols + k);
                vi[j] = __builtin_nontemporal_load(vals + k);
            }
        }
        T xv[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j) xv[j] = x[ci[j]];
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const uint32_t k = k0 + threadIdx.x + uint32_t(j) * kBlock;
            if (k < k1) prod[k - k0] = vi[j] * xv[j];
        }
        __syncthreads();
        bool grouped = false;
        if constexpr (!kOrdered) grouped = (k1 - k0) >= kGroupRowNnz * (r1 - r0);
        if (!grouped) {
            // Loop bounds uniform in a wavefront (wave_row_sums is collective).
            for (uint32_t row = row1; row - (threadIdx.x & 63u) < r1; row += kBlock) {
                const bool live = row < r1;
                if (row != row1) {
                    rb = live ? rowp[row] : 0u;
                    re = live ? rowp[row + 1] : 0u;
                    if (live) {
                        pre = epi.load(row);
                        ini = init(row);
                    }
                }
                T s;
                if constexpr (kOrdered) {
                    s = live ? ordered_sum(prod, rb - k0, re - k0, ini) : ini;
                } else {
                    const bool longer = live && re - rb > kWaveRowNnz;
                    s = live && !longer ? ordered_sum(prod, rb - k0, re - k0, ini) : ini;
                    const T t = wave_row_sums(prod, rb - k0, re - k0, longer);
                    if (longer) s = ini + t;
                }
                if (live) part += epi.apply(row, s, pre);
            }
        } else {
            if constexpr (!kOrdered) {
                // Long rows (FP32 only, no ordering contract): kGroupLanes
                // lanes per row, strided partial sums combined by a shuffle
                // tree, row sums staged in LDS; then one thread per row
                // applies the epilogue, so the epilogue's loads are issued
                // once, together.
                __shared__ T rsum[kMaxRowsPerBlock];
                const uint32_t g = threadIdx.x / kGroupLanes, lane = threadIdx.x % kGroupLanes;
                for (uint32_t row0 = r0; row0 < r1; row0 += kBlock / kGroupLanes) {
                    const uint32_t row = row0 + g;
                    T s = T(0);
                    if (row < r1 && rowp[row + 1] - rowp[row] <= kGroupRowMax)
                        for (uint32_t k = rowp[row] - k0 + lane; k < rowp[row + 1] - k0; k += kGroupLanes)
                            s += prod[k];
#pragma unroll
                    for (int off = int(kGroupLanes) / 2; off > 0; off >>= 1) s += __shfl_xor(s, off, kGroupLanes);
                    if (row < r1 && lane == 0) rsum[row - r0] = s;
                }
                __syncthreads();
                for (uint32_t row = row1; row - (threadIdx.x & 63u) < r1; row += kBlock) {
                    const bool live = row < r1;
                    if (row != row1) {
                        rb = live ? rowp[row] : 0u;
                        re = live ? rowp[row + 1] : 0u;
                        if (live) {
                            pre = epi.load(row);
                            ini = init(row);
                        }
                    }
                    const bool longer = live && re - rb > kGroupRowMax;
                    const T t = wave_row_sums(prod, rb - k0, re - k0, longer);
                    if (live) part += epi.apply(row, ini + (longer ? t : rsum[row - r0]), pre);
                }
            }
        }
    } else if (kOrdered) {
        // One long row: streamed in chunks, a single thread keeps the
        // sequential sum while the other wavefronts fill the next chunk.
        constexpr uint32_t kHalf = uint32_t(kStreamNnz) / 2;
        T s = init(r0);
        auto fill = [&](uint32_t base, T* dst, uint32_t first, uint32_t step) {
            const uint32_t len = min(k1 - base, kHalf);
            for (uint32_t k = first; k < len; k += 4 * step) {
                T v[4];
                uint32_t c[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const uint32_t kk = k + uint32_t(u) * step;
                    c[u] = kk < len ? cols[base + kk] : 0u;
                    v[u] = kk < len ? vals[base + kk] : T(0);
                }
                T xv[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) xv[u] = x[c[u]];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (k + uint32_t(u) * step < len) dst[k + uint32_t(u) * step] = v[u] * xv[u];
            }
        };
        fill(k0, prod, threadIdx.x, kBlock);
        __syncthreads();
        uint32_t h = 0;
        for (uint32_t base = k0; base < k1; base += kHalf, h ^= 1u) {
            if (threadIdx.x >= 64) {
                if (base + kHalf < k1) fill(base + kHalf, prod + (h ^ 1u) * kHalf, threadIdx.x - 64, kBlock - 64);
            } else if (threadIdx.x == 0) {
                s = ordered_sum(prod + h * kHalf, 0u, min(k1 - base, kHalf), s);
            }
            __syncthreads();
        }
        if (threadIdx.x == 0) part = epi(r0, s);
    } else {
        // One long row, FP32: per-thread strided sums, then a block tree. Eight
        // products per thread are loaded before they are added, so their
        // gathers are in flight together.
        __shared__ T tred[kBlock / 64];
        T s = T(0);
        for (uint32_t k = k0 + threadIdx.x; k < k1; k += 8 * kBlock) {
            T v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const uint32_t kk = k + uint32_t(u) * kBlock;
                v[u] = kk < k1 ? vals[kk] * x[cols[kk]] : T(0);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) s += v[u];
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
        if ((threadIdx.x & 63) == 0) tred[threadIdx.x >> 6] = s;
        __syncthreads();
        if (threadIdx.x == 0) part = epi(r0, init(r0) + (((tred[0] + tred[1]) + tred[2]) + tred[3]));
    }
    return part;
}

template <class T, class Init, class Epi>
__global__ __launch_bounds__(kBlock) void spmv_stream_kernel(const uint2* __restrict__ blocks, uint32_t nb,
                                                             const uint32_t* __restrict__ rowp,
                                                             const uint32_t* __restrict__ cols,
                                                             const T* __restrict__ vals, const T* __restrict__ x,
                                                             Init init, Epi epi) {
    const uint32_t b = xcd_block(blockIdx.x, nb);
    const double part = stream_rows<T>(blocks[b], blocks[b + 1], rowp, cols, vals, x, init, epi);
    if (Epi::kPartial) {
        __shared__ double red[4];
        const double bs = block_sum(part, red);
        if (threadIdx.x == 0) epi.store_partial(blockIdx.x, bs);
    }
}

// ------------------------------------------------------------- SELL-64 --
//
// Sliced ELL: rows in slices of 64 (one wavefront, one row per lane); inside
// a slice the q-th entry of every row is stored together, so entry (slice, q,
// lane) sits at soff[slice] + q * 64 + lane, and a lane adds its slots in
// order. Rows shorter than the slice's width end in padding slots (column
// kSellPad, value 0) that the sum skips. Every load of values and columns is
// a unit-stride 256 B (FP32) or 512 B (FP64) wavefront access.
// FP64 copies keep each row's CSR entry order in its slots, so rows are
// summed exactly as the CSR-stream kernel sums them (bit-identical results).
// FP32 copies sort each row's slots by column: then the gathers of slot q are
// the q-th neighbours of 64 consecutive rows, which in a bandwidth-reducing
// ordering lie close together (few cache lines per gather).
constexpr uint32_t kSellRows = 64;
constexpr uint32_t kSellPad = 0xFFFFFFFFu;
constexpr int kSellUnroll = 8;  // slots in flight per lane

template <class T, class Init, class Epi>
__global__ __launch_bounds__(kBlock) void spmv_sell_kernel(uint32_t n, uint32_t ns, uint32_t nblk,
                                                           const uint32_t* __restrict__ soff,
                                                           const uint32_t* __restrict__ cols,
                                                           const T* __restrict__ vals, const T* __restrict__ x,
                                                           Init init, Epi epi) {
#pragma clang fp contract(off)
    __shared__ double red[4];
    const uint32_t b = xcd_block(blockIdx.x, nblk);
    const uint32_t slice = b * (kBlock / kSellRows) + threadIdx.x / kSellRows;
    const uint32_t lane = threadIdx.x % kSellRows;
    const uint32_t row = slice * kSellRows + lane;
    double part = 0.0;
    if (slice < ns) {
        typename Epi::Pre pre{};
        T s = T(0);
        if (row < n) {
            pre = epi.load(row);
            s = init(row);
        }
        const uint32_t e = soff[slice + 1];
        for (uint32_t k = soff[slice] + lane; k < e; k += kSellRows * kSellUnroll) {
            uint32_t c[kSellUnroll];
            T v[kSellUnroll];
#pragma unroll
            for (int j = 0; j < kSellUnroll; ++j) {
                const uint32_t kk = k + uint32_t(j) * kSellRows;
                c[j] = kSellPad;
                v[j] = T(0);
                if (kk < e) {
                    c[j] = __builtin_nontemporal_load(cols + kk);
                    v[j] = __builtin_nontemporal_load(vals + kk);
                }
            }
            // Unconditional gathers (padding reads x[0]) keep all of them in
            // flight together; the select leaves s untouched on padding.
            T xv[kSellUnroll];
#pragma unroll
            for (int j = 0; j < kSellUnroll; ++j) xv[j] = x[c[j] == kSellPad ? 0u : c[j]];
#pragma unroll
            for (int j = 0; j < kSellUnroll; ++j) s = c[j] == kSellPad ? s : s + v[j] * xv[j];
        }
        if (row < n) part = epi.apply(row, s, pre);
    }
    if (Epi::kPartial) {
        const double bs = block_sum(part, red);
        if (threadIdx.x == 0) epi.store_partial(blockIdx.x, bs);
    }
}

// Half-precision smoothing copy of a column-sorted FP32 SELL matrix: the
// values of D^-1 A (each row divided by its diagonal, so the diagonal is 1
// and M-matrix off-diagonals lie in [-1, 0]) rounded to FP16, 2 B per slot
// and no padding beyond the SELL slots: a slice of width w whose slots start
// at k0 = soff[slice] owns the 32-bit words k0/2 .. k0/2 + 32w - 1. Word
// k0/2 + p * 64 + lane (p < w/2) holds slot 2p of the lane's row in its low
// half and slot 2p + 1 in its high half; when w is odd, the last slot of
// lanes l and l + 32 shares word k0/2 + (w/2) * 64 + l (low half lane l).
// In 16-bit units slot (q, lane) sits at half_slot(k0, w, q, lane). Sums and
// epilogues run in FP32.
__host__ __device__ __forceinline__ uint32_t half_slot(uint32_t k0, uint32_t w, uint32_t q, uint32_t lane) {
    return (q | 1u) < w ? k0 + (q & ~1u) * kSellRows + 2 * lane + (q & 1u)
                        : k0 + q * kSellRows + ((lane & 31u) << 1 | lane >> 5);
}
__device__ __forceinline__ uint32_t f32_to_f16_bits(float v) {
    return uint32_t(__builtin_bit_cast(uint16_t, static_cast<_Float16>(v)));
}
__device__ __forceinline__ float f16_bits_to_f32(uint32_t h) {
    return static_cast<float>(__builtin_bit_cast(_Float16, uint16_t(h)));
}

// Compact columns of the half copy. In a slice whose slot rows each span at
// most 65533 columns, hbase[soff[slice] / 64 + q] is the middle of slot q's
// column range and hcol16, laid out like hvals, holds each slot's offset from
// its base as int16, -32768 marking padding; the bases are wave-uniform scalar
// loads, so a slot costs 2 B of column and 2 B of value. Slices flagged in
// hwide keep the 4 B columns of the FP32 copy.
constexpr int32_t kHalfPadOff = -32768;
template <class Init, class Epi>
__global__ __launch_bounds__(kBlock) void spmv_sell_half_compact_kernel(
    uint32_t n, uint32_t ns, uint32_t nblk, const uint32_t* __restrict__ soff, const uint8_t* __restrict__ hwide,
    const uint32_t* __restrict__ hbase, const uint32_t* __restrict__ hcol16, const uint32_t* __restrict__ cols, const uint32_t* __restrict__ hvals, const float* __restrict__ x, Init init,
    Epi epi) {
#pragma clang fp contract(off)
    static_assert(kSellUnroll % 2 == 0, "slot pairs");
    static_assert(!Epi::kPartial, "no block partials on the half copy");
    const uint32_t b = xcd_block(blockIdx.x, nblk);
    const uint32_t slice = b * (kBlock / kSellRows) + threadIdx.x / kSellRows;
    const uint32_t lane = threadIdx.x % kSellRows;
    const uint32_t row = slice * kSellRows + lane;
    if (slice >= ns) return;
    typename Epi::Pre pre{};
    float s = 0.0f;
    if (row < n) {
        pre = epi.load(row);
        s = init(row);
    }
    const uint32_t k0 = __builtin_amdgcn_readfirstlane(soff[slice]);
    const uint32_t w_slots = (__builtin_amdgcn_readfirstlane(soff[slice + 1]) - k0) / kSellRows;
    const uint32_t h0 = k0 / 2;  // word offset of the slice's slot pairs
    const bool wide = __builtin_amdgcn_readfirstlane(uint32_t(hwide[slice])) != 0u;
    const uint32_t* base = hbase + k0 / kSellRows;
    // A slice's odd last slot (two rows per word: lane l's in the low half,
    // lane l + 32's in the high half) is read as the last pair's low half, so
    // its loads and gather go out with the rest of the row's.
    const uint32_t tail_q = (w_slots & 1u) ? w_slots - 1 : ~0u;
    const uint32_t tail_word = h0 + (w_slots / 2) * kSellRows + (lane & 31u);
    const uint32_t tail_shift = (lane >> 5) * 16u;
    for (uint32_t q = 0; q < w_slots; q += kSellUnroll) {
        uint32_t vw[kSellUnroll / 2];
        uint32_t c[kSellUnroll];
        bool pad[kSellUnroll];
        if (wide) {
#pragma unroll
            for (int j = 0; j < kSellUnroll; ++j) {
                const bool ok = q + uint32_t(j) < w_slots;
                const uint32_t cc = ok ? __builtin_nontemporal_load(cols + k0 + (q + j) * kSellRows + lane) : kSellPad;
                pad[j] = cc == kSellPad;
                c[j] = pad[j] ? 0u : cc;
            }
        } else {
            uint32_t dw[kSellUnroll / 2];
#pragma unroll
            for (int p = 0; p < kSellUnroll / 2; ++p) {
                const uint32_t qp = q + 2 * uint32_t(p);
                const bool tl = qp == tail_q;
                const uint32_t wi = tl ? tail_word : h0 + (q / 2 + uint32_t(p)) * kSellRows + lane;
                const uint32_t d = qp < w_slots ? __builtin_nontemporal_load(hcol16 + wi) : 0x80008000u;
                dw[p] = tl ? (((d >> tail_shift) & 0xffffu) | 0x80000000u) : d;
            }
#pragma unroll
            for (int j = 0; j < kSellUnroll; ++j) {
                const int32_t off = int32_t(int16_t((j & 1) ? (dw[j / 2] >> 16) : (dw[j / 2] & 0xffffu)));
                pad[j] = off == kHalfPadOff;
                const uint32_t bq = q + uint32_t(j) < w_slots ? base[q + j] : 0u;
                c[j] = pad[j] ? 0u : uint32_t(int32_t(bq) + off);
            }
        }
#pragma unroll
        for (int p = 0; p < kSellUnroll / 2; ++p) {
            const uint32_t qp = q + 2 * uint32_t(p);
            const bool tl = qp == tail_q;
            const uint32_t wi = tl ? tail_word : h0 + (q / 2 + uint32_t(p)) * kSellRows + lane;
            const uint32_t v = qp < w_slots ? __builtin_nontemporal_load(hvals + wi) : 0u;
            vw[p] = tl ? ((v >> tail_shift) & 0xffffu) : v;
        }
        float xv[kSellUnroll];
#pragma unroll
        for (int j = 0; j < kSellUnroll; ++j) xv[j] = x[c[j]];
#pragma unroll
        for (int j = 0; j < kSellUnroll; ++j) {
            const float v = f16_bits_to_f32((j & 1) ? (vw[j / 2] >> 16) : (vw[j / 2] & 0xffffu));
            s = pad[j] ? s : s + v * xv[j];
        }
    }
    if (row < n) epi.apply(row, s, pre);
}

// Bases of the compact columns: thread per (slice, slot) row of 64 lanes,
// the middle of its non-padding columns' range (0 when all are padding).
static __global__ __launch_bounds__(kBlock) void sell_half_base_kernel(uint64_t slots64,
                                                                      const uint32_t* __restrict__ scols,
                                                                      uint32_t* __restrict__ hbase) {
    const uint64_t t = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (t >= slots64) return;
    uint32_t lo = 0xffffffffu, hi = 0;
    for (uint32_t l = 0; l < kSellRows; ++l) {
        const uint32_t c = scols[t * kSellRows + l];
        if (c == kSellPad) continue;
        lo = c < lo ? c : lo;
        hi = c > hi ? c : hi;
    }
    hbase[t] = lo > hi ? 0u : lo + (hi - lo) / 2;
}

// Offsets of the compact columns, one thread per lane of every slice (the
// padding rows of the last slice included: their slots are padding, so every
// half word the kernel reads is written); a slice with an offset outside
// int16 is flagged wide (every writer stores 1).
static __global__ __launch_bounds__(kBlock) void sell_half_cols_kernel(uint32_t rows, const uint32_t* __restrict__ soff,
                                                                      const uint32_t* __restrict__ scols,
                                                                      const uint32_t* __restrict__ hbase,
                                                                      uint32_t* __restrict__ hcol16,
                                                                      uint8_t* __restrict__ hwide) {
    const uint32_t r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= rows) return;
    const uint32_t slice = r / kSellRows, lane = r % kSellRows;
    const uint32_t k0 = soff[slice], w = (soff[slice + 1] - k0) / kSellRows;
    bool fits = true;
    auto off_of = [&](uint32_t q) -> uint32_t {
        const uint32_t c = scols[k0 + q * kSellRows + lane];
        if (c == kSellPad) return 0x8000u;
        const int64_t d = int64_t(c) - int64_t(hbase[k0 / kSellRows + q]);
        if (d < -32767 || d > 32767) {
            fits = false;
            return 0x8000u;
        }
        return uint32_t(uint16_t(int16_t(d)));
    };
    for (uint32_t p = 0; 2 * p + 1 < w; ++p)
        hcol16[k0 / 2 + p * kSellRows + lane] = off_of(2 * p) | (off_of(2 * p + 1) << 16);
    if (w & 1u) reinterpret_cast<uint16_t*>(hcol16)[half_slot(k0, w, w - 1, lane)] = uint16_t(off_of(w - 1));
    if (!fits) hwide[slice] = 1;
}

// Fills the half copy from the FP32 SELL values and the FP32 inverse
// diagonal, one thread per lane of every slice (padding rows, r >= n, get
// zero halves).
static __global__ __launch_bounds__(kBlock) void sell_half_values_kernel(uint32_t n, uint32_t rows,
                                                                  const uint32_t* __restrict__ soff,
                                                                  const float* __restrict__ s32,
                                                                  const float* __restrict__ inv_diag,
                                                                  uint32_t* __restrict__ hvals) {
#pragma clang fp contract(off)
    const uint32_t r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= rows) return;
    const uint32_t slice = r / kSellRows, lane = r % kSellRows;
    const uint32_t k0 = soff[slice], w = (soff[slice + 1] - k0) / kSellRows;
    const bool live = r < n;
    const float inv = live ? inv_diag[r] : 0.0f;
    auto half_of = [&](uint32_t q) -> uint32_t {
        return live ? f32_to_f16_bits(s32[k0 + q * kSellRows + lane] * inv) : 0u;
    };
    for (uint32_t p = 0; 2 * p + 1 < w; ++p)
        hvals[k0 / 2 + p * kSellRows + lane] = half_of(2 * p) | (half_of(2 * p + 1) << 16);
    if (w & 1u) reinterpret_cast<uint16_t*>(hvals)[half_slot(k0, w, w - 1, lane)] = uint16_t(half_of(w - 1));
}

// Column-sorted SELL: entry k of row r goes to the slot of its rank among
// the row's columns (ascending), so slot q of 64 consecutive rows points the
// same way for every row and the gathers of one slot stay close together.
// Changes the summation order: FP32 copies only.
template <class T>
__global__ __launch_bounds__(kBlock) void sell_scatter_sorted_kernel(uint32_t n, const uint32_t* __restrict__ rowp,
                                                                     const uint32_t* __restrict__ cols,
                                                                     const uint32_t* __restrict__ soff,
                                                                     const T* __restrict__ src, T* __restrict__ dst) {
    const uint32_t r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= n) return;
    const uint32_t base = soff[r / kSellRows] + r % kSellRows;
    const uint32_t b = rowp[r], e = rowp[r + 1];
    for (uint32_t k = b; k < e; ++k) {
        const uint32_t c = cols[k];
        uint32_t rank = 0;
        for (uint32_t k2 = b; k2 < e; ++k2) rank += (cols[k2] < c || (cols[k2] == c && k2 < k)) ? 1u : 0u;
        dst[base + rank * kSellRows] = src[k];
    }
}

// CSR entry k of row r (k-th of the row: q = k - rowp[r]) -> SELL slot
// soff[r / 64] + q * 64 + r % 64.
template <class T>
__global__ __launch_bounds__(kBlock) void sell_scatter_kernel(uint32_t n, const uint32_t* __restrict__ rowp,
                                                              const uint32_t* __restrict__ soff,
                                                              const T* __restrict__ src, T* __restrict__ dst) {
    const uint32_t r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= n) return;
    const uint32_t base = soff[r / kSellRows] + r % kSellRows;
    const uint32_t b = rowp[r], e = rowp[r + 1];
    for (uint32_t k = b; k < e; ++k) dst[base + (k - b) * kSellRows] = src[k];
}

template <class T>
struct InitZero {
    __device__ T operator()(uint32_t) const { return T(0); }
};
template <class T>
struct InitFrom {
    const T* v;
    __device__ T operator()(uint32_t row) const { return v[row]; }
};

// Epilogue functors: load(row) fetches the row's inputs (issued early by
// the kernel), apply(row, s, pre) finishes the row from its sum s.
struct NoPre {};

// y = A x
template <class T>
struct EpiStore {
    static constexpr bool kPartial = false;
    using Pre = NoPre;
    T* y;
    __device__ Pre load(uint32_t) const { return {}; }
    __device__ double apply(uint32_t row, T s, const Pre&) const {
        y[row] = s;
        return 0.0;
    }
    __device__ double operator()(uint32_t row, T s) const { return apply(row, s, load(row)); }
    __device__ void store_partial(uint32_t, double) const {}
};

// y = A x, partial += w[row] * y[row]   (p^T A p)
template <class T>
struct EpiStoreDot {
    static constexpr bool kPartial = true;
    struct Pre {
        T w;
    };
    T* y;
    const T* w;
    double* partial;
    __device__ Pre load(uint32_t row) const { return {w[row]}; }
    __device__ double apply(uint32_t row, T s, const Pre& p) const {
        y[row] = s;
        return double(p.w) * double(s);
    }
    __device__ double operator()(uint32_t row, T s) const { return apply(row, s, load(row)); }
    __device__ void store_partial(uint32_t b, double v) const { partial[b] = v; }
};

// r = b - A x, partial += r^2 (optional)
template <class T, bool kNorm>
struct EpiResidual {
    static constexpr bool kPartial = kNorm;
    struct Pre {
        T b;
    };
    const T* b;
    T* r;
    double* partial;
    __device__ Pre load(uint32_t row) const { return {b[row]}; }
    __device__ double apply(uint32_t row, T s, const Pre& p) const {
#pragma clang fp contract(off)
        const T v = p.b - s;
        r[row] = v;
        return kNorm ? double(v) * double(v) : 0.0;
    }
    __device__ double operator()(uint32_t row, T s) const { return apply(row, s, load(row)); }
    __device__ void store_partial(uint32_t bb, double v) const { partial[bb] = v; }
};

// Damped Jacobi sweep (amg_preconditioner.h:2394-2405):
// xn = x + omega * (inv_diag * (b - A x))
template <class T>
struct EpiJacobi {
    static constexpr bool kPartial = false;
    struct Pre {
        T b, x, inv;
    };
    const T* b;
    const T* x;
    const T* inv_diag;
    T* xn;
    T omega;
    __device__ Pre load(uint32_t row) const { return {b[row], x[row], inv_diag[row]}; }
    __device__ double apply(uint32_t row, T s, const Pre& p) const {
#pragma clang fp contract(off)
        const T delta = p.inv * (p.b - s);
        xn[row] = p.x + omega * delta;
        return 0.0;
    }
    __device__ double operator()(uint32_t row, T s) const { return apply(row, s, load(row)); }
    __device__ void store_partial(uint32_t, double) const {}
};

// Chebyshev step (three-term recurrence, Jacobi-preconditioned):
// dn = c1 * d + c2 * (inv_diag * (b - A x)), xn = x + dn, d <- dn.
// kFirst: the step that starts the recurrence (no previous direction).
template <class T, bool kFirst>
struct EpiCheb {
    static constexpr bool kPartial = false;
    struct Pre {
        T b, x, inv, d;
    };
    const T* b;
    const T* x;
    const T* inv_diag;
    T* d;
    T* xn;
    T c1, c2;
    __device__ Pre load(uint32_t row) const { return {b[row], x[row], inv_diag[row], kFirst ? T(0) : d[row]}; }
    __device__ double apply(uint32_t row, T s, const Pre& p) const {
#pragma clang fp contract(off)
        const T delta = p.inv * (p.b - s);
        const T dn = kFirst ? c2 * delta : c1 * p.d + c2 * delta;
        d[row] = dn;
        xn[row] = p.x + dn;
        return 0.0;
    }
    __device__ double operator()(uint32_t row, T s) const { return apply(row, s, load(row)); }
    __device__ void store_partial(uint32_t, double) const {}
};

// Chebyshev step on the row-scaled half copy: dn = c1 * d + c2 * (bt - B x)
// with B = D^-1 A and bt = D^-1 b, xn = x + dn, d <- dn (FP32).
template <bool kFirst>
struct EpiChebHalf {
    static constexpr bool kPartial = false;
    struct Pre {
        float bt, x, d;
    };
    const float* bt;
    const float* x;
    float* d;
    float* xn;
    float c1, c2;
    __device__ Pre load(uint32_t row) const { return {bt[row], x[row], kFirst ? 0.0f : d[row]}; }
    __device__ double apply(uint32_t row, float s, const Pre& p) const {
#pragma clang fp contract(off)
        const float delta = p.bt - s;
        const float dn = kFirst ? c2 * delta : c1 * p.d + c2 * delta;
        d[row] = dn;
        xn[row] = p.x + dn;
        return 0.0;
    }
};

// Prolongation x_i += sum_c P_ic xc_c accumulated onto x_i in entry order
// (amg_preconditioner.h:2432-2436): init = x, store back.
template <class T>
struct EpiAssign {
    static constexpr bool kPartial = false;
    using Pre = NoPre;
    T* y;
    __device__ Pre load(uint32_t) const { return {}; }
    __device__ double apply(uint32_t row, T s, const Pre&) const {
        y[row] = s;
        return 0.0;
    }
    __device__ double operator()(uint32_t row, T s) const { return apply(row, s, load(row)); }
    __device__ void store_partial(uint32_t, double) const {}
};

// -------------------------------------------------------------- vectors --

// First sweep from x = 0: A*0 = 0, so x = omega * (inv_diag * b).
// First Chebyshev step from x = 0: d = c2 * (inv_diag * b), x = d.
template <class T>
__global__ __launch_bounds__(kBlock) void cheb_first_kernel(uint32_t n, const T* __restrict__ b,
                                                           const T* __restrict__ inv_diag, T c2,
                                                           T* __restrict__ d, T* __restrict__ x) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) {
        const T v = c2 * (inv_diag[i] * b[i]);
        d[i] = v;
        x[i] = v;
    }
}

// First Chebyshev step from x = 0 that also keeps bt = D^-1 b for the
// half-copy steps: the same d and x as cheb_first_kernel.
static __global__ __launch_bounds__(kBlock) void cheb_first_half_kernel(uint32_t n, const float* __restrict__ b,
                                                                const float* __restrict__ inv_diag, float c2,
                                                                float* __restrict__ bt, float* __restrict__ d,
                                                                float* __restrict__ x) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) {
        const float t = inv_diag[i] * b[i];
        bt[i] = t;
        const float v = c2 * t;
        d[i] = v;
        x[i] = v;
    }
}

// bt = D^-1 b (post-smoothing without a pre-smoothing pass).
static __global__ __launch_bounds__(kBlock) void scale_by_kernel(uint32_t n, const float* __restrict__ b,
                                                         const float* __restrict__ inv_diag, float* __restrict__ bt) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) bt[i] = inv_diag[i] * b[i];
}

template <class T>
__global__ __launch_bounds__(kBlock) void jacobi_first_kernel(uint32_t n, const T* __restrict__ b,
                                                             const T* __restrict__ inv_diag, T omega,
                                                             T* __restrict__ x) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) x[i] = omega * (inv_diag[i] * b[i]);
}

template <class T>
__global__ __launch_bounds__(kBlock) void fill_kernel(uint32_t n, T v, T* __restrict__ x) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) x[i] = v;
}

template <class S, class D>
__global__ __launch_bounds__(kBlock) void convert_kernel(uint32_t n, const S* __restrict__ s, D* __restrict__ d) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) d[i] = D(s[i]);
}

// dst[new_of_old[i]] = src[i]  (caller ordering -> solve ordering)
template <class S, class D>
__global__ __launch_bounds__(kBlock) void scatter_perm_kernel(uint32_t n, const uint32_t* __restrict__ new_of_old,
                                                             const S* __restrict__ src, D* __restrict__ dst) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) dst[new_of_old[i]] = D(src[i]);
}

// dst[i] = src[new_of_old[i]]  (solve ordering -> caller ordering)
template <class S, class D>
__global__ __launch_bounds__(kBlock) void gather_perm_kernel(uint32_t n, const uint32_t* __restrict__ new_of_old,
                                                            const S* __restrict__ src, D* __restrict__ dst) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) dst[i] = D(src[new_of_old[i]]);
}

// Partial dot products a.b over grid-stride chunks.
template <class T>
__global__ __launch_bounds__(kBlock) void dot_partial_kernel(uint32_t n, const T* __restrict__ a,
                                                            const T* __restrict__ b, double* __restrict__ partial) {
    __shared__ double red[4];
    double v = 0.0;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
        v += double(a[i]) * double(b[i]);
    v = block_sum(v, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = v;
}

// PCG update (cg_solver.h:285-294): alpha = rsold / pAp; the update is
// skipped when the curvature or alpha is invalid (the solver then stops with
// x untouched, as the reference does). partial += r^2.
static __global__ __launch_bounds__(kBlock) void cg_update_kernel(uint32_t n, double rsold, const double* __restrict__ pAp_ptr,
                                                          const double* __restrict__ p, const double* __restrict__ Ap,
                                                          double* __restrict__ x, double* __restrict__ r,
                                                          double* __restrict__ partial) {
#pragma clang fp contract(off)
    __shared__ double red[4];
    const double pAp = *pAp_ptr;
    const double alpha = rsold / pAp;
    const bool ok = pAp > 0.0 && isfinite(pAp) && isfinite(alpha);
    double v = 0.0;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        double ri = r[i];
        if (ok) {
            x[i] += alpha * p[i];
            ri -= alpha * Ap[i];
            r[i] = ri;
        }
        v += ri * ri;
    }
    v = block_sum(v, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = v;
}

// p = z + beta p
static __global__ __launch_bounds__(kBlock) void cg_direction_kernel(uint32_t n, double beta, const double* __restrict__ z,
                                                             double* __restrict__ p) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) p[i] = z[i] + beta * p[i];
}

template <class T>
__global__ __launch_bounds__(kBlock) void copy_kernel(uint32_t n, const T* __restrict__ s, T* __restrict__ d) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) d[i] = s[i];
}

// -------------------------------------------------------- coarse solve --

// Replays the dense partial-pivot elimination of the coarsest level
// (amg_preconditioner.h:2603-2663) with factors computed once at setup. One
// wavefront, order n <= 17 (16 unknowns, bordered); nr unknowns (n or n - 1),
// the border's right-hand side is 0. Lane i owns component i: a forward step
// updates every component at once, each with the operations of the sequential
// elimination. The back substitution subtracts a row's terms in ascending
// column order, a chain that only lane ii can follow, so its products are
// formed by the lanes and read in order, by lane reads: 17 FGMRES steps on 67k
// rows take 3580 us so, 3680 with shuffles (11 us a solve of order 16). One lane
// with its arrays in scratch memory took 24 us a solve.
template <class T>
__device__ __forceinline__ void coarse_lu_solve(uint32_t n, uint32_t nr, const uint32_t* __restrict__ piv,
                                                const double* __restrict__ factor, const double* __restrict__ upper,
                                                const T* r, T* x, double* sm /* 2 * 17 * 17 */) {
#pragma clang fp contract(off)
    const uint32_t lane = threadIdx.x & 63u;
    double* F = sm;
    double* U = sm + 17 * 17;
    for (uint32_t k = lane; k < n * n; k += 64) {
        F[k] = factor[k];
        U[k] = upper[k];
    }
    double b = lane < nr ? double(r[lane]) : 0.0;
    const uint32_t pv = lane < n ? piv[lane] : 0u;
    wave_fence();
    for (uint32_t k = 0; k < n; ++k) {
        const int p = __builtin_amdgcn_readlane(int(pv), int(k));
        const double bk = lane_value(b, int(k)), bp = lane_value(b, p);
        if (lane == k) b = bp;
        else if (int(lane) == p) b = bk;
        if (lane > k && lane < n) b -= F[k * n + lane] * bp;
    }
    double s = 0.0;  // lane i: component i of the solution once it is known
    for (uint32_t ii = n; ii-- > 0;) {
        // Products of row ii, lane j holds upper[ii][j] s[j].
        const double t = lane > ii && lane < n ? U[ii * n + lane] * s : 0.0;
        double sum = lane_value(b, int(ii));
        for (uint32_t j = ii + 1; j < n; ++j) sum -= lane_value(t, int(j));
        if (lane == ii) s = sum / U[ii * n + ii];
    }
    if (lane < nr) x[lane] = T(s);
}

template <class T>
__global__ __launch_bounds__(64) void coarse_lu_kernel(uint32_t n, uint32_t nr, const uint32_t* __restrict__ piv,
                                 const double* __restrict__ factor, const double* __restrict__ upper,
                                 const T* __restrict__ r, T* __restrict__ x) {
    __shared__ double sm[2 * 17 * 17];
    coarse_lu_solve<T>(n, nr, piv, factor, upper, r, x, sm);
}

// Partial sums of v over grid-stride chunks (the mean of the constant null
// space), in double.
template <class T>
__global__ __launch_bounds__(kBlock) void sum_partial_kernel(uint32_t n, const T* __restrict__ v,
                                                             double* __restrict__ partial) {
    __shared__ double red[4];
    double a = 0.0;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) a += double(v[i]);
    a = block_sum(a, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = a;
}

// v -= sum / count, sum read from device memory (amg_preconditioner.h:
// 1310-1319: mean = sum / n, then v_i - mean).
template <class T>
__global__ __launch_bounds__(kBlock) void subtract_mean_kernel(uint32_t n, T* __restrict__ v,
                                                               const double* __restrict__ sum, double count) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) v[i] = v[i] - T(sum[0] / count);
}

// v -= c m with c read from device memory (one null-space mode,
// null_space.h:67-74).
__global__ __launch_bounds__(kBlock) static void remove_mode_kernel(uint32_t n, double* __restrict__ v,
                                                                    const double* __restrict__ m,
                                                                    const double* __restrict__ c) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) v[i] -= c[0] * m[i];
}

}  // namespace cfdxhip
