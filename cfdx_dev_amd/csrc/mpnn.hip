// Learned preconditioner stage: forward, backward and Adam kernels (HIP,
// gfx950). Layout and algorithm are described in mpnn.hpp.
//
// Tiling: the training kernels work on tiles of 64 nodes per 256-thread
// workgroup; inference gives each wavefront its own 16-node sub-tiles on a
// persistent grid. The gather phase gives each node 4 lanes of 8 channels
// (16-byte BF16 rows), with neighbour loads issued in batches of eight; the
// dense phase gives each wavefront 16 nodes and runs 16x16x16 BF16 MFMAs on
// LDS tiles. Parameter gradients are written as per-tile partials (one row of
// kMpnnParams floats per tile) and summed in tile order: no atomics, the
// result does not depend on scheduling.
#include "mpnn.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <stdexcept>

#include "kernels.hpp"
#include "parallel.h"

namespace cfdxhip {

#define MPNN_HIP(expr)                                                                            \
    do {                                                                                          \
        hipError_t e_ = (expr);                                                                   \
        if (e_ != hipSuccess)                                                                     \
            throw std::runtime_error(std::string("HIP error ") + hipGetErrorString(e_) + " at " + \
                                     __FILE__ + ":" + std::to_string(__LINE__));                  \
    } while (0)

namespace {

constexpr int kTile = 64;   // nodes per workgroup
constexpr int kLd = 68;     // LDS row stride (elements) of 64-wide BF16 tiles
constexpr int kLd32 = 36;   // LDS row stride of 32-wide BF16 tiles
constexpr int kMaxPartBlocks = 4096;

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <class T>
T* mpnn_alloc(uint64_t count) {
    if (count == 0) count = 1;
    void* p = nullptr;
    MPNN_HIP(hipMalloc(&p, count * sizeof(T)));
    return static_cast<T*>(p);
}
template <class T>
void mpnn_free(T*& p) {
    if (p) (void)hipFree(p);
    p = nullptr;
}

// Round-to-nearest-even FP32 -> BF16 (NaN kept quiet).
__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return uint16_t((u >> 16) | 0x40u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return uint16_t(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t b) { return __uint_as_float(uint32_t(b) << 16); }
__device__ __forceinline__ uint32_t pack2(float a, float b) { return uint32_t(f2bf(a)) | (uint32_t(f2bf(b)) << 16); }

// Eight channels [8q, 8q + 8) of node j: BF16 hidden states (kept packed,
// four registers per row, until they are accumulated) or FP32 rows.
struct LoadBf8 {
    using Raw = uint4;
    const uint16_t* h;
    uint32_t q;
    __device__ __forceinline__ Raw raw(uint32_t j) const {
        return *reinterpret_cast<const uint4*>(h + size_t(j) * kHid + 8 * q);
    }
    __device__ __forceinline__ static void unpack(const Raw& u, float* v) {
        const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            v[2 * t] = __uint_as_float(w[t] << 16);
            v[2 * t + 1] = __uint_as_float(w[t] & 0xffff0000u);
        }
    }
    __device__ __forceinline__ void operator()(uint32_t j, float* v) const { unpack(raw(j), v); }
};
struct LoadF8 {
    struct Raw {
        float4 a, b;
    };
    const float* g;
    uint32_t q;
    __device__ __forceinline__ Raw raw(uint32_t j) const {
        return {*reinterpret_cast<const float4*>(g + size_t(j) * kHid + 8 * q),
                *reinterpret_cast<const float4*>(g + size_t(j) * kHid + 8 * q + 4)};
    }
    __device__ __forceinline__ static void unpack(const Raw& r, float* v) {
        v[0] = r.a.x, v[1] = r.a.y, v[2] = r.a.z, v[3] = r.a.w;
        v[4] = r.b.x, v[5] = r.b.y, v[6] = r.b.z, v[7] = r.b.w;
    }
    __device__ __forceinline__ void operator()(uint32_t j, float* v) const { unpack(raw(j), v); }
};

// m[c] = sum_{j != i} w_ij x_j[8q + c], w_ij = (-a_ij s_i) s_j, in entry
// order. Neighbour indices, then the neighbours' rows, are loaded in batches
// of eight so that their latencies overlap.
template <class Load>
__device__ __forceinline__ void gather8(uint32_t i, const uint32_t* __restrict__ rowp,
                                        const uint32_t* __restrict__ cols, const float* __restrict__ vals,
                                        const float* __restrict__ s, const Load& ld, float* m) {
#pragma unroll
    for (int c = 0; c < 8; ++c) m[c] = 0.0f;
    const float si = s[i];
    const uint32_t k0 = rowp[i], k1 = rowp[i + 1];
    for (uint32_t k = k0; k < k1; k += 8) {
        uint32_t jj[8];
        float ww[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const bool ok = k + u < k1;
            jj[u] = ok ? cols[k + u] : i;
            ww[u] = ok ? vals[k + u] : 0.0f;
        }
        float sj[8];
        typename Load::Raw raw[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            sj[u] = s[jj[u]];
            raw[u] = ld.raw(jj[u]);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (jj[u] == i) continue;
            const float w = (-ww[u] * si) * sj[u];
            float hv[8];
            ld.unpack(raw[u], hv);
#pragma unroll
            for (int c = 0; c < 8; ++c) m[c] += w * hv[c];
        }
    }
}

// D (16x16, FP32) += A (16 x K) * B (K x 16), A row-major in LDS with stride
// lda, B supplied transposed (Bt[n][k], stride ldb). Lane l feeds
// A[l%16][k0 + 4(l/16) + 0..3] and Bt[l%16][k0 + 4(l/16) + 0..3] per K step of
// 16; D comes back as D[4(l/16) + j][l%16], j = 0..3.
__device__ __forceinline__ f32x4 mfma_tile(const uint16_t* A, int lda, const uint16_t* Bt, int ldb, int K,
                                           f32x4 acc) {
    const int lane = threadIdx.x & 63;
    const uint16_t* pa = A + (lane & 15) * lda + 4 * (lane >> 4);
    const uint16_t* pb = Bt + (lane & 15) * ldb + 4 * (lane >> 4);
    for (int k = 0; k < K; k += 16) {
        const bf16x4 a = *reinterpret_cast<const bf16x4*>(pa + k);
        const bf16x4 b = *reinterpret_cast<const bf16x4*>(pb + k);
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
    }
    return acc;
}

// rho and 1/rho, computed once per forward pass into scal[3], scal[4].
__global__ void rho_kernel(double* scal, uint32_t n) {
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        const double rho = std::sqrt(scal[0] / double(n));
        scal[3] = rho;
        scal[4] = rho > 0.0 ? 1.0 / rho : 0.0;
    }
}
__device__ __forceinline__ float inv_rho_of(const double* scal, uint32_t) { return float(scal[4]); }
__device__ __forceinline__ float rho_of(const double* scal, uint32_t) { return float(scal[3]); }

// s_i = sqrt(inv_diag_i); partial[block] = sum (r_i s_i)^2 (grid stride).
__global__ __launch_bounds__(kBlock) void scale_kernel(uint32_t n, const float* __restrict__ r,
                                                      const float* __restrict__ inv_diag, float* __restrict__ s,
                                                      double* __restrict__ partial) {
    __shared__ double red[4];
    double acc = 0.0;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        const float si = std::sqrt(inv_diag[i]);
        s[i] = si;
        const double v = double(r[i]) * double(si);
        acc += v * v;
    }
    acc = block_sum(acc, red);
    if (threadIdx.x == 0) partial[blockIdx.x] = acc;
}

// h0 = relu(u w_in + b_in); thread per (node, channel), 8 nodes per block.
__global__ __launch_bounds__(kBlock) void encode_kernel(uint32_t n, const float* __restrict__ r,
                                                       const float* __restrict__ s, const double* __restrict__ scal,
                                                       const float* __restrict__ p, uint16_t* __restrict__ h0,
                                                       uint32_t* __restrict__ mask) {
    const uint64_t t = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    const uint32_t i = uint32_t(t >> 5), c = uint32_t(t & 31);
    const float inv = inv_rho_of(scal, n);
    float z = 0.0f;
    if (i < n) {
        const float u = r[i] * s[i] * inv;
        z = u * p[c] + p[kHid + c];
        h0[size_t(i) * kHid + c] = f2bf(std::max(z, 0.0f));
    }
    const uint64_t bits = __ballot(z > 0.0f);
    if (mask && i < n && c == 0) mask[i] = uint32_t(bits >> (threadIdx.x & 32));
}

// Inference encoder: the rows encode_kernel writes, eight channels (one
// 16-byte store) per thread.
__global__ __launch_bounds__(kBlock) void encode8_kernel(uint32_t n, const float* __restrict__ r,
                                                        const float* __restrict__ s,
                                                        const double* __restrict__ scal,
                                                        const float* __restrict__ p, uint16_t* __restrict__ h0) {
#pragma clang fp contract(off)
    const uint64_t t = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    const uint32_t i = uint32_t(t >> 2), q = uint32_t(t & 3);
    if (i >= n) return;
    const float u = r[i] * s[i] * inv_rho_of(scal, n);
    float h[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const float z = u * p[8 * q + c] + p[kHid + 8 * q + c];
        h[c] = std::max(z, 0.0f);
    }
    *reinterpret_cast<uint4*>(h0 + size_t(i) * kHid + 8 * q) =
        make_uint4(pack2(h[0], h[1]), pack2(h[2], h[3]), pack2(h[4], h[5]), pack2(h[6], h[7]));
}

// One training message-passing layer: X = [h_i ; sum_j w_ij h_j] (64 x 64,
// BF16 in LDS), h_out = relu(X W + b) + h_i, and each node's ReLU mask for the
// backward pass. Inference runs layer_wave_kernel (the same values).
__global__ __launch_bounds__(kBlock) void layer_kernel(uint32_t n, const uint32_t* __restrict__ rowp,
                                                      const uint32_t* __restrict__ cols,
                                                      const float* __restrict__ vals, const float* __restrict__ s,
                                                      const uint16_t* __restrict__ hin, uint16_t* __restrict__ hout,
                                                      const uint16_t* __restrict__ wt_g,
                                                      const float* __restrict__ bias, uint32_t* __restrict__ mask) {
    __shared__ __align__(16) uint16_t X[kTile * kLd];
    __shared__ __align__(16) uint16_t Wt[kHid * kLd];
    __shared__ float Y[kTile * (kHid + 1)];
    __shared__ uint8_t Mk[kTile * kHid];
    const int tid = threadIdx.x;
    const uint32_t node0 = blockIdx.x * kTile;
    for (int e = tid; e < kHid * 2 * kHid; e += kBlock) Wt[(e >> 6) * kLd + (e & 63)] = wt_g[e];
    // 4 lanes per node, 8 channels per lane.
    const int il = tid >> 2, q = tid & 3;
    {
        const uint32_t i = node0 + il;
        uint4 hv = {0u, 0u, 0u, 0u};
        float m[8];
        if (i < n) {
            hv = *reinterpret_cast<const uint4*>(hin + size_t(i) * kHid + 8 * q);
            gather8(i, rowp, cols, vals, s, LoadBf8{hin, uint32_t(q)}, m);
        } else {
#pragma unroll
            for (int c = 0; c < 8; ++c) m[c] = 0.0f;
        }
        uint2* xh = reinterpret_cast<uint2*>(X + il * kLd + 8 * q);
        xh[0] = make_uint2(hv.x, hv.y);
        xh[1] = make_uint2(hv.z, hv.w);
        uint2* xm = reinterpret_cast<uint2*>(X + il * kLd + kHid + 8 * q);
        xm[0] = make_uint2(pack2(m[0], m[1]), pack2(m[2], m[3]));
        xm[1] = make_uint2(pack2(m[4], m[5]), pack2(m[6], m[7]));
    }
    __syncthreads();
    const int wave = tid >> 6, lane = tid & 63;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        acc = mfma_tile(X + wave * 16 * kLd, kLd, Wt + nt * 16 * kLd, kLd, 2 * kHid, acc);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = wave * 16 + 4 * (lane >> 4) + j;
            const int col = nt * 16 + (lane & 15);
            const float z = acc[j] + bias[col];
            Y[row * (kHid + 1) + col] = std::max(z, 0.0f) + bf2f(X[row * kLd + col]);
            Mk[row * kHid + col] = z > 0.0f ? 1 : 0;
        }
    }
    __syncthreads();
    {
        const uint32_t i = node0 + il;
        if (i < n) {
            const float* y = Y + il * (kHid + 1) + 8 * q;
            *reinterpret_cast<uint4*>(hout + size_t(i) * kHid + 8 * q) =
                make_uint4(pack2(y[0], y[1]), pack2(y[2], y[3]), pack2(y[4], y[5]), pack2(y[6], y[7]));
        }
    }
    if (tid < kTile && node0 + tid < n) {
        uint32_t bits = 0;
        for (int cc = 0; cc < kHid; ++cc) bits |= uint32_t(Mk[tid * kHid + cc]) << cc;
        mask[node0 + tid] = bits;
    }
}

// gather8 split into stages, so a wavefront can issue the row offsets and the
// first batch of neighbour indices of its next node while it gathers the
// current one. The sums are gather8's: batches in order, entries in order.
struct NbrBatch {
    uint32_t k0 = 0, k1 = 0;
    uint32_t jj[8];
    float ww[8];
};
__device__ __forceinline__ void batch_fill(NbrBatch& b, uint32_t i, const uint32_t* __restrict__ cols,
                                           const float* __restrict__ vals) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const bool ok = b.k0 + u < b.k1;
        b.jj[u] = ok ? cols[b.k0 + u] : i;
        b.ww[u] = ok ? vals[b.k0 + u] : 0.0f;
    }
}
template <class Load>
__device__ __forceinline__ void gather8_from(const NbrBatch& b, uint32_t i, float si,
                                             const uint32_t* __restrict__ rowp, const uint32_t* __restrict__ cols,
                                             const float* __restrict__ vals, const float* __restrict__ s,
                                             const Load& ld, float* m) {
#pragma unroll
    for (int c = 0; c < 8; ++c) m[c] = 0.0f;
    {
        float sj[8];
        typename Load::Raw raw[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            sj[u] = s[b.jj[u]];
            raw[u] = ld.raw(b.jj[u]);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (b.jj[u] == i) continue;
            const float w = (-b.ww[u] * si) * sj[u];
            float hv[8];
            ld.unpack(raw[u], hv);
#pragma unroll
            for (int c = 0; c < 8; ++c) m[c] += w * hv[c];
        }
    }
    for (uint32_t k = b.k0 + 8; k < b.k1; k += 8) {
        uint32_t jj[8];
        float ww[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const bool ok = k + u < b.k1;
            jj[u] = ok ? cols[k + u] : i;
            ww[u] = ok ? vals[k + u] : 0.0f;
        }
        float sj[8];
        typename Load::Raw raw[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            sj[u] = s[jj[u]];
            raw[u] = ld.raw(jj[u]);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (jj[u] == i) continue;
            const float w = (-ww[u] * si) * sj[u];
            float hv[8];
            ld.unpack(raw[u], hv);
#pragma unroll
            for (int c = 0; c < 8; ++c) m[c] += w * hv[c];
        }
    }
}

// Inference layer: the arithmetic of layer_kernel (bit-identical output),
// with each wavefront owning its X and Y tiles in LDS and working through
// 16-node sub-tiles on its own, no workgroup barrier after the weights are
// staged once per workgroup. The grid is persistent: the workgroups on one
// XCD take one contiguous eighth of the sub-tiles, so that XCD's L2 serves a
// contiguous window of neighbour rows. kDec applies the decoder to the
// rounded output rows and writes e (the last layer, no h_out array), as
// decode_kernel would.
constexpr int kSub = 16;  // nodes per wavefront sub-tile
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
template <bool kDec>
__global__ __launch_bounds__(kBlock) void layer_wave_kernel(uint32_t n, const uint32_t* __restrict__ rowp,
                                                           const uint32_t* __restrict__ cols,
                                                           const float* __restrict__ vals,
                                                           const float* __restrict__ s,
                                                           const uint16_t* __restrict__ hin,
                                                           uint16_t* __restrict__ hout,
                                                           const uint16_t* __restrict__ wt_g,
                                                           const float* __restrict__ bias,
                                                           const double* __restrict__ scal,
                                                           const float* __restrict__ p, float* __restrict__ e) {
    constexpr int kWaves = kBlock / 64;
    __shared__ __align__(16) uint16_t Wt[kHid * kLd];
    __shared__ __align__(16) uint16_t Xs[kWaves][kSub * kLd];
    __shared__ float Ys[kWaves][kSub * (kHid + 1)];
    const int tid = threadIdx.x;
    for (int e8 = tid; e8 < kHid * 2 * kHid / 8; e8 += kBlock) {
        const uint4 v = reinterpret_cast<const uint4*>(wt_g)[e8];
        uint2* d = reinterpret_cast<uint2*>(Wt + (e8 >> 3) * kLd + 8 * (e8 & 7));
        d[0] = make_uint2(v.x, v.y);
        d[1] = make_uint2(v.z, v.w);
    }
    __syncthreads();
    const int wave = tid >> 6, lane = tid & 63;
    uint16_t* X = Xs[wave];
    float* Y = Ys[wave];
    const int il = lane >> 2, q = lane & 3;
    float bcol[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) bcol[nt] = bias[nt * 16 + (lane & 15)];
    // This XCD's contiguous range of sub-tiles, shared by its workgroups.
    const uint32_t nsub = (n + kSub - 1) / kSub;
    const uint32_t xcd = blockIdx.x % kXcds, local = blockIdx.x / kXcds;
    const uint32_t per_xcd = gridDim.x / kXcds;
    const uint32_t span = (nsub + kXcds - 1) / kXcds;
    const uint32_t first = xcd * span, last = std::min(nsub, first + span);
    const uint32_t stride = per_xcd * kWaves;
    uint32_t sub = first + local * kWaves + wave;
    // The first batch of this lane's node in the next sub-tile is loaded
    // while the current one is gathered.
    NbrBatch cur;
    {
        const uint32_t i = sub * kSub + il;
        if (sub < last && i < n) {
            cur.k0 = rowp[i];
            cur.k1 = rowp[i + 1];
            batch_fill(cur, i, cols, vals);
        }
    }
    for (; sub < last; sub += stride) {
        const uint32_t i = sub * kSub + il;
        const uint32_t sub_n = sub + stride, i_n = sub_n * kSub + il;
        const bool has_n = sub_n < last && i_n < n;
        uint32_t nk0 = 0, nk1 = 0;
        if (has_n) {
            nk0 = rowp[i_n];
            nk1 = rowp[i_n + 1];
        }
        uint4 hv = {0u, 0u, 0u, 0u};
        float m[8];
        if (i < n) {
            hv = *reinterpret_cast<const uint4*>(hin + size_t(i) * kHid + 8 * q);
            gather8_from(cur, i, s[i], rowp, cols, vals, s, LoadBf8{hin, uint32_t(q)}, m);
        } else {
#pragma unroll
            for (int c = 0; c < 8; ++c) m[c] = 0.0f;
        }
        cur.k0 = nk0;
        cur.k1 = nk1;
        if (has_n) batch_fill(cur, i_n, cols, vals);
        uint2* xh = reinterpret_cast<uint2*>(X + il * kLd + 8 * q);
        xh[0] = make_uint2(hv.x, hv.y);
        xh[1] = make_uint2(hv.z, hv.w);
        uint2* xm = reinterpret_cast<uint2*>(X + il * kLd + kHid + 8 * q);
        xm[0] = make_uint2(pack2(m[0], m[1]), pack2(m[2], m[3]));
        xm[1] = make_uint2(pack2(m[4], m[5]), pack2(m[6], m[7]));
        wave_sync();
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            acc = mfma_tile(X, kLd, Wt + nt * 16 * kLd, kLd, 2 * kHid, acc);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int row = 4 * (lane >> 4) + j;
                const int col = nt * 16 + (lane & 15);
                const float z = acc[j] + bcol[nt];
                Y[row * (kHid + 1) + col] = std::max(z, 0.0f) + bf2f(X[row * kLd + col]);
            }
        }
        wave_sync();
        if constexpr (kDec) {
            float yv = 0.0f;
            if (i < n) {
                const float* y = Y + il * (kHid + 1) + 8 * q;
                const float* w = p + kOffWout + 8 * q;
                float v[8];
#pragma unroll
                for (int c = 0; c < 8; ++c) v[c] = bf2f(f2bf(y[c]));
#pragma unroll
                for (int c = 0; c < 8; ++c) yv += v[c] * w[c];
            }
            yv += __shfl_xor(yv, 1, 4);
            yv += __shfl_xor(yv, 2, 4);
            if (i < n && q == 0) e[i] = rho_of(scal, n) * s[i] * (yv + p[kOffWout + kHid]);
        } else if (i < n) {
            const float* y = Y + il * (kHid + 1) + 8 * q;
            *reinterpret_cast<uint4*>(hout + size_t(i) * kHid + 8 * q) =
                make_uint4(pack2(y[0], y[1]), pack2(y[2], y[3]), pack2(y[4], y[5]), pack2(y[6], y[7]));
        }
        wave_sync();  // X and Y are rewritten by the next sub-tile
    }
}

// e_i = rho s_i (h_i . w_out + b_out); 4 lanes per node, 8 channels each.
__global__ __launch_bounds__(kBlock) void decode_kernel(uint32_t n, const uint16_t* __restrict__ h,
                                                       const float* __restrict__ s, const double* __restrict__ scal,
                                                       const float* __restrict__ p, float* __restrict__ e) {
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    const uint32_t i = t >> 2, q = t & 3;
    const float* w = p + kOffWout + 8 * q;
    float y = 0.0f;
    if (i < n) {
        float v[8];
        LoadBf8{h, q}(i, v);
#pragma unroll
        for (int c = 0; c < 8; ++c) y += v[c] * w[c];
    }
    y += __shfl_xor(y, 1, 4);
    y += __shfl_xor(y, 2, 4);
    if (i < n && q == 0) e[i] = rho_of(scal, n) * s[i] * (y + p[kOffWout + kHid]);
}

// Sum of acc over the 8 node slots of a 64-node tile, per channel, into
// out[c] (thread tid < 32 holds channel tid's total on return).
__device__ __forceinline__ float tile_channel_sum(float acc, float* red /* 8 x 32 */) {
    const int tid = threadIdx.x;
    red[(tid >> 5) * kHid + (tid & 31)] = acc;
    __syncthreads();
    float t = 0.0f;
    if (tid < kHid)
        for (int k = 0; k < 8; ++k) t += red[k * kHid + tid];
    __syncthreads();
    return t;
}

// Decoder backward: gy = ge rho s; gh = gy w_out; partials of w_out, b_out.
__global__ __launch_bounds__(kBlock) void decode_bwd_kernel(uint32_t n, const float* __restrict__ ge,
                                                           const float* __restrict__ s,
                                                           const double* __restrict__ scal,
                                                           const uint16_t* __restrict__ h, const float* __restrict__ p,
                                                           float* __restrict__ gh, float* __restrict__ gpart) {
    __shared__ float red[8 * kHid];
    const int tid = threadIdx.x, c = tid & 31, sub = tid >> 5;
    const uint32_t node0 = blockIdx.x * kTile;
    const float rho = rho_of(scal, n);
    const float wc = p[kOffWout + c];
    float aw = 0.0f, ab = 0.0f;
    for (int il = sub; il < kTile; il += 8) {
        const uint32_t i = node0 + il;
        if (i >= n) continue;
        const float gy = ge[i] * rho * s[i];
        gh[size_t(i) * kHid + c] = gy * wc;
        aw += gy * bf2f(h[size_t(i) * kHid + c]);
        ab += gy;
    }
    const float tw = tile_channel_sum(aw, red);
    const float tb = tile_channel_sum(ab, red);
    float* out = gpart + size_t(blockIdx.x) * kMpnnParams;
    if (tid < kHid) out[kOffWout + tid] = tw;
    if (tid == 0) out[kOffWout + kHid] = tb;  // every channel slot saw the same gy
}

// Layer backward. In: gh = dL/dh_out, the layer's relu mask, h_prev.
// Out: gh2 = gh + (dL/dX)[:, :32] (residual + self path), gm = (dL/dX)[:, 32:],
// per-tile partials of dL/dW (X^T gz) and dL/db (sum gz). Bound by the latency
// of the neighbour gathers, so by the tiles resident: 23 KB of LDS a tile hold
// six a CU, which takes the 1050 tiles of 67k nodes in one go (47 KB, with
// dL/dX and the FP32 gz in places of their own, held three: 18.2 us
// a layer, now 15.5).
__global__ __launch_bounds__(kBlock) void layer_bwd_kernel(
    uint32_t n, const uint32_t* __restrict__ rowp, const uint32_t* __restrict__ cols, const float* __restrict__ vals,
    const float* __restrict__ s, const uint16_t* __restrict__ hprev, const uint32_t* __restrict__ mask,
    const uint16_t* __restrict__ w_g, const float* __restrict__ gh, float* __restrict__ gh2, float* __restrict__ gm,
    float* __restrict__ gpart, uint32_t layer_off) {
    constexpr int kXt = 2 * kHid * kLd, kGz = kTile * kLd32, kGzt = kHid * kLd, kG = kTile * (2 * kHid + 1);
    __shared__ __align__(16) uint16_t W[2 * kHid * kLd32];  // [f][c]
    __shared__ float GB[4 * kHid];                          // per-wavefront column sums of gz
    __shared__ __align__(16) uint16_t tile[std::max(kXt + kGz + kGzt, 2 * kG)];
    uint16_t* XT = tile;                        // [f][node]
    uint16_t* GZ = tile + kXt;                  // [node][c]
    uint16_t* GZT = tile + kXt + kGz;           // [c][node]
    float* G = reinterpret_cast<float*>(tile);  // dL/dX [node][f], in their place once both products are formed
    const int tid = threadIdx.x;
    const uint32_t node0 = blockIdx.x * kTile;
    for (int e = tid; e < 2 * kHid * kHid; e += kBlock) W[(e >> 5) * kLd32 + (e & 31)] = w_g[e];
    // 4 lanes per node, 8 channels per lane.
    const int il = tid >> 2, q = tid & 3;
    const uint32_t i = node0 + il;
    float ghv[8], m[8], hv[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) ghv[c] = m[c] = hv[c] = 0.0f;
    uint32_t mk = 0;
    if (i < n) {
        LoadBf8{hprev, uint32_t(q)}(i, hv);
        gather8(i, rowp, cols, vals, s, LoadBf8{hprev, uint32_t(q)}, m);
        LoadF8{gh, uint32_t(q)}(i, ghv);
        mk = mask[i] >> (8 * q);
    }
    float gzs[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int f = 8 * q + c;
        const float gz = ((mk >> c) & 1u) ? ghv[c] : 0.0f;
        XT[f * kLd + il] = f2bf(hv[c]);  // exact: hv holds BF16 values
        XT[(kHid + f) * kLd + il] = f2bf(m[c]);
        const uint16_t gzb = f2bf(gz);
        GZ[il * kLd32 + f] = gzb;
        GZT[f * kLd + il] = gzb;
        gzs[c] = gz;
    }
    const int wave = tid >> 6, lane = tid & 63;
    // dL/db: column sums of the FP32 gz, 16 nodes a wavefront, then wavefronts in order.
#pragma unroll
    for (int d = 4; d < 64; d <<= 1)
#pragma unroll
        for (int c = 0; c < 8; ++c) gzs[c] += __shfl_xor(gzs[c], d);
    if (lane < 4)
#pragma unroll
        for (int c = 0; c < 8; ++c) GB[wave * kHid + 8 * q + c] = gzs[c];
    __syncthreads();
    // dL/dX = GZ (64 x 32) * W^T (32 x 64): Bt[f][c] = W[f][c].
    f32x4 dx[4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
        dx[nt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        dx[nt] = mfma_tile(GZ + wave * 16 * kLd32, kLd32, W + nt * 16 * kLd32, kLd32, kHid, dx[nt]);
    }
    // dL/dW = X^T (64 x 64 nodes) * GZ (64 x 32): A = XT rows f, Bt = GZT rows c.
    float* out = gpart + size_t(blockIdx.x) * kMpnnParams + layer_off;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        acc = mfma_tile(XT + wave * 16 * kLd, kLd, GZT + nt * 16 * kLd, kLd, kTile, acc);
#pragma unroll
        for (int j = 0; j < 4; ++j) out[(wave * 16 + 4 * (lane >> 4) + j) * kHid + nt * 16 + (lane & 15)] = acc[j];
    }
    if (tid < kHid) out[2 * kHid * kHid + tid] = GB[tid] + GB[kHid + tid] + GB[2 * kHid + tid] + GB[3 * kHid + tid];
    __syncthreads();
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            G[(wave * 16 + 4 * (lane >> 4) + j) * (2 * kHid + 1) + nt * 16 + (lane & 15)] = dx[nt][j];
    __syncthreads();
    if (i < n) {
        const float* gr = G + il * (2 * kHid + 1);
        float4* o2 = reinterpret_cast<float4*>(gh2 + size_t(i) * kHid + 8 * q);
        o2[0] = make_float4(ghv[0] + gr[8 * q], ghv[1] + gr[8 * q + 1], ghv[2] + gr[8 * q + 2], ghv[3] + gr[8 * q + 3]);
        o2[1] = make_float4(ghv[4] + gr[8 * q + 4], ghv[5] + gr[8 * q + 5], ghv[6] + gr[8 * q + 6],
                            ghv[7] + gr[8 * q + 7]);
        float4* om = reinterpret_cast<float4*>(gm + size_t(i) * kHid + 8 * q);
        om[0] = make_float4(gr[kHid + 8 * q], gr[kHid + 8 * q + 1], gr[kHid + 8 * q + 2], gr[kHid + 8 * q + 3]);
        om[1] = make_float4(gr[kHid + 8 * q + 4], gr[kHid + 8 * q + 5], gr[kHid + 8 * q + 6], gr[kHid + 8 * q + 7]);
    }
}

// gh_out = gh2 + sum_j w_ij gm_j (the mixing is symmetric for symmetric A).
__global__ __launch_bounds__(kBlock) void mix_t_kernel(uint32_t n, const uint32_t* __restrict__ rowp,
                                                      const uint32_t* __restrict__ cols,
                                                      const float* __restrict__ vals, const float* __restrict__ s,
                                                      const float* __restrict__ gm, const float* __restrict__ gh2,
                                                      float* __restrict__ gh_out) {
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    const uint32_t i = t >> 2, q = t & 3;
    if (i >= n) return;
    float acc[8], base[8];
    gather8(i, rowp, cols, vals, s, LoadF8{gm, q}, acc);
    LoadF8{gh2, q}(i, base);
    float4* out = reinterpret_cast<float4*>(gh_out + size_t(i) * kHid + 8 * q);
    out[0] = make_float4(base[0] + acc[0], base[1] + acc[1], base[2] + acc[2], base[3] + acc[3]);
    out[1] = make_float4(base[4] + acc[4], base[5] + acc[5], base[6] + acc[6], base[7] + acc[7]);
}

// Encoder backward: partials of w_in (sum u gz) and b_in (sum gz).
__global__ __launch_bounds__(kBlock) void encode_bwd_kernel(uint32_t n, const float* __restrict__ r,
                                                           const float* __restrict__ s,
                                                           const double* __restrict__ scal,
                                                           const float* __restrict__ gh,
                                                           const uint32_t* __restrict__ mask,
                                                           float* __restrict__ gpart) {
    __shared__ float red[8 * kHid];
    const int tid = threadIdx.x, c = tid & 31, sub = tid >> 5;
    const uint32_t node0 = blockIdx.x * kTile;
    const float inv = inv_rho_of(scal, n);
    float aw = 0.0f, ab = 0.0f;
    for (int il = sub; il < kTile; il += 8) {
        const uint32_t i = node0 + il;
        if (i >= n) continue;
        const float g = ((mask[i] >> c) & 1u) ? gh[size_t(i) * kHid + c] : 0.0f;
        aw += r[i] * s[i] * inv * g;
        ab += g;
    }
    const float tw = tile_channel_sum(aw, red);
    const float tb = tile_channel_sum(ab, red);
    float* out = gpart + size_t(blockIdx.x) * kMpnnParams;
    if (tid < kHid) {
        out[tid] = tw;
        out[kHid + tid] = tb;
    }
}

// out[y][p] = sum of gpart[b][p] over b in [y * per, min((y + 1) * per, rows))
// in row order. The parameter gradient is reduced in two such stages with a
// grouping fixed by the tile count (grad_chunk tiles, then all chunk sums), so
// the sum is deterministic and the reduction has enough parallelism.
__global__ __launch_bounds__(kBlock) void grad_reduce_kernel(uint32_t rows, uint32_t per,
                                                            const float* __restrict__ gpart,
                                                            float* __restrict__ out) {
    const uint32_t p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= uint32_t(kMpnnParams)) return;
    const uint32_t b0 = blockIdx.y * per;
    const uint32_t b1 = std::min(rows, b0 + per);
    float acc = 0.0f;
    for (uint32_t b = b0; b < b1; ++b) acc += gpart[size_t(b) * kMpnnParams + p];
    out[size_t(blockIdx.y) * kMpnnParams + p] = acc;
}

// Adam (Kingma & Ba 2015, Algorithm 1) with bias corrections c1 = 1/(1-b1^t),
// c2 = 1/(1-b2^t).
__global__ __launch_bounds__(kBlock) void adam_kernel(uint32_t count, float* __restrict__ p, float* __restrict__ m,
                                                     float* __restrict__ v, const float* __restrict__ g, float lr,
                                                     float b1, float b2, float eps, float c1, float c2) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= count) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi * c1) / (std::sqrt(vi * c2) + eps);
}

// BF16 copies of the layer weights: w[l][f][c] and wt[l][c][f].
__global__ __launch_bounds__(kBlock) void weights_bf16_kernel(const float* __restrict__ p, uint16_t* __restrict__ w,
                                                             uint16_t* __restrict__ wt) {
    const uint32_t t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= uint32_t(kMpnnLayers * 2 * kHid * kHid)) return;
    const uint32_t l = t / (2 * kHid * kHid), e = t % (2 * kHid * kHid);
    const uint32_t f = e / kHid, c = e % kHid;
    const uint16_t b = f2bf(p[2 * kHid + l * kLayerStride + e]);
    w[l * 2 * kHid * kHid + e] = b;
    wt[l * 2 * kHid * kHid + c * 2 * kHid + f] = b;
}

// out = x + a * y
// partial[block] = sum a_i^2, partial[stride + block] = sum b_i^2 (grid
// stride, kMaxPartBlocks stride).
__global__ __launch_bounds__(kBlock) void sumsq2_kernel(uint32_t n, const float* __restrict__ a,
                                                        const float* __restrict__ b, double* __restrict__ partial) {
    __shared__ double red[4];
    double sa = 0.0, sb = 0.0;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock) {
        sa += double(a[i]) * double(a[i]);
        sb += double(b[i]) * double(b[i]);
    }
    sa = block_sum(sa, red);
    sb = block_sum(sb, red);
    if (threadIdx.x == 0) {
        partial[blockIdx.x] = sa;
        partial[kMaxPartBlocks + blockIdx.x] = sb;
    }
}

__global__ __launch_bounds__(kBlock) void axpy_kernel(uint32_t n, const float* __restrict__ x, float a,
                                                     const float* __restrict__ y, float* __restrict__ out) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) out[i] = x[i] + a * y[i];
}

// ge = -Aw / (e.r); loss = 1/2 v.Av / (e.r).
__global__ __launch_bounds__(kBlock) void loss_grad_kernel(uint32_t n, const float* __restrict__ aw,
                                                          const double* __restrict__ scal, float* __restrict__ ge) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) ge[i] = float(-double(aw[i]) / scal[1]);
}
__global__ void loss_value_kernel(const double* __restrict__ scal, double* __restrict__ loss) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *loss = 0.5 * scal[2] / scal[1];
}

inline uint32_t grid_of(uint64_t n) { return uint32_t((n + kBlock - 1) / kBlock); }
inline uint32_t tiles_of(uint32_t n) { return (n + kTile - 1) / kTile; }

// Tiles a thread of the first reduction stage adds, one after the other; the
// second adds the chunk sums the same way, so the two serial lengths are kept
// alike: the square root of the tile count (2.1M nodes: second stage 63 us,
// 177 with chunks of 64 and 477 with chunks of 24, which suit 67k nodes; the
// first stage 294, 304 and 309). Up to 24 tiles take one stage.
inline uint32_t grad_chunk(uint32_t tiles) {
    uint32_t c = 24;
    while (uint64_t(c) * c < tiles) ++c;
    return c;
}
inline uint32_t grad_chunks(uint32_t tiles) { return (tiles + grad_chunk(tiles) - 1) / grad_chunk(tiles); }
inline uint32_t red_grid(uint32_t n) { return std::min<uint32_t>(grid_of(n), kMaxPartBlocks); }
// Persistent inference grid: 256 CUs x 4 resident workgroups (VGPR-bound).
constexpr uint32_t kWaveGrid = 256 * 4;

}  // namespace

Mpnn::Mpnn(int device) : device_(device) {
    MPNN_HIP(hipSetDevice(device_));
    p_ = mpnn_alloc<float>(kMpnnParams);
    m_ = mpnn_alloc<float>(kMpnnParams);
    v_ = mpnn_alloc<float>(kMpnnParams);
    grad_ = mpnn_alloc<float>(kMpnnParams);
    w_ = mpnn_alloc<uint16_t>(kMpnnLayers * 2 * kHid * kHid);
    wt_ = mpnn_alloc<uint16_t>(kMpnnLayers * 2 * kHid * kHid);
    scal_ = mpnn_alloc<double>(8);
    part_ = mpnn_alloc<double>(2 * kMaxPartBlocks);  // two partial arrays (sumsq2_kernel)
    MPNN_HIP(hipMemset(p_, 0, kMpnnParams * sizeof(float)));
    MPNN_HIP(hipMemset(m_, 0, kMpnnParams * sizeof(float)));
    MPNN_HIP(hipMemset(v_, 0, kMpnnParams * sizeof(float)));
    MPNN_HIP(hipMemset(w_, 0, kMpnnLayers * 2 * kHid * kHid * sizeof(uint16_t)));
    MPNN_HIP(hipMemset(wt_, 0, kMpnnLayers * 2 * kHid * kHid * sizeof(uint16_t)));
}

Mpnn::~Mpnn() {
    (void)hipSetDevice(device_);
    (void)hipDeviceSynchronize();
    mpnn_free(p_);
    mpnn_free(m_);
    mpnn_free(v_);
    mpnn_free(grad_);
    mpnn_free(w_);
    mpnn_free(wt_);
    mpnn_free(scal_);
    mpnn_free(part_);
    mpnn_free(s_);
    for (auto& h : h_) mpnn_free(h);
    for (auto& mk : mask_) mpnn_free(mk);
    mpnn_free(gh_);
    mpnn_free(gh2_);
    mpnn_free(gm_);
    mpnn_free(gpart_);
    for (auto& t : t_) mpnn_free(t);
    free_host_vectors();
    mpnn_free(pairs_r);
    mpnn_free(pairs_e);
}

void Mpnn::ensure(uint32_t n) {
    if (n <= cap_) return;
    MPNN_HIP(hipDeviceSynchronize());
    mpnn_free(s_);
    for (auto& h : h_) mpnn_free(h);
    for (auto& mk : mask_) mpnn_free(mk);
    mpnn_free(gh_);
    mpnn_free(gh2_);
    mpnn_free(gm_);
    mpnn_free(gpart_);
    for (auto& t : t_) mpnn_free(t);
    gpart_cap_ = 0;
    s_ = mpnn_alloc<float>(n);
    for (auto& h : h_) h = mpnn_alloc<uint16_t>(uint64_t(n) * kHid);
    for (auto& t : t_) t = mpnn_alloc<float>(n);
    cap_ = n;
}

const Mpnn::HostVectors& Mpnn::host_vectors(uint32_t n) {
    if (n > host_cap_) {
        MPNN_HIP(hipDeviceSynchronize());
        free_host_vectors();
        for (int k = 0; k < 2; ++k) {
            MPNN_HIP(hipHostMalloc(reinterpret_cast<void**>(&host_.h[k]), n * sizeof(float), hipHostMallocMapped));
            MPNN_HIP(hipHostGetDevicePointer(reinterpret_cast<void**>(&host_.d[k]), host_.h[k], 0));
        }
        MPNN_HIP(hipHostMalloc(reinterpret_cast<void**>(&host_.hgrad), kMpnnParams * sizeof(float),
                               hipHostMallocDefault));
        host_.r = mpnn_alloc<float>(n);
        host_.g = mpnn_alloc<float>(n);
        host_.e = mpnn_alloc<float>(n);
        host_.grad = mpnn_alloc<float>(kMpnnParams);
        host_cap_ = n;
    }
    return host_;
}

void Mpnn::free_host_vectors() {
    host_cap_ = 0;
    for (float* h : {host_.h[0], host_.h[1], host_.hgrad})
        if (h) (void)hipHostFree(h);
    host_.h[0] = host_.h[1] = host_.d[0] = host_.d[1] = host_.hgrad = nullptr;
    for (float** f : {&host_.r, &host_.g, &host_.e, &host_.grad}) mpnn_free(*f);
}

void Mpnn::reserve_pairs(uint32_t n, uint32_t count) {
    if (pairs_n != n || count > pairs_cap) {
        MPNN_HIP(hipDeviceSynchronize());
        mpnn_free(pairs_r);
        mpnn_free(pairs_e);
        pairs_r = mpnn_alloc<float>(uint64_t(n) * count);
        pairs_e = mpnn_alloc<float>(uint64_t(n) * count);
        pairs_cap = count;
    }
    pairs_n = n;
    pairs_count = 0;
}

void Mpnn::refresh_bf16(hipStream_t s) {
    weights_bf16_kernel<<<grid_of(kMpnnLayers * 2 * kHid * kHid), kBlock, 0, s>>>(p_, w_, wt_);
}

void Mpnn::set_params(const float* host) {
    MPNN_HIP(hipMemcpy(p_, host, kMpnnParams * sizeof(float), hipMemcpyHostToDevice));
    MPNN_HIP(hipMemset(m_, 0, kMpnnParams * sizeof(float)));
    MPNN_HIP(hipMemset(v_, 0, kMpnnParams * sizeof(float)));
    step_ = 0;
    refresh_bf16(nullptr);
    MPNN_HIP(hipDeviceSynchronize());
}

void Mpnn::get_params(float* host) const {
    MPNN_HIP(hipDeviceSynchronize());
    MPNN_HIP(hipMemcpy(host, p_, kMpnnParams * sizeof(float), hipMemcpyDeviceToHost));
}

void Mpnn::forward(DeviceAmg& amg, const float* r, float* e, bool keep) {
    const Level0View g = amg.level0();
    const uint32_t n = g.n;
    ensure(n);
    if (keep) {
        for (auto& mk : mask_)
            if (!mk) mk = mpnn_alloc<uint32_t>(cap_);
    }
    hipStream_t st = amg.stream();
    if (keep) last_r_ = r;
    const uint32_t rg = red_grid(n);
    scale_kernel<<<rg, kBlock, 0, st>>>(n, r, g.inv_diag, s_, part_);
    reduce_partials_kernel<<<1, 1024, 0, st>>>(part_, rg, kMaxPartBlocks, scal_, nullptr);
    rho_kernel<<<1, 1, 0, st>>>(scal_, n);
    const uint32_t tiles = tiles_of(n);
    auto wt_of = [&](int l) { return wt_ + l * 2 * kHid * kHid; };
    auto bias_of = [&](int l) { return p_ + 2 * kHid + l * kLayerStride + 2 * kHid * kHid; };
    if (keep) {
        // Training keeps every layer's input and ReLU mask for the backward pass.
        const uint32_t gn = uint32_t((uint64_t(n) * kHid + kBlock - 1) / kBlock);
        encode_kernel<<<gn, kBlock, 0, st>>>(n, r, s_, scal_, p_, h_[0], mask_[0]);
        for (int l = 0; l < kMpnnLayers; ++l)
            layer_kernel<<<tiles, kBlock, 0, st>>>(n, g.rowp, g.cols, g.vals, s_, h_[l], h_[l + 1], wt_of(l),
                                                         bias_of(l), mask_[l + 1]);
        decode_kernel<<<grid_of(uint64_t(n) * 4), kBlock, 0, st>>>(n, h_[kMpnnLayers], s_, scal_, p_, e);
        return;
    }
    // Inference: encoder rows in one vectorised pass, the decoder fused into
    // the last layer, wavefront-independent sub-tiles on a persistent grid (a
    // multiple of the XCD count, at most the workgroups that fit at once).
    static_assert(kMpnnLayers >= 2, "fused first and last layers");
    const uint32_t subs = (n + kSub - 1) / kSub;
    const uint32_t wg = std::max<uint32_t>(
        kXcds, std::min<uint32_t>(kWaveGrid, (subs + 4 * kXcds - 1) / (4 * kXcds) * kXcds));
    encode8_kernel<<<grid_of(uint64_t(n) * 4), kBlock, 0, st>>>(n, r, s_, scal_, p_, h_[0]);
    for (int l = 0; l + 1 < kMpnnLayers; ++l)
        layer_wave_kernel<false><<<wg, kBlock, 0, st>>>(n, g.rowp, g.cols, g.vals, s_, h_[l], h_[l + 1], wt_of(l),
                                                         bias_of(l), scal_, p_, nullptr);
    const int last = kMpnnLayers - 1;
    layer_wave_kernel<true><<<wg, kBlock, 0, st>>>(n, g.rowp, g.cols, g.vals, s_, h_[last], nullptr, wt_of(last),
                                                    bias_of(last), scal_, p_, e);
}

void Mpnn::backward(DeviceAmg& amg, const float* ge, float* grad_dev) {
    const Level0View g = amg.level0();
    const uint32_t n = g.n;
    hipStream_t st = amg.stream();
    const uint32_t tiles = tiles_of(n);
    if (!gh_) {
        gh_ = mpnn_alloc<float>(uint64_t(cap_) * kHid);
        gh2_ = mpnn_alloc<float>(uint64_t(cap_) * kHid);
        gm_ = mpnn_alloc<float>(uint64_t(cap_) * kHid);
    }
    // tile partials plus one row per chunk of the two-stage reduction
    // (never fewer for more tiles)
    const uint32_t cap_tiles = tiles_of(cap_);
    const uint64_t need = (uint64_t(cap_tiles) + grad_chunks(cap_tiles)) * kMpnnParams;
    if (gpart_cap_ < need) {
        MPNN_HIP(hipStreamSynchronize(st));
        mpnn_free(gpart_);
        gpart_ = mpnn_alloc<float>(need);
        gpart_cap_ = need;
    }
    decode_bwd_kernel<<<tiles, kBlock, 0, st>>>(n, ge, s_, scal_, h_[kMpnnLayers], p_, gh_, gpart_);
    for (int l = kMpnnLayers - 1; l >= 0; --l) {
        const uint32_t off = 2 * kHid + l * kLayerStride;
        layer_bwd_kernel<<<tiles, kBlock, 0, st>>>(n, g.rowp, g.cols, g.vals, s_, h_[l], mask_[l + 1],
                                                   w_ + l * 2 * kHid * kHid, gh_, gh2_, gm_, gpart_, off);
        mix_t_kernel<<<grid_of(uint64_t(n) * 4), kBlock, 0, st>>>(n, g.rowp, g.cols, g.vals, s_, gm_, gh2_, gh_);
    }
    encode_bwd_kernel<<<tiles, kBlock, 0, st>>>(n, last_r_, s_, scal_, gh_, mask_[0], gpart_);
    const uint32_t chunk = grad_chunk(tiles), chunks = grad_chunks(tiles);
    if (chunks <= 1) {
        grad_reduce_kernel<<<grid_of(kMpnnParams), kBlock, 0, st>>>(tiles, tiles, gpart_, grad_dev);
    } else {
        // Chunk sums go to the rows after the tiles' rows (the buffer holds
        // tiles + chunks rows, see the allocation above), then are summed.
        float* csum = gpart_ + size_t(tiles) * kMpnnParams;
        grad_reduce_kernel<<<dim3(grid_of(kMpnnParams), chunks), kBlock, 0, st>>>(tiles, chunk, gpart_, csum);
        grad_reduce_kernel<<<grid_of(kMpnnParams), kBlock, 0, st>>>(chunks, chunks, csum, grad_dev);
    }
}

void Mpnn::adam_step(const float* grad_dev, float lr, hipStream_t s) {
    ++step_;
    const double b1 = 0.9, b2 = 0.999;
    const float c1 = float(1.0 / (1.0 - std::pow(b1, double(step_))));
    const float c2 = float(1.0 / (1.0 - std::pow(b2, double(step_))));
    adam_kernel<<<grid_of(kMpnnParams), kBlock, 0, s>>>(kMpnnParams, p_, m_, v_, grad_dev, lr, float(b1), float(b2),
                                                        1e-8f, c1, c2);
    refresh_bf16(s);
}

bool Mpnn::apply(DeviceAmg& amg, const float* r, float* z, std::string& err, double* network_reduction) {
    const uint32_t n = amg.level0().n;
    ensure(n);
    float* e = t_[0];
    float* res = t_[1];
    float* zv = t_[2];
    forward(amg, r, e, false);
    amg.residual32(r, e, res);
    if (network_reduction) {
        const uint32_t rg = red_grid(n);
        sumsq2_kernel<<<rg, kBlock, 0, amg.stream()>>>(n, r, res, part_);
        reduce_partials_kernel<<<2, 1024, 0, amg.stream()>>>(part_, rg, kMaxPartBlocks, scal_ + 5, nullptr);
        double h[2] = {0.0, 0.0};
        MPNN_HIP(hipMemcpyAsync(h, scal_ + 5, sizeof(h), hipMemcpyDeviceToHost, amg.stream()));
        MPNN_HIP(hipStreamSynchronize(amg.stream()));
        *network_reduction = h[0] > 0.0 ? 1.0 - std::sqrt(h[1] / h[0]) : 1.0;
    }
    if (!amg.vcycle32(res, zv)) {
        err = "learned stage: V-cycle failed";
        return false;
    }
    axpy_kernel<<<grid_of(n), kBlock, 0, amg.stream()>>>(n, e, 1.0f, zv, z);
    return true;
}

bool Mpnn::train_step(DeviceAmg& amg, const float* r, const float* e, float lr, double* loss_dev,
                      std::string& err) {
    const uint32_t n = amg.level0().n;
    ensure(n);
    hipStream_t st = amg.stream();
    float* enn = t_[0];
    float* u = t_[1];
    float* a = t_[2];
    float* b = t_[3];
    float* v = t_[4];
    forward(amg, r, enn, true);
    const uint32_t g = grid_of(n), rg = red_grid(n);
    axpy_kernel<<<g, kBlock, 0, st>>>(n, e, -1.0f, enn, u);  // u = e - N(r)
    amg.spmv32(u, a);                                        // a = A u
    if (!amg.vcycle32(a, b)) {                               // b = V A u
        err = "training: V-cycle failed";
        return false;
    }
    axpy_kernel<<<g, kBlock, 0, st>>>(n, u, -1.0f, b, v);    // v = E u
    amg.spmv32(v, a);                                        // a = A v
    dot_partial_kernel<float><<<rg, kBlock, 0, st>>>(n, v, a, part_);
    reduce_partials_kernel<<<1, 1024, 0, st>>>(part_, rg, kMaxPartBlocks, scal_ + 2, nullptr);
    dot_partial_kernel<float><<<rg, kBlock, 0, st>>>(n, e, r, part_);
    reduce_partials_kernel<<<1, 1024, 0, st>>>(part_, rg, kMaxPartBlocks, scal_ + 1, nullptr);
    if (!amg.vcycle32(a, b)) {                               // b = V A v
        err = "training: V-cycle failed";
        return false;
    }
    axpy_kernel<<<g, kBlock, 0, st>>>(n, v, -1.0f, b, u);    // u = E v
    amg.spmv32(u, a);                                        // a = A E E u
    loss_grad_kernel<<<g, kBlock, 0, st>>>(n, a, scal_, b);  // b = dL/dN(r)
    if (loss_dev) loss_value_kernel<<<1, 1, 0, st>>>(scal_, loss_dev);
    backward(amg, b, grad_);
    adam_step(grad_, lr, st);
    return true;
}

// ------------------------------------------------- host-vector entries --

namespace {
struct Scoped {
    void* p = nullptr;
    explicit Scoped(size_t bytes) { MPNN_HIP(hipMalloc(&p, bytes ? bytes : 1)); }
    ~Scoped() { (void)hipFree(p); }
    template <class T>
    T* as() const { return static_cast<T*>(p); }
};
}  // namespace

// The host-vector entries' vectors stay with the object. The network works in
// FP32, so the host converts the caller's doubles into pinned memory that the
// reordering kernels read and write across the bus, and the call waits once, at
// its end. (Pageable copies of the doubles and a device allocation per vector
// and call, which waits for the device when it is freed, took 100 of the 445 us
// of a 67k-node estimate and gradient.)
namespace {
template <class S, class D>
void convert_host(uint32_t n, const S* from, D* to) {
    auto run = [&](uint64_t b, uint64_t e, uint32_t) {
        for (uint64_t i = b; i < e; ++i) to[i] = D(from[i]);
    };
    if (n < (1u << 20)) run(0, n, 0);  // below a millisecond: cheaper than starting threads
    else parallel_chunks(n, 0, run);
}
}  // namespace

void mpnn_forward_host(Mpnn& m, DeviceAmg& amg, const double* r, double* e) {
    const uint32_t n = amg.level0().n;
    hipStream_t st = amg.stream();
    const Mpnn::HostVectors& v = m.host_vectors(n);
    convert_host(n, r, v.h[0]);
    scatter_perm_kernel<float, float><<<grid_of(n), kBlock, 0, st>>>(n, amg.device_perm0(), v.d[0], v.r);
    m.forward(amg, v.r, v.e, false);
    gather_perm_kernel<float, float><<<grid_of(n), kBlock, 0, st>>>(n, amg.device_perm0(), v.e, v.d[1]);
    MPNN_HIP(hipStreamSynchronize(st));
    convert_host(n, v.h[1], e);
}

void mpnn_vjp_host(Mpnn& m, DeviceAmg& amg, const double* r, const double* ge, float* grad) {
    const uint32_t n = amg.level0().n;
    hipStream_t st = amg.stream();
    const Mpnn::HostVectors& v = m.host_vectors(n);
    convert_host(n, r, v.h[0]);
    scatter_perm_kernel<float, float><<<grid_of(n), kBlock, 0, st>>>(n, amg.device_perm0(), v.d[0], v.r);
    m.forward(amg, v.r, v.e, true);
    convert_host(n, ge, v.h[1]);
    scatter_perm_kernel<float, float><<<grid_of(n), kBlock, 0, st>>>(n, amg.device_perm0(), v.d[1], v.g);
    m.backward(amg, v.g, v.grad);
    MPNN_HIP(hipMemcpyAsync(v.hgrad, v.grad, kMpnnParams * sizeof(float), hipMemcpyDeviceToHost, st));
    MPNN_HIP(hipStreamSynchronize(st));
    std::copy_n(v.hgrad, kMpnnParams, grad);
}

void mpnn_adam_host(Mpnn& m, const float* grad, float lr) {
    Scoped gd(kMpnnParams * 4);
    MPNN_HIP(hipMemcpy(gd.p, grad, kMpnnParams * 4, hipMemcpyHostToDevice));
    m.adam_step(gd.as<float>(), lr, nullptr);
    MPNN_HIP(hipDeviceSynchronize());
}

bool mpnn_collect(Mpnn& m, DeviceAmg& amg, const double* b, const std::vector<uint64_t>& iterations, double tol,
                  uint32_t& got, SolveStats& st, std::string& err) {
    const uint32_t n = amg.level0().n;
    m.reserve_pairs(n, uint32_t(iterations.size()));
    Scoped bd(size_t(n) * 8);
    MPNN_HIP(hipMemcpy(bd.p, b, size_t(n) * 8, hipMemcpyHostToDevice));
    const bool ok = amg.collect_pairs(bd.as<double>(), iterations, tol, m.pairs_r, m.pairs_e, got, st, err);
    m.pairs_count = ok ? got : 0;
    return ok;
}

bool mpnn_train(Mpnn& m, DeviceAmg& amg, uint32_t steps, float lr, double* losses, std::string& err) {
    const uint32_t n = amg.level0().n;
    if (m.pairs_count == 0 || m.pairs_n != n) {
        err = "training needs pairs collected on this hierarchy";
        return false;
    }
    Scoped ld(size_t(steps) * 8);
    for (uint32_t k = 0; k < steps; ++k) {
        const size_t off = size_t(k % m.pairs_count) * n;
        if (!m.train_step(amg, m.pairs_r + off, m.pairs_e + off, lr, ld.as<double>() + k, err)) return false;
    }
    MPNN_HIP(hipStreamSynchronize(amg.stream()));
    if (losses) MPNN_HIP(hipMemcpy(losses, ld.p, size_t(steps) * 8, hipMemcpyDeviceToHost));
    return true;
}

}  // namespace cfdxhip
