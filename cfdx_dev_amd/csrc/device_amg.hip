// Device-resident AMG hierarchy, V-cycle, PCG and FGMRES.
//
// Reference anchors:
//   V-cycle / smoother / coarsest   core/linalg/amg_preconditioner.h:2369-2443, :2564-2666
//   PCG (true residual every iter.) core/linalg/cg_solver.h:45-569
//   FGMRES(restart)                 core/linalg/gmres_solver.h:28-600
//
// The hierarchy is stored in a locality ("solve") ordering: reverse
// Cuthill-McKee on level 0, and on every coarser level the order in which
// aggregates first appear in the finer level's ordering. Rows keep the
// reference's entry order (columns are relabelled, not re-sorted), and the
// restriction rows list fine points in the reference's ascending order, so
// each per-row sum is evaluated in the reference's order: the FP64 V-cycle
// is bit-identical to the reference's apply() whatever the ordering.

#include "device_amg.hpp"

#include <algorithm>
#include <atomic>
#include <array>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>
#include <mutex>
#include <numeric>
#include <stdexcept>

#include "coarse_tail.hpp"
#include "device_util.hpp"
#include "kernels.hpp"

namespace cfdxhip {

namespace {

constexpr uint32_t kLastSweeps = 24;  // Jacobi sweeps of a coarsest level without dense factors
constexpr uint32_t kGsStride = 4096;  // partial stride (and grid cap) of the Gram-Schmidt reductions
constexpr uint32_t kScalars = 1024;   // device scalar slots
constexpr uint32_t kRestartMax = 120;  // largest FGMRES restart
constexpr uint32_t kGsCoefSlot = 512; // Gram-Schmidt update coefficients (2 * kRestartMax + 2 slots)
constexpr uint32_t kPcgScalars = 8;   // scalar slots the PCG uses

// Row blocks of the CSR-stream SpMV: consecutive rows up to a target of
// entries (and kMaxRowsPerBlock rows); a row longer than the target is a
// block of its own. The target is the kernel's LDS capacity `cap`, less on
// the small coarse levels so that they keep about 1024 workgroups: a level of
// 42K entries in 11 blocks of 4096 left 245 of the 256 CUs idle.
std::vector<uint2> row_blocks(const std::vector<uint32_t>& rowp, uint32_t cap) {
    const uint32_t n = uint32_t(rowp.size() - 1);
    const uint32_t target = std::clamp<uint32_t>(rowp[n] / 1024, 512, cap);
    std::vector<uint2> b{make_uint2(0, 0)};
    uint32_t row = 0;
    while (row < n) {
        const uint32_t start = row++;
        while (row < n && row - start < uint32_t(kMaxRowsPerBlock) && rowp[row + 1] - rowp[start] <= target) ++row;
        b.push_back(make_uint2(row, rowp[row]));
    }
    return b;
}

// Workgroups (and so dot-product partials) of one SpMV launch in
// precision T.
template <class T>
uint32_t spmv_groups(const DevCsr& M) {
    if (M.nslices) return (M.nslices + kBlock / kSellRows - 1) / (kBlock / kSellRows);
    return sizeof(T) == 8 ? M.nblocks : M.nblocks32;
}

// Padded slots allowed over the CSR entry count before a matrix keeps the
// CSR-stream SpMV, the smallest matrix given a SELL copy, and the longest row
// (one lane sums a row; the column-sorted copy ranks a row's entries in
// O(len^2)).
constexpr double kSellMaxPad = 0.25;
constexpr uint32_t kSellMinRows = 4096;
constexpr uint32_t kSellMaxWidth = 64;

// Slot offsets of the SELL-64 layout of a CSR pattern: slice s holds
// 64 * (longest row of the slice) slots. Returns false (CSR stays the SpMV
// format) when padding exceeds kSellMaxPad, a row is longer than
// kSellMaxWidth or the slots overflow 32 bits.
bool sell_offsets(const std::vector<uint32_t>& rowp, std::vector<uint32_t>& soff) {
    const uint32_t n = uint32_t(rowp.size() - 1);
    if (n < kSellMinRows) return false;
    const uint32_t ns = (n + kSellRows - 1) / kSellRows;
    soff.assign(size_t(ns) + 1, 0);
    uint64_t total = 0;
    for (uint32_t sl = 0; sl < ns; ++sl) {
        const uint32_t r1 = std::min<uint32_t>(n, (sl + 1) * kSellRows);
        uint32_t w = 0;
        for (uint32_t r = sl * kSellRows; r < r1; ++r) w = std::max(w, rowp[r + 1] - rowp[r]);
        if (w > kSellMaxWidth) return false;
        total += uint64_t(w) * kSellRows;
        if (total >= uint64_t(kSellPad)) return false;
        soff[sl + 1] = uint32_t(total);
    }
    return double(total) <= (1.0 + kSellMaxPad) * double(rowp[n]);
}

// Gives D (CSR already on the device) its SELL-64 copy when the pattern
// suits it.
void build_sell(DevCsr& D, const std::vector<uint32_t>& rowp, hipStream_t s) {
    std::vector<uint32_t> soff;
    if (!sell_offsets(rowp, soff)) return;
    D.nslices = uint32_t(soff.size() - 1);
    D.sell_entries = soff.back();
    const uint32_t slots = soff.back();
    D.soff = upload(soff, s);
    if (D.v64) {
        D.scols = dalloc<uint32_t>(slots);
        fill_kernel<uint32_t><<<grid_for(slots), kBlock, 0, s>>>(slots, kSellPad, D.scols);
        sell_scatter_kernel<uint32_t><<<grid_for(D.n), kBlock, 0, s>>>(D.n, D.rowp, D.soff, D.cols, D.scols);
        D.s64 = dalloc<double>(slots);
    }
    if (D.v32) {
        D.scols32 = dalloc<uint32_t>(slots);
        fill_kernel<uint32_t><<<grid_for(slots), kBlock, 0, s>>>(slots, kSellPad, D.scols32);
        sell_scatter_sorted_kernel<uint32_t><<<grid_for(D.n), kBlock, 0, s>>>(D.n, D.rowp, D.cols, D.soff, D.cols,
                                                                                D.scols32);
        D.s32 = dalloc<float>(slots);
    }
    sell_values(D, s, true);
}

// Relabels a CSR: row i -> rp[i], column j -> cp[j], entry order kept.
void permute_csr(const HCsr& A, const std::vector<uint32_t>& rp, const std::vector<uint32_t>& cp,
                 std::vector<uint32_t>& rowp, std::vector<uint32_t>& cols, std::vector<uint32_t>& src) {
    const uint32_t n = A.n;
    rowp.assign(size_t(n) + 1, 0);
    for (uint32_t i = 0; i < n; ++i) rowp[rp[i] + 1] = A.rowp[i + 1] - A.rowp[i];
    for (uint32_t i = 0; i < n; ++i) rowp[i + 1] += rowp[i];
    cols.resize(A.nnz());
    src.resize(A.nnz());
    parallel_for(n, 0, [&](uint64_t i) {
        uint32_t w = rowp[rp[i]];
        for (uint32_t k = A.rowp[i]; k < A.rowp[i + 1]; ++k, ++w) {
            cols[w] = cp[A.cols[k]];
            src[w] = k;
        }
    });
}

}  // namespace

// Fills the SELL values of D from its CSR values (padding slots hold 0, from
// the first fill on).
void sell_values(DevCsr& D, hipStream_t s, bool first) {
    if (!D.nslices) return;
    const uint32_t slots = uint32_t(D.sell_entries);
    if (D.s64) {
        if (first) fill_kernel<double><<<grid_for(slots), kBlock, 0, s>>>(slots, 0.0, D.s64);
        sell_scatter_kernel<double><<<grid_for(D.n), kBlock, 0, s>>>(D.n, D.rowp, D.soff, D.v64, D.s64);
    }
    if (D.s32) {
        if (first) fill_kernel<float><<<grid_for(slots), kBlock, 0, s>>>(slots, 0.0f, D.s32);
        sell_scatter_sorted_kernel<float><<<grid_for(D.n), kBlock, 0, s>>>(D.n, D.rowp, D.cols, D.soff, D.v32,
                                                                             D.s32);
    }
}

DeviceAmg::~DeviceAmg() { release(); }

void DeviceAmg::release() {
    auto free_csr = [](DevCsr& m) {
        dfree(m.rowp);
        dfree(m.cols);
        dfree(m.blocks);
        dfree(m.blocks32);
        dfree(m.v64);
        dfree(m.v32);
        dfree(m.soff);
        dfree(m.scols);
        dfree(m.scols32);
        dfree(m.hvals);
        dfree(m.hbase);
        dfree(m.hcol16);
        dfree(m.hwide);
        m.half_words = 0;
        m.half_bytes = 0;
        dfree(m.s64);
        dfree(m.s32);
        m.nslices = 0;
    };
    for (auto& L : lv_) {
        free_csr(L.A);
        free_csr(L.P);
        free_csr(L.R);
        dfree(L.inv64);
        dfree(L.inv32);
        dfree(L.bt32);
        dfree(L.x64[0]);
        dfree(L.x64[1]);
        dfree(L.b64);
        dfree(L.r64);
        dfree(L.x32[0]);
        dfree(L.x32[1]);
        dfree(L.b32);
        dfree(L.r32);
        dfree(L.d64);
        dfree(L.d32);
    }
    lv_.clear();
    dfree(lu_.piv);
    dfree(lu_.factor);
    dfree(lu_.upper);
    lu_ = DevCoarseLU{};
    dfree(tail_.mem);
    tail_ = Tail{};
    dfree(d_perm0_);
    dfree(partials_);
    dfree(aux_part_);
    dfree(cns_r64_);
    dfree(cns_r32_);
    dfree(scal_);
    if (h_scal_) (void)hipHostFree(h_scal_);
    h_scal_ = nullptr;
    for (auto*& p : work_) dfree(p);
    work_.clear();
    for (auto*& p : work32_) dfree(p);
    work32_.clear();
    for (auto*& p : basis_) dfree(p);
    basis_.clear();
    basis_m_ = 0;
    release_refresh();
}

bool DeviceAmg::build(const HostHierarchy& h, const AmgConfig& cfg, bool reorder, bool want64, bool want32,
                      hipStream_t stream, std::string& err, std::vector<RefreshLevel>* adopt) {
    release();
    stream_ = stream;
    omega_ = h.omega;
    pre_ = cfg.pre;
    post_ = cfg.post;
    has64_ = want64;
    has32_ = want32;
    cns_ = cfg.constant_null_space;
    smoother64_ = cfg.smoother64;
    smoother32_ = cfg.smoother32;
    cheb_degree_ = cfg.cheb_degree;
    cheb_degree_coarse_ = cfg.cheb_degree_coarse;
    cheb_ratio_ = cfg.cheb_ratio;
    if ((smoother64_ == SMOOTHER_CHEBYSHEV || smoother32_ == SMOOTHER_CHEBYSHEV) && !h.lambda_max.empty() &&
        h.lambda_max.size() != h.lv.size()) {
        err = "Chebyshev smoother requires the eigenvalue estimates of every level";
        return false;
    }
    set_chebyshev(h);
    const size_t L = h.lv.size();
    if (L == 0) {
        err = "empty hierarchy";
        return false;
    }
    lv_.resize(L);
    // CFDXHIP_SETUP_TRACE=1 prints the phase times to stderr.
    const bool trace = std::getenv("CFDXHIP_SETUP_TRACE") != nullptr;
    auto tick = std::chrono::steady_clock::now();
    auto phase = [&](const char* what) {
        if (!trace) return;
        HIP_OK(hipStreamSynchronize(stream_));
        const auto now = std::chrono::steady_clock::now();
        std::fprintf(stderr, "[build] %s %.3f s\n", what, std::chrono::duration<double>(now - tick).count());
        tick = now;
    };
    // ---- orderings
    for (size_t l = 0; l < L; ++l) {
        const uint32_t n = h.lv[l].A.n;
        auto& perm = lv_[l].new_of_old;
        const bool last_dense = (l + 1 == L) && n <= 16;
        if (!reorder || last_dense) {
            perm.resize(n);
            std::iota(perm.begin(), perm.end(), 0u);
        } else if (l == 0) {
            perm = rcm_ordering(h.lv[0].A);
        } else {
            const auto& agg = h.lv[l - 1].aggregate;
            const auto& fp = lv_[l - 1].new_of_old;
            std::vector<uint32_t> key(n, std::numeric_limits<uint32_t>::max());
            for (uint32_t i = 0; i < agg.size(); ++i) key[agg[i]] = std::min(key[agg[i]], fp[i]);
            std::vector<uint32_t> order(n);
            std::iota(order.begin(), order.end(), 0u);
            std::sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) {
                return key[a] != key[b] ? key[a] < key[b] : a < b;
            });
            perm.resize(n);
            for (uint32_t p = 0; p < n; ++p) perm[order[p]] = p;
        }
    }
    phase("orderings");
    // ---- matrices
    std::vector<uint32_t> rowp, cols, src;
    std::vector<TailPatterns> small(L);  // A, R, P of the levels the coarse end may take
    auto upload_csr = [&](DevCsr& D, const HCsr& H, const std::vector<uint32_t>& rp,
                          const std::vector<uint32_t>& cp, uint32_t ncols, TailPatterns::Pattern* keep) {
        permute_csr(H, rp, cp, rowp, cols, src);
        if (keep) *keep = {rowp, cols};
        D.n = H.n;
        D.ncols = ncols;
        D.nnz = H.nnz();
        D.rowp = upload(rowp, stream_);
        D.cols = upload(cols, stream_);
        const auto blk = row_blocks(rowp, StreamNnz<double>::value);
        D.nblocks = uint32_t(blk.size() - 1);
        D.blocks = upload(blk, stream_);
        const auto blk32 = row_blocks(rowp, StreamNnz<float>::value);
        D.nblocks32 = uint32_t(blk32.size() - 1);
        D.blocks32 = upload(blk32, stream_);
        std::vector<double> v64(H.nnz());
        for (size_t k = 0; k < v64.size(); ++k) v64[k] = H.vals[src[k]];
        if (has64_) D.v64 = upload(v64, stream_);
        if (has32_) {
            std::vector<float> v32(v64.size());
            for (size_t k = 0; k < v32.size(); ++k) v32[k] = float(v64[k]);
            D.v32 = upload(v32, stream_);
        }
        build_sell(D, rowp, stream_);
        HIP_OK(hipStreamSynchronize(stream_));
    };
    for (size_t l = 0; l < L; ++l) {
        const HostLevel& H = h.lv[l];
        DevLevel& D = lv_[l];
        D.n = H.A.n;
        TailPatterns* keep = D.n <= kTailMaxRows ? &small[l] : nullptr;
        upload_csr(D.A, H.A, D.new_of_old, D.new_of_old, H.A.n, keep ? &keep->m[0] : nullptr);
        std::vector<double> inv(D.n);
        for (uint32_t i = 0; i < D.n; ++i) inv[D.new_of_old[i]] = H.inv_diag[i];
        if (has64_) {
            D.inv64 = upload(inv, stream_);
            D.x64[0] = dalloc<double>(D.n);
            D.x64[1] = dalloc<double>(D.n);
            D.b64 = dalloc<double>(D.n);
            D.r64 = dalloc<double>(D.n);
            if (smoother64_ == SMOOTHER_CHEBYSHEV) D.d64 = dalloc<double>(D.n);
        }
        if (has32_) {
            std::vector<float> inv32(D.n);
            for (uint32_t i = 0; i < D.n; ++i) inv32[i] = float(inv[i]);
            D.inv32 = upload(inv32, stream_);
            D.x32[0] = dalloc<float>(D.n);
            D.x32[1] = dalloc<float>(D.n);
            D.b32 = dalloc<float>(D.n);
            D.r32 = dalloc<float>(D.n);
            if (smoother32_ == SMOOTHER_CHEBYSHEV) D.d32 = dalloc<float>(D.n);
            if (l == 0 && cfg.half_finest && smoother32_ == SMOOTHER_CHEBYSHEV && D.A.nslices) build_half_copy(D);
        }
        HIP_OK(hipStreamSynchronize(stream_));
        if (l + 1 < L) {
            const auto& cperm = lv_[l + 1].new_of_old;
            upload_csr(D.P, H.P, D.new_of_old, cperm, H.P.ncols, keep ? &keep->m[2] : nullptr);
            // R = P^T in the reference order: coarse row c lists fine rows
            // ascending in the reference numbering.
            HCsr R;
            R.n = H.P.ncols;
            R.ncols = H.P.n;
            R.rowp.assign(size_t(R.n) + 1, 0);
            for (uint32_t c : H.P.cols) ++R.rowp[c + 1];
            for (uint32_t c = 0; c < R.n; ++c) R.rowp[c + 1] += R.rowp[c];
            R.cols.resize(H.P.nnz());
            R.vals.resize(H.P.nnz());
            std::vector<uint32_t> cur(R.rowp.begin(), R.rowp.end() - 1);
            for (uint32_t i = 0; i < H.P.n; ++i)
                for (uint32_t q = H.P.rowp[i]; q < H.P.rowp[i + 1]; ++q) {
                    const uint32_t c = H.P.cols[q];
                    R.cols[cur[c]] = i;
                    R.vals[cur[c]] = H.P.vals[q];
                    ++cur[c];
                }
            upload_csr(D.R, R, cperm, D.new_of_old, H.P.n, keep ? &keep->m[1] : nullptr);
        }
    }
    phase("matrices, transfers, SELL copies");
    // ---- coarsest dense LU
    const HostLevel& C = h.lv.back();
    if (C.A.n <= 16) {
        CoarseLU lu;
        lu_.ok = factor_coarsest(C.A, lu, cfg.constant_null_space);
        lu_.n = lu.n;
        if (lu_.ok) {
            lu_.piv = upload(lu.piv, stream_);
            lu_.factor = upload(lu.factor, stream_);
            lu_.upper = upload(lu.upper, stream_);
        }
    }
    build_tail(small);
    const uint32_t n0 = lv_[0].n;
    d_perm0_ = upload(lv_[0].new_of_old, stream_);
    partial_stride_ = std::max<uint64_t>({spmv_groups<double>(lv_[0].A), spmv_groups<float>(lv_[0].A), 4096});
    partials_ = dalloc<double>(std::max<uint64_t>(partial_stride_ * 8, uint64_t(kGsStride) * (2 * kRestartMax + 3)));
    aux_part_ = dalloc<double>(4096);
    if (cns_) {
        if (has64_) cns_r64_ = dalloc<double>(lv_[0].n);
        if (has32_) cns_r32_ = dalloc<float>(lv_[0].n);
    }
    scal_ = dalloc<double>(kScalars);
    HIP_OK(hipMemset(scal_, 0, kScalars * sizeof(double)));
    HIP_OK(hipHostMalloc(reinterpret_cast<void**>(&h_scal_), kScalars * sizeof(double), hipHostMallocMapped));
    HIP_OK(hipHostGetDevicePointer(reinterpret_cast<void**>(&scal_host_), h_scal_, 0));
    std::fill_n(h_scal_, kScalars, 0.0);
    // The last slots but one: the polled tickets.
    h_done_ = reinterpret_cast<unsigned long long*>(h_scal_ + kScalars - 16);
    done_ = reinterpret_cast<unsigned long long*>(scal_host_ + kScalars - 16);
    ticket_ = 0;
    (void)n0;
    HIP_OK(hipStreamSynchronize(stream_));
    phase("coarsest factors, work arrays");
    const bool ok = build_refresh(h, err, adopt);
    phase("refresh state");
    return ok;
}

// ------------------------------------------------------------ V-cycle --

template <class T>
static const T* vals_of(const DevCsr& m);
template <>
const double* vals_of<double>(const DevCsr& m) {
    return m.v64;
}
template <>
const float* vals_of<float>(const DevCsr& m) {
    return m.v32;
}
template <class T>
static T* const* x_of(DevLevel& L);
template <>
double* const* x_of<double>(DevLevel& L) {
    return L.x64;
}
template <>
float* const* x_of<float>(DevLevel& L) {
    return L.x32;
}
template <class T>
static T* b_of(DevLevel& L);
template <>
double* b_of<double>(DevLevel& L) {
    return L.b64;
}
template <>
float* b_of<float>(DevLevel& L) {
    return L.b32;
}
template <class T>
static T* r_of(DevLevel& L);
template <>
double* r_of<double>(DevLevel& L) {
    return L.r64;
}
template <>
float* r_of<float>(DevLevel& L) {
    return L.r32;
}
template <class T>
static const T* inv_of(const DevLevel& L);
template <>
const double* inv_of<double>(const DevLevel& L) {
    return L.inv64;
}
template <>
const float* inv_of<float>(const DevLevel& L) {
    return L.inv32;
}

template <class T>
static const T* sell_vals_of(const DevCsr& m);
template <>
const double* sell_vals_of<double>(const DevCsr& m) {
    return m.s64;
}
template <>
const float* sell_vals_of<float>(const DevCsr& m) {
    return m.s32;
}
template <class T>
static const uint32_t* sell_cols_of(const DevCsr& m);
template <>
const uint32_t* sell_cols_of<double>(const DevCsr& m) {
    return m.scols;
}
template <>
const uint32_t* sell_cols_of<float>(const DevCsr& m) {
    return m.scols32;
}

template <class T, class Init, class Epi>
static void launch_spmv(const DevCsr& M, const T* x, Init init, Epi epi, hipStream_t s) {
    if (M.nslices) {
        const uint32_t g = spmv_groups<T>(M);
        spmv_sell_kernel<T, Init, Epi><<<g, kBlock, 0, s>>>(M.n, M.nslices, g, M.soff, sell_cols_of<T>(M),
                                                            sell_vals_of<T>(M), x, init, epi);
        return;
    }
    const uint32_t nb = sizeof(T) == 8 ? M.nblocks : M.nblocks32;
    if (nb == 0) return;
    spmv_stream_kernel<T, Init, Epi><<<nb, kBlock, 0, s>>>(sizeof(T) == 8 ? M.blocks : M.blocks32, nb, M.rowp, M.cols,
                                                                  vals_of<T>(M), x, init, epi);
}

template <class T>
void DeviceAmg::spmv_jacobi_sweeps(DevLevel& L, const T* b, T*& x, uint32_t sweeps, bool from_zero) {
    T* const* xs = x_of<T>(L);
    const T om = T(omega_);
    uint32_t s = 0;
    if (from_zero && sweeps > 0) {
        jacobi_first_kernel<T><<<grid_for(L.n), kBlock, 0, stream_>>>(L.n, b, inv_of<T>(L), om, x);
        if (cns_) remove_mean<T>(x, L.n);
        s = 1;
    }
    for (; s < sweeps; ++s) {
        T* xn = (x == xs[0]) ? xs[1] : xs[0];
        launch_spmv<T>(L.A, x, InitZero<T>{}, EpiJacobi<T>{b, x, inv_of<T>(L), xn, om}, stream_);
        x = xn;
        if (cns_) remove_mean<T>(x, L.n);
    }
}

void DeviceAmg::set_chebyshev_lambda(const std::vector<double>& lambda_max) {
    cheb_c1_.assign(lambda_max.size(), {});
    cheb_c2_.assign(lambda_max.size(), {});
    cheb_deg_.assign(lambda_max.size(), cheb_degree_);
    for (size_t l = 0; l < lambda_max.size(); ++l) {
        if (l > 0 && cheb_degree_coarse_ > 0) cheb_deg_[l] = cheb_degree_coarse_;
        chebyshev_coefficients(lambda_max[l], cheb_ratio_, cheb_deg_[l], cheb_c1_[l], cheb_c2_[l]);
    }
    upload_tail();
}

template <class T>
static T* d_of(DevLevel& L);
template <>
double* d_of<double>(DevLevel& L) {
    return L.d64;
}
template <>
float* d_of<float>(DevLevel& L) {
    return L.d32;
}

template <class T>
void DeviceAmg::chebyshev_sweeps(uint32_t l, const T* b, T*& x, bool from_zero) {
    DevLevel& L = lv_[l];
    T* const* xs = x_of<T>(L);
    T* d = d_of<T>(L);
    const auto& c1 = cheb_c1_[l];
    const auto& c2 = cheb_c2_[l];
    const uint32_t deg = cheb_deg_[l];
    uint32_t k = 0;
    if (from_zero && deg > 0) {
        cheb_first_kernel<T><<<grid_for(L.n), kBlock, 0, stream_>>>(L.n, b, inv_of<T>(L), T(c2[0]), d, x);
        if (cns_) remove_mean<T>(x, L.n);
        k = 1;
    }
    for (; k < deg; ++k) {
        T* xn = (x == xs[0]) ? xs[1] : xs[0];
        if (k == 0)
            launch_spmv<T>(L.A, x, InitZero<T>{},
                           EpiCheb<T, true>{b, x, inv_of<T>(L), d, xn, T(0), T(c2[0])}, stream_);
        else
            launch_spmv<T>(L.A, x, InitZero<T>{},
                           EpiCheb<T, false>{b, x, inv_of<T>(L), d, xn, T(c1[k]), T(c2[k])}, stream_);
        x = xn;
        if (cns_) remove_mean<T>(x, L.n);
    }
}

// Half-copy word offsets from the slice widths; values from the FP32 copy.
void DeviceAmg::build_half_copy(DevLevel& L) {
    DevCsr& A = L.A;
    std::vector<uint32_t> soff(size_t(A.nslices) + 1);
    HIP_OK(hipMemcpyAsync(soff.data(), A.soff, soff.size() * 4, hipMemcpyDeviceToHost, stream_));
    HIP_OK(hipStreamSynchronize(stream_));
    A.half_words = A.sell_entries / 2;  // 2 B per slot; slices are 64 slots a column, so even
    A.hvals = dalloc<uint32_t>(A.half_words);
    L.bt32 = dalloc<float>(L.n);
    const uint32_t rows = A.nslices * kSellRows;  // every lane of every slice, padding rows included
    sell_half_values_kernel<<<grid_for(rows), kBlock, 0, stream_>>>(L.n, rows, A.soff, A.s32, L.inv32, A.hvals);
    // Compact columns where a slice's slot rows fit int16 offsets.
    const uint64_t slots64 = A.sell_entries / kSellRows;
    A.hbase = dalloc<uint32_t>(slots64);
    A.hcol16 = dalloc<uint32_t>(A.half_words);
    A.hwide = dalloc<uint8_t>(A.nslices);
    fill_kernel<uint8_t><<<grid_for(A.nslices), kBlock, 0, stream_>>>(A.nslices, uint8_t(0), A.hwide);
    sell_half_base_kernel<<<uint32_t((slots64 + kBlock - 1) / kBlock), kBlock, 0, stream_>>>(slots64, A.scols32,
                                                                                            A.hbase);
    sell_half_cols_kernel<<<grid_for(rows), kBlock, 0, stream_>>>(rows, A.soff, A.scols32, A.hbase, A.hcol16,
                                                                  A.hwide);
    std::vector<uint8_t> wide(A.nslices);
    HIP_OK(hipMemcpyAsync(wide.data(), A.hwide, A.nslices, hipMemcpyDeviceToHost, stream_));
    HIP_OK(hipStreamSynchronize(stream_));
    uint64_t bytes = 4 * (uint64_t(A.nslices) + 1) + A.nslices;  // slot offsets, flags
    for (uint32_t s = 0; s < A.nslices; ++s) {
        const uint64_t slots = soff[s + 1] - soff[s];
        bytes += wide[s] ? slots * 2 + slots * 4 : slots * 4 + slots / kSellRows * 4;
    }
    A.half_bytes = bytes;
}

// One launch over the half copy (compact columns where they fit).
template <class Epi>
static void half_step(const DevLevel& L, const float* x, Epi epi, uint32_t g, hipStream_t s) {
    const DevCsr& A = L.A;
    spmv_sell_half_compact_kernel<InitZero<float>, Epi><<<g, kBlock, 0, s>>>(
        L.n, A.nslices, g, A.soff, A.hwide, A.hbase, A.hcol16, A.scols32, A.hvals, x, InitZero<float>{}, epi);
}

// Chebyshev steps of the finest level in an FP32 V-cycle on the half copy:
// the recurrence of chebyshev_sweeps with B = D^-1 A and bt = D^-1 b.
void DeviceAmg::chebyshev_sweeps_half(const float* b, float*& x, bool from_zero) {
    DevLevel& L = lv_[0];
    float* const* xs = x_of<float>(L);
    float* d = L.d32;
    const auto& c1 = cheb_c1_[0];
    const auto& c2 = cheb_c2_[0];
    const uint32_t deg = cheb_deg_[0];
    const uint32_t g = spmv_groups<float>(L.A);
    uint32_t k = 0;
    if (from_zero && deg > 0) {
        cheb_first_half_kernel<<<grid_for(L.n), kBlock, 0, stream_>>>(L.n, b, L.inv32, float(c2[0]), L.bt32, d, x);
        half_bt_for_ = b;
        if (cns_) remove_mean<float>(x, L.n);
        k = 1;
    } else if (deg > 0 && half_bt_for_ != b) {
        scale_by_kernel<<<grid_for(L.n), kBlock, 0, stream_>>>(L.n, b, L.inv32, L.bt32);
        half_bt_for_ = b;
    }
    for (; k < deg; ++k) {
        float* xn = (x == xs[0]) ? xs[1] : xs[0];
        if (k == 0)
            half_step(L, x, EpiChebHalf<true>{L.bt32, x, d, xn, 0.0f, float(c2[0])}, g, stream_);
        else
            half_step(L, x, EpiChebHalf<false>{L.bt32, x, d, xn, float(c1[k]), float(c2[k])}, g, stream_);
        x = xn;
        if (cns_) remove_mean<float>(x, L.n);
    }
    if (!from_zero) half_bt_for_ = nullptr;  // the next V-cycle's b may reuse the buffer
}

template <class T>
void DeviceAmg::smooth(uint32_t l, const T* b, T*& x, uint32_t sweeps, bool from_zero) {
    const uint32_t kind = sizeof(T) == 8 ? smoother64_ : smoother32_;
    if constexpr (sizeof(T) == 4) {
        if (l == 0 && kind == SMOOTHER_CHEBYSHEV && lv_[0].A.hvals) {
            chebyshev_sweeps_half(b, x, from_zero);
            return;
        }
    }
    if (kind == SMOOTHER_CHEBYSHEV)
        chebyshev_sweeps<T>(l, b, x, from_zero);
    else
        spmv_jacobi_sweeps<T>(lv_[l], b, x, sweeps, from_zero);
}

namespace {

// A matrix packed for the coarse end: rows of at most kTailLaneRow entries in
// lanes, longer ones listed. src: the CSR entry of each stored value (lane
// slots, then the long rows' entries).
struct TailPack {
    uint32_t first[kTailWaves], count[kTailWaves];
    std::vector<uint32_t> ctl, src;
    std::vector<uint16_t> cols, lcols;
    std::vector<uint4> groups, lrows;
    uint32_t lane_values = 0;
};

// False when a lane would hold more than kTailBatches.
bool pack_tail(const std::vector<uint32_t>& rowp, const std::vector<uint32_t>& cols, uint32_t ncols, TailPack& t) {
    const uint32_t n = uint32_t(rowp.size() - 1);
    auto len = [&](uint32_t r) { return rowp[r + 1] - rowp[r]; };
    std::vector<uint32_t> rows, longs;
    uint64_t grouped = 0;  // entries of rows that share a group
    for (uint32_t r = 0; r < n; ++r) {
        (len(r) <= kTailLaneRow ? rows : longs).push_back(r);
        if (len(r) > kTailLaneRow && len(r) < kTailChunk / 2) grouped += len(r);
    }
    // Groups of longer rows, about one for each wavefront; a row of half a
    // chunk and more is alone.
    std::stable_sort(longs.begin(), longs.end(), [&](uint32_t a, uint32_t b) { return len(a) > len(b); });
    const uint32_t target = uint32_t(std::min<uint64_t>(kTailChunk, grouped / kTailWaves + kTailLaneRow));
    for (size_t i = 0; i < longs.size();) {
        uint4 g = make_uint4(uint32_t(t.lcols.size()), 0, uint32_t(t.lrows.size()), 0);
        do {
            const uint32_t r = longs[i];
            t.lrows.push_back(make_uint4(r, g.y, g.y + len(r), 0));
            t.lcols.insert(t.lcols.end(), cols.begin() + rowp[r], cols.begin() + rowp[r + 1]);
            g.y += len(r);
            ++g.w;
            ++i;
        } while (i < longs.size() && g.w < 64 && len(longs[i - g.w]) < kTailChunk / 2 &&
                 g.y + len(longs[i]) <= target);
        t.groups.push_back(g);
    }
    auto need = [&](uint32_t r) { return std::max<uint32_t>(1, (len(r) + 7) / 8); };
    std::stable_sort(rows.begin(), rows.end(), [&](uint32_t a, uint32_t b) { return need(a) > need(b); });
    // Longest first over the lanes, back and forth: neighbouring lanes, and
    // so the lanes of a wavefront, end up with like counts.
    std::vector<std::vector<uint32_t>> lane(kTailThreads);
    for (size_t i = 0; i < rows.size(); ++i) {
        const uint32_t pos = uint32_t(i % kTailThreads);
        lane[(i / kTailThreads) % 2 ? kTailThreads - 1 - pos : pos].push_back(rows[i]);
    }
    uint32_t total = 0;
    for (uint32_t w = 0; w < kTailWaves; ++w) {
        uint32_t most = 0;
        for (uint32_t l = 0; l < 64; ++l) {
            uint32_t c = 0;
            for (uint32_t r : lane[w * 64 + l]) c += need(r);
            most = std::max(most, c);
        }
        if (most > kTailBatches) return false;
        t.first[w] = total;
        t.count[w] = most;
        total += most;
    }
    t.lane_values = total * 512;
    t.ctl.assign(size_t(total) * 64, 0);
    t.cols.assign(t.lane_values, uint16_t(ncols));
    t.src.assign(t.lane_values, kTailPad);
    for (uint32_t w = 0; w < kTailWaves; ++w)
        for (uint32_t l = 0; l < 64; ++l) {
            uint32_t at = t.first[w];
            for (uint32_t r : lane[w * 64 + l])
                for (uint32_t q = 0; q < need(r); ++q, ++at) {
                    t.ctl[size_t(at) * 64 + l] = r | (q == 0 ? kTailStart : 0u) | (q + 1 == need(r) ? kTailEnd : 0u);
                    for (uint32_t j = 0; j < 8 && 8 * q + j < len(r); ++j) {
                        const uint32_t k = rowp[r] + 8 * q + j;
                        t.cols[(size_t(at) * 64 + l) * 8 + j] = uint16_t(cols[k]);
                        t.src[((size_t(at) * 4 + j / 2) * 64 + l) * 2 + j % 2] = k;
                    }
                }
        }
    for (const uint4& m : t.lrows)
        for (uint32_t k = rowp[m.x]; k < rowp[m.x + 1]; ++k) t.src.push_back(k);
    return true;
}

}  // namespace

// The levels one workgroup runs: the longest run of levels down to the
// coarsest, at least two, whose matrices fit its lanes and whose vectors fit
// LDS (160 KiB). Mean removals of the constant null space are launches
// between the sweeps: such hierarchies keep the launches.
void DeviceAmg::build_tail(const std::vector<TailPatterns>& small) {
    Tail& t = tail_;
    const uint32_t L = uint32_t(lv_.size());
    t.first = L;
    if (cns_ || !has64_) return;
    constexpr uint32_t kLds = 160 * 1024;
    constexpr uint32_t stage_cells = kTailWaves * kTailChunk;  // the coarsest factors use it too
    static_assert(stage_cells >= 2 * 17 * 17, "coarse_lu_solve's arrays");
    std::vector<std::array<TailPack, 3>> packs;  // A, R, P of the levels, coarsest first
    uint32_t cells = 0;
    while (t.first > 0 && L - t.first < kTailMaxLevels) {
        const DevLevel& D = lv_[t.first - 1];
        const uint32_t more = 2 * D.n + 2;
        if (D.n > kTailMaxRows || D.A.nnz > 4 * uint64_t(kTailThreads) * kTailLaneRow) break;
        if ((cells + more + 3 * (D.n + 1) + stage_cells) * sizeof(double) > kLds) break;
        std::array<TailPack, 3> p;
        bool ok = true;
        for (int m = 0; ok && m < (t.first == L ? 1 : 3); ++m) {
            const DevCsr& M = m == 0 ? D.A : m == 1 ? D.R : D.P;
            const auto& pattern = small[t.first - 1].m[m];
            ok = pack_tail(pattern.rowp, pattern.cols, M.ncols, p[m]);
        }
        if (!ok) break;
        packs.push_back(std::move(p));
        cells += more;
        --t.first;
    }
    if (L - t.first < 2) {
        t.first = L;
        return;
    }
    // One allocation and one copy: the arrays one after the other, then the
    // values, which a kernel gathers, and the level descriptors.
    std::vector<unsigned char> image;
    auto put = [&](const auto& v) {
        const size_t at = (image.size() + 15) & ~size_t(15);
        image.resize(at + v.size() * sizeof(v[0]));
        if (!v.empty()) std::memcpy(image.data() + at, v.data(), v.size() * sizeof(v[0]));
        return at;
    };
    struct Places {
        size_t ctl, cols, groups, lrows, lcols, src, vals;
    };
    std::vector<std::array<Places, 3>> places(L - t.first);
    size_t values = 0;
    auto matrices = [&](uint32_t k) { return t.first + k + 1 == L ? 1 : 3; };
    for (uint32_t k = 0; k < places.size(); ++k)
        for (int m = 0; m < matrices(k); ++m) {
            const TailPack& p = packs[places.size() - 1 - k][m];
            places[k][m] = {put(p.ctl), put(p.cols), put(p.groups), put(p.lrows), put(p.lcols), put(p.src), values};
            values += (p.src.size() + 1) & ~size_t(1);
        }
    const size_t first_value = (image.size() + 15) & ~size_t(15), levels = first_value + values * 8;
    t.mem = dalloc<unsigned char>(levels + places.size() * sizeof(TailLevel));
    HIP_OK(hipMemcpy(t.mem, image.data(), image.size(), hipMemcpyHostToDevice));
    t.host.resize(L - t.first);
    uint32_t at = 0;
    for (uint32_t k = 0; k < t.host.size(); ++k) {
        const uint32_t l = t.first + k;
        DevLevel& D = lv_[l];
        TailLevel& H = t.host[k];
        std::memset(&H, 0, sizeof(H));
        H.inv = D.inv64;
        H.x = at;
        H.b = at + D.n + 1;
        at += 2 * D.n + 2;
        for (int m = 0; m < matrices(k); ++m) {
            const TailPack& p = packs[t.host.size() - 1 - k][m];
            const Places& o = places[k][m];
            const DevCsr& M = m == 0 ? D.A : m == 1 ? D.R : D.P;
            TailMat& X = m == 0 ? H.A : m == 1 ? H.R : H.P;
            X.n = M.n;
            X.ngroups = uint32_t(p.groups.size());
            std::copy(p.first, p.first + kTailWaves, X.first);
            std::copy(p.count, p.count + kTailWaves, X.count);
            X.ctl = reinterpret_cast<const uint32_t*>(t.mem + o.ctl);
            X.cols = reinterpret_cast<const uint4*>(t.mem + o.cols);
            X.groups = reinterpret_cast<const uint4*>(t.mem + o.groups);
            X.lrows = reinterpret_cast<const uint4*>(t.mem + o.lrows);
            X.lcols = reinterpret_cast<const uint16_t*>(t.mem + o.lcols);
            double* v = reinterpret_cast<double*>(t.mem + first_value) + o.vals;
            X.vals = v;
            X.lvals = v + p.lane_values;
            const uint32_t n = uint32_t(p.src.size());
            const uint32_t* src = reinterpret_cast<const uint32_t*>(t.mem + o.src);
            tail_values_kernel<<<grid_for(n), kBlock, 0, stream_>>>(n, src, M.v64, v);
            if (m == 0) t.refill.push_back({l, n, src, v});
        }
    }
    t.cells = at;
    t.stage = at + 3 * (lv_[t.first].n + 1);
    t.lds_bytes = (t.stage + stage_cells) * sizeof(double);
    t.dev = reinterpret_cast<TailLevel*>(t.mem + levels);
    for (const auto kernel : {coarse_tail_kernel<false>, coarse_tail_kernel<true>})
        HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   int(kLds)));
    upload_tail();
}

// The level descriptors, which carry the Chebyshev coefficients.
void DeviceAmg::upload_tail() {
    Tail& t = tail_;
    if (!t.dev) return;
    for (size_t k = 0; k < t.host.size() && t.first + k < cheb_deg_.size(); ++k) {
        const size_t l = t.first + k;
        TailLevel& H = t.host[k];
        H.degree = cheb_deg_[l];
        std::copy(cheb_c1_[l].begin(), cheb_c1_[l].end(), H.c1);
        std::copy(cheb_c2_[l].begin(), cheb_c2_[l].end(), H.c2);
    }
    HIP_OK(hipMemcpyAsync(t.dev, t.host.data(), t.host.size() * sizeof(t.host[0]), hipMemcpyHostToDevice, stream_));
    HIP_OK(hipStreamSynchronize(stream_));
}

void DeviceAmg::refill_tail() {
    for (const auto& f : tail_.refill)
        tail_values_kernel<<<grid_for(f.n), kBlock, 0, stream_>>>(f.n, f.src, lv_[f.level].A.v64, f.dst);
}

template <class T>
bool DeviceAmg::vcycle_t(uint32_t l, const T* b, T*& x) {
    DevLevel& L = lv_[l];
    T* const* xs = x_of<T>(L);
    x = xs[0];
    if constexpr (sizeof(T) == 8) {
        if (l == tail_.first) {
            const bool dense = lv_.back().n <= 16;
            if (dense && !lu_.ok) return false;
            const auto kernel =
                smoother64_ == SMOOTHER_CHEBYSHEV ? coarse_tail_kernel<true> : coarse_tail_kernel<false>;
            kernel<<<1, kTailThreads, tail_.lds_bytes, stream_>>>(
                tail_.dev, uint32_t(tail_.host.size()), tail_.cells, tail_.stage, omega_, pre_, post_, kLastSweeps,
                TailLu{dense ? lu_.n : 0u, lu_.piv, lu_.factor, lu_.upper}, b, x);
            return true;
        }
    }
    if (l + 1 == lv_.size()) {
        if (L.n <= 16) {
            if (!lu_.ok) return false;
            coarse_lu_kernel<T><<<1, 64, 0, stream_>>>(lu_.n, L.n, lu_.piv, lu_.factor, lu_.upper, b, x);
            if (cns_) remove_mean<T>(x, L.n);
            return true;
        }
        spmv_jacobi_sweeps<T>(L, b, x, kLastSweeps, true);
        return true;
    }
    const bool cheb = (sizeof(T) == 8 ? smoother64_ : smoother32_) == SMOOTHER_CHEBYSHEV;
    if (cheb ? cheb_deg_[l] > 0 : pre_ > 0) {
        smooth<T>(l, b, x, pre_, true);
    } else {
        fill_kernel<T><<<grid_for(L.n), kBlock, 0, stream_>>>(L.n, T(0), x);
    }
    T* r = r_of<T>(L);
    launch_spmv<T>(L.A, x, InitZero<T>{}, EpiResidual<T, false>{b, r, nullptr}, stream_);
    DevLevel& Cl = lv_[l + 1];
    T* bc = b_of<T>(Cl);
    launch_spmv<T>(L.R, r, InitZero<T>{}, EpiStore<T>{bc}, stream_);
    if (cns_) remove_mean<T>(bc, Cl.n);
    T* xc = nullptr;
    if (!vcycle_t<T>(l + 1, bc, xc)) return false;
    launch_spmv<T>(L.P, xc, InitFrom<T>{x}, EpiAssign<T>{x}, stream_);
    if (cns_) remove_mean<T>(x, L.n);
    smooth<T>(l, b, x, post_, false);
    return true;
}

template <class T>
void DeviceAmg::remove_mean(T* v, uint32_t n) {
    const uint32_t gs = grid_stride(n);
    sum_partial_kernel<T><<<gs, kBlock, 0, stream_>>>(n, v, aux_part_);
    reduce_partials_kernel<<<1, 1024, 0, stream_>>>(aux_part_, gs, gs, scal_ + 450, nullptr);
    subtract_mean_kernel<T><<<grid_for(n), kBlock, 0, stream_>>>(n, v, scal_ + 450, double(n));
}

void DeviceAmg::project_out(const double* modes, uint32_t count, double* v) {
    const uint32_t n = lv_[0].n;
    const uint32_t gs = grid_stride(n);
    for (uint32_t q = 0; q < count; ++q) {
        const double* m = modes + size_t(q) * n;
        dot_partial_kernel<double><<<gs, kBlock, 0, stream_>>>(n, v, m, aux_part_);
        reduce_partials_kernel<<<1, 1024, 0, stream_>>>(aux_part_, gs, gs, scal_ + 460, nullptr);
        remove_mode_kernel<<<grid_for(n), kBlock, 0, stream_>>>(n, v, m, scal_ + 460);
    }
}

void DeviceAmg::to_solve_order(const double* caller, double* solve, uint32_t count) {
    const uint32_t n = lv_[0].n;
    for (uint32_t q = 0; q < count; ++q)
        scatter_perm_kernel<double, double><<<grid_for(n), kBlock, 0, stream_>>>(n, d_perm0_, caller + size_t(q) * n,
                                                                             solve + size_t(q) * n);
}

// With the constant null space the application works on r minus its mean
// and returns z minus its mean (amg_preconditioner.h:1191-1203).
bool DeviceAmg::vcycle64(const double* r, double* z) {
    double* x = nullptr;
    const uint32_t n = lv_[0].n;
    if (cns_) {
        HIP_OK(hipMemcpyAsync(cns_r64_, r, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
        remove_mean<double>(cns_r64_, n);
        r = cns_r64_;
    }
    if (!vcycle_t<double>(0, r, x)) return false;
    HIP_OK(hipMemcpyAsync(z, x, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
    if (cns_) remove_mean<double>(z, n);
    return true;
}

bool DeviceAmg::vcycle32(const float* r, float* z) {
    float* x = nullptr;
    const uint32_t n = lv_[0].n;
    if (cns_) {
        HIP_OK(hipMemcpyAsync(cns_r32_, r, size_t(n) * 4, hipMemcpyDeviceToDevice, stream_));
        remove_mean<float>(cns_r32_, n);
        r = cns_r32_;
    }
    if (!vcycle_t<float>(0, r, x)) return false;
    HIP_OK(hipMemcpyAsync(z, x, size_t(n) * 4, hipMemcpyDeviceToDevice, stream_));
    if (cns_) remove_mean<float>(z, n);
    return true;
}

// ------------------------------------------------------------ helpers --

// out: a slot of base, whose sums the same slots of h_scal_ receive as well
// (null: they stay on the device).
void DeviceAmg::reduce(const double* partials, uint32_t n, uint32_t count, double* out, uint64_t stride,
                       const double* base) {
    reduce_partials_kernel<<<count, 1024, 0, stream_>>>(partials, n, uint32_t(stride ? stride : partial_stride_), out,
                                                        base ? scal_host_ + (out - base) : nullptr);
}

// Waits for the reduced scalars of slots first..first + count and leaves them at
// the start of h_scal_.
bool DeviceAmg::fetch_scalars(uint32_t count, uint32_t first) {
    HIP_OK(hipStreamSynchronize(stream_));
    if (first) std::copy_n(h_scal_ + first, count, h_scal_);
    return true;
}

// Waits until the first `count` workgroups of the kernel launched last have
// signalled ticket_. Polling pinned memory sees them sooner than a stream synchronisation
// (17 FGMRES steps on 67k rows: 3780 us so, 3890 that way); a launch that takes
// longer than some milliseconds, or fails, is left to the runtime.
void DeviceAmg::await(int count) {
    const volatile unsigned long long* done = h_done_;
    for (int k = 0; k < count; ++k)
        for (uint32_t spin = 0; done[k] != ticket_; ++spin) {
            if (spin > 200000u) {
                HIP_OK(hipStreamSynchronize(stream_));
                break;
            }
            __builtin_ia32_pause();
        }
    std::atomic_thread_fence(std::memory_order_acquire);
}

static double* need_vec(std::vector<double*>& pool, size_t idx, uint32_t n) {
    while (pool.size() <= idx) pool.push_back(dalloc<double>(n));
    return pool[idx];
}
static float* need_vec32(std::vector<float*>& pool, size_t idx, uint32_t n) {
    while (pool.size() <= idx) pool.push_back(dalloc<float>(n));
    return pool[idx];
}

// -------------------------------------------------------- device apply --

namespace {
// An application's residual into the solve order. A non-finite entry marks the
// call (the host's flag, and the call's number for apply_out_kernel) and enters
// as zero, so that it reaches no workspace.
template <class T>
__global__ __launch_bounds__(kBlock) void apply_in_kernel(uint32_t n, const uint32_t* __restrict__ new_of_old,
                                                         const double* __restrict__ r, T* __restrict__ out,
                                                         unsigned long long call,
                                                         unsigned long long* __restrict__ bad,
                                                         int* __restrict__ seen) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    double v = r[i];
    if (!isfinite(v)) {
        *bad = call;
        seen[0] = 1;
        v = 0.0;
    }
    out[new_of_old[i]] = T(v);
}

// The correction out to the caller's order, unless the call is marked.
template <class T>
__global__ __launch_bounds__(kBlock) void apply_out_kernel(uint32_t n, const uint32_t* __restrict__ new_of_old,
                                                          const T* __restrict__ z, double* __restrict__ out,
                                                          unsigned long long call,
                                                          const unsigned long long* __restrict__ bad,
                                                          int* __restrict__ seen) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n || *bad == call) return;
    const double v = double(z[new_of_old[i]]);
    if (!isfinite(v)) seen[1] = 1;
    out[i] = v;
}
}  // namespace

namespace {

__global__ __launch_bounds__(kBlock) void damped_jacobi_action_kernel(uint32_t n, const double* __restrict__ inv,
                                                                      const double* __restrict__ r,
                                                                      double* __restrict__ z) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) z[i] = 0.7 * inv[i] * r[i];
}

}  // namespace

bool DeviceAmg::bounded_action(const double* r, double* z, std::string& err) {
    if (!(max_image_ratio > 0.0)) return true;
    const uint32_t n = lv_[0].n;
    const uint32_t gs = grid_stride(n);
    double* img = need_vec(work_, 15, n);
    // |A z| and |r| (slots 400, 401); hypre_amg.cpp:305-317.
    auto inspect = [&]() {
        launch_spmv<double>(lv_[0].A, z, InitZero<double>{}, EpiStore<double>{img}, stream_);
        dot_partial_kernel<double><<<gs, kBlock, 0, stream_>>>(n, img, img, partials_);
        dot_partial_kernel<double><<<gs, kBlock, 0, stream_>>>(n, r, r, partials_ + partial_stride_);
        reduce(partials_, gs, 2, scal_ + 400, 0, scal_);
        fetch_scalars(2, 400);
        const double an = std::sqrt(h_scal_[0]), rn = std::sqrt(h_scal_[1]);
        if (!std::isfinite(an) || !std::isfinite(rn) || !(rn > 0.0) || !(an > 0.0)) return rn == 0.0 && an == 0.0;
        return an / rn <= max_image_ratio;
    };
    if (inspect()) return true;
    ++bounded_fallbacks;
    damped_jacobi_action_kernel<<<grid_for(n), kBlock, 0, stream_>>>(n, lv_[0].inv64, r, z);
    if (inspect()) return true;
    err = "bounded AMG action and Jacobi fallback both unsafe";
    return false;
}

bool DeviceAmg::apply_caller(const double* r_caller, double* z_caller, bool fp32, std::string& err) {
    const uint32_t n = lv_[0].n;
    const uint32_t g = grid_for(n);
    if (fp32 ? !has32_ : !has64_) {
        err = fp32 ? "no FP32 hierarchy" : "no FP64 hierarchy";
        return false;
    }
    // Non-finite entries are seen on the way in and out, so that a good call
    // waits once; a residual that holds any leaves z as it is. seen: [0] in, [1]
    // out, read by the host; *bad: the number of the last call that was refused.
    int* seen = reinterpret_cast<int*>(h_scal_ + kScalars - 1);
    int* d_seen = reinterpret_cast<int*>(scal_host_ + kScalars - 1);
    unsigned long long* bad = reinterpret_cast<unsigned long long*>(scal_ + kScalars - 1);
    const unsigned long long call = ++apply_calls_;
    const_cast<volatile int*>(seen)[0] = const_cast<volatile int*>(seen)[1] = 0;
    auto flagged = [&](int k) { return const_cast<volatile int*>(seen)[k] != 0; };
    const bool bounded = max_image_ratio > 0.0;
    bool ok;
    if (fp32) {
        float* rs = need_vec32(work32_, 4, n);
        float* zs = need_vec32(work32_, 5, n);
        double* r64 = bounded ? need_vec(work_, 13, n) : nullptr;
        if (bounded) {
            // The bounded test works on the FP64 result: convert, test, reorder.
            apply_in_kernel<double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, r_caller, r64, call, bad, d_seen);
            convert_kernel<double, float><<<g, kBlock, 0, stream_>>>(n, r64, rs);
        } else {
            apply_in_kernel<float><<<g, kBlock, 0, stream_>>>(n, d_perm0_, r_caller, rs, call, bad, d_seen);
        }
        if (cns_) ok = vcycle32(rs, zs);
        else ok = vcycle_t<float>(0, rs, zs);
        if (ok && bounded) {
            double* z64 = need_vec(work_, 14, n);
            convert_kernel<float, double><<<g, kBlock, 0, stream_>>>(n, zs, z64);
            if (!apply_bounded(r64, z64, seen, err)) return false;
            apply_out_kernel<double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, z64, z_caller, call, bad, d_seen);
        } else if (ok) {
            apply_out_kernel<float><<<g, kBlock, 0, stream_>>>(n, d_perm0_, zs, z_caller, call, bad, d_seen);
        }
    } else {
        double* rs = need_vec(work_, 13, n);
        double* zs = need_vec(work_, 14, n);
        apply_in_kernel<double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, r_caller, rs, call, bad, d_seen);
        if (cns_) ok = vcycle64(rs, zs);
        else ok = vcycle_t<double>(0, rs, zs);
        if (ok && bounded && !apply_bounded(rs, zs, seen, err)) return false;
        if (ok) apply_out_kernel<double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, zs, z_caller, call, bad, d_seen);
    }
    HIP_OK(hipStreamSynchronize(stream_));
    if (flagged(0)) {
        err = "non-finite residual";
        return false;
    }
    if (!ok) {
        err = "native AMG V-cycle failed: singular coarsest level";
        return false;
    }
    if (flagged(1)) {
        err = "native AMG V-cycle failed: non-finite correction";
        return false;
    }
    return true;
}

// The bounded test of an application, unless its residual is refused anyway.
bool DeviceAmg::apply_bounded(const double* r, double* z, const int* seen, std::string& err) {
    HIP_OK(hipStreamSynchronize(stream_));
    if (*const_cast<const volatile int*>(seen)) {
        err = "non-finite residual";
        return false;
    }
    return bounded_action(r, z, err);
}

// ---------------------------------------------------------------- PCG --

bool DeviceAmg::pcg(const double* b_caller, double* x_caller, uint64_t max_iter, double tol, SolveStats& st,
                    std::string& err, const double* ns_modes, uint32_t ns_count) {
    if (!has64_) {
        err = "PCG requires the FP64 hierarchy";
        return false;
    }
    PcgWork w;
    for (uint32_t k = 0; k < 7; ++k) w.vec[k] = need_vec(work_, k, lv_[0].n);
    w.partials = partials_;
    w.stride = partial_stride_;
    w.scal = scal_;
    return pcg_in(w, b_caller, x_caller, max_iter, tol, st, err, ns_modes, ns_count);
}

uint64_t DeviceAmg::pcg_work_bytes(uint64_t align) const {
    const auto up = [align](uint64_t b) { return (b + align - 1) / align * align; };
    return 7 * up(uint64_t(n()) * 8) + up(3 * partial_stride_ * 8) + up(kPcgScalars * 8);
}

DeviceAmg::PcgWork DeviceAmg::pcg_work_at(unsigned char* base, uint64_t align) const {
    const auto up = [align](uint64_t b) { return (b + align - 1) / align * align; };
    PcgWork w;
    uint64_t off = 0;
    for (uint32_t k = 0; k < 7; ++k) {
        w.vec[k] = reinterpret_cast<double*>(base + off);
        off += up(uint64_t(n()) * 8);
    }
    w.partials = reinterpret_cast<double*>(base + off);
    w.stride = partial_stride_;
    off += up(3 * partial_stride_ * 8);
    w.scal = reinterpret_cast<double*>(base + off);
    return w;
}

bool DeviceAmg::pcg_in(const PcgWork& w, const double* b_caller, double* x_caller, uint64_t max_iter, double tol,
                       SolveStats& st, std::string& err, const double* ns_modes, uint32_t ns_count) {
    const auto t0 = std::chrono::steady_clock::now();
    if (!has64_) {
        err = "PCG requires the FP64 hierarchy";
        return false;
    }
    st = SolveStats{};
    DevLevel& L0 = lv_[0];
    const uint32_t n = L0.n;
    double* b = w.vec[0];
    double* x = w.vec[1];
    double* r = w.vec[2];
    double* rv = w.vec[3];
    double* z = w.vec[4];
    double* p = w.vec[5];
    double* Ap = w.vec[6];
    double* const scal = w.scal;
    const uint64_t stride = w.stride;
    const uint32_t g = grid_for(n);
    scatter_perm_kernel<double, double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, b_caller, b);
    scatter_perm_kernel<double, double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, x_caller, x);
    const uint32_t nbA = spmv_groups<double>(L0.A);
    const uint32_t gs = grid_stride(n);
    double* P0 = w.partials;
    double* P1 = w.partials + stride;
    double* P2 = w.partials + 2 * stride;
    const bool ns = ns_modes && ns_count > 0;
    // scal slots: 0 |b|^2, 1 |rv|^2, 2 pAp, 3 |r|^2, 4 r.z, 5 |rv|^2 (iteration)
    if (ns) project_out(ns_modes, ns_count, x);
    dot_partial_kernel<double><<<gs, kBlock, 0, stream_>>>(n, b, b, P0);
    launch_spmv<double>(L0.A, x, InitZero<double>{}, EpiResidual<double, true>{b, rv, P1}, stream_);
    reduce(P0, gs, 1, scal + 0, stride, scal);
    if (ns) {
        // the initial residual is projected (cg_solver.h:147-156)
        project_out(ns_modes, ns_count, rv);
        dot_partial_kernel<double><<<gs, kBlock, 0, stream_>>>(n, rv, rv, P1);
        reduce(P1, gs, 1, scal + 1, stride, scal);
    } else {
        reduce(P1, nbA, 1, scal + 1, stride, scal);
    }
    fetch_scalars(2);
    const double bnorm = std::sqrt(h_scal_[0]);
    const double r0 = std::sqrt(h_scal_[1]);
    const double ref = bnorm > 0.0 ? bnorm : r0;
    const double tol_abs = tol * ref;
    auto finish = [&](uint32_t status, uint64_t it, double res) {
        st.status = status;
        st.iterations = it;
        st.residual = res;
        st.residual_relative = ref > 0.0 ? res / ref : 0.0;
        if (on_iterate_) on_iterate_(~uint64_t(0), x);
        gather_perm_kernel<double, double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, x, x_caller);
        HIP_OK(hipStreamSynchronize(stream_));
        st.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
        return true;
    };
    if (on_iterate_) on_iterate_(0, x);
    auto true_residual = [&]() {
        launch_spmv<double>(L0.A, x, InitZero<double>{}, EpiResidual<double, true>{b, rv, P1}, stream_);
        reduce(P1, nbA, 1, scal + 5, stride, scal);
        fetch_scalars(6);
        return std::sqrt(h_scal_[5]);
    };
    st.min_true = std::numeric_limits<double>::infinity();
    if (!std::isfinite(r0) || !std::isfinite(bnorm)) return finish(2, 0, r0);
    if (r0 <= tol_abs) return finish(0, 0, r0);
    HIP_OK(hipMemcpyAsync(r, rv, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
    auto precondition = [&]() {
        ++st.pc_applications;
        if (!vcycle64(r, z) || !bounded_action(r, z, err)) return false;
        if (ns) project_out(ns_modes, ns_count, z);
        return true;
    };
    if (!precondition()) return finish(3, 0, true_residual());
    HIP_OK(hipMemcpyAsync(p, z, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
    dot_partial_kernel<double><<<gs, kBlock, 0, stream_>>>(n, r, z, P0);
    reduce(P0, gs, 1, scal + 4, stride, scal);
    fetch_scalars(5);
    double rsold = h_scal_[4];
    if (!std::isfinite(rsold)) return finish(2, 0, true_residual());
    if (!(rsold > 0.0)) return finish(3, 0, true_residual());
    double last_repl = std::numeric_limits<double>::infinity();
    for (uint64_t it = 1; it <= max_iter; ++it) {
        launch_spmv<double>(L0.A, p, InitZero<double>{}, EpiStoreDot<double>{Ap, p, P0}, stream_);
        if (ns) {
            project_out(ns_modes, ns_count, Ap);
            dot_partial_kernel<double><<<gs, kBlock, 0, stream_>>>(n, p, Ap, P0);
            reduce(P0, gs, 1, scal + 2, stride);
        } else {
            reduce(P0, nbA, 1, scal + 2, stride);
        }
        cg_update_kernel<<<gs, kBlock, 0, stream_>>>(n, rsold, scal + 2, p, Ap, x, r, P2);
        if (ns) {
            project_out(ns_modes, ns_count, x);
            project_out(ns_modes, ns_count, r);
            dot_partial_kernel<double><<<gs, kBlock, 0, stream_>>>(n, r, r, P2);
        }
        if (on_iterate_) on_iterate_(it, x);
        if (!precondition()) {
            const double tr = true_residual();
            return finish(3, it, tr);
        }
        dot_partial_kernel<double><<<gs, kBlock, 0, stream_>>>(n, r, z, P0);
        launch_spmv<double>(L0.A, x, InitZero<double>{}, EpiResidual<double, true>{b, rv, P1}, stream_);
        reduce_list_kernel<<<3, 1024, 0, stream_>>>(PartialList{{P2, P0, P1}, {gs, gs, uint32_t(nbA)}}, scal + 3,
                                                    scal_host_ + 3, done_, ++ticket_);
        await(3);
        const double pAp = h_scal_[2];
        if (!(pAp > 0.0) || !std::isfinite(pAp)) return finish(3, it, true_residual());
        if (!std::isfinite(rsold / pAp)) return finish(2, it, true_residual());
        const double rec2 = h_scal_[3];
        const double rsnew = h_scal_[4];
        const double tr = std::sqrt(h_scal_[5]);
        if (!std::isfinite(rec2) || !std::isfinite(tr)) return finish(2, it, tr);
        if (!std::isfinite(rsnew)) return finish(2, it, tr);
        st.max_true = std::max(st.max_true, tr);
        st.min_true = std::min(st.min_true, tr);
        if (tr <= tol_abs) return finish(0, it, tr);
        const double rec = std::sqrt(rec2);
        const double gap = std::abs(tr - rec);
        const double sc = std::max(tr, rec);
        st.max_gap = std::max(st.max_gap, gap);
        const bool progress = tr < 0.5 * last_repl;
        const bool collapsed = !(rsnew > 0.0);
        const bool adaptive = std::isfinite(rec) && sc > 0.0 && gap > 0.25 * sc && progress;
        const bool repair = collapsed && progress;
        if (collapsed && !repair) return finish(1, it, tr);
        if (adaptive || repair) {
            ++st.replacements;
            if (st.first_replacement == 0) st.first_replacement = it;
            st.last_replacement = it;
            last_repl = tr;
            HIP_OK(hipMemcpyAsync(r, rv, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
            if (ns) project_out(ns_modes, ns_count, r);
            if (!precondition()) return finish(3, it, tr);
            dot_partial_kernel<double><<<gs, kBlock, 0, stream_>>>(n, r, z, P0);
            reduce(P0, gs, 1, scal + 4, stride, scal);
            fetch_scalars(5);
            const double rz = h_scal_[4];
            if (!std::isfinite(rz) || !(rz > 0.0)) return finish(3, it, tr);
            HIP_OK(hipMemcpyAsync(p, z, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
            rsold = rz;
            continue;
        }
        const double beta = rsnew / rsold;
        cg_direction_kernel<<<g, kBlock, 0, stream_>>>(n, beta, z, p);
        if (ns) project_out(ns_modes, ns_count, p);
        rsold = rsnew;
    }
    return finish(1, max_iter, true_residual());
}

// ------------------------------------------------------------- FGMRES --

namespace {

// Arnoldi orthogonalisation: classical Gram-Schmidt with delayed
// reorthogonalisation (DCGS2; Swirydowicz, Langou, Ananthan, Yang and Thomas,
// "Low synchronization Gram-Schmidt and generalized minimal residual
// algorithms", Numer. Linear Algebra Appl. 28 (2021) e2343). Step j reads the
// basis twice: one pass of products, one pass that reorthogonalises the
// previous step's vector u = V_j and orthogonalises w. Basis vectors are
// padded to a multiple of 64 entries with zeros and read as pairs.
constexpr int kGsTile = 12;
inline uint32_t gs_tiles(uint32_t j) { return j == 0 ? 1u : (j + kGsTile - 1) / kGsTile; }

// Products of step j over row pairs (u = V_j):
//   partials[k]        = V_k . w    for k < j,  partials[j]      = u . w
//   partials[j + 1 + k] = V_k . u   for k < j,  partials[2j + 1] = u . u
//   partials[2j + 2]   = w . w
// blockIdx.y takes kGsTile basis vectors; the sums of a workgroup are formed by
// wavefronts, stored, and closed by one thread a sum (one block sum after the
// other, two barriers each, took 10.9 us a step of 67k rows,
// averaged over a cycle of 17; 9.1 us so, most of it the loads).
__global__ __launch_bounds__(kBlock) void gs_dot_kernel(uint32_t npairs, size_t ld, uint32_t j,
                                                       const double* __restrict__ V, const double* __restrict__ w,
                                                       double* __restrict__ partials, uint32_t stride) {
#pragma clang fp contract(off)
    constexpr int kSums = 2 * kGsTile + 3;
    __shared__ double red[kSums][4];
    const double2* up = reinterpret_cast<const double2*>(V + size_t(j) * ld);
    const double2* wp = reinterpret_cast<const double2*>(w);
    const uint32_t k0 = blockIdx.y * kGsTile;
    double aw[kGsTile], au[kGsTile];
#pragma unroll
    for (int t = 0; t < kGsTile; ++t) aw[t] = au[t] = 0.0;
    double uw = 0.0, uu = 0.0, ww = 0.0;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < npairs; i += gridDim.x * kBlock) {
        const double2 wv = wp[i];
        const double2 uv = up[i];
#pragma unroll
        for (int t = 0; t < kGsTile; ++t) {
            if (k0 + t < j) {
                const double2 v = reinterpret_cast<const double2*>(V + size_t(k0 + t) * ld)[i];
                aw[t] += v.x * wv.x;
                aw[t] += v.y * wv.y;
                au[t] += v.x * uv.x;
                au[t] += v.y * uv.y;
            }
        }
        if (k0 == 0) {
            uw += uv.x * wv.x;
            uw += uv.y * wv.y;
            uu += uv.x * uv.x;
            uu += uv.y * uv.y;
            ww += wv.x * wv.x;
            ww += wv.y * wv.y;
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    auto close_wave = [&](int slot, double v) {
        v = wave_sum(v);
        if (lane == 0) red[slot][wave] = v;
    };
#pragma unroll
    for (int t = 0; t < kGsTile; ++t) {
        if (k0 + t < j) {
            close_wave(t, aw[t]);
            close_wave(kGsTile + t, au[t]);
        }
    }
    if (k0 == 0) {
        close_wave(2 * kGsTile, uw);
        close_wave(2 * kGsTile + 1, uu);
        close_wave(2 * kGsTile + 2, ww);
    }
    __syncthreads();
    const int s = threadIdx.x;
    if (s >= kSums) return;
    uint32_t slot;
    if (s < 2 * kGsTile) {
        const uint32_t k = k0 + uint32_t(s % kGsTile);
        if (k >= j) return;
        slot = s < kGsTile ? k : j + 1 + k;
    } else {
        if (k0 != 0) return;
        slot = s == 2 * kGsTile ? j : 2 * j + uint32_t(s - 2 * kGsTile);
    }
    partials[size_t(slot) * stride + blockIdx.x] = ((red[s][0] + red[s][1]) + red[s][2]) + red[s][3];
}

// The coefficients of step j's update from its reduced products d = [V_k . w
// (k <= j), V_k . u (k < j), u . u, w . w], as the host computes them, and a
// last one that is 0 when the host will end the cycle before the update: so the
// update follows at once, and the host reads both steps' results in one wait.
__global__ __launch_bounds__(64) void gs_coef_kernel(uint32_t j, const double* __restrict__ d,
                                                    double* __restrict__ coef) {
#pragma clang fp contract(off)
    const double *c = d, *sv = d + j + 1;
    const double alpha = d[2 * j + 1], an = sqrt(d[2 * j + 2]);
    for (uint32_t k = threadIdx.x; k < j; k += 64) {
        coef[k] = sv[k];
        coef[j + k] = c[k];
    }
    if (threadIdx.x != 0) return;
    double nu = 1.0, hjj = c[0];
    bool go = isfinite(an) && isfinite(alpha);
    if (j > 0) {
        double ss = 0.0, sc = 0.0;
        for (uint32_t k = 0; k < j; ++k) {
            ss += sv[k] * sv[k];
            sc += sv[k] * c[k];
        }
        const double nu2 = alpha - ss;
        go = go && nu2 > 0.5 * alpha;
        nu = sqrt(nu2);
        hjj = (c[j] - sc) / nu;
    }
    coef[2 * j] = nu;
    coef[2 * j + 1] = hjj;
    coef[2 * j + 2] = go ? 1.0 : 0.0;
}

// Update of step j with coef = [s_0..s_{j-1}, c_0..c_{j-1}, nu, h_jj, go]:
//   V_j <- (V_j - sum_k s_k V_k) / nu          (j > 0; V_0 is final)
//   w   <- w - sum_k c_k V_k - h_jj V_j
// and the partials of |w|^2.
constexpr uint32_t kGsCoef = 2 * kRestartMax + 3;
__global__ __launch_bounds__(kBlock) void gs_update_kernel(uint32_t npairs, size_t ld, uint32_t j,
                                                          double* __restrict__ V, const double* __restrict__ coef,
                                                          double* __restrict__ w, double* __restrict__ partials) {
#pragma clang fp contract(off)
    __shared__ double red[4];
    __shared__ double cs[kGsCoef];
    for (uint32_t k = threadIdx.x; k < 2 * j + 3; k += kBlock) cs[k] = coef[k];
    __syncthreads();
    if (cs[2 * j + 2] == 0.0) return;
    const double nu = cs[2 * j], hjj = cs[2 * j + 1];
    double2* up = reinterpret_cast<double2*>(V + size_t(j) * ld);
    double2* wp = reinterpret_cast<double2*>(w);
    double nrm = 0.0;
    for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < npairs; i += gridDim.x * kBlock) {
        double2 u = up[i], x = wp[i];
        for (uint32_t k = 0; k < j; ++k) {
            const double2 v = reinterpret_cast<const double2*>(V + size_t(k) * ld)[i];
            u.x -= cs[k] * v.x;
            u.y -= cs[k] * v.y;
            x.x -= cs[j + k] * v.x;
            x.y -= cs[j + k] * v.y;
        }
        if (j > 0) {
            u.x = u.x / nu;
            u.y = u.y / nu;
            up[i] = u;
        }
        x.x -= hjj * u.x;
        x.y -= hjj * u.y;
        wp[i] = x;
        nrm += x.x * x.x;
        nrm += x.y * x.y;
    }
    const double sum = block_sum(nrm, red);
    if (threadIdx.x == 0) partials[blockIdx.x] = sum;
}

__global__ __launch_bounds__(kBlock) void scale_copy_kernel(uint32_t n, const double* __restrict__ w,
                                                           const double* __restrict__ sc_ptr, double* __restrict__ v) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) v[i] = w[i] / *sc_ptr;
}

__global__ __launch_bounds__(kBlock) void scale_sqrt_copy_kernel(uint32_t n, const double* __restrict__ w,
                                                                const double* __restrict__ sq_ptr,
                                                                double* __restrict__ v) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) v[i] = w[i] / sqrt(*sq_ptr);
}

// x += y
__global__ __launch_bounds__(kBlock) void add_into_kernel(uint32_t n, const double* __restrict__ y,
                                                         double* __restrict__ x) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) x[i] += y[i];
}

// x += sum_j y_j Z_j (y on device)
__global__ __launch_bounds__(kBlock) void basis_axpy_kernel(uint32_t n, size_t ld, uint32_t m,
                                                           const double* __restrict__ Z, const double* __restrict__ y,
                                                           double* __restrict__ x) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    double xi = x[i];
    for (uint32_t j = 0; j < m; ++j) xi += y[j] * Z[size_t(j) * ld + i];
    x[i] = xi;
}

}  // namespace

Level0View DeviceAmg::level0() const {
    Level0View v;
    if (lv_.empty()) return v;
    v.n = lv_[0].n;
    v.rowp = lv_[0].A.rowp;
    v.cols = lv_[0].A.cols;
    v.vals = lv_[0].A.v32;
    v.inv_diag = lv_[0].inv32;
    return v;
}

void DeviceAmg::spmv32(const float* x, float* y) {
    launch_spmv<float>(lv_[0].A, x, InitZero<float>{}, EpiStore<float>{y}, stream_);
}

void DeviceAmg::residual32(const float* b, const float* x, float* r) {
    launch_spmv<float>(lv_[0].A, x, InitZero<float>{}, EpiResidual<float, false>{b, r, nullptr}, stream_);
}

namespace {
// e = xf - xk, r = b - A xk (r given), both to FP32.
__global__ __launch_bounds__(kBlock) void pair_kernel(uint32_t n, const double* __restrict__ xf,
                                                     const double* __restrict__ xk, const double* __restrict__ r,
                                                     float* __restrict__ rout, float* __restrict__ eout) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) {
        eout[i] = float(xf[i] - xk[i]);
        rout[i] = float(r[i]);
    }
}
}  // namespace

bool DeviceAmg::collect_pairs(const double* b_caller, const std::vector<uint64_t>& iterations, double tol,
                              float* r_out, float* e_out, uint32_t& got, SolveStats& st, std::string& err) {
    got = 0;
    if (!has64_ || lv_.empty()) {
        err = "pair collection requires the FP64 hierarchy";
        return false;
    }
    const uint32_t n = lv_[0].n;
    const size_t K = iterations.size();
    std::vector<double*> rec(K, nullptr);
    for (auto& p : rec) p = dalloc<double>(n);
    double* xf = dalloc<double>(n);
    double* xc = dalloc<double>(n);
    std::vector<uint8_t> have(K, 0);
    on_iterate_ = [&](uint64_t it, const double* xs) {
        if (it == ~uint64_t(0)) {
            HIP_OK(hipMemcpyAsync(xf, xs, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
            return;
        }
        for (size_t k = 0; k < K; ++k)
            if (iterations[k] == it) {
                HIP_OK(hipMemcpyAsync(rec[k], xs, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
                have[k] = 1;
            }
    };
    bool ok = false;
    try {
        HIP_OK(hipMemsetAsync(xc, 0, size_t(n) * 8, stream_));
        ok = pcg(b_caller, xc, 100000, tol, st, err);
    } catch (...) {
        on_iterate_ = nullptr;
        for (auto& p : rec) dfree(p);
        dfree(xf);
        dfree(xc);
        throw;
    }
    on_iterate_ = nullptr;
    if (ok && st.status == 0) {
        // b in the solve ordering into xc, then r_k = b - A x_k.
        double* bs = xc;
        scatter_perm_kernel<double, double><<<grid_for(n), kBlock, 0, stream_>>>(n, d_perm0_, b_caller, bs);
        double* rk = need_vec(work_, 2, n);
        for (size_t k = 0; k < K; ++k) {
            if (!have[k]) continue;
            launch_spmv<double>(lv_[0].A, rec[k], InitZero<double>{}, EpiResidual<double, false>{bs, rk, nullptr},
                                stream_);
            pair_kernel<<<grid_for(n), kBlock, 0, stream_>>>(n, xf, rec[k], rk, r_out + size_t(got) * n,
                                                             e_out + size_t(got) * n);
            ++got;
        }
        HIP_OK(hipStreamSynchronize(stream_));
    } else if (ok) {
        err = "pair collection: PCG did not converge (status " + std::to_string(st.status) + ")";
        ok = false;
    }
    for (auto& p : rec) dfree(p);
    dfree(xf);
    dfree(xc);
    return ok;
}

void DeviceAmg::ensure_basis(uint32_t n, uint32_t mcap, size_t ld) {
    (void)n;
    if (basis_m_ >= mcap) return;
    for (auto*& p : basis_) dfree(p);
    basis_.clear();
    basis_.push_back(dalloc<double>(uint64_t(mcap + 1) * ld));
    basis_.push_back(dalloc<double>(uint64_t(mcap) * ld));
    basis_.push_back(dalloc<double>(ld));
    HIP_OK(hipMemsetAsync(basis_[0], 0, uint64_t(mcap + 1) * ld * 8, stream_));
    HIP_OK(hipMemsetAsync(basis_[2], 0, ld * 8, stream_));
    basis_m_ = mcap;
}

bool DeviceAmg::gram_schmidt_seconds(uint32_t j, uint32_t repeat, double& dot_s, double& update_s,
                                     std::string& err) {
    if (lv_.empty() || !lv_[0].A.v64) {
        err = "no FP64 finest level";
        return false;
    }
    const uint32_t n = lv_[0].n;
    if (j + 1 > kRestartMax || j >= n) {
        err = "Arnoldi step out of range";
        return false;
    }
    if (repeat == 0) repeat = 1;
    const uint32_t mcap = std::min<uint32_t>(kRestartMax, n);
    const size_t ld = (size_t(n) + 63) / 64 * 64;
    const uint32_t npairs = uint32_t((uint64_t(n) + 1) / 2);
    ensure_basis(n, mcap, ld);
    double* V = basis_[0];
    double* w = basis_[2];
    const double fill = 1.0 / std::sqrt(double(n));
    for (uint32_t k = 0; k <= j; ++k) fill_kernel<double><<<grid_for(n), kBlock, 0, stream_>>>(n, fill, V + k * ld);
    fill_kernel<double><<<grid_for(n), kBlock, 0, stream_>>>(n, fill, w);
    double* hc = h_scal_ + kGsCoefSlot;
    for (uint32_t k = 0; k < 2 * j; ++k) hc[k] = 1e-3;
    hc[2 * j] = 1.0;
    hc[2 * j + 1] = 1e-3;
    hc[2 * j + 2] = 1.0;
    HIP_OK(hipMemcpyAsync(scal_ + kGsCoefSlot, hc, (2 * j + 3) * sizeof(double), hipMemcpyHostToDevice, stream_));
    const uint32_t gp = std::min<uint32_t>(grid_stride(npairs), kGsStride);
    hipEvent_t e[3];
    for (auto& ev : e) HIP_OK(hipEventCreate(&ev));
    HIP_OK(hipEventRecord(e[0], stream_));
    for (uint32_t r = 0; r < repeat; ++r) {
        gs_dot_kernel<<<dim3(gp, gs_tiles(j)), kBlock, 0, stream_>>>(npairs, ld, j, V, w, partials_, kGsStride);
        reduce(partials_, gp, 2 * j + 3, scal_ + 16, kGsStride, scal_);
    }
    HIP_OK(hipEventRecord(e[1], stream_));
    for (uint32_t r = 0; r < repeat; ++r) {
        gs_update_kernel<<<gp, kBlock, 0, stream_>>>(npairs, ld, j, V, scal_ + kGsCoefSlot, w, partials_);
        reduce(partials_, gp, 1, scal_ + 304, kGsStride, scal_);
    }
    HIP_OK(hipEventRecord(e[2], stream_));
    HIP_OK(hipStreamSynchronize(stream_));
    float ms0 = 0.0f, ms1 = 0.0f;
    HIP_OK(hipEventElapsedTime(&ms0, e[0], e[1]));
    HIP_OK(hipEventElapsedTime(&ms1, e[1], e[2]));
    for (auto& ev : e) (void)hipEventDestroy(ev);
    dot_s = double(ms0) * 1e-3 / repeat;
    update_s = double(ms1) * 1e-3 / repeat;
    return true;
}

bool DeviceAmg::fgmres(const double* b_caller, double* x_caller, int restart, uint64_t max_iter, double tol,
                       bool mixed, SolveStats& st, std::string& err, LearnedControl* learned) {
    const auto t0 = std::chrono::steady_clock::now();
    if (!has64_ && !mixed) {
        err = "FP64 FGMRES preconditioner requires the FP64 hierarchy";
        return false;
    }
    if (mixed && !has32_) {
        err = "mixed-precision FGMRES requires the FP32 hierarchy";
        return false;
    }
    if (!lv_[0].A.v64) {
        err = "FGMRES requires the FP64 finest operator";
        return false;
    }
    st = SolveStats{};
    st.min_true = std::numeric_limits<double>::infinity();
    DevLevel& L0 = lv_[0];
    const uint32_t n = L0.n;
    const int rmin = 10, rmax = int(kRestartMax);
    int cur = std::clamp(restart, rmin, rmax);
    if (n < uint32_t(cur)) cur = int(n);
    // Basis storage: V (rmax+1), Z (rmax) and w, FP64, allocated for the
    // largest restart this solve can reach. Each vector is padded to ld
    // entries; the padding of V and w stays zero (the Gram-Schmidt kernels
    // read row pairs).
    const uint32_t mcap = uint32_t(std::min<int>(rmax, int(n)));
    const size_t ld = (size_t(n) + 63) / 64 * 64;
    const uint32_t npairs = uint32_t((uint64_t(n) + 1) / 2);
    ensure_basis(n, mcap, ld);
    double* V = basis_[0];
    double* Z = basis_[1];
    double* w = basis_[2];
    double* b = need_vec(work_, 0, n);
    double* x = need_vec(work_, 1, n);
    double* r = need_vec(work_, 2, n);
    double* bestx = need_vec(work_, 4, n);
    double* dy = need_vec(work_, 7, n);  // small device buffer for y (n >= m)
    float* r32 = mixed ? need_vec32(work32_, 0, n) : nullptr;
    float* z32 = mixed ? need_vec32(work32_, 1, n) : nullptr;
    const uint32_t g = grid_for(n);
    const uint32_t gs = std::min<uint32_t>(grid_stride(n), kGsStride);
    const uint32_t gp = std::min<uint32_t>(grid_stride(npairs), kGsStride);
    const uint32_t nbA = spmv_groups<double>(L0.A);
    scatter_perm_kernel<double, double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, b_caller, b);
    scatter_perm_kernel<double, double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, x_caller, x);
    double* P0 = partials_;
    dot_partial_kernel<double><<<gs, kBlock, 0, stream_>>>(n, b, b, P0);
    reduce(P0, gs, 1, scal_, 0, scal_);
    fetch_scalars(1);
    const double bn = std::sqrt(h_scal_[0]);
    auto finish = [&](uint32_t status, uint64_t it, double res) {
        st.status = status;
        st.iterations = it;
        st.residual = res;
        st.residual_relative = res / std::max(bn, 1e-300);
        gather_perm_kernel<double, double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, x, x_caller);
        HIP_OK(hipStreamSynchronize(stream_));
        st.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
        return true;
    };
    if (!std::isfinite(bn)) return finish(2, 0, bn);
    const double tolv = tol * bn;
    auto true_res = [&]() {
        launch_spmv<double>(L0.A, x, InitZero<double>{}, EpiResidual<double, true>{b, r, P0}, stream_);
        reduce(P0, nbA, 1, scal_, 0, scal_);
        fetch_scalars(1);
        return std::sqrt(h_scal_[0]);
    };
    if (bn == 0.0) {
        // Homogeneous system (core/linalg/gmres_solver.h:74-135, :180-196):
        // with A x0 != 0, solve A y = -A x0 from y = 0 and certify x0 + y
        // against ||A x0||; with A x0 == 0, x0 is the solution.
        const double ax0 = true_res();  // r = -A x0 (solve ordering)
        auto done = [&](uint32_t status, uint64_t it, double res, double rel) {
            st.status = status;
            st.iterations = it;
            st.residual = res;
            st.residual_relative = rel;
            gather_perm_kernel<double, double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, x, x_caller);
            HIP_OK(hipStreamSynchronize(stream_));
            st.seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
            return true;
        };
        if (!std::isfinite(ax0)) return done(2, 0, ax0, ax0);
        if (ax0 > 0.0) {
            double* rc = need_vec(work_, 10, n);
            double* yc = need_vec(work_, 11, n);
            double* xc = need_vec(work_, 12, n);
            gather_perm_kernel<double, double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, r, rc);
            gather_perm_kernel<double, double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, x, xc);
            fill_kernel<double><<<g, kBlock, 0, stream_>>>(n, 0.0, yc);
            SolveStats sh;
            if (!fgmres(rc, yc, restart, max_iter, tol, mixed, sh, err, learned)) return false;
            add_into_kernel<<<g, kBlock, 0, stream_>>>(n, yc, xc);
            scatter_perm_kernel<double, double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, xc, x);
            fill_kernel<double><<<g, kBlock, 0, stream_>>>(n, 0.0, b);
            const double res = true_res();
            const double rel = res / ax0;
            const bool certified = std::isfinite(res) && std::isfinite(rel) && rel <= tol;
            done(certified ? 0u : (sh.status == 3 ? 3u : 2u), sh.iterations, res, rel);
            st.reorthogonalisations = sh.reorthogonalisations;
            st.pc_applications = sh.pc_applications;
            return true;
        }
        dot_partial_kernel<double><<<gs, kBlock, 0, stream_>>>(n, x, x, P0);
        reduce(P0, gs, 1, scal_, 0, scal_);
        fetch_scalars(1);
        const double ref_scale = std::max({std::sqrt(h_scal_[0]), 1.0, 1e-300});
        return done(ax0 <= tol * ref_scale ? 0u : 2u, 0, ax0, ax0 / ref_scale);
    }
    if (learned && (!mixed || !learned->stage)) {
        err = "the learned stage runs inside mixed-precision FGMRES only";
        return false;
    }
    bool stage_on = learned != nullptr;
    const bool judged = learned && learned->min_reduction >= 0.0;  // negative: the stage stays on
    std::vector<double> hist;  // residual estimate after each iteration (hist[0] = initial)
    auto precondition = [&](const double* v, double* z) {
        ++st.pc_applications;
        if (!mixed) return vcycle64(v, z) && bounded_action(v, z, err);
        convert_kernel<double, float><<<g, kBlock, 0, stream_>>>(n, v, r32);
        if (stage_on) {
            ++learned->applications;
            double red = 1.0;
            if (!learned->stage->apply(*this, r32, z32, err, &red)) return false;
            if (judged && red < learned->min_reduction) {
                // this application's z is kept; the next ones are plain V-cycles
                stage_on = false;
                ++learned->fallbacks;
            }
        } else if (!vcycle32(r32, z32)) {
            return false;
        }
        convert_kernel<float, double><<<g, kBlock, 0, stream_>>>(n, z32, z);
        return bounded_action(v, z, err);
    };
    auto monitor = [&](double est) {
        hist.push_back(est);
        if (!stage_on || !judged || hist.size() <= learned->window) return;
        const size_t k = hist.size() - 1;
        const double a = hist[k - learned->window], b2 = hist[k];
        const double red = a > 0.0 ? 1.0 - std::pow(b2 / a, 1.0 / double(learned->window)) : 0.0;
        if (red < learned->min_reduction) {
            stage_on = false;
            ++learned->fallbacks;
        }
    };
    double beta = true_res();
    if (!std::isfinite(beta)) return finish(2, 0, beta);
    if (beta <= tolv) return finish(0, 0, beta);
    hist.push_back(beta);
    uint64_t its = 0;
    double prev_cycle = beta, best = beta;
    HIP_OK(hipMemcpyAsync(bestx, x, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
    std::vector<double> H, cs, sn, gv, yv;
    while (its < max_iter) {
        const uint32_t m = uint32_t(cur);
        H.assign(size_t(m + 1) * m, 0.0);
        cs.assign(m, 0.0);
        sn.assign(m, 0.0);
        gv.assign(m + 1, 0.0);
        yv.assign(m, 0.0);
        auto Hr = [&](size_t i, size_t j) -> double& { return H[i * m + j]; };
        beta = true_res();
        if (!std::isfinite(beta)) {
            HIP_OK(hipMemcpyAsync(x, bestx, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
            return finish(2, its, best);
        }
        if (beta <= tolv) break;
        // v_0 = r / beta
        h_scal_[0] = beta;
        HIP_OK(hipMemcpyAsync(scal_ + 8, h_scal_, 8, hipMemcpyHostToDevice, stream_));
        scale_copy_kernel<<<g, kBlock, 0, stream_>>>(n, r, scal_ + 8, V);
        gv[0] = beta;
        uint32_t used = 0;
        double est = beta;
        bool brk = false;
        // Column jj of H from its raw entries col[0..jj+1]: earlier rotations,
        // then its own, applied to g.
        auto close_column = [&](uint32_t jj, const std::vector<double>& col) {
            for (uint32_t i = 0; i <= jj + 1; ++i) Hr(i, jj) = col[i];
            for (uint32_t i = 0; i < jj; ++i) {
                const double h0 = Hr(i, jj), h1 = Hr(i + 1, jj);
                Hr(i, jj) = cs[i] * h0 + sn[i] * h1;
                Hr(i + 1, jj) = -sn[i] * h0 + cs[i] * h1;
            }
            const double a = Hr(jj, jj), b2 = Hr(jj + 1, jj);
            const double rho = std::hypot(a, b2);
            if (rho > 0.0) {
                cs[jj] = a / rho;
                sn[jj] = b2 / rho;
                Hr(jj, jj) = rho;
                Hr(jj + 1, jj) = 0.0;
                const double gj = gv[jj], gj1 = gv[jj + 1];
                gv[jj] = cs[jj] * gj + sn[jj] * gj1;
                gv[jj + 1] = -sn[jj] * gj + cs[jj] * gj1;
            }
        };
        // Column j-1 waits for step j: its last entry is |u| nu and the
        // others gain |u| s once u = V_j is reorthogonalised.
        std::vector<double> pend(m + 1, 0.0);
        double pend_norm = 0.0;
        for (uint32_t j = 0; j < m && its < max_iter; ++j) {
            double* vj = V + size_t(j) * ld;
            double* zj = Z + size_t(j) * ld;
            if (!precondition(vj, zj)) {
                HIP_OK(hipMemcpyAsync(x, bestx, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
                return finish(3, its, best);
            }
            // w = A z_j
            launch_spmv<double>(L0.A, zj, InitZero<double>{}, EpiStore<double>{w}, stream_);
            const uint32_t cnt = 2 * j + 3;
            gs_dot_kernel<<<dim3(gp, gs_tiles(j)), kBlock, 0, stream_>>>(npairs, ld, j, V, w, partials_, kGsStride);
            reduce(partials_, gp, cnt, scal_ + 16, kGsStride);
            gs_coef_kernel<<<1, 64, 0, stream_>>>(j, scal_ + 16, scal_ + kGsCoefSlot);
            gs_update_kernel<<<gp, kBlock, 0, stream_>>>(npairs, ld, j, V, scal_ + kGsCoefSlot, w, partials_);
            reduce_step_kernel<<<1, 1024, 0, stream_>>>(partials_, gp, scal_ + 304, scal_host_ + 304, cnt, scal_ + 16,
                                                        scal_host_ + 16, done_, ++ticket_);
            await(1);
            const double* c = h_scal_ + 16;           // V_k . w, k <= j
            const double* sv = h_scal_ + 16 + j + 1;  // V_k . u, k < j
            const double alpha = h_scal_[16 + 2 * j + 1];
            const double an = std::sqrt(h_scal_[16 + 2 * j + 2]);
            if (!std::isfinite(an) || !std::isfinite(alpha)) {
                HIP_OK(hipMemcpyAsync(x, bestx, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
                return finish(2, its, best);
            }
            double nu = 1.0, hjj = c[0];
            if (j > 0) {
                double ss = 0.0, sc = 0.0;
                for (uint32_t k = 0; k < j; ++k) {
                    ss += sv[k] * sv[k];
                    sc += sv[k] * c[k];
                }
                const double nu2 = alpha - ss;
                for (uint32_t k = 0; k < j; ++k) pend[k] += pend_norm * sv[k];
                if (!(nu2 > 0.5 * alpha)) {
                    // u kept less than half its length against V: it is not
                    // reorthogonalised here. Column j-1 closes with the
                    // remaining length and the cycle ends before step j.
                    pend[j] = pend_norm * std::sqrt(std::max(nu2, 0.0));
                    close_column(j - 1, pend);
                    est = std::abs(gv[j]);
                    break;
                }
                ++st.reorthogonalisations;
                nu = std::sqrt(nu2);
                pend[j] = pend_norm * nu;
                close_column(j - 1, pend);
                hjj = (c[j] - sc) / nu;
            }
            const double hn = std::sqrt(h_scal_[304]);
            if (!std::isfinite(hn)) {
                HIP_OK(hipMemcpyAsync(x, bestx, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
                return finish(2, its, best);
            }
            // Column j as far as it is known: |w| stands in for |u| nu.
            for (uint32_t k = 0; k < j; ++k) pend[k] = c[k];
            pend[j] = hjj;
            pend[j + 1] = hn;
            pend_norm = hn;
            const double floor_ = 4096.0 * std::numeric_limits<double>::epsilon() * std::max(an, 1e-300);
            const bool bd = hn <= floor_ && an > 0.0;
            {
                // Residual estimate: column j rotated by the earlier rotations
                // and its own (the last one only scales |g_j|).
                double a = pend[j];
                for (uint32_t i = 0; i < j; ++i) {
                    const double h0 = i == 0 ? pend[0] : a, h1 = pend[i + 1];
                    a = -sn[i] * h0 + cs[i] * h1;
                }
                const double rho = std::hypot(a, hn);
                est = rho > 0.0 ? std::abs(gv[j]) * (hn / rho) : 0.0;
            }
            ++its;
            ++used;
            monitor(est);
            if (bd || est <= tolv || j + 1 == m || its >= max_iter) {
                close_column(j, pend);
                est = std::abs(gv[j + 1]);
                brk = bd;
                break;
            }
            // u = w / |w| is the next step's preconditioner input.
            scale_sqrt_copy_kernel<<<g, kBlock, 0, stream_>>>(n, w, scal_ + 304, V + size_t(j + 1) * ld);
        }
        if (used == 0) break;
        std::fill(yv.begin(), yv.end(), 0.0);
        for (size_t i = used; i-- > 0;) {
            double s = gv[i];
            for (size_t jj = i + 1; jj < used; ++jj) s -= Hr(i, jj) * yv[jj];
            const double dg = Hr(i, i);
            double hs = std::abs(dg);
            for (size_t k = 0; k < used; ++k) hs = std::max(hs, std::abs(Hr(k, i)));
            const double fl = 128.0 * std::numeric_limits<double>::epsilon() * std::max(hs, 1e-300);
            if (std::abs(dg) <= fl) {
                if (std::abs(s) <= fl) {
                    yv[i] = 0.0;
                    continue;
                }
                double br = true_res();
                if (!std::isfinite(br) || best < br) {
                    HIP_OK(hipMemcpyAsync(x, bestx, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
                    br = best;
                }
                return finish(2, its, br);
            }
            yv[i] = s / dg;
        }
        HIP_OK(hipMemcpyAsync(dy, yv.data(), used * 8, hipMemcpyHostToDevice, stream_));
        basis_axpy_kernel<<<g, kBlock, 0, stream_>>>(n, ld, used, Z, dy, x);
        beta = true_res();
        if (!std::isfinite(beta)) {
            HIP_OK(hipMemcpyAsync(x, bestx, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
            return finish(2, its, best);
        }
        st.max_true = std::max(st.max_true, beta);
        st.min_true = std::min(st.min_true, beta);
        if (beta < best) {
            best = beta;
            HIP_OK(hipMemcpyAsync(bestx, x, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
        }
        if (beta <= tolv) return finish(0, its, beta);
        if (brk) {
            if (best < beta) {
                HIP_OK(hipMemcpyAsync(x, bestx, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
                beta = best;
            }
            return finish(2, its, beta);
        }
        const double red = beta / std::max(prev_cycle, 1e-300);
        if (red > 0.1 * 2.0)
            cur = cur > rmax - 5 ? rmax : cur + 5;
        else if (red < 0.1 * 0.5)
            cur = std::max(rmin, cur - 5);
        if (n < uint32_t(cur)) cur = int(n);
        prev_cycle = beta;
    }
    if (best < beta) {
        HIP_OK(hipMemcpyAsync(x, bestx, size_t(n) * 8, hipMemcpyDeviceToDevice, stream_));
        beta = best;
    }
    return finish(beta <= tolv ? 0 : 1, its, beta);
}

// ------------------------------------------------------------ SpMV API --

bool DeviceAmg::level_kernel_seconds(uint32_t level, uint32_t precision, uint32_t kind, uint32_t repeat,
                                     double& sec, std::string& err) {
    if (level >= lv_.size() || precision > 2 || kind > 1) {
        err = "invalid level or kernel";
        return false;
    }
    if (precision == 2 && !lv_[level].A.hvals) {
        err = "no half smoothing copy on this level";
        return false;
    }
    if ((precision == 0 && !has64_) || (precision == 1 && !has32_)) {
        err = "hierarchy precision not built";
        return false;
    }
    DevLevel& L = lv_[level];
    if (repeat == 0) repeat = 1;
    hipEvent_t e0, e1;
    HIP_OK(hipEventCreate(&e0));
    HIP_OK(hipEventCreate(&e1));
    auto run = [&](auto tag) {
        using T = decltype(tag);
        T* const* xs = x_of<T>(L);
        T* b = b_of<T>(L);
        fill_kernel<T><<<grid_for(L.n), kBlock, 0, stream_>>>(L.n, T(1), xs[0]);
        fill_kernel<T><<<grid_for(L.n), kBlock, 0, stream_>>>(L.n, T(1), b);
        HIP_OK(hipEventRecord(e0, stream_));
        for (uint32_t k = 0; k < repeat; ++k) {
            if (kind == 0)
                launch_spmv<T>(L.A, xs[0], InitZero<T>{}, EpiStore<T>{xs[1]}, stream_);
            else
                launch_spmv<T>(L.A, xs[0], InitZero<T>{}, EpiJacobi<T>{b, xs[0], inv_of<T>(L), xs[1], T(omega_)},
                               stream_);
        }
        HIP_OK(hipEventRecord(e1, stream_));
    };
    if (precision == 0) {
        run(double{});
    } else if (precision == 1) {
        run(float{});
    } else {
        // one Chebyshev step on the half copy (kind ignored)
        float* const* xs = x_of<float>(L);
        fill_kernel<float><<<grid_for(L.n), kBlock, 0, stream_>>>(L.n, 1.0f, xs[0]);
        fill_kernel<float><<<grid_for(L.n), kBlock, 0, stream_>>>(L.n, 1.0f, L.bt32);
        fill_kernel<float><<<grid_for(L.n), kBlock, 0, stream_>>>(L.n, 0.0f, L.d32);
        half_bt_for_ = nullptr;
        const uint32_t g = spmv_groups<float>(L.A);
        HIP_OK(hipEventRecord(e0, stream_));
        for (uint32_t k = 0; k < repeat; ++k)
            half_step(L, xs[0], EpiChebHalf<false>{L.bt32, xs[0], L.d32, xs[1], 0.5f, 0.5f}, g, stream_);
        HIP_OK(hipEventRecord(e1, stream_));
    }
    HIP_OK(hipStreamSynchronize(stream_));
    float ms = 0.0f;
    HIP_OK(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    sec = double(ms) * 1e-3 / repeat;
    return true;
}

bool DeviceAmg::spmv_caller(uint32_t precision, const void* x_caller, void* y_caller, uint32_t repeat,
                            double& sec, std::string& err) {
    DevLevel& L0 = lv_[0];
    const uint32_t n = L0.n;
    const uint32_t g = grid_for(n);
    if (repeat == 0) repeat = 1;
    hipEvent_t e0, e1;
    HIP_OK(hipEventCreate(&e0));
    HIP_OK(hipEventCreate(&e1));
    if (precision == 0) {
        if (!has64_) {
            err = "no FP64 hierarchy";
            return false;
        }
        double* xs = need_vec(work_, 5, n);
        double* ys = need_vec(work_, 6, n);
        scatter_perm_kernel<double, double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, (const double*)x_caller, xs);
        HIP_OK(hipEventRecord(e0, stream_));
        for (uint32_t k = 0; k < repeat; ++k)
            launch_spmv<double>(L0.A, xs, InitZero<double>{}, EpiStore<double>{ys}, stream_);
        HIP_OK(hipEventRecord(e1, stream_));
        gather_perm_kernel<double, double><<<g, kBlock, 0, stream_>>>(n, d_perm0_, ys, (double*)y_caller);
    } else {
        if (!has32_) {
            err = "no FP32 hierarchy";
            return false;
        }
        float* xs = need_vec32(work32_, 2, n);
        float* ys = need_vec32(work32_, 3, n);
        scatter_perm_kernel<float, float><<<g, kBlock, 0, stream_>>>(n, d_perm0_, (const float*)x_caller, xs);
        HIP_OK(hipEventRecord(e0, stream_));
        for (uint32_t k = 0; k < repeat; ++k)
            launch_spmv<float>(L0.A, xs, InitZero<float>{}, EpiStore<float>{ys}, stream_);
        HIP_OK(hipEventRecord(e1, stream_));
        gather_perm_kernel<float, float><<<g, kBlock, 0, stream_>>>(n, d_perm0_, ys, (float*)y_caller);
    }
    HIP_OK(hipStreamSynchronize(stream_));
    float ms = 0.0f;
    HIP_OK(hipEventElapsedTime(&ms, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    sec = double(ms) * 1e-3 / double(repeat);
    return true;
}

// ------------------------------------------------- allocation-free PCG --

// Work memory of the allocation-free PCG entry point. Each GPU the library
// runs on holds its own copy of this array until the process ends, and every
// call on that GPU shares it. Host code never passes `scratch` itself to a
// kernel (on the host the name is a stand-in, not a device address): it
// passes the address hipGetSymbolAddress returns for the current device.
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

bool noalloc_scratch(int device, unsigned char*& ptr, std::string& err) {
    static std::mutex mu;
    static std::vector<unsigned char*> per_device;
    std::lock_guard<std::mutex> lock(mu);
    if (device < 0) {
        err = "allocation-free PCG: invalid device ordinal";
        return false;
    }
    if (per_device.size() <= size_t(device)) per_device.resize(size_t(device) + 1, nullptr);
    if (!per_device[size_t(device)]) {
        int current = -1;
        if (hipGetDevice(&current) != hipSuccess || current != device) {
            err = "allocation-free PCG: the handle's device is not current";
            return false;
        }
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            err = std::string("allocation-free PCG: hipGetSymbolAddress failed: ") + hipGetErrorString(e);
            return false;
        }
        per_device[size_t(device)] = static_cast<unsigned char*>(p);
    }
    ptr = per_device[size_t(device)];
    return true;
}

}  // namespace cfdxhip
