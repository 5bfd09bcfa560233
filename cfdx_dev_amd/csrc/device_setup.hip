// Smoothed-aggregation hierarchy construction and numeric refresh
// (update_values with an unchanged pattern) on the device, so a SIMPLE
// corrector that reassembles the pressure matrix on the device never sends
// the hierarchy through the host.
//
// Construction (build_sa_device) follows the host restatement step by step:
// strength graph, its transpose and the symmetrised union, P smoothing,
// Galerkin symbolic and numeric products and the 1e-30 pruning are HIP
// kernels (one thread per row, or per output entry for the products); the
// greedy aggregation is a sequential seed order and runs on the host between
// them. Patterns come out sorted and duplicate-free whatever the order of
// atomically taken cursors, and every value keeps the reference's operation
// order, so the hierarchy is bit-identical to the host construction.
//
// Reference anchors (core/linalg/amg_preconditioner.h unless noted):
//   strength graph                 :1466-1509
//   SA aggregation, P smoothing    :1887-2044
//   Galerkin symbolic / numeric    core/linalg/galerkin_csr_product.h:33-212
//   update_values (transactional)  :245-314
//   build_diagonal                 :1401-1421
//   damping certificate            :1324-1399
//   numeric_into_existing          core/linalg/galerkin_csr_product.h:183-212
//
// Every value is computed as the host restatement computes it (same
// operations, same order, no FMA contraction), so the refreshed hierarchy
// is bit-identical to a host refresh:
//   * AP = A P and C = P^T (AP): one thread per output entry, contributions
//     in the reference's accumulation order (see galerkin_ap_entries_kernel);
//     entries with |c| <= 1e-30 are the pruned ones, and a refresh whose
//     pruned set differs from setup's is rejected;
//   * the inverse diagonal, the Gershgorin bound max_i sum_j |a_ij| /
//     sqrt(d_i d_j) (maxima are exact in any order), and the Lanczos estimate
//     of lambda_max(D^-1 A) with the host's fixed 8192-row block sums.
// All of it runs in the reference ordering on reference-ordered copies of
// the patterns; the committed values are then gathered into the solve-ordered
// CSR and SELL copies the V-cycle reads. Nothing is written to those before
// every check has passed: a failed refresh leaves the previous hierarchy
// untouched.

#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <limits>

#include "device_amg.hpp"
#include "device_util.hpp"

namespace cfdxhip {

namespace {

enum RefreshFlag : int {
    kBadInput = 0,    // non-finite value in the new finest matrix
    kBadDiagonal,     // zero / non-finite diagonal
    kBadProduct,      // non-finite A P or P^T (A P) entry
    kPatternChanged,  // the 1e-30 pruning keeps a different set of entries
    kBadGershgorin,   // the damping certificate cannot be formed
    kFlagCount
};

constexpr uint32_t kLanczosRows = 8192;  // block of the host's deterministic sums

__global__ __launch_bounds__(kBlock) void finite_check_kernel(uint64_t n, const double* __restrict__ v,
                                                              int* __restrict__ flags) {
    const uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i < n && !isfinite(v[i])) flags[kBadInput] = 1;
}

__device__ __forceinline__ uint32_t lower_bound_u32(const uint32_t* __restrict__ a, uint32_t lo, uint32_t hi,
                                                    uint32_t key) {
    while (lo < hi) {
        const uint32_t mid = lo + ((hi - lo) >> 1);
        if (a[mid] < key) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// build_diagonal: inv[i] = 1 / a_ii, failing on |a_ii| <= 1e-30. Columns
// ascend strictly, so the diagonal is found by bisection: a scan of the rows
// that span a coarse level took one lane 340 us.
__global__ __launch_bounds__(kBlock) void inv_diag_kernel(uint32_t n, const uint32_t* __restrict__ rowp,
                                                          const uint32_t* __restrict__ cols,
                                                          const double* __restrict__ vals, double* __restrict__ inv,
                                                          int* __restrict__ flags) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const uint32_t e = rowp[i + 1], k = lower_bound_u32(cols, rowp[i], e, i);
    const double d = k < e && cols[k] == i ? vals[k] : 0.0;
    if (!isfinite(d) || fabs(d) <= 1e-30) {
        flags[kBadDiagonal] = 1;
        inv[i] = 0.0;
        return;
    }
    const double r = 1.0 / d;
    if (!isfinite(r)) flags[kBadDiagonal] = 1;
    inv[i] = r;
}

// acc + the values of the lanes in `m`, in lane order.
__device__ __forceinline__ double add_lanes(double acc, double v, uint64_t m) {
#pragma clang fp contract(off)
    for (; m; m &= m - 1) acc += lane_value(v, __builtin_ctzll(m));
    return acc;
}

// Galerkin numeric products (galerkin_csr_product.h's numeric pass). The
// reference accumulates row by row: for AP, apv[i, c] += a_ij p_jc over A's
// entries (i, j) in row order; for P^T AP, cv[c, k] += p_ic apv[i, k] over the
// fine rows i of the transpose plan in ascending order. A given output entry
// receives its contributions in that same order (each A entry matches at most
// one P entry of the column, each fine row at most one AP entry), so summing
// them per entry from 0 gives the reference's values bit for bit.
//
// AP: one thread per output entry (i, c). Its contributions are the j common
// to A's row i and to the fine rows of c (column c of P), both ascending: the
// thread walks the shorter list and looks each j up in the other. On the
// coarse levels some rows of A span the level: walking those for each of their
// AP entries took 1.24 ms on a level of 4.6K rows. Entries where both lists
// are long are walked by the whole wavefront, 64 candidates at a time, the
// hits added in order.
__global__ __launch_bounds__(kBlock) void galerkin_ap_entries_kernel(
    uint64_t m, const uint32_t* __restrict__ ap_row, const uint32_t* __restrict__ ap_col,
    const uint32_t* __restrict__ arow, const uint32_t* __restrict__ acol, const double* __restrict__ aval,
    const uint32_t* __restrict__ prow, const uint32_t* __restrict__ pcol, const double* __restrict__ pval,
    const uint32_t* __restrict__ t_off, const uint32_t* __restrict__ t_row, const uint32_t* __restrict__ t_pos,
    double* __restrict__ apv, int* __restrict__ flags) {
#pragma clang fp contract(off)
    const uint64_t p = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    const bool live = p < m;
    uint32_t col = 0, a0 = 0, a1 = 0, t0 = 0, t1 = 0;
    if (live) {
        const uint32_t i = ap_row[p];
        col = ap_col[p];
        a0 = arow[i];
        a1 = arow[i + 1];
        t0 = t_off[col];
        t1 = t_off[col + 1];
    }
    // Dependent steps of the two walks: a row's P entries are few, a lookup in
    // A's row halves it.
    const uint32_t by_a = 2 * (a1 - a0), by_t = (t1 - t0) * (33u - __clz(a1 - a0));
    const bool walk_t = by_t < by_a;
    const bool heavy = (walk_t ? by_t : by_a) > 512;
    double acc = 0.0;
    if (live && !heavy) {
        if (walk_t) {
            for (uint32_t t = t0; t < t1; ++t) {
                const uint32_t j = t_row[t], k = lower_bound_u32(acol, a0, a1, j);
                if (k < a1 && acol[k] == j) acc += aval[k] * pval[prow[j] + t_pos[t]];
            }
        } else {
            for (uint32_t k = a0; k < a1; ++k) {
                const uint32_t j = acol[k], e = prow[j + 1];
                const uint32_t q = lower_bound_u32(pcol, prow[j], e, col);
                if (q < e && pcol[q] == col) acc += aval[k] * pval[q];
            }
        }
    }
    const uint32_t lane = threadIdx.x & 63u;
    for (uint64_t hm = __ballot(live && heavy); hm; hm &= hm - 1) {
        const int src = __builtin_ctzll(hm);
        const uint32_t c = __builtin_amdgcn_readlane(col, src), b0 = __builtin_amdgcn_readlane(a0, src),
                       b1 = __builtin_amdgcn_readlane(a1, src), u0 = __builtin_amdgcn_readlane(t0, src),
                       u1 = __builtin_amdgcn_readlane(t1, src);
        const bool wt = __builtin_amdgcn_readlane(uint32_t(walk_t), src) != 0;
        double s = 0.0;
        for (uint32_t base = wt ? u0 : b0, end = wt ? u1 : b1; base < end; base += 64) {
            const uint32_t x = base + lane;
            bool hit = false;
            double v = 0.0;
            if (x < end) {
                if (wt) {
                    const uint32_t j = t_row[x], k = lower_bound_u32(acol, b0, b1, j);
                    hit = k < b1 && acol[k] == j;
                    if (hit) v = aval[k] * pval[prow[j] + t_pos[x]];
                } else {
                    const uint32_t j = acol[x], e = prow[j + 1];
                    const uint32_t q = lower_bound_u32(pcol, prow[j], e, c);
                    hit = q < e && pcol[q] == c;
                    if (hit) v = aval[x] * pval[q];
                }
            }
            s = add_lanes(s, v, __ballot(hit));
        }
        if (int(lane) == src) acc = s;
    }
    if (live) {
        apv[p] = acc;
        if (!isfinite(acc)) flags[kBadProduct] = 1;
    }
}

// P^T (AP), three kinds of coarse row by their length and their count of fine
// rows. Each kind takes the fine rows in order and adds their AP entries
// (distinct columns) into the row's slots in LDS, so each slot receives its
// terms in the reference's order.
//   * up to kLightRow entries and kLightFine fine rows (nearly all): 16 lanes,
//     sixteen rows a workgroup;
//   * up to kTileCols entries and kMidFine fine rows: a wavefront;
//   * the rest, rows that span a coarse level: a workgroup for every
//     kTileCols columns, 32 fine rows at a time. Each wavefront writes the
//     products of two of them into a 32 x kTileCols table and marks them in
//     the columns' masks; then a thread a column adds the marked ones in order.
//     One wavefront a row, fine row after fine row, took 7 ms on a level of 2K
//     coarse rows.
constexpr uint32_t kLightRow = 64, kLightFine = 24, kTileCols = 512, kMidFine = 64, kTileFine = 32;
constexpr uint32_t kTileBytes = kTileFine * kTileCols * 8 + kTileCols * 16 + 2 * kTileFine * 16;

__device__ __forceinline__ int c_row_kind(uint32_t len, uint32_t fine) {
    return len <= kLightRow && fine <= kLightFine ? 0 : len <= kTileCols && fine <= kMidFine ? 1 : 2;
}

// Counts (null lists) or lists the mid rows and the heavy rows' tiles; their
// order does not matter.
__global__ __launch_bounds__(kBlock) void c_row_kinds_kernel(uint32_t nc, const uint32_t* __restrict__ c_off,
                                                             const uint32_t* __restrict__ t_off,
                                                             uint32_t* __restrict__ cnt, uint32_t* __restrict__ mid,
                                                             uint2* __restrict__ heavy) {
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= nc) return;
    const uint32_t len = c_off[c + 1] - c_off[c];
    const int kind = c_row_kind(len, t_off[c + 1] - t_off[c]);
    if (kind == 1) {
        const uint32_t at = atomicAdd(&cnt[0], 1u);
        if (mid) mid[at] = c;
    } else if (kind == 2) {
        const uint32_t tiles = max(1u, (len + kTileCols - 1) / kTileCols), at = atomicAdd(&cnt[1], tiles);
        if (heavy)
            for (uint32_t t = 0; t < tiles; ++t) heavy[at + t] = make_uint2(c, t);
    }
}

struct CProduct {
    const uint32_t *t_off, *t_row, *t_pos, *prow;
    const double* pval;
    const uint32_t *ap_off, *ap_col;
    const double* apv;
    const uint32_t *c_off, *c_col;
    double* cv;
    const uint8_t* keep_mask;  // null at setup
    int* flags;
};

// Position of col in the ascending cols[0, n) (LDS), or n.
__device__ __forceinline__ uint32_t find_col(const uint32_t* cols, uint32_t n, uint32_t col) {
    uint32_t lo = 0, hi = n;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (cols[mid] < col) lo = mid + 1;
        else hi = mid;
    }
    return lo < n && cols[lo] == col ? lo : n;
}

__device__ __forceinline__ void store_c(const CProduct& g, uint32_t at, double v) {
    g.cv[at] = v;
    if (!isfinite(v)) g.flags[kBadProduct] = 1;
    if (g.keep_mask && (fabs(v) > 1e-30) != (g.keep_mask[at] != 0)) g.flags[kPatternChanged] = 1;
}

// kLanes lanes a row of at most kLen entries; rows from `list`, or the light
// ones of all rows.
template <uint32_t kLanes, uint32_t kLen>
__global__ __launch_bounds__(kBlock) void galerkin_c_rows_kernel(uint32_t count, const uint32_t* __restrict__ list,
                                                                 CProduct g) {
#pragma clang fp contract(off)
    constexpr uint32_t kGroups = kBlock / kLanes;
    __shared__ double accs[kGroups][kLen];
    __shared__ uint32_t colss[kGroups][kLen];
    const uint32_t grp = threadIdx.x / kLanes, lane = threadIdx.x % kLanes;
    const uint32_t q = blockIdx.x * kGroups + grp;
    if (q >= count) return;
    const uint32_t c = list ? list[q] : q;
    const uint32_t rb = g.c_off[c], len = g.c_off[c + 1] - rb, t0 = g.t_off[c], t1 = g.t_off[c + 1];
    if (!list && c_row_kind(len, t1 - t0) != 0) return;
    double* acc = accs[grp];
    uint32_t* cols = colss[grp];
    for (uint32_t k = lane; k < len; k += kLanes) {
        acc[k] = 0.0;
        cols[k] = g.c_col[rb + k];
    }
    wave_fence();
    bool missing = false;
    // The next fine row's offsets are loaded while the current one is added.
    uint32_t p0 = 0, p1 = 0;
    double wgt = 0.0;
    auto fetch = [&](uint32_t t) {
        const uint32_t i = g.t_row[t];
        p0 = g.ap_off[i];
        p1 = g.ap_off[i + 1];
        wgt = g.pval[g.prow[i] + g.t_pos[t]];
    };
    if (t0 < t1) fetch(t0);
    for (uint32_t t = t0; t < t1; ++t) {
        const uint32_t b = p0, e = p1;
        const double w = wgt;
        if (t + 1 < t1) fetch(t + 1);
        for (uint32_t p = b + lane; p < e; p += kLanes) {
            const double v = g.apv[p];
            const uint32_t pos = find_col(cols, len, g.ap_col[p]);
            if (pos < len) acc[pos] += w * v;
            else missing = true;
        }
        wave_fence();
    }
    if (missing) g.flags[kBadProduct] = 1;
    for (uint32_t k = lane; k < len; k += kLanes) store_c(g, rb + k, acc[k]);
}

__global__ __launch_bounds__(1024) void galerkin_c_tiles_kernel(const uint2* __restrict__ list, CProduct g) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) unsigned char tile_lds[];
    double* table = reinterpret_cast<double*>(tile_lds);  // [fine][column]
    double* acc = table + kTileFine * kTileCols;
    uint32_t* cols = reinterpret_cast<uint32_t*>(acc + kTileCols);
    uint32_t* mask = cols + kTileCols;
    uint4* meta = reinterpret_cast<uint4*>(mask + kTileCols);  // two sets: AP row begin, end, weight
    const uint32_t tid = threadIdx.x, wave = tid >> 6, lane = tid & 63u;
    const uint32_t c = list[blockIdx.x].x, tile = list[blockIdx.x].y;
    const uint32_t row0 = g.c_off[c], row1 = g.c_off[c + 1];
    const uint32_t rb = row0 + tile * kTileCols, len = min(row1 - rb, kTileCols);
    const uint32_t t0 = g.t_off[c], t1 = g.t_off[c + 1];
    if (tid < len) {
        cols[tid] = g.c_col[rb + tid];
        acc[tid] = 0.0;
        mask[tid] = 0u;
    }
    // Columns this tile answers for: up to the next tile's first.
    const bool first = tile == 0, last = rb + len == row1;
    const uint32_t lo = first || len == 0 ? 0u : g.c_col[rb], hi = last ? 0xffffffffu : g.c_col[rb + len];
    auto fetch = [&](uint32_t t) {
        uint4 m = make_uint4(0, 0, 0, 0);
        if (t < t1) {
            const uint32_t i = g.t_row[t];
            const double w = g.pval[g.prow[i] + g.t_pos[t]];
            m = make_uint4(g.ap_off[i], g.ap_off[i + 1], uint32_t(__double2loint(w)), uint32_t(__double2hiint(w)));
        }
        return m;
    };
    if (tid < kTileFine) meta[tid] = fetch(t0 + tid);
    __syncthreads();
    bool missing = false;
    uint32_t set = 0;
    for (uint32_t r = t0; r < t1; r += kTileFine, set ^= 1u) {
        uint4 next = make_uint4(0, 0, 0, 0);
        if (tid < kTileFine) next = fetch(r + kTileFine + tid);
        for (uint32_t f = wave; f < kTileFine && r + f < t1; f += 16) {
            const uint4 m = meta[set * kTileFine + f];
            const double w = __hiloint2double(int(m.w), int(m.z));
            uint32_t b = __builtin_amdgcn_readfirstlane(m.x);
            const uint32_t e = __builtin_amdgcn_readfirstlane(m.y);
            if (!first && e - b > 128) b = lower_bound_u32(g.ap_col, b, e, lo);
            for (uint32_t p = b; p < e; p += 64) {
                const bool in = p + lane < e;
                const uint32_t col = in ? g.ap_col[p + lane] : 0xffffffffu;
                if (in && col >= lo && (last || col < hi)) {
                    const double v = g.apv[p + lane];
                    const uint32_t pos = find_col(cols, len, col);
                    if (pos < len) {
                        table[f * kTileCols + pos] = w * v;
                        atomicOr(&mask[pos], 1u << f);
                    } else {
                        missing = true;
                    }
                }
                if (!last && __ballot(in && col >= hi)) break;
            }
        }
        __syncthreads();
        if (tid < len) {
            uint32_t m = mask[tid];
            if (m) {
                double a = acc[tid];
                for (; m; m &= m - 1) a += table[__builtin_ctz(m) * kTileCols + tid];
                acc[tid] = a;
                mask[tid] = 0u;
            }
        }
        if (tid < kTileFine) meta[(set ^ 1u) * kTileFine + tid] = next;
        __syncthreads();
    }
    if (missing) g.flags[kBadProduct] = 1;
    if (tid < len) store_c(g, rb + tid, acc[tid]);
}

// Row index of every entry of a CSR pattern.
__global__ __launch_bounds__(kBlock) void row_index_kernel(uint32_t n, const uint32_t* __restrict__ off,
                                                           uint32_t* __restrict__ row) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    for (uint32_t k = off[i]; k < off[i + 1]; ++k) row[k] = i;
}

// ---- Damping certificate and Lanczos bounds, all levels in one launch: a
// level is a few microseconds of work, and a launch each (with a scalar sent
// back to the host after every dot product) made 1800 launches of a refresh.

// The level of workgroup wg: views[l].*first <= wg < views[l + 1].*first.
__device__ __forceinline__ uint32_t level_of(const RefreshView* __restrict__ views, uint32_t wg) {
    uint32_t l = 0;
    while (wg >= views[l + 1].first_wg) ++l;
    return l;
}

// Normalised Gershgorin row sums sum_j |a_ij| / (sqrt(d_i) sqrt(d_j)),
// d = 1 / inv; per-workgroup maxima. flags: kFlagCount per level.
__global__ __launch_bounds__(kBlock) void gershgorin_sd_kernel(const RefreshView* __restrict__ views, uint32_t slot,
                                                               double* __restrict__ sd, int* __restrict__ flags) {
#pragma clang fp contract(off)
    const uint32_t l = level_of(views, blockIdx.x);
    const RefreshView& L = views[l];
    const uint32_t i = (blockIdx.x - L.first_wg) * kBlock + threadIdx.x;
    if (i >= L.n) return;
    const double v = L.rinv[slot][i];
    double s = 0.0;
    if (!(v > 0.0) || !isfinite(v)) {
        flags[l * kFlagCount + kBadGershgorin] = 1;
    } else {
        const double d = 1.0 / v;
        if (!(d > 0.0) || !isfinite(d)) flags[l * kFlagCount + kBadGershgorin] = 1;
        else s = sqrt(d);
    }
    sd[L.row0 + i] = s;
}

// Rows above kGershgorinRow entries, listed longest first: one wavefront each, 64
// terms formed at a time and added in order, a chain of 6 ns an entry. Coarse
// levels hold their long rows side by side: with the wavefront that holds a row
// of 64 also summing its long ones, a refresh of 222k cells spent 1204 us here.
// With a wavefront each the whole refresh went from 6410 to 5398 us.
constexpr uint32_t kGershgorinRow = 48;
__global__ __launch_bounds__(kBlock) void gershgorin_long_kernel(const RefreshView* __restrict__ views, uint32_t slot,
                                                                 uint32_t count, const uint2* __restrict__ list,
                                                                 const double* __restrict__ sd_all,
                                                                 double* __restrict__ sums) {
#pragma clang fp contract(off)
    const uint32_t w = (blockIdx.x * kBlock + threadIdx.x) >> 6, lane = threadIdx.x & 63u;
    if (w >= count) return;
    const uint2 at = list[w];
    const RefreshView& L = views[at.x];
    const double* sd = sd_all + L.row0;
    const uint32_t* cols = L.acol;
    const double* vals = L.aval[slot];
    const uint32_t e = L.arow[at.y + 1];
    const double s0 = sd[at.y];
    double s = 0.0;
    bool wrong = false;
    for (uint32_t k = L.arow[at.y]; k < e; k += 64) {
        double t = 0.0;
        const bool in = k + lane < e;
        if (in) {
            const double sc = s0 * sd[cols[k + lane]];
            if (!(sc > 0.0) || !isfinite(sc)) wrong = true;
            t = fabs(vals[k + lane]) / sc;
        }
        s = add_lanes(s, t, __ballot(in));
    }
    if (__ballot(wrong)) s = NAN;
    if (lane == 0) sums[L.row0 + at.y] = s;
}

__global__ __launch_bounds__(kBlock) void gershgorin_rows_kernel(const RefreshView* __restrict__ views, uint32_t slot,
                                                                 const double* __restrict__ sd_all,
                                                                 const double* __restrict__ long_sums,
                                                                 double* __restrict__ block_max,
                                                                 int* __restrict__ flags) {
#pragma clang fp contract(off)
    __shared__ double sm[kBlock];
    const uint32_t l = level_of(views, blockIdx.x);
    const RefreshView& L = views[l];
    const double* sd = sd_all + L.row0;
    const uint32_t* cols = L.acol;
    const double* vals = L.aval[slot];
    const uint32_t i = (blockIdx.x - L.first_wg) * kBlock + threadIdx.x;
    const bool live = i < L.n;
    const uint32_t b = live ? L.arow[i] : 0u, e = live ? L.arow[i + 1] : 0u;
    const double si = live ? sd[i] : 0.0;
    double rs = 0.0;
    bool bad = false;
    if (e - b > kGershgorinRow) {
        rs = long_sums[L.row0 + i];
    } else {
        for (uint32_t k = b; k < e; ++k) {
            const double sc = si * sd[cols[k]];
            if (!(sc > 0.0) || !isfinite(sc)) bad = true;
            rs += fabs(vals[k]) / sc;
        }
    }
    if (live && (bad || !isfinite(rs))) {
        flags[l * kFlagCount + kBadGershgorin] = 1;
        rs = 0.0;
    }
    sm[threadIdx.x] = rs;
    __syncthreads();
    for (uint32_t s = kBlock / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) sm[threadIdx.x] = fmax(sm[threadIdx.x], sm[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) block_max[blockIdx.x] = sm[0];
}

// out[l] = maximum over level l's workgroups.
__global__ __launch_bounds__(1024) void max_reduce_kernel(const RefreshView* __restrict__ views,
                                                          const double* __restrict__ v, double* __restrict__ out) {
    __shared__ double sm[1024];
    double m = 0.0;
    for (uint32_t i = views[blockIdx.x].first_wg + threadIdx.x; i < views[blockIdx.x + 1].first_wg; i += 1024)
        m = fmax(m, v[i]);
    sm[threadIdx.x] = m;
    __syncthreads();
    for (uint32_t s = 512; s > 0; s >>= 1) {
        if (threadIdx.x < s) sm[threadIdx.x] = fmax(sm[threadIdx.x], sm[threadIdx.x + s]);
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.x] = sm[0];
}

// ---- Lanczos on D^-1/2 A D^-1/2, the host estimate's arithmetic. Vectors
// live in the solve ordering next to the committed solve-ordered matrix
// (rows keep the reference's entry order, so each row sum is the host's);
// the dot products visit rows in the reference order through new_of_old, in
// 256-row tiles (tile_tree_sum) whose sums lanczos_total_kernel adds in the
// host's blocks of 8192 rows. A level whose recurrence has ended (stop) skips
// the launches that remain.

__device__ __forceinline__ double lanczos_start(uint32_t i) {
    const uint32_t h = i * 2654435761u + 0x9e3779b9u;
    return double(h >> 8) * (1.0 / 16777216.0) - 0.5;
}

struct LanczosVectors {
    double *sq, *v, *vp, *w, *u, *tile;
};

// The workgroup's tile sum of x (one value a thread).
__device__ __forceinline__ void store_tile(double x, double* __restrict__ tile) {
#pragma clang fp contract(off)
    __shared__ double red[4];
    x = wave_sum(x);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
    __syncthreads();
    if (threadIdx.x == 0) tile[blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

__global__ __launch_bounds__(kBlock) void lanczos_init_kernel(const RefreshView* __restrict__ views,
                                                              LanczosState* __restrict__ st, LanczosVectors z) {
#pragma clang fp contract(off)
    const uint32_t l = level_of(views, blockIdx.x);
    const RefreshView& L = views[l];
    const uint32_t i = (blockIdx.x - L.first_wg) * kBlock + threadIdx.x;
    double x = 0.0;
    if (i < L.n) {
        const uint32_t p = L.perm[i];
        const double v = lanczos_start(i);
        z.v[L.row0 + p] = v;
        z.sq[L.row0 + i] = sqrt(L.inv[i]);
        z.vp[L.row0 + i] = 0.0;
        x = v * v;
    }
    if (blockIdx.x == L.first_wg && threadIdx.x == 0) {
        st[l].count = st[l].stop = 0;
        st[l].beta[0] = 0.0;
    }
    store_tile(x, z.tile);
}

// The ordered total of a level's tile sums, then what the host's loop does
// with it. kWhat 0: |v| at the start; 1: alpha; 2: beta and the stop rule.
template <int kWhat>
__global__ __launch_bounds__(1024) void lanczos_total_kernel(const RefreshView* __restrict__ views, uint32_t steps,
                                                             LanczosState* __restrict__ states,
                                                             const double* __restrict__ tile) {
#pragma clang fp contract(off)
    constexpr uint32_t kTiles = kLanczosRows / kBlock;
    const RefreshView& L = views[blockIdx.x];
    LanczosState& S = states[blockIdx.x];
    if (S.stop) return;
    const uint32_t nt = views[blockIdx.x + 1].first_wg - L.first_wg, nb = (nt + kTiles - 1) / kTiles;
    const double* t = tile + L.first_wg;
    __shared__ double sm[1024];
    double total = 0.0;
    for (uint32_t b0 = 0; b0 < nb; b0 += 1024) {
        const uint32_t b = b0 + threadIdx.x;
        double acc = 0.0;
        if (b < nb) {
            double v[kTiles];
#pragma unroll
            for (uint32_t k = 0; k < kTiles; ++k) v[k] = b * kTiles + k < nt ? t[b * kTiles + k] : 0.0;
#pragma unroll
            for (uint32_t k = 0; k < kTiles; ++k)
                if (b * kTiles + k < nt) acc += v[k];
        }
        sm[threadIdx.x] = acc;
        __syncthreads();
        if (threadIdx.x == 0) total = ordered_sum<false>(sm, 0u, min(nb - b0, 1024u), total);
        __syncthreads();
    }
    if (threadIdx.x != 0) return;
    if (kWhat == 0) {
        S.norm = sqrt(total);
    } else if (kWhat == 1) {
        S.a = total;
        S.alpha[S.count] = total;
        S.bprev = S.beta[S.count];
        ++S.count;
    } else {
        const double bn = sqrt(total);
        if (!(bn > 1e-14 * fabs(S.a)) || S.count == min(steps, L.n)) {
            S.stop = 1;
        } else {
            S.beta[S.count] = bn;
            S.b = bn;
        }
    }
}

// v /= |v| and u = sq v.
__global__ __launch_bounds__(kBlock) void lanczos_scale_kernel(const RefreshView* __restrict__ views,
                                                               const LanczosState* __restrict__ st,
                                                               LanczosVectors z) {
#pragma clang fp contract(off)
    const uint32_t l = level_of(views, blockIdx.x);
    const RefreshView& L = views[l];
    const uint32_t i = (blockIdx.x - L.first_wg) * kBlock + threadIdx.x;
    if (i >= L.n) return;
    const double v = z.v[L.row0 + i] / st[l].norm;
    z.v[L.row0 + i] = v;
    z.u[L.row0 + i] = z.sq[L.row0 + i] * v;
}

// w = sq (A u): w_i = sq_i sum_q a_iq (sq_j v_j) in each row's entry order.
struct EpiScaled {
    struct Pre {
        double d;
    };
    const double* d;
    double* y;
    __device__ Pre load(uint32_t row) const { return {d[row]}; }
    __device__ double apply(uint32_t row, double s, const Pre& p) const {
        y[row] = p.d * s;
        return 0.0;
    }
    __device__ double operator()(uint32_t row, double s) const { return apply(row, s, load(row)); }
};
__global__ __launch_bounds__(kBlock) void lanczos_spmv_kernel(const RefreshView* __restrict__ views,
                                                              const LanczosState* __restrict__ st,
                                                              LanczosVectors z) {
    uint32_t l = 0;
    while (blockIdx.x >= views[l + 1].first_block) ++l;
    if (st[l].stop) return;
    const RefreshView& L = views[l];
    const uint32_t b = xcd_block(blockIdx.x - L.first_block, views[l + 1].first_block - L.first_block);
    stream_rows<double>(L.blocks[b], L.blocks[b + 1], L.rowp, L.cols, L.vals, z.u + L.row0, InitZero<double>{},
                        EpiScaled{z.sq + L.row0, z.w + L.row0});
}

// Tile sums of w v.
__global__ __launch_bounds__(kBlock) void lanczos_dot_kernel(const RefreshView* __restrict__ views,
                                                             const LanczosState* __restrict__ st, LanczosVectors z) {
#pragma clang fp contract(off)
    const uint32_t l = level_of(views, blockIdx.x);
    if (st[l].stop) return;
    const RefreshView& L = views[l];
    const uint32_t i = (blockIdx.x - L.first_wg) * kBlock + threadIdx.x;
    double x = 0.0;
    if (i < L.n) {
        const uint32_t p = L.row0 + L.perm[i];
        x = z.w[p] * z.v[p];
    }
    store_tile(x, z.tile);
}

// w = (w - a v) - b_prev vp, and the tile sums of w w.
__global__ __launch_bounds__(kBlock) void lanczos_update_kernel(const RefreshView* __restrict__ views,
                                                                const LanczosState* __restrict__ st,
                                                                LanczosVectors z) {
#pragma clang fp contract(off)
    const uint32_t l = level_of(views, blockIdx.x);
    if (st[l].stop) return;
    const RefreshView& L = views[l];
    const uint32_t i = (blockIdx.x - L.first_wg) * kBlock + threadIdx.x;
    double x = 0.0;
    if (i < L.n) {
        const uint32_t p = L.row0 + L.perm[i];
        const double w = (z.w[p] - st[l].a * z.v[p]) - st[l].bprev * z.vp[p];
        z.w[p] = w;
        x = w * w;
    }
    store_tile(x, z.tile);
}

// vp = v, v = w / b, u = sq v.
__global__ __launch_bounds__(kBlock) void lanczos_next_kernel(const RefreshView* __restrict__ views,
                                                              const LanczosState* __restrict__ st, LanczosVectors z) {
#pragma clang fp contract(off)
    const uint32_t l = level_of(views, blockIdx.x);
    if (st[l].stop) return;
    const RefreshView& L = views[l];
    const uint32_t i = (blockIdx.x - L.first_wg) * kBlock + threadIdx.x;
    if (i >= L.n) return;
    const uint32_t p = L.row0 + i;
    z.vp[p] = z.v[p];
    const double v = z.w[p] / st[l].b;
    z.v[p] = v;
    z.u[p] = z.sq[p] * v;
}

// Committed values in the solve ordering: CSR copies of either precision.
__global__ __launch_bounds__(kBlock) void commit_values_kernel(uint64_t n, const uint32_t* __restrict__ idx,
                                                               const double* __restrict__ src,
                                                               double* __restrict__ v64, float* __restrict__ v32) {
    const uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i >= n) return;
    const double v = src[idx[i]];
    if (v64) v64[i] = v;
    if (v32) v32[i] = float(v);
}
__global__ __launch_bounds__(kBlock) void commit_diagonal_kernel(uint32_t n, const uint32_t* __restrict__ perm,
                                                                 const double* __restrict__ src,
                                                                 double* __restrict__ d64, float* __restrict__ d32) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const uint32_t p = perm[i];
    if (d64) d64[p] = src[i];
    if (d32) d32[p] = float(src[i]);
}

template <class T>
__global__ __launch_bounds__(kBlock) void gather_idx_kernel(uint64_t n, const uint32_t* __restrict__ idx,
                                                            const double* __restrict__ src, T* __restrict__ dst) {
    const uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i < n) dst[i] = T(src[idx[i]]);
}

inline uint32_t grid64(uint64_t n) { return uint32_t((n + kBlock - 1) / kBlock); }

// ---- hierarchy construction kernels (smoothed aggregation) ------------------

// Exclusive scan of 32-bit counts into 64-bit offsets: per-tile sums, a
// sequential scan of the tile sums, then each tile's local scan.
constexpr uint32_t kScanItems = 16;
constexpr uint32_t kScanTile = kBlock * kScanItems;

__global__ __launch_bounds__(kBlock) void scan_tile_sums_kernel(uint64_t n, const uint32_t* __restrict__ in,
                                                                uint64_t* __restrict__ tile_sum) {
    __shared__ uint64_t sm[kBlock];
    const uint64_t base = uint64_t(blockIdx.x) * kScanTile;
    uint64_t s = 0;
    for (uint32_t k = 0; k < kScanItems; ++k) {
        const uint64_t i = base + uint64_t(k) * kBlock + threadIdx.x;
        if (i < n) s += in[i];
    }
    sm[threadIdx.x] = s;
    __syncthreads();
    for (uint32_t st = kBlock / 2; st > 0; st >>= 1) {
        if (threadIdx.x < st) sm[threadIdx.x] += sm[threadIdx.x + st];
        __syncthreads();
    }
    if (threadIdx.x == 0) tile_sum[blockIdx.x] = sm[0];
}

__global__ void scan_tiles_kernel(uint32_t nt, uint64_t* __restrict__ tile_sum, uint64_t* __restrict__ total) {
    if (blockIdx.x != 0 || threadIdx.x != 0) return;
    uint64_t run = 0;
    for (uint32_t t = 0; t < nt; ++t) {
        const uint64_t v = tile_sum[t];
        tile_sum[t] = run;
        run += v;
    }
    *total = run;
}

__global__ __launch_bounds__(kBlock) void scan_apply_kernel(uint64_t n, const uint32_t* __restrict__ in,
                                                            const uint64_t* __restrict__ tile_off,
                                                            uint64_t* __restrict__ out) {
    __shared__ uint64_t sm[kBlock];
    const uint64_t base = uint64_t(blockIdx.x) * kScanTile + uint64_t(threadIdx.x) * kScanItems;
    uint32_t v[kScanItems];
    uint64_t s = 0;
#pragma unroll
    for (uint32_t k = 0; k < kScanItems; ++k) {
        const uint64_t i = base + k;
        v[k] = i < n ? in[i] : 0u;
        s += v[k];
    }
    sm[threadIdx.x] = s;
    __syncthreads();
    for (uint32_t off = 1; off < kBlock; off <<= 1) {
        const uint64_t t = threadIdx.x >= off ? sm[threadIdx.x - off] : 0;
        __syncthreads();
        sm[threadIdx.x] += t;
        __syncthreads();
    }
    uint64_t run = tile_off[blockIdx.x] + sm[threadIdx.x] - s;
#pragma unroll
    for (uint32_t k = 0; k < kScanItems; ++k) {
        const uint64_t i = base + k;
        if (i < n) out[i] = run;
        run += v[k];
    }
}

__global__ __launch_bounds__(kBlock) void narrow_u32_kernel(uint64_t n, const uint64_t* __restrict__ in,
                                                            uint32_t* __restrict__ out) {
    const uint64_t i = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (i < n) out[i] = uint32_t(in[i]);
}

// strength_graph (amg_preconditioner.h:1466-1509 as restated on the host):
// rows whose |row sum| exceeds 0.9 |a_ii| have no strong connections; else a
// neighbour is strong when it is opposite in sign to the diagonal (or, with
// no such neighbour, any neighbour) and |a_ij| + eps >= theta max.
__global__ __launch_bounds__(kBlock) void strength_count_kernel(uint32_t n, const uint32_t* __restrict__ arow,
                                                                const uint32_t* __restrict__ acol,
                                                                const double* __restrict__ aval,
                                                                const double* __restrict__ inv, double theta,
                                                                double* __restrict__ thr, int8_t* __restrict__ mode,
                                                                uint32_t* __restrict__ cnt) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const double eps = 2.220446049250313080847e-16;
    const double di = 1.0 / inv[i];
    double row_sum = di, opp = 0.0, absmax = 0.0;
    for (uint32_t k = arow[i]; k < arow[i + 1]; ++k) {
        if (acol[k] == i) continue;
        const double v = aval[k];
        row_sum += v;
        absmax = absmax < fabs(v) ? fabs(v) : absmax;
        if (di * v < 0.0) opp = opp < fabs(v) ? fabs(v) : opp;
    }
    mode[i] = -1;
    cnt[i] = 0;
    if (fabs(row_sum) > fabs(di) * 0.9) return;
    const bool use_opp = opp > 0.0;
    const double sc = use_opp ? opp : absmax;
    if (!(sc > 0.0) || !isfinite(sc)) return;
    mode[i] = use_opp ? 1 : 0;
    const double t = theta * sc;
    thr[i] = t;
    uint32_t c = 0;
    for (uint32_t k = arow[i]; k < arow[i + 1]; ++k) {
        const uint32_t j = acol[k];
        const double v = aval[k];
        if (j == i || j >= n) continue;
        if (use_opp && di * v >= 0.0) continue;
        if (fabs(v) + eps < t) continue;
        ++c;
    }
    cnt[i] = c;
}

__global__ __launch_bounds__(kBlock) void strength_fill_kernel(uint32_t n, const uint32_t* __restrict__ arow,
                                                               const uint32_t* __restrict__ acol,
                                                               const double* __restrict__ aval,
                                                               const double* __restrict__ inv,
                                                               const double* __restrict__ thr,
                                                               const int8_t* __restrict__ mode,
                                                               const uint64_t* __restrict__ soff,
                                                               uint32_t* __restrict__ scol) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n || mode[i] < 0) return;
    const double eps = 2.220446049250313080847e-16;
    const double di = 1.0 / inv[i];
    const double t = thr[i];
    uint64_t w = soff[i];
    for (uint32_t k = arow[i]; k < arow[i + 1]; ++k) {
        const uint32_t j = acol[k];
        const double v = aval[k];
        if (j == i || j >= n) continue;
        if (mode[i] == 1 && di * v >= 0.0) continue;
        if (fabs(v) + eps < t) continue;
        scol[w++] = j;
    }
}

// Transpose of a pattern: counts per column, then each entry placed through
// a per-column cursor; the segments are sorted afterwards, so the result is
// the ascending transpose whatever order the cursors were taken in.
__global__ __launch_bounds__(kBlock) void col_count_kernel(uint32_t n, const uint64_t* __restrict__ off,
                                                           const uint32_t* __restrict__ col,
                                                           uint32_t* __restrict__ cnt) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    for (uint64_t k = off[i]; k < off[i + 1]; ++k) atomicAdd(&cnt[col[k]], 1u);
}

__global__ __launch_bounds__(kBlock) void col_fill_kernel(uint32_t n, const uint64_t* __restrict__ off,
                                                          const uint32_t* __restrict__ col,
                                                          const uint64_t* __restrict__ toff,
                                                          uint32_t* __restrict__ cursor, uint32_t* __restrict__ tcol) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    for (uint64_t k = off[i]; k < off[i + 1]; ++k) {
        const uint32_t j = col[k];
        const uint32_t pos = atomicAdd(&cursor[j], 1u);
        tcol[toff[j] + pos] = i;
    }
}

template <class K>
__device__ void sift_down(K* a, uint64_t root, uint64_t end) {
    while (true) {
        uint64_t child = 2 * root + 1;
        if (child >= end) return;
        if (child + 1 < end && a[child] < a[child + 1]) ++child;
        if (!(a[root] < a[child])) return;
        const K t = a[root];
        a[root] = a[child];
        a[child] = t;
        root = child;
    }
}

// Ascending sort of a[0, n): insertion sort for short segments, heap sort
// otherwise.
template <class K>
__device__ void sort_segment(K* a, uint64_t n) {
    if (n <= 32) {
        for (uint64_t i = 1; i < n; ++i) {
            const K v = a[i];
            uint64_t j = i;
            while (j > 0 && v < a[j - 1]) {
                a[j] = a[j - 1];
                --j;
            }
            a[j] = v;
        }
        return;
    }
    for (uint64_t s = n / 2; s-- > 0;) sift_down(a, s, n);
    for (uint64_t e = n; e-- > 1;) {
        const K t = a[0];
        a[0] = a[e];
        a[e] = t;
        sift_down(a, 0, e);
    }
}

template <class K>
__global__ __launch_bounds__(kBlock) void segment_sort_kernel(uint32_t n, const uint64_t* __restrict__ off,
                                                              K* __restrict__ a) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n) sort_segment(a + off[i], off[i + 1] - off[i]);
}

// Symmetrised neighbourhood: the sorted union of S_i and (S^T)_i.
__global__ __launch_bounds__(kBlock) void merge_count_kernel(uint32_t n, const uint64_t* __restrict__ soff,
                                                             const uint32_t* __restrict__ scol,
                                                             const uint64_t* __restrict__ toff,
                                                             const uint32_t* __restrict__ tcol,
                                                             uint32_t* __restrict__ cnt) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    uint64_t a = soff[i], ae = soff[i + 1], b = toff[i], be = toff[i + 1];
    uint32_t c = 0;
    while (a < ae || b < be) {
        if (b >= be || (a < ae && scol[a] < tcol[b])) ++a;
        else if (a >= ae || tcol[b] < scol[a]) ++b;
        else {
            ++a;
            ++b;
        }
        ++c;
    }
    cnt[i] = c;
}

__global__ __launch_bounds__(kBlock) void merge_fill_kernel(uint32_t n, const uint64_t* __restrict__ soff,
                                                            const uint32_t* __restrict__ scol,
                                                            const uint64_t* __restrict__ toff,
                                                            const uint32_t* __restrict__ tcol,
                                                            const uint64_t* __restrict__ noff,
                                                            uint32_t* __restrict__ ncol) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    uint64_t a = soff[i], ae = soff[i + 1], b = toff[i], be = toff[i + 1], w = noff[i];
    while (a < ae || b < be) {
        if (b >= be || (a < ae && scol[a] < tcol[b])) ncol[w++] = scol[a++];
        else if (a >= ae || tcol[b] < scol[a]) ncol[w++] = tcol[b++];
        else {
            ncol[w++] = scol[a];
            ++a;
            ++b;
        }
    }
}

constexpr uint32_t kSmoothShortRow = 32;  // rows at least this long take the sort path

// One damped-Jacobi smoothing step of the tentative prolongator, row
// normalised, with the restated drop / filter / fallback rules
// (amg_preconditioner.h:1968-2044; keep_own: the own-aggregate entry
// survives the filter, and a row whose own-aggregate weight falls below
// filter * largest keeps its tentative row). Row i works in scratch at arow[i] + i (row length
// + 1 slots): distinct aggregates in first-seen order, their sums in entry
// order, then sorted by aggregate id.
__global__ __launch_bounds__(kBlock) void smooth_rows_kernel(
    uint32_t n, const uint32_t* __restrict__ arow, const uint32_t* __restrict__ acol,
    const double* __restrict__ aval, const double* __restrict__ inv, const uint32_t* __restrict__ agg,
    double filter, int keep_own, uint32_t* __restrict__ scol, double* __restrict__ sval, uint64_t* __restrict__ keys,
    uint32_t* __restrict__ cnt, unsigned long long* __restrict__ fallbacks) {
#pragma clang fp contract(off)
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const double w = 2.0 / 3.0;
    const uint64_t base = uint64_t(arow[i]) + i;
    uint32_t* oc = scol + base;
    double* ov = sval + base;
    const uint32_t len = arow[i + 1] - arow[i];
    uint32_t d = 0;
    if (len < kSmoothShortRow) {
        // Short rows: distinct aggregates in first-seen order, then sorted.
        auto acc = [&](uint32_t c, double v) {
            for (uint32_t q = 0; q < d; ++q)
                if (oc[q] == c) {
                    ov[q] += v;
                    return;
                }
            oc[d] = c;
            ov[d] = 0.0;
            ov[d] += v;
            ++d;
        };
        acc(agg[i], 1.0);
        for (uint32_t k = arow[i]; k < arow[i + 1]; ++k) acc(agg[acol[k]], -w * inv[i] * aval[k]);
        for (uint32_t q = 1; q < d; ++q) {
            const uint32_t c = oc[q];
            const double v = ov[q];
            uint32_t r = q;
            while (r > 0 && c < oc[r - 1]) {
                oc[r] = oc[r - 1];
                ov[r] = ov[r - 1];
                --r;
            }
            oc[r] = c;
            ov[r] = v;
        }
    } else {
        // Long rows: sort (aggregate, entry index) keys, the own-aggregate
        // term as index 0, so each aggregate's terms are added in the same
        // order (own term, then entries in row order) as the short path.
        uint64_t* key = keys + base;
        key[0] = uint64_t(agg[i]) << 32;
        for (uint32_t k = 0; k < len; ++k) key[k + 1] = (uint64_t(agg[acol[arow[i] + k]]) << 32) | uint64_t(k + 1);
        sort_segment(key, uint64_t(len) + 1);
        for (uint32_t q = 0; q <= len; ++q) {
            const uint32_t c = uint32_t(key[q] >> 32);
            const uint32_t idx = uint32_t(key[q] & 0xffffffffu);
            const double v = idx == 0 ? 1.0 : -w * inv[i] * aval[arow[i] + idx - 1];
            if (d == 0 || oc[d - 1] != c) {
                oc[d] = c;
                ov[d] = 0.0;
                ov[d] += v;
                ++d;
            } else {
                ov[d - 1] += v;
            }
        }
    }
    double sum = 0.0;
    for (uint32_t q = 0; q < d; ++q)
        if (isfinite(ov[q]) && fabs(ov[q]) > 1e-14) sum += ov[q];
    const uint32_t own_c = agg[i];
    if (!isfinite(sum) || fabs(sum) <= 1e-14) {
        oc[0] = own_c;
        ov[0] = 1.0;
        cnt[i] = 1;
        atomicAdd(fallbacks, 1ull);
        return;
    }
    double largest = 0.0;
    double own_w = 0.0;
    for (uint32_t q = 0; q < d; ++q) {
        const double x = fabs(ov[q] / sum);
        largest = largest < x ? x : largest;
        if (oc[q] == own_c) own_w = ov[q] / sum;
    }
    if (keep_own && !(own_w >= filter * largest)) {
        // the smoothed row would hand the point away from its own aggregate:
        // tentative row
        oc[0] = own_c;
        ov[0] = 1.0;
        cnt[i] = 1;
        atomicAdd(fallbacks, 1ull);
        return;
    }
    uint32_t m = 0;
    for (uint32_t q = 0; q < d; ++q) {
        const double nv = ov[q] / sum;
        const bool own = keep_own && oc[q] == own_c;
        if (isfinite(nv) && (own ? nv != 0.0 : (fabs(nv) > 1e-14 && fabs(nv) >= filter * largest))) {
            oc[m] = oc[q];
            ov[m] = nv;
            ++m;
        }
    }
    double kept = 0.0;
    for (uint32_t q = 0; q < m; ++q) kept += ov[q];
    if (isfinite(kept) && fabs(kept) > 1e-14) {
        for (uint32_t q = 0; q < m; ++q) ov[q] /= kept;
    } else {
        m = 0;
    }
    if (m == 0) {
        oc[0] = own_c;
        ov[0] = 1.0;
        m = 1;
        atomicAdd(fallbacks, 1ull);
    }
    cnt[i] = m;
}

// Copies row i's first (dst_off[i+1] - dst_off[i]) entries from scratch at
// src_base(i) to the compact arrays.
template <class T>
__global__ __launch_bounds__(kBlock) void compact_from_rows_kernel(uint32_t n, const uint32_t* __restrict__ arow,
                                                                   const uint64_t* __restrict__ dst_off,
                                                                   const T* __restrict__ src, T* __restrict__ dst) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const uint64_t s = uint64_t(arow[i]) + i;
    for (uint64_t q = dst_off[i]; q < dst_off[i + 1]; ++q) dst[q] = src[s + (q - dst_off[i])];
}

template <class T>
__global__ __launch_bounds__(kBlock) void compact_from_offsets_kernel(uint32_t n,
                                                                      const uint64_t* __restrict__ src_off,
                                                                      const uint64_t* __restrict__ dst_off,
                                                                      const T* __restrict__ src,
                                                                      T* __restrict__ dst) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const uint64_t s = src_off[i];
    for (uint64_t q = dst_off[i]; q < dst_off[i + 1]; ++q) dst[q] = src[s + (q - dst_off[i])];
}

// Sorted, de-duplicated segment: returns its new length.
__device__ uint32_t sort_unique(uint32_t* a, uint64_t n) {
    sort_segment(a, n);
    uint32_t m = 0;
    for (uint64_t q = 0; q < n; ++q)
        if (m == 0 || a[q] != a[m - 1]) a[m++] = a[q];
    return m;
}

// AP pattern (galerkin_csr_product.h:33-148): row i = sorted union of the P
// rows of i's A neighbours. ub: the candidate count.
__global__ __launch_bounds__(kBlock) void ap_bound_kernel(uint32_t n, const uint32_t* __restrict__ arow,
                                                          const uint32_t* __restrict__ acol,
                                                          const uint32_t* __restrict__ prow,
                                                          uint32_t* __restrict__ ub) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    uint32_t c = 0;
    for (uint32_t k = arow[i]; k < arow[i + 1]; ++k) c += prow[acol[k] + 1] - prow[acol[k]];
    ub[i] = c;
}

__global__ __launch_bounds__(kBlock) void ap_pattern_kernel(uint32_t n, const uint32_t* __restrict__ arow,
                                                            const uint32_t* __restrict__ acol,
                                                            const uint32_t* __restrict__ prow,
                                                            const uint32_t* __restrict__ pcol,
                                                            const uint64_t* __restrict__ boff,
                                                            uint32_t* __restrict__ buf, uint32_t* __restrict__ cnt) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    uint32_t* b = buf + boff[i];
    uint64_t w = 0;
    for (uint32_t k = arow[i]; k < arow[i + 1]; ++k) {
        const uint32_t j = acol[k];
        for (uint32_t q = prow[j]; q < prow[j + 1]; ++q) b[w++] = pcol[q];
    }
    cnt[i] = sort_unique(b, w);
}

// Transpose plan of P: coarse column c lists (fine row i, position of c in
// P's row i) for ascending i, packed as i << 32 | position.
__global__ __launch_bounds__(kBlock) void t_count_kernel(uint32_t n, const uint32_t* __restrict__ prow,
                                                         const uint32_t* __restrict__ pcol,
                                                         uint32_t* __restrict__ cnt) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    for (uint32_t q = prow[i]; q < prow[i + 1]; ++q) atomicAdd(&cnt[pcol[q]], 1u);
}

__global__ __launch_bounds__(kBlock) void t_fill_kernel(uint32_t n, const uint32_t* __restrict__ prow,
                                                        const uint32_t* __restrict__ pcol,
                                                        const uint64_t* __restrict__ toff,
                                                        uint32_t* __restrict__ cursor, uint64_t* __restrict__ key) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    for (uint32_t q = prow[i]; q < prow[i + 1]; ++q) {
        const uint32_t c = pcol[q];
        const uint32_t pos = atomicAdd(&cursor[c], 1u);
        key[toff[c] + pos] = (uint64_t(i) << 32) | uint64_t(q - prow[i]);
    }
}

__global__ __launch_bounds__(kBlock) void t_split_kernel(uint64_t m, const uint64_t* __restrict__ key,
                                                         uint32_t* __restrict__ t_row, uint32_t* __restrict__ t_pos) {
    const uint64_t k = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (k >= m) return;
    t_row[k] = uint32_t(key[k] >> 32);
    t_pos[k] = uint32_t(key[k] & 0xffffffffu);
}

// P^T (AP) pattern: coarse row c = sorted union of the AP rows of the fine
// rows holding column c.
__global__ __launch_bounds__(kBlock) void c_bound_kernel(uint32_t nc, const uint32_t* __restrict__ t_off,
                                                         const uint32_t* __restrict__ t_row,
                                                         const uint32_t* __restrict__ ap_off,
                                                         uint32_t* __restrict__ ub) {
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= nc) return;
    uint32_t s = 0;
    for (uint32_t t = t_off[c]; t < t_off[c + 1]; ++t) s += ap_off[t_row[t] + 1] - ap_off[t_row[t]];
    ub[c] = s;
}

__global__ __launch_bounds__(kBlock) void c_pattern_kernel(uint32_t nc, const uint32_t* __restrict__ t_off,
                                                           const uint32_t* __restrict__ t_row,
                                                           const uint32_t* __restrict__ ap_off,
                                                           const uint32_t* __restrict__ ap_col,
                                                           const uint64_t* __restrict__ boff,
                                                           uint32_t* __restrict__ buf, uint32_t* __restrict__ cnt) {
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= nc) return;
    uint32_t* b = buf + boff[c];
    uint64_t w = 0;
    for (uint32_t t = t_off[c]; t < t_off[c + 1]; ++t) {
        const uint32_t i = t_row[t];
        for (uint32_t p = ap_off[i]; p < ap_off[i + 1]; ++p) b[w++] = ap_col[p];
    }
    cnt[c] = sort_unique(b, w);
}

// The kept coarse entries (|c| > 1e-30) of each row, in order.
__global__ __launch_bounds__(kBlock) void prune_count_kernel(uint32_t nc, const uint32_t* __restrict__ c_off,
                                                             const double* __restrict__ cv,
                                                             uint32_t* __restrict__ cnt) {
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= nc) return;
    uint32_t k = 0;
    for (uint32_t p = c_off[c]; p < c_off[c + 1]; ++p) k += fabs(cv[p]) > 1e-30;
    cnt[c] = k;
}

__global__ __launch_bounds__(kBlock) void prune_fill_kernel(uint32_t nc, const uint32_t* __restrict__ c_off,
                                                            const uint32_t* __restrict__ c_col,
                                                            const double* __restrict__ cv,
                                                            const uint64_t* __restrict__ noff,
                                                            uint32_t* __restrict__ ncol, double* __restrict__ nval,
                                                            uint32_t* __restrict__ keep,
                                                            uint8_t* __restrict__ mask) {
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= nc) return;
    uint64_t w = noff[c];
    for (uint32_t p = c_off[c]; p < c_off[c + 1]; ++p) {
        const bool k = fabs(cv[p]) > 1e-30;
        mask[p] = k;
        if (k) {
            ncol[w] = c_col[p];
            nval[w] = cv[p];
            keep[w] = p;
            ++w;
        }
    }
}

}  // namespace

// A P numeric of a transfer.
static void launch_galerkin_ap(const DeviceAmg::RefreshLevel& R, const double* aval, int* flags, hipStream_t s) {
    galerkin_ap_entries_kernel<<<grid64(R.apnnz), kBlock, 0, s>>>(R.apnnz, R.ap_row, R.ap_col, R.arow, R.acol, aval,
                                                                  R.prow, R.pcol, R.pval, R.t_off, R.t_row, R.t_pos,
                                                                  R.apv, flags);
}

// P^T (AP) numeric of a transfer.
static void launch_galerkin_c(const DeviceAmg::RefreshLevel& R, const uint8_t* keep_mask, int* flags,
                              hipStream_t s) {
    const CProduct g{R.t_off, R.t_row, R.t_pos, R.prow, R.pval, R.ap_off, R.ap_col, R.apv,
                     R.c_off, R.c_col, R.cv,    keep_mask, flags};
    galerkin_c_rows_kernel<16, kLightRow><<<(R.nc + 15) / 16, kBlock, 0, s>>>(R.nc, nullptr, g);
    if (R.c_nmid) galerkin_c_rows_kernel<64, kTileCols><<<(R.c_nmid + 3) / 4, kBlock, 0, s>>>(R.c_nmid, R.c_mid, g);
    if (R.c_nheavy) galerkin_c_tiles_kernel<<<R.c_nheavy, 1024, kTileBytes, s>>>(R.c_heavy, g);
}

// Lists of the mid and heavy coarse rows of a transfer.
static void list_c_rows(DeviceAmg::RefreshLevel& R, hipStream_t s) {
    HIP_OK(hipFuncSetAttribute(reinterpret_cast<const void*>(galerkin_c_tiles_kernel),
                               hipFuncAttributeMaxDynamicSharedMemorySize, int(kTileBytes)));
    uint32_t* cnt = dalloc<uint32_t>(2);
    uint32_t h[2] = {0, 0};
    HIP_OK(hipMemsetAsync(cnt, 0, 8, s));
    c_row_kinds_kernel<<<grid64(R.nc), kBlock, 0, s>>>(R.nc, R.c_off, R.t_off, cnt, nullptr, nullptr);
    HIP_OK(hipMemcpyAsync(h, cnt, 8, hipMemcpyDeviceToHost, s));
    HIP_OK(hipStreamSynchronize(s));
    R.c_nmid = h[0];
    R.c_nheavy = h[1];
    R.c_mid = dalloc<uint32_t>(R.c_nmid);
    R.c_heavy = dalloc<uint2>(R.c_nheavy);
    if (h[0] || h[1]) {
        HIP_OK(hipMemsetAsync(cnt, 0, 8, s));
        c_row_kinds_kernel<<<grid64(R.nc), kBlock, 0, s>>>(R.nc, R.c_off, R.t_off, cnt, R.c_mid, R.c_heavy);
        HIP_OK(hipStreamSynchronize(s));
    }
    dfree(cnt);
}

void DeviceAmg::release_refresh() {
    for (auto& R : rf_) free_refresh_level(R);
    rf_.clear();
    dfree(rf_flags_);
    dfree(rf_work_);
    dfree(rf_view_);
    dfree(rf_lz_);
    dfree(rf_ub_);
    dfree(rf_long_);
    rf_nlong_ = 0;
    rf_view_host_.clear();
    rf_cur_ = 0;
}

void DeviceAmg::free_refresh_level(RefreshLevel& R) {
    for (uint32_t** p : {&R.arow, &R.acol, &R.src, &R.perm, &R.prow, &R.pcol, &R.ap_off, &R.ap_col, &R.ap_row,
                         &R.c_off, &R.c_col, &R.t_off, &R.t_row, &R.t_pos, &R.keep})
        dfree(*p);
    for (double** p : {&R.aval[0], &R.aval[1], &R.inv[0], &R.inv[1], &R.pval, &R.apv, &R.cv}) dfree(*p);
    dfree(R.keep_mask);
    dfree(R.c_mid);
    dfree(R.c_heavy);
}

bool DeviceAmg::build_refresh(const HostHierarchy& h, std::string& err, std::vector<RefreshLevel>* adopt) {
    release_refresh();
    const size_t L = h.lv.size();
    if (L != lv_.size() || (adopt && adopt->size() != L)) {
        err = "refresh plan: hierarchy depth mismatch";
        return false;
    }
    if (adopt) {
        rf_ = std::move(*adopt);
        adopt->clear();
    } else {
        rf_.resize(L);
    }
    for (size_t l = 0; l < L; ++l) {
        const HostLevel& H = h.lv[l];
        RefreshLevel& R = rf_[l];
        if (!adopt) {
            R.n = H.A.n;
            R.nnz = H.A.nnz();
            R.arow = upload(H.A.rowp, stream_);
            R.acol = upload(H.A.cols, stream_);
            R.aval[0] = upload(H.A.vals, stream_);
            R.inv[0] = upload(H.inv_diag, stream_);
            if (l + 1 < L) {
                R.nc = H.P.ncols;
                R.pnnz = H.P.nnz();
                R.prow = upload(H.P.rowp, stream_);
                R.pcol = upload(H.P.cols, stream_);
                R.pval = upload(H.P.vals, stream_);
                R.apnnz = H.ap_col.size();
                R.ap_off = upload(H.ap_off, stream_);
                R.ap_col = upload(H.ap_col, stream_);
                R.cnnz = H.c_col.size();
                R.c_off = upload(H.c_off, stream_);
                R.c_col = upload(H.c_col, stream_);
                R.t_off = upload(H.t_off, stream_);
                R.t_row = upload(H.t_row, stream_);
                R.t_pos = upload(H.t_pos, stream_);
                std::vector<uint8_t> mask(R.cnnz, 0);
                for (uint32_t p : H.c_keep) mask[p] = 1;
                R.keep_mask = upload(mask, stream_);
                R.keep = upload(H.c_keep, stream_);
            }
        }
        if (R.n != H.A.n || R.nnz != H.A.nnz()) {
            err = "refresh plan: level size mismatch";
            return false;
        }
        if (!R.aval[1]) R.aval[1] = dalloc<double>(R.nnz);
        if (!R.inv[1]) R.inv[1] = dalloc<double>(R.n);
        if (l + 1 < L) {
            if (!R.apv) R.apv = dalloc<double>(R.apnnz);
            if (!R.cv) R.cv = dalloc<double>(R.cnnz);
            if (!R.ap_row) {
                R.ap_row = dalloc<uint32_t>(R.apnnz);
                row_index_kernel<<<grid64(R.n), kBlock, 0, stream_>>>(R.n, R.ap_off, R.ap_row);
            }
            if (!R.c_mid) list_c_rows(R, stream_);
        }
        // src: solve-ordered CSR position -> reference entry (rows relabelled
        // by the solve ordering, entry order kept).
        const auto& perm = lv_[l].new_of_old;
        std::vector<uint32_t> newp(size_t(R.n) + 1, 0);
        for (uint32_t i = 0; i < R.n; ++i) newp[perm[i] + 1] = H.A.rowp[i + 1] - H.A.rowp[i];
        for (uint32_t i = 0; i < R.n; ++i) newp[i + 1] += newp[i];
        std::vector<uint32_t> src(R.nnz);
        for (uint32_t i = 0; i < R.n; ++i) {
            uint32_t w = newp[perm[i]];
            for (uint32_t k = H.A.rowp[i]; k < H.A.rowp[i + 1]; ++k) src[w++] = k;
        }
        R.src = upload(src, stream_);
        R.perm = upload(perm, stream_);
    }
    {
        std::vector<uint2> rows_;
        auto length = [&](uint2 r) { return h.lv[r.x].A.rowp[r.y + 1] - h.lv[r.x].A.rowp[r.y]; };
        for (uint32_t l = 0; l < L; ++l)
            for (uint32_t i = 0; i < rf_[l].n; ++i)
                if (const uint2 r{l, i}; length(r) > kGershgorinRow) rows_.push_back(r);
        std::stable_sort(rows_.begin(), rows_.end(), [&](uint2 a, uint2 b) { return length(a) > length(b); });
        rf_nlong_ = uint32_t(rows_.size());
        if (rf_nlong_) rf_long_ = upload(rows_, stream_);
    }
    // What the batched kernels see of the levels.
    rf_view_host_.assign(L + 1, RefreshView{});
    uint32_t wg = 0, blk = 0, rows = 0;
    for (size_t l = 0; l <= L; ++l) {
        RefreshView& V = rf_view_host_[l];
        V.first_wg = wg;
        V.first_block = blk;
        V.row0 = rows;
        if (l == L) break;
        const RefreshLevel& R = rf_[l];
        const DevLevel& D = lv_[l];
        V.n = R.n;
        V.blocks = D.A.blocks;
        V.rowp = D.A.rowp;
        V.cols = D.A.cols;
        V.vals = D.A.v64;
        V.inv = D.inv64;
        V.perm = R.perm;
        V.arow = R.arow;
        V.acol = R.acol;
        for (int k = 0; k < 2; ++k) {
            V.aval[k] = R.aval[k];
            V.rinv[k] = R.inv[k];
        }
        wg += grid64(R.n);
        blk += D.A.nblocks;
        rows += R.n;
    }
    rf_view_ = upload(rf_view_host_, stream_);
    rf_flags_ = dalloc<int>(kFlagCount * L);
    rf_lz_ = dalloc<LanczosState>(L);
    rf_ub_ = dalloc<double>(L);
    // Five Lanczos vectors over all rows, tile sums (Gershgorin: row scales
    // and workgroup maxima).
    rf_work_ = dalloc<double>(5 * uint64_t(rows) + wg);
    rf_cur_ = 0;
    const RefreshLevel& C = rf_.back();
    rf_coarsest_ = HCsr{};
    if (C.n <= 16) {
        const HCsr& A = h.lv.back().A;
        rf_coarsest_.n = rf_coarsest_.ncols = A.n;
        rf_coarsest_.rowp = A.rowp;
        rf_coarsest_.cols = A.cols;
        rf_coarsest_.vals = A.vals;
    }
    HIP_OK(hipStreamSynchronize(stream_));
    return true;
}

void DeviceAmg::launch_gershgorin(uint32_t slot) {
    const RefreshView& end = rf_view_host_.back();
    double* sd = rf_work_;
    double* bmax = rf_work_ + 5 * uint64_t(end.row0);
    gershgorin_sd_kernel<<<end.first_wg, kBlock, 0, stream_>>>(rf_view_, slot, sd, rf_flags_);
    double* sums = rf_work_ + end.row0;
    if (rf_nlong_)
        gershgorin_long_kernel<<<(rf_nlong_ + 3) / 4, kBlock, 0, stream_>>>(rf_view_, slot, rf_nlong_, rf_long_, sd,
                                                                            sums);
    gershgorin_rows_kernel<<<end.first_wg, kBlock, 0, stream_>>>(rf_view_, slot, sd, sums, bmax, rf_flags_);
    max_reduce_kernel<<<uint32_t(rf_.size()), 1024, 0, stream_>>>(rf_view_, bmax, rf_ub_);
}

// Fetches the levels' flags and Gershgorin bounds and, for a dense coarsest
// level, its values of `slot`.
void DeviceAmg::read_refresh(bool coarsest, uint32_t slot) {
    rf_host_flags_.resize(kFlagCount * rf_.size());
    rf_host_ub_.resize(rf_.size());
    HIP_OK(hipMemcpyAsync(rf_host_flags_.data(), rf_flags_, rf_host_flags_.size() * sizeof(int),
                          hipMemcpyDeviceToHost, stream_));
    HIP_OK(hipMemcpyAsync(rf_host_ub_.data(), rf_ub_, rf_host_ub_.size() * 8, hipMemcpyDeviceToHost, stream_));
    if (coarsest)
        HIP_OK(hipMemcpyAsync(rf_coarsest_.vals.data(), rf_.back().aval[slot], rf_coarsest_.vals.size() * 8,
                              hipMemcpyDeviceToHost, stream_));
    HIP_OK(hipStreamSynchronize(stream_));
}

bool DeviceAmg::gershgorin_bound(bool& certified, double& mb) const {
    mb = 0.0;
    certified = true;
    for (size_t l = 0; l < rf_.size() && certified; ++l) {
        const double ub = rf_host_ub_[l];
        if (rf_host_flags_[l * kFlagCount + kBadGershgorin] || !std::isfinite(ub) || !(ub > 0.0)) certified = false;
        else mb = std::max(mb, ub);
    }
    return true;
}

std::vector<double> DeviceAmg::lanczos_bounds(const AmgConfig& cfg) {
    // Lanczos estimate of lambda_max(D^-1 A) per level on the committed
    // solve-ordered FP64 matrices (the host estimate's arithmetic).
    const uint32_t steps = cfg.lambda_iterations;
    if (steps > kLanczosMax) throw std::runtime_error("too many Lanczos steps");
    const RefreshView& end = rf_view_host_.back();
    const uint32_t L = uint32_t(lv_.size()), g = end.first_wg;
    const uint64_t n = end.row0;
    double* q = rf_work_;
    const LanczosVectors z{q, q + n, q + 2 * n, q + 3 * n, q + 4 * n, q + 5 * n};
    lanczos_init_kernel<<<g, kBlock, 0, stream_>>>(rf_view_, rf_lz_, z);
    lanczos_total_kernel<0><<<L, 1024, 0, stream_>>>(rf_view_, steps, rf_lz_, z.tile);
    lanczos_scale_kernel<<<g, kBlock, 0, stream_>>>(rf_view_, rf_lz_, z);
    for (uint32_t k = 0; k < steps; ++k) {
        lanczos_spmv_kernel<<<end.first_block, kBlock, 0, stream_>>>(rf_view_, rf_lz_, z);
        lanczos_dot_kernel<<<g, kBlock, 0, stream_>>>(rf_view_, rf_lz_, z);
        lanczos_total_kernel<1><<<L, 1024, 0, stream_>>>(rf_view_, steps, rf_lz_, z.tile);
        lanczos_update_kernel<<<g, kBlock, 0, stream_>>>(rf_view_, rf_lz_, z);
        lanczos_total_kernel<2><<<L, 1024, 0, stream_>>>(rf_view_, steps, rf_lz_, z.tile);
        if (k + 1 < steps) lanczos_next_kernel<<<g, kBlock, 0, stream_>>>(rf_view_, rf_lz_, z);
    }
    std::vector<LanczosState> st(L);
    HIP_OK(hipMemcpyAsync(st.data(), rf_lz_, L * sizeof(LanczosState), hipMemcpyDeviceToHost, stream_));
    HIP_OK(hipStreamSynchronize(stream_));
    std::vector<double> lambda;
    for (const LanczosState& S : st)
        lambda.push_back(tridiag_max_eigenvalue(std::vector<double>(S.alpha, S.alpha + S.count),
                                                std::vector<double>(S.beta, S.beta + S.count)));
    return lambda;
}

bool DeviceAmg::finish_setup(const AmgConfig& cfg, double& omega, std::vector<double>& lambda, std::string& err) {
    bool certified = false;
    double mb = 0.0;
    const auto t0 = std::chrono::steady_clock::now();
    HIP_OK(hipMemsetAsync(rf_flags_, 0, sizeof(int) * kFlagCount * rf_.size(), stream_));
    launch_gershgorin(rf_cur_);
    read_refresh(false, rf_cur_);
    gershgorin_bound(certified, mb);
    lambda.clear();
    if (cfg.wants_lambda()) lambda = lanczos_bounds(cfg);
    if (std::getenv("CFDXHIP_SETUP_TRACE"))
        std::fprintf(stderr, "[build] damping certificate and eigenvalue bounds %.3f s\n",
                     std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count());
    double wv = 0.0;
    if (certified) {
        wv = std::min(cfg.omega, 1.8 / mb);
        certified = std::isfinite(wv) && wv > 0.0 && wv < 2.0;
    }
    if (!certified) {
        if (cfg.require_certificate) {
            err = "Jacobi stability certificate requires positive finite diagonals and a finite Gershgorin bound";
            return false;
        }
        wv = cfg.omega;
    }
    omega_ = wv;
    omega = wv;
    if (!lambda.empty()) set_chebyshev_lambda(lambda);
    return true;
}

bool DeviceAmg::refresh_device(const double* d_vals, const AmgConfig& cfg, double& omega, std::vector<double>& lambda,
                               std::string& err, bool& pattern_changed) {
    pattern_changed = false;
    if (rf_.empty()) {
        err = "numeric update requires an existing hierarchy";
        return false;
    }
    const uint32_t stg = rf_cur_ ^ 1u;
    const size_t L = rf_.size();
    // Every level is recomputed into the staged slot; the error flags, the
    // Gershgorin bounds and the coarsest values come back together. A level
    // that follows a failed one computes on what it finds (patterns are
    // fixed), and the first failure in the order of the checks is reported.
    HIP_OK(hipMemsetAsync(rf_flags_, 0, sizeof(int) * kFlagCount * L, stream_));
    // Level 0 values come in the caller's (reference) order.
    HIP_OK(hipMemcpyAsync(rf_[0].aval[stg], d_vals, rf_[0].nnz * 8, hipMemcpyDeviceToDevice, stream_));
    finite_check_kernel<<<grid64(rf_[0].nnz), kBlock, 0, stream_>>>(rf_[0].nnz, rf_[0].aval[stg], rf_flags_);
    for (size_t l = 0; l < L; ++l) {
        RefreshLevel& R = rf_[l];
        int* flags = rf_flags_ + l * kFlagCount;
        inv_diag_kernel<<<grid64(R.n), kBlock, 0, stream_>>>(R.n, R.arow, R.acol, R.aval[stg], R.inv[stg], flags);
        if (l + 1 == L) break;
        launch_galerkin_ap(R, R.aval[stg], flags, stream_);
        launch_galerkin_c(R, R.keep_mask, flags, stream_);
        RefreshLevel& N = rf_[l + 1];
        gather_idx_kernel<double><<<grid64(N.nnz), kBlock, 0, stream_>>>(N.nnz, R.keep, R.cv, N.aval[stg]);
    }
    launch_gershgorin(stg);
    const bool dense = rf_.back().n <= 16;
    read_refresh(dense, stg);
    for (size_t l = 0; l < L; ++l) {
        const int* f = rf_host_flags_.data() + l * kFlagCount;
        if (f[kBadInput]) err = "non-finite matrix value";
        else if (f[kBadDiagonal]) err = "invalid or zero diagonal at level " + std::to_string(l);
        else if (f[kBadProduct]) err = "non-finite Galerkin product at level " + std::to_string(l);
        else if (f[kPatternChanged]) {
            err = "Galerkin pattern changed at level " + std::to_string(l + 1);
            pattern_changed = true;
        } else {
            continue;
        }
        return false;
    }
    // Damping certificate on the staged values.
    bool certified = false;
    double mb = 0.0;
    gershgorin_bound(certified, mb);
    double wv = 0.0;
    if (certified) {
        wv = std::min(cfg.omega, 1.8 / mb);
        certified = std::isfinite(wv) && wv > 0.0 && wv < 2.0;
    }
    if (!certified) {
        if (cfg.require_certificate) {
            err = "Jacobi stability certificate failed on refreshed values";
            return false;
        }
        wv = omega_;
    }
    // Coarsest dense LU from the refreshed coarsest values (at most 16 rows).
    CoarseLU lu;
    bool lu_ok = false;
    if (dense) lu_ok = factor_coarsest(rf_coarsest_, lu, cns_);
    // Commit: values into the solve-ordered CSR / SELL copies, inverse
    // diagonals, damping, Chebyshev coefficients, coarsest factors.
    for (size_t l = 0; l < L; ++l) {
        RefreshLevel& R = rf_[l];
        DevLevel& D = lv_[l];
        commit_values_kernel<<<grid64(R.nnz), kBlock, 0, stream_>>>(R.nnz, R.src, R.aval[stg], D.A.v64, D.A.v32);
        commit_diagonal_kernel<<<grid64(R.n), kBlock, 0, stream_>>>(R.n, R.perm, R.inv[stg], D.inv64, D.inv32);
        sell_values(D.A, stream_, false);
        if (D.A.hvals) {
            const uint32_t rows = D.A.nslices * kSellRows;
            sell_half_values_kernel<<<grid_for(rows), kBlock, 0, stream_>>>(D.n, rows, D.A.soff, D.A.s32, D.inv32,
                                                                             D.A.hvals);
        }
    }
    refill_tail();
    rf_cur_ = stg;
    omega_ = wv;
    omega = wv;
    // Eigenvalue estimates of the committed hierarchy (they decide no
    // acceptance, so they are formed after the commit, on the solve-ordered
    // copies).
    lambda.clear();
    if (cfg.wants_lambda()) {
        lambda = lanczos_bounds(cfg);
        set_chebyshev_lambda(lambda);
    }
    if (dense) {
        lu_.ok = lu_ok;
        if (lu_ok) {
            if (!lu_.piv) {
                lu_.piv = dalloc<uint32_t>(lu.piv.size());
                lu_.factor = dalloc<double>(lu.factor.size());
                lu_.upper = dalloc<double>(lu.upper.size());
            }
            HIP_OK(hipMemcpyAsync(lu_.piv, lu.piv.data(), lu.piv.size() * 4, hipMemcpyHostToDevice, stream_));
            HIP_OK(hipMemcpyAsync(lu_.factor, lu.factor.data(), lu.factor.size() * 8, hipMemcpyHostToDevice, stream_));
            HIP_OK(hipMemcpyAsync(lu_.upper, lu.upper.data(), lu.upper.size() * 8, hipMemcpyHostToDevice, stream_));
        }
    }
    HIP_OK(hipStreamSynchronize(stream_));
    return true;
}

bool DeviceAmg::level_values(size_t level, std::vector<double>& vals) const {
    if (level >= rf_.size()) return false;
    const RefreshLevel& R = rf_[level];
    vals.resize(R.nnz);
    HIP_OK(hipMemcpy(vals.data(), R.aval[rf_cur_], R.nnz * 8, hipMemcpyDeviceToHost));
    return true;
}

// ------------------------------------------ hierarchy construction (SA) --

namespace {

// Exclusive scan of n counts into out[0..n] (out[n] = total); returns the
// total. tiles: scratch of at least ceil(n / kScanTile) + 1 entries.
uint64_t scan_counts(const uint32_t* cnt, uint64_t* out, uint64_t n, hipStream_t s) {
    const uint32_t nt = uint32_t((n + kScanTile - 1) / kScanTile);
    uint64_t* tiles = dalloc<uint64_t>(uint64_t(nt) + 1);
    if (nt) scan_tile_sums_kernel<<<nt, kBlock, 0, s>>>(n, cnt, tiles);
    scan_tiles_kernel<<<1, 1, 0, s>>>(nt, tiles, out + n);
    if (nt) scan_apply_kernel<<<nt, kBlock, 0, s>>>(n, cnt, tiles, out);
    uint64_t total = 0;
    HIP_OK(hipMemcpyAsync(&total, out + n, 8, hipMemcpyDeviceToHost, s));
    HIP_OK(hipStreamSynchronize(s));
    dfree(tiles);
    return total;
}

template <class T>
std::vector<T> download(const T* d, uint64_t n, hipStream_t s) {
    std::vector<T> h(n);
    if (n) HIP_OK(hipMemcpyAsync(h.data(), d, n * sizeof(T), hipMemcpyDeviceToHost, s));
    HIP_OK(hipStreamSynchronize(s));
    return h;
}

// 64-bit offsets narrowed to a CSR's 32-bit row offsets (total checked by
// the caller).
uint32_t* narrow_offsets(const uint64_t* off, uint64_t n, hipStream_t s) {
    uint32_t* o = dalloc<uint32_t>(n + 1);
    narrow_u32_kernel<<<grid64(n + 1), kBlock, 0, s>>>(n + 1, off, o);
    return o;
}

}  // namespace

bool DeviceAmg::build_sa_device(const uint32_t* d_rowp, const uint32_t* d_cols, const double* d_vals, uint32_t n,
                                const AmgConfig& cfg, hipStream_t stream, HostHierarchy& host,
                                std::vector<RefreshLevel>& levels, std::string& err) {
    host = HostHierarchy{};
    for (auto& R : levels) free_refresh_level(R);
    levels.clear();
    auto fail = [&](const std::string& m) {
        for (auto& R : levels) free_refresh_level(R);
        levels.clear();
        host = HostHierarchy{};
        err = m;
        return false;
    };
    int* flags = dalloc<int>(kFlagCount);
    struct FlagsGuard {
        int*& f;
        ~FlagsGuard() { dfree(f); }
    } guard{flags};
    int hflags[kFlagCount];
    auto flagged = [&](int which) {
        HIP_OK(hipMemcpyAsync(hflags, flags, sizeof(hflags), hipMemcpyDeviceToHost, stream));
        HIP_OK(hipStreamSynchronize(stream));
        return hflags[which] != 0;
    };
    HIP_OK(hipMemsetAsync(flags, 0, sizeof(int) * kFlagCount, stream));
    // Level 0: the caller's matrix, copied.
    RefreshLevel L0;
    L0.n = n;
    {
        uint32_t last = 0;
        HIP_OK(hipMemcpyAsync(&last, d_rowp + n, 4, hipMemcpyDeviceToHost, stream));
        HIP_OK(hipStreamSynchronize(stream));
        L0.nnz = last;
    }
    L0.arow = dalloc<uint32_t>(uint64_t(n) + 1);
    L0.acol = dalloc<uint32_t>(L0.nnz);
    L0.aval[0] = dalloc<double>(L0.nnz);
    L0.inv[0] = dalloc<double>(n);
    HIP_OK(hipMemcpyAsync(L0.arow, d_rowp, (uint64_t(n) + 1) * 4, hipMemcpyDeviceToDevice, stream));
    HIP_OK(hipMemcpyAsync(L0.acol, d_cols, L0.nnz * 4, hipMemcpyDeviceToDevice, stream));
    HIP_OK(hipMemcpyAsync(L0.aval[0], d_vals, L0.nnz * 8, hipMemcpyDeviceToDevice, stream));
    levels.push_back(L0);
    inv_diag_kernel<<<grid64(n), kBlock, 0, stream>>>(n, L0.arow, L0.acol, L0.aval[0], L0.inv[0], flags);
    if (flagged(kBadDiagonal)) return fail("invalid or zero diagonal on finest level");
    // CFDXHIP_SETUP_TRACE=1 prints each level's phase times to stderr.
    const bool trace = std::getenv("CFDXHIP_SETUP_TRACE") != nullptr;
    auto clock = [&]() {
        if (trace) HIP_OK(hipStreamSynchronize(stream));
        return std::chrono::steady_clock::now();
    };
    auto secs = [](std::chrono::steady_clock::time_point a, std::chrono::steady_clock::time_point b) {
        return std::chrono::duration<double>(b - a).count();
    };
    unsigned long long* d_fallbacks = reinterpret_cast<unsigned long long*>(dalloc<uint64_t>(1));
    HIP_OK(hipMemsetAsync(d_fallbacks, 0, 8, stream));
    while (levels.back().n > 16 && levels.size() < cfg.max_levels) {
        RefreshLevel& R = levels.back();
        const uint32_t nl = R.n;
        const uint32_t g = grid64(nl);
        const auto c0 = clock();
        // ---- strength graph S and its transpose
        double* thr = dalloc<double>(nl);
        int8_t* mode = dalloc<int8_t>(nl);
        uint32_t* cnt = dalloc<uint32_t>(nl);
        uint64_t* soff = dalloc<uint64_t>(uint64_t(nl) + 1);
        strength_count_kernel<<<g, kBlock, 0, stream>>>(nl, R.arow, R.acol, R.aval[0], R.inv[0], cfg.theta, thr,
                                                        mode, cnt);
        const uint64_t snnz = scan_counts(cnt, soff, nl, stream);
        uint32_t* scol = dalloc<uint32_t>(snnz);
        strength_fill_kernel<<<g, kBlock, 0, stream>>>(nl, R.arow, R.acol, R.aval[0], R.inv[0], thr, mode, soff,
                                                       scol);
        dfree(thr);
        dfree(mode);
        HIP_OK(hipMemsetAsync(cnt, 0, uint64_t(nl) * 4, stream));
        col_count_kernel<<<g, kBlock, 0, stream>>>(nl, soff, scol, cnt);
        uint64_t* toff = dalloc<uint64_t>(uint64_t(nl) + 1);
        scan_counts(cnt, toff, nl, stream);
        uint32_t* tcol = dalloc<uint32_t>(snnz);
        HIP_OK(hipMemsetAsync(cnt, 0, uint64_t(nl) * 4, stream));
        col_fill_kernel<<<g, kBlock, 0, stream>>>(nl, soff, scol, toff, cnt, tcol);
        segment_sort_kernel<uint32_t><<<g, kBlock, 0, stream>>>(nl, toff, tcol);
        // ---- symmetrised neighbourhood, greedy aggregation on the host
        merge_count_kernel<<<g, kBlock, 0, stream>>>(nl, soff, scol, toff, tcol, cnt);
        uint64_t* noff = dalloc<uint64_t>(uint64_t(nl) + 1);
        const uint64_t nnn = scan_counts(cnt, noff, nl, stream);
        if (nnn > UINT32_MAX) return fail("strength graph too large for 32-bit offsets");
        uint32_t* ncol = dalloc<uint32_t>(nnn);
        merge_fill_kernel<<<g, kBlock, 0, stream>>>(nl, soff, scol, toff, tcol, noff, ncol);
        dfree(soff);
        dfree(scol);
        dfree(toff);
        dfree(tcol);
        const auto c1 = clock();
        std::vector<uint64_t> hnoff64 = download(noff, uint64_t(nl) + 1, stream);
        std::vector<uint32_t> hncol = download(ncol, nnn, stream);
        dfree(noff);
        dfree(ncol);
        std::vector<uint32_t> hnoff(hnoff64.begin(), hnoff64.end());
        hnoff64 = {};
        std::vector<uint32_t> agg;
        const uint32_t nc = greedy_aggregation(nl, hnoff, hncol, agg);
        hnoff = {};
        hncol = {};
        if (levels.size() == 1) {
            std::vector<uint32_t> members(nc, 0);
            for (uint32_t a : agg) ++members[a];
            for (uint32_t m : members) host.singleton_aggregates += m == 1;
        }
        uint32_t* d_agg = upload(agg, stream);
        const auto c2 = clock();
        // ---- smoothed prolongator
        const uint64_t scratch = R.nnz + nl;
        uint32_t* pscol = dalloc<uint32_t>(scratch);
        double* psval = dalloc<double>(scratch);
        uint64_t* pskey = dalloc<uint64_t>(scratch);
        smooth_rows_kernel<<<g, kBlock, 0, stream>>>(nl, R.arow, R.acol, R.aval[0], R.inv[0], d_agg, cfg.filter,
                                                     cfg.keep_own ? 1 : 0, pscol, psval, pskey, cnt, d_fallbacks);
        dfree(pskey);
        if (nc == 0 || nc >= nl || coarsening_too_slow(cfg, nc, nl)) {
            dfree(pscol);
            dfree(psval);
            dfree(cnt);
            dfree(d_agg);
            break;
        }
        uint64_t* poff = dalloc<uint64_t>(uint64_t(nl) + 1);
        const uint64_t pnnz = scan_counts(cnt, poff, nl, stream);
        if (pnnz > UINT32_MAX) return fail("prolongator too large for 32-bit offsets");
        R.nc = nc;
        R.pnnz = pnnz;
        R.prow = narrow_offsets(poff, nl, stream);
        R.pcol = dalloc<uint32_t>(pnnz);
        R.pval = dalloc<double>(pnnz);
        compact_from_rows_kernel<uint32_t><<<g, kBlock, 0, stream>>>(nl, R.arow, poff, pscol, R.pcol);
        compact_from_rows_kernel<double><<<g, kBlock, 0, stream>>>(nl, R.arow, poff, psval, R.pval);
        dfree(pscol);
        dfree(psval);
        dfree(poff);
        host.lv.emplace_back();
        host.lv.back().aggregate = std::move(agg);
        dfree(d_agg);
        const auto c3 = clock();
        // ---- Galerkin symbolic: AP, transpose plan, P^T (AP)
        ap_bound_kernel<<<g, kBlock, 0, stream>>>(nl, R.arow, R.acol, R.prow, cnt);
        uint64_t* boff = dalloc<uint64_t>(uint64_t(nl) + 1);
        const uint64_t apub = scan_counts(cnt, boff, nl, stream);
        uint32_t* buf = dalloc<uint32_t>(apub);
        ap_pattern_kernel<<<g, kBlock, 0, stream>>>(nl, R.arow, R.acol, R.prow, R.pcol, boff, buf, cnt);
        uint64_t* apoff = dalloc<uint64_t>(uint64_t(nl) + 1);
        const uint64_t apnnz = scan_counts(cnt, apoff, nl, stream);
        if (apnnz > UINT32_MAX) return fail("Galerkin product too large for 32-bit offsets");
        R.apnnz = apnnz;
        R.ap_off = narrow_offsets(apoff, nl, stream);
        R.ap_col = dalloc<uint32_t>(apnnz);
        compact_from_offsets_kernel<uint32_t><<<g, kBlock, 0, stream>>>(nl, boff, apoff, buf, R.ap_col);
        dfree(buf);
        dfree(boff);
        dfree(apoff);
        dfree(cnt);
        const uint32_t gc = grid64(nc);
        uint32_t* ccnt = dalloc<uint32_t>(nc);
        HIP_OK(hipMemsetAsync(ccnt, 0, uint64_t(nc) * 4, stream));
        t_count_kernel<<<g, kBlock, 0, stream>>>(nl, R.prow, R.pcol, ccnt);
        uint64_t* toff64 = dalloc<uint64_t>(uint64_t(nc) + 1);
        scan_counts(ccnt, toff64, nc, stream);
        uint64_t* tkey = dalloc<uint64_t>(pnnz);
        HIP_OK(hipMemsetAsync(ccnt, 0, uint64_t(nc) * 4, stream));
        t_fill_kernel<<<g, kBlock, 0, stream>>>(nl, R.prow, R.pcol, toff64, ccnt, tkey);
        segment_sort_kernel<uint64_t><<<gc, kBlock, 0, stream>>>(nc, toff64, tkey);
        R.t_off = narrow_offsets(toff64, nc, stream);
        R.t_row = dalloc<uint32_t>(pnnz);
        R.t_pos = dalloc<uint32_t>(pnnz);
        t_split_kernel<<<grid64(pnnz), kBlock, 0, stream>>>(pnnz, tkey, R.t_row, R.t_pos);
        dfree(tkey);
        dfree(toff64);
        c_bound_kernel<<<gc, kBlock, 0, stream>>>(nc, R.t_off, R.t_row, R.ap_off, ccnt);
        uint64_t* cboff = dalloc<uint64_t>(uint64_t(nc) + 1);
        const uint64_t cub = scan_counts(ccnt, cboff, nc, stream);
        uint32_t* cbuf = dalloc<uint32_t>(cub);
        c_pattern_kernel<<<gc, kBlock, 0, stream>>>(nc, R.t_off, R.t_row, R.ap_off, R.ap_col, cboff, cbuf, ccnt);
        uint64_t* coff = dalloc<uint64_t>(uint64_t(nc) + 1);
        const uint64_t cnnz = scan_counts(ccnt, coff, nc, stream);
        if (cnnz > UINT32_MAX) return fail("Galerkin product too large for 32-bit offsets");
        R.cnnz = cnnz;
        R.c_off = narrow_offsets(coff, nc, stream);
        R.c_col = dalloc<uint32_t>(cnnz);
        compact_from_offsets_kernel<uint32_t><<<gc, kBlock, 0, stream>>>(nc, cboff, coff, cbuf, R.c_col);
        dfree(cbuf);
        dfree(cboff);
        dfree(coff);
        const auto c4 = clock();
        // ---- Galerkin numeric and the 1e-30 pruning
        R.apv = dalloc<double>(apnnz);
        R.cv = dalloc<double>(cnnz);
        R.ap_row = dalloc<uint32_t>(apnnz);
        row_index_kernel<<<g, kBlock, 0, stream>>>(nl, R.ap_off, R.ap_row);
        launch_galerkin_ap(R, R.aval[0], flags, stream);
        list_c_rows(R, stream);
        launch_galerkin_c(R, nullptr, flags, stream);
        if (flagged(kBadProduct))
            return fail("invalid Galerkin coarse matrix from level " + std::to_string(levels.size() - 1));
        prune_count_kernel<<<gc, kBlock, 0, stream>>>(nc, R.c_off, R.cv, ccnt);
        uint64_t* noff2 = dalloc<uint64_t>(uint64_t(nc) + 1);
        const uint64_t knnz = scan_counts(ccnt, noff2, nc, stream);
        dfree(ccnt);
        RefreshLevel N;
        N.n = nc;
        N.nnz = knnz;
        N.arow = narrow_offsets(noff2, nc, stream);
        N.acol = dalloc<uint32_t>(knnz);
        N.aval[0] = dalloc<double>(knnz);
        N.inv[0] = dalloc<double>(nc);
        R.keep = dalloc<uint32_t>(knnz);
        R.keep_mask = dalloc<uint8_t>(cnnz);
        prune_fill_kernel<<<gc, kBlock, 0, stream>>>(nc, R.c_off, R.c_col, R.cv, noff2, N.acol, N.aval[0], R.keep,
                                                     R.keep_mask);
        dfree(noff2);
        inv_diag_kernel<<<gc, kBlock, 0, stream>>>(nc, N.arow, N.acol, N.aval[0], N.inv[0], flags);
        if (trace) {
            const auto c5 = clock();
            std::fprintf(stderr,
                         "[setup] level %zu: n %u nnz %llu -> %u: strength+graph %.3f s, greedy (host, with "
                         "copies) %.3f s, P smoothing %.3f s, Galerkin symbolic %.3f s, numeric+prune %.3f s\n",
                         levels.size() - 1, nl, (unsigned long long)R.nnz, nc, secs(c0, c1), secs(c1, c2),
                         secs(c2, c3), secs(c3, c4), secs(c4, c5));
        }
        if (flagged(kBadDiagonal)) {
            // The own-aggregate variant ends the hierarchy at the current
            // level instead (no reference counterpart: the reference rejects).
            if (!cfg.keep_own) {
                levels.push_back(N);
                return fail("invalid Galerkin coarse matrix or zero diagonal at level " +
                            std::to_string(levels.size() - 1));
            }
            free_refresh_level(N);
            RefreshLevel& T = levels.back();
            for (uint32_t** p : {&T.prow, &T.pcol, &T.ap_off, &T.ap_col, &T.ap_row, &T.c_off, &T.c_col,
                                 &T.t_off, &T.t_row, &T.t_pos, &T.keep})
                dfree(*p);
            for (double** p : {&T.pval, &T.apv, &T.cv}) dfree(*p);
            dfree(T.keep_mask);
            T.nc = 0;
            T.pnnz = T.apnnz = T.cnnz = 0;
            dfree(T.c_mid);
            dfree(T.c_heavy);
            T.c_nmid = T.c_nheavy = 0;
            host.lv.pop_back();
            break;
        }
        levels.push_back(N);
    }
    {
        uint64_t fb = 0;
        HIP_OK(hipMemcpyAsync(&fb, d_fallbacks, 8, hipMemcpyDeviceToHost, stream));
        HIP_OK(hipStreamSynchronize(stream));
        host.fallback_rows = fb;
        uint64_t* p = reinterpret_cast<uint64_t*>(d_fallbacks);
        dfree(p);
    }
    // Host mirror: matrices, inverse diagonals, aggregates and transfers.
    host.lv.resize(levels.size());
    for (size_t l = 0; l < levels.size(); ++l) {
        RefreshLevel& R = levels[l];
        HostLevel& H = host.lv[l];
        H.A.n = H.A.ncols = R.n;
        H.A.rowp = download(R.arow, uint64_t(R.n) + 1, stream);
        H.A.cols = download(R.acol, R.nnz, stream);
        H.A.vals = download(R.aval[0], R.nnz, stream);
        H.inv_diag = download(R.inv[0], R.n, stream);
        if (l + 1 < levels.size()) {
            H.P.n = R.n;
            H.P.ncols = R.nc;
            H.P.rowp = download(R.prow, uint64_t(R.n) + 1, stream);
            H.P.cols = download(R.pcol, R.pnnz, stream);
            H.P.vals = download(R.pval, R.pnnz, stream);
        } else {
            H.aggregate.clear();
        }
    }
    return true;
}

}  // namespace cfdxhip
