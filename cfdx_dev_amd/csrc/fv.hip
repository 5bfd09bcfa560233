// Finite-volume geometry and pressure-system assembly on the device.
//
// Reference anchors (physics/steady_incompressible_solver.h unless noted):
//   face geometry (triangle fan)     core/geometry/face_geometry.h:50-90
//   cell centre / volume             core/geometry/cell_geometry.h:49-147
//   build_fv_geometry (2 passes)     physics/finite_volume_transport.h:92-175
//   gauss_gradient_with_boundary     :1634-1750
//   make_mass_flux                   :1842-1905
//   orthogonal coefficient           :1914-1935
//   non-orthogonal (deferred) flux   :1941-1965
//   Rhie-Chow internal flux          :1967-2029
//   corrector assembly               :8048-8181, CSR + gauge :8599-8652
//   scalar diffusion assembly        core/solvers/scalar_diffusion.h:39-163
//
// The assemblies take one row a thread and evaluate every face from both of its
// cells. The reference accumulates the diagonal and the boundary sources in
// global face order; a row visits its cell's faces in ascending face id, so
// every value is bit-identical to the reference (FMA contraction is off). No
// atomics.

#include "fv.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <stdexcept>

#include "amg_setup.h"
#include "kernels.hpp"
#include "parallel.h"

namespace cfdxhip {

#define HIP_OK(expr)                                                                              \
    do {                                                                                          \
        hipError_t e_ = (expr);                                                                   \
        if (e_ != hipSuccess)                                                                     \
            throw std::runtime_error(std::string("HIP error ") + hipGetErrorString(e_) + " at " + \
                                     __FILE__ + ":" + std::to_string(__LINE__));                  \
    } while (0)

namespace {

template <class T>
T* dalloc(uint64_t count) {
    if (count == 0) count = 1;
    void* p = nullptr;
    HIP_OK(hipMalloc(&p, count * sizeof(T)));
    return static_cast<T*>(p);
}
template <class T>
void dfree(T*& p) {
    if (p) (void)hipFree(p);
    p = nullptr;
}
template <class T>
T* upload(const T* h, uint64_t n) {
    T* d = dalloc<T>(n);
    if (n) HIP_OK(hipMemcpy(d, h, n * sizeof(T), hipMemcpyHostToDevice));
    return d;
}
template <class T>
void download(T* h, const T* d, uint64_t n) {
    if (n && h) HIP_OK(hipMemcpy(h, d, n * sizeof(T), hipMemcpyDeviceToHost));
}
inline uint32_t grid_for(uint64_t n) { return uint32_t((n + kBlock - 1) / kBlock); }

struct D3 {
    double x, y, z;
};
__device__ __forceinline__ D3 d3(double x, double y, double z) { return {x, y, z}; }
__device__ __forceinline__ D3 add3(D3 a, D3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ D3 sub3(D3 a, D3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ D3 mul3(D3 a, double s) { return {a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ double dot3(D3 a, D3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ double mag3(D3 a) { return sqrt(a.x * a.x + a.y * a.y + a.z * a.z); }
__device__ __forceinline__ D3 cross3(D3 a, D3 b) {
    return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

struct Soa3 {
    double *x, *y, *z;
    __device__ D3 get(uint32_t i) const { return {x[i], y[i], z[i]}; }
    __device__ void set(uint32_t i, D3 v) const {
        x[i] = v.x;
        y[i] = v.y;
        z[i] = v.z;
    }
};

// -------------------------------------------------------------- geometry --

__global__ __launch_bounds__(kBlock) void face_geometry_kernel(uint32_t nf, const double* __restrict__ px,
                                                              const double* __restrict__ py,
                                                              const double* __restrict__ pz,
                                                              const uint32_t* __restrict__ foff,
                                                              const uint32_t* __restrict__ fvtx, Soa3 fc, Soa3 fs,
                                                              int* __restrict__ err) {
#pragma clang fp contract(off)
    const uint32_t f = blockIdx.x * kBlock + threadIdx.x;
    if (f >= nf) return;
    const uint32_t off = foff[f], nv = foff[f + 1] - off;
    if (nv < 3) {
        err[0] = 1;
        return;
    }
    const uint32_t v0 = fvtx[off];
    const D3 p0 = d3(px[v0], py[v0], pz[v0]);
    D3 S = d3(0.0, 0.0, 0.0), wc = d3(0.0, 0.0, 0.0);
    double tri = 0.0;
    for (uint32_t k = 1; k + 1 < nv; ++k) {
        const uint32_t va = fvtx[off + k], vb = fvtx[off + k + 1];
        const D3 pa = d3(px[va], py[va], pz[va]);
        const D3 pb = d3(px[vb], py[vb], pz[vb]);
        const D3 tS = mul3(cross3(sub3(pa, p0), sub3(pb, p0)), 0.5);
        const double ta = mag3(tS);
        S = add3(S, tS);
        wc = add3(wc, mul3(add3(add3(p0, pa), pb), ta / 3.0));
        tri += ta;
    }
    const double area = mag3(S);
    if (!(tri > 0.0) || !(area > 0.0) || !isfinite(area)) err[0] = 1;
    fc.set(f, mul3(wc, 1.0 / tri));
    fs.set(f, S);
}

// Cell centre: area-weighted face-centre mean (orientation independent).
__global__ __launch_bounds__(kBlock) void cell_centre_kernel(uint32_t nc, const uint32_t* __restrict__ coff,
                                                            const uint32_t* __restrict__ cf, Soa3 fc, Soa3 fs,
                                                            Soa3 cc) {
#pragma clang fp contract(off)
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= nc) return;
    D3 ws = d3(0.0, 0.0, 0.0);
    double total = 0.0;
    for (uint32_t k = coff[c]; k < coff[c + 1]; ++k) {
        const uint32_t f = cf[k];
        const double a = mag3(fs.get(f));
        ws = add3(ws, mul3(fc.get(f), a));
        total += a;
    }
    cc.set(c, total > 0.0 ? mul3(ws, 1.0 / total) : d3(0.0, 0.0, 0.0));
}

__global__ __launch_bounds__(kBlock) void orient_kernel(uint32_t nf, const uint32_t* __restrict__ owner,
                                                       const int32_t* __restrict__ neigh, Soa3 fc, Soa3 fs,
                                                       Soa3 cc) {
#pragma clang fp contract(off)
    const uint32_t f = blockIdx.x * kBlock + threadIdx.x;
    if (f >= nf) return;
    const uint32_t o = owner[f];
    const D3 d = neigh[f] >= 0 ? sub3(cc.get(uint32_t(neigh[f])), cc.get(o)) : sub3(fc.get(f), cc.get(o));
    const D3 s = fs.get(f);
    if (dot3(s, d) < 0.0) fs.set(f, mul3(s, -1.0));
}

__global__ __launch_bounds__(kBlock) void cell_volume_kernel(uint32_t nc, const uint32_t* __restrict__ coff,
                                                            const uint32_t* __restrict__ cf,
                                                            const uint32_t* __restrict__ owner, Soa3 fc, Soa3 fs,
                                                            Soa3 cc, double* __restrict__ vol,
                                                            int* __restrict__ err) {
#pragma clang fp contract(off)
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= nc) return;
    const D3 centre = cc.get(c);
    double sv = 0.0;
    for (uint32_t k = coff[c]; k < coff[c + 1]; ++k) {
        const uint32_t f = cf[k];
        const D3 s = owner[f] == c ? fs.get(f) : mul3(fs.get(f), -1.0);
        sv += dot3(sub3(fc.get(f), centre), s);
    }
    sv /= 3.0;
    const double v = fabs(sv);
    if (!(v > 0.0) || !isfinite(v)) err[0] = 2;
    vol[c] = v;
}

// ---------------------------------------------------------- gradient ----

// Slot stencils: geometry-only data of the cell-wise face loops, built once
// per mesh in slot-major order (entry q * nc + c belongs to the q-th face of
// cell c in its face-list order). A cell loop then reads them coalesced
// instead of gathering the face and neighbour-cell arrays face by face.
//   other: the cell across an internal face, -1 for a boundary face, -2 for
//          an EMPTY face or an unused slot;
//   face:  the face; the top bit is set on the side of a cell that does not
//          own it (also where such a cell lists a boundary face, which the
//          mesh's addressing admits): face_of() makes it an index;
//   w:     the distance weight dn / (dc + dn) of an internal face (the
//          Green-Gauss face interpolation);
//   s:     the face area vector oriented out of the cell.
constexpr uint32_t kFaceReversed = 0x80000000u;
struct Slots {
    int32_t* other;
    uint32_t* face;
    double* w;
    Soa3 s;

    __device__ __forceinline__ static uint32_t face_of(uint32_t entry) { return entry & ~kFaceReversed; }
};

__global__ __launch_bounds__(kBlock) void slot_build_kernel(uint32_t nc, uint32_t D, const uint32_t* __restrict__ coff,
                                                           const uint32_t* __restrict__ cf,
                                                           const uint32_t* __restrict__ owner,
                                                           const int32_t* __restrict__ neigh,
                                                           const uint32_t* __restrict__ patch, uint32_t npatch,
                                                           const uint8_t* __restrict__ kind, Soa3 fc, Soa3 fs,
                                                           Soa3 cc, const double* __restrict__ vol,
                                                           const uint32_t* __restrict__ face_old,
                                                           double4* __restrict__ cell, Slots sl,
                                                           uint8_t* __restrict__ slot_sorted,
                                                           int* __restrict__ err) {
#pragma clang fp contract(off)
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= nc) return;
    const uint32_t deg = coff[c + 1] - coff[c];
    const D3 centre = cc.get(c);
    cell[c] = make_double4(centre.x, centre.y, centre.z, vol[c]);
    for (uint32_t q = 0; q < D; ++q) {
        const size_t idx = size_t(q) * nc + c;
        if (q >= deg) {
            sl.other[idx] = -2;
            sl.face[idx] = 0;
            sl.w[idx] = 0.0;
            sl.s.set(idx, d3(0.0, 0.0, 0.0));
            continue;
        }
        const uint32_t f = cf[coff[c] + q];
        // The slot's place in the cell's faces by caller id (a face listed
        // twice keeps its order).
        const uint32_t id = face_old[f];
        uint32_t before = 0;
        for (uint32_t x = 0; x < deg; ++x) {
            const uint32_t other = face_old[cf[coff[c] + x]];
            before += other < id || (other == id && x < q);
        }
        slot_sorted[size_t(before) * nc + c] = uint8_t(q);
        const bool own = owner[f] == c;
        sl.face[idx] = own ? f : f | kFaceReversed;
        sl.s.set(idx, own ? fs.get(f) : mul3(fs.get(f), -1.0));
        if (neigh[f] >= 0) {
            const uint32_t other = own ? uint32_t(neigh[f]) : owner[f];
            const double dc = mag3(sub3(fc.get(f), centre));
            const double dn = mag3(sub3(cc.get(other), fc.get(f)));
            if (!(dc + dn > 0.0) || !isfinite(dc + dn)) err[0] = 30;
            sl.other[idx] = int32_t(other);
            sl.w[idx] = dn / (dc + dn);
        } else {
            const uint32_t pp = patch[f];
            sl.other[idx] = pp < npatch && kind[pp] == 1 ? -2 : -1;
            sl.w[idx] = 0.0;
        }
    }
}

// Cells go to workgroups by xcd_block: each XCD takes one contiguous range, so
// that the records a cell and its neighbours share are fetched into one L2
// rather than into most of them (a 222k-cell channel's pressure rows: 40 us in
// launch order, 31 so).
__device__ __forceinline__ uint32_t cell_block() { return xcd_block(blockIdx.x, gridDim.x); }

// Slots a thread loads together: the loads of one slot depend on each other
// (cell id, then that cell's record), so a thread that walks them one by one
// waits for two round trips a face. Enough waves are resident to hide most of
// it: the gradient of a 128^3 box takes 157 us one by one, 151 by threes, 146
// by sixes, which cost half again the registers.
constexpr uint32_t kSlotBatch = 3, kRowBatch = 2;

// gauss_gradient_with_boundary over the slot stencils. bc arrays are per
// patch: type 0 none/zero-gradient, 1 fixed value, 2 fixed gradient. The field
// value of cell i is p[i * ps]; kRec writes one record (gx, gy, gz, 0) a cell,
// else three arrays. Bound by the slots' 36 bytes a face and side.
template <bool kRec>
__global__ __launch_bounds__(kBlock) void gauss_gradient_kernel(
    uint32_t nc, uint32_t D, Slots sl, const uint32_t* __restrict__ patch, uint32_t npatch,
    const uint8_t* __restrict__ bct, const double* __restrict__ bcv, Soa3 fc, Soa3 cc, const double* __restrict__ vol,
    const double* __restrict__ p, uint32_t ps, double* __restrict__ grad) {
#pragma clang fp contract(off)
    const uint32_t c = cell_block() * kBlock + threadIdx.x;
    if (c >= nc) return;
    const double pc = p[size_t(c) * ps];
    D3 sum = d3(0.0, 0.0, 0.0);
    for (uint32_t q0 = 0; q0 < D; q0 += kSlotBatch) {
        int32_t o[kSlotBatch];
        double po[kSlotBatch], w[kSlotBatch];
        D3 S[kSlotBatch];
#pragma unroll
        for (uint32_t j = 0; j < kSlotBatch; ++j) {
            const size_t idx = size_t(min(q0 + j, D - 1)) * nc + c;
            o[j] = q0 + j < D ? sl.other[idx] : -2;
            w[j] = sl.w[idx];
            S[j] = sl.s.get(idx);
        }
#pragma unroll
        for (uint32_t j = 0; j < kSlotBatch; ++j) po[j] = p[size_t(o[j] >= 0 ? uint32_t(o[j]) : c) * ps];
#pragma unroll
        for (uint32_t j = 0; j < kSlotBatch; ++j) {
            if (o[j] == -2) continue;
            const D3 Sf = S[j];
            double vf = pc;
            if (o[j] >= 0) {
                vf = w[j] * pc + (1.0 - w[j]) * po[j];
            } else {
                const uint32_t f = sl.face_of(sl.face[size_t(q0 + j) * nc + c]);
                const uint32_t pp = patch[f];
                if (pp < npatch) {
                    if (bct[pp] == 1) {
                        vf = bcv[pp];
                    } else if (bct[pp] == 2) {
                        const D3 out = mul3(Sf, 1.0 / mag3(Sf));
                        vf += bcv[pp] * dot3(sub3(fc.get(f), cc.get(c)), out);
                    }
                }
            }
            sum = add3(sum, mul3(Sf, vf));
        }
    }
    const double invV = 1.0 / vol[c];
    if (kRec) {
        reinterpret_cast<double4*>(grad)[c] = make_double4(sum.x * invV, sum.y * invV, sum.z * invV, 0.0);
    } else {
        grad[c] = sum.x * invV;
        grad[nc + c] = sum.y * invV;
        grad[2 * size_t(nc) + c] = sum.z * invV;
    }
}

__global__ __launch_bounds__(kBlock) void mass_flux_kernel(uint32_t nf, uint32_t nc, const uint32_t* __restrict__ owner,
                                                          const int32_t* __restrict__ neigh,
                                                          const uint32_t* __restrict__ patch, uint32_t npatch,
                                                          const uint8_t* __restrict__ kind,
                                                          const uint8_t* __restrict__ vbt,
                                                          const double* __restrict__ vbv, double rho, Soa3 fs,
                                                          const double* __restrict__ U, double* __restrict__ phi) {
#pragma clang fp contract(off)
    const uint32_t f = blockIdx.x * kBlock + threadIdx.x;
    if (f >= nf) return;
    const uint32_t o = owner[f];
    D3 Uf = d3(U[o], U[nc + o], U[2 * size_t(nc) + o]);
    if (neigh[f] >= 0) {
        const uint32_t n = uint32_t(neigh[f]);
        const D3 Un = d3(U[n], U[nc + n], U[2 * size_t(nc) + n]);
        Uf = add3(mul3(Uf, 1.0 - 0.5), mul3(Un, 0.5));
    } else {
        const uint32_t pp = patch[f];
        if (pp < npatch && (kind[pp] == 1 || kind[pp] == 2)) {
            phi[f] = 0.0;
            return;
        }
        if (pp < npatch && vbt[pp] == 1) Uf = d3(vbv[3 * pp], vbv[3 * pp + 1], vbv[3 * pp + 2]);
    }
    phi[f] = rho * dot3(Uf, fs.get(f));
}

// ---------------------------------------------------------- pressure ----

// Orthogonal coefficient (S.e)(dAU e.e)/|d| of a face and the flux of the
// gradient g beyond its orthogonal part; false when the geometry does not
// admit them.
__device__ __forceinline__ bool face_pressure_terms(D3 Sf, D3 dv, D3 dAU, D3 g, double& coeff, double& flux) {
#pragma clang fp contract(off)
    const double d = mag3(dv);
    const double area = mag3(Sf);
    if (!(d > 0.0) || !isfinite(d) || !(area > 0.0) || !isfinite(area)) return false;
    const D3 e = d3(dv.x / d, dv.y / d, dv.z / d);
    const double oa = dot3(Sf, e);
    if (!(oa > 0.0) || !isfinite(oa)) return false;
    const double rfn = dAU.x * e.x * e.x + dAU.y * e.y * e.y + dAU.z * e.z * e.z;
    coeff = rfn * oa / d;
    const double full = dAU.x * g.x * Sf.x + dAU.y * g.y * Sf.y + dAU.z * g.z * Sf.z;
    const double impl = rfn * dot3(g, e) * oa;
    flux = full - impl;
    return isfinite(coeff) && isfinite(flux);
}

// The cell fields of one assembly as a record a cell, (x, y, z, w), in the
// internal numbering: read in the caller's order, written as one 32-byte
// record, so that a permuted mesh costs one scattered access a cell instead of
// one a field, and a neighbour's fields arrive together. v: 3 x nc.
__global__ __launch_bounds__(kBlock) void pack_cells_kernel(uint32_t nc, const uint32_t* __restrict__ to,
                                                           const double* __restrict__ v,
                                                           const double* __restrict__ w, double4* __restrict__ rec) {
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= nc) return;
    rec[to ? to[c] : c] = make_double4(v[c], v[size_t(nc) + c], v[2 * size_t(nc) + c], w[c]);
}

// The momentum predictor's fields: (U, mu) and (body - grad p, 0) a cell.
// Viscosity must be finite and non-negative; flags[0] = 1 when any is positive
// (diffusion active).
__global__ __launch_bounds__(kBlock) void pack_momentum_kernel(
    uint32_t nc, const uint32_t* __restrict__ to, const double* __restrict__ U, const double* __restrict__ mu,
    const double* __restrict__ gradp, const double* __restrict__ body, double4* __restrict__ rec,
    double4* __restrict__ source, int* __restrict__ flags, int* __restrict__ err) {
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= nc) return;
    const size_t n1 = nc;
    const uint32_t i = to ? to[c] : c;
    const double m = mu[c];
    if (!(m >= 0.0) || !isfinite(m)) err[0] = 40;
    if (m > 0.0) flags[0] = 1;
    double s[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) s[k] = (body ? body[k * n1 + c] : 0.0) - gradp[k * n1 + c];
    rec[i] = make_double4(U[c], U[n1 + c], U[2 * n1 + c], m);
    source[i] = make_double4(s[0], s[1], s[2], 0.0);
}

__global__ __launch_bounds__(kBlock) void fetch_bcs_kernel(uint32_t words, const double* __restrict__ from,
                                                          double* __restrict__ to, int* __restrict__ flags) {
    for (uint32_t i = threadIdx.x; i < words; i += kBlock) to[i] = from[i];
    if (flags && threadIdx.x < 4) flags[threadIdx.x] = 0;
}

// Records (x, y, z, w) a cell out to the caller's order: v 3 x nc, w nc.
__global__ __launch_bounds__(kBlock) void unpack_cells_kernel(uint32_t nc, const uint32_t* __restrict__ from,
                                                             const double4* __restrict__ rec,
                                                             double* __restrict__ v, double* __restrict__ w) {
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= nc) return;
    const double4 r = rec[from ? from[c] : c];
    v[c] = r.x;
    v[size_t(nc) + c] = r.y;
    v[2 * size_t(nc) + c] = r.z;
    w[c] = r.w;
}

// Where the rows of an assembled matrix go: internal cell c fills the entries
// from start[c] (~0: the row is left out) and right-hand side entry row[c];
// rank[k * nc + c] is the entry, counted from the row's start, of the cell's
// k-th slot in ascending caller face id (kNoEntry: boundary face or column
// left out; equal for faces that join one pair, of which there are some when
// shared), diag[c] that of the diagonal.
constexpr uint16_t kNoEntry = 0xffffu;
struct RowMap {
    const uint32_t *start, *row;
    const uint16_t *rank, *diag;
    int shared;
};

// Builds them from a plan's pattern (caller numbering, rows ascending; row and
// column ref left out): one internal cell a thread.
__global__ __launch_bounds__(kBlock) void map_rows_kernel(uint32_t nc, uint32_t D, const uint32_t* __restrict__ coff,
                                                          const uint8_t* __restrict__ slot_sorted,
                                                          const int32_t* __restrict__ other,
                                                          const uint32_t* __restrict__ cell_old,
                                                          const uint32_t* __restrict__ rowp,
                                                          const uint32_t* __restrict__ cols, uint32_t ref,
                                                          uint32_t* __restrict__ start, uint32_t* __restrict__ row,
                                                          uint16_t* __restrict__ rank, uint16_t* __restrict__ diag) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= nc) return;
    const uint32_t c = cell_old[i], deg = coff[i + 1] - coff[i];
    const bool kept = c != ref;
    const uint32_t r = c - (c > ref ? 1u : 0u), lo = kept ? rowp[r] : 0u, hi = kept ? rowp[r + 1] : 0u;
    auto place = [&](uint32_t col) {
        uint32_t a = lo, b = hi;
        while (a < b) {
            const uint32_t mid = a + ((b - a) >> 1);
            if (cols[mid] < col) a = mid + 1;
            else b = mid;
        }
        return uint16_t(a - lo);
    };
    start[i] = kept ? lo : 0xffffffffu;
    row[i] = kept ? r : 0xffffffffu;
    diag[i] = kept ? place(r) : kNoEntry;
    for (uint32_t k = 0; k < D; ++k) {
        uint16_t at = kNoEntry;
        if (kept && k < deg) {
            const int32_t o = other[size_t(slot_sorted[size_t(k) * nc + i]) * nc + i];
            const uint32_t oc = o >= 0 ? cell_old[o] : ref;
            if (o >= 0 && oc != ref) at = place(oc - (oc > ref ? 1u : 0u));
        }
        rank[size_t(k) * nc + i] = at;
    }
}

// A wave's rows from LDS to the matrix: row i of the wave (its length len and
// first nonzero start held by lane i) lies at rows + i * stride. Eight lanes
// share a row, so that a row of a randomly numbered mesh is written in one or
// two requests rather than one a value: those go to memory in 32-byte pieces.
__device__ __forceinline__ void store_rows(const double* rows, uint32_t stride, uint32_t start, uint32_t len,
                                           double* __restrict__ vals) {
    const uint32_t lane = threadIdx.x & 63u, e = lane & 7u;
#pragma unroll
    for (uint32_t r0 = 0; r0 < 64; r0 += 8) {
        const uint32_t r = r0 + (lane >> 3);
        const uint32_t at = __shfl(start, r), n = __shfl(len, r);
        for (uint32_t k = e; k < n; k += 8) vals[size_t(at) + k] = rows[r * stride + k];
    }
}

// The block's own records in LDS: on the curve most neighbours of a cell lie in
// its block, and gathers through L1 bound the kernels that take all of a
// neighbour's fields from memory.
struct Near {
    double2* at;  // [half][kBlock]
    uint32_t first;

    __device__ __forceinline__ void put(uint32_t k, double4 v) const {
        at[2 * k * kBlock + threadIdx.x] = make_double2(v.x, v.y);
        at[(2 * k + 1) * kBlock + threadIdx.x] = make_double2(v.z, v.w);
    }
    __device__ __forceinline__ bool has(uint32_t c) const { return c - first < uint32_t(kBlock); }
    __device__ __forceinline__ double4 get(uint32_t k, uint32_t c) const {
        const double2 a = at[2 * k * kBlock + (c - first)], b = at[(2 * k + 1) * kBlock + (c - first)];
        return make_double4(a.x, a.y, b.x, b.y);
    }
};

// LDS of a workgroup that assembles rows of up to D + 1 entries beside nrec
// staged records: the rows take the records' place once those are read.
// Hexahedra (6 slots) take 36 KB and polyhedra up to kRowSlots 50 KB, so three
// or more workgroups, what the registers allow, share a CU's 160 KB.
constexpr uint32_t kRowSlots = 12;
constexpr uint32_t kMomNear = 2;  // records a momentum row stages: cell, fields
inline size_t row_lds(uint32_t D, uint32_t nrec) {
    return size_t(kBlock) * 8 * (D + std::max(4 * nrec, D + 1));
}

// One row of the pressure system per thread (internal cell c): continuity in
// cell-face list order (+-phiHbyA, -+Rhie-Chow flux of the pressure), the
// diagonal = internal coefficients then fixed-pressure boundary coefficients,
// both in ascending caller face id, off-diagonals 0 - coefficient of each
// joining face, rhs = -continuity + boundary sources; weights are the default
// w = 1/2. Every face is evaluated from both of its cells: its flux changes
// sign and its coefficient is the same to the last bit from either side
// (differences, the area vector and so the unit vector negate exactly, and the
// weighted sums commute), so nothing has to pass between the cells. Bound by
// memory: 36 bytes of stencil a slot, three 32-byte records a cell that its
// neighbours share, the row's values; the arithmetic is free beside it (taking
// it out changed nothing). kLds: the slots' coefficients wait for the second
// order in LDS, the block's records are staged and the rows leave by
// store_rows; else (many slots a cell) coefficients wait in sbuf and values
// are written one by one. On a 128^3 box of randomly numbered cells: 312 us;
// 587 with values written one by one and all neighbours' records read from
// memory (294 of it the writes, 125 the gathers); 762 as a pass over faces
// that scattered its terms to the cells, one over cells and one over nonzeros.
template <bool kLds>
__global__ __launch_bounds__(kBlock) void pressure_row_kernel(
    uint32_t nc, uint32_t D, const uint32_t* __restrict__ coff, const uint8_t* __restrict__ slot_sorted, Slots sl,
    const uint32_t* __restrict__ patch, uint32_t npatch, const uint8_t* __restrict__ pbt,
    const double* __restrict__ pbv, double rho, Soa3 fc, const double4* __restrict__ cell,
    const double4* __restrict__ fields, const double4* __restrict__ grad, const double* __restrict__ phi,
    double* __restrict__ sbuf, RowMap rm, double* __restrict__ vals, double* __restrict__ rhs,
    int* __restrict__ err) {
#pragma clang fp contract(off)
    extern __shared__ double2 row_shared[];
    const uint32_t first = cell_block() * kBlock;
    const bool live = first + threadIdx.x < nc;
    const uint32_t c = live ? first + threadIdx.x : nc - 1;  // the last block's spare threads only keep step
    double* lds = reinterpret_cast<double*>(row_shared);
    double* cbuf = kLds ? lds + threadIdx.x : sbuf + c;
    const size_t cs = kLds ? size_t(kBlock) : size_t(nc);
    const Near near{reinterpret_cast<double2*>(lds + size_t(D) * kBlock), first};
    const uint32_t deg = live ? coff[c + 1] - coff[c] : 0;
    const double4 C = cell[c], A = fields[c], G = grad[c];
    if (kLds) {
        near.put(0, C);
        near.put(1, A);
        near.put(2, G);
        __syncthreads();
    }
    const double wh = 0.5;
    const D3 ra = d3(wh * C.w * A.x, wh * C.w * A.y, wh * C.w * A.z);
    const D3 gh = d3(wh * G.x, wh * G.y, wh * G.z);
    double cont = 0.0;
    bool fixed = false;
    for (uint32_t q0 = 0; q0 < D; q0 += kRowBatch) {
        int32_t o[kRowBatch];
        uint32_t f[kRowBatch];
        double ph[kRowBatch];
        D3 S[kRowBatch];
        double4 Cn[kRowBatch], An[kRowBatch], Gn[kRowBatch];
#pragma unroll
        for (uint32_t j = 0; j < kRowBatch; ++j) {
            const size_t idx = size_t(min(q0 + j, D - 1)) * nc + c;
            o[j] = q0 + j < deg ? sl.other[idx] : -3;
            f[j] = sl.face[idx];
            S[j] = sl.s.get(idx);
        }
#pragma unroll
        for (uint32_t j = 0; j < kRowBatch; ++j) {
            const uint32_t n = o[j] >= 0 ? uint32_t(o[j]) : c;
            ph[j] = phi[sl.face_of(f[j])];
            if (kLds && near.has(n)) {
                Cn[j] = near.get(0, n);
                An[j] = near.get(1, n);
                Gn[j] = near.get(2, n);
            } else {
                Cn[j] = cell[n];
                An[j] = fields[n];
                Gn[j] = grad[n];
            }
        }
#pragma unroll
        for (uint32_t j = 0; j < kRowBatch; ++j) {
            if (o[j] == -3) continue;
            double cf = 0.0;
            cont += f[j] & kFaceReversed ? -ph[j] : ph[j];
            if (o[j] >= 0) {
                const D3 dAU = add3(ra, d3(wh * Cn[j].w * An[j].x, wh * Cn[j].w * An[j].y, wh * Cn[j].w * An[j].z));
                const D3 gp = add3(gh, d3(wh * Gn[j].x, wh * Gn[j].y, wh * Gn[j].z));
                const D3 dv = d3(Cn[j].x - C.x, Cn[j].y - C.y, Cn[j].z - C.z);
                double ic = 0.0, nof = 0.0;
                if (!face_pressure_terms(S[j], dv, dAU, gp, ic, nof)) err[0] = 3;
                cf = rho * ic;
                cont -= rho * (ic * (An[j].w - A.w) + nof);
            } else {
                const uint32_t pp = patch[sl.face_of(f[j])];
                fixed |= pp < npatch && pbt[pp] == 1;
            }
            cbuf[(q0 + j) * cs] = cf;
        }
    }
    if (kLds) __syncthreads();  // the rows take the records' place
    const uint32_t start = rm.start[c], stride = D + 1;
    double* row = kLds ? lds + size_t(D) * kBlock + threadIdx.x * stride : vals + size_t(start);
    double d = 0.0;
    uint32_t len = 0;
    if (rm.shared && start != 0xffffffffu) {
        for (uint32_t k = 0; k < deg; ++k) {
            const uint16_t r = rm.rank[size_t(k) * nc + c];
            if (r != kNoEntry) row[r] = 0.0;
        }
    }
    for (uint32_t k = 0; k < deg; ++k) {
        const double cf = cbuf[slot_sorted[size_t(k) * nc + c] * cs];
        d += cf;
        const uint16_t r = rm.rank[size_t(k) * nc + c];
        if (r == kNoEntry) continue;
        len = max(len, uint32_t(r) + 1u);
        row[r] = (rm.shared ? row[r] : 0.0) - cf;
    }
    double b = -cont;
    if (fixed) {
        const D3 dAU = d3(C.w * A.x, C.w * A.y, C.w * A.z);
        for (uint32_t k = 0; k < deg; ++k) {
            const size_t idx = size_t(slot_sorted[size_t(k) * nc + c]) * nc + c;
            if (sl.other[idx] >= 0) continue;
            const uint32_t f = sl.face_of(sl.face[idx]);
            const uint32_t pp = patch[f];
            if (!(pp < npatch && pbt[pp] == 1)) continue;
            double bc = 0.0, def = 0.0;
            if (!face_pressure_terms(sl.s.get(idx), sub3(fc.get(f), d3(C.x, C.y, C.z)), dAU, d3(G.x, G.y, G.z), bc,
                                     def)) {
                err[0] = 3;
                continue;
            }
            d += rho * bc;
            b += rho * (bc * (pbv[pp] - A.w) + def);
        }
    }
    const bool kept = live && start != 0xffffffffu;
    if (kept) {
        const uint32_t r = rm.diag[c];
        row[r] = d;
        len = max(len, r + 1u);
        rhs[rm.row[c]] = b;
    }
    if (kLds) {
        wave_fence();
        store_rows(lds + size_t(D) * kBlock + (threadIdx.x & ~63u) * stride, stride, start, kept ? len : 0, vals);
    }
}

// CSR values of the diffusion system: diagonal from diag[], off-diagonals
// 0 - coeff(f1) - coeff(f2) ... over the faces joining the pair.
__global__ __launch_bounds__(kBlock) void csr_values_kernel(uint64_t nnz, const uint32_t* __restrict__ nz_row_diag,
                                                           const uint32_t* __restrict__ nzf_off,
                                                           const uint32_t* __restrict__ nzf,
                                                           const double* __restrict__ diag,
                                                           const double* __restrict__ coeff,
                                                           double* __restrict__ vals) {
#pragma clang fp contract(off)
    const uint64_t k = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (k >= nnz) return;
    const uint32_t dr = nz_row_diag[k];
    if (dr != 0xffffffffu) {
        vals[k] = diag[dr];
        return;
    }
    double v = 0.0;
    for (uint32_t q = nzf_off[k]; q < nzf_off[k + 1]; ++q) v -= coeff[nzf[q]];
    vals[k] = v;
}

__global__ __launch_bounds__(kBlock) void gather_u32idx_kernel(uint64_t n, const uint32_t* __restrict__ src_idx,
                                                              const double* __restrict__ src,
                                                              double* __restrict__ dst) {
    const uint64_t k = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (k < n) dst[k] = src[src_idx[k]];
}

// ---------------------------------------------------------- diffusion ---

__global__ __launch_bounds__(kBlock) void diffusion_face_kernel(uint32_t nf, const uint32_t* __restrict__ owner,
                                                               const int32_t* __restrict__ neigh, double gamma,
                                                               Soa3 fc, Soa3 fs, Soa3 cc,
                                                               const double* __restrict__ fval,
                                                               double* __restrict__ g, int* __restrict__ err) {
#pragma clang fp contract(off)
    const uint32_t f = blockIdx.x * kBlock + threadIdx.x;
    if (f >= nf) return;
    const uint32_t o = owner[f];
    const double area = mag3(fs.get(f));
    if (!(area > 0.0)) err[0] = 4;
    g[f] = 0.0;
    double d = 0.0;
    if (neigh[f] >= 0) {
        d = mag3(sub3(cc.get(uint32_t(neigh[f])), cc.get(o)));
    } else if (isfinite(fval[f])) {
        d = mag3(sub3(fc.get(f), cc.get(o)));
    } else {
        return;
    }
    if (!(d > 2.220446049250313e-16)) {
        err[0] = 4;
        return;
    }
    g[f] = gamma * area / d;
}

__global__ __launch_bounds__(kBlock) void diffusion_cell_kernel(uint32_t nc, const uint32_t* __restrict__ coff,
                                                               const uint32_t* __restrict__ cfs,
                                                               const int32_t* __restrict__ neigh, Soa3 fs,
                                                               const double* __restrict__ vol,
                                                               const double* __restrict__ source,
                                                               const double* __restrict__ fval,
                                                               const uint8_t* __restrict__ fneu,
                                                               const double* __restrict__ g,
                                                               double* __restrict__ diag, double* __restrict__ rhs) {
#pragma clang fp contract(off)
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= nc) return;
    double d = 0.0;
    double b = source[c] * vol[c];
    for (uint32_t k = coff[c]; k < coff[c + 1]; ++k) {
        const uint32_t f = cfs[k];
        if (neigh[f] >= 0) {
            d += g[f];
        } else if (isfinite(fval[f])) {
            if (!fneu[f]) {
                d += g[f];
                b += g[f] * fval[f];
            } else {
                b += fval[f] * mag3(fs.get(f));
            }
        }
    }
    diag[c] = 0.0 + d;
    rhs[c] = b;
}

// Caller-ordered AoS copy of an internally ordered SoA triple: entry i of the
// caller's numbering is internal entry map[i].
__global__ __launch_bounds__(kBlock) void soa_to_aos_kernel(uint32_t n, const uint32_t* __restrict__ map, Soa3 s,
                                                           double* __restrict__ aos) {
    const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const uint32_t j = map[i];
    aos[3 * size_t(i)] = s.x[j];
    aos[3 * size_t(i) + 1] = s.y[j];
    aos[3 * size_t(i) + 2] = s.z[j];
}

__global__ __launch_bounds__(kBlock) void gather_u8_kernel(uint64_t n, const uint32_t* __restrict__ src_idx,
                                                          const uint8_t* __restrict__ src, uint8_t* __restrict__ dst) {
    const uint64_t k = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
    if (k < n) dst[k] = src[src_idx[k]];
}

// ------------------------------------------------------ momentum side ---
//
// Reference anchors:
//   compute_scalar_gradient_with_boundary   physics/finite_volume_transport.h:505-586
//   weighted_least_squares_gradient_robust  core/fvm/least_squares_gradient.h:77-205
//   compute_boundary_aware_wls_gradient     physics/finite_volume_transport.h:606-715
//   compute_nonorthogonal_diffusion_face_fluxes                         :717-874
//   assemble_scalar_equation (UPWIND, cell viscosity)                   :882-1310
//   assemble_momentum_component             physics/steady_incompressible_solver.h:3262-3311
//   relax_momentum_equation                 :3728-3770
//   rAU / build_hbya                        :7816-7836 / :6430-6465
//   velocity correction                     :9545-9557
//   make_rhie_chow_mass_flux                :2063-2217
//
// The three velocity components share the flux, the viscosity and the
// boundary-condition types, so their matrices are identical: one value array
// (and one diagonal) serves all three, each component keeping its own RHS.
// A row visits its cell's faces in ascending order, the order of the reference's
// global face loop, so the per-cell sums are bit-identical (FMA contraction is
// off).

constexpr int kMaxCellFaces = 10;  // WLS stencil: one sample per cell face

// std::max(x, 0.0) and std::clamp(x, 0, 1) exactly (signed zeros included).
__device__ __forceinline__ double max0(double x) { return x < 0.0 ? 0.0 : x; }
__device__ __forceinline__ double clamp01(double v) { return v < 0.0 ? 0.0 : (1.0 < v ? 1.0 : v); }
__device__ __forceinline__ double mag2_3(D3 a) { return a.x * a.x + a.y * a.y + a.z * a.z; }

// boundary_normal_distance: finite_volume_transport.h:247-269.
__device__ __forceinline__ bool boundary_normal_distance(D3 Sf, D3 Cf, D3 Cc, double V, double& out) {
#pragma clang fp contract(off)
    const double area = mag3(Sf);
    if (!(area > 0.0) || !isfinite(area)) return false;
    const double dn = fabs(dot3(sub3(Cf, Cc), Sf)) / area;
    if (!(dn > 0.0) || !isfinite(dn)) {
        if (V > 0.0 && isfinite(V)) {
            const double dn2 = sqrt(V);
            if (dn2 > 0.0 && isfinite(dn2)) {
                out = dn2;
                return true;
            }
        }
        return false;
    }
    out = dn;
    return true;
}

// WLS fit cache. The weighted design matrix of compute_boundary_aware_wls_gradient
// depends on the geometry and on which boundary faces are fixed-value (their
// sample is the face centre, otherwise the centre's normal projection), not
// on the field. wls_build_kernel runs the one-sided Jacobi factorisation once
// per cell and keeps, slot-major, each sample's rotated design row (a0, a1,
// a2), its weight 1/|d| (fac) and its normal distance (nd, boundary samples),
// and per cell the singular values (sig, 3 x nc), the right singular vectors
// (V, 9 x nc, row-major per cell), the condition estimate (cond) and meta:
// bit 0 geometry finite, bit 1 rank == requested dimension, bits 2-7 the
// descending singular-value order (2 bits each).
struct WlsCache {
    double *a0, *a1, *a2, *fac, *nd;
    double *sig, *V, *cond;
    uint32_t* meta;
};

__global__ __launch_bounds__(kBlock) void wls_build_kernel(uint32_t nc, const uint32_t* __restrict__ coff, Slots sl,
                                                          const uint32_t* __restrict__ patch, uint32_t npatch,
                                                          const uint8_t* __restrict__ bct, Soa3 fc, Soa3 cc, int dim,
                                                          WlsCache wc, int* __restrict__ err) {
#pragma clang fp contract(off)
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= nc) return;
    const size_t n1 = nc;
    const uint32_t deg = coff[c + 1] - coff[c];
    const D3 centre = cc.get(c);
    if (deg > uint32_t(kMaxCellFaces)) {
        err[0] = 34;
        return;
    }
    double A[kMaxCellFaces][3];
    int slot_of[kMaxCellFaces];
    bool geo_ok = isfinite(centre.x) && isfinite(centre.y) && isfinite(centre.z);
    int ns = 0;
    for (uint32_t q = 0; q < deg; ++q) {
        const size_t idx = size_t(q) * nc + c;
        const int32_t o = sl.other[idx];
        if (o == -2) continue;
        D3 pt;
        if (o >= 0) {
            pt = cc.get(uint32_t(o));
            wc.nd[idx] = 0.0;
        } else {
            const uint32_t f = sl.face_of(sl.face[idx]);
            const uint32_t pp = patch[f];
            const uint8_t t = pp < npatch ? bct[pp] : 0;
            const D3 sf = sl.s.get(idx);
            const double area = mag3(sf);
            if (!(area > 0.0) || !isfinite(area)) {
                err[0] = 35;
                return;
            }
            const D3 normal = mul3(sf, 1.0 / area);
            const double nd = dot3(sub3(fc.get(f), centre), normal);
            if (!(nd > 0.0) || !isfinite(nd)) {
                err[0] = 36;
                return;
            }
            wc.nd[idx] = nd;
            pt = t == 1 ? fc.get(f) : add3(centre, mul3(normal, nd));
        }
        const D3 d = sub3(pt, centre);
        const double r2 = mag2_3(d);
        if (!(r2 > 0.0) || !isfinite(r2)) geo_ok = false;
        const double factor = 1.0 / sqrt(r2);
        if (!isfinite(factor)) geo_ok = false;
        wc.fac[idx] = factor;
#pragma unroll
        for (int i = 0; i < kMaxCellFaces; ++i)
            if (i == ns) {
                A[i][0] = factor * d.x;
                A[i][1] = factor * d.y;
                A[i][2] = factor * d.z;
                slot_of[i] = int(q);
            }
        ++ns;
    }
    double Vm[3][3] = {{1.0, 0.0, 0.0}, {0.0, 1.0, 0.0}, {0.0, 0.0, 1.0}};
    double sigma[3] = {0.0, 0.0, 0.0};
    int order[3] = {0, 1, 2};
    bool rank_ok = false;
    double cond = INFINITY;
    if (geo_ok) {
        constexpr double eps = 2.220446049250313e-16;
        for (int sweep = 0; sweep < 40; ++sweep) {
            bool changed = false;
#pragma unroll
            for (int p = 0; p < 2; ++p) {
#pragma unroll
                for (int k = p + 1; k < 3; ++k) {
                    double alpha = 0.0, beta = 0.0, gamma = 0.0;
#pragma unroll
                    for (int i = 0; i < kMaxCellFaces; ++i)
                        if (i < ns) {
                            alpha += A[i][p] * A[i][p];
                            beta += A[i][k] * A[i][k];
                            gamma += A[i][p] * A[i][k];
                        }
                    if (!(alpha > 0.0) || !(beta > 0.0)) continue;
                    if (fabs(gamma) <= 8.0 * eps * sqrt(alpha * beta)) continue;
                    const double tau = (beta - alpha) / (2.0 * gamma);
                    const double t = copysign(1.0, tau) / (fabs(tau) + sqrt(1.0 + tau * tau));
                    const double cs = 1.0 / sqrt(1.0 + t * t);
                    const double sn = cs * t;
#pragma unroll
                    for (int i = 0; i < kMaxCellFaces; ++i)
                        if (i < ns) {
                            const double op = A[i][p], ok2 = A[i][k];
                            A[i][p] = cs * op - sn * ok2;
                            A[i][k] = sn * op + cs * ok2;
                        }
#pragma unroll
                    for (int r = 0; r < 3; ++r) {
                        const double op = Vm[r][p], ok2 = Vm[r][k];
                        Vm[r][p] = cs * op - sn * ok2;
                        Vm[r][k] = sn * op + cs * ok2;
                    }
                    changed = true;
                }
            }
            if (!changed) break;
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            double s2 = 0.0;
#pragma unroll
            for (int i = 0; i < kMaxCellFaces; ++i)
                if (i < ns) s2 += A[i][j] * A[i][j];
            sigma[j] = sqrt(s2);
        }
        // Descending, ties in index order (the reference's three-element sort
        // is an insertion sort).
        if (sigma[order[1]] > sigma[order[0]]) {
            const int tmp = order[0];
            order[0] = order[1];
            order[1] = tmp;
        }
        if (sigma[order[2]] > sigma[order[1]]) {
            const int tmp = order[1];
            order[1] = order[2];
            order[2] = tmp;
            if (sigma[order[1]] > sigma[order[0]]) {
                const int tmp2 = order[0];
                order[0] = order[1];
                order[1] = tmp2;
            }
        }
        const double scale = sigma[order[0]];
        const double cutoff = 128.0 * eps * scale;
        int rank = 0;
#pragma unroll
        for (int j = 0; j < 3; ++j)
            if (sigma[order[j]] > cutoff) ++rank;
        if (dim == 2 && rank == 3 && sigma[order[2]] <= 1e-10 * sigma[order[0]]) rank = 2;
        const bool full_rank = rank == dim;
        const double min_pivot = full_rank ? sigma[order[dim - 1]] : 0.0;
        cond = full_rank && min_pivot > 0.0 ? scale / min_pivot : INFINITY;
        rank_ok = full_rank && rank > 0;
    }
#pragma unroll
    for (int i = 0; i < kMaxCellFaces; ++i)
        if (i < ns) {
            const size_t idx = size_t(slot_of[i]) * nc + c;
            wc.a0[idx] = A[i][0];
            wc.a1[idx] = A[i][1];
            wc.a2[idx] = A[i][2];
        }
#pragma unroll
    for (int j = 0; j < 3; ++j) wc.sig[j * n1 + c] = sigma[j];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int j = 0; j < 3; ++j) wc.V[(3 * r + j) * n1 + c] = Vm[r][j];
    wc.cond[c] = cond;
    wc.meta[c] = (geo_ok ? 1u : 0u) | (rank_ok ? 2u : 0u) | (uint32_t(order[0]) << 2) |
                 (uint32_t(order[1]) << 4) | (uint32_t(order[2]) << 6);
}

// K scalar fields at once (the velocity components share the stencil): the
// boundary-aware Green-Gauss gradient (compute_scalar_gradient_with_boundary),
// replaced by the cached WLS fit where it is certified. Field k's boundary
// value at patch p is bcv[p * bstride + k]; bct: 0 zero-gradient, 1 fixed
// value, 2 fixed gradient. K = 1: one field, its gradient as three arrays; the
// Green-Gauss pass comes first for every cell, for the errors it raises on
// fixed gradients. K = 3: velocity records (u, v, w, .) and gradients as three
// records a cell; boundary types are 0 and 1, for which finite samples make a
// finite Green-Gauss sum, so only cells whose fit is refused take that pass and
// the others read neither area vectors nor weights: bound by the 36 bytes of
// fit a slot (80^3 cells: 72 us; 136 with both passes and gathers from memory).
// gate: skip the whole pass unless diffusion is active.
template <int K>
__global__ __launch_bounds__(kBlock) void wls_gradient_kernel(
    uint32_t nc, const uint32_t* __restrict__ coff, Slots sl, const uint32_t* __restrict__ patch, uint32_t npatch,
    const uint8_t* __restrict__ bct, const double* __restrict__ bcv, uint32_t bstride, Soa3 fc, Soa3 fs, Soa3 cc,
    const double* __restrict__ vol, int dim, double limit, WlsCache wc, const double* __restrict__ field,
    double* __restrict__ grad, uint8_t* __restrict__ fallback, const int* __restrict__ gate, int* __restrict__ err) {
#pragma clang fp contract(off)
    static_assert(K == 1 || K == 3);
    __shared__ double2 near_lds[K == 3 ? 2 * kBlock : 1];
    if (gate && !gate[0]) return;
    const uint32_t first = cell_block() * kBlock, c = first + threadIdx.x;
    const Near near{near_lds, first};
    const double4* rec = reinterpret_cast<const double4*>(field);
    double value[K];
    if constexpr (K == 3) {
        if (c < nc) {
            const double4 r = rec[c];
            near.put(0, r);
            value[0] = r.x;
            value[1] = r.y;
            value[2] = r.z;
        }
        __syncthreads();
    }
    if (c >= nc) return;
    if constexpr (K == 1) value[0] = field[c];
    auto sample = [&](uint32_t i, double* v) {
        if constexpr (K == 3) {
            const double4 r = near.has(i) ? near.get(0, i) : rec[i];
            v[0] = r.x;
            v[1] = r.y;
            v[2] = r.z;
        } else {
            v[0] = field[i];
        }
    };
    const size_t n1 = nc;
    const uint32_t deg = coff[c + 1] - coff[c];
    const double V = vol[c];
    if (K == 3 && (!(V > 0.0) || !isfinite(V))) {
        err[0] = 33;
        return;
    }
    D3 g[K];
    // Green-Gauss with boundary values (compute_scalar_gradient_with_boundary).
    auto green_gauss = [&]() {
        const D3 centre = cc.get(c);
        D3 sum[K];
#pragma unroll
        for (int k = 0; k < K; ++k) sum[k] = d3(0.0, 0.0, 0.0);
        for (uint32_t q = 0; q < deg; ++q) {
            const size_t idx = size_t(q) * nc + c;
            const int32_t o = sl.other[idx];
            if (o == -2) continue;
            const D3 Sf = sl.s.get(idx);
            double fv[K];
            if (o >= 0) {
                const double w = sl.w[idx];
                double other[K];
                sample(uint32_t(o), other);
#pragma unroll
                for (int k = 0; k < K; ++k) fv[k] = w * value[k] + (1.0 - w) * other[k];
            } else {
                const uint32_t f = sl.face_of(sl.face[idx]);
                const uint32_t pp = patch[f];
                const uint8_t t = pp < npatch ? bct[pp] : 0;
                double dn = 0.0;
                if (t == 2 && !boundary_normal_distance(fs.get(f), fc.get(f), centre, V, dn)) {
                    err[0] = 31;
                    return false;
                }
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    fv[k] = value[k];
                    if (t == 1) fv[k] = bcv[size_t(pp) * bstride + k];
                    else if (t == 2) fv[k] = value[k] + bcv[size_t(pp) * bstride + k] * dn;
                }
            }
#pragma unroll
            for (int k = 0; k < K; ++k) {
                if (!isfinite(fv[k])) {
                    err[0] = 32;
                    return false;
                }
                sum[k] = add3(sum[k], mul3(Sf, fv[k]));
            }
        }
        if (!(V > 0.0) || !isfinite(V)) {
            err[0] = 33;
            return false;
        }
#pragma unroll
        for (int k = 0; k < K; ++k) g[k] = d3(sum[k].x / V, sum[k].y / V, sum[k].z / V);
        return true;
    };
    if (K == 1 && !green_gauss()) return;
    // The cached WLS fit: rhs_i = fac_i (value_i - value); proj_j = sum_i
    // a_ij rhs_i (sample order); g += V e_j proj_j / sigma_j^2 (descending).
    const uint32_t meta = wc.meta[c];
    const double cond = wc.cond[c];
    const bool certified = (meta & 1u) && (meta & 2u) && isfinite(cond) && cond <= limit;
    bool any_fallback = !certified;
    bool use[K];
    D3 fit[K];
#pragma unroll
    for (int k = 0; k < K; ++k) use[k] = false;
    if (certified) {
        const int o0 = int((meta >> 2) & 3u), o1 = int((meta >> 4) & 3u), o2 = int((meta >> 6) & 3u);
        double proj[K][3];
#pragma unroll
        for (int k = 0; k < K; ++k) {
            use[k] = isfinite(value[k]);
            proj[k][0] = proj[k][1] = proj[k][2] = 0.0;
        }
        for (uint32_t q = 0; q < deg; ++q) {
            const size_t idx = size_t(q) * nc + c;
            const int32_t o = sl.other[idx];
            if (o == -2) continue;
            const double fac = wc.fac[idx];
            const double a[3] = {wc.a0[idx], wc.a1[idx], wc.a2[idx]};
            const double aj0 = o0 == 0 ? a[0] : (o0 == 1 ? a[1] : a[2]);
            const double aj1 = o1 == 0 ? a[0] : (o1 == 1 ? a[1] : a[2]);
            const double aj2 = o2 == 0 ? a[0] : (o2 == 1 ? a[1] : a[2]);
            double sv[K];
            if (o >= 0) {
                sample(uint32_t(o), sv);
            } else {
                const uint32_t pp = patch[sl.face_of(sl.face[idx])];
                const uint8_t t = pp < npatch ? bct[pp] : 0;
                const double nd = wc.nd[idx];
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    if (t == 1) sv[k] = bcv[size_t(pp) * bstride + k];
                    else sv[k] = value[k] + nd * (t == 2 ? bcv[size_t(pp) * bstride + k] : 0.0);
                }
            }
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const double dv = sv[k] - value[k];
                if (!isfinite(dv)) use[k] = false;
                const double rhs = fac * dv;
                proj[k][0] += aj0 * rhs;
                proj[k][1] += aj1 * rhs;
                proj[k][2] += aj2 * rhs;
            }
        }
        const int ord[3] = {o0, o1, o2};
#pragma unroll
        for (int k = 0; k < K; ++k) {
            double x[3] = {0.0, 0.0, 0.0};
            if (use[k]) {
                for (int oi = 0; oi < dim; ++oi) {
                    const int j = ord[oi];
                    const double sj = wc.sig[j * n1 + c];
                    const double coeff = proj[k][oi] / (sj * sj);
#pragma unroll
                    for (int r = 0; r < 3; ++r) x[r] += wc.V[(3 * r + j) * n1 + c] * coeff;
                }
                use[k] = isfinite(x[0]) && isfinite(x[1]) && isfinite(x[2]);
            }
            fit[k] = d3(x[0], x[1], x[2]);
        }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) any_fallback |= !use[k];
    if (K == 3 && any_fallback && !green_gauss()) return;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const D3 r = use[k] ? fit[k] : g[k];
        if constexpr (K == 3) {
            reinterpret_cast<double4*>(grad)[3 * size_t(c) + k] = make_double4(r.x, r.y, r.z, 0.0);
        } else {
            grad[c] = r.x;
            grad[n1 + c] = r.y;
            grad[2 * n1 + c] = r.z;
        }
    }
    if (fallback) fallback[c] = any_fallback ? 1 : 0;
}

// needs_nonorthogonal_gradient scan (finite_volume_transport.h:987-1021) of the
// geometry: an internal or boundary face with a tangential part above 1e-12
// |S_f| sets flags[its patch] (internal: flags[npatch]), one whose geometry
// does not define it flags[npatch + 1 + its patch]. Boundary faces count only
// where the patch's velocity is fixed, which the caller looks up.
__global__ __launch_bounds__(kBlock) void nonorth_scan_kernel(uint32_t nf, const uint32_t* __restrict__ owner,
                                                             const int32_t* __restrict__ neigh,
                                                             const uint32_t* __restrict__ patch, uint32_t npatch,
                                                             const uint8_t* __restrict__ kind, Soa3 fc, Soa3 fs,
                                                             Soa3 cc, int* __restrict__ flags) {
#pragma clang fp contract(off)
    const uint32_t f = blockIdx.x * kBlock + threadIdx.x;
    if (f >= nf) return;
    const int32_t nr = neigh[f];
    uint32_t pp = npatch;
    if (nr < 0) {
        pp = patch[f];
        if (pp >= npatch || kind[pp] == 1) return;
    }
    const uint32_t o = owner[f];
    const D3 sf = fs.get(f);
    const double area = mag3(sf);
    const D3 d = nr >= 0 ? sub3(cc.get(uint32_t(nr)), cc.get(o)) : sub3(fc.get(f), cc.get(o));
    const double sd = dot3(sf, d);
    const double d2 = dot3(d, d);
    if (!(area > 0.0) || !(sd > 0.0) || !(d2 > 0.0) || !isfinite(area) || !isfinite(sd) || !isfinite(d2)) {
        flags[npatch + 1 + pp] = 1;
        return;
    }
    const double alpha = area * area / sd;
    const D3 tangential = sub3(sf, mul3(d, alpha));
    if (mag3(tangential) > 1e-12 * area) flags[pp] = 1;
}

// One momentum row per thread (internal cell c), its faces in ascending caller
// face id (the reference's face loop order): the upwind/diffusion coefficient
// of each face on the diagonal and on the row's entry, flux divergence,
// tangential diffusion fluxes (needs) and boundary sources; then the
// bounded-convection correction, sources and the equation relaxation
// (relax: alpha < 1). As in the pressure rows every face is evaluated from both
// of its cells: conductances and interpolation weights come out the same to the
// last bit and fluxes negated, as long as the one quantity that is not
// symmetric, the weight along the line from the owner, is taken from the
// owner's side. out: (rhs, relaxed diagonal) a cell. On 80^3 jittered cells,
// randomly numbered: 155 us; 162 with the gradients staged as well (LDS then
// leaves two workgroups a CU instead of three), 162 with the face's data read
// one slot ahead; 368 as a pass over faces that scattered five terms to the
// cells' slots, one over cells and one over nonzeros.
__global__ __launch_bounds__(kBlock) void momentum_row_kernel(
    uint32_t nc, uint32_t D, const uint32_t* __restrict__ coff, const uint8_t* __restrict__ slot_sorted, Slots sl,
    const uint32_t* __restrict__ patch, uint32_t npatch, const uint8_t* __restrict__ vbt,
    const double* __restrict__ vbv, Soa3 fc, const double4* __restrict__ cell, const double4* __restrict__ fields,
    const double4* __restrict__ source, const double4* __restrict__ ugrad, const double* __restrict__ phi,
    int bounded, int nonorthogonal, const int* __restrict__ flags, int relax, double alpha_u, RowMap rm,
    double* __restrict__ vals, double4* __restrict__ out, int* __restrict__ err) {
#pragma clang fp contract(off)
    extern __shared__ double2 row_shared[];
    const uint32_t first = cell_block() * kBlock;
    const bool live = first + threadIdx.x < nc;
    const uint32_t c = live ? first + threadIdx.x : nc - 1;  // the last block's spare threads only keep step
    const bool needs = nonorthogonal && flags[0];
    const Near near{row_shared, first};
    const uint32_t stride = D + 1;
    double* rows = reinterpret_cast<double*>(row_shared + kMomNear * 2 * kBlock);
    double* row = rows + threadIdx.x * stride;
    const uint32_t deg = live ? coff[c + 1] - coff[c] : 0;
    const double4 C = cell[c], A = fields[c];
    double4 G[3];
    near.put(0, C);
    near.put(1, A);
    if (needs) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            G[k] = ugrad[3 * size_t(c) + k];
        }
    }
    __syncthreads();
    const D3 Cc = d3(C.x, C.y, C.z);
    if (rm.shared)
        for (uint32_t k = 0; k < stride; ++k) row[k] = 0.0;
    double diag = 0.0, div = 0.0;
    double rhs[3] = {0.0, 0.0, 0.0}, def[3] = {0.0, 0.0, 0.0};
    uint32_t len = 0;
    // A slot's place, then its ids, then the face's and the neighbour's data
    // depend on each other: the first two are read ahead.
    auto place = [&](uint32_t k) {
        return k < deg ? size_t(slot_sorted[size_t(k) * nc + c]) * nc + c : size_t(c);
    };
    size_t idx = place(0), idx1 = place(1);
    int32_t o1 = sl.other[idx];
    uint32_t f1 = sl.face[idx];
    for (uint32_t k = 0; k < deg; ++k) {
        const size_t at = idx;
        const int32_t o = o1;
        const uint32_t fr = f1, f = sl.face_of(fr);
        const bool reversed = fr != f;
        const double Fo = phi[f];
        const D3 Sf = sl.s.get(at), Cf = fc.get(f);
        idx = idx1;
        o1 = sl.other[idx];
        f1 = sl.face[idx];
        idx1 = place(k + 2);
        if (!isfinite(Fo)) err[0] = 42;
        if (o == -2) continue;
        const double F = reversed ? -Fo : Fo;
        const double area = mag3(Sf);
        if (o >= 0) {
            const uint32_t n = uint32_t(o);
            const bool in = near.has(n);
            const double4 Nn = in ? near.get(0, n) : cell[n];
            const double gn = in ? near.get(1, n).w : fields[n].w, go = A.w;
            const D3 Cn = d3(Nn.x, Nn.y, Nn.z);
            const D3 line = sub3(Cn, Cc);
            const double distance = mag3(line);
            if (!(distance > 0.0) || !(area > 0.0)) err[0] = 43;
            const double d_own = fabs(dot3(sub3(Cf, Cc), Sf)) / area;
            const double d_oth = fabs(dot3(sub3(Cn, Cf), Sf)) / area;
            if (!(d_own > 0.0) || !(d_oth > 0.0) || !isfinite(d_own) || !isfinite(d_oth)) err[0] = 44;
            double Dc = 0.0;
            if (go > 0.0 && gn > 0.0) Dc = area / (d_own / go + d_oth / gn);
            if (needs) {
                const double sd = dot3(Sf, line);
                const double alpha = area * area / sd;
                const D3 tangential = sub3(Sf, mul3(line, alpha));
                if (mag3(tangential) > 1e-12 * area) {
                    const double area_projection = fabs(sd) / area;
                    if (!(area_projection > 0.0)) err[0] = 45;
                    const double gamma_face = Dc / alpha;
                    const double d2_line = mag2_3(line);
                    if (!(d2_line > 0.0) || !isfinite(d2_line)) err[0] = 46;
                    const double along =
                        reversed ? dot3(sub3(Cf, Cn), sub3(Cc, Cn)) : dot3(sub3(Cf, Cc), line);
                    const double w = 1.0 - clamp01(along / d2_line);
                    const double wc = reversed ? 1.0 - w : w, wn = reversed ? w : 1.0 - w;
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        const double4 N = ugrad[3 * size_t(n) + q];
                        const D3 gf = add3(mul3(d3(G[q].x, G[q].y, G[q].z), wc), mul3(d3(N.x, N.y, N.z), wn));
                        const double flux = gamma_face * dot3(gf, tangential);
                        if (!isfinite(flux)) err[0] = 47;
                        def[q] += flux;
                    }
                }
            }
            diag += Dc + max0(F);
            div += F;
            const uint16_t r = rm.rank[size_t(k) * nc + c];
            len = max(len, uint32_t(r) + 1u);
            row[r] = (rm.shared ? row[r] : 0.0) - (Dc + max0(-F));
        } else {
            const uint32_t pp = patch[f];
            const bool fixed = pp < npatch && vbt[pp] == 1;
            double distance = 0.0;
            if (!boundary_normal_distance(Sf, Cf, Cc, C.w, distance) || !(distance > 0.0) || !(area > 0.0))
                err[0] = 48;
            if (fixed) {
                const double Dc = A.w * area / distance;
                if (needs) {
                    const D3 d = sub3(Cf, Cc);
                    const double sd = dot3(Sf, d);
                    const double alpha = area * area / sd;
                    const D3 tangential = sub3(Sf, mul3(d, alpha));
                    if (mag3(tangential) > 1e-12 * area) {
#pragma unroll
                        for (int q = 0; q < 3; ++q) {
                            const double flux = A.w * dot3(d3(G[q].x, G[q].y, G[q].z), tangential);
                            if (!isfinite(flux)) err[0] = 47;
                            def[q] += flux;
                        }
                    }
                }
                diag += Dc + max0(F);
#pragma unroll
                for (int q = 0; q < 3; ++q) rhs[q] += (Dc + max0(-F)) * vbv[3 * size_t(pp) + q];
            } else {
                diag += bounded ? F : max0(F);
                if (!bounded && F < 0.0) {
                    def[0] -= F * A.x;
                    def[1] -= F * A.y;
                    def[2] -= F * A.z;
                }
            }
            div += F;
        }
    }
    if (bounded) diag -= div;
    const double V = C.w;
    diag -= 0.0 * V;
    if (live && (!(diag > 0.0) || !isfinite(diag))) err[0] = 49;
    const double4 src = source[c];
    rhs[0] += src.x * V;
    rhs[1] += src.y * V;
    rhs[2] += src.z * V;
#pragma unroll
    for (int q = 0; q < 3; ++q) rhs[q] += def[q];
    if (relax) {
        const double added = diag * (1.0 / alpha_u - 1.0);
        diag += added;
        rhs[0] += added * A.x;
        rhs[1] += added * A.y;
        rhs[2] += added * A.z;
    }
    if (live) {
        const uint32_t r = rm.diag[c];
        row[r] = diag;
        len = max(len, r + 1u);
        out[c] = make_double4(rhs[0], rhs[1], rhs[2], diag);
    }
    wave_fence();
    store_rows(rows + (threadIdx.x & ~63u) * stride, stride, rm.start[c], live ? len : 0, vals);
}

// rAU = 1 / diag and HbyA_k = rAU (rhs_k + grad_p_k V - sum_{j != r} a_rj U_k[j])
// with the row's entries in storage order.
__global__ __launch_bounds__(kBlock) void hbya_kernel(uint32_t n, const uint32_t* __restrict__ rowp,
                                                     const uint32_t* __restrict__ cols,
                                                     const double* __restrict__ vals, const double* __restrict__ rhs,
                                                     const double* __restrict__ diag,
                                                     const double* __restrict__ gradp, const double* __restrict__ vol,
                                                     const double* __restrict__ U, double* __restrict__ rau,
                                                     double* __restrict__ hbya, int* __restrict__ err) {
#pragma clang fp contract(off)
    const uint32_t r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= n) return;
    const size_t n1 = n;
    const double a = diag[r];
    if (!(a > 0.0) || !isfinite(a)) err[0] = 50;
    const double ra = 1.0 / a;
    double h[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) h[k] = rhs[k * n1 + r] + gradp[k * n1 + r] * vol[r];
    for (uint32_t j = rowp[r]; j < rowp[r + 1]; ++j) {
        const uint32_t col = cols[j];
        if (col == r) continue;
        const double v = vals[j];
#pragma unroll
        for (int k = 0; k < 3; ++k) h[k] -= v * U[k * n1 + col];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double hb = ra * h[k];
        if (!isfinite(hb)) err[0] = 51;
        rau[k * n1 + r] = ra;
        hbya[k * n1 + r] = hb;
    }
}

// U = HbyA - rAU grad_p V.
__global__ __launch_bounds__(kBlock) void velocity_correct_kernel(uint32_t nc, const double* __restrict__ hbya,
                                                                 const double* __restrict__ rau,
                                                                 const double* __restrict__ gradp,
                                                                 const double* __restrict__ vol,
                                                                 double* __restrict__ U) {
#pragma clang fp contract(off)
    const uint32_t c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= nc) return;
    const size_t n1 = nc;
#pragma unroll
    for (int k = 0; k < 3; ++k) U[k * n1 + c] = hbya[k * n1 + c] - rau[k * n1 + c] * gradp[k * n1 + c] * vol[c];
}

// Rhie-Chow face mass flux from HbyA and p (make_rhie_chow_mass_flux,
// HBYA_PREDICTOR contract, w = 1/2): rho H_f.S_f minus the pressure
// correction (internal: rhie_chow_pressure_flux_internal; fixed-pressure
// boundary: the boundary coefficient and deferred flux); EMPTY and SYMMETRY
// faces carry no flux.
__global__ __launch_bounds__(kBlock) void rhie_chow_flux_kernel(
    uint32_t nf, uint32_t nc, const uint32_t* __restrict__ owner, const int32_t* __restrict__ neigh,
    const uint32_t* __restrict__ patch, uint32_t npatch, const uint8_t* __restrict__ kind,
    const uint8_t* __restrict__ vbt, const double* __restrict__ vbv, const uint8_t* __restrict__ pbt,
    const double* __restrict__ pbv, double rho, Soa3 fc, Soa3 fs, Soa3 cc, const double* __restrict__ vol,
    const double* __restrict__ H, const double* __restrict__ p, const double4* __restrict__ grad,
    const double* __restrict__ rAU, double* __restrict__ phi, int* __restrict__ err) {
#pragma clang fp contract(off)
    const uint32_t f = blockIdx.x * kBlock + threadIdx.x;
    if (f >= nf) return;
    const size_t n2 = 2 * size_t(nc);
    const uint32_t o = owner[f];
    D3 Hf = d3(H[o], H[nc + o], H[n2 + o]);
    double correction = 0.0;
    const D3 Sf = fs.get(f);
    // rAU must be finite and positive; every cell is some face's.
    auto invalid = [&](uint32_t i) {
        const double a = rAU[i], b = rAU[nc + i], c = rAU[n2 + i];
        return !(a > 0.0 && b > 0.0 && c > 0.0 && isfinite(a) && isfinite(b) && isfinite(c));
    };
    if (invalid(o) || (neigh[f] >= 0 && invalid(uint32_t(neigh[f])))) err[0] = 53;
    if (neigh[f] >= 0) {
        const uint32_t n = uint32_t(neigh[f]);
        const D3 Hn = d3(H[n], H[nc + n], H[n2 + n]);
        const double wn = 0.5, wo = 1.0 - wn;
        Hf = add3(mul3(Hf, 1.0 - wn), mul3(Hn, wn));
        const D3 dAU = d3(wo * vol[o] * rAU[o] + wn * vol[n] * rAU[n],
                          wo * vol[o] * rAU[nc + o] + wn * vol[n] * rAU[nc + n],
                          wo * vol[o] * rAU[n2 + o] + wn * vol[n] * rAU[n2 + n]);
        const double4 go = grad[o], gn = grad[n];
        const D3 gp = d3(wo * go.x + wn * gn.x, wo * go.y + wn * gn.y, wo * go.z + wn * gn.z);
        const D3 dv = sub3(cc.get(n), cc.get(o));
        double ic = 0.0, nofl = 0.0;
        if (!face_pressure_terms(Sf, dv, dAU, gp, ic, nofl)) {
            err[0] = 52;
            return;
        }
        correction = rho * (ic * (p[n] - p[o]) + nofl);
    } else {
        const uint32_t pp = patch[f];
        if (pp < npatch && (kind[pp] == 1 || kind[pp] == 2)) {
            phi[f] = 0.0;
            return;
        }
        if (pp < npatch) {
            if (vbt[pp] == 1) Hf = d3(vbv[3 * pp], vbv[3 * pp + 1], vbv[3 * pp + 2]);
            if (pbt[pp] == 1) {
                const D3 dv = sub3(fc.get(f), cc.get(o));
                const double d = mag3(dv);
                if (!(d > 0.0) || !isfinite(d)) {
                    err[0] = 52;
                    return;
                }
                const double4 go = grad[o];
                const D3 gp = d3(go.x, go.y, go.z);
                const D3 dAU = d3(vol[o] * rAU[o], vol[o] * rAU[nc + o], vol[o] * rAU[n2 + o]);
                double ic = 0.0, def = 0.0;
                if (!face_pressure_terms(Sf, dv, dAU, gp, ic, def)) {
                    err[0] = 52;
                    return;
                }
                correction = rho * (ic * (pbv[pp] - p[o]) + def);
            }
        }
    }
    phi[f] = rho * dot3(Hf, Sf) - correction;
}

}  // namespace

// ==================================================================== FvMesh

// Internal numbering. A caller's cells may be numbered without locality (the
// benchmark boxes are a random permutation), and a kernel that gathers cell or
// face data through such ids reads a whole cache line per 8-byte value. The
// handle therefore keeps the mesh in its own order: cells along a Hilbert
// curve through their centres, faces grouped by owner in that order
// (caller order within an owner). Every kernel runs on the internal arrays;
// the public methods take and return caller-ordered fields and permute them
// once on the way in and out. Each cell keeps its caller face list order
// (cfaces) and visits faces in ascending caller face id where the reference
// accumulates in face order (cfaces_sorted), so every value is unchanged.

namespace {

// Hilbert index of a point of the 2^16 cube (J. Skilling, Programming the
// Hilbert curve, AIP Conf. Proc. 707, 2004): the axes' bits are turned into
// the curve's transposed index from the top bit down, then interleaved.
uint64_t hilbert_key(uint32_t x, uint32_t y, uint32_t z) {
    uint32_t a[3] = {x, y, z};
    for (uint32_t q = 1u << 15; q > 1; q >>= 1) {
        const uint32_t low = q - 1;
        for (int i = 0; i < 3; ++i) {
            if (a[i] & q) {
                a[0] ^= low;
            } else {
                const uint32_t t = (a[0] ^ a[i]) & low;
                a[0] ^= t;
                a[i] ^= t;
            }
        }
    }
    a[1] ^= a[0];
    a[2] ^= a[1];
    uint32_t t = 0;
    for (uint32_t q = 1u << 15; q > 1; q >>= 1)
        if (a[2] & q) t ^= q - 1;
    uint64_t key = 0;
    for (int b = 15; b >= 0; --b)
        for (int i = 0; i < 3; ++i) key = (key << 1) | (((a[i] ^ t) >> b) & 1u);
    return key;
}

// Cells in the order of a Hilbert curve through their vertices' means, each
// axis scaled by the distribution of the cells along it (grids are stretched
// towards walls by factors of a thousand: equal steps of the key then hold
// equally many cells). Ties keep the caller's order. The order only sets where
// values lie: it needs no accuracy, and takes any coordinates.
void curve_ordering(uint32_t nc, const uint32_t* coff, const uint32_t* cf, const uint32_t* foff,
                    const uint32_t* fvtx, const double* px, const double* py, const double* pz,
                    std::vector<uint32_t>& order) {
    constexpr uint32_t kBins = 1u << 16;
    std::vector<double> centre[3];
    for (auto& v : centre) v.resize(nc);
    parallel_for(nc, 0, [&](uint64_t c) {
        double s[3] = {0.0, 0.0, 0.0};
        uint32_t n = 0;
        for (uint32_t k = coff[c]; k < coff[c + 1]; ++k)
            for (uint32_t q = foff[cf[k]]; q < foff[cf[k] + 1]; ++q, ++n) {
                s[0] += px[fvtx[q]];
                s[1] += py[fvtx[q]];
                s[2] += pz[fvtx[q]];
            }
        for (int d = 0; d < 3; ++d) centre[d][c] = n ? s[d] / n : 0.0;
    });
    std::vector<uint16_t> axis[3];
    for (int d = 0; d < 3; ++d) {
        axis[d].resize(nc);
        double lo = INFINITY, hi = -INFINITY;
        for (double v : centre[d])
            if (std::isfinite(v)) lo = std::min(lo, v), hi = std::max(hi, v);
        const double scale = hi > lo ? (kBins - 1) / (hi - lo) : 0.0;
        std::vector<uint64_t> below(kBins + 1, 0);
        auto bin = [&](double v) {
            const double b = (v - lo) * scale;
            return b >= 0.0 && b <= kBins - 1 ? uint32_t(b) : 0u;
        };
        for (double v : centre[d]) ++below[bin(v) + 1];
        for (uint32_t b = 0; b < kBins; ++b) below[b + 1] += below[b];
        parallel_for(nc, 0, [&](uint64_t c) {
            const uint32_t b = bin(centre[d][c]);
            axis[d][c] = uint16_t((below[b] + below[b + 1]) / 2 * (kBins - 1) / nc);
        });
    }
    std::vector<uint64_t> key(nc);
    parallel_for(nc, 0, [&](uint64_t c) { key[c] = hilbert_key(axis[0][c], axis[1][c], axis[2][c]); });
    // Counting sort by 12 bits at a time, stable.
    order.resize(nc);
    std::iota(order.begin(), order.end(), 0u);
    std::vector<uint32_t> next(nc);
    for (int shift = 0; shift < 48; shift += 12) {
        std::vector<uint32_t> at(4097, 0);
        for (uint32_t c = 0; c < nc; ++c) ++at[((key[c] >> shift) & 4095u) + 1];
        for (int b = 0; b < 4096; ++b) at[b + 1] += at[b];
        for (uint32_t i = 0; i < nc; ++i) next[at[(key[order[i]] >> shift) & 4095u]++] = order[i];
        order.swap(next);
    }
}

Slots slots_of(const FvMesh& m) {
    return Slots{m.slot_other, m.slot_face, m.slot_w, Soa3{m.slot_sx, m.slot_sy, m.slot_sz}};
}
WlsCache wls_of(const FvMesh& m) {
    return WlsCache{m.wls_a0, m.wls_a1, m.wls_a2, m.wls_fac, m.wls_nd, m.wls_sig, m.wls_V, m.wls_cond, m.wls_meta};
}
}  // namespace

void PressurePlan::release() {
    for (uint32_t** p : {&rowp, &cols, &nz_row_diag, &nzf_off, &nzf}) dfree(*p);
    release_maps();
}

void PressurePlan::release_maps() {
    for (uint32_t** p : {&row_start, &row_of}) dfree(*p);
    for (uint16_t** p : {&slot_rank, &diag_rank}) dfree(*p);
}

FvMesh::~FvMesh() { release(); }

void FvMesh::release() {
    for (double** p : {&px, &py, &pz, &fcx, &fcy, &fcz, &fsx, &fsy, &fsz, &ccx, &ccy, &ccz, &vol, &vol_caller,
                       &work_coeff, &work_diag, &work_grad,
                       &mom_ugrad, &bc_f64, &slot_coeff,
                       &wls_a0, &wls_a1, &wls_a2, &wls_fac, &wls_nd, &wls_sig, &wls_V, &wls_cond})
        dfree(*p);
    for (uint32_t** p : {&foff, &fvtx, &owner, &coff, &cfaces, &cfaces_sorted, &patch, &cell_new, &cell_old,
                         &face_new, &face_old})
        dfree(*p);
    for (auto& b : scratch) dfree(b.first);
    scratch.clear();
    dfree(scratch_u8);
    release_slots();
    dfree(wls_meta);
    dfree(neigh);
    dfree(patch_kind);
    if (h_err) (void)hipHostFree(h_err);
    h_err = err = nullptr;
    if (bc_host) (void)hipHostFree(bc_host);
    bc_host = nullptr;
    dfree(mom_flags);
    pressure_full.release();
    pressure_red.release();
}

// Lines of 16 values that the neighbours and the faces of 64 consecutive cells
// lie in, summed over up to 128 such windows spread over the mesh: cells in
// the order `at` (cell of each place), places cell_place and face_place (null:
// the caller's order). fewest: the lines that so many values take at least.
uint64_t FvMesh::touched_lines(const uint32_t* at, const uint32_t* cell_place, const uint32_t* face_place,
                               uint64_t* fewest) const {
    const uint32_t windows = (nc + 63) / 64, taken = std::min<uint32_t>(windows, 128);
    std::vector<uint32_t> cells, faces;
    uint64_t lines = 0, least = 0;
    for (uint32_t s = 0; s < taken; ++s) {
        const uint64_t first = uint64_t(s) * windows / taken * 64;
        cells.clear();
        faces.clear();
        for (uint64_t i = first; i < std::min<uint64_t>(first + 64, nc); ++i) {
            const uint32_t c = at ? at[i] : uint32_t(i);
            for (uint32_t k = h_coff[c]; k < h_coff[c + 1]; ++k) {
                const uint32_t f = h_cf[k];
                faces.push_back(face_place ? face_place[f] : f);
                if (h_neigh[f] < 0) continue;
                const uint32_t n = h_owner[f] == c ? uint32_t(h_neigh[f]) : h_owner[f];
                cells.push_back(cell_place ? cell_place[n] : n);
            }
        }
        for (auto* v : {&cells, &faces}) {
            std::sort(v->begin(), v->end());
            v->erase(std::unique(v->begin(), v->end()), v->end());
            least += (v->size() + 15) / 16;
            for (size_t k = 0; k < v->size(); ++k) lines += k == 0 || (*v)[k] / 16 != (*v)[k - 1] / 16;
        }
    }
    if (fewest) *fewest = least;
    return lines;
}

void FvMesh::create(int device, uint64_t np_, const double* hx, const double* hy, const double* hz, uint64_t nf_,
                    const uint32_t* hfoff, const uint32_t* hfvtx, const uint32_t* hown, const int32_t* hnei,
                    uint64_t nc_, const uint32_t* hcoff, const uint32_t* hcf, uint64_t npatch_,
                    const uint32_t* hpatch, const uint8_t* hkind) {
    if (nf_ >= UINT32_MAX || nc_ >= UINT32_MAX || np_ >= UINT32_MAX) throw std::invalid_argument("mesh too large");
    dev = device;
    HIP_OK(hipSetDevice(dev));
    np = uint32_t(np_);
    nf = uint32_t(nf_);
    nc = uint32_t(nc_);
    npatch = uint32_t(npatch_);
    // Host copies (caller numbering) for the sparsity plans.
    h_owner.assign(hown, hown + nf);
    h_neigh.assign(hnei, hnei + nf);
    h_coff.assign(hcoff, hcoff + nc + 1);
    h_cf.assign(hcf, hcf + h_coff[nc]);
    h_patch.assign(hpatch, hpatch + nf);
    h_kind.assign(hkind, hkind + npatch);
    h_patch_boundary.assign(std::max<uint32_t>(npatch, 1), 0);
    for (uint32_t f = 0; f < nf; ++f) {
        if (h_owner[f] >= nc || h_neigh[f] >= int64_t(nc)) throw std::invalid_argument("face addressing out of range");
        if (h_neigh[f] < 0 && h_patch[f] < npatch) h_patch_boundary[h_patch[f]] = 1;
    }
    for (uint32_t k = 0; k < h_coff[nc]; ++k)
        if (h_cf[k] >= nf) throw std::invalid_argument("cell face index out of range");
    for (uint32_t k = 0; k < hfoff[nf]; ++k)
        if (hfvtx[k] >= np) throw std::invalid_argument("face vertex out of range");
    // Keep the caller's numbering when the accesses of 64 consecutive cells
    // touch about as few lines in it as on the curve (at most half as many
    // again): then no field is permuted at all.
    // Lexicographic numberings of boxes and channels touch 1.05 times the
    // curve's lines, random ones 9 times. A 222k-cell channel kept as numbered
    // assembles its pressure in 71 us, moved onto the curve in 81 (its fields
    // pass through gathers); a random 128^3 box assembled as
    // numbered would fetch a line for each of its 66M values.
    // The curve itself touches 1.4 to 1.7 times the fewest lines that any
    // order could, so a numbering within twice the fewest (lexicographic ones
    // take 1.2 to 1.6 times) is kept without laying the curve.
    std::vector<uint32_t> cold(nc), cnew(nc), fnew(nf), fold(nf);
    uint64_t fewest = 0;
    const uint64_t caller = touched_lines(nullptr, nullptr, nullptr, &fewest);
    identity_order = caller <= 2 * fewest;
    if (!identity_order) {
        // Cells along the curve, faces by internal owner, caller order within one.
        curve_ordering(nc, h_coff.data(), h_cf.data(), hfoff, hfvtx, hx, hy, hz, cold);
        for (uint32_t i = 0; i < nc; ++i) cnew[cold[i]] = i;
        std::vector<uint32_t> cnt(uint64_t(nc) + 1, 0);
        for (uint32_t f = 0; f < nf; ++f) ++cnt[cnew[h_owner[f]] + 1];
        for (uint32_t c = 0; c < nc; ++c) cnt[c + 1] += cnt[c];
        for (uint32_t f = 0; f < nf; ++f) {
            const uint32_t pos = cnt[cnew[h_owner[f]]]++;
            fold[pos] = f;
            fnew[f] = pos;
        }
        const uint64_t curve = touched_lines(cold.data(), cnew.data(), fnew.data(), nullptr);
        identity_order = 2 * caller <= 3 * curve;
    }
    if (identity_order) {
        std::iota(cnew.begin(), cnew.end(), 0u);
        std::iota(cold.begin(), cold.end(), 0u);
        std::iota(fold.begin(), fold.end(), 0u);
        std::iota(fnew.begin(), fnew.end(), 0u);
    }
    // Internal arrays.
    {
        std::vector<uint32_t> o(nf), pt(nf), fo(uint64_t(nf) + 1, 0), fv;
        std::vector<int32_t> nb(nf);
        for (uint32_t i = 0; i < nf; ++i) {
            const uint32_t f = fold[i];
            o[i] = cnew[h_owner[f]];
            nb[i] = h_neigh[f] >= 0 ? int32_t(cnew[uint32_t(h_neigh[f])]) : -1;
            pt[i] = h_patch[f];
            fo[i + 1] = fo[i] + (hfoff[f + 1] - hfoff[f]);
        }
        fv.resize(fo[nf]);
        parallel_for(nf, 0, [&](uint64_t i) {
            const uint32_t f = fold[i];
            std::copy(hfvtx + hfoff[f], hfvtx + hfoff[f + 1], fv.begin() + fo[i]);
        });
        owner = upload(o.data(), nf);
        neigh = upload(nb.data(), nf);
        patch = upload(pt.data(), nf);
        foff = upload(fo.data(), uint64_t(nf) + 1);
        fvtx = upload(fv.data(), fv.size());
    }
    {
        std::vector<uint32_t> co(uint64_t(nc) + 1, 0), cf(h_cf.size()), cfs(h_cf.size());
        for (uint32_t i = 0; i < nc; ++i) {
            const uint32_t c = cold[i];
            co[i + 1] = co[i] + (h_coff[c + 1] - h_coff[c]);
        }
        parallel_for(nc, 0, [&](uint64_t i) {
            const uint32_t c = cold[i];
            const uint32_t b = h_coff[c], e = h_coff[c + 1];
            std::vector<uint32_t> sorted(h_cf.begin() + b, h_cf.begin() + e);
            std::sort(sorted.begin(), sorted.end());
            for (uint32_t k = 0; k < e - b; ++k) {
                cf[co[i] + k] = fnew[h_cf[b + k]];
                cfs[co[i] + k] = fnew[sorted[k]];
            }
        });
        coff = upload(co.data(), co.size());
        cfaces = upload(cf.data(), cf.size());
        cfaces_sorted = upload(cfs.data(), cfs.size());
    }
    cell_new = upload(cnew.data(), nc);
    cell_old = upload(cold.data(), nc);
    face_new = upload(fnew.data(), nf);
    face_old = upload(fold.data(), nf);
    h_cell_new = std::move(cnew);
    h_face_new = std::move(fnew);
    px = upload(hx, np);
    py = upload(hy, np);
    pz = upload(hz, np);
    patch_kind = upload(hkind, npatch);
    for (double** p : {&fcx, &fcy, &fcz, &fsx, &fsy, &fsz}) *p = dalloc<double>(nf);
    for (double** p : {&ccx, &ccy, &ccz, &vol, &vol_caller}) *p = dalloc<double>(nc);
    // The error flags are host memory that kernels write only when they refuse
    // something: the host reads and clears them without a copy or a launch.
    HIP_OK(hipHostMalloc(reinterpret_cast<void**>(&h_err), 4 * sizeof(int), hipHostMallocMapped));
    HIP_OK(hipHostGetDevicePointer(reinterpret_cast<void**>(&err), h_err, 0));
    clear_err();
    HIP_OK(hipStreamCreate(&stream));
    compute_geometry();
    gather_u32idx_kernel<<<grid_for(nc), kBlock, 0, stream>>>(nc, cell_new, vol, vol_caller);
    HIP_OK(hipStreamSynchronize(stream));
}

double* FvMesh::scr(size_t slot, uint64_t count) {
    if (scratch.size() <= slot) scratch.resize(slot + 1, {nullptr, 0});
    auto& b = scratch[slot];
    if (b.second < count) {
        dfree(b.first);
        b.first = dalloc<double>(count);
        b.second = count;
    }
    return b.first;
}

void FvMesh::cells_in(const double* caller, double* internal, int comps) {
    if (identity_order) {
        HIP_OK(hipMemcpyAsync(internal, caller, uint64_t(comps) * nc * 8, hipMemcpyDeviceToDevice, stream));
        return;
    }
    for (int k = 0; k < comps; ++k)
        gather_u32idx_kernel<<<grid_for(nc), kBlock, 0, stream>>>(nc, cell_old, caller + size_t(k) * nc,
                                                                  internal + size_t(k) * nc);
}

void FvMesh::cells_out(const double* internal, double* caller, int comps) {
    if (internal == caller) return;
    if (identity_order) {
        HIP_OK(hipMemcpyAsync(caller, internal, uint64_t(comps) * nc * 8, hipMemcpyDeviceToDevice, stream));
        return;
    }
    for (int k = 0; k < comps; ++k)
        gather_u32idx_kernel<<<grid_for(nc), kBlock, 0, stream>>>(nc, cell_new, internal + size_t(k) * nc,
                                                                  caller + size_t(k) * nc);
}

void FvMesh::faces_in(const double* caller, double* internal) {
    if (identity_order) {
        HIP_OK(hipMemcpyAsync(internal, caller, uint64_t(nf) * 8, hipMemcpyDeviceToDevice, stream));
        return;
    }
    gather_u32idx_kernel<<<grid_for(nf), kBlock, 0, stream>>>(nf, face_old, caller, internal);
}

void FvMesh::faces_out(const double* internal, double* caller) {
    if (internal == caller) return;
    if (identity_order) {
        HIP_OK(hipMemcpyAsync(caller, internal, uint64_t(nf) * 8, hipMemcpyDeviceToDevice, stream));
        return;
    }
    gather_u32idx_kernel<<<grid_for(nf), kBlock, 0, stream>>>(nf, face_new, internal, caller);
}

// Caller-ordered input as an internal array: the caller's own buffer when the
// numbering is kept, else a permuted copy in scratch slot `slot`.
const double* FvMesh::cin(const double* caller, size_t slot, int comps) {
    if (identity_order) return caller;
    double* b = scr(slot, uint64_t(comps) * nc);
    cells_in(caller, b, comps);
    return b;
}
const double* FvMesh::fin(const double* caller, size_t slot) {
    if (identity_order) return caller;
    double* b = scr(slot, nf);
    faces_in(caller, b);
    return b;
}
// Where a kernel writes a caller-ordered output (the caller's buffer when the
// numbering is kept); cells_out / faces_out then move it if needed.
double* FvMesh::cout_buf(double* caller, size_t slot, int comps) {
    return identity_order ? caller : scr(slot, uint64_t(comps) * nc);
}
double* FvMesh::fout_buf(double* caller, size_t slot) { return identity_order ? caller : scr(slot, nf); }

// Before the first kernel of a call (every call that may raise a flag ends
// synchronised, so none is in flight).
void FvMesh::clear_err() {
    for (int k = 0; k < 4; ++k) const_cast<volatile int*>(h_err)[k] = 0;
}

// After the call's synchronisation.
void FvMesh::check_err(const char* what) {
    const int code = *const_cast<volatile int*>(h_err);
    if (code == 0) return;
    clear_err();
    throw std::domain_error(std::string(what) + " (code " + std::to_string(code) + ")");
}

void FvMesh::compute_geometry() {
    clear_err();
    const Soa3 fc{fcx, fcy, fcz}, fs{fsx, fsy, fsz}, cc{ccx, ccy, ccz};
    face_geometry_kernel<<<grid_for(nf), kBlock, 0, stream>>>(nf, px, py, pz, foff, fvtx, fc, fs, err);
    cell_centre_kernel<<<grid_for(nc), kBlock, 0, stream>>>(nc, coff, cfaces, fc, fs, cc);
    orient_kernel<<<grid_for(nf), kBlock, 0, stream>>>(nf, owner, neigh, fc, fs, cc);
    cell_volume_kernel<<<grid_for(nc), kBlock, 0, stream>>>(nc, coff, cfaces, owner, fc, fs, cc, vol, err);
    HIP_OK(hipStreamSynchronize(stream));
    check_err("invalid face or cell geometry");
}

void FvMesh::geometry_out(double* fc_aos, double* fs_aos, double* cc_aos, double* vol_out) {
    double* tmp = dalloc<double>(3 * uint64_t(std::max(nf, nc)));
    auto out3 = [&](Soa3 s, uint32_t n, const uint32_t* map, double* h) {
        if (!h) return;
        soa_to_aos_kernel<<<grid_for(n), kBlock, 0, stream>>>(n, map, s, tmp);
        HIP_OK(hipStreamSynchronize(stream));
        download(h, tmp, 3 * uint64_t(n));
    };
    out3(Soa3{fcx, fcy, fcz}, nf, face_new, fc_aos);
    out3(Soa3{fsx, fsy, fsz}, nf, face_new, fs_aos);
    out3(Soa3{ccx, ccy, ccz}, nc, cell_new, cc_aos);
    download(vol_out, vol_caller, nc);
    dfree(tmp);
}

// Slot stencils (geometry only): built on first use.
void FvMesh::ensure_slots() {
    if (slots_built) return;
    uint32_t D = 0;
    for (uint32_t c = 0; c < nc; ++c) D = std::max(D, h_coff[c + 1] - h_coff[c]);
    if (D > 255) throw std::invalid_argument("cells with more than 255 faces are not supported");
    if (nf > kFaceReversed) throw std::invalid_argument("cell stencils: more than 2^31 faces are not supported");
    slot_D = D;
    const uint64_t m = uint64_t(D) * nc;
    release_slots();  // of an attempt that failed
    cell_rec = dalloc<double4>(nc);
    slot_other = dalloc<int32_t>(m);
    slot_face = dalloc<uint32_t>(m);
    slot_w = dalloc<double>(m);
    slot_sx = dalloc<double>(m);
    slot_sy = dalloc<double>(m);
    slot_sz = dalloc<double>(m);
    // Each cell's slots in ascending caller face id (the order of the
    // reference's face loop accumulations).
    slot_sorted = dalloc<uint8_t>(m);
    const Soa3 fc{fcx, fcy, fcz}, fs{fsx, fsy, fsz}, cc{ccx, ccy, ccz};
    clear_err();
    slot_build_kernel<<<grid_for(nc), kBlock, 0, stream>>>(nc, D, coff, cfaces, owner, neigh, patch, npatch,
                                                           patch_kind, fc, fs, cc, vol, face_old, cell_rec, slots_of(*this),
                                                           slot_sorted, err);
    HIP_OK(hipStreamSynchronize(stream));
    check_err("cell stencils: degenerate face distances");
    slots_built = true;
}

void FvMesh::release_slots() {
    slots_built = false;
    for (double** p : {&slot_w, &slot_sx, &slot_sy, &slot_sz}) dfree(*p);
    dfree(slot_other);
    dfree(slot_face);
    dfree(slot_sorted);
    dfree(cell_rec);
}

// WLS fit cache for one set of boundary types (fixed value or not, per patch).
void FvMesh::ensure_wls_cache(const uint8_t* h_bt, const uint8_t* d_bt) {
    ensure_slots();
    std::vector<uint8_t> key(npatch);
    for (uint32_t p = 0; p < npatch; ++p) key[p] = h_bt[p] == 1 ? 1 : 0;
    if (wls_meta && key == wls_key) return;
    if (slot_D > uint32_t(kMaxCellFaces))
        throw std::invalid_argument("boundary WLS: cells with more than " + std::to_string(kMaxCellFaces) +
                                    " faces are not supported");
    const uint64_t m = uint64_t(slot_D) * nc;
    if (!wls_meta) {
        for (double** p : {&wls_a0, &wls_a1, &wls_a2, &wls_fac, &wls_nd}) *p = dalloc<double>(m);
        wls_sig = dalloc<double>(3 * uint64_t(nc));
        wls_V = dalloc<double>(9 * uint64_t(nc));
        wls_cond = dalloc<double>(nc);
        wls_meta = dalloc<uint32_t>(nc);
    }
    wls_key.clear();
    const Soa3 fc{fcx, fcy, fcz}, cc{ccx, ccy, ccz};
    clear_err();
    wls_build_kernel<<<grid_for(nc), kBlock, 0, stream>>>(nc, coff, slots_of(*this), patch, npatch, d_bt, fc, cc,
                                                          stencil_dimension(), wls_of(*this), err);
    HIP_OK(hipStreamSynchronize(stream));
    check_err("boundary WLS: degenerate boundary face or normal distance");
    wls_key = key;
}

// Records (gx, gy, gz, 0) per internal cell of the field p[i * ps].
void FvMesh::gauss_gradient_internal(const uint8_t* d_bct, const double* d_bcv, const double* p, uint32_t ps) {
    if (!work_grad) work_grad = dalloc<double>(4 * uint64_t(nc));
    ensure_slots();
    gauss_gradient_kernel<true><<<grid_for(nc), kBlock, 0, stream>>>(
        nc, slot_D, slots_of(*this), patch, npatch, d_bct, d_bcv, Soa3{fcx, fcy, fcz},
        Soa3{ccx, ccy, ccz}, vol, p, ps, work_grad);
}

void FvMesh::gauss_gradient_device(const uint8_t* d_bct, const double* d_bcv, const double* d_p, double* d_grad) {
    const double* p_i = cin(d_p, 9, 1);
    double* g_i = cout_buf(d_grad, 8, 3);
    ensure_slots();
    gauss_gradient_kernel<false><<<grid_for(nc), kBlock, 0, stream>>>(
        nc, slot_D, slots_of(*this), patch, npatch, d_bct, d_bcv, Soa3{fcx, fcy, fcz},
        Soa3{ccx, ccy, ccz}, vol, p_i, 1, g_i);
    cells_out(g_i, d_grad, 3);
}

void FvMesh::mass_flux_device(const uint8_t* d_vbt, const double* d_vbv, double rho, const double* d_U,
                              double* d_phi) {
    const Soa3 fs{fsx, fsy, fsz};
    const double* u_i = cin(d_U, 0, 3);
    double* phi_i = fout_buf(d_phi, 4);
    mass_flux_kernel<<<grid_for(nf), kBlock, 0, stream>>>(nf, nc, owner, neigh, patch, npatch, patch_kind, d_vbt,
                                                          d_vbv, rho, fs, u_i, phi_i);
    faces_out(phi_i, d_phi);
}

// Sparsity of the pressure system: diagonal + face neighbours, sorted per
// row (sparse_matrix.h:76-131 canonical order); with reference-cell
// elimination the row/column `ref` is dropped and indices above it shift.
const PressurePlan& FvMesh::pressure_plan(bool eliminate, uint32_t ref) {
    PressurePlan& full = pressure_full;
    if (!full.rowp) {
        full.release();  // of an attempt that failed
        // Row c: {c} and the other cell of each internal face of c, sorted,
        // duplicates (several faces joining one pair) merged with their faces
        // listed in ascending face id. Two passes over the cell->face lists.
        std::vector<uint32_t> cnt(uint64_t(nc) + 1, 0), fcnt(uint64_t(nc) + 1, 0);
        auto row_entries = [&](uint32_t c, std::vector<std::pair<uint32_t, uint32_t>>& r) {
            r.clear();
            r.push_back({c, 0xffffffffu});
            for (uint32_t k = h_coff[c]; k < h_coff[c + 1]; ++k) {
                const uint32_t f = h_cf[k];
                if (h_neigh[f] < 0) continue;
                const uint32_t other = h_owner[f] == c ? uint32_t(h_neigh[f]) : h_owner[f];
                r.push_back({other, f});
            }
            std::sort(r.begin(), r.end());
        };
        parallel_chunks(nc, 0, [&](uint64_t b, uint64_t e, uint32_t) {
            std::vector<std::pair<uint32_t, uint32_t>> r;
            for (uint64_t c = b; c < e; ++c) {
                row_entries(uint32_t(c), r);
                uint32_t u = 0;
                for (size_t q = 0; q < r.size(); ++q) u += (q == 0 || r[q].first != r[q - 1].first);
                cnt[c + 1] = u;
                fcnt[c + 1] = uint32_t(r.size() - 1);
            }
        });
        for (uint32_t c = 0; c < nc; ++c) {
            cnt[c + 1] += cnt[c];
            fcnt[c + 1] += fcnt[c];
        }
        const uint64_t nnz = cnt[nc];
        std::vector<uint32_t> rowp(cnt.begin(), cnt.end()), cols(nnz), rdiag(nnz), nzf_off(nnz + 1, 0),
            nzf(fcnt[nc]);
        parallel_chunks(nc, 0, [&](uint64_t b, uint64_t e, uint32_t) {
            std::vector<std::pair<uint32_t, uint32_t>> r;
            for (uint64_t c = b; c < e; ++c) {
                row_entries(uint32_t(c), r);
                uint64_t w = rowp[c];
                uint32_t fw = fcnt[c];
                for (size_t q = 0; q < r.size();) {
                    const uint32_t col = r[q].first;
                    cols[w] = col;
                    rdiag[w] = col == c ? uint32_t(c) : 0xffffffffu;
                    while (q < r.size() && r[q].first == col) {
                        if (r[q].second != 0xffffffffu) nzf[fw++] = r[q].second;
                        ++q;
                    }
                    nzf_off[w + 1] = fw;
                    ++w;
                }
            }
        });
        // Device slot maps address the internal numbering: the diagonal's
        // internal row and the joining faces' internal ids (still listed in
        // ascending caller face id).
        for (auto& v : rdiag)
            if (v != 0xffffffffu) v = h_cell_new[v];
        for (auto& f : nzf) f = h_face_new[f];
        full.n = nc;
        full.nnz = nnz;
        full.h_rowp = std::move(rowp);
        full.h_cols = std::move(cols);
        full.shared_pairs = nnz != uint64_t(nc) + fcnt[nc];
        full.cols = upload(full.h_cols.data(), full.h_cols.size());
        full.nz_row_diag = upload(rdiag.data(), rdiag.size());
        full.nzf_off = upload(nzf_off.data(), nzf_off.size());
        full.nzf = upload(nzf.data(), nzf.size());
        full.rowp = upload(full.h_rowp.data(), full.h_rowp.size());  // last: the plan is whole
    }
    if (!eliminate) return full;
    PressurePlan& red = pressure_red;
    if (!red.rowp || red.ref != ref) {
        red.release();
        std::vector<uint32_t> rowp{0}, cols;
        rowp.reserve(nc);
        cols.reserve(full.nnz);
        for (uint32_t c = 0; c < nc; ++c) {
            if (c == ref) continue;
            for (uint32_t k = full.h_rowp[c]; k < full.h_rowp[c + 1]; ++k) {
                const uint32_t j = full.h_cols[k];
                if (j != ref) cols.push_back(j < ref ? j : j - 1);
            }
            rowp.push_back(uint32_t(cols.size()));
        }
        red.n = nc - 1;
        red.nnz = cols.size();
        red.ref = ref;
        red.h_rowp = std::move(rowp);
        red.h_cols = std::move(cols);
        red.shared_pairs = full.shared_pairs;
        red.cols = upload(red.h_cols.data(), red.h_cols.size());
        red.rowp = upload(red.h_rowp.data(), red.h_rowp.size());
    }
    return red;
}

// The plan with its row maps, which only the assemblies need: the calls that
// read nothing but the pattern take meshes that have no slot stencils.
const PressurePlan& FvMesh::row_plan(bool eliminate, uint32_t ref) {
    pressure_plan(eliminate, ref);
    PressurePlan& plan = eliminate ? pressure_red : pressure_full;
    if (!plan.row_start) map_rows(plan, eliminate ? ref : 0xffffffffu);
    return plan;
}

// A pattern query is followed by assemblies: lays the maps out ahead where the
// mesh has stencils. What fails here is raised by the assembly that meets it.
void FvMesh::prepare_rows(bool eliminate, uint32_t ref) {
    try {
        row_plan(eliminate, ref);
    } catch (const std::exception&) {
        (void)hipGetLastError();
    }
}

// Row maps of plan (row and column ref left out; ~0: none).
void FvMesh::map_rows(PressurePlan& plan, uint32_t ref) {
    ensure_slots();
    plan.release_maps();  // of an attempt that failed
    plan.row_of = dalloc<uint32_t>(nc);
    plan.slot_rank = dalloc<uint16_t>(uint64_t(slot_D) * nc);
    plan.diag_rank = dalloc<uint16_t>(nc);
    uint32_t* start = dalloc<uint32_t>(nc);
    map_rows_kernel<<<grid_for(nc), kBlock, 0, stream>>>(nc, slot_D, coff, slot_sorted, slot_other, cell_old,
                                                         plan.rowp, plan.cols, ref, start, plan.row_of,
                                                         plan.slot_rank, plan.diag_rank);
    plan.row_start = start;  // last: the maps are whole
}

bool FvMesh::has_fixed_pressure(const uint8_t* h_pbt) const {
    for (uint32_t p = 0; p < npatch; ++p)
        if (h_patch_boundary[p] && h_pbt[p] == 1) return true;
    return false;
}

const PressurePlan& FvMesh::pressure_assemble_device(const uint8_t* h_pbt, const double* h_pbv, double rho,
                                                     const double* d_rAU, const double* d_phi, const double* d_p,
                                                     uint64_t ref, double* d_vals, double* d_rhs) {
    const bool fixed = has_fixed_pressure(h_pbt);
    const bool eliminate = !fixed && nc > 1 && ref < nc;
    const PressurePlan& plan = row_plan(eliminate, uint32_t(eliminate ? ref : 0));
    upload_bcs(nullptr, nullptr, h_pbt, h_pbv, true, nullptr);
    const uint32_t npp = std::max<uint32_t>(npatch, 1);
    const uint8_t* d_pbt = bc_u8 + npp;
    const double* d_pbv = bc_f64 + 3 * size_t(npp);
    clear_err();
    const Soa3 fc{fcx, fcy, fcz};
    double4* rec = reinterpret_cast<double4*>(scr(5, 4 * uint64_t(nc)));
    pack_cells_kernel<<<grid_for(nc), kBlock, 0, stream>>>(nc, identity_order ? nullptr : cell_new, d_rAU, d_p, rec);
    const double* phi_i = fin(d_phi, 4);
    // A kept numbering has p at hand as an array of its own: a quarter of the
    // lines (256^3 cells in lattice order: 885 us, 1030 from records).
    if (identity_order) gauss_gradient_internal(d_pbt, d_pbv, d_p, 1);
    else gauss_gradient_internal(d_pbt, d_pbv, &rec->w, 4);
    const RowMap rm{plan.row_start, plan.row_of, plan.slot_rank, plan.diag_rank, plan.shared_pairs ? 1 : 0};
    const double4* grad = reinterpret_cast<const double4*>(work_grad);
    if (slot_D <= kRowSlots) {
        pressure_row_kernel<true><<<grid_for(nc), kBlock, row_lds(slot_D, 3), stream>>>(
            nc, slot_D, coff, slot_sorted, slots_of(*this), patch, npatch, d_pbt, d_pbv, rho, fc, cell_rec, rec, grad,
            phi_i, nullptr, rm, d_vals, d_rhs, err);
    } else {
        if (!slot_coeff) slot_coeff = dalloc<double>(uint64_t(slot_D) * nc);
        pressure_row_kernel<false><<<grid_for(nc), kBlock, 0, stream>>>(
            nc, slot_D, coff, slot_sorted, slots_of(*this), patch, npatch, d_pbt, d_pbv, rho, fc, cell_rec, rec, grad,
            phi_i, slot_coeff, rm, d_vals, d_rhs, err);
    }
    HIP_OK(hipStreamSynchronize(stream));
    check_err("pressure_face_orthogonal_coefficient: invalid face geometry or orientation");
    return plan;
}

const PressurePlan& FvMesh::diffusion_assemble_device(double gamma, const double* d_source, const double* d_fval,
                                                      const uint8_t* d_fneu, double* d_vals, double* d_rhs) {
    if (!work_coeff) work_coeff = dalloc<double>(nf);
    if (!work_diag) work_diag = dalloc<double>(nc);
    const PressurePlan& plan = pressure_plan(false, 0);
    clear_err();
    const Soa3 fc{fcx, fcy, fcz}, fs{fsx, fsy, fsz}, cc{ccx, ccy, ccz};
    const double* src_i = cin(d_source, 3, 1);
    const double* fval_i = fin(d_fval, 7);
    double* rhs_i = cout_buf(d_rhs, 8, 1);
    const uint8_t* fneu_i = d_fneu;
    if (!identity_order) {
        if (!scratch_u8) scratch_u8 = dalloc<uint8_t>(nf);
        gather_u8_kernel<<<grid_for(nf), kBlock, 0, stream>>>(nf, face_old, d_fneu, scratch_u8);
        fneu_i = scratch_u8;
    }
    diffusion_face_kernel<<<grid_for(nf), kBlock, 0, stream>>>(nf, owner, neigh, gamma, fc, fs, cc, fval_i,
                                                               work_coeff, err);
    diffusion_cell_kernel<<<grid_for(nc), kBlock, 0, stream>>>(nc, coff, cfaces_sorted, neigh, fs, vol, src_i, fval_i,
                                                               fneu_i, work_coeff, work_diag, rhs_i);
    csr_values_kernel<<<grid_for(plan.nnz), kBlock, 0, stream>>>(plan.nnz, plan.nz_row_diag, plan.nzf_off,
                                                                 plan.nzf, work_diag, work_coeff, d_vals);
    cells_out(rhs_i, d_rhs, 1);
    HIP_OK(hipStreamSynchronize(stream));
    check_err("assemble_cell_diffusion_matrix: invalid geometry");
    return plan;
}

// ============================================================ momentum side

void FvMesh::ensure_momentum_work() {
    if (mom_flags) return;
    ensure_slots();
    if (!mom_ugrad) mom_ugrad = dalloc<double>(12 * uint64_t(nc));
    // Which patches (last: the internal faces) hold non-orthogonal faces, and
    // which ones faces that do not say: geometry, so found once.
    const uint32_t nflag = 2 * (npatch + 1);
    int* flags = dalloc<int>(std::max<uint32_t>(nflag, 4));
    h_nonorth.assign(nflag, 0);
    HIP_OK(hipMemsetAsync(flags, 0, nflag * sizeof(int), stream));
    nonorth_scan_kernel<<<grid_for(nf), kBlock, 0, stream>>>(nf, owner, neigh, patch, npatch, patch_kind,
                                                             Soa3{fcx, fcy, fcz}, Soa3{fsx, fsy, fsz},
                                                             Soa3{ccx, ccy, ccz}, flags);
    HIP_OK(hipStreamSynchronize(stream));
    download(h_nonorth.data(), flags, nflag);
    mom_flags = flags;
}

// Boundary data per patch into the persistent device buffer (no allocation per
// call): bc_f64 = [3 velocity values | pressure value], bc_u8 = [velocity type |
// pressure type], written by the host into pinned memory and fetched by one
// small kernel, which also clears the call's device flags. Pressure types other
// than 1 read as zero-gradient unless raw_pbt. (Two copies of a few
// bytes and a fill took 10 us of a 222k-cell pressure assembly's 90.)
void FvMesh::upload_bcs(const uint8_t* h_vbt, const double* h_vbv, const uint8_t* h_pbt, const double* h_pbv,
                        bool raw_pbt, int* flags) {
    const size_t npp = std::max<uint32_t>(npatch, 1);
    const uint32_t words = uint32_t(4 * npp + (2 * npp + 7) / 8);
    if (!bc_host) {
        if (!bc_f64) bc_f64 = dalloc<double>(words);
        bc_u8 = reinterpret_cast<uint8_t*>(bc_f64 + 4 * npp);
        HIP_OK(hipHostMalloc(reinterpret_cast<void**>(&bc_host), words * 8, hipHostMallocMapped));
        h_bc_u8 = reinterpret_cast<uint8_t*>(bc_host + 4 * npp);
    }
    std::memset(bc_host, 0, words * 8);
    for (uint32_t p = 0; p < npatch; ++p) {
        if (h_vbt) h_bc_u8[p] = h_vbt[p] == 1 ? 1 : 0;
        if (h_pbt) h_bc_u8[npp + p] = raw_pbt ? h_pbt[p] : (h_pbt[p] == 1 ? 1 : 0);
        for (int k = 0; k < 3; ++k)
            if (h_vbv) bc_host[3 * size_t(p) + k] = h_vbv[3 * size_t(p) + k];
        if (h_pbv) bc_host[3 * npp + p] = h_pbv[p];
    }
    double* from = nullptr;
    HIP_OK(hipHostGetDevicePointer(reinterpret_cast<void**>(&from), bc_host, 0));
    fetch_bcs_kernel<<<1, kBlock, 0, stream>>>(words, from, bc_f64, flags);
}

int FvMesh::stencil_dimension() const {
    for (uint8_t k : h_kind)
        if (k == 1) return 2;
    return 3;
}

void FvMesh::wls_gradient_device(const uint8_t* h_bt, const double* h_bv, double limit, const double* d_field,
                                 double* d_grad, uint8_t* d_fallback) {
    if (!(limit >= 1.0) || !std::isfinite(limit)) throw std::invalid_argument("boundary WLS: invalid condition limit");
    uint8_t* d_bt = upload(h_bt, std::max<uint32_t>(npatch, 1));
    double* d_bv = upload(h_bv, std::max<uint32_t>(npatch, 1));
    clear_err();
    const Soa3 fc{fcx, fcy, fcz}, fs{fsx, fsy, fsz}, cc{ccx, ccy, ccz};
    double* g_i = cout_buf(d_grad, 8, 3);
    try {
        ensure_wls_cache(h_bt, d_bt);
    } catch (...) {
        dfree(d_bt);
        dfree(d_bv);
        throw;
    }
    const double* f_i = cin(d_field, 0, 1);
    wls_gradient_kernel<1><<<grid_for(nc), kBlock, 0, stream>>>(nc, coff, slots_of(*this), patch, npatch, d_bt, d_bv, 1, fc,
                                                                fs, cc, vol, stencil_dimension(), limit, wls_of(*this), f_i,
                                                                g_i, d_fallback, nullptr, err);
    cells_out(g_i, d_grad, 3);
    HIP_OK(hipStreamSynchronize(stream));
    dfree(d_bt);
    dfree(d_bv);
    check_err("boundary WLS gradient: invalid geometry, boundary data or stencil size");
}

// One stream-ordered pass, synchronised once at the end for the error flag. The
// velocity gradients are only computed when a face that counts is
// non-orthogonal (geometry and boundary types: known on the host) and diffusion
// is active (a device flag that the packing kernel sets from the viscosity).
const PressurePlan& FvMesh::momentum_assemble_device(const uint8_t* h_vbt, const double* h_vbv, const double* d_mu,
                                                     const double* d_phi, const double* d_gradp,
                                                     const double* d_body, const double* d_U, bool bounded,
                                                     double alpha, double* d_vals, double* d_rhs, double* d_diag) {
    if (!(alpha > 0.0 && alpha <= 1.0)) throw std::invalid_argument("relax_momentum_equation: invalid relaxation");
    const PressurePlan& plan = row_plan(false, 0);
    ensure_momentum_work();
    upload_bcs(h_vbt, h_vbv, nullptr, nullptr, false, mom_flags);
    const uint8_t* d_vbt = bc_u8;
    const double* d_vbv = bc_f64;
    ensure_wls_cache(h_bc_u8, d_vbt);
    const Soa3 fc{fcx, fcy, fcz}, fs{fsx, fsy, fsz}, cc{ccx, ccy, ccz};
    bool nonorthogonal = h_nonorth[npatch], undefined = h_nonorth[2 * npatch + 1];
    for (uint32_t p = 0; p < npatch; ++p) {
        if (h_bc_u8[p] != 1) continue;
        nonorthogonal = nonorthogonal || h_nonorth[p];
        undefined = undefined || h_nonorth[npatch + 1 + p];
    }
    auto records = [&](size_t slot) { return reinterpret_cast<double4*>(scr(slot, 4 * uint64_t(nc))); };
    double4 *rec = records(0), *source = records(1), *out = records(2);
    const double* phi_i = fin(d_phi, 4);
    clear_err();
    pack_momentum_kernel<<<grid_for(nc), kBlock, 0, stream>>>(nc, identity_order ? nullptr : cell_new, d_U, d_mu,
                                                              d_gradp, d_body, rec, source, mom_flags, err);
    if (nonorthogonal)
        wls_gradient_kernel<3><<<grid_for(nc), kBlock, 0, stream>>>(
            nc, coff, slots_of(*this), patch, npatch, d_vbt, d_vbv, 3, fc, fs, cc, vol, stencil_dimension(), 1.e8,
            wls_of(*this), &rec->x, mom_ugrad, nullptr, mom_flags, err);
    const RowMap rm{plan.row_start, plan.row_of, plan.slot_rank, plan.diag_rank, plan.shared_pairs ? 1 : 0};
    momentum_row_kernel<<<grid_for(nc), kBlock, size_t(kBlock) * 8 * (4 * kMomNear + slot_D + 1), stream>>>(
        nc, slot_D, coff, slot_sorted, slots_of(*this), patch, npatch, d_vbt, d_vbv, fc, cell_rec, rec, source,
        reinterpret_cast<const double4*>(mom_ugrad), phi_i, bounded ? 1 : 0, nonorthogonal ? 1 : 0, mom_flags,
        alpha != 1.0 ? 1 : 0, alpha, rm, d_vals, out, err);
    unpack_cells_kernel<<<grid_for(nc), kBlock, 0, stream>>>(nc, identity_order ? nullptr : cell_new, out, d_rhs,
                                                             d_diag);
    HIP_OK(hipStreamSynchronize(stream));
    check_err("assemble_momentum_component: invalid viscosity, flux or geometry, or non-positive diagonal");
    if (undefined)
        throw std::domain_error("assemble_momentum_component: invalid viscosity, flux or geometry, or non-positive "
                                "diagonal (code 41)");
    return plan;
}

void FvMesh::momentum_hbya_device(const double* d_vals, const double* d_rhs, const double* d_diag,
                                  const double* d_gradp, const double* d_U, double* d_rau, double* d_hbya) {
    const PressurePlan& plan = pressure_plan(false, 0);
    clear_err();
    hbya_kernel<<<grid_for(nc), kBlock, 0, stream>>>(nc, plan.rowp, plan.cols, d_vals, d_rhs, d_diag, d_gradp,
                                                     vol_caller, d_U, d_rau, d_hbya, err);
    HIP_OK(hipStreamSynchronize(stream));
    check_err("HbyA: invalid momentum diagonal or non-finite HbyA");
}

void FvMesh::velocity_correct_device(const double* d_hbya, const double* d_rau, const double* d_gradp,
                                     double* d_U) {
    velocity_correct_kernel<<<grid_for(nc), kBlock, 0, stream>>>(nc, d_hbya, d_rau, d_gradp, vol_caller, d_U);
    HIP_OK(hipStreamSynchronize(stream));
}

void FvMesh::rhie_chow_flux_device(const uint8_t* h_vbt, const double* h_vbv, const uint8_t* h_pbt,
                                   const double* h_pbv, double rho, const double* d_hbya, const double* d_p,
                                   const double* d_rau, double* d_phi) {
    upload_bcs(h_vbt, h_vbv, h_pbt, h_pbv, false, nullptr);
    const uint32_t npp = std::max<uint32_t>(npatch, 1);
    const uint8_t* d_vbt = bc_u8;
    const uint8_t* d_pbt = bc_u8 + npp;
    const double* d_vbv = bc_f64;
    const double* d_pbv = bc_f64 + 3 * size_t(npp);
    const Soa3 fc{fcx, fcy, fcz}, fs{fsx, fsy, fsz}, cc{ccx, ccy, ccz};
    clear_err();
    const double* h_i = cin(d_hbya, 6, 3);
    const double* rau_i = cin(d_rau, 5, 3);
    const double* p_i = cin(d_p, 9, 1);
    double* phi_i = fout_buf(d_phi, 4);
    gauss_gradient_internal(d_pbt, d_pbv, p_i, 1);
    rhie_chow_flux_kernel<<<grid_for(nf), kBlock, 0, stream>>>(nf, nc, owner, neigh, patch, npatch, patch_kind,
                                                               d_vbt, d_vbv, d_pbt, d_pbv, rho, fc, fs, cc, vol, h_i,
                                                               p_i, reinterpret_cast<const double4*>(work_grad), rau_i, phi_i,
                                                               err);
    faces_out(phi_i, d_phi);
    HIP_OK(hipStreamSynchronize(stream));
    check_err("make_rhie_chow_mass_flux: inverse momentum diagonal must be finite and positive, or invalid face");
}

// ------------------------------------------------ face-list operators --
//
// Green-Gauss gradient and divergence straight from a face list on caller
// device arrays (runtime/gpu/cuda_kernels.cu:7-97): no mesh handle, so no
// cell-to-face map; each face adds its contribution to its owner and (when
// neighbour >= 0) subtracts it from its neighbour through FP64 atomics, in
// no fixed order, as the reference does. Faces whose owner or neighbour lies
// outside [0, n_cells) are skipped and raise *bad.

namespace {

// Per-cell accumulation of a chunk of faces. Face lists come grouped by owner
// as a rule, so a chunk's owners, and its neighbours one cell or one row of
// cells away, lie in a window of cells that fits LDS: those contributions are
// added there and reach memory as one atomic a cell and component, 64
// consecutive cells an instruction. Contributions outside the window, and the
// chunks whose owners spread over more than the window (an ungrouped list), go
// to memory one by one. On a 160^3 lattice (12.4M faces; every contribution a
// global atomic took 1369 us for the gradient, 489 us for the divergence) the
// atomics to memory fall from 18 to about 7 a cell.
constexpr uint32_t kFacePer = 8;                       // faces a thread
constexpr uint32_t kFaceChunk = kFacePer * kBlock;
template <int C>
struct FaceWindow {
    static constexpr uint32_t kCells = C == 3 ? 1280 : 4096;
};

// term(f, o, nb, add): calls add(cell, c, value) for the face's contributions.
template <int C, class Term>
__device__ __forceinline__ void accumulate_faces(uint64_t nf, uint64_t nc, const uint32_t* __restrict__ owner,
                                                 const int64_t* __restrict__ neighbour, double* const (&out)[C],
                                                 int* bad, Term term) {
    constexpr uint32_t kW = FaceWindow<C>::kCells;
    __shared__ double win[C][kW];
    __shared__ uint32_t range[2];
    const uint64_t f0 = uint64_t(blockIdx.x) * kFaceChunk;
    uint32_t ow[kFacePer];
    uint32_t lo = 0xffffffffu, hi = 0;
#pragma unroll
    for (uint32_t k = 0; k < kFacePer; ++k) {
        const uint64_t f = f0 + k * kBlock + threadIdx.x;
        ow[k] = f < nf ? owner[f] : 0xffffffffu;
        if (ow[k] < nc) {
            lo = min(lo, ow[k]);
            hi = max(hi, ow[k]);
        }
    }
    if (threadIdx.x == 0) {
        range[0] = 0xffffffffu;
        range[1] = 0;
    }
    for (uint32_t w = threadIdx.x; w < kW; w += kBlock)
#pragma unroll
        for (int c = 0; c < C; ++c) win[c][w] = 0.0;
    __syncthreads();
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        lo = min(lo, uint32_t(__shfl_xor(int(lo), off, 64)));
        hi = max(hi, uint32_t(__shfl_xor(int(hi), off, 64)));
    }
    if ((threadIdx.x & 63) == 0) {
        atomicMin(&range[0], lo);
        atomicMax(&range[1], hi);
    }
    __syncthreads();
    const uint32_t base = range[0];
    // Nothing valid: base stays above every cell and no contribution arises.
    const uint32_t width = range[1] >= base && range[1] - base < kW ? kW : 0;
    auto add = [&](uint64_t cell, int c, double v) {
        const uint64_t w = cell - base;
        if (w < width) unsafeAtomicAdd(&win[c][w], v);
        else atomicAdd(out[c] + cell, v);
    };
#pragma unroll
    for (uint32_t k = 0; k < kFacePer; ++k) {
        const uint64_t f = f0 + k * kBlock + threadIdx.x;
        if (f >= nf) break;
        const uint64_t o = ow[k];
        const int64_t nb = neighbour[f];
        if (o >= nc || nb >= int64_t(nc)) {
            atomicOr(bad, 1);
            continue;
        }
        term(f, o, nb, add);
    }
    __syncthreads();
    for (uint32_t w = threadIdx.x; w < width; w += kBlock)
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const double v = win[c][w];
            if (v != 0.0) atomicAdd(out[c] + base + w, v);
        }
}

__global__ __launch_bounds__(kBlock) void face_gradient_kernel(uint64_t nf, uint64_t nc, const double* __restrict__ phi,
                                                               const double* __restrict__ sx,
                                                               const double* __restrict__ sy,
                                                               const double* __restrict__ sz,
                                                               const uint32_t* __restrict__ owner,
                                                               const int64_t* __restrict__ neighbour, double* gx,
                                                               double* gy, double* gz, int* bad) {
#pragma clang fp contract(off)
    double* const out[3] = {gx, gy, gz};
    accumulate_faces<3>(nf, nc, owner, neighbour, out, bad, [&](uint64_t f, uint64_t o, int64_t nb, auto add) {
        const double vf = nb >= 0 ? 0.5 * (phi[o] + phi[nb]) : phi[o];
        const double t[3] = {vf * sx[f], vf * sy[f], vf * sz[f]};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            add(o, c, t[c]);
            if (nb >= 0) add(uint64_t(nb), c, -t[c]);
        }
    });
}

__global__ __launch_bounds__(kBlock) void inverse_volume_scale_kernel(uint64_t nc, const double* __restrict__ vol,
                                                                      double* gx, double* gy, double* gz) {
#pragma clang fp contract(off)
    for (uint64_t c = blockIdx.x * uint64_t(kBlock) + threadIdx.x; c < nc; c += uint64_t(gridDim.x) * kBlock) {
        const double inv = vol[c] > 0.0 ? 1.0 / vol[c] : 0.0;
        gx[c] *= inv;
        gy[c] *= inv;
        gz[c] *= inv;
    }
}

__global__ __launch_bounds__(kBlock) void face_divergence_kernel(uint64_t nf, uint64_t nc,
                                                                 const double* __restrict__ phi_face,
                                                                 const uint32_t* __restrict__ owner,
                                                                 const int64_t* __restrict__ neighbour, double* div,
                                                                 int* bad) {
    double* const out[1] = {div};
    accumulate_faces<1>(nf, nc, owner, neighbour, out, bad, [&](uint64_t f, uint64_t o, int64_t nb, auto add) {
        const double v = phi_face[f];
        add(o, 0, v);
        if (nb >= 0) add(uint64_t(nb), 0, -v);
    });
}

// Clears the outputs (null: absent) and the index flag.
__global__ __launch_bounds__(kBlock) void face_clear_kernel(uint64_t n, double* a, double* b, double* c, int* bad) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *bad = 0;
    for (uint64_t i = blockIdx.x * uint64_t(kBlock) + threadIdx.x; i < n; i += uint64_t(gridDim.x) * kBlock) {
        a[i] = 0.0;
        if (b) b[i] = 0.0;
        if (c) c[i] = 0.0;
    }
}

uint32_t face_grid(uint64_t n) { return uint32_t(std::min<uint64_t>((n + kBlock - 1) / kBlock, 1u << 20)) + (n == 0); }

uint32_t chunks(uint64_t n_faces) {
    const uint64_t c = (n_faces + kFaceChunk - 1) / kFaceChunk;
    if (c > 0x7fffffffu) throw std::invalid_argument("face list too long");
    return uint32_t(c);
}

// Stream-ordered flag for one call; false when any face index was out of
// range.
template <class F>
bool with_index_flag(hipStream_t s, F launch) {
    int* bad = nullptr;
    HIP_OK(hipMallocAsync(reinterpret_cast<void**>(&bad), sizeof(int), s));
    launch(bad);
    HIP_OK(hipGetLastError());
    int h = 0;
    HIP_OK(hipMemcpyAsync(&h, bad, sizeof(int), hipMemcpyDeviceToHost, s));
    HIP_OK(hipFreeAsync(bad, s));
    HIP_OK(hipStreamSynchronize(s));
    return h == 0;
}

}  // namespace

bool face_gradient_gauss(const double* phi, const double* sx, const double* sy, const double* sz,
                         const uint32_t* owner, const int64_t* neighbour, const double* volume, uint64_t n_faces,
                         uint64_t n_cells, double* gx, double* gy, double* gz, hipStream_t s) {
    return with_index_flag(s, [&](int* bad) {
        face_clear_kernel<<<face_grid(n_cells), kBlock, 0, s>>>(n_cells, gx, gy, gz, bad);
        if (n_faces)
            face_gradient_kernel<<<chunks(n_faces), kBlock, 0, s>>>(n_faces, n_cells, phi, sx, sy, sz, owner,
                                                                       neighbour, gx, gy, gz, bad);
        inverse_volume_scale_kernel<<<face_grid(n_cells), kBlock, 0, s>>>(n_cells, volume, gx, gy, gz);
    });
}

bool face_divergence(const double* phi_face, const uint32_t* owner, const int64_t* neighbour, uint64_t n_faces,
                     uint64_t n_cells, double* div, hipStream_t s) {
    return with_index_flag(s, [&](int* bad) {
        face_clear_kernel<<<face_grid(n_cells), kBlock, 0, s>>>(n_cells, div, nullptr, nullptr, bad);
        if (n_faces)
            face_divergence_kernel<<<chunks(n_faces), kBlock, 0, s>>>(n_faces, n_cells, phi_face, owner,
                                                                         neighbour, div, bad);
    });
}

}  // namespace cfdxhip
