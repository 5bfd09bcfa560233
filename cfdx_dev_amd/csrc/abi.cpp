// C ABI of libcfdxhip (declared in include/cfdxhip.h). Every entry point
// catches exceptions and reports a status; the failure text is kept on the
// handle (NativeAMGPreconditioner::last_error, core/linalg/hypre_amg.h:89-96).

#include "cfdxhip.h"

#include <hip/hip_runtime.h>

#include <chrono>
#include <cmath>
#include <limits>
#include <cstring>
#include <exception>
#include <memory>
#include <new>
#include <stdexcept>
#include <algorithm>
#include <string>
#include <vector>

#include "amg_setup.h"
#include "device_amg.hpp"
#include "fv.hpp"
#include "mesh_gen.h"
#include "mpnn.hpp"

using namespace cfdxhip;

struct cfdxhip_amg {
    cfdxhip_amg_options opt{};
    AmgConfig cfg{};
    HostHierarchy host;
    std::unique_ptr<DeviceAmg> dev;
    hipStream_t stream = nullptr;
    std::string error;
    double host_setup_s = 0.0, device_setup_s = 0.0;
    double update_s = 0.0;  // wall time of the last successful update_values
    uint64_t hierarchy_builds = 0, numeric_updates = 0;
    // configure_* knobs (hypre_amg.cpp:97-135)
    uint32_t cf_cap = 0;
    double max_coarsening_fraction = 1.0;
    double max_image_ratio = 0.0;
    bool ready = false;
    // After a device refresh the level values live on the device only; the
    // host mirror keeps the patterns, transfers and aggregates.
    bool values_on_device = false;
};

struct cfdxhip_mpnn {
    std::unique_ptr<Mpnn> m;
    int32_t device = 0;
    std::string error;
};

struct cfdxhip_host_mesh {
    HostMesh m;
};

struct cfdxhip_fv {
    FvMesh mesh;
    std::string error;
};

namespace {

const char* kEmpty = "";

cfdxhip_status fail(cfdxhip_amg* h, cfdxhip_status s, const std::string& msg) {
    if (h) h->error = msg;
    return s;
}

template <class F>
cfdxhip_status guarded(cfdxhip_amg* h, F&& f) {
    try {
        return f();
    } catch (const std::bad_alloc&) {
        return fail(h, CFDXHIP_ERR_OUT_OF_MEMORY, "host allocation failed");
    } catch (const std::exception& e) {
        const std::string w = e.what();
        const bool dev = w.rfind("HIP error", 0) == 0;
        return fail(h, dev ? CFDXHIP_ERR_DEVICE : CFDXHIP_ERR_INTERNAL, w);
    } catch (...) {
        return fail(h, CFDXHIP_ERR_INTERNAL, "unknown exception");
    }
}

void configure(cfdxhip_amg* h) {
    AmgConfig c;
    c.method = h->opt.method == CFDXHIP_AMG_BOOMER_STYLE ? AMG_BOOMER_STYLE : AMG_SMOOTHED_AGGREGATION;
    // NativeAMGPreconditioner::setup policies: hypre_amg.cpp:172-186, :208.
    if (h->opt.policy == CFDXHIP_POLICY_LOW) {
        c.omega = 0.65;
        c.pre = c.post = 2;
        c.max_levels = 15;
    } else if (h->opt.policy == CFDXHIP_POLICY_FAST) {
        c.omega = 0.75;
    }
    c.require_certificate = h->opt.require_smoother_certificate != 0;
    c.theta = h->opt.strength_threshold;
    c.filter = h->opt.prolongator_filter;
    c.keep_own = h->opt.filter_keeps_aggregate != 0;
    c.threads = h->opt.host_threads;
    c.smoother64 = h->opt.smoother;
    c.smoother32 = h->opt.smoother_fp32;
    c.cheb_degree = h->opt.chebyshev_degree;
    c.cheb_degree_coarse = h->opt.chebyshev_degree_coarse;
    c.cheb_ratio = h->opt.chebyshev_ratio;
    c.cf_cap = h->cf_cap;
    c.max_coarsening_fraction = h->max_coarsening_fraction;
    c.constant_null_space = h->opt.constant_null_space != 0;
    c.half_finest = h->opt.smoother_fp16_finest != 0;
    h->cfg = c;
}

// bounded_fine_diagonal (hypre_amg.cpp:141-161): every row's diagonal is
// finite and |a_ii| >= 1e-12 max_j |a_ij| > 0.
bool bounded_fine_diagonal(const HCsr& A, const double* vals) {
    for (uint32_t i = 0; i < A.n; ++i) {
        double diag = 0.0, scale = 0.0;
        for (uint32_t k = A.rowp[i]; k < A.rowp[i + 1]; ++k) {
            if (A.cols[k] == i) diag += vals[k];
            scale = std::max(scale, std::abs(vals[k]));
        }
        if (!(scale > 0.0) || !std::isfinite(scale) || !std::isfinite(diag) || std::abs(diag) < 1e-12 * scale)
            return false;
    }
    return true;
}

// A changed setup option invalidates the hierarchy (hypre_amg.cpp:100-103):
// setup must run again.
void drop_hierarchy(cfdxhip_amg* h) {
    if (h->dev && h->opt.device >= 0) (void)hipSetDevice(h->opt.device);
    h->dev.reset();
    h->host = HostHierarchy{};
    h->ready = false;
    h->values_on_device = false;
}

void fill_result(const SolveStats& st, cfdxhip_result* r) {
    if (!r) return;
    std::memset(r, 0, sizeof(*r));
    r->status = st.status;
    r->iterations = st.iterations;
    r->residual = st.residual;
    r->residual_relative = st.residual_relative;
    r->residual_replacements = st.replacements;
    r->max_true_recursive_gap = st.max_gap;
    r->min_true_residual = st.min_true;
    r->max_true_residual = st.max_true;
    r->first_residual_replacement = st.first_replacement;
    r->last_residual_replacement = st.last_replacement;
    r->solve_seconds = st.seconds;
    r->preconditioner_applications = st.pc_applications;
}

struct DevBuf {
    void* p = nullptr;
    explicit DevBuf(size_t bytes) {
        if (hipMalloc(&p, bytes ? bytes : 1) != hipSuccess) throw std::runtime_error("HIP error: hipMalloc failed");
    }
    ~DevBuf() {
        if (p) (void)hipFree(p);
    }
    template <class T>
    T* as() const {
        return static_cast<T*>(p);
    }
};

void hip_check(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string("HIP error ") + hipGetErrorString(e) + " in " + what);
}

template <class F>
cfdxhip_status fv_guarded(cfdxhip_fv* fv, F&& f) {
    try {
        hip_check(hipSetDevice(fv->mesh.dev), "hipSetDevice");
        const cfdxhip_status s = f();
        if (s == CFDXHIP_OK) fv->error.clear();
        return s;
    } catch (const std::domain_error& e) {
        fv->error = e.what();
        return CFDXHIP_ERR_NUMERIC;
    } catch (const std::invalid_argument& e) {
        fv->error = e.what();
        return CFDXHIP_ERR_INVALID_ARGUMENT;
    } catch (const std::bad_alloc&) {
        fv->error = "host allocation failed";
        return CFDXHIP_ERR_OUT_OF_MEMORY;
    } catch (const std::exception& e) {
        fv->error = e.what();
        return std::string(e.what()).rfind("HIP error", 0) == 0 ? CFDXHIP_ERR_DEVICE : CFDXHIP_ERR_INTERNAL;
    }
}

}  // namespace

extern "C" {

const char* cfdxhip_version(void) { return "cfdxhip 0.1 (gfx950)"; }

void cfdxhip_amg_options_default(cfdxhip_amg_options* o) {
    if (!o) return;
    std::memset(o, 0, sizeof(*o));
    o->method = CFDXHIP_AMG_SMOOTHED_AGGREGATION;
    o->policy = CFDXHIP_POLICY_BALANCED;
    o->require_smoother_certificate = 1;
    o->precision = CFDXHIP_PRECISION_FP64;
    o->reorder = 1;
    o->host_threads = 0;
    o->device = 0;
    o->strength_threshold = 0.25;
    o->prolongator_filter = 0.0;
    o->smoother = CFDXHIP_SMOOTHER_JACOBI;
    o->smoother_fp32 = CFDXHIP_SMOOTHER_JACOBI;
    o->chebyshev_degree = 3;
    o->chebyshev_ratio = 30.0;
}

cfdxhip_status cfdxhip_amg_create(const cfdxhip_amg_options* options, cfdxhip_amg** out) {
    if (!out) return CFDXHIP_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    auto* h = new (std::nothrow) cfdxhip_amg();
    if (!h) return CFDXHIP_ERR_OUT_OF_MEMORY;
    if (options) h->opt = *options;
    else cfdxhip_amg_options_default(&h->opt);
    if (h->opt.method > 1 || h->opt.policy > 2 || h->opt.precision > 1 ||
        !(h->opt.strength_threshold >= 0.0 && h->opt.strength_threshold <= 1.0) ||
        !(h->opt.prolongator_filter >= 0.0 && h->opt.prolongator_filter < 1.0) || h->opt.smoother > 1 ||
        h->opt.smoother_fp32 > 1 || h->opt.smoother_fp16_finest > 1 ||
        ((h->opt.smoother == CFDXHIP_SMOOTHER_CHEBYSHEV || h->opt.smoother_fp32 == CFDXHIP_SMOOTHER_CHEBYSHEV) &&
         (h->opt.chebyshev_degree < 1 || h->opt.chebyshev_degree > 16 || h->opt.chebyshev_degree_coarse > 16 ||
          !(h->opt.chebyshev_ratio > 1.0) ||
          !std::isfinite(h->opt.chebyshev_ratio)))) {
        delete h;
        return CFDXHIP_ERR_INVALID_ARGUMENT;
    }
    configure(h);
    // device < 0: host-only handle (hierarchy construction and introspection,
    // no device work), used to check the host setup without a GPU.
    const cfdxhip_status s = h->opt.device < 0 ? CFDXHIP_OK : guarded(h, [&]() {
        hip_check(hipSetDevice(h->opt.device), "hipSetDevice");
        hip_check(hipStreamCreate(&h->stream), "hipStreamCreate");
        return CFDXHIP_OK;
    });
    if (s != CFDXHIP_OK) {
        delete h;
        return s;
    }
    *out = h;
    return CFDXHIP_OK;
}

void cfdxhip_amg_destroy(cfdxhip_amg* h) {
    if (!h) return;
    try {
        if (h->opt.device >= 0) {
            (void)hipSetDevice(h->opt.device);
            h->dev.reset();
            if (h->stream) (void)hipStreamDestroy(h->stream);
        }
    } catch (...) {
    }
    delete h;
}

const char* cfdxhip_amg_last_error(const cfdxhip_amg* h) { return h ? h->error.c_str() : kEmpty; }

// Setup from host (device == false) or device CSR arrays. Host-only
// handles build on the host. Device handles build smoothed aggregation on
// the device (build_sa_device) and Boomer-style C/F on the host; the
// damping certificate and Chebyshev bounds are computed on the device.
static cfdxhip_status setup_common(cfdxhip_amg* h, size_t n, const uint32_t* rowp, const uint32_t* cols,
                                   const double* vals, bool device) {
    if (!h) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (n == 0 || n >= UINT32_MAX || !rowp || !cols || !vals)
        return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "AMG setup requires a non-empty CSR matrix");
    const bool host_only = h->opt.device < 0;
    if (device && host_only) return fail(h, CFDXHIP_ERR_NOT_READY, "host-only handle has no device");
    return guarded(h, [&]() {
        if (!host_only) hip_check(hipSetDevice(h->opt.device), "hipSetDevice");
        const auto t0 = std::chrono::steady_clock::now();
        // Host copy of the CSR (validation, host construction, the mirror).
        HCsr A;
        A.n = A.ncols = uint32_t(n);
        A.rowp.resize(n + 1);
        if (device) hip_check(hipMemcpy(A.rowp.data(), rowp, (n + 1) * 4, hipMemcpyDeviceToHost), "copy row offsets");
        else A.rowp.assign(rowp, rowp + n + 1);
        if (A.rowp[0] != 0) return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "row_offsets[0] must be 0");
        for (size_t i = 0; i < n; ++i)
            if (A.rowp[i + 1] < A.rowp[i])
                return fail(h, CFDXHIP_ERR_SETUP_FAILED,
                            "native AMG hierarchy construction failed: AMG setup requires a non-empty, square, "
                            "finalized CSR matrix");
        const size_t nnz = A.rowp[n];
        A.cols.resize(nnz);
        A.vals.resize(nnz);
        if (device) {
            hip_check(hipMemcpy(A.cols.data(), cols, nnz * 4, hipMemcpyDeviceToHost), "copy columns");
            hip_check(hipMemcpy(A.vals.data(), vals, nnz * 8, hipMemcpyDeviceToHost), "copy values");
        } else {
            A.cols.assign(cols, cols + nnz);
            A.vals.assign(vals, vals + nnz);
        }
        if (h->cfg.constant_null_space && csr_is_valid(A) && !has_constant_null_space(A))
            return fail(h, CFDXHIP_ERR_SETUP_FAILED,
                        "native AMG hierarchy construction failed: invalid finest matrix, dimensions, CSR, or "
                        "null-space contract");
        if (h->max_image_ratio > 0.0 && (h->cfg.require_certificate || !bounded_fine_diagonal(A, A.vals.data())))
            return fail(h, CFDXHIP_ERR_SETUP_FAILED,
                        "bounded AMG action requires nonsymmetric Krylov and finite nonzero diagonal");
        HostHierarchy staged;
        std::string err;
        if (host_only) {
            if (!build_hierarchy(A, h->cfg, staged, err))
                return fail(h, CFDXHIP_ERR_SETUP_FAILED, "native AMG hierarchy construction failed: " + err);
            const auto t1 = std::chrono::steady_clock::now();
            h->host = std::move(staged);
            h->dev.reset();
            h->host_setup_s = std::chrono::duration<double>(t1 - t0).count();
            h->device_setup_s = 0.0;
            h->ready = true;
            h->values_on_device = false;
            ++h->hierarchy_builds;
            h->error.clear();
            return CFDXHIP_OK;
        }
        if (!csr_is_valid(A))
            return fail(h, CFDXHIP_ERR_SETUP_FAILED,
                        "native AMG hierarchy construction failed: AMG setup requires a non-empty, square, finalized "
                        "CSR matrix");
        AmgConfig cfg = h->cfg;
        cfg.host_bounds = false;
        std::vector<DeviceAmg::RefreshLevel> plan;
        struct PlanGuard {
            std::vector<DeviceAmg::RefreshLevel>& p;
            ~PlanGuard() {
                for (auto& R : p) DeviceAmg::free_refresh_level(R);
            }
        } guard{plan};
        const bool gpu_sa = cfg.method == AMG_SMOOTHED_AGGREGATION;
        if (gpu_sa) {
            std::unique_ptr<DevBuf> brow, bcol, bval;
            const uint32_t* drow = rowp;
            const uint32_t* dcol = cols;
            const double* dval = vals;
            if (!device) {
                brow = std::make_unique<DevBuf>((n + 1) * 4);
                bcol = std::make_unique<DevBuf>(nnz * 4);
                bval = std::make_unique<DevBuf>(nnz * 8);
                hip_check(hipMemcpy(brow->p, rowp, (n + 1) * 4, hipMemcpyHostToDevice), "copy row offsets");
                hip_check(hipMemcpy(bcol->p, cols, nnz * 4, hipMemcpyHostToDevice), "copy columns");
                hip_check(hipMemcpy(bval->p, vals, nnz * 8, hipMemcpyHostToDevice), "copy values");
                drow = brow->as<uint32_t>();
                dcol = bcol->as<uint32_t>();
                dval = bval->as<double>();
            }
            if (!DeviceAmg::build_sa_device(drow, dcol, dval, uint32_t(n), cfg, h->stream, staged, plan, err))
                return fail(h, CFDXHIP_ERR_SETUP_FAILED, "native AMG hierarchy construction failed: " + err);
        } else if (!build_hierarchy(A, cfg, staged, err)) {
            return fail(h, CFDXHIP_ERR_SETUP_FAILED, "native AMG hierarchy construction failed: " + err);
        }
        const auto t1 = std::chrono::steady_clock::now();
        auto dev = std::make_unique<DeviceAmg>();
        const bool want32 = h->opt.precision == CFDXHIP_PRECISION_FP32;
        if (!dev->build(staged, cfg, h->opt.reorder != 0, true, want32, h->stream, err, gpu_sa ? &plan : nullptr))
            return fail(h, CFDXHIP_ERR_SETUP_FAILED, err);
        double omega = 0.0;
        std::vector<double> lambda;
        if (!dev->finish_setup(h->cfg, omega, lambda, err))
            return fail(h, CFDXHIP_ERR_SETUP_FAILED, "native AMG hierarchy construction failed: " + err);
        staged.omega = omega;
        staged.lambda_max = std::move(lambda);
        const auto t2 = std::chrono::steady_clock::now();
        // Transactional commit: the previous hierarchy survives any failure above.
        h->host = std::move(staged);
        h->dev = std::move(dev);
        h->dev->max_image_ratio = h->max_image_ratio;
        h->host_setup_s = std::chrono::duration<double>(t1 - t0).count();
        h->device_setup_s = std::chrono::duration<double>(t2 - t1).count();
        h->ready = true;
        h->values_on_device = false;
        ++h->hierarchy_builds;
        h->error.clear();
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_amg_setup(cfdxhip_amg* h, size_t n, const uint32_t* rowp, const uint32_t* cols,
                                 const double* vals) {
    return setup_common(h, n, rowp, cols, vals, false);
}

cfdxhip_status cfdxhip_amg_setup_device(cfdxhip_amg* h, size_t n, const uint32_t* rowp, const uint32_t* cols,
                                        const double* vals) {
    return setup_common(h, n, rowp, cols, vals, true);
}

static cfdxhip_status update_host(cfdxhip_amg* h, const double* vals);

static cfdxhip_status update_common(cfdxhip_amg* h, const double* vals, bool device) {
    if (!h) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready || !vals)
        return fail(h, CFDXHIP_ERR_NOT_READY, "native AMG numeric update requires an existing compatible hierarchy");
    if (device && !h->dev) return fail(h, CFDXHIP_ERR_NOT_READY, "host-only handle has no device hierarchy");
    if (!h->dev) return update_host(h, vals);
    return guarded(h, [&]() {
        const auto t0 = std::chrono::steady_clock::now();
        hip_check(hipSetDevice(h->opt.device), "hipSetDevice");
        const double* dv = vals;
        std::unique_ptr<DevBuf> staging;
        if (!device) {
            const size_t nnz = h->host.lv[0].A.nnz();
            staging = std::make_unique<DevBuf>(nnz * 8);
            hip_check(hipMemcpy(staging->p, vals, nnz * 8, hipMemcpyHostToDevice), "copy values");
            dv = staging->as<double>();
        }
        if (h->max_image_ratio > 0.0 || h->cfg.constant_null_space) {
            const HCsr& A0 = h->host.lv[0].A;
            std::vector<double> hv;
            const double* check = vals;
            if (device) {
                hv.resize(A0.nnz());
                hip_check(hipMemcpy(hv.data(), vals, hv.size() * 8, hipMemcpyDeviceToHost), "copy values");
                check = hv.data();
            }
            if (h->max_image_ratio > 0.0 && !bounded_fine_diagonal(A0, check))
                return fail(h, CFDXHIP_ERR_NUMERIC, "bounded AMG update requires safe diagonal");
            if (h->cfg.constant_null_space && !has_constant_null_space(A0, check))
                return fail(h, CFDXHIP_ERR_NUMERIC, "native AMG numeric update failed: null-space contract");
        }
        double omega = 0.0;
        std::vector<double> lambda;
        std::string err;
        bool pattern = false;
        bool ok = false;
        try {
            ok = h->dev->refresh_device(dv, h->cfg, omega, lambda, err, pattern);
        } catch (...) {
            // A device error part-way may leave the hierarchy inconsistent.
            h->ready = false;
            throw;
        }
        if (!ok)
            return fail(h, pattern ? CFDXHIP_ERR_PATTERN_CHANGED : CFDXHIP_ERR_NUMERIC,
                        "native AMG numeric update failed: " + err);
        h->host.omega = omega;
        if (!lambda.empty()) h->host.lambda_max = std::move(lambda);
        h->values_on_device = true;
        ++h->numeric_updates;
        h->update_s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
        h->error.clear();
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_amg_update_values(cfdxhip_amg* h, const double* vals) { return update_common(h, vals, false); }
cfdxhip_status cfdxhip_amg_update_values_device(cfdxhip_amg* h, const double* vals) {
    return update_common(h, vals, true);
}

// Host-only handles: the host restatement of the refresh.
static cfdxhip_status update_host(cfdxhip_amg* h, const double* vals) {
    if (h->max_image_ratio > 0.0 && !bounded_fine_diagonal(h->host.lv[0].A, vals))
        return fail(h, CFDXHIP_ERR_NUMERIC, "bounded AMG update requires safe diagonal");
    return guarded(h, [&]() {
        const auto t0 = std::chrono::steady_clock::now();
        HostHierarchy staged = h->host;
        std::string err;
        if (!refresh_hierarchy(staged, h->cfg, vals, err)) {
            const bool pattern = err.find("pattern") != std::string::npos;
            return fail(h, pattern ? CFDXHIP_ERR_PATTERN_CHANGED : CFDXHIP_ERR_NUMERIC,
                        "native AMG numeric update failed: " + err);
        }
        h->host = std::move(staged);
        ++h->numeric_updates;
        h->update_s = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
        h->error.clear();
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_amg_apply(cfdxhip_amg* h, const double* r, double* z) {
    if (!h) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready) return fail(h, CFDXHIP_ERR_NOT_READY, "native AMG preconditioner has not been set up");
    if (!h->dev) return fail(h, CFDXHIP_ERR_NOT_READY, "host-only handle has no device hierarchy");
    if (!r || !z) return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "null vector");
    return guarded(h, [&]() {
        hip_check(hipSetDevice(h->opt.device), "hipSetDevice");
        const uint32_t n = h->dev->n();
        for (uint32_t i = 0; i < n; ++i)
            if (!std::isfinite(r[i])) return fail(h, CFDXHIP_ERR_NUMERIC, "non-finite residual");
        DevBuf dr(size_t(n) * 8), dz(size_t(n) * 8);
        hip_check(hipMemcpy(dr.p, r, size_t(n) * 8, hipMemcpyHostToDevice), "copy r");
        std::string err;
        if (!h->dev->apply_caller(dr.as<double>(), dz.as<double>(), h->opt.precision == CFDXHIP_PRECISION_FP32, err))
            return fail(h, CFDXHIP_ERR_NUMERIC, err);
        hip_check(hipMemcpy(z, dz.p, size_t(n) * 8, hipMemcpyDeviceToHost), "copy z");
        for (uint32_t i = 0; i < n; ++i)
            if (!std::isfinite(z[i])) return fail(h, CFDXHIP_ERR_NUMERIC, "native AMG V-cycle failed: non-finite correction");
        h->error.clear();
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_amg_apply_device(cfdxhip_amg* h, const double* r, double* z) {
    if (!h) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready) return fail(h, CFDXHIP_ERR_NOT_READY, "native AMG preconditioner has not been set up");
    if (!h->dev) return fail(h, CFDXHIP_ERR_NOT_READY, "host-only handle has no device hierarchy");
    if (!r || !z) return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "null vector");
    return guarded(h, [&]() {
        hip_check(hipSetDevice(h->opt.device), "hipSetDevice");
        std::string err;
        if (!h->dev->apply_caller(r, z, h->opt.precision == CFDXHIP_PRECISION_FP32, err))
            return fail(h, CFDXHIP_ERR_NUMERIC, err);
        h->error.clear();
        return CFDXHIP_OK;
    });
}

static cfdxhip_status solve_common(cfdxhip_amg* h, const double* b, double* x, bool device, bool fgmres,
                                   int restart, size_t max_iter, double tol, cfdxhip_result* result) {
    if (!h) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready) return fail(h, CFDXHIP_ERR_NOT_READY, "native AMG preconditioner has not been set up");
    if (!h->dev) return fail(h, CFDXHIP_ERR_NOT_READY, "host-only handle has no device hierarchy");
    if (!b || !x || max_iter == 0 || !(tol > 0.0) || !std::isfinite(tol))
        return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "invalid solve arguments");
    return guarded(h, [&]() {
        hip_check(hipSetDevice(h->opt.device), "hipSetDevice");
        const uint32_t n = h->dev->n();
        SolveStats st;
        std::string err;
        bool ok;
        const bool mixed = h->opt.precision == CFDXHIP_PRECISION_FP32;
        if (device) {
            ok = fgmres ? h->dev->fgmres(b, x, restart, max_iter, tol, mixed, st, err)
                        : h->dev->pcg(b, x, max_iter, tol, st, err);
        } else {
            DevBuf db(size_t(n) * 8), dx(size_t(n) * 8);
            hip_check(hipMemcpy(db.p, b, size_t(n) * 8, hipMemcpyHostToDevice), "copy b");
            hip_check(hipMemcpy(dx.p, x, size_t(n) * 8, hipMemcpyHostToDevice), "copy x");
            ok = fgmres ? h->dev->fgmres(db.as<double>(), dx.as<double>(), restart, max_iter, tol, mixed, st, err)
                        : h->dev->pcg(db.as<double>(), dx.as<double>(), max_iter, tol, st, err);
            hip_check(hipMemcpy(x, dx.p, size_t(n) * 8, hipMemcpyDeviceToHost), "copy x");
        }
        if (!ok) return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, err);
        fill_result(st, result);
        h->error.clear();
        return CFDXHIP_OK;
    });
}

namespace {

double hypot_norm(const double* v, size_t n) {
    double s = 0.0;
    for (size_t i = 0; i < n; ++i) s = std::hypot(s, v[i]);
    return s;
}

double seq_dot(const double* a, const double* b, size_t n) {
    double s = 0.0;
    for (size_t i = 0; i < n; ++i) s += a[i] * b[i];
    return s;
}

}  // namespace

cfdxhip_status cfdxhip_amg_solve_cg_projected(cfdxhip_amg* h, const double* b, double* x, size_t max_iter,
                                              double tol, const double* basis, size_t basis_count,
                                              cfdxhip_result* result) {
    if (!h) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready) return fail(h, CFDXHIP_ERR_NOT_READY, "native AMG preconditioner has not been set up");
    if (!h->dev) return fail(h, CFDXHIP_ERR_NOT_READY, "host-only handle has no device hierarchy");
    if (!b || !x || !basis || basis_count == 0 || max_iter == 0 || !(tol > 0.0) || !std::isfinite(tol))
        return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "invalid solve arguments");
    return guarded(h, [&]() {
        hip_check(hipSetDevice(h->opt.device), "hipSetDevice");
        const uint32_t n = h->dev->n();
        // NullSpaceProjector construction (null_space.h:22-51).
        std::vector<double> modes;
        for (size_t q = 0; q < basis_count; ++q) {
            std::vector<double> v(basis + q * n, basis + (q + 1) * n);
            for (double e : v)
                if (!std::isfinite(e)) return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "null space basis contains non-finite values");
            const double input_norm = hypot_norm(v.data(), n);
            if (!(input_norm > 0.0))
                return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "null space basis contains a zero vector");
            for (int pass = 0; pass < 2; ++pass)
                for (size_t a = 0; a < q; ++a) {
                    const double* m = modes.data() + a * n;
                    const double c = seq_dot(v.data(), m, n);
                    for (uint32_t i = 0; i < n; ++i) v[i] -= c * m[i];
                }
            const double norm = hypot_norm(v.data(), n);
            const double threshold =
                64.0 * std::numeric_limits<double>::epsilon() * std::sqrt(double(n)) * input_norm;
            if (!(norm > threshold) || !std::isfinite(norm))
                return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "null space basis is linearly dependent");
            const double inv = 1.0 / norm;
            for (double& e : v) e *= inv;
            modes.insert(modes.end(), v.begin(), v.end());
        }
        // Applicability (cg_solver.h:74-81): b compatible, A m ~ 0.
        double comp = 0.0;
        for (size_t q = 0; q < basis_count; ++q) {
            const double c = seq_dot(b, modes.data() + q * n, n);
            comp += c * c;
        }
        const HCsr& A0 = h->host.lv[0].A;
        std::vector<double> vals;
        if (h->values_on_device) h->dev->level_values(0, vals);
        const double* av = h->values_on_device ? vals.data() : A0.vals.data();
        const double anorm = hypot_norm(av, A0.nnz());
        double worst = 0.0;
        std::vector<double> y(n);
        for (size_t q = 0; q < basis_count; ++q) {
            const double* m = modes.data() + q * n;
            for (uint32_t i = 0; i < n; ++i) {
                double sum = 0.0;
                for (uint32_t k = A0.rowp[i]; k < A0.rowp[i + 1]; ++k) sum += av[k] * m[A0.cols[k]];
                y[i] = sum;
            }
            worst = std::max(worst, hypot_norm(y.data(), n) / std::max(anorm, std::numeric_limits<double>::min()));
        }
        if (!(std::sqrt(std::max(0.0, comp)) <= 1e-14 + 1e-12 * hypot_norm(b, n)) || !(worst <= 1e-12)) {
            if (result) {
                std::memset(result, 0, sizeof(*result));
                result->status = CFDXHIP_SOLVER_NOT_APPLICABLE;
            }
            h->error.clear();
            return CFDXHIP_OK;
        }
        DevBuf db(size_t(n) * 8), dx(size_t(n) * 8), dm(modes.size() * 8), ds(modes.size() * 8);
        hip_check(hipMemcpy(db.p, b, size_t(n) * 8, hipMemcpyHostToDevice), "copy b");
        hip_check(hipMemcpy(dx.p, x, size_t(n) * 8, hipMemcpyHostToDevice), "copy x");
        hip_check(hipMemcpy(dm.p, modes.data(), modes.size() * 8, hipMemcpyHostToDevice), "copy basis");
        h->dev->to_solve_order(dm.as<double>(), ds.as<double>(), uint32_t(basis_count));
        SolveStats st;
        std::string err;
        const bool ok = h->dev->pcg(db.as<double>(), dx.as<double>(), max_iter, tol, st, err, ds.as<double>(),
                                    uint32_t(basis_count));
        hip_check(hipMemcpy(x, dx.p, size_t(n) * 8, hipMemcpyDeviceToHost), "copy x");
        if (!ok) return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, err);
        fill_result(st, result);
        h->error.clear();
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_amg_solve_cg_device_noalloc(cfdxhip_amg* h, const double* b, double* x, size_t max_iter,
                                                   double tol, cfdxhip_result* result) {
    if (!h) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready) return fail(h, CFDXHIP_ERR_NOT_READY, "native AMG preconditioner has not been set up");
    if (!h->dev) return fail(h, CFDXHIP_ERR_NOT_READY, "host-only handle has no device hierarchy");
    if (!b || !x || max_iter == 0 || !(tol > 0.0) || !std::isfinite(tol))
        return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "invalid solve arguments");
    if (h->max_image_ratio > 0.0)
        return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "allocation-free PCG: the bounded action is not supported");
    return guarded(h, [&]() {
        hip_check(hipSetDevice(h->opt.device), "hipSetDevice");
        const uint64_t need = h->dev->pcg_work_bytes(kNoAllocAlign);
        if (need > kNoAllocScratchBytes)
            return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT,
                        "allocation-free PCG: " + std::to_string(h->dev->n()) + " unknowns need " +
                            std::to_string(need) + " bytes of work memory, more than its fixed " +
                            std::to_string(kNoAllocScratchBytes) + "-byte array");
        unsigned char* base = nullptr;
        std::string err;
        if (!noalloc_scratch(h->opt.device, base, err)) return fail(h, CFDXHIP_ERR_DEVICE, err);
        SolveStats st;
        if (!h->dev->pcg_in(h->dev->pcg_work_at(base, kNoAllocAlign), b, x, max_iter, tol, st, err))
            return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, err);
        fill_result(st, result);
        h->error.clear();
        return CFDXHIP_OK;
    });
}
cfdxhip_status cfdxhip_amg_solve_cg(cfdxhip_amg* h, const double* b, double* x, size_t max_iter, double tol,
                                    cfdxhip_result* result) {
    return solve_common(h, b, x, false, false, 0, max_iter, tol, result);
}
cfdxhip_status cfdxhip_amg_solve_fgmres(cfdxhip_amg* h, const double* b, double* x, int restart, size_t max_iter,
                                        double tol, cfdxhip_result* result) {
    if (h && restart <= 0) return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "restart must be positive");
    return solve_common(h, b, x, false, true, restart, max_iter, tol, result);
}
cfdxhip_status cfdxhip_amg_solve_cg_device(cfdxhip_amg* h, const double* b, double* x, size_t max_iter,
                                           double tol, cfdxhip_result* result) {
    return solve_common(h, b, x, true, false, 0, max_iter, tol, result);
}
cfdxhip_status cfdxhip_amg_solve_fgmres_device(cfdxhip_amg* h, const double* b, double* x, int restart,
                                               size_t max_iter, double tol, cfdxhip_result* result) {
    if (h && restart <= 0) return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "restart must be positive");
    return solve_common(h, b, x, true, true, restart, max_iter, tol, result);
}

cfdxhip_status cfdxhip_amg_num_levels(const cfdxhip_amg* h, size_t* levels) {
    if (!h || !levels) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready) return CFDXHIP_ERR_NOT_READY;
    *levels = h->host.lv.size();
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_level_info(const cfdxhip_amg* h, size_t level, size_t* n, size_t* nnz, size_t* pnnz) {
    if (!h || !n || !nnz || !pnnz) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready) return CFDXHIP_ERR_NOT_READY;
    if (level >= h->host.lv.size()) return CFDXHIP_ERR_INVALID_ARGUMENT;
    const HostLevel& L = h->host.lv[level];
    *n = L.A.n;
    *nnz = L.A.nnz();
    *pnnz = L.P.nnz();
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_level_matrix(const cfdxhip_amg* h, size_t level, uint32_t* rowp, uint32_t* cols,
                                        double* vals) {
    if (!h || !rowp || !cols || !vals) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready) return CFDXHIP_ERR_NOT_READY;
    if (level >= h->host.lv.size()) return CFDXHIP_ERR_INVALID_ARGUMENT;
    const HCsr& A = h->host.lv[level].A;
    std::memcpy(rowp, A.rowp.data(), A.rowp.size() * 4);
    std::memcpy(cols, A.cols.data(), A.cols.size() * 4);
    if (h->values_on_device && h->dev) {
        try {
            (void)hipSetDevice(h->opt.device);
            std::vector<double> v;
            if (!h->dev->level_values(level, v) || v.size() != A.vals.size()) return CFDXHIP_ERR_INTERNAL;
            std::memcpy(vals, v.data(), v.size() * 8);
        } catch (...) {
            return CFDXHIP_ERR_DEVICE;
        }
        return CFDXHIP_OK;
    }
    std::memcpy(vals, A.vals.data(), A.vals.size() * 8);
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_level_transfer(const cfdxhip_amg* h, size_t level, uint64_t* agg, uint32_t* prowp,
                                          uint32_t* pcols, double* pvals) {
    if (!h || !agg || !prowp || !pcols || !pvals) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready) return CFDXHIP_ERR_NOT_READY;
    if (level + 1 >= h->host.lv.size()) return CFDXHIP_ERR_INVALID_ARGUMENT;
    const HostLevel& L = h->host.lv[level];
    for (size_t i = 0; i < L.aggregate.size(); ++i) agg[i] = L.aggregate[i];
    std::memcpy(prowp, L.P.rowp.data(), L.P.rowp.size() * 4);
    std::memcpy(pcols, L.P.cols.data(), L.P.cols.size() * 4);
    std::memcpy(pvals, L.P.vals.data(), L.P.vals.size() * 8);
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_smoother_omega(const cfdxhip_amg* h, double* omega) {
    if (!h || !omega) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready) return CFDXHIP_ERR_NOT_READY;
    *omega = h->host.omega;
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_level_lambda_max(const cfdxhip_amg* h, size_t level, double* lambda_max) {
    if (!h || !lambda_max) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready || h->host.lambda_max.empty()) return CFDXHIP_ERR_NOT_READY;
    if (level >= h->host.lambda_max.size()) return CFDXHIP_ERR_INVALID_ARGUMENT;
    *lambda_max = h->host.lambda_max[level];
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_set_chebyshev_levels(cfdxhip_amg* h, uint32_t degree, uint32_t degree_coarse,
                                                double ratio) {
    if (!h) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (degree < 1 || degree > 16 || degree_coarse > 16 || !(ratio > 1.0) || !std::isfinite(ratio))
        return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT,
                    "Chebyshev degree must be in [1, 16], the coarse degree in [0, 16], and ratio > 1");
    if (!h->ready || h->host.lambda_max.empty())
        return fail(h, CFDXHIP_ERR_NOT_READY, "no Chebyshev smoother configured on a set-up hierarchy");
    return guarded(h, [&]() {
        if (h->dev) {
            hip_check(hipSetDevice(h->opt.device), "hipSetDevice");
            try {
                h->dev->set_chebyshev_params(h->host, degree, degree_coarse, ratio);
            } catch (...) {
                // The device's coefficients may be the old ones.
                h->ready = false;
                throw;
            }
        }
        h->opt.chebyshev_degree = degree;
        h->opt.chebyshev_degree_coarse = degree_coarse;
        h->opt.chebyshev_ratio = ratio;
        h->cfg.cheb_degree = degree;
        h->cfg.cheb_degree_coarse = degree_coarse;
        h->cfg.cheb_ratio = ratio;
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_amg_set_chebyshev(cfdxhip_amg* h, uint32_t degree, double ratio) {
    if (!h) return CFDXHIP_ERR_INVALID_ARGUMENT;
    return cfdxhip_amg_set_chebyshev_levels(h, degree, h->opt.chebyshev_degree_coarse, ratio);
}

cfdxhip_status cfdxhip_amg_counters(const cfdxhip_amg* h, uint64_t* coarse_size, uint64_t* hierarchy_builds,
                                    uint64_t* numeric_updates) {
    if (!h || !coarse_size || !hierarchy_builds || !numeric_updates) return CFDXHIP_ERR_INVALID_ARGUMENT;
    const auto& lv = h->host.lv;
    *coarse_size = !h->ready || lv.empty() ? 0 : lv.size() < 2 ? lv[0].A.n : lv[1].A.n;
    *hierarchy_builds = h->hierarchy_builds;
    *numeric_updates = h->numeric_updates;
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_configure_cf_interpolation_limit(cfdxhip_amg* h, size_t max_entries) {
    if (!h) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (max_entries == 1 || max_entries > UINT32_MAX)
        return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "AMG C/F row cap must be 0 or >=2");
    if (h->cf_cap != max_entries) drop_hierarchy(h);
    h->cf_cap = uint32_t(max_entries);
    configure(h);
    h->error.clear();
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_cf_interpolation_limit(const cfdxhip_amg* h, size_t* max_entries) {
    if (!h || !max_entries) return CFDXHIP_ERR_INVALID_ARGUMENT;
    *max_entries = h->cf_cap;
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_configure_max_coarsening_fraction(cfdxhip_amg* h, double fraction) {
    if (!h) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!std::isfinite(fraction) || fraction < 0.5 || fraction > 1.0)
        return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "AMG coarsening fraction must lie in [0.5,1]");
    if (h->max_coarsening_fraction != fraction) drop_hierarchy(h);
    h->max_coarsening_fraction = fraction;
    configure(h);
    h->error.clear();
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_configure_bounded_nonsymmetric_action(cfdxhip_amg* h, double max_image_ratio) {
    if (!h) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!std::isfinite(max_image_ratio) ||
        (max_image_ratio != 0.0 && (max_image_ratio < 1.0 || max_image_ratio > 1e6)))
        return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "AMG bounded-action ratio must be 0 or in [1,1e6]");
    if (h->max_image_ratio != max_image_ratio) drop_hierarchy(h);
    h->max_image_ratio = max_image_ratio;
    if (h->dev) h->dev->bounded_fallbacks = 0;
    h->error.clear();
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_bounded_action_fallbacks(const cfdxhip_amg* h, uint64_t* fallbacks) {
    if (!h || !fallbacks) return CFDXHIP_ERR_INVALID_ARGUMENT;
    *fallbacks = h->dev ? h->dev->bounded_fallbacks : 0;
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_complexity(const cfdxhip_amg* h, double* operator_complexity, double* grid_complexity) {
    if (!h || !operator_complexity || !grid_complexity) return CFDXHIP_ERR_INVALID_ARGUMENT;
    *operator_complexity = *grid_complexity = 0.0;
    const auto& lv = h->host.lv;
    if (!h->ready || lv.empty() || lv[0].A.nnz() == 0) return CFDXHIP_OK;
    double nnz = 0.0, rows = 0.0;
    for (const HostLevel& L : lv) {
        nnz += double(L.A.nnz());
        rows += double(L.A.n);
    }
    *operator_complexity = nnz / double(lv[0].A.nnz());
    *grid_complexity = rows / double(lv[0].A.n);
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_prolongation_stats(const cfdxhip_amg* h, uint64_t* first_nnz, double* row_sum_min,
                                              double* row_sum_max) {
    if (!h || !first_nnz || !row_sum_min || !row_sum_max) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready) return CFDXHIP_ERR_NOT_READY;
    const auto& lv = h->host.lv;
    if (lv.size() < 2 || lv[0].P.n == 0) return CFDXHIP_ERR_INVALID_ARGUMENT;  // hierarchy of one level
    const HCsr& P = lv[0].P;
    double lo = std::numeric_limits<double>::infinity(), hi = -lo;
    for (uint32_t i = 0; i < P.n; ++i) {
        double sum = 0.0;
        for (uint32_t k = P.rowp[i]; k < P.rowp[i + 1]; ++k) sum += P.vals[k];
        lo = std::min(lo, sum);
        hi = std::max(hi, sum);
    }
    *first_nnz = P.nnz();
    *row_sum_min = lo;
    *row_sum_max = hi;
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_setup_seconds(const cfdxhip_amg* h, double* hs, double* ds) {
    if (!h || !hs || !ds) return CFDXHIP_ERR_INVALID_ARGUMENT;
    *hs = h->host_setup_s;
    *ds = h->device_setup_s;
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_update_seconds(const cfdxhip_amg* h, double* seconds) {
    if (!h || !seconds) return CFDXHIP_ERR_INVALID_ARGUMENT;
    *seconds = h->update_s;
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_level_kernel_seconds(cfdxhip_amg* h, size_t level, uint32_t precision, uint32_t kind,
                                                uint32_t repeat, double* seconds) {
    if (!h || !seconds) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready || !h->dev) return fail(h, CFDXHIP_ERR_NOT_READY, "not set up on a device");
    return guarded(h, [&]() {
        hip_check(hipSetDevice(h->opt.device), "hipSetDevice");
        std::string err;
        if (!h->dev->level_kernel_seconds(uint32_t(level), precision, kind, repeat, *seconds, err))
            return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, err);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_amg_gram_schmidt_seconds(cfdxhip_amg* h, uint32_t j, uint32_t repeat, double* dot_seconds,
                                                double* update_seconds) {
    if (!h || !dot_seconds || !update_seconds) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready || !h->dev) return fail(h, CFDXHIP_ERR_NOT_READY, "not set up on a device");
    return guarded(h, [&]() {
        hip_check(hipSetDevice(h->opt.device), "hipSetDevice");
        std::string err;
        if (!h->dev->gram_schmidt_seconds(j, repeat, *dot_seconds, *update_seconds, err))
            return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, err);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_amg_coarse_end(const cfdxhip_amg* h, size_t* first_level) {
    if (!h || !first_level) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready || !h->dev) return CFDXHIP_ERR_NOT_READY;
    *first_level = h->dev->coarse_end_level();
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_level_spmv_format(const cfdxhip_amg* h, size_t level, uint32_t* format,
                                             uint64_t* stored_entries, uint64_t* slices) {
    if (!h || !format || !stored_entries || !slices) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready || !h->dev) return CFDXHIP_ERR_NOT_READY;
    if (level >= h->dev->num_levels()) return CFDXHIP_ERR_INVALID_ARGUMENT;
    const DevCsr& A = h->dev->level_matrix(level);
    *format = A.nslices ? 1u : 0u;
    *stored_entries = A.nslices ? A.sell_entries : A.nnz;
    *slices = A.nslices;
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_level_spmv_bytes(const cfdxhip_amg* h, size_t level, uint32_t precision,
                                            uint64_t* matrix_bytes) {
    if (!h || !matrix_bytes || precision > 2) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready || !h->dev) return CFDXHIP_ERR_NOT_READY;
    if (level >= h->dev->num_levels()) return CFDXHIP_ERR_INVALID_ARGUMENT;
    const DevCsr& A = h->dev->level_matrix(level);
    if (precision == 2) {
        if (!A.hvals) return CFDXHIP_ERR_NOT_READY;
        *matrix_bytes = A.half_bytes;
        return CFDXHIP_OK;
    }
    if ((precision == 0 && !A.v64) || (precision == 1 && !A.v32)) return CFDXHIP_ERR_NOT_READY;
    const uint64_t sv = precision == 0 ? 8 : 4;
    if (!A.nslices)
        *matrix_bytes = A.nnz * (sv + 4) + 4 * (uint64_t(A.n) + 1);
    else
        *matrix_bytes = A.sell_entries * (sv + 4) + 4 * (uint64_t(A.nslices) + 1);
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_amg_spmv_device(cfdxhip_amg* h, uint32_t precision, const void* x, void* y, uint32_t repeat,
                                       double* seconds) {
    if (!h) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h->ready || !h->dev) return fail(h, CFDXHIP_ERR_NOT_READY, "not set up on a device");
    if (!x || !y || precision > 1) return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "invalid SpMV arguments");
    return guarded(h, [&]() {
        hip_check(hipSetDevice(h->opt.device), "hipSetDevice");
        double sec = 0.0;
        std::string err;
        if (!h->dev->spmv_caller(precision, x, y, repeat, sec, err)) return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, err);
        if (seconds) *seconds = sec;
        return CFDXHIP_OK;
    });
}

// ------------------------------------------------------------------ mesh --

cfdxhip_status cfdxhip_mesh_generate(const cfdxhip_mesh_spec* spec, cfdxhip_host_mesh** out) {
    if (!spec || !out) return CFDXHIP_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    try {
        MeshSpec s;
        s.kind = spec->kind;
        s.nx = spec->nx;
        s.ny = spec->ny;
        s.nz = spec->nz;
        s.lx = spec->lx;
        s.ly = spec->ly;
        s.lz = spec->lz;
        s.jitter = spec->jitter;
        s.wall_layers = spec->wall_layers;
        s.first_aspect = spec->first_aspect;
        s.growth = spec->growth;
        s.step_height_fraction = spec->step_height_fraction;
        s.step_length_fraction = spec->step_length_fraction;
        s.permute = spec->permute;
        s.seed = spec->seed;
        if (s.kind > 2 || s.jitter < 0.0 || s.jitter >= 0.5) return CFDXHIP_ERR_INVALID_ARGUMENT;
        auto* m = new cfdxhip_host_mesh();
        m->m = generate_mesh(s);
        *out = m;
        return CFDXHIP_OK;
    } catch (const std::bad_alloc&) {
        return CFDXHIP_ERR_OUT_OF_MEMORY;
    } catch (...) {
        return CFDXHIP_ERR_INVALID_ARGUMENT;
    }
}

cfdxhip_status cfdxhip_mesh_sizes_get(const cfdxhip_host_mesh* mm, cfdxhip_mesh_sizes* s) {
    if (!mm || !s) return CFDXHIP_ERR_INVALID_ARGUMENT;
    const HostMesh& m = mm->m;
    s->n_points = m.px.size();
    s->n_faces = m.owner.size();
    s->n_internal_faces = m.n_internal_faces;
    s->n_cells = m.n_cells;
    s->n_face_vertices = m.fvtx.size();
    s->n_cell_faces = m.cfaces.size();
    s->n_patches = m.n_patches;
    return CFDXHIP_OK;
}

cfdxhip_status cfdxhip_mesh_copy(const cfdxhip_host_mesh* mm, double* px, double* py, double* pz, uint32_t* foff,
                                 uint32_t* fvtx, uint32_t* owner, int32_t* neigh, uint32_t* coff, uint32_t* cfaces,
                                 uint32_t* patch_of_face, uint8_t* patch_kind, uint32_t* cell_ijk) {
    if (!mm) return CFDXHIP_ERR_INVALID_ARGUMENT;
    const HostMesh& m = mm->m;
    auto cp = [](void* dst, const auto& v) {
        if (dst && !v.empty()) std::memcpy(dst, v.data(), v.size() * sizeof(v[0]));
    };
    cp(px, m.px);
    cp(py, m.py);
    cp(pz, m.pz);
    cp(foff, m.foff);
    cp(fvtx, m.fvtx);
    cp(owner, m.owner);
    cp(neigh, m.neigh);
    cp(coff, m.coff);
    cp(cfaces, m.cfaces);
    cp(patch_of_face, m.patch_of_face);
    cp(patch_kind, m.patch_kind);
    cp(cell_ijk, m.cell_ijk);
    return CFDXHIP_OK;
}

void cfdxhip_mesh_destroy(cfdxhip_host_mesh* m) { delete m; }

// ----------------------------------------------------------------- fv --

cfdxhip_status cfdxhip_fv_create(int32_t device, size_t np, const double* px, const double* py, const double* pz,
                                 size_t nf, const uint32_t* foff, const uint32_t* fvtx, const uint32_t* owner,
                                 const int32_t* neigh, size_t nc, const uint32_t* coff, const uint32_t* cf,
                                 size_t npatch, const uint32_t* patch, const uint8_t* kind, cfdxhip_fv** out) {
    if (!out || !px || !py || !pz || !foff || !fvtx || !owner || !neigh || !coff || !cf || !patch ||
        (npatch && !kind) || nf == 0 || nc == 0 || device < 0)
        return CFDXHIP_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    auto* fv = new (std::nothrow) cfdxhip_fv();
    if (!fv) return CFDXHIP_ERR_OUT_OF_MEMORY;
    fv->mesh.dev = device;
    const cfdxhip_status s = fv_guarded(fv, [&]() {
        fv->mesh.create(device, np, px, py, pz, nf, foff, fvtx, owner, neigh, nc, coff, cf, npatch, patch, kind);
        return CFDXHIP_OK;
    });
    if (s != CFDXHIP_OK) {
        delete fv;
        return s;
    }
    *out = fv;
    return CFDXHIP_OK;
}

void cfdxhip_fv_destroy(cfdxhip_fv* fv) {
    if (!fv) return;
    (void)hipSetDevice(fv->mesh.dev);
    if (fv->mesh.stream) (void)hipStreamDestroy(fv->mesh.stream);
    fv->mesh.stream = nullptr;
    delete fv;
}

const char* cfdxhip_fv_last_error(const cfdxhip_fv* fv) { return fv ? fv->error.c_str() : kEmpty; }

cfdxhip_status cfdxhip_fv_geometry(cfdxhip_fv* fv, double* fc, double* fs, double* cc, double* vol) {
    if (!fv) return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        fv->mesh.geometry_out(fc, fs, cc, vol);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_gauss_gradient(cfdxhip_fv* fv, const uint8_t* bct, const double* bcv, const double* p,
                                         double* grad) {
    if (!fv || !p || !grad || (fv->mesh.npatch && (!bct || !bcv))) return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        FvMesh& m = fv->mesh;
        const uint32_t np_ = std::max<uint32_t>(m.npatch, 1);
        DevBuf dt(np_), dv(size_t(np_) * 8), dp(size_t(m.nc) * 8), dg(size_t(m.nc) * 24);
        if (m.npatch) {
            hip_check(hipMemcpy(dt.p, bct, m.npatch, hipMemcpyHostToDevice), "copy");
            hip_check(hipMemcpy(dv.p, bcv, size_t(m.npatch) * 8, hipMemcpyHostToDevice), "copy");
        }
        hip_check(hipMemcpy(dp.p, p, size_t(m.nc) * 8, hipMemcpyHostToDevice), "copy");
        m.gauss_gradient_device(dt.as<uint8_t>(), dv.as<double>(), dp.as<double>(), dg.as<double>());
        hip_check(hipStreamSynchronize(m.stream), "sync");
        hip_check(hipMemcpy(grad, dg.p, size_t(m.nc) * 24, hipMemcpyDeviceToHost), "copy");
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_mass_flux(cfdxhip_fv* fv, const uint8_t* vbt, const double* vbv, double rho,
                                    const double* U, double* phi) {
    if (!fv || !U || !phi || (fv->mesh.npatch && (!vbt || !vbv))) return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        FvMesh& m = fv->mesh;
        const uint32_t np_ = std::max<uint32_t>(m.npatch, 1);
        DevBuf dt(np_), dv(size_t(np_) * 24), du(size_t(m.nc) * 24), dphi(size_t(m.nf) * 8);
        if (m.npatch) {
            hip_check(hipMemcpy(dt.p, vbt, m.npatch, hipMemcpyHostToDevice), "copy");
            hip_check(hipMemcpy(dv.p, vbv, size_t(m.npatch) * 24, hipMemcpyHostToDevice), "copy");
        }
        hip_check(hipMemcpy(du.p, U, size_t(m.nc) * 24, hipMemcpyHostToDevice), "copy");
        m.mass_flux_device(dt.as<uint8_t>(), dv.as<double>(), rho, du.as<double>(), dphi.as<double>());
        hip_check(hipStreamSynchronize(m.stream), "sync");
        hip_check(hipMemcpy(phi, dphi.p, size_t(m.nf) * 8, hipMemcpyDeviceToHost), "copy");
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_pressure_pattern(cfdxhip_fv* fv, const uint8_t* pbt, size_t ref, size_t* n_rows,
                                           size_t* nnz, uint32_t* rowp, uint32_t* cols) {
    if (!fv || !n_rows || !nnz || (fv->mesh.npatch && !pbt)) return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        FvMesh& m = fv->mesh;
        const bool fixed = m.npatch ? m.has_fixed_pressure(pbt) : false;
        const bool eliminate = !fixed && m.nc > 1 && ref < m.nc;
        const PressurePlan& pl = m.pressure_plan(eliminate, uint32_t(eliminate ? ref : 0));
        m.prepare_rows(eliminate, uint32_t(eliminate ? ref : 0));
        *n_rows = pl.n;
        *nnz = pl.nnz;
        if (rowp) std::memcpy(rowp, pl.h_rowp.data(), pl.h_rowp.size() * 4);
        if (cols) std::memcpy(cols, pl.h_cols.data(), pl.h_cols.size() * 4);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_pressure_assemble_device(cfdxhip_fv* fv, const uint8_t* pbt, const double* pbv, double rho,
                                                   const double* rAU, const double* phi, const double* p, size_t ref,
                                                   double* values, double* rhs) {
    if (!fv || !rAU || !phi || !p || !values || !rhs || (fv->mesh.npatch && (!pbt || !pbv)) || !std::isfinite(rho))
        return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        std::vector<uint8_t> t(std::max<uint32_t>(fv->mesh.npatch, 1), 0);
        std::vector<double> v(t.size(), 0.0);
        if (fv->mesh.npatch) {
            std::memcpy(t.data(), pbt, fv->mesh.npatch);
            std::memcpy(v.data(), pbv, size_t(fv->mesh.npatch) * 8);
        }
        fv->mesh.pressure_assemble_device(t.data(), v.data(), rho, rAU, phi, p, ref, values, rhs);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_pressure_assemble(cfdxhip_fv* fv, const uint8_t* pbt, const double* pbv, double rho,
                                            const double* rAU, const double* phi, const double* p, size_t ref,
                                            double* values, double* rhs) {
    if (!fv || !rAU || !phi || !p || !values || !rhs) return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        FvMesh& m = fv->mesh;
        size_t n = 0, nnz = 0;
        const cfdxhip_status s = cfdxhip_fv_pressure_pattern(fv, pbt, ref, &n, &nnz, nullptr, nullptr);
        if (s != CFDXHIP_OK) return s;
        DevBuf dr(size_t(m.nc) * 24), dphi(size_t(m.nf) * 8), dp(size_t(m.nc) * 8), dv(nnz * 8), db(n * 8);
        hip_check(hipMemcpy(dr.p, rAU, size_t(m.nc) * 24, hipMemcpyHostToDevice), "copy");
        hip_check(hipMemcpy(dphi.p, phi, size_t(m.nf) * 8, hipMemcpyHostToDevice), "copy");
        hip_check(hipMemcpy(dp.p, p, size_t(m.nc) * 8, hipMemcpyHostToDevice), "copy");
        const cfdxhip_status s2 = cfdxhip_fv_pressure_assemble_device(fv, pbt, pbv, rho, dr.as<double>(),
                                                                      dphi.as<double>(), dp.as<double>(), ref,
                                                                      dv.as<double>(), db.as<double>());
        if (s2 != CFDXHIP_OK) return s2;
        hip_check(hipMemcpy(values, dv.p, nnz * 8, hipMemcpyDeviceToHost), "copy");
        hip_check(hipMemcpy(rhs, db.p, n * 8, hipMemcpyDeviceToHost), "copy");
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_diffusion_assemble(cfdxhip_fv* fv, double gamma, const double* source, const double* fval,
                                             const uint8_t* fneu, size_t* nnz, uint32_t* rowp, uint32_t* cols,
                                             double* values, double* rhs) {
    if (!fv || !nnz || !(gamma > 0.0) || !std::isfinite(gamma)) return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        FvMesh& m = fv->mesh;
        const PressurePlan& pl = m.pressure_plan(false, 0);
        *nnz = pl.nnz;
        if (!rowp && !cols && !values && !rhs) return CFDXHIP_OK;
        if (!source || !fval || !fneu || !rowp || !cols || !values || !rhs) return CFDXHIP_ERR_INVALID_ARGUMENT;
        DevBuf ds(size_t(m.nc) * 8), dfv(size_t(m.nf) * 8), dfn(m.nf), dv(pl.nnz * 8), db(size_t(m.nc) * 8);
        hip_check(hipMemcpy(ds.p, source, size_t(m.nc) * 8, hipMemcpyHostToDevice), "copy");
        hip_check(hipMemcpy(dfv.p, fval, size_t(m.nf) * 8, hipMemcpyHostToDevice), "copy");
        hip_check(hipMemcpy(dfn.p, fneu, m.nf, hipMemcpyHostToDevice), "copy");
        m.diffusion_assemble_device(gamma, ds.as<double>(), dfv.as<double>(), dfn.as<uint8_t>(), dv.as<double>(),
                                    db.as<double>());
        std::memcpy(rowp, pl.h_rowp.data(), pl.h_rowp.size() * 4);
        std::memcpy(cols, pl.h_cols.data(), pl.h_cols.size() * 4);
        hip_check(hipMemcpy(values, dv.p, pl.nnz * 8, hipMemcpyDeviceToHost), "copy");
        hip_check(hipMemcpy(rhs, db.p, size_t(m.nc) * 8, hipMemcpyDeviceToHost), "copy");
        return CFDXHIP_OK;
    });
}

// ------------------------------------------------------ momentum side --

namespace {
void h2d(void* d, const void* h, size_t bytes) { hip_check(hipMemcpy(d, h, bytes, hipMemcpyHostToDevice), "copy"); }
void d2h(void* h, const void* d, size_t bytes) { hip_check(hipMemcpy(h, d, bytes, hipMemcpyDeviceToHost), "copy"); }
}  // namespace

cfdxhip_status cfdxhip_gradient_gauss_device(const double* phi, const double* sx, const double* sy,
                                             const double* sz, const uint32_t* owner, const int64_t* neighbour,
                                             const double* volume, size_t n_faces, size_t n_cells, double* gx,
                                             double* gy, double* gz, void* stream) {
    if (n_cells == 0 || !phi || !volume || !gx || !gy || !gz || (n_faces && (!sx || !sy || !sz || !owner || !neighbour)))
        return CFDXHIP_ERR_INVALID_ARGUMENT;
    try {
        return face_gradient_gauss(phi, sx, sy, sz, owner, neighbour, volume, n_faces, n_cells, gx, gy, gz,
                                   static_cast<hipStream_t>(stream))
                   ? CFDXHIP_OK
                   : CFDXHIP_ERR_INVALID_ARGUMENT;
    } catch (const std::exception&) {
        return CFDXHIP_ERR_DEVICE;
    }
}

cfdxhip_status cfdxhip_divergence_device(const double* phi_face, const uint32_t* owner, const int64_t* neighbour,
                                         size_t n_faces, size_t n_cells, double* div, void* stream) {
    if (n_cells == 0 || !div || (n_faces && (!phi_face || !owner || !neighbour))) return CFDXHIP_ERR_INVALID_ARGUMENT;
    try {
        return face_divergence(phi_face, owner, neighbour, n_faces, n_cells, div, static_cast<hipStream_t>(stream))
                   ? CFDXHIP_OK
                   : CFDXHIP_ERR_INVALID_ARGUMENT;
    } catch (const std::exception&) {
        return CFDXHIP_ERR_DEVICE;
    }
}

cfdxhip_status cfdxhip_fv_wls_gradient(cfdxhip_fv* fv, const uint8_t* bct, const double* bcv, double condition_limit,
                                       const double* field, double* grad, size_t* fallback_cells) {
    if (!fv || !field || !grad || (fv->mesh.npatch && (!bct || !bcv))) return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        FvMesh& m = fv->mesh;
        std::vector<uint8_t> t(std::max<uint32_t>(m.npatch, 1), 0);
        std::vector<double> v(t.size(), 0.0);
        if (m.npatch) {
            std::memcpy(t.data(), bct, m.npatch);
            std::memcpy(v.data(), bcv, size_t(m.npatch) * 8);
        }
        DevBuf df(size_t(m.nc) * 8), dg(size_t(m.nc) * 24), dfb(m.nc);
        h2d(df.p, field, size_t(m.nc) * 8);
        m.wls_gradient_device(t.data(), v.data(), condition_limit, df.as<double>(), dg.as<double>(),
                              dfb.as<uint8_t>());
        d2h(grad, dg.p, size_t(m.nc) * 24);
        if (fallback_cells) {
            std::vector<uint8_t> fb(m.nc);
            d2h(fb.data(), dfb.p, m.nc);
            size_t count = 0;
            for (uint8_t b : fb) count += b;
            *fallback_cells = count;
        }
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_momentum_pattern(cfdxhip_fv* fv, size_t* n_rows, size_t* nnz, uint32_t* rowp,
                                           uint32_t* cols) {
    if (!fv || !n_rows || !nnz) return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        const PressurePlan& pl = fv->mesh.pressure_plan(false, 0);
        fv->mesh.prepare_rows(false, 0);
        *n_rows = pl.n;
        *nnz = pl.nnz;
        if (rowp) std::memcpy(rowp, pl.h_rowp.data(), pl.h_rowp.size() * 4);
        if (cols) std::memcpy(cols, pl.h_cols.data(), pl.h_cols.size() * 4);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_momentum_assemble_device(cfdxhip_fv* fv, const uint8_t* vbt, const double* vbv,
                                                   const double* mu, const double* phi, const double* grad_p,
                                                   const double* body, const double* U, int32_t bounded,
                                                   double alpha_u, double* values, double* rhs, double* diag) {
    if (!fv || !mu || !phi || !grad_p || !U || !values || !rhs || !diag || (fv->mesh.npatch && (!vbt || !vbv)))
        return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        fv->mesh.momentum_assemble_device(vbt, vbv, mu, phi, grad_p, body, U, bounded != 0, alpha_u, values, rhs,
                                          diag);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_momentum_assemble(cfdxhip_fv* fv, const uint8_t* vbt, const double* vbv, const double* mu,
                                            const double* phi, const double* grad_p, const double* body,
                                            const double* U, int32_t bounded, double alpha_u, double* values,
                                            double* rhs, double* diag) {
    if (!fv || !mu || !phi || !grad_p || !U || !values || !rhs || !diag || (fv->mesh.npatch && (!vbt || !vbv)))
        return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        FvMesh& m = fv->mesh;
        const size_t nc = m.nc, nf = m.nf;
        const PressurePlan& pl = m.pressure_plan(false, 0);
        DevBuf dmu(nc * 8), dphi(nf * 8), dgp(nc * 24), dbody(body ? nc * 24 : 8), du(nc * 24), dv(pl.nnz * 8),
            drhs(nc * 24), dd(nc * 8);
        h2d(dmu.p, mu, nc * 8);
        h2d(dphi.p, phi, nf * 8);
        h2d(dgp.p, grad_p, nc * 24);
        if (body) h2d(dbody.p, body, nc * 24);
        h2d(du.p, U, nc * 24);
        m.momentum_assemble_device(vbt, vbv, dmu.as<double>(), dphi.as<double>(), dgp.as<double>(),
                                   body ? dbody.as<double>() : nullptr, du.as<double>(), bounded != 0, alpha_u,
                                   dv.as<double>(), drhs.as<double>(), dd.as<double>());
        d2h(values, dv.p, pl.nnz * 8);
        d2h(rhs, drhs.p, nc * 24);
        d2h(diag, dd.p, nc * 8);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_momentum_hbya_device(cfdxhip_fv* fv, const double* values, const double* rhs,
                                               const double* diag, const double* grad_p, const double* U, double* rAU,
                                               double* HbyA) {
    if (!fv || !values || !rhs || !diag || !grad_p || !U || !rAU || !HbyA) return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        fv->mesh.momentum_hbya_device(values, rhs, diag, grad_p, U, rAU, HbyA);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_momentum_hbya(cfdxhip_fv* fv, const double* values, const double* rhs, const double* diag,
                                        const double* grad_p, const double* U, double* rAU, double* HbyA) {
    if (!fv || !values || !rhs || !diag || !grad_p || !U || !rAU || !HbyA) return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        FvMesh& m = fv->mesh;
        const size_t nc = m.nc;
        const PressurePlan& pl = m.pressure_plan(false, 0);
        DevBuf dv(pl.nnz * 8), drhs(nc * 24), dd(nc * 8), dgp(nc * 24), du(nc * 24), dr(nc * 24), dh(nc * 24);
        h2d(dv.p, values, pl.nnz * 8);
        h2d(drhs.p, rhs, nc * 24);
        h2d(dd.p, diag, nc * 8);
        h2d(dgp.p, grad_p, nc * 24);
        h2d(du.p, U, nc * 24);
        m.momentum_hbya_device(dv.as<double>(), drhs.as<double>(), dd.as<double>(), dgp.as<double>(),
                               du.as<double>(), dr.as<double>(), dh.as<double>());
        d2h(rAU, dr.p, nc * 24);
        d2h(HbyA, dh.p, nc * 24);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_velocity_correct_device(cfdxhip_fv* fv, const double* HbyA, const double* rAU,
                                                  const double* grad_p, double* U) {
    if (!fv || !HbyA || !rAU || !grad_p || !U) return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        fv->mesh.velocity_correct_device(HbyA, rAU, grad_p, U);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_velocity_correct(cfdxhip_fv* fv, const double* HbyA, const double* rAU,
                                           const double* grad_p, double* U) {
    if (!fv || !HbyA || !rAU || !grad_p || !U) return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        FvMesh& m = fv->mesh;
        const size_t nc = m.nc;
        DevBuf dh(nc * 24), dr(nc * 24), dg(nc * 24), du(nc * 24);
        h2d(dh.p, HbyA, nc * 24);
        h2d(dr.p, rAU, nc * 24);
        h2d(dg.p, grad_p, nc * 24);
        m.velocity_correct_device(dh.as<double>(), dr.as<double>(), dg.as<double>(), du.as<double>());
        d2h(U, du.p, nc * 24);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_rhie_chow_flux_device(cfdxhip_fv* fv, const uint8_t* vbt, const double* vbv,
                                                const uint8_t* pbt, const double* pbv, double rho, const double* HbyA,
                                                const double* p, const double* rAU, double* phi) {
    if (!fv || !HbyA || !p || !rAU || !phi || !std::isfinite(rho) ||
        (fv->mesh.npatch && (!vbt || !vbv || !pbt || !pbv)))
        return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        fv->mesh.rhie_chow_flux_device(vbt, vbv, pbt, pbv, rho, HbyA, p, rAU, phi);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_fv_rhie_chow_flux(cfdxhip_fv* fv, const uint8_t* vbt, const double* vbv, const uint8_t* pbt,
                                         const double* pbv, double rho, const double* HbyA, const double* p,
                                         const double* rAU, double* phi) {
    if (!fv || !HbyA || !p || !rAU || !phi || !std::isfinite(rho) ||
        (fv->mesh.npatch && (!vbt || !vbv || !pbt || !pbv)))
        return CFDXHIP_ERR_INVALID_ARGUMENT;
    return fv_guarded(fv, [&]() {
        FvMesh& m = fv->mesh;
        const size_t nc = m.nc, nf = m.nf;
        DevBuf dh(nc * 24), dp(nc * 8), dr(nc * 24), dphi(nf * 8);
        h2d(dh.p, HbyA, nc * 24);
        h2d(dp.p, p, nc * 8);
        h2d(dr.p, rAU, nc * 24);
        m.rhie_chow_flux_device(vbt, vbv, pbt, pbv, rho, dh.as<double>(), dp.as<double>(), dr.as<double>(),
                                dphi.as<double>());
        d2h(phi, dphi.p, nf * 8);
        return CFDXHIP_OK;
    });
}

}  // extern "C"

// ------------------------------------------------------ learned stage --

namespace {
cfdxhip_status mfail(cfdxhip_mpnn* m, cfdxhip_status s, const std::string& msg) {
    if (m) m->error = msg;
    return s;
}
template <class F>
cfdxhip_status mguarded(cfdxhip_mpnn* m, F&& f) {
    try {
        return f();
    } catch (const std::bad_alloc&) {
        return mfail(m, CFDXHIP_ERR_OUT_OF_MEMORY, "host allocation failed");
    } catch (const std::exception& e) {
        const std::string w = e.what();
        return mfail(m, w.rfind("HIP error", 0) == 0 ? CFDXHIP_ERR_DEVICE : CFDXHIP_ERR_INTERNAL, w);
    } catch (...) {
        return mfail(m, CFDXHIP_ERR_INTERNAL, "unknown exception");
    }
}
// The network runs on the finest FP32 operator of a set-up device hierarchy
// on the same device.
cfdxhip_status check_pair(cfdxhip_mpnn* m, const cfdxhip_amg* h) {
    if (!m) return CFDXHIP_ERR_INVALID_ARGUMENT;
    if (!h) return mfail(m, CFDXHIP_ERR_INVALID_ARGUMENT, "no AMG handle");
    if (!h->ready || !h->dev) return mfail(m, CFDXHIP_ERR_NOT_READY, "AMG handle has no device hierarchy");
    if (h->opt.precision != CFDXHIP_PRECISION_FP32)
        return mfail(m, CFDXHIP_ERR_INVALID_ARGUMENT, "the learned stage needs an FP32 (mixed) hierarchy");
    if (h->opt.device != m->device) return mfail(m, CFDXHIP_ERR_INVALID_ARGUMENT, "handles on different devices");
    return CFDXHIP_OK;
}
}  // namespace

extern "C" {

size_t cfdxhip_mpnn_param_count(void) { return size_t(kMpnnParams); }

cfdxhip_status cfdxhip_mpnn_create(int32_t device, cfdxhip_mpnn** out) {
    if (!out || device < 0) return CFDXHIP_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    auto* m = new (std::nothrow) cfdxhip_mpnn();
    if (!m) return CFDXHIP_ERR_OUT_OF_MEMORY;
    m->device = device;
    const cfdxhip_status s = mguarded(m, [&]() {
        m->m = std::make_unique<Mpnn>(device);
        return CFDXHIP_OK;
    });
    if (s != CFDXHIP_OK) {
        delete m;
        return s;
    }
    *out = m;
    return CFDXHIP_OK;
}

void cfdxhip_mpnn_destroy(cfdxhip_mpnn* m) {
    if (!m) return;
    try {
        (void)hipSetDevice(m->device);
        m->m.reset();
    } catch (...) {
    }
    delete m;
}

const char* cfdxhip_mpnn_last_error(const cfdxhip_mpnn* m) { return m ? m->error.c_str() : kEmpty; }

cfdxhip_status cfdxhip_mpnn_set_params(cfdxhip_mpnn* m, const float* params, size_t count) {
    if (!m || !params || count != size_t(kMpnnParams)) return mfail(m, CFDXHIP_ERR_INVALID_ARGUMENT, "bad parameters");
    for (size_t i = 0; i < count; ++i)
        if (!std::isfinite(params[i])) return mfail(m, CFDXHIP_ERR_INVALID_ARGUMENT, "non-finite parameter");
    return mguarded(m, [&]() {
        hip_check(hipSetDevice(m->device), "hipSetDevice");
        m->m->set_params(params);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_mpnn_get_params(cfdxhip_mpnn* m, float* params, size_t count) {
    if (!m || !params || count != size_t(kMpnnParams)) return mfail(m, CFDXHIP_ERR_INVALID_ARGUMENT, "bad buffer");
    return mguarded(m, [&]() {
        hip_check(hipSetDevice(m->device), "hipSetDevice");
        m->m->get_params(params);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_mpnn_forward(cfdxhip_mpnn* m, cfdxhip_amg* h, const double* r, double* e) {
    const cfdxhip_status c = check_pair(m, h);
    if (c != CFDXHIP_OK) return c;
    if (!r || !e) return mfail(m, CFDXHIP_ERR_INVALID_ARGUMENT, "null vector");
    return mguarded(m, [&]() {
        hip_check(hipSetDevice(m->device), "hipSetDevice");
        mpnn_forward_host(*m->m, *h->dev, r, e);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_mpnn_vjp(cfdxhip_mpnn* m, cfdxhip_amg* h, const double* r, const double* ge, float* grad) {
    const cfdxhip_status c = check_pair(m, h);
    if (c != CFDXHIP_OK) return c;
    if (!r || !ge || !grad) return mfail(m, CFDXHIP_ERR_INVALID_ARGUMENT, "null vector");
    return mguarded(m, [&]() {
        hip_check(hipSetDevice(m->device), "hipSetDevice");
        mpnn_vjp_host(*m->m, *h->dev, r, ge, grad);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_mpnn_adam_step(cfdxhip_mpnn* m, const float* grad, float lr) {
    if (!m || !grad || !(lr > 0.0f)) return mfail(m, CFDXHIP_ERR_INVALID_ARGUMENT, "bad Adam arguments");
    return mguarded(m, [&]() {
        hip_check(hipSetDevice(m->device), "hipSetDevice");
        mpnn_adam_host(*m->m, grad, lr);
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_mpnn_collect_pairs(cfdxhip_mpnn* m, cfdxhip_amg* h, const double* b,
                                          const uint64_t* iterations, uint32_t count, double tol,
                                          uint32_t* collected, cfdxhip_result* solve) {
    const cfdxhip_status c = check_pair(m, h);
    if (c != CFDXHIP_OK) return c;
    if (!b || !iterations || count == 0 || !(tol > 0.0) || !h->dev)
        return mfail(m, CFDXHIP_ERR_INVALID_ARGUMENT, "bad collection arguments");
    return mguarded(m, [&]() {
        hip_check(hipSetDevice(m->device), "hipSetDevice");
        std::vector<uint64_t> its(iterations, iterations + count);
        uint32_t got = 0;
        SolveStats st;
        std::string err;
        const bool ok = mpnn_collect(*m->m, *h->dev, b, its, tol, got, st, err);
        if (collected) *collected = got;
        fill_result(st, solve);
        if (!ok) return mfail(m, CFDXHIP_ERR_NUMERIC, err);
        m->error.clear();
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_mpnn_train(cfdxhip_mpnn* m, cfdxhip_amg* h, uint32_t steps, float lr, double* losses) {
    const cfdxhip_status c = check_pair(m, h);
    if (c != CFDXHIP_OK) return c;
    if (steps == 0 || !(lr > 0.0f)) return mfail(m, CFDXHIP_ERR_INVALID_ARGUMENT, "bad training arguments");
    return mguarded(m, [&]() {
        hip_check(hipSetDevice(m->device), "hipSetDevice");
        std::string err;
        if (!mpnn_train(*m->m, *h->dev, steps, lr, losses, err)) return mfail(m, CFDXHIP_ERR_NOT_READY, err);
        m->error.clear();
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_mpnn_set_fallback(cfdxhip_mpnn* m, double min_reduction, uint32_t window) {
    if (!m || !(min_reduction <= 1.0) || window == 0 || window > 64)
        return mfail(m, CFDXHIP_ERR_INVALID_ARGUMENT, "bad fallback arguments");
    m->m->fallback_min_reduction = min_reduction;
    m->m->fallback_window = window;
    return CFDXHIP_OK;
}

static cfdxhip_status learned_common(cfdxhip_amg* h, cfdxhip_mpnn* m, const double* b, double* x, bool device,
                                     int restart, size_t max_iter, double tol, cfdxhip_result* result) {
    const cfdxhip_status c = check_pair(m, h);
    if (c != CFDXHIP_OK) {
        if (h && m) h->error = m->error;
        return c;
    }
    if (!b || !x || max_iter == 0 || restart <= 0 || !(tol > 0.0) || !std::isfinite(tol))
        return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, "invalid solve arguments");
    return guarded(h, [&]() {
        hip_check(hipSetDevice(h->opt.device), "hipSetDevice");
        const uint32_t n = h->dev->n();
        SolveStats st;
        std::string err;
        LearnedControl lc;
        lc.stage = m->m.get();
        lc.min_reduction = m->m->fallback_min_reduction;
        lc.window = m->m->fallback_window;
        bool ok;
        if (device) {
            ok = h->dev->fgmres(b, x, restart, max_iter, tol, true, st, err, &lc);
        } else {
            DevBuf db(size_t(n) * 8), dx(size_t(n) * 8);
            hip_check(hipMemcpy(db.p, b, size_t(n) * 8, hipMemcpyHostToDevice), "copy b");
            hip_check(hipMemcpy(dx.p, x, size_t(n) * 8, hipMemcpyHostToDevice), "copy x");
            ok = h->dev->fgmres(db.as<double>(), dx.as<double>(), restart, max_iter, tol, true, st, err, &lc);
            hip_check(hipMemcpy(x, dx.p, size_t(n) * 8, hipMemcpyDeviceToHost), "copy x");
        }
        if (!ok) return fail(h, CFDXHIP_ERR_INVALID_ARGUMENT, err);
        fill_result(st, result);
        if (result) {
            result->learned_stage_applications = lc.applications;
            result->learned_stage_fallbacks = lc.fallbacks;
        }
        h->error.clear();
        return CFDXHIP_OK;
    });
}

cfdxhip_status cfdxhip_amg_solve_fgmres_learned(cfdxhip_amg* h, cfdxhip_mpnn* m, const double* b, double* x,
                                                int restart, size_t max_iter, double tol, cfdxhip_result* result) {
    return learned_common(h, m, b, x, false, restart, max_iter, tol, result);
}

cfdxhip_status cfdxhip_amg_solve_fgmres_learned_device(cfdxhip_amg* h, cfdxhip_mpnn* m, const double* b,
                                                       double* x, int restart, size_t max_iter, double tol,
                                                       cfdxhip_result* result) {
    return learned_common(h, m, b, x, true, restart, max_iter, tol, result);
}

}  // extern "C"
