// Device-resident AMG hierarchy and Krylov solvers (HIP).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <functional>
#include <string>
#include <vector>

#include "amg_setup.h"

namespace cfdxhip {

struct DevCsr {
    uint32_t n = 0, ncols = 0;
    uint64_t nnz = 0;
    uint32_t* rowp = nullptr;
    uint32_t* cols = nullptr;
    uint2* blocks = nullptr;  // CSR-stream row blocks of FP64 launches (nblocks + 1 boundaries: row, first entry)
    uint32_t nblocks = 0;
    uint2* blocks32 = nullptr;  // the same for FP32 launches (smaller blocks)
    uint32_t nblocks32 = 0;
    double* v64 = nullptr;
    float* v32 = nullptr;
    // SELL-64 copy used by the SpMV when the slices pad little (nslices > 0).
    uint32_t nslices = 0;
    uint64_t sell_entries = 0;  // stored slots, padding included
    uint32_t* soff = nullptr;   // nslices + 1 slot offsets
    uint32_t* scols = nullptr;  // FP64 copy: CSR entry order within a row
    double* s64 = nullptr;
    uint32_t* scols32 = nullptr;  // FP32 copy: slots sorted by column
    float* s32 = nullptr;
    // Half smoothing copy (finest level, FP32 V-cycle): FP16 values of D^-1 A,
    // 2 B per SELL slot (slot pairs of a row per word; a slice's odd last slot
    // two rows per word), the slice's words from soff[slice] / 2.
    uint32_t* hvals = nullptr;
    uint64_t half_words = 0;
    // Compact columns of the half copy: per-slot-row bases, int16 offsets
    // laid out like hvals, and the slices that keep 4 B columns.
    uint32_t* hbase = nullptr;
    uint32_t* hcol16 = nullptr;
    uint8_t* hwide = nullptr;
    uint64_t half_bytes = 0;  // bytes one half-copy step streams for the matrix
};

struct DevLevel {
    uint32_t n = 0;
    DevCsr A, P, R;  // P: n x n_coarse, R = P^T: n_coarse x n
    double* inv64 = nullptr;
    float* inv32 = nullptr;
    double* x64[2] = {nullptr, nullptr};
    double* b64 = nullptr;
    double* r64 = nullptr;
    float* x32[2] = {nullptr, nullptr};
    float* b32 = nullptr;
    float* r32 = nullptr;
    double* d64 = nullptr;  // Chebyshev direction (allocated when selected)
    float* d32 = nullptr;
    float* bt32 = nullptr;  // D^-1 b of the half-copy Chebyshev steps
    // Host mirror of the solve-ordering permutation (new index of old row).
    std::vector<uint32_t> new_of_old;
};

// Levels of the FP64 V-cycle's single-launch coarse end (layout:
// coarse_tail.hpp).
constexpr int kTailWaves = 8;

struct TailMat {
    uint32_t n;                  // rows
    uint32_t ngroups;            // groups of longer rows
    uint32_t first[kTailWaves];  // first batch of each wavefront
    uint32_t count[kTailWaves];
    const uint32_t* ctl;         // [batch][lane]
    const uint4* cols;           // [batch][lane]: eight 16-bit columns
    const double* vals;          // [batch][pair of slots][lane]
    const uint4* groups;         // first entry, entries, first row in lrows, rows
    const uint4* lrows;          // row, first and end product in its group
    const uint16_t* lcols;
    const double* lvals;
};

// x and b: offsets of the level's vectors in LDS (n + 1 cells each, the last
// one of x holds 1.0). R and P lead to the next level; the last has none.
struct TailLevel {
    TailMat A, R, P;
    const double* inv;
    uint32_t x, b;
    uint32_t degree;       // Chebyshev degree
    double c1[16], c2[16];  // its coefficients
};

struct DevCoarseLU {
    bool ok = false;
    uint32_t n = 0;
    uint32_t* piv = nullptr;
    double* factor = nullptr;
    double* upper = nullptr;
};

struct SolveStats {
    uint32_t status = 3;
    uint64_t iterations = 0;
    double residual = 0.0, residual_relative = 0.0;
    uint64_t replacements = 0;
    double max_gap = 0.0, min_true = 0.0, max_true = 0.0;
    uint64_t first_replacement = 0, last_replacement = 0;
    uint64_t pc_applications = 0;
    uint64_t reorthogonalisations = 0;  // FGMRES second Gram-Schmidt passes
    double seconds = 0.0;
};

// Fills the SELL-64 values of a matrix from its CSR values (no-op without a
// SELL copy); first: the padding slots too.
void sell_values(DevCsr& D, hipStream_t s, bool first);

// Work memory of the allocation-free PCG: a fixed device array of
// kNoAllocScratchBytes per GPU (file-scope in device_amg.hip), laid out in
// kNoAllocAlign-byte aligned parts. noalloc_scratch returns its address on
// `device`, which must be current; the address is looked up once per device.
constexpr uint64_t kNoAllocScratchBytes = uint64_t(128) << 20;
constexpr uint64_t kNoAllocAlign = 256;
bool noalloc_scratch(int device, unsigned char*& ptr, std::string& err);

class DeviceAmg;

// One level as the refresh's batched kernels see it: a launch covers all
// levels, each with a range of workgroups (first_* of the next entry ends it).
struct RefreshView {
    uint32_t n;
    uint32_t first_wg;     // 256-row workgroups (elementwise kernels, 256-row tiles)
    uint32_t first_block;  // CSR-stream row blocks
    uint32_t row0;         // offset of the level's rows in the work vectors
    // solve ordering
    const uint2* blocks;
    const uint32_t* rowp;
    const uint32_t* cols;
    const double* vals;
    const double* inv;
    const uint32_t* perm;  // new_of_old
    // reference ordering, current and staged values
    const uint32_t* arow;
    const uint32_t* acol;
    const double* aval[2];
    const double* rinv[2];
};

// Lanczos scalars of a level.
constexpr uint32_t kLanczosMax = 32;
struct LanczosState {
    double norm, a, bprev, b;
    uint32_t count, stop;
    double alpha[kLanczosMax], beta[kLanczosMax];
};

// A preconditioner stage run ahead of (and around) the FP32 V-cycle inside
// mixed FGMRES: z = stage(r) on FP32 vectors in the solve ordering.
class PreconditionerStage {
public:
    virtual ~PreconditionerStage() = default;
    // network_reduction (when not null) receives 1 - |r - A e| / |r| for the
    // stage's own error estimate e, before its V-cycle.
    virtual bool apply(DeviceAmg& amg, const float* r, float* z, std::string& err,
                       double* network_reduction = nullptr) = 0;
};

// Learned-stage control of one mixed FGMRES solve. The stage is dropped for
// the rest of the solve (plain V-cycle, counted as a fallback) once a residual
// reduction drops below min_reduction: the network's own, 1 - |r - A N(r)| /
// |r|, at any application (the network judged by the residual its estimate
// leaves), or the FGMRES one per iteration over the last `window` iterations,
// 1 - (|g_k| / |g_{k-window}|)^(1/window) from the Givens estimates.
struct LearnedControl {
    PreconditionerStage* stage = nullptr;
    double min_reduction = 0.5;
    uint32_t window = 5;
    uint64_t applications = 0;
    uint64_t fallbacks = 0;
};

// Finest-level operator as the learned stage sees it (solve ordering, FP32).
struct Level0View {
    uint32_t n = 0;
    const uint32_t* rowp = nullptr;
    const uint32_t* cols = nullptr;
    const float* vals = nullptr;
    const float* inv_diag = nullptr;
};

class DeviceAmg {
public:
    // Reference-ordered state of the device numeric refresh, per level: A's
    // pattern and values (current and staged), the staged inverse diagonal,
    // the maps to the solve-ordered copies, and for each transfer P and the
    // Galerkin plan (AP and P^T AP patterns, transpose plan, kept entries).
    struct RefreshLevel {
        uint32_t n = 0;
        uint64_t nnz = 0;
        uint32_t* arow = nullptr;
        uint32_t* acol = nullptr;
        double* aval[2] = {nullptr, nullptr};  // values (current, staged)
        double* inv[2] = {nullptr, nullptr};  // inverse diagonal (current, staged)
        uint32_t* src = nullptr;   // solve-ordered CSR position -> reference entry
        uint32_t* perm = nullptr;  // new_of_old
        uint32_t nc = 0;
        uint64_t pnnz = 0, apnnz = 0, cnnz = 0;
        uint32_t* prow = nullptr;
        uint32_t* pcol = nullptr;
        double* pval = nullptr;
        uint32_t* ap_off = nullptr;
        uint32_t* ap_col = nullptr;
        uint32_t* ap_row = nullptr;  // row of each AP entry
        double* apv = nullptr;
        uint32_t* c_off = nullptr;
        uint32_t* c_col = nullptr;
        // Coarse rows the Galerkin product gives a wavefront or a workgroup
        // (row, tile of columns) each; the others share a wavefront.
        uint32_t* c_mid = nullptr;
        uint2* c_heavy = nullptr;
        uint32_t c_nmid = 0, c_nheavy = 0;
        double* cv = nullptr;
        uint32_t* t_off = nullptr;
        uint32_t* t_row = nullptr;
        uint32_t* t_pos = nullptr;
        uint8_t* keep_mask = nullptr;  // per unpruned coarse entry: kept at setup
        uint32_t* keep = nullptr;      // kept coarse entry -> unpruned index
    };
    DeviceAmg() = default;
    ~DeviceAmg();
    DeviceAmg(const DeviceAmg&) = delete;
    DeviceAmg& operator=(const DeviceAmg&) = delete;

    // Uploads a host hierarchy (reference ordering) into the solve ordering.
    // adopt: the device-side construction's reference-ordered levels (from
    // build_sa_device), taken over as the refresh state instead of uploading
    // the host mirror's. The damping and eigenvalue bounds may be left to
    // finish_setup.
    bool build(const HostHierarchy& h, const AmgConfig& cfg, bool reorder, bool want64, bool want32,
               hipStream_t stream, std::string& err, std::vector<RefreshLevel>* adopt = nullptr);
    // Smoothed-aggregation hierarchy built on the device from a device CSR
    // (reference ordering): strength graph, its transpose and symmetrised
    // union, P smoothing, Galerkin symbolic and numeric products and the
    // 1e-30 pruning are HIP kernels; only the greedy aggregation (a
    // sequential seed order) runs on the host. Results are bit-identical to
    // build_hierarchy. `host` receives the mirror the ordering, upload and
    // introspection need (matrices, inverse diagonals, aggregates, P), and
    // `levels` the device arrays for build(adopt).
    static bool build_sa_device(const uint32_t* d_rowp, const uint32_t* d_cols, const double* d_vals, uint32_t n,
                                const AmgConfig& cfg, hipStream_t stream, HostHierarchy& host,
                                std::vector<RefreshLevel>& levels, std::string& err);
    static void free_refresh_level(RefreshLevel& R);
    // Damping certificate (normalised Gershgorin bound over all levels) and,
    // for a Chebyshev smoother, the Lanczos eigenvalue estimates of the set-up
    // hierarchy, computed on the device as build_hierarchy computes them.
    bool finish_setup(const AmgConfig& cfg, double& omega, std::vector<double>& lambda, std::string& err);
    // Numeric refresh on the device (update_values): new finest-level values
    // d_vals (device, caller order = the setup matrix's entry order). Galerkin
    // products, inverse diagonals, damping certificate and (for Chebyshev)
    // eigenvalue estimates are recomputed on the device exactly as the host
    // refresh computes them. Transactional: on failure nothing changes.
    // pattern_changed: the 1e-30 pruning would keep a different set of
    // coarse entries. omega / lambda receive the committed values.
    bool refresh_device(const double* d_vals, const AmgConfig& cfg, double& omega, std::vector<double>& lambda,
                        std::string& err, bool& pattern_changed);
    // Current values of a level's matrix in the reference order (host copy).
    bool level_values(size_t level, std::vector<double>& vals) const;

    uint32_t n() const { return lv_.empty() ? 0 : lv_[0].n; }
    // One V-cycle z = M^{-1} r. r, z: device vectors in the SOLVE ordering of
    // level 0, precision T. Returns false if the coarse solve is unusable.
    bool vcycle64(const double* r, double* z);
    bool vcycle32(const float* r, float* z);
    // z = M^{-1} r on caller-ordered FP64 device vectors (the handle's
    // precision: FP32 V-cycles convert on the way in and out). Fails on a
    // non-finite r (before any work) or z.
    bool apply_caller(const double* r, double* z, bool fp32, std::string& err);

    // Bounded action for nonsymmetric Krylov use (hypre_amg.cpp:293-326):
    // with max_image_ratio > 0, a preconditioner result z whose image A z is
    // not finite or exceeds max_image_ratio |r| is replaced by the damped
    // Jacobi action 0.7 D^-1 r, and the application fails if that does not
    // pass either. 0 disables.
    double max_image_ratio = 0.0;
    uint64_t bounded_fallbacks = 0;
    // r, z: solve-ordered FP64 vectors of level 0.
    bool bounded_action(const double* r, double* z, std::string& err);

    // Device memory the PCG works in: seven FP64 n-vectors (b, x, r, true
    // residual, z, p, Ap), three partial-sum arrays of `stride` doubles and
    // the device scalar slots.
    struct PcgWork {
        double* vec[7] = {};
        double* partials = nullptr;
        uint64_t stride = 0;
        double* scal = nullptr;
    };
    // Krylov solvers on caller-ordered device vectors (FP64).
    // ns_modes (may be null): ns_count orthonormal null-space modes, device
    // vectors in the solve ordering, projected out at the reference's points
    // (cg_solver.h:93,149,203,262,295-297,517,558).
    bool pcg(const double* b, double* x, uint64_t max_iter, double tol, SolveStats& st, std::string& err,
             const double* ns_modes = nullptr, uint32_t ns_count = 0);
    // PCG in caller-provided work memory: allocates no device memory.
    bool pcg_in(const PcgWork& w, const double* b, double* x, uint64_t max_iter, double tol, SolveStats& st,
                std::string& err, const double* ns_modes = nullptr, uint32_t ns_count = 0);
    // v -= (v . m) m for each of `count` modes (solve ordering, level 0).
    void project_out(const double* modes, uint32_t count, double* v);
    // Solve-ordered copy of caller-ordered device vector(s).
    void to_solve_order(const double* caller, double* solve, uint32_t count);
    // Bytes of a PcgWork laid out from one base address (each part aligned
    // to `align` bytes), and that layout.
    uint64_t pcg_work_bytes(uint64_t align) const;
    PcgWork pcg_work_at(unsigned char* base, uint64_t align) const;
    bool fgmres(const double* b, double* x, int restart, uint64_t max_iter, double tol, bool mixed,
                SolveStats& st, std::string& err, LearnedControl* learned = nullptr);
    // Runs FP64 PCG from x = 0 to tol on b (caller order, device) and returns
    // (residual, error) pairs at the requested iterations: r_k = b - A x_k,
    // e_k = x_final - x_k, FP32, solve ordering, pair k at r_out + k n.
    bool collect_pairs(const double* b, const std::vector<uint64_t>& iterations, double tol, float* r_out,
                       float* e_out, uint32_t& got, SolveStats& st, std::string& err);
    Level0View level0() const;
    // y = A x on the finest level, FP32, solve ordering.
    void spmv32(const float* x, float* y);
    // r = b - A x on the finest level, FP32, solve ordering.
    void residual32(const float* b, const float* x, float* r);
    const uint32_t* device_perm0() const { return d_perm0_; }
    // Seconds per launch of a level's SpMV (kind 0: y = A x) or fused Jacobi
    // sweep (kind 1) on the level's own buffers (x = b = 1), HIP events.
    size_t num_levels() const { return lv_.size(); }
    const DevCsr& level_matrix(size_t l) const { return lv_[l].A; }
    // First level of the FP64 V-cycle's single-launch coarse end (the number
    // of levels: none).
    uint32_t coarse_end_level() const { return tail_.first; }
    bool level_kernel_seconds(uint32_t level, uint32_t precision, uint32_t kind, uint32_t repeat, double& sec,
                              std::string& err);
    // Seconds per launch of the Gram-Schmidt passes of Arnoldi step j.
    bool gram_schmidt_seconds(uint32_t j, uint32_t repeat, double& dot_s, double& update_s, std::string& err);
    // y = A x on caller-ordered device vectors; returns seconds per launch.
    bool spmv_caller(uint32_t precision, const void* x, void* y, uint32_t repeat, double& sec, std::string& err);

    // Changes the Chebyshev degree / interval ratio of a built hierarchy
    // (coefficients only; the eigenvalue estimates are kept).
    void set_chebyshev_params(const HostHierarchy& h, uint32_t degree, uint32_t degree_coarse, double ratio) {
        cheb_degree_ = degree;
        cheb_degree_coarse_ = degree_coarse;
        cheb_ratio_ = ratio;
        set_chebyshev(h);
    }

    hipStream_t stream() const { return stream_; }

private:
    template <class T>
    bool vcycle_t(uint32_t l, const T* b, T*& x);
    // Mean removal of the constant null space on n entries (device-side
    // sum, fixed tree).
    template <class T>
    void remove_mean(T* v, uint32_t n);
    template <class T>
    void spmv_jacobi_sweeps(DevLevel& L, const T* b, T*& x, uint32_t sweeps, bool from_zero);
    template <class T>
    void chebyshev_sweeps(uint32_t l, const T* b, T*& x, bool from_zero);
    void chebyshev_sweeps_half(const float* b, float*& x, bool from_zero);
    void build_half_copy(DevLevel& L);
    template <class T>
    void smooth(uint32_t l, const T* b, T*& x, uint32_t sweeps, bool from_zero);
    void set_chebyshev(const HostHierarchy& h) { set_chebyshev_lambda(h.lambda_max); }
    void set_chebyshev_lambda(const std::vector<double>& lambda_max);
    bool build_refresh(const HostHierarchy& h, std::string& err, std::vector<RefreshLevel>* adopt = nullptr);
    // Normalised Gershgorin bound over all levels of the refresh state's
    // values `slot` (the damping certificate's input).
    // Launches it for all levels (results in rf_host_ after read_refresh).
    void launch_gershgorin(uint32_t slot);
    void read_refresh(bool coarsest, uint32_t slot);
    bool gershgorin_bound(bool& certified, double& mb) const;
    // Lanczos eigenvalue estimates of every level's committed matrix.
    std::vector<double> lanczos_bounds(const AmgConfig& cfg);
    void release_refresh();
    void release();
    // stride 0: the hierarchy's own partial-sum stride; src null: scal_.
    void reduce(const double* partials, uint32_t n, uint32_t count, double* out, uint64_t stride = 0,
                const double* base = nullptr);
    bool fetch_scalars(uint32_t count, uint32_t first = 0);

    // The FP64 V-cycle's single-launch coarse end (coarse_tail.hpp): its
    // first level (the number of levels: none), the level descriptors on the
    // host and the device, the LDS layout, and what refills the packed
    // matrices from the levels' CSR values.
    struct Tail {
        struct Refill {
            uint32_t level, n;
            const uint32_t* src;
            double* dst;
        };
        uint32_t first = 0, cells = 0, stage = 0, lds_bytes = 0;
        std::vector<TailLevel> host;
        TailLevel* dev = nullptr;
        std::vector<Refill> refill;
        unsigned char* mem = nullptr;  // its device arrays
    };
    // Host patterns of a level's A, R and P in the solve ordering.
    struct TailPatterns {
        struct Pattern {
            std::vector<uint32_t> rowp, cols;
        };
        Pattern m[3];
    };
    void build_tail(const std::vector<TailPatterns>& small);
    void upload_tail();  // after new Chebyshev coefficients
    void refill_tail();  // after new values of the levels' CSR copies
    Tail tail_;

    std::vector<DevLevel> lv_;
    std::vector<RefreshLevel> rf_;
    uint32_t rf_cur_ = 0;        // which aval holds the committed values
    int* rf_flags_ = nullptr;    // refresh error flags, per level
    double* rf_work_ = nullptr;  // Lanczos vectors and tile sums, Gershgorin rows
    RefreshView* rf_view_ = nullptr;  // the levels as the batched kernels see them
    std::vector<RefreshView> rf_view_host_;
    LanczosState* rf_lz_ = nullptr;
    double* rf_ub_ = nullptr;        // Gershgorin bound per level
    uint2* rf_long_ = nullptr;     // (level, row) of the levels' long rows, longest first
    uint32_t rf_nlong_ = 0;
    std::vector<int> rf_host_flags_;
    std::vector<double> rf_host_ub_;
    HCsr rf_coarsest_;               // pattern and fetched values of the coarsest level
    DevCoarseLU lu_;
    double omega_ = 0.7;
    uint32_t pre_ = 6, post_ = 6;
    uint32_t smoother64_ = SMOOTHER_JACOBI, smoother32_ = SMOOTHER_JACOBI;
    uint32_t cheb_degree_ = 3;
    uint32_t cheb_degree_coarse_ = 0;  // levels below the finest; 0: cheb_degree_
    double cheb_ratio_ = 30.0;
    std::vector<std::vector<double>> cheb_c1_, cheb_c2_;  // per level
    std::vector<uint32_t> cheb_deg_;                       // per level
    bool has64_ = false, has32_ = false;
    const float* half_bt_for_ = nullptr;  // the b whose D^-1 b the finest level's bt32 holds
    // Called by pcg with (iteration, x in the solve ordering) after every
    // update of x, with iteration 0 for the initial guess and UINT64_MAX for
    // the returned iterate.
    std::function<void(uint64_t, const double*)> on_iterate_;
    hipStream_t stream_ = nullptr;
    uint32_t* d_perm0_ = nullptr;  // new_of_old of level 0 on device
    // Krylov work (caller size n0), FP64.
    double* partials_ = nullptr;    // 8 partial arrays
    double* aux_part_ = nullptr;    // partial sums of the mean and null-space projections
    bool cns_ = false;              // constant null space
    double* cns_r64_ = nullptr;     // level-0 right-hand side with its mean removed
    float* cns_r32_ = nullptr;
    uint64_t partial_stride_ = 0;
    double* scal_ = nullptr;        // device scalars
    double* h_scal_ = nullptr;      // pinned host mirror
    unsigned long long *h_done_ = nullptr, *done_ = nullptr, ticket_ = 0;  // tickets of awaited kernels (pinned)
    void await(int count);
    unsigned long long apply_calls_ = 0;
    bool apply_bounded(const double* r, double* z, const int* seen, std::string& err);
    double* scal_host_ = nullptr;  // h_scal_ as the device addresses it
    std::vector<double*> work_;     // generic FP64 n-vectors
    std::vector<float*> work32_;
    std::vector<double*> basis_;    // FGMRES V (m+1), Z (m) and w, padded
    void ensure_basis(uint32_t n, uint32_t mcap, size_t ld);
    uint32_t basis_m_ = 0;
};

}  // namespace cfdxhip
