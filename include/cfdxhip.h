/*
 * cfdxhip — MI355X-native pressure-correction solve for CFDX (C ABI).
 *
 * Drop-in boundary for the reference's pressure path:
 *   - the linear-solver interface (Preconditioner / NativeAMGPreconditioner /
 *     solve_cg_prepared / solve_fgmres), core/linalg/preconditioner.h:18-28,
 *     core/linalg/hypre_amg.h:26-101, core/linalg/cg_solver.h:653-667,
 *     core/linalg/gmres_solver.h:678-692;
 *   - the face-loop pressure assembly of the SIMPLE corrector,
 *     physics/steady_incompressible_solver.h:8048-8181 and :8599-8652, and the
 *     canonical Poisson assembly core/solvers/scalar_diffusion.h:39-163.
 *
 * Conventions
 *   - Every entry point returns a cfdxhip_status and never throws; the reason
 *     of the latest failure on a handle is available from *_last_error
 *     (mirrors NativeAMGPreconditioner::last_error, hypre_amg.h:89-96).
 *   - Pointers are host pointers unless the name ends in _device, in which
 *     case they are device pointers on the handle's device and the call is
 *     ordered on the handle's stream.
 *   - CSR: uint32 row offsets [n+1], uint32 columns strictly ascending per
 *     row, double values (core/linalg/sparse_matrix.h:27-31).
 *   - One handle per host thread: handles are not reentrant.
 */
#ifndef CFDXHIP_H
#define CFDXHIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef enum cfdxhip_status {
    CFDXHIP_OK = 0,
    CFDXHIP_ERR_INVALID_ARGUMENT = 1,
    CFDXHIP_ERR_NOT_READY = 2,
    CFDXHIP_ERR_PATTERN_CHANGED = 3,
    CFDXHIP_ERR_SETUP_FAILED = 4,
    CFDXHIP_ERR_NUMERIC = 5,
    CFDXHIP_ERR_DEVICE = 6,
    CFDXHIP_ERR_OUT_OF_MEMORY = 7,
    CFDXHIP_ERR_INTERNAL = 8
} cfdxhip_status;

/* SolverStatus, core/linalg/solver_status.h:18-23. */
enum {
    CFDXHIP_SOLVER_CONVERGED = 0,
    CFDXHIP_SOLVER_MAX_ITER_REACHED = 1,
    CFDXHIP_SOLVER_DIVERGED = 2,
    CFDXHIP_SOLVER_NOT_APPLICABLE = 3
};

/* SolverResult (core/linalg/solver_status.h:45-72) plus solve metrics. */
typedef struct cfdxhip_result {
    uint32_t status;
    uint32_t reserved0;
    uint64_t iterations;
    double residual;          /* absolute FP64 true residual ||b - A x||_2 */
    double residual_relative; /* residual / ||b||_2 */
    uint64_t residual_replacements;
    double max_true_recursive_gap;
    double min_true_residual;
    double max_true_residual;
    uint64_t first_residual_replacement;
    uint64_t last_residual_replacement;
    /* metrics of this build */
    double solve_seconds;          /* wall time of the solve call */
    uint64_t preconditioner_applications;
    uint64_t learned_stage_applications;
    uint64_t learned_stage_fallbacks;
} cfdxhip_result;

/* NativeAMGMethod (hypre_amg.h:19-22). */
enum { CFDXHIP_AMG_BOOMER_STYLE = 0, CFDXHIP_AMG_SMOOTHED_AGGREGATION = 1 };
/* AMGMemoryPolicy (hypre_amg.h:13-17). */
enum { CFDXHIP_POLICY_LOW = 0, CFDXHIP_POLICY_BALANCED = 1, CFDXHIP_POLICY_FAST = 2 };
/* Precision of the V-cycle (hierarchy values, smoother, transfers). */
enum { CFDXHIP_PRECISION_FP64 = 0, CFDXHIP_PRECISION_FP32 = 1 };
/* V-cycle smoother. JACOBI is the reference's damped Jacobi
 * (amg_preconditioner.h:2369-2409: pre/post sweeps, certified omega).
 * CHEBYSHEV has no counterpart inside the reference's V-cycle: the textbook
 * Jacobi-preconditioned three-term Chebyshev recurrence of chebyshev_degree
 * steps per smoothing on [1.1 lambda / ratio, 1.1 lambda], lambda being a
 * 20-step Lanczos estimate of lambda_max(D^-1 A) per level. (The
 * reference's standalone ChebyshevSmoother, chebyshev_smoother.h:11-118, uses
 * a different update and is not on its V-cycle path.) */
enum { CFDXHIP_SMOOTHER_JACOBI = 0, CFDXHIP_SMOOTHER_CHEBYSHEV = 1 };

typedef struct cfdxhip_amg_options {
    uint32_t method;                       /* CFDXHIP_AMG_* (default smoothed aggregation) */
    uint32_t policy;                       /* CFDXHIP_POLICY_* (default balanced) */
    uint32_t require_smoother_certificate; /* 1: fail setup without the omega certificate */
    uint32_t precision;                    /* V-cycle precision for apply/FGMRES */
    uint32_t reorder;                      /* 1: locality ordering of the hierarchy (default) */
    uint32_t host_threads;                 /* 0: all host cores for setup */
    int32_t device;                        /* HIP device ordinal; < 0: host-only handle
                                              (setup + introspection, no device work) */
    double strength_threshold;             /* theta, default 0.25 (hypre_amg.cpp:203) */
    double prolongator_filter;             /* SA P filter, default 0 (amg_preconditioner.h:2020-2033) */
    uint32_t filter_keeps_aggregate;       /* 1: the filter never drops a point's own-aggregate
                                              entry, a point whose smoothed own-aggregate weight
                                              is below filter x its largest keeps its tentative
                                              row, and coarsening stops before a level whose
                                              Galerkin product has a zero diagonal. No reference
                                              counterpart: the reference rejects a hierarchy
                                              whose filtered P loses a whole column (zero coarse
                                              diagonal). Default 0. */
    uint32_t smoother;                     /* CFDXHIP_SMOOTHER_* of FP64 V-cycles (default JACOBI) */
    uint32_t smoother_fp32;                /* CFDXHIP_SMOOTHER_* of FP32 V-cycles (default JACOBI) */
    uint32_t chebyshev_degree;             /* Chebyshev steps per pre/post smoothing (default 3) */
    uint32_t chebyshev_degree_coarse;      /* steps on levels below the finest; 0: chebyshev_degree
                                              (default 0) */
    double chebyshev_ratio;                /* upper / lower end of the damped interval (default 30) */
    uint32_t constant_null_space;          /* 1: the constant vector spans A's null space
                                              (hypre_amg.h:35; amg_preconditioner.h:49,84,
                                              1191-1203,2369-2443,2590-2666): setup and
                                              update_values require every row sum within
                                              256 eps max(1, largest row 1-norm) of zero; each
                                              application removes the mean of r and of z, the
                                              V-cycle removes it after every smoothing sweep,
                                              restriction and prolongation, and the dense
                                              coarsest solve is bordered by ones. Means are
                                              fixed-tree sums on the device (not the
                                              reference's left-to-right sum). Default 0. */
    uint32_t smoother_fp16_finest;         /* 1: in FP32 V-cycles with the Chebyshev smoother, the
                                              finest level's Chebyshev steps read an FP16 copy of
                                              D^-1 A (each row divided by its diagonal, 2 B per
                                              SELL-64 slot, no padding beyond the slots; columns
                                              as int16 offsets from a per-slot-row base where a
                                              slice allows) with bt = D^-1 b, summing in FP32
                                              (the same values whatever the column layout); its
                                              residual,
                                              restriction and every other level keep the FP32
                                              values. Only where the finest level is stored as
                                              SELL-64; ignored otherwise. No reference
                                              counterpart (the reference has no reduced-
                                              precision V-cycle). Default 0. */
} cfdxhip_amg_options;

typedef struct cfdxhip_amg cfdxhip_amg;

/* Fills defaults: smoothed aggregation, balanced policy, certificate on,
 * FP64, reordering on, device 0. */
void cfdxhip_amg_options_default(cfdxhip_amg_options* options);

/* NativeAMGPreconditioner(...) + configure(AMGMemoryPolicy): hypre_amg.h:35-49. */
cfdxhip_status cfdxhip_amg_create(const cfdxhip_amg_options* options, cfdxhip_amg** out);
/* Preconditioner::setup(const SparseMatrix&): hypre_amg.cpp:163-236. Copies A. */
cfdxhip_status cfdxhip_amg_setup(cfdxhip_amg* h, size_t n, const uint32_t* row_offsets,
                                 const uint32_t* columns, const double* values);
/* Preconditioner::update_values: hypre_amg.cpp:238-286. Same pattern required. */
cfdxhip_status cfdxhip_amg_update_values(cfdxhip_amg* h, const double* values);
/* Preconditioner::apply(r, z): hypre_amg.cpp:288-330. One V-cycle, z = M^{-1} r. */
cfdxhip_status cfdxhip_amg_apply(cfdxhip_amg* h, const double* r, double* z);
/* Device-pointer lifecycle for device-resident drivers (the coupled Schur
 * AMG applies inside FGMRES, core/linalg/coupled_amg_schur.h:791-798):
 * setup from a device CSR; numeric update from device values, recomputed on
 * the device (Galerkin products, diagonals, damping certificate, Chebyshev
 * bounds) with the same values, decisions and errors as the host update,
 * transactional; one V-cycle on device vectors in the caller's ordering. */
cfdxhip_status cfdxhip_amg_setup_device(cfdxhip_amg* h, size_t n, const uint32_t* row_offsets,
                                        const uint32_t* columns, const double* values);
cfdxhip_status cfdxhip_amg_update_values_device(cfdxhip_amg* h, const double* values);
cfdxhip_status cfdxhip_amg_apply_device(cfdxhip_amg* h, const double* r, double* z);
/* solve_cg_prepared(A, b, x, pc, max_iter, tol): cg_solver.h:653-667.
 * x: initial guess in, solution out. */
cfdxhip_status cfdxhip_amg_solve_cg(cfdxhip_amg* h, const double* b, double* x, size_t max_iter,
                                    double tolerance, cfdxhip_result* result);
/* solve_fgmres(A, b, x, restart, max_iter, tol, pc): gmres_solver.h:678-692,
 * FP64 outer iteration; the V-cycle runs in options.precision. */
cfdxhip_status cfdxhip_amg_solve_fgmres(cfdxhip_amg* h, const double* b, double* x, int restart,
                                        size_t max_iter, double tolerance, cfdxhip_result* result);
/* Device-resident variants (b, x on the device, caller ordering). */
cfdxhip_status cfdxhip_amg_solve_cg_device(cfdxhip_amg* h, const double* b, double* x, size_t max_iter,
                                           double tolerance, cfdxhip_result* result);
cfdxhip_status cfdxhip_amg_solve_fgmres_device(cfdxhip_amg* h, const double* b, double* x, int restart,
                                               size_t max_iter, double tolerance, cfdxhip_result* result);
/* solve_cg_prepared(A, b, x, pc, max_iter, tol, {}, {}, &projector)
 * (cg_solver.h:653-667) with a NullSpaceProjector (null_space.h:20-162)
 * built from basis_count vectors of length n (row-major, caller ordering):
 * two modified Gram-Schmidt passes and normalisation per vector, on the
 * host; a zero, non-finite or dependent vector is CFDXHIP_ERR_INVALID_ARGUMENT
 * (the reference throws). The solve returns NOT_APPLICABLE (iterations 0,
 * residuals 0) unless b is compatible (|P_N b| <= 1e-14 + 1e-12 |b|) and the
 * basis is a null space of A (|A m| <= 1e-12 |A|_F per mode). x, the initial
 * residual, every preconditioned residual, A p, the updated x and r, a
 * replaced residual and each new direction are projected; the convergence
 * test stays on the unprojected FP64 true residual. Host pointers. */
cfdxhip_status cfdxhip_amg_solve_cg_projected(cfdxhip_amg* h, const double* b, double* x, size_t max_iter,
                                              double tol, const double* basis, size_t basis_count,
                                              cfdxhip_result* result);
/* Allocation-free variant of cfdxhip_amg_solve_cg_device. No counterpart in
 * the reference: it is for callers that cannot allocate device memory (code
 * under HIP graph capture, tight serving loops, harnesses that forbid
 * hipMalloc). The PCG's work memory (seven FP64 n-vectors, partial sums,
 * scalars) comes from a fixed 128 MiB array that the library holds on each
 * GPU it runs on until the process ends; the call allocates nothing. Systems
 * needing more than that (about 2.39M unknowns) are rejected with
 * CFDXHIP_ERR_INVALID_ARGUMENT before any device work. Every call on one GPU
 * shares that array, so calls that overlap on one GPU (two handles on
 * different streams or threads) race. Results equal cfdxhip_amg_solve_cg_device
 * bit for bit. */
cfdxhip_status cfdxhip_amg_solve_cg_device_noalloc(cfdxhip_amg* h, const double* b, double* x, size_t max_iter,
                                                   double tolerance, cfdxhip_result* result);
/* NativeAMGPreconditioner::last_error: hypre_amg.h:89-96. Never NULL. */
const char* cfdxhip_amg_last_error(const cfdxhip_amg* h);
void cfdxhip_amg_destroy(cfdxhip_amg* h);

/* Hierarchy introspection (hierarchy_level_sizes / _nnz, hypre_amg.h:57-66,
 * and the first aggregation, amg_preconditioner.h:349-355). Matrices and
 * transfers are returned in the caller's (reference) ordering. */
cfdxhip_status cfdxhip_amg_num_levels(const cfdxhip_amg* h, size_t* levels);
cfdxhip_status cfdxhip_amg_level_info(const cfdxhip_amg* h, size_t level, size_t* n, size_t* nnz,
                                      size_t* prolongation_nnz);
cfdxhip_status cfdxhip_amg_level_matrix(const cfdxhip_amg* h, size_t level, uint32_t* row_offsets,
                                        uint32_t* columns, double* values);
cfdxhip_status cfdxhip_amg_level_transfer(const cfdxhip_amg* h, size_t level, uint64_t* aggregate,
                                          uint32_t* p_row_offsets, uint32_t* p_columns, double* p_values);
cfdxhip_status cfdxhip_amg_smoother_omega(const cfdxhip_amg* h, double* omega);
/* coarse_size(), hierarchy_builds(), numeric_updates() (hypre_amg.h:72,86-87):
 * size of the first coarse level (the finest level's when the hierarchy has
 * one level; amg_preconditioner.h:343-347), successful setups, successful
 * numeric updates. */
cfdxhip_status cfdxhip_amg_counters(const cfdxhip_amg* h, uint64_t* coarse_size, uint64_t* hierarchy_builds,
                                    uint64_t* numeric_updates);
/* Lanczos estimate of lambda_max(D^-1 A) on a level, the Chebyshev
 * smoother's interval anchor. CFDXHIP_ERR_NOT_READY unless a Chebyshev
 * smoother is configured. No reference counterpart. */
cfdxhip_status cfdxhip_amg_level_lambda_max(const cfdxhip_amg* h, size_t level, double* lambda_max);
/* Changes the Chebyshev degree and interval ratio of a set-up hierarchy that
 * uses a Chebyshev smoother (coefficients only, no new setup); the coarse
 * levels' degree is kept. No reference counterpart. */
cfdxhip_status cfdxhip_amg_set_chebyshev(cfdxhip_amg* h, uint32_t degree, double ratio);
/* As cfdxhip_amg_set_chebyshev, with the degree of the levels below the
 * finest (0: the finest level's degree). No reference counterpart. */
cfdxhip_status cfdxhip_amg_set_chebyshev_levels(cfdxhip_amg* h, uint32_t degree, uint32_t degree_coarse,
                                                double ratio);
/* configure_cf_interpolation_limit / cf_interpolation_limit (hypre_amg.h:
 * 51-54, hypre_amg.cpp:97-110): cap on the entries of a C/F (Boomer-style)
 * interpolation row. Rows above it keep their max_entries largest |w| (ties:
 * lower coarse index), renormalised to sum 1 (amg_preconditioner.h:
 * 1840-1883); a kept sum below 1e-12 of the kept |w| fails setup. 0 = no
 * cap (default); 1 is rejected with CFDXHIP_ERR_INVALID_ARGUMENT. A changed
 * cap drops the current hierarchy: setup must run again. */
cfdxhip_status cfdxhip_amg_configure_cf_interpolation_limit(cfdxhip_amg* h, size_t max_entries);
cfdxhip_status cfdxhip_amg_cf_interpolation_limit(const cfdxhip_amg* h, size_t* max_entries);
/* configure_max_coarsening_fraction (hypre_amg.h:55-58, hypre_amg.cpp:
 * 112-121): coarsening stops before a level that keeps at least `fraction`
 * of the unknowns (amg_preconditioner.h:161-175). fraction in [0.5, 1]; 1
 * (default) disables. A change drops the current hierarchy. */
cfdxhip_status cfdxhip_amg_configure_max_coarsening_fraction(cfdxhip_amg* h, double fraction);
/* configure_bounded_nonsymmetric_action / bounded_action_fallbacks
 * (hypre_amg.h:59-63, hypre_amg.cpp:123-139,293-326), for nonsymmetric
 * Krylov use: after each preconditioner application z = M r (apply, FGMRES,
 * PCG), a z whose image A z is not finite or exceeds max_image_ratio |r| is
 * replaced by the damped Jacobi action 0.7 D^-1 r (counted as a fallback);
 * if that fails the same test the application fails. 0 disables (default);
 * otherwise [1, 1e6]. Setup then requires a handle created with
 * require_smoother_certificate = 0 and a finest diagonal with
 * |a_ii| >= 1e-12 max_j |a_ij| (update_values checks the latter again). A
 * change drops the current hierarchy. The allocation-free PCG rejects such a
 * handle. */
cfdxhip_status cfdxhip_amg_configure_bounded_nonsymmetric_action(cfdxhip_amg* h, double max_image_ratio);
cfdxhip_status cfdxhip_amg_bounded_action_fallbacks(const cfdxhip_amg* h, uint64_t* fallbacks);
/* operator_complexity(), grid_complexity() (hypre_amg.h:75-76,
 * amg_preconditioner.h:376-390): sum of nnz (rows) over the levels divided
 * by the finest level's; 0 before setup. */
cfdxhip_status cfdxhip_amg_complexity(const cfdxhip_amg* h, double* operator_complexity, double* grid_complexity);
/* first_prolongation_nnz(), prolongation_row_sum_min/max() (hypre_amg.h:
 * 77,83-84; amg_preconditioner.h:412-430,1166-1190): entries and extreme
 * row sums of the finest level's P. CFDXHIP_ERR_INVALID_ARGUMENT for a
 * hierarchy of one level. */
cfdxhip_status cfdxhip_amg_prolongation_stats(const cfdxhip_amg* h, uint64_t* first_nnz, double* row_sum_min,
                                              double* row_sum_max);
/* Seconds spent in the last setup: host construction, device upload. */
cfdxhip_status cfdxhip_amg_setup_seconds(const cfdxhip_amg* h, double* host_seconds, double* device_seconds);
/* Wall seconds of the last successful update_values (host or device entry). */
cfdxhip_status cfdxhip_amg_update_seconds(const cfdxhip_amg* h, double* seconds);

/* Plain CSR SpMV on the device, y = A x, FP64 (sparse_matrix.h:226-242).
 * Kept for measurement: runs the hierarchy's finest-level kernel on the
 * caller-ordered vectors. repeat >= 1 launches back to back; the kernel time
 * of the last batch (HIP events on the handle's stream) is returned. */
cfdxhip_status cfdxhip_amg_spmv_device(cfdxhip_amg* h, uint32_t precision, const void* x, void* y,
                                       uint32_t repeat, double* seconds_per_launch);
/* Measurement: seconds per launch of one hierarchy level's kernel on the
 * level's own buffers, timed with HIP events on the handle's stream.
 * kind 0: y = A x; kind 1: the fused damped-Jacobi sweep. precision 0 FP64,
 * 1 FP32, 2 one Chebyshev step on the finest level's FP16 copy (kind
 * ignored; smoother_fp16_finest). No reference counterpart. */
cfdxhip_status cfdxhip_amg_level_kernel_seconds(cfdxhip_amg* h, size_t level, uint32_t precision, uint32_t kind,
                                                uint32_t repeat, double* seconds);
/* Measurement: seconds per launch of the two Gram-Schmidt passes of FGMRES
 * Arnoldi step j (0 <= j < 120, j < n) on the finest level's size: the product
 * pass over j + 1 basis vectors and w, and the update pass (each with its
 * partial-sum reduction), HIP events on the handle's stream, on placeholder
 * basis values. No reference counterpart. */
cfdxhip_status cfdxhip_amg_gram_schmidt_seconds(cfdxhip_amg* h, uint32_t j, uint32_t repeat, double* dot_seconds,
                                                double* update_seconds);
/* First level that the FP64 V-cycle runs in its single-launch coarse end (the
 * number of levels: none). Diagnostics only. No reference counterpart. */
cfdxhip_status cfdxhip_amg_coarse_end(const cfdxhip_amg* h, size_t* first_level);
/* Storage the device SpMV of a level's matrix streams: format 0 = CSR
 * stream (stored_entries = nnz, slices = 0), 1 = SELL-64 (slices of 64 rows,
 * stored_entries = slots including padding). Measurement only: the byte
 * counts of a level's kernels follow from it. No reference counterpart. */
cfdxhip_status cfdxhip_amg_level_spmv_format(const cfdxhip_amg* h, size_t level, uint32_t* format,
                                             uint64_t* stored_entries, uint64_t* slices);
/* Bytes the device SpMV of a level's matrix streams for the matrix itself
 * (values, 4 B columns, row or slice offsets; x and y not included), for
 * precision 0 (FP64), 1 (FP32) or 2 (the FP16 smoothing copy: 2 B values,
 * int16 column offsets and per-slot-row bases, or 4 B columns in slices that
 * keep them, slot offsets and slice flags). Measurement only. No reference
 * counterpart. */
cfdxhip_status cfdxhip_amg_level_spmv_bytes(const cfdxhip_amg* h, size_t level, uint32_t precision,
                                            uint64_t* matrix_bytes);

/* ------------------------------------------------------------ meshes ---- */

/* Synthetic unstructured hex meshes (inputs of the workloads). */
enum { CFDXHIP_MESH_BOX = 0, CFDXHIP_MESH_EXTRUDED_2D = 1, CFDXHIP_MESH_CHANNEL_STEP = 2 };
typedef struct cfdxhip_mesh_spec {
    uint32_t kind;
    uint32_t nx, ny, nz;
    double lx, ly, lz;
    double jitter;
    uint32_t wall_layers;
    uint32_t permute;
    double first_aspect;
    double growth;
    double step_height_fraction;
    double step_length_fraction;
    uint64_t seed;
} cfdxhip_mesh_spec;

typedef struct cfdxhip_host_mesh cfdxhip_host_mesh;
typedef struct cfdxhip_mesh_sizes {
    uint64_t n_points, n_faces, n_internal_faces, n_cells, n_face_vertices, n_cell_faces, n_patches;
} cfdxhip_mesh_sizes;

cfdxhip_status cfdxhip_mesh_generate(const cfdxhip_mesh_spec* spec, cfdxhip_host_mesh** out);
cfdxhip_status cfdxhip_mesh_sizes_get(const cfdxhip_host_mesh* m, cfdxhip_mesh_sizes* sizes);
/* Copies the mesh arrays; any pointer may be NULL to skip that array.
 * patch_kind: 0 wall, 1 empty, 2 symmetry (PatchType, mesh/boundary.h:31-40).
 * patch_of_face: patch id of boundary faces, UINT32_MAX for internal faces.
 * cell_ijk: lattice coordinates of each cell (3 per cell). */
cfdxhip_status cfdxhip_mesh_copy(const cfdxhip_host_mesh* m, double* px, double* py, double* pz,
                                 uint32_t* face_offsets, uint32_t* face_vertices, uint32_t* owner,
                                 int32_t* neighbour, uint32_t* cell_offsets, uint32_t* cell_faces,
                                 uint32_t* patch_of_face, uint8_t* patch_kind, uint32_t* cell_ijk);
void cfdxhip_mesh_destroy(cfdxhip_host_mesh* m);

/* ------------------------------------------- finite-volume assembly ---- */

/* Device-resident mesh: points, face->vertex CSR, owner/neighbour (neighbour
 * -1 on boundary faces), cell->face CSR, patch id per face (UINT32_MAX for
 * internal faces) and patch kinds (0 wall, 1 empty, 2 symmetry). Geometry is
 * computed on the device at creation: build_fv_geometry,
 * physics/finite_volume_transport.h:92-175. */
typedef struct cfdxhip_fv cfdxhip_fv;
cfdxhip_status cfdxhip_fv_create(int32_t device, size_t n_points, const double* px, const double* py,
                                 const double* pz, size_t n_faces, const uint32_t* face_offsets,
                                 const uint32_t* face_vertices, const uint32_t* owner, const int32_t* neighbour,
                                 size_t n_cells, const uint32_t* cell_offsets, const uint32_t* cell_faces,
                                 size_t n_patches, const uint32_t* patch_of_face, const uint8_t* patch_kind,
                                 cfdxhip_fv** out);
void cfdxhip_fv_destroy(cfdxhip_fv* fv);
const char* cfdxhip_fv_last_error(const cfdxhip_fv* fv);
/* Geometry copy-out: xyz triplets per face / cell, volumes. NULL skips. */
cfdxhip_status cfdxhip_fv_geometry(cfdxhip_fv* fv, double* face_centres, double* face_area_vectors,
                                   double* cell_centres, double* cell_volumes);
/* gauss_gradient_with_boundary, steady_incompressible_solver.h:1634-1750.
 * bc_type per patch: 0 zero-gradient, 1 fixed value, 2 fixed gradient.
 * grad: 3 x n_cells, component-major. */
cfdxhip_status cfdxhip_fv_gauss_gradient(cfdxhip_fv* fv, const uint8_t* bc_type, const double* bc_value,
                                         const double* p, double* grad);
/* make_mass_flux, steady_incompressible_solver.h:1842-1905. vbc_type per
 * patch: 0 zero-gradient, 1 fixed value (3 values per patch). U: 3 x n_cells. */
cfdxhip_status cfdxhip_fv_mass_flux(cfdxhip_fv* fv, const uint8_t* vbc_type, const double* vbc_value, double rho,
                                    const double* U, double* phi);
/* Sparsity of the pressure system (steady_incompressible_solver.h:8599-8652):
 * with no fixed-pressure patch the reference cell is eliminated. row_offsets
 * and columns may be NULL to query sizes. */
cfdxhip_status cfdxhip_fv_pressure_pattern(cfdxhip_fv* fv, const uint8_t* pbc_type, size_t reference_cell,
                                           size_t* n_rows, size_t* nnz, uint32_t* row_offsets, uint32_t* columns);
/* SIMPLE corrector assembly (steady_incompressible_solver.h:8048-8181):
 * values of the pattern above and the RHS. rAU: 3 x n_cells, phiHbyA: per
 * face, p: per cell. Host pointers. */
cfdxhip_status cfdxhip_fv_pressure_assemble(cfdxhip_fv* fv, const uint8_t* pbc_type, const double* pbc_value,
                                            double rho, const double* rAU, const double* phiHbyA, const double* p,
                                            size_t reference_cell, double* values, double* rhs);
/* Same with device pointers (rAU, phiHbyA, p, values, rhs). */
cfdxhip_status cfdxhip_fv_pressure_assemble_device(cfdxhip_fv* fv, const uint8_t* pbc_type,
                                                   const double* pbc_value, double rho, const double* rAU,
                                                   const double* phiHbyA, const double* p, size_t reference_cell,
                                                   double* values, double* rhs);
/* assemble_cell_diffusion_matrix (core/solvers/scalar_diffusion.h:39-163):
 * face_value NaN = unprescribed face; face_is_neumann selects q_n faces.
 * Pattern: diagonal + face neighbours (n_cells rows). */
cfdxhip_status cfdxhip_fv_diffusion_assemble(cfdxhip_fv* fv, double gamma, const double* source,
                                             const double* face_value, const uint8_t* face_is_neumann,
                                             size_t* nnz, uint32_t* row_offsets, uint32_t* columns,
                                             double* values, double* rhs);

/* Green-Gauss gradient from a face list on device arrays, without a mesh
 * handle; replaces cfdx_cuda_gradient_gauss (runtime/gpu/cuda_kernels.cu:
 * 43-65). Face value 1/2 (phi_o + phi_n) where neighbour >= 0, phi_o
 * elsewhere; owner += phi_f S_f, neighbour -= phi_f S_f; then g /= V (0
 * where V <= 0). Per-cell sums arrive through FP64 atomics in no fixed
 * order, as in the reference. phi, volume, gx, gy, gz: n_cells; sx, sy, sz,
 * owner, neighbour: n_faces. stream: a hipStream_t (NULL: the null stream);
 * the call synchronises it. Status codes replace the reference's
 * exceptions: CFDXHIP_ERR_INVALID_ARGUMENT when an owner or neighbour index
 * is out of range (such faces are skipped), CFDXHIP_ERR_DEVICE on a HIP
 * failure. */
cfdxhip_status cfdxhip_gradient_gauss_device(const double* phi, const double* sx, const double* sy,
                                             const double* sz, const uint32_t* owner, const int64_t* neighbour,
                                             const double* volume, size_t n_faces, size_t n_cells, double* gx,
                                             double* gy, double* gz, void* stream);
/* Face-list divergence, div[o] += phi_face[f], div[n] -= phi_face[f]
 * (neighbour >= 0), on device arrays; replaces cfdx_cuda_divergence
 * (runtime/gpu/cuda_kernels.cu:67-97). Same conventions as
 * cfdxhip_gradient_gauss_device. */
cfdxhip_status cfdxhip_divergence_device(const double* phi_face, const uint32_t* owner, const int64_t* neighbour,
                                         size_t n_faces, size_t n_cells, double* div, void* stream);

/* ---------------------------------------- momentum side of SIMPLE ---- */

/* compute_boundary_aware_wls_gradient (physics/finite_volume_transport.h:
 * 606-715): per-cell weighted least-squares gradient of a scalar cell field
 * (one-sided Jacobi fit, core/fvm/least_squares_gradient.h:77-205), kept at
 * the boundary-aware Green-Gauss value (:505-586) where the fit is not
 * rank- and condition-certified. bc_type per patch: 0 zero-gradient,
 * 1 fixed value, 2 fixed gradient (bc_value holds the value or gradient).
 * condition_limit: the reference's argument (1e8). grad: 3 x n_cells.
 * fallback_cells (may be NULL): cells left at Green-Gauss. Cells may have at
 * most 10 faces. Host pointers. */
cfdxhip_status cfdxhip_fv_wls_gradient(cfdxhip_fv* fv, const uint8_t* bc_type, const double* bc_value,
                                       double condition_limit, const double* field, double* grad,
                                       size_t* fallback_cells);
/* Sparsity of the momentum equations: every cell, its diagonal and its face
 * neighbours, columns ascending (n_cells rows). NULL arrays query sizes. */
cfdxhip_status cfdxhip_fv_momentum_pattern(cfdxhip_fv* fv, size_t* n_rows, size_t* nnz, uint32_t* row_offsets,
                                           uint32_t* columns);
/* The SIMPLE momentum predictor's three equations as the reference builds
 * them: assemble_momentum_component (cell-viscosity overload,
 * steady_incompressible_solver.h:3262-3311 over finite_volume_transport.h:
 * 882-1310: UPWIND, bounded or not, orthogonal conductance plus the
 * non-orthogonal correction from the WLS velocity gradients), then
 * relax_momentum_equation (:3728-3770) with alpha_u in (0, 1]. vbc_type per
 * patch: 1 fixed value (3 values per patch), otherwise zero-gradient. mu:
 * cell viscosity; phi: face mass flux; grad_p: 3 x n_cells; body: 3 x n_cells
 * force density or NULL; U: current velocity 3 x n_cells (convected field
 * and relaxation state). The three component matrices are identical, so
 * values (the momentum pattern) and diag (n_cells, relaxed) are written once;
 * rhs is 3 x n_cells. Host pointers. */
cfdxhip_status cfdxhip_fv_momentum_assemble(cfdxhip_fv* fv, const uint8_t* vbc_type, const double* vbc_value,
                                            const double* mu, const double* phi, const double* grad_p,
                                            const double* body, const double* U, int32_t bounded, double alpha_u,
                                            double* values, double* rhs, double* diag);
/* Same with device pointers (vbc arrays stay on the host). */
cfdxhip_status cfdxhip_fv_momentum_assemble_device(cfdxhip_fv* fv, const uint8_t* vbc_type,
                                                   const double* vbc_value, const double* mu, const double* phi,
                                                   const double* grad_p, const double* body, const double* U,
                                                   int32_t bounded, double alpha_u, double* values, double* rhs,
                                                   double* diag);
/* rAU = 1 / diag (steady_incompressible_solver.h:7816-7836, SIMPLE) and
 * HbyA = rAU (rhs + grad_p V - sum of off-diagonal a U) (build_hbya
 * :6430-6465), from the assembled equations and the predicted velocity U.
 * rAU, HbyA: 3 x n_cells. Host pointers. */
cfdxhip_status cfdxhip_fv_momentum_hbya(cfdxhip_fv* fv, const double* values, const double* rhs, const double* diag,
                                        const double* grad_p, const double* U, double* rAU, double* HbyA);
cfdxhip_status cfdxhip_fv_momentum_hbya_device(cfdxhip_fv* fv, const double* values, const double* rhs,
                                               const double* diag, const double* grad_p, const double* U, double* rAU,
                                               double* HbyA);
/* Post-solve velocity U = HbyA - rAU grad_p V (steady_incompressible_solver.h:
 * 9545-9557), grad_p of the corrected pressure. Host / device pointers. */
cfdxhip_status cfdxhip_fv_velocity_correct(cfdxhip_fv* fv, const double* HbyA, const double* rAU,
                                           const double* grad_p, double* U);
cfdxhip_status cfdxhip_fv_velocity_correct_device(cfdxhip_fv* fv, const double* HbyA, const double* rAU,
                                                  const double* grad_p, double* U);
/* Post-solve face flux: make_rhie_chow_mass_flux (steady_incompressible_solver.h:
 * 2063-2217) with the corrector's arguments (HBYA_PREDICTOR, linear weights,
 * Gauss pressure gradient). Host / device pointers (BC arrays on the host). */
cfdxhip_status cfdxhip_fv_rhie_chow_flux(cfdxhip_fv* fv, const uint8_t* vbc_type, const double* vbc_value,
                                         const uint8_t* pbc_type, const double* pbc_value, double rho,
                                         const double* HbyA, const double* p, const double* rAU, double* phi);
cfdxhip_status cfdxhip_fv_rhie_chow_flux_device(cfdxhip_fv* fv, const uint8_t* vbc_type, const double* vbc_value,
                                                const uint8_t* pbc_type, const double* pbc_value, double rho,
                                                const double* HbyA, const double* p, const double* rAU,
                                                double* phi);

/* ------------------------------------------------------------------------
 * Learned preconditioner stage. No reference counterpart (the reference has
 * no learned component). A 4-layer message-passing network, hidden width 32,
 * on the graph of the finest operator of a set-up FP32 (mixed) hierarchy:
 * features are the symmetrically scaled couplings -a_ij / sqrt(a_ii a_jj)
 * and the scaled residual r_i / sqrt(a_ii). Inside mixed FGMRES the stage is
 * z = N(r) + V(r - A N(r)), V one FP32 V-cycle. BF16 MFMA, FP32 accumulation.
 * The graph must be symmetric (the pressure Laplacian is).
 * ------------------------------------------------------------------------ */
typedef struct cfdxhip_mpnn cfdxhip_mpnn;

/* Number of network parameters (8417). Layout: w_in[32], b_in[32]; per layer
 * l = 0..3 at 64 + 2080 l: W_l[64][32] row-major (rows: [h; m] features),
 * b_l[32]; then w_out[32], b_out. */
size_t cfdxhip_mpnn_param_count(void);
cfdxhip_status cfdxhip_mpnn_create(int32_t device, cfdxhip_mpnn** out);
void cfdxhip_mpnn_destroy(cfdxhip_mpnn* m);
const char* cfdxhip_mpnn_last_error(const cfdxhip_mpnn* m);
/* Sets the FP32 parameters (resets the Adam moments and step count). */
cfdxhip_status cfdxhip_mpnn_set_params(cfdxhip_mpnn* m, const float* params, size_t count);
cfdxhip_status cfdxhip_mpnn_get_params(cfdxhip_mpnn* m, float* params, size_t count);
/* e = N(r) on the graph of h's finest level; host FP64 vectors, caller order. */
cfdxhip_status cfdxhip_mpnn_forward(cfdxhip_mpnn* m, cfdxhip_amg* h, const double* r, double* e);
/* grad = d(ge . N(r)) / d params (the network's backward pass). */
cfdxhip_status cfdxhip_mpnn_vjp(cfdxhip_mpnn* m, cfdxhip_amg* h, const double* r, const double* ge, float* grad);
/* One Adam step (beta1 0.9, beta2 0.999, eps 1e-8) with a host gradient. */
cfdxhip_status cfdxhip_mpnn_adam_step(cfdxhip_mpnn* m, const float* grad, float lr);
/* Solver-generated training pairs: FP64 PCG from x = 0 to tol on b (host,
 * caller order) with h's FP64 V-cycle; at each listed iteration k the pair
 * (r_k = b - A x_k, e_k = x_final - x_k) is kept on the device. */
cfdxhip_status cfdxhip_mpnn_collect_pairs(cfdxhip_mpnn* m, cfdxhip_amg* h, const double* b,
                                          const uint64_t* iterations, uint32_t count, double tol,
                                          uint32_t* collected, cfdxhip_result* solve);
/* `steps` Adam steps over the collected pairs (cyclically), minimising
 * 1/2 |(I - V A)(e - N(r))|_A^2 / (e^T r). losses[steps] (optional) receives
 * each step's loss. */
cfdxhip_status cfdxhip_mpnn_train(cfdxhip_mpnn* m, cfdxhip_amg* h, uint32_t steps, float lr, double* losses);
/* Fallback rule: inside a learned solve the stage is dropped for the rest of
 * the solve (plain V-cycle, counted in learned_stage_fallbacks) once a
 * residual reduction drops below min_reduction: the network's own,
 * 1 - |r - A N(r)| / |r|, at any application, or the FGMRES reduction per
 * iteration over the last `window` iterations, 1 - (|g_k| /
 * |g_{k-window}|)^(1/window) from the Givens estimates (default 0.5, window 3;
 * min_reduction <= 1; a negative value keeps the stage on). */
cfdxhip_status cfdxhip_mpnn_set_fallback(cfdxhip_mpnn* m, double min_reduction, uint32_t window);
/* Mixed FGMRES with the learned stage ahead of the FP32 V-cycle (host or
 * device vectors). Same contract as cfdxhip_amg_solve_fgmres. */
cfdxhip_status cfdxhip_amg_solve_fgmres_learned(cfdxhip_amg* h, cfdxhip_mpnn* m, const double* b, double* x,
                                                int restart, size_t max_iter, double tol, cfdxhip_result* result);
cfdxhip_status cfdxhip_amg_solve_fgmres_learned_device(cfdxhip_amg* h, cfdxhip_mpnn* m, const double* b,
                                                       double* x, int restart, size_t max_iter, double tol,
                                                       cfdxhip_result* result);

/* ------------------------------------------------------------------------
 * Linear-system capture files (.cfdxlin, CFDX_LINEAR_REPLAY_V1): read and
 * write the reference's replay format (core/linalg/linear_system_capture.h:
 * 165-284: write_linear_system_capture, read_linear_system_capture), byte for
 * byte, with its FNV-1a checksum and limits (rows <= 2,000,000,
 * nnz <= 100,000,000). The reference's file-level validation applies: square
 * finalized CSR with strictly ascending columns, finite values, known enum
 * values, 0 < max_iterations <= 1e8, finite tolerance > 0.
 * ------------------------------------------------------------------------ */
typedef struct cfdxhip_capture cfdxhip_capture;
typedef struct cfdxhip_capture_info {
    uint64_t n;               /* rows = columns */
    uint64_t nnz;
    uint64_t max_iterations;
    uint64_t checksum;        /* read: the file's; write: ignored (computed) */
    uint32_t problem;         /* LinearProblemKind 0..5 (linear_solver_models.h:11-18) */
    uint32_t null_space;      /* NullSpaceModel 0..1 (:59) */
    uint32_t scaling;         /* LinearScalingModel 0..4 (:61) */
    uint32_t reserved;
    double tolerance;
} cfdxhip_capture_info;

/* Parses and verifies a capture (checksum, CSR, limits). On failure the
 * reason is in cfdxhip_capture_last_error() (per thread). */
cfdxhip_status cfdxhip_capture_read(const char* path, cfdxhip_capture** out);
cfdxhip_status cfdxhip_capture_info_get(const cfdxhip_capture* capture, cfdxhip_capture_info* info);
/* Copies the system out: row_offsets[n+1], columns[nnz], values[nnz],
 * rhs[n], initial_solution[n]. */
cfdxhip_status cfdxhip_capture_copy(const cfdxhip_capture* capture, uint32_t* row_offsets, uint32_t* columns,
                                    double* values, double* rhs, double* initial_solution);
void cfdxhip_capture_destroy(cfdxhip_capture* capture);
/* Writes a capture atomically (temporary file + rename); checksum_out
 * (optional) receives the checksum written. */
cfdxhip_status cfdxhip_capture_write(const char* path, const cfdxhip_capture_info* info, const uint32_t* row_offsets,
                                     const uint32_t* columns, const double* values, const double* rhs,
                                     const double* initial_solution, uint64_t* checksum_out);
const char* cfdxhip_capture_last_error(void);

/* Version string of the library build. */
const char* cfdxhip_version(void);

#ifdef __cplusplus
}
#endif

#endif /* CFDXHIP_H */
