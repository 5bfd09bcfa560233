// Device-resident finite-volume mesh, geometry, pressure assembly and the
// momentum side of the SIMPLE corrector.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

namespace cfdxhip {

// CSR sparsity of an assembled system and the maps that fill its values.
struct PressurePlan {
    uint32_t n = 0;
    uint64_t nnz = 0;
    uint32_t ref = 0;
    std::vector<uint32_t> h_rowp, h_cols;
    uint32_t* rowp = nullptr;
    uint32_t* cols = nullptr;
    // full system only: per nonzero, the diagonal's row (or ~0u) and the
    // faces joining the pair, ascending
    uint32_t* nz_row_diag = nullptr;
    uint32_t* nzf_off = nullptr;
    uint32_t* nzf = nullptr;
    // Per internal cell: its row's first nonzero and its row (~0: left out), and
    // the places in that row of its slots' neighbours, slot-major in ascending
    // caller face id, and of the diagonal (0xffff: none).
    uint32_t *row_start = nullptr, *row_of = nullptr;
    uint16_t *slot_rank = nullptr, *diag_rank = nullptr;
    bool shared_pairs = false;  // some pair of cells is joined by several faces

    void release();
    void release_maps();
};

struct FvMesh {
    int dev = 0;
    hipStream_t stream = nullptr;
    uint32_t np = 0, nf = 0, nc = 0, npatch = 0;
    double *px = nullptr, *py = nullptr, *pz = nullptr;
    uint32_t *foff = nullptr, *fvtx = nullptr, *owner = nullptr, *coff = nullptr, *cfaces = nullptr;
    uint32_t* cfaces_sorted = nullptr;  // each cell's faces in ascending caller face id (internal ids)
    // internal numbering: new_of_old / old_of_new for cells and faces
    uint32_t *cell_new = nullptr, *cell_old = nullptr, *face_new = nullptr, *face_old = nullptr;
    std::vector<uint32_t> h_cell_new, h_face_new;
    bool identity_order = false;  // the caller's numbering is kept (no permutation)
    int32_t* neigh = nullptr;
    uint32_t* patch = nullptr;
    uint8_t* patch_kind = nullptr;
    // geometry (SoA)
    double *fcx = nullptr, *fcy = nullptr, *fcz = nullptr;
    double *fsx = nullptr, *fsy = nullptr, *fsz = nullptr;
    double *ccx = nullptr, *ccy = nullptr, *ccz = nullptr;
    double* vol = nullptr;
    double* vol_caller = nullptr;  // cell volumes in the caller's numbering
    int *err = nullptr, *h_err = nullptr;  // error flags: device and host address of pinned memory
    // work
    double *work_coeff = nullptr, *work_diag = nullptr, *work_grad = nullptr;
    // momentum side: velocity WLS gradients (three records a cell), flags, and
    // per patch (last: internal faces) whether faces are non-orthogonal, then
    // whether their geometry leaves that undefined
    double* mom_ugrad = nullptr;
    int* mom_flags = nullptr;
    std::vector<int> h_nonorth;
    double* slot_coeff = nullptr;  // coefficients per slot, where they do not fit LDS
    // per-patch boundary data of a call: device buffer (bc_u8 in its tail) and
    // its pinned host side
    uint8_t* bc_u8 = nullptr;
    double* bc_f64 = nullptr;
    double* bc_host = nullptr;
    uint8_t* h_bc_u8 = nullptr;
    PressurePlan pressure_full, pressure_red;
    // host copies of the addressing
    std::vector<uint32_t> h_owner, h_coff, h_cf, h_patch;
    std::vector<int32_t> h_neigh;
    std::vector<uint8_t> h_kind;
    std::vector<uint8_t> h_patch_boundary;  // per patch: owns at least one boundary face
    // slot stencils (slot-major, slot_D slots per cell) and the WLS fit cache
    uint32_t slot_D = 0;
    bool slots_built = false;
    uint8_t* slot_sorted = nullptr;  // per cell, its slots in ascending caller face id
    int32_t* slot_other = nullptr;
    double4* cell_rec = nullptr;  // (centre, volume) per cell
    uint32_t* slot_face = nullptr;
    double *slot_w = nullptr, *slot_sx = nullptr, *slot_sy = nullptr, *slot_sz = nullptr;
    double *wls_a0 = nullptr, *wls_a1 = nullptr, *wls_a2 = nullptr, *wls_fac = nullptr, *wls_nd = nullptr;
    double *wls_sig = nullptr, *wls_V = nullptr, *wls_cond = nullptr;
    uint32_t* wls_meta = nullptr;
    std::vector<uint8_t> wls_key;
    // scratch for fields moved into the internal numbering (slot -> buffer)
    std::vector<std::pair<double*, uint64_t>> scratch;
    uint8_t* scratch_u8 = nullptr;

    FvMesh() = default;
    ~FvMesh();
    FvMesh(const FvMesh&) = delete;
    FvMesh& operator=(const FvMesh&) = delete;

    void create(int device, uint64_t np, const double* px, const double* py, const double* pz, uint64_t nf,
                const uint32_t* foff, const uint32_t* fvtx, const uint32_t* owner, const int32_t* neigh,
                uint64_t nc, const uint32_t* coff, const uint32_t* cf, uint64_t npatch, const uint32_t* patch,
                const uint8_t* kind);
    void compute_geometry();
    void geometry_out(double* fc_aos, double* fs_aos, double* cc_aos, double* vol);
    void gauss_gradient_device(const uint8_t* d_bct, const double* d_bcv, const double* d_p, double* d_grad);
    void mass_flux_device(const uint8_t* d_vbt, const double* d_vbv, double rho, const double* d_U, double* d_phi);
    const PressurePlan& pressure_plan(bool eliminate, uint32_t ref);
    const PressurePlan& row_plan(bool eliminate, uint32_t ref);
    void prepare_rows(bool eliminate, uint32_t ref);
    bool has_fixed_pressure(const uint8_t* h_pbt) const;
    const PressurePlan& pressure_assemble_device(const uint8_t* h_pbt, const double* h_pbv, double rho,
                                                 const double* d_rAU, const double* d_phi, const double* d_p,
                                                 uint64_t ref, double* d_vals, double* d_rhs);
    const PressurePlan& diffusion_assemble_device(double gamma, const double* d_source, const double* d_fval,
                                                  const uint8_t* d_fneu, double* d_vals, double* d_rhs);
    // Momentum side (device pointers; velocity BCs per patch on the host:
    // type 1 fixed value with 3 values, otherwise zero-gradient).
    void wls_gradient_device(const uint8_t* h_bt, const double* h_bv, double limit, const double* d_field,
                             double* d_grad, uint8_t* d_fallback);
    const PressurePlan& momentum_assemble_device(const uint8_t* h_vbt, const double* h_vbv, const double* d_mu,
                                                 const double* d_phi, const double* d_gradp, const double* d_body,
                                                 const double* d_U, bool bounded, double alpha, double* d_vals,
                                                 double* d_rhs, double* d_diag);
    void momentum_hbya_device(const double* d_vals, const double* d_rhs, const double* d_diag,
                              const double* d_gradp, const double* d_U, double* d_rau, double* d_hbya);
    void velocity_correct_device(const double* d_hbya, const double* d_rau, const double* d_gradp, double* d_U);
    void rhie_chow_flux_device(const uint8_t* h_vbt, const double* h_vbv, const uint8_t* h_pbt,
                               const double* h_pbv, double rho, const double* d_hbya, const double* d_p,
                               const double* d_rau, double* d_phi);
    void ensure_momentum_work();
    void upload_bcs(const uint8_t* h_vbt, const double* h_vbv, const uint8_t* h_pbt, const double* h_pbv, bool raw_pbt, int* flags);
    void clear_err();
    int stencil_dimension() const;
    double* scr(size_t slot, uint64_t count);
    void cells_in(const double* caller, double* internal, int comps);
    void cells_out(const double* internal, double* caller, int comps);
    void faces_in(const double* caller, double* internal);
    void faces_out(const double* internal, double* caller);
    const double* cin(const double* caller, size_t slot, int comps);
    const double* fin(const double* caller, size_t slot);
    double* cout_buf(double* caller, size_t slot, int comps);
    double* fout_buf(double* caller, size_t slot);
    void ensure_slots();
    void release_slots();
    void ensure_wls_cache(const uint8_t* h_bt, const uint8_t* d_bt);
    void gauss_gradient_internal(const uint8_t* d_bct, const double* d_bcv, const double* p, uint32_t ps);
    void map_rows(PressurePlan& plan, uint32_t ref);
    uint64_t touched_lines(const uint32_t* at, const uint32_t* cell_place, const uint32_t* face_place,
                           uint64_t* fewest) const;
    void check_err(const char* what);
    void release();
};

// Face-list Green-Gauss gradient and divergence on caller device arrays
// (runtime/gpu/cuda_kernels.cu:7-97), on stream s, which they synchronise.
// False when an owner or neighbour index is out of range.
bool face_gradient_gauss(const double* phi, const double* sx, const double* sy, const double* sz,
                         const uint32_t* owner, const int64_t* neighbour, const double* volume, uint64_t n_faces,
                         uint64_t n_cells, double* gx, double* gy, double* gz, hipStream_t s);
bool face_divergence(const double* phi_face, const uint32_t* owner, const int64_t* neighbour, uint64_t n_faces,
                     uint64_t n_cells, double* div, hipStream_t s);

}  // namespace cfdxhip
