"""cfdx_dev_amd: MI355X-native pressure-correction solve for CFDX.

Python mirror of the reference's solver interface over the C ABI of
libcfdxhip.so:

* :class:`NativeAMGPreconditioner` follows core/linalg/hypre_amg.h:26-101
  (setup / update_values / apply return ``bool`` and keep ``last_error``);
* :meth:`NativeAMGPreconditioner.solve_cg` follows solve_cg_prepared
  (core/linalg/cg_solver.h:653-667) and returns a :class:`SolverResult`
  mirroring core/linalg/solver_status.h:45-72;
* :meth:`NativeAMGPreconditioner.solve_fgmres` follows solve_fgmres
  (core/linalg/gmres_solver.h:678-692).

All numerical work runs in libcfdxhip.so on the GPU; nothing here computes.
"""
from __future__ import annotations

import ctypes as C
import os
from dataclasses import dataclass, field

import numpy as np

from . import _native
from ._native import AmgOptions, MeshSizes, MeshSpec, Result

CONVERGED, MAX_ITER_REACHED, DIVERGED, NOT_APPLICABLE = 0, 1, 2, 3
STATUS_NAMES = {0: "converged", 1: "max_iter_reached", 2: "diverged", 3: "not_applicable"}

METHODS = {"boomer": 0, "directcf": 0, "sa": 1, "smoothed_aggregation": 1}
POLICIES = {"low": 0, "balanced": 1, "fast": 2}
PRECISIONS = {"fp64": 0, "fp32": 1}
SMOOTHERS = {"jacobi": 0, "chebyshev": 1}


@dataclass
class SolverResult:
    status: int
    iterations: int
    residual: float
    residual_relative: float
    residual_replacements: int = 0
    solve_seconds: float = 0.0
    preconditioner_applications: int = 0
    extra: dict = field(default_factory=dict)

    def converged(self) -> bool:
        return self.status == CONVERGED

    @staticmethod
    def from_c(r: Result) -> "SolverResult":
        return SolverResult(
            status=r.status,
            iterations=r.iterations,
            residual=r.residual,
            residual_relative=r.residual_relative,
            residual_replacements=r.residual_replacements,
            solve_seconds=r.solve_seconds,
            preconditioner_applications=r.preconditioner_applications,
            extra={
                "max_true_recursive_gap": r.max_true_recursive_gap,
                "min_true_residual": r.min_true_residual,
                "max_true_residual": r.max_true_residual,
                "learned_stage_applications": r.learned_stage_applications,
                "learned_stage_fallbacks": r.learned_stage_fallbacks,
            },
        )


def _u32(a):
    return np.ascontiguousarray(a, dtype=np.uint32)


def _f64(a):
    return np.ascontiguousarray(a, dtype=np.float64)


class NativeAMGPreconditioner:
    """GPU AMG preconditioner with the reference's lifecycle (hypre_amg.h:26-101)."""

    def __init__(self, method: str = "sa", policy: str = "balanced", precision: str = "fp64",
                 require_smoother_certificate: bool = True, reorder: bool = True,
                 host_threads: int = 0, device: int = 0, strength_threshold: float = 0.25,
                 prolongator_filter: float = 0.0, filter_keeps_aggregate: bool = False,
                 smoother: str = "jacobi", smoother_fp32: str = "jacobi", chebyshev_degree: int = 3,
                 chebyshev_ratio: float = 30.0, chebyshev_degree_coarse: int = 0,
                 constant_null_space: bool = False, smoother_fp16_finest: bool = False):
        self._lib = _native.load()
        opt = AmgOptions()
        self._lib.cfdxhip_amg_options_default(C.byref(opt))
        opt.method = METHODS[method]
        opt.policy = POLICIES[policy]
        opt.precision = PRECISIONS[precision]
        opt.require_smoother_certificate = int(require_smoother_certificate)
        opt.reorder = int(reorder)
        opt.host_threads = host_threads
        opt.device = device
        opt.strength_threshold = strength_threshold
        opt.prolongator_filter = prolongator_filter
        opt.filter_keeps_aggregate = int(filter_keeps_aggregate)
        opt.smoother = SMOOTHERS[smoother]
        opt.smoother_fp32 = SMOOTHERS[smoother_fp32]
        opt.chebyshev_degree = chebyshev_degree
        opt.chebyshev_degree_coarse = chebyshev_degree_coarse
        opt.chebyshev_ratio = chebyshev_ratio
        opt.constant_null_space = int(constant_null_space)
        opt.smoother_fp16_finest = int(smoother_fp16_finest)
        h = C.c_void_p()
        st = self._lib.cfdxhip_amg_create(C.byref(opt), C.byref(h))
        if st != 0:
            raise RuntimeError(f"cfdxhip_amg_create failed with status {st}")
        self._h = h
        self.n = 0
        self.last_status = 0

    def __del__(self):
        h = getattr(self, "_h", None)
        if h:
            self._lib.cfdxhip_amg_destroy(h)
            self._h = None

    def last_error(self) -> str:
        return self._lib.cfdxhip_amg_last_error(self._h).decode()

    def _ok(self, st: int) -> bool:
        self.last_status = st
        return st == 0

    def setup(self, n, row_offsets, columns, values) -> bool:
        self.n = int(n)
        return self._ok(self._lib.cfdxhip_amg_setup(self._h, self.n, _u32(row_offsets), _u32(columns),
                                                    _f64(values)))

    def update_values(self, values) -> bool:
        return self._ok(self._lib.cfdxhip_amg_update_values(self._h, _f64(values)))

    # Device-pointer lifecycle (raw device addresses as ints or c_void_p).
    def setup_device(self, n, row_offsets_ptr, columns_ptr, values_ptr) -> bool:
        self.n = int(n)
        return self._ok(self._lib.cfdxhip_amg_setup_device(self._h, self.n, row_offsets_ptr, columns_ptr,
                                                           values_ptr))

    def update_values_device(self, values_ptr) -> bool:
        return self._ok(self._lib.cfdxhip_amg_update_values_device(self._h, values_ptr))

    def apply_device(self, r_ptr, z_ptr) -> bool:
        return self._ok(self._lib.cfdxhip_amg_apply_device(self._h, r_ptr, z_ptr))

    def update_seconds(self) -> float:
        v = C.c_double()
        self._lib.cfdxhip_amg_update_seconds(self._h, C.byref(v))
        return v.value

    def apply(self, r):
        z = np.empty(self.n, dtype=np.float64)
        if not self._ok(self._lib.cfdxhip_amg_apply(self._h, _f64(r), z)):
            return None
        return z

    def solve_cg(self, b, x, max_iter=1000, tolerance=1e-12) -> SolverResult:
        """x is updated in place (initial guess in, solution out)."""
        assert x.dtype == np.float64 and x.flags.c_contiguous
        res = Result()
        if not self._ok(self._lib.cfdxhip_amg_solve_cg(self._h, _f64(b), x, max_iter, tolerance, C.byref(res))):
            raise RuntimeError(self.last_error())
        return SolverResult.from_c(res)

    def solve_fgmres(self, b, x, restart=30, max_iter=1000, tolerance=1e-12) -> SolverResult:
        assert x.dtype == np.float64 and x.flags.c_contiguous
        res = Result()
        if not self._ok(self._lib.cfdxhip_amg_solve_fgmres(self._h, _f64(b), x, restart, max_iter, tolerance,
                                                           C.byref(res))):
            raise RuntimeError(self.last_error())
        return SolverResult.from_c(res)

    def solve_cg_projected(self, b, x, basis, max_iter=1000, tol=1e-12) -> SolverResult:
        """PCG with the null-space projector of `basis` (rows; cg_solver.h:
        653-667). x is updated in place."""
        basis = np.ascontiguousarray(np.atleast_2d(basis), dtype=np.float64)
        r = Result()
        st = self._lib.cfdxhip_amg_solve_cg_projected(self._h, _f64(b), x, max_iter, tol, basis, basis.shape[0],
                                                      C.byref(r))
        if st != 0:
            raise RuntimeError(f"status {st}: {self.last_error()}")
        return SolverResult.from_c(r)

    def solve_fgmres_learned(self, b, x, stage: "LearnedStage", restart=30, max_iter=1000,
                             tolerance=1e-12) -> SolverResult:
        """Mixed FGMRES with the learned stage ahead of the FP32 V-cycle."""
        assert x.dtype == np.float64 and x.flags.c_contiguous
        res = Result()
        st = self._lib.cfdxhip_amg_solve_fgmres_learned(self._h, stage._h, _f64(b), x, restart, max_iter, tolerance,
                                                        C.byref(res))
        if not self._ok(st):
            raise RuntimeError(self.last_error())
        return SolverResult.from_c(res)

    # ---- hierarchy introspection (reference ordering) ----
    def num_levels(self) -> int:
        v = C.c_size_t()
        self._lib.cfdxhip_amg_num_levels(self._h, C.byref(v))
        return v.value

    def level_info(self, level):
        n, nnz, pn = C.c_size_t(), C.c_size_t(), C.c_size_t()
        st = self._lib.cfdxhip_amg_level_info(self._h, level, C.byref(n), C.byref(nnz), C.byref(pn))
        if st != 0:
            raise IndexError(level)
        return n.value, nnz.value, pn.value

    def level_matrix(self, level):
        n, nnz, _ = self.level_info(level)
        rp = np.empty(n + 1, np.uint32)
        cols = np.empty(nnz, np.uint32)
        vals = np.empty(nnz, np.float64)
        self._lib.cfdxhip_amg_level_matrix(self._h, level, rp, cols, vals)
        return rp, cols, vals

    def level_transfer(self, level):
        n, _, pn = self.level_info(level)
        agg = np.empty(n, np.uint64)
        rp = np.empty(n + 1, np.uint32)
        cols = np.empty(pn, np.uint32)
        vals = np.empty(pn, np.float64)
        st = self._lib.cfdxhip_amg_level_transfer(self._h, level, agg, rp, cols, vals)
        if st != 0:
            raise IndexError(level)
        return agg, rp, cols, vals

    def level_kernel_seconds(self, level: int, precision: str = "fp64", kind: str = "spmv", repeat: int = 10):
        """Seconds per launch of a level's SpMV ("spmv") or fused Jacobi sweep
        ("jacobi"); precision "fp16": one Chebyshev step on the finest
        level's FP16 smoothing copy."""
        v = C.c_double()
        st = self._lib.cfdxhip_amg_level_kernel_seconds(self._h, level, {**PRECISIONS, "fp16": 2}[precision],
                                                        {"spmv": 0, "jacobi": 1}[kind], repeat, C.byref(v))
        if st != 0:
            raise RuntimeError(self.last_error())
        return v.value

    def gram_schmidt_seconds(self, j: int, repeat: int = 10):
        """(product pass, update pass) seconds per launch of FGMRES Arnoldi
        step j on the finest level's size (measurement only)."""
        d, u = C.c_double(), C.c_double()
        st = self._lib.cfdxhip_amg_gram_schmidt_seconds(self._h, j, repeat, C.byref(d), C.byref(u))
        if st != 0:
            raise RuntimeError(self.last_error())
        return d.value, u.value

    def coarse_end(self) -> int:
        """First level that the FP64 V-cycle runs in its single-launch coarse
        end (num_levels(): none)."""
        v = C.c_size_t()
        st = self._lib.cfdxhip_amg_coarse_end(self._h, C.byref(v))
        if st != 0:
            raise RuntimeError(f"cfdxhip_amg_coarse_end failed with status {st}")
        return v.value

    def level_spmv_format(self, level: int):
        """(format, stored_entries, slices) of the storage a level's device
        SpMV streams: "csr" (stored_entries = nnz) or "sell64" (slots of
        64-row slices, padding included)."""
        f, e, sl = C.c_uint32(), C.c_uint64(), C.c_uint64()
        st = self._lib.cfdxhip_amg_level_spmv_format(self._h, level, C.byref(f), C.byref(e), C.byref(sl))
        if st != 0:
            raise RuntimeError(f"cfdxhip_amg_level_spmv_format failed with status {st}")
        return ("csr", "sell64")[f.value], int(e.value), int(sl.value)

    def level_spmv_bytes(self, level: int, precision: str = "fp32") -> int:
        """Bytes one device SpMV of the level streams for the matrix (values,
        columns, offsets; x and y excluded), in the storage it uses
        ("fp16": the finest level's FP16 smoothing copy)."""
        v = C.c_uint64()
        st = self._lib.cfdxhip_amg_level_spmv_bytes(self._h, level, {**PRECISIONS, "fp16": 2}[precision],
                                                    C.byref(v))
        if st != 0:
            raise RuntimeError(f"cfdxhip_amg_level_spmv_bytes failed with status {st}")
        return int(v.value)

    def _check(self, st):
        if st != 0:
            raise RuntimeError(f"status {st}: {self.last_error()}")

    def configure_cf_interpolation_limit(self, max_entries: int):
        """C/F interpolation row cap, 0 or >= 2 (hypre_amg.h:51-54); a change
        drops the hierarchy (setup again)."""
        self._check(self._lib.cfdxhip_amg_configure_cf_interpolation_limit(self._h, max_entries))

    def cf_interpolation_limit(self) -> int:
        v = C.c_size_t()
        self._check(self._lib.cfdxhip_amg_cf_interpolation_limit(self._h, C.byref(v)))
        return int(v.value)

    def configure_max_coarsening_fraction(self, fraction: float):
        """Stop coarsening before a level keeping >= fraction of the unknowns
        (hypre_amg.h:55-58); [0.5, 1], 1 disables."""
        self._check(self._lib.cfdxhip_amg_configure_max_coarsening_fraction(self._h, fraction))

    def configure_bounded_nonsymmetric_action(self, max_image_ratio: float):
        """Bounded preconditioner action for nonsymmetric Krylov use
        (hypre_amg.h:59-63); 0 disables, else [1, 1e6]."""
        self._check(self._lib.cfdxhip_amg_configure_bounded_nonsymmetric_action(self._h, max_image_ratio))

    def bounded_action_fallbacks(self) -> int:
        v = C.c_uint64()
        self._check(self._lib.cfdxhip_amg_bounded_action_fallbacks(self._h, C.byref(v)))
        return int(v.value)

    def operator_complexity(self) -> float:
        return self._complexity()[0]

    def grid_complexity(self) -> float:
        return self._complexity()[1]

    def _complexity(self):
        a, b = C.c_double(), C.c_double()
        self._check(self._lib.cfdxhip_amg_complexity(self._h, C.byref(a), C.byref(b)))
        return a.value, b.value

    def prolongation_stats(self):
        """(first_prolongation_nnz, row_sum_min, row_sum_max) of the finest P."""
        n, lo, hi = C.c_uint64(), C.c_double(), C.c_double()
        self._check(self._lib.cfdxhip_amg_prolongation_stats(self._h, C.byref(n), C.byref(lo), C.byref(hi)))
        return int(n.value), lo.value, hi.value

    def counters(self):
        """(coarse_size, hierarchy_builds, numeric_updates), hypre_amg.h:72,86-87."""
        a, b, c = C.c_uint64(), C.c_uint64(), C.c_uint64()
        self._lib.cfdxhip_amg_counters(self._h, C.byref(a), C.byref(b), C.byref(c))
        return a.value, b.value, c.value

    def set_chebyshev(self, degree: int, ratio: float = 30.0, degree_coarse=None) -> bool:
        """New Chebyshev degree / ratio on a set-up hierarchy; degree_coarse
        (levels below the finest, 0 = degree) is kept when None."""
        if degree_coarse is None:
            self.last_status = self._lib.cfdxhip_amg_set_chebyshev(self._h, degree, ratio)
        else:
            self.last_status = self._lib.cfdxhip_amg_set_chebyshev_levels(self._h, degree, degree_coarse, ratio)
        return self.last_status == 0

    def level_lambda_max(self, level: int) -> float:
        v = C.c_double()
        st = self._lib.cfdxhip_amg_level_lambda_max(self._h, level, C.byref(v))
        if st != 0:
            raise RuntimeError(f"cfdxhip_amg_level_lambda_max failed with status {st}")
        return v.value

    def smoother_omega(self) -> float:
        v = C.c_double()
        self._lib.cfdxhip_amg_smoother_omega(self._h, C.byref(v))
        return v.value

    def setup_seconds(self):
        a, b = C.c_double(), C.c_double()
        self._lib.cfdxhip_amg_setup_seconds(self._h, C.byref(a), C.byref(b))
        return a.value, b.value


@dataclass
class Mesh:
    px: np.ndarray
    py: np.ndarray
    pz: np.ndarray
    face_offsets: np.ndarray
    face_vertices: np.ndarray
    owner: np.ndarray
    neighbour: np.ndarray
    cell_offsets: np.ndarray
    cell_faces: np.ndarray
    patch_of_face: np.ndarray
    patch_kind: np.ndarray
    cell_ijk: np.ndarray
    n_cells: int
    n_faces: int
    n_internal_faces: int
    n_patches: int


MESH_KINDS = {"box": 0, "extruded2d": 1, "channel_step": 2}


def generate_mesh(kind="box", nx=8, ny=8, nz=8, lx=1.0, ly=1.0, lz=1.0, jitter=0.0, wall_layers=0,
                  first_aspect=0.0, growth=0.0, step_height_fraction=0.0, step_length_fraction=0.0,
                  permute=False, seed=0) -> Mesh:
    """Synthetic unstructured hex mesh built by libcfdxhip's generator."""
    lib = _native.load()
    s = MeshSpec()
    s.kind = MESH_KINDS[kind]
    s.nx, s.ny, s.nz = nx, ny, nz
    s.lx, s.ly, s.lz = lx, ly, lz
    s.jitter = jitter
    s.wall_layers = wall_layers
    s.first_aspect = first_aspect
    s.growth = growth
    s.step_height_fraction = step_height_fraction
    s.step_length_fraction = step_length_fraction
    s.permute = int(permute)
    s.seed = seed
    h = C.c_void_p()
    st = lib.cfdxhip_mesh_generate(C.byref(s), C.byref(h))
    if st != 0:
        raise ValueError(f"mesh generation failed (status {st})")
    try:
        z = MeshSizes()
        lib.cfdxhip_mesh_sizes_get(h, C.byref(z))
        a = dict(
            px=np.empty(z.n_points, np.float64), py=np.empty(z.n_points, np.float64),
            pz=np.empty(z.n_points, np.float64), face_offsets=np.empty(z.n_faces + 1, np.uint32),
            face_vertices=np.empty(z.n_face_vertices, np.uint32), owner=np.empty(z.n_faces, np.uint32),
            neighbour=np.empty(z.n_faces, np.int32), cell_offsets=np.empty(z.n_cells + 1, np.uint32),
            cell_faces=np.empty(z.n_cell_faces, np.uint32), patch_of_face=np.empty(z.n_faces, np.uint32),
            patch_kind=np.empty(z.n_patches, np.uint8), cell_ijk=np.empty(3 * z.n_cells, np.uint32),
        )
        order = ["px", "py", "pz", "face_offsets", "face_vertices", "owner", "neighbour", "cell_offsets",
                 "cell_faces", "patch_of_face", "patch_kind", "cell_ijk"]
        lib.cfdxhip_mesh_copy(h, *[a[k].ctypes.data_as(C.c_void_p) for k in order])
    finally:
        lib.cfdxhip_mesh_destroy(h)
    return Mesh(**a, n_cells=int(z.n_cells), n_faces=int(z.n_faces), n_internal_faces=int(z.n_internal_faces),
                n_patches=int(z.n_patches))


def _ptr(a):
    return a.ctypes.data_as(C.c_void_p)


def gradient_gauss_device(phi, sx, sy, sz, owner, neighbour, volume, n_faces, n_cells, gx, gy, gz, stream=None):
    """Face-list Green-Gauss gradient on device pointers (ints or c_void_p):
    the drop-in for the reference's cfdx_cuda_gradient_gauss
    (runtime/gpu/cuda_kernels.cu:43-65). Raises on a bad index or HIP error."""
    st = _native.load().cfdxhip_gradient_gauss_device(phi, sx, sy, sz, owner, neighbour, volume, n_faces, n_cells,
                                                      gx, gy, gz, stream)
    if st != 0:
        raise RuntimeError(f"cfdxhip_gradient_gauss_device failed with status {st}")


def divergence_device(phi_face, owner, neighbour, n_faces, n_cells, div, stream=None):
    """Face-list divergence on device pointers: the drop-in for the
    reference's cfdx_cuda_divergence (runtime/gpu/cuda_kernels.cu:67-97)."""
    st = _native.load().cfdxhip_divergence_device(phi_face, owner, neighbour, n_faces, n_cells, div, stream)
    if st != 0:
        raise RuntimeError(f"cfdxhip_divergence_device failed with status {st}")


class FvMesh:
    """Device-resident mesh with the pressure-path face kernels (geometry,
    Green-Gauss gradient, mass flux, SIMPLE pressure assembly, Poisson
    assembly). Mirrors the data the reference's corrector consumes
    (physics/steady_incompressible_solver.h:8048-8181)."""

    def __init__(self, mesh: Mesh, device: int = 0):
        self._lib = _native.load()
        self.mesh = mesh
        self.keep = [np.ascontiguousarray(a) for a in (
            mesh.px, mesh.py, mesh.pz, mesh.face_offsets, mesh.face_vertices, mesh.owner, mesh.neighbour,
            mesh.cell_offsets, mesh.cell_faces, mesh.patch_of_face, mesh.patch_kind)]
        k = self.keep
        h = C.c_void_p()
        st = self._lib.cfdxhip_fv_create(device, len(mesh.px), _ptr(k[0]), _ptr(k[1]), _ptr(k[2]), mesh.n_faces,
                                         _ptr(k[3]), _ptr(k[4]), _ptr(k[5]), _ptr(k[6]), mesh.n_cells, _ptr(k[7]),
                                         _ptr(k[8]), mesh.n_patches, _ptr(k[9]), _ptr(k[10]), C.byref(h))
        if st != 0:
            raise RuntimeError(f"cfdxhip_fv_create failed with status {st}")
        self._h = h

    def __del__(self):
        h = getattr(self, "_h", None)
        if h:
            self._lib.cfdxhip_fv_destroy(h)
            self._h = None

    def last_error(self):
        return self._lib.cfdxhip_fv_last_error(self._h).decode()

    def _check(self, st):
        if st != 0:
            raise RuntimeError(f"status {st}: {self.last_error()}")

    def geometry(self):
        m = self.mesh
        fc = np.empty(3 * m.n_faces)
        fs = np.empty(3 * m.n_faces)
        cc = np.empty(3 * m.n_cells)
        vol = np.empty(m.n_cells)
        self._check(self._lib.cfdxhip_fv_geometry(self._h, _ptr(fc), _ptr(fs), _ptr(cc), _ptr(vol)))
        return fc, fs, cc, vol

    def gauss_gradient(self, bc_type, bc_value, p):
        g = np.empty(3 * self.mesh.n_cells)
        self._check(self._lib.cfdxhip_fv_gauss_gradient(self._h, np.ascontiguousarray(bc_type, np.uint8),
                                                        _f64(bc_value), _f64(p), g))
        return g

    def mass_flux(self, vbc_type, vbc_value, rho, U):
        phi = np.empty(self.mesh.n_faces)
        self._check(self._lib.cfdxhip_fv_mass_flux(self._h, np.ascontiguousarray(vbc_type, np.uint8),
                                                   _f64(vbc_value), rho, _f64(U), phi))
        return phi

    def pressure_pattern(self, pbc_type, reference_cell=0):
        n, nnz = C.c_size_t(), C.c_size_t()
        t = np.ascontiguousarray(pbc_type, np.uint8)
        self._check(self._lib.cfdxhip_fv_pressure_pattern(self._h, t, reference_cell, C.byref(n), C.byref(nnz),
                                                          None, None))
        rp = np.empty(n.value + 1, np.uint32)
        cols = np.empty(nnz.value, np.uint32)
        self._check(self._lib.cfdxhip_fv_pressure_pattern(self._h, t, reference_cell, C.byref(n), C.byref(nnz),
                                                          _ptr(rp), _ptr(cols)))
        return rp, cols

    def pressure_assemble(self, pbc_type, pbc_value, rho, rAU, phi, p, reference_cell=0):
        rp, cols = self.pressure_pattern(pbc_type, reference_cell)
        vals = np.empty(len(cols))
        rhs = np.empty(len(rp) - 1)
        self._check(self._lib.cfdxhip_fv_pressure_assemble(self._h, np.ascontiguousarray(pbc_type, np.uint8),
                                                           _f64(pbc_value), rho, _f64(rAU), _f64(phi), _f64(p),
                                                           reference_cell, vals, rhs))
        return rp, cols, vals, rhs

    # --------------------------------------------------- momentum side --
    def wls_gradient(self, bc_type, bc_value, field, condition_limit=1e8):
        """compute_boundary_aware_wls_gradient (physics/finite_volume_transport.h:606-715):
        (grad 3 x n, number of cells left at the Green-Gauss gradient)."""
        g = np.empty(3 * self.mesh.n_cells)
        fb = C.c_size_t()
        self._check(self._lib.cfdxhip_fv_wls_gradient(self._h, np.ascontiguousarray(bc_type, np.uint8),
                                                      _f64(bc_value), condition_limit, _f64(field), g,
                                                      C.byref(fb)))
        return g, fb.value

    def momentum_pattern(self):
        n, nnz = C.c_size_t(), C.c_size_t()
        self._check(self._lib.cfdxhip_fv_momentum_pattern(self._h, C.byref(n), C.byref(nnz), None, None))
        rp = np.empty(n.value + 1, np.uint32)
        cols = np.empty(nnz.value, np.uint32)
        self._check(self._lib.cfdxhip_fv_momentum_pattern(self._h, C.byref(n), C.byref(nnz), _ptr(rp), _ptr(cols)))
        return rp, cols

    def momentum_assemble(self, vbc_type, vbc_value, mu, phi, grad_p, body, U, bounded=True, alpha=1.0):
        """The SIMPLE predictor's relaxed momentum equations
        (steady_incompressible_solver.h:3262-3311, 3728-3770): one matrix for
        the three components. Returns (rowp, cols, vals, rhs (3 x n), diag)."""
        rp, cols = self.momentum_pattern()
        n = self.mesh.n_cells
        vals = np.empty(len(cols))
        rhs = np.empty(3 * n)
        diag = np.empty(n)
        body_arr = None if body is None else _f64(body)
        b = None if body_arr is None else _ptr(body_arr)
        self._check(self._lib.cfdxhip_fv_momentum_assemble(self._h, np.ascontiguousarray(vbc_type, np.uint8),
                                                           _f64(vbc_value), _f64(mu), _f64(phi), _f64(grad_p), b,
                                                           _f64(U), int(bool(bounded)), alpha, vals, rhs, diag))
        return rp, cols, vals, rhs, diag

    def momentum_hbya(self, vals, rhs, diag, grad_p, U):
        """rAU and HbyA (3 x n each): steady_incompressible_solver.h:7816-7836, 6430-6465."""
        n = self.mesh.n_cells
        rau = np.empty(3 * n)
        hbya = np.empty(3 * n)
        self._check(self._lib.cfdxhip_fv_momentum_hbya(self._h, _f64(vals), _f64(rhs), _f64(diag), _f64(grad_p),
                                                       _f64(U), rau, hbya))
        return rau, hbya

    def velocity_correct(self, hbya, rau, grad_p):
        U = np.empty(3 * self.mesh.n_cells)
        self._check(self._lib.cfdxhip_fv_velocity_correct(self._h, _f64(hbya), _f64(rau), _f64(grad_p), U))
        return U

    def rhie_chow_flux(self, vbc_type, vbc_value, pbc_type, pbc_value, rho, hbya, p, rau):
        """make_rhie_chow_mass_flux (steady_incompressible_solver.h:2063-2217)."""
        phi = np.empty(self.mesh.n_faces)
        self._check(self._lib.cfdxhip_fv_rhie_chow_flux(self._h, np.ascontiguousarray(vbc_type, np.uint8),
                                                        _f64(vbc_value), np.ascontiguousarray(pbc_type, np.uint8),
                                                        _f64(pbc_value), rho, _f64(hbya), _f64(p), _f64(rau), phi))
        return phi

    def diffusion_assemble(self, gamma, source, face_value, face_is_neumann):
        nnz = C.c_size_t()
        self._check(self._lib.cfdxhip_fv_diffusion_assemble(self._h, gamma, None, None, None, C.byref(nnz), None,
                                                            None, None, None))
        n = self.mesh.n_cells
        rp = np.empty(n + 1, np.uint32)
        cols = np.empty(nnz.value, np.uint32)
        vals = np.empty(nnz.value)
        rhs = np.empty(n)
        src = _f64(source)
        fv = _f64(face_value)
        fn = np.ascontiguousarray(face_is_neumann, np.uint8)
        self._check(self._lib.cfdxhip_fv_diffusion_assemble(self._h, gamma, _ptr(src), _ptr(fv), _ptr(fn),
                                                            C.byref(nnz), _ptr(rp), _ptr(cols), _ptr(vals),
                                                            _ptr(rhs)))
        return rp, cols, vals, rhs


class LearnedStage:
    """Message-passing network stage of mixed FGMRES (no reference
    counterpart): forward, backward, Adam and training run in libcfdxhip's HIP
    kernels on the graph of a set-up FP32 hierarchy."""

    def __init__(self, device: int = 0, params=None):
        self._lib = _native.load()
        h = C.c_void_p()
        st = self._lib.cfdxhip_mpnn_create(device, C.byref(h))
        if st != 0:
            raise RuntimeError(f"cfdxhip_mpnn_create failed with status {st}")
        self._h = h
        self.nparams = int(self._lib.cfdxhip_mpnn_param_count())
        if params is not None:
            self.set_params(params)

    def __del__(self):
        h = getattr(self, "_h", None)
        if h:
            self._lib.cfdxhip_mpnn_destroy(h)
            self._h = None

    def last_error(self) -> str:
        return (self._lib.cfdxhip_mpnn_last_error(self._h) or b"").decode()

    def _check(self, st):
        if st != 0:
            raise RuntimeError(f"status {st}: {self.last_error()}")

    @staticmethod
    def initial_params(seed: int = 0, out_scale: float = 0.1) -> np.ndarray:
        """Seeded initialisation (layout of cfdxhip_mpnn_param_count): w_in ~
        N(0, 1), layer weights ~ U(+-sqrt(6/96)/2), w_out ~ out_scale N(0, 1/32),
        biases 0. A small w_out starts the stage close to the plain V-cycle."""
        H, L = 32, 4
        stride = 2 * H * H + H
        off_out = 2 * H + L * stride
        rng = np.random.default_rng(seed)
        p = np.zeros(off_out + H + 1)
        p[0:H] = rng.standard_normal(H)
        lim = np.sqrt(6.0 / (3 * H)) / 2
        for l in range(L):
            o = 2 * H + l * stride
            p[o:o + 2 * H * H] = rng.uniform(-lim, lim, 2 * H * H)
        p[off_out:off_out + H] = out_scale * rng.standard_normal(H) / np.sqrt(H)
        return p.astype(np.float32)

    def set_params(self, p):
        p = np.ascontiguousarray(p, dtype=np.float32)
        self._check(self._lib.cfdxhip_mpnn_set_params(self._h, p, p.size))

    def get_params(self):
        p = np.empty(self.nparams, np.float32)
        self._check(self._lib.cfdxhip_mpnn_get_params(self._h, p, p.size))
        return p

    def forward(self, amg: NativeAMGPreconditioner, r):
        e = np.empty(amg.n)
        self._check(self._lib.cfdxhip_mpnn_forward(self._h, amg._h, _f64(r), e))
        return e

    def vjp(self, amg: NativeAMGPreconditioner, r, ge):
        g = np.empty(self.nparams, np.float32)
        self._check(self._lib.cfdxhip_mpnn_vjp(self._h, amg._h, _f64(r), _f64(ge), g))
        return g

    def adam_step(self, grad, lr):
        self._check(self._lib.cfdxhip_mpnn_adam_step(self._h, np.ascontiguousarray(grad, dtype=np.float32), lr))

    def collect_pairs(self, amg: NativeAMGPreconditioner, b, iterations, tol=1e-10):
        its = np.ascontiguousarray(iterations, dtype=np.uint64)
        got = C.c_uint32()
        res = Result()
        self._check(self._lib.cfdxhip_mpnn_collect_pairs(self._h, amg._h, _f64(b), its, len(its), tol,
                                                          C.byref(got), C.byref(res)))
        return got.value, SolverResult.from_c(res)

    def train(self, amg: NativeAMGPreconditioner, steps, lr):
        losses = np.empty(steps)
        self._check(self._lib.cfdxhip_mpnn_train(self._h, amg._h, steps, lr, losses))
        return losses

    def set_fallback(self, min_reduction=0.5, window=3):
        """Drop the stage once a residual reduction falls below min_reduction:
        the network's own, 1 - |r - A N(r)|/|r|, at any application, or
        FGMRES's per iteration over `window` iterations (negative: never)."""
        self._check(self._lib.cfdxhip_mpnn_set_fallback(self._h, min_reduction, window))


# ----------------------------------------------------- capture files --

PROBLEMS = {"general": 0, "pressure_poisson": 1, "diffusion": 2, "momentum": 3, "scalar_transport": 4,
            "coupled_pressure_velocity": 5}


@dataclass
class LinearSystemCapture:
    """One captured system (core/linalg/linear_system_capture.h:73-83)."""
    rowp: np.ndarray
    cols: np.ndarray
    vals: np.ndarray
    rhs: np.ndarray
    initial_solution: np.ndarray
    problem: int = 0
    null_space: int = 0
    scaling: int = 0
    max_iterations: int = 1000
    tolerance: float = 1e-12
    checksum: int = 0

    @property
    def n(self) -> int:
        return len(self.rowp) - 1


def read_capture(path) -> LinearSystemCapture:
    """Reads a .cfdxlin file (CFDX_LINEAR_REPLAY_V1); raises ValueError with
    the reader's reason when the file is rejected."""
    lib = _native.load()
    h = C.c_void_p()
    if lib.cfdxhip_capture_read(os.fsencode(path), C.byref(h)) != 0:
        raise ValueError((lib.cfdxhip_capture_last_error() or b"").decode())
    try:
        info = _native.CaptureInfo()
        lib.cfdxhip_capture_info_get(h, C.byref(info))
        n, nnz = info.n, info.nnz
        rp, cols = np.empty(n + 1, np.uint32), np.empty(nnz, np.uint32)
        vals, rhs, x0 = np.empty(nnz), np.empty(n), np.empty(n)
        lib.cfdxhip_capture_copy(h, rp, cols, vals, rhs, x0)
        return LinearSystemCapture(rp, cols, vals, rhs, x0, info.problem, info.null_space, info.scaling,
                                   info.max_iterations, info.tolerance, info.checksum)
    finally:
        lib.cfdxhip_capture_destroy(h)


def write_capture(path, cap: LinearSystemCapture) -> int:
    """Writes a .cfdxlin file; returns its checksum. Raises ValueError when
    the system fails the format's validation."""
    lib = _native.load()
    info = _native.CaptureInfo()
    info.n = cap.n
    info.nnz = len(cap.vals)
    info.max_iterations = cap.max_iterations
    info.problem, info.null_space, info.scaling = cap.problem, cap.null_space, cap.scaling
    info.tolerance = cap.tolerance
    out = C.c_uint64()
    st = lib.cfdxhip_capture_write(os.fsencode(path), C.byref(info), _u32(cap.rowp), _u32(cap.cols), _f64(cap.vals),
                                   _f64(cap.rhs), _f64(cap.initial_solution), C.byref(out))
    if st != 0:
        raise ValueError((lib.cfdxhip_capture_last_error() or b"").decode())
    return out.value
