"""Workloads whose time this library is judged by.

One case is one pass of work that a SIMPLE pressure-correction program asks
the library for, through the Python classes or the C ABI: assembling the
momentum and pressure equations, applying and refreshing the AMG
preconditioner, solving, correcting velocity and flux, the learned stage's
forward and backward pass, and the face-list operators. The meshes are the
project's own families (jittered, wall-clustered and natural-order boxes, the
channel with a step, the 2-D Poisson square) between 1.7K and 4M cells.

listed() are the fixed cases, draw() gives more of the same ranges.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import cfdx_dev_amd as cx
import cfdx_dev_amd.workloads as W
from cfdx_dev_amd import _native

# Mixed-precision settings of the benchmark and the replay tool.
MIXED = dict(precision="fp32", smoother_fp32="chebyshev", chebyshev_degree=9, chebyshev_degree_coarse=1,
             chebyshev_ratio=240.0, smoother_fp16_finest=True)
FILTERED = dict(prolongator_filter=0.2, filter_keeps_aggregate=True)


def listed():
    return [
        # The smallest call: one FP64 V-cycle on the smoke test's box, where
        # launches and synchronisations are everything.
        dict(name="vcycle64_box12", kind="vcycle", mesh="box", nx=12, ny=12, nz=12, precision="fp64"),
        # One FP64 V-cycle (the plain AMG-PCG's preconditioner, damped Jacobi)
        # on the channel mesh the learned stage is trained on; ragged rows.
        dict(name="vcycle64_channel", kind="vcycle", mesh="channel", nx=80, ny=32, nz=30, precision="fp64"),
        # One mixed V-cycle (FP32, Chebyshev, FP16 finest level) on a
        # wall-clustered box: what mixed FGMRES does every iteration.
        dict(name="vcycle_mixed_walls96", kind="vcycle", mesh="walls", nx=96, ny=96, nz=96, precision="mixed"),
        # Whole solve, small plain problem: 2-D Poisson, FP64 PCG to 1e-10 on
        # the classical C/F hierarchy, host vectors in and out.
        dict(name="pcg_poisson2d_128", kind="pcg2d", n=128),
        # Whole solve, mixed FGMRES(30) to 1e-8 on the channel.
        dict(name="fgmres_channel", kind="fgmres", mesh="channel", nx=80, ny=32, nz=30),
        # Numeric refresh of the hierarchy with a new corrector's matrix, then
        # the V-cycle that uses it.
        dict(name="refresh_channel", kind="refresh", mesh="channel", nx=120, ny=48, nz=44),
        # Pressure equation of one corrector on a randomly numbered 2.1M-cell
        # box, reference cell eliminated.
        dict(name="pressure_box128", kind="pressure", mesh="box", nx=128, ny=128, nz=128, permute=True),
        # The same on a locally numbered channel with a fixed-pressure outlet.
        dict(name="pressure_channel", kind="pressure", mesh="channel", nx=120, ny=48, nz=44, permute=False),
        # Three relaxed momentum equations on a randomly numbered jittered box.
        dict(name="momentum_box80", kind="momentum", mesh="box", nx=80, ny=81, nz=79, permute=True, bounded=True),
        # rAU / HbyA, velocity correction and Rhie-Chow flux after the solve.
        dict(name="correct_channel", kind="correct", mesh="channel", nx=160, ny=64, nz=58, permute=False),
        # Training side of the learned stage: estimate and parameter gradient.
        dict(name="learned_channel", kind="learned", mesh="channel", nx=80, ny=32, nz=30),
        # Face-list gradient and divergence on caller arrays, 4.1M cells.
        dict(name="face_ops_160", kind="face", nx=160, ny=160, nz=160),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["vcycle", "vcycle", "pcg2d", "fgmres", "refresh", "pressure", "pressure", "momentum",
                       "correct", "learned", "face"])
    if kind == "pcg2d":
        return dict(kind=kind, n=_log_int(rng, 20, 128))
    if kind == "face":
        a = _log_int(rng, 12, 150)
        return dict(kind=kind, nx=a, ny=a + rng.randrange(0, 10), nz=a + rng.randrange(0, 10))
    # Cells along y, up to the listed sizes; the channel is 3 x 1 x 1.
    box, channel = dict(vcycle=(88, 56), fgmres=(0, 31), refresh=(0, 47), pressure=(120, 70), momentum=(76, 56),
                        correct=(70, 60), learned=(0, 31))[kind]
    mesh = rng.choice(["box", "channel"]) if box else "channel"
    if kind == "vcycle" and rng.random() < 0.3:
        mesh = "walls"
    if mesh == "channel":
        a = _log_int(rng, 16, channel)
        c = dict(kind=kind, mesh=mesh, nx=2 * a + rng.randrange(0, a // 2), ny=a, nz=a - rng.randrange(0, 5))
    else:
        a = _log_int(rng, 12, box)
        c = dict(kind=kind, mesh=mesh, nx=a + rng.randrange(0, 8), ny=a, nz=a + rng.randrange(0, 8))
    if kind == "vcycle":
        c["precision"] = rng.choice(["fp64", "mixed"])
        if mesh == "walls":
            c["precision"] = "mixed"
    if kind in ("pressure", "momentum", "correct"):
        c["permute"] = rng.random() < 0.5
    if kind == "momentum":
        c["bounded"] = rng.random() < 0.7
    return c


# ------------------------------------------------------------------ inputs --

def _mesh(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    permute = case.get("permute", True)
    if case["mesh"] == "channel":
        return cx.generate_mesh("channel_step", nx, ny, nz, lx=3.0, first_aspect=500.0, growth=1.15,
                                step_height_fraction=1.0 / 3.0, step_length_fraction=0.25, permute=permute,
                                seed=seed % 100000)
    if case["mesh"] == "walls":
        return cx.generate_mesh("box", nx, ny, nz, jitter=0.10, permute=permute, seed=seed % 100000,
                                wall_layers=max(1, round(30 * ny / 256)), first_aspect=1000.0)
    return cx.generate_mesh("box", nx, ny, nz, jitter=0.15, permute=permute, seed=seed % 100000)


def _boundary(case, m):
    """(velocity types, velocity values, pressure types, pressure values) per
    patch: a lid-driven box, or the channel with inlet, walls and a
    fixed-pressure outlet."""
    vt = np.ones(m.n_patches, np.uint8)
    vv = np.zeros(3 * m.n_patches)
    pt = np.zeros(m.n_patches, np.uint8)
    pv = np.zeros(m.n_patches)
    if case["mesh"] == "channel":
        vv[0:3] = [1.0, 0.0, 0.0]
        vt[1] = 0
        pt[1] = 1
    else:
        vv[9:12] = [1.0, 0.0, 0.0]
    return vt, vv, pt, pv


def _fields(case, m, seed):
    """Cell fields of a corrector: smooth velocity, pressure and pressure
    gradient plus a little noise, log-normal 1/a_P (its scale leaves the
    matrix diagonal near one), viscosity, and a face flux near U.S."""
    rng = np.random.default_rng([seed, 17])
    n = m.n_cells
    ijk = m.cell_ijk.reshape(-1, 3)
    x = (ijk + 0.5) / np.asarray([case["nx"], case["ny"], case["nz"]], dtype=float)

    def smooth(count, mean):
        out = np.full(n, float(mean))
        for _ in range(count):
            k = rng.integers(1, 5, size=3)
            out += rng.normal() / float(k @ k) * np.sin(2.0 * math.pi * (x @ k) + rng.uniform(0.0, 2.0 * math.pi))
        return out + 0.01 * rng.standard_normal(n)

    U = np.concatenate([smooth(4, 1.0), smooth(4, 0.0), smooth(4, 0.0)])
    p = smooth(4, 0.0)
    gp = np.concatenate([smooth(2, 0.0) for _ in range(3)])
    sigma = rng.uniform(0.5, 1.5)
    rau = np.repeat((float(n) ** (-1.0 / 3.0) * np.exp(sigma * (smooth(6, 0.0) - 0.5)))[None], 3, 0).ravel()
    mu = 1e-3 * np.exp(0.3 * smooth(2, 0.0))
    noise = rng.standard_normal(m.n_faces)
    return dict(U=U, p=p, gp=gp, rau=rau, mu=mu, noise=noise)


def _system(case, seed):
    """A pressure matrix and right-hand side of the case's family, as the
    corrector hands them to the solver."""
    dims = (case["nx"], case["ny"], case["nz"])
    m = _mesh(case, seed)
    if case["mesh"] == "channel":
        return W.c3_channel(seed % 400, dims=dims, seed=seed % 100000, mesh=m)
    fv = cx.FvMesh(m)
    g = W.correlated_gaussian(m, dims, max(2.0, min(dims) / 16.0), seed % 100000 + 1)
    rau = np.repeat(np.exp((1.5 if case["mesh"] == "walls" else 1.0) * g)[None], 3, 0).ravel()
    pt, pv = np.zeros(m.n_patches, np.uint8), np.zeros(m.n_patches)
    zf, zc = np.zeros(m.n_faces), np.zeros(m.n_cells)
    rp, cols = fv.pressure_pattern(pt, 0)
    rows = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    _, _, vals, _ = fv.pressure_assemble(pt, pv, 1.0, rau, zf, zc, 0)
    scale = 1.0 / vals[cols == rows].mean()
    b = np.random.default_rng([seed, 2]).standard_normal(m.n_cells)
    b -= b.mean()
    # The coefficients are linear in 1/a_P, so the unit-mean-diagonal system
    # is the scaled one.
    return W.PressureSystem("case", m, len(rp) - 1, rp, cols, vals * scale, np.ascontiguousarray(b[1:]), rau * scale,
                            dict(fv=fv))


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda")


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _check(ok, what):
    if not ok:
        raise RuntimeError(what)


def _amg(s, **opt):
    h = cx.NativeAMGPreconditioner(method="sa", **opt)
    _check(h.setup(s.n, s.rowp, s.cols, s.vals), h.last_error())
    return h


def _lattice_faces(nx, ny, nz):
    """Internal and boundary faces of an nx x ny x nz lattice: owner,
    neighbour (-1 outside) and axis of the normal, internal faces first."""
    cell = np.arange(nx * ny * nz, dtype=np.int64).reshape(nz, ny, nx)
    own, nei, axis, side = [], [], [], []
    for ax, (lo, hi) in enumerate((((slice(None), slice(None), slice(0, -1)), (slice(None), slice(None), slice(1, None))),
                                   ((slice(None), slice(0, -1)), (slice(None), slice(1, None))),
                                   ((slice(0, -1),), (slice(1, None),)))):
        a, b = cell[lo].ravel(), cell[hi].ravel()
        own.append(a), nei.append(b), axis.append(np.full(a.size, ax, np.int8)), side.append(np.ones(a.size))
    for ax, sel in enumerate(((slice(None), slice(None)), (slice(None),), ())):
        for sgn, at in ((-1.0, 0), (1.0, -1)):
            a = cell[sel + (at,)].ravel()
            own.append(a), nei.append(np.full(a.size, -1)), axis.append(np.full(a.size, ax, np.int8))
            side.append(np.full(a.size, sgn))
    own, nei, axis, side = (np.concatenate(v) for v in (own, nei, axis, side))
    order = np.lexsort((nei, own, nei < 0))
    return own[order], nei[order], axis[order], side[order]


def _face_inputs(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    own, nei, axis, side = _lattice_faces(nx, ny, nz)
    rng = np.random.default_rng([seed, 5])
    nf, nc = len(own), nx * ny * nz
    h = 1.0 / nx
    s = rng.normal(0.0, 0.05 * h * h, size=(3, nf))
    s[axis, np.arange(nf)] += side * h * h
    vol = h ** 3 * rng.uniform(0.8, 1.2, nc)
    phi = rng.standard_normal(nc)
    flux = rng.standard_normal(nf) * h * h
    return dict(phi=phi, sx=s[0], sy=s[1], sz=s[2], owner=own.astype(np.uint32), neighbour=nei.astype(np.int64),
                volume=vol, flux=flux)


def _learned_ge(r, rng):
    """Gradient of the training loss at a small estimate: -A e / (e.r) is
    about -r, up to its scale."""
    return -r * (1.0 + 0.1 * rng.standard_normal(len(r)))


def _poisson2d_source(case, seed):
    return np.random.default_rng([seed, 3]).standard_normal(case["n"] ** 2)


# ----------------------------------------------------------------- prepare --

def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    lib = _native.load()
    if kind in ("vcycle", "fgmres", "refresh", "learned"):
        s = _system(case, seed)
        rng = np.random.default_rng([seed, 7])
        if kind == "vcycle":
            opt = dict(MIXED, **FILTERED) if case["precision"] == "mixed" else (
                FILTERED if case["mesh"] == "channel" else {})
            st["h"] = _amg(s, **opt)
            st["r"] = _dev(rng.standard_normal(s.n))
            st["z"] = torch.empty(s.n, dtype=torch.float64, device="cuda")
        elif kind == "fgmres":
            st["h"] = _amg(s, **MIXED, **FILTERED)
            st["b"] = _dev(s.b)
            st["x"] = torch.empty(s.n, dtype=torch.float64, device="cuda")
        elif kind == "refresh":
            st["h"] = _amg(s, **MIXED, **FILTERED)
            # The next corrector's matrix: 1/a_P moved by a few percent.
            rows = np.repeat(np.arange(s.n), np.diff(s.rowp))
            d = np.exp(0.05 * rng.standard_normal(s.n))
            st["vals"] = _dev(s.vals * d[rows] * d[s.cols])
            st["r"] = _dev(rng.standard_normal(s.n))
            st["z"] = torch.empty(s.n, dtype=torch.float64, device="cuda")
        else:
            st["h"] = _amg(s, precision="fp32", smoother_fp32="chebyshev", **FILTERED)
            st["net"] = cx.LearnedStage(params=cx.LearnedStage.initial_params(seed % 100000, out_scale=1.0))
            st["r"] = s.b + 0.1 * np.linalg.norm(s.b) / math.sqrt(s.n) * rng.standard_normal(s.n)
            st["ge"] = _learned_ge(st["r"], rng)
    elif kind == "pcg2d":
        n = case["n"]
        m = cx.generate_mesh("extruded2d", n, n, 1)
        fv = cx.FvMesh(m)
        fval = np.full(m.n_faces, np.nan)
        outer = np.arange(m.n_internal_faces, m.n_faces)
        fval[outer[m.patch_kind[m.patch_of_face[outer]] != 1]] = 0.0
        rp, cols, vals, rhs = fv.diffusion_assemble(1.0, _poisson2d_source(case, seed), fval,
                                                    np.zeros(m.n_faces, np.uint8))
        # The reference's default hierarchy; smoothed aggregation fills in here.
        h = cx.NativeAMGPreconditioner(method="boomer")
        _check(h.setup(len(rp) - 1, rp, cols, vals), h.last_error())
        st.update(h=h, b=rhs)
    elif kind in ("pressure", "momentum", "correct"):
        m = _mesh(case, seed)
        fv = cx.FvMesh(m)
        f = _fields(case, m, seed)
        vt, vv, pt, pv = _boundary(case, m)
        phi = fv.mass_flux(vt, vv, 1.0, f["U"])
        phi = phi * (1.0 + 0.01 * f["noise"])
        st.update(fv=fv, lib=lib, vt=vt, vv=vv, pt=pt, pv=pv, n=m.n_cells, nf=m.n_faces)
        for k in ("U", "p", "gp", "rau", "mu"):
            st[k] = _dev(f[k])
        st["phi"] = _dev(phi)
        n = m.n_cells
        f64 = dict(dtype=torch.float64, device="cuda")
        if kind == "pressure":
            rp, cols = fv.pressure_pattern(pt, 0)
            st["vals"] = torch.empty(len(cols), **f64)
            st["rhs"] = torch.empty(len(rp) - 1, **f64)
        else:
            rp, cols = fv.momentum_pattern()
            st["vals"] = torch.empty(len(cols), **f64)
            st["rhs"], st["diag"] = torch.empty(3 * n, **f64), torch.empty(n, **f64)
            if kind == "correct":
                # The assembled momentum system the predictor left behind.
                _momentum(st, True)
                st["rauo"], st["hbya"] = torch.empty(3 * n, **f64), torch.empty(3 * n, **f64)
                st["Unew"], st["phinew"] = torch.empty(3 * n, **f64), torch.empty(m.n_faces, **f64)
    elif kind == "face":
        f = _face_inputs(case, seed)
        st.update({k: _dev(v) if v.dtype != np.uint32 else _dev(v.view(np.int32)) for k, v in f.items()})
        nc = len(f["phi"])
        st["g"] = [torch.empty(nc, dtype=torch.float64, device="cuda") for _ in range(3)]
        st["div"] = torch.empty(nc, dtype=torch.float64, device="cuda")
        st.update(n=nc, nf=len(f["owner"]))
    torch.cuda.synchronize()
    return st


def _momentum(st, bounded):
    fv = st["fv"]
    e = st["lib"].cfdxhip_fv_momentum_assemble_device(
        fv._h, st["vt"], st["vv"], _ptr(st["mu"]), _ptr(st["phi"]), _ptr(st["gp"]), None, _ptr(st["U"]),
        int(bounded), 0.7, _ptr(st["vals"]), _ptr(st["rhs"]), _ptr(st["diag"]))
    _check(e == 0, fv.last_error())


# --------------------------------------------------------------------- run --

def run(state):
    st = state
    case = st["case"]
    kind = case["kind"]
    if kind == "vcycle":
        _check(st["h"].apply_device(_ptr(st["r"]), _ptr(st["z"])), st["h"].last_error())
        return st["z"]
    if kind == "fgmres":
        h = st["h"]
        st["x"].zero_()
        res = _native.Result()
        e = h._lib.cfdxhip_amg_solve_fgmres_device(h._h, _ptr(st["b"]), _ptr(st["x"]), 30, 1000, 1e-8,
                                                   ctypes.byref(res))
        _check(e == 0 and res.status == 0, h.last_error())
        return st["x"]
    if kind == "refresh":
        h = st["h"]
        _check(h.update_values_device(_ptr(st["vals"])), h.last_error())
        _check(h.apply_device(_ptr(st["r"]), _ptr(st["z"])), h.last_error())
        return st["z"]
    if kind == "learned":
        return st["net"].forward(st["h"], st["r"]), st["net"].vjp(st["h"], st["r"], st["ge"])
    if kind == "pcg2d":
        x = np.zeros(len(st["b"]))
        res = st["h"].solve_cg(st["b"], x, 1000, 1e-10)
        _check(res.status == 0, "PCG did not converge")
        return x
    if kind == "face":
        cx.gradient_gauss_device(_ptr(st["phi"]), _ptr(st["sx"]), _ptr(st["sy"]), _ptr(st["sz"]), _ptr(st["owner"]),
                                 _ptr(st["neighbour"]), _ptr(st["volume"]), st["nf"], st["n"],
                                 *[_ptr(g) for g in st["g"]])
        cx.divergence_device(_ptr(st["flux"]), _ptr(st["owner"]), _ptr(st["neighbour"]), st["nf"], st["n"],
                             _ptr(st["div"]))
        return (*st["g"], st["div"])
    fv, lib = st["fv"], st["lib"]
    if kind == "pressure":
        e = lib.cfdxhip_fv_pressure_assemble_device(fv._h, st["pt"], st["pv"], 1.0, _ptr(st["rau"]), _ptr(st["phi"]),
                                                    _ptr(st["p"]), 0, _ptr(st["vals"]), _ptr(st["rhs"]))
        _check(e == 0, fv.last_error())
        return st["vals"], st["rhs"]
    if kind == "momentum":
        _momentum(st, case["bounded"])
        return st["vals"], st["rhs"], st["diag"]
    # correct: the corrector's steps around the pressure solve, whose pressure
    # and pressure gradient are in hand.
    e = lib.cfdxhip_fv_momentum_hbya_device(fv._h, _ptr(st["vals"]), _ptr(st["rhs"]), _ptr(st["diag"]),
                                            _ptr(st["gp"]), _ptr(st["U"]), _ptr(st["rauo"]), _ptr(st["hbya"]))
    e = e or lib.cfdxhip_fv_rhie_chow_flux_device(fv._h, st["vt"], st["vv"], st["pt"], st["pv"], 1.0,
                                                  _ptr(st["hbya"]), _ptr(st["p"]), _ptr(st["rauo"]),
                                                  _ptr(st["phinew"]))
    e = e or lib.cfdxhip_fv_velocity_correct_device(fv._h, _ptr(st["hbya"]), _ptr(st["rauo"]), _ptr(st["gp"]),
                                                    _ptr(st["Unew"]))
    _check(e == 0, fv.last_error())
    return st["rauo"], st["hbya"], st["phinew"], st["Unew"]


# -------------------------------------------------------------------- work --

def _cells(case):
    n = case["nx"] * case["ny"] * case["nz"]
    if case.get("mesh") == "channel":
        n = int(n * (1.0 - 0.25 * 0.5))  # the step takes a quarter of the length, about half of the y cells
    return n


def work(case):
    """Inputs read once and outputs written once, and operations. Meshes:
    cells n, faces about 3 n, 7 matrix entries a row; a hierarchy is about
    twice its finest matrix."""
    kind = case["kind"]
    if kind == "pcg2d":
        n = case["n"] ** 2  # about 10 iterations of 14 passes over 5-point rows
        return dict(bytes=n * (2 * 5 * 12 + 16.0), flops=10 * 14 * 2 * n * 10.0)
    n = _cells(case)
    nf, nnz = 3 * n, 7 * n
    if kind == "face":
        return dict(bytes=nf * (24 + 12 + 8 + 12) + n * (8 + 8 + 24 + 8.0), flops=nf * 12.0)
    if kind == "pressure":
        # 1/a_P, p, centres, volumes; face vectors, flux, addressing; matrix and right-hand side
        return dict(bytes=n * (24 + 8 + 24 + 8 + 8) + nf * (24 + 8 + 8) + nnz * 8.0, flops=nf * 90.0)
    if kind == "momentum":
        return dict(bytes=n * (24 + 24 + 8 + 24 + 8 + 24 + 8) + nf * (24 + 8 + 8 + 24) + nnz * 8.0,
                    flops=nf * 200.0 + n * 300.0)
    if kind == "correct":
        # HbyA from the matrix; flux from HbyA, p, rAU; velocity
        return dict(bytes=nnz * 12 + n * (24 * 3 + 8 * 2 + 24 * 2) + nf * (24 + 8 + 8) + n * (24 * 2 + 40) + n * 96.0,
                    flops=nnz * 6 + nf * 100.0)
    if kind == "learned":
        # 4 layers forward twice, once backward: 64 x 32 products
        return dict(bytes=nnz * 8 + n * (2 * 8 + 8 + 4.0), flops=n * (2 * 4 + 2 * 4) * 2 * 64 * 32.0)
    if kind == "refresh":
        # matrix in, two Galerkin products a level, every copy out; 20 Lanczos steps
        return dict(bytes=nnz * (8 + 2 * (8 + 4 + 2)) + n * 16.0, flops=nnz * 2 * (20 * 2 + 60.0))
    passes = 17 if kind == "fgmres" or case["precision"] == "mixed" else 12
    if kind == "fgmres":  # about 15 iterations
        return dict(bytes=nnz * (12 + 4 + 8) + n * 16.0, flops=15 * (passes + 2) * nnz * 2.0)
    return dict(bytes=nnz * 2 * (12.0 if passes == 12 else 6.0) + n * 16, flops=passes * 2 * nnz * 2.0)


def tolerance(case):
    kind = case["kind"]
    if kind == "face":
        return dict(rel=1e-14)  # six FP64 terms a cell; seen 1.5e-16
    if kind == "pressure":
        return dict(rel=5e-14)  # FP64; seen 1.2e-14
    if kind in ("momentum", "correct"):
        return dict(rel=4e-12)  # FP64; thin wall cells cancel four digits: seen 1.0e-12
    if kind in ("vcycle", "refresh"):
        # FP32 sums in another order (another row numbering): seen 3.2e-6
        return dict(rel=1e-12) if case.get("precision") == "fp64" else dict(rel=1.5e-5)
    if kind == "learned":
        return dict(rel=2e-2)  # BF16 states and products: seen 5e-3 on the estimate
    if kind == "pcg2d":
        return dict(rel=6e-10)  # stops at a residual of 1e-10: seen 1.4e-10
    return dict(rel=2e-5)  # stops at a residual of 1e-8: seen 6e-6 on the worst-conditioned channel


# ------------------------------------------------------------------- exact --

def _bincount3(idx, v, n):
    return np.stack([np.bincount(idx, v[:, k], n) for k in range(3)], 1)


def _geometry(m):
    """Face centres, area vectors (out of the owner), cell centres, volumes:
    quadrilateral faces as triangle fans, cells from their faces."""
    pts = np.stack([m.px, m.py, m.pz], 1)
    v = pts[m.face_vertices.reshape(-1, 4)]
    S = np.zeros((m.n_faces, 3))
    wc = np.zeros_like(S)
    tri = np.zeros(m.n_faces)
    for a, b in ((1, 2), (2, 3)):
        t = 0.5 * np.cross(v[:, a] - v[:, 0], v[:, b] - v[:, 0])
        ta = np.linalg.norm(t, axis=1)
        S += t
        wc += (v[:, 0] + v[:, a] + v[:, b]) * (ta / 3.0)[:, None]
        tri += ta
    fc = wc / tri[:, None]
    n, ni = m.n_cells, m.n_internal_faces
    o, nb = m.owner.astype(np.int64), m.neighbour[:ni].astype(np.int64)
    area = np.linalg.norm(S, axis=1)
    den = np.bincount(o, area, n) + np.bincount(nb, area[:ni], n)
    cc = (_bincount3(o, fc * area[:, None], n) + _bincount3(nb, (fc * area[:, None])[:ni], n)) / den[:, None]
    d = np.where(np.arange(m.n_faces)[:, None] < ni, 0.0, fc) - cc[o]
    d[:ni] += cc[nb]
    S = np.where((np.einsum("ij,ij->i", S, d) < 0.0)[:, None], -S, S)
    vol = np.bincount(o, np.einsum("ij,ij->i", fc - cc[o], S), n)
    vol -= np.bincount(nb, np.einsum("ij,ij->i", fc[:ni] - cc[nb], S[:ni]), n)
    return fc, S, cc, np.abs(vol) / 3.0, o, nb


def _green_gauss(m, geo, pt, pv, p):
    fc, S, cc, vol, o, nb = geo
    ni, n = m.n_internal_faces, m.n_cells
    do = np.linalg.norm(fc[:ni] - cc[o[:ni]], axis=1)
    dn = np.linalg.norm(fc[:ni] - cc[nb], axis=1)
    w = dn / (do + dn)
    vf = np.empty(m.n_faces)
    vf[:ni] = w * p[o[:ni]] + (1.0 - w) * p[nb]
    pp = m.patch_of_face[ni:].astype(np.int64)
    vf[ni:] = np.where(pt[pp] == 1, pv[pp], p[o[ni:]])
    t = S * vf[:, None]
    return (_bincount3(o, t, n) - _bincount3(nb, t[:ni], n)) / vol[:, None]


def _face_pressure(m, geo, pt, pv, rau, p, g):
    """Orthogonal coefficient and Rhie-Chow pressure flux of every face (zero
    on boundary faces without a fixed pressure), rho = 1, weights 1/2."""
    fc, S, cc, vol, o, nb = geo
    ni = m.n_internal_faces
    pp = m.patch_of_face[ni:].astype(np.int64)
    fixed = pt[pp] == 1
    dA = rau.reshape(3, -1).T * vol[:, None]
    d = fc - cc[o]
    d[:ni] = cc[nb] - cc[o[:ni]]
    D = dA[o].copy()
    D[:ni] = 0.5 * (D[:ni] + dA[nb])
    G = g[o].copy()
    G[:ni] = 0.5 * (G[:ni] + g[nb])
    dp = np.zeros(m.n_faces)
    dp[:ni] = p[nb] - p[o[:ni]]
    dp[ni:] = pv[pp] - p[o[ni:]]
    dist = np.linalg.norm(d, axis=1)
    e = d / dist[:, None]
    oa = np.einsum("ij,ij->i", S, e)
    rfn = (D * e * e).sum(1)
    coef = rfn * oa / dist
    flux = coef * dp + (D * G * S).sum(1) - rfn * np.einsum("ij,ij->i", G, e) * oa
    on = np.ones(m.n_faces, bool)
    on[ni:] = fixed
    return np.where(on, coef, 0.0), np.where(on, flux, 0.0), on


def _csr_order(n, o, nb):
    rows = np.concatenate([np.arange(n), o, nb])
    cols = np.concatenate([np.arange(n), nb, o])
    return np.argsort(rows * n + cols, kind="stable"), rows, cols


def _mass_flux(m, geo, vt, vv, U):
    fc, S, cc, vol, o, nb = geo
    ni = m.n_internal_faces
    Uc = U.reshape(3, -1).T
    Uf = Uc[o].copy()
    Uf[:ni] = 0.5 * (Uf[:ni] + Uc[nb])
    pp = m.patch_of_face[ni:].astype(np.int64)
    Uf[ni:] = np.where((vt[pp] == 1)[:, None], vv.reshape(-1, 3)[pp], Uf[ni:])
    f = np.einsum("ij,ij->i", Uf, S)
    f[ni:][m.patch_kind[pp] != 0] = 0.0
    return f


def _momentum_exact(m, geo, vt, vv, f, phi, bounded, alpha):
    fc, S, cc, vol, o, nb = geo
    ni, n = m.n_internal_faces, m.n_cells
    oi = o[:ni]
    pp = m.patch_of_face[ni:].astype(np.int64)
    fixed = vt[pp] == 1
    vb = vv.reshape(-1, 3)[pp]
    U, mu = f["U"].reshape(3, -1).T, f["mu"]
    # Inverse-distance weighted least-squares gradients of U; a zero-gradient
    # boundary face adds the sample (normal projection, own value).
    area = np.linalg.norm(S, axis=1)
    nrm = S / area[:, None]
    nd = np.einsum("ij,ij->i", fc - cc[o], nrm)
    M = np.zeros((n, 3, 3))
    R = np.zeros((n, 3, 3))
    d = cc[nb] - cc[oi]
    dU = U[nb] - U[oi]
    db = np.where(fixed[:, None], (fc - cc[o])[ni:], nrm[ni:] * nd[ni:, None])
    dUb = np.where(fixed[:, None], vb - U[o[ni:]], 0.0)
    for a in range(3):
        for b in range(3):
            w = d[:, a] * d[:, b] / (d * d).sum(1)
            M[:, a, b] = np.bincount(oi, w, n) + np.bincount(nb, w, n) + np.bincount(
                o[ni:], db[:, a] * db[:, b] / (db * db).sum(1), n)
            w = d[:, a] * dU[:, b] / (d * d).sum(1)
            R[:, a, b] = np.bincount(oi, w, n) + np.bincount(nb, w, n) + np.bincount(
                o[ni:], db[:, a] * dUb[:, b] / (db * db).sum(1), n)
    grad = np.linalg.solve(M, R)  # [cell, direction, component]
    # Diffusion, upwind convection and the tangential diffusion flux per face.
    # The area vector splits as alpha d + tangential, alpha = |S|^2 / (S.d).
    dist = fc - cc[o]
    dist[:ni] = d
    sd = np.einsum("ij,ij->i", S, dist)
    al = area * area / sd
    tang = S - dist * al[:, None]
    tang[np.linalg.norm(tang, axis=1) <= 1e-12 * area] = 0.0
    do = np.abs(np.einsum("ij,ij->i", fc - cc[o], S)) / area
    dn = np.abs(np.einsum("ij,ij->i", (cc[nb] - fc[:ni]), S[:ni])) / area[:ni]
    D = np.empty(m.n_faces)
    D[:ni] = area[:ni] / (do[:ni] / mu[oi] + dn / mu[nb])
    D[ni:] = mu[o[ni:]] * area[ni:] / do[ni:]
    w = 1.0 - np.clip(np.einsum("ij,ij->i", (fc - cc[o])[:ni], d) / (d * d).sum(1), 0.0, 1.0)
    gf = grad[o].copy()
    gf[:ni] = gf[:ni] * w[:, None, None] + grad[nb] * (1.0 - w)[:, None, None]
    gam = mu[o].copy()
    gam[:ni] = D[:ni] / al[:ni]
    nof = gam[:, None] * np.einsum("fdc,fd->fc", gf, tang)
    bnd = np.zeros(m.n_faces, bool)
    bnd[ni:] = fixed
    nof[ni:][~fixed] = 0.0
    t_on = np.where(bnd | (np.arange(m.n_faces) < ni), D + np.maximum(phi, 0.0),
                    phi if bounded else np.maximum(phi, 0.0))
    t_no = np.where(bnd | (np.arange(m.n_faces) < ni), D + np.maximum(-phi, 0.0), 0.0)
    diag = np.bincount(o, t_on, n) + np.bincount(nb, t_no[:ni], n)
    div = np.bincount(o, phi, n) - np.bincount(nb, phi[:ni], n)
    rhs = _bincount3(o, nof, n) - _bincount3(nb, nof[:ni], n)
    rhs += _bincount3(o[ni:], np.where(fixed[:, None], t_no[ni:, None] * vb, 0.0), n)
    if bounded:
        diag = diag - div
    else:
        back = ~fixed & (phi[ni:] < 0.0)
        rhs -= _bincount3(o[ni:], np.where(back[:, None], phi[ni:, None] * U[o[ni:]], 0.0), n)
    rhs -= f["gp"].reshape(3, -1).T * vol[:, None]
    added = diag * (1.0 / alpha - 1.0)
    diag = diag + added
    rhs += added[:, None] * U
    order, rows, cols = _csr_order(n, oi, nb)
    vals = np.concatenate([diag, -t_no[:ni], -t_on[:ni]])[order]
    return vals, np.ascontiguousarray(rhs.T).ravel(), diag, rows[order], cols[order]


def _mpnn_exact(case, seed):
    """The message-passing network in float64 without BF16 rounding, and the
    gradient of sum ge e with respect to its parameters."""
    s = _system(case, seed)
    rng = np.random.default_rng([seed, 7])
    r = s.b + 0.1 * np.linalg.norm(s.b) / math.sqrt(s.n) * rng.standard_normal(s.n)
    ge = torch.from_numpy(_learned_ge(r, rng))
    p = torch.from_numpy(cx.LearnedStage.initial_params(seed % 100000, out_scale=1.0).astype(np.float64))
    p.requires_grad_(True)
    rows = np.repeat(np.arange(s.n), np.diff(s.rowp))
    cols = s.cols.astype(np.int64)
    on = rows == cols
    diag = np.empty(s.n)
    diag[rows[on]] = s.vals[on]
    sc = 1.0 / np.sqrt(diag)
    w = -s.vals[~on] * sc[rows[~on]] * sc[cols[~on]]
    i, j, w, sc = (torch.from_numpy(a) for a in (rows[~on], cols[~on], w, sc))
    u = torch.from_numpy(r) * sc
    rho = torch.sqrt((u * u).mean())
    H = 32
    h = torch.relu((u / rho)[:, None] * p[:H] + p[H:2 * H])
    for l in range(4):
        o = 2 * H + l * (2 * H * H + H)
        mix = torch.zeros_like(h).index_add(0, i, w[:, None] * h[j])
        h = torch.relu(torch.cat([h, mix], 1) @ p[o:o + 2 * H * H].reshape(2 * H, H) + p[o + 2 * H * H:o + 2 * H * H + H]) + h
    o = 2 * H + 4 * (2 * H * H + H)
    e = rho * sc * (h @ p[o:o + H] + p[o + H])
    (grad,) = torch.autograd.grad((e * ge).sum(), p)
    return e.detach().numpy(), grad.numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("vcycle", "refresh"):
        # Defined by the hierarchy the library builds.
        return None
    if kind == "pcg2d":
        # Cell-centred 5-point Dirichlet Laplacian on the unit square: its
        # eigenvectors are the sine (DST-II) modes. Cell order: row by row.
        n = case["n"]
        k = np.arange(1, n + 1)
        Q = np.sin(math.pi * np.outer(np.arange(n) + 0.5, k) / n) * math.sqrt(2.0 / n)
        Q[:, -1] /= math.sqrt(2.0)
        lam = (2.0 * n * np.sin(math.pi * k / (2.0 * n))) ** 2
        f = _poisson2d_source(case, seed).reshape(n, n)
        return (Q @ ((Q.T @ f @ Q) / (lam[:, None] + lam[None, :])) @ Q.T).ravel()
    if kind == "fgmres":
        return _exact_solution(case, seed)
    if kind == "learned":
        return _mpnn_exact(case, seed)
    if kind == "face":
        f = _face_inputs(case, seed)
        own, nei, n = f["owner"].astype(np.int64), f["neighbour"], len(f["phi"])
        inn = nei >= 0
        vf = np.where(inn, 0.5 * (f["phi"][own] + f["phi"][np.maximum(nei, 0)]), f["phi"][own])
        out = [(np.bincount(own, vf * f[s], n) - np.bincount(nei[inn], (vf * f[s])[inn], n)) / f["volume"]
               for s in ("sx", "sy", "sz")]
        return (*out, np.bincount(own, f["flux"], n) - np.bincount(nei[inn], f["flux"][inn], n))
    m = _mesh(case, seed)
    geo = _geometry(m)
    fc, S, cc, vol, o, nb = geo
    ni, n = m.n_internal_faces, m.n_cells
    f = _fields(case, m, seed)
    vt, vv, pt, pv = _boundary(case, m)
    phi = _mass_flux(m, geo, vt, vv, f["U"]) * (1.0 + 0.01 * f["noise"])
    if kind == "pressure":
        g = _green_gauss(m, geo, pt, pv, f["p"])
        coef, flux, on = _face_pressure(m, geo, pt, pv, f["rau"], f["p"], g)
        diag = np.bincount(o, coef, n) + np.bincount(nb, coef[:ni], n)
        net = phi - np.where(np.arange(m.n_faces) < ni, flux, 0.0)
        rhs = -(np.bincount(o, net, n) - np.bincount(nb, net[:ni], n))
        rhs += np.bincount(o[ni:], flux[ni:], n)
        order, rows, cols = _csr_order(n, o[:ni], nb)
        vals = np.concatenate([diag, -coef[:ni], -coef[:ni]])[order]
        if not pt.any():
            keep = (rows[order] != 0) & (cols[order] != 0)
            return vals[keep], rhs[1:]
        return vals, rhs
    if kind == "momentum":
        vals, rhs, diag, _, _ = _momentum_exact(m, geo, vt, vv, f, phi, case["bounded"], 0.7)
        return vals, rhs, diag
    vals, rhs, diag, rows, cols = _momentum_exact(m, geo, vt, vv, f, phi, True, 0.7)
    U = f["U"].reshape(3, -1)
    gp, rhs = f["gp"].reshape(3, -1), rhs.reshape(3, -1)
    off = rows != cols
    ra = 1.0 / diag
    hb = np.stack([ra * (rhs[k] + gp[k] * vol - np.bincount(rows[off], vals[off] * U[k][cols[off]], n))
                   for k in range(3)])
    rau = np.repeat(ra[None], 3, 0)
    g = _green_gauss(m, geo, pt, pv, f["p"])
    _, flux, _ = _face_pressure(m, geo, pt, pv, rau.ravel(), f["p"], g)
    return rau.ravel(), hb.ravel(), _mass_flux(m, geo, vt, vv, hb.ravel()) - flux, (hb - rau * gp * vol).ravel()


def _exact_solution(case, seed):
    """A x = b by Jacobi-preconditioned conjugate gradients in float64 with
    one restart from the true residual."""
    if _cells(case) > 80000:
        return None
    s = _system(case, seed)
    A = torch.sparse_csr_tensor(torch.from_numpy(s.rowp.astype(np.int64)), torch.from_numpy(s.cols.astype(np.int64)),
                                torch.from_numpy(s.vals), size=(s.n, s.n))
    rows = np.repeat(np.arange(s.n), np.diff(s.rowp))
    inv = torch.from_numpy(1.0 / s.vals[rows == s.cols])
    b = torch.from_numpy(s.b)
    x = torch.zeros_like(b)
    for goal in (1e-11, 1e-13):
        r = b - A @ x
        z = inv * r
        p, rz = z.clone(), r @ z
        for _ in range(6000):
            q = A @ p
            a = rz / (p @ q)
            x += a * p
            r -= a * q
            if torch.linalg.norm(r) <= goal * torch.linalg.norm(b):
                break
            z = inv * r
            rz, old = r @ z, rz
            p = z + (rz / old) * p
    return x.numpy()
