"""Pressure and momentum assembly by rows, one thread a cell, against the oracle bit for bit
where the bookkeeping branches: pairs of cells joined by one, two or four faces
(every quad whole, halved, or a fan of triangles, in shuffled face order), up to
24 slots a cell (more than LDS holds the coefficients of), cells short of, at
and past a workgroup, and the row and column of a reference cell left out at
the start, inside and at the end of the numbering."""
import numpy as np
import pytest

import cfdx_dev_amd as cx

pytestmark = pytest.mark.gpu


def split_faces(m, pieces, seed, inner_only=False):
    """m with every quad (or the internal ones) in `pieces` faces, internal faces first, each group shuffled."""
    rng = np.random.default_rng(seed)
    fo, fv = m.face_offsets.astype(int), m.face_vertices.astype(int)
    pts = [list(a) for a in (m.px, m.py, m.pz)]
    faces, parent = [], []
    for f in range(m.n_faces):
        v = list(fv[fo[f]:fo[f + 1]])
        if pieces == 1 or (inner_only and m.neighbour[f] < 0):
            parts = [v]
        elif pieces == 2:
            parts = [[v[0], v[1], v[2]], [v[0], v[2], v[3]]]
        else:
            mid = len(pts[0])
            for a in pts:
                a.append(float(np.mean([a[i] for i in v])))
            parts = [[v[i], v[(i + 1) % 4], mid] for i in range(4)]
        faces += parts
        parent += [f] * len(parts)
    parent = np.array(parent)
    inner = np.flatnonzero(m.neighbour[parent] >= 0)
    outer = np.flatnonzero(m.neighbour[parent] < 0)
    order = np.concatenate([rng.permutation(inner), rng.permutation(outer)])
    children = [[] for _ in range(m.n_faces)]
    for new, old in enumerate(order):
        children[parent[old]].append(new)
    cells = [[] for _ in range(m.n_cells)]
    for c in range(m.n_cells):
        for f in m.cell_faces[m.cell_offsets[c]:m.cell_offsets[c + 1]]:
            cells[c] += children[f]
        cells[c] = list(rng.permutation(cells[c]))
    fl = [faces[i] for i in order]
    par = parent[order]

    def offsets(lists, dtype):
        return np.concatenate([[0], np.cumsum([len(x) for x in lists])]).astype(dtype)

    return cx.Mesh(px=np.array(pts[0]), py=np.array(pts[1]), pz=np.array(pts[2]),
                   face_offsets=offsets(fl, m.face_offsets.dtype),
                   face_vertices=np.concatenate(fl).astype(m.face_vertices.dtype), owner=m.owner[par],
                   neighbour=m.neighbour[par], cell_offsets=offsets(cells, m.cell_offsets.dtype),
                   cell_faces=np.concatenate(cells).astype(m.cell_faces.dtype), patch_of_face=m.patch_of_face[par],
                   patch_kind=m.patch_kind, cell_ijk=m.cell_ijk, n_cells=m.n_cells, n_faces=len(fl),
                   n_internal_faces=len(inner), n_patches=m.n_patches)


def same(oracle, m, ref, fixed):
    g = oracle.geometry(m)
    fv = cx.FvMesh(m)
    rng = np.random.default_rng(3)
    nc = m.n_cells
    pt = np.zeros(m.n_patches, np.uint8)
    pv = rng.normal(size=m.n_patches)
    if fixed:
        pt[1] = 1
        pt[m.n_patches - 1] = 1
    rau, p, phi = np.exp(rng.normal(size=3 * nc)), rng.normal(size=nc), rng.normal(size=m.n_faces)
    grad = oracle.gauss_gradient(m, g, pt, pv, p)
    a = oracle.pressure_assemble(m, g, pt, pv, 0.7, rau, phi, p, grad, ref)
    for _ in range(2):  # a second call on a used handle
        got = fv.pressure_assemble(pt, pv, 0.7, rau, phi, p, ref)
        for x, y in zip(got, (a["rowp"], a["cols"], a["vals"], a["rhs"])):
            assert np.array_equal(x, y)


@pytest.mark.parametrize("dims", [(3, 3, 2), (8, 8, 4), (11, 8, 3)])
@pytest.mark.parametrize("pieces", [1, 2, 4])
def test_split_faces_fixed_pressure(oracle, dims, pieces):
    m = cx.generate_mesh("box", *dims, jitter=0.05, permute=True, seed=4)
    same(oracle, split_faces(m, pieces, 7), 0, True)


@pytest.mark.parametrize("pieces", [1, 2])
@pytest.mark.parametrize("where", ["first", "inside", "last"])
def test_reference_cell_left_out(oracle, pieces, where):
    m = split_faces(cx.generate_mesh("box", 9, 7, 5, jitter=0.05, permute=where == "inside", seed=5), pieces, 8)
    same(oracle, m, {"first": 0, "inside": m.n_cells // 2, "last": m.n_cells - 1}[where], False)


def test_empty_and_stepped(oracle):
    same(oracle, cx.generate_mesh("extruded2d", 20, 15, 1), 7, False)
    same(oracle, cx.generate_mesh("channel_step", 24, 12, 4, lx=3.0, jitter=0.05, permute=True, seed=9,
                                  step_height_fraction=1.0 / 3.0, step_length_fraction=0.25), 0, True)


@pytest.mark.parametrize("pieces", [1, 2])
@pytest.mark.parametrize("dims", [(8, 8, 4), (11, 8, 3)])
@pytest.mark.parametrize("jitter", [0.0, 0.05])  # orthogonal or not: without or with velocity gradients
@pytest.mark.parametrize("bounded", [True, False])
def test_momentum_rows(oracle, dims, pieces, jitter, bounded):
    m = cx.generate_mesh("box", *dims, jitter=jitter, permute=True, seed=6)
    if pieces > 1:  # wall faces stay whole: ten faces a cell at the most
        m = cx.generate_mesh("extruded2d", dims[0], dims[1] * dims[2], 1, jitter=jitter, permute=True, seed=6)
        m = split_faces(m, pieces, 9, inner_only=True)
    g = oracle.geometry(m)
    rng = np.random.default_rng(5)
    nc = m.n_cells
    U, gp, body = (rng.normal(size=3 * nc) for _ in range(3))
    mu = np.exp(rng.normal(size=nc)) * (rng.uniform(size=nc) > 0.1)
    vt = np.zeros(m.n_patches, np.uint8)
    vt[0] = vt[1] = 1
    vv = rng.normal(size=3 * m.n_patches)
    phi = 0.01 * oracle.mass_flux(m, g, vt, vv, 1.0, U)
    mu += 1.0  # keeps the diagonal positive
    want = oracle.momentum_assemble(m, g, vt, vv, mu, phi, gp, body, U, bounded, 0.7)
    got = cx.FvMesh(m).momentum_assemble(vt, vv, mu, phi, gp, body, U, bounded=bounded, alpha=0.7)
    assert np.array_equal(got[0], want["rowp"]) and np.array_equal(got[1], want["cols"])
    assert np.array_equal(got[2], want["vals"][0])
    assert np.array_equal(got[3], want["rhs"].ravel())
    assert np.array_equal(got[4], want["diag"][0])
