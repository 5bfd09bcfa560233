"""Finite-volume handles at the edges of what they take, against the oracle
bit for bit: a cell that lists a boundary face another cell owns; cells of
more faces than the slot stencils hold, which the assemblies by rows refuse
and every other call takes."""
import numpy as np
import pytest

import cfdx_dev_amd as cx

pytestmark = pytest.mark.gpu


def foreign_boundary_face(m, inside):
    """m with one boundary face listed by a second cell as well: the owner's
    neighbour, at the end of its list (inside False) or in its middle."""
    f = m.n_internal_faces + 5
    own = int(m.owner[f])
    g = np.flatnonzero((m.neighbour >= 0) & ((m.owner == own) | (m.neighbour == own)))[0]
    c = int(m.neighbour[g] if m.owner[g] == own else m.owner[g])
    lists = [list(m.cell_faces[m.cell_offsets[i]:m.cell_offsets[i + 1]]) for i in range(m.n_cells)]
    lists[c].insert(2 if inside else len(lists[c]), f)
    off = np.concatenate([[0], np.cumsum([len(x) for x in lists])]).astype(m.cell_offsets.dtype)
    d = {k: getattr(m, k) for k in m.__dataclass_fields__}
    d.update(cell_offsets=off, cell_faces=np.concatenate(lists).astype(m.cell_faces.dtype))
    return cx.Mesh(**d), int(m.patch_of_face[f])


@pytest.mark.parametrize("inside", [False, True])
@pytest.mark.parametrize("permute", [False, True])
def test_boundary_face_of_another_cell(oracle, inside, permute):
    m, patch = foreign_boundary_face(cx.generate_mesh("box", 7, 6, 5, jitter=0.1, permute=permute, seed=3), inside)
    g = oracle.geometry(m)
    fv = cx.FvMesh(m)
    rng = np.random.default_rng(2)
    nc = m.n_cells
    p, pv = rng.normal(size=nc), rng.normal(size=m.n_patches)
    pt = np.zeros(m.n_patches, np.uint8)
    for t in (0, 1, 2):
        pt[patch] = t
        assert np.array_equal(fv.gauss_gradient(pt, pv, p), oracle.gauss_gradient(m, g, pt, pv, p))
    pt[:] = 0
    rau, phi = np.exp(rng.normal(size=3 * nc)), rng.normal(size=m.n_faces)
    a = oracle.pressure_assemble(m, g, pt, pv, 0.9, rau, phi, p, oracle.gauss_gradient(m, g, pt, pv, p), 4)
    for x, y in zip(fv.pressure_assemble(pt, pv, 0.9, rau, phi, p, 4), (a["rowp"], a["cols"], a["vals"], a["rhs"])):
        assert np.array_equal(x, y)


def fan_faces(m, k):
    """m with every quad in a fan of 4 k triangles around its mean (each edge in k pieces)."""
    pts = [list(a) for a in (m.px, m.py, m.pz)]
    fo, fv = m.face_offsets.astype(int), m.face_vertices.astype(int)
    faces, parent = [], []
    for f in range(m.n_faces):
        v = fv[fo[f]:fo[f + 1]]
        ring = []
        for i in range(4):
            for j in range(k):
                ring.append(len(pts[0]))
                for a in pts:
                    a.append(a[v[i]] + (a[v[(i + 1) % 4]] - a[v[i]]) * j / k)
        mid = len(pts[0])
        for a in pts:
            a.append(float(np.mean([a[i] for i in v])))
        faces += [[ring[i], ring[(i + 1) % len(ring)], mid] for i in range(len(ring))]
        parent += [f] * (4 * k)
    par = np.array(parent)
    cells = [np.concatenate([np.flatnonzero(par == f) for f in m.cell_faces[m.cell_offsets[c]:m.cell_offsets[c + 1]]])
             for c in range(m.n_cells)]
    d = {key: getattr(m, key) for key in m.__dataclass_fields__}
    d.update(px=np.array(pts[0]), py=np.array(pts[1]), pz=np.array(pts[2]),
             face_offsets=(3 * np.arange(len(faces) + 1)).astype(m.face_offsets.dtype),
             face_vertices=np.concatenate(faces).astype(m.face_vertices.dtype), owner=m.owner[par],
             neighbour=m.neighbour[par],
             cell_offsets=np.concatenate([[0], np.cumsum([len(c) for c in cells])]).astype(m.cell_offsets.dtype),
             cell_faces=np.concatenate(cells).astype(m.cell_faces.dtype), patch_of_face=m.patch_of_face[par],
             n_faces=len(faces), n_internal_faces=int((m.neighbour[par] >= 0).sum()))
    return cx.Mesh(**d)


@pytest.mark.parametrize("k,slots", [(10, True), (11, False)])  # 240 and 264 faces a cell
@pytest.mark.parametrize("first", ["pattern", "assemble"])
def test_cells_of_many_faces(oracle, k, slots, first):
    m = fan_faces(cx.generate_mesh("box", 3, 2, 2), k)
    g = oracle.geometry(m)
    fv = cx.FvMesh(m)
    rng = np.random.default_rng(6)
    nc = m.n_cells
    pt, pv = np.zeros(m.n_patches, np.uint8), np.zeros(m.n_patches)
    rau, p, phi = np.exp(rng.normal(size=3 * nc)), rng.normal(size=nc), rng.normal(size=m.n_faces)
    a = oracle.pressure_assemble(m, g, pt, pv, 1.0, rau, phi, p, oracle.gauss_gradient(m, g, pt, pv, p), 0)

    def assemble():
        if slots:
            got = fv.pressure_assemble(pt, pv, 1.0, rau, phi, p, 0)
            for x, y in zip(got, (a["rowp"], a["cols"], a["vals"], a["rhs"])):
                assert np.array_equal(x, y)
            return
        for _ in range(2):  # refused as often as it is asked
            with pytest.raises(RuntimeError, match="255 faces"):
                fv.pressure_assemble(pt, pv, 1.0, rau, phi, p, 0)

    if first == "assemble":
        assemble()
    for x, y in zip(fv.pressure_pattern(pt, 0), (a["rowp"], a["cols"])):
        assert np.array_equal(x, y)
    fval = np.where(m.neighbour < 0, 0.5, np.nan)
    fneu, src = np.zeros(m.n_faces, np.uint8), rng.normal(size=nc)
    for x, y in zip(fv.diffusion_assemble(1.3, src, fval, fneu), oracle.diffusion_assemble(m, g, 1.3, src, fval, fneu)):
        assert np.array_equal(x, y)
    rp, cols = fv.momentum_pattern()
    vals, diag = rng.normal(size=len(cols)), np.exp(rng.normal(size=nc))
    rhs, gp, U = (rng.normal(size=3 * nc) for _ in range(3))
    want = oracle.momentum_hbya(rp, cols, np.tile(vals, 3), rhs, np.tile(diag, 3), gp, g[3], U)
    for x, y in zip(fv.momentum_hbya(vals, rhs, diag, gp, U), want):
        assert np.array_equal(x, y)
    assemble()
