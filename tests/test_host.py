"""Host logic of librkdg without a GPU: exported symbols, mesh generation and ingest,
config parser, .plt writer, state dump, basis exchange (CPU)."""
import ctypes
import json
import os
import re

import numpy as np
import pytest

from rkdg_heter_calculate_amd import Grid, _lib as L
from rkdg_heter_calculate_amd.solver import freestream_state

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
GOLD = os.path.join(ROOT, "tests", "golden")


def test_library_exports_every_declared_symbol():
    with open(os.path.join(ROOT, "include", "rkdg.h")) as f:
        text = f.read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    names = set(re.findall(r"\b(rkdg_[a-z0-9_]+)\s*\(", text))
    lib = ctypes.CDLL(L.LIB_PATH)
    missing = [n for n in sorted(names) if not hasattr(lib, n)]
    assert not missing, missing
    assert len(names) >= 40
    # and the Python binding knows every one of them
    bound = {n for n, _, _ in L.SIGNATURES}
    assert names <= bound, names - bound


def check_connectivity(g, periodic, lx=None, ly=None):
    E = g.n_elements
    ex, ey = g.element_coords()
    cross = (ex[:, 1] - ex[:, 0]) * (ey[:, 2] - ey[:, 0]) - (ey[:, 1] - ey[:, 0]) * (ex[:, 2] - ex[:, 0])
    assert (cross > 0).all()  # CCW
    for e in range(E):
        for k in range(3):
            n = g.neighbour[e, k]
            if n < 0:
                assert not periodic
                continue
            s = g.shared_edge[e, k]
            assert g.neighbour[n, s] == e and g.shared_edge[n, s] == k
            # same physical edge (up to a period), opposite direction
            a = np.array([ex[e, (k + 1) % 3], ey[e, (k + 1) % 3]])
            b = np.array([ex[e, (k + 2) % 3], ey[e, (k + 2) % 3]])
            c = np.array([ex[n, (s + 1) % 3], ey[n, (s + 1) % 3]])
            d = np.array([ex[n, (s + 2) % 3], ey[n, (s + 2) % 3]])
            sh = (a - d)
            if periodic:
                sh = sh - np.round(sh / [lx, ly]) * [lx, ly]
            assert np.allclose(sh, 0, atol=1e-12)
            assert np.allclose((a - d) - (b - c), 0, atol=1e-12)


@pytest.mark.parametrize("periodic", [True, False])
def test_splitquad_connectivity(periodic):
    g = Grid.splitquad(9, 7, 0.0, 0.0, 10.0, 7.0, periodic=periodic, diagonal=1, jitter=0.2, seed=3)
    assert g.n_elements == 2 * 9 * 7
    check_connectivity(g, periodic, 10.0, 7.0)
    if not periodic:
        nb = (g.neighbour < 0).sum()
        assert nb == 2 * (9 + 7)
        assert (g.boundary[g.neighbour < 0] == L.BC_OUTFLOW).all()


def test_splitquad_jitter_and_seed():
    n = 16
    a = Grid.splitquad(n, n, 0.0, 0.0, 10.0, 10.0, periodic=True, diagonal=1, jitter=0.2, seed=42)
    b = Grid.splitquad(n, n, 0.0, 0.0, 10.0, 10.0, periodic=True, diagonal=1, jitter=0.2, seed=42)
    c = Grid.splitquad(n, n, 0.0, 0.0, 10.0, 10.0, periodic=True, diagonal=1, jitter=0.2, seed=43)
    assert np.array_equal(a.vx, b.vx) and np.array_equal(a.tri, b.tri)
    assert not np.array_equal(a.vx, c.vx)
    h = 10.0 / n
    i = np.arange((n + 1) * (n + 1)) % (n + 1)
    j = np.arange((n + 1) * (n + 1)) // (n + 1)
    dx, dy = a.vx - i * h, a.vy - j * h
    assert np.abs(dx).max() <= 0.2 * h and np.abs(dy).max() <= 0.2 * h
    bnd = (i == 0) | (i == n) | (j == 0) | (j == n)
    assert np.all(dx[bnd] == 0) and np.all(dy[bnd] == 0)
    # both diagonals occur
    d0 = Grid.splitquad(n, n, 0.0, 0.0, 10.0, 10.0, periodic=True, diagonal=0)
    assert not np.array_equal(a.tri, d0.tri)


def write_reference_mesh(tmp_path, d, with_header_neigh=True):
    """Reconstructs the reference mesh files from the fixture (headers as the originals)."""
    inp = tmp_path / "input"
    inp.mkdir()
    E, NV = d["tri"].shape[0], d["vertices"].shape[0]
    (inp / "Vertice.dat").write_text("#vertist data\n" + "\n".join(f"{float(x)!r} {float(y)!r}" for x, y in d["vertices"]) + "\n")
    (inp / "ElemVertice.dat").write_text("#ElemVertex Data\n" + "\n".join(" ".join(map(str, r)) for r in d["tri"]) + "\n")
    (inp / "ElemNeigh.dat").write_text(("#ElemNeigh data\n" if with_header_neigh else "") +
                                      "\n".join(" ".join(map(str, r)) for r in d["neigh"]) + "\n")
    (inp / "ElemEdge.dat").write_text("#Elemside data\n" + "\n".join(" ".join(map(str, r)) for r in d["edge"]) + "\n")
    (inp / "EdgeVertice.dat").write_text("#Sidelist data\n" + "\n".join(" ".join(map(str, r)) for r in d["edge_vertices"]) + "\n")
    (inp / "ElemDepart.dat").write_text("\n".join(map(str, d["partition"])) + "\n")
    conf = tmp_path / "mesh.conf"
    conf.write_text(f"trianglenum {E}\nverticenum {NV}\nedgenum {d['edge_vertices'].shape[0]}\n"
                    f"trivertice_filename {inp}/ElemVertice.dat\ntrineigh_filename {inp}/ElemNeigh.dat\n"
                    f"triedge_filename {inp}/ElemEdge.dat\nvertice_filename {inp}/Vertice.dat\n"
                    f"edgevertice_filename {inp}/EdgeVertice.dat\noutput_filename out.plt\n")
    return str(conf), str(inp / "ElemDepart.dat")


def test_reader_reproduces_reference_grid_setup(tmp_path):
    d = np.load(os.path.join(GOLD, "naca_grid.npz"))
    conf, part = write_reference_mesh(tmp_path, d)
    g = Grid.read(conf, part, box=15.0)
    E = g.n_elements
    assert E == d["tri"].shape[0]
    assert np.array_equal(g.tri, d["tri"]) and np.array_equal(g.neighbour, d["neigh"])
    assert np.array_equal(g.partition, d["partition"])
    rn, rse, rflag = d["ref_neighbour"], d["ref_shared_edge"], d["ref_flag"]
    for e in range(E):
        for k in range(3):
            if g.neighbour[e, k] >= 0:
                assert g.shared_edge[e, k] == rse[k, e]
            else:
                ghost = rn[k, e]
                assert g.boundary[e, k] == rflag[ghost]
    assert (g.boundary[g.neighbour < 0] == L.BC_FARFIELD).sum() == 64
    assert (g.boundary[g.neighbour < 0] == L.BC_REFLECTION).sum() == 130


def test_reader_rejects_inconsistent_edges(tmp_path):
    d = dict(np.load(os.path.join(GOLD, "naca_grid.npz")))
    nb = d["neigh"].copy()
    e = int(np.nonzero((nb >= 0).all(axis=1))[0][0])
    nb[e, 0], nb[e, 1] = nb[e, 1], nb[e, 0]
    d["neigh"] = nb
    conf, part = write_reference_mesh(tmp_path, d)
    with pytest.raises(L.RkdgError) as ei:
        Grid.read(conf, part)
    assert ei.value.code == L.ERR_MESH


def test_reader_missing_file(tmp_path):
    with pytest.raises(L.RkdgError) as ei:
        Grid.read(str(tmp_path / "nope.conf"))
    assert ei.value.code == L.ERR_IO


def config_get(path, key):
    lib = L.load()
    buf = ctypes.create_string_buffer(4096)
    L.check(lib.rkdg_config_get(path.encode(), key.encode(), buf, 4096), None, "config")
    return buf.value.decode("latin-1")


def test_config_parser_matches_reference_values(tmp_path):
    with open(os.path.join(GOLD, "config_values.json")) as f:
        gold = json.load(f)
    for name, entry in gold.items():
        p = tmp_path / (name + ".txt")
        p.write_text(entry["text"])
        for k, v in zip(entry["keys"], entry["values"]):
            assert config_get(str(p), k) == v, (name, k)


def cxx_g(v):
    """C++ ostream default formatting (%g, 6 significant digits)."""
    return "%g" % v


def test_plt_writer_format(tmp_path):
    g = Grid.splitquad(3, 2, 0.0, 0.0, 1.5, 1.0, periodic=False, diagonal=0)
    E, NV = g.n_elements, g.n_vertices
    rng = np.random.default_rng(0)
    U = np.zeros((4, 3, E))
    U[0, 0] = rng.uniform(0.9, 1.1, E)
    U[1, 0] = rng.uniform(-0.1, 0.1, E)
    U[2, 0] = rng.uniform(-0.1, 0.1, E)
    U[3, 0] = rng.uniform(2.4, 2.6, E)
    path = str(tmp_path / "s.plt")
    g.write_plt(path, U, 3)
    txt = open(path).read()

    def block(vals):
        s = ""
        for i, v in enumerate(vals):
            s += v + "  "
            if i % 6 == 0:
                s += "\n"
        return s

    r, u, v = U[0, 0], U[1, 0] / U[0, 0], U[2, 0] / U[0, 0]
    p = 0.4 * (U[3, 0] - 0.5 * r * (u * u + v * v))
    ma = np.sqrt(u * u + v * v) / np.sqrt(1.4 * p / r)
    exp = ("TITLE=RKDG\nVARIABLES=X , Y , rho , u , v , p, Ma , FLAG\n"
           f"ZONE T= T1 N= {NV} , E= {E} , ZONETYPE=FETRIANGLE\nDATAPACKING=BLOCK\n"
           "VARLOCATION=([1-2]=NODAL,[3-8]=CELLCENTERED)\nDT=(SINGLE SINGLE SINGLE SINGLE SINGLE SINGLE SINGLE SINGLE)\n")
    exp += block([cxx_g(x) for x in g.vx]) + block([cxx_g(y) for y in g.vy]) + "\n"
    for arr in (r, u, v, p, ma):
        exp += block([cxx_g(x) for x in arr]) + "\n"
    exp += block(["1"] * E) + "\n"
    for t in g.tri:
        exp += f"{t[0] + 1}    {t[1] + 1}    {t[2] + 1}\n"
    assert txt == exp


def test_state_dump_round_trip(tmp_path):
    lib = L.load()
    U = np.random.default_rng(1).normal(size=(4, 6, 33))
    path = str(tmp_path / "st.bin").encode()
    L.check(lib.rkdg_dump_state(path, 6, 33, 1.25, L.dptr(U)), None, "dump")
    V = np.zeros_like(U)
    t = ctypes.c_double()
    L.check(lib.rkdg_load_state(path, 6, 33, ctypes.byref(t), L.dptr(V)), None, "load")
    assert np.array_equal(U, V) and t.value == 1.25
    assert lib.rkdg_load_state(path, 6, 34, ctypes.byref(t), L.dptr(V)) == L.ERR_IO


@pytest.mark.parametrize("P", [1, 2, 3])
def test_basis_exchange_round_trip_and_mean(P):
    """element -> native -> element recovers the reference coefficients; the mode-0
    coefficient (cell mean) is the same in both bases."""
    lib = L.load()
    g = Grid.splitquad(6, 5, 0.0, 0.0, 3.0, 2.0, periodic=False, diagonal=1, jitter=0.2, seed=1)
    ex, ey = g.element_coords()
    ex, ey = np.ascontiguousarray(ex), np.ascontiguousarray(ey)
    Np = (P + 1) * (P + 2) // 2
    E = g.n_elements
    U = np.random.default_rng(P).normal(size=(4, Np, E))
    D = np.zeros_like(U)
    B = np.zeros_like(U)
    L.check(lib.rkdg_convert_basis(P, E, L.dptr(ex), L.dptr(ey), L.BASIS_ELEMENT, L.dptr(U), L.dptr(D)), None, "c")
    L.check(lib.rkdg_convert_basis(P, E, L.dptr(ex), L.dptr(ey), L.BASIS_NATIVE, L.dptr(D), L.dptr(B)), None, "c")
    assert np.allclose(B, U, rtol=1e-12, atol=1e-12 * np.abs(U).max())
    assert np.allclose(D[:, 0], U[:, 0], rtol=1e-13, atol=1e-14)


def test_freestream_state_matches_reference_formula():
    fs = freestream_state(1.4, 5.0, 0.4, 1.0, 1.0)
    ut = np.sqrt(1.4) * 0.4
    al = 5.0 * np.arctan(1.0) * 4 / 180
    assert np.allclose(fs, [1.0, ut * np.cos(al), ut * np.sin(al), 0.5 * ut * ut + 1 / 0.4], rtol=1e-15)


def test_edge_normals_follow_from_inverse_jacobian():
    """The stage kernels derive edge k's outward normal times its length as 2A s_k with
    s_0 = xi + eta, s_1 = -xi, s_2 = -eta (xi, eta: rows of the inverse Jacobian of the
    affine map, 2A its determinant).  Checked against the vertex formulas of
    src/triangleinfo.cpp:171-189 (edge k opposite vertex k, CCW) on random triangles."""
    rng = np.random.default_rng(5)
    n = 0
    while n < 300:
        x, y = rng.uniform(-1, 1, 3), rng.uniform(-1, 1, 3)
        det = (x[1] - x[0]) * (y[2] - y[0]) - (x[2] - x[0]) * (y[1] - y[0])
        if abs(det) < 1e-2:
            continue
        if det < 0:
            x[[1, 2]], y[[1, 2]] = x[[2, 1]], y[[2, 1]]
            det = -det
        n += 1
        xi = np.array([y[2] - y[0], -(x[2] - x[0])]) / det
        eta = np.array([-(y[1] - y[0]), x[1] - x[0]]) / det
        area = 0.5 * det
        s = [xi + eta, -xi, -eta]
        nl = [np.array([y[2] - y[1], x[1] - x[2]]), np.array([y[0] - y[2], x[2] - x[0]]),
              np.array([y[1] - y[0], x[0] - x[1]])]
        for k in range(3):
            assert np.allclose(2 * area * s[k], nl[k], rtol=1e-12, atol=1e-13), (k, x, y)
            # outward: the normal points away from the opposite vertex
            mid = 0.5 * np.array([x[(k + 1) % 3] + x[(k + 2) % 3], y[(k + 1) % 3] + y[(k + 2) % 3]])
            assert np.dot(s[k], mid - np.array([x[k], y[k]])) > 0


def test_create_rejects_clockwise_elements():
    """Because the kernels derive normals from the inverse Jacobian, rkdg_create refuses an
    element given clockwise (the mesh contract of rkdg.h) before touching the device."""
    from rkdg_heter_calculate_amd import Solver
    g = Grid.splitquad(4, 4, periodic=True)
    g.tri[5] = g.tri[5][[0, 2, 1]]
    with pytest.raises(L.RkdgError) as ei:
        Solver(g, degree=1)
    assert ei.value.code == L.ERR_MESH and "clockwise" in str(ei.value)


def _batch_create(grids, **kw):
    from rkdg_heter_calculate_amd.solver import make_params, mesh_view
    lib = L.load()
    views = [mesh_view(g) for g in grids]
    meshes = (L.Mesh * len(grids))(*views)
    params = (L.Params * len(grids))(*[make_params(**kw) for _ in grids])
    h = ctypes.c_void_p()
    rc = lib.rkdg_batch_create(len(grids), meshes, params, ctypes.byref(h))
    msg = lib.rkdg_batch_last_error(None)
    msg = msg.decode() if msg else ""
    if rc == 0:
        lib.rkdg_batch_destroy(h)
    return rc, msg


@pytest.mark.parametrize("fault", ["shared_edge", "asymmetric", "tag"])
def test_create_rejects_inconsistent_connectivity(fault):
    """A shared-edge index outside 0..2, a one-sided neighbour relation or an unknown
    boundary tag is refused by rkdg_create and rkdg_batch_create before the device is
    touched: the kernels would read another element's traces or an undefined ghost."""
    from rkdg_heter_calculate_amd import Solver
    g = Grid.splitquad(4, 4, periodic=False)
    e, k = next((e, k) for e in range(g.n_elements) for k in range(3) if g.neighbour[e, k] >= 0)
    if fault == "shared_edge":
        g.shared_edge[e, k] = 3
    elif fault == "asymmetric":
        n = g.neighbour[e, k]
        g.neighbour[e, k] = next(x for x in range(g.n_elements) if x not in (e, n))
    else:
        eb, kb = next((e, k) for e in range(g.n_elements) for k in range(3) if g.neighbour[e, k] < 0)
        g.boundary[eb, kb] = 7
    with pytest.raises(L.RkdgError) as ei:
        Solver(g, degree=1, dt_policy="max", cfl=0.3)
    assert ei.value.code == L.ERR_MESH
    rc, msg = _batch_create([Grid.splitquad(3, 3, periodic=True), g], degree=1, dt_policy="max", cfl=0.3)
    assert rc == L.ERR_MESH, (rc, msg)


def test_create_rejects_an_empty_mesh():
    """n_elements < 1 is an argument error, reported before any device call."""
    from rkdg_heter_calculate_amd.solver import make_params
    lib = L.load()
    m = L.Mesh()
    m.n_elements, m.n_vertices = 0, 0
    prm = make_params(degree=2)
    h = ctypes.c_void_p()
    assert lib.rkdg_create(ctypes.byref(m), ctypes.byref(prm), ctypes.byref(h)) == L.ERR_ARG
    assert lib.rkdg_batch_create(0, None, None, ctypes.byref(h)) == L.ERR_ARG


@pytest.mark.parametrize("degree,n,msg", [(1, (1 << 29), "too many elements"),
                                           (3, 13_500_000, "above 4 GiB"),
                                           (2, 22_500_000, "above 4 GiB")])
def test_create_rejects_meshes_beyond_the_addressing_limits(degree, n, msg):
    """Up to 2^29 - 1 elements (neighbour ids carry the edge index in two bits) and every
    device array below 4 GiB (32-bit byte offsets): larger meshes are argument errors,
    reported before any array is read or any device call (the arrays here hold 3 entries)."""
    from rkdg_heter_calculate_amd.solver import make_params
    lib = L.load()
    d = (ctypes.c_double * 3)()
    i = (ctypes.c_int32 * 9)()
    m = L.Mesh()
    m.n_vertices, m.n_elements = 3, n
    m.vx = m.vy = ctypes.cast(d, L.P_double)
    m.tri = m.neighbour = ctypes.cast(i, L.P_int32)
    prm = make_params(degree=degree)
    h = ctypes.c_void_p()
    assert lib.rkdg_create(ctypes.byref(m), ctypes.byref(prm), ctypes.byref(h)) == L.ERR_ARG
    assert msg in lib.rkdg_last_error(None).decode()


def _batch_create_each(grids, params):
    """rkdg_batch_create with one parameter set per mesh; (status, message)."""
    from rkdg_heter_calculate_amd.solver import make_params, mesh_view
    lib = L.load()
    views = [mesh_view(g) for g in grids]
    meshes = (L.Mesh * len(grids))(*views)
    prm = (L.Params * len(grids))(*[make_params(**p) for p in params])
    h = ctypes.c_void_p()
    rc = lib.rkdg_batch_create(len(grids), meshes, prm, ctypes.byref(h))
    msg = lib.rkdg_batch_last_error(None)
    if rc == 0:
        lib.rkdg_batch_destroy(h)
    return rc, msg.decode() if msg else ""


@pytest.mark.parametrize("field,a,b", [("limiter", False, True), ("dt_fixed", 0.01, 0.02),
                                       ("reduction_threads", 512, 64), ("block", 256, 128), ("device", 0, 1)])
def test_batch_rejects_per_instance_fields_it_cannot_honour(field, a, b):
    """Every field but the mesh, the initial state and cfl is one per launch: a batch whose
    instances disagree on one is refused before the device is touched, not run with
    instance 0's value."""
    g = Grid.splitquad(4, 4, periodic=True)
    base = dict(degree=2, dt_policy="fixed" if field == "dt_fixed" else "reference", cfl=0.2)
    p0, p1 = dict(base), dict(base)
    p0[field], p1[field] = a, b
    rc, msg = _batch_create_each([g, g], [p0, p1])
    assert rc == L.ERR_ARG, (rc, msg)


def test_batch_free_stream_must_agree_only_where_far_field_edges_use_it():
    ff = Grid.splitquad(4, 4, periodic=False, bc=L.BC_FARFIELD)
    per = Grid.splitquad(4, 4, periodic=True)
    fa, fb = [1.0, 0.5, 0.0, 2.6], [1.2, 0.0, 0.3, 2.9]
    rc, msg = _batch_create_each([ff, per, ff], [dict(degree=2, freestream=fa), dict(degree=2, freestream=fb),
                                                  dict(degree=2, freestream=fb)])
    assert rc == L.ERR_ARG and "free stream" in msg, (rc, msg)
    # the periodic instance never reads its free stream: accepted (the device is reached,
    # which this container lacks, so anything but an argument error)
    rc, msg = _batch_create_each([ff, per, ff], [dict(degree=2, freestream=fa), dict(degree=2, freestream=fb),
                                                  dict(degree=2, freestream=fa)])
    assert rc != L.ERR_ARG, (rc, msg)


@pytest.mark.parametrize("block", [32, 192, 320])
def test_batch_rejects_a_block_that_does_not_tile_256(block):
    g = Grid.splitquad(4, 4, periodic=True)
    rc, msg = _batch_create_each([g], [dict(degree=2, block=block)])
    assert rc == L.ERR_ARG and "block" in msg, (rc, msg)


def test_batch_rejects_missing_vertex_arrays():
    from rkdg_heter_calculate_amd.solver import make_params, mesh_view
    lib = L.load()
    g = Grid.splitquad(4, 4, periodic=True)
    v = mesh_view(g)
    v.vy = None
    meshes = (L.Mesh * 1)(v)
    prm = (L.Params * 1)(make_params(degree=2))
    h = ctypes.c_void_p()
    assert lib.rkdg_batch_create(1, meshes, prm, ctypes.byref(h)) == L.ERR_ARG


def _assert_same_mesh(a, b, tags=True):
    assert (a.n_elements, a.n_vertices) == (b.n_elements, b.n_vertices)
    assert np.array_equal(a.vx, b.vx) and np.array_equal(a.vy, b.vy)  # 17 significant digits
    assert np.array_equal(a.tri, b.tri) and np.array_equal(a.neighbour, b.neighbour)
    assert np.array_equal(a.shared_edge, b.shared_edge)
    if tags:
        assert np.array_equal(a.boundary, b.boundary)


@pytest.mark.parametrize("periodic", [False, True])
def test_mesh_writer_round_trip_split_quad(tmp_path, periodic):
    """rkdg_grid_write then rkdg_grid_read gives back the same arrays (boundary tags are not
    part of the format; the reader derives them), periodic seams included."""
    g = Grid.splitquad(9, 7, 0.0, 0.0, 2.0, 1.5, periodic=periodic, diagonal=1, jitter=0.2, seed=13)
    g.partition = (np.arange(g.n_elements) * 5 // g.n_elements).astype(np.int32)
    g.write(tmp_path)
    lines = {f: (tmp_path / f).read_text().splitlines() for f in
             ("Vertice.dat", "ElemVertice.dat", "ElemNeigh.dat", "ElemEdge.dat", "EdgeVertice.dat", "ElemDepart.dat")}
    E, NV = g.n_elements, g.n_vertices
    # one header line each, except ElemNeigh and ElemDepart (src/unstructuredgrid.cpp:193-305)
    assert len(lines["Vertice.dat"]) == NV + 1 and lines["Vertice.dat"][0].startswith("#")
    assert len(lines["ElemVertice.dat"]) == E + 1 and len(lines["ElemEdge.dat"]) == E + 1
    assert len(lines["ElemNeigh.dat"]) == E and not lines["ElemNeigh.dat"][0].startswith("#")
    assert len(lines["ElemDepart.dat"]) == E
    # edges: each interior edge once, each boundary edge once
    nb = g.neighbour
    n_edges = int((nb < 0).sum() + (nb >= 0).sum() // 2)
    assert len(lines["EdgeVertice.dat"]) == n_edges + 1
    conf = (tmp_path / "mesh.conf").read_text()
    assert f"trianglenum {E}" in conf and f"edgenum {n_edges}" in conf
    eid = np.array([list(map(int, s.split())) for s in lines["ElemEdge.dat"][1:]])
    for e in range(E):
        for k in range(3):
            n = nb[e, k]
            if n >= 0:
                assert eid[e, k] == eid[n, g.shared_edge[e, k]]
    r = Grid.read(str(tmp_path / "mesh.conf"), str(tmp_path / "ElemDepart.dat"), box=1e9)
    _assert_same_mesh(g, r, tags=False)
    assert np.array_equal(r.partition, g.partition)
    assert (r.boundary[r.neighbour < 0] == L.BC_REFLECTION).all()


def test_mesh_writer_round_trip_naca(tmp_path):
    d = np.load(os.path.join(GOLD, "naca_grid.npz"))
    conf, part = write_reference_mesh(tmp_path, d)
    g = Grid.read(conf, part, box=15.0)
    out = tmp_path / "written"
    out.mkdir()
    g.write(out)
    r = Grid.read(str(out / "mesh.conf"), str(out / "ElemDepart.dat"), box=15.0)
    _assert_same_mesh(g, r)
    assert np.array_equal(r.partition, g.partition)


@pytest.mark.skipif("libasan" in os.environ.get("LD_PRELOAD", ""), reason="the sanitizer maps its own shadow memory")
def test_host_loops_without_threads(tmp_path):
    """Where no thread can be started (no address space for its stack) the host loops run on the
    caller's thread: the same values, and no exception out of the C entry."""
    import subprocess
    import sys
    prog = tmp_path / "no_threads.py"
    prog.write_text("""
import resource, sys
import numpy as np
from rkdg_heter_calculate_amd import Grid, _lib as L
g = Grid.splitquad(80, 80, 0.0, 0.0, 1.0, 1.0, periodic=False, diagonal=1, jitter=0.2, seed=1)
ex, ey = (np.ascontiguousarray(a) for a in g.element_coords())
U = np.random.default_rng(0).uniform(-1, 1, (4, 6, g.n_elements))
a, b = np.empty_like(U), np.empty_like(U)
conv = lambda out: L.load().rkdg_convert_basis(2, g.n_elements, L.dptr(ex), L.dptr(ey), 1, L.dptr(U), L.dptr(out))
with open("/proc/self/statm") as f:
    used = int(f.read().split()[0]) * resource.getpagesize()
resource.setrlimit(resource.RLIMIT_AS, (used + (1 << 20), resource.RLIM_INFINITY))
rc = conv(a)
resource.setrlimit(resource.RLIMIT_AS, (resource.RLIM_INFINITY, resource.RLIM_INFINITY))
assert rc == 0 and conv(b) == 0 and np.array_equal(a, b)
print("same")
""")
    env = dict(os.environ, RKDG_HOST_THREADS="8", PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, str(prog)], capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0 and r.stdout.strip() == "same", (r.returncode, r.stdout, r.stderr[-1000:])
