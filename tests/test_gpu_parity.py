"""GPU (librkdg) against the CPU oracle on the same seeded inputs.

The oracle restates the reference's per-element-basis algorithm; the GPU evolves the
same polynomials in a reference-element basis.  States are compared in the reference's
basis through the library's own exchange (rkdg_get_state, RKDG_BASIS_ELEMENT), with the
relative L2 norm per conserved variable.  Bar: 1e-12 for the plain FP64 form.
"""
import numpy as np
import pytest

from oracle import pyoracle as po
from rkdg_heter_calculate_amd import Grid, Solver, riemann4_params, vortex_params, BC_FARFIELD, BC_OUTFLOW, BC_REFLECTION
from helpers import make_pair, rel_l2, vortex_grid, vortex_ic

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.mark.parametrize("P", [1, 2, 3])
@pytest.mark.parametrize("flux", ["lf", "roe"])
def test_single_stage_matches_oracle(P, flux):
    print(f"case: single stage P{P} {flux}", flush=True)
    g = vortex_grid(8, jitter=0.2, diagonal=1, seed=3)
    o, s = make_pair(g, P=P, flux=flux)
    U0 = vortex_ic(o)
    s.set_state(U0)
    dt = 0.01
    for st in range(3):
        o.stage(st, dt)
        s.stage(st, dt)
        err = rel_l2(s.get_state(), o.get_state(), o.mass())
        assert np.all(err < TOL), (st, err)


def test_reference_workload_100_steps():
    """64x64 periodic split-quad vortex, P1, LF, CFL 0.3, reference dt subset, 100 steps."""
    print("case: 64x64 P1 vortex 100 steps", flush=True)
    g = vortex_grid(64)
    o, s = make_pair(g, P=1, flux="lf", dt_policy="reference", cfl=0.3)
    U0 = vortex_ic(o)
    s.set_state(U0)
    assert abs(s.compute_dt() - o.compute_dt()) <= 1e-14 * o.compute_dt()
    n, t = s.advance(100)
    no, to, _ = o.advance(100)
    assert n == 100 and no == 100
    assert abs(t - to) <= 1e-12 * to
    err = rel_l2(s.get_state(), o.get_state(), o.mass())
    print("relative L2 per variable", err)
    assert np.all(err < TOL), err


@pytest.mark.parametrize("P", [2, 3])
def test_jittered_steps(P):
    print(f"case: jittered P{P} 10 steps", flush=True)
    g = vortex_grid(16, jitter=0.2, diagonal=1, seed=11)
    o, s = make_pair(g, P=P, flux="lf", dt_policy="max", cfl=0.3)
    s.set_state(vortex_ic(o))
    s.advance(10)
    o.advance(10)
    err = rel_l2(s.get_state(), o.get_state(), o.mass())
    assert np.all(err < TOL), err


@pytest.mark.parametrize("P,prec", [(2, "fp64"), (1, "fp64"), (3, "fp64"), (2, "fp32"), (3, "fp32"), (2, "bf16"),
                                    (3, "bf16")])
def test_boundaries_match_oracle(P, prec):
    """Far-field, wall and transmissive edges (per-edge treatment of the ghost kernel), in the
    FP64 kernels and in the precision kernels (one partial 256-element tile).  BF16: 1e-3
    relative L2 per variable (measured 0.6-4.4e-4; the free stream's rho v is a fifth of its
    rho u, so the same absolute error, 0.4-2.6e-4 over the four variables, is a larger
    fraction of it than on the vortex workloads' 2e-4 bar), the residual of the means to 2e-2."""
    print(f"case: boundaries P{P} {prec}", flush=True)
    g = Grid.splitquad(12, 10, 0.0, 0.0, 10.0, 8.0, periodic=False, diagonal=1, jitter=0.15, seed=5)
    bnd = g.boundary.copy()
    # left/bottom far field, top wall, right transmissive
    ex, ey = g.element_coords()
    for e in range(g.n_elements):
        for k in range(3):
            if g.neighbour[e, k] < 0:
                mx = 0.5 * (ex[e, (k + 1) % 3] + ex[e, (k + 2) % 3])
                my = 0.5 * (ey[e, (k + 1) % 3] + ey[e, (k + 2) % 3])
                bnd[e, k] = BC_FARFIELD if (mx < 1e-9 or my < 1e-9) else (BC_REFLECTION if my > 8 - 1e-9 else BC_OUTFLOW)
    g.boundary = bnd
    fs = (1.0, 0.5, 0.1, 2.63)
    for flux in ("lf", "roe"):
        o, s = make_pair(g, P=P, flux=flux, dt_policy="max", cfl=0.2 if P < 3 else 0.1, freestream=fs)
        if prec != "fp64":
            s = Solver(g, degree=P, flux=flux, dt_policy="max", cfl=0.2 if P < 3 else 0.1, precision=prec,
                       freestream=fs)
        vp = vortex_params(uinf=0.5, vinf=0.1, xc=4.0, yc=4.0, lx=0.0, ly=0.0)
        o.project(1, vp)
        s.set_state(o.get_state())
        s.advance(8)
        o.advance(8)
        err = rel_l2(s.get_state(), o.get_state(), o.mass())
        print(f"{flux}: relative L2 per variable {err}", flush=True)
        assert np.all(err < {"fp64": TOL, "fp32": MX_TOL, "bf16": 1e-3}[prec]), (flux, err)
        print("residual of the means, GPU and oracle:", s.residual(), o.residual_change(), flush=True)
        # the reference's residual (max change of the rho and rhoE means), reduced over tiles
        assert np.allclose(s.residual(), o.residual_change(), rtol={"fp64": 1e-9, "fp32": 1e-3, "bf16": 2e-2}[prec],
                           atol=1e-15)


def test_limiter_matches_oracle():
    print("case: TVB limiter", flush=True)
    g = Grid.splitquad(24, 24, 0.0, 0.0, 1.0, 1.0, periodic=False, diagonal=1, jitter=0.2, seed=9)
    o, s = make_pair(g, P=1, flux="roe", limiter=True, dt_policy="max", cfl=0.2, tvb_M=50.0)
    o.project(2, riemann4_params())
    s.set_state(o.get_state())
    s.advance(6)
    o.advance(6)
    err = rel_l2(s.get_state(), o.get_state(), o.mass())
    print("relative L2 per variable", err, flush=True)
    assert np.all(err < 1e-12), err
    assert np.array_equal(s.flags(), o.flags())


def test_locality_order_is_transparent():
    print("case: reordering", flush=True)
    g = vortex_grid(20, jitter=0.2, diagonal=1, seed=2)
    o, s = make_pair(g, P=2, dt_policy="reference", cfl=0.3)
    U0 = vortex_ic(o)
    rng = np.random.default_rng(0)
    order = rng.permutation(g.n_elements).astype(np.int32)
    s2 = Solver(g, order=order, degree=2, dt_policy="reference", cfl=0.3)
    s.set_state(U0)
    s2.set_state(U0)
    s.advance(5)
    s2.advance(5)
    err = rel_l2(s2.get_state(), s.get_state(), o.mass())
    assert np.all(err < 1e-14), err


def test_run_twice_bitwise():
    print("case: determinism", flush=True)
    g = vortex_grid(32, jitter=0.2, diagonal=1, seed=4)
    o, s = make_pair(g, P=2)
    U0 = vortex_ic(o)
    s.set_state(U0)
    s.advance(7)
    a = s.get_state(basis=1)
    s.set_state(U0)
    s.advance(7)
    b = s.get_state(basis=1)
    assert np.array_equal(a, b)


@pytest.mark.parametrize("P", [2, 1])  # (the other FP64 forms: test_gpu_forms.py)
def test_advance_counts_steps_per_call(P):
    print(f"case: advance step counts and end time P{P}", flush=True)
    g = vortex_grid(16, jitter=0.2, diagonal=1, seed=5)
    s = Solver(g, degree=P, dt_policy="fixed", dt_fixed=1e-3)
    s.project_ic(1, vortex_params())
    n1, t1 = s.advance(5)
    n2, t2 = s.advance(5)
    assert (n1, n2) == (5, 5)
    assert abs(t1 - 5e-3) < 1e-15 and abs(t2 - 1e-2) < 1e-15
    # an end time inside the next steps stops the run there, the last step clipped
    n3, t3 = s.advance(50, t_end=0.0125)
    assert n3 == 3 and abs(t3 - 0.0125) < 1e-15
    n4, t4 = s.advance(10, t_end=0.0125)
    assert n4 == 0 and t4 == t3
    s.close()


def test_p1_pipelined_tiles_match_oracle(monkeypatch):
    """P1 LF FP64 above 65,536 elements runs the register-pipelined persistent tile (next tile's image loaded into
    registers during the current tile). 528 full tiles and a partial one on 256 workgroups
    (RKDG_PERSIST=1 on a 256-CU part) give each workgroup two or three tiles, so the
    prefetch chain (data one tile ahead, halo ids two, halo offsets three) runs; the result
    must equal the one-tile-per-workgroup staged kernel bit for bit and the oracle to 1e-12."""
    print("case: P1 LF pipelined persistent tiles", flush=True)
    g = Grid.splitquad(260, 260, 0.0, 0.0, 10.0, 10.0, periodic=True, diagonal=1, jitter=0.2, seed=21)
    assert g.n_elements == 135200
    monkeypatch.setenv("RKDG_PERSIST", "1")
    o, s = make_pair(g, P=1, flux="lf", dt_policy="max", cfl=0.3)
    monkeypatch.setenv("RKDG_PIPE", "0")
    monkeypatch.delenv("RKDG_PERSIST")
    r = Solver(g, degree=1, flux="lf", dt_policy="max", cfl=0.3)
    o.project(1, vortex_params())
    U0 = o.get_state()
    s.set_state(U0)
    r.set_state(U0)
    s.advance(4)
    r.advance(4)
    o.advance(4)
    assert np.array_equal(s.get_state(), r.get_state())
    err = rel_l2(s.get_state(), o.get_state(), o.mass())
    assert np.all(err < TOL), err
    assert np.allclose(s.residual(), o.residual_change(), rtol=1e-9, atol=1e-15)


@pytest.mark.parametrize("P,flux", [(2, "lf"), (2, "roe"), (1, "roe")])
def test_pipelined_image_tiles_match_staged_and_oracle(monkeypatch, P, flux):
    """RKDG_PIPE=1: persistent staged tiles whose next image is requested during the current
    tile's update (step-start loads first, then a fixed count of direct loads).  529 tiles on
    256 workgroups (RKDG_PERSIST=1) give each workgroup two or three tiles, so both the
    prefetching body and the last-tile body run; against the one-tile-per-workgroup staged
    kernel (same arithmetic, evaluated one edge point at a time) and the oracle."""
    print(f"case: pipelined image tiles P{P} {flux}", flush=True)
    g = Grid.splitquad(260, 260, 0.0, 0.0, 10.0, 10.0, periodic=True, diagonal=1, jitter=0.2, seed=22)
    monkeypatch.setenv("RKDG_PIPE", "1")
    monkeypatch.setenv("RKDG_PERSIST", "1")
    o, s = make_pair(g, P=P, flux=flux, dt_policy="max", cfl=0.3)
    monkeypatch.setenv("RKDG_PIPE", "0")
    monkeypatch.delenv("RKDG_PERSIST")
    r = Solver(g, degree=P, flux=flux, dt_policy="max", cfl=0.3)
    o.project(1, vortex_params())
    U0 = o.get_state()
    s.set_state(U0)
    r.set_state(U0)
    s.advance(4)
    r.advance(4)
    o.advance(4)
    Us, Ur = s.get_state(), r.get_state()
    print("equal to the staged kernel bit for bit:", bool(np.array_equal(Us, Ur)), flush=True)
    assert np.all(rel_l2(Us, Ur, o.mass()) < 1e-14)
    err = rel_l2(Us, o.get_state(), o.mass())
    assert np.all(err < TOL), err
    (ts, ns), (tr, nr) = s.time(), r.time()
    assert ns == nr == 4 and abs(ts - tr) <= 1e-13 * tr
    assert np.allclose(s.residual(), o.residual_change(), rtol=1e-9, atol=1e-15)
    s.close()
    r.close()


def test_timed_steps_equal_advance():
    """The measurement entry point rkdg_time_steps takes exactly the steps of rkdg_advance
    (graph-replayed pairs after an odd step count, device dt)."""
    print("case: time_steps vs advance", flush=True)
    g = vortex_grid(16, jitter=0.2, diagonal=1, seed=6)
    a = Solver(g, degree=2, dt_policy="max", cfl=0.3)
    b = Solver(g, degree=2, dt_policy="max", cfl=0.3)
    for s in (a, b):
        s.project_ic(1, vortex_params())
        s.advance(1)
    a.advance(7)
    ms = b.time_steps(7)
    assert ms > 0
    assert np.array_equal(a.get_state(), b.get_state())
    assert a.time() == b.time()
    a.close()
    b.close()


@pytest.mark.parametrize("P,staged", [(2, False), (2, True), (1, True), (3, False)])
def test_batch_equals_single(P, staged, monkeypatch):
    print(f"case: batch vs single P{P} staged={staged}", flush=True)
    if staged:
        monkeypatch.setenv("RKDG_BATCH_STAGED", "1")  # the batch's staged tiles from the start
    import ctypes
    from rkdg_heter_calculate_amd import _lib as L
    from rkdg_heter_calculate_amd.solver import make_params, mesh_view
    lib = L.load()
    grids = [vortex_grid(n, jitter=0.2, diagonal=1, seed=n) for n in (6, 11, 17)]
    meshes = (L.Mesh * 3)()
    views = [mesh_view(gr) for gr in grids]
    for i, v in enumerate(views):
        meshes[i] = v
    params = (L.Params * 3)()
    cfl0 = 0.25 if P <= 2 else 0.15  # inside each degree's stable range
    for i in range(3):
        params[i] = make_params(degree=P, dt_policy="max", cfl=cfl0 + 0.02 * i)
    h = ctypes.c_void_p()
    L.bcheck(lib.rkdg_batch_create(3, meshes, params, ctypes.byref(h)), None, "batch_create")
    vp = np.array(vortex_params(), dtype=np.float64)
    for i in range(3):
        L.bcheck(lib.rkdg_batch_project_ic(h, i, 1, L.dptr(vp), len(vp)), h, "project")
    L.bcheck(lib.rkdg_batch_advance(h, 9, 1), h, "advance")
    L.bcheck(lib.rkdg_batch_sync(h), h, "sync")
    for i, gr in enumerate(grids):
        s = Solver(gr, degree=P, dt_policy="max", cfl=cfl0 + 0.02 * i)
        s.project_ic(1, vortex_params())
        s.advance(9)
        Np = (P + 1) * (P + 2) // 2
        Ub = np.empty((4, Np, gr.n_elements))
        L.bcheck(lib.rkdg_batch_get_state(h, i, 1, L.dptr(Ub)), h, "get")
        # both are FP64 forms of the same scheme; they may fuse multiply-adds differently
        Us = s.get_state(basis=1)
        for v in range(4):
            assert np.linalg.norm(Ub[v] - Us[v]) <= 1e-13 * np.linalg.norm(Us[v]), (i, v)
    lib.rkdg_batch_destroy(h)


def naca_files(tmp_path):
    import os
    from test_host import write_reference_mesh
    d = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "naca_grid.npz"))
    return write_reference_mesh(tmp_path, d)


@pytest.mark.parametrize("rhoref,pref", [(1.0, 1.0), (1.3, 2.0)])
def test_naca_reference_case_matches_oracle(tmp_path, rhoref, pref):
    """The reference's own case: NACA0012, Mach 0.4, alpha 5 deg, CFL 0.18, P2, LF, far field
    and slip walls from the barycentre box, reference dt subset, 11 steps.  With rho_ref != 1
    the start state keeps the reference's p / (rho_ref (gamma - 1)) energy
    (src/cudarkdgsolver.cu:354) while the far field uses p / (gamma - 1)
    (src/rkdgadvance.cpp:34)."""
    print(f"case: NACA0012 reference case rhoref={rhoref} pref={pref}", flush=True)
    from rkdg_heter_calculate_amd import IC_FREESTREAM, freestream_state
    conf, part = naca_files(tmp_path)
    g = Grid.read(conf, part, box=15.0)
    fs = freestream_state(1.4, 5.0, 0.4, rhoref, pref)
    o, s = make_pair(g, P=2, flux="lf", dt_policy="reference", cfl=0.18, freestream=fs)
    ic = [1.4, 5.0 * np.arctan(1.0) * 4 / 180, 0.4, rhoref, pref]
    o.project(0, ic)
    s.project_ic(IC_FREESTREAM, ic)
    # the exchange through the element basis is an L2 projection: round-off in the modes
    assert np.allclose(s.get_state(), o.get_state(), rtol=0, atol=1e-13 * max(1.0, np.abs(o.get_state()).max()))
    for _ in range(11):
        dto = o.compute_dt()
        assert abs(s.step() - dto) <= 1e-12 * dto
        o.advance(1)
    err = rel_l2(s.get_state(), o.get_state(), o.mass())
    print("relative L2 per variable", err)
    assert np.all(err < TOL), err
    # the reference's residual: max change of the rho / rhoE means over the last step
    assert np.allclose(s.residual(), o.residual_change(), rtol=1e-9, atol=1e-15)


def test_solver_driver_runs_reference_case(tmp_path):
    print("case: rkdg_solver driver", flush=True)
    import os
    import subprocess
    from rkdg_heter_calculate_amd import IC_FREESTREAM
    conf, part = naca_files(tmp_path)
    main = tmp_path / "main.conf"
    main.write_text(f"title naca\ngamma 1.4\nalpha 5.0\nmach 0.4\ncfl 0.18\nrhoref 1.0\npref 1.0\ntime 1\n"
                    f"gridconf {conf}\nsolutionfile {tmp_path}/solution.plt\nlogfile {tmp_path}/log.dat\n"
                    f"residualfile {tmp_path}/residual.dat\nprintinterval 100\nloghistory Y\n"
                    f"threadsperblock 512\nreductionthreads 512\n")
    exe = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rkdg_heter_calculate_amd",
                       "bin", "rkdg_solver")
    r = subprocess.run([exe, str(main), "--partition", part, "--dump", str(tmp_path / "state.bin"), "--quiet"],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    res = (tmp_path / "residual.dat").read_text().splitlines()
    assert res[0] == "N, rho" and len(res) == 12 and res[-1].startswith("11 ")
    plt = (tmp_path / "solution.plt").read_text().splitlines()
    assert plt[0] == "TITLE=RKDG" and "E= 9340" in plt[2]
    # the dumped state equals the API's result for the same case
    g = Grid.read(conf, part, box=15.0)
    s = Solver(g, order=g.locality_order(), degree=2, dt_policy="reference", cfl=0.18)
    s.project_ic(IC_FREESTREAM, [1.4, 5.0 * np.arctan(1.0) * 4 / 180, 0.4, 1.0, 1.0])
    s.advance(11)
    from rkdg_heter_calculate_amd import _lib as L
    import ctypes
    U = np.zeros((4, 6, g.n_elements))
    t = ctypes.c_double()
    L.check(L.load().rkdg_load_state(str(tmp_path / "state.bin").encode(), 6, g.n_elements, ctypes.byref(t),
                                     L.dptr(U)), None, "load")
    Us = s.get_state()
    assert np.allclose(U, Us, rtol=1e-13, atol=1e-14)


# ---- precision form: FP32 MFMA contractions, FP64 state / means / update ----------------
MX_TOL = 1e-6  # relative L2 per variable against the FP64 oracle


@pytest.mark.parametrize("P", [1, 2, 3])
@pytest.mark.parametrize("flux", ["lf", "roe"])
def test_precision_form_single_stage(P, flux):
    print(f"case: FP32-MFMA single stage P{P} {flux}", flush=True)
    g = vortex_grid(8, jitter=0.2, diagonal=1, seed=3)
    o, _ = make_pair(g, P=P, flux=flux)
    U0 = vortex_ic(o)
    s = Solver(g, degree=P, flux=flux, dt_policy="max", cfl=0.3, precision="fp32")
    s.set_state(U0)
    for st in range(3):
        o.stage(st, 0.01)
        s.stage(st, 0.01)
        err = rel_l2(s.get_state(), o.get_state(), o.mass())
        assert np.all(err < MX_TOL), (st, err)
        assert np.all(err > 0)  # really computed in reduced precision


def test_precision_form_vortex_steps():
    print("case: FP32-MFMA 50 steps P2", flush=True)
    g = vortex_grid(32, jitter=0.2, diagonal=1, seed=5)
    o, _ = make_pair(g, P=2, flux="lf", dt_policy="max", cfl=0.3)
    s = Solver(g, degree=2, flux="lf", dt_policy="max", cfl=0.3, precision="fp32")
    s.set_state(vortex_ic(o))
    s.advance(50)
    o.advance(50)
    err = rel_l2(s.get_state(), o.get_state(), o.mass())
    print("relative L2 vs FP64 oracle", err)
    assert np.all(err < MX_TOL), err


@pytest.mark.parametrize("P,flux", [(2, "roe"), (3, "lf"), (3, "roe")])
def test_precision_form_staged_tiles_with_halos(P, flux):
    """The precision kernels (P2: lane per element on 256-element tiles; P3: four lanes per element
    on 128-element tiles) on a mesh of several tiles (halos gathered from other tiles, padded
    lanes in the last tile): 10 steps against the oracle."""
    print(f"case: FP32-MFMA staged tiles P{P} {flux}", flush=True)
    g = vortex_grid(20, jitter=0.2, diagonal=1, seed=13)  # 800 triangles: 4 tiles, the last one partial
    o, _ = make_pair(g, P=P, flux=flux, dt_policy="max", cfl=0.2)
    U0 = vortex_ic(o)  # (projects into the oracle's state)
    s = Solver(g, degree=P, flux=flux, dt_policy="max", cfl=0.2, precision="fp32")
    s.set_state(U0)
    s.advance(10)
    o.advance(10)
    err = rel_l2(s.get_state(), o.get_state(), o.mass())
    print("relative L2 vs FP64 oracle", err)
    assert np.all(err < MX_TOL), err
    assert np.all(err > 0)
    assert np.allclose(s.residual(), o.residual_change(), rtol=1e-3, atol=1e-15)
    assert tuple(s.tiles().values()) == ((2, 128, 0) if P == 3 else (1, 256, 0))
    # the 64-element form (RKDG_PX=0) rounds differently: a different result shows that the
    # tiles' kernel ran
    import os
    os.environ["RKDG_PX"] = "0"
    try:
        m = Solver(g, degree=P, flux=flux, dt_policy="max", cfl=0.2, precision="fp32")
    finally:
        del os.environ["RKDG_PX"]
    m.set_state(U0)
    m.advance(10)
    assert not np.array_equal(m.get_state(), s.get_state())
    assert np.all(rel_l2(m.get_state(), o.get_state(), o.mass()) < MX_TOL)


def test_precision_form_boundaries_and_limiter():
    print("case: FP32-MFMA boundaries + limiter", flush=True)
    g = Grid.splitquad(24, 24, 0.0, 0.0, 1.0, 1.0, periodic=False, diagonal=1, jitter=0.2, seed=9)
    o, _ = make_pair(g, P=1, flux="roe", limiter=True, dt_policy="max", cfl=0.2)
    o.project(2, riemann4_params())
    s = Solver(g, degree=1, flux="roe", limiter=True, dt_policy="max", cfl=0.2, precision="fp32")
    s.set_state(o.get_state())
    s.advance(5)
    o.advance(5)
    err = rel_l2(s.get_state(), o.get_state(), o.mass())
    assert np.all(err < 1e-5), err


@pytest.mark.parametrize("P", [1, 2, 3])
def test_precision_form_batch_equals_single(P):
    print(f"case: FP32-MFMA batch vs single P{P}", flush=True)
    import ctypes
    from rkdg_heter_calculate_amd import _lib as L
    from rkdg_heter_calculate_amd.solver import make_params, mesh_view
    lib = L.load()
    grids = [vortex_grid(n, jitter=0.2, diagonal=1, seed=n) for n in (7, 12)]
    meshes = (L.Mesh * 2)()
    views = [mesh_view(gr) for gr in grids]
    for i, v in enumerate(views):
        meshes[i] = v
    params = (L.Params * 2)()
    cfl = 0.3 if P <= 2 else 0.2
    for i in range(2):
        params[i] = make_params(degree=P, dt_policy="max", cfl=cfl, precision="fp32")
    h = ctypes.c_void_p()
    L.bcheck(lib.rkdg_batch_create(2, meshes, params, ctypes.byref(h)), None, "batch_create")
    vp = np.array(vortex_params(), dtype=np.float64)
    for i in range(2):
        L.bcheck(lib.rkdg_batch_project_ic(h, i, 1, L.dptr(vp), len(vp)), h, "project")
    L.bcheck(lib.rkdg_batch_advance(h, 6, 1), h, "advance")
    L.bcheck(lib.rkdg_batch_sync(h), h, "sync")
    for i, gr in enumerate(grids):
        s = Solver(gr, degree=P, dt_policy="max", cfl=cfl, precision="fp32")
        s.project_ic(1, vortex_params())
        s.advance(6)
        Ub = np.empty((4, (P + 1) * (P + 2) // 2, gr.n_elements))
        L.bcheck(lib.rkdg_batch_get_state(h, i, 1, L.dptr(Ub)), h, "get")
        Us = s.get_state(basis=1)
        if P <= 2:
            # both run the same staged MFMA tile kernel on the same tiles
            assert np.array_equal(Ub, Us), i
        else:
            # P3: the batch runs four lanes per element, the single solver the FP32 image
            # tiles; two FP32 forms of one scheme, each within 1e-6 of the FP64 form
            for v in range(4):
                assert np.linalg.norm(Ub[v] - Us[v]) <= 2e-6 * np.linalg.norm(Us[v]), (i, v)
    lib.rkdg_batch_destroy(h)


class _TinyGrid:
    """A hand-made mesh: one triangle with a far-field, a slip-wall and a transmissive edge."""

    def __init__(self):
        self.vx = np.array([0.0, 1.0, 0.2])
        self.vy = np.array([0.0, 0.1, 0.9])
        self.tri = np.array([[0, 1, 2]], dtype=np.int32)
        self.neighbour = np.full((1, 3), -1, dtype=np.int32)
        self.shared_edge = np.zeros((1, 3), dtype=np.int32)
        self.boundary = np.array([[BC_FARFIELD, BC_REFLECTION, BC_OUTFLOW]], dtype=np.int32)
        self.n_elements, self.n_vertices = 1, 3

    def element_coords(self):
        return self.vx[self.tri], self.vy[self.tri]


@pytest.mark.parametrize("P", [1, 2, 3])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_tiny_meshes_match_oracle(P, prec):
    """The smallest inputs: one triangle (every edge a different boundary kind) and one split
    quad (two triangles, far field): a tile of one or two live lanes and 255 padded ones."""
    print(f"case: tiny meshes P{P} {prec}", flush=True)
    fs = (1.0, 0.3, -0.2, 2.6)
    for g in (_TinyGrid(), Grid.splitquad(1, 1, 0.0, 0.0, 1.0, 1.0, periodic=False, diagonal=1, bc=BC_FARFIELD)):
        o, s = make_pair(g, P=P, flux="roe", dt_policy="max", cfl=0.1, freestream=fs)
        if prec == "fp32":
            s = Solver(g, degree=P, flux="roe", dt_policy="max", cfl=0.1, precision="fp32", freestream=list(fs))
        o.project(1, vortex_params(uinf=0.3, vinf=-0.2, xc=0.4, yc=0.4, lx=0.0, ly=0.0, beta=1.0))
        s.set_state(o.get_state())
        s.advance(3)
        o.advance(3)
        err = rel_l2(s.get_state(), o.get_state(), o.mass())
        assert np.all(err < (TOL if prec == "fp64" else MX_TOL)), (g.n_elements, err)


def test_non_physical_state_is_reported_with_the_element():
    """A negative density mean is reported as RKDG_ERR_NONPHYSICAL naming the caller's element
    (the device position maps back through the locality order); a batch names the instance."""
    print("case: non-physical state report", flush=True)
    import ctypes
    from rkdg_heter_calculate_amd import _lib as L
    from rkdg_heter_calculate_amd.solver import make_params, mesh_view
    g = vortex_grid(8, jitter=0.2, diagonal=1, seed=9)
    s = Solver(g, degree=2, dt_policy="max", cfl=0.3)
    s.project_ic(1, vortex_params())
    U = s.get_state()
    U[0, 0, 37] = -0.5
    with pytest.raises(L.RkdgError) as ei:
        s.set_state(U)
    assert ei.value.code == L.ERR_NONPHYSICAL and "element 37" in str(ei.value), str(ei.value)
    s.close()
    lib = L.load()
    grids = [vortex_grid(6, seed=1), g]
    views = [mesh_view(x) for x in grids]
    meshes = (L.Mesh * 2)(*views)
    params = (L.Params * 2)(*[make_params(degree=2, dt_policy="max", cfl=0.3) for _ in grids])
    h = ctypes.c_void_p()
    L.bcheck(lib.rkdg_batch_create(2, meshes, params, ctypes.byref(h)), None, "batch_create")
    vp = np.array(vortex_params(), dtype=np.float64)
    L.bcheck(lib.rkdg_batch_project_ic(h, 0, 1, L.dptr(vp), len(vp)), h, "project")
    Ub = np.ascontiguousarray(U)
    rc = lib.rkdg_batch_set_state(h, 1, 1, L.dptr(Ub))
    if rc == 0:
        rc = lib.rkdg_batch_sync(h)
    msg = lib.rkdg_batch_last_error(h).decode()
    lib.rkdg_batch_destroy(h)
    assert rc == L.ERR_NONPHYSICAL and "instance 1" in msg, (rc, msg)


def test_compute_dt_leaves_time_and_step_count():
    """rkdg_compute_dt on a live context refreshes only the CFL reduction: the simulated
    time and step count stay, and the next step takes the dt it returned."""
    print("case: compute_dt on a live context", flush=True)
    g = vortex_grid(12, jitter=0.2, diagonal=1, seed=5)
    o, s = make_pair(g, P=2, flux="lf", dt_policy="max", cfl=0.3)
    s.set_state(vortex_ic(o))
    s.advance(5)
    t0, n0 = s.time()
    dt = s.compute_dt()
    assert s.time() == (t0, n0)
    assert s.step() == dt
    t1, n1 = s.time()
    assert n1 == n0 + 1 and abs(t1 - (t0 + dt)) <= 1e-15 * t1
    o.advance(5)
    assert abs(o.compute_dt() - dt) <= 1e-13 * dt


def test_tiles_whose_halo_does_not_fit_the_staged_image():
    """A caller order that keeps the mesh's row-major numbering: 256 consecutive elements of a
    64x64 split-quad mesh span two rows, so a tile's halo (about 130 elements) exceeds the 96
    slots of the staged LDS image.  FP64 runs the global-gather tiles, the FP32 precision form
    the four-lanes-per-element kernel, both against the oracle; BF16, which needs the staged
    tiles, is refused with an error instead of running anything else."""
    print("case: halo beyond the staged image (identity order, 64x64)", flush=True)
    g = vortex_grid(64, jitter=0.2, diagonal=1, seed=17)
    order = np.arange(g.n_elements, dtype=np.int32)
    o, s = make_pair(g, P=2, flux="lf", dt_policy="max", cfl=0.3, order=order)
    U0 = vortex_ic(o)
    s.set_state(U0)
    s.advance(5)
    o.advance(5)
    err = rel_l2(s.get_state(), o.get_state(), o.mass())
    print("fp64 relative L2", err, flush=True)
    assert np.all(err < TOL), err
    s.close()
    f = Solver(g, order=order, degree=2, flux="lf", dt_policy="max", cfl=0.3, precision="fp32")
    f.set_state(U0)
    f.advance(5)
    err = rel_l2(f.get_state(), o.get_state(), o.mass())
    print("fp32 relative L2", err, flush=True)
    assert np.all(err < MX_TOL), err
    f.close()
    with pytest.raises(Exception, match="halo does not fit"):
        Solver(g, order=order, degree=2, flux="lf", dt_policy="max", cfl=0.3, precision="bf16")


@pytest.mark.parametrize("P", [1, 2, 3])
def test_limiter_branches_match_oracle(P):
    """One stage of dt = 0 (LF, whose wave speed takes cell means only) applies the limiter to the
    start state: cells within M h^2, beyond it, near vacuum and with negative pressures at points,
    so that every combination of its two halves is entered and left out, flags included."""
    print(f"case: limiter branches P{P}", flush=True)
    g = Grid.splitquad(24, 19, 0.0, 0.0, 1.0, 1.0, periodic=False, diagonal=1, jitter=0.2, seed=9)
    o, s = make_pair(g, P=P, flux="lf", limiter=True, dt_policy="max", cfl=0.1, tvb_M=50.0)
    rng = np.random.default_rng(P)
    E = g.n_elements
    U = rng.uniform(-1, 1, s.state_shape())
    U *= (10.0 ** rng.uniform(-6, -0.5, E))[None, None, :]   # deviations from tiny to a third of the mean
    rho = 10.0 ** rng.uniform(-2, 0, E)
    p = 10.0 ** rng.uniform(-5, 2, E)
    U *= rho[None, None, :]
    U[0, 0], U[1, 0], U[2, 0] = rho, 0.3 * rho, -0.2 * rho
    U[3, 0] = p / 0.4 + 0.5 * rho * 0.13
    U[:3, 1:, :E // 3] = 0.0  # a third with smooth density and momentum: limited in rho E, not scaled
    U[3, 1:, :E // 3] = 0.02 * U[3, 0, :E // 3] * rng.uniform(-1, 1, U[3, 1:, :E // 3].shape)
    s.set_state(U, basis=1)
    o.set_state(s.get_state())
    s.stage(0, 0.0)
    o.stage(0, 0.0)
    fs, fo = s.flags(), o.flags()
    assert set(np.unique(fo)) == {0, 1, 2, 3}
    assert np.array_equal(fs, fo)
    err = rel_l2(s.get_state(), o.get_state(), o.mass())
    assert np.all(err < TOL), err
    s.close()
