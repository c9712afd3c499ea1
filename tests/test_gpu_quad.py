"""The four-lanes-per-element forms (FP64 at P3, with Roe, and for LF on small meshes; the
precision forms at P3) at the sizes where their tiles can go wrong: partial tiles of 16 elements
per wave and 64 or 128 per workgroup, tiles whose edges are all boundary or halo edges, and a
caller order they must leave to the general kernels.  Against the oracle, FP64 at 1e-12."""
import numpy as np
import pytest

from rkdg_heter_calculate_amd import (BASIS_NATIVE, BC_FARFIELD, BC_OUTFLOW, BC_REFLECTION, IC_VORTEX, Batch, Grid,
                                      Solver, vortex_params)
from rkdg_heter_calculate_amd import _lib as L
from helpers import make_pair, rel_l2, vortex_grid, vortex_ic

pytestmark = pytest.mark.gpu
TOL = 1e-12

# triangles: 4, 32, 62, 64, 66, 126, 130, 522 (wave, tile and layout-tile remainders)
SIZES = [(2, 1), (4, 4), (31, 1), (8, 4), (11, 3), (9, 7), (5, 13), (9, 29)]


def noisy_state(s, seed):
    """A state near a uniform flow whose traces differ at every point (native basis)."""
    rng = np.random.default_rng(seed)
    U = 0.02 * rng.uniform(-1, 1, s.state_shape())
    U[:, 0] += np.array([1.0, 0.3, 0.2, 2.6])[:, None]
    return U


@pytest.mark.parametrize("P,flux", [(1, "lf"), (1, "roe"), (2, "lf"), (2, "roe"), (3, "lf"), (3, "roe")])
@pytest.mark.parametrize("bc", [0, BC_FARFIELD, BC_OUTFLOW, BC_REFLECTION])
def test_tile_remainders(P, flux, bc):
    for nx, ny in SIZES:
        if bc == 0 and min(nx, ny) < 3:
            continue  # not a manifold periodic mesh
        print(f"case: quad tiles P{P} {flux} bc {bc} {nx}x{ny}", flush=True)
        g = Grid.splitquad(nx, ny, 0.0, 0.0, 10.0, 10.0 * ny / nx, periodic=bc == 0, diagonal=1, jitter=0.2, seed=nx,
                           bc=bc or BC_OUTFLOW)
        fs = [1.0, 0.3, 0.2, 2.6]
        o, s = make_pair(g, P=P, flux=flux, dt_policy="max", cfl=0.1, freestream=fs)
        s.set_state(noisy_state(s, nx), basis=1)
        o.set_state(s.get_state())
        s.advance(3)
        o.advance(3)
        err = rel_l2(s.get_state(), o.get_state(), o.mass())
        assert np.all(err < TOL), (nx, ny, err)
        assert np.allclose(s.residual(), o.residual_change(), rtol=1e-9, atol=1e-14)
        s.close()


# Three steps at CFL 0.1 move a mode by at most about its deviation (0.06 over the modes, 0.2 the
# smallest mean): bf16 rounds each by 2^-9 twice, 3 * 0.3 * 0.06 * 2^-8 / 0.2 = 1e-3; FP32 rounds
# point values and fluxes up to 3 by 2^-24, 3 * 0.3 * 3 * 2^-24 / 0.2 = 8e-7.
@pytest.mark.parametrize("prec,tol", [("fp32", 1e-6), ("bf16", 1e-3)])
@pytest.mark.parametrize("flux", ["lf", "roe"])
@pytest.mark.parametrize("bc", [0, BC_FARFIELD, BC_OUTFLOW, BC_REFLECTION])
def test_p3_precision_tile_remainders(bc, flux, prec, tol):
    """The P3 precision form's tiles at the same sizes, and (the last) a row-major order whose tiles
    hold more halo edges than the form admits."""
    for nx, ny, row_major in [(*n, False) for n in SIZES] + [(32, 12, True), (44, 12, True)]:
        if bc == 0 and min(nx, ny) < 3:
            continue
        print(f"case: P3 {prec} tiles {flux} bc {bc} {nx}x{ny} row-major {row_major}", flush=True)
        g = Grid.splitquad(nx, ny, 0.0, 0.0, 10.0, 10.0 * ny / nx, periodic=bc == 0, diagonal=1, jitter=0.2, seed=nx,
                           bc=bc or BC_OUTFLOW)
        kw = dict(order=np.arange(g.n_elements, dtype=np.int32)) if row_major else {}
        o, _ = make_pair(g, P=3, flux=flux, dt_policy="max", cfl=0.1, freestream=[1.0, 0.3, 0.2, 2.6])
        s = Solver(g, degree=3, flux=flux, dt_policy="max", cfl=0.1, freestream=[1.0, 0.3, 0.2, 2.6], precision=prec, **kw)
        s.set_state(noisy_state(s, nx), basis=1)
        o.set_state(s.get_state())
        s.advance(3)
        o.advance(3)
        err = rel_l2(s.get_state(), o.get_state(), o.mass())
        assert np.all(err < tol), (nx, ny, err)
        assert np.all(err > 0)
        s.close()


@pytest.mark.parametrize("P,flux", [(2, "roe"), (3, "lf")])
def test_against_the_one_lane_form(P, flux, monkeypatch):
    """The same run with RKDG_QUAD=0: other roundings (the kernels differ), the same scheme."""
    print(f"case: quad against one-lane P{P} {flux}", flush=True)
    g = vortex_grid(45, jitter=0.2, diagonal=1, seed=5)
    kw = dict(degree=P, flux=flux, dt_policy="max", cfl=0.15)
    s = Solver(g, **kw)
    monkeypatch.setenv("RKDG_QUAD", "0")
    r = Solver(g, **kw)
    U0 = noisy_state(s, 3)
    for x in (s, r):
        x.set_state(U0, basis=1)
        x.advance(10)
    Us, Ur = s.get_state(basis=1), r.get_state(basis=1)
    assert not np.array_equal(Us, Ur)
    assert np.linalg.norm(Us - Ur) < 1e-13 * np.linalg.norm(Ur)


@pytest.mark.parametrize("P", [2, 3])
@pytest.mark.parametrize("nx", [32, 33, 64])
def test_row_major_orders_at_the_halo_limit(P, nx):
    """The caller's row-major numbering: a tile of 64 (128) elements is a strip of one or two rows
    with 64-70 (up to 132) tile-boundary edges, on both sides of what the form holds."""
    print(f"case: quad halo limit P{P} nx {nx}", flush=True)
    g = Grid.splitquad(nx, 12, 0.0, 0.0, 10.0, 10.0, periodic=True, diagonal=1, jitter=0.2, seed=3)
    o, s = make_pair(g, P=P, flux="roe", dt_policy="max", cfl=0.1, order=np.arange(g.n_elements, dtype=np.int32))
    s.set_state(noisy_state(s, nx), basis=1)
    o.set_state(s.get_state())
    s.advance(3)
    o.advance(3)
    err = rel_l2(s.get_state(), o.get_state(), o.mass())
    assert np.all(err < TOL), err
    s.close()


def test_an_order_it_does_not_admit_and_an_end_time():
    """A random caller order (tiles with more halo edges than the form holds) runs the general
    kernel; an end time inside the third step clips it."""
    print("case: quad not admitted, end time", flush=True)
    g = vortex_grid(20, jitter=0.2, diagonal=1, seed=2)
    order = np.random.default_rng(0).permutation(g.n_elements).astype(np.int32)
    o, s = make_pair(g, P=3, flux="roe", dt_policy="max", cfl=0.1, order=order)
    U0 = vortex_ic(o)
    s.set_state(U0)
    s.advance(3)
    o.advance(3)
    assert np.all(rel_l2(s.get_state(), o.get_state(), o.mass()) < TOL)
    s.close()
    q = Solver(g, degree=3, flux="roe", dt_policy="max", cfl=0.1)
    q.set_state(U0)
    dt = q.compute_dt()
    n, t = q.advance(10, t_end=2.5 * dt)
    assert n == 3 and abs(t - 2.5 * dt) < 1e-15
    q.close()


@pytest.mark.parametrize("P,flux", [(1, "roe"), (2, "lf"), (2, "roe"), (3, "lf")])
def test_batch_instances_equal_single_meshes(P, flux):
    """A batch without a caller block runs the same tiles as a single mesh (instances start on
    256-element boundaries, so their tiles hold the same elements): the same bits.  24, 130 and 512
    triangles: a partial tile, a partial layout tile and two full ones."""
    print(f"case: quad batch P{P} {flux}", flush=True)
    grids = [Grid.splitquad(nx, ny, 0.0, 0.0, 10.0, 10.0, periodic=True, diagonal=1, jitter=0.2, seed=nx)
             for nx, ny in ((4, 3), (5, 13), (16, 16))]
    kw = dict(degree=P, flux=flux, dt_policy="max", cfl=0.1)
    b = Batch(grids, [kw] * 3)
    assert b.tiles()["staged"] == 2
    singles = [Solver(g, **kw) for g in grids]
    for i, s in enumerate(singles):
        U = noisy_state(s, i)
        b.set_state(i, U, BASIS_NATIVE)
        s.set_state(U, BASIS_NATIVE)
    b.advance(5)
    b.sync()
    for i, s in enumerate(singles):
        s.advance(5)
        assert np.array_equal(b.get_state(i, BASIS_NATIVE), s.get_state(BASIS_NATIVE)), i
        assert b.time(i) == s.time()[0]
    # the configuration reported can be given back, after another one
    default = b.tiles()
    b.set_tiles(0, 256, 8)
    assert b.tiles() == {"staged": 0, "block": 256, "per_cu": 8}
    b.set_tiles(**default)
    assert b.tiles() == default
    for i, s in enumerate(singles):
        b.set_state(i, U := noisy_state(s, i), BASIS_NATIVE)
        s.set_state(U, BASIS_NATIVE)
        s.advance(2)
    b.advance(2)
    b.sync()
    for i, s in enumerate(singles):
        assert np.array_equal(b.get_state(i, BASIS_NATIVE), s.get_state(BASIS_NATIVE)), i
    for block, per_cu in ((64 if P == 3 else 128, 0), (default["block"], 4)):
        with pytest.raises(L.RkdgError):
            b.set_tiles(2, block, per_cu)
    b.close()


def test_the_allocation_free_step_takes_meshes_above_the_small_tiles_limit():
    """4,194,304 elements fill the allocation-free step's 65,536 tiles at 64 elements per tile; a
    larger mesh runs the 256-element tiles and is accepted."""
    print("case: step_noalloc P1 Roe 4,199,202 triangles", flush=True)
    s = Solver(Grid.splitquad(1449, 1449, 0.0, 0.0, 10.0, 10.0, periodic=True), degree=1, flux="roe", dt_policy="max", cfl=0.3)
    s.project_ic(IC_VORTEX, vortex_params())
    dt = s.compute_dt()
    L.check(L.load().rkdg_step_noalloc(s.h, dt, None, None), s.h, "step_noalloc")
    assert np.all(np.isfinite(s.get_state(basis=1)))
    s.close()
