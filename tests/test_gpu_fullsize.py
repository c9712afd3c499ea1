"""GPU against the oracle at the workloads' full sizes (the oracle takes seconds there).

* the 512x512 jittered vortex mesh of the P2 benchmark (seed 2024, 524,288 triangles,
  XCD-remapped sweep, halo capacity checked per tile), 5 steps, in the FP64 form (1e-12) on
  8,192 four-lanes-per-element tiles and on the 2,048 staged tiles that larger meshes run, and
  in the FP32-MFMA form (1e-6, staged tiles);
* the 1024x1024 four-quadrant Riemann mesh (seed 2025, 2,097,152 triangles), P1, Roe,
  TVB M = 50 with positivity scaling, 3 steps (1e-12, equal limiter flags);
* the same problem shrunk to 64x64 and run to t = 0.3 (about 3,500 steps), where the
  limiter's decisions could drift apart: relative L2 and the fraction of equal flags;
* the P3 Roe vortex mesh family at 1024x1024 (seed 2026, 2,097,152 triangles), 2 steps, in the
  FP64 form (1e-12) and the precision form's FP32 (1e-6) and BF16 (2e-4) contractions.
"""
import numpy as np
import pytest

from oracle import pyoracle as po
from rkdg_heter_calculate_amd import IC_RIEMANN4, IC_VORTEX, Solver, vortex_params
from rkdg_heter_calculate_amd.workloads import riemann_p1, vortex_grid, vortex_p3
from helpers import rel_l2

pytestmark = pytest.mark.gpu

_REF = {}


def oracle_for(g, **kw):
    ex, ey = g.element_coords()
    return po.Oracle(ex, ey, g.neighbour, g.shared_edge, g.boundary, **kw)


def vortex_512_reference():
    if "v512" not in _REF:
        g = vortex_grid(512)  # seed 2024, jitter 0.2, seed-chosen diagonals
        o = oracle_for(g, P=2, flux=0, dt_policy=1, cfl=0.3)
        o.project(1, vortex_params())
        U0 = o.get_state()
        n, t, _ = o.advance(5)
        _REF["v512"] = (g, U0, o.get_state(), t, o.mass())
    return _REF["v512"]


@pytest.mark.parametrize("prec,tol,quad", [("fp64", 1e-12, "1"), ("fp64", 1e-12, "0"), ("fp32", 1e-6, "0")])
def test_vortex_p2_512_matches_oracle(prec, tol, quad, monkeypatch):
    print(f"case: 512x512 P2 vortex 5 steps {prec} RKDG_QUAD={quad}", flush=True)
    monkeypatch.setenv("RKDG_QUAD", quad)
    g, U0, Uo, to, M = vortex_512_reference()
    assert g.n_elements == 524288
    s = Solver(g, degree=2, flux="lf", dt_policy="max", cfl=0.3, precision=prec)
    assert tuple(s.tiles().values()) == ((2, 64, 0) if quad == "1" else (1, 256, 0))
    s.set_state(U0)
    n, t = s.advance(5)
    # the time sums CFL dts of cell means: 1e-13 in FP64, the form's bar in FP32
    assert n == 5 and abs(t - to) <= (1e-13 if prec == "fp64" else tol) * to
    Us = s.get_state()
    err = rel_l2(Us, Uo, M)
    linf = [float(np.max(np.abs(Us[v] - Uo[v])) / np.max(np.abs(Uo[v]))) for v in range(4)]
    print("relative L2 per variable", err, "relative Linf", linf, flush=True)
    assert np.all(err < tol), err
    s.close()


def vortex_p3_1024_reference():
    if "p3" not in _REF:
        g, kw, vp, _ = vortex_p3(1024)  # the P3 workload's mesh family at 2.1M triangles
        o = oracle_for(g, P=3, flux=1, dt_policy=1, cfl=kw["cfl"])
        o.project(1, vp)
        U0 = o.get_state()
        n, t, _ = o.advance(2)
        _REF["p3"] = (g, kw, U0, o.get_state(), t, o.mass())
    return _REF["p3"]


@pytest.mark.parametrize("prec,tol", [("fp64", 1e-12), ("fp32", 1e-6), ("bf16", 2e-4)])
def test_vortex_p3_1024_matches_oracle(prec, tol):
    """P3 Roe on 2,097,152 triangles, 2 steps: the four-lanes-per-element tiles of the FP64 form
    and of the precision forms (128 elements, halo capacity checked per tile) against the
    oracle."""
    print(f"case: 1024x1024 P3 Roe vortex 2 steps {prec}", flush=True)
    g, kw, U0, Uo, to, M = vortex_p3_1024_reference()
    assert g.n_elements == 2097152
    s = Solver(g, precision=prec, **kw)
    assert tuple(s.tiles().values()) == (2, 128, 0)
    s.set_state(U0)
    n, t = s.advance(2)
    assert n == 2 and abs(t - to) <= (1e-13 if prec == "fp64" else tol) * to
    Us = s.get_state()
    err = rel_l2(Us, Uo, M)
    print("relative L2 per variable", err, flush=True)
    assert np.all(err < tol), err
    s.close()


def test_riemann_p1_1024_three_steps_match_oracle():
    print("case: 1024x1024 four-quadrant Riemann P1 Roe TVB 3 steps", flush=True)
    g, kw, ic, _ = riemann_p1(1024)
    assert g.n_elements == 2097152
    o = oracle_for(g, P=1, flux=1, limiter=1, dt_policy=1, cfl=kw["cfl"], tvb_M=kw["tvb_M"])
    o.project(2, ic)
    s = Solver(g, **kw)
    s.project_ic(IC_RIEMANN4, ic)
    # exact cell averages on both sides (two clipping codes, exchanged through the element basis)
    assert np.all(rel_l2(s.get_state(), o.get_state(), o.mass()) < 1e-14)
    s.advance(3)
    o.advance(3)
    err = rel_l2(s.get_state(), o.get_state(), o.mass())
    fs, fo = s.flags(), o.flags()
    print("relative L2 per variable", err, "limited cells", int((fo != 0).sum()), flush=True)
    assert np.all(err < 1e-12), err
    assert np.array_equal(fs, fo)
    assert (fo != 0).sum() > 1000  # the limiter is active along the four discontinuities


def test_riemann_p1_64_to_t03_against_oracle():
    """About 3,500 steps through shocks and contacts: limiter decisions switch on round-off
    (the GPU's reciprocal and square root differ from IEEE division in the last bits), and
    the problem amplifies such differences.  The bar is therefore the oracle's own
    sensitivity: the same run with its start state perturbed by 1e-15 (relative, seeded)."""
    print("case: 64x64 four-quadrant Riemann P1 Roe TVB to t = 0.3", flush=True)
    g, kw, ic, t_end = riemann_p1(64)

    def oracle_run(perturb):
        o = oracle_for(g, P=1, flux=1, limiter=1, dt_policy=1, cfl=kw["cfl"], tvb_M=kw["tvb_M"])
        o.project(2, ic)
        if perturb:
            U = o.get_state()
            o.set_state(U * (1 + 1e-15 * np.random.default_rng(1).standard_normal(U.shape)))
        n, t, _ = o.advance(1000000, t_end=t_end)
        return o, n, t

    o, no, to = oracle_run(False)
    p, _, _ = oracle_run(True)
    s = Solver(g, **kw)
    s.project_ic(IC_RIEMANN4, ic)
    n = 0
    t = 0.0
    while t < t_end:
        k, t = s.advance(5000, t_end=t_end)
        n += k
        if k == 0:
            break
    assert n == no and abs(t - to) <= 1e-12
    M = o.mass()
    err = rel_l2(s.get_state(), o.get_state(), M)
    sens = rel_l2(p.get_state(), o.get_state(), M)
    fs, fo, fp = s.flags(), o.flags(), p.flags()
    agree, agree_p = float(np.mean(fs == fo)), float(np.mean(fp == fo))
    print(f"{n} steps to t = {t}: relative L2 per variable {err} (oracle vs its 1e-15 perturbation: {sens}); "
          f"flags agree on {agree:.4f} of the cells ({agree_p:.4f} for the perturbed oracle; "
          f"{int((fo != 0).sum())} limited)", flush=True)
    assert np.all(err < 4 * sens + 1e-9), (err, sens)
    assert agree > 0.97, agree
