"""State exchange on the device: caller order and both bases, transfers below and above the
one-copy limit (1.5 MiB) and the 8 MiB chunks, reads inside a step."""
import ctypes
import math

import numpy as np
import pytest

from rkdg_heter_calculate_amd import BASIS_ELEMENT, BASIS_NATIVE, IC_VORTEX, Batch, Grid, Solver, vortex_params
from rkdg_heter_calculate_amd import _lib as L
from helpers import vortex_grid

pytestmark = pytest.mark.gpu


def random_state(P, E, seed):
    rng = np.random.default_rng(seed)
    U = 0.05 * rng.uniform(-1, 1, (4, (P + 1) * (P + 2) // 2, E))
    U[:, 0] += np.array([1.0, 0.2, -0.1, 2.5])[:, None]
    return U


def host_convert(P, g, U, from_basis):
    ex, ey = (np.ascontiguousarray(a) for a in g.element_coords())
    out = np.empty_like(U)
    assert L.load().rkdg_convert_basis(P, g.n_elements, L.dptr(ex), L.dptr(ey), from_basis, L.dptr(U), L.dptr(out)) == 0
    return out


MX, MY = (0, 1, 0, 2, 1, 0, 3, 2, 1, 0), (0, 0, 1, 0, 1, 2, 0, 1, 2, 3)


def exact_element_basis(P, g, U):
    """Native -> element coefficients in extended precision: the native basis is the Cholesky factor
    of the monomials' moments, the element basis Gram-Schmidt of the scaled monomials, both as
    polynomials in xi, eta with exact moments."""
    ld = np.longdouble
    n = (P + 1) * (P + 2) // 2
    fact = [ld(math.factorial(k)) for k in range(20)]
    moment = lambda a, b: 2 * fact[a] * fact[b] / fact[a + b + 2]  # noqa: E731
    G = np.array([[moment(MX[a] + MX[b], MY[a] + MY[b]) for b in range(n)] for a in range(n)])
    Lc = np.zeros((n, n), ld)
    for i in range(n):
        for j in range(i + 1):
            t = G[i, j] - np.dot(Lc[i, :j], Lc[j, :j])
            Lc[i, j] = np.sqrt(t) if i == j else t / Lc[j, j]
    C = np.zeros((n, n), ld)  # psi_i = sum_m C[i][m] mono_m
    for i in range(n):
        e = np.zeros(n, ld)
        e[i] = 1
        for r in range(n):
            C[r, i] = (e[r] - np.dot(Lc[r, :r], C[:r, i])) / Lc[r, r]
    ex, ey = (c.astype(ld) for c in g.element_coords())
    isq = 1 / np.sqrt(((ex[:, 1] - ex[:, 0]) * (ey[:, 2] - ey[:, 0]) - (ex[:, 2] - ex[:, 0]) * (ey[:, 1] - ey[:, 0])) / 2)
    index = {(MX[m], MY[m]): m for m in range(n)}

    def times(c, x):  # c: coordinate; x: polynomials [n][E]
        d1, d2 = (c[:, 1] - c[:, 0]) * isq, (c[:, 2] - c[:, 0]) * isq
        out = -(d1 + d2) / 3 * x
        for m in range(n):
            if (MX[m] + 1, MY[m]) in index:
                out[index[MX[m] + 1, MY[m]]] += d1 * x[m]
            if (MX[m], MY[m] + 1) in index:
                out[index[MX[m], MY[m] + 1]] += d2 * x[m]
        return out

    inner = lambda a, b: np.einsum("ie,ij,je->e", a, G, b)  # noqa: E731
    parent = (0, 0, 0, 1, 2, 2, 3, 4, 5, 5)
    mono, phi, out = [], [], np.empty(U.shape, ld)
    u = np.einsum("vie,im->vme", U.astype(ld), C)
    for k in range(n):
        if k == 0:
            f = np.zeros((n, g.n_elements), ld)
            f[0] = 1
        else:
            f = times(ey if k in (2, 5, 9) else ex, mono[parent[k]])
        mono.append(f)
        for q in phi:
            f = f - inner(mono[k], q) / inner(q, q) * q
        phi.append(f)
        for v in range(4):
            out[v, k] = inner(u[v], f) / inner(f, f)
    return out


# 4 triangles; 192 B each at P2: 8192 triangles are the 1.5 MiB limit, 87,382 two chunks and a
# rest, 264,992 more chunks than the ring holds
@pytest.mark.parametrize("P,nx,ny", [(1, 2, 1), (2, 64, 64), (2, 17, 241), (2, 43691, 1), (3, 364, 364), (1, 3, 86)])
def test_round_trip_is_exact_in_the_native_basis(P, nx, ny):
    print(f"case: exchange P{P} {nx}x{ny}", flush=True)
    g = Grid.splitquad(nx, ny, 0.0, 0.0, float(nx), float(ny), periodic=False, diagonal=1, jitter=0.2, seed=1)
    s = Solver(g, degree=P)
    U = random_state(P, g.n_elements, nx)
    s.set_state(U, BASIS_NATIVE)
    assert np.array_equal(s.get_state(BASIS_NATIVE), U)
    s.close()


@pytest.mark.parametrize("P", [1, 2, 3])
@pytest.mark.parametrize("ly", [10.0, 3.0])
def test_element_basis_is_no_further_from_exact_than_the_host_conversion(P, ly):
    """The reference's basis is not normalised: on small elements its conversion amplifies
    rounding (7e-11 at P3 here), so the bound is what rkdg_convert_basis (36-point quadrature on
    the host) is off by, and 8 ulp of the largest coefficient where that is less."""
    print(f"case: exchange element basis P{P} {ly}", flush=True)
    g = Grid.splitquad(31, 17, 0.0, 0.0, 10.0, ly, periodic=False, diagonal=1, jitter=0.24, seed=4)
    s = Solver(g, degree=P)
    U = random_state(P, g.n_elements, 3)
    s.set_state(U, BASIS_NATIVE)
    want, host, got = exact_element_basis(P, g, U), host_convert(P, g, U, BASIS_NATIVE), s.get_state(BASIS_ELEMENT)
    floor = 8 * 2.0 ** -52 * float(np.max(np.abs(want)))
    off = [float(np.max(np.abs(x - want))) for x in (host, got)]
    print("host and device are off by", off, flush=True)
    assert off[1] <= max(off[0], floor)
    # and back: a round trip through the element basis
    s.set_state(got, BASIS_ELEMENT)
    back = host_convert(P, g, host, BASIS_ELEMENT)
    assert np.max(np.abs(s.get_state(BASIS_NATIVE) - U)) <= max(np.max(np.abs(back - U)), floor)
    s.close()


def test_batch_instances_keep_to_their_own_block():
    print("case: exchange batch", flush=True)
    grids = [vortex_grid(n, jitter=0.2, diagonal=1, seed=n) for n in (5, 16, 11)]
    b = Batch(grids, [dict(degree=2, dt_policy="max", cfl=0.2)] * 3)
    U = [random_state(2, g.n_elements, i) for i, g in enumerate(grids)]
    for i in (1, 0, 2):
        b.set_state(i, U[i], BASIS_NATIVE)
    for i in range(3):
        assert np.array_equal(b.get_state(i, BASIS_NATIVE), U[i])
        want, host = exact_element_basis(2, grids[i], U[i]), host_convert(2, grids[i], U[i], BASIS_NATIVE)
        assert np.max(np.abs(b.get_state(i, BASIS_ELEMENT) - want)) <= np.max(np.abs(host - want))
    b.close()


@pytest.mark.parametrize("P,prec", [(1, "fp64"), (2, "fp64"), (3, "fp64"), (2, "fp32"), (3, "bf16")])
def test_reading_inside_a_step_changes_nothing(P, prec):
    """get_state and flags after every stage (the latest stage and the step-start state are both
    live then) against the same stages unread."""
    print(f"case: exchange inside a step P{P} {prec}", flush=True)
    g = vortex_grid(24, jitter=0.2, diagonal=1, seed=3)
    kw = dict(degree=P, flux="roe", dt_policy="max", cfl=0.1, precision=prec, limiter=P == 1)
    a, b = Solver(g, **kw), Solver(g, **kw)
    U = random_state(P, g.n_elements, 5)
    for s in (a, b):
        s.set_state(U, BASIS_NATIVE)
    for _ in range(2):
        for st in range(3):
            a.stage(st, 1e-3)
            b.stage(st, 1e-3)
            b.get_state(BASIS_ELEMENT)
            b.flags()
    assert np.array_equal(a.get_state(BASIS_NATIVE), b.get_state(BASIS_NATIVE))
    assert np.array_equal(a.flags(), b.flags())
    a.close()
    b.close()


@pytest.mark.parametrize("P,limiter,n", [(2, False, 64), (1, True, 48), (3, False, 170)])
def test_reading_beside_steps_on_another_stream_changes_nothing(P, limiter, n):
    """get_state and flags while rkdg_step_noalloc works on a caller's stream: what they return is of
    no one stage, but the steps must come out as if unread (the rows have a buffer of their own; at
    P3 here the state crosses one variable at a time)."""
    print(f"case: exchange beside steps P{P}", flush=True)
    lib, hip = L.load(), ctypes.CDLL("libamdhip64.so")
    g = vortex_grid(n, jitter=0.2, diagonal=1, seed=3)
    kw = dict(degree=P, flux="roe", dt_policy="max", cfl=0.1, limiter=limiter)
    a, b = Solver(g, **kw), Solver(g, **kw)
    for s in (a, b):
        s.project_ic(IC_VORTEX, vortex_params())
    dt = a.compute_dt()
    stream = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0
    for _ in range(4):
        for _ in range(100):
            L.check(lib.rkdg_step_noalloc(b.h, dt, None, stream), b.h, "step_noalloc")
        for _ in range(5):
            b.get_state(BASIS_ELEMENT)
            b.flags()
        assert hip.hipStreamSynchronize(stream) == 0
        for _ in range(100):
            L.check(lib.rkdg_step_noalloc(a.h, dt, None, None), a.h, "step_noalloc")
        assert np.array_equal(a.get_state(BASIS_NATIVE), b.get_state(BASIS_NATIVE))
        assert np.array_equal(a.flags(), b.flags())
    assert hip.hipStreamDestroy(stream) == 0
    a.close()
    b.close()
