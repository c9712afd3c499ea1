"""The limiter where its shortcuts could decide differently from the full evaluation."""
from decimal import Decimal, getcontext
from fractions import Fraction

import numpy as np
import pytest

from rkdg_heter_calculate_amd import BASIS_NATIVE, Grid, Solver, riemann4_params
from helpers import make_pair, rel_l2, vortex_grid

pytestmark = pytest.mark.gpu


def near_vacuum(E):
    """P1 states with one density mode, whose density at two edge points is about 1e-9 of the mean
    and whose pressure there is about -5e-8 (exact arithmetic): rho = 1 + T c there, momentum m and
    energy 1 constant.  Kept are modes whose product T c rounds towards zero: 1 - fl(T |c|), the
    density that a bound over all points forms, is then above the exact one, by up to 1e-16, which is
    1e-7 of it, and its kinetic energy below the energy."""
    getcontext().prec = 60
    cp = Fraction(0.5 + float(np.sqrt(15.0)) / 10.0)  # the edge rule's outer point
    T = float(Fraction(Decimal(18).sqrt()) * (cp - Fraction(1, 3)))  # psi_1 there
    rng = np.random.default_rng(7)
    U = np.zeros((4, 3, E))
    U[0, 0] = U[3, 0] = 1.0
    n = 0
    while n < E:
        c = (1.0 - rng.uniform(0.8e-9, 1.2e-9)) / T
        rho, bound = 1 - Fraction(T) * Fraction(c), 1 - Fraction(T * c)
        x = (bound - rho) / rho
        if x < Fraction(4, 10 ** 8):
            continue
        m = float((Decimal(2 * rho.numerator) / Decimal(rho.denominator) *
                   (1 + Decimal(x.numerator) / Decimal(2 * x.denominator))).sqrt())
        p = 1 - Fraction(m) ** 2 / (2 * rho)  # pressure over (gamma - 1)
        assert Fraction(-1, 10 ** 6) < p < Fraction(-1, 10 ** 8)
        U[0, 1, n], U[1, 0, n] = -c, m
        n += 1
    return U


def test_positivity_is_not_skipped_near_vacuum():
    """The points of an element are left out where bounds on density and pressure rule the scaling
    out.  Near vacuum the bound's own rounding is of the size of the pressure."""
    print("case: limiter near vacuum", flush=True)
    g = vortex_grid(16)
    s = Solver(g, degree=1, flux="lf", limiter=True, tvb_M=1e30, dt_policy="fixed", dt_fixed=1e-3)
    s.set_state(near_vacuum(g.n_elements), BASIS_NATIVE)
    s.stage(0, 0.0)  # leaves the state as it is, then the limiter
    f = s.flags()
    print("scaled", int((f == 2).sum()), "of", f.size, flush=True)
    assert np.all(f == 2)
    s.close()


@pytest.mark.parametrize("P", [1, 2])
@pytest.mark.parametrize("nx,ny", [(256, 192), (223, 221), (250, 280), (280, 251)])
def test_limiter_on_both_sides_of_the_warm_rule(P, nx, ny):
    """98,304 elements and 98,566, 140,000 and 140,560: the launches in which some workgroups look at
    every point and those in which only the elements do that may need it decide alike."""
    print(f"case: limiter P{P} {nx}x{ny}", flush=True)
    g = Grid.splitquad(nx, ny, 0.0, 0.0, 1.0, ny / nx, periodic=False, diagonal=1, jitter=0.2, seed=9)
    o, s = make_pair(g, P=P, flux="lf", limiter=True, dt_policy="max", cfl=0.2 if P == 1 else 0.1, tvb_M=50.0)
    o.project(2, riemann4_params())
    s.set_state(o.get_state())
    s.advance(3)
    o.advance(3)
    err = rel_l2(s.get_state(), o.get_state(), o.mass())
    assert np.all(err < 1e-12), err
    assert np.array_equal(s.flags(), o.flags())
    assert (o.flags() != 0).sum() > 100
    s.close()
