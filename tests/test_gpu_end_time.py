"""Runs that reach their end time: what the launches after it cost."""
import time

import pytest

from rkdg_heter_calculate_amd import IC_VORTEX, Solver, vortex_params
from rkdg_heter_calculate_amd.workloads import vortex_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32", "bf16"])
def test_steps_past_the_end_time_load_no_tile(prec, monkeypatch):
    """advance launches its steps in chunks, so up to 31 steps follow the one that reaches the end
    time.  On the staged tiles (P2, 2,048 of them) 96 such launches take what launches cost, 5-7% of
    32 steps; a tile image loaded before the end time is looked at made it 32%."""
    print(f"case: steps past the end time P2 {prec}", flush=True)
    monkeypatch.setenv("RKDG_QUAD", "0")
    s = Solver(vortex_grid(512), degree=2, dt_policy="max", cfl=0.3, precision=prec)
    s.project_ic(IC_VORTEX, vortex_params())
    s.advance(40)
    t = s.time()[0]

    def ms(t_end):
        best = 1e9
        for _ in range(5):
            s.sync()
            t0 = time.perf_counter()
            n, tn = s.advance(32, t_end=t_end)
            best = min(best, time.perf_counter() - t0)
            assert (n, tn) == (0, t) if t_end == t else n == 32
        return best * 1e3

    idle, active = ms(t), ms(1e9)
    print(f"32 steps past the end {idle:.3f} ms, 32 steps {active:.3f} ms", flush=True)
    assert idle < 0.15 * active
    s.close()
