"""step(0) reports the last executed iteration, also one of a profile."""
import pytest

import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("plane", [0, 2])
def test_report_follows_a_profile(plane):
    case = P.make_case(shape=(16, 32, 32), core="sine", noise=1e-2, sigma_mu=0.004)
    g, h = P.gpu_solver(case), P.gpu_solver(case)
    try:
        for s in (g, h):
            s.set_tuning([1, 1, 1, 1, plane])
        g.step(2)
        g.profile(3)
        last, ref = g.step(0), h.step(5)
        for key in ("xinorm", "xiave", "e_elastic", "e_core", "e_stress", "e_total", "e_core_ref"):
            assert last[key] == ref[key], key
        assert last["steps_done"] == 0
    finally:
        g.close()
        h.close()
