"""A handle's core model changed by set_core_coef.

set_core_coef turns the coupled (2) and Fourier (4, 9) models into the sine
series, whose update is another kernel with other tiles.  From then on the
handle does what one created with the series does, bit for bit: the same
kernels on the same inputs, so field and scalars are compared exactly.
"""
import numpy as np
import pytest

import problems as P

pytestmark = pytest.mark.gpu

SCALARS = ("xinorm", "xiave", "e_elastic", "e_core", "e_stress", "e_total", "e_core_ref", "steps_done", "converged")


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("core", ["extended", "fourier", "pyrII"])
@pytest.mark.parametrize("nz", [32, 48, 64, 128, 256, 512])
def test_switched_handle_equals_a_series_handle(nz, core, precision):
    shape = (8, 16, nz)
    print(f"case: {core} -> series at nz {nz}, precision {precision}", flush=True)
    other = P.make_case(shape=shape, core=core, noise=1e-2, sigma_mu=0.004)
    case = P.make_case(shape=shape, core="series", ncoef=4, noise=1e-2, sigma_mu=0.004)
    a, b = P.gpu_solver(other, precision=precision), P.gpu_solver(case, precision=precision)
    try:
        # the coupled and Fourier models' only tile shape, which the handle keeps
        b.set_tuning([1, 1, 1, 0, 0])
        a.step(3)
        a.set_xi(case["xi0"])
        a.set_core_coef(case["core_par"], case["nm"])
        for n, tol in ((5, 0.0), (25, 0.0), (3, 1e30)):
            ra, rb = a.step(n, tol=tol), b.step(n, tol=tol)
            for key in SCALARS:
                assert ra[key] == rb[key], (n, key, ra[key], rb[key])
        assert np.array_equal(a.get_xi(), b.get_xi())
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("nz", [32, 128])
def test_recorded_run_outlives_a_switch(nz):
    """A recorded run keeps its own model: the reverse pass recomputes its
    states with that model's kernels, whatever the handle does by then."""
    case = P.make_case(shape=(8, 16, nz), core="extended", noise=1e-2, sigma_mu=0.004)
    series = P.make_case(shape=(8, 16, nz), core="series", ncoef=4, noise=1e-2, sigma_mu=0.004)
    rng = np.random.default_rng(5)
    seed = rng.standard_normal((3, 8, 16, nz)) + 1j * rng.standard_normal((3, 8, 16, nz))
    out = []
    for switch in (False, True):
        g = P.gpu_solver(case)
        try:
            g.tape_record(5, 3)
            if switch:
                g.set_core_coef(series["core_par"], series["nm"])
            out.append(g.tape_backward(seed, 7))
        finally:
            g.close()
    for x, y in zip(*out):
        assert np.array_equal(np.asarray(x), np.asarray(y))
