"""Conductivity iteration with fused x and z kernels (32 to 512 points).

A run of n iterations inside one call carries the forward z transform from
iteration to iteration; it equals the oracle's n iterations and n runs of one
iteration.  Tolerance: an iteration rounds each value in at most 6 passes of
at most 9 radix stages, a few ulp (2.2e-16) each relative to the largest
value, so three iterations stay below 1e-12 of it.
"""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _layers(n, seed):
    rng = np.random.default_rng(seed)
    return rng.uniform(0.5, 2.0, n), rng.uniform(-0.5, 0.5, n)


@pytest.mark.parametrize("shape", [
    (32, 8, 8), (8, 8, 32),        # only the x / only the z kernel; the smallest grids
    (32, 40, 64), (64, 24 * 2, 32),  # rows that tiles of 16 lines cross, odd factors in y
    (128, 8, 256), (256, 16, 128), (512, 8, 32), (32, 8, 512),
])
def test_run_of_three_matches_oracle(shape):
    import pfdd_gl
    print(f"case: conductivity run of 3 {shape}", flush=True)
    rng = np.random.default_rng(11)
    four = oracle.set_scale(oracle.prim((1, 0, 0), (0.5, 0.8660254037844386, 0), (0, 0, 1))[0], 1, 1, 1)[0]
    c = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    sig, dsig = _layers(shape[1], 5)
    El, eps0, rate = 0.7, 1.3, 0.05 * np.prod(shape)
    g = pfdd_gl.CondSolver(shape, four, sig, dsig, El, eps0, rate)
    try:
        g.set_c(c)
        r = g.step(3)
        got = g.get_c()
        g.set_c(c)
        for _ in range(3):
            r1 = g.step(1)
        assert np.array_equal(got, g.get_c()) and r == r1
        ref = c.copy()
        for _ in range(3):
            ref, o = oracle.cond_step(ref, four, sig, dsig, El, eps0, rate)
        assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref))
        for key in ("conductivity", "javerage_re", "condxinorm", "condxiave", "conductivity_repeat"):
            assert abs(r[key] - o[key]) <= 1e-9 * max(abs(o[key]), 1e-300), (key, r[key], o[key])
    finally:
        g.close()


def test_non_finite_field_is_refused_and_the_handle_stays_usable():
    import pfdd_gl
    print("case: conductivity run from a field with a NaN", flush=True)
    shape = (32, 16, 32)
    sig, dsig = _layers(shape[1], 6)
    rng = np.random.default_rng(12)
    c = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    bad = c.copy()
    bad[3, 4, 5] = np.nan
    g = pfdd_gl.CondSolver(shape, np.eye(3), sig, dsig, 0.7, 1.3, 0.05)
    try:
        g.set_c(bad)
        for n in (1, 3):
            with pytest.raises(pfdd_gl.PfddError):
                g.step(n)
        g.set_c(c)
        first = g.step(2)
        g.set_c(c)
        assert g.step(2) == first
    finally:
        g.close()
