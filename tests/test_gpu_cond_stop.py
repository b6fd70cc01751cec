"""A conductivity run stops at the iteration whose sums are not finite.

The field stays as that iteration left it, whatever the number of iterations
that were asked for, and also where only the total overflows and no block's
share of it.  The iteration is affine in c and for large c linear, so a field
is scaled to put the first iteration's |dc|^2 above the largest double.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("log_total", [309, 320])  # of |dc|^2: the blocks' shares are finite / are not
@pytest.mark.parametrize("shape", [
    (64, 32, 64),                 # fused x and z kernels
    (48, 32, 40), (48, 16, 128),  # separate ones; only the z kernel is fused
    (128, 16, 48),                # only the x kernel is fused
])
def test_field_stays_where_the_run_stopped(shape, log_total):
    import pfdd_gl
    print(f"case: conductivity overflow at 1e{log_total} on {shape}", flush=True)
    rng = np.random.default_rng(21)
    c = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    sig, dsig = rng.uniform(0.5, 2.0, shape[1]), rng.uniform(-0.5, 0.5, shape[1])
    g = pfdd_gl.CondSolver(shape, np.eye(3), sig, dsig, 0.7, 1.3, 0.05 * np.prod(shape))
    try:
        g.set_c(1e6 * c)
        dc = g.step(1)["condxinorm"] / 1e6
        big = 10.0 ** (log_total / 2) / dc * c
        assert np.all(np.isfinite(big))
        left = []
        for n in (1, 2, 5):
            g.set_c(big)
            with pytest.raises(pfdd_gl.PfddError):
                g.step(n)
            left.append(g.get_c())
        assert np.all(np.isfinite(left[0])) and not np.array_equal(left[0], big)
        for n, got in zip((2, 5), left[1:]):
            assert np.array_equal(got, left[0]), n
        # the handle is as good as new
        g.set_c(c)
        first = g.step(3)
        h = pfdd_gl.CondSolver(shape, np.eye(3), sig, dsig, 0.7, 1.3, 0.05 * np.prod(shape))
        try:
            h.set_c(c)
            assert h.step(3) == first and np.array_equal(h.get_c(), g.get_c())
        finally:
            h.close()
    finally:
        g.close()
