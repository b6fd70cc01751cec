"""The update fused with the next iteration's forward transform.

Inside a run of several iterations the update kernel transforms its own
result forward (line and plane form); the last iteration of a run does not,
and a run of one iteration uses neither.  Both sequences do the same
arithmetic on every cell, so a run of n iterations equals n runs of one
iteration bit for bit, for every tile shape, radix plan and core model.
"""
import numpy as np
import pytest

import problems as P

pytestmark = pytest.mark.gpu

FRANK = ((1, 0, 0), (0.5, 0.8660254037844386, 0), (0, 0, 1))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("shape,systems,core,choice", [
    ((8, 8, 8), "one", "sine", [1, 1, 1, 1, 0]),         # the smallest lines; tiles larger than the field
    ((16, 8, 16), "basal3", "sine", [0, 0, 0, 0, 0]),
    ((16, 8, 16), "basal3", "sine", [3, 1, 1, 2, 0]),    # one radix-16 stage
    ((8, 40, 48), "basal3", "perfect", [4, 1, 1, 1, 0]),
    ((8, 40, 40), "basal3", "series", [2, 1, 1, 2, 0]),  # 40-point lines, a partial last tile
    ((8, 16, 96), "basal3", "mpea", [1, 1, 1, 0, 0]),
    ((8, 16, 128), "basal3", "sine", [0, 1, 1, 0, 0]),
    ((8, 16, 128), "basal3", "sine", [5, 1, 1, 2, 0]),
    ((8, 8, 256), "basal3", "extended", [3, 1, 1, 0, 0]),
    ((8, 8, 512), "one", "sine", [2, 1, 1, 2, 0]),
    ((16, 16, 32), "basal3", "bcc", [1, 1, 1, 1, 0]),
    ((16, 32, 32), "basal3", "fourier", [1, 1, 1, 1, 2]),
    ((16, 48, 48), "basal3", "sine", [1, 1, 1, 1, 2]),
    ((64, 64, 64), "one", "sine", [1, 1, 1, 1, 2]),
])
def test_run_equals_single_iterations(precision, shape, systems, core, choice):
    print(f"case: {shape} {systems} {core} tuning {choice} precision {precision}: step(5) vs 5 x step(1)", flush=True)
    xo = None
    S = 1 if systems == "one" else 3
    if core == "sine":  # with frozen cells
        xo = np.zeros((S,) + shape)
        xo[:, shape[0] // 2, 1:4, shape[2] // 2] = 1.0
    case = P.make_case(shape=shape, systems=systems, core=core, noise=1e-2, sigma_mu=0.004, xo=xo)
    a, b = P.gpu_solver(case, precision=precision), P.gpu_solver(case, precision=precision)
    try:
        a.set_tuning(choice)
        b.set_tuning(choice)
        ra = a.step(5)
        for _ in range(5):
            rb = b.step(1)
        assert ra["steps_done"] == 5
        xa, xb = a.get_xi(), b.get_xi()
        assert np.array_equal(xa, xb), float(np.max(np.abs(xa - xb)))
        for key in ("xinorm", "xiave", "e_elastic", "e_core", "e_stress", "e_total"):
            assert ra[key] == rb[key], key
    finally:
        a.close()
        b.close()


def test_run_counters_over_runs_of_every_kind():
    """A run counts its own iterations and reports its own end, whatever ran
    on the handle before it: runs that were not waited for, converged runs,
    empty runs, graph replays (20 iterations and more)."""
    case = P.make_case(shape=(32, 32, 32), systems="basal3", core="sine", noise=1e-2, sigma_mu=0.004)
    g = P.gpu_solver(case)
    try:
        g.step(3, sync=False)
        for n, tol, done in ((2, 0.0, 0), (50, 1e30, 1), (4, 0.0, 0), (0, 0.0, 0), (25, 0.0, 0), (25, 1e30, 1),
                             (3, 1e-300, 0)):
            r = g.step(n, tol=tol)
            assert (r["steps_done"], r["converged"]) == (1 if done else n, done), (n, tol, r)
            g.step(1, sync=False)
        h = P.gpu_solver(case)
        try:
            h.step(3 + 2 + 1 + 4 + 25 + 1 + 3 + 7)
            assert np.array_equal(g.get_xi(), h.get_xi())
        finally:
            h.close()
    finally:
        g.close()


def test_gradients_do_not_depend_on_the_tuning():
    """Reverse mode on a handle tuned to the plane iteration sums its blocks as
    on any other.  Tolerance: the sums over 1e5 cells are taken in another
    order, each term below the largest (error below 1e5 u = 2e-11 of it,
    typically its square root)."""
    case = P.make_case(shape=(32, 32, 32), systems="basal3", core="sine", noise=1e-2, sigma_mu=0.004)
    rng = np.random.default_rng(5)
    seed = rng.standard_normal((3, 32, 32, 32)) + 1j * rng.standard_normal((3, 32, 32, 32))
    out = []
    for choice in ([1, 1, 1, 1, 0], [1, 1, 1, 1, 2], [0, 1, 1, 2, 2]):
        g = P.gpu_solver(case)
        try:
            g.set_tuning(choice)
            g.tape_record(5, 3)
            out.append(g.tape_backward(seed, 2))
        finally:
            g.close()
    for got in out[1:]:
        for a, b in zip(got, out[0]):
            assert np.max(np.abs(np.asarray(a) - np.asarray(b))) <= 2e-11 * np.max(np.abs(np.asarray(b)))
