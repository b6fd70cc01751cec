"""Fields that reach the host in several chunks (2 MiB slots, 16 MiB and more,
or the spread components of the output fields), and the stress of captured
runs."""
import numpy as np
import pytest

import oracle
import problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,shape", [(0, (128, 128, 128)), (0, (160, 96, 80)), (1, (96, 96, 80)), (1, (8, 8, 8))])
def test_field_round_trip(precision, shape):
    print(f"case: set_xi / get_xi {shape} precision {precision}", flush=True)
    case = P.make_case(shape=shape, systems="one", noise=1e-2)
    g = P.gpu_solver(case, precision=precision)
    try:
        rng = np.random.default_rng(3)
        x = rng.standard_normal((1,) + shape) + 1j * rng.standard_normal((1,) + shape)
        g.set_xi(x)
        want = x if precision == 0 else x.astype(np.complex64).astype(np.complex128)
        for _ in range(2):
            assert np.array_equal(g.get_xi(), want)
    finally:
        g.close()


def test_output_fields_over_several_chunks():
    """48 x 48 x 32: the six components (1.1 MiB each) lie across the slots."""
    print("case: output-step fields 48x48x32 x 3", flush=True)
    case = P.make_case(shape=(48, 48, 32), noise=1e-2, sigma_mu=0.004, loops=[(0, 2, 16, 8, 8, 5)])
    m = case["mat"]
    BB, eps, mod = P.oracle_B(case)
    st = P.oracle_state(case, BB)
    g = P.gpu_solver(case)
    try:
        st.step(case["tau"])
        g.step(1)
        FF = oracle.fmatrix(case["shape"], m["C44"], m["C12"], mod["mu"], mod["xnu"], eps, case["geo"]["four"])
        d = oracle.diagnostics(st.data_fftw, st.xi, FF, eps, m, mod["mu"], case["sigma_rot"], fields=True)
        _, _, de, ds = g.diag_fields(case["sigma_rot"])
        for got, want in ((de, d["data_eps"]), (ds, d["data_sigma"])):
            assert np.max(np.abs(got - want)) <= 1e-9 * np.max(np.abs(want))
    finally:
        g.close()


def test_new_stress_reaches_captured_runs():
    """Runs of 20 iterations and more replay captured kernels; set_tau between
    them, alone or with short runs, acts as on a fresh handle."""
    print("case: set_tau between captured runs, 32^3", flush=True)
    case = P.make_case(shape=(32, 32, 32), systems="basal3", noise=1e-2, sigma_mu=0.004)
    tau = np.asarray(case["tau"], float)
    g, h = P.gpu_solver(case), P.gpu_solver(case)
    try:
        for scale, n in ((1.0, 20), (1.5, 20), (-0.5, 3), (2.0, 30), (0.25, 45)):
            g.set_tau(scale * tau)
            g.step(n)
            h.set_tau(scale * tau)
            for _ in range(n):
                h.step(1)
        assert np.array_equal(g.get_xi(), h.get_xi())
    finally:
        g.close()
        h.close()
