"""The register update (nz of 32 to 512) over the lengths of its sine series.

One to eight terms, with and without a per-cell amplitude and frozen cells:
the run of five iterations in one call (the update that also transforms
forward) equals five runs of one bit for bit, since both do the same
arithmetic on every cell, and the field and scalars agree with the oracle
within the tolerances of the parity tests (FP64 1e-9, FP32 1e-5 relative).
"""
import numpy as np
import pytest

import problems as P

pytestmark = pytest.mark.gpu

SCALARS = (("xinorm", "xinorm"), ("xiave", "xiave"), ("E_el", "e_elastic"), ("E_core", "e_core"),
           ("E_stress", "e_stress"), ("E_total", "e_total"))


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("amplitude", [False, True])
@pytest.mark.parametrize("nz,plan", [(32, 1), (128, 1), (128, 4)])  # 128: both radix plans
@pytest.mark.parametrize("ncoef", [1, 2, 3, 4, 5, 8])
def test_series_of_every_length(ncoef, nz, plan, amplitude, masked, precision):
    shape = (8, 16, nz)
    print(f"case: {ncoef} terms, nz {nz} plan {plan}, amplitude {amplitude}, masked {masked}, precision {precision}",
          flush=True)
    xo = None
    if masked:
        xo = np.zeros((3,) + shape)
        xo[:, 2:4, 5:9, nz // 2] = 1.0
        xo[1, 7, 15, nz - 1] = xo[0, 0, 0, 0] = 1.0
    amp = P.amplitude_field(shape, 3, seed=31) if amplitude else None
    # coefficients that differ from system to system and do not vanish
    case = P.make_case(shape=shape, core="series", ncoef=max(2, ncoef), noise=1e-2, sigma_mu=0.004, xo=xo, amp=amp)
    if ncoef == 1:
        par = np.ascontiguousarray(case["core_par"].reshape(3, -1)[:, :1])
        case.update(core_par=par.reshape(-1), nm=1, gpu_core=dict(case["gpu_core"], coef=par.reshape(-1), ncoef=1))
    a, b = P.gpu_solver(case, precision), P.gpu_solver(case, precision)
    st = P.oracle_state(case)
    tol = 1e-9 if precision == 0 else 1e-5
    try:
        for s in (a, b):
            s.set_tuning([plan, 1, 1, 1, 0])
        ra = a.step(5)
        for _ in range(5):
            rb, ref = b.step(1), st.step(case["tau"])
        xa = a.get_xi()
        assert np.array_equal(xa, b.get_xi())
        for want, got in SCALARS:
            assert ra[got] == rb[got], got
            if abs(ref[want]) > 1e-12:
                assert abs(ra[got] - ref[want]) <= tol * abs(ref[want]), (got, ra[got], ref[want])
        assert np.max(np.abs(xa - st.xi)) <= tol * np.max(np.abs(st.xi))
    finally:
        a.close()
        b.close()
