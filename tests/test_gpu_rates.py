"""The linear athermal law's exponential form on the device (stz_law.h,
large_rate) around its two limits, y = Omega eps0 sbar / theta = 10 and 19.1,
against the oracle, which evaluates the reference's cosh and tanh: stresses,
chi, ddev after one advection step and the substep counts.  The two forms
agree to rounding, a few units in the last place per substep."""
import numpy as np
import pytest

from oracle.pyoracle import Oracle
from stz_amd import ShearSim
from stz_amd.problems import simple_shear

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("theta_K", [400.0, 560.0, 700.0])
def test_rates_around_the_limits_of_the_exponential_form(theta_K):
    print("case rates", theta_K, flush=True)
    p = simple_shear(64, 40, theta_K=theta_K)
    z = p["stz"]
    o, g = Oracle(p), ShearSim(p, "fp64")
    planes = np.zeros((10,) + g.plane_shape)
    # sbar around 1, around both limits and beyond, along x
    at = [10 * z["theta"] / z["Omegaeps0"], 19.1 * z["theta"] / z["Omegaeps0"], 1.0]
    sbar = np.concatenate([a * (1 + np.array([-1e-2, -1e-6, -1e-15, 0, 1e-15, 1e-6, 1e-2])) for a in at] +
                          [np.linspace(0.9, 3.0, 64 - 21)])
    planes[5] = sbar[None, :]
    planes[6] = 0.03 + 1e-3 * np.linspace(0, 1, 42)[:, None]
    for s in (o, g):
        s.set_fields(planes)
        s.time = 2.0
        s.record_decisions(True)
        s.advection_step(0.05)
    G, F = g.get_fields(), o.get_fields()
    trips_g, trips_o = g.get_decisions() >> 24, o.get_decisions() >> 24
    assert trips_o.max() > 1
    # a count may turn on the last place of a rate (none has)
    assert np.count_nonzero(trips_g != trips_o) <= 1
    # each trip changes sbar and chi by rates good to some 4 ulp; up to 255 trips
    for k in (5, 6, 9):
        tol = 4 * 2.3e-16 * max(4, int(trips_o.max()))
        assert np.abs(G[k] - F[k]).max() <= tol * np.abs(F[k]).max(), k
    g.close()
