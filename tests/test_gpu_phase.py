"""The nonlinear factor exp(i theta) of complex64 fields: its modulus over many steps."""

import numpy as np
import pytest
from scipy.constants import c, epsilon_0

pytestmark = pytest.mark.gpu

N, DZ, STEPS = 1024, 1e-5, 200


# Without loss, and with a propagator of ones (products by it and by 1/N^2 are
# exact), only the modulus of the phase factor and unbiased roundings change the
# power.  The series of sine and cosine keep |f|^2 - 1 below 6e-12; the roundings
# of a step (some eight of 3e-8 a point, independent over 2^20 points) add
# 2e-10 / sqrt(steps) = 1.4e-11 to the mean per step.  Bound: 1e-10.
@pytest.mark.parametrize("theta", [0.12, 0.25, 0.4])
def test_mean_power_change_per_step(gpu, theta):
    from nlse_amd import NLSE

    s = NLSE(0, 1.0, 1e-2, -1e-9, None, 1.0, NX=N, NY=N, Isat=np.inf)
    s.delta_z = DZ
    s.n2 = -theta / (s.k / 2 * c * epsilon_0 * DZ)
    s.propagator = np.ones((N, N), np.complex64)
    rng = np.random.default_rng(int(100 * theta))
    E = np.sqrt(rng.uniform(0.96, 1.0, (N, N))) * np.exp(2j * np.pi * rng.random((N, N)))
    E = E.astype(np.complex64)
    out = s.out_field(E, (STEPS - 0.5) * DZ, normalize=False, verbose=False)

    def power(A):
        return float((A.real.astype(np.float64) ** 2 + A.imag.astype(np.float64) ** 2).sum())

    change = (power(out) / power(E) - 1) / STEPS
    print(f"phase {theta}: power change per step {change:.2e}")
    assert abs(change) < 1e-10
