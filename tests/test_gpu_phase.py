"""The nonlinear factor exp(-a + i theta) of complex64 fields: its modulus over many
steps, and its value over the ranges of its forms."""

import numpy as np
import pytest
from scipy.constants import c, epsilon_0

pytestmark = pytest.mark.gpu

N, DZ, STEPS = 1024, 1e-5, 200


# Without loss, and with a propagator of ones (products by it and by 1/N^2 are
# exact), only the modulus of the phase factor and unbiased roundings change the
# power.  The series of sine and cosine keep |f|^2 - 1 below 6e-12; the roundings
# of a step (some eight of 3e-8 a point, independent over 2^20 points) add
# 2e-10 / sqrt(steps) = 1.4e-11 to the mean per step.  Bound: 1e-10.  Past pi/2
# the FP32 evaluation of the factor leaves up to 5.4e-10 (between pi/2 and pi).
@pytest.mark.parametrize("theta,bound", [(0.12, 1e-10), (0.25, 1e-10), (0.4, 1e-10), (2.5, 1e-9), (7.0, 1e-9),
                                         (300.0, 1e-9)])
def test_mean_power_change_per_step(gpu, theta, bound):
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
    assert abs(change) < bound


# both sides of the limits of the short, half-angle and reduced forms (1/4, pi/2,
# 2^16) and far beyond; losses on both sides of 1/8 and 80, and gain
PHASES = [0.2, 0.26, 1.57, 1.58, 3.2, 100.0, 65536.0, 65600.0, 1e9]
LOSSES = [0.0, 0.12, 0.13, 0.7, 5.0, 79.0, 81.0, -0.13, -3.0, -79.0]


# The operator with V = theta + i a, one wave per combination of ranges.  FP32
# sine, cosine and exponential of one rounding each and the products round to
# less than 5e-7 of the larger of |A| and |A| e^{-a}.
def test_factor_of_points(gpu):
    import torch
    from nlse_amd import kernels_hip as K

    rng = np.random.default_rng(4)
    th = np.repeat(np.array(PHASES)[:, None, None], len(LOSSES), 1) * rng.uniform(0.98, 1.0, (1, 1, 64))
    a = np.array(LOSSES)[None, :, None] * rng.uniform(0.99, 1.0, (len(PHASES), 1, 64))
    V = (th * rng.choice([-1, 1], th.shape) + 1j * a).astype(np.complex64).reshape(-1, 64)
    A = np.exp(2j * np.pi * rng.random(V.shape)).astype(np.complex64)
    t = torch.from_numpy(A).to(gpu)
    K.nl_prop(t, torch.zeros(A.shape, dtype=torch.float32, device=gpu), 1.0, 0.0, torch.from_numpy(V).to(gpu), 0.0, np.inf)
    aa, tt = V.imag.astype(np.float64), V.real.astype(np.float64)
    ref = A.astype(np.complex128) * np.exp(-aa + 1j * tt)
    err = np.abs(t.cpu().numpy() - ref) / np.maximum(1.0, np.exp(-aa))
    print("largest error", err.max(), "at", V.reshape(-1)[err.argmax()])
    assert err.max() < 5e-7


# The sweeps' form with one loss for all points: one step with a propagator of
# ones, theta = V.  The transforms round a point of unit modulus by 2e-7 (rms).
@pytest.mark.parametrize("alpha", [0.0, 0.24, 0.26, 8.0, -0.5])
@pytest.mark.parametrize("nx", [256, 1024])
def test_factor_in_a_step(gpu, nx, alpha):
    from nlse_amd import NLSE

    ny = 2 * len(PHASES)
    ny = 1 << (ny - 1).bit_length()
    s = NLSE(alpha, 1.0, 1e-2, -1e-9, None, 2.0, NX=nx, NY=ny, Isat=np.inf)
    s.delta_z, s.k, s.n2 = 1.0, 2.0, 0.0
    rng = np.random.default_rng(nx)
    scale = np.resize(np.array(PHASES), (ny, 1))
    s.V = (scale * rng.uniform(-1, 1, (ny, nx))).astype(np.float32)
    s.propagator = np.ones((ny, nx), np.complex64)
    E = np.exp(2j * np.pi * rng.random((ny, nx))).astype(np.complex64)
    out = s.out_field(E, 0.5, normalize=False, verbose=False)
    ref = E.astype(np.complex128) * np.exp(-alpha / 2 + 1j * s.V.astype(np.float64))
    err = np.abs(out - ref) / max(1.0, np.exp(-alpha / 2))
    print(nx, alpha, f"rms {np.sqrt((err**2).mean()):.2e} max {err.max():.2e}")
    assert np.sqrt((err**2).mean()) < 5e-7 and err.max() < 3e-6
