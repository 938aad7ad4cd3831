"""Slabs past 32-bit offsets: a 3-D field of 1024 x 1024 x 512 points, 2^32 bytes, whose
columns along the first axis are addressed by 64 bits.

A transform rounds a point a few times per axis, a step twice as often and in its
propagator: below 1e-6 relative (rms) against 64 bits."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPE = (1024, 1024, 512)


def _field(seed):
    import torch

    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.randn(SHAPE, generator=g, dtype=torch.complex64, device="cuda")


def _err(out, ref):
    import torch

    d = ref.sub_(out)
    return float(torch.linalg.vector_norm(torch.view_as_real(d)) / torch.linalg.vector_norm(torch.view_as_real(out)))


def test_transforms(gpu):
    import torch
    from nlse_amd.fft import HipFFTPlan

    plan = HipFFTPlan(SHAPE, np.complex64, 3)
    A = _field(1)
    ref = torch.fft.fftn(A.to(torch.complex128))
    B = A.clone()
    plan.fft(B)
    forward = _err(B, ref)
    plan.ifft(B)
    back = _err(B, A.to(torch.complex128))
    print(f"forward {forward:.2e}, there and back {back:.2e}")
    assert forward < 1e-6 and back < 1e-6


@pytest.mark.parametrize("kind", ["separable", "dense"])
def test_linear_step(gpu, kind):
    import torch
    from nlse_amd.engine import NL1_DTYPE, SLOT_FULL, Plan

    ny, nx, nt = SHAPE
    rng = np.random.default_rng(3)
    px, py, pt = (np.exp(-2j * np.pi * rng.random(n)) for n in (nx, ny, nt))
    dev = lambda p: torch.from_numpy(p).to("cuda")  # noqa: E731
    table = (dev(py)[:, None] * dev(px)[None, :]).to(torch.complex64).to(torch.complex128)[..., None] * dev(pt)
    plan = Plan(ny, nx, 1, ndim=3, nt=nt)
    if kind == "separable":
        plan.set_propagator_sep(px, py)
        plan.set_propagator_t(pt)
    else:
        plan.set_propagator_3d_c128(table)
    plan.set_nl1(SLOT_FULL, np.zeros(1, NL1_DTYPE))
    A = _field(2)
    ref = torch.fft.fftn(A.to(torch.complex128))
    ref *= table
    ref = torch.fft.ifftn(ref)
    plan.run(A, 1, 0)
    err = _err(A, ref)
    print(kind, plan.config(), f"{err:.2e}")
    assert err < 1e-6
