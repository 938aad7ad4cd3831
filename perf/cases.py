"""Performance cases of the split-step engine.

Each case is one ``out_field`` call as a program makes it: the solver object,
its potential and its input field exist, the field is propagated over
``steps`` steps and comes back.  The cases cover the solver classes of the
main path (2-D, two components, 3-D pulses, 1-D lines, uneven batches), both
step kinds (``single``: one nonlinear application per step, ``double``:
Strang), local and nonlocal response, complex64 and complex128 fields, host
and device input, and grids from latency-bound (256^2) to 4096^2.  The learned
corrector is not among them: it is an opt-in addition beside the split-step
path.

Grids are powers of two (what the engine takes); what is ragged in use is the
aspect ratio, the number of realisations, of steps and of fields.
"""

import math

import numpy as np
import torch

C0 = 299792458.0
EPS0 = 8.8541878188e-12
WVL = 780e-9
WAIST = 2.23e-3
WINDOW = 4 * WAIST
ALPHA, POWER, N2, N12, ISAT = 20.0, 1.05, -1.6e-9, -1e-10, 1e5
PULSE_WINDOW = (4e-3, 4e-3, 2e-12)
PULSE_N2, PULSE_D0, PULSE_T0 = -1e-9, -1e-26, 200e-15
L = 10e-3


def _case(name, kind, ny, nx, steps, **kw):
    c = dict(kind=kind, ny=ny, nx=nx, nt=1, lead=0, steps=steps, dz=1e-5, precision="single", potential=True,
             nl_points=0.0, dtype="complex64", omega=0.0, host=False, fields=0)
    c.update(kw)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # the README example: 512^2 beam over 10 mm in a potential, numpy in
        # and numpy out, the call most users make first
        _case("readme_512", "nlse", 512, 512, 1000, host=True),
        # the smallest 2-D grid of ordinary use, Strang steps: launch latency
        _case("strang_256", "nlse", 256, 256, 200, precision="double", potential=False),
        # a parameter scan: 18 realisations of a small non-square grid with
        # their own n2, through leading-dimension broadcasting
        _case("scan_18x128x256", "nlse", 128, 256, 301, lead=18),
        # the everyday large field: 2048^2 with a potential, local response
        _case("local_2048", "nlse", 2048, 2048, 201),
        # the grid sweep of the published 2-D benchmark (20 steps, no
        # potential) at the largest supported grid
        _case("sweep_4096", "nlse", 4096, 4096, 20, potential=False, dz=1e-4),
        # the headline workload: 2048^2 speckle field, nonlocal response of
        # 20 um (kernel of 25 x 25 points), potential
        _case("nonlocal_2048", "nlse", 2048, 2048, 201, dz=5e-6, nl_points=4.6),
        # nonlocal response with Strang steps (two convolutions per step)
        _case("nonlocal_strang_1024", "nlse", 1024, 1024, 101, precision="double", nl_points=4.6),
        # two coupled components with Rabi coupling in a potential
        _case("cnlse_1024", "cnlse", 1024, 1024, 101, omega=2e3),
        # pulse propagation with dispersion: 512 x 512 x 64 points
        _case("pulse_512x512x64", "nlse3d", 512, 512, 51, nt=64, potential=False),
        # 1-D parameter scan: 250 lines of 1024 points over the full length
        _case("lines_250x1024", "nlse1d", 1, 1024, 1000, lead=250),
        # 64 simulations of different grids advanced together
        _case("uneven_64", "uneven", 0, 0, 500, fields=64, potential=False),
        # double-precision field, nonlocal response
        _case("c128_nonlocal_1024", "nlse", 1024, 1024, 51, nl_points=4.6, dtype="complex128"),
    ]


# grid-point-steps of a drawn case, at most
_MOST = 6e8


def _steps(rng, points, cap=1000):
    most = max(12, min(cap, int(_MOST / points)))
    return int(round(math.exp(rng.uniform(math.log(11), math.log(most)))))


def draw(rng):
    pick = rng.choice(["nlse", "nlse", "nlse", "nonlocal", "nonlocal", "cnlse", "nlse3d", "nlse1d", "uneven", "c128"])
    prec = rng.choice(["single", "single", "double"])
    pot = rng.random() < 0.6
    if pick == "nlse3d":
        ny, nx, nt = 2 ** rng.randint(7, 9), 2 ** rng.randint(7, 9), 2 ** rng.randint(4, 7)
        return _case(None, "nlse3d", ny, nx, _steps(rng, 2 * ny * nx * nt), nt=nt, potential=False, precision=prec)
    if pick == "nlse1d":
        nx, lead = 2 ** rng.randint(8, 12), rng.randint(1, 400)
        return _case(None, "nlse1d", 1, nx, rng.randint(100, 1000), lead=lead, potential=pot, precision=prec)
    if pick == "uneven":
        return _case(None, "uneven", 0, 0, rng.randint(20, 300), fields=rng.randint(5, 64), potential=False,
                     precision=prec)
    top = 11 if pick in ("nlse", "nonlocal") else 10
    ny, nx = 2 ** rng.randint(7, top), 2 ** rng.randint(7, top)
    if pick == "nlse" and rng.random() < 0.25:
        nx = 4096
    lead = 0
    if rng.random() < 0.4 and ny * nx <= 1 << 19:
        lead = rng.randint(2, max(3, min(24, (1 << 22) // (ny * nx))))
    points = ny * nx * max(1, lead)
    if pick == "cnlse":
        return _case(None, "cnlse", ny, nx, _steps(rng, 2 * points), lead=lead, potential=pot, precision=prec,
                     omega=rng.choice([0.0, 2e3]))
    if pick == "c128":
        nl = rng.choice([0.0, rng.randint(1, 4) + 0.6])
        return _case(None, "nlse", ny, nx, _steps(rng, (8 if nl else 2) * points, 200), lead=lead, potential=pot,
                     precision=prec, nl_points=nl, dtype="complex128")
    nl = rng.randint(1, 8) + 0.6 if pick == "nonlocal" else 0.0
    return _case(None, "nlse", ny, nx, _steps(rng, (4 if nl else 1) * points), lead=lead, potential=pot,
                 precision=prec, nl_points=nl, host=rng.random() < 0.2)


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _axis(window, n):
    return torch.arange(n, dtype=torch.float64, device="cuda") * (window / n) - window / 2


def _noise(shape, g, amp=0.01):
    n = torch.randn((2,) + tuple(shape), generator=g, dtype=torch.float32, device="cuda").double()
    return 1 + amp * torch.complex(n[0], n[1])


def _beam(ny, nx):
    x, y = _axis(WINDOW, nx), _axis(WINDOW, ny)
    return torch.exp(-(x[None, :] ** 2 + y[:, None] ** 2) / WAIST**2)


def _speckle(shape, g):
    """Random phases low-passed to 1/8 of the band, unit mean intensity."""
    ph = torch.rand(shape, generator=g, dtype=torch.float32, device="cuda").double() * (2 * math.pi)
    S = torch.fft.fft2(torch.polar(torch.ones_like(ph), ph))
    ky = torch.fft.fftfreq(shape[-2], device="cuda").abs() <= 1 / 16
    kx = torch.fft.fftfreq(shape[-1], device="cuda").abs() <= 1 / 16
    S = torch.fft.ifft2(S * (ky[:, None] & kx[None, :]))
    return S / S.abs().square().mean((-2, -1), keepdim=True).sqrt()


def _pulse_power(nt):
    """Energy for a peak power of 1 W of the sech pulse on its time grid."""
    t = np.linspace(-PULSE_WINDOW[2] / 2, PULSE_WINDOW[2] / 2, nt)
    return float(np.sum(1.0 / np.cosh(t / PULSE_T0) ** 2) * (t[1] - t[0]))


def _uneven_list(case, seed):
    """Grid, n2, power and Isat of every field of an uneven batch.  The grids
    belong to the case, the material to the seed."""
    grids = np.random.default_rng(2 + case["fields"])
    rng = np.random.default_rng(seed)
    return [dict(n=int(grids.choice([256, 512, 1024])), n2=-(10 ** rng.uniform(-10, -8)), power=rng.uniform(0.1, 2.0),
                 isat=10 ** rng.uniform(4, 6)) for _ in range(case["fields"])]


def _scan_n2(case, dims):
    """n2 of each realisation of a scan, shaped to broadcast over the field."""
    return np.linspace(N2, -1e-10, case["lead"]).reshape((case["lead"],) + (1,) * dims)


def _potential(case):
    if case["kind"] == "nlse1d":
        r2 = _axis(WINDOW, case["nx"]) ** 2
    else:
        r2 = _axis(WINDOW, case["nx"])[None, :] ** 2 + _axis(WINDOW, case["ny"])[:, None] ** 2
    return (-1e-4 * torch.exp(-r2 / (140e-6) ** 2)).float()


def _fields(case, seed):
    """The input field(s) of a case, complex, on the GPU."""
    g = _gen(seed)
    kind, lead = case["kind"], ((case["lead"],) if case["lead"] else ())
    dtype = getattr(torch, case["dtype"])
    if kind == "uneven":
        return [(_beam(f["n"], f["n"]) * _noise((f["n"], f["n"]), g)).to(dtype) for f in _uneven_list(case, seed)]
    if kind == "nlse1d":
        x = _axis(WINDOW, case["nx"])
        return (torch.exp(-(x**2) / WAIST**2) * _noise(lead + (case["nx"],), g)).to(dtype)
    if kind == "nlse3d":
        wx, wy, wt = PULSE_WINDOW
        x, y = _axis(wx, case["nx"]), _axis(wy, case["ny"])
        t = torch.linspace(-wt / 2, wt / 2, case["nt"], dtype=torch.float64, device="cuda")
        E = torch.exp(-(x[None, :, None] ** 2 + y[:, None, None] ** 2) / 1e-6) / torch.cosh(t / PULSE_T0)
        return (E * _noise(E.shape, g)).to(dtype)
    comp = (2,) if kind == "cnlse" else ()
    shape = lead + comp + (case["ny"], case["nx"])
    mod = 1 + _speckle(shape, g) if case["nl_points"] > 0 else _noise(shape, g)
    return (_beam(case["ny"], case["nx"]) * mod).to(dtype)


def prepare(case, seed):
    from nlse_amd import CNLSE, NLSE, NLSE_1d, NLSE_3d, NLSEBatch

    kind, ny, nx = case["kind"], case["ny"], case["nx"]
    E = _fields(case, seed)
    if kind == "uneven":
        sims = []
        for f in _uneven_list(case, seed):
            s = NLSE(ALPHA, f["power"], WINDOW, f["n2"], None, L, NX=f["n"], NY=f["n"], Isat=f["isat"], wvl=WVL)
            s.delta_z = case["dz"]
            sims.append(s)
        sim = NLSEBatch(sims)
    elif kind == "nlse3d":
        sim = NLSE_3d(alpha=0, energy=_pulse_power(case["nt"]), window=list(PULSE_WINDOW), n2=PULSE_N2, D0=PULSE_D0,
                      vg=1.0, V=None, L=L, NX=nx, NY=ny, NZ=case["nt"], Isat=np.inf, wvl=WVL)
        sim.delta_z = case["dz"]
    else:
        n2 = _scan_n2(case, 1 if kind == "nlse1d" else 2) if case["lead"] else N2
        kw = dict(alpha=ALPHA, power=POWER, window=WINDOW, n2=n2, V=None, L=L, NX=nx, Isat=ISAT, wvl=WVL,
                  nl_length=case["nl_points"] * WINDOW / nx)
        if kind == "nlse1d":
            sim = NLSE_1d(**kw)
        elif kind == "cnlse":
            sim = CNLSE(NY=ny, n12=N12, omega=case["omega"] or None, **kw)
        else:
            sim = NLSE(NY=ny, **kw)
        sim.delta_z = case["dz"]
        if case["potential"]:
            sim.V = _potential(case).cpu().numpy()
    if case["host"]:
        E = E.cpu().numpy()
    return {"sim": sim, "E": E, "z": (case["steps"] - 0.5) * case["dz"], "precision": case["precision"],
            "uneven": kind == "uneven"}


def run(state):
    sim, E, z, precision = state["sim"], state["E"], state["z"], state["precision"]
    if state["uneven"]:
        return sim.out_field(E, z, precision=precision)
    return sim.out_field(E, z, precision=precision, verbose=False)


# ------------------------------------------------------------------ work
def work(case):
    """A pass cannot do without reading the input field (and the potential)
    and writing the result, and the transforms and pointwise operations of
    its steps: 5 n log2 n operations per transform, forward and inverse per
    step, a complex product per point for the propagator, about 30
    operations per point for a nonlinear application, and for a nonlocal
    response the forward and inverse transform of a real array."""
    kind = case["kind"]
    item = 16 if case["dtype"] == "complex128" else 8
    if kind == "uneven":
        grids = [(f["n"], f["n"], 1) for f in _uneven_list(case, 0)]
    else:
        reps = max(1, case["lead"]) * (2 if kind == "cnlse" else 1)
        grids = [(case["ny"], case["nx"], case["nt"])] * reps
    apps = 2 if case["precision"] == "double" else 1
    nbytes = flops = 0.0
    for ny, nx, nt in grids:
        n = ny * nx * nt
        per = 10.0 * math.log2(n) + 6 + apps * 30.0
        if case["nl_points"] > 0:
            per += apps * (5.0 * math.log2(n) + 2)
        nbytes += 2.0 * item * n
        flops += n * per * case["steps"]
    if case["potential"] and kind != "uneven":
        nbytes += 4.0 * case["ny"] * case["nx"]
    return {"bytes": nbytes, "flops": flops}


# ----------------------------------------------------------------- exact
def _wavenumbers(window, n):
    return 2 * math.pi * torch.fft.fftfreq(n, d=window / n, dtype=torch.float64, device="cuda")


def _k0_kernel(nl_length, dx):
    """The nonlocal response: K0(r/d) on (6d+1)^2 points, the singular centre
    set to the largest finite value, unit sum."""
    from scipy import special

    d = nl_length // dx
    x = np.arange(-3 * d, 3 * d + 1)
    K = special.kn(0, np.hypot(*np.meshgrid(x, x)) / d)
    m = K.shape[0] // 2
    K[m, m] = np.nanmax(K[~np.isinf(K)])
    return torch.from_numpy(K / K.sum()).cuda()


def _same_convolution(K, ny, nx):
    """I -> the zero-padded linear convolution with K, the central NY x NX."""
    kh, kw = K.shape
    py, px = ny + kh - 1, nx + kw - 1
    py, px = py + py % 2, px + px % 2
    KF = torch.fft.rfft2(K, s=(py, px))
    a, b = (kh - 1) // 2, (kw - 1) // 2
    return lambda I: torch.fft.irfft2(torch.fft.rfft2(I, s=(py, px)) * KF, s=(py, px))[..., a:a + ny, b:b + nx]


def _propagate(A, prop, dims, nonlinear, case, coupling=None):
    """`steps` split steps: the linear step, then N(dz); or N(dz/2), the
    linear step, N(dz/2)."""
    dz, double = case["dz"], case["precision"] == "double"
    for _ in range(case["steps"]):
        if double:
            A = nonlinear(A, dz / 2)
        A = torch.fft.ifftn(torch.fft.fftn(A, dim=dims) * prop, dim=dims)
        A = nonlinear(A, dz / 2 if double else dz)
        if coupling is not None and not double:
            A = coupling(A)
    return A


def _normalised(E, target, cell, dims):
    E = E.to(torch.complex128)
    p = E.abs().square().sum(dims, keepdim=True) * cell * C0 * EPS0 / 2
    return E * torch.sqrt(target / p)


def _table(*phase):
    """exp(-i sum of the phases) as the complex64 table the step is defined with."""
    total = phase[0]
    for p in phase[1:]:
        total = total + p
    return torch.polar(torch.ones_like(total), -total).to(torch.complex64).to(torch.complex128)


def _single_field(E, case, n2, power, isat, V=None, conv=None):
    k = 2 * math.pi / WVL
    ny, nx = E.shape[-2:]
    cell = (WINDOW / nx) * (WINDOW / ny)
    A = _normalised(E, power, cell, (-2, -1))
    kx, ky = _wavenumbers(WINDOW, nx), _wavenumbers(WINDOW, ny)
    prop = _table(0.5 * (kx[None, :] ** 2 + ky[:, None] ** 2) / k * case["dz"])
    g, i0 = k / 2 * n2 * C0 * EPS0, 2 * isat / (EPS0 * C0)
    # a complex128 field sees k/2 V in the potential's own float32
    vk = 0.0 if V is None else ((V * np.float32(k / 2)).double() if case["dtype"] == "complex128" else k / 2 * V.double())

    def nonlinear(A, dz):
        I = A.abs().square()
        if conv is not None:
            I = conv(I)
        phase = dz * (g * I / (1 + I / i0) + vk)
        return A * torch.polar(torch.full_like(phase, math.exp(-dz * ALPHA / 2)), phase)

    return _propagate(A, prop, (-2, -1), nonlinear, case)


def exact(case, seed):
    """What `run` returns, by torch's transforms in 64 bits."""
    kind, ny, nx = case["kind"], case["ny"], case["nx"]
    k = 2 * math.pi / WVL
    E = _fields(case, seed)
    if kind == "uneven":
        return [_single_field(e, case, f["n2"], f["power"], f["isat"]) for e, f in zip(E, _uneven_list(case, seed))]
    V = _potential(case) if case["potential"] else None
    if kind == "nlse":
        n2 = torch.from_numpy(_scan_n2(case, 2)).cuda() if case["lead"] else N2
        conv = None
        if case["nl_points"] > 0:
            conv = _same_convolution(_k0_kernel(case["nl_points"] * WINDOW / nx, WINDOW / nx), ny, nx)
        out = _single_field(E, case, n2, POWER, ISAT, V, conv)
    elif kind == "nlse1d":
        n2 = torch.from_numpy(_scan_n2(case, 1)).cuda() if case["lead"] else N2
        dx = WINDOW / nx
        A = _normalised(E, POWER, dx * dx, (-1,))
        phase = 0.5 * _wavenumbers(WINDOW, nx) ** 2 / k * case["dz"]
        prop = torch.polar(torch.ones_like(phase), -phase)
        g, i0 = k / 2 * n2 * C0 * EPS0, 2 * ISAT / (EPS0 * C0)
        vk = 0.0 if V is None else k / 2 * V.double()

        def nonlinear(A, dz):
            I = A.abs().square()
            phase = dz * (g * I / (1 + I / i0) + vk)
            return A * torch.polar(torch.full_like(phase, math.exp(-dz * ALPHA / 2)), phase)

        out = _propagate(A, prop, (-1,), nonlinear, case)
    elif kind == "nlse3d":
        wx, wy, wt = PULSE_WINDOW
        nt = case["nt"]
        dt = wt / (nt - 1)
        A = _normalised(E, _pulse_power(nt), (wx / nx) * (wy / ny) * dt, (-3, -2, -1))
        kx, ky = _wavenumbers(wx, nx), _wavenumbers(wy, ny)
        om = 2 * math.pi * torch.fft.fftfreq(nt, d=dt, dtype=torch.float64, device="cuda")
        prop2 = _table(0.5 * (kx[None, :] ** 2 + ky[:, None] ** 2) / k * case["dz"])
        ph = PULSE_D0 / 2 * om**2
        prop = prop2[:, :, None] * torch.polar(torch.ones_like(ph), -ph)
        g = k / 2 * PULSE_N2 * C0 * EPS0

        def nonlinear(A, dz):
            phase = dz * g * A.abs().square()
            return A * torch.polar(torch.ones_like(phase), phase)

        out = _propagate(A, prop, (-3, -2, -1), nonlinear, case)
    else:  # two components; the second has the first's material
        n2 = torch.from_numpy(_scan_n2(case, 2)).cuda() if case["lead"] else N2
        A = _normalised(E, POWER, (WINDOW / nx) * (WINDOW / ny), (-2, -1))
        kx, ky = _wavenumbers(WINDOW, nx), _wavenumbers(WINDOW, ny)
        prop = _table(0.5 * (kx[None, :] ** 2 + ky[:, None] ** 2) / k * case["dz"])
        gs, gc, i0 = k / 2 * n2 * C0 * EPS0, k / 2 * N12 * C0 * EPS0, 2 * ISAT / (EPS0 * C0)
        vk = 0.0 if V is None else k / 2 * V.double()

        def nonlinear(A, dz):
            I1, I2 = (A[..., i, :, :].abs().square() for i in (0, 1))
            sat = 1 / (1 + I1 / i0 + I2 / i0)
            loss = torch.exp(-dz * ALPHA / 2 * sat)
            f1 = torch.polar(loss, dz * (gs * I1 * sat + gc * I2 * sat + vk))
            f2 = torch.polar(loss, dz * (gs * I2 * sat + gc * I1 * sat + vk))
            return A * torch.stack([f1, f2], dim=-3)

        coupling = None
        if case["omega"]:
            w = case["omega"] / 2 * case["dz"]
            cw, sw = math.cos(w), math.sin(w)

            def coupling(A):
                a, b = A[..., 0, :, :], A[..., 1, :, :]
                return torch.stack([cw * a - 1j * sw * b, cw * b - 1j * sw * a], dim=-3)

        out = _propagate(A, prop, (-2, -1), nonlinear, case, coupling)
    return out.cpu().numpy() if case["host"] else out
