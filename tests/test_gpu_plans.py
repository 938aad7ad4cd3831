"""The plans that the launch rules choose between, at the edges of their ranges.

Bounds, against the complex64 oracle: both sides round a field a few times per
step (the engine once per transform stage, the oracle once per transform and
operator), at most about 4e-7 relative together, and a float32 phase of theta
adds theta * 2.4e-7; twelve steps of small phase or three of phases up to 8 stay
below 7e-6 even if every rounding adds up.  The bound is 1e-5.  complex128:
1e-10, as FP64 rounding (1e-15 per step) and equal table roundings allow."""

import numpy as np
import pytest

import oracle
from conftest import rel_l2

pytestmark = pytest.mark.gpu

C64, C128 = 1e-5, 1e-10
waist = 2.23e-3
window = 4 * waist
DZ = 1e-5


def _material(nx, ny=None, **extra):
    kw = dict(alpha=20, power=1.05, window=[window, window * (ny or nx) / nx], n2=-1.6e-9, V=None, L=1.0, NX=nx,
              Isat=1e5)
    if ny is not None:
        kw["NY"] = ny
    kw.update(extra)
    return kw


def _pair(name, kw, V=None, loss_saturates=False):
    import nlse_amd

    out = []
    for mod in (nlse_amd, oracle):
        s = getattr(mod, name)(**kw)
        s.delta_z = DZ
        s.V = V
        s.loss_saturates = loss_saturates
        out.append(s)
    return out


def _beam(lead, ny, nx, seed, dtype=np.complex64):
    rng = np.random.default_rng(seed)
    y, x = (np.arange(ny) - ny / 2) / nx * window, (np.arange(nx) - nx / 2) / nx * window
    G = np.exp(-(x[None, :] ** 2 + y[:, None] ** 2) / waist**2)
    shape = tuple(lead) + (ny, nx)
    return (G * (1 + 0.01 * (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)))).astype(dtype)


# 2^18 points and fewer take the small-field plans
@pytest.mark.parametrize("lead,ny,nx,precision", [
    ((), 8, 8, "single"), ((), 16, 4096, "double"), ((), 512, 512, "single"), ((), 512, 1024, "double"),
    ((), 2048, 128, "single"), ((), 2048, 256, "single"), ((4,), 256, 256, "double"), ((5,), 256, 256, "single"),
    ((3,), 32, 64, "single"), ((17,), 64, 16, "double")])
def test_small_field_plans(gpu, lead, ny, nx, precision):
    g, o = _pair("NLSE", _material(nx, ny), V=(1e-4 * np.cos(np.arange(ny * nx))).reshape(ny, nx).astype(np.float32))
    E = _beam(lead, ny, nx, ny + nx)
    out = g.out_field(E, 11.5 * DZ, precision=precision, verbose=False)
    err = rel_l2(out, o.out_field(E, 11.5 * DZ, precision))
    print(lead, ny, nx, precision, g._engine.config(), f"{err:.2e}")
    assert err < C64


def test_stack_plans(gpu):
    """Row sets and tiles of stacks of 1024^2 fields: 16 points per lane from 2^21
    points, tiles of 4 columns past 48 MiB; a single field and a requested set
    keep theirs.  Tiles and stores do not change a bit."""
    from nlse_amd import NLSE

    E = _beam((7,), 1024, 1024, 5)

    def run(k, **att):
        s = NLSE(**_material(1024, 1024))
        s.delta_z = DZ
        for a, b in att.items():
            setattr(s, a, b)
        return s.out_field(E[:k] if k else E[0], 3.5 * DZ, verbose=False), s._engine.config()

    one, c1 = run(0)
    two, c2 = run(2)
    six, c6 = run(6)
    seven, c7 = run(7)
    wide, cw = run(7, col_width=8)
    eight, c8 = run(7, row_points=8)
    assert (c1[0], c2[0], c6[0], c7[0], c8[0]) == (8, 16, 16, 16, 8)
    assert (c2[1], c6[1], c7[1], cw[1]) == (8, 8, 4, 8)
    assert np.array_equal(two, six[:2]) and np.array_equal(six, seven[:6]) and np.array_equal(seven, wide)
    assert np.array_equal(eight[0], one)
    half, ch = NLSE(**_material(1024, 512)), None
    half.delta_z = DZ
    half.out_field(_beam((2,), 512, 1024, 6), 1.5 * DZ, verbose=False)
    ch = half._engine.config()
    assert ch[0] == 8  # 2^20 points
    o = oracle.NLSE(**_material(1024, 1024))
    o.delta_z = DZ
    err = rel_l2(two, o.out_field(E[:2], 3.5 * DZ))
    print(c1, c2, c6, c7, cw, ch, f"{err:.2e}")
    assert err < C64


# phases a step of about 0.007, 0.7 (past the short series), 7 (past both), with
# one loss for all points or one that varies, small or past its series
@pytest.mark.parametrize("n2", [-1.6e-9, -1.6e-7, -1.6e-6])
@pytest.mark.parametrize("general", ["", "saturating", "complex V"])
@pytest.mark.parametrize("alpha", [20, 5e4])
@pytest.mark.parametrize("nx", [256, 1024])
def test_phase_and_loss_ranges(gpu, n2, general, alpha, nx):
    ny = 64 if nx == 256 else 512
    V = 1e-3 * np.cos(np.arange(ny * nx)).reshape(ny, nx)
    V = (V + 0.2j * V).astype(np.complex64) if general == "complex V" else V.astype(np.float32)
    kw = _material(nx, ny, n2=n2, alpha=alpha)
    E = _beam((), ny, nx, 3)
    g, o = _pair("NLSE", kw, V=V, loss_saturates=general == "saturating")
    err = rel_l2(g.out_field(E, 2.5 * DZ, verbose=False), o.out_field(E, 2.5 * DZ))
    Ew = E.astype(np.complex128)
    gw, ow = _pair("NLSE", kw, V=V, loss_saturates=general == "saturating")
    errw = rel_l2(gw.out_field(Ew, 2.5 * DZ, verbose=False), ow.out_field(Ew, 2.5 * DZ))
    print(n2, general, alpha, nx, f"{err:.2e} {errw:.2e}")
    assert err < C64 and errw < C128


@pytest.mark.parametrize("n2", [-1.6e-9, -1.6e-7, -1.6e-6])
@pytest.mark.parametrize("dtype,bound", [(np.complex64, C64), (np.complex128, C128)])
def test_two_component_phase_ranges(gpu, n2, dtype, bound):
    g, o = _pair("CNLSE", _material(256, 64, n2=n2, n12=0.3 * n2))
    E = _beam((2,), 64, 256, 9, dtype)
    err = rel_l2(g.out_field(E, 2.5 * DZ, verbose=False), o.out_field(E, 2.5 * DZ))
    print(n2, dtype.__name__, f"{err:.2e}")
    assert err < bound


# 1-D runs: one line, odd counts, the last count of the few-lines plan and the
# next (2^17 / (N/4) lines, at 512 and 2048 points 2^17 / (N/8), 2^16 / (N/8))
@pytest.mark.parametrize("nx,lead", [(16, 1), (64, 7), (256, 1), (256, 2048), (256, 2049), (512, 3), (1024, 512),
                                     (1024, 513), (2048, 256), (2048, 257), (4096, 2)])
@pytest.mark.parametrize("precision", ["single", "double"])
def test_line_counts(gpu, nx, lead, precision):
    kw = _material(nx, Isat=np.inf if lead == 7 else 1e5)
    kw["window"] = window
    g, o = _pair("NLSE_1d", kw, V=(1e-4 * np.cos(np.arange(nx))).astype(np.float32))
    E = _beam((lead,), 1, nx, nx + lead)[:, 0]
    err = rel_l2(g.out_field(E, 11.5 * DZ, precision=precision, verbose=False), o.out_field(E, 11.5 * DZ, precision))
    print(nx, lead, precision, f"{err:.2e}")
    assert err < C64


@pytest.mark.parametrize("nx,lead", [(256, 3), (512, 1), (1024, 512), (1024, 513), (2048, 2)])
def test_line_pair_counts(gpu, nx, lead):
    kw = _material(nx, n12=-3e-10)
    kw["window"] = window
    g, o = _pair("CNLSE_1d", kw)
    E = _beam((lead, 2), 1, nx, nx + lead)[..., 0, :]
    err = rel_l2(g.out_field(E, 11.5 * DZ, verbose=False), o.out_field(E, 11.5 * DZ))
    print(nx, lead, f"{err:.2e}")
    assert err < C64


# nonlocal row kernels: 4 points per lane up to 256-point lines, and up to 2^19
# points of pairs at 512 and 1024
@pytest.mark.parametrize("lead,ny,nx", [((), 64, 16), ((), 16, 32), ((), 64, 128), ((3,), 128, 256), ((4,), 512, 512),
                                        ((5,), 512, 512), ((), 1024, 1024), ((2,), 1024, 1024), ((), 64, 2048)])
def test_nonlocal_row_plans(gpu, lead, ny, nx):
    g, o = _pair("NLSE", _material(nx, ny, nl_length=1.6 * window / nx),
                 V=(1e-4 * np.cos(np.arange(ny * nx))).reshape(ny, nx).astype(np.float32))
    E = _beam(lead, ny, nx, nx)
    err = rel_l2(g.out_field(E, 3.5 * DZ, precision="double", verbose=False), o.out_field(E, 3.5 * DZ, "double"))
    print(lead, ny, nx, f"{err:.2e}")
    assert err < C64


def test_batch_of_mixed_plans(gpu):
    """Members under and over 2^18 points, square and not, equal their own runs."""
    from nlse_amd import NLSE, NLSEBatch

    def sims():
        out = []
        for i, (ny, nx) in enumerate([(256, 256), (512, 512), (512, 1024), (1024, 256), (2048, 128), (128, 2048),
                                      (1024, 1024)]):
            s = NLSE(**_material(nx, ny, n2=-(1 + i) * 1e-9))
            s.delta_z = DZ
            if i % 2:
                s.V = (1e-4 * np.cos(np.arange(ny * nx))).reshape(ny, nx).astype(np.float32)
            out.append(s)
        return out

    fields = [_beam((), s.NY, s.NX, i) for i, s in enumerate(sims())]
    for precision in ("single", "double"):
        outs = NLSEBatch(sims()).out_field(fields, 4.5 * DZ, precision)
        for s, E, out in zip(sims(), fields, outs):
            assert np.array_equal(out, s.out_field(E, 4.5 * DZ, precision=precision, verbose=False)), (s.NY, s.NX, precision)


# complex128: each kind of potential, with and without saturation, one and two
# lines per block, and stores beyond the written-through size
@pytest.mark.parametrize("vdtype", [None, np.float32, np.complex64, np.float64, np.complex128])
@pytest.mark.parametrize("lead,ny,nx", [((), 8, 16), ((3,), 64, 128), ((), 512, 64), ((4,), 1024, 1024)])
def test_complex128_plans(gpu, vdtype, lead, ny, nx):
    V = None
    if vdtype is not None:
        V = 1e-4 * np.cos(np.arange(ny * nx)).reshape(ny, nx)
        V = (V * (1 + 0.1j) if np.dtype(vdtype).kind == "c" else V).astype(vdtype)
    g, o = _pair("NLSE", _material(nx, ny, Isat=np.inf if vdtype is None else 1e5), V=V)
    E = _beam(lead, ny, nx, nx, np.complex128)
    err = rel_l2(g.out_field(E, 2.5 * DZ, precision="double", verbose=False), o.out_field(E, 2.5 * DZ, "double"))
    print(vdtype, lead, ny, nx, f"{err:.2e}")
    assert err < C128


# stores of 8, 16, 32 and 64 contiguous bytes a row (lines of 16 to 128 points,
# tiles of 1 to 8 columns) in stacks on both sides of 16 and 48 MiB: what decides
# between stores back and through changes no bit.  All stacks have more points
# than the small-field plans, and the same row sets
@pytest.mark.parametrize("comp", [1, 2])
@pytest.mark.parametrize("ny,nx,counts", [(256, 16, (80, 640, 1540)), (256, 32, (40, 320, 770)), (128, 64, (40, 320, 770)),
                                          (64, 128, (40, 320, 770)), (4096, 8, (10, 80, 193))])
def test_stores_back_or_through(gpu, ny, nx, counts, comp):
    name, kw = ("NLSE", _material(nx, ny)) if comp == 1 else ("CNLSE", _material(nx, ny, n12=-3e-10))
    E = _beam((2,) if comp == 2 else (), ny, nx, ny)
    scale = np.linspace(0.5, 1.0, counts[-1], dtype=np.float32).reshape((-1,) + (1,) * E.ndim)
    ref = None
    for k in counts:
        g, o = _pair(name, kw)
        out = g.out_field(E * scale[:k], 1.5 * DZ, normalize=False, verbose=False)
        if ref is None:
            ref = out[:3]
            want = o.out_field(E * scale[:3], 1.5 * DZ, normalize=False)
            assert rel_l2(ref, want) < C64
        assert np.array_equal(out[:3], ref), k


def _sized(sim, prop):
    sim.propagator = prop.copy()
    return sim


# dense propagators: every column tile gives the same bits
@pytest.mark.parametrize("name,ny,nx", [("NLSE", 16, 64), ("NLSE", 128, 128), ("CNLSE", 512, 32), ("NLSE", 1024, 64),
                                        ("CNLSE", 2048, 64), ("NLSE", 4096, 32)])
def test_dense_propagator_tiles(gpu, name, ny, nx):
    kw = _material(nx, ny, **({"n12": -3e-10} if name == "CNLSE" else {}))
    comp = (2,) if name == "CNLSE" else ()
    rng = np.random.default_rng(ny)
    prop = np.exp(-1j * rng.random(comp + (ny, nx))).astype(np.complex64)
    E = _beam((2,) + comp, ny, nx, nx)
    outs = {}
    for w in (0, 1, 2, 4, 8, 16, 32):
        g, o = (_sized(s, prop) for s in _pair(name, kw))
        g.col_width = w
        out = g.out_field(E, 2.5 * DZ, verbose=False)
        outs[g._engine.config()[1]] = out
    err = rel_l2(out, o.out_field(E, 2.5 * DZ))
    print(name, ny, nx, sorted(outs), f"{err:.2e}")
    assert err < C64 and len(outs) >= 3
    for w, x in outs.items():
        assert np.array_equal(x, out), w


# 3-D fields: a dense complex128 table, and its column tiles
@pytest.mark.parametrize("shape", [(8, 16, 32), (256, 16, 8), (1024, 8, 16)])
def test_dense_3d_propagator_tiles(gpu, shape):
    import nlse_amd

    ny, nx, nt = shape
    kw = dict(alpha=0, energy=1e-9, window=[4e-3, 4e-3, 2e-12], n2=-1e-9, D0=-1e-26, vg=1.0, V=None, L=1.0, NX=nx, NY=ny,
              NZ=nt, Isat=np.inf)
    rng = np.random.default_rng(ny)
    prop = np.exp(-1j * rng.random(shape))
    E = (1 + 0.1 * rng.standard_normal(shape) + 0.1j * rng.standard_normal(shape)).astype(np.complex64)
    outs = []
    for w in (0, 1, 2, 4, 8, 16, 32):
        g, o = (_sized(getattr(m, "NLSE_3d")(**kw), prop) for m in (nlse_amd, oracle))
        g.delta_z = o.delta_z = DZ
        g.col_width = w
        outs.append(g.out_field(E, 2.5 * DZ, verbose=False))
    err = rel_l2(outs[0], o.out_field(E, 2.5 * DZ))
    print(shape, f"{err:.2e}")
    assert err < C64 and all(np.array_equal(x, outs[0]) for x in outs)
