"""The step's band table (pencils outside the dealiasing sphere are neither
transformed nor moved), its whole-spectrum form for unprojected data, the
kx = 0 plane factor that stands in for the symmetrized velocity, and both
forms of the integrating factor, against the CPU oracle.

Tolerance: relative L2 1e-11 after a few FP64 steps, that of the other FP64
step tests (rounding of 27 transforms a step, about 1e-15 each), and 1e-6 in
FP32 (about 1e-7 each).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
TOL = 1e-11
TOL32 = 1e-6


def rel(a, b):
    return np.linalg.norm((a - b).ravel()) / max(np.linalg.norm(b.ravel()), 1e-300)


def spectrum(n, seed):
    """Every mode but the unstored kx = n/2 ones, not conjugate-symmetric on
    kx = 0: what a caller may put without a projection."""
    rng = np.random.default_rng(seed)
    shp = (n, n, n // 2 + 1, 3)
    a = rng.standard_normal(shp) + 1j * rng.standard_normal(shp)
    kx = np.arange(n // 2 + 1)
    k1 = np.where(np.arange(n) <= n // 2, np.arange(n), np.arange(n) - n)
    k2 = k1[:, None, None] ** 2 + k1[None, :, None] ** 2 + kx[None, None, :] ** 2
    a *= (1.0 / (1.0 + k2))[..., None]
    a[:, :, n // 2] = 0
    return a


@pytest.mark.parametrize("n, dealias, projected, dk, nu", [
    (16, "SMOOTH", False, (1.0, 1.0, 1.0), 0.02),
    (32, "SMOOTH", True, (1.0, 1.0, 1.0), 0.02),
    (32, "TWO_THIRDS", False, (1.0, 1.0, 1.0), 0.02),
    (48, "SMOOTH", False, (1.0, 1.0, 1.0), 0.02),
    (48, "TWO_THIRDS", True, (1.0, 1.0, 1.0), 0.02),
    # ky = n/2 and kz = n/2 inside the sphere (kx = n/2, which is not stored, never is)
    (64, "SMOOTH", True, (1.0, 0.5, 0.75), 0.02),
    (64, "TWO_THIRDS", True, (1.25, 1.0, 0.5), 0.02),
    (32, "SMOOTH", True, (1.0, 1.0, 1.0), 2.0),     # damping of the last modes above exp(-1/2) per step
    (128, "TWO_THIRDS", True, (1.0, 1.0, 1.0), 0.02),
])
def test_step(oracle, n, dealias, projected, dk, nu):
    import bfps_amd as B
    w0 = spectrum(n, n)
    print("case: band n=%d %s projected=%s dk=%s nu=%g" % (n, dealias, projected, dk, nu), flush=True)
    fs = B.vorticity_equation("t", n, dkx=dk[0], dky=dk[1], dkz=dk[2], precision="double", dealias=dealias)
    fs.nu, fs.famplitude, fs.forcing_type = nu, 0.3, "linear"
    o = oracle.Solver(n, precision="double", dealias=dealias, dk=dk)
    o.set_physics(nu, "linear", 0.3, 2.0, 4.0)
    o.set_cfield("vorticity", w0)
    if projected:
        fs.io_checkpoint(read=True, data=w0)
        o.io_projection()
    else:
        fs.cvorticity = w0
    for _ in range(3):
        fs.step(0.005)
        o.step(0.005)
    e = rel(fs.cvorticity, o.get_cfield("vorticity"))
    print("  rel", e, flush=True)
    assert e < TOL


@pytest.mark.parametrize("n, dealias, projected", [
    (32, "TWO_THIRDS", True), (32, "SMOOTH", False),     # one launch a stage over the (z, x) slab of a y
    (64, "TWO_THIRDS", True), (64, "TWO_THIRDS", False), (64, "SMOOTH", False),  # the same, FP32 only
    (48, "TWO_THIRDS", False),
    (128, "TWO_THIRDS", True), (128, "SMOOTH", False),   # x pass in registers, FP32 only
])
def test_step_single(oracle, n, dealias, projected):
    import bfps_amd as B
    w0 = spectrum(n, n + 2).astype(np.complex64)
    print("case: band fp32 n=%d %s projected=%s" % (n, dealias, projected), flush=True)
    fs = B.vorticity_equation("t", n, precision="single", dealias=dealias)
    fs.nu, fs.famplitude, fs.forcing_type = 0.02, 0.3, "linear"
    o = oracle.Solver(n, precision="double", dealias=dealias)
    o.set_physics(0.02, "linear", 0.3, 2.0, 4.0)
    o.set_cfield("vorticity", w0.astype(np.complex128))
    if projected:
        fs.io_checkpoint(read=True, data=w0)
        o.io_projection()
    else:
        fs.cvorticity = w0
    for _ in range(2):
        fs.step(0.005)
        o.step(0.005)
    e = rel(fs.cvorticity, o.get_cfield("vorticity"))
    print("  rel", e, flush=True)
    assert e < TOL32


@pytest.mark.parametrize("precision, dealias, projected", [
    ("single", "SMOOTH", True), ("single", "TWO_THIRDS", True), ("single", "SMOOTH", False),
    ("double", "TWO_THIRDS", True)])
def test_every_band_pass_shape(precision, dealias, projected):
    """Every shape of the step's z passes, persistent ones among them, by a
    step at 256^3 from a field that fills the sphere (and, unprojected, what
    lies beyond it) evenly: as the built-in shapes, which the steps above check,
    to rounding."""
    import bfps_amd as B
    n = 256
    print("case: band pass shapes %s %s projected=%s" % (precision, dealias, projected), flush=True)
    fs = B.vorticity_equation("t", n, precision=precision, dealias=dealias, plan_rigor="FFTW_ESTIMATE")
    fs.nu, fs.forcing_type = 0.0005, "none"
    rng = np.random.default_rng(n)
    real = np.float32 if precision == "single" else np.float64
    w0 = rng.standard_normal((n, n, n // 2 + 1, 6), dtype=real).view(fs.cdtype)
    w0 *= 0.01  # dt k u is about a quarter: the nonlinear term is a good part of the step
    w0[:, :, n // 2] = 0

    def step(index):
        for kind in ("z_inv", "z_fwd"):
            fs.set_pass_shape(kind, index)
        if projected:
            fs.io_checkpoint(read=True, data=w0)
        else:
            fs.cvorticity = w0
        start = fs.cvorticity if index == 0 else None
        fs.step(0.005)
        return start, fs.cvorticity

    start, want = step(0)
    assert rel(want, start) > 0.05
    shapes = fs.pass_shapes()["z_inv"][3]
    assert shapes > 8
    for index in range(1, shapes):
        e = rel(step(index)[1], want)
        print("  shape %d %s rel %.3e" % (index, fs.pass_shapes()["z_inv"][:2] + fs.pass_shapes()["z_inv"][4:], e), flush=True)
        assert e < (TOL32 if precision == "single" else TOL)
    fs.close()


@pytest.mark.parametrize("n, dealias, dk", [
    (32, "SMOOTH", (1.0, 1.0, 1.0)),
    # ky = n/2 and kz = n/2 inside the sphere
    (64, "SMOOTH", (1.0, 0.5, 0.75)),
    (32, "TWO_THIRDS", (1.25, 1.0, 0.5)),
])
def test_gradient(oracle, n, dealias, dk):
    """Velocity and its gradient in real space, component by component."""
    import bfps_amd as B
    print("case: band gradient n=%d %s dk=%s" % (n, dealias, dk), flush=True)
    fs = B.vorticity_equation("t", n, dkx=dk[0], dky=dk[1], dkz=dk[2], precision="double", dealias=dealias)
    o = oracle.Solver(n, precision="double", dealias=dealias, dk=dk)
    w0 = spectrum(n, n + 1)
    fs.io_checkpoint(read=True, data=w0)
    o.set_cfield("vorticity", w0)
    o.io_projection()
    fs.velocity_rspace()
    o.velocity_rspace()
    assert rel(fs.get_rfield(B.capi.RVELOCITY), o.get_rfield("rvelocity")) < TOL
    fs.gradient_rspace()
    o.gradient_rspace()
    got, want = fs.get_rfield(B.capi.RGRADIENT), o.get_rfield("gradient")
    errors = [rel(got[..., c], want[..., c]) for c in range(9)]
    print("  rel", errors, flush=True)
    assert max(errors) < TOL


@pytest.mark.parametrize("x", [0.7, 1.4, 3.0])
def test_strong_damping(x):
    """FP64 decay of modes so small that nothing else acts on them (squares of
    1e-120 against modes of 1e-120 times exp(-64 x)), where nu dt kM^2 = x
    damps the last modes by more than exp(-1/2) a step: the error of each mode
    (against its exponential in extended precision) is that of a step with one
    rounded exponential per factor.

    The factors are the same every step, so their rounding adds up over the
    64 steps, to about 8e-15 in the mean over the modes; the roundings of the
    stages and projections of a step differ and add up to about 1e-15.  A
    product of two rounded exponentials gives 1.3 times as much: the bound is
    1.15 times, and the mean over 10^5 modes does not move by more than a
    percent from one spectrum to another."""
    import bfps_amd as B
    n, steps = 64, 64
    kM, scale = n // 2 - 1, 1e-120
    dt = 2.0 ** -7
    nu = x / (dt * kM ** 2)
    print("case: strong damping nu dt kM^2 = %g" % x, flush=True)
    fs = B.vorticity_equation("t", n, precision="double")
    fs.nu, fs.forcing_type = nu, "none"
    w = spectrum(n, 9) * scale
    fs.io_checkpoint(read=True, data=w)
    w0 = fs.cvorticity
    for _ in range(steps):
        fs.step(dt)
    got = fs.cvorticity
    kx = np.arange(n // 2 + 1.0)[None, None, :]
    k1 = np.where(np.arange(n) <= n // 2, np.arange(n), np.arange(n) - n).astype(np.float64)
    k2 = kx ** 2 + k1[:, None, None] ** 2 + k1[None, :, None] ** 2
    inside = (k2 < kM ** 2) & (k2 > 0)

    def mean_error(w, start):
        """Of the mode's vorticity projected on its value at the start."""
        a, b = w[inside] / scale, start[inside] / scale  # (products stay above 1e-308)
        along = (a * b.conj()).sum(-1).real / (np.abs(b) ** 2).sum(-1)
        want = np.exp(-np.longdouble(nu) * np.longdouble(dt) * steps * k2[inside].astype(np.longdouble))
        return np.sqrt(np.mean(((along - want) / want).astype(np.float64) ** 2))

    f, half, back = np.exp(-nu * dt * k2), np.exp(-nu * dt / 2 * k2), np.exp(nu * dt / 2 * k2)
    v = np.random.default_rng(1).standard_normal(k2.shape)
    r = v.copy()
    for _ in range(steps):
        r2 = 0.25 * (3 * r * half + r * f * back)
        r = (r * half + 2 * r2) * (half * (1.0 / 3))
    one = mean_error(scale * r[..., None].astype(np.complex128), scale * v[..., None].astype(np.complex128))
    e = mean_error(got, w0)
    print("  mean error of a mode %.3e, with one exponential a factor %.3e" % (e, one), flush=True)
    assert e < 1.15 * one


def test_inverse_factors_beyond_32_bits(oracle):
    """One step whose last modes are damped by exp(-260): the second stage's
    inverse factors reach exp(130), beyond a 32-bit number's range.  The field
    is so small (1e-120) that they do not raise the nonlinear term to it."""
    import bfps_amd as B
    n, dt = 32, 0.005
    nu = 260 / (dt * (n // 2 - 1) ** 2)
    print("case: inverse factors up to exp(130)", flush=True)
    w0 = spectrum(n, 3) * 1e-120
    fs = B.vorticity_equation("t", n, precision="double")
    fs.nu, fs.forcing_type = nu, "none"
    fs.io_checkpoint(read=True, data=w0)
    fs.step(dt)
    o = oracle.Solver(n, precision="double")
    o.set_physics(nu, "none", 0.0, 2.0, 4.0)
    o.set_cfield("vorticity", w0)
    o.io_projection()
    o.step(dt)
    e = rel(fs.cvorticity, o.get_cfield("vorticity"))
    print("  rel", e, flush=True)
    assert e < TOL


def test_put_switches_the_table(oracle):
    """An unprojected put, then a projection, then steps: each form in turn,
    and the same in a box of an ensemble beside a projected one."""
    import bfps_amd as B
    n, dt = 32, 0.005
    w = spectrum(n, 5)

    def reference(projected):
        o = oracle.Solver(n, precision="double")
        o.set_physics(0.02, "none", 0.0, 2.0, 4.0)
        o.set_cfield("vorticity", w)
        if projected:
            o.io_projection()
        o.step(dt)
        return o.get_cfield("vorticity")

    fs = B.vorticity_equation("t", n, precision="double")
    fs.nu, fs.forcing_type = 0.02, "none"
    for projected in (True, False, True):
        if projected:
            fs.io_checkpoint(read=True, data=w)
        else:
            fs.cvorticity = w
        fs.step(dt)
        assert rel(fs.cvorticity, reference(projected)) < TOL
    ens = B.ensemble([n, n], precision="double")
    for projected in (True, False, True):
        for i, b in enumerate(ens.boxes):
            b.nu, b.forcing_type = 0.02, "none"
            if i == 0 or projected:
                b.io_checkpoint(read=True, data=w)
            else:
                b.cvorticity = w
        ens.step(dt, with_particles=False)
        assert rel(ens.boxes[0].cvorticity, reference(True)) < TOL
        assert rel(ens.boxes[1].cvorticity, reference(projected)) < TOL
