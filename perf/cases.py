"""Timed cases of the solver: what a program that drives it asks for, from one
step of a 16^3 box to ten steps of a 512^3 box with 2^22 tracers.

Kinds of case:

* ``run``: `steps` steps of ``NSVEparticles_step``, then what such a run takes
  to the host: the vorticity and the tracers' whole state (`read` =
  "checkpoint"), or the tracer positions and the velocity spectrum of a run
  between two checkpoints ("positions").
* ``gradient``: the velocity gradient in real space and its nine components
  at every tracer.
* ``stats``: one ``NSVEparticles_do_stats``: moments, histograms, spectra,
  velocity and Lagrangian acceleration at the tracers.
* ``field_stats``: ``field.compute_stats`` of a real-space field handed in.
* ``forward`` / ``inverse``: `fields` fields of host data, one after the other
  through ``put``, ``dft`` or ``ift``, and ``get``.
* ``ensemble``: `steps` steps of boxes of several sizes, then the vorticity
  and the tracer positions of every box.
"""
import math
from fractions import Fraction

import numpy as np
import torch

import bfps_amd as B

BOX = 2 * np.pi
MAXIMUM = 8.0  # histogram half range of the statistics (velocity, vorticity)


def listed():
    return [
        # one step of the smallest box: nothing but latency and launches
        dict(name="step_16_f32", kind="run", n=16, precision="single", dealias="SMOOTH", np=0, nb=1, m=1, steps=1,
             read="checkpoint"),
        # the regression run's box: 32^3, 10^4 tracers, 8 steps between checkpoints
        dict(name="regression_32_f32", kind="run", n=32, precision="single", dealias="SMOOTH", np=10000, nb=1, m=1,
             steps=8, read="checkpoint"),
        # the plain method: 64^3 in FP64, two-thirds rule, 32 steps, no tracers
        dict(name="plain_64_f64", kind="run", n=64, precision="double", dealias="TWO_THIRDS", np=0, nb=1, m=1,
             steps=32, read="checkpoint"),
        # a small production box: many steps, then a checkpoint
        dict(name="run_128_f32", kind="run", n=128, precision="single", dealias="SMOOTH", np=100000, nb=2, m=1,
             steps=64, read="checkpoint"),
        # decaying turbulence without tracers under the two-thirds rule
        dict(name="twothirds_256_f32", kind="run", n=256, precision="single", dealias="TWO_THIRDS", np=0, nb=1, m=1,
             steps=48, read="checkpoint"),
        # FP64 with tracers whose positions are written every 10 steps
        dict(name="run_256_f64", kind="run", n=256, precision="double", dealias="SMOOTH", np=2 ** 20, nb=4, m=1,
             steps=10, read="positions"),
        # the benchmark's workload: 512^3 FP32, 2^22 tracers, positions every 10 steps
        dict(name="run_512_f32", kind="run", n=512, precision="single", dealias="SMOOTH", np=2 ** 22, nb=6, m=2,
             steps=10, read="positions"),
        # velocity-gradient samples of a 256^3 box
        dict(name="gradient_256_f32", kind="gradient", n=256, precision="single", np=2 ** 19, nb=6, m=2),
        # the statistics of a run, every niter_stat steps
        dict(name="stats_128_f64", kind="stats", n=128, precision="double", np=50000, nb=2, m=1),
        # postprocessing of stored fields: real to spectral, spectral to real
        dict(name="forward_128_f32", kind="forward", n=128, precision="single", ncomp=3, fields=1),
        dict(name="inverse_64_f64", kind="inverse", n=64, precision="double", ncomp=9, fields=1),
        # a parameter study: boxes of uneven size and tracer number advanced together
        dict(name="ensemble_f32", kind="ensemble", n32=8, n48=8, n64=6, n128=2, precision="single", np=8000, nb=2,
             m=1, steps=32),
    ]


def draw(rng):
    kind = rng.choice(["run"] * 6 + ["gradient", "stats", "field_stats", "forward", "inverse", "ensemble"])
    precision = rng.choice(["single", "single", "double"])
    if kind == "ensemble":
        return dict(kind=kind, n32=rng.randint(1, 12), n48=rng.randint(0, 12), n64=rng.randint(0, 8),
                    n128=rng.randint(0, 2), precision="single", np=int(math.exp(rng.uniform(math.log(1e3), math.log(3e4)))),
                    nb=rng.randint(1, 4), m=rng.randint(0, 2), steps=rng.randint(4, 40))
    n = rng.choice([16, 32, 48, 64, 128, 128, 256, 256])
    if kind in ("forward", "inverse"):
        return dict(kind=kind, n=min(n, 128), precision=precision, ncomp=rng.choice([1, 3, 9 if n <= 64 else 3]),
                    fields=rng.randint(1, 6))
    if kind == "field_stats":
        return dict(kind=kind, n=min(n, 128), precision=precision, bins=rng.randint(64, 1024))
    nb = min(rng.choice([1, 1, 2, 3, 4, 4, 5, 6, 7, 8, 10]), n // 2 - 1)
    tracers = int(math.exp(rng.uniform(math.log(1e3), math.log(n ** 3 / 16 if n >= 64 else 2e4))))
    if kind in ("gradient", "stats"):
        if kind == "stats":
            precision = "double"
            n = min(n, 128)
        return dict(kind=kind, n=n, precision=precision, np=min(tracers, 2 ** 18), nb=nb, m=rng.randint(0, 2))
    return dict(kind=kind, n=n, precision=precision, dealias=rng.choice(["SMOOTH", "SMOOTH", "TWO_THIRDS"]),
                np=rng.choice([0, tracers, tracers]), nb=nb, m=rng.randint(0, 2),
                steps=rng.randint(1, 64 if n <= 128 else 12), read="checkpoint" if n <= 128 else "positions")


# ------------------------------------------------------------------ inputs
def _cut(n, dealias):
    return float(n // 2 - 1) if dealias == "SMOOTH" else float(n // 3 - 1)


def _viscosity(n):
    return 0.003 * (256.0 / n) ** (4.0 / 3.0)


def _vorticity(n, seed, dtype, dealias="SMOOTH"):
    """Vorticity of a random solenoidal real velocity with E(k) ~ k^(-5/3) up
    to |k_i| = kc and energy 1/2, [ky][kz][kx][3]."""
    kc = max(2, min(n // 3 - 2, 40))
    rng = np.random.default_rng(seed)
    k1 = np.arange(-kc, kc + 1, dtype=np.float64)
    ky, kz, kx = np.meshgrid(k1, k1, np.arange(kc + 1.0), indexing="ij")
    k = np.stack([kx, ky, kz])
    k2 = (k ** 2).sum(0)
    u = rng.standard_normal((3,) + k2.shape) + 1j * rng.standard_normal((3,) + k2.shape)
    u *= np.where(k2 > 0, np.maximum(k2, 1.0) ** (-11.0 / 12.0), 0.0)
    # a real field: the kx = 0 plane is its own mirror image
    u[..., 0] = 0.5 * (u[..., 0] + np.conj(u[:, ::-1, ::-1, 0]))
    u -= k * ((k * u).sum(0) / np.maximum(k2, 1.0))
    u *= np.where((k2 > 0) & (k2 < _cut(n, dealias) ** 2), 1.0, 0.0)
    energy = 0.5 * (np.where(kx == 0, 1.0, 2.0) * (np.abs(u) ** 2).sum(0)).sum()
    w = 1j * np.cross(k, u * math.sqrt(0.5 / energy), axis=0)
    out = np.zeros((n, n, n // 2 + 1, 3), dtype)
    at = np.where(k1 >= 0, k1, k1 + n).astype(np.int64)
    out[np.ix_(at, at, np.arange(kc + 1))] = np.moveaxis(w, 0, -1)
    return out


def _positions(count, seed):
    return np.random.default_rng(seed + 7).random((count, 3)) * BOX


def _complex(case):
    return np.complex64 if case["precision"] == "single" else np.complex128


def _real(case):
    return np.float32 if case["precision"] == "single" else np.float64


def _host_field(case, seed, i=0):
    """Host data of the transform and field statistics cases."""
    n, nc = case["n"], case.get("ncomp", 3)
    rng = np.random.default_rng(seed + 3 + 1000 * i)
    if case["kind"] == "inverse":
        # modes of a real field: conjugate pairs on kx = 0, none at n / 2
        a = rng.standard_normal((n, n, n // 2 + 1, nc)) + 1j * rng.standard_normal((n, n, n // 2 + 1, nc))
        flip = -np.arange(n) % n
        a[:, :, 0] = 0.5 * (a[:, :, 0] + np.conj(a[flip][:, flip][:, :, 0]))
        a[n // 2] = 0
        a[:, n // 2] = 0
        a[:, :, n // 2] = 0
        return a.astype(_complex(case))
    return (rng.standard_normal((n, n, n, nc)) * 1.5).astype(_real(case))


def _boxes(case):
    return [s for s in (32, 48, 64, 128) for _ in range(case["n%d" % s])]


def _box_tracers(case, i):
    return case["np"] // 4 + (case["np"] * (i * 7 % 16)) // 8  # uneven sets


def _solver(case, seed):
    fs = B.vorticity_equation("case", case["n"], precision=case["precision"], dealias=case.get("dealias", "SMOOTH"))
    fs.nu, fs.forcing_type, fs.famplitude, fs.fk0, fs.fk1 = _viscosity(case["n"]), "linear", 0.5, 2.0, 4.0
    fs.io_checkpoint(True, data=_vorticity(case["n"], seed, _complex(case), case.get("dealias", "SMOOTH")))
    ps = None
    if case["np"]:
        ps = B.particles_system(fs, case["np"], case["nb"], case["m"], 4, step_idx=1)
        ps.put(_positions(case["np"], seed))
    return fs, ps


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("forward", "inverse", "field_stats"):
        fs = B.vorticity_equation("case", case["n"], precision=case["precision"])
        nc = case.get("ncomp", 3)
        return dict(case=case, fs=fs, field=B.field(fs, nc),
                    data=[_host_field(case, seed, i) for i in range(case.get("fields", 1))])
    if kind == "ensemble":
        sizes = _boxes(case)
        ens = B.ensemble(sizes, precision=case["precision"])
        systems = []
        for i, (box, n) in enumerate(zip(ens.boxes, sizes)):
            box.nu, box.forcing_type, box.famplitude = _viscosity(n) * (1 + 0.1 * (i % 4)), "linear", 0.5
            box.io_checkpoint(True, data=_vorticity(n, seed + 100 * i, _complex(case)))
            ps = B.particles_system(box, _box_tracers(case, i), case["nb"], case["m"], 4, step_idx=1)
            ps.put(_positions(_box_tracers(case, i), seed + 100 * i))
            systems.append(ps)
        return dict(case=case, ens=ens, systems=systems, dt=[0.5 / n for n in sizes])
    fs, ps = _solver(case, seed)
    return dict(case=case, fs=fs, ps=ps)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "run":
        fs, ps = state["fs"], state["ps"]
        for _ in range(case["steps"]):
            B.NSVEparticles_step(fs, 0.5 / case["n"])
        if case["read"] == "checkpoint":
            out = {"vorticity": fs.cvorticity}
            if ps is not None:
                out["positions"], out["history"] = ps.get()[:2]
            return out
        out = {"spectrum": fs.cospectrum("velocity", "velocity")}
        if ps is not None:
            out["positions"] = ps.getParticlesPositions()
        return out
    if kind == "gradient":
        state["fs"].gradient_rspace()
        return state["ps"].sample("gradient")
    if kind == "stats":
        return B.NSVEparticles_do_stats(state["fs"], state["ps"], MAXIMUM, 4 * MAXIMUM)
    if kind == "ensemble":
        for _ in range(case["steps"]):
            state["ens"].step(state["dt"])
        return {"vorticity": np.concatenate([b.cvorticity.reshape(-1) for b in state["ens"].boxes]),
                "positions": np.concatenate([p.getParticlesPositions() for p in state["systems"]])}
    f = state["field"]
    out = []
    for data in state["data"]:
        f.put(data, kind != "inverse")
        if kind == "field_stats":
            return f.compute_stats(MAXIMUM / math.sqrt(3.0), case["bins"])
        if kind == "forward":
            f.dft()
        else:
            f.ift()
        out.append(f.get())
    return out


# ------------------------------------------------------------------ work
def _transform_flops(n, ncomp):
    return ncomp * 2.5 * n ** 3 * 3 * math.log2(n)


def _box_work(n, es, tracers, nb, steps):
    """Bytes and operations of `steps` steps: the three components of the
    vorticity and the tracers' state and newest right-hand side read and
    written once a step; 27 transforms of one component and the pointwise
    work of three stages, and (2 nb + 2)^3 stencil points of 3 components a
    tracer."""
    pts = (2 * nb + 2) ** 3
    return (steps * (6 * n ** 3 * es + 168 * tracers),
            steps * (_transform_flops(n, 27) + 3 * 100 * n ** 3 + 8 * pts * tracers))


def work(case):
    kind = case["kind"]
    es = 4 if case["precision"] == "single" else 8
    if kind == "ensemble":
        total = [0, 0]
        for i, n in enumerate(_boxes(case)):
            t = _box_tracers(case, i)
            b, f = _box_work(n, es, t, case["nb"], case["steps"])
            total[0] += b + 3 * n ** 3 * es + 24 * t
            total[1] += f
        return {"bytes": total[0], "flops": total[1]}
    n, tracers = case["n"], case.get("np", 0)
    vol = n ** 3 * es
    if kind == "run":
        b, f = _box_work(n, es, tracers, case["nb"], case["steps"])
        b += 3 * vol + 120 * tracers if case["read"] == "checkpoint" else 24 * tracers
        return {"bytes": b, "flops": f}
    pts = (2 * case.get("nb", 0) + 2) ** 3
    if kind == "gradient":
        return {"bytes": 3 * vol + 96 * tracers, "flops": _transform_flops(n, 9) + 20 * pts * tracers}
    if kind == "stats":
        return {"bytes": 3 * vol + 72 * tracers, "flops": _transform_flops(n, 18) + 16 * pts * tracers + 400 * n ** 3}
    if kind == "field_stats":
        return {"bytes": 3 * vol, "flops": _transform_flops(n, 3) + 200 * n ** 3}
    nc = case["ncomp"] * case["fields"]
    return {"bytes": 2 * nc * vol, "flops": _transform_flops(n, nc)}


# ------------------------------------------------------------------ 64-bit values
def _dev(a):
    a = torch.from_numpy(np.ascontiguousarray(a))
    a = a.to("cuda" if torch.cuda.is_available() else "cpu")
    return a.to(torch.complex128 if a.is_complex() else torch.float64)


class _Flow:
    """The vorticity equation in 64 bits with torch's transforms; fields
    [component][ky][kz][kx] and [component][y][z][x]."""

    def __init__(self, n, dealias, vorticity, nu):
        self.n, self.nu = n, nu
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        k1 = torch.arange(n, dtype=torch.float64, device=dev)
        k1 = torch.where(k1 <= n // 2, k1, k1 - n)
        self.k = [torch.arange(n // 2 + 1, dtype=torch.float64, device=dev)[None, None, :], k1[:, None, None],
                  k1[None, :, None]]
        self.k2 = self.k[0] ** 2 + self.k[1] ** 2 + self.k[2] ** 2
        self.kM2 = _cut(n, dealias) ** 2
        self.inside = self.k2 <= self.kM2
        self.ik2 = torch.where(self.k2 > 0, 1.0 / torch.clamp(self.k2, min=1.0), 0.0)
        if dealias == "SMOOTH":
            self.filter = torch.exp(-36.0 * (self.k2 / self.kM2) ** 18)
        else:
            self.filter = (self.k2 < self.kM2).double()
        w = _dev(vorticity).permute(3, 0, 1, 2)
        self.w = self.solenoidal(w * (self.k2 < self.kM2))
        self.band = ((self.k2 >= 4.0) & (self.k2 <= 16.0)).double()

    def solenoidal(self, a):
        d = (self.k[0] * a[0] + self.k[1] * a[1] + self.k[2] * a[2]) * self.ik2
        return torch.stack([a[c] - d * self.k[c] for c in range(3)]) * (self.k2 > 0)

    def curl(self, a):
        k = self.k
        return 1j * torch.stack([k[1] * a[2] - k[2] * a[1], k[2] * a[0] - k[0] * a[2], k[0] * a[1] - k[1] * a[0]])

    def velocity(self, w):
        return self.curl(w) * (self.ik2 * self.inside)

    def real(self, a):
        n = self.n
        return torch.stack([torch.fft.irfftn(c, s=(n, n, n), norm="forward") for c in a])

    def spectral(self, a):
        return torch.stack([torch.fft.rfftn(c) for c in a])

    def nonlinear(self, w):
        u = self.real(self.velocity(w))
        r = torch.linalg.cross(u, self.real(w), dim=0) / float(self.n) ** 3
        return self.solenoidal(self.curl(self.spectral(r) * self.filter) + 0.5 * w * self.band)

    def step(self, dt):
        f1 = torch.exp(-self.nu * self.k2 * dt)
        fh = torch.exp(-self.nu * self.k2 * dt / 2)
        fp = torch.where(self.inside, torch.exp(torch.clamp(self.nu * self.k2 * dt / 2, max=600.0)), 0.0)
        w0 = self.w
        w1 = (w0 + dt * self.nonlinear(w0)) * f1 * self.inside
        w2 = 0.25 * (3 * w0 * fh + (w1 + dt * self.nonlinear(w1)) * fp) * self.inside
        self.w = self.solenoidal((w0 * fh + 2 * (w2 + dt * self.nonlinear(w2))) * (fh / 3.0) * self.inside)

    def shells(self, a):
        """[shell][i][j] sums of Re a_i conj a_j, kx > 0 counted twice."""
        count = int(math.sqrt(self.kM2)) + 2
        at = torch.sqrt(self.k2).long().expand(self.inside.shape)[self.inside]
        twice = torch.where(self.k[0] == 0, 1.0, 2.0).expand(self.inside.shape)[self.inside]
        v = a[:, self.inside]
        out = torch.zeros(count, 3, 3, dtype=torch.float64, device=v.device)
        for i in range(3):
            for j in range(3):
                out[:, i, j] = torch.bincount(at, weights=twice * (v[i] * v[j].conj()).real, minlength=count)[:count]
        return out.cpu().numpy()

    def host(self, a):
        a = a.clone()
        a[..., self.n // 2] = 0
        return a.permute(1, 2, 3, 0)


def _polynomials(n, m):
    """Coefficients (lowest first) of the 2n + 2 weights of (n, m)."""
    def basis(nodes, node):
        c = [Fraction(1)]
        for o in nodes:
            if o != node:
                d = Fraction(1, node - o)
                c = [(c[i - 1] if i else 0) * d - (c[i] if i < len(c) else 0) * o * d for i in range(len(c) + 1)]
        return c

    def at(c, d, x):  # d-th derivative at x = 0 or 1
        return sum(c[i] * math.perm(i, d) for i in range(d, len(c)) if x or i == d)

    left, right = range(-n, n + 1), range(1 - n, n + 2)
    out = []
    for node in range(-n, n + 2):
        if m == 0:
            out.append([float(v) for v in basis(range(-n, n + 2), node)])
            continue
        a, b = (basis(s, node) if node in s else [Fraction(0)] for s in (left, right))
        low = [at(a, d, 0) / math.factorial(d) for d in range(m + 1)]
        rhs = [float(at(b, d, 1) - at(low, d, 1)) for d in range(m + 1)]
        mat = [[float(math.perm(i, d)) for i in range(m + 1, 2 * m + 2)] for d in range(m + 1)]
        out.append([float(v) for v in low] + list(np.linalg.solve(np.array(mat), np.array(rhs))))
    return torch.tensor(out, dtype=torch.float64)


def _interpolate(f, pos, n, nb, m):
    """Components of f ([c][y][z][x]) at the positions: [np][c]."""
    w, c = 2 * nb + 2, f.shape[0]
    poly = _polynomials(nb, m).to(f.device)
    flat = f.reshape(c, -1)
    out = []
    for p in pos.split(max(1, 2 ** 25 // w // c)):
        h = BOX / n
        inbox = p - torch.floor(p / BOX) * BOX
        cell = torch.floor(inbox / h)
        x = inbox / h - cell
        wt = torch.zeros(*x.shape, w, dtype=torch.float64, device=f.device)
        for q in range(poly.shape[1] - 1, -1, -1):
            wt = wt * x[..., None] + poly[:, q]
        node = (cell.long()[..., None] + torch.arange(-nb, nb + 2, device=f.device)) % n
        acc = torch.zeros(c, len(p), dtype=torch.float64, device=f.device)
        for jy in range(w):
            for jz in range(w):
                at = (node[:, 1, jy] * n + node[:, 2, jz])[:, None] * n + node[:, 0]
                acc += (flat[:, at] * wt[:, 0]).sum(-1) * (wt[:, 1, jy] * wt[:, 2, jz])
        out.append(acc.T)
    return torch.cat(out)


def _tracers(case, seed):
    return _dev(_positions(case["np"], seed))


def _advance(flow, case, pos, steps):
    """`steps` steps of flow and tracers; the tracers' newest four slopes."""
    past, n = [], flow.n
    for s in range(steps):
        if pos is not None:
            past = [_interpolate(flow.real(flow.velocity(flow.w)), pos, n, case["nb"], case["m"])] + past[:3]
            c = {1: [1.0], 2: [1.5, -0.5], 3: [23 / 12, -16 / 12, 5 / 12], 4: [55 / 24, -59 / 24, 37 / 24, -9 / 24]}
            pos = pos + 0.5 / n * sum(a * r for a, r in zip(c[min(s + 1, 4)], past))
        flow.step(0.5 / n)
    return pos, past


def _moments(v, estimate):
    """Rows min, means of the powers 1..8, max of each value; minimum and
    maximum start at zero (the magnitude's minimum at its estimate)."""
    v = list(v) + [torch.sqrt((v ** 2).sum(0))]
    out = np.zeros((10, 4))
    for i, x in enumerate(v):
        out[0, i] = min(estimate if i == 3 else 0.0, float(x.min()))
        out[9, i] = max(0.0, float(x.max()))
        p = torch.ones_like(x)
        for k in range(1, 9):
            p = p * x
            out[k, i] = float(p.mean())
    return out


def _cost(n, tracers, nb, steps, ncomp=3):
    """Rough seconds of the 64-bit values on this card."""
    return steps * (0.5 * (n / 512) ** 3 + 0.01 + ncomp / 3 * (tracers * (2 * nb + 2) ** 3 / 1.5e10 + (2 * nb + 2) ** 2 * 2e-4))


def exact(case, seed):
    kind = case["kind"]
    if kind == "ensemble":
        sizes = _boxes(case)
        if sum(_cost(n, _box_tracers(case, i), case["nb"], case["steps"]) for i, n in enumerate(sizes)) > 18:
            return None
        fields, points = [], []
        for i, n in enumerate(sizes):
            flow = _Flow(n, "SMOOTH", _vorticity(n, seed + 100 * i, _complex(case)), _viscosity(n) * (1 + 0.1 * (i % 4)))
            pos, _ = _advance(flow, case, _dev(_positions(_box_tracers(case, i), seed + 100 * i)), case["steps"])
            fields.append(flow.host(flow.w).reshape(-1))
            points.append(pos)
        return {"vorticity": torch.cat(fields), "positions": torch.cat(points)}
    n = case["n"]
    if kind in ("forward", "inverse"):
        out = []
        for i in range(case["fields"]):
            v = _dev(_host_field(case, seed, i))
            if kind == "forward":  # [c][y][z][x] -> [ky][kz][kx][c]
                f = torch.stack([torch.fft.rfftn(c) for c in v.permute(3, 1, 0, 2)]).permute(1, 2, 3, 0).clone()
                f[:, :, n // 2] = 0
            else:
                f = torch.stack([torch.fft.irfftn(c, s=(n, n, n), norm="forward") for c in v.permute(3, 0, 1, 2)])
                f = f.permute(2, 1, 3, 0)
            out.append(f)
        return out
    if kind == "field_stats":
        v = _dev(_host_field(case, seed)).permute(3, 1, 0, 2)
        flow = _Flow(n, "SMOOTH", np.zeros((n, n, n // 2 + 1, 3), np.complex128), 1.0)
        return {"moments": _moments(v, MAXIMUM), "histograms": None,
                "cospectrum": flow.shells(flow.spectral(v) / float(n) ** 3)}
    steps = case.get("steps", 1)
    if _cost(n, case["np"], case["nb"], steps, 9 if kind == "gradient" else 3) > 18:
        return None
    flow = _Flow(n, case.get("dealias", "SMOOTH"), _vorticity(n, seed, _complex(case), case.get("dealias", "SMOOTH")),
                 _viscosity(n))
    pos = _tracers(case, seed) if case["np"] else None
    if kind == "run":
        pos, past = _advance(flow, case, pos, steps)
        out = {}
        if case["read"] == "checkpoint":
            out["vorticity"] = flow.host(flow.w)
            if pos is not None:
                zero = torch.zeros_like(pos)
                out["history"] = torch.stack(([zero] + past[:3] + [zero] * 3)[:4])
        else:
            out["spectrum"] = flow.shells(flow.velocity(flow.w))
        if pos is not None:
            out["positions"] = pos
        return out
    u = flow.velocity(flow.w)
    if kind == "gradient":
        within = (flow.k2 < flow.kM2).double()
        g = torch.stack([1j * flow.k[j] * u[i] * within for j in range(3) for i in range(3)])
        return _interpolate(flow.real(g), pos, n, case["nb"], case["m"])
    # the statistics of vorticity and velocity, then velocity and acceleration at the tracers
    out = {}
    for name, a, top in (("vorticity", flow.w, 4 * MAXIMUM), ("velocity", u, MAXIMUM)):
        out[name] = {"moments": _moments(flow.real(a), top), "histograms": None, "cospectrum": flow.shells(a)}
    ur = flow.real(u)
    out["tracers0/velocity"] = _interpolate(ur, pos, n, case["nb"], case["m"])
    p = torch.zeros_like(u[0])
    for i in range(3):
        for j in range(3):
            p -= flow.k[i] * flow.k[j] * torch.fft.rfftn(ur[i] * ur[j]) * flow.filter
    p *= flow.ik2 * flow.inside / float(n) ** 3
    acc = torch.stack([(0.5 * flow.band - flow.nu * flow.k2) * u[c] - 1j * flow.k[c] * p for c in range(3)]) * flow.inside
    out["tracers0/acceleration"] = _interpolate(flow.real(acc), pos, n, case["nb"], case["m"])
    return out
