"""Host copies through the pinned chunks: every layout and number of
components comes back bit for bit (no arithmetic: equality), in one chunk and
in several, from two threads at once, and tracer rows in global-index order."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def B():
    import bfps_amd
    bfps_amd.capi.load()
    return bfps_amd


def host_data(fs, nc, real, seed):
    rng = np.random.default_rng(seed)
    n = fs.nx
    if real:
        return rng.standard_normal((n, n, n, nc)).astype(fs.rdtype)
    a = (rng.standard_normal(fs.cshape(nc)) + 1j * rng.standard_normal(fs.cshape(nc))).astype(fs.cdtype)
    a[:, :, n // 2] = 0
    return a


# 16^3: one chunk; 48^3 FP64 with 9 components: 8 MB, uneven last chunk;
# 128^3: more chunks than slots
@pytest.mark.parametrize("n, precision, nc", [(16, "single", 1), (48, "double", 9), (32, "single", 9),
                                              (128, "single", 3), (128, "double", 1)])
def test_round_trip(B, n, precision, nc):
    print("case: transfer n=%d %s nc=%d" % (n, precision, nc), flush=True)
    fs = B.vorticity_equation("t", n, precision=precision, plan_rigor="FFTW_ESTIMATE")
    f = B.field(fs, nc)
    for real in (True, False, True):
        a = host_data(fs, nc, real, n + nc)
        f.put(a, real)
        assert np.array_equal(f.get(), a)
    if nc == 3:
        w = host_data(fs, 3, False, 5)
        fs.cvorticity = w
        assert np.array_equal(fs.cvorticity, w)


def test_two_threads(B):
    """Two contexts share the process's slots."""
    bad = []

    def work(seed):
        fs = B.vorticity_equation("t%d" % seed, 64, precision="double", plan_rigor="FFTW_ESTIMATE")
        f = B.field(fs, 3)
        for i in range(6):
            a = host_data(fs, 3, bool(i % 2), seed + i)
            f.put(a, bool(i % 2))
            if not np.array_equal(f.get(), a):
                bad.append((seed, i))
        f.close()
        fs.close()

    th = [threading.Thread(target=work, args=(100 * t,)) for t in range(3)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad


def test_tracer_rows(B):
    """State and samples of tracers whose slots are not in index order."""
    n, np_ = 32, 70001  # 1.7 MB of positions: several chunks, uneven
    fs = B.vorticity_equation("t", n, precision="double", plan_rigor="FFTW_ESTIMATE")
    rng = np.random.default_rng(3)
    ps = B.particles_system(fs, np_, 1, 1, 3, step_idx=1)
    pos, rhs = rng.random((np_, 3)) * 6, rng.standard_normal((3, np_, 3))
    idx = rng.permutation(np_).astype(np.int64)
    ps.put(pos, rhs, idx)
    order = np.argsort(idx, kind="stable")
    p, r, i, si = ps.get()
    assert np.array_equal(p, pos[order]) and np.array_equal(r, rhs[:, order]) and np.array_equal(i, np.arange(np_))
    assert si == ps.get_step_idx() == 1
    assert np.array_equal(ps.getParticlesPositions(), p) and np.array_equal(ps.getParticlesRhs(), r)
    assert np.array_equal(ps.getParticlesIndexes(), i)
    # a field linear in x, sampled by cubic splines away from the wrap: its own value
    f = B.field(fs, 3)
    x = np.arange(n) * (2 * np.pi / n)
    a = np.zeros((n, n, n, 3))
    a[..., 0], a[..., 1], a[..., 2] = x[None, None, :], x[None, :, None], x[:, None, None]
    f.put(a, True)
    s = ps.sample_compute_field(f)
    inside = ((p > 2 * x[1]) & (p < x[-3])).all(axis=1)
    # Horner sums of three weights: a few roundings of values below 2 pi
    assert np.abs(s - p)[inside].max() < 1e-13
