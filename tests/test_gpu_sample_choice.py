"""Gradient samples whose trials choose the tracer kernel form (the first tracer
call) or that follow a velocity loop's choice, and after new positions, against
the global gather on the same states.  All forms sum the same products of FP64 weights and
field values in FP64, in other orders; up to 12^3 terms of order the largest
gradient: 1e-12 of it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,n,count,nb,m", [("single", 64, 20000, 4, 1), ("single", 64, 100, 2, 0),
                                                    ("double", 64, 5000, 5, 2), ("single", 48, 3000, 3, 1)])
@pytest.mark.parametrize("steps_first", [0, 2])
def test_gradient_samples(monkeypatch, precision, n, count, nb, m, steps_first):
    import bfps_amd as B
    from bfps_amd import ic
    print("case: gradient samples %s n=%d np=%d nb=%d steps first %d" % (precision, n, count, nb, steps_first), flush=True)

    def run(form):
        if form:
            monkeypatch.setenv("BFPSH_TRACER_KERNEL", form)
        else:
            monkeypatch.delenv("BFPSH_TRACER_KERNEL", raising=False)
        fs = B.vorticity_equation("t", n, precision=precision)
        fs.nu = 0.01
        fs.io_checkpoint(read=True, data=ic.solenoidal_vorticity(n, seed=5, k0=4.0, dtype=fs.cdtype))
        ps = B.particles_system(fs, count, nb, m, 4, step_idx=1)
        ps.put(ic.uniform_positions(count, seed=nb))
        out = []
        for steps in (steps_first, 2):
            for _ in range(steps):
                B.NSVEparticles_step(fs, 0.01)
            fs.gradient_rspace()
            out.append(ps.sample("gradient"))
        ps.put(ic.uniform_positions(count, seed=nb + 1))
        out.append(ps.sample("gradient"))
        return out

    for a, b in zip(run(None), run("gather")):
        print("  ", np.abs(a - b).max() / np.abs(b).max(), flush=True)
        assert np.abs(a - b).max() <= 1e-12 * np.abs(b).max()
