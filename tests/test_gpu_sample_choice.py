"""Which tracer kernel form runs: the fastest velocity loop's, whatever the first
tracer call is, and between samples of a set without a loop the fastest sample's.
Gradient samples on these routes, and after new positions, against
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


def test_loop_form_after_gradient_samples():
    """10^5 tracers with 2 neighbours in 128^3 FP64: the loop takes half the
    time by the gather (64 us against 126), the 9-plane sample less by columns
    (271 us against 292).  The loop runs in its own form after one gradient
    sample, or several, as it does when it comes first."""
    import bfps_amd as B
    from bfps_amd import ic
    print("case: loop form after gradient samples", flush=True)

    def forms(samples):
        fs = B.vorticity_equation("t", 128, precision="double")
        fs.nu = 0.01
        fs.io_checkpoint(read=True, data=ic.solenoidal_vorticity(128, seed=5, k0=4.0, dtype=fs.cdtype))
        ps = B.particles_system(fs, 100000, 2, 1, 4, step_idx=1)
        ps.put(ic.uniform_positions(100000, seed=3))
        fs.gradient_rspace()
        fs.profile(True)
        before = []
        for _ in range(samples):
            fs.profile(True)
            ps.sample("gradient")
            before += [k for k in fs.profile_report() if k.startswith("sample9")]
        fs.profile(True)
        B.NSVEparticles_step(fs, 0.001)
        loop = [k for k in fs.profile_report() if k.startswith("interp_ab")]
        fs.gradient_rspace()
        fs.profile(True)
        ps.sample("gradient")
        after = [k for k in fs.profile_report() if k.startswith("sample9")]
        fs.close()
        return before, loop, after

    _, loop, after = forms(0)
    print("  loop first:", loop, after, flush=True)
    for samples in (1, 3):
        before, l, a = forms(samples)
        print("  after %d samples:" % samples, before, l, a, flush=True)
        assert l == loop and a == after
        assert before[0] == after[0]  # one form for a single sample before the steps and for all after it
        if samples > 1:
            assert before[1:] == ["sample9_col"] * (samples - 1)
