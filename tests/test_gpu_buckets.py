"""Tracer sets above 2^20, whose buckets come from the radix sort (those below
are counted), with an odd count: each kernel form, and the automatic choice,
whose trials pass through the bucket counts of all forms on the same buffers.
The reference is a set of the first tracers alone, which the counting path
buckets: a tracer's sums do not depend on the others, so both sets agree to
1e-13 of the largest value where the form is the same (that of equal FP64 sums
in another order), 1e-12 across forms."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
COUNT, FEW = 2 ** 20 + 1, 5001


@pytest.mark.parametrize("form", ["column", "brick", "gather", None])
def test_sorted_buckets(monkeypatch, form):
    import bfps_amd as B
    from bfps_amd import ic
    n, nb, m = 128, 2, 1
    pos = ic.uniform_positions(COUNT, seed=11)
    pos[3000:4000] = pos[3000:4000] * 0.01 + 1.0  # a crowded bucket
    pos[4000:4100] -= 2 * np.pi

    def run(positions, kernel):
        if kernel:
            monkeypatch.setenv("BFPSH_TRACER_KERNEL", kernel)
        else:
            monkeypatch.delenv("BFPSH_TRACER_KERNEL", raising=False)
        fs = B.vorticity_equation("t", n, precision="single")
        fs.nu, fs.forcing_type = 0.01, "linear"
        fs.io_checkpoint(read=True, data=ic.solenoidal_vorticity(n, seed=5, k0=4.0, dtype=fs.cdtype))
        ps = B.particles_system(fs, len(positions), nb, m, 2, step_idx=1)
        ps.put(positions)
        out = []
        for _ in range(2):
            for _ in range(2):
                B.NSVEparticles_step(fs, 0.5 / n)
            fs.gradient_rspace()
            out.append(ps.sample("gradient")[:FEW])
            fs.velocity_rspace()
            out.append(ps.sample("velocity")[:FEW])
        p, r, _, _ = ps.get()
        fs.close()
        return out + [p[:FEW]] + [h[:FEW] for h in r]

    print("case: sorted buckets, %d tracers, form %s" % (COUNT, form), flush=True)
    many, few = run(pos, form), run(pos[:FEW], form or "gather")
    for a, b in zip(many, few):
        e = np.abs(a - b).max()
        print("  ", e / max(1.0, np.abs(b).max()), flush=True)
        assert e <= (1e-13 if form else 1e-12) * max(1.0, np.abs(b).max())
