"""FP64 tracers with 4 to 6 neighbours in the narrow columns (16 x 16 cells,
16 x 8 for n = 6) against the brick kernel on the same case: the same FP64 sums
in another order, up to 2744 products of order one, so 1e-13 of the largest
value (the tolerance of the wide FP64 columns)."""
import numpy as np
import pytest

from test_gpu_parity import _fp32_tracer_run as tracer_run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nb,m", [(64, 4, 1), (128, 4, 0), (64, 5, 2), (64, 6, 2), (128, 6, 0)])
def test_narrow_columns(monkeypatch, n, nb, m):
    import bfps_amd as B
    from bfps_amd import ic
    print("case: fp64 narrow columns n=%d nb=%d m=%d" % (n, nb, m), flush=True)
    pos = ic.uniform_positions(15000, seed=60 + nb)
    h = 2 * np.pi / n
    pos[:20] -= 2 * np.pi
    pos[20:40] += 4 * np.pi
    # several batches in one y step, tracers on cell faces, empty columns
    pos[1000:4000] = np.array([5.5, 40.0, 9.5]) * h + np.random.default_rng(nb).random((3000, 3)) * 4 * h
    pos[4000:4100] = np.round(pos[4000:4100] / h) * h
    gp, grhs, gsi, gv, gg = tracer_run(B, n, nb, m, pos, "column", monkeypatch, precision="double")
    bp, brhs, bsi, bv, bg = tracer_run(B, n, nb, m, pos, "brick", monkeypatch, precision="double")
    assert gsi == bsi == 4
    for a, b in ((gp, bp), (grhs, brhs), (gv, bv), (gg, bg)):
        print("  ", np.abs(a - b).max() / np.abs(b).max(), flush=True)
        assert np.abs(a - b).max() <= 1e-13 * max(1.0, np.abs(b).max())
