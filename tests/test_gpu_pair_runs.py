"""GPU test of the row-tiled pair of Chebyshev steps (csrc/mg.hip,
k_smooth_pair_rows) over runs of x planes of every length modulo its unrolled
march, of rows a wavefront or half of one holds, and on both sides of the plane size up to which it addresses a run by
32-bit byte offsets (the x-plane tiles above): bit-identical to two flat
steps."""
import numpy as np
import pytest

import sfp
from sfp import scenes

pytestmark = pytest.mark.gpu


# 129 tile columns of y leave one run a column: of all planes up to 56, then two
@pytest.mark.parametrize("n", [(1, 1290, 196), (2, 1290, 196), (3, 1290, 200), (4, 1290, 196), (5, 1290, 196),
                               (56, 1290, 196), (57, 1290, 196), (3, 16380, 256), (3, 16388, 256),
                               # two rows a wavefront: 22 of a tile's, a tile of one, odd counts, short rows
                               (40, 22, 128), (41, 23, 128), (60, 67, 100), (3, 133, 124), (128, 128, 128),
                               (61, 45, 80), (41, 23, 132), (20, 41, 160)])
@pytest.mark.parametrize("pre", [False, True])
def test_runs_match_two_steps(n, pre):
    for kind in ("magnetic", "pressure") if (n[0] in (3, 5) or n[2] <= 160) and n[1] < 2000 else ("magnetic",):
        print(f"[case] pair runs {kind} {n} pre {pre}", flush=True)
        sc = scenes.random_pressure_scene(n, seed=3) if kind == "pressure" else scenes.magnetic_scene(n, seed=3)
        which = 0 if kind == "pressure" else 1
        with sfp.Context.for_scene(sc, max_iters=1) as ctx:
            (ctx.pressure_project if which == 0 else ctx.magnetic_solve)(sc)
            act = ctx.export_level32(which, 0)["diag"] > 0
            rng = np.random.default_rng(5)
            b, x1, d1 = (rng.standard_normal(act.shape, dtype=np.float32) * act for _ in range(3))
            pair, steps = ctx.smooth_pair(which, 0, b, x1, None if pre else d1, 0.31, 0.72, 0.27, 0.66)
            again, _ = ctx.smooth_pair(which, 0, b, x1, None if pre else d1, 0.31, 0.72, 0.27, 0.66)
        assert np.abs(steps).max() > 0
        np.testing.assert_array_equal(pair, steps)
        np.testing.assert_array_equal(again, pair)
