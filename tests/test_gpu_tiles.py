"""GPU test of the V-cycle's small levels in few launches (csrc/mg_tile.hip):
several Chebyshev steps and the restriction over overlapping tiles, and the
coarse end of the cycle in one block, against level-by-level launches of the
same arithmetic: the preconditioned vector is the same bit for bit."""
import numpy as np
import pytest

import sfp
from sfp import scenes

pytestmark = pytest.mark.gpu


# extents at the tiles' edges: one cell thick, z rows of 1 to 3 cells past a
# group of four, tiles cut by the grid's end, rows split over several tiles
# (z halos), the largest level the tiles take (2^19 cells) and one past it,
# the first level in the one-block tail (16 x 16 x 16) and just above it
@pytest.mark.parametrize("kind,n", [
    ("magnetic", (16, 16, 16)), ("magnetic", (17, 16, 16)), ("magnetic", (1, 40, 37)),
    ("magnetic", (40, 1, 62)), ("pressure", (21, 19, 18)), ("magnetic", (34, 30, 129)),
    ("pressure", (65, 65, 66)), ("magnetic", (128, 64, 64)), ("magnetic", (129, 64, 64)),
])
@pytest.mark.parametrize("degree,coarse", [(3, 5), (2, 3), (1, 8)])
def test_tiles_match_level_by_level(kind, n, degree, coarse):
    print(f"[case] tiles {kind} {n} degree {degree}/{coarse}", flush=True)
    sc = scenes.random_pressure_scene(n, seed=7) if kind == "pressure" else scenes.magnetic_scene(n, seed=7)
    which = 0 if kind == "pressure" else 1
    with sfp.Context.for_scene(sc, cheby_degree=degree, coarse_cheby_degree=coarse,
                               pressure_coarse_cheby_degree=coarse, max_iters=2) as ctx:
        (ctx.pressure_project if which == 0 else ctx.magnetic_solve)(sc)
        diag = ctx.export_level32(which, 0)["diag"]
        r = np.random.default_rng(4).standard_normal(diag.shape) * (diag > 0)
        z = {}
        for tail in (False, True):
            ctx.set_vcycle_tail(tail)
            z[tail] = ctx.precondition(which, r)
            np.testing.assert_array_equal(z[tail], ctx.precondition(which, r))  # no race
    assert np.abs(z[False]).max() > 0
    np.testing.assert_array_equal(z[True], z[False])


# coarsest levels of 18, 6 and 2 cells (2 mod 4: rows of the dense inverse that
# share 16-byte groups), under first levels of thousands of cells to a handful
@pytest.mark.parametrize("kind,n,coarsest,iters", [
    ("magnetic", (33, 27, 45), 4, True), ("pressure", (64, 96, 96), 4, True), ("magnetic", (96, 90, 64), 4, True),
    ("magnetic", (2, 4, 5), 4, False), ("pressure", (10, 9, 6), 4, False), ("magnetic", (5, 1, 2), 2, False),
])
@pytest.mark.parametrize("coarse", [1, 2, 3, 5])
def test_coarsest_levels_of_two_mod_four_cells(kind, n, coarsest, iters, coarse):
    """One application, and whole solves, as level by level bit for bit."""
    print(f"[case] 2 mod 4 {kind} {n} coarse degree {coarse}", flush=True)
    sc = scenes.random_pressure_scene(n, seed=7) if kind == "pressure" else scenes.magnetic_scene(n, seed=7)
    which = 0 if kind == "pressure" else 1
    out = {}
    with sfp.Context.for_scene(sc, mg_coarsest=coarsest, coarse_cheby_degree=coarse,
                               pressure_coarse_cheby_degree=coarse, max_iters=100) as ctx:
        for tail in (False, True):
            ctx.set_vcycle_tail(tail)
            ctx.reset_warm_start()
            solved = (ctx.pressure_project if which == 0 else ctx.magnetic_solve)(sc)
            assert np.prod(ctx.level_dims(which, ctx.num_levels(which) - 1)) % 4 == 2
            diag = ctx.export_level32(which, 0)["diag"]
            r = np.random.default_rng(4).standard_normal(diag.shape) * (diag > 0)
            out[tail] = (ctx.precondition(which, r), solved)
    assert np.abs(out[False][0]).max() > 0
    np.testing.assert_array_equal(out[True][0], out[False][0])
    if iters:
        (v0, p0, st0), (v1, p1, st1) = ((s[0], s[1], s[2]) for s in (out[False][1], out[True][1]))
        assert st1["converged"] and st1["iterations"] == st0["iterations"]
        for a, b in zip([*v1, *p1], [*v0, *p0]):
            np.testing.assert_array_equal(a, b)
