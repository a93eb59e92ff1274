"""GPU test of the lists of active chunks: the kernels over the flat cell index
on the 256-cell chunks that hold an active cell, against the same kernels on
every chunk."""
import numpy as np
import pytest

import sfp
from sfp import scenes

pytestmark = pytest.mark.gpu

EVERY = 18 + 32  # the default step pairs, no lists


# chunks of whole z rows, of several and across them; a last chunk in part; the
# row-pair kernel's segments (193 to 256 cells per row, one and several tile
# columns, more planes than one activity mask holds); groups of four and pairs
# of cells that cross z rows, planes and the array's ends (nz = 1, 2, 3 mod 4,
# with and without whole groups in a plane and in the grid)
GRIDS = [(96, 90, 64), (84, 82, 80), (67, 83, 100), (36, 80, 200), (96, 90, 256), (160, 72, 196),
         (83, 89, 91), (82, 80, 81), (81, 81, 82), (75, 85, 87), (82, 84, 86)]


@pytest.mark.parametrize("n", GRIDS)
def test_lists_change_nothing(n):
    """A V-cycle and whole solves: the same bits."""
    print(f"[case] active chunks {n}", flush=True)
    sc = scenes.random_pressure_scene(n, 5)
    r = np.random.default_rng(2).normal(size=n)
    got = {}
    for mask in (18, EVERY):
        with sfp.Context.for_scene(sc, tol=1e-8) as ctx:
            ctx.set_fused_pairs(mask)
            vel, p, st = ctx.pressure_project(sc)
            active = ctx.export_level32(0, 0)["diag"] > 0
            z = ctx.precondition(0, r * active) * active
            again = ctx.pressure_project(sc, reproject=True)[1]
        got[mask] = (z, p, vel, st["iterations"], again)
    cells = active.ravel()
    cells = np.concatenate([cells, np.zeros(-cells.size % 256, bool)]).reshape(-1, 256)
    assert 0 < cells.any(axis=1).sum() < len(cells)
    a, b = got[18], got[EVERY]
    np.testing.assert_array_equal(a[0], b[0])
    assert a[3] == b[3] and np.all(a[1][~active] == 0)
    for x, y in [(a[1], b[1]), (a[4], b[4]), *zip(a[2], b[2])]:
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("n", [(84, 82, 80), (36, 80, 200), (83, 89, 91)])
def test_a_new_active_set(n):
    """Solves of other liquids before leave nothing behind: the same bits as a
    new context's, from an empty container, a full one and other pools."""
    print(f"[case] active chunks, new set {n}", flush=True)
    sc = scenes.random_pressure_scene(n, 5)
    with sfp.Context.for_scene(sc, tol=1e-8) as ctx:
        want = ctx.pressure_project(sc)
    with sfp.Context.for_scene(sc, tol=1e-8, max_iters=6) as ctx:
        for phi in (np.full(n, 1.0), np.full(n, -1.0), sc["phi"][::-1].copy(), -sc["phi"]):
            ctx.pressure_project(dict(sc, phi=phi))
        ctx.set_params(max_iters=200)
        got = ctx.pressure_project(sc)
    assert got[2]["iterations"] == want[2]["iterations"]
    np.testing.assert_array_equal(got[1], want[1])
    for a, b in zip(got[0], want[0]):
        np.testing.assert_array_equal(a, b)
