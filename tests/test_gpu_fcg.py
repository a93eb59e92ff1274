"""GPU test of the flexible CG's iterates: the solution after k iterations, its
directions kept as FP32 preconditioned residuals and summed up to twelve at a
time, against the textbook recurrence in numpy around the library's own
preconditioner and operator."""
import numpy as np
import pytest
import torch

import sfp
from sfp import scenes
from sfp.learn import apply_full

pytestmark = pytest.mark.gpu


def np_fcg(ctx, which, k, active):
    """x after 1 .. k iterations from 0 (Notay's FCG with one direction)."""
    op = ctx.export_level(which, 0)
    r = op["rhs"] * active
    x = np.zeros_like(r)
    p = q = pq = None
    out = []
    for _ in range(k):
        z = ctx.precondition(which, r).astype(np.float64) * active
        w = apply_full(op["diag"], op["cpl"], z) * active
        beta = 0.0 if p is None else float(np.vdot(z, q)) / pq
        p = z if p is None else z - beta * p
        q = w if q is None else w - beta * q
        pq = float(np.vdot(z, w)) if beta == 0.0 else float(np.vdot(p, q))
        alpha = float(np.vdot(z, r)) / pq
        x = x + alpha * p
        r = r - alpha * q
        out.append(x)
    return out


# odd and even cell counts, reductions added by their readers (the first three)
# and by finalize launches, x-plane tiles and flat kernels, an active set of
# part of the grid and all of it
@pytest.mark.parametrize("kind,n", [("pressure", (19, 21, 23)), ("magnetic", (24, 20, 28)),
                                    ("pressure", (48, 48, 48)), ("magnetic", (90, 88, 86)),
                                    ("pressure", (83, 89, 91))])
def test_iterates_match_the_recurrence(kind, n):
    """1 to 17 iterations: below, at and past the twelve whose directions are
    pending at once. Both sides run the same FP32 cycle on residuals equal to
    FP64 rounding, so they differ by that rounding times the few hundred
    operations between, and where a residual rounds to the other FP32 value
    (2^-24 of it): 1e-7 of the solution's change per iteration at the most."""
    print(f"[case] fcg iterates {kind} {n}", flush=True)
    sc = scenes.random_pressure_scene(n, 9) if kind == "pressure" else scenes.magnetic_scene(n, seed=9)
    which = 0 if kind == "pressure" else 1
    got = {}
    with sfp.Context.for_scene(sc, tol=1e-300) as ctx:
        for k in (1, 2, 7, 8, 12, 13, 17):
            ctx.set_params(max_iters=k)
            ctx.reset_warm_start()
            x, st = (ctx.pressure_project(sc)[1:] if which == 0 else ctx.magnetic_solve(sc)[::2])
            assert st["iterations"] == k
            got[k] = x
        active = ctx.export_level32(which, 0)["diag"] > 0
        want = np_fcg(ctx, which, 17, active)
    scale = np.abs(want[-1]).max()
    for k, x in got.items():
        assert np.all(x[~active] == 0)
        np.testing.assert_allclose(x, want[k - 1], rtol=0, atol=1e-7 * scale)
    # a planted mistake in the recurrence (a direction left out) is caught
    assert np.abs(want[1] - want[0]).max() > 100 * 1e-7 * scale


# rings shorter than, equal to and of no whole number of batches of four; small
# grids (batches of any length) and larger ones; solves of up to three rings
@pytest.mark.parametrize("kind,n", [("pressure", (19, 21, 23)), ("magnetic", (24, 20, 28)),
                                    ("pressure", (83, 89, 91)), ("magnetic", (90, 88, 86))])
def test_short_rings_give_the_same_solution(kind, n):
    """Fewer kept residuals (as where memory is short): the same bits, however
    often the solution is brought up to date, from a warm start too, and no
    memory is allocated by a solve longer than the ring."""
    print(f"[case] ring {kind} {n}", flush=True)
    sc = scenes.random_pressure_scene(n, 9) if kind == "pressure" else scenes.magnetic_scene(n, seed=9)
    out = {}
    with sfp.Context.for_scene(sc, tol=1e-12, max_iters=4) as ctx:
        run = ctx.pressure_project if kind == "pressure" else ctx.magnetic_solve
        run(sc)
        free = torch.cuda.mem_get_info()[0]
        for tol, most in ((1e-12, 100), (1e-300, 14)):
            ctx.set_params(tol=tol, max_iters=most)
            for ring in (12, 1, 3, 4, 7):
                ctx.set_ring(ring)
                ctx.reset_warm_start()
                passes = [run(sc), run(sc, reproject=True) if kind == "pressure" else run(sc)]
                out[ring] = [(p[2]["iterations"], p[0], p[1]) for p in passes]
                for (it, *arrays), (it0, *arrays0) in zip(out[ring], out[12]):
                    assert it == it0
                    for a, b in zip(arrays, arrays0):
                        for x, y in zip(a, b):
                            np.testing.assert_array_equal(x, y)
            assert out[12][0][0] > 7  # longer than every short ring
        assert torch.cuda.mem_get_info()[0] == free
