"""GPU test of how a solve ends: the check of its true residual, the velocity
or field update and the caller's copies are enqueued behind the batch that is
expected to converge, and run by the host's decision everywhere else. With the
kernel timings on, a solve never does the former."""
import time

import numpy as np
import pytest
import torch

import sfp
from sfp import scenes

pytestmark = pytest.mark.gpu


def passes(sc, kind, profiled, params):
    """Two passes (the second from a warm start: Reproject, or the next
    magnetic solve of the same scene), each (arrays, stats)."""
    out = []
    with sfp.Context.for_scene(sc, **params) as ctx:
        ctx.profile(profiled)
        for warm in (False, True):
            if kind == "pressure":
                vel, x, st = ctx.pressure_project(sc, reproject=warm)
            else:
                x, vel, st = ctx.magnetic_solve(sc)
            out.append(([x, *vel], st))
    return out


# a small grid (batches of any length) and a larger one (batches of four); a
# tolerance met at once, within, at the end of and after the first batch, and
# never; as many iterations as allowed, and none
@pytest.mark.parametrize("kind,n", [("pressure", (19, 21, 23)), ("magnetic", (24, 20, 28)),
                                    ("magnetic", (90, 88, 86))])
@pytest.mark.parametrize("tol,max_iters", [(0.9, 50), (1e-2, 50), (1e-4, 50), (1e-8, 50), (1e-8, 6),
                                           (1e-8, 0), (1e-300, 14)])
def test_ends_alike(kind, n, tol, max_iters):
    """The two ways run the same kernels in the same order: equal results."""
    print(f"[case] solve end {kind} {n} {tol} {max_iters}", flush=True)
    sc = scenes.random_pressure_scene(n, 9) if kind == "pressure" else scenes.magnetic_scene(n, seed=9)
    params = dict(tol=tol, max_iters=max_iters)
    for (got, st), (want, st0) in zip(passes(sc, kind, False, params), passes(sc, kind, True, params)):
        for key in ("iterations", "converged", "rel_residual", "unknowns"):
            assert st[key] == st0[key], key
        assert st["iterations"] <= max_iters and st["converged"] == (st["rel_residual"] <= tol)
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a, b)


def test_zero_right_hand_side_and_shared_outputs():
    """A zero field gives a zero potential from a warm start too; outputs that
    lie over inputs get the values of separate ones."""
    print("[case] solve end, zero right-hand side, shared outputs", flush=True)
    sc = scenes.magnetic_scene((24, 20, 28), seed=9)
    ptr = lambda ts: [t.data_ptr() for t in ts]  # noqa: E731
    dev = lambda a: torch.tensor(np.ascontiguousarray(a), dtype=torch.float64, device="cuda:0")  # noqa: E731
    with sfp.Context.for_scene(sc, tol=1e-8) as ctx:
        want_x, want_f, _ = ctx.magnetic_solve(sc)
        phi = dev(sc["phi"])
        field = [dev(h) for h in sc["hext"]]
        zero = [torch.zeros_like(h) for h in field]
        x = torch.full_like(phi, 3.0)
        torch.cuda.synchronize()
        st = ctx.magnetic_solve_device(phi.data_ptr(), ptr(zero), sc["chi"], sc["band"], x.data_ptr())
        assert st["iterations"] == 0 and st["converged"] and not x.any()
        ctx.reset_warm_start()
        # the field over the external field, the potential over its first array
        ctx.magnetic_solve_device(phi.data_ptr(), ptr(field), sc["chi"], sc["band"], None, ptr(field))
        for a, b in zip(field, want_f):
            np.testing.assert_array_equal(a.cpu().numpy(), b)
        field = [dev(h) for h in sc["hext"]]
        torch.cuda.synchronize()
        ctx.reset_warm_start()
        ctx.magnetic_solve_device(phi.data_ptr(), ptr(field), sc["chi"], sc["band"], field[0].data_ptr())
        np.testing.assert_array_equal(field[0].flatten()[:phi.numel()].cpu().numpy(), want_x.flatten())
    sc = scenes.random_pressure_scene((19, 21, 23), 9)
    with sfp.Context.for_scene(sc, tol=1e-8) as ctx:
        want_v, want_p, _ = ctx.pressure_project(sc)
        phi, frac, us = dev(sc["phi"]), [dev(a) for a in sc["fraction"]], [dev(a) for a in sc["solid_velocity"]]
        vel = [dev(a) for a in sc["velocity"]]
        jump = [dev(a) for a in sc["jump"]] if sc.get("jump") is not None else None
        torch.cuda.synchronize()
        ctx.pressure_project_device(ptr(vel), phi.data_ptr(), ptr(frac), ptr(us),
                                    None if jump is None else ptr(jump), sc["vol_error"], phi.data_ptr())
        np.testing.assert_array_equal(phi.cpu().numpy(), want_p)
        for a, b in zip(vel, want_v):
            np.testing.assert_array_equal(a.cpu().numpy(), b)


# grids whose kernels write every cell, and skip groups of inactive ones
@pytest.mark.parametrize("n", [(64, 64, 64), (128, 132, 128)])
def test_non_finite_input_leaves_nothing_behind(n):
    """A projection of NaN velocities on a full container fails to converge;
    the next one, on a pool, is that of a new context."""
    print(f"[case] solve end after NaN {n}", flush=True)
    pool = scenes.random_pressure_scene(n, 9)
    full = dict(pool, phi=np.full_like(pool["phi"], -1.0), velocity=[np.full_like(v, np.nan) for v in pool["velocity"]])
    with sfp.Context.for_scene(pool, tol=1e-8) as ctx:
        want_v, want_p, want = ctx.pressure_project(pool)
    with sfp.Context.for_scene(pool, tol=1e-8, max_iters=5) as ctx:
        bad = ctx.pressure_project(full)[2]
        assert not bad["converged"]
        ctx.set_params(max_iters=200)
        vel, p, st = ctx.pressure_project(pool)
    assert st["converged"] and st["iterations"] == want["iterations"]
    np.testing.assert_array_equal(p, want_p)
    for a, b in zip(vel, want_v):
        np.testing.assert_array_equal(a, b)


# odd nz: the matvec's rows and the update's groups of cells are not the same
@pytest.mark.parametrize("n", [(19, 21, 23), (83, 89, 91)])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_non_finite_input_leaves_nothing_behind_on_odd_rows(n, value):
    """As above, and after infinities: the next projection and re-projection
    are those of a new context."""
    print(f"[case] solve end after {value} {n}", flush=True)
    pool = scenes.random_pressure_scene(n, 9)
    full = dict(pool, phi=np.full_like(pool["phi"], -1.0), velocity=[np.full_like(v, value) for v in pool["velocity"]])

    def both(ctx):
        return [ctx.pressure_project(pool, reproject=again) for again in (False, True)]

    with sfp.Context.for_scene(pool, tol=1e-8) as ctx:
        want = both(ctx)
    with sfp.Context.for_scene(pool, tol=1e-8, max_iters=5) as ctx:
        assert not ctx.pressure_project(full)[2]["converged"]
        ctx.set_params(max_iters=200)
        got = both(ctx)
    for (vel, p, st), (want_v, want_p, want_st) in zip(got, want):
        assert st["converged"] and st["iterations"] == want_st["iterations"]
        np.testing.assert_array_equal(p, want_p)
        for a, b in zip(vel, want_v):
            np.testing.assert_array_equal(a, b)


def test_input_error_of_a_failed_call_stays_its_own():
    """The flag left up by a call that failed before reading it (the hook
    raises it from the host) changes neither a magnetic solve nor a
    projection; an open boundary face is still reported, each time."""
    print("[case] input error left behind", flush=True)
    sc = scenes.magnetic_scene((24, 20, 28), seed=9)
    with sfp.Context.for_scene(sc, tol=1e-8) as ctx:
        want = ctx.magnetic_solve(sc)
        ctx.raise_input_error()
        ctx.reset_warm_start()
        x, field, st = ctx.magnetic_solve(sc)
    assert st["converged"] and st["iterations"] == want[2]["iterations"]
    for a, b in zip([x, *field], [want[0], *want[1]]):
        np.testing.assert_array_equal(a, b)
    sc = scenes.random_pressure_scene((19, 21, 23), 9)
    broken = dict(sc, phi=np.full_like(sc["phi"], -1.0), fraction=[np.zeros_like(f) for f in sc["fraction"]])
    with sfp.Context.for_scene(sc, tol=1e-8) as ctx:
        want = ctx.pressure_project(sc)
        for _ in range(2):
            with pytest.raises(sfp.SfpError):
                ctx.pressure_project(broken)
            with pytest.raises(sfp.SfpError):
                ctx.pressure_project(sc, reproject=True)
            ctx.raise_input_error()
            vel, p, st = ctx.pressure_project(sc)
            assert st["iterations"] == want[2]["iterations"]
            for a, b in zip([p, *vel], [want[1], *want[0]]):
                np.testing.assert_array_equal(a, b)


def test_nothing_to_solve_returns_early():
    """A projection without liquid, and one refused for an open boundary face,
    end soon after the assembly: well below half of the share of a projection's
    time that its set-up and first batch take (0.39 at 64^3; 0.1 without)."""
    print("[case] nothing to solve 64", flush=True)
    n = (64, 64, 64)
    faces = lambda v: [torch.full(tuple(n[b] + (b == a) for b in range(3)), v, dtype=torch.float64,  # noqa: E731
                                  device="cuda:0") for a in range(3)]
    ptr = lambda ts: [t.data_ptr() for t in ts]  # noqa: E731
    closed = faces(0.0)
    for a in range(3):
        closed[a].select(a, 0).fill_(1.0)
        closed[a].select(a, n[a]).fill_(1.0)
    Y = torch.arange(64, dtype=torch.float64, device="cuda:0").reshape(1, -1, 1)
    pool = ((Y - 31.7) / 64).expand(n).contiguous()
    best = {}
    for what, phi, frac in (("pool", pool, closed), ("air", torch.ones_like(pool), closed), ("open", pool, faces(0.0))):
        vel, us, p = faces(0.1), faces(0.0), torch.full_like(pool, 3.0)
        torch.cuda.synchronize()
        with sfp.Context(n, 1 / 64, (0, 0, 0)) as ctx:
            for _ in range(40):
                began = time.perf_counter()
                try:
                    st = ctx.pressure_project_device(ptr(vel), phi.data_ptr(), ptr(frac), ptr(us), None, 0.0, p.data_ptr())
                    assert what != "open"
                except sfp.SfpError:
                    assert what == "open"
                best[what] = min(best.get(what, 1.0), time.perf_counter() - began)
            if what == "air":
                assert st["unknowns"] == 0 and st["converged"] and not p.any()
                assert ctx.pressure_project_device(ptr(vel), phi.data_ptr(), ptr(frac), ptr(us), None, 0.0,
                                                   p.data_ptr(), reproject=True)["unknowns"] == 0
    assert best["air"] < 0.2 * best["pool"] and best["open"] < 0.2 * best["pool"], best


# one level, below and above the grids whose host waits for the assembly
@pytest.mark.parametrize("n", [(4, 3, 4), (24, 20, 28), (140, 132, 136)])
def test_empty_projections_between_full_ones(n):
    """With and without liquid in turn: as in new contexts, bit for bit."""
    print(f"[case] empty between full {n}", flush=True)
    pool = scenes.random_pressure_scene(n, 9)
    air = dict(pool, phi=np.ones_like(pool["phi"]))
    drop = np.ones_like(pool["phi"])
    drop[-1, -1, -1] = -0.5  # one liquid cell, the grid's last
    drop = dict(pool, phi=drop)
    want = {}
    for k, sc in (("pool", pool), ("drop", drop)):
        with sfp.Context.for_scene(sc, tol=1e-8) as ctx:
            want[k] = ctx.pressure_project(sc)
    assert want["drop"][2]["unknowns"] == 1
    with sfp.Context.for_scene(pool, tol=1e-8) as ctx:
        for k, sc in (("air", air), ("pool", pool), ("air", air), ("drop", drop), ("air", air), ("pool", pool)):
            vel, p, st = ctx.pressure_project(sc)
            if k == "air":
                assert st["unknowns"] == 0 and st["converged"] and not p.any()
                for a, b in zip(vel, sc["velocity"]):
                    np.testing.assert_array_equal(a, b)
                continue
            for key in ("unknowns", "iterations", "converged"):
                assert st[key] == want[k][2][key]
            for a, b in zip([p, *vel], [want[k][1], *want[k][0]]):
                np.testing.assert_array_equal(a, b)


def test_reprojection_without_unknowns_has_no_pressure():
    """Its pressure is 0, as the projection's before it, not what an earlier
    call left in the library's buffers."""
    print("[case] re-projection without unknowns", flush=True)
    pool = scenes.random_pressure_scene((24, 20, 28), 9)
    air = dict(pool, phi=np.ones_like(pool["phi"]))
    with sfp.Context.for_scene(pool, tol=1e-8) as ctx:
        assert ctx.pressure_project(pool)[1].any()
        ctx.pressure_project(air, want_pressure=False)
        vel, p, st = ctx.pressure_project(air, reproject=True)
    assert st["unknowns"] == 0 and st["converged"] and not p.any()
    for a, b in zip(vel, air["velocity"]):
        np.testing.assert_array_equal(a, b)
