"""GPU test of calls that run out of device memory: each allocation of a call is
made to fail in turn (on the host, by asking the allocator for more than there
is); the call reports it and the next one is that of a new context."""
import numpy as np
import pytest

import sfp
from sfp import learn, scenes

pytestmark = pytest.mark.gpu


def _pressure(ctx, sc):
    return ctx.pressure_project(sc)


def _reproject(ctx, sc):
    first = ctx.pressure_project(sc)
    return first + ctx.pressure_project(sc, reproject=True)


def _magnetic(ctx, sc):
    ctx.reset_warm_start()
    return ctx.magnetic_solve(sc)


def _arrays(got):
    return [a for g in got if not isinstance(g, dict) for a in (g if isinstance(g, list) else [g])]


# a small system; one with lists of active cells and the row pairs' segments; the
# network's buffers; levels made again for another coarsest extent
@pytest.mark.parametrize("kind,n,call", [("pressure", (19, 21, 23), _reproject), ("pressure", (72, 60, 132), _pressure),
                                         ("magnetic", (24, 20, 28), _magnetic), ("learned", (32, 32, 32), _magnetic)])
def test_failed_allocations_leave_nothing_half_made(kind, n, call):
    print(f"[case] out of memory {kind} {n}", flush=True)
    sc = scenes.random_pressure_scene(n, 9) if kind == "pressure" else scenes.magnetic_scene(n, seed=9)
    params = dict(tol=1e-6)
    if kind == "learned":
        weights, meta = learn.load_weights()
        params.update(learn.learned_params(meta))

    def context():
        ctx = sfp.Context.for_scene(sc)
        if kind == "learned":
            ctx.set_network(weights)
        ctx.set_params(**params)
        return ctx

    with context() as ctx:
        want = _arrays(call(ctx, sc))
    failures = 0
    for after in range(400):
        with context() as ctx:
            sfp.lib().sfp_test_fail_allocation(after)
            try:
                call(ctx, sc)
                failed = False
            except sfp.SfpError:
                failed = True
            finally:
                sfp.lib().sfp_test_fail_allocation(-1)
            for a, b in zip(_arrays(call(ctx, sc)), want):
                np.testing.assert_array_equal(a, b)
        if not failed:
            break
        failures += 1
    assert 20 < failures < 400


def test_failed_allocation_of_other_levels():
    """A change of the coarsest extent whose levels do not fit, and back."""
    print("[case] out of memory, coarsest extent", flush=True)
    sc = scenes.magnetic_scene((24, 20, 28), seed=9)
    with sfp.Context.for_scene(sc, tol=1e-6) as ctx:
        want = _arrays(_magnetic(ctx, sc))
        for after in range(0, 48, 5):
            ctx.set_params(mg_coarsest=2)
            sfp.lib().sfp_test_fail_allocation(after)
            try:
                with pytest.raises(sfp.SfpError):
                    _magnetic(ctx, sc)
            finally:
                sfp.lib().sfp_test_fail_allocation(-1)
            ctx.set_params(mg_coarsest=4)
            for a, b in zip(_arrays(_magnetic(ctx, sc)), want):
                np.testing.assert_array_equal(a, b)
