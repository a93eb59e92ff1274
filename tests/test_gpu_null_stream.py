"""GPU test of a busy null stream: a new context's (or network's) arrays are
cleared in the order of its own stream's work, however much other work of the
program waits on the null stream."""
import ctypes as C

import numpy as np
import pytest

import sfp
from sfp import learn, scenes

pytestmark = pytest.mark.gpu


class Busy:
    """Some 0.15 s of clears of 4 GiB on the null stream of the library's runtime."""

    def __enter__(self):
        self.hip, self.p, self.n = sfp.lib(), C.c_void_p(), 4 << 30
        assert self.hip.hipMalloc(C.byref(self.p), C.c_size_t(self.n)) == 0
        for _ in range(150):
            assert self.hip.hipMemsetAsync(self.p, C.c_int(0), C.c_size_t(self.n), None) == 0
        return self

    def waiting(self):
        return self.hip.hipStreamQuery(None) != 0

    def __exit__(self, *exc):
        assert self.hip.hipStreamSynchronize(None) == 0
        assert self.hip.hipFree(self.p) == 0


def test_new_contexts_beside_a_busy_null_stream():
    print("[case] busy null stream, solves", flush=True)
    pool = scenes.random_pressure_scene((40, 36, 44), 9)
    big = scenes.random_pressure_scene((140, 132, 136), 9)
    mag = scenes.magnetic_scene((64, 64, 64), seed=9)
    weights, meta = learn.load_weights()

    # (closing a context waits for the device: whether the null stream was still
    # at work is asked before)
    def project(sc, waiting):
        with sfp.Context.for_scene(sc, tol=1e-8) as ctx:
            vel, p, st = ctx.pressure_project(sc)
            assert waiting()
            return [p, *vel], (st["unknowns"], st["iterations"])

    def solve(network, waiting):
        with sfp.Context.for_scene(mag, tol=1e-8) as ctx:
            if network:
                ctx.set_network(weights)
                ctx.set_params(**learn.learned_params(meta))
            x, field, st = ctx.magnetic_solve(mag)
            assert waiting()
            return [x, *field], st["iterations"]

    for call, arg in ((project, pool), (project, big), (solve, False), (solve, True)):
        want, counts = call(arg, lambda: True)
        with Busy() as busy:
            got, counts_busy = call(arg, busy.waiting)
        assert counts_busy == counts
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a, b)


def test_new_networks_beside_a_busy_null_stream():
    print("[case] busy null stream, network", flush=True)
    weights, _ = learn.load_weights()
    rng = np.random.default_rng(3)
    x = rng.standard_normal((2, 16, 16, 16, 4), dtype=np.float32)
    t = rng.standard_normal((2, 16, 16, 16), dtype=np.float32)

    def gradients(waiting):
        with sfp.UNet(2, 16, 16, 16, training=True) as net:
            net.set_params(weights)
            got = net.gradients(x, t)
            assert waiting()
            return got

    loss, grads = gradients(lambda: True)
    with Busy() as busy:
        loss_busy, grads_busy = gradients(busy.waiting)
    assert loss_busy == loss
    np.testing.assert_array_equal(grads_busy, grads)
