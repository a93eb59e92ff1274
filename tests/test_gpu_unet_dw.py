"""GPU test of the convolutions' weight gradients at the edges of their tiling,
in whole numbers: a network whose last convolution sees small integers as its
input and its output's gradient, so every sum is exact and has one value."""
import numpy as np
import pytest

import sfp
import unet_params as U

pytestmark = pytest.mark.gpu


# the smallest volume; planes in one, several and partly filled columns along
# each axis; more column runs than blocks; voxels in whole and partial units of 32
@pytest.mark.parametrize("shape", [(1, 4, 4, 4), (2, 8, 12, 20), (1, 8, 40, 36), (1, 12, 4, 68), (3, 16, 36, 4),
                                   (1, 20, 132, 36), (5, 32, 32, 32)])
def test_weight_gradients_of_integers(shape):
    print(f"[case] weight gradient of integers shape={shape}", flush=True)
    rng = np.random.default_rng(sum(shape))
    p = np.zeros(sfp.unet_param_count(), np.float32)
    mix = rng.integers(-1, 2, (16, 4))
    w0, w1 = U.conv_weights(p, 0), U.conv_weights(p, 1)
    w0[13, :, :4] = mix                      # a0 = relu(mix x) from the centre tap
    w1[13] = np.eye(16)                      # e0 = a0; the decoder adds 0: s0 = e0
    U.conv_bias(p, 9)[:] = 1.0               # d0 = 1
    head = rng.permutation(np.repeat([-1.0, 1.0], 8))  # sum 0: the output is 0
    p[U.OFF_HEAD:U.OFF_HEAD + 16] = head
    # |s0| <= 8 and |g| <= 4 (over the count): sums below 2^24 units of 1 / count
    x = rng.integers(-2, 3, shape + (4,))
    t = rng.integers(-2, 3, shape)
    nv = int(np.prod(shape))
    count = 1 << (nv.bit_length() - 1)       # a power of two, so the mean's division is exact
    m = np.zeros(nv)
    m[rng.permutation(nv)[:count]] = 1.0
    m = m.reshape(shape)
    with sfp.UNet(*shape, training=True) as net:
        net.set_params(p)
        got = [net.gradients(x.astype(np.float32), t.astype(np.float32), m.astype(np.float32))[1]
               for _ in range(2)]
    assert np.array_equal(got[0], got[1])
    s0 = np.maximum(x @ mix.T, 0).astype(np.float64)
    dz = -2.0 * m * t / count
    want = np.zeros(p.size)
    ww = U.conv_weights(want, 9)
    pad = np.pad(s0, ((0, 0), (1, 1), (1, 1), (1, 1), (0, 0)))
    for tap in range(27):
        dx, dy, dzz = tap // 9, tap // 3 % 3, tap % 3
        v = pad[:, dx:dx + shape[1], dy:dy + shape[2], dzz:dzz + shape[3]]
        ww[tap] = np.outer(head, np.einsum("bxyz,bxyzc->c", dz, v))
    U.conv_bias(want, 9)[:] = head * dz.sum()
    want[U.OFF_HEAD:U.OFF_HEAD + 16] = dz.sum()
    want[U.OFF_HEAD + 16] = dz.sum()
    np.testing.assert_array_equal(got[0], want.astype(np.float32))
