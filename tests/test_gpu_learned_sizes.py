"""The network's convolution layers at the ends of the sizes that st_net_conv_test takes."""
import numpy as np
import pytest

from stokes_to_amd.steady import conv_test

pytestmark = pytest.mark.gpu


def test_weight_gradient_of_more_than_2_31_values():
    """128^3 voxels, 1024 output channels: the gradient of the output has 2^31 values.  It is
    nonzero at a few voxels, among them the first and the last, so that the sums over the
    voxels are short; whole numbers, so that they are exact."""
    R, cin, cout = 128, 16, 1024
    rng = np.random.default_rng(1)
    at = np.r_[0, R ** 3 - 1, rng.integers(0, R ** 3, 30)]
    x = rng.integers(-3, 4, (R, R, R, cin)).astype(np.float32)
    g = np.zeros((R ** 3, cout), np.float32)
    g[at] = rng.integers(-3, 4, (at.size, cout))
    gw, gb = conv_test(R, 27, cin, cout, 0, 2, x.reshape(-1), np.zeros(27 * cin * cout), None, g.reshape(-1))
    ref = np.zeros((27, cin, cout))
    pad = np.pad(x, [(1, 1)] * 3 + [(0, 0)])
    for v in set(at.tolist()):
        i, j, k = np.unravel_index(v, (R,) * 3)
        ref += pad[i:i + 3, j:j + 3, k:k + 3].reshape(27, cin, 1) * g[v]
    assert np.array_equal(gw.reshape(ref.shape), ref)
    assert np.array_equal(gb, g[sorted(set(at.tolist()))].sum(axis=0))
