"""Input gradients of more tiles than the device holds at once: the stride phases are put into the order in which the launch ends first, which
is not the order of a launch that is told how to split."""
import numpy as np
import pytest

from common import rand_conv_inputs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    import __graft_entry__ as ge
    return ge.load_package().HipBackend(0)


@pytest.mark.parametrize("shape", [      # N, H, W, C, kh, kw, O, stride: 128x64 tiles
    (150, 24, 20, 48, 5, 5, 16, 2),      # 2.2 tiles to a unit
    (201, 23, 21, 36, 3, 3, 16, 2),      # 3.0, odd extents: phases of different sizes
    (230, 24, 20, 64, 5, 5, 16, 2),      # 3.4
    (180, 24, 40, 64, 5, 2, 32, 2),      # 5.3, phases of 3 and 2 taps
    (150, 16, 90, 20, 4, 7, 16, 3),      # nine phases: three launches, in the order they always had
])
def test_order_of_the_phases_changes_no_bit(be, shape):
    print("shape", shape, flush=True)
    N, H, W, C, kh, kw, O, s = shape
    _, k, dy = rand_conv_inputs(61, *shape)
    _, _, dy2 = rand_conv_inputs(62, *shape)
    half = N // 2
    got = be.conv2d_input_grad(dy, k, s, (H, W))
    pair = be.conv2d_input_grad_pair(dy[:half], dy2[:half], k, s, (H, W))
    be.lib.dh_debug_force_splitk(1)
    try:
        want = be.conv2d_input_grad(dy, k, s, (H, W))
        want_pair = be.conv2d_input_grad_pair(dy[:half], dy2[:half], k, s, (H, W))
    finally:
        be.lib.dh_debug_force_splitk(0)
    np.testing.assert_array_equal(got, want)
    for a, b in zip(pair, want_pair):
        np.testing.assert_array_equal(a, b)
