"""The general convolution kernel (csrc/conv_igemm.inc: channel counts that no wide load fits) and the slice sums
behind it, on the sizes where its addresses can go wrong, against float64 sums."""
import numpy as np
import pytest

from common import rand_conv_inputs, same_pad

pytestmark = pytest.mark.gpu

# N, H, W, C, kh, kw, O, stride
SHAPES = [
    (1, 5, 5, 1, 1, 1, 1, 1),        # one element each way, one slab that is nearly empty
    (2, 9, 7, 18, 4, 4, 30, 2),      # single loads on both operands, 32 columns
    (3, 11, 9, 20, 3, 3, 34, 2),     # 16-byte loads on the activations only
    (3, 11, 9, 18, 3, 3, 36, 2),     # ... on the filter only
    (2, 12, 13, 20, 5, 3, 36, 2),    # ... on both; rectangular filter
    (2, 12, 13, 17, 5, 5, 70, 2),    # 128 x 128 tiles, rows and columns left over
    (9, 17, 10, 7, 3, 2, 130, 1),    # two column tiles
    (1, 10, 10, 6, 2, 2, 10, 3),     # stride phases without any tap
    (20, 33, 33, 18, 4, 4, 30, 2),   # a filter gradient of tens of slices
]


@pytest.fixture(scope="module")
def be():
    import __graft_entry__ as ge
    return ge.load_package().HipBackend(0)


def products(be, x, k, dy, s):
    pads = (same_pad(x.shape[1], k.shape[0], s)[0], same_pad(x.shape[2], k.shape[1], s)[0])
    return {"fwd": be.conv2d(x, k, (s, s)), "dx": be.conv2d_input_grad(dy, k, s, x.shape[1:3]),
            "dk": be.conv2d_kernel_grad(dy, x, s, pads)}


@pytest.mark.parametrize("splits", [0, 1, 21])
@pytest.mark.parametrize("shape", SHAPES)
def test_general_kernel(be, orc64, shape, splits):
    """Element by element within the error of any fp32 summation of n products, n 2^-24 times the sum of their
    magnitudes (n + 2: the products' own rounding, and the float64 sums' rounding to fp32); splits: the library's own choice, none,
    and 21 slices, one run of 16 loads and a remainder."""
    print("shape", shape, "splits", splits, flush=True)
    x, k, dy = rand_conv_inputs(41, *shape)
    N, H, W, C, kh, kw, O, s = shape
    exact = products(orc64, x, k, dy, s)
    mag = products(orc64, np.abs(x), np.abs(k), np.abs(dy), s)
    terms = {"fwd": kh * kw * C, "dx": kh * kw * O, "dk": dy.shape[0] * dy.shape[1] * dy.shape[2]}
    be.lib.dh_debug_force_generic_conv(1)
    be.lib.dh_debug_force_splitk(splits)
    try:
        got = products(be, x, k, dy, s)
    finally:
        be.lib.dh_debug_force_splitk(0)
        be.lib.dh_debug_force_generic_conv(0)
    for op in got:
        bound = (terms[op] + 2) * 2.0 ** -24 * mag[op].astype(np.float64) + 1e-37
        err = np.abs(got[op].astype(np.float64) - exact[op].astype(np.float64))
        assert got[op].shape == exact[op].shape, op
        assert (err <= bound).all(), (op, float((err / bound).max()))


@pytest.mark.parametrize("splits", [1, 2, 3])
@pytest.mark.parametrize("channels", [5, 17, 33, 49, 65, 97])
def test_slabs_in_flight(be, orc64, channels, splits):
    """Contractions of 1, 2, 3, 4, 5 and 7 slabs (forward; input gradient two more channels), whole and in shares of one slab and more:
    the two slabs that are loaded ahead may lie past the share or past the end."""
    test_general_kernel(be, orc64, (2, 6, 7, channels, 1, 1, channels + 2, 1), splits)


@pytest.mark.parametrize("shape", [(2, 9, 7, 18, 4, 4, 30, 2), (26, 10, 10, 30, 5, 5, 3, 2), (40, 16, 16, 18, 4, 4, 30, 1)])
def test_shares_of_four_and_eight_slabs(be, orc64, shape):
    """Either side of the rule for the smallest share, with the library's own choice of the split."""
    test_general_kernel(be, orc64, shape, 0)


@pytest.mark.parametrize("splits", [1, 2])
@pytest.mark.parametrize("channels", [49, 65, 97, 113, 145, 289])
def test_register_sets(be, orc64, channels, splits):
    """Shares of 2 to 19 slabs, odd and even, on either side of the rule for the second register set (more than 4, input gradient more
    than 6); on all tile shapes."""
    for out in (5, 37, 66):
        test_general_kernel(be, orc64, (2, 3, 5, channels, 1, 1, out, 1), splits)      # filter gradient: 2 slabs
        test_general_kernel(be, orc64, (2, 3, 5, out, 1, 1, channels, 1), splits)
    test_general_kernel(be, orc64, (2, 6 + channels % 3, 7, 17, 1, 1, 70, 1), splits)  # 6, 7 and 8 slabs
    test_general_kernel(be, orc64, (5, 6, 5, channels, 1, 1, 37, 1), splits)           # 10 slabs


@pytest.mark.parametrize("channels", [99, 131])
def test_register_sets_with_many_workgroups(be, orc64, channels):
    """More than two workgroups per unit: one set for 7 slabs, two for 9."""
    test_general_kernel(be, orc64, (40, 41, 41, channels, 1, 1, 3, 1), 1)
