"""Small launches, whose workgroups have an output tile of 16x16 to 32x32 each and share the contraction among their wavefronts: all four tiles, 16-byte
and single loads, remainders of rows, columns and of the contraction, fewer steps than wavefronts, stride phases without a tap."""
import numpy as np
import pytest
import torch   # before the library: whichever comes first brings the HIP runtime that both use

from common import convolutions, rand_conv_inputs, same_pad
from test_gpu_conv_odd_columns import guarded, result
from test_gpu_conv_split_products import products64

pytestmark = pytest.mark.gpu

# product, tile it must take, (N, H, W, C, kh, kw, O, stride)
CASES = [
    ("fwd", "16x16,8", (1, 16, 16, 128, 5, 5, 252, 2)),    # 100 steps, 16-byte loads of x, remainder of columns
    ("fwd", "16x16,8", (1, 12, 13, 37, 3, 3, 29, 1)),      # 333 k: single loads, a lane's k in two taps
    ("fwd", "32x16,8", (3, 27, 19, 48, 3, 3, 80, 1)),      # 14 steps for 8 wavefronts
    ("fwd", "32x32,8", (20, 33, 33, 18, 4, 4, 30, 2)),
    ("fwd", "32x32,4", (10, 40, 40, 10, 2, 2, 100, 2)),    # 40 k: two steps for four wavefronts
    ("dx", "16x16,8", (1, 32, 32, 64, 5, 5, 128, 2)),      # phases of 9, 6, 6 and 4 taps
    ("dx", "16x16,8", (8, 12, 13, 37, 3, 3, 29, 1)),
    ("dx", "32x16,8", (4, 20, 21, 64, 3, 3, 96, 1)),
    ("dx", "32x16,8", (20, 24, 25, 34, 3, 3, 37, 1)),      # single loads
    ("dx", "32x32,4", (4, 8, 9, 513, 1, 1, 96, 1)),        # one tap
    ("dx", "32x32,4", (40, 21, 19, 40, 1, 1, 100, 2)),     # three of four phases have no tap: zeros
    ("dx", "32x32,8", (6, 24, 25, 64, 3, 3, 64, 1)),
    ("dx", "32x32,8", (1, 30, 28, 512, 5, 5, 48, 2)),      # fewer steps than wavefronts in some phases
    ("dk", "16x16,8", (1, 12, 13, 37, 3, 3, 29, 1)),
    ("dk", "32x16,8", (4, 16, 16, 64, 5, 5, 64, 2)),
    ("dk", "32x32,4", (3, 16, 16, 96, 5, 5, 128, 2)),      # six steps for four wavefronts
    ("dk", "32x32,8", (2, 32, 32, 64, 5, 5, 128, 2)),
]


@pytest.fixture(scope="module")
def A():
    import __graft_entry__ as ge
    return ge.load_package().hipabi


@pytest.fixture(scope="module")
def be(A):
    return A.HipBackend(0)


def product(be, what, x, k, dy, shape):
    N, H, W, C, kh, kw, O, s = shape
    if what == "fwd":
        return be.conv2d(x, k, (s, s))
    if what == "dx":
        return be.conv2d_input_grad(dy, k, s, (H, W))
    return be.conv2d_kernel_grad(dy, x, s, (same_pad(H, kh, s)[0], same_pad(W, kw, s)[0]))


@pytest.mark.parametrize("case", CASES)
def test_small_launches(A, be, orc64, case):
    """Against 64-bit sums: a share of the contraction is rounded once per 16 products in either of its two parts, the shares of 8 wavefronts are added in either
    part and the parts once, by 2^-23 of the magnitudes at most (the matrix cores may cut off); a step left out or counted twice is hundreds of times that."""
    what, tile, shape = case
    print("case", case, flush=True)
    if A.device_info()["compute_units"] != 256:
        pytest.skip("the tiles are those of a device with 256 compute units")
    N, H, W, C, kh, kw, O, s = shape
    x, k, dy = rand_conv_inputs(71, *shape)
    A.profile_enable(1)
    A.profile_reset()
    try:
        got = product(be, what, x, k, dy, shape)
        tags = [r["name"] for r in A.profile_read()]
    finally:
        A.profile_enable(0)
    assert tags == ["conv_tiny<%s,%s>" % (what, tile)]
    np.testing.assert_array_equal(got, product(be, what, x, k, dy, shape))
    orc64.set_threads(8)
    want = product(orc64, what, x, k, dy, shape)
    size = product(orc64, what, np.abs(x), np.abs(k), np.abs(dy), shape)
    contraction = {"fwd": kh * kw * C, "dx": kh * kw * O, "dk": N * H * W}[what]
    bound = (contraction / 8 / 16 + 12) * 2.0 ** -23 * size
    assert (np.abs(got - want) <= bound).all(), np.max(np.abs(got - want) / np.maximum(bound, 1e-300))


@pytest.mark.parametrize("case", [   # tiled, us / here, us
    ("fwd", (44, 25, 25, 92, 3, 3, 16, 1)),     # 27.5 / 42.8: half of a tile's columns past the end
    ("fwd", (97, 34, 32, 5, 4, 4, 45, 2)),      # 11.8 / 19.6: single loads
    ("fwd", (7, 29, 29, 192, 5, 5, 48, 2)),     # 23.7 / 29.0
    ("dx", (420, 8, 6, 48, 1, 1, 112, 1)),      # 9.9 / 11.8: many results, a short contraction
    ("dk", (141, 7, 7, 113, 5, 5, 43, 2)),      # 27.6 / 34.3
])
def test_small_launches_that_tiled_kernels_do_faster(A, be, case):
    what, shape = case
    print("case", case, flush=True)
    if A.device_info()["compute_units"] != 256:
        pytest.skip("the choice is that of a device with 256 compute units")
    x, k, dy = rand_conv_inputs(78, *shape)
    with convolutions("any") as tags:
        product(be, what, x, k, dy, shape)
    assert len(tags) == 1 and tags[0].startswith("conv_igemm"), tags


@pytest.mark.parametrize("act", ["none", "leaky", "tanh"])
@pytest.mark.parametrize("what", ["fwd", "dx"])
def test_bias_and_activation(A, be, what, act):
    """(product + bias) through the activation, as from the product alone."""
    shape = (2, 9, 7, 19, 3, 3, 21, 1)
    N, H, W, C, kh, kw, O, s = shape
    x, k, dy = rand_conv_inputs(72, *shape)
    bias = np.random.default_rng(73).standard_normal(O if what == "fwd" else C).astype(np.float32)
    kind = {"none": A.ACT_NONE, "leaky": A.ACT_LEAKY, "tanh": A.ACT_TANH}[act]
    z = product(be, what, x, k, dy, shape) + bias
    want = {"none": z, "leaky": np.where(z < 0, np.float32(0.2) * z, z), "tanh": np.tanh(z)}[act]
    got = be.conv2d(x, k, (s, s), bias=bias, act=kind, alpha=0.2) if what == "fwd" else be.conv2d_input_grad(dy, k, s, (H, W), bias=bias, act=kind, alpha=0.2)
    np.testing.assert_allclose(got, want, rtol=0 if act != "tanh" else 1e-6, atol=0 if act != "tanh" else 1e-7)


@pytest.mark.parametrize("what", ["fwd", "dx", "dk"])
@pytest.mark.parametrize("odd", ["infinity", "large", "many large"])
def test_sums_that_parts_overflow_on(be, orc, what, odd):
    """An infinity; products that bf16 parts overflow on (2^80 and more) in one wavefront's share; in all of them, where each share is below that and their sum is not."""
    shape = (2, 6, 7, 32, 3, 3, 24, 1)
    N, H, W, C, kh, kw, O, s = shape
    x, k, dy = (np.abs(t) + np.float32(0.5) for t in rand_conv_inputs(74, *shape))
    if odd == "infinity":
        x[1, 2, 3, 4] = k[1, 1, 4, 5] = dy[1, 2, 3, 5] = np.inf
    elif odd == "large":
        x[1, 2, 3, 4] = k[1, 1, 4, 5] = dy[1, 2, 3, 5] = 2.0 ** 60
    else:
        x, k, dy = (t * np.float32(2.0 ** 37) for t in (x, k, dy))
    orc.set_threads(8)
    got, want = product(be, what, x, k, dy, shape), product(orc, what, x, k, dy, shape)
    np.testing.assert_array_equal(np.isfinite(got), np.isfinite(want))
    fine = np.isfinite(want)
    np.testing.assert_allclose(got[fine], want[fine], rtol=288 * 2.0 ** -23, atol=0)     # all terms positive: 288 roundings at most


GENERAL = [   # launches that the general kernel would take: channel counts that its wide loads or the buffer-load kernel do not fit
    ("fwd", (1, 12, 13, 37, 3, 3, 29, 1)),
    ("fwd", (20, 33, 33, 18, 4, 4, 30, 2)),
    ("fwd", (10, 40, 40, 10, 2, 2, 100, 2)),
    ("fwd", (2, 6, 6, 16, 3, 3, 17, 1)),      # 4.5 steps for 8 wavefronts, 16-byte loads
    ("fwd", (1, 9, 9, 1, 1, 1, 5, 1)),        # one product per sum
    ("dx", (8, 12, 13, 37, 3, 3, 29, 1)),
    ("dx", (10, 21, 19, 40, 1, 1, 100, 2)),   # three of four phases have no tap
    ("dx", (3, 9, 9, 5, 1, 1, 1, 1)),
    ("dx", (2, 7, 7, 6, 3, 3, 24, 2)),        # 16-byte loads
    ("dk", (1, 12, 13, 37, 3, 3, 29, 1)),
    ("dk", (5, 3, 4, 7, 2, 2, 9, 1)),
    ("dk", (1, 1, 1, 7, 1, 1, 9, 1)),
]


@pytest.mark.parametrize("case", GENERAL)
def test_no_part_of_a_product_is_left_out(A, be, case):
    """Where the general kernel would multiply in fp32.  At most one product of a sum is not zero here, and 32-bit arithmetic rounds it once.  Of nine products of bf16
    parts the one of the high parts is exact; the others add up to 2^-7 of the product at most, of which the last two steps of that sum may cut off 2^-23 each and
    the steps before them (at most 2^-15 of it) less: 2^-28.  (Six of the nine are 2^-27 off as a rule, 2^-24 at most.)"""
    what, shape = case
    print("case", case, flush=True)
    N, H, W, C, kh, kw, O, s = shape
    x, k, dy = rand_conv_inputs(75, *shape)
    if what == "dk":
        alone = np.zeros_like(x)        # one pixel of one image
        alone[N // 2, H // 2, W // 2] = x[N // 2, H // 2, W // 2]
        x = alone
    else:
        of = x if what == "fwd" else dy
        step = (kh, kw) if what == "fwd" else (-(-kh // s), -(-kw // s))
        alone = np.zeros_like(of)       # one channel of pixels so far apart that no result meets two
        at = np.s_[:, ::step[0], ::step[1], of.shape[3] // 2]
        alone[at] = of[at]
        x, dy = (alone, dy) if what == "fwd" else (x, alone)
    A.profile_enable(1)
    A.profile_reset()
    try:
        got = product(be, what, x, k, dy, shape)
        tags = [r["name"] for r in A.profile_read()]
    finally:
        A.profile_enable(0)
    assert len(tags) == 1 and tags[0].startswith("conv_tiny<" + what)
    exact = products64(x, k, dy, s)[what]
    np.testing.assert_array_less(np.abs(got - exact), 0.5 * np.spacing(np.abs(got)) + 2.0 ** -28 * np.abs(exact) + 1e-300)


@pytest.mark.parametrize("apart", ["none", "operand", "filter", "bias", "result", "all"])
@pytest.mark.parametrize("shape", [
    (2, 9, 7, 32, 3, 3, 48, 1),     # what the buffer-load kernel would take
    (2, 9, 7, 24, 3, 3, 40, 1),     # 16-byte loads and stores
    (1, 11, 10, 36, 3, 3, 44, 2),   # 16-byte stores only
    (1, 12, 13, 37, 3, 3, 29, 1),   # neither
])
@pytest.mark.parametrize("what", ["fwd", "dx", "dk"])
def test_any_address(A, orc64, what, shape, apart):
    """Every operand, the bias or the result 4 bytes past a multiple of 16, through every activation, between words that stay as they are.  The product is held to 64-bit
    sums (bound of test_small_launches), the rest to that product and the bias: exact where the activation is a multiplication or none, else
    within two roundings of tanh and exp in 32 bits."""
    print(what, shape, apart, flush=True)
    N, H, W, C, kh, kw, O, s = shape
    (ph, Ho), (pw, Wo) = A.same_pad(H, kh, s), A.same_pad(W, kw, s)
    lib, P = A.load(), torch.Tensor.data_ptr
    A.check(lib.dh_init(0))
    x, k, dy = rand_conv_inputs(76, *shape)
    ncols = C if what == "dx" else O
    bias = np.random.default_rng(77).standard_normal(ncols).astype(np.float32)

    def placed(a, name):
        first = int(apart in (name, "all"))
        whole = torch.full((a.size + 8,), float("nan"), device="cuda")
        part = whole[first:first + a.size]
        part.copy_(torch.from_numpy(np.ascontiguousarray(a).reshape(-1)))
        assert P(part) % 16 == 4 * first
        return part

    first = int(apart in ("result", "all"))
    xd, kd, yd, bd = placed(x, "operand"), placed(k, "filter"), placed(dy, "filter" if what == "dk" else "operand"), placed(bias, "bias")
    shape_out = {"fwd": dy.shape, "dx": x.shape, "dk": k.shape}[what]

    def run(b, act):
        whole, out = guarded(shape_out, first)
        if what == "fwd":
            A.check(lib.dh_conv2d_fwd(P(xd), P(kd), out, N, H, W, C, kh, kw, O, s, s, ph // 2, pw // 2, Ho, Wo, b, act, 0.2, None))
        elif what == "dx":
            A.check(lib.dh_conv2d_dx(P(yd), P(kd), out, N, Ho, Wo, O, kh, kw, C, s, s, ph // 2, pw // 2, H, W, b, act, 0.2, None))
        else:
            A.check(lib.dh_conv2d_dk(P(xd), P(yd), out, N, H, W, C, Ho, Wo, O, kh, kw, s, s, ph // 2, pw // 2, None))
        return result(whole, shape_out, first)

    with convolutions("any") as tags:
        plain = run(None, A.ACT_NONE)
    assert len(tags) == 1 and tags[0].startswith("conv_tiny<" + what), tags
    exact, size = (products64(f(x), f(k), f(dy), s)[what] for f in (np.asarray, np.abs))
    contraction = {"fwd": kh * kw * C, "dx": kh * kw * O, "dk": N * Ho * Wo}[what]
    assert (np.abs(plain - exact) <= (contraction / 8 / 16 + 12) * 2.0 ** -23 * size).all()
    if what == "dk":
        return
    for b in (None, bias):
        z = plain if b is None else plain + b
        for act, want in {A.ACT_NONE: z, A.ACT_RELU: np.where(z < 0, np.float32(0), z), A.ACT_LEAKY: np.where(z < 0, np.float32(0.2) * z, z),
                          A.ACT_TANH: np.tanh(z.astype(np.float64)), A.ACT_SIGMOID: 1 / (1 + np.exp(-z.astype(np.float64)))}.items():
            got = run(None if b is None else P(bd), act)
            if act in (A.ACT_TANH, A.ACT_SIGMOID):
                np.testing.assert_allclose(got, want, rtol=1e-6, atol=1e-6, err_msg=str(act))
            else:
                np.testing.assert_array_equal(got, want, err_msg=str(act))
