"""The convolution kernels form fp32 products from bf16 parts (csrc/conv_igemm.inc, csrc/conv_small.hip; the image layer's
filter gradient multiplies in fp32).  Two properties of that: it is no less accurate than the general kernel, which
multiplies in fp32 (each against float64 sums; dense, sparse and small operands, sums of one sign), and operands whose
parts are not finite -- infinities, NaNs, magnitudes next to the largest float -- give what plain fp32 arithmetic
gives, in single and paired launches and with either tile width."""
import numpy as np
import pytest

from common import RTOL, ATOL, convolutions, rand_conv_inputs, same_pad

pytestmark = pytest.mark.gpu

# N, H, W, C, kh, kw, O, stride: one per way an operand tile is staged (32, 64 and 128 columns, whole and partial
# tiles, batch a multiple of 16 or not, split and unsplit contraction)
SHAPES = [
    (3, 9, 7, 32, 3, 3, 24, 1),
    (16, 8, 8, 16, 5, 5, 64, 2),
    (17, 10, 9, 48, 4, 4, 80, 2),
    (16, 16, 16, 64, 5, 5, 160, 2),
    (5, 12, 12, 144, 3, 3, 260, 1),
    # the kernels of the image layer: whole rows, and rows, strips, channel tiles and segments that are part empty
    (3, 64, 64, 3, 5, 5, 64, 2),
    (16, 38, 36, 3, 5, 5, 48, 2),
    (18, 22, 20, 2, 5, 5, 64, 2),
    (9, 19, 17, 4, 4, 4, 36, 1),
]

# Which kernel forms them: launches as small as these leave the tiled one for conv_tiny, two input gradients are too large for that.
WAYS = [(shape, way) for shape in SHAPES[:5] for way in ("tiled", "small")] + [(shape, "image") for shape in SHAPES[5:]]
TOO_LARGE = [(SHAPES[3], "dx"), (SHAPES[4], "dx")]
IMAGE = dict(zip(SHAPES[5:], [("fwd_rows", "dx_col2im", "dk_thin"), ("fwd_rows", "dx_few_channels", "dk_thin"),
                              ("fwd_thin", "dx_col2im", "conv_igemm"), ("fwd_thin", "conv_igemm", "dk_thin")]))


def kernel_of(way, shape, op):
    if way == "image":
        return IMAGE[shape][("fwd", "dx", "dk").index(op)]
    if way == "small" and (shape, op) not in TOO_LARGE:
        return "conv_tiny"
    C, O = shape[3], shape[6]
    return "conv_igemm_fast" if {"fwd": C % 16 == 0, "dx": O % 16 == 0, "dk": C % 4 == 0 and O % 4 == 0}[op] else "conv_igemm"


@pytest.fixture(scope="module")
def be():
    import __graft_entry__ as ge
    return ge.load_package().HipBackend(0)


def product(be, op, x, k, dy, s):
    H, W = x.shape[1:3]
    if op == "fwd":
        return be.conv2d(x, k, (s, s))
    if op == "dx":
        return be.conv2d_input_grad(dy, k, s, (H, W))
    return be.conv2d_kernel_grad(dy, x, s, (same_pad(H, k.shape[0], s)[0], same_pad(W, k.shape[1], s)[0]))


def products(be, x, k, dy, s):
    return {op: product(be, op, x, k, dy, s) for op in ("fwd", "dx", "dk")}


def products_by(be, way, shape, x, k, dy, ops=("fwd", "dx", "dk")):
    """The products, each by the kernel that `way` names."""
    import __graft_entry__ as ge
    if way == "small" and ge.load_package().hipabi.device_info()["compute_units"] != 256:
        pytest.skip("which launches are small ones is that of a device with 256 compute units")
    got = {}
    for op in ops:
        with convolutions(way) as tags:
            got[op] = product(be, op, x, k, dy, shape[-1])
        print("  %s: %s" % (op, tags), flush=True)
        assert [t.split("<")[0] for t in tags] == [kernel_of(way, shape, op)]
    return got


@pytest.mark.parametrize("scale", ["one", "wide", "tiny"])
@pytest.mark.parametrize("shape,way", WAYS)
def test_no_less_accurate_than_fp32_products(be, orc64, shape, way, scale):
    """Error against float64 sums, in the 2-norm over a result of thousands of elements: at most 1.1 times that of
    the fp32 kernel (equal in expectation or better; the ratio of two such norms scatters by a few percent).
    wide: magnitudes over 20 binades, so that the low parts of large values meet the high parts of small ones.
    tiny: activations around 1e-35, whose low parts bf16 holds as subnormals only, unless they are scaled first."""
    print("shape", shape, way, scale, flush=True)
    x, k, dy = rand_conv_inputs(11, *shape)
    if scale == "wide":
        rng = np.random.default_rng(12)
        x, dy = (a * np.exp2(rng.uniform(-10, 10, a.shape)).astype(np.float32) for a in (x, dy))
    if scale == "tiny":
        x, dy = x * np.float32(1e-35), dy * np.float32(1e-35)
    s = shape[-1]
    got = products_by(be, way, shape, x, k, dy)
    be.lib.dh_debug_force_generic_conv(1)
    try:
        plain = products(be, x, k, dy, s)
    finally:
        be.lib.dh_debug_force_generic_conv(0)
    exact = products(orc64, x, k, dy, s)
    for op in got:
        e64 = exact[op].astype(np.float64)
        err, yard = (np.linalg.norm(r[op].astype(np.float64) - e64) for r in (got, plain))
        norm = np.linalg.norm(e64)
        print("  %s: relative error %.3g, fp32 products %.3g" % (op, err / norm, yard / norm), flush=True)
        # 6e-8: both results end in one rounding to fp32
        assert err <= max(1.1 * yard, 6e-8 * norm), op


@pytest.mark.parametrize("what", ["inf", "nan", "largest"])
@pytest.mark.parametrize("shape,way", WAYS)
def test_operands_without_finite_parts(be, orc, shape, way, what):
    print("shape", shape, way, what, flush=True)
    x, k, dy = rand_conv_inputs(13, *shape)
    odd = {"inf": np.inf, "nan": np.nan, "largest": -np.finfo(np.float32).max}[what]
    k[np.abs(k) < 1e-4] = 1e-4    # no infinity times zero that only one order of the sums would meet
    c = min(3, x.shape[3] - 1)
    # (the filter gradient of a thin input multiplies the last columns by the zeros past a row's end as well)
    w = -1 if x.shape[3] > 4 else x.shape[2] // 2
    x[0, 1, 2, c] = odd
    x[-1, -1, w, -1] = -odd
    dy[0, 1, 1, 1] = odd
    if what == "largest":
        x *= np.float32(0.25)     # leaves room for the sums; rounds to infinity only at the full magnitude below
        x[0, 1, 2, c], x[-1, -1, w, -1] = odd, -odd
        k *= np.float32(0.01)
        dy[np.abs(dy) < 1] *= np.float32(0.25)
    s = shape[-1]
    with np.errstate(all="ignore"):
        exp = products(orc, x, k, dy, s)
    got = products_by(be, way, shape, x, k, dy)
    for op in got:
        g, e = got[op], exp[op]
        np.testing.assert_array_equal(np.isnan(g), np.isnan(e), err_msg=op)
        np.testing.assert_array_equal(np.isposinf(g), np.isposinf(e), err_msg=op)
        np.testing.assert_array_equal(np.isneginf(g), np.isneginf(e), err_msg=op)
        fine = np.isfinite(e)
        mag = np.abs(e[fine & (np.abs(e) < 1e20)]).max() if (fine & (np.abs(e) < 1e20)).any() else 1.0
        np.testing.assert_allclose(g[fine], e[fine], rtol=RTOL, atol=ATOL * max(1.0, float(mag)), err_msg=op)


def products64(x, k, dy, s):
    """The three products in float64, one filter tap at a time."""
    x, k, dy = (a.astype(np.float64) for a in (x, k, dy))
    N, H, W, C = x.shape
    kh, kw, _, O = k.shape
    Ho, Wo = dy.shape[1:3]
    pt, pl = (same_pad(n, f, s)[0] // 2 for n, f in ((H, kh), (W, kw)))
    xp = np.zeros((N, max((Ho - 1) * s + kh, H + pt), max((Wo - 1) * s + kw, W + pl), C))
    xp[:, pt:pt + H, pl:pl + W] = x
    y, dxp, dk = np.zeros((N, Ho, Wo, O)), np.zeros_like(xp), np.zeros_like(k)
    for i in range(kh):
        for j in range(kw):
            at = np.s_[:, i:i + (Ho - 1) * s + 1:s, j:j + (Wo - 1) * s + 1:s]
            y += xp[at] @ k[i, j]
            dxp[at] += dy @ k[i, j].T
            dk[i, j] = xp[at].reshape(-1, C).T @ dy.reshape(-1, O)
    return {"fwd": y, "dx": dxp[:, pt:pt + H, pl:pl + W], "dk": dk}


SPARSE = [(shape, way, op) for shape, way in WAYS for op in ("fwd", "dx", "dk")]


@pytest.mark.parametrize("live", ["one", 0.1, 0.5, "positive"])
@pytest.mark.parametrize("shape,way,op", SPARSE)
def test_no_less_accurate_on_sparse_operands(be, shape, way, op, live):
    """As above where few of a sum's products are not zero (activations and gradients behind a relu): fp32 rounds
    such a sum once per product, and the parts of one product must not cost more.  one: one product on average;
    positive: all of them, of one sign.  1.1: the three products of parts that are left out add 3 % to the error of a
    single product, the rest is the scatter of two norms over thousands of elements."""
    print("shape", shape, way, op, live, flush=True)
    x, k, dy = rand_conv_inputs(17, *shape)
    s = shape[-1]
    rng = np.random.default_rng(18)
    terms = {"fwd": k[..., 0].size, "dx": k[:, :, 0].size / s ** 2, "dk": dy[..., 0].size}[op]
    if live == "positive":
        x, k, dy = np.abs(x), np.abs(k), np.abs(dy)
    else:
        part = 1.0 / terms if live == "one" else live
        if op == "dx":
            dy = np.where(rng.random(dy.shape) < part, dy, np.float32(0))
        else:
            x = np.where(rng.random(x.shape) < part, x, np.float32(0))
    got = products_by(be, way, shape, x, k, dy, (op,))[op].astype(np.float64)
    be.lib.dh_debug_force_generic_conv(1)
    try:
        plain = product(be, op, x, k, dy, s).astype(np.float64)
    finally:
        be.lib.dh_debug_force_generic_conv(0)
    exact = products64(x, k, dy, s)[op]
    err, yard, norm = np.linalg.norm(got - exact), np.linalg.norm(plain - exact), np.linalg.norm(exact)
    print("  relative error %.3g, fp32 products %.3g: %.2f" % (err / norm, yard / norm, err / yard), flush=True)
    assert err <= 1.1 * yard


@pytest.mark.parametrize("what", ["small times large", "subnormal times large", "small beside ordinary"])
@pytest.mark.parametrize("shape,way", WAYS)
def test_small_operands(be, shape, way, what):
    """Operands whose parts bf16 holds only in part (below 2^-109) or not at all, where their products count: beside
    a large partner, or as the one small image (filter gradient: the one small channel) of a tile of ordinary ones.
    The slice of the result that they make is as close to float64 sums as the fp32 kernel's (1.1: as above)."""
    print("shape", shape, way, what, flush=True)
    s = shape[-1]
    x, k, dy = rand_conv_inputs(19, *shape)
    inputs = {"fwd": (x, k, dy), "dx": (x, k, dy), "dk": (x, k, dy)}
    where = {"fwd": np.s_[:], "dx": np.s_[:], "dk": np.s_[:]}
    if what == "small beside ordinary":
        x0, dy0, xc = x.copy(), dy.copy(), x.copy()
        x0[0] *= np.float32(1e-36)
        dy0[0] *= np.float32(1e-36)
        xc[..., 0] *= np.float32(1e-36)
        inputs = {"fwd": (x0, k, dy), "dx": (x, k, dy0), "dk": (xc, k, dy)}
        where = {"fwd": np.s_[0], "dx": np.s_[0], "dk": np.s_[:, :, 0]}
    else:
        small, large = (np.float32(v) for v in ((1e-37, 1e16) if what == "small times large" else (1e-41, 1e20)))
        inputs = {"fwd": (x * small, k * large, dy), "dx": (x, k * large, dy * small), "dk": (x * small, k, dy * large)}
    for op in inputs:
        got = products_by(be, way, shape, *inputs[op], (op,))[op]
        be.lib.dh_debug_force_generic_conv(1)
        try:
            plain = product(be, op, *inputs[op], s)
        finally:
            be.lib.dh_debug_force_generic_conv(0)
        exact = products64(*inputs[op], s)[op][where[op]]
        err, yard = (np.linalg.norm(r[where[op]].astype(np.float64) - exact) for r in (got, plain))
        norm = np.linalg.norm(exact)
        print("  %s: relative error %.3g, fp32 products %.3g" % (op, err / norm, yard / norm), flush=True)
        assert err <= 1.1 * yard, op


@pytest.mark.parametrize("op", ["fwd", "dx"])
def test_tile_width_changes_no_result_beside_infinities(be, op):
    """The two tile widths that a launch may be measured with give the same bits where an infinity makes part of a
    tile form its products again in fp32: one filter column of the 160, whose neighbours stay finite."""
    shape = (16, 16, 16, 64, 5, 5, 160, 2) if op == "fwd" else (16, 16, 16, 160, 5, 5, 64, 2)
    x, k, dy = rand_conv_inputs(23, *shape)
    if op == "fwd":
        k[2, 2, 3, 5] = np.inf
    else:
        k[2, 2, 5, 3] = np.inf
    got = []
    be.lib.dh_debug_force_splitk(1)
    try:
        for width in (64, 128):
            be.lib.dh_debug_force_tile_width(width)
            got.append(be.conv2d(x, k, (2, 2)) if op == "fwd" else be.conv2d_input_grad(dy, k, 2, x.shape[1:3]))
    finally:
        be.lib.dh_debug_force_tile_width(0)
        be.lib.dh_debug_force_splitk(0)
    assert np.isfinite(got[0][..., 6:]).all() and not np.isfinite(got[0][..., 5]).all()
    np.testing.assert_array_equal(got[0], got[1])


# the pixel order of tiles that span two pixels (batch half the tile height: 128 rows 128 or 64 wide, 64 rows), a batch
# that is no multiple of 16, and the image layer
PAIRS = [(64, 8, 8, 144, 5, 5, 160, 2), (64, 8, 8, 32, 5, 5, 64, 2), (32, 2, 4, 16, 2, 2, 48, 2), (5, 9, 7, 32, 3, 3, 48, 1),
         (3, 64, 64, 3, 5, 5, 64, 2)]


@pytest.mark.parametrize("odd", [np.inf, np.nan, 1e30])
@pytest.mark.parametrize("where", ["first", "second", "filter"])
@pytest.mark.parametrize("shape", PAIRS)
def test_operands_without_finite_parts_in_paired_launches(be, orc, shape, where, odd):
    """Operands whose products are formed again in fp32 (infinity, NaN, a sum beyond 2^80) in either instance of a
    paired launch or in the filter, and in the single launches: the results are the oracle's, non-finite ones where
    it has them.  The odd values sit where every tap they meet is inside the image."""
    print("shape", shape, where, odd, flush=True)
    N, H, W, C, kh, kw, O, s = shape
    (x1, k, dy1), (x2, _, dy2) = (rand_conv_inputs(seed, *shape) for seed in (29, 31))
    k[np.abs(k) < 1e-4] = 1e-4
    i, j = dy1.shape[1] // 2, dy1.shape[2] // 2
    if where == "filter":
        k[kh // 2, kw // 2, C - 1, O - 3] = odd
    else:
        (x1 if where == "first" else x2)[N // 2, H // 2, W // 2, C - 1] = odd
        (dy1 if where == "first" else dy2)[N - 1, i, j, 1] = odd
    pads = (same_pad(H, kh, s)[0], same_pad(W, kw, s)[0])
    orc.set_threads(8)
    with np.errstate(all="ignore"):
        exp1, exp2 = products(orc, x1, k, dy1, s), products(orc, x2, k, dy2, s)
        both = exp1["dk"] + exp2["dk"]
    got = {"fwd 1": (be.conv2d(x1, k, (s, s)), exp1["fwd"]), "dx 2": (be.conv2d_input_grad(dy2, k, s, (H, W)), exp2["dx"]),
           "dk 2": (be.conv2d_kernel_grad(dy2, x2, s, pads), exp2["dk"])}
    y1, y2 = be.conv2d_pair(x1, x2, k, (s, s))
    got.update({"pair fwd 1": (y1, exp1["fwd"]), "pair fwd 2": (y2, exp2["fwd"])})
    if C % 16 == 0:
        g1, g2 = be.conv2d_input_grad_pair(dy1, dy2, k, s, (H, W))
        got.update({"pair dx 1": (g1, exp1["dx"]), "pair dx 2": (g2, exp2["dx"])})
    got["pair dk"] = (be.conv2d_kernel_grad_pair(dy1, x1, dy2, x2, s, pads), both)
    for op, (g, e) in got.items():
        for kind in (np.isnan, np.isposinf, np.isneginf):
            np.testing.assert_array_equal(kind(g), kind(e), err_msg=op)
        fine = np.isfinite(e)
        plain = np.abs(e[fine & (np.abs(e) < 1e20)])
        np.testing.assert_allclose(g[fine], e[fine], rtol=RTOL, atol=ATOL * max(1.0, float(plain.max(initial=0))), err_msg=op)


@pytest.mark.parametrize("way", ["tiled", "small", "pair"])
@pytest.mark.parametrize("shape", [
    (1, 3, 3, 16, 3, 3, 20, 1),       # less than one slab of 16 output pixels
    (5, 1, 1, 48, 1, 1, 8, 1),        # an image a pixel
    (37, 1, 2, 20, 2, 1, 144, 1),     # two, runs of eight over four images, the last slab part empty
    (7, 2, 5, 32, 3, 3, 48, 1),       # runs that cross rows and images
    (9, 7, 3, 12, 5, 4, 36, 2),       # a row of two pixels, most taps of a pixel in the padding
    (17, 6, 6, 260, 2, 2, 136, 2),    # 128 x 128 tiles, rows and columns left over
])
def test_filter_gradient_of_any_batch(be, shape, way):
    """Batches that are no multiple of 16: the output pixels of a slab are decoded eight at a time and may belong to any
    rows and images.  Element by element within the error of any fp32 summation of n products (n + 2: their own
    rounding and the last one's)."""
    print("shape", shape, way, flush=True)
    H, W, s = shape[1], shape[2], shape[-1]
    (x, k, dy), (x2, _, dy2) = (rand_conv_inputs(seed, *shape) for seed in (37, 41))
    pads = (same_pad(H, shape[4], s)[0], same_pad(W, shape[5], s)[0])
    exact, mag = (products64(f(x), k, f(dy), s)["dk"] for f in (np.asarray, np.abs))
    terms = dy[..., 0].size
    if way == "pair":
        with convolutions(way) as tags:
            got = be.conv2d_kernel_grad_pair(dy, x, dy2, x2, s, pads)
        assert tags[0].startswith("conv_igemm_fast<dk"), tags
        exact, mag = (a + products64(f(x2), k, f(dy2), s)["dk"] for a, f in ((exact, np.asarray), (mag, np.abs)))
        terms *= 2
    else:
        got = products_by(be, way, shape, x, k, dy, ("dk",))["dk"]
    assert (np.abs(got - exact) <= (terms + 2) * 2.0 ** -24 * mag).all()
