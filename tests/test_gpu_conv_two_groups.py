"""Launches whose workgroups are two groups of four wavefronts, each with half of the workgroup's k-slabs: shares that are odd or shorter
than the rest, whole and split, remainders of rows and columns, batches that are and are not a multiple of 16, two operand pairs, stride phases of unequal
length, values that are not finite in one group's slabs."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from common import convolutions, rand_conv_inputs, same_pad
from test_gpu_conv_split_products import products64

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# product, instances, (N, H, W, C, kh, kw, O, stride), cut: workgroups' share of slabs and slices of the longest tile
CASES = [
    ("fwd", 1, (37, 27, 19, 48, 3, 3, 80, 1), (27, 1)),      # whole, 27 slabs: 14 and 13; 37 images, 80 of 128 columns
    ("fwd", 1, (16, 24, 20, 80, 3, 3, 196, 1), (23, 2)),     # two slices, the second a slab less; 68 columns in the second tile
    ("fwd", 2, (16, 15, 13, 64, 5, 5, 128, 1), (20, 5)),     # pair
    ("dx", 1, (40, 13, 12, 196, 3, 3, 112, 1), (32, 2)),     # remainder of rows, image-major
    ("dx", 2, (48, 9, 9, 128, 3, 3, 160, 1), (23, 4)),       # pair
    ("dx", 1, (21, 13, 15, 224, 5, 5, 160, 2), (20, 5)),     # phases of 9, 6, 6 and 4 taps and of different extents
    ("dx", 2, (32, 13, 11, 100, 5, 5, 144, 2), (18, 5)),     # ... in a pair, a slab is 16 images of one pixel
    ("dk", 1, (6, 33, 31, 20, 5, 5, 68, 1), (8, 48)),        # smallest share, any batch, many slices shared by threads
    ("dk", 1, (16, 19, 17, 20, 5, 5, 68, 1), (8, 41)),       # a slab is 16 images of one pixel
    ("dk", 2, (16, 19, 17, 20, 5, 5, 132, 1), (20, 33)),     # two pairs of operands
    ("dk", 1, (7, 40, 40, 32, 3, 3, 96, 1), (9, 78)),
]


# enough slabs for two groups with those in the padding, not without
NARROW = [("dx", 1, (421, 2, 2, 240, 3, 3, 240, 1)), ("fwd", 2, (160, 3, 2, 208, 5, 5, 96, 1)), ("dx", 2, (208, 2, 4, 128, 4, 4, 176, 1))]

# as long by the estimate, longer in two groups: 186 / 196, 104 / 111 and 116 / 122 us
ONE_GROUP = [("dk", 2, (181, 7, 5, 288, 5, 5, 336, 2)), ("dk", 2, (245, 5, 5, 320, 5, 5, 176, 2)), ("dk", 1, (64, 42, 42, 80, 3, 3, 80, 1))]


def plan(case, tmp_path_factory):
    """Groups, share, slices and workgroups of a launch of square tiles; 0 groups: it takes narrower ones."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not found")
    exe = str(tmp_path_factory.getbasetemp() / "two_groups_plan")
    if not os.path.exists(exe):
        subprocess.run([hipcc, "--cuda-host-only", "-O1", "-std=c++17", "-Wno-unused-function", "-I" + os.path.join(ROOT, "include"),
                        "-I" + os.path.join(ROOT, "dcgan-cuda_amd", "csrc"), "-o", exe, os.path.join(ROOT, "tests", "two_groups_plan.hip")], check=True)
    what, instances, (N, H, W, C, kh, kw, O, s) = case[:3]
    out = subprocess.run([exe, what] + [str(v) for v in (N, H, W, C, O, kh, s, instances)], capture_output=True, text=True, check=True).stdout
    return tuple(map(int, out.split()))


@pytest.mark.parametrize("case", CASES)
def test_cut_into_two_groups(case, tmp_path_factory):
    """The launches below are the ones this file is about, and no unit gets two workgroups."""
    groups, per, slices, workgroups = plan(case, tmp_path_factory)
    assert (groups, (per, slices)) == (2, case[3]) and workgroups <= 256


@pytest.mark.parametrize("case", NARROW)
def test_slabs_in_the_padding_do_not_count(case, tmp_path_factory):
    assert plan(case, tmp_path_factory)[0] == 0


@pytest.mark.parametrize("case", ONE_GROUP)
def test_filter_gradients_of_long_shares(case, tmp_path_factory):
    assert plan(case, tmp_path_factory)[0] == 1


def launch(be, what, x, x2, k, dy, dy2, shape, instances):
    """The product by a launch of 128x128 tiles: what the plans above are plans of."""
    with convolutions("any") as tags:
        got = products(be, what, x, x2, k, dy, dy2, shape, instances)
    assert tags == ["conv_igemm_fast<%s,128x128>" % what]
    return got


def products(be, what, x, x2, k, dy, dy2, shape, instances):
    N, H, W, C, kh, kw, O, s = shape
    pads = (same_pad(H, kh, s)[0], same_pad(W, kw, s)[0])
    if what == "fwd":
        return be.conv2d_pair(x, x2, k, (s, s)) if instances == 2 else (be.conv2d(x, k, (s, s)),)
    if what == "dx":
        return be.conv2d_input_grad_pair(dy, dy2, k, s, (H, W)) if instances == 2 else (be.conv2d_input_grad(dy, k, s, (H, W)),)
    return (be.conv2d_kernel_grad_pair(dy, x, dy2, x2, s, pads) if instances == 2 else be.conv2d_kernel_grad(dy, x, s, pads),)


def exact(orc64, what, x, x2, k, dy, dy2, shape, instances):
    N, H, W, C, kh, kw, O, s = shape
    pads = (same_pad(H, kh, s)[0], same_pad(W, kw, s)[0])
    one = {"fwd": lambda a, g: orc64.conv2d(a, k, (s, s)), "dx": lambda a, g: orc64.conv2d_input_grad(g, k, s, (H, W)),
           "dk": lambda a, g: orc64.conv2d_kernel_grad(g, a, s, pads)}[what]
    both = [one(x, dy)] + ([one(x2, dy2)] if instances == 2 else [])
    return (both[0] + both[-1],) if what == "dk" and instances == 2 else tuple(both)


@pytest.fixture(scope="module")
def be():
    import __graft_entry__ as ge
    return ge.load_package().HipBackend(0)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_sums_of_both_groups(be, orc64, case):
    """Against 64-bit sums.  A sum is rounded once per slab of 16 products in either of its two parts and once per slice, by 2^-23 of the
    magnitudes added up at most (the matrix cores may cut off); the products themselves are good for 2^-24.  A slab that is missing or counted
    twice is some hundred times that."""
    what, instances, shape, _ = case
    print("case", case, flush=True)
    N, H, W, C, kh, kw, O, s = shape
    x, k, dy = rand_conv_inputs(51, *shape)
    x2, _, dy2 = rand_conv_inputs(52, *shape)
    orc64.set_threads(8)
    got = launch(be, what, x, x2, k, dy, dy2, shape, instances)
    again = products(be, what, x, x2, k, dy, dy2, shape, instances)
    want = exact(orc64, what, x, x2, k, dy, dy2, shape, instances)
    size = exact(orc64, what, *(np.abs(t) for t in (x, x2, k, dy, dy2)), shape, instances)
    contraction = {"fwd": kh * kw * C, "dx": kh * kw * O, "dk": N * H * W * instances}[what]
    for g, a, w, m in zip(got, again, want, size):
        np.testing.assert_array_equal(g, a)
        assert (np.abs(g - w) <= (contraction / 16 + 4) * 2.0 ** -23 * m).all(), np.max(np.abs(g - w) / m)


@pytest.mark.gpu
@pytest.mark.parametrize("tap", [(0, 0), (2, 2)])   # in the first group's slabs, in the second's
def test_infinity_in_one_groups_slabs(be, orc, tap):
    """One filter element is infinite: the infinities of its column are those of plain fp32 arithmetic; the other columns keep their values,
    from either kind of products."""
    shape = CASES[0][2]
    x, k, dy = rand_conv_inputs(53, *shape)
    plain = be.conv2d(x, k, (1, 1))
    k[tap[0], tap[1], 5, 33] = np.inf
    orc.set_threads(8)
    got, want = be.conv2d(x, k, (1, 1)), orc.conv2d(x, k, (1, 1))
    others = np.arange(shape[6]) != 33
    np.testing.assert_array_equal(np.isposinf(got[..., 33]), np.isposinf(want[..., 33]))
    np.testing.assert_array_equal(np.isneginf(got[..., 33]), np.isneginf(want[..., 33]))
    np.testing.assert_allclose(got[..., others], plain[..., others], rtol=0, atol=2.0 ** -23 * 31 * 432 * 0.02)


@pytest.mark.gpu
@pytest.mark.parametrize("odd", [np.inf, np.nan, 1e30])
@pytest.mark.parametrize("case,instance", [(case, i) for case in CASES for i in range(case[1])])
def test_values_without_finite_parts(be, orc64, case, instance, odd):
    """An infinity, a NaN, a value that bf16 parts overflow on, in either instance: one in the first image and one in the last, in the first and in the last channel,
    where every tap that they meet is inside the image.  Results of a forward product or an input gradient that they reach have them in different slabs; a
    filter gradient has them at the beginning and at the end of its contraction.  What is not finite is that of plain arithmetic; the rest is as near
    to 64-bit sums as any fp32 summation of n products, n 2^-24 of the magnitudes (n + 2: their own rounding and the last one's)."""
    what, instances, shape, _ = case
    print("case", case, instance, odd, flush=True)
    N, H, W, C, kh, kw, O, s = shape
    ins = [list(rand_conv_inputs(seed, *shape)) for seed in (54, 55)]
    ins[1][1] = ins[0][1]
    ins[0][1][np.abs(ins[0][1]) < 1e-4] = 1e-4      # no infinity times zero
    Ho, Wo = ins[0][2].shape[1:3]
    pt, pl = same_pad(H, kh, s)[0] // 2, same_pad(W, kw, s)[0] // 2
    if what == "fwd":
        t = ins[instance][0]
        t[0, H // 2, W // 2, 0] = odd
        t[N - 1, H // 2, W // 2, C - 1] = -odd
    else:                                           # first and last pixel of dy whose window is inside
        t = ins[instance][2]
        t[0, -(-pt // s), -(-pl // s), 0] = odd
        t[N - 1, (H - kh + pt) // s, (W - kw + pl) // s, O - 1] = -odd
    (x, k, dy), (x2, _, dy2) = ins
    orc64.set_threads(8)
    with np.errstate(all="ignore"):
        want = exact(orc64, what, x, x2, k, dy, dy2, shape, instances)
        size = exact(orc64, what, *(np.abs(t) for t in (x, x2, k, dy, dy2)), shape, instances)
    got = launch(be, what, x, x2, k, dy, dy2, shape, instances)
    terms = {"fwd": kh * kw * C, "dx": kh * kw * O, "dk": N * Ho * Wo * instances}[what]
    assert odd == 1e30 or not all(np.isfinite(w).all() for w in want)
    for g, w, m in zip(got, want, size):
        for kind in (np.isnan, np.isposinf, np.isneginf):
            np.testing.assert_array_equal(kind(g), kind(w))
        fine = np.isfinite(w)
        err, bound = np.abs(g[fine].astype(np.float64) - w[fine]), (terms + 2) * 2.0 ** -24 * m[fine].astype(np.float64)
        assert (err <= bound).all(), np.max(err / bound)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_no_less_accurate_than_fp32_products(be, case):
    """Error against float64 sums in the 2-norm, at most 1.1 times that of the general kernel, which multiplies in fp32 (the ratio of two such norms
    scatters by a few percent)."""
    what, instances, shape, _ = case
    print("case", case, flush=True)
    s = shape[-1]
    (x, k, dy), (x2, _, dy2) = (rand_conv_inputs(seed, *shape) for seed in (56, 57))
    got = launch(be, what, x, x2, k, dy, dy2, shape, instances)
    be.lib.dh_debug_force_generic_conv(1)
    try:
        plain = [products(be, what, a, None, k, g, None, shape, 1)[0] for a, g in ((x, dy), (x2, dy2))[:instances]]
    finally:
        be.lib.dh_debug_force_generic_conv(0)
    want = [products64(a, k, g, s)[what] for a, g in ((x, dy), (x2, dy2))[:instances]]
    if what == "dk":
        plain, want = [sum(plain)], [sum(want)]
    for g, p, w in zip(got, plain, want):
        err, yard = np.linalg.norm(g - w), np.linalg.norm(p - w)
        print("  relative error %.3g, fp32 products %.3g: %.2f" % (err / np.linalg.norm(w), yard / np.linalg.norm(w), err / yard), flush=True)
        assert err <= 1.1 * yard
