"""The write-out of the buffer-load convolution kernel and the sums of its slices: every activation with and without a
bias, whole and split, with 16-byte and with single stores, and filter gradients whose many slices are shared by
several threads."""
import numpy as np
import pytest
import torch   # before the library: whichever comes first brings the HIP runtime that both use

from common import convolutions, rand_conv_inputs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    import __graft_entry__ as ge
    A = ge.load_package().hipabi
    A.check(A.load().dh_init(0))
    return A


def device(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def room(n, offset):
    """A device tensor of n floats whose address is a multiple of 16 plus 4 * offset."""
    return torch.full((n + 4,), np.nan, device="cuda")[offset:offset + n]


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("shape", [(3, 9, 7, 16, 3, 3, 36, 1), (2, 20, 20, 16, 3, 3, 132, 1)])   # one and two column tiles, remainders
def test_activations(A, shape, splits, offset):
    """The activation of (product + bias), element by element, from the product alone as the same launch plan gives it: exact
    where the activation is one multiplication or none, else within 1e-6 (two roundings of tanh and exp in 32 bits)."""
    print("shape", shape, "splits", splits, "offset", offset, flush=True)
    N, H, W, C, kh, kw, O, s = shape
    x, k, _ = rand_conv_inputs(5, *shape)
    rng = np.random.default_rng(6)
    bias = rng.standard_normal(O).astype(np.float32)
    bias[:3] = -np.inf, np.nan, np.inf
    lib, P = A.load(), torch.Tensor.data_ptr
    (ph, Ho), (pw, Wo) = A.same_pad(H, kh, s), A.same_pad(W, kw, s)
    xd, kd, bd = device(x), device(k), room(O, offset)
    bd.copy_(device(bias))
    geom = (N, H, W, C, kh, kw, O, s, s, ph // 2, pw // 2, Ho, Wo)

    def run(b, act, alpha):
        y = room(N * Ho * Wo * O, offset)
        A.check(lib.dh_conv2d_fwd(P(xd), P(kd), P(y), *geom, b, act, alpha, None))
        return y.cpu().numpy().reshape(-1, O)

    lib.dh_debug_force_splitk(splits)
    try:
        plain = run(None, A.ACT_NONE, 0.0)
        assert np.isfinite(plain).all()
        for b in (None, bias):
            z = plain if b is None else plain + b
            below = z < 0
            expected = {
                A.ACT_NONE: z,
                A.ACT_RELU: np.where(below, np.float32(0), z),
                A.ACT_LEAKY: np.where(below, np.float32(0.2) * z, z),
                A.ACT_TANH: np.tanh(z.astype(np.float64)),
                A.ACT_SIGMOID: 1 / (1 + np.exp(-z.astype(np.float64))),
            }
            for act, exp in expected.items():
                got = run(None if b is None else P(bd), act, 0.2)
                if act in (A.ACT_TANH, A.ACT_SIGMOID):
                    np.testing.assert_allclose(got, exp, rtol=1e-6, atol=1e-6, err_msg=str(act))
                else:
                    np.testing.assert_array_equal(got, exp, err_msg=str(act))
    finally:
        lib.dh_debug_force_splitk(0)


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("shape", [  # tile of the filter gradient
    (9, 27, 19, 48, 3, 3, 80, 1),    # 128 x 128, 48 of 128 columns past the end
    (9, 27, 19, 16, 3, 3, 64, 1),    # 128 x 64
    (9, 27, 19, 16, 3, 3, 20, 1),    # 128 x 32
    (9, 27, 19, 16, 2, 2, 64, 1),    # 64 x 64
])
def test_many_slices(A, shape, offset):
    """One thread an output and eight sharing its slices (58, 97 and 145 of them, 193 paired: counts that eight does not
    divide), every tile with the same number; single and paired, against float64.  Tolerance: a partial sum of K products of numbers
    in (-1, 1) is about sqrt(K) / 3, each of up to K roundings at most 2^-25 of that, and they add up as their root:
    K / 3 * 2^-25, taken six times."""
    print("shape", shape, "offset", offset, flush=True)
    N, H, W, C, kh, kw, O, s = shape
    (ph, Ho), (pw, Wo) = A.same_pad(H, kh, s), A.same_pad(W, kw, s)
    lib, P = A.load(), torch.Tensor.data_ptr
    ins = [rand_conv_inputs(seed, *shape)[::2] for seed in (7, 8)]
    pad = torch.nn.functional.pad
    exp = []
    for x, dy in ins:
        xp = pad(torch.from_numpy(x).double(), (0, 0, pw // 2, pw - pw // 2, ph // 2, ph - ph // 2)).numpy()
        exp.append(np.stack([np.einsum("bijc,bijo->co", xp[:, i:i + Ho, j:j + Wo], dy.astype(np.float64), optimize=True)
                             for i in range(kh) for j in range(kw)]).reshape(kh, kw, C, O))
    dev = [(device(x), device(dy)) for x, dy in ins]
    geom = (N, H, W, C, Ho, Wo, O, kh, kw, s, s, ph // 2, pw // 2)
    tol = N * Ho * Wo * 2.0 ** -24
    for splits in (63, 64, 100, 200):
        lib.dh_debug_force_splitk(splits)
        try:
            d = room(kh * kw * C * O, offset)
            A.check(lib.dh_conv2d_dk(P(dev[0][0]), P(dev[0][1]), P(d), *geom, None))
            got = d.cpu().numpy().reshape(kh, kw, C, O)
            np.testing.assert_allclose(got, exp[0], rtol=0, atol=tol, err_msg="%d splits" % splits)
            again = room(kh * kw * C * O, offset)
            A.check(lib.dh_conv2d_dk(P(dev[0][0]), P(dev[0][1]), P(again), *geom, None))
            np.testing.assert_array_equal(got, again.cpu().numpy().reshape(kh, kw, C, O))
            A.check(lib.dh_conv2d_dk_pair(P(dev[0][0]), P(dev[0][1]), P(dev[1][0]), P(dev[1][1]), P(d), *geom, None))
            np.testing.assert_allclose(d.cpu().numpy().reshape(kh, kw, C, O), exp[0] + exp[1], rtol=0, atol=2 * tol,
                                       err_msg="%d splits, pair" % splits)
        finally:
            lib.dh_debug_force_splitk(0)


@pytest.mark.parametrize("shape", [  # either side of the rule for the smallest share of a small launch
    (4, 16, 16, 64, 3, 3, 64, 1),    # shares of 4 slabs, 9 slices
    (1, 16, 16, 80, 4, 4, 64, 1),    # 80 slabs, 20 slices
    (1, 16, 16, 96, 4, 4, 64, 1),    # 96 slabs: shares of 8
    (9, 16, 16, 80, 4, 4, 144, 1),   # 18 x 80 slabs and more: shares of 8
])
def test_small_launches(A, shape):
    """Forward product and input gradient of the tiled kernel with its own split against the same launch cut differently (one slice):
    two orders of the sums differ by at most n 2^-24 of the sum of the magnitudes, here bounded by that of the largest."""
    print("shape", shape, flush=True)
    be = A.HipBackend(0)
    N, H, W, C, kh, kw, O, s = shape
    x, k, dy = rand_conv_inputs(9, *shape)
    with convolutions("tiled", level=2) as tags:
        got = be.conv2d(x, k, (s, s)), be.conv2d_input_grad(dy, k, s, (H, W))
    assert all(t.startswith(("conv_igemm_fast<", "hbm:")) for t in tags) and any("splitk_reduce" in t for t in tags), tags
    mag = be.conv2d(np.abs(x), np.abs(k), (s, s)), be.conv2d_input_grad(np.abs(dy), np.abs(k), s, (H, W))
    be.lib.dh_debug_force_splitk(1)
    try:
        whole = be.conv2d(x, k, (s, s)), be.conv2d_input_grad(dy, k, s, (H, W))
    finally:
        be.lib.dh_debug_force_splitk(0)
    for g, w, m, n in zip(got, whole, mag, (kh * kw * C, kh * kw * O)):
        assert np.abs(g - w).max() <= 2.0 ** -24 * n * m.max()


def filter_gradient_float64(A, x, dy, kh, kw, s):
    N, H, W, C = x.shape
    _, Ho, Wo, O = dy.shape
    ph, pw = A.same_pad(H, kh, s)[0], A.same_pad(W, kw, s)[0]
    xp = np.pad(x.astype(np.float64), ((0, 0), (ph // 2, ph - ph // 2), (pw // 2, pw - pw // 2), (0, 0)))
    return np.stack([np.einsum("bijc,bijo->co", xp[:, i:i + Ho * s:s, j:j + Wo * s:s][:, :Ho, :Wo], dy.astype(np.float64), optimize=True)
                     for i in range(kh) for j in range(kw)]).reshape(kh, kw, C, O)


@pytest.mark.parametrize("shape", [
    # one slab a slice, as many slices as slabs: 63, 64 and 65 of them, the bound of the sharing between the first two
    (9, 14, 8, 48, 3, 3, 80, 1),
    (8, 16, 8, 48, 3, 3, 80, 1),
    (5, 16, 13, 48, 3, 3, 80, 1),
    # 62 and 64 of them in the paired launch, which has twice the slabs
    (8, 31, 2, 48, 3, 3, 80, 1),
    (8, 16, 4, 48, 3, 3, 80, 1),
    # a tile is one tap, whose pixels outside the image are left out: 81 slices in the middle, 25 in the corners, where some of
    # the eight threads have none
    (16, 9, 9, 128, 9, 9, 32, 1),
])
def test_shared_slices_at_the_bound(A, shape):
    """Tolerance as in test_many_slices."""
    print("shape", shape, flush=True)
    N, H, W, C, kh, kw, O, s = shape
    (ph, Ho), (pw, Wo) = A.same_pad(H, kh, s), A.same_pad(W, kw, s)
    lib, P = A.load(), torch.Tensor.data_ptr
    ins = [rand_conv_inputs(seed, *shape)[::2] for seed in (7, 8)]
    exp = [filter_gradient_float64(A, x, dy, kh, kw, s) for x, dy in ins]
    dev = [(device(x), device(dy)) for x, dy in ins]
    geom = (N, H, W, C, Ho, Wo, O, kh, kw, s, s, ph // 2, pw // 2)
    tol = N * Ho * Wo * 2.0 ** -24
    lib.dh_debug_force_splitk(200)
    try:
        d = room(kh * kw * C * O, 0)
        A.check(lib.dh_conv2d_dk(P(dev[0][0]), P(dev[0][1]), P(d), *geom, None))
        np.testing.assert_allclose(d.cpu().numpy().reshape(kh, kw, C, O), exp[0], rtol=0, atol=tol)
        A.check(lib.dh_conv2d_dk_pair(P(dev[0][0]), P(dev[0][1]), P(dev[1][0]), P(dev[1][1]), P(d), *geom, None))
        np.testing.assert_allclose(d.cpu().numpy().reshape(kh, kw, C, O), exp[0] + exp[1], rtol=0, atol=2 * tol)
    finally:
        lib.dh_debug_force_splitk(0)


@pytest.mark.parametrize("shape", [  # as in test_small_launches, and a launch of position-major rows
    (4, 16, 16, 64, 3, 3, 64, 1),
    (1, 16, 16, 80, 4, 4, 64, 1),
    (16, 4, 4, 64, 5, 5, 128, 2),
])
def test_small_paired_launches(A, shape):
    """Two instances in one launch against the single launches cut into one slice each; bound as in test_small_launches."""
    print("shape", shape, flush=True)
    be = A.HipBackend(0)
    N, H, W, C, kh, kw, O, s = shape
    (ph, Ho), (pw, Wo) = A.same_pad(H, kh, s), A.same_pad(W, kw, s)
    lib, P = A.load(), torch.Tensor.data_ptr
    ins = [rand_conv_inputs(seed, *shape) for seed in (9, 10)]
    k = ins[0][1]
    kd, xd, dyd = device(k), [device(x) for x, _, _ in ins], [device(dy) for _, _, dy in ins]
    y, dx = [torch.empty_like(t) for t in dyd], [torch.empty_like(t) for t in xd]
    fwd = (N, H, W, C, kh, kw, O, s, s, ph // 2, pw // 2, Ho, Wo)
    adj = (N, Ho, Wo, O, kh, kw, C, s, s, ph // 2, pw // 2, H, W)
    A.check(lib.dh_conv2d_fwd_pair(P(xd[0]), P(xd[1]), P(kd), P(y[0]), P(y[1]), *fwd, None, A.ACT_NONE, 0.0, None))
    A.check(lib.dh_conv2d_dx_pair(P(dyd[0]), P(dyd[1]), P(kd), P(dx[0]), P(dx[1]), *adj, None, A.ACT_NONE, 0.0, None))
    for i, (x, _, dy) in enumerate(ins):
        mag = be.conv2d(np.abs(x), np.abs(k), (s, s)), be.conv2d_input_grad(np.abs(dy), np.abs(k), s, (H, W))
        lib.dh_debug_force_splitk(1)
        try:
            whole = be.conv2d(x, k, (s, s)), be.conv2d_input_grad(dy, k, s, (H, W))
        finally:
            lib.dh_debug_force_splitk(0)
        for g, w, m, n in zip((y[i].cpu().numpy(), dx[i].cpu().numpy()), whole, mag, (kh * kw * C, kh * kw * O)):
            assert np.abs(g - w).max() <= 2.0 ** -24 * n * m.max()


@pytest.mark.parametrize("generic", [0, 1])
@pytest.mark.parametrize("splits", [0, 1, 2])
@pytest.mark.parametrize("shape", [(2, 6, 6, 16, 3, 3, 16, 1), (2, 6, 6, 32, 3, 3, 70, 1), (2, 6, 6, 32, 3, 3, 132, 1)])
def test_negative_zeros(A, shape, splits, generic):
    """Sums of products that all underflow from below are -0, and stay that without a bias, with the activations that keep it; in
    which launch they are formed makes no difference."""
    print("shape", shape, "splits", splits, "generic", generic, flush=True)
    be = A.HipBackend(0)
    N, H, W, C, kh, kw, O, s = shape
    x, k = np.full((N, H, W, C), 1e-30, np.float32), np.full((kh, kw, C, O), -1e-30, np.float32)
    be.lib.dh_debug_force_splitk(splits)
    be.lib.dh_debug_force_generic_conv(generic)
    try:
        for act in (A.ACT_NONE, A.ACT_RELU, A.ACT_LEAKY):
            y = be.conv2d(x, k, (s, s), act=act, alpha=0.2)
            inner = y[:, 1:-1, 1:-1]     # no tap in the padding, whose products are 0
            assert (inner == 0).all() and np.signbit(inner).all(), act
    finally:
        be.lib.dh_debug_force_splitk(0)
        be.lib.dh_debug_force_generic_conv(0)


@pytest.mark.parametrize("shape", [(9, 27, 19, 48, 3, 3, 80, 1), (16, 9, 9, 128, 9, 9, 32, 1)])
def test_negative_zeros_of_filter_gradients(A, shape):
    """The same in whole filter gradients (in a split one the slices' own zeros may have either sign)."""
    be = A.HipBackend(0)
    N, H, W, C, kh, kw, O, s = shape
    pads = (A.same_pad(H, kh, s)[0], A.same_pad(W, kw, s)[0])
    be.lib.dh_debug_force_splitk(1)
    try:
        d = be.conv2d_kernel_grad(np.full((N, H, W, O), -1e-30, np.float32), np.full((N, H, W, C), 1e-30, np.float32), s, pads)
    finally:
        be.lib.dh_debug_force_splitk(0)
    assert (d == 0).all() and np.signbit(d).all()
