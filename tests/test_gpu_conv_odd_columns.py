"""Results whose columns are no multiple of 4: the write-out of launches that are large enough turns 32 x 32 tiles in LDS.  Around the widths where that begins, the tiles' edges
and remainders, direct and from slices, with and without a result that starts at 16 bytes; nothing outside the result is written."""
import numpy as np
import pytest
import torch

from common import ATOL, RTOL, rand_conv_inputs, same_pad

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def A():
    import __graft_entry__ as ge
    A = ge.load_package().hipabi
    A.check(A.load().dh_init(0))
    return A


def guarded(shape, first):
    """(whole buffer, pointer to its part that is the result): 64 words around it, which starts `first` words past 256 bytes."""
    n = int(np.prod(shape))
    whole = torch.full((n + 128,), 7.5, device="cuda")
    return whole, whole.data_ptr() + 4 * (64 + first)


def result(whole, shape, first):
    torch.cuda.synchronize()
    n, got = int(np.prod(shape)), whole.cpu().numpy()
    assert (got[:64 + first] == 7.5).all() and (got[64 + first + n:] == 7.5).all()
    return got[64 + first:64 + first + n].reshape(shape)


def workgroups(rows, columns, slices):
    bm, bn = (128, 32) if columns <= 32 else (64 if rows <= 64 else 128, 64 if columns <= 64 or rows <= 64 else 128)
    return -(-rows // bm) * -(-columns // bn) * slices


def turned(rows, columns, slices):
    """The rule of the launch, on a device with 256 units."""
    return workgroups(rows, columns, slices) * (2 if slices > 1 else 4) >= 256


@pytest.mark.parametrize("many", [False, True])      # rows enough that they are turned
@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("shape", [      # N, H, W, C, kh, kw, O, stride
    (3, 9, 11, 16, 3, 3, 17, 1),         # the narrowest that is turned
    (2, 10, 9, 18, 3, 3, 15, 1),         # columns one way are, the other way not
    (3, 13, 7, 23, 3, 2, 31, 1),         # one tile, almost full
    (2, 11, 12, 33, 3, 3, 34, 2),        # two columns in the second tile of 32
    (3, 10, 10, 49, 2, 2, 50, 1),        # 18 in the second
    (2, 17, 9, 65, 3, 3, 63, 1),
    (5, 12, 13, 81, 3, 3, 98, 2),        # tiles of 128
    (2, 15, 16, 127, 1, 1, 129, 1),      # and one column past one
    (9, 30, 31, 37, 3, 3, 101, 1),       # many rows, the last tile a part
    (4, 16, 16, 24, 3, 3, 40, 1),        # multiples of 4 at any address
])
@pytest.mark.parametrize("first", [0, 1])
def test_write_out(A, orc, shape, splits, first, many):
    N, H, W, C, kh, kw, O, s = shape
    if many:
        N = -(-64 * 128 // (-(-H // s) * -(-W // s)))
        shape = (N,) + shape[1:]
    print("shape", shape, "splits", splits, "first", first, flush=True)
    dk_splits = 160 if many and splits > 1 else splits
    (ph, Ho), (pw, Wo) = A.same_pad(H, kh, s), A.same_pad(W, kw, s)
    x, k, dy = rand_conv_inputs(71, *shape)
    bias, bias_c = np.linspace(-0.5, 0.5, O).astype(np.float32), np.linspace(-0.3, 0.3, C).astype(np.float32)
    orc.set_threads(8)
    exp = (orc.relu_leaky(orc.bias_add(orc.conv2d(x, k, (s, s)), bias), 0.2),
           orc.tanh(orc.bias_add(orc.conv2d_input_grad(dy, k, s, (H, W)), bias_c)),
           orc.conv2d_kernel_grad(dy, x, s, (same_pad(H, kh, s)[0], same_pad(W, kw, s)[0])))
    dx, dk, ddy, db, dbc = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x, k, dy, bias, bias_c))
    lib, p = A.load(), torch.Tensor.data_ptr
    fwd = (N, H, W, C, kh, kw, O, s, s, ph // 2, pw // 2, Ho, Wo)
    adj = (N, Ho, Wo, O, kh, kw, C, s, s, ph // 2, pw // 2, H, W)
    fil = (N, H, W, C, Ho, Wo, O, kh, kw, s, s, ph // 2, pw // 2)
    (wy, y), (wx, gx), (wk, gk) = (guarded(e.shape, first) for e in exp)
    if many and A.device_info()["compute_units"] == 256:
        slices = min(splits, -(-kh * kw * C // 16))
        assert turned(N * Ho * Wo, O, slices) and (s > 1 or turned(N * H * W, C, min(splits, -(-kh * kw * O // 16))))
        assert splits == 1 or turned(kh * kw * C, O, dk_splits)
    lib.dh_debug_force_splitk(splits)
    try:
        A.check(lib.dh_conv2d_fwd(p(dx), p(dk), y, *fwd, p(db), A.ACT_LEAKY, 0.2, None))
        A.check(lib.dh_conv2d_dx(p(ddy), p(dk), gx, *adj, p(dbc), A.ACT_TANH, 0.0, None))
        lib.dh_debug_force_splitk(dk_splits)
        A.check(lib.dh_conv2d_dk(p(dx), p(ddy), gk, *fil, None))
    finally:
        lib.dh_debug_force_splitk(0)
    for what, whole, e in zip(("fwd", "dx", "dk"), (wy, wx, wk), exp):
        # sums of N*Ho*Wo products of U(-1,1) values: the filter gradient's absolute tolerance follows their magnitude
        scale = max(1.0, float(np.abs(e).max())) if what == "dk" else 1.0
        np.testing.assert_allclose(result(whole, e.shape, first), e, rtol=RTOL, atol=ATOL * scale, err_msg=what)


@pytest.mark.parametrize("first", [0, 1])
def test_whole_filter_gradient(A, orc, first):
    """Turned in one slice: 22 x 3 tiles, both ends a part."""
    N, H, W, C, kh, kw, O, s = shape = (2, 4, 5, 309, 3, 3, 303, 1)
    assert turned(kh * kw * C, O, 1)
    x, k, dy = rand_conv_inputs(73, *shape)
    orc.set_threads(8)
    want = orc.conv2d_kernel_grad(dy, x, s, (same_pad(H, kh, s)[0], same_pad(W, kw, s)[0]))
    xd, yd = (torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (x, dy))
    whole, gk = guarded(k.shape, first)
    lib = A.load()
    lib.dh_debug_force_splitk(1)
    try:
        A.check(lib.dh_conv2d_dk(xd.data_ptr(), yd.data_ptr(), gk, N, H, W, C, H, W, O, kh, kw, s, s, 1, 1, None))
    finally:
        lib.dh_debug_force_splitk(0)
    np.testing.assert_allclose(result(whole, k.shape, first), want, rtol=RTOL, atol=ATOL * max(1.0, float(np.abs(want).max())))


@pytest.mark.parametrize("shape", [      # N, H, W, C, kh, kw, O, stride
    (40, 60, 61, 90, 1, 1, 1, 1),        # one column: chunks of four rows
    (3, 21, 20, 91, 1, 1, 33, 1),        # the last chunk one element past the end
    (3, 21, 20, 93, 3, 3, 66, 2),        # two
    (3, 20, 21, 97, 2, 2, 103, 1),       # three
    (1, 1, 1, 120, 1, 1, 3, 1),          # filter gradient over three elements
    (1, 1, 2, 120, 1, 1, 1, 1),          # and over two
    (1, 1, 1, 120, 1, 1, 5, 1),          # five
])
@pytest.mark.parametrize("first", [0, 1, 3])
def test_rows_read_16_bytes_at_a_time(A, orc, shape, first):
    """Filter and gradient that end and begin beside NaNs, at any address: nothing outside them gets into a result."""
    print("shape", shape, "first", first, flush=True)
    N, H, W, C, kh, kw, O, s = shape
    (ph, Ho), (pw, Wo) = A.same_pad(H, kh, s), A.same_pad(W, kw, s)
    x, k, dy = rand_conv_inputs(72, *shape)
    orc.set_threads(8)
    exp = orc.conv2d(x, k, (s, s)), orc.conv2d_kernel_grad(dy, x, s, (same_pad(H, kh, s)[0], same_pad(W, kw, s)[0]))

    def among_nans(a):
        whole = torch.full((a.size + 128,), float("nan"), device="cuda")
        whole[64 + first:64 + first + a.size] = torch.from_numpy(np.ascontiguousarray(a).reshape(-1)).cuda()
        return whole, whole.data_ptr() + 4 * (64 + first)

    dx = torch.from_numpy(np.ascontiguousarray(x)).cuda()
    (wf, f), (wd, d) = among_nans(k), among_nans(dy)
    (wy, y), (wk, gk) = (guarded(e.shape, 0) for e in exp)
    lib = A.load()
    lib.dh_debug_force_splitk(1)
    lib.dh_debug_force_generic_conv(1)
    try:
        A.check(lib.dh_conv2d_fwd(dx.data_ptr(), f, y, N, H, W, C, kh, kw, O, s, s, ph // 2, pw // 2, Ho, Wo, None, A.ACT_NONE, 0.0, None))
        A.check(lib.dh_conv2d_dk(dx.data_ptr(), d, gk, N, H, W, C, Ho, Wo, O, kh, kw, s, s, ph // 2, pw // 2, None))
    finally:
        lib.dh_debug_force_generic_conv(0)
        lib.dh_debug_force_splitk(0)
    for what, whole, e in zip(("fwd", "dk"), (wy, wk), exp):
        scale = max(1.0, float(np.abs(e).max())) if what == "dk" else 1.0
        np.testing.assert_allclose(result(whole, e.shape, 0), e, rtol=RTOL, atol=ATOL * scale, err_msg=what)
