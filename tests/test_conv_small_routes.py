"""A small launch that the tiled kernels do faster by cutting it into slices, where there is no memory for slices: on a ninth stream, and on a stream being captured whose
arena would have to grow.  It takes the kernel without slices.  On a HIP runtime without a device (tests/fake_launches.cc); each case is a process of its own."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "dcgan-cuda_amd", "lib", "libdcgan_hip.so")

PRELUDE = """
import ctypes as C, sys
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
lib = C.CDLL(sys.argv[2])
fake.fake_launched.restype = C.c_char_p
p = [C.c_void_p((i + 1) << 40) for i in range(3)]
# N, H, W, C, O, k: stride 1, a split launch of the tiled kernels
SMALL = {"fwd": (44, 25, 25, 92, 16, 3), "dx": (1, 7, 6, 10, 150, 5), "dk": (46, 7, 7, 113, 43, 5)}
LARGE = (64, 8, 8, 256, 512, 5)
def call(what, shape, stream):
    N, H, W, ci, co, k = shape
    pad = (k - 1) // 2
    st = C.c_void_p(stream)
    if what == "fwd":
        rc = lib.dh_conv2d_fwd(*p, N, H, W, ci, k, k, co, 1, 1, pad, pad, H, W, None, 0, C.c_float(0), st)
    elif what == "dx":
        rc = lib.dh_conv2d_dx(*p, N, H, W, co, k, k, ci, 1, 1, pad, pad, H, W, None, 0, C.c_float(0), st)
    else:
        rc = lib.dh_conv2d_dk(*p, N, H, W, ci, H, W, co, k, k, 1, 1, pad, pad, st)
    return rc, fake.fake_launched().decode().split()
def tiled(got):
    rc, names = got
    assert rc == 0 and len(names) == 2 and "conv_igemm" in names[0] and "splitk_reduce" in names[1], got
def tiny(got):
    rc, names = got
    assert rc == 0 and len(names) == 1 and "conv_tiny" in names[0], got
assert lib.dh_init(0) == 0
"""

CASES = {
    "a ninth stream": """
for stream in range(1, 9):
    for what in SMALL:
        tiled(call(what, SMALL[what], stream))
for what in SMALL:
    tiny(call(what, SMALL[what], 9))
    tiled(call(what, SMALL[what], 3))
rc, names = call("fwd", LARGE, 9)
assert rc != 0 and not names        # as ever
""",
    "under capture": """
fake.fake_capture(1)
before = fake.fake_allocations()
for what in SMALL:
    tiny(call(what, SMALL[what], 1))
assert fake.fake_allocations() == before
fake.fake_capture(0)
tiled(call("dk", SMALL["dk"], 1))
assert lib.dh_workspace_reserve(C.c_size_t(256 << 20)) == 0     # (the default stream's)
fake.fake_capture(1)
for what in SMALL:
    tiled(call(what, SMALL[what], 0))
    tiny(call(what, SMALL[what], 2))
""",
}


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    headers = "/opt/rocm/include"
    if not os.path.exists(os.path.join(headers, "hip", "hip_runtime_api.h")):
        pytest.skip("no HIP headers")
    so = str(tmp_path_factory.mktemp("fake") / "libfake_launches.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + headers, "-fPIC", "-shared", "-o", so,
                    os.path.join(ROOT, "tests", "fake_launches.cc")], check=True)
    return so


@pytest.mark.parametrize("case", sorted(CASES))
def test_route(fake, case):
    if not os.path.exists(LIB):
        import __graft_entry__ as ge
        ge.build()
    res = subprocess.run([sys.executable, "-c", PRELUDE + CASES[case], fake, LIB], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout + res.stderr
