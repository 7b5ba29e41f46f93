"""Which way a large copy to the host goes, on a HIP runtime of two devices in host memory (tests/fake_hip.cc): through the ring of
pinned chunks only where source, thread and library are on one device, else by the runtime's copy, which finds the device of the
memory by itself.  Without a GPU; each case is a process of its own, since the library keeps its device."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "dcgan-cuda_amd", "lib", "libdcgan_hip.so")

PRELUDE = """
import ctypes as C, sys, threading
import numpy as np
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
lib = C.CDLL(sys.argv[2])
DEVICE, PINNED, MANAGED, MB = 0, 1, 2, 1 << 20
kept = []
def memory(nbytes, kind=DEVICE, device=0):
    raw = np.zeros(nbytes + 4096, np.uint8)
    kept.append(raw)                 # the fake runtime goes on knowing its address
    a = raw[-raw.ctypes.data % 4096:][:nbytes]
    a[:] = np.random.default_rng(nbytes).integers(0, 256, nbytes)
    if kind is not None:
        fake.fake_declare(C.c_void_p(a.ctypes.data), C.c_size_t(nbytes), kind, device)
    return a
def read(src, out=None, nbytes=None, rc=0, fail_at=-1, no_pinned=0):
    out = np.zeros(src.size, np.uint8) if out is None else out
    fake.fake_reset(fail_at, no_pinned)
    got = lib.dh_memcpy_d2h(C.c_void_p(out.ctypes.data), C.c_void_p(src.ctypes.data), C.c_size_t(nbytes or src.size))
    assert (got == 0) == (rc == 0), (got, rc)
    if got == 0:
        assert (out[:nbytes or src.size] == np.ctypeslib.as_array(C.cast(src.ctypes.data, C.POINTER(C.c_uint8)), (nbytes or src.size,))).all()
    route = {(True, False): "ring", (False, True): "runtime"}.get((fake.fake_launches() > 0, fake.fake_copies() > 0), "both or none")
    return route
def in_thread(fn):
    got = []
    t = threading.Thread(target=lambda: got.append(fn()))
    t.start(); t.join()
    return got[0]
def expect(got, want):
    assert got == want, (got, want)
"""

CASES = {
    "one device": """
lib.dh_init(0)
for mb in (4, 13, 4, 9):
    expect(read(memory(mb * MB + 12)), "ring")
for nbytes in (1024, 512 << 10, MB, 2 * MB - 4):
    expect(read(memory(nbytes)), "runtime")       # what gains nothing by the ring
expect(read(memory(2 * MB)), "ring")
""",
    "library on the second device": """
lib.dh_init(1)
expect(read(memory(5 * MB, device=1)), "ring")
expect(read(memory(5 * MB, device=0)), "runtime")
""",
    "memory of the other device": """
lib.dh_init(0)
expect(read(memory(5 * MB, device=1)), "runtime")
expect(read(memory(5 * MB, device=0)), "ring")
expect(read(memory(5 * MB, device=1)), "runtime")
""",
    "thread on another device than the library": """
lib.dh_init(1)
a = memory(5 * MB, device=1)
expect(in_thread(lambda: read(a)), "runtime")      # a thread's current device is the first until it says otherwise
expect(read(a), "ring")
fake.hipSetDevice(0)
expect(read(a), "runtime")
expect(read(memory(5 * MB, device=0)), "runtime")
fake.hipSetDevice(1)
expect(read(a), "ring")
""",
    "both devices in turn": """
for i in range(3):
    for d in (0, 1):
        lib.dh_init(d)
        expect(read(memory(5 * MB + 4 * i, device=d)), "ring")
""",
    "host memory that the device knows": """
lib.dh_init(0)
expect(read(memory(5 * MB), out=memory(5 * MB, PINNED)), "runtime")
expect(read(memory(5 * MB, MANAGED)), "runtime")
expect(read(memory(5 * MB, PINNED)), "runtime")
""",
    "not one allocation": """
lib.dh_init(0)
both = memory(8 * MB, None)
fake.fake_declare(C.c_void_p(both.ctypes.data), C.c_size_t(4 * MB), DEVICE, 0)
fake.fake_declare(C.c_void_p(both.ctypes.data + 4 * MB), C.c_size_t(4 * MB), DEVICE, 0)
expect(read(both), "runtime")
expect(read(both[:4 * MB]), "ring")
expect(read(both[4 * MB:]), "ring")
expect(read(memory(5 * MB, None)), "runtime")      # whatever it is, the runtime decides
""",
    "refused pointers": """
lib.dh_init(0)
fake.fake_reset(-1, 0)
a = memory(5 * MB)
assert lib.dh_memcpy_d2h(None, C.c_void_p(a.ctypes.data), C.c_size_t(a.size)) != 0
assert lib.dh_memcpy_d2h(C.c_void_p(a.ctypes.data), None, C.c_size_t(a.size)) != 0
assert fake.fake_launches() == 0 and fake.fake_copies() == 2
""",
    "a stream is captured": """
lib.dh_init(0)
a, small = memory(5 * MB), memory(4096)
for i in range(2):
    fake.fake_capture(1)
    read(small, rc=1)
    expect(read(a, rc=1), "both or none")
    fake.fake_capture(0)
    expect(read(a), "ring")
    expect(read(small), "runtime")
""",
    "errors on the way": """
lib.dh_init(0)
a = memory(9 * MB)
expect(read(a, no_pinned=1), "runtime")            # no ring to be had
for at in (0, 1, 15, 16, 20, 35):
    read(a, rc=1, fail_at=at)                      # the helpers end, the call says so
expect(read(a), "ring")
""",
}


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    headers = "/opt/rocm/include"
    if not os.path.exists(os.path.join(headers, "hip", "hip_runtime_api.h")):
        pytest.skip("no HIP headers")
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + headers, "-fPIC", "-shared", "-o", so,
                    os.path.join(ROOT, "tests", "fake_hip.cc")], check=True)
    return so


@pytest.mark.parametrize("case", sorted(CASES))
def test_route(fake, case):
    if not os.path.exists(LIB):
        import __graft_entry__ as ge
        ge.build()
    res = subprocess.run([sys.executable, "-c", PRELUDE + CASES[case], fake, LIB], capture_output=True, text=True, timeout=120)
    assert res.returncode == 0, res.stdout + res.stderr
