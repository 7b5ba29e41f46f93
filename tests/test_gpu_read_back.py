"""Large copies to the host, which go through a ring of pinned chunks: every byte arrives, behind the work already queued, for
lengths around the chunk and ring sizes, and from several threads at once."""
import ctypes as C
import threading

import numpy as np
import pytest
import torch   # before the library: whichever comes first brings the HIP runtime that both use

pytestmark = pytest.mark.gpu

CHUNK, RING = 256 << 10, 4 << 20


@pytest.fixture(scope="module")
def A():
    import __graft_entry__ as ge
    A = ge.load_package().hipabi
    A.check(A.load().dh_init(0))
    return A


def read(A, src, nbytes):
    out = np.full(nbytes + 8, 0xa5, np.uint8)
    A.check(A.load().dh_memcpy_d2h(C.c_void_p(out.ctypes.data + 4), C.c_void_p(src), C.c_size_t(nbytes)))
    assert (out[:4] == 0xa5).all() and (out[-4:] == 0xa5).all()
    return out[4:-4]


@pytest.mark.parametrize("nbytes", [2 * CHUNK - 4, 2 * CHUNK, 2 * CHUNK + 4, 2 * CHUNK + 2, 1 << 20,
                                    8 * CHUNK - 4, 8 * CHUNK, 8 * CHUNK + 4, 8 * CHUNK + 2, 9 * CHUNK, RING - 4, RING, RING + 4,
                                    RING + CHUNK + 16, 3 * RING + 12, 13 << 20])
@pytest.mark.parametrize("offset", [0, 4, 16])
def test_lengths(A, nbytes, offset):
    print("bytes", nbytes, "offset", offset, flush=True)
    a = torch.randint(0, 256, (nbytes + 64,), dtype=torch.uint8, device="cuda")
    exp = a.cpu().numpy()
    for _ in range(2):
        np.testing.assert_array_equal(read(A, a.data_ptr() + offset, nbytes), exp[offset:offset + nbytes])


@pytest.mark.parametrize("nbytes", [(3 << 20) - 4, 3 << 20, (3 << 20) + 4, (6 << 20) + CHUNK, (8 << 20) - 4, 8 << 20, (8 << 20) + 4,
                                    (9 << 20) + 3 * CHUNK + 8, 17 << 20, (24 << 20) + 2 * CHUNK - 4])
def test_lengths_around_the_pieces_of_an_event(A, nbytes):
    """Two or four pieces to an event, slots that are filled again, a last chunk of fewer pieces."""
    print("bytes", nbytes, flush=True)
    a = torch.randint(0, 256, (nbytes,), dtype=torch.uint8, device="cuda")
    np.testing.assert_array_equal(read(A, a.data_ptr(), nbytes), a.cpu().numpy())


def test_behind_queued_work(A):
    a = torch.zeros(3 << 20, device="cuda")
    for i in range(5):
        b = a
        for _ in range(20):
            b = b + 1
        a = b
        got = read(A, a.data_ptr(), a.numel() * 4).view(np.float32)
        assert (got == 20 * (i + 1)).all()


def test_threads(A):
    srcs = [torch.full((700000 + 1000 * i,), float(i + 1), device="cuda") for i in range(4)]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        for _ in range(6):
            if not (read(A, srcs[i].data_ptr(), srcs[i].numel() * 4).view(np.float32) == i + 1).all():
                bad.append(i)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.parametrize("nbytes", [64 << 10, 5 << 20])
def test_into_pinned_memory(A, nbytes):
    """The runtime's way, whatever the size."""
    src = torch.arange(nbytes // 4, device="cuda", dtype=torch.float32)
    out = torch.empty(nbytes // 4, pin_memory=True)
    A.check(A.load().dh_memcpy_d2h(C.c_void_p(out.data_ptr()), C.c_void_p(src.data_ptr()), C.c_size_t(nbytes)))
    assert torch.equal(out, torch.arange(nbytes // 4, dtype=torch.float32))


@pytest.mark.parametrize("nbytes", [64 << 10, 5 << 20])
def test_refused_while_a_stream_is_captured(A, nbytes):
    """As the blocking copy is, whatever the size and whether the ring is there already."""
    lib, st, graph = A.load(), C.c_void_p(), C.c_void_p()
    src = torch.full((nbytes // 4,), 3.0, device="cuda")
    out = np.zeros(nbytes // 4, np.float32)
    assert lib.hipStreamCreateWithFlags(C.byref(st), 1) == 0    # kept: a stream whose capture was ended by an error cannot be waited for
    for _ in range(2):
        torch.cuda.synchronize()
        assert lib.hipStreamBeginCapture(st, 0) == 0
        rc = lib.dh_memcpy_d2h(C.c_void_p(out.ctypes.data), C.c_void_p(src.data_ptr()), C.c_size_t(nbytes))
        lib.hipStreamEndCapture(st, C.byref(graph))             # an error too
        lib.hipGetLastError()
        assert rc != 0 and (out == 0).all()
        assert (read(A, src.data_ptr(), nbytes).view(np.float32) == 3.0).all()
