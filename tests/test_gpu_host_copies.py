"""Host copies through pinned slots: sizes around the smallest that takes them and
around whole chunks, unaligned host memory, pinned host memory, and several threads
with streams of their own at once.  Bytes stay the same."""
import ctypes
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from gtt import operators as ops  # noqa: E402

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.fixture(scope="module")
def lib():
    L = ops.load()
    h2d, d2h, stream = (L._ZN3gtt8copy_h2dEPvPKvm, L._ZN3gtt8copy_d2hEPvPKvm, L._ZN3gtt18set_current_streamEPv)
    for f in (h2d, d2h):
        f.argtypes, f.restype = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t], None
    stream.argtypes, stream.restype = [ctypes.c_void_p], None
    return h2d, d2h, stream


def round_trip(lib, nbytes, seed, shift=0, pinned=False):
    src = np.random.default_rng(seed).integers(0, 256, nbytes + 16, dtype=np.uint8)[shift:shift + nbytes]
    if pinned:
        keep = torch.from_numpy(src.copy()).pin_memory()
        src = keep.numpy()
    dev = torch.zeros(nbytes + 64, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    back = np.full(nbytes + 64, 7, np.uint8)
    lib[0](dev.data_ptr(), src.ctypes.data, nbytes)
    lib[1](back.ctypes.data + shift, dev.data_ptr(), nbytes)
    return (np.array_equal(back[shift:shift + nbytes], src) and (back[:shift] == 7).all()
            and (back[shift + nbytes:] == 7).all() and not dev[nbytes:].any().item())


@pytest.mark.parametrize("nbytes", [1, 4 * MB - 1, 4 * MB, 4 * MB + 1, 8 * MB, 8 * MB + 4097, 16 * MB - 1, 16 * MB,
                                    32 * MB - 3, 32 * MB + 1, 71 * MB + 5])
def test_round_trip(lib, nbytes):
    print("CASE host copy", nbytes, flush=True)
    assert round_trip(lib, nbytes, nbytes)
    assert round_trip(lib, nbytes, nbytes + 1, shift=3)
    assert round_trip(lib, nbytes, nbytes + 2, pinned=True)


def test_threads(lib):
    print("CASE host copies of six threads", flush=True)
    ok = [False] * 6

    def work(i):
        s = torch.cuda.Stream()
        lib[2](s.cuda_stream)
        ok[i] = all(round_trip(lib, (5 + 5 * i) * MB + i, 10 * i + r) for r in range(3))
        lib[2](None)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(ok)
