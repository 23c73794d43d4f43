"""hip_h2d, hip_d2h and hip_d2h_rows: bytes arrive whole at every edge of the
staging (small copies up to 128 KiB, downloads from 2 MiB on in 4 MiB blocks
with 512 KiB to a thread), rows lose their padding, pinned memory is a copy's
own source and destination, and threads that share one context do not mix
their bytes."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.fixture(scope="module")
def dev(trlm):
    return trlm.Device()


def roundtrip(dev, n, seed):
    x = np.random.default_rng(seed).integers(0, 256, n, np.uint8)
    p = dev.upload(x)
    got = dev.download(p, n, np.uint8)
    dev.free(p)
    return np.array_equal(x, got)


@pytest.mark.parametrize("n", [0, 1, 3, 4096, MB // 8 - 1, MB // 8, MB // 8 + 1, 2 * MB - 1, 2 * MB, 2 * MB + 1, MB // 2 + 65, 4 * MB - 1, 4 * MB,
                               4 * MB + 1, 8 * MB, 8 * MB + 7, 12 * MB + 3])
def test_round_trip(dev, n):
    dev.current()
    assert roundtrip(dev, n, n)


@pytest.mark.parametrize("row_bytes,pitch,rows", [
    (4, 16, 5),                          # short rows
    (31769 * 4, 31772 * 4, 1),           # one row
    (31769 * 4, 31772 * 4, 33),          # exactly the rows of one block
    (31769 * 4, 31772 * 4, 34),          # one row over
    (31769 * 4, 31772 * 4, 101),         # several blocks and a remainder
    (1000, 1000, 9000),                  # no padding
    (4 * MB - 16, 4 * MB, 3),            # one row to a block
    (4 * MB + 5, 4 * MB + 16, 2),        # rows longer than a block
    (4, 16, 0), (0, 16, 3),
])
def test_rows(dev, row_bytes, pitch, rows):
    dev.current()
    fn = dev.hip.hip_d2h_rows
    fn.argtypes, fn.restype = [C.c_void_p, C.c_void_p, C.c_uint64, C.c_uint64, C.c_uint64], None
    n = max(rows - 1, 0) * pitch + row_bytes     # the last row ends the allocation: nothing beyond it is read
    x = np.random.default_rng(rows).integers(0, 256, n, np.uint8)
    p = dev.upload(x)
    got = np.full(rows * row_bytes + 64, 7, np.uint8)
    fn(got.ctypes.data, p, pitch, row_bytes, rows)
    dev.free(p)
    want = [x[r * pitch:r * pitch + row_bytes] for r in range(rows)]
    assert np.array_equal(got[:rows * row_bytes], np.concatenate(want) if want else got[:0])
    assert (got[rows * row_bytes:] == 7).all()


@pytest.mark.parametrize("row_bytes,pitch,rows", [(4096, 4096, 1), (4, 16, 5), (31769 * 4, 31772 * 4, 34),
                                                  (4 * MB + 5, 4 * MB + 16, 2)])
def test_pinned_memory(dev, row_bytes, pitch, rows):
    dev.current()
    with open("/proc/self/maps") as fh:     # the HIP runtime that libtrlm_hip.so loaded
        hip = C.CDLL(sorted({line.split()[-1] for line in fh if "libamdhip64.so" in line})[0])
    fn = dev.hip.hip_d2h_rows
    fn.argtypes, fn.restype = [C.c_void_p, C.c_void_p, C.c_uint64, C.c_uint64, C.c_uint64], None
    n = (rows - 1) * pitch + row_bytes
    mem = [C.c_void_p() for _ in range(2)]
    for m in mem:
        assert hip.hipHostMalloc(C.byref(m), C.c_size_t(n + 64), C.c_uint(0)) == 0
    a, b = [np.ctypeslib.as_array(C.cast(m, C.POINTER(C.c_uint8)), (n + 64,)) for m in mem]
    a[:n] = np.random.default_rng(rows).integers(0, 256, n, np.uint8)
    p = dev.empty(n)
    dev.hip.hip_h2d(p, a.ctypes.data, n)
    b[:] = 7
    dev.hip.hip_d2h(b.ctypes.data, p, n)
    assert np.array_equal(a[:n], b[:n]) and (b[n:] == 7).all()
    b[:] = 7
    fn(b.ctypes.data, p, pitch, row_bytes, rows)
    dev.free(p)
    assert np.array_equal(b[:rows * row_bytes], np.concatenate([a[r * pitch:r * pitch + row_bytes] for r in range(rows)]))
    assert (b[rows * row_bytes:] == 7).all()
    for m in mem:
        assert hip.hipHostFree(m) == 0


def test_threads_share_a_context(dev):
    ok = []

    def work(k):
        dev.current()
        ok.append(all(roundtrip(dev, n, 10 * k + n) for n in (100, 70001, 3 * MB, 9 * MB + 1)))

    th = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert ok == [True] * 4
