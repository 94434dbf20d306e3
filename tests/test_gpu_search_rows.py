"""Row offsets of the stand-alone search: its lists together may pass 2^31 and
2^32 entries, which the int64 row_ptr of the call promises to hold."""
import ctypes as C

import numpy as np
import pytest

from spatialpy_amd import _abi

pytestmark = pytest.mark.gpu

SCAN = "_ZN3ssa18exclusive_scan_i64EP12ihipStream_tPKiPlxPv"        # exclusive_scan_i64(stream, in, out, n, tmp)
SCAN_TMP = "_ZN3ssa14scan_tmp_bytesExm"                             # scan_tmp_bytes(n, bytes of a sum)
CSR = "_ZN3ssa9csr_listsEP12ihipStream_tiiPKiPKlS3_PKdPiPd"         # csr_lists(stream, m, W, deg, row, oi, or, ci, cr)


class Device:
    """Device arrays through the HIP runtime of the library."""

    def __init__(self):
        self.lib = _abi.load_library()
        self.held = []

    def __enter__(self):
        return self

    def __exit__(self, *_):
        self.lib.hipDeviceSynchronize()
        for p in self.held:
            self.lib.hipFree(p)

    def empty(self, nbytes):
        p = C.c_void_p()
        assert self.lib.hipMalloc(C.byref(p), C.c_size_t(max(nbytes, 8))) == 0
        self.held.append(p)
        return p

    def array(self, a):
        p = self.empty(a.nbytes)
        assert self.lib.hipMemcpy(p, a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes), 1) == 0
        return p

    def read(self, p, dtype, count, at=0):
        count, at = int(count), int(at)
        out = np.zeros(count, dtype)
        assert self.lib.hipMemcpy(out.ctypes.data_as(C.c_void_p), C.c_void_p(p.value + at * out.itemsize),
                                  C.c_size_t(out.nbytes), 2) == 0
        return out


@pytest.mark.parametrize("n", [1, 2, 5, 1023, 1024, 1025, 1 << 20, (1 << 20) + 1025])
@pytest.mark.parametrize("total", [1 << 31, (1 << 32) + 7, 1 << 40])
def test_offsets_past_32_bits(n, total):
    top = min(2 * total // n + 1, 2 ** 31 - 1)
    lengths = np.random.default_rng(n).integers(0, top, n).astype(np.int32)
    lengths[0] = top
    with Device() as d:
        size = d.lib[SCAN_TMP]
        size.restype, size.argtypes = C.c_size_t, [C.c_longlong, C.c_size_t]
        scan = d.lib[SCAN]
        scan.restype, scan.argtypes = None, [C.c_void_p, C.c_void_p, C.c_void_p, C.c_longlong, C.c_void_p]
        src, dst, tmp = d.array(lengths), d.empty(8 * (n + 1)), d.empty(size(n, 8))
        scan(None, src, dst, n, tmp)
        got = d.read(dst, np.int64, n + 1)
    assert np.array_equal(got, np.concatenate([[0], np.cumsum(lengths, dtype=np.int64)]))


def test_rows_are_written_past_32_bits():
    deg = np.array([2, 1, 0, 3], np.int32)
    row = np.array([0, 2 ** 31 - 1, 2 ** 31, 2 ** 32 + 5], np.int64)
    m, W, total = 4, 3, 2 ** 32 + 8
    oi = np.arange(W * m, dtype=np.int32) + 100
    orr = np.arange(W * m) + 0.5
    with Device() as d:
        csr = d.lib[CSR]
        csr.restype = None
        csr.argtypes = [C.c_void_p, C.c_int, C.c_int] + [C.c_void_p] * 6
        ci, cr = d.empty(4 * total), d.empty(8 * total)
        csr(None, m, W, d.array(deg), d.array(row), d.array(oi), d.array(orr), ci, cr)
        for i in range(m):
            assert np.array_equal(d.read(ci, np.int32, deg[i], row[i]), oi.reshape(W, m)[:deg[i], i])
            assert np.array_equal(d.read(cr, np.float64, deg[i], row[i]), orr.reshape(W, m)[:deg[i], i])
