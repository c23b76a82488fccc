"""CRC-32 at the edges of its kernel's steps (8 KB) and chunks (64 KB), past 256
and 65,536 chunks (the levels of its power table) and past 1,024 (several a
block), against zlib."""
import ctypes
import zlib

import numpy as np
import pytest

from tac_gpu import device, errors, lib

pytestmark = pytest.mark.gpu


def _crc(buf, shift, n):
    out = ctypes.c_uint32(0)
    errors.check(lib.tac_crc32_device(ctypes.c_void_p(buf.ptr.value + shift), n,
                                      ctypes.byref(out), None))
    return out.value


@pytest.mark.parametrize("n", [1, 15, 16, 17, 1023, 8191, 8192, 8193, 65_535, 65_536, 65_537,
                               131_072, 1_023 * 65_536 + 9, 1_025 * 65_536 + 1, 256 * 65_536 - 1, 256 * 65_536, 257 * 65_536 + 3])
def test_crc_chunk_edges(gpu, n):
    data = np.random.default_rng(n).integers(0, 256, n + 16, dtype=np.uint8)
    buf = device.DeviceArray.from_host(data)
    for shift in (0, 1, 8, 15):
        want = zlib.crc32(data[shift:shift + n].tobytes())
        assert _crc(buf, shift, n) == want


def test_crc_past_65536_chunks(gpu):
    piece = np.random.default_rng(9).integers(0, 256, 1 << 26, dtype=np.uint8)
    n = (65_536 + 3) * 65_536 + 77
    buf = device.DeviceArray((n,), np.uint8)
    want = 0
    for at in range(0, n, piece.size):
        part = piece[:min(piece.size, n - at)]
        errors.check(lib.tac_gpu_memcpy_htod(ctypes.c_void_p(buf.ptr.value + at),
                                             ctypes.c_void_p(part.ctypes.data), part.size))
        want = zlib.crc32(part.tobytes(), want)
    assert _crc(buf, 0, n) == want
