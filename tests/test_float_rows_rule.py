"""Which plain products of 32-bit rows go to the kernel of many rows (no GPU: the library is asked for a chip of 256 units, and of fewer)."""
import ctypes

import pytest

from sharpinference_amd.ops import lib


def takes(M, N, units=256):
    fn = lib.load().sharpi_gemm_tiled_many_rows
    fn.argtypes, fn.restype = [ctypes.c_int] * 3, ctypes.c_int
    return bool(fn(M, N, units))


# rows, columns, us of the tiled kernel and of the other at K = 2,048
TIMED = [(573, 2048, 68.3, 71.8), (573, 2816, 85.2, 71.6), (573, 3072, 84.8, 71.9), (573, 5120, 117.5, 122.9), (573, 8192, 198.3, 217.1),
         (350, 2816, 54.9, 71.6), (350, 5120, 86.3, 72.2), (350, 8192, 117.5, 123.0), (400, 8192, 194.3, 125.0), (400, 2048, 52.5, 70.9),
         (800, 2048, 84.7, 71.5), (800, 5120, 193.3, 138.5), (1024, 2048, 84.9, 72.5), (1024, 5120, 197.3, 241.9), (1024, 8192, 314.3, 247.3),
         (2048, 2048, 194.7, 128.4), (2048, 3072, 229.8, 243.2), (2048, 4096, 307.8, 247.7), (64, 2048, 35.7, 69.8), (64, 32000, 93.1, 82.1),
         (100, 16384, 93.9, 74.3), (192, 16384, 120.4, 126.3), (7, 8192, 37.1, 32.3), (7, 24576, 49.7, 40.4), (32, 8192, 37.6, 41.8),
         (32, 20000, 55.4, 42.7)]


@pytest.mark.parametrize("M,N,tiled,rows", TIMED)
def test_the_faster_kernel_is_taken(M, N, tiled, rows):
    assert takes(M, N) == (rows < tiled and (M, N) != (7, 8192))          # (under half a block a unit is left where it was)


def test_rounds_are_the_chip_s():
    # 352 blocks beside 704 tiled ones: one round each on 256 units, three and four on 64
    assert not takes(1024, 2816) and takes(1024, 2816, 64)
    assert not takes(0, 2816) and not takes(573, 0) and not takes(573, 2816, 0)
