"""The conversion to bfloat16 that every kernel stores with: each of the 2^32 floats against rounding to nearest even by integer steps."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def test_every_float_rounds_to_the_nearest_even_bfloat16():
    from sharpinference_amd import ops

    n = 1 << 26
    for start in range(-2 ** 31, 2 ** 31, n):
        bits = torch.arange(start, start + n, device=DEV, dtype=torch.int64)
        got = ops.cast(bits.to(torch.int32).view(torch.float32), torch.bfloat16).view(torch.int16).to(torch.int64) & 0xFFFF
        u = bits & 0xFFFFFFFF
        want = (u + 0x7FFF + ((u >> 16) & 1)) >> 16
        nan = (u & 0x7FFFFFFF) > 0x7F800000
        assert bool(torch.where(nan, (got & 0x7FFF) > 0x7F80, got == want).all()), start
        assert bool((got == torch.where(nan, (u >> 16) | 0x40, want)).all()), f"a NaN's bits at {start}"
