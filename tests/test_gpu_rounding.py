"""The conversions to bfloat16 that kernels store with, a value at a time and in pairs, against rounding to nearest even by integer steps."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rounded(bits):
    u = bits & 0xFFFFFFFF
    nan = (u & 0x7FFFFFFF) > 0x7F800000
    return torch.where(nan, (u >> 16) | 0x40, (u + 0x7FFF + ((u >> 16) & 1)) >> 16), nan


def test_every_float_rounds_to_the_nearest_even_bfloat16():
    from sharpinference_amd import ops

    n = 1 << 26
    for start in range(-2 ** 31, 2 ** 31, n):
        bits = torch.arange(start, start + n, device=DEV, dtype=torch.int64)
        got = ops.cast(bits.to(torch.int32).view(torch.float32), torch.bfloat16).view(torch.int16).to(torch.int64) & 0xFFFF
        want, nan = _rounded(bits)
        assert bool(torch.where(nan, (got & 0x7FFF) > 0x7F80, got == want).all()), start
        assert bool((got == want).all()), f"a NaN's bits at {start}"


def test_every_float_rounds_so_in_a_pair_too():
    """Rows by eights are stored a pair of values in one conversion: -0 + b is b, and neighbours differ in all their bits."""
    from sharpinference_amd import ops

    n = 1 << 26
    for start in range(0, 2 ** 32, n):
        bits = (torch.arange(start, start + n, device=DEV, dtype=torch.int64) * 0x9E3779B1) & 0xFFFFFFFF        # (odd: every pattern once)
        b = torch.where(bits >= 2 ** 31, bits - 2 ** 32, bits).to(torch.int32).view(torch.float32)
        got = ops.add_bias(torch.full((1, n), -0.0, dtype=torch.bfloat16, device=DEV), b).view(torch.int16).to(torch.int64)[0] & 0xFFFF
        assert bool((got == _rounded(bits)[0]).all()), start
