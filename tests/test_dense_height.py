"""Which products of many rows go to tiles of one height (no GPU: 256 units are assumed)."""
import pytest
import torch

from sharpinference_amd import ops


@pytest.mark.parametrize("M,N,K,gated,height", [
    (3000, 2816, 2048, True, 160), (1664, 2816, 2048, True, 128), (2048, 8192, 2048, False, 256), (908, 10240, 1408, True, 160),
    (2049, 8192, 2048, False, 0),                                      # more than 256 tall tiles
    (1400, 2816, 2048, True, 0), (509, 2048, 2816, True, 0),           # under half a round
    (547, 8192, 2816, True, 0), (1056, 7168, 2816, True, 0), (1331, 7168, 2816, True, 160),        # the rate that is asked for
    (1401, 10240, 3584, True, 0), (1247, 16384, 5120, True, 0), (33, 2816, 2048, True, 0), (0, 2816, 2048, False, 0),
    (3000, 2824, 2048, False, 0), (3000, 2816, 2112, False, 0), (3000, 2832, 2048, True, 0),      # not stored tile by tile, or halves not in tiles
    # few rows of many columns, which the weight-streaming kernel or the library has; what lies outside of the sizes that were timed
    (1, 32768, 2048, True, 0), (8, 40960, 1408, True, 0), (32, 32768, 2048, True, 0), (33, 65536, 2048, False, 0), (299, 28672, 2048, True, 0),
    (300, 28672, 2048, True, 160), (300, 32768, 2048, True, 0), (8192, 2048, 2048, True, 256), (8192, 1920, 2048, True, 0),
    (1500, 2816, 1408, True, 128), (1500, 2816, 1280, True, 0), (1500, 2816, 128, False, 0)])
def test_heights(M, N, K, gated, height):
    assert ops.dense_height(M, N, K, gated) == height


def test_a_height_is_of_the_device_that_asks(monkeypatch):
    assert ops.dense_height(3000, 2816, 2048, True) == 160
    monkeypatch.setattr(ops, "compute_units", lambda device=None: 64)
    assert ops.dense_height(3000, 2816, 2048, True) == 0             # more than a tall tile a unit
    monkeypatch.undo()
    assert ops.dense_height(3000, 2816, 2048, True) == 160


def test_few_rows_ask_nothing_further(monkeypatch):
    """Short steps wait for the host: neither the device nor the matrix is looked at for them."""
    monkeypatch.setattr(ops, "compute_units", lambda device=None: 1 / 0)
    assert ops.dense_height(8, 16384, 2048, True) == 0
    assert ops._dense_height_of(torch.zeros(8, 2048, dtype=torch.bfloat16), None, torch.bfloat16, True) == 0
