"""Which products of many rows go to tiles of one height (no GPU: 256 units are assumed)."""
import pytest

from sharpinference_amd import ops


@pytest.mark.parametrize("M,N,K,gated,height", [
    (3000, 2816, 2048, True, 160), (1664, 2816, 2048, True, 128), (2048, 8192, 2048, False, 256), (908, 10240, 1408, True, 160),
    (2049, 8192, 2048, False, 0),                                      # more than 256 tall tiles
    (1400, 2816, 2048, True, 0), (509, 2048, 2816, True, 0),           # under half a round
    (547, 8192, 2816, True, 0), (1056, 7168, 2816, True, 0), (1331, 7168, 2816, True, 160),        # the rate that is asked for
    (1401, 10240, 3584, True, 0), (1247, 16384, 5120, True, 0), (33, 2816, 2048, True, 0), (0, 2816, 2048, False, 0),
    (3000, 2824, 2048, False, 0), (3000, 2816, 2112, False, 0), (3000, 2832, 2048, True, 0)])      # not stored tile by tile, or halves not in tiles
def test_heights(M, N, K, gated, height):
    assert ops.dense_height(M, N, K, gated) == height
