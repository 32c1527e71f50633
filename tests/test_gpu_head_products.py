"""Products per head on the matrix cores: both tile sizes, the steps requested ahead and what is left behind them."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("T, H, N, K", [(513, 8, 128, 512), (530, 2, 1028, 128), (1025, 9, 20, 648), (1600, 6, 44, 1192), (4200, 3, 4, 72), (200, 64, 128, 512)])
def test_both_tile_sizes_give_the_same_sums(T, H, N, K, gated):
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(T)
    x, w = torch.randn(T, H * K, generator=g).bfloat16(), torch.randn(H, N, K, generator=g).bfloat16()
    gate = torch.randn(T, 3 + H * N, generator=g).bfloat16() if gated else None

    def run(a, b):
        out = torch.zeros(b - a, H * N, dtype=torch.bfloat16, device=DEV)
        return ops.head_gemm(x[a:b].contiguous().to(DEV), 0, K, w.to(DEV), out, 0, N, **(dict(gate=gate[a:b].contiguous().to(DEV), gate_off=3) if gated else {})).cpu()

    whole = run(0, T)                                       # above 64 tiles of 64 x 64
    for a, b in [(0, 1), (1, 18), (T - 33, T)]:             # below, or of few tokens (64 heads, 33 tokens: above)
        assert torch.equal(whole[a:b], run(a, b))
    xs, ws = x.double().view(T, H, K).transpose(0, 1), w.double()
    scale = torch.sigmoid(gate.double()[:, 3:].reshape(T, H, N)) if gated else 1.0
    want = (xs @ ws.transpose(1, 2).contiguous()).transpose(0, 1) * scale
    room = (xs.abs() @ ws.abs().transpose(1, 2).contiguous()).transpose(0, 1) * scale
    # one rounding of the result to 8 bits, K of its sum to 24 (and what the gate's exponential leaves, below 2^-20)
    bound = want.abs() * (2.0 ** -8 + 2.0 ** -20) + room * K * 2.0 ** -24 + 1e-30
    assert bool(((whole.double().view(T, H, N) - want).abs() <= bound).all())
