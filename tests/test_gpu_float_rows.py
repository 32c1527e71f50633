"""The grouped 32-bit product of many rows sums as the tiled product does, bit for bit: every height of its tiles, one and several
tiles a group, the shortest sums, columns that end inside a block, gathered rows and rows of their own."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("counts", [[1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 80, 128, 129], [0, 700, 0, 3, 64, 0, 27, 200]])
@pytest.mark.parametrize("N,K", [(4100, 32), (3077, 64), (3200, 96), (2999, 352)])
def test_rows_are_the_tiled_products(counts, N, K):
    from sharpinference_amd import ops
    g = torch.Generator(device=DEV).manual_seed(N + K)
    E, M = len(counts), sum(counts)
    assert M > 24 * E and (M // 64 + E) * -(-N // 128) >= 384          # (what the kernel is chosen for)
    ids = torch.cat([torch.full((c,), e, dtype=torch.int32) for e, c in enumerate(counts)])
    ids = ids[torch.randperm(M, generator=torch.Generator().manual_seed(M))].view(-1, 1).to(DEV)
    rt = ops.moe_permute(ids, torch.ones(ids.shape, device=DEV), E)
    x = torch.randn(M, K, device=DEV, generator=g)
    w = torch.randn(E, N, K, device=DEV, generator=g)
    x[0, 0], w[E - 1, N - 1, K - 1] = float("inf"), float("nan")       # stay with their row and their column
    got = ops.grouped_gemm(x, w, rt.offsets, rt.sorted_token, M)
    own = ops.grouped_gemm(x[rt.sorted_token.long()].contiguous(), w, rt.offsets, None, M)
    off = rt.offsets.tolist()
    for e in range(E):
        rows = rt.sorted_token[off[e]:off[e + 1]].long()
        if len(rows):
            want = ops.gemm_tiled(x[rows].contiguous(), w[e].contiguous())
            for y in (got, own):
                assert torch.equal(y[off[e]:off[e + 1]].nan_to_num(1.5), want.nan_to_num(1.5)), e


@pytest.mark.parametrize("M,N,K", [(573, 2817, 64), (1, 16385, 32), (32, 16400, 96), (65, 16001, 32), (448, 7300, 64), (130, 32000, 32), (450, 16390, 32)])
def test_plain_rows_are_the_tiled_products(M, N, K):
    """Sizes that go to the kernel of many rows (one round of its blocks, two, several; few rows of many columns) and, cut
    into few rows and columns, to the tiled one."""
    from sharpinference_amd import ops
    g = torch.Generator(device=DEV).manual_seed(M + N)
    x, w = torch.randn(M, K, device=DEV, generator=g), torch.randn(N, K, device=DEV, generator=g)
    x[0, 0], w[N - 1, K - 1] = float("inf"), float("nan")
    got = ops.gemm_tiled(x, w)
    for r in range(0, M, max(1, M // 3)):
        for c in (0, N // 2, N - 33):
            part = ops.gemm_tiled(x[r:r + 15].contiguous(), w[c:c + 33].contiguous())
            assert torch.equal(got[r:r + 15, c:c + 33].nan_to_num(1.5), part.nan_to_num(1.5)), (r, c)
