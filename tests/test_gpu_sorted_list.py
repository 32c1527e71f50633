"""The expert-sorted list at the numbers of pairs where it is made in another way, or in one more window of rows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,k,E,identity", [(1024, 1, 16, 0), (1025, 1, 1024, 0), (1024, 2, 16, 0), (683, 3, 60, 4), (512, 8, 128, 0), (4097, 1, 16, 0), (8192, 1, 7, 0), (2731, 3, 600, 40), (4096, 6, 64, 0), (4097, 6, 64, 3), (3000, 8, 9, 9)])
def test_every_pair_has_one_row_among_its_experts(T, k, E, identity):
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(T + k)
    score = torch.rand(T, E + identity, generator=g) + torch.linspace(0, 0.5, E + identity)
    ids, w = score.topk(k).indices.to(torch.int32), torch.rand(T, k, generator=g)
    rt = ops.moe_permute(ids.to(DEV), w.to(DEV), E, False, identity > 0)
    off, token, weight, inv = (t.cpu() for t in (rt.offsets, rt.sorted_token, rt.sorted_w, rt.inv_pos))
    count = torch.bincount(ids.flatten().long(), minlength=E + identity)[:E]
    assert off[:E + 1].tolist() == [0] + count.cumsum(0).tolist()
    real = ids < E
    row = inv.view(T, k)[real].long()
    assert torch.equal(row.sort().values, torch.arange(int(count.sum())))
    assert torch.equal(token[row].long(), torch.arange(T)[:, None].expand(T, k)[real]) and torch.equal(weight[row], w[real])
    expert = ids[real].long()
    assert bool(((off[expert] <= row) & (row < off[expert + 1])).all())
