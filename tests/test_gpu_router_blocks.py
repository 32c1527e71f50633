"""The router's blocks of experts and tokens, at the numbers where another block begins: the same bits from every one, and the picks in order."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("xd,wd", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("E,hidden", [(1, 8), (8, 520), (9, 512), (16, 5120), (17, 1032), (33, 64), (70, 512), (257, 16), (5, 75)])
def test_every_block_gives_the_same_bits_and_picks_in_order(E, hidden, xd, wd):
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(E + hidden)
    k = min(E, 6)
    x = torch.randn(1030, hidden, generator=g).to(xd).to(DEV)
    w = (torch.randn(E, hidden, generator=g) / hidden ** 0.5).to(wd).to(DEV)
    corr = (torch.randn(E, generator=g) * 0.3).to(DEV)
    for kw in ({}, {"correction": corr}):
        whole = ops.router_topk(x, w, k, ops.GATE_SIGMOID, want_gates=True, **kw)
        rank = whole[2] + corr if kw else whole[2]
        assert torch.equal(whole[0].long(), rank.sort(dim=1, descending=True, stable=True).indices[:, :k])
        assert torch.equal(whole[1], torch.gather(whole[2], 1, whole[0].long()))
        for n in (1, 63, 65, 257, 1023):
            assert all(torch.equal(a, b[:n]) for a, b in zip(ops.router_topk(x[:n], w, k, ops.GATE_SIGMOID, want_gates=True, **kw), whole))


@pytest.mark.parametrize("xd,wd", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16), (torch.float32, torch.float32)])
@pytest.mark.parametrize("E,hidden", [(2, 64), (3, 1032), (4, 512), (6, 72), (24, 520), (25, 264), (65, 2056), (300, 64)])
def test_every_choice_of_blocks_gives_the_same_bits(E, hidden, xd, wd):
    """The steps at which other numbers of experts, tokens and waves are taken: 256, 512, 1,024 and 2,048 tokens."""
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(E + hidden)
    x = torch.randn(2050, hidden, generator=g).to(xd).to(DEV)
    w = (torch.randn(E, hidden, generator=g) / hidden ** 0.5).to(wd).to(DEV)
    few = [ops.router_topk(x[a:a + 50], w, 2, ops.GATE_SOFTMAX_PICKED, want_gates=True) for a in range(0, 2050, 50)]
    want = [torch.cat(parts) for parts in zip(*few)]
    for n in (256, 257, 512, 513, 1024, 1025, 2048, 2050):
        assert all(torch.equal(a, b[:n]) for a, b in zip(ops.router_topk(x[:n], w, 2, ops.GATE_SOFTMAX_PICKED, want_gates=True), want)), n
    logits = x.double() @ w.double().t()
    terms = x.double().abs() @ w.double().abs().t()          # a lane's chain of hidden / 64 products, six sums of lanes
    assert bool(((want[2].double() - logits).abs() <= (hidden / 64 + 16) * 2.0 ** -24 * terms).all())


@pytest.mark.parametrize("E", [16, 70])
def test_ties_and_values_that_are_no_numbers(E):
    from sharpinference_amd import ops

    x = torch.ones(20, 64, device=DEV).bfloat16()
    w = torch.zeros(E, 64, device=DEV).bfloat16()
    w[E - 2] = 1.0
    w[3] = 1.0
    ids, _ = ops.router_topk(x, w, 4, ops.GATE_SOFTMAX_PICKED)
    assert ids.cpu().tolist() == [[3, E - 2, 0, 1]] * 20
    x[7] = float("nan")
    ids, _ = ops.router_topk(x, w, 4, ops.GATE_SOFTMAX_PICKED)
    assert ids[:7].cpu().tolist() + ids[8:].cpu().tolist() == [[3, E - 2, 0, 1]] * 19
    assert len(set(ids[7].tolist())) == 4 and 0 <= int(ids[7].min()) and int(ids[7].max()) < E
