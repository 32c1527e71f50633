"""The router's register-blocked logits (64 tokens and more) and the list of many pairs, at the edges of their blocks."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("xd,wd", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("E,hidden", [(3, 8), (16, 1032), (63, 512), (66, 520), (130, 2056)])
def test_a_tokens_logits_are_the_same_bits_in_every_batch(E, hidden, xd, wd):
    """A block a token, four experts a wave, four tokens a block: every logit is one chain in the width's order."""
    from sharpinference_amd import ops
    g = torch.Generator().manual_seed(E)
    x = torch.randn(259, hidden, generator=g).to(xd).to(DEV)
    w = (torch.randn(E, hidden, generator=g) / hidden ** 0.5).to(wd).to(DEV)
    bias = torch.randn(E, generator=g).to(DEV)
    want = x.double() @ w.double().t() + bias.double()
    few = [ops.router_topk(x[a:a + 37], w, 2, ops.GATE_SOFTMAX_PICKED, want_gates=True, bias=bias) for a in range(0, 259, 37)]
    for n in (64, 67, 256, 257, 259):
        got = ops.router_topk(x[:n], w, 2, ops.GATE_SOFTMAX_PICKED, want_gates=True, bias=bias)
        for one, parts in zip(got, zip(*few)):
            assert torch.equal(one, torch.cat(parts)[:n])
        # a lane's chain of hidden / 64 products, six sums of lanes, the bias
        terms = x[:n].double().abs() @ w.double().abs().t() + bias.double().abs()
        assert bool(((got[2].double() - want[:n]).abs() <= (hidden / 64 + 16) * 2.0 ** -24 * terms).all())


@pytest.mark.parametrize("T,k,E,shared,identity", [(1, 1, 1, True, 0), (63, 3, 5, False, 0), (2049, 4, 66, False, 8), (1366, 6, 130, True, 0),
                                                   (9000, 1, 3, True, 0), (700, 8, 1024, False, 0)])
def test_the_sorted_list_and_its_plan(T, k, E, shared, identity):
    from sharpinference_amd import ops
    g = torch.Generator().manual_seed(T)
    score = torch.rand(T, E + identity, generator=g) + torch.linspace(0, 0.7, E + identity)       # uneven groups, some empty
    ids = score.topk(k).indices.to(torch.int32)
    w = torch.rand(T, k, generator=g)
    rt = ops.moe_permute(ids.to(DEV), w.to(DEV), E, shared, identity > 0)
    off, st, sw, inv = (t.cpu() for t in (rt.offsets, rt.sorted_token, rt.sorted_w, rt.inv_pos))
    count = torch.bincount(ids.flatten().long(), minlength=E + identity)[:E]
    assert off[:E + 1].tolist() == [0] + count.cumsum(0).tolist()
    real = ids < E
    row = inv.view(T, k)[real].long()
    assert row.unique().numel() == row.numel()
    assert torch.equal(st[row].long(), torch.arange(T)[:, None].expand(T, k)[real]) and torch.equal(sw[row], w[real])
    assert bool(((off[:-1 if not shared else -2][ids[real].long()] <= row) & (row < off[1 + ids[real].long()])).all())
    if shared:
        assert off[E + 1] == off[E] + T and st[T * k:].tolist() == list(range(T)) and bool((sw[T * k:] == 1).all())
        count = torch.cat([count, torch.tensor([T])])
    # the plan: every group's parts once, the heaviest units first, dealt to the XCDs row by row in turning direction
    sib = lambda c: -(-c // 128)
    parts = lambda s: 2 if s <= 2 else 4 if s <= 4 else 8 if s <= 8 else 16
    groups = [(i, sib(c)) for i, c in enumerate(count.tolist()) if c]
    groups.sort(key=lambda t: (-t[1] * (16 // parts(t[1])), t[0]))
    units = [[i, p, parts(s), s] for i, s in groups for p in range(parts(s))]
    plan = rt.plan.cpu()
    stride = (plan.numel() - 16) // 8
    for x in range(8):
        mine = [units[8 * r + (7 - x if r & 1 else x)] for r in range(-(-len(units) // 8)) if 8 * r + (7 - x if r & 1 else x) < len(units)]
        lists = plan[x * stride:(x + 1) * stride]
        assert int(lists[0]) == len(mine) and lists[1:1 + 4 * len(mine)].view(-1, 4).tolist() == mine
    assert int(plan[8 * stride:].abs().max()) == 0
