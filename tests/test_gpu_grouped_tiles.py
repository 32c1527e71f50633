"""The grouped product of many rows at the edges of its tiles: every height of a tile, one and several siblings, the shortest
sums, columns that end inside a tile and inside a block, slots cut in two, and more groups than it keeps offsets of."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def routed(counts, shared=False):
    from sharpinference_amd import ops
    ids = torch.cat([torch.full((c,), e, dtype=torch.int32) for e, c in enumerate(counts)])
    ids = ids[torch.randperm(len(ids), generator=torch.Generator().manual_seed(len(ids)))].view(-1, 1).to(DEV)
    return ops.moe_permute(ids, torch.ones(ids.shape, device=DEV), len(counts), shared_group=shared)


HEIGHTS = [1, 31, 32, 33, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 224, 225, 255, 256, 257, 513]


@pytest.mark.parametrize("counts", [HEIGHTS, HEIGHTS[::-1], [700], [0, 256, 0, 0, 9]])
@pytest.mark.parametrize("N,K", [(20, 64), (264, 128), (320, 192), (272, 320), (1056, 128), (96, 1152), (32, 576)])
def test_every_height_of_a_tile(counts, N, K):
    from sharpinference_amd import ops
    g = torch.Generator().manual_seed(N + K)
    x = torch.randn(sum(counts), K, generator=g).bfloat16()
    w = (torch.randn(len(counts), N, K, generator=g) * 0.1).bfloat16()
    rt = routed(counts)
    token, offsets = rt.sorted_token.cpu().long(), rt.offsets.cpu().tolist()
    want = torch.cat([x[token[a:b]].double() @ w[e].double().T for e, (a, b) in enumerate(zip(offsets, offsets[1:]))])
    size = torch.cat([x[token[a:b]].double().abs() @ w[e].double().abs().T for e, (a, b) in enumerate(zip(offsets, offsets[1:]))])
    forms = [w.to(DEV)] + ([ops.pack_weight(w.to(DEV), keep_rows=False)] if ops.can_pack(w) else [])
    for form in forms:
        exact = ops.gemm_grouped(x.to(DEV), form, rt, True, torch.float32).cpu().double()
        # a sum of K products in 32 bits
        assert bool(((exact - want).abs() <= K * 2 ** -24 * size + 1e-30).all())
        got = ops.gemm_grouped(x.to(DEV), form, rt, True, torch.bfloat16).cpu()
        assert torch.equal(got, exact.float().bfloat16())
        # rows of their own order, read from an address that is no multiple of 16
        flat = torch.empty(x.numel() + 1, dtype=torch.bfloat16, device=DEV)
        flat[1:] = x[token].reshape(-1).to(DEV)
        assert torch.equal(ops.gemm_grouped(flat[1:].view(x.shape), form, rt, False, torch.bfloat16).cpu(), got)
        if N % 32 == 0:
            gate, up = exact.float().bfloat16().float().chunk(2, 1)
            act = ops.gemm_grouped_swiglu(x.to(DEV), form, rt, None).cpu().float()
            ref = gate / (1 + torch.exp(-gate)) * up
            # a result rounded to 8 bits, and the exponential's and the quotient's last places
            assert bool(((act - ref).abs() <= 2 ** -8 * ref.abs() + 1e-30).all())


@pytest.mark.parametrize("off", [1, 2, 5])
def test_weights_may_begin_at_any_address(off):
    """The same bits as from an address that is a multiple of 16, and no copy of the weights."""
    from sharpinference_amd import ops
    g = torch.Generator().manual_seed(off)
    counts, N, K = [3, 0, 290, 64, 31], 320, 192
    x = torch.randn(sum(counts), K, generator=g).bfloat16().to(DEV)
    w = (torch.randn(len(counts), N, K, generator=g) * 0.1).bfloat16().to(DEV)
    rt = routed(counts)
    flat = torch.empty(w.numel() + off, dtype=torch.bfloat16, device=DEV)
    flat[off:] = w.reshape(-1)
    own = flat[off:].view(w.shape)
    assert own.data_ptr() % 16
    for gather in (True, False):
        assert torch.equal(ops.gemm_grouped(x, own, rt, gather, torch.float32), ops.gemm_grouped(x, w, rt, gather, torch.float32))
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        got = ops.gemm_grouped_swiglu(x, own, rt, None, gather)
        assert torch.cuda.max_memory_allocated() - before < w.numel() * 2
        assert torch.equal(got, ops.gemm_grouped_swiglu(x, w, rt, None, gather))


def test_more_groups_than_offsets_are_kept_of():
    from sharpinference_amd import ops
    g = torch.Generator().manual_seed(3)
    counts = [1] * 1024
    rt = routed(counts, shared=True)
    x = torch.randn(1024, 64, generator=g).bfloat16()
    w = (torch.randn(1025, 16, 64, generator=g) * 0.1).bfloat16()
    got = ops.gemm_grouped(x.to(DEV), w.to(DEV), rt, True, torch.float32).cpu().double()
    rows = x[rt.sorted_token.cpu().long()].double()
    want = torch.cat([torch.einsum("tk,tnk->tn", rows[:1024], w[:1024].double()), rows[1024:] @ w[1024].double().T])
    assert float((got - want).abs().max()) <= 64 * 2 ** -24 * float((rows.abs().max() * w.abs().max() * 64))
