"""Prompt attention where its stages and layouts can go wrong: pages whose size is no power of two, starts and ends inside
a 16-key block, a 32-key chunk and a stage, kept tokens before a window, every swizzle of the key rows, half a tile of
value columns, pages behind no visible key (given back: -1 in the table, whatever page 0 holds), and caches that begin at any address."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def reference(q, k, v, p, start, keep, scale, cap, sink):
    """One query row [nh, hd] over keys [L, nkv, hd] in 64 bits."""
    rep = q.shape[0] // k.shape[1]
    seen = torch.tensor([j for j in range(p + 1) if j >= start or j < keep])
    s = torch.einsum("hd,khd->hk", q.double(), k[seen].double().repeat_interleave(rep, 1)) * scale
    if cap:
        s = cap * torch.tanh(s / cap)
    if sink:
        s = torch.cat([s, torch.zeros(s.shape[0], 1, dtype=torch.float64)], 1)
    w = s.softmax(-1)[:, :len(seen)]
    return torch.einsum("hk,khd->hd", w, v[seen].double().repeat_interleave(rep, 1))


@pytest.mark.parametrize("nh,nkv,hd,vd,ps", [(8, 8, 128, 128, 48), (16, 2, 192, 128, 16), (3, 1, 64, 48, 80), (4, 2, 32, 96, 32),
                                             (2, 2, 96, 64, 112), (6, 3, 160, 96, 128), (2, 1, 192, 192, 144)])
@pytest.mark.parametrize("kind,window,keep,start,rows", [(0, 0, 0, 0, 1), (0, 0, 0, 61, 130), (1, 70, 0, 139, 67), (2, 33, 0, 200, 129),
                                                         (2, 90, 20, 333, 66), (2, 64, 100, 140, 65), (1, 160, 0, 150, 33)])
def test_stages_chunks_and_pages(nh, nkv, hd, vd, ps, kind, window, keep, start, rows):
    from sharpinference_amd import ops
    g = torch.Generator().manual_seed(hd + vd + ps + start)
    L, cap, sink = start + rows, 30.0 if ps == 48 else 0.0, ps == 32
    pages = (L + ps - 1) // ps
    k, v = (torch.randn(L, nkv, n, generator=g).bfloat16() for n in (hd, vd))
    q = torch.randn(rows, nh, hd, generator=g).bfloat16()
    first = lambda p: (p // window) * window if kind == 1 else max(0, p - window + 1) if kind == 2 else 0
    # page 0 belongs to nobody and holds what must not be read; keys past the end are finite
    kc = torch.zeros(pages + 1, nkv, ps, hd, dtype=torch.bfloat16)
    vc = torch.zeros(pages + 1, nkv, vd, ps, dtype=torch.bfloat16)
    kc[0], vc[0] = float("nan"), float("nan")
    order = torch.randperm(pages, generator=g) + 1
    table = torch.full((1, pages), -1, dtype=torch.int32)
    for i in range(pages):
        a, b = i * ps, min(L, (i + 1) * ps)
        if not (a < keep or b > first(start)):
            continue
        kc[order[i], :, :b - a] = k[a:b].transpose(0, 1)
        vc[order[i], :, :, :b - a] = v[a:b].permute(1, 2, 0)
        table[0, i] = int(order[i])
    positions = torch.arange(start, L, dtype=torch.int32, device=DEV)
    scale, got = 1.0 / math.sqrt(hd), {}
    for tile in (ops.PREFILL_TILE_TOKENS, ops.PREFILL_TILE_TOKENS // 2):
        tiles = torch.tensor([(0, o, min(tile, rows - o)) for o in range(0, rows, tile)], dtype=torch.int32, device=DEV)
        got[tile] = ops.attention_prefill(q.reshape(rows, nh * hd).to(DEV), kc.to(DEV), vc.to(DEV), table.to(DEV), positions, tiles, kind,
                                          window, scale, nh, nkv, hd, tile_tokens=tile, softcap=cap, sink=sink, vd=vd, keep=keep)
    a, b = got.values()
    assert torch.equal(a, b)
    a = a.cpu().double().view(rows, nh, vd)
    for t in sorted({0, 1, 15, 16, 31, 32, 63, 64, 65, 127, 128, rows - 1} & set(range(rows))):
        want = reference(q[t], k, v, start + t, first(start + t), keep, scale, cap, sink)
        # half a step of a bfloat16 result, and probabilities of 16 bits over values below 6
        assert bool(((a[t] - want).abs() <= 2 ** -8 * want.abs() + 6 * 2 ** -14).all()), (t, float((a[t] - want).abs().max()))


@pytest.mark.parametrize("nh,nkv,hd,vd", [(8, 2, 128, 128), (2, 1, 192, 96), (3, 3, 32, 96)])
@pytest.mark.parametrize("off", [(1, 0), (0, 2), (7, 5)])
def test_caches_may_begin_at_any_address(nh, nkv, hd, vd, off):
    """The same bits as from addresses that are multiples of 16, and no copy of the caches."""
    from sharpinference_amd import ops
    g = torch.Generator().manual_seed(hd + off[0])
    pages, ps, rows, start = 40, 16, 130, 300
    kc, vc = torch.randn(pages, nkv, ps, hd, generator=g).bfloat16().to(DEV), torch.randn(pages, nkv, vd, ps, generator=g).bfloat16().to(DEV)
    q = torch.randn(rows, nh * hd, generator=g).bfloat16().to(DEV)
    table = torch.randperm(pages, generator=g).int()[None, :27].contiguous().to(DEV)
    positions = torch.arange(start, start + rows, dtype=torch.int32, device=DEV)

    def moved(t, n):
        flat = torch.empty(t.numel() + n, dtype=t.dtype, device=DEV)
        flat[n:] = t.reshape(-1)
        return flat[n:].view(t.shape)

    own = moved(kc, off[0]), moved(vc, off[1])
    assert any(t.data_ptr() % 16 for t in own)
    for tile in (ops.PREFILL_TILE_TOKENS, ops.PREFILL_TILE_TOKENS // 2):
        tiles = torch.tensor([(0, o, min(tile, rows - o)) for o in range(0, rows, tile)], dtype=torch.int32, device=DEV)
        run = lambda k, v: ops.attention_prefill(q, k, v, table, positions, tiles, 0, 0, hd ** -0.5, nh, nkv, hd, tile_tokens=tile, vd=vd)
        want = run(kc, vc)
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        got = run(*own)
        assert torch.cuda.max_memory_allocated() - before < kc.numel() * 2
        assert torch.equal(got, want)
