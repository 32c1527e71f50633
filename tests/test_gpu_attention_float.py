"""The 32-bit path's attention on the float matrix instruction (csrc/attention_float.hip) against float64 and against the
kernel with one (token, head) a block, which serves pages that are not whole 16-key blocks."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _pages(rows, ps, transposed, fill):
    """Rows [L, nkv, d] of each entry in pages [n, nkv, ps, d] (values: [n, nkv, d, ps]) dealt out backwards; slots past an
    entry's end hold `fill`."""
    nkv, d = rows[0].shape[1:]
    counts = [-(-r.shape[0] // ps) for r in rows]
    n = sum(counts) + 1
    pool = torch.full((n, nkv, ps, d), fill)
    bt = torch.full((len(rows), max(counts)), -1, dtype=torch.int32)
    page = n - 1
    for e, r in enumerate(rows):
        for b in range(counts[e]):
            seg = r[b * ps:(b + 1) * ps]
            pool[page, :, :seg.shape[0]] = seg.transpose(0, 1)
            bt[e, b] = page
            page -= 1
    return (pool.transpose(2, 3).contiguous() if transposed else pool), bt


def _exact(q, ks, vs, entry, pos, kind, window, scale, keep, softcap, sinks, gate):
    T, nh, _ = q.shape
    out = torch.zeros(T, nh, vs[0].shape[2], dtype=torch.float64)
    for t in range(T):
        p = int(pos[t])
        k, v = ks[entry[t]].double(), vs[entry[t]].double()
        G = nh // k.shape[1]
        start = p // window * window if kind == 1 else max(0, p - window + 1) if kind == 2 else 0
        seen = torch.tensor([j for j in range(p + 1) if j >= start or j < keep])
        for h in range(nh):
            s = (k[seen, h // G] @ q[t, h].double()) * scale
            if softcap:
                s = softcap * torch.tanh(s / softcap)
            e = torch.exp(s - s.max())
            den = e.sum() + (torch.exp(sinks[h].double() - s.max()) if sinks is not None else 0.0)
            out[t, h] = (e @ v[seen, h // G]) / den * (torch.sigmoid(gate[t, h].double()) if gate is not None else 1.0)
    return out


@pytest.mark.parametrize("nh,nkv,hd,vd,kind,window,ps,extras", [
    (4, 1, 128, 128, 0, 0, 16, False), (10, 2, 64, 64, 1, 24, 64, True), (34, 2, 128, 128, 2, 50, 32, True),
    (3, 3, 192, 128, 1, 40, 16, False), (8, 4, 64, 64, 0, 0, 128, True), (6, 2, 128, 128, 2, 7, 48, True)])
def test_float_rows_share_their_keys(nh, nkv, hd, vd, kind, window, ps, extras):
    from sharpinference_amd import ops
    g = torch.Generator().manual_seed(nh * hd + ps)
    lens = [1, 17, 70, 16, 131]                    # single tokens, edges of the 16-key blocks
    counts = [1, 1, 37, 16, 5]                     # the step's tokens of each: the last ones, flat rows cut anywhere
    ks = [torch.randn(n, nkv, hd, generator=g) for n in lens]
    vs = [torch.randn(n, nkv, vd, generator=g) for n in lens]
    entry = [e for e, c in enumerate(counts) for _ in range(c)]
    pos = [n - c + i for n, c in zip(lens, counts) for i in range(c)]
    T, scale = len(entry), 1.0 / math.sqrt(hd)
    q = torch.randn(T, nh, hd, generator=g)
    keep, softcap = (20 if kind else 0, 15.0) if extras else (0, 0.0)
    sinks = torch.randn(nh, generator=g) if extras else None
    gate = torch.randn(T, nh + 3, generator=g) if extras else None

    def run(page, sel=None, fill=float("nan")):
        """Slots that were never written hold `fill`: none of it may reach a row."""
        kc, bt = _pages(ks, page, False, fill)
        vc, _ = _pages(vs, page, True, fill)
        idx = torch.arange(T) if sel is None else torch.tensor(sel)
        out = ops.attention_generic(q[idx].reshape(len(idx), -1).contiguous().to(DEV), kc.to(DEV), vc.to(DEV), bt.to(DEV),
                                    torch.tensor(entry, dtype=torch.int32)[idx].to(DEV),
                                    torch.tensor(pos, dtype=torch.int32)[idx].to(DEV), kind, window, scale, nh, nkv, hd, vd,
                                    softcap=softcap, sink=sinks.to(DEV) if extras else False, keep=keep,
                                    gate=(gate[idx].contiguous().to(DEV), 2) if extras else None)
        return out.cpu().view(len(idx), nh, vd)

    want = _exact(q, ks, vs, entry, pos, kind, window, scale, keep, softcap, sinks, gate[:, 2:] if extras else None)
    got, general = run(ps), run(8)
    # a score's rounding: (hd / 2 + 2) steps of 2^-24 of its terms' sizes, felt twice by a weight (over and under the line),
    # and 2^-24 a key of the sums
    size = max(float((q[t].abs().view(nkv, -1, hd) @ ks[entry[t]].abs().permute(1, 2, 0)).max()) for t in range(T)) * scale
    bound = 2.0 ** -24 * (2 * (hd / 2 + 2) * size + 2 * max(lens)) * max(float(v.abs().max()) for v in vs)
    err, err_general = (got - want).abs(), (general - want).abs()
    assert float(err.max()) <= bound, (float(err.max()), bound)
    assert float(err.square().mean().sqrt()) <= 1.25 * float(err_general.square().mean().sqrt()), "rounds more than one row a block"
    # the same bits whoever shares the tile, and whatever lies in unwritten slots
    assert torch.equal(run(ps, fill=0.0), got)
    for sel in ([0, 1], list(range(5, 30)), [T - 1]):
        assert torch.equal(run(ps, sel), got[sel])


def test_a_later_tokens_infinity_stays_with_it():
    """A value that is no number reaches the rows that see its key, no other row of the tile."""
    from sharpinference_amd import ops
    g = torch.Generator().manual_seed(1)
    L, nh, nkv, hd = 24, 4, 2, 64
    k, v = torch.randn(L, nkv, hd, generator=g), torch.randn(L, nkv, hd, generator=g)
    q = torch.randn(L, nh * hd, generator=g).to(DEV)
    zeros, pos = torch.zeros(L, dtype=torch.int32, device=DEV), torch.arange(L, dtype=torch.int32, device=DEV)

    def run():
        kc, bt = _pages([k], 32, False, 0.0)
        vc, _ = _pages([v], 32, True, 0.0)
        return ops.attention_generic(q, kc.to(DEV), vc.to(DEV), bt.to(DEV), zeros, pos, 0, 0, 0.125, nh, nkv, hd).cpu().view(L, nh, hd)
    before = run()
    v[18, 1, 5] = float("inf")
    after = run()
    assert torch.isinf(after[18:, 2:, 5]).all()
    after[18:, 2:, 5] = before[18:, 2:, 5]
    assert torch.equal(after, before)
