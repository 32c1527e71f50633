"""Steps of many tokens turn their values into the cache's pages in blocks of their own: the same bits as the same tokens in
portions small enough to go token by token."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}


class _Step:
    def __init__(self, positions, slot=0):
        T = len(positions)
        i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
        self.n_entries, self.n_tokens = 1, T
        self.positions, self.entry_of_token = i32(positions), i32([0] * T)
        self.cu_tokens, self.state_slots = i32([0, T]), i32([slot])


def _slots(kind, T, pages, ps, g):
    """A prompt's pages in shuffled order from the first place on, or from another, tokens anywhere, or some not stored."""
    if kind in ("pages", "shifted"):
        first = 0 if kind == "pages" else 5
        order = torch.randperm(pages, generator=g)
        place = torch.arange(T) + first
        return (order[place // ps] * ps + place % ps).to(torch.int32)
    slots = torch.randperm(pages * ps, generator=g)[:T].to(torch.int32)
    if kind == "holes":
        slots[torch.rand(T, generator=g) < 0.4] = -1
    return slots if kind != "none" else torch.full((T,), -1, dtype=torch.int32)


CASES = [("pages", 65, 16, 128), ("pages", 200, 32, 64), ("shifted", 83, 16, 128), ("shifted", 131, 48, 72), ("anywhere", 96, 16, 136),
         ("holes", 79, 16, 8), ("none", 70, 16, 128), ("pages", 130, 16, 24)]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("kind, T, ps, vd", CASES)
@pytest.mark.parametrize("layout", [0, 1])
def test_rotated_heads_and_values_of_a_long_step(kind, T, ps, vd, layout, dtype):
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(T + vd)
    nh, nkv, hd, r, pages = 5, 3, 128, 32, T // ps + 3
    width = (nh + nkv) * hd + nkv * vd
    qkv = torch.randn(T, width + 8, generator=g).to(DT[dtype]).to(DEV)
    bias = torch.randn(width, generator=g).to(DEV) if T % 2 else None
    freq = torch.tensor([300.0 ** (-2.0 * i / r) for i in range(r // 2)], device=DEV)
    slots = _slots(kind, T, pages, ps, g).to(DEV)
    pos = (torch.arange(T) * 7).to(torch.int32).to(DEV)
    got, caches = [], []
    for portion in (T, 50):
        kc = torch.zeros(pages, nkv, ps, hd, dtype=DT[dtype], device=DEV)
        vc = torch.zeros(pages, nkv, vd, ps, dtype=DT[dtype], device=DEV)
        out = [ops.rope_kv(qkv[i:i + portion], kc, vc, slots[i:i + portion], pos[i:i + portion], freq, True, 1e-5, (40.0, 0.1), nh, nkv, hd,
                           layout, bias, vd, 8) for i in range(0, T, portion)]
        got.append(torch.cat(out).float())
        caches.append((kc.float(), vc.float()))
    assert torch.equal(caches[0][1], caches[1][1])
    assert torch.equal(got[0], got[1]) and torch.equal(caches[0][0], caches[1][0])


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("kind, T, ps, vd", CASES)
@pytest.mark.parametrize("form", ["run", "pairs", "mixed", "bias", "conv", "conv3", "keys", "maps", "whole", "whole of many heads"])
def test_prepared_heads_and_values_of_a_long_step(kind, T, ps, vd, form, dtype):
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(T + vd + len(form))
    nh, nkv, hd, r, pages = 64 if form == "whole of many heads" else 6, 2, 128, 32, T // ps + 3
    vd = hd if form == "keys" else vd
    qn, kn, vn = nh * hd, nkv * hd, 0 if form == "keys" else nkv * vd
    C, taps = qn + kn + vn, {"conv": 4, "conv3": 3}.get(form, 0)
    proj = torch.randn(T, C + 8, generator=g).to(DT[dtype]).to(DEV)
    other = torch.randn(T, vn + 16, generator=g).to(DT[dtype]).to(DEV)
    whole = form.startswith("whole")
    wq, wk = (torch.rand(n, generator=g).to(DEV) + 0.5 for n in ((qn, kn) if whole else (hd, hd)))
    conv = torch.randn(C, taps, generator=g).to(DEV) if taps else None
    bias = torch.randn(C, generator=g).to(DEV) if form == "bias" else None
    freq = torch.tensor([300.0 ** (-2.0 * i / r) for i in range(r // 2)], device=DEV)
    slots = _slots(kind, T, pages, ps, g).to(DEV)
    results = []
    for portion in (T, 50):
        kc = torch.zeros(pages, nkv, ps, hd, dtype=DT[dtype], device=DEV)
        vc = torch.zeros(pages, nkv, vd, ps, dtype=DT[dtype], device=DEV)
        tail = torch.zeros(2, taps - 1, C, device=DEV) if taps else None
        out = []
        for i in range(0, T, portion):
            n = min(portion, T - i)
            out.append(ops.qk_prep(proj[i:i + n], 0, qn, None if form == "keys" else qn + kn, nh, nkv, hd, vd, _Step(list(range(i, i + n)), 1), kc, vc,
                                   slots[i:i + n], ops.NORM_WHOLE if whole else ops.NORM_PER_HEAD, wq, wk, 1e-5, freq,
                                   ops.PAIRS_INTERLEAVED if form == "pairs" else ops.PAIRS_HALF_SPLIT, 1.0,
                                   conv, tail, bias=bias, maps=2 if form == "maps" else 1,
                                   v_mix=(other[i:i + n], 16, 0.3) if form == "mixed" else None))
        results.append((torch.cat(out), kc, vc) + ((tail,) if taps else ()))
    for a, b in zip(*results):
        assert torch.equal(a, b)
