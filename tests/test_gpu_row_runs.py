"""Row kernels that take eight channels a thread: the bits of the forms that take any width, or the plain arithmetic in double."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}
# float: a sum of squares over at most 16 terms a lane and 6 of the lanes, halved by the root, and five roundings behind it; bfloat16: its own
TOL = {"float32": 16 * 2.0 ** -24, "bfloat16": 2.0 ** -8}


class _Step:
    def __init__(self, lens, slots):
        i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
        cu = [0]
        for n in lens:
            cu.append(cu[-1] + n)
        self.n_entries, self.n_tokens = len(lens), cu[-1]
        self.cu_tokens, self.state_slots = i32(cu), i32(slots)
        self.entry_of_token = i32([e for e, n in enumerate(lens) for _ in range(n)])
        self.positions = i32([p for n in lens for p in range(n)])


def _shifted(x):
    """The same values two columns further on, in rows too wide to be read by eights."""
    wide = torch.zeros(x.shape[0], x.shape[1] + 3, dtype=x.dtype, device=x.device)
    wide[:, 2:2 + x.shape[1]] = x
    return wide


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("lens, C", [([1], 8), ([2, 1, 3, 4], 2056), ([1] * 20, 64), ([3, 250, 1, 2, 9], 264), ([300], 2048), ([5, 4, 257], 40)])
def test_four_taps_by_eights_give_the_bits_of_a_channel_at_a_time(lens, C, dtype):
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(C + len(lens))
    T = sum(lens)
    u = (torch.randn(T, C, generator=g) * 2).to(DT[dtype]).to(DEV)
    w, b = torch.randn(C, 4, generator=g).to(DEV), torch.randn(C, generator=g).to(DEV) if C != 64 else None
    held = torch.randn(len(lens) + 2, 3, C, generator=g).to(DEV)
    ctx, out = _Step(lens, list(range(len(lens), 0, -1))), []
    for rows, off in ((u, 0), (_shifted(u), 2)):
        tail = held.clone()
        out.append((ops.short_conv(rows, off, C, w, b, tail, ctx), tail))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("lens, C", [([3, 250, 1, 2, 9], 2056), ([100, 1, 3], 6144), ([8000, 1, 300], 64), ([700, 1, 3], 6000), ([70000], 8), ([1] * 300, 7048), ([1, 2] * 300, 7000)])
def test_four_taps_by_eights_in_longer_steps(lens, C, dtype):
    """Two and four tokens a thread, narrow rows side by side in a block; single tokens, whose rows before are all in the tail."""
    test_four_taps_by_eights_give_the_bits_of_a_channel_at_a_time(lens, C, dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T, groups, size", [(1, 1, 8), (70, 5, 24), (3, 16, 128), (33, 2, 192), (9, 3, 512), (5, 2, 520), (2, 3, 1024)])
@pytest.mark.parametrize("act, first, weighted", [("silu", False, True), ("silu", True, True), ("sigmoid", False, False)])
def test_parts_in_neighbouring_lanes(T, groups, size, act, first, weighted, dtype):
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(T + size)
    N, off, eps = groups * size, 16, 1e-3
    o = (torch.randn(T, N, generator=g) * 5).to(DEV)
    w = torch.randn(N, generator=g).to(DEV) if weighted else None
    gp = (torch.randn(T, off + N + 8, generator=g) * 2).to(DT[dtype]).to(DEV)
    got = ops.group_norm_gate(o, w, eps, groups, DT[dtype], gp, off, ops.GATE_SILU if act == "silu" else ops.GATE_SIGMOID_ACT, gate_first=first)
    z = gp.double()[:, off:off + N]
    gate = torch.sigmoid(z) * (z if act == "silu" else 1.0)
    x = o.double() * gate if first else o.double()
    x = x.view(T, groups, size)
    want = (x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps)).reshape(T, N) * (w.double() if weighted else 1.0) * (1.0 if first else gate)
    assert float(((got.double() - want).abs() - TOL[dtype] * want.abs()).max()) <= 2.0 ** -60
    if not first:
        heads = ops.head_norm_gate(o, w[:size].contiguous() if weighted else torch.ones(size, device=DEV), eps, groups, size, DT[dtype], gp, off)
        want = (x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps) * (w.double()[:size] if weighted else 1.0)).reshape(T, N) * torch.sigmoid(z) * z
        assert float(((heads.double() - want).abs() - TOL[dtype] * want.abs()).max()) <= 2.0 ** -60


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("size", [8, 16, 24, 64, 96, 128, 192, 256, 320, 512, 520, 1024])
@pytest.mark.parametrize("first", [False, True])
def test_parts_in_neighbouring_lanes_give_the_bits_of_a_wave_a_part(size, first, dtype):
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(size)
    T, groups, eps = 9, 5, 1e-3
    N = groups * size
    o = (torch.randn(T, N, generator=g) * 5).to(DEV)
    w = torch.randn(N, generator=g).to(DEV)
    gates = (torch.randn(T, N, generator=g) * 2).to(DT[dtype]).to(DEV)
    wide = _shifted(gates)               # (gates that cannot be read by eights: a wave a part)
    for act in (ops.GATE_SILU, ops.GATE_SIGMOID_ACT):
        by = [ops.group_norm_gate(o, w, eps, groups, DT[dtype], x, off, act, gate_first=first) for x, off in ((gates, 0), (wide, 2))]
        assert torch.equal(*by)
    if not first:
        assert torch.equal(*[ops.head_norm_gate(o, w[:size].contiguous(), eps, groups, size, DT[dtype], x, off) for x, off in ((gates, 0), (wide, 2))])


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T, groups, size", [(1229, 5, 8), (6145, 1, 16), (770, 8, 24), (410, 15, 64), (2049, 3, 40)])
@pytest.mark.parametrize("first", [False, True])
def test_many_parts_of_up_to_64_channels(T, groups, size, first, dtype):
    """More parts than go a wave each: the same parts in portions that do, for their bits."""
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(T)
    N, cut = groups * size, T // 2
    o, w = (torch.randn(T, N, generator=g) * 5).to(DEV), torch.randn(N, generator=g).to(DEV)
    gates = (torch.randn(T, N, generator=g) * 2).to(DT[dtype]).to(DEV)
    go = lambda a, b: ops.group_norm_gate(o[a:b].contiguous(), w, 1e-3, groups, DT[dtype], gates[a:b].contiguous(), 0, ops.GATE_SILU, gate_first=first)
    assert torch.equal(go(0, T), torch.cat([go(0, cut), go(cut, T)]))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T, H, e, gate", [(1, 1, 8, True), (70, 8, 128, False), (3, 5, 136, True), (9, 2, 512, True), (4, 3, 520, True)])
def test_differences_of_maps_in_neighbouring_lanes(T, H, e, gate, dtype):
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(T + e)
    a = torch.randn(T, H, 2, e, generator=g).to(DT[dtype]).to(DEV)
    proj = torch.randn(T, 11 + H, generator=g).to(DT[dtype]).to(DEV)
    lam, eps, post = 0.62, 1e-5, 0.7
    d = a[:, :, 0].double() - lam * a[:, :, 1].double()
    mul = post / torch.sqrt(d.pow(2).mean(-1, keepdim=True) + eps)
    if gate:
        mul = mul * torch.sigmoid(proj[:, 11:].double())[:, :, None]
    want = d * mul
    got = ops.map_difference(a.reshape(T, -1), H, e, lam, eps, post, proj if gate else None, 11).double().view(T, H, e)
    # (a difference keeps the error of its two terms and of lambda's float)
    terms = (a[:, :, 0].double().abs() + a[:, :, 1].double().abs()) * mul * 2.0 ** -23
    assert float(((got - want).abs() - TOL[dtype] * want.abs() - terms).max()) <= 2.0 ** -60


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("e", [8, 16, 24, 64, 96, 128, 192, 256, 320, 512])
def test_differences_of_maps_in_neighbouring_lanes_give_the_bits_of_a_wave_a_head(e, dtype):
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(e)
    T, H = 9, 5
    flat = torch.randn(T * H * 2 * e, generator=g).to(DT[dtype]).to(DEV)
    proj = torch.randn(T, 11 + H, generator=g).to(DT[dtype]).to(DEV)
    moved = torch.cat([flat[:1], flat])[1:]          # (one element on: no 16-byte loads, a wave a head)
    assert torch.equal(*[ops.map_difference(x.view(T, -1), H, e, 0.62, 1e-5, 0.7, proj, 11) for x in (flat, moved)])


@pytest.mark.parametrize("T, N", [(1, 8), (70, 2056), (5, 1000), (3, 12), (5000, 8), (301, 72), (257, 24)])
def test_columns_side_by_side_add_as_one_by_one(T, N):
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(T + N)
    x, b = (torch.randn(T, N, generator=g) * 3).to(DEV), torch.randn(N, generator=g).to(DEV)
    for dtype in DT.values():
        y = x.to(dtype)
        assert torch.equal(ops.add_bias(y.clone(), b), (y.float() + b).to(dtype))


def _prepared_by_eights_and_one_by_one(turn, form, nh, nkv, hd, T, dtype):
    """The same rows aligned for runs of eight and shifted, so that they are staged an element at a time: the same bits."""
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(hd + T + len(form))
    vd, r, ps = 40, 16, 16
    keys, whole, maps = "keys" in form, "whole" in form, 2 if "maps" in form else 1
    r, vd = min(r, hd // maps), hd if keys else vd
    if turn == "none" or (r < 16 and turn == "halves"):
        r = 0
    qn, kn, vn, pages = nh * hd, nkv * hd, 0 if keys else nkv * vd, T // ps + 3
    C, taps = qn + kn + vn, 3 if "conv3" in form else 6 if "conv6" in form else 4 if "conv" in form else 0
    proj = torch.randn(T, C + 8, generator=g).to(DT[dtype]).to(DEV)
    wq, wk = (torch.rand(n, generator=g).to(DEV) + 0.5 for n in ((qn, kn) if whole else (hd, hd)))
    conv = torch.randn(C, taps, generator=g).to(DEV) if taps else None
    freq = torch.tensor([300.0 ** (-2.0 * i / r) for i in range(r // 2)], device=DEV) if r else None
    slots = torch.randperm(pages * ps, generator=g)[:T].to(torch.int32).to(DEV)
    held = torch.randn(4, max(taps - 1, 1), C, generator=g).to(DEV)
    ctx, results = _Step([1, 2, T - 4, 1], [3, 0, 2, 1]), []
    for rows, off in ((proj, 0), (_shifted(proj), 2)):           # (rows that cannot be read by eights are staged)
        kc = torch.zeros(pages, nkv, ps, hd, dtype=DT[dtype], device=DEV)
        vc = torch.zeros(pages, nkv, vd, ps, dtype=DT[dtype], device=DEV)
        tail = held.clone() if taps else None
        q = ops.qk_prep(rows, off, off + qn, None if keys else off + qn + kn, nh, nkv, hd, vd, ctx, kc, vc, slots,
                        ops.NORM_WHOLE if whole else ops.NORM_PER_HEAD, wq, wk, 1e-5, freq,
                        ops.PAIRS_INTERLEAVED if turn == "pairs" else ops.PAIRS_HALF_SPLIT, 1.0, conv, tail, maps=maps)
        results.append((q, kc, vc) + ((tail,) if taps else ()))
    for i, (a, b) in enumerate(zip(*results)):
        if turn != "halves" or i > 1:
            assert torch.equal(a, b)
            continue
        # (scalar rows round the other of a high half's two products: one rounding of a term and one of the sum on either side)
        tol = 3 * 2.0 ** -24 if dtype == "float32" else 2.0 ** -8 + 3 * 2.0 ** -24
        a, b = a.double(), b.double()
        assert bool(((a - b).abs() <= tol * (a.abs() + b.abs()) + 3 * 2.0 ** -24 * b.abs().amax(-1, keepdim=True)).all())


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T", [9, 70])
@pytest.mark.parametrize("hd", [16, 64, 96, 128, 192, 256, 512])
@pytest.mark.parametrize("form", ["conv", "conv3", "keys", "maps", "maps conv", "whole", "whole conv", "whole keys"])
@pytest.mark.parametrize("turn", ["none", "pairs", "halves"])
def test_heads_by_runs_give_the_bits_of_the_staged_form(turn, form, hd, T, dtype):
    _prepared_by_eights_and_one_by_one(turn, form, 4 if hd > 256 else 6, 2, hd, T, dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T", [9, 70, 300])
@pytest.mark.parametrize("form", ["conv", "conv3", "keys", "maps"])
def test_heads_in_several_turns_give_the_bits_of_the_staged_form(form, T, dtype):
    _prepared_by_eights_and_one_by_one("halves", form, 64, 2, 192, T, dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("form, nh, hd, T", [("conv", 16, 192, 711), ("conv", 16, 192, 712), ("whole conv3", 16, 192, 712), ("conv3", 6, 64, 500), ("conv3", 6, 64, 501),
                                             ("conv6", 6, 64, 1000), ("whole conv6", 6, 64, 1001), ("conv6", 6, 16, 70), ("maps conv6", 6, 128, 70), ("conv6", 2, 64, 9)])
def test_convolved_heads_on_both_sides_of_the_choices(form, nh, hd, T, dtype):
    """Lanes a step, tokens and lanes of more than four taps, values beside or apart."""
    _prepared_by_eights_and_one_by_one("pairs", form, nh, 2, hd, T, dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_plain_heads_have_the_same_bits_in_steps_of_any_size(dtype):
    """A turn a block, two and four, neighbouring tokens on a die or not."""
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(5)
    T, nh, nkv, hd, vd, ps = 300, 40, 2, 192, 40, 16
    qn, kn, pages = nh * hd, nkv * hd, 20
    proj = torch.randn(T, qn + kn + nkv * vd, generator=g).to(DT[dtype]).to(DEV)
    wq, wk = (torch.rand(hd, generator=g).to(DEV) + 0.5 for _ in range(2))
    freq = torch.tensor([300.0 ** (-2.0 * i / 64) for i in range(32)], device=DEV)
    slots, results = torch.randperm(pages * ps, generator=g)[:T].to(torch.int32).to(DEV), []
    for portion in (300, 70, 33, 7):
        kc = torch.zeros(pages, nkv, ps, hd, dtype=DT[dtype], device=DEV)
        vc = torch.zeros(pages, nkv, vd, ps, dtype=DT[dtype], device=DEV)
        out = []
        for i in range(0, T, portion):
            n = min(portion, T - i)
            ctx = _Step([n], [0])
            ctx.positions += i
            out.append(ops.qk_prep(proj[i:i + n], 0, qn, qn + kn, nh, nkv, hd, vd, ctx, kc, vc, slots[i:i + n], ops.NORM_PER_HEAD, wq, wk, 1e-5, freq,
                                   ops.PAIRS_HALF_SPLIT))
        results.append((torch.cat(out), kc, vc))
    for other in results[1:]:
        for a, b in zip(results[0], other):
            assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T", [1, 3, 2050])
@pytest.mark.parametrize("hidden", [8, 520, 5120, 1032])
def test_embedding_by_runs(hidden, T, dtype):
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(T + hidden)
    table = torch.randn(300, hidden, generator=g).to(DT[dtype]).to(DEV)
    ids = torch.randint(0, 300, (T,), generator=g).to(torch.int32).to(DEV)
    assert torch.equal(ops.embed_gather(ids, table, scale=1.7), table[ids.long()].float() * 1.7)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("T", [9, 70])
@pytest.mark.parametrize("nh, hd", [(64, 128), (40, 192)])             # (more than 1,024 lanes: aligned rows are staged, too)
@pytest.mark.parametrize("form", ["whole", "whole conv", "whole conv3", "whole keys", "whole maps", "whole maps conv"])
@pytest.mark.parametrize("turn", ["none", "pairs", "halves"])
def test_aligned_rows_too_wide_for_runs(turn, form, nh, hd, T, dtype):
    _prepared_by_eights_and_one_by_one(turn, form, nh, 2, hd, T, dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("hd, r, vd, layout", [(128, 128, 128, 1), (128, 32, 128, 1), (32, 16, 32, 1), (64, 64, 64, 1), (256, 96, 256, 1), (256, 256, 256, 1),
                                               (64, 0, 64, 1), (128, 32, 40, 0), (64, 64, 72, 0), (256, 128, 8, 0), (32, 8, 24, 0), (128, 64, 72, 1)])
@pytest.mark.parametrize("T", [7, 70, 744, 746])       # (eleven heads: 8,184 and 8,206 waves, on both sides of the choice)
@pytest.mark.parametrize("norm", [True, False])
def test_rotated_heads_by_runs_give_the_bits_of_a_wave_a_head(norm, T, hd, r, vd, layout, dtype, nh=5, nkv=3):
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(hd + r + T)
    ps = 16
    width, pages = (nh + nkv) * hd + nkv * vd, T // ps + 3
    rows = torch.randn(T, width, generator=g).to(DT[dtype]).to(DEV)
    bias = torch.randn(width, generator=g).to(DEV)
    freq = torch.tensor([300.0 ** (-2.0 * i / r) for i in range(r // 2)], device=DEV) if r else None
    slots = torch.randperm(pages * ps, generator=g)[:T].to(torch.int32).to(DEV)
    pos, out = (torch.arange(T) * 7).to(torch.int32).to(DEV), []
    for extra in (0, 3):                 # (rows of another stride: a wave a head)
        qkv = torch.nn.functional.pad(rows, (0, extra)) if extra else rows
        kc = torch.zeros(pages, nkv, ps, hd, dtype=DT[dtype], device=DEV)
        vc = torch.zeros(pages, nkv, vd, ps, dtype=DT[dtype], device=DEV)
        out.append((ops.rope_kv(qkv, kc, vc, slots, pos, freq, norm, 1e-5, (40.0, 0.1), nh, nkv, hd, layout, bias, vd, extra), kc, vc))
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("hd, r, vd, layout", [(32, 16, 32, 1), (64, 64, 64, 1), (128, 32, 128, 1), (64, 0, 72, 0), (64, 64, 72, 0), (128, 128, 40, 0), (256, 96, 256, 1)])
@pytest.mark.parametrize("T", [190, 191])              # (43 heads: 8,170 and 8,213 waves)
def test_rotated_heads_of_wide_rows(T, hd, r, vd, layout, dtype):
    """Rows narrow beside a block's threads always go a wave a head; these do not."""
    test_rotated_heads_by_runs_give_the_bits_of_a_wave_a_head(True, T, hd, r, vd, layout, dtype, nh=29, nkv=7)


@pytest.mark.parametrize("maps", [2, 1])
def test_which_product_of_a_split_pairs_high_half_is_rounded(maps):
    """Several maps (the staged form by eights did them): the cosine's; plain heads: the sine's.  Computed in double from the kernel's own cosines and sines."""
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(maps)
    T, nh, nkv, hd, r, ps = 70, 4, 2, 128, 64, 16
    C, half, pages = (nh + 2 * nkv) * hd, r // 2, T // ps + 1
    freq = torch.tensor([300.0 ** (-2.0 * i / r) for i in range(half)], device=DEV)
    ctx, slots = _Step([T], [0]), torch.arange(T, dtype=torch.int32, device=DEV)

    def rotated(rows):
        kc = torch.zeros(pages, nkv, ps, hd, device=DEV)
        vc = torch.zeros(pages, nkv, hd, ps, device=DEV)
        ops.qk_prep(rows, 0, nh * hd, (nh + nkv) * hd, nh, nkv, hd, hd, ctx, kc, vc, slots, inv_freq=freq, pair_layout=ops.PAIRS_HALF_SPLIT, maps=maps)
        keys = kc.transpose(1, 2).reshape(pages * ps, nkv, maps, hd // maps)[:T]
        return keys[..., :half].double(), keys[..., half:r].double()

    unit = torch.zeros(T, C, device=DEV)
    unit[:, nh * hd:(nh + nkv) * hd].view(T, nkv, maps, hd // maps)[..., :half] = 1.0
    cos, sin = rotated(unit)
    rows = torch.randn(T, C, generator=g).to(DEV)
    low, high = rotated(rows)
    x = rows[:, nh * hd:(nh + nkv) * hd].view(T, nkv, maps, hd // maps).double()
    a, b = x[..., :half], x[..., half:r]
    rounded = lambda v: v.float().double()
    assert torch.equal(low, rounded(a * cos - rounded(b * sin)))
    assert torch.equal(high, rounded(a * sin + rounded(b * cos)) if maps > 1 else rounded(b * cos + rounded(a * sin)))
