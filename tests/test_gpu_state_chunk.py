"""Long entries through a recurrent state with one decay a head, run as matrix products over segments, against the
recurrence in 64 bits."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}


class _Step:
    def __init__(self, lens, starts, slots):
        self.n_entries, self.n_tokens = len(lens), sum(lens)
        cu = np.concatenate([[0], np.cumsum(lens)])
        self.lens, self.cu = lens, cu
        self.cu_tokens = torch.tensor(cu, dtype=torch.int32, device=DEV)
        self.state_slots = torch.tensor(slots, dtype=torch.int32, device=DEV)
        self.positions = torch.cat([torch.arange(s, s + n) for s, n in zip(starts, lens)]).to(torch.int32).to(DEV)


def _recurrence(mode, q, k, v, gates, par, cap, freqs, k_scale):
    """Token by token in 64 bits: q, k [T, G, d], v [T, H, e] -> (o [T, H, e], S [H, d, e])."""
    T, H, e = v.shape
    q, k = (t.repeat_interleave(H // t.shape[1], 1) for t in (q, k))
    S, n, m = torch.zeros(H, q.shape[2], e, dtype=torch.float64), torch.zeros(H, q.shape[2], dtype=torch.float64), torch.zeros(H, dtype=torch.float64)
    out = torch.zeros(T, H, e, dtype=torch.float64)
    if freqs is not None:
        half = freqs.shape[0]
        ang = (torch.arange(T, dtype=torch.float32)[:, None] * freqs[None]).double()[:, None]       # (the angle is a float product)
        turn = lambda x: torch.cat([x[..., :half] * ang.cos() - x[..., half:2 * half] * ang.sin(),
                                    x[..., half:2 * half] * ang.cos() + x[..., :half] * ang.sin(), x[..., 2 * half:]], -1)
        q, k = turn(q), turn(k)
    for t in range(T):
        if mode == "gates":
            i, f = (cap * torch.tanh((gates[t, a:a + H] + p) / cap) for a, p in ((0, par[0]), (H, par[1])))
            f = torch.nn.functional.logsigmoid(f)
            new = torch.maximum(f + m, i)
            a, b, m = torch.exp(f + m - new), torch.exp(i - new), new
            n = a[:, None] * n + b[:, None] * k[t]
        elif mode == "space":
            b = torch.nn.functional.softplus(gates[t, :H] + par[0])
            a = torch.exp(-torch.exp(par[1]) * b)
        else:
            a, b = par[0], torch.full((H,), k_scale, dtype=torch.float64)
        S = a[:, None, None] * S + (b[:, None] * k[t])[:, :, None] * v[t][:, None]
        out[t] = (S * q[t][:, :, None]).sum(1)
        if mode == "gates":
            out[t] /= (torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-m)) + 1e-6)[:, None]
        elif mode == "space":
            out[t] += par[2][:, None] * v[t]
    return out, S


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("mode, H, G, dk, dv", [("gates", 2, 2, 128, 128), ("gates", 3, 3, 64, 64), ("space", 4, 2, 128, 64),
                                               ("space", 2, 1, 64, 128), ("fixed", 2, 2, 128, 128), ("fixed", 2, 2, 64, 64)])
def test_segments_as_matrix_products_are_as_exact_as_the_walk(dtype, mode, H, G, dk, dv):
    """Entries at the edges of segments (128 tokens) and of tiles (16), single tokens among them, from states that earlier
    steps left: outputs and states against the recurrence in 64 bits, over all entries together no further off than 1.1
    times what the token-by-token walk of the same rows is.  (One entry's few rows say little by themselves: where n . q
    cancels, a row's error is that of its sums over a small remainder, whichever way they are ordered; an entry alone is
    held to 1e-5, a hundred roundings of its largest term.)"""
    from sharpinference_amd import ops

    assert ops.walk_takes_chunks(dk, dv)
    g = torch.Generator().manual_seed(dk + dv + H)
    code = {"gates": ops.WALK_EXP_GATES, "space": ops.WALK_STATE_SPACE, "fixed": ops.WALK_FIXED_DECAY}[mode]
    before, lens, slots = [3, 0, 17, 1, 0, 130, 2], [300, 128, 1, 129, 15, 16, 257], [2, 0, 3, 6, 5, 1, 7]
    cap, k_scale = 8.0, (dk ** -0.5 if mode == "fixed" else 1.0)
    q_scale = dk ** -0.5 if mode == "gates" else 1.0
    freqs = 10000.0 ** (-torch.arange(dk // 4, dtype=torch.float32) / (dk // 4)) if mode == "fixed" else None
    par = {"gates": (torch.randn(H, generator=g), torch.randn(H, generator=g)),
           "space": (torch.randn(H, generator=g) * 0.5, torch.randn(H, generator=g) * 0.5 - 1.0, torch.randn(H, generator=g)),
           "fixed": (1.0 - 2.0 ** (-3.0 - torch.arange(H) * 4.0),)}[mode]
    rows = [torch.randn(b + n, 2 * G * dk + H * dv, generator=g).to(DT[dtype]) for b, n in zip(before, lens)]
    gates = [torch.randn(b + n, 2 * H, generator=g) * 2.0 + (torch.tensor([0.0] * H + [3.0] * H) if mode == "gates" else -2.0)
             for b, n in zip(before, lens)]

    def run(segmented):
        state = torch.zeros(9, *ops.walk_state_shape(H, dk, dv, code), device=DEV)
        got = None
        for part in (0, 1):
            ns, at = (before, [0] * len(lens)) if part == 0 else (lens, before)
            live = [i for i, n in enumerate(ns) if n > 0]
            ctx = _Step([ns[i] for i in live], [at[i] for i in live], [slots[i] for i in live])
            segments = None
            if segmented and part:
                segments = tuple(torch.from_numpy(x).to(DEV) for x in ops.gla_segments(ctx.lens, ctx.cu))
            x = torch.cat([rows[i][at[i]:at[i] + ns[i]] for i in live]).to(DEV)
            z = torch.cat([gates[i][at[i]:at[i] + ns[i]] for i in live]).to(DEV) if mode != "fixed" else None
            got = ops.state_walk(x, 0, G * dk, 2 * G * dk, H // G, z, tuple(p.to(DEV) for p in par), cap, q_scale, code, state, ctx, H, dk, dv,
                                 segments=segments, inv_freq=freqs.to(DEV) if freqs is not None else None, k_scale=k_scale)
        return got.cpu().double(), state

    (chunk, chunk_state), (walk, walk_state) = run(True), run(False)
    at, errors = 0, {"outputs": [], "states": []}
    for i, (b, n) in enumerate(zip(before, lens)):
        x = rows[i].double()
        q, k = x[:, :G * dk].reshape(-1, G, dk) * q_scale, x[:, G * dk:2 * G * dk].reshape(-1, G, dk)
        want, S = _recurrence(mode, q, k, x[:, 2 * G * dk:].reshape(-1, H, dv), gates[i].double(), [p.double() for p in par], cap, freqs, k_scale)
        want = want[b:].reshape(n, -1)
        rel = lambda got, ref: float((got - ref).norm() / ref.norm())
        errors["outputs"].append((rel(chunk[at:at + n], want), rel(walk[at:at + n], want)))
        s_chunk, s_walk = (ops.walk_state_matrices(s[slots[i]], dk, dv, code) for s in (chunk_state, walk_state))
        errors["states"].append(tuple(rel(s[0].cpu().double(), S) for s in (s_chunk, s_walk)))
        for a, w in zip(s_chunk[1:], s_walk[1:]):
            if a is not None:
                assert float((a - w).abs().max()) <= 1e-5 * float(w.abs().max() + 1)
        at += n
    for what, pairs in errors.items():
        e_chunk, e_walk = (float(np.sqrt(np.mean([p[j] ** 2 for p in pairs]))) for j in (0, 1))
        print(mode, dtype, what, f"chunks {e_chunk:.2e} walk {e_walk:.2e}")
        assert e_chunk <= 1.1 * e_walk and max(p[0] for p in pairs) < 1e-5, (what, pairs)
    if mode == "gates":                                            # every slice keeps a copy of the normaliser and the maximum
        tail = chunk_state[slots][:, :, :, dk * 8:dk * 8 + dk + 1]
        assert torch.equal(tail, tail[:, :, :1].expand_as(tail))
    assert float(chunk_state[[4, 8]].abs().max()) == 0.0           # slots no entry names


def _modes(mode, H, dk, g):
    """(code, parameters, frequencies, keys' scale) of a mode, as the layers that walk such states have them."""
    from sharpinference_amd import ops

    code = {"gates": ops.WALK_EXP_GATES, "space": ops.WALK_STATE_SPACE, "fixed": ops.WALK_FIXED_DECAY}[mode]
    par = {"gates": (torch.randn(H, generator=g), torch.randn(H, generator=g)),
           "space": (torch.randn(H, generator=g) * 0.5, torch.randn(H, generator=g) * 0.5 - 1.0, torch.randn(H, generator=g)),
           "fixed": (1.0 - 2.0 ** (-3.0 - torch.arange(H) * 4.0),)}[mode]
    freqs = 10000.0 ** (-torch.arange(dk // 4, dtype=torch.float32) / (dk // 4)) if mode == "fixed" else None
    return code, tuple(p.to(DEV) for p in par), freqs.to(DEV) if freqs is not None else None, dk ** -0.5 if mode == "fixed" else 1.0


def _walk(mode, lens, rows, gates, modes, H, dk, dv, segmented=True, state=None):
    from sharpinference_amd import ops

    code, par, freqs, k_scale = modes
    ctx = _Step(lens, [0] * len(lens), range(len(lens)))
    segments = tuple(torch.from_numpy(x).to(DEV) for x in ops.gla_segments(ctx.lens, ctx.cu)) if segmented else None
    state = torch.zeros(len(lens), *ops.walk_state_shape(H, dk, dv, code), device=DEV) if state is None else state
    out = ops.state_walk(rows, 0, H * dk, 2 * H * dk, 1, gates, par, 8.0, dk ** -0.5, code, state, ctx, H, dk, dv,
                         segments=segments, inv_freq=freqs, k_scale=k_scale)
    return out.view(-1, H, dv), state


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("mode, dk, dv", [("gates", 128, 128), ("space", 128, 64), ("fixed", 64, 128)])
def test_what_is_no_number_stays_with_its_token_and_later_ones(dtype, mode, dk, dv):
    """A token's value, key, query or gate that is infinite or no number: tokens before it have the same bits as without it,
    whichever tile and segment they share with it; a value spoils one output column alone, from its token on."""
    g = torch.Generator().manual_seed(dk + dv)
    H, lens = 2, [300, 40]
    n = sum(lens)
    modes = _modes(mode, H, dk, g)
    rows = torch.randn(n, 2 * H * dk + H * dv, generator=g).to(DT[dtype]).to(DEV)
    gates = torch.randn(n, 2 * H, generator=g).to(DEV) if mode != "fixed" else None
    clean = _walk(mode, lens, rows, gates, modes, H, dk, dv)[0]
    v_col = lambda h, c: 2 * H * dk + h * dv + c
    for bad in (float("inf"), float("nan")):
        for t, h, c in ((5, 0, 17), (141, 1, dv - 1), (287, 0, 0), (299, 1, 33), (333, 0, 1)):
            x = rows.clone()
            x[t, v_col(h, c)] = bad
            got = _walk(mode, lens, x, gates, modes, H, dk, dv)[0]
            spoilt = torch.zeros_like(clean, dtype=torch.bool)
            spoilt[t:300 if t < 300 else n, h, c] = True
            assert torch.equal(got[~spoilt], clean[~spoilt])
            assert not bool(got[spoilt].isfinite().any())
        for t in (6, 141, 287, 333):
            for what in ("key", "query", "gate"):
                x, z = rows.clone(), gates
                if what == "gate":
                    if gates is None:
                        continue
                    z = gates.clone()
                    z[t, 0] = bad
                else:
                    x[t, 3 if what == "query" else H * dk + 3] = bad
                got = _walk(mode, lens, x, z, modes, H, dk, dv)[0]
                assert torch.equal(got[:t], clean[:t]) and torch.equal(got[:, 1], clean[:, 1])



@pytest.mark.parametrize("mode", ["space", "fixed"])
def test_decays_of_zero_forget_what_was_before(mode):
    """A step size so large, or a stored decay, that a token's decay is 0: its logarithm is minus infinity, what follows is what
    the walk of the whole entry makes of it, here and in the state that is left."""
    g = torch.Generator().manual_seed(11)
    H, dk, dv, lens = 2, 128, 64, [300, 90]
    modes = list(_modes(mode, H, dk, g))
    rows = torch.randn(sum(lens), 2 * H * dk + H * dv, generator=g).to(DEV)
    gates = None
    if mode == "space":
        gates = torch.randn(sum(lens), 2 * H, generator=g).to(DEV)
        modes[1][1][0] = 100.0                                     # exp(100) is beyond float: every decay of the head is 0
        modes[1][1][1] = 60.0                                      # 1e26: finite logarithms, decays of 0 where the step is not tiny
    else:
        modes[1][0][0] = 0.0
    (got, state), (want, walked) = (_walk(mode, lens, rows, gates, modes, H, dk, dv, s) for s in (True, False))
    # an output is one product of 128 and two of a head's own sums: a few roundings of the largest
    assert float((got - want).abs().max()) <= 2e-6 * float(want.abs().max())
    assert float((state - walked).abs().max()) <= 2e-6 * float(walked.abs().max())



def test_scratch_is_for_entries_of_several_segments_alone():
    """200 decoding requests beside one prompt of three segments: what is allocated beside the outputs are two states a
    segment of the prompt."""
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(3)
    H, dk, dv, lens = 4, 128, 128, [1] * 100 + [300] + [1] * 100
    modes = _modes("fixed", H, dk, g)
    rows = torch.randn(sum(lens), 3 * H * dk, generator=g).to(DEV)
    state = torch.zeros(len(lens), *ops.walk_state_shape(H, dk, dv, ops.WALK_FIXED_DECAY), device=DEV)
    code, par, freqs, k_scale = modes
    ctx = _Step(lens, [0] * len(lens), range(len(lens)))
    segs, ents = ops.gla_segments(ctx.lens, ctx.cu)
    segments = (torch.from_numpy(segs).to(DEV), torch.from_numpy(ents).to(DEV), ops.segment_counts(lens))
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    out = ops.state_walk(rows, 0, H * dk, 2 * H * dk, 1, None, par, 8.0, dk ** -0.5, code, state, ctx, H, dk, dv, segments=segments,
                         inv_freq=freqs, k_scale=k_scale)
    one = state[0].numel() * 4
    # (the allocator leaves up to a MiB behind a large tensor in its block; a place for every segment would be 106 MB)
    assert torch.cuda.max_memory_allocated() - before <= out.numel() * 4 + 2 * 3 * one + (1 << 20)
    want, walked = _walk("fixed", lens, rows, None, modes, H, dk, dv, False)
    assert float((out.view_as(want) - want).abs().max()) <= 2e-6 * float(want.abs().max())
    assert float((state - walked).abs().max()) <= 2e-6 * float(walked.abs().max())


@pytest.mark.parametrize("pad, lens", [(0, [20]), (0, [100]), (0, [300]), (0, [128, 31]), (3, [300, 20, 1])])
def test_one_entry_alone_and_rows_that_cannot_be_read_in_sixteen_bytes(pad, lens):
    """One entry below the chunk form's tokens, of one segment, of several; rows of odd strides take the walk in segments."""
    g = torch.Generator().manual_seed(sum(lens))
    H, dk, dv = 2, 128, 128
    modes = _modes("gates", H, dk, g)
    rows = torch.randn(sum(lens), 3 * H * dk + pad, generator=g).to(torch.bfloat16).to(DEV)
    gates = torch.randn(sum(lens), 2 * H, generator=g).to(DEV)
    (got, state), (want, walked) = (_walk("gates", lens, rows, gates, modes, H, dk, dv, s) for s in (True, False))
    assert float((got - want).norm() / want.norm()) < 1e-5
    assert float((state - walked).abs().max()) <= 1e-5 * float(walked.abs().max() + 1)
