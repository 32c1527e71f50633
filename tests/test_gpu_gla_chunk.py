"""Gated linear attention's segments as matrix products: against the recurrence in 64 bits, no further from it than the walk, at
the edges of blocks of 16 tokens and of segments, with decays of 0, of 1 and near 1, and with values that are no number, which stay with their
token and later ones."""
import types

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def recurrence(q, k, v, alpha, S):
    out = []
    for t in range(q.shape[0]):
        S = alpha[t][:, :, None] * S + k[t][:, :, None] * v[t][:, None, :]
        out.append((S * q[t][:, :, None]).sum(1))
    return torch.stack(out), S


def step(lens, slots):
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    return types.SimpleNamespace(n_entries=len(lens), n_tokens=int(cu[-1]), max_entry_len=max(lens), cu=cu,
                                 state_slots=torch.tensor(slots, dtype=torch.int32, device=DEV), cu_tokens=torch.from_numpy(cu).to(DEV))


def run(proj, alpha, state, ctx, H, dk, dv, pad, segmented=True):
    from sharpinference_amd import ops
    lens = np.diff(ctx.cu).tolist()
    segments = tuple(torch.from_numpy(x).to(DEV) for x in ops.gla_segments(lens, ctx.cu)) if segmented else None
    state = state.clone()
    o = ops.gla_walk(proj, pad, pad + H * dk, pad + 2 * H * dk, alpha, dk ** -0.5, state, ctx, H, dk, dv, segments=segments)
    return o, state


def inputs(lens, H, dk, dv, pad, dtype, tau, seed, decay=None):
    from sharpinference_amd import ops
    g = torch.Generator(device=DEV).manual_seed(seed)
    T = sum(lens)
    proj = torch.randn(T, pad + H * (2 * dk + dv) + 8, device=DEV, generator=g).to(dtype)
    alpha = torch.sigmoid(2 * torch.randn(T, H * dk, device=DEV, generator=g) + 1) ** (1 / tau)
    some = torch.rand(T, H * dk, device=DEV, generator=g)
    alpha = torch.where(some < 0.01, torch.zeros_like(alpha), torch.where(some > 0.99, torch.ones_like(alpha), alpha))
    if decay is not None:
        alpha = torch.full_like(alpha, decay)
    state = torch.randn(len(lens) + 1, *ops.gla_state_shape(H, dk, dv), device=DEV, generator=g)
    return proj, alpha.contiguous(), state


def errors_of(proj, alpha, state, ctx, H, dk, dv, pad):
    """Of the products and of the segments walked (the same numbers in rows that lie off the borders the products need): outputs' and
    states' distances from 64 bits, over the results' root mean square."""
    from sharpinference_amd import ops
    lens = np.diff(ctx.cu).tolist()
    got, left = run(proj, alpha, state, ctx, H, dk, dv, pad)
    moved = torch.cat([proj[:, 5:], proj[:, :5]], 1).contiguous()
    walk, walk_left = run(moved, alpha, state, ctx, H, dk, dv, pad - 5)
    assert torch.equal(left[0], state[0])                                # nobody's slot
    p = proj.double()
    part = lambda a, n: p[:, a:a + H * n].reshape(-1, H, n)
    q, k, v, a = part(pad, dk) * dk ** -0.5, part(pad + H * dk, dk), part(pad + 2 * H * dk, dv), alpha.double().view(-1, H, dk)
    S0 = ops.gla_state_matrices(state, dk, dv).double()
    errors = np.zeros((2, 2))
    for e in range(len(lens)):
        rows = slice(int(ctx.cu[e]), int(ctx.cu[e + 1]))
        want, S = recurrence(q[rows], k[rows], v[rows], a[rows], S0[e + 1])
        for i, (o, st) in enumerate(((got, left), (walk, walk_left))):
            errors[i] += [float((o[rows].double().view(want.shape) - want).pow(2).sum() / want.pow(2).mean()),
                          float((ops.gla_state_matrices(st[e + 1:e + 2], dk, dv)[0].double() - S).pow(2).sum() / S.pow(2).mean())]
    return np.sqrt(errors / np.array([got.numel(), len(lens) * H * dk * dv]))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H, dk, dv, tau", [(2, 128, 128, 16.0), (3, 64, 128, 1.0), (1, 128, 64, 0.3), (2, 64, 64, 40.0), (1, 128, 128, 200.0)])
@pytest.mark.parametrize("lens", [[128], [1, 15, 16, 17], [129, 2], [33, 127, 260], [400]])
def test_segments_as_products_are_no_further_from_64_bits_than_the_walk(dtype, H, dk, dv, tau, lens):
    pad = 8
    proj, alpha, state = inputs(lens, H, dk, dv, pad, dtype, tau, sum(lens) + dk)
    ours, walks = errors_of(proj, alpha, state, step(lens, [i + 1 for i in range(len(lens))]), H, dk, dv, pad)
    assert (ours <= walks).all(), (ours, walks)


@pytest.mark.parametrize("lens", [[128], [1900]])
@pytest.mark.parametrize("loss", [1e-4, 2e-4, 3e-4, 1.3e-3, 1e-2])
def test_equal_decays_near_one_are_no_further_from_64_bits_than_the_walk(loss, lens):
    """Products of equal floats 1 - a all round to one side: what is lost adds up from token to token and from segment to segment."""
    H, dk, dv, pad = 1, 128, 64, 8
    proj, alpha, state = inputs(lens, H, dk, dv, pad, torch.bfloat16, 1.0, 11, decay=1 - loss)
    ours, walks = errors_of(proj, alpha, state, step(lens, [1]), H, dk, dv, pad)
    assert (ours <= walks).all(), (ours, walks)


@pytest.mark.parametrize("what", ["v", "k", "q", "alpha"])
@pytest.mark.parametrize("at", [3, 40, 127, 128, 200])
def test_what_is_no_number_stays_with_its_token_and_later_ones(what, at):
    H, dk, dv, pad, lens = 2, 128, 64, 8, [260, 20]
    proj, alpha, state = inputs(lens, H, dk, dv, pad, torch.bfloat16, 16.0, 5)
    ctx = step(lens, [0, 1])
    clean, left = run(proj, alpha, state, ctx, H, dk, dv, pad)
    for bad in (float("inf"), float("nan")):
        p, a = proj.clone(), alpha.clone()
        if what == "alpha":
            a[at, 7] = bad
        else:
            p[at, pad + {"q": 0, "k": H * dk, "v": 2 * H * dk}[what] + 7] = bad
        o, st = run(p, a, state, ctx, H, dk, dv, pad)
        assert torch.equal(o[:at], clean[:at]) and torch.equal(o[260:], clean[260:])
        assert torch.equal(o[:, dv:], clean[:, dv:])                     # the other head
        assert not bool(o[at, :dv].isfinite().all())
        assert torch.equal(st[1], left[1]) and (what == "q") == bool(st[0].isfinite().all())


def test_rows_off_the_borders_are_walked():
    H, dk, dv, lens = 2, 64, 64, [300]
    proj, alpha, state = inputs(lens, H, dk, dv, 8, torch.bfloat16, 4.0, 9)
    ctx = step(lens, [0])
    want, left = run(proj, alpha, state, ctx, H, dk, dv, 8)
    got, st = run(torch.cat([proj[:, 5:], proj[:, :5]], 1).contiguous(), alpha, state, ctx, H, dk, dv, 3)
    assert float((got - want).abs().max()) <= 1e-5 * float(want.abs().max()) and float((st - left).abs().max()) <= 1e-5 * float(left.abs().max())


@pytest.mark.parametrize("H, dk, dv", [(2, 128, 64), (1, 64, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("cuts", [[[129]], [[300], [0], [7]], [[128, 257, 31], [1]], [[400, 16], [128]]])
def test_a_callers_own_segments_may_be_longer_than_a_chunk(cuts, dtype, H, dk, dv):
    """Lists that ops.gla_segments would not make: segments of more tokens than a chunk, and of none."""
    from sharpinference_amd import ops
    lens, pad = [sum(c) for c in cuts], 8
    proj, alpha, state = inputs(lens, H, dk, dv, pad, dtype, 16.0, sum(lens))
    ctx = step(lens, list(range(len(lens))))
    segs, ents = [], []
    for e, c in enumerate(cuts):
        ents.append((len(segs), len(c)))
        for n, m in enumerate(c):
            segs.append((e, int(ctx.cu[e]) + sum(c[:n]), m, int(n == len(c) - 1)))
    lists = tuple(torch.tensor(x, dtype=torch.int32, device=DEV) for x in (segs, ents))
    left = state.clone()
    got = ops.gla_walk(proj, pad, pad + H * dk, pad + 2 * H * dk, alpha, dk ** -0.5, left, ctx, H, dk, dv, segments=lists)
    want, want_left = run(proj, alpha, state, ctx, H, dk, dv, pad, segmented=False)
    # both within 4e-7 of 64 bits (above), the largest of some thousand differences within 6 times that
    for a, b in ((got, want), (left, want_left)):
        assert float((a - b).abs().max()) <= 5e-6 * float(b.pow(2).mean().sqrt())
    assert torch.equal(left[len(lens)], state[len(lens)])                # nobody's slot
    for e, n in enumerate(lens):
        if n == 0:
            assert torch.equal(left[e], state[e])
