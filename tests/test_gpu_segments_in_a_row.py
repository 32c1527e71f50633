"""Gated linear attention over entries of one to twenty segments: the states handed from segment to segment, eight requested at a time."""
import numpy as np
import pytest
import torch

from test_gpu_gla_chunk import inputs, recurrence, run, step

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("H, dk, dv", [(3, 64, 64), (2, 24, 20)])
@pytest.mark.parametrize("lens, slots", [([128 * 9 + 5, 3, 128 * 8], [2, 0, 1]), ([128 * 20], [1]), ([200, 128 * 16 + 1], [0, 2])])
def test_states_pass_through_every_segment(H, dk, dv, lens, slots):
    ctx = step(lens, slots)
    proj, alpha, state = inputs(lens, H, dk, dv, 8, torch.float32, 16.0, sum(lens))
    state = state if state.shape[0] > max(slots) else torch.cat([state, state])
    got, left = run(proj, alpha, state, ctx, H, dk, dv, 8)
    whole, whole_left = run(proj, alpha, state, ctx, H, dk, dv, 8, segmented=False)
    # two orders of the same float sums: each is within some 1e-6 of a result of order sqrt(dk) in 64 bits
    for a, b in ((got, whole), (left, whole_left)):
        assert float((a - b).abs().max()) <= 2e-5 * float(b.abs().max())
    e = int(np.argmax(lens))
    t0, t1 = int(ctx.cu[e]), int(ctx.cu[e + 1])
    q, k, v = (proj[t0:t1, 8 + o:8 + o + H * d].double().view(-1, H, d) for o, d in ((0, dk), (H * dk, dk), (2 * H * dk, dv)))
    if dk == 64:      # the state's layout is [ceil(dv / 8), rows, 8] with rows in the walk's order: from nothing here, so none has to be read
        empty = torch.zeros_like(state)
        out, _ = run(proj, alpha, empty, ctx, H, dk, dv, 8)
        want, _ = recurrence(q * dk ** -0.5, k, v, alpha[t0:t1].double().view(-1, H, dk), torch.zeros(H, dk, dv, dtype=torch.float64, device=DEV))
        assert float((out[t0:t1].double().view(-1, H, dv) - want).abs().max()) <= 2e-5 * float(want.abs().max())


@pytest.mark.parametrize("H, dk, dv", [(3, 64, 64), (2, 24, 20)])
def test_states_at_any_address(H, dk, dv):
    from sharpinference_amd import ops

    lens, slots = [128 * 9 + 5, 3, 128 * 2], [2, 0, 1]
    ctx = step(lens, slots)
    proj, alpha, state = inputs(lens, H, dk, dv, 8, torch.float32, 16.0, sum(lens))
    segments = tuple(torch.from_numpy(x).to(DEV) for x in ops.gla_segments(lens, ctx.cu))
    results = []
    for first in (0, 1, 2):              # (elements from a multiple of 16 bytes on)
        held = torch.zeros(state.numel() + first, device=DEV)[first:].view(state.shape)
        held.copy_(state)
        o = ops.gla_walk(proj, 8, 8 + H * dk, 8 + 2 * H * dk, alpha, dk ** -0.5, held, ctx, H, dk, dv, segments=segments)
        results.append((o, held))
    for a, b in zip(*results[1:]):       # (both are walked)
        assert torch.equal(a, b)
    for a, b in zip(*results[:2]):       # (the first in products where the sizes allow it: the bound of the two orders above)
        assert float((a - b).abs().max()) <= 2e-5 * float(b.abs().max())
