"""Runs of shared rows merged by a wave a row and by waves of 256 elements."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T, H, R, runs", [(1, 3, 4, 5), (5, 5, 252, 5), (3, 7, 260, 4), (3, 7, 260, 5), (2, 6, 512, 9), (2, 1, 512, 70), (1, 3, 1100, 6)])
def test_the_runs_merged(T, H, R, runs):
    from sharpinference_amd import ops

    g = torch.Generator().manual_seed(R + runs)
    o, ml = torch.randn(T, H, runs, R, generator=g), torch.rand(T, H, runs, 2, generator=g) + 0.5
    seen = torch.tensor([1 + (runs - 1 + t) % (runs + 1) for t in range(T)])      # runs of each token, the first all, the second one too many
    pos, sink = (seen * 64 - 1).to(torch.int32), torch.randn(H, generator=g)
    out = torch.zeros(T, H * R, dtype=torch.bfloat16, device=DEV)
    dev = [t.to(DEV) for t in (o, ml, pos, sink)]
    ops._run("sharpi_attention_latent_merge", ops._ptr(dev[0]), ops._ptr(dev[1]), ops._ptr(dev[2]), None, T, ops._ptr(dev[3]), ops._ptr(out), H, R, 64, runs, 0,
             ops._stream())
    got = out.cpu().double().view(T, H, R)
    for t in range(T):
        n = int(seen[t])
        if n > runs:
            assert bool(got[t].isnan().all())               # sized for fewer keys than the token sees
        elif n == 1:
            assert bool((got[t] == 0).all())                # nothing to merge: whoever made the run stored the result
        else:
            w = torch.exp(ml[t, :, :n, 0].double())
            want = (o[t, :, :n].double() * w[..., None]).sum(1) / ((w * ml[t, :, :n, 1].double()).sum(1) + torch.exp(sink.double()))[:, None]
            room = (o[t, :, :n].double().abs() * w[..., None]).sum(1) / ((w * ml[t, :, :n, 1].double()).sum(1) + torch.exp(sink.double()))[:, None]
            # one rounding to 8 bits; weights and sums in 24 bits (an exponential within four places, a place a run)
            assert bool(((got[t] - want).abs() <= want.abs() * 2.0 ** -8 + room * (2 * n + 16) * 2.0 ** -23).all())
