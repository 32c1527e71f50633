"""Prompt portions over expanded keys and values against the shared latent rows and the plain models in 64 bits."""
import pytest
import torch

import plain_pagonex
import plain_rigodra

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _tokens(n, vocab, seed):
    return torch.randint(vocab, (n,), generator=torch.Generator().manual_seed(seed)).tolist()


@pytest.mark.parametrize("H, dn, dr, dv, R, page", [(2, 64, 32, 64, 64, 16), (3, 128, 64, 128, 512, 16), (1, 64, 32, 64, 320, 48), (2, 128, 32, 64, 128, 32)])
def test_expanded_keys_and_values_are_the_products(H, dn, dr, dv, R, page):
    """Pages that begin and end inside a sequence, entries of one key, pages of the cache in any order; keys that are not
    there hold the nearest one's values.  Bound: a chain of R products and one rounding to bfloat16."""
    from types import SimpleNamespace

    from sharpinference_amd import ops

    if not ops.latent_expand_ok(torch.bfloat16, dn, dr, dv, R):
        pytest.skip("no flash kernel of these widths")
    g = torch.Generator().manual_seed(R + H)
    spans = [(0, 300), (130, 131), (0, 1), (5, 257), (256, 384)]
    n_pages = 60
    rows = torch.randn(n_pages, 1, page, R + dr, generator=g).to(torch.bfloat16).to(DEV)
    per = (384 + page - 1) // page
    order = torch.randperm(n_pages, generator=g)
    table = torch.stack([order[torch.arange(per) + (5 * e) % (n_pages - per)] for e in range(len(spans))]).to(torch.int32)
    for e, (lo, _) in enumerate(spans):
        table[e, :lo // page] = -1                                # pages behind a window went back
    listed = [(e, b, lo, hi) for e, (lo, hi) in enumerate(spans) for b in range(lo // 128, (hi - 1) // 128 + 1)]
    w = (torch.randn(H, dn + dv, R, generator=g) * R ** -0.5).to(torch.bfloat16).to(DEV)
    k, v = ops.latent_expand(rows, SimpleNamespace(block_table=table.to(DEV)), torch.tensor(listed, dtype=torch.int32, device=DEV), w, dn, dr, dv, R)
    flat, wd = rows.double().reshape(-1, R + dr), w.double()
    for i, (e, b, lo, hi) in enumerate(listed):
        keys = (torch.arange(128) + 128 * b).clamp(lo, hi - 1)
        at = (table[e][keys // page].long() * page + keys % page).to(DEV)
        c, turned = flat[at][:, :R], rows.reshape(-1, R + dr)[at][:, R:]
        both = torch.einsum("kr,hnr->hkn", c, wd)
        bound = torch.einsum("kr,hnr->hkn", c.abs(), wd.abs()) * R * 2.0 ** -24 + both.abs() * 2.0 ** -8
        assert bool(((k[i][..., :dn].double() - both[..., :dn]).abs() <= bound[..., :dn]).all())
        assert bool(((v[i].double().transpose(1, 2) - both[..., dn:]).abs() <= bound[..., dn:]).all())
        assert torch.equal(k[i][..., dn:], turned[None].expand(H, -1, -1))


def _latent_only(name):
    """Small models of latent attention alone (no router whose choice could fall either way)."""
    mixer = {"heads": 4, "dim": 64, "rot_dim": 32, "vdim": 64, "kv_rank": 128, "scale": 96 ** -0.5, "rot": {"base": 1000.0, "dims": 32}}
    if name == "rigodra":                                          # every key in sight, pairs in two halves
        layers = [dict(mixer, q_rank=64, rot={"base": 1000.0, "dims": n}) for n in (32, 16, 32)]
        return {"architecture": "Rigodra", "vocab": 128, "width": 128, "norm": {"eps": 1e-5}, "postln_alpha": 1.7,
                "layers": [{"type": "latent_attention", "mixer": m, "mlp": None} for m in layers]}
    layers = [dict(mixer, q_rank=64, mask={"size": s}) for s in (96, 40, 300)]      # windows
    return {"architecture": "Pagonex", "vocab": 128, "width": 128, "norm": {"eps": 1e-5}, "logit_scale": 1.0, "canon": {"taps": 2},
            "layers": [{"type": "latent_attention", "mixer": m, "mlp": None} for m in layers]}


@pytest.mark.parametrize("name, plain", [("rigodra", plain_rigodra), ("pagonex", plain_pagonex)])
def test_prompts_over_expanded_keys_are_as_exact_as_over_the_shared_rows(name, plain, tmp_path, monkeypatch):
    """Portions of 33 to 200 tokens, alone, beside each other and beside decoding requests (side by side, and scattered, which
    keeps to the shared rows), first portions and later ones: every row of logits against the plain model in 64 bits, both
    ways.  The two round in different places, so a row may be further off one way; over all rows the expanded
    form's error is held to 1.05 times the other's."""
    from sharpinference_amd import load_config
    from sharpinference_amd.engine import Engine, StepEntry
    from sharpinference_amd.parts import latent_attention as L
    from sharpinference_amd.weights.loader import write_random_model

    cfg, d = _latent_only(name), str(tmp_path / name)
    write_random_model(load_config(cfg), d, 7, std=0.1, std_by_suffix={"embed": 1.0})
    reqs = {r: _tokens(n, 128, i) for i, (r, n) in enumerate({"a": 345, "b": 64, "c": 233, "d": 40}.items())}
    steps = [[("a", 130), ("b", 33)], [("b", 1), ("c", 200)], [("b", 1), ("a", 129), ("c", 1)], [("b", 1), ("c", 1), ("d", 37), ("a", 70)],
             [("d", 1), ("a", 1), ("b", 1), ("c", 1)], [("a", 15), ("c", 30), ("d", 2)], [("b", 26)]]
    expanded = []
    real = L.LatentAttention._attend_expanded
    monkeypatch.setattr(L.LatentAttention, "_attend_expanded", lambda self, *a: expanded.append(1) or real(self, *a))

    def run(least):
        monkeypatch.setattr(L, "EXPAND_FROM_TOKENS", least)
        monkeypatch.setattr(L, "EXPAND_FROM_PAIRS", 0)             # (steps this small would not pay)
        eng = Engine(d, dtype="bfloat16", max_num_seqs=4, kv_tokens=1200, max_model_len=512, max_tokens_per_step=512, decode_graphs=False)
        got, at = {r: [] for r in reqs}, {r: 0 for r in reqs}
        for r in reqs:
            eng.add_request(r)
        for step in steps:
            o = eng.step([StepEntry(r, reqs[r][at[r]:at[r] + n], tuple(range(n))) for r, n in step]).cpu()
            i = 0
            for r, n in step:
                got[r].append(o[i:i + n])
                i += n
                at[r] += n
        return {r: torch.cat(v).double() for r, v in got.items()}

    new, shared = run(32), None
    # three layers in the first, second and fourth step (the third's single tokens are scattered); in the fourth the layer
    # with a window of 40 sees too few keys a query to pay
    assert len(expanded) == (9 if name == "rigodra" else 8)
    expanded.clear()
    shared = run(1 << 30)
    assert not expanded
    raw, w = plain.read_config(d), plain.load_weights(d, torch.float64)
    errs = []
    for r, toks in reqs.items():
        n = new[r].shape[0]
        want = plain.forward(raw, w, toks[:n]).double()
        errs.append(torch.stack([(x[r] - want).norm(dim=-1) / want.norm(dim=-1) for x in (new, shared)]))
    e_new, e_shared = torch.cat(errs, dim=1).pow(2).mean(dim=1).sqrt().tolist()
    print(f"{name}: expanded {e_new:.3e} shared {e_shared:.3e}")
    assert e_new <= 1.05 * e_shared and float(torch.cat(errs, dim=1)[0].max()) < 0.1


@pytest.mark.parametrize("name, plain", [("rigodra", plain_rigodra), ("pagonex", plain_pagonex)])
def test_portions_left_out_of_the_expansion_keep_to_the_shared_rows(name, plain, tmp_path, monkeypatch):
    """Portions of few tokens, as those that would lose by an expansion of a long context, before, between and behind
    portions that are expanded, beside each other, and beside decoding requests: every row of logits against the plain model
    in 64 bits, held to what the shared rows alone give (1.05 times over all rows: the two round in different places)."""
    from sharpinference_amd import load_config
    from sharpinference_amd.engine import Engine, StepEntry
    from sharpinference_amd.parts import latent_attention as L
    from sharpinference_amd.weights.loader import write_random_model

    cfg, d = _latent_only(name), str(tmp_path / name)
    write_random_model(load_config(cfg), d, 7, std=0.1, std_by_suffix={"embed": 1.0})
    reqs = {r: _tokens(300, 128, i) for i, r in enumerate("abcdef")}
    steps = [[("a", 9), ("b", 130), ("c", 5), ("d", 20)], [("e", 1), ("f", 1), ("a", 70), ("c", 100), ("b", 17), ("d", 140)],
             [("b", 150), ("e", 2), ("c", 120), ("a", 30), ("f", 40)], [("a", 1), ("d", 60), ("b", 1), ("c", 1), ("e", 19)]]
    left_out = []
    real = L.LatentAttention._attend_shared
    monkeypatch.setattr(L.LatentAttention, "_attend_shared", lambda self, q, *a: left_out.append(q.shape[0]) or real(self, q, *a))
    monkeypatch.setattr(L, "_few_queries_lose", lambda n, *a: n < 40)
    monkeypatch.setattr(L, "EXPAND_FROM_PAIRS", 0)
    monkeypatch.setattr(L, "STRETCH_US", 0.0)

    def run(least):
        monkeypatch.setattr(L, "EXPAND_FROM_TOKENS", least)
        eng = Engine(d, dtype="bfloat16", max_num_seqs=6, kv_tokens=2000, max_model_len=512, max_tokens_per_step=512, decode_graphs=False)
        got, at = {r: [] for r in reqs}, {r: 0 for r in reqs}
        for r in reqs:
            eng.add_request(r)
        for step in steps:
            o = eng.step([StepEntry(r, reqs[r][at[r]:at[r] + n], tuple(range(n))) for r, n in step]).cpu()
            i = 0
            for r, n in step:
                got[r].append(o[i:i + n])
                i += n
                at[r] += n
        return {r: torch.cat(v).double() for r, v in got.items()}

    new = run(1)
    # three layers a step; what each step leaves over the shared rows, a stretch a call
    assert left_out == [9, 25] * 3 + [17, 2] * 3 + [2, 30] * 3 + [19, 1, 2] * 3
    shared = run(1 << 30)
    raw, w = plain.read_config(d), plain.load_weights(d, torch.float64)
    errs = []
    for r, toks in reqs.items():
        n = new[r].shape[0]
        want = plain.forward(raw, w, toks[:n]).double()
        errs.append(torch.stack([(x[r] - want).norm(dim=-1) / want.norm(dim=-1) for x in (new, shared)]))
    e_new, e_shared = torch.cat(errs, dim=1).pow(2).mean(dim=1).sqrt().tolist()
    print(f"{name}: some left out {e_new:.3e} shared {e_shared:.3e}")
    assert e_new <= 1.05 * e_shared and float(torch.cat(errs, dim=1)[0].max()) < 0.1


def test_only_layers_that_can_expand_have_the_pages_planned(tmp_path):
    """Layers with a gate for every output element, and layers in 32 bits, keep to the shared rows: their steps list no pages."""
    import tiny_kuvonex
    from sharpinference_amd import load_config
    from sharpinference_amd.engine import Engine
    from sharpinference_amd.parts.latent_attention import LatentPages
    from sharpinference_amd.weights.loader import write_random_model

    def planned(cfg, dtype):
        d = str(tmp_path / cfg["architecture"])
        write_random_model(load_config(cfg), d, 7, std=0.1)
        eng = Engine(d, dtype=dtype, max_num_seqs=1, kv_tokens=64, max_model_len=64, max_tokens_per_step=64, decode_graphs=False)
        return sum(isinstance(p, LatentPages) for p in eng.runner.planners)

    gated = _latent_only("rigodra")
    assert planned(gated, "bfloat16") == 1 and planned(gated, "float32") == 0
    assert planned(next(iter(tiny_kuvonex.CONFIGS.values())), "bfloat16") == 0
