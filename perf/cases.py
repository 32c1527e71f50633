"""The work the framework is timed on: steps of the engine, as a serving program calls them.

A pass is one step of continuous batching through `Engine.step`: requests that are being decoded bring
a token each, new prompts bring all of theirs (a prompt longer than a step goes in portions), the
logits of every request's last token come back, and the new prompts' requests end.  A case names

    model, size   the design and its layers' sizes (those of the benchmark's shapes, fewer layers)
    dtype         bfloat16, as models are served, or float32, as traces are replayed
    requests      requests that decode one token each, with `context` tokens in the cache
    prompts       new prompts of up to `tokens` tokens each (every further one is somewhat shorter)

Weights are random, drawn by the engine from a seed; a branch's last matrix is drawn smaller than the
rest and gates, sinks, decays and convolutions wider, so that every mechanism has its say.
"""
import math

import torch

from sharpinference_amd import load_config
from sharpinference_amd.engine import Engine, StepEntry
from sharpinference_amd.registry import build_model
from sharpinference_amd.weights.loader import RandomSource

STEP_TOKENS = 8192          # the most tokens a step takes
DECODE_LIMIT = 4096         # a decoding request that has grown to this many tokens starts again from its prompt


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    def case(name, model, size, requests=0, context=0, prompts=0, tokens=0, dtype="bfloat16"):
        return dict(name=name, model=model, size=size, dtype=dtype, requests=requests, context=context, prompts=prompts, tokens=tokens)
    return [
        # one user in a chat: every kernel's latency and the launches between them
        case("llama4 decode 1", "llama4", "scout", requests=1, context=700),
        # the benchmark's headline: a small batch that streams the experts' weights
        case("llama4 decode 8", "llama4", "scout", requests=8, context=2048),
        # reading one prompt: the first token's latency
        case("llama4 prompt 2048", "llama4", "scout", prompts=1, tokens=2048),
        # a long document, in portions of a step
        case("llama4 prompt 20011", "llama4", "scout", prompts=1, tokens=20011),
        # continuous batching: three new prompts beside the tokens of those that decode
        case("llama4 mixed", "llama4", "scout", requests=29, context=1100, prompts=3, tokens=457),
        # replaying a trace in 32 bits
        case("llama4 float32", "llama4", "w2048", requests=5, context=300, prompts=2, tokens=301, dtype="float32"),
        # a full batch of decoding requests, experts in groups, latent keys
        case("kuvonex decode 64", "kuvonex", "w2048", requests=64, context=1500),
        # prompts through each of the other designs
        case("rigodra prompt 2048", "rigodra", "w4096", prompts=1, tokens=2048),
        case("pazatar prompt 1900", "pazatar", "w2048", prompts=1, tokens=1900),
        case("nosedra mixed", "nosedra", "w2048", requests=16, context=900, prompts=2, tokens=1024),
        case("fovosun prompts 4 x 500", "fovosun", "w2048", prompts=4, tokens=500),
        case("pagonex prompt 3000", "pagonex", "w2048", prompts=1, tokens=3000),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    model = rng.choice(["llama4", "llama4", "llama4", "kuvonex", "rigodra", "pazatar", "nosedra", "fovosun", "pagonex"])
    size = rng.choice(["scout", "scout", "w2048"]) if model == "llama4" else rng.choice(["w2048", "w2048", "w4096"])
    kind = rng.choice(["decode", "prompt", "mixed"])
    dtype = "float32" if size == "w2048" and rng.random() < 0.15 else "bfloat16"
    most = 400 if dtype == "float32" else 4096
    c = dict(model=model, size=size, dtype=dtype, requests=0, context=0, prompts=0, tokens=0)
    if kind != "prompt":
        c.update(requests=spread(1, 64), context=spread(16, min(2500, 4 * most)))
    if kind != "decode":
        prompts = spread(1, 6)
        c.update(prompts=prompts, tokens=spread(16, most // prompts))
    return c


def prompt_lengths(case):
    return [max(1, case["tokens"] - j * (case["tokens"] // 9 + 1)) for j in range(case["prompts"])]


# ---------------------------------------------------------------------------
# the models
# ---------------------------------------------------------------------------
# the Scout layers' sizes: the published Llama 4 Scout configuration
SCOUT = dict(width=5120, layers=4, heads=40, kv_heads=8, experts=16, top=1, ff=8192, dense=16384, vocab=202048, rope_scaling={
    "rope_type": "llama3", "factor": 16.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0, "original_max_position_embeddings": 8192})
SIZES = {
    "w2048": dict(width=2048, layers=4, heads=16, vocab=32000, experts=64, top=6, ff=1408, groups=(8, 4), identity=8, q_rank=768,
                  dense=8192, kv_heads=4, decay_rank=64, delta_heads=16),
    "w4096": dict(width=4096, layers=4, heads=64, vocab=32000, experts=32, top=4, ff=2048, groups=(4, 2), identity=4, q_rank=1536,
                  dense=14336, kv_heads=8, decay_rank=128, delta_heads=32),
}


def rot(base, dims, **scaling):
    return {"base": base, "dims": dims, **({"scaling": scaling} if scaling else {})}


def llama4(z):
    return {"architectures": ["Llama4ForCausalLM"], "hidden_size": z["width"], "num_hidden_layers": z["layers"],
            "num_attention_heads": z["heads"], "num_key_value_heads": z["kv_heads"], "head_dim": 128, "vocab_size": z["vocab"],
            "intermediate_size": z["ff"], "intermediate_size_mlp": z["dense"], "num_local_experts": z["experts"],
            "num_experts_per_tok": z["top"], "interleave_moe_layer_step": 1, "attention_chunk_size": 8192, "use_qk_norm": True,
            "attn_temperature_tuning": True, "floor_scale": 8192, "attn_scale": 0.1, "rms_norm_eps": 1e-5, "rope_theta": 500000.0,
            "rope_scaling": z.get("rope_scaling"), "no_rope_layers": [int((i + 1) % 4 != 0) for i in range(z["layers"])],
            "tie_word_embeddings": False, "max_position_embeddings": 40960, "torch_dtype": "bfloat16"}


def kuvonex(z):
    mixer = {"heads": z["heads"], "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "scale": 192 ** -0.5, "rot": rot(10000.0, 64)}
    mlp = {"kind": "moe", "expert": {"ff": z["ff"]},
           "router": {"experts": z["experts"], "top": z["top"], "groups": {"count": z["groups"][0], "keep": z["groups"][1]}}}
    layers = [{"type": "latent_attention", "mixer": dict(mixer), "mlp": mlp} for _ in range(z["layers"])]
    layers[-1]["mixer"]["kv_from"] = z["layers"] - 2
    return {"architecture": "Kuvonex", "vocab": z["vocab"], "width": z["width"], "norm": {"eps": 1e-5}, "embedding": {"scale": 1.0},
            "layers": layers}


def rigodra(z):
    latent = {"heads": z["heads"], "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": z["q_rank"], "kv_rank": 512, "scale": 192 ** -0.5,
              "mask": {"size": 1024}, "rot": rot(10000.0, 64)}
    attn = {"heads": z["heads"], "kv_heads": z["heads"] // 8, "dim": 192, "vdim": 128, "scale": 192 ** -0.5, "v_mix": True,
            "mask": {"size": 1024, "keep_first": 64}, "rot": rot(10000.0, 64)}
    moe = {"kind": "moe", "expert": {"ff": z["ff"]}, "shared": {"ff": z["ff"]},
           "router": {"experts": z["experts"] - z["identity"], "top": z["top"], "identity": z["identity"],
                      "groups": {"count": z["groups"][0], "keep": z["groups"][1]}}}
    dense = {"kind": "dense", "ff": z["ff"] * z["top"]}
    layers = [("latent_attention", latent, moe), ("attention", attn, moe), ("attention", attn, moe), ("latent_attention", latent, dense)]
    return {"architecture": "Rigodra", "vocab": z["vocab"], "width": z["width"], "norm": {"eps": 1e-5}, "postln_alpha": 1.7,
            "layers": [{"type": t, "mixer": m, "mlp": f} for t, m, f in layers]}


def pazatar(z):
    attention = {"heads": z["heads"] // 2 if z["width"] == 4096 else z["heads"], "kv_heads": z["kv_heads"], "dim": 128, "vdim": 128,
                 "scale": 128 ** -0.5, "mask": {"size": 1024}}
    left = dict(attention, conv=4, softcap=50.0, mask={"size": 512}, rot=rot(20000.0, 64, factor=8.0, low=1.0, high=4.0, original=2048))
    attention = dict(attention, rot=rot(10000.0, 128, factor=8.0, original=1024, fast=32.0, slow=1.0))
    right = {"heads": attention["heads"], "dim": 128, "vdim": 128, "tau": 16.0, "decay_rank": z["decay_rank"]}
    layers = [("attention", attention) if i % 2 == 0 else ("parallel", {"left": left, "right": right}) for i in range(z["layers"])]
    return {"architecture": "Pazatar", "vocab": z["vocab"], "width": z["width"], "norm": {"eps": 1e-5},
            "layers": [{"type": t, "mixer": m, "mlp": {"kind": "dense", "ff": z["dense"]}} for t, m in layers],
            "loop": {"start": 0, "stop": z["layers"], "times": 1}}


def nosedra(z):
    heads = z["width"] // 128
    left = {"heads": heads, "kv_heads": z["kv_heads"], "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "rot": rot(1000000.0, 64, factor=4.0)}
    right = {"heads": heads, "dim": 128, "vdim": 128, "gate_cap": 10.0}
    space = {"heads": 2 * z["width"] // 64, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}
    both = {"left": left, "right": right, "left_scale": 1.0, "right_scale": 1.0}
    return {"architecture": "Nosedra", "vocab": z["vocab"], "width": z["width"], "norm": {"eps": 1e-5}, "token_side": {"dim": 256},
            "logit_softcap": 50.0, "layers": [{"type": t, "mixer": space if t == "mamba2" else both, "mlp": {"kind": "dense", "ff": z["dense"]}}
                                              for t in ("parallel", "parallel", "mamba2", "parallel")]}


def fovosun(z):
    heads = z["width"] // 128
    base = {"heads": heads, "kv_heads": heads // 8, "dim": 64, "vdim": 128, "scale": 64 ** -0.5, "diff": 0.3}
    windowed = dict(base, rot=rot(10000.0, 64), mask={"size": 1024})
    conv = dict(base, conv=4, q_temp={"coef": 0.1, "every": 1024})
    ret = {"heads": heads, "dim": 128, "vdim": 128, "decay": [1.0 - 2.0 ** (-5 - 3 * h / heads) for h in range(heads)], "rot": rot(1000000.0, 64)}
    mlp = {"kind": "moe", "expert": {"ff": z["ff"], "limit": 7.0}, "router": {"experts": z["experts"], "top": z["top"]},
           "shared": {"ff": z["ff"], "limit": 3.0}}
    return {"architecture": "Fovosun", "vocab": z["vocab"], "width": z["width"], "norm": {"eps": 1e-5}, "embedding": {"scale": 1.0},
            "streams": 4, "layers": [{"type": t, "mixer": m, "mlp": mlp} for t, m in
                                     (("attention_2", windowed), ("attention", conv), ("retention", ret), ("attention_2", windowed))]}


def pagonex(z):
    delta = {"heads": z["delta_heads"], "kv_heads": z["delta_heads"] // 2, "dim": 128, "vdim": 128, "conv": 4, "decay_rank": 128, "gate_rank": 128}
    latent = {"heads": z["heads"], "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": z["q_rank"], "kv_rank": 512, "scale": 192 ** -0.5,
              "mask": {"size": 1024}, "rot": rot(10000.0, 64, factor=8.0, original=1024, fast=32.0, slow=1.0)}
    mlp = {"kind": "moe", "expert": {"ff": z["ff"], "limit": 7.0}, "router": {"experts": z["experts"], "top": z["top"], "scale": 2.5},
           "shared": {"ff": z["ff"], "limit": 3.0}}
    layers = [("channel_delta", delta), ("latent_attention", latent), ("latent_attention", dict(latent, kv_from=1)), ("channel_delta", delta)]
    return {"architecture": "Pagonex", "vocab": z["vocab"], "width": z["width"], "norm": {"eps": 1e-5}, "canon": {"taps": 4},
            "embedding": {"bigram": {"buckets": 100003, "mul_prev": 10007, "mul_cur": 257}}, "logit_scale": 1.0,
            "layers": [{"type": t, "mixer": m, "mlp": mlp} for t, m in layers]}


MAKERS = dict(llama4=llama4, kuvonex=kuvonex, rigodra=rigodra, pazatar=pazatar, nosedra=nosedra, fovosun=fovosun, pagonex=pagonex)


def config_of(case):
    return MAKERS[case["model"]](SCOUT if case["size"] == "scout" else SIZES[case["size"]])


def deviations(case):
    """What the weights' standard deviations are where they are not 0.02, by the end of a tensor's name (the first that fits)."""
    small = 0.2 / math.sqrt((SCOUT if case["size"] == "scout" else SIZES[case["size"]])["ff"])
    return {
        "llama4": {"embed_tokens.weight": 1.0, "down_proj": small, "down_proj.weight": small},
        "kuvonex": {"embed": 6.0, ".sink": 1.0, ".correction": 0.1},
        "rigodra": {".router": 0.1, ".vmix": 0.5},
        "pazatar": {"embed": 0.5, ".conv": 0.5, ".a2.b": 1.5},
        "nosedra": {"embed": 1.0, ".conv": 0.5, ".i.b": 1.0, ".f.b": 2.0, ".sink": 1.0, ".dt_bias": 1.0, ".A_log": 0.7, ".D": 1.0},
        "fovosun": {"embed": 1.0, ".conv": 0.5, ".in": 0.7, ".out": 0.7, ".mix": 0.6, ".router": 0.1,
                    ".lq1": 0.1, ".lk1": 0.1, ".lq2": 0.1, ".lk2": 0.1},
        "pagonex": {"embed": 1.0, "bigram": 0.3, ".conv": 0.5, "canon1": 0.3, "canon2": 0.3, ".A_log": 1.0, ".dt_bias": 1.0, ".router": 0.1},
    }[case["model"]]


# ---------------------------------------------------------------------------
# a pass
# ---------------------------------------------------------------------------
def tokens_of(case, seed):
    """(the decoding requests' tokens: those in the cache, then the ones fed one a pass; the new prompts' tokens)"""
    vocab = (SCOUT if case["size"] == "scout" else SIZES[case["size"]])["vocab"]
    g = torch.Generator().manual_seed(seed)
    lengths = [max(1, case["context"] - 3 * i) for i in range(case["requests"])]
    held = [torch.randint(vocab, (n + 64,), generator=g).tolist() for n in lengths]
    return [(t[:-64], t[-64:]) for t in held], [torch.randint(vocab, (n,), generator=g).tolist() for n in prompt_lengths(case)]


def prepare(case, seed):
    held, prompts = tokens_of(case, seed)
    most = max([len(p) for p in prompts] + [DECODE_LIMIT if held else 0]) + 16
    engine = Engine(config=config_of(case), weight_seed=seed, weight_std_by_suffix=deviations(case), dtype=case["dtype"],
                    max_num_seqs=len(held) + len(prompts), max_tokens_per_step=STEP_TOKENS, max_model_len=most,
                    kv_tokens=len(held) * DECODE_LIMIT + sum(len(p) + 16 for p in prompts) + 16)
    state = dict(engine=engine, held=held, prompts=prompts, step=0)
    begin_decoding(state)
    return state


def begin_decoding(state):
    """The decoding requests' prompts into the cache, several in a step."""
    engine, entries, room = state["engine"], [], STEP_TOKENS
    for i, (prompt, _) in enumerate(state["held"]):
        engine.add_request(("decode", i))
        if len(prompt) > room:
            engine.step(entries)
            entries, room = [], STEP_TOKENS
        entries.append(StepEntry(("decode", i), prompt))
        room -= len(prompt)
    if entries:
        engine.step(entries)
    state["grown"] = 0


def run(state):
    engine, held, prompts = state["engine"], state["held"], state["prompts"]
    if held and len(held[0][0]) + state["grown"] >= DECODE_LIMIT:      # as long as a request may get: from the start again
        for i in range(len(held)):
            engine.free_request(("decode", i))
        begin_decoding(state)
    place = state["step"] % 64
    entries = [StepEntry(("decode", i), (after[place],), (0,)) for i, (_, after) in enumerate(held)]
    for j, prompt in enumerate(prompts):
        engine.add_request(("prompt", j))
        while len(prompt) > STEP_TOKENS:                               # a long prompt: all but its last portion
            engine.step([StepEntry(("prompt", j), prompt[:STEP_TOKENS])])
            prompt = prompt[STEP_TOKENS:]
        entries.append(StepEntry(("prompt", j), prompt, (len(prompt) - 1,)))
    logits = engine.step(entries)
    for j in range(len(prompts)):
        engine.free_request(("prompt", j))
    state["step"] += 1
    state["grown"] += 1
    return logits


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: every weight the tokens need once (of routed experts those that a token is expected to pick),
    what the cache holds of the context, the logits.  Flops: two a weight and token, and the attention's
    products or the states' updates."""
    cfg, wide = config_of(case), 2 if case["dtype"] == "bfloat16" else 4
    z = SCOUT if case["size"] == "scout" else SIZES[case["size"]]
    spans = [(max(1, case["context"] - 3 * i), 1) for i in range(case["requests"])] + [(0, n) for n in prompt_lengths(case)]
    tokens, rows = sum(n for _, n in spans), len(spans)
    reached = 1.0 - (1.0 - z["top"] / z["experts"]) ** tokens
    size, flops = 0.0, 0.0
    for name, spec in build_model(load_config(cfg)).param_specs().items():
        n = math.prod(spec.shape)
        if "embed" in name or "bigram" in name:
            size += min(n, tokens * spec.shape[-1]) * wide
            head = name == "embed" and case["model"] in ("pazatar", "rigodra")           # the embedding is the head too
            if head:
                size, flops = size + n * wide, flops + 2.0 * n * rows
        elif "head" in name:
            size, flops = size + n * wide, flops + 2.0 * n * rows
        elif ".experts." in name or ".mlp.e" in name:
            size, flops = size + n * wide * reached, flops + 2.0 * n * tokens * z["top"] / z["experts"]
        else:
            size, flops = size + n * wide, flops + (2.0 * n * tokens if len(spec.shape) == 2 else 0.0)

    def pairs(window=None, chunk=None):
        total = 0.0
        for start, n in spans:
            for a in range(start, start + n):
                total += a % chunk + 1 if chunk else min(a + 1, window) if window else a + 1
        return total

    def keys(window=None):
        return sum(min(s + n, n + window) if window else s + n for s, n in spans)

    if case["model"] == "llama4":
        for roped in cfg["no_rope_layers"]:
            flops += 4.0 * z["heads"] * 128 * pairs(chunk=8192 if roped else None)
            size += 2 * z["kv_heads"] * 128 * wide * keys(8192 if roped else None)
    else:
        for layer in cfg["layers"]:
            m = layer["mixer"]
            for mix in ([m["left"], m["right"]] if layer["type"] == "parallel" else [m]):
                window = (mix.get("mask") or {}).get("size")
                if "kv_rank" in mix:
                    flops += 2.0 * mix["heads"] * (mix["dim"] + mix["rot_dim"] + mix["vdim"]) * pairs(window)
                    size += (mix["kv_rank"] + mix["rot_dim"]) * wide * keys(window)
                elif "kv_heads" in mix and layer["type"] != "channel_delta":
                    chunked = case["model"] == "pazatar"
                    maps = 2 if "diff" in mix else 1
                    flops += 2.0 * maps * mix["heads"] * (mix["dim"] + mix["vdim"]) * (pairs(chunk=window) if chunked else pairs(window))
                    size += mix["kv_heads"] * (maps * mix["dim"] + mix["vdim"]) * wide * keys(window)
                else:
                    cells = mix["heads"] * mix["vdim"] * mix.get("dim", mix.get("state", 0))
                    flops += (7.0 if layer["type"] == "channel_delta" else 5.0) * cells * tokens
                    size += 2 * 4 * cells * rows
    return {"bytes": size + 4 * z["vocab"] * rows, "flops": flops}


def tolerance(case):
    # bfloat16: four times the distance to `exact` (0.5 to 1 % measured), held at 3 %; where a row's router chooses otherwise between
    # two experts of nearly equal score that row moves by the share of that expert in it, and the worst of its values with it
    # (a prompt's last row then lies 2 to 5 % off).  float32: 1e-6 to 7e-6 measured
    if case["dtype"] == "bfloat16":
        return {"rel": 0.03, "max": 0.9}
    return {"rel": 1e-4, "max": 0.01}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def rms(x, w=1.0):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5) * w


def layer_norm(x, w, b):
    c = x - x.mean(-1, keepdim=True)
    return rms(c, w) + b


def silu(x):
    return x * torch.sigmoid(x)


def rotate(x, pos, freqs, halves, magnitude=1.0):
    """The first 2 len(freqs) elements of x [N, heads, d]: a pair (a, b) turns by pos * freq; pairs are neighbours or lie in two halves."""
    f = torch.tensor(freqs, dtype=torch.float64, device=x.device)
    a = pos.double()[:, None, None] * f
    cos, sin, n = a.cos() * magnitude, a.sin() * magnitude, len(freqs)
    x = x.clone()
    one, two = (x[..., :n].clone(), x[..., n:2 * n].clone()) if halves else (x[..., 0:2 * n:2].clone(), x[..., 1:2 * n:2].clone())
    first, second = one * cos - two * sin, two * cos + one * sin
    if halves:
        x[..., :n], x[..., n:2 * n] = first, second
    else:
        x[..., 0:2 * n:2], x[..., 1:2 * n:2] = first, second
    return x


def frequencies(base, dims, s=None):
    """(frequencies, magnitude): plain, divided by a factor, stretched between two wavelengths, or ramped between two numbers of turns."""
    f = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
    if not s:
        return f, 1.0
    factor = s["factor"]
    if "fast" in s:
        place = [dims * math.log(s["original"] / (2 * math.pi * t)) / (2 * math.log(base)) for t in (s["fast"], s["slow"])]
        lo, hi = max(math.floor(place[0]), 0), min(math.ceil(place[1]), dims - 1)
        ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(dims // 2)]
        return [x / factor * r + x * (1.0 - r) for x, r in zip(f, ramp)], 0.1 * math.log(factor) + 1.0
    if "original" in s:
        out = []
        for x in f:
            t = (s["original"] * x / (2 * math.pi) - s["low"]) / (s["high"] - s["low"])
            t = min(max(t, 0.0), 1.0)
            out.append((1.0 - t) * x / factor + t * x)
        return out, 1.0
    return [x / factor for x in f], 1.0


class Exact:
    """One pass in 64 bits: whole sequences side by side, `spans` (first row, rows) of each in the flat batch."""

    def __init__(self, case, seed):
        self.case, self.cfg = case, config_of(case)
        self.z = SCOUT if case["size"] == "scout" else SIZES[case["size"]]
        dtype = torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32
        self.weights = RandomSource(build_model(load_config(self.cfg)).param_specs(), seed, dtype, torch.device("cuda:0"),
                                    stored_dtype=torch.bfloat16, std_by_suffix=deviations(case), generate_on_device=True)
        held, prompts = tokens_of(case, seed)
        sequences = [prompt + after[:1] for prompt, after in held] + prompts
        self.spans, at = [], 0
        for s in sequences:
            self.spans.append((at, len(s)))
            at += len(s)
        self.tokens = torch.tensor([t for s in sequences for t in s], device="cuda")
        self.pos = torch.cat([torch.arange(len(s), device="cuda") for s in sequences])

    def w(self, name):
        return self.weights.get(name).double()

    def linear(self, x, name):
        return x @ self.w(name).T

    def conv(self, u, w, b=0.0):
        out = torch.empty_like(u)
        for a, n in self.spans:
            padded = torch.cat([u.new_zeros(w.shape[1] - 1, u.shape[1]), u[a:a + n]])
            out[a:a + n] = b + sum(padded[j:j + n] * w[:, j] for j in range(w.shape[1]))
        return out

    def attend(self, q, k, v, scale, window=None, chunk=None, keep=0, cap=None, sink=None):
        """q [N, H, d], k [N, G, d], v [N, G, e]; `sink` [H]: one more term of the denominator."""
        H, G = q.shape[1], k.shape[1]
        out = q.new_empty(q.shape[0], H, v.shape[2])
        for a, n in self.spans:
            kt, vt = (t[a:a + n].repeat_interleave(H // G, 1).transpose(0, 1).contiguous() for t in (k, v))
            kt = kt.transpose(1, 2).contiguous()
            for o in range(0, n, 256):
                i = torch.arange(o, min(o + 256, n), device=q.device)[:, None]
                j = torch.arange(n, device=q.device)[None]
                see = j <= i
                if window:
                    see = see & ((i - j < window) | (j < keep))
                if chunk:
                    see = see & (i // chunk == j // chunk)
                s = torch.bmm(q[a + o:a + o + i.shape[0]].transpose(0, 1).contiguous(), kt) * scale
                if cap:
                    s = cap * torch.tanh(s / cap)
                s = s.masked_fill(~see, -math.inf)
                if sink is not None:
                    s = torch.cat([s, sink[:, None, None].expand(H, i.shape[0], 1)], -1)
                p = torch.softmax(s, -1)[..., :n]
                out[a + o:a + o + i.shape[0]] = torch.bmm(p.contiguous(), vt).transpose(0, 1)
        return out

    def walk(self, inputs, state, step):
        """step(state, inputs of a token) -> (state, output), over all sequences side by side."""
        most = max(n for _, n in self.spans)
        padded = []
        for x in inputs:
            p = x.new_zeros(len(self.spans), most, *x.shape[1:])
            for i, (a, n) in enumerate(self.spans):
                p[i, :n] = x[a:a + n]
            padded.append(p)
        outs = []
        for t in range(most):
            state, o = step(state, *(p[:, t] for p in padded))
            outs.append(o)
        outs = torch.stack(outs, 1)
        return torch.cat([outs[i, :n] for i, (_, n) in enumerate(self.spans)])

    def experts(self, ids, weights, unit, h):
        """Sum over the picks of weight * unit(rows, expert)."""
        y = torch.zeros_like(h)
        for e in ids.unique().tolist():
            rows, slot = (ids == e).nonzero(as_tuple=True)
            y[rows] += weights[rows, slot, None] * unit(h[rows], e)
        return y

    def logits(self):
        last = torch.tensor([a + n - 1 for a, n in self.spans], device="cuda")
        return getattr(self, self.case["model"])(last)

    # -- Llama 4 -----------------------------------------------------------
    def llama4(self, last):
        z, cfg = self.z, self.cfg
        x = self.weights.get("model.embed_tokens.weight")[self.tokens].double()
        scaling = z.get("rope_scaling")
        freqs, _ = frequencies(500000.0, 128, scaling and {"factor": scaling["factor"], "low": scaling["low_freq_factor"],
                                                           "high": scaling["high_freq_factor"], "original": scaling["original_max_position_embeddings"]})
        for i, roped in enumerate(cfg["no_rope_layers"]):
            p = f"model.layers.{i}."
            h = rms(x, self.w(p + "input_layernorm.weight"))
            q, k, v = (self.linear(h, f"{p}self_attn.{n}_proj.weight").reshape(len(h), -1, 128) for n in "qkv")
            if roped:
                q, k = rms(rotate(q, self.pos, freqs, False)), rms(rotate(k, self.pos, freqs, False))
            else:
                q = q * (1.0 + 0.1 * torch.log(torch.floor((self.pos.double() + 1.0) / 8192) + 1.0))[:, None, None]
            o = self.attend(q, k, v, 128 ** -0.5, chunk=8192 if roped else None)
            x = x + self.linear(o.reshape(len(h), -1), p + "self_attn.o_proj.weight")
            h = rms(x, self.w(p + "post_attention_layernorm.weight"))
            f = p + "feed_forward."
            s, ids = self.linear(h, f + "router.weight").topk(z["top"], -1)
            y = torch.zeros_like(h)
            g, u, d = (self.weights.get(f"{f}experts.{n}_proj") for n in ("gate", "up", "down"))
            for e in ids.unique().tolist():
                rows, slot = (ids == e).nonzero(as_tuple=True)
                r = h[rows] * torch.sigmoid(s[rows, slot])[:, None]
                y[rows] += (silu(r @ g[e].double().T) * (r @ u[e].double().T)) @ d[e].double().T
            f += "shared_expert."
            x = x + y + self.linear(silu(self.linear(h, f + "gate_proj.weight")) * self.linear(h, f + "up_proj.weight"), f + "down_proj.weight")
        return self.linear(rms(x[last], self.w("model.norm.weight")), "lm_head.weight")

    # -- latent attention --------------------------------------------------
    def latent_rows(self, h, p, m, halves):
        y = self.linear(h, p + "dkv")
        f, mag = frequencies(m["rot"]["base"], m["rot"]["dims"], m["rot"].get("scaling"))
        return rms(y[:, :512], self.w(p + "dkv.norm")), rotate(y[:, None, 512:], self.pos, f, halves, mag)

    def latent(self, h, p, m, kept, halves):
        """Attention over keys and values expanded from the kept rows, before the last projection."""
        H, d = m["heads"], m["dim"]
        c, turned = kept
        q = self.linear(rms(self.linear(h, p + "dq"), self.w(p + "dq.norm")), p + "uq") if "q_rank" in m else self.linear(h, p + "q")
        q = q.reshape(len(h), H, -1)
        f, mag = frequencies(m["rot"]["base"], m["rot"]["dims"], m["rot"].get("scaling"))
        q = torch.cat([q[..., :d], rotate(q[..., d:], self.pos, f, halves, mag)], -1)
        k = torch.cat([self.linear(c, p + "uk").reshape(len(c), H, d), turned.expand(-1, H, -1)], -1)
        sink = self.w(p + "sink") if self.case["model"] == "kuvonex" else None
        return self.attend(q, k, self.linear(c, p + "uv").reshape(len(c), H, -1), m["scale"], window=(m.get("mask") or {}).get("size"),
                           sink=sink).reshape(len(h), -1)

    def best_groups(self, choice, router, ranks):
        n, keep = router["groups"]["count"], router["groups"]["keep"]
        g = choice.reshape(len(choice), n, -1)
        best = g.topk(ranks, -1).values.sum(-1).topk(keep, -1).indices
        open_ = torch.zeros(len(choice), n, dtype=torch.bool, device=choice.device).scatter_(1, best, True)
        return choice.masked_fill(~open_.repeat_interleave(g.shape[2], 1), -math.inf)

    def kuvonex(self, last):
        x = self.weights.get("embed")[self.tokens].double()
        kept = {}
        for i, layer in enumerate(self.cfg["layers"]):
            p, m, r = f"l{i}.mix.", layer["mixer"], layer["mlp"]["router"]
            kept[i] = kept[m["kv_from"]] if "kv_from" in m else self.latent_rows(x, p, m, False)
            o = self.latent(x, p, m, kept[i], False) * torch.sigmoid(self.linear(x, p + "g"))
            x = x + rms(self.linear(o, p + "o"), self.w(f"l{i}.norm1"))
            p = f"l{i}.mlp."
            s = torch.sigmoid(self.linear(x, p + "router"))
            ids = self.best_groups(s + self.w(p + "correction"), r, 2).topk(r["top"], -1).indices
            y = self.experts(ids, s.gather(1, ids), lambda t, e: self.linear(
                silu(self.linear(t, f"{p}e{e}.gate")) * self.linear(t, f"{p}e{e}.up"), f"{p}e{e}.down"), x)
            x = x + rms(y, self.w(f"l{i}.norm2"))
        return self.linear(rms(x[last], self.w("final.norm")), "head")

    def rigodra(self, last):
        def norm(t, name):
            return layer_norm(t, self.w(name), self.w(name + ".b"))

        def relu2(t, p):
            return self.linear(torch.relu(self.linear(t, p + "up")).pow(2), p + "down")
        x, first = norm(self.weights.get("embed")[self.tokens].double(), "embed.norm"), None
        for i, layer in enumerate(self.cfg["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            if layer["type"] == "attention":
                H, G = m["heads"], m["kv_heads"]
                f, _ = frequencies(m["rot"]["base"], m["rot"]["dims"])
                q = rotate(rms(self.linear(x, p + "q").reshape(len(x), H, -1), self.w(p + "q.norm")), self.pos, f, True)
                k = rotate(rms(self.linear(x, p + "k").reshape(len(x), G, -1), self.w(p + "k.norm")), self.pos, f, True)
                v = self.linear(x, p + "v").reshape(len(x), G, -1)
                if first is None:
                    first = v
                else:
                    v = (1.0 - self.w(p + "vmix")) * v + self.w(p + "vmix") * first
                o = self.attend(q, k, v, m["scale"], window=m["mask"]["size"], keep=m["mask"]["keep_first"])
                o = (o * torch.sigmoid(self.linear(x, p + "g"))[:, :, None]).reshape(len(x), -1)
            else:
                o = self.latent(x, p, m, self.latent_rows(x, p, m, True), True)
            x = norm(1.7 * x + self.linear(o, p + "o"), f"l{i}.norm1")
            p = f"l{i}.mlp."
            if layer["mlp"]["kind"] == "dense":
                u = self.linear(x, p + "up")
                y = self.linear(0.5 * u * (1.0 + torch.erf(u / math.sqrt(2.0))), p + "down")
            else:
                r = layer["mlp"]["router"]
                s = torch.softmax(self.linear(x, p + "router"), -1)
                ids = self.best_groups(s + self.w(p + "correction"), r, 1).topk(r["top"], -1).indices
                y = self.experts(ids, s.gather(1, ids), lambda t, e: relu2(t, f"{p}e{e}.") if e < r["experts"] else t, x) + relu2(x, p + "shared.")
            x = norm(1.7 * x + y, f"l{i}.norm2")
        return self.linear(norm(x[last], "final.norm"), "embed")

    # -- recurrent states --------------------------------------------------
    def zero_state(self, m):
        return torch.zeros(len(self.spans), m["heads"], m.get("dim", m.get("state")), m["vdim"], dtype=torch.float64, device="cuda")

    def pazatar(self, last):
        x = self.weights.get("embed")[self.tokens].double() + self.w("loop.step")[0]
        N = len(x)

        def update(S, q, k, v, alpha):
            S = alpha[..., None] * S + k[..., None] * v[:, :, None]
            return S, (S * q[..., None]).sum(2)
        for i, layer in enumerate(self.cfg["layers"]):
            h, p, m = rms(x, self.w(f"l{i}.norm1")), f"l{i}.mix.", layer["mixer"]
            if layer["type"] == "attention":
                k = self.linear(h, p + "k")
                v = k.reshape(N, m["kv_heads"], -1)
                f, mag = frequencies(m["rot"]["base"], m["rot"]["dims"], m["rot"]["scaling"])
                q, k = (rotate(rms(t, self.w(p + n + ".norm")).reshape(N, -1, 128), self.pos, f, False, mag)
                        for n, t in (("q", self.linear(h, p + "q")), ("k", k)))
                y = self.linear(self.attend(q, k, v, m["scale"], chunk=m["mask"]["size"]).reshape(N, -1), p + "o")
            else:
                a, b, s = m["left"], m["right"], p + "left."
                q, k, v = (self.conv(self.linear(h, s + n), self.w(s + n + ".conv")).reshape(N, -1, 128) for n in "qkv")
                f, _ = frequencies(a["rot"]["base"], a["rot"]["dims"], a["rot"]["scaling"])
                q, k = (rotate(rms(t, self.w(s + n + ".norm")), self.pos, f, True) for n, t in (("q", q), ("k", k)))
                left = self.attend(q, k, v, a["scale"], chunk=a["mask"]["size"], cap=a["softcap"],
                                   sink=torch.zeros(a["heads"], dtype=torch.float64, device="cuda"))
                left = self.linear(left.reshape(N, -1), s + "o")
                s = p + "right."
                q, k, v = (self.linear(h, s + n).reshape(N, -1, 128) for n in "qkv")
                decay = self.linear(self.linear(h, s + "a1"), s + "a2") + self.w(s + "a2.b")
                decay = torch.exp(torch.nn.functional.logsigmoid(decay) / b["tau"]).reshape(N, -1, 128)
                o = rms(self.walk((q * 128 ** -0.5, k, v, decay), self.zero_state(b), update), self.w(s + "norm")).reshape(N, -1)
                right = self.linear(o * silu(self.linear(h, s + "g")), s + "o")
                y = 0.5 * (rms(left, self.w(p + "left.out")) + rms(right, self.w(s + "out")))
            x = x + rms(y, self.w(f"l{i}.norm1b"))
            h = rms(x, self.w(f"l{i}.norm2"))
            x = x + rms(self.linear(torch.relu(self.linear(h, f"l{i}.mlp.up")).pow(2), f"l{i}.mlp.down"), self.w(f"l{i}.norm2b"))
        return self.linear(rms(x[last], self.w("final.norm")), "embed")

    def nosedra(self, last):
        x = self.weights.get("embed")[self.tokens].double()
        N, softplus = len(x), torch.nn.functional.softplus

        def memory(state, q, k, v, log_i, log_f):
            S, n, top = state
            new = torch.maximum(log_f + top, log_i)
            keep, take = torch.exp(log_f + top - new)[..., None], torch.exp(log_i - new)[..., None]
            S, n = keep[..., None] * S + (take * k)[..., None] * v[:, :, None], keep * n + take * k
            den = torch.maximum((n * q).sum(-1).abs(), torch.exp(-new)) + 1e-6
            return (S, n, new), (S * q[..., None]).sum(2) / den[..., None]

        def space(S, u, B, C, dt, decay):
            S = decay[..., None, None] * S + (dt[..., None] * B)[..., None] * u[:, :, None]
            return S, (S * C[..., None]).sum(2)
        for i, layer in enumerate(self.cfg["layers"]):
            h, p, m = rms(x, 1.0 + self.w(f"l{i}.norm1")), f"l{i}.mix.", layer["mixer"]
            if layer["type"] == "parallel":
                a, b, s = m["left"], m["right"], p + "left."
                q, k, v = (self.linear(h, s + n).reshape(N, -1, 128) for n in "qkv")
                f, _ = frequencies(a["rot"]["base"], a["rot"]["dims"], a["rot"]["scaling"])
                q, k = (rms(rotate(t, self.pos, f, True)) for t in (q, k))
                o = self.attend(q, k, v, a["scale"], sink=self.w(s + "sink")).reshape(N, -1) * torch.sigmoid(self.linear(h, s + "g"))
                x = x + self.linear(o, s + "o")
                s = p + "right."
                q, k, v = (self.linear(h, s + n).reshape(N, -1, 128) for n in "qkv")
                log_i, log_f = (10.0 * torch.tanh((self.linear(h, s + n) + self.w(f"{s}{n}.b")) / 10.0) for n in "if")
                S = self.zero_state(b)
                o = self.walk((q * 128 ** -0.5, k, v, log_i, -softplus(-log_f)), (S, S[..., 0].clone(), S[..., 0, 0].clone()), memory)
                o = rms(o).reshape(N, -1) * self.w(s + "norm") * torch.sigmoid(self.linear(h, s + "g"))
                x = x + self.linear(o, s + "o")
            else:
                H, e, d, G = m["heads"], m["vdim"], m["state"], m["groups"]
                inner = H * e
                u = self.linear(h, p + "in")
                c = silu(self.conv(u[:, inner:2 * inner + 2 * G * d].contiguous(), self.w(p + "conv"), self.w(p + "conv.b")))
                v = c[:, :inner].reshape(N, H, e)
                B, C = (t.reshape(N, G, d).repeat_interleave(H // G, 1) for t in c[:, inner:].chunk(2, 1))
                dt = softplus(u[:, 2 * inner + 2 * G * d:] + self.w(p + "dt_bias"))
                y = self.walk((v, B, C, dt, torch.exp(-torch.exp(self.w(p + "A_log")) * dt)), self.zero_state(m), space)
                y = (y + self.w(p + "D")[:, None] * v).reshape(N, inner) * silu(u[:, :inner])
                y = rms(y.reshape(N, m["norm_groups"], -1)).reshape(N, inner) * self.w(p + "norm")
                x = x + self.linear(y, p + "o")
            h, p = rms(x, 1.0 + self.w(f"l{i}.norm2")), f"l{i}.mlp."
            g = torch.nn.functional.gelu(self.linear(h, p + "gate") + self.w(p + "gate.b"), approximate="tanh")
            x = x + self.linear(g * (self.linear(h, p + "up") + self.w(p + "up.b")), p + "down") + self.w(p + "down.b")
            p = f"l{i}.side."
            e = self.weights.get("side.embed")[self.tokens, i * 256:(i + 1) * 256].double()
            g = torch.nn.functional.gelu(self.linear(x, p + "gate"), approximate="tanh")
            x = x + rms(self.linear(g * e, p + "proj"), self.w(p + "norm"))
        return 50.0 * torch.tanh(self.linear(rms(x[last], 1.0 + self.w("final.norm")), "head") / 50.0)

    def unit(self, h, p, limit):
        g, u = self.linear(h, p + "gate").clamp(max=limit), self.linear(h, p + "up").clamp(-limit, limit)
        return self.linear(g * torch.sigmoid(1.702 * g) * (u + 1.0), p + "down")

    def fovosun(self, last):
        x = self.weights.get("embed")[self.tokens].double()
        N, lanes = len(x), x[None].repeat(4, 1, 1)

        def update(S, q, k, v):
            S = decay[:, None, None] * S + k[..., None] * v[:, :, None]
            return S, (S * q[..., None]).sum(2)
        for i, layer in enumerate(self.cfg["layers"]):
            m, f = layer["mixer"], layer["mlp"]
            for n in (1, 2):
                p = f"l{i}.hc{n}."
                h = rms(torch.einsum("s,stw->tw", self.w(p + "in"), lanes), self.w(f"l{i}.norm{n}"))
                s = f"l{i}.mix."
                if n == 2:
                    s = f"l{i}.mlp."
                    val, ids = (self.linear(h, s + "router") + self.w(s + "router.b")).topk(f["router"]["top"], -1)
                    y = self.experts(ids, torch.softmax(val, -1), lambda t, e: self.unit(t, f"{s}e{e}.", f["expert"]["limit"]), h)
                    y = y + self.unit(h, s + "shared.", f["shared"]["limit"])
                elif layer["type"] == "retention":
                    decay = torch.tensor(m["decay"], dtype=torch.float64, device="cuda")
                    q, k, v = (self.linear(h, s + t).reshape(N, -1, 128) for t in "qkv")
                    fr, _ = frequencies(m["rot"]["base"], m["rot"]["dims"])
                    q, k = rotate(q, self.pos, fr, True), rotate(k, self.pos, fr, True) * 128 ** -0.5
                    o = rms(self.walk((q, k, v), self.zero_state(m), update)).reshape(N, -1) * silu(self.linear(h, s + "g"))
                    y = self.linear(o, s + "o")
                else:
                    have = self.weights.specs
                    q, k, v = (self.linear(h, s + t) + (self.w(f"{s}{t}.b") if f"{s}{t}.b" in have else 0.0) for t in "qkv")
                    if m.get("conv"):
                        q, k, v = (self.conv(t, self.w(f"{s}{c}.conv")) for c, t in (("q", q), ("k", k), ("v", v)))
                    q, k, v = q.reshape(N, -1, 64), k.reshape(N, -1, 64), v.reshape(N, -1, 128)
                    if m.get("rot"):
                        fr, _ = frequencies(m["rot"]["base"], m["rot"]["dims"])
                        q, k = rotate(q, self.pos, fr, True), rotate(k, self.pos, fr, True)
                    if m.get("q_temp"):
                        q = q * (1.0 + 0.1 * torch.log(torch.floor((self.pos.double() + 1.0) / 1024) + 1.0))[:, None, None]
                    one, two = (self.attend(q[:, a::2], k[:, a::2], v, m["scale"], window=(m.get("mask") or {}).get("size")) for a in (0, 1))
                    lam = sum(t * torch.exp((self.w(f"{s}lq{a}") * self.w(f"{s}lk{a}")).sum()) for a, t in ((1, 1.0), (2, -1.0))) + m["diff"]
                    o = rms(one - lam * two) * (1.0 - m["diff"])
                    if s + "g" in have:
                        o = o * torch.sigmoid(self.linear(h, s + "g"))[:, :, None]
                    y = self.linear(o.reshape(N, -1), s + "o")
                lanes = torch.einsum("sr,stw->rtw", self.w(p + "mix"), lanes) + self.w(p + "out")[:, None, None] * y
        return self.linear(rms(lanes[:, last].sum(0), self.w("final.norm")), "head")

    def pagonex(self, last):
        big = self.cfg["embedding"]["bigram"]
        before = torch.cat([self.tokens[:1], self.tokens[:-1]])
        row = torch.where(self.pos == 0, big["buckets"], (before * big["mul_prev"] + self.tokens * big["mul_cur"]) % big["buckets"])
        x = self.weights.get("embed")[self.tokens].double() + self.weights.get("bigram")[row].double()
        N, kept = len(x), {}

        def norm(t, name):
            return layer_norm(t, self.w(name), self.w(name + ".b"))

        def update(S, q, k, v, g, beta):
            S = g[..., None] * S
            S = S + k[..., None] * (beta[..., None] * (v - (S * k[..., None]).sum(2)))[:, :, None]
            return S, (S * q[..., None]).sum(2)
        for i, layer in enumerate(self.cfg["layers"]):
            p, m, f = f"l{i}.mix.", layer["mixer"], layer["mlp"]
            h = x + self.conv(x, self.w(f"l{i}.canon1"))
            if layer["type"] == "channel_delta":
                q, k, v = (silu(self.conv(self.linear(h, p + n), self.w(f"{p}{n}.conv"))).reshape(N, -1, 128) for n in "qkv")
                q, k = (t / torch.sqrt(t.pow(2).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
                q, k = (t.repeat_interleave(m["heads"] // m["kv_heads"], 1) for t in (q * 128 ** -0.5, k))
                zed = (self.linear(self.linear(h, p + "a1"), p + "a2") + self.w(p + "dt_bias")).reshape(N, -1, 128)
                g = torch.exp(-torch.exp(self.w(p + "A_log"))[:, None] * torch.nn.functional.softplus(zed))
                o = self.walk((q, k, v, g, torch.sigmoid(self.linear(h, p + "b"))), self.zero_state(m), update)
                gate = torch.sigmoid(self.linear(self.linear(h, p + "g1"), p + "g2")).reshape(N, -1, 128)
                o = (rms(o, self.w(p + "norm")) * gate).reshape(N, -1)
            else:
                kept[i] = kept[m["kv_from"]] if "kv_from" in m else self.latent_rows(h, p, m, False)
                o = self.latent(h, p, m, kept[i], False)
            x = x + norm(self.linear(o, p + "o"), f"l{i}.norm1")
            h, p, r = x + self.conv(x, self.w(f"l{i}.canon2")), f"l{i}.mlp.", f["router"]
            val, ids = torch.softmax(self.linear(h, p + "router"), -1).topk(r["top"], -1)
            y = self.experts(ids, val / (val.sum(-1, keepdim=True) + 1e-20) * r["scale"],
                             lambda t, e: self.unit(t, f"{p}e{e}.", f["expert"]["limit"]), h) + self.unit(h, p + "shared.", f["shared"]["limit"])
            x = x + norm(y, f"l{i}.norm2")
        return self.linear(norm(x[last], "final.norm"), "head")


def exact(case, seed):
    with torch.no_grad():
        return Exact(case, seed).logits()
