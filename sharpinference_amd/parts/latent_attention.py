"""The latent attention mixer: keys and values of all heads kept as one low-rank row per token."""
from __future__ import annotations

from types import SimpleNamespace
from typing import Dict, List, Optional, Tuple

import numpy as np
import torch

from .. import ops
from ..cache.spec import KVSpec, WINDOW_NONE, WINDOW_SLIDING
from ..ops.lib import PREFILL_TILE_TOKENS
from ..ops.profile import section
from .attention import _WORK_LISTS, prompt_tile_tokens, prompt_tiles
from .base import HostStep, LayerCache, ParamSpec, Part, StepContext, StepPlanner, TensorSource


# A step's prompt portions attend over expanded keys and values where their queries times the keys of their spans are at least
# EXPAND_FROM_TOKENS times the keys to expand (a key's expansion costs about what 28 pairs save), and, times the heads, at
# least EXPAND_FROM_PAIRS (the two launches more), and where the whole of it saves time (_saved).  Microseconds of a step through
# four such layers over the shared rows and over expanded keys: 64 heads behind 2,000 keys, 40 tokens 1,177 / 1,354, 64: 1,757 /
# 1,347, 400: 3,213 / 1,595; behind none, 100 tokens 961 / 928, 400: 1,262 / 979; 16 heads behind 2,000, 40 tokens 1,140 / 1,031;
# behind none, 200 tokens 977 / 947, 700: 1,054 / 1,001.  A window makes the queries see fewer pairs than that, and the shared
# rows' kernel no faster: 2,000 tokens of 64 heads, window 64: 2,486 / 1,292, window 16: 2,345 / 1,273.
EXPAND_FROM_TOKENS = 32
EXPAND_FROM_PAIRS = 1 << 19
EXPAND_MAX_BYTES = 2 << 30         # ... and the expanded keys and values take at most this much for the layer's time: the
                                   # portions with the most keys give way


def _few_queries_lose(n: int, span: int, keys: int, heads: int, context: int, tile: int) -> bool:
    """Whether a portion of few queries (fewer than make up for their keys) is the slower for an expansion of its keys beside
    portions that pay.  Either way one block a head walks the keys, in microseconds: the expansion 0.8 for 1,024 keys and head,
    the flash kernel 0.05 a key (0.075 in tiles of the full height), the shared rows 0.13 a key of a run and 150 of
    launches.  A step through four layers, expanded / left out: 2,000 tokens and 2 behind 32,000 keys, 64 heads 17,470 /
    11,060, 16 heads 12,430 / 9,970; 1,000 tokens and 4 behind 24,000, 64 heads 10,330 / 10,070, 16 heads 6,940 / 9,360; behind
    6,000, 64 heads 3,130 / 3,340."""
    expanded = 0.8 * keys * heads / 1024 + (0.05 if tile < PREFILL_TILE_TOKENS else 0.075) * span
    return n < EXPAND_FROM_TOKENS and expanded > 0.13 * min(ops.latent_run_keys(context, True), span) + 150.0


# What a step leaves over the shared rows goes in stretches of neighbouring rows, five launches more each: a layer's time with the
# host that makes them, in microseconds (the first: as FIRST_STRETCH times the pairs of the expansion's two launches).
STRETCH_US = 75.0
FIRST_STRETCH = 20
PAIR_US = 5.0 / (1 << 20)          # (a layer's time for a query, a key and a head: 6.5 over the shared rows, 1.5 in the flash kernel)


def _saved(pairs: int, keys: int, span: int, heads: int, context: int, tile: int) -> float:
    """What an expansion saves a layer, in microseconds: `pairs` of query and key, `keys` to expand, `span` keys of the longest
    portion, which one block walks in either form.  Measured, a layer of four with experts behind them, and this: 64 heads, 200
    tokens 26 / 15, 400 107 / 55, 1,500 692 / 668, 40 behind 2,000 -37 / -46, 64 behind 2,000 106 / 95; 16 heads, 400 tokens 33 / 38,
    1,500 160 / 211, 100 behind 2,000 141 / 150.  A stretch took 30 to 60 of it (up to 90 where nothing else kept the GPU busy).
    Steps of 8 single tokens beside a portion, expanded / shared, microseconds: 64 heads, 200 tokens 1,940 / 1,860, 400 2,071 / 2,377,
    64 behind 2,000 2,407 / 2,705; 16 heads, 400 tokens 1,991 / 1,917, 700 2,081 / 2,215, 64 behind 2,000 2,050 / 2,634; two single
    tokens around 700 tokens of 64 heads 2,407 / 2,957."""
    walk = 0.13 * min(ops.latent_run_keys(context, True), span) - (0.05 if tile < PREFILL_TILE_TOKENS else 0.075) * span
    return walk + PAIR_US * pairs * heads - 0.8 * keys * heads / 1024


class LatentPages(StepPlanner):
    """Which of a step's prompt portions attend over expanded keys and values, seen through a window by `heads` heads of
    `width` elements of key and value.  For them the list of pages of 128 keys (entry, page of its sequence, first key that
    is there, end of the keys), the block table of a cache that holds just those, and their tiles; for the other portions
    the stretches of neighbouring rows and their tiles, counted from the stretch's first row."""

    def __init__(self, window_kind: int, window: int, heads: int, width: int):
        self.spec = KVSpec(1, 1, window_kind, window)
        self.heads, self.key_bytes = int(heads), 2 * int(heads) * int(width)
        self.key = f"latent pages {window_kind} {window} {heads} {width}"

    def plan(self, host: HostStep) -> Tuple[List[np.ndarray], dict]:
        nothing = [np.zeros(0, dtype=np.int32)] * 4, dict(pages=0)
        long = [e for e, n in enumerate(host.lens) if n > 1]
        if not long:
            return nothing
        tile = prompt_tile_tokens(host.lens)
        context = max(host.starts[e] + host.lens[e] for e in range(host.n_entries))
        spans = {}                                                # the entries' (first key, end, first page, end)
        for e in long:
            lo, hi = self.spec.first_visible(host.starts[e]), host.starts[e] + host.lens[e]
            spans[e] = (lo, hi, lo // ops.LATENT_PAGE_KEYS, (hi - 1) // ops.LATENT_PAGE_KEYS + 1)
        keys = {e: (end - first) * ops.LATENT_PAGE_KEYS for e, (_, _, first, end) in spans.items()}
        chosen = [e for e, (lo, hi, _, _) in spans.items()
                  if not _few_queries_lose(host.lens[e], hi - lo, keys[e], self.heads, context, tile)]
        while chosen and sum(keys[e] for e in chosen) * self.key_bytes > EXPAND_MAX_BYTES:
            chosen.remove(max(chosen, key=keys.__getitem__))
        pairs, all_keys = sum(host.lens[e] * (spans[e][1] - spans[e][0]) for e in chosen), sum(keys[e] for e in chosen)
        if not chosen or pairs < EXPAND_FROM_TOKENS * all_keys or pairs * self.heads < EXPAND_FROM_PAIRS:
            return nothing
        rest, other, single = [], [], []                          # (first row, end, first tile, end, entries) of what is left out
        rows, expanded = host.cu_tokens.tolist(), set(chosen)
        for e in (e for e in range(host.n_entries) if e not in expanded):
            a, b = rows[e], rows[e + 1]
            of = single if host.lens[e] == 1 else rest
            if not of or of[-1][1] != a:
                of.append([a, a, len(other), 0, []])
            if of is rest:
                other += prompt_tiles(host, [e], tile, rest[-1][0])
            of[-1][1], of[-1][3] = b, len(other)
            of[-1][4].append(e)
        rest += [[a, b, 0, 0, entries] for a, b, _, _, entries in single]
        price = FIRST_STRETCH * EXPAND_FROM_PAIRS * PAIR_US + STRETCH_US * (len(rest) - 1) if rest else 0.0
        if _saved(pairs, all_keys, max(spans[e][1] - spans[e][0] for e in chosen), self.heads, context, tile) < price:
            return nothing
        pages = []
        table = np.full((host.n_entries, max(spans[e][3] for e in chosen)), -1, dtype=np.int32)
        for e in chosen:
            lo, hi, first, end = spans[e]
            table[e, first:end] = np.arange(len(pages), len(pages) + end - first, dtype=np.int32)
            pages += [(e, b, lo, hi) for b in range(first, end)]
        tiles = prompt_tiles(host, chosen, tile)
        arrays = [np.asarray(x, dtype=np.int32).reshape(-1) for x in (pages, table, tiles, other)]
        return arrays, dict(pages=len(pages), entries=host.n_entries, keys=len(pages) * ops.LATENT_PAGE_KEYS, tile=tile, rest=rest)

    def attach(self, ctx: StepContext, views: List[torch.Tensor], facts: dict) -> None:
        n = facts["pages"]
        ctx.extras[self.key] = (views[0].view(n, 4), views[1].view(facts["entries"], -1), views[2].view(-1, 3), views[3].view(-1, 3),
                                facts) if n else None


class LatentAttention(Part):
    """Attention whose cache holds, per token, a latent c [rank] and one rotated key part [dr]
    shared by all heads, instead of per-head keys and values.

    With h the input: q = W_q h, per head [dn unrotated | dr rotated]; W_dkv h gives rank + dr
    elements, the first rank RMS-normed (weight ``dkv.norm``) into c, the last dr rotated into the
    shared key part.  A head's unrotated key is W_uk c and its value W_uv c; its score against a
    key is (q_n . W_uk c + q_r . k_r) * scale.  Neither keys nor values are kept: the
    unrotated query is taken through W_uk first (q_n^T W_uk) c, so that all heads attend over the
    cached rows [c | k_r] themselves (the score is one dot product over rank + dr elements, the
    weighted sum of the rows' first rank elements is taken through W_uv afterwards).  Softmax in
    float, with ``sink``: one learned term exp(sink_h) more in the denominator, without key or
    value.  With ``gate`` the heads' outputs are multiplied by sigmoid(W_g h) before W_o.
    Prompt portions of some length are the exception: for them the keys and values of the rows they see are
    expanded, used in the flash kernel and dropped (csrc/latent_expand.hip), which costs a third of the
    products; the cache is the same.

    ``q_rank``: queries come through a latent of their own, q = W_uq rms_norm(W_dq h) (weight
    ``dq.norm``), instead of W_q h.

    ``own_latent=False``: the layer has no W_dkv and attends over the rows another layer stored
    (the schedule hands it that layer's cache with ``write=False``).  ``window_kind`` / ``window``: which
    keys this layer sees; ``kept`` (kind, window): which the shared rows have to be kept for, where layers
    with different windows read them (default: this layer's own).  ``rotary``: any object with
    ``table(device)`` (float32 frequencies of the rotated pairs, at most dr / 2), a ``pair_layout`` and a
    ``magnitude`` (of cos and sin).  The kernels turn pairs (2i, 2i + 1); with the layout "half" (pairs (i, i + r / 2)) the
    rows of W_q (or W_uq) and W_dkv that make the rotated parts are put in that order when they are loaded: a score
    is a sum over the part's elements, so it does not change when queries and keys are reordered alike.
    """

    NAMES = {"q": "q", "dq": "dq", "dq_norm": "dq.norm", "uq": "uq", "dkv": "dkv", "dkv_norm": "dkv.norm", "uk": "uk", "uv": "uv", "sink": "sink", "g": "g", "o": "o"}

    def __init__(self, hidden: int, num_heads: int, nope_dim: int, rope_dim: int, v_dim: int, rank: int, rotary,
                 norm_eps: float, scale: float, sink: bool = True, gate: bool = True, own_latent: bool = True,
                 window_kind: int = WINDOW_NONE, window: int = 0, names: Optional[Dict[str, str]] = None,
                 q_rank: Optional[int] = None, kept: Optional[Tuple[int, int]] = None):
        if rank < 1 or rank > ops.LATENT_MAX_RANK:
            raise ValueError(f"a latent of {rank} elements is not taken: 1 to {ops.LATENT_MAX_RANK}")
        if min(num_heads, nope_dim, rope_dim, v_dim) < 1:
            raise ValueError("heads and head sizes must be positive")
        if rotary is not None and (rotary.pair_layout not in ("interleaved", "half") or rotary.rotary_dim > rope_dim):
            raise ValueError("the rotated part takes interleaved or half-split pairs, at most as many as it is wide")
        self.hidden, self.nh, self.dn, self.dr, self.dv, self.rank = (int(hidden), int(num_heads), int(nope_dim),
                                                                     int(rope_dim), int(v_dim), int(rank))
        self.rotary, self.eps, self.scale = rotary, float(norm_eps), float(scale)
        self.has_sink, self.has_gate, self.own_latent = bool(sink), bool(gate), bool(own_latent)
        self.window_kind, self.window = int(window_kind), int(window)
        self.kept = (self.window_kind, self.window) if kept is None else (int(kept[0]), int(kept[1]))
        self.q_rank = int(q_rank) if q_rank else 0
        if self.q_rank < 0:
            raise ValueError("the query latent's width must be positive")
        self.w_uq = None
        self.w_q_norm: Optional[torch.Tensor] = None       # float32 [q_rank]
        self.names = {**self.NAMES, **(names or {})}
        self.w_in = None                                   # [q (or dq) | g | dkv] rows: one product of the input
        self.w_uk_t: Optional[torch.Tensor] = None         # [heads, rank, dn]: W_uk per head, transposed
        self.w_uv: Optional[torch.Tensor] = None           # [heads, dv, rank]
        self.w_ukv: Optional[torch.Tensor] = None          # [heads, dn + dv, rank]: both row by row, where prompts expand keys
        self.pages = LatentPages(self.window_kind, self.window, self.nh, self.dn + self.dr + self.dv)
        self.w_o = None
        self.w_norm: Optional[torch.Tensor] = None         # float32 [rank]
        self.w_sink: Optional[torch.Tensor] = None         # float32 [heads]

    # -- what it needs --------------------------------------------------------
    def step_planners(self):
        return (_WORK_LISTS, self.pages) if self.w_ukv is not None else (_WORK_LISTS,)     # (known once the weights are there)

    def cache_spec(self) -> KVSpec:
        return KVSpec(1, self.rank + self.dr, *self.kept, self.rank, values_in_keys=True)

    @property
    def q_dim(self) -> int:
        return self.nh * (self.dn + self.dr)

    @property
    def o_dim(self) -> int:
        return self.nh * self.dv

    def param_specs(self, prefix: str) -> Dict[str, ParamSpec]:
        n = self.names
        specs = {
            prefix + n["uk"]: ParamSpec((self.nh * self.dn, self.rank)),
            prefix + n["uv"]: ParamSpec((self.o_dim, self.rank)),
            prefix + n["o"]: ParamSpec((self.hidden, self.o_dim)),
        }
        if self.q_rank:
            specs[prefix + n["dq"]] = ParamSpec((self.q_rank, self.hidden))
            specs[prefix + n["dq_norm"]] = ParamSpec((self.q_rank,), "norm_weight")
            specs[prefix + n["uq"]] = ParamSpec((self.q_dim, self.q_rank))
        else:
            specs[prefix + n["q"]] = ParamSpec((self.q_dim, self.hidden))
        if self.own_latent:
            specs[prefix + n["dkv"]] = ParamSpec((self.rank + self.dr, self.hidden))
            specs[prefix + n["dkv_norm"]] = ParamSpec((self.rank,), "norm_weight")
        if self.has_sink:
            specs[prefix + n["sink"]] = ParamSpec((self.nh,))
        if self.has_gate:
            specs[prefix + n["g"]] = ParamSpec((self.o_dim, self.hidden))
        return specs

    def _pair_order(self) -> Optional[torch.Tensor]:
        """Where each element of a rotated part comes from when its pairs are to lie side by side; None: they do."""
        if self.rotary is None or self.rotary.pair_layout == "interleaved":
            return None
        r = self.rotary.rotary_dim
        turned = torch.arange(r).view(2, r // 2).t().reshape(-1)
        return torch.cat([turned, torch.arange(r, self.dr)])

    def _query_rows(self, w: torch.Tensor) -> torch.Tensor:
        order = self._pair_order()
        if order is None:
            return w
        rows = torch.cat([torch.arange(self.dn), self.dn + order])
        return w.view(self.nh, self.dn + self.dr, -1)[:, rows.to(w.device)].reshape(w.shape).contiguous()

    def _latent_rows(self, w: torch.Tensor) -> torch.Tensor:
        order = self._pair_order()
        if order is None:
            return w
        return w[torch.cat([torch.arange(self.rank), self.rank + order]).to(w.device)].contiguous()

    def load(self, prefix: str, source: TensorSource) -> None:
        n = self.names
        parts = [source.get(prefix + n["dq"]) if self.q_rank else self._query_rows(source.get(prefix + n["q"]))]
        if self.q_rank:
            self.w_q_norm = source.get(prefix + n["dq_norm"]).float().contiguous()
            self.w_uq = ops.pack_weight(self._query_rows(source.get(prefix + n["uq"])))
        if self.has_gate:
            parts.append(source.get(prefix + n["g"]))
        if self.own_latent:
            parts.append(self._latent_rows(source.get(prefix + n["dkv"])))
            self.w_norm = source.get(prefix + n["dkv_norm"]).float().contiguous()
        dt = torch.float32 if any(p.dtype == torch.float32 for p in parts) else parts[0].dtype
        fused = torch.empty(sum(p.shape[0] for p in parts), self.hidden, dtype=dt, device=parts[0].device)
        o = 0
        for p in parts:
            fused[o:o + p.shape[0]].copy_(p)
            o += p.shape[0]
        self.w_in = ops.pack_weight(fused)
        uk = source.get(prefix + n["uk"]).to(dt)
        self.w_uk_t = uk.view(self.nh, self.dn, self.rank).transpose(1, 2).contiguous()
        self.w_uv = source.get(prefix + n["uv"]).to(dt).view(self.nh, self.dv, self.rank).contiguous()
        # (with a gate per output element the shared form rounds once, behind the gate; the flash kernel would round before it too)
        if dt == torch.bfloat16 and uk.is_cuda and not self.has_gate and ops.latent_expand_ok(dt, self.dn, self.dr, self.dv, self.rank):
            self.w_ukv = torch.cat([uk.view(self.nh, self.dn, self.rank), self.w_uv], dim=1).contiguous()
        self.w_o = ops.pack_weight(source.get(prefix + n["o"]))
        if self.has_sink:
            self.w_sink = source.get(prefix + n["sink"]).float().contiguous()

    # -- compute --------------------------------------------------------------
    def forward(self, x: torch.Tensor, ctx: StepContext, cache: LayerCache) -> torch.Tensor:
        g = cache.group
        T = x.shape[0]
        D = self.rank + self.dr
        width = 2 if ctx.act_dtype == torch.bfloat16 else 4
        n_in = self.w_in.shape[0]
        g_off = self.q_rank or self.q_dim
        kv_off = g_off + (self.o_dim if self.has_gate else 0)
        with section("q|g|dkv", nbytes=width * n_in * (self.hidden + T) + width * T * self.hidden, flops=2.0 * T * self.hidden * n_in):
            proj = ops.linear(x, self.w_in, ctx.act_dtype)
        store = self.own_latent and cache.write
        if self.own_latent and not cache.write:
            raise ValueError("a latent layer with a down projection of its own must own its cache")
        inv_freq = self.rotary.table(x.device) if self.rotary is not None else None
        rows = (cache.k, g.slot_mapping) if store else (None, None)
        common = (ctx.positions, inv_freq, self.w_norm, self.eps, self.nh, self.dn, self.dr, self.rank)
        magnitude = getattr(self.rotary, "magnitude", 1.0)
        pages = self._pages_to_expand(ctx, proj)
        q_full = None if pages is not None else torch.empty(T, self.nh * D, dtype=ctx.act_dtype, device=x.device)
        if self.q_rank:
            with section("latents + cache write", nbytes=width * T * (2 * self.q_rank + 2 * D)):
                cq = ops.latent_prep(None, 0, kv_off if store else None, None, *rows, *common, magnitude=magnitude, kv=proj,
                                     q_latent=(proj, 0, self.w_q_norm))
            with section("uq", nbytes=width * (self.q_dim * self.q_rank + T * (self.q_rank + self.q_dim)), flops=2.0 * T * self.q_dim * self.q_rank):
                q = ops.linear(cq, self.w_uq, ctx.act_dtype)
            if q_full is not None:
                with section("rotary", nbytes=width * T * 2 * self.nh * self.dr):
                    ops.latent_prep(q, 0, None, q_full, None, None, *common, magnitude=magnitude)
        else:
            q = proj
            if q_full is not None or store:
                with section("latent + rotary + cache write", nbytes=width * T * (2 * self.nh * self.dr + 2 * D)):
                    ops.latent_prep(q, 0, kv_off if store else None, q_full, *rows, *common, magnitude=magnitude)
        gate = proj if self.has_gate else None
        if pages is not None:
            o = self._attend_expanded(q, pages, ctx, cache, inv_freq, magnitude)
        else:
            o = torch.empty(T, self.o_dim, dtype=ctx.act_dtype, device=x.device)
            self._attend_shared(q, q_full, gate, g_off, o, ctx, cache)
        with section("o", nbytes=width * self.hidden * (self.o_dim + T) + width * T * self.o_dim, flops=2.0 * T * self.hidden * self.o_dim):
            return ops.linear(o, self.w_o, ctx.act_dtype)

    def _attend_shared(self, q: torch.Tensor, q_full: torch.Tensor, gate: Optional[torch.Tensor], g_off: int, o: torch.Tensor, ctx,
                       cache: LayerCache) -> None:
        """Attention over the shared rows into o [T, o_dim]: queries through W_uk (q_full holds their rotated parts), the
        weighted latents through W_uv."""
        T, D, width = q.shape[0], self.rank + self.dr, q.element_size()
        with section("q through uk", nbytes=width * (self.nh * self.dn * self.rank + T * self.nh * (self.dn + self.rank)),
                     flops=2.0 * T * self.nh * self.dn * self.rank):
            ops.head_gemm(q, 0, self.dn + self.dr, self.w_uk_t, q_full, 0, D)
        with section("attention", nbytes=lambda: self._keys_held(ctx) * D * width + T * self.nh * (D + self.rank) * width,
                     flops=lambda: 2.0 * self._keys_read(ctx) * self.nh * (D + self.rank)):
            o_lat = ops.attention_latent(q_full, cache.k, cache.group, ctx, self.scale, self.nh, self.rank, self.dr, sink=self.w_sink,
                                         window_kind=self.window_kind, window=self.window)
        with section("uv + gate", nbytes=width * (self.o_dim * self.rank + T * (self.nh * self.rank + 2 * self.o_dim)),
                     flops=2.0 * T * self.o_dim * self.rank):
            ops.head_gemm(o_lat, 0, self.rank, self.w_uv, o, 0, self.dv, gate=gate, gate_off=g_off)

    def _pages_to_expand(self, ctx: StepContext, proj: torch.Tensor):
        """The step's pages where prompt portions of it attend over expanded keys and values, else None: bfloat16 layers of
        widths the kernels take, portions long enough to pay for the expansion (single tokens and the
        rest keep to the shared rows)."""
        if self.w_ukv is None or ctx.act_dtype != torch.bfloat16 or proj.shape[1] % 8 or self.window_kind not in (WINDOW_NONE, WINDOW_SLIDING):
            return None
        return ctx.extras.get(self.pages.key)

    def _attend_expanded(self, q: torch.Tensor, pages, ctx: StepContext, cache: LayerCache, inv_freq: Optional[torch.Tensor],
                         magnitude: float) -> torch.Tensor:
        listed, table, tiles, other, facts = pages
        T, hd = q.shape[0], self.dn + self.dr
        with section("expand uk, uv", nbytes=2 * facts["keys"] * (self.rank + self.dr + self.nh * (hd + self.dv)),
                     flops=2.0 * facts["keys"] * self.nh * (self.dn + self.dv) * self.rank):
            k, v = ops.latent_expand(cache.k, cache.group, listed, self.w_ukv, self.dn, self.dr, self.dv, self.rank)
        with section("rotary", nbytes=2 * T * 2 * self.nh * hd):
            qr = ops.latent_queries(q, ctx.positions, inv_freq, magnitude, self.nh, self.dn, self.dr)
        with section("attention", nbytes=2 * (facts["keys"] + T) * self.nh * (hd + self.dv),
                     flops=lambda: 2.0 * self._keys_read(ctx) * self.nh * (hd + self.dv)):
            o = ops.attention_prefill(qr, k, v, table, ctx.positions, tiles, self.window_kind, self.window, self.scale, self.nh,
                                      self.nh, hd, tile_tokens=facts["tile"], sink=self.w_sink, vd=self.dv)
        # the step's other rows, over the shared rows: its single tokens, and the stretches of portions that do not pay
        for a, b, t0, t1, entries in facts["rest"]:
            single = t0 == t1
            alone = SimpleNamespace(entry_of_token=ctx.entry_of_token[a:b], positions=ctx.positions[a:b], n_decode=b - a if single else 0,
                                    decode_tokens=None, n_prefill_tiles=t1 - t0, prefill_tiles=None if single else other[t0:t1],
                                    prefill_tile_tokens=facts["tile"], entry_lens=[ctx.entry_lens[e] for e in entries],
                                    entry_starts=[ctx.entry_starts[e] for e in entries])
            q_full = torch.empty(b - a, self.nh * (self.rank + self.dr), dtype=q.dtype, device=q.device)
            ops.latent_prep(q[a:b], 0, None, q_full, None, None, alone.positions, inv_freq, self.w_norm, self.eps, self.nh, self.dn, self.dr,
                            self.rank, magnitude=magnitude)
            self._attend_shared(q[a:b], q_full, None, 0, o[a:b], alone, cache)
        return o

    def _keys_read(self, ctx: StepContext) -> int:
        spec = KVSpec(1, 1, self.window_kind, self.window)
        return sum(p - spec.first_visible(p) + 1 for s, n in zip(ctx.entry_starts, ctx.entry_lens) for p in range(s, s + n))

    def _keys_held(self, ctx: StepContext) -> int:
        spec = KVSpec(1, 1, self.window_kind, self.window)
        return sum(s + n - spec.first_visible(s) for s, n in zip(ctx.entry_starts, ctx.entry_lens))
