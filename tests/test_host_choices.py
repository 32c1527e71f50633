"""Choices the host makes without a GPU: the shapes of the few-rows product's launches, the
benchmark's refusal of more than one GPU, the byte counts its roofline is priced with."""
import json
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_few_rows_launch_shapes_follow_the_rows_and_the_compute_units():
    from sharpinference_amd import ops

    # the waves that split K are the same whatever the rows: a row's sums do not change with the batch
    assert {ops.skinny_plan(N, K, rb, g)[1] for N in (5120, 7168, 16384, 202048) for K in (5120, 8192)
            for rb in (1, 2, 4) for g in (1, 2, 9, 17)} == {8}
    # one block of rows: two tiles a block (two K units in flight), wide or not
    assert ops.skinny_plan(7168, 5120, 1)[0] == 2 and ops.skinny_plan(202048, 5120, 1)[0] == 2
    assert ops.skinny_plan(16384, 5120, 1, 9, act=True)[0] == 2
    # ... unless that makes between one and two blocks per compute unit: the merged down projection of one token
    assert ops.skinny_plan(5120, 8192, 1, 2)[0] == 1 and ops.skinny_plan(5120, 8192, 1, 9)[0] == 2
    assert ops.skinny_plan(5120, 5120, 1, 1)[0] == 2            # 160 blocks: every unit has at most one
    assert ops.skinny_plan(16384, 5120, 1, 1, act=True)[0] == 2  # the gated form pairs tiles: never one
    # more rows: four tiles for wide matrices
    assert ops.skinny_plan(16384, 5120, 4, 17)[0] == 4 and ops.skinny_plan(5120, 8192, 4, 17)[0] == 2


def test_the_decode_attention_s_runs_cover_every_window():
    """The decode attention cuts a token's visible keys into runs of 256, counted from the 16-key
    block that holds the first visible key, and sizes its workspace for a bound on the contexts.
    The bound's runs cover every token below it: all keys, chunks, and sliding windows that start
    inside a 16-key block (a window of 257 keys that starts at key 15 spans two runs)."""
    from sharpinference_amd import ops
    from sharpinference_amd.cache.spec import KVSpec, WINDOW_CHUNK, WINDOW_NONE, WINDOW_SLIDING

    run = ops.DECODE_RUN_KEYS
    assert run % 16 == 0
    specs = [KVSpec(1, 16, WINDOW_NONE, 0)] + [KVSpec(1, 16, kind, w) for kind in (WINDOW_CHUNK, WINDOW_SLIDING)
                                                for w in (1, 17, 24, 250, 256, 300, 1000, 4099)]
    for context in (1, 15, 16, 17, 255, 256, 257, 511, 513, 4096, 4097, 9000):
        bound = ops.decode_max_splits(context)
        assert bound == (context - 1) // run + 1            # the runs a context spans from key 0
        for spec in specs:
            for p in {0, context // 3, context - 2, context - 1} - {-1}:
                if p < 0:
                    continue
                s = spec.first_visible(p)
                wanted = ((p >> 4) - (s >> 4)) // (run // 16) + 1     # what the kernels walk (attention_decode.hip)
                assert (s >> 4) * 16 + wanted * run > p               # ... reaches the token's own key
                assert (s >> 4) * 16 + (wanted - 1) * run <= p        # ... with no run to spare
                assert wanted <= bound, (context, spec, p)


def test_benchmark_refuses_more_than_one_gpu():
    out = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True, timeout=120)
    assert out.returncode == 2
    assert len(out.stdout.strip().splitlines()) == 1 and "one GPU" in out.stdout


def test_roofline_bytes_count_every_weight_once_and_the_live_cache():
    sys.path.insert(0, ROOT)
    import bench
    from sharpinference_amd import load_config

    cfg = load_config(dict(bench.SCOUT, num_hidden_layers=48, no_rope_layers=[0 if (l + 1) % 4 == 0 else 1 for l in range(48)]))
    H, I, V = cfg.hidden_size, cfg.intermediate_size, cfg.vocab_size
    attn = H * (cfg.num_attention_heads + 2 * cfg.num_key_value_heads) * cfg.head_dim + cfg.num_attention_heads * cfg.head_dim * H
    expert = 3 * H * I
    router = cfg.num_local_experts * H
    ctx, batch, distinct = 2100, 8, 6.5
    kv = 2 * cfg.num_key_value_heads * cfg.head_dim * ctx * batch
    want = 2 * (48 * (attn + router + (distinct + 1) * expert + kv) + V * H)
    got = bench.decode_step_bytes(cfg, 48, batch, ctx, distinct)
    assert abs(got - want) / want < 0.01, (got, want)
    json.dumps({"bytes": got})


def test_attention_work_lists_cut_a_step_into_decode_tokens_and_tiles():
    """What the attention parts ask the step function to upload: the tokens of entries of one
    token, and tiles of the longer entries: 64-token tiles while a step holds few prompt tokens,
    128-token tiles beyond; every token of a longer entry lies in exactly one tile, tiles do
    not cross entries."""
    import numpy as np
    from sharpinference_amd.parts.attention import SHORT_PROMPT_TOKENS, AttentionWorkLists
    from sharpinference_amd.parts.base import HostStep

    def plan(lens):
        cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        host = HostStep(n_entries=len(lens), n_tokens=int(cu[-1]), lens=list(lens), starts=[7 * i for i in range(len(lens))], cu_tokens=cu)
        (dec, tiles), facts = AttentionWorkLists().plan(host)
        return cu, dec, tiles.reshape(-1, 3), facts

    cu, dec, tiles, facts = plan([1, 130, 1, 2, 64])
    assert dec.tolist() == [0, 131] and facts["n_dec"] == 2 and not facts["all_decode"]
    assert facts["tile"] == 64 and facts["n_tiles"] == len(tiles) == 3 + 1 + 1
    assert tiles.tolist() == [[1, 1, 64], [1, 65, 64], [1, 129, 2], [3, 132, 2], [4, 134, 64]]
    cu, dec, tiles, facts = plan([1, 1, 1])
    assert facts["all_decode"] and facts["n_tiles"] == 0 and tiles.size == 0 and dec.tolist() == [0, 1, 2]
    for lens in ([SHORT_PROMPT_TOKENS], [SHORT_PROMPT_TOKENS + 1], [700, 1, 900, 300], [4096, 5]):
        cu, dec, tiles, facts = plan(lens)
        assert facts["tile"] == (64 if sum(n for n in lens if n > 1) <= SHORT_PROMPT_TOKENS else 128)
        covered = np.zeros(int(cu[-1]), dtype=np.int32)
        for e, t0, rows in tiles.tolist():
            assert 1 <= rows <= facts["tile"] and cu[e] <= t0 and t0 + rows <= cu[e + 1]
            covered[t0:t0 + rows] += 1
        want = np.concatenate([np.full(n, 1 if n > 1 else 0) for n in lens])
        assert covered.tolist() == want.tolist()
    # under a graph's trial run the lists hold harmless contents of the same sizes
    host = HostStep(n_entries=3, n_tokens=3, lens=[1, 1, 1], starts=[5, 6, 7], cu_tokens=np.arange(4, dtype=np.int32))
    arrays, _ = AttentionWorkLists().plan(host)
    null = AttentionWorkLists().null(host, arrays)
    assert [a.size for a in null] == [a.size for a in arrays] and null[0].tolist() == [0, 1, 2]


def test_recurrent_states_take_products_only_where_they_are_the_faster_form():
    """A layer's choice between walking all entries and running the long ones as matrix products, at steps where both were timed
    (microseconds of the walk, and of the products behind the walk of the short entries)."""
    from types import SimpleNamespace

    import numpy as np

    from sharpinference_amd import ops
    from sharpinference_amd.parts.base import HostStep
    from sharpinference_amd.parts.linear_attention import WALK_SEGMENTS
    from sharpinference_amd.parts.matrix_memory import _segments_for

    def takes(lens, nh, dk, dv, turned=False):
        cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        arrays, facts = WALK_SEGMENTS.plan(HostStep(len(lens), int(cu[-1]), list(lens), [0] * len(lens), cu))
        ctx = SimpleNamespace(extras={}, n_entries=len(lens), n_tokens=int(cu[-1]), max_entry_len=max(lens))
        WALK_SEGMENTS.attach(ctx, arrays, facts)
        chosen = _segments_for(ctx, nh, dk, dv, turned)
        assert chosen is None or tuple(chosen[2]) == ops.segment_counts(lens)
        return chosen is not None

    for lens, nh, dk, dv, turned, walk, products in (
            ([64] + [1] * 256, 64, 128, 64, False, 185, 219), ([200] + [1] * 256, 64, 128, 64, False, 193, 352),
            ([300] + [1] * 256, 128, 128, 64, False, 384, 639), ([64] + [1] * 256, 16, 128, 128, True, 97, 154),
            ([200] + [1] * 256, 32, 128, 128, False, 247, 427), ([64] + [1] * 64, 32, 128, 128, True, 65, 100), ([96] + [1] * 64, 16, 128, 128, True, 77, 97),
            ([1000, 900] + [1] * 16, 16, 128, 128, False, 736, 97), ([2000], 16, 128, 128, False, 1436, 76),
            ([2000], 64, 128, 64, False, 1072, 140), ([500] * 4, 16, 128, 128, True, 353, 119), ([1500] + [1] * 64, 4, 64, 64, True, 606, 46),
            ([64], 64, 128, 64, False, 34, 20), ([64] * 6, 16, 128, 128, False, 60, 25), ([64] * 30, 16, 128, 128, True, 136, 109)):
        assert takes(lens, nh, dk, dv, turned) == (products < walk), (lens[0], len(lens), nh)
    assert not takes([63] * 3, 16, 128, 128) and not takes([1] * 64, 16, 128, 128)        # steps without a list


def test_segments_are_cut_to_what_the_kernels_hold():
    """The tokens of a segment and those from which an entry is run in products are the library's own numbers, checked when it is
    loaded; every list keeps to them, its entries of several segments first and the short ones last."""
    import numpy as np

    from sharpinference_amd import ops
    from sharpinference_amd.ops import lib

    assert lib._BUILT_WITH["sharpi_state_segment_tokens"] == ops.GLA_SEGMENT_TOKENS
    assert lib._BUILT_WITH["sharpi_state_chunk_from"] == ops.WALK_CHUNK_FROM
    lens = [1, 300, 31, 32, 128, 129, 7, 1000]
    cu = np.concatenate([[0], np.cumsum(lens)])
    segs, ents = ops.gla_segments(lens, cu)
    assert int(segs[:, 2].max()) == ops.GLA_SEGMENT_TOKENS
    for e, (first, count) in enumerate(ents):
        mine = segs[first:first + count]
        assert (mine[:, 0] == e).all() and mine[:, 3].tolist() == [0] * (count - 1) + [1]
        assert mine[:, 1].tolist() == [cu[e] + 128 * i for i in range(count)] and mine[:, 2].sum() == lens[e]
    assert [segs[first, 0] for first, _ in ents] == list(range(len(lens)))                # (every entry's own, whatever the order)
    several, long = ops.segment_counts(lens)
    single = ents[segs[:, 0], 1] == 1
    assert (several, long) == (3 + 2 + 8, 3 + 2 + 8 + 2) and not single[:several].any() and single[several:].all()
    assert (segs[several:long, 2] >= ops.WALK_CHUNK_FROM).all() and (segs[long:, 2] < ops.WALK_CHUNK_FROM).all()


def test_segments_are_listed_for_the_layers_that_may_take_them():
    """Layers with a decay per key channel, which walk their segments, have lists from 512 tokens on; layers with one decay a head,
    whose segments are products, from 64."""
    import numpy as np

    from sharpinference_amd.parts.base import HostStep
    from sharpinference_amd.parts.linear_attention import GatedLinearAttention
    from sharpinference_amd.parts.matrix_memory import MatrixMemory

    parts = GatedLinearAttention.__new__(GatedLinearAttention), MatrixMemory.__new__(MatrixMemory)
    for n, made in ((63, [0, 0]), (64, [0, 1]), (511, [0, 1]), (512, [1, 1])):
        lens = [1, n, 5]
        cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        host = HostStep(3, int(cu[-1]), lens, [0] * 3, cu)
        assert [int(p.step_planners()[0].plan(host)[1]["n_segs"] > 0) for p in parts] == made
    assert parts[0].step_planners()[0].key != parts[1].step_planners()[0].key


def _latent_pages(lens, starts, kind=0, window=0, heads=64, width=320):
    """The step's plan of a latent layer -> (entries whose keys are expanded, pages, block table, tiles, the other tiles, facts)"""
    import numpy as np

    from sharpinference_amd.parts.base import HostStep
    from sharpinference_amd.parts.latent_attention import LatentPages

    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    (pages, table, tiles, other), facts = LatentPages(kind, window, heads, width).plan(HostStep(len(lens), int(cu[-1]), lens, starts, cu))
    pages = pages.reshape(-1, 4).tolist()
    return sorted({p[0] for p in pages}), pages, table.reshape(len(lens), -1), tiles.reshape(-1, 3).tolist(), other.reshape(-1, 3).tolist(), facts


def test_prompt_portions_expand_their_keys_where_it_is_the_faster_form():
    from sharpinference_amd.cache.spec import WINDOW_SLIDING

    # a long prompt beside a few tokens behind a long context: the context's keys stay as they are
    chosen, pages, table, tiles, other, facts = _latent_pages([2000, 2], [0, 30000])
    assert chosen == [0] and len(pages) == 16 and table[0, :16].tolist() == list(range(16)) and int(table[1].max()) == -1
    assert sum(t[2] for t in tiles) == 2000 and other == [[1, 0, 2]] and facts["rest"] == [[2000, 2002, 0, 1, [1]]]
    assert _latent_pages([2000, 2], [0, 30000], heads=16)[0] == [0]
    # ... unless the flash kernel walks them faster than the shared rows are walked
    assert _latent_pages([1000, 4], [0, 24000], heads=16)[0] == [0, 1] and _latent_pages([1000, 4], [0, 3000])[0] == [0, 1]
    assert _latent_pages([2000, 2], [0, 30000], WINDOW_SLIDING, 1024)[0] == [0, 1]
    assert _latent_pages([2000, 300], [0, 20000])[0] == [0, 1]                    # (queries enough for their keys)
    # a context whose expanded keys would not fit leaves the other prompts theirs
    assert _latent_pages([2000, 4000], [0, 60000])[0] == [0] and _latent_pages([2000, 4000], [0, 60000], heads=16)[0] == [0, 1]
    # too little work in all, portions that are too short
    assert _latent_pages([80], [0], heads=16)[0] == [] and _latent_pages([100] * 6, [0] * 6, heads=16)[0] == list(range(6))
    assert _latent_pages([31, 1, 1], [2000, 5, 6])[0] == [] and _latent_pages([64, 1, 1], [2000, 5, 6])[0] == [0]
    assert _latent_pages([40], [2000])[0] == [] and _latent_pages([40], [2000], heads=16)[0] == [0]
    assert _latent_pages([1] * 8, [2000] * 8)[0] == []
    # what is left out: neighbouring portions together, the single tokens apart
    far = 30000
    chosen, _, _, tiles, other, facts = _latent_pages([1, 1, 5, 9, 1000, 3, 900, 2, 4], [9, 9, far, far, 0, far, 64, far, far])
    assert chosen == [4, 6]
    assert facts["rest"] == [[2, 16, 0, 2, [2, 3]], [1016, 1019, 2, 3, [5]], [1919, 1925, 3, 5, [7, 8]], [0, 2, 0, 0, [0, 1]]]
    assert other == [[2, 0, 5], [3, 5, 9], [5, 0, 3], [7, 0, 2], [8, 2, 4]]
    assert [t for t in tiles if t[0] == 6][0][:2] == [6, 1019] and sum(t[2] for t in tiles) == 1900
    # rows left to the shared form, a stretch each for neighbours: only where the prompts' work is enough for the launches
    assert _latent_pages([1, 700, 1, 1], [9, 0, 9, 9])[5]["rest"] == [[0, 1, 0, 0, [0]], [701, 703, 0, 0, [2, 3]]]
    for n, heads, behind, alone, beside, around in ((200, 64, 0, 1, 0, 0), (1000, 16, 0, 1, 1, 1), (400, 64, 0, 1, 1, 0), (100, 16, 2000, 1, 1, 1), (1500, 16, 0, 1, 1, 1)):
        chosen = [_latent_pages(lens, [behind if n > 1 else 50 for n in lens], heads=heads)[0] for lens in ([n], [1] * 8 + [n], [1, n, 1])]
        assert [len(c) for c in chosen] == [alone, beside, around], (n, heads, behind, chosen)
