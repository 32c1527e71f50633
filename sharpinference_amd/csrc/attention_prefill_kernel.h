// Attention for entries of several tokens (prompt portions): flash attention on the matrix cores
// over the paged cache, causal and window masks applied per element.
//
// A block owns a tile of up to 128 consecutive tokens of one entry and one query head; each of its
// four waves takes 32 of the tokens (or, for tiles of up to 64 tokens, 16: a row's sums are the same
// either way).  As in the decode kernel everything is transposed:
//   S^T[key, q]  = K[key, :] . Q[q, :]          A = K block, B = Q^T
//   O^T[d, q]   += V^T[d, key] * P^T[key, q]    A = V^T block (values are stored transposed
//                                               inside a page), B = P^T
// and the S^T accumulator of a lane is the B operand of the second product once exponentiated
// and split into a bfloat16 pair hi + lo (two products: the probabilities keep ~16 bits; the row's
// sum is taken from the unrounded values).  Softmax state (a reference maximum and the sum per query)
// is float, kept in base-2 units (scores times log2 e, the hardware's exp2).
// The keys of a query are always visited in the same chunks (pairs of 16-key blocks at absolute
// positions), whatever tile it sits in.
//
// Keys and values go from the cache straight into LDS (loads that write LDS, no registers between), a
// stage of 64 keys ahead: wave w fetches the stage's 16-key block w, so a stage needs one page number a
// wave, itself requested a stage earlier, and a barrier covers 96 products of a wave.  The cache's order
// is kept in 16-byte pieces; a key row's are XORed with row bits so that the operand reads are free
// of bank conflicts (k_swizzle).  Heads of one kv head run on one die and share its L2.
//
// What bounds it: per 32 keys and 32 rows a wave issues 48 products of 16 cycles (128-wide heads) and about
// 150 vector instructions a lane for the softmax, on one SIMD that two waves share.
// 40 heads of 128 sharing 8 key heads, 8,192 tokens: 1,041 us (660 TFLOP/s, the pair's second product not counted); 1,452 us with
// 32-key chunks on their way through registers and divisions by the page size in every chunk.  2,048 tokens: 98 us (133); 64 heads of
// 192 / 128, window 1,024, 2,048 tokens: 139 us (180); 16 heads, 1,900 tokens: 49 us (75).  Three prompts of 400 tokens in
// tiles of 64: 32 us (35).  On 32x32x16 products, eight consecutive keys a lane, it took 904, 76, 111 and 47 us: other sums of the
// same exactness, whose roundings turned routers' near ties in whole models; these are the bits of the kernel before.
#pragma once
#include <type_traits>

#include "common.h"
#include "lds_loads.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

#ifndef SHARPI_PREFILL_P_PAIR
// 1: probabilities enter the second product as a bfloat16 pair hi + lo.  0 (hi alone) is faster, but then
// rounds every probability to 8 bits, which the comparison with a float softmax does not forgive where
// the softmax is sharp: random mixed traces at a weight scale of 0.08 left the derived bfloat16 bound by
// up to a quarter in 4 of 60, none with the pair.
#define SHARPI_PREFILL_P_PAIR 1
#endif
constexpr int kPreWaves = 4;
constexpr int kTileTokens = 32 * kPreWaves;          // 128 tokens per block at most

// LDS layouts.  The LDS serves a 16-byte read of a wave in four turns of two octets of lanes: one
// octet holding operand rows 0..7 and one holding rows 8..15 of the neighbouring lane group (measured
// with the bank-conflict counter).  The 16 pieces of 16
// bytes that a turn reads must fall into the 16 different 16-byte groups of the 256-byte bank space:
// a piece's number is XORed with row bits, as many as rows share a group.
template <int HD> __device__ __forceinline__ constexpr int k_swizzle(int row) {
  return HD % 128 == 0 ? (row & 15) : HD % 64 == 0 ? ((row >> 1) & 7) : ((row >> 2) & 3);
}
// values: a 16-key block is kept as rows of 32 bytes, one a value column: a wave's 8-byte reads are 512 bytes in a row.

constexpr float kLazyMax = 8.0f;                     // how far the row maximum may outgrow its reference
// the reference before a row has seen a key: finite, so that a masked score (-inf) minus it is
// -inf and its probability 0, and far below any score, so that the first key moves it
constexpr float kNoMax = -1.0e30f;

struct PrefillArgs {
  const void *q, *k_cache, *v_cache;
  const int *block_table, *positions, *tiles;
  void* out;
  int n_tiles, tile_tokens, window_kind, window;
  float scale;
  int nh, nkv, page_size, max_blocks, num_pages;
  float softcap;
  int sink;
  const float* sink_vals;
  int keep;                    // a window's first tokens that stay visible (0: none)
  const void* gate;            // bf16, column h of row t gates head h of token t (null: no gate)
  int gate_stride;
};

__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  const bf16x2 p = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, p);
}

template <int HD, int VD>
constexpr int prefill_waves_a_simd() { return kPreWaves * 16 * (HD + (VD + 31) / 32 * 32) * 4 <= 80 * 1024 ? 2 : 1; }   // by the LDS two blocks need

// DIRECT: the caches begin at 16-byte addresses (40 heads of 128, 2,048 tokens: 102 us, 146 from odd ones).
template <int HD, int VD, int kQT, bool DIRECT>
__global__ __launch_bounds__(kPreWaves* kWave, (prefill_waves_a_simd<HD, VD>())) void attn_prefill_kernel(
    const bf16_t* __restrict__ q, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
    const int* __restrict__ block_table, const int* __restrict__ positions, const int* __restrict__ tiles,
    bf16_t* __restrict__ out, int window_kind, int window, float scale, int nh, int nkv, int page_size,
    int max_blocks, int num_pages, float softcap, int sink, const float* __restrict__ sink_vals, int keep,
    const bf16_t* __restrict__ gate, int gate_stride) {
  constexpr int WAVES = kPreWaves, kWaveTokens = 16 * kQT;
  constexpr int NJ = HD / 32;                       // product steps of a score
  constexpr int ND = VD / 16;                       // 16-column tiles of the values
  constexpr int VL = (VD + 31) / 32;                // loads of a 16-key block of values (32 columns each; half of the last may be idle)
  constexpr int CH = HD / 8;                        // 16-byte pieces of a key row
  constexpr int KL = HD / 32;                       // loads of a 16-key block of keys (64 pieces each)
  constexpr int KB = 16 * HD * 2, VB = VL * 1024;   // LDS bytes of a 16-key block
  constexpr int STAGE = WAVES * (KB + VB);          // a stage: WAVES blocks of keys, then as many of values
  constexpr int SUBS = WAVES / 2;                   // 32-key chunks of a stage
  static_assert(HD % 32 == 0 && VD % 16 == 0 && WAVES % 2 == 0, "sizes the layouts are made for");
  __shared__ __attribute__((aligned(1024))) char smem[2 * STAGE];

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  // Tiles run from the last backwards (later tiles of a prompt see more keys, and the longest blocks should start first),
  // heads fastest.  Blocks go to the 8 dies round-robin, so where the heads divide by 8 a die takes neighbouring
  // heads: those of one kv head read the same keys and values out of one L2.
  const int linear = blockIdx.x + blockIdx.y * gridDim.x;
  const int ti = gridDim.y - 1 - linear / nh;
  const int hx = linear % nh;
  const int h = nh % 8 == 0 ? (hx % 8) * (nh / 8) + hx / 8 : hx;
  const int kvh = h / (nh / nkv);
  const int entry = tiles[ti * 3], tok0 = tiles[ti * 3 + 1], rows = tiles[ti * 3 + 2];
  const int pos0 = positions[tok0];
  const int* bt = block_table + (size_t)entry * max_blocks;
  auto first_key = [&](int p) {                       // the first key position p sees (kept ones apart)
    if (window_kind == 1) return (p / window) * window;
    if (window_kind == 2) return max(p - window + 1, 0);
    return 0;
  };

  // this wave's tokens: per column tile, the lane's query row, its position, its first key
  const int wrow0 = w * kWaveTokens;
  int qpos[kQT], qstart[kQT];
  bool qok[kQT];
  bf16x8 qf[kQT][NJ];
#pragma unroll
  for (int c = 0; c < kQT; ++c) {
    const int row = wrow0 + c * 16 + r;
    qok[c] = row < rows;
    qpos[c] = pos0 + row;
    qstart[c] = first_key(qpos[c]);
    // rows beyond the tile's last read its last row; their scores are masked and their output is never stored
    const bf16_t* src = q + ((size_t)(tok0 + min(row, rows - 1)) * nh + h) * HD + g * 8;
#pragma unroll
    for (int j = 0; j < NJ; ++j) qf[c][j] = *reinterpret_cast<const bf16x8*>(src + j * 32);
  }
  // waited for here: the compiler would wait where they are first used, inside the loop, and so in every
  // stage for the loads of the next one, which it does not know of
#pragma unroll
  for (int c = 0; c < kQT; ++c)
#pragma unroll
    for (int j = 0; j < NJ; ++j) asm volatile("" : "+v"(qf[c][j]));
  const bool wave_has_rows = wrow0 < rows;
  const bool wave_full = wrow0 + kWaveTokens <= rows;                 // all 32 rows exist
  const int wave_first_pos = pos0 + wrow0;
  const int wave_last = pos0 + min(rows, wrow0 + kWaveTokens) - 1;    // last position of this wave's rows
  const int wave_last_start = first_key(wave_last);                   // first key the wave's last row may see
  const int wave_first = first_key(wave_first_pos);                   // first key the wave's first row may see
  const float scale_log2 = scale * 1.4426950408889634f;               // softmax in base 2: exp(x) = 2^(x log2 e)
  const float cap_log2 = softcap * 1.4426950408889634f;               // capped scores: cap * tanh(score / cap), in base-2 units
  const float scale_by_cap = softcap > 0.f ? scale / softcap : 0.f;
  // Stages are WAVES 16-key blocks aligned to absolute positions; blocks count from the sequence's start.
  const int first = first_key(pos0);                // the first key of the tile's first row
  const int b_first_seen = first >> 4;
  const int b_win = b_first_seen & ~(WAVES - 1);
  const int b_last = (pos0 + rows - 1) >> 4;
  // with kept first tokens the walk begins at their stages (blocks below b_kept) and goes on where the window begins
  const int b_kept = WAVES * ((keep + 16 * WAVES - 1) / (16 * WAVES));
  const int b_first = keep > 0 ? 0 : b_win;
  auto after = [&](int b) { return b + WAVES >= b_kept && b + WAVES < b_win ? b_win : b + WAVES; };
  // The block that wave w fetches of the stage at b: its own, or, where no row sees that one (behind the tile's last key,
  // between kept tokens and window, before the window), the nearest that some row sees: its keys are masked, its values
  // are the sequence's own and meet probabilities of zero.
  auto block_of = [&](int b) {
    int bb = min(b + w, b_last);
    if (bb < b_first_seen && (bb << 4) >= keep) bb = keep > 0 ? (keep - 1) >> 4 : b_first_seen;
    return bb;
  };
  const int per_page = page_size >> 4;              // 16-key blocks of a page
  const uint32_t page_inv = per_page > 1 ? 0xffffffffu / (uint32_t)per_page + 1 : 0;   // bb / per_page = high word of bb * page_inv (exact below 2^32 / per_page)
  auto page_slot = [&](int bb) { return per_page > 1 ? (int)__umulhi((uint32_t)bb, page_inv) : bb; };
  auto page_at = [&](int bb) { return bt[min(page_slot(bb), max_blocks - 1)]; };

  // where this lane's pieces of a 16-key block lie (bytes from the block's start)
  uint32_t k_off[KL];
#pragma unroll
  for (int n = 0; n < KL; ++n) {
    const int f = n * kWave + lane, lrow = f / CH, piece = f % CH;
    k_off[n] = (uint32_t)(lrow * HD + (piece ^ k_swizzle<HD>(lrow)) * 8) * 2;
  }
  uint32_t v_off[VL];
#pragma unroll
  for (int n = 0; n < VL; ++n) {
    const int d = n * 32 + (lane >> 1);
    v_off[n] = (uint32_t)(min(d, VD - 1) * page_size + (lane & 1) * 8) * 2;
  }
  const uint32_t lds0 = lds_address(smem);
  auto fetch = [&](int bb, int page_raw, int buf) {   // 16-key block bb, of the page that page_at gave
    const int page = min(max(__builtin_amdgcn_readfirstlane(page_raw), 0), num_pages - 1);   // a table that is wrong reads a wrong page, never outside
    const int off = min(max((bb - page_slot(bb) * per_page) << 4, 0), page_size - 16);
    const long long head = (long long)page * nkv + kvh;
    const u32x4 kr = buffer_of(k_cache + (head * page_size + off) * HD, KB);
    const u32x4 vr = buffer_of(v_cache + head * VD * page_size + off, (uint32_t)((VD - 1) * page_size + 16) * 2);
    const uint32_t at = lds0 + buf * STAGE;
    uint32_t k_to[KL], v_to[VL];
#pragma unroll
    for (int n = 0; n < KL; ++n) k_to[n] = at + w * KB + n * 1024;
#pragma unroll
    for (int n = 0; n < VL; ++n) v_to[n] = at + WAVES * KB + w * VB + n * 1024;
    bring_all_to_lds<DIRECT, KL>(kr, k_off, 0, k_to);
    bring_all_to_lds<DIRECT, VL>(vr, v_off, 0, v_to);
  };

  // where this lane reads its operands (bytes): piece 4j + g of key row r, keys 4g .. 4g + 3 of value column r
  int k_at[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) k_at[j] = r * HD * 2 + ((4 * j + g) ^ k_swizzle<HD>(r)) * 16;
  const int v_at = WAVES * KB + r * 32 + g * 8;

  float m[kQT], l[kQT];
  f32x4 acc[kQT][ND];
#pragma unroll
  for (int c = 0; c < kQT; ++c) {
    m[c] = kNoMax;
    l[c] = 0.f;
#pragma unroll
    for (int d = 0; d < ND; ++d) acc[c][d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  // One 32-key chunk: keys (b0 << 4) .. + 31, chunk `sub` of the stage in the buffer at `buf`.
  auto chunk = [&](int b0, const char* buf, auto sub_tag, bool whole) {
    constexpr int sub = decltype(sub_tag)::value;
    f32x4 s[kQT][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int c = 0; c < kQT; ++c) s[c][u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(buf + k_at[j] + (sub * 2 + u) * KB);
#pragma unroll
        for (int c = 0; c < kQT; ++c) s[c][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[c][j], s[c][u], 0, 0, 0);
      }
    }
    // the lane holds S^T[key = 16 * (b0 + u) + 4g + i][query row c * 16 + r]; scores go to base-2 units
    if (softcap > 0.f) {
#pragma unroll
      for (int c = 0; c < kQT; ++c)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) s[c][u][i] = cap_log2 * tanhf(s[c][u][i] * scale_by_cap);
    } else {
#pragma unroll
      for (int c = 0; c < kQT; ++c)
#pragma unroll
        for (int u = 0; u < 2; ++u) s[c][u] *= scale_log2;
    }
    if (!whole) {
#pragma unroll
      for (int c = 0; c < kQT; ++c)
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = ((b0 + u) << 4) + 4 * g + i;
            const bool ok = qok[c] && (key >= qstart[c] || key < keep) && key <= qpos[c];
            s[c][u][i] = ok ? s[c][u][i] : -INFINITY;
          }
    }
    float lmax[kQT];
    bool grown = false;
#pragma unroll
    for (int c = 0; c < kQT; ++c) {
      float lm = s[c][0][0];
#pragma unroll
      for (int x = 1; x < 8; ++x) lm = fmaxf(lm, s[c][x >> 2][x & 3]);
      lmax[c] = lm;
      grown = grown || lm - m[c] > kLazyMax;
    }
    // m is a reference, not the running maximum: a row moves it only when the chunk's largest
    // score lies more than kLazyMax (base-2 units) above it.  Probabilities then reach 2^kLazyMax
    // at most, which float sums carry easily.  Most chunks move no row of the wave: they need
    // no exchange between lanes and no rescaling.  The rule is the row's own (its four lanes
    // hold the same m and, once exchanged, the same maximum), so what a row ends up with does
    // not depend on the rows it shares a wave with.
    if (__builtin_amdgcn_ballot_w64(grown) != 0) {   // wave-uniform
#pragma unroll
      for (int c = 0; c < kQT; ++c) {
        float cm = lmax[c];
        cm = reduce16(cm, MaxOf{});
        cm = reduce32(cm, MaxOf{});
        const bool move = cm - m[c] > kLazyMax;
        const float corr = move ? __builtin_amdgcn_exp2f(m[c] - cm) : 1.0f;
        m[c] = move ? cm : m[c];
        l[c] *= corr;
#pragma unroll
        for (int d = 0; d < ND; ++d) acc[c][d] *= corr;
      }
    }
    u32x4 pf[kQT];
#if SHARPI_PREFILL_P_PAIR
    u32x4 pf_lo[kQT];
#endif
#pragma unroll
    for (int c = 0; c < kQT; ++c) {
      float ls = 0.f;
#pragma unroll
      for (int x = 0; x < 8; x += 2) {
        const float e0 = __builtin_amdgcn_exp2f(s[c][x >> 2][x & 3] - m[c]);              // masked: 2^-inf = 0
        const float e1 = __builtin_amdgcn_exp2f(s[c][x >> 2][(x & 3) + 1] - m[c]);
        ls += e0;
        ls += e1;
        const uint32_t hi = bf16_pair(e0, e1);                                            // round to nearest even
        pf[c][x >> 1] = hi;
#if SHARPI_PREFILL_P_PAIR
        pf_lo[c][x >> 1] = bf16_pair(e0 - __uint_as_float(hi << 16), e1 - __uint_as_float(hi & 0xffff0000u));
#endif
      }
      l[c] += ls;
    }
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      // lane (column r, group g): keys 4g..4g+3 of the chunk's first block, then of its second
      const uint2 v0 = *reinterpret_cast<const uint2*>(buf + v_at + (sub * 2) * VB + d * 512);
      const uint2 v1 = *reinterpret_cast<const uint2*>(buf + v_at + (sub * 2 + 1) * VB + d * 512);
      const bf16x8 vf = __builtin_bit_cast(bf16x8, u32x4{v0.x, v0.y, v1.x, v1.y});
#pragma unroll
      for (int c = 0; c < kQT; ++c) {
        acc[c][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, __builtin_bit_cast(bf16x8, pf[c]), acc[c][d], 0, 0, 0);
#if SHARPI_PREFILL_P_PAIR
        acc[c][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, __builtin_bit_cast(bf16x8, pf_lo[c]), acc[c][d], 0, 0, 0);
#endif
      }
    }
  };

  int b_next = after(b_first);
  int page_next = 0;
  {
    const int bb = block_of(b_first);
    fetch(bb, page_at(bb), 0);
    if (b_next <= b_last) page_next = page_at(block_of(b_next));
  }
  int par = 0;
  for (int b = b_first; b <= b_last;) {
    lds_loads_wait();                                  // this wave's part of the stage, and the next page number
    __syncthreads();                                   // every wave's part; and the other buffer has been read
    const int b_two = after(b_next);
    if (b_next <= b_last) {
      fetch(block_of(b_next), page_next, par ^ 1);
      if (b_two <= b_last) page_next = page_at(block_of(b_two));
    }
    const char* buf = smem + par * STAGE;
    auto one = [&](auto sub_tag) {
      constexpr int sub = decltype(sub_tag)::value;
      const int b0 = b + 2 * sub, k0 = b0 << 4;
      // does any row of this wave see a key of this chunk?  does every row see all of them?
      if (!wave_has_rows || k0 > wave_last || (k0 + 32 <= wave_first && k0 >= keep)) return;
      const bool whole = wave_full && k0 + 31 <= wave_first_pos && (k0 >= wave_last_start || k0 + 32 <= keep);
      chunk(b0, buf, sub_tag, whole);
    };
    one(std::integral_constant<int, 0>{});
    if constexpr (SUBS > 1) one(std::integral_constant<int, 1>{});
    static_assert(SUBS <= 2, "a stage is one or two chunks");
    par ^= 1;
    b = b_next;
    b_next = b_two;
  }

#pragma unroll
  for (int c = 0; c < kQT; ++c) {
    float L = l[c];
    L = reduce16(L, SumOf{});
    L = reduce32(L, SumOf{});
    if (!qok[c]) continue;
    // a key of score 0 (or of the head's learned score) without a value: 2^(score log2 e - reference) more
    if (sink) L += __builtin_amdgcn_exp2f((sink_vals ? sink_vals[h] * 1.4426950408889634f : 0.f) - m[c]);
    float inv = L > 0.f ? 1.0f / L : 0.f;
    const size_t token = tok0 + wrow0 + c * 16 + r;
    if (gate) inv *= 1.0f / (1.0f + expf(-bf16_to_f32(gate[token * gate_stride + h])));
    bf16_t* orow = out + (token * nh + h) * VD;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      // lane holds O^T[d*16 + 4g + i][query row]
      const f32x4 o = acc[c][d] * inv;
      uint2 packed;
      packed.x = f32_to_bf16_pair(o[0], o[1]);
      packed.y = f32_to_bf16_pair(o[2], o[3]);
      *reinterpret_cast<uint2*>(orow + d * 16 + 4 * g) = packed;
    }
  }
}

template <int HD, int VD>
static int launch_prefill(const PrefillArgs& a, hipStream_t stream) {
  dim3 grid(a.nh, a.n_tiles);
#define PRE_QT(QTV, DIR)                                                                                                 \
  attn_prefill_kernel<HD, VD, QTV, DIR><<<grid, kPreWaves * kWave, 0, stream>>>(                                                    \
      (const bf16_t*)a.q, (const bf16_t*)a.k_cache, (const bf16_t*)a.v_cache, a.block_table, a.positions, a.tiles,        \
      (bf16_t*)a.out, a.window_kind, a.window, a.scale, a.nh, a.nkv, a.page_size, a.max_blocks, a.num_pages, a.softcap,   \
      a.sink, a.sink_vals, a.keep, (const bf16_t*)a.gate, a.gate_stride)
  const bool direct = whole_pieces(a.k_cache, a.v_cache), full = a.tile_tokens == kTileTokens;
  if (direct && full) PRE_QT(2, true);
  else if (direct) PRE_QT(1, true);
  else if (full) PRE_QT(2, false);
  else PRE_QT(1, false);
#undef PRE_QT
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}
