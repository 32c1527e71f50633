// Attention of the 32-bit path over the paged cache on the float matrix instruction: what attention_generic.hip computes, for
// float rows of the widths it is compiled for and pages of whole 16-key blocks.
//
// Up to 16 (token, head) rows of one kv head walk the keys together: the heads of the group for as many neighbouring
// tokens as fill the tile; a block takes one of a tile's runs of tokens of one entry.
// The four waves take the 16-key blocks in turn by their number in the sequence; S^T = K Q^T and O^T = V^T P^T on
// v_mfma_f32_16x16x4_f32, so that a lane's four exponentiated scores are the second product's operand as they lie,
// and keys and values come straight from memory, four neighbouring elements (keys) a lane.  A row's sums depend on
// (first key, position) alone: keys it does not see add nothing, whoever shares its tile.
//
// Bound: the float matrix instruction (64 products of 16 x 16 x 4 a block of keys at 128 wide heads, for 16 rows) and the
// latency of a wave's loads.  The walk of one row a block read every key once a row, a lane a key: 573 rows of 16 heads
// over 4 kv heads, up to 301 keys: 400 -> 45 us a layer.  Single tokens (a block a kv head and token, where the walk of
// one row had one a head) gain as well: one token of 16 heads behind 30 keys 19 -> 15 us, 2,000 250 -> 99, 16,000 1,990 ->
// 915; 64 tokens behind 2,000 1,102 -> 175.
#include "common.h"

using f32x4 = __attribute__((__vector_size__(4 * sizeof(float)))) float;

constexpr int kFlWaves = 4;

struct FloatAttention {
  const float *q, *k, *v;
  const int *block_table, *entry_of_token, *positions;
  float* out;
  int window_kind, window;
  float scale;
  int n_tokens, nh, nkv, page_size, max_blocks, num_pages;
  float softcap;
  int sink;
  const float* sink_vals;
  int keep;
  const float* gate;
  int gate_stride, tile_tokens;
};

__device__ __forceinline__ int first_key(const FloatAttention& a, int p) {
  if (a.window_kind == 1) return p / a.window * a.window;
  if (a.window_kind == 2) return max(0, p - a.window + 1);
  return 0;
}

template <int HD, int VD>
__global__ __launch_bounds__(kFlWaves* kWave) void attn_float_kernel(FloatAttention a) {
  constexpr int NJ = HD / 16, ND = VD / 16;
  __shared__ f32x4 acc_s[kFlWaves][ND][kWave];
  __shared__ float m_s[kFlWaves][16], l_s[kFlWaves][16];
  const int lane = threadIdx.x & (kWave - 1), w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int G = a.nh / a.nkv, hp = 16 / a.tile_tokens, head_tiles = (G + hp - 1) / hp;
  const int kvh = blockIdx.y / head_tiles, ht = blockIdx.y - kvh * head_tiles;
  // this block's run: the blockIdx.z-th stretch of the tile's tokens that belong to one entry
  const int t0 = blockIdx.x * a.tile_tokens, t1 = min(t0 + a.tile_tokens, a.n_tokens);
  int from = t0, to = t0 + 1;
  for (int z = 0;; ++z) {
    const int e = a.entry_of_token[from];
    to = from + 1;
    while (to < t1 && a.entry_of_token[to] == e) ++to;
    if (z == (int)blockIdx.z) break;
    if (to >= t1) return;
    from = to;
  }
  const int entry = a.entry_of_token[from];
  const int* bt = a.block_table + (size_t)entry * a.max_blocks;

  // the lane's row
  const int token = t0 + r / hp, in_group = ht * hp + r % hp;
  const bool row_ok = token >= from && token < to && in_group < G;
  const int head = kvh * G + (in_group < G ? in_group : G - 1);
  const int p = row_ok ? a.positions[token] : -1;              // (no key lies at or before -1)
  const int start = row_ok ? first_key(a, p) : 0;
  f32x4 qf[NJ];
  {
    const float* qrow = a.q + ((size_t)(row_ok ? token : from) * a.nh + head) * HD + 4 * g;
#pragma unroll
    for (int j = 0; j < NJ; ++j) qf[j] = *reinterpret_cast<const f32x4*>(qrow + 16 * j);
  }
  // the run's key blocks: those of kept first tokens, then from its rows' lowest first key to their highest position
  int lo = row_ok ? start : INT_MAX, hi = p;
#pragma unroll
  for (int x = 1; x < 16; x <<= 1) {
    lo = min(lo, __shfl_xor(lo, x, kWave));
    hi = max(hi, __shfl_xor(hi, x, kWave));
  }
  const int b_first = __builtin_amdgcn_readfirstlane(lo) >> 4, b_last = __builtin_amdgcn_readfirstlane(hi) >> 4;
  const int b_kept = a.keep > 0 ? min((a.keep + 15) >> 4, b_first) : 0;
  const int n_blocks = b_kept + b_last - b_first + 1;

  float m = -INFINITY, l = 0.f;
  f32x4 acc[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int i = 0; i < n_blocks; ++i) {
    const int b = i < b_kept ? i : b_first + i - b_kept;
    if ((b & (kFlWaves - 1)) != w) continue;                   // (the same for the whole wave)
    const int key0 = b << 4, blk = key0 / a.page_size;
    const int page = blk < a.max_blocks ? bt[blk] : -1;
    const bool there = page >= 0 && page < a.num_pages;
    const size_t base = (size_t)(there ? page : 0) * a.nkv + kvh;
    const int off = key0 - blk * a.page_size;
    const float* kr = a.k + (base * a.page_size + off + r) * HD + 4 * g;
    const float* vr = a.v + (base * VD + r) * a.page_size + off + 4 * g;
    f32x4 kf[NJ], vf[ND];
#pragma unroll
    for (int j = 0; j < NJ; ++j) kf[j] = *reinterpret_cast<const f32x4*>(kr + 16 * j);
#pragma unroll
    for (int d = 0; d < ND; ++d) vf[d] = *reinterpret_cast<const f32x4*>(vr + (size_t)(16 * d) * a.page_size);
    f32x4 s0 = f32x4{0.f, 0.f, 0.f, 0.f}, s1 = s0;             // two chains: a score's roundings are halved
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        f32x4& s = x & 1 ? s1 : s0;
        s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][x], qf[j][x], s, 0, 0, 0);
      }
    float sc[4], mb = -INFINITY;
    int hidden = 0;                                            // of the lane's four keys, for its row
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int key = key0 + 4 * g + x;
      float t = (s0[x] + s1[x]) * a.scale;
      if (a.softcap > 0.f) t = a.softcap * tanhf(t / a.softcap);
      const bool seen = there && key <= p && (key >= start || key < a.keep);
      sc[x] = seen ? t : -INFINITY;
      hidden |= seen ? 0 : 1 << x;
      mb = fmaxf(mb, sc[x]);
    }
    mb = reduce16(mb, MaxOf{});
    mb = reduce32(mb, MaxOf{});
    const float m_new = fmaxf(m, mb);
    const float ref = m_new > -INFINITY ? m_new : 0.f;         // (nothing seen yet: every term is exp(-inf) = 0)
    const float corr = expf(m - ref);
    float pe[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) pe[x] = expf(sc[x] - ref);
    l = l * corr + ((pe[0] + pe[1]) + (pe[2] + pe[3]));
    m = m_new;
    if (__any(corr != 1.0f)) {
#pragma unroll
      for (int d = 0; d < ND; ++d) acc[d] *= corr;
    }
    // Products with a row's hidden keys are 0 * value: a value that is no number (a slot not yet written, a later token's)
    // must not reach the row, so those are taken out of the product and added to the rows that see them.
    bool odd = false;
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int x = 0; x < 4; ++x) odd |= !(fabsf(vf[d][x]) < INFINITY);
    if (__any(odd)) {
      for (int kg = 0; kg < 4; ++kg)
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const float pk = __shfl(pe[x], r + 16 * kg, kWave);
          const bool seen = __shfl(hidden >> x & 1, r + 16 * kg, kWave) == 0;
#pragma unroll
          for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int y = 0; y < 4; ++y) {
              const float val = __shfl(vf[d][x], 4 * g + y + 16 * kg, kWave);
              if (seen && !(fabsf(val) < INFINITY)) acc[d][y] = fmaf(pk, val, acc[d][y]);
            }
        }
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int x = 0; x < 4; ++x) vf[d][x] = fabsf(vf[d][x]) < INFINITY ? vf[d][x] : 0.f;
    }
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int x = 0; x < 4; ++x) acc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[d][x], pe[x], acc[d], 0, 0, 0);
  }
  l = reduce16(l, SumOf{});                               // the row's four lanes hold a quarter of its keys each
  l = reduce32(l, SumOf{});
#pragma unroll
  for (int d = 0; d < ND; ++d) acc_s[w][d][lane] = acc[d];
  if (g == 0) {
    m_s[w][r] = m;
    l_s[w][r] = l;
  }
  __syncthreads();
  if (!row_ok) return;
  float M = m_s[0][r];
#pragma unroll
  for (int x = 1; x < kFlWaves; ++x) M = fmaxf(M, m_s[x][r]);
  float f[kFlWaves], L = 0.f;
#pragma unroll
  for (int x = 0; x < kFlWaves; ++x) {
    f[x] = m_s[x][r] > -INFINITY ? expf(m_s[x][r] - M) : 0.f;
    L += l_s[x][r] * f[x];
  }
  if (a.sink) L += expf((a.sink_vals ? a.sink_vals[head] : 0.f) - M);    // (every row sees at least its own key: M is finite)
  const float open = a.gate ? 1.0f / (1.0f + expf(-a.gate[(size_t)token * a.gate_stride + head])) : 1.0f;
  float* orow = a.out + ((size_t)token * a.nh + head) * VD + 4 * g;
  for (int d = w; d < ND; d += kFlWaves) {                     // the waves share the output's tiles
    f32x4 o = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int x = 0; x < kFlWaves; ++x) o += acc_s[x][d][lane] * f[x];
#pragma unroll
    for (int x = 0; x < 4; ++x) o[x] = L > 0.f ? o[x] / L * open : 0.f;
    *reinterpret_cast<f32x4*>(orow + 16 * d) = o;
  }
}

// Whether float rows of these sizes go this way (attention_generic.hip asks); the same arguments as there.
bool attention_float_takes(const void* q, const void* k, const void* v, const void* out, int hd, int vd, int page_size) {
  if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15) return false;
  return page_size % 16 == 0 && ((hd == 64 && vd == 64) || (hd == 128 && vd == 128) || (hd == 192 && vd == 128));
}

int attention_float(const float* q, const float* k, const float* v, const int* block_table, const int* entry_of_token,
                    const int* positions, float* out, int window_kind, int window, float scale, int n_tokens, int nh, int nkv, int hd,
                    int vd, int page_size, int max_blocks, int num_pages, float softcap, int sink, const float* sink_vals, int keep,
                    const float* gate, int gate_stride, hipStream_t stream) {
  int hp = 1;                                        // heads of a tile: the group's, up to 16; the rest of the 16 rows are tokens
  while (hp < 16 && hp < nh / nkv) hp *= 2;
  const int tb = 16 / hp;
  const FloatAttention a{q, k, v, block_table, entry_of_token, positions, out, window_kind, window, scale, n_tokens, nh, nkv, page_size,
                         max_blocks, num_pages, softcap, sink, sink_vals, keep, gate, gate_stride, tb};
  const int rows = nkv * ceil_div(nh / nkv, hp);
  if (rows > 65535) return SHARPI_ERR_ARG;
  const dim3 grid(ceil_div(n_tokens, tb), rows, tb), block(kFlWaves * kWave);
  if (hd == 64) attn_float_kernel<64, 64><<<grid, block, 0, stream>>>(a);
  else if (hd == 128) attn_float_kernel<128, 128><<<grid, block, 0, stream>>>(a);
  else attn_float_kernel<192, 128><<<grid, block, 0, stream>>>(a);
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}
