// Position encoding, weightless per-head norm, query temperature and the cache write, one kernel.
//
// Input  qkv [T, (nh + nkv) * hd + nkv * vd]: q heads, then k heads (hd wide), then v heads (vd wide,
// usually hd) of each token; an optional bias of the row's width (float) is added to every
// token's row first, in float.
// q head : rotate (if inv_freq) -> norm (if qk_norm) -> * temperature (if temp_tuning) -> q_out
// k head : rotate (if inv_freq) -> norm (if qk_norm) -> cache K at slot_mapping[t]
// v head : cache V at slot_mapping[t]
// Rotation is on the first rotary_dim elements of a head (the rest pass through unrotated), in
// pairs (2i, 2i+1) (interleaved) or (i, i + rotary_dim/2) (half-split), with
// angle = float(pos) * inv_freq[i], i < rotary_dim/2, all in float.  The norm runs over the whole head.
// Cache layout of one layer: keys [page][kv head][page_size][hd], values transposed inside the page,
// [page][kv head][hd][page_size] (so that the matrix-core kernels read runs of keys for one
// value column); slot = page * page_size + offset;
// a negative slot means "do not store" (the layer reads another layer's cache).
#include "common.h"
#include "value_pages.h"

template <typename T>
__global__ void rope_kv_kernel(const T* __restrict__ qkv, T* __restrict__ q_out, T* __restrict__ k_cache,
                               T* __restrict__ v_cache, const int* __restrict__ slot_mapping,
                               const int* __restrict__ positions, const float* __restrict__ inv_freq,
                               const float* __restrict__ bias,
                               int qk_norm, float eps, int temp_tuning, float floor_scale, float attn_scale,
                               int nh, int nkv, int hd, int vd, int page_size, int half_split, int rotary_dim,
                               int row_stride) {
  const int t = blockIdx.x;
  const int head = blockIdx.y;            // 0..nh-1 q, nh..nh+nkv-1 k, then v
  const int lane = threadIdx.x;           // one wave
  const int half = hd >> 1;
  const size_t head_at = head < nh + nkv ? (size_t)head * hd : (size_t)(nh + nkv) * hd + (size_t)(head - nh - nkv) * vd;
  const T* src = qkv + (size_t)t * row_stride + head_at;
  const float* hb = bias ? bias + head_at : nullptr;
  const int pos = positions[t];
  const bool is_q = head < nh;
  const bool is_k = !is_q && head < nh + nkv;
  const int slot = slot_mapping[t];

  if (!is_q && !is_k) {  // v: plain copy into the cache
    if (slot < 0) return;
    const int kvh = head - nh - nkv;
    T* dst = v_cache + ((size_t)(slot / page_size) * nkv + kvh) * vd * page_size + (slot % page_size);
    for (int d = lane; d < vd; d += kWave)
      dst[(size_t)d * page_size] = hb ? from_f32<T>(to_f32<T>(src[d]) + hb[d]) : src[d];
    return;
  }
  if (is_k && slot < 0) return;

  // pairs handled by this lane: i = lane, lane + 64, ... (hd <= 512).  Pair i < rotary_dim/2 is a
  // rotary pair, at elements (2i, 2i+1) or (i, i + rotary_dim/2); the pairs after them are the
  // neighbouring elements of the unrotated rest.
  const int rot_pairs = rotary_dim >> 1;
  float x0[4], x1[4];
  int e0[4], e1[4];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = lane + j * kWave;
    x0[j] = 0.f;
    x1[j] = 0.f;
    e0[j] = e1[j] = 0;
    if (i < half) {
      if (i >= rot_pairs) {
        e0[j] = 2 * i;
        e1[j] = 2 * i + 1;
      } else if (half_split) {
        e0[j] = i;
        e1[j] = i + rot_pairs;
      } else {
        e0[j] = 2 * i;
        e1[j] = 2 * i + 1;
      }
      float a = to_f32<T>(src[e0[j]]);
      float b = to_f32<T>(src[e1[j]]);
      if (hb) {
        a += hb[e0[j]];
        b += hb[e1[j]];
      }
      if (inv_freq && i < rot_pairs) {
        const float ang = (float)pos * inv_freq[i];
        const float c = cosf(ang);
        const float s = sinf(ang);
        const float ra = fmaf(a, c, -(b * s));       // (written out: the vector form below has the same bits)
        const float rb = fmaf(b, c, a * s);
        a = ra;
        b = rb;
      }
      x0[j] = a;
      x1[j] = b;
      ss += fmaf(b, b, a * a);
    }
  }
  float mul = 1.0f;
  if (qk_norm) {
    const float total = wave_sum(ss);
    mul = 1.0f / sqrtf(total / (float)hd + eps);
  }
  float post = 1.0f;
  if (is_q && temp_tuning) {
    post = 1.0f + attn_scale * logf(floorf(((float)pos + 1.0f) / floor_scale) + 1.0f);
  }
  T* dst;
  if (is_q) {
    dst = q_out + ((size_t)t * nh + head) * hd;
  } else {
    const int kvh = head - nh;
    dst = k_cache + (((size_t)(slot / page_size) * nkv + kvh) * page_size + (slot % page_size)) * hd;
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = lane + j * kWave;
    if (i < half) {
      float a = x0[j], b = x1[j];
      if (qk_norm) {
        a *= mul;
        b *= mul;
      }
      if (is_q && temp_tuning) {
        a *= post;
        b *= post;
      }
      dst[e0[j]] = from_f32<T>(a);
      dst[e1[j]] = from_f32<T>(b);
    }
  }
}

// The same for head sizes 32, 64, 128, 256 whose rotary width is a multiple of 8 (pairs split in halves: of 16; runs beyond it
// pass through): a thread per run of 8 elements, 16-byte accesses; the hd/8 lanes of a head are neighbours in a wave, sum their
// squares with shuffles and hand each other the partners of split pairs.  Blocks (token, y) share a token's heads between
// them, 256 runs each, so that a handful of decode tokens still spreads over many compute units.  The token's angles are the
// same for every head: a block computes each of them once, into LDS (four sines and cosines in every thread were the kernel's
// time).  Steps of many tokens leave the values to blocks of their own behind the tokens' (value_pages.h).
// Interleaved pairs of heads as wide as their values (PAIRS false) keep the sums this form always had: eight squares a lane, then the lanes.  The
// others (PAIRS) add their squares pair by pair in the general kernel's order, through LDS, and have its bits, so that a row has the same
// bits however many tokens come with it (they come here in steps of many tokens alone).
// Bound: the rows' bytes.  40 + 8 heads of 128 and 8 of values, us: 2,048 tokens 24.2 -> 12.6 (104 -> 54.7 for 8,192, 235 MB: 4.3 TB/s, about
// a copy's rate); 1,950 tokens with split pairs (a wave a head before), 16 + 8 heads 25.3 -> 12.3, 16 + 4 19.2 -> 10.8 (with the lanes' order of
// the sum, other bits than a wave a head, 10.9 and 9.7).
constexpr int kRopeMaxAngles = 128;              // hd <= 256
// A wave's sums of a pair's two squares: a head of L lanes has 4 L, at 5 L from the head before (neighbouring heads' reads in different banks).
constexpr int kRopeWavePairs = 5 * kWave;
constexpr int kRopeChipWaves = 256 * 32;         // 256 compute units of 32 waves
constexpr int kRopeNarrow = 1024;     // q and k elements of a token up to which half of a block's threads and more would have no run
constexpr int kRopeSplitTokens = 64;             // up to so many tokens a step, a token's heads lie in several blocks

// what a wave's lanes stored to LDS is there for its other lanes (a wave's LDS accesses stay in their order; the compiler has to keep it)
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <typename T, bool PAIRS>
__global__ __launch_bounds__(256) void rope_kv_vec_kernel(
    const T* __restrict__ qkv, T* __restrict__ q_out, T* __restrict__ k_cache, T* __restrict__ v_cache,
    const int* __restrict__ slot_mapping, const int* __restrict__ positions, const float* __restrict__ inv_freq,
    const float* __restrict__ bias, int qk_norm, float eps, int temp_tuning, float floor_scale, float attn_scale,
    int n_tokens, int nh, int nkv, int hd, int vd, int page_size, int half_split, int rotary_dim, int row_stride, int values_apart) {
  constexpr size_t kTile = kValueLds<T> > 4 * kRopeWavePairs * sizeof(float) ? kValueLds<T> : 4 * kRopeWavePairs * sizeof(float);
  __shared__ __attribute__((aligned(16))) char tile[kTile];     // (value blocks: their tile; the others: their waves' pairs of squares)
  __shared__ int tile_slots[kValueTokens];
  __shared__ __attribute__((aligned(16))) float cs_tab[kRopeMaxAngles], sn_tab[kRopeMaxAngles];
  if (blockIdx.x >= n_tokens) {                    // (values_apart: the blocks behind the tokens')
    const size_t v_at = (size_t)(nh + nkv) * hd;
    values_to_pages<T>(blockIdx.x - n_tokens, n_tokens, nkv, vd, page_size, slot_mapping, v_cache, reinterpret_cast<T*>(tile), tile_slots,
                       [&](int t, int c, float* v) {
      load8(qkv + (size_t)t * row_stride + v_at + c, v);
      if (bias) {
        float b8[8];
        load8(bias + v_at + c, b8);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] += b8[j];
      }
    });
    return;
  }
  const int t = blockIdx.x;
  const int per_head = hd >> 3;                    // lanes per head: 4, 8, 16 or 32
  const int chunks = (nh + (values_apart ? nkv : 2 * nkv)) * per_head;
  const int pos = positions[t];
  const int slot = slot_mapping[t];
  const T* src = qkv + (size_t)t * row_stride;
  float post = 1.0f;
  if (temp_tuning) post = 1.0f + attn_scale * logf(floorf(((float)pos + 1.0f) / floor_scale) + 1.0f);
  if (inv_freq) {
    if (threadIdx.x < rotary_dim / 2) {
      const float ang = (float)pos * inv_freq[threadIdx.x];
      cs_tab[threadIdx.x] = cosf(ang);
      sn_tab[threadIdx.x] = sinf(ang);
    }
    __syncthreads();
  }
  // a thread's run within a head is the same in every turn of the loop (the block size is a multiple
  // of the lanes per head), and so are its angles
  const int run = threadIdx.x % per_head;
  const int half_runs = rotary_dim / 16;           // (split pairs: runs of the low half)
  const bool rotates = inv_freq != nullptr && run * 8 < rotary_dim;
  const bool low = run < half_runs;
  const int mate = (threadIdx.x & (kWave - 1)) + (low ? half_runs : -half_runs);
  const int ang = !rotates ? 0 : PAIRS && half_split ? (low ? run : run - half_runs) * 8 : run * 4;      // the run's first angle
  float cs4[4], sn4[4];                            // (interleaved pairs keep their four)
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    cs4[j] = rotates ? cs_tab[ang + j] : 1.f;
    sn4[j] = rotates ? sn_tab[ang + j] : 0.f;
  }
  for (int base = blockIdx.y * blockDim.x; base < chunks; base += gridDim.y * blockDim.x) {
    const int ci = base + threadIdx.x;
    const bool valid = ci < chunks;
    const int head = valid ? ci / per_head : 0;
    const bool is_q = head < nh;
    const bool is_k = !is_q && head < nh + nkv;
    float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (valid) {
      load8(src + (size_t)head * hd + run * 8, x);
      if (bias) {
        float b8[8];
        load8(bias + (size_t)head * hd + run * 8, b8);
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] += b8[j];
      }
    }
    [[maybe_unused]] float other[8];   // (PAIRS: split pairs' partners, turned as x is)
    if (PAIRS && half_split && inv_freq) {      // every lane takes part in the shuffles
#pragma unroll
      for (int j = 0; j < 8; ++j) other[j] = __shfl(x[j], mate & (kWave - 1), kWave);
      if (rotates && (is_q || is_k)) {
        float c[8], sn[8];
        load8(cs_tab + ang, c);
        load8(sn_tab + ang, sn);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float own = x[j];
          x[j] = fmaf(own, c[j], low ? -(other[j] * sn[j]) : other[j] * sn[j]);
          other[j] = fmaf(other[j], c[j], low ? own * sn[j] : -(own * sn[j]));
        }
      }
    } else if (rotates && (is_q || is_k)) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float a = x[2 * j], b = x[2 * j + 1];
        x[2 * j] = fmaf(a, cs4[j], -(b * sn4[j]));
        x[2 * j + 1] = PAIRS ? fmaf(b, cs4[j], a * sn4[j]) : fmaf(a, sn4[j], b * cs4[j]);
      }
    }
    if (qk_norm) {
      float ss = 0.f;
      if constexpr (PAIRS) {
        float* const head_pairs = reinterpret_cast<float*>(tile) + threadIdx.x / kWave * kRopeWavePairs + (threadIdx.x & (kWave - 1)) / per_head * 5 * per_head;
        if (!(half_split && rotates)) {
          *reinterpret_cast<float4*>(head_pairs + 4 * run) = make_float4(fmaf(x[1], x[1], x[0] * x[0]), fmaf(x[3], x[3], x[2] * x[2]),
                                                                         fmaf(x[5], x[5], x[4] * x[4]), fmaf(x[7], x[7], x[6] * x[6]));
        } else if (low) {
#pragma unroll
          for (int j = 0; j < 8; j += 4)
            *reinterpret_cast<float4*>(head_pairs + 8 * run + j) =
                make_float4(fmaf(other[j], other[j], x[j] * x[j]), fmaf(other[j + 1], other[j + 1], x[j + 1] * x[j + 1]),
                            fmaf(other[j + 2], other[j + 2], x[j + 2] * x[j + 2]), fmaf(other[j + 3], other[j + 3], x[j + 3] * x[j + 3]));
        }
        wave_lds_fence();
        ss = (head_pairs[run] + head_pairs[run + 2 * per_head]) + (head_pairs[run + per_head] + head_pairs[run + 3 * per_head]);
        wave_lds_fence();
      } else if (valid && (is_q || is_k)) {
        ss = fmaf(x[0], x[0], x[1] * x[1]);
#pragma unroll
        for (int j = 2; j < 8; ++j) ss = fmaf(x[j], x[j], ss);
      }
      ss = group_sum(ss, per_head);
      const float mul = 1.0f / sqrtf(ss / (float)hd + eps);
      if (is_q || is_k) {
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] *= mul;
      }
    }
    if (!valid) continue;
    if (is_q) {
      if (temp_tuning) {
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] *= post;
      }
      store8(q_out + ((size_t)t * nh + head) * hd + run * 8, x);
    } else if (slot >= 0) {
      const size_t page = (size_t)(slot / page_size);
      const int off = slot % page_size;
      if (is_k) {
        store8(k_cache + ((page * nkv + (head - nh)) * page_size + off) * hd + run * 8, x);
      } else {
        T* dst = v_cache + (page * nkv + (head - nh - nkv)) * hd * page_size + off;
#pragma unroll
        for (int j = 0; j < 8; ++j) dst[(size_t)(run * 8 + j) * page_size] = from_f32<T>(x[j]);
      }
    }
  }
}

SHARPI_EXPORT int sharpi_rope_kv(const void* qkv, void* q_out, void* k_cache, void* v_cache, int dtype,
                                 const int* slot_mapping, const int* positions, const float* inv_freq,
                                 const float* bias, int qk_norm, float eps, int temp_tuning, float floor_scale, float attn_scale,
                                 int n_tokens, int nh, int nkv, int hd, int vd, int page_size, int pair_layout,
                                 int rotary_dim, int row_stride, hipStream_t stream) {
  if (n_tokens <= 0) return SHARPI_OK;
  // pair_layout: 0 = pairs (2i, 2i+1), 1 = pairs (i, i + rotary_dim/2); rotary_dim even, <= hd
  if (pair_layout < 0 || pair_layout > 1) return SHARPI_ERR_ARG;
  if (inv_freq == nullptr) rotary_dim = 0;
  else if (rotary_dim <= 0 || (rotary_dim & 1) || rotary_dim > hd) return SHARPI_ERR_ARG;
  if (hd <= 0 || (hd & 1) || hd > 512 || vd <= 0 || nh <= 0 || nkv <= 0 || page_size <= 0) return SHARPI_ERR_ARG;
  if (nh + 2 * nkv > 65535) return SHARPI_ERR_ARG;
  // rows of qkv may be wider than q, k and v (further columns behind them): row_stride elements a row, 0 = dense
  const int row_width = (nh + nkv) * hd + nkv * vd;
  if (row_stride == 0) row_stride = row_width;
  if (row_stride < row_width) return SHARPI_ERR_ARG;
  if (temp_tuning && !(floor_scale > 0.f)) return SHARPI_ERR_ARG;
  dim3 grid(n_tokens, nh + 2 * nkv), block(kWave);
  if (dtype != DT_F32 && dtype != DT_BF16) return SHARPI_ERR_ARG;
  // few tokens (decode): a token's heads over several blocks, for the compute units' sake; many tokens: one block
  // per token, which then computes its angles once for all heads, and blocks of their own for the values
  // (narrow rows, which leave most of a block's threads idle, keep their values: 4 + 2 heads of 64 in floats, unturned, 3,000 tokens 8.2 -> 11.0 us with
  // blocks apart; and go a wave a head where they have the choice: split pairs, 5 + 1 heads of 64, 8,192 tokens 19.5 -> 23 us by runs)
  const int row_lanes = (nh + 2 * nkv) * hd / 8;
  const bool many = n_tokens > kRopeSplitTokens && row_lanes > (rotary_dim > 0 ? 128 : 192);
  const auto at16 = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  const bool pairs = pair_layout || vd != hd;
  // (the forms that have the general kernel's bits go there until its waves are more than the chip holds at once: us, a wave a head / runs, split
  // pairs: 1 token of 16 + 4 heads 2.8 / 3.6, 64 3.3 / 4.0, 200 4.3 / 4.8, 400 6.0 / 5.3; 100 tokens of 40 + 8 4.4 / 5.8, 200 6.6 / 6.1)
  const bool by_runs = !pairs || (many && (nh + nkv) * hd > kRopeNarrow && (long long)n_tokens * (nh + 2 * nkv) > kRopeChipWaves);
  if (by_runs && (hd == 32 || hd == 64 || hd == 128 || hd == 256) && vd % 8 == 0 &&
      rotary_dim % (pair_layout ? 16 : 8) == 0 && (row_stride & 7) == 0 && at16(qkv) && at16(q_out) && at16(k_cache) && at16(bias)) {
    const int tiles = many ? value_tiles(n_tokens, nkv * vd) : 0;
    const dim3 vgrid(n_tokens + tiles, many ? 1 : ceil_div((nh + 2 * nkv) * (hd >> 3), 256));
#define ROPE_GO(T, PAIRS)                                                                                                               \
  rope_kv_vec_kernel<T, PAIRS><<<vgrid, 256, 0, stream>>>((const T*)qkv, (T*)q_out, (T*)k_cache, (T*)v_cache, slot_mapping, positions, inv_freq, \
                                                   bias, qk_norm, eps, temp_tuning, floor_scale, attn_scale, n_tokens, nh, nkv, hd, vd,   \
                                                   page_size, pair_layout, rotary_dim, row_stride, many)
    if (dtype == DT_F32 && pairs) ROPE_GO(float, true);
    else if (dtype == DT_F32) ROPE_GO(float, false);
    else if (pairs) ROPE_GO(bf16_t, true);
    else ROPE_GO(bf16_t, false);
#undef ROPE_GO
    SHARPI_CHECK_LAUNCH();
    return SHARPI_OK;
  }
  if (dtype == DT_F32)
    rope_kv_kernel<float><<<grid, block, 0, stream>>>((const float*)qkv, (float*)q_out, (float*)k_cache,
                                                     (float*)v_cache, slot_mapping, positions, inv_freq, bias, qk_norm,
                                                     eps, temp_tuning, floor_scale, attn_scale, nh, nkv, hd, vd,
                                                     page_size, pair_layout, rotary_dim, row_stride);
  else if (dtype == DT_BF16)
    rope_kv_kernel<bf16_t><<<grid, block, 0, stream>>>((const bf16_t*)qkv, (bf16_t*)q_out, (bf16_t*)k_cache,
                                                      (bf16_t*)v_cache, slot_mapping, positions, inv_freq, bias,
                                                      qk_norm, eps, temp_tuning, floor_scale, attn_scale, nh, nkv,
                                                      hd, vd, page_size, pair_layout, rotary_dim, row_stride);
  else
    return SHARPI_ERR_ARG;
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}
