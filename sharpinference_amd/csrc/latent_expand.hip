// Latent attention of prompt portions over keys and values of their own: the cached rows [c (R) | rotated part (dr)] of the
// keys a step's portions see are expanded once, per head, into K [page, head, key, dn + dr] and V [page, head, dv, key]
// of a cache that lives for the step (pages of 128 keys), which the flash kernel then walks like any other
// (attention_prefill_kernel.h).
//
// A query row costs dn + dr + dv products a key this way instead of 2 R + dr over the shared rows (320 against 1,088 at 128 + 64
// wide heads over a latent of 512), and the flash kernel's 32 rows a wave feed two products with what one LDS read
// brings; the expansion costs (dn + dv) R products a key and head, whatever the number of queries.  So steps with few
// prompt tokens and decoding requests keep to the shared rows (the rule: parts/latent_attention.py).
// Rounding: keys and values are rounded to bfloat16 here, where the other form rounds the query taken through W_uk and the
// weighted sum of latents.
//
// latent_expand: a block is (page, head, 128 weight rows of K or of V), a product of R steps.  Bound: the matrix
// instruction and the LDS: a wave takes 64 weight rows (straight from memory, they stay in L2) against 64 keys, so that a
// key fragment read from LDS feeds four products.  Keys are rows of the result for V (a lane then stores four
// neighbouring keys of a value row), weights for K (four neighbouring elements of a key).
// 2,048 keys, 64 heads: 102 us (34 GFLOP; the weights a block reads from L2 bound it); a prompt of 2,048 tokens there,
// window 1,024: 1,630 us a layer over the shared rows (with both products per head), 315 over expanded keys.
#include <type_traits>

#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

constexpr int kPageKeys = 128;
constexpr int kExpThreads = 256;
constexpr int kExpK = 64;                      // elements of the latent a stage
constexpr int kExpLd = kExpK + 8;              // an LDS row: 16-byte reads of 16 rows fall into different banks

SHARPI_EXPORT int sharpi_latent_page_keys() { return kPageKeys; }

__global__ __launch_bounds__(kExpThreads, 2) void latent_expand_kernel(
    const bf16_t* __restrict__ rows, const int* __restrict__ block_table, const int* __restrict__ list,
    const bf16_t* __restrict__ w, bf16_t* __restrict__ k_out, bf16_t* __restrict__ v_out, int H, int dn, int dr, int dv, int R,
    int page_size, int max_blocks, int num_pages) {
  __shared__ __attribute__((aligned(16))) bf16_t cs[2][kPageKeys][kExpLd];
  const int page = blockIdx.x, h = blockIdx.y;
  const int entry = list[4 * page], key0 = list[4 * page + 1] * kPageKeys;
  const int lo = list[4 * page + 2], hi = list[4 * page + 3];        // the entry's keys that are there: lo <= key < hi
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wid = tid >> 6, r = lane & 15, g = lane >> 4;
  const int D = R + dr, N = dn + dv;
  const int* bt = block_table + (size_t)entry * max_blocks;
  // a key outside is read as the nearest that is there: finite values that meet probabilities of zero
  auto row_at = [&](int i) {
    const int key = min(max(key0 + i, lo), hi - 1);
    const int blk = key / page_size;
    const int p = min(max(blk < max_blocks ? bt[blk] : 0, 0), num_pages - 1);
    return rows + ((size_t)p * page_size + key % page_size) * D;
  };
  // the thread's four rows of every stage, and its 16 bytes of them
  const bf16_t* src[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) src[i] = row_at((tid >> 3) + 32 * i) + (tid & 7) * 8;

  // this block's 128 weight rows: of K, or of V
  const int k_blocks = (dn + 127) / 128;
  const bool values = (int)blockIdx.z >= k_blocks;
  const int n0 = ((int)blockIdx.z - (values ? k_blocks : 0)) * 128 + (wid & 1) * 64;   // the wave's 64 of them, and its 64 keys
  const int m0 = (wid >> 1) * 64;
  const bool live = n0 < (values ? dv : dn);
  const bf16_t* wp = w + ((size_t)h * N + (live ? n0 : 0) + (values ? dn : 0) + r) * R + g * 8;

  // the rotated part, the same for every head
  if (blockIdx.z == 0) {
    for (int idx = tid; idx < kPageKeys * (dr / 8); idx += kExpThreads) {
      const int i = idx / (dr / 8), c = idx % (dr / 8) * 8;
      *reinterpret_cast<uint4*>(k_out + (((size_t)page * H + h) * kPageKeys + i) * (dn + dr) + dn + c) =
          *reinterpret_cast<const uint4*>(row_at(i) + R + c);
    }
  }
  f32x4 acc[4][4];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int m = 0; m < 4; ++m) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](u32x4 (&st)[4], int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) st[i] = *reinterpret_cast<const u32x4*>(src[i] + k0);
  };
  auto weights = [&](bf16x8 (&f)[2][4], int k0) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int t = 0; t < 4; ++t) f[j][t] = *reinterpret_cast<const bf16x8*>(wp + (size_t)(16 * t) * R + k0 + 32 * j);
  };
  auto stash = [&](int buf, const u32x4 (&st)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(&cs[buf][(tid >> 3) + 32 * i][(tid & 7) * 8]) = st[i];
  };
  auto products = [&](int buf, const bf16x8 (&f)[2][4], auto values_tag) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      bf16x8 c[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) c[m] = *reinterpret_cast<const bf16x8*>(&cs[buf][m0 + 16 * m + r][32 * j + 8 * g]);
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if constexpr (decltype(values_tag)::value)
            acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c[m], f[j][t], acc[t][m], 0, 0, 0);
          else
            acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[j][t], c[m], acc[t][m], 0, 0, 0);
        }
    }
  };
  // (loads beyond the last stage read the last again: none sits behind a branch)
  const int last = R - kExpK;
  auto walk = [&](auto values_tag) {
    u32x4 st[4];
    bf16x8 wf[2][2][4];
    fetch(st, 0);
    weights(wf[0], 0);
    stash(0, st);
    __syncthreads();
    for (int k0 = 0;; k0 += 2 * kExpK) {
      fetch(st, min(k0 + kExpK, last));
      weights(wf[1], min(k0 + kExpK, last));
      __builtin_amdgcn_sched_barrier(0);
      products(0, wf[0], values_tag);
      __builtin_amdgcn_sched_barrier(0);
      if (k0 + kExpK >= R) break;
      stash(1, st);
      __syncthreads();
      fetch(st, min(k0 + 2 * kExpK, last));
      weights(wf[0], min(k0 + 2 * kExpK, last));
      __builtin_amdgcn_sched_barrier(0);
      products(1, wf[1], values_tag);
      __builtin_amdgcn_sched_barrier(0);
      if (k0 + 2 * kExpK >= R) break;
      stash(0, st);
      __syncthreads();
    }
  };
  auto pack = [](const f32x4& v) {
    uint2 o;
    o.x = f32_to_bf16_pair(v[0], v[1]);
    o.y = f32_to_bf16_pair(v[2], v[3]);
    return o;
  };
  if (values) {                                     // (the same for the whole block)
    walk(std::true_type{});
    if (!live) return;
    // lane: value row n0 + 16 t + r, keys m0 + 16 m + 4 g ..
    bf16_t* dst = v_out + (((size_t)page * H + h) * dv + n0 + r) * kPageKeys + m0 + 4 * g;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int m = 0; m < 4; ++m) *reinterpret_cast<uint2*>(dst + (size_t)(16 * t) * kPageKeys + 16 * m) = pack(acc[t][m]);
  } else {
    walk(std::false_type{});
    if (!live) return;
    // lane: key m0 + 16 m + r, elements n0 + 16 t + 4 g ..
    bf16_t* dst = k_out + (((size_t)page * H + h) * kPageKeys + m0 + r) * (dn + dr) + n0 + 4 * g;
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int t = 0; t < 4; ++t) *reinterpret_cast<uint2*>(dst + (size_t)(16 * m) * (dn + dr) + 16 * t) = pack(acc[t][m]);
  }
}

// Whether heads of these widths are expanded: whole strips of 64 weight rows, whole stages of the latent.
SHARPI_EXPORT int sharpi_latent_expand_takes(int dn, int dr, int dv, int R) {
  return dn > 0 && dv > 0 && dr >= 0 && R > 0 && dn % 64 == 0 && dv % 64 == 0 && dr % 8 == 0 && R % kExpK == 0;
}

// rows [num_pages * page_size, R + dr]; block_table [entries, max_blocks]; list int [n_pages, 4] = (entry, number of the page
// in its sequence, first key that is there, end of the keys that are there); w [H, dn + dv, R]: a head's key rows, then its
// value rows; k_out [n_pages, H, 128, dn + dr], v_out [n_pages, H, dv, 128].  bfloat16 throughout.
SHARPI_EXPORT int sharpi_latent_expand(const void* rows, const int* block_table, const int* list, const void* w, void* k_out,
                                       void* v_out, int n_pages, int H, int dn, int dr, int dv, int R, int page_size,
                                       int max_blocks, int num_pages, hipStream_t stream) {
  if (n_pages <= 0) return SHARPI_OK;
  if (!sharpi_latent_expand_takes(dn, dr, dv, R) || H <= 0 || H > 65535 || page_size <= 0 || max_blocks <= 0 || num_pages <= 0) return SHARPI_ERR_ARG;
  if (((uintptr_t)rows | (uintptr_t)w | (uintptr_t)k_out | (uintptr_t)v_out) & 15) return SHARPI_ERR_ARG;
  const dim3 grid(n_pages, H, ceil_div(dn, 128) + ceil_div(dv, 128));
  latent_expand_kernel<<<grid, kExpThreads, 0, stream>>>((const bf16_t*)rows, block_table, list, (const bf16_t*)w, (bf16_t*)k_out,
                                                        (bf16_t*)v_out, H, dn, dr, dv, R, page_size, max_blocks, num_pages);
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}

// ---------------------------------------------------------------------------
// The queries of the expanded form: per token the heads' [dn | dr] side by side, the leading pairs (2i, 2i + 1) of the last dr
// elements turned by position * inv_freq[i] (cos and sin times `magnitude`), in float, rounded once.
// ---------------------------------------------------------------------------
constexpr int kQueryMaxPairs = 128;

__global__ __launch_bounds__(256) void latent_queries_kernel(const bf16_t* __restrict__ q, int ldq, const int* __restrict__ positions,
                                                             const float* __restrict__ inv_freq, int n_pairs, float magnitude,
                                                             bf16_t* __restrict__ out, int H, int dn, int dr) {
  __shared__ float cs[kQueryMaxPairs], sn[kQueryMaxPairs];
  const int t = blockIdx.x;
  const float p = (float)positions[t];
  for (int i = threadIdx.x; i < n_pairs; i += blockDim.x) {
    const float ang = p * inv_freq[i];
    cs[i] = cosf(ang) * magnitude;
    sn[i] = sinf(ang) * magnitude;
  }
  __syncthreads();
  const int width = dn + dr, pieces = H * width / 8;
  const bf16_t* src = q + (size_t)t * ldq;
  bf16_t* dst = out + (size_t)t * H * width;
  for (int idx = threadIdx.x; idx < pieces; idx += blockDim.x) {
    const int c = idx * 8 % width;                  // (a piece of 8 lies in one head, and in one part of it)
    uint4 v = *reinterpret_cast<const uint4*>(src + idx * 8);
    if (c >= dn) {
      uint32_t* x = reinterpret_cast<uint32_t*>(&v);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int pair = (c - dn) / 2 + i;
        if (pair < n_pairs) {
          const float a = bf16_bits_to_f32(x[i] & 0xffffu), b = bf16_bits_to_f32(x[i] >> 16);
          x[i] = f32_to_bf16_pair(a * cs[pair] - b * sn[pair], b * cs[pair] + a * sn[pair]);
        }
      }
    }
    *reinterpret_cast<uint4*>(dst + idx * 8) = v;
  }
}

SHARPI_EXPORT int sharpi_latent_queries(const void* q, int ldq, const int* positions, const float* inv_freq, int n_pairs, float magnitude,
                                        void* out, int n_tokens, int H, int dn, int dr, hipStream_t stream) {
  if (n_tokens <= 0) return SHARPI_OK;
  if (H <= 0 || dn <= 0 || dn % 8 || dr < 0 || dr % 8 || ldq % 8 || ldq < H * (dn + dr) || n_pairs < 0 || n_pairs > kQueryMaxPairs ||
      2 * n_pairs > dr || (n_pairs && !inv_freq) || (((uintptr_t)q | (uintptr_t)out) & 15)) return SHARPI_ERR_ARG;
  latent_queries_kernel<<<n_tokens, 256, 0, stream>>>((const bf16_t*)q, ldq, positions, inv_freq, n_pairs, magnitude, (bf16_t*)out, H, dn, dr);
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}
