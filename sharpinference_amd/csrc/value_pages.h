// Values on their way into the paged cache, for steps of many tokens.
//
// A page keeps a value channel's tokens side by side ([page][kv head][channel][page_size]), a projection's row keeps a token's
// channels side by side.  A block that stores one token's channels therefore writes single elements a page apart, and the other tokens
// of the same 32 bytes are written by other blocks on other dies, each of which sends its piece to memory by itself.  Here a block of 256 threads
// turns 16 tokens x 128 channels in LDS and stores runs of eight tokens of a channel, 16 bytes at once where their slots are
// neighbours (a prompt's pages), element by element where they are not; a page of 16 tokens leaves as whole lines.
#pragma once
#include "common.h"

constexpr int kValueTokens = 16;
constexpr int kValueCols = 128;
constexpr int kValueThreads = 256;
// elements from a channel's tokens to the next channel's in LDS: a column read by neighbouring lanes falls into different banks
template <typename T> constexpr int kValuePitch = sizeof(T) == 2 ? 18 : 17;
template <typename T> constexpr size_t kValueLds = (size_t)kValueCols * kValuePitch<T> * sizeof(T);

__host__ __device__ inline int value_tiles(int n_tokens, int channels) {
  return ((n_tokens + kValueTokens - 1) / kValueTokens) * ((channels + kValueCols - 1) / kValueCols);
}

// Tile `tile` of value_tiles(n_tokens, nkv * vd); vd % 8 == 0.  gather(t, c, v) gives channels c .. c + 7 of the nkv * vd of token t as
// floats.  lds: kValueLds<T> bytes, slots: LDS of kValueTokens ints.  Every thread of a block of kValueThreads or more calls it.
template <typename T, typename G>
__device__ __forceinline__ void values_to_pages(int tile, int n_tokens, int nkv, int vd, int page_size, const int* __restrict__ slot_mapping,
                                                T* __restrict__ v_cache, T* lds, int* slots, const G& gather) {
  constexpr int P = kValuePitch<T>;
  const int across = (nkv * vd + kValueCols - 1) / kValueCols;
  const int t0 = tile / across * kValueTokens, c0 = tile % across * kValueCols;
  int own = -1;
  if (threadIdx.x < kValueTokens && t0 + (int)threadIdx.x < n_tokens) own = slot_mapping[t0 + threadIdx.x];
  if (threadIdx.x < kValueTokens) slots[threadIdx.x] = own;
  if (!__syncthreads_or(own >= 0)) return;         // (a layer that reads another's cache)
  if (threadIdx.x < kValueThreads) {
    const int tok = threadIdx.x >> 4, run = threadIdx.x & 15;
    const int t = t0 + tok, c = c0 + run * 8;
    if (t < n_tokens && c < nkv * vd) {
      float v[8];
      gather(t, c, v);
#pragma unroll
      for (int j = 0; j < 8; ++j) lds[(run * 8 + j) * P + tok] = from_f32<T>(v[j]);
    }
  }
  __syncthreads();
  const int col = threadIdx.x >> 1, first = (threadIdx.x & 1) * 8, c = c0 + col;
  if (threadIdx.x >= kValueThreads || c >= nkv * vd) return;
  int s[8];
  bool run = true;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    s[j] = slots[first + j];
    run = run && s[j] == s[0] + j;
  }
  const T* src = lds + col * P + first;
  const int g = c / vd, d = c % vd;
  const auto place = [&](int slot) { return (((size_t)(slot / page_size) * nkv + g) * vd + d) * page_size + slot % page_size; };
  if (run && s[0] >= 0 && s[0] % 8 == 0 && page_size % 8 == 0 && ((uintptr_t)v_cache & 15) == 0) {
    union {
      T e[8];
      uint4 q[sizeof(T) / 2];
    } o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o.e[j] = src[j];
    uint4* dst = reinterpret_cast<uint4*>(v_cache + place(s[0]));
#pragma unroll
    for (int j = 0; j < (int)(sizeof(T) / 2); ++j) dst[j] = o.q[j];
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (s[j] >= 0) v_cache[place(s[j])] = src[j];
  }
}
