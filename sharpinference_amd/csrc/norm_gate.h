// Behind a recurrence: every part (a head, a group of channels) of a token's row divided by its root mean square, times a weight a
// channel, times a gate; for parts of up to 1,024 channels, a multiple of 8.  A part lies in neighbouring lanes of a wave, eight
// channels a lane and turn, 16-byte accesses; its squares are added in the order of the kernels for any width, so the bits are theirs.
// Bound: the gate's exponential and division, and bytes (a wave a part, one channel a lane and turn, spent as much again on two-byte
// loads and stores).  us: 3,000 rows of 16 x 128 24.4 -> 12.6, 1,950 rows of 8 x 512, gated first 26.0 -> 13.8 (squares added as the lanes
// come, with other bits, 11.6 and 13.4).
#pragma once
#include "common.h"

// what multiplies: nothing, z / (1 + exp(-z)) as a product or as a quotient, 1 / (1 + exp(-z))
enum : int { PART_GATE_NONE = 0, PART_GATE_SILU = 1, PART_GATE_SIGMOID = 2, PART_GATE_SILU_QUOTIENT = 3 };
__device__ __forceinline__ float part_gate(int act, float z) {
  if (act == PART_GATE_SILU_QUOTIENT) return z / (1.0f + expf(-z));
  const float s = 1.0f / (1.0f + expf(-z));
  return act == PART_GATE_SILU ? z * s : s;
}

struct PartNorm {
  const float* o;          // [pairs, gd], (token, part) pairs, parts fastest
  const float* w;          // part p's weights at w + p * w_step, or null
  int w_step;
  float eps;
  const void* proj;        // gates: element (token t, part p, channel d) at t * stride + g_off + p * gd + d (act: none, null)
  int stride, g_off, act, gate_first;
  void* out;               // [pairs, gd]
  int pairs, G, gd;
};

constexpr int kPartChipWaves = 256 * 24;   // 256 compute units of 24 waves

inline bool part_norm_wide(const PartNorm& a) {
  const auto at16 = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  // (parts of up to 64 channels, an element a lane of a wave: until those waves are most of what the chip holds at once, a lane's eight exponentials one
  // after the other take longer: us, a wave a part / here, 4 parts of 64: 1 token 2.5 / 3.2, 500 2.9 / 3.6, 1,000 3.3 / 3.7, 2,048 4.2 / 4.0, 5,000 7.3 / 5.0)
  if (a.gd <= kWave && a.pairs <= kPartChipWaves) return false;
  return a.gd % 8 == 0 && a.gd <= 1024 && a.pairs <= (1 << 25) && at16(a.o) && at16(a.w) && at16(a.out) &&
         (a.act == PART_GATE_NONE || (a.stride % 8 == 0 && a.g_off % 8 == 0 && at16(a.proj)));
}

// R: runs of 8 a lane (two where a part has more than 512 channels)
template <typename T, int R>
__global__ __launch_bounds__(256) void part_norm_kernel(PartNorm a, int log_lanes) {
  const unsigned idx = blockIdx.x * 256u + threadIdx.x;
  const int pair = idx >> log_lanes, li = idx & ((1 << log_lanes) - 1);
  const bool there = pair < a.pairs;
  const int t = there ? pair / a.G : 0, p = there ? pair - t * a.G : 0;
  const T* gate = a.act ? (const T*)a.proj + (size_t)t * a.stride + a.g_off + (size_t)p * a.gd : nullptr;
  float x[R][8];
  Run8<T> z[R];
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int d = (li + u * kWave) * 8;
    const bool live = there && d < a.gd;
#pragma unroll
    for (int j = 0; j < 8; ++j) x[u][j] = 0.f;
    if (!live) continue;
    load8(a.o + (size_t)pair * a.gd + d, x[u]);
    if (gate) z[u].load(gate + d);
  }
#pragma unroll
  for (int u = 0; u < R; ++u) {
    if (gate && a.gate_first && there && (li + u * kWave) * 8 < a.gd) {
      float g[8];
      z[u].floats(g);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[u][j] *= part_gate(a.act, g[j]);
    }
  }
  const float ss = row_square_sum(x, 1 << log_lanes);
  const float inv = rsqrtf(ss / (float)a.gd + a.eps);
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int d = (li + u * kWave) * 8;
    if (!there || d >= a.gd) continue;
    if (a.w) {
      float wv[8];
      load8(a.w + (size_t)p * a.w_step + d, wv);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[u][j] = x[u][j] * inv * wv[j];
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[u][j] *= inv;
    }
    if (gate && !a.gate_first) {
      float g[8];
      z[u].floats(g);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[u][j] *= part_gate(a.act, g[j]);
    }
    store8((T*)a.out + (size_t)pair * a.gd + d, x[u]);
  }
}

template <typename T> static void part_norm_launch(const PartNorm& a, hipStream_t stream) {
  int log_lanes = 0;
  while ((8 << log_lanes) < a.gd && log_lanes < 6) ++log_lanes;
  const unsigned blocks = (unsigned)((((long long)a.pairs << log_lanes) + 255) / 256);
  if (a.gd > 512) part_norm_kernel<T, 2><<<blocks, 256, 0, stream>>>(a, log_lanes);
  else part_norm_kernel<T, 1><<<blocks, 256, 0, stream>>>(a, log_lanes);
}
