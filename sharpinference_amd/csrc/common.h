// Shared device helpers for the gfx950 kernels: storage types, conversions, wave reductions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define SHARPI_OK 0
#define SHARPI_ERR_ARG 1001   // a size or option the kernel does not take
#define SHARPI_ERR_LAUNCH 1002

#define SHARPI_CHECK_LAUNCH()                                   \
  do {                                                          \
    hipError_t e__ = hipGetLastError();                         \
    if (e__ != hipSuccess) return (int)e__;                     \
  } while (0)

#define SHARPI_EXPORT extern "C" __attribute__((visibility("default")))

constexpr int kWave = 64;

// bfloat16 as raw bits; conversions are round-to-nearest-even, NaN kept quiet.
struct bf16_t {
  uint16_t bits;
};

__device__ __forceinline__ float bf16_to_f32(bf16_t v) {
  return __uint_as_float(((uint32_t)v.bits) << 16);
}
__device__ __forceinline__ float bf16_bits_to_f32(uint32_t bits16) {
  return __uint_as_float(bits16 << 16);
}
// One instruction for two values (rounding by integer steps, with a NaN's bits selected, took seven a value and was half of
// what small row kernels issued; 3,000 tokens: activation in the grouped product's epilogue 295 -> 280 us, expanded keys 46.5 -> 37.8).
__device__ __forceinline__ uint32_t f32_to_bf16_pair(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) float f32x2_t;
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
  const f32x2_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}
__device__ __forceinline__ bf16_t f32_to_bf16(float f) {
  bf16_t r;
  r.bits = __builtin_bit_cast(uint16_t, (__bf16)f);
  return r;
}

template <typename T> __device__ __forceinline__ float to_f32(T v);
template <> __device__ __forceinline__ float to_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ float to_f32<bf16_t>(bf16_t v) { return bf16_to_f32(v); }

template <typename T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16_t from_f32<bf16_t>(float v) { return f32_to_bf16(v); }

// eight consecutive elements as floats (p must be 16-byte aligned for bfloat16, 32 for float)
__device__ __forceinline__ void load8(const float* p, float* v) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  const float4 b = *reinterpret_cast<const float4*>(p + 4);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
__device__ __forceinline__ void load8(const bf16_t* p, float* v) {
  const uint4 a = *reinterpret_cast<const uint4*>(p);
  v[0] = bf16_bits_to_f32(a.x & 0xffffu); v[1] = bf16_bits_to_f32(a.x >> 16);
  v[2] = bf16_bits_to_f32(a.y & 0xffffu); v[3] = bf16_bits_to_f32(a.y >> 16);
  v[4] = bf16_bits_to_f32(a.z & 0xffffu); v[5] = bf16_bits_to_f32(a.z >> 16);
  v[6] = bf16_bits_to_f32(a.w & 0xffffu); v[7] = bf16_bits_to_f32(a.w >> 16);
}
__device__ __forceinline__ void store8(float* p, const float* v) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ __forceinline__ void store8(bf16_t* p, const float* v) {
  const uint4 o = make_uint4(f32_to_bf16_pair(v[0], v[1]), f32_to_bf16_pair(v[2], v[3]), f32_to_bf16_pair(v[4], v[5]), f32_to_bf16_pair(v[6], v[7]));
  *reinterpret_cast<uint4*>(p) = o;
}

// Eight neighbouring elements as they lie in memory.
template <typename T> struct Run8;
template <> struct Run8<float> {
  float4 a, b;
  __device__ __forceinline__ void load(const float* p) {
    a = *reinterpret_cast<const float4*>(p);
    b = *reinterpret_cast<const float4*>(p + 4);
  }
  __device__ __forceinline__ void floats(float (&v)[8]) const {
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
};
template <> struct Run8<bf16_t> {
  uint4 a;
  __device__ __forceinline__ void load(const bf16_t* p) { a = *reinterpret_cast<const uint4*>(p); }
  __device__ __forceinline__ void floats(float (&v)[8]) const { load8(reinterpret_cast<const bf16_t*>(&a), v); }
};

// The gated unit of a feed-forward, one element: act(s g) * (s u), with the activation a code that
// the caller passes (shared with the Python side): SiLU x / (1 + exp(-x)), or GELU in its tanh form
// 0.5 x (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3))).  One definition for the activation kernel and
// for the products that apply it in their epilogue, so both give the same bits.
// ACT_SWISH_CLAMP is the clamped form: g = min(g, limit), u = clamp(u, -limit, limit), then
// g sigmoid(1.702 g) * (u + 1); its limit travels beside the code (GatedAct).
enum : int { ACT_SILU = 1, ACT_GELU_TANH = 2, ACT_SWISH_CLAMP = 3 };
constexpr float kSwishSlope = 1.702f;
struct GatedAct {
  int code;
  float limit;      // ACT_SWISH_CLAMP only
};
static inline __host__ __device__ bool act_known(int act) {
  return act == ACT_SILU || act == ACT_GELU_TANH || act == ACT_SWISH_CLAMP;
}
static inline __host__ __device__ bool act_known(GatedAct a) {
  return act_known(a.code) && (a.code != ACT_SWISH_CLAMP || a.limit > 0.f);
}
template <int ACT> __device__ __forceinline__ float gated_f32(float limit, float g, float u) {
  if constexpr (ACT == ACT_SWISH_CLAMP) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return (g / (1.0f + expf(-kSwishSlope * g))) * (u + 1.0f);
  } else if constexpr (ACT == ACT_GELU_TANH) {
    const float t = tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g));
    return (0.5f * g * (1.0f + t)) * u;
  } else {
    return (g / (1.0f + expf(-g))) * u;
  }
}
__device__ __forceinline__ float gated_f32(GatedAct act, float g, float u, float s, bool scaled) {
  if (scaled) {
    g *= s;
    u *= s;
  }
  if (act.code == ACT_SWISH_CLAMP) return gated_f32<ACT_SWISH_CLAMP>(act.limit, g, u);
  if (act.code == ACT_GELU_TANH) return gated_f32<ACT_GELU_TANH>(act.limit, g, u);
  return gated_f32<ACT_SILU>(act.limit, g, u);
}

// An activation without a gate, one element (feed-forwards down(f(up x))).  Codes shared with the Python side: the
// square of relu; GELU in its tanh form; SiLU; GELU as x times the normal distribution function (erf).
// One definition for the activation kernel and for the products that apply it in their epilogue.
enum : int { UACT_NONE = 0, UACT_RELU2 = 1, UACT_GELU_TANH = 2, UACT_SILU = 3, UACT_GELU = 4 };
static inline __host__ __device__ bool uact_known(int f) { return f >= UACT_RELU2 && f <= UACT_GELU; }
__device__ __forceinline__ float ungated_f32(int f, float v) {
  if (f == UACT_RELU2) {
    const float r = fmaxf(v, 0.f);
    return r * r;
  }
  if (f == UACT_GELU_TANH) return 0.5f * v * (1.0f + tanhf(0.7978845608028654f * (v + 0.044715f * v * v * v)));
  if (f == UACT_GELU) return 0.5f * v * (1.0f + erff(v * 0.7071067811865476f));
  return v / (1.0f + expf(-v));
}

// Compute units of the current device (256 where none can be asked).
static inline int compute_units() {
  static int units[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (units[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    units[dev] = n;
  }
  return units[dev];
}

// dtype codes shared with the Python side
enum : int { DT_F32 = 0, DT_BF16 = 1 };

// Sums and maxima over a wave, in the pairs of lane ^ 32, 16, 8, 4, 2, 1, by register moves alone (a trip through LDS a
// step, as shuffles go, was most of a small norm's chain).  A swap of two copies of a value's halves or rows gives each lane
// both operands of its pair; inside a row of 16 a rotation by 8 pairs lane ^ 8, and as lanes 8 apart are then the same, one by 4
// pairs lane ^ 4, and so on.  Every lane of the wave takes part.  (The swap's results by __uint_as_float: __builtin_bit_cast of a
// vector's element takes element 0.)  Norm with router of one token 7.2 -> 6.3 us.
template <int ROR> __device__ __forceinline__ float row_rotated(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + ROR, 0xf, 0xf, true));
}
template <typename F> __device__ __forceinline__ float reduce32(float v, const F& f) {
  const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
template <typename F> __device__ __forceinline__ float reduce16(float v, const F& f) {
  const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(p[0]), __uint_as_float(p[1]));
}
struct SumOf { __device__ __forceinline__ float operator()(float a, float b) const { return a + b; } };
struct MaxOf { __device__ __forceinline__ float operator()(float a, float b) const { return fmaxf(a, b); } };
template <typename F> __device__ __forceinline__ float wave_reduce(float v, const F& f) {
  v = reduce16(reduce32(v, f), f);
  v = f(v, row_rotated<8>(v));
  v = f(v, row_rotated<4>(v));
  v = f(v, row_rotated<2>(v));
  return f(v, row_rotated<1>(v));
}
__device__ __forceinline__ float wave_sum(float v) { return wave_reduce(v, SumOf{}); }
__device__ __forceinline__ float wave_max(float v) { return wave_reduce(v, MaxOf{}); }

// Sums over groups of `lanes` neighbouring lanes (a power of two, the same for the wave), in the pairs of lane ^ lanes / 2, ..., 1.
__device__ __forceinline__ float group_sum(float v, int lanes) {
  if (lanes >= 16) {
    if (lanes >= 64) v = reduce32(v, SumOf{});
    if (lanes >= 32) v = reduce16(v, SumOf{});
    v += row_rotated<8>(v);
    v += row_rotated<4>(v);
    v += row_rotated<2>(v);
    return v + row_rotated<1>(v);
  }
  for (int off = lanes >> 1; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  return v;
}

// Two values of which the lanes of a pair (lane ^ 32, 16, 8) exchange one: afterwards `a` holds the lower lane's pair of values, one in each
// lane, and `b` the upper lane's.
template <int BIT> __device__ __forceinline__ void pair_swap(float& a, float& b) {
  if constexpr (BIT == 8) {
    const int ia = __builtin_bit_cast(int, a), ib = __builtin_bit_cast(int, b);
    a = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(ia, ib, 0x118, 0xf, 0xc, false));   // (row_shr:8 into lanes 8 .. 15)
    b = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(ib, ia, 0x108, 0xf, 0x3, false));   // (row_shl:8 into lanes 0 .. 7)
  } else {
    const auto p = BIT == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false)
                             : __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(p[0]);
    b = __uint_as_float(p[1]);
  }
}
// the value of lane ^ 4, 2, 1
template <int BIT> __device__ __forceinline__ float lane_xor(float v) {
  const int i = __builtin_bit_cast(int, v);
  if constexpr (BIT == 4) {
    const int up = __builtin_amdgcn_update_dpp(0, i, 0x104, 0xf, 0x5, false);                       // (row_shl:4 into lanes 0 .. 3, 8 .. 11)
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(up, i, 0x114, 0xf, 0xa, false));   // (row_shr:4 into the others)
  } else {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, i, BIT == 2 ? 0x4e : 0xb1, 0xf, 0xf, true));
  }
}

// Sum of the squares of a row that lies in `lanes` neighbouring lanes (a power of two, the same for the wave), eight elements on end a lane and
// turn, zeros behind its end; in the order of a wave that takes one element a lane and turn: a chain over the elements 64 apart, then
// the 64 in the pairs of place ^ 32, 16, 8, 4, 2, 1.  So a row has the same bits here as in the kernels for any width.  More than one turn: 64 lanes.
// Lanes 8 apart hold the chain's elements, in the same place of their eight: they exchange them until every lane has whole chains.
template <int R> __device__ __forceinline__ float row_square_sum(const float (&x)[R][8], int lanes) {
  if (R > 1 || lanes == 64) {
    float s = 0.f;
#pragma unroll
    for (int u = 0; u < R; ++u) {
      float y[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = x[u][j];
#pragma unroll
      for (int j = 0; j < 4; ++j) pair_swap<32>(y[j], y[j + 4]);
#pragma unroll
      for (int j = 0; j < 4; ++j) pair_swap<16>(y[j / 2 * 4 + j % 2], y[j / 2 * 4 + j % 2 + 2]);
#pragma unroll
      for (int j = 0; j < 4; ++j) pair_swap<8>(y[2 * j], y[2 * j + 1]);
#pragma unroll
      for (int i = 0; i < 8; ++i) s = fmaf(y[i], y[i], s);
    }
    s += lane_xor<4>(s);
    s += lane_xor<2>(s);
    s += lane_xor<1>(s);
    s = reduce16(reduce32(s, SumOf{}), SumOf{});
    return s + row_rotated<8>(s);
  }
  float y[8], s[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) y[j] = x[0][j];
  if (lanes == 32) {
#pragma unroll
    for (int j = 0; j < 4; ++j) pair_swap<16>(y[j], y[j + 4]);
#pragma unroll
    for (int j = 0; j < 4; ++j) pair_swap<8>(y[j / 2 * 4 + j % 2], y[j / 2 * 4 + j % 2 + 2]);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      s[j] = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) s[j] = fmaf(y[2 * i + j], y[2 * i + j], s[j]);
      s[j] += lane_xor<4>(s[j]);
      s[j] += lane_xor<2>(s[j]);
      s[j] += lane_xor<1>(s[j]);
      s[j] = reduce16(s[j], SumOf{});
      s[j] += row_rotated<8>(s[j]);
    }
    return s[0] + s[1];
  }
  if (lanes == 16) {
#pragma unroll
    for (int j = 0; j < 4; ++j) pair_swap<8>(y[j], y[j + 4]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      s[j] = fmaf(y[4 + j], y[4 + j], fmaf(y[j], y[j], 0.f));
      s[j] += lane_xor<4>(s[j]);
      s[j] += lane_xor<2>(s[j]);
      s[j] += lane_xor<1>(s[j]);
      s[j] += row_rotated<8>(s[j]);
    }
    return (s[0] + s[2]) + (s[1] + s[3]);
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    s[j] = fmaf(y[j], y[j], 0.f);
    if (lanes >= 8) s[j] += lane_xor<4>(s[j]);
    if (lanes >= 4) s[j] += lane_xor<2>(s[j]);
    if (lanes >= 2) s[j] += lane_xor<1>(s[j]);
  }
  return ((s[0] + s[4]) + (s[2] + s[6])) + ((s[1] + s[5]) + (s[3] + s[7]));
}

// Block-wide sum for blocks of up to 1024 threads; `red` is LDS of >= 16 floats.
// The result is the same in every thread; the order of additions is fixed.
__device__ __forceinline__ float block_sum(float v, float* red) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = threadIdx.x >> 6;
  const int nw = (blockDim.x + kWave - 1) >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) red[wid] = v;
  __syncthreads();
  float t = 0.f, part[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) part[i] = red[i];   // (all requested before the first is added)
#pragma unroll
  for (int i = 0; i < 16; ++i) t = i < nw ? t + part[i] : t;
  return t;
}

static inline int ceil_div(int a, int b) { return (a + b - 1) / b; }
