// Segments of long entries through gated linear attention (a decay per key channel; the recurrence: linear_attention.hip) as
// matrix products: what the segmented walk's two phases make, a block of eight waves a (segment, head).
//
// With D_ts the product of the decays of tokens s + 1 .. t (per key channel) and S_0 the state before the segment:
//   o_t = (q_t D_t,-1)^T S_0 + sum_(s <= t) [sum_i q_ti k_si D_tsi] v_s,   S_end = D_end,-1 S_0 + sum_s (k_s D_end,s) v_s^T.
// A factor D_ts belongs to neither t nor s alone, and dividing two running products would overflow.  So a pair is taken at a
// border between s and t: D_ts = (product from the border to t) (product from s + 1 to the border), both at most 1.  A wave
// has 16 tokens in registers (lane (i, g): a quarter of token i's channels); inside them the borders are those of halves of 2, 4,
// 8 and 16 tokens, a product of the 16 x 16 tile each, of which the pairs with that border are kept (X: from the start of the
// token's half, Y: behind the token to its end; both double their reach by the product of the other half's decays).  Between the
// waves' tokens the border is the later block's start: keys times Y lie in LDS for all, queries times X take on the decays of the
// blocks between from block to block.
//
// Decays, scores and states are float as in the walk (v_mfma_f32_16x16x4_f32); what is summed over tokens or over a
// state is summed in double (v_mfma_f64_16x16x4_f64: products of floats are exact, half the rate; with float sums the errors
// against 64 bits were 1.1 to 3 times the walk's, whose sums are short).  Scores come transposed (keys down, queries across) and are the next product's operand in their registers; the columns of values are dealt to the
// tiles so that a lane's reads of values and states are four neighbours.  A zero weight times a value that is no number
// would spoil earlier tokens: where a wave's tokens hold one, their own pairs are summed one by one.
//
// The products of decays are formed in double and rounded once: of halves for X and Y, of blocks for the queries on their way, of a whole
// segment for its state, which keeps them in double.  A product of floats 1 - a and 1 - b drops a b where that is less than half a
// place of the result, always to the same side: with products of floats, doubled from pairs on, the state's error after 1,900
// tokens of decays 1 - 2e-4 was 1.7e-5 (the walk's 7.5e-7, now 1.7e-7), of decays about 1 - 2.5e-4 1.07e-6 (5.3e-7, now 8.6e-8).
//
// Bound: what a block's waves do one after the other, and how many blocks a unit holds.  A wave makes, for 128 x 128, 400 double
// products of 64 cycles on average (32 a block of tokens up to its own, 256 for the state) and 270 float ones of 32; outputs of 128
// key channels keep 34 to 48 of their 256 registers a lane in scratch, those of 64 none.  LDS: 608 bytes a key channel and 256 or 512
// (float) a value column, 59 KB (bf16, 64 x 64: two blocks a unit) to 152 (float, 128 x 128).  All launches of a call, bf16, us of the
// walk's phases and of the products: 16 heads of 128 x 128, 1,900 tokens 216 -> 116, 512 tokens 110 -> 105; 32 heads, 4,000 tokens 711 ->
// 386; 16 heads of 64 x 64, two of 600 72 -> 41.  Errors against 64 bits, 1,900 tokens: outputs 1.25e-7 -> 1.07e-7, state 7.7e-8 -> 4.6e-8.
#include "gla_chunk.h"

#include <type_traits>

#include "state_walk.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int kBlockTokens = 16, kGlaWaves = kSeg / kBlockTokens, kGlaThreads = kGlaWaves * kWave;
constexpr int kSliceCols = 8;            // value columns of a state slice (linear_attention.hip)

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// the neighbouring lane's value
__device__ __forceinline__ float neighbour(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), 0xB1, 0xF, 0xF, true));
}

// A score is eight chains of channels: a sum's rounding grows with its length.
constexpr int kChains = 4;
__device__ __forceinline__ f32x4 sum_of(const f32x4* c) { return (c[0] + c[1]) + (c[2] + c[3]); }

// Sums of values and of states are of doubles: products of floats, exact, on the double matrix instruction (half the float one's
// rate); its result's register v holds row g + 4 v.
typedef __attribute__((ext_vector_type(4))) double f64x4;
__device__ __forceinline__ f64x4 mfma4(double a, double b, f64x4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }

template <typename T> __device__ __forceinline__ void read4(const T* p, float* v) {
  if constexpr (sizeof(T) == 4) {
    const f32x4 x = *reinterpret_cast<const f32x4*>(p);
    v[0] = x[0]; v[1] = x[1]; v[2] = x[2]; v[3] = x[3];
  } else {
    const uint2 x = *reinterpret_cast<const uint2*>(p);
    v[0] = bf16_bits_to_f32(x.x & 0xffffu); v[1] = bf16_bits_to_f32(x.x >> 16);
    v[2] = bf16_bits_to_f32(x.y & 0xffffu); v[3] = bf16_bits_to_f32(x.y >> 16);
  }
}

// Tokens t0 .. t0 + nt - 1 (kSeg at most) of segment `seg`: `begins` and `ends` where they are its first and its last, `last` where the
// segment is its entry's last.
template <typename T, int DK, int DV, bool FINAL>
__device__ __forceinline__ void gla_chunk(const GlaChunkArgs& a, int seg, int h, int e, int t0, int nt, bool begins, bool ends, bool last) {
  constexpr int CH = DK / 4, RPL = DK / 8, NH = DV / 64, NT = DV / 16;
  constexpr int LDV = DV + 16;
  // keys times Y; before, of every block of 16 tokens the products of the decays of its pairs (rows 0 .. 7 of the block), fours (8 .. 11)
  // and eights (12, 13); 16-byte pieces swizzled (k_piece)
  __shared__ __attribute__((aligned(16))) float ks[kSeg][DK];
  __shared__ __attribute__((aligned(16))) T vs[kSeg][LDV];
  __shared__ __attribute__((aligned(16))) float bt[kGlaWaves][DK];     // the products of the blocks' decays,
  __shared__ double bd[kGlaWaves][DK];                                 // and before they are rounded
  __shared__ int odd[kGlaWaves];                                       // whether a block's values hold one that is no number
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));        // (a chunk's addresses are formed in it: kept from one to the next they would fill the registers)
  const int lane = tid & (kWave - 1), wid = __builtin_amdgcn_readfirstlane(tid >> 6), i = lane & 15, g = lane >> 4;
  const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
  const int I = wid < 4 ? wid : 11 - wid;                              // blocks of 16 tokens: waves of one SIMD get an early and a late one
  auto k_piece = [](int t, int piece) { return piece ^ (t & 7); };

  if (tid < kGlaWaves) odd[tid] = 0;
  const T* proj = (const T*)a.proj;
  const int t = I * kBlockTokens + i;
  const bool live = t < nt;
  const size_t row = (size_t)max(t0 + min(t, nt - 1), 0);              // (no token: one that exists, unused)
  // a block's decays of one channel a thread, for their products
  constexpr int COLUMNS = kGlaWaves * DK / kGlaThreads;
  float f[COLUMNS][kBlockTokens];
#pragma unroll
  for (int n = 0; n < COLUMNS; ++n) {
    const int J = (tid + n * kGlaThreads) / DK, ch = tid % DK;
#pragma unroll
    for (int x = 0; x < kBlockTokens; ++x) {
      const int tx = J * kBlockTokens + x;
      f[n][x] = a.alpha[(size_t)max(t0 + min(tx, nt - 1), 0) * (size_t)(a.nh * DK) + h * DK + ch];
      f[n][x] = tx < nt ? f[n][x] : 1.f;
    }
  }
  float k[CH], X[CH], Y[CH], q[FINAL ? CH : 1];
#pragma unroll
  for (int m = 0; m < CH; m += 8) {
    load8(proj + row * a.stride + a.k_off + h * DK + CH * g + m, k + m);
    load8(a.alpha + row * (size_t)(a.nh * DK) + h * DK + CH * g + m, X + m);
    if constexpr (FINAL) load8(proj + row * a.stride + a.q_off + h * DK + CH * g + m, q + m);
  }
#pragma unroll
  for (int n = 0; n < COLUMNS; ++n) {
    const int J = (tid + n * kGlaThreads) / DK, ch = tid % DK;
    auto put = [&](int node, double d) { ks[J * kBlockTokens + node][k_piece(node, ch >> 2) * 4 + (ch & 3)] = (float)d; };
    double d[8];
#pragma unroll
    for (int x = 0; x < 8; ++x) put(x, d[x] = (double)f[n][2 * x] * (double)f[n][2 * x + 1]);
#pragma unroll
    for (int x = 0; x < 4; ++x) put(8 + x, d[x] = d[2 * x] * d[2 * x + 1]);
#pragma unroll
    for (int x = 0; x < 2; ++x) put(12 + x, d[x] = d[2 * x] * d[2 * x + 1]);
    bd[J][ch] = d[0] * d[1];
    bt[J][ch] = (float)(d[0] * d[1]);
  }
  __syncthreads();
  // values into LDS
  constexpr int PV = 16 / (int)sizeof(T);
  for (int idx = tid; idx < kSeg * (DV / PV); idx += kGlaThreads) {
    const int tv = idx / (DV / PV), c = (idx % (DV / PV)) * PV;
    uint4 raw = make_uint4(0, 0, 0, 0);
    if (tv < nt) raw = *reinterpret_cast<const uint4*>(proj + (size_t)(t0 + tv) * a.stride + a.v_off + h * DV + c);
    *reinterpret_cast<uint4*>(&vs[tv][c]) = raw;
    bool bad;
    if constexpr (sizeof(T) == 4) {
      auto is = [](uint32_t x) { return (x & 0x7f800000u) == 0x7f800000u; };
      bad = is(raw.x) || is(raw.y) || is(raw.z) || is(raw.w);
    } else {
      auto is = [](uint32_t x) { return (x & 0x7f80u) == 0x7f80u || (x & 0x7f800000u) == 0x7f800000u; };
      bad = is(raw.x) || is(raw.y) || is(raw.z) || is(raw.w);
    }
    if (bad) odd[tv / kBlockTokens] = 1;
  }
#pragma unroll
  for (int m = 0; m < CH; ++m) {
    k[m] = live ? k[m] : 0.f;
    X[m] = live ? X[m] : 1.f;
    Y[m] = 1.f;
    if constexpr (FINAL) q[m] = live ? q[m] * a.q_scale : 0.f;
  }
  // the pairs of the wave's own tokens: lane (i, g) gets query i with keys 4 g + 0..3
  f32x4 own = f32x4{0.f, 0.f, 0.f, 0.f};
  auto tile = [&](auto scaled_tag) {
    constexpr bool scaled = decltype(scaled_tag)::value;
    f32x4 all = zero;
#pragma unroll
    for (int m0 = 0; m0 < CH; m0 += CH / 2) {
      f32x4 c[kChains];
#pragma unroll
      for (int m = m0; m < m0 + CH / 2; ++m) {
        c[m % kChains] = mfma4(scaled ? k[m] * Y[m] : k[m], scaled ? q[m] * X[m] : q[m], m < m0 + kChains ? zero : c[m % kChains]);
        if (m % 4 == 3) asm volatile("" : "+v"(c[m % kChains]));       // (all scaled operands ahead would not fit the registers)
      }
      all = m0 == 0 ? sum_of(c) : all + sum_of(c);
    }
    return all;
  };
  if constexpr (FINAL) {
    const f32x4 c = tile(std::false_type{});
#pragma unroll
    for (int v = 0; v < 4; ++v) own[v] = 4 * g + v == i ? c[v] : 0.f;
  }
  auto level = [&](auto half_tag) {
    constexpr int H = decltype(half_tag)::value;
    if constexpr (FINAL) {
      const f32x4 c = tile(std::true_type{});
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int s = 4 * g + v;
        if ((s ^ i) < 2 * H && (i & H) && !(s & H)) own[v] = c[v];
      }
    }
    const bool up = i & H;
    const int node = (H == 2 ? 0 : H == 4 ? 8 : 12) + ((i / H) ^ 1);   // the other half
#pragma unroll
    for (int m = 0; m < CH; m += 4) {
      f32x4 p;
      if constexpr (H == 1) p = f32x4{neighbour(X[m]), neighbour(X[m + 1]), neighbour(X[m + 2]), neighbour(X[m + 3])};
      else p = *reinterpret_cast<const f32x4*>(&ks[I * kBlockTokens + node][k_piece(node, (CH * g + m) / 4) * 4]);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        X[m + x] *= up ? p[x] : 1.f;
        Y[m + x] *= up ? 1.f : p[x];
        asm volatile("" : "+v"(X[m + x]), "+v"(Y[m + x]));             // (a few channels after the others, for the registers' sake)
      }
    }
  };
  level(std::integral_constant<int, 1>{});
  level(std::integral_constant<int, 2>{});
  level(std::integral_constant<int, 4>{});
  level(std::integral_constant<int, 8>{});
#pragma unroll
  for (int m = 0; m < CH; m += 4) {
    *reinterpret_cast<f32x4*>(&ks[t][k_piece(t, (CH * g + m) / 4) * 4]) = f32x4{k[m] * Y[m], k[m + 1] * Y[m + 1], k[m + 2] * Y[m + 2], k[m + 3] * Y[m + 3]};
  }
  __syncthreads();

  const size_t seg_floats = (size_t)(DV / kSliceCols) * DK * kSliceCols;
  float* S_seg = a.seg_state + ((size_t)seg * a.nh + h) * seg_floats;
  const int blocks = (nt + kBlockTokens - 1) / kBlockTokens;           // (those behind hold no token)
  if (FINAL && I < blocks) {
    float qx[FINAL ? CH : 1];
    f64x4 acc[NT];
#pragma unroll
    for (int m = 0; m < CH; ++m) qx[m] = q[m] * X[m];
#pragma unroll
    for (int c = 0; c < NT; ++c) acc[c] = f64x4{0.0, 0.0, 0.0, 0.0};
    // tile c of the outputs has columns 64 (c / 4) + 4 (row) + c % 4: one read brings a lane four tiles' operands
    auto add_values = [&](const f32x4& w, int J) {
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int hi = 0; hi < NH; ++hi) {
          float v[4];
          read4<T>(&vs[J * kBlockTokens + 4 * g + m][64 * hi + 4 * i], v);
#pragma unroll
          for (int c = 0; c < 4; ++c) acc[4 * hi + c] = mfma4((double)v[c], (double)w[m], acc[4 * hi + c]);
        }
    };
    if (!odd[I]) {
      add_values(own, I);
    } else {
      for (int s = 0; s < kBlockTokens; ++s) {
        const float mine = s % 4 == 0 ? own[0] : s % 4 == 1 ? own[1] : s % 4 == 2 ? own[2] : own[3];
        const float w = __shfl(mine, (s / 4) * 16 + i, kWave);
        if (i < s) continue;
#pragma unroll
        for (int hi = 0; hi < NH; ++hi)
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            float x[4];
            read4<T>(&vs[I * kBlockTokens + s][64 * hi + 4 * g + 16 * v], x);
#pragma unroll
            for (int c = 0; c < 4; ++c) acc[4 * hi + c][v] += (double)w * (double)x[c];
          }
      }
    }
    auto take_on = [&](int J) {                                        // the decays of block J
#pragma unroll
      for (int m = 0; m < CH; m += 4) {
        const f32x4 b = *reinterpret_cast<const f32x4*>(&bt[J][CH * g + m]);
#pragma unroll
        for (int x = 0; x < 4; ++x) qx[m + x] *= b[x];
      }
    };
    for (int J = I - 1; J >= 0; --J) {
      f32x4 all = zero;
      const int tk = J * kBlockTokens + i;
#pragma unroll
      for (int m0 = 0; m0 < CH; m0 += CH / 2) {
        f32x4 cs[kChains];
#pragma unroll
        for (int m = m0; m < m0 + CH / 2; m += 4) {
          const f32x4 kk = *reinterpret_cast<const f32x4*>(&ks[tk][k_piece(tk, (CH * g + m) / 4) * 4]);
#pragma unroll
          for (int x = 0; x < 4; ++x)
            cs[(m + x) % kChains] = mfma4(kk[x], qx[m + x], m + x < m0 + kChains ? zero : cs[(m + x) % kChains]);
        }
        all = m0 == 0 ? sum_of(cs) : all + sum_of(cs);
      }
      add_values(all, J);
      take_on(J);
    }
    // the state before the segment: channel CH g + m lies in row group 2 g + m / RPL, place m % RPL
#pragma unroll
    for (int m = 0; m < CH; ++m) {
      const int place = (m % RPL) * 8 + 2 * g + m / RPL;
#pragma unroll
      for (int hi = 0; hi < NH; ++hi) {
        const f32x4 s0 = *reinterpret_cast<const f32x4*>(S_seg + ((size_t)(8 * hi + (i >> 1)) * DK + place) * kSliceCols + 4 * (i & 1));
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[4 * hi + c] = mfma4((double)s0[c], (double)qx[m], acc[4 * hi + c]);
      }
      if (m % 8 == 7) __builtin_amdgcn_sched_barrier(0);               // (all the state's reads ahead would not fit the registers)
    }
    if (live) {
      float* o = a.out + (size_t)(t0 + t) * (size_t)(a.nh * DV) + h * DV + 4 * g;
#pragma unroll
      for (int hi = 0; hi < NH; ++hi)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          *reinterpret_cast<f32x4*>(o + 64 * hi + 16 * v) = f32x4{(float)acc[4 * hi][v], (float)acc[4 * hi + 1][v], (float)acc[4 * hi + 2][v], (float)acc[4 * hi + 3][v]};
    }
  }
  const bool to_slot = FINAL && ends && last;
  if (FINAL && ends && !last) return;
  if (FINAL && !ends) __syncthreads();                                 // (the outputs above have read what is written below)

  // The state: a wave has 16 rows of it (two neighbouring places of all eight row groups) and 64 columns at a time.
  constexpr int RW = DK / 16;                                          // waves over the rows, the others over the columns
  const int r = 2 * (wid % RW) + (i >> 3), g8 = i & 7, ch = g8 * RPL + r;
  float* S_to = to_slot ? a.state + ((size_t)a.state_slots[e] * a.nh + h) * seg_floats : S_seg;
  for (int hi = wid / RW; hi < NH; hi += kGlaWaves / RW) {
    f64x4 acc[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = f64x4{0.0, 0.0, 0.0, 0.0};
    double keep = 1.0;                                                 // the decays of the blocks behind J
    for (int J = blocks - 1; J >= 0; --J) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int tk = J * kBlockTokens + 4 * u + g;
        const double kv = (double)ks[tk][k_piece(tk, ch >> 2) * 4 + (ch & 3)] * keep;
        float v[4];
        read4<T>(&vs[tk][64 * hi + 4 * i], v);
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] = mfma4((double)v[c], kv, acc[c]);
      }
      keep *= bd[J][ch];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const size_t at = ((size_t)(8 * hi + 2 * v + (g >> 1)) * DK + r * 8 + g8) * kSliceCols + 4 * (g & 1);
      double s[4] = {acc[0][v], acc[1][v], acc[2][v], acc[3][v]};
      if (FINAL || !begins) {
        const f32x4 s0 = *reinterpret_cast<const f32x4*>(S_seg + at);
#pragma unroll
        for (int c = 0; c < 4; ++c) s[c] += keep * (double)s0[c];
      }
      *reinterpret_cast<f32x4*>(S_to + at) = f32x4{(float)s[0], (float)s[1], (float)s[2], (float)s[3]};
    }
    if (!FINAL && hi == 0 && g == 0) {
      float* d = a.seg_decay + ((size_t)seg * a.nh + h) * DK + ch;
      *d = begins ? (float)keep : (float)(keep * (double)*d);
    }
  }
}

// FINAL: outputs, and the state in its slot where the segment is its entry's last; else what the segment makes of nothing and
// the product of its decays.  The step's own lists cut segments to kSeg tokens; a longer one, of a caller's own list, goes in
// chunks of so many, the state between them where the segment's state is kept.
template <typename T, int DK, int DV, bool FINAL>
__global__ __launch_bounds__(kGlaThreads, 2) void gla_chunk_kernel(GlaChunkArgs a) {
  const int seg = blockIdx.x, h = blockIdx.y;
  const int e = a.segs[4 * seg], first = a.segs[4 * seg + 1], tokens = a.segs[4 * seg + 2];
  const bool last = a.segs[4 * seg + 3] != 0;
  if (!FINAL && last) return;                                          // (nobody reads it)
  for (int done = 0;; done += kSeg) {
    const bool ends = tokens - done <= kSeg;
    gla_chunk<T, DK, DV, FINAL>(a, seg, h, e, first + done, ends ? max(tokens - done, 0) : kSeg, done == 0, ends, last);
    if (ends) return;
    __syncthreads();
  }
}

bool gla_chunk_takes(int dtype, int stride, int q_off, int k_off, int v_off, const GlaChunkArgs& a, int dk, int dv) {
  const int piece = dtype == DT_F32 ? 4 : 8;
  if (!((dk == 64 || dk == 128) && (dv == 64 || dv == 128))) return false;
  if (stride % piece || q_off % piece || k_off % piece || v_off % piece) return false;
  return (((uintptr_t)a.proj | (uintptr_t)a.alpha | (uintptr_t)a.out | (uintptr_t)a.state | (uintptr_t)a.seg_state) & 15) == 0;
}

void gla_chunk_launch(int dtype, const GlaChunkArgs& a, int dk, int dv, int n_segs, bool final, hipStream_t stream) {
  const dim3 grid(n_segs, a.nh);
#define GC(T, DKV, DVV)                                                                      \
  do {                                                                                       \
    if (final) gla_chunk_kernel<T, DKV, DVV, true><<<grid, kGlaThreads, 0, stream>>>(a);      \
    else gla_chunk_kernel<T, DKV, DVV, false><<<grid, kGlaThreads, 0, stream>>>(a);           \
  } while (0)
#define GC_T(T)                                   \
  do {                                            \
    if (dk == 64 && dv == 64) GC(T, 64, 64);      \
    else if (dk == 64) GC(T, 64, 128);            \
    else if (dv == 64) GC(T, 128, 64);            \
    else GC(T, 128, 128);                         \
  } while (0)
  if (dtype == DT_F32) GC_T(float);
  else GC_T(bf16_t);
#undef GC_T
#undef GC
}
