// Segments of long entries through a recurrent state with one decay per (token, head), as matrix products.
//
// The recurrence (state_walk.hip) over a segment of up to 128 tokens that starts from S_0, with G_t the sum of
// the logarithms of the decays up to and with token t:
//     o_t   = exp(G_t) S_0^T q_t + sum_(s <= t) exp(G_t - G_s) b_s (k_s . q_t) v_s
//     S_end = exp(G_end) S_0 + sum_s exp(G_end - G_s) b_s k_s v_s^T
// and with exponential gates the same with exp(G_t - G_s + i_s - m_t) for the weights, m_t = max(G_t + m_0,
// max_(s <= t)(G_t - G_s + i_s)), and the normaliser's n_t . q_t as the plain sum of the weighted scores.  A
// weight's exponent is u_s - r_t with u_s = i_s - G_s (or -G_s) and r_t = m_t - G_t (or -G_t): sums over the
// segment, kept in double and handed on as pairs of floats, so that a weight is as exact as one exponential of a
// small difference, where the walk multiplied up to 128 factors.
//
// A block (eight waves) is one (segment, head), all value columns.  state_chunk_local makes what a segment
// makes of nothing (K^T times weighted V), state_chunk_final the outputs and, for an entry's last segment, the new
// state.  A wave has 16 queries; scores come transposed (keys down, queries across), so that the weighted scores are the next product's
// operand without leaving their registers, and so does O^T.  Scores of bfloat16 q and k use the bfloat16
// instruction (its products are exact, its sums float); the other products v_mfma_f32_16x16x4_f32: states,
// weights and sums stay float.
//
// Bound: the float matrix instruction, 0.8 k of them a wave and full segment, against a token at a time in the walk
// (0.7 us a token, whatever the width of the chip).  All launches of a call, microseconds before and after: 16 heads of 128 x 128
// with exponential gates, 2,048 tokens 1,445 -> 88, 8,192 tokens 5,743 -> 260, prompts of 1,024 and 910 tokens beside 16
// single ones 734 -> 88; 64 state-space heads of 128 x 64, 2,048 tokens 1,072 -> 140; 16 heads with a fixed decay,
// 2,048 tokens 947 -> 104.
#include <type_traits>

#include "state_walk.h"

using f32x4 = __attribute__((__vector_size__(4 * sizeof(float)))) float;
using bf16x8 = __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16;

constexpr int kChunkWaves = 8;
constexpr int kChunkThreads = kChunkWaves * kWave;
constexpr int kPadK = 8, kPadV = 16;   // elements behind an LDS row of k and of v (bfloat16: banks 4 and 8 apart from row to row)

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// what a segment's tokens weigh, per token: weight(t, s) = exp((uh_s - rh_t) + (ul_s - rl_t)) b_s
struct SegWeights {
  float uh[kSeg], ul[kSeg], b[kSeg], rh[kSeg], rl[kSeg], inter[kSeg], e[kSeg], end[kSeg];
  float inter_end, log_decay, m_end;
  int odd[kChunkWaves];              // whether a wave staged a value that is no number
};

__device__ __forceinline__ void split(double x, float& hi, float& lo) {
  hi = (float)x;
  lo = isinf(hi) ? 0.f : (float)(x - (double)hi);
}

// Logarithms of decays below this count as it: such a decay is 0 in float, and so are the products it is in, while sums
// of 128 of them still carry the others' logarithms (a decay of 0 itself would make them infinite, and differences of
// infinite sums are no numbers).
constexpr double kLeastLog = -1e4;
__device__ __forceinline__ double log_of_decay(double x) { return x < kLeastLog ? kLeastLog : x; }

// By one wave: two neighbouring tokens a lane.  LOCAL: from nothing (the maximum starts at minus infinity).
template <int MODE, bool LOCAL>
__device__ void segment_weights(SegWeights& w, const WalkArgs& a, int h, int t0, int nt, float m_start, int lane) {
  double f[2], i[2], b[2];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    const int t = 2 * lane + x;
    const bool live = t < nt;
    f[x] = 0.0;
    i[x] = MODE == WALK_EXP_GATES ? -INFINITY : 0.0;
    b[x] = 0.0;
    if (MODE == WALK_FIXED_DECAY) {
      if (live) f[x] = log_of_decay(log((double)a.p0[h])), b[x] = a.k_scale;
    } else if (live) {
      const float* row = a.gates + (size_t)(t0 + t) * a.gate_stride;
      if (MODE == WALK_EXP_GATES) {
        i[x] = a.cap * tanhf((row[h] + a.p0[h]) / a.cap);
        f[x] = log_sigmoid_f32(a.cap * tanhf((row[a.nh + h] + a.p1[h]) / a.cap));
        b[x] = 1.0;
      } else {
        const float dt = softplus_f32(row[h] + a.p0[h]);
        f[x] = log_of_decay(-expf(a.p1[h]) * dt);
        b[x] = dt;
      }
    }
  }
  // a logarithm that is no number stays out of the sums (a lane's first token has the pair's less the second) and is put back
  // into those from its token on
  const uint64_t odd0 = __ballot(!(fabs(f[0]) < INFINITY)), odd1 = __ballot(!(fabs(f[1]) < INFINITY));
  if (odd0 >> lane & 1) f[0] = 0.0;
  if (odd1 >> lane & 1) f[1] = 0.0;
  double upto = f[0] + f[1];                         // inclusive sums over the lanes
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const double x = __shfl_up(upto, o, kWave);
    if (lane >= o) upto += x;
  }
  double G1 = upto, G0 = upto - f[1];
  if (odd0 | odd1) {
    const uint64_t from = 1ull << lane, odd = (odd0 | odd1) & (from - 1);     // of earlier lanes, then of the lane's own tokens
    if (odd || (odd0 & from)) G0 = NAN;
    if (odd || ((odd0 | odd1) & from)) G1 = NAN;
  }
  const double u0 = i[0] - G0, u1 = i[1] - G1;
  double r0 = -G0, r1 = -G1, r_end, inter0 = G0, inter1 = G1;
  const double G_end = __shfl(G1, kWave - 1, kWave);          // (tokens beyond the segment add nothing)
  if (MODE == WALK_EXP_GATES) {
    double top = fmax(u0, u1);
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
      const double x = __shfl_up(top, o, kWave);
      if (lane >= o) top = fmax(top, x);
    }
    double before = __shfl_up(top, 1, kWave);
    if (lane == 0) before = -INFINITY;
    const double m0 = LOCAL ? -INFINITY : (double)m_start;
    r0 = fmax(fmax(before, u0), m0);
    r1 = fmax(top, m0);
    r_end = __shfl(r1, kWave - 1, kWave);
    inter0 = m0 - r0;
    inter1 = m0 - r1;
    if (lane == 0) w.inter_end = LOCAL ? 0.f : expf((float)(m0 - r_end)), w.m_end = (float)(G_end + r_end);
    w.e[2 * lane] = expf(-(float)(G0 + r0));
    w.e[2 * lane + 1] = expf(-(float)(G1 + r1));
  } else {
    r_end = -G_end;
    if (lane == 0) w.inter_end = LOCAL ? 0.f : expf((float)G_end);
  }
  if (lane == 0) w.log_decay = (float)G_end;
  const double u[2] = {u0, u1}, r[2] = {r0, r1}, inter[2] = {inter0, inter1};
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    const int t = 2 * lane + x;
    split(u[x], w.uh[t], w.ul[t]);
    split(r[x], w.rh[t], w.rl[t]);
    w.b[t] = (float)b[x];
    w.inter[t] = LOCAL ? 0.f : expf((float)inter[x]);
    w.end[t] = t < nt ? expf((float)(u[x] - r_end)) * (float)b[x] : 0.f;
  }
}

template <typename KT> __device__ __forceinline__ KT zero_of();
template <> __device__ __forceinline__ float zero_of<float>() { return 0.f; }
template <> __device__ __forceinline__ bf16_t zero_of<bf16_t>() { return bf16_t{0}; }

// The largest magnitudes of 16 bytes' elements so far, as their bits (of bfloat16 two by two), and whether one of them is infinite
// or no number.
template <typename T> struct Magnitudes;
template <> struct Magnitudes<float> {
  uint32_t most = 0;
  __device__ __forceinline__ void add(uint32_t x) { most = max(most, x & 0x7fffffffu); }
  __device__ __forceinline__ bool odd() const { return most >= 0x7f800000u; }
};
template <> struct Magnitudes<bf16_t> {
  using u16x2 = __attribute__((__vector_size__(4))) unsigned short;
  u16x2 most = {0, 0};
  __device__ __forceinline__ void add(uint32_t x) { most = __builtin_elementwise_max(most, __builtin_bit_cast(u16x2, x & 0x7fff7fffu)); }
  __device__ __forceinline__ bool odd() const { return most[0] >= 0x7f80 || most[1] >= 0x7f80; }
};

// `rows` (a multiple of 16) rows of W elements from column `off` of proj into LDS rows of W + kPad, zeros beyond nt; 16-byte loads.
// Returns whether the thread's elements hold one that is no number.
template <typename T, typename KT, int W, int LD>
__device__ __forceinline__ bool stage_rows(KT* dst, const T* __restrict__ proj, int stride, int off, int t0, int nt, int rows) {
  constexpr int V = 16 / (int)sizeof(T);
  Magnitudes<T> seen;
  for (int idx = threadIdx.x; idx < rows * (W / V); idx += kChunkThreads) {
    const int t = idx / (W / V), c = (idx % (W / V)) * V;
    const T* src = proj + (size_t)(t0 + min(t, nt - 1)) * stride + off + c;
    KT* to = dst + t * LD + c;
    uint4 raw = *reinterpret_cast<const uint4*>(src);
    if (t >= nt) raw = make_uint4(0, 0, 0, 0);
    seen.add(raw.x);
    seen.add(raw.y);
    seen.add(raw.z);
    seen.add(raw.w);
    if constexpr (sizeof(KT) == sizeof(T)) {
      *reinterpret_cast<uint4*>(to) = raw;
    } else {
      float x[V];
      load8(reinterpret_cast<const T*>(&raw), x);
#pragma unroll
      for (int i = 0; i < V; i += 4)
        *reinterpret_cast<float4*>(to + i) = make_float4(x[i], x[i + 1], x[i + 2], x[i + 3]);
    }
  }
  return seen.odd();
}

// rotary positions on staged floats: element i of a row with element i + half
template <int W>
__device__ __forceinline__ void turn_rows(float* rows, const int* __restrict__ positions, const float* __restrict__ inv_freq, int t0,
                                          int nt, int half) {
  for (int idx = threadIdx.x; idx < nt * half; idx += kChunkThreads) {
    const int t = idx / half, i = idx % half;
    const float ang = (float)positions[t0 + t] * inv_freq[i];
    const float cs = cosf(ang), sn = sinf(ang);
    float* r = rows + t * (W + kPadK);
    const float x = r[i], y = r[i + half];
    r[i] = x * cs - y * sn;
    r[i + half] = y * cs + x * sn;
  }
}

// sum_s end_s k_s v_s^T (and the normaliser's sum) of a staged segment, plus inter_end times `from` where there is one,
// into the state's slices at `to`.  A tile has 16 rows, two neighbouring r of all eight row groups, so that its
// columns are stored 16 bytes a lane and 512 in a row; a wave has one tile and all columns (64 rows: half of them).
template <typename T, typename KT, int DK, int NCT, int MODE>
__device__ __forceinline__ void segment_state(const SegWeights& w, const KT* k_s, const T* v_s, int rows, const float* from, float* to) {
  constexpr int RPL = DK / 8, DV = NCT * 16, NOFF = RPL * 64;
  constexpr int RW = DK / 16, CW = NCT * RW / kChunkWaves;        // waves over the rows; column tiles of a wave
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x >> 6, g = lane >> 4, i = lane & 15;
  const int r = wid % RW * 2 + (i >> 3), g8 = i & 7, ct0 = wid / RW * CW;
  const int slice = walk_slice_floats(DK, MODE);
  const size_t at = (size_t)(2 * ct0 + (g >> 1)) * slice + r * 64 + 8 * g8 + 4 * (g & 1);
  float4 old[CW];
  if (from) {
#pragma unroll
    for (int ct = 0; ct < CW; ++ct) old[ct] = *reinterpret_cast<const float4*>(from + at + (size_t)(2 * ct) * slice);
  }
  f32x4 acc[CW];
  float nsum = 0.f;
#pragma unroll
  for (int ct = 0; ct < CW; ++ct) acc[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int t0 = 0; t0 < rows; t0 += 16) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int t = t0 + 4 * u + g;
      const float kv = to_f32<KT>(k_s[t * (DK + kPadK) + g8 * RPL + r]) * w.end[t];
      if (MODE == WALK_EXP_GATES) nsum += kv;
#pragma unroll
      for (int ct = 0; ct < CW; ++ct) acc[ct] = mfma_f32(to_f32<T>(v_s[t * (DV + kPadV) + (ct0 + ct) * 16 + i]), kv, acc[ct]);
    }
  }
  const float keep = w.inter_end;
#pragma unroll
  for (int ct = 0; ct < CW; ++ct) {
    float4 x = make_float4(acc[ct][0], acc[ct][1], acc[ct][2], acc[ct][3]);
    if (from) x = make_float4(fmaf(keep, old[ct].x, x.x), fmaf(keep, old[ct].y, x.y), fmaf(keep, old[ct].z, x.z), fmaf(keep, old[ct].w, x.w));
    *reinterpret_cast<float4*>(to + at + (size_t)(2 * ct) * slice) = x;
  }
  if (MODE == WALK_EXP_GATES && ct0 == 0) {
    nsum = reduce16(nsum, SumOf{});
    nsum = reduce32(nsum, SumOf{});
    const int n_at = NOFF + ((r >> 2) * 8 + g8) * 4 + (r & 3);
    if (from) nsum = fmaf(keep, from[n_at], nsum);
    for (int cb = g; cb < 2 * NCT; cb += 4) to[(size_t)cb * slice + n_at] = nsum;     // (every slice has its copy)
  }
  if (MODE == WALK_EXP_GATES && threadIdx.x < 2 * NCT) to[(size_t)threadIdx.x * slice + NOFF + DK] = w.m_end;
}

template <typename T, int DK, int NCT, int MODE>
__global__ __launch_bounds__(kChunkThreads) void state_chunk_local_kernel(const WalkArgs a) {
  constexpr int DV = NCT * 16;
  constexpr bool TURN = MODE == WALK_FIXED_DECAY;
  using KT = std::conditional_t<TURN, float, T>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  KT* k_s = reinterpret_cast<KT*>(smem);
  T* v_s = reinterpret_cast<T*>(k_s + kSeg * (DK + kPadK));
  SegWeights& w = *reinterpret_cast<SegWeights*>(v_s + kSeg * (DV + kPadV));
  const int h = blockIdx.x;
  const int* sg = a.segs + 4 * blockIdx.y;
  const int t0 = sg[1], nt = min(sg[2], kSeg);
  if (sg[3] != 0 || nt <= 0) return;                 // nobody starts from what an entry's last segment makes
  const int rows = (nt + 15) / 16 * 16;
  const T* proj = static_cast<const T*>(a.proj);
  stage_rows<T, KT, DK, DK + kPadK>(k_s, proj, a.stride, a.k_off + (h / a.heads_per_group) * DK, t0, nt, rows);
  stage_rows<T, T, DV, DV + kPadV>(v_s, proj, a.stride, a.v_off + h * DV, t0, nt, rows);
  if (threadIdx.x >= kChunkThreads - kWave) segment_weights<MODE, true>(w, a, h, t0, nt, 0.f, threadIdx.x & (kWave - 1));
  __syncthreads();
  if constexpr (TURN) {
    if (a.rot_dim > 0) {
      turn_rows<DK>(k_s, a.positions, a.inv_freq, t0, nt, a.rot_dim >> 1);
      __syncthreads();
    }
  }
  const int ncb = DV / kWalkCols, slice = walk_slice_floats(DK, MODE);
  float* to = a.seg_local + ((size_t)blockIdx.y * a.nh + h) * ncb * slice;
  segment_state<T, KT, DK, NCT, MODE>(w, k_s, v_s, rows, nullptr, to);
  if (threadIdx.x == 0) a.seg_decay[(size_t)blockIdx.y * a.nh + h] = w.log_decay;
}

template <typename T, int DK, int NCT, int MODE>
__device__ __forceinline__ void state_chunk_final_block(const WalkArgs& a) {
  constexpr int DV = NCT * 16, RPL = DK / 8, NOFF = RPL * 64;
  constexpr int EL = DK / 4;                         // elements of a query a lane holds: rows (g + 4 gh) RPL + r, gh = 0, 1
  constexpr bool TURN = MODE == WALK_FIXED_DECAY;
  using KT = std::conditional_t<TURN, float, T>;
  constexpr bool HALF = sizeof(KT) == 2;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  KT* k_s = reinterpret_cast<KT*>(smem);
  T* v_s = reinterpret_cast<T*>(k_s + kSeg * (DK + kPadK));
  SegWeights& w = *reinterpret_cast<SegWeights*>(v_s + kSeg * (DV + kPadV));
  const int h = blockIdx.x, lane = threadIdx.x & (kWave - 1), wid = threadIdx.x >> 6, g = lane >> 4, i = lane & 15;
  const int* sg = a.segs + 4 * blockIdx.y;
  const int e = sg[0], t0 = sg[1], nt = min(sg[2], kSeg);
  const bool last = sg[3] != 0;
  const bool only = last && t0 == a.cu_tokens[e];    // an entry's only segment starts from the slot
  if (nt <= 0 || (only ? nt < kChunkFrom : (int)blockIdx.y >= a.n_scratch)) return;
  const int rows = (nt + 15) / 16 * 16, tiles = rows / 16;
  const T* proj = static_cast<const T*>(a.proj);
  const int ncb = DV / kWalkCols, slice = walk_slice_floats(DK, MODE);
  const size_t per_head = (size_t)ncb * slice;
  float* slot = a.state + ((size_t)a.state_slots[e] * a.nh + h) * per_head;
  const float* from = only ? slot : a.seg_start + ((size_t)blockIdx.y * a.nh + h) * per_head;
  const int q_col = a.q_off + (h / a.heads_per_group) * DK, k_col = a.k_off + (h / a.heads_per_group) * DK;

  // the wave's tile of 16 queries and their elements; the two tiles of a SIMD's waves (w and w + 4) have as many keys
  // together as any other two
  const int qt = wid < 4 ? wid : 11 - wid;
  const bool live = qt < tiles;
  __attribute__((aligned(16))) KT q[EL];
  if constexpr (TURN) {
    // q is turned in LDS, where k lies afterwards
    stage_rows<T, KT, DK, DK + kPadK>(k_s, proj, a.stride, q_col, t0, nt, rows);
    __syncthreads();
    if (a.rot_dim > 0) {
      turn_rows<DK>(k_s, a.positions, a.inv_freq, t0, nt, a.rot_dim >> 1);
      __syncthreads();
    }
  }
  {
    const int t = min(qt * 16 + i, nt - 1);
#pragma unroll
    for (int gh = 0; gh < 2; ++gh) {
      const int row = (g + 4 * gh) * RPL;
#pragma unroll
      for (int r = 0; r < RPL; r += 16 / (int)sizeof(KT)) {
        const KT* src;
        if constexpr (TURN) src = k_s + t * (DK + kPadK) + row + r;
        else src = proj + (size_t)(t0 + t) * a.stride + q_col + row + r;
        *reinterpret_cast<uint4*>(&q[gh * RPL + r]) = *reinterpret_cast<const uint4*>(src);
      }
    }
  }
  if constexpr (TURN) __syncthreads();
  stage_rows<T, KT, DK, DK + kPadK>(k_s, proj, a.stride, k_col, t0, nt, rows);
  const bool odd_v = __any(stage_rows<T, T, DV, DV + kPadV>(v_s, proj, a.stride, a.v_off + h * DV, t0, nt, rows));
  if (lane == 0) w.odd[wid] = odd_v;
  if (wid == kChunkWaves - 1) segment_weights<MODE, false>(w, a, h, t0, nt, MODE == WALK_EXP_GATES ? from[NOFF + DK] : 0.f, lane);

  // the part of the start state, S_0^T q (its weight comes afterwards: nothing here waits for the staged rows)
  f32x4 acc[NCT];
  float den = 0.f;
#pragma unroll
  for (int ct = 0; ct < NCT; ++ct) acc[ct] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (live) {
    const float* src = from + (size_t)(i >> 3) * slice + 8 * g + (i & 7);
    float s[2][4][NCT];                              // four rows' columns asked for ahead of the four that are multiplied
    auto ask = [&](int b) {                          // four neighbouring rows of every row group
      const int gh = b / (RPL / 4), r = b % (RPL / 4) * 4;
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) s[b & 1][u][ct] = src[(size_t)(2 * ct) * slice + (r + u) * 64 + 32 * gh];
    };
    ask(0);
#pragma unroll
    for (int b = 0; b < RPL / 2; ++b) {
      if (b + 1 < RPL / 2) ask(b + 1);
      const int gh = b / (RPL / 4), r = b % (RPL / 4) * 4;
      float4 n0 = make_float4(0.f, 0.f, 0.f, 0.f);
      if (MODE == WALK_EXP_GATES) n0 = *reinterpret_cast<const float4*>(from + NOFF + ((r >> 2) * 8 + g + 4 * gh) * 4);
      const float n4[4] = {n0.x, n0.y, n0.z, n0.w};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float qv = to_f32<KT>(q[gh * RPL + r + u]);
        if (MODE == WALK_EXP_GATES) den = fmaf(n4[u], qv, den);
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) acc[ct] = mfma_f32(s[b & 1][u][ct], qv, acc[ct]);
      }
    }
  }
  __syncthreads();
  if constexpr (TURN) {
    if (a.rot_dim > 0) {
      turn_rows<DK>(k_s, a.positions, a.inv_freq, t0, nt, a.rot_dim >> 1);
      __syncthreads();
    }
  }

  const int t = qt * 16 + i;
  if (live) {
    const float inter = w.inter[t] * a.q_scale, rh = w.rh[t], rl = w.rl[t];
    den *= inter;
#pragma unroll
    for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[ct][v] *= inter;
    // the segment's own keys, 16 at a time
    const auto keys = [&](int kb, auto apart) {
      f32x4 sc = f32x4{0.f, 0.f, 0.f, 0.f};
      const KT* krow = k_s + (kb * 16 + i) * (DK + kPadK);
      if constexpr (HALF) {
#pragma unroll
        for (int st = 0; st < EL / 8; ++st) {
          const int gh = st * 8 / RPL, r = st * 8 % RPL;
          const bf16x8 kf = *reinterpret_cast<const bf16x8*>(krow + (g + 4 * gh) * RPL + r);
          sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, *reinterpret_cast<const bf16x8*>(&q[st * 8]), sc, 0, 0, 0);
        }
      } else {
        f32x4 sums[4] = {sc, sc, sc, sc};              // four chains: half the rounding of one
#pragma unroll
        for (int st = 0; st < EL / 4; ++st) {
          const int gh = st * 4 / RPL, r = st * 4 % RPL;
          const float4 kf = *reinterpret_cast<const float4*>(krow + (g + 4 * gh) * RPL + r);
          const float kv[4] = {kf.x, kf.y, kf.z, kf.w};
#pragma unroll
          for (int j = 0; j < 4; ++j) sums[j] = mfma_f32(kv[j], q[st * 4 + j], sums[j]);
        }
        sc = (sums[0] + sums[1]) + (sums[2] + sums[3]);
      }
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int s = kb * 16 + 4 * g + v;
        const float p = s <= t ? sc[v] * a.q_scale * (expf((w.uh[s] - rh) + (w.ul[s] - rl)) * w.b[s]) : 0.f;
        if (MODE == WALK_EXP_GATES) den += p;
        if constexpr (decltype(apart)::value) {
          for (int kg = 0; kg < 4; ++kg) {
            const float ps = __shfl(p, i + 16 * kg, kWave);
            const T* row = v_s + (kb * 16 + 4 * kg + v) * (DV + kPadV) + 4 * g;
            const bool sees = kb * 16 + 4 * kg + v <= t;
#pragma unroll
            for (int ct = 0; ct < NCT; ++ct)
#pragma unroll
              for (int y = 0; y < 4; ++y) {
                const float x = to_f32<T>(row[ct * 16 + y]);
                if (sees && !(fabsf(x) < INFINITY)) acc[ct][y] = fmaf(ps, x, acc[ct][y]);
              }
          }
        }
#pragma unroll
        for (int ct = 0; ct < NCT; ++ct) {
          float x = to_f32<T>(v_s[s * (DV + kPadV) + ct * 16 + i]);
          if constexpr (decltype(apart)::value) x = fabsf(x) < INFINITY ? x : 0.f;
          acc[ct] = mfma_f32(x, p, acc[ct]);
        }
      }
    };
    // Among the queries' own 16 tokens a later one's weight is 0, and 0 times a value that is no number is none: where the
    // segment holds such values, they are taken out of that product and added to the queries that see them.
    int odd = 0;
#pragma unroll
    for (int x = 0; x < kChunkWaves; ++x) odd |= w.odd[x];
    const int plain = __builtin_amdgcn_readfirstlane(odd ? qt - 1 : qt);
    for (int kb = 0; kb <= plain; ++kb) keys(kb, std::false_type{});
    if (plain < qt) keys(qt, std::true_type{});
    float inv = 1.f;
    if (MODE == WALK_EXP_GATES) {
      den = reduce16(den, SumOf{});
      den = reduce32(den, SumOf{});
      inv = fmaxf(fabsf(den), w.e[t]) + kWalkFloor;
    }
    if (t < nt) {
      float* orow = a.out + (size_t)(t0 + t) * a.nh * DV + (size_t)h * DV + 4 * g;
      const float skip = MODE == WALK_STATE_SPACE ? a.p2[h] : 0.f;
#pragma unroll
      for (int ct = 0; ct < NCT; ++ct) {
        float y[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          y[v] = acc[ct][v];
          if (MODE == WALK_EXP_GATES) y[v] = y[v] / inv;
          if (MODE == WALK_STATE_SPACE) y[v] = fmaf(skip, to_f32<T>(v_s[t * (DV + kPadV) + ct * 16 + 4 * g + v]), y[v]);
        }
        *reinterpret_cast<float4*>(orow + ct * 16) = make_float4(y[0], y[1], y[2], y[3]);
      }
    }
  }
  if (!last) return;
  __syncthreads();                                   // (the slot may be what the other waves still read)
  segment_state<T, KT, DK, NCT, MODE>(w, k_s, v_s, rows, from, slot);
}

template <typename T, int DK, int NCT, int MODE>
__global__ __launch_bounds__(kChunkThreads) void state_chunk_final_kernel(const WalkArgs a) { state_chunk_final_block<T, DK, NCT, MODE>(a); }

// A fixed decay's keys are floats in LDS, so one block fits a unit; its registers may be those of two waves a SIMD (104 -> 71 us
// for 2,048 tokens of 16 heads of 128 x 128; the others, two blocks a unit, lose by it: 87 -> 124 us for 64 state-space heads).
template <typename T, int DK, int NCT>
__global__ __launch_bounds__(kChunkThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void state_chunk_final_turned_kernel(const WalkArgs a) {
  state_chunk_final_block<T, DK, NCT, WALK_FIXED_DECAY>(a);
}

// 1 where long entries of heads of dk key and dv value channels take the chunk form
SHARPI_EXPORT int sharpi_state_chunk_takes(int dk, int dv) { return (dk == 64 || dk == 128) && (dv == 64 || dv == 128); }

SHARPI_EXPORT int sharpi_state_chunk_from() { return kChunkFrom; }
SHARPI_EXPORT int sharpi_state_segment_tokens() { return kSeg; }

bool state_chunk_takes(const WalkArgs& a, int dtype) {
  const int V = dtype == DT_BF16 ? 8 : 4;            // 16-byte loads of every head's rows, 16-byte stores of the outputs
  return sharpi_state_chunk_takes(a.dk, a.dv) && a.stride % V == 0 && a.q_off % V == 0 && a.k_off % V == 0 &&
         a.v_off % V == 0 && reinterpret_cast<uintptr_t>(a.proj) % 16 == 0 && reinterpret_cast<uintptr_t>(a.out) % 16 == 0;
}

template <typename T, int DK, int NCT, int MODE>
static int launch_chunk(const WalkArgs& a, bool final, hipStream_t stream) {
  constexpr size_t kt = MODE == WALK_FIXED_DECAY ? sizeof(float) : sizeof(T);
  constexpr size_t lds = kSeg * (DK + kPadK) * kt + kSeg * (NCT * 16 + kPadV) * sizeof(T) + sizeof(SegWeights);
  static_assert(lds <= 160 * 1024, "a block's LDS");
  const dim3 grid(a.nh, !final ? a.n_scratch : a.n_long < 0 ? a.n_segs : a.n_long);
  void (*kern)(const WalkArgs) = state_chunk_local_kernel<T, DK, NCT, MODE>;
  if (final) {
    if constexpr (MODE == WALK_FIXED_DECAY) kern = state_chunk_final_turned_kernel<T, DK, NCT>;
    else kern = state_chunk_final_kernel<T, DK, NCT, MODE>;
  }
  if (lds > 48 * 1024) {
    const hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
  }
  kern<<<grid, kChunkThreads, lds, stream>>>(a);
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}

template <typename T, int MODE>
static int chunk_sizes(const WalkArgs& a, bool final, hipStream_t stream) {
  if (a.dk == 64) return a.dv == 64 ? launch_chunk<T, 64, 4, MODE>(a, final, stream) : launch_chunk<T, 64, 8, MODE>(a, final, stream);
  return a.dv == 64 ? launch_chunk<T, 128, 4, MODE>(a, final, stream) : launch_chunk<T, 128, 8, MODE>(a, final, stream);
}

template <typename T>
static int chunk_mode(const WalkArgs& a, int mode, bool final, hipStream_t stream) {
  if (mode == WALK_EXP_GATES) return chunk_sizes<T, WALK_EXP_GATES>(a, final, stream);
  if (mode == WALK_STATE_SPACE) return chunk_sizes<T, WALK_STATE_SPACE>(a, final, stream);
  return chunk_sizes<T, WALK_FIXED_DECAY>(a, final, stream);
}

int state_chunk_local(const WalkArgs& a, int dtype, int mode, hipStream_t stream) {
  return dtype == DT_F32 ? chunk_mode<float>(a, mode, false, stream) : chunk_mode<bf16_t>(a, mode, false, stream);
}
int state_chunk_final(const WalkArgs& a, int dtype, int mode, hipStream_t stream) {
  return dtype == DT_F32 ? chunk_mode<float>(a, mode, true, stream) : chunk_mode<bf16_t>(a, mode, true, stream);
}
