// Matrix-valued recurrent states with one scalar decay per (token, head), walked token by token.
//
// Per head a state S [dk, dv] (float) moves as S_t = a_t S_(t-1) + b_t k_t v_t^T and gives o_t = S_t^T q_t.
// Two designs of mixer share the walk; they differ in where a_t and b_t come from and in what is done
// with o_t:
//   WALK_EXP_GATES  (a matrix memory with exponential gates): from pre-activations x_i, x_f of a token's
//       head, i = cap tanh((x_i + bias_i) / cap), f = log_sigmoid(cap tanh((x_f + bias_f) / cap)), a running
//       maximum m_t = max(f + m_(t-1), i) (m starts at 0), a_t = exp(f + m_(t-1) - m_t), b_t = exp(i - m_t);
//       beside S a vector n_t = a_t n_(t-1) + b_t k_t; the output is o_t / (max(|n_t . q_t|, exp(-m_t)) + 1e-6).
//   WALK_STATE_SPACE (a selective state space): dt = softplus(x_dt + bias_dt), a_t = exp(-exp(A_log) dt),
//       b_t = dt; k and q are the state's input and output vectors, shared by the heads of a group; the
//       output is o_t + D v_t.
//   WALK_FIXED_DECAY (retention): a_t is one stored number per head and b_t one number for the layer (the
//       keys' scale); q and k are first turned by rotary positions on their leading elements (pairs (i, i +
//       r/2), angle = position x frequency, in float, on the staged floats), the output is o_t itself.
// Everything but the reading of q, k, v is float: the gates, their logarithms and exponentials, the
// running maximum, the state, the sums.
//
// Work: a block (one wave) = (entry, head, 8 value columns).  Lane (g, j) keeps RPL = DKP / 8 rows
// g RPL .. g RPL + RPL - 1 of column j in registers (DKP = dk rounded up to 32, 64, 128 or 256; rows
// beyond dk stay zero).  Tokens are staged 8 at a time into LDS (8 KB a block at 128 rows: with 16 a
// CU held ten waves and the walk took 1.4 times as long; with 4 the gates' arithmetic, done once a
// stage, weighs more): q and k as floats in the order the
// lanes read them, the stage's gates computed side by side (the running maximum by a scan over
// the lanes whose order is fixed by the chunk), then the wave walks the stage's tokens.  A request's
// state lies slice by slice, [heads, ceil(dv / 8), slice], a slice = RPL x 64 floats of S in the
// lanes' order (row g RPL + r of column j at r 64 + 8 g + j), and, for the exponential gates, DKP
// floats of n and the maximum m (each slice its own copy: the blocks of a head do not wait for
// each other).
//
// A long entry alone in its step would leave most of the chip idle.  Since a_t is one number per head,
// a stretch of tokens acts on the state as S -> D S + L with D the product of its decays and L what
// the stretch makes of a zero state, so the entry is cut into segments that are walked side by side:
// WALK_LOCAL walks every segment but an entry's last from nothing (for the exponential gates the
// maximum starts at minus infinity: the first token then enters with weight 1) and keeps L, its
// maximum and the summed logarithms of the decays; a short kernel turns these into the segments' true
// start states one after the other (for the gates, with m' = max(F + m, m_L):
// S' = exp(F + m - m') S + exp(m_L - m') L); WALK_FINAL walks every segment from its start state,
// writes the outputs, and the entry's last segment leaves the new state in the slot.
#include "norm_gate.h"
#include "state_walk.h"

enum : int { WALK_WHOLE = 0, WALK_LOCAL = 1, WALK_FINAL = 2 };
constexpr int kWalkChunk = 8;      // tokens staged at a time

SHARPI_EXPORT int sharpi_state_walk_cols() { return kWalkCols; }

SHARPI_EXPORT int sharpi_state_walk_slice_floats(int dk, int mode) {
  const int dkp = dk <= 32 ? 32 : dk <= 64 ? 64 : dk <= 128 ? 128 : 256;
  return walk_slice_floats(dkp, mode);
}

// 16 bytes of a row as floats
__device__ __forceinline__ void load16(const float* p, float* v) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}
__device__ __forceinline__ void load16(const bf16_t* p, float* v) { load8(p, v); }

// where row `row` (= g RPL + r) of a staged q or k vector lies in LDS: four rows of a lane together,
// the eight row groups side by side (a lane reads float4s, the wave 32 consecutive words)
template <int RPL>
__device__ __forceinline__ int staged_at(int row) {
  const int g = row / RPL, r = row % RPL;
  return ((r >> 2) * 8 + g) * 4 + (r & 3);
}

template <typename T, int RPL, int MODE, int PHASE>
__global__ __launch_bounds__(kWave) void state_walk_kernel(
    const T* __restrict__ proj, int stride, int q_off, int k_off, int v_off, int heads_per_group,
    const float* __restrict__ gates, int gate_stride, const float* __restrict__ p0, const float* __restrict__ p1,
    const float* __restrict__ p2, float cap, float q_scale, float* __restrict__ state,
    const int* __restrict__ state_slots, const int* __restrict__ cu_tokens, float* __restrict__ out, int nh, int dk,
    int dv, int ncb, int vec, const int* __restrict__ segs, float* __restrict__ seg_local,
    const float* __restrict__ seg_start, float* __restrict__ seg_decay, const int* __restrict__ positions,
    const float* __restrict__ inv_freq, int rot_dim, float k_scale, int below, int n_scratch) {
  constexpr int DKP = RPL * 8;
  constexpr int V = 16 / (int)sizeof(T);            // elements of a 16-byte load
  __shared__ __attribute__((aligned(16))) float q_s[PHASE == WALK_LOCAL ? 1 : kWalkChunk][DKP];     // (no outputs, no queries)
  __shared__ __attribute__((aligned(16))) float k_s[kWalkChunk][DKP];
  __shared__ float v_s[kWalkChunk][kWalkCols];
  __shared__ float a_s[kWalkChunk], b_s[kWalkChunk], e_s[kWalkChunk];
  const int cb = blockIdx.x, h = blockIdx.y;
  const int lane = threadIdx.x, g = lane >> 3, j = lane & 7;
  const int slice = walk_slice_floats(DKP, MODE);
  int e, t_first, t_end;
  bool last = true;
  if (PHASE == WALK_WHOLE) {
    e = blockIdx.z;
    t_first = cu_tokens[e];
    t_end = cu_tokens[e + 1];
    if (t_end - t_first >= below) return;           // (the chunk form has the others)
  } else {
    const int* sg = segs + 4 * blockIdx.z;
    e = sg[0];
    t_first = sg[1];
    t_end = t_first + sg[2];
    last = sg[3] != 0;
    if (PHASE == WALK_LOCAL && last) return;        // nobody starts from what an entry's last segment makes
  }
  if (t_end <= t_first) return;
  const size_t seg_at = (((size_t)blockIdx.z * nh + h) * ncb + cb) * slice;
  float* st = state + (((size_t)state_slots[e] * nh + h) * ncb + cb) * slice;      // the request's slot
  const bool from_slot = PHASE != WALK_FINAL || (last && t_first == cu_tokens[e]);     // (an entry's only segment)
  if (!from_slot && (int)blockIdx.z >= n_scratch) return;
  const float* from = from_slot ? st : seg_start + seg_at;
  const int c = cb * kWalkCols + j;
  const int qk_head = h / heads_per_group;

  float S[RPL], n[RPL];
  float m_run = 0.f, log_decay = 0.f;
  if (PHASE == WALK_LOCAL) {
#pragma unroll
    for (int r = 0; r < RPL; ++r) S[r] = 0.f, n[r] = 0.f;
    m_run = -INFINITY;
  } else {
#pragma unroll
    for (int r = 0; r < RPL; ++r) S[r] = from[r * 64 + lane];
    if (MODE == WALK_EXP_GATES) {
      const float4* nsrc = reinterpret_cast<const float4*>(from + RPL * 64);
#pragma unroll
      for (int r4 = 0; r4 < RPL / 4; ++r4) {
        const float4 x = nsrc[r4 * 8 + g];
        n[r4 * 4] = x.x; n[r4 * 4 + 1] = x.y; n[r4 * 4 + 2] = x.z; n[r4 * 4 + 3] = x.w;
      }
      m_run = from[RPL * 64 + DKP];
    }
  }
  float par0 = 0.f, par1 = 0.f, par2 = 0.f;     // the head's constants
  if (MODE == WALK_EXP_GATES) {
    par0 = p0[h];
    par1 = p1[h];
  } else if (MODE == WALK_FIXED_DECAY) {
    par0 = p0[h];                 // the head's decay
    par1 = logf(par0);
  } else {
    par0 = p0[h];                 // dt bias
    par1 = -expf(p1[h]);          // -exp(A_log)
    par2 = p2[h];                 // D
  }

  for (int t0 = t_first; t0 < t_end; t0 += kWalkChunk) {
    const int nt = min(kWalkChunk, t_end - t0);
    __syncthreads();
    // stage q and k (floats, the lanes' order), v, and the tokens' gates
    if (vec) {                                       // 16-byte loads: every head's q and k begin on a 16-byte border
      constexpr int VPR = DKP / V;                   // loads of a row
      for (int idx = lane; idx < kWalkChunk * VPR; idx += kWave) {
        const int tt = idx / VPR, row0 = (idx % VPR) * V;
        float qv[V], kv[V];
#pragma unroll
        for (int i = 0; i < V; ++i) qv[i] = 0.f, kv[i] = 0.f;
        if (tt < nt && row0 < dk) {
          const T* base = proj + (size_t)(t0 + tt) * stride + (size_t)qk_head * dk + row0;
          load16(base + q_off, qv);
          load16(base + k_off, kv);
        }
#pragma unroll
        for (int i = 0; i < V; i += 4) {             // four rows of a lane lie together
          const int at = staged_at<RPL>(row0 + i);
          if (PHASE != WALK_LOCAL) *reinterpret_cast<float4*>(&q_s[tt][at]) = make_float4(qv[i] * q_scale, qv[i + 1] * q_scale, qv[i + 2] * q_scale, qv[i + 3] * q_scale);
          *reinterpret_cast<float4*>(&k_s[tt][at]) = make_float4(kv[i], kv[i + 1], kv[i + 2], kv[i + 3]);
        }
      }
    } else
    for (int idx = lane; idx < kWalkChunk * DKP; idx += kWave) {
      const int tt = idx / DKP, row = idx % DKP;
      float qv = 0.f, kv = 0.f;
      if (tt < nt && row < dk) {
        const T* base = proj + (size_t)(t0 + tt) * stride + (size_t)qk_head * dk + row;
        qv = to_f32<T>(base[q_off]) * q_scale;
        kv = to_f32<T>(base[k_off]);
      }
      const int at = staged_at<RPL>(row);
      if (PHASE != WALK_LOCAL) q_s[tt][at] = qv;
      k_s[tt][at] = kv;
    }
    for (int idx = lane; idx < kWalkChunk * kWalkCols; idx += kWave) {
      const int tt = idx / kWalkCols, jj = idx % kWalkCols;
      const int cc = cb * kWalkCols + jj;
      v_s[tt][jj] = (tt < nt && cc < dv) ? to_f32<T>(proj[(size_t)(t0 + tt) * stride + v_off + (size_t)h * dv + cc]) : 0.f;
    }
    if (MODE == WALK_FIXED_DECAY) {
      if (lane < nt) {
        a_s[lane] = par0;
        b_s[lane] = k_scale;
      }
      if (PHASE == WALK_LOCAL) log_decay += (float)nt * par1;
      if (rot_dim > 0) {
        // rotary positions on the staged floats: element i of a head with element i + rot_dim / 2
        __syncthreads();
        const int half = rot_dim >> 1;
        for (int idx = lane; idx < nt * half; idx += kWave) {
          const int tt = idx / half, i = idx % half;
          const float ang = (float)positions[t0 + tt] * inv_freq[i];
          const float cs = cosf(ang), sn = sinf(ang);
          const int at0 = staged_at<RPL>(i), at1 = staged_at<RPL>(i + half);
          const float ku = k_s[tt][at0], kv = k_s[tt][at1];
          k_s[tt][at0] = ku * cs - kv * sn;
          k_s[tt][at1] = kv * cs + ku * sn;
          if (PHASE != WALK_LOCAL) {
            const float qu = q_s[tt][at0], qv = q_s[tt][at1];
            q_s[tt][at0] = qu * cs - qv * sn;
            q_s[tt][at1] = qv * cs + qu * sn;
          }
        }
      }
    } else {
      const bool live = lane < nt;
      const float* grow = gates + (size_t)(t0 + (live ? lane : 0)) * gate_stride;
      if (MODE == WALK_EXP_GATES) {
        // (F, I) of a stretch of tokens: its summed log forget gates, and what its input gates alone would
        // make of the maximum; stretches combine as (F1 + F2, max(I1 + F2, I2)).  Lanes beyond the chunk
        // hold the neutral stretch (0, -inf).
        float F = 0.f, I = -INFINITY;
        if (live) {
          I = cap * tanhf((grow[h] + par0) / cap);
          F = log_sigmoid_f32(cap * tanhf((grow[nh + h] + par1) / cap));
        }
        const float log_i = I, log_f = F;
#pragma unroll
        for (int off = 1; off < kWalkChunk; off <<= 1) {
          const float Fp = __shfl_up(F, off, kWave), Ip = __shfl_up(I, off, kWave);
          if (lane >= off) {
            I = fmaxf(Ip + F, I);
            F = Fp + F;
          }
        }
        const float m_t = fmaxf(m_run + F, I);
        float m_before = __shfl_up(m_t, 1, kWave);
        if (lane == 0) m_before = m_run;
        if (live) {
          a_s[lane] = expf(log_f + m_before - m_t);
          b_s[lane] = expf(log_i - m_t);
          e_s[lane] = expf(-m_t);
        }
        m_run = __shfl(m_t, nt - 1, kWave);
        if (PHASE == WALK_LOCAL) log_decay += __shfl(F, nt - 1, kWave);
      } else {
        float la = 0.f;
        if (live) {
          const float dt = softplus_f32(grow[h] + par0);
          la = par1 * dt;
          a_s[lane] = expf(la);
          b_s[lane] = dt;
        }
        if (PHASE == WALK_LOCAL) {
#pragma unroll
          for (int off = 1; off < kWalkChunk; off <<= 1) la += __shfl_xor(la, off, kWave);
          log_decay += la;
        }
      }
    }
    __syncthreads();
    for (int tt = 0; tt < nt; ++tt) {
      const float a = a_s[tt], b = b_s[tt];
      const float vj = v_s[tt][j];
      const float bv = b * vj;
      float acc = 0.f, nq = 0.f;
      const float4* k4 = reinterpret_cast<const float4*>(&k_s[tt][0]);
      const float4* q4 = reinterpret_cast<const float4*>(&q_s[PHASE == WALK_LOCAL ? 0 : tt][0]);
#pragma unroll
      for (int r4 = 0; r4 < RPL / 4; ++r4) {
        const float4 kk = k4[r4 * 8 + g], qq = q4[r4 * 8 + g];
        const float kr[4] = {kk.x, kk.y, kk.z, kk.w}, qr[4] = {qq.x, qq.y, qq.z, qq.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = r4 * 4 + i;
          S[r] = fmaf(kr[i], bv, a * S[r]);
          if (PHASE != WALK_LOCAL) acc = fmaf(S[r], qr[i], acc);
          if (MODE == WALK_EXP_GATES) {
            n[r] = fmaf(kr[i], b, a * n[r]);
            if (PHASE != WALK_LOCAL) nq = fmaf(n[r], qr[i], nq);
          }
        }
      }
      if (PHASE == WALK_LOCAL) continue;
      acc += row_rotated<8>(acc);
      acc = reduce16(acc, SumOf{});
      acc = reduce32(acc, SumOf{});
      float y;
      if (MODE == WALK_EXP_GATES) {
        nq += row_rotated<8>(nq);
        nq = reduce16(nq, SumOf{});
        nq = reduce32(nq, SumOf{});
        y = acc / (fmaxf(fabsf(nq), e_s[tt]) + kWalkFloor);
      } else if (MODE == WALK_FIXED_DECAY) {
        y = acc;
      } else {
        y = fmaf(par2, vj, acc);
      }
      if (g == 0 && c < dv) out[(size_t)(t0 + tt) * nh * dv + (size_t)h * dv + c] = y;
    }
  }
  if (PHASE == WALK_FINAL && !last) return;
  if (PHASE == WALK_LOCAL) {
    st = seg_local + seg_at;
    if (cb == 0 && lane == 0) seg_decay[(size_t)blockIdx.z * nh + h] = log_decay;
  }
#pragma unroll
  for (int r = 0; r < RPL; ++r) st[r * 64 + lane] = S[r];
  if (MODE == WALK_EXP_GATES) {
    if (j == 0) {
      float4* ndst = reinterpret_cast<float4*>(st + RPL * 64);
#pragma unroll
      for (int r4 = 0; r4 < RPL / 4; ++r4) ndst[r4 * 8 + g] = make_float4(n[r4 * 4], n[r4 * 4 + 1], n[r4 * 4 + 2], n[r4 * 4 + 3]);
    }
    if (lane == 0) st[RPL * 64 + DKP] = m_run;
  }
}

// The segments' start states, one entry's after the other: start(first) = the slot's state, start(s + 1) =
// what segment s makes of start(s).  A thread owns one float of a (head, 8 value columns) slice (of S or,
// for the gates, of n) and keeps it in a register; it asks for eight segments' local values before it
// uses the first (they do not depend on the chain), then moves along them.
constexpr int kCombineThreads = 256;
constexpr int kCombineAhead = 8;

template <int MODE>
__global__ __launch_bounds__(kCombineThreads) void state_walk_combine_kernel(
    const float* __restrict__ state, const int* __restrict__ state_slots, const int* __restrict__ cu_tokens,
    const int* __restrict__ segs, const int* __restrict__ ent_segs,
    const float* __restrict__ seg_local, float* __restrict__ seg_start, const float* __restrict__ seg_decay, int nh,
    int ncb, int dkp, int n_scratch) {
  const int h = blockIdx.y, e = segs ? segs[4 * blockIdx.z] : blockIdx.z;
  if (segs && segs[4 * blockIdx.z + 1] != cu_tokens[e]) return;     // (an entry's first segment has the entry's blocks)
  const int first = ent_segs[2 * e], count = ent_segs[2 * e + 1];
  if (count <= 1 || first + count > n_scratch) return;      // nothing (one segment starts from the slot)
  const int slice = walk_slice_floats(dkp, MODE);
  const int moved = (dkp / 8) * 64 + (MODE == WALK_EXP_GATES ? dkp : 0);     // S and n; the maximum lies behind them
  const int idx = blockIdx.x * kCombineThreads + threadIdx.x;              // over the head's slices
  if (idx >= ncb * moved) return;
  const int cb = idx / moved, i = idx % moved;
  const size_t per_seg = (size_t)nh * ncb * slice;
  const size_t at = ((size_t)h * ncb + cb) * slice;
  const float* slot = state + (size_t)state_slots[e] * per_seg + at;
  float cur = slot[i];
  float m = MODE == WALK_EXP_GATES ? slot[moved] : 0.f;
  seg_start[(size_t)first * per_seg + at + i] = cur;
  if (MODE == WALK_EXP_GATES && i == 0) seg_start[(size_t)first * per_seg + at + moved] = m;
  for (int s0 = first; s0 + 1 < first + count; s0 += kCombineAhead) {
    const int n = min(kCombineAhead, first + count - 1 - s0);
    float loc[kCombineAhead], F[kCombineAhead], m_loc[kCombineAhead];
#pragma unroll
    for (int u = 0; u < kCombineAhead; ++u) {
      const int s = s0 + min(u, n - 1);                // (addresses clamped: no load behind a branch)
      loc[u] = seg_local[(size_t)s * per_seg + at + i];
      F[u] = seg_decay[(size_t)s * nh + h];
      m_loc[u] = MODE == WALK_EXP_GATES ? seg_local[(size_t)s * per_seg + at + moved] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < kCombineAhead; ++u) {
      if (u < n) {
        float wa, wb = 1.f;
        if (MODE == WALK_EXP_GATES) {
          const float m_new = fmaxf(F[u] + m, m_loc[u]);
          wa = expf(F[u] + m - m_new);
          wb = expf(m_loc[u] - m_new);
          m = m_new;
        } else {
          wa = expf(F[u]);
        }
        cur = fmaf(wa, cur, wb * loc[u]);
        const size_t to = (size_t)(s0 + u + 1) * per_seg + at;
        seg_start[to + i] = cur;
        if (MODE == WALK_EXP_GATES && i == 0) seg_start[to + moved] = m;
      }
    }
  }
}

template <typename T, int RPL, int MODE, int PHASE>
static void launch_walk_phase(const WalkArgs& a, int ncb, int vec, hipStream_t stream, int below = 0x7fffffff) {
  dim3 grid(ncb, a.nh, PHASE == WALK_WHOLE ? a.n_entries : PHASE == WALK_LOCAL ? a.n_scratch : a.n_segs);
  state_walk_kernel<T, RPL, MODE, PHASE><<<grid, kWave, 0, stream>>>(
      (const T*)a.proj, a.stride, a.q_off, a.k_off, a.v_off, a.heads_per_group, a.gates, a.gate_stride, a.p0, a.p1, a.p2,
      a.cap, a.q_scale, a.state, a.state_slots, a.cu_tokens, a.out, a.nh, a.dk, a.dv, ncb, vec, a.segs, a.seg_local,
      a.seg_start, a.seg_decay, a.positions, a.inv_freq, a.rot_dim, a.k_scale, below, a.n_scratch);
}

template <typename T, int RPL, int MODE>
static int launch_walk_rpl(const WalkArgs& a, int ncb, int vec, hipStream_t stream) {
  if (!a.segs) {
    launch_walk_phase<T, RPL, MODE, WALK_WHOLE>(a, ncb, vec, stream);
    SHARPI_CHECK_LAUNCH();
    return SHARPI_OK;
  }
  constexpr int dtype = sizeof(T) == 4 ? DT_F32 : DT_BF16;
  const bool chunks = state_chunk_takes(a, dtype);
  if (chunks && a.n_long < a.n_segs) {                        // (first: what the passes leave each other stays in the caches)
    launch_walk_phase<T, RPL, MODE, WALK_WHOLE>(a, ncb, vec, stream, kChunkFrom);
    SHARPI_CHECK_LAUNCH();
  }
  if (a.n_scratch > 0) {
    if (chunks) {
      const int rc = state_chunk_local(a, dtype, MODE, stream);
      if (rc != SHARPI_OK) return rc;
    } else {
      launch_walk_phase<T, RPL, MODE, WALK_LOCAL>(a, ncb, vec, stream);
      SHARPI_CHECK_LAUNCH();
    }
    // blocks of every entry, or of every segment that may be the first of one, whichever are fewer
    const int moved = RPL * 64 + (MODE == WALK_EXP_GATES ? RPL * 8 : 0);
    const dim3 grid(ceil_div(ncb * moved, kCombineThreads), a.nh, min(a.n_entries, a.n_scratch));
    state_walk_combine_kernel<MODE><<<grid, kCombineThreads, 0, stream>>>(
        a.state, a.state_slots, a.cu_tokens, a.n_scratch < a.n_entries ? a.segs : nullptr, a.ent_segs, a.seg_local, a.seg_start,
        a.seg_decay, a.nh, ncb, RPL * 8, a.n_scratch);
    SHARPI_CHECK_LAUNCH();
  }
  if (chunks) return a.n_long != 0 ? state_chunk_final(a, dtype, MODE, stream) : SHARPI_OK;
  launch_walk_phase<T, RPL, MODE, WALK_FINAL>(a, ncb, vec, stream);
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}

template <typename T, int MODE>
static int launch_state_walk(const WalkArgs& a, hipStream_t stream) {
  const int ncb = ceil_div(a.dv, kWalkCols);
  constexpr int V = 16 / (int)sizeof(T);
  const int vec = a.dk % V == 0 && a.stride % V == 0 && a.q_off % V == 0 && a.k_off % V == 0 &&
                  reinterpret_cast<uintptr_t>(a.proj) % 16 == 0;
  if (a.dk <= 32) return launch_walk_rpl<T, 4, MODE>(a, ncb, vec, stream);
  if (a.dk <= 64) return launch_walk_rpl<T, 8, MODE>(a, ncb, vec, stream);
  if (a.dk <= 128) return launch_walk_rpl<T, 16, MODE>(a, ncb, vec, stream);
  if (a.dk <= 256) return launch_walk_rpl<T, 32, MODE>(a, ncb, vec, stream);
  return SHARPI_ERR_ARG;
}

static int state_walk_any(const WalkArgs& a, int dtype, int mode, hipStream_t stream) {
  if (a.n_entries <= 0) return SHARPI_OK;
  if (a.nh <= 0 || a.nh > 65535 || a.n_entries > 65535 || a.dk <= 0 || a.dk > 256 || a.dv <= 0 || a.heads_per_group <= 0) return SHARPI_ERR_ARG;
  if (mode != WALK_EXP_GATES && mode != WALK_STATE_SPACE && mode != WALK_FIXED_DECAY) return SHARPI_ERR_ARG;
  if (mode == WALK_FIXED_DECAY) {
    if (!a.p0 || a.rot_dim < 0 || (a.rot_dim & 1) || a.rot_dim > a.dk || (a.rot_dim > 0 && (!a.positions || !a.inv_freq))) return SHARPI_ERR_ARG;
  } else if (!a.gates || !a.p0 || !a.p1 || (mode == WALK_STATE_SPACE && !a.p2) || (mode == WALK_EXP_GATES && !(a.cap > 0.f))) {
    return SHARPI_ERR_ARG;
  }
  if (dtype != DT_F32 && dtype != DT_BF16) return SHARPI_ERR_ARG;
  if (a.segs && (!a.ent_segs || (a.n_scratch > 0 && (!a.seg_local || !a.seg_start || !a.seg_decay)) || a.n_segs < a.n_entries || a.n_segs > 65535 || a.n_scratch < 0 || a.n_scratch > a.n_segs || a.n_long > a.n_segs ||
                 (a.n_long >= 0 && a.n_long < a.n_scratch))) return SHARPI_ERR_ARG;
  if (mode == WALK_EXP_GATES) {
    if (dtype == DT_F32) return launch_state_walk<float, WALK_EXP_GATES>(a, stream);
    return launch_state_walk<bf16_t, WALK_EXP_GATES>(a, stream);
  }
  if (mode == WALK_FIXED_DECAY) {
    if (dtype == DT_F32) return launch_state_walk<float, WALK_FIXED_DECAY>(a, stream);
    return launch_state_walk<bf16_t, WALK_FIXED_DECAY>(a, stream);
  }
  if (dtype == DT_F32) return launch_state_walk<float, WALK_STATE_SPACE>(a, stream);
  return launch_state_walk<bf16_t, WALK_STATE_SPACE>(a, stream);
}

// proj [T, stride] (dtype): q and k of head h at columns q_off / k_off + (h / heads_per_group) dk, v at
// v_off + h dv.  gates float [T, gate_stride]: WALK_EXP_GATES reads columns h (input gate) and nh + h
// (forget gate), p0 / p1 their biases [nh], cap the gates' cap; WALK_STATE_SPACE reads column h (the
// step size before its softplus), p0 its bias, p1 A_log, p2 D (all [nh]); WALK_FIXED_DECAY reads no gates:
// p0 the heads' decays [nh], k_scale the keys' scale, and positions int [T], inv_freq float [rot_dim / 2]
// turn the leading rot_dim elements of q and k (rot_dim 0: no rotation).  state float [slots, nh,
// ceil(dv / 8), slice]; out float [T, nh dv].
SHARPI_EXPORT int sharpi_state_walk(const void* proj, int dtype, int stride, int q_off, int k_off, int v_off,
                                    int heads_per_group, const float* gates, int gate_stride, const float* p0,
                                    const float* p1, const float* p2, float cap, float q_scale, int mode, float* state,
                                    const int* state_slots, const int* cu_tokens, float* out, int n_entries, int nh,
                                    int dk, int dv, const int* positions, const float* inv_freq, int rot_dim, float k_scale,
                                    hipStream_t stream) {
  const WalkArgs a{proj, stride, q_off, k_off, v_off, heads_per_group, gates, gate_stride, p0, p1, p2, cap, q_scale, state,
                   state_slots, cu_tokens, out, n_entries, nh, dk, dv, nullptr, nullptr, 0, 0, 0, nullptr, nullptr, nullptr,
                   positions, inv_freq, rot_dim, k_scale};
  return state_walk_any(a, dtype, mode, stream);
}

// The same walk with long entries cut into segments that are walked side by side (results equal to
// rounding).  segs int [n_segs, 4] = (entry, first row, tokens, 1 if the entry's last), an entry's one after the
// other, those of entries with several first, then those of at least kChunkFrom tokens (n_long up to there; -1: not known); ent_segs int
// [n_entries, 2] = (first segment, segments).  An entry's only segment starts from its slot and leaves into it; the first
// n_scratch segments, which hold all others, have their place in seg_local and seg_start float [n_scratch, nh,
// ceil(dv / 8), slice] and seg_decay float [n_scratch, nh].
SHARPI_EXPORT int sharpi_state_walk_segmented(const void* proj, int dtype, int stride, int q_off, int k_off, int v_off,
                                              int heads_per_group, const float* gates, int gate_stride, const float* p0,
                                              const float* p1, const float* p2, float cap, float q_scale, int mode,
                                              float* state, const int* state_slots, const int* cu_tokens, float* out,
                                              int n_entries, int nh, int dk, int dv, const int* segs, const int* ent_segs,
                                              int n_segs, int n_scratch, int n_long, float* seg_local, float* seg_start, float* seg_decay,
                                              const int* positions, const float* inv_freq, int rot_dim, float k_scale,
                                              hipStream_t stream) {
  if (!segs) return SHARPI_ERR_ARG;
  const WalkArgs a{proj, stride, q_off, k_off, v_off, heads_per_group, gates, gate_stride, p0, p1, p2, cap, q_scale, state,
                   state_slots, cu_tokens, out, n_entries, nh, dk, dv, segs, ent_segs, n_segs, n_scratch, n_long, seg_local, seg_start, seg_decay,
                   positions, inv_freq, rot_dim, k_scale};
  return state_walk_any(a, dtype, mode, stream);
}

// ---------------------------------------------------------------------------
// Behind a walk: o float [T, G * gd] in G equal parts, each divided by its root mean square, times a
// weight per channel, times a gate act(z) read from columns g_off.. of proj [T, stride] (act: 0 none,
// 1 SiLU, 2 sigmoid).  gate_first: the gate multiplies o BEFORE the statistics are taken (the norm
// then sees the gated values); otherwise after the weight.  A wave a (token, part), where norm_gate.h does not take the parts' width.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void group_norm_gate_kernel(const float* __restrict__ o, const float* __restrict__ w,
                                                               float eps, const T* __restrict__ proj, int stride,
                                                               int g_off, int act, int gate_first, T* __restrict__ out,
                                                               int n_tokens, int G, int gd) {
  const int pair = blockIdx.x * 4 + (threadIdx.x >> 6);     // (token, part), parts fastest
  const int lane = threadIdx.x & (kWave - 1);
  if (pair >= n_tokens * G) return;
  const int t = pair / G, p = pair % G;
  const float* x = o + (size_t)pair * gd;
  const T* gate = act ? proj + (size_t)t * stride + g_off + (size_t)p * gd : nullptr;
  float ss = 0.f;
  for (int d = lane; d < gd; d += kWave) {
    float v = x[d];
    if (gate && gate_first) v *= part_gate(act, to_f32<T>(gate[d]));
    ss = fmaf(v, v, ss);
  }
  ss = wave_sum(ss);
  const float inv = rsqrtf(ss / (float)gd + eps);
  for (int d = lane; d < gd; d += kWave) {
    float v = x[d];
    if (gate && gate_first) v *= part_gate(act, to_f32<T>(gate[d]));
    float y = w ? v * inv * w[(size_t)p * gd + d] : v * inv;      // (w null: a norm without a weight)
    if (gate && !gate_first) y *= part_gate(act, to_f32<T>(gate[d]));
    out[(size_t)pair * gd + d] = from_f32<T>(y);
  }
}

SHARPI_EXPORT int sharpi_group_norm_gate(const float* o, const float* w, float eps, const void* proj, int dtype,
                                         int stride, int g_off, int act, int gate_first, void* out, int n_tokens, int G,
                                         int gd, hipStream_t stream) {
  if (n_tokens <= 0) return SHARPI_OK;
  if (G <= 0 || gd <= 0 || act < 0 || act > 2 || (act && !proj)) return SHARPI_ERR_ARG;
  const PartNorm parts{o, w, gd, eps, proj, stride, g_off, act, gate_first, out, n_tokens * G, G, gd};
  if ((dtype == DT_F32 || dtype == DT_BF16) && part_norm_wide(parts)) {
    if (dtype == DT_F32) part_norm_launch<float>(parts, stream);
    else part_norm_launch<bf16_t>(parts, stream);
    SHARPI_CHECK_LAUNCH();
    return SHARPI_OK;
  }
  const int blocks = ceil_div(n_tokens * G, 4);
  if (dtype == DT_F32)
    group_norm_gate_kernel<float><<<blocks, 256, 0, stream>>>(o, w, eps, (const float*)proj, stride, g_off, act, gate_first,
                                                               (float*)out, n_tokens, G, gd);
  else if (dtype == DT_BF16)
    group_norm_gate_kernel<bf16_t><<<blocks, 256, 0, stream>>>(o, w, eps, (const bf16_t*)proj, stride, g_off, act,
                                                                gate_first, (bf16_t*)out, n_tokens, G, gd);
  else
    return SHARPI_ERR_ARG;
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}

// ---------------------------------------------------------------------------
// A short causal convolution over time on C channels of proj [T, stride] (columns c_off..), with a
// bias, then SiLU: y_t = silu(b + sum_j w[:, j] u_(t - taps + 1 + j)) (w float [C, taps]; the last
// column is the current token's).  Before an entry's first row of the step the inputs come from the
// request's tail, float [slots, taps - 1, C] (its last taps - 1 inputs, oldest first; zeros for a new
// request).  A second kernel moves the tails on.  Sums in float, the current token's term last.
// ---------------------------------------------------------------------------
constexpr int kConvMaxTaps = 8;

template <typename T>
__global__ __launch_bounds__(256) void short_conv_kernel(const T* __restrict__ proj, int stride, int c_off,
                                                          const float* __restrict__ w, const float* __restrict__ bias,
                                                          int taps, const float* __restrict__ tail,
                                                          const int* __restrict__ state_slots,
                                                          const int* __restrict__ entry_of_token,
                                                          const int* __restrict__ cu_tokens, T* __restrict__ out, int C) {
  const int t = blockIdx.x;
  const int ch = blockIdx.y * blockDim.x + threadIdx.x;
  if (ch >= C) return;
  const int e = entry_of_token[t];
  const int local = t - cu_tokens[e];
  const float* tl = tail ? tail + (size_t)state_slots[e] * (taps - 1) * C : nullptr;
  float acc = bias ? bias[ch] : 0.f;
  for (int jx = 0; jx < taps; ++jx) {
    const int back = taps - 1 - jx;           // how many tokens before this one
    float u;
    if (back <= local) u = to_f32<T>(proj[(size_t)(t - back) * stride + c_off + ch]);
    else u = tl[(size_t)(taps - 1 + local - back) * C + ch];
    acc = fmaf(w[(size_t)ch * taps + jx], u, acc);
  }
  out[(size_t)t * C + ch] = from_f32<T>(acc / (1.0f + expf(-acc)));
}

// Four taps, channels by eights: a thread takes eight channels of S consecutive tokens, so that their weights (128 bytes) and the rows
// that several of them read are read once (one channel and tap at a time: 1,950 tokens of 6,144 channels 75.4 -> 21.4 us).  A block's
// threads are 2^log_cols runs of channels by as many groups of tokens as that leaves room for.
constexpr int kConvThreads = 256;
template <typename T, int S>
__global__ __launch_bounds__(kConvThreads) void short_conv4_kernel(const T* __restrict__ proj, int stride, int c_off, const float* __restrict__ w,
                                                           const float* __restrict__ bias, const float* __restrict__ tail,
                                                           const int* __restrict__ state_slots, const int* __restrict__ entry_of_token,
                                                           const int* __restrict__ cu_tokens, T* __restrict__ out, int n_tokens, int C, int log_cols) {
  const int run = threadIdx.x & ((1 << log_cols) - 1), group = threadIdx.x >> log_cols;
  const int t0 = (blockIdx.x * (kConvThreads >> log_cols) + group) * S, ch = ((blockIdx.y << log_cols) + run) * 8;
  if (ch >= C || t0 >= n_tokens) return;
  const T* src = proj + c_off + ch;
  int e[S], local[S];
#pragma unroll
  for (int i = 0; i < S; ++i) e[i] = entry_of_token[min(t0 + i, n_tokens - 1)];
  Run8<T> row[S + 3];                              // rows t0 - 3 ..
#pragma unroll
  for (int i = 0; i < S + 3; ++i) row[i].load(src + (size_t)min(max(t0 - 3 + i, 0), n_tokens - 1) * stride);
  float4 wv[8];
  float b8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 8; ++j) wv[j] = *reinterpret_cast<const float4*>(w + (size_t)(ch + j) * 4);
  if (bias) load8(bias + ch, b8);
#pragma unroll
  for (int i = 0; i < S; ++i) local[i] = t0 + i - cu_tokens[e[i]];
#pragma unroll
  for (int i = 0; i < S; ++i) {
    const int t = t0 + i;
    if (t >= n_tokens) break;
    float held[3][8];                              // (an entry's first three tokens: what its tail holds of the rows before, requested together)
    if (local[i] < 3) {
      const float* tl = tail + ((size_t)state_slots[e[i]] * 3 + local[i]) * C + ch;
#pragma unroll
      for (int x = 0; x < 3; ++x)
        if (3 - x > local[i]) load8(tl + (size_t)x * C, held[x]);
    }
    float acc[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = b8[j];
#pragma unroll
    for (int x = 0; x < 4; ++x) {                  // 3 - x tokens back
      float u[8];
      row[i + x].floats(u);
      if (x < 3 && 3 - x > local[i])
#pragma unroll
        for (int j = 0; j < 8; ++j) u[j] = held[x][j];
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] = fmaf(x == 0 ? wv[j].x : x == 1 ? wv[j].y : x == 2 ? wv[j].z : wv[j].w, u[j], acc[j]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = acc[j] / (1.0f + expf(-acc[j]));
    store8(out + (size_t)t * C + ch, acc);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void short_conv_tail_kernel(const T* __restrict__ proj, int stride, int c_off, int taps,
                                                               float* __restrict__ tail, const int* __restrict__ state_slots,
                                                               const int* __restrict__ cu_tokens, int C) {
  const int e = blockIdx.x;
  const int ch = blockIdx.y * blockDim.x + threadIdx.x;
  if (ch >= C) return;
  const int first = cu_tokens[e], L = cu_tokens[e + 1] - first;
  if (L <= 0) return;
  float* tl = tail + (size_t)state_slots[e] * (taps - 1) * C;
  float keep[kConvMaxTaps];
  for (int i = 0; i < taps - 1; ++i) {        // the new row i is the input at local index L - (taps - 1) + i
    const int li = L - (taps - 1) + i;
    keep[i] = li >= 0 ? to_f32<T>(proj[(size_t)(first + li) * stride + c_off + ch]) : tl[(size_t)(taps - 1 + li) * C + ch];
  }
  for (int i = 0; i < taps - 1; ++i) tl[(size_t)i * C + ch] = keep[i];
}

SHARPI_EXPORT int sharpi_short_conv(const void* proj, int dtype, int stride, int c_off, const float* w, const float* bias,
                                    int taps, float* tail, const int* state_slots, const int* entry_of_token,
                                    const int* cu_tokens, void* out, int n_tokens, int n_entries, int C, int update_tail,
                                    hipStream_t stream) {
  if (n_tokens <= 0) return SHARPI_OK;
  if (C <= 0 || taps < 1 || taps > kConvMaxTaps || (taps > 1 && !tail) || n_entries <= 0 || ceil_div(C, 256) > 65535) return SHARPI_ERR_ARG;
  if (dtype != DT_F32 && dtype != DT_BF16) return SHARPI_ERR_ARG;
  dim3 grid(n_tokens, ceil_div(C, 256)), tgrid(n_entries, ceil_div(C, 256));
  const auto at16 = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  // Four taps by eights where there is enough for it: a channel a lane has an eighth of a thread's exponentials and its weights' lines to itself, and a step of single
  // tokens reads three rows of floats a token whatever the form.  us, a channel a lane / two tokens a thread / four: 1 token of 6,144 channels
  // 5.0 / 6.2 / 6.3, 64 6.6 / 7.2 / 9.0, 100 8.2 / 7.3 / 9.1, 500 22 / 11.0 / 11.9, 5,000 187 / 51.7 / 50.6; 2,048 tokens of 64 5.4 / 6.3 / 8.0, of 512 9.4 / 6.7 /
  // 8.4; single tokens, 6,144 channels: 200 18.9 / 23.4 / 23.9, 300 26.9 / 25.7 / 26.5, 500 42 / 35.3 / 35.3.
  const long long many = (long long)n_tokens * C;
  const bool by_eights = many >> (n_tokens < 8LL * n_entries ? 21 : 19) != 0;
  if (by_eights && taps == 4 && C % 8 == 0 && stride % 8 == 0 && c_off % 8 == 0 && at16(proj) && at16(w) && at16(bias) && at16(tail) && at16(out)) {
    const int s = many >> 22 ? 4 : 2;
    int log_cols = 0;
    while ((1 << log_cols) < C / 8 && (1 << log_cols) < kConvThreads) ++log_cols;
    const dim3 grid8(ceil_div(n_tokens, s * (kConvThreads >> log_cols)), ceil_div(C / 8, 1 << log_cols));
#define CONV4(T, SV)                                                                                                           \
  short_conv4_kernel<T, SV><<<grid8, kConvThreads, 0, stream>>>((const T*)proj, stride, c_off, w, bias, tail, state_slots, entry_of_token, \
                                                       cu_tokens, (T*)out, n_tokens, C, log_cols)
    if (dtype == DT_F32) {
      if (s == 4) CONV4(float, 4); else CONV4(float, 2);
    } else {
      if (s == 4) CONV4(bf16_t, 4); else CONV4(bf16_t, 2);
    }
#undef CONV4
    SHARPI_CHECK_LAUNCH();
    if (update_tail) {
      if (dtype == DT_F32)
        short_conv_tail_kernel<float><<<tgrid, 256, 0, stream>>>((const float*)proj, stride, c_off, taps, tail, state_slots, cu_tokens, C);
      else
        short_conv_tail_kernel<bf16_t><<<tgrid, 256, 0, stream>>>((const bf16_t*)proj, stride, c_off, taps, tail, state_slots, cu_tokens, C);
    }
  } else if (dtype == DT_F32) {
    short_conv_kernel<float><<<grid, 256, 0, stream>>>((const float*)proj, stride, c_off, w, bias, taps, tail, state_slots,
                                                        entry_of_token, cu_tokens, (float*)out, C);
    SHARPI_CHECK_LAUNCH();
    if (taps > 1 && update_tail)
      short_conv_tail_kernel<float><<<tgrid, 256, 0, stream>>>((const float*)proj, stride, c_off, taps, tail, state_slots,
                                                                cu_tokens, C);
  } else {
    short_conv_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)proj, stride, c_off, w, bias, taps, tail,
                                                         state_slots, entry_of_token, cu_tokens, (bf16_t*)out, C);
    SHARPI_CHECK_LAUNCH();
    if (taps > 1 && update_tail)
      short_conv_tail_kernel<bf16_t><<<tgrid, 256, 0, stream>>>((const bf16_t*)proj, stride, c_off, taps, tail, state_slots,
                                                                 cu_tokens, C);
  }
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}
