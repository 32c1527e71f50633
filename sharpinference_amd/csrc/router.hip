// MoE routing on the device: router logits, gate, top-k, and the expert-sorted row list.
//
// router_topk: one block per token, or per two or four tokens when there are many.
// logits[e] = Wr[e, :] . x[t, :] in float (a wave takes two or four neighbouring experts at a time, or one, and goes on behind
// those of the block's other waves; lanes stride over the hidden width, so the order of the additions depends on the width only).
// gate 0 = sigmoid over every expert, gate 1 = softmax over every expert.  The k picks scan
// ascending with a strict >, so the lowest index wins a tie; the weight of a pick is its gate
// value; renorm divides the k weights by their sum.
//
// moe_permute: one block. Counts rows per expert, prefix-sums them into offsets[E + 1] and
// writes, in expert order, the token and weight of every (token, pick) pair plus the inverse
// map inv_pos[t * k + j] = row in that order, and the plan that the grouped product of many rows
// walks (grouped_plan.h: units of sibling row tiles dealt to the XCDs).  With shared_group the list gets one
// more group after the experts: every token once, weight 1 (an always-on expert that shares the
// experts' weight tensor); offsets then has n_experts + 2 entries and the row arrays n_tokens more.
// Picks of n_experts and above (identity experts: the token's own row is their output) get no row: the list
// then ends at offsets[n_experts], before its room does.  The two do not come together.
#include "common.h"
#include "grouped_plan.h"

constexpr int kMaxExperts = 1024;

// One thread: gate the logits g[0 .. n_experts) in place, pick k of them (ascending scan with a
// strict >, so the lowest index wins a tie) into ids / w.
// `choice` (or null) is scratch of n_experts + n_groups floats and turns the choice apart from the
// weights: experts are then picked by g[e] + corr[e] (corr may be null), among the experts of the
// `keep` best of n_groups equal groups of neighbours only (a group's rank: the sum of its
// group_top largest choice scores; the lowest index wins a tie; the others' choice scores count as
// minus infinity), and a pick's weight stays its gate value g[e].
constexpr int kMaxGroupTop = 2;

__device__ void gate_and_pick(float* g, int n_experts, int k, int gate, int renorm, int* ids, float* w,
                              float* gate_out, float* choice = nullptr, const float* corr = nullptr,
                              int n_groups = 1, int keep = 1, int group_top = kMaxGroupTop) {
  if (gate == 2) {
    // the logits themselves rank the experts; the picks' weights are the softmax over the picked logits alone
  } else if (gate == 0) {
    for (int e = 0; e < n_experts; ++e) g[e] = 1.0f / (1.0f + expf(-g[e]));
  } else {
    float mx = g[0];
    for (int e = 1; e < n_experts; ++e) mx = fmaxf(mx, g[e]);
    float sum = 0.f;
    for (int e = 0; e < n_experts; ++e) {
      g[e] = expf(g[e] - mx);
      sum += g[e];
    }
    const float inv = 1.0f / sum;
    for (int e = 0; e < n_experts; ++e) g[e] *= inv;
  }
  if (gate_out)
    for (int e = 0; e < n_experts; ++e) gate_out[e] = g[e];
  const float* by = g;               // what the picks are ranked by
  if (choice) {
    for (int e = 0; e < n_experts; ++e) choice[e] = corr ? g[e] + corr[e] : g[e];
    if (n_groups > 1 && keep < n_groups) {
      const int per = n_experts / n_groups;
      float* rank = choice + n_experts;
      for (int q = 0; q < n_groups; ++q) {
        // the sum of the group's group_top largest choice scores (of all of them in a smaller group)
        float top[kMaxGroupTop];
        for (int i = 0; i < kMaxGroupTop; ++i) top[i] = -INFINITY;
        for (int e = q * per; e < (q + 1) * per; ++e) {
          float v = choice[e];
          for (int i = 0; i < kMaxGroupTop; ++i)
            if (v > top[i]) {
              const float o = top[i];
              top[i] = v;
              v = o;
            }
        }
        float r = 0.f;
        for (int i = 0; i < group_top && i < per; ++i) r += top[i];
        rank[q] = r;
      }
      for (int j = 0; j < keep; ++j) {       // the kept groups are marked with +infinity
        int best = -1;
        float bv = -INFINITY;
        for (int q = 0; q < n_groups; ++q)
          if (rank[q] != INFINITY && (best < 0 || rank[q] > bv)) {
            bv = rank[q];
            best = q;
          }
        rank[best] = INFINITY;
      }
      for (int q = 0; q < n_groups; ++q)
        if (rank[q] != INFINITY)
          for (int e = q * per; e < (q + 1) * per; ++e) choice[e] = -INFINITY;
    }
    by = choice;
  }
  float wsum = 0.f;
  for (int j = 0; j < k; ++j) {
    int best = -1;
    float bv = -INFINITY;
    for (int e = 0; e < n_experts; ++e) {
      bool taken = false;
      for (int i = 0; i < j; ++i) taken |= (ids[i] == e);
      if (!taken && (best < 0 || by[e] > bv)) {
        bv = by[e];
        best = e;
      }
    }
    ids[j] = best;
    w[j] = g[best];
    wsum += g[best];
  }
  if (gate == 2) {
    float mx = w[0];
    for (int j = 1; j < k; ++j) mx = fmaxf(mx, w[j]);
    float sum = 0.f;
    for (int j = 0; j < k; ++j) {
      w[j] = expf(w[j] - mx);
      sum += w[j];
    }
    const float inv = 1.0f / sum;
    for (int j = 0; j < k; ++j) w[j] *= inv;
    return;
  }
  if (renorm && k > 1 && wsum > 0.f)
    for (int j = 0; j < k; ++j) w[j] /= wsum;
}

// The same by one wave, for up to 64 picks: lanes gate and rank experts lane, lane + 64, ..., a pick is a wave-wide
// maximum (the lowest index wins a tie), pick j's id and weight stay in lane j until they are written.  The
// additions over picks are in the picks' order, as one thread makes them.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// index of the largest v[i], i < n, that is not marked in the lanes' masks (bit i / 64 of lane i % 64); -1: none
__device__ __forceinline__ int wave_argmax(const float* v, int n, int lane, uint32_t taken, float* best_v) {
  int best = -1;
  float bv = -INFINITY;
  for (int i = lane, b = 0; i < n; i += kWave, ++b) {
    const float x = v[i];
    if (!(taken >> b & 1u) && (best < 0 || x > bv)) {
      bv = x;
      best = i;
    }
  }
  // the lanes that hold the largest; of several the one of the lowest index (none equal to it: only values that are no number are left)
  const float mx = wave_max(best >= 0 ? bv : -INFINITY);
  unsigned long long at = __ballot(best >= 0 && bv == mx);
  if (at == 0) at = __ballot(best >= 0);
  if (at == 0) {
    *best_v = -INFINITY;
    return -1;
  }
  if (n > kWave && (at & (at - 1)) != 0) {
    int low = (at >> lane & 1) != 0 ? best : 0x7fffffff;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) low = min(low, __shfl_xor(low, off, kWave));
    at = __ballot(best == low);
  }
  const int src = __ffsll((long long)at) - 1;
  *best_v = __shfl(bv, src, kWave);
  best = __shfl(best, src, kWave);
  return best;
}

__device__ void gate_and_pick_wave(float* g, int n_experts, int k, int gate, int renorm, int* ids, float* w, float* gate_out,
                                   float* choice, const float* corr, int n_groups, int keep, float w_scale, int lane, int group_top = kMaxGroupTop) {
  if (gate == 0) {
    for (int e = lane; e < n_experts; e += kWave) g[e] = 1.0f / (1.0f + expf(-g[e]));
  } else if (gate == 1) {
    float mx = -INFINITY, sum = 0.f;
    for (int e = lane; e < n_experts; e += kWave) mx = fmaxf(mx, g[e]);
    mx = wave_max(mx);
    for (int e = lane; e < n_experts; e += kWave) {
      g[e] = expf(g[e] - mx);
      sum += g[e];
    }
    const float inv = 1.0f / wave_sum(sum);
    for (int e = lane; e < n_experts; e += kWave) g[e] *= inv;
  }
  if (gate_out)
    for (int e = lane; e < n_experts; e += kWave) gate_out[e] = g[e];
  const float* by = g;
  if (choice) {
    for (int e = lane; e < n_experts; e += kWave) choice[e] = corr ? g[e] + corr[e] : g[e];
    if (n_groups > 1 && keep < n_groups) {
      const int per = n_experts / n_groups;
      float* rank = choice + n_experts;
      wave_lds_sync();
      for (int q = lane; q < n_groups; q += kWave) {
        float top[kMaxGroupTop];
        for (int i = 0; i < kMaxGroupTop; ++i) top[i] = -INFINITY;
        for (int e = q * per; e < (q + 1) * per; ++e) {
          float v = choice[e];
          for (int i = 0; i < kMaxGroupTop; ++i)
            if (v > top[i]) {
              const float o = top[i];
              top[i] = v;
              v = o;
            }
        }
        float r = 0.f;
        for (int i = 0; i < group_top && i < per; ++i) r += top[i];
        rank[q] = r;
      }
      wave_lds_sync();
      uint32_t kept = 0;                   // bit b: group lane + 64 b
      for (int j = 0; j < keep; ++j) {
        float bv;
        const int best = wave_argmax(rank, n_groups, lane, kept, &bv);
        if (best >= 0 && best % kWave == lane) kept |= 1u << (best / kWave);
      }
      for (int q = lane, b = 0; q < n_groups; q += kWave, ++b)
        if (!(kept >> b & 1u))
          for (int e = q * per; e < (q + 1) * per; ++e) choice[e] = -INFINITY;
    }
    by = choice;
  }
  wave_lds_sync();
  uint32_t taken = 0;
  int my_id = 0;
  float my_w = 0.f;
  for (int j = 0; j < k; ++j) {
    float bv;
    int best = wave_argmax(by, n_experts, lane, taken, &bv);
    if (best < 0) best = 0;                // (cannot be: k <= n_experts)
    if (best % kWave == lane) taken |= 1u << (best / kWave);
    if (lane == j) {
      my_id = best;
      my_w = g[best];
    }
  }
  if (gate == 2) {
    float mx = __shfl(my_w, 0, kWave);
    for (int j = 1; j < k; ++j) mx = fmaxf(mx, __shfl(my_w, j, kWave));
    my_w = expf(my_w - mx);
    float sum = 0.f;
    for (int j = 0; j < k; ++j) sum += __shfl(my_w, j, kWave);
    my_w *= 1.0f / sum;
  } else if (renorm && k > 1) {
    float sum = 0.f;
    for (int j = 0; j < k; ++j) sum += __shfl(my_w, j, kWave);
    if (sum > 0.f) my_w /= sum;
  }
  if (lane < k) {
    ids[lane] = my_id;
    w[lane] = w_scale != 1.0f ? my_w * w_scale : my_w;
  }
}

// One wave: s[i] = wrow . xr[i] for TT rows, in float.  Lanes stride over the width in runs of 8
// (one fused multiply-add chain per lane and row, in ascending order), then the lanes are summed:
// the order of the additions depends on the width only, and each row has its own accumulator, so
// a token's logit is the same bits whatever TT is and whichever kernel calls this.
template <typename T, typename TW, int TT>
__device__ __forceinline__ void wave_dot_rows(const T* const (&xr)[TT], const TW* __restrict__ wrow, int hidden,
                                              int lane, float (&out)[TT]) {
  float s[TT];
#pragma unroll
  for (int i = 0; i < TT; ++i) s[i] = 0.f;
  if ((hidden & 7) == 0) {
    // Q runs are fetched before the first is added: a row is a dozen dependent round trips
    // to the cache otherwise, and the kernel is nothing but their latency
    constexpr int Q = TT == 1 ? 4 : 2;
    int c = lane * 8;
    for (; c + (Q - 1) * kWave * 8 < hidden; c += Q * kWave * 8) {
      float a[TT][Q][8], b[Q][8];
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        load8(wrow + c + q * kWave * 8, b[q]);
#pragma unroll
        for (int i = 0; i < TT; ++i) load8(xr[i] + c + q * kWave * 8, a[i][q]);
      }
#pragma unroll
      for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
          for (int j = 0; j < 8; ++j) s[i] = fmaf(a[i][q][j], b[q][j], s[i]);
    }
    for (; c < hidden; c += kWave * 8) {
      float b[8];
      load8(wrow + c, b);
#pragma unroll
      for (int i = 0; i < TT; ++i) {
        float a[8];
        load8(xr[i] + c, a);
#pragma unroll
        for (int j = 0; j < 8; ++j) s[i] = fmaf(a[j], b[j], s[i]);
      }
    }
  } else {
    for (int c = lane; c < hidden; c += kWave) {
      const float b = to_f32<TW>(wrow[c]);
#pragma unroll
      for (int i = 0; i < TT; ++i) s[i] = fmaf(to_f32<T>(xr[i][c]), b, s[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < TT; ++i) out[i] = wave_sum(s[i]);
}

// One wave: the EE x TT products of EE router rows and TT token rows, bit for bit those of wave_dot_rows (the same chain
// a lane, the lanes added in the same pairs); hidden % 8 == 0.  What bounds it: a row read for one product
// costs the cache's 64 bytes a cycle more than its eight multiply-adds a lane, so a row is read for EE or TT of them,
// the next run's loads are sent before this run is added (not at 16 products, where they cost the registers that let
// the block's other waves cover them), and the lanes' sums go up the tree together: half of them by half of the lanes.  Lane v * 64 / (EE * TT) returns product v = ee * TT + i.
template <typename T, typename TW, int EE, int TT>
__device__ __forceinline__ float wave_dots(const T* const (&xr)[TT], const TW* const (&wrow)[EE], int hidden, int lane) {
  constexpr int N = EE * TT;
  float s[N];
#pragma unroll
  for (int v = 0; v < N; ++v) s[v] = 0.f;
  const auto add = [&](const Run8<TW> (&wc)[EE], const Run8<T> (&xc)[TT]) {
    float a[TT][8];
#pragma unroll
    for (int i = 0; i < TT; ++i) xc[i].floats(a[i]);
#pragma unroll
    for (int e = 0; e < EE; ++e) {
      float b[8];
      wc[e].floats(b);
#pragma unroll
      for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) s[e * TT + i] = fmaf(a[i][j], b[j], s[e * TT + i]);
    }
  };
  const auto load = [&](int c, Run8<TW> (&wc)[EE], Run8<T> (&xc)[TT]) {
#pragma unroll
    for (int e = 0; e < EE; ++e) wc[e].load(wrow[e] + c);
#pragma unroll
    for (int i = 0; i < TT; ++i) xc[i].load(xr[i] + c);
  };
  int c = lane * 8;
  if constexpr (N == 16) {
    for (; c < hidden; c += kWave * 8) {
      Run8<TW> wc[EE];
      Run8<T> xc[TT];
      load(c, wc, xc);
      add(wc, xc);
    }
  } else {
    Run8<TW> w0[EE], w1[EE];
    Run8<T> x0[TT], x1[TT];
    if (c < hidden) load(c, w0, x0);
    while (c < hidden) {
      const int c1 = c + kWave * 8, c2 = c1 + kWave * 8;
      if (c1 < hidden) load(c1, w1, x1);
      __builtin_amdgcn_sched_barrier(0);
      add(w0, x0);
      if (c1 >= hidden) break;
      if (c2 < hidden) load(c2, w0, x0);
      __builtin_amdgcn_sched_barrier(0);
      add(w1, x1);
      c = c2;
    }
  }
  int off = kWave / 2;
#pragma unroll
  for (int m = N / 2; m > 0; m >>= 1, off >>= 1) {
    const bool high = lane & off;
#pragma unroll
    for (int v = 0; v < m; ++v) {
      if (off >= 16) {                  // (a swap leaves each lane both terms of its product's sum)
        const auto p = off == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(s[v]), __float_as_uint(s[v + m]), false, false)
                                 : __builtin_amdgcn_permlane16_swap(__float_as_uint(s[v]), __float_as_uint(s[v + m]), false, false);
        s[v] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
      } else {
        const float other = __shfl_xor(high ? s[v] : s[v + m], off, kWave);
        s[v] = (high ? s[v + m] : s[v]) + other;
      }
    }
  }
  for (; off > 0; off >>= 1) s[0] += __shfl_xor(s[0], off, kWave);
  return s[0];
}

template <typename T, typename TW, int EE, int TT>
__global__ __launch_bounds__(1024) void router_topk_kernel(const T* __restrict__ x, const TW* __restrict__ wr,
                                                           int* __restrict__ topk_ids,
                                                           float* __restrict__ topk_w,
                                                           float* __restrict__ gate_out, int n_tokens, int hidden,
                                                           int n_experts, int k, int gate, int renorm,
                                                           const float* __restrict__ corr, int n_groups, int keep,
                                                           int split_choice, const float* __restrict__ bias, float w_scale, int group_top) {
  // TT tokens per block: a router row is fetched once for all of them.
  extern __shared__ float router_lds[];
  float* const g_s = router_lds;             // [TT][n_experts]: logits, then gates
  float* const choice_s = g_s + TT * n_experts;   // [TT][n_experts + n_groups] when the choice has scores of its own
  const auto g = [&](int i) { return g_s + i * n_experts; };
  const int t0 = blockIdx.x * TT;
  const int lane = threadIdx.x & (kWave - 1);
  const int w = threadIdx.x >> 6;
  const int nw = blockDim.x >> 6;
  const T* xr[TT];
#pragma unroll
  for (int i = 0; i < TT; ++i) xr[i] = x + (size_t)min(t0 + i, n_tokens - 1) * hidden;   // beyond the last: computed, not kept
  if constexpr (EE > 0) {
    constexpr int N = EE * TT, W = kWave / N;
    for (int e0 = w * EE; e0 < n_experts; e0 += nw * EE) {
      const TW* wrow[EE];
#pragma unroll
      for (int x = 0; x < EE; ++x) wrow[x] = wr + (size_t)min(e0 + x, n_experts - 1) * hidden;
      const float v = wave_dots<T, TW, EE, TT>(xr, wrow, hidden, lane);
      const int e = e0 + lane / W / TT;
      if (lane % W == 0 && e < n_experts) g(lane / W % TT)[e] = bias ? v + bias[e] : v;
    }
  } else for (int e = w; e < n_experts; e += nw) {
    float v[TT];
    wave_dot_rows<T, TW, TT>(xr, wr + (size_t)e * hidden, hidden, lane, v);
    if (lane == 0) {
#pragma unroll
      for (int i = 0; i < TT; ++i) g(i)[e] = bias ? v[i] + bias[e] : v[i];
    }
  }
  __syncthreads();
  if (k <= kWave) {                          // a wave a token
    for (int i = w; i < TT && t0 + i < n_tokens; i += nw) {
      const int t = t0 + i;
      gate_and_pick_wave(g(i), n_experts, k, gate, renorm, topk_ids + (size_t)t * k, topk_w + (size_t)t * k,
                         gate_out ? gate_out + (size_t)t * n_experts : nullptr,
                         split_choice ? choice_s + (size_t)i * (n_experts + n_groups) : nullptr, corr, n_groups, keep, w_scale, lane, group_top);
    }
  } else if (threadIdx.x < TT && t0 + threadIdx.x < n_tokens) {
    const int t = t0 + threadIdx.x;
    gate_and_pick(g(threadIdx.x), n_experts, k, gate, renorm, topk_ids + (size_t)t * k, topk_w + (size_t)t * k,
                  gate_out ? gate_out + (size_t)t * n_experts : nullptr,
                  split_choice ? choice_s + (size_t)threadIdx.x * (n_experts + n_groups) : nullptr, corr, n_groups, keep, group_top);
    if (w_scale != 1.0f)
      for (int j = 0; j < k; ++j) topk_w[(size_t)t * k + j] *= w_scale;
  }
}

// Residual add + RMSNorm + router in one launch, for a few decode tokens: one block per token
// forms h += delta, normalises it (the arithmetic of the norm kernel: a thread per run of 8, the
// same statistics), stores the normalised row in `out` for the experts and keeps a copy in LDS,
// from which its waves then compute the router's logits (wave_dot_rows over the stored, rounded
// values: the bits of the router kernel) and one thread picks.  hidden % 8 == 0, hidden <= 8192.
constexpr int kFusedMaxHidden = 8192;

template <typename TW, typename TWR>
__global__ __launch_bounds__(1024) void add_rmsnorm_router_kernel(
    float* __restrict__ h, const bf16_t* __restrict__ delta, const TW* __restrict__ w, bf16_t* __restrict__ out,
    int hidden, float eps, const TWR* __restrict__ wr, int* __restrict__ topk_ids, float* __restrict__ topk_w,
    int n_experts, int k, int gate, int renorm) {
  __shared__ float red[16];
  __shared__ float g[1][kMaxExperts];
  __shared__ __attribute__((aligned(16))) bf16_t row[kFusedMaxHidden];
  const int t = blockIdx.x;
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = threadIdx.x >> 6;
  const int nw = blockDim.x >> 6;
  float* hr = h + (size_t)t * hidden;
  const int c = threadIdx.x * 8;
  float x[8], wk[8];
  float ss = 0.f;
  if (c < hidden) {
    load8(hr + c, x);
    if (w) load8(w + c, wk);
    if (delta) {
      float d[8];
      load8(delta + (size_t)t * hidden + c, d);
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] += d[j];
      store8(hr + c, x);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += x[j] * x[j];
  }
  const float total = block_sum(ss, red);
  const float s = 1.0f / sqrtf(total / (float)hidden + eps);
  if (c < hidden) {
    float y[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) y[j] = w ? (x[j] * s) * wk[j] : x[j] * s;
    store8(out + (size_t)t * hidden + c, y);
    store8(row + c, y);            // the same rounding: what the router would read back from memory
  }
  __syncthreads();
  const bf16_t* xr[1] = {row};
  for (int e = wv; e < n_experts; e += nw) {
    float v[1];
    wave_dot_rows<bf16_t, TWR, 1>(xr, wr + (size_t)e * hidden, hidden, lane, v);
    if (lane == 0) g[0][e] = v[0];
  }
  __syncthreads();
  if (k <= kWave) {
    if (wv == 0)
      gate_and_pick_wave(g[0], n_experts, k, gate, renorm, topk_ids + (size_t)t * k, topk_w + (size_t)t * k, nullptr, nullptr, nullptr,
                         1, 1, 1.0f, lane);
  } else if (threadIdx.x == 0) {
    gate_and_pick(g[0], n_experts, k, gate, renorm, topk_ids + (size_t)t * k, topk_w + (size_t)t * k, nullptr);
  }
}

// h [T, hidden] float (updated), delta [T, hidden] bf16 or null, w the norm's weights (bf16 or float, or
// null), out [T, hidden] bf16, wr [n_experts, hidden] (bf16 or float): what sharpi_add_rmsnorm then
// sharpi_router_topk give, in one launch.
SHARPI_EXPORT int sharpi_add_rmsnorm_router(float* h, const void* delta, const void* w, int w_dtype, void* out,
                                            int n_tokens, int hidden, float eps, const void* wr, int wr_dtype,
                                            int* topk_ids, float* topk_w, int n_experts, int k, int gate,
                                            int renorm, hipStream_t stream) {
  if (n_tokens <= 0) return SHARPI_OK;
  if (hidden <= 0 || (hidden & 7) || hidden > kFusedMaxHidden || !(eps > 0.f)) return SHARPI_ERR_ARG;
  if (n_experts <= 0 || n_experts > kMaxExperts || k <= 0 || k > n_experts || gate < 0 || gate > 1) return SHARPI_ERR_ARG;
  dim3 grid(n_tokens), block(1024);
#define FUSED_LAUNCH(TWV, TWRV)                                                                                  \
  add_rmsnorm_router_kernel<TWV, TWRV><<<grid, block, 0, stream>>>(h, (const bf16_t*)delta, (const TWV*)w,      \
                                                                   (bf16_t*)out, hidden, eps, (const TWRV*)wr,  \
                                                                   topk_ids, topk_w, n_experts, k, gate, renorm)
  const bool wf = w == nullptr || w_dtype == DT_F32;
  if (!wf && w_dtype != DT_BF16) return SHARPI_ERR_ARG;
  if (wr_dtype == DT_BF16) {
    if (wf) FUSED_LAUNCH(float, bf16_t); else FUSED_LAUNCH(bf16_t, bf16_t);
  } else if (wr_dtype == DT_F32) {
    if (wf) FUSED_LAUNCH(float, float); else FUSED_LAUNCH(bf16_t, float);
  } else {
    return SHARPI_ERR_ARG;
  }
#undef FUSED_LAUNCH
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}

// The experts a wave takes together (0: one at a time, with several runs of its row on their way), the tokens a block, the waves a block.  Every
// choice gives the same bits.
// Up to 256 tokens a block each: the chip has a unit for every one.  Behind that tokens share the experts' rows, two a block up to 512
// (where those rows are bfloat16; floats fill the registers), then four.  While the blocks still have a unit each, many waves
// hide each other's loads, so few experts are dealt to more of them; behind 1,024 tokens blocks share units, and four experts a wave with half of
// the waves cost the fewest loads and conversions a product.  Many float rows want the waves back there: their tokens' rows leave the
// cache before the next turn.
// Chosen from 2,737 sizes (1 to 1,024 experts, 1 to 8,192 tokens, widths of 512 to 5,120, the four pairs of types) and compared on 2,620 others with one
// expert a wave of sixteen, four from 64 experts, and four tokens from 257 on: none more than 6 % slower, 1.35 times as fast in the mean; with two
// tokens up to 1,023 and eight waves of four at every number of experts, up to 1.9 times slower than that: 1.09.  us, the one / the other / now: bfloat16, 1,000 rows 2,048 wide of 512
// experts 53 / 76 / 53, 600 of 96 13.4 / 21.2 / 13.4, 1,024 of 2 5.4 / 9.6 / 5.4, 8,192 rows 5,120 wide of 16 78 / 34 / 34, 300 of 16 10.7 / 7.2 / 7.2;
// floats, 1,024 wide, 600 of 2 4.9 / 9.0 / 4.9.  The same tried with tiles of 16 x 16 on the bfloat16 matrix instruction: 3,000 rows of 64 15.9
// for 25, but errors against 64 bits 1.15 to 1.3 times these.
struct RouterShape {
  int ee, tt, waves;
};
static RouterShape router_shape(int n_tokens, int hidden, int n_experts, bool x_float, bool w_float) {
  if (hidden & 7) return {0, n_tokens >= 64 ? 4 : 1, n_experts >= 16 ? 16 : n_experts >= 8 ? 8 : 4};       // (no runs of 8)
  const bool shared = n_tokens > 1024;               // blocks of four tokens share a unit
  int ee, tt = n_tokens <= 256 ? 1 : n_tokens <= 512 && !w_float ? 2 : 4;
  if (n_experts <= 2) ee = 0;
  else if (n_experts <= 4) ee = shared ? 2 : 0;
  else if (n_experts <= 8) ee = shared ? (w_float && !x_float ? 4 : 2) : tt == 2 ? 2 : 0;
  else if (shared || n_experts > 24) ee = 4;
  else if (tt == 1) ee = n_experts <= 16 && !x_float ? 0 : 4;
  else ee = x_float || w_float ? 4 : 2;
  if (tt == 2 && ee == 0) tt = 4;
  if (shared && n_experts <= 4 && ee == 2) tt = 2;   // (a wave a token for the picks)
  int most = 16;
  if (shared) most = x_float && n_tokens > 2048 && hidden >= 2048 && hidden * n_experts >= 3 << 17 ? 16 : 8;
  else if (x_float && w_float && n_tokens > 256 && hidden > 1024) most = 8;
  const int full = ceil_div(n_experts, ee ? ee : 1);
  return {ee, tt, min(most, max(ee == 0 ? 4 : tt, full))};
}

// corr (float [n_experts] or null): added to the gate values for the choice only.  n_groups, keep:
// picks come from the `keep` best of n_groups equal groups of neighbouring experts (1, 1: no groups), a group
// ranked by the sum of its group_top (1 or 2) largest choice scores.
// bias (float [n_experts] or null): added to the logits.  gate 0: sigmoid; 1: softmax over all experts;
// 2: the largest logits are picked and their weights are the softmax over the picked logits alone.
// w_scale multiplies the picks' weights at the end.
SHARPI_EXPORT int sharpi_router_topk(const void* x, int x_dtype, const void* wr, int w_dtype, int* topk_ids,
                                     float* topk_w, float* gate_out, int n_tokens, int hidden, int n_experts,
                                     int k, int gate, int renorm, const float* corr, int n_groups, int keep,
                                     const float* bias, float w_scale, int group_top, hipStream_t stream) {
  if (n_tokens <= 0) return SHARPI_OK;
  if (hidden <= 0 || n_experts <= 0 || n_experts > kMaxExperts || k <= 0 || k > n_experts) return SHARPI_ERR_ARG;
  if (gate < 0 || gate > 2) return SHARPI_ERR_ARG;
  if (n_groups < 1 || keep < 1 || keep > n_groups || n_experts % n_groups != 0 || k > keep * (n_experts / n_groups)) return SHARPI_ERR_ARG;
  if (group_top < 1 || group_top > kMaxGroupTop) return SHARPI_ERR_ARG;
  const int split_choice = corr != nullptr || keep < n_groups;
  const RouterShape shape = router_shape(n_tokens, hidden, n_experts, x_dtype == DT_F32, w_dtype == DT_F32);
  const int ee = shape.ee, tt = shape.tt, waves = shape.waves;
  dim3 grid(ceil_div(n_tokens, tt)), block(kWave * waves);
  const size_t lds = (size_t)tt * (n_experts + (split_choice ? n_experts + n_groups : 0)) * sizeof(float);
#define ROUTER_LAUNCH_AT(TX, TWT, EEV, TTV)                                                                      \
  router_topk_kernel<TX, TWT, EEV, TTV><<<grid, block, lds, stream>>>((const TX*)x, (const TWT*)wr, topk_ids, topk_w, \
                                                                      gate_out, n_tokens, hidden, n_experts, k, gate, \
                                                                      renorm, corr, n_groups, keep, split_choice, bias, w_scale, group_top)
#define ROUTER_LAUNCH_TT(TX, TWT, EEV)                                                                           \
  do {                                                                                                           \
    if (tt == 4) ROUTER_LAUNCH_AT(TX, TWT, EEV, 4);                                                              \
    else if (tt == 1) ROUTER_LAUNCH_AT(TX, TWT, EEV, 1);                                                         \
    else if constexpr (EEV == 2 || (EEV == 4 && sizeof(TWT) == 2)) ROUTER_LAUNCH_AT(TX, TWT, EEV, 2);            \
  } while (0)
#define ROUTER_LAUNCH(TX, TWT)                                                                                   \
  do {                                                                                                           \
    if (ee == 4) ROUTER_LAUNCH_TT(TX, TWT, 4);                                                                   \
    else if (ee == 2) ROUTER_LAUNCH_TT(TX, TWT, 2);                                                              \
    else ROUTER_LAUNCH_TT(TX, TWT, 0);                                                                           \
  } while (0)
  if (x_dtype == DT_F32 && w_dtype == DT_F32) ROUTER_LAUNCH(float, float);
  else if (x_dtype == DT_BF16 && w_dtype == DT_BF16) ROUTER_LAUNCH(bf16_t, bf16_t);
  else if (x_dtype == DT_BF16 && w_dtype == DT_F32) ROUTER_LAUNCH(bf16_t, float);
  else if (x_dtype == DT_F32 && w_dtype == DT_BF16) ROUTER_LAUNCH(float, bf16_t);
  else return SHARPI_ERR_ARG;
#undef ROUTER_LAUNCH
#undef ROUTER_LAUNCH_TT
#undef ROUTER_LAUNCH_AT
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}

// One block: the expert-sorted list of the (token, pick) pairs.  Every thread of the block calls it; the pairs must be visible to the block.
//
// Bound: latency, one block's chain of loads, counters and sums, and its scattered stores: a wave that stores to 64 lines takes 64 cycles and more of
// its unit, so the list is put in order in LDS, a window of rows after the other, and leaves by whole lines.  A thread requests all its pairs (and
// up to 24 weights) at once and keeps them (KEEP a thread; 0: more pairs than it can, read again for the second pass and stored one by one); an
// expert has up to 16 counters, a lane takes the one of its number, and what the counter held is the pair's place behind the counter's first row;
// every group counts the units before its own from one number a group.
// 24 pairs a thread are what its 128 registers and the window's LDS hold; beyond 24,576 pairs (8,192 tokens of four picks or more) the list is made as
// before, and costs what it did: 49,152 pairs 53 us, 65,536 82.
// us, pairs read, counted and stored one by one in two passes before: 18,000 pairs of 64 experts 24.8 -> 17.5, 9,984 17.5 -> 13.0, 8,192 of 28 and of
// 16 10.7 -> 8.4 and 10.8 -> 7.8.
constexpr unsigned kPlanRankParts = 32;        // (above kPlanMaxParts)
constexpr int kPermuteThreads = 1024;
constexpr int kPermuteCounters = 1024;         // counters of all experts
constexpr int kMaxCopies = 16;                 // counters an expert
template <int KEEP> constexpr int kPermuteWindow = KEEP <= 1 ? 1 : KEEP <= 8 ? KEEP * 1024 : 16384;    // rows put in order at a time
static_assert(kPermuteCounters >= kMaxExperts && kPermuteCounters <= kPermuteThreads, "a counter for every expert, a thread for every counter");

template <int KEEP>
__device__ void permute_block(const int* __restrict__ topk_ids, const float* __restrict__ topk_w,
                              int* __restrict__ offsets, int* __restrict__ sorted_token,
                              float* __restrict__ sorted_w, int* __restrict__ inv_pos, int* __restrict__ plan,
                              int n_pairs, int k, int n_experts, int shared_group, int* count, int* counters, int* spare,
                              int* plan_scratch, int* row_token, float* row_weight) {
  constexpr int kAhead = 8;                  // pairs a thread has in flight where it does not keep them
  constexpr bool kWeights = KEEP > 0 && KEEP <= 24;
  constexpr int step = kPermuteThreads;
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  int log_copies = 0;
  if (KEEP > 0)
    while ((2 << log_copies) <= kMaxCopies && (n_experts << (log_copies + 1)) <= kPermuteCounters) ++log_copies;
  const int n_counters = n_experts << log_copies, copy = lane & ((1 << log_copies) - 1);
  const auto counter = [&](int id) { return (id << log_copies) + copy; };
  // i / k by a product: exact while i k < 2^32 (kept pairs are fewer than 2^15, k at most 2^10)
  const unsigned part_k = k > 1 ? (unsigned)(0xffffffffu / (unsigned)k + 1) : 0;
  const auto token_of = [&](int i) { return k > 1 ? (int)__umulhi((unsigned)i, part_k) : i; };
  int pair[KEEP > 0 ? KEEP : 1];             // the pair's expert, then its counter and (times kPermuteCounters) what that held; -1: no row
  float weight[kWeights ? KEEP : 1];
  if constexpr (KEEP > 0) {
#pragma unroll
    for (int x = 0; x < KEEP; ++x) {
      if (x % kAhead == 0 && x * step >= n_pairs) break;
      const int i = min(tid + x * step, n_pairs - 1);
      pair[x] = topk_ids[i];
      if (kWeights) weight[x] = topk_w[i];
    }
  }
  counters[tid] = 0;
  __syncthreads();
  if constexpr (KEEP > 0) {
    int* const mine = spare + tid;           // (pairs without a row count here: no branch, all on their way together)
#pragma unroll
    for (int x = 0; x < KEEP; ++x) {
      if (x % kAhead == 0 && x * step >= n_pairs) break;
      const bool real = tid + x * step < n_pairs && pair[x] < n_experts;
      const int c = counter(pair[x]);
      const int was = atomicAdd(real ? counters + c : mine, 1);
      pair[x] = real ? was * kPermuteCounters + c : -1;
    }
  } else {
    for (int i0 = tid; i0 < n_pairs; i0 += kAhead * step) {
      int id[kAhead];
#pragma unroll
      for (int x = 0; x < kAhead; ++x) id[x] = topk_ids[min(i0 + x * step, n_pairs - 1)];
#pragma unroll
      for (int x = 0; x < kAhead; ++x)
        if (i0 + x * step < n_pairs && id[x] < n_experts) atomicAdd(counters + counter(id[x]), 1);
    }
  }
  __syncthreads();
  // the rows before each counter's: a sum over the wave's counters, then over the waves before it
  const int held = tid < n_counters ? counters[tid] : 0;
  int upto = held;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int o = __shfl_up(upto, off, kWave);
    if (lane >= off) upto += o;
  }
  if (lane == kWave - 1) plan_scratch[tid / kWave] = upto;
  __syncthreads();
  int before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kPermuteThreads / kWave; ++w) {
    const int sum = plan_scratch[w];
    before += w < tid / kWave ? sum : 0;
    all += sum;
  }
  if (tid < n_counters) {
    counters[tid] = before + upto - held;
    if (copy == 0) offsets[tid >> log_copies] = before + upto - held;
  }
  if (tid == 0) {
    offsets[n_experts] = all;
    // an always-on expert as one more group: every token once, in token order, with weight 1
    if (shared_group) {
      offsets[n_experts + 1] = all + n_pairs / k;
      count[n_experts] = n_pairs / k;
    }
  }
  __syncthreads();
  for (int e = tid; e < n_experts; e += step) count[e] = (e + 1 < n_experts ? counters[(e + 1) << log_copies] : all) - counters[e << log_copies];
  // (an identity expert: no product, no row; whoever sums the pairs asks the id)
  if constexpr (KEEP > 0) {
    constexpr int W = kPermuteWindow<KEEP>;
#pragma unroll
    for (int x = 0; x < KEEP; ++x) {
      if (x % kAhead == 0 && x * step >= n_pairs) break;
      const int i = tid + x * step;
      if (pair[x] >= 0) pair[x] = counters[(unsigned)pair[x] % kPermuteCounters] + (unsigned)pair[x] / kPermuteCounters;
      if (i < n_pairs) inv_pos[i] = max(pair[x], 0);
    }
    if constexpr (KEEP == 1) {               // (a store a thread: no order to wait for)
      if (n_pairs > 0 && pair[0] >= 0) {
        sorted_token[pair[0]] = token_of(tid);
        sorted_w[pair[0]] = weight[0];
      }
    } else for (int w0 = 0; w0 < all; w0 += W) {
      if (w0 > 0) __syncthreads();           // (the window before has left)
#pragma unroll
      for (int x = 0; x < KEEP; ++x) {
        if (x % kAhead == 0 && x * step >= n_pairs) break;
        const int r = pair[x] - w0, i = tid + x * step;
        if (pair[x] >= 0 && r >= 0 && r < W) {
          row_token[r] = token_of(i);
          row_weight[r] = kWeights ? weight[x] : topk_w[i];
        }
      }
      __syncthreads();
      for (int r = tid; r < min(W, all - w0); r += step) {
        sorted_token[w0 + r] = row_token[r];
        sorted_w[w0 + r] = row_weight[r];
      }
    }
  }
  if (shared_group) {
    for (int t = threadIdx.x; t < n_pairs / k; t += blockDim.x) {
      sorted_token[n_pairs + t] = t;
      sorted_w[n_pairs + t] = 1.0f;
    }
  }
  if (plan) {
    // The plan of the grouped product (grouped_plan.h).  Groups: the experts, and the always-on
    // group (every token once) if there is one.  Every group with rows gives plan_parts units;
    // units in the order of their weight (then of group and part) are dealt to the XCDs row by
    // row, rows alternating in direction so that the XCDs' loads stay level.
    const int n_groups = n_experts + (shared_group ? 1 : 0);
    const int stride = plan_stride(n_groups);
    __syncthreads();
    // a group's weight and units as one number that orders groups as the deal does and tells their units; 0: no rows
    int* rank = plan_scratch;
    for (int g = threadIdx.x; g < n_groups; g += step) {
      const int sg = plan_siblings(count[g]);
      rank[g] = count[g] == 0 ? 0 : plan_weight(sg) * (int)kPlanRankParts + plan_parts(sg);
    }
    __syncthreads();
    for (int g = threadIdx.x; g < n_groups; g += step) {
      if (count[g] == 0) continue;
      const int sg = plan_siblings(count[g]);
      const int wg = plan_weight(sg), pg = plan_parts(sg);
      // units that come before this group's: of heavier groups all, of equally heavy ones those of lower index
      int before = 0;
#pragma unroll 8
      for (int j = 0; j < n_groups; ++j) {
        const int wj = (unsigned)rank[j] / kPlanRankParts;
        before += wj > wg || (wj == wg && j < g) ? (unsigned)rank[j] % kPlanRankParts : 0;
      }
      for (int part = 0; part < pg; ++part) {
        const int u = before + part;
        const int pos = u / kPlanXcds;
        const int xcd = (pos & 1) ? kPlanXcds - 1 - u % kPlanXcds : u % kPlanXcds;
        int* pu = plan + xcd * stride + 1 + 4 * pos;
        pu[0] = g;
        pu[1] = part;
        pu[2] = pg;
        pu[3] = sg;
      }
    }
    if (threadIdx.x >= kWave && threadIdx.x < 2 * kWave) {       // (the second wave: the first has groups to place)
      int units = 0;
      for (int g = threadIdx.x - kWave; g < n_groups; g += kWave) units += (unsigned)rank[g] % kPlanRankParts;
#pragma unroll
      for (int off = kWave / 2; off > 0; off >>= 1) units += __shfl_xor(units, off, kWave);
      const int x = threadIdx.x - kWave;
      if (x < kPlanXcds) {
        // XCD x holds one unit of every full row of 8, and of the last row its own if it exists
        const int rows = units / kPlanXcds, left = units % kPlanXcds;
        plan[x * stride] = rows + (((rows & 1) ? kPlanXcds - 1 - x : x) < left ? 1 : 0);
      }
    }
    if (threadIdx.x < kPlanCounters) plan[plan_counters_at(n_groups) + threadIdx.x] = 0;
  }
  if constexpr (KEEP == 0) {
    __syncthreads();                         // (the counts are taken: the counters go on as the next rows)
    for (int i0 = tid; i0 < n_pairs; i0 += kAhead * step) {
      int id[kAhead], row[kAhead];
      float wt[kAhead];
#pragma unroll
      for (int x = 0; x < kAhead; ++x) {
        const int i = min(i0 + x * step, n_pairs - 1);
        id[x] = topk_ids[i];
        wt[x] = topk_w[i];
      }
#pragma unroll
      for (int x = 0; x < kAhead; ++x)
        row[x] = i0 + x * step < n_pairs && id[x] < n_experts ? atomicAdd(counters + counter(id[x]), 1) : -1;
#pragma unroll
      for (int x = 0; x < kAhead; ++x)
        if (const int i = i0 + x * step; i < n_pairs) {
          if (row[x] >= 0) {
            sorted_token[row[x]] = (unsigned)i / (unsigned)k;
            sorted_w[row[x]] = wt[x];
          }
          inv_pos[i] = max(row[x], 0);
        }
    }
  }
}

template <int KEEP>
__global__ __launch_bounds__(kPermuteThreads) void moe_permute_kernel(const int* __restrict__ topk_ids,
                                                           const float* __restrict__ topk_w,
                                                           int* __restrict__ offsets,
                                                           int* __restrict__ sorted_token,
                                                           float* __restrict__ sorted_w,
                                                           int* __restrict__ inv_pos, int* __restrict__ plan,
                                                           int n_pairs, int k, int n_experts, int shared_group) {
  __shared__ int count[kMaxExperts + 1];
  __shared__ int counters[kPermuteCounters];
  __shared__ int spare[kPermuteThreads];
  __shared__ int plan_scratch[kMaxExperts + 1];
  __shared__ int row_token[kPermuteWindow<KEEP>];
  __shared__ float row_weight[kPermuteWindow<KEEP>];
  permute_block<KEEP>(topk_ids, topk_w, offsets, sorted_token, sorted_w, inv_pos, plan, n_pairs, k, n_experts,
                shared_group, count, counters, spare, plan_scratch, row_token, row_weight);
}

// plan: plan_ints(n_experts + shared_group) ints (grouped_plan.h) for the grouped product of many rows, or null.
SHARPI_EXPORT int sharpi_moe_permute(const int* topk_ids, const float* topk_w, int* offsets, int* sorted_token,
                                     float* sorted_w, int* inv_pos, int* plan, int plan_len, int n_tokens, int k,
                                     int n_experts, int shared_group, int identity, hipStream_t stream) {
  if (shared_group && identity) return SHARPI_ERR_ARG;
  if (n_experts <= 0 || n_experts > kMaxExperts || k <= 0) return SHARPI_ERR_ARG;
  if (n_tokens < 0) return SHARPI_ERR_ARG;
  if (plan && plan_len < plan_ints(n_experts + (shared_group ? 1 : 0))) return SHARPI_ERR_ARG;
  const int n_pairs = n_tokens * k;
#define PERMUTE(KEEPV)                                                                                                          \
  moe_permute_kernel<KEEPV><<<1, kPermuteThreads, 0, stream>>>(topk_ids, topk_w, offsets, sorted_token, sorted_w, inv_pos, plan, n_pairs, k, \
                                                    n_experts, shared_group)
  // (as few pairs a thread as hold them all: 2 for 8 at 2,048 pairs 6.4 -> 5.4 us, 4 for 8 at 4,096 6.9 -> 6.4; stored one by one, as 1 a thread is,
  // these took 6.3 and 8.7)
  if (n_pairs <= 1024) PERMUTE(1);
  else if (n_pairs <= 2 * 1024) PERMUTE(2);
  else if (n_pairs <= 4 * 1024) PERMUTE(4);
  else if (n_pairs <= 8 * 1024) PERMUTE(8);
  else if (n_pairs <= 24 * 1024) PERMUTE(24);
  else PERMUTE(0);
#undef PERMUTE
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}

SHARPI_EXPORT int sharpi_grouped_plan_ints(int n_groups) { return plan_ints(n_groups); }
SHARPI_EXPORT int sharpi_router_max_experts() { return kMaxExperts; }
SHARPI_EXPORT int sharpi_add_rmsnorm_router_max_hidden() { return kFusedMaxHidden; }
