// What lies between an attention layer's input projections and its attention kernel, for layers
// that norm before they rotate: an optional short causal convolution over time on every channel
// of q, k and v, an RMS norm of q and of k with learned weights (per head, one weight vector
// shared by the heads; or over the whole projection, one weight per channel), rotary positions on
// the first r elements of every head (pairs interleaved or split in halves, cos and sin times a
// magnitude), and the write of keys and values into the paged cache.  Values may be the keys as
// they were before norm and rotation (a layer without a value projection).  Further options: a bias
// per projected channel (float, added to the row as it is gathered; not together with a
// convolution), a query temperature 1 + c ln(floor((p + 1) / f) + 1) on q, and heads that hold
// several score maps side by side (`maps`): norm weights and cache rows stay per head, the rotation
// works on each map's own leading elements, and the queries leave expanded, one row of the head's
// width per (head, map) with that map's elements in their place and zeros elsewhere, so that an
// attention kernel over keys of the head's width computes each map's scores on its own; and values mixed with
// those of another layer, (1 - c) v + c v_other, in float on their way into the cache.
//
// Rows of widths and offsets that are multiples of 8, and heads of up to 512, go to qk_prep_run_kernel; the others, and norms over projections of more
// than 1,024 lanes (q and kv heads times hd / 8 rounded up to a power of two), as follows.
// One block per token, or, in steps of few tokens, one per (token, kv head): the block then takes
// that kv head's key and value and the query heads that read it, so that a decode step still fills
// the chip (what a row's sums are made of and their order do not depend on the split).  The token's
// row is gathered into LDS as floats (the convolution reads up to taps - 1 earlier rows: of this
// step where the entry has them, otherwise the tail that the request's state slot carries), the
// sums of squares are taken in an order that depends on the row alone, and everything after the
// projection is float arithmetic rounded once, on the way out.
#include "common.h"
#include "value_pages.h"

constexpr int kPrepThreads = 256;
constexpr int kPrepMaxTaps = 8;
constexpr int kPrepTapsAhead = 3;     // taps whose rows and weights are on their way together (any number but four)
constexpr int kPrepSplitTokens = 64;  // up to so many tokens a step, a token's heads are spread over nkv blocks
// Values of convolved rows go in blocks of their own by tiles of 16 tokens from more tokens on: a tile's thread gathers one run after the other, which
// of few tiles is the step's longest chain.  Apart / beside, times as fast as with the
// whole row staged, in the mean: three taps, 300 tokens 1.22 / 1.25, 700 1.13 / 1.17, but 1,400 1.12 / 1.07; eight taps, 300 1.11 / 1.24, 700 1.04 / 1.16, and
// at 5,000 single shapes 0.85 / 0.99: with more than four taps always beside, and so keys that are the values, which a tile would convolve twice.
constexpr int kPrepBesideFewTaps = 500;
constexpr int kPrepMaxHeads = 1024;   // q heads + kv heads whose inverse norms are kept in LDS

enum : int { NORM_NONE = 0, NORM_PER_HEAD = 1, NORM_WHOLE = 2 };

struct PrepArgs {
  const void* proj;        // [T, stride]
  int stride, q_off, k_off, v_off;   // v_off < 0: the values are the keys before norm and rotation
  int nh, nkv, hd, vd;
  const float* conv_w;     // [q + k + v channels, taps] or null
  int taps;
  float* tail;             // [slots, taps - 1, channels]: the last projected rows of each request
  const int* state_slots;  // [entries]
  const int* entry_of_token;
  const int* cu_tokens;
  const int* positions;
  int norm_mode;
  const float* q_norm_w;   // [hd] or [nh * hd]
  const float* k_norm_w;   // [hd] or [nkv * hd]
  float eps;
  const float* inv_freq;   // [rotary_dim / 2] or null
  int rotary_dim, half_split;
  float magnitude;
  void* q_out;             // [T, nh * hd]
  void* k_cache;           // [pages, nkv, page_size, hd]
  void* v_cache;           // [pages, nkv, vd, page_size]
  const int* slot_mapping; // [T], -1: store nothing
  int page_size;
  int parts;               // blocks a token: 1, or nkv (a kv head and its query heads each)
  const float* bias;       // [q + k + v channels] or null
  int temp_on;             // query temperature
  float temp_floor, temp_scale;
  int maps;                // score maps a head (1: the plain layout of q_out; > 1: q_out [T, nh * maps * hd], expanded)
  const void* v_other;     // another layer's projections of the same tokens (null: values as they are)
  int v_other_stride, v_other_off;
  float v_mix;             // c
  int values_apart;        // values go in blocks of their own behind the tokens' (value_pages.h)
  int values_beside;       // (runs) few tokens: a token's values go in a block of their own, the last of its column
  int n_tokens;
  int by8;                 // every offset, stride and width a multiple of 8 (and split halves): eight channels a thread
};

constexpr int kPrepMaxTurns = 256;    // rotary pairs whose cosines and sines a block keeps (a map of up to 512 elements)
static_assert(kPrepThreads == kValueThreads, "a block of either kind");

// Channels c .. c + 7 of q | k | v of token t, column col of its projected row, through the convolution or with the bias (wide
// rows).  TAPS: 0 none, 4 four with their weights on multiples of 32 bytes, -1 any number.
template <typename T, int TAPS>
__device__ __forceinline__ void prep_gather8(const PrepArgs& a, int t, int c, int col, int C, float* y) {
  const T* proj = (const T*)a.proj;
  if constexpr (TAPS != 0) {
    if constexpr (TAPS == 4) {
      // The four rows, as they lie in memory or, of an entry's first three tokens, in the tail, and the eight channels' weights (32 floats on
      // end, 16 bytes a load) are all requested before the first is used; a weight and a row at a time the loads' number and latency were
      // the kernel's time (1900 tokens of 4096 channels: 62 -> 35 us).
      float4 cw[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) cw[i] = *reinterpret_cast<const float4*>(a.conv_w + (size_t)(c + i) * 4);
      const auto add = [&](int j, const float* v) {
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = fmaf(j == 0 ? cw[i].x : j == 1 ? cw[i].y : j == 2 ? cw[i].z : cw[i].w, v[i], j == 0 ? 0.f : y[i]);
      };
      const int e = a.entry_of_token[t], li = t - a.cu_tokens[e];          // (the token's place in its entry)
      const T* rows = proj + (size_t)t * a.stride + col;
      if (li >= 3) {
        Run8<T> u[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) u[j].load(rows - (size_t)(3 - j) * a.stride);
        float v[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          u[j].floats(v);
          add(j, v);
        }
      } else {
        const float* tail = a.tail + ((size_t)a.state_slots[e] * 3 + li) * C + c;
        Run8<T> own;
        float v[3][8];
        own.load(rows);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          if (3 - j > li) load8(tail + (size_t)j * C, v[j]);
          else load8(rows - (size_t)(3 - j) * a.stride, v[j]);
        }
#pragma unroll
        for (int j = 0; j < 3; ++j) add(j, v[j]);
        own.floats(v[0]);
        add(3, v[0]);
      }
      return;
    }
    const int e = a.entry_of_token[t];
    const int li = t - a.cu_tokens[e];                 // the token's place in its entry
    const float* tail = a.tail + (size_t)a.state_slots[e] * (a.taps - 1) * C;
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] = 0.f;
    // (several taps' rows and weights requested together: one after the other, 8 tokens of three taps and 8 + 1 heads of 64 took 9.4 us, so 7.9)
#pragma unroll 1
    for (int j0 = 0; j0 < a.taps; j0 += kPrepTapsAhead) {
      float u[kPrepTapsAhead][8], cw[kPrepTapsAhead][8];
#pragma unroll
      for (int x = 0; x < kPrepTapsAhead; ++x) {
        const int j = min(j0 + x, a.taps - 1), back = a.taps - 1 - j;      // this tap reads the row `back` tokens ago
        if (back <= li) load8(proj + (size_t)(t - back) * a.stride + col, u[x]);
        else load8(tail + (size_t)(a.taps - 1 + li - back) * C + c, u[x]);
#pragma unroll
        for (int i = 0; i < 8; ++i) cw[x][i] = a.conv_w[(size_t)(c + i) * a.taps + j];
      }
#pragma unroll
      for (int x = 0; x < kPrepTapsAhead; ++x) {
        if (j0 + x >= a.taps) break;
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = fmaf(cw[x][i], u[x][i], y[i]);
      }
    }
    return;
  }
  load8(proj + (size_t)t * a.stride + col, y);
  if (a.bias) {
    float b8[8];
    load8(a.bias + c, b8);
#pragma unroll
    for (int i = 0; i < 8; ++i) y[i] += b8[i];
  }
}

// Values mixed with another layer's: channels c .. c + 7 of the values of token t.
template <typename T>
__device__ __forceinline__ void prep_mix8(const PrepArgs& a, int t, int c, float* v) {
  if (!a.v_other) return;
  const T* other = (const T*)a.v_other + (size_t)t * a.v_other_stride + a.v_other_off + c;
  float u[8];
  load8(other, u);
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j] = fmaf(1.0f - a.v_mix, v[j], a.v_mix * u[j]);
}

template <typename T, int TAPS>
__global__ __launch_bounds__(kPrepThreads) void qk_prep_kernel(PrepArgs a) {
  extern __shared__ __attribute__((aligned(32))) float row[];          // q | k | v of the token, as floats (values apart: q | k)
  __shared__ float red[16];
  __shared__ float inv[kPrepMaxHeads];
  if (blockIdx.x >= a.n_tokens) {          // (values_apart: the blocks behind the tokens')
    const bool own = a.v_off >= 0;
    const int v0 = own ? (a.nh + a.nkv) * a.hd : a.nh * a.hd, all_c = (a.nh + a.nkv) * a.hd + (own ? a.nkv * a.vd : 0);
    values_to_pages<T>(blockIdx.x - a.n_tokens, a.n_tokens, a.nkv, a.vd, a.page_size, a.slot_mapping, (T*)a.v_cache,
                       reinterpret_cast<T*>(row), reinterpret_cast<int*>(inv), [&](int tt, int c, float* v) {
      prep_gather8<T, TAPS>(a, tt, v0 + c, (own ? a.v_off : a.k_off) + c, all_c, v);
      prep_mix8<T>(a, tt, c, v);
    });
    return;
  }
  const int t = blockIdx.x;
  // the heads this block takes: all, or kv head blockIdx.y with its query heads
  const int per_kv = a.nh / a.nkv;
  const int qh0 = a.parts > 1 ? blockIdx.y * per_kv : 0, qh1 = a.parts > 1 ? qh0 + per_kv : a.nh;
  const int kh0 = a.parts > 1 ? blockIdx.y : 0, kh1 = a.parts > 1 ? kh0 + 1 : a.nkv;
  const bool every_qk = a.norm_mode == NORM_WHOLE;   // a norm over the whole projection reads all of q and of k
  const int qn = a.nh * a.hd, kn = a.nkv * a.hd;
  const bool own_v = a.v_off >= 0;
  const int vn = own_v ? a.nkv * a.vd : 0;
  const int C = qn + kn + vn;
  const T* proj = (const T*)a.proj;
  const bool all = a.parts == 1;                     // (then no channel or head needs asking)
  auto mine = [&](int c) {
    if (all) return true;
    if (c < qn) return every_qk || (c / a.hd >= qh0 && c / a.hd < qh1);
    if (c < qn + kn) return every_qk || ((c - qn) / a.hd >= kh0 && (c - qn) / a.hd < kh1);
    return (c - qn - kn) / a.vd >= kh0 && (c - qn - kn) / a.vd < kh1;
  };

  // 1. gather, through the convolution where there is one
  const int upto = a.values_apart ? qn + kn : C;
  if (a.by8) {
    // eight consecutive channels a thread, 16-byte loads (the sums of a channel are those of the scalar form)
    for (int c = threadIdx.x * 8; c < upto; c += kPrepThreads * 8) {
      if (!mine(c)) continue;
      const int col = c < qn ? a.q_off + c : c < qn + kn ? a.k_off + (c - qn) : a.v_off + (c - qn - kn);
      float y[8];
      prep_gather8<T, TAPS>(a, t, c, col, C, y);
      store8(row + c, y);
    }
  } else if (a.taps > 0) {
    const int e = a.entry_of_token[t];
    const int li = t - a.cu_tokens[e];                 // the token's place in its entry
    const float* tail = a.tail + (size_t)a.state_slots[e] * (a.taps - 1) * C;
    for (int c = threadIdx.x; c < upto; c += kPrepThreads) {
      if (!mine(c)) continue;
      const int col = c < qn ? a.q_off + c : c < qn + kn ? a.k_off + (c - qn) : a.v_off + (c - qn - kn);
      float y = 0.f;
      for (int j = 0; j < a.taps; ++j) {
        const int back = a.taps - 1 - j;               // this tap reads the row `back` tokens ago
        float u;
        if (back <= li) u = to_f32<T>(proj[(size_t)(t - back) * a.stride + col]);
        else u = tail[(size_t)(a.taps - 1 + li - back) * C + c];
        y = fmaf(a.conv_w[(size_t)c * a.taps + j], u, y);
      }
      row[c] = y;
    }
  } else {
    for (int c = threadIdx.x; c < upto; c += kPrepThreads) {
      if (!mine(c)) continue;
      const int col = c < qn ? a.q_off + c : c < qn + kn ? a.k_off + (c - qn) : a.v_off + (c - qn - kn);
      const float u = to_f32<T>(proj[(size_t)t * a.stride + col]);
      row[c] = a.bias ? u + a.bias[c] : u;
    }
  }
  __syncthreads();

  // 2. values leave as they are (a layer without a value projection stores its unnormed keys)
  const int slot = a.slot_mapping ? a.slot_mapping[t] : -1;
  if (slot >= 0 && !a.values_apart) {
    const int page = slot / a.page_size, off = slot % a.page_size;
    T* vc = (T*)a.v_cache;
    const float* vsrc = own_v ? row + qn + kn : row + qn;
    for (int i = kh0 * a.vd + threadIdx.x; i < kh1 * a.vd; i += kPrepThreads) {
      const int g = i / a.vd, d = i % a.vd;
      float v = vsrc[i];
      if (a.v_other) v = fmaf(1.0f - a.v_mix, v, a.v_mix * to_f32<T>(((const T*)a.v_other)[(size_t)t * a.v_other_stride + a.v_other_off + i]));
      vc[(((size_t)page * a.nkv + g) * a.vd + d) * a.page_size + off] = from_f32<T>(v);
    }
  }

  // 3. inverse norms
  const int lane = threadIdx.x & (kWave - 1), wid = threadIdx.x >> 6;
  const int heads = a.nh + a.nkv;
  if (a.norm_mode == NORM_PER_HEAD) {
    for (int h = wid; h < heads; h += kPrepThreads / kWave) {
      if (!all && !(h < a.nh ? (h >= qh0 && h < qh1) : (h - a.nh >= kh0 && h - a.nh < kh1))) continue;
      const float* x = row + (size_t)h * a.hd;         // (q heads then k heads lie back to back)
      float ss = 0.f;
      for (int d = lane; d < a.hd; d += kWave) ss = fmaf(x[d], x[d], ss);
      ss = wave_sum(ss);
      if (lane == 0) inv[h] = rsqrtf(ss / (float)a.hd + a.eps);
    }
  } else if (a.norm_mode == NORM_WHOLE) {
    float sq = 0.f, sk = 0.f;
    for (int c = threadIdx.x; c < qn; c += kPrepThreads) sq = fmaf(row[c], row[c], sq);
    for (int c = threadIdx.x; c < kn; c += kPrepThreads) sk = fmaf(row[qn + c], row[qn + c], sk);
    sq = block_sum(sq, red);
    sk = block_sum(sk, red);
    const float iq = rsqrtf(sq / (float)qn + a.eps), ik = rsqrtf(sk / (float)kn + a.eps);
    for (int h = threadIdx.x; h < heads; h += kPrepThreads) inv[h] = h < a.nh ? iq : ik;
  }
  __syncthreads();

  // 4. norm, rotation, and out: a thread takes a pair of a head (or two elements that do not turn)
  const float pos = (float)a.positions[t];
  __shared__ float cs_tab[kPrepMaxTurns], sn_tab[kPrepMaxTurns];      // the token's angles are the same for every head and map
  if (a.inv_freq) {
    for (int i = threadIdx.x; i < a.rotary_dim / 2; i += kPrepThreads) {
      const float ang = pos * a.inv_freq[i];
      cs_tab[i] = cosf(ang) * a.magnitude;
      sn_tab[i] = sinf(ang) * a.magnitude;
    }
    __syncthreads();
  }
  const int sd = a.hd / a.maps;                          // width of one map of a head (the head's, with one map)
  const int half_hd = a.hd / 2, half_sd = sd / 2, half_r = a.rotary_dim / 2;
  T* qo = (T*)a.q_out + (size_t)t * qn * a.maps;
  T* kc = (T*)a.k_cache;
  const float temp = a.temp_on ? 1.0f + a.temp_scale * logf(floorf((pos + 1.0f) / a.temp_floor) + 1.0f) : 1.0f;
  if (a.by8) {
    // Eight consecutive elements a thread, 16-byte stores.  A run in the low half of a map's rotated part comes
    // with its partner run half the rotated width on (the thread turns both); a run behind the rotated part passes.
    const int runs = sd / 8, low = half_r / 8, rot_runs = a.rotary_dim / 8;
    const int per_map = runs - low;                      // work items of a map: low runs (each with its partner) and the rest
    const int page = slot >= 0 ? slot / a.page_size : 0, off = slot >= 0 ? slot % a.page_size : 0;
    for (int i = threadIdx.x; i < heads * a.maps * per_map; i += kPrepThreads) {
      const int hs = i / per_map, wi = i % per_map;
      const int h = hs / a.maps, mp = hs % a.maps, at = mp * sd;
      if (!all && !(h < a.nh ? (h >= qh0 && h < qh1) : (h - a.nh >= kh0 && h - a.nh < kh1))) continue;
      const bool is_q = h < a.nh, turns = wi < low;
      if (!is_q && slot < 0) continue;
      const int e0 = at + (turns ? wi * 8 : (rot_runs + (wi - low)) * 8);      // first element inside the head
      const int e1 = e0 + half_r;                                               // the partner run (turning runs only)
      float x0[8], x1[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      load8(row + (size_t)h * a.hd + e0, x0);
      if (turns) load8(row + (size_t)h * a.hd + e1, x1);
      if (a.norm_mode != NORM_NONE) {
        const float* w = is_q ? a.q_norm_w : a.k_norm_w;
        const int wbase = a.norm_mode == NORM_WHOLE ? (is_q ? h : h - a.nh) * a.hd : 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          x0[j] = x0[j] * inv[h] * w[wbase + e0 + j];
          if (turns) x1[j] = x1[j] * inv[h] * w[wbase + e1 + j];
        }
      }
      if (turns) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float c = cs_tab[wi * 8 + j], sn = sn_tab[wi * 8 + j];
          const float y0 = fmaf(x0[j], c, -(x1[j] * sn)), y1 = fmaf(x0[j], sn, x1[j] * c);
          x0[j] = y0;
          x1[j] = y1;
        }
      }
      if (is_q) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          x0[j] *= temp;
          x1[j] *= temp;
        }
        if (a.maps == 1) {
          store8(qo + (size_t)h * a.hd + e0, x0);
          if (turns) store8(qo + (size_t)h * a.hd + e1, x1);
        } else {
          const float zero[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
          T* qr = qo + ((size_t)h * a.maps + mp) * a.hd;
          for (int mm = 0; mm < a.maps; ++mm) {
            const int sh = (mm - mp) * sd;
            store8(qr + e0 + sh, mm == mp ? x0 : zero);
            if (turns) store8(qr + e1 + sh, mm == mp ? x1 : zero);
          }
        }
      } else {
        T* kr = kc + (((size_t)page * a.nkv + (h - a.nh)) * a.page_size + off) * a.hd;
        store8(kr + e0, x0);
        if (turns) store8(kr + e1, x1);
      }
    }
    return;
  }
  for (int i = threadIdx.x; i < heads * half_hd; i += kPrepThreads) {
    const int hs = i / half_sd, pi = i % half_sd;         // (head, map) and the pair inside the map
    const int h = hs / a.maps, mp = hs % a.maps, at = mp * sd;
    if (!all && !(h < a.nh ? (h >= qh0 && h < qh1) : (h - a.nh >= kh0 && h - a.nh < kh1))) continue;
    int d0, d1;
    bool turns;
    if (pi < half_r) {
      turns = true;
      d0 = a.half_split ? pi : 2 * pi;
      d1 = a.half_split ? pi + half_r : 2 * pi + 1;
    } else {
      turns = false;
      d0 = a.rotary_dim + 2 * (pi - half_r);
      d1 = d0 + 1;
    }
    const bool is_q = h < a.nh;
    d0 += at;
    d1 += at;
    float x0 = row[(size_t)h * a.hd + d0], x1 = row[(size_t)h * a.hd + d1];
    if (a.norm_mode != NORM_NONE) {
      const float* w = is_q ? a.q_norm_w : a.k_norm_w;
      const int wbase = a.norm_mode == NORM_WHOLE ? (is_q ? h : h - a.nh) * a.hd : 0;
      x0 = x0 * inv[h] * w[wbase + d0];
      x1 = x1 * inv[h] * w[wbase + d1];
    }
    if (turns && a.inv_freq) {
      const float c = cs_tab[pi], s = sn_tab[pi];
      const float y0 = fmaf(x0, c, -(x1 * s)), y1 = fmaf(x1, c, x0 * s);
      x0 = y0;
      x1 = y1;
    }
    if (is_q) {
      x0 *= temp;
      x1 *= temp;
      if (a.maps == 1) {
        qo[(size_t)h * a.hd + d0] = from_f32<T>(x0);
        qo[(size_t)h * a.hd + d1] = from_f32<T>(x1);
      } else {
        // the (head, map)'s own row of the head's width: the map's elements in place, zeros in the other maps' places
        T* qr = qo + ((size_t)h * a.maps + mp) * a.hd;
        for (int mm = 0; mm < a.maps; ++mm) {
          const int sh = (mm - mp) * sd;
          qr[d0 + sh] = from_f32<T>(mm == mp ? x0 : 0.f);
          qr[d1 + sh] = from_f32<T>(mm == mp ? x1 : 0.f);
        }
      }
    } else if (slot >= 0) {
      const int page = slot / a.page_size, off = slot % a.page_size;
      T* kr = kc + (((size_t)page * a.nkv + (h - a.nh)) * a.page_size + off) * a.hd;
      kr[d0] = from_f32<T>(x0);
      kr[d1] = from_f32<T>(x1);
    }
  }
}

// The same for rows whose widths and offsets are multiples of 8 (pairs split in halves: the rotated width of 16): nothing is staged.  A head
// lies in neighbouring lanes of a wave, eight elements a lane (hd / 8 of them rounded up to a power of two); its sum of
// squares and the partner run of a split rotation come by lane exchange, 16-byte accesses throughout.  A block has a thread for
// every run of a token's heads where that is at most 1,024 (a norm over the whole projection asks for it), else blocks (token, y) share them; steps of many
// tokens leave the values to blocks of their own behind the tokens' (value_pages.h).
// Bound: a block's chain of latencies, so a run and its norm's weights are requested before the angles are formed, and the next before one is
// worked on; in short steps the values of a token, another chain, go in a block beside those of its heads.  us, 16 + 4 heads
// of 128, staged through LDS before: 1,900 tokens, norms over the projections 22.3 -> 12.7 (their squares added as the lanes come, with other bits,
// 11.7), two maps a head 21.9 -> 13.0, four taps with the tail's launch 37.9 -> 28.1; 8 tokens, a norm a head 4.6 -> 4.4 (weights and values behind
// the rest: 5.0), over the projections 7.7 -> 5.1, four taps 11.4 -> 7.9 (a tap of the tail at a time: 14.2), three taps 11.8 -> 9.6 (a tap at a
// time: 11.8).  64 + 8 heads of 192: 2,048 tokens (a block of 256 for three turns, each behind the one before) 40.9 -> 35; floats, 200 tokens
// four turns a block 9.9, two 9.0 (8.9 before), 64 tokens with neighbours on several dies 5.8, on one 5.5 (5.25 before).
constexpr int kRunMaxThreads = 1024;
// Convolved rows go by runs up to so many lanes a step: a gather's rows and weights fill the registers, so of a block of nine or ten waves a
// unit holds one at a time, and with enough tokens to fill the chip the staged form's blocks of four waves, several a unit, are through sooner.  us with
// the tail's launch, bfloat16, four taps, a norm a head, staged / runs: 16 + 2 heads of 192, 300 tokens 16.1 / 14.9, 1,400 29.0 / 37.9, 5,000 77.6 / 116; 32 + 8
// of 128, 300 20.7 / 16.1, 1,400 43.2 / 45.7, 2,800 69.9 / 85.3; 16 + 4 of 128, 1,400 24.3 / 23.2, 2,800 39.8 / 38.7.
// More than four taps are chains of several gathers: by runs up to 1,000 tokens (eight taps, times as fast as staged before values went apart: 300 tokens
// 1.24, 1,400 1.09 in the mean, but single shapes 0.85), and not in rows of up to 32 lanes, half a wave, whose chain is all there is (floats, 2 + 1 heads of
// 64, 33 single tokens: staged 10.3, runs 11.4).
constexpr long kRunMuch = 400 * 1024;
// Rows of more lanes than these go in turns of blocks of 256 beyond so much, a norm over the projection aside, for the same reason (plain rows of 32 + 8
// heads of 96, 6,000 tokens: one block 55, in turns 32; 20 + 4 of 192 interleaved, 3,000 tokens 30 and 20).
constexpr int kRunFullBlock = 512;
// Few taps of interleaved pairs, which are staged an element a thread, likewise beyond 500 tokens in rows of up to half a block (three taps, 8 + 2 heads of
// 64, 1,500 tokens: staged 13.0, runs 16.8), and beyond 1,000 in any.
constexpr int kRunManyTaps = 1000, kRunNarrow = 32, kRunHalfBlock = 128;

// How the squares of a norm are added.  RUN_LANES: eight a lane, then the lanes.  RUN_ROW and RUN_WHOLE, a norm over the projection: in the staged
// form's order, with its bits.  (Plain rows had the first before the others came here, and keep it.)  A rotation's multiply-adds are
// written out in every form: of the two products of a split pair's high half the one that is rounded is the one that the staged form by eights rounds.
enum : int { RUN_LANES = 0, RUN_ROW = 1, RUN_WHOLE = 2 };

template <typename T, int TAPS, int SUMS>
__global__ __launch_bounds__(kRunMaxThreads, TAPS != 0 ? 5 : 8) void qk_prep_run_kernel(PrepArgs a, int log_lanes) {
  __shared__ float cs_tab[kPrepMaxTurns], sn_tab[kPrepMaxTurns];
  __shared__ float red[2][kPrepThreads / kWave];
  extern __shared__ __attribute__((aligned(32))) float row[];          // (a norm over the whole projection: q | k of the token)
  __shared__ __attribute__((aligned(16))) char tile[kValueLds<T>];
  const int qn = a.nh * a.hd, kn = a.nkv * a.hd, runs = a.hd / 8, heads = a.nh + a.nkv;
  const bool own_v = a.v_off >= 0;
  const int v_at = own_v ? qn + kn : qn, v_col = own_v ? a.v_off : a.k_off, C = qn + kn + (own_v ? a.nkv * a.vd : 0);
  if (a.values_apart && blockIdx.x >= a.n_tokens) {     // (the blocks behind the tokens', y of them side by side)
    const int v = (blockIdx.x - a.n_tokens) * gridDim.y + blockIdx.y;
    if (v < value_tiles(a.n_tokens, a.nkv * a.vd))
      values_to_pages<T>(v, a.n_tokens, a.nkv, a.vd, a.page_size, a.slot_mapping, (T*)a.v_cache, reinterpret_cast<T*>(tile),
                         reinterpret_cast<int*>(cs_tab), [&](int tt, int c, float* x) {
        prep_gather8<T, TAPS>(a, tt, v_at + c, v_col + c, C, x);
        prep_mix8<T>(a, tt, c, x);
      });
    return;
  }
  // (short steps: neighbouring tokens on one die, whose cache gathers the values' columns)
  const int t = a.values_beside ? (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8 : blockIdx.x;
  if (t >= a.n_tokens) return;
  const int slot = a.slot_mapping ? a.slot_mapping[t] : -1;
  // a thread's run inside a head is the same in every turn
  const int li = threadIdx.x & ((1 << log_lanes) - 1);
  const bool in = li < runs;
  const int parts = gridDim.y - a.values_beside, step = parts * blockDim.x;
  const bool values_only = (int)blockIdx.y >= parts;
  int base = blockIdx.y * blockDim.x;
  constexpr bool kAhead = TAPS == 0 && SUMS != RUN_WHOLE;
  Run8<T> raw;                             // (without a convolution) the next turn's run, on its way, and a head's norm weights
  Run8<float> weight;
  const auto column = [&](int h) { return (h < a.nh ? a.q_off + h * a.hd : a.k_off + (h - a.nh) * a.hd) + li * 8; };
  const auto request = [&]() {
    const int h = (base + (int)threadIdx.x) >> log_lanes;
    if (!in || h >= heads) return;
    if (TAPS == 0) raw.load((const T*)a.proj + (size_t)t * a.stride + column(h));
    if (kAhead && a.norm_mode != NORM_NONE) weight.load((h < a.nh ? a.q_norm_w : a.k_norm_w) + li * 8);
  };
  if (!values_only) request();
  const float pos = (float)a.positions[t];
  if (a.inv_freq && !values_only) {
    for (int i = threadIdx.x; i < a.rotary_dim / 2; i += blockDim.x) {
      float sn, cs;
      sincosf(pos * a.inv_freq[i], &sn, &cs);
      cs_tab[i] = cs * a.magnitude;
      sn_tab[i] = sn * a.magnitude;
    }
    __syncthreads();
  }
  const int page = slot >= 0 ? slot / a.page_size : 0, off = slot >= 0 ? slot % a.page_size : 0;
  const float temp = a.temp_on ? 1.0f + a.temp_scale * logf(floorf((pos + 1.0f) / a.temp_floor) + 1.0f) : 1.0f;
  const int map_runs = a.maps > 1 ? runs / a.maps : runs, mp = a.maps > 1 ? li / map_runs : 0, lm = li - mp * map_runs;
  const int half_runs = a.rotary_dim / 16;               // split pairs: runs of the low half of the rotated part
  const bool low = lm < half_runs, turns = a.inv_freq && in && lm * 8 < a.rotary_dim;
  const int mate = (int)threadIdx.x + (low ? half_runs : -half_runs);
  const int ang = a.half_split ? (low ? lm : lm - half_runs) * 8 : lm * 4;     // the run's first angle
  for (bool more = !values_only; more;) {
    const int h = (base + (int)threadIdx.x) >> log_lanes;
    const bool is_q = h < a.nh, live = in && h < heads;
    float xs[1][8] = {{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}};
    float(&x)[8] = xs[0];
    if (live) {
      if constexpr (TAPS == 0) {
        raw.floats(x);
        if (a.bias) {
          float b8[8];
          load8(a.bias + h * a.hd + li * 8, b8);
#pragma unroll
          for (int j = 0; j < 8; ++j) x[j] += b8[j];
        }
      } else {
        prep_gather8<T, TAPS>(a, t, h * a.hd + li * 8, column(h), C, x);
      }
    }
    base += step;
    more = base < (heads << log_lanes);
    float w8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (kAhead && live && a.norm_mode != NORM_NONE) weight.floats(w8);
    if (more) request();
    if (a.norm_mode != NORM_NONE) {                      // every lane takes part in the exchanges (a lane without a run holds zeros)
      if (!kAhead && live) load8((is_q ? a.q_norm_w : a.k_norm_w) + (SUMS == RUN_WHOLE ? (is_q ? h : h - a.nh) * a.hd : 0) + li * 8, w8);
      float inv;
      if constexpr (SUMS != RUN_WHOLE) {
        float ss = 0.f;
        if constexpr (SUMS == RUN_LANES) {
#pragma unroll
          for (int j = 0; j < 8; ++j) ss = fmaf(x[j], x[j], ss);
          ss = group_sum(ss, 1 << log_lanes);
        } else {
          ss = row_square_sum(xs, 1 << log_lanes);
        }
        inv = rsqrtf(ss / (float)a.hd + a.eps);
      } else {                                           // (one turn)
        if (live) store8(row + h * a.hd + li * 8, x);
        __syncthreads();
        if (threadIdx.x < kPrepThreads) {                // (the staged form's threads, chains and pairs)
          float sq = 0.f, sk = 0.f;
#pragma unroll 4
          for (int c = threadIdx.x; c < qn; c += kPrepThreads) sq = fmaf(row[c], row[c], sq);
#pragma unroll 4
          for (int c = threadIdx.x; c < kn; c += kPrepThreads) sk = fmaf(row[qn + c], row[qn + c], sk);
          sq = wave_sum(sq);
          sk = wave_sum(sk);
          if (threadIdx.x % kWave == 0) {
            red[0][threadIdx.x / kWave] = sq;
            red[1][threadIdx.x / kWave] = sk;
          }
        }
        __syncthreads();
        float total = 0.f;
#pragma unroll
        for (int i = 0; i < kPrepThreads / kWave; ++i) total += red[is_q ? 0 : 1][i];
        inv = rsqrtf(total / (float)(is_q ? qn : kn) + a.eps);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = x[j] * inv * w8[j];
    }
    if (a.inv_freq) {
      if (a.half_split) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float other = __shfl(x[j], mate & (kWave - 1), kWave);
          if (turns) {
            const float c = cs_tab[ang + j], sn = low ? -sn_tab[ang + j] : sn_tab[ang + j];
            x[j] = SUMS == RUN_LANES || low ? fmaf(x[j], c, other * sn) : fmaf(other, sn, x[j] * c);
          }
        }
      } else if (turns) {
#pragma unroll
        for (int j = 0; j < 8; j += 2) {
          const float lo = x[j], hi = x[j + 1], c = cs_tab[ang + j / 2], sn = sn_tab[ang + j / 2];
          x[j] = fmaf(lo, c, -(hi * sn));
          x[j + 1] = fmaf(hi, c, lo * sn);
        }
      }
    }
    if (live) {
      if (is_q) {
        if (a.temp_on) {
#pragma unroll
          for (int j = 0; j < 8; ++j) x[j] *= temp;
        }
        T* q = (T*)a.q_out + ((size_t)t * a.nh + h) * a.maps * a.hd + li * 8;
        if (a.maps == 1) {
          store8(q, x);
        } else {                                         // the map's own row of the head's width, zeros in the other maps' rows
          const float zero[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
          for (int mm = 0; mm < a.maps; ++mm) store8(q + (size_t)mm * a.hd, mm == mp ? x : zero);
        }
      } else if (slot >= 0) {
        store8((T*)a.k_cache + (((size_t)page * a.nkv + (h - a.nh)) * a.page_size + off) * a.hd + li * 8, x);
      }
    }
  }
  if (slot < 0 || a.values_apart || (a.values_beside && !values_only)) return;
  const int v_part = a.values_beside ? 0 : blockIdx.y, v_parts = a.values_beside ? 1 : gridDim.y;
  for (int i = (v_part * blockDim.x + threadIdx.x) * 8; i < a.nkv * a.vd; i += v_parts * blockDim.x * 8) {
    float v[8];
    prep_gather8<T, TAPS>(a, t, v_at + i, v_col + i, C, v);
    prep_mix8<T>(a, t, i, v);
    const int g = i / a.vd, d = i % a.vd;
    T* dst = (T*)a.v_cache + (((size_t)page * a.nkv + g) * a.vd + d) * a.page_size + off;
#pragma unroll
    for (int j = 0; j < 8; ++j) dst[(size_t)j * a.page_size] = from_f32<T>(v[j]);
  }
}

// The convolution's tail after a step: the last taps - 1 projected rows of each entry's request
// (rows of this step where the entry brought enough, what the slot held before otherwise).  A
// thread takes one channel of one entry, reads everything it needs and only then writes.
template <typename T>
__global__ void conv_tail_kernel(const T* __restrict__ proj, int stride, int q_off, int k_off, int v_off, int qn, int kn,
                                 int vn, int taps, float* __restrict__ tail, const int* __restrict__ state_slots,
                                 const int* __restrict__ cu_tokens) {
  const int e = blockIdx.y;
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  const int C = qn + kn + vn;
  if (c >= C) return;
  const int col = c < qn ? q_off + c : c < qn + kn ? k_off + (c - qn) : v_off + (c - qn - kn);
  const int first = cu_tokens[e], len = cu_tokens[e + 1] - first;
  float* mine = tail + (size_t)state_slots[e] * (taps - 1) * C + c;
  float keep[kPrepMaxTaps];
  for (int s = 0; s < taps - 1; ++s) {
    const int li = len - (taps - 1) + s;               // the row that ends up in place s
    keep[s] = li >= 0 ? to_f32<T>(proj[(size_t)(first + li) * stride + col]) : mine[(size_t)(taps - 1 + li) * C];
  }
  for (int s = 0; s < taps - 1; ++s) mine[(size_t)s * C] = keep[s];
}

// proj [T, stride] of `dtype`; q at columns q_off.., k at k_off.., v at v_off.. (v_off < 0: values
// are the unnormed keys, vd must equal hd).  conv_w float [channels, taps] (taps 0: none), tail float
// [slots, taps - 1, channels].  norm_mode 0 none / 1 per head (weights [hd]) / 2 whole projection
// (weights [nh*hd], [nkv*hd]).  inv_freq float [rotary_dim / 2] or null.  Caches K [pages, nkv,
// page_size, hd], V [pages, nkv, vd, page_size]; slot_mapping null or -1: nothing is stored.
// bias float [q + k + v channels] or null (only without a convolution); temp_on: q times
// 1 + temp_scale ln(floor((pos + 1) / temp_floor) + 1); maps > 1: hd is the width of a head's maps
// together, rotary_dim <= hd / maps, and q_out is [T, nh * maps * hd].  v_other (of `dtype`, or null): rows of
// v_other_stride elements whose columns v_other_off .. hold another layer's values: what is stored is
// (1 - v_mix) v + v_mix v_other.
SHARPI_EXPORT int sharpi_qk_prep(const void* proj, int dtype, int stride, int q_off, int k_off, int v_off, int n_tokens,
                                 int n_entries, int nh, int nkv, int hd, int vd, const float* conv_w, int taps, float* tail,
                                 const int* state_slots, const int* entry_of_token, const int* cu_tokens,
                                 const int* positions, int norm_mode, const float* q_norm_w, const float* k_norm_w,
                                 float eps, const float* inv_freq, int rotary_dim, int half_split, float magnitude,
                                 void* q_out, void* k_cache, void* v_cache, const int* slot_mapping, int page_size,
                                 int update_tail, const float* bias, int temp_on, float temp_floor, float temp_scale,
                                 int maps, const void* v_other, int v_other_stride, int v_other_off, float v_mix,
                                 hipStream_t stream) {
  if (n_tokens <= 0) return SHARPI_OK;
  if (v_other && (v_other_off < 0 || v_other_off + nkv * vd > v_other_stride)) return SHARPI_ERR_ARG;
  if (maps < 1 || hd % (2 * maps) || rotary_dim > hd / maps) return SHARPI_ERR_ARG;
  if ((bias && taps > 0) || (temp_on && !(temp_floor > 0.f))) return SHARPI_ERR_ARG;
  if (nh <= 0 || nkv <= 0 || hd <= 0 || hd % 2 || vd <= 0 || nh + nkv > kPrepMaxHeads) return SHARPI_ERR_ARG;
  if (taps < 0 || taps == 1 || taps > kPrepMaxTaps || (taps > 0 && (!conv_w || !tail || !state_slots || !cu_tokens || !entry_of_token)))
    return SHARPI_ERR_ARG;
  if (norm_mode < 0 || norm_mode > 2 || (norm_mode && (!q_norm_w || !k_norm_w))) return SHARPI_ERR_ARG;
  if (rotary_dim < 0 || rotary_dim % 2 || rotary_dim > hd || (rotary_dim > 0 && !inv_freq)) return SHARPI_ERR_ARG;
  if (v_off < 0 && vd != hd) return SHARPI_ERR_ARG;
  if (slot_mapping && (!k_cache || !v_cache || page_size <= 0)) return SHARPI_ERR_ARG;
  const int qn = nh * hd, kn = nkv * hd, vn = v_off >= 0 ? nkv * vd : 0;
  const size_t lds = (size_t)(qn + kn + vn) * sizeof(float);
  if (lds > 60 * 1024) return SHARPI_ERR_ARG;
  const int parts = (n_tokens <= kPrepSplitTokens && nkv > 1 && nkv <= 65535 && nh % nkv == 0) ? nkv : 1;
  auto at16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 32 == 0; };
  const int sd = hd / maps;
  if (rotary_dim / 2 > kPrepMaxTurns) return SHARPI_ERR_ARG;
  const bool wide = sd % 8 == 0 && vd % 8 == 0 && stride % 8 == 0 && q_off % 8 == 0 && k_off % 8 == 0 && (v_off < 0 || v_off % 8 == 0) &&
                    at16(proj) && at16(q_out) && at16(k_cache) && at16(tail) && at16(bias);
  const bool other_wide = !v_other || (at16(v_other) && v_other_stride % 8 == 0 && v_other_off % 8 == 0);
  const int by8 = wide && (half_split || rotary_dim == 0) && rotary_dim % 16 == 0;
  const bool taps4 = taps == 4 && at16(conv_w);
  const int lanes = hd <= 64 ? (hd <= 8 ? 1 : hd <= 16 ? 2 : hd <= 32 ? 4 : 8) : hd <= 128 ? 16 : hd <= 256 ? 32 : 64;
  const int items = (nh + nkv) * lanes;
  const bool much = (long)n_tokens * items > kRunMuch;
  // a thread for every run where a block can have them; of a few tokens 256 a block, or the launch would leave the chip empty (a
  // norm over the projection aside, whose sums need them together)
  const bool together = items <= kRunMaxThreads && (norm_mode == NORM_WHOLE || (n_tokens > kPrepSplitTokens && !(much && items > kRunFullBlock)));
  const bool chains = taps > 4 || (taps > 0 && !taps4 && !by8 && n_tokens > kPrepBesideFewTaps);
  const bool convolved = taps == 0 || (!much && (!chains || (n_tokens <= kRunManyTaps && items > (n_tokens <= kPrepBesideFewTaps ? kRunNarrow : kRunHalfBlock))));
  const bool by_runs = wide && other_wide && convolved && rotary_dim % (half_split ? 16 : 8) == 0 && hd <= 512 && at16(q_norm_w) && at16(k_norm_w) &&
                       (norm_mode != NORM_WHOLE || together);
  // (a step stores all its tokens or, without slots, none)
  const int beside_up_to = taps == 0 || (taps4 && v_off >= 0) ? kPrepSplitTokens : taps <= 4 && v_off >= 0 && (by8 || by_runs) ? kPrepBesideFewTaps : n_tokens;
  const bool v_apart = wide && other_wide && n_tokens > beside_up_to && slot_mapping != nullptr;
  const int tiles = v_apart ? value_tiles(n_tokens, nkv * vd) : 0;
  PrepArgs a{proj, stride, q_off, k_off, v_off, nh, nkv, hd, vd, conv_w, taps, tail, state_slots, entry_of_token,
             cu_tokens, positions, norm_mode, q_norm_w, k_norm_w, eps, rotary_dim > 0 ? inv_freq : nullptr, rotary_dim,
             half_split, magnitude, q_out, k_cache, v_cache, slot_mapping, page_size, parts, bias, temp_on, temp_floor,
             temp_scale, maps, v_other, v_other_stride, v_other_off, v_mix, v_apart, 0, n_tokens, by8};
  if (dtype != DT_F32 && dtype != DT_BF16) return SHARPI_ERR_ARG;
  // (no gather by eights in a block that takes an element a thread: the form without one, whose registers leave room for more waves)
  const int form = taps == 0 || !(by_runs || by8 || v_apart) ? 0 : taps4 ? 4 : -1;
#define PREP_BY_TAPS(GO, ...)                                               \
  do {                                                                      \
    if (dtype == DT_F32) {                                                  \
      if (form == 0) GO(float, 0, ##__VA_ARGS__); else if (form == 4) GO(float, 4, ##__VA_ARGS__); else GO(float, -1, ##__VA_ARGS__);    \
    } else {                                                                \
      if (form == 0) GO(bf16_t, 0, ##__VA_ARGS__); else if (form == 4) GO(bf16_t, 4, ##__VA_ARGS__); else GO(bf16_t, -1, ##__VA_ARGS__); \
    }                                                                       \
  } while (0)
  if (by_runs) {
    const int threads = together ? max(kValueThreads, ceil_div(items, kWave) * kWave) : kPrepThreads;
    // not together: a block a turn of few tokens; of more two turns or so a block, of many four, to share the angles
    const int turns = ceil_div(items, threads), y = ceil_div(turns, n_tokens <= kPrepSplitTokens ? 1 : n_tokens <= 4 * kPrepSplitTokens ? 2 : 4);
    a.values_beside = !v_apart && slot_mapping != nullptr;
    const dim3 rgrid(a.values_beside ? 8 * ceil_div(n_tokens, 8) : n_tokens + ceil_div(tiles, y), y + a.values_beside);
    const size_t row_lds = norm_mode == NORM_WHOLE ? (size_t)(qn + kn) * sizeof(float) : 0;
    const bool plain = (half_split || rotary_dim == 0) && taps == 0 && maps == 1 && v_off >= 0;
#define RUN_GO(T, TAPSV, SUMSV) qk_prep_run_kernel<T, TAPSV, SUMSV><<<rgrid, threads, row_lds, stream>>>(a, __builtin_ctz(lanes))
    if (norm_mode == NORM_WHOLE) PREP_BY_TAPS(RUN_GO, RUN_WHOLE);
    else if (!plain) PREP_BY_TAPS(RUN_GO, RUN_ROW);
    else if (dtype == DT_F32) RUN_GO(float, 0, RUN_LANES);
    else RUN_GO(bf16_t, 0, RUN_LANES);
#undef RUN_GO
    SHARPI_CHECK_LAUNCH();
  } else {
    dim3 pgrid(n_tokens + tiles, parts);               // (values apart: one part)
    const size_t row_lds = v_apart ? (size_t)(qn + kn) * sizeof(float) : lds, tile_lds = dtype == DT_F32 ? kValueLds<float> : kValueLds<bf16_t>;
    const size_t prep_lds = v_apart && row_lds < tile_lds ? tile_lds : row_lds;
#define PREP_GO(T, TAPSV) qk_prep_kernel<T, TAPSV><<<pgrid, kPrepThreads, prep_lds, stream>>>(a)
    PREP_BY_TAPS(PREP_GO);
#undef PREP_GO
    SHARPI_CHECK_LAUNCH();
  }
#undef PREP_BY_TAPS
  if (taps > 0 && update_tail) {
    dim3 grid(ceil_div(qn + kn + vn, 256), n_entries);
    if (dtype == DT_F32)
      conv_tail_kernel<float><<<grid, 256, 0, stream>>>((const float*)proj, stride, q_off, k_off, v_off, qn, kn, vn, taps,
                                                        tail, state_slots, cu_tokens);
    else
      conv_tail_kernel<bf16_t><<<grid, 256, 0, stream>>>((const bf16_t*)proj, stride, q_off, k_off, v_off, qn, kn, vn, taps,
                                                         tail, state_slots, cu_tokens);
    SHARPI_CHECK_LAUNCH();
  }
  return SHARPI_OK;
}
