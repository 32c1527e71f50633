// C[M, N] = A[M, K] * W[N, K]^T in 32 bits, on the float matrix instruction (no reduced precision).
//
// The 32-bit path's matrix product, also the fallback for sizes the bfloat16 kernels refuse.
// Every output element is four chains of float fused multiply-adds, added at the end (their roundings are
// half of one chain's), in an order of k that depends on k alone (of 32 k, chain 2 h + c takes places i, i + 4,
// i + 8, i + 12 of sixteen number h, i = 2 c and 2 c + 1: a lane reads four neighbouring k at once), so a row's
// result depends neither on how many other rows are in the batch nor on where the row sits in it nor on the
// tile's height.  The grouped form runs E products at
// once: rows [off[e], off[e+1]) of the (expert-sorted) row list use W[e]; A's rows may be gathered
// through `a_rows`.
//
// Bound: the float matrix instruction (151 TFLOP/s in a large product of the library here, twice
// what unpacked vector FMAs can reach) for many rows, the weights' bytes for few.  A block makes a
// tile of BM rows x 64 columns with 4 waves; k is staged 32 at a time through two LDS buffers (rows
// of 36 floats: 16-byte reads without bank conflicts), the next two pieces in registers meanwhile.
// 573 rows, 6 of 64 experts each, 2,048 wide, gate|up of 2,816 columns: 1,750 -> 506 us (weights alone 214, products
// 263); 573 x 2,048 x 2,048: 270 -> 74 us; 7 x 32,000 x 2,048: 265 -> 46 us.
#include "common.h"

using f32x4 = __attribute__((__vector_size__(4 * sizeof(float)))) float;

constexpr int BN = 64, BK = 32, LDK = BK + 4;
constexpr int kChains = 4;
constexpr int kTiledThreads = 256;

// four consecutive elements at k; VEC: whole fours, aligned.  Places beyond the row are read inside it: `mask4` clears
// them when the values are used (a select beside the load would wait for it at once).
template <typename T, bool VEC>
__device__ __forceinline__ f32x4 load4(const T* __restrict__ row, int k, int K) {
  f32x4 v;
  if constexpr (VEC) {
    const int kc = min(k, K - 4);
    if constexpr (sizeof(T) == 4) {
      v = *reinterpret_cast<const f32x4*>(row + kc);
    } else {
      const uint2 u = *reinterpret_cast<const uint2*>(row + kc);
      v[0] = bf16_bits_to_f32(u.x & 0xffffu);
      v[1] = bf16_bits_to_f32(u.x >> 16);
      v[2] = bf16_bits_to_f32(u.y & 0xffffu);
      v[3] = bf16_bits_to_f32(u.y >> 16);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = to_f32<T>(row[min(k + j, K - 1)]);
  }
  return v;
}
__device__ __forceinline__ f32x4 mask4(f32x4 v, int k, int K) {
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = k + j < K ? v[j] : 0.f;
  return v;
}

// Waves lie WR x (4 / WR) over the tile; a wave has RM x RN squares of 16 x 16: BM = WR * RM * 16, 64 = (4 / WR) * RN * 16.
template <typename T, typename TO, int WR, int RM, int RN, bool VEC>
__global__ __launch_bounds__(kTiledThreads) void gemm_tiled_kernel(const T* __restrict__ A, const T* __restrict__ W,
                                                                   TO* __restrict__ C, int M, int N, int K,
                                                                   const int* __restrict__ a_rows,
                                                                   const int* __restrict__ group_offsets, int groups) {
  constexpr int BM = WR * RM * 16;
  static_assert((4 / WR) * RN * 16 == BN, "the waves cover the tile's columns");
  __shared__ float As[2][BM * LDK];
  __shared__ float Ws[2][BN * LDK];
  __shared__ int found[2];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wid = tid >> 6;
  const int columns = (N + BN - 1) / BN;
  const int tile = blockIdx.x / columns, n0 = (blockIdx.x - tile * columns) * BN;
  int m0 = tile * BM, row_end = M;
  if (group_offsets) {
    // this block's group and tile: tiles are numbered group by group
    if (tid == 0) found[0] = -1;
    __syncthreads();
    if (wid == 0) {
      int before = 0;
      for (int e0 = 0; e0 < groups; e0 += kWave) {
        const int e = e0 + lane;
        const int lo = e < groups ? group_offsets[e] : 0;
        const int n = e < groups ? (group_offsets[e + 1] - lo + BM - 1) / BM : 0;
        int upto = n;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
          const int x = __shfl_up(upto, o, kWave);
          if (lane >= o) upto += x;
        }
        const int first = before + upto - n;
        if (tile >= first && tile < first + n) {
          found[0] = e;
          found[1] = lo + (tile - first) * BM;
        }
        before += __shfl(upto, kWave - 1, kWave);
        if (before > tile) break;
      }
    }
    __syncthreads();
    const int e = found[0];
    if (e < 0) return;
    m0 = found[1];
    row_end = group_offsets[e + 1];
    W += (size_t)e * N * K;
  }

  // Loader: thread tid brings the four k at lk of rows lr, lr + 32, ...; rows outside are read as the last one inside
  // (what comes of them is not stored).
  const int lr = tid >> 3, lk = (tid & 7) * 4;
  constexpr int AL = BM >= 32 ? BM / 32 : 1;
  const T* a_src[AL];
  const T* w_src[2];
#pragma unroll
  for (int i = 0; i < AL; ++i) {
    const int m = min(m0 + (BM >= 32 ? lr + 32 * i : lr & (BM - 1)), row_end - 1);
    a_src[i] = A + (size_t)(a_rows ? a_rows[m] : m) * K;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) w_src[i] = W + (size_t)min(n0 + lr + 32 * i, N - 1) * K;

  struct Pieces {
    f32x4 a[AL], w[2];
  };
  auto fetch = [&](Pieces& r, int k0) {
#pragma unroll
    for (int i = 0; i < AL; ++i) r.a[i] = load4<T, VEC>(a_src[i], k0 + lk, K);
#pragma unroll
    for (int i = 0; i < 2; ++i) r.w[i] = load4<T, VEC>(w_src[i], k0 + lk, K);
  };
  auto stage = [&](int buf, const Pieces& r, int k0) {
#pragma unroll
    for (int i = 0; i < AL; ++i)
      if (BM >= 32 || lr < BM) *reinterpret_cast<f32x4*>(&As[buf][(lr + 32 * i) * LDK + lk]) = mask4(r.a[i], k0 + lk, K);
#pragma unroll
    for (int i = 0; i < 2; ++i) *reinterpret_cast<f32x4*>(&Ws[buf][(lr + 32 * i) * LDK + lk]) = mask4(r.w[i], k0 + lk, K);
  };

  const int wr = (wid % WR) * RM * 16, wc = (wid / WR) * RN * 16;
  const int fr = lane & 15, fk = (lane >> 4) * 4;
  f32x4 acc[RM][RN][kChains];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
      for (int c = 0; c < kChains; ++c) acc[i][j][c] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto products = [&](int buf) {
#pragma unroll
    for (int kk = 0; kk < BK; kk += 16) {
      f32x4 a[RM], w[RN];
#pragma unroll
      for (int i = 0; i < RM; ++i) a[i] = *reinterpret_cast<const f32x4*>(&As[buf][(wr + 16 * i + fr) * LDK + kk + fk]);
#pragma unroll
      for (int j = 0; j < RN; ++j) w[j] = *reinterpret_cast<const f32x4*>(&Ws[buf][(wc + 16 * j + fr) * LDK + kk + fk]);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < RM; ++i)
#pragma unroll
          for (int j = 0; j < RN; ++j) {
            f32x4& c = acc[i][j][kk / 16 * 2 + s / 2];
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][s], w[j][s], c, 0, 0, 0);
          }
    }
  };
  // Two pieces of k are on their way while one is multiplied; a buffer is written behind the barrier that ends its
  // last reading.  Pieces beyond K are read clamped and never multiplied.
  Pieces even, odd;
  fetch(even, 0);
  fetch(odd, BK);
  stage(0, even, 0);
  __syncthreads();
  for (int k0 = 0;; k0 += 2 * BK) {
    fetch(even, k0 + 2 * BK);
    products(0);
    if (k0 + BK >= K) break;
    stage(1, odd, k0 + BK);
    __syncthreads();
    fetch(odd, k0 + 3 * BK);
    products(1);
    if (k0 + 2 * BK >= K) break;
    stage(0, even, k0 + 2 * BK);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int m = m0 + wr + 16 * i + (lane >> 4) * 4 + v;
      if (m >= row_end) continue;
#pragma unroll
      for (int j = 0; j < RN; ++j) {
        const int n = n0 + wc + 16 * j + fr;
        if (n < N) C[(size_t)m * N + n] = from_f32<TO>((acc[i][j][0][v] + acc[i][j][1][v]) + (acc[i][j][2][v] + acc[i][j][3][v]));
      }
    }
}

template <typename T, typename TO, int WR, int RM, int RN>
static void launch_tiled(const T* A, const T* W, TO* C, int M, int N, int K, const int* a_rows, const int* go, int groups,
                         int row_tiles, hipStream_t stream) {
  const dim3 grid(ceil_div(N, BN) * row_tiles), block(kTiledThreads);
  // four k at once: whole fours in a row, rows and bases on multiples of a load's width
  const bool vec = K % 4 == 0 && ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(W)) % (4 * sizeof(T))) == 0;
  if (vec)
    gemm_tiled_kernel<T, TO, WR, RM, RN, true><<<grid, block, 0, stream>>>(A, W, C, M, N, K, a_rows, go, groups);
  else
    gemm_tiled_kernel<T, TO, WR, RM, RN, false><<<grid, block, 0, stream>>>(A, W, C, M, N, K, a_rows, go, groups);
}

// The tile's height: the smallest of 16, 32, 64 that holds the rows of a group (their mean: a group a little larger
// takes a second tile), halved while fewer than 384 blocks would start (a unit then waits on one block's loads).
// Microseconds at heights 16 / 32 / 64, K = 2,048: 7 rows x 2,048 columns 26 / 35 / 51; 300 x 2,048: 50 / 55 / 60
// (160 blocks of 64 rows); 573 x 2,048: 73 / 74 / 86 (288 blocks); 573 x 2,816: 99 / 89 / 84 (396); 2,048 x 8,192:
// 881 / 690 / 596; 64 experts, 2,816 columns, rows an expert 14: 305 / 329 / 473; 28: 497 / 394 / 483; 54: 787 / 601 / 506.
// 128 rows were no faster anywhere (96, 98, 603 us at the last three plain sizes).
template <typename T, typename TO>
static int run_tiled(const T* A, const T* W, TO* C, int M, int N, int K, const int* a_rows, const int* go, int groups, hipStream_t stream) {
  const int rows = go ? ceil_div(M, min(M, groups)) : M;
  auto tiles = [&](int bm) { return go ? M / bm + min(M, groups) : ceil_div(M, bm); };
  int bm = rows <= 16 ? 16 : rows <= 32 ? 32 : 64;
  while (bm > 16 && (int64_t)tiles(bm) * ceil_div(N, BN) < 384) bm /= 2;
  if ((int64_t)tiles(bm) * ceil_div(N, BN) > 0x7fffffff) return SHARPI_ERR_ARG;
  if (bm == 16) launch_tiled<T, TO, 1, 1, 1>(A, W, C, M, N, K, a_rows, go, groups, tiles(16), stream);
  else if (bm == 32) launch_tiled<T, TO, 1, 2, 1>(A, W, C, M, N, K, a_rows, go, groups, tiles(32), stream);
  else launch_tiled<T, TO, 2, 2, 2>(A, W, C, M, N, K, a_rows, go, groups, tiles(64), stream);
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}

// dtype: storage of A and W; out_dtype: storage of C.
// groups == 0: plain product of M rows. groups > 0: grouped, M = rows of all groups together.
SHARPI_EXPORT int sharpi_gemm_tiled(const void* A, const void* W, void* C, int dtype, int out_dtype, int M, int N,
                                    int K, const int* a_rows, const int* group_offsets, int groups,
                                    hipStream_t stream) {
  if (M <= 0) return SHARPI_OK;
  if (N <= 0 || K <= 0 || groups < 0 || groups > 65535) return SHARPI_ERR_ARG;
  if (groups > 0 && group_offsets == nullptr) return SHARPI_ERR_ARG;
  if (ceil_div(M, 64) > 65535) return SHARPI_ERR_ARG;
  const int* go = groups > 0 ? group_offsets : nullptr;
  if (dtype == DT_F32 && out_dtype == DT_F32)
    return run_tiled<float, float>((const float*)A, (const float*)W, (float*)C, M, N, K, a_rows, go, groups, stream);
  if (dtype == DT_BF16 && out_dtype == DT_BF16)
    return run_tiled<bf16_t, bf16_t>((const bf16_t*)A, (const bf16_t*)W, (bf16_t*)C, M, N, K, a_rows, go, groups, stream);
  if (dtype == DT_BF16 && out_dtype == DT_F32)
    return run_tiled<bf16_t, float>((const bf16_t*)A, (const bf16_t*)W, (float*)C, M, N, K, a_rows, go, groups, stream);
  return SHARPI_ERR_ARG;
}
