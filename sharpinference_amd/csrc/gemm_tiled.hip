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
// 573 x 2,048 x 2,048: 270 -> 74 us; 7 x 32,000 x 2,048: 265 -> 46 us.  Many rows have a kernel of their own below, in groups and outside of them.
#include "common.h"
#include "lds_loads.h"

#include <type_traits>

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

// The group (found[0], -1: none) and first row (found[1]) of tile number `tile`: tiles of BM rows are numbered group by group.
template <int BM>
__device__ __forceinline__ void find_tile(int tile, const int* __restrict__ group_offsets, int groups, int* found) {
  const int lane = threadIdx.x & (kWave - 1);
  if (threadIdx.x == 0) found[0] = -1;
  __syncthreads();
  if (threadIdx.x < kWave) {
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
    find_tile<BM>(tile, group_offsets, groups, found);
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

// The product of 32-bit rows where there are many (in groups: between them): a block takes up to 64 rows (of a group) against 128
// weight rows.  Every wave has all the rows (in steps of 16: a tile is multiplied no higher than its rows go) and 32 of the
// columns, so that nothing is done for rows that are not there, which in tiles of 64 x 64, two waves high, was a third
// of the products at 54 rows a group.  Both operands go straight into LDS, 32 of k a stage (whole 128-byte lines, their 16-byte
// pieces XORed with row bits), two stages ahead; the LDS reads of half a stage run beside the products of the half before.
// Two blocks stay on a compute unit.  The sums are the tiled kernel's, bit for bit.
// 64 experts, six picks, us before and now: gate|up 2,816 x 2,048, 300 tokens 380 -> 337, 573 tokens 576 -> 438 (91 TFLOP/s of the rows
// there are), 1,600 tokens 1,213 -> 953 (116); down 2,048 x 1,408, 573 tokens 300 -> 228; 32 experts of 4,096 x 4,096, 573 tokens,
// four picks 1,054 -> 768.  Weights that one tile alone reads come with the streaming hint: 300 tokens 331 -> 311.  What is left: the last round of blocks, and tiles whose rows end 1 to 15 short of a step.
constexpr int kRowsBM = 64, kRowsBN = 128, kRowsRing = 3, kRowsWaves = 4;
constexpr int kRowsA = kRowsBM * BK * 4, kRowsStage = kRowsA + kRowsBN * BK * 4;      // LDS bytes: A's rows, then W's

__device__ __forceinline__ int rows_piece(int row, int piece) { return piece ^ ((row >> 1) & 7); }

// STREAM: the weights with the streaming hint.
template <int RM, bool STREAM>
__device__ __forceinline__ void float_rows_tile(const float* __restrict__ A, uint32_t a_bytes, const float* __restrict__ W,
                                                float* __restrict__ C, int N, int K, const int* __restrict__ a_rows, int m0, int row_end,
                                                int n0, const char* smem) {
  constexpr int RN = 2, WL = kRowsBN / 8 / kRowsWaves, AL = (2 * RM + kRowsWaves - 1) / kRowsWaves, LOADS = WL + AL;
  const int lane = threadIdx.x & (kWave - 1), wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // a load brings 8 rows of a stage, lane l the row l / 8 at place l % 8; rows outside are read as the last one inside
  uint32_t w_off[WL], a_off[AL];
  int a_load[AL];
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int row = (wid * WL + i) * 8 + (lane >> 3);
    w_off[i] = (uint32_t)min(n0 + row, N - 1) * (uint32_t)K * 4 + rows_piece(row, lane & 7) * 16;
  }
#pragma unroll
  for (int i = 0; i < AL; ++i) {
    a_load[i] = min(wid * AL + i, 2 * RM - 1);
    const int row = a_load[i] * 8 + (lane >> 3), m = min(m0 + row, row_end - 1);
    a_off[i] = (uint32_t)(a_rows ? a_rows[m] : m) * (uint32_t)K * 4 + rows_piece(row, lane & 7) * 16;
  }
  // waited for here: the compiler's own waits must not fall among the loads below, which it does not know of
#pragma unroll
  for (int i = 0; i < AL; ++i) asm volatile("" : "+v"(a_off[i]));
  const u32x4 wb = buffer_of(W, (uint32_t)N * (uint32_t)K * 4), ab = buffer_of(A, a_bytes);
  const uint32_t lds0 = lds_address(smem);
  const int stages = K / BK;
  auto send = [&](int s, int place) {
#pragma unroll
    for (int i = 0; i < AL; ++i) load_to_lds(ab, a_off[i], s * (BK * 4), lds0 + place * kRowsStage + a_load[i] * 1024);
#pragma unroll
    for (int i = 0; i < WL; ++i) load_to_lds<STREAM>(wb, w_off[i], s * (BK * 4), lds0 + place * kRowsStage + kRowsA + (wid * WL + i) * 1024);
  };

  f32x4 acc[RM][RN][kChains];
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
      for (int c = 0; c < kChains; ++c) acc[i][j][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int fr = lane & 15, fg = lane >> 4;
  int at[2];                                    // this lane's piece of a half stage, in row fr
#pragma unroll
  for (int h = 0; h < 2; ++h) at[h] = fr * 128 + rows_piece(fr, h * 4 + fg) * 16;
  f32x4 a[2][RM], w[2][RN];
  auto read = [&](auto half_tag, int place) {
    constexpr int h = decltype(half_tag)::value;
    const char* p = smem + place * kRowsStage + at[h];
#pragma unroll
    for (int i = 0; i < RM; ++i) a[h][i] = *reinterpret_cast<const f32x4*>(p + i * 2048);
#pragma unroll
    for (int j = 0; j < RN; ++j) w[h][j] = *reinterpret_cast<const f32x4*>(p + kRowsA + (wid * RN + j) * 2048);
  };
  auto products = [&](auto half_tag) {
    constexpr int h = decltype(half_tag)::value;
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j) {
          f32x4& c = acc[i][j][h * 2 + s / 2];
          c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[h][i][s], w[h][j][s], c, 0, 0, 0);
        }
  };
  using Half0 = std::integral_constant<int, 0>;
  using Half1 = std::integral_constant<int, 1>;
  send(0, 0);
  if (stages > 1) send(1, 1);
  // a stage is there when the wave's own loads of it are (those of the next one may be under way) and everyone has said so; the place
  // of the stage before is free then
  if (stages > 1) lds_loads_wait<LOADS>();
  else lds_loads_wait<0>();
  __syncthreads();
  read(Half0{}, 0);
  int place = 0, ahead = 2;
  for (int s = 0; s + 1 < stages; ++s) {
    read(Half1{}, place);
    if (s + 2 < stages) send(s + 2, ahead);
    ahead = ahead + 1 == kRowsRing ? 0 : ahead + 1;
    products(Half0{});
    place = place + 1 == kRowsRing ? 0 : place + 1;
    if (s + 2 < stages) lds_loads_wait<LOADS>();
    else lds_loads_wait<0>();
    __syncthreads();
    read(Half0{}, place);
    products(Half1{});
  }
  read(Half1{}, place);
  products(Half0{});
  products(Half1{});
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int m = m0 + 16 * i + fg * 4 + v;
      if (m >= row_end) continue;
#pragma unroll
      for (int j = 0; j < RN; ++j) {
        const int n = n0 + (wid * RN + j) * 16 + fr;
        if (n < N) C[(size_t)m * N + n] = (acc[i][j][0][v] + acc[i][j][1][v]) + (acc[i][j][2][v] + acc[i][j][3][v]);
      }
    }
}

__global__ __launch_bounds__(kRowsWaves* kWave, 2) void gemm_float_rows_kernel(const float* __restrict__ A, uint32_t a_bytes,
                                                                               const float* __restrict__ W, float* __restrict__ C, int M,
                                                                               int N, int K, const int* __restrict__ a_rows,
                                                                               const int* __restrict__ group_offsets, int groups) {
  __shared__ __attribute__((aligned(1024))) char smem[kRowsRing * kRowsStage];
  __shared__ int found[2];
  const int columns = (N + kRowsBN - 1) / kRowsBN;
  const int tile = blockIdx.x / columns, n0 = (blockIdx.x - tile * columns) * kRowsBN;
  int m0 = tile * kRowsBM, row_end = M;
  bool alone = M <= kRowsBM;                       // no other tile reads these weights
  if (group_offsets) {
    find_tile<kRowsBM>(tile, group_offsets, groups, found);
    const int e = __builtin_amdgcn_readfirstlane(found[0]);
    if (e < 0) return;
    m0 = __builtin_amdgcn_readfirstlane(found[1]);
    row_end = group_offsets[e + 1];
    alone = row_end - group_offsets[e] <= kRowsBM;
    W += (size_t)e * N * K;
  }
  const int rows = min(row_end - m0, kRowsBM);
#define ROWS_TILE(RMV)                                                                                             \
  do {                                                                                                             \
    if (alone) float_rows_tile<RMV, true>(A, a_bytes, W, C, N, K, a_rows, m0, row_end, n0, smem);                   \
    else float_rows_tile<RMV, false>(A, a_bytes, W, C, N, K, a_rows, m0, row_end, n0, smem);                        \
  } while (0)
  if (rows <= 16) ROWS_TILE(1);
  else if (rows <= 32) ROWS_TILE(2);
  else if (rows <= 48) ROWS_TILE(3);
  else ROWS_TILE(4);
#undef ROWS_TILE
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
template <typename F> static int tiled_height(int rows, int N, const F& tiles) {
  int bm = rows <= 16 ? 16 : rows <= 32 ? 32 : 64;
  while (bm > 16 && (int64_t)tiles(bm) * ceil_div(N, BN) < 384) bm /= 2;
  return bm;
}

// Plain products of 32-bit rows: the kernel of many rows (64 x 128 a block) or the tiled one.  Beyond 32 rows the former only where the
// latter would take tiles of 64 rows (lower ones are faster, 573 x 2,048 68 and 72 us, 350 x 2,816 55 and 72, but for 33 to 48 rows of 16,384
// columns, 62 and 57) and its rounds of the chip take less time.  us a round at K = 2,048, two blocks a unit here: 123; up to one a unit 73; a few
// blocks behind whole rounds 40, more of them as much as a round.  Three blocks a unit there: 117; up to 15/8 a unit 78, up to two 90.
// Tiled / this: 573 x 2,816 85 / 72; 2,048 x 2,048 195 / 128, x 3,072 230 / 243 (left); 400 x 8,192 194 / 125; 1,024 x 5,120 197 / 242 (left);
// 800 x 5,120 193 / 139.  Up to 32 rows from half a block a unit on: 7 x 24,576 50 / 40, x 32,000 58 / 58, 32 x 32,000 62 / 61, 7 x 16,384 40 / 35.
// Of 1,665 sizes (1 to 2,048 rows, 512 to 65,536 columns, K 512 to 8,192, weights from memory) 537 are taken, none slower by more
// than 1 %, 1.25 times as fast in the mean.
static bool plain_goes_to_rows(int M, int N, int units) {
  const int64_t here = (int64_t)ceil_div(M, kRowsBM) * ceil_div(N, kRowsBN);
  if (M <= 32) return 2 * here >= units;
  const auto tiles = [&](int bm) { return ceil_div(M, bm); };
  if (tiled_height(M, N, tiles) < 64) return false;
  const int64_t there = (int64_t)tiles(64) * ceil_div(N, BN);
  const int64_t here_left = here % (2 * units), there_left = there % (3 * units);
  int64_t here_us = here / (2 * units) * 123, there_us = there / (3 * units) * 117;
  if (here_left) here_us += here <= units ? 73 : here_us && 16 * here_left <= units ? 40 : 123;
  if (there_left) there_us += 8 * there_left <= 15 * units ? 78 : there_left <= 2 * units ? 90 : 117;
  return here_us < there_us;
}

template <typename T, typename TO>
static int run_tiled(const T* A, const T* W, TO* C, int M, int N, int K, const int* a_rows, const int* go, int groups, int a_total, hipStream_t stream) {
  const int rows = go ? ceil_div(M, min(M, groups)) : M;
  auto tiles = [&](int bm) { return go ? M / bm + min(M, groups) : ceil_div(M, bm); };
  if constexpr (std::is_same<T, float>::value && std::is_same<TO, float>::value) {
    // Groups of more than 24 rows (their mean) that make 384 blocks or more (one and a half a unit).  us, tiled / this, gate|up of 64
    // experts at 19 rows an expert: 315 / 318; 28: 380 / 337; 16 experts of 36 rows, 528 blocks: 120 / 120; 4 of 150 rows and 256
    // columns, 16 blocks: 12 / 21.  Offsets are of 32 bits: operands of 4 GB and more take the tiled kernel, as odd k do.
    const int64_t blocks = (int64_t)tiles(kRowsBM) * ceil_div(N, kRowsBN);
    const bool fits = K % BK == 0 && (reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(W)) % 16 == 0 &&
                      (int64_t)a_total * K * 4 < (1LL << 32) && (int64_t)N * K * 4 < (1LL << 32) && blocks <= 0x7fffffff;
    const bool here = go ? rows > 24 && blocks >= 384 : plain_goes_to_rows(M, N, compute_units());
    if (fits && here) {
      gemm_float_rows_kernel<<<(unsigned)blocks, kRowsWaves * kWave, 0, stream>>>(A, (uint32_t)((int64_t)a_total * K * 4), W, C, M, N, K,
                                                                                  a_rows, go, groups);
      SHARPI_CHECK_LAUNCH();
      return SHARPI_OK;
    }
  }
  const int bm = tiled_height(rows, N, tiles);
  if ((int64_t)tiles(bm) * ceil_div(N, BN) > 0x7fffffff) return SHARPI_ERR_ARG;
  if (bm == 16) launch_tiled<T, TO, 1, 1, 1>(A, W, C, M, N, K, a_rows, go, groups, tiles(16), stream);
  else if (bm == 32) launch_tiled<T, TO, 1, 2, 1>(A, W, C, M, N, K, a_rows, go, groups, tiles(32), stream);
  else launch_tiled<T, TO, 2, 2, 2>(A, W, C, M, N, K, a_rows, go, groups, tiles(64), stream);
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}

// Whether a plain product of 32-bit rows goes to the kernel of many rows on a chip of `units` units (what the choice is, for tests of it).
SHARPI_EXPORT int sharpi_gemm_tiled_many_rows(int M, int N, int units) {
  return M > 0 && N > 0 && units > 0 && plain_goes_to_rows(M, N, units);
}

// dtype: storage of A and W; out_dtype: storage of C.
// a_total: rows of A.  groups == 0: plain product of M rows. groups > 0: grouped, M = rows of all groups together.
SHARPI_EXPORT int sharpi_gemm_tiled(const void* A, const void* W, void* C, int dtype, int out_dtype, int M, int N,
                                    int K, const int* a_rows, const int* group_offsets, int groups, int a_total,
                                    hipStream_t stream) {
  if (M <= 0) return SHARPI_OK;
  if (N <= 0 || K <= 0 || groups < 0 || groups > 65535) return SHARPI_ERR_ARG;
  if (groups > 0 && group_offsets == nullptr) return SHARPI_ERR_ARG;
  if (ceil_div(M, 64) > 65535) return SHARPI_ERR_ARG;
  const int* go = groups > 0 ? group_offsets : nullptr;
  if (dtype == DT_F32 && out_dtype == DT_F32)
    return run_tiled<float, float>((const float*)A, (const float*)W, (float*)C, M, N, K, a_rows, go, groups, a_total, stream);
  if (dtype == DT_BF16 && out_dtype == DT_BF16)
    return run_tiled<bf16_t, bf16_t>((const bf16_t*)A, (const bf16_t*)W, (bf16_t*)C, M, N, K, a_rows, go, groups, a_total, stream);
  if (dtype == DT_BF16 && out_dtype == DT_F32)
    return run_tiled<bf16_t, float>((const bf16_t*)A, (const bf16_t*)W, (float*)C, M, N, K, a_rows, go, groups, a_total, stream);
  return SHARPI_ERR_ARG;
}
