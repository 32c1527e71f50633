// One matrix times many rows (prompt-sized steps) with the activation behind it: act(g) * u with (g | u) = x[M, K] * W[N, K]^T, or relu(y)^2 of
// y = x W^T, of products rounded to bfloat16 (what a separate activation kernel would have read), on the grouped product's tiles
// (gemm_grouped_kernel.h).  act 0 and relu2 0: the product itself.
//
// Bound: what a unit reads from LDS and multiplies (tiles of 256 x 256: 1.37 PFLOP/s in whole rounds of the chip), and the last round:
// a block is one tile and stays alone on a unit, so that 2.5 rounds take as long as three.  Every output is one chain over k in ascending order
// however the rows are cut, and the caller cuts them where the rounds come out whole: tiles of 128 to 256 rows, all of one height.  No
// tickets and no plan as the grouped product has: the tiles are alike.  Blocks go to the dies round-robin; a die takes neighbouring tiles,
// kDenseColumns column blocks wide, so that its 32 units read the same few rows and weights through its L2 (8,192 x 5,120 x 5,120, 1, 2, 4,
// 8 and 16 wide: 396, 346, 334, 331, 339 us; 8,192 x 16,384 x 5,120: 1,075, 1,004, 1,002, 993, 1,042).
// us, the library's product and a kernel for the activation, and this: 3,000 x 2,816 x 2,048 50 -> 37, 1,664 x 2,816 x 2,048 32 -> 29,
// 908 x 10,240 x 1,408 46 -> 32, 1,225 x 8,192 x 2,048 48 -> 42, 5,216 x 2,816 x 2,816 73 -> 72.  In whole steps, beside kernels that leave
// other things in the caches: 3,000 x 2,816 x 2,048 59 -> 44, 1,900 x 8,192 x 2,048 with the squared relu 66 -> 57, 1,664 x 2,816 x 2,048 35 both ways.
#include "gemm_grouped_kernel.h"

constexpr int kDenseColumns = 4;       // column blocks side by side in a die's walk

template <int MT, bool ACT>
__global__ __launch_bounds__(GW* kWave, 2) void dense_gemm_kernel(const bf16_t* __restrict__ x, uint32_t x_bytes,
                                                                  const bf16_t* __restrict__ W, bf16_t* __restrict__ out, int M, int N,
                                                                  int K, int row_tiles, GatedAct act, int relu2) {
  __shared__ __attribute__((aligned(1024))) char smem[kGroupedLds];
  constexpr int kCols = ACT ? columns_of(kMaxNT) / 2 : columns_of(kMaxNT);
  const int nb = ((ACT ? N / 2 : N) + kCols - 1) / kCols;
  const int slots = gridDim.x, die = blockIdx.x % kXcds;
  const int slot = die * (slots / kXcds) + min(die, slots % kXcds) + blockIdx.x / kXcds;
  const int c0 = slot / (kDenseColumns * row_tiles) * kDenseColumns, left = slot - c0 * row_tiles, wide = min(kDenseColumns, nb - c0);
  const int row0 = left / wide * (MT * 32), row_end = min(M, row0 + MT * 32);
  int next = 0;
  grouped_tile<bf16_t, MT, kMaxNT, true, ACT, true>(x, x_bytes, W, out, N, K, nullptr, nullptr, act, relu2, row0, row_end,
                                                    (c0 + left % wide) * kCols, false, smem, nullptr, next);
}

// W stored tile by tile, [N/16][K/128][16 runs of 8 k][16 rows][8]; height: rows of a tile, a multiple of 32 from 128 to 256.  act > 0: W holds
// gate rows, then up rows, and out is [M, N/2]; act 0: out is [M, N], and relu2 may be set.
SHARPI_EXPORT int sharpi_gemm_dense(const void* x, const void* W, void* out, int M, int N, int K, int height, int act, float limit, int relu2,
                                    hipStream_t stream) {
  if (M <= 0) return SHARPI_OK;
  const bool gated = act > 0;
  if (height <= 0 || N <= 0 || N % (gated ? 32 : 16) || K <= 0 || K % 128 || !whole_pieces(x, W)) return SHARPI_ERR_ARG;
  if ((long long)N * K > 0x7fffffffLL || (long long)M * K > 0x7fffffffLL) return SHARPI_ERR_ARG;
  const GatedAct ga{act, limit};
  if (act < 0 || (gated && (relu2 || !act_known(ga)))) return SHARPI_ERR_ARG;      // (unknown codes: the output's width hangs on them)
  const int row_tiles = ceil_div(M, height), cols = columns_of(kMaxNT) / (gated ? 2 : 1);
  const dim3 grid((unsigned)(row_tiles * ceil_div(gated ? N / 2 : N, cols))), block(GW * kWave);
#define GD_FORM(MTV, ACTV)                                                                                                    \
  dense_gemm_kernel<MTV, ACTV><<<grid, block, 0, stream>>>((const bf16_t*)x, grouped_x_bytes(M, K), (const bf16_t*)W, (bf16_t*)out, M, N, K, \
                                                           row_tiles, ga, relu2)
#define GD(MTV)                    \
  case MTV * 32:                   \
    if (gated) GD_FORM(MTV, true); \
    else GD_FORM(MTV, false);      \
    break
  switch (height) {
    GD(4); GD(5); GD(6); GD(7); GD(8);
    default: return SHARPI_ERR_ARG;
  }
#undef GD
#undef GD_FORM
  SHARPI_CHECK_LAUNCH();
  return SHARPI_OK;
}
