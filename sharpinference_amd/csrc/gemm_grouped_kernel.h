// Grouped matrix product for routed experts with many rows (prefill):
//   out[row, :] = x[a_rows[row], :] * W[e]^T   for the rows of expert e in the expert-sorted list,
// bfloat16 inputs, float accumulation on the matrix cores.
//
// The product is bound by reading the experts' weights while few rows share them, and by what a
// compute unit can fetch and multiply once many do.  A block takes up to 256 rows of its expert against
// 256 weight rows: an expert's weights are then read once for every 256 of its rows, and a unit fetches
// 64 KB for 256 x 256 x 64 products (128 rows against 512 weight rows: 80 KB, and an expert of 129 to 256
// rows pulled its weights through two units).  An expert with more rows is cut into sibling tiles of equal height, and the
// blocks that multiply the SAME weight rows by sibling tiles start side by side on one XCD, so that the
// weights cross the memory interface about once all the same (grouped_plan.h says how the routing kernel
// lays that out; the host never learns the routing).  The tile's work is compiled for every height in
// steps of 32 rows, and a block takes the one that holds its rows.
//  * The blocks are persistent: as many as there are compute units (each holds one), every block
//    taking the next slot of its XCD's walk from a ticket counter until none is left, then slots
//    of other XCDs.  Experts of very different loads, whose tiles take very different times, are
//    so levelled at run time; with blocks dealt out beforehand an XCD that drew a block more than
//    its units can hold at once ran a second round alone.  The caller may bound the number of
//    blocks, to leave compute units to other work that runs beside the product.
//  * The 8 waves stand 2 (halves of the rows) x 4 (64 weight rows each); both operands go from memory
//    straight into LDS (loads that write LDS: no registers, so the ring is as deep as the LDS allows):
//    weights 32 of K a step, three steps ahead, in the order the packed matrix has them (1 KB a 16-row
//    tile and step, read back without conflicts); x rows (gathered through a_rows) 64 of K at a time, whole
//    128-byte lines, a stage ahead, their 16-byte pieces XORed with row bits (xs_piece).  One barrier a step; a wave
//    waits for its own loads of the step by count and the barrier makes them everyone's.  Tiles of up to 128 rows, whose steps are
//    short beside a barrier and a latency, go a stage of 64 at a time, weights and rows two or three stages ahead.
//  * W is the A operand (rows = n), x the B operand: a lane ends up with 4 consecutive n of one
//    row; bfloat16 results of two tiles are exchanged between lanes and stored as runs of 64 bytes a row.  Each output is one chain over k in ascending order, so a
//    row's result does not depend on which other rows share its tile, nor on which block took it.
//  * SwiGLU form (ACT): W holds gate rows [0, N/2) and up rows [N/2, N) of every expert; a wave's
//    tiles are two gate tiles and the up tiles of the same 32 columns, so a lane ends up with both
//    products of its outputs, rounds them to bfloat16 (what a separate activation kernel would have
//    read) and stores act(s g) * (s u), s the row's score: out is [rows, N/2] and the gate|up
//    rows never go to memory.
//  * The plain form may square the relu of its results (relu2: feed-forwards without a gate), rounded to
//    bfloat16 first (what a separate activation kernel would have read).
// Measured, 16 experts, up (2 x 8,192 rows of 5,120) + down, us, beside tiles of 128 x 512 whose weights went straight to
// registers: 8,192 tokens 1,328 + 647 (1,420 + 700), 2,048 tokens of uneven load 576 + 269 (587 + 264), 1,190 tokens 463 + 241
// (488 + 250); 64 experts of 1,408 x 2,048, six picks, 3,000 tokens 291 + 137 (327 + 157), 1,664 tokens 192 + 100 (235 + 110).
// Tiles of up to 128 rows, a step and a stage at a time: 28 experts of 2,048 x 4,096, 43 rows each 104 -> 97, 71 rows 110 -> 104; 16 of
// 5,120 x 8,192, 19 rows each 238 -> 223.  Where an expert's rows about
// fill a tile of 128 the product stays behind tiles of 128 x 512: 64 of 2,048 x 1,408, 111 rows 97 (90), 32 of 4,096 x 2,048,
// 75 rows 114 (106), 28 of 2,048 x 4,096, 71 rows 104 (92).
// Parts taken out, 4,096 tokens even (up, 656 us): no loads 465 (1.48 PFLOP/s), no products 538, weights and products without x rows
// 615: the weights' 2.7 GB and the products each need about 460, and neither hides the other whole.
// Limits: K % 64 == 0, N % 4 == 0 (N % 32 == 0 in the SwiGLU form).
#pragma once
#include <type_traits>

#include "common.h"
#include "grouped_plan.h"
#include "lds_loads.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int GM = 256;                // rows per tile: two of the plan's
static_assert(GM % kPlanTileRows == 0, "the plan's units stay level");
constexpr int GW = 8;                  // waves per block
constexpr int GWC = 4;                 // of them side by side along the columns, the others along the rows
constexpr int kMaxNT = 4;              // 16-row weight tiles per wave: this many, or half where a slot is cut
constexpr int columns_of(int nt) { return 16 * nt * GWC; }   // weight rows (output columns) of a block
constexpr int GK = 64;                 // K of a stage of x rows: two steps of 32
constexpr int kXcds = kPlanXcds;       // accelerator dies, each with its own L2
// LDS: rings of weights (steps of 32 of K) and x rows (stages of 64), see grouped_tile.
constexpr int kGroupedLds = 144 * 1024;
constexpr int kOffsetsKept = 1025;     // of more groups the rows are read from memory
static_assert(GM == 2 * 16 * 8, "tile heights are compiled in steps of 32 rows up to 256");

// Where 16-byte piece `piece` of x row `row` of a stage is kept.  The LDS serves a 16-byte read of a wave in four
// turns of two octets of lanes, one from operand rows 0..7 and one from rows 8..15 (measured with the bank-conflict
// counter); with the exclusive or the sixteen pieces of a turn fall into the sixteen different 16-byte groups of the bank space.
__device__ __forceinline__ int xs_piece(int row, int piece) { return piece ^ ((row >> 1) & 7); }

// The work of one tile of up to MT * 32 rows against 16 * NT * GWC weight rows.  DIRECT: both operands begin at 16-byte
// addresses; else the pieces go through registers, a latency of memory a step (16 experts of 8,192 x 5,120, 2,048 rows: 433 us, 1,041
// from an odd address).
template <typename TO, int MT, int NT, bool PACKED, bool ACT, bool DIRECT>
__device__ __forceinline__ void grouped_tile(const bf16_t* __restrict__ x, uint32_t x_bytes, const bf16_t* __restrict__ We,
                                             TO* __restrict__ out, int N, int K, const int* __restrict__ a_rows,
                                             const float* __restrict__ act_scale, GatedAct act, int relu2, int tile_row0, int row_end,
                                             int col_base, bool stream, const char* smem, int* counter, int& next) {
  static_assert(!ACT || NT % 2 == 0, "the SwiGLU form pairs gate tiles with up tiles");
  constexpr int HT = ACT ? NT / 2 : NT;         // tiles of distinct output columns per wave
  const int n_out = ACT ? N / 2 : N;            // output columns
  constexpr int TILES = NT * GWC;               // weight tiles of the block
  constexpr int WL = (TILES + GW - 1) / GW;     // loads of weights a wave and step
  constexpr int XL = (4 * MT + GW - 1) / GW;    // loads of x rows a wave and stage (8 rows each)
  // The rings: of tall tiles two stages of x rows (32 KB each) and four steps of weights (16 KB), filled a step at a time, weights three
  // steps ahead; of tiles of up to 128 rows (half as much of x) three stages of both, of which a cut slot's (half of the weights, too)
  // has four, filled a stage at a time.
  constexpr int RS = MT > 4 ? 2 : NT == kMaxNT ? 3 : 4;
  constexpr bool STAGED = RS > 2;
  constexpr int kWStep = 1024 * (MT > 4 ? 16 : TILES), kXStage = MT > 4 ? 32768 : 16384, kXAt = 2 * RS * kWStep;
  constexpr int GL = XL + 2 * WL;               // a wave's loads of a stage
  static_assert(TILES * 1024 <= kWStep && MT * 32 * GK * 2 <= kXStage && kXAt + RS * kXStage <= kGroupedLds, "the rings hold a tile");
  const int lane = threadIdx.x & (kWave - 1);
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int wr = wid / GWC, wc = wid % GWC;

  // Weights: tile lt of the block is tile lt % NT of column wave lt / NT.  A tile that lies beyond the last column (or its rows that do)
  // is read as the last that exists, never stored.
  // Packed layout (the matrix stored as [N/16][K/128][16 runs of 8 k][16 rows][8]): a step of a tile is 1 KB in a row.
  // Row layout: lane (row l % 16, run l / 16) reads 16 bytes of its row; in LDS both lie as [run][row].  Where weights come a stage at a
  // time a load takes whole lines, 8 rows of 128 bytes, as those of x rows do.  The streaming hint goes with whole lines only: of half a
  // line the other half came from memory once more.  us with tiles of 128 x 512, half lines and the hint, half lines without, lines
  // without and lines with it: 16 experts of 8,192 x 5,120, 300 rows 281, 382, 308, 259, 234; 64 of 2,816 x 2,048, 300 tokens 186,
  // 234, 187, 172, 162; 20 of 1,408 x 960 (caches hold them from call to call) 33, 33, 25, 23, 26.
  constexpr bool LINES = STAGED && !PACKED;
  constexpr uint32_t kWStepBytes = PACKED ? 1024 : 64;
  uint32_t w_off[LINES ? 2 : 1][WL];
  int w_tile[WL];
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int lt = (wid * WL + i) % TILES;      // (fewer tiles than waves: fetched twice, to the same place)
    const int t = lt % NT;
    int n = col_base + (lt / NT) * HT * 16 + (t % HT) * 16;
    w_tile[i] = lt;
    if constexpr (PACKED) {
      if (n >= n_out) n = n_out - 16;
      if (ACT && t >= HT) n += n_out;
      w_off[0][i] = (uint32_t)n * (uint32_t)K * 2 + lane * 16;
    } else {
#pragma unroll
      for (int u = 0; u < (LINES ? 2 : 1); ++u) {
        const int row = LINES ? u * 8 + (lane >> 3) : lane & 15, piece = LINES ? xs_piece(row, lane & 7) : lane >> 4;
        w_off[u][i] = (uint32_t)(min(n + row, n_out - 1) + (ACT && t >= HT ? n_out : 0)) * (uint32_t)K * 2 + piece * 16;
      }
    }
  }
  f32x4 acc[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int mb = 0; mb < MT; ++mb) acc[t][mb] = f32x4{0.f, 0.f, 0.f, 0.f};

  const u32x4 wb = buffer_of(We, (uint32_t)N * (uint32_t)K * 2), xb = buffer_of(x, x_bytes);
  const uint32_t lds0 = lds_address(smem);
  const int steps = K / 32, stages = K / GK;
  auto load_w = [&](int s, int place) {         // weights of step s into the ring
    const int u = LINES ? s & 1 : 0;
    const uint32_t step = LINES ? (s >> 1) * (GK * 2) : s * kWStepBytes;
    uint32_t at[WL], off[WL];
#pragma unroll
    for (int i = 0; i < WL; ++i) {
      at[i] = lds0 + (LINES ? (place >> 1) * 2 * kWStep + w_tile[i] * 2048 + u * 1024 : place * kWStep + w_tile[i] * 1024);
      off[i] = LINES ? (u ? w_off[LINES][i] : w_off[0][i]) : w_off[0][i];
    }
    if (DIRECT && stream && (PACKED || LINES)) bring_all_to_lds<true, WL, true>(wb, off, step, at);
    else bring_all_to_lds<DIRECT, WL>(wb, off, step, at);
  };
#pragma unroll
  for (int s = 0; s < (STAGED ? 2 * RS - 2 : 3); ++s)   // (on their way while the rows' places are looked up)
    if (s < 2 || s < steps) load_w(s, s);
  // x rows: a load brings 8 rows of 128 bytes, lane l row l / 8 at place l % 8.  Rows beyond the expert's last read its last row again
  // (what such rows produce is never stored).
  uint32_t x_off[XL];
  int x_load[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int li = min(wid * XL + i, 4 * MT - 1);
    const int lrow = li * 8 + (lane >> 3);
    const int row = min(tile_row0 + lrow, row_end - 1);
    x_load[i] = li;
    x_off[i] = (uint32_t)(a_rows ? a_rows[row] : row) * (uint32_t)K * 2 + xs_piece(lrow, lane & 7) * 16;
  }
  // waited for here: the compiler's own waits must not fall among the loads below, which it does not know of
#pragma unroll
  for (int i = 0; i < XL; ++i) asm volatile("" : "+v"(x_off[i]));
  auto load_x = [&](int c, int place) {         // x rows of stage c
    uint32_t at[XL];
#pragma unroll
    for (int i = 0; i < XL; ++i) at[i] = lds0 + kXAt + place * kXStage + x_load[i] * 1024;
    bring_all_to_lds<DIRECT, XL>(xb, x_off, c * (GK * 2), at);
  };
#pragma unroll
  for (int c = 0; c < RS - 1; ++c)
    if (c == 0 || c < stages) load_x(c, c);

  // operand addresses (bytes): fragment t of a step lies at w_at + t * 1024 (lines: 2048), row group mb of a stage's half at x_at + mb * 2048
  int w_at[2];
#pragma unroll
  for (int hh = 0; hh < 2; ++hh)
    w_at[hh] = LINES ? wc * NT * 2048 + r * 128 + xs_piece(r, hh * 4 + g) * 16 : wc * NT * 1024 + lane * 16 + hh * kWStep;
  int x_at[2];
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) x_at[hh] = kXAt + (wr * MT * 16 + r) * 128 + xs_piece(r, hh * 4 + g) * 16;
  // LDS reads run beside products: a step begins with its weights and half of its row groups in registers, reads the
  // other half while the first is multiplied, and the next step's first part while the other half is (with all reads of a step ahead
  // of its products, the LDS and the matrix cores took turns).
  constexpr int H0 = (MT + 1) / 2, H1 = MT / 2;
  bf16x8 wf[2][NT], x0[H0], x1[H1 > 0 ? H1 : 1];
  int place = 0;                                // of this stage in the rings
  auto arrive = [&](int s, auto half_tag) {     // step s is in LDS, and everyone has read step s - 1
    constexpr int hh = decltype(half_tag)::value;
    // This step's loads: counted is what was sent behind them.  (The first x rows were sent last: everything is waited for.)
    if constexpr (STAGED) {                     // whole stages: those behind it
      if (hh == 1) return;                      // (came with the step before)
      const int behind = stages - 1 - (s >> 1);
      if (s == 0) lds_loads_wait<0>();
      else if (RS == 4 && behind >= 2) lds_loads_wait<2 * GL>();
      else if (behind >= 1) lds_loads_wait<GL>();
      else lds_loads_wait<0>();
    } else {                                    // two steps of weights and, in a stage's second step, the next stage's x rows
      if (s > 0 && s + 2 < steps) lds_loads_wait<hh == 0 ? 2 * WL : 2 * WL + XL>();
      else lds_loads_wait<0>();
    }
    __syncthreads();
  };
  auto send = [&](int s, auto half_tag) {       // the loads that take the place of step s - 1, or of the stage before
    constexpr int hh = decltype(half_tag)::value;
    if constexpr (STAGED) {
      const int c = (s >> 1) + RS - 1, to = place == 0 ? RS - 1 : place - 1;
      if (hh == 0 && c < stages) {
        load_x(c, to);
        load_w(2 * c, 2 * to);
        load_w(2 * c + 1, 2 * to + 1);
      }
    } else {
      if (hh == 0 && (s >> 1) + 1 < stages) load_x((s >> 1) + 1, place ^ 1);
      if (s + 3 < steps) load_w(s + 3, (s + 3) & 3);
    }
  };
  auto read_first = [&](auto half_tag) {
    constexpr int hh = decltype(half_tag)::value;
#pragma unroll
    for (int t = 0; t < NT; ++t) wf[hh][t] = *reinterpret_cast<const bf16x8*>(smem + w_at[hh] + t * (LINES ? 2048 : 1024));
#pragma unroll
    for (int mb = 0; mb < H0; ++mb) x0[mb] = *reinterpret_cast<const bf16x8*>(smem + x_at[hh] + mb * 2048);
  };
  // the order the compiler is to keep: a read, then its share of the products
  auto in_turn = [&](auto reads_tag, auto products_tag) {
    constexpr int R = decltype(reads_tag)::value, P = decltype(products_tag)::value, kShare = R > 0 && P > R ? P / (R > 0 ? R : 1) : 1;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x8, kShare, 0);
    }
  };
  auto step = [&](int s, auto half_tag, auto last_tag) {
    constexpr int hh = decltype(half_tag)::value;
    constexpr bool last = decltype(last_tag)::value;
#pragma unroll
    for (int mb = 0; mb < H1; ++mb) x1[mb] = *reinterpret_cast<const bf16x8*>(smem + x_at[hh] + (H0 + mb) * 2048);
    auto row_products = [&](const bf16x8& rows, int mb) {
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[t][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[hh][t], rows, acc[t][mb], 0, 0, 0);
    };
#pragma unroll
    for (int mb = 0; mb < H0; ++mb) row_products(x0[mb], mb);
    in_turn(std::integral_constant<int, H1>{}, std::integral_constant<int, H0 * NT>{});
    if constexpr (hh == 1) {
      const int turn = place == RS - 1 ? 1 - RS : 1;
      place += turn;
      w_at[0] += turn * 2 * kWStep;
      w_at[1] += turn * 2 * kWStep;
      x_at[0] += turn * kXStage;
      x_at[1] += turn * kXStage;
    }
    if constexpr (!last) {
      __builtin_amdgcn_sched_barrier(0);        // products of the first half stay ahead of the barrier, those of the other behind it
      arrive(s + 1, std::integral_constant<int, hh ^ 1>{});
      __builtin_amdgcn_sched_barrier(0);
      read_first(std::integral_constant<int, hh ^ 1>{});
    }
    // this half's products, with the reads above and, half way through, the loads that fill the place step s has left
    constexpr int kBefore = H1 / 2;
#pragma unroll
    for (int mb = 0; mb < kBefore; ++mb) row_products(x1[mb], H0 + mb);
    if constexpr (!last) {
      in_turn(std::integral_constant<int, NT + H0>{}, std::integral_constant<int, kBefore * NT>{});
      __builtin_amdgcn_sched_barrier(0);
      send(s + 1, std::integral_constant<int, hh ^ 1>{});
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int mb = kBefore; mb < H1; ++mb) row_products(x1[mb], H0 + mb);
  };
  using Half0 = std::integral_constant<int, 0>;
  using Half1 = std::integral_constant<int, 1>;
  arrive(0, Half0{});
  send(0, Half0{});
  read_first(Half0{});
  for (int c = 0; c + 1 < stages; ++c) {
    step(2 * c, Half0{}, std::false_type{});
    step(2 * c + 1, Half1{}, std::false_type{});
  }
  step(steps - 2, Half0{}, std::false_type{});
  step(steps - 1, Half1{}, std::true_type{});

  if (counter && threadIdx.x == 0) next = atomicAdd(counter, 1);   // the block's next slot: on its way while the results are stored
  const int n_base = col_base + wc * HT * 16, row0 = tile_row0 + wr * MT * 16;
  // lane holds out[row0 + mb*16 + r][n_base + t*16 + 4g + 0..3]
  auto store4 = [&](int row, int t, const f32x4& v) {
    const int n = n_base + t * 16 + 4 * g;
    if (row >= row_end || n >= n_out) return;
    TO* dst = out + (size_t)row * n_out + n;
    if constexpr (sizeof(TO) == 4) *reinterpret_cast<f32x4*>(dst) = v;
    else *reinterpret_cast<uint2*>(dst) = make_uint2(f32_to_bf16_pair(v[0], v[1]), f32_to_bf16_pair(v[2], v[3]));
  };
  // Tiles t and t + 1 of a row: lanes 16 apart exchange halves, one ends up with eight columns of tile t and the other with eight of
  // tile t + 1; a row's 32 columns are then stored as one run of 64 bytes (wide: rows and out begin at 16-byte addresses).
  const bool wide = sizeof(TO) == 2 && ((n_out & 7) | (int)((uintptr_t)out & 15)) == 0;
  auto store_pair = [&](int row, int t, const f32x4& v, const f32x4& w) {
    if (!wide) {
      store4(row, t, v);
      store4(row, t + 1, w);
      return;
    }
    const auto lo = __builtin_amdgcn_permlane16_swap(f32_to_bf16_pair(v[0], v[1]), f32_to_bf16_pair(w[0], w[1]), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(f32_to_bf16_pair(v[2], v[3]), f32_to_bf16_pair(w[2], w[3]), false, false);
    const int n = n_base + (t + (g & 1)) * 16 + 4 * (g & 2);
    if (row < row_end && n < n_out) *reinterpret_cast<uint4*>(out + (size_t)row * n_out + n) = make_uint4(lo[0], hi[0], lo[1], hi[1]);
  };
  auto store_tiles = [&](int row, auto value) {        // value(t): tile t of the row group
    if constexpr (HT % 2 == 0) {
#pragma unroll
      for (int t = 0; t < HT; t += 2) store_pair(row, t, value(t), value(t + 1));
    } else {
#pragma unroll
      for (int t = 0; t < HT; ++t) store4(row, t, value(t));
    }
  };
  auto rounded = [](float v) { return bf16_to_f32(f32_to_bf16(v)); };
  if constexpr (ACT) {
    // The code is chosen once for the tile: a choice an element made the unrolled epilogue larger than the instruction cache (10 us of a
    // slot's 55: 64 experts of 2 x 1,408 x 2,048, six picks, 3,000 tokens 281 us, 268 with the choice a tile and the runs; with the
    // hardware's power of two and reciprocal for expf and the division, as exact but other bits, 261).
    auto store_gated = [&](auto code_tag) {
#pragma unroll
      for (int mb = 0; mb < MT; ++mb) {
        if (row0 + mb * 16 >= row_end) break;   // (the wave's: no rows from here on)
        const int row = row0 + mb * 16 + r;
        const float sc = act_scale && row < row_end ? act_scale[row] : 1.0f;
        store_tiles(row, [&](int h) {
          f32x4 o;
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = gated_f32<decltype(code_tag)::value>(act.limit, rounded(acc[h][mb][i]) * sc, rounded(acc[h + HT][mb][i]) * sc);
          return o;
        });
      }
    };
    if (act.code == ACT_SWISH_CLAMP) store_gated(std::integral_constant<int, ACT_SWISH_CLAMP>{});
    else if (act.code == ACT_GELU_TANH) store_gated(std::integral_constant<int, ACT_GELU_TANH>{});
    else store_gated(std::integral_constant<int, ACT_SILU>{});
  } else {
    // (Row groups without rows are not skipped here: little is done for them, and the branches cost more.  64 experts of 2,048 x 1,408,
    // 300 tokens 76.6 us, 78.0 with the skip, 1,600 tokens 95.7 and 98.4; 32 of 4,096 x 2,048, 300 tokens 98.1 and 99.3.)
#pragma unroll
    for (int mb = 0; mb < MT; ++mb)
      store_tiles(row0 + mb * 16 + r, [&](int t) {
        f32x4 v = acc[t][mb];
        if (relu2) {
#pragma unroll
          for (int i = 0; i < 4; ++i) v[i] = ungated_f32(UACT_RELU2, rounded(v[i]));
        }
        return v;
      });
  }
}

template <typename TO, int NT, bool PACKED, bool ACT, bool DIRECT>
__global__ __launch_bounds__(GW* kWave, 2) void grouped_gemm_kernel(
    const bf16_t* __restrict__ x, uint32_t x_bytes, const bf16_t* __restrict__ W, TO* __restrict__ out, int N, int K,
    const int* __restrict__ a_rows, const float* __restrict__ act_scale, GatedAct act, int relu2,
    const int* __restrict__ group_offsets, const int* __restrict__ plan, int n_groups, int nb) {
  __shared__ __attribute__((aligned(1024))) char smem[kGroupedLds];
  __shared__ int s_slot, s_total[kXcds], s_rows[kXcds], s_taken[kXcds];
  __shared__ int4 s_unit[kWave + 1];
  __shared__ int s_offset[kOffsetsKept];
  constexpr int GN = columns_of(NT);
  constexpr int kCols = ACT ? GN / 2 : GN;   // output columns of a block
  const int n_out = ACT ? N / 2 : N;
  // The blocks stay (one to a compute unit, as many as there are units) and take work until none is
  // left.  Workgroups go to the 8 XCDs round-robin by their linear id, so this block sits on XCD
  // blockIdx.x % 8 and walks that XCD's units first, slot by slot: a unit's column blocks times its
  // siblings, the siblings of a column block side by side.  The slots of an XCD are handed out by a
  // ticket counter; when its own XCD's are gone a block takes slots of the next XCD's walk.
  //
  // A walk is only a few slots per block long: slots that fill no whole round of the XCD's blocks would leave most of them idle for
  // a slot's time at the end.  Those last slots are therefore cut by columns into two (16 experts of 13 to 396 rows, 8,192 ->
  // 5,120: 313 us where they were cut only if the halves fitted one round, 294 always; quarters, 318, read the x rows too often;
  // a first round nearly full, 28 experts of 2,048 x 4,096, 71 rows each, 104 halved, 112 whole).
  // A walk with work for a quarter of its blocks cuts its groups into tiles of half the rows: twice as many blocks, and the deeper rings
  // (one matrix of 2,048 x 4,096, 130 rows 53 -> 37 us, 700 rows 58 -> 40; 8 groups of 512 x 512, 250 rows each 18.8 -> 16.0;
  // from half of the blocks on nothing changed).
  if (n_groups < kOffsetsKept)
    for (int i = threadIdx.x; i <= n_groups; i += GW * kWave) s_offset[i] = group_offsets[i];
  __syncthreads();
  // The unit lists are read by waves, a unit a lane (every thread after the other through the 16 units of each XCD
  // that 64 groups make cost 40 us a product: 16 rows an expert, 64 experts of 2,816 x 2,048: 173 -> 135 us).
  int* counters = const_cast<int*>(plan) + plan_counters_at(n_groups);
  const int home = blockIdx.x % kXcds;
  const int per_xcd = ((int)gridDim.x + kXcds - 1) / kXcds;   // blocks whose first walk is one XCD's
  const int lane = threadIdx.x & (kWave - 1);
  // The plan counts siblings of kPlanTileRows rows; here a group's rows are cut into tiles of GM, or half of that where the
  // walk has little work (the deal stays level, and the tall tiles, which take longest, still come first in a walk).
  auto offset_of = [&](int e) { return n_groups < kOffsetsKept ? s_offset[e] : group_offsets[e]; };
  auto siblings_of = [&](int e, int rows) { return (offset_of(e + 1) - offset_of(e) + rows - 1) / rows; };
  auto unit_slots = [&](const int* pu, int rows) {
    return (plan_part_first(pu[1] + 1, pu[2], nb) - plan_part_first(pu[1], pu[2], nb)) * siblings_of(pu[0], rows);
  };
  // units j0 .. j0 + 63 of a walk into LDS: (slots before it, group, siblings, first column block), and all their slots
  auto list_units = [&](const int* px, int n_units, int j0, int rows) {
    __syncthreads();
    if (threadIdx.x < kWave) {
      const int* pu = px + 1 + 4 * min(j0 + lane, n_units - 1);
      const int u_group = pu[0], u_sib = siblings_of(pu[0], rows), u_col = plan_part_first(pu[1], pu[2], nb);
      const int slots = j0 + lane < n_units ? unit_slots(pu, rows) : 0;
      int upto = slots;
#pragma unroll
      for (int o = 1; o < kWave; o <<= 1) {
        const int up = __shfl_up(upto, o, kWave);
        if (lane >= o) upto += up;
      }
      s_unit[lane] = make_int4(j0 + lane < n_units ? upto - slots : 0x7fffffff, u_group, u_sib, u_col);
      if (lane == kWave - 1) s_unit[kWave] = make_int4(upto, 0, 0, 0);
    }
    __syncthreads();
  };
  static_assert(GW == kXcds, "a wave counts the slots of one XCD's walk");
  {
    const int x = threadIdx.x >> 6;
    const int* px = plan + x * plan_stride(n_groups);
    const int n_units = px[0];
    int total = 0, total_low = 0;
    for (int j = lane; j < n_units; j += kWave) {
      total += unit_slots(px + 1 + 4 * j, GM);
      total_low += unit_slots(px + 1 + 4 * j, GM / 2);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      total += __shfl_xor(total, o, kWave);
      total_low += __shfl_xor(total_low, o, kWave);
    }
    if (lane == 0) {
      const bool low = 4 * total <= per_xcd;
      s_total[x] = low ? total_low : total;
      s_rows[x] = low ? GM / 2 : GM;
    }
  }
  __syncthreads();
  for (int q = 0; q < kXcds; ++q) {
    const int xcd = (home + q) % kXcds;
    const int* px = plan + xcd * plan_stride(n_groups);
    const int n_units = px[0];
    const int total = __builtin_amdgcn_readfirstlane(s_total[xcd]);   // slots of this walk
    const int whole = total / per_xcd * per_xcd;   // slots of whole rounds: taken as they are
    const int rest = total - whole;
    const int cut = DIRECT && rest > 0 ? 2 : 1;
    const int rows_most = __builtin_amdgcn_readfirstlane(s_rows[xcd]);
    const int tickets = whole + rest * cut;
    if (q == 1) {                                  // its own walk is done: which others still have slots
      if (threadIdx.x < kXcds) s_taken[threadIdx.x] = __hip_atomic_load(&counters[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
    }
    if (q > 0 && s_taken[xcd] >= tickets) continue;
    if (n_units > 0 && n_units <= kWave) list_units(px, n_units, 0, rows_most);
    int next = -1;                                 // thread 0: the ticket taken at the end of the slot before, if there was one
    for (;;) {
      if (threadIdx.x == 0) s_slot = next >= 0 ? next : atomicAdd(&counters[xcd], 1);
      next = -1;
      __syncthreads();
      const int ticket = __builtin_amdgcn_readfirstlane(s_slot);      // (what is found through LDS is the same for all lanes: scalars again)
      __syncthreads();
      if (ticket >= tickets) break;                // this walk is done
      const int width = ticket < whole ? 1 : cut;  // this slot is 1 / width of a column block
      int slot = ticket < whole ? ticket : whole + (ticket - whole) / width;
      const int piece = ticket < whole ? 0 : (ticket - whole) % width;
      int e = -1, n_sib = 1, col0 = 0;
      for (int j0 = 0; j0 < n_units && e < 0; j0 += kWave) {
        if (n_units > kWave) list_units(px, n_units, j0, rows_most);
        const int mine = s_unit[lane].x;             // this lane's unit begins behind so many slots (of these units)
        const int last = __builtin_amdgcn_readfirstlane(s_unit[kWave].x);
        if (slot < last) {
          const int at = __popcll((unsigned long long)__ballot(mine <= slot)) - 1;
          const int4 u = s_unit[at];
          e = __builtin_amdgcn_readfirstlane(u.y);
          n_sib = __builtin_amdgcn_readfirstlane(u.z);
          col0 = __builtin_amdgcn_readfirstlane(u.w);
          slot -= __builtin_amdgcn_readfirstlane(u.x);
        } else {
          slot -= last;
        }
      }
      if (e < 0) break;                            // (behind the walk's last unit: not reached)
      const int sib = slot % n_sib;
      const int nblock = col0 + slot / n_sib;
      const int col_base = nblock * kCols + piece * (kCols / width);
      if (col_base >= n_out) continue;
      const int first_row = offset_of(e), last_row = offset_of(e + 1);
      const int height = plan_height(last_row - first_row, n_sib);
      const int row0 = first_row + sib * height;
      const int row_end = min(last_row, row0 + height);
      const int n_rows = row_end - row0;
      if (n_rows <= 0) continue;
      const bf16_t* We = W + (size_t)e * N * K;
      // (the streaming hint only where no sibling reads the same weights: a pure read reaches 6.9 TB/s with it, 6.2 without)
#define GTILE(MTV, NTV) \
  grouped_tile<TO, MTV, NTV, PACKED, ACT, DIRECT>(x, x_bytes, We, out, N, K, a_rows, act_scale, act, relu2, row0, row_end, col_base, n_sib == 1, smem, &counters[xcd], next)
#define GT1(MTV, NTV) case MTV: GTILE(MTV, NTV); break
#define GT(NTV)                                                                                                  \
  switch ((n_rows + 31) >> 5) {                                                                                  \
    GT1(1, NTV); GT1(2, NTV); GT1(3, NTV); GT1(4, NTV); GT1(5, NTV); GT1(6, NTV); GT1(7, NTV); GT1(8, NTV);      \
  }
      if constexpr (DIRECT) {
        if (width == 1) GT(NT)
        else GT(NT / 2)
      } else {                                     // (two heights are compiled: such a product waits for its operands)
        if (n_rows <= 64) GTILE(2, NT);
        else GTILE(8, NT);
      }
#undef GT
#undef GT1
#undef GTILE
    }
  }
  // the last block to leave sets the counters back for the next product that reads this plan
  if (threadIdx.x == 0) {
    if (atomicAdd(&counters[kXcds], 1) == (int)gridDim.x - 1) {
      for (int i = 0; i <= kXcds; ++i) counters[i] = 0;
    }
  }
}

static bool grouped_args_ok(int x_rows, int n_rows, int N, int K, int n_groups, int packed, const int* group_offsets,
                            const int* plan) {
  if (N <= 0 || (N & 3) || K <= 0 || K % GK != 0 || n_groups <= 0) return false;
  if (packed && ((N & 15) || (K & 127))) return false;
  if (!group_offsets || !plan) return false;
  // the kernel addresses x and one group's weights with 32-bit element offsets
  return (long long)N * K <= 0x7fffffffLL && x_rows > 0 && (long long)x_rows * K <= 0x7fffffffLL;
}

static uint32_t grouped_x_bytes(int x_rows, int K) {
  const unsigned long long bytes = 2ull * x_rows * K;       // below 2^32: grouped_args_ok
  return (uint32_t)bytes;
}

// As many blocks as stay at once (one to a compute unit), fewer if there is less work (a slot may
// be cut in two) or if the caller bounds them (max_blocks > 0: the compute units left over
// are for other work).
static dim3 grouped_grid(int n_rows, int n_groups, int nb, int max_blocks) {
  long long blocks = 2LL * kXcds * plan_slots_bound(n_rows, n_groups, nb);
  const long long stay = compute_units();
  if (blocks > stay) blocks = stay;
  if (max_blocks > 0 && blocks > max_blocks) blocks = max_blocks;
  return dim3((unsigned)(blocks < 1 ? 1 : blocks));
}

