// Y[M, N] = X[M, K] * W[N, K]^T of bf16 for prompts, and the gated form act(X W^T) * (X W2^T), in tiles of up to 352 rows x 256 W rows
// (wide_tile.h).  Results are bf16 or float32, sums float32 in the order of K: a row's result depends on that row alone.
//
// What bounds it: the matrix cores at the clock that the chip holds under them (8,192 rows x 28,672 x 4,096, gated: 90 us a round of
// tiles of 256 rows, 1,530 TFLOP/s), and how even its rounds over the compute units are.  So
//  - one workgroup a compute unit goes through tiles, and the next tile's first two steps are on their way while one ends and its
//    results are stored: with a workgroup a tile the same product took 1,372 us, now 1,261 (2,048 rows 367 -> 331);
//  - the height of the tiles is chosen for the matrix, and a last round of half the units or fewer is of tiles of half the height;
//  - the gate costs ten instructions and two of the transcendental unit a number, 1 us a tile more than those two with nothing that makes up for
//    their argument's rounding (8,192 rows x 28,672 x 4,096 1,292 us / 1,278), whose error grows with the gate; expf and a division: 6 us a tile;
//  - W's rows lie in LDS in such an order that bf16 results leave 16 bytes a lane.
#include "wide_tile.h"
#include "hal_api.h"

#include <algorithm>

#define WG_DIES 8     // of the gfx950 parts that this library is built for (a wrong count costs cache hits only)
#define WG_UNITS 32   // compute units of a die
#define WG_PANEL 4    // row tiles that are gone through column by column

struct WideArgs {
  const bf16_t *X, *W, *W2;
  int ldx, ldw;
  void* Y;
  int ldy, f32, M, N, K;
  int rows, row_tiles, col_tiles;  // rows of a tile: row_tiles * rows >= M
  hal_gate gate;
};

// Where a tile's operands are: base addresses, the bytes from there on that are rows of its own.
struct wg_place {
  const bf16_t *x, *w, *w2;
  uint32_t x_bytes, w_bytes;
  int row0, row_end, n0;
};
template <bool GATED>
__device__ __forceinline__ wg_place wg_place_of(const WideArgs& a, int tile) {
  const int panel = tile / (WG_PANEL * a.col_tiles), in_panel = tile % (WG_PANEL * a.col_tiles), high = min(WG_PANEL, a.row_tiles - panel * WG_PANEL);
  constexpr int COLS = GATED ? WT_COLS / 2 : WT_COLS;
  wg_place p;
  p.n0 = in_panel / high * COLS, p.row0 = (panel * WG_PANEL + in_panel % high) * a.rows, p.row_end = min(a.M, p.row0 + a.rows);
  p.x = a.X + (size_t)p.row0 * a.ldx, p.x_bytes = ((uint32_t)(p.row_end - p.row0 - 1) * a.ldx + a.K) * 2;
  p.w = a.W + (size_t)p.n0 * a.ldw, p.w_bytes = ((uint32_t)(min(COLS, a.N - p.n0) - 1) * a.ldw + a.K) * 2;
  p.w2 = GATED ? a.W2 + (size_t)p.n0 * a.ldw : p.w;
  return p;
}

// sigmoid(z), to some 2^-22 of it: 1 over 1 + exp(-z) by the reciprocal and a step of Newton's, and the exponential as a power of two behind which
// is brought in what its argument's rounding lost.  (z is held where the power is finite: from there on down its reciprocal is 0, and up 1.)
__device__ __forceinline__ float wg_sigmoid(float z) {
  constexpr double LN_2 = 0.6931471805599453;
  constexpr float LOG2_E = 1.4426950408889634f, HIGH = (float)LN_2, LOW = (float)(LN_2 - (double)HIGH);
  const float b = __builtin_amdgcn_fmed3f(z, -88.5f, 88.5f), t = b * -LOG2_E;
  const float rest = fmaf(t, -LOW, fmaf(t, -HIGH, -b)), power = __builtin_amdgcn_exp2f(t);
  const float d = 1.0f + fmaf(power, rest, power), y = __builtin_amdgcn_rcpf(d);
  return fmaf(fmaf(-d, y, 1.0f), y, y);
}
__device__ __forceinline__ float wg_gated(const hal_gate& a, float g, float u) {
  float z = g;
  if (a.act == HAL_ACT_CLAMPED) {
    g = fminf(g, a.limit), u = fminf(fmaxf(u, -a.limit), a.limit) + a.up_shift;
    z = a.alpha * g;
  } else if (a.act == HAL_ACT_GELU_TANH) {  // 0.5 (1 + tanh(y)) = sigmoid(2 y)
    z = 1.5957691216057308f * (g + 0.044715f * g * g * g);
  }
  return g * wg_sigmoid(z) * u;
}

template <bool GATED, int NI>
__device__ __forceinline__ void wg_store(const WideArgs& a, const wg_place& p, int wave, int lane, wt_f32x4 (&acc)[NI][4]) {
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = p.row0 + (wave / 4 * NI + i) * 16 + lane % 16;
    if (r >= p.row_end) continue;
    const size_t row = (size_t)r * a.ldy;
    if (GATED) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int k = 0; k < 4; ++k) acc[i][j][k] = wg_gated(a.gate, acc[i][j][k], acc[i][j + 2][k]);
    }
    // (bf16: a lane's four columns of each of two neighbouring blocks lie beside each other, see wg_tiles)
#pragma unroll
    for (int h = 0; h < (GATED ? 1 : 2); ++h) {
      const int n = p.n0 + wave % 4 * (GATED ? 32 : 64) + h * 32;
      const wt_f32x4 v = acc[i][2 * h], u = acc[i][2 * h + 1];
      if (a.f32) {
        const int c = n + lane / 16 * 4;
        if (c < a.N) *(wt_f32x4*)((float*)a.Y + row + c) = v;
        if (c + 16 < a.N) *(wt_f32x4*)((float*)a.Y + row + c + 16) = u;
      } else {
        const int c = n + lane / 16 * 8;
        const uint4 all = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(u[0], u[1]), pack_bf16x2(u[2], u[3]));
        bf16_t* to = (bf16_t*)a.Y + row + c;
        if (c + 4 < a.N && a.ldy % 8 == 0) {
          *(uint4*)to = all;
        } else {
          if (c < a.N) *(uint2*)to = make_uint2(all.x, all.y);
          if (c + 4 < a.N) *(uint2*)(to + 4) = make_uint2(all.z, all.w);
        }
      }
    }
  }
}

// Tiles of at most 32 * NI rows: `tile` and every `apart`-th after it below `end`, the next one's first pieces on their way while one's results are stored;
// or, of one tile, a half of 32 * NI rows (0 or 1; -1: all of it).
template <bool GATED, int NI, bool ONCE>
__device__ __forceinline__ void wg_tiles(const WideArgs& a, const wt_lds& lds, int wave, int tile, int apart, int end, int half) {
  using P = wt_part<NI>;
  int lane = threadIdx.x % 64;
  const int oct = lane / 8, c = ((lane % 8) ^ hal_turn(wave % 2 * 8 + oct)) * 16, steps = a.K / WT_TK;
  wg_place here = wg_place_of<GATED>(a, tile);
  if (half >= 0) {
    const int skip = half ? min(32 * NI, here.row_end - here.row0) : 0;
    here.row_end = half ? here.row_end : min(here.row_end, here.row0 + 32 * NI);
    if (here.row0 + skip >= here.row_end) return;
    here.row0 += skip, here.x += (size_t)skip * a.ldx;
    here.x_bytes = ((uint32_t)(here.row_end - here.row0 - 1) * a.ldx + a.K) * 2;
  }
  wg_place next = here;
  // (rows past the end lie past the operand's bytes and are read as zeros)
  uint32_t xo[P::loads(0) + P::loads(1)];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int u = 0; u < P::loads(p); ++u) {
      uint32_t& to = xo[p * P::loads(0) + u];
      to = (uint32_t)(wt_octet_row<NI>(wt_octet<NI>(wave, p, u), p) + oct) * (uint32_t)(a.ldx * 2) + c;
      asm("v_mov_b32 %0, %1" : "=v"(to) : "v"(to));  // (one register, not the pair that a multiplication with addition writes)
    }
  // A wave's 64 W rows are two halves of 32 (GATED: the gate's and the up projection's), a half two blocks of 16, of which a lane of a result has
  // rows 4 q .. + 3 (q = lane / 16).  For results of bf16 these are rows 8 q .. and 8 q + 4 .. of the half's 32, so that they leave as one store.
  const int in_block = wave % 2 * 8 + oct, in_half = a.f32 ? wave / 2 % 2 * 16 + in_block : in_block / 4 * 8 + wave / 2 % 2 * 4 + in_block % 4;
  const uint32_t row = (uint32_t)a.ldw * 2, wo = (uint32_t)(wave / 4 * (GATED ? 32 : 64) + in_half) * row + c;
  auto bring_x = [&](auto part, char* to, int step) {
    constexpr int p = decltype(part)::value;
    const bool over = step >= steps;
    const hal_memory X = hal_memory_at(over ? next.x : here.x, over ? next.x_bytes : here.x_bytes);
    const uint32_t at = (uint32_t)(over ? step - steps : step) * (WT_TK * 2);
#pragma unroll
    for (int u = 0; u < P::loads(p); ++u) hal_load_lds(X, xo[p * P::loads(0) + u], at, to + wt_octet<NI>(wave, p, u) * 1024);
  };
  auto bring_w = [&](int half_of_w, char* to, int step) {
    const bool over = step >= steps;
    const hal_memory W = hal_memory_at(half_of_w ? (over ? next.w2 : here.w2) : over ? next.w : here.w, over ? next.w_bytes : here.w_bytes);
    const uint32_t at = (uint32_t)(over ? step - steps : step) * (WT_TK * 2);
#pragma unroll
    for (int u = 0; u < 2; ++u) hal_load_lds<ONCE ? HAL_ONCE : 0>(W, wo + (GATED ? u * 64 : u * 128 + half_of_w * 32) * row, at, to + (wave + 8 * u) * 1024);
  };
  wt_begin<NI>(lds, bring_x, bring_w);
  for (;;) {
    tile += apart;
    const bool more = half < 0 && tile < end;
    if (more) next = wg_place_of<GATED>(a, tile);
    wt_f32x4 acc[NI][4];
    wt_steps<NI>(lds, wave, lane, steps, acc, bring_x, bring_w);
    asm volatile("" : "+v"(lane));  // (or what follows from it would be kept in registers over the products)
    wg_store<GATED, NI>(a, here, wave, lane, acc);
    if (!more) break;
    here = next;
  }
  wt_end();
}

// A die takes an eighth of the tiles, neighbours in an order that goes through WG_PANEL row tiles column by column, so that its 32
// workgroups read few different rows.  Its last round, if at most half of its units have a tile in it, is of tiles of half the height.
// ONCE: one row tile, so that W is read once and passes the caches by.
template <bool GATED, int NI, bool ONCE>
__global__ void __launch_bounds__(512, 2) gemm_wide_kernel(WideArgs a) {
  WT_LDS(lds);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int tiles = a.row_tiles * a.col_tiles, die = blockIdx.x % WG_DIES, at = blockIdx.x / WG_DIES, apart = gridDim.x / WG_DIES;
  const int first = (int)((long long)tiles * die / WG_DIES), mine = (int)((long long)tiles * (die + 1) / WG_DIES) - first;
  const int rest = mine % WG_UNITS, whole = rest <= WG_UNITS / 2 ? mine - rest : mine;
  if (at < whole) wg_tiles<GATED, NI, ONCE>(a, lds, wave, first + at, apart, first + whole, -1);
  if (at < 2 * (mine - whole)) {
    __syncthreads();
    wg_tiles<GATED, (NI + 1) / 2, false>(a, lds, wave, first + whole + at / 2, 0, 0, at % 2);
  }
}

#define WG_LEAST 4  // fewest blocks of 16 rows of a wave

// What tiles of NI blocks a wave cost: microseconds a round of 4,096 k, 8,192 rows x 28,672 gated in 8 to 28 rounds (halves of fewer than four
// blocks from short products), and what a round of halves pays beside that, its first pieces not being on their way before it.
static int wg_round(int ni) {
  static const int us[WT_MOST + 1] = {0, 0, 42, 50, 57, 66, 75, 83, 90, 101, 117, 125};
  return us[ni];
}
#define WG_APART 6
struct WideCut {
  int blocks, cost;
};
// The height of the tiles whose rounds over the compute units end first.  A result's bits do not depend on it.
static WideCut wg_cut(int M, int N, bool gated) {
  const int col_tiles = ((gated ? 2 * N : N) + WT_COLS - 1) / WT_COLS;
  WideCut best = {0, 0};
  for (int ni = WG_LEAST; ni <= WT_MOST; ++ni) {
    const long long tiles = (long long)((M + 32 * ni - 1) / (32 * ni)) * col_tiles, each = (tiles + WG_DIES - 1) / WG_DIES;
    const int rest = (int)(each % WG_UNITS);
    const long long cost = each / WG_UNITS * wg_round(ni) + (rest == 0 ? 0 : rest <= WG_UNITS / 2 ? wg_round((ni + 1) / 2) + WG_APART : wg_round(ni));
    if (best.blocks == 0 || cost < best.cost) best = {ni, (int)std::min(cost, 1ll << 30)};
  }
  return best;
}

// Whether this kernel is to take a product that the library could take too, both sides in us.  Where tiles leave much of the chip idle, the library cuts K
// as well: 1,000 rows x 4,096 x 14,336 114.8 there, 123.8 here (the tiles do 0.35 of what a full chip does in their time), x 4,096 x 4,096 39.5 / 40.5,
// 500 x 6,144 x 4,096 36.6 / 39.4 (0.26), but 1,000 x 6,144 x 4,096 53.0 / 51.3 (0.52), 2,048 x 4,096 x 4,096 61.3 / 56.8 (0.71), 3,000 x 6,144 x 4,096
// 142.0 / 114.7; over a short K it is the slower one all the same (500 x 6,144 x 1,536 22.5 / 18.4, 500 x 4,096 x 2,048 21.4 / 20.8, 500 x 2,048 x 2,048
// 20.7 / 19.9).  bf16 results whose tiles of 256 x 256 fill two rounds and more to the last unit are its best: 8,192 x 4,096 x 4,096 182.6 / 186.2,
// x 14,336 598 / 626, but 8,192 x 5,120 x 3,072 (2.5 rounds) 290 / 183, 8,192 x 3,072 x 8,192 (1.5) 301 / 278.  Float32 results cost it more: 2,250 x 20,608 x 4,096
// 368 / 296, 3,000 x 6,144 x 1,536 72 / 55, 8,192 x 6,144 x 4,096 309 / 282.  Gated, beside the kernel that multiplies (before the gate's last us a tile): 2,048 x 28,672 x 4,096 340 + 36 / 331,
// 8,192 x 28,672 x 4,096 1,238 + 128 / 1,261, 500 x 28,672 x 4,096 95 + 12 / 96, 2,250 x 22,016 x 4,096 377 + 32 / 285.
extern "C" int hal_gemm_bf16_wide_pays(int M, int N, int K, int gated, int f32) {
  if (M <= 64 || N < 4 || K < 2 * WT_TK) return 0;
  const double n = gated ? 2.0 * N : N, full = (double)M * n / (256.0 * 65536.0) * wg_round(8), part = full / wg_cut(M, N, gated != 0).cost;
  const double tiles = (double)((M + 255) / 256) * ((N + 255) / 256), rounds = (tiles + 255) / 256;
  const bool exact = !gated && !f32 && rounds >= 2 && tiles >= 0.97 * 256 * (long long)rounds && M % 256 == 0 && N % 256 == 0;
  return !exact && part >= (K <= 2048 ? 0.15 : 0.5);
}

// Whether there is a form for these sizes and distances of rows; operands begin at multiples of 16 bytes besides.
extern "C" int hal_gemm_bf16_wide_takes(int M, int N, int K, int ldx, int ldw) {
  return M > 0 && N >= 4 && N % 4 == 0 && K >= 2 * WT_TK && K % (2 * WT_TK) == 0 && ldx >= K && ldw >= K && ldx % 8 == 0 && ldw % 8 == 0 && ldx < (1 << 21) &&
         ldw < (1 << 21);
}

// X [M, K], W (and W2 of a gated product: W is the gate's) [N, K] bf16, Y [M, N] of bf16 or float32.  height: blocks of 16 rows of a wave (0: as
// it is best), for tests and measurements.
extern "C" int hal_gemm_bf16_wide(const void* X, int ldx, const void* W, const void* W2, int ldw, void* Y, int ldy, int y_dtype, int act, float limit,
                                  float alpha, float up_shift, int M, int N, int K, int height, hipStream_t stream) {
  HAL_REQUIRE(hal_gemm_bf16_wide_takes(M, N, K, ldx, ldw) && ((uintptr_t)X | (uintptr_t)W | (uintptr_t)W2) % 16 == 0, "hal_gemm_bf16_wide: M=%d N=%d K=%d, rows of %d and %d, or their places", M, N, K, ldx, ldw);
  HAL_REQUIRE(ldy >= N && ldy % 4 == 0 && (uintptr_t)Y % 16 == 0, "hal_gemm_bf16_wide: results' rows of %d, or their place", ldy);
  HAL_REQUIRE(y_dtype == HAL_F32 || y_dtype == HAL_BF16, "hal_gemm_bf16_wide: result dtype %d", y_dtype);
  HAL_REQUIRE(act >= HAL_ACT_SILU && act <= HAL_ACT_CLAMPED, "hal_gemm_bf16_wide: activation %d", act);
  HAL_REQUIRE(height == 0 || (height >= WG_LEAST && height <= WT_MOST), "hal_gemm_bf16_wide: height %d", height);
  const bool gated = W2 != nullptr;
  const int ni = height ? height : wg_cut(M, N, gated).blocks, rows = 32 * ni;
  const int row_tiles = (M + rows - 1) / rows, col_tiles = ((gated ? 2 * N : N) + WT_COLS - 1) / WT_COLS;
  const long long tiles = (long long)row_tiles * col_tiles;
  HAL_REQUIRE(tiles < (1ll << 28), "hal_gemm_bf16_wide: M=%d N=%d exceed the grid limit", M, N);
  const WideArgs a = {(const bf16_t*)X, (const bf16_t*)W, (const bf16_t*)W2, ldx, ldw, Y, ldy, y_dtype == HAL_F32, M, N, K, rows, row_tiles, col_tiles,
                      {act, limit, alpha, up_shift}};
  // workgroups of a die: one a unit, or of fewer tiles one each, or two where they are cut in two
  const long long each = (tiles + WG_DIES - 1) / WG_DIES;
  const int blocks = each > WG_UNITS / 2 ? WG_UNITS : 2 * (int)each;
#define WG_LAUNCH(NI_)                                                                                                                         \
  case NI_:                                                                                                                                    \
    if (gated && once) hipLaunchKernelGGL((gemm_wide_kernel<true, NI_, true>), dim3(WG_DIES * blocks), dim3(512), 0, stream, a);                \
    else if (gated) hipLaunchKernelGGL((gemm_wide_kernel<true, NI_, false>), dim3(WG_DIES * blocks), dim3(512), 0, stream, a);                  \
    else if (once) hipLaunchKernelGGL((gemm_wide_kernel<false, NI_, true>), dim3(WG_DIES * blocks), dim3(512), 0, stream, a);                   \
    else hipLaunchKernelGGL((gemm_wide_kernel<false, NI_, false>), dim3(WG_DIES * blocks), dim3(512), 0, stream, a);                            \
    break
  const bool once = row_tiles == 1;
  switch (ni) {
    WG_LAUNCH(4);
    WG_LAUNCH(5);
    WG_LAUNCH(6);
    WG_LAUNCH(7);
    WG_LAUNCH(8);
    WG_LAUNCH(9);
    WG_LAUNCH(10);
    WG_LAUNCH(11);
  }
#undef WG_LAUNCH
  HAL_LAUNCH_CHECK();
  return 0;
}
