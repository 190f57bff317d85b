// Products in groups: Y_g = X_g * W_g^T for g = 0 .. G-1, one launch for all groups.
//
// A group is a head (every group has the same rows, its operands are column ranges of
// wider rows: the per-head projections of a latent attention) or an expert of a mixture
// (the groups' rows are slices of one sorted list of (token, choice) pairs whose bounds
// are on the device; rows of X are gathered and rows of Y scattered through index
// arrays).  W is [G, N, K] with row length ldw.  The epilogue can multiply by the sigmoid
// of a float32 gate (heads), or compute the clamped gated activation of two products
// (experts: W the gate's weight, W2 the up projection's), write float32 or bf16, or add
// into a float32 destination.  Accumulation is float32 throughout; a row's result depends
// on that row alone, up to the order in which the kernels add its terms.
//
// Five kernels.  For any element type and any sizes tiles of 64 x 64 on the vector units
// (grouped_fma_kernel).  For bf16 operands whose addresses allow 16-byte loads the matrix cores
// (v_mfma_f32_16x16x32_bf16): a kernel for at most 16 rows a group that reads both operands straight
// from memory (grouped_skinny_kernel), and tiles of 128 x 128 staged through registers and LDS
// (grouped_mfma_kernel).  Where moreover whole lines can go straight into LDS (K of whole 64s) and
// results leave as vector stores: streaming tiles of 64 x 128 for experts of few rows and for heads
// (grouped_stream_kernel), and tiles of up to 352 x 256 for prompts' experts (grouped_wide_kernel).
// gg_experts_kernel says which of the four takes an expert's product, and why.
#include "wide_tile.h"
#include "hal_api.h"
#include <math.h>

#include <algorithm>
#include <type_traits>

struct GroupedArgs {
  const void* X;
  int ldx, x_group_cols, x_col0;
  const void* W;
  const void* W2;
  long long w_group_stride;
  int ldw;
  void* Y;
  int ldy, y_group_cols, y_col0, y_dtype, y_add;
  int M, N, K, G;
  int x_rows;
  const int* group_offsets;  // [G + 1] or null
  const int* tile_offsets;   // [G + 1] with group_offsets
  const int* row_src;        // or null
  int src_div;
  const int* row_dst;  // or null
  const float* gate;   // or null
  int ldg;
  int gate_group_cols, gate_cols;  // the gate of group g, column n: gate[row][g * gate_group_cols + (gate_cols ? n : 0)]
  float limit, alpha, up_shift;
  int act;  // without W2: 0 the product as it is, 1 the square of its positive part
  int turn;  // the streaming tiles begin at different places of K
};

#define GG_ROWS 128  // rows of a workgroup's tile (what the tile offsets count in)
#define GG_TM 64     // the vector-unit kernel takes them in two halves of 64 rows, 64 columns at a time
#define GG_TN 64
#define GG_TK 16

// which group and which rows a workgroup serves; false: nothing
__device__ __forceinline__ bool gg_locate(const GroupedArgs& a, int& g, int& row0, int& row_end) {
  if (a.group_offsets == nullptr) {
    g = blockIdx.z;
    row0 = blockIdx.y * GG_ROWS;
    row_end = a.M;
    return row0 < row_end;
  }
  const int tile = blockIdx.y;
  if (tile >= a.tile_offsets[a.G]) return false;
  int lo = 0, hi = a.G;  // the last group whose first tile is <= tile
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2;
    if (a.tile_offsets[mid] <= tile) lo = mid; else hi = mid;
  }
  g = lo;
  row0 = a.group_offsets[g] + (tile - a.tile_offsets[g]) * GG_ROWS;
  row_end = a.group_offsets[g + 1];
  return row0 < row_end;
}

__device__ __forceinline__ float gg_sigmoid(float z) { return 1.0f / (1.0f + __expf(-z)); }

__device__ __forceinline__ void gg_store(const GroupedArgs& a, int g, int i, int n, float v, float v2,
                                         bool gated) {
  if (gated) {
    const float gg = fminf(v, a.limit);
    const float uu = fminf(fmaxf(v2, -a.limit), a.limit);
    v = gg * gg_sigmoid(a.alpha * gg) * (uu + a.up_shift);
  }
  if (!gated && a.act == 1) {
    v = fmaxf(v, 0.f);
    v = v * v;
  }
  const int dst = a.row_dst ? a.row_dst[i] : i;
  const size_t col = (size_t)g * a.y_group_cols + a.y_col0 + n;
  if (a.gate) v *= gg_sigmoid(a.gate[(size_t)dst * a.ldg + (size_t)g * a.gate_group_cols + (a.gate_cols ? n : 0)]);
  const size_t at = (size_t)dst * a.ldy + col;
  if (a.y_dtype == HAL_F32) {
    float* y = (float*)a.Y;
    y[at] = a.y_add ? y[at] + v : v;
  } else {
    ((bf16_t*)a.Y)[at] = f32_to_bf16(v);
  }
}

template <typename T, bool GATED>
__global__ void __launch_bounds__(256) grouped_fma_kernel(GroupedArgs a) {
  int g, row0, row_end;
  if (!gg_locate(a, g, row0, row_end)) return;
  row0 += (blockIdx.x % (GG_ROWS / GG_TM)) * GG_TM;  // which half of the tile's rows
  if (row0 >= row_end) return;
  const int n0 = (blockIdx.x / (GG_ROWS / GG_TM)) * GG_TN;
  __shared__ float As[GG_TK][GG_TM + 4];
  __shared__ float Bs[GG_TK][GG_TN + 4];
  __shared__ float B2s[GATED ? GG_TK : 1][GG_TN + 4];
  __shared__ int src_rows[GG_TM];
  const int tid = threadIdx.x;
  if (tid < GG_TM) {
    const int i = row0 + tid;
    int s = -1;
    if (i < row_end) s = a.row_src ? a.row_src[i] / a.src_div : i;
    src_rows[tid] = s;
  }
  __syncthreads();
  const T* X = (const T*)a.X + (size_t)g * a.x_group_cols + a.x_col0;
  const T* W = (const T*)a.W + (size_t)g * a.w_group_stride;
  const T* W2 = GATED ? (const T*)a.W2 + (size_t)g * a.w_group_stride : nullptr;
  const int tm = (tid / 16) * 4, tn = (tid % 16) * 4;
  float acc[4][4] = {}, acc2[4][4] = {};
  // a thread brings element (r, kk) of each tile, r = tid / 4 (+ 0), kk = (tid % 4) * 4 .. + 3
  const int lr = tid / 4, lk = (tid % 4) * 4;
  for (int k0 = 0; k0 < a.K; k0 += GG_TK) {
    const int s = src_rows[lr];
    const int n = n0 + lr;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = k0 + lk + j;
      const bool kin = k < a.K;
      As[lk + j][lr] = (s >= 0 && kin) ? to_f32(X[(size_t)s * a.ldx + k]) : 0.f;
      Bs[lk + j][lr] = (n < a.N && kin) ? to_f32(W[(size_t)n * a.ldw + k]) : 0.f;
      if (GATED) B2s[lk + j][lr] = (n < a.N && kin) ? to_f32(W2[(size_t)n * a.ldw + k]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GG_TK; ++kk) {
      float av[4], bv[4], b2v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        av[i] = As[kk][tm + i];
        bv[i] = Bs[kk][tn + i];
        if (GATED) b2v[i] = B2s[kk][tn + i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          acc[i][j] = fmaf(av[i], bv[j], acc[i][j]);
          if (GATED) acc2[i][j] = fmaf(av[i], b2v[j], acc2[i][j]);
        }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = row0 + tm + i;
    if (r >= row_end) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tn + j;
      if (n < a.N) gg_store(a, g, r, n, acc[i][j], acc2[i][j], GATED);
    }
  }
}

typedef __attribute__((ext_vector_type(8))) __bf16 gg_bf16x8;
typedef __attribute__((ext_vector_type(4))) float gg_f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t gg_u32x4;

__device__ __forceinline__ gg_bf16x8 gg_frag(const bf16_t* p, bool valid) {
  gg_u32x4 raw = {0u, 0u, 0u, 0u};
  if (valid) raw = *(const gg_u32x4*)p;
  return __builtin_bit_cast(gg_bf16x8, raw);
}

// bf16 on the matrix cores: a workgroup of four waves takes 128 rows x 128 columns, a wave
// 64 x 64 (sixteen 16 x 16 results).  K goes through LDS 64 at a time: every thread brings
// 16-byte pieces (eight k of one row) of the X rows and of the W rows, the next stage's while
// this one is multiplied, and puts them down in the instruction's operand order, so that a
// wave reads an operand (16 rows x 32 k) as one contiguous KiB: lane l holds row l % 16 and
// the eight k from (l / 16) * 8 on.  Lane l of a result holds W row (column) l % 16 and the
// X rows 4 * (l / 16) .. + 3, so a store instruction writes runs of 16 neighbouring columns.
// K, ldx, ldw and the column offsets are multiples of 8 and the bases 16-byte aligned.
#define GM_TK 64
// Where the piece of eight k (q of four in step ks of 32 k) of row r of a 16-row tile lies in
// the tile-step's KiB: at lane q * 16 + r of the operand, with r's bits turned by q and ks, so
// that the sixteen lanes of a store (two rows, eight pieces) meet sixteen different banks, and
// the sixteen lanes of a load (one q, sixteen rows) still read one contiguous quarter KiB.
__device__ __forceinline__ int gm_slot(int q, int r, int ks) { return q * 16 + (r ^ (q << 2) ^ (ks << 1)); }
__device__ __forceinline__ int gm_lds_offset(int row, int kc) {  // kc: which piece of eight k
  return (((row / 16) * (GM_TK / 32) + kc / 4) * 64 + gm_slot(kc % 4, row % 16, kc / 4)) * 8;
}

// GATED: the tile's 128 W rows are, for each of the two column halves of the waves, 32 rows of
// the gate's weight and the same 32 rows of the up projection's, so a wave holds both products
// of its 32 result columns at the same lanes and the workgroup writes 64 columns.
template <bool GATED>
__global__ void __launch_bounds__(256, 2) grouped_mfma_kernel(GroupedArgs a) {
  int g, row0, row_end;
  if (!gg_locate(a, g, row0, row_end)) return;
  constexpr int COLS = GATED ? GG_ROWS / 2 : GG_ROWS;  // result columns of a workgroup
  constexpr int WCOLS = COLS / 2;                      // of a wave
  const int n0 = blockIdx.x * COLS;
  __shared__ __attribute__((aligned(16))) bf16_t As[GG_ROWS * GM_TK];
  __shared__ __attribute__((aligned(16))) bf16_t Bs[GG_ROWS * GM_TK];
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int wm = wave / 2, wn = wave % 2;
  const bf16_t* X = (const bf16_t*)a.X + (size_t)g * a.x_group_cols + a.x_col0;
  const bf16_t* W = (const bf16_t*)a.W + (size_t)g * a.w_group_stride;
  const bf16_t* W2 = GATED ? (const bf16_t*)a.W2 + (size_t)g * a.w_group_stride : nullptr;
  // the four pieces a thread brings of each operand: rows tid / 8 + 32 i, piece tid % 8
  const int kc = tid % 8;
  const bf16_t* xp[4];
  const bf16_t* wp[4];
  int at[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = tid / 8 + 32 * i;
    at[i] = gm_lds_offset(row, kc);
    const int r = row0 + row;
    xp[i] = nullptr;
    if (r < row_end) xp[i] = X + (size_t)(a.row_src ? a.row_src[r] / a.src_div : r) * a.ldx + kc * 8;
    int n = n0 + row;
    const bf16_t* from = W;
    if (GATED) {
      n = n0 + (row / 64) * WCOLS + row % WCOLS;
      if (row % 64 >= WCOLS) from = W2;
    }
    wp[i] = n < a.N ? from + (size_t)n * a.ldw + kc * 8 : nullptr;
  }
  gg_u32x4 rx[4], rw[4];
  auto bring = [&](int k0) {
    const bool kin = k0 + kc * 8 < a.K;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      rx[i] = gg_u32x4{0u, 0u, 0u, 0u};
      rw[i] = gg_u32x4{0u, 0u, 0u, 0u};
      if (xp[i] && kin) rx[i] = *(const gg_u32x4*)(xp[i] + k0);
      if (wp[i] && kin) rw[i] = *(const gg_u32x4*)(wp[i] + k0);
    }
  };
  gg_f32x4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = gg_f32x4{0.f, 0.f, 0.f, 0.f};
  const bool active = row0 + wm * 64 < row_end && n0 + wn * WCOLS < a.N;  // a wave without rows or columns only carries
  bring(0);
  for (int k0 = 0; k0 < a.K; k0 += GM_TK) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *(gg_u32x4*)&As[at[i]] = rx[i];
      *(gg_u32x4*)&Bs[at[i]] = rw[i];
    }
    __syncthreads();
    if (k0 + GM_TK < a.K) bring(k0 + GM_TK);
    if (active) {
#pragma unroll
      for (int ks = 0; ks < GM_TK / 32; ++ks) {
        gg_bf16x8 xa[4], wa[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int slot = gm_slot(lane / 16, lane % 16, ks);
          xa[i] = *(const gg_bf16x8*)&As[(((wm * 4 + i) * (GM_TK / 32) + ks) * 64 + slot) * 8];
          wa[i] = *(const gg_bf16x8*)&Bs[(((wn * 4 + i) * (GM_TK / 32) + ks) * 64 + slot) * 8];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[i], wa[j], acc[i][j], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  if (!active) return;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const int r = row0 + wm * 64 + i * 16 + (lane / 16) * 4 + jj;
      if (r >= row_end) continue;
#pragma unroll
      for (int j = 0; j < (GATED ? 2 : 4); ++j) {
        const int n = n0 + wn * WCOLS + j * 16 + lane % 16;
        if (n < a.N) gg_store(a, g, r, n, acc[i][j][jj], GATED ? acc[i][j + 2][jj] : 0.f, GATED);
      }
    }
}

// The experts' products of prompts (rows sorted by group): tiles of up to 352 rows x 256 W rows (GATED:
// 128 of the gate's weight and the same 128 of the up projection's) by eight waves, a wave half the
// tile's rows x 64 W rows, one workgroup a compute unit.
//
// What bounds it: weights that come from memory while the matrix cores work at the clock that the chip holds under them.  Tiles are as large as
// the registers hold, so that an expert's rows make one or two, and wide_tile.h says how a tile's steps go.  (4,000 to 5,440 rows of 4096 x 4096 in one round take 104 to
// 136 us as rows of one group and 148 to 158 as rows of 16, whose 537 MB of weights take 106 at the memory's rate.)  Weights' rows are a power of two apart and
// meet in a few of the memory's channels: rows a line further apart made prompts' products 5% faster, and those of decode steps, whose kernel reads whole
// matrices in their order, 7% slower.
//
// A group's rows are cut into the fewest tiles of at most so many rows (gw_height) and these are made equally high,
// in steps of 32 rows, so that workgroups take equally long.  Workgroup b runs on compute die b % 8, and
// each die has an L2 of its own, so die x takes the x-th eighth of the list of all tiles, which goes
// through a group's row tiles (eight at a time) column by column: one die reads an expert's weights,
// once (tiles of two experts side by side cost a third more reads from memory and 8% of the time).
//
// Measured beside a schedule in which every wave read, loaded and multiplied for itself with one barrier a step, us: 9,000 rows of 16 experts, 4096 x 4096 302 ->
// 280 (1,080 TFLOP/s; tiles of 128 x 128 in registers and LDS 469); 18,000 rows of 64, gate and up 1024 x 4096 each, 330 -> 320; 49,152 rows 730 -> 698;
// 2,400 rows of 8, gate and up 14336 x 4096, 554 -> 551; 3,600 rows of 64 249 -> 234; 16 groups of 60, 128, 210, 280 and 340 rows 133 -> 129, 137 -> 135, 155 -> 150, 167 -> 159, 181 -> 170.
// The weights of a group with one row tile, which are read once, pass the caches by (with two or three row tiles side by side 2 to 3% slower): 16 groups of 60, 210, 280 and 340 rows
// 129 -> 120, 150 -> 133, 159 -> 136, 170 -> 147; 18,000 rows of 64, gate and up 320 -> 305, down 227 -> 219; 2,400 of 8 551 -> 530.
#define GW_ROWS 352
#define GW_COLS 256
#define GW_TK 64
#define GW_PANEL 8
#define GG_UNITS 256  // compute units of the gfx950 parts that this library is built for

// column n and the three behind it of the row that goes to row dst
template <bool GATED>
__device__ __forceinline__ void gw_store(const GroupedArgs& a, int dst, int n, gg_f32x4 v, gg_f32x4 v2) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (GATED) {
      const float gg = fminf(v[j], a.limit);
      const float uu = fminf(fmaxf(v2[j], -a.limit), a.limit);
      v[j] = gg * gg_sigmoid(a.alpha * gg) * (uu + a.up_shift);
    } else if (a.act == 1) {
      const float p = fmaxf(v[j], 0.f);
      v[j] = p * p;
    }
  }
  const size_t at = (size_t)dst * a.ldy + a.y_col0 + n;
  if (a.y_dtype == HAL_F32) *(gg_f32x4*)((float*)a.Y + at) = v;
  else *(uint2*)((bf16_t*)a.Y + at) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
}

// The rows of X, K columns from `col0` on: up to the end of the last row's, so that rows that overlap (a row
// length below K, or 0 where one row stands for all) lie in the range like any others.
__device__ __forceinline__ hal_memory gw_rows_of_x(const GroupedArgs& a, int col0) {
  return hal_memory_at((const bf16_t*)a.X + col0, ((uint32_t)(a.x_rows - 1) * a.ldx + a.K) * 2);
}

// The lane's number, counted anew at every call: kept over a tile's products, it and what follows from it would take registers.
__device__ __forceinline__ int gw_lane() {
  int zero = 0;
  asm volatile("" : "+v"(zero));
  return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, zero));
}

// What one wave does for a tile of at most 32 * NI rows.  ONCE: the group has one row tile, so that its weights are read once.
template <bool GATED, int NI, bool ONCE>
__device__ __forceinline__ void gw_wave(const GroupedArgs& a, int wave, int g, int row0, int row_end, int n0, const wt_lds& lds) {
  using P = wt_part<NI>;
  const int lane = gw_lane(), oct = lane / 8, c = ((lane % 8) ^ hal_turn(wave % 2 * 8 + oct)) * 16;
  const size_t w_at = (size_t)g * a.w_group_stride;
  const hal_memory W = hal_memory_at((const bf16_t*)a.W + w_at, (uint32_t)a.N * a.ldw * 2);
  const hal_memory W2 = hal_memory_at((const bf16_t*)(GATED ? a.W2 : a.W) + w_at, (uint32_t)a.N * a.ldw * 2);
  const hal_memory X = gw_rows_of_x(a, a.x_col0);
  const int last = a.K / GW_TK - 1;
  // rows past the end are read from the last one, columns as zeros: nothing of them is stored
  uint32_t xo[P::loads(0) + P::loads(1)];
#pragma unroll
  for (int p = 0; p < 2; ++p)
#pragma unroll
    for (int u = 0; u < P::loads(p); ++u) {
      int r = row0 + wt_octet_row<NI>(wt_octet<NI>(wave, p, u), p) + oct;
      r = r < row_end ? r : row_end - 1;
      uint32_t& to = xo[p * P::loads(0) + u];
      to = (uint32_t)(a.row_src ? a.row_src[r] / a.src_div : r) * (uint32_t)(a.ldx * 2) + c;
      asm("v_mov_b32 %0, %1" : "=v"(to) : "v"(to));  // (one register, not the pair that a multiplication with addition writes)
    }
  // (GATED: of a wave's 64 W rows the first 32 are the gate's and the others the up projection's)
  const uint32_t row = (uint32_t)a.ldw * 2, wo = (uint32_t)(n0 + (GATED ? wave * 8 : wave / 4 * 64 + wave % 4 * 8) + oct) * row + c;
  auto bring_x = [&](auto part, char* to, int step) {
    constexpr int p = decltype(part)::value;
#pragma unroll
    for (int u = 0; u < P::loads(p); ++u) hal_load_lds(X, xo[p * P::loads(0) + u], (uint32_t)min(step, last) * (GW_TK * 2), to + wt_octet<NI>(wave, p, u) * 1024);
  };
  auto bring_w = [&](int half, char* to, int step) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
      hal_load_lds<ONCE ? HAL_ONCE : 0>(half ? W2 : W, wo + (GATED ? u * 64 : u * 128 + half * 32) * row, (uint32_t)min(step, last) * (GW_TK * 2), to + (wave + 8 * u) * 1024);
  };
  gg_f32x4 acc[NI][4];
  wt_begin<NI>(lds, bring_x, bring_w);
  wt_steps<NI>(lds, wave, lane, last + 1, acc, bring_x, bring_w);
  wt_end();
  const int end_lane = gw_lane();
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = row0 + (wave / 4 * NI + i) * 16 + end_lane % 16;
    if (r >= row_end) continue;
    const int dst = a.row_dst ? a.row_dst[r] : r;
#pragma unroll
    for (int j = 0; j < (GATED ? 2 : 4); ++j) {
      const int n = n0 + wave % 4 * (GATED ? 32 : 64) + j * 16 + end_lane / 16 * 4;
      if (n < a.N) gw_store<GATED>(a, dst, n, acc[i][j], GATED ? acc[i][j + 2] : acc[i][j]);
    }
  }
}

// Which tile is a workgroup's `turn`-th, written to `found` (group, first row, end row, column tile, whether
// there is one more after it, whether the group has no other row tile; group -1: none),
// by its first wave: the groups' rows in tiles of at most `most`, equally high in steps of 32.  A lane counts a
// run of neighbouring groups (one where there are up to 64), so that one sum over the wave serves any number:
// 64 at a time, 512 groups of 512 x 2048 (gate and up) took 27.9 us for 3 tokens of 10 and 69.0 for 8, now 23.4 and 62.7.
__device__ __forceinline__ void gw_find(const GroupedArgs& a, int most, int col_tiles, int turn, int* found) {
  const int lane = gw_lane();
  const int each = (a.G + 63) / 64;
  const int first = min(a.G, lane * each), last = min(a.G, first + each);
  auto tiles_of = [&](int g) { return (a.group_offsets[g + 1] - a.group_offsets[g] + most - 1) / most; };
  int mine = 0;
  for (int g = first; g < last; ++g) mine += tiles_of(g);
  int upto = mine;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int v = __shfl_up(upto, off, 64);
    if (lane >= off) upto += v;
  }
  const long long units = (long long)__shfl(upto, 63, 64) * col_tiles;
  const int die = blockIdx.x % 8;
  const long long unit = units * die / 8 + blockIdx.x / 8 + (long long)turn * (gridDim.x / 8), end_of_die = units * (die + 1) / 8;
  if (lane == 0) found[0] = -1, found[4] = unit + gridDim.x / 8 < end_of_die;
  if (unit >= end_of_die) return;
  int before = upto - mine;  // row tiles of the groups before
  if (unit < (long long)before * col_tiles || unit >= (long long)upto * col_tiles) return;
  for (int g = first; g < last; ++g) {  // (one lane: its groups have the tile)
    const int begin = a.group_offsets[g], end = a.group_offsets[g + 1], n = (end - begin + most - 1) / most;
    if (unit < (long long)(before + n) * col_tiles) {
      const int in_group = (int)(unit - (long long)before * col_tiles);
      const int panel = in_group / (GW_PANEL * col_tiles), in_panel = in_group % (GW_PANEL * col_tiles);
      const int high = min(GW_PANEL, n - panel * GW_PANEL);         // row tiles of this panel
      const int rows = ((end - begin + n - 1) / n + 31) / 32 * 32;  // of each of the group's tiles
      found[0] = g;
      found[1] = begin + (panel * GW_PANEL + in_panel % high) * rows;
      found[2] = min(end, found[1] + rows);
      found[3] = in_panel / high;
      found[5] = n == 1;
      return;
    }
    before += n;
  }
}

// How high the wide tiles may be is chosen from the groups' sizes: the least of rounds of tiles, one a compute unit,
// times what the highest tile asks of the second-level cache (X and W rows of a step: its rows and GW_COLS).  A result's
// bits do not depend on it.  One group over a tile's height can be one more round: 18,000 rows dealt to 64 experts
// at random (281 +- 17 each), gate and up, took 387 us in tiles of at most 320 rows (just over two rounds), 391 of at most
// 256 (four of half the height), and now, of at most 352, 311.
// (The first wave's work; the same in all its lanes.)
#define GW_HEIGHTS 4
#define GW_LEAST_ROWS 192
__device__ __forceinline__ int gw_height(const GroupedArgs& a, int col_tiles) {
  constexpr int heights[GW_HEIGHTS] = {GW_ROWS, 320, 256, GW_LEAST_ROWS};
  const int lane = threadIdx.x % 64, each = (a.G + 63) / 64;
  const int first = min(a.G, lane * each), last = min(a.G, first + each);
  int tiles[GW_HEIGHTS] = {}, high[GW_HEIGHTS] = {}, most = 0;
  for (int g = first; g < last; ++g) {
    const int rows = a.group_offsets[g + 1] - a.group_offsets[g];
    most = max(most, rows);
#pragma unroll
    for (int h = 0; h < GW_HEIGHTS; ++h) {
      const int n = max(1, (rows + heights[h] - 1) / heights[h]);
      tiles[h] += rows > 0 ? n : 0;
      high[h] = max(high[h], (rows + n - 1) / n);
    }
  }
  if (!__any(most > GW_LEAST_ROWS)) return GW_ROWS;  // (they are all the same)
  int best = 0;
  long long least = 0;
#pragma unroll
  for (int h = 0; h < GW_HEIGHTS; ++h) {
#pragma unroll
    for (int off = 32; off; off >>= 1) {
      tiles[h] += __shfl_xor(tiles[h], off, 64);
      high[h] = max(high[h], __shfl_xor(high[h], off, 64));
    }
    const long long cost = ((long long)tiles[h] * col_tiles + GG_UNITS - 1) / GG_UNITS * ((high[h] + 31) / 32 * 32 + GW_COLS);
    if (h == 0 || cost < least) best = heights[h], least = cost;
  }
  return best;
}

template <bool GATED>
__global__ void __launch_bounds__(512, 2) grouped_wide_kernel(GroupedArgs a, int col_tiles) {
  WT_LDS(lds);
  __shared__ __attribute__((aligned(64))) int found[6];
  __shared__ int most;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  if (wave == 0) most = gw_height(a, col_tiles);
  // (as many workgroups as tiles of GW_ROWS can be, and one a compute unit: lower ones are some workgroups' second)
  for (int turn = 0;; ++turn) {
    __syncthreads();  // the tile before is done with the buffers and `found`
    if (wave == 0) gw_find(a, most, col_tiles, turn, found);
    __syncthreads();
    const int g = __builtin_amdgcn_readfirstlane(found[0]), more = __builtin_amdgcn_readfirstlane(found[4]);
    if (g < 0) return;
    const int row0 = __builtin_amdgcn_readfirstlane(found[1]), row_end = __builtin_amdgcn_readfirstlane(found[2]);
    const int n0 = __builtin_amdgcn_readfirstlane(found[3]) * (GATED ? GW_COLS / 2 : GW_COLS);
    const int rows = row_end - row0, once = __builtin_amdgcn_readfirstlane(found[5]);
    // (equal heights in steps of 32 can leave a group's last tile empty)
#define GW_WAVE(NI_)                                                             \
  do {                                                                           \
    if (once) gw_wave<GATED, NI_, true>(a, wave, g, row0, row_end, n0, lds);      \
    else gw_wave<GATED, NI_, false>(a, wave, g, row0, row_end, n0, lds);          \
  } while (0)
    if (rows <= 0);
    else if (rows <= 64) GW_WAVE(2);
    else if (rows <= 128) GW_WAVE(4);
    else if (rows <= 160) GW_WAVE(5);
    else if (rows <= 192) GW_WAVE(6);
    else if (rows <= 224) GW_WAVE(7);
    else if (rows <= 256) GW_WAVE(8);
    else if (rows <= 288) GW_WAVE(9);
    else if (rows <= 320) GW_WAVE(10);
    else GW_WAVE(11);
#undef GW_WAVE
    if (!more) return;
  }
}

// Groups of few rows (decode steps, short prompts): what counts is that the weights come at the memory's
// rate, and come once.  Tiles of at most 64 rows x 128 W rows (GATED: 64 and 64) by four waves, a wave all
// rows x 32 W rows; whole lines straight into three LDS buffers, two steps of 64 k under way while one is
// multiplied, and two workgroups a compute unit.
// Measured beside grouped_skinny_kernel, whose loads take half lines and which goes through the weights
// once for every 16 rows, events around the call: 48 tokens, 4 of 16 experts of 4096 x 4096 (537 MB): 143 ->
// 106 us; 16 tokens: 113 -> 104; 64 tokens: 178 -> 107; 48 tokens, 6 of 64 experts of 1024 x 4096, gate and
// up: 211 -> 184.  All workgroups at one place of K (see `begin`): 122 instead of 106.
// The weights of a group with one row tile pass the caches by, those of a group with several, side by side, do not.  None / all of groups of fewer than 48
// rows on average / by group, us: 2,500 rows, 12 of 64 groups of 150, down of 4096 x 1024 123 / 139 / 120, gate and up of 1024 x 4096 220 / 213 / 210; 500
// rows of 16 groups of 4096 x 4096, one of 300, 113 / 108 / 105; 900 rows of those, evenly, 111 / 111 / 101; 384 rows of 64, evenly, 182 / 161 / 162.
#define GT_ROWS 64
#define GT_ROWS_A_GROUP 48  // the streaming tiles are for fewer rows a group, on average
#define GT_COLS 128
#define GT_A_BYTES (GT_ROWS * GW_TK * 2)
#define GT_BUFFER ((GT_ROWS + GT_COLS) * GW_TK * 2)
// HEADS: every group has all rows, columns of its own in X and Y, and perhaps a gate on its result.  The
// tiles' shape is as good for many rows there, as K is a head's few hundred and the rows are what is read:
// 32 heads of K = 192, N = 128 with a gate: 17 rows 13.6 -> 8.0 us, 64 26.0 -> 9.6, 1,000 38.7 -> 15.2, 3,000
// 51.6 -> 34.6 beside the tiles of 128 (K = 128, N = 192: 10.1 -> 6.6, 17.2 -> 7.7, 21.3 -> 15.5, 41.5 -> 36.4),
// whose loads go through registers and wait for each other.
// A K of one step has no loads on their way while another step is multiplied: 128 heads of 64 x 64, 4,000 rows 67.3 us
// against 67.6, but 8,000 rows 131 / 121.
#define GT_ONE_STEP_ROWS 4096
typedef __attribute__((ext_vector_type(4), aligned(4))) float gt_f32x4_any;  // (a gate's rows begin at any float)
// ONCE: the group has one row tile, so that its weights are read once.
template <bool GATED, bool HEADS, bool ONCE, int NI>
__device__ __forceinline__ void gt_wave(const GroupedArgs& a, int g, int row0, int row_end, int n0, char* b0, char* b1,
                                        char* b2) {
  constexpr int AI = NI / 2, LOADS = AI + 4;
  const int steps = a.K / GW_TK;
  // Few rows: workgroups begin at different places of K and go round, since rows of W that lie a power of two
  // apart, all read at one place of K at a time, meet in a few of the memory's channels.  (Prompts' products add in
  // the order of K, as in the other tiles: their bits do not depend on which of the three the rows' number takes.)
  const int begin = a.turn ? (n0 / (GATED ? GT_COLS / 2 : GT_COLS) * 7 + g * 13) % steps : 0;
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int lr = wave * 8 + lane / 8, c = ((lane % 8) ^ hal_turn(lr % 16)) * 16;
  // (GATED: of every 32 W rows, a wave's, the first 16 are the gate's and the others the up projection's)
  const void* w0 = GATED && wave % 4 >= 2 ? a.W2 : a.W;
  const hal_memory W = hal_memory_at((const bf16_t*)w0 + (size_t)g * a.w_group_stride, (uint32_t)a.N * a.ldw * 2);
  const hal_memory X = gw_rows_of_x(a, a.x_col0 + (HEADS ? g * a.x_group_cols : 0));
  uint32_t xo[AI], wo[4];
#pragma unroll
  for (int i = 0; i < AI; ++i) {
    int r = row0 + lr + 32 * i;
    r = r < row_end ? r : row_end - 1;
    xo[i] = (uint32_t)(a.row_src ? a.row_src[r] / a.src_div : r) * (uint32_t)(a.ldx * 2) + c;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    int n = GATED ? n0 + i * 16 + lr % 16 : n0 + i * 32 + lr;
    n = n < a.N ? n : a.N - 1;
    wo[i] = (uint32_t)n * (uint32_t)(a.ldw * 2) + c;
  }
  auto bring = [&](char* lds, int step) {
    step = (step < steps ? step : steps - 1) + begin;
    const uint32_t at = (uint32_t)(step < steps ? step : step - steps) * (GW_TK * 2);
#pragma unroll
    for (int i = 0; i < AI; ++i) hal_load_lds(X, xo[i], at, lds + (i * 4 + wave) * 1024);
#pragma unroll
    for (int i = 0; i < 4; ++i) hal_load_lds<ONCE ? HAL_ONCE : 0>(W, wo[i], at, lds + GT_A_BYTES + (i * 4 + wave) * 1024);
  };
  const int q = lane / 16, r16 = lane % 16;
  const int get[2] = {r16 * 128 + (q ^ hal_turn(r16)) * 16, r16 * 128 + ((q + 4) ^ hal_turn(r16)) * 16};
  gg_f32x4 acc[NI][2];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = gg_f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](const char* lds) {
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      gg_bf16x8 w[2], x[NI];
#pragma unroll
      for (int j = 0; j < 2; ++j) w[j] = *(const gg_bf16x8*)(lds + GT_A_BYTES + (wave * 2 + j) * 2048 + get[half]);
#pragma unroll
      for (int i = 0; i < NI; ++i) x[i] = *(const gg_bf16x8*)(lds + i * 2048 + get[half]);
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j], x[i], acc[i][j], 0, 0, 0);
    }
  };
  // the steps that do not fill a turn through the buffers, one at a time
  const int odd = steps % 3;
  for (int s = 0; s < odd; ++s) {
    bring(b0, s);
    hal_meet<0>();
    multiply(b0);
    hal_meet<0>();
  }
  bring(b0, odd);
  bring(b1, odd + 1);
  auto advance = [&](int s, const char* mine, char* free) {
    hal_meet<LOADS>();  // (this step's pieces are there, the next one's may be on their way)
    bring(free, s + 2);
    multiply(mine);
  };
  for (int s = odd; s < steps; s += 3) {
    advance(s, b0, b2);
    advance(s + 1, b1, b0);
    advance(s + 2, b2, b1);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // LDS is not given back while loads are on their way into it
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = row0 + i * 16 + r16;
    if (r >= row_end) continue;
    const int dst = a.row_dst ? a.row_dst[r] : r;
#pragma unroll
    for (int j = 0; j < (GATED ? 1 : 2); ++j) {
      const int n = n0 + wave * (GATED ? 16 : 32) + j * 16 + q * 4;
      if (n >= a.N) continue;
      if (HEADS && a.gate) {
        const float* at = a.gate + (size_t)dst * a.ldg + (size_t)g * a.gate_group_cols + (a.gate_cols ? n : 0);
        gt_f32x4_any by;
        if (a.gate_cols) by = *(const gt_f32x4_any*)at;
        else by = gt_f32x4_any{at[0], at[0], at[0], at[0]};
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[i][j][v] *= gg_sigmoid(by[v]);
      }
      gw_store<GATED>(a, dst, (HEADS ? g * a.y_group_cols : 0) + n, acc[i][j], GATED ? acc[i][1] : acc[i][j]);
    }
  }
}

// ONE: there are so few rows that every group has one tile, and no second form of the loop (8 requests of six experts each, a step of four layers:
// 1,088 us, with both forms 1,092 to 1,097).
template <bool GATED, bool HEADS, bool ONE>
__global__ void __launch_bounds__(256, 2) grouped_stream_kernel(GroupedArgs a, int col_tiles) {
  __shared__ __attribute__((aligned(16))) char b0[GT_BUFFER], b1[GT_BUFFER], b2[GT_BUFFER];
  __shared__ __attribute__((aligned(64))) int found[6];
  int g, row0, row_end, col, once = ONE;
  if (HEADS) {
    // a die takes neighbouring heads, a head's columns beside each other: they read the same rows
    const int in_group = (a.M + GT_ROWS - 1) / GT_ROWS * col_tiles, die = blockIdx.x % 8;
    const long long units = (long long)a.G * in_group, unit = units * die / 8 + blockIdx.x / 8;
    if (unit >= units * (die + 1) / 8) return;
    g = (int)(unit / in_group), row0 = (int)(unit % in_group) / col_tiles * GT_ROWS;
    row_end = min(a.M, row0 + GT_ROWS), col = (int)(unit % in_group) % col_tiles;
  } else {
    if (threadIdx.x < 64) gw_find(a, GT_ROWS, col_tiles, 0, found);
    __syncthreads();
    g = __builtin_amdgcn_readfirstlane(found[0]);
    if (g < 0) return;
    row0 = __builtin_amdgcn_readfirstlane(found[1]), row_end = __builtin_amdgcn_readfirstlane(found[2]);
    col = __builtin_amdgcn_readfirstlane(found[3]);
    if (!ONE) once = __builtin_amdgcn_readfirstlane(found[5]);
  }
  const int n0 = col * (GATED ? GT_COLS / 2 : GT_COLS);
  const int rows = row_end - row0;
  if (rows <= 0) return;
#define GT_WAVE(NI_)                                                                             \
  do {                                                                                           \
    if (ONE || (!HEADS && once)) gt_wave<GATED, HEADS, !HEADS, NI_>(a, g, row0, row_end, n0, b0, b1, b2); \
    else gt_wave<GATED, HEADS, false, NI_>(a, g, row0, row_end, n0, b0, b1, b2);                  \
  } while (0)
  if (rows <= 32) GT_WAVE(2);
  else GT_WAVE(4);
#undef GT_WAVE
}

// bf16, few rows a group (decode steps): a workgroup takes 64 rows of W (GATED: 32 of the
// gate's weight and the same 32 of the up projection's) and the tile's rows 16 at a time.  Its
// four waves split K between them and read both operands straight from memory in the
// instruction's operand order, four steps of 32 k in flight at a time and no barrier on the
// way; their sums meet in LDS and are added in rising wave number.
#define GS_U 4
template <bool GATED>
__global__ void __launch_bounds__(256) grouped_skinny_kernel(GroupedArgs a) {
  int g, row0, row_end;
  if (!gg_locate(a, g, row0, row_end)) return;
  constexpr int COLS = GATED ? 32 : 64;
  const int n0 = blockIdx.x * COLS;
  __shared__ __attribute__((aligned(16))) float red[4][4][256];
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int r = lane % 16, q = lane / 16;
  const bf16_t* X = (const bf16_t*)a.X + (size_t)g * a.x_group_cols + a.x_col0;
  const bf16_t* W = (const bf16_t*)a.W + (size_t)g * a.w_group_stride;
  const bf16_t* W2 = GATED ? (const bf16_t*)a.W2 + (size_t)g * a.w_group_stride : nullptr;
  const bf16_t* wrow[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    const int n = n0 + (GATED ? f % 2 : f) * 16 + r;
    const bf16_t* from = (GATED && f >= 2) ? W2 : W;
    wrow[f] = n < a.N ? from + (size_t)n * a.ldw + q * 8 : nullptr;
  }
  const int steps = (a.K + 31) / 32;
  const int s_begin = (int)((long long)steps * wave / 4), s_end = (int)((long long)steps * (wave + 1) / 4);
  for (int r0 = row0; r0 < row_end; r0 += 16) {
    const int i = r0 + r;
    const bf16_t* xrow = nullptr;
    if (i < row_end) xrow = X + (size_t)(a.row_src ? a.row_src[i] / a.src_div : i) * a.ldx + q * 8;
    gg_f32x4 acc[4];
#pragma unroll
    for (int f = 0; f < 4; ++f) acc[f] = gg_f32x4{0.f, 0.f, 0.f, 0.f};
    for (int step = s_begin; step < s_end; step += GS_U) {
      gg_bf16x8 xa[GS_U], wa[GS_U][4];
#pragma unroll
      for (int u = 0; u < GS_U; ++u) {
        const int k = (step + u) * 32;
        const bool kin = step + u < s_end && k + q * 8 < a.K;
        xa[u] = gg_frag(xrow + k, kin && xrow != nullptr);
#pragma unroll
        for (int f = 0; f < 4; ++f) wa[u][f] = gg_frag(wrow[f] + k, kin && wrow[f] != nullptr);
      }
#pragma unroll
      for (int u = 0; u < GS_U; ++u)
#pragma unroll
        for (int f = 0; f < 4; ++f)
          acc[f] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[u], wa[u][f], acc[f], 0, 0, 0);
    }
#pragma unroll
    for (int f = 0; f < 4; ++f) *(gg_f32x4*)&red[wave][f][lane * 4] = acc[f];
    __syncthreads();
    // wave w adds up result w of all waves (GATED: waves 0 and 1, each the gate's and the up's)
    if (wave < (GATED ? 2 : 4)) {
      gg_f32x4 sum = gg_f32x4{0.f, 0.f, 0.f, 0.f}, sum2 = gg_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        sum += *(const gg_f32x4*)&red[w][wave][lane * 4];
        if (GATED) sum2 += *(const gg_f32x4*)&red[w][wave + 2][lane * 4];
      }
      const int n = n0 + wave * 16 + r;
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const int row = r0 + q * 4 + jj;
        if (row < row_end && n < a.N) gg_store(a, g, row, n, sum[jj], sum2[jj], GATED);
      }
    }
    __syncthreads();
  }
}

// The most tiles of `rows` rows that M listed rows of G groups have: a tile has a row at least, and is full or
// its group's last.  (A workgroup without a tile has to find that out: with one for every group's last tile, 8 rows of
// 256 groups of 2048 x 2048, gate and up, took 43.2 us, now 26.0.)
static long long gw_most_tiles(int M, int G, int rows) {
  const long long n = ((long long)M + rows - 1) / rows + G;
  return n < M ? n : M;
}

// Which kernel takes experts' products whose sizes and addresses allow any of them (bf16, loads and vector
// stores without bounds): M listed rows of G groups, N x K weights.  All sides were timed on 2 to 512 groups
// of 256 to 14,336 x 256 to 14,336, rows dealt to the groups at random.
//
// Up to 16 rows a group: the streaming tiles, but not where they fill the chip badly (about as many
// groups have rows as M random picks meet).  Fewer of them than half of the compute units: 4 rows of 16
// groups of 4096 x 4096 (116 tiles) 26.9 us against 26.3 of the kernel for few rows, whose workgroups are
// smaller; 4096 x 8192, 2 of 8 groups (60) 42.5 / 36.4; 2048 x 512, 4 of 32 (61) 7.3 / 6.5, but 4608 x 4096,
// 4 of 16 (131) 36.4 / 45.8.  (These before the streaming tiles' weights passed the caches by; since then 4 rows of 16 groups of 4096 x 4096 34.6 streaming / 25.1,
// 12 of 64 of 1024 x 4096, gate and up (176 tiles), 36.1 / 45.8, 24 of 64 65.8 / 74.5, 8 of 16 of 4096 x 4096 (206) 39.5 / 49.3, in single calls.)  Or, of rows of up to 1,024, the second
// round of two tiles a unit just begun, with less than a row a group (the others are bound by the reads of all weights).  Streaming / few rows, us, at 1.06, 1.12, 1.19 and 1.25
// rounds: 64 groups of 4096 x 1024 33.6 / 30.5, 34.4 / 30.9, 36.3 / 32.6, 36.7 / 35.7; 256 of 2048 x 768 at 1.03 to 1.19 27.2 / 24.1, 27.9 / 25.3, 28.8 / 24.7; 64 of 2048 x 512 20.4 / 19.1,
// 21.8 / 19.6, 22.3 / 20.0; 64 of 1024 x 1024, gate and up, 33.2 / 33.2, 34.1 / 34.0, 36.0 / 34.7; before the round, at 0.97 to 1.0, 25.3 / 28.5, 20.3 / 21.1, 14.8 / 17.5 and 25.3 / 29.7.  Of longer rows the streaming
// tiles are the faster ones there too: 256 of 512 x 1536, gate and up, 46.4 / 51.5 to 48.2 / 53.7; 512 of 512 x 2048 60.5 / 61.6 to 64.0 / 65.0, 128 of 768 x 2048 58.8 / 61.9 to 63.1 / 65.0; 48 rows of 64 of
// 1024 x 4096, 1.06 rounds, 109.6 / 121.3.  (A third round: 48 of 64 of 4096 x 1024, 2.1, 56.7 / 58.4; 90 of 64, 3.0, 70.4 / 77.5.)  With a row or more in a group 1.02 to 0.57 of the other's time at any fraction of a round
// (4608 x 4096, 16 groups, 1.12 rounds: 48 rows 122 / 124, 256 rows 124 / 192).
//
// From 48 rows a group on the wide tiles, one a unit, where they fill the chip: below five eighths of a
// round, and where a second round has just begun, the streaming tiles end earlier (200 rows of each of
// 8 groups of 1024 x 4096, gate and up, 64 wide tiles: 102 us against 61; 16 of 256 x 2048, 32: 47.6 / 18.0;
// with 256 tiles, 16 of 4096 x 4096 at 200 rows: 0.69 of the streaming tiles' time), and
// where those would be more than one and a half rounds over a long K, tiles of 128 in registers (4096 x
// 14336, 8 groups at 200 rows: wide 356, streaming 395, 128: 328; 512 x 2048, 32 groups, gate and up: 62.8,
// 61.8, 56.3; over a short K, 2048 x 256, 16 groups: 20.4, 18.2, 25.6).
// The kernel for few rows and the tiles of 128 take what the others' conditions leave.
// (the tiles that a group of `rows` rows on average has: the rows vary by their root, so that a group of about
// a tile's has one tile or two)
static double gg_tiles_a_group(double rows, int tile) {
  double n = 0;
  for (double k = 0; tile * k < rows + 4 * sqrt(rows); k += 1) n += 0.5 * erfc((tile * k - rows) / sqrt(2 * rows));
  return n;
}
// The lines above were measured with wide tiles of at most so many rows, and are drawn by their number still.  The higher ones
// that gw_height now chooses only end earlier or alike (3,600 rows of 64 groups 196 -> 197 us, 9,000 of 16 327 -> 286): where a line
// would lie with them was not measured.
#define GG_WIDE_ROWS 256
enum { GG_FEW_ROWS = 0, GG_STREAM = 1, GG_WIDE = 2, GG_TILES_128 = 3 };
static int gg_experts_kernel(int M, int N, int K, int G, bool gated) {
  const double rows = (double)M / G;
  const bool stream = K % GW_TK == 0 && K >= 4 * GW_TK && N >= GT_COLS, wide = K % (2 * GW_TK) == 0 && N >= GW_COLS;
  const int n_of = gated ? 2 * N : N;  // W rows that tiles are cut from
  const int stream_cols = (n_of + GT_COLS - 1) / GT_COLS, wide_cols = (n_of + GW_COLS - 1) / GW_COLS;
  if (M / G <= 16) {
    const double tiles = G * (1.0 - pow(1.0 - 1.0 / G, (double)M)) * stream_cols, rounds = tiles / (2 * GG_UNITS);
    const bool begun = M < G && K <= 1024 && rounds > 1.0 && rounds < 1.2;
    return stream && tiles >= GG_UNITS / 2 && !begun ? GG_STREAM : GG_FEW_ROWS;
  }
  if (stream && M / G < GT_ROWS_A_GROUP) return GG_STREAM;
  const double wide_tiles = G * gg_tiles_a_group(rows, GG_WIDE_ROWS) * wide_cols;
  const double stream_tiles = G * gg_tiles_a_group(rows, GT_ROWS) * stream_cols;
  // (groups of many tiles make these lower where one more is needed, and the round begun is a short one)
  const bool begun = rows < 2 * GG_WIDE_ROWS && wide_tiles > 1.02 * GG_UNITS && wide_tiles < 1.1 * GG_UNITS;
  const bool wide_fills = wide_tiles >= 0.625 * GG_UNITS && !begun;
  if (wide && (wide_fills || !stream)) return GG_WIDE;
  return stream && (stream_tiles <= 3 * GG_UNITS || K < 2048 || rows >= 512) ? GG_STREAM : GG_TILES_128;
}

// The choice above, for tests.
extern "C" int hal_grouped_gemm_experts_kernel(int M, int N, int K, int G, int gated) {
  return gg_experts_kernel(M, N, K, G, gated != 0);
}

extern "C" int hal_grouped_gemm(const void* X, int ldx, int x_group_cols, int x_col0, const void* W,
                                const void* W2, long long w_group_stride, int ldw, int dtype,
                                void* Y, int ldy, int y_group_cols, int y_col0, int y_dtype,
                                int y_add, int M, int N, int K, int G, int x_rows, const int* group_offsets,
                                const int* tile_offsets, const int* row_src, int src_div,
                                const int* row_dst, const float* gate, int ldg, int gate_per_group,
                                float limit, float up_shift,
                                float alpha, int act, int allow_mfma, hipStream_t stream) {
  HAL_REQUIRE(act == 0 || (act == 1 && W2 == nullptr), "hal_grouped_gemm: activation %d", act);
  HAL_REQUIRE(M >= 0 && N > 0 && K > 0 && G > 0, "hal_grouped_gemm: bad sizes M=%d N=%d K=%d G=%d", M, N,
              K, G);
  HAL_REQUIRE(dtype == HAL_F32 || dtype == HAL_BF16, "hal_grouped_gemm: operand dtype %d", dtype);
  HAL_REQUIRE(y_dtype == HAL_F32 || y_dtype == HAL_BF16, "hal_grouped_gemm: result dtype %d", y_dtype);
  HAL_REQUIRE(!y_add || y_dtype == HAL_F32, "hal_grouped_gemm: only a float32 result is added into");
  HAL_REQUIRE((group_offsets == nullptr) == (tile_offsets == nullptr),
              "hal_grouped_gemm: group and tile offsets come together");
  HAL_REQUIRE(src_div > 0, "hal_grouped_gemm: src_div %d", src_div);
  HAL_REQUIRE(G <= 65535, "hal_grouped_gemm: %d groups", G);
  if (M == 0) return 0;
  GroupedArgs a;
  a.X = X; a.ldx = ldx; a.x_group_cols = x_group_cols; a.x_col0 = x_col0;
  a.W = W; a.W2 = W2; a.w_group_stride = w_group_stride; a.ldw = ldw;
  a.Y = Y; a.ldy = ldy; a.y_group_cols = y_group_cols; a.y_col0 = y_col0; a.y_dtype = y_dtype;
  a.y_add = y_add;
  a.M = M; a.N = N; a.K = K; a.G = G;
  a.x_rows = x_rows;
  a.group_offsets = group_offsets; a.tile_offsets = tile_offsets;
  a.row_src = row_src; a.src_div = src_div; a.row_dst = row_dst;
  a.gate = gate; a.ldg = ldg; a.limit = limit; a.alpha = alpha; a.act = act; a.up_shift = up_shift;
  a.gate_group_cols = gate_per_group ? 1 : y_group_cols;
  a.gate_cols = gate_per_group ? 0 : 1;
  const int row_tiles = (M + GG_ROWS - 1) / GG_ROWS;
  // (a list of M rows cut into G groups has at most M / tile + G tiles, each group's last one partly filled)
  dim3 grid((N + GG_TN - 1) / GG_TN * (GG_ROWS / GG_TM), group_offsets ? row_tiles + G : row_tiles,
            group_offsets ? 1 : G);
  HAL_REQUIRE(grid.y <= 65535, "hal_grouped_gemm: %u row tiles", grid.y);
  const bool aligned = K % 8 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && x_group_cols % 8 == 0 &&
                       x_col0 % 8 == 0 && w_group_stride % 8 == 0 && ((uintptr_t)X % 16 == 0) &&
                       ((uintptr_t)W % 16 == 0) && (W2 == nullptr || (uintptr_t)W2 % 16 == 0);
  // Experts (rows listed by group) whose sizes and addresses are such that loads and vector stores need no
  // bounds take one of four kernels (gg_experts_kernel), heads of more than 16 rows the streaming tiles (figures
  // there; faster from 17 to 8,000 rows at K of 128 to 512).  The others: of few rows the kernel that keeps many
  // loads in flight instead of staging tiles, of more tiles of 128.
  const long long rows_per_group = group_offsets ? M / G : M;
  const bool whole = dtype == HAL_BF16 && allow_mfma && aligned && !y_add && x_rows > 0 && N % 4 == 0 && ldy % 4 == 0 && y_col0 % 4 == 0 &&
                     y_group_cols % 4 == 0 && (uintptr_t)Y % 16 == 0 && (long long)N * ldw * 2 < (1ll << 31) &&
                     ((long long)x_rows * ldx + K) * 2 < (1ll << 31);
  const bool plain = whole && group_offsets && gate == nullptr && x_group_cols == 0 && y_group_cols == 0;
  const bool heads = whole && !group_offsets && !W2 && row_src == nullptr && row_dst == nullptr && (act == 0 || gate == nullptr);
  const int stream_cols = ((W2 ? 2 * N : N) + GT_COLS - 1) / GT_COLS, wide_cols = ((W2 ? 2 * N : N) + GW_COLS - 1) / GW_COLS;
  const int kernel = plain ? gg_experts_kernel(M, N, K, G, W2 != nullptr) : rows_per_group <= 16 ? GG_FEW_ROWS : GG_TILES_128;
  a.turn = heads || rows_per_group < GT_ROWS_A_GROUP;
  if (kernel == GG_STREAM) {
    const long long units = gw_most_tiles(M, G, GT_ROWS) * stream_cols, blocks = 8 * ((units + 7) / 8);
    HAL_REQUIRE(blocks < (1ll << 31), "hal_grouped_gemm: %lld workgroups", blocks);
    const bool one = M <= GT_ROWS;
    if (W2 && one) hipLaunchKernelGGL((grouped_stream_kernel<true, false, true>), dim3((unsigned)blocks), dim3(256), 0, stream, a, stream_cols);
    else if (W2) hipLaunchKernelGGL((grouped_stream_kernel<true, false, false>), dim3((unsigned)blocks), dim3(256), 0, stream, a, stream_cols);
    else if (one) hipLaunchKernelGGL((grouped_stream_kernel<false, false, true>), dim3((unsigned)blocks), dim3(256), 0, stream, a, stream_cols);
    else hipLaunchKernelGGL((grouped_stream_kernel<false, false, false>), dim3((unsigned)blocks), dim3(256), 0, stream, a, stream_cols);
  } else if (kernel == GG_WIDE) {
    const long long most = gw_most_tiles(M, G, GW_LEAST_ROWS) * wide_cols, units = std::min(most, std::max(gw_most_tiles(M, G, GW_ROWS) * wide_cols, (long long)GG_UNITS));
    const long long blocks = 8 * ((units + 7) / 8);
    HAL_REQUIRE(blocks < (1ll << 31), "hal_grouped_gemm: %lld workgroups", blocks);
    if (W2) hipLaunchKernelGGL(grouped_wide_kernel<true>, dim3((unsigned)blocks), dim3(512), 0, stream, a, wide_cols);
    else hipLaunchKernelGGL(grouped_wide_kernel<false>, dim3((unsigned)blocks), dim3(512), 0, stream, a, wide_cols);
  } else if (heads && K % GW_TK == 0 && rows_per_group > 16 && (K > GW_TK || M <= GT_ONE_STEP_ROWS)) {
    const long long units = (long long)((M + GT_ROWS - 1) / GT_ROWS) * G * stream_cols, blocks = 8 * ((units + 7) / 8);
    HAL_REQUIRE(blocks < (1ll << 31) && (long long)M * stream_cols < (1ll << 31), "hal_grouped_gemm: %lld workgroups", blocks);
    hipLaunchKernelGGL((grouped_stream_kernel<false, true, false>), dim3((unsigned)blocks), dim3(256), 0, stream, a, stream_cols);
  } else if (dtype == HAL_BF16 && allow_mfma && aligned && kernel == GG_FEW_ROWS) {
    grid.x = W2 ? (N + 31) / 32 : (N + 63) / 64;
    if (W2) hipLaunchKernelGGL(grouped_skinny_kernel<true>, grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL(grouped_skinny_kernel<false>, grid, dim3(256), 0, stream, a);
  } else if (dtype == HAL_BF16 && allow_mfma && aligned) {
    grid.x = W2 ? (N + GG_ROWS / 2 - 1) / (GG_ROWS / 2) : (N + GG_ROWS - 1) / GG_ROWS;
    if (W2) hipLaunchKernelGGL(grouped_mfma_kernel<true>, grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL(grouped_mfma_kernel<false>, grid, dim3(256), 0, stream, a);
  } else if (dtype == HAL_BF16) {
    if (W2) hipLaunchKernelGGL((grouped_fma_kernel<bf16_t, true>), grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((grouped_fma_kernel<bf16_t, false>), grid, dim3(256), 0, stream, a);
  } else {
    if (W2) hipLaunchKernelGGL((grouped_fma_kernel<float, true>), grid, dim3(256), 0, stream, a);
    else hipLaunchKernelGGL((grouped_fma_kernel<float, false>), grid, dim3(256), 0, stream, a);
  }
  HAL_LAUNCH_CHECK();
  return 0;
}
