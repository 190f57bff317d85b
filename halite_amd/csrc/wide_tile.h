// The products of one tile of up to 352 rows x 256 W rows by eight waves, for the kernels of prompts: a wave takes half of the
// tile's rows (NI blocks of 16) and 64 W rows, K goes 64 at a time through two buffers in LDS that the loads fill by themselves.
#pragma once

#include "hal_lds.h"

#include <type_traits>

typedef __attribute__((ext_vector_type(8))) __bf16 wt_bf16x8;
typedef __attribute__((ext_vector_type(4))) float wt_f32x4;

#define WT_TK 64    // k of a step: whole 128-byte lines
#define WT_COLS 256  // W rows of a tile
#define WT_MOST 11   // most blocks of 16 rows of a wave

// A wave's rows in two parts; the loads of a part that every wave makes a step (eight rows of either half of the tile each; an odd
// part's last ones have rows for four waves, the others' bring their rows before those again).
template <int NI>
struct wt_part {
  static constexpr int blocks(int p) { return p ? NI / 2 : (NI + 1) / 2; }
  static constexpr int first(int p) { return p ? (NI + 1) / 2 : 0; }
  static constexpr int loads(int p) { return (blocks(p) + 1) / 2; }
};
#define WT_PART_BYTES(p) (wt_part<WT_MOST>::blocks(p) * 2 * 16 * WT_TK * 2)  // of X: both halves of the tile
#define WT_HALF_BYTES (WT_COLS / 2 * WT_TK * 2)                // of W: 32 rows of each of four waves' 64

// The two buffers: parts of X and halves of W, each an array of its own (see hal_load_lds).
struct wt_lds {
  char *x[2][2], *w[2][2];
};
#define WT_LDS(name)                                                                                                              \
  __shared__ __attribute__((aligned(16))) char name##_x00[WT_PART_BYTES(0)], name##_x01[WT_PART_BYTES(1)], name##_w00[WT_HALF_BYTES], \
      name##_w01[WT_HALF_BYTES], name##_x10[WT_PART_BYTES(0)], name##_x11[WT_PART_BYTES(1)], name##_w10[WT_HALF_BYTES],                \
      name##_w11[WT_HALF_BYTES];                                                                                                    \
  const wt_lds name = {{{name##_x00, name##_x01}, {name##_x10, name##_x11}}, {{name##_w00, name##_w01}, {name##_w10, name##_w11}}}

// Which eight rows load u of a wave brings of part p: the octet's place in the part, and its row in the tile.
template <int NI>
__device__ __forceinline__ int wt_octet(int wave, int p, int u) {
  const int o = wave + 8 * u;
  return o < 4 * wt_part<NI>::blocks(p) ? o : o >= 8 ? o - 8 : o - 4;
}
template <int NI>
__device__ __forceinline__ int wt_octet_row(int octet, int p) {
  const int n = wt_part<NI>::blocks(p), block = octet / 2;
  return (block / n * NI + wt_part<NI>::first(p) + block % n) * 16 + octet % 2 * 8;
}

template <int LEFT>
__device__ __forceinline__ void wt_meet_left() {  // the newest LEFT loads may be on their way, this phase's operands from LDS too
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(LEFT) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}
// The end of a phase: all that it read of LDS is there.  (Its products have waited for most of it, but not for what the next phase multiplies,
// and that place is asked for anew by the other group of waves before this one's next products.)
__device__ __forceinline__ void wt_meet() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Where a lane's piece of an operand lies in a block of 16 rows x 64 k (k: which 32 of them).
__device__ __forceinline__ int wt_get(int lane, int k) { return lane % 16 * 128 + ((lane / 16 + 4 * k) ^ hal_turn(lane % 16)) * 16; }

// acc = X * W^T over `steps` (an even number) steps of 64 k.  bring_x(part, to, step) makes wt_part::loads loads of a part of X into `to`,
// bring_w(half, to, step) two loads of a half of W: of eight rows each, octet wave + 8 u of the half, which is of 32 neighbouring W rows of each
// wave's 64.  wt_begin asks for the first two steps; wt_steps asks for two steps past the end too, in the order and into the places in which wt_begin
// would ask for the first two of a tile that follows: they may be those, and that tile then begins with wt_steps.
//
// What bounds it: the matrix cores at the clock that the chip holds under them, given that they always have work and that the
// workgroups of a compute die read the same lines at the same time (then a step's 64 KB come in 0.7 us, products take 1.0 to 1.4;
// workgroups at different places of K need 1.5 to 2.0 us a step).  A SIMD has two waves, one of waves 0-3 and one of 4-7, and these take turns: while one
// multiplies, the other reads its next operands and asks for new pieces; a barrier ends each turn, and waves 4-7 are one turn behind.
// A step is four such phases of a wave, a part of its rows times half of its columns each, in an order in which one operand
// stays: (x0, A) (x0, B) (x1, B) (x1, A), A being the half of W that the step before ended without, so that a half's registers are free when its
// next piece is read.  What phase p read of LDS is asked for anew in phase p + 2 (both groups of waves have ended phase p by then, with which its
// reads have come, see wt_meet), for the step after next, six phases before it is read: loads have the time of five to arrive.
// WT_SLIM blocks and more leave no registers for a part of X: there a phase is a part of the rows times all columns over 32 of the 64 k.
#define WT_SLIM 10  // from so many blocks on
template <int NI, typename BringX, typename BringW>
__device__ __forceinline__ void wt_begin(const wt_lds& lds, BringX&& bring_x, BringW&& bring_w) {
  constexpr std::integral_constant<int, 0> first{};
  constexpr std::integral_constant<int, 1> second{};
  if constexpr (NI < WT_SLIM) {
    bring_w(0, lds.w[0][0], 0), bring_x(first, lds.x[0][0], 0), bring_w(1, lds.w[0][1], 0);
    bring_x(second, lds.x[0][1], 0), bring_w(1, lds.w[1][1], 1), bring_x(first, lds.x[1][0], 1), bring_w(0, lds.w[1][0], 1);
  } else {
    bring_w(0, lds.w[0][0], 0), bring_w(1, lds.w[0][1], 0), bring_x(first, lds.x[0][0], 0), bring_x(second, lds.x[0][1], 0);
    bring_w(0, lds.w[1][0], 1), bring_w(1, lds.w[1][1], 1);
  }
}

template <int NI, typename BringX, typename BringW>
__device__ __forceinline__ void wt_steps(const wt_lds& lds, int wave, int lane, int steps, wt_f32x4 (&acc)[NI][4], BringX&& bring_x, BringW&& bring_w) {
  using P = wt_part<NI>;
  constexpr int H0 = P::blocks(0), H1 = P::blocks(1), L0 = P::loads(0), L1 = P::loads(1);
  constexpr std::integral_constant<int, 0> first{};
  constexpr std::integral_constant<int, 1> second{};
  const int wm = wave / 4, wn = wave % 4, get0 = wt_get(lane, 0);
  auto of_x = [&](const char* from, int n, int i, int at) { return *(const wt_bf16x8*)(from + (wm * n + i) * 2048 + at); };
  auto of_w = [&](const char* from, int j, int at) { return *(const wt_bf16x8*)(from + (wn * 2 + j) * 2048 + at); };
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = wt_f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (NI < WT_SLIM) {
    const int get[2] = {get0, wt_get(lane, 1)};
    wt_bf16x8 x[H0][2], w[2][2][2];
    auto read_x = [&](const char* from, int n) {
#pragma unroll
      for (int i = 0; i < H0; ++i)
#pragma unroll
        for (int k = 0; k < 2; ++k)
          if (i < n) x[i][k] = of_x(from, n, i, get[k]);
    };
    auto read_w = [&](const char* from, int half) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int k = 0; k < 2; ++k) w[half][j][k] = of_w(from, j, get[k]);
    };
    auto products = [&](int part, int half) {
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int i = 0; i < H0; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            if (i < P::blocks(part)) {
              wt_f32x4& to = acc[P::first(part) + i][half * 2 + j];
              to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[half][j][k], x[i][k], to, 0, 0, 0);
            }
      wt_meet();
    };
    wt_meet_left<L0 + L1 + 6>();
    read_w(lds.w[0][0], 0);
    if (wave >= 4) wt_meet();
    auto step = [&](int s, int b) {
      read_x(lds.x[b][0], H0);
      bring_x(second, lds.x[!b][1], s + 1);
      wt_meet_left<L0 + 2 * L1 + 4>();
      products(0, b);
      read_w(lds.w[b][!b], !b);
      bring_w(b, lds.w[b][b], s + 2);
      wt_meet_left<L0 + L1 + 6>();
      products(0, !b);
      read_x(lds.x[b][1], H1);
      bring_x(first, lds.x[b][0], s + 2);
      wt_meet_left<2 * L0 + L1 + 4>();
      products(1, !b);
      read_w(lds.w[!b][!b], !b);
      bring_w(!b, lds.w[b][!b], s + 2);
      wt_meet_left<L0 + L1 + 6>();
      products(1, b);
    };
    for (int s = 0; s < steps; s += 2) {
      step(s, 0);
      step(s + 1, 1);
    }
  } else {
    wt_bf16x8 x[H0], w[2][4];
    // (where operands lie is worked out anew for every phase: kept, the places would take registers that are not there)
    auto place = [&](int k) {
      int at = get0 ^ 64 * k;
      asm volatile("" : "+v"(at));
      return at;
    };
    auto read_x = [&](const char* from, int n, int k) {
      const int at = place(k);
#pragma unroll
      for (int i = 0; i < H0; ++i)
        if (i < n) x[i] = of_x(from, n, i, at);
    };
    auto read_w = [&](char* const (&from)[2], int k) {
      const int at = place(k);
#pragma unroll
      for (int j = 0; j < 4; ++j) w[k][j] = of_w(from[j / 2], j % 2, at);
    };
    auto products = [&](int part, int k) {
#pragma unroll
      for (int i = 0; i < H0; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (i < P::blocks(part)) {
            wt_f32x4& to = acc[P::first(part) + i][j];
            to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[k][j], x[i], to, 0, 0, 0);
          }
      wt_meet();
    };
    // Parts of X are read in the first and third phase and in the second and fourth, W for 32 of the k in the second and for the next step's
    // other 32 in the fourth: all are asked for anew two phases after their last read, four before the next.
    wt_meet_left<L1 + 4>();
    read_w(lds.w[0], 0);
    if (wave >= 4) wt_meet();
    auto step = [&](int s, int b) {
      read_x(lds.x[b][0], H0, 0);
      bring_x(first, lds.x[!b][0], s + 1);
      wt_meet_left<L0 + 4>();
      products(0, 0);
      read_x(lds.x[b][1], H1, 0);
      read_w(lds.w[b], 1);
      bring_x(second, lds.x[!b][1], s + 1);
      wt_meet_left<L0 + L1 + 4>();
      products(1, 0);
      read_x(lds.x[b][0], H0, 1);
      wt_meet_left<L0 + L1>();
      products(0, 1);
      read_x(lds.x[b][1], H1, 1);
      read_w(lds.w[!b], 0);
      bring_w(0, lds.w[b][0], s + 2), bring_w(1, lds.w[b][1], s + 2);
      wt_meet_left<L1 + 4>();
      products(1, 1);
    };
    for (int s = 0; s < steps; s += 2) {
      step(s, 0);
      step(s + 1, 1);
    }
  }
  if (wave < 4) wt_meet();
}

// LDS is neither given back nor used anew while loads are on their way into it.
__device__ __forceinline__ void wt_end() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
