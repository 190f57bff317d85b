// C[M, N] = X[M, K] W[N, K]^T for up to 64 rows of bf16 X (decode steps of many requests; from how many on, the callers' rules say): what counts is that W
// comes at the memory's rate.  Both operands go in whole 128-byte lines straight into LDS, two to five steps of 64 k on
// their way while one is multiplied (v_mfma_f32_16x16x32_bf16, float32 sums).  A workgroup of four waves takes all rows
// and 64 or 128 rows of W (of a gated product half of them the gate's and half the up projection's, act(gate) * up in the
// epilogue).  W rows are the instruction's first operand, so lane l of a result holds row l % 16 and the four neighbouring
// columns 4 * (l / 16) .. + 3: one vector store.
//
// A matrix of few rows fills the chip by its K: cut into parts, a workgroup each, whose float32 sums go to planes of their
// own that the kernel which reads the result adds up in order (the norm, the rotation: they are launched
// anyway; a workgroup of the product that waited for the others' sums would cost a trip through memory for few
// workgroups, and one more kernel its launch).
//
// What bounds it: the 20 bytes a clock that a compute unit gets from the second-level cache, of which X takes a third
// (tiles of 128) or a half (of 64), and a start of about 3 us.  64 rows, events around graphs of calls on changing weights, beside the
// library's product: 6144 x 4096 18.1 -> 13.8 us, 4096 x 4096 15.4 -> 10.6, 4096 x 14336 41.3 -> 26.6,
// gate and up of 14336 x 4096 with SiLU 55.1 + 5.1 (a kernel of its own) -> 49.5, 128256 x 4096 225 -> 204.
#include "hal_lds.h"
#include "hal_api.h"

typedef __attribute__((ext_vector_type(8))) __bf16 gs_bf16x8;
typedef __attribute__((ext_vector_type(4))) float gs_f32x4;

#define GS_K 64  // of a step
#define GS_MAX_ROWS 64
#define GS_UNITS 256  // compute units of the gfx950 parts that this library is built for

struct StreamArgs {
  const bf16_t* X;
  int ldx;
  const bf16_t *W, *W2;
  int ldw;
  void* Y;
  bool f32;
  int M, N, K, tiles, parts;
  hal_gate act;
};

// Tiles of 64 go through six buffers, one workgroup a compute unit; of 128 through three, two workgroups, or six (`gs_deep`).
template <int NI, int COLS, bool GATED, int BUFFERS>
__global__ void __launch_bounds__(256)
gemm_stream_kernel(StreamArgs a) {
  constexpr int NJ = COLS / 64, AI = NI / 2, WI = COLS / 32, LOADS = AI + WI;
  constexpr int A_BYTES = NI * 16 * GS_K * 2, BYTES = A_BYTES + COLS * GS_K * 2, WIDE = GATED ? COLS / 2 : COLS;
  __shared__ __attribute__((aligned(16))) char b0[BYTES], b1[BYTES], b2[BYTES], b3[BUFFERS > 3 ? BYTES : 16], b4[BUFFERS > 3 ? BYTES : 16],
      b5[BUFFERS > 3 ? BYTES : 16];
  const int tile = blockIdx.x % a.tiles, part = blockIdx.x / a.tiles, n0 = tile * WIDE;
  const int all = a.K / GS_K, first = (int)((long long)all * part / a.parts);
  const int steps = (int)((long long)all * (part + 1) / a.parts) - first;
  // Workgroups of one part begin at different places of K and go round: rows of W that lie a power of two
  // apart, all read at one place of K at a time, meet in a few of the memory's channels.
  const int begin = a.parts > 1 ? 0 : (tile * 7) % steps;
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int lr = wave * 8 + lane / 8, c = ((lane % 8) ^ hal_turn(lr % 16)) * 16;
  // (GATED: of every 32 W rows in LDS the first 16 are the gate's and the others the up projection's; where a wave has 16
  // only, 8 and 8: either way a wave's loads are of one of the two)
  const bool up = GATED && (COLS == 128 ? wave >= 2 : wave % 2 == 1);
  const uint32_t w_bytes = (uint32_t)a.N * a.ldw * 2, x_bytes = ((uint32_t)(a.M - 1) * a.ldx + a.K) * 2;
  const hal_memory W = hal_memory_at(up ? a.W2 : a.W, w_bytes), X = hal_memory_at(a.X, x_bytes);
  uint32_t xo[AI], wo[WI];
  // rows and columns past the end are read from the last one: nothing of them is stored
#pragma unroll
  for (int i = 0; i < AI; ++i) {
    const int r = lr + 32 * i;
    xo[i] = (uint32_t)(r < a.M ? r : a.M - 1) * (uint32_t)(a.ldx * 2) + c;
  }
#pragma unroll
  for (int i = 0; i < WI; ++i) {
    int n = i * 32 + lr;
    if (GATED) n = COLS == 128 ? i * 16 + lr % 16 : n / 16 * 8 + n % 8;
    n = n0 + n < a.N ? n0 + n : a.N - 1;
    wo[i] = (uint32_t)n * (uint32_t)(a.ldw * 2) + c;
  }
  // (no branch, so that the compiler knows which loads may be on their way: steps past the end, which fill the last turn
  // through the buffers, are read from past the operands' bytes, and are zeros)
  auto bring = [&](char* lds, int step) {
    const bool past = step >= steps;
    step += begin;
    const uint32_t at = (uint32_t)(first + (step < steps ? step : step - steps)) * (GS_K * 2);
#pragma unroll
    for (int i = 0; i < AI; ++i) hal_load_lds(X, past ? x_bytes : xo[i] + at, 0, lds + (i * 4 + wave) * 1024);
#pragma unroll
    for (int i = 0; i < WI; ++i) hal_load_lds<HAL_ONCE>(W, past ? w_bytes : wo[i] + at, 0, lds + A_BYTES + (i * 4 + wave) * 1024);
  };
  const int q = lane / 16, r16 = lane % 16;
  const int get[2] = {r16 * 128 + (q ^ hal_turn(r16)) * 16, r16 * 128 + ((q + 4) ^ hal_turn(r16)) * 16};
  gs_f32x4 acc[NI][NJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = gs_f32x4{0.f, 0.f, 0.f, 0.f};
  auto advance = [&](int s, const char* mine, char* free) {
    hal_meet<(BUFFERS - 2) * LOADS>();  // (this step's pieces are there, the next ones' may be on their way)
    bring(free, s + BUFFERS - 1);
    gs_bf16x8 w[2][NJ], x[2][NI];
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) w[half][j] = *(const gs_bf16x8*)(mine + A_BYTES + (wave * NJ + j) * 2048 + get[half]);
#pragma unroll
      for (int i = 0; i < NI; ++i) x[half][i] = *(const gs_bf16x8*)(mine + i * 2048 + get[half]);
    }
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int i = 0; i < NI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[half][j], x[half][i], acc[i][j], 0, 0, 0);
  };
  bring(b0, 0);
  bring(b1, 1);
  if constexpr (BUFFERS == 3) {
    for (int s = 0; s < steps; s += 3) {
      advance(s, b0, b2);
      advance(s + 1, b1, b0);
      advance(s + 2, b2, b1);
    }
  } else {
    bring(b2, 2);
    bring(b3, 3);
    bring(b4, 4);
    for (int s = 0; s < steps; s += 6) {
      advance(s, b0, b5);
      advance(s + 1, b1, b0);
      advance(s + 2, b2, b1);
      advance(s + 3, b3, b2);
      advance(s + 4, b4, b3);
      advance(s + 5, b5, b4);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // LDS is not given back while loads are on their way into it
  auto store = [&](int r, int n, gs_f32x4 v, gs_f32x4 u) {
    if (r >= a.M || n >= a.N) return;
    if (GATED) {
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = hal_gated(a.act, v[k], u[k]);
    }
    const size_t at = ((size_t)part * a.M + r) * a.N + n;
    if (a.f32) *(gs_f32x4*)((float*)a.Y + at) = v;
    else *(uint2*)((bf16_t*)a.Y + at) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
  };
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int r = i * 16 + r16;
    if constexpr (GATED && COLS == 64) {  // a wave's 16 rows of W: lanes q of 0 and 1 have the gate's, q + 2 the same columns' up
      gs_f32x4 u;
#pragma unroll
      for (int k = 0; k < 4; ++k) u[k] = __shfl_xor(acc[i][0][k], 32, HAL_WAVE);
      if (q < 2) store(r, n0 + wave * 8 + q * 4, acc[i][0], u);
    } else if constexpr (GATED) {
      store(r, n0 + wave * 16 + q * 4, acc[i][0], acc[i][1]);
    } else {
#pragma unroll
      for (int j = 0; j < NJ; ++j) store(r, n0 + (wave * NJ + j) * 16 + q * 4, acc[i][j], acc[i][j]);
    }
  }
}

// How a product of 17 to 64 rows is cut: columns of a tile and parts of K, or no parts where the library's is to be
// taken.  One workgroup a compute unit and as near to all of them as it goes is the fastest of all
// cuts (4096 x 14336, tiles of 128 in 4 to 16 parts: 38.9, 34.5, 30.1, 30.9, 25.9 at 8 = 256 workgroups, 34.3, 31.0, 29.2, 28.2 us);
// where tiles of 64 and of 128 fill the chip alike those of 64, with half as many planes to be added up afterwards.
// More tiles than units: tiles of 128, two a unit, no parts.  A gated product has no parts (its epilogue needs the sums).
struct StreamCut {
  int cols, parts;
};
static StreamCut gs_cut(int N, int K, bool gated, bool may_part) {
  const int n = gated ? 2 * N : N, steps = K / GS_K;
  StreamCut best = {0, 0};
  int most = 0;
  for (int cols = 64; cols <= 128; cols += 64) {
    const int tiles = (n + cols - 1) / cols;
    if (tiles > GS_UNITS) continue;
    int parts = may_part && !gated ? GS_UNITS / tiles : 1;
    parts = parts > steps / 4 ? steps / 4 : parts;
    if (parts >= 1 && tiles * parts > most) most = tiles * parts, best = {cols, parts};
  }
  if ((n + 127) / 128 > GS_UNITS) return {128, 1};
  return most >= GS_UNITS * 5 / 8 ? best : StreamCut{0, 0};
}

// Whether tiles of 128 go through six buffers: a compute unit has one of them then, so where there are no more tiles than units, and
// where the longer start is made up for by the steps behind it.  Three / six buffers, us, at 48 rows: 161 tiles of K 4,096 39.7 / 37.0, 250 52.2 / 50.8,
// gated 172 42.9 / 40.5, but gated 224 (which have the memory's rate) 49.2 / 49.5; 250 of 2,048 31.0 / 31.4; in parts 48 tiles x 5 of 4,096
// 13.8 / 15.1, 97 x 2 25.5 / 27.2; at 17 rows 161 36.9 / 35.5, 172 42.5 / 39.8, 250 50.8 / 49.2.  The lines are the cautious ones: of K 3,072
// 161 tiles 34.6 / 29.4 at 48 rows and 31.9 / 31.7 at 64, 204 35.3 / 32.5 and 34.1 / 33.9, 250 38.0 / 37.0 and 37.5 / 37.8, gated 172 32.8 / 32.3 and
// 35.5 / 35.6, 192 35.7 / 33.9 and 36.9 / 37.0, 224 36.0 / 36.0; 250 of 3,584 42.9 / 43.2 and 42.5 / 43.5; of 2,560 gated 172 32.0 / 32.0; of 5,120
// gated 172 57.0 / 57.4 and 59.2 / 59.7 (17 rows 55.7 / 53.8), 224 60.3 / 61.0; gated 192 of 4,096 43.9 / 42.7, 204 45.0 / 44.5.
static bool gs_deep(int K, bool gated, int tiles, int parts) {
  return parts == 1 && K >= 4096 && tiles <= (gated ? GS_UNITS * 3 / 4 : GS_UNITS);
}

// The cut above: parts of K, 0 for none (may_part: the reader adds up planes).
extern "C" int hal_gemm_bf16_stream_parts(int N, int K, int gated, int may_part) {
  if (K % GS_K || K < 4 * GS_K || N % 4 || N < 128) return 0;
  return gs_cut(N, K, gated != 0, may_part != 0).parts;
}

// X [M, K], W (and W2 of a gated product: W is the gate's) [N, K] bf16, up to 64 rows.  parts: what
// hal_gemm_bf16_stream_parts returned; 1: Y [M, N] of bf16 or float32, more: float32 planes [parts][M][N] whose sum is the result.
extern "C" int hal_gemm_bf16_stream(const void* X, int ldx, const void* W, const void* W2, int ldw, void* Y, int y_dtype,
                                    int parts, int act, float limit, float alpha, float up_shift, int M, int N, int K,
                                    hipStream_t stream) {
  HAL_REQUIRE(M > 0 && M <= GS_MAX_ROWS, "hal_gemm_bf16_stream: %d rows", M);
  const int cut = hal_gemm_bf16_stream_parts(N, K, W2 != nullptr, parts > 1);
  HAL_REQUIRE(parts >= 1 && parts == cut, "hal_gemm_bf16_stream: N=%d K=%d in %d parts", N, K, parts);
  HAL_REQUIRE(ldx >= K && ldw >= K && ldx % 8 == 0 && ldw % 8 == 0 && (uintptr_t)X % 16 == 0 && (uintptr_t)W % 16 == 0 &&
                  (uintptr_t)W2 % 16 == 0 && (uintptr_t)Y % 16 == 0,
              "hal_gemm_bf16_stream: rows of %d and %d, or their places", ldx, ldw);
  HAL_REQUIRE((long long)N * ldw * 2 < (1ll << 31) && (long long)M * ldx * 2 < (1ll << 31), "hal_gemm_bf16_stream: more bytes than offsets reach");
  HAL_REQUIRE((y_dtype == HAL_F32 || y_dtype == HAL_BF16) && (parts == 1 || y_dtype == HAL_F32), "hal_gemm_bf16_stream: result dtype %d", y_dtype);
  HAL_REQUIRE(act >= HAL_ACT_SILU && act <= HAL_ACT_CLAMPED, "hal_gemm_bf16_stream: activation %d", act);
  const int cols = gs_cut(N, K, W2 != nullptr, parts > 1).cols, tiles = ((W2 ? 2 * N : N) + cols - 1) / cols;
  const StreamArgs a = {(const bf16_t*)X, ldx, (const bf16_t*)W, (const bf16_t*)W2, ldw, Y, y_dtype == HAL_F32, M, N, K, tiles, parts,
                        {act, limit, alpha, up_shift}};
  const bool deep = cols == 64 || gs_deep(K, W2 != nullptr, tiles, parts);
#define GS_LAUNCH(NI_, COLS_, GATED_)                                                                                                  \
  do {                                                                                                                                 \
    if (deep) hipLaunchKernelGGL((gemm_stream_kernel<NI_, COLS_, GATED_, 6>), dim3(tiles * parts), dim3(256), 0, stream, a);            \
    else hipLaunchKernelGGL((gemm_stream_kernel<NI_, COLS_, GATED_, COLS_ == 64 ? 6 : 3>), dim3(tiles * parts), dim3(256), 0, stream, a); \
  } while (0)
#define GS_ROWS(COLS_, GATED_)             \
  if (M <= 32) GS_LAUNCH(2, COLS_, GATED_); \
  else GS_LAUNCH(4, COLS_, GATED_)
  if (W2) {
    if (cols == 64) { GS_ROWS(64, true); }
    else { GS_ROWS(128, true); }
  } else {
    if (cols == 64) { GS_ROWS(64, false); }
    else { GS_ROWS(128, false); }
  }
#undef GS_ROWS
#undef GS_LAUNCH
  HAL_LAUNCH_CHECK();
  return 0;
}
