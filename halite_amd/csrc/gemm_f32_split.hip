// C[M, N] = A[M, K] * W[N, K]^T of float32 for prompts, on the matrix cores' bf16 instruction, as exact as float32 sums are
// (a published method: Henry, Tang, Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", 2019): a float32 number is the sum of three bf16 numbers (x = hi + mid + lo: hi = bf16(x), mid = bf16(x - hi),
// lo = x - hi - mid, exactly, as 8 + 8 + 8 significant bits and two signs hold 24), a product of two bf16 numbers is exact in
// float32, and six of the nine products of two such sums are added up in float32.  The other three are left out: mid * lo and
// lo * mid are at most 2^-25 of the product each, together (with lo * lo) under 2^-24, which is what its own rounding to
// float32 takes.  bf16 ends at 2^-133, float32 at 2^-149, so every number is multiplied by 2^16 (SP_SCALE) first, and a sum by
// 2^-32 at the end: then no bit of any number is lost.  (Without: 2^-116 times N(0, 1) 2.2e-6, 2^-124 5.6e-4.)  Numbers from
// 2^112 and sums from 2^96 on become infinities by that, and are taken again as below.
//
// The instruction cuts its sums off where a float32 addition rounds, and a float32 addition to a long sum loses more than one
// to a short one, so how often a sum of full size goes through either decides the error.  Two stages of 32 k at a time start from
// nothing, each with its five small products first, and are added to the total by a float32 addition; a total takes 128 stages
// at most (SP_WALK), the next one is added to it where it lies in memory.  Distance to 64 bits over the result's norm, for
// K = 4,096 in four parts / two / one, 14,336 in four, 8,192 in one: N(0, 1) times N(0, 0.02) 1.4e-7 / 1.5e-7 / 1.8e-7, 2.0e-7, 1.9e-7;
// the same without signs, where every sum is of full size, 0.5e-7 / 0.7e-7 / 1.2e-7, 0.7e-7, 0.9e-7.  The float32 instruction's tiles
// (gemm_f32.hip) 4.1e-7, 4.2e-7, 4.1e-7 and 1.25e-7, 1.04e-7, 1.02e-7; its kernel for up to 128 rows 5.7e-7 (K = 4,096), 1.1e-6 (14,336) and
// 2.4e-7, 4.6e-7.  (A total from each stage: 2.2e-7 and 1.65e-7 in one part of 4,096, and without walks 2.3e-7 for 8,192 without signs;
// one sum of all six products over 64 stages: 7e-7, over all of 14,336: 1.9e-6.)
//
// What bounds it: the instruction at the clock that the chip holds under it (1,340 TFLOP/s of bf16 products, the
// library's largest bf16 products reach 1,555), given that nothing else stands in the way.  So
//  - a workgroup takes 256 x 128 results, a wave of eight 64 x 64: numbers come from the second-level cache at 16 to 20 bytes a clock and
//    unit whoever asks, and 128 x 128 asks for a third more of them a product (500 rows x 28,672 x 4,096: 609 and 698 us; the
//    tiles of 128 and of 64 rows are for steps that leave units without a tile of 256);
//  - every number is taken apart once a workgroup, on its way from memory through registers into LDS, where six planes (hi, mid, lo of
//    A and W) lie in the operands' order;
//  - the order of work within a stage is spelled out in groups of four products with the loads, conversions and LDS accesses that go
//    beside them: left to the compiler, conversions stood in front of a stage's products (686 us), or registers spilled;
//  - one barrier a stage, before its last product: by then the next stage lies in LDS, and its first operands are read beside
//    that product.
// Measured beside the float32 instruction's tiles, 500 rows, us: x 28,672 x 4,096 990 -> 602; 32,000 x 4,096 1,095 -> 629; 4,096 x 14,336
// 500 -> 294; 6,144 x 4,096 207 -> 154; 4,096 x 4,096 142 -> 98; 2,048 rows x 28,672 x 4,096 3,600 -> 2,226 (216 TFLOP/s).  (The scale costs
// two multiplications beside seven instructions a pair of numbers, 15 to 30 us of 600; the additions that every second stage spares
// give that back.)
//
// A matrix of few columns fills the chip by its K, cut into parts whose sums go to planes that one more kernel adds up in order.  How many
// depends on the matrix alone, so that a row's result is its own, whatever rows are beside it.
#include "hal_lds.h"
#include "hal_api.h"
#include <algorithm>

#define SP_SCALE 65536.f  // 2^-149, float32's smallest number, is bf16's smallest, 2^-133, then
#define SP_BN 128  // columns of a tile
#define SP_BN_LOW 96  // of 256 rows, where fewer end earlier
#define SP_BK 32  // k of a stage: a row's 128-byte line
#define SP_THREADS 512
#define SP_XCDS 8     // dies of the gfx950 parts that this library is built for (a wrong count costs cache hits only)
#define SP_UNITS 256  // compute units of the same
#define SP_MOST_PARTS 8
#define SP_WALK 128   // most stages whose sums go into one total
#define SP_PLANES (64ll << 20)  // bytes of planes up to which all rows go at once
#define SP_ROW_LIMIT (1 << 22)  // numbers of a row: 256 of them lie within 32-bit offsets

typedef __attribute__((ext_vector_type(8))) __bf16 sp_bf16x8;
typedef __attribute__((ext_vector_type(4))) float sp_f32x4;

// Where the eight k from 8 q on of row r of a block of 16 rows lie in the block's KiB: a wave's operand is the whole KiB, each
// of its turns through LDS (see hal_turn) a quarter of it; and the 8-byte stores of four rows meet all banks.
__device__ __forceinline__ int sp_slot(int q, int r) { return (q * 16 + (r ^ (12 * q & 15))) * 16; }

// two neighbouring numbers, times the scale, as three words of two bf16 (minus: (-1, 0) and (0, -1) of bf16)
typedef __attribute__((ext_vector_type(2))) __bf16 sp_bf16x2;
__device__ __forceinline__ void sp_split(float a, float b, const uint32_t (&minus)[2], uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  const sp_bf16x2 first = __builtin_bit_cast(sp_bf16x2, minus[0]), second = __builtin_bit_cast(sp_bf16x2, minus[1]);
  a *= SP_SCALE, b *= SP_SCALE;
  hi = pack_bf16x2(a, b);
  const sp_bf16x2 h = __builtin_bit_cast(sp_bf16x2, hi);
  a = __builtin_amdgcn_fdot2_f32_bf16(h, first, a, false), b = __builtin_amdgcn_fdot2_f32_bf16(h, second, b, false);
  mid = pack_bf16x2(a, b);
  const sp_bf16x2 m = __builtin_bit_cast(sp_bf16x2, mid);
  a = __builtin_amdgcn_fdot2_f32_bf16(m, first, a, false), b = __builtin_amdgcn_fdot2_f32_bf16(m, second, b, false);
  lo = pack_bf16x2(a, b);
}

struct SplitArgs {
  const float *A, *W;
  float* C;
  int lda, ldw, ldc, M, N, K, tiles_m, tiles_n, parts;
  long long plane;  // numbers from one part's results to the next one's
};

// WALKS: for parts of more than SP_WALK stages.
template <int BM, int BN, bool WALKS>
__global__ void __launch_bounds__(SP_THREADS, BM == 64 ? 4 : 2)
gemm_f32_split_kernel(SplitArgs g) {
  constexpr int WM = BM / 64, WN = 8 / WM, NI = 4, NJ = BN / 16 / WN;  // WM x WN waves of NI x NJ results of 16 x 16
  constexpr int AL = BM / 64, LOADS = AL + 2;                             // a wave's loads a stage, eight rows each
  constexpr int A_PLANE = BM * 64, W_PLANE = SP_BN * 64, W_AT = 3 * A_PLANE, BYTES = 3 * (A_PLANE + W_PLANE);
  __shared__ __attribute__((aligned(16))) char lds[2 * BYTES];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int n_tiles = g.tiles_m * g.tiles_n * g.parts, die = blockIdx.x % SP_XCDS, rest = n_tiles % SP_XCDS;
  const int id = die * (n_tiles / SP_XCDS) + min(die, rest) + blockIdx.x / SP_XCDS;
  const int m0 = (id % g.tiles_m) * BM, n0 = (id / g.tiles_m % g.tiles_n) * BN, part = id / g.tiles_m / g.tiles_n;
  const int rows_here = min(BM, g.M - m0), cols_here = min(BN, g.N - n0);
  const int all = (g.K + SP_BK - 1) / SP_BK, part_first = (int)((long long)all * part / g.parts);
  const int part_stages = (int)((long long)all * (part + 1) / g.parts) - part_first, walks = WALKS ? (part_stages + SP_WALK - 1) / SP_WALK : 1;
  const uint32_t a_bytes = ((uint32_t)(rows_here - 1) * g.lda + g.K) * 4, w_bytes = ((uint32_t)(cols_here - 1) * g.ldw + g.K) * 4;
  const hal_memory a_all = hal_memory_at(g.A + (size_t)m0 * g.lda, a_bytes), w_all = hal_memory_at(g.W + (size_t)n0 * g.ldw, w_bytes);
  uint32_t minus[2] = {0x0000bf80u, 0xbf800000u};
  asm volatile("" : "+s"(minus[0]), "+s"(minus[1]));  // (as inline constants they would be taken for float32)

  // load i of a wave: rows 8 (8 i + wave) .. + 7 of the operand
  const int lr = lane / 8, piece = lane % 8;
  int put_at = (wave / 2) * 1024 + sp_slot(piece / 2, wave % 2 * 8 + lr) + piece % 2 * 8;
  // (rows past the end begin past the operands' bytes and are read as zeros)
  const uint32_t a_from = ((uint32_t)(wave * 8 + lr) * g.lda + piece * 4) * 4, w_from = ((uint32_t)(wave * 8 + lr) * g.ldw + piece * 4) * 4;
  sp_f32x4 p[LOADS];
  int first = 0, k_end = 0;  // the walk's first stage, and where its numbers end
  auto ask = [&](int stage, int i) {
    const int k = (first + stage) * SP_BK;
    const bool in = k + piece * 4 < k_end;  // (K is a multiple of 4; what lies past the end is read as zeros)
    const uint32_t apart = (uint32_t)(i < AL ? i * 64 * g.lda : (i - AL) * 64 * g.ldw) * 4 + (uint32_t)k * 4;
    p[i] = __builtin_bit_cast(sp_f32x4, __builtin_amdgcn_raw_buffer_load_b128(i < AL ? a_all : w_all, in ? (i < AL ? a_from : w_from) + apart : ~0u, 0, 0));
  };
  auto put = [&](int i) {
    uint32_t words[3][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) sp_split(p[i][2 * h], p[i][2 * h + 1], minus, words[0][h], words[1][h], words[2][h]);
    char* to = lds + put_at + (i < AL ? i * 4096 : W_AT + (i - AL) * 4096);
#pragma unroll
    for (int k = 0; k < 3; ++k) *(uint2*)(to + k * (i < AL ? A_PLANE : W_PLANE)) = make_uint2(words[k][0], words[k][1]);
  };
  const int wm = wave / WN, wn = wave % WN;
  int get_a = wm * NI * 1024 + sp_slot(lane / 16, lane % 16), get_w = W_AT + wn * NJ * 1024 + sp_slot(lane / 16, lane % 16);
  sp_f32x4 acc[NI][NJ], total[NI][NJ];
  auto of_a = [&](int k, int i) { return *(const sp_bf16x8*)(lds + get_a + k * A_PLANE + i * 1024); };
  auto of_w = [&](int k, int j) { return *(const sp_bf16x8*)(lds + get_w + k * W_PLANE + j * 1024); };
  auto meet = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  sp_bf16x8 a_hi[NI], a_mid[NI], a_lo[NI], w_even[NJ], w_odd[NJ], w_mid[NJ], w_lo[NJ];
  // The last of stage s's six products (w_hi: W's high parts), and the first five of the stage after it, which lies in
  // `mine` (its own: w_next), in groups of NJ instructions; beside them the stage after that goes from registers to
  // `next`, and one more is asked for.  `fresh`: the sums so far go to the totals, and new ones begin.
  auto turn = [&](int s, int to_mine, sp_bf16x8 (&w_hi)[NJ], sp_bf16x8 (&w_next)[NJ], const bool fresh) {
    // (one register each, whichever buffer it is: the compiler would keep both)
    get_a += to_mine, get_w += to_mine, put_at -= to_mine;
    asm volatile("" : "+v"(get_a), "+v"(get_w), "+v"(put_at));
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // (where few operands wait in registers, and early enough to lie in LDS at the barrier)
        const int at = t * 4 + i, load = at == 1 || at == 3 ? at / 2 : at >= 9 && at % 2 ? (at - 5) / 2 : LOADS;
        if (load < LOADS) {
          put(load);
          ask(s + 3, load);
        }
        if (t == 0) {
          a_lo[i] = of_a(2, i);
          if (i < NJ) w_next[i] = of_w(0, i);
        }
        if (t == 1) {
          a_mid[i] = of_a(1, i);
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            if (fresh) total[i][j] += acc[i][j];
        }
        if (t == 2 && i < NJ) w_mid[i] = of_w(1, i);
        if (t == 3) a_hi[i] = of_a(0, i);
        if (t == 4 && i < NJ) w_lo[i] = of_w(2, i);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const sp_bf16x8 w = t == 0 ? w_hi[j] : t < 3 ? w_next[j] : t < 5 ? w_mid[j] : w_lo[j];
          const sp_bf16x8 a = t == 1 ? a_lo[i] : t == 2 || t == 3 ? a_mid[i] : a_hi[i];
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, a, t == 1 && fresh ? sp_f32x4{0.f, 0.f, 0.f, 0.f} : acc[i][j], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    meet();
  };
  float* C = g.C + part * g.plane;
  const bool vectors = g.ldc % 4 == 0 && (uintptr_t)C % 16 == 0;
  bool odd = false;
  get_a += BYTES, get_w += BYTES;
  for (int walk = 0; walk < walks; ++walk) {
    first = part_first + part_stages * walk / walks;
    const int stages = part_first + part_stages * (walk + 1) / walks - first;
    k_end = min(g.K, (first + stages) * SP_BK);
    // (the stage before the first one: zeros)
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      a_hi[i] = sp_bf16x8{};
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = total[i][j] = sp_f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) w_odd[j] = sp_bf16x8{};
#pragma unroll
    for (int i = 0; i < LOADS; ++i) ask(0, i);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) put(i), ask(1, i);
    meet();
    for (int s = 0; s < stages; s += 2) {  // (stages past the end are zeros; left in the middle, the loop would need more registers)
      turn(s - 1, -BYTES, w_odd, w_even, true);
      turn(s, BYTES, w_even, w_odd, false);
    }
    // (the last product of the last stage)
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w_odd[j], a_hi[i], acc[i][j], 0, 0, 0);
    int l = lane;
    asm volatile("" : "+v"(l));  // (or where the results lie would be kept in registers over the walk)
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int r = (wm * NI + i) * 16 + l % 16;
      if (r >= rows_here) continue;
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int c = (wn * NJ + j) * 16 + l / 16 * 4;
        float* at = C + (size_t)(m0 + r) * g.ldc + n0 + c;
        sp_f32x4 sum = (total[i][j] + acc[i][j]) * (1.f / SP_SCALE / SP_SCALE);
        if (vectors && c + 3 < cols_here) {
          if (walk) sum += *(const sp_f32x4*)at;
          *(sp_f32x4*)at = sum;
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          if (c + v >= cols_here) continue;
          if (!(vectors && c + 3 < cols_here)) at[v] = sum[v] += walk ? at[v] : 0.f;
          odd |= !(fabsf(sum[v]) <= 3.4028235e38f);
        }
      }
    }
  }
  if (!__any(odd)) return;
  // Infinities and NaN among the operands, and numbers whose scaled parts are infinities, have no parts: every result that is not
  // finite (they all are not then) is taken again as a float32 sum, by the whole wave.
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "agent");
  const int k_begin = part_first * SP_BK;
  k_end = min(g.K, (part_first + part_stages) * SP_BK);
  for (int r = wm * 64; r < min(rows_here, wm * 64 + 64); ++r) {
    const float* a = g.A + (size_t)(m0 + r) * g.lda;
    const int c = wn * NJ * 16 + lane;
    const bool mine = lane < NJ * 16 && c < cols_here;
    const float v = mine ? __hip_atomic_load(C + (size_t)(m0 + r) * g.ldc + n0 + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.f;
    uint64_t todo = __ballot(!(fabsf(v) <= 3.4028235e38f));
    if (todo == 0) continue;
    bool nan = false;  // (a row with one: so are all its results)
    for (int k = k_begin + lane; k < k_end; k += 64) nan |= a[k] != a[k];
    if (__any(nan)) {
      if (mine) C[(size_t)(m0 + r) * g.ldc + n0 + c] = __builtin_nanf("");
      continue;
    }
    for (; todo; todo &= todo - 1) {
      const int n = n0 + wn * NJ * 16 + __builtin_ctzll(todo);
      const float* w = g.W + (size_t)n * g.ldw;
      float sum = 0.f;
      for (int k = k_begin + lane; k < k_end; k += 64) sum = fmaf(a[k], w[k], sum);
      sum = wave_sum(sum);
      if (lane == 0) C[(size_t)(m0 + r) * g.ldc + n] = sum;
    }
  }
}

// The parts' planes [rows][pitch], added up in order, four columns a thread.
__global__ void __launch_bounds__(256)
gemm_f32_planes_kernel(const float* __restrict__ planes, long long plane, int pitch, float* __restrict__ C, int ldc, int N, int parts) {
  const uint32_t at = (blockIdx.x * 256 + threadIdx.x) * 4;  // (a plane is 64 MiB or 1,024 rows of 8,192 at most)
  if (at >= (uint32_t)plane) return;
  const int r = at / (uint32_t)pitch, c = at % (uint32_t)pitch;
  sp_f32x4 v[SP_MOST_PARTS];
#pragma unroll
  for (int p = 0; p < SP_MOST_PARTS; ++p)
    if (p < parts) v[p] = *(const sp_f32x4*)(planes + p * plane + at);
#pragma unroll
  for (int p = 1; p < SP_MOST_PARTS; ++p)
    if (p < parts) v[0] += v[p];
  float* to = C + (size_t)r * ldc + c;
  if (c + 3 < N && ldc % 4 == 0 && (uintptr_t)C % 16 == 0) {
    *(sp_f32x4*)to = v[0];
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (c + e < N) to[e] = v[0][e];
  }
}

// Into how many parts K is cut: as many as it takes for 128 workgroups a tile of 256 rows, so that 500 rows of a matrix of 4,096 columns
// fill the chip once (one part 268 us, two 165, four 104, eight with twice the planes 117).
static int sp_parts(int N) {
  const int tiles_n = (N + SP_BN - 1) / SP_BN;
  return std::min(SP_MOST_PARTS, std::max(1, SP_UNITS / 2 / tiles_n));
}
static int sp_pitch(int N) { return (N + 3) / 4 * 4; }
// rows whose planes are held at once: whole tiles, as many as take SP_PLANES bytes, but 1,024 at least
static int sp_rows_at_once(int M, int N) {
  const long long fit = SP_PLANES / ((long long)sp_parts(N) * sp_pitch(N) * 4) / 256 * 256;
  return (int)std::min((long long)M, std::max(1024ll, fit));
}

// Whether a product is taken here, and how many float32 numbers of planes it needs (0: none).  More rows than 64: at 65 / 96 rows this
// and the kernel that splits K over a workgroup's waves take 39 / 40 and 73 / 75 us for 4,096 x 4,096, 58 / 60 and 69 / 75 for
// 6,144 x 4,096, 83 / 87 and 99 / 107 for 16,384 x 3,072, 183 / 186 and 240 / 267 for 28,672 x 4,096; below, that one reads a wide W at
// the memory's rate (28,672 x 4,096 at 64 rows in tiles of 64 columns 147).  Rows of 2,048 numbers or more: of
// 1,024 the planes' kernel costs what the parts gain (4,096 columns, 500 rows 45 us here, 41 there; 16,384 columns 90 / 139).
extern "C" int hal_gemm_f32_split_takes(const float* A, int lda, const float* W, int ldw, int M, int K) {
  return (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0 && M > 64 && K >= 2048 && K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && lda < SP_ROW_LIMIT && ldw < SP_ROW_LIMIT;
}
extern "C" long long hal_gemm_f32_split_planes(int M, int N) {
  return sp_parts(N) == 1 ? 0 : (long long)sp_parts(N) * sp_rows_at_once(M, N) * sp_pitch(N);
}

// How tiles of 256 rows go over the compute units: all of SP_BN columns, all of SP_BN_LOW, or SP_BN for whole rounds and SP_BN_LOW behind them (`first` columns
// are the former's; K in one part), and what that costs beside rounds of SP_BN.
struct SplitCut {
  int first;
  double rounds;
};
// (500 rows x 6,144 x 4,096 in parts, all lower: 153 -> 140 us; x 28,672 x 4,096, one round and a lower one for 448 tiles: 584 -> 574, less than the quarter of a round
// that it spares, as the chip holds a higher clock with a quarter of its units idle; 200 rows x 20,608 x 4,096 268 -> 239, 400 x 32,000 x 4,096 610 -> 596.)
#define SP_LOW_ROUND 0.79
static SplitCut sp_cut(int M, int N, int parts) {
  const long long rows = (M + 255) / 256;
  auto tiles = [&](int n, int cols) { return rows * ((n + cols - 1) / cols) * parts; };
  auto rounds = [&](long long n) { return (double)((n + SP_UNITS - 1) / SP_UNITS); };
  SplitCut best = {N, rounds(tiles(N, SP_BN))};
  if (SP_LOW_ROUND * rounds(tiles(N, SP_BN_LOW)) < best.rounds) best = {0, SP_LOW_ROUND * rounds(tiles(N, SP_BN_LOW))};
  const long long whole = tiles(N, SP_BN) / SP_UNITS, cols = whole * SP_UNITS / rows;
  if (parts == 1 && whole > 0 && cols > 0 && cols * SP_BN < N) {
    const double then = (double)(cols * rows + SP_UNITS - 1) / SP_UNITS;  // (a few units may stay without a tile)
    const double cost = (double)(long long)then + SP_LOW_ROUND * rounds(tiles(N - (int)cols * SP_BN, SP_BN_LOW)) + 0.02;
    if (cost < best.rounds) best = {(int)cols * SP_BN, cost};
  }
  return best;
}

// The rows of a tile: those whose rounds over the compute units are expected to end first, in microseconds a round of 128 stages (500 rows x 28,672 x
// 4,096 in tiles of 64 / 128 / 256: 743 / 730 / 629; 200 rows 396 / 356 / 304; 128 rows 207 / 195 / 304; 128 x 16,384 x 3,072 91 / 136 / 201;
// 128, 256 and 500 x 4,096 x 4,096 40 / 54 / 82, 68 / 63 / 89, 126 / 118 / 104).  A result's bits do not depend on it.
static int sp_tile_rows(int M, int N) {
  const long long n = (long long)((N + SP_BN - 1) / SP_BN) * sp_parts(N);
  auto cost = [&](int rows, int round) { return round * (((M + rows - 1) / rows * n + SP_UNITS - 1) / SP_UNITS); };
  const double low = (double)cost(64, 100), middle = (double)cost(128, 175), high = 300 * sp_cut(M, N, sp_parts(N)).rounds;
  return high <= middle && high <= low ? 256 : middle <= low ? 128 : 64;
}

extern "C" int hal_gemm_f32_split(const float* A, int lda, const float* W, int ldw, float* C, int ldc, float* planes, int M, int N, int K,
                                  hipStream_t stream) {
  HAL_REQUIRE(M > 0 && N > 0 && hal_gemm_f32_split_takes(A, lda, W, ldw, M, K), "hal_gemm_f32_split: M=%d N=%d K=%d", M, N, K);
  HAL_REQUIRE(lda >= K && ldw >= K && ldc >= N, "hal_gemm_f32_split: leading dimensions %d %d %d", lda, ldw, ldc);
  HAL_REQUIRE((uintptr_t)C % 4 == 0 && (uintptr_t)planes % 16 == 0, "hal_gemm_f32_split: addresses");
  const int parts = sp_parts(N), rows = parts == 1 ? M : sp_rows_at_once(M, N), pitch = sp_pitch(N);
  HAL_REQUIRE(parts == 1 || planes != nullptr, "hal_gemm_f32_split: no planes for %d parts", parts);
  const bool walks = ((K + SP_BK - 1) / SP_BK + parts - 1) / parts > SP_WALK;  // (parts differ by one stage at most)
  for (int m = 0; m < M; m += rows) {
    const int here = std::min(rows, M - m), tile = sp_tile_rows(here, N), tiles_m = (here + tile - 1) / tile;
    const long long plane = (long long)here * pitch;
    float* to = C + (size_t)m * ldc;
    const int first = tile == 256 ? sp_cut(here, N, parts).first : N;
#define SP_LAUNCH(BM_, BN_)                                                                                                               \
  do {                                                                                                                                    \
    if (walks) hipLaunchKernelGGL((gemm_f32_split_kernel<BM_, BN_, true>), dim3((unsigned)blocks), dim3(SP_THREADS), 0, stream, g);         \
    else hipLaunchKernelGGL((gemm_f32_split_kernel<BM_, BN_, false>), dim3((unsigned)blocks), dim3(SP_THREADS), 0, stream, g);              \
  } while (0)
    for (int low = 0; low < 2; ++low) {  // the columns of the wider tiles, and those behind them
      const int n0 = low ? first : 0, cols = low ? N - first : first, per = low ? SP_BN_LOW : SP_BN;
      if (cols <= 0) continue;
      const int tiles = (cols + per - 1) / per;
      const long long blocks = (long long)tiles_m * tiles * parts;
      HAL_REQUIRE(blocks < (1ll << 31), "hal_gemm_f32_split: M=%d N=%d exceed the grid limit", M, N);
      const SplitArgs g = {A + (size_t)m * lda, W + (size_t)n0 * ldw, (parts > 1 ? planes : to) + n0, lda, ldw, parts > 1 ? pitch : ldc, here, cols, K,
                           tiles_m, tiles, parts, plane};
      if (low) SP_LAUNCH(256, SP_BN_LOW);
      else if (tile == 256) SP_LAUNCH(256, SP_BN);
      else if (tile == 64) SP_LAUNCH(64, SP_BN);
      else SP_LAUNCH(128, SP_BN);
    }
#undef SP_LAUNCH
    if (parts > 1)
      hipLaunchKernelGGL(gemm_f32_planes_kernel, dim3((unsigned)((plane / 4 + 255) / 256)), dim3(256), 0, stream, planes, plane, pitch, to, ldc, N, parts);
    HAL_LAUNCH_CHECK();
  }
  return 0;
}
