// The generalized delta rule (see delta_rule.hip for what it computes) for heads of 64 over segments of several
// tokens, in chunks of 16 tokens as products on the matrix cores' float32 instruction
// (v_mfma_f32_16x16x4_f32: multiply and add in float32, none of the reduced-precision modes).
//
// Within a chunk let G_t be the product of the decays w_1 .. w_t (per key channel, G_0 = 1) and
// S_t = diag(G_t) Z_t.  Then Z_t = Z_(t-1) - e~_t q_t + k~_t v_t^T with q_t = u~_t^T Z_(t-1), where
//   u~_t = u_t G_(t-1),  e~_t = a_t u_t / G_t,  k~_t = k_t / G_t,  r~_t = r_t G_t,
// so that with the products L = U~ E~^T, M = U~ K~^T (below the diagonal), E = R~ E~^T and K = R~ K~^T (up
// to it) the chunk's rows are, in terms of the state Z_0 = S_0 before it,
//   Q = Wu Z_0 + Wm V          Wu = (I + L)^-1 U~,  Wm = (I + L)^-1 M   (forward substitution)
//   O = X Z_0 + N V            X = R~ - E Wu,       N = K - E Wm
//   S_n = diag(G_n) (Z_0 + K~^T V - E~^T Q).
// A decay is at least exp(-rate): 1 / G is at most exp(16 rate), 2e17 for the largest rate that the host lets through, which
// float32 holds far from its ends (k~ of keys above 1e21 would not be held, where the walk holds them).
//
// Two kernels.  delta_chunk_prep_kernel makes a chunk's record (Wu, X, E~, K~, Wm, N, G_n) for all chunks
// side by side, a wave a (chunk, head).  delta_chunk_scan_kernel walks a segment's chunks, a workgroup a
// (segment, head).  Norm, weight and gate of the heads are applied before the rows are written.
//
// What bounds it: the making of the records by vector instructions (some 2,800 a chunk and head) and the records' way to
// memory (2,250 tokens of 64 heads: 87 us, 300 MB), the walk by its chain of chunks, 1.6 us each where one request is long (52
// dependent instructions of 32 clocks are 0.8).  Measured with 64 heads beside the walk token by token and the norm and
// gate in a pass of their own: requests of 225, 450, 675 and 900 tokens 505 -> 192 us, one of 2,048 690 -> 290, one of 8,192
// 2,640 -> 1,150, one of 300 128 -> 61, 32 of 16 tokens each 125 -> 86.  Distance from 64 bits (2-norm) of the normed rows
// 1.55e-7 beside 1.47e-7, of the states 1.0e-7 beside 0.96e-7, largest differences 2.5e-7 beside 3.1e-7; at a rate of 2.5 and
// decays next to exp(-2.5) 5.4e-7 beside 4.6e-7 and 6.3e-8 beside 4.7e-8, next to 1 1.8e-7 beside 1.7e-7 and 2.4e-7 each.
#include "hal_lds.h"
#include "hal_api.h"

#define DK_D 64          // channels of a head
#define DK_TOKENS 16     // of a chunk
#define DK_RANKS 64      // entries of tanh(x1) that the prep kernel holds at a time
#define DK_HEADS 4       // heads (waves) of a workgroup of the prep kernel
#define DK_TILES (DK_D / 16)
#define DK_MAX_RATE 2.5f  // of the decay: exp(16 * 2.5) = 2e17 in 1 / G

typedef __attribute__((ext_vector_type(4))) float dk_f32x4;

// A chunk's record, in floats: four matrices of 16 rows of 64 (+ 4, so that the lanes of an LDS read meet
// different banks), two of 16 rows of 16 (+ 4), 64 decays; then, in LDS alone, the chunk's values and gates.
enum {
  DK_ROW = DK_D + 4,
  DK_SMALL = 20,
  DK_WU = 0,
  DK_X = 16 * DK_ROW,
  DK_E = 32 * DK_ROW,
  DK_K = 48 * DK_ROW,
  DK_WM = 64 * DK_ROW,
  DK_N = DK_WM + 16 * DK_SMALL,
  DK_G = DK_N + 16 * DK_SMALL,
  DK_RECORD = 20 * 256,  // whole KiB
  DK_VALUES = DK_RECORD,
  DK_GATES = DK_VALUES + 16 * DK_D,
  DK_BUFFER = DK_GATES + 16 * DK_D,
};
static_assert(DK_G + DK_D <= DK_RECORD, "a record");

// (the reciprocal and one step of Newton's; where 1 + exp(-x) is infinite the step would make a NaN of it)
__device__ __forceinline__ float dk_sigmoid(float x) {
  const float e = 1.0f + expf(-x), d = e > 1e37f ? 1e37f : e, y = __builtin_amdgcn_rcpf(d);
  return fmaf(fmaf(-d, y, 1.0f), y, y);
}

__device__ __forceinline__ void dk_wave_sync() {  // LDS of one wave: what its lanes wrote can be read by the others
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int BY>
__device__ __forceinline__ float dk_rotated(float x) {  // inside every 16 lanes
  return __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0x120 + BY, 0xf, 0xf, false));
}

// Chunks of the segments before segment `upto` (all lanes of a wave together).
__device__ __forceinline__ int dk_chunks_before(const int* __restrict__ seg_q_len, int upto) {
  const int lane = threadIdx.x % HAL_WAVE;
  int n = 0;
  for (int s = lane; s < upto; s += HAL_WAVE) n += (seg_q_len[s] + DK_TOKENS - 1) / DK_TOKENS;
#pragma unroll
  for (int off = 1; off < HAL_WAVE; off <<= 1) n += __shfl_xor(n, off, HAL_WAVE);
  return __builtin_amdgcn_readfirstlane(n);
}

// The segment of a chunk and the chunk's place in it; false: there are fewer chunks.
__device__ __forceinline__ bool dk_locate(const int* __restrict__ seg_q_len, int n_segs, int chunk, int& seg, int& place) {
  const int lane = threadIdx.x % HAL_WAVE;
  int before = 0;
  for (int s0 = 0; s0 < n_segs; s0 += HAL_WAVE) {
    const int mine = s0 + lane < n_segs ? (seg_q_len[s0 + lane] + DK_TOKENS - 1) / DK_TOKENS : 0;
    int upto = mine;
#pragma unroll
    for (int off = 1; off < HAL_WAVE; off <<= 1) {
      const int v = __shfl_up(upto, off, HAL_WAVE);
      if (lane >= off) upto += v;
    }
    const unsigned long long past = __builtin_amdgcn_ballot_w64(before + upto > chunk);
    if (past) {
      const int at = __builtin_ctzll(past);
      seg = s0 + at;
      place = __builtin_amdgcn_readfirstlane(chunk - before - __shfl(upto - mine, at, HAL_WAVE));
      return true;
    }
    before += __shfl(upto, HAL_WAVE - 1, HAL_WAVE);
  }
  return false;
}

// ---- a chunk's record: a wave takes one head of one chunk.  Lane l is key channel l with all tokens in registers
// (running products and the substitution need no other lane), and for the products on the matrix cores token l % 16
// with the channels 16 j + 4 g .. + 3 (g = l / 16); the rows change sides through LDS.
// The products of decays and what they multiply are made in 64 bits and rounded once: chains of float32 ones
// showed in the results (distance from 64 bits of a head's normed rows 2.8e-7 instead of 1.7e-7).
template <typename W, bool VEC>  // (VEC: rows of W2 are whole vectors of four, and lie at multiples of one)
__global__ void __launch_bounds__(DK_HEADS * HAL_WAVE, 4)
delta_chunk_prep_kernel(const float* __restrict__ r, int ldr, const float* __restrict__ k, int ldk,
                        const float* __restrict__ a_raw, int lda, const float* __restrict__ x1, int ldx1,
                        const W* __restrict__ w2, const W* __restrict__ w0, const W* __restrict__ a_bias, int lora,
                        float decay_rate, float unit_eps, const int* __restrict__ seg_q_start,
                        const int* __restrict__ seg_q_len, int n_segs, float* __restrict__ records, int H) {
  constexpr int ROOM = 4 * 16 * DK_SMALL;  // of a wave: 16 rows of 64, or the four products
  static_assert(ROOM >= 16 * DK_ROW, "rows fit the room");
  __shared__ __attribute__((aligned(16))) float tl[DK_TOKENS][DK_RANKS + 4];
  __shared__ __attribute__((aligned(16))) float rooms[DK_HEADS][ROOM];
  int seg, place;
  if (!dk_locate(seg_q_len, n_segs, blockIdx.x, seg, place)) return;  // (the same in all waves)
  const int lane = threadIdx.x % HAL_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / HAL_WAVE);
  const int tok = lane % 16, g = lane / 16;
  const int t0 = seg_q_start[seg] + place * DK_TOKENS;
  const int left = seg_q_len[seg] - place * DK_TOKENS, n = left < DK_TOKENS ? left : DK_TOKENS;
  const bool real = blockIdx.y * DK_HEADS + wave < H;  // (a wave without a head works on the last one's and writes nothing)
  const int h = real ? blockIdx.y * DK_HEADS + wave : H - 1;
  const size_t ch0 = (size_t)h * DK_D;
  float* const room = rooms[wave];
  float* const mine = room + tok * DK_ROW + 4 * g;  // for the matrix cores

  // the tokens' rows, on their way while the decays are made
  float kc[DK_TOKENS], ac[DK_TOKENS], rc[DK_TOKENS];
#pragma unroll
  for (int t = 0; t < DK_TOKENS; ++t) {
    const size_t row = t0 + (t < n ? t : n - 1);
    kc[t] = (k + row * ldk + ch0)[lane];
    ac[t] = (a_raw + row * lda + ch0)[lane];
    rc[t] = (r + row * ldr + ch0)[lane];
  }

  // W2 tanh(x1): rows are tokens, columns channels
  dk_f32x4 z[DK_TILES];
#pragma unroll
  for (int j = 0; j < DK_TILES; ++j) z[j] = dk_f32x4{0.f, 0.f, 0.f, 0.f};
  for (int j0 = 0; j0 < lora; j0 += DK_RANKS) {
    __syncthreads();
    for (int i = threadIdx.x; i < DK_TOKENS * DK_RANKS; i += DK_HEADS * HAL_WAVE) {
      const int it = i / DK_RANKS, ij = i % DK_RANKS;
      tl[it][ij] = it < n && j0 + ij < lora ? tanhf(x1[(size_t)(t0 + it) * ldx1 + j0 + ij]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int jb = 0; jb < DK_RANKS / 16; ++jb) {
      float w[DK_TILES][4];
      const int at = j0 + 16 * jb + 4 * g;  // (past the rank tanh(x1) is 0 and any weight will do)
      if (VEC) {
#pragma unroll
        for (int j = 0; j < DK_TILES; ++j) load4(w2 + (ch0 + 16 * j + tok) * lora + (at < lora ? at : 0), w[j]);
      } else {
#pragma unroll
        for (int j = 0; j < DK_TILES; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) w[j][i] = to_f32(w2[(ch0 + 16 * j + tok) * lora + (at + i < lora ? at + i : 0)]);
      }
      const dk_f32x4 x = *(const dk_f32x4*)&tl[tok][16 * jb + 4 * g];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < DK_TILES; ++j) z[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], w[j][i], z[j], 0, 0, 0);
    }
  }
#pragma unroll
  for (int j = 0; j < DK_TILES; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) room[(4 * g + i) * DK_ROW + 16 * j + tok] = z[j][i];
  dk_wave_sync();
  float zc[DK_TOKENS];
#pragma unroll
  for (int t = 0; t < DK_TOKENS; ++t) zc[t] = room[t * DK_ROW + lane];
  dk_wave_sync();
#pragma unroll
  for (int t = 0; t < DK_TOKENS; ++t) room[t * DK_ROW + lane] = kc[t];
  dk_wave_sync();
  float kk = 0.f;
#pragma unroll
  for (int j = 0; j < DK_TILES; ++j) {
    const dk_f32x4 v = *(const dk_f32x4*)(mine + 16 * j);
#pragma unroll
    for (int i = 0; i < 4; ++i) kk = fmaf(v[i], v[i], kk);
  }
  kk += __shfl_xor(kk, 16, HAL_WAVE);
  kk += __shfl_xor(kk, 32, HAL_WAVE);
  const double unit = 1.0 / sqrt((double)kk + (double)unit_eps);  // of token l % 16
  dk_wave_sync();

  __builtin_amdgcn_sched_barrier(0);
  // what the tokens contribute; a place past the chunk's tokens decays nothing and adds nothing
  const float bias0 = to_f32(w0[ch0 + lane]), bias_a = to_f32(a_bias[ch0 + lane]);
  // (what lies past the record's bytes is not written: a wave without a head has a record of none)
  const hal_memory rec = hal_memory_at(records + ((size_t)blockIdx.x * H + h) * DK_RECORD, real ? DK_RECORD * 4 : 0);
  auto put = [&](float value, int at, bool if_lane = true) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(value), rec, if_lane ? lane * 4 : DK_RECORD * 4, at * 4, 0);
  };
  float x[2][DK_TOKENS], y[2][DK_TOKENS];  // U~ and R~, M and K; then Wu and X, Wm and N
  double G = 1.0;
#pragma unroll
  for (int t = 0; t < DK_TOKENS; ++t) {
    const double of_t = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(unit), t), __builtin_amdgcn_readlane(__double2loint(unit), t));
    const double u = (double)kc[t] * of_t, before = G;
    const float w = expf(-decay_rate * dk_sigmoid(zc[t] + bias0));
    G = before * (double)(t < n ? w : 1.f);
    double inverse = (double)__builtin_amdgcn_rcpf((float)G);
    inverse = fma(fma(-G, inverse, 1.0), inverse, inverse);
    const float ut = (float)(u * before), et = (float)((double)dk_sigmoid(ac[t] + bias_a) * u * inverse);
    const float kt = (float)((double)kc[t] * inverse), rt = (float)((double)rc[t] * G);
    x[0][t] = t < n ? ut : 0.f, y[0][t] = t < n ? rt : 0.f;
    kc[t] = t < n ? kt : 0.f, ac[t] = t < n ? et : 0.f;
    if (t % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (registers: four tokens' numbers at a time)
  }
#pragma unroll
  for (int t = 0; t < DK_TOKENS; ++t) put(ac[t], DK_E + t * DK_ROW), put(kc[t], DK_K + t * DK_ROW);
  put((float)G, DK_G);
  __builtin_amdgcn_sched_barrier(0);

  // the four products of the chunk's tokens with each other; lane l of a result holds column (earlier
  // token) l % 16 and the rows (tokens) 4 g + i
  dk_f32x4 f[4][DK_TILES];  // u~, r~, e~, k~
  auto turned = [&](const float (&rows)[DK_TOKENS], dk_f32x4 (&to)[DK_TILES]) {
#pragma unroll
    for (int t = 0; t < DK_TOKENS; ++t) room[t * DK_ROW + lane] = rows[t];
    dk_wave_sync();
#pragma unroll
    for (int j = 0; j < DK_TILES; ++j) to[j] = *(const dk_f32x4*)(mine + 16 * j);
    dk_wave_sync();
  };
  turned(x[0], f[0]);
  turned(y[0], f[1]);
  turned(ac, f[2]);
  turned(kc, f[3]);
  dk_f32x4 m[4];  // L, E, M, K
#pragma unroll
  for (int j = 0; j < DK_TILES; ++j) {
    dk_f32x4 part[4];  // (a sum of its own for every 16 channels)
#pragma unroll
    for (int p = 0; p < 4; ++p) part[p] = dk_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int p = 0; p < 4; ++p)
        part[p] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[p % 2][j][i], f[2 + p / 2][j][i], part[p], 0, 0, 0);
#pragma unroll
    for (int p = 0; p < 4; ++p) m[p] = j == 0 ? part[p] : m[p] + part[p];
  }
#pragma unroll
  for (int p = 0; p < 4; ++p)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 4 * g + i;
      const bool seen = p % 2 == 0 ? tok < row : tok <= row;  // L and M: what came before; E and K: the token itself too
      room[(p * 16 + row) * DK_SMALL + tok] = seen ? m[p][i] : 0.f;
    }
  dk_wave_sync();

  __builtin_amdgcn_sched_barrier(0);
  // forward substitution, a lane a column: key channel l of U~ and R~, and (sixteen lanes) a column of M and K.
  // A row's factors are the same in all lanes.
  const float *L = room, *E = room + 16 * DK_SMALL;
#pragma unroll
  for (int row = 0; row < DK_TOKENS; ++row) {
    if (row % 2 == 0) __builtin_amdgcn_sched_barrier(0);  // (registers: the factors of two rows at a time)
    x[1][row] = room[(32 + row) * DK_SMALL + tok];
    y[1][row] = room[(48 + row) * DK_SMALL + tok];
#pragma unroll
    for (int s = 0; s <= row; s += 4) {
      const dk_f32x4 l = *(const dk_f32x4*)&L[row * DK_SMALL + s];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (s + i < row) {
          x[0][row] = fmaf(-l[i], x[0][s + i], x[0][row]);
          x[1][row] = fmaf(-l[i], x[1][s + i], x[1][row]);
        }
    }
#pragma unroll
    for (int s = 0; s <= row; s += 4) {
      const dk_f32x4 e = *(const dk_f32x4*)&E[row * DK_SMALL + s];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (s + i <= row) {
          y[0][row] = fmaf(-e[i], x[0][s + i], y[0][row]);
          y[1][row] = fmaf(-e[i], x[1][s + i], y[1][row]);
        }
    }
  }
#pragma unroll
  for (int t = 0; t < DK_TOKENS; ++t) put(x[0][t], DK_WU + t * DK_ROW), put(y[0][t], DK_X + t * DK_ROW);
  // (sixteen lanes have a column of the others; a branch around the stores would take the sums into it, and keep all factors for them)
#pragma unroll
  for (int t = 0; t < DK_TOKENS; ++t) put(x[1][t], DK_WM + t * DK_SMALL, lane < 16), put(y[1][t], DK_N + t * DK_SMALL, lane < 16);
}

struct DeltaGate {  // of the heads' results: y / rms(y over the head) * weight * sigmoid(z)
  const float* z;
  int ldz;
  const void* weight;
  int w_dtype;
  float eps;
};

// ---- the walk.  Four waves carry the state, 16 value channels each in registers (rows 16 j + 4 g + i of column
// l % 16, g = l / 16: which k of a product an instruction takes is free as long as both operands agree, so the
// accumulators are the second operand of the next product as they are): 52 instructions of 32 clocks a chunk, of
// which Q's and E~^T Q's wait for each other.  Four more waves on the same SIMDs do what nothing waits for: they bring
// records, values and gates, two chunks ahead; a chunk behind they make its rows from the state that the first
// four left in LDS; and another chunk behind they norm, gate and write them, a token sixteen lanes.  One barrier a
// chunk.  (Four arrays and not one, so that the compiler can tell a load into one from a read of another.)
#define DK_LOADS 7  // of a wave a chunk: five of the record, one of the values, one of the gates
template <typename T>
__global__ void __launch_bounds__(512)
delta_chunk_scan_kernel(const float* __restrict__ records, const float* __restrict__ v, int ldv, float* __restrict__ state,
                        const int* __restrict__ seg_q_start, const int* __restrict__ seg_q_len,
                        const int* __restrict__ token_slot, DeltaGate gate, T* __restrict__ out, int H) {
  __shared__ __attribute__((aligned(16))) float b0[DK_BUFFER], b1[DK_BUFFER], b2[DK_BUFFER], b3[DK_BUFFER];
  __shared__ __attribute__((aligned(16))) float starts[2][4][DK_TILES][HAL_WAVE * 4];  // the state before a chunk, by wave
  __shared__ __attribute__((aligned(16))) float made[2][DK_TOKENS * DK_ROW];           // a chunk's rows
  const int s = blockIdx.x, h = blockIdx.y;
  const int lane = threadIdx.x % HAL_WAVE, role = __builtin_amdgcn_readfirstlane(threadIdx.x / HAL_WAVE), wave = role % 4;
  const int col16 = lane % 16, g = lane / 16, col = wave * 16 + col16;
  const int t0 = seg_q_start[s], n = seg_q_len[s];
  if (n <= 0) return;
  const int chunks = (n + DK_TOKENS - 1) / DK_TOKENS;
  const dk_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  const int own16 = col16 * DK_SMALL + 4 * g, own64 = col16 * DK_ROW + 4 * g, across = 4 * g * DK_ROW + col16;

  if (role < 4) {
    float* st = state + ((size_t)token_slot[t0] * H + h) * DK_D * DK_D + col;
    dk_f32x4 Z[DK_TILES];
#pragma unroll
    for (int j = 0; j < DK_TILES; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) Z[j][i] = st[(16 * j + 4 * g + i) * DK_D];
    __builtin_amdgcn_s_setprio(2);  // (the other waves have time)
    auto advance = [&](int c, const float* mine) {
      hal_meet<0>();
      dk_f32x4 val, wu[DK_TILES], kt[DK_TILES], et[DK_TILES], add[DK_TILES], gone[DK_TILES], qs[DK_TILES];
      const dk_f32x4 wm = *(const dk_f32x4*)(mine + DK_WM + own16);
#pragma unroll
      for (int j = 0; j < DK_TILES; ++j) wu[j] = *(const dk_f32x4*)(mine + DK_WU + own64 + 16 * j);
#pragma unroll
      for (int i = 0; i < 4; ++i) val[i] = mine[DK_VALUES + (4 * g + i) * DK_D + col];
#pragma unroll
      for (int j = 0; j < DK_TILES; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) kt[j][i] = mine[DK_K + across + i * DK_ROW + 16 * j];
#pragma unroll
      for (int j = 0; j < DK_TILES; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) et[j][i] = mine[DK_E + across + i * DK_ROW + 16 * j];
#pragma unroll
      for (int j = 0; j < DK_TILES; ++j) *(dk_f32x4*)&starts[c & 1][wave][j][lane * 4] = Z[j];
      // (sums of their own for every 16 key channels, added up in the end: as short chains as the walk's token by token)
      dk_f32x4 q = zero;
#pragma unroll
      for (int j = 0; j < DK_TILES; ++j) qs[j] = add[j] = gone[j] = zero;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < DK_TILES; ++j) qs[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wu[j][i], Z[j][i], qs[j], 0, 0, 0);
        q = __builtin_amdgcn_mfma_f32_16x16x4f32(wm[i], val[i], q, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < DK_TILES; ++j) add[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[j][i], val[i], add[j], 0, 0, 0);
      q = (qs[0] + qs[1]) + (qs[2] + qs[3]) + q;
      // key channels 16 j + l % 16 are the rows of the first operand
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < DK_TILES; ++j) gone[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(et[j][i], q[i], gone[j], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < DK_TILES; ++j) Z[j] = (Z[j] + (add[j] - gone[j])) * *(const dk_f32x4*)(mine + DK_G + 16 * j + 4 * g);
    };
    for (int c = 0; c < chunks; c += 4) {
      advance(c, b0);
      if (c + 1 < chunks) advance(c + 1, b1);
      if (c + 2 < chunks) advance(c + 2, b2);
      if (c + 3 < chunks) advance(c + 3, b3);
    }
#pragma unroll
    for (int j = 0; j < DK_TILES; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) st[(16 * j + 4 * g + i) * DK_D] = Z[j][i];
    hal_meet<0>();  // (the others are two chunks behind)
    hal_meet<0>();
    return;
  }

  const float* const rec0 = records + ((size_t)dk_chunks_before(seg_q_len, s) * H + h) * DK_RECORD;
  const size_t first = (size_t)h * DK_D;
  const uint32_t in_row = col16 * 16, in_record = lane * 16;
  // (no branch: past the end the last chunk comes again and is not used)
  auto bring = [&](int chunk, float* to) {
    const int c = chunk < chunks ? chunk : chunks - 1;
    const hal_memory rec = hal_memory_at(rec0 + (size_t)c * H * DK_RECORD, DK_RECORD * 4);
#pragma unroll
    for (int j = 0; j < 5; ++j) hal_load_lds(rec, in_record, (j * 4 + wave) * 1024, to + (j * 4 + wave) * 256);
    const int before = c * DK_TOKENS, have = n - before < DK_TOKENS ? n - before : DK_TOKENS;
    int tok = wave * 4 + g;
    tok = tok < have ? tok : have - 1;
    const size_t row = t0 + before;
    const hal_memory values = hal_memory_at(v + row * ldv + first, (uint32_t)((have - 1) * ldv + DK_D) * 4);
    const hal_memory gates = hal_memory_at(gate.z + row * gate.ldz + first, (uint32_t)((have - 1) * gate.ldz + DK_D) * 4);
    hal_load_lds(values, (uint32_t)(tok * ldv) * 4 + in_row, 0, to + DK_VALUES + wave * 256);
    hal_load_lds(gates, (uint32_t)(tok * gate.ldz) * 4 + in_row, 0, to + DK_GATES + wave * 256);
  };
  // of the rows that are written this lane has token 4 wave + g, columns 4 (l % 16) .. + 3
  const int mine_at = (4 * wave + g) * DK_ROW + 4 * col16;
  float weight[4];
#pragma unroll
  for (int i = 0; i < 4; ++i)  // (one by one, once a workgroup: the weight may begin anywhere)
    weight[i] = gate.w_dtype == HAL_F32 ? ((const float*)gate.weight)[first + 4 * col16 + i] : to_f32(((const bf16_t*)gate.weight)[first + 4 * col16 + i]);
  dk_f32x4 zg = zero;  // the gates of the chunk that is written next
  T* const to = out + (size_t)(t0 + 4 * wave + g) * H * DK_D + first + 4 * col16;
  // Turn c: the record of chunk c - 1 is in `last`, that of chunk c + 2 goes to `free`.
  auto turn = [&](int c, const float* last, float* free) {
    hal_meet<DK_LOADS>();  // (chunk c is there, the next one may be on its way)
    bring(c + 2, free);
    __builtin_amdgcn_sched_barrier(0);
    dk_f32x4 Z[DK_TILES], x[DK_TILES], os[DK_TILES], val;
    bool odd = false;
#pragma unroll
    for (int j = 0; j < DK_TILES; ++j) {
      Z[j] = *(const dk_f32x4*)&starts[(c + 1) & 1][wave][j][lane * 4];
      x[j] = *(const dk_f32x4*)(last + DK_X + own64 + 16 * j);
      os[j] = zero;
    }
    const dk_f32x4 nn = *(const dk_f32x4*)(last + DK_N + own16);
    const dk_f32x4 ready = *(const dk_f32x4*)&made[c & 1][mine_at];
    const dk_f32x4 z_next = *(const dk_f32x4*)(last + DK_GATES + wave * 256 + lane * 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      val[i] = last[DK_VALUES + (4 * g + i) * DK_D + col];
      odd = odd || !(fabsf(val[i]) < INFINITY);
    }
    // An infinite or missing number among the values: the product over the chunk's tokens would bring it (times 0)
    // to the tokens before it, so it is left out of it and the rows from it on are made NaN by hand.
    int bad = DK_TOKENS;
    if (__builtin_amdgcn_ballot_w64(odd)) {
#pragma unroll
      for (int i = 3; i >= 0; --i)
        if (!(fabsf(val[i]) < INFINITY)) bad = 4 * g + i, val[i] = 0.f;
      bad = min(bad, __shfl_xor(bad, 16, HAL_WAVE));
      bad = min(bad, __shfl_xor(bad, 32, HAL_WAVE));
    }
    dk_f32x4 o = zero;  // chunk c - 1's rows (turn 0 and the last one make rows of nothing, which are not written)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int j = 0; j < DK_TILES; ++j) os[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j][i], Z[j][i], os[j], 0, 0, 0);
      o = __builtin_amdgcn_mfma_f32_16x16x4f32(nn[i], val[i], o, 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    // chunk c - 2's rows, while those products run
    float sq = ready[0] * ready[0] + ready[1] * ready[1] + (ready[2] * ready[2] + ready[3] * ready[3]);
    sq += dk_rotated<8>(sq);
    sq += dk_rotated<4>(sq);
    sq += dk_rotated<2>(sq);
    sq += dk_rotated<1>(sq);
    const float rstd = 1.0f / sqrtf(sq / (float)DK_D + gate.eps);
    float put[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) put[i] = ready[i] * rstd * weight[i] * dk_sigmoid(zg[i]);
    zg = z_next;
    if (c >= 2 && (c - 2) * DK_TOKENS + 4 * wave + g < n) store4(to + (size_t)(c - 2) * DK_TOKENS * H * DK_D, put);
    __builtin_amdgcn_sched_barrier(0);
    o = (os[0] + os[1]) + (os[2] + os[3]) + o;
#pragma unroll
    for (int i = 0; i < 4; ++i) made[(c + 1) & 1][(4 * g + i) * DK_ROW + col] = 4 * g + i >= bad ? __builtin_nanf("") : o[i];
  };
  bring(0, b0);
  bring(1, b1);
  for (int c = 0; c < chunks + 2; c += 4) {
    turn(c, b3, b2);
    if (c + 1 < chunks + 2) turn(c + 1, b0, b3);
    if (c + 2 < chunks + 2) turn(c + 2, b1, b0);
    if (c + 3 < chunks + 2) turn(c + 3, b2, b1);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // LDS is not given back while loads are on their way into it
}

// floats of room for the records of a step of n_tokens in n_segs segments (every segment's last chunk may be a short one)
extern "C" long long hal_delta_chunks_room(int n_tokens, int n_segs, int H) {
  return ((long long)n_tokens / DK_TOKENS + n_segs) * H * DK_RECORD;
}

// Whether heads of D channels, a decay of that rate, and rows of values and gates of that length and place have kernels here.
extern "C" int hal_delta_chunks_fit(int D, float decay_rate, const float* v, int ldv, const float* z, int ldz) {
  return D == DK_D && decay_rate <= DK_MAX_RATE && ldv % 4 == 0 && ldv < (1 << 24) && (uintptr_t)v % 16 == 0 && ldz % 4 == 0 &&
         ldz < (1 << 24) && (uintptr_t)z % 16 == 0;
}

// Arguments as of hal_delta_rule; z [T, H * D] float32 with rows of ldz, weight [H * D]: out[t] = norm over each head
// of o[t], times weight times sigmoid(z), of type `dtype`.  records: room for hal_delta_chunks_room floats.
extern "C" int hal_delta_chunks(const float* r, int ldr, const float* k, int ldk, const float* v, int ldv, const float* a_raw,
                                int lda, const float* x1, int ldx1, const void* w2, const void* w0, const void* a_bias,
                                int w_dtype, int lora, float decay_rate, float unit_eps, float* records, float* state,
                                const int* seg_q_start, const int* seg_q_len, const int* token_slot, const float* z, int ldz,
                                const void* weight, int weight_dtype, float eps, void* out, int dtype, int n_tokens, int n_segs,
                                int H, int D, hipStream_t stream) {
  HAL_REQUIRE(n_tokens >= 0 && n_segs >= 0 && H > 0 && lora > 0, "hal_delta_chunks: bad sizes T=%d segments=%d heads=%d lora=%d",
              n_tokens, n_segs, H, lora);
  HAL_REQUIRE(hal_delta_chunks_fit(D, decay_rate, v, ldv, z, ldz),
              "hal_delta_chunks: no kernel for heads of %d, rate %f, rows of values of %d, of gates of %d", D, decay_rate, ldv, ldz);
  HAL_REQUIRE(H <= 65535, "hal_delta_chunks: %d heads exceed the grid limit", H);
  HAL_REQUIRE(ldr >= H * D && ldk >= H * D && ldv >= H * D && lda >= H * D && ldz >= H * D && ldx1 >= lora, "hal_delta_chunks: rows too short");
  HAL_REQUIRE((w_dtype == HAL_F32 || w_dtype == HAL_BF16) && (weight_dtype == HAL_F32 || weight_dtype == HAL_BF16) &&
                  (dtype == HAL_F32 || dtype == HAL_BF16),
              "hal_delta_chunks: dtypes %d, %d, %d", w_dtype, weight_dtype, dtype);
  HAL_REQUIRE(z && weight && out && records && state, "hal_delta_chunks: arguments missing");
  HAL_REQUIRE((uintptr_t)records % 16 == 0 && (uintptr_t)out % (dtype == HAL_F32 ? 16 : 8) == 0, "hal_delta_chunks: records or results off a vector");
  if (n_tokens == 0 || n_segs == 0) return 0;
  const dim3 all((unsigned)(n_tokens / DK_TOKENS + n_segs), (H + DK_HEADS - 1) / DK_HEADS);
#define DK_PREP(W_, VEC_)                                                                                                     \
  hipLaunchKernelGGL((delta_chunk_prep_kernel<W_, VEC_>), all, dim3(DK_HEADS * HAL_WAVE), 0, stream, r, ldr, k, ldk, a_raw, lda, \
                     x1, ldx1, (const W_*)w2, (const W_*)w0, (const W_*)a_bias, lora, decay_rate, unit_eps, seg_q_start,        \
                     seg_q_len, n_segs, records, H)
  const bool vec = lora % 4 == 0 && (uintptr_t)w2 % (w_dtype == HAL_F32 ? 16 : 8) == 0;
  if (w_dtype == HAL_F32) {
    if (vec) DK_PREP(float, true);
    else DK_PREP(float, false);
  } else {
    if (vec) DK_PREP(bf16_t, true);
    else DK_PREP(bf16_t, false);
  }
#undef DK_PREP
  HAL_LAUNCH_CHECK();
  const DeltaGate gate = {z, ldz, weight, weight_dtype, eps};
#define DK_SCAN(T_)                                                                                                        \
  hipLaunchKernelGGL(delta_chunk_scan_kernel<T_>, dim3(n_segs, H), dim3(512), 0, stream, records, v, ldv, state, seg_q_start, \
                     seg_q_len, token_slot, gate, (T_*)out, H)
  if (dtype == HAL_F32) DK_SCAN(float);
  else DK_SCAN(bf16_t);
#undef DK_SCAN
  HAL_LAUNCH_CHECK();
  return 0;
}
