// Small kernels around a latent attention and a mixture of experts.  All arithmetic is
// float32; T is the element type of activations (float or bf16).
//
//   * RMSNorm of the float32 stream with one or two weights at once (the two norms of a
//     block whose mixer and feed-forward read the same rows), x * rstd * w in float32 and
//     one rounding at the end;
//   * the step between the down projections of a latent attention and its cache: norms of
//     the query latent and of the key/value latent, and the key and value rows that the
//     paged attention kernels take;
//   * column ranges copied head by head;
//   * the product of a router's few columns, in parts of K;
//   * the router of a mixture of experts: scores, the chosen `top` (also by corrected scores and
//     among the best groups of neighbours), their weights;
//   * a counting sort of the (token, choice) pairs by expert, on the device;
//   * the weighted sum of the chosen experts' results, added into the stream.
#include "hal_common.h"
#include "hal_api.h"

// ---------------------------------------------------------------------------------
// out1[r] = T(x * rstd * w1), out2[r] = T(x * rstd * w2) with x = h[rows ? rows[r] : r]
// ---------------------------------------------------------------------------------
template <typename T>
__global__ void norm_pair_kernel(const float* __restrict__ h, const int* __restrict__ rows,
                                 const void* __restrict__ w1, const void* __restrict__ w2, int w_dtype,
                                 float eps, T* __restrict__ out1, T* __restrict__ out2, int d) {
  __shared__ float scratch[16];
  const int r = blockIdx.x;
  const float* hr = h + (size_t)(rows ? rows[r] : r) * d;
  float ss = 0.f;
  for (int i = threadIdx.x; i < d; i += blockDim.x) {
    const float x = hr[i];
    ss += x * x;
  }
  const float total = block_sum(ss, scratch);
  const float rstd = 1.0f / sqrtf(total / (float)d + eps);
  for (int i = threadIdx.x; i < d; i += blockDim.x) {
    const float x = hr[i] * rstd;
    out1[(size_t)r * d + i] = from_f32<T>(x * load_as_f32(w1, w_dtype, i));
    if (w2) out2[(size_t)r * d + i] = from_f32<T>(x * load_as_f32(w2, w_dtype, i));
  }
}

// The same with the row held in registers: one pass over memory, four numbers an access, all loads (the weights' too) issued
// before the first use.  d is a multiple of 4 and at most 4 * MAXV * blockDim.x, rows and weights lie at multiples of
// four numbers.  Many rows: NP_MAXV vectors a thread, so that a compute unit holds rows in every phase (bound by memory: 3,000
// rows of 4,096 with two weights 38.5 -> 27.4 us, 98 MB).  Few: one, for the shortest code, which is
// mostly fetched (8 rows 7.0 -> 4.5 us; with NP_MAXV vectors 9.9).
#define NP_MAXV 8
template <typename T, bool PAIR, int MAXV>
__global__ void norm_pair_vec_kernel(const float* __restrict__ h, const int* __restrict__ rows,
                                     const void* __restrict__ w1, const void* __restrict__ w2, int w_dtype,
                                     float eps, T* __restrict__ out1, T* __restrict__ out2, int d) {
  __shared__ float scratch[16];
  const int r = blockIdx.x, nv = d / 4;
  const float* hr = h + (size_t)(rows ? rows[r] : r) * d;
  float x[MAXV][4], a[MAXV][4], b[MAXV][4];
#pragma unroll
  for (int u = 0; u < MAXV; ++u) {
    const int v = threadIdx.x + u * blockDim.x;
    if (v < nv) load4(hr + v * 4, x[u]);
  }
#pragma unroll
  for (int u = 0; u < MAXV; ++u) {
    const int v = threadIdx.x + u * blockDim.x;
    if (v < nv) {
      load4_any(w1, w_dtype, (size_t)v * 4, a[u]);
      if (PAIR) load4_any(w2, w_dtype, (size_t)v * 4, b[u]);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < MAXV; ++u)
    if (threadIdx.x + u * blockDim.x < nv) {
#pragma unroll
      for (int i = 0; i < 4; ++i) ss += x[u][i] * x[u][i];
    }
  const float total = block_sum(ss, scratch);
  const float rstd = 1.0f / sqrtf(total / (float)d + eps);
#pragma unroll
  for (int u = 0; u < MAXV; ++u) {
    const int v = threadIdx.x + u * blockDim.x;
    if (v < nv) {
      float y[4], z[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[u][i] *= rstd;
        y[i] = x[u][i] * a[u][i];
        if (PAIR) z[i] = x[u][i] * b[u][i];
      }
      store4(out1 + (size_t)r * d + v * 4, y);
      if (PAIR) store4(out2 + (size_t)r * d + v * 4, z);
    }
  }
}

extern "C" int hal_norm_pair(const float* h, const int* rows, const void* w1, const void* w2,
                             int w_dtype, float eps, void* out1, void* out2, int dtype, int n_rows,
                             int d, hipStream_t stream) {
  HAL_REQUIRE(n_rows >= 0 && d > 0, "hal_norm_pair: bad sizes rows=%d d=%d", n_rows, d);
  HAL_REQUIRE(dtype == HAL_F32 || dtype == HAL_BF16, "hal_norm_pair: dtype %d", dtype);
  HAL_REQUIRE((w2 == nullptr) == (out2 == nullptr), "hal_norm_pair: a second weight and a second result come together");
  if (n_rows == 0) return 0;
  if (d % 4 == 0 && d <= 4096 * NP_MAXV && ((uintptr_t)h | (uintptr_t)w1 | (uintptr_t)w2 | (uintptr_t)out1 | (uintptr_t)out2) % 16 == 0) {
    const int maxv = n_rows < 256 && d <= 4096 ? 1 : NP_MAXV, lanes = ((d / 4 + maxv - 1) / maxv + 63) / 64 * 64;
#define NP_LAUNCH(T_, PAIR_, MAXV_) \
  hipLaunchKernelGGL((norm_pair_vec_kernel<T_, PAIR_, MAXV_>), dim3(n_rows), dim3(lanes), 0, stream, h, rows, w1, w2, w_dtype, eps, (T_*)out1, (T_*)out2, d)
#define NP_BY_ROWS(T_, PAIR_)                    \
  do {                                           \
    if (maxv == 1) NP_LAUNCH(T_, PAIR_, 1);      \
    else NP_LAUNCH(T_, PAIR_, NP_MAXV);          \
  } while (0)
    if (dtype == HAL_F32 && w2) NP_BY_ROWS(float, true);
    else if (dtype == HAL_F32) NP_BY_ROWS(float, false);
    else if (w2) NP_BY_ROWS(bf16_t, true);
    else NP_BY_ROWS(bf16_t, false);
#undef NP_BY_ROWS
#undef NP_LAUNCH
    HAL_LAUNCH_CHECK();
    return 0;
  }
  int threads = ((d + 3) / 4 + 63) / 64 * 64;
  if (threads > 1024) threads = 1024;
  if (dtype == HAL_F32)
    hipLaunchKernelGGL(norm_pair_kernel<float>, dim3(n_rows), dim3(threads), 0, stream, h, rows, w1, w2,
                       w_dtype, eps, (float*)out1, (float*)out2, d);
  else
    hipLaunchKernelGGL(norm_pair_kernel<bf16_t>, dim3(n_rows), dim3(threads), 0, stream, h, rows, w1,
                       w2, w_dtype, eps, (bf16_t*)out1, (bf16_t*)out2, d);
  HAL_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------------
// The same with what a layer left to be added: h[t] <- (h[t] + beside[t]) + s[t], s the weighted sum of a mixture's experts
// (as hal_moe_combine adds it up), then the norms of the new row.  With `rows` those rows alone, and h stays as it is (the
// last norm reads a few).  A thread holds its part of the new row; the rows of up to four experts are on their way together.
// Bound by memory; what is saved is the stream's way out and back, twice, and two launches.  Three passes / this one, six experts, a row
// beside and an extra one, two weights, us: 8 rows of 4,096 5.2 / 4.1, 64 8.3 / 4.4, 300 21.7 / 10.8, 3,000 130 / 101 (540 MB); 8,192 of
// 2,048 with four 146 / 114.  One group of four numbers a thread where a workgroup can have as many (3,000 rows: two groups 105, four
// 109, eight 121: a group's rows wait for the group's before).
// ---------------------------------------------------------------------------------
struct AddedRows {
  const float* beside;  // [T, d], or null
  const float* y;       // [T * top, d]
  const float* wgt;     // [T, top]
  const float* extra;   // [T, d], or null
  const float* gate;    // [T] with rows of ld_gate, or null: sigmoid(gate) times `extra`
  int ld_gate, top;
};
template <typename T, bool PAIR, int MAXV>
__global__ void __launch_bounds__(1024) norm_added_vec_kernel(float* __restrict__ h, AddedRows e, const int* __restrict__ rows,
                                                              const void* __restrict__ w1, const void* __restrict__ w2, int w_dtype,
                                                              float eps, T* __restrict__ out1, T* __restrict__ out2, int d) {
  __shared__ float scratch[16];
  const int r = blockIdx.x, nv = d / 4;
  const size_t t = rows ? rows[r] : r;
  const float eg = e.gate ? 1.0f / (1.0f + expf(-e.gate[t * e.ld_gate])) : 1.0f;
  const float* w = e.wgt + t * e.top;
  float x[MAXV][4];
  float ss = 0.f;
#pragma unroll
  for (int u = 0; u < MAXV; ++u) {
    const int v = threadIdx.x + u * blockDim.x;
    if (v >= nv) continue;
    float b[4], s[4] = {0.f, 0.f, 0.f, 0.f};
    load4(h + t * d + v * 4, x[u]);
    if (e.beside) load4_once(e.beside + t * d + v * 4, b);
    if (e.extra) load4_once(e.extra + t * d + v * 4, s);
    const float* at = e.y + t * e.top * d + v * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) s[i] *= eg;
    for (int j0 = 0; j0 < e.top; j0 += 4) {
      float part[4][4], c[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int which = j0 + j < e.top ? j0 + j : j0;  // (past the end: a row that is there, not added)
        load4_once(at + (size_t)which * d, part[j]);
        c[j] = w[which];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j0 + j >= e.top) break;
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] += c[j] * part[j][i];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (e.beside) x[u][i] += b[i];
      x[u][i] += s[i];
      ss += x[u][i] * x[u][i];
    }
    if (!rows) store4(h + t * d + v * 4, x[u]);
  }
  const float total = block_sum(ss, scratch);
  const float rstd = 1.0f / sqrtf(total / (float)d + eps);
#pragma unroll
  for (int u = 0; u < MAXV; ++u) {
    const int v = threadIdx.x + u * blockDim.x;
    if (v >= nv) continue;
    float a[4], b[4], y[4], z[4];
    load4_any(w1, w_dtype, (size_t)v * 4, a);
    if (PAIR) load4_any(w2, w_dtype, (size_t)v * 4, b);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[u][i] *= rstd;
      y[i] = x[u][i] * a[i];
      if (PAIR) z[i] = x[u][i] * b[i];
    }
    store4(out1 + (size_t)r * d + v * 4, y);
    if (PAIR) store4(out2 + (size_t)r * d + v * 4, z);
  }
}

// Rows of a multiple of four numbers up to NA_MOST, at places of 16 bytes.
#define NA_MOST 16384
extern "C" int hal_norm_pair_added(float* h, const float* beside, const float* y, const float* wgt, const float* extra,
                                   const float* extra_gate, int ld_gate, int top, const int* rows, const void* w1, const void* w2,
                                   int w_dtype, float eps, void* out1, void* out2, int dtype, int n_rows, int d, hipStream_t stream) {
  HAL_REQUIRE(n_rows >= 0 && d > 0 && d % 4 == 0 && d <= NA_MOST && top > 0 && y && wgt, "hal_norm_pair_added: bad sizes rows=%d d=%d top=%d",
              n_rows, d, top);
  HAL_REQUIRE(dtype == HAL_F32 || dtype == HAL_BF16, "hal_norm_pair_added: dtype %d", dtype);
  HAL_REQUIRE((w2 == nullptr) == (out2 == nullptr), "hal_norm_pair_added: a second weight and a second result come together");
  HAL_REQUIRE(((uintptr_t)h | (uintptr_t)beside | (uintptr_t)y | (uintptr_t)extra | (uintptr_t)w1 | (uintptr_t)w2 | (uintptr_t)out1 |
               (uintptr_t)out2) % 16 == 0, "hal_norm_pair_added: rows must be 16-byte aligned");
  if (n_rows == 0) return 0;
  const AddedRows e = {beside, y, wgt, extra, extra ? extra_gate : nullptr, ld_gate, top};
  const int v = d <= 4096 ? 1 : 4;
  const int lanes = ((d / 4 + v - 1) / v + 63) / 64 * 64;
#define NA_LAUNCH(T_, PAIR_, V_) \
  hipLaunchKernelGGL((norm_added_vec_kernel<T_, PAIR_, V_>), dim3(n_rows), dim3(lanes), 0, stream, h, e, rows, w1, w2, w_dtype, eps, (T_*)out1, (T_*)out2, d)
#define NA_BY_WIDTH(T_, PAIR_)            \
  do {                                    \
    if (v == 1) NA_LAUNCH(T_, PAIR_, 1);  \
    else NA_LAUNCH(T_, PAIR_, 4);         \
  } while (0)
  if (dtype == HAL_F32 && w2) NA_BY_WIDTH(float, true);
  else if (dtype == HAL_F32) NA_BY_WIDTH(float, false);
  else if (w2) NA_BY_WIDTH(bf16_t, true);
  else NA_BY_WIDTH(bf16_t, false);
#undef NA_BY_WIDTH
#undef NA_LAUNCH
  HAL_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------------
// a [T, lda] float32 holds, per token, the query latent (q_rank, from column q_col0; none
// if q_rank == 0), then at kv_col0 the key/value latent (kv_rank) and the shared rotated key
// part (rot, not normed).
//   cq[t]         = T(rmsnorm(query latent) * wq)
//   k row of t    = [rotated part (not yet rotated) | T(rmsnorm(latent) * wkv) | 0 ...]   (D)
//   v row of t    = [0 ...                          | the same                 | 0 ...]   (D)
// in the packed rows `qkv` at columns k_col0 and k_col0 + D.
// ---------------------------------------------------------------------------------
template <typename T>
__global__ void latent_prep_kernel(const float* __restrict__ a, int lda, int q_col0, int q_rank,
                                   int kv_col0, int kv_rank, int rot, int D, const void* wq,
                                   const void* wkv, int w_dtype, float eps, T* __restrict__ cq,
                                   T* __restrict__ qkv, int row_stride, int k_col0) {
  __shared__ float scratch[16];
  const int t = blockIdx.x;
  const float* ar = a + (size_t)t * lda;
  if (q_rank > 0) {
    float ss = 0.f;
    for (int i = threadIdx.x; i < q_rank; i += blockDim.x) ss += ar[q_col0 + i] * ar[q_col0 + i];
    const float rstd = 1.0f / sqrtf(block_sum(ss, scratch) / (float)q_rank + eps);
    for (int i = threadIdx.x; i < q_rank; i += blockDim.x)
      cq[(size_t)t * q_rank + i] = from_f32<T>(ar[q_col0 + i] * rstd * load_as_f32(wq, w_dtype, i));
  }
  float ss = 0.f;
  for (int i = threadIdx.x; i < kv_rank; i += blockDim.x) ss += ar[kv_col0 + i] * ar[kv_col0 + i];
  const float rstd = 1.0f / sqrtf(block_sum(ss, scratch) / (float)kv_rank + eps);
  T* k = qkv + (size_t)t * row_stride + k_col0;
  T* v = k + D;
  for (int i = threadIdx.x; i < D; i += blockDim.x) {
    float kx = 0.f, vx = 0.f;
    if (i < rot) {
      kx = ar[kv_col0 + kv_rank + i];
    } else if (i < rot + kv_rank) {
      const int c = i - rot;
      // rounded once, so that keys and values hold the same number
      kx = vx = to_f32(from_f32<T>(ar[kv_col0 + c] * rstd * load_as_f32(wkv, w_dtype, c)));
    }
    k[i] = from_f32<T>(kx);
    v[i] = from_f32<T>(vx);
  }
}

// The same where all sizes, columns and addresses are multiples of four numbers and 256 threads hold the latents in
// registers (LP_MAXV vectors each of the query's, one of the key's): every load on its way before the first sum, both
// sums at once.  3,000 tokens of 1,536 + 192 + 64, heads of 256: 17.5 -> 10.6 us (33 MB), 8 tokens 8.1 -> 4.8.
#define LP_MAXV 4
#define LP_THREADS 256
template <typename T>
__global__ void __launch_bounds__(LP_THREADS)
latent_prep_vec_kernel(const float* __restrict__ a, int lda, int q_col0, int q_rank, int kv_col0, int kv_rank, int rot, int D,
                       const void* wq, const void* wkv, int w_dtype, float eps, T* __restrict__ cq,
                       T* __restrict__ qkv, int row_stride, int k_col0) {
  __shared__ float sums[2][LP_THREADS / HAL_WAVE];
  const int t = blockIdx.x, tid = threadIdx.x, qv = q_rank / 4;
  const float* ar = a + (size_t)t * lda;
  float x[LP_MAXV][4], w[LP_MAXV][4], c[4] = {0.f, 0.f, 0.f, 0.f}, wc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < LP_MAXV; ++u) {
    const int v = tid + u * LP_THREADS;
    if (v < qv) load4(ar + q_col0 + v * 4, x[u]);
  }
  // thread tid has the key row's numbers 4 tid .. 4 tid + 3: the rotated part, then the latent, then zeros
  const int i = tid * 4, in_latent = i - rot;
  const bool latent = in_latent >= 0 && in_latent < kv_rank;
  if (i < rot) load4(ar + kv_col0 + kv_rank + i, c);
  else if (latent) load4(ar + kv_col0 + in_latent, c), load4_any(wkv, w_dtype, in_latent, wc);
#pragma unroll
  for (int u = 0; u < LP_MAXV; ++u) {
    const int v = tid + u * LP_THREADS;
    if (v < qv) load4_any(wq, w_dtype, (size_t)v * 4, w[u]);
  }
  float sq = 0.f, sk = 0.f;
#pragma unroll
  for (int u = 0; u < LP_MAXV; ++u)
    if (tid + u * LP_THREADS < qv) {
#pragma unroll
      for (int k = 0; k < 4; ++k) sq += x[u][k] * x[u][k];
    }
  if (latent) {
#pragma unroll
    for (int k = 0; k < 4; ++k) sk += c[k] * c[k];
  }
#pragma unroll
  for (int off = HAL_WAVE / 2; off; off /= 2) {
    sq += __shfl_xor(sq, off, HAL_WAVE);
    sk += __shfl_xor(sk, off, HAL_WAVE);
  }
  if (tid % HAL_WAVE == 0) sums[0][tid / HAL_WAVE] = sq, sums[1][tid / HAL_WAVE] = sk;
  __syncthreads();
  sq = sk = 0.f;
#pragma unroll
  for (int k = 0; k < LP_THREADS / HAL_WAVE; ++k) sq += sums[0][k], sk += sums[1][k];
  if (q_rank > 0) {
    const float rstd = 1.0f / sqrtf(sq / (float)q_rank + eps);
#pragma unroll
    for (int u = 0; u < LP_MAXV; ++u) {
      const int v = tid + u * LP_THREADS;
      if (v < qv) {
#pragma unroll
        for (int k = 0; k < 4; ++k) x[u][k] = x[u][k] * rstd * w[u][k];
        store4(cq + (size_t)t * q_rank + v * 4, x[u]);
      }
    }
  }
  if (i < D) {
    const float rstd = 1.0f / sqrtf(sk / (float)kv_rank + eps);
    float kx[4], vx[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      // (rounded once, so that keys and values hold the same number)
      vx[k] = latent ? to_f32(from_f32<T>(c[k] * rstd * wc[k])) : 0.f;
      kx[k] = latent ? vx[k] : c[k];
    }
    T* k = qkv + (size_t)t * row_stride + k_col0 + i;
    store4(k, kx);
    store4(k + D, vx);
  }
}

extern "C" int hal_latent_prep(const float* a, int lda, int q_col0, int q_rank, int kv_col0,
                               int kv_rank, int rot, int D, const void* wq, const void* wkv,
                               int w_dtype, float eps, void* cq, void* qkv, int row_stride,
                               int k_col0, int dtype, int n_tokens, hipStream_t stream) {
  HAL_REQUIRE(n_tokens >= 0 && kv_rank > 0 && rot >= 0 && q_rank >= 0 && D >= rot + kv_rank,
              "hal_latent_prep: bad sizes T=%d q_rank=%d kv_rank=%d rot=%d D=%d", n_tokens, q_rank, kv_rank,
              rot, D);
  HAL_REQUIRE(q_col0 >= 0 && kv_col0 >= 0 && q_col0 + q_rank <= lda && kv_col0 + kv_rank + rot <= lda &&
                  k_col0 >= 0 && k_col0 + 2 * D <= row_stride,
              "hal_latent_prep: columns outside the rows");
  HAL_REQUIRE(dtype == HAL_F32 || dtype == HAL_BF16, "hal_latent_prep: dtype %d", dtype);
  if (n_tokens == 0) return 0;
  if (!((q_col0 | q_rank | kv_col0 | kv_rank | rot | D | lda | row_stride | k_col0) % 4) && q_rank <= 4 * LP_MAXV * LP_THREADS &&
      D <= 4 * LP_THREADS && ((uintptr_t)a | (uintptr_t)wq | (uintptr_t)wkv | (uintptr_t)cq | (uintptr_t)qkv) % 16 == 0) {
    if (dtype == HAL_F32)
      hipLaunchKernelGGL(latent_prep_vec_kernel<float>, dim3(n_tokens), dim3(LP_THREADS), 0, stream, a, lda, q_col0, q_rank, kv_col0,
                         kv_rank, rot, D, wq, wkv, w_dtype, eps, (float*)cq, (float*)qkv, row_stride, k_col0);
    else
      hipLaunchKernelGGL(latent_prep_vec_kernel<bf16_t>, dim3(n_tokens), dim3(LP_THREADS), 0, stream, a, lda, q_col0, q_rank, kv_col0,
                         kv_rank, rot, D, wq, wkv, w_dtype, eps, (bf16_t*)cq, (bf16_t*)qkv, row_stride, k_col0);
    HAL_LAUNCH_CHECK();
    return 0;
  }
  if (dtype == HAL_F32)
    hipLaunchKernelGGL(latent_prep_kernel<float>, dim3(n_tokens), dim3(256), 0, stream, a, lda, q_col0,
                       q_rank, kv_col0, kv_rank, rot, D, wq, wkv, w_dtype, eps, (float*)cq, (float*)qkv,
                       row_stride, k_col0);
  else
    hipLaunchKernelGGL(latent_prep_kernel<bf16_t>, dim3(n_tokens), dim3(256), 0, stream, a, lda, q_col0,
                       q_rank, kv_col0, kv_rank, rot, D, wq, wkv, w_dtype, eps, (bf16_t*)cq,
                       (bf16_t*)qkv, row_stride, k_col0);
  HAL_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------------
// y[t, h * ys + y0 + j] = x[t, h * xs + x0 + j] for j < n, and zero for the `n_zero` columns
// from h * ys + z0 on
// ---------------------------------------------------------------------------------
// (V: what is copied at once, a number or, where all sizes, columns and addresses allow it, 16 bytes: 3,000 tokens of 32
// heads of 64 bf16 11.5 -> 6.4 us; the arguments count in V)
template <typename V>
__global__ void head_cols_kernel(const V* __restrict__ x, int ldx, int xs, int x0, V* __restrict__ y,
                                 int ldy, int ys, int y0, int n, int z0, int n_zero, int H) {
  const int t = blockIdx.x;
  const int per = n + n_zero;
  for (int e = threadIdx.x; e < H * per; e += blockDim.x) {
    const int h = e / per, j = e % per;
    if (j < n) y[(size_t)t * ldy + h * ys + y0 + j] = x[(size_t)t * ldx + h * xs + x0 + j];
    else y[(size_t)t * ldy + h * ys + z0 + (j - n)] = V{};
  }
}

extern "C" int hal_head_cols(const void* x, int ldx, int xs, int x0, void* y, int ldy, int ys, int y0,
                             int n, int z0, int n_zero, int H, int dtype, int n_tokens,
                             hipStream_t stream) {
  HAL_REQUIRE(n_tokens >= 0 && H > 0 && n >= 0 && n_zero >= 0, "hal_head_cols: bad sizes");
  HAL_REQUIRE(x0 >= 0 && x0 + n <= xs && H * xs <= ldx && y0 >= 0 && y0 + n <= ys && z0 >= 0 &&
                  z0 + n_zero <= ys && H * ys <= ldy,
              "hal_head_cols: columns outside the rows");
  HAL_REQUIRE(dtype == HAL_F32 || dtype == HAL_BF16, "hal_head_cols: dtype %d", dtype);
  if (n_tokens == 0 || n + n_zero == 0) return 0;
  const int v = dtype == HAL_F32 ? 4 : 8;  // numbers of 16 bytes
  if (!((ldx | xs | x0 | ldy | ys | y0 | n | z0 | n_zero) % v) && ((uintptr_t)x | (uintptr_t)y) % 16 == 0)
    hipLaunchKernelGGL(head_cols_kernel<uint4>, dim3(n_tokens), dim3(256), 0, stream, (const uint4*)x, ldx / v, xs / v, x0 / v,
                       (uint4*)y, ldy / v, ys / v, y0 / v, n / v, z0 / v, n_zero / v, H);
  else if (dtype == HAL_F32)
    hipLaunchKernelGGL(head_cols_kernel<uint32_t>, dim3(n_tokens), dim3(256), 0, stream, (const uint32_t*)x, ldx,
                       xs, x0, (uint32_t*)y, ldy, ys, y0, n, z0, n_zero, H);
  else
    hipLaunchKernelGGL(head_cols_kernel<uint16_t>, dim3(n_tokens), dim3(256), 0, stream, (const uint16_t*)x,
                       ldx, xs, x0, (uint16_t*)y, ldy, ys, y0, n, z0, n_zero, H);
  HAL_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------------
// x[i] *= s
// ---------------------------------------------------------------------------------
__global__ void scale_f32_kernel(float* __restrict__ x, size_t n, float s) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] *= s;
}

extern "C" int hal_scale_f32(float* x, long long n, float s, hipStream_t stream) {
  HAL_REQUIRE(n >= 0, "hal_scale_f32: n=%lld", n);
  if (n == 0) return 0;
  hipLaunchKernelGGL(scale_f32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, x, (size_t)n, s);
  HAL_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------------
#define MOE_MAX_EXPERTS 1024
// Router: z [T, E] float32 logits.  score = sigmoid(z) (or, softmax == 1, the softmax over
// the experts); the `top` largest scores (the lower index wins a tie); weights = the chosen
// scores, divided by their sum + norm_eps if `normalize`, times `scale`.  `correction` (or null)
// [E]: added to the scores for the choice alone.  `groups` > 0: the experts form so many equal
// groups of neighbours, and only experts of the `keep` groups with the largest sums of their two
// largest (corrected) scores are chosen from (the lower group wins a tie).
//
// One wave a token: lane l holds the scores of the experts l, l + 64, ... in W words (W is the
// build for so many experts: the code of a step that runs once is mostly fetched, so it is kept
// short).  A score is shown to all lanes by reading it from its lane at a uniform index.
// ---------------------------------------------------------------------------------
struct MoeChoice {
  int softmax, normalize;
  float norm_eps, scale;
  const void* correction;
  int c_dtype, groups, keep;
};
__device__ __forceinline__ float lane_value(float v, int lane) {
  return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane));
}
// how many of the first n numbers (lane l of word w holds number w * 64 + l) come before lane's own
// ones: larger, or equal and of a lower index
template <int W>
__device__ __forceinline__ void places_before(const float (&v)[W], int n, int lane, int (&before)[W]) {
#pragma unroll
  for (int u = 0; u < W; ++u) before[u] = 0;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const int m = n - w * HAL_WAVE < HAL_WAVE ? n - w * HAL_WAVE : HAL_WAVE;
    for (int l = 0; l < m; ++l) {
      const float x = lane_value(v[w], l);
#pragma unroll
      for (int u = 0; u < W; ++u)
        before[u] += (x > v[u] || (x == v[u] && w * HAL_WAVE + l < u * HAL_WAVE + lane)) ? 1 : 0;
    }
  }
}

// The scores of experts outside the best groups become -infinity.  Lane g (word g / 64) holds what
// belongs to group g.
template <int W>
__device__ __forceinline__ void moe_close_groups(float (&s)[W], int E, int groups, int keep, int lane) {
  const int per = E / groups;
  float first[W], second[W];  // a group's two largest
#pragma unroll
  for (int u = 0; u < W; ++u) first[u] = second[u] = -INFINITY;
  int g = 0, in_group = 0;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const int m = E - w * HAL_WAVE < HAL_WAVE ? E - w * HAL_WAVE : HAL_WAVE;
    for (int l = 0; l < m; ++l) {
      const float x = lane_value(s[w], l);
#pragma unroll
      for (int u = 0; u < W; ++u)
        if (lane + u * HAL_WAVE == g) second[u] = fmaxf(second[u], fminf(first[u], x)), first[u] = fmaxf(first[u], x);
      if (++in_group == per) in_group = 0, ++g;
    }
  }
  if (per > 1) {
#pragma unroll
    for (int u = 0; u < W; ++u) first[u] += second[u];
  }
  int before[W];
  places_before<W>(first, groups, lane, before);
#pragma unroll
  for (int u = 0; u < W; ++u) {
    const int e = lane + u * HAL_WAVE, mine = e < E ? e / per : 0;
    int place = 0;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const int got = __shfl(before[w], mine % HAL_WAVE, HAL_WAVE);
      if (w == mine / HAL_WAVE) place = got;
    }
    if (place >= keep) s[u] = -INFINITY;
  }
}

// ---------------------------------------------------------------------------------
// Z[p] = X W^T over the p-th part of K, for a bf16 W [N, K] of few rows (a router's): float32 planes [parts][M][N], which
// whoever reads the logits adds up in order.
//
// What bounds it: a matrix of 64 columns is four tiles of an instruction, so that a whole product of few rows has four workgroups, each
// of which waits for its K numbers a row alone.  In parts of K, four waves a part whose sums meet in LDS, one tile of columns a
// workgroup: 8 rows, 64 x 4,096: 7.7 -> 2.9 us (the small-batch product before); 48 rows, 16 x 4,096: 6.0 -> 4.3 (the library).
// Both operands come straight from memory in the instruction's order, four steps of 32 k at a time.
// ---------------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(8))) __bf16 nw_bf16x8;
typedef __attribute__((ext_vector_type(4))) float nw_f32x4;
#define NW_WAVES 4
template <int MT>  // tiles of 16 rows
__global__ void __launch_bounds__(NW_WAVES * HAL_WAVE)
narrow_product_kernel(const bf16_t* __restrict__ X, int ldx, const bf16_t* __restrict__ W, int ldw, float* __restrict__ Z, int M, int N, int K) {
  constexpr int U = 4;  // steps of 32 k at a time
  __shared__ __attribute__((aligned(16))) float sums[NW_WAVES][MT][256];
  const int lane = threadIdx.x % HAL_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / HAL_WAVE);
  const int n0 = blockIdx.x * 16, part = blockIdx.y, parts = gridDim.y;
  const int r = lane % 16, q = lane / 16, all = K / 32, shares = parts * NW_WAVES, mine = part * NW_WAVES + wave;
  const int begin = (int)((long long)all * mine / shares), end = (int)((long long)all * (mine + 1) / shares);
  // (rows and columns past the end are read from the last one: nothing of them is stored)
  const bf16_t* x[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) x[i] = X + (size_t)min(i * 16 + r, M - 1) * ldx + q * 8;
  const bf16_t* w = W + (size_t)min(n0 + r, N - 1) * ldw + q * 8;
  nw_f32x4 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i] = nw_f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s = begin; s < end; s += U) {
    nw_bf16x8 a[U][MT], b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(s + u, end - 1) * 32;  // (past the share's end the last step's numbers come again and are not multiplied)
#pragma unroll
      for (int i = 0; i < MT; ++i) a[u][i] = *(const nw_bf16x8*)(x[i] + k);
      b[u] = *(const nw_bf16x8*)(w + k);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (s + u >= end) break;
#pragma unroll
      for (int i = 0; i < MT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[u], a[u][i], acc[i], 0, 0, 0);
    }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) *(nw_f32x4*)&sums[wave][i][lane * 4] = acc[i];
  __syncthreads();
  // lane l of a tile's result holds row l % 16 and columns 4 (l / 16) .. + 3; wave v adds up tile v
  if (wave >= MT) return;
  nw_f32x4 sum = *(const nw_f32x4*)&sums[0][wave][lane * 4];
#pragma unroll
  for (int v = 1; v < NW_WAVES; ++v) sum += *(const nw_f32x4*)&sums[v][wave][lane * 4];
  const int m = wave * 16 + r, n = n0 + q * 4;
  if (m >= M) return;
  float* to = Z + ((size_t)part * M + m) * N + n;
  if (N % 4 == 0 && n < N) {
    *(nw_f32x4*)to = sum;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) to[e] = sum[e];
  }
}

// Into how many parts K is cut; 0: the product is not taken.  Up to 64 rows (8 rows, 64 x 4,096: 7.7 us as one product, 2.9 in
// parts; 64 rows: 6.2 and 4.5); at 65 rows and more the tiles of 64 columns that read X once take 10.6 us against the library's 6.2,
// and no number of rows up to 8,192 turned that.  Past 256 columns (256 x 2,048, 64 rows: 5.3 and 3.6, of which the reader
// of eight planes gives 1.1 back) the whole product has workgroups enough.
#define NW_MAX_ROWS 64
#define NW_MAX_COLS 256
extern "C" int hal_narrow_product_parts(const void* X, int ldx, const void* W, int ldw, int M, int N, int K) {
  if (M <= 0 || M > NW_MAX_ROWS || N <= 0 || N > NW_MAX_COLS || K % 32 || K < 512) return 0;
  if (ldx % 8 || ldw % 8 || (uintptr_t)X % 16 || (uintptr_t)W % 16) return 0;
  return K >= 2048 ? 8 : K / 256;  // (at least two steps of 32 k a wave)
}

extern "C" int hal_narrow_product(const void* X, int ldx, const void* W, int ldw, float* Z, int parts, int M, int N, int K, hipStream_t stream) {
  HAL_REQUIRE(parts > 0 && parts == hal_narrow_product_parts(X, ldx, W, ldw, M, N, K), "hal_narrow_product: M=%d N=%d K=%d in %d parts", M, N, K, parts);
  HAL_REQUIRE(ldx >= K && ldw >= K && (uintptr_t)Z % 16 == 0, "hal_narrow_product: rows of %d and %d, or the planes' place", ldx, ldw);
  const dim3 grid((N + 15) / 16, parts), block(NW_WAVES * HAL_WAVE);
#define NW_LAUNCH(MT_) \
  hipLaunchKernelGGL((narrow_product_kernel<MT_>), grid, block, 0, stream, (const bf16_t*)X, ldx, (const bf16_t*)W, ldw, Z, M, N, K)
  if (M <= 16) NW_LAUNCH(1);
  else if (M <= 32) NW_LAUNCH(2);
  else NW_LAUNCH(4);
#undef NW_LAUNCH
  HAL_LAUNCH_CHECK();
  return 0;
}

// a router's logits: rows of `ld`, in planes that are added up
#define MOE_MAX_PLANES 8
struct MoeLogits {
  const float* at;
  int ld, planes;
  long long plane;
};
template <int W>
__device__ __forceinline__ void moe_route_token(const MoeLogits& z, int E, int top, const MoeChoice& how,
                                                int* __restrict__ idx, float* __restrict__ wgt, int t, int lane) {
  const float* zr = z.at + (size_t)t * z.ld;
  float s[W], w[W];  // what the choice is made by, and the scores as weights
  float zmax = -INFINITY;
#pragma unroll
  for (int u = 0; u < W; ++u) {
    const int e = lane + u * HAL_WAVE;
    s[u] = -INFINITY;
    if (e < E) {
      float part[MOE_MAX_PLANES];  // (all asked for before they are added up)
#pragma unroll
      for (int p = 0; p < MOE_MAX_PLANES; ++p) part[p] = p < z.planes ? zr[(size_t)p * z.plane + e] : 0.f;
      s[u] = part[0];
#pragma unroll
      for (int p = 1; p < MOE_MAX_PLANES; ++p)
        if (p < z.planes) s[u] += part[p];
    }
    zmax = fmaxf(zmax, s[u]);
  }
  if (how.softmax) {
    zmax = wave_max(zmax);
    float part = 0.f;
#pragma unroll
    for (int u = 0; u < W; ++u) {
      w[u] = expf(s[u] - zmax);  // (0 beyond the experts)
      part += w[u];
    }
    const float denom = wave_sum(part);
#pragma unroll
    for (int u = 0; u < W; ++u) w[u] = w[u] / denom;
  } else {
#pragma unroll
    for (int u = 0; u < W; ++u) w[u] = 1.0f / (1.0f + expf(-s[u]));
  }
#pragma unroll
  for (int u = 0; u < W; ++u) {
    const int e = lane + u * HAL_WAVE;
    s[u] = w[u];
    if (how.correction && e < E) s[u] += load_as_f32(how.correction, how.c_dtype, e);
    if (e >= E || s[u] != s[u]) s[u] = -INFINITY;  // (a choice among numbers that are none is some choice)
  }
  if (how.groups > 0) moe_close_groups<W>(s, E, how.groups, how.keep, lane);
  if constexpr (W <= 2) {  // few experts: every expert's place among all
    int place[W];
    places_before<W>(s, E, lane, place);
    float part = 0.f;
#pragma unroll
    for (int u = 0; u < W; ++u) part += (lane + u * HAL_WAVE < E && place[u] < top) ? w[u] : 0.f;
    const float sum = wave_sum(part) + how.norm_eps;
#pragma unroll
    for (int u = 0; u < W; ++u) {
      if (lane + u * HAL_WAVE >= E || place[u] >= top) continue;
      idx[(size_t)t * top + place[u]] = lane + u * HAL_WAVE;
      wgt[(size_t)t * top + place[u]] = (how.normalize ? w[u] / sum : w[u]) * how.scale;
    }
  } else {  // each of the `top` rounds finds the largest that is left across the wave
    float sum = 0.f, mine[W];
    int place[W];
#pragma unroll
    for (int u = 0; u < W; ++u) place[u] = -1;
    for (int j = 0; j < top; ++j) {
      float best = -INFINITY;
      int best_e = MOE_MAX_EXPERTS;
#pragma unroll
      for (int u = 0; u < W; ++u)  // rising index: the lower one stays on a tie
        if (lane + u * HAL_WAVE < E && place[u] < 0 && (s[u] > best || best_e == MOE_MAX_EXPERTS)) best = s[u], best_e = lane + u * HAL_WAVE;
#pragma unroll
      for (int off = HAL_WAVE / 2; off > 0; off >>= 1) {
        const float ob = __shfl_xor(best, off, HAL_WAVE);
        const int oe = __shfl_xor(best_e, off, HAL_WAVE);
        if (oe < MOE_MAX_EXPERTS && (best_e == MOE_MAX_EXPERTS || ob > best || (ob == best && oe < best_e))) best = ob, best_e = oe;
      }
      float own = 0.f;
#pragma unroll
      for (int u = 0; u < W; ++u)
        if (lane + u * HAL_WAVE == best_e) place[u] = j, own = w[u];  // taken
      sum += lane_value(own, __builtin_amdgcn_readfirstlane(best_e % HAL_WAVE));
    }
    sum += how.norm_eps;
#pragma unroll
    for (int u = 0; u < W; ++u) {
      mine[u] = (how.normalize ? w[u] / sum : w[u]) * how.scale;
      if (place[u] < 0) continue;
      idx[(size_t)t * top + place[u]] = lane + u * HAL_WAVE;
      wgt[(size_t)t * top + place[u]] = mine[u];
    }
  }
}

template <int W>
__global__ void __launch_bounds__(HAL_WAVE) moe_route_kernel(MoeLogits z, int E, int top, MoeChoice how,
                                                             int* __restrict__ idx, float* __restrict__ wgt, int n_tokens) {
  moe_route_token<W>(z, E, top, how, idx, wgt, blockIdx.x, threadIdx.x);
}

static int moe_check_choice(const MoeChoice& how, int E, int top) {
  HAL_REQUIRE(how.c_dtype == HAL_F32 || how.c_dtype == HAL_BF16, "router: a correction of type %d", how.c_dtype);
  HAL_REQUIRE(how.groups >= 0 && (how.groups == 0 || (E % how.groups == 0 && how.keep > 0 && how.keep <= how.groups &&
                                                      top <= E / how.groups * how.keep)),
              "router: %d of %d experts in %d groups of which %d are kept", top, E, how.groups, how.keep);
  return 0;
}

#define MOE_BY_WORDS(LAUNCH_, MOST_)               \
  do {                                             \
    if (E <= HAL_WAVE) LAUNCH_(1);                 \
    else if (E <= 2 * HAL_WAVE) LAUNCH_(2);        \
    else if (E <= 4 * HAL_WAVE) LAUNCH_(4);        \
    else if (MOST_ > 4) LAUNCH_(MOST_);            \
  } while (0)

extern "C" int hal_moe_route(const float* z, int ldz, int planes, long long plane, int E, int top, int softmax, int normalize, float norm_eps,
                             float scale, const void* correction, int c_dtype, int groups, int keep, int* idx,
                             float* wgt, int n_tokens, hipStream_t stream) {
  const MoeChoice how = {softmax, normalize, norm_eps, scale, correction, c_dtype, groups, keep};
  HAL_REQUIRE(planes >= 1 && planes <= MOE_MAX_PLANES, "router: logits in %d planes", planes);
  const MoeLogits logits = {z, ldz, planes, plane};
  HAL_REQUIRE(n_tokens >= 0 && E > 0 && E <= MOE_MAX_EXPERTS && top > 0 && top <= E && ldz >= E,
              "hal_moe_route: bad sizes T=%d E=%d top=%d", n_tokens, E, top);
  if (int rc = moe_check_choice(how, E, top)) return rc;
  if (n_tokens == 0) return 0;
#define MOE_ROUTE(W_) \
  hipLaunchKernelGGL(moe_route_kernel<W_>, dim3(n_tokens), dim3(HAL_WAVE), 0, stream, logits, E, top, how, idx, wgt, n_tokens)
  MOE_BY_WORDS(MOE_ROUTE, 16);
#undef MOE_ROUTE
  HAL_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------------
// Counting sort of the n = T * top pairs by expert, one workgroup.  offsets [E + 1]: where
// each expert's pairs begin in `sorted`; tile_offsets [E + 1]: the same counted in tiles of
// `tile` rows, each expert's count rounded up; sorted [n]: pair numbers (token * top +
// choice), expert by expert.  The order inside an expert is not fixed; nothing that is
// computed from it depends on it.
// ---------------------------------------------------------------------------------
// (idx without __restrict__: the kernel that routes and sorts in one has just written it)
__device__ __forceinline__ void moe_sort_pairs(const int* idx, int n, int E, int tile,
                                               int* __restrict__ offsets, int* __restrict__ tile_offsets,
                                               int* __restrict__ sorted, int* count, int* cursor) {
  for (int e = threadIdx.x; e < E; e += blockDim.x) count[e] = 0;
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int e = idx[i];
    if (e >= 0 && e < E) atomicAdd(&count[e], 1);
  }
  __syncthreads();
  if (threadIdx.x < HAL_WAVE) {  // the first wave: running sums, 64 experts at a time
    const int lane = threadIdx.x;
    int at = 0, tiles = 0;
    for (int e0 = 0; e0 < E; e0 += HAL_WAVE) {
      const int e = e0 + lane, c = e < E ? count[e] : 0, ct = (c + tile - 1) / tile;
      int sum = c, sum_t = ct;
#pragma unroll
      for (int off = 1; off < HAL_WAVE; off <<= 1) {
        const int a = __shfl_up(sum, off, HAL_WAVE), b = __shfl_up(sum_t, off, HAL_WAVE);
        if (lane >= off) sum += a, sum_t += b;
      }
      if (e < E) {
        offsets[e] = cursor[e] = at + sum - c;
        tile_offsets[e] = tiles + sum_t - ct;
      }
      at += __shfl(sum, HAL_WAVE - 1, HAL_WAVE);
      tiles += __shfl(sum_t, HAL_WAVE - 1, HAL_WAVE);
    }
    if (lane == 0) {
      offsets[E] = at;
      tile_offsets[E] = tiles;
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    const int e = idx[i];
    if (e >= 0 && e < E) sorted[atomicAdd(&cursor[e], 1)] = i;
  }
}

__global__ void __launch_bounds__(1024) moe_sort_kernel(const int* __restrict__ idx, int n, int E, int tile,
                                                        int* __restrict__ offsets,
                                                        int* __restrict__ tile_offsets,
                                                        int* __restrict__ sorted) {
  __shared__ int count[MOE_MAX_EXPERTS];
  __shared__ int cursor[MOE_MAX_EXPERTS];
  moe_sort_pairs(idx, n, E, tile, offsets, tile_offsets, sorted, count, cursor);
}

// Both in one workgroup, for steps of few tokens and up to 256 experts: its waves take the tokens in
// turn, then all of it sorts the pairs.
template <int W>
__global__ void __launch_bounds__(1024) moe_route_sort_kernel(MoeLogits z, int E, int top, MoeChoice how, int* __restrict__ idx,
                                                              float* __restrict__ wgt, int n_tokens, int tile,
                                                              int* __restrict__ offsets, int* __restrict__ tile_offsets,
                                                              int* __restrict__ sorted) {
  __shared__ int count[MOE_MAX_EXPERTS];
  __shared__ int cursor[MOE_MAX_EXPERTS];
  const int wave = threadIdx.x / HAL_WAVE, lane = threadIdx.x % HAL_WAVE;
  for (int t = wave; t < n_tokens; t += blockDim.x / HAL_WAVE)
    moe_route_token<W>(z, E, top, how, idx, wgt, t, lane);
  __threadfence_block();
  __syncthreads();
  moe_sort_pairs(idx, n_tokens * top, E, tile, offsets, tile_offsets, sorted, count, cursor);
}

extern "C" int hal_moe_route_sort(const float* z, int ldz, int planes, long long plane, int E, int top, int softmax, int normalize, float norm_eps,
                                  float scale, const void* correction, int c_dtype, int groups, int keep,
                                  int* idx, float* wgt, int n_tokens, int tile, int* offsets, int* tile_offsets,
                                  int* sorted, hipStream_t stream) {
  const MoeChoice how = {softmax, normalize, norm_eps, scale, correction, c_dtype, groups, keep};
  HAL_REQUIRE(planes >= 1 && planes <= MOE_MAX_PLANES, "router: logits in %d planes", planes);
  const MoeLogits logits = {z, ldz, planes, plane};
  HAL_REQUIRE(n_tokens >= 0 && E > 0 && E <= 4 * HAL_WAVE && top > 0 && top <= E && ldz >= E && tile > 0,
              "hal_moe_route_sort: bad sizes T=%d E=%d top=%d", n_tokens, E, top);
  if (int rc = moe_check_choice(how, E, top)) return rc;
  int waves = n_tokens < 4 ? 4 : (n_tokens < 16 ? n_tokens : 16);
#define MOE_ROUTE_SORT(W_)                                                                                                    \
  hipLaunchKernelGGL(moe_route_sort_kernel<W_>, dim3(1), dim3(waves * HAL_WAVE), 0, stream, logits, E, top, how, idx, wgt,    \
                     n_tokens, tile, offsets, tile_offsets, sorted)
  MOE_BY_WORDS(MOE_ROUTE_SORT, 4);
#undef MOE_ROUTE_SORT
  HAL_LAUNCH_CHECK();
  return 0;
}

extern "C" int hal_moe_sort(const int* idx, int n, int E, int tile, int* offsets, int* tile_offsets,
                            int* sorted, hipStream_t stream) {
  HAL_REQUIRE(n >= 0 && E > 0 && E <= MOE_MAX_EXPERTS && tile > 0, "hal_moe_sort: bad sizes n=%d E=%d", n, E);
  hipLaunchKernelGGL(moe_sort_kernel, dim3(1), dim3(1024), 0, stream, idx, n, E, tile, offsets,
                     tile_offsets, sorted);
  HAL_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------------
// h[t, :] += sum_j wgt[t, j] * y[t * top + j, :] (+ extra[t, :])   (y float32 [T * top, d])
// ---------------------------------------------------------------------------------
__global__ void moe_combine_kernel(float* __restrict__ h, const float* __restrict__ y,
                                   const float* __restrict__ wgt, const float* __restrict__ extra,
                                   const float* __restrict__ extra_gate, int ld_gate, int top, int d, bool overwrite) {
  const int t = blockIdx.x;
  const float eg = extra_gate ? 1.0f / (1.0f + expf(-extra_gate[(size_t)t * ld_gate])) : 1.0f;
  // (a step of few tokens spreads a row over several workgroups: blockIdx.y takes every gridDim.y-th run of columns)
  for (int i = blockIdx.y * blockDim.x + threadIdx.x; i < d; i += blockDim.x * gridDim.y) {
    float s = extra ? eg * extra[(size_t)t * d + i] : 0.f;
    for (int j = 0; j < top; ++j) s += wgt[(size_t)t * top + j] * y[((size_t)t * top + j) * d + i];
    h[(size_t)t * d + i] = overwrite ? s : h[(size_t)t * d + i] + s;
  }
}

// The same four columns a thread, the rows of up to four experts in flight together (the sum's order is
// the same).  Bound by memory: 3,000 tokens of 6 experts, width 4096, with an extra row, 442 MB: 86 us
// (5.1 TB/s), 147 us with a column a thread, which waits for an expert's row before it asks for the
// next; 2,250 tokens of 4 experts without one: 32 us, 69 us.
__global__ void __launch_bounds__(256)
moe_combine_vec_kernel(float* __restrict__ h, const float* __restrict__ y, const float* __restrict__ wgt,
                       const float* __restrict__ extra, const float* __restrict__ extra_gate, int ld_gate, int top,
                       int d, bool overwrite) {
  const int t = blockIdx.x;
  const int i = (blockIdx.y * blockDim.x + threadIdx.x) * 4;
  if (i >= d) return;
  const float* w = wgt + (size_t)t * top;
  const float* rows = y + (size_t)t * top * d + i;
  float* out = h + (size_t)t * d + i;
  float4 before = make_float4(0.f, 0.f, 0.f, 0.f), e = before;
  if (!overwrite) before = *(const float4*)out;
  if (extra) e = *(const float4*)(extra + (size_t)t * d + i);
  const float eg = extra_gate ? 1.0f / (1.0f + expf(-extra_gate[(size_t)t * ld_gate])) : 1.0f;
  float s[4] = {eg * e.x, eg * e.y, eg * e.z, eg * e.w};
  for (int j0 = 0; j0 < top; j0 += 4) {
    float4 v[4];
    float c[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = j0 + u < top ? j0 + u : j0;  // (past the end: a row that is there, not added)
      v[u] = *(const float4*)(rows + (size_t)j * d);
      c[u] = w[j];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (j0 + u >= top) break;
      s[0] += c[u] * v[u].x, s[1] += c[u] * v[u].y, s[2] += c[u] * v[u].z, s[3] += c[u] * v[u].w;
    }
  }
  *(float4*)out = overwrite ? make_float4(s[0], s[1], s[2], s[3])
                            : make_float4(before.x + s[0], before.y + s[1], before.z + s[2], before.w + s[3]);
}

extern "C" int hal_moe_combine(float* h, const float* y, const float* wgt, const float* extra,
                               const float* extra_gate, int ld_gate, int top, int d, int n_tokens,
                               int overwrite, hipStream_t stream) {
  HAL_REQUIRE(n_tokens >= 0 && top > 0 && d > 0, "hal_moe_combine: bad sizes");
  if (n_tokens == 0) return 0;
  // many rows of whole 16-byte pieces: four columns a thread (for few rows the launch is what
  // counts: 4.8 us either way at 8 rows)
  if (n_tokens >= 64 && d % 4 == 0 && ((uintptr_t)h | (uintptr_t)y | (uintptr_t)extra) % 16 == 0) {
    const int quads = d / 4, block = quads >= 256 ? 256 : (quads + 63) / 64 * 64;
    hipLaunchKernelGGL(moe_combine_vec_kernel, dim3(n_tokens, (quads + block - 1) / block), dim3(block), 0, stream, h, y,
                       wgt, extra, extra_gate, ld_gate, top, d, overwrite != 0);
    HAL_LAUNCH_CHECK();
    return 0;
  }
  int threads = (d + 63) / 64 * 64;
  if (threads > 256) threads = 256;
  int parts = 1;  // workgroups a row, so that a decode step has a few hundred of them
  while (parts < 16 && n_tokens * parts < 256 && d / (threads * parts * 2) >= 1) parts *= 2;
  hipLaunchKernelGGL(moe_combine_kernel, dim3(n_tokens, parts), dim3(threads), 0, stream, h, y, wgt, extra, extra_gate, ld_gate, top, d, overwrite != 0);
  HAL_LAUNCH_CHECK();
  return 0;
}
