// The sampler: one block per row of float32 logits.
//   greedy (temperature 0 or top_k 1): first index of the maximum, and its
//     log-probability under softmax(logits);
//   otherwise z = logits / temperature, p = softmax(z), the reference's filters
//     (top-k, top-p, min-p), and the first token, in index order, whose cumulative
//     kept probability exceeds u * (kept mass).  u comes from a counter-based
//     generator keyed by (seed, draw index) of the row's request, so a request's
//     tokens do not depend on what else is in the batch.  The log-probability is
//     that of the temperature-scaled distribution before filtering.
// NaN logits count as -1e5.  src/halite/transformers/infer/engine/sampler.py:17-60
#include "hal_common.h"
#include "hal_api.h"
#include <mutex>
#include <string.h>

#define SAMPLE_THREADS 1024
#define SAMPLE_BINS 2048  // two per thread

__device__ __forceinline__ float clean_logit(float x) { return x != x ? -1e5f : x; }

// order-preserving map of a float to an unsigned key
__device__ __forceinline__ uint32_t sort_key(float x) {
  const uint32_t u = __float_as_uint(x);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// the float that a key stands for
__device__ __forceinline__ float key_value(uint32_t key) {
  return __uint_as_float((key & 0x80000000u) ? (key & 0x7fffffffu) : ~key);
}

__device__ __forceinline__ float uniform_draw(uint64_t seed, uint32_t index) {
  uint64_t x = seed * 0x9E3779B97F4A7C15ull + ((uint64_t)index + 1ull) * 0xD1B54A32D192ED03ull;
  x ^= x >> 30;
  x *= 0xBF58476D1CE4E5B9ull;
  x ^= x >> 27;
  x *= 0x94D049BB133111EBull;
  x ^= x >> 31;
  return (float)(x >> 40) * (1.0f / 16777216.0f);
}

// Sum of `v` over the threads after this one (exclusive), for a block of SAMPLE_THREADS
// threads; `tmp` holds one entry per wave.  Ends with a barrier, so `tmp` can be used
// again at once.
__device__ __forceinline__ unsigned long long block_suffix_u64(unsigned long long v,
                                                               unsigned long long* tmp) {
  const int lane = threadIdx.x % HAL_WAVE, wave = threadIdx.x / HAL_WAVE;
  unsigned long long inc = v;
#pragma unroll
  for (int off = 1; off < HAL_WAVE; off <<= 1) {
    const uint32_t lo = __shfl_down((uint32_t)inc, off, HAL_WAVE);
    const uint32_t hi = __shfl_down((uint32_t)(inc >> 32), off, HAL_WAVE);
    if (lane + off < HAL_WAVE) inc += ((unsigned long long)hi << 32) | lo;
  }
  if (lane == 0) tmp[wave] = inc;
  __syncthreads();
  unsigned long long after = 0ull;
  for (int w = wave + 1; w < SAMPLE_THREADS / HAL_WAVE; ++w) after += tmp[w];
  __syncthreads();
  return inc - v + after;
}

struct ArgMax {
  float v;
  int i;
};

__device__ __forceinline__ ArgMax argmax_merge(ArgMax a, ArgMax b) {
  if (b.v > a.v || (b.v == a.v && b.i < a.i)) return b;
  return a;
}

__global__ void __launch_bounds__(SAMPLE_THREADS)
sample_kernel(const float* __restrict__ logits, int ld, int V,
              const float* __restrict__ temperature, const int* __restrict__ top_k,
              const float* __restrict__ top_p, const float* __restrict__ min_p,
              const uint64_t* __restrict__ seeds, const int* __restrict__ draw_index,
              int* __restrict__ out_token, float* __restrict__ out_logprob,
              uint32_t* __restrict__ key_rows) {
  __shared__ float red[16];
  __shared__ float red2[16];
  __shared__ ArgMax amax_s[16];
  __shared__ int chosen_thread;
  __shared__ int last_thread;
  __shared__ unsigned long long hist[2][SAMPLE_BINS];
  __shared__ unsigned long long scan_tmp[SAMPLE_THREADS / HAL_WAVE];
  __shared__ unsigned long long whole_mass;
  __shared__ unsigned long long found_above[2];
  __shared__ uint32_t found_bin[2];
  __shared__ int found_any[2];

  const int row = blockIdx.x, tid = threadIdx.x;
  const int lane = tid % HAL_WAVE, wave = tid / HAL_WAVE;
  const float* x = logits + (size_t)row * ld;
  const float T = temperature[row];
  const int k = top_k[row];
  const bool greedy = (T == 0.f) || (k == 1);
  const float inv_scale = greedy ? 1.f : T;

  // ---- one pass: maximum (with its first index) and sum of exp(z - max), z = x / T ----
  // Each thread keeps a running maximum and a sum relative to it (the online form of
  // softmax's denominator); four logits per load where the row allows it.
  ArgMax am = {-INFINITY, 0x7fffffff};
  float part = 0.f;
  // the keys of the row (order-preserving integers of z) are kept for the later passes
  uint32_t* keys = (key_rows && !greedy) ? key_rows + (size_t)row * V : nullptr;
  auto key_of = [&](float xv) { return sort_key(clean_logit(xv) / inv_scale); };
  auto take = [&](float xv, int i) {
    const float z = clean_logit(xv) / inv_scale;
    if (z > am.v) {
      part = part * expf(am.v - z) + 1.f;  // am.v = -inf gives part * 0
      am.v = z;
      am.i = i;
    } else if (z != -INFINITY) {  // (-inf adds nothing; with am.v still -inf it would add NaN)
      part += expf(z - am.v);
    }
  };
  if (ld % 4 == 0 && ((uintptr_t)logits % 16) == 0) {
    const int n4 = V / 4;
    const bool keys4 = keys && V % 4 == 0;  // rows of keys start on 16 bytes then
#pragma unroll 4
    for (int v = tid; v < n4; v += SAMPLE_THREADS) {
      const float4 q = *(const float4*)(x + 4 * v);
      take(q.x, 4 * v), take(q.y, 4 * v + 1), take(q.z, 4 * v + 2), take(q.w, 4 * v + 3);
      if (keys4)
        *(uint4*)(keys + 4 * v) = make_uint4(key_of(q.x), key_of(q.y), key_of(q.z), key_of(q.w));
      else if (keys)
        keys[4 * v] = key_of(q.x), keys[4 * v + 1] = key_of(q.y), keys[4 * v + 2] = key_of(q.z),
                 keys[4 * v + 3] = key_of(q.w);
    }
    for (int i = 4 * n4 + tid; i < V; i += SAMPLE_THREADS) {
      take(x[i], i);
      if (keys) keys[i] = key_of(x[i]);
    }
  } else {
    for (int i = tid; i < V; i += SAMPLE_THREADS) {
      take(x[i], i);
      if (keys) keys[i] = key_of(x[i]);
    }
  }
  // combine the threads: the block's maximum, then the sums rescaled to it
  ArgMax mine_am = am;
#pragma unroll
  for (int off = HAL_WAVE / 2; off > 0; off >>= 1) {
    ArgMax o;
    o.v = __shfl_xor(am.v, off, HAL_WAVE);
    o.i = __shfl_xor(am.i, off, HAL_WAVE);
    am = argmax_merge(am, o);
  }
  if (lane == 0) amax_s[wave] = am;
  __syncthreads();
  am = amax_s[0];
  for (int w = 1; w < SAMPLE_THREADS / HAL_WAVE; ++w) am = argmax_merge(am, amax_s[w]);
  const float m = am.v;
  part = (mine_am.v == -INFINITY) ? 0.f : part * expf(mine_am.v - m);
  const float total = block_sum(part, red);

  if (greedy) {
    if (tid == 0) {
      out_token[row] = am.i < V ? am.i : 0;  // (a row of nothing but -inf has no maximum)
      out_logprob[row] = -logf(total);  // z_max - m - log(total)
    }
    return;
  }

  // ---- filters: the kept set is { key(z_i) >= key_min } and exp(z_i - m) >= min_p --
  // Both thresholds are the key at which a sum over the tokens in descending order of
  // their keys first reaches a target: the number of tokens reaches k (top-k), the mass
  // reaches top_p of the reference mass (top-p).  That key is found digit by digit
  // (11 + 11 + 10 bits) from histograms over the tokens that share the digits found so
  // far: three passes over the row instead of one per bit.  Masses are summed as
  // integers (2^-40 of the largest token's), so the sums do not depend on their order.
  auto key_at = [&](int i) { return keys ? keys[i] : sort_key(clean_logit(x[i]) / inv_scale); };
  const float tp = top_p[row];
  const float mp = min_p[row];
  const bool want_k = k > 0 && k < V, want_p = tp < 1.f;
  uint32_t key_min = 0;
  if (want_k || want_p) {
    auto fixed = [&](uint32_t key) {
      return (unsigned long long)(expf(key_value(key) - m) * 1099511627776.0f);
    };
    // one search: the digits found so far, the sum over all keys above them, the target
    uint32_t prefix[2] = {0u, 0u};
    unsigned long long above[2] = {0ull, 0ull}, target[2] = {(unsigned long long)(k > 0 ? k : 0), 0ull};
    auto descend = [&](bool on_k, bool on_p) {
      const bool on[2] = {on_k, on_p};
      prefix[0] = on_k ? 0u : prefix[0], prefix[1] = on_p ? 0u : prefix[1];
      above[0] = on_k ? 0ull : above[0], above[1] = on_p ? 0ull : above[1];
#pragma unroll 1
      for (int level = 0; level < 3; ++level) {
        const int shift = level == 0 ? 21 : (level == 1 ? 10 : 0);
        const int up = level == 0 ? 32 : (level == 1 ? 21 : 10);  // bits below `up` are open
        for (int b = tid; b < 2 * SAMPLE_BINS; b += SAMPLE_THREADS) (&hist[0][0])[b] = 0ull;
        __syncthreads();
        for (int i = tid; i < V; i += SAMPLE_THREADS) {
          const uint32_t key = key_at(i);
          const uint32_t high = level == 0 ? 0u : key >> up;
          const uint32_t bin = (key >> shift) & (SAMPLE_BINS - 1) & ((1u << (up - shift)) - 1u);
          if (on[0] && high == prefix[0]) atomicAdd(&hist[0][bin], 1ull);
          if (on[1] && high == prefix[1]) atomicAdd(&hist[1][bin], fixed(key));
        }
        __syncthreads();
        if (level == 0 && on[1]) {
          // the whole mass, as the histogram has it: the reference of top-p unless the
          // caller has set another
          unsigned long long all = hist[1][2 * tid] + hist[1][2 * tid + 1];
          all += block_suffix_u64(all, scan_tmp);
          if (tid == 0) whole_mass = all;
          __syncthreads();
          if (target[1] == ~0ull) {
            const double t = (double)tp * (double)whole_mass;
            target[1] = (unsigned long long)t;
          }
        }
#pragma unroll
        for (int sidx = 0; sidx < 2; ++sidx) {
          if (!on[sidx]) continue;
          // bins in descending order: thread t has bins 2t+1 and 2t
          const unsigned long long h1 = hist[sidx][2 * tid + 1], h0 = hist[sidx][2 * tid];
          const unsigned long long higher = above[sidx] + block_suffix_u64(h1 + h0, scan_tmp);
          if (tid == 0) found_bin[sidx] = 0u, found_above[sidx] = above[sidx] + 0ull, found_any[sidx] = 0;
          __syncthreads();
          if (higher < target[sidx] && higher + h1 >= target[sidx]) {
            found_bin[sidx] = 2 * tid + 1, found_above[sidx] = higher, found_any[sidx] = 1;
          } else if (higher + h1 < target[sidx] && higher + h1 + h0 >= target[sidx]) {
            found_bin[sidx] = 2 * tid, found_above[sidx] = higher + h1, found_any[sidx] = 1;
          }
          __syncthreads();
          // a target of zero, or one beyond the whole sum, is met by no bin: the first
          // keeps the largest key only, the second every key
          if (!found_any[sidx]) {
            if (target[sidx] == 0ull) {
              int top = -1;
              if (h1 != 0ull) top = 2 * tid + 1; else if (h0 != 0ull) top = 2 * tid;
              if (top >= 0) atomicMax(&found_bin[sidx], (uint32_t)top);
            }
            __syncthreads();
          }
          prefix[sidx] = (prefix[sidx] << (up - shift)) | found_bin[sidx];
          above[sidx] = found_above[sidx];
          __syncthreads();
        }
      }
    };
    const bool p_after_k = want_k && want_p && mp > 0.f;  // top-p refers to what top-k kept
    target[1] = ~0ull;                                    // top_p of the whole mass
    if (!p_after_k) {
      descend(want_k, want_p);
      if (want_k) key_min = prefix[0];
      if (want_p && prefix[1] > key_min) key_min = prefix[1];
    } else {
      descend(true, false);
      key_min = prefix[0];
      // with min_p the reference renormalises after top-k, so top-p refers to the
      // mass that top-k kept
      unsigned long long kept = 0ull;
      for (int i = tid; i < V; i += SAMPLE_THREADS) {
        const uint32_t key = key_at(i);
        if (key >= key_min) kept += fixed(key);
      }
      kept += block_suffix_u64(kept, scan_tmp);
      if (tid == 0) whole_mass = kept;
      __syncthreads();
      target[1] = (unsigned long long)((double)tp * (double)whole_mass);
      __syncthreads();
      descend(false, true);
      if (prefix[1] > key_min) key_min = prefix[1];
    }
  }

  // ---- inverse CDF over the kept tokens in index order -----------------------------
  // A wave owns a contiguous run of tokens and reads it 64 tokens at a time; a prefix
  // sum over the waves' kept masses finds the wave that holds the target, and that wave
  // walks its run again with a prefix sum over each 64 tokens.
  const int n_waves = SAMPLE_THREADS / HAL_WAVE;
  const int run_len = ((V + n_waves - 1) / n_waves + HAL_WAVE - 1) / HAL_WAVE * HAL_WAVE;
  const int begin = wave * run_len;
  const int end = begin + run_len < V ? begin + run_len : V;
  auto kept_mass_of = [&](int i, float& z) {
    if (i >= end) return 0.f;
    const uint32_t key = key_at(i);
    if (key < key_min) return 0.f;
    z = key_value(key);
    const float e = expf(z - m);
    return e >= mp ? e : 0.f;
  };
  float mine = 0.f, zz;
  for (int i = begin + lane; i < end; i += HAL_WAVE) mine += kept_mass_of(i, zz);
  const float wave_mass = wave_sum(mine);
  if (tid == 0) {
    chosen_thread = 0x7fffffff;
    last_thread = -1;
  }
  if (lane == 0) red2[wave] = wave_mass;
  __syncthreads();
  float before = 0.f, kept_mass = 0.f;
  for (int w = 0; w < n_waves; ++w) {
    if (w < wave) before += red2[w];
    kept_mass += red2[w];
  }
  const float target = uniform_draw(seeds[row], (uint32_t)draw_index[row]) * kept_mass;
  if (lane == 0 && wave_mass > 0.f) {
    atomicMax(&last_thread, wave);
    if (before + wave_mass > target) atomicMin(&chosen_thread, wave);
  }
  __syncthreads();
  int pick = chosen_thread;
  if (pick == 0x7fffffff) pick = last_thread;  // rounding left the target at the very end
  if (pick < 0) pick = 0;                      // nothing is kept anywhere: token 0 below
  if (wave != pick) return;
  float run = before;
  int tok = -1, last_kept = -1;
  float z_tok = 0.f, z_last = 0.f;
  for (int i0 = begin; i0 < end && tok < 0; i0 += HAL_WAVE) {
    float z = 0.f;
    const float e = kept_mass_of(i0 + lane, z);
    float incl = e;
#pragma unroll
    for (int off = 1; off < HAL_WAVE; off <<= 1) {
      const float up = __shfl_up(incl, off, HAL_WAVE);
      if (lane >= off) incl += up;
    }
    const unsigned long long kept_lanes = __builtin_amdgcn_ballot_w64(e > 0.f);
    const unsigned long long hit = __builtin_amdgcn_ballot_w64(e > 0.f && run + incl > target);
    if (kept_lanes) {
      const int hi = 63 - __builtin_clzll(kept_lanes);
      last_kept = i0 + hi;
      z_last = __shfl(z, hi, HAL_WAVE);
    }
    if (hit) {
      const int lo = __builtin_ctzll(hit);
      tok = i0 + lo;
      z_tok = __shfl(z, lo, HAL_WAVE);
    }
    run += __shfl(incl, HAL_WAVE - 1, HAL_WAVE);
  }
  if (tok < 0) {
    tok = last_kept >= 0 ? last_kept : (am.i < V ? am.i : 0);
    z_tok = last_kept >= 0 ? z_last : m;
  }
  if (lane == 0) {
    out_token[row] = tok;
    out_logprob[row] = z_tok - m - logf(total);
  }
}

// `key_rows`: room for n_rows * V 32-bit words that the kernel may use between its
// passes, or null (every pass then derives the keys from the logits again).
extern "C" int hal_sample(const float* logits, int ld, int n_rows, int V, const float* temperature,
                          const int* top_k, const float* top_p, const float* min_p,
                          const uint64_t* seeds, const int* draw_index, int* out_token,
                          float* out_logprob, uint32_t* key_rows, hipStream_t stream) {
  HAL_REQUIRE(n_rows >= 0 && V > 0 && ld >= V, "hal_sample: bad sizes rows=%d V=%d ld=%d", n_rows,
              V, ld);
  if (n_rows == 0) return 0;
  hipLaunchKernelGGL(sample_kernel, dim3(n_rows), dim3(SAMPLE_THREADS), 0, stream, logits, ld, V,
                     temperature, top_k, top_p, min_p, seeds, draw_index, out_token, out_logprob,
                     key_rows);
  HAL_LAUNCH_CHECK();
  return 0;
}

// ---- no row has a filter: the row is spread over ROW_PARTS blocks ---------------------------
// Greedy rows and rows that draw from the whole temperature-scaled distribution need the
// row's maximum, the sum of exp(z - maximum) and, for a draw, one walk to the token at which
// the cumulative probability passes u: no thresholds.  Stage one: a block takes a contiguous
// share of a row and leaves its maximum, the first index of that maximum and the sum of
// exp(z - maximum), z = logit / temperature (the logit itself for a greedy row).  Stage two
// joins a row's shares in order (ties go to the lower index, as everywhere); for a draw it
// finds the share in which the running sum passes u * total and walks that share, a quarter
// per wave, as the one-block kernel walks the row.  Same generator, same rule, same
// log-probability as there; sums are added in another order, so a draw within rounding of a
// token's edge may fall to its neighbour.
#define ROW_PARTS 32
#define PART_THREADS 256

__device__ __forceinline__ int part_share(int V) { return ((V + ROW_PARTS - 1) / ROW_PARTS + 3) / 4 * 4; }
// The logits begin + tid, begin + tid + PART_THREADS, ... below `end`, PART_BATCH of them asked for
// before the first is worked on (a share of a vocabulary of up to 131,072 is one batch): these passes are
// bound by the trips to memory, which a load at a time takes one after the other.  64 rows of 128,256 with
// top-p: a pass over the rows 10.6 -> 10.1 us, the first one, which keeps its batch, 20.9 -> 15.1 us, a
// histogram 19.4 -> 12.7 us on average (where it also leaves out what the row does not search by).  Places of the
// batch that lie past the share are passed over by all threads at once: worked through by none of them, 200 rows
// of 1,000 logits without filters took 23.0 us, of 32,000 29.9, and take 16.5 and 23.4 so.  (Asking and working as two functions
// schedules better than as one: a call of 64 rows with top-p 59.8 us / 60.7.)
#define PART_BATCH 16
template <bool WHOLE>
__device__ __forceinline__ void ask_batch(const float* x, int from, int end, float (&v)[PART_BATCH]) {
#pragma unroll
  for (int u = 0; u < PART_BATCH; ++u) {
    if (!WHOLE && from + u * PART_THREADS >= end) break;
    const int i = from + u * PART_THREADS + (int)threadIdx.x;
    v[u] = x[i < end ? i : from];
  }
}
template <bool WHOLE, typename F>
__device__ __forceinline__ void use_batch(const float (&v)[PART_BATCH], int from, int end, F&& each) {
#pragma unroll
  for (int u = 0; u < PART_BATCH; ++u) {
    if (!WHOLE && from + u * PART_THREADS >= end) break;
    const int i = from + u * PART_THREADS + (int)threadIdx.x;
    if (i < end) each(v[u], i, u);
  }
}
template <typename F>
__device__ __forceinline__ void for_part(const float* x, int begin, int end, F&& each) {
  for (int from = begin; from < end; from += PART_BATCH * PART_THREADS) {
    float v[PART_BATCH];
    if (from + (PART_BATCH - 1) * PART_THREADS < end) ask_batch<true>(x, from, end, v), use_batch<true>(v, from, end, each);
    else ask_batch<false>(x, from, end, v), use_batch<false>(v, from, end, each);
  }
}

// a row is greedy if it has no temperature array (all rows greedy), a temperature of 0 or top_k 1
__device__ __forceinline__ float row_scale_of(const float* temperature, const int* top_k, int row) {
  if (!temperature) return 0.f;
  const float T = temperature[row];
  return (T == 0.f || (top_k && top_k[row] == 1)) ? 0.f : T;
}

__global__ void __launch_bounds__(PART_THREADS)
row_part_kernel(const float* __restrict__ logits, int ld, int V,
                const float* __restrict__ temperature, const int* __restrict__ top_k,
                float* __restrict__ parts) {
  __shared__ ArgMax amax_s[PART_THREADS / HAL_WAVE];
  __shared__ float red[16];
  const int row = blockIdx.y, part = blockIdx.x, tid = threadIdx.x;
  const int lane = tid % HAL_WAVE, wave = tid / HAL_WAVE;
  const int share = part_share(V);
  const int begin = part * share;
  const int end = begin + share < V ? begin + share : V;
  const float* x = logits + (size_t)row * ld;
  const float T = row_scale_of(temperature, top_k, row);
  const float inv_scale = T == 0.f ? 1.f : T;
  ArgMax am = {-INFINITY, 0x7fffffff};
  float z_of[PART_BATCH];
  for_part(x, begin, end, [&](float v, int i, int u) {
    const float z = clean_logit(v) / inv_scale;
    z_of[u] = z;
    if (z > am.v) am.v = z, am.i = i;  // a thread's indices rise: the first maximum stays
  });
#pragma unroll
  for (int off = HAL_WAVE / 2; off > 0; off >>= 1) {
    ArgMax o;
    o.v = __shfl_xor(am.v, off, HAL_WAVE);
    o.i = __shfl_xor(am.i, off, HAL_WAVE);
    am = argmax_merge(am, o);
  }
  if (lane == 0) amax_s[wave] = am;
  __syncthreads();
  am = amax_s[0];
  for (int w = 1; w < PART_THREADS / HAL_WAVE; ++w) am = argmax_merge(am, amax_s[w]);
  float sum = 0.f;
  if (share <= PART_BATCH * PART_THREADS) {  // the batch is the share
    if (begin + (PART_BATCH - 1) * PART_THREADS < end) {
#pragma unroll
      for (int u = 0; u < PART_BATCH; ++u)
        if (begin + tid + u * PART_THREADS < end) sum += expf(z_of[u] - am.v);
    } else {
#pragma unroll
      for (int u = 0; u < PART_BATCH; ++u) {
        if (begin + u * PART_THREADS >= end) break;
        if (begin + tid + u * PART_THREADS < end) sum += expf(z_of[u] - am.v);
      }
    }
  } else {
    for_part(x, begin, end, [&](float v, int, int) { sum += expf(clean_logit(v) / inv_scale - am.v); });
  }
  sum = block_sum(sum, red);
  if (tid == 0) {
    float* p = parts + ((size_t)row * ROW_PARTS + part) * 4;
    p[0] = am.v;
    p[1] = __int_as_float(am.i);
    p[2] = begin < end ? sum : 0.f;
  }
}

__global__ void __launch_bounds__(PART_THREADS)
row_join_kernel(const float* __restrict__ logits, int ld, int V, const float* __restrict__ parts,
                const float* __restrict__ temperature, const int* __restrict__ top_k,
                const uint64_t* __restrict__ seeds, const int* __restrict__ draw_index,
                int* __restrict__ out_token, float* __restrict__ out_logprob) {
  __shared__ float quarter_mass[PART_THREADS / HAL_WAVE];
  const int row = blockIdx.x, tid = threadIdx.x;
  const int lane = tid % HAL_WAVE, wave = tid / HAL_WAVE;
  // every wave joins the shares for itself (32 values)
  ArgMax am = {-INFINITY, 0x7fffffff};
  float sum = 0.f;
  if (lane < ROW_PARTS) {
    const float* p = parts + ((size_t)row * ROW_PARTS + lane) * 4;
    am.v = p[0], am.i = __float_as_int(p[1]), sum = p[2];
  }
  ArgMax best = am;
#pragma unroll
  for (int off = HAL_WAVE / 2; off > 0; off >>= 1) {
    ArgMax o;
    o.v = __shfl_xor(best.v, off, HAL_WAVE);
    o.i = __shfl_xor(best.i, off, HAL_WAVE);
    best = argmax_merge(best, o);
  }
  const float m = best.v;
  const float scaled = (am.v == -INFINITY) ? 0.f : sum * expf(am.v - m);
  const float total = wave_sum(scaled);
  const float T = row_scale_of(temperature, top_k, row);
  if (T == 0.f) {  // greedy
    if (tid == 0) {
      out_token[row] = best.i < V ? best.i : 0;
      out_logprob[row] = -logf(total);
    }
    return;
  }
  // the share in which the running sum (shares in order) passes the target
  const float target = uniform_draw(seeds[row], (uint32_t)draw_index[row]) * total;
  float incl = scaled;
#pragma unroll
  for (int off = 1; off < HAL_WAVE; off <<= 1) {
    const float up = __shfl_up(incl, off, HAL_WAVE);
    if (lane >= off) incl += up;
  }
  const unsigned long long some = __builtin_amdgcn_ballot_w64(scaled > 0.f);
  const unsigned long long hit = __builtin_amdgcn_ballot_w64(scaled > 0.f && incl > target);
  // rounding may leave the target at the very end: the last share that holds anything
  // (a row of nothing but -inf holds nothing anywhere: share 0 then, and token 0 below)
  const int part = hit ? __builtin_ctzll(hit) : (some ? 63 - __builtin_clzll(some) : 0);
  const float before_part = __shfl(incl - scaled, part, HAL_WAVE);

  // the share is walked as the one-block kernel walks a row: a quarter per wave
  const float* x = logits + (size_t)row * ld;
  const int share = part_share(V);
  const int p_begin = part * share, p_end = p_begin + share < V ? p_begin + share : V;
  constexpr int n_waves = PART_THREADS / HAL_WAVE;
  const int run_len = ((p_end - p_begin + n_waves - 1) / n_waves + HAL_WAVE - 1) / HAL_WAVE * HAL_WAVE;
  const int begin = p_begin + wave * run_len;
  const int end = begin + run_len < p_end ? begin + run_len : p_end;
  auto mass_of = [&](int i, float& z) {
    if (i >= end) return 0.f;
    z = clean_logit(x[i]) / T;
    return expf(z - m);
  };
  float mine = 0.f, zz;
  for (int i = begin + lane; i < end; i += HAL_WAVE) mine += mass_of(i, zz);
  const float wave_mass = wave_sum(mine);
  if (lane == 0) quarter_mass[wave] = wave_mass;
  __syncthreads();
  float before = before_part;
  int pick = -1, last = -1;
  for (int w = 0; w < n_waves; ++w) {
    if (quarter_mass[w] > 0.f) last = w;
    if (pick < 0 && quarter_mass[w] > 0.f && before + quarter_mass[w] > target) pick = w;
    if (pick < 0) before += quarter_mass[w];
  }
  if (pick < 0) {  // rounding again: the last quarter that holds anything, from its start
    pick = last < 0 ? 0 : last;
    before = before_part;
    for (int w = 0; w < pick; ++w) before += quarter_mass[w];
  }
  if (wave != pick) return;
  float run = before;
  int tok = -1, last_kept = -1;
  float z_tok = 0.f, z_last = 0.f;
  for (int i0 = begin; i0 < end && tok < 0; i0 += HAL_WAVE) {
    float z = 0.f;
    const float e = mass_of(i0 + lane, z);
    float inc = e;
#pragma unroll
    for (int off = 1; off < HAL_WAVE; off <<= 1) {
      const float up = __shfl_up(inc, off, HAL_WAVE);
      if (lane >= off) inc += up;
    }
    const unsigned long long kept_lanes = __builtin_amdgcn_ballot_w64(e > 0.f);
    const unsigned long long found = __builtin_amdgcn_ballot_w64(e > 0.f && run + inc > target);
    if (kept_lanes) {
      const int hi = 63 - __builtin_clzll(kept_lanes);
      last_kept = i0 + hi;
      z_last = __shfl(z, hi, HAL_WAVE);
    }
    if (found) {
      const int lo = __builtin_ctzll(found);
      tok = i0 + lo;
      z_tok = __shfl(z, lo, HAL_WAVE);
    }
    run += __shfl(inc, HAL_WAVE - 1, HAL_WAVE);
  }
  if (tok < 0) {
    tok = last_kept >= 0 ? last_kept : (best.i < V ? best.i : 0);
    z_tok = last_kept >= 0 ? z_last : m;
  }
  if (lane == 0) {
    out_token[row] = tok;
    out_logprob[row] = z_tok - m - logf(total);
  }
}

// ---- rows with filters, spread over many blocks -----------------------------------------
// A row's passes are shared by ROW_PARTS blocks each; what a pass over 64 rows of 128,256 costs is its
// launch, the logits' way from memory (33 MB, 6.5 us) and about fifty instructions a logit where it takes
// an exponential.  So a row is passed over three times, and once with its share alone:
//   filt_max_kernel     its maximum;
//   filt_coarse_kernel  the sum of exponentials, and how many logits and what mass lie in each of 256 bins of
//                       the distance from the maximum (an eighth wide; the last takes the rest);
//   filt_list_kernel    the keys in the bin that holds the threshold, as lists in memory, and the mass of what lies
//                       before that bin, a share;
//   filt_pick_kernel    (a block a row) the threshold among them, by radix selection over the bits in which
//                       they differ, with it the kept mass of every share, and the draw.
// Distances are monotone in the keys, so the bins hold the keys in order, and counts and masses are integers: the
// thresholds are the same keys as the one-block kernel's, and the shares' kept masses do not depend on an order either.  The drawn token may differ where
// the draw is within rounding of a token's edge, since the kept masses are made in another way.  A row with top-k, top-p and min-p
// all at once, where top-p refers to what top-k kept, is searched twice: top-k first (filt_find_kernel), then (`late`) top-p
// of the mass that top-k kept.
// 64 rows of 128,256 with top-p: 12.2 + 14.4 + 11.3 + 20.0 us of kernels, a call 59.7.  (A pass over the rows for the kept masses and the search and the
// draw as kernels of their own: 12.4 + 14.7 + 10.7 + 12.8 + 9.8 + 8.3, 69.  With a share's logits asked for before what their work needs is there
// the two middle passes take 1.5 and 5 us more.)
struct FiltRow {
  float m;        // maximum of z
  int best;       // its first index
  uint32_t key_min;              // late rows: of their first search
  unsigned long long kept_by_k;  // and the mass of the keys that it kept
};
static_assert(sizeof(FiltRow) == 24, "a row's state is 6 words");
#define FILT_BINS 256
// greedy; top-k is searched; top-p is searched beside it; top-p is searched after it (late)
enum { FILT_GREEDY = 1, FILT_K = 2, FILT_P = 4, FILT_P_LATE = 8 };

struct FiltParams {
  const float *temperature, *top_p, *min_p;
  const int* top_k;
};

// (all four parameters are asked for at once: one after the other, each is a trip to memory)
__device__ __forceinline__ int filt_flags(const FiltParams& p, int V, int row) {
  const float T = p.temperature[row], tp = p.top_p[row], mp = p.min_p[row];
  const int k = p.top_k[row];
  const bool want_k = (k > 0) & (k < V), want_p = tp < 1.f;
  // with min_p the reference renormalises after top-k, so top-p refers to what top-k kept
  const bool late = want_k & want_p & (mp > 0.f);
  const int flags = (want_k ? FILT_K : 0) | (want_p ? (late ? FILT_P_LATE : FILT_P) : 0);
  return (T == 0.f) | (k == 1) ? FILT_GREEDY : flags;
}

// the bin of a z (the last one also where there is no distance: a maximum that is infinite)
__device__ __forceinline__ int filt_bin(float z, float m) { return (int)fminf((m - z) * 8.0f, (float)(FILT_BINS - 1)); }
// a key's mass, in units of 2^-40 of the largest
__device__ __forceinline__ unsigned long long filt_fixed(float e) { return (unsigned long long)(e * 1099511627776.0f); }

__global__ void __launch_bounds__(PART_THREADS, 8)  // (eight blocks a compute unit: 64 rows at once)
filt_max_kernel(const float* __restrict__ logits, int ld, int V, FiltParams params, float* __restrict__ parts,
                unsigned long long* __restrict__ hist) {  // [rows][2][FILT_BINS]
  __shared__ ArgMax amax_s[PART_THREADS / HAL_WAVE];
  const int row = blockIdx.y, part = blockIdx.x, tid = threadIdx.x;
  const int lane = tid % HAL_WAVE, wave = tid / HAL_WAVE;
  constexpr int MINE = 2 * FILT_BINS / ROW_PARTS;  // of the row's bins, which start at zero
  if (tid < MINE) hist[(size_t)row * 2 * FILT_BINS + part * MINE + tid] = 0ull;
  const int share = part_share(V);
  const int begin = part * share;
  const int end = begin + share < V ? begin + share : V;
  const float* x = logits + (size_t)row * ld;
  const float T = row_scale_of(params.temperature, params.top_k, row);
  const float scale = T == 0.f ? 1.f : T;
  // The quotient rises with the logit, so the largest logit has the largest z, and only logits next to it can
  // share that z: those alone are divided to find the first (all, where quotients run into the type's ends).
  ArgMax am = {-INFINITY, 0x7fffffff};
  float held[PART_BATCH];
  float top = -INFINITY;
  const bool one_batch = share <= PART_BATCH * PART_THREADS;
  for_part(x, begin, end, [&](float v, int, int u) {
    held[u] = clean_logit(v);
    top = fmaxf(top, held[u]);
  });
  am.v = top / scale;
  const float near = fabsf(am.v) > 1e-30f && fabsf(am.v) < INFINITY ? top - fabsf(top) * 1e-6f : -INFINITY;
  auto first = [&](float v, int i) {
    if (v >= near && am.i == 0x7fffffff && am.v > -INFINITY && v / scale == am.v) am.i = i;
  };
  if (one_batch) {
#pragma unroll
    for (int u = 0; u < PART_BATCH; ++u) {
      const int i = begin + tid + u * PART_THREADS;
      if (i < end) first(held[u], i);
    }
  } else {
    for_part(x, begin, end, [&](float v, int i, int) { first(clean_logit(v), i); });
  }
#pragma unroll
  for (int off = HAL_WAVE / 2; off > 0; off >>= 1) {
    ArgMax o;
    o.v = __shfl_xor(am.v, off, HAL_WAVE);
    o.i = __shfl_xor(am.i, off, HAL_WAVE);
    am = argmax_merge(am, o);
  }
  if (lane == 0) amax_s[wave] = am;
  __syncthreads();
  if (tid != 0) return;
  for (int w = 1; w < PART_THREADS / HAL_WAVE; ++w) am = argmax_merge(am, amax_s[w]);
  float* p = parts + ((size_t)row * ROW_PARTS + part) * 4;
  p[0] = am.v;
  p[1] = __int_as_float(am.i);
}

__global__ void __launch_bounds__(PART_THREADS)
filt_coarse_kernel(const float* __restrict__ logits, int ld, int V, FiltParams params, float* __restrict__ parts,
                   FiltRow* __restrict__ rows, unsigned long long* __restrict__ hist) {
  __shared__ uint32_t count_s[FILT_BINS];
  __shared__ unsigned long long mass_s[FILT_BINS];
  __shared__ float red[16];
  static_assert(FILT_BINS == PART_THREADS, "a thread a bin");
  const int row = blockIdx.y, part = blockIdx.x, tid = threadIdx.x, lane = tid % HAL_WAVE;
  const int flags = filt_flags(params, V, row);
  const bool on_k = (flags & FILT_K) != 0, on_p = (flags & (FILT_P | FILT_P_LATE)) != 0;
  const int share = part_share(V);
  const int begin = part * share, end = begin + share < V ? begin + share : V;
  const float* x = logits + (size_t)row * ld;
  count_s[tid] = 0u;
  mass_s[tid] = 0ull;
  // every wave joins the shares' maxima for itself
  ArgMax best = {-INFINITY, 0x7fffffff};
  if (lane < ROW_PARTS) {
    const float* p = parts + ((size_t)row * ROW_PARTS + lane) * 4;
    best.v = p[0], best.i = __float_as_int(p[1]);
  }
#pragma unroll
  for (int off = HAL_WAVE / 2; off > 0; off >>= 1) {
    ArgMax o;
    o.v = __shfl_xor(best.v, off, HAL_WAVE);
    o.i = __shfl_xor(best.i, off, HAL_WAVE);
    best = argmax_merge(best, o);
  }
  const float m = best.v;
  if (part == 0 && tid == 0) {
    FiltRow r;
    r.m = m, r.best = best.i, r.key_min = 0u, r.kept_by_k = 0ull;
    rows[row] = r;
  }
  __syncthreads();
  const float T = row_scale_of(params.temperature, params.top_k, row), scale = T == 0.f ? 1.f : T;
  float sum = 0.f;
  for_part(x, begin, end, [&](float v, int, int) {
    const float z = clean_logit(v) / scale, e = expf(z - m);
    sum += e;
    const int bin = filt_bin(z, m);
    if (on_p) atomicAdd(&mass_s[bin], filt_fixed(e));
    if (on_k) atomicAdd(&count_s[bin], 1u);
  });
  sum = block_sum(sum, red);
  if (tid == 0) parts[((size_t)row * ROW_PARTS + part) * 4 + 2] = begin < end && m > -INFINITY ? sum : 0.f;
  unsigned long long* h = hist + (size_t)row * 2 * FILT_BINS;
  if (on_k && count_s[tid]) atomicAdd(&h[tid], (unsigned long long)count_s[tid]);
  if (on_p && mass_s[tid]) atomicAdd(&h[FILT_BINS + tid], mass_s[tid]);
}

// Where a row's thresholds lie: for each of the two searches the bin and the sum over the bins before it (nearer the
// maximum).  A block of at least FILT_BINS threads, all of which get the result.
struct FiltPlace {
  bool on[2];     // top-k, top-p
  bool largest[2];  // the target is nothing: the largest key alone is kept
  int bin[2];
  unsigned long long before[2], target[2];
  int list;  // the bin whose keys are listed: that of the higher threshold; -1: none
};
__device__ __forceinline__ FiltPlace filt_place(const unsigned long long* __restrict__ h, const FiltParams& params, int V, int row,
                                                const FiltRow& r, int late) {
  __shared__ unsigned long long wave_sums[2][FILT_BINS / HAL_WAVE];
  __shared__ unsigned long long before_s[2];
  __shared__ int bin_s[2];
  const int tid = threadIdx.x, lane = tid % HAL_WAVE, wave = tid / HAL_WAVE;
  const int flags = filt_flags(params, V, row);
  FiltPlace f;
  f.on[0] = !late && (flags & FILT_K) != 0;
  f.on[1] = (flags & (late ? FILT_P_LATE : FILT_P)) != 0;
  f.list = -1;
  f.largest[0] = f.largest[1] = false;
  if (!f.on[0] && !f.on[1]) return f;
  unsigned long long own[2] = {0ull, 0ull}, upto[2];
  if (tid < FILT_BINS) own[0] = h[tid], own[1] = h[FILT_BINS + tid];  // (zeros where there is no such search)
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    upto[w] = own[w];
#pragma unroll
    for (int off = 1; off < HAL_WAVE; off <<= 1) {
      const uint32_t lo = __shfl_up((uint32_t)upto[w], off, HAL_WAVE), hi = __shfl_up((uint32_t)(upto[w] >> 32), off, HAL_WAVE);
      if (lane >= off) upto[w] += ((unsigned long long)hi << 32) | lo;
    }
    if (lane == HAL_WAVE - 1 && tid < FILT_BINS) wave_sums[w][wave] = upto[w];
  }
  if (tid < 2) bin_s[tid] = FILT_BINS - 1, before_s[tid] = 0ull;
  __syncthreads();
  unsigned long long all = 0ull;
#pragma unroll
  for (int w = 0; w < FILT_BINS / HAL_WAVE; ++w) {
    if (w < wave) upto[0] += wave_sums[0][w], upto[1] += wave_sums[1][w];
    all += wave_sums[1][w];
  }
  f.target[0] = (unsigned long long)params.top_k[row];
  // top-p of the whole mass, as the bins have it, or of what top-k kept
  f.target[1] = (unsigned long long)((double)params.top_p[row] * (double)(late ? r.kept_by_k : all));
#pragma unroll
  for (int w = 0; w < 2; ++w)
    if (tid < FILT_BINS && f.on[w] && upto[w] - own[w] < f.target[w] && upto[w] >= f.target[w]) bin_s[w] = tid, before_s[w] = upto[w] - own[w];
  __syncthreads();
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    f.bin[w] = bin_s[w], f.before[w] = before_s[w];
    f.largest[w] = f.on[w] && f.target[w] == 0ull;
    if (f.largest[w]) f.bin[w] = 0;
    if (f.on[w] && !f.largest[w] && (f.list < 0 || f.bin[w] < f.list)) f.list = f.bin[w];
  }
  if (f.largest[0] || f.largest[1]) f.list = -1;  // (nothing to search for: the largest key is the threshold)
  return f;
}

// What a share keeps for certain (its mass, to `kept`), and the keys among which the row's threshold lies, at the share's own place in the
// row's list (their number is the fourth of the share's `parts`).  The logits that are not surely below the threshold's bin, a few in
// a hundred, are gathered first and then go through quotient and exponential together; masses are added up as integers, so that their
// order does not matter.
__global__ void __launch_bounds__(PART_THREADS)
filt_list_kernel(const float* __restrict__ logits, int ld, int V, FiltParams params, const FiltRow* __restrict__ rows, int late,
                 const unsigned long long* __restrict__ hist, float* __restrict__ parts, float* __restrict__ kept,
                 uint32_t* __restrict__ lists) {  // [rows][V]
  __shared__ float found[PART_BATCH * PART_THREADS];
  __shared__ unsigned long long mass_s[PART_THREADS / HAL_WAVE];
  __shared__ int n_found, n_listed;
  const int row = blockIdx.y, part = blockIdx.x, tid = threadIdx.x;
  const int flags = filt_flags(params, V, row);
  if (flags == FILT_GREEDY || (late && !(flags & FILT_P_LATE))) return;
  const int share = part_share(V);
  const int begin = part * share, end = begin + share < V ? begin + share : V;
  const float* x = logits + (size_t)row * ld;
  const FiltRow r = rows[row];
  if (tid == 0) n_listed = 0;
  const FiltPlace f = filt_place(hist + (size_t)row * 2 * FILT_BINS, params, V, row, r, late);
  const bool largest = f.largest[0] || f.largest[1];  // the largest key alone is kept; without a search and that, every key
  const float T = params.temperature[row], mp = params.min_p[row];
  // A bound a 100,000th of the numbers that it is made of below what counts: the bin's end, or without a search the largest key or min-p's.
  const float wide = 1e-5f * (fabsf(r.m) + 32.f) * T;
  float low = f.list < 0 || f.list == FILT_BINS - 1 ? -INFINITY : (r.m - 0.125f * (f.list + 1)) * T - wide;
  if (f.list < 0 && (largest || mp > 0.f)) low = (largest ? r.m : r.m + logf(mp)) * T - wide;
  const uint32_t top = sort_key(r.m);
  uint32_t* list = lists + (size_t)row * V + begin;
  unsigned long long mass = 0ull;
  for (int from = begin; from < end; from += PART_BATCH * PART_THREADS) {
    const int to = from + PART_BATCH * PART_THREADS < end ? from + PART_BATCH * PART_THREADS : end;
    if (tid == 0) n_found = 0;
    __syncthreads();
    auto gather = [&](float v, int, int) {
      v = clean_logit(v);
      if (v >= low) found[atomicAdd(&n_found, 1)] = v;
    };
    for_part(x, from, to, gather);
    __syncthreads();
    for (int i = tid; i < n_found; i += PART_THREADS) {
      const float z = found[i] / T;
      const int bin = f.list < 0 ? 0 : filt_bin(z, r.m);
      const bool sure = f.list < 0 ? !largest || sort_key(z) >= top : bin < f.list;
      if (sure) {
        const float e = expf(z - r.m);
        if (e >= mp) mass += filt_fixed(e);
      } else if (bin == f.list) {
        list[atomicAdd(&n_listed, 1)] = sort_key(z);
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int off = HAL_WAVE / 2; off; off >>= 1) {
    const uint32_t lo = __shfl_xor((uint32_t)mass, off, HAL_WAVE), hi = __shfl_xor((uint32_t)(mass >> 32), off, HAL_WAVE);
    mass += ((unsigned long long)hi << 32) | lo;
  }
  if (tid % HAL_WAVE == 0) mass_s[tid / HAL_WAVE] = mass;
  __syncthreads();
  if (tid != 0) return;
  for (int w = 1; w < PART_THREADS / HAL_WAVE; ++w) mass += mass_s[w];
  kept[(size_t)row * ROW_PARTS + part] = (float)mass * (1.0f / 1099511627776.0f);
  parts[((size_t)row * ROW_PARTS + part) * 4 + 3] = __int_as_float(n_listed);
}

// The smallest key that a row keeps by the searches of this pass, by a block a row; all its threads get it.  `listed`: lane l's is how many keys share l has.  The keys of the row's list are searched bit by
// bit of those in which they differ, ten at a time from the top, from histograms over the keys that share the bits found so far (the keys of a bin
// differ in some eighteen bits: two rounds).  A wave has two shares' keys.  (Every block of another pass finding it for itself: 24 us more there.)
#define PICK_THREADS 1024
#define FILT_DIGIT 10
#define FILT_STAGED 4096  // keys of a list that are kept in LDS
struct FiltSearch {
  unsigned long long bins[1 << FILT_DIGIT], tmp[PICK_THREADS / HAL_WAVE], above;
  uint32_t staged[FILT_STAGED], ends[2], bin;
  int first[ROW_PARTS + 1];  // the shares' first keys, counted over the row
};
static_assert((1 << FILT_DIGIT) == PICK_THREADS && SAMPLE_THREADS == PICK_THREADS && PICK_THREADS / HAL_WAVE * 2 == ROW_PARTS, "a thread a bin, a wave two shares");
// What a wave does with each key of each of its shares.
template <typename F>
__device__ __forceinline__ void filt_each(const FiltSearch& s, const uint32_t* keys, int V, F&& what) {
  const int lane = threadIdx.x % HAL_WAVE, wave = threadIdx.x / HAL_WAVE, share = part_share(V);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int part = 2 * wave + h, first = s.first[part], n = s.first[part + 1] - first;
    for (int k = lane; k < n; k += HAL_WAVE) what(first + k < FILT_STAGED ? s.staged[first + k] : keys[part * share + k], part);
  }
}
__device__ __forceinline__ uint32_t filt_search(FiltSearch& s, const FiltPlace& f, const FiltRow& r, int listed, const uint32_t* keys, int V, int late) {
  const int tid = threadIdx.x, lane = tid % HAL_WAVE, wave = tid / HAL_WAVE, share = part_share(V);
  uint32_t key_min = late ? r.key_min : 0u;
  if (f.largest[0] || f.largest[1]) key_min = sort_key(r.m);
  if (wave == 0) {
    int upto = f.list >= 0 ? listed : 0;
#pragma unroll
    for (int off = 1; off < ROW_PARTS; off <<= 1) {
      const int v = __shfl_up(upto, off, HAL_WAVE);
      if (lane >= off) upto += v;
    }
    if (lane < ROW_PARTS) s.first[lane + 1] = upto;
    if (lane == 0) s.first[0] = 0, s.ends[0] = 0xffffffffu, s.ends[1] = 0u;
  }
  __syncthreads();
  if (s.first[ROW_PARTS] == 0) return key_min;
  uint32_t lowest = 0xffffffffu, highest = 0u;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int part = 2 * wave + h, first = s.first[part], n = s.first[part + 1] - first;
    for (int k = lane; k < n; k += HAL_WAVE) {
      const uint32_t key = keys[part * share + k];
      if (first + k < FILT_STAGED) s.staged[first + k] = key;
      lowest = min(lowest, key), highest = max(highest, key);
    }
  }
#pragma unroll
  for (int off = HAL_WAVE / 2; off; off >>= 1) lowest = min(lowest, (uint32_t)__shfl_xor((int)lowest, off, HAL_WAVE)), highest = max(highest, (uint32_t)__shfl_xor((int)highest, off, HAL_WAVE));
  if (lane == 0) atomicMin(&s.ends[0], lowest), atomicMax(&s.ends[1], highest);
  __syncthreads();
  lowest = s.ends[0];
  const uint32_t range = s.ends[1] - lowest;
#pragma unroll 1
  for (int w = 0; w < 2; ++w) {
    if (!f.on[w] || f.bin[w] != f.list) continue;
    const unsigned long long target = f.target[w] - f.before[w];
    uint32_t prefix = 0u;
    unsigned long long above = 0ull;
    int bits = range ? 32 - __builtin_clz(range) : 0;
#pragma unroll 1
    while (bits > 0) {
      const int take = bits < FILT_DIGIT ? bits : FILT_DIGIT, shift = bits - take;
      s.bins[tid] = 0ull;
      if (tid == 0) s.bin = 0u, s.above = above;
      __syncthreads();
      filt_each(s, keys, V, [&](uint32_t key, int) {
        const uint32_t rel = key - lowest;
        if (((unsigned long long)rel >> bits) != prefix) return;
        atomicAdd(&s.bins[(rel >> shift) & ((1u << take) - 1u)], w == 1 ? filt_fixed(expf(key_value(key) - r.m)) : 1ull);
      });
      __syncthreads();
      // in descending order
      const unsigned long long own = s.bins[tid], higher = above + block_suffix_u64(own, s.tmp);
      if (higher < target && higher + own >= target) s.bin = tid, s.above = higher;
      __syncthreads();
      prefix = (prefix << take) | s.bin;
      above = s.above;
      bits = shift;
      __syncthreads();
    }
    key_min = max(key_min, lowest + prefix);
  }
  return key_min;
}

// The first search of late rows: the smallest key that top-k keeps, and the mass of those that it keeps.
__global__ void __launch_bounds__(PICK_THREADS)
filt_find_kernel(FiltRow* __restrict__ rows, const unsigned long long* __restrict__ hists, FiltParams params, int V, const float* __restrict__ parts,
                 const uint32_t* __restrict__ lists) {
  __shared__ FiltSearch s;
  const int row = blockIdx.x, tid = threadIdx.x;
  if (!(filt_flags(params, V, row) & FILT_P_LATE)) return;
  const unsigned long long* hist = hists + (size_t)row * 2 * FILT_BINS;
  const uint32_t* keys = lists + (size_t)row * V;
  const FiltRow r = rows[row];
  const int lane = tid % HAL_WAVE, listed = lane < ROW_PARTS ? __float_as_int(parts[((size_t)row * ROW_PARTS + lane) * 4 + 3]) : 0;
  const FiltPlace f = filt_place(hist, params, V, row, r, 0);
  const uint32_t key_min = filt_search(s, f, r, listed, keys, V, 0);
  unsigned long long kept = tid < f.bin[0] ? hist[FILT_BINS + tid] : 0ull;
  filt_each(s, keys, V, [&](uint32_t key, int) { kept += key >= key_min ? filt_fixed(expf(key_value(key) - r.m)) : 0ull; });
  kept += block_suffix_u64(kept, s.tmp);  // (thread 0: of all)
  if (tid == 0) rows[row].key_min = key_min, rows[row].kept_by_k = kept;
}

__device__ __forceinline__ float kept_mass_of(float v, float T, uint32_t key_min, float m, float mp, float& z) {
  const uint32_t key = sort_key(clean_logit(v) / T);
  if (key < key_min) return 0.f;
  z = key_value(key);
  const float e = expf(z - m);
  return e >= mp ? e : 0.f;
}

// The threshold, what every share keeps, and the draw, a block a row: the share in which the running kept mass passes u * (kept mass), then the walk
// through that share as four waves would walk it, a quarter each, 64 logits at a time.  Sixteen waves make the masses and the running sums inside
// every 64 and leave them in LDS; the sums over a quarter's runs of 64 and the runs' order are then a few additions.
#define PICK_QUARTERS 4
__global__ void __launch_bounds__(PICK_THREADS)
filt_pick_kernel(const float* __restrict__ logits, int ld, int V, FiltParams params, const FiltRow* __restrict__ rows, int any_late,
                 const unsigned long long* __restrict__ hists, const float* __restrict__ parts, const float* __restrict__ kept,
                 const uint32_t* __restrict__ lists, const uint64_t* __restrict__ seeds, const int* __restrict__ draw_index,
                 int* __restrict__ out_token, float* __restrict__ out_logprob) {
  constexpr int RUNS = 16, WAVES = PICK_THREADS / HAL_WAVE, MINE = RUNS * PICK_QUARTERS / WAVES;  // runs in LDS a quarter; of a wave
  __shared__ float e_s[PICK_QUARTERS][RUNS][HAL_WAVE], z_s[PICK_QUARTERS][RUNS][HAL_WAVE], inc_s[PICK_QUARTERS][RUNS][HAL_WAVE];
  __shared__ float quarter_mass[PICK_QUARTERS], kept_s[ROW_PARTS];
  __shared__ FiltSearch search;
  const int row = blockIdx.x, tid = threadIdx.x;
  const int lane = tid % HAL_WAVE, wave = __builtin_amdgcn_readfirstlane(tid / HAL_WAVE);
  const FiltRow r = rows[row];
  // (what is read here does not wait for the search)
  typedef __attribute__((ext_vector_type(4), aligned(4))) float any4;  // (the room's parts begin at any float)
  any4 of_part = {0.f, 0.f, 0.f, 0.f};
  if (lane < ROW_PARTS) of_part = *(const any4*)(parts + ((size_t)row * ROW_PARTS + lane) * 4);
  const float for_sure = kept[(size_t)row * ROW_PARTS + 2 * wave + lane % 2];
  const uint64_t seed = seeds[row];
  const uint32_t drawn = (uint32_t)draw_index[row];
  const int flags = filt_flags(params, V, row);
  const float total = wave_sum(of_part.z);
  if (flags == FILT_GREEDY) {
    if (tid == 0) {
      out_token[row] = r.best < V ? r.best : 0;
      out_logprob[row] = -logf(total);
    }
    return;
  }
  const int late = any_late && (flags & FILT_P_LATE) ? 1 : 0;
  const uint32_t* keys = lists + (size_t)row * V;
  const FiltPlace f = filt_place(hists + (size_t)row * 2 * FILT_BINS, params, V, row, r, late);
  const uint32_t key_min = filt_search(search, f, r, __float_as_int(of_part.w), keys, V, late);
  {
    const float mp = params.min_p[row];
    unsigned long long listed[2] = {0ull, 0ull};
    filt_each(search, keys, V, [&](uint32_t key, int part) {
      if (key < key_min) return;
      const float e = expf(key_value(key) - r.m);
      if (e >= mp) listed[part % 2] += filt_fixed(e);
    });
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int off = HAL_WAVE / 2; off; off >>= 1) {
        const uint32_t lo = __shfl_xor((uint32_t)listed[h], off, HAL_WAVE), hi = __shfl_xor((uint32_t)(listed[h] >> 32), off, HAL_WAVE);
        listed[h] += ((unsigned long long)hi << 32) | lo;
      }
      if (lane == h) kept_s[2 * wave + h] = for_sure + (float)listed[h] * (1.0f / 1099511627776.0f);
    }
  }
  __syncthreads();
  auto running = [&](float v) {
    float inc = v;
#pragma unroll
    for (int off = 1; off < HAL_WAVE; off <<= 1) {
      const float up = __shfl_up(inc, off, HAL_WAVE);
      if (lane >= off) inc += up;
    }
    return inc;
  };
  const float mass = lane < ROW_PARTS ? kept_s[lane] : 0.f;
  const float incl = running(mass);
  const float kept_mass = __shfl(incl, HAL_WAVE - 1, HAL_WAVE);
  const float target = uniform_draw(seed, drawn) * kept_mass;
  const unsigned long long some = __builtin_amdgcn_ballot_w64(mass > 0.f);
  const unsigned long long hit = __builtin_amdgcn_ballot_w64(mass > 0.f && incl > target);
  // (the largest key is always kept, so some share holds something)
  const int part = hit ? __builtin_ctzll(hit) : (some ? 63 - __builtin_clzll(some) : 0);
  const float before_part = __shfl(incl - mass, part, HAL_WAVE);

  const float* x = logits + (size_t)row * ld;
  const int share = part_share(V);
  const int p_begin = part * share, p_end = p_begin + share < V ? p_begin + share : V;
  const int run_len = ((p_end - p_begin + PICK_QUARTERS - 1) / PICK_QUARTERS + HAL_WAVE - 1) / HAL_WAVE * HAL_WAVE;
  const float T = params.temperature[row], mp = params.min_p[row];
  auto quarter_end = [&](int q) { return p_begin + (q + 1) * run_len < p_end ? p_begin + (q + 1) * run_len : p_end; };
  {  // (a wave's runs are all of one quarter)
    const int q = wave * MINE / RUNS, run0 = wave * MINE % RUNS, from = p_begin + q * run_len, end = quarter_end(q);
    float held[MINE];
#pragma unroll
    for (int u = 0; u < MINE; ++u) {
      const int i = from + (run0 + u) * HAL_WAVE + lane;
      held[u] = i < end ? x[i] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < MINE; ++u) {
      float z = 0.f;
      const float e = from + (run0 + u) * HAL_WAVE + lane < end ? kept_mass_of(held[u], T, key_min, r.m, mp, z) : 0.f;
      e_s[q][run0 + u][lane] = e, z_s[q][run0 + u][lane] = z, inc_s[q][run0 + u][lane] = running(e);
    }
  }
  __syncthreads();
  // (a wave past the quarters begins at the share's end or behind it and has no runs)
  const int begin = p_begin + wave * run_len, end = quarter_end(wave);
  const int runs = end > begin ? (end - begin + HAL_WAVE - 1) / HAL_WAVE : 0;
  float mine = 0.f, zz = 0.f;
  for (int u = 0; u < runs && u < RUNS; ++u) mine += e_s[wave][u][lane];
  for (int i = begin + RUNS * HAL_WAVE + lane; i < end; i += HAL_WAVE) mine += kept_mass_of(x[i], T, key_min, r.m, mp, zz);
  const float wave_mass = wave_sum(mine);
  if (lane == 0 && wave < PICK_QUARTERS) quarter_mass[wave] = wave_mass;
  __syncthreads();
  float before = before_part;
  int pick = -1, last = -1;
  for (int w = 0; w < PICK_QUARTERS; ++w) {
    if (quarter_mass[w] > 0.f) last = w;
    if (pick < 0 && quarter_mass[w] > 0.f && before + quarter_mass[w] > target) pick = w;
    if (pick < 0) before += quarter_mass[w];
  }
  if (pick < 0) {  // rounding left the target at the very end: the last quarter that holds anything
    pick = last < 0 ? 0 : last;
    before = before_part;
    for (int w = 0; w < pick; ++w) before += quarter_mass[w];
  }
  if (wave != pick) return;
  float run = before;
  int tok = -1, last_kept = -1;
  float z_tok = 0.f, z_last = 0.f;
  for (int u = 0; u < runs && tok < 0; ++u) {
    const int i0 = begin + u * HAL_WAVE;
    float z = 0.f, e = 0.f, inc;
    if (u < RUNS) {
      e = e_s[wave][u][lane], z = z_s[wave][u][lane], inc = inc_s[wave][u][lane];
    } else {
      if (i0 + lane < end) e = kept_mass_of(x[i0 + lane], T, key_min, r.m, mp, z);
      inc = running(e);
    }
    const unsigned long long kept_lanes = __builtin_amdgcn_ballot_w64(e > 0.f);
    const unsigned long long found = __builtin_amdgcn_ballot_w64(e > 0.f && run + inc > target);
    if (kept_lanes) {
      const int hi = 63 - __builtin_clzll(kept_lanes);
      last_kept = i0 + hi;
      z_last = __shfl(z, hi, HAL_WAVE);
    }
    if (found) {
      const int lo = __builtin_ctzll(found);
      tok = i0 + lo;
      z_tok = __shfl(z, lo, HAL_WAVE);
    }
    run += __shfl(inc, HAL_WAVE - 1, HAL_WAVE);
  }
  if (tok < 0) {
    tok = last_kept >= 0 ? last_kept : (r.best < V ? r.best : 0);
    z_tok = last_kept >= 0 ? z_last : r.m;
  }
  if (lane == 0) {
    out_token[row] = tok;
    out_logprob[row] = z_tok - r.m - logf(total);
  }
}

static int launch_row_parts(const float* logits, int ld, int n_rows, int V, const float* temperature,
                            const int* top_k, const uint64_t* seeds, const int* draw_index,
                            float* parts, int* out_token, float* out_logprob, hipStream_t stream) {
  hipLaunchKernelGGL(row_part_kernel, dim3(ROW_PARTS, n_rows), dim3(PART_THREADS), 0, stream, logits,
                     ld, V, temperature, top_k, parts);
  HAL_LAUNCH_CHECK();
  hipLaunchKernelGGL(row_join_kernel, dim3(n_rows), dim3(PART_THREADS), 0, stream, logits, ld, V,
                     parts, temperature, top_k, seeds, draw_index, out_token, out_logprob);
  HAL_LAUNCH_CHECK();
  return 0;
}

// Greedy decoding of every row: first index of the maximum and its log-probability under
// softmax(logits).  `parts` has room for n_rows * 32 * 4 floats.
extern "C" int hal_sample_greedy(const float* logits, int ld, int n_rows, int V, float* parts,
                                 int* out_token, float* out_logprob, hipStream_t stream) {
  HAL_REQUIRE(n_rows >= 0 && V > 0 && ld >= V, "hal_sample_greedy: bad sizes rows=%d V=%d ld=%d",
              n_rows, V, ld);
  HAL_REQUIRE(n_rows <= 65535, "hal_sample_greedy: %d rows exceed the grid limit", n_rows);
  if (n_rows == 0) return 0;
  HAL_REQUIRE(parts != nullptr, "hal_sample_greedy: no room for the partial results");
  return launch_row_parts(logits, ld, n_rows, V, nullptr, nullptr, nullptr, nullptr, parts, out_token,
                          out_logprob, stream);
}

// ---- greedy decoding without any allocation ---------------------------------------------
// The partial results of hal_sample_greedy in memory that the library itself holds: one
// array per GPU, there from the moment the library is loaded until the process ends.
#define STATIC_GREEDY_ROWS 1024
static __device__ __align__(256) float scratch[STATIC_GREEDY_ROWS * ROW_PARTS * 4];  // 512 KiB

#define STATIC_MAX_DEVICES 64
static float* g_scratch_of_device[STATIC_MAX_DEVICES];  // the array's address on each GPU
static std::mutex g_scratch_lock;

// The address of this GPU's copy of `scratch`.  The array's name means nothing to host
// code; the address is asked for once per device, with that device current.
static int scratch_of_current_device(float** out) {
  int dev = -1;
  HAL_CHECK_HIP(hipGetDevice(&dev));
  HAL_REQUIRE(dev >= 0 && dev < STATIC_MAX_DEVICES, "hal_sample_greedy_static: device %d of at most %d",
              dev, STATIC_MAX_DEVICES);
  std::lock_guard<std::mutex> hold(g_scratch_lock);
  if (g_scratch_of_device[dev] == nullptr) {
    float* ptr = nullptr;
    HAL_CHECK_HIP(hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)));
    HAL_REQUIRE(ptr != nullptr, "hal_sample_greedy_static: the scratch array has no address on device %d", dev);
    g_scratch_of_device[dev] = ptr;
  }
  *out = g_scratch_of_device[dev];
  return 0;
}

extern "C" int hal_sample_greedy_static_max_rows() { return STATIC_GREEDY_ROWS; }

// hal_sample_greedy for callers that cannot allocate: the partial results go to the
// library's own array on the current GPU instead of to `parts`.  Calls no hipMalloc, no
// hipFree and no routine that allocates; launches the same two kernels.  Nothing in the
// array has to start at zero: the first kernel writes every word that the second reads (32
// shares of every row), so what an earlier call left does no harm.  All calls on a GPU
// share the array: two calls whose kernels may overlap (different streams, different host
// threads) race; calls on one stream follow each other and are safe.
extern "C" int hal_sample_greedy_static(const float* logits, int ld, int n_rows, int V,
                                        int* out_token, float* out_logprob, hipStream_t stream) {
  HAL_REQUIRE(n_rows >= 0 && V > 0 && ld >= V, "hal_sample_greedy_static: bad sizes rows=%d V=%d ld=%d",
              n_rows, V, ld);
  HAL_REQUIRE(n_rows <= STATIC_GREEDY_ROWS,
              "hal_sample_greedy_static: %d rows, the scratch array holds the partial results of at most %d",
              n_rows, STATIC_GREEDY_ROWS);
  if (n_rows == 0) return 0;
  HAL_REQUIRE(logits && out_token && out_logprob, "hal_sample_greedy_static: arguments missing");
  float* parts = nullptr;
  if (int rc = scratch_of_current_device(&parts)) return rc;
  return launch_row_parts(logits, ld, n_rows, V, nullptr, nullptr, nullptr, nullptr, parts, out_token,
                          out_logprob, stream);
}

// Rows without filters (no top-k beyond 1, no top-p, no min-p): greedy rows (temperature 0
// or top_k 1) and draws from the whole temperature-scaled distribution, as hal_sample gives
// them.  `parts` has room for n_rows * 32 * 4 floats.
extern "C" int hal_sample_unfiltered(const float* logits, int ld, int n_rows, int V,
                                     const float* temperature, const int* top_k,
                                     const uint64_t* seeds, const int* draw_index, float* parts,
                                     int* out_token, float* out_logprob, hipStream_t stream) {
  HAL_REQUIRE(n_rows >= 0 && V > 0 && ld >= V, "hal_sample_unfiltered: bad sizes rows=%d V=%d ld=%d",
              n_rows, V, ld);
  HAL_REQUIRE(n_rows <= 65535, "hal_sample_unfiltered: %d rows exceed the grid limit", n_rows);
  if (n_rows == 0) return 0;
  HAL_REQUIRE(parts && temperature && top_k && seeds && draw_index,
              "hal_sample_unfiltered: arguments missing");
  return launch_row_parts(logits, ld, n_rows, V, temperature, top_k, seeds, draw_index, parts,
                          out_token, out_logprob, stream);
}

// Rows with filters (and greedy or unfiltered ones among them), every row spread over 32
// blocks in every pass.  `any_late`: some row has top-k, top-p and min-p all at once (its
// second search costs two launches more; a wrong 0 leaves such a row without top-p).
// Room: `parts` n_rows * 32 * 4 floats, `kept` n_rows * 32 floats, `state` n_rows * 6
// words, `hist` n_rows * 2 * 256 64-bit words, `lists` n_rows * V words.
extern "C" int hal_sample_spread(const float* logits, int ld, int n_rows, int V,
                                 const float* temperature, const int* top_k, const float* top_p,
                                 const float* min_p, const uint64_t* seeds, const int* draw_index,
                                 float* parts, float* kept, void* state, void* hist, uint32_t* lists, int any_late,
                                 int* out_token, float* out_logprob, hipStream_t stream) {
  HAL_REQUIRE(n_rows >= 0 && V > 0 && ld >= V, "hal_sample_spread: bad sizes rows=%d V=%d ld=%d",
              n_rows, V, ld);
  HAL_REQUIRE(n_rows <= 65535, "hal_sample_spread: %d rows exceed the grid limit", n_rows);
  if (n_rows == 0) return 0;
  HAL_REQUIRE(temperature && top_k && top_p && min_p && seeds && draw_index && parts && kept &&
                  state && hist && lists && ((uintptr_t)state % 8) == 0 && ((uintptr_t)hist % 8) == 0,
              "hal_sample_spread: arguments missing");
  FiltRow* rows = (FiltRow*)state;
  unsigned long long* h = (unsigned long long*)hist;
  const FiltParams params = {temperature, top_p, min_p, top_k};
  const dim3 shares(ROW_PARTS, n_rows);
  hipLaunchKernelGGL(filt_max_kernel, shares, dim3(PART_THREADS), 0, stream, logits, ld, V, params, parts, h);
  hipLaunchKernelGGL(filt_coarse_kernel, shares, dim3(PART_THREADS), 0, stream, logits, ld, V, params, parts, rows, h);
  hipLaunchKernelGGL(filt_list_kernel, shares, dim3(PART_THREADS), 0, stream, logits, ld, V, params, rows, 0, h, parts, kept, lists);
  if (any_late) {  // rows with top-k, top-p and min-p all at once: what top-k keeps, and the second search's list
    hipLaunchKernelGGL(filt_find_kernel, dim3(n_rows), dim3(PICK_THREADS), 0, stream, rows, h, params, V, parts, lists);
    hipLaunchKernelGGL(filt_list_kernel, shares, dim3(PART_THREADS), 0, stream, logits, ld, V, params, rows, 1, h, parts, kept, lists);
  }
  hipLaunchKernelGGL(filt_pick_kernel, dim3(n_rows), dim3(PICK_THREADS), 0, stream, logits, ld, V, params, rows, any_late, h, parts,
                     kept, lists, seeds, draw_index, out_token, out_logprob);
  HAL_LAUNCH_CHECK();
  return 0;
}

// ---- a step's rows as the host has them -------------------------------------------------
// A row's parameters as they lie in one buffer of 7 n words, so that one copy brings a step's: seeds (64 bits), temperature, top_p,
// min_p (float32), top_k, draw index.  Returns what holds for all rows, which decides how they are sampled; -1: a draw index beyond 32 bits.  (As two dozen numpy
// calls on 64 rows this was 25 of the 50 us that the host had to do before a step's first launch.)
enum { SAMPLE_ALL_GREEDY = 1, SAMPLE_UNFILTERED = 2, SAMPLE_LATE = 4 };
extern "C" int hal_sample_pack(const double* temperature, const double* top_p, const double* min_p, const long long* top_k,
                               const long long* seeds, const long long* draws, int n, int V, int* words) {
  bool all_greedy = true, unfiltered = true, late = false;
  float* f = (float*)(words + 2 * (size_t)n);
  int* w = words + 5 * (size_t)n;
  for (int r = 0; r < n; ++r) {
    if (draws[r] != (int)draws[r]) return -1;
    const bool greedy = temperature[r] == 0 || top_k[r] == 1;
    const bool by_k = top_k[r] > 0 && top_k[r] < V, by_p = top_p[r] < 1.0, by_min = min_p[r] > 0.0;
    all_greedy &= greedy;
    unfiltered &= greedy || !(by_k || by_p || by_min);
    // (top-k, top-p and min-p all at once: top-p then refers to what top-k kept, two searches one after the other)
    late |= !greedy && by_k && by_p && by_min;
    memcpy(words + 2 * (size_t)r, &seeds[r], 8);
    f[r] = greedy ? 0.f : (float)temperature[r], f[n + r] = (float)top_p[r], f[2 * (size_t)n + r] = (float)min_p[r];
    w[r] = greedy ? 1 : (int)(top_k[r] < 0x7fffffffll ? top_k[r] : 0x7fffffffll), w[n + r] = (int)draws[r];
  }
  return (all_greedy ? SAMPLE_ALL_GREEDY : 0) | (unfiltered ? SAMPLE_UNFILTERED : 0) | (late ? SAMPLE_LATE : 0);
}

// The words of room a row: a histogram and its state (64-bit words, so they come first in the room), its blocks' partial results and kept
// masses, a list as long as the row; partial results alone where no row is filtered.
extern "C" long long hal_sample_row_words(int flags, int V) {
  if (flags & (SAMPLE_ALL_GREEDY | SAMPLE_UNFILTERED)) return ROW_PARTS * 4;
  return 4 * FILT_BINS + 6 + ROW_PARTS * 4 + ROW_PARTS + (long long)V;
}

// Samples n rows by such a buffer on the GPU.  `flags`: what hal_sample_pack returned.  `room`: hal_sample_row_words for each of the rows that go
// over it at a time, from a multiple of 8 bytes on: `at_once` of those with filters, all others.  `out`: n tokens, then n log-probabilities.
extern "C" int hal_sample_packed(const float* logits, int ld, int n, int V, const int* packed, int flags, int* room, int at_once, int* out,
                                 hipStream_t stream) {
  HAL_REQUIRE(n >= 0 && V > 0 && ld >= V && at_once > 0, "hal_sample_packed: bad sizes rows=%d V=%d ld=%d, %d at once", n, V, ld, at_once);
  if (n == 0) return 0;
  HAL_REQUIRE(logits && packed && room && out && (uintptr_t)packed % 8 == 0 && (uintptr_t)room % 8 == 0, "hal_sample_packed: arguments missing");
  const uint64_t* seeds = (const uint64_t*)packed;
  const float *temperature = (const float*)(packed + 2 * (size_t)n), *top_p = temperature + n, *min_p = top_p + n;
  const int *top_k = packed + 5 * (size_t)n, *draws = top_k + n;
  float* logprobs = (float*)(out + n);
  if (flags & SAMPLE_ALL_GREEDY) return hal_sample_greedy(logits, ld, n, V, (float*)room, out, logprobs, stream);
  if (flags & SAMPLE_UNFILTERED) return hal_sample_unfiltered(logits, ld, n, V, temperature, top_k, seeds, draws, (float*)room, out, logprobs, stream);
  int* hist = room;
  int* state = hist + (size_t)at_once * 4 * FILT_BINS;
  float* parts = (float*)(state + (size_t)at_once * 6);
  float* kept = parts + (size_t)at_once * ROW_PARTS * 4;
  uint32_t* lists = (uint32_t*)(kept + (size_t)at_once * ROW_PARTS);
  for (int r = 0; r < n; r += at_once) {
    if (hal_sample_spread(logits + (size_t)r * ld, ld, n - r < at_once ? n - r : at_once, V, temperature + r, top_k + r, top_p + r, min_p + r, seeds + r,
                          draws + r, parts, kept, state, hist, lists, flags & SAMPLE_LATE ? 1 : 0, out + r, logprobs + r, stream))
      return 1;
  }
  return 0;
}
