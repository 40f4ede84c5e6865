// Token sampling on the logits rows of the lm_head: temperature, top-k, top-p (nucleus) filtering,
// the filtered distribution, the probability of a drafted token, and an inverse-CDF draw -- the
// Sampler of phase0/specsample.py:36-107 (dist, sample_logits, accept's residual draw) on the GPU.
//
// Definition, per logits row x[V] (bf16):
//   z_v = x_v / max(temp, 1e-6) (fp32);
//   top-k (0 < k < V): keep z_v >= the k-th largest z (counted with multiplicity);
//   weights w_v = floor(2^40 * e^(z_v - max z)) as exact integers, 0 for masked tokens, with e^d from
//     samp_exp below (fixed fp64 operations, so every build computes the same integers);
//   top-p (0 < p < 1): with the kept tokens ordered by (z desc, id asc; -0 and +0 are one value),
//     keep a token iff the weight of the tokens before it is <= floor(p * W) (W = the sum of the
//     kept weights, p * W one fp64 product);
//   the distribution is w' / W' over what is kept;
//   a draw with uniform u in [0, 1) is the first id v (ascending) whose inclusive prefix of w'' exceeds
//     floor(u * W''), where w'' is w' with the drafted token's weight removed when a draft is given
//     (the residual of the speculative-sampling rule); when nothing is left (W'' == 0) the draw is the
//     first id of maximal w'.
// Integer weights make every sum independent of the reduction order, so a row's results do not depend
// on the launch shape.  Greedy rows (temp <= 0) draw the first id of maximal x.
#include <algorithm>
#include <math.h>

#include "common.h"

namespace flyai {

constexpr int kSampThreads = 1024;
constexpr int kSampWaves = kSampThreads / 64;

// order-preserving key of a finite fp32 value: larger value <=> larger key (-0 keyed as +0)
__device__ __forceinline__ uint32_t f32_key(float z) {
  const uint32_t u = z == 0.f ? 0u : __float_as_uint(z);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float key_f32(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// floor(2^40 * e^d) for d <= 0, by Cody-Waite range reduction (d = k ln2 + r, |r| <= ln2 / 2, ln2 split
// into a 32-bit head, so k * head is exact, and a tail) and the degree-13 Taylor polynomial of e^r
// (truncation error below 5e-18), each fp64 operation rounded on its own (no fused multiply-add):
// within one unit of the exact floor.  d below -27.75 gives 0 (2^40 e^d < 1 there).
__device__ __forceinline__ uint64_t samp_weight(float z, float zmax) {
#pragma clang fp contract(off)
  const double d = (double)z - (double)zmax;
  if (!(d >= -27.75)) return 0;
  const double k = rint(d * 0x1.71547652b82fep+0);
  const double r = (d - k * 0x1.62e42feep-1) - k * 0x1.a39ef35793c76p-33;
  double p = 0x1.6124613a86d09p-33;
  p = p * r + 0x1.1eed8eff8d898p-29;
  p = p * r + 0x1.ae64567f544e4p-26;
  p = p * r + 0x1.27e4fb7789f5cp-22;
  p = p * r + 0x1.71de3a556c734p-19;
  p = p * r + 0x1.a01a01a01a01ap-16;
  p = p * r + 0x1.a01a01a01a01ap-13;
  p = p * r + 0x1.6c16c16c16c17p-10;
  p = p * r + 0x1.1111111111111p-7;
  p = p * r + 0x1.5555555555555p-5;
  p = p * r + 0x1.5555555555555p-3;
  p = p * r + 0x1p-1;
  p = p * r + 1.0;
  p = p * r + 1.0;
  return (uint64_t)floor(ldexp(p, (int)k + 40));
}

// block sums over the 1024 threads through LDS (one slot per wave)
template <class T>
__device__ __forceinline__ T block_sum(T v, T* red) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  T s = 0;
#pragma unroll
  for (int w = 0; w < kSampWaves; ++w) s += red[w];
  return s;
}

__device__ __forceinline__ uint32_t block_max_u32(uint32_t v, uint32_t* red) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v = max(v, (uint32_t)__shfl_xor((int)v, o, 64));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  uint32_t m = 0;
#pragma unroll
  for (int w = 0; w < kSampWaves; ++w) m = max(m, red[w]);
  return m;
}

struct SampShared {
  uint64_t hist[256];
  uint64_t red64[kSampWaves];
  uint32_t red32[kSampWaves];
  uint64_t scan[kSampThreads];
  uint64_t sel_above;  // weight (or count) above the selected bin
  uint32_t sel_prefix;
  int sel_found;
};

// Radix selection over the 32-bit keys of the kept tokens, 8 bits per pass from the top: the key of
// the token where the running total of `mass` (counts for top-k, weights for top-p), taken in
// descending key order, first exceeds `limit`.  Returns the key; *above gets the total mass of the
// kept tokens with larger keys.  If the total never exceeds limit, returns 0 with *above = total.
template <class KeyOf, class MassOf>
__device__ uint32_t radix_select(int V, KeyOf key_of, MassOf mass_of, uint64_t limit, uint64_t* above, SampShared& sh) {
  uint32_t prefix = 0;
  uint64_t run = 0;  // mass of tokens above the current prefix's range
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int b = threadIdx.x; b < 256; b += kSampThreads) sh.hist[b] = 0;
    __syncthreads();
    const uint32_t hi_mask = shift == 24 ? 0u : (0xffffffffu << (shift + 8));
    for (int v = threadIdx.x; v < V; v += kSampThreads) {
      uint32_t k;
      uint64_t m;
      if (!key_of(v, &k)) continue;
      if ((k & hi_mask) != (prefix & hi_mask)) continue;
      m = mass_of(v);
      if (m) atomicAdd((unsigned long long*)&sh.hist[(k >> shift) & 0xff], (unsigned long long)m);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      int found = -1;
      uint64_t r = run;
      for (int b = 255; b >= 0; --b) {
        if (r + sh.hist[b] > limit) {
          found = b;
          break;
        }
        r += sh.hist[b];
      }
      sh.sel_found = found;
      sh.sel_above = r;
      sh.sel_prefix = found >= 0 ? (prefix | ((uint32_t)found << shift)) : 0u;
    }
    __syncthreads();
    if (sh.sel_found < 0) {
      *above = sh.sel_above;
      return 0u;
    }
    prefix = sh.sel_prefix;
    run = sh.sel_above;
  }
  *above = run;
  return prefix;
}

// One row by one kSampThreads workgroup, for any logits (NaN, infinities, denormal quotients) and with no
// workspace: every pass reads the row again.  Inlined into sample_rows_kernel: a function call there takes 128
// registers and scratch memory instead of 66 and none (512 greedy rows of 512 logits 32 us instead of 4.9).
__device__ __forceinline__ void sample_row_general(SampShared& sh, int row, const uint16_t* __restrict__ logits, int V, float temp,
                                   int top_k, float top_p, const int32_t* __restrict__ draft,
                                   const double* __restrict__ u, float* __restrict__ p_draft,
                                   int32_t* __restrict__ draw, float* __restrict__ probs) {
  const uint16_t* x = logits + (size_t)row * V;
  const int tid = threadIdx.x;
  const int d = draft ? draft[row] : -1;
  const int C = (V + kSampThreads - 1) / kSampThreads;  // ids of thread t for ordered scans: [tC, tC+C)

  if (!(temp > 0.f)) {  // greedy: the first id of maximal x
    uint32_t best = 0;
    for (int v = tid; v < V; v += kSampThreads) best = max(best, f32_key(bf2f(x[v])));
    best = block_max_u32(best, sh.red32);
    int first = V;
    for (int v = tid; v < V; v += kSampThreads)
      if (f32_key(bf2f(x[v])) == best) { first = v; break; }
    // smallest id among the threads' first hits
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) first = min(first, __shfl_xor(first, o, 64));
    __syncthreads();
    if ((tid & 63) == 0) sh.red32[tid >> 6] = (uint32_t)first;
    __syncthreads();
    int arg = V;
    for (int w = 0; w < kSampWaves; ++w) arg = min(arg, (int)sh.red32[w]);
    if (tid == 0) {
      if (draw) draw[row] = arg;
      if (p_draft) p_draft[row] = (d == arg) ? 1.f : 0.f;
    }
    if (probs)
      for (int v = tid; v < V; v += kSampThreads) probs[(size_t)row * V + v] = v == arg ? 1.f : 0.f;
    return;
  }
  const float tdiv = fmaxf(temp, 1e-6f);
  auto zof = [&](int v) __attribute__((always_inline)) { return __fdiv_rn(bf2f(x[v]), tdiv); };

  // top-k: the k-th largest key, counted with multiplicity
  uint32_t kth = 0;
  if (top_k > 0 && top_k < V) {
    uint64_t above = 0;
    kth = radix_select(V, [&](int v, uint32_t* k) { *k = f32_key(zof(v)); return true; },
                       [&](int) { return (uint64_t)1; }, (uint64_t)(top_k - 1), &above, sh);
  }
  auto kept_k = [&](int v, uint32_t* k) __attribute__((always_inline)) {
    *k = f32_key(zof(v));
    return *k >= kth;
  };
  // max z, then the weights' total
  uint32_t mkey = 0;
  for (int v = tid; v < V; v += kSampThreads) mkey = max(mkey, f32_key(zof(v)));
  mkey = block_max_u32(mkey, sh.red32);
  const float zmax = key_f32(mkey);
  uint64_t wsum = 0;
  for (int v = tid; v < V; v += kSampThreads) {
    uint32_t k;
    if (kept_k(v, &k)) wsum += samp_weight(zof(v), zmax);
  }
  const uint64_t W = block_sum(wsum, sh.red64);

  // top-p: the boundary key and how many of its ties (in id order) are kept
  uint32_t pkey = 0;
  uint64_t tie_keep = ~0ull;  // ties at pkey kept (all when top-p is off)
  if (top_p > 0.f && top_p < 1.f) {
    const uint64_t T = (uint64_t)floor((double)top_p * (double)W);
    // the boundary: the first token (descending order) whose inclusive running weight exceeds T; every
    // token above it is kept (its preceding weight is <= T), every token below it is dropped
    uint64_t above = 0;
    pkey = radix_select(V, kept_k, [&](int v) { return samp_weight(zof(v), zmax); }, T, &above, sh);
    if (pkey != 0u) {
      // tie j (0-based, id order) of the boundary value is kept iff above + j * wb <= T (tie 0 always is)
      const uint64_t wb = samp_weight(key_f32(pkey), zmax);
      tie_keep = wb == 0 ? ~0ull : (T - above) / wb + 1;
    }
  }
  // ordered pass 1: per-thread counts of boundary ties (for tie ranks) and kept weights
  const int v0 = tid * C, v1 = min(V, v0 + C);
  uint64_t my_ties = 0;
  if (pkey != 0u)
    for (int v = v0; v < v1; ++v) {
      uint32_t k;
      if (kept_k(v, &k) && k == pkey) ++my_ties;
    }
  __syncthreads();
  sh.scan[tid] = my_ties;
  __syncthreads();
  // exclusive prefix of tie counts (thread 0 serial scan of 1024 values; a small fraction of the work)
  if (tid == 0) {
    uint64_t acc = 0;
    for (int t = 0; t < kSampThreads; ++t) {
      const uint64_t c = sh.scan[t];
      sh.scan[t] = acc;
      acc += c;
    }
  }
  __syncthreads();
  const uint64_t tie_base = sh.scan[tid];
  auto final_w = [&](int v, uint64_t* tie_rank) __attribute__((always_inline)) -> uint64_t {
    uint32_t k;
    if (!kept_k(v, &k)) return 0;
    if (pkey != 0u) {
      if (k < pkey) return 0;
      if (k == pkey) {
        const bool keep = *tie_rank < tie_keep;
        ++*tie_rank;
        if (!keep) return 0;
      }
    }
    return samp_weight(zof(v), zmax);
  };
  // ordered pass 2: kept weights per thread (W'), the draft's weight, the first maximal weight
  uint64_t my_w = 0, wd = 0, best_w = 0;
  int best_v = V;
  {
    uint64_t tr = tie_base;
    for (int v = v0; v < v1; ++v) {
      const uint64_t w = final_w(v, &tr);
      my_w += w;
      if (v == d) wd = w;
      if (w > best_w) { best_w = w; best_v = v; }
    }
  }
  const uint64_t Wk = block_sum(my_w, sh.red64);
  const uint64_t Wd = block_sum(wd, sh.red64);
  if (tid == 0 && p_draft) p_draft[row] = (d >= 0 && Wk > 0) ? (float)((double)Wd / (double)Wk) : 0.f;
  if (probs) {
    uint64_t tr = tie_base;
    for (int v = v0; v < v1; ++v) {
      const uint64_t w = final_w(v, &tr);
      probs[(size_t)row * V + v] = Wk > 0 ? (float)((double)w / (double)Wk) : 0.f;
    }
  }
  if (!(draw && u)) return;
  // the draw: residual weights (draft removed), inverse CDF in id order
  const uint64_t my_r = my_w - wd;
  __syncthreads();
  sh.scan[tid] = my_r;
  __syncthreads();
  if (tid == 0) {
    uint64_t acc = 0;
    for (int t = 0; t < kSampThreads; ++t) {
      const uint64_t c = sh.scan[t];
      sh.scan[t] = acc;
      acc += c;
    }
    sh.sel_above = acc;  // W''
  }
  __syncthreads();
  const uint64_t Wr = sh.sel_above;
  if (Wr == 0) {  // nothing left: the first id of maximal kept weight
    // first maximum across threads: max weight, then the smallest id holding it
    __syncthreads();
    sh.scan[tid] = best_w;
    __syncthreads();
    if (tid == 0) {
      uint64_t bw = 0;
      for (int t = 0; t < kSampThreads; ++t) bw = sh.scan[t] > bw ? sh.scan[t] : bw;
      sh.hist[0] = bw;
    }
    __syncthreads();
    const int cand = best_w == sh.hist[0] ? best_v : V;
    int m = cand;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = min(m, __shfl_xor(m, o, 64));
    __syncthreads();
    if ((tid & 63) == 0) sh.red32[tid >> 6] = (uint32_t)m;
    __syncthreads();
    if (tid == 0) {
      int a = V;
      for (int w = 0; w < kSampWaves; ++w) a = min(a, (int)sh.red32[w]);
      draw[row] = a < V ? a : 0;  // every weight 0 (a non-finite row): the first id, as argmax of zeros
    }
    return;
  }
  double uu = u[row];
  if (!(uu >= 0.0)) uu = 0.0;  // u below 0 (or NaN) draws as 0; u >= 1 is held at Wr - 1 below
  uint64_t target = (uint64_t)(uu * (double)Wr);
  if (target >= Wr) target = Wr - 1;
  const uint64_t base = sh.scan[tid];
  if (target >= base && target < base + my_r) {
    uint64_t acc = base, tr = tie_base;
    for (int v = v0; v < v1; ++v) {
      uint64_t w = final_w(v, &tr);
      if (v == d) w = 0;
      acc += w;
      if (acc > target) {
        draw[row] = v;
        break;
      }
    }
  }
}

__global__ __launch_bounds__(kSampThreads) void sample_rows_kernel(
    const uint16_t* __restrict__ logits, int V, float temp, int top_k, float top_p,
    const int32_t* __restrict__ draft, const double* __restrict__ u, float* __restrict__ p_draft,
    int32_t* __restrict__ draw, float* __restrict__ probs) {
  __shared__ SampShared sh;
  sample_row_general(sh, blockIdx.x, logits, V, temp, top_k, top_p, draft, u, p_draft, draw, probs);
}

// The same, called: for the rows that the split path leaves to it, so that its code does not sit among that path's
// (inlined there one row of 128,256 logits without top-k and top-p takes 19.1 us instead of 18.2).
__device__ __attribute__((noinline)) void sample_row_general_call(SampShared& sh, int row, const uint16_t* __restrict__ logits,
                                                                  int V, float temp, int top_k, float top_p,
                                                                  const int32_t* __restrict__ draft,
                                                                  const double* __restrict__ u, float* __restrict__ p_draft,
                                                                  int32_t* __restrict__ draw, float* __restrict__ probs) {
  sample_row_general(sh, row, logits, V, temp, top_k, top_p, draft, u, p_draft, draw, probs);
}

// ---- a row split over many workgroups ---------------------------------------------------------------
// One workgroup a row (sample_row_general) leaves all but R of the 256 CUs idle and reads the row about
// ten times: the fp64 weights of 201,088 tokens alone are 60 us of one CU's fp64 rate.  With a workspace
// the row is cut into chunks of consecutive ids (at most 64) and each pass is one launch over
// (chunk, row), so the passes are bound by their launches and one round trip to memory:
//   sample_max_kernel    each chunk's (largest key, first id of it), and whether the row needs the general path;
//   sample_hist_kernel   the row's histogram of key / 32 over the tokens of non-zero weight: counts (for
//                        top-k) and weight sums (for top-p); without either, each chunk's weight sum;
//   sample_codes_kernel  (one launch for top-k, one for top-p) the bin the boundary lies in, and for each
//                        chunk the weight above that bin and the count of each of the bin's 32 keys;
//   sample_final_kernel  one workgroup a row: the boundary key and its ties, every chunk's kept weight
//                        from those sums, the drafted token's weight, and the draw -- only the chunk
//                        that holds it is read again;
//   sample_probs_rows_kernel  the probabilities, when asked for.
// The key is the logit's 16 bits in value order; z = x / temp does not decrease with it, and equal z of
// different keys need a quotient that overflows or gets near the denormals, so rows with NaN, +inf, such
// a quotient or a zero that is none take sample_row_general in the final kernel.  Sums are of integers:
// the results are the general path's bit for bit.
// 8 rows x 201,088, temperature 0.8, top-p 0.95: 656 us (one workgroup a row) -> 35 us; 6 rows without top-k
// and top-p: 346 -> 21 us.
constexpr int kChunkThreads = 256;
constexpr int kMaxChunks = 64;
constexpr int kChunkStep = kChunkThreads * 8;  // ids of one iteration of a chunk's loop
constexpr int kMinChunk = 2 * kChunkStep;      // two iterations: less, and the launch outweighs the loads
constexpr int kBins = 2048, kBinKeys = 32;     // key >> 5, key & 31
constexpr int kRowsAtOnce = 256;               // rows of one set of launches; more rows reuse the workspace
// Greedy rows of few chunks stay with one workgroup: there is little to divide, and the split path's second launch
// costs more; a workgroup a row takes any number of rows in one launch.  One workgroup / split, us: V 512 1 row
// 2.8 / 4.9, 512 rows 5.0 / 11.1; V 8,192 4.6 / 6.0 and 10.9 / 15.8; V 12,288 5.5 / 6.0 and 10.8 / 14.4; V 16,384 1 row
// 7.0 / 6.1, 256 rows 10.0 / 10.5, 512 14.0 / 15.5; V 20,480 1 row 8.2 / 6.0, 512 16.6 / 16.8, 1,024 44.8 / 35.3.
inline bool greedy_one_workgroup(int R, int V) { return V <= (R >= kRowsAtOnce ? 4 : 3) * kMinChunk; }

struct SampPlan {
  int V, chunk, n_chunks;
  float tdiv, tiny, top_p;  // z = x / tdiv; 0 < |x| < tiny sends a row to the general path
  int top_k;                // 0: off
  int use_p, greedy, vec;   // vec: rows may be read 16 bytes at a time
};

struct SampRow {
  uint64_t wts[kBins];
  uint32_t cnt[kBins];
  uint64_t above[kMaxChunks];            // weight of the chunk's tokens above the boundary bin
  uint64_t best[kMaxChunks];             // largest key << 32 | ~first id
  uint32_t flag[kMaxChunks];
  uint32_t cc[2][kMaxChunks][kBinKeys];  // [top-k, top-p]: the chunk's tokens of each key of the boundary bin
  uint32_t tie_before[kMaxChunks];
  // the boundary bins with the totals above them, and top-p's limit (sample_codes_kernel)
  uint64_t kabove, pabove, plimit;
  int32_t kbin, pbin;
  uint32_t kkey, pkey;  // the boundary keys
  uint64_t kept, tie_keep;
  int32_t arg;
};

// the 16 bits of a bf16 in value order (-0 as +0), and back
__device__ __forceinline__ uint32_t bf_key(uint16_t b) {
  return (b & 0x8000u) ? (b == 0x8000u ? 0x8000u : (~(uint32_t)b & 0xffffu)) : (b | 0x8000u);
}
__device__ __forceinline__ float key_bf(uint32_t k) {
  return bf2f((uint16_t)((k & 0x8000u) ? (k & 0x7fffu) : (~k & 0xffffu)));
}
__device__ __forceinline__ uint64_t key_weight(uint32_t k, float tdiv, float zmax) {
  return samp_weight(__fdiv_rn(key_bf(k), tdiv), zmax);
}

template <class T>
__device__ __forceinline__ T wave_incl_scan(T v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const T y = __shfl_up(v, o, 64);
    if (lane >= o) v += y;
  }
  return v;
}

// exclusive prefix over the workgroup's NT threads; *total gets the sum
template <int NT, class T>
__device__ __forceinline__ T block_excl_scan(T v, T* red, T* total) {
  const T incl = wave_incl_scan(v);
  const int wave = threadIdx.x >> 6;
  __syncthreads();  // the last use of red is over
  if ((threadIdx.x & 63) == 63) red[wave] = incl;
  __syncthreads();
  T base = 0, sum = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) {
    base += w < wave ? red[w] : (T)0;
    sum += red[w];
  }
  *total = sum;
  return base + incl - v;
}

// f(id, bits) for the thread's ids of [c0, c1), in steps of 8 consecutive ids a thread
template <class F>
__device__ __forceinline__ void for_chunk(const uint16_t* __restrict__ x, int c0, int c1, int vec, F&& f) {
  for (int b = c0 + (int)threadIdx.x * 8; b < c1; b += kChunkStep) {
    if (vec && b + 8 <= c1) {
      const uint4 q = *reinterpret_cast<const uint4*>(x + b);
      const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) f(b + j, (uint16_t)((j & 1) ? w[j >> 1] >> 16 : w[j >> 1] & 0xffffu));
    } else {
      const int n = min(8, c1 - b);
      for (int j = 0; j < n; ++j) f(b + j, x[b + j]);
    }
  }
}

struct RowMax {
  float zmax;
  uint32_t general;
  uint64_t best;
};

struct ChunkShared {
  uint64_t red[kSampWaves];
  RowMax mx;
  uint64_t tot[kBinKeys], above;
  uint32_t kkey, pkey, rank;
  int bin;
};

// the row's maximum over its chunks, by every thread of the workgroup
__device__ __forceinline__ RowMax row_max(const SampPlan& p, const SampRow& r, ChunkShared& sh) {
  if (threadIdx.x < 64) {
    const int c = threadIdx.x;
    uint64_t b = c < p.n_chunks ? r.best[c] : 0;
    uint32_t fl = c < p.n_chunks ? r.flag[c] : 0;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      const uint64_t y = __shfl_xor(b, o, 64);
      b = y > b ? y : b;
      fl |= __shfl_xor(fl, o, 64);
    }
    if (c == 0) {
      sh.mx.best = b;
      sh.mx.zmax = p.greedy ? 0.f : __fdiv_rn(key_bf((uint32_t)(b >> 32)), p.tdiv);
      sh.mx.general = !p.greedy && (fl || sh.mx.zmax == INFINITY);
    }
  }
  __syncthreads();
  return sh.mx;
}

// The bin, taken from the largest key down, where the running total of mass(bin) first exceeds limit
// (sh.bin, or -1) and the total above it (sh.above).
template <int NT, class Mass>
__device__ __forceinline__ void find_bin(Mass&& mass, uint64_t limit, ChunkShared& sh) {
  constexpr int kPer = kBins / NT;
  uint64_t m[kPer], sum = 0, total;
#pragma unroll
  for (int j = 0; j < kPer; ++j) {
    m[j] = mass(kBins - 1 - ((int)threadIdx.x * kPer + j));
    sum += m[j];
  }
  uint64_t run = block_excl_scan<NT>(sum, sh.red, &total);
  if (threadIdx.x == 0 && total <= limit) {
    sh.bin = -1;
    sh.above = total;
  }
  if (run <= limit && limit < run + sum) {  // one thread, if any
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
      if (run <= limit && limit < run + m[j]) {
        sh.bin = kBins - 1 - ((int)threadIdx.x * kPer + j);
        sh.above = run;
      }
      run += m[j];
    }
  }
  __syncthreads();
}

// totals over the chunks of the boundary bin's 32 keys, to sh.tot
__device__ __forceinline__ void bin_totals(const SampPlan& p, const uint32_t (&cc)[kMaxChunks][kBinKeys], ChunkShared& sh) {
  if (threadIdx.x < 64) {  // lane = half of the chunks x key
    const int k = threadIdx.x & 31;
    uint32_t n = 0;
    for (int c = threadIdx.x >> 5; c < p.n_chunks; c += 2) n += cc[c][k];
    n += __shfl_xor(n, 32, 64);
    if (threadIdx.x < 32) sh.tot[k] = n;
  }
  __syncthreads();
}

// The k-th largest key (0 when fewer than k tokens have weight): its bin is known, its totals go to sh.tot.
__device__ __forceinline__ uint32_t resolve_k(const SampPlan& p, const SampRow& r, ChunkShared& sh) {
  if (r.kbin < 0) return 0;
  bin_totals(p, r.cc[0], sh);
  if (threadIdx.x == 0) {
    uint64_t run = r.kabove;
    int k = kBinKeys - 1;
    while (k > 0 && run + sh.tot[k] <= (uint64_t)(p.top_k - 1)) run += sh.tot[k--];
    sh.kkey = (uint32_t)(r.kbin * kBinKeys + k);
  }
  __syncthreads();
  return sh.kkey;
}

// The bin of top-p's boundary over the tokens of key >= kkey (kbin: kkey's bin) to sh.bin, the weight above it
// to sh.above; returns the limit floor(p W).
template <int NT>
__device__ __forceinline__ uint64_t find_p_bin(const SampPlan& p, const SampRow& r, float zmax, int kbin, uint32_t kkey,
                                               ChunkShared& sh) {
  uint64_t part = 0;  // the kept weight of kkey's bin (sh.tot holds its counts)
  if (kbin >= 0 && threadIdx.x < 64) {
    const uint32_t key = (uint32_t)(kbin * kBinKeys) + (threadIdx.x & 31);
    part = (threadIdx.x < 32 && key >= kkey) ? sh.tot[threadIdx.x] * key_weight(key, p.tdiv, zmax) : 0;
  }
  uint64_t total;
  block_excl_scan<NT>(part, sh.red, &total);
  const uint64_t kpart = total;
  auto mass = [&](int b) { return b > kbin ? r.wts[b] : (b == kbin ? kpart : (uint64_t)0); };
  uint64_t sum = 0;
  for (int b = threadIdx.x; b < kBins; b += NT) sum += mass(b);
  block_excl_scan<NT>(sum, sh.red, &total);
  const uint64_t limit = (uint64_t)floor((double)p.top_p * (double)total);
  find_bin<NT>(mass, limit, sh);
  return limit;
}

__global__ __launch_bounds__(kChunkThreads) void sample_max_kernel(const uint16_t* __restrict__ logits, SampPlan p,
                                                                   SampRow* __restrict__ rows) {
  __shared__ uint64_t best_s[kChunkThreads / 64];
  __shared__ uint32_t flag_s[kChunkThreads / 64];
  const int c = blockIdx.x, tid = threadIdx.x;
  SampRow& r = rows[blockIdx.y];
  const int c0 = c * p.chunk, c1 = min(p.V, c0 + p.chunk);
  if (p.top_k || p.use_p)
    for (int b = c * kChunkThreads + tid; b < kBins; b += p.n_chunks * kChunkThreads) {
      r.wts[b] = 0;
      r.cnt[b] = 0;
    }
  uint32_t bk = 0, fl = 0;
  int bi = 0x7fffffff;
  for_chunk(logits + (size_t)blockIdx.y * p.V, c0, c1, p.vec, [&](int v, uint16_t bits) {
    const uint32_t k = bf_key(bits);
    const float ax = fabsf(bf2f(bits));
    fl |= (ax != ax) || bits == 0x7f80u || (ax > 0.f && ax < p.tiny);
    if (k > bk || bi == 0x7fffffff) { bk = k; bi = v; }
  });
  uint64_t best = bi == 0x7fffffff ? 0 : ((uint64_t)bk << 32) | (uint32_t)~bi;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const uint64_t y = __shfl_xor(best, o, 64);
    best = y > best ? y : best;
    fl |= __shfl_xor(fl, o, 64);
  }
  if ((tid & 63) == 0) { best_s[tid >> 6] = best; flag_s[tid >> 6] = fl; }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kChunkThreads / 64; ++w) {
      best = best_s[w] > best ? best_s[w] : best;
      fl |= flag_s[w];
    }
    r.best[c] = best;
    r.flag[c] = fl;
  }
}

__global__ __launch_bounds__(kChunkThreads) void sample_hist_kernel(const uint16_t* __restrict__ logits, SampPlan p,
                                                                    SampRow* __restrict__ rows) {
  __shared__ uint64_t wts[kBins];
  __shared__ uint32_t cnt[kBins];
  __shared__ ChunkShared sh;
  const int c = blockIdx.x, tid = threadIdx.x;
  SampRow& r = rows[blockIdx.y];
  const RowMax mx = row_max(p, r, sh);
  if (mx.general) return;  // uniform over the workgroup
  const int c0 = c * p.chunk, c1 = min(p.V, c0 + p.chunk);
  const uint16_t* x = logits + (size_t)blockIdx.y * p.V;
  if (!p.top_k && !p.use_p) {
    uint64_t sum = 0, total;
    for_chunk(x, c0, c1, p.vec, [&](int, uint16_t bits) { sum += samp_weight(__fdiv_rn(bf2f(bits), p.tdiv), mx.zmax); });
    block_excl_scan<kChunkThreads>(sum, sh.red, &total);
    if (tid == 0) r.above[c] = total;
    return;
  }
  for (int b = tid; b < kBins; b += kChunkThreads) {
    wts[b] = 0;
    cnt[b] = 0;
  }
  __syncthreads();
  for_chunk(x, c0, c1, p.vec, [&](int, uint16_t bits) {
    const uint64_t w = samp_weight(__fdiv_rn(bf2f(bits), p.tdiv), mx.zmax);
    if (!w) return;
    const uint32_t b = bf_key(bits) / kBinKeys;
    if (p.use_p) atomicAdd((unsigned long long*)&wts[b], (unsigned long long)w);
    if (p.top_k) atomicAdd(&cnt[b], 1u);
  });
  __syncthreads();
  for (int b = tid; b < kBins; b += kChunkThreads) {
    if (wts[b]) atomicAdd((unsigned long long*)&r.wts[b], (unsigned long long)wts[b]);
    if (cnt[b]) atomicAdd(&r.cnt[b], cnt[b]);
  }
}

// which = 0: the boundary bin of top-k; 1: of top-p, among the tokens top-k keeps
__global__ __launch_bounds__(kChunkThreads) void sample_codes_kernel(const uint16_t* __restrict__ logits, SampPlan p,
                                                                     SampRow* __restrict__ rows, int which) {
  __shared__ ChunkShared sh;
  __shared__ uint32_t cc[kBinKeys];
  const int c = blockIdx.x, tid = threadIdx.x;
  SampRow& r = rows[blockIdx.y];
  const RowMax mx = row_max(p, r, sh);
  if (mx.general) return;  // uniform over the workgroup
  if (tid < kBinKeys) cc[tid] = 0;
  uint32_t kkey = 0;
  uint64_t limit = 0;
  if (which == 0) {
    find_bin<kChunkThreads>([&](int b) { return (uint64_t)r.cnt[b]; }, (uint64_t)(p.top_k - 1), sh);
  } else {
    if (p.top_k) kkey = resolve_k(p, r, sh);
    limit = find_p_bin<kChunkThreads>(p, r, mx.zmax, p.top_k ? r.kbin : -1, kkey, sh);
  }
  const int bin = sh.bin;
  if (c == 0 && tid == 0) {  // read by the next launch only
    if (which == 0) {
      r.kbin = bin;
      r.kabove = sh.above;
    } else {
      r.pbin = bin;
      r.pabove = sh.above;
      r.plimit = limit;
      r.kkey = kkey;
    }
  }
  const int c0 = c * p.chunk, c1 = min(p.V, c0 + p.chunk);
  uint64_t sum = 0, total;
  for_chunk(logits + (size_t)blockIdx.y * p.V, c0, c1, p.vec, [&](int, uint16_t bits) {
    const uint32_t k = bf_key(bits);
    if (k < kkey || (int)(k / kBinKeys) < bin) return;
    const uint64_t w = samp_weight(__fdiv_rn(bf2f(bits), p.tdiv), mx.zmax);
    if (!w) return;
    if ((int)(k / kBinKeys) > bin) sum += w;
    else atomicAdd(&cc[k % kBinKeys], 1u);
  });
  block_excl_scan<kChunkThreads>(sum, sh.red, &total);  // (its barriers also end the counting)
  if (tid == 0) r.above[c] = total;
  if (tid < kBinKeys) r.cc[which][c][tid] = cc[tid];
}

__global__ __launch_bounds__(kSampThreads) void sample_final_kernel(
    const uint16_t* __restrict__ logits, SampPlan p, SampRow* __restrict__ rows, float temp, int top_k,
    const int32_t* __restrict__ draft, const double* __restrict__ u, float* __restrict__ p_draft,
    int32_t* __restrict__ draw, float* __restrict__ probs) {
  __shared__ union { SampShared gen; ChunkShared ch; } un;
  __shared__ uint64_t tot_s[kMaxChunks];   // each chunk's kept weight
  __shared__ uint64_t base_s[kMaxChunks];  // ... of the chunks before it
  __shared__ uint32_t tie_s[kMaxChunks];   // boundary ties of the chunks before it
  __shared__ uint64_t wk_s, wtab[kBinKeys], tot_k[kBinKeys];
  __shared__ uint32_t cc_s[kMaxChunks][kBinKeys + 1];
  __shared__ int hit_s;
  ChunkShared& sh = un.ch;
  const int row = blockIdx.x, tid = threadIdx.x;
  SampRow& r = rows[row];
  const uint16_t* x = logits + (size_t)row * p.V;
  // every load that does not wait for another one first
  const int which = p.use_p ? 1 : 0;
  const int d = draft ? draft[row] : -1;
  const int pbin = p.use_p ? r.pbin : -1, kbin = p.top_k ? r.kbin : -1;
  const int bin = p.use_p ? pbin : kbin;
  const uint64_t limit = p.use_p ? r.plimit : (uint64_t)(p.top_k - 1);
  const uint64_t above = p.use_p ? r.pabove : r.kabove;
  uint32_t kkey = p.use_p && p.top_k ? r.kkey : 0, pkey = 0;
  double uu = draw && u ? u[row] : 0.0;
  const uint64_t chunk_above = tid < p.n_chunks ? r.above[tid] : 0;
  if (bin >= 0)
    for (int i = tid; i < p.n_chunks * kBinKeys; i += kSampThreads) cc_s[i / kBinKeys][i % kBinKeys] = r.cc[which][i / kBinKeys][i % kBinKeys];
  const int dc = d >= 0 && d < p.V ? d / p.chunk : -1;
  const uint32_t dkey = dc >= 0 ? bf_key(x[d]) : 0;
  const RowMax mx = row_max(p, r, sh);
  if (p.greedy) {
    const int arg = (int)~(uint32_t)mx.best;
    if (tid == 0) {
      if (draw) draw[row] = arg;
      if (p_draft) p_draft[row] = d == arg ? 1.f : 0.f;
      r.arg = arg;
    }
    return;
  }
  if (mx.general) {
    __syncthreads();  // every thread has read the union's other side
    sample_row_general_call(un.gen, row, logits, p.V, temp, top_k, p.top_p, draft, u, p_draft, draw, probs);
    return;
  }
  // the boundary key: the first, from the bin's largest down, whose running total exceeds the limit
  uint64_t tie_keep = 0;
  if (bin >= 0) {
    if (tid < 64) {
      const int k = kBinKeys - 1 - (tid & 31);  // lanes in descending order of key
      uint32_t n = 0;
      if (tid < kBinKeys)
        for (int c = 0; c < p.n_chunks; ++c) n += cc_s[c][k];
      const uint64_t w = key_weight((uint32_t)(bin * kBinKeys + k), p.tdiv, mx.zmax);
      const uint64_t mass = p.use_p ? n * w : (uint64_t)n;
      const uint64_t incl = wave_incl_scan(mass);
      if (tid < kBinKeys) {
        wtab[k] = w;
        tot_k[k] = above + incl - mass;
        if (above + incl > limit && above + incl - mass <= limit) sh.pkey = (uint32_t)(bin * kBinKeys + k);
      }
    }
    __syncthreads();
    if (p.use_p) {
      pkey = sh.pkey;
      // tie j (0-based, id order) of the boundary key is kept iff the weight before it is <= the limit
      tie_keep = (limit - tot_k[pkey % kBinKeys]) / wtab[pkey % kBinKeys] + 1;
    } else {
      kkey = sh.pkey;
    }
  }
  if (tid < kMaxChunks) {
    const int c = tid;
    uint64_t w = chunk_above, ties = 0;
    if (bin >= 0 && c < p.n_chunks) {
      const uint32_t first = p.use_p ? pkey + 1 : kkey;  // keys of the bin from here on are kept whole
      for (int k = kBinKeys - 1; k >= 0 && (uint32_t)(bin * kBinKeys + k) >= first; --k) w += cc_s[c][k] * wtab[k];
      if (p.use_p) ties = cc_s[c][pkey % kBinKeys];
    }
    const uint64_t before = wave_incl_scan(ties) - ties;
    const uint64_t keep = before >= tie_keep ? 0 : min(ties, tie_keep - before);
    if (p.use_p && bin >= 0) w += keep * wtab[pkey % kBinKeys];
    const uint64_t incl = wave_incl_scan(w);
    tot_s[c] = w;
    base_s[c] = incl - w;
    tie_s[c] = (uint32_t)before;
    if (c < p.n_chunks) r.tie_before[c] = (uint32_t)before;
    if (c == kMaxChunks - 1) wk_s = incl;
  }
  __syncthreads();
  const uint64_t Wk = wk_s;
  // the drafted token's weight; as a boundary tie it counts if its rank among the ties is kept
  uint64_t Wd = 0;
  if (dc >= 0) {
    const uint32_t k = dkey;
    bool kept = k >= kkey && (pbin < 0 || k >= pkey);
    if (kept && pbin >= 0 && k == pkey) {  // uniform over the workgroup
      uint32_t n = 0, rank;
      for (int v = dc * p.chunk + tid; v < d; v += kSampThreads) n += bf_key(x[v]) == pkey;
      block_excl_scan<kSampThreads>(n, reinterpret_cast<uint32_t*>(sh.red), &rank);
      kept = tie_s[dc] + (uint64_t)rank < tie_keep;
    }
    if (kept) Wd = key_weight(k, p.tdiv, mx.zmax);
  }
  if (tid == 0) {
    if (p_draft) p_draft[row] = (d >= 0 && Wk > 0) ? (float)((double)Wd / (double)Wk) : 0.f;
    r.kept = Wk;
    r.tie_keep = tie_keep;
    r.kkey = kkey;
    r.pkey = pkey;
    r.pbin = pbin;
  }
  if (!(draw && u)) return;
  const uint64_t Wr = Wk - Wd;
  if (Wr == 0) {  // nothing but the drafted token is left, or nothing at all
    if (tid == 0) draw[row] = Wk ? d : 0;
    return;
  }
  if (!(uu >= 0.0)) uu = 0.0;  // u below 0 (or NaN) draws as 0; u >= 1 is held at Wr - 1 below
  uint64_t target = (uint64_t)(uu * (double)Wr);
  if (target >= Wr) target = Wr - 1;
  if (tid < kMaxChunks) {  // the chunk whose residual weight holds the target
    const uint64_t lo = base_s[tid] - (dc >= 0 && tid > dc ? Wd : 0);
    const uint64_t w = tot_s[tid] - (tid == dc ? Wd : 0);
    if (target >= lo && target < lo + w) {
      hit_s = tid;
      sh.above = lo;
    }
  }
  __syncthreads();
  const int c = hit_s;
  const uint64_t left = target - sh.above;
  const int c0 = c * p.chunk, c1 = min(p.V, c0 + p.chunk);
  const int per = (c1 - c0 + kSampThreads - 1) / kSampThreads;
  const int v0 = min(c1, c0 + tid * per), v1 = min(c1, v0 + per);
  uint32_t my_ties = 0, all_ties;
  if (pbin >= 0)
    for (int v = v0; v < v1; ++v) my_ties += bf_key(x[v]) == pkey;
  const uint32_t rank0 = tie_s[c] + block_excl_scan<kSampThreads>(my_ties, reinterpret_cast<uint32_t*>(sh.red), &all_ties);
  auto weight = [&](int v, uint64_t& rank) __attribute__((always_inline)) -> uint64_t {
    const uint32_t k = bf_key(x[v]);
    if (k < kkey || (pbin >= 0 && (k < pkey || (k == pkey && rank++ >= tie_keep))) || v == d) return 0;
    return key_weight(k, p.tdiv, mx.zmax);
  };
  uint64_t my = 0, all, rank = rank0;
  for (int v = v0; v < v1; ++v) my += weight(v, rank);
  uint64_t run = block_excl_scan<kSampThreads>(my, sh.red, &all);
  if (left >= run && left < run + my) {
    rank = rank0;
    for (int v = v0; v < v1; ++v) {
      run += weight(v, rank);
      if (run > left) {
        draw[row] = v;
        break;
      }
    }
  }
}

__global__ __launch_bounds__(kChunkThreads) void sample_probs_rows_kernel(const uint16_t* __restrict__ logits, SampPlan p,
                                                                          const SampRow* __restrict__ rows,
                                                                          float* __restrict__ probs) {
  __shared__ ChunkShared sh;
  const int c = blockIdx.x;
  const SampRow& r = rows[blockIdx.y];
  const int c0 = c * p.chunk, c1 = min(p.V, c0 + p.chunk);
  const uint16_t* x = logits + (size_t)blockIdx.y * p.V;
  float* o = probs + (size_t)blockIdx.y * p.V;
  if (p.greedy) {
    for (int v = c0 + (int)threadIdx.x; v < c1; v += kChunkThreads) o[v] = v == r.arg ? 1.f : 0.f;
    return;
  }
  const RowMax mx = row_max(p, r, sh);
  if (mx.general) return;  // written by the general path
  uint64_t before = r.tie_before[c];
  for (int b0 = c0; b0 < c1; b0 += kChunkThreads) {  // one id a thread: the boundary ties stay in id order
    const int v = b0 + (int)threadIdx.x;
    const uint32_t k = v < c1 ? bf_key(x[v]) : 0;
    bool keep = v < c1 && k >= r.kkey;
    if (r.pbin >= 0) {
      const uint32_t tie = v < c1 && k == r.pkey;
      uint32_t n;
      const uint32_t rank = block_excl_scan<kChunkThreads>(tie, reinterpret_cast<uint32_t*>(sh.red), &n);
      keep = keep && k >= r.pkey && (!tie || before + rank < r.tie_keep);
      before += n;
    }
    const uint64_t w = keep ? key_weight(k, p.tdiv, mx.zmax) : 0;
    if (v < c1) o[v] = r.kept ? (float)((double)w / (double)r.kept) : 0.f;
  }
}

// A draw from a given probability vector (the reference's Sampler.sample(probs)): weights
// floor(p_v * 2^40), then the same inverse-CDF rule; all-zero -> the first maximal id (0).
__global__ __launch_bounds__(kSampThreads) void sample_probs_kernel(const float* __restrict__ p, int V, double u,
                                                                    int32_t* __restrict__ out) {
  __shared__ SampShared sh;
  const int tid = threadIdx.x;
  const int C = (V + kSampThreads - 1) / kSampThreads;
  const int v0 = tid * C, v1 = min(V, v0 + C);
  uint64_t my = 0;
  for (int v = v0; v < v1; ++v) my += (uint64_t)((double)fmaxf(p[v], 0.f) * 0x1p40);
  sh.scan[tid] = my;
  __syncthreads();
  if (tid == 0) {
    uint64_t acc = 0;
    for (int t = 0; t < kSampThreads; ++t) {
      const uint64_t c = sh.scan[t];
      sh.scan[t] = acc;
      acc += c;
    }
    sh.sel_above = acc;
  }
  __syncthreads();
  const uint64_t W = sh.sel_above;
  if (W == 0) {
    if (tid == 0) out[0] = 0;
    return;
  }
  uint64_t target = (uint64_t)(u * (double)W);
  if (target >= W) target = W - 1;
  const uint64_t base = sh.scan[tid];
  if (target >= base && target < base + my) {
    uint64_t acc = base;
    for (int v = v0; v < v1; ++v) {
      acc += (uint64_t)((double)fmaxf(p[v], 0.f) * 0x1p40);
      if (acc > target) {
        out[0] = v;
        break;
      }
    }
  }
}

}  // namespace flyai

using namespace flyai;

extern "C" int flyai_sample_rows(const uint16_t* logits, int32_t R, int32_t V, float temp, int32_t top_k,
                                 float top_p, const int32_t* draft, const double* u, float* p_draft,
                                 int32_t* draw, float* probs, flyai_stream_t stream) {
  FLYAI_REQUIRE(R >= 0 && V > 0, "sample_rows: bad shape");
  FLYAI_REQUIRE(logits, "sample_rows: null logits");
  FLYAI_REQUIRE(top_k >= 0, "sample_rows: top_k must be >= 0");
  FLYAI_REQUIRE(!(draw && !u && temp > 0.f), "sample_rows: a sampled draw needs u");
  if (R == 0) return FLYAI_OK;
  hipLaunchKernelGGL(sample_rows_kernel, dim3(R), dim3(kSampThreads), 0, as_stream(stream), logits, V, temp, top_k,
                     top_p, draft, u, p_draft, draw, probs);
  return check_launch("sample_rows");
}

extern "C" size_t flyai_sample_workspace_bytes(int32_t R, int32_t V) {
  return R > 0 && V > 0 ? (size_t)std::min(R, kRowsAtOnce) * sizeof(SampRow) : 0;
}

extern "C" int flyai_sample_rows_ws(const uint16_t* logits, int32_t R, int32_t V, float temp, int32_t top_k,
                                    float top_p, const int32_t* draft, const double* u, float* p_draft,
                                    int32_t* draw, float* probs, void* workspace, flyai_stream_t stream) {
  FLYAI_REQUIRE(R >= 0 && V > 0, "sample_rows: bad shape");
  FLYAI_REQUIRE(logits, "sample_rows: null logits");
  FLYAI_REQUIRE(top_k >= 0, "sample_rows: top_k must be >= 0");
  FLYAI_REQUIRE(!(draw && !u && temp > 0.f), "sample_rows: a sampled draw needs u");
  if (R == 0) return FLYAI_OK;
  FLYAI_REQUIRE(workspace && ((uintptr_t)workspace & 7) == 0, "sample_rows: the workspace must be 8-byte aligned");
  hipStream_t s = as_stream(stream);
  if (!(temp > 0.f) && greedy_one_workgroup(R, V)) {
    hipLaunchKernelGGL(sample_rows_kernel, dim3(R), dim3(kSampThreads), 0, s, logits, V, temp, top_k, top_p, draft, u, p_draft,
                       draw, probs);
    return check_launch("sample_rows");
  }
  SampPlan p;
  p.V = V;
  const int steps = (int)(((int64_t)V + (int64_t)kMaxChunks * kChunkStep - 1) / ((int64_t)kMaxChunks * kChunkStep));
  p.chunk = std::max(kMinChunk, steps * kChunkStep);
  p.n_chunks = (int)(((int64_t)V + p.chunk - 1) / p.chunk);
  p.greedy = !(temp > 0.f);
  p.tdiv = fmaxf(temp, 1e-6f);
  p.tiny = p.tdiv * 0x1p-99f;
  p.top_k = top_k < V ? top_k : 0;
  p.top_p = top_p;
  p.use_p = top_p > 0.f && top_p < 1.f;
  p.vec = V % 8 == 0 && ((uintptr_t)logits & 15) == 0;
  SampRow* ws = static_cast<SampRow*>(workspace);
  for (int r0 = 0; r0 < R; r0 += kRowsAtOnce) {
    const int n = std::min(R - r0, kRowsAtOnce);
    const uint16_t* x = logits + (size_t)r0 * V;
    auto at = [&](auto* q, size_t step) { return q ? q + step * r0 : q; };
    const dim3 grid(p.n_chunks, n), block(kChunkThreads);
    hipLaunchKernelGGL(sample_max_kernel, grid, block, 0, s, x, p, ws);
    if (!p.greedy) {
      hipLaunchKernelGGL(sample_hist_kernel, grid, block, 0, s, x, p, ws);
      if (p.top_k) hipLaunchKernelGGL(sample_codes_kernel, grid, block, 0, s, x, p, ws, 0);
      if (p.use_p) hipLaunchKernelGGL(sample_codes_kernel, grid, block, 0, s, x, p, ws, 1);
    }
    hipLaunchKernelGGL(sample_final_kernel, dim3(n), dim3(kSampThreads), 0, s, x, p, ws, temp, top_k, at(draft, 1),
                       at(u, 1), at(p_draft, 1), at(draw, 1), at(probs, V));
    if (probs) hipLaunchKernelGGL(sample_probs_rows_kernel, grid, block, 0, s, x, p, ws, at(probs, V));
    const int rc = check_launch("sample_rows");
    if (rc) return rc;
  }
  return FLYAI_OK;
}

extern "C" int flyai_sample_probs(const float* probs, int32_t V, double u, int32_t* out, flyai_stream_t stream) {
  FLYAI_REQUIRE(probs && out && V > 0, "sample_probs: bad arguments");
  FLYAI_REQUIRE(u >= 0.0 && u < 1.0, "sample_probs: u must be in [0, 1)");
  hipLaunchKernelGGL(sample_probs_kernel, dim3(1), dim3(kSampThreads), 0, as_stream(stream), probs, V, u, out);
  return check_launch("sample_probs");
}
