// ss_sample.hip - non-greedy sampling of the next token on the device.
//
// k_sample follows ss_sample (tensor.c:363-451) step by step over the logits
// the LM head left in HBM, in one workgroup:
//   1. x_i = logit_i / T (NaN logits become -FLT_MAX), softmax (tensor.c:154-173);
//   2. top-k: probabilities below the k-th largest (NaN counted as 0 for the
//      ranking, as the reference's sort key) become 0;
//   3. top-p: going down the probabilities in descending order, the cutoff is
//      the probability at which the running sum of the positive ones first
//      reaches top_p; probabilities below it become 0;
//   4. renormalise, draw r from xorshift64 (state passed in, advanced state
//      written back), return the first index whose cumulative probability
//      exceeds r (vocab - 1 when none does).
// The reference sorts all probabilities (qsort) and sums sequentially in
// fp32. Here the k-th largest value and the top-p cutoff come from radix
// selections over the float bit patterns (non-negative floats order like
// their bits), 8 bits per pass with LDS histograms; sums are exact fixed
// point (each probability truncated to a multiple of 2^-52) in uint64, so
// they do not depend on the order the atomics land in. The cumulative
// search is a two-level scan: per-thread chunk sums, a workgroup scan, then
// one sequential walk inside the chunk that holds r. The index differs from
// the reference's only when r lies within the reference's fp32 rounding of a
// cumulative boundary.
//
// One workgroup reads a 128256-entry row some 15 times, 25 us each: 373 us.
// Rows of more than kOneGroup entries go over many workgroups instead, in a
// few short launches (launch_sample), with the same fixed-point sums and the
// same comparisons, so the same index. A softmax term e = exp(x - max) is
// computed before its probability p = e * inv is known; p does not decrease
// with e, so the k-th largest p is that of the k-th largest e.

#include <float.h>
#include <math.h>

#include "ss_device.h"
#include "ss_kernels.h"

namespace ssk {
namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / kWave;
constexpr int kOneGroup = 1024;                // rows up to this: k_sample alone
constexpr int kTile = 1024;                    // entries per workgroup of the others
constexpr int kTileThreads = 256;
constexpr int kBins = 2048;                    // by key >> 19 (sign 0, exponent, 4 bits of the mantissa): e, p <= 1
constexpr int kCand = 2048;                    // candidates the top-k path keeps in LDS
constexpr int kPairs = 288;                    // up to this many are compared each with all, more are sorted
constexpr int kMaxTopK = 1024;                 // top_k it takes
constexpr double kFix = 4503599627370496.0;   // 2^52: probabilities (each <= 1, sums <= ~1)
constexpr double kFixE = 1099511627776.0;     // 2^40: softmax terms (each <= 1, up to 2^18 of them)

// a probability as fixed point; NaN and non-positive values count 0, values
// are clamped to 2 (a probability never exceeds 1 + rounding)
__device__ __forceinline__ uint64_t fix(float p) {
  return p > 0.f ? (uint64_t)((double)fminf(p, 2.0f) * kFix) : 0ull;
}
// the sum at which top-p cuts off (at least one step: the largest value always stays)
__device__ __forceinline__ uint64_t top_p_target(float top_p) {
  const uint64_t t = (uint64_t)((double)top_p * kFix);
  return t > 0 ? t : 1ull;
}
// sort key of tensor.c:384-385 (NaN ranks as 0)
__device__ __forceinline__ uint32_t key(float p) { return __float_as_uint(p == p ? p : 0.f); }

__device__ __forceinline__ uint64_t wave_sum_u64(uint64_t v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
  return v;
}

struct Shared {
  float f[kWaves];
  uint64_t u[kWaves];
  uint32_t hist[256];
  uint64_t hsum[256];
  uint32_t sel, kk;
  int first;
  uint64_t above;
  int done;
};

__device__ float block_max(float v, Shared& sh) {
  v = wave_max(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh.f[threadIdx.x >> 6] = v;
  __syncthreads();
  float m = sh.f[0];
  for (int w = 1; w < kWaves; ++w) m = fmaxf(m, sh.f[w]);
  return m;
}

__device__ uint64_t block_sum(uint64_t v, Shared& sh) {
  v = wave_sum_u64(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh.u[threadIdx.x >> 6] = v;
  __syncthreads();
  uint64_t t = 0;
  for (int w = 0; w < kWaves; ++w) t += sh.u[w];
  return t;
}

__device__ int block_min_i(int v, Shared& sh) {
  __syncthreads();
  if (threadIdx.x == 0) sh.first = 0x7fffffff;
  __syncthreads();
  atomicMin(&sh.first, v);
  __syncthreads();
  return sh.first;
}

// The k-th largest key (1 <= k <= V), MSB first.
__device__ uint32_t kth_largest(const float* p, int V, int k, Shared& sh) {
  uint32_t prefix = 0, mask = 0;
  uint32_t kk = (uint32_t)k;
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int b = threadIdx.x; b < 256; b += kThreads) sh.hist[b] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < V; i += kThreads) {
      const uint32_t u = key(p[i]);
      if ((u & mask) == prefix) atomicAdd(&sh.hist[(u >> shift) & 255u], 1u);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t acc = 0, b = 255;
      for (;; --b) {
        if (acc + sh.hist[b] >= kk || b == 0) break;
        acc += sh.hist[b];
      }
      sh.sel = b;
      sh.kk = kk - acc;
    }
    __syncthreads();
    prefix |= sh.sel << shift;
    mask |= 255u << shift;
    kk = sh.kk;
    __syncthreads();
  }
  return prefix;
}

// The top-p cutoff: the largest positive value v with sum(p >= v, p > 0)
// reaching target (fixed point), or 0 when the positive values never do.
__device__ float top_p_cutoff(const float* p, int V, uint64_t target, Shared& sh) {
  uint32_t prefix = 0, mask = 0;
  uint64_t above = 0;   // sum of the values whose key is above the current prefix range
  for (int shift = 24; shift >= 0; shift -= 8) {
    for (int b = threadIdx.x; b < 256; b += kThreads) sh.hsum[b] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < V; i += kThreads) {
      const float v = p[i];
      if (!(v > 0.f)) continue;
      const uint32_t u = __float_as_uint(v);
      if ((u & mask) == prefix) atomicAdd(reinterpret_cast<unsigned long long*>(&sh.hsum[(u >> shift) & 255u]),
                                          (unsigned long long)fix(v));
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      int b = 255;
      uint64_t acc = above;
      for (; b >= 0; --b) {
        if (acc + sh.hsum[b] >= target) break;
        acc += sh.hsum[b];
      }
      sh.done = b < 0;
      sh.sel = b < 0 ? 0u : (uint32_t)b;
      sh.above = acc;
    }
    __syncthreads();
    if (sh.done) return 0.f;   // uniform: the positive values sum to less than top_p
    prefix |= sh.sel << shift;
    mask |= 255u << shift;
    above = sh.above;
    __syncthreads();
  }
  return __uint_as_float(prefix);
}

__device__ uint64_t advance(uint64_t st) {   // xorshift64, tensor.c:341-343
  st ^= st << 13;
  st ^= st >> 7;
  st ^= st << 17;
  return st;
}
// r as fixed point: (float)(st >> 11) / (float)2^53
__device__ uint64_t draw_fix(uint64_t st) {
  const float r = (float)(st >> 11) / (float)(1ull << 53);
  return (uint64_t)((double)r * kFix);
}
__device__ void put_result(const SampleArgs& a, int idx, uint64_t st) {
  *a.out = idx;
  *a.rng_out = st;
  if (a.tokens) {
    const int pos = *a.dpos;
    a.tokens[pos + 1] = idx;
    *a.dpos = pos + 1;
  }
}

// The whole of ss_sample in one workgroup. HAVE: the softmax terms are in
// a.probs already; inv: the factor that makes them probabilities.
template <bool HAVE>
__device__ void sample_one_group(const SampleArgs& a, Shared& sh, float inv = 0.f) {
  const int V = a.V, tid = threadIdx.x;
  float* p = a.probs;
  uint64_t s = 0;
  int nan_at = 0x7fffffff;

  // 1. temperature and softmax (tensor.c:374-381, 154-173)
  if constexpr (!HAVE) {
    float mx = -FLT_MAX;
    for (int i = tid; i < V; i += kThreads) {
      const float l = a.logits[i];
      const float x = l != l ? -FLT_MAX : l / a.temperature;
      p[i] = x;
      mx = fmaxf(mx, x);
    }
    mx = block_max(mx, sh);
    for (int i = tid; i < V; i += kThreads) {
      const float e = expf(p[i] - mx);
      p[i] = e;
      s += e > 0.f ? (uint64_t)((double)e * kFixE) : 0ull;   // e <= 1
      if (e != e) nan_at = min(nan_at, i);
    }
    const bool nan_sum = block_min_i(nan_at, sh) != 0x7fffffff;
    const uint64_t esum = block_sum(s, sh);
    inv = nan_sum ? NAN : 1.0f / (float)((double)esum / kFixE);
  }
  for (int i = tid; i < V; i += kThreads) p[i] *= inv;
  __syncthreads();

  // 2. top-k (tensor.c:390-396)
  if (a.top_k > 0 && a.top_k < V) {
    const float th = __uint_as_float(kth_largest(p, V, a.top_k, sh));
    for (int i = tid; i < V; i += kThreads)
      if (p[i] < th) p[i] = 0.f;
    __syncthreads();
  }

  // 3. top-p (tensor.c:398-417)
  if (a.top_p > 0.f && a.top_p < 1.0f) {
    const uint64_t target = top_p_target(a.top_p);
    const float cutoff = top_p_cutoff(p, V, target, sh);
    for (int i = tid; i < V; i += kThreads)
      if (p[i] < cutoff) p[i] = 0.f;
    __syncthreads();
  }

  // 4. renormalise (tensor.c:423-429); a NaN probability makes the sum NaN
  nan_at = 0x7fffffff;
  s = 0;
  for (int i = tid; i < V; i += kThreads) {
    const float v = p[i];
    s += fix(v);
    if (v != v) nan_at = min(nan_at, i);
  }
  const int first_nan = block_min_i(nan_at, sh);
  const uint64_t psum = block_sum(s, sh);
  if (first_nan == 0x7fffffff && psum > 0) {
    const float pinv = 1.0f / (float)((double)psum / kFix);
    for (int i = tid; i < V; i += kThreads) p[i] *= pinv;
  }
  __syncthreads();

  // 5. draw (tensor.c:341-343, 431-442): first i with r < cdf_i, i before any
  // NaN (a NaN term makes every later comparison false)
  const uint64_t st = advance(a.rng), rf = draw_fix(st);
  const int C = (V + kThreads - 1) / kThreads;   // contiguous chunk per thread
  const int i0 = min(tid * C, V), i1 = min(i0 + C, V);
  uint64_t cs = 0;
  for (int i = i0; i < i1; ++i) cs += fix(p[i]);
  // exclusive scan of the chunk sums over the workgroup
  uint64_t incl = cs;
  const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint64_t o = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += o;
  }
  __syncthreads();
  if (lane == kWave - 1) sh.u[wave] = incl;
  __syncthreads();
  uint64_t base = incl - cs;
  for (int w = 0; w < wave; ++w) base += sh.u[w];
  int found = 0x7fffffff;
  if (i0 < i1 && rf < base + cs) {
    uint64_t c = base;
    for (int i = i0; i < i1; ++i) {
      c += fix(p[i]);
      if (rf < c) {
        found = i;
        break;
      }
    }
  }
  found = block_min_i(found, sh);
  if (tid != 0) return;
  put_result(a, found < first_nan && found < V ? found : V - 1, st);
}

__global__ void __launch_bounds__(kThreads) k_sample(const SampleArgs a) {
  __shared__ Shared sh;
  sample_one_group<false>(a, sh);
}

// ---- many workgroups ---------------------------------------------------------
// Scratch of a row (SampleArgs::probs): p or e per entry, the boundary list or
// the candidates, the histogram, and the per-workgroup values.
struct Work {
  float* e;            // [V] softmax terms
  float* list;         // [V] values of the boundary bin (top-p), or [2 * kCand] candidates (index, e)
  uint64_t* hist;      // [kBins] counts of e (top-k) or sums of p (top-p) per bin
  uint64_t* esum;      // [nb] fixed-point sums of e
  uint64_t* psum;      // [nb] of the kept p, then of their renormalised values
  float* mx;           // [nb]
  uint32_t* nan;       // [nb] nonzero: a term is NaN
  uint32_t* count;     // [1] list entries
  float* cut;          // [2] cutoff, renormalisation factor
};
__host__ __device__ inline size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }
__host__ __device__ inline Work work_of(float* base, int V, size_t* bytes) {
  const int nb = (V + kTile - 1) / kTile;
  uint8_t* p = reinterpret_cast<uint8_t*>(base);
  size_t o = 0;
  auto take = [&](size_t n) {
    uint8_t* q = p + o;
    o += up256(n);
    return q;
  };
  Work w;
  w.e = reinterpret_cast<float*>(take(sizeof(float) * (size_t)V));
  w.list = reinterpret_cast<float*>(take(sizeof(float) * (size_t)(V > 2 * kCand ? V : 2 * kCand)));
  w.hist = reinterpret_cast<uint64_t*>(take(sizeof(uint64_t) * kBins));
  w.esum = reinterpret_cast<uint64_t*>(take(sizeof(uint64_t) * nb));
  w.psum = reinterpret_cast<uint64_t*>(take(sizeof(uint64_t) * nb));
  w.mx = reinterpret_cast<float*>(take(sizeof(float) * nb));
  w.nan = reinterpret_cast<uint32_t*>(take(sizeof(uint32_t) * nb));
  w.count = reinterpret_cast<uint32_t*>(take(sizeof(uint32_t)));
  w.cut = reinterpret_cast<float*>(take(2 * sizeof(float)));
  if (bytes) *bytes = o;
  return w;
}

// sum, maximum or or over a workgroup of W waves (red: W slots), in every thread
template <int W>
__device__ __forceinline__ uint64_t group_sum(uint64_t v, uint64_t* red) {
  v = wave_sum_u64(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  uint64_t t = 0;
#pragma unroll
  for (int i = 0; i < W; ++i) t += red[i];
  return t;
}
// sum of n values (the per-workgroup sums of an earlier launch)
template <int W>
__device__ __forceinline__ uint64_t total(const uint64_t* p, int n, uint64_t* red) {
  uint64_t v = 0;
  for (int i = threadIdx.x; i < n; i += W * kWave) v += p[i];
  return group_sum<W>(v, red);
}
template <int W>
__device__ __forceinline__ bool any_nan(const Work& w, int nb, uint64_t* red) {
  uint64_t v = 0;
  for (int i = threadIdx.x; i < nb; i += W * kWave) v += w.nan[i];
  return group_sum<W>(v, red) != 0;
}
// sum of v over the threads of a workgroup of W waves before this one; all: over every thread
template <int W>
__device__ __forceinline__ uint64_t sum_before(uint64_t v, uint64_t* red, uint64_t& all) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint64_t incl = v;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint64_t o = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += o;
  }
  __syncthreads();
  if (lane == 63) red[wave] = incl;
  __syncthreads();
  uint64_t before = incl - v;
  all = 0;
  for (int i = 0; i < W; ++i) {
    if (i < wave) before += red[i];
    all += red[i];
  }
  return before;
}
__device__ __forceinline__ float inv_of(uint64_t esum) { return 1.0f / (float)((double)esum / kFixE); }

constexpr int kTW = kTileThreads / kWave, kTK = kTile / kTileThreads;

// 1. the row's maximum of logit / temperature; the histogram starts at zero
__global__ void __launch_bounds__(kTileThreads) k_smp_max(const SampleArgs a) {
  __shared__ float red[kTW];
  const Work w = work_of(a.probs, a.V, nullptr);
  const int i0 = blockIdx.x * kTile + threadIdx.x;
  float mx = -FLT_MAX;
#pragma unroll
  for (int k = 0; k < kTK; ++k) {
    const float l = a.logits[min(i0 + k * kTileThreads, a.V - 1)];
    mx = fmaxf(mx, l != l ? -FLT_MAX : l / a.temperature);
  }
  mx = wave_max(mx);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
  for (int i = blockIdx.x * kTileThreads + threadIdx.x; i < kBins; i += gridDim.x * kTileThreads) w.hist[i] = 0;
  if (blockIdx.x == 0 && threadIdx.x == 0) *w.count = 0;
  __syncthreads();
  if (threadIdx.x == 0) w.mx[blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
}

// 2. the softmax terms, their sum, and (COUNT) how many fall into each bin
template <bool COUNT>
__global__ void __launch_bounds__(kTileThreads) k_smp_exp(const SampleArgs a) {
  __shared__ float redf[kTW];
  __shared__ uint64_t red[kTW];
  __shared__ uint32_t hist[COUNT ? kBins : 1];
  const Work w = work_of(a.probs, a.V, nullptr);
  const int tid = threadIdx.x;
  float l[kTK];
#pragma unroll
  for (int k = 0; k < kTK; ++k) l[k] = a.logits[min((int)blockIdx.x * kTile + k * kTileThreads + tid, a.V - 1)];
  float mx = -FLT_MAX;
  for (int i = tid; i < (int)gridDim.x; i += kTileThreads) mx = fmaxf(mx, w.mx[i]);
  mx = wave_max(mx);
  if ((tid & 63) == 0) redf[tid >> 6] = mx;
  if constexpr (COUNT)
    for (int i = tid; i < kBins; i += kTileThreads) hist[i] = 0;
  __syncthreads();
  mx = fmaxf(fmaxf(redf[0], redf[1]), fmaxf(redf[2], redf[3]));
  uint64_t s = 0;
  bool nan = false;
#pragma unroll
  for (int k = 0; k < kTK; ++k) {
    const int i = blockIdx.x * kTile + k * kTileThreads + tid;
    if (i >= a.V) break;
    const float x = l[k] != l[k] ? -FLT_MAX : l[k] / a.temperature;
    const float e = expf(x - mx);
    w.e[i] = e;
    s += e > 0.f ? (uint64_t)((double)e * kFixE) : 0ull;   // e <= 1
    nan = nan || e != e;
    if constexpr (COUNT)
      if (e > 0.f) atomicAdd(&hist[__float_as_uint(e) >> 19], 1u);
  }
  s = group_sum<kTW>(s, red);
  const bool nans = group_sum<kTW>(nan ? 1 : 0, red) != 0;
  if (tid == 0) {
    w.esum[blockIdx.x] = s;
    w.nan[blockIdx.x] = nans;
  }
  if constexpr (COUNT)
    for (int i = tid; i < kBins; i += kTileThreads)
      if (hist[i]) atomicAdd(reinterpret_cast<unsigned long long*>(&w.hist[i]), (unsigned long long)hist[i]);
}

// The largest bin at which the sum of hist over it and the bins above reaches
// target, or -1; above: the sum over the bins above it (over all when -1).
// 256 threads, 8 bins each.
__device__ int find_bin(const uint64_t* hist, uint64_t target, uint64_t* red, int* sel, uint64_t* sel_above, uint64_t& above) {
  static_assert(kBins == 8 * kTileThreads, "eight bins per thread");
  const int tid = threadIdx.x, top = kBins - 1 - 8 * tid;   // thread 0 takes the highest bins
  uint64_t h[8], s = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    h[k] = hist[top - k];
    s += h[k];
  }
  uint64_t incl = s;   // inclusive scan over the workgroup
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const uint64_t o = __shfl_up(incl, off, kWave);
    if ((tid & 63) >= off) incl += o;
  }
  if (tid == 0) *sel = -1;
  if ((tid & 63) == 63) red[tid >> 6] = incl;
  __syncthreads();
  uint64_t base = incl - s;
  for (int i = 0; i < tid >> 6; ++i) base += red[i];
  if (tid == kTileThreads - 1) *sel_above = base + s;   // everything; replaced below when a bin reaches the target
  __syncthreads();
  if (base < target && base + s >= target) {
    int k = 0;
    while (base + h[k] < target) base += h[k++];
    *sel = top - k;
    *sel_above = base;
  }
  __syncthreads();
  above = *sel_above;
  return *sel;
}

// ---- 0 < top_k <= kMaxTopK: the candidates ---------------------------------
// 3. every term that may belong to the k largest: those of the bin the k-th
// falls into and above (and a few rounding steps below: their p may equal
// the k-th's). Terms of 0 are left out: their probability is 0 in any case.
__global__ void __launch_bounds__(kTileThreads) k_smp_gather(const SampleArgs a) {
  __shared__ uint64_t red[kTW], sa;
  __shared__ int sel;
  const Work w = work_of(a.probs, a.V, nullptr);
  float e[kTK];
#pragma unroll
  for (int k = 0; k < kTK; ++k) e[k] = w.e[min((int)blockIdx.x * kTile + k * kTileThreads + (int)threadIdx.x, a.V - 1)];
  uint64_t above;
  const int bin = find_bin(w.hist, (uint64_t)a.top_k, red, &sel, &sa, above);
  const uint32_t low = bin <= 0 ? 1u : ((uint32_t)bin << 19) - 8u;
#pragma unroll
  for (int k = 0; k < kTK; ++k) {
    const int i = blockIdx.x * kTile + k * kTileThreads + threadIdx.x;
    if (i < a.V && e[k] > 0.f && __float_as_uint(e[k]) >= low) {
      const uint32_t at = atomicAdd(w.count, 1u);
      if (at < (uint32_t)kCand) {
        w.list[2 * at] = __int_as_float(i);
        w.list[2 * at + 1] = e[k];
      }
    }
  }
}

// v[0 .. n - 1], n a power of two up to kCand, in descending order (bitonic).
// The pairs of a step up to 64 apart lie within one wave's 128 entries, so
// only wider steps meet at a barrier.
__device__ void sort_descending(uint64_t* v, int n) {
  __syncthreads();
  for (int k = 2; k <= n; k <<= 1)
    for (int j = k >> 1; j > 0; j >>= 1) {
      for (int t = threadIdx.x; t < n / 2; t += kThreads) {
        const int i = ((t & ~(j - 1)) << 1) | (t & (j - 1));
        const uint64_t x = v[i], y = v[i + j];
        if ((x < y) == ((i & k) == 0)) {
          v[i] = y;
          v[i + j] = x;
        }
      }
      if (j > 64 || (j == 1 && k > 64))   // (after j = 1 the next step's pairs are k apart)
        __syncthreads();
      else
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  __syncthreads();
}
__device__ __forceinline__ int pow2_from(int n) {   // the power of two at or above n
  int p = 2;
  while (p < n) p <<= 1;
  return p;
}

// 4. the k-th largest, the top-p cutoff, the renormalisation and the draw over
// the candidates, whose order in the list does not matter. Up to kPairs are each
// compared with all others by 8 threads, which takes the square of their
// number. More are sorted, by probability, then what is kept by index, with
// running sums over each order. Calls over 3000 entries, in pairs and sorted:
// top_k 200 39 and 46 us, 300 50 and 50, 1000 463 and 66 (one workgroup: 84).
// More than kCand (ties, a flat row): the whole row in this workgroup, from its
// softmax terms on; with room for 4096, 3000 equal entries took 100 us, 79 so.
__global__ void __launch_bounds__(kThreads) k_smp_topk(const SampleArgs a) {
  __shared__ Shared sh;
  __shared__ uint64_t ent[kCand];   // sorted: probability (its bits) << 32 | index
  __shared__ float p[kPairs];       // in pairs
  __shared__ int idx[kPairs];
  __shared__ uint32_t th, cut;
  __shared__ int found;
  const Work w = work_of(a.probs, a.V, nullptr);
  const int tid = threadIdx.x, nb = (a.V + kTile - 1) / kTile;
  const int n = (int)*w.count;
  const bool nan = any_nan<kWaves>(w, nb, sh.u);
  const float inv = inv_of(total<kWaves>(w.esum, nb, sh.u));
  if (n > kCand) {
    sample_one_group<true>(a, sh, nan ? NAN : inv);
    return;
  }
  const uint64_t st = advance(a.rng), rf = draw_fix(st);
  const bool topp = a.top_p > 0.f && a.top_p < 1.0f;
  const uint64_t target = top_p_target(a.top_p);
  const bool sorted = n > kPairs;
  const int pn = sorted ? pow2_from(n) : n;
  for (int i = tid; i < pn; i += kThreads) {
    const float q = i < n ? w.list[2 * i + 1] * inv : 0.f;
    const uint32_t at = i < n ? __float_as_uint(w.list[2 * i]) : 0u;
    if (sorted) {
      ent[i] = (uint64_t)__float_as_uint(q) << 32 | at;
    } else {
      p[i] = q;
      idx[i] = (int)at;
    }
  }
  if (tid == 0) {
    th = 0;
    cut = 0;
    found = 0x7fffffff;
  }
  __syncthreads();
  auto ep = [&](int i) { return __uint_as_float((uint32_t)(ent[i] >> 32)); };
  const int part = tid & 7;
  // f(i) for i < m, by the 8 threads of an aligned group
  auto each = [&](int m, auto f) {
    for (int i = tid >> 3; i < m; i += kThreads / 8) f(i);
  };
  auto sum8u = [](uint64_t v) {
    v += __shfl_xor(v, 1, kWave);
    v += __shfl_xor(v, 2, kWave);
    return v + __shfl_xor(v, 4, kWave);
  };
  // the running sum of v(i) over i < m (at most kCand) in order: f(i, sum through i - 1, v(i))
  auto running = [&](int m, auto v, auto f) {
    constexpr int C = kCand / kThreads;
    uint64_t x[C], s = 0, all;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int i = C * tid + c;
      x[c] = i < m ? v(i) : 0ull;
      s += x[c];
    }
    uint64_t before = sum_before<kWaves>(s, sh.u, all);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (C * tid + c < m) f(C * tid + c, before, x[c]);
      before += x[c];
    }
    __syncthreads();
  };
  // what is left of m of them in pairs, given the least that stays and the
  // factor: the first index whose cumulative probability exceeds r
  auto draw_pairs = [&](int m, float low, float pinv) {
    each(m, [&](int i) {
      uint64_t c = 0;
      for (int j = part; j < m; j += 8) c += p[j] >= low && idx[j] <= idx[i] ? fix(p[j] * pinv) : 0ull;
      c = sum8u(c);
      if (part == 0 && p[i] >= low && rf < c) atomicMin(&found, idx[i]);
    });
  };
  auto factor = [&](uint64_t s) {
    s = group_sum<kWaves>(s, sh.u);
    return s > 0 ? 1.0f / (float)((double)s / kFix) : 1.0f;
  };
  uint64_t s = 0;
  if (!sorted) {
    each(n, [&](int i) {   // the k-th largest p (p >= 0: its bits order like its value)
      uint64_t c = 0;      // greater ones, and (high half) equal ones
      for (int j = part; j < n; j += 8) c += p[j] > p[i] ? 1ull : p[j] == p[i] ? 1ull << 32 : 0ull;
      c = sum8u(c);
      const uint32_t gt = (uint32_t)c, eq = (uint32_t)(c >> 32);
      if (part == 0 && gt < (uint32_t)a.top_k && gt + eq >= (uint32_t)a.top_k) th = __float_as_uint(p[i]);
    });
    __syncthreads();
    const float tk = __uint_as_float(th);
    if (topp) {
      each(n, [&](int i) {   // the largest p whose sum with those above it reaches the target
        uint64_t v = 0;
        for (int j = part; j < n; j += 8) v += p[j] >= tk && p[j] >= p[i] ? fix(p[j]) : 0ull;
        v = sum8u(v);
        if (part == 0 && p[i] >= tk && v >= target) atomicMax(&cut, __float_as_uint(p[i]));
      });
      __syncthreads();
    }
    const float low = fmaxf(tk, __uint_as_float(cut));
    for (int i = tid; i < n; i += kThreads) s += p[i] >= low ? fix(p[i]) : 0ull;
    draw_pairs(n, low, factor(s));
  } else {
    sort_descending(ent, pn);
    const float tk = n >= a.top_k ? ep(a.top_k - 1) : 0.f;
    if (topp)
      running(n, [&](int i) { return ep(i) >= tk ? fix(ep(i)) : 0ull; },
              [&](int i, uint64_t before, uint64_t v) {   // the first to reach the target
                if (before < target && before + v >= target) cut = (uint32_t)(ent[i] >> 32);
              });
    const float low = fmaxf(tk, __uint_as_float(cut));
    uint64_t kept = 0;
    for (int i = tid; i < n; i += kThreads) {
      s += ep(i) >= low ? fix(ep(i)) : 0ull;
      kept += ep(i) >= low;
    }
    const float pinv = factor(s);
    const int m = (int)group_sum<kWaves>(kept, sh.u);   // they come first
    if (m > kPairs) {
      const int pm = pow2_from(m);
      __syncthreads();
      for (int i = tid; i < pm; i += kThreads) ent[i] = i < m ? ~ent[i] << 32 | ent[i] >> 32 : 0ull;   // ~index, p
      sort_descending(ent, pm);
      running(m, [&](int i) { return fix(__uint_as_float((uint32_t)ent[i]) * pinv); },
              [&](int i, uint64_t before, uint64_t v) {
                if (rf < before + v) atomicMin(&found, (int)~(uint32_t)(ent[i] >> 32));
              });
    } else {
      if (tid < m) {
        p[tid] = ep(tid);
        idx[tid] = (int)(uint32_t)ent[tid];
      }
      __syncthreads();
      draw_pairs(m, low, pinv);
    }
  }
  __syncthreads();
  if (tid == 0) put_result(a, !nan && found < a.V ? found : a.V - 1, st);
}

// ---- no top-k: the whole distribution ----------------------------------------
// 3. the probabilities and (HIST) their sums per bin, or their whole sum
template <bool HIST>
__global__ void __launch_bounds__(kTileThreads) k_smp_prob(const SampleArgs a) {
  __shared__ uint64_t red[kTW];
  __shared__ uint64_t hist[HIST ? kBins : 1];
  const Work w = work_of(a.probs, a.V, nullptr);
  const int tid = threadIdx.x;
  if constexpr (HIST)
    for (int i = tid; i < kBins; i += kTileThreads) hist[i] = 0;
  const float inv = inv_of(total<kTW>(w.esum, gridDim.x, red));
  uint64_t s = 0;
#pragma unroll
  for (int k = 0; k < kTK; ++k) {
    const int i = blockIdx.x * kTile + k * kTileThreads + tid;
    if (i >= a.V) break;
    const float p = w.e[i] * inv;
    w.e[i] = p;
    s += fix(p);
    if constexpr (HIST)
      if (p > 0.f)
        atomicAdd(reinterpret_cast<unsigned long long*>(&hist[__float_as_uint(p) >> 19]), (unsigned long long)fix(p));
  }
  s = group_sum<kTW>(s, red);
  if (tid == 0) w.psum[blockIdx.x] = s;
  if constexpr (HIST)
    for (int i = tid; i < kBins; i += kTileThreads)
      if (hist[i]) atomicAdd(reinterpret_cast<unsigned long long*>(&w.hist[i]), (unsigned long long)hist[i]);
}

// 4. the values of the bin the top-p cutoff lies in
__global__ void __launch_bounds__(kTileThreads) k_smp_boundary(const SampleArgs a) {
  __shared__ uint64_t red[kTW], sa;
  __shared__ int sel;
  const Work w = work_of(a.probs, a.V, nullptr);
  float p[kTK];
#pragma unroll
  for (int k = 0; k < kTK; ++k) p[k] = w.e[min((int)blockIdx.x * kTile + k * kTileThreads + (int)threadIdx.x, a.V - 1)];
  uint64_t above;
  const int bin = find_bin(w.hist, top_p_target(a.top_p), red, &sel, &sa, above);
#pragma unroll
  for (int k = 0; k < kTK; ++k) {
    const int i = blockIdx.x * kTile + k * kTileThreads + threadIdx.x;
    if (i < a.V && p[k] > 0.f && (int)(__float_as_uint(p[k]) >> 19) == bin) w.list[atomicAdd(w.count, 1u)] = p[k];
  }
}

// 5. the cutoff within that bin, and the renormalisation (CUT false: of everything)
template <bool CUT>
__global__ void __launch_bounds__(kTileThreads) k_smp_cutoff(const SampleArgs a) {
  __shared__ uint64_t red[kTW], sa, bins[256];
  __shared__ int sel;
  const Work w = work_of(a.probs, a.V, nullptr);
  const int tid = threadIdx.x, nb = (a.V + kTile - 1) / kTile;
  uint64_t s = 0;
  uint32_t prefix = 0;
  if constexpr (CUT) {
    const uint64_t target = top_p_target(a.top_p);
    uint64_t above;
    const int bin = find_bin(w.hist, target, red, &sel, &sa, above);
    s = above;   // everything when no bin reaches the target: the cutoff is 0
    if (bin >= 0) {
      // the remaining 19 bits of the key, 7, 6 and 6 at a time
      const int n = (int)*w.count;
      prefix = (uint32_t)bin << 19;
      uint32_t mask = ~0u << 19;
      for (int shift = 12; shift >= 0; shift -= 6) {
        const uint32_t width = shift == 12 ? 128 : 64;
        __syncthreads();
        bins[tid] = 0;
        __syncthreads();
        for (int i = tid; i < n; i += kTileThreads) {
          const uint32_t u = __float_as_uint(w.list[i]);
          if ((u & mask) == prefix)
            atomicAdd(reinterpret_cast<unsigned long long*>(&bins[(u >> shift) & (width - 1)]),
                      (unsigned long long)fix(__uint_as_float(u)));
        }
        __syncthreads();
        if (tid == 0) {
          int b = (int)width - 1;
          uint64_t acc = above;
          for (; b > 0; --b) {   // some bin reaches the target: their sum does
            if (acc + bins[b] >= target) break;
            acc += bins[b];
          }
          sel = b;
          sa = acc;
        }
        __syncthreads();
        prefix |= (uint32_t)sel << shift;
        mask |= (width - 1) << shift;
        above = sa;
      }
      // all keys of the last bin are equal: its sum is the cutoff's own
      s = above + bins[sel];
    }
  } else {
    s = total<kTW>(w.psum, nb, red);
  }
  if (tid == 0) {
    w.cut[0] = __uint_as_float(prefix);
    w.cut[1] = s > 0 ? 1.0f / (float)((double)s / kFix) : 1.0f;
  }
}

// 6. the renormalised sum of each tile
__global__ void __launch_bounds__(kTileThreads) k_smp_sums(const SampleArgs a) {
  __shared__ uint64_t red[kTW];
  const Work w = work_of(a.probs, a.V, nullptr);
  const float low = w.cut[0], pinv = w.cut[1];
  uint64_t s = 0;
#pragma unroll
  for (int k = 0; k < kTK; ++k) {
    const int i = blockIdx.x * kTile + k * kTileThreads + threadIdx.x;
    const float p = w.e[min(i, a.V - 1)];
    s += i < a.V && p >= low ? fix(p * pinv) : 0ull;
  }
  s = group_sum<kTW>(s, red);
  if (threadIdx.x == 0) w.psum[blockIdx.x] = s;
}

// 7. the tile the draw falls into, and the entry in it
__global__ void __launch_bounds__(kThreads) k_smp_draw(const SampleArgs a) {
  __shared__ uint64_t red[kWaves], base;
  __shared__ int tile, found;
  const Work w = work_of(a.probs, a.V, nullptr);
  const int tid = threadIdx.x, nb = (a.V + kTile - 1) / kTile;
  const uint64_t st = advance(a.rng), rf = draw_fix(st);
  const bool nan = any_nan<kWaves>(w, nb, red);
  const float low = w.cut[0], pinv = w.cut[1];
  if (tid == 0) {
    tile = -1;
    found = 0x7fffffff;
  }
  uint64_t done = 0;
  for (int b0 = 0; b0 < nb; b0 += kThreads) {
    const uint64_t v = b0 + tid < nb ? w.psum[b0 + tid] : 0ull;
    uint64_t all;
    const uint64_t before = done + sum_before<kWaves>(v, red, all);
    if (v > 0 && rf >= before && rf < before + v) {
      tile = b0 + tid;
      base = before;
    }
    done += all;
    __syncthreads();
  }
  const int t = tile;
  if (t >= 0) {   // uniform
    const int i = t * kTile + tid;
    const float p = w.e[min(i, a.V - 1)];
    const uint64_t v = i < a.V && p >= low ? fix(p * pinv) : 0ull;
    uint64_t all;
    const uint64_t c = base + sum_before<kWaves>(v, red, all) + v;
    if (i < a.V && rf < c) atomicMin(&found, i);
  }
  __syncthreads();
  if (tid == 0) put_result(a, !nan && found < a.V ? found : a.V - 1, st);
}
static_assert(kPairs <= kThreads, "k_smp_topk: a thread per pair's end");
static_assert(kTile == kThreads, "k_smp_draw: one entry per thread");

}  // namespace

size_t sample_scratch_bytes(int V) {
  if (V <= kOneGroup) return sizeof(float) * (size_t)V;
  size_t bytes = 0;
  work_of(nullptr, V, &bytes);
  return bytes;
}

hipError_t launch_sample(const SampleArgs& a, hipStream_t s) {
  if (a.V <= 0 || !a.logits || !a.probs || !a.out || !a.rng_out || !(a.temperature > 0.f) ||
      (a.tokens && !a.dpos))
    return hipErrorInvalidValue;
  // Rows of up to kOneGroup entries (one per thread) and a top_k past the
  // candidates' space stay with one workgroup. The whole call, one workgroup
  // and many: 128256 entries with top_k 40 and top_p 0.95 407 and 33 us, with
  // top_p alone 341 and 56 us, with neither 200 and 36 us; 4097 entries 98 and
  // 30, 73 and 46, 41 and 35 us. What remains is four (six) launches and the
  // wait for them.
  const bool topk = a.top_k > 0 && a.top_k < a.V, topp = a.top_p > 0.f && a.top_p < 1.0f;
  if (a.V <= kOneGroup || (topk && a.top_k > kMaxTopK)) {
    hipLaunchKernelGGL(k_sample, dim3(1), dim3(kThreads), 0, s, a);
    return hipGetLastError();
  }
  const dim3 nb((a.V + kTile - 1) / kTile), th(kTileThreads);
  hipLaunchKernelGGL(k_smp_max, nb, th, 0, s, a);
  if (topk) {
    hipLaunchKernelGGL(k_smp_exp<true>, nb, th, 0, s, a);
    hipLaunchKernelGGL(k_smp_gather, nb, th, 0, s, a);
    hipLaunchKernelGGL(k_smp_topk, dim3(1), dim3(kThreads), 0, s, a);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_smp_exp<false>, nb, th, 0, s, a);
  if (topp) {
    hipLaunchKernelGGL(k_smp_prob<true>, nb, th, 0, s, a);
    hipLaunchKernelGGL(k_smp_boundary, nb, th, 0, s, a);
    hipLaunchKernelGGL(k_smp_cutoff<true>, dim3(1), th, 0, s, a);
  } else {
    hipLaunchKernelGGL(k_smp_prob<false>, nb, th, 0, s, a);
    hipLaunchKernelGGL(k_smp_cutoff<false>, dim3(1), th, 0, s, a);
  }
  hipLaunchKernelGGL(k_smp_sums, nb, th, 0, s, a);
  hipLaunchKernelGGL(k_smp_draw, dim3(1), dim3(kThreads), 0, s, a);
  return hipGetLastError();
}

}  // namespace ssk
