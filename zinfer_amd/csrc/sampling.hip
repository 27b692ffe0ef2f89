// Sampling on the device with the reference's order of operations
// (src/sampling/sampler.zig:18-91): penalties on seen tokens, the k largest adjusted logits
// in descending order (lower id first among equals), exp((l / T) - max) in 32-bit with
// 64-bit sums, the min-p prefix, the top-p prefix on the renormalised kept set, then the
// draw u * kept_sum walked down the candidates.  One workgroup per row; k <= 1024.
#include "zf_common.h"

#define SMP_THREADS 1024
#define SMP_MAX_K 1024

// order-preserving map float -> uint32 (larger float, larger key)
__device__ __forceinline__ uint32_t float_key(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// ---------------------------------------------------------------- penalties, in place
// For every (row, token, count) triple: repetition (negative logits multiplied, others
// divided), presence, frequency, in this order (sampler.zig:186-201).
__global__ void apply_penalties_kernel(float* __restrict__ logits, const int* __restrict__ rows,
                                       const int* __restrict__ tokens,
                                       const int* __restrict__ counts,
                                       const float* __restrict__ params, int n, int V) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int row = rows[i];
  const float rep = params[row * 3 + 0], pres = params[row * 3 + 1], freq = params[row * 3 + 2];
  float* p = logits + (size_t)row * V + tokens[i];
  float a = *p;
  if (rep > 0.f && rep != 1.f) a = a < 0.f ? a * rep : a / rep;
  a -= pres;
  a -= (float)counts[i] * freq;
  *p = a;
}

extern "C" int zf_apply_penalties(float* logits, const int* rows, const int* tokens,
                                  const int* counts, const float* params, int n, int V,
                                  hipStream_t stream) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(apply_penalties_kernel, dim3((n + 255) / 256), dim3(256), 0, stream, logits,
                     rows, tokens, counts, params, n, V);
  ZF_CHECK_LAUNCH();
}

// ---------------------------------------------------------------- top-k sampling
// params per row: temperature, top_p, min_p (float), top_k (int), u (double, in [0, 1)).
struct SampleRow {
  float temperature, top_p, min_p;
  int top_k;
  double u;
};

// One pass of a radix select, by the first wave: the bin (from the top) in which the s_remaining-th
// largest of the counted keys lies; the prefix takes the bin's 8 bits, s_remaining becomes the rank
// within the bin.  A lane holds four bins; what lies above its own comes from the lanes behind it.
__device__ __forceinline__ void narrow(const unsigned* hist, unsigned prefix, int shift,
                                       unsigned& s_prefix, unsigned& s_remaining) {
  if (threadIdx.x >= ZF_WAVE) return;
  const int lane = threadIdx.x;
  const unsigned want = s_remaining;
  unsigned h[4], above = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) above += h[i] = hist[4 * lane + i];
  const unsigned own = above;
#pragma unroll
  for (int off = 1; off < ZF_WAVE; off <<= 1) {
    const unsigned v = __shfl_down(above, off, ZF_WAVE);
    if (lane + off < ZF_WAVE) above += v;
  }
  above -= own;                              // keys in the bins of the lanes behind this one
  // (all lanes' bins together hold at least `want` keys, so exactly one bin takes it)
#pragma unroll
  for (int i = 3; i >= 0; --i) {
    if (above < want && above + h[i] >= want) {
      s_prefix = prefix | ((unsigned)(4 * lane + i) << shift);
      s_remaining = want - above;
    }
    above += h[i];
  }
}

// A workgroup a row.  Two passes over the row do for the usual k: the first leaves every thread
// with the largest of its 1/1024 of the row, the k-th largest of those 1024 is a bound that at least
// k elements reach and, with k elements scattered over the row, few more, and the second collects
// what reaches it; sorted by (value, id) the first k of these are the answer.  Only where more than
// 1024 elements reach the bound (k in the hundreds, a row of equal logits) the k-th key is found by
// a radix select over the whole row and gathered in id order.  What bounds it: one compute unit
// draws a row of 152 k logits in about 8 us a pass.  Measured (V = 151936, k = 50, 4 rows): 307 us with
// the radix select alone (six passes, a thread walking the bins), now 29.
__global__ __launch_bounds__(SMP_THREADS) void sample_topk_kernel(
    const float* __restrict__ logits, const SampleRow* __restrict__ params,
    int* __restrict__ out, int V) {
  __shared__ unsigned hist[256];
  __shared__ unsigned s_prefix, s_remaining;
  __shared__ float cval[SMP_MAX_K];
  __shared__ int cidx[SMP_MAX_K];
  __shared__ unsigned scan[SMP_THREADS];
  __shared__ unsigned s_count;
  const float* row = logits + (size_t)blockIdx.x * V;
  const SampleRow prm = params[blockIdx.x];
  const int tid = threadIdx.x;
  int k = prm.top_k <= 0 || prm.top_k > V ? V : prm.top_k;
  if (k > SMP_MAX_K) k = SMP_MAX_K;     // the host refuses such rows before launching

  // f(value, id) for the thread's part of the row, until enough(), which is asked every eight loads
  auto each = [&](auto&& f, auto&& enough) {
    if (V % 4 == 0 && ((uintptr_t)row & 15) == 0) {
      for (int i0 = tid; i0 < V / 4; i0 += 8 * SMP_THREADS) {
        float4 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (i0 + u * SMP_THREADS < V / 4) v[u] = ((const float4*)row)[i0 + u * SMP_THREADS];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          const int i = i0 + u * SMP_THREADS;
          if (i >= V / 4) break;
          f(v[u].x, 4 * i);
          f(v[u].y, 4 * i + 1);
          f(v[u].z, 4 * i + 2);
          f(v[u].w, 4 * i + 3);
        }
        if (enough()) break;
      }
    } else {
      for (int i = tid; i < V; i += SMP_THREADS) f(row[i], i);
    }
  };
  if (tid == 0) s_count = 0;
  uint32_t mine = 0;                         // (no float has the key 0 but a NaN, which none may reach)
  each([&](float v, int) { mine = max(mine, float_key(v)); }, [] { return false; });
  if (tid == 0) {
    s_prefix = 0;
    s_remaining = (unsigned)min(k, SMP_THREADS);
  }
  for (int pass = 0; pass < 4; ++pass) {
    const int shift = 24 - 8 * pass;
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
    const unsigned prefix = s_prefix;
    const unsigned mask = pass == 0 ? 0u : (0xffffffffu << (shift + 8));
    if ((mine & mask) == prefix) atomicAdd(&hist[(mine >> shift) & 0xff], 1u);
    __syncthreads();
    narrow(hist, prefix, shift, s_prefix, s_remaining);
    __syncthreads();
  }
  const uint32_t bound = s_prefix;
  each([&](float v, int i) {
    if (float_key(v) >= bound) {
      const unsigned at = atomicAdd(&s_count, 1u);
      if (at < SMP_MAX_K) {
        cval[at] = v;
        cidx[at] = i;
      }
    }
  }, [&] { return *(volatile unsigned*)&s_count > SMP_MAX_K; });      // (they go to the radix select)
  __syncthreads();
  int found = (int)s_count;
  __syncthreads();
  if (found > SMP_MAX_K) {
    // radix select: the key of the k-th largest element, 8 bits a pass from the top
    if (tid == 0) {
      s_prefix = 0;
      s_remaining = (unsigned)k;
    }
    for (int pass = 0; pass < 4; ++pass) {
      const int shift = 24 - 8 * pass;
      if (tid < 256) hist[tid] = 0;
      __syncthreads();
      const unsigned prefix = s_prefix;
      const unsigned mask = pass == 0 ? 0u : (0xffffffffu << (shift + 8));
      for (int i = tid; i < V; i += SMP_THREADS) {
        const uint32_t key = float_key(row[i]);
        if ((key & mask) == prefix) atomicAdd(&hist[(key >> shift) & 0xff], 1u);
      }
      __syncthreads();
      narrow(hist, prefix, shift, s_prefix, s_remaining);
      __syncthreads();
    }
    const uint32_t kth = s_prefix;
    const unsigned want_equal = s_remaining;

    // gather: everything above the k-th key, then the lowest ids among those equal to it.
    //    Threads own contiguous index ranges so that the block-wide scans are in id order.
    const int per = (V + SMP_THREADS - 1) / SMP_THREADS;
    const int lo = tid * per, hi = min(V, lo + per);
    unsigned n_gt = 0, n_eq = 0;
    for (int i = lo; i < hi; ++i) {
      const uint32_t key = float_key(row[i]);
      n_gt += key > kth;
      n_eq += key == kth;
    }
    // exclusive scans of n_gt and n_eq over the threads
    unsigned off_gt, off_eq, total_gt;
    scan[tid] = n_gt;
    __syncthreads();
    for (int d = 1; d < SMP_THREADS; d <<= 1) {
      const unsigned v = tid >= d ? scan[tid - d] : 0;
      __syncthreads();
      scan[tid] += v;
      __syncthreads();
    }
    off_gt = scan[tid] - n_gt;
    total_gt = scan[SMP_THREADS - 1];
    __syncthreads();
    scan[tid] = n_eq;
    __syncthreads();
    for (int d = 1; d < SMP_THREADS; d <<= 1) {
      const unsigned v = tid >= d ? scan[tid - d] : 0;
      __syncthreads();
      scan[tid] += v;
      __syncthreads();
    }
    off_eq = scan[tid] - n_eq;
    __syncthreads();
    for (int i = lo; i < hi; ++i) {
      const float v = row[i];
      const uint32_t key = float_key(v);
      if (key > kth) {
        cval[off_gt] = v;
        cidx[off_gt] = i;
        ++off_gt;
      } else if (key == kth) {
        if (off_eq < want_equal) {
          cval[total_gt + off_eq] = v;
          cidx[total_gt + off_eq] = i;
        }
        ++off_eq;
      }
    }
    if (tid == 0) s_count = total_gt + want_equal;      // == k
    __syncthreads();
  }
  const int n = min(k, (int)s_count);

  // sorted: larger first, the lower id among equals (bitonic over the next power of two).  `zeros`:
  // -0 and 0 are equal, as the reference compares; which elements are among the k goes by the
  // keys, where -0 lies below 0.
  auto sort = [&](int have, bool zeros) {
    int slots = ZF_WAVE;
    while (slots < have) slots <<= 1;
    if (tid >= have && tid < slots) {
      cval[tid] = __uint_as_float(0xffffffffu);         // the lowest key
      cidx[tid] = 0x7fffffff;
    }
    __syncthreads();
    auto key_of = [&](float v) { return float_key(zeros && v == 0.f ? 0.f : v); };
    for (int size = 2; size <= slots; size <<= 1) {
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        const int i = tid, jj = tid ^ stride;
        if (jj > i && i < slots) {
          const bool up = (i & size) == 0;      // this half ends up in "before" order
          const float vi = cval[i], vj = cval[jj];
          const int ii = cidx[i], ij = cidx[jj];
          const uint32_t ki = key_of(vi), kj = key_of(vj);
          const bool i_before_j = ki > kj || (ki == kj && ii < ij);
          if (i_before_j != up) {
            cval[i] = vj;
            cval[jj] = vi;
            cidx[i] = ij;
            cidx[jj] = ii;
          }
        }
        __syncthreads();
      }
    }
  };
  static_assert(SMP_THREADS == SMP_MAX_K, "a thread an element");
  if (found <= SMP_MAX_K) sort(found, false);           // (the gather above left exactly the k)
  const bool low_zero = tid < n && __float_as_uint(cval[tid]) == 0x80000000u;
  if (__syncthreads_or(low_zero) || found > SMP_MAX_K) sort(n, true);

  // the reference's walk: 32-bit exponentials, then, by one thread, 64-bit sums
  const float T = prm.temperature, max_scaled = cval[0] / T;
  __syncthreads();
  if (tid < n) cval[tid] = expf(cval[tid] / T - max_scaled);
  __syncthreads();
  if (tid == 0) {
    double sum = 0.0;
#pragma unroll 8
    for (int i = 0; i < n; ++i) sum += (double)cval[i];
    int result = cidx[0];
    if (sum > 0.0) {
      int keep = n;
      const float min_p = fminf(fmaxf(prm.min_p, 0.f), 1.f);
      if (min_p > 0.f) {
        const float thr = cval[0] * min_p;
        keep = 0;
        while (keep < n && cval[keep] >= thr) ++keep;
        if (keep < 1) keep = 1;
        sum = 0.0;
        for (int i = 0; i < keep; ++i) sum += (double)cval[i];
      }
      const float top_p = fminf(fmaxf(prm.top_p, 0.f), 1.f);
      if (top_p < 1.f) {
        double cum = 0.0;
        int np = 0;
        while (np < keep) {
          cum += (double)cval[np] / sum;
          ++np;
          if (cum >= (double)top_p) break;
        }
        if (np < 1) np = 1;
        if (np < keep) keep = np;
      }
      double kept = 0.0;
      for (int i = 0; i < keep; ++i) kept += (double)cval[i];
      if (kept > 0.0) {
        double thr = prm.u * kept;
        result = cidx[keep - 1];
        for (int i = 0; i < keep; ++i) {
          thr -= (double)cval[i];
          if (thr <= 0.0) {
            result = cidx[i];
            break;
          }
        }
      }
    }
    out[blockIdx.x] = result;
  }
}

extern "C" int zf_sample_topk(const float* logits, const void* params, int* out, int n, int V,
                              hipStream_t stream) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(sample_topk_kernel, dim3(n), dim3(SMP_THREADS), 0, stream, logits,
                     (const SampleRow*)params, out, V);
  ZF_CHECK_LAUNCH();
}
