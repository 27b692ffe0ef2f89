// A feed-forward layer made of many small experts, of which every token uses a few.
//
//   router:  z = R h + r            32-bit; the `top` largest z are chosen (the lower index
//            wins a tie), and their weights are the soft-max over the chosen z alone;
//            or (scoring 1) s = sigmoid(z), the choice goes by s + correction among the experts
//            of the best groups (a group of neighbours is marked by its two largest choice
//            scores added), and the weights are the chosen s over their sum (+ 1e-20)
//   expert:  g = min(Wg h, limit), u = clamp(Wu h, -limit, limit)      (limit <= 0: no clamp)
//            y = g * sigmoid(alpha * g) * (u + shift)
//            out = Wd y
//            or, without a gate: y = act(Wu h) with one of the plain activations
//   layer:   out[t] = sum over the chosen experts of weight * expert(h[t])
//
// Expert matrices are stacked: gate_up [E, 2 * ff, W] (an expert's gate rows, then its up
// rows) and down [E, W, ff].  Three kernels that stream the weights of the chosen experts
// token by token (float32, and bfloat16 sizes that the kernels for few tokens further down do
// not take); every token's result depends on that token alone and its sums run in a
// fixed order, so a token gives the same bits whatever else is in the batch:
//
//  * moe_route         a workgroup per four tokens, or sixteen (route16_takes)
//  * moe_gate_up       grid (token * slot, groups of outputs): y[t, slot, :] of the expert in
//                      that slot, the token's row staged in LDS as 32-bit numbers
//  * moe_down          grid (token, groups of outputs): out[t, n] (=, or += into) the weighted
//                      sum over the slots in slot order, 32-bit
//
// With `ids` null every token uses expert 0 with weight 1 (an expert that all tokens share).
#include <type_traits>

#include "zf_common.h"

#define MOE_MAX_EXPERTS 1024

#define MOE_ROUTE_TOKENS 4     // tokens a workgroup routes: one wave each for the choice
#define MOE_ROUTE_WAVES 16     // waves of the workgroup: the experts' logits are dealt over them

template <typename T> struct Vec4 {};
template <> struct Vec4<float> {
  static __device__ __forceinline__ void load(const float* p, float (&v)[4]) {
    const float4 x = *(const float4*)p;
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
  }
};
template <> struct Vec4<bf16_t> {
  static __device__ __forceinline__ void load(const bf16_t* p, float (&v)[4]) {
    const uint2 x = *(const uint2*)p;
    v[0] = __uint_as_float(x.x << 16); v[1] = __uint_as_float(x.x & 0xffff0000u);
    v[2] = __uint_as_float(x.y << 16); v[3] = __uint_as_float(x.y & 0xffff0000u);
  }
};

// A workgroup of 16 waves takes four tokens.  Logits: wave w forms those of the experts w,
// w + 16, ... for all four tokens at once (a piece of the router's row is loaded once and meets
// the four tokens' pieces; every token's sum runs over its own row in a fixed order).  Choice:
// wave w then ranks token w's logits.
template <typename T>
__global__ __launch_bounds__(MOE_ROUTE_WAVES * ZF_WAVE) void moe_route_kernel(
    const T* __restrict__ h, const float* __restrict__ router, const float* __restrict__ bias,
    int* __restrict__ ids, float* __restrict__ weights, int n_tokens, int W, int E, int top,
    int scoring, const float* __restrict__ correction, int n_groups, int keep_groups,
    int mark_top, int normalize, float weight_scale, int n_extra, float* __restrict__ extra) {
  __shared__ float zs[MOE_ROUTE_TOKENS][MOE_MAX_EXPERTS], shares[MOE_ROUTE_TOKENS][MOE_MAX_EXPERTS];
  __shared__ int chosens[MOE_ROUTE_TOKENS][MOE_MAX_EXPERTS];
  __shared__ unsigned char kepts[MOE_ROUTE_TOKENS][MOE_MAX_EXPERTS];
  const int wave = threadIdx.x / ZF_WAVE, lane = threadIdx.x % ZF_WAVE;
  const int t0 = blockIdx.x * MOE_ROUTE_TOKENS;
  const T* rows[MOE_ROUTE_TOKENS];
#pragma unroll
  for (int k = 0; k < MOE_ROUTE_TOKENS; ++k) rows[k] = h + (size_t)min(t0 + k, n_tokens - 1) * W;
  // (rows E .. E + n_extra - 1 of the router are no experts: their sigmoids go to `extra`)
  for (int e = wave; e < E + n_extra; e += MOE_ROUTE_WAVES) {
    const float* r = router + (size_t)e * W;
    float dot[MOE_ROUTE_TOKENS];
#pragma unroll
    for (int k = 0; k < MOE_ROUTE_TOKENS; ++k) dot[k] = 0.f;
    if (W % 4 == 0) {
#pragma unroll 4
      for (int i = lane * 4; i < W; i += ZF_WAVE * 4) {
        const float4 rv = *(const float4*)(r + i);
#pragma unroll
        for (int k = 0; k < MOE_ROUTE_TOKENS; ++k) {
          float x[4];
          Vec4<T>::load(rows[k] + i, x);
          dot[k] = fmaf(x[0], rv.x, dot[k]);
          dot[k] = fmaf(x[1], rv.y, dot[k]);
          dot[k] = fmaf(x[2], rv.z, dot[k]);
          dot[k] = fmaf(x[3], rv.w, dot[k]);
        }
      }
    } else {
      for (int i = lane; i < W; i += ZF_WAVE) {
        const float rv = r[i];
#pragma unroll
        for (int k = 0; k < MOE_ROUTE_TOKENS; ++k)
          dot[k] = fmaf(load_as_float<T>(rows[k] + i), rv, dot[k]);
      }
    }
    const float be = (bias != nullptr && e < E) ? bias[e] : 0.f;
#pragma unroll
    for (int k = 0; k < MOE_ROUTE_TOKENS; ++k) {
      const float z = wave_sum(dot[k]);
      if (lane == 0) {
        if (e < E) zs[k][e] = z + be;
        else if (t0 + k < n_tokens)
          extra[(size_t)(t0 + k) * n_extra + (e - E)] = 1.0f / (1.0f + expf(-z));
      }
    }
  }
  __syncthreads();
  const int t = t0 + wave;
  if (wave >= MOE_ROUTE_TOKENS || t >= n_tokens) return;
  float* z = zs[wave];
  float* share = shares[wave];
  int* chosen = chosens[wave];
  if (scoring != 0) {
    // scores s = sigmoid(z), or the soft-max over all of z (kept in `share`), choice scores
    // s + correction (in `z`)
    float zmax = 0.f, zsum = 1.f;
    if (scoring == 2) {
      zmax = -INFINITY;
      for (int e = lane; e < E; e += ZF_WAVE) zmax = fmaxf(zmax, z[e]);
      zmax = wave_max(zmax);
      zsum = 0.f;
      for (int e = lane; e < E; e += ZF_WAVE) zsum += expf(z[e] - zmax);
      zsum = wave_sum(zsum);
    }
    for (int e = lane; e < E; e += ZF_WAVE) {
      const float sc = scoring == 2 ? expf(z[e] - zmax) / zsum : 1.0f / (1.0f + expf(-z[e]));
      share[e] = sc;
      z[e] = sc + (correction != nullptr ? correction[e] : 0.f);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    if (n_groups > 0 && keep_groups < n_groups) {
      // a group's mark: its two largest choice scores added (its one score, if it has one)
      float* mark = (float*)chosen;
      unsigned char* kept = kepts[wave];
      const int size = E / n_groups;
      for (int g = lane; g < n_groups; g += ZF_WAVE) {
        float a = -INFINITY, b = -INFINITY;
        for (int e = g * size; e < (g + 1) * size; ++e) {
          const float v = z[e];
          if (v > a) { b = a; a = v; } else if (v > b) { b = v; }
        }
        mark[g] = (size > 1 && mark_top > 1) ? a + b : a;
        kept[g] = 0;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __builtin_amdgcn_wave_barrier();
      for (int k = 0; k < keep_groups; ++k) {
        float best = -INFINITY;
        int arg = 0x7fffffff;
        for (int g = lane; g < n_groups; g += ZF_WAVE) {
          const float v = mark[g];
          if (!kept[g] && (v > best || arg == 0x7fffffff)) { best = v; arg = g; }
        }
#pragma unroll
        for (int off = ZF_WAVE / 2; off > 0; off >>= 1) {
          const float ob = __shfl_xor(best, off, ZF_WAVE);
          const int oa = __shfl_xor(arg, off, ZF_WAVE);
          if (oa != 0x7fffffff && (arg == 0x7fffffff || ob > best || (ob == best && oa < arg))) {
            best = ob; arg = oa;
          }
        }
        if (lane == 0 && arg != 0x7fffffff) kept[arg] = 1;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_wave_barrier();
      }
      // outside the kept groups nothing can be chosen
      for (int e = lane; e < E; e += ZF_WAVE)
        if (!kept[e / size]) z[e] = -INFINITY;
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __builtin_amdgcn_wave_barrier();
    }
    float sum = 0.f;
    for (int k = 0; k < top; ++k) {
      float best = -INFINITY;
      int arg = 0x7fffffff;
      for (int e = lane; e < E; e += ZF_WAVE) {
        const float v = z[e];
        if (v > best) { best = v; arg = e; }
      }
#pragma unroll
      for (int off = ZF_WAVE / 2; off > 0; off >>= 1) {
        const float ob = __shfl_xor(best, off, ZF_WAVE);
        const int oa = __shfl_xor(arg, off, ZF_WAVE);
        if (ob > best || (ob == best && oa < arg)) { best = ob; arg = oa; }
      }
      if (arg == 0x7fffffff) arg = 0;
      sum += share[arg];
      if (lane == 0) {
        chosen[k] = arg;
        z[arg] = -INFINITY;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      __builtin_amdgcn_wave_barrier();
    }
    for (int k = lane; k < top; k += ZF_WAVE) {
      ids[(size_t)t * top + k] = chosen[k];
      const float sh = share[chosen[k]];
      weights[(size_t)t * top + k] = (normalize ? sh / (sum + 1e-20f) : sh) * weight_scale;
    }
    return;
  }
  // `top` rounds of: the largest remaining logit, the lowest index among equals
  float first = 0.f, sum = 0.f;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int arg = 0x7fffffff;
    for (int e = lane; e < E; e += ZF_WAVE) {
      const float v = z[e];
      if (v > best) { best = v; arg = e; }
    }
#pragma unroll
    for (int off = ZF_WAVE / 2; off > 0; off >>= 1) {
      const float ob = __shfl_xor(best, off, ZF_WAVE);
      const int oa = __shfl_xor(arg, off, ZF_WAVE);
      if (ob > best || (ob == best && oa < arg)) { best = ob; arg = oa; }
    }
    if (arg == 0x7fffffff) arg = 0;            // nothing but NaN or -inf left
    if (k == 0) first = best;
    const float e_k = expf(best - first);       // the first chosen logit is the largest
    sum += e_k;
    if (lane == 0) {
      chosen[k] = arg;
      share[k] = e_k;
      z[arg] = -INFINITY;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
  }
  for (int k = lane; k < top; k += ZF_WAVE) {
    ids[(size_t)t * top + k] = chosen[k];
    weights[(size_t)t * top + k] = share[k] / sum;
  }
}

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float moe_f32x4_t;

// Up to 128 router rows, 16 tokens a tile.  The logits are 32-bit MFMAs (16x16x4: rows of the
// router against the tokens, h widened), K dealt into 64 spans, eight to a group: a group's spans
// are added in pairs, then the groups, so a token's logits do not depend on the tokens beside it
// nor on how many there are.  Then a wave ranks a token's logits all at once: an expert's rank is
// the number of experts before it (larger, or equal and of a lower index), one pass over a row in
// LDS instead of a round of twelve lane exchanges for every chosen one.
//   * many tokens: a workgroup of 16 waves takes a tile, two groups at a time.
//   * else (SPLIT): one compute unit draws a router of 256 KB in 8 us, so a workgroup of eight
//     waves takes one group of K and 32 rows of the router, leaves its sums in `ws` and adds one to
//     the tile's counter; the one that finds the count complete adds the groups and chooses.  Sums
//     and counter go through to memory (agent scope), where every XCD sees them; the counter is
//     back at zero when the kernel ends.  (Up to 1024 workgroups: with 2048 of them 1024 tokens of
//     W = 2048 and 128 rows took 86 us, without the split 60.)
// What it takes is said at route16_takes.  Without a release fence a decode step's 32 rows take 9.8
// us where they took 11.3, 33 rows 12.5 and 15.2.
#if defined(__HIP_DEVICE_COMPILE__) && !defined(__gfx950__)
#error "moe_route16_kernel's hand-over between workgroups is written for gfx950's memory"
#endif
#define MOE_ROUTE16_ROWS 128
#define MOE_ROUTE16_GROUPS 8
#define MOE_ROUTE16_SPLIT_TILES 64       // up to so many tiles of 16 tokens are split

// numbers of K in a span, and groups that hold any
static __host__ __device__ __forceinline__ int route16_span(int W) { return (W + 2047) / 2048 * 32; }
static __host__ __device__ __forceinline__ int route16_groups(int W) {
  return (W + 8 * route16_span(W) - 1) / (8 * route16_span(W));
}

__device__ __forceinline__ void store_agent(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// (two floats side by side, from a multiple of 8 bytes)
__device__ __forceinline__ void load2_agent(const float* p, float& a, float& b) {
  const unsigned long long v = __hip_atomic_load((const unsigned long long*)p, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
  a = __uint_as_float((uint32_t)v);
  b = __uint_as_float((uint32_t)(v >> 32));
}

// eight consecutive values of a row as floats; at or beyond k_end they are 0
template <typename T, bool VEC>
__device__ __forceinline__ void route_load8(const T* __restrict__ row, int k, int k_end,
                                            float (&v)[8]) {
  if constexpr (VEC) {             // (W a multiple of 8: all eight or none)
    if (k < k_end) {
      if constexpr (sizeof(T) == 2) {
        const uint4 x = *(const uint4*)(row + k);
        const uint32_t p[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          v[2 * c] = __uint_as_float(p[c] << 16);
          v[2 * c + 1] = __uint_as_float(p[c] & 0xffff0000u);
        }
      } else {
        const float4 x = *(const float4*)(row + k), y = *(const float4*)(row + k + 4);
        v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
        v[4] = y.x; v[5] = y.y; v[6] = y.z; v[7] = y.w;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = 0.f;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = k + i < k_end ? load_as_float<T>(row + k + i) : 0.f;
  }
}

// f(0) + .. + f(7), added in pairs
template <typename F>
__device__ __forceinline__ moe_f32x4_t sum8(F f) {
  return ((f(0) + f(1)) + (f(2) + f(3))) + ((f(4) + f(5)) + (f(6) + f(7)));
}

__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

// how many of row[0 .. n4 * 4) come before (v, e): larger, or equal with a lower index (NaN: none).
// No branches: the lanes of a wave part at every comparison.  BLOCK: e lies in the BLOCK-th 64 for
// the whole wave (-1: anywhere), so that only numbers of that 64 need their index compared.
// (Where 16 waves choose among 128, the comparisons are what the kernel spends its time on: 16
// tokens, W = 64 in 24 us with branches, 20 without, 13 by blocks.)
template <int BLOCK>
__device__ __forceinline__ int rank_before(const float* row, int n4, float v, int e) {
  int rank = 0;
  const int lo = BLOCK < 0 ? 0 : min(n4, 16 * BLOCK), hi = BLOCK < 0 ? n4 : min(n4, 16 * BLOCK + 16);
  auto each = [&](int from, int to, auto before) {
#pragma unroll 4
    for (int j = from; j < to; ++j) {
      const float4 o = *(const float4*)(row + 4 * j);
      rank += before(o.x, 4 * j);
      rank += before(o.y, 4 * j + 1);
      rank += before(o.z, 4 * j + 2);
      rank += before(o.w, 4 * j + 3);
    }
  };
  if constexpr (BLOCK > 0) each(0, lo, [&](float o, int) { return (int)(o >= v); });
  each(lo, hi, [&](float o, int i) { return (int)(o > v) + ((int)(o == v) & (int)(i < e)); });
  if constexpr (BLOCK >= 0) each(hi, n4, [&](float o, int) { return (int)(o > v); });
  return rank;
}

// one wave: token t's logits in `z` (LDS, -inf from E up to a multiple of 4) to its experts and
// weights; share and chosen: room for as many numbers
__device__ __forceinline__ void route_choose(float* z, float* share, int* chosen, int* __restrict__ ids,
                             float* __restrict__ weights, int t, int E, int top, int scoring,
                             const float* __restrict__ correction, int n_groups, int keep_groups,
                             int mark_top, int normalize, float weight_scale, int lane) {
  const int n4 = (E + 3) / 4;
  if (scoring != 0) {
    // scores s = sigmoid(z), or the soft-max over all of z (kept in `share`), choice scores
    // s + correction (in `z`)
    float zmax = 0.f, zsum = 1.f;
    if (scoring == 2) {
      zmax = -INFINITY;
      for (int e = lane; e < E; e += ZF_WAVE) zmax = fmaxf(zmax, z[e]);
      zmax = wave_max(zmax);
      zsum = 0.f;
      for (int e = lane; e < E; e += ZF_WAVE) zsum += expf(z[e] - zmax);
      zsum = wave_sum(zsum);
    }
    for (int e = lane; e < E; e += ZF_WAVE) {
      const float sc = scoring == 2 ? expf(z[e] - zmax) / zsum : 1.0f / (1.0f + expf(-z[e]));
      share[e] = sc;
      z[e] = sc + (correction != nullptr ? correction[e] : 0.f);
    }
    wave_lds_fence();
    if (n_groups > 0 && keep_groups < n_groups) {
      // a group's mark: its two largest choice scores added (its one score, if it has one)
      float* mark = (float*)chosen;
      const int size = E / n_groups, g4 = (n_groups + 3) / 4;
      for (int q = lane; q < 4 * g4; q += ZF_WAVE) {
        float a = -INFINITY, b = -INFINITY;
        if (q < n_groups)
          for (int e = q * size; e < (q + 1) * size; ++e) {
            const float v = z[e];
            if (v > a) { b = a; a = v; } else if (v > b) { b = v; }
          }
        // (a sum of +inf and -inf ranks last, as -inf does)
        const float m = (size > 1 && mark_top > 1) ? a + b : a;
        mark[q] = m == m ? m : -INFINITY;
      }
      wave_lds_fence();
      // outside the kept groups nothing can be chosen
      bool out[2] = {false, false};
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int e = lane + ZF_WAVE * i;
        if (e < E) out[i] = rank_before<-1>(mark, g4, mark[e / size], e / size) >= keep_groups;
      }
      wave_lds_fence();
#pragma unroll
      for (int i = 0; i < 2; ++i)
        if (out[i]) z[lane + ZF_WAVE * i] = -INFINITY;
      wave_lds_fence();
    }
  }
  // the chosen in the order of their scores; where nothing but NaN or -inf is left, expert 0
  for (int k = lane; k < top; k += ZF_WAVE) chosen[k] = -1;
  wave_lds_fence();
  auto place = [&](auto BLOCK) {
    const int e = lane + ZF_WAVE * decltype(BLOCK)::value;
    const float v = e < E ? z[e] : -INFINITY;
    const int rank = rank_before<decltype(BLOCK)::value>(z, n4, v, e);
    if (v > -INFINITY && rank < top) chosen[rank] = e;
  };
  place(std::integral_constant<int, 0>{});
  if (E > ZF_WAVE) place(std::integral_constant<int, 1>{});
  wave_lds_fence();
  if (scoring == 0) {
    const float first = chosen[0] >= 0 ? z[chosen[0]] : -INFINITY;
    for (int k = lane; k < top; k += ZF_WAVE)
      share[k] = expf((chosen[k] >= 0 ? z[chosen[k]] : -INFINITY) - first);
    wave_lds_fence();
    float sum = 0.f;
    for (int k = 0; k < top; ++k) sum += share[k];
    for (int k = lane; k < top; k += ZF_WAVE) {
      ids[(size_t)t * top + k] = max(chosen[k], 0);
      weights[(size_t)t * top + k] = share[k] / sum;
    }
    return;
  }
  float sum = 0.f;
  for (int k = 0; k < top; ++k) sum += share[max(chosen[k], 0)];
  for (int k = lane; k < top; k += ZF_WAVE) {
    const int e = max(chosen[k], 0);
    ids[(size_t)t * top + k] = e;
    weights[(size_t)t * top + k] = (normalize ? share[e] / (sum + 1e-20f) : share[e]) * weight_scale;
  }
}

template <typename T, bool VEC, bool SPLIT>
__global__ __launch_bounds__((SPLIT ? 8 : 16) * ZF_WAVE) void moe_route16_kernel(
    const T* __restrict__ h, const float* __restrict__ router, const float* __restrict__ bias,
    int* __restrict__ ids, float* __restrict__ weights, int n_tokens, int W, int E, int top,
    int scoring, const float* __restrict__ correction, int n_groups, int keep_groups,
    int mark_top, int normalize, float weight_scale, int n_extra, float* __restrict__ extra,
    float* __restrict__ ws, int* __restrict__ counters) {
  constexpr int WAVES = SPLIT ? 8 : 16;
  __shared__ moe_f32x4_t part[WAVES][2][ZF_WAVE];
  __shared__ __attribute__((aligned(16))) float zs[16][MOE_ROUTE16_ROWS];
  __shared__ __attribute__((aligned(16))) float shares[16][MOE_ROUTE16_ROWS];
  __shared__ __attribute__((aligned(16))) int chosens[16][MOE_ROUTE16_ROWS];
  __shared__ int arrived;
  const int wave = threadIdx.x / ZF_WAVE, lane = threadIdx.x % ZF_WAVE;
  const int r = lane % 16, g = lane / 16, tile = SPLIT ? blockIdx.y : blockIdx.x, t0 = tile * 16;
  const int rows = E + n_extra, chunks = (rows + 31) / 32;        // 32 rows of the router
  const int span = route16_span(W), groups = route16_groups(W);
  const T* row = h + (size_t)min(t0 + r, n_tokens - 1) * W;
  // column lane % 16 is a token, the four numbers are rows 4 (lane / 16) + i of the 16-row tile
  auto take = [&](int chunk, int half, moe_f32x4_t z) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = chunk * 32 + 16 * half + 4 * g + i;
      if (e < E) {
        zs[r][e] = z[i] + (bias != nullptr ? bias[e] : 0.f);
      } else {
        if (e < rows && t0 + r < n_tokens)
          extra[(size_t)(t0 + r) * n_extra + (e - E)] = 1.0f / (1.0f + expf(-z[i]));
        if (e < MOE_ROUTE16_ROWS) zs[r][e] = -INFINITY;           // no candidates
      }
    }
  };
  const int c0 = SPLIT ? blockIdx.x / groups : 0, c1 = SPLIT ? c0 + 1 : chunks;
  const int grp0 = SPLIT ? blockIdx.x % groups : 0, grp1 = SPLIT ? grp0 + 1 : groups;
  for (int chunk = c0; chunk < c1; ++chunk) {
    const float *ra = router + (size_t)min(chunk * 32 + r, rows - 1) * W,
                *rb = router + (size_t)min(chunk * 32 + 16 + r, rows - 1) * W;
    moe_f32x4_t lo = {0.f, 0.f, 0.f, 0.f}, hi = lo;                  // of the groups' halves
    for (int grp = grp0; grp < grp1; grp += WAVES / 8) {
      const int k_begin = ((grp + wave / 8) * 8 + wave % 8) * span, k_end = min(W, k_begin + span);
      // (eight sums side by side, one an element of a lane's eight: sums of few terms, added in
      // pairs)
      moe_f32x4_t acc[8][2];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        acc[i][0] = acc[i][1] = moe_f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll (SPLIT ? 2 : 1)                // (sixteen waves have 128 registers each)
      for (int k0 = k_begin; k0 < k_end; k0 += 32) {
        float x[8], a[8], b[8];
        route_load8<T, VEC>(row, k0 + 8 * g, k_end, x);
        route_load8<float, VEC>(ra, k0 + 8 * g, k_end, a);
        route_load8<float, VEC>(rb, k0 + 8 * g, k_end, b);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], x[i], acc[i][0], 0, 0, 0);
          acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[i], x[i], acc[i][1], 0, 0, 0);
        }
      }
#pragma unroll
      for (int half = 0; half < 2; ++half)
        part[wave][half][lane] = sum8([&](int i) { return acc[i][half]; });
      __syncthreads();
      if (wave < 2) {
        moe_f32x4_t z = sum8([&](int s) { return part[s][wave][lane]; });
        if constexpr (WAVES > 8) z += sum8([&](int s) { return part[8 + s][wave][lane]; });
        if (grp < MOE_ROUTE16_GROUPS / 2) lo += z; else hi += z;
      }
      __syncthreads();
    }
    if constexpr (SPLIT) {
      // [tile][chunk][half][lane][group][4]
      if (wave < 2) {
        float* p = ws + ((((size_t)tile * chunks + chunk) * 2 + wave) * ZF_WAVE + lane) *
                            (MOE_ROUTE16_GROUPS * 4) + grp0 * 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) store_agent(p + i, lo[i] + hi[i]);
        // The stores have reached memory before the count says so: on gfx950 agent-scope stores go
        // through the L2 and count down vmcnt once they are there.  (A release fence says the same
        // in the language's terms, but writes the whole L2 back, which is what the kernels before
        // this one left there.)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
    } else if (wave < 2) {
      take(chunk, wave, lo + hi);
    }
  }
  __syncthreads();
  if constexpr (SPLIT) {
    const int all = chunks * groups;
    if (threadIdx.x == 0)
      arrived = __hip_atomic_fetch_add(counters + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (arrived != all - 1) return;
    // The others' sums are read behind the count: agent-scope loads pass the caches here, and none of
    // them is issued before the count has come back.  (An acquire fence would drop what the caches
    // hold for it: a decode step's router 10.3 -> 11.1 us.)
    __atomic_signal_fence(__ATOMIC_ACQUIRE);
    if (threadIdx.x == 0)
      __hip_atomic_store(counters + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (wave < 2 * chunks) {            // (at most 128 rows: 8 halves of 16, one a wave)
      const float* p = ws + (((size_t)tile * chunks * 2 + wave) * ZF_WAVE + lane) *
                                (MOE_ROUTE16_GROUPS * 4);
      float v[MOE_ROUTE16_GROUPS * 4];
#pragma unroll
      for (int i = 0; i < MOE_ROUTE16_GROUPS * 4; i += 2) {
        v[i] = v[i + 1] = 0.f;
        if (i < 4 * groups) load2_agent(p + i, v[i], v[i + 1]);
      }
      take(wave / 2, wave % 2, sum8([&](int grp) {
        return moe_f32x4_t{v[4 * grp], v[4 * grp + 1], v[4 * grp + 2], v[4 * grp + 3]};
      }));
    }
    __syncthreads();
  }
  for (int k = wave; k < 16 && t0 + k < n_tokens; k += WAVES)
    route_choose(zs[k], shares[k], chosens[k], ids, weights, t0 + k, E, top, scoring, correction,
                 n_groups, keep_groups, mark_top, normalize, weight_scale, lane);
}

// Which calls the kernel for 16 tokens a tile takes.  By the router's sizes: W from 2048 on, or from
// 1024 on and 32 rows or more.  (Narrower ones are at the cost of a launch either way, or spend
// their time on the choice, which only as many waves as tokens work at: 4 rows of 768 7.4 us,
// four tokens a workgroup 6.6; 128 rows of 256 19.7, 16.3.)  In bfloat16 also by the tokens: up to
// `few` through the sums in `ws`; and above 1024, where four tokens a workgroup fill the chip more
// than once, from W = 512 on and any number of rows.  Measured, us, this and that: W = 2048, 32
// rows: 8 tokens 9.1 and 16.5, 256 12.5 and 16.7, 1024 17.1 and 17.3, 2048 17.1 and 29.0; 128 rows:
// 16.5 and 49.7, 37.9 and 50.4, 60.0 and 51.1, 60.3 and 96.8; 8 rows: 8 tokens 8.1 and 9.5, 256
// 11.0 and 9.7; W = 4096, 64 rows: 12.1 and 45.4, 18.7 and 46.0, 36.2 and 46.5, 49.9 and 87.9.  In
// float32 the same kernel for any number of tokens, so that a token's logits do not depend on it.
static bool route16_takes(int T, int W, int rows, bool f32, bool sums) {
  if (rows > MOE_ROUTE16_ROWS) return false;
  if (!f32 && T > 1024) return W >= 512;
  if (W < 1024 || (W < 2048 && rows < 32)) return false;
  const int few = W >= 3072 ? 512 : rows < 32 ? 64 : 256;
  return f32 || (sums && T <= few);
}

// ws: float32 [64 tiles][(E + n_extra + 31) / 32][4096] and counters [64] at zero (both or neither;
// the counters are at zero again when the kernel ends): what up to 1024 tokens and 128 router rows
// use to spread over workgroups.
extern "C" int zf_moe_route(const void* h, int dtype, const float* router, const float* bias,
                            int* ids, float* weights, int T, int W, int E, int top,
                            int scoring, const float* correction, int n_groups, int keep_groups,
                            int mark_top, int normalize, float weight_scale, int n_extra,
                            float* extra, float* ws, int* counters, hipStream_t stream) {
  if (T <= 0) return 0;
  if (E <= 0 || E > MOE_MAX_EXPERTS || top <= 0 || top > E || scoring < 0 || scoring > 2 ||
      n_extra < 0 || (n_extra > 0 && extra == nullptr) || mark_top < 1 || mark_top > 2 ||
      n_groups < 0 || (n_groups > 0 && (E % n_groups != 0 || keep_groups < 1 ||
                                        keep_groups > n_groups ||
                                        top > keep_groups * (E / n_groups))))
    return -2;
  const int rows = E + n_extra;
  const bool sums = ws != nullptr && counters != nullptr;
  if (route16_takes(T, W, rows, dtype == ZF_F32, sums)) {
    const bool vec = W % 8 == 0 && ((uintptr_t)h | (uintptr_t)router) % 16 == 0;
    const int tiles = (T + 15) / 16, parts = (rows + 31) / 32 * route16_groups(W);
    const bool split = sums && tiles <= MOE_ROUTE16_SPLIT_TILES && tiles * parts <= 1024;
#define MOE_ROUTE16_AS(TT, V, S, G, B)                                                           \
  hipLaunchKernelGGL((moe_route16_kernel<TT, V, S>), G, dim3(B), 0, stream, (const TT*)h,        \
                     router, bias, ids, weights, T, W, E, top, scoring, correction, n_groups,    \
                     keep_groups, mark_top, normalize, weight_scale, n_extra, extra, ws, counters)
#define MOE_ROUTE16(TT, V)                                                                       \
  do {                                                                                           \
    if (split) MOE_ROUTE16_AS(TT, V, true, dim3(parts, tiles), 512);                             \
    else MOE_ROUTE16_AS(TT, V, false, dim3(tiles), 1024);                                        \
  } while (0)
    if (dtype == ZF_F32) {
      if (vec) MOE_ROUTE16(float, true); else MOE_ROUTE16(float, false);
    } else {
      if (vec) MOE_ROUTE16(bf16_t, true); else MOE_ROUTE16(bf16_t, false);
    }
#undef MOE_ROUTE16_AS
#undef MOE_ROUTE16
    ZF_CHECK_LAUNCH();
  }
  const dim3 grid((T + MOE_ROUTE_TOKENS - 1) / MOE_ROUTE_TOKENS), block(MOE_ROUTE_WAVES * ZF_WAVE);
  if (dtype == ZF_F32)
    hipLaunchKernelGGL(moe_route_kernel<float>, grid, block, 0, stream, (const float*)h, router,
                       bias, ids, weights, T, W, E, top, scoring, correction, n_groups,
                       keep_groups, mark_top, normalize, weight_scale, n_extra, extra);
  else
    hipLaunchKernelGGL(moe_route_kernel<bf16_t>, grid, block, 0, stream, (const bf16_t*)h, router,
                       bias, ids, weights, T, W, E, top, scoring, correction, n_groups,
                       keep_groups, mark_top, normalize, weight_scale, n_extra, extra);
  ZF_CHECK_LAUNCH();
}

// the activation of an expert's two products
__device__ __forceinline__ float gated_unit(float g, float u, float limit, float alpha,
                                            float shift) {
  if (limit > 0.f) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
  }
  return g * (1.0f / (1.0f + expf(-alpha * g))) * (u + shift);
}

// dot product of a weight row with a vector held in LDS as floats, lanes side by side; a
// bfloat16 row whose length is a multiple of 8 comes as 16-byte loads
template <typename T>
__device__ __forceinline__ float row_dot_lds(const T* __restrict__ w, const float* __restrict__ x,
                                             int n, int lane) {
  float dot = 0.f;
  if constexpr (sizeof(T) == 2) {
    if (n % 8 == 0) {
      for (int i = lane * 8; i < n; i += ZF_WAVE * 8) {
        const uint4 v = *(const uint4*)(w + i);
        const uint32_t p[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          dot = fmaf(__uint_as_float(p[c] << 16), x[i + 2 * c], dot);
          dot = fmaf(__uint_as_float(p[c] & 0xffff0000u), x[i + 2 * c + 1], dot);
        }
      }
      return dot;
    }
  }
  for (int i = lane; i < n; i += ZF_WAVE) dot = fmaf(load_as_float<T>(w + i), x[i], dot);
  return dot;
}

// the same between two rows in global memory
template <typename T>
__device__ __forceinline__ float row_dot(const T* __restrict__ w, const T* __restrict__ y, int n,
                                         int lane) {
  float dot = 0.f;
  if constexpr (sizeof(T) == 2) {
    if (n % 8 == 0) {
      for (int i = lane * 8; i < n; i += ZF_WAVE * 8) {
        const uint4 a = *(const uint4*)(w + i);
        const uint4 b = *(const uint4*)(y + i);
        const uint32_t p[4] = {a.x, a.y, a.z, a.w}, q[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          dot = fmaf(__uint_as_float(p[c] << 16), __uint_as_float(q[c] << 16), dot);
          dot = fmaf(__uint_as_float(p[c] & 0xffff0000u), __uint_as_float(q[c] & 0xffff0000u), dot);
        }
      }
      return dot;
    }
  }
  for (int i = lane; i < n; i += ZF_WAVE)
    dot = fmaf(load_as_float<T>(w + i), load_as_float<T>(y + i), dot);
  return dot;
}

#define MOE_WAVES 4
#define MOE_GU_PER_WAVE 4      // outputs of y a wave computes, one after the other

// GATED: gate_up [E, 2 ff, W] and the gated activation; else `gate_up` holds the up rows alone,
// [E, ff, W], and y = activation_value(up, act) (`act` by the numbers of zf_common.h).
template <typename T, bool GATED>
__global__ __launch_bounds__(MOE_WAVES * ZF_WAVE) void moe_gate_up_kernel(
    const T* __restrict__ h, const T* __restrict__ gate_up, const int* __restrict__ ids,
    T* __restrict__ y, int W, int ff, int slots, float limit, float alpha, float shift, int act,
    int n_experts) {
  extern __shared__ __attribute__((aligned(16))) float xs[];       // the token's row, [W]
  const int ts = blockIdx.x, t = ts / slots;
  const int e = ids != nullptr ? ids[ts] : 0;
  if (e >= n_experts) return;                      // an output of the router without an expert
  const int wave = threadIdx.x / ZF_WAVE, lane = threadIdx.x % ZF_WAVE;
  const T* row = h + (size_t)t * W;
  for (int i = threadIdx.x; i < W; i += blockDim.x) xs[i] = load_as_float<T>(row + i);
  __syncthreads();
  const T* we = gate_up + (size_t)e * (GATED ? 2 : 1) * ff * W;
  const int j0 = (blockIdx.y * MOE_WAVES + wave) * MOE_GU_PER_WAVE;
  if (j0 >= ff) return;
  if constexpr (sizeof(T) == 2) {
    if (W % 8 == 0) {
      // the wave's outputs side by side: eight 16-byte loads in flight for every piece of the
      // token's row (an output beyond the last repeats the last one and is not stored)
      float dg[MOE_GU_PER_WAVE], du[MOE_GU_PER_WAVE];
      const T* gr[MOE_GU_PER_WAVE];
#pragma unroll
      for (int o = 0; o < MOE_GU_PER_WAVE; ++o) {
        dg[o] = du[o] = 0.f;
        gr[o] = we + (size_t)min(j0 + o, ff - 1) * W;
      }
#pragma unroll 2
      for (int i = lane * 8; i < W; i += ZF_WAVE * 8) {
        uint4 a[MOE_GU_PER_WAVE], b[MOE_GU_PER_WAVE];
#pragma unroll
        for (int o = 0; o < MOE_GU_PER_WAVE; ++o) {
          a[o] = *(const uint4*)(gr[o] + i);
          if constexpr (GATED) b[o] = *(const uint4*)(gr[o] + (size_t)ff * W + i);
        }
        const float4 x0 = *(const float4*)(xs + i), x1 = *(const float4*)(xs + i + 4);
        const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
        for (int o = 0; o < MOE_GU_PER_WAVE; ++o) {
          const uint32_t p[4] = {a[o].x, a[o].y, a[o].z, a[o].w};
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            dg[o] = fmaf(__uint_as_float(p[c] << 16), x[2 * c], dg[o]);
            dg[o] = fmaf(__uint_as_float(p[c] & 0xffff0000u), x[2 * c + 1], dg[o]);
          }
          if constexpr (GATED) {
            const uint32_t q[4] = {b[o].x, b[o].y, b[o].z, b[o].w};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
              du[o] = fmaf(__uint_as_float(q[c] << 16), x[2 * c], du[o]);
              du[o] = fmaf(__uint_as_float(q[c] & 0xffff0000u), x[2 * c + 1], du[o]);
            }
          }
        }
      }
#pragma unroll
      for (int o = 0; o < MOE_GU_PER_WAVE; ++o) {
        const float g = wave_sum(dg[o]);
        float r;
        if constexpr (GATED) r = gated_unit(g, wave_sum(du[o]), limit, alpha, shift);
        else r = activation_value(g, act);
        if (lane == 0 && j0 + o < ff) store_from_float<T>(y + (size_t)ts * ff + j0 + o, r);
      }
      return;
    }
  }
  for (int j = j0; j < j0 + MOE_GU_PER_WAVE && j < ff; ++j) {
    const float g = wave_sum(row_dot_lds<T>(we + (size_t)j * W, xs, W, lane));
    float r;
    if constexpr (GATED) {
      const float u = wave_sum(row_dot_lds<T>(we + (size_t)(ff + j) * W, xs, W, lane));
      r = gated_unit(g, u, limit, alpha, shift);
    } else {
      r = activation_value(g, act);
    }
    if (lane == 0) store_from_float<T>(y + (size_t)ts * ff + j, r);
  }
}

// gated != 0: gate_up [E, 2 ff, W]; else [E, ff, W] and the plain activation `act`
extern "C" int zf_moe_gate_up(const void* h, const void* gate_up, int dtype, const int* ids,
                              void* y, int T, int W, int ff, int slots, float limit, float alpha,
                              float shift, int gated, int act, int n_experts,
                              hipStream_t stream) {
  if (T <= 0) return 0;
  if (W <= 0 || ff <= 0 || slots <= 0 || (size_t)W * sizeof(float) > 64 * 1024 || act < 0 ||
      act > 4)
    return -2;
  const int per_wg = MOE_WAVES * MOE_GU_PER_WAVE;
  dim3 grid(T * slots, (ff + per_wg - 1) / per_wg);
  const size_t smem = (size_t)W * sizeof(float);
#define MOE_GU_LAUNCH(TT, G)                                                                      \
  hipLaunchKernelGGL((moe_gate_up_kernel<TT, G>), grid, dim3(MOE_WAVES * ZF_WAVE), smem, stream, \
                     (const TT*)h, (const TT*)gate_up, ids, (TT*)y, W, ff, slots, limit, alpha,  \
                     shift, act, n_experts)
  if (dtype == ZF_F32) {
    if (gated) MOE_GU_LAUNCH(float, true); else MOE_GU_LAUNCH(float, false);
  } else {
    if (gated) MOE_GU_LAUNCH(bf16_t, true); else MOE_GU_LAUNCH(bf16_t, false);
  }
  ZF_CHECK_LAUNCH();
}

#define MOE_DOWN_PER_WAVE 4

template <typename T>
__global__ __launch_bounds__(MOE_WAVES * ZF_WAVE) void moe_down_kernel(
    const T* __restrict__ y, const T* __restrict__ down, const int* __restrict__ ids,
    const float* __restrict__ weights, float* __restrict__ out, int W, int ff, int slots,
    int add, int n_experts, const T* __restrict__ h) {
  const int t = blockIdx.x;
  const int wave = threadIdx.x / ZF_WAVE, lane = threadIdx.x % ZF_WAVE;
  const int n0 = (blockIdx.y * MOE_WAVES + wave) * MOE_DOWN_PER_WAVE;
  if (n0 >= W) return;
  if constexpr (sizeof(T) == 2) {
    if (ff % 8 == 0) {
      // the wave's outputs side by side; a lane adds its pieces over all slots (in slot order)
      // before the lanes are added up, so there is one sum over the wave per output
      float tot[MOE_DOWN_PER_WAVE], same[MOE_DOWN_PER_WAVE];
#pragma unroll
      for (int o = 0; o < MOE_DOWN_PER_WAVE; ++o) tot[o] = same[o] = 0.f;
      for (int s = 0; s < slots; ++s) {
        const int ts = t * slots + s;
        const int e = ids != nullptr ? ids[ts] : 0;
        const float c = weights != nullptr ? weights[ts] : 1.0f;
        if (e >= n_experts) {                      // no expert: the token's own row, weighted
#pragma unroll
          for (int o = 0; o < MOE_DOWN_PER_WAVE; ++o)
            same[o] = fmaf(c, load_as_float<T>(h + (size_t)t * W + min(n0 + o, W - 1)), same[o]);
          continue;
        }
        const T* yr = y + (size_t)ts * ff;
        const T* wr[MOE_DOWN_PER_WAVE];
#pragma unroll
        for (int o = 0; o < MOE_DOWN_PER_WAVE; ++o)
          wr[o] = down + ((size_t)e * W + min(n0 + o, W - 1)) * ff;
        float part[MOE_DOWN_PER_WAVE];
#pragma unroll
        for (int o = 0; o < MOE_DOWN_PER_WAVE; ++o) part[o] = 0.f;
        for (int i = lane * 8; i < ff; i += ZF_WAVE * 8) {
          uint4 a[MOE_DOWN_PER_WAVE];
#pragma unroll
          for (int o = 0; o < MOE_DOWN_PER_WAVE; ++o) a[o] = *(const uint4*)(wr[o] + i);
          const uint4 b = *(const uint4*)(yr + i);
          const uint32_t q[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
          for (int o = 0; o < MOE_DOWN_PER_WAVE; ++o) {
            const uint32_t p[4] = {a[o].x, a[o].y, a[o].z, a[o].w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
              part[o] = fmaf(__uint_as_float(p[k] << 16), __uint_as_float(q[k] << 16), part[o]);
              part[o] = fmaf(__uint_as_float(p[k] & 0xffff0000u),
                             __uint_as_float(q[k] & 0xffff0000u), part[o]);
            }
          }
        }
#pragma unroll
        for (int o = 0; o < MOE_DOWN_PER_WAVE; ++o) tot[o] = fmaf(c, part[o], tot[o]);
      }
#pragma unroll
      for (int o = 0; o < MOE_DOWN_PER_WAVE; ++o) {
        const float total = wave_sum(tot[o]) + same[o];
        if (lane == 0 && n0 + o < W) {
          float* dst = out + (size_t)t * W + n0 + o;
          *dst = add ? *dst + total : total;
        }
      }
      return;
    }
  }
  for (int n = n0; n < n0 + MOE_DOWN_PER_WAVE && n < W; ++n) {
    float total = 0.f;
    for (int s = 0; s < slots; ++s) {
      const int ts = t * slots + s;
      const int e = ids != nullptr ? ids[ts] : 0;
      if (e >= n_experts) {
        total += (weights != nullptr ? weights[ts] : 1.0f) * load_as_float<T>(h + (size_t)t * W + n);
        continue;
      }
      const T* wr = down + ((size_t)e * W + n) * ff;
      const T* yr = y + (size_t)ts * ff;
      const float dot = wave_sum(row_dot<T>(wr, yr, ff, lane));
      total += (weights != nullptr ? weights[ts] : 1.0f) * dot;
    }
    if (lane == 0) {
      float* o = out + (size_t)t * W + n;
      *o = add ? *o + total : total;
    }
  }
}

extern "C" int zf_moe_down(const void* y, const void* down, int dtype, const int* ids,
                           const float* weights, float* out, int T, int W, int ff, int slots,
                           int add, int n_experts, const void* h, hipStream_t stream) {
  if (T <= 0) return 0;
  if (W <= 0 || ff <= 0 || slots <= 0) return -2;
  const int per_wg = MOE_WAVES * MOE_DOWN_PER_WAVE;
  dim3 grid(T, (W + per_wg - 1) / per_wg);
  if (dtype == ZF_F32)
    hipLaunchKernelGGL(moe_down_kernel<float>, grid, dim3(MOE_WAVES * ZF_WAVE), 0, stream,
                       (const float*)y, (const float*)down, ids, weights, out, W, ff, slots, add,
                       n_experts, (const float*)h);
  else
    hipLaunchKernelGGL(moe_down_kernel<bf16_t>, grid, dim3(MOE_WAVES * ZF_WAVE), 0, stream,
                       (const bf16_t*)y, (const bf16_t*)down, ids, weights, out, W, ff, slots,
                       add, n_experts, (const bf16_t*)h);
  ZF_CHECK_LAUNCH();
}

// ---------------------------------------------------------------- the activation alone
// out[t, j] = act(gu[t, j], gu[t, ff + j]) for a gate/up product that a plain matrix kernel
// made (an expert that every token uses)
template <typename T>
__global__ void gated_act_kernel(const T* __restrict__ gu, T* __restrict__ out, int ff, size_t n,
                                 float limit, float alpha, float shift,
                                 const float* __restrict__ row_factor, int factor_stride) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const size_t t = i / ff, j = i % ff;
  const float g = load_as_float<T>(gu + t * 2 * ff + j);
  const float u = load_as_float<T>(gu + t * 2 * ff + ff + j);
  float r = gated_unit(g, u, limit, alpha, shift);
  if (row_factor != nullptr) r *= row_factor[t * factor_stride];
  store_from_float<T>(out + i, r);
}

extern "C" int zf_gated_act(const void* gu, void* out, int dtype, int T, int ff, float limit,
                            float alpha, float shift, const float* row_factor,
                            int factor_stride, hipStream_t stream) {
  const size_t n = (size_t)T * ff;
  if (n == 0) return 0;
  const unsigned blocks = (unsigned)((n + 255) / 256);
  if (dtype == ZF_F32)
    hipLaunchKernelGGL(gated_act_kernel<float>, dim3(blocks), dim3(256), 0, stream,
                       (const float*)gu, (float*)out, ff, n, limit, alpha, shift, row_factor,
                       factor_stride);
  else
    hipLaunchKernelGGL(gated_act_kernel<bf16_t>, dim3(blocks), dim3(256), 0, stream,
                       (const bf16_t*)gu, (bf16_t*)out, ff, n, limit, alpha, shift, row_factor,
                       factor_stride);
  ZF_CHECK_LAUNCH();
}

// =====================================================================================
//  Up to 16 tokens (bfloat16, matrices pre-tiled): every used expert's matrices are read once
//  for all tokens that chose it, 16 rows of a matrix against those tokens as columns of 16x16x32
//  MFMAs.  Token by token, 8 tokens with 4 of 32 experts each read 32 experts' worth where about
//  21 are used; the kernels are bound by that reading, and a CU alone draws no more than about a
//  256th of what the chip does, so both kernels spread it over all of them.
//    * moe_few_up    a workgroup of four waves per (unit, 16 outputs), K dealt to the waves in
//                    blocks of 64, the partials added in wave order; the activation in the
//                    epilogue.  A unit is an expert and up to 16 of its pairs (token, slot): the
//                    workgroup of pair p finds with a few ballots over the ids whether p starts a
//                    unit, else it ends.  The first workgroups take 16 outputs each of the expert
//                    that all tokens share, if there is one.
//    * moe_few_down  a workgroup of sixteen waves per 8 outputs, for all experts: (unit of up to 8
//                    pairs, piece of ff) after piece by each wave.  The 16 rows and columns of an
//                    MFMA are 8 outputs and 8 pairs at two neighbouring blocks of 64 of ff: only
//                    the products of like halves are used, and 2048 outputs make 256 workgroups.
//                    Partials in LDS, added per pair every fourth piece side by side, per token
//                    in slot order, the shared expert last.  (Fetching the next piece's operands before a
//                    piece's products was no faster; a workgroup per unit and 32 outputs whose last
//                    one to arrive adds the sums took 10 % less at W = 4096, 64 experts and 8
//                    tokens, 15 % more at 16 tokens, and more in the decode step.)
//  The matrices lie as the matrix kernels' pre-tiled ones, [rows / 16][K / 64][2][64 lanes][8]: a
//  wave's load is consecutive memory.  A column of an MFMA depends on its own token alone
//  and all sums have a fixed order: a token's bits do not depend on the others.
//  Measured (MI355X, both kernels in a graph, us, against the token-by-token kernels): W = 2048, ff
//  = 768, 32 experts, 4 a token: 1 token 18 -> 17.6, 8 tokens 55 -> 46 (21 experts: 24.6 for the
//  first, 5.9 TB/s, 22 for the second), 16 tokens 90 -> 71; W = 4096, ff = 1024, 64 experts, 8 a
//  token: 1 token 50 -> 42, 8 tokens 241 -> 204 (6.1 and 5.1 TB/s), 16 tokens 448 -> 283.
// =====================================================================================
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 moe_bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t moe_u32x4_t;

#define MOE_FEW_TOKENS 16
#define MOE_FEW_PAIRS 256

// (weights are read once a step: loads that need not stay in the caches)
__device__ __forceinline__ moe_u32x4_t few_load_w(const bf16_t* p) {
  return __builtin_nontemporal_load((const moe_u32x4_t*)p);
}

// Whether pair p, of expert e, starts a unit: up to 16 pairs of one expert, in their order; then
// `column` (LDS, the wave's own) holds them, -1 where there are fewer.  The same in every lane.
// Ids from n_experts on name no expert.  (A token may name an expert twice: 17 pairs, two units.)
__device__ __forceinline__ bool few_columns(const int* __restrict__ ids, int P, int p, int e,
                                            int n_experts, int lane, int* column) {
  if (e >= n_experts) return false;
  int id[4];
  unsigned long long uses[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int i = 64 * c + lane;
    id[c] = i < P ? ids[i] : -1;
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) uses[c] = __ballot(id[c] == e);
  int rank = 0;                              // pairs of this expert before p
#pragma unroll
  for (int c = 0; c < 4; ++c)
    if (p >= 64 * c)
      rank += __popcll(p >= 64 * c + 64 ? uses[c] : uses[c] & ((1ull << (p - 64 * c)) - 1));
  if (rank % 16 != 0) return false;
  if (lane < 16) column[lane] = -1;
  __builtin_amdgcn_wave_barrier();
  int before = -rank;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int at = before + __popcll(uses[c] & ((1ull << lane) - 1));
    if (id[c] == e && at >= 0 && at < 16) column[at] = 64 * c + lane;
    before += __popcll(uses[c]);
  }
  wave_lds_fence();
  return true;
}

// n (even) numbers, eight apart: four sums side by side, added in pairs
__device__ __forceinline__ float few_sum(const float* p, int n) {
  float a[4] = {0.f, 0.f, 0.f, 0.f};
  int q = 0;
#pragma unroll 4
  for (; q + 4 <= n; q += 4)
#pragma unroll
    for (int i = 0; i < 4; ++i) a[i] += p[8 * (q + i)];
  if (q < n) {
    a[0] += p[8 * q];
    a[1] += p[8 * q + 8];
  }
  return (a[0] + a[1]) + (a[2] + a[3]);
}

template <bool GATED>
__global__ __launch_bounds__(256) void moe_few_up_kernel(
    const bf16_t* __restrict__ h, const bf16_t* __restrict__ w, const int* __restrict__ ids,
    bf16_t* __restrict__ y, int T, int W, int ff, int top, float limit, float alpha, float shift,
    int act, int n_experts, const bf16_t* __restrict__ shared_w, bf16_t* __restrict__ shared_y,
    int shared_ff, float s_limit, float s_alpha, float s_shift, const float* __restrict__ factor,
    int factor_stride) {
  __shared__ moe_f32x4_t part[4][2][ZF_WAVE];
  __shared__ int column[4][16];
  const int wave = threadIdx.x / ZF_WAVE, lane = threadIdx.x % ZF_WAVE;
  const int r = lane % 16, g = lane / 16, shared_blocks = shared_ff / 16, blocks = W / 64;
  const bool shared = (int)blockIdx.x < shared_blocks;
  int pair, token, j0;                         // pair: this lane's column, -1: none
  const bf16_t *wg, *wu;
  if (shared) {
    j0 = blockIdx.x * 16;
    pair = r < T ? r : -1;
    token = r < T ? r : 0;
    wg = shared_w + (size_t)(j0 / 16) * blocks * 1024;
    wu = wg + (size_t)(shared_ff / 16) * blocks * 1024;
  } else {
    const int P = T * top, b = blockIdx.x - shared_blocks, p = b % P;
    j0 = b / P * 16;
    const int e = ids[p];
    if (!few_columns(ids, P, p, e, n_experts, lane, column[wave])) return;
    pair = column[wave][r];
    token = (pair >= 0 ? pair : p) / top;
    wg = w + ((size_t)e * (GATED ? 2 : 1) * ff + j0) / 16 * blocks * 1024;
    wu = wg + (size_t)(ff / 16) * blocks * 1024;
  }
  wg += lane * 8;
  wu += lane * 8;
  const bf16_t* x = h + (size_t)token * W + 16 * g;
  // Four sums side by side, of either half of even and odd blocks, closed every four blocks: one sum
  // over a wave's whole share of K is further off than the lane sums of the row-by-row kernel
  // (4096 columns, of the activations 0.043 % rounded the other way than the 64-bit ones, so 0.016
  // %, row by row 0.017 %).
  moe_f32x4_t sg[2][2], su[2][2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 2; ++i) sg[j][i] = su[j][i] = moe_f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto take = [&](auto J, int kb) {
    constexpr int j = decltype(J)::value;
    moe_u32x4_t xf[2], gf[2], uf[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      gf[i] = few_load_w(wg + (size_t)kb * 1024 + i * 512);
      if constexpr (GATED) uf[i] = few_load_w(wu + (size_t)kb * 1024 + i * 512);
      xf[i] = *(const moe_u32x4_t*)(x + kb * 64 + i * 8);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      sg[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const moe_bf16x8_t*)&gf[i],
                                                         *(const moe_bf16x8_t*)&xf[i], sg[j][i], 0, 0, 0);
      if constexpr (GATED)
        su[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const moe_bf16x8_t*)&uf[i],
                                                           *(const moe_bf16x8_t*)&xf[i], su[j][i], 0, 0, 0);
    }
  };
  int kb = wave;
  moe_f32x4_t ag = {0.f, 0.f, 0.f, 0.f}, au = ag;
  auto close = [&]() {
    ag += (sg[0][0] + sg[0][1]) + (sg[1][0] + sg[1][1]);
    if constexpr (GATED) au += (su[0][0] + su[0][1]) + (su[1][0] + su[1][1]);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i) sg[j][i] = su[j][i] = moe_f32x4_t{0.f, 0.f, 0.f, 0.f};
  };
#pragma unroll 1
  for (; kb + 4 < blocks; kb += 8) {
    take(std::integral_constant<int, 0>{}, kb);
    take(std::integral_constant<int, 1>{}, kb + 4);
    if (kb & 8) close();
  }
  if (kb < blocks) take(std::integral_constant<int, 0>{}, kb);
  close();
  part[wave][0][lane] = ag;
  part[wave][1][lane] = au;
  __syncthreads();
  if (wave != 0 || pair < 0) return;
  ag = (ag + part[1][0][lane]) + (part[2][0][lane] + part[3][0][lane]);
  au = (au + part[1][1][lane]) + (part[2][1][lane] + part[3][1][lane]);
  // column r is the pair, the four numbers are outputs j0 + 4 g + i
  const float f = shared && factor != nullptr ? factor[(size_t)pair * factor_stride] : 1.0f;
  uint32_t v[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float o;
    if constexpr (GATED)
      o = shared ? gated_unit(ag[i], au[i], s_limit, s_alpha, s_shift)
                 : gated_unit(ag[i], au[i], limit, alpha, shift);
    else
      o = activation_value(ag[i], act);
    v[i] = float_to_bf16(shared ? o * f : o);
  }
  bf16_t* dst = (shared ? shared_y + (size_t)pair * shared_ff : y + (size_t)pair * ff) + j0 + 4 * g;
  *(uint2*)dst = make_uint2(v[0] | v[1] << 16, v[2] | v[3] << 16);
}

__global__ __launch_bounds__(1024) void moe_few_down_kernel(
    const bf16_t* __restrict__ y, const bf16_t* __restrict__ down, const int* __restrict__ ids,
    const float* __restrict__ weights, float* __restrict__ out, int T, int W, int ff, int top,
    int add, int n_experts, const bf16_t* __restrict__ h, int piece,
    const bf16_t* __restrict__ shared_w, const bf16_t* __restrict__ shared_y, int shared_ff) {
  __shared__ int n_units, id[MOE_FEW_PAIRS], expert[MOE_FEW_PAIRS];
  __shared__ float share[MOE_FEW_PAIRS];
  __shared__ __attribute__((aligned(16))) short pairs[MOE_FEW_PAIRS][8];   // of a unit; -1: it has fewer
  extern __shared__ __attribute__((aligned(16))) float sums[];   // [pair][2 pieces][8], then shared's
  const int wave = threadIdx.x / ZF_WAVE, lane = threadIdx.x % ZF_WAVE;
  const int r = lane % 16, g = lane / 16, n0 = blockIdx.x * 8, P = T * top;
  const int blocks = ff / 64, pieces = (blocks + 2 * piece - 1) / (2 * piece);
  const int s_blocks = shared_ff / 64, s_pieces = (s_blocks + 2 * piece - 1) / (2 * piece);
  float* s_sums = sums + (size_t)P * pieces * 16;
  // what the sums at the end want, asked for now
  const int t = threadIdx.x / 8, n = threadIdx.x % 8;
  const float before = add && t < T ? out[(size_t)t * W + n0 + n] : 0.f;
  if (wave == 1)
    for (int i = lane; i < P; i += ZF_WAVE) share[i] = weights[i];
  // one wave lists the units, in the order of their first pairs
  if (wave == 0) {
    // This lane's pairs: experts, ranks among their expert's pairs, and the pair that starts their unit.
    // Pair j's own rank is there when its turn comes.
    int mine[4], rank[4] = {0, 0, 0, 0}, lead[4] = {0, 0, 0, 0};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int i = 64 * c + lane;
      mine[c] = i < P ? ids[i] : n_experts;
      if (i < P) id[i] = mine[c];
      *(moe_u32x4_t*)&pairs[i][0] = moe_u32x4_t{~0u, ~0u, ~0u, ~0u};
    }
#pragma unroll
    for (int cj = 0; cj < 4; ++cj)
      for (int j = 0; j < min(64, P - 64 * cj); ++j) {
        const int e = __builtin_amdgcn_readlane(mine[cj], j);
        const bool starts = __builtin_amdgcn_readlane(rank[cj], j) % 8 == 0;
#pragma unroll
        for (int c = cj; c < 4; ++c)
          if (64 * c < P) {
            const bool same = mine[c] == e && (c > cj || j <= lane);
            if (same && starts) lead[c] = 64 * cj + j;
            rank[c] += same && (c > cj || j < lane);
          }
      }
    unsigned long long first[4];
    int units = 0, before[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      first[c] = __ballot(mine[c] < n_experts && rank[c] % 8 == 0);
      before[c] = units;
      units += __popcll(first[c]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (mine[c] < n_experts) {
        const int cl = lead[c] / 64, l = lead[c] % 64;
        const unsigned long long f = cl == 0 ? first[0] : cl == 1 ? first[1] : cl == 2 ? first[2] : first[3];
        const int unit = (cl == 0 ? before[0] : cl == 1 ? before[1] : cl == 2 ? before[2] : before[3]) +
                         __popcll(f & ((1ull << l) - 1));
        pairs[unit][rank[c] % 8] = (short)(64 * c + lane);
        if (rank[c] % 8 == 0) expert[unit] = mine[c];
      }
    if (lane == 0) n_units = units;
  }
  __syncthreads();
  const int jobs = n_units * pieces + s_pieces, half = r / 8;
  for (int q = wave; q < jobs; q += 16) {
    const bool shared = q < s_pieces;
    const int unit = (q - s_pieces) / pieces, c = shared ? q : (q - s_pieces) % pieces;
    const int nb = shared ? s_blocks : blocks;
    int pair;
    const bf16_t *wr, *x;
    // (the two halves of the blocks in a sum each, the pieces' sums four side by side: the outputs of ff
    // = 4096 from given activations 1.34e-7 off with one sum, 1.04e-7 so, 1.05e-7 row by row)
    // rows r and columns r: output n0 + r % 8 and pair r % 8 at the blocks 2 i + r / 8
    for (int p0 = 0; p0 < (shared ? T : 8); p0 += 8) {
      if (shared) {
        pair = p0 + r % 8 < T ? p0 + r % 8 : -1;
        wr = shared_w;
        x = shared_y + (size_t)max(pair, 0) * shared_ff;
      } else {
        pair = pairs[unit][r % 8];
        wr = down + (size_t)expert[unit] * W * ff;
        x = y + (size_t)(pair >= 0 ? pair : pairs[unit][0]) * ff;
      }
      wr += (size_t)(n0 / 16) * nb * 1024 + (g * 16 + n0 % 16 + r % 8) * 8;
      x += 16 * g;
      const int b0 = c * 2 * piece, b1 = min(nb, b0 + 2 * piece);
      moe_f32x4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll 4
      for (int kb = b0; kb < b1; kb += 2) {
        // (behind an odd last block the upper half repeats it against zeros)
        const bool in = kb + half < b1;
        const int k = in ? kb + half : kb;
        moe_u32x4_t wf[2], xf[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          wf[i] = few_load_w(wr + (size_t)k * 1024 + i * 512);
          xf[i] = *(const moe_u32x4_t*)(x + k * 64 + i * 8);
          if (!in) wf[i] = xf[i] = moe_u32x4_t{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const moe_bf16x8_t*)&wf[i],
                                                           *(const moe_bf16x8_t*)&xf[i], acc[i], 0, 0, 0);
      }
      // rows 4 g + i of column r: like halves are g / 2 == half
      if (pair >= 0 && g / 2 == half)
        *(moe_f32x4_t*)((shared ? s_sums + ((size_t)pair * s_pieces + c) * 16
                                : sums + ((size_t)pair * pieces + c) * 16) + 8 * half + 4 * (g % 2)) =
            acc[0] + acc[1];
    }
  }
  __syncthreads();
  if (t >= T) return;
  float total = 0.f, same = 0.f;
  for (int s = 0; s < top; ++s) {
    const int ts = t * top + s;
    const float c = share[ts];
    if (id[ts] >= n_experts) {                  // no expert: the token's own row, weighted
      same = fmaf(c, bf16_to_float(h[(size_t)t * W + n0 + n]), same);
      continue;
    }
    total = fmaf(c, few_sum(sums + (size_t)ts * pieces * 16 + n, 2 * pieces), total);
  }
  total += same;
  if (add) total += before;
  if (s_pieces > 0) total += few_sum(s_sums + (size_t)t * s_pieces * 16 + n, 2 * s_pieces);
  out[(size_t)t * W + n0 + n] = total;
}

// The whole feed-forward of up to 16 tokens: y (work space, bfloat16 [T, top, ff]) and out float32
// [T, W] (=, add: +=).  gated: gate_up [E, 2 ff, W]; else [E, ff, W] and the plain activation
// `act`; every expert's matrices pre-tiled.  Ids from n_experts on name no expert: their term is
// the weight times h[t].  shared_ff > 0: an expert that all tokens share is added, pre-tiled as
// well, its activations times factor[t * factor_stride] if given, in shared_y [T, shared_ff].
// Rows and matrices 16-byte aligned.
extern "C" int zf_moe_few(const void* h, const void* gate_up, const void* down, const int* ids,
                          const float* weights, void* y, float* out, int T, int W, int ff, int top,
                          float limit, float alpha, float shift, int add, int gated, int act,
                          int n_experts, const void* shared_gate_up, const void* shared_down,
                          void* shared_y, int shared_ff, float s_limit, float s_alpha,
                          float s_shift, const float* factor, int factor_stride,
                          hipStream_t stream) {
  if (T <= 0) return 0;
  if (T > MOE_FEW_TOKENS || W <= 0 || ff <= 0 || top <= 0 || W % 64 != 0 || ff % 64 != 0 ||
      T * top > MOE_FEW_PAIRS || n_experts <= 0 || act < 0 || act > 4 || shared_ff < 0 ||
      shared_ff % 64 != 0 || (shared_ff > 0 && !gated))
    return -2;
  const uintptr_t all = (uintptr_t)h | (uintptr_t)gate_up | (uintptr_t)down | (uintptr_t)y |
                        (uintptr_t)out | (uintptr_t)shared_gate_up | (uintptr_t)shared_down |
                        (uintptr_t)shared_y;
  if (all % 16 != 0) return -2;
  const dim3 up_grid(shared_ff / 16 + T * top * (ff / 16));
#define MOE_FEW_UP(G)                                                                             \
  hipLaunchKernelGGL(moe_few_up_kernel<G>, up_grid, dim3(256), 0, stream, (const bf16_t*)h,       \
                     (const bf16_t*)gate_up, ids, (bf16_t*)y, T, W, ff, top, limit, alpha, shift, \
                     act, n_experts, (const bf16_t*)shared_gate_up, (bf16_t*)shared_y, shared_ff, \
                     s_limit, s_alpha, s_shift, factor, factor_stride)
  if (gated) MOE_FEW_UP(true); else MOE_FEW_UP(false);
#undef MOE_FEW_UP
  // pieces of 2 x 128 of ff, larger ones where the partials of 16 tokens would not fit 48 KB of
  // LDS (by the layer's sizes alone: a token's sums must not depend on how many tokens there are).
  // Pieces of up to 8 blocks, their sums in four accumulators, were 4 to 8 % slower for one or two tokens of
  // top 1 and 2 (W = 2048, ff = 512, us 12.3 for 13.1) and 2 to 4 % faster only for some of eight and more.
  int piece = 2;
  const auto pieces = [](int width, int p) { return (width / 64 + 2 * p - 1) / (2 * p); };
  const auto lds = [&](int tokens, int p) {
    return (size_t)tokens * (top * pieces(ff, p) + pieces(shared_ff, p)) * 64;
  };
  while (lds(MOE_FEW_TOKENS, piece) > 48 * 1024 && piece < (ff + shared_ff) / 64) piece *= 2;
  if (lds(T, piece) > 48 * 1024) return -2;
  hipLaunchKernelGGL(moe_few_down_kernel, dim3(W / 8), dim3(1024), lds(T, piece), stream,
                     (const bf16_t*)y, (const bf16_t*)down, ids, weights, out, T, W, ff, top, add,
                     n_experts, (const bf16_t*)h, piece, (const bf16_t*)shared_down,
                     (const bf16_t*)shared_y, shared_ff);
  ZF_CHECK_LAUNCH();
}

// =====================================================================================
//  Many tokens (bfloat16): the (token, slot) pairs are sorted by expert, and every expert's
//  pairs run through MFMA tiles of 128 pairs against that expert's matrices.
//
//  * moe_sort      one workgroup: counts per expert, the pairs in expert order (`sorted`: the
//                  pair at a place, `place`: the place of a pair), and the list of tiles
//                  (expert, first place, places), their number in n_tiles[0].
//  * moe_grouped   grid (tile, columns): GATED: y[place, j] = act(gate, up) of the pair's token
//                  (rows of h gathered through `sorted`); else o[place, n] = down y[place] in
//                  32-bit.  A row's result depends on that row and the expert's matrix alone
//                  (sums along K in a fixed order), not on the rows beside it in the tile.
//  * moe_combine   out[t] (=, +=) sum over the slots, in slot order, of weight * o[place].
// =====================================================================================
#define MOE_TILE_ROWS 128

__global__ __launch_bounds__(1024) void moe_sort_kernel(
    const int* __restrict__ ids, int P, int E, int* __restrict__ sorted, int* __restrict__ place,
    int* __restrict__ tile_expert, int* __restrict__ tile_row0, int* __restrict__ tile_rows,
    int* __restrict__ n_tiles) {
  __shared__ int count[MOE_MAX_EXPERTS], start[MOE_MAX_EXPERTS], cursor[MOE_MAX_EXPERTS];
  for (int e = threadIdx.x; e < E; e += blockDim.x) { count[e] = 0; cursor[e] = 0; }
  __syncthreads();
  for (int i = threadIdx.x; i < P; i += blockDim.x) atomicAdd(&count[ids[i]], 1);
  __syncthreads();
  if (threadIdx.x == 0) {
    int at = 0, tiles = 0;
    for (int e = 0; e < E; ++e) {
      start[e] = at;
      for (int r = 0; r < count[e]; r += MOE_TILE_ROWS) {
        tile_expert[tiles] = e;
        tile_row0[tiles] = at + r;
        tile_rows[tiles] = min(MOE_TILE_ROWS, count[e] - r);
        ++tiles;
      }
      at += count[e];
    }
    n_tiles[0] = tiles;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < P; i += blockDim.x) {
    const int e = ids[i];
    const int at = start[e] + atomicAdd(&cursor[e], 1);
    sorted[at] = i;
    place[i] = at;
  }
}

extern "C" int zf_moe_sort(const int* ids, int P, int E, int* sorted, int* place, int* tile_expert,
                           int* tile_row0, int* tile_rows, int* n_tiles, hipStream_t stream) {
  if (P <= 0) return 0;
  if (E <= 0 || E > MOE_MAX_EXPERTS) return -2;
  hipLaunchKernelGGL(moe_sort_kernel, dim3(1), dim3(1024), 0, stream, ids, P, E, sorted, place,
                     tile_expert, tile_row0, tile_rows, n_tiles);
  ZF_CHECK_LAUNCH();
}

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float moe_f32x16_t;

#define MOE_BK 64
#define MOE_LD (MOE_BK + 8)      // row stride in LDS (bfloat16): 16-byte reads of 8 lanes cover all banks

// 4 waves as 2 x 2: a wave takes 64 of the tile's 128 rows and 32 of the 64 columns of each of
// the MOE_NB weight tiles (GATED: the gate rows of MOE_NB / 2 groups of 64 outputs, then the up
// rows of the same outputs; else MOE_NB neighbouring groups of 64 outputs).  Two tiles, three
// workgroups to a CU, ran faster than four tiles with one or two, and loads issued one step
// ahead faster than two.  What bounds the loop with a few hundred rows an expert is the
// experts' matrices coming from memory: the tiles of one expert are dealt to workgroups whose
// numbers are equal modulo 8, which share an XCD and so its L2.
// v_mfma_f32_32x32x16_bf16: a lane holds row (or column) lane % 32 and k 8 (lane / 32) .. + 8
// of an operand, and of the result column lane % 32, rows 8 (r / 4) + 4 (lane / 32) + r % 4.
#define MOE_NB 2                 // weight tiles of 64 rows a workgroup holds
#define MOE_HALF (MOE_NB / 2)
// MODE 0: the down pass; 1: gate and up with the gated activation; 2: up alone, w [E, N, K], with
// the plain activation `act`.
// TILED: every expert's matrices pre-tiled (K a multiple of 64, their rows of 16).  ONCE: mostly one
// tile of rows an expert, so that nobody reads the matrices again and their loads need not stay in
// the caches.
template <int MODE, bool TILED, bool ONCE>
__global__ __launch_bounds__(256) void moe_grouped_kernel(
    const bf16_t* __restrict__ a, long long lda, const int* __restrict__ sorted, int top,
    const bf16_t* __restrict__ w, const int* __restrict__ tile_expert,
    const int* __restrict__ tile_row0, const int* __restrict__ tile_rows,
    const int* __restrict__ n_tiles, void* __restrict__ out, int N, int K, float limit,
    float alpha, float shift, int act, int n_experts) {
  constexpr bool GATED = MODE == 1;
  constexpr bool GATHER = MODE != 0;            // rows of h found through the sort
  __shared__ __attribute__((aligned(16))) bf16_t as[MOE_TILE_ROWS * MOE_LD];
  __shared__ __attribute__((aligned(16))) bf16_t bs[MOE_NB * 64 * MOE_LD];
  // gridDim.x is a multiple of 8: workgroup x takes tile (x % 8) * (gridDim.x / 8) + x / 8, so
  // that neighbouring tiles (the same expert's) run on one XCD at about the same time
  const int tile = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
  if (tile >= n_tiles[0]) return;
  const int e = tile_expert[tile], row0 = tile_row0[tile], nrows = tile_rows[tile];
  if (e >= n_experts) return;                      // an output of the router without an expert
  const int c0 = blockIdx.y * 64 * (GATED ? MOE_HALF : MOE_NB);
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int wm = wave / 2, wn = wave % 2;

  // what this thread stages: rows tid / 8 + 32 i of the pairs' tile (i < 4) and of the
  // weight tiles (i < 2 MOE_NB), 8 values at k0 + 8 (tid % 8)
  const int sr = tid / 8, sk = (tid % 8) * 8;
  // of pre-tiled matrices ([rows / 16][K / 64][2][64][8]; MOE_BK = 64: a step is one block of 64)
  // consecutive threads take consecutive memory: piece p = tid + 256 i is lane p % 64 of half
  // (p / 64) % 2 of row group p / 128, i.e. row 16 (p / 128) + p % 16 at k 16 (p % 64 / 16) + 8
  // half (through the row mapping above the same loads scattered 16-byte pieces: 5 to 10 % of
  // the kernel's time)
  const bf16_t* ap[4];
  const bf16_t* bp[2 * MOE_NB];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = sr + 32 * i;
    ap[i] = nullptr;
    if (r < nrows) {
      const int src = GATHER ? sorted[row0 + r] / top : row0 + r;
      ap[i] = a + (size_t)src * lda;
    }
  }
#pragma unroll
  for (int i = 0; i < 2 * MOE_NB; ++i) {
    const int r = TILED ? 16 * ((tid + 256 * i) / 128) + tid % 16 : sr + 32 * i;
    const int br = r % 64, bt = r / 64;              // row br of weight tile bt
    size_t wrow;
    bool ok;
    if (GATED) {                                     // the first half of the tiles: gate; then up
      const int j = c0 + (bt % MOE_HALF) * 64 + br;
      ok = j < N;
      wrow = (size_t)e * 2 * N + (size_t)(bt / MOE_HALF) * N + j;
    } else {
      const int n = c0 + bt * 64 + br;
      ok = n < N;
      wrow = (size_t)e * N + n;
    }
    bp[i] = !ok ? nullptr
        : TILED ? w + wrow / 16 * (K / 64) * 1024 + tid % 128 * 8 : w + wrow * K + sk;
  }
  moe_f32x16_t acc[2][MOE_NB];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < MOE_NB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const moe_u32x4_t zero = {0u, 0u, 0u, 0u};
  moe_u32x4_t ra[4], rb[2 * MOE_NB];
  auto fetch = [&](int k0) {
    const bool in_k = k0 + sk < K;                   // K is a multiple of 8
#pragma unroll
    for (int i = 0; i < 4; ++i)
      ra[i] = (ap[i] != nullptr && in_k) ? *(const moe_u32x4_t*)(ap[i] + k0 + sk) : zero;
#pragma unroll
    for (int i = 0; i < 2 * MOE_NB; ++i)
      if (bp[i] == nullptr || !(TILED || in_k))
        rb[i] = zero;
      else if constexpr (ONCE)
        rb[i] = few_load_w(bp[i] + (size_t)k0 * 16);
      else
        rb[i] = *(const moe_u32x4_t*)(bp[i] + (TILED ? (size_t)k0 * 16 : (size_t)k0));
  };
  fetch(0);
  for (int k0 = 0; k0 < K; k0 += MOE_BK) {
    __syncthreads();                                 // the tiles of the step before are done with
#pragma unroll
    for (int i = 0; i < 4; ++i) *(moe_u32x4_t*)(as + (sr + 32 * i) * MOE_LD + sk) = ra[i];
#pragma unroll
    for (int i = 0; i < 2 * MOE_NB; ++i)
      *(moe_u32x4_t*)(bs + (TILED ? (16 * ((tid + 256 * i) / 128) + tid % 16) * MOE_LD +
                                        tid % 64 / 16 * 16 + tid % 128 / 64 * 8
                                  : (sr + 32 * i) * MOE_LD + sk)) = rb[i];
    __syncthreads();
    if (k0 + MOE_BK < K) fetch(k0 + MOE_BK);         // in flight while the MFMAs run
#pragma unroll
    for (int ks = 0; ks < MOE_BK; ks += 16) {
      moe_bf16x8_t af[2], bf[MOE_NB];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        af[i] = *(const moe_bf16x8_t*)(as + (wm * 64 + i * 32 + lane % 32) * MOE_LD + ks + 8 * (lane / 32));
#pragma unroll
      for (int j = 0; j < MOE_NB; ++j)
        bf[j] = *(const moe_bf16x8_t*)(bs + (j * 64 + wn * 32 + lane % 32) * MOE_LD + ks + 8 * (lane / 32));
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < MOE_NB; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bf[j], acc[i][j], 0, 0, 0);
    }
  }
  const int col = wn * 32 + lane % 32;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = wm * 64 + i * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4;
      if (row >= nrows) continue;
      if (GATED) {
#pragma unroll
        for (int j = 0; j < MOE_HALF; ++j)
          if (c0 + j * 64 + col < N)
            ((bf16_t*)out)[(size_t)(row0 + row) * N + c0 + j * 64 + col] =
                float_to_bf16(gated_unit(acc[i][j][r], acc[i][MOE_HALF + j][r], limit, alpha, shift));
      } else if (MODE == 2) {
#pragma unroll
        for (int j = 0; j < MOE_NB; ++j)
          if (c0 + j * 64 + col < N)
            ((bf16_t*)out)[(size_t)(row0 + row) * N + c0 + j * 64 + col] =
                float_to_bf16(activation_value(acc[i][j][r], act));
      } else {
#pragma unroll
        for (int j = 0; j < MOE_NB; ++j)
          if (c0 + j * 64 + col < N)
            ((float*)out)[(size_t)(row0 + row) * N + c0 + j * 64 + col] = acc[i][j][r];
      }
    }
}

// mode 1: a = h [T, K] (rows gathered), w = gate_up [E, 2 N, K], out = y bfloat16 [P, N];
// mode 2: the same with w = up [E, N, K] and the plain activation `act`;
// mode 0: a = y [P, K], w = down [E, N, K], out = o float32 [P, N].  K a multiple of 8.
// w_tiled 1: matrices pre-tiled; 2: and mostly read once (ONCE above).
extern "C" int zf_moe_grouped(const void* a, long long lda, const int* sorted, int top,
                              const void* w, const int* tile_expert, const int* tile_row0,
                              const int* tile_rows, const int* n_tiles, void* out, int max_tiles,
                              int N, int K, int mode, float limit, float alpha, float shift,
                              int act, int n_experts, int w_tiled, hipStream_t stream) {
  if (max_tiles <= 0) return 0;
  if (N <= 0 || K <= 0 || K % 8 != 0 || top <= 0 || mode < 0 || mode > 2 || act < 0 || act > 4 ||
      (w_tiled && (K % 64 != 0 || N % 16 != 0)))
    return -2;
  max_tiles = (max_tiles + 7) / 8 * 8;
#define MOE_GROUPED_LAUNCH(MODE, COLS)                                                           \
  if (w_tiled == 2) MOE_GROUPED_LAUNCH_AS(MODE, true, true, COLS);                               \
  else if (w_tiled) MOE_GROUPED_LAUNCH_AS(MODE, true, false, COLS);                              \
  else MOE_GROUPED_LAUNCH_AS(MODE, false, false, COLS)
#define MOE_GROUPED_LAUNCH_AS(MODE, TILED, ONCE, COLS)                                           \
  hipLaunchKernelGGL((moe_grouped_kernel<MODE, TILED, ONCE>), dim3(max_tiles, (N + (COLS) - 1) / (COLS)), \
                     dim3(256), 0, stream, (const bf16_t*)a, lda, sorted, top, (const bf16_t*)w, \
                     tile_expert, tile_row0, tile_rows, n_tiles, out, N, K, limit, alpha, shift, \
                     act, n_experts)
  if (mode == 1) {
    MOE_GROUPED_LAUNCH(1, 64 * MOE_HALF);
  } else if (mode == 2) {
    MOE_GROUPED_LAUNCH(2, 64 * MOE_NB);
  } else {
    MOE_GROUPED_LAUNCH(0, 64 * MOE_NB);
  }
  ZF_CHECK_LAUNCH();
}

__global__ __launch_bounds__(256) void moe_combine_kernel(
    const float* __restrict__ o, const int* __restrict__ place, const float* __restrict__ weights,
    float* __restrict__ out, int W, int slots, int add, const int* __restrict__ ids,
    int n_experts, const bf16_t* __restrict__ h) {
  const int t = blockIdx.x;
  for (int n = blockIdx.y * blockDim.x + threadIdx.x; n < W; n += gridDim.y * blockDim.x) {
    float total = 0.f;
    for (int s = 0; s < slots; ++s) {
      const int ts = t * slots + s;
      // an output of the router without an expert hands the token's own row on
      const float v = (ids != nullptr && ids[ts] >= n_experts)
          ? bf16_to_float(h[(size_t)t * W + n]) : o[(size_t)place[ts] * W + n];
      total += weights[ts] * v;
    }
    float* dst = out + (size_t)t * W + n;
    *dst = add ? *dst + total : total;
  }
}

extern "C" int zf_moe_combine(const float* o, const int* place, const float* weights, float* out,
                              int T, int W, int slots, int add, const int* ids, int n_experts,
                              const void* h, hipStream_t stream) {
  if (T <= 0) return 0;
  if (W <= 0 || slots <= 0) return -2;
  int gy = (W + 255) / 256;
  if (gy > 64) gy = 64;
  hipLaunchKernelGGL(moe_combine_kernel, dim3(T, gy), dim3(256), 0, stream, o, place, weights,
                     out, W, slots, add, ids, n_experts, (const bf16_t*)h);
  ZF_CHECK_LAUNCH();
}
