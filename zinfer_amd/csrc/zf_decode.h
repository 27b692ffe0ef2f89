// The arithmetic of the bfloat16 decode attention on a wave's 64 keys, for every kernel that decodes.
// Keys and values lie in tiled pools, as attention.hip lays them out.
#pragma once
#include "zf_common.h"

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_t;
typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2_t;

// 2^x for x <= 0 as the bare v_exp_f32 (1 ulp; -inf gives 0, results below 2^-126 may come
// out as 0): exp2f() wraps the same instruction in five more that rescale such tiny results,
// which a soft-max term does not need.
__device__ __forceinline__ float exp2_raw(float x) { return __builtin_amdgcn_exp2f(x); }

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  return pack_bf16x2(lo, hi);
}

// keeps elements [n_lo, n_hi) of the 4 bfloat16 in v (element 0 in the low bits), zeroes the rest
__device__ __forceinline__ u32x2_t keep_range4(u32x2_t v, int n_lo, int n_hi) {
  uint64_t x = ((uint64_t)v[1] << 32) | v[0];
  n_lo = max(0, min(4, n_lo));
  n_hi = max(0, min(4, n_hi));
  uint64_t m = 0;
  if (n_hi > n_lo) {
    const uint64_t hi = n_hi == 4 ? ~0ull : ((1ull << (16 * n_hi)) - 1);
    const uint64_t lo = (1ull << (16 * n_lo)) - 1;
    m = hi & ~lo;
  }
  x &= m;
  return u32x2_t{(uint32_t)x, (uint32_t)(x >> 32)};
}

#define DEC_SPLIT 256
#define DEC_WAVE_KEYS 64

// The scores of a wave's 64 keys against the G query columns, their soft-max terms and the
// product with the values.  kf, vf and qf are the MFMA operands as the loads leave them; m, l
// and o the wave's maximum, sum and un-normalised output.  One order of operations for every
// kernel that decodes.
//
// PATCH: key kb + pn (0 <= pn < 64; pn < 0: none) is not what kf and vf hold for it but the
// row k_new / v_new in LDS (the token's own key and value, which the cache did not hold yet
// when the loads were asked for).  Its scores come from MFMAs of their own over a tile that
// holds the row in its place, and land in the lanes and registers that hold that key's scores
// anyway: an MFMA's output element depends on its own row and column alone, so the scores, and
// with them everything after, are the bits that operands read from the cache would give.
// NG: groups of 16 keys, 4 or 2.
template <int HD, bool PATCH, int NG>
__device__ __forceinline__ void decode_scores(const u32x4_t (&kf)[NG][HD / 32],
                                              const bf16x8_t (&qf)[HD / 32], int kb, int k_begin,
                                              int k_end, int qd, float scale_log2e, float& m,
                                              float& l, float (&sc)[4 * NG], int pn,
                                              const bf16_t* k_new) {
  f32x4_t st[NG];
#pragma unroll
  for (int h = 0; h < NG; ++h) {
    st[h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int stp = 0; stp < HD / 32; ++stp)
      st[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8_t*)&kf[h][stp], qf[stp],
                                                      st[h], 0, 0, 0);
  }
  const int hn = pn / 16, jn = pn % 16, lane16 = threadIdx.x % 16;
  if constexpr (PATCH) {
    if (pn >= 0) {
      // lane (j, qd) holds of a 16-key tile the row j, elements 32 stp + 8 qd .. + 7
      f32x4_t sn = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int stp = 0; stp < HD / 32; ++stp) {
        u32x4_t kx = *(const u32x4_t*)(k_new + stp * 32 + 8 * qd);
        if (lane16 != jn) kx = u32x4_t{0, 0, 0, 0};
        sn = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8_t*)&kx, qf[stp], sn, 0, 0, 0);
      }
      // its scores: element jn % 4 of the lanes with qd = jn / 4, in group hn
#pragma unroll
      for (int h = 0; h < NG; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (h == hn && r == jn % 4 && qd == jn / 4) st[h][r] = sn[r];
    }
  }
  // st[h][r]: key kb + 16 h + 4 qd + r, query column j
#pragma unroll
  for (int h = 0; h < NG; ++h)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = kb + 16 * h + 4 * qd + r;
      const float v = (key >= k_begin && key < k_end) ? st[h][r] * scale_log2e : -INFINITY;
      sc[h * 4 + r] = v;
      m = fmaxf(m, v);
    }
  m = apart_max<16>(m);
  m = apart_max<32>(m);
#pragma unroll
  for (int e = 0; e < 4 * NG; ++e) {
    sc[e] = exp2_raw(sc[e] - m);
    l += sc[e];
  }
  l = apart_sum<16>(l);
  l = apart_sum<32>(l);
}
template <int HD, bool PATCH, int NG>
__device__ __forceinline__ void decode_values(const u32x2_t (&vf)[NG][HD / 16],
                                              const float (&sc)[4 * NG], int kb, int k_begin,
                                              int k_end, int qd, f32x4_t (&o)[HD / 16], int pn,
                                              const bf16_t* v_new) {
  const int hn = pn / 16, jn = pn % 16, lane16 = threadIdx.x % 16;
#pragma unroll
  for (int hh = 0; hh < NG / 2; ++hh) {     // two MFMAs of 32 keys: groups 2 hh and 2 hh + 1
    u32x4_t pk = u32x4_t{pack_bf16(sc[8 * hh + 0], sc[8 * hh + 1]),
                         pack_bf16(sc[8 * hh + 2], sc[8 * hh + 3]),
                         pack_bf16(sc[8 * hh + 4], sc[8 * hh + 5]),
                         pack_bf16(sc[8 * hh + 6], sc[8 * hh + 7])};
    const bf16x8_t pf = *(bf16x8_t*)&pk;
    const int b0 = kb + 32 * hh + 4 * qd, b1 = b0 + 16;
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) {
      // stale or poisoned rows outside [k_begin, k_end) are zeroed: 0 * NaN would spoil the sum
      u32x2_t v0 = keep_range4(vf[2 * hh][dt], k_begin - b0, k_end - b0);
      u32x2_t v1 = keep_range4(vf[2 * hh + 1][dt], k_begin - b1, k_end - b1);
      if constexpr (PATCH) {
        // the lanes with qd = jn / 4 hold the values of keys 4 qd .. 4 qd + 3 at head
        // element 16 dt + j, 16 bits each
        if (pn >= 0 && hn / 2 == hh && qd == jn / 4) {
          const uint32_t vn = v_new[16 * dt + lane16];
          u32x2_t& v = hn % 2 ? v1 : v0;
          const int w = (jn % 4) / 2, sh = 16 * (jn % 2);
          v[w] = (v[w] & ~(0xffffu << sh)) | (vn << sh);
        }
      }
      u32x4_t vv = u32x4_t{v0[0], v0[1], v1[0], v1[1]};
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(bf16x8_t*)&vv, pf, o[dt], 0, 0, 0);
    }
  }
}
template <int HD, bool PATCH = false>
__device__ __forceinline__ void decode_attend(const u32x4_t (&kf)[4][HD / 32],
                                              const u32x2_t (&vf)[4][HD / 16],
                                              const bf16x8_t (&qf)[HD / 32], int kb, int k_begin,
                                              int k_end, int qd, float scale_log2e, float& m,
                                              float& l, f32x4_t (&o)[HD / 16], int pn = -1,
                                              const bf16_t* k_new = nullptr,
                                              const bf16_t* v_new = nullptr) {
  float sc[16];
  decode_scores<HD, PATCH, 4>(kf, qf, kb, k_begin, k_end, qd, scale_log2e, m, l, sc, pn, k_new);
  decode_values<HD, PATCH, 4>(vf, sc, kb, k_begin, k_end, qd, o, pn, v_new);
}
