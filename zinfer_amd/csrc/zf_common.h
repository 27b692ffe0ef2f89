// Shared device helpers for the gfx950 kernels: bfloat16 <-> float, wave (64 lanes) and
// block reductions, element loads templated on the storage type.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define ZF_WAVE 64

typedef uint16_t bf16_t;  // raw bfloat16 bits

// bits << 16 (src/tensor/formats/bfloat16.zig:3-6 of the reference)
__device__ __forceinline__ float bf16_to_float(bf16_t b) {
  return __uint_as_float(((uint32_t)b) << 16);
}

// round to nearest even, (bits + 0x7fff + lsb) >> 16 (bfloat16.zig:8-13), a NaN stays a NaN:
// gfx950 has an instruction for it (v_cvt_pk_bf16_f32), which the cast below becomes; it
// gives the same 16 bits as the formula for every one of the 2^32 inputs
__device__ __forceinline__ bf16_t float_to_bf16(float f) {
  const __bf16 b = (__bf16)f;
  return *(const bf16_t*)&b;
}
// two values in one register, `lo` in the low half
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  typedef __bf16 bf16x2_native __attribute__((ext_vector_type(2)));
  typedef float floatx2_native __attribute__((ext_vector_type(2)));
  const bf16x2_native v = __builtin_convertvector(floatx2_native{lo, hi}, bf16x2_native);
  return *(const uint32_t*)&v;
}

template <typename T> __device__ __forceinline__ float load_as_float(const T* p);
template <> __device__ __forceinline__ float load_as_float<float>(const float* p) { return *p; }
template <> __device__ __forceinline__ float load_as_float<bf16_t>(const bf16_t* p) {
  return bf16_to_float(*p);
}
template <typename T> __device__ __forceinline__ void store_from_float(T* p, float v);
template <> __device__ __forceinline__ void store_from_float<float>(float* p, float v) { *p = v; }
template <> __device__ __forceinline__ void store_from_float<bf16_t>(bf16_t* p, float v) {
  *p = float_to_bf16(v);
}

// Between what a wave's lanes lay down in LDS and what its other lanes read there (or the other way round): a
// wave's LDS accesses run in order, this keeps the compiler from moving them.  No instruction.
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The value of lane l xor OFF, OFF 1, 2, 4 or 8: register moves within a row of 16 lanes instead of a
// shuffle's way through LDS (about 60 cycles a step).  OFF 4 takes the quads of four lanes with
// an even number from the quad behind and those with an odd one from the quad before.
template <int CTRL, int BANKS = 0xf>
__device__ __forceinline__ float lane_move(float v, float old) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), CTRL,
                                                    0xf, BANKS, BANKS == 0xf));
}
template <int OFF>
__device__ __forceinline__ float lane_xor(float v) {
  static_assert(OFF == 1 || OFF == 2 || OFF == 4 || OFF == 8, "within a row of 16 lanes");
  if constexpr (OFF == 1) return lane_move<0xB1>(v, v);           // quad_perm [1, 0, 3, 2]
  else if constexpr (OFF == 2) return lane_move<0x4E>(v, v);      // quad_perm [2, 3, 0, 1]
  else if constexpr (OFF == 8) return lane_move<0x128>(v, v);     // row_ror 8
  else return lane_move<0x114, 0xA>(v, lane_move<0x104, 0x5>(v, v));   // row_shl 4, row_shr 4
}
// f of the values of lanes l and l xor OFF, OFF 32 or 16: the two copies that the swap leaves hold the
// wave's halves (the rows of 16 of each half) lane by lane
template <int OFF, typename F>
__device__ __forceinline__ float lanes_apart(float v, F f) {
  static_assert(OFF == 32 || OFF == 16, "a half or a row");
  typedef unsigned int lanes_u2 __attribute__((ext_vector_type(2)));
  const uint32_t u = __float_as_uint(v);
  const lanes_u2 r = OFF == 32 ? __builtin_amdgcn_permlane32_swap(u, u, false, false)
                               : __builtin_amdgcn_permlane16_swap(u, u, false, false);
  return f(__uint_as_float(r.x), __uint_as_float(r.y));
}
template <int OFF>
__device__ __forceinline__ float apart_sum(float v) {
  return lanes_apart<OFF>(v, [](float a, float b) { return a + b; });
}
template <int OFF>
__device__ __forceinline__ float apart_max(float v) {
  return lanes_apart<OFF>(v, [](float a, float b) { return fmaxf(a, b); });
}
// all N lanes of a group (N a power of two up to 64, all of the wave's lanes active) get f over
// the group, paired off as lane l with l xor N / 2, then N / 4, .. 1
template <int N, typename F>
__device__ __forceinline__ float lanes_reduce(float v, F f) {
  if constexpr (N >= 64) v = lanes_apart<32>(v, f);
  if constexpr (N >= 32) v = lanes_apart<16>(v, f);
  if constexpr (N >= 16) v = f(v, lane_xor<8>(v));
  // (behind a step of 8 lane l xor 12 holds what lane l xor 4 does: row_ror 4 is one move)
  if constexpr (N >= 16) v = f(v, lane_move<0x124>(v, v));
  else if constexpr (N >= 8) v = f(v, lane_xor<4>(v));
  if constexpr (N >= 4) v = f(v, lane_xor<2>(v));
  if constexpr (N >= 2) v = f(v, lane_xor<1>(v));
  return v;
}
template <int N>
__device__ __forceinline__ float lanes_sum(float v) {
  return lanes_reduce<N>(v, [](float a, float b) { return a + b; });
}
// Every number of v summed over n neighbouring lanes (a power of two up to 64, the same in the
// whole wave), paired off the other way: lane l with l xor 1, then 2, .. n / 2.  The lanes of a
// quad hold the same sum by the time the quads meet, so the mirrors of eight and sixteen lanes do
// for l xor 4 and 8.
template <int N>
__device__ __forceinline__ void lanes_sum_up(float (&v)[N], int n) {
  auto each = [&](auto f) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = f(v[i]);
  };
  // (Left as early as a group is done: with a branch for every step that is not taken, walks over
  // tokens that add up few lanes took longer: 32 heads of 16 x 64, 64 tokens 49.6 us for 43.8.)
  if (n <= 1) return;
  each([](float x) { return x + lane_xor<1>(x); });
  if (n <= 2) return;
  each([](float x) { return x + lane_xor<2>(x); });
  if (n <= 4) return;
  each([](float x) { return x + lane_move<0x141>(x, x); });      // row_half_mirror
  if (n <= 8) return;
  each([](float x) { return x + lane_move<0x140>(x, x); });      // row_mirror
  if (n <= 16) return;
  each([](float x) { return apart_sum<16>(x); });
  if (n <= 32) return;
  each([](float x) { return apart_sum<32>(x); });
}
// lanes_sum for a number of lanes that is known when the kernel runs
__device__ __forceinline__ float lanes_sum_down(float v, int n) {
  if (n > 32) v = apart_sum<32>(v);
  if (n > 16) v = apart_sum<16>(v);
  if (n > 8) v += lane_xor<8>(v);
  if (n > 4) v += lane_xor<4>(v);
  if (n > 2) v += lane_xor<2>(v);
  if (n > 1) v += lane_xor<1>(v);
  return v;
}
__device__ __forceinline__ float wave_sum(float v) { return lanes_sum<ZF_WAVE>(v); }
__device__ __forceinline__ float wave_max(float v) {
  return lanes_reduce<ZF_WAVE>(v, [](float a, float b) { return fmaxf(a, b); });
}

// RMSNorm over a head and rotation of its pairs (i, i + hd / 2) for the 8 elements a lane
// holds: x0 = elements 4 li .. 4 li + 3 of the head, x1 = those hd / 2 further on; LPH lanes
// side by side hold the head (src/kernel/norm/basic.zig:5-22 and src/kernel/rope/basic.zig:5-30
// of the reference: x / sqrt(mean(x^2) + eps) * gain, then (x0 c - x1 s, x1 c + x0 s) with the
// angle of (position, pair)).  Every lane of the LPH calls it (the sum goes over all of them);
// a lane that is not `active` holds zeros and keeps them.  The gains and the angles' cosines
// and sines of the lane's elements are loaded apart (a null table: none), so that a kernel
// can ask for them early.  One function for the kernel that writes the cache and for the
// decode attention that does the same work itself, so that both round alike.
struct HeadCoef {
  float g0[4], g1[4], c[4], sn[4];
  bool has_gain, has_rotation;
};
__device__ __forceinline__ void load_head_coef(HeadCoef& cf, int li, int hd,
                                               const float* __restrict__ gain,
                                               const float* __restrict__ cos_t,
                                               const float* __restrict__ sin_t, int pos) {
  // hd % 8 == 0 and 4 li < hd / 2: each group of four is one 16-byte load (as four 4-byte
  // loads they were two thirds of the load instructions of the kernels that call this)
  const int half = hd / 2;
  cf.has_gain = gain != nullptr;
  cf.has_rotation = cos_t != nullptr;
  float4 g0 = float4{1.f, 1.f, 1.f, 1.f}, g1 = g0, c = g0, sn = float4{0.f, 0.f, 0.f, 0.f};
  if (cf.has_gain) {
    g0 = *(const float4*)(gain + 4 * li);
    g1 = *(const float4*)(gain + half + 4 * li);
  }
  if (cf.has_rotation) {
    c = *(const float4*)(cos_t + (size_t)pos * half + 4 * li);
    sn = *(const float4*)(sin_t + (size_t)pos * half + 4 * li);
  }
  cf.g0[0] = g0.x; cf.g0[1] = g0.y; cf.g0[2] = g0.z; cf.g0[3] = g0.w;
  cf.g1[0] = g1.x; cf.g1[1] = g1.y; cf.g1[2] = g1.z; cf.g1[3] = g1.w;
  cf.c[0] = c.x; cf.c[1] = c.y; cf.c[2] = c.z; cf.c[3] = c.w;
  cf.sn[0] = sn.x; cf.sn[1] = sn.y; cf.sn[2] = sn.z; cf.sn[3] = sn.w;
}
// the same head at another position: the gains stay, cosines and sines are loaded anew
__device__ __forceinline__ void load_head_rotation(HeadCoef& cf, int li, int hd,
                                                   const float* __restrict__ cos_t,
                                                   const float* __restrict__ sin_t, int pos) {
  if (!cf.has_rotation) return;
  const int half = hd / 2;
  const float4 c = *(const float4*)(cos_t + (size_t)pos * half + 4 * li);
  const float4 sn = *(const float4*)(sin_t + (size_t)pos * half + 4 * li);
  cf.c[0] = c.x; cf.c[1] = c.y; cf.c[2] = c.z; cf.c[3] = c.w;
  cf.sn[0] = sn.x; cf.sn[1] = sn.y; cf.sn[2] = sn.z; cf.sn[3] = sn.w;
}
template <int LPH>
__device__ __forceinline__ void head_norm_rotate(float (&x0)[4], float (&x1)[4], int hd,
                                                 bool active, float eps, const HeadCoef& cf) {
  // every product and sum below is rounded on its own: fused multiply-adds, formed or not as
  // the code around a call happens to be scheduled, would let two kernels that call this
  // disagree in the last bit
#pragma clang fp contract(off)
  if (cf.has_gain) {
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) ss += x0[e] * x0[e] + x1[e] * x1[e];
    ss = lanes_sum<LPH>(ss);
    const float inv = 1.0f / sqrtf(ss / (float)hd + eps);
    if (active) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x0[e] = x0[e] * inv * cf.g0[e];
        x1[e] = x1[e] * inv * cf.g1[e];
      }
    }
  }
  if (active && cf.has_rotation) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float r0 = x0[e] * cf.c[e] - x1[e] * cf.sn[e];
      const float r1 = x1[e] * cf.c[e] + x0[e] * cf.sn[e];
      x0[e] = r0;
      x1[e] = r1;
    }
  }
}

// Sum over a block of up to 1024 threads; every thread gets the result.  `red` is LDS for
// at least 16 floats.  The order of the additions depends only on the block size.
__device__ __forceinline__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  const int wave = threadIdx.x / ZF_WAVE, lane = threadIdx.x % ZF_WAVE;
  const int nwaves = (blockDim.x + ZF_WAVE - 1) / ZF_WAVE;
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  // (four reads in flight at a time; a wave that is not there repeats the last one's)
  float total = 0.f;
  for (int w0 = 0; w0 < nwaves; w0 += 4) {
    float p[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) p[w] = red[min(w0 + w, nwaves - 1)];
#pragma unroll
    for (int w = 0; w < 4; ++w)
      if (w0 + w < nwaves) total += p[w];
  }
  return total;
}

// An activation alone, by number (32-bit arithmetic): 0 gelu(z) = z/2 (1 + erf(z / sqrt 2)),
// 1 its tanh form, 2 silu(z) = z / (1 + exp(-z)), 3 max(z, 0)^2, 4 tanh(z).
__device__ __forceinline__ float activation_value(float z, int kind) {
  if (kind == 0) return 0.5f * z * (1.0f + erff(z * 0.70710678118654752440f));
  if (kind == 1)
    return 0.5f * z * (1.0f + tanhf(0.79788456080286535588f * (z + 0.044715f * z * z * z)));
  if (kind == 3) { const float r = fmaxf(z, 0.f); return r * r; }
  if (kind == 4) return tanhf(z);
  return z / (1.0f + expf(-z));
}

// dtype codes shared with the Python side
#define ZF_F32 0
#define ZF_BF16 1

#define ZF_CHECK_LAUNCH() return (int)hipGetLastError()
