// The gated delta rule: a matrix S [d, dv] a head that every token decays and then corrects
// towards its own value,
//
//   S <- g_t S;   w = beta_t (v_t - S^T k_t);   S <- S + k_t w^T;   o_t = S^T q_t
//
// with one decay g_t = exp(-exp(A) softplus(z_a + dt)) and one step size beta_t = sigmoid(z_b) a
// head and token, and the short convolutions that feed it.  All arithmetic is 32-bit.
//
//  * short_conv        rows of a projection -> silu(causal convolution over time a channel, plus a
//                      bias); the leading channels are heads that are made unit vectors (and the
//                      first of those multiplied by a scale).  The taps - 1 rows before a step come
//                      from the request's state.
//  * short_conv_state  the state takes the step's last taps - 1 rows.
//  * delta_recurrence  the recurrence over the rows of a step, sequence by sequence.
//  * delta_chunk_*     the same for long portions, sixteen tokens at a time as 32-bit matrix products.
//
// With r = S^T k and p = S^T q of the matrix *before* the token (both formed in one pass over
// it), w = beta (v - g r), o = g p + (q . k) w and S <- g S + k w^T: the same numbers as the
// four lines above with one pass over S less.
#include "zf_common.h"

#include <type_traits>

__device__ __forceinline__ float dl_silu(float z) { return z / (1.0f + expf(-z)); }
// silu of what leaves in TO (for bfloat16 through the bare exponential and reciprocal)
template <typename TO> __device__ __forceinline__ float dl_silu_to(float z) {
  if constexpr (sizeof(TO) == 2)
    return z * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
  return dl_silu(z);
}
#define DL_STEP_TAPS 8          // most taps of a decode step in one kernel
__device__ __forceinline__ float dl_softplus(float z) {
  return z > 20.f ? z : log1pf(expf(z));
}

// The sum over the CG lanes (a power of two up to 64, aligned) that share a
// column, in every one of them, through the data-parallel lane moves: neighbours, pairs, then the
// mirrored half row and row (a lane and its mirror hold sums over different halves).
template <int CTRL>
__device__ __forceinline__ float dl_move(float v) {
  // (every lane has a source lane: the value a lane without one would keep is never used)
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(v), __float_as_int(v), CTRL,
                                                    0xf, 0xf, true));
}
template <int CG>
__device__ __forceinline__ float dl_lanes_sum(float v) {
  if constexpr (CG >= 2) v += dl_move<0xB1>(v);      // quad_perm [1, 0, 3, 2]
  if constexpr (CG >= 4) v += dl_move<0x4E>(v);      // quad_perm [2, 3, 0, 1]
  if constexpr (CG >= 8) v += dl_move<0x141>(v);     // row_half_mirror
  if constexpr (CG >= 16) v += dl_move<0x140>(v);    // row_mirror
  if constexpr (CG >= 32) {
    // rows of 16 lanes in pairs: one copy takes its odd rows from the other's even rows and
    // gives its own odd rows for them, so the two copies hold a pair's two rows lane by lane
    typedef unsigned int dl_u2 __attribute__((ext_vector_type(2)));
    const dl_u2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r.x) + __uint_as_float(r.y);
    if constexpr (CG >= 64) {
      const dl_u2 q = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
      v = __uint_as_float(q.x) + __uint_as_float(q.y);      // the wave's two halves
    }
  }
  return v;
}

// ------------------------------------------------------------------ short convolutions
// src [T, >= C] (row stride given), taps [C, n] float32 (the last column is the token's own), bias
// float32 [C] or null, out [T, C] in float32 or bfloat16.  Channels [0, unit_heads * hd) are heads of hd that leave as unit vectors
// x / sqrt(sum x^2 + unit_eps), the first scaled_heads of them times `scale`.  State of a
// request: [n - 1, C] floats at state + slot * state_stride + state_off, oldest row first.
// Grid (token, block of channels): the first head_blocks blocks hold hpb whole heads each, a
// head in one, two or four whole waves and a thread a channel (a head wider than the workgroup:
// a thread several channels), the others DL_CONV_THREADS plain channels.  A head's sum of
// squares is added up over a wave's lanes and then over the head's waves in their order.
// update_state (only when every sequence of the step brings one token: a thread is then the
// only reader of its channel's kept rows): the state is moved on by this kernel.
#define DL_CONV_THREADS 256
#define DL_CONV_MAX_TAPS 8
#define DL_CONV_ROWS_AHEAD 8     // tokens whose rows a thread of the rows' form asks for at once
#define DL_CONV_PER_THREAD 4     // channels a thread takes of a head wider than the workgroup

template <typename T, typename TO>
__global__ __launch_bounds__(DL_CONV_THREADS) void short_conv_kernel(
    const T* __restrict__ src, long long src_stride, const float* __restrict__ taps, int n_taps,
    const float* __restrict__ bias, float* __restrict__ state, long long state_stride,
    long long state_off, const int* __restrict__ state_slots, const int* __restrict__ seq_index,
    const int* __restrict__ q_start, TO* __restrict__ out, int C, int unit_heads, int hd,
    int scaled_heads, float scale, float unit_eps, int update_state, int head_blocks, int hpb) {
#pragma clang fp contract(off)
  __shared__ float sq[DL_CONV_THREADS / ZF_WAVE];
  const int t = blockIdx.x;
  const int s = seq_index[t];
  const int i0 = t - q_start[s];                       // the token's place in its portion
  float* st = state + (size_t)state_slots[s] * state_stride + state_off;
  const int hist = n_taps - 1;
  auto conv = [&](int c) -> float {
    float x[DL_CONV_MAX_TAPS];
#pragma unroll
    for (int j = 0; j < DL_CONV_MAX_TAPS; ++j) {
      x[j] = 0.f;
      if (j < n_taps) {
        const int back = hist - j;                     // rows before the token's own
        if (back <= i0) x[j] = load_as_float<T>(src + (size_t)(t - back) * src_stride + c);
        else x[j] = st[(size_t)(hist + i0 - back) * C + c];
      }
    }
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < DL_CONV_MAX_TAPS; ++j)
      if (j < n_taps) acc = acc + taps[(size_t)c * n_taps + j] * x[j];
    if (update_state) {
      // the kept rows move on by one: rows 1 .. of what was read, then the token's own
#pragma unroll
      for (int j = 1; j < DL_CONV_MAX_TAPS; ++j)
        if (j < n_taps) st[(size_t)(j - 1) * C + c] = x[j];
    }
    return dl_silu_to<TO>(bias != nullptr ? acc + bias[c] : acc);
  };
  TO* o = out + (size_t)t * C;
  const int b = blockIdx.y;
  if (b >= head_blocks) {
    const int c = unit_heads * hd + (b - head_blocks) * DL_CONV_THREADS + threadIdx.x;
    if (c < C) store_from_float<TO>(o + c, conv(c));
    return;
  }
  // a head takes tph threads, whole waves of them (hpb heads a block), a thread `per` channels
  const int tph = DL_CONV_THREADS / hpb;
  const int per = (hd + tph - 1) / tph;
  const int head = b * hpb + threadIdx.x / tph;
  const int d0 = threadIdx.x % tph;
  const bool mine = head < unit_heads;
  float v[DL_CONV_PER_THREAD];
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < DL_CONV_PER_THREAD; ++j) {
    v[j] = 0.f;
    const int dd = d0 + j * tph;
    if (j < per && mine && dd < hd) v[j] = conv(head * hd + dd);
    ss += v[j] * v[j];
  }
  // over the lanes of a wave, then over the head's waves in their order
  ss = dl_lanes_sum<16>(ss);
  ss = apart_sum<16>(ss);
  ss = apart_sum<32>(ss);
  const int wave = threadIdx.x / ZF_WAVE, wph = tph / ZF_WAVE;
  if (threadIdx.x % ZF_WAVE == 0) sq[wave] = ss;
  __syncthreads();
  if (!mine) return;
  float total = 0.f;
  for (int w = 0; w < wph; ++w) total += sq[(wave / wph) * wph + w];
  float inv = 1.0f / sqrtf(total + unit_eps);
  if (head < scaled_heads) inv = inv * scale;
#pragma unroll
  for (int j = 0; j < DL_CONV_PER_THREAD; ++j) {
    const int dd = d0 + j * tph;
    if (j < per && dd < hd) store_from_float<TO>(o + head * hd + dd, v[j] * inv);
  }
}

// The same in rows of pieces: a thread takes V neighbouring channels (16 bytes of a row) of TT tokens
// one behind the other and keeps the rows before the token in registers, NT of them with the
// token's own (n_taps <= NT; the rows further back meet taps of zero).  The same products and
// sums in the same order as above.  A head that leaves as a unit vector is lph lanes side by side
// (hd = lph * V, lph a power of two up to 64; a workgroup is one wave, so heads never straddle
// one): its squares are added over a thread's channels and then over the lanes, whatever the
// portion.  With a thread a channel that read every row once a tap, 2048 tokens of 4096 channels,
// half of them in heads of 128, took 87 us, so 25; a decode step's eight tokens 5.3 and 4.8.
// Grid (blocks of TT tokens, blocks of channels).
template <typename T, typename TO, int V, int NT, bool UNIT>
__global__ __launch_bounds__(DL_CONV_THREADS) void short_conv_rows_kernel(
    const T* __restrict__ src, long long src_stride, const float* __restrict__ taps, int n_taps,
    const float* __restrict__ bias, float* __restrict__ state, long long state_stride,
    long long state_off, const int* __restrict__ state_slots, const int* __restrict__ seq_index,
    const int* __restrict__ q_start, TO* __restrict__ out, int n_tokens, int C, int TT,
    int update_state, int unit_heads, int lph, int scaled_heads, float scale, float unit_eps) {
#pragma clang fp contract(off)
  const int c = (blockIdx.y * blockDim.x + threadIdx.x) * V;
  if (c >= C) return;
  const int hist = n_taps - 1;
  float tp[NT][V], b[V], w[NT][V];
  if (n_taps == NT) {
    float flat[V * NT];
#pragma unroll
    for (int i = 0; i < V * NT; i += 4) {
      const float4 f = *(const float4*)(taps + (size_t)c * NT + i);
      flat[i] = f.x; flat[i + 1] = f.y; flat[i + 2] = f.z; flat[i + 3] = f.w;
    }
#pragma unroll
    for (int k = 0; k < NT; ++k)
#pragma unroll
      for (int v = 0; v < V; ++v) tp[k][v] = flat[v * NT + k];
  } else {
#pragma unroll
    for (int k = 0; k < NT; ++k)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const int j = k - (NT - n_taps);
        tp[k][v] = j >= 0 ? taps[(size_t)(c + v) * n_taps + j] : 0.f;
      }
  }
#pragma unroll
  for (int v = 0; v < V; v += 4) {
    float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
    if (bias != nullptr) f = *(const float4*)(bias + c + v);
    b[v] = f.x; b[v + 1] = f.y; b[v + 2] = f.z; b[v + 3] = f.w;
  }
  typedef typename std::conditional<sizeof(T) == 2, uint4, float4>::type raw_t;      // V channels
  auto raw_row = [&](int t) { return *(const raw_t*)(src + (size_t)t * src_stride + c); };
  auto open_row = [&](const raw_t& r, float (&x)[V]) {
    if constexpr (sizeof(T) == 2) {
      const uint32_t u[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        x[2 * i] = __uint_as_float(u[i] << 16);
        x[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
      }
    } else {
      x[0] = r.x; x[1] = r.y; x[2] = r.z; x[3] = r.w;
    }
  };
  // the rows before token t: of its portion, or of the request's state
  auto rows_before = [&](int t, int s, const float* st) {
    const int i0 = t - q_start[s];
#pragma unroll
    for (int k = 0; k < NT - 1; ++k) {
      const int back = NT - 1 - k;
#pragma unroll
      for (int v = 0; v < V; ++v) w[k][v] = 0.f;
      if (back <= hist) {
        if (back <= i0) {
          open_row(raw_row(t - back), w[k]);
        } else {
#pragma unroll
          for (int v = 0; v < V; v += 4) {
            const float4 f = *(const float4*)(st + (size_t)(hist + i0 - back) * C + c + v);
            w[k][v] = f.x; w[k][v + 1] = f.y; w[k][v + 2] = f.z; w[k][v + 3] = f.w;
          }
        }
      }
    }
  };
  auto emit = [&](int t) {
    float acc[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
      acc[v] = 0.f;
#pragma unroll
      for (int k = 0; k < NT; ++k) acc[v] = acc[v] + tp[k][v] * w[k][v];
      acc[v] = dl_silu_to<TO>(bias != nullptr ? acc[v] + b[v] : acc[v]);
    }
    if (UNIT && c < unit_heads * lph * V) {
      float ss = 0.f;
#pragma unroll
      for (int v = 0; v < V; ++v) ss += acc[v] * acc[v];
      ss = lanes_sum_down(ss, lph);
      float inv = 1.0f / sqrtf(ss + unit_eps);
      if (c < scaled_heads * lph * V) inv = inv * scale;
#pragma unroll
      for (int v = 0; v < V; ++v) acc[v] = acc[v] * inv;
    }
    TO* o = out + (size_t)t * C + c;
    if constexpr (sizeof(TO) == 2) {
      *(uint4*)o = make_uint4(pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]),
                              pack_bf16x2(acc[4], acc[5]), pack_bf16x2(acc[6], acc[7]));
    } else {
#pragma unroll
      for (int v = 0; v < V; v += 4)
        *(float4*)(o + v) = make_float4(acc[v], acc[v + 1], acc[v + 2], acc[v + 3]);
    }
  };
  auto move_on = [&]() {
#pragma unroll
    for (int k = 0; k + 1 < NT; ++k)
#pragma unroll
      for (int v = 0; v < V; ++v) w[k][v] = w[k + 1][v];
  };
  const int first = blockIdx.x * TT, last = min(n_tokens, first + TT);
  const int s0 = seq_index[first];
  if (TT == DL_CONV_ROWS_AHEAD && last - first == TT && seq_index[last - 1] == s0) {
    // tokens of one sequence: their rows are asked for all at once
    raw_t raw[DL_CONV_ROWS_AHEAD];
#pragma unroll
    for (int u = 0; u < DL_CONV_ROWS_AHEAD; ++u) raw[u] = raw_row(first + u);
    rows_before(first, s0, state + (size_t)state_slots[s0] * state_stride + state_off);
#pragma unroll
    for (int u = 0; u < DL_CONV_ROWS_AHEAD; ++u) {
      open_row(raw[u], w[NT - 1]);
      emit(first + u);
      move_on();
    }
    return;
  }
  int seq = -1;
  for (int t = first; t < last; ++t) {
    const int s = seq_index[t];
    float* st = state + (size_t)state_slots[s] * state_stride + state_off;
    if (s != seq) rows_before(t, s, st);
    seq = s;
    open_row(raw_row(t), w[NT - 1]);
    emit(t);
    if (update_state) {
      // the kept rows move on by one: the last n_taps - 1 rows of the window
#pragma unroll
      for (int k = 1; k < NT; ++k)
        if (k >= NT - hist) {
#pragma unroll
          for (int v = 0; v < V; v += 4)
            *(float4*)(st + (size_t)(k - (NT - hist)) * C + c + v) =
                make_float4(w[k][v], w[k][v + 1], w[k][v + 2], w[k][v + 3]);
        }
    }
    move_on();
  }
}

// The state after a step: the last n - 1 rows the convolution has seen.  Grid (sequence, block of
// channels), a thread a channel.
template <typename T>
__global__ __launch_bounds__(DL_CONV_THREADS) void short_conv_state_kernel(
    const T* __restrict__ src, long long src_stride, int n_taps, float* __restrict__ state,
    long long state_stride, long long state_off, const int* __restrict__ state_slots,
    const int* __restrict__ q_start, int C) {
  const int s = blockIdx.x;
  const int first = q_start[s], len = q_start[s + 1] - first;
  const int c = blockIdx.y * DL_CONV_THREADS + threadIdx.x;
  if (len <= 0 || c >= C) return;
  float* st = state + (size_t)state_slots[s] * state_stride + state_off;
  const int hist = n_taps - 1;
  // row r of the new state is the portion's row len - hist + r, or (before the portion) the
  // old state's row r + len, which lies behind the row being written: ascending r is safe
  for (int r = 0; r < hist; ++r) {
    const int i = len - hist + r;
    st[(size_t)r * C + c] = i >= 0 ? load_as_float<T>(src + (size_t)(first + i) * src_stride + c)
                                   : st[(size_t)(r + len) * C + c];
  }
}

extern "C" int zf_short_conv(const void* src, int dtype, long long src_stride, const float* taps,
                             int n_taps, const float* bias, float* state, long long state_stride,
                             long long state_off, const int* state_slots, const int* seq_index,
                             const int* q_start, void* out, int out_dtype, int T, int n_seqs, int C,
                             int unit_heads, int hd, int scaled_heads, float scale,
                             float unit_eps, int single_tokens, hipStream_t stream) {
  if (T <= 0) return 0;
  if (C <= 0 || n_taps < 1 || n_taps > DL_CONV_MAX_TAPS || unit_heads < 0 || hd < 1 ||
      (size_t)unit_heads * hd > (size_t)C || scaled_heads > unit_heads || n_seqs < 1 ||
      (single_tokens && T != n_seqs) || hd > DL_CONV_THREADS * DL_CONV_PER_THREAD ||
      (dtype == ZF_F32 && out_dtype != ZF_F32))
    return -2;
  // a head takes whole waves (one, two or four): as many heads a block as fit
  const int hw = hd > 128 ? 4 : (hd > 64 ? 2 : 1);
  const int hpb = DL_CONV_THREADS / (hw * ZF_WAVE);
  const int head_blocks = (unit_heads + hpb - 1) / hpb;
  const int plain = C - unit_heads * hd;
  const dim3 grid(T, head_blocks + (plain + DL_CONV_THREADS - 1) / DL_CONV_THREADS);
  const dim3 sgrid(n_seqs, (C + DL_CONV_THREADS - 1) / DL_CONV_THREADS);
  const int V = dtype == ZF_F32 ? 4 : 8;
  // heads of V, 2 V, .. 64 V channels: whole lanes of a wave
  const int lph = unit_heads > 0 && hd % V == 0 ? hd / V : 0;
  const bool rows = (unit_heads == 0 || (lph > 0 && lph <= ZF_WAVE && (lph & (lph - 1)) == 0)) &&
                    C % V == 0 && src_stride % V == 0 && state_stride % 4 == 0 &&
                    state_off % 4 == 0 && (uintptr_t)src % 16 == 0 && (uintptr_t)out % 16 == 0 &&
                    (uintptr_t)taps % 16 == 0 && (uintptr_t)bias % 16 == 0 &&
                    (uintptr_t)state % 16 == 0;
  const int threads = 64;
  // (a wave across all channels leaves most of the chip idle, and a head's sum over its lanes is one
  // more chain a token: 512 tokens of 64 channels four a workgroup 6.9 us, two 5.6, through the other
  // kernel 6.1; 1024 tokens eight a workgroup 8.7 us, through the other kernel 7.3)
  const int TT = single_tokens ? 1
                 : unit_heads > 0 && C <= 64 * V && T < 2048 ? 2
                 : T >= 1024 ? 8 : T >= 256 ? 4 : 2;
  const dim3 rgrid((T + TT - 1) / TT, (C / V + threads - 1) / threads);
#define DL_CONV_ROWS(TT_, TO_, V_, N_)                                                            \
  if (unit_heads > 0) DL_CONV_ROWS_OF(TT_, TO_, V_, N_, true);                                   \
  else DL_CONV_ROWS_OF(TT_, TO_, V_, N_, false)
#define DL_CONV_ROWS_OF(TT_, TO_, V_, N_, U_)                                                     \
  hipLaunchKernelGGL((short_conv_rows_kernel<TT_, TO_, V_, N_, U_>), rgrid, dim3(threads), 0, stream,\
                     (const TT_*)src, src_stride, taps, n_taps, bias, state, state_stride,       \
                     state_off, state_slots, seq_index, q_start, (TO_*)out, T, C, TT, single_tokens, \
                     unit_heads, lph, scaled_heads, scale, unit_eps)
#define DL_CONV_LAUNCH(TT_, TO_, V_)                                                              \
  if (rows) {                                                                                    \
    if (n_taps <= 4) { DL_CONV_ROWS(TT_, TO_, V_, 4); }                                          \
    else { DL_CONV_ROWS(TT_, TO_, V_, 8); }                                                      \
  } else {                                                                                       \
    hipLaunchKernelGGL((short_conv_kernel<TT_, TO_>), grid, dim3(DL_CONV_THREADS), 0, stream,    \
                       (const TT_*)src, src_stride, taps, n_taps, bias, state, state_stride,     \
                       state_off, state_slots, seq_index, q_start, (TO_*)out, C, unit_heads, hd, \
                       scaled_heads, scale, unit_eps, single_tokens, head_blocks, hpb);          \
  }                                                                                              \
  if (!single_tokens && n_taps > 1)                                                              \
    hipLaunchKernelGGL(short_conv_state_kernel<TT_>, sgrid, dim3(DL_CONV_THREADS), 0, stream,    \
                       (const TT_*)src, src_stride, n_taps, state, state_stride, state_off,      \
                       state_slots, q_start, C)
  if (dtype == ZF_F32) { DL_CONV_LAUNCH(float, float, 4); }
  else if (out_dtype == ZF_F32) { DL_CONV_LAUNCH(bf16_t, float, 8); }
  else { DL_CONV_LAUNCH(bf16_t, bf16_t, 8); }
  ZF_CHECK_LAUNCH();
}

// ------------------------------------------------------------------ the recurrence
#define DL_STAGE 16            // tokens staged in LDS at a time
#define DL_MAX_LANES 64        // lanes that share a column's key channels
#define DL_PF 4                // 16-byte pieces of q and of k, and values of v, a thread fetches ahead

// A thread holds R key channels of one value column of S; CG lanes side by side hold the
// column's P = CG * R channels (zeros beyond d).  A request's matrices lie [head][column][P] in
// its state, so a thread's channels are consecutive.  Grid (column tiles, heads, sequences).
// qkv float32 [T, C]: q heads at q_off, k heads at k_off (KH heads of d each), v heads at v_off
// (H heads of dv); ab float32 [T, 2 H]: the decays' numbers z_a, then the step sizes' z_b.
// Sixteen tokens at a time lie in LDS; the next sixteen are asked for before these are walked
// (16-byte pieces, where the rows' offsets allow: VEC), and a token's operands are read from LDS
// while the token before it is computed.
template <int R, int CG, bool VEC>
__global__ __launch_bounds__(256) void delta_recurrence_kernel(
    const float* __restrict__ qkv, int C, int q_off, int k_off, int v_off,
    const float* __restrict__ ab, const float* __restrict__ a_log,
    const float* __restrict__ dt_bias, float* __restrict__ state, long long state_stride,
    const int* __restrict__ state_slots, const int* __restrict__ q_start, float* __restrict__ out,
    int H, int KH, int d, int dv, int cols, int longest) {
  // (fused multiply-adds as the compiler forms them: this one kernel walks every portion up to
  // `longest` tokens, so every cut of a sequence into such gets the same instructions)
  extern __shared__ float lds[];
  const int P = CG * R;
  float* qs = lds;                          // [DL_STAGE][P]
  float* ks = qs + DL_STAGE * P;            // [DL_STAGE][P]
  float* vs = ks + DL_STAGE * P;            // [DL_STAGE][cols]
  float* gs = vs + DL_STAGE * cols;         // [DL_STAGE] decay
  float* bs = gs + DL_STAGE;                // [DL_STAGE] step size
  float* ds = bs + DL_STAGE;                // [DL_STAGE] q . k
  float* os = ds + DL_STAGE;                // [DL_STAGE][cols] the stage's outputs
  const int h = blockIdx.y, seq = blockIdx.z;
  const int kh = h / (H / KH);
  const int first = q_start[seq], len = q_start[seq + 1] - first;
  if (len <= 0 || len > longest) return;
  const int tid = threadIdx.x, nthreads = blockDim.x;
  const int cg = tid % CG, col_l = tid / CG;
  const int col = blockIdx.x * cols + col_l;
  const bool live = col < dv;
  float* S_mem = state + (size_t)state_slots[seq] * state_stride
                 + ((size_t)h * dv + (live ? col : 0)) * P + cg * R;
  float S[R];
  if constexpr (R % 4 == 0) {
#pragma unroll
    for (int r = 0; r < R; r += 4) {
      const float4 v = live ? *(const float4*)(S_mem + r) : make_float4(0.f, 0.f, 0.f, 0.f);
      S[r] = v.x; S[r + 1] = v.y; S[r + 2] = v.z; S[r + 3] = v.w;
    }
  } else {
#pragma unroll
    for (int r = 0; r < R; r += 2) {
      const float2 v = live ? *(const float2*)(S_mem + r) : make_float2(0.f, 0.f);
      S[r] = v.x; S[r + 1] = v.y;
    }
  }
  const float decay_rate = expf(a_log[h]);
  const float dtb = dt_bias[h];
  const int P4 = P / 4;
  // what a thread fetches ahead: pieces tid, tid + nthreads, ... of the stage's q and k rows,
  // one value of its v columns, and (the first threads) a token's two numbers
  float4 fq[DL_PF], fk[DL_PF];
  float fv[DL_PF], fa = 0.f, fb = 0.f;
  const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
  auto fetch = [&](int t0, int n) {
    if constexpr (VEC) {
#pragma unroll
      for (int j = 0; j < DL_PF; ++j) {
        const int i = tid + j * nthreads;
        fq[j] = fk[j] = zero4;
        if (i < n * P4) {
          const int tok = i / P4, c = (i % P4) * 4;
          const float* row = qkv + (size_t)(first + t0 + tok) * C;
          if (c < d) {
            fq[j] = *(const float4*)(row + q_off + kh * d + c);
            fk[j] = *(const float4*)(row + k_off + kh * d + c);
          }
        }
      }
#pragma unroll
      for (int j = 0; j < DL_PF; ++j) {
        const int i = tid + j * nthreads;
        fv[j] = 0.f;
        if (i < n * cols) {
          const int tok = i / cols, c = blockIdx.x * cols + i % cols;
          if (c < dv) fv[j] = qkv[(size_t)(first + t0 + tok) * C + v_off + h * dv + c];
        }
      }
      if (tid < n) {
        const float* z = ab + (size_t)(first + t0 + tid) * 2 * H;
        fa = z[h];
        fb = z[H + h];
      }
    }
  };
  auto stage = [&](int t0, int n) {
    if constexpr (VEC) {
#pragma unroll
      for (int j = 0; j < DL_PF; ++j) {
        const int i = tid + j * nthreads;
        if (i < n * P4) {
          *(float4*)(qs + 4 * i) = fq[j];
          *(float4*)(ks + 4 * i) = fk[j];
        }
      }
#pragma unroll
      for (int j = 0; j < DL_PF; ++j)
        if (tid + j * nthreads < n * cols) vs[tid + j * nthreads] = fv[j];
      if (tid < n) {
        gs[tid] = expf(-(decay_rate * dl_softplus(fa + dtb)));
        bs[tid] = 1.0f / (1.0f + expf(-fb));
      }
    } else {
      for (int i = tid; i < n * P; i += nthreads) {
        const int tok = i / P, c = i % P;
        const float* row = qkv + (size_t)(first + t0 + tok) * C;
        qs[i] = c < d ? row[q_off + kh * d + c] : 0.f;
        ks[i] = c < d ? row[k_off + kh * d + c] : 0.f;
      }
      for (int i = tid; i < n * cols; i += nthreads) {
        const int tok = i / cols, c = blockIdx.x * cols + i % cols;
        vs[i] = c < dv ? qkv[(size_t)(first + t0 + tok) * C + v_off + h * dv + c] : 0.f;
      }
      if (tid < n) {
        const float* z = ab + (size_t)(first + t0 + tid) * 2 * H;
        gs[tid] = expf(-(decay_rate * dl_softplus(z[h] + dtb)));
        bs[tid] = 1.0f / (1.0f + expf(-z[H + h]));
      }
    }
  };
  fetch(0, min(DL_STAGE, len));
  for (int t0 = 0; t0 < len; t0 += DL_STAGE) {
    const int n = min(DL_STAGE, len - t0);
    __syncthreads();                        // the tokens staged before are done with
    stage(t0, n);
    __syncthreads();
    if (t0 + DL_STAGE < len) fetch(t0 + DL_STAGE, min(DL_STAGE, len - t0 - DL_STAGE));
    // q . k of every staged token: sixteen lanes a token
    for (int tok = tid / 16; tok < n; tok += nthreads / 16) {
      float dot = 0.f;
      for (int c = tid % 16; c < P; c += 16) dot += qs[tok * P + c] * ks[tok * P + c];
      dot = dl_lanes_sum<16>(dot);
      if (tid % 16 == 0) ds[tok] = dot;
    }
    __syncthreads();
    // a token's operands are read a token ahead
    float kk[R], qq[R], g, b, v, qk;

    auto read = [&](int tok) {
      const float* qrow = qs + tok * P + cg * R;
      const float* krow = ks + tok * P + cg * R;
      if constexpr (R % 4 == 0) {
#pragma unroll
        for (int r = 0; r < R; r += 4) {
          const float4 kv = *(const float4*)(krow + r);
          const float4 qv = *(const float4*)(qrow + r);
          kk[r] = kv.x; kk[r + 1] = kv.y; kk[r + 2] = kv.z; kk[r + 3] = kv.w;
          qq[r] = qv.x; qq[r + 1] = qv.y; qq[r + 2] = qv.z; qq[r + 3] = qv.w;
        }
      } else {
#pragma unroll
        for (int r = 0; r < R; r += 2) {
          const float2 kv = *(const float2*)(krow + r);
          const float2 qv = *(const float2*)(qrow + r);
          kk[r] = kv.x; kk[r + 1] = kv.y;
          qq[r] = qv.x; qq[r + 1] = qv.y;
        }
      }
      g = gs[tok]; b = bs[tok]; v = vs[tok * cols + col_l]; qk = ds[tok];
    };
    read(0);
    for (int tok = 0; tok < n; ++tok) {
      float r0 = 0.f, r1 = 0.f, p0 = 0.f, p1 = 0.f;
      float kc[R];
#pragma unroll
      for (int r = 0; r < R; r += 2) {
        kc[r] = kk[r]; kc[r + 1] = kk[r + 1];
        r0 += kk[r] * S[r]; r1 += kk[r + 1] * S[r + 1];
        p0 += qq[r] * S[r]; p1 += qq[r + 1] * S[r + 1];
      }
      const float gc = g, bc = b, vc = v, qkc = qk;
      if (tok + 1 < n) read(tok + 1);
      const float rs = dl_lanes_sum<CG>(r0 + r1), ps = dl_lanes_sum<CG>(p0 + p1);
      const float w = bc * (vc - gc * rs);
#pragma unroll
      for (int r = 0; r < R; ++r) S[r] = gc * S[r] + kc[r] * w;
      if (cg == 0) os[tok * cols + col_l] = gc * ps + qkc * w;
    }
    // the stage's outputs leave side by side (the next stage's barrier stands between these
    // reads and the next writes)
    __syncthreads();
    for (int i = tid; i < n * cols; i += nthreads) {
      const int tok = i / cols, c = blockIdx.x * cols + i % cols;
      if (c < dv) out[(size_t)(first + t0 + tok) * H * dv + (size_t)h * dv + c] = os[i];
    }
  }
  if (live) {
    if constexpr (R % 4 == 0) {
#pragma unroll
      for (int r = 0; r < R; r += 4)
        *(float4*)(S_mem + r) = make_float4(S[r], S[r + 1], S[r + 2], S[r + 3]);
    } else {
#pragma unroll
      for (int r = 0; r < R; r += 2) *(float2*)(S_mem + r) = make_float2(S[r], S[r + 1]);
    }
  }
}

// R * CG >= d is the padded key size P the state is laid out with; cols * CG threads a workgroup
// (a multiple of 64, at most 256).  Sequences that bring more than `longest` tokens are left out.
extern "C" int zf_delta_recurrence(const float* qkv, int C, int q_off, int k_off, int v_off,
                                   const float* ab, const float* a_log, const float* dt_bias,
                                   float* state, long long state_stride, const int* state_slots,
                                   const int* q_start, float* out, int n_seqs, int H, int KH,
                                   int d, int dv, int R, int CG, int cols, int longest,
                                   hipStream_t stream) {
  if (n_seqs <= 0) return 0;
  const int threads = cols * CG;
  if (H < 1 || KH < 1 || H % KH != 0 || d < 1 || dv < 1 || CG < 1 || CG > DL_MAX_LANES ||
      (CG & (CG - 1)) != 0 || R * CG < d || cols < 1 || threads > 256 || threads % ZF_WAVE != 0 ||
      ZF_WAVE % CG != 0)
    return -2;
  const dim3 grid((dv + cols - 1) / cols, H, n_seqs), block(threads);
  const size_t smem = (size_t)(DL_STAGE * (2 * R * CG + 2 * cols) + 3 * DL_STAGE) * sizeof(float);
  // 16-byte pieces: every row offset a multiple of four floats, and few enough pieces a thread
  const bool vec = C % 4 == 0 && q_off % 4 == 0 && k_off % 4 == 0 && d % 4 == 0 &&
                   ((uintptr_t)qkv % 16) == 0 &&
                   DL_STAGE * (R * CG / 4) <= DL_PF * threads && DL_STAGE * cols <= DL_PF * threads &&
                   DL_STAGE <= threads;
#define DL_REC_LAUNCH(RR, GG)                                                                    \
  if (R == RR && CG == GG) {                                                                     \
    if (vec)                                                                                     \
      hipLaunchKernelGGL((delta_recurrence_kernel<RR, GG, true>), grid, block, smem, stream,     \
                         qkv, C, q_off, k_off, v_off, ab, a_log, dt_bias, state, state_stride,   \
                         state_slots, q_start, out, H, KH, d, dv, cols, longest);                         \
    else                                                                                         \
      hipLaunchKernelGGL((delta_recurrence_kernel<RR, GG, false>), grid, block, smem, stream,    \
                         qkv, C, q_off, k_off, v_off, ab, a_log, dt_bias, state, state_stride,   \
                         state_slots, q_start, out, H, KH, d, dv, cols, longest);                         \
    launched = true;                                                                             \
  }
  bool launched = false;
  // (the padded key sizes 8, 12, 16, 24, 32, 48, 64, 96, 128, 192, 256)
  DL_REC_LAUNCH(8, 1) DL_REC_LAUNCH(12, 1) DL_REC_LAUNCH(8, 2) DL_REC_LAUNCH(12, 2)
  DL_REC_LAUNCH(8, 4) DL_REC_LAUNCH(12, 4) DL_REC_LAUNCH(8, 8) DL_REC_LAUNCH(12, 8)
  DL_REC_LAUNCH(8, 16) DL_REC_LAUNCH(12, 16) DL_REC_LAUNCH(16, 16)
  if (!launched) return -2;
  ZF_CHECK_LAUNCH();
}

// ------------------------------------------------------------------ a decode step, whole
// One token a sequence (bfloat16 rows): a workgroup a (q/k head, sequence) runs the convolutions of its channels
// and moves their kept rows on, makes q and k unit vectors, walks the token for the value heads that share them,
// norms each of these and applies gain and gate.  As three kernels a layer of 8 tokens took 4.7 + 9.8 + 4.6 us for
// 16 heads of 128 x 128 on 8, each waiting for its first loads; here the matrices are asked for ahead of all else:
// 10.7 us; 1 to 64 sequences gain 1 to 7 % of a pass of four layers.  Thread (vl, cg) = (tid / CG, tid % CG) holds the channels 8 cg .. + 8 of RV neighbouring
// columns of the heads side by side; CG = d / 8.
struct DeltaStep {
  const bf16_t *src, *gate;
  const float *taps, *ab, *a_log, *dt_bias, *gain;
  float* state;
  const int* state_slots;
  bf16_t* out;
  long long src_stride, gate_stride, out_stride, state_stride, conv_at;
  int n_taps, H, KH, d, dv, CG;
  float scale, unit_eps, norm_eps;
};
template <int RV>
__global__ __launch_bounds__(1024) void delta_step_kernel(DeltaStep p) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  __shared__ float s_unit[3];               // 1 / |q| times the scale, 1 / |k|, q . k of the unit vectors
  const int d = p.d, dv = p.dv, HG = p.H / p.KH, N = HG * dv, C = 2 * p.KH * d + p.H * dv, CG = p.CG;
  float* qs = lds;                          // [d]
  float* ks = qs + d;
  float* vs = ks + d;                       // [N]
  float* os = vs + N;                       // [N]
  float* gs = os + N;                       // [HG] decay
  float* bs = gs + HG;                      // [HG] step size
  const int kh = blockIdx.x, s = blockIdx.y, tid = threadIdx.x, nt = blockDim.x;
  const int wave = tid / ZF_WAVE, lane = tid % ZF_WAVE, waves = nt / ZF_WAVE;
  float* slot = p.state + (size_t)p.state_slots[s] * p.state_stride;
  const int cg = tid % CG, col = tid / CG * RV;
  const bool live = col < N;                // (dv is a multiple of RV: a thread's columns are one head's)
  float* S_mem = slot + ((size_t)kh * N + (live ? col : 0)) * d + cg * 8;
  float S[RV][8];
#pragma unroll
  for (int r = 0; r < RV; ++r) {
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f), b = a;
    if (live) {
      a = *(const float4*)(S_mem + (size_t)r * d);
      b = *(const float4*)(S_mem + (size_t)r * d + 4);
    }
    S[r][0] = a.x; S[r][1] = a.y; S[r][2] = a.z; S[r][3] = a.w;
    S[r][4] = b.x; S[r][5] = b.y; S[r][6] = b.z; S[r][7] = b.w;
  }
  const int hist = p.n_taps - 1;
  for (int i = tid; i < 2 * d + N; i += nt) {
    const int c = i < d ? kh * d + i : i < 2 * d ? p.KH * d + kh * d + i - d : 2 * p.KH * d + kh * N + i - 2 * d;
    const float x = bf16_to_float(p.src[(size_t)s * p.src_stride + c]);
    float* kept = slot + p.conv_at + c;
    float w[DL_STEP_TAPS - 1];
#pragma unroll
    for (int k = 0; k < DL_STEP_TAPS - 1; ++k) w[k] = k < hist ? kept[(size_t)k * C] : 0.f;
    float acc = 0.f;
#pragma unroll
    for (int k = 0; k < DL_STEP_TAPS - 1; ++k)
      if (k < hist) {
        acc += p.taps[(size_t)c * p.n_taps + k] * w[k];
        kept[(size_t)k * C] = k + 1 < hist ? w[k + 1 < DL_STEP_TAPS - 1 ? k + 1 : k] : x;
      }
    acc += p.taps[(size_t)c * p.n_taps + hist] * x;
    lds[i] = dl_silu_to<float>(acc);        // q, k and v side by side
  }
  for (int j = tid; j < HG; j += nt) {
    const int h = kh * HG + j;
    const float* z = p.ab + (size_t)s * 2 * p.H;
    gs[j] = expf(-(expf(p.a_log[h]) * dl_softplus(z[h] + p.dt_bias[h])));
    bs[j] = 1.0f / (1.0f + expf(-z[p.H + h]));
  }
  __syncthreads();
  if (wave == 0) {
    float qq = 0.f, kk = 0.f, qk = 0.f;
    for (int c = lane; c < d; c += ZF_WAVE) {
      qq = fmaf(qs[c], qs[c], qq);
      kk = fmaf(ks[c], ks[c], kk);
      qk = fmaf(qs[c], ks[c], qk);
    }
    qq = wave_sum(qq);
    kk = wave_sum(kk);
    qk = wave_sum(qk);
    if (lane == 0) {
      const float iq = 1.0f / sqrtf(qq + p.unit_eps) * p.scale, ik = 1.0f / sqrtf(kk + p.unit_eps);
      s_unit[0] = iq;
      s_unit[1] = ik;
      s_unit[2] = qk * iq * ik;
    }
  }
  __syncthreads();
  if (live) {
    const float iq = s_unit[0], ik = s_unit[1], qk = s_unit[2];
    const int j = col / dv;
    const float g = gs[j], b = bs[j];
    float k8[8], rs[RV], ps[RV];
#pragma unroll
    for (int e = 0; e < 8; ++e) k8[e] = ks[cg * 8 + e] * ik;
#pragma unroll
    for (int r = 0; r < RV; ++r) {
      float r0 = 0.f, r1 = 0.f, p0 = 0.f, p1 = 0.f;
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        r0 = fmaf(k8[e], S[r][e], r0);
        r1 = fmaf(k8[e + 1], S[r][e + 1], r1);
        p0 = fmaf(qs[cg * 8 + e], S[r][e], p0);
        p1 = fmaf(qs[cg * 8 + e + 1], S[r][e + 1], p1);
      }
      rs[r] = r0 + r1;
      ps[r] = p0 + p1;
    }
    lanes_sum_up(rs, CG);
    lanes_sum_up(ps, CG);
#pragma unroll
    for (int r = 0; r < RV; ++r) {
      const float w = b * (vs[col + r] - g * rs[r]);
#pragma unroll
      for (int e = 0; e < 8; ++e) S[r][e] = g * S[r][e] + k8[e] * w;
      if (cg == 0) os[col + r] = g * (ps[r] * iq) + qk * w;
      *(float4*)(S_mem + (size_t)r * d) = make_float4(S[r][0], S[r][1], S[r][2], S[r][3]);
      *(float4*)(S_mem + (size_t)r * d + 4) = make_float4(S[r][4], S[r][5], S[r][6], S[r][7]);
    }
  }
  __syncthreads();
  for (int j = wave; j < HG; j += waves) {
    float ss = 0.f;
    for (int x = lane; x < dv; x += ZF_WAVE) ss = fmaf(os[j * dv + x], os[j * dv + x], ss);
    const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)dv + p.norm_eps);
    const size_t at = (size_t)(kh * HG + j) * dv;
    for (int x = lane; x < dv; x += ZF_WAVE) {
      const float gv = bf16_to_float(p.gate[(size_t)s * p.gate_stride + at + x]);
      p.out[(size_t)s * p.out_stride + at + x] =
          float_to_bf16(os[j * dv + x] * inv * p.gain[x] * (gv * (1.0f / (1.0f + expf(-gv)))));
    }
  }
}

// Columns a thread, 0: not these sizes.
static int delta_step_columns(int H, int KH, int d, int dv) {
  const int CG = d / 8;
  if (H < 1 || KH < 1 || H % KH != 0 || d % 8 != 0 || CG < 1 || CG > 16 || (CG & (CG - 1)) != 0 || dv < 1)
    return 0;
  for (int rv = 1; rv <= 8; rv *= 2)
    if (dv % rv == 0 && (long long)(H / KH) * dv / rv * CG <= 1024) return rv;
  return 0;
}

// A step of one token a sequence: src bfloat16 rows [n_seqs, >= C], taps [C][n_taps]; the convolutions' kept rows
// at conv_at of a slot, behind the matrices; slots 16-byte aligned.  gain [dv], gate and out rows [H dv].
extern "C" int zf_delta_step(const void* src, long long src_stride, const float* taps, int n_taps,
                             const float* ab, const float* a_log, const float* dt_bias, float* state,
                             long long state_stride, long long conv_at, const int* state_slots,
                             const float* gain, const void* gate, long long gate_stride, void* out,
                             long long out_stride, int n_seqs, int H, int KH, int d, int dv, float scale,
                             float unit_eps, float norm_eps, hipStream_t stream) {
  if (n_seqs <= 0) return 0;
  const int rv = delta_step_columns(H, KH, d, dv);
  if (rv == 0 || n_taps < 1 || n_taps > DL_STEP_TAPS || state_stride % 4 != 0 || (uintptr_t)state % 16 != 0)
    return -2;
  const int HG = H / KH, N = HG * dv;
  const DeltaStep p{(const bf16_t*)src, (const bf16_t*)gate, taps, ab, a_log, dt_bias, gain, state, state_slots,
                    (bf16_t*)out, src_stride, gate_stride, out_stride, state_stride, conv_at, n_taps, H, KH, d, dv,
                    d / 8, scale, unit_eps, norm_eps};
  const int threads = (N / rv * (d / 8) + ZF_WAVE - 1) / ZF_WAVE * ZF_WAVE;
  const size_t smem = (size_t)(2 * d + 2 * N + 2 * HG) * sizeof(float);
  const dim3 grid(KH, n_seqs);
  if (rv == 1) hipLaunchKernelGGL(delta_step_kernel<1>, grid, dim3(threads), smem, stream, p);
  else if (rv == 2) hipLaunchKernelGGL(delta_step_kernel<2>, grid, dim3(threads), smem, stream, p);
  else if (rv == 4) hipLaunchKernelGGL(delta_step_kernel<4>, grid, dim3(threads), smem, stream, p);
  else hipLaunchKernelGGL(delta_step_kernel<8>, grid, dim3(threads), smem, stream, p);
  ZF_CHECK_LAUNCH();
}

// ------------------------------------------------------------------ long portions in chunks
// Sixteen tokens at a time as products.  With G_t the sum of the chunk's log decays up to token t, the
// matrix S0 ahead of the chunk and w_t = beta_t (v_t - exp(G_t) S0^T k_t - sum over i < t of
// exp(G_t - G_i) (k_t . k_i) w_i),
//   W = Tb (V - exp(G) (K S0)),   Tb = (I + L)^-1 diag(beta),  L_ti = beta_t exp(G_t - G_i) k_t . k_i, i < t
//   O = exp(G) (Q S0) + M W,      M_ti = exp(G_t - G_i) q_t . k_i, i <= t
//   S = exp(G_15) S0 + K^T (exp(G_15 - G) W)
// (the chunked form by its triangular system: Yang, Wang, Zhang, Shen and Kim, "Parallelizing Linear
// Transformers with the Delta Rule over Sequence Length", 2024; with decays Yang, Kautz and Hatamizadeh,
// "Gated Delta Networks", 2024).
// Everything is 32-bit: v_mfma_f32_16x16x4_f32, expf, fused multiply-adds; no ratio of decays exceeds 1.
// A token that is not finite reaches itself and the tokens behind it, as in the walk: the triangular
// matrices hold zeros above their diagonals, whatever the token brings, but such zeros against its
// numbers in a product would reach every row.  What it brings stays in S, so a sequence that leaves an
// S that is not finite is walked once more, with its numbers taken out of those products first (a look
// at every chunk cost all sequences 4 to 8 %, the one at the end 0.5 us).
//   * delta_chunk_prepare  a wave a (chunk, head): Tb, M and the decays, all chunks side by side.
//   * delta_chunk_walk     a workgroup of four waves a (16 value columns, head, sequence) walks the
//                          chunks with S in the accumulators of the waves, d / 64 blocks of 16 key
//                          channels each.
// The walk token by token is bound by the vector units' issue: some 100 instructions a token and
// wave, 2.5 waves to a SIMD; here a chunk costs a wave 28 MFMAs of 32 cycles (d = 128), 32 the one that
// forms its outputs.
// Measured (16 heads of 128 x 128, a step of 2048 tokens of five prompts, the longest 680, us): 290
// walked, 87 + 15 in chunks; on inputs of such sizes 2.3 to 3.3e-7 off the 64-bit rule behind 200 to 2000
// tokens, the walk 2.9e-7 to 1.1e-6.
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float dl_f32x4_t;
#define DL_CHUNK 16
#define DL_CHUNK_FLOATS (2 * DL_CHUNK * DL_CHUNK + 2 * DL_CHUNK)   // Tb, M, exp(G), exp(G_15 - G)

// where chunk c of a sequence keeps its numbers: below (all tokens) / 16 + sequences + 1, no two alike
__device__ __forceinline__ size_t dl_chunk_at(int first, int seq, int c, int H, int h) {
  return ((size_t)(first / DL_CHUNK + seq + c) * H + h) * DL_CHUNK_FLOATS;
}

template <int ND>
__global__ __launch_bounds__(64) void delta_chunk_prepare_kernel(
    const float* __restrict__ qkv, int C, int q_off, int k_off, const float* __restrict__ ab,
    const float* __restrict__ a_log, const float* __restrict__ dt_bias,
    const int* __restrict__ q_start, float* __restrict__ ws, int H, int KH, int longest) {
  __shared__ float L[DL_CHUNK][DL_CHUNK + 1], log_g[DL_CHUNK], beta[DL_CHUNK];
  const int h = blockIdx.y, seq = blockIdx.z, lane = threadIdx.x, m = lane % 16, g = lane / 16;
  const int first = q_start[seq], len = q_start[seq + 1] - first;
  const int t0 = blockIdx.x * DL_CHUNK;
  if (len <= longest || t0 >= len) return;
  const int n = min(DL_CHUNK, len - t0), kh = h / (H / KH);
  constexpr int d = 16 * ND;
  const dl_f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  const float* row = qkv + (size_t)(first + t0 + min(m, n - 1)) * C + kh * d + 4 * g;
  dl_f32x4_t kk = zero, qk = zero, kf[ND], qf[ND];
#pragma unroll
  for (int b = 0; b < ND; ++b) {
    kf[b] = *(const dl_f32x4_t*)(row + k_off + 16 * b);
    qf[b] = *(const dl_f32x4_t*)(row + q_off + 16 * b);
  }
  if (lane < 16) {
    const float* z = ab + (size_t)(first + t0 + min(lane, n - 1)) * 2 * H;
    const float za = z[h], zb = z[H + h];
    // a token that is not there decays nothing and corrects nothing; exp(-110) is 0 as a float, and
    // sums of such stay finite
    const float v = -(expf(a_log[h]) * dl_softplus(za + dt_bias[h]));
    log_g[lane] = lane >= n ? 0.f : v < -110.f ? -110.f : v;
    beta[lane] = lane < n ? 1.0f / (1.0f + expf(-zb)) : 0.f;
  }
  // (rows of a token that is not there repeat the last one's; their columns are masked below)
#pragma unroll
  for (int b = 0; b < ND; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      kk = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[b][i], kf[b][i], kk, 0, 0, 0);
      qk = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[b][i], kf[b][i], qk, 0, 0, 0);
    }
  __syncthreads();
  // Column m is token i = m, the four rows are tokens t = 4 g + r.  The decays between two tokens
  // are added up from the earlier one on: the difference of two sums from the chunk's start would lose
  // the digits that a token which forgets everything has taken.
  float* dst = ws + dl_chunk_at(first, seq, blockIdx.x, H, h);
  float since = 0.f, start = 0.f, whole = 0.f, ratio[4];
#pragma unroll
  for (int t = 0; t < DL_CHUNK; ++t) {
    const float v = log_g[t];
    whole += v;
    since = t > m ? since + v : 0.f;
    if (t == m) start = whole;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (t == 4 * g + r) ratio[r] = t >= m ? expf(since) : 0.f;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int t = 4 * g + r;
    L[t][m] = t > m && m < n ? beta[t] * ratio[r] * kk[r] : 0.f;
    dst[DL_CHUNK * DL_CHUNK + t * DL_CHUNK + m] = t >= m && m < n ? ratio[r] * qk[r] : 0.f;
  }
  if (lane < 16) {
    dst[2 * DL_CHUNK * DL_CHUNK + lane] = expf(start);
    dst[2 * DL_CHUNK * DL_CHUNK + DL_CHUNK + lane] = expf(since);
  }
  __syncthreads();
  // (I + L)^-1, a column a lane, row after row
  if (lane < 16) {
    float x[DL_CHUNK];
#pragma unroll
    for (int t = 0; t < DL_CHUNK; ++t) {
      float v = t == lane ? 1.f : 0.f;
#pragma unroll
      for (int i = 0; i < t; ++i) v = fmaf(-L[t][i], x[i], v);
      x[t] = v;
    }
    const float b = beta[lane];
#pragma unroll
    for (int t = 0; t < DL_CHUNK; ++t) dst[t * DL_CHUNK + lane] = t >= lane ? x[t] * b : 0.f;
  }
}

// acc += the 16 x 16 lower triangular matrix whose row m holds `tri` at columns 4 g + i, times x.
// CAREFUL: of a column's rows (4 g + r, the column's lanes 16 apart) those from its first number on that
// is not finite are not finite, and the ones before have not met it.
template <bool CAREFUL>
__device__ __forceinline__ dl_f32x4_t dl_triangle(const dl_f32x4_t& tri, dl_f32x4_t x,
                                                  dl_f32x4_t acc, int g) {
  int bad = DL_CHUNK;
  if constexpr (CAREFUL) {
#pragma unroll
    for (int r = 3; r >= 0; --r)
      if (!(fabsf(x[r]) < INFINITY)) {
        bad = 4 * g + r;
        x[r] = 0.f;
      }
    bad = min(bad, __shfl_xor(bad, 16));
    bad = min(bad, __shfl_xor(bad, 32));
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(tri[i], x[i], acc, 0, 0, 0);
  if constexpr (CAREFUL) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (4 * g + r >= bad) acc[r] = NAN;
  }
  return acc;
}

// (as many registers as leave a CU the workgroups that one walk alone would: with three of four, four
// portions of 1024 tokens of 32 heads took 250 us for 215)
template <int ND>
__global__ __launch_bounds__(256, ND == 8 ? 4 : 5) void delta_chunk_walk_kernel(
    const float* __restrict__ qkv, int C, int q_off, int k_off, int v_off, float* __restrict__ state,
    long long state_stride, const int* __restrict__ state_slots, const int* __restrict__ q_start,
    const float* __restrict__ ws, float* __restrict__ out, int H, int KH, int dv, int longest) {
  constexpr int d = 16 * ND, B = ND / 4, LD = d + 4, LM = DL_CHUNK + 4;
  constexpr int PIECES = DL_CHUNK * d / 4 / 256;          // 16-byte pieces of K (and of Q) a thread
  static_assert(ND % 4 == 0 && PIECES >= 1, "blocks of channels for four waves");
  __shared__ __attribute__((aligned(16))) float ks[DL_CHUNK][LD], qs[DL_CHUNK][LD];
  __shared__ __attribute__((aligned(16))) float mats[2][DL_CHUNK][LM];   // Tb, M
  __shared__ float vs[DL_CHUNK][DL_CHUNK + 1], decays[2][DL_CHUNK];
  __shared__ dl_f32x4_t red[4][2][64];
  const int h = blockIdx.y, seq = blockIdx.z, kh = h / (H / KH);
  const int first = q_start[seq], len = q_start[seq + 1] - first;
  if (len <= longest) return;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
  const int m = lane % 16, g = lane / 16, col0 = blockIdx.x * 16;
  // S: row 4 g + r of block wave * B + b is key channel 16 (wave B + b) + 4 g + r, column m
  float* S_mem = state + (size_t)state_slots[seq] * state_stride + ((size_t)h * dv + col0 + m) * d
                 + 16 * wave * B + 4 * g;
  dl_f32x4_t S[B];
  dl_f32x4_t fk[PIECES], fq[PIECES];
  float fv, fm[2], fd;
  auto fetch = [&](int t0) {
    const int n = min(DL_CHUNK, len - t0);
#pragma unroll
    for (int j = 0; j < PIECES; ++j) {
      const int i = tid + 256 * j, tok = i / (d / 4), c = i % (d / 4) * 4;
      const float* row = qkv + (size_t)(first + t0 + min(tok, n - 1)) * C + kh * d + c;
      fk[j] = *(const dl_f32x4_t*)(row + k_off);
      fq[j] = *(const dl_f32x4_t*)(row + q_off);
    }
    const int tok = tid / 16;
    fv = qkv[(size_t)(first + t0 + min(tok, n - 1)) * C + v_off + h * dv + col0 + tid % 16];
    const float* src = ws + dl_chunk_at(first, seq, t0 / DL_CHUNK, H, h);
    fm[0] = src[tid];
    fm[1] = src[256 + tid];
    fd = src[512 + tid % 32];
  };
  auto walk = [&](auto CAREFUL_) __attribute__((always_inline)) {
    constexpr bool CAREFUL = decltype(CAREFUL_)::value;
#pragma unroll
    for (int b = 0; b < B; ++b) S[b] = *(const dl_f32x4_t*)(S_mem + 16 * b);
    fetch(0);
    for (int t0 = 0; t0 < len; t0 += DL_CHUNK) {
      const int n = min(DL_CHUNK, len - t0);
      __syncthreads();                        // the chunk before is done with
#pragma unroll
      for (int j = 0; j < PIECES; ++j) {
        const int i = tid + 256 * j, tok = i / (d / 4), c = i % (d / 4) * 4;
        *(dl_f32x4_t*)&ks[tok][c] = fk[j];
        *(dl_f32x4_t*)&qs[tok][c] = fq[j];
      }
      vs[tid / 16][tid % 16] = fv;
      mats[0][tid / 16][tid % 16] = fm[0];
      mats[1][tid / 16][tid % 16] = fm[1];
      if (tid < 32) decays[tid / 16][tid % 16] = fd;
      __syncthreads();
      if (t0 + DL_CHUNK < len) fetch(t0 + DL_CHUNK);
      // this wave's channels' share of K S0 and Q S0 (element i of a lane's four channels in MFMA i,
      // where S has the same ones as element i of its rows)
      dl_f32x4_t pk = {0.f, 0.f, 0.f, 0.f}, pq = pk;
#pragma unroll
      for (int b = 0; b < B; ++b) {
        const dl_f32x4_t kv = *(const dl_f32x4_t*)&ks[m][16 * (wave * B + b) + 4 * g];
        const dl_f32x4_t qv = *(const dl_f32x4_t*)&qs[m][16 * (wave * B + b) + 4 * g];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          pk = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[i], S[b][i], pk, 0, 0, 0);
          pq = __builtin_amdgcn_mfma_f32_16x16x4f32(qv[i], S[b][i], pq, 0, 0, 0);
        }
      }
      red[wave][0][lane] = pk;
      red[wave][1][lane] = pq;
      __syncthreads();
      // rows 4 g + r are tokens, column m a value column; every wave forms W for its own channels
      const dl_f32x4_t sk = (red[0][0][lane] + red[1][0][lane]) + (red[2][0][lane] + red[3][0][lane]);
      const dl_f32x4_t tb = *(const dl_f32x4_t*)&mats[0][m][4 * g];
      dl_f32x4_t x;
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = fmaf(-decays[0][4 * g + r], sk[r], vs[4 * g + r][m]);
      const dl_f32x4_t W = dl_triangle<CAREFUL>(tb, x, dl_f32x4_t{0.f, 0.f, 0.f, 0.f}, g);
      const float whole = decays[0][DL_CHUNK - 1];
      float cw[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) cw[i] = decays[1][4 * g + i] * W[i];
#pragma unroll
      for (int b = 0; b < B; ++b) {
        float kt[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) kt[i] = ks[4 * g + i][16 * (wave * B + b) + m];
        S[b] = S[b] * whole;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          S[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[i], cw[i], S[b], 0, 0, 0);
      }
      if (wave == t0 / DL_CHUNK % 4) {        // the outputs, the waves in turn
        const dl_f32x4_t sq = (red[0][1][lane] + red[1][1][lane]) + (red[2][1][lane] + red[3][1][lane]);
        const dl_f32x4_t mv = *(const dl_f32x4_t*)&mats[1][m][4 * g];
        dl_f32x4_t o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = decays[0][4 * g + r] * sq[r];
        o = dl_triangle<CAREFUL>(mv, W, o, g);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (4 * g + r < n)
            out[(size_t)(first + t0 + 4 * g + r) * H * dv + (size_t)h * dv + col0 + m] = o[r];
      }
    }
  };
  walk(std::false_type{});
  bool finite = true;
#pragma unroll
  for (int b = 0; b < B; ++b)
#pragma unroll
    for (int i = 0; i < 4; ++i) finite = finite && fabsf(S[b][i]) < INFINITY;
  if (__syncthreads_or(!finite)) walk(std::true_type{});
#pragma unroll
  for (int b = 0; b < B; ++b) *(dl_f32x4_t*)(S_mem + 16 * b) = S[b];
}

// The sequences that bring more than `longest` tokens (max_len: what the longest one brings), in chunks;
// d 64 or 128 (the padded key size too), dv a multiple of 16, 16-byte aligned rows; ws: (T / 16 +
// n_seqs + 1) * H * DL_CHUNK_FLOATS floats.
extern "C" int zf_delta_chunks(const float* qkv, int C, int q_off, int k_off, int v_off,
                               const float* ab, const float* a_log, const float* dt_bias,
                               float* state, long long state_stride, const int* state_slots,
                               const int* q_start, float* out, float* ws, int n_seqs, int max_len,
                               int H, int KH, int d, int dv, int longest, hipStream_t stream) {
  if (n_seqs <= 0 || max_len <= longest) return 0;
  if (H < 1 || KH < 1 || H % KH != 0 || (d != 64 && d != 128) || dv < 16 || dv % 16 != 0 ||
      (C | q_off | k_off) % 4 != 0 || state_stride % 4 != 0 ||
      (((uintptr_t)qkv | (uintptr_t)state) % 16) != 0 || ws == nullptr || longest < 0)
    return -2;
  const dim3 pgrid((max_len + DL_CHUNK - 1) / DL_CHUNK, H, n_seqs), wgrid(dv / 16, H, n_seqs);
#define DL_CHUNKS(ND)                                                                            \
  do {                                                                                           \
    hipLaunchKernelGGL((delta_chunk_prepare_kernel<ND>), pgrid, dim3(64), 0, stream, qkv, C, q_off, \
                       k_off, ab, a_log, dt_bias, q_start, ws, H, KH, longest);                  \
    hipLaunchKernelGGL((delta_chunk_walk_kernel<ND>), wgrid, dim3(256), 0, stream, qkv, C, q_off, \
                       k_off, v_off, state, state_stride, state_slots, q_start, ws, out, H, KH, dv, \
                       longest);                                                                 \
  } while (0)
  if (d == 64) DL_CHUNKS(4); else DL_CHUNKS(8);
#undef DL_CHUNKS
  ZF_CHECK_LAUNCH();
}
