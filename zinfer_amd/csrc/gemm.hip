// Matrix products C[M,N] = A[M,K] * W[N,K]^T (the weight is [out, in], as in the reference:
// y[r] = sum_c W[r,c] x[c], src/tensor/storage/store.zig:286-319).
//
//  * gemm_f32: float32 operands, 32-bit MFMAs, any sizes: the true 32-bit path.  One order of
//    the sum whatever M is and wherever the row lies in the batch, so a token's result does not
//    depend on how the batch was cut.
//  * gemm_fma: 32-bit FMA for mixed storage types, any sizes.  Every output element is the sum
//    of its products in ascending k, whatever M is and wherever the row lies in the batch.
#include <type_traits>

#include "zf_common.h"

#define GF_BM 64
#define GF_BN 64
#define GF_BK 16

template <typename TA, typename TW, typename TO, bool ACC>
__global__ __launch_bounds__(256) void gemm_fma_kernel(const TA* __restrict__ A,
                                                       const TW* __restrict__ W,
                                                       TO* __restrict__ C, int M, int N, int K) {
  __shared__ float As[GF_BK][GF_BM + 4];
  __shared__ float Ws[GF_BK][GF_BN + 4];
  const int tid = threadIdx.x;
  const int tx = tid % 16, ty = tid / 16;       // 16 x 16 threads, each 4 x 4 outputs
  const int m0 = blockIdx.y * GF_BM, n0 = blockIdx.x * GF_BN;
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

  // each thread loads 4 elements of A and 4 of W per k-tile: row = tid / 4, k = (tid % 4) * 4..
  const int lr = tid / 4, lk = (tid % 4) * 4;
  for (int k0 = 0; k0 < K; k0 += GF_BK) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = k0 + lk + i;
      const int am = m0 + lr, wn = n0 + lr;
      As[lk + i][lr] = (am < M && k < K) ? load_as_float<TA>(A + (size_t)am * K + k) : 0.f;
      Ws[lk + i][lr] = (wn < N && k < K) ? load_as_float<TW>(W + (size_t)wn * K + k) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < GF_BK; ++kk) {
      float a[4], w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = Ws[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= N) continue;
      TO* c = C + (size_t)m * N + n;
      if (ACC)
        store_from_float<TO>(c, load_as_float<TO>(c) + acc[i][j]);
      else
        store_from_float<TO>(c, acc[i][j]);
    }
  }
}

template <typename TA, typename TW, typename TO>
static void launch_fma(const void* A, const void* W, void* C, int M, int N, int K, int accumulate,
                       hipStream_t stream) {
  dim3 grid((N + GF_BN - 1) / GF_BN, (M + GF_BM - 1) / GF_BM);
  if (accumulate)
    hipLaunchKernelGGL((gemm_fma_kernel<TA, TW, TO, true>), grid, dim3(256), 0, stream,
                       (const TA*)A, (const TW*)W, (TO*)C, M, N, K);
  else
    hipLaunchKernelGGL((gemm_fma_kernel<TA, TW, TO, false>), grid, dim3(256), 0, stream,
                       (const TA*)A, (const TW*)W, (TO*)C, M, N, K);
}

// dtypes: ZF_F32 / ZF_BF16 for a, w, out, a and w not both float32 (zf_gemm_f32 takes those).
// accumulate: out += (else out =).
extern "C" int zf_gemm_fma(const void* A, int a_dtype, const void* W, int w_dtype, void* C,
                           int c_dtype, int M, int N, int K, int accumulate,
                           hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  const int key = a_dtype * 4 + w_dtype * 2 + c_dtype;
  switch (key) {
    case 2: launch_fma<float, bf16_t, float>(A, W, C, M, N, K, accumulate, stream); break;
    case 3: launch_fma<float, bf16_t, bf16_t>(A, W, C, M, N, K, accumulate, stream); break;
    case 4: launch_fma<bf16_t, float, float>(A, W, C, M, N, K, accumulate, stream); break;
    case 5: launch_fma<bf16_t, float, bf16_t>(A, W, C, M, N, K, accumulate, stream); break;
    case 6: launch_fma<bf16_t, bf16_t, float>(A, W, C, M, N, K, accumulate, stream); break;
    case 7: launch_fma<bf16_t, bf16_t, bf16_t>(A, W, C, M, N, K, accumulate, stream); break;
    default: return -1;
  }
  ZF_CHECK_LAUNCH();
}

// =====================================================================================
//  bfloat16 MFMA kernels (gfx950): v_mfma_f32_32x32x16_bf16 and v_mfma_f32_16x16x32_bf16,
//  fp32 accumulation.  A is [M, K] bfloat16, W is [N, K] bfloat16, both with K contiguous,
//  which is the operand order the instruction wants: every lane feeds 8 consecutive k of
//  one row of A and of one row of W.
// =====================================================================================
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_t;
typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2_t;

// XCD-aware tile order.  Consecutive workgroups go to different XCDs (8 of them, each with its
// own L2), so workgroup b takes place (b % 8) * per_xcd + b / 8 of the tile order: one XCD
// then walks neighbouring tiles.  The order runs through groups of at most GROUP tile rows,
// down the rows of a group first, so that the tiles an XCD walks share W tiles in its L2.  The
// rows are dealt evenly over the groups (9 rows in groups of 8: 5 + 4, not 8 + 1): a group of
// one row would send an XCD through every W tile on its own.
template <int GROUP>
__device__ __forceinline__ void tile_of_workgroup(int b, int tiles_m, int tiles_n, int& tm,
                                                  int& tn) {
  const int nblocks = tiles_m * tiles_n;
  {
    const int base = nblocks / 8, rem = nblocks % 8;
    const int xcd = b % 8, idx = b / 8;
    b = xcd * base + min(xcd, rem) + idx;   // XCD x owns base (+1 if x < rem) tiles in a row
  }
  const int ngroups = (tiles_m + GROUP - 1) / GROUP;
  const int rows = tiles_m / ngroups, longer = tiles_m % ngroups;   // the first groups: rows + 1
  const int in_longer = (rows + 1) * tiles_n;
  int first_m, gsize, at;
  if (b < longer * in_longer) {
    gsize = rows + 1;
    first_m = (b / in_longer) * gsize;
    at = b % in_longer;
  } else {
    const int bb = b - longer * in_longer, in_group = rows * tiles_n;
    gsize = rows;
    first_m = longer * (rows + 1) + (bb / in_group) * rows;
    at = bb % in_group;
  }
  tm = first_m + at % gsize;
  tn = at / gsize;
}

// ------------------------------------------------------------------ 32-bit MFMA product
// A, W and the sums are float32 throughout: v_mfma_f32_16x16x4_f32 multiplies and adds in full
// 32-bit precision, at 256 flops a cycle and CU (154 TFLOP/s; a VALU loop of scalar FMAs gets
// half of that at best and, with 4 x 4 outputs a thread, one LDS word per FMA, a tenth).
//
// One order of the sum for every number of rows, so that a token's result does not depend on
// how the batch was cut: K is dealt in eight spans (F32_SPAN below, a function of K alone), each
// summed from zero in ascending steps of 32, and the spans are added in ascending order to zero.
// Inside a step of 32 a lane's group g = lane / 16 holds k = 8 g .. 8 g + 7, and MFMA j takes
// element j of every group, which lets 16-byte loads of rows feed the operands as they are.
// Three kernels follow that order:
//   * up to 64 rows, bound by reading W (one user of the 0.6B shape's float32 weights: 1.9 GB a
//     token): a workgroup of eight waves, one span each, takes 16 rows of W (32 with a wide
//     output) for all tokens; a wave's loads of a step are 16 whole lines of 128 bytes, straight
//     into the operands, up to two steps in flight; the eight partials meet in LDS.  For narrow outputs
//     every span is a workgroup, and a second kernel adds the spans (gemm_f32_spans_kernel).
//   * above, bound by the MFMAs: tiles through a ring of LDS stages (gemm_f32_ring_kernel); of other
//     sizes, alignments and outputs tiles of 128 x 128, 64 x 64 or 32 x 32 through LDS (rows of 36
//     words: the 16-byte operand reads of 16 rows fall into different banks), the next step's
//     loads in flight during the products.  The largest tile that still gives 256 workgroups.
// Measured (weights from HBM, us, against the scalar loop of 64 x 64 tiles before): 4 tokens into
// 1024 outputs over K = 3072 290 -> 13, 6144 x 1024 107 -> 8.2, 151936 x 1024 474 -> 120 (5.2
// TB/s), 4096 x 12288 1254 -> 64; 256 tokens into 1024 x 3072 350 -> 17, 6144 x 1024 163 -> 30;
// 2048 tokens into 24576 x 4096 10925 -> 2970 (139 TFLOP/s; the vendor's product 154).  Up to 64
// rows the streaming kernel wins or draws (48 tokens: 24576 x 4096 240 us, the tiles at 96: 258).
static __host__ __device__ __forceinline__ int f32_span(int K) { return (K + 255) / 256 * 32; }
#define F32_SPANS 8

// four consecutive k of one row; what lies at or beyond k_end is 0
template <bool VEC>
__device__ __forceinline__ f32x4_t f32_load4(const float* __restrict__ row, int k, int k_end) {
  if constexpr (VEC) {        // K a multiple of 4 and 16-byte aligned rows: all four or none
    return k < k_end ? *(const f32x4_t*)(row + k) : f32x4_t{0.f, 0.f, 0.f, 0.f};
  } else {
    f32x4_t v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = k + i < k_end ? row[k + i] : 0.f;
    return v;
  }
}

// outputs n .. n + 3 of row m (sum: their 32-bit sums); vec: 16-byte stores are aligned
template <typename TO, bool ACC>
__device__ __forceinline__ void f32_store4(TO* __restrict__ C, int m, int n, int N, bool vec,
                                           f32x4_t sum) {
  TO* c = C + (size_t)m * N + n;
  if constexpr (std::is_same<TO, float>::value) {
    if (vec && n + 3 < N) {
      if constexpr (ACC) sum = *(const f32x4_t*)c + sum;
      *(f32x4_t*)c = sum;
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (n + i < N) store_from_float<TO>(c + i, ACC ? load_as_float<TO>(c + i) + sum[i] : sum[i]);
}

// GLU (RG 2, one group of tokens): W is a gate's N rows and then an up projection's N rows; the two
// row groups are the same rows of both, and silu(gate) * up of the 32-bit sums is stored: the bits of
// the product and zf_swiglu behind it, without the launch and the way through memory (4 tokens,
// 6144 rows of 1024: 8.1 + 4.7 -> 9.1 us in the trace).
template <typename TO, bool ACC, int RG, int MT, bool VEC, int SETS, bool GLU = false>
__global__ __launch_bounds__(F32_SPANS * 64) void gemm_f32_stream_kernel(
    const float* __restrict__ A, const float* __restrict__ W, TO* __restrict__ C, int M, int N,
    int K, int span, bool vec_out) {
  __shared__ f32x4_t part[F32_SPANS][RG * MT][64];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, r = lane % 16, g = lane / 16;
  static_assert(!GLU || (RG == 2 && MT == 1 && !ACC), "a gate's and an up projection's rows");
  const int n0 = blockIdx.x * 16 * (GLU ? 1 : RG), m0 = blockIdx.y * 16 * MT;
  // rows beyond the matrices read its last row; nothing of theirs is stored
  const float* w[RG];
  const float* a[MT];
#pragma unroll
  for (int i = 0; i < RG; ++i)
    w[i] = W + (size_t)(GLU ? i * N + min(n0 + r, N - 1) : min(n0 + 16 * i + r, N - 1)) * K;
#pragma unroll
  for (int i = 0; i < MT; ++i) a[i] = A + (size_t)min(m0 + 16 * i + r, M - 1) * K;
  f32x4_t acc[RG][MT];
#pragma unroll
  for (int i = 0; i < RG; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // SETS 2, two steps in flight: the next but one is asked for behind the products that free its registers.
  // SETS 1, a loop that asks for a few steps and then multiplies them: fewer registers and so more waves.
  const int k_first = wave * span, k_end = min(K, k_first + span);
  f32x4_t wf[SETS][RG][2], af[SETS][MT][2];
  auto load = [&](int b, int k0) __attribute__((always_inline)) {      // (steps beyond the span: zeros)
    const int k = k0 + 8 * g;
#pragma unroll
    for (int i = 0; i < RG; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) wf[b][i][h] = f32_load4<VEC>(w[i], k + 4 * h, k_end);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) af[b][i][h] = f32_load4<VEC>(a[i], k + 4 * h, k_end);
  };
  auto multiply = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int i = 0; i < RG; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[b][i][s / 4][s % 4], af[b][j][s / 4][s % 4],
                                                           acc[i][j], 0, 0, 0);
  };
  if constexpr (SETS == 1) {
#pragma unroll (RG * MT >= 4 ? 1 : RG * MT == 2 ? 2 : 4)
    for (int k0 = k_first; k0 < k_end; k0 += 32) {
      load(0, k0);
      multiply(0);
    }
  } else {
    load(0, k_first);
    __builtin_amdgcn_sched_barrier(0);
    load(1, k_first + 32);
    __builtin_amdgcn_sched_barrier(0);
    for (int k0 = k_first; k0 < k_end; k0 += 64) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        if (b == 1 && k0 + 32 >= k_end) break;
        multiply(b);
        __builtin_amdgcn_sched_barrier(0);
        if (k0 + 64 < k_end) {
          load(b, k0 + 32 * (2 + b));
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < RG; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) part[wave][i * MT + j][lane] = acc[i][j];
  __syncthreads();
  if constexpr (GLU) {
    if (threadIdx.x >= 64) return;
    f32x4_t gate = f32x4_t{0.f, 0.f, 0.f, 0.f}, up = gate;
#pragma unroll
    for (int s = 0; s < F32_SPANS; ++s) {
      gate += part[s][0][lane];
      up += part[s][1][lane];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) gate[e] = gate[e] / (1.0f + expf(-gate[e])) * up[e];
    if (m0 + r < M) f32_store4<TO, false>(C, m0 + r, n0 + 4 * g, N, vec_out, gate);
    return;
  }
  if (threadIdx.x >= RG * MT * 64) return;
  // a lane's column is a token, its four rows are outputs: tile `wave` of the RG x MT ones
  f32x4_t sum = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < F32_SPANS; ++s) sum += part[s][wave][lane];
  const int m = m0 + 16 * (wave % MT) + r, n = n0 + 16 * (wave / MT) + 4 * g;
  if (m < M) f32_store4<TO, ACC>(C, m, n, N, vec_out, sum);
}

// The streaming kernel's product with every span of 16 rows in a wave and a workgroup of its own:
// the spans' sums go to ws [F32_SPANS][M][N], and the kernel that adds them, in span order, joins
// what comes behind (the residual, the norm).  For outputs whose row groups leave most of the
// chip idle: a group's eight waves together on one CU wait for its matrix core (32 cycles an MFMA,
// whatever the number of tokens) and for one another's loads.  DEPTH batches of BATCH steps in flight.
// In the trace, 4 tokens into 1024 outputs over K = 2048 and 3072, the mean of both: 14.2 -> 5.3 us, the
// kernel that adds them in the place of the norm's (4.6 -> 4.5); deeper batches in the eight waves' own
// kernel alone had reached 8.6 and 13.6 us in a chain (12.2 and 17.0 before, 8.4 and 9.9 so).
template <int MT>
__global__ __launch_bounds__(64) void gemm_f32_spans_kernel(const float* __restrict__ A,
                                                            const float* __restrict__ W,
                                                            float* __restrict__ ws, int M, int N,
                                                            int K, int span) {
  constexpr int BATCH = MT == 1 ? 4 : MT == 2 ? 2 : 1, DEPTH = MT == 4 ? 4 : 3, STEP = 32 * BATCH;
  const int lane = threadIdx.x, r = lane % 16, g = lane / 16;
  const int n0 = blockIdx.x * 16, k0 = blockIdx.y * span;
  const float* w = W + (size_t)min(n0 + r, N - 1) * K + 8 * g;
  const float* a[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) a[j] = A + (size_t)min(16 * j + r, M - 1) * K + 8 * g;
  f32x4_t acc[MT], wf[DEPTH][BATCH][2], af[DEPTH][BATCH][MT][2];
#pragma unroll
  for (int j = 0; j < MT; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto load = [&](int b, int k) {
#pragma unroll
    for (int u = 0; u < BATCH; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        wf[b][u][h] = *(const f32x4_t*)(w + k + 32 * u + 4 * h);
#pragma unroll
        for (int j = 0; j < MT; ++j) af[b][u][j][h] = *(const f32x4_t*)(a[j] + k + 32 * u + 4 * h);
      }
  };
  auto step = [&](const f32x4_t (&wv)[2], const f32x4_t (&av)[MT][2]) {
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
      for (int j = 0; j < MT; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[s / 4][s % 4], av[j][s / 4][s % 4], acc[j],
                                                      0, 0, 0);
  };
  auto compute = [&](int b) {
#pragma unroll
    for (int u = 0; u < BATCH; ++u) step(wf[b][u], af[b][u]);
  };
  const int len = max(0, min(K - k0, span)), nb = len / STEP;
  // The first DEPTH batches at once; from then on a batch is asked for behind the products of the
  // one whose registers it takes.  Every branch is the wave's.
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if (d < nb) load(d, k0 + d * STEP);
  int b = 0;
  for (; b + 2 * DEPTH <= nb; b += DEPTH)
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      __builtin_amdgcn_sched_barrier(0);
      compute(d);
      __builtin_amdgcn_sched_barrier(0);
      load(d, k0 + (b + DEPTH + d) * STEP);
    }
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    __builtin_amdgcn_sched_barrier(0);
    if (b + d < nb) compute(d);
    __builtin_amdgcn_sched_barrier(0);
    if (b + DEPTH + d < nb) load(d, k0 + (b + DEPTH + d) * STEP);
  }
#pragma unroll
  for (int d = 0; d < DEPTH - 1; ++d)
    if (b + DEPTH + d < nb) compute(d);
  for (int k = nb * STEP; k < len; k += 32) {       // steps that make no batch, the last one in part
    f32x4_t wv[2], av[MT][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      wv[h] = f32_load4<true>(w + k0, k + 4 * h, len - 8 * g);
#pragma unroll
      for (int j = 0; j < MT; ++j) av[j][h] = f32_load4<true>(a[j] + k0, k + 4 * h, len - 8 * g);
    }
    step(wv, av);
  }
#pragma unroll
  for (int j = 0; j < MT; ++j) {
    const int m = 16 * j + r, n = n0 + 4 * g;
    if (m < M && n < N) *(f32x4_t*)(ws + ((size_t)blockIdx.y * M + m) * N + n) = acc[j];
  }
}

// B x B outputs a workgroup of 2 x 2 waves; ST steps of 32 of K between two barriers: the small
// tiles have little to multiply in a step, and a barrier with one step's loads in flight takes 0.45
// us (256 tokens into 1024 outputs over K = 3072, tiles of 32: 42 us with 96 barriers, 29 with 24;
// 4096 outputs over 1024, tiles of 64: 31.8 -> 28.9 with two steps; with more than 512 of those the
// LDS that two steps take costs more, 24576 x 4096 at 96 tokens 258 -> 282 us).
template <typename TO, bool ACC, int B, int ST, bool VEC>
__global__ __launch_bounds__(256) void gemm_f32_tile_kernel(
    const float* __restrict__ A, const float* __restrict__ W, TO* __restrict__ C, int M, int N,
    int K, int span, bool vec_out) {
  constexpr int F = B / 32, L = B / 32;      // 16-wide fragments a wave and side; loads a thread
  constexpr int LD = 32 * ST + 4;            // (rows 4 words apart modulo the 64 banks)
  __shared__ __attribute__((aligned(16))) float As[2][B][LD];
  __shared__ __attribute__((aligned(16))) float Ws[2][B][LD];
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64, r = lane % 16, g = lane / 16;
  const int n0 = blockIdx.x * B, m0 = blockIdx.y * B;
  const int wm = (wave % 2) * (B / 2), wn = (wave / 2) * (B / 2);
  const int lr = tid / 8, lk = (tid % 8) * 4;        // staging: 32 rows x 128 bytes a pass
  const float *ap[L], *wp[L];
#pragma unroll
  for (int i = 0; i < L; ++i) {
    ap[i] = A + (size_t)min(m0 + lr + 32 * i, M - 1) * K;
    wp[i] = W + (size_t)min(n0 + lr + 32 * i, N - 1) * K;
  }
  f32x4_t acc[F][F], sum[F][F], ar[ST][L], wr[ST][L];
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) acc[i][j] = sum[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int steps = (K + 31) / 32, per = span / 32;
  auto fetch = [&](int st) {                         // (steps beyond the last are zeros)
#pragma unroll
    for (int s = 0; s < ST; ++s)
#pragma unroll
      for (int i = 0; i < L; ++i) {
        ar[s][i] = f32_load4<VEC>(ap[i], (st + s) * 32 + lk, K);
        wr[s][i] = f32_load4<VEC>(wp[i], (st + s) * 32 + lk, K);
      }
  };
  fetch(0);
  int in_span = 0;
  for (int st = 0; st < steps; st += ST) {
    const int b = st / ST % 2;
#pragma unroll
    for (int s = 0; s < ST; ++s)
#pragma unroll
      for (int i = 0; i < L; ++i) {
        *(f32x4_t*)&As[b][lr + 32 * i][32 * s + lk] = ar[s][i];
        *(f32x4_t*)&Ws[b][lr + 32 * i][32 * s + lk] = wr[s][i];
      }
    // one barrier a stage: the buffer written next was last read before the barrier of this one
    __syncthreads();
    if (st + ST < steps) fetch(st + ST);
#pragma unroll
    for (int s = 0; s < ST; ++s) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        f32x4_t wf[F], af[F];
#pragma unroll
        for (int i = 0; i < F; ++i) {
          wf[i] = *(const f32x4_t*)&Ws[b][wn + 16 * i + r][32 * s + 8 * g + 4 * h];
          af[i] = *(const f32x4_t*)&As[b][wm + 16 * i + r][32 * s + 8 * g + 4 * h];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < F; ++i)
#pragma unroll
            for (int j = 0; j < F; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[i][e], af[j][e], acc[i][j], 0, 0, 0);
      }
      // a span ends behind its last step (steps beyond K add zeros to a span that is empty)
      if (++in_span == per || st + s + 1 == steps) {
        in_span = 0;
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
          for (int j = 0; j < F; ++j) {
            sum[i][j] += acc[i][j];
            acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
          }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j) {
      const int m = m0 + wm + 16 * j + r, n = n0 + wn + 16 * i + 4 * g;
      if (m < M) f32_store4<TO, ACC>(C, m, n, N, vec_out, sum[i][j]);
    }
}

// The same products from aligned operands and whole steps (K % 32 == 0) over more than 64 rows: BM x BN
// outputs a group of 2 x 2 waves, both operands copied straight into a ring of NS stages of one step each.
// The kernel above asks for a stage's numbers, multiplies the stage before, and only then lays them
// down; here a stage's copies are NS - 1 stages old when they are waited for.  A stage's row is a line of
// 128 bytes: its eight 16-byte pieces, in the order 0 2 4 6 1 3 5 7, permuted by the row, so that the
// operand reads of 16 rows (piece 2 g + h of lane group g) fall into different banks.  The operands of a
// half step are read behind the products of the half before.
// KG 2: two groups of waves, each its own ring and four of the eight spans; the second lays its spans'
// sums down for the first, which adds them in order: twice the waves where the tiles are few and
// every wave is one chain of products.
// Measured, us, as the kernel above -> here (the chosen tile): 256 rows into 4096 over 1024 26.4 -> 21.0, into
// 6144 43.5 -> 29.5, into 1024 over 2048 19.9 -> 12.2, over 3072 28.8 -> 16.9; 131 rows 23.9 -> 17.1, 42.5 ->
// 20.9, 19.5 -> 11.4, 28.4 -> 16.3; 2048 rows into 24576 over 4096 3920 -> 2970 (139 TFLOP/s; the MFMAs 154).
// Tiles in the order of tile_of_workgroup: row by row of tiles, a wide W was read once for each (100 rows
// into 151936 over 1024 501 us, so 360).
template <int BM, int BN, int KG, bool ACC>
__global__ __launch_bounds__(256 * KG) void gemm_f32_ring_kernel(
    const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M, int N,
    int K, int span, int tiles_m, int tiles_n) {
  // (the host pass, which only needs the launch stub, does not know the buffer descriptor type)
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NS = KG == 2 ? 4 : 3;                      // stages
  constexpr int FM = BM / 32, FN = BN / 32;                // 16-wide fragments a wave and side
  constexpr int A_PLACES = BM * 8, W_PLACES = BN * 8;      // 16-byte pieces of a step of 32
  constexpr int AC = A_PLACES / 256, WC = W_PLACES / 256, COPIES = AC + WC;      // copies a thread
  constexpr int STAGE = A_PLACES + W_PLACES;
  __shared__ u32x4_t stage0[KG * STAGE];
  __shared__ u32x4_t stage1[KG * STAGE];
  __shared__ u32x4_t stage2[KG * STAGE];
  __shared__ u32x4_t stage3[NS > 3 ? KG * STAGE : 1];
  __shared__ f32x4_t spans[KG > 1 ? F32_SPANS / 2 * FM * FN * 256 : 1];
  const int kg = KG > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / 256) : 0;
  auto stage_of = [&](auto IDX) __attribute__((always_inline)) -> u32x4_t* {
    constexpr int I = decltype(IDX)::value % NS;
    if constexpr (I == 0) return stage0 + kg * STAGE;
    else if constexpr (I == 1) return stage1 + kg * STAGE;
    else if constexpr (I == 2) return stage2 + kg * STAGE;
    else return stage3 + kg * STAGE;
  };
  const int tid = threadIdx.x % 256, wave = tid / 64, lane = tid % 64, r = lane % 16, g = lane / 16;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);      // the LDS address is a scalar
  int tm, tn;
  tile_of_workgroup<8>(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int wm = (wave % 2) * (BM / 2), wn = (wave / 2) * (BN / 2);
  const __amdgpu_buffer_rsrc_t a_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)(A + (size_t)m0 * K), 0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t w_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)(W + (size_t)n0 * K), 0, 0x7fffffff, 0x00020000);
  // place p is row p / 8, slot p % 8, number q = slot ^ (row / 2 % 8) of the order above (rows beyond the
  // matrices: the last one; nothing of theirs is stored)
  auto source = [&](int p, int rows) __attribute__((always_inline)) {
    const int row = p / 8, q = (p % 8) ^ ((row >> 1) & 7);
    return ((uint32_t)min(row, rows - 1) * (uint32_t)K + (((q & 3) << 1) | (q >> 2)) * 4) * 4;
  };
  uint32_t asrc[AC], wsrc[WC];
#pragma unroll
  for (int c = 0; c < AC; ++c) asrc[c] = source(tid + 256 * c, M - m0);
#pragma unroll
  for (int c = 0; c < WC; ++c) wsrc[c] = source(tid + 256 * c, N - n0);
  // this group's steps: from `first` on; steps behind the last are the last again, and not added
  const int steps = K / 32, per = span / 32, last = steps - 1, first = kg * (F32_SPANS / 2) * per;
  const int stages = KG > 1 ? min(F32_SPANS / 2 * per, steps) : steps;
  auto copies = [&](int stage, u32x4_t* to) __attribute__((always_inline)) {
    const uint32_t at = (uint32_t)min(first + stage, last) * 128;
#pragma unroll
    for (int c = 0; c < AC; ++c)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          a_rsrc, (__attribute__((address_space(3))) void*)(to + wave_u * 64 + c * 256), 16, asrc[c], at, 0, 0);
#pragma unroll
    for (int c = 0; c < WC; ++c)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          w_rsrc, (__attribute__((address_space(3))) void*)(to + A_PLACES + wave_u * 64 + c * 256), 16, wsrc[c],
          at, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4_t acc[FN][FM], sum[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[i][j] = sum[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int at[2];      // piece 2 g + h of row r: number g + 4 h
#pragma unroll
  for (int h = 0; h < 2; ++h) at[h] = r * 8 + ((g + 4 * h) ^ (r >> 1));
  f32x4_t af[2][FM], wf[2][FN];
  auto read = [&](const u32x4_t* from, auto H) __attribute__((always_inline)) {
    constexpr int h = decltype(H)::value;
#pragma unroll
    for (int j = 0; j < FM; ++j) af[h][j] = *(const f32x4_t*)&from[(wm + 16 * j) * 8 + at[h]];
#pragma unroll
    for (int i = 0; i < FN; ++i) wf[h][i] = *(const f32x4_t*)&from[A_PLACES + (wn + 16 * i) * 8 + at[h]];
    __builtin_amdgcn_sched_barrier(0);
  };
  auto multiply = [&](auto H) __attribute__((always_inline)) {
    constexpr int h = decltype(H)::value;
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[h][i][e], af[h][j][e], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  copies(0, stage_of(I0{}));
  copies(1, stage_of(I1{}));
  copies(2, stage_of(I2{}));
  if constexpr (NS > 3) copies(3, stage_of(I3{}));
  constexpr int FIRST = (NS - 1) * COPIES, AHEAD = (NS - 2) * COPIES;      // younger copies at a meeting
  static_assert(FIRST < 64, "the wait counts them");
  __builtin_amdgcn_s_waitcnt(0x0f70 | (FIRST & 15) | ((FIRST >> 4) << 14));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  read(stage_of(I0{}), I0{});
  int in_span = 0, span_at = 0;
  // Stage t: ahead of its second half the wave waits for the next stage's copies and its own reads and
  // meets the others, behind which this stage's places take the copies of stage t + NS.
  auto step = [&](int t, auto IDX) __attribute__((always_inline)) {
    read(stage_of(IDX), I1{});
    multiply(I0{});
    __builtin_amdgcn_s_waitcnt(0x0070 | (AHEAD & 15) | ((AHEAD >> 4) << 14));     // vmcnt(AHEAD) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read(stage_of(std::integral_constant<int, decltype(IDX)::value + 1>{}), I0{});
    copies(t + NS, stage_of(IDX));
    multiply(I1{});
    const int now = first + t;
    if (++in_span == per || now == last) {          // a span ends
      const bool take = now <= last && (KG == 1 || span_at < F32_SPANS / 2);
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) {
          if (KG > 1 && kg == 1) {
            if (take) spans[((span_at * FN + i) * FM + j) * 256 + tid] = acc[i][j];
          } else if (take) {
            sum[i][j] += acc[i][j];
          }
          acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
      in_span = 0;
      ++span_at;
    }
  };
  int t = 0;
  for (; t + NS <= stages; t += NS) {
    step(t, I0{});
    step(t + 1, I1{});
    step(t + 2, I2{});
    if constexpr (NS > 3) step(t + 3, I3{});
  }
  if (t < stages) {
    step(t, I0{});
    if (t + 1 < stages) {
      step(t + 1, I1{});
      if constexpr (NS > 3)
        if (t + 2 < stages) step(t + 2, I2{});
    }
  }
  // nothing may still be on its way into LDS when the workgroup ends
  __builtin_amdgcn_s_waitcnt(0x0f70);       // vmcnt(0)
  if constexpr (KG > 1) {
    __syncthreads();
    if (kg == 1) return;
    const int more = (steps - F32_SPANS / 2 * per + per - 1) / per;      // spans the second group has (none: < 1)
    for (int s = 0; s < more; ++s)
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) sum[i][j] += spans[((s * FN + i) * FM + j) * 256 + tid];
  }
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      const int m = m0 + wm + 16 * j + r, n = n0 + wn + 16 * i + 4 * g;
      if (m < M) f32_store4<float, ACC>(C, m, n, N, true, sum[i][j]);
    }
#endif
}

// Whether the streaming kernel keeps two steps in flight: not in spans of one step, not where the outputs are so
// many that more waves a CU do as well, and of few rows not where they are one and a half workgroups of 16 a CU or
// two.  Measured, us, one step / two: 1 row into 1024 over 1024 6.1 / 5.2, over 4096 17.7 / 12.0, into 16384 over 4096
// 53.8 / 51.0, into 65536 over 256 13.6 / 15.4, over 1024 49.7 / 49.7; 17 into 6144 over 4096 43.9 / 40.8, into
// 16384 over 320 9.0 / 9.2, into 32768 over 256 12.8 / 14.4, over 320 16.0 / 17.1, over 1024 44.8 / 44.7; 1 into 6144
// over 768 6.7 / 7.2, over 2048 15.8 / 15.3, 16 over 768 8.5 / 8.4.  Of rows that are not aligned, number by number,
// only into few outputs over a long K: 4 into 4096 over 541 6.9 / 7.6, over 1743 20.5 / 18.6.
static bool f32_two_sets(int M, int N, int K, bool vec) {
  if (K <= 256 || N >= (M <= 16 ? 65536 : 24576)) return false;
  if (!vec) return N <= 4096 && K > 1280;
  return M > 8 || N <= 4096 || N > 8192 || K >= 2048;
}

template <typename TO, bool ACC, bool VEC>
static void launch_f32(const float* A, const float* W, TO* C, int M, int N, int K, bool vec_out,
                       hipStream_t stream) {
  const int span = f32_span(K);
#define F32_STREAM(RG, MT, SETS)                                                                 \
  hipLaunchKernelGGL((gemm_f32_stream_kernel<TO, ACC, RG, MT, VEC, SETS>),                       \
                     dim3((N + 16 * RG - 1) / (16 * RG), (M + 16 * MT - 1) / (16 * MT)),         \
                     dim3(F32_SPANS * 64), 0, stream, A, W, C, M, N, K, span, vec_out)
#define F32_TILE(B, ST)                                                                          \
  hipLaunchKernelGGL((gemm_f32_tile_kernel<TO, ACC, B, ST, VEC>), dim3((N + B - 1) / B,              \
                     (M + B - 1) / B), dim3(256), 0, stream, A, W, C, M, N, K, span, vec_out)
  const auto tiles = [&](int b) { return (long long)((M + b - 1) / b) * ((N + b - 1) / b); };
  if (M <= 16) {
    const bool two = f32_two_sets(M, N, K, VEC);
    if (N >= 16384) {
      if (two) F32_STREAM(2, 1, 2); else F32_STREAM(2, 1, 1);
    } else {
      if (two) F32_STREAM(1, 1, 2); else F32_STREAM(1, 1, 1);
    }
  } else if (M <= 32) {
    if (f32_two_sets(M, N, K, VEC)) F32_STREAM(1, 2, 2); else F32_STREAM(1, 2, 1);
  } else if (M <= 64) {
    F32_STREAM(1, 4, 1);
  } else if (VEC && std::is_same<TO, float>::value && vec_out && K > 0 && K % 32 == 0 &&
             (K > 32 || tiles(32) <= 768)) {
    // Up to three tiles of 32 x 32 a CU those, from K = 768 on (1024 where they are more than two) with two
    // groups of waves (us, one group / two: 65 rows into 2048 over 256 4.5 / 5.3, over 512 6.4 / 6.4, over 1024
    // 9.7 / 8.7; 152 into 4096 over 512 11.2 / 12.7, over 1024 19.0 / 19.1; 131 over 1024, 640 tiles, so 17.1,
    // 32 x 64 20.6); behind that 32 x 64 (256 rows, 1024 tiles, 21.9 and 21.0), and 64 x 64 where those are many
    // and K long (1024 rows into 7168 over 2048 237 us, 32 x 64 245; 2048 into 6144 over 1024 209 and 203) or
    // they are very many (2000 into 32768 over 64 124, 32 x 64 141).  One step of 32 over more tiles leaves a
    // ring nothing to run ahead of: the tiles below (2000 into 32768 91 us, 32 x 64 here 114).
#define F32_RING(BM, BN, KG)                                                                   \
  hipLaunchKernelGGL((gemm_f32_ring_kernel<BM, BN, KG, ACC>),                                  \
                     dim3(((N + BN - 1) / BN) * ((M + BM - 1) / BM)), dim3(256 * KG), 0, stream, A, W, \
                     (float*)C, M, N, K, span, (M + BM - 1) / BM, (N + BN - 1) / BN)
    if (tiles(32) <= 768 && K >= (tiles(32) <= 512 ? 768 : 1024)) F32_RING(32, 32, 2);
    else if (tiles(32) <= 768) F32_RING(32, 32, 1);
    else if (tiles(64) >= (K >= 2048 ? 1024 : 8192)) F32_RING(64, 64, 1);
    else F32_RING(32, 64, 1);
#undef F32_RING
  } else if (tiles(128) >= 256) {
    F32_TILE(128, 1);
  } else if (tiles(64) > 512) {
    F32_TILE(64, 1);
  } else if (tiles(64) >= 256) {
    F32_TILE(64, 2);
  } else {
    F32_TILE(32, 4);
  }
#undef F32_STREAM
#undef F32_TILE
}

// out = A W^T (accumulate: out += A W^T); A and W float32, out float32 or bfloat16; any sizes,
// any alignment of the elements
extern "C" int zf_gemm_f32(const void* A, const void* W, void* C, int c_dtype, int M, int N, int K,
                           int accumulate, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K < 0 || (c_dtype != ZF_F32 && c_dtype != ZF_BF16)) return -1;
  const bool vec = K % 4 == 0 && ((uintptr_t)A | (uintptr_t)W) % 16 == 0;
  const bool vec_out = N % 4 == 0 && (uintptr_t)C % 16 == 0;
  const float *a = (const float*)A, *w = (const float*)W;
#define F32_GO(TO, ACC)                                                            \
  do {                                                                             \
    if (vec) launch_f32<TO, ACC, true>(a, w, (TO*)C, M, N, K, vec_out, stream);    \
    else launch_f32<TO, ACC, false>(a, w, (TO*)C, M, N, K, vec_out, stream);       \
  } while (0)
  if (c_dtype == ZF_F32) {
    if (accumulate) F32_GO(float, true); else F32_GO(float, false);
  } else {
    if (accumulate) return -1;
    F32_GO(bf16_t, false);
  }
#undef F32_GO
  ZF_CHECK_LAUNCH();
}

// out [M, I] = silu(A Wg^T) * (A Wu^T) of W [2 I, K], the gate's rows before the up projection's; up
// to 16 rows, float32 throughout, any sizes and alignment of the elements.
extern "C" int zf_gemm_f32_swiglu(const float* A, const float* W, float* C, int M, int I, int K,
                                  hipStream_t stream) {
  if (M <= 0 || I <= 0) return 0;
  if (M > 16 || K < 0) return -1;
  const bool vec = K % 4 == 0 && ((uintptr_t)A | (uintptr_t)W) % 16 == 0;
  const bool vec_out = I % 4 == 0 && (uintptr_t)C % 16 == 0;
  const dim3 grid((I + 15) / 16);
#define F32_GLU(VEC, SETS)                                                                             \
  hipLaunchKernelGGL((gemm_f32_stream_kernel<float, false, 2, 1, VEC, SETS, true>), grid,              \
                     dim3(F32_SPANS * 64), 0, stream, A, W, C, M, I, K, f32_span(K), vec_out)
  const bool two = K > 256;       // (1 row, 3072 pairs over 1024 10.4 us, so 9.2; 24576 over 256 11.9, 14.8)
  if (vec) {
    if (two) F32_GLU(true, 2); else F32_GLU(true, 1);
  } else {
    if (two) F32_GLU(false, 2); else F32_GLU(false, 1);
  }
#undef F32_GLU
  ZF_CHECK_LAUNCH();
}

#define EPI_STORE_BF16 0
#define EPI_STORE_F32 1
#define EPI_ACC_F32 2
// SwiGLU fused into the product: the rows of W alternate in groups of 16 between the gate
// and the up projection (gate 0..15, up 0..15, gate 16..31, ...); the output is
// silu(gate) * up as bfloat16 [M, N / 2]  (a_j = g_j / (1 + exp(-g_j)) * u_j, cpu.zig:130-147)
#define EPI_SWIGLU 3

// the same with the tanh form of gelu and a bias a row of W (float32 [N] in W's order, or null):
// gelu(gate + b_gate) * (up + b_up)
#define EPI_GEGLU 4
// an activation on the bfloat16 that EPI_STORE_BF16 would store, stored as bfloat16 (up to 16 tokens)
#define EPI_ACT 5
// bfloat16, float32 or an activation on the bfloat16, as SkinnyNorm::act says
#define EPI_MANY 6
#define MANY_BF16 -1
#define MANY_F32 -2
#define EPI_GLU(E) ((E) == EPI_SWIGLU || (E) == EPI_GEGLU)

__device__ __forceinline__ float swiglu_f(float g, float u) { return g / (1.0f + expf(-g)) * u; }
// gelu(g) = g / 2 (1 + tanh(v)), the tanh through one exponential: 1 - 2 / (e^2v + 1)
__device__ __forceinline__ float geglu_f(float g, float u) {
  const float v = 0.79788456080286535588f * (g + 0.044715f * g * g * g);
  const float e = __builtin_amdgcn_exp2f(v * 2.8853900817779268f);
  return g * (1.0f - __builtin_amdgcn_rcpf(e + 1.0f)) * u;
}
template <int EPI> __device__ __forceinline__ float glu_f(float g, float u) {
  return EPI == EPI_GEGLU ? geglu_f(g, u) : swiglu_f(g, u);
}

// ---------------------------------------------------------------- large M: LDS-tiled
// Block tile BM x BN x 64, waves laid out (BM/WM) x (BN/WN), each wave WM x WN through
// 32x32x16 MFMAs.  Tiles are staged through LDS with rows padded to 72 elements (144 bytes)
// so that the 16-byte operand reads of 8 neighbouring rows fall on distinct banks; the next
// tile's global loads are in flight while the current one is multiplied.
#define TK 64
#define LDS_ROW 72

// Pre-tiled weights (WT): W is stored as [N / 16][K / 64][2][64][8]: the 16 rows x 64 k of a
// tile lie together (2 KB) in the order in which the lanes of a 16x16x32 MFMA pair consume
// them (chunk c of lane l = 16 g + r holds row r, k = 16 g + 8 c .. + 8), so that one wave
// load of the weight-streaming kernel is 1 KB of consecutive memory.  This kernel reads the
// same layout 16 bytes at a time.
__device__ __forceinline__ size_t tiled_offset(int n, int k, int K) {
  const int kk = k % 64;
  return ((size_t)(n / 16) * (K / 64) + k / 64) * 1024 + ((kk % 16) / 8) * 512 +
         ((kk / 16) * 16 + n % 16) * 8 + kk % 8;
}

template <int BM, int BN, int WM, int WN, int EPI, bool WT>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void gemm_bf16_tile_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ Cv, int M,
    int N, int K, int tiles_m, int tiles_n) {
  constexpr int NWM = BM / WM, NWN = BN / WN;
  constexpr int NT = NWM * NWN * 64;
  constexpr int FM = WM / 32, FN = WN / 32;
  constexpr int A_CHUNKS = BM * 8 / NT;   // 16-byte chunks per thread per tile
  constexpr int B_CHUNKS = BN * 8 / NT;
  static_assert(BM * 8 % NT == 0 && BN * 8 % NT == 0, "tile does not divide over the threads");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  bf16_t* lds = (bf16_t*)lds_raw;
  // stage s: A at s*(BM+BN)*LDS_ROW, W after it
  constexpr int STAGE = (BM + BN) * LDS_ROW;

  int tm, tn;
  tile_of_workgroup<(BM >= 128 ? 8 : 1024 / BM)>(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  const int tid = threadIdx.x;
  const int wave = tid / 64, lane = tid % 64;
  const int wm = wave / NWN, wn = wave % NWN;

  f32x16_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  u32x4_t areg[A_CHUNKS], breg[B_CHUNKS];

  // which 16 bytes of the W tile a thread moves: (row of the tile, k offset).  Plain layout:
  // 8 consecutive threads take the 8 chunks of a row.  Pre-tiled: 128 consecutive threads
  // take the 128 chunks of a 16-row group in the order they lie in memory (chunk p = 64 c +
  // 16 g + r holds row r, k = 16 g + 8 c), so their loads are consecutive 16-byte pieces.
  auto b_chunk = [&](int chunk, int& row, int& kc) {
    if (WT) {
      const int p = chunk % 128;
      row = (chunk / 128) * 16 + p % 16;
      kc = ((p % 64) / 16) * 16 + (p / 64) * 8;
    } else {
      row = chunk / 8;
      kc = (chunk % 8) * 8;
    }
  };

  auto gload = [&](int k0) {
#pragma unroll
    for (int c = 0; c < A_CHUNKS; ++c) {
      const int chunk = tid + c * NT;
      const int row = chunk / 8, kc = (chunk % 8) * 8;
      const int m = min(m0 + row, M - 1);
      if (k0 + kc < K)
        areg[c] = *(const u32x4_t*)(A + (size_t)m * K + k0 + kc);
      else
        areg[c] = u32x4_t{0, 0, 0, 0};
    }
#pragma unroll
    for (int c = 0; c < B_CHUNKS; ++c) {
      int row, kc;
      b_chunk(tid + c * NT, row, kc);
      const int n = min(n0 + row, N - 1);
      if (k0 + kc < K)
        breg[c] = *(const u32x4_t*)(W + (WT ? tiled_offset(n, k0 + kc, K)
                                            : (size_t)n * K + k0 + kc));
      else
        breg[c] = u32x4_t{0, 0, 0, 0};
    }
  };
  auto lstore = [&](int stage) {
    bf16_t* a_s = lds + stage * STAGE;
    bf16_t* b_s = a_s + BM * LDS_ROW;
#pragma unroll
    for (int c = 0; c < A_CHUNKS; ++c) {
      const int chunk = tid + c * NT;
      const int row = chunk / 8, kc = (chunk % 8) * 8;
      *(u32x4_t*)(a_s + row * LDS_ROW + kc) = areg[c];
    }
#pragma unroll
    for (int c = 0; c < B_CHUNKS; ++c) {
      int row, kc;
      b_chunk(tid + c * NT, row, kc);
      *(u32x4_t*)(b_s + row * LDS_ROW + kc) = breg[c];
    }
  };

  const int ktiles = (K + TK - 1) / TK;
  gload(0);
  lstore(0);
  __syncthreads();
  for (int kt = 0; kt < ktiles; ++kt) {
    const int stage = kt & 1;
    if (kt + 1 < ktiles) gload((kt + 1) * TK);
    const bf16_t* a_s = lds + stage * STAGE + (wm * WM) * LDS_ROW;
    const bf16_t* b_s = lds + stage * STAGE + BM * LDS_ROW + (wn * WN) * LDS_ROW;
#pragma unroll
    for (int ks = 0; ks < TK / 16; ++ks) {
      bf16x8_t af[FM], bfr[FN];
      const int koff = ks * 16 + (lane / 32) * 8;
#pragma unroll
      for (int i = 0; i < FM; ++i)
        af[i] = *(const bf16x8_t*)(a_s + (i * 32 + lane % 32) * LDS_ROW + koff);
#pragma unroll
      for (int j = 0; j < FN; ++j)
        bfr[j] = *(const bf16x8_t*)(b_s + (j * 32 + lane % 32) * LDS_ROW + koff);
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[i], bfr[j], acc[i][j], 0, 0, 0);
    }
    if (kt + 1 < ktiles) lstore(stage ^ 1);
    __syncthreads();
  }

  // D[i][j] of a 32x32 block: j = lane % 32, i = 8 * (r / 4) + 4 * (lane / 32) + r % 4
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int n = n0 + wn * WN + j * 32 + lane % 32;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + wm * WM + i * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4;
        if (EPI == EPI_SWIGLU) {
          // columns 0..15 of the 32-wide block are gate, 16..31 the matching up columns
          const float other = __shfl_xor(acc[i][j][r], 16, 64);
          if (lane % 32 < 16 && m < M && n < N)
            ((bf16_t*)Cv)[(size_t)m * (N / 2) + (n / 32) * 16 + n % 16] =
                float_to_bf16(swiglu_f(acc[i][j][r], other));
          continue;
        }
        if (m < M && n < N) {
          const size_t off = (size_t)m * N + n;
          if (EPI == EPI_STORE_BF16)
            ((bf16_t*)Cv)[off] = float_to_bf16(acc[i][j][r]);
          else if (EPI == EPI_STORE_F32)
            ((float*)Cv)[off] = acc[i][j][r];
          else
            ((float*)Cv)[off] += acc[i][j][r];
        }
      }
    }
}

__device__ __forceinline__ float4 sum4(const float4& a, const float4& b) {
  return float4{a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w};
}

// Epilogue through LDS of the kernels whose waves hold 32-row x 32-column MFMA results: a
// 32x32 result has a lane's 16 values in 16 different rows, so direct stores would be 2 or 4
// bytes wide in runs of 64 bytes.  Each wave lays 32 rows of WN columns of its tile (rows mw.., columns
// nw..) down in its own slab (32 rows of WN + 4 floats) and reads them back along the rows, 16
// bytes per lane.  All waves of the workgroup call it together.
template <int FM, int FN, int WN, int EPI>
__device__ __forceinline__ void store_through_slab(f32x16_t (&acc)[FM][FN], float* slab, int mw,
                                                   int nw, int M, int N, void* Cv, int lane,
                                                   const float* glu_bias = nullptr) {
  static_assert(WN == 32 * FN, "column blocks");
  constexpr int SLAB_ROW = WN + 4;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        slab[(8 * (r / 4) + 4 * (lane / 32) + r % 4) * SLAB_ROW + j * 32 + lane % 32] = acc[i][j][r];
    __syncthreads();
    if (EPI_GLU(EPI)) {
      // 16 gate columns, then the 16 up columns that belong to them: 8 outputs per lane
      constexpr int LPR = WN / 16;                  // lanes per row
#pragma unroll
      for (int it = 0; it < 32 * LPR / 64; ++it) {
        const int row = it * (64 / LPR) + lane / LPR, q = lane % LPR;
        const int m = mw + i * 32 + row;
        const int c = (q / 2) * 32 + (q % 2) * 8;   // first gate column inside the wave's tile
        const int n = nw + c;
        if (m < M && n < N) {
          const float* src = slab + row * SLAB_ROW + c;
          float4 g0 = *(const float4*)src, g1 = *(const float4*)(src + 4);
          float4 u0 = *(const float4*)(src + 16), u1 = *(const float4*)(src + 20);
          if (EPI == EPI_GEGLU && glu_bias != nullptr) {
            g0 = sum4(g0, *(const float4*)(glu_bias + n));
            g1 = sum4(g1, *(const float4*)(glu_bias + n + 4));
            u0 = sum4(u0, *(const float4*)(glu_bias + n + 16));
            u1 = sum4(u1, *(const float4*)(glu_bias + n + 20));
          }
          const u32x4_t v = u32x4_t{
              pack_bf16x2(glu_f<EPI>(g0.x, u0.x), glu_f<EPI>(g0.y, u0.y)),
              pack_bf16x2(glu_f<EPI>(g0.z, u0.z), glu_f<EPI>(g0.w, u0.w)),
              pack_bf16x2(glu_f<EPI>(g1.x, u1.x), glu_f<EPI>(g1.y, u1.y)),
              pack_bf16x2(glu_f<EPI>(g1.z, u1.z), glu_f<EPI>(g1.w, u1.w))};
          *(u32x4_t*)((bf16_t*)Cv + (size_t)m * (N / 2) + (n / 32) * 16 + (n % 32)) = v;
        }
      }
    } else if (EPI == EPI_STORE_BF16) {
      constexpr int LPR = WN / 8;
#pragma unroll
      for (int it = 0; it < 32 * LPR / 64; ++it) {
        const int row = it * (64 / LPR) + lane / LPR, c = (lane % LPR) * 8;
        const int m = mw + i * 32 + row, n = nw + c;
        if (m < M && n < N) {
          const float* src = slab + row * SLAB_ROW + c;
          const float4 x0 = *(const float4*)src, x1 = *(const float4*)(src + 4);
          const u32x4_t v = u32x4_t{pack_bf16x2(x0.x, x0.y), pack_bf16x2(x0.z, x0.w),
                                    pack_bf16x2(x1.x, x1.y), pack_bf16x2(x1.z, x1.w)};
          *(u32x4_t*)((bf16_t*)Cv + (size_t)m * N + n) = v;
        }
      }
    } else {
      constexpr int LPR = WN / 4;
#pragma unroll
      for (int it = 0; it < 32 * LPR / 64; ++it) {
        const int row = it * (64 / LPR) + lane / LPR, c = (lane % LPR) * 4;
        const int m = mw + i * 32 + row, n = nw + c;
        if (m < M && n < N) {
          float4 x = *(const float4*)(slab + row * SLAB_ROW + c);
          float4* dst = (float4*)((float*)Cv + (size_t)m * N + n);
          if (EPI == EPI_ACC_F32) {
            const float4 old = *dst;
            x = float4{old.x + x.x, old.y + x.y, old.z + x.z, old.w + x.w};
          }
          *dst = x;
        }
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------- large M, pre-tiled W: W not staged
// Tiles of BM tokens x BN outputs, k-tiles of TKM.  Only the tokens go through LDS; every wave
// takes its W operands straight from the pre-tiled matrix (16-byte pieces that lie in runs of
// 256 bytes), one k-tile ahead in registers.  That halves the LDS traffic per MFMA against
// the kernel above, whose LDS is as busy as its MFMAs.  With the waves side by side along the
// outputs (WM == BM) no two of them load the same part of W.
// ADMA: the tokens' k-tiles go from memory into LDS by direct-to-LDS loads (a wave instruction
// copies 64 x 16 bytes to one LDS address + 16 bytes a lane), not through registers: no
// registers hold them on the way, and the stores into LDS and their waits are gone (1 to 2 %
// at 2048 and 8192 tokens).  Such a copy lands as consecutive bytes, so instead of padded rows
// the 16-byte pieces of a row are permuted (piece c of row r lies at place c ^ ((r >> 1) & 7)
// of its 128 bytes): the 16 rows a quarter wave reads then fall into 16 different groups of
// banks.  Two stages in two arrays, so that the compiler knows which reads wait for which
// copies; the barrier is a bare s_barrier behind a wait that lets the W loads issued since
// (younger than the copies) stay in flight.
// TAIL: the tiles beyond the last whole round of the chip (the tile order's last `tail` ones)
// are shared by tail_split workgroups each, along K: workgroups [whole, whole + tail *
// tail_split) of the grid, which leave float32 partials [tail][tail_split][BM][BN] in tail_ws
// for tile_tail_reduce_kernel; a short last round then takes 1 / tail_split of a tile's time
// instead of a whole one.
// KG == 2: two groups of waves in one workgroup, each the whole tile over half of the
// workgroup's k-tiles (its own stages in LDS, its own W), for products whose tiles are so few
// that a CU holds one workgroup: twice the waves to hide a load behind, and no more traffic
// than one group has.  At the end each group hands one of its two column blocks to the other
// through LDS (half the tile's rows at a time), adds what it is handed (first half of K plus
// second half, whichever group adds) and stores the block it kept.
template <int BM, int BN, int WM, int WN, int EPI, int TKM = TK, bool W2 = false,
          bool ADMA = false, bool TAIL = false, int KG = 1>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64 * KG) void gemm_bf16_tile_wdirect_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ Cv, int M,
    int N, int K, int tiles_m, int tiles_n, int whole, int tail_split,
    float* __restrict__ tail_ws, const float* __restrict__ glu_bias) {
  // (the host pass, which only needs the launch stub, does not know the buffer descriptor type)
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NWN = BN / WN, NT = (BM / WM) * NWN * 64;       // (NT: the threads of a group)
  constexpr int FM = WM / 32, FN = WN / 32;
  constexpr int LROW = TKM + 8, KCH = TKM / 8;      // LDS row in elements; 16-byte chunks per row
  static_assert(BM * KCH % NT == 0 && TKM % 64 == 0, "tile does not divide over the threads");
  static_assert(KG == 1 || (KG == 2 && ADMA && !TAIL && FN == 2 && FM % 2 == 0),
                "two groups: tokens copied straight into LDS, two column blocks a wave");
  constexpr int A_CHUNKS = BM * KCH / NT;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  bf16_t* lds = (bf16_t*)lds_raw;       // two stages of BM rows of LROW elements

  // which tile, and which of how many parts of its k-tiles
  int tile = blockIdx.x, kpart = blockIdx.y, kparts = gridDim.y;
  bool in_tail = false;
  if constexpr (TAIL) {
    if ((int)blockIdx.x >= whole) {
      in_tail = true;
      tile = whole + ((int)blockIdx.x - whole) / tail_split;
      kpart = ((int)blockIdx.x - whole) % tail_split;
      kparts = tail_split;
    }
  }
  int tm, tn;
  tile_of_workgroup<(BM >= 128 ? 8 : 1024 / BM)>(tile, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  // (a group's threads count from 0: what follows is one group's view)
  const int kgrp = KG > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / NT) : 0;
  const int tid = KG > 1 ? (int)threadIdx.x % NT : (int)threadIdx.x;
  if (KG > 1) {
    kpart = kpart * KG + kgrp;
    kparts *= KG;
  }
  const int wave = tid / 64, lane = tid % 64;
  const int wm = wave / NWN, wn = wave % NWN;

  f32x16_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  // W operand of MFMA (j, ks): column n = n0 + wn * WN + 32 j + lane % 32, k = 16 ks +
  // 8 (lane / 32) .. + 8 of the k-tile: piece 64 (lane / 32) + 16 ks + n % 16 of the 16-row
  // group n / 16.  Groups beyond N are clamped (their columns are never stored).
  // (loaded through a buffer descriptor on the tile's first group: a 32-bit offset per lane
  // and one all lanes share instead of a 64-bit address per lane, which issues faster and
  // needs no address arithmetic)
  const int grp0 = min(n0 / 16, N / 16 - 1);
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(W + (size_t)grp0 * (K / 64) * 1024), 0, 0x7fffffff, 0x00020000);
  uint32_t wbase[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int n = n0 + wn * WN + j * 32 + lane % 32;
    const int grp = min(n / 16, N / 16 - 1) - grp0;
    wbase[j] = ((uint32_t)grp * (uint32_t)(K / 64) * 1024 + ((lane / 32) * 64 + n % 16) * 8) * 2;
  }
  u32x4_t wreg[W2 ? 2 : 1][TKM / 16][FN];
  auto gload_w = [&](auto BUF, int kt, int ks) {
    constexpr int B = decltype(BUF)::value;
    const uint32_t at = ((uint32_t)kt * (TKM / 64) + ks / 4) * 2048 + (ks % 4) * 256;
#pragma unroll
    for (int j = 0; j < FN; ++j)
      wreg[B][ks][j] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, wbase[j], at, 0);
  };
  // gridDim.y workgroups share a tile's k-tiles (split-K for products with few tiles); each
  // then leaves a float32 partial [gridDim.y, M, N] in Cv for skinny_reduce_kernel
  const int kt_all = K / TKM;
  const int kt0 = (int)((long long)kpart * kt_all / kparts);
  const int ktiles = (int)((long long)(kpart + 1) * kt_all / kparts);
  if (gridDim.y > 1) Cv = (float*)Cv + (size_t)blockIdx.y * M * N;
  using Buf0 = std::integral_constant<int, 0>;
  using Buf1 = std::integral_constant<int, 1>;

  if constexpr (ADMA) {
    static_assert(TKM == 64, "direct-to-LDS tokens: k-tiles of 64 (rows of 8 pieces)");
    __shared__ u32x4_t a_stages0[KG * BM * 8];
    __shared__ u32x4_t a_stages1[KG * BM * 8];
    u32x4_t* const a_stage0 = a_stages0 + kgrp * (BM * 8);
    u32x4_t* const a_stage1 = a_stages1 + kgrp * (BM * 8);
    // the places this thread fills: place p = tid + c NT is row p / 8, slot p % 8, and takes
    // piece slot ^ ((row >> 1) & 7) of the row's 128 bytes (rows beyond M: the last row)
    uint32_t asrc[A_CHUNKS];
#pragma unroll
    for (int c = 0; c < A_CHUNKS; ++c) {
      const int p = tid + c * NT, row = p / 8, piece = (p % 8) ^ ((row >> 1) & 7);
      asrc[c] = (uint32_t)(min(m0 + row, M - 1) - m0) * (uint32_t)K + piece * 8;
    }
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(A + (size_t)m0 * K), 0, 0x7fffffff, 0x00020000);
    const int wave_u = __builtin_amdgcn_readfirstlane(wave);      // the LDS address is a scalar
    auto dma_a = [&](int k0, u32x4_t* stage) {
#pragma unroll
      for (int c = 0; c < A_CHUNKS; ++c)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            a_rsrc, (__attribute__((address_space(3))) void*)(stage + (wave_u * 64 + c * NT)), 16,
            asrc[c] * 2, (uint32_t)k0 * 2, 0, 0);
    };
    // the operand of MFMA row block i, k-step ks: row 32 i + lane % 32, piece 2 ks + lane / 32
    int a_at[TKM / 16];
#pragma unroll
    for (int ks = 0; ks < TKM / 16; ++ks)
      a_at[ks] = (wm * WM + lane % 32) * 8 + ((2 * ks + lane / 32) ^ (((lane % 32) >> 1) & 7));
    // (in this order, kept by the scheduling barriers: the first step's wait counts on it)
    dma_a(kt0 * TKM, a_stage0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < TKM / 16; ++ks) gload_w(Buf0{}, kt0, ks);
    __builtin_amdgcn_sched_barrier(0);
    if (W2) {
#pragma unroll
      for (int ks = 0; ks < TKM / 16; ++ks) gload_w(Buf1{}, min(kt0 + 1, ktiles - 1), ks);
      __builtin_amdgcn_sched_barrier(0);
    }
    // Before a step: its tokens' copies have landed (the last of them is older than the 6 W
    // loads of the step before that were issued behind it, which may stay in flight), then
    // all waves meet: every wave has also read its last operands out of the other stage.
    static_assert(FN == 2 && TKM == 64 && A_CHUNKS == 4, "the wait counts the loads behind the last copy");
    auto meet = [&]() {
      __builtin_amdgcn_s_waitcnt(0x0f76);     // vmcnt(6)
      __builtin_amdgcn_s_barrier();
    };
    // A k-step's MFMAs run output block by output block, so that a W register is free after
    // the first FM of them.  What else a wave issues follows single MFMAs: the next k-step's
    // FM operand reads behind the first FM MFMAs, then (k-steps 0 and 1) two of the next
    // tile's four copies, then the two W loads that refill this k-step's registers, the
    // second behind the last MFMA.  (All copies in one place hold the wave, and with it its
    // MFMAs, while the CU's one path to memory takes them one by one.)
    auto step = [&](int kt, const u32x4_t* cur, u32x4_t* other, auto BUF) {
      constexpr int B = decltype(BUF)::value;
      meet();
      const int wnxt = min(kt + (W2 ? 2 : 1), ktiles - 1);
      const uint32_t next_k0 = (uint32_t)min(kt + 1, ktiles - 1) * TKM * 2;
      __builtin_amdgcn_sched_barrier(0);
      u32x4_t af[2][FM];
#pragma unroll
      for (int i = 0; i < FM; ++i) af[0][i] = cur[a_at[0] + i * 256];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const uint32_t w_at = ((uint32_t)wnxt * (TKM / 64) + ks / 4) * 2048 + (ks % 4) * 256;
#pragma unroll
        for (int m = 0; m < 2 * FM; ++m) {
          const int j = m / FM, i = m % FM;
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              *(const bf16x8_t*)&af[ks % 2][i], *(const bf16x8_t*)&wreg[B][ks][j], acc[i][j],
              0, 0, 0);
          if (m < FM && ks < 3) af[(ks + 1) % 2][m] = cur[a_at[ks + 1] + m * 256];
          // copies 2 ks and 2 ks + 1 of the four: behind the first two MFMAs of the second block
          if (ks < 2 && (m == FM || (FM > 2 && m == FM + 1))) {
            const int c0 = 2 * ks + (FM == 2 ? 0 : m - FM), c1 = FM == 2 ? c0 + 2 : c0 + 1;
#pragma unroll
            for (int c = c0; c < c1; ++c)
              __builtin_amdgcn_raw_ptr_buffer_load_lds(
                  a_rsrc, (__attribute__((address_space(3))) void*)(other + (wave_u * 64 + c * NT)),
                  16, asrc[c] * 2, next_k0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);      // (older than the W loads that follow)
          }
          if (m == 2 * FM - 2) wreg[B][ks][0] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, wbase[0], w_at, 0);
          if (m == 2 * FM - 1) wreg[B][ks][1] = __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, wbase[1], w_at, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    if (W2) {       // an even number of k-tiles (the launch sees to it)
      for (int kt = kt0; kt < ktiles; kt += 2) {
        step(kt, a_stage0, a_stage1, Buf0{});
        step(kt + 1, a_stage1, a_stage0, Buf1{});
      }
    } else {
      int kt = kt0;
      for (; kt + 1 < ktiles; kt += 2) {
        step(kt, a_stage0, a_stage1, Buf0{});
        step(kt + 1, a_stage1, a_stage0, Buf0{});
      }
      if (kt < ktiles) step(kt, a_stage0, a_stage1, Buf0{});
    }
    // the last step copied its own tile once more: nothing may still be on its way into LDS
    // when the workgroup ends
    __builtin_amdgcn_s_waitcnt(0x0f70);       // vmcnt(0)
  } else {
  u32x4_t areg[A_CHUNKS];
  const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(A + (size_t)m0 * K), 0, 0x7fffffff, 0x00020000);
  uint32_t a_from[A_CHUNKS];
#pragma unroll
  for (int c = 0; c < A_CHUNKS; ++c) {
    const int chunk = tid + c * NT;
    const int row = chunk / KCH, kc = (chunk % KCH) * 8;
    a_from[c] = ((uint32_t)(min(m0 + row, M - 1) - m0) * (uint32_t)K + kc) * 2;
  }
  auto gload_a = [&](int k0) {
#pragma unroll
    for (int c = 0; c < A_CHUNKS; ++c)
      areg[c] = __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, a_from[c], (uint32_t)k0 * 2, 0);
  };
  auto lstore = [&](int stage) {
    bf16_t* a_s = lds + stage * BM * LROW;
#pragma unroll
    for (int c = 0; c < A_CHUNKS; ++c) {
      const int chunk = tid + c * NT;
      const int row = chunk / KCH, kc = (chunk % KCH) * 8;
      *(u32x4_t*)(a_s + row * LROW + kc) = areg[c];
    }
  };

  gload_a(kt0 * TKM);
#pragma unroll
  for (int ks = 0; ks < TKM / 16; ++ks) gload_w(Buf0{}, kt0, ks);
  if (W2) {
#pragma unroll
    for (int ks = 0; ks < TKM / 16; ++ks) gload_w(Buf1{}, min(kt0 + 1, ktiles - 1), ks);
  }
  lstore(0);
  __syncthreads();
  // One k-tile per step: MFMAs on LDS stage `stage`; meanwhile the tokens of tile kt + 1
  // travel through registers into the other stage, and every k-step's W registers are
  // refilled right after their last use with their part of tile kt + 1 (W2: of tile kt + 2,
  // from the other of two register sets, so that a miss in L2 has two k-tiles to arrive).
  // No branches around the loads (the last steps load their own tile once more), so the
  // compiler can count the loads in flight and waits for no younger one; the scheduling
  // barriers keep it from sinking the loads down to their first use, which would expose
  // their whole latency.
  auto step = [&](int kt, int stage, auto BUF) {
    constexpr int B = decltype(BUF)::value;
    const int nxt = min(kt + 1, ktiles - 1);
    const int wnxt = W2 ? min(kt + 2, ktiles - 1) : nxt;
    gload_a(nxt * TKM);
    __builtin_amdgcn_sched_barrier(0);
    const bf16_t* a_s = lds + stage * BM * LROW + (wm * WM) * LROW;
    // the token operands of k-step ks + 1 are read from LDS while the MFMAs of ks run
    bf16x8_t af[2][FM];
#pragma unroll
    for (int i = 0; i < FM; ++i)
      af[0][i] = *(const bf16x8_t*)(a_s + (i * 32 + lane % 32) * LROW + (lane / 32) * 8);
#pragma unroll
    for (int ks = 0; ks < TKM / 16; ++ks) {
      if (ks + 1 < TKM / 16) {
        const int koff = (ks + 1) * 16 + (lane / 32) * 8;
#pragma unroll
        for (int i = 0; i < FM; ++i)
          af[(ks + 1) % 2][i] = *(const bf16x8_t*)(a_s + (i * 32 + lane % 32) * LROW + koff);
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              af[ks % 2][i], *(const bf16x8_t*)&wreg[B][ks][j], acc[i][j], 0, 0, 0);
      gload_w(BUF, wnxt, ks);
      __builtin_amdgcn_sched_barrier(0);
    }
    lstore(stage ^ 1);
    __syncthreads();
  };
  if (W2) {       // an even number of k-tiles (the launch sees to it)
    for (int kt = kt0; kt < ktiles; kt += 2) {
      step(kt, 0, Buf0{});
      step(kt + 1, 1, Buf1{});
    }
  } else {
    for (int kt = kt0; kt < ktiles; ++kt) step(kt, (kt - kt0) & 1, Buf0{});
  }
  }

  // (the main loop's last barrier has freed the token stages; the launch sizes the LDS for
  // stages and slabs)
  if constexpr (KG == 2) {
    // Half the tile's rows at a time: every wave lays down the column block it gives away
    // (group 0 its second, group 1 its first) where its partner in the other group finds it.
    constexpr int HALF = FM / 2, PER_WAVE = HALF * 16 * 64;
    float* const xch = (float*)lds_raw;
    float* const mine = xch + (size_t)(kgrp * (NT / 64) + wave) * PER_WAVE;
    const float* const theirs = xch + (size_t)((1 - kgrp) * (NT / 64) + wave) * PER_WAVE;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      __syncthreads();          // (the round before has been read)
#pragma unroll
      for (int ii = 0; ii < HALF; ++ii)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int i = half * HALF + ii;
          mine[(ii * 16 + r) * 64 + lane] = kgrp == 0 ? acc[i][1][r] : acc[i][0][r];
        }
      __syncthreads();
#pragma unroll
      for (int ii = 0; ii < HALF; ++ii)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int i = half * HALF + ii;
          const float v = theirs[(ii * 16 + r) * 64 + lane];
          // kept block = first half of K + second half of K, in either group
          const float mine0 = acc[i][0][r], mine1 = acc[i][1][r];
          acc[i][0][r] = kgrp == 0 ? mine0 + v : mine0;
          acc[i][1][r] = kgrp == 0 ? mine1 : v + mine1;
        }
    }
    __syncthreads();            // the slabs lie where the blocks were handed over
    f32x16_t kept[FM][1];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) kept[i][0][r] = kgrp == 0 ? acc[i][0][r] : acc[i][1][r];
    float* slab32 = (float*)lds_raw + (size_t)(kgrp * (NT / 64) + wave) * 32 * (32 + 4);
    store_through_slab<FM, 1, 32, EPI>(kept, slab32, m0 + wm * WM, n0 + wn * WN + 32 * kgrp, M, N,
                                       Cv, lane, glu_bias);
    return;
  }
  float* slab = (float*)lds_raw + (size_t)wave * 32 * (WN + 4);
  if constexpr (TAIL) {
    if (in_tail) {      // (uniform over the workgroup) the whole tile as it is, rows beyond M too
      float* part = tail_ws + ((size_t)(tile - whole) * tail_split + kpart) * BM * BN;
      store_through_slab<FM, FN, WN, EPI_STORE_F32>(acc, slab, wm * WM, wn * WN, BM, BN, part, lane);
      return;
    }
  }
  store_through_slab<FM, FN, WN, EPI>(acc, slab, m0 + wm * WM, n0 + wn * WN, M, N, Cv, lane,
                                      glu_bias);
#endif
}

// The partials of the tiles that gemm_bf16_tile_wdirect_kernel<.., TAIL> split along K, added
// in split order, with the product's epilogue at the tile's place.  Grid (tail tiles, BM / 8):
// a workgroup takes 8 rows of a tile, a thread 8 columns of a row (SwiGLU: 4 gate columns and
// the 4 up columns that belong to them, which lie 16 further on).
template <int BM, int BN, int EPI>
__global__ __launch_bounds__(BN) void tile_tail_reduce_kernel(
    const float* __restrict__ ws, void* __restrict__ Cv, int M, int N, int tiles_m, int tiles_n,
    int whole, int split, const float* __restrict__ glu_bias) {
  static_assert(BN % 32 == 0 && BM % 8 == 0, "a row is BN / 8 threads");
  constexpr int TPR = BN / 8;                        // threads per row
  const int t = blockIdx.x;
  int tm, tn;
  tile_of_workgroup<(BM >= 128 ? 8 : 1024 / BM)>(whole + t, tiles_m, tiles_n, tm, tn);
  const int row = blockIdx.y * 8 + threadIdx.x / TPR, q = threadIdx.x % TPR;
  const int m = tm * BM + row;
  const int c0 = EPI_GLU(EPI) ? (q / 4) * 32 + (q % 4) * 4 : q * 8;
  const int c1 = EPI_GLU(EPI) ? c0 + 16 : c0 + 4;
  const int n = tn * BN + c0;
  if (m >= M || n >= N) return;
  const float* part = ws + ((size_t)t * split * BM + row) * BN;
  float4 x0 = float4{0.f, 0.f, 0.f, 0.f}, x1 = x0;
  for (int k = 0; k < split; ++k) {
    const float4 p0 = *(const float4*)(part + (size_t)k * BM * BN + c0);
    const float4 p1 = *(const float4*)(part + (size_t)k * BM * BN + c1);
    x0.x += p0.x; x0.y += p0.y; x0.z += p0.z; x0.w += p0.w;
    x1.x += p1.x; x1.y += p1.y; x1.z += p1.z; x1.w += p1.w;
  }
  if (EPI_GLU(EPI)) {
    if (EPI == EPI_GEGLU && glu_bias != nullptr) {
      x0 = sum4(x0, *(const float4*)(glu_bias + n));
      x1 = sum4(x1, *(const float4*)(glu_bias + n + 16));
    }
    const u32x2_t v = u32x2_t{pack_bf16x2(glu_f<EPI>(x0.x, x1.x), glu_f<EPI>(x0.y, x1.y)),
                              pack_bf16x2(glu_f<EPI>(x0.z, x1.z), glu_f<EPI>(x0.w, x1.w))};
    *(u32x2_t*)((bf16_t*)Cv + (size_t)m * (N / 2) + (n / 32) * 16 + (n % 32)) = v;
  } else if (EPI == EPI_STORE_BF16) {
    *(u32x4_t*)((bf16_t*)Cv + (size_t)m * N + n) =
        u32x4_t{pack_bf16x2(x0.x, x0.y), pack_bf16x2(x0.z, x0.w), pack_bf16x2(x1.x, x1.y),
                pack_bf16x2(x1.z, x1.w)};
  } else {
    float4* dst = (float4*)((float*)Cv + (size_t)m * N + n);
    if (EPI == EPI_ACC_F32) {
      const float4 o0 = dst[0], o1 = dst[1];
      x0 = float4{o0.x + x0.x, o0.y + x0.y, o0.z + x0.z, o0.w + x0.w};
      x1 = float4{o1.x + x1.x, o1.y + x1.y, o1.z + x1.z, o1.w + x1.w};
    }
    dst[0] = x0;
    dst[1] = x1;
  }
}

// ---------------------------------------------------------------- large M: 256-token tiles, one workgroup to a CU
// Tiles of 256 tokens x BN outputs (128, 192 or 256), one workgroup of 4 waves (2 x 2) per
// CU, each wave alone on its SIMD with a tile of 128 x BN / 2 (up to 256 accumulator
// registers).  The kernel above moves (BM + BN) / (BM * BN) bytes per flop from L2 through a
// CU's vector memory path, which at 128 x 256 tiles is as busy as the MFMAs; here it is half
// to two thirds of that.  Both operands go from memory into LDS by direct-to-LDS loads in
// k-tiles of 64: a row of tokens is then one whole line of 128 bytes (as pieces of 64 bytes, in
// k-tiles of 32, every line was fetched from L2 twice), its eight 16-byte pieces permuted
// (piece c of row r at place c ^ ((r >> 1) & 7): the 16 rows that an operand read takes fall into
// different groups of banks), W as it lies in the pre-tiled matrix.  The LDS holds two or three
// stages of either operand (separate arrays, so that the compiler knows which reads wait for
// which copies): two of the tokens and three of W at 256 outputs, all of the 160 KB.
// A tile is two k-steps of 32; the operands of the next k-step are read behind the MFMAs of
// the one before.  Between the two the wave waits for the copies of the next tile (those of W
// two tiles ahead stay in flight) and meets the others, which have then read all of this tile;
// the second k-step and the next tile's first one then issue the copies that take the places so
// freed.  A wave issues one instruction at a time, so what is not an MFMA follows single
// MFMAs, evenly spread.
// v_mfma_f32_16x16x32_bf16 and not 32x32x16: the chip's power is what large products run into
// on data that is not zeros, and with half the accumulator traffic a flop these take less of it;
// both add in the same order (the results are the same bits as those of the kernels above).
// W's rows are the first operand, so that a lane's four sums are four outputs of one token.
// Measured, weights from HBM, TFLOP/s, k-tiles of 32 in a ring of four with 32x32x16 -> k-tiles
// of 64 -> stages as here -> 16x16x32: 2048 tokens into 24576 over 4096 1290 -> 1349 -> 1351 -> 1390;
// 8192 into 51200 over 5120 1353 -> 1414 -> 1428 -> 1456; 8192 into 5120 over 25600 1207 -> 1195 ->
// 1333 -> 1355; on zeros, which power does not limit, 8192 into 24576 over 4096 1619 -> 1729 -> 2050 ->
// 1844.

// which of a k-step's cnt copies follows MFMA m of nm (-1: none): evenly spread
constexpr int copy_after(int m, int nm, int cnt) {
  for (int d = 0; d < cnt; ++d)
    if (m == (d + 1) * nm / cnt - 1) return d;
  return -1;
}
// how many of the nr operand reads have been issued before MFMA m: one behind every second MFMA
constexpr int reads_before(int m, int nr) { return (m + 1) / 2 < nr ? (m + 1) / 2 : nr; }

// What the kernels leave whose waves hold FM x FN blocks of 16 tokens x 16 outputs with W's rows as the
// first operand: lane 16 g + c has outputs 4 g .. 4 g + 3 of token c of a block; the wave's first
// token and output are mw and nw.  Two blocks of tokens at a time.
// (256 accumulators stay where the MFMAs left them until their block is stored: the compiler would take
// all of them into the other half of the registers ahead of the first branch, and where two epilogues
// follow spill 15 to 60.  Measured, us, without -> with: 4096 tokens into 5120 over 25600 added, its last round split,
// 769 -> 734, SwiGLU pairs of 2048 tokens into 24576 over 4096 291 -> 284, 8192 added into 4096 over 12288
// 575 -> 558, GEGLU pairs of 8192 into 51200 over 5120 2894 -> 2911.)
template <int FM, int FN>
__device__ __forceinline__ f32x4_t block_of(const f32x4_t& sums) {
  f32x4_t v = sums;
  if constexpr (FM * FN >= 64) asm volatile("" : "+a"(v));
  return v;
}
// float32: 16 bytes a lane as they are, 64 bytes of a row in a run.
template <int FM, int FN, bool ADD>
__device__ __forceinline__ void store_blocks_f32(const f32x4_t (&acc)[FM][FN], float* to, int mw, int nw, int M,
                                                 int N, int lane) {
  const int tok = lane % 16, n4 = 4 * (lane / 16);
#pragma unroll
  for (int i = 0; i < FM; i += 2) {
    f32x4_t old[2][FN];
#pragma unroll
    for (int ii = 0; ii < 2; ++ii) {
      const int m = mw + 16 * (i + ii) + tok;
      if constexpr (ADD)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          if (m < M && nw + 16 * j < N) old[ii][j] = *(const f32x4_t*)(to + (size_t)m * N + nw + 16 * j + n4);
    }
#pragma unroll
    for (int ii = 0; ii < 2; ++ii) {
      const int m = mw + 16 * (i + ii) + tok;
#pragma unroll
      for (int j = 0; j < FN; ++j)
        if (m < M && nw + 16 * j < N) {
          const f32x4_t v = block_of<FM, FN>(acc[i + ii][j]);
          *(f32x4_t*)(to + (size_t)m * N + nw + 16 * j + n4) = ADD ? old[ii][j] + v : v;
        }
    }
  }
}
// bfloat16: through a slab of the wave's own in LDS (16 bytes more a row than its outputs: the rows begin
// in different banks), which is then read along the rows.
template <int FN, int EPI>
__host__ __device__ constexpr int slab_places() {
  return 32 * ((EPI_GLU(EPI) ? FN * 8 : FN * 16) / 8 + 1);
}
template <int FM, int FN, int EPI>
__device__ __forceinline__ void store_blocks_bf16(const f32x4_t (&acc)[FM][FN], void* Cv, u32x4_t* slab, int mw,
                                                  int nw, int M, int N, int lane, const float* glu_bias) {
  constexpr int LPR = (EPI_GLU(EPI) ? FN * 8 : FN * 16) / 8, ROW = LPR + 1;
  const int tok = lane % 16, n4 = 4 * (lane / 16);
#pragma unroll
  for (int i = 0; i < FM; i += 2) {
#pragma unroll
    for (int ii = 0; ii < 2; ++ii) {
      u32x2_t* row = (u32x2_t*)(slab + (16 * ii + tok) * ROW) + lane / 16;
      if constexpr (EPI_GLU(EPI)) {       // gate columns, then the up columns that belong to them
#pragma unroll
        for (int j = 0; j < FN; j += 2) {
          f32x4_t g = block_of<FM, FN>(acc[i + ii][j]), u = block_of<FM, FN>(acc[i + ii][j + 1]);
          if constexpr (EPI == EPI_GEGLU)
            if (glu_bias != nullptr && nw + 16 * j < N) {
              g += *(const f32x4_t*)(glu_bias + nw + 16 * j + n4);
              u += *(const f32x4_t*)(glu_bias + nw + 16 * j + 16 + n4);
            }
          row[2 * j] = u32x2_t{pack_bf16x2(glu_f<EPI>(g[0], u[0]), glu_f<EPI>(g[1], u[1])),
                               pack_bf16x2(glu_f<EPI>(g[2], u[2]), glu_f<EPI>(g[3], u[3]))};
        }
      } else {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const f32x4_t v = block_of<FM, FN>(acc[i + ii][j]);
          row[4 * j] = u32x2_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        }
      }
    }
    wave_fence();               // the slab is written
    const int n_out = EPI_GLU(EPI) ? N / 2 : N, nw_out = EPI_GLU(EPI) ? nw / 2 : nw;
#pragma unroll
    for (int it = 0; it < (32 * LPR + 63) / 64; ++it) {
      const int at = it * 64 + lane, m = mw + 16 * i + at / LPR, n = nw_out + at % LPR * 8;
      if (32 * LPR % 64 == 0 || at < 32 * LPR) {
        const u32x4_t v = slab[at / LPR * ROW + at % LPR];
        if (m < M && n < n_out) *(u32x4_t*)((bf16_t*)Cv + (size_t)m * n_out + n) = v;
      }
    }
    wave_fence();               // and read, before it is written again
  }
}

// How K is shared: T256_WHOLE not; T256_SPLIT in gridDim.y parts of whole 128, as even as they come (a
// part's sums go to Cv + part * M * N); T256_TAIL the tiles of the order's last, short round, from
// `whole` on, by tail_split workgroups each, which leave float32 partials [tail][tail_split][256][BN] in
// tail_ws for tile_tail_reduce_kernel (the parts of one tile lie a multiple of the tail apart in the
// grid: where 8 divides the tail, in one XCD).
enum { T256_WHOLE = 0, T256_SPLIT = 1, T256_TAIL = 2 };

template <int BN, int EPI, int MODE = T256_WHOLE>
__global__ __launch_bounds__(256) void gemm_bf16_tile256_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ Cv, int M,
    int N, int K, int tiles_m, int tiles_n, const float* __restrict__ glu_bias, int whole,
    int tail_split, float* __restrict__ tail_ws) {
  // (the host pass, which only needs the launch stub, does not know the buffer descriptor type)
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int BM = 256, NT = 256, WM = 128, WN = BN / 2, FM = WM / 16, FN = WN / 16;
  static_assert(BN == 128 || BN == 192 || BN == 256, "tile width");
  constexpr int NA = BN == 128 ? 3 : 2, NW = 3;                 // stages of tokens and of W
  constexpr int A_PLACES = BM * 8, W_PLACES = BN * 8;           // 16-byte pieces of a k-tile of 64
  constexpr int A_CHUNKS = A_PLACES / NT, W_CHUNKS = W_PLACES / NT;     // copies per thread
  constexpr int CHUNKS = A_CHUNKS + W_CHUNKS;
  constexpr int PART1 = CHUNKS / 2;         // copies behind a tile's second k-step; the rest behind
                                            // the next one's first
  __shared__ u32x4_t a_stage0[A_PLACES];
  __shared__ u32x4_t a_stage1[A_PLACES];
  __shared__ u32x4_t a_stage2[NA > 2 ? A_PLACES : 1];
  __shared__ u32x4_t w_stage0[W_PLACES];
  __shared__ u32x4_t w_stage1[W_PLACES];
  __shared__ u32x4_t w_stage2[W_PLACES];
  auto a_stage = [&](auto IDX) __attribute__((always_inline)) -> u32x4_t* {
    constexpr int I = decltype(IDX)::value % NA;
    if constexpr (I == 0) return a_stage0;
    else if constexpr (I == 1) return a_stage1;
    else return a_stage2;
  };
  auto w_stage = [&](auto IDX) __attribute__((always_inline)) -> u32x4_t* {
    constexpr int I = decltype(IDX)::value % NW;
    if constexpr (I == 0) return w_stage0;
    else if constexpr (I == 1) return w_stage1;
    else return w_stage2;
  };

  int tile = blockIdx.x, part = MODE == T256_SPLIT ? blockIdx.y : 0, parts = MODE == T256_SPLIT ? gridDim.y : 1;
  const bool in_tail = MODE == T256_TAIL && tile >= whole;
  if (in_tail) {
    const int tail = tiles_m * tiles_n - whole;
    part = (tile - whole) / tail;
    parts = tail_split;
    tile = whole + (tile - whole) % tail;
  }
  int tm, tn;
  tile_of_workgroup<8>(tile, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;

  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int wm = wave / 2, wn = wave % 2;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);        // the LDS address is a scalar

  f32x4_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // Sources, as a base all lanes share plus a 32-bit offset per lane.  Tokens: place p =
  // tid + 256 c is row p / 8 = tid / 8 + 32 c, slot p % 8, and takes piece slot ^ ((row >> 1) & 7)
  // of the row's 128 bytes (rows beyond M: the last row).  W: place q = tid + 256 c of the stage is
  // piece q % 128 of the tile's 16-row group q / 128, as in memory: [8-k half][k-step of 16][output].
  // Groups beyond N are clamped (never stored).
  const int unit0 = MODE == T256_WHOLE ? 0 : (int)((long long)part * (K / 128) / parts);
  const int units = MODE == T256_WHOLE ? K / 128 : (int)((part + 1ll) * (K / 128) / parts) - unit0;
  const char* a_tile = (const char*)(A + (size_t)m0 * K + (size_t)unit0 * 128);
  uint32_t asrc[A_CHUNKS];
#pragma unroll
  for (int c = 0; c < A_CHUNKS; ++c) {
    const int row = tid / 8 + 32 * c, piece = (tid % 8) ^ ((tid / 16) & 7);
    asrc[c] = ((uint32_t)(min(m0 + row, M - 1) - m0) * (uint32_t)K + piece * 8) * 2;
  }
  const int kt64 = K / 64;
  const int grp0 = min(n0 / 16, N / 16 - 1);
  const char* w_tile = (const char*)(W + ((size_t)grp0 * kt64 + 2 * unit0) * 1024);
  uint32_t wsrc[W_CHUNKS];
#pragma unroll
  for (int c = 0; c < W_CHUNKS; ++c) {
    const int grp = min(n0 / 16 + tid / 128 + 2 * c, N / 16 - 1) - grp0;
    wsrc[c] = (uint32_t)grp * (uint32_t)kt64 * 2048 + (tid % 128) * 16;
  }
  // (tiles behind the last one are the last one again)
  const int ktiles = 2 * units, klast = ktiles - 1;
  // The copies address memory through buffer descriptors (the tile's first token row, the
  // tile's first group of W; no bound that the offsets could reach): base, an offset per
  // lane and one all lanes share, so that a copy costs no address arithmetic and issues
  // faster than one with a 64-bit address per lane.
  const __amdgpu_buffer_rsrc_t a_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)a_tile, 0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t w_rsrc =
      __builtin_amdgcn_make_buffer_rsrc((void*)w_tile, 0, 0x7fffffff, 0x00020000);
  auto copy_a = [&](int t, u32x4_t* stage, int c) __attribute__((always_inline)) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        a_rsrc, (__attribute__((address_space(3))) void*)(stage + (wave_u * 64 + c * NT)), 16,
        asrc[c], (uint32_t)min(t, klast) * 128, 0, 0);
  };
  auto copy_w = [&](int t, u32x4_t* stage, int c) __attribute__((always_inline)) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        w_rsrc, (__attribute__((address_space(3))) void*)(stage + (wave_u * 64 + c * NT)), 16,
        wsrc[c], (uint32_t)min(t, klast) * 2048, 0, 0);
  };
  // Copy q of those that are issued between the meeting of tile t - 1 and that of tile t (whose
  // number is IDX modulo the stages): the tokens of tile t + NA - 1 first, then W of tile t + NW - 1.
  auto copy_one = [&](int t, auto IDX, auto Q) __attribute__((always_inline)) {
    constexpr int q = decltype(Q)::value, I = decltype(IDX)::value;
    if constexpr (q < A_CHUNKS) copy_a(t + NA - 1, a_stage(std::integral_constant<int, I + NA - 1>{}), q);
    else copy_w(t + NW - 1, w_stage(std::integral_constant<int, I + NW - 1>{}), q - A_CHUNKS);
  };
  // what may still be in flight at the meeting of tile t, whose next tile has landed
  constexpr int LATER = NA == 3 ? CHUNKS : W_CHUNKS;
  // MFMA operands of k-step ks (0, 1) of a stage: tokens of row block i at a_at[ks] + 128 i,
  // outputs of column block j at w_at[ks] + 128 j (row or output lane % 16, k = 32 ks + 8 (lane / 16) .. + 8)
  int a_at[2], w_at[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    a_at[ks] = (wm * WM + lane % 16) * 8 + ((4 * ks + lane / 16) ^ ((lane % 16) >> 1));
    w_at[ks] = wn * (WN / 16) * 128 + (lane / 16 % 2) * 64 + (2 * ks + lane / 32) * 16 + lane % 16;
  }
  constexpr int NR = FM + FN;       // operand reads from LDS per k-step
  u32x4_t af[2][FM], wf[2][FN];
  // operand read number c of k-step ks of a tile: the FM token blocks, then the FN output blocks
  auto reads = [&](auto& self, auto IDX, auto KS, auto C0, auto CNT) __attribute__((always_inline)) -> void {
    constexpr int ks = decltype(KS)::value, c = decltype(C0)::value, n = decltype(CNT)::value;
    if constexpr (n > 0) {
      if constexpr (c < FM) af[ks][c] = a_stage(IDX)[a_at[ks] + c * 128];
      else wf[ks][c - FM] = w_stage(IDX)[w_at[ks] + (c - FM) * 128];
      self(self, IDX, KS, std::integral_constant<int, c + 1>{}, std::integral_constant<int, n - 1>{});
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  // The FM * FN MFMAs of k-step KS; behind them the reads of k-step READ_KS of tile READ, and cnt
  // copies from q0 on of tile t's (its number INTO).
  auto k_step = [&](auto KS, int t, auto INTO, auto Q0, auto CNT, auto READ, auto READ_KS)
                    __attribute__((always_inline)) {
    constexpr int ks = decltype(KS)::value, q0 = decltype(Q0)::value, cnt = decltype(CNT)::value;
    constexpr int NM = FM * FN;
    static_assert(2 * NR <= NM, "every read has an MFMA to follow");
    auto run = [&](auto& self, auto MI) __attribute__((always_inline)) -> void {
      constexpr int m = decltype(MI)::value, i = m / FN, j = m % FN;
      if constexpr (m < NM) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *(const bf16x8_t*)&wf[ks][j], *(const bf16x8_t*)&af[ks][i], acc[i][j], 0, 0, 0);
        constexpr int d = copy_after(m, NM, cnt), r0 = reads_before(m, NR), r1 = reads_before(m + 1, NR);
        reads(reads, READ, READ_KS, std::integral_constant<int, r0>{}, std::integral_constant<int, r1 - r0>{});
        if constexpr (d >= 0) copy_one(t, INTO, std::integral_constant<int, q0 + (d >= 0 ? d : 0)>{});
        __builtin_amdgcn_sched_barrier(0);
        self(self, std::integral_constant<int, m + 1>{});
      }
    };
    run(run, I0{});
  };
  // prologue: tile 0, what of tile 1 belongs before tile 0's own copies, and the first part of those
#pragma unroll
  for (int c = 0; c < A_CHUNKS; ++c) copy_a(0, a_stage0, c);
#pragma unroll
  for (int c = 0; c < W_CHUNKS; ++c) copy_w(0, w_stage0, c);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (NA == 3)
#pragma unroll
    for (int c = 0; c < A_CHUNKS; ++c) copy_a(1, a_stage1, c);
#pragma unroll
  for (int c = 0; c < W_CHUNKS; ++c) copy_w(1, w_stage1, c);
  __builtin_amdgcn_sched_barrier(0);
  auto first = [&](auto& self, auto Q) __attribute__((always_inline)) -> void {
    if constexpr (decltype(Q)::value < PART1) {
      copy_one(0, I0{}, Q);
      self(self, std::integral_constant<int, decltype(Q)::value + 1>{});
    }
  };
  first(first, I0{});
  __builtin_amdgcn_sched_barrier(0);
  constexpr int BEHIND = PART1 + (NA == 3 ? A_CHUNKS : 0) + W_CHUNKS;
  __builtin_amdgcn_s_waitcnt(0x0f70 | (BEHIND & 15) | ((BEHIND >> 4) << 14));     // vmcnt(BEHIND)
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  reads(reads, I0{}, I0{}, I0{}, std::integral_constant<int, NR>{});
  auto step = [&](int t, auto IDX) __attribute__((always_inline)) {
    using NXT = std::integral_constant<int, decltype(IDX)::value + 1>;
    k_step(I0{}, t, IDX, std::integral_constant<int, PART1>{}, std::integral_constant<int, CHUNKS - PART1>{},
           IDX, I1{});
    // (and every LDS read done: the meeting frees this tile's places)
    __builtin_amdgcn_s_waitcnt(0x0070 | (LATER & 15) | ((LATER >> 4) << 14));     // vmcnt(LATER) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    k_step(I1{}, t + 1, NXT{}, I0{}, std::integral_constant<int, PART1>{}, NXT{}, I0{});
  };
  // Whole turns round the stages in one loop, what is left of a turn behind it (one way in and one
  // way out: with more the accumulators move between registers).  K % 128 == 0: an even number of tiles.
  constexpr int TURN = NA == 2 ? 6 : 3;
  int kt = 0;
  for (; kt + TURN <= ktiles; kt += TURN) {
    step(kt, I0{});
    step(kt + 1, I1{});
    step(kt + 2, std::integral_constant<int, 2>{});
    if constexpr (TURN == 6) {
      step(kt + 3, std::integral_constant<int, 3>{});
      step(kt + 4, std::integral_constant<int, 4>{});
      step(kt + 5, std::integral_constant<int, 5>{});
    }
  }
  if (kt < ktiles) {
    step(kt, I0{});
    if (TURN == 6 || kt + 1 < ktiles) step(kt + 1, I1{});
    if constexpr (TURN == 6)
      if (kt + 2 < ktiles) {
        step(kt + 2, std::integral_constant<int, 2>{});
        step(kt + 3, std::integral_constant<int, 3>{});
      }
  }
  // nothing may still be on its way into LDS when a stage becomes the epilogue's slabs or the
  // workgroup ends
  __builtin_amdgcn_s_waitcnt(0x0f70);       // vmcnt(0)
  __syncthreads();
  const int mw = m0 + wm * WM, nw = n0 + wn * WN;
  if constexpr (MODE == T256_SPLIT) Cv = (float*)Cv + (size_t)part * M * N;
  if constexpr (MODE == T256_TAIL)
    if (in_tail) {        // the whole tile, rows and columns beyond the matrices too
      store_blocks_f32<FM, FN, false>(acc, tail_ws + ((size_t)(tile - whole) * parts + part) * BM * BN, wm * WM,
                                      wn * WN, BM, BN, lane);
      return;
    }
  if constexpr (EPI == EPI_STORE_F32 || EPI == EPI_ACC_F32) {
    store_blocks_f32<FM, FN, EPI == EPI_ACC_F32>(acc, (float*)Cv, mw, nw, M, N, lane);
  } else {
    constexpr int SLAB = slab_places<FN, EPI>();
    static_assert(2 * SLAB <= A_PLACES, "the slabs of two waves fit a stage of tokens");
    store_blocks_bf16<FM, FN, EPI>(acc, Cv, (wm == 0 ? a_stage0 : a_stage1) + wn * SLAB, mw, nw, M, N, lane,
                                   glu_bias);
  }
#endif
}

template <int BN>
static int launch_tile256(const void* A, const void* W, void* C, int M, int N, int K, int epi,
                          hipStream_t stream, const float* glu_bias = nullptr) {
  if (N % 16 != 0 || K % 128 != 0) return -3;
  const int tiles_m = (M + 255) / 256, tiles_n = (N + BN - 1) / BN;
  const dim3 grid(tiles_m * tiles_n), block(256);
#define ZF_T256(E)                                                                             \
  hipLaunchKernelGGL((gemm_bf16_tile256_kernel<BN, E>), grid, block, 0, stream,                \
                     (const bf16_t*)A, (const bf16_t*)W, C, M, N, K, tiles_m, tiles_n,         \
                     glu_bias, 0, 1, (float*)nullptr)
  if (epi == EPI_STORE_BF16) ZF_T256(EPI_STORE_BF16);
  else if (epi == EPI_STORE_F32) ZF_T256(EPI_STORE_F32);
  else if (epi == EPI_SWIGLU) ZF_T256(EPI_SWIGLU);
  else if (epi == EPI_GEGLU) ZF_T256(EPI_GEGLU);
  else ZF_T256(EPI_ACC_F32);
#undef ZF_T256
  return (int)hipGetLastError();
}

// The 256 x 256 tiles with the tile order's tiles from `whole` on shared by `split` workgroups each
// along K (ws: float32 [tiles - whole][split][256][256]) and the kernel that adds their partials;
// every epilogue.
static int launch_tile256_tail(const void* A, const void* W, void* C, void* ws, int M, int N, int K,
                               int epi, int whole, int split, hipStream_t stream,
                               const float* glu_bias = nullptr) {
  const int tiles_m = (M + 255) / 256, tiles_n = (N + 255) / 256;
  const long long tiles = (long long)tiles_m * tiles_n, tail = tiles - whole;
  if (N % 16 != 0 || K % 128 != 0 || ws == nullptr) return -3;
  if (split < 2 || split > K / 128 || whole < 0 || tail <= 0 || whole + tail * split > 0x7fffffffLL) return -3;
  const dim3 grid((unsigned)(whole + tail * split)), block(256);
#define ZF_T256T(E)                                                                            \
  do {                                                                                         \
    hipLaunchKernelGGL((gemm_bf16_tile256_kernel<256, E, T256_TAIL>), grid, block, 0, stream,  \
                       (const bf16_t*)A, (const bf16_t*)W, C, M, N, K, tiles_m, tiles_n,       \
                       glu_bias, whole, split, (float*)ws);                                    \
    hipLaunchKernelGGL((tile_tail_reduce_kernel<256, 256, E>), dim3((unsigned)tail, 32),       \
                       dim3(256), 0, stream, (const float*)ws, C, M, N, tiles_m, tiles_n,      \
                       whole, split, glu_bias);                                                \
  } while (0)
  if (epi == EPI_STORE_BF16) ZF_T256T(EPI_STORE_BF16);
  else if (epi == EPI_STORE_F32) ZF_T256T(EPI_STORE_F32);
  else if (epi == EPI_SWIGLU) ZF_T256T(EPI_SWIGLU);
  else if (epi == EPI_GEGLU) ZF_T256T(EPI_GEGLU);
  else ZF_T256T(EPI_ACC_F32);
#undef ZF_T256T
  return (int)hipGetLastError();
}

// ---------------------------------------------------------------- large M: smaller tiles, both operands in a ring
// Tiles of BM tokens x BN outputs for products of few tiles, one workgroup of 4 waves (2 x 2) to a CU: k-tiles
// of 64 of both operands in a ring of NS stages, copied straight into LDS as in the kernel above, the copies of
// a stage NS - 1 k-tiles old when they are waited for.  With one workgroup to a CU nothing else hides a
// load, and the kernel that takes W straight into registers is one k-tile ahead: 200 tokens into 4096 over
// 2048, 64 x 64, 12.0 -> 7.7 us; 768 tokens, 128 x 128, 20.8 -> 16.3; 2048 into 2048 over 2048 22.1 -> 18.2,
// over 4096 39.0 -> 31.2; 200 into 6144 over 4096, 128 x 64, 24.5 -> 22.3.  From two workgroups to a CU on it
// is behind (512 into 7168 over 5120 45.5 -> 47.9: half the flops a byte of LDS that the 256-token tiles have).
// The same bits.  SPLIT: gridDim.y parts of K, a part's sums at Cv + part * M * N.
template <int BM, int BN, int EPI, bool SPLIT>
__global__ __launch_bounds__(256) void gemm_bf16_ring_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ Cv, int M, int N, int K,
    int tiles_m, int tiles_n, const float* __restrict__ glu_bias) {
  // (the host pass, which only needs the launch stub, does not know the buffer descriptor type)
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NT = 256, WM = BM / 2, WN = BN / 2, FM = WM / 16, FN = WN / 16;
  constexpr int NS = BM + BN >= 384 ? 3 : BM + BN >= 256 ? 4 : 5;
  constexpr int A_PLACES = BM * 8, W_PLACES = BN * 8, STAGE = A_PLACES + W_PLACES;
  constexpr int A_CHUNKS = A_PLACES / NT, W_CHUNKS = W_PLACES / NT, COPIES = A_CHUNKS + W_CHUNKS;
  __shared__ u32x4_t stage0[STAGE];
  __shared__ u32x4_t stage1[STAGE];
  __shared__ u32x4_t stage2[STAGE];
  __shared__ u32x4_t stage3[NS > 3 ? STAGE : 1];
  __shared__ u32x4_t stage4[NS > 4 ? STAGE : 1];
  auto stage_of = [&](auto IDX) __attribute__((always_inline)) -> u32x4_t* {
    constexpr int I = decltype(IDX)::value % NS;
    if constexpr (I == 0) return stage0;
    else if constexpr (I == 1) return stage1;
    else if constexpr (I == 2) return stage2;
    else if constexpr (I == 3) return stage3;
    else return stage4;
  };
  int tm, tn;
  tile_of_workgroup<(BM >= 128 ? 8 : 1024 / BM)>(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64, wm = wave / 2, wn = wave % 2;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);        // the LDS address is a scalar
  f32x4_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // sources and operands as in the kernel above
  const int kt_all = K / 64, kt0 = SPLIT ? (int)((long long)blockIdx.y * kt_all / gridDim.y) : 0;
  const int ktiles = SPLIT ? (int)((blockIdx.y + 1ll) * kt_all / gridDim.y) - kt0 : kt_all;
  const int grp0 = min(n0 / 16, N / 16 - 1);
  const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(A + (size_t)m0 * K + (size_t)kt0 * 64), 0, 0x7fffffff, 0x00020000);
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(W + ((size_t)grp0 * kt_all + kt0) * 1024), 0, 0x7fffffff, 0x00020000);
  uint32_t asrc[A_CHUNKS], wsrc[W_CHUNKS];
#pragma unroll
  for (int c = 0; c < A_CHUNKS; ++c) {
    const int row = tid / 8 + 32 * c, piece = (tid % 8) ^ ((tid / 16) & 7);
    asrc[c] = ((uint32_t)(min(m0 + row, M - 1) - m0) * (uint32_t)K + piece * 8) * 2;
  }
#pragma unroll
  for (int c = 0; c < W_CHUNKS; ++c) {
    const int grp = min(n0 / 16 + tid / 128 + 2 * c, N / 16 - 1) - grp0;
    wsrc[c] = (uint32_t)grp * (uint32_t)kt_all * 2048 + (tid % 128) * 16;
  }
  auto copies = [&](auto& self, int t, u32x4_t* to, auto Q, auto CNT) __attribute__((always_inline)) -> void {
    constexpr int q = decltype(Q)::value;
    if constexpr (decltype(CNT)::value > 0) {
      const uint32_t at = (uint32_t)min(t, ktiles - 1);      // (behind the last one: the last one again)
      if constexpr (q < A_CHUNKS)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            a_rsrc, (__attribute__((address_space(3))) void*)(to + wave_u * 64 + q * NT), 16, asrc[q], at * 128, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            w_rsrc, (__attribute__((address_space(3))) void*)(to + A_PLACES + wave_u * 64 + (q - A_CHUNKS) * NT), 16,
            wsrc[q - A_CHUNKS], at * 2048, 0, 0);
      self(self, t, to, std::integral_constant<int, q + 1>{}, std::integral_constant<int, decltype(CNT)::value - 1>{});
    }
  };
  int a_at[2], w_at[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    a_at[ks] = (wm * WM + lane % 16) * 8 + ((4 * ks + lane / 16) ^ ((lane % 16) >> 1));
    w_at[ks] = A_PLACES + wn * (WN / 16) * 128 + (lane / 16 % 2) * 64 + (2 * ks + lane / 32) * 16 + lane % 16;
  }
  constexpr int NR = FM + FN, NM = FM * FN;
  u32x4_t af[2][FM], wf[2][FN];
  auto reads = [&](auto& self, const u32x4_t* from, auto KS, auto C0, auto CNT) __attribute__((always_inline)) -> void {
    constexpr int ks = decltype(KS)::value, c = decltype(C0)::value, n = decltype(CNT)::value;
    if constexpr (n > 0) {
      if constexpr (c < FM) af[ks][c] = from[a_at[ks] + c * 128];
      else wf[ks][c - FM] = from[w_at[ks] + (c - FM) * 128];
      self(self, from, KS, std::integral_constant<int, c + 1>{}, std::integral_constant<int, n - 1>{});
    }
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  using I3 = std::integral_constant<int, 3>;
  using I4 = std::integral_constant<int, 4>;
  using NONE = I0;
  using ALL = std::integral_constant<int, COPIES>;
  // k-step KS's MFMAs; behind the first ones the reads of the next k-step (READ_KS of `from`), spread over
  // them cnt copies of k-tile t
  auto k_step = [&](auto KS, const u32x4_t* from, auto READ_KS, int t, u32x4_t* into, auto CNT)
                    __attribute__((always_inline)) {
    constexpr int ks = decltype(KS)::value, cnt = decltype(CNT)::value;
    auto run = [&](auto& self, auto MI) __attribute__((always_inline)) -> void {
      constexpr int m = decltype(MI)::value, i = m / FN, j = m % FN;
      if constexpr (m < NM) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *(const bf16x8_t*)&wf[ks][j], *(const bf16x8_t*)&af[ks][i], acc[i][j], 0, 0, 0);
        constexpr int r0 = 2 * m < NR ? 2 * m : NR, r1 = 2 * m + 2 < NR ? 2 * m + 2 : NR;
        reads(reads, from, READ_KS, std::integral_constant<int, r0>{}, std::integral_constant<int, r1 - r0>{});
        constexpr int c0 = m * cnt / NM, c1 = (m + 1) * cnt / NM;
        copies(copies, t, into, std::integral_constant<int, c0>{}, std::integral_constant<int, c1 - c0>{});
        __builtin_amdgcn_sched_barrier(0);
        self(self, std::integral_constant<int, m + 1>{});
      }
    };
    run(run, I0{});
  };
  copies(copies, 0, stage0, I0{}, ALL{});
  __builtin_amdgcn_sched_barrier(0);
  copies(copies, 1, stage1, I0{}, ALL{});
  __builtin_amdgcn_sched_barrier(0);
  copies(copies, 2, stage2, I0{}, ALL{});
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (NS > 3) copies(copies, 3, stage3, I0{}, ALL{});
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (NS > 4) copies(copies, 4, stage4, I0{}, ALL{});
  __builtin_amdgcn_sched_barrier(0);
  constexpr int FIRST = (NS - 1) * COPIES, AHEAD = (NS - 2) * COPIES;      // younger copies at a meeting
  static_assert(FIRST < 64, "the wait counts them");
  __builtin_amdgcn_s_waitcnt(0x0f70 | (FIRST & 15) | ((FIRST >> 4) << 14));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  reads(reads, stage0, I0{}, I0{}, std::integral_constant<int, NR>{});
  auto step = [&](int t, auto IDX) __attribute__((always_inline)) {
    k_step(I0{}, stage_of(IDX), I1{}, 0, stage0, NONE{});
    // the next k-tile has landed, and (every read done) all waves have read this one
    __builtin_amdgcn_s_waitcnt(0x0070 | (AHEAD & 15) | ((AHEAD >> 4) << 14));     // vmcnt(AHEAD) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    k_step(I1{}, stage_of(std::integral_constant<int, decltype(IDX)::value + 1>{}), I0{}, t + NS, stage_of(IDX), ALL{});
  };
  int t = 0;
  for (; t + NS <= ktiles; t += NS) {
    step(t, I0{});
    step(t + 1, I1{});
    step(t + 2, I2{});
    if constexpr (NS > 3) step(t + 3, I3{});
    if constexpr (NS > 4) step(t + 4, I4{});
  }
  if (t < ktiles) {
    step(t, I0{});
    if (t + 1 < ktiles) {
      step(t + 1, I1{});
      if constexpr (NS > 3)
        if (t + 2 < ktiles) {
          step(t + 2, I2{});
          if constexpr (NS > 4)
            if (t + 3 < ktiles) step(t + 3, I3{});
        }
    }
  }
  // nothing may still be on its way into LDS when a stage becomes the slabs or the workgroup ends
  __builtin_amdgcn_s_waitcnt(0x0f70);       // vmcnt(0)
  __syncthreads();
  const int mw = m0 + wm * WM, nw = n0 + wn * WN;
  if constexpr (SPLIT) Cv = (float*)Cv + (size_t)blockIdx.y * M * N;
  if constexpr (EPI == EPI_STORE_F32 || EPI == EPI_ACC_F32) {
    store_blocks_f32<FM, FN, EPI == EPI_ACC_F32>(acc, (float*)Cv, mw, nw, M, N, lane);
  } else {
    constexpr int SLAB = slab_places<FN, EPI>();
    static_assert(4 * SLAB <= STAGE, "the waves' slabs fit a stage");
    store_blocks_bf16<FM, FN, EPI>(acc, Cv, stage0 + wave * SLAB, mw, nw, M, N, lane, glu_bias);
  }
#endif
}

template <int BM, int BN>
static int launch_ring(const void* A, const void* W, void* C, int M, int N, int K, int epi, hipStream_t stream,
                       const float* glu_bias = nullptr) {
  if (N % 16 != 0 || K % 64 != 0 || K <= 0) return -3;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
#define ZF_RING(E)                                                                             \
  hipLaunchKernelGGL((gemm_bf16_ring_kernel<BM, BN, E, false>), dim3(tiles_m * tiles_n), dim3(256), 0, stream, \
                     (const bf16_t*)A, (const bf16_t*)W, C, M, N, K, tiles_m, tiles_n, glu_bias)
  if (epi == EPI_STORE_BF16) ZF_RING(EPI_STORE_BF16);
  else if (epi == EPI_STORE_F32) ZF_RING(EPI_STORE_F32);
  else if (epi == EPI_SWIGLU) ZF_RING(EPI_SWIGLU);
  else if (epi == EPI_GEGLU) ZF_RING(EPI_GEGLU);
  else ZF_RING(EPI_ACC_F32);
#undef ZF_RING
  return (int)hipGetLastError();
}
// the float32 partials [ksplit, M, N] of the product in ws
template <int BM, int BN>
static int launch_ring_parts(const void* A, const void* W, void* ws, int M, int N, int K, int ksplit,
                             hipStream_t stream) {
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  hipLaunchKernelGGL((gemm_bf16_ring_kernel<BM, BN, EPI_STORE_F32, true>), dim3(tiles_m * tiles_n, ksplit),
                     dim3(256), 0, stream, (const bf16_t*)A, (const bf16_t*)W, ws, M, N, K, tiles_m, tiles_n,
                     (const float*)nullptr);
  return (int)hipGetLastError();
}

// adds the float32 partials [ksplit, M, N] in split order and applies the epilogue (defined
// with the weight-streaming kernel below)
static int launch_reduce(const void* ws, void* C, int M, int N, int ksplit, int epi,
                         hipStream_t stream);

template <int BM, int BN, int WM, int WN, int TKM = TK, bool W2 = false, bool ADMA = false,
          int KG = 1>
static int launch_tile_wdirect(const void* A, const void* W, void* C, int M, int N, int K, int epi,
                               hipStream_t stream, void* ws = nullptr, int ksplit = 1,
                               bool reduce = true, const float* glu_bias = nullptr) {
  if (N % 16 != 0 || K % TKM != 0) return -3;
  // every part (and every group of waves in it) an even number of k-tiles
  if (W2 && (K / TKM) % (2 * ksplit * KG) != 0) return -3;
  if (KG > 1 && (K / TKM) % (ksplit * KG) != 0) return -3;      // the groups meet step by step
  if (ksplit > 1 && (ws == nullptr || EPI_GLU(epi) || ksplit > K / TKM)) return -3;
  constexpr int NT = (BM / WM) * (BN / WN) * 64 * KG;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const dim3 grid(tiles_m * tiles_n, ksplit), block(NT);
  const int final_epi = epi;
  constexpr size_t stages = (size_t)2 * BM * (TKM + 8) * sizeof(bf16_t);
  constexpr size_t slabs = (size_t)(BM / WM) * (BN / WN) * 32 * (WN + 4) * sizeof(float);
  // two groups: the column blocks handed over (half of every wave's rows, one block)
  constexpr size_t handed = (size_t)KG * (BM / WM) * (BN / WN) * (WM / 64) * 16 * 64 * sizeof(float);
  // (with the tokens copied straight into LDS the stages are arrays of the kernel's own)
  const size_t smem = KG > 1 ? handed : ADMA ? slabs : stages > slabs ? stages : slabs;
  static_assert(KG == 1 || handed >= (size_t)KG * (BM / WM) * (BN / WN) * 32 * 36 * sizeof(float),
                "the slabs of the two groups' waves fit where the blocks are handed over");
#define ZF_WD(E)                                                                              \
  do {                                                                                        \
    auto kern = gemm_bf16_tile_wdirect_kernel<BM, BN, WM, WN, E, TKM, W2, ADMA, false, KG>;   \
    if (smem > 64 * 1024 || KG > 1) {                                                         \
      hipError_t e = hipFuncSetAttribute((const void*)kern,                                   \
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem); \
      if (e != hipSuccess) return (int)e;                                                     \
    }                                                                                         \
    hipLaunchKernelGGL(kern, grid, block, smem, stream, (const bf16_t*)A, (const bf16_t*)W, C, \
                       M, N, K, tiles_m, tiles_n, 0, 1, (float*)nullptr, glu_bias);           \
  } while (0)
  void* const final_c = C;
  if (ksplit > 1) {
    epi = EPI_STORE_F32;
    C = ws;
  }
  if (epi == EPI_STORE_BF16) ZF_WD(EPI_STORE_BF16);
  else if (epi == EPI_STORE_F32) ZF_WD(EPI_STORE_F32);
  else if (epi == EPI_SWIGLU) ZF_WD(EPI_SWIGLU);
  else if (epi == EPI_GEGLU) ZF_WD(EPI_GEGLU);
  else ZF_WD(EPI_ACC_F32);
#undef ZF_WD
  if (ksplit > 1 && reduce) return launch_reduce(ws, final_c, M, N, ksplit, final_epi, stream);
  return (int)hipGetLastError();
}

// The 128 x 256 tiles with the tile order's tiles from `whole` on shared by `split` workgroups
// each along K (ws: float32 [tiles - whole][split][128][256]) and the kernel that adds their
// partials; every epilogue.
template <bool W2>
static int launch_tile_tail(const void* A, const void* W, void* C, void* ws, int M, int N, int K,
                            int epi, int whole, int split, hipStream_t stream,
                            const float* glu_bias = nullptr) {
  constexpr int BM = 128, BN = 256, WM = 128, WN = 64, NT = 256;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const long long tiles = (long long)tiles_m * tiles_n;
  if (N % 16 != 0 || K % TK != 0 || ws == nullptr) return -3;
  if (split < 2 || split > K / TK || whole < 0 || whole >= tiles) return -3;
  if (W2 && (K / TK) % (2 * split) != 0) return -3;
  const long long tail = tiles - whole;
  if (whole + tail * split > 0x7fffffffLL) return -3;
  const dim3 grid((unsigned)(whole + tail * split)), block(NT);
  constexpr size_t smem = (size_t)(BM / WM) * (BN / WN) * 32 * (WN + 4) * sizeof(float);
  static_assert(smem <= 64 * 1024, "the slabs fit the default limit");
#define ZF_WT(E)                                                                              \
  do {                                                                                        \
    hipLaunchKernelGGL((gemm_bf16_tile_wdirect_kernel<BM, BN, WM, WN, E, TK, W2, true, true>), \
                       grid, block, smem, stream, (const bf16_t*)A, (const bf16_t*)W, C, M, N, \
                       K, tiles_m, tiles_n, whole, split, (float*)ws, glu_bias);              \
    hipLaunchKernelGGL((tile_tail_reduce_kernel<BM, BN, E>), dim3((unsigned)tail, BM / 8),    \
                       dim3(BN), 0, stream, (const float*)ws, C, M, N, tiles_m, tiles_n,      \
                       whole, split, glu_bias);                                               \
  } while (0)
  if (epi == EPI_STORE_BF16) ZF_WT(EPI_STORE_BF16);
  else if (epi == EPI_STORE_F32) ZF_WT(EPI_STORE_F32);
  else if (epi == EPI_SWIGLU) ZF_WT(EPI_SWIGLU);
  else if (epi == EPI_GEGLU) ZF_WT(EPI_GEGLU);
  else ZF_WT(EPI_ACC_F32);
#undef ZF_WT
  return (int)hipGetLastError();
}

template <int BM, int BN, int WM, int WN, bool WT>
static int launch_tile(const void* A, const void* W, void* C, int M, int N, int K, int epi,
                       hipStream_t stream) {
  constexpr int NT = (BM / WM) * (BN / WN) * 64;
  const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  const int nblocks = tiles_m * tiles_n;
  const size_t smem = (size_t)2 * (BM + BN) * LDS_ROW * sizeof(bf16_t);
#define ZF_TILE_LAUNCH(E)                                                                      \
  do {                                                                                         \
    auto kern = gemm_bf16_tile_kernel<BM, BN, WM, WN, E, WT>;                                  \
    if (smem > 64 * 1024) {                                                                    \
      hipError_t e = hipFuncSetAttribute((const void*)kern,                                    \
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem); \
      if (e != hipSuccess) return (int)e;                                                      \
    }                                                                                          \
    hipLaunchKernelGGL(kern, dim3(nblocks), dim3(NT), smem, stream, (const bf16_t*)A,          \
                       (const bf16_t*)W, C, M, N, K, tiles_m, tiles_n);                        \
  } while (0)
  if (epi == EPI_STORE_BF16) ZF_TILE_LAUNCH(EPI_STORE_BF16);
  else if (epi == EPI_STORE_F32) ZF_TILE_LAUNCH(EPI_STORE_F32);
  else if (epi == EPI_SWIGLU) ZF_TILE_LAUNCH(EPI_SWIGLU);
  else ZF_TILE_LAUNCH(EPI_ACC_F32);
#undef ZF_TILE_LAUNCH
  return (int)hipGetLastError();
}

// variant, plain W: 0 = 128x128 (waves 64x64), 4 = 256x256 (waves 128x64, 8 waves);
//          pre-tiled W (w_tiled; N % 16 == 0 and K % 64 == 0), taken straight from memory
//          into the MFMA operands: 6 = 128x128 (waves 64x64), 16 = 128x128 with k-tiles of 128
//          and the waves side by side (128x32: for few tiles; K % 128 == 0), 10 = 128x256
//          (waves 128x64: no two waves load the same part of W, two workgroups share a CU,
//          and W is loaded two k-tiles ahead when their number is even).  10 copies the
//          tokens straight into LDS, and so does 6 from 384 tiles on: with two workgroups to
//          most CUs that was 2 to 18 % faster (qkv at 1024 and 2048 tokens), with one 10 to
//          34 % slower (512 tokens, or 256 tiles at 1024: nothing hides the copies' longer
//          way).  12 = the tiles of 10 with two groups of four waves in a workgroup,
//          each over half of K (K % 256 == 0): for 256 tiles or fewer, where a CU has one
//          workgroup either way.  20, 21 and 22 = 256 tokens x 256, 192 and 128 (K % 128 == 0).
//          30, 31 and 32 = 128x128, 128x64 and 64x64 with both operands in a ring of LDS stages.
//          7 = 6 with the tokens through registers at any size, 11 = 10 by another number: no rule
//          asks for them, callers that name a kernel may.
extern "C" int zf_gemm_bf16_tile(const void* A, const void* W, void* C, int M, int N, int K,
                                 int epi, int variant, int w_tiled, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K % 8 != 0 || (epi == EPI_SWIGLU && N % 32 != 0)) return -3;
  if (w_tiled) {
    if (N % 16 != 0 || K % 64 != 0) return -3;
    if (variant == 6 && (long long)((M + 127) / 128) * ((N + 127) / 128) >= 384)
      return launch_tile_wdirect<128, 128, 64, 64, TK, false, true>(A, W, C, M, N, K, epi, stream);
    if (variant == 6 || variant == 7)
      return launch_tile_wdirect<128, 128, 64, 64>(A, W, C, M, N, K, epi, stream);
    if (variant == 16)
      return launch_tile_wdirect<128, 128, 128, 32, 128>(A, W, C, M, N, K, epi, stream);
    if (variant == 10 || variant == 11) {
      if (K % (2 * TK) == 0)     // W two k-tiles ahead: an even number of k-tiles
        return launch_tile_wdirect<128, 256, 128, 64, TK, true, true>(A, W, C, M, N, K, epi,
                                                                      stream);
      return launch_tile_wdirect<128, 256, 128, 64, TK, false, true>(A, W, C, M, N, K, epi,
                                                                     stream);
    }
    if (variant == 20) return launch_tile256<256>(A, W, C, M, N, K, epi, stream);
    if (variant == 21) return launch_tile256<192>(A, W, C, M, N, K, epi, stream);
    if (variant == 22) return launch_tile256<128>(A, W, C, M, N, K, epi, stream);
    if (variant == 30) return launch_ring<128, 128>(A, W, C, M, N, K, epi, stream);
    if (variant == 31) return launch_ring<128, 64>(A, W, C, M, N, K, epi, stream);
    if (variant == 32) return launch_ring<64, 64>(A, W, C, M, N, K, epi, stream);
    if (variant == 12)         // the tiles of 10 with two groups of waves, each half of K
      return launch_tile_wdirect<128, 256, 128, 64, TK, true, true, 2>(A, W, C, M, N, K, epi,
                                                                       stream);
    return -4;
  }
  switch (variant) {
    case 0: return launch_tile<128, 128, 64, 64, false>(A, W, C, M, N, K, epi, stream);
    case 4: return launch_tile<256, 256, 128, 64, false>(A, W, C, M, N, K, epi, stream);
    default: return -4;
  }
}

// The 128 x 256 tiles of variant 10 on pre-tiled W where the tiles do not end on a whole round
// of the chip: the first `whole` tiles of the tile order run one workgroup each, the rest
// `split` workgroups each along K, so that the last round is as short as its share of the
// work (512 tokens into 34816 outputs, K = 5120: 544 tiles for 512 places, 210 -> 150 us).
// ws: float32 [tiles - whole][split][128][256].
extern "C" int zf_gemm_bf16_tile_tail(const void* A, const void* W, void* C, void* ws, int M,
                                      int N, int K, int epi, int whole, int split,
                                      hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K % 8 != 0 || (epi == EPI_SWIGLU && N % 32 != 0)) return -3;
  if (K % (2 * TK) == 0 && (K / TK) % (2 * split) == 0)
    return launch_tile_tail<true>(A, W, C, ws, M, N, K, epi, whole, split, stream);
  return launch_tile_tail<false>(A, W, C, ws, M, N, K, epi, whole, split, stream);
}

// The 256 x 256 tiles of variant 20 (K % 128 == 0) with the tiles from `whole` on shared by `split`
// workgroups each along K; ws: float32 [tiles - whole][split][256][256].
extern "C" int zf_gemm_bf16_tile256_tail(const void* A, const void* W, void* C, void* ws, int M,
                                         int N, int K, int epi, int whole, int split,
                                         hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (epi == EPI_SWIGLU && N % 32 != 0) return -3;
  return launch_tile256_tail(A, W, C, ws, M, N, K, epi, whole, split, stream);
}

// 17 to 128 tokens on pre-tiled W.  The weight-streaming kernel below re-reads the tokens for
// every 16 * RG rows of W, which at 64 tokens is as much traffic as W itself; here a workgroup
// takes 128 rows of W, its 4 waves side by side along them, the tokens of a k-tile go through
// LDS once for all of them, and the k-tiles are 128 or 256 wide so that 32 or 64 KB of W are
// in flight per workgroup.  ksplit workgroups share a tile's K (ws: float32 [ksplit, M, N])
// when the tiles do not fill the chip.
//   M <= 32: tiles of 32 tokens, K % 256 == 0;  M <= 64: 64 tokens;  M <= 128: 128 tokens;
//   both K % 128 == 0.
// Above 128 tokens: tiles of 64 tokens again, for a few hundred tokens on a narrow output
// whose 128-token tiles would leave most CUs idle (512 tokens into 6144 outputs: 384 tiles
// of 64 x 128 against 192 of 128 x 128, 41 -> 35 us).
extern "C" int zf_gemm_bf16_mid(const void* A, const void* W, void* C, void* ws, int M, int N,
                                int K, int epi, int ksplit, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (ksplit < 1 || (epi == EPI_SWIGLU && N % 32 != 0)) return -3;
  if (M > 128)
    return launch_tile_wdirect<64, 128, 64, 32, 128>(A, W, C, M, N, K, epi, stream, ws, ksplit);
  if (M <= 32)
    return launch_tile_wdirect<32, 128, 32, 32, 256>(A, W, C, M, N, K, epi, stream, ws, ksplit);
  if (M <= 64)
    return launch_tile_wdirect<64, 128, 64, 32, 128>(A, W, C, M, N, K, epi, stream, ws, ksplit);
  return launch_tile_wdirect<128, 128, 128, 32, 128>(A, W, C, M, N, K, epi, stream, ws, ksplit);
}

// The same product for 17 to 128 tokens with ksplit >= 2 workgroups along K, left as float32
// partials [ksplit, M, N] in ws for a kernel of the caller's that adds them on its way.
extern "C" int zf_gemm_bf16_mid_partials(const void* A, const void* W, void* ws, int M, int N,
                                         int K, int ksplit, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (ksplit < 2 || ws == nullptr || M > 128) return -3;
  if (M <= 32)
    return launch_tile_wdirect<32, 128, 32, 32, 256>(A, W, ws, M, N, K, EPI_STORE_F32, stream, ws,
                                                     ksplit, false);
  if (M <= 64)
    return launch_tile_wdirect<64, 128, 64, 32, 128>(A, W, ws, M, N, K, EPI_STORE_F32, stream, ws,
                                                     ksplit, false);
  return launch_tile_wdirect<128, 128, 128, 32, 128>(A, W, ws, M, N, K, EPI_STORE_F32, stream, ws,
                                                     ksplit, false);
}

enum { NORM_NONE = 0, NORM_FOLD = 1, NORM_GIVEN = 2 };

// What the weight-streaming kernel needs to know of an RMSNorm around it.
//   before the product: NORM_FOLD   gain, eps: the rows come as the 32-bit residual stream;
//                       NORM_GIVEN  eps, sq_in [sq_groups][16]: the rows come as
//                                   bfloat16(x * gain) with the sums of x^2 per 16 columns,
//                                   as the kernel that produced x left them (EMIT);
//   after it (EMIT, with the residual epilogue): gain_out, xg_out [M, N], sq_out [N / 16][16]
//                                   for the norm that reads the sum next.
struct SkinnyNorm {
  const float* gain;
  float eps;
  const float* sq_in;
  int sq_groups;
  const float* gain_out;
  bf16_t* xg_out;
  float* sq_out;
  const float* glu_bias;       // (EPI_GEGLU) a bias a row of W, or null
  int act;                     // (EPI_ACT) which activation (activation_value)
};

// The 128 x 128 tiled product on pre-tiled W with ksplit workgroups per tile along K, for
// products whose tiles alone do not fill the chip (a few hundred tokens, a narrow output).
// ws: float32 [ksplit, M, N]; epi: store bf16, store f32 or add into f32.
extern "C" int zf_gemm_bf16_tile_splitk(const void* A, const void* W, void* C, void* ws, int M,
                                        int N, int K, int epi, int ksplit, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (ksplit < 2 || ksplit > 64 || epi == EPI_SWIGLU) return -3;
  if (K % 128 == 0)      // the waves side by side along the outputs: W is loaded once
    return launch_tile_wdirect<128, 128, 128, 32, 128>(A, W, C, M, N, K, epi, stream, ws, ksplit);
  return launch_tile_wdirect<128, 128, 64, 64>(A, W, C, M, N, K, epi, stream, ws, ksplit);
}

// ---------------------------------------------------------------- small M: weight streaming
// For M <= 64 the product is bound by reading W once from HBM.  A workgroup owns 16 * RG rows
// of W (output features) and all M tokens; its 8 waves (times KSPLIT workgroups along
// gridDim.y) split K between them in steps of 64: each lane loads 2 x 16 bytes of one row, 4
// lanes cover a 128-byte line.  W is the first MFMA operand, the tokens (read through L2,
// they are small, and reused for the RG row groups) the second (v_mfma_f32_16x16x32_bf16).
// The waves' partial sums are added through LDS in wave order; with KSPLIT > 1 the
// workgroups write float32 partials to a workspace [KSPLIT, M, N] that
// skinny_reduce_kernel adds in split order.  Nothing depends on timing.  No LDS staging of W:
// nothing of it is reused.
//
// NORM: the tokens come as the float32 residual stream and the RMSNorm before the product is
// folded in.  The product is linear, so  W (x * gain * inv) = inv * W (x * gain): the lanes
// feed bfloat16(x * gain) to the MFMAs, add up x^2 on the way (the workgroup sees all of K
// when there is no split over workgroups), and the epilogue scales each token's sums by
// inv = 1 / sqrt(mean(x^2) + eps), all in 32-bit  (n = x w / sqrt(mean(x^2) + eps),
// src/kernel/core/cpu.zig:38-48 of the reference).
// `block` of the workgroups along the outputs, `part` of `parts` along K.
// DEEP: two register sets of loads, for a workgroup that has a CU to itself.
template <int MT, int RG, int EPI, bool WT, int NORM, int NW, bool EMIT, bool DEEP = true>
__device__ __forceinline__ void skinny_product(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ Cv, int M,
    int N, int K, const SkinnyNorm& nrm, int block, int part_k, int parts) {
  constexpr int NSS = NORM == NORM_GIVEN ? NW * 4 : NW;
  __shared__ float part[NW][RG * MT][64][4];
  // a token's sums side by side: inv_rms reads four at a time, and the tokens' rows of NSS + 4
  // words begin in different banks (one by one, 32 sums made 8B decode steps 1 % slower)
  __shared__ __attribute__((aligned(16))) float ssum[MT][16][NSS + 4];
  const float* __restrict__ gain = nrm.gain;
  const float eps = nrm.eps;
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int n0 = block * (16 * RG);
  const int g = lane / 16;
  // plain layout: row pointer, k added later; pre-tiled: the lane's 16 bytes of chunk 0 of
  // the row group's first tile, tiles of 64 k are 1024 elements apart, chunk 1 is 512 on
  const bf16_t* wrow[RG];
#pragma unroll
  for (int r = 0; r < RG; ++r)
    wrow[r] = WT ? W + (size_t)(n0 / 16 + r) * (K / 64) * 1024 + lane * 8
                 : W + (size_t)min(n0 + r * 16 + lane % 16, N - 1) * K;
  const bf16_t* arow[MT];
  const float* xrow[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    arow[t] = A + (size_t)min(t * 16 + lane % 16, M - 1) * K;
    xrow[t] = (const float*)A + (size_t)min(t * 16 + lane % 16, M - 1) * K;
  }
  // lanes of tokens beyond M load nothing and feed zeros
  bool tok[MT];
  float ss[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    tok[t] = t * 16 + lane % 16 < M;
    ss[t] = 0.f;
  }

  f32x4_t acc[RG][MT];
#pragma unroll
  for (int r = 0; r < RG; ++r)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[r][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const u32x4_t zero = u32x4_t{0, 0, 0, 0};
  const int kstride = NW * 64 * parts;
  int k0 = (part_k * NW + wave) * 64;
  // What the epilogue reads from memory is asked for now, so that it has arrived when the
  // last weights have: the residual and the next norm's gains (wave 0 writes the outputs of
  // one row group and up to 16 tokens), and the producer's sums of squares.
  constexpr bool PRE_EPI = EMIT && RG * MT == 1;
  float4 pre_c = float4{0.f, 0.f, 0.f, 0.f}, pre_g = float4{0.f, 0.f, 0.f, 0.f};
  if (PRE_EPI && wave == 0 && parts == 1) {
    const int token = lane % 16, n = n0 + 4 * (lane / 16);
    if (token < M && n + 3 < N) {
      pre_c = *(const float4*)((const float*)Cv + (size_t)token * N + n);
      pre_g = *(const float4*)(nrm.gain_out + n);
    }
  }
  // The producer's sums of squares per 16 columns, [groups][16 tokens]: thread (p, j) takes groups p,
  // p + NSS, ... of token j.  Asked for behind the weights' first loads (in front of them the
  // addresses of 16 loads a thread, most of them beyond the groups of a narrow row, held the
  // weights up) and added up in norm_sums, which runs behind the last product; the rest, the NSS
  // sums of a token, follows in order of p (inv_rms).
  constexpr int SQ_PRE = NORM == NORM_GIVEN ? 16 : 1;
  float sqv[SQ_PRE];
  auto norm_ask = [&]() {
    if constexpr (NORM == NORM_GIVEN) {
      const int j = tid % 16, p = tid / 16;
#pragma unroll
      for (int i = 0; i < SQ_PRE; ++i) {
        sqv[i] = 0.f;
        if (i * NSS < nrm.sq_groups)             // (uniform)
          sqv[i] = nrm.sq_in[min(p + i * NSS, nrm.sq_groups - 1) * 16 + j];
      }
    }
  };
  auto norm_sums = [&]() {
    if constexpr (NORM == NORM_GIVEN) {
      const int j = tid % 16, p = tid / 16;
      float v = 0.f;
#pragma unroll
      for (int i = 0; i < SQ_PRE; ++i) v += p + i * NSS < nrm.sq_groups ? sqv[i] : 0.f;
      for (int gidx = p + SQ_PRE * NSS; gidx < nrm.sq_groups; gidx += NSS)
        v += nrm.sq_in[gidx * 16 + j];
      ssum[0][j][p] = v;
    }
  };
  // blocks of 64 of K that are this wave's (the same in its lanes: branches on it are scalar)
  const int cnt = __builtin_amdgcn_readfirstlane(k0 < K ? (K - 1 - k0) / kstride + 1 : 0);
  bool asked = false;                            // (the same in every wave)
  if constexpr (WT && NORM != NORM_FOLD && EPI_GLU(EPI) && RG * MT == 2) {
    // a short K: both blocks of a wave at once (the loop below waits for one before it asks for the
    // next: 6144 x 1024 with SwiGLU, one token, 5.7 -> 5.5 us; eight tokens 6.0 -> 5.6)
    if (K <= 2 * kstride) {
      asked = true;
      u32x4_t w0[2][RG], w1[2][RG], a0[2][MT], a1[2][MT];
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (u < cnt) {
          const int kk = k0 + u * kstride;
#pragma unroll
          for (int r = 0; r < RG; ++r) {
            const bf16_t* tile = wrow[r] + (size_t)(kk / 64) * 1024;
            w0[u][r] = __builtin_nontemporal_load((const u32x4_t*)tile);
            w1[u][r] = __builtin_nontemporal_load((const u32x4_t*)(tile + 512));
          }
#pragma unroll
          for (int t = 0; t < MT; ++t) {
            a0[u][t] = tok[t] ? *(const u32x4_t*)(arow[t] + kk + g * 16) : zero;
            a1[u][t] = tok[t] ? *(const u32x4_t*)(arow[t] + kk + g * 16 + 8) : zero;
          }
        }
      norm_ask();
#pragma unroll
      for (int u = 0; u < 2; ++u)
        if (u < cnt) {
#pragma unroll
          for (int r = 0; r < RG; ++r)
#pragma unroll
            for (int t = 0; t < MT; ++t) {
              acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  *(bf16x8_t*)&w0[u][r], *(bf16x8_t*)&a0[u][t], acc[r][t], 0, 0, 0);
              acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  *(bf16x8_t*)&w1[u][r], *(bf16x8_t*)&a1[u][t], acc[r][t], 0, 0, 0);
            }
        }
      k0 = K;
    }
  }
  if constexpr (WT && !DEEP && RG * MT == 1) {
    // four blocks in flight in one register set (other workgroups of the CU load meanwhile)
    static_assert(NORM == NORM_NONE, "plain products");
    for (; k0 + 3 * kstride < K; k0 += 4 * kstride) {
      u32x4_t w0[4], w1[4], a0[4], a1[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int kk = k0 + u * kstride;
        const bf16_t* tile = wrow[0] + (size_t)(kk / 64) * 1024;
        w0[u] = __builtin_nontemporal_load((const u32x4_t*)tile);
        w1[u] = __builtin_nontemporal_load((const u32x4_t*)(tile + 512));
        a0[u] = tok[0] ? *(const u32x4_t*)(arow[0] + kk + g * 16) : zero;
        a1[u] = tok[0] ? *(const u32x4_t*)(arow[0] + kk + g * 16 + 8) : zero;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(bf16x8_t*)&w0[u], *(bf16x8_t*)&a0[u],
                                                            acc[0][0], 0, 0, 0);
        acc[0][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(bf16x8_t*)&w1[u], *(bf16x8_t*)&a1[u],
                                                            acc[0][0], 0, 0, 0);
      }
    }
  }
  if constexpr (WT && DEEP && NORM != NORM_FOLD && (RG * MT == 1 || (RG * MT == 2 && !EPI_GLU(EPI)))) {
    asked = true;
    // Pre-tiled weights (no bounds checks; K % 64 == 0), up to two MFMA tiles per k-step:
    // batches of UNR k-steps in two register sets, the next batch asked for before the
    // MFMAs of the one that has arrived, so that a wave always has loads in flight.  The
    // paths below are laid out so that every wait has a known number of younger loads.
    // (Measured in a replayed graph at 1 and 8 tokens, 4096 x 4096, 4096 x 12288 and
    // 6144 x 4096: 0.1 to 1.0 us less than waiting for each batch before asking for the
    // next; the gate/up product with its three workgroups to a CU loses by it and keeps the
    // plain loop below.)
    constexpr int UNR = RG * MT == 1 ? 4 : 2;
    u32x4_t w0[2][UNR][RG], w1[2][UNR][RG], a0[2][UNR][MT], a1[2][UNR][MT];
    auto load_some = [&](auto BUF, auto COUNT, int kb) {
      constexpr int B = decltype(BUF)::value;
#pragma unroll
      for (int u = 0; u < decltype(COUNT)::value; ++u) {
        const int kk = kb + u * kstride;
#pragma unroll
        for (int r = 0; r < RG; ++r) {
          const bf16_t* tile = wrow[r] + (size_t)(kk / 64) * 1024;
          w0[B][u][r] = __builtin_nontemporal_load((const u32x4_t*)tile);
          w1[B][u][r] = __builtin_nontemporal_load((const u32x4_t*)(tile + 512));
        }
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          a0[B][u][t] = tok[t] ? *(const u32x4_t*)(arow[t] + kk + g * 16) : zero;
          a1[B][u][t] = tok[t] ? *(const u32x4_t*)(arow[t] + kk + g * 16 + 8) : zero;
        }
      }
    };
    auto compute_some = [&](auto BUF, auto COUNT) {
      constexpr int B = decltype(BUF)::value;
#pragma unroll
      for (int u = 0; u < decltype(COUNT)::value; ++u)
#pragma unroll
        for (int r = 0; r < RG; ++r)
#pragma unroll
          for (int t = 0; t < MT; ++t) {
            acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                *(bf16x8_t*)&w0[B][u][r], *(bf16x8_t*)&a0[B][u][t], acc[r][t], 0, 0, 0);
            acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                *(bf16x8_t*)&w1[B][u][r], *(bf16x8_t*)&a1[B][u][t], acc[r][t], 0, 0, 0);
          }
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    using All = std::integral_constant<int, UNR>;
    auto load = [&](auto BUF, int kb) { load_some(BUF, All{}, kb); };
    auto compute = [&](auto BUF) { compute_some(BUF, All{}); };
    // The blocks that make no whole batch come first, in the other register set, with the first
    // batch behind them: their loads are in flight together (one block after the other behind
    // the batches waited for each: 1024 outputs over K = 3072 5.7 -> 5.2 us).  A path of its own
    // for every number of them: where paths with and without such blocks meet again the compiler
    // waits for every load before the second batch is asked for (4096 x 4096, eight tokens 9.1 us
    // where they did, 8.8 here).
    const int nb = cnt / UNR, rem = cnt % UNR;
    const int bstride = UNR * kstride;
    auto go = [&](auto REM) {
      constexpr int R = decltype(REM)::value;
      if constexpr (R > 0) load_some(B1{}, REM, k0);
      k0 += R * kstride;
      if (nb == 0) {
        norm_ask();
        if constexpr (R > 0) compute_some(B1{}, REM);
        return;
      }
      load(B0{}, k0);
      norm_ask();
      if constexpr (R > 0) {
        __builtin_amdgcn_sched_barrier(0);
        compute_some(B1{}, REM);
        __builtin_amdgcn_sched_barrier(0);
      }
      int b = 0;
      for (; b + 2 < nb; b += 2) {
        load(B1{}, k0 + (b + 1) * bstride);
        __builtin_amdgcn_sched_barrier(0);
        compute(B0{});
        __builtin_amdgcn_sched_barrier(0);
        load(B0{}, k0 + (b + 2) * bstride);
        __builtin_amdgcn_sched_barrier(0);
        compute(B1{});
        __builtin_amdgcn_sched_barrier(0);
      }
      if (nb - b == 2) {
        load(B1{}, k0 + (b + 1) * bstride);
        __builtin_amdgcn_sched_barrier(0);
        compute(B0{});
        __builtin_amdgcn_sched_barrier(0);
        compute(B1{});
      } else {
        compute(B0{});
      }
    };
    if (rem == 0) go(std::integral_constant<int, 0>{});
    else if (rem == 1) go(std::integral_constant<int, 1>{});
    else if constexpr (UNR > 2) {
      if (rem == 2) go(std::integral_constant<int, 2>{});
      else go(std::integral_constant<int, 3>{});
    }
    k0 = K;
  }
  if (!asked) norm_ask();
  for (; k0 < K; k0 += kstride) {
    const int k = k0 + g * 16;
    u32x4_t w0[RG], w1[RG];
#pragma unroll
    for (int r = 0; r < RG; ++r) {
      if (WT) {       // N % 16 == 0 and K % 64 == 0: nothing to clamp, nothing to zero-fill
        const bf16_t* tile = wrow[r] + (size_t)(k0 / 64) * 1024;
        w0[r] = __builtin_nontemporal_load((const u32x4_t*)tile);
        w1[r] = __builtin_nontemporal_load((const u32x4_t*)(tile + 512));
      } else {
        w0[r] = (k < K) ? __builtin_nontemporal_load((const u32x4_t*)(wrow[r] + k)) : zero;
        w1[r] = (k + 8 < K) ? __builtin_nontemporal_load((const u32x4_t*)(wrow[r] + k + 8)) : zero;
      }
    }
    u32x4_t a0[MT], a1[MT];
    if (NORM == NORM_FOLD) {       // K % 64 == 0 here: 16 floats of x and of the gain per lane
      float4 gv[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) gv[c] = *(const float4*)(gain + k + 4 * c);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        float4 xv[4];
#pragma unroll
        for (int c = 0; c < 4; ++c)
          xv[c] = tok[t] ? *(const float4*)(xrow[t] + k + 4 * c) : float4{0.f, 0.f, 0.f, 0.f};
        uint32_t pk[8];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          ss[t] += xv[c].x * xv[c].x + xv[c].y * xv[c].y + xv[c].z * xv[c].z + xv[c].w * xv[c].w;
          pk[2 * c] = pack_bf16x2(xv[c].x * gv[c].x, xv[c].y * gv[c].y);
          pk[2 * c + 1] = pack_bf16x2(xv[c].z * gv[c].z, xv[c].w * gv[c].w);
        }
        a0[t] = u32x4_t{pk[0], pk[1], pk[2], pk[3]};
        a1[t] = u32x4_t{pk[4], pk[5], pk[6], pk[7]};
      }
    } else {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        a0[t] = (tok[t] && k < K) ? *(const u32x4_t*)(arow[t] + k) : zero;
        a1[t] = (tok[t] && k + 8 < K) ? *(const u32x4_t*)(arow[t] + k + 8) : zero;
      }
    }
#pragma unroll
    for (int r = 0; r < RG; ++r)
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *(bf16x8_t*)&w0[r], *(bf16x8_t*)&a0[t], acc[r][t], 0, 0, 0);
        acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            *(bf16x8_t*)&w1[r], *(bf16x8_t*)&a1[t], acc[r][t], 0, 0, 0);
      }
  }
#pragma unroll
  for (int r = 0; r < RG; ++r)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) part[wave][r * MT + t][lane][e] = acc[r][t][e];
  if (NORM == NORM_FOLD) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      float v = ss[t];
      v = apart_sum<16>(v);
      v = apart_sum<32>(v);
      if (lane < 16) ssum[t][lane][wave] = v;
    }
  }
  norm_sums();
  __syncthreads();
  // the token's 1 / sqrt(mean(x^2) + eps): the partial sums in a fixed order
  auto inv_rms = [&](int t, int j) {
    static_assert(NSS % 4 == 0, "read four at a time");
    if (NORM == NORM_NONE) return 1.0f;
    float tot = 0.f;
#pragma unroll
    for (int w = 0; w < NSS; w += 4) {
      const float4 v = *(const float4*)&ssum[t][j][w];
      tot += v.x;
      tot += v.y;
      tot += v.z;
      tot += v.w;
    }
    return 1.0f / sqrtf(tot / (float)K + eps);
  };
  if (EPI_GLU(EPI)) {
    // row groups alternate gate / up: the pair (2 p, 2 p + 1) gives 16 outputs per token
    for (int item = tid; item < (RG / 2) * MT * 64; item += NW * 64) {
      const int pt = item / 64, l = item % 64;
      const int p = pt / MT, t = pt % MT;
      float g[4] = {0.f, 0.f, 0.f, 0.f}, u[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          g[e] += part[w][(2 * p) * MT + t][l][e];
          u[e] += part[w][(2 * p + 1) * MT + t][l][e];
        }
      const int token = t * 16 + l % 16;
      if (token < M) {
        const float inv = inv_rms(t, l % 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int n = n0 / 2 + p * 16 + 4 * (l / 16) + e;      // column of the [M, N / 2] output
          if (2 * n < N) {
            float gv = g[e] * inv, uv = u[e] * inv;
            if (EPI == EPI_GEGLU && nrm.glu_bias != nullptr) {
              const float* b = nrm.glu_bias + n0 + p * 32 + 4 * (l / 16) + e;
              gv += b[0];
              uv += b[16];
            }
            ((bf16_t*)Cv)[(size_t)token * (N / 2) + n] = float_to_bf16(glu_f<EPI>(gv, uv));
          }
        }
      }
    }
    return;
  }
  for (int item = tid; item < RG * MT * 64; item += NW * 64) {
    const int rt = item / 64, l = item % 64;
    const int r = rt / MT, t = rt % MT;
    float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w)
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] += part[w][rt][l][e];
    // D[i][j]: i = 4 * (l / 16) + e is the W row (output feature), j = l % 16 the token
    const int token = t * 16 + l % 16;
    float sq = 0.f;
    if (token < M) {
      const float inv = inv_rms(t, l % 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] *= inv;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = n0 + r * 16 + 4 * (l / 16) + e;
        if (n < N) {
          if (parts > 1) {
            ((float*)Cv)[((size_t)part_k * M + token) * N + n] = s[e];   // workspace
          } else {
            const size_t off = (size_t)token * N + n;
            if (EPI == EPI_STORE_BF16) {
              ((bf16_t*)Cv)[off] = float_to_bf16(s[e]);
            } else if (EPI == EPI_ACT) {
              ((bf16_t*)Cv)[off] =
                  float_to_bf16(activation_value(bf16_to_float(float_to_bf16(s[e])), nrm.act));
            } else if (EPI == EPI_STORE_F32 || (EPI == EPI_MANY && nrm.act == MANY_F32)) {
              ((float*)Cv)[off] = s[e];
            } else if (EPI == EPI_MANY) {
              const bf16_t v = float_to_bf16(s[e]);
              ((bf16_t*)Cv)[off] = nrm.act == MANY_BF16
                  ? v : float_to_bf16(activation_value(bf16_to_float(v), nrm.act));
            } else {
              const float old = PRE_EPI ? ((const float*)&pre_c)[e] : ((float*)Cv)[off];
              const float v = old + s[e];
              ((float*)Cv)[off] = v;
              if (EMIT) {   // what the RMSNorm after this sum needs: v * gain, and v^2
                const float go = PRE_EPI ? ((const float*)&pre_g)[e] : nrm.gain_out[n];
                nrm.xg_out[off] = float_to_bf16(v * go);
                sq += v * v;
              }
            }
          }
        }
      }
    }
    if (EMIT) {
      // the 16 columns of this row group: 4 per lane, lanes l, l + 16, l + 32, l + 48 of a
      // token; every item is a whole wave here (RG * MT * 64 items, NW * 64 threads)
      sq = apart_sum<16>(sq);
      sq = apart_sum<32>(sq);
      if (l < 16) nrm.sq_out[(size_t)(n0 / 16 + r) * 16 + l] = sq;
    }
  }
}

template <int MT, int RG, int EPI, bool WT, int NORM, int NW = 8, bool EMIT = false>
__global__ __launch_bounds__(NW * 64) void gemm_bf16_skinny_kernel(
    const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, void* __restrict__ Cv, int M,
    int N, int K, SkinnyNorm nrm) {
  skinny_product<MT, RG, EPI, WT, NORM, NW, EMIT>(A, W, Cv, M, N, K, nrm, blockIdx.x, blockIdx.y,
                                                  gridDim.y);
}

// Several products of up to 16 tokens over the same K in one launch, a row group of 16 a
// workgroup: products that read the same rows or lie ready together, each too narrow for the chip
// and as long as a launch.  In traces, 16 tokens: four of 2048 x 2048 and one of 16 x 2048 with a tanh
// 4 x 5.6 + 6.3 + 3.7 -> 10.5 us, 6144 and 16 x 2048 7.6 + 6.3 -> 9.6; 8 tokens: 3072, 6144 and 32 x
// 2048 5.3 + 7.1 + 5.9 -> 10.2, twice 2048 x 2048 10.2 -> 5.8.  Two workgroups and more a CU in one
// register set: with the streaming kernel's two sets, one a CU, the first took 16.2 us.
// Every product's bits are those of a launch of its own.
#define ZF_MANY_PRODUCTS 6
struct ManyProducts {
  const bf16_t* a[ZF_MANY_PRODUCTS];
  const bf16_t* w[ZF_MANY_PRODUCTS];
  void* c[ZF_MANY_PRODUCTS];
  int n[ZF_MANY_PRODUCTS];
  int tiled[ZF_MANY_PRODUCTS];
  int act[ZF_MANY_PRODUCTS];       // an activation's number, MANY_BF16 or MANY_F32
  int end[ZF_MANY_PRODUCTS];       // workgroups of this product and the ones before
  int count;
};
__global__ __launch_bounds__(512, 4) void gemm_bf16_many_kernel(ManyProducts p, int M, int K) {
  int i = 0, first = 0;
  while (i + 1 < p.count && (int)blockIdx.x >= p.end[i]) first = p.end[i++];
  SkinnyNorm nrm{};
  nrm.act = p.act[i];
  if (p.tiled[i])
    skinny_product<1, 1, EPI_MANY, true, NORM_NONE, 8, false, false>(p.a[i], p.w[i], p.c[i], M, p.n[i], K, nrm,
                                                              blockIdx.x - first, 0, 1);
  else
    skinny_product<1, 1, EPI_MANY, false, NORM_NONE, 8, false, false>(p.a[i], p.w[i], p.c[i], M, p.n[i], K,
                                                               nrm, blockIdx.x - first, 0, 1);
}

// `products`: count, n, tiled and act as above, end filled here; every operand bfloat16 with K
// contiguous, K % 8 == 0 (pre-tiled: K % 64 == 0, n % 16 == 0) and 16-byte aligned.
extern "C" int zf_gemm_bf16_many(ManyProducts* products, int M, int K, hipStream_t stream) {
  if (M <= 0) return 0;
  if (M > 16 || K <= 0 || K % 8 != 0 || products->count < 1 || products->count > ZF_MANY_PRODUCTS)
    return -3;
  int end = 0;
  for (int i = 0; i < products->count; ++i) {
    if (products->n[i] <= 0 || products->act[i] > 4 ||
        (products->tiled[i] && (K % 64 != 0 || products->n[i] % 16 != 0)) ||
        (((uintptr_t)products->a[i] | (uintptr_t)products->w[i]) % 16) != 0)
      return -3;
    products->end[i] = end += (products->n[i] + 15) / 16;
  }
  hipLaunchKernelGGL(gemm_bf16_many_kernel, dim3(end), dim3(512), 0, stream, *products, M, K);
  return (int)hipGetLastError();
}

// VEC: four outputs a thread with 16-byte loads (M * N a multiple of 4, so that every
// partial starts on a 16-byte boundary); else one output a thread.
template <int EPI, bool VEC>
__global__ void skinny_reduce_kernel(const float* __restrict__ ws, void* __restrict__ Cv,
                                     size_t mn, int ksplit) {
  if (VEC) {
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
    if (i >= mn) return;
    float4 s = float4{0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < ksplit; ++k) {
      const float4 p = *(const float4*)(ws + (size_t)k * mn + i);
      s.x += p.x; s.y += p.y; s.z += p.z; s.w += p.w;
    }
    if (EPI == EPI_STORE_BF16) {
      *(u32x2_t*)((bf16_t*)Cv + i) = u32x2_t{pack_bf16x2(s.x, s.y), pack_bf16x2(s.z, s.w)};
    } else if (EPI == EPI_STORE_F32) {
      *(float4*)((float*)Cv + i) = s;
    } else {
      float4* dst = (float4*)((float*)Cv + i);
      const float4 old = *dst;
      *dst = float4{old.x + s.x, old.y + s.y, old.z + s.z, old.w + s.w};
    }
    return;
  }
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= mn) return;
  float s = 0.f;
  for (int k = 0; k < ksplit; ++k) s += ws[(size_t)k * mn + i];
  if (EPI == EPI_STORE_BF16)
    ((bf16_t*)Cv)[i] = float_to_bf16(s);
  else if (EPI == EPI_STORE_F32)
    ((float*)Cv)[i] = s;
  else
    ((float*)Cv)[i] += s;
}

static int launch_reduce(const void* ws, void* C, int M, int N, int ksplit, int epi,
                         hipStream_t stream) {
  const size_t mn = (size_t)M * N;
  const bool vec = mn % 4 == 0;
  const unsigned blocks = (unsigned)(((vec ? mn / 4 : mn) + 255) / 256);
#define ZF_REDUCE(E)                                                                           \
  do {                                                                                         \
    if (vec)                                                                                   \
      hipLaunchKernelGGL((skinny_reduce_kernel<E, true>), dim3(blocks), dim3(256), 0, stream,  \
                         (const float*)ws, C, mn, ksplit);                                     \
    else                                                                                       \
      hipLaunchKernelGGL((skinny_reduce_kernel<E, false>), dim3(blocks), dim3(256), 0, stream, \
                         (const float*)ws, C, mn, ksplit);                                     \
  } while (0)
  if (epi == EPI_STORE_BF16) ZF_REDUCE(EPI_STORE_BF16);
  else if (epi == EPI_STORE_F32) ZF_REDUCE(EPI_STORE_F32);
  else if (epi == EPI_ACC_F32) ZF_REDUCE(EPI_ACC_F32);
  else return -3;
#undef ZF_REDUCE
  return (int)hipGetLastError();
}

// The split-K partials of a residual sum whose reader is an RMSNorm: one workgroup per token
// adds the partials in split order into the 32-bit residual row (as skinny_reduce_kernel
// does), keeps the row in registers, and writes the norm of the sum,
// n = x * gain / sqrt(mean(x^2) + eps) (src/kernel/core/cpu.zig:38-48 of the reference), as
// bfloat16: the reduce and the norm kernel in one, the row read once.  N % 4 == 0, N <= 8192
// (8 float4 per thread with 256 threads; wider rows get up to 1024 threads).
template <typename TO>
__global__ __launch_bounds__(1024) void reduce_sum_norm_kernel(
    const float* __restrict__ ws, float* __restrict__ C, const float* __restrict__ gain,
    TO* __restrict__ normed, int M, int N, int ksplit, float eps) {
  __shared__ float red[16];
  const int m = blockIdx.x, n4 = N / 4, nt = blockDim.x;      // 8 * nt >= n4
  float4* row = (float4*)(C + (size_t)m * N);
  const float4* part = (const float4*)(ws + (size_t)m * N);
  const size_t kstride = (size_t)M * n4;
  float4 v[8];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int c = threadIdx.x + i * nt;
    v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (c < n4) {
      float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 8
      for (int k = 0; k < ksplit; ++k) {          // independent loads, added in split order
        const float4 p = part[k * kstride + c];
        s.x += p.x; s.y += p.y; s.z += p.z; s.w += p.w;
      }
      const float4 old = row[c];
      v[i] = make_float4(old.x + s.x, old.y + s.y, old.z + s.z, old.w + s.w);
      row[c] = v[i];
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) ss += v[i].x * v[i].x + v[i].y * v[i].y + v[i].z * v[i].z + v[i].w * v[i].w;
  ss = block_sum(ss, red);
  const float inv = 1.0f / sqrtf(ss / (float)N + eps);
  TO* o = normed + (size_t)m * N;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int c = threadIdx.x + i * nt;
    if (c < n4) {
      const float4 g = ((const float4*)gain)[c];
      const float4 y = make_float4(v[i].x * inv * g.x, v[i].y * inv * g.y, v[i].z * inv * g.z,
                                   v[i].w * inv * g.w);
      if constexpr (std::is_same<TO, float>::value)
        *(float4*)(o + 4 * c) = y;
      else
        *(u32x2_t*)(o + 4 * c) = u32x2_t{pack_bf16x2(y.x, y.y), pack_bf16x2(y.z, y.w)};
    }
  }
}

// C += A W^T in 32-bit with ksplit >= 2 workgroups along K, and normed = bfloat16 RMSNorm of
// the sum's rows, from the kernel that adds the partials.  M <= 128: the kernels for 17 to 128
// tokens; above: 128 x 128 tiles.  W pre-tiled; ws: float32 [ksplit, M, N].
extern "C" int zf_gemm_bf16_splitk_sum_norm(const void* A, const void* W, void* C, void* ws,
                                            const float* gain, float eps, void* normed, int M,
                                            int N, int K, int ksplit, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (ksplit < 2 || ksplit > 64 || N % 16 != 0 || N > 8192 || ws == nullptr) return -3;
  int rc;
  if (M <= 32)
    rc = launch_tile_wdirect<32, 128, 32, 32, 256>(A, W, C, M, N, K, EPI_ACC_F32, stream, ws,
                                                   ksplit, false);
  else if (M <= 64)
    rc = launch_tile_wdirect<64, 128, 64, 32, 128>(A, W, C, M, N, K, EPI_ACC_F32, stream, ws,
                                                   ksplit, false);
  else if (K % 128 == 0)
    rc = launch_tile_wdirect<128, 128, 128, 32, 128>(A, W, C, M, N, K, EPI_ACC_F32, stream, ws,
                                                     ksplit, false);
  else
    rc = launch_tile_wdirect<128, 128, 64, 64>(A, W, C, M, N, K, EPI_ACC_F32, stream, ws, ksplit,
                                               false);
  if (rc != 0) return rc;
  // a thread per 4 columns up to 1024 threads: every load of a row is in flight at once
  const int threads = N / 4 >= 1024 ? 1024 : (N / 4 > 256 ? 512 : 256);
  hipLaunchKernelGGL(reduce_sum_norm_kernel<bf16_t>, dim3(M), dim3(threads), 0, stream, (const float*)ws,
                     (float*)C, gain, (bf16_t*)normed, M, N, ksplit, eps);
  return (int)hipGetLastError();
}

// out = A W^T (accumulate: out += A W^T), all float32, up to 64 rows, one workgroup a span of K and
// row group; ws: float32 [F32_SPANS, M, N].  The bits of zf_gemm_f32.  K and N multiples of 4 and
// 16-byte aligned operands.  With a gain (accumulate only, N <= 8192) normed = the rows' RMSNorm,
// the bits of zf_rmsnorm (its 256 threads a row), from the kernel that adds the spans.
extern "C" int zf_gemm_f32_spans(const float* A, const float* W, float* C, float* ws, int M, int N,
                                 int K, int accumulate, const float* gain, float eps, float* normed,
                                 hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 64 || K <= 0 || K % 4 != 0 || N % 4 != 0 || ws == nullptr ||
      (((uintptr_t)A | (uintptr_t)W | (uintptr_t)C | (uintptr_t)ws | (uintptr_t)gain |
        (uintptr_t)normed) % 16) != 0)
    return -1;
  if (gain != nullptr && (!accumulate || N > 8192)) return -1;
  const dim3 grid((N + 15) / 16, F32_SPANS);
  const int span = f32_span(K);
  if (M <= 16)
    hipLaunchKernelGGL(gemm_f32_spans_kernel<1>, grid, dim3(64), 0, stream, A, W, ws, M, N, K, span);
  else if (M <= 32)
    hipLaunchKernelGGL(gemm_f32_spans_kernel<2>, grid, dim3(64), 0, stream, A, W, ws, M, N, K, span);
  else
    hipLaunchKernelGGL(gemm_f32_spans_kernel<4>, grid, dim3(64), 0, stream, A, W, ws, M, N, K, span);
  if (gain != nullptr) {
    hipLaunchKernelGGL(reduce_sum_norm_kernel<float>, dim3(M), dim3(256), 0, stream, ws, C, gain,
                       normed, M, N, F32_SPANS, eps);
    return (int)hipGetLastError();
  }
  return launch_reduce(ws, C, M, N, F32_SPANS, accumulate ? EPI_ACC_F32 : EPI_STORE_F32, stream);
}

// The product with 128 x 256 tiles split along K (for a long K on a narrow output at several
// hundred tokens) and the kernel that adds the partials.  (K / 64) % (2 ksplit) == 0; ws:
// float32 [ksplit, M, N]; epi: store bf16, store f32 or add into f32.
extern "C" int zf_gemm_bf16_wide_splitk(const void* A, const void* W, void* C, void* ws, int M,
                                        int N, int K, int epi, int ksplit, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (ksplit < 2 || ksplit > 64 || epi == EPI_SWIGLU || ws == nullptr) return -3;
  return launch_tile_wdirect<128, 256, 128, 64, TK, true, true>(A, W, C, M, N, K, epi, stream, ws,
                                                                ksplit);
}

// The same with 128 x 256 tiles (two workgroups to a CU, no two waves load the same part of
// W): for a long K on a narrow output, where few of these tiles, each split many times, run
// faster than the 128 x 128 tiles.  (K / 64) % (2 ksplit) == 0.
extern "C" int zf_gemm_bf16_wide_splitk_sum_norm(const void* A, const void* W, void* C, void* ws,
                                                 const float* gain, float eps, void* normed,
                                                 int M, int N, int K, int ksplit,
                                                 hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (ksplit < 2 || ksplit > 64 || N % 16 != 0 || N > 8192 || ws == nullptr) return -3;
  const int rc = launch_tile_wdirect<128, 256, 128, 64, TK, true, true>(
      A, W, C, M, N, K, EPI_ACC_F32, stream, ws, ksplit, false);
  if (rc != 0) return rc;
  const int threads = N / 4 >= 1024 ? 1024 : (N / 4 > 256 ? 512 : 256);
  hipLaunchKernelGGL(reduce_sum_norm_kernel<bf16_t>, dim3(M), dim3(threads), 0, stream, (const float*)ws,
                     (float*)C, gain, (bf16_t*)normed, M, N, ksplit, eps);
  return (int)hipGetLastError();
}

// The product through the ring's tiles (30 to 32 as zf_gemm_bf16_tile's variants, 33: 128 x 256) split along K:
// ws float32 [ksplit, M, N], then the kernel that adds the partials: with a gain C += and normed = bfloat16
// RMSNorm of the rows (N <= 8192), else the epilogue (store bf16, store f32, add into f32).
extern "C" int zf_gemm_bf16_ring_splitk(const void* A, const void* W, void* C, void* ws, int M, int N, int K,
                                        int epi, int shape, int ksplit, const float* gain, float eps,
                                        void* normed, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (N % 16 != 0 || K % 64 != 0 || ksplit < 2 || ksplit > 64 || ksplit > K / 64 || ws == nullptr || EPI_GLU(epi))
    return -3;
  if (gain != nullptr && (N > 8192 || epi != EPI_ACC_F32)) return -3;
  int rc = -4;
  if (shape == 30) rc = launch_ring_parts<128, 128>(A, W, ws, M, N, K, ksplit, stream);
  else if (shape == 31) rc = launch_ring_parts<128, 64>(A, W, ws, M, N, K, ksplit, stream);
  else if (shape == 32) rc = launch_ring_parts<64, 64>(A, W, ws, M, N, K, ksplit, stream);
  else if (shape == 33) rc = launch_ring_parts<128, 256>(A, W, ws, M, N, K, ksplit, stream);
  if (rc != 0) return rc;
  if (gain == nullptr) return launch_reduce(ws, C, M, N, ksplit, epi, stream);
  const int threads = N / 4 >= 1024 ? 1024 : (N / 4 > 256 ? 512 : 256);
  hipLaunchKernelGGL(reduce_sum_norm_kernel<bf16_t>, dim3(M), dim3(threads), 0, stream, (const float*)ws,
                     (float*)C, gain, (bf16_t*)normed, M, N, ksplit, eps);
  return (int)hipGetLastError();
}

// C += A W^T in 32-bit through 256 x 256 tiles split along K: ws float32 [ksplit, M, N], K of at
// least ksplit times 128.  With a gain normed = bfloat16 RMSNorm of the rows (N <= 8192), from the
// kernel that adds the partials.
extern "C" int zf_gemm_bf16_tile256_splitk(const void* A, const void* W, void* C, void* ws, int M,
                                           int N, int K, int ksplit, const float* gain, float eps,
                                           void* normed, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (N % 16 != 0 || K % 128 != 0 || ksplit < 2 || ksplit > K / 128 || ws == nullptr) return -3;
  if (gain != nullptr && N > 8192) return -3;
  const int tiles_m = (M + 255) / 256, tiles_n = (N + 255) / 256;
  hipLaunchKernelGGL((gemm_bf16_tile256_kernel<256, EPI_STORE_F32, T256_SPLIT>),
                     dim3(tiles_m * tiles_n, ksplit), dim3(256), 0, stream, (const bf16_t*)A,
                     (const bf16_t*)W, ws, M, N, K, tiles_m, tiles_n, nullptr, 0, 1, (float*)nullptr);
  if (gain == nullptr) return launch_reduce(ws, C, M, N, ksplit, EPI_ACC_F32, stream);
  const int threads = N / 4 >= 1024 ? 1024 : (N / 4 > 256 ? 512 : 256);
  hipLaunchKernelGGL(reduce_sum_norm_kernel<bf16_t>, dim3(M), dim3(threads), 0, stream,
                     (const float*)ws, (float*)C, gain, (bf16_t*)normed, M, N, ksplit, eps);
  return (int)hipGetLastError();
}

template <int MT, int RG, bool WT, int NORM = NORM_NONE, bool EMIT = false>
static int launch_skinny(const void* A, const void* W, void* C, void* ws, int M, int N, int K,
                         int epi, int ksplit, hipStream_t stream, SkinnyNorm nrm = SkinnyNorm{},
                         bool reduce = true) {
  constexpr int NW = 8;
  const dim3 grid((N + 16 * RG - 1) / (16 * RG), ksplit), block(NW * 64);
  void* dst = ksplit > 1 ? ws : C;
  if (NORM != NORM_NONE && (ksplit != 1 || epi == EPI_ACC_F32)) return -3;
  if (EMIT) {
    if (ksplit != 1 || epi != EPI_ACC_F32) return -3;
    hipLaunchKernelGGL((gemm_bf16_skinny_kernel<MT, RG, EPI_ACC_F32, WT, NORM_NONE, NW, true>), grid,
                       block, 0, stream, (const bf16_t*)A, (const bf16_t*)W, dst, M, N, K, nrm);
    return (int)hipGetLastError();
  }
  if (epi == EPI_GEGLU) {
    if constexpr (WT && NORM == NORM_NONE) {
      if (RG < 2 || ksplit != 1 || N % 32 != 0) return -3;
      hipLaunchKernelGGL((gemm_bf16_skinny_kernel<MT, (RG < 2 ? 2 : RG), EPI_GEGLU, WT, NORM, NW>),
                         grid, block, 0, stream, (const bf16_t*)A, (const bf16_t*)W, dst, M, N, K, nrm);
      return (int)hipGetLastError();
    }
    return -3;
  }
  if (epi == EPI_SWIGLU) {
    if (RG < 2 || ksplit != 1 || N % 32 != 0) return -3;
    hipLaunchKernelGGL((gemm_bf16_skinny_kernel<MT, (RG < 2 ? 2 : RG), EPI_SWIGLU, WT, NORM, NW>), grid,
                       block, 0, stream, (const bf16_t*)A, (const bf16_t*)W, dst, M, N, K, nrm);
    return (int)hipGetLastError();
  }
  if (epi == EPI_STORE_BF16)
    hipLaunchKernelGGL((gemm_bf16_skinny_kernel<MT, RG, EPI_STORE_BF16, WT, NORM, NW>), grid, block, 0,
                       stream, (const bf16_t*)A, (const bf16_t*)W, dst, M, N, K, nrm);
  else if (epi == EPI_STORE_F32)
    hipLaunchKernelGGL((gemm_bf16_skinny_kernel<MT, RG, EPI_STORE_F32, WT, NORM, NW>), grid, block, 0,
                       stream, (const bf16_t*)A, (const bf16_t*)W, dst, M, N, K, nrm);
  else
    hipLaunchKernelGGL((gemm_bf16_skinny_kernel<MT, RG, EPI_ACC_F32, WT, NORM_NONE, NW>), grid, block, 0,
                       stream, (const bf16_t*)A, (const bf16_t*)W, dst, M, N, K, nrm);
  if (ksplit > 1 && reduce) return launch_reduce(ws, C, M, N, ksplit, epi, stream);
  return (int)hipGetLastError();
}

// C += A W^T in 32-bit by the weight-streaming kernel with ksplit >= 2 workgroups along K, and
// normed = bfloat16 RMSNorm of the sum's rows from the kernel that adds the partials: for
// narrow outputs whose row groups alone leave CUs idle (320 of them on 256 CUs).  M <= 64,
// W pre-tiled, N a multiple of 16 * rg; ws: float32 [ksplit, M, N].
extern "C" int zf_gemm_bf16_skinny_sum_norm(const void* A, const void* W, void* C, void* ws,
                                            const float* gain, float eps, void* normed, int M,
                                            int N, int K, int rg, int ksplit,
                                            hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 64 || ksplit < 2 || ksplit > 16 || K % 64 != 0 || N % (16 * rg) != 0 || N > 8192 ||
      ws == nullptr)
    return -3;
  const int mt = (M + 15) / 16;
  int rc = -4;
#define ZF_SKS(MT, RG)                                                                         \
  rc = launch_skinny<MT, RG, true>(A, W, C, ws, M, N, K, EPI_ACC_F32, ksplit, stream,          \
                                   SkinnyNorm{}, false)
  if (rg == 1) { if (mt == 1) ZF_SKS(1, 1); else if (mt == 2) ZF_SKS(2, 1); else if (mt == 3) ZF_SKS(3, 1); else ZF_SKS(4, 1); }
  if (rg == 2) { if (mt == 1) ZF_SKS(1, 2); else if (mt == 2) ZF_SKS(2, 2); else if (mt == 3) ZF_SKS(3, 2); else ZF_SKS(4, 2); }
  if (rg == 4) { if (mt == 1) ZF_SKS(1, 4); else if (mt == 2) ZF_SKS(2, 4); else if (mt == 3) ZF_SKS(3, 4); else ZF_SKS(4, 4); }
#undef ZF_SKS
  if (rc != 0) return rc;
  const int threads = N / 4 >= 1024 ? 1024 : (N / 4 > 256 ? 512 : 256);
  hipLaunchKernelGGL(reduce_sum_norm_kernel<bf16_t>, dim3(M), dim3(threads), 0, stream, (const float*)ws,
                     (float*)C, gain, (bf16_t*)normed, M, N, ksplit, eps);
  return (int)hipGetLastError();
}

// rg: row groups of 16 per workgroup (1, 2 or 4); ksplit: workgroups along K (1..16), which
// needs a float32 workspace of ksplit * M * N elements when > 1; w_tiled: W is pre-tiled
// (N % 16 == 0, K % 64 == 0, N a multiple of 16 * rg).  keep_parts: ws keeps the parts
// [ksplit, M, N] for a kernel of the caller's that adds them.
extern "C" int zf_gemm_bf16_skinny(const void* A, const void* W, void* C, void* ws, int M, int N,
                                   int K, int epi, int rg, int ksplit, int w_tiled,
                                   int keep_parts, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K % 8 != 0 || M > 64 || ksplit < 1 || ksplit > 16 || (ksplit > 1 && ws == nullptr))
    return -3;
  if (keep_parts && (ksplit < 2 || epi != EPI_STORE_F32)) return -3;
  const int mt = (M + 15) / 16;
  if (w_tiled && (N % (16 * rg) != 0 || K % 64 != 0)) return -3;
#define ZF_SK(MT, RG)                                                                         \
  return w_tiled ? launch_skinny<MT, RG, true>(A, W, C, ws, M, N, K, epi, ksplit, stream, SkinnyNorm{}, !keep_parts) \
                 : launch_skinny<MT, RG, false>(A, W, C, ws, M, N, K, epi, ksplit, stream, SkinnyNorm{}, !keep_parts)
  if (rg == 1) { if (mt == 1) ZF_SK(1, 1); if (mt == 2) ZF_SK(2, 1); if (mt == 3) ZF_SK(3, 1); ZF_SK(4, 1); }
  if (rg == 2) { if (mt == 1) ZF_SK(1, 2); if (mt == 2) ZF_SK(2, 2); if (mt == 3) ZF_SK(3, 2); ZF_SK(4, 2); }
  if (rg == 4) { if (mt == 1) ZF_SK(1, 4); if (mt == 2) ZF_SK(2, 4); if (mt == 3) ZF_SK(3, 4); ZF_SK(4, 4); }
#undef ZF_SK
  return -4;
}

// C [M <= 16, N] = act(bfloat16(A W^T)) as bfloat16 by the weight-streaming kernel, W pre-tiled; the
// bits of the product and of the activation's own kernel behind it.  That kernel moves 0.5 MB at
// 16 tokens and 7168 outputs and takes 4.7 us of a decode step; here the values are in registers
// (product and activation 12.8 -> 8.4 us).
extern "C" int zf_gemm_bf16_act(const void* A, const void* W, void* C, int M, int N, int K, int rg,
                                int kind, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 16 || K % 64 != 0 || N % (16 * rg) != 0 || kind < 0 || kind > 4) return -3;
  SkinnyNorm nrm{};
  nrm.act = kind;
#define ZF_ACT(RG)                                                                              \
  hipLaunchKernelGGL((gemm_bf16_skinny_kernel<1, RG, EPI_ACT, true, NORM_NONE, 8>),             \
                     dim3(N / (16 * RG)), dim3(512), 0, stream, (const bf16_t*)A,               \
                     (const bf16_t*)W, C, M, N, K, nrm);                                        \
  return (int)hipGetLastError()
  if (rg == 1) { ZF_ACT(1); }
  if (rg == 2) { ZF_ACT(2); }
  if (rg == 4) { ZF_ACT(4); }
#undef ZF_ACT
  return -4;
}

// out[M, N / 2] = gelu(A Wg^T + bg) * (A Wu^T + bu) with W's and bias's rows alternating in groups
// of 16 (EPI_GEGLU), W pre-tiled.  way: 0 tiles (number: the variant of zf_gemm_bf16_tile), 1 the
// 128 x 256 tiles with the last round split along K (number: whole, split), 2 for 17 to 128
// tokens, 3 weight streaming (number: rg), 4 the 256 x 256 tiles with the last round split (number: whole).
extern "C" int zf_gemm_geglu(const void* A, const void* W, const float* bias, void* C, void* ws,
                             int M, int N, int K, int way, int number, int split,
                             hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (N % 32 != 0 || K % 64 != 0) return -3;
  constexpr int E = EPI_GEGLU;
  if (way == 1) {
    if (K % (2 * TK) == 0 && (K / TK) % (2 * split) == 0)
      return launch_tile_tail<true>(A, W, C, ws, M, N, K, E, number, split, stream, bias);
    return launch_tile_tail<false>(A, W, C, ws, M, N, K, E, number, split, stream, bias);
  }
  if (way == 4) return launch_tile256_tail(A, W, C, ws, M, N, K, E, number, split, stream, bias);
  if (way == 2) {
    if (M > 128) return -3;
    if (M <= 32)
      return launch_tile_wdirect<32, 128, 32, 32, 256>(A, W, C, M, N, K, E, stream, nullptr, 1, true, bias);
    if (M <= 64)
      return launch_tile_wdirect<64, 128, 64, 32, 128>(A, W, C, M, N, K, E, stream, nullptr, 1, true, bias);
    return launch_tile_wdirect<128, 128, 128, 32, 128>(A, W, C, M, N, K, E, stream, nullptr, 1, true, bias);
  }
  if (way == 3) {
    if (M > 64 || N % (16 * number) != 0) return -3;
    const int mt = (M + 15) / 16;
    SkinnyNorm nrm{};
    nrm.glu_bias = bias;
#define ZF_GSK(MT, RG) \
  return launch_skinny<MT, RG, true>(A, W, C, nullptr, M, N, K, E, 1, stream, nrm)
    if (number == 2) { if (mt == 1) ZF_GSK(1, 2); if (mt == 2) ZF_GSK(2, 2); if (mt == 3) ZF_GSK(3, 2); ZF_GSK(4, 2); }
    if (number == 4) { if (mt == 1) ZF_GSK(1, 4); if (mt == 2) ZF_GSK(2, 4); if (mt == 3) ZF_GSK(3, 4); ZF_GSK(4, 4); }
#undef ZF_GSK
    return -4;
  }
  switch (number) {
    case 6:
      if ((long long)((M + 127) / 128) * ((N + 127) / 128) >= 384)
        return launch_tile_wdirect<128, 128, 64, 64, TK, false, true>(A, W, C, M, N, K, E, stream, nullptr, 1, true, bias);
      return launch_tile_wdirect<128, 128, 64, 64>(A, W, C, M, N, K, E, stream, nullptr, 1, true, bias);
    case 10:
      if (K % (2 * TK) == 0)
        return launch_tile_wdirect<128, 256, 128, 64, TK, true, true>(A, W, C, M, N, K, E, stream, nullptr, 1, true, bias);
      return launch_tile_wdirect<128, 256, 128, 64, TK, false, true>(A, W, C, M, N, K, E, stream, nullptr, 1, true, bias);
    case 12:
      return launch_tile_wdirect<128, 256, 128, 64, TK, true, true, 2>(A, W, C, M, N, K, E, stream, nullptr, 1, true, bias);
    case 16:
      return launch_tile_wdirect<128, 128, 128, 32, 128>(A, W, C, M, N, K, E, stream, nullptr, 1, true, bias);
    case 20: return launch_tile256<256>(A, W, C, M, N, K, E, stream, bias);
    case 21: return launch_tile256<192>(A, W, C, M, N, K, E, stream, bias);
    case 30: return launch_ring<128, 128>(A, W, C, M, N, K, E, stream, bias);
    case 31: return launch_ring<128, 64>(A, W, C, M, N, K, E, stream, bias);
    case 32: return launch_ring<64, 64>(A, W, C, M, N, K, E, stream, bias);
    case 22: return launch_tile256<128>(A, W, C, M, N, K, E, stream, bias);
    default: return -4;
  }
}

// The same product with the RMSNorm before it folded in: X is the float32 residual stream
// [M, K], gain float32 [K]; W must be pre-tiled, M <= 64, no split over workgroups; epi is
// store-bf16, store-f32 or SwiGLU.
extern "C" int zf_norm_gemm_bf16_skinny(const float* X, const float* gain, float eps, const void* W,
                                        void* C, int M, int N, int K, int epi, int rg,
                                        hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  const int mt = (M + 15) / 16;
  if (M > 64 || K % 64 != 0 || N % (16 * rg) != 0 || epi == EPI_ACC_F32) return -3;
  SkinnyNorm nrm{};
  nrm.gain = gain;
  nrm.eps = eps;
#define ZF_NSK(MT, RG) \
  return launch_skinny<MT, RG, true, NORM_FOLD>(X, W, C, nullptr, M, N, K, epi, 1, stream, nrm)
  if (rg == 1) { if (mt == 1) ZF_NSK(1, 1); if (mt == 2) ZF_NSK(2, 1); if (mt == 3) ZF_NSK(3, 1); ZF_NSK(4, 1); }
  if (rg == 2) { if (mt == 1) ZF_NSK(1, 2); if (mt == 2) ZF_NSK(2, 2); if (mt == 3) ZF_NSK(3, 2); ZF_NSK(4, 2); }
  if (rg == 4) { if (mt == 1) ZF_NSK(1, 4); if (mt == 2) ZF_NSK(2, 4); if (mt == 3) ZF_NSK(3, 4); ZF_NSK(4, 4); }
#undef ZF_NSK
  return -4;
}

// The same product for rows that come already multiplied by the norm's gain, as bfloat16
// XG [M <= 16, K], with the sums of squares of the un-normed rows per 16 columns,
// sq [sq_groups][16] (token j of group g at sq[g * 16 + j]), as zf_gemm_bf16_skinny_emit
// leaves them: out = (XG W^T) / sqrt(sum_g sq[g][token] / K + eps).
extern "C" int zf_gemm_bf16_skinny_given(const void* XG, const float* sq, int sq_groups, float eps,
                                         const void* W, void* C, int M, int N, int K, int epi,
                                         int rg, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 16 || K % 64 != 0 || N % (16 * rg) != 0 || epi == EPI_ACC_F32 || sq_groups < 1)
    return -3;
  SkinnyNorm nrm{};
  nrm.eps = eps;
  nrm.sq_in = sq;
  nrm.sq_groups = sq_groups;
  if (rg == 1) return launch_skinny<1, 1, true, NORM_GIVEN>(XG, W, C, nullptr, M, N, K, epi, 1, stream, nrm);
  if (rg == 2) return launch_skinny<1, 2, true, NORM_GIVEN>(XG, W, C, nullptr, M, N, K, epi, 1, stream, nrm);
  if (rg == 4) return launch_skinny<1, 4, true, NORM_GIVEN>(XG, W, C, nullptr, M, N, K, epi, 1, stream, nrm);
  return -4;
}

// C += A W^T (C the float32 residual stream [M <= 16, N], W pre-tiled) and, for the RMSNorm
// that reads C next: xg_out [M, N] = bfloat16(C * gain_out), sq_out [N / 16][16] = sums of
// C^2 over each group of 16 columns (tokens beyond M: 0).
extern "C" int zf_gemm_bf16_skinny_emit(const void* A, const void* W, float* C,
                                        const float* gain_out, void* xg_out, float* sq_out, int M,
                                        int N, int K, int rg, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 16 || K % 64 != 0 || N % (16 * rg) != 0) return -3;
  SkinnyNorm nrm{};
  nrm.gain_out = gain_out;
  nrm.xg_out = (bf16_t*)xg_out;
  nrm.sq_out = sq_out;
  if (rg == 1) return launch_skinny<1, 1, true, NORM_NONE, true>(A, W, C, nullptr, M, N, K, EPI_ACC_F32, 1, stream, nrm);
  if (rg == 2) return launch_skinny<1, 2, true, NORM_NONE, true>(A, W, C, nullptr, M, N, K, EPI_ACC_F32, 1, stream, nrm);
  return -4;
}

// ---------------------------------------------------------------- measurement: MFMAs alone
// What the matrix cores sustain on given operands with nothing else to do: every wave keeps
// four token operands (32 rows x 16 k each) and two weight operands (32 outputs x 16 k) in
// registers and runs `iters` rounds of the eight 32x32x16 products between them into eight
// accumulators, so that operands change from one instruction to the next as they do in the
// products above.  On operands that toggle the multipliers the chip's power limit, not its
// clock, sets the rate; the rate this reaches is what the tiled products are measured
// against.  src: bfloat16 [6][64][8], operand f of lane l at src[f][l] (a lane holds row or
// output l % 32, k 8 (l / 32) .. + 8); operands 0-3 tokens, 4-5 weights.  The first wave of
// the first workgroup leaves its accumulators in out [8][32][32] (accumulator n = tokens
// n % 4 against weights n / 4: iters times their product).
__global__ __launch_bounds__(256) void mfma_loop_kernel(const u32x4_t* __restrict__ src,
                                                        float* __restrict__ out, int iters) {
  const int lane = threadIdx.x % 64;
  u32x4_t a[4], b[2];
#pragma unroll
  for (int f = 0; f < 4; ++f) a[f] = src[f * 64 + lane];
#pragma unroll
  for (int f = 0; f < 2; ++f) b[f] = src[(4 + f) * 64 + lane];
  f32x16_t acc[8];
#pragma unroll
  for (int n = 0; n < 8; ++n)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[n][r] = 0.f;
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int n = 0; n < 8; ++n)
      acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*(const bf16x8_t*)&a[n % 4],
                                                       *(const bf16x8_t*)&b[n / 4], acc[n], 0, 0, 0);
  }
  if (blockIdx.x == 0 && threadIdx.x < 64) {
#pragma unroll
    for (int n = 0; n < 8; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        out[(n * 32 + 8 * (r / 4) + 4 * (lane / 32) + r % 4) * 32 + lane % 32] = acc[n][r];
  } else {
    // (every other wave's sums must count for something, or the compiler drops its loop)
    float s = 0.f;
#pragma unroll
    for (int n = 0; n < 8; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) s += acc[n][r];
    if (s == 1234.5678f && iters < 0) out[0] = s;
  }
}

// workgroups of four waves; 2 * 32 * 32 * 16 * 8 flops a wave and round
extern "C" int zf_mfma_loop(const void* src, float* out, int workgroups, int iters,
                            hipStream_t stream) {
  if (workgroups < 1 || workgroups > 65536 || iters < 1 || iters > (1 << 22)) return 1;
  hipLaunchKernelGGL(mfma_loop_kernel, dim3(workgroups), dim3(256), 0, stream,
                     (const u32x4_t*)src, out, iters);
  ZF_CHECK_LAUNCH();
}
