// All layers of a decoder in one launch, for a decode step of very few tokens (pre-norm layers:
// RMSNorm, grouped-query attention with normed and rotated heads, RMSNorm, SwiGLU; bfloat16).
//
// In launches of their own a layer's six kernels each ramp up and drain while memory idles (26 us a layer
// of the 0.6B shape, whose 31 MB of weights take 4.5 at 7 TB/s; 81 of 55 at the 8B shape).  Here a layer
// takes 15 us and 69: the weights, and where these are few the five times that rows travel between all
// workgroups (1.9 us each, the words' way alone).  Decode steps of one token of Qwen3 shapes behind 120 tokens, four layers and
// the head, before and after: 0.6B 197 -> 164 us, 1.7B 285 -> 244, 4B 372 -> 350, 8B 560 -> 527; where
// row groups deal out unevenly, as at 14B, the phases' ends cost what the launches' did, and such steps keep a launch a
// product (ops/decode_layers.py, `pays`, has the lines and both sides' figures).  Two tokens 0.6B 196 -> 168, 8B 544 ->
// 521; three 200 -> 179, 547 -> 535; four tokens of the 0.6B and 1.7B shapes 202 -> 187 and 291 -> 273: what the
// workgroups hand each other grows with the tokens.
//
// One workgroup a CU stays for the whole step.  Its first DL_CW waves stream weights and multiply:
// each holds the next RING tiles (16 rows x 64 of K, 2 KB) of its own in registers and asks for one
// more with every one it takes, through matrices, layers and waits alike, so that memory is read
// while rows travel between workgroups.  The other four waves gather the rows a phase reads, add up
// its sums, run norms, residual, activation and attention, and hand the result on.
//
// Rows travel between workgroups as words of 8 bytes, 4 of data and 4 that say of which layer they
// are (`epoch`): a word that carries the epoch carries its data, so a reader waits for the words
// themselves and nothing else orders the workgroups.  They are written and read by buffer accesses of 8
// or 16 bytes past the XCDs' own caches (sc1).  What this rests on: an aligned 8-byte half of such an
// access arrives whole, and a reader's loads are issued anew at every look (an asm statement that may
// change memory stands ahead of them, so that the compiler neither joins nor hoists them).  A phase's
// words are overwritten a layer later at the earliest, and whoever is about to write them has read,
// directly or through others, what every workgroup made from the last ones; two sets of words in turn
// leave another layer between.
//
// Workgroups that are resident at once do the step: they arrive one after the other, and what there is
// to do is dealt among those that have come when all have or, where another stream or process holds
// CUs, `meet_ticks` later; whoever comes then leaves again.  So no workgroup waits for one that has no CU,
// whatever runs beside (a cooperative launch promises the same from a queue of its own: 15 us a step to
// go there and back, and half a microsecond more for every later kernel of the process).
// Launches side by side: a step holds every CU it got until its end, so two engines that decode at once run
// their steps one behind the other, where launches a product fill each other's gaps (us a step, two engines of one
// user each, drawing included: 0.6B 952 and 969, eight layers of the 8B shape 1165 and 1047; of three users 1302
// and 1064, 1304 and 1105), and beside another's whole prompts a step waits for CUs once and not at every product (0.6B
// 682 and 5019 us a step, while a prompt of 2048 tokens through four layers of the 8B shape takes 8.2 ms and 3.4).
// However few have come `meet_most` later, one included, do it: a launch that held CUs until it had more could
// wait for another that does the same.  Fewer than `need`, whose shares would not fit a phase's sums, take
// theirs a piece at a time (FEW, below), in the same order of sums.
// Every wait ends: a reader that has looked DL_SPINS times gives up for its workgroup, which leaves
// without handing on what it owes, so that the others leave in turn: what follows from words that did
// not come is neither handed on nor written to the pools.  The rows that go to the head are then NaN and
// `status` is 1.
//
// A product's sums run in the order of the kernel that has a launch of its own for it (gemm.hip's
// weight-streaming product, K dealt to eight waves in blocks of 64), whoever takes them.
#include <type_traits>

#include "zf_common.h"
#include "zf_decode.h"

#define DL_CW 8                  // waves that stream and multiply
#define DL_THREADS 768
#define DL_HD 128                // head size
#define DL_WAVE_KEYS 32          // keys a wave of the attention takes
#define DL_SPLIT 128             // keys a workgroup takes
#define DL_PART (DL_HD + 2)      // words of a split's partial result: O, max, sum
#define DL_SPINS (1 << 21)
#define DL_CLOSED (1u << 31)
#define DL_UNITS 16              // most units of 16 outputs a workgroup has in a phase, times tokens
#define DL_FF_UNITS 32           // and at gate/up, where a unit is two row groups
#define DL_RUNS (3 * DL_UNITS + 2 * DL_FF_UNITS)
#define DL_ATT 8                 // most splits of contexts a workgroup has
#define DL_COPIES 4
#define DL_TOKENS 4              // most of a step
// a run: the first tile of a row group, whether a phase begins and ends with it, which product's
#define DL_RUN_TILE 0x0fffffffu
#define DL_RUN_FIRST (1u << 28)
#define DL_RUN_LAST (1u << 29)

typedef unsigned long long dl_word;

struct DecodeLayer {
  const bf16_t* w[4];            // q/k/v, output, gate/up (rows in turn by 16), down: pre-tiled
  const float* q_gain;           // null: no norm of the heads
  const float* k_gain;
  const float* ff_gain;          // of the norm ahead of gate/up
  const float* next_gain;        // of the norm that reads the stream behind the layer
  bf16_t* k_pool;
  bf16_t* v_pool;
};

// Where a launch's workgroups meet (zero at first), in lines of their own.
struct DecodeMeet {
  alignas(128) unsigned arrived;         // and DL_CLOSED: whoever comes leaves again
  alignas(128) dl_word go;               // the step's number and how many do it
  alignas(128) unsigned decided;
  alignas(128) unsigned epoch;           // of the last launch's last layer
};

struct DecodeLayers {
  const DecodeLayer* layers;
  int tokens, n_layers, hidden, ff, nH, nKV, page_size, max_pages, max_splits;
  float eps_in, eps_ff, eps_head, scale_log2e;
  const float* cos_t;            // [table_rows, hd / 2], null: no rotation
  const float* sin_t;
  int table_rows;
  const int* positions;
  const int* slot_mapping;
  const int* block_table;
  const int* ctx_len;
  float* x;                      // [M, hidden] the stream, in place
  bf16_t* xg;                    // [M, hidden] bfloat16(x * gain) of the norm that reads it next, in place
  float* sq;                     // [hidden / 16][16] the sums of x^2 over 16 columns, in place
  dl_word* words;                // zero at first
  DecodeMeet* meet;
  int need;                      // workgroups whose shares of a phase fit its sums
  int meet_ticks;                // of 10 ns that the workgroups which have come wait for the others
  int meet_most;                 // and while they are fewer than `need`
  int spin_from;                 // looks of a wait that count as taken (0)
  int* status;
};

// What nothing writes while the kernel runs is read by scalar loads; the kernel's arguments where they
// lie, where they are used.
#define DL_CONST const __attribute__((address_space(4)))
#define DL_GLOBAL __attribute__((address_space(1)))
typedef DL_CONST DecodeLayers* DecodeArgs;
template <typename T>
__device__ __forceinline__ DL_CONST T* dl_const(const T* p) { return (DL_CONST T*)(uintptr_t)p; }
// from a pointer that itself came from memory
template <typename V>
__device__ __forceinline__ V dl_global(const void* p) { return *(const DL_GLOBAL V*)(uintptr_t)p; }
// 16 or 8 bytes a lane that are read once
template <typename V>
__device__ __forceinline__ V dl_stream(const void* p, size_t uniform, uint32_t lane_bytes) {
  return __builtin_nontemporal_load(
      (const DL_GLOBAL V*)((const DL_GLOBAL char*)(uintptr_t)p + uniform + lane_bytes));
}
__device__ __forceinline__ int dl_uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// LDS alone is handed over: loads of weights stay in flight
__device__ __forceinline__ void dl_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The words of a set, numbers of 16 bytes (two words).  Rows that every workgroup reads lie DL_COPIES
// times, for a part of the readers each (1024 numbers read by 256 workgroups: 2.4 us from one copy, 1.9
// from four, the words' way included).
struct DecodeWords {
  uint32_t qkv, attn, mid, mid_sq, next, next_sq, act, part, all;
};
__host__ __device__ inline DecodeWords dl_words(int M, int hidden, int ff, int nH, int nKV,
                                                int max_splits) {
  DecodeWords w;
  const uint32_t row = M * hidden / 4 * DL_COPIES, sq = M * hidden / 32 * DL_COPIES;
  w.qkv = 0;
  w.attn = w.qkv + M * (nH + 2 * nKV) * (DL_HD / 4);
  w.mid = w.attn + M * nH * (DL_HD / 4) * DL_COPIES;
  w.mid_sq = w.mid + row;
  w.next = w.mid_sq + sq;
  w.next_sq = w.next + row;
  w.act = w.next_sq + sq;
  w.part = w.act + M * ff / 4 * DL_COPIES;
  w.all = w.part + M * nH * max_splits * (DL_PART / 2);
  return w;
}
// bytes of LDS a row of the phases' inputs takes: 16 more than its numbers, so that the rows of
// several tokens begin in different banks
__host__ __device__ inline int dl_row(int hidden, int ff, int nH) {
  const int q = nH * DL_HD;
  int k = hidden > ff ? hidden : ff;
  if (q > k) k = q;
  return k * 2 + 16;
}

template <int M>
struct alignas(16) DecodeShared {
  float o[4][16][DL_HD];
  float m[4][16], l[4][16];
  bf16_t q[18][DL_HD + 8];       // query heads; row 16: the new key; row 17: the new value
  float part[DL_FF_UNITS * 2][DL_CW][16];         // (unit, token) by wave; at gate/up two for each
  float turn[M][2][DL_HD / 2];   // cosines and sines of the tokens' positions
  size_t blk[DL_ATT][4][2];      // where the 16-key groups of the workgroup's splits lie in the pools
  size_t put[DL_ATT];            // and the 16-row group of the token's own key and value
  int item[DL_ATT];              // kv head, split << 8, token << 16 and whether it holds the token's own
  uint32_t runs[DL_RUNS];        // the row groups of a layer's products that are this workgroup's
  float res[M > 1 ? 256 : 1];    // the stream's elements of this workgroup (one token: in registers)
  int n_runs, late, n_att;
  int dead;
  int wg, wgs;                   // this workgroup's number among those that do the step; none: it leaves
  unsigned base;
};

template <typename T>
__device__ __forceinline__ T dl_get(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void dl_put(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One thread of a workgroup: its number among those that do the step, and how many these are.  What a
// launch leaves in `meet` is changed by the last of its workgroups to have decided.
__device__ __forceinline__ void dl_meet(const DecodeLayers& p, int& wg, int& wgs, unsigned& base) {
  DecodeMeet* meet = p.meet;
  base = dl_get(&meet->epoch);
  const dl_word tag = (dl_word)(base + 1) << 32;
  const unsigned all = gridDim.x;
  const unsigned mine = __hip_atomic_fetch_add(&meet->arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  wg = mine & ~DL_CLOSED;
  wgs = 0;
  if (mine & DL_CLOSED) return;
  if (mine + 1 == all) {
    dl_put(&meet->go, tag | all);
    wgs = all;
    return;
  }
  const long long first = wall_clock64();
  for (;;) {
    const dl_word go = dl_get(&meet->go);
    if ((go ^ tag) >> 32 == 0) {
      wgs = (int)(uint32_t)go;
      return;
    }
    __builtin_amdgcn_s_sleep(1);
    const long long waited = wall_clock64() - first;
    if (waited < p.meet_ticks) continue;
    const unsigned come = dl_get(&meet->arrived);
    if ((come & DL_CLOSED) || (come < (unsigned)p.need && waited < p.meet_most)) continue;
    const unsigned n = __hip_atomic_fetch_or(&meet->arrived, DL_CLOSED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((n & DL_CLOSED) || n == all) continue;       // (another says, or the last to come does)
    dl_put(&meet->go, tag | n);
  }
}

template <int M, int BATCH>
__global__ __launch_bounds__(DL_THREADS) void decode_layers_kernel(DecodeLayers p) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  DecodeShared<M>& sh = *(DecodeShared<M>*)smem;
  float* s_sq = (float*)(smem + sizeof(DecodeShared<M>));                  // [M][hidden / 16]
  char* s_rows = (char*)(s_sq + (size_t)M * (p.hidden / 16));              // [M] rows
  const int row_bytes = dl_row(p.hidden, p.ff, p.nH);
  const int tid = threadIdx.x;
  const int wave = dl_uniform(tid / 64);

  if (tid == DL_CW * 64) dl_meet(p, sh.wg, sh.wgs, sh.base);
  dl_barrier();
  const int wg = dl_uniform(sh.wg), wgs = dl_uniform(sh.wgs);
  if (tid == DL_CW * 64) {        // the last to have decided makes the meeting ready for the next launch
    const unsigned before = __hip_atomic_fetch_add(&p.meet->decided, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (before + 1 == gridDim.x) {
      dl_put(&p.meet->arrived, 0u);
      dl_put(&p.meet->decided, 0u);
      dl_put(&p.meet->epoch, sh.base + p.n_layers);
    }
  }
  if (wg >= wgs) return;

  // the four products of a layer: units (a row group of 16, a pair of them at gate/up) are dealt
  // to the workgroups in turn; where they do not come out even, another product's go on from there
  const int qkv_units = (p.nH + 2 * p.nKV) * (DL_HD / 16), sum_units = p.hidden / 16, ff_units = p.ff / 16;
  const int extra = sum_units % wgs;
  const int qkv_first = (wg + wgs - extra) % wgs, ff_first = (qkv_first + wgs - qkv_units % wgs) % wgs;
  auto count = [&](int first, int units) { return first < units ? (units - first + wgs - 1) / wgs : 0; };
  const int n_qkv = count(qkv_first, qkv_units), n_sum = count(wg, sum_units), n_ff = count(ff_first, ff_units);

  // split `item` of a context as entry n, by threads t = 0 .. 7; false: the context does not reach it
  auto put_split = [&](int item, int n, int t) __attribute__((always_inline)) {
    const int kvh = item % p.nKV, s = (item / p.nKV) % M, sp = item / (p.nKV * M), ps = p.page_size;
    const int ctx = p.ctx_len[s];
    if (sp * DL_SPLIT >= ctx) return false;
    if (t < 8) {
      const int kb = sp * DL_SPLIT + (t / 2) * DL_WAVE_KEYS, end = min(ctx, kb + DL_WAVE_KEYS);
      // (a group without a key may have no page: it reads the group of one that exists and is masked)
      const int key = kb + 16 * (t % 2) < end ? kb + 16 * (t % 2) : kb;
      sh.blk[n][t / 2][t % 2] = kb >= end ? 0
          : (((size_t)p.block_table[(size_t)s * p.max_pages + key / ps] * p.nKV + kvh) * ps + key % ps) *
                DL_HD;
    }
    if (t == 0) {
      const int slot = p.slot_mapping[s], own = (ctx - 1) / DL_SPLIT == sp;
      sh.item[n] = kvh | sp << 8 | s << 16 | own << 24;
      // the row within the sixteen in the low bits
      sh.put[n] = ((((size_t)(slot / ps) * p.nKV + kvh) * ps + (slot % ps) / 16 * 16) * DL_HD) |
                  (size_t)(slot % 16);
    }
    return true;
  };
  const int n_splits = p.max_splits * M * p.nKV;
  const bool few = wgs < p.need;
  if (!few && tid < 64) {         // the splits of contexts that are this workgroup's
    int n = 0;
    for (int item = wg; item < n_splits; item += wgs)
      if (put_split(item, n, tid)) ++n;
    if (tid == 0) sh.n_att = n;
  }
  if (tid == 64) sh.dead = 0;
  if (!few && tid == 64) {
    // in the order of the layer; `late` is the first run behind the attention (-1: there is none)
    int n = 0, late = -1;
    for (int m = 0; m < 4; ++m) {
      const int before = n, per = (m == 1 ? p.nH * DL_HD : m == 3 ? p.ff : p.hidden) / 64;
      if (m > 0 && late < 0) late = n;
      const int units = m == 0 ? qkv_units : m == 2 ? ff_units : sum_units;
      for (int u = m == 0 ? qkv_first : m == 2 ? ff_first : wg; u < units; u += wgs)
        for (int r = 0; r < (m == 2 ? 2 : 1); ++r) {
          const uint32_t rg = m == 2 ? 2 * u + r : u;
          sh.runs[n] = ((uint32_t)m << 30) | (n == before ? DL_RUN_FIRST : 0u) | rg * per;
          ++n;
        }
      if (n > before) sh.runs[n - 1] |= DL_RUN_LAST;
      else if (late == n) late = -1;
    }
    sh.n_runs = n;
    sh.late = late;
  }
  if (p.cos_t != nullptr && tid >= 128)
    for (int i = tid - 128; i < M * DL_HD; i += DL_THREADS - 128) {
      const int s = i / DL_HD, d = i % DL_HD, row = min(max(p.positions[s], 0), p.table_rows - 1);
      sh.turn[s][d / (DL_HD / 2)][d % (DL_HD / 2)] =
          (d < DL_HD / 2 ? p.cos_t : p.sin_t)[(size_t)row * (DL_HD / 2) + d % (DL_HD / 2)];
    }
  dl_barrier();
  const int n_att = few ? 0 : dl_uniform(sh.n_att);
  volatile __attribute__((address_space(3))) int* dead =
      (volatile __attribute__((address_space(3))) int*)&sh.dead;

  if (few && wave < DL_CW) return;
  if (wave < DL_CW) {
    // ------------------------------------------------------------ streaming and multiplying
    const int lane = tid % 64, g = lane / 16, j = min(lane % 16, M - 1);
    // tiles of a row group that are this wave's: blocks wave, wave + 8, ..
    auto tiles_of = [&](int k) __attribute__((always_inline)) { return (k / 64 - wave + DL_CW - 1) / DL_CW; };
    const int h_tiles = tiles_of(p.hidden), q_tiles = tiles_of(p.nH * DL_HD), ff_tiles = tiles_of(p.ff);
    auto tiles = [&](uint32_t m) __attribute__((always_inline)) { return m == 1 ? q_tiles : m == 3 ? ff_tiles : h_tiles; };
    auto run_at = [&](int i) __attribute__((always_inline)) { return (uint32_t)dl_uniform(sh.runs[i]); };
    DL_CONST DecodeLayer* layers = dl_const(p.layers);
    const int n_layers = p.n_layers;
    const int n_runs = dl_uniform(sh.n_runs), late = dl_uniform(sh.late);
    if (n_runs == 0) {              // (attention alone)
      for (int i = 0; i < 3 * n_att * n_layers; ++i) dl_barrier();
      return;
    }
    // Where the next tiles come from: run lr of layer li, and the run behind it.  Past a phase's last run
    // the rest of a batch, and past the last layer all, is loads of nothing: descriptors of no bytes.
    int li = 0, lr = -1, left = 0, next_left = 0;
    bool ends = false, next_ends = false;       // the run is its phase's last one
    const char *at = nullptr, *next_at = nullptr;
    // the matrices of layer li and, asked for a layer ahead, of the one behind it
    const bf16_t *w_h = layers[0].w[0], *w_o = layers[0].w[1], *w_gu = layers[0].w[2], *w_d = layers[0].w[3];
    const bf16_t *n_h, *n_o, *n_gu, *n_d;
    bool ahead = false;
    auto look_ahead = [&]() __attribute__((always_inline)) {
      if (ahead) return;
      ahead = true;
      DL_CONST DecodeLayer& n = layers[min(li + 1, n_layers - 1)];
      n_h = n.w[0];
      n_o = n.w[1];
      n_gu = n.w[2];
      n_d = n.w[3];
    };
    look_ahead();
    auto look = [&]() __attribute__((always_inline)) {
      if (++lr == n_runs) {
        lr = 0;
        look_ahead();
        ++li;
        w_h = n_h;
        w_o = n_o;
        w_gu = n_gu;
        w_d = n_d;
        ahead = false;
      }
      if (li >= n_layers) {
        next_left = 0;
        next_ends = true;
        return;
      }
      const uint32_t run = run_at(lr);
      next_left = tiles(run >> 30);
      next_ends = run & DL_RUN_LAST;
      const uint32_t m = run >> 30;
      // (read here and then chosen among: a choice of variables puts them into memory)
      const bf16_t *w0_ = w_h, *w1_ = w_o, *w2_ = w_gu, *w3_ = w_d;
      const bf16_t* w = m & 2 ? (m & 1 ? w3_ : w2_) : (m & 1 ? w1_ : w0_);
      next_at = (const char*)w + ((size_t)(run & DL_RUN_TILE) + wave) * 2048;
    };
    auto next_run = [&]() __attribute__((always_inline)) {
      at = next_at;
      left = next_left;
      ends = next_ends;
      look();
    };
    look();
    const uint32_t lane_at = lane * 16;
    constexpr int NT = 2;           // read once
    // two batches of pairs of tiles (three pairs a batch, 24 KB a wave under way: one user of the 0.6B and
    // 8B shapes 17.3 and 138.0 ms; two pairs 17.8 and 138.3, four 17.7 and 139.0)
    u32x4_t w0[2][BATCH][2], w1[2][BATCH][2];
    auto ask = [&](int b) __attribute__((always_inline)) {
      if (left <= 0) next_run();
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        if (i > 0 && left <= 0 && !ends) next_run();
        const __amdgpu_buffer_rsrc_t one =
            __builtin_amdgcn_make_buffer_rsrc((void*)at, 0, left > 0 ? 2048 : 0, 0x00020000);
        const __amdgpu_buffer_rsrc_t two =
            __builtin_amdgcn_make_buffer_rsrc((void*)(at + 2048 * DL_CW), 0, left > 1 ? 2048 : 0, 0x00020000);
        w0[b][i][0] = __builtin_amdgcn_raw_buffer_load_b128(one, lane_at, 0, NT);
        w1[b][i][0] = __builtin_amdgcn_raw_buffer_load_b128(one, lane_at + 1024, 0, NT);
        w0[b][i][1] = __builtin_amdgcn_raw_buffer_load_b128(two, lane_at, 0, NT);
        w1[b][i][1] = __builtin_amdgcn_raw_buffer_load_b128(two, lane_at + 1024, 0, NT);
        at += 2 * 2048 * DL_CW;
        left -= 2;
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // (in this order: a wait in the loop below counts the loads that are younger on every way there)
    ask(0);
    ask(1);

    // What is multiplied now.  A pair's rows are read from LDS ahead of it.  A batch is asked for anew
    // when all of it is multiplied, and where a phase ends with it, when its sums have been handed on:
    // loads that are under way hold up the words that others wait for.
    int cl = 0, cr = -1, todo = 0, ci = 0, seen = 0;      // (barriers of the attention's)
    bool last = false, done = false, alive = true;
    const char* arow = s_rows + (size_t)j * row_bytes + g * 32 + wave * 128;
    const char* a = arow;
    f32x4_t acc0 = f32x4_t{0.f, 0.f, 0.f, 0.f}, acc1 = acc0;
    u32x4_t a00, a01, a10, a11;
    auto rows = [&]() __attribute__((always_inline)) {
      a00 = *(const u32x4_t*)a;
      a01 = *(const u32x4_t*)(a + 16);
      a10 = *(const u32x4_t*)(a + 128 * DL_CW);     // (one too many may follow a row's last: in LDS too)
      a11 = *(const u32x4_t*)(a + 128 * DL_CW + 16);
      a += 2 * 128 * DL_CW;
    };
    auto run = [&]() __attribute__((always_inline)) {
      const uint32_t r = run_at(cr);
      todo = tiles(r >> 30);
      last = r & DL_RUN_LAST;
      a = arow;
    };
    auto begin = [&]() __attribute__((always_inline)) {   // the next phase, its rows in LDS
      done = false;
      if (++cr == n_runs) {
        cr = 0;
        if (late < 0)
          for (int i = 0; i < 3 * n_att; ++i) dl_barrier();
        if (++cl == n_layers) {
          alive = false;
          done = true;
          return;
        }
      }
      ci = 0;
      if (cr == late)
        for (int i = seen; i < 3 * n_att; ++i) dl_barrier();
      seen = 0;
      run();
      dl_barrier();
      rows();
    };
    begin();
    // (one way out, at the end of a round: where others met the way back the waits would be for loads
    // that were asked for just now)
    while (alive) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
          if (!done) {
            acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(bf16x8_t*)&w0[b][i][0], *(bf16x8_t*)&a00, acc0, 0,
                                                           0, 0);
            if (todo > 1)
              acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(bf16x8_t*)&w0[b][i][1], *(bf16x8_t*)&a10, acc1,
                                                             0, 0, 0);
            acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(bf16x8_t*)&w1[b][i][0], *(bf16x8_t*)&a01, acc0, 0,
                                                           0, 0);
            if (todo > 1)
              acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(bf16x8_t*)&w1[b][i][1], *(bf16x8_t*)&a11, acc1,
                                                             0, 0, 0);
            todo -= 2;
            if (todo <= 0) {
              if (lane % 16 < M) *(f32x4_t*)&sh.part[ci + lane % 16][wave][4 * (lane / 16)] = acc0 + acc1;
              acc0 = acc1 = f32x4_t{0.f, 0.f, 0.f, 0.f};
              ci += M;
              done = last;
              if (!last) {
                ++cr;
                run();
              }
            }
            if (!done) rows();
          }
          __builtin_amdgcn_sched_barrier(0);
        }
        bool leave = false;
        if (done && alive) {
          leave = dl_uniform(*dead) != 0;
          dl_barrier();               // the sums are there
          dl_barrier();               // and handed on
          if (n_att > 0 && cr + 1 == late) {
            dl_barrier();             // and the attention's rows have come
            seen = 1;
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        ask(b);
        __builtin_amdgcn_sched_barrier(0);
        if (done && alive) {
          look_ahead();
          if (leave) alive = false;
          else begin();
        }
      }
    }
    return;
  }

  // -------------------------------------------------------------- rows, sums and attention
  const int cwave = wave - DL_CW;
  // What is formed from a thread's number or the arguments is formed where it is used: hoisted out of
  // the layers' loop it takes the registers that the attention's keys and values need.
  auto thread = [&]() __attribute__((always_inline)) {
    uint32_t t = tid - DL_CW * 64;
    asm volatile("" : "+v"(t));
    return t;
  };
  auto args = [&]() __attribute__((always_inline)) {
    DecodeArgs a = (DecodeArgs)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    return a;
  };
  const DecodeWords at = dl_words(M, p.hidden, p.ff, p.nH, p.nKV, p.max_splits);
  const unsigned base = dl_uniform(sh.base);
  const int groups = p.hidden / 16, n_layers = p.n_layers, nH = p.nH, G = p.nH / p.nKV;
  const uint32_t copy = wg % DL_COPIES;
  // words are read and written past the caches that belong to one XCD (sc1)
  const __amdgpu_buffer_rsrc_t words =
      __builtin_amdgcn_make_buffer_rsrc(p.words, 0, (int)(2 * 16 * at.all), 0x00020000);
  constexpr int SC1 = 16;
  auto load2 = [&](uint32_t lane_bytes, uint32_t from) __attribute__((always_inline)) {
    return __builtin_amdgcn_raw_buffer_load_b128(words, lane_bytes, from, SC1);
  };
  auto store2 = [&](uint32_t lane_bytes, uint32_t to, uint32_t d0, uint32_t d1, unsigned epoch) __attribute__((always_inline)) {
    __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{d0, epoch, d1, epoch}, words, lane_bytes, to, SC1);
  };
  // look() loads and says (a lane) whether words are missing; until none of the wave's are (true), or the
  // workgroup has given up
  const int spin_from = p.spin_from;
  auto wait_for = [&](auto look) __attribute__((always_inline)) {
    for (int spin = spin_from;; ++spin) {
      asm volatile("" ::: "memory");
      const bool missing = look();
      if (__builtin_amdgcn_ballot_w64(missing) == 0) return true;
      if (spin >= DL_SPINS) *dead = 1;
      if ((spin & 15) == 15 && dl_uniform(*dead) != 0) return false;
    }
  };
  // `n` pairs of words behind one another from pair `from`, a pair a thread, N at a time; to(number, data)
  auto gather_some = [&](auto N, uint32_t from, uint32_t n, unsigned epoch, auto to) __attribute__((always_inline)) {
    const uint32_t t = thread();
    u32x4_t v[decltype(N)::value];
    wait_for([&]() __attribute__((always_inline)) {
      uint32_t bad = 0;
#pragma unroll
      for (int i = 0; i < decltype(N)::value; ++i) v[i] = load2(t * 16, (from + i * 256) * 16);
#pragma unroll
      for (int i = 0; i < decltype(N)::value; ++i)
        bad |= t + i * 256 < n ? (v[i][1] ^ epoch) | (v[i][3] ^ epoch) : 0u;
      return bad != 0;
    });
#pragma unroll
    for (int i = 0; i < decltype(N)::value; ++i)
      if (t + i * 256 < n) to(t + i * 256, u32x2_t{v[i][0], v[i][2]});
  };
  auto gather = [&](uint32_t from, uint32_t n, unsigned epoch, auto to) __attribute__((always_inline)) {
    uint32_t i = 0;
    auto some = [&](auto N) __attribute__((always_inline)) {
      gather_some(N, from + i, n - i, epoch, [&](uint32_t w, u32x2_t d) __attribute__((always_inline)) { to(i + w, d); });
      i += decltype(N)::value * 256;
    };
    while (i + 1024 < n) some(std::integral_constant<int, 8>{});
    if (i + 512 < n) some(std::integral_constant<int, 4>{});
    else if (i + 256 < n) some(std::integral_constant<int, 2>{});
    else if (i < n) some(std::integral_constant<int, 1>{});
  };
  // rows of n numbers a token
  auto gather_rows = [&](uint32_t from, int n, unsigned epoch) __attribute__((always_inline)) {
#pragma unroll
    for (int tok = 0; tok < M; ++tok)
      gather(from + tok * (n / 4), n / 4, epoch,
             [&](uint32_t w, u32x2_t d) __attribute__((always_inline)) { *(u32x2_t*)(s_rows + (size_t)tok * row_bytes + w * 8) = d; });
  };
  // rows that a norm reads next: the sums of squares of each 16 columns as well
  auto gather_normed = [&](uint32_t from, uint32_t from_sq, unsigned epoch) __attribute__((always_inline)) {
    gather_rows(from + copy * (M * p.hidden / 4), p.hidden, epoch);
    gather(from_sq + copy * (M * groups / 2), M * groups / 2, epoch,
           [&](uint32_t w, u32x2_t d) __attribute__((always_inline)) { *(u32x2_t*)(s_sq + 2 * w) = d; });
  };
  // 1 / sqrt(mean(x^2) + eps) of every token, the same in every lane
  auto inv_rms = [&](float eps, float (&inv)[M]) {
    const uint32_t lane = thread() % 64;
#pragma unroll
    for (int tok = 0; tok < M; ++tok) {
      float v = 0.f;
      for (int i = lane; i < groups; i += 64) v += s_sq[tok * groups + i];
      inv[tok] = 1.0f / sqrtf(wave_sum(v) / (float)p.hidden + eps);
      asm volatile("" : "+v"(inv[tok]));      // (while the other waves multiply, not behind them)
    }
  };
  // Epilogues: sixteen threads a (unit, token), one a row of the unit.  The sum over the waves:
  auto sum_waves = [&](uint32_t pair, uint32_t r) __attribute__((always_inline)) {
    float v[DL_CW];
#pragma unroll
    for (int w = 0; w < DL_CW; ++w) v[w] = sh.part[pair][w][r];
    float s = v[0];
#pragma unroll
    for (int w = 1; w < DL_CW; ++w) s += v[w];
    return s;
  };
  // four lanes' values as two words each of the four holds
  auto quad_words = [&](float v, uint32_t r, uint32_t& d0, uint32_t& d1) __attribute__((always_inline)) {
    const float o = lane_xor<1>(v);
    const uint32_t mine = r % 2 ? pack_bf16x2(o, v) : pack_bf16x2(v, o);
    const uint32_t other = __float_as_uint(lane_xor<2>(__uint_as_float(mine)));
    d0 = r & 2 ? other : mine;
    d1 = r & 2 ? mine : other;
  };
  // this thread's (unit, token) and its row, formed where they are used (as are the addresses that follow
  // from them: kept through the layers they were spilled, a load of 0.5 us in every epilogue)
  struct Place {
    uint32_t r, pair, tok, unit;
  };
  auto place = [&]() __attribute__((always_inline)) {
    const uint32_t t = thread();
    return Place{t % 16, t / 16, t / 16 % M, t / 16 / M};
  };
  // the stream's element it keeps
  auto column = [&](const Place& e) __attribute__((always_inline)) { return (wg + e.unit * wgs) * 16 + e.r; };
  // FEW: the workgroups are fewer than `need`.  These four waves do the products too, so many units of a
  // phase at a time, and find their splits of contexts as they go; the other eight have left.
  auto all_layers = [&](auto few_) __attribute__((always_inline)) {
    constexpr bool FEW = decltype(few_)::value;
    constexpr int PIECE = DL_UNITS / M, FF_PIECE = DL_FF_UNITS / M;
    const bool keeps = place().unit < (uint32_t)n_sum;
    float res = 0.f;
    if (!FEW && keeps) {
      const Place e = place();
      res = p.x[(size_t)e.tok * p.hidden + column(e)];
      if constexpr (M > 1) sh.res[thread()] = res;
    }
    // The sum joins the stream's element, and what the next norm needs of the result goes to the words
    // at `to` and `to_sq`, or (last) back to memory.  Of a piece the units from k0 on, whose elements lie
    // in memory and whose gains are read here.
    auto residual = [&](float gain, const float* gains, int k0, uint32_t to, uint32_t to_sq, unsigned epoch, bool last) __attribute__((always_inline)) {
      Place e = place();
      if (FEW ? e.unit >= (uint32_t)min(PIECE, n_sum - k0) : !keeps) return;
      if constexpr (FEW) e.unit += k0;
      const uint32_t e_r = e.r, e_tok = e.tok, keeps_at = column(e);
      float* mine = FEW ? args()->x + (size_t)e_tok * args()->hidden + keeps_at : nullptr;
      if constexpr (FEW) gain = dl_global<float>(gains + keeps_at);
      float now = FEW ? *mine : M > 1 ? sh.res[thread()] : res;
      now += sum_waves(e.pair, e_r);
      if constexpr (FEW) *mine = now;
      else if constexpr (M > 1) sh.res[thread()] = now;
      else res = now;
      const float sq = lanes_sum<16>(now * now);
      uint32_t d0, d1;
      quad_words(now * gain, e_r, d0, d1);
      const uint32_t c = e_r % DL_COPIES;
      const uint32_t row = (c * M + e_tok) * p.hidden + (keeps_at & ~3u);       // numbers, 4 a pair of words
      if (!last) {
        store2(row * 4, to * 16, d0, d1, epoch);
        if (e_r < DL_COPIES)
          __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{__float_as_uint(sq), epoch}, words,
                                                ((e_r * M + e_tok) * groups + keeps_at / 16) * 8, to_sq * 16, SC1);
        return;
      }
      const DecodeArgs pp = args();
      const size_t n = (size_t)e_tok * p.hidden + keeps_at;
      pp->x[n] = now;
      if (c == 0) *(u32x2_t*)(pp->xg + n) = u32x2_t{d0, d1};
      if (e_r == 0) pp->sq[(size_t)(keeps_at / 16) * 16 + e_tok] = sq;
    };

    bool split = false;             // a context of more than one split: the partials are merged
    for (int s = 0; s < M; ++s) split = split || dl_const(p.ctx_len)[s] > DL_SPLIT;

    // A split's part of the norm's gains and of the keys and values that the cache holds: asked for while
    // the other waves run the down product of the layer before, behind whose loads they may wait.
    f32x4_t g0 = f32x4_t{1.f, 1.f, 1.f, 1.f}, g1 = g0;
    u32x4_t kf[2][DL_HD / 32];
    u32x2_t vf[2][DL_HD / 16];
    auto ask_keys = [&](int layer, int att) __attribute__((always_inline)) {
      if ((!FEW && att >= n_att) || layer >= n_layers) return;
      DL_CONST DecodeLayer& L = dl_const(args()->layers)[layer];
      const uint32_t t = thread(), lane = t % 64, l16 = t % 16;
      const int item = dl_uniform(sh.item[att]);
      const int kb = (item >> 8 & 255) * DL_SPLIT + cwave * DL_WAVE_KEYS;
      if (L.q_gain != nullptr) {
        const float* gain = (int)t / 16 < G ? L.q_gain : L.k_gain;
        g0 = dl_global<f32x4_t>(gain + 4 * l16);
        g1 = dl_global<f32x4_t>(gain + DL_HD / 2 + 4 * l16);
      }
      if (kb >= dl_const(p.ctx_len)[item >> 16 & 255]) return;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x2_t b = *(const u32x2_t*)&sh.blk[att][cwave][h];
        const size_t blk = ((size_t)(uint32_t)dl_uniform(b[0]) | (size_t)(uint32_t)dl_uniform(b[1]) << 32) * 2;
#pragma unroll
        for (int stp = 0; stp < DL_HD / 32; ++stp)
          kf[h][stp] = dl_stream<u32x4_t>(L.k_pool, blk + stp * 1024, lane * 16);
#pragma unroll
        for (int dt = 0; dt < DL_HD / 16; ++dt)
          vf[h][dt] = dl_stream<u32x2_t>(L.v_pool, blk + dt * 512, lane * 8);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (!FEW) ask_keys(0, 0);
    // The units [k0, k0 + n) of product m, which begin at `first`, into the sums: what the other eight waves do,
    // two of them a wave.
    auto multiply = [&](int layer, int m, int first, int k0, int n) __attribute__((always_inline)) {
      const DecodeArgs pp = args();
      DL_CONST DecodeLayer& L = dl_const(pp->layers)[layer];
      const int lane = thread() % 64, per = (m == 1 ? nH * DL_HD : m == 3 ? pp->ff : pp->hidden) / 64;
      for (int i = 0; i < (m == 2 ? 2 * n : n); ++i) {
        const size_t rg = m == 2 ? 2 * (first + (k0 + i / 2) * wgs) + i % 2 : first + (k0 + i) * wgs;
        for (int w = cwave; w < DL_CW; w += 4) {
          const int tiles = (per - w + DL_CW - 1) / DL_CW;
          const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc(
              (void*)((const char*)L.w[m] + (rg * per + w) * 2048), 0, max(per - w, 0) * 2048, 0x00020000);
          const char* a = s_rows + (size_t)min(lane % 16, M - 1) * row_bytes + (lane / 16) * 32 + w * 128;
          f32x4_t acc[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
          constexpr int AHEAD = 8;
          for (int t = 0; t < tiles; t += AHEAD) {
            u32x4_t w0[AHEAD], w1[AHEAD];
#pragma unroll
            for (int b = 0; b < AHEAD; ++b) {
              w0[b] = __builtin_amdgcn_raw_buffer_load_b128(from, lane * 16, (t + b) * DL_CW * 2048, 2);
              w1[b] = __builtin_amdgcn_raw_buffer_load_b128(from, lane * 16 + 1024, (t + b) * DL_CW * 2048, 2);
            }
#pragma unroll
            for (int b = 0; b < AHEAD; ++b)
              if (t + b < tiles) {
                const u32x4_t a0 = *(const u32x4_t*)(a + (t + b) * DL_CW * 128);
                const u32x4_t a1 = *(const u32x4_t*)(a + (t + b) * DL_CW * 128 + 16);
                acc[b % 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8_t*)&w0[b], *(const bf16x8_t*)&a0,
                                                                     acc[b % 2], 0, 0, 0);
                acc[b % 2] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8_t*)&w1[b], *(const bf16x8_t*)&a1,
                                                                     acc[b % 2], 0, 0, 0);
              }
          }
          if (lane % 16 < M) *(f32x4_t*)&sh.part[i * M + lane % 16][w][4 * (lane / 16)] = acc[0] + acc[1];
        }
      }
    };

    // false: given up
    auto run_layer = [&](int layer) __attribute__((always_inline)) {
      DL_CONST DecodeLayer& L = dl_const(args()->layers)[layer];
      const unsigned epoch = base + layer + 1;
      const uint32_t set = (epoch & 1) * at.all;
      float ff_gain = 0.f, next_gain = 0.f;
      if (!FEW && keeps) {
        const uint32_t at = column(place());
        ff_gain = dl_global<float>(L.ff_gain + at);
        next_gain = dl_global<float>(L.next_gain + at);
      }
      // ---- q, k and v
      if (n_qkv > 0) {
        const uint32_t t = thread();
        if (layer == 0) {
          const DecodeArgs pp = args();
          const uint32_t per = p.hidden / 8;
          for (uint32_t i = t; i < M * per; i += 256)
            *(u32x4_t*)(s_rows + (size_t)(i / per) * row_bytes + (i % per) * 16) = *((const u32x4_t*)pp->xg + i);
          for (uint32_t i = t; i < M * (uint32_t)groups; i += 256)
            s_sq[i] = pp->sq[(size_t)(i % groups) * 16 + i / groups];
        } else {
          // (the rows the layer before left, under its own epoch)
          const uint32_t before = ((epoch - 1) & 1) * at.all;
          gather_normed(before + at.next, before + at.next_sq, epoch - 1);
        }
        dl_barrier();
        float inv[M];
        inv_rms(p.eps_in, inv);
        const bool leave = dl_uniform(*dead) != 0;
        for (int k0 = 0; k0 == 0 || (FEW && k0 < n_qkv); k0 += PIECE) {
          const int n = FEW ? min(PIECE, n_qkv - k0) : n_qkv;
          if (FEW && !leave) multiply(layer, 0, qkv_first, k0, n);
          dl_barrier();
          if (leave) { dl_barrier(); return false; }
          const Place e = place();
          if (e.unit < (uint32_t)n) {
            float f = inv[0];
#pragma unroll
            for (int tok = 1; tok < M; ++tok) f = e.tok == tok ? inv[tok] : f;
            uint32_t d0, d1;
            quad_words(sum_waves(e.pair, e.r) * f, e.r, d0, d1);
            if (e.r % 4 == 0)
              store2((e.tok * qkv_units + qkv_first + (k0 + e.unit) * wgs) * 64 + e.r * 4, (set + at.qkv) * 16, d0,
                     d1, epoch);
          }
          dl_barrier();
        }
      }
      // ---- attention, a split of a context at a time
      for (int turn = 0, split_at = wg; FEW ? split_at < n_splits : turn < n_att; ++turn, split_at += wgs) {
        const uint32_t t = thread();
        const int att = FEW ? 0 : turn;
        if constexpr (FEW) {
          if (!put_split(split_at, 0, t)) continue;
          dl_barrier();
          ask_keys(layer, 0);
        }
        const DecodeArgs pp = args();
        const int item = dl_uniform(sh.item[att]);
        const int kvh = item & 255, sp = item >> 8 & 255, s = item >> 16 & 255;
        const bool own = item >> 24;
        const int ctx = dl_const(pp->ctx_len)[s], pos = ctx - 1;
        const int lane = t % 64, j = lane % 16, qd = lane / 16;
        const int kb = sp * DL_SPLIT + cwave * DL_WAVE_KEYS, k_end = min(ctx, kb + DL_WAVE_KEYS);
        const bool has_keys = kb < k_end;
        const int hi = t / 16, l16 = t % 16, n_items = own ? G + 1 : G;
        // the head's words: elements 4 l16 .. + 3 and 64 further on; the new value: 8 elements a thread
        const uint32_t row = (set + at.qkv + s * (qkv_units * 4)) * 16;
        const uint32_t head_at = (hi < G ? kvh * G + hi : nH + kvh) * (DL_HD / 4 * 16) + l16 * 16;
        u32x4_t r0, r1, v0, v1;
        bool came = wait_for([&]() __attribute__((always_inline)) {
          r0 = load2(head_at, row);
          r1 = load2(head_at, row + DL_HD / 8 * 16);
          const uint32_t bad = (r0[1] ^ epoch) | (r0[3] ^ epoch) | (r1[1] ^ epoch) | (r1[3] ^ epoch);
          return hi < n_items && bad != 0;
        });
        if (own && cwave == 0) {
          const uint32_t value_at = row + (nH + p.nKV + kvh) * (DL_HD / 4 * 16);
          came &= wait_for([&]() __attribute__((always_inline)) {
            v0 = load2(l16 * 32, value_at);
            v1 = load2(l16 * 32, value_at + 16);
            return ((v0[1] ^ epoch) | (v0[3] ^ epoch) | (v1[1] ^ epoch) | (v1[3] ^ epoch)) != 0;
          });
        }
        const size_t put = sh.put[att];
        const int r = put % 16;
        {
          float x0[4], x1[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            x0[e] = bf16_to_float((bf16_t)(r0[2 * (e / 2)] >> (16 * (e % 2))));
            x1[e] = bf16_to_float((bf16_t)(r1[2 * (e / 2)] >> (16 * (e % 2))));
          }
          HeadCoef cf;
          cf.has_gain = L.q_gain != nullptr;
          cf.has_rotation = p.cos_t != nullptr;
          const f32x4_t c = *(const f32x4_t*)&sh.turn[s][0][4 * l16], sn = *(const f32x4_t*)&sh.turn[s][1][4 * l16];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            cf.g0[e] = g0[e];
            cf.g1[e] = g1[e];
            cf.c[e] = c[e];
            cf.sn[e] = sn[e];
          }
          head_norm_rotate<16>(x0, x1, DL_HD, true, pp->eps_head, cf);
          if (hi < n_items) {
            const u32x2_t y0 = u32x2_t{pack_bf16x2(x0[0], x0[1]), pack_bf16x2(x0[2], x0[3])};
            const u32x2_t y1 = u32x2_t{pack_bf16x2(x1[0], x1[1]), pack_bf16x2(x1[2], x1[3])};
            bf16_t* dst = sh.q[hi < G ? hi : 16];
            *(u32x2_t*)(dst + 4 * l16) = y0;
            *(u32x2_t*)(dst + DL_HD / 2 + 4 * l16) = y1;
            if (hi == G && came) {  // element d of row r at [d / 32][16 ((d % 32) / 8) + r][d % 8]
              auto* grp = (DL_GLOBAL bf16_t*)(uintptr_t)L.k_pool + (put & ~(size_t)15);
              const int d0 = 4 * l16, at0 = (d0 / 32) * 512 + (((d0 % 32) / 8) * 16 + r) * 8 + d0 % 8;
              *(DL_GLOBAL u32x2_t*)(grp + at0) = y0;
              *(DL_GLOBAL u32x2_t*)(grp + at0 + (DL_HD / 64) * 512) = y1;
            }
          }
          if (own && came && t < DL_HD / 8) {   // [d / 16][16 (r / 4) + d % 16][r % 4]
            *(u32x4_t*)(sh.q[17] + 8 * l16) = u32x4_t{v0[0], v0[2], v1[0], v1[2]};
            auto* grp = (DL_GLOBAL bf16_t*)(uintptr_t)L.v_pool + (put & ~(size_t)15) + (r / 4) * 64 + r % 4;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const int d = 8 * l16 + i;
              grp[(d / 16) * 256 + (d % 16) * 4] =
                  (bf16_t)((i < 4 ? v0 : v1)[(i / 2) % 2 * 2] >> (16 * (i % 2)));
            }
          }
        }
        dl_barrier();
        const bool lost = dl_uniform(*dead) != 0;       // (nothing of this split is handed on)
        float m = -INFINITY, l = 0.f;
        f32x4_t o[DL_HD / 16];
#pragma unroll
        for (int dt = 0; dt < DL_HD / 16; ++dt) o[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (has_keys) {
          bf16x8_t qf[DL_HD / 32];
#pragma unroll
          for (int st = 0; st < DL_HD / 32; ++st) {
            u32x4_t v = *(const u32x4_t*)(sh.q[min(j, G - 1)] + st * 32 + 8 * qd);
            qf[st] = *(bf16x8_t*)&v;
          }
          // the token's own key and value, which the cache did not hold when it was read, where its lanes
          // hold a key's elements 32 stp + 8 qd .. + 7 (lane j: key j of the group) and four keys' values
          // (lane j: element 16 dt + j of keys 4 qd .. + 3)
          if (pos >= kb && pos < kb + DL_WAVE_KEYS) {
            const int jn = (pos - kb) % 16;
            auto patch = [&](u32x4_t (&k)[DL_HD / 32], u32x2_t (&v)[DL_HD / 16]) __attribute__((always_inline)) {
#pragma unroll
              for (int stp = 0; stp < DL_HD / 32; ++stp) {
                const u32x4_t kx = *(const u32x4_t*)(sh.q[16] + stp * 32 + 8 * qd);
                if (j == jn) k[stp] = kx;
              }
              const uint32_t keep = jn % 2 ? 0x0000ffffu : 0xffff0000u;
#pragma unroll
              for (int dt = 0; dt < DL_HD / 16; ++dt) {
                const uint32_t vn = (uint32_t)sh.q[17][16 * dt + j] << (16 * (jn % 2));
                if (qd == jn / 4) {
                  if ((jn % 4) / 2 == 0) v[dt][0] = (v[dt][0] & keep) | vn;
                  else v[dt][1] = (v[dt][1] & keep) | vn;
                }
              }
            };
            if (pos - kb < 16) patch(kf[0], vf[0]);
            else patch(kf[1], vf[1]);
          }
          float sc[8];
          decode_scores<DL_HD, false, 2>(kf, qf, kb, kb, k_end, qd, p.scale_log2e, m, l, sc, -1, nullptr);
          decode_values<DL_HD, false, 2>(vf, sc, kb, kb, k_end, qd, o, -1, nullptr);
        }
        if (j < G) {
#pragma unroll
          for (int dt = 0; dt < DL_HD / 16; ++dt) *(f32x4_t*)&sh.o[cwave][j][dt * 16 + 4 * qd] = o[dt];
        }
        if (qd == 0) {
          sh.m[cwave][j] = m;
          sh.l[cwave][j] = l;
        }
        dl_barrier();
        // a head a wave, two elements a lane
        for (int col = cwave; col < G; col += 4) {
          float pm[4], mx = -INFINITY;
#pragma unroll
          for (int w = 0; w < 4; ++w) pm[w] = sh.m[w][col];
#pragma unroll
          for (int w = 0; w < 4; ++w) mx = fmaxf(mx, pm[w]);
          float a0 = 0.f, a1 = 0.f, den = 0.f;
#pragma unroll
          for (int w = 0; w < 4; ++w) {         // (a wave without keys has max -inf: weight 0)
            const float f = exp2_raw(pm[w] - mx);
            const float2 ov = *(const float2*)&sh.o[w][col][2 * lane];
            a0 = fmaf(f, ov.x, a0);
            a1 = fmaf(f, ov.y, a1);
            den = fmaf(f, sh.l[w][col], den);
          }
          const int head = s * nH + kvh * G + col;
          if (lost) continue;
          if (ctx <= DL_SPLIT) {
            const uint32_t mine = pack_bf16x2(a0 / den, a1 / den);
            const uint32_t other = __float_as_uint(lane_xor<1>(__uint_as_float(mine)));
            const uint32_t d0 = lane % 2 ? other : mine, d1 = lane % 2 ? mine : other;
            // copies lane % 2 and lane % 2 + 2
            const uint32_t to = ((lane % 2) * M * nH * (DL_HD / 4) + head * (DL_HD / 4) + lane / 2) * 16;
            store2(to, (set + at.attn) * 16, d0, d1, epoch);
            store2(to, (set + at.attn + 2 * M * nH * (DL_HD / 4)) * 16, d0, d1, epoch);
          } else {
            const uint32_t to = (set + at.part + (head * p.max_splits + sp) * (DL_PART / 2)) * 16;
            store2(lane * 16, to, __float_as_uint(a0), __float_as_uint(a1), epoch);
            if (lane == 0) store2(DL_HD / 2 * 16, to, __float_as_uint(mx), __float_as_uint(den), epoch);
          }
        }
        if constexpr (!FEW) ask_keys(layer, att + 1);
        dl_barrier();               // (the next split's partial outputs go where these are)
      }
      // ---- contexts of several splits: eight elements of a head a wave, eight splits side by side
      if (split) {
        const int lane = thread() % 64, d8 = lane % 8, slot = lane / 8;
        constexpr int pieces = DL_HD / 8;
        for (int item = cwave * wgs + wg; item < M * nH * pieces; item += 4 * wgs) {
          const int piece = item % pieces, head = item / pieces, s = M == 1 ? 0 : head / nH;
          const int last = (dl_const(args()->ctx_len)[s] - 1) / DL_SPLIT;
          if (last == 0) continue;
          const uint32_t from = (set + at.part + head * p.max_splits * (DL_PART / 2)) * 16;
          float mx = -INFINITY, acc = 0.f, den = 0.f;
          bool came = true;
          for (int sp0 = 0; sp0 <= last; sp0 += 8) {
            const uint32_t mine = min(sp0 + slot, last) * (DL_PART * 8);
            u32x4_t ml;
            u32x2_t v;
            came &= wait_for([&]() __attribute__((always_inline)) {
              v = __builtin_amdgcn_raw_buffer_load_b64(words, mine + (piece * 8 + d8) * 8, from, SC1);
              ml = load2(mine + DL_HD * 8, from);
              return ((v[1] ^ epoch) | (ml[1] ^ epoch) | (ml[3] ^ epoch)) != 0;
            });
            const float pm = sp0 + slot <= last ? __uint_as_float(ml[0]) : -INFINITY;
            const float most = fmaxf(mx, pm);
            const float f0 = most == mx ? 1.f : exp2_raw(mx - most), f1 = most == pm ? 1.f : exp2_raw(pm - most);
            const float w = sp0 + slot <= last ? f1 : 0.f;
            acc = fmaf(w, __uint_as_float(v[0]), acc * f0);
            den = fmaf(w, __uint_as_float(ml[2]), den * f0);
            mx = most;
          }
          float top = fmaxf(mx, lane_xor<8>(mx));
          top = apart_max<16>(top);
          top = apart_max<32>(top);
          const float f = exp2_raw(mx - top);
          acc *= f;
          den *= f;
          acc += lane_xor<8>(acc);
          den += lane_xor<8>(den);
          acc = apart_sum<16>(acc);
          den = apart_sum<16>(den);
          acc = apart_sum<32>(acc);
          den = apart_sum<32>(den);
          uint32_t d0, d1;
          quad_words(acc / den, d8, d0, d1);
          if (came && slot == 0)
            store2((((d8 % 4) * M * nH + head) * (DL_HD / 4) + piece * 2 + d8 / 4) * 16, (set + at.attn) * 16, d0,
                   d1, epoch);
        }
      }
      // ---- the attention's output into the stream
      if (n_sum > 0) {
        gather_rows(set + at.attn + copy * (M * nH * (DL_HD / 4)), nH * DL_HD, epoch);
        dl_barrier();
        const bool leave = dl_uniform(*dead) != 0;
        for (int k0 = 0; k0 == 0 || (FEW && k0 < n_sum); k0 += PIECE) {
          if (FEW && !leave) multiply(layer, 1, wg, k0, min(PIECE, n_sum - k0));
          dl_barrier();
          if (leave) { dl_barrier(); return false; }
          residual(ff_gain, L.ff_gain, k0, set + at.mid, set + at.mid_sq, epoch, false);
          dl_barrier();
        }
      }
      // ---- gate and up
      if (n_ff > 0) {
        gather_normed(set + at.mid, set + at.mid_sq, epoch);
        dl_barrier();
        float inv[M];
        inv_rms(p.eps_ff, inv);
        const bool leave = dl_uniform(*dead) != 0;
        for (int k0 = 0; k0 == 0 || (FEW && k0 < n_ff); k0 += FF_PIECE) {
          const int n = FEW ? min(FF_PIECE, n_ff - k0) : n_ff;
          if (FEW && !leave) multiply(layer, 2, ff_first, k0, n);
          dl_barrier();
          if (leave) { dl_barrier(); return false; }
          const uint32_t e_r = place().r;
          for (uint32_t e = place().pair; e < (uint32_t)n * M; e += 16) {
            const uint32_t tok = e % M, unit = e / M;
            float f = inv[0];
#pragma unroll
            for (int k = 1; k < M; ++k) f = tok == k ? inv[k] : f;
            const float gv = sum_waves(2 * M * unit + tok, e_r) * f, uv = sum_waves((2 * unit + 1) * M + tok, e_r) * f;
            uint32_t d0, d1;
            quad_words(gv / (1.0f + expf(-gv)) * uv, e_r, d0, d1);
            const uint32_t row = (e_r % DL_COPIES) * M + tok;
            store2((row * (p.ff / 4) + (ff_first + (k0 + unit) * wgs) * 4 + e_r / 4) * 16, (set + at.act) * 16, d0,
                   d1, epoch);
          }
          dl_barrier();
        }
      }
      // ---- down into the stream
      if (n_sum > 0) {
        gather_rows(set + at.act + copy * (M * p.ff / 4), p.ff, epoch);
        dl_barrier();
        if constexpr (!FEW) ask_keys(layer + 1, 0);
        const bool leave = dl_uniform(*dead) != 0;
        for (int k0 = 0; k0 == 0 || (FEW && k0 < n_sum); k0 += PIECE) {
          if (FEW && !leave) multiply(layer, 3, wg, k0, min(PIECE, n_sum - k0));
          dl_barrier();
          if (leave) { dl_barrier(); return false; }
          residual(next_gain, L.next_gain, k0, set + at.next, set + at.next_sq, epoch, layer + 1 == n_layers);
          dl_barrier();
        }
        return true;
      }
      if constexpr (!FEW) ask_keys(layer + 1, 0);
      return dl_uniform(*dead) == 0;
    };
    for (int layer = 0; layer < n_layers; ++layer)
      if (!run_layer(layer)) break;
    const DecodeArgs pp = args();
    if (dl_uniform(*dead) != 0) {
      Place e = place();
      for (; e.unit < (uint32_t)n_sum; e.unit += PIECE) {
        const size_t n = (size_t)e.tok * p.hidden + column(e);
        pp->x[n] = __uint_as_float(0x7fc00000u);
        pp->xg[n] = 0x7fc0;
      }
      __hip_atomic_store(pp->status, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  };
  if (few) all_layers(std::true_type{});
  else all_layers(std::false_type{});
}

template <int M>
static size_t dl_lds(const DecodeLayers& p) {
  // (behind the rows the 1040 bytes that a wave reads ahead of a row's end)
  const size_t need = sizeof(DecodeShared<M>) + (size_t)M * (p.hidden / 16) * 4 +
                      (size_t)M * dl_row(p.hidden, p.ff, p.nH) + 2 * 2 * 128 * DL_CW;
  const size_t alone = 84 * 1024;          // more than half of a CU's: one workgroup a CU
  return need > alone ? need : alone;
}

// bytes of `words` for M tokens
extern "C" long long zf_decode_layers_words(int M, int hidden, int ff, int nH, int nKV, int max_splits) {
  return 2 * 16 * (long long)dl_words(M, hidden, ff, nH, nKV, max_splits).all;
}

// Everything in `p` is device memory but p itself; rows and tables 16-byte aligned; a sequence a
// token.  The grid is one workgroup a CU.
extern "C" int zf_decode_layers(const DecodeLayers* args, int workgroups, hipStream_t stream) {
  DecodeLayers p = *args;
  const int M = p.tokens;
  if (M < 1 || M > DL_TOKENS || p.n_layers < 1 || workgroups < 1) return -3;
  if (p.hidden % 64 != 0 || p.ff % 64 != 0 || p.hidden < 512 || p.ff < 512 || p.nKV < 1 || p.nKV > 255 ||
      p.nH % p.nKV != 0 || p.nH / p.nKV > 15 || p.nH * DL_HD < 512 || p.page_size % 16 != 0 ||
      p.max_splits < 1 || p.max_splits > 255)
    return -3;
  int units = (p.nH + 2 * p.nKV) * (DL_HD / 16), table = (p.max_pages * p.page_size + DL_SPLIT - 1) / DL_SPLIT;
  if (p.hidden / 16 > units) units = p.hidden / 16;
  if (table > p.max_splits) return -3;
  const int per = DL_UNITS / M, ff_per = DL_FF_UNITS / M, splits = M * p.nKV * table;
  p.need = (units + per - 1) / per;
  if ((p.ff / 16 + ff_per - 1) / ff_per > p.need) p.need = (p.ff / 16 + ff_per - 1) / ff_per;
  if ((splits + DL_ATT - 1) / DL_ATT > p.need) p.need = (splits + DL_ATT - 1) / DL_ATT;
  if ((p.cos_t == nullptr) != (p.sin_t == nullptr) || (p.cos_t != nullptr && p.table_rows < 1)) return -3;
  const size_t lds = M == 1 ? dl_lds<1>(p) : M == 2 ? dl_lds<2>(p) : M == 3 ? dl_lds<3>(p) : dl_lds<4>(p);
  if (lds > 160 * 1024) return -3;
  void* params[] = {&p};
  const void* kernel = M == 1   ? (const void*)decode_layers_kernel<1, 3>
                       : M == 2 ? (const void*)decode_layers_kernel<2, 3>
                       : M == 3 ? (const void*)decode_layers_kernel<3, 3>
                                : (const void*)decode_layers_kernel<4, 3>;
  hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return (int)e;
  return (int)hipLaunchKernel(kernel, dim3(workgroups), dim3(DL_THREADS), params, lds, stream);
}
