// Single-token decode (one query row per request): the key layout's kernel
// for Sq = 1.
//
// One query row leaves the matrix cores nothing to do (a 32x32 tile would
// hold one live column), and the time is the time to read K and V once, so
// this kernel streams both straight from memory into registers and computes
// with the vector ALU: no LDS stage, no transposing read, no barrier in the
// main loop, and short enough that a small call is not spent on fetching its
// instructions. Math and results are fwd_kernel's (fmha_kernel.h), with P
// rounded to the input type for the PV product and all sums in fp32.
//
// A work item is (request b, KV split, head h). Its keys are cut into steps of
// STEP keys; wave w of the W waves takes steps w, w + W, ... In a step one load
// instruction reads KPI key rows, LPK = DPAD / 8 lanes to a row and 16 bytes
// to a lane, U instructions for K and U for V. Every lane group of LPK lanes
// keeps its own online-softmax state (running maximum m, row sum l, 8 output
// dims per lane) over the keys it sees; the states meet once, at the end:
// across the wave's groups by lane exchanges, across the waves through LDS.
// The K registers of the next step are loaded as soon as a step's scores are
// known and its V registers as soon as its products are done, so that one of
// the two is always in flight.
//
// What bounds it: memory reads for long caches (8 waves keep 64 KB in flight per
// workgroup; reads that the caches serve are bound by that and by the vector ALU, where
// the MFMA key kernel's DMA keeps 128 KB in flight: kernel_of in fmha_api.hip draws
// the line), the chain length -> table -> K -> V -> combine for short ones.
// Measured against the MFMA key kernel at Sq = 1 (D 128 unless said, K/V from three
// rotating sets): B16 H16 KV 1024-4096 pages of 16 125 -> 59-68 us, B8 H32 KV 2048
// D 96 65 -> 33 us, D 64 KV 4096 pages of 16 96 -> 53 us, D 256 B8 H8 KV 2048 31.6
// -> 25.5 us, B4 H32 KV 512 10.8 -> 9.8 us, B1 H1 KV 512 8.2 -> 7.8 us. Steps of 32
// keys at D 128 (twice the registers, one workgroup per CU) measured 0-8% slower
// except on the shortest calls (B1 H1 KV 512 7.4 us); 4 waves 1-7% slower; the heads
// of a key range as neighbours instead of a head's splits 7% slower.
#pragma once
#include "fmha_kernel.h"

namespace fgw_mha {

template <bool BF16_, int DPAD_>
struct DCfg {
  static constexpr bool BF16 = BF16_;
  static constexpr int DPAD = DPAD_;
  static constexpr int W = 8;
  static constexpr int THREADS = 64 * W;
  static constexpr int ROWS_TILE = 1;
  static constexpr int BN = 32;              // keys per block of the split partition
  static constexpr int LPK = DPAD / 8;       // lanes per key row
  static constexpr int KPI = 64 / LPK;       // key rows per load instruction
  static constexpr int STEP = DPAD == 256 ? 8 : (DPAD == 128 ? 16 : 32);  // keys per step
  static constexpr int U = STEP / KPI;       // load instructions per step, of K and of V
  static_assert(DPAD == 32 || DPAD == 64 || DPAD == 128 || DPAD == 256, "head-dim tiles");
  static_assert(U >= 2 && U % 2 == 0 && BN % STEP == 0, "whole steps per block, weights in pairs");
};

// Eight fp16/bf16 values of a 16-byte chunk as fp32.
template <bool BF16>
__device__ __forceinline__ void unpack8(u32x4 x, float (&f)[8]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const u32 w = x[i];  // (a bit cast of x[i] itself would read element 0)
    if constexpr (BF16) {
      f[2 * i] = __uint_as_float(w << 16);
      f[2 * i + 1] = __uint_as_float(w & 0xffff0000u);
    } else {
      const f16x2 h = __builtin_bit_cast(f16x2, w);
      f[2 * i] = (float)h[0];
      f[2 * i + 1] = (float)h[1];
    }
  }
}

// Two values rounded to the input type.
template <bool BF16>
__device__ __forceinline__ void round_pair(float& a, float& b) {
  const u32 w = Elem<BF16>::pack2(a, b);
  if constexpr (BF16) {
    a = __uint_as_float(w << 16);
    b = __uint_as_float(w & 0xffff0000u);
  } else {
    const f16x2 h = __builtin_bit_cast(f16x2, w);
    a = (float)h[0];
    b = (float)h[1];
  }
}

// x plus its value in the lane that the DPP control names (within rows of 16 lanes).
template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
  const int y = __builtin_amdgcn_update_dpp(0, (int)__float_as_uint(x), CTRL, 0xf, 0xf, true);
  return x + __uint_as_float((u32)y);
}

// Sum over the LPK lanes of a key row, in every lane of it: neighbours, pairs
// of neighbours, halves of 8, halves of 16, rows of 16.
template <int LPK>
__device__ __forceinline__ float row_sum(float x) {
  x = dpp_add<0xB1>(x);                             // quad_perm [1, 0, 3, 2]
  x = dpp_add<0x4E>(x);                             // quad_perm [2, 3, 0, 1]
  if constexpr (LPK >= 8) x = dpp_add<0x141>(x);    // row_half_mirror
  if constexpr (LPK >= 16) x = dpp_add<0x140>(x);   // row_mirror
  if constexpr (LPK >= 32) {
    const auto sw = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
  }
  return x;
}

// The state of one lane: its group's running maximum (log2 units) and row sum,
// and the lane's eight output dims.
struct DecodeState {
  float m, l;
  float acc[8];
};

// Scores of a step's keys (log2 units), key u KPI + lane / LPK in s[u]. Lanes
// past D (dim_live false) hold a copy of the row's last chunk and add nothing.
template <class C>
__device__ __forceinline__ void step_scores(const u32x4 (&k)[C::U], const float (&q)[8],
                                            bool dim_live, float (&s)[C::U]) {
#pragma unroll
  for (int u = 0; u < C::U; ++u) {
    float f[8];
    unpack8<C::BF16>(k[u], f);
    float a = q[0] * f[0], b = q[1] * f[1];
#pragma unroll
    for (int i = 2; i < 8; i += 2) {
      a = __builtin_fmaf(q[i], f[i], a);
      b = __builtin_fmaf(q[i + 1], f[i + 1], b);
    }
    s[u] = row_sum<C::LPK>(dim_live ? a + b : 0.0f);
    // Fence: the scheduler would otherwise unpack every key first and hold
    // all the fp32 values at once.
    if (u % 2) __builtin_amdgcn_sched_barrier(0);
  }
}

// Online softmax of a step: m moves to the running maximum, l and acc follow,
// s[u] becomes the key's weight exp2(s - m).
template <class C>
__device__ __forceinline__ void step_softmax(float (&s)[C::U], DecodeState& st) {
  float mx = st.m;
#pragma unroll
  for (int u = 0; u < C::U; ++u) mx = fmaxf(mx, s[u]);
  const float alpha = __builtin_amdgcn_exp2f(st.m - mx);
  st.m = mx;
  float sum = 0.0f;
#pragma unroll
  for (int u = 0; u < C::U; ++u) {
    s[u] = __builtin_amdgcn_exp2f(s[u] - mx);
    sum += s[u];
  }
  // The row sum is of the fp32 weights, the products take them rounded to the
  // input type: the operator's rounding points, the same in every kernel.
#pragma unroll
  for (int u = 0; u < C::U; u += 2) round_pair<C::BF16>(s[u], s[u + 1]);
  st.l = __builtin_fmaf(st.l, alpha, sum);
#pragma unroll
  for (int i = 0; i < 8; ++i) st.acc[i] *= alpha;
}

template <class C>
__device__ __forceinline__ void step_values(const u32x4 (&v)[C::U], const float (&p)[C::U],
                                            DecodeState& st) {
#pragma unroll
  for (int u = 0; u < C::U; ++u) {
    float f[8];
    unpack8<C::BF16>(v[u], f);
#pragma unroll
    for (int i = 0; i < 8; ++i) st.acc[i] = __builtin_fmaf(p[u], f[i], st.acc[i]);
    if (u % 2) __builtin_amdgcn_sched_barrier(0);
  }
}

// What the steps of one work item share.
struct DecodeItem {
  const int32_t* table_b;
  const char* kb;  // K and V of head h at pool row 0
  const char* vb;
  int64_t row_bytes;
  int len, end;  // live keys; steps n < end
};

// Page ids of step n, lane u (mod U) the one of load instruction u's rows:
// page_size % KPI == 0, so they all lie in one page. Clamped to the table; an
// id past the live pages is not used.
template <class C>
__device__ __forceinline__ int32_t step_ids(const FwdParams& p, const int32_t* table_b, int n,
                                            int lane) {
  const u32 pos = (u32)n * C::STEP + (u32)(lane % C::U * C::KPI);
  const u32 pg = div_page(pos, p.page_magic, p.page_shift);
  const u32 last = (u32)p.width - 1u;
  return table_b[pg < last ? pg : last];
}

// The rows of step n's load instructions, lane u (mod U) instruction u's: byte
// offset of the first one in the pool, and bytes from there to the end of the
// last live one (0 where no row is below len or the page id lies outside the
// pool).
struct StepRows {
  int64_t off;
  u32 size;
};
template <class C>
__device__ __forceinline__ StepRows step_rows(const FwdParams& p, const DecodeItem& it, int n,
                                              int32_t id, int lane) {
  const int pos = n * C::STEP + lane % C::U * C::KPI;
  const u32 pg = div_page((u32)pos, p.page_magic, p.page_shift);
  const int64_t row = (int64_t)id * p.page_size + ((u32)pos - pg * (u32)p.page_size);
  const int live = it.len - pos;
  const bool ok = live > 0 && row >= 0 && row < p.pool_rows;
  const u32 rows = (u32)(live < C::KPI ? live : C::KPI);
  return StepRows{ok ? row * it.row_bytes : 0,
                  ok ? (rows - 1u) * (u32)it.row_bytes + (u32)p.dim * 2u : 0u};
}

// The K or V rows of one step. Every instruction reads through a buffer
// descriptor of its own rows, so that lanes of rows at or past len (or of a
// page outside the pool) read zeros without a branch. NT: non-temporal.
template <class C, bool NT>
__device__ __forceinline__ void load_step(const char* base, const StepRows& r, u32 lane_off,
                                          u32x4 (&x)[C::U]) {
#pragma unroll
  for (int u = 0; u < C::U; ++u) {
    const u32 lo = __builtin_amdgcn_readlane((u32)r.off, u);
    const u32 hi = __builtin_amdgcn_readlane((u32)((uint64_t)r.off >> 32), u);
    const u32 size = __builtin_amdgcn_readlane(r.size, u);
    const char* first = base + (int64_t)(((uint64_t)hi << 32) | lo);
    const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(first), (short)0, (int)size,
                                                        0x00027000);
    x[u] = __builtin_bit_cast(
        u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)lane_off, 0, NT ? 2 : 0));
  }
}

// Steps n, n + W, ... < end of one wave.
template <class C, bool NT>
__device__ __forceinline__ void decode_steps(const FwdParams& p, const DecodeItem& it, int n,
                                             int32_t ids, const float (&q)[8], DecodeState& st,
                                             int lane, u32 lane_off) {
  const bool dim_live = lane % C::LPK * 8 < p.dim;
  u32x4 k[C::U], v[C::U];
  StepRows rows = step_rows<C>(p, it, n, ids, lane);
  ids = step_ids<C>(p, it.table_b, n + C::W, lane);
  load_step<C, NT>(it.kb, rows, lane_off, k);
  load_step<C, NT>(it.vb, rows, lane_off, v);
  for (;;) {
    float s[C::U];
    step_scores<C>(k, q, dim_live, s);
    if ((n + 1) * C::STEP > it.len) {
#pragma unroll
      for (int u = 0; u < C::U; ++u)
        s[u] = n * C::STEP + u * C::KPI + lane / C::LPK < it.len ? s[u] : -INFINITY;
    }
    n += C::W;
    const bool more = n < it.end;
    if (more) {
      rows = step_rows<C>(p, it, n, ids, lane);
      // The ids of the step after before the rows: the wait for those rows
      // then covers them.
      ids = step_ids<C>(p, it.table_b, n + C::W, lane);
      load_step<C, NT>(it.kb, rows, lane_off, k);
    }
    step_softmax<C>(s, st);
    step_values<C>(v, s, st);
    if (!more) return;
    load_step<C, NT>(it.vb, rows, lane_off, v);
  }
}

// The wave's lane groups' states into one, in the lanes of group 0 (and all
// others): rescaled to the common maximum and summed.
template <class C>
__device__ __forceinline__ void merge_groups(DecodeState& st) {
  float top = st.m;
#pragma unroll
  for (int x = C::LPK; x < 64; x *= 2) top = fmaxf(top, __shfl_xor(top, x, 64));
  const float w = __builtin_amdgcn_exp2f(st.m - top);
  st.m = top;
  st.l *= w;
#pragma unroll
  for (int i = 0; i < 8; ++i) st.acc[i] *= w;
#pragma unroll
  for (int x = C::LPK; x < 64; x *= 2) {
    st.l += __shfl_xor(st.l, x, 64);
#pragma unroll
    for (int i = 0; i < 8; ++i) st.acc[i] += __shfl_xor(st.acc[i], x, 64);
  }
}

template <class C>
__global__ __launch_bounds__(C::THREADS, 4) void decode_kernel(FwdParams p_arg,
                                                               const int32_t* __restrict__ table,
                                                               const int32_t* __restrict__ lengths) {
  __shared__ float sm[C::W], sl[C::W];
  __shared__ __attribute__((aligned(16))) float so[C::W * C::DPAD];
  __shared__ int32_t pre[kMaxBalancedBatch + 1];
  __shared__ int32_t merge_flag;
  // The parameters, read again where a part needs them (as in fwd_kernel)
  // instead of held in scalar registers across the steps.
  const FwdParams& p = p_arg;
  auto kernarg = []() {
    typedef const __attribute__((address_space(4))) FwdParams* KP;
    KP kp = (KP)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(kp));
    return (const FwdParams*)kp;
  };
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int chunk = lane % C::LPK;
  const int64_t row_bytes = (int64_t)p.heads * p.dim * 2;
  const int capacity = p.width * p.page_size;
  // The lane's byte offset in a load instruction's rows (lanes past D: the
  // row's last chunk).
  const int last_chunk = p.dim / 8 - 1;
  const u32 lane_off = (u32)(lane / C::LPK) * (u32)row_bytes +
                       16u * (u32)(chunk < last_chunk ? chunk : last_chunk);

  const bool balanced = p.mode == 1 && p.split_keys > 0;
  int work = p.work;
  if (balanced) {
    balanced_prefix(p, lengths, capacity, pre, wave, lane);
    work = __builtin_amdgcn_readfirstlane(pre[p.batch]) * p.heads;
  }
  const ProgramItems items = key_items(work);

  for (int i = 0; i < items.count; ++i) {
    FwdParams p = *kernarg();
    // Even splits: request, head, split (split fastest). Balanced ones:
    // request, split, head, since the splits of a request are not a constant.
    int b, h, split, nsplit = p.splits;
    const int w = items.first + i * items.step;
    if (balanced) {
      const int g = w / p.heads;
      h = w - g * p.heads;
      b = balanced_request(pre, p.batch, g, split, nsplit);
    } else {
      b = w / (p.splits * p.heads);
      const int r = w - b * (p.splits * p.heads);
      h = r / p.splits;
      split = r - h * p.splits;
    }
    DecodeItem it;
    it.table_b = table + (int64_t)b * p.width;
    it.kb = static_cast<const char*>(p.k) + (int64_t)h * p.dim * 2;
    it.vb = static_cast<const char*>(p.v) + (int64_t)h * p.dim * 2;
    it.row_bytes = row_bytes;
    constexpr int kSteps = C::BN / C::STEP;
    // The wave's first page ids for a full cache, read together with the
    // length instead of after it; a shorter length that moves the split's
    // first key reads them again.
    const int guess = split_bound((capacity + C::BN - 1) / C::BN, split, nsplit) * kSteps + wave;
    int32_t ids = step_ids<C>(p, it.table_b, guess, lane);
    // The lane's eight dims of q, scaled to log2 units (zero past D).
    float q[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (chunk * 8 < p.dim) {
      const u16* qp = static_cast<const u16*>(p.q) + ((int64_t)b * p.heads + h) * p.dim;
      unpack8<C::BF16>(load16(qp + 8 * chunk), q);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) q[j] *= p.scale_log2;

    int len = lengths[b];
    len = len < 0 ? 0 : (len > capacity ? capacity : len);
    const int nblk = (len + C::BN - 1) / C::BN;
    const int n = split_bound(nblk, split, nsplit) * kSteps + wave;
    it.len = len;
    it.end = split_bound(nblk, split + 1, nsplit) * kSteps;

    DecodeState st;
    st.m = kNegBig;
    st.l = 0.0f;
#pragma unroll
    for (int j = 0; j < 8; ++j) st.acc[j] = 0.0f;
    if (n < it.end) {
      if (n != guess) ids = step_ids<C>(p, it.table_b, n, lane);
      if (stream_kv(p, stream_probe(p, table, lengths, b, (n - wave) * C::STEP, lane), row_bytes, lane))
        decode_steps<C, true>(p, it, n, ids, q, st, lane, lane_off);
      else
        decode_steps<C, false>(p, it, n, ids, q, st, lane, lane_off);
    }
    merge_groups<C>(st);
    p = *kernarg();

    // The waves' states through LDS.
    if (i > 0) __syncthreads();  // the previous item's are read
    if (lane == 0) {
      sm[wave] = st.m;
      sl[wave] = st.l;
    }
    if (lane < C::LPK) {
      float* o = so + wave * C::DPAD + 8 * chunk;
      *reinterpret_cast<f32x4*>(o) = f32x4{st.acc[0], st.acc[1], st.acc[2], st.acc[3]};
      *reinterpret_cast<f32x4*>(o + 4) = f32x4{st.acc[4], st.acc[5], st.acc[6], st.acc[7]};
    }
    __syncthreads();
    const int d0 = 4 * tid;
    if (d0 < p.dim) {
      float top = kNegBig;
#pragma unroll
      for (int k = 0; k < C::W; ++k) top = fmaxf(top, sm[k]);
      float tot = 0.0f;
      f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int k = 0; k < C::W; ++k) {
        const float wt = __builtin_amdgcn_exp2f(sm[k] - top);
        tot += sl[k] * wt;
        acc += *reinterpret_cast<const f32x4*>(so + k * C::DPAD + d0) * wt;
      }
      store_row<C>(p, b, h, split, 0, d0, acc, 1.0f / fmaxf(tot, 1.0e-30f));
      if (p.mode == 1 && tid == 0) {
        float* lp = p.lse + ((int64_t)b * p.heads + h) * p.splits + split;
        if (p.arrivals != nullptr)
          __hip_atomic_store(lp, lse_of(top, tot), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else
          *lp = lse_of(top, tot);
      }
    }
    if (p.mode == 1 && p.arrivals != nullptr)
      arrive_and_merge<C::BF16, C::THREADS, C::ROWS_TILE, kFusedMergeMaxChunk<C::DPAD>>(
          p, b, h, 0, nsplit, reinterpret_cast<unsigned char*>(&merge_flag), tid);
  }
}

// Resident workgroups per CU (the launch bound's registers; LDS allows more).
constexpr int kDecodeWgPerCu = 2;

// Shapes this kernel takes: load instructions whose rows lie in one page and
// span less than 2^31 bytes (a descriptor's offsets are 32 bits).
inline bool decode_takes(int dpad, int64_t row_bytes, int page_size) {
  const int kpi = 64 / (dpad / 8);
  return page_size % kpi == 0 && row_bytes * kpi < (int64_t(1) << 31);
}

template <bool BF16, int DPAD>
hipError_t launch_decode(const FwdParams& p, int grid, hipStream_t stream) {
  using C = DCfg<BF16, DPAD>;
  decode_kernel<C><<<dim3(grid), dim3(C::THREADS), 0, stream>>>(p, p.table, p.lengths);
  return hipGetLastError();
}

}  // namespace fgw_mha
