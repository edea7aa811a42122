// Half-tile prefill: 128 query rows per work item, its key blocks shared out
// between the two wave groups.
//
// The prefill layout's items (fmha_prefill.h) are 256 query rows, one per CU;
// with fewer tiles than CUs, or causal tiles of very different lengths, most
// CUs wait for the longest item. Here a work item is 128 rows: waves 0-3 (group
// A) and 4-7 (group B) hold the same four sets of 32 rows, A takes the even
// and B the odd 64-key blocks, and their softmax states meet in LDS at the end.
// A step (two blocks) takes 1.3 to 1.7 times one block there, so an item of the
// same keys takes 0.65 to 0.85 of the time and there are twice as many, without
// the fp32 partials and the second launch of a KV split. Which plans take it, and
// what it measured: half_tiles in fmha_api.hip.
//
// The groups ping-pong as in fmha_prefill.h (matrix phase of one against
// vector phase of the other, a barrier between phases). Block j is block
// n = j / 2 of group j % 2: its scores are computed in phase j, its softmax runs
// in phase j + 1 and its PV product in phase j + 2. K and V of block j lie in
// ring slot 2 (j % 2) + n % 2. Every wave issues its share of K block p + 3 and
// V block p + 1 at the start of phase p: the slots' last readers were K block
// p - 1 in phase p - 1 and V block p - 3 in phase p - 1. The wait at the end of
// phase p leaves the loads of phases p - 1 and p in flight, so K block p + 1 and
// V block p - 1 (both issued in phase p - 2) have landed.
//
// What bounds it: no unit alone. At head-dim tile 64 (causal B1 H16 S4096) the CUs
// are busy 0.82 of the time, and of that the vector ALU 0.43 and the matrix cores 0.25
// (0.65 of it beside vector work); waves wait 0.22 of their cycles, at the phases'
// barriers and for operands, and the staged rows and states cost 0.13 in LDS bank
// conflicts. At 128 the K/V DMA adds to it, twice as much per row (every block serves
// 128 rows instead of 256).
#pragma once
#include "fmha_prefill.h"

namespace fgw_mha {

template <bool BF16_, int DPAD_, int ROWS_>
struct HCfg : PCfg<BF16_, DPAD_, ROWS_> {
  using P = PCfg<BF16_, DPAD_, ROWS_>;
  static constexpr int LAYOUT = kLayoutQuery;
  static constexpr int GROUP = 4;  // waves per group
  static constexpr int ROWS_TILE = GROUP * P::ROWS_WAVE;
  // After the rings: (m, l) of group B's lanes.
  static constexpr int STATE_BYTES = GROUP * 64 * 8;
  static constexpr int LDS_BYTES = P::RING_BYTES + STATE_BYTES;
  static constexpr int IPW = P::INSTR_PER_WAVE;
  static_assert(ROWS_ != kRowsBlock, "row groups");
  // Group B's O in the K ring, group A's staged output rows in the V ring.
  static_assert(GROUP * P::DT * 4096 <= P::NKSLOT * P::TILE_BYTES, "O fits the K ring");
  static_assert(GROUP * 32 * kStagedRowBytes<P> <= P::NVSLOT * P::TILE_BYTES,
                "staged rows fit the V ring");
};

template <class C>
__global__ __launch_bounds__(C::THREADS) void half_kernel(FwdParams p_arg,
                                                          const int32_t* __restrict__ table,
                                                          const int32_t* __restrict__ lengths) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[C::LDS_BYTES];
  const u32 kring_lds = lds_address(smem);
  const u32 vring_lds = kring_lds + (u32)(C::NKSLOT * C::TILE_BYTES);
  unsigned char* const vring = smem + C::NKSLOT * C::TILE_BYTES;

  // The parameters, read again per work item and for the output (as in
  // prefill_kernel).
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
  const int il = lane & 31, hh = lane >> 5;
  const Lanes<C> ln(lane);
  const int64_t row_bytes = (int64_t)p.heads * p.dim * 2;
  const DmaLanes<C> dl(lane, wave, row_bytes);
  const RowDma<C> rd(dl, p.dim, wave, lane);

  // Work items in the orders of prefill_kernel: one XCD's programs share a
  // contiguous, interleaved range, or the items go longest first over all (b, h).
  const int grid = gridDim.x;
  const bool longest_first = p.longest_first != 0;
  ProgramItems items = key_items(p.work);
  if (longest_first)
    items = ProgramItems{(int)blockIdx.x, grid,
                         (int)blockIdx.x < p.work ? (p.work - 1 - (int)blockIdx.x) / grid + 1 : 0};
  const int capacity = p.width * p.page_size;

  for (int it = 0; it < items.count; ++it) {
    const FwdParams p = *kernarg();  // this item's copy
    const bool group_a = opaque_uniform(wave) < C::GROUP;
    const int group = group_a ? 0 : 1;
    int w = items.first + it * items.step, split, qt;
    if (longest_first) {
      const int bhs = p.batch * p.heads;
      const int run = w / (p.splits * bhs);
      w -= run * (p.splits * bhs);
      qt = p.q_tiles - 1 - run;
      split = w / bhs;
      w -= split * bhs;
    } else {
      split = w % p.splits;
      w /= p.splits;
      qt = p.causal ? p.q_tiles - 1 - w % p.q_tiles : w % p.q_tiles;
      w /= p.q_tiles;
    }
    const int h = w % p.heads, b = w / p.heads;
    const int32_t* table_b = table + (int64_t)b * p.width;
    const char* kb = static_cast<const char*>(p.k) + (int64_t)h * p.dim * 2;
    const char* vb = static_cast<const char*>(p.v) + (int64_t)h * p.dim * 2;
    const int q0 = qt * C::ROWS_TILE;
    const int row_base = q0 + wave % C::GROUP * C::ROWS_WAVE;
    const int qrow = row_base + il;
    const int tile_last = (q0 + C::ROWS_TILE < p.sq ? q0 + C::ROWS_TILE : p.sq) - 1;

    u32x4 qf[C::KK];
    {
      const int dim = opaque_uniform(p.dim), hq = opaque_lane(hh);
      const u16* qp =
          static_cast<const u16*>(p.q) + (((int64_t)b * p.sq + qrow) * p.heads + h) * p.dim;
#pragma unroll
      for (int kk = 0; kk < C::KK; ++kk) {
        const int d = 16 * kk + 8 * hq;
        u32x4 val = {0u, 0u, 0u, 0u};
        if (qrow < p.sq && d < dim)
          val = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(qp + d));
        qf[kk] = val;
      }
    }

    int len = lengths[b];
    len = len < 0 ? 0 : (len > capacity ? capacity : len);
    int max_vis = p.causal ? len - p.sq + tile_last + 1 : len;
    max_vis = max_vis < 0 ? 0 : (max_vis > len ? len : max_vis);
    const int nblk = (max_vis + C::BN - 1) / C::BN;
    const int blk_begin = split_bound(nblk, split, p.splits);
    const int N = split_bound(nblk, split + 1, p.splits) - blk_begin;
    const int key0 = blk_begin * C::BN;

    // Rows of this wave and their visible key counts; blocks that end above
    // wmin hold keys some row of the wave cannot see and are masked.
    int wmin = p.causal ? len - p.sq + row_base + 1 : len;
    wmin = wmin < 0 ? 0 : (wmin > len ? len : wmin);
    int vis = p.causal ? len - p.sq + qrow + 1 : len;
    vis = vis < 0 ? 0 : (vis > len ? len : vis);

    float m = kNegBig, l = 0.0f;
    f32x16 o[C::DT];
#pragma unroll
    for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
      for (int v = 0; v < 16; ++v) o[dt][v] = 0.0f;

    __syncthreads();  // the previous work item no longer reads or stages in the rings

    if (N > 0) {
      // Offsets of the window that V's next block lies in, and of the next
      // one: K's next block is two ahead of V's.
      BlockWindow win0{0, window_offset<C>(p, table_b, row_bytes, key0, N, len, 0, wave, lane)};
      BlockWindow win1{1, window_offset<C>(p, table_b, row_bytes, key0, N, len, 1, wave, lane)};
      auto slot_of = [](int j) { return (u32)((2 * (j & 1) + ((j >> 1) & 1)) * C::TILE_BYTES); };
      // This wave's share of the K (V) tile of block j < N.
      auto issue = [&](int j, auto is_v) {
        constexpr bool V = decltype(is_v)::value;
        const char* base = V ? vb : kb;
        const u32 dst = (V ? vring_lds : kring_lds) + slot_of(j);
        const bool second = j / C::WINDOW != win0.w;
#pragma unroll
        for (int q = 0; q < C::IPW; ++q) {
          const int at = j % C::WINDOW * C::IPW + q;
          const int64_t off = second ? readlane64(win1.off, at) : readlane64(win0.off, at);
          if ((int32_t)((uint64_t)off >> 32) >= 0) {
            issue_row_group<C>(base + off, V ? rd.v[q] : rd.k[q], V ? rd.v_live[q] : rd.k_live[q],
                               dst + 1024u * (u32)(q * C::NWQ + wave));
          } else {
            int pos0 = key0 + j * C::BN;
            asm volatile("" : "+s"(pos0));  // no per-block induction variables for the rare path
            issue_slow_tile<C, V>(p, table_b, base, row_bytes, pos0, len, dst, wave, lane, q);
          }
        }
      };
      constexpr std::true_type on{};
      constexpr std::false_type off{};
      // The loads of phase p: K block p + 3, V block p + 1.
      auto issue_phase = [&](int ph) {
        if (ph + 3 < N) issue(ph + 3, off);
        const int jv = ph + 1;
        if (jv < N) {
          issue(jv, on);
          if ((jv + 1) / C::WINDOW != win0.w) {  // V's next block enters the next window
            win0 = win1;
            win1 = BlockWindow{win0.w + 1, window_offset<C>(p, table_b, row_bytes, key0, N, len,
                                                            win0.w + 1, wave, lane)};
          }
        }
      };
      // The end of phase p: everything issued before phase p - 1 has landed.
      // Those two phases issued K blocks p + 2, p + 3 and V blocks p, p + 1,
      // as far as they exist.
      auto wait_phase = [&](int ph) {
        if (ph + 3 < N)
          wait_vm<4 * C::IPW>();
        else if (ph + 2 < N)
          wait_vm<3 * C::IPW>();
        else if (ph + 1 < N)
          wait_vm<2 * C::IPW>();
        else if (ph < N)
          wait_vm<C::IPW>();
        else
          wait_vm<0>();
      };

      issue(0, off);
      if (1 < N) issue(1, off);
      if (2 < N) issue(2, off);
      issue(0, on);
      // K block 0 has landed; K blocks 1 and 2 and V block 0 may be in flight.
      if (2 < N)
        wait_vm<3 * C::IPW>();
      else if (1 < N)
        wait_vm<2 * C::IPW>();
      else
        wait_vm<C::IPW>();
      // Q's registers are waited for here, once (see prefill_kernel).
#pragma unroll
      for (int kk = 0; kk < C::KK; ++kk) asm volatile("" ::"v"(qf[kk]));
      __syncthreads();

      f32x16 s[C::ST];
      u32x4 pf[C::KS];
      const OperandAddr<C> ad(ln, kring_lds, vring_lds);
      // M(n) of this group: PV of its block n - 1, QK^T of its block n; odd =
      // n % 2 (a compile-time constant in the unrolled loops).
      auto mphase = [&](auto odd, auto pv, auto qk) {
        const u32 ks = (u32)((2 * group + (int)odd) * C::TILE_BYTES);
        const u32 vs = (u32)((2 * group + ((int)odd ^ 1)) * C::TILE_BYTES);
        matrix_phase<C, decltype(pv)::value, decltype(qk)::value>(ad, ks, vs, qf, pf, s, o);
      };
      const int vis4 = vis - 4 * hh;
      // S(n) of this group: softmax of its block n.
      auto sphase = [&](int n) {
        int pos0 = key0 + (2 * n + group) * C::BN;
        if (pos0 + C::BN > wmin) {
          asm volatile("" : "+s"(pos0));
          mask_from<C>(s, vis4 - pos0);
        }
        online_softmax<C>(s, m, l, o, p.scale_log2, pf);
      };
      constexpr std::integral_constant<int, 0> even{};
      constexpr std::integral_constant<int, 1> odd{};
      const int NA = (N + 1) >> 1, NB = N >> 1;  // blocks of groups A and B
      // Phases 2n and 2n + 1 for n = 0 .. NA, straight-line per group.
      if (group_a) {
        auto body = [&](int n, auto par) {
          issue_phase(2 * n);
          mphase(par, on, on);
          wait_phase(2 * n);
          __syncthreads();
          issue_phase(2 * n + 1);
          sphase(n);
          wait_phase(2 * n + 1);
          __syncthreads();
        };
        issue_phase(0);
        mphase(even, off, on);
        wait_phase(0);
        __syncthreads();
        issue_phase(1);
        sphase(0);
        wait_phase(1);
        __syncthreads();
        int n = 1;
        for (; n + 2 <= NA; n += 2) {
          body(n, odd);
          body(n + 1, even);
        }
        if (n < NA) {
          body(n, odd);
          ++n;
        }
        mphase(NA & 1, on, off);
        wait_phase(2 * NA);  // this wave's share of V for group B's last phase
        __syncthreads();
        __syncthreads();
      } else {
        auto body = [&](int n, auto par) {
          issue_phase(2 * n);
          sphase(n - 1);
          wait_phase(2 * n);
          __syncthreads();
          issue_phase(2 * n + 1);
          mphase(par, on, on);
          wait_phase(2 * n + 1);
          __syncthreads();
        };
        issue_phase(0);
        wait_phase(0);
        __syncthreads();
        issue_phase(1);
        if (NB > 0) mphase(even, off, on);
        wait_phase(1);
        __syncthreads();
        int n = 1;
        for (; n + 2 <= NB; n += 2) {
          body(n, odd);
          body(n + 1, even);
        }
        if (n < NB) {
          body(n, odd);
          ++n;
        }
        // n = NB (or 1 without a block): the last block's softmax and PV, then
        // the phases that only group A has.
        if (NB > 0) {
          issue_phase(2 * NB);
          sphase(NB - 1);
          wait_phase(2 * NB);
          __syncthreads();
          issue_phase(2 * NB + 1);
          mphase(NB & 1, on, off);
          wait_phase(2 * NB + 1);
          __syncthreads();
        }
        for (int k = NB > 0 ? NB + 1 : 1; k <= NA; ++k) {
          __syncthreads();
          __syncthreads();
        }
      }
    }

    // Group B's state to group A through LDS: no DMA is in flight and no wave
    // reads the rings.
    float* const state = reinterpret_cast<float*>(smem + C::RING_BYTES);
    const int gw = opaque_uniform(wave) % C::GROUP, lo = opaque_lane(lane);
    if (!group_a) {
      state[gw * 128 + lo] = m;
      state[gw * 128 + 64 + lo] = l;
      f32x4* dst = reinterpret_cast<f32x4*>(smem + gw * C::DT * 4096);
#pragma unroll
      for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
        for (int gq = 0; gq < 4; ++gq)
          dst[(dt * 4 + gq) * 64 + lo] =
              f32x4{o[dt][4 * gq], o[dt][4 * gq + 1], o[dt][4 * gq + 2], o[dt][4 * gq + 3]};
    }
    __syncthreads();
    if (!group_a) continue;  // the barrier at the item top joins the groups again

    {
      const float mb = state[gw * 128 + lo], lb = state[gw * 128 + 64 + lo];
      const float top = fmaxf(m, mb);
      const float wa = __builtin_amdgcn_exp2f(m - top), wb = __builtin_amdgcn_exp2f(mb - top);
      const f32x4* src = reinterpret_cast<const f32x4*>(smem + gw * C::DT * 4096);
#pragma unroll
      for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
        for (int gq = 0; gq < 4; ++gq) {
          const f32x4 x = src[(dt * 4 + gq) * 64 + lo];
#pragma unroll
          for (int i = 0; i < 4; ++i) o[dt][4 * gq + i] = o[dt][4 * gq + i] * wa + x[i] * wb;
        }
      m = top;
      l = l * wa + lb * wb;
    }
    const FwdParams po = *kernarg();
    const int ho = opaque_lane(hh), qr = row_base + opaque_lane(il);
    const float tot = pair_sum(l), inv = 1.0f / fmaxf(tot, 1.0e-30f);
    const bool f32 = po.mode == 1;
    if (po.dim == C::DPAD) {
      float* fdst = f32 ? po.parts + ((((int64_t)b * po.heads + h) * po.splits + split) * po.sq +
                                      row_base) * C::DPAD
                        : nullptr;
      unsigned char* bdst = f32 ? nullptr
                                : static_cast<unsigned char*>(po.out) +
                                      (((int64_t)b * po.sq + row_base) * po.heads + h) * C::DPAD * 2;
      store_rows_staged<C>(vring + gw * 32 * kStagedRowBytes<C>, lane, o, inv, f32, fdst, bdst,
                           (int64_t)po.heads * C::DPAD * 2, po.sq - row_base);
    } else if (qr < po.sq) {
#pragma unroll
      for (int dt = 0; dt < C::DT; ++dt)
#pragma unroll
        for (int gq = 0; gq < 4; ++gq) {
          const int d0 = 32 * dt + 8 * gq + 4 * ho;
          if (d0 < po.dim) {
            f32x4 val = {o[dt][4 * gq], o[dt][4 * gq + 1], o[dt][4 * gq + 2], o[dt][4 * gq + 3]};
            store_row<C>(po, b, h, split, qr, d0, val, inv);
          }
        }
    }
    if (f32 && ho == 0 && qr < po.sq)
      po.lse[(((int64_t)b * po.heads + h) * po.splits + split) * po.sq + qr] = lse_of(m, tot);
  }
}

// One workgroup per work item where the plan has as many programs as items
// (p.work is the variant's own item count).
template <bool BF16, int DPAD, int ROWS>
hipError_t launch_half(const FwdParams& p, int grid, hipStream_t stream) {
  using C = HCfg<BF16, DPAD, ROWS>;
  half_kernel<C><<<dim3(grid), dim3(C::THREADS), 0, stream>>>(p, p.table, p.lengths);
  return hipGetLastError();
}

}  // namespace fgw_mha
