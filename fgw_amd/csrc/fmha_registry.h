// Host-side table of the compiled kernel instantiations.
#pragma once
#include <hip/hip_runtime.h>

#include "fmha_params.h"

namespace fgw_mha {

typedef hipError_t (*FwdLaunchFn)(const FwdParams&, int, hipStream_t);
typedef int (*OccupancyFn)();

struct FwdEntry {
  FwdLaunchFn launch;
  OccupancyFn occupancy;
};

// Head-dim tiles with a compiled kernel: 32, 64, 128, 256 (D padded to a
// power of two, cube_general.py:31).
inline int dim_tile(int dim) {
  int t = 32;
  while (t < dim) t *= 2;
  return t;
}

// The kernel of (dtype, head-dim tile, layout, stages); stages 0 is the
// instantiation's default, 1 the key layout's single-stage variant (tile 128).
FwdEntry fwd_entry(bool bf16, int dpad, int layout, int stages = 0);
// The prefill layout's row-group kernel of (dtype, head-dim tile, rows mode).
FwdLaunchFn prefill_rows_entry(bool bf16, int dpad, int rows);
// The row-group kernel of (dtype, head-dim tile, key or query layout, stages).
FwdLaunchFn groups_entry(bool bf16, int dpad, int layout, int stages);
// The key layout's kernel with non-temporal loads (kStream) of (dtype, head-dim
// tile, stages); null for tile 32.
FwdLaunchFn stream_entry(bool bf16, int dpad, int stages);
// The query layout's kernel of eight waves (kDual), head-dim tile 256.
FwdLaunchFn dual_entry(bool bf16);
// The half-tile kernel of (dtype, head-dim tile, rows mode).
FwdLaunchFn half_entry(bool bf16, int dpad, int rows);
// The key layout's kernel of (dtype, head-dim tile) for Sq = 1.
FwdLaunchFn decode_entry(bool bf16, int dpad);
hipError_t launch_merge(bool bf16, const MergeParams& p, hipStream_t stream);
hipError_t launch_gather(const GatherParams& p, hipStream_t stream);
hipError_t launch_pack(const PackParams& p, int total_pages, hipStream_t stream);
hipError_t launch_group_merge(bool bf16, const GroupMergeParams& p, int groups, hipStream_t stream);

}  // namespace fgw_mha

// Explicit instantiation lists, expanded once per translation unit.
#define FGW_MHA_FOR_DPAD_LO(X, BF) X(BF, 32) X(BF, 64)
#define FGW_MHA_FOR_DPAD_HI(X, BF) X(BF, 128) X(BF, 256)
#define FGW_MHA_INSTANTIATE(BF, DP)                                                         \
  template hipError_t launch_fwd<BF, DP, kLayoutQuery>(const FwdParams&, int, hipStream_t); \
  template hipError_t launch_fwd<BF, DP, kLayoutKey>(const FwdParams&, int, hipStream_t);   \
  template int occupancy_fwd<BF, DP, kLayoutQuery>();                                       \
  template int occupancy_fwd<BF, DP, kLayoutKey>();
// The key layout's single-stage variant: head-dim tile 128 (two workgroups per CU).
#define FGW_MHA_INSTANTIATE_KEY_SINGLE(BF)                                                  \
  template hipError_t launch_fwd<BF, 128, kLayoutKey, 1>(const FwdParams&, int, hipStream_t); \
  template int occupancy_fwd<BF, 128, kLayoutKey, 1>();
#define FGW_MHA_EXTERN_KEY_SINGLE(BF)                                                              \
  extern template hipError_t launch_fwd<BF, 128, kLayoutKey, 1>(const FwdParams&, int, hipStream_t); \
  extern template int occupancy_fwd<BF, 128, kLayoutKey, 1>();
// The prefill layout exists for head-dim tiles 64 and 128.
#define FGW_MHA_FOR_PREFILL_LO(X, BF) X(BF, 64)
#define FGW_MHA_FOR_PREFILL_HI(X, BF) X(BF, 128)
#define FGW_MHA_INSTANTIATE_PREFILL(BF, DP)                                   \
  template hipError_t launch_prefill<BF, DP>(const FwdParams&, int, hipStream_t); \
  template int occupancy_prefill<BF, DP>();
#define FGW_MHA_EXTERN_PREFILL(BF, DP)                                               \
  extern template hipError_t launch_prefill<BF, DP>(const FwdParams&, int, hipStream_t); \
  extern template int occupancy_prefill<BF, DP>();
// The prefill layout's row-group variants (RowsMode in fmha_prefill.h): 1 for
// pages that key blocks straddle, 2 for head dims below their tile.
#define FGW_MHA_FOR_PREFILL_ROWS(X, BF) X(BF, 64, 1) X(BF, 128, 1) X(BF, 64, 2) X(BF, 128, 2)
#define FGW_MHA_INSTANTIATE_PREFILL_ROWS(BF, DP, RM) \
  template hipError_t launch_prefill<BF, DP, RM>(const FwdParams&, int, hipStream_t);
#define FGW_MHA_EXTERN_PREFILL_ROWS(BF, DP, RM) \
  extern template hipError_t launch_prefill<BF, DP, RM>(const FwdParams&, int, hipStream_t);
// The row-group kernels of the key layout (every head-dim tile, and the
// single-stage variant of tile 128) and of the query layout.
#define FGW_MHA_FOR_GROUPS(X, BF)                                                              \
  X(BF, 32, kLayoutKey, 0) X(BF, 64, kLayoutKey, 0) X(BF, 128, kLayoutKey, 0)                  \
  X(BF, 256, kLayoutKey, 0) X(BF, 128, kLayoutKey, 1) X(BF, 32, kLayoutQuery, 0)               \
  X(BF, 64, kLayoutQuery, 0) X(BF, 128, kLayoutQuery, 0) X(BF, 256, kLayoutQuery, 0)
#define FGW_MHA_INSTANTIATE_GROUPS(BF, DP, LY, ST) \
  template hipError_t launch_fwd<BF, DP, LY, ST, kGroups>(const FwdParams&, int, hipStream_t);
#define FGW_MHA_EXTERN_GROUPS(BF, DP, LY, ST) \
  extern template hipError_t launch_fwd<BF, DP, LY, ST, kGroups>(const FwdParams&, int, hipStream_t);
// The key layout's kernels with non-temporal loads.
#define FGW_MHA_FOR_STREAM(X, BF) X(BF, 64, 0) X(BF, 128, 0) X(BF, 256, 0) X(BF, 128, 1)
#define FGW_MHA_INSTANTIATE_STREAM(BF, DP, ST) \
  template hipError_t launch_fwd<BF, DP, kLayoutKey, ST, kStream>(const FwdParams&, int, hipStream_t);
#define FGW_MHA_EXTERN_STREAM(BF, DP, ST) \
  extern template hipError_t launch_fwd<BF, DP, kLayoutKey, ST, kStream>(const FwdParams&, int, \
                                                                         hipStream_t);
// The query layout's eight-wave kernel, head-dim tile 256.
#define FGW_MHA_INSTANTIATE_DUAL(BF) \
  template hipError_t launch_fwd<BF, 256, kLayoutQuery, 0, kDual>(const FwdParams&, int, hipStream_t);
// The half-tile kernel (128 query rows), both head-dim tiles, whole and padded
// head dims.
#define FGW_MHA_INSTANTIATE_HALF(BF, DP, RM) \
  template hipError_t launch_half<BF, DP, RM>(const FwdParams&, int, hipStream_t);
#define FGW_MHA_EXTERN_HALF(BF, DP, RM) \
  extern template hipError_t launch_half<BF, DP, RM>(const FwdParams&, int, hipStream_t);
// The key layout's single-token kernel (Sq = 1), every head-dim tile.
#define FGW_MHA_FOR_DECODE(X, BF) X(BF, 32) X(BF, 64) X(BF, 128) X(BF, 256)
#define FGW_MHA_INSTANTIATE_DECODE(BF, DP) \
  template hipError_t launch_decode<BF, DP>(const FwdParams&, int, hipStream_t);
#define FGW_MHA_EXTERN_DECODE(BF, DP) \
  extern template hipError_t launch_decode<BF, DP>(const FwdParams&, int, hipStream_t);
#define FGW_MHA_EXTERN(BF, DP)                                                                     \
  extern template hipError_t launch_fwd<BF, DP, kLayoutQuery>(const FwdParams&, int, hipStream_t); \
  extern template hipError_t launch_fwd<BF, DP, kLayoutKey>(const FwdParams&, int, hipStream_t);   \
  extern template int occupancy_fwd<BF, DP, kLayoutQuery>();                                       \
  extern template int occupancy_fwd<BF, DP, kLayoutKey>();
