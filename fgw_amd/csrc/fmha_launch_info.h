// Which kernel a plan's call launches, and how. For tests and diagnostics of
// this library only: not part of the C ABI (include/fgw_mha.h), which leaves
// the choice of a kernel variant open.
#pragma once
#include "../../include/fgw_mha.h"

namespace fgw_mha {

// The forward kernels (order: _lib.KERNELS in fgw_amd/_lib.py).
enum Kernel : int32_t {
  kKernelQuery = 0,      // fwd_kernel, query layout
  kKernelQueryGroups,    // its row-group variant
  kKernelQueryDual,      // its eight-wave variant (head-dim tile 256)
  kKernelKey,            // fwd_kernel, key layout
  kKernelKeyGroups,      // its row-group variant
  kKernelKeyStream,      // its variant with non-temporal loads
  kKernelDecode,         // decode_kernel (Sq = 1)
  kKernelPrefill,        // prefill_kernel
  kKernelPrefillGroups,  // its row-group variant
  kKernelPrefillPadded,  // the same for head dims below their tile
  kKernelHalf,           // half_kernel
  kKernelHalfPadded,     // the same for head dims below their tile
};

struct LaunchInfo {
  int32_t kernel;         // Kernel
  int32_t threads;        // per program
  int32_t rows_per_item;  // query rows of a work item
  int32_t q_tiles;        // ceil(Sq / rows of its query tiles)
  int32_t work_items;
  int32_t grid;           // programs
  int64_t stream_bytes;   // FwdParams::stream_bytes
  int32_t longest_first;  // FwdParams::longest_first
};

}  // namespace fgw_mha

// Fills `info` for a call of fgw_mha_fwd with this plan. Host arithmetic only; the
// status codes of the ABI.
extern "C" int fgw_internal_launch_info(const fgw_mha_shape* shape, const fgw_mha_plan_t* plan,
                                        fgw_mha::LaunchInfo* info);
