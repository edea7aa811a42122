// BF16 instantiations of the half-tile kernel.
#include "fmha_half.h"
#include "fmha_registry.h"

namespace fgw_mha {
FGW_MHA_FOR_PREFILL_ROWS(FGW_MHA_INSTANTIATE_HALF, true)
}  // namespace fgw_mha
