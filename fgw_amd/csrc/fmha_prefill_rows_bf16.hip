// BF16 instantiations of the prefill layout's row-group variants.
#include "fmha_prefill.h"
#include "fmha_registry.h"

namespace fgw_mha {
FGW_MHA_FOR_PREFILL_ROWS(FGW_MHA_INSTANTIATE_PREFILL_ROWS, true)
}  // namespace fgw_mha
