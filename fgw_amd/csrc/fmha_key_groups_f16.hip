// F16 instantiations of the key layout's row-group kernels.
#include "fmha_kernel.h"
#include "fmha_registry.h"

namespace fgw_mha {
FGW_MHA_FOR_KEY_GROUPS(FGW_MHA_INSTANTIATE_KEY_GROUPS, false)
}  // namespace fgw_mha
