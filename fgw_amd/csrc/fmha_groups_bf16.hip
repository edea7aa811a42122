// BF16 instantiations of the key and query layouts' row-group kernels, of
// the key layout's with non-temporal loads and of the query layout's eight-wave one.
#include "fmha_kernel.h"
#include "fmha_registry.h"

namespace fgw_mha {
FGW_MHA_FOR_GROUPS(FGW_MHA_INSTANTIATE_GROUPS, true)
FGW_MHA_FOR_STREAM(FGW_MHA_INSTANTIATE_STREAM, true)
FGW_MHA_INSTANTIATE_DUAL(true)
}  // namespace fgw_mha
