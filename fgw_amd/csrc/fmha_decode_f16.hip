// F16 instantiations of the single-token decode kernel.
#include "fmha_decode.h"
#include "fmha_registry.h"

namespace fgw_mha {
FGW_MHA_FOR_DECODE(FGW_MHA_INSTANTIATE_DECODE, false)
}  // namespace fgw_mha
