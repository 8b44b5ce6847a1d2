// bwd_pair_kernel (fhog_bwd_pair.h) for rows of 512 bytes (2-byte D = 256, fp32
// D = 128), in the compiler's default scheduling: for instruction-level
// parallelism it spills in the loop (first backward at B4 N2048 H16 D256 causal
// 942 against 691 us).
#include "fhog_bwd_pair.h"

namespace fhog {

#define FHOG_INST(T, D, C) template hipError_t launch_bwd_pair<T, D, C>(const BwdParams<T>&, hipStream_t);
FHOG_INST(__bf16, 256, true)
FHOG_INST(__bf16, 256, false)
FHOG_INST(_Float16, 256, true)
FHOG_INST(_Float16, 256, false)
FHOG_INST(float, 128, true)
FHOG_INST(float, 128, false)
#undef FHOG_INST

}  // namespace fhog
