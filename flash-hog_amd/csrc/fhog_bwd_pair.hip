// bwd_pair_kernel (fhog_bwd_pair.h) for rows of up to 256 bytes, scheduled for
// instruction-level parallelism (build.py).
#include "fhog_bwd_pair.h"

namespace fhog {

#define FHOG_INST(T, D, C) template hipError_t launch_bwd_pair<T, D, C>(const BwdParams<T>&, hipStream_t);
FHOG_INST(__bf16, 64, true)
FHOG_INST(__bf16, 64, false)
FHOG_INST(__bf16, 128, true)
FHOG_INST(__bf16, 128, false)
FHOG_INST(_Float16, 64, true)
FHOG_INST(_Float16, 64, false)
FHOG_INST(_Float16, 128, true)
FHOG_INST(_Float16, 128, false)
FHOG_INST(float, 64, true)
FHOG_INST(float, 64, false)
#undef FHOG_INST

}  // namespace fhog
