// Instantiates the FP64 pair kernels (see pmx_pair.h), with the option of the
// mixed ones: 118 registers fewer spilled in the PME form.
#include <hip/hip_runtime.h>

#include "pmx_pair.h"

namespace pmx {

#define PMX_X(C, LJ, CS, BIG) PMX_PAIR_MODES(, false, C, LJ, CS, BIG)
PMX_PAIR_CASES(PMX_X)
#undef PMX_X
#define PMX_X(C, LJ, CS, BIG) PMX_BATCH_PAIR_KERNEL(, false, C, LJ, CS, BIG)
PMX_BATCH_PAIR_CASES(PMX_X)
#undef PMX_X

}  // namespace pmx
