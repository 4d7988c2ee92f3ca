// Instantiates the mixed pair kernels (see pmx_pair.h).  Compiled with
// -structurizecfg-skip-uniform-regions: the branches of the pair loop on list
// bits and ballots are uniform, and turning them into the linear form that
// divergent branches need cost three register copies per cluster pair and 23
// VGPRs (95 -> 72): 67.0 -> 60.5 us a launch at 26,000 atoms, 1.18 -> 1.07 ms
// at 1,000,000.
#include <hip/hip_runtime.h>

#include "pmx_pair.h"

namespace pmx {

#define PMX_X(C, LJ, CS, BIG) PMX_PAIR_MODES(, true, C, LJ, CS, BIG)
PMX_PAIR_CASES(PMX_X)
#undef PMX_X
#define PMX_X(C, LJ, CS, BIG) PMX_BATCH_PAIR_KERNEL(, true, C, LJ, CS, BIG)
PMX_BATCH_PAIR_CASES(PMX_X)
#undef PMX_X

}  // namespace pmx
