// The mixed pair kernels, compiled in a file of their own (pmx_pair.hip) with
// a compiler option that the rest does not take: every form that pmx.hip
// launches, declared here and instantiated there.
#pragma once

#include "pmx_batch.h"

namespace pmx {

// X(COUL, LJSW, CSW, BIGLJ) for the cases of run_pair_phase
#define PMX_PAIR_CASES(X)                    \
  X(COUL_PME, SW_C2, SW_CUTOFF, false)       \
  X(COUL_PME, SW_NONE, SW_ANY, false)        \
  X(COUL_PME, SW_ANY, SW_ANY, false)         \
  X(COUL_PME, SW_ANY, SW_ANY, true)          \
  X(COUL_CUTOFF, SW_C2, SW_C1, false)        \
  X(COUL_CUTOFF, SW_NONE, SW_ANY, false)     \
  X(COUL_CUTOFF, SW_ANY, SW_ANY, false)      \
  X(COUL_CUTOFF, SW_ANY, SW_ANY, true)       \
  X(COUL_NONE, SW_ANY, SW_ANY, false)        \
  X(COUL_NONE, SW_ANY, SW_ANY, true)
// and for those of batch_case
#define PMX_BATCH_PAIR_CASES(X)              \
  X(COUL_PME, SW_C2, SW_CUTOFF, false)       \
  X(COUL_PME, SW_NONE, SW_ANY, false)        \
  X(COUL_PME, SW_ANY, SW_ANY, false)         \
  X(COUL_PME, SW_ANY, SW_ANY, true)

#define PMX_PAIR_KERNEL(EXT, C, LJ, CS, BIG, MODE)                                                                   \
  EXT template __global__ void k_pair<true, C, LJ, CS, BIG, MODE>(                                                   \
      PairParams, int, const int2 *__restrict__, const int *__restrict__, const int *__restrict__,                   \
      int *__restrict__, const int4 *__restrict__, int4 *, int, const unsigned short *__restrict__,                  \
      const float4 *__restrict__, const float4 *__restrict__, const int *__restrict__, const int *__restrict__,      \
      const double *__restrict__, const float4 *__restrict__, unsigned long long *__restrict__, PairOut);
#define PMX_BATCH_PAIR_KERNEL(EXT, C, LJ, CS, BIG)                                                              \
  EXT template __global__ void k_batch<OpPair<true, C, LJ, CS, BIG>>(                                           \
      const OpPair<true, C, LJ, CS, BIG>::Args *__restrict__, const int *__restrict__, const int *__restrict__, \
      BatchStep);

#define PMX_X(C, LJ, CS, BIG)                          \
  PMX_PAIR_KERNEL(extern, C, LJ, CS, BIG, kPairPlain)  \
  PMX_PAIR_KERNEL(extern, C, LJ, CS, BIG, kPairPrune)  \
  PMX_PAIR_KERNEL(extern, C, LJ, CS, BIG, kPairStats)
PMX_PAIR_CASES(PMX_X)
#undef PMX_X
#define PMX_X(C, LJ, CS, BIG) PMX_BATCH_PAIR_KERNEL(extern, C, LJ, CS, BIG)
PMX_BATCH_PAIR_CASES(PMX_X)
#undef PMX_X

}  // namespace pmx
