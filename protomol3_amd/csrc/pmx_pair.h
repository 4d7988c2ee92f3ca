// The pair kernels, compiled in files of their own (pmx_pair.hip: mixed,
// pmx_pair64.hip: FP64) with a compiler option that the rest does not take:
// every form that pmx.hip launches, declared here and instantiated there.
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

#define PMX_PAIR_KERNEL(EXT, M, C, LJ, CS, BIG, MODE)                                                             \
  EXT template __global__ void k_pair<M, C, LJ, CS, BIG, MODE>(                                                   \
      PairParams, int, const int2 *__restrict__, const int *__restrict__, const int *__restrict__,                \
      int *__restrict__, const int4 *__restrict__, int4 *, int, const unsigned short *__restrict__,               \
      const Real4<PairReal<M>>::type *__restrict__, const float4 *__restrict__, const int *__restrict__,          \
      const int *__restrict__, const double *__restrict__, const Real4<PairReal<M>>::type *__restrict__,          \
      AccT<M>::type *__restrict__, PairOut);
#define PMX_BATCH_PAIR_KERNEL(EXT, M, C, LJ, CS, BIG)                                                        \
  EXT template __global__ void k_batch<OpPair<M, C, LJ, CS, BIG>>(                                           \
      const OpPair<M, C, LJ, CS, BIG>::Args *__restrict__, const int *__restrict__, const int *__restrict__, \
      BatchStep);
// every kernel of one case and form
#define PMX_PAIR_MODES(EXT, M, C, LJ, CS, BIG)           \
  PMX_PAIR_KERNEL(EXT, M, C, LJ, CS, BIG, kPairPlain)    \
  PMX_PAIR_KERNEL(EXT, M, C, LJ, CS, BIG, kPairPrune)    \
  PMX_PAIR_KERNEL(EXT, M, C, LJ, CS, BIG, kPairStats)

template <bool MIXED>
using PairReal = typename std::conditional<MIXED, float, double>::type;

#define PMX_X(C, LJ, CS, BIG)                 \
  PMX_PAIR_MODES(extern, true, C, LJ, CS, BIG) \
  PMX_PAIR_MODES(extern, false, C, LJ, CS, BIG)
PMX_PAIR_CASES(PMX_X)
#undef PMX_X
#define PMX_X(C, LJ, CS, BIG)                        \
  PMX_BATCH_PAIR_KERNEL(extern, true, C, LJ, CS, BIG) \
  PMX_BATCH_PAIR_KERNEL(extern, false, C, LJ, CS, BIG)
PMX_BATCH_PAIR_CASES(PMX_X)
#undef PMX_X

}  // namespace pmx
