// Batched launches: one launch runs a kernel over the blocks of many systems.
//
// A batch is a set of systems of one context that share the kernel case (form,
// force kinds, PME order).  Each kernel of the MD step (and of a force pass)
// gets, per batch, a
// table with one argument block per system in device memory, the first block
// of every system (first[s], first[nsys] = all blocks) and the system of every
// block (b2s).  Block b then does the work of block b - first[s] of system
// b2s[b] in a launch of first[s + 1] - first[s] blocks, through the same
// kernel body as the single-system launch, so a system's results do not depend
// on the batch it runs in.
//
// The list rebuild runs on the device: per step a small kernel marks the
// systems whose atoms moved more than half the skin since their last build
// (the displacement record of the step's kick-drift), and the blocks of the
// rebuild kernels of the other systems return at once.
#pragma once

#include "pmx_kernels.h"

namespace pmx {

// Per-launch values shared by the systems of a batched step.
struct BatchStep {
  int k;                          // step within the chunk
  int opening;                    // 1: step 0 of the chunk opens the run (half kick)
  const unsigned char *need;      // per system: the list is rebuilt at this step
};

template <class Op>
__global__ void __launch_bounds__(Op::kBlock, Op::kMinBlocks) k_batch(const typename Op::Args *__restrict__ tab,
                                                                      const int *__restrict__ b2s,
                                                                      const int *__restrict__ first, BatchStep st) {
  // the blocks of one XCD take a contiguous range of the table (whole
  // systems share its L2)
  const int b = xcd_block(blockIdx.x, gridDim.x);
  const int s = __builtin_amdgcn_readfirstlane(b2s[b]);
  if (Op::kGated && !st.need[s]) return;
  const int f = first[s];
  Op::run(tab[s], b - f, first[s + 1] - f, st);
}

// The kick of step k of a chunk for a system whose kick parameters are `base`
// (half0 relative to the chunk's first step in *base.step_dev): step 0 of an
// opening chunk gets one half kick, every other step the previous step's
// closing and its own opening half kick.
__device__ inline Kick batch_kick(const Kick &base, double h, int k, bool opening) {
  Kick kk = base;
  const bool half = opening && k == 0;
  kk.h_kick = (half ? 0.5 : 1.0) * h;
  kk.nhalf = half ? 1 : 2;
  kk.half0 = half ? 2ull * (unsigned long long)k : 2ull * (unsigned long long)k - 1ull;
  return kk;
}

// ---- list rebuild (gated) ----

struct OpBin {
  struct Args {
    int n;
    const double *xorig;
    BinParams p;
    uint32_t *key, *hist;
    double *xwrap;
    int *refcell;
  };
  static constexpr int kBlock = 256, kMinBlocks = 1;
  static constexpr bool kGated = true;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    bin_body(bid, nbk, a.n, a.xorig, a.p, a.key, a.xwrap, a.refcell, a.hist, nullptr);
  }
};

struct OpScanColumns {
  struct Args {
    uint32_t *hist, *start, *cursor;
    int nbins, ncols, nzb, n, nsuper;
    int2 *sc_info;
    int *sc_col, *colsc;
  };
  static constexpr int kBlock = kScanBlock, kMinBlocks = 1;
  static constexpr bool kGated = true;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    scan_columns_body(a.hist, a.nbins, a.start, a.cursor, a.ncols, a.nzb, a.n, a.nsuper, a.sc_info, a.sc_col,
                      a.colsc);
  }
};

struct OpScatter {
  struct Args {
    int n;
    const uint32_t *key;
    uint32_t *cursor;
    int *perm;
  };
  static constexpr int kBlock = 256, kMinBlocks = 1;
  static constexpr bool kGated = true;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    scatter_body(bid, nbk, a.n, a.key, a.cursor, a.perm);
  }
};

template <class R>
struct OpSplitFill {
  struct Args {
    int nsuper;
    const int2 *sc_info;
    SortedBins sb;
    const double *xwrap, *q;
    int *permp, *slot;
    const int *type;
    typename Real4<R>::type *xs;
    double4 *xs64;
    int *ts;
    const double *xorig;
    const double *minv;
    double4 *xbuild;
    float4 *sorg, *ctr, *half, *sctr, *shalf;
    int *nmaskwork;
    double qpair;
    PmeParams pme;
    PmeSlots<R> rec;
  };
  static constexpr int kBlock = 256, kMinBlocks = 1;
  static constexpr bool kGated = true;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    split_fill_body<R>(bid, nbk, a.nsuper, a.sc_info, a.sb, a.xwrap, a.permp, a.slot, a.q, a.type, a.xs, a.xs64,
                       a.ts, a.xorig, a.minv, a.xbuild, a.sorg, a.ctr, a.half, a.sctr, a.shalf, a.nmaskwork, a.qpair, a.pme,
                       a.rec);
  }
};

struct OpBuildList {
  struct Args {
    ListParams q;
    const int *sc_col, *colsc;
    const float4 *sctr, *shalf, *ctr, *half;
    int4 *entries;
    int *count, *ecost, *cost_out;
    MaskArgs ma;
    int *nmaskwork, *overflow;
  };
  static constexpr int kBlock = kListBlock, kMinBlocks = 1;
  static constexpr bool kGated = true;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    build_list_body(bid, nbk, a.q, a.sc_col, a.colsc, a.sctr, a.shalf, a.ctr, a.half, a.entries, a.count, a.ecost,
                    a.cost_out, a.ma, a.nmaskwork, a.overflow);
  }
};

struct OpRuns {
  struct Args {
    int nsuper, cap;
    const int *count, *cost, *ecost;
    int2 *runs;
    int *ntiles;
  };
  static constexpr int kBlock = kRunsBlock, kMinBlocks = 1;
  static constexpr bool kGated = true;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    runs_body(bid, nbk, a.nsuper, a.count, a.cost, a.ecost, a.cap, kCutBatch, a.runs, a.ntiles);
  }
};

// ---- force pass and integration ----

template <class R>
struct OpKickDrift {
  struct Args {
    int n;
    Kick kick;
    double h;
    const int *perm;
    const double *fout;
    const double4 *xbuild;
    double *v, *x;
    typename Real4<R>::type *xs;
    const double4 *xs64;
    const float4 *sorg;
    unsigned *dmax;  // displacement record of the chunk, one word per step
    PmeParams pme;
    PmeSlots<R> rec;
  };
  static constexpr int kBlock = 256, kMinBlocks = 1;
  static constexpr bool kGated = false;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &st) {
    kick_drift_body<R>(bid, nbk, a.n, batch_kick(a.kick, a.h, st.k, st.opening), a.h, a.perm, a.fout, a.v, a.x,
                       a.xbuild, a.xs, a.xs64, a.sorg, a.dmax + st.k, a.pme, a.rec);
  }
};

template <bool MIXED, int P>
struct OpPmeSpreadZ {
  using T = typename std::conditional<MIXED, float, double>::type;
  struct Args {
    PmeParams p;
    FftPlan pl;
    const int2 *tcol;
    const int *colsc;
    const typename Real4<T>::type *pmw;
    const int2 *pmb;
    const Cx<T> *tw;
    Cx<T> *spec;
  };
  static constexpr int kBlock = kPmeBlock, kMinBlocks = kPmeWaves<T>;
  static constexpr bool kGated = false;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    pme_spread_z_body<MIXED, P>(bid, nbk, a.p, a.pl, a.tcol, a.colsc, a.pmw, a.pmb, a.tw, a.spec);
  }
};

template <bool MIXED, int P>
struct OpPmeSpreadZLong : OpPmeSpreadZ<MIXED, P> {
  using typename OpPmeSpreadZ<MIXED, P>::Args;
  static constexpr int kMinBlocks = 2;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    pme_spread_z_body<MIXED, P, true>(bid, nbk, a.p, a.pl, a.tcol, a.colsc, a.pmw, a.pmb, a.tw, a.spec);
  }
};

template <bool MIXED, int COUL, int LJSW, int CSW, bool BIGLJ>
struct OpPair {
  using R4 = typename Real4<typename std::conditional<MIXED, float, double>::type>::type;
  struct Args {
    PairParams pp;
    const int2 *runs;
    const int *ntiles, *count;
    int *tilectr;
    int4 *entries;
    int cap;
    const unsigned short *masks;
    const R4 *xs;
    const float4 *sorg;
    const int *ts, *perm;
    const double *ljtab;
    const R4 *ljt;
    typename AccT<MIXED>::type *facc;
    PairOut out;
  };
  static constexpr int kBlock = kPairBlock, kMinBlocks = MIXED ? 4 : 3;
  static constexpr bool kGated = false;
  // the runs in contiguous shares per wave (schedule 0)
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    pair_body<MIXED, COUL, LJSW, CSW, BIGLJ, kPairPlain>(bid, nbk, a.pp, 0, a.runs, a.ntiles, a.count, a.tilectr,
                                                         a.entries, a.entries, a.cap, a.masks, a.xs, a.sorg, a.ts,
                                                         a.perm, a.ljtab, a.ljt, a.facc, a.out);
  }
};

template <class T>
struct OpFftY {
  struct Args {
    PmeParams p;
    FftPlan pl;
    int llog;
    bool inverse;
    const Cx<T> *tw;
    Cx<T> *spec;
  };
  static constexpr int kBlock = kPmeBlock, kMinBlocks = kPmeWaves<T>;
  static constexpr bool kGated = false;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    fft_y_body<T>(bid, nbk, a.p, a.pl, a.llog, a.inverse, a.tw, a.spec);
  }
};

template <class T>
struct OpFftYLong : OpFftY<T> {
  using typename OpFftY<T>::Args;
  static constexpr int kMinBlocks = 2;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    fft_y_body<T, true>(bid, nbk, a.p, a.pl, a.llog, a.inverse, a.tw, a.spec);
  }
};

template <class T>
struct OpFftXConv {
  struct Args {
    PmeParams p;
    FftPlan pl;
    int llog, threads;
    const Cx<T> *tw;
    const T *theta;
    Cx<T> *spec;
    double *epart;
  };
  static constexpr int kBlock = kPmeBlock, kMinBlocks = kPmeWaves<T>;
  static constexpr bool kGated = false;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    fft_x_conv_body<T>(bid, nbk, a.p, a.pl, a.llog, a.threads, a.tw, a.theta, a.spec, a.epart);
  }
};

template <class T>
struct OpFftXConvLong : OpFftXConv<T> {
  using typename OpFftXConv<T>::Args;
  static constexpr int kMinBlocks = 2;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    fft_x_conv_body<T, true>(bid, nbk, a.p, a.pl, a.llog, a.threads, a.tw, a.theta, a.spec, a.epart);
  }
};

template <class T>
struct OpFftPlane {
  struct Args {
    PmeParams p;
    FftPlan ply, plx;
    int threads;
    const Cx<T> *twy, *twx;
    const T *theta;
    Cx<T> *spec;
    double *epart;
  };
  static constexpr int kBlock = kPmeBlock, kMinBlocks = kPmeWaves<T>;
  static constexpr bool kGated = false;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    fft_plane_conv_body<T>(bid, nbk, a.p, a.ply, a.plx, a.threads, a.twy, a.twx, a.theta, a.spec, a.epart);
  }
};

template <bool MIXED, int P>
struct OpPmeZGather {
  using T = typename std::conditional<MIXED, float, double>::type;
  struct Args {
    PmeParams p;
    FftPlan pl;
    const int2 *tcol;
    const int *colsc;
    const typename Real4<T>::type *pmw;
    const int2 *pmb;
    const Cx<T> *tw, *spec;
    typename AccT<MIXED>::type *facc;
  };
  static constexpr int kBlock = kPmeBlock, kMinBlocks = kPmeWaves<T>;
  static constexpr bool kGated = false;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    pme_z_gather_body<MIXED, P>(bid, nbk, a.p, a.pl, a.tcol, a.colsc, a.pmw, a.pmb, a.tw, a.spec, a.facc);
  }
};

template <bool MIXED, int P>
struct OpPmeZGatherLong : OpPmeZGather<MIXED, P> {
  using typename OpPmeZGather<MIXED, P>::Args;
  static constexpr int kMinBlocks = 2;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    pme_z_gather_body<MIXED, P, true>(bid, nbk, a.p, a.pl, a.tcol, a.colsc, a.pmw, a.pmb, a.tw, a.spec, a.facc);
  }
};

template <bool MIXED, int COUL, int LJSW, int CSW>
struct OpFixups {
  using Args = FixupArgs<MIXED>;
  static constexpr int kBlock = 256, kMinBlocks = 1;
  static constexpr bool kGated = false;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    fixups_body<MIXED, COUL, LJSW, CSW>(bid, nbk, a);
  }
};

// unsort of step k's forces, kick and drift of step k + 1
template <bool MIXED, class R>
struct OpUnsortKickDrift {
  struct Args {
    int n;
    Kick kick;
    double h;
    const int *perm;
    typename AccT<MIXED>::type *facc;
    int *tilectr, *nborder;
    const double4 *xbuild;
    double *v, *x;
    typename Real4<R>::type *xs;
    const double4 *xs64;
    const float4 *sorg;
    unsigned *dmax;
    PmeParams pme;
    PmeSlots<R> rec;
  };
  static constexpr int kBlock = 256, kMinBlocks = 1;
  static constexpr bool kGated = false;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &st) {
    unsort_kick_drift_body<MIXED, R>(bid, nbk, a.n, batch_kick(a.kick, a.h, st.k + 1, false), a.h, a.perm, a.facc,
                                     a.tilectr, a.nborder, a.v, a.x, a.xbuild, a.xs, a.xs64, a.sorg,
                                     a.dmax + st.k + 1, a.pme, a.rec);
  }
};

template <bool MIXED>
struct OpUnsortForces {
  struct Args {
    int n;
    const int *slot;
    typename AccT<MIXED>::type *facc;
    double *fout;
    int *tilectr, *nborder;
  };
  static constexpr int kBlock = 256, kMinBlocks = 1;
  static constexpr bool kGated = false;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    unsort_forces_body<MIXED>(bid, nbk, a.n, a.slot, a.facc, a.fout, a.tilectr, a.nborder);
  }
};

// The end of a force pass with energies, one more block a system than the forces take.
template <bool MIXED>
struct OpUnsortEnergy {
  struct Args {
    int n;
    const int *slot;
    typename AccT<MIXED>::type *facc;
    double *fout;
    int *tilectr, *nborder;
    EnergyArgs e;
  };
  static constexpr int kBlock = kEndBlock, kMinBlocks = 1;
  static constexpr bool kGated = false;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    unsort_energy_body<MIXED>(bid, a.n, a.slot, a.facc, a.fout, a.tilectr, a.nborder, a.e);
  }
};

struct OpOut {
  using Args = OutArgs;
  static constexpr int kBlock = 256, kMinBlocks = 1;
  static constexpr bool kGated = false;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) { out_body(bid, nbk, a); }
};

// backups for a restore, cleared overflow flags and displacement record
struct OpChunkBegin {
  struct Args {
    long long m3;
    const double *x, *v, *f;
    double *xbak, *vbak, *fbak;
    int *overflow;
    unsigned *dmax;
    int nrec;
  };
  static constexpr int kBlock = 256, kMinBlocks = 1;
  static constexpr bool kGated = false;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &) {
    chunk_begin_body(bid, nbk, a.m3, a.x, a.v, a.f, a.xbak, a.vbak, a.fbak, a.overflow, a.dmax, a.nrec);
  }
};

// the closing half kick after the chunk's last step (st.k = its length)
struct OpHalfKick {
  struct Args {
    int n;
    Kick kick;
    double h;
    const double *fout, *minv;
    double *v;
  };
  static constexpr int kBlock = 256, kMinBlocks = 1;
  static constexpr bool kGated = false;
  __device__ static void run(const Args &a, int bid, int nbk, const BatchStep &st) {
    Kick kk = a.kick;
    kk.h_kick = 0.5 * a.h;
    kk.nhalf = 1;
    kk.half0 = 2ull * (unsigned long long)st.k - 1ull;
    half_kick_body(bid, nbk, a.n, kk, a.fout, a.minv, a.v);
  }
};

// ---- per-system bookkeeping of a batch ----

struct BatchSys {
  const unsigned *dmax;          // the chunk's displacement record
  float lim2;                    // (skin / 2)^2
  int force;                     // rebuild at step 0 of the chunk whatever the displacement
  unsigned long long *step_dev;  // first step of the chunk
  int *overflow;
  long long *rebuilds;           // device count of the builds in the batch
};

// need[s]: system s rebuilds its list at step k (first thread of each
// system); the count of builds goes up.
static __global__ void k_batch_need(int nsys, const BatchSys *__restrict__ bs, int k, unsigned char *__restrict__ need) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nsys) return;
  const BatchSys b = bs[s];
  const float d = __uint_as_float(b.dmax[k]);
  const bool r = (k == 0 && b.force) || d > b.lim2;
  need[s] = r ? 1 : 0;
  if (r) ++*b.rebuilds;
}

// The chunk's first step index of every system (base[s]) and the overflow
// flags of the last chunk gathered into one array for the host.
static __global__ void k_batch_steps(int nsys, const BatchSys *__restrict__ bs, const unsigned long long *__restrict__ base) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < nsys) *bs[s].step_dev = base[s];
}

static __global__ void k_batch_clear(int nsys, const BatchSys *__restrict__ bs) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < nsys) bs[s].overflow[0] = bs[s].overflow[1] = 0;
}

static __global__ void k_batch_flags(int nsys, const BatchSys *__restrict__ bs, int *__restrict__ out) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s < nsys) out[s] = *bs[s].overflow;
}

}  // namespace pmx
