// pmx: C-ABI implementation (include/pmx.h) -- host orchestration of the
// gfx950 kernels in pmx_kernels.h.  One HIP stream per context; all device
// state of a system stays resident between calls.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <thread>
#include <tuple>
#include <type_traits>
#include <vector>

#include "../../include/pmx.h"
#include "pmx_kernels.h"
#include "pmx_pair.h"

using namespace pmx;

struct pmx_ctx {
  int device = 0;
  int cus = 256;  // compute units of the device
  void *scratch = nullptr;  // device address of this device's copy of `scratch` (no-allocation force pass)
  hipStream_t stream = nullptr;   // main stream: sort, list, pair kernel, boundary pairs, finalize
  hipStream_t stream2 = nullptr;  // PME, exclusion correction and bonded terms, concurrent with the pair kernel
  // batched launches: pinned host staging (grown as needed) and the fork/join
  // events, kept from one batch to the next
  void *batch_host = nullptr;
  size_t batch_host_bytes = 0;
  hipEvent_t batch_fork = nullptr, batch_join = nullptr;
  std::string err;
};

// Scratch of pmx_sys_compute_noalloc: the per-pass partial results, counters
// and records of a force pass (per-tile energies and pair statistics, the
// boundary-pair records and their counters) live here instead of in the
// system's own buffers.  Each device holds one copy for the life of the
// process, shared by every call on that device.  In host code the name is a
// stand-in, not a device address: host code uses only the address
// hipGetSymbolAddress returns for the current device (pmx_ctx::scratch).
constexpr size_t kScratchBytes = 32ull << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

// Device address of `scratch` per device, looked up once per device (with
// that device current) by the first pmx_ctx_create on it.
constexpr int kMaxDevices = 64;
void *g_scratch_addr[kMaxDevices] = {};

struct DevBuf {
  void *p = nullptr;
  size_t bytes = 0;
  bool listed = false;  // registered in Sys::all (freed by pmx_sys_destroy)
};

// A pinned host block (host_get, host_put).
struct HostBuf {
  void *p = nullptr;
  size_t bytes = 0;
};

// Timed stages: sort (+ integrate), list (+ accumulator zeroing), pair,
// spread (with the z transform, and with the exclusion correction and bonded
// terms where these go with it; only where it runs on the main stream, by
// default below kSpread2From atoms), fft (+ convolution, after the spread
// where that runs on the second stream), gather (with the inverse z transform), fixups (exclusion
// correction and bonded terms, where they run on the second stream), finalize
// (boundary pairs, with them those terms where they follow the pair kernel, and
// the force unsort).  Events: 0 start, 1 sorted,
// 2 list built and accumulators zeroed, 4 spread done = fork (main stream), 3
// pair done (main stream), 5 fft, 6 gather, 7 correction + bonded done
// (second stream), 8 end.  The second stream's stages run beside the pair
// kernel.
constexpr int kStages = 8;
constexpr int kStageEv[kStages][2] = {{0, 1}, {1, 2}, {4, 3}, {2, 4}, {4, 5}, {5, 6}, {6, 7}, {7, 8}};
static_assert(kStages == PMX_STAGES, "stage count of the C ABI");

// Results of a force pass, in device memory (Sys::eout).
struct PassResults {
  double e[4];  // Coulomb, LJ, reciprocal, correction
  long long np[1];
  unsigned long long hash[1];
  int overflow[2];
};

struct Sys {
  pmx_ctx *ctx = nullptr;
  pmx_sys_desc d{};
  bool mixed = false;
  int n = 0, npad = 0, ncl = 0, nsuper = 0, ncols = 0;  // nsuper: upper bound (slots = 64 nsuper)
  // host copies
  std::vector<double> q, lj;
  std::vector<float> lj32;         // FP32 copy of lj (source of ljt32)
  std::vector<int> type;
  std::vector<int4> etab;          // de-duplicated exclusion table a1 a2 cls
  std::vector<int> eptr;           // CSR of partners per atom (orig index)
  std::vector<int2> elist;
  double alpha = 0, self_e = 0, charged_e = 0;
  double qpair = 1.0;              // charge factor of the pair pass (0: PME real term off)
  Box box{};
  BinParams bin{};
  PairParams pp{};
  ListParams lp{};
  PmeParams pme{}, pme_g{};  // the same but for the tiles: spread, gather
  FftPlan plx{}, ply{}, plz{};
  bool pme_on = false;
  int cap = 0, maxmaskwork = 0, ntiles_cap = 0;
  // launch shapes the autotuner may change (pmx_sys_set_tuning)
  int tune_fft_lines = 16;     // most lines per FFT block
  int tune_pair_blocks = 0;    // pair-kernel blocks per CU (0: as many as fit)
  int tune_schedule = 0;       // 0: runs round robin over the waves; 1: later runs from a counter
  int tune_spread_stream2 = 0; // 1: the PME spread runs on the second stream, beside the pair kernel
  int tune_fixup_main = 0;     // 1: exclusion correction and bonded terms on the main stream after the pair kernel
                               // (default 1 below kFixupMainBelow atoms)
  int tune_fft_planes = 1;     // 1: y, x and convolution passes in one launch per plane on small planes
  bool fft_plane = false;      // the plane launch is in use
  int border_blocks = 4;       // blocks of the boundary-pair pass
  int tune_prune = 1;          // 1: the first pair pass after a list build prunes the list's cluster pairs
  bool prune_pending = false;  // a list was built and its first pair pass has not run
  int pair_grid = 0;           // blocks of the pair-kernel launch
  RunCut cut = kCutBeside;     // how the list is cut into runs
  long long nbins = 0;
  int nscanblocks = 0;
  int recip_blocks = 0, term_blocks = 0;  // blocks of the x pass and of the atoms' terms
  int xlog = 0, ylog = 0;              // lines of a block of the x and y passes (log2)
  size_t lds_z = 0, lds_g = 0, lds_y = 0, lds_x = 0, lds_p = 0;  // dynamic LDS of the PME launches
  int thr_z = 256, thr_g = 256, thr_y = 256, thr_x = 256, thr_p = 256;  // and their block sizes
  int thr_gb = 256, thr_pb = 256;  // gather and plane in batched launches
  // device buffers
  std::vector<DevBuf *> all;
  DevBuf xorig, xwrap, q_d, type_d, key, hist, start, cursor, scansum, perm, permp, slot, refcell, xs, xs64, ts,
      sc_info, sc_col, colsc, sctr, shalf, sorg, ctr, half, entries, count, ecost, lcost, runs, nmaskwork, masks, overflow, ntiles, tilectr, ljtab, ljt32, facc, fout,
      pair_e, npairs, hash, eptr_d, elist_d, cptr_d, clist_d, corr_e, recip_e, eout, np_out, hash_out, pmw, pmb, tcol, spec, theta, twx, twy, twz, border, nborder, border_acc;
  // (overflow, np_out and hash_out are parts of eout: one copy brings a pass's results)
  int maxborder = 65536;
  // results
  long long last_np = 0;
  unsigned long long last_hash = 0;
  float stage_ms[kStages] = {0};
  hipEvent_t *ev = nullptr;                    // event set of the current timed call
  hipEvent_t fork_ev = nullptr, join_ev = nullptr;  // main stream <-> second stream per force pass
  std::vector<std::vector<hipEvent_t>> evsets;  // one set of kStages + 1 per timed call since timing_begin
  size_t evused = 0;
  bool timing_active = false;                   // MD steps record events (timing_begin .. timing_end)
  bool have_positions = false;
  bool cached = false;
  bool list_valid = false;             // entries, counts and work of a built list are in place
  enum { kInPartials, kInResults, kInHeld } energies_at = kInPartials;  // where the last pass's energies are:
                                       // its partials, eout, md.held (the partials may be gone)
  bool acc_clean = false;              // force accumulators and pass counters are zero
  bool dry = false;                    // size only: allocations are counted, nothing runs
  unsigned long long dry_bytes = 0;
  // pinned staging of this system's copies to and from the host, in chunks
  // beyond kStageChunks x kStageChunk bytes (stage_ev: a chunk's copy is done)
  HostBuf stage;
  bool staged = false;  // the stage holds the last pass's results and forces (batched passes); cleared by
                        // whatever may write new ones
  bool recorded = false;  // a pass was recorded into a graph, whose replays the host does not see: never staged
  hipEvent_t stage_ev[4] = {nullptr, nullptr, nullptr, nullptr};
  // device-resident MD state
  struct Md {
    bool on = false;
    int nb = 0, na = 0;
    double h = 0, skin = 0;
    DevBuf mptr, bonds, bpar, angles, apar, minv, v, xbuild, xbak, vbak, fbak, dmax, bond_e, ke_e, held;
    int chunk = 16;
    long long steps = 0, rebuilds = 0, rollbacks = 0;
    bool forces_valid = false;
    int integrator = PMX_MD_LEAPFROG;
    double vdt = 1, fdt = 0, ndt = 0, fc = 0;  // Langevin half-kick constants
    unsigned long long seed = 0;
    // two chunks in flight: backups, displacement records and their pinned
    // host copies (per slot: kMaxChunk displacements + the overflow flag)
    unsigned *host = nullptr;
    hipEvent_t chunk_ev[2] = {nullptr, nullptr};
    // chunks captured as HIP graphs, keyed by (steps, first, slot); the
    // chunk's first step index is written to step_dev before each launch
    bool graphs = false;
    DevBuf step_dev;
    std::map<long long, hipGraphExec_t> gexec;
  } md;
};
constexpr int kMaxChunk = 128;
constexpr int kFixupMainBelow = 100000;  // atoms; default of PMX_TUNE_FIXUP_STREAM
// Atoms from which the charge spread runs beside the pair kernel by default
// (PMX_TUNE_SPREAD_STREAM): below, the PME chain is the longer branch.
constexpr int kSpread2From = 10000;
constexpr double kInvTimeFactor = 0.02045482828087295;  // protomol/base/PMConstants.cpp:54
constexpr double kBoltzmann = 0.001987191;              // protomol/base/PMConstants.cpp:70

int fail(pmx_ctx *c, int code, const std::string &m) {
  if (c) c->err = m;
  return code;
}

#define HIPCHK(expr)                                                                        \
  do {                                                                                      \
    hipError_t _e = (expr);                                                                 \
    if (_e != hipSuccess) return fail(s->ctx, PMX_ERR_HIP, std::string(#expr ": ") + hipGetErrorString(_e)); \
  } while (0)

// Runtime calls that may synchronize the device (allocation, free, pinned
// allocation, event and stream creation, synchronous copies) can invalidate a
// stream capture that another thread has in progress, so they and the
// captures themselves are serialized on this lock.
std::recursive_mutex g_rt_mu;
using RtLock = std::lock_guard<std::recursive_mutex>;

// Device block cache.  Systems come and go (a request loop builds one per
// request), so released device blocks are kept per device in size classes
// (powers of 2 split in quarters above 4 KiB) and handed to the next request
// of the same class instead of going back to hipFree / hipMalloc.  A block is
// released only after the streams that used it are synchronized.  When
// hipMalloc fails, the cached blocks of that device are freed and the
// allocation is tried once more.  Guarded by g_rt_mu.
size_t size_class(size_t bytes) {
  if (bytes <= 4096) return bytes <= 256 ? 256 : (size_t)1 << (64 - __builtin_clzll(bytes - 1));
  const int e = 63 - __builtin_clzll(bytes);  // 2^e <= bytes < 2^(e+1)
  const size_t q = (size_t)1 << (e - 2);
  return (bytes + q - 1) / q * q;
}
std::map<int, std::multimap<size_t, void *>> g_block_cache;
size_t g_cached_bytes = 0;
constexpr size_t kBlockCacheMax = 16ull << 30;  // cached bytes kept per process, at most

void *block_get(int device, size_t cls) {
  auto &m = g_block_cache[device];
  auto it = m.find(cls);
  if (it != m.end()) {
    void *p = it->second;
    m.erase(it);
    g_cached_bytes -= cls;
    return p;
  }
  void *p = nullptr;
  if (hipMalloc(&p, cls) == hipSuccess) return p;
  for (auto &kv : m) hipFree(kv.second), g_cached_bytes -= kv.first;
  m.clear();
  p = nullptr;
  return hipMalloc(&p, cls) == hipSuccess ? p : nullptr;
}

void block_put(int device, void *p, size_t cls) {
  if (!p) return;
  if (g_cached_bytes + cls > kBlockCacheMax) {
    hipFree(p);
    return;
  }
  g_block_cache[device].emplace(cls, p);
  g_cached_bytes += cls;
}

// Pinned host blocks, cached the same way (size classes, guarded by g_rt_mu):
// a copy between device and pageable memory goes through the runtime's own
// staging, about 20 us each and one after the other; copies to a pinned block
// are queued together and waited for once.  The cache is bounded and goes
// back to the system with the last context.
std::multimap<size_t, void *> g_host_cache;
size_t g_host_cached = 0;
int g_contexts = 0;
constexpr size_t kHostCacheMax = 256ull << 20;

void host_put(HostBuf &b) {
  if (!b.p) return;
  RtLock lk(g_rt_mu);
  if (g_host_cached + b.bytes > kHostCacheMax || g_contexts == 0) {
    hipHostFree(b.p);
  } else {
    g_host_cache.emplace(b.bytes, b.p);
    g_host_cached += b.bytes;
  }
  b = HostBuf{};
}

// At least `bytes`; a large enough block is kept (no copy may be in flight).
bool host_get(HostBuf &b, size_t bytes) {
  if (b.p && b.bytes >= bytes) return true;
  host_put(b);
  RtLock lk(g_rt_mu);
  const size_t c = size_class(std::max<size_t>(bytes, 4096));
  const auto it = g_host_cache.find(c);
  if (it != g_host_cache.end()) {
    b.p = it->second;
    g_host_cache.erase(it);
    g_host_cached -= c;
  } else if (hipHostMalloc(&b.p, c, hipHostMallocDefault) != hipSuccess) {
    b.p = nullptr;
    return false;
  }
  b.bytes = c;
  return true;
}

int dalloc(Sys *s, DevBuf &b, size_t bytes) {
  if (bytes == 0) bytes = 8;
  if (s->dry) {
    s->dry_bytes += size_class(bytes);
    return PMX_OK;
  }
  RtLock lk(g_rt_mu);
  if (b.p && b.bytes >= bytes) return PMX_OK;
  if (b.p) {
    // a growing buffer: its last users must be done before the block is reused
    hipStreamSynchronize(s->ctx->stream);
    hipStreamSynchronize(s->ctx->stream2);
    block_put(s->ctx->device, b.p, b.bytes);
  }
  const size_t cls = size_class(bytes);
  b.p = block_get(s->ctx->device, cls);
  if (!b.p) return fail(s->ctx, PMX_ERR_OOM, "hipMalloc failed (" + std::to_string(cls) + " bytes)");
  b.bytes = cls;
  if (!b.listed) s->all.push_back(&b);
  b.listed = true;
  return PMX_OK;
}

template <class T>
T *P(DevBuf &b) {
  return reinterpret_cast<T *>(b.p);
}

unsigned nblk(long long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// Abramowitz-free alpha choice (NonbondedPMEwaldSystemForce.h:520-537).
double choose_alpha(double rc, double acc) {
  double a = 1.0;
  while (std::erfc(a * rc) / rc >= acc) a *= 2.0;
  double lo = 0., hi = a;
  for (int i = 0; i < 100; ++i) {
    a = 0.5 * (lo + hi);
    if (std::erfc(a * rc) / rc >= acc)
      lo = a;
    else
      hi = a;
  }
  return a;
}

// The transform of length n as a product of the kernels' radices: the fewest
// passes (each costs two block barriers and a trip through LDS), and among
// those the smallest largest radix.
bool make_plan(int n, FftPlan &pl) {
  static const int kRad[] = {10, 9, 8, 6, 5, 4, 3, 2};
  int best[12], cur[12], nbest = 0;
  auto search = [&](auto &self, int m, int depth) -> void {
    if (m == 1) {
      const int big = *std::max_element(cur, cur + depth), was = nbest ? *std::max_element(best, best + nbest) : 0;
      if (!nbest || depth < nbest || (depth == nbest && big < was)) {
        nbest = depth;
        std::copy(cur, cur + depth, best);
      }
      return;
    }
    if (depth >= 12 || (nbest && depth >= nbest)) return;
    for (int r : kRad)
      if (m % r == 0 && (depth == 0 || r <= cur[depth - 1])) {
        cur[depth] = r;
        self(self, m / r, depth + 1);
      }
  };
  pl = FftPlan{};
  pl.n = n;
  if (n < 2) return false;
  search(search, n, 0);
  pl.nrad = nbest;
  pl.magic_n = div_magic((unsigned)n);
  unsigned ns = 1;
  for (int s = 0; s < nbest; ++s) {
    pl.rad[s] = best[s];
    pl.magic[s] = ns > 1 ? div_magic(ns) : 0u;
    ns *= (unsigned)best[s];
  }
  return nbest > 0;
}

void bspline_host(int order, double w, double *th, double *dth) {
  if (order == 2) {
    th[0] = 1.0 - w;
    th[1] = w;
    dth[0] = -1.0;
    dth[1] = 1.0;
    return;
  }
  th[order - 1] = 0.0;
  th[1] = w;
  th[0] = 1.0 - w;
  for (int k = 2; k < order - 1; k++) {
    double div = 1.0 / k;
    th[k] = div * w * th[k - 1];
    for (int j = 1; j < k; j++) th[k - j] = div * ((w + j) * th[k - j - 1] + (k + 1 - j - w) * th[k - j]);
    th[0] = div * (1 - w) * th[0];
  }
  dth[0] = -th[0];
  for (int j = 1; j <= order - 1; j++) dth[j] = th[j - 1] - th[j];
  double div = 1.0 / (order - 1.0);
  th[order - 1] = div * w * th[order - 2];
  for (int j = 1; j < order - 1; j++)
    th[order - 1 - j] = div * ((w + j) * th[order - j - 2] + (order - j - w) * th[order - 1 - j]);
  th[0] = div * (1 - w) * th[0];
}

SwitchC make_switch(int kind, double on, double rc) {
  SwitchC s{};
  s.kind = kind;
  s.rc2 = rc * rc;
  s.on2 = on * on;
  double t = rc * rc - on * on;
  s.s1 = kind == SW_C2 ? 1.0 / (t * t * t) : 0.0;
  s.s2 = rc * rc - 3.0 * on * on;
  s.s3 = kind == SW_C2 ? 4.0 / (t * t * t) : 0.0;
  s.c15_1 = 1.5 / rc;
  s.c05_3 = 0.5 / (rc * rc * rc);
  s.c15_3 = 1.5 / (rc * rc * rc);
  return s;
}

int validate(pmx_ctx *c, const pmx_sys_desc *d) {
  if (!d) return fail(c, PMX_ERR_ARG, "null descriptor");
  if (d->n <= 0 || d->ntypes <= 0 || d->nexcl < 0) return fail(c, PMX_ERR_ARG, "bad sizes");
  if (!d->charge || !d->type || !d->lj || (d->nexcl > 0 && !d->excl)) return fail(c, PMX_ERR_ARG, "null array");
  if (d->ntypes > kMaxTypesTotal) return fail(c, PMX_ERR_UNSUPPORTED, "more than 4096 LJ types");
  for (int k = 0; k < 3; ++k)
    if (!(d->box[k] > 0)) return fail(c, PMX_ERR_ARG, "box edge must be > 0");
  if (d->lj_switch < 0 || d->lj_switch > 3 || d->coul_kind < 0 || d->coul_kind > 2)
    return fail(c, PMX_ERR_ARG, "bad force kind");
  if (d->lj_switch == SW_NONE && d->coul_kind == COUL_NONE) return fail(c, PMX_ERR_ARG, "no force selected");
  if (d->lj_switch != SW_NONE && !(d->lj_rc > 0)) return fail(c, PMX_ERR_ARG, "LJ cutoff must be > 0");
  if (d->lj_switch == SW_C2 && !(d->lj_on >= 0 && d->lj_on < d->lj_rc))
    return fail(c, PMX_ERR_ARG, "C2 switching function: 0 <= switchon < cutoff");
  if (d->coul_kind != COUL_NONE && !(d->coul_rc > 0)) return fail(c, PMX_ERR_ARG, "Coulomb cutoff must be > 0");
  if (d->coul_kind == COUL_CUTOFF && d->coul_switch == SW_C2 && !(d->coul_on >= 0 && d->coul_on < d->coul_rc))
    return fail(c, PMX_ERR_ARG, "C2 switching function: 0 <= switchon < cutoff");
  if (d->coul_kind == COUL_CUTOFF && (d->coul_switch < 1 || d->coul_switch > 3))
    return fail(c, PMX_ERR_ARG, "bad Coulomb switching function");
  if (d->coul_kind == COUL_PME) {
    if (d->coul_switch != SW_CUTOFF && d->coul_switch != SW_C1)
      return fail(c, PMX_ERR_ARG, "PME real term takes the Cutoff or C1 switching function");
    const int p = d->pme_order;
    if (p < 2 || p % 2 != 0 || p > 8) return fail(c, PMX_ERR_ARG, "PMEwald order must be even, 2..8");
    for (int k = 0; k < 3; ++k)
      if (d->pme_grid[k] < p) return fail(c, PMX_ERR_ARG, "PMEwald grid must be >= order");
    if (!(d->pme_accuracy > 0) && !(d->pme_alpha > 0)) return fail(c, PMX_ERR_ARG, "PMEwald accuracy > 0");
    if ((d->pme_terms & 7) == 0) return fail(c, PMX_ERR_ARG, "no PME term selected");
  }
  if (!(d->cellsize > 0)) return fail(c, PMX_ERR_ARG, "cellsize must be > 0");
  if (d->precision != PMX_FP64 && d->precision != PMX_MIXED) return fail(c, PMX_ERR_ARG, "bad precision");
  double rcmax = std::max(d->lj_switch ? d->lj_rc : 0.0, d->coul_kind ? d->coul_rc : 0.0);
  for (int k = 0; k < 3; ++k)
    if (rcmax > 0.5 * d->box[k])
      return fail(c, PMX_ERR_UNSUPPORTED, "cutoff larger than half the box (multiple images per pair)");
  for (int i = 0; i < d->n; ++i)
    if (d->type[i] < 0 || d->type[i] >= d->ntypes) return fail(c, PMX_ERR_ARG, "atom type out of range");
  for (int e = 0; e < d->nexcl; ++e) {
    int a = d->excl[3 * e], b = d->excl[3 * e + 1], cl = d->excl[3 * e + 2];
    if (a < 0 || b < 0 || a >= d->n || b >= d->n || cl < 0 || cl > 2)
      return fail(c, PMX_ERR_ARG, "exclusion entry out of range");
  }
  return PMX_OK;
}

// Launch shapes of the PME passes.  Beside the pair kernel's four blocks of
// 80 registers a CU has 64 VGPRs a lane left on each SIMD, which is room for one
// block of 512 threads or two of 256, and about 38 KB of LDS; the passes stay
// within that (which take 512 threads: see below).
//  - Tiles of the spread and gather passes: tx x ty lines along z.  Wider
//    tiles repeat less of an atom's work (each tile that an atom's stencil
//    touches visits it: (tx + p - 1)(ty + p - 1) / (tx ty) tiles) and write
//    longer segments; 8 x 4 where that still gives at least 4 tiles per CU.
//    Where the spread has the device to itself (main stream, batches) tiles of
//    twice the LDS in blocks of 512 threads did no better: 9,000 atoms on 192 x
//    192 x 48 points 104 us a step with, 103 without, on 256 x 256 x 64 at order
//    8 196 and 185, in FP64 269 and 247; 200,000 atoms on 192^3 306 and 303.
//  - y pass: 8 neighbouring lines (64- or 128-byte segments), x pass: 8
//    (contiguous anyway), fewer while that leaves fewer than two blocks per
//    CU; at most tune_fft_lines.
// The compute units are a constant, not the device's: the gather adds an FP32
// partial per tile and the x pass an energy partial per block, so other tiles
// or lines would give other last bits on a partition of the device.
constexpr int kShapeCus = 256;
int fft_blocking(Sys *s) {
  PmeParams &pm = s->pme, &pg = s->pme_g;
  const size_t cx = s->mixed ? 8 : 16;
  const int small = 256 * kFftPerThread;  // points of a block of 256 threads
  // the larger of the charge sums (16 bytes a point of two lines) and the
  // transforms (a complex number), and the twiddles (of LONG passes in memory)
  auto lds = [&](const PmeParams &q, size_t per_point) {
    return per_point * (size_t)(q.tx * q.ty / 2) * pme_line(q.nz, q.order) + (q.nz > kFftMax ? 0 : cx * (q.nz + 1));
  };
  auto tiles = [&](PmeParams &q, int tx, size_t per_point) {
    q.tx = tx;
    q.ty = 4;
    while (q.tx * q.ty > 2 && lds(q, per_point) > 36864) {
      if (q.tx > 4)
        q.tx /= 2;
      else if (q.ty > 1)
        q.ty /= 2;
      else
        q.tx /= 2;
    }
    q.ntx = (q.nx + q.tx - 1) / q.tx;
    q.nty = (q.ny + q.ty - 1) / q.ty;
  };
  pg = pm;
  const bool wide = (long long)pm.nx * pm.ny >= 32ll * 4 * kShapeCus;
  tiles(pg, wide ? 8 : 4, cx);
  tiles(pm, wide ? 8 : 4, 16);
  s->lds_z = lds(pm, 16);
  s->lds_g = lds(pg, cx);
  auto lines = [&](int n, int other) {
    int l = 0;
    while (l < 3 && (2 << l) <= s->tune_fft_lines && ((long long)n << (l + 1)) <= small) ++l;
    while (l > 0 && (1 << l) >= 2 * other) --l;
    while (l > 2 && (long long)pm.nzh * ((other + (1 << l) - 1) >> l) < 2 * kShapeCus) --l;
    return l;
  };
  s->ylog = lines(pm.ny, pm.nx);
  s->xlog = lines(pm.nx, pm.ny);
  s->lds_y = cx * (((size_t)(pm.ny | 1) << s->ylog) + (pm.ny > kFftMax ? 0 : pm.ny));
  s->lds_x = cx * (((size_t)(pm.nx | 1) << s->xlog) + (pm.nx > kFftMax ? 0 : pm.nx));
  s->lds_p = cx * ((size_t)(pm.nx | 1) * pm.ny + pm.nx + pm.ny);
  // threads: a line needs n / kFftPerThread; the tiles and planes transform
  // as many lines at a time as the block has threads for.  Planes and the
  // gather take 512, which finds room beside the pair kernel's four blocks of 80
  // registers: a step of 4,000 / 9,400 / 13,800 / 26,000 / 1,000,000 atoms
  // 65.9 / 80.5 / 87.1 / 105.5 / 1,501 us with 256, 63.7 / 75.7 / 78.0 /
  // 97.3 / 1,465 with 512.  The spread and the line passes on large grids do
  // better with two blocks of 256 (1,000,000 atoms 1,465 -> 1,592 and 1,527; a y
  // pass of 216 x 240 x 240 points whose blocks of 512 waited for the pair kernel's
  // last ones took 0.70 ms instead of 0.1), and
  // so do planes and gather in batches, which fill the device (64 systems 24.0
  // ms with 256, 24.8 with 512; 16 in FP64 14.0 and 14.9).
  auto threads = [&](int n, int l) { return ((long long)n << l) > small ? 512 : 256; };
  s->thr_z = threads(pm.nz, 0);
  s->thr_g = kPmeBlock;
  s->thr_gb = threads(pm.nz, 0);
  s->thr_y = threads(pm.ny, s->ylog);
  s->thr_x = threads(pm.nx, s->xlog);
  s->thr_p = kPmeBlock;
  s->thr_pb = threads(std::max(pm.nx, pm.ny), 0);
  s->fft_plane = s->tune_fft_planes && pm.nx * pm.ny <= kFftPlanePoints && s->lds_p <= 36864;
  s->recip_blocks = s->fft_plane ? pm.nzh : pm.nzh * ((pm.ny + (1 << s->xlog) - 1) >> s->xlog);
  // the columns of the sort that can hold atoms whose stencils touch a row or
  // column of tiles: places from the first base's to the last base's cell,
  // widened by half the skin (an atom's way since the sort)
  std::vector<int2> tc;
  const double m = 0.5 * s->md.skin + 1e-3;
  auto window = [&](int nt, int tl, int K, double L, int ncol) {
    const int p = pm.order, back = (p - 1) / 2;
    const double h = L / K, w = L / ncol;
    for (int t = 0; t < nt; ++t) {
      const double lo = (t * tl - p + 1 + back) * h - m, hi = (t * tl + tl + back) * h + m;
      const long long a = (long long)std::floor(lo / w), b = (long long)std::floor(hi / w);
      if (b - a + 1 >= ncol)
        tc.push_back(make_int2(0, ncol));
      else
        tc.push_back(make_int2((int)(((a % ncol) + ncol) % ncol), (int)(b - a + 1)));
    }
  };
  for (const PmeParams *q : {&pm, &pg}) {
    window(q->ntx, q->tx, q->nx, s->box.L[0], q->ncx);
    window(q->nty, q->ty, q->ny, s->box.L[1], q->ncy);
  }
  if (int rc = dalloc(s, s->tcol, 8 * tc.size())) return rc;
  if (int rc = dalloc(s, s->recip_e, 8 * (size_t)s->recip_blocks)) return rc;
  HIPCHK(hipMemcpyAsync(s->tcol.p, tc.data(), 8 * tc.size(), hipMemcpyHostToDevice, s->ctx->stream));
  HIPCHK(hipStreamSynchronize(s->ctx->stream));
  return PMX_OK;
}

template <bool MIXED>
void run_pair_phase(Sys *s, bool stats, int phase);

int setup(Sys *s) {
  const pmx_sys_desc &d = s->d;
  s->acc_clean = false;  // buffers are (re)allocated below
  s->list_valid = false;
  s->mixed = d.precision == PMX_MIXED;
  s->n = d.n;
  s->q.assign(d.charge, d.charge + d.n);
  s->type.assign(d.type, d.type + d.n);
  s->lj.assign(d.lj, d.lj + (size_t)d.ntypes * d.ntypes * 4);

  // Exclusions (ExclusionTable.cpp:103-120): the correction table holds each
  // pair once, in insertion order, with the class it was first added with
  // (its filter set orders pairs on (a1, a2) only, ExclusionTable.cpp:20-27);
  // the lookup class of a pair is the last one added.
  std::set<std::pair<int, int>> seen;
  std::map<std::pair<int, int>, int> cls;
  s->etab.clear();
  for (int e = 0; e < d.nexcl; ++e) {
    int a = d.excl[3 * e], b = d.excl[3 * e + 1], c = d.excl[3 * e + 2];
    if (a > b) std::swap(a, b);
    if (c != 0 && a != b && !seen.count({a, b})) {
      s->etab.push_back(make_int4(a, b, c, 0));
      seen.insert({a, b});
    }
    if (a != b) cls[{a, b}] = c;
  }
  std::vector<std::vector<int2>> part(d.n);
  for (auto &kv : cls) {
    if (kv.second == 0) continue;
    part[kv.first.first].push_back(make_int2(kv.first.second, kv.second));
    part[kv.first.second].push_back(make_int2(kv.first.first, kv.second));
  }
  s->eptr.assign(d.n + 1, 0);
  s->elist.clear();
  for (int a = 0; a < d.n; ++a) {
    std::sort(part[a].begin(), part[a].end(), [](int2 x, int2 y) { return x.x < y.x; });
    s->eptr[a] = (int)s->elist.size();
    for (auto &v : part[a]) s->elist.push_back(v);
  }
  s->eptr[d.n] = (int)s->elist.size();

  // Box (PeriodicBoundaryConditions.cpp:32-77)
  Box &bx = s->box;
  for (int k = 0; k < 3; ++k) {
    bx.L[k] = d.box[k];
    bx.Linv[k] = 1.0 / d.box[k];
    bx.o[k] = d.origin[k];
    double a = d.origin[k] - d.box[k] * 0.5, b = d.origin[k] + d.box[k] * 0.5;
    bx.mn[k] = std::min(a, b);
    double mx = std::max(a, b);
    bx.H[k] = mx - bx.mn[k];
    bx.H2[k] = bx.H[k] * 0.5;
  }
  bx.Lr[0] = (bx.L[1] * bx.L[2]) / (bx.L[0] * (bx.L[1] * bx.L[2]));
  bx.Lr[1] = (bx.L[2] * bx.L[0]) / (bx.L[1] * (bx.L[2] * bx.L[0]));
  bx.Lr[2] = (bx.L[0] * bx.L[1]) / (bx.L[2] * (bx.L[0] * bx.L[1]));
  {
    double dx = (bx.L[0] * 0.5) * (bx.L[0] * 0.5), dy = (bx.L[1] * 0.5) * (bx.L[1] * 0.5),
           dz = (bx.L[2] * 0.5) * (bx.L[2] * 0.5);
    bx.D = std::min(dx, std::min(dy, dz));
  }

  // Binning parameters: x-y columns about one supercluster (64 atoms) wide
  // and deep, z bins of about two atoms per column; reference cell grid
  // (CubicCellManager.cpp:46-65, ArrayCellListStructure.cpp:40-42).
  BinParams &bp = s->bin;
  bp.box = bx;
  const double vol = bx.L[0] * bx.L[1] * bx.L[2];
  const double rho = std::max(1, d.n) / vol;
  const double a_sc = std::cbrt(kSuperSize / rho);
  bp.ncx = (int)std::max(1L, std::min(1024L, std::lround(bx.L[0] / a_sc)));
  bp.ncy = (int)std::max(1L, std::min(1024L, std::lround(bx.L[1] / a_sc)));
  {
    const double area = (bx.L[0] / bp.ncx) * (bx.L[1] / bp.ncy);
    const long long nzb = std::lround(bx.L[2] * rho * area / 2.0);
    bp.nzb = (int)std::max(1LL, std::min(1LL << 16, nzb));
  }
  bp.cxinv = bp.ncx / bx.L[0];
  bp.cyinv = bp.ncy / bx.L[1];
  bp.zinv = bp.nzb / bx.L[2];
  s->ncols = bp.ncx * bp.ncy;
  // each column's last supercluster may be partly padding
  s->nsuper = (d.n + kSuperSize - 1) / kSuperSize + s->ncols;
  s->npad = s->nsuper * kSuperSize;
  s->ncl = s->npad / kClusterSize;
  for (int k = 0; k < 3; ++k) {
    double H = bx.H[k];
    double e = H / std::max(1.0, std::floor(H / d.cellsize));
    bp.rc_inv[k] = 1.0 / e;
    bp.rc_n[k] = std::max(1, (int)std::floor(H / e + 1.0e-14));
    bp.delta[k] = bx.o[k] - bx.mn[k];
  }
  s->nbins = (long long)s->ncols * bp.nzb;
  s->nscanblocks = (int)((s->nbins + kScanBlock - 1) / kScanBlock);

  // Pair parameters
  PairParams &pp = s->pp;
  pp.box = bx;
  pp.has_lj = d.lj_switch != SW_NONE;
  pp.lj = make_switch(pp.has_lj ? d.lj_switch : SW_CUTOFF, d.lj_on, pp.has_lj ? d.lj_rc : 0.0);
  pp.coul = d.coul_kind;
  if (d.coul_kind == COUL_CUTOFF)
    pp.co = make_switch(d.coul_switch, d.coul_on, d.coul_rc);
  else if (d.coul_kind == COUL_PME)
    pp.co = make_switch(d.coul_switch, 0.0, d.coul_rc);
  else
    pp.co = make_switch(SW_CUTOFF, 0.0, 0.0);
  const double rcmax = std::max(pp.has_lj ? d.lj_rc : 0.0, d.coul_kind ? d.coul_rc : 0.0);
  pp.rc2max = rcmax * rcmax;
  const double Lmax = std::max(bx.L[0], std::max(bx.L[1], bx.L[2]));
  const double eps = s->mixed ? std::ldexp(1.0, -24) : std::ldexp(1.0, -53);
  // |delta r2| bound: coordinates rounded once (<= L eps), differences and
  // image shift (<= 3 L eps per component), squares and sums (3 rc^2 eps).
  pp.guard = 4.0 * (2.0 * std::sqrt(3.0) * rcmax * 3.0 * Lmax * eps + 3.0 * pp.rc2max * eps);
  pp.csf = d.csf;
  pp.ntypes = d.ntypes;
  for (int k = 0; k < 3; ++k) {
    pp.Lhi[k] = origin_round(bx.L[k]);
    pp.Llo[k] = bx.L[k] - pp.Lhi[k];
  }

  s->pme_on = d.coul_kind == COUL_PME;
  // PME without -real: the pair pass still decides membership (pair
  // statistics) but its Coulomb part sees zero charges
  s->qpair = s->pme_on && !(d.pme_terms & PMX_PME_REAL) ? 0.0 : 1.0;
  s->alpha = 0;
  s->self_e = s->charged_e = 0;
  if (s->pme_on) {
    s->alpha = d.pme_alpha > 0 ? d.pme_alpha : choose_alpha(d.coul_rc, d.pme_accuracy);
    pp.alpha = s->alpha;
    pp.a2pi = 2.0 * s->alpha / std::sqrt(M_PI);
    if (d.pme_terms & PMX_PME_CORR) {
      double q2 = 0, qs = 0;
      for (int i = 0; i < d.n; ++i) q2 += d.charge[i] * d.charge[i];
      for (int i = 0; i < d.n; ++i) qs += d.charge[i];
      s->self_e = -q2 * s->alpha / std::sqrt(M_PI);
      if (std::fabs(qs * 0.00268283) > 1.0e-5) s->charged_e = -M_PI / (2.0 * vol * s->alpha * s->alpha) * qs * qs;
    }
  }

  // List parameters
  ListParams &lp = s->lp;
  const double margin = 4.0 * Lmax * std::ldexp(1.0, -23) + 1e-4;
  for (int k = 0; k < 3; ++k) {
    lp.L[k] = (float)bx.L[k];
    lp.Linv[k] = (float)(1.0 / bx.L[k]);
  }
  lp.skin = (float)s->md.skin;
  lp.rlist2 = (float)((rcmax + margin + s->md.skin) * (rcmax + margin + s->md.skin));
  s->pp.prune_r2 = (double)lp.rlist2 * (1.0 + 1e-5);
  auto direct = [&](auto &c) {
    using R = std::decay_t<decltype(c.guard)>;
    c = std::decay_t<decltype(c)>{};
    c.lj.load(pp.lj);
    c.co.load(pp.co);
    c.ljkind = pp.lj.kind;
    c.cokind = pp.co.kind;
    c.rmax2 = !pp.has_lj ? c.co.rc2 : (pp.coul == COUL_NONE ? c.lj.rc2 : std::max(c.lj.rc2, c.co.rc2));
    c.guard = (R)pp.guard;
    c.near2 = std::nextafter(c.rmax2 + c.guard, (R)INFINITY);
    c.in2 = std::nextafter(c.rmax2 - c.guard, (R)0);
    c.pa = (R)(0.3275911 * pp.alpha);
    c.ke = (R)((sizeof(R) == 4 ? -1.4426950408889634 : -1.0) * pp.alpha * pp.alpha);
    c.a2pi = (R)pp.a2pi;
    c.csf = (R)pp.csf;
    c.prune_r2 = (R)pp.prune_r2;
    for (int k = 0; k < 3; ++k) {
      c.hi[k] = (R)pp.Lhi[k];
      c.lo[k] = (R)pp.Llo[k];
      c.inv[k] = (R)bx.Linv[k];
    }
  };
  direct(s->pp.dc);
  direct(s->pp.dd);
  lp.rc = (float)rcmax;
  lp.ncl = s->ncl;
  lp.nsuper = s->nsuper;
  {
    // supercluster pruning radius: the list radius plus a slack that covers
    // the FP32 rounding of the boxes; column reach from the column widths
    // (atoms of columns kx + 1 apart are more than kx widths apart in x)
    const double rl = rcmax + margin + s->md.skin + 0.02;
    lp.rlist2_sc = (float)(rl * rl);
    lp.ncx = bp.ncx;
    lp.ncy = bp.ncy;
    lp.kx = (int)std::floor(rl / (bx.L[0] / bp.ncx)) + 1;
    lp.ky = (int)std::floor(rl / (bx.L[1] / bp.ncy)) + 1;
  }
  {
    // generous per-supercluster capacity from the cluster density
    const double rho_cl = s->ncl / vol;
    const double reach = 2.0 * rcmax + 24.0;
    long long c = (long long)std::ceil(rho_cl * reach * reach * reach) + 64;
    s->cap = (int)std::min<long long>(c, s->ncl);
    s->cap = (s->cap + kTileEntries - 1) / kTileEntries * kTileEntries;
  }
  lp.cap = s->cap;
  s->ntiles_cap = kMaxRuns + 2 * s->nsuper;  // a run touches one supercluster or more
  s->maxmaskwork = std::max(1024, s->nsuper * 128);

  int rc;
  auto A = [&](DevBuf &b, size_t bytes) { return dalloc(s, b, bytes); };
  const size_t N = d.n, NP = s->npad;
  if ((rc = A(s->xorig, 24 * N)) || (rc = A(s->xwrap, 24 * N)) || (rc = A(s->q_d, 8 * N)) ||
      (rc = A(s->type_d, 4 * N)) || (rc = A(s->key, 4 * N)) || (rc = A(s->hist, 16 * ((s->nbins + 3) / 4))) ||
      (rc = A(s->start, 16 * ((s->nbins + 3) / 4))) || (rc = A(s->cursor, 16 * ((s->nbins + 3) / 4))) ||
      (rc = A(s->scansum, 4 * (size_t)s->nscanblocks)) || (rc = A(s->perm, 4 * N)) ||
      (rc = A(s->permp, 4 * NP)) ||
      (rc = A(s->slot, 4 * N)) || (rc = A(s->refcell, 4 * N)) || (rc = A(s->xs, 32 * NP)) ||
      (rc = A(s->xs64, 32 * NP)) || (rc = A(s->ts, 4 * NP)) || (rc = A(s->sc_info, 8 * (size_t)s->nsuper)) ||
      (rc = A(s->sc_col, 4 * (size_t)s->nsuper)) || (rc = A(s->colsc, 4 * ((size_t)s->ncols + 1))) ||
      (rc = A(s->sctr, 16 * (size_t)s->nsuper)) || (rc = A(s->shalf, 16 * (size_t)s->nsuper)) ||
      (rc = A(s->sorg, 16 * (size_t)s->nsuper)) ||
      (rc = A(s->ctr, 16 * (size_t)s->ncl)) ||
      (rc = A(s->half, 16 * (size_t)s->ncl)) || (rc = A(s->entries, 16 * (size_t)s->nsuper * s->cap)) ||
      (rc = A(s->count, 4 * (size_t)s->nsuper)) || (rc = A(s->lcost, 4 * (size_t)s->nsuper)) ||
      (rc = A(s->ecost, 4 * (size_t)s->nsuper * s->cap)) ||
      (rc = A(s->runs, 8 * ((size_t)kMaxRuns + 1))) ||
      (rc = A(s->nmaskwork, 8)) || (rc = A(s->masks, 16 * 8 * (size_t)s->maxmaskwork)) ||
      (rc = A(s->ntiles, 16)) ||
      (rc = A(s->tilectr, 8)) || (rc = A(s->ljtab, 8 * s->lj.size())) ||
      (rc = A(s->ljt32, 4 * s->lj.size())) || (rc = A(s->facc, 24 * NP)) ||
      (rc = A(s->fout, 24 * N)) || (rc = A(s->pair_e, 16 * (size_t)s->ntiles_cap)) ||
      (rc = A(s->npairs, 8 * (size_t)s->ntiles_cap)) || (rc = A(s->hash, 8 * (size_t)s->ntiles_cap)) ||
      (rc = A(s->eptr_d, 4 * (N + 1))) || (rc = A(s->elist_d, 8 * s->elist.size())) ||
      (rc = A(s->eout, 64)) || (rc = A(s->border, 8 * (size_t)s->maxborder)) ||
      (rc = A(s->nborder, 8)) || (rc = A(s->border_acc, 32)))
    return rc;
  if (s->eout.p) {
    s->np_out.p = P<PassResults>(s->eout)->np;
    s->hash_out.p = P<PassResults>(s->eout)->hash;
    s->overflow.p = P<PassResults>(s->eout)->overflow;
  }
  s->term_blocks = (int)nblk((long long)NP, 256);
  // the correction table by atom (each entry listed for both of its atoms)
  std::vector<int> cptr;
  std::vector<int2> clist;
  if (!s->dry) {
    cptr.assign(N + 1, 0);
    for (const int4 &e : s->etab) {
      ++cptr[e.x + 1];
      ++cptr[e.y + 1];
    }
    for (size_t a = 0; a < N; ++a) cptr[a + 1] += cptr[a];
    clist.resize(2 * s->etab.size());
    std::vector<int> at(cptr.begin(), cptr.end() - 1);
    for (const int4 &e : s->etab) {
      clist[at[e.x]++] = make_int2(e.y, e.z);
      clist[at[e.y]++] = make_int2(e.x, e.z);
    }
  }
  if ((rc = A(s->cptr_d, 4 * (N + 1))) || (rc = A(s->clist_d, 16 * s->etab.size()))) return rc;
  // boundary pairs grow with the pair count: one block per 16 superclusters
  s->border_blocks = std::min(128, std::max(4, (int)(s->nsuper / 16)));
  if ((rc = A(s->corr_e, 8 * (size_t)s->term_blocks))) return rc;
  if (s->dry) {
    // PME buffers as allocated below (grid records, tile windows, half
    // spectrum, influence table, twiddles, energy partials bounded by ny * nzh)
    if (s->pme_on) {
      const size_t nx = d.pme_grid[0], ny = d.pme_grid[1], nz = d.pme_grid[2], nzh = nz / 2 + 1;
      const size_t GH = nx * ny * nzh, cxb = s->mixed ? 8 : 16, rb = s->mixed ? 4 : 8;
      for (size_t b : {(s->mixed ? 16 : 32) * NP, 8 * NP, 4 * (nx + ny + 4), cxb * GH, rb * GH, cxb * nx, cxb * ny,
                       cxb * nz, 8 * ny * nzh})
        s->dry_bytes += size_class(b);
    }
    return PMX_OK;
  }

  hipStream_t st = s->ctx->stream;
  // the cell histogram starts cleared; each rebuild's scan clears it again
  // (with the padding to whole groups of four that the scan reads)
  hipLaunchKernelGGL(k_fill_u32, dim3(nblk(s->nbins + 3, 256)), dim3(256), 0, st, P<uint32_t>(s->hist), 0u,
                     (s->nbins + 3) / 4 * 4);
  {
    RtLock lk(g_rt_mu);
    // the fork and join order the two streams of one device only (the host
    // never waits on them), so they need no system-scope fence
    if (!s->fork_ev) HIPCHK(hipEventCreateWithFlags(&s->fork_ev, hipEventDisableTiming | hipEventDisableSystemFence));
    if (!s->join_ev) HIPCHK(hipEventCreateWithFlags(&s->join_ev, hipEventDisableTiming | hipEventDisableSystemFence));
  }
  HIPCHK(hipMemcpyAsync(s->q_d.p, s->q.data(), 8 * N, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(s->type_d.p, s->type.data(), 4 * N, hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(s->ljtab.p, s->lj.data(), 8 * s->lj.size(), hipMemcpyHostToDevice, st));
  // FP32 copy for the mixed pair kernel when the table does not fit its LDS
  s->lj32.assign(s->lj.begin(), s->lj.end());
  HIPCHK(hipMemcpyAsync(s->ljt32.p, s->lj32.data(), 4 * s->lj32.size(), hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(s->eptr_d.p, s->eptr.data(), 4 * (N + 1), hipMemcpyHostToDevice, st));
  if (!s->elist.empty())
    HIPCHK(hipMemcpyAsync(s->elist_d.p, s->elist.data(), 8 * s->elist.size(), hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(s->cptr_d.p, cptr.data(), 4 * cptr.size(), hipMemcpyHostToDevice, st));
  if (!clist.empty())
    HIPCHK(hipMemcpyAsync(s->clist_d.p, clist.data(), 8 * clist.size(), hipMemcpyHostToDevice, st));

  if (s->pme_on) {
    PmeParams &pm = s->pme;
    pm.nx = d.pme_grid[0];
    pm.ny = d.pme_grid[1];
    pm.nz = d.pme_grid[2];
    pm.nzh = pm.nz / 2 + 1;
    pm.order = d.pme_order;
    pm.hxr = pm.nx / bx.L[0];
    pm.hyr = pm.ny / bx.L[1];
    pm.hzr = pm.nz / bx.L[2];
    pm.offx = -(pm.order - 1) / 2 + pm.nx;
    pm.offy = -(pm.order - 1) / 2 + pm.ny;
    pm.offz = -(pm.order - 1) / 2 + pm.nz;
    if (!make_plan(pm.nx, s->plx) || !make_plan(pm.ny, s->ply) || !make_plan(pm.nz, s->plz))
      return fail(s->ctx, PMX_ERR_UNSUPPORTED, "PME grid sizes must be products of 2, 3 and 5");
    if (std::max(pm.nx, std::max(pm.ny, pm.nz)) > (s->mixed ? kFftMaxLong<float> : kFftMaxLong<double>))
      return fail(s->ctx, PMX_ERR_UNSUPPORTED, "PME grid axes have at most 10125 points (5120 in FP64)");
    pm.ncx = bp.ncx;
    pm.ncy = bp.ncy;
    const size_t GH = (size_t)pm.nx * pm.ny * pm.nzh;
    const size_t cxb = s->mixed ? 8 : 16;
    if ((rc = A(s->pmw, (s->mixed ? 16 : 32) * NP)) || (rc = A(s->pmb, 8 * NP)) || (rc = A(s->spec, cxb * GH)) ||
        (rc = A(s->theta, (s->mixed ? 4 : 8) * GH)) || (rc = A(s->twx, cxb * pm.nx)) ||
        (rc = A(s->twy, cxb * pm.ny)) || (rc = A(s->twz, cxb * pm.nz)))
      return rc;
    // Influence function on the half spectrum (Grid.h:237-341 with the
    // tables of Grid.h:526-575 and dftmod :589-600).
    const int p = pm.order;
    std::vector<double> th0(p), dth0(p);
    bspline_host(p, 0.0, th0.data(), dth0.data());
    auto dftmod = [&](int nn, std::vector<double> &out) {
      out.resize(nn);
      for (int i = 0; i < nn; i++) {
        double sc = 0.0, ss = 0.0;
        for (int j = 0; j < p; j++) {
          double x = M_PI * 2.0 * i * j / (double)nn;
          sc += th0[j] * std::cos(x);
          ss += th0[j] * std::sin(x);
        }
        out[i] = 1.0 / (sc * sc + ss * ss);
      }
    };
    std::vector<double> bxm, bym, bzm;
    dftmod(pm.nx, bxm);
    dftmod(pm.ny, bym);
    dftmod(pm.nz, bzm);
    const double W = bx.L[0], Lh = bx.L[1], Hh = bx.L[2];
    const double Wr = 1.0 / W, Lr = 1.0 / Lh, Hr = 1.0 / Hh, V = W * Lh * Hh;
    const double fac = M_PI * M_PI / (s->alpha * s->alpha);
    std::vector<double> ex(pm.nx), ey(pm.ny), ez(pm.nzh);
    for (int i = 0; i < pm.nx; i++) {
      int i0 = i <= pm.nx / 2 ? i : i - pm.nx;
      ex[i] = std::exp(-fac * (i0 * Wr) * (i0 * Wr));
    }
    for (int j = 0; j < pm.ny; j++) {
      int j0 = j <= pm.ny / 2 ? j : j - pm.ny;
      ey[j] = std::exp(-fac * (j0 * Lr) * (j0 * Lr));
    }
    for (int k = 0; k < pm.nzh; k++) ez[k] = std::exp(-fac * (k * Hr) * (k * Hr));
    std::vector<double> th(GH);
    const double piVr = 1.0 / (M_PI * V);
    for (int i = 0; i < pm.nx; i++) {
      int i0 = i <= pm.nx / 2 ? i : i - pm.nx;
      double mi = i0 * Wr, exi = ex[i] * piVr;
      for (int j = 0; j < pm.ny; j++) {
        int j0 = j <= pm.ny / 2 ? j : j - pm.ny;
        double bxy = bxm[i] * bym[j], mj = j0 * Lr, mij = mi * mi + mj * mj, exy = exi * ey[j];
        for (int k = 0; k < pm.nzh; k++) {
          double v = 0.0;
          if (i != 0 || j != 0 || k != 0) {
            double mk = k * Hr, m2 = mij + mk * mk;
            v = bxy * bzm[k] * exy * ez[k] / m2;
          }
          th[((size_t)k * pm.ny + j) * pm.nx + i] = v;  // the spectrum's layout [k][j][i]
        }
      }
    }
    // uploads on the system's stream; the host arrays live until the
    // synchronisation at the end of the set-up
    std::vector<double> tw64[3];
    std::vector<float> tw32[3], thf;
    auto tw = [&](int axis, int nn, DevBuf &b) -> hipError_t {
      std::vector<double> &t = tw64[axis];
      t.resize(2 * nn);
      for (int m = 0; m < nn; ++m) {
        t[2 * m] = std::cos(-2.0 * M_PI * m / nn);
        t[2 * m + 1] = std::sin(-2.0 * M_PI * m / nn);
      }
      if (s->mixed) {
        tw32[axis].assign(t.begin(), t.end());
        return hipMemcpyAsync(b.p, tw32[axis].data(), 4 * tw32[axis].size(), hipMemcpyHostToDevice, st);
      }
      return hipMemcpyAsync(b.p, t.data(), 8 * t.size(), hipMemcpyHostToDevice, st);
    };
    HIPCHK(tw(0, pm.nx, s->twx));
    HIPCHK(tw(1, pm.ny, s->twy));
    HIPCHK(tw(2, pm.nz, s->twz));
    if (s->mixed) {
      thf.assign(th.begin(), th.end());
      HIPCHK(hipMemcpyAsync(s->theta.p, thf.data(), 4 * GH, hipMemcpyHostToDevice, st));
    } else {
      HIPCHK(hipMemcpyAsync(s->theta.p, th.data(), 8 * GH, hipMemcpyHostToDevice, st));
    }
    if ((rc = fft_blocking(s))) return rc;
    HIPCHK(hipStreamSynchronize(st));  // the host tables above are still alive
  }
  HIPCHK(hipStreamSynchronize(st));
  if (s->mixed)  // the pair-kernel grid (phase -1 sizes it)
    run_pair_phase<true>(s, false, -1);
  else
    run_pair_phase<false>(s, false, -1);
  s->cached = true;
  return PMX_OK;
}

// Launches of the kernels templated on the force kinds: the pair kernel
// (phase 0, main stream), the boundary pairs (phase 1, main stream), the
// exclusion correction with the bonded terms (phase 2, second stream), or all
// three fixups in one launch on the main stream (phase 3); the fixups are one
// kernel with different block ranges.
template <bool MIXED>
FixupArgs<MIXED> fixup_args(Sys *s, bool stats, bool border_here, bool rest_here, int *nblocks);

// Blocks per CU of a pair-kernel launch of `runs` least runs: at least 1, at
// most those of as many waves on the device.
int pair_blocks_of(int per_cu, int runs) { return std::min(per_cu, runs / (kPairBlock / kWave) / 256); }

// Resident blocks per CU of a pair kernel, at least 1.  Each caller keeps its
// kernel's value in a function-local static, initialized once even under
// concurrent first calls.
int pair_blocks_per_cu(const void *kernel) {
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, kPairBlock, 0) != hipSuccess || per_cu < 1)
    per_cu = 1;
  return per_cu;
}

template <bool MIXED, int C, int LJ, int CS, bool BIGLJ = false>
void launch_pair_phase(Sys *s, bool stats, int phase) {
  hipStream_t st = phase == 2 ? s->ctx->stream2 : s->ctx->stream;
  const bool border_here = phase == 1 || phase == 3, rest_here = phase == 2 || phase == 3;
  using R4 = typename Real4<typename std::conditional<MIXED, float, double>::type>::type;
  auto *facc = P<typename AccT<MIXED>::type>(s->facc);
  if (phase < 0) {
    // as many blocks as are resident at once (the schedules assign each
    // wave its first tile, or its whole run, statically)
    static const int fit =
        pair_blocks_per_cu(reinterpret_cast<const void *>(k_pair<MIXED, C, LJ, CS, BIGLJ, kPairPlain>));
    // the least number of the list's runs is that of the waves: of the mixed
    // form for the device it is cut for, whatever this one is
    const bool grid = s->pme_on && (s->d.pme_terms & PMX_PME_RECIP);
    s->cut = !MIXED ? kCut64 : grid ? kCutBeside : kCutAlone;
    const int per_cu = pair_blocks_of(fit, s->cut.min_runs);
    if (!MIXED) s->cut.min_runs = per_cu * (kPairBlock / kWave) * 256;
    // knob > 0: blocks per CU; 0: as many as fit; < 0: that many fewer
    const int bpc = s->tune_pair_blocks > 0 ? std::min(s->tune_pair_blocks, per_cu)
                                            : std::max(1, per_cu + s->tune_pair_blocks);
    s->pair_grid = std::max(1, s->ctx->cus * bpc);
    return;
  }
  if (phase == 0) {
    const unsigned grid = (unsigned)s->pair_grid;
    PairOut out{P<double>(s->pair_e), P<long long>(s->npairs), P<unsigned long long>(s->hash),
                P<int2>(s->border), P<int>(s->nborder), s->maxborder, P<int>(s->overflow),
                P<unsigned long long>(s->border_acc)};
    // the list prune runs in the first pass after a build, at the build
    // positions (a pruned cluster pair cannot gain a member before the next
    // build only when judged there); not in a pass that counts pairs, nor
    // for tables beyond the LDS size, which are rare
    const bool prune = !BIGLJ && !stats && s->tune_prune && s->prune_pending;
    s->prune_pending = false;
    const R4 *ljt = MIXED ? reinterpret_cast<const R4 *>(s->ljt32.p) : reinterpret_cast<const R4 *>(s->ljtab.p);
#define PMX_PAIR_ARGS                                                                                              \
  s->pp, s->tune_schedule, P<int2>(s->runs), P<int>(s->ntiles), P<int>(s->count), P<int>(s->tilectr),            \
      P<int4>(s->entries), P<int4>(s->entries), s->cap, P<unsigned short>(s->masks), P<R4>(s->xs),                 \
      P<float4>(s->sorg), P<int>(s->ts), P<int>(s->permp), P<double>(s->ljtab), ljt, facc, out
    if (stats)
      hipLaunchKernelGGL((k_pair<MIXED, C, LJ, CS, BIGLJ, kPairStats>), dim3(grid), dim3(kPairBlock), 0, st,
                         PMX_PAIR_ARGS);
    else if (prune)
      hipLaunchKernelGGL((k_pair<MIXED, C, LJ, CS, false, kPairPrune>), dim3(grid), dim3(kPairBlock), 0, st,
                         PMX_PAIR_ARGS);
    else
      hipLaunchKernelGGL((k_pair<MIXED, C, LJ, CS, BIGLJ, kPairPlain>), dim3(grid), dim3(kPairBlock), 0, st,
                         PMX_PAIR_ARGS);
#undef PMX_PAIR_ARGS
    return;
  }
  int nfix = 0;
  const FixupArgs<MIXED> a = fixup_args<MIXED>(s, stats, border_here, rest_here, &nfix);
  if (nfix > 0)
    hipLaunchKernelGGL((k_fixups<MIXED, C, LJ, CS>), dim3(nfix), dim3(256), 0, st, a);
}

// Arguments of k_fixups for one force pass: the boundary pairs
// (border_here), the exclusion correction and the bonded terms (rest_here);
// *nblocks gets the launch's block count.
template <bool MIXED>
FixupArgs<MIXED> fixup_args(Sys *s, bool stats, bool border_here, bool rest_here, int *nblocks) {
  using R4 = typename Real4<typename std::conditional<MIXED, float, double>::type>::type;
  FixupArgs<MIXED> a{};
  a.border_blocks = border_here ? s->border_blocks : 0;
  a.pp = s->pp;
  a.stats = stats ? 1 : 0;
  a.border = P<int2>(s->border);
  a.nborder = P<int>(s->nborder);
  a.maxborder = s->maxborder;
  a.xs = P<R4>(s->xs);
  a.sorg = P<float4>(s->sorg);
  a.ts = P<int>(s->ts);
  a.perm = P<int>(s->permp);
  a.xorig = P<double>(s->xorig);
  a.ljtab = P<double>(s->ljtab);
  a.eptr = P<int>(s->eptr_d);
  a.elist = P<int2>(s->elist_d);
  a.border_e = P<unsigned long long>(s->border_acc);
  a.border_stat = P<unsigned long long>(s->border_acc) + 2;
  const bool corr = s->pme_on && (s->d.pme_terms & PMX_PME_CORR) && !s->etab.empty();
  const bool bonded = s->md.on && s->md.nb + s->md.na > 0;
  a.npad = s->npad;
  a.q = P<double>(s->q_d);
  a.alpha = s->alpha;
  a.csf = s->d.csf;
  a.corr_e = P<double>(s->corr_e);
  if (corr) {
    a.at.eptr = P<int>(s->cptr_d);
    a.at.excl = P<int2>(s->clist_d);
  }
  if (bonded) {
    a.at.mptr = P<int2>(s->md.mptr);
    a.at.bond = P<int>(s->md.bonds);
    a.at.bpar = P<double2>(s->md.bpar);
    a.at.angle = P<int4>(s->md.angles);
    a.at.apar = P<double2>(s->md.apar);
    a.bond_e = P<double>(s->md.bond_e);
  }
  a.facc = P<typename AccT<MIXED>::type>(s->facc);
  *nblocks = a.border_blocks + (rest_here && (corr || bonded) ? s->term_blocks : 0);
  return a;
}

template <bool MIXED>
void run_pair_phase(Sys *s, bool stats, int phase) {
  const int lj = s->d.lj_switch, cs = s->d.coul_switch;
  if (s->d.ntypes > kMaxTypes && lj != SW_NONE) {
    // LJ table too large for the kernel's LDS: read from the caches
    if (s->pp.coul == COUL_PME)
      launch_pair_phase<MIXED, COUL_PME, SW_ANY, SW_ANY, true>(s, stats, phase);
    else if (s->pp.coul == COUL_CUTOFF)
      launch_pair_phase<MIXED, COUL_CUTOFF, SW_ANY, SW_ANY, true>(s, stats, phase);
    else
      launch_pair_phase<MIXED, COUL_NONE, SW_ANY, SW_ANY, true>(s, stats, phase);
    return;
  }
  if (s->pp.coul == COUL_PME) {
    if (lj == SW_C2 && cs == SW_CUTOFF)
      launch_pair_phase<MIXED, COUL_PME, SW_C2, SW_CUTOFF>(s, stats, phase);
    else if (lj == SW_NONE)
      launch_pair_phase<MIXED, COUL_PME, SW_NONE, SW_ANY>(s, stats, phase);
    else
      launch_pair_phase<MIXED, COUL_PME, SW_ANY, SW_ANY>(s, stats, phase);
  } else if (s->pp.coul == COUL_CUTOFF) {
    if (lj == SW_C2 && cs == SW_C1)
      launch_pair_phase<MIXED, COUL_CUTOFF, SW_C2, SW_C1>(s, stats, phase);
    else if (lj == SW_NONE)
      launch_pair_phase<MIXED, COUL_CUTOFF, SW_NONE, SW_ANY>(s, stats, phase);
    else
      launch_pair_phase<MIXED, COUL_CUTOFF, SW_ANY, SW_ANY>(s, stats, phase);
  } else {
    launch_pair_phase<MIXED, COUL_NONE, SW_ANY, SW_ANY>(s, stats, phase);
  }
}

// The atoms' grid records, for the kernels that write them (null without PME).
template <class R>
PmeSlots<R> pme_slots(Sys *s) {
  if (!s->pme_on || !(s->d.pme_terms & PMX_PME_RECIP)) return PmeSlots<R>{nullptr, nullptr};
  return PmeSlots<R>{P<typename Real4<R>::type>(s->pmw), P<int2>(s->pmb)};
}

// Charge spread with the z transform (order: even, 2..8); with: the atoms'
// terms in the same launch (blocks of 256 threads).
template <bool MIXED>
void run_spread(Sys *s, hipStream_t st, bool with = false) {
  using T = typename std::conditional<MIXED, float, double>::type;
  using T4 = typename Real4<T>::type;
  int nterms = 0;
  FixupArgs<MIXED> terms{};
  if (with) terms = fixup_args<MIXED>(s, false, false, true, &nterms);
#define PMX_SPREAD_ARGS \
  s->pme, s->plz, P<int2>(s->tcol), P<int>(s->colsc), P<T4>(s->pmw), P<int2>(s->pmb), P<Cx<T>>(s->twz), P<Cx<T>>(s->spec)
#define PMX_SPREAD(ORD)                                                                                             \
  if (nterms)                                                                                                       \
    hipLaunchKernelGGL((k_pme_spread_terms<MIXED, ORD>), dim3(s->pme.ntx * s->pme.nty + nterms), dim3(s->thr_z),    \
                       s->lds_z, st, PMX_SPREAD_ARGS, terms);                                                       \
  else if (s->pme.nz > kFftMax)                                                                                     \
    hipLaunchKernelGGL((k_pme_spread_z<MIXED, ORD, true>), dim3(s->pme.ntx * s->pme.nty), dim3(s->thr_z), s->lds_z, \
                       st, PMX_SPREAD_ARGS);                                                                        \
  else                                                                                                              \
    hipLaunchKernelGGL((k_pme_spread_z<MIXED, ORD>), dim3(s->pme.ntx * s->pme.nty), dim3(s->thr_z), s->lds_z, st,   \
                       PMX_SPREAD_ARGS)
  switch (s->pme.order) {
    case 2: PMX_SPREAD(2); break;
    case 4: PMX_SPREAD(4); break;
    case 6: PMX_SPREAD(6); break;
    default: PMX_SPREAD(8); break;
  }
#undef PMX_SPREAD
#undef PMX_SPREAD_ARGS
}

// The transforms and the force gather on the second stream.
template <bool MIXED>
int run_pme(Sys *s, bool timing) {
  using T = typename std::conditional<MIXED, float, double>::type;
  using T4 = typename Real4<T>::type;
  using Acc = typename AccT<MIXED>::type;
  hipStream_t st = s->ctx->stream2;
  const PmeParams &pm = s->pme, &pg = s->pme_g;
  if (s->d.pme_terms & PMX_PME_RECIP) {
    if (s->fft_plane) {
      hipLaunchKernelGGL((k_fft_plane_conv<T>), dim3(pm.nzh), dim3(s->thr_p), s->lds_p, st, pm, s->ply, s->plx,
                         P<Cx<T>>(s->twy), P<Cx<T>>(s->twx), P<T>(s->theta), P<Cx<T>>(s->spec), P<double>(s->recip_e));
    } else {
      const int yb = pm.nzh * ((pm.nx + (1 << s->ylog) - 1) >> s->ylog);
      auto y = [&](bool inverse) {
        auto go = [&](auto kernel) {
          hipLaunchKernelGGL(kernel, dim3(yb), dim3(s->thr_y), s->lds_y, st, pm, s->ply, s->ylog, inverse,
                             P<Cx<T>>(s->twy), P<Cx<T>>(s->spec));
        };
        if (pm.ny > kFftMax)
          go(k_fft_y<T, true>);
        else
          go(k_fft_y<T>);
      };
      auto x = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(s->recip_blocks), dim3(s->thr_x), s->lds_x, st, pm, s->plx, s->xlog,
                           P<Cx<T>>(s->twx), P<T>(s->theta), P<Cx<T>>(s->spec), P<double>(s->recip_e));
      };
      y(false);
      if (pm.nx > kFftMax)
        x(k_fft_x_conv<T, true>);
      else
        x(k_fft_x_conv<T>);
      y(true);
    }
    if (timing) hipEventRecord(s->ev[5], st);
#define PMX_GATHER_ARGS                                                                                              \
  dim3(pg.ntx * pg.nty), dim3(s->thr_g), s->lds_g, st, pg, s->plz, P<int2>(s->tcol) + pm.ntx + pm.nty,               \
      P<int>(s->colsc), P<T4>(s->pmw), P<int2>(s->pmb), P<Cx<T>>(s->twz), P<Cx<T>>(s->spec), P<Acc>(s->facc)
#define PMX_GATHER(ORD)                                                                                              \
  if (pm.nz > kFftMax)                                                                                               \
    hipLaunchKernelGGL((k_pme_z_gather<MIXED, ORD, true>), PMX_GATHER_ARGS);                                         \
  else                                                                                                               \
    hipLaunchKernelGGL((k_pme_z_gather<MIXED, ORD>), PMX_GATHER_ARGS)
    switch (pm.order) {
      case 2: PMX_GATHER(2); break;
      case 4: PMX_GATHER(4); break;
      case 6: PMX_GATHER(6); break;
      default: PMX_GATHER(8); break;
    }
#undef PMX_GATHER
#undef PMX_GATHER_ARGS
  } else if (timing) {
    hipEventRecord(s->ev[5], st);
  }
  if (timing) hipEventRecord(s->ev[6], st);
  return PMX_OK;
}

EnergyArgs energy_args(Sys *s, bool stats) {
  const bool recip = s->pme_on && (s->d.pme_terms & PMX_PME_RECIP);
  const bool corr = s->pme_on && (s->d.pme_terms & PMX_PME_CORR) && !s->etab.empty();
  return {s->ntiles_cap, P<int>(s->ntiles), P<double>(s->pair_e), s->mixed ? 1 : 0, recip ? s->recip_blocks : 0,
          P<double>(s->recip_e), corr ? s->term_blocks : 0, P<double>(s->corr_e), P<long long>(s->npairs),
          P<unsigned long long>(s->hash), stats ? 1 : 0, P<unsigned long long>(s->border_acc),
          P<unsigned long long>(s->border_acc) + 2, P<double>(s->eout), P<long long>(s->np_out),
          P<unsigned long long>(s->hash_out)};
}

// The energies of the last pass added up: into eout for pmx_md_get_state, or
// aside before its partials go, where eout keeps the last evaluation's.
void reduce_energies(Sys *s, bool aside) {
  if (s->energies_at != Sys::kInPartials) return;
  EnergyArgs a = energy_args(s, false);
  if (aside) {
    PassResults *const h = P<PassResults>(s->md.held);
    a.out = h->e;
    a.out_np = h->np;
    a.out_hash = h->hash;
  }
  hipLaunchKernelGGL(k_reduce_energy, dim3(1), dim3(kEndBlock), 0, s->ctx->stream, a);
  s->energies_at = aside ? Sys::kInHeld : Sys::kInResults;
}

void timing_begin_call(Sys *s, bool timing) {
  if (!timing) return;
  RtLock lk(g_rt_mu);
  if (s->evused == s->evsets.size()) {
    std::vector<hipEvent_t> set(kStages + 1);
    for (auto &e : set) hipEventCreate(&e);
    s->evsets.push_back(set);
  }
  s->ev = s->evsets[s->evused++].data();
  hipEventRecord(s->ev[0], s->ctx->stream);
}

// Cell sort of the current positions and the cluster-pair list built from it
// (the reference rebuilds its cell lists at every force evaluation,
// ForceGroup.cpp:57; the MD path rebuilds when the skin requires it).
// Work tiles of the current list for the current schedule and pair grid.
unsigned runs_blocks(Sys *s) { return (unsigned)std::min<long long>(256, nblk(s->nsuper, kRunsBlock / kWave)); }
void make_runs(Sys *s, hipStream_t st) {
  hipLaunchKernelGGL(k_runs, dim3(runs_blocks(s)), dim3(kRunsBlock), 0, st, s->nsuper, P<int>(s->count),
                     P<int>(s->lcost), P<int>(s->ecost), s->cap, s->cut, P<int2>(s->runs), P<int>(s->ntiles));
}

SortedBins sorted_bins(Sys *s) {
  return {s->n, s->nbins, P<uint32_t>(s->key), P<uint32_t>(s->start), P<int>(s->perm)};
}

MaskArgs mask_args(Sys *s) {
  return {P<int>(s->permp),           P<int>(s->slot), P<int>(s->eptr_d), P<int2>(s->elist_d),
          P<unsigned short>(s->masks), s->maxmaskwork};
}

// clear: a pass begins, with its overflow flag cleared.
int rebuild(Sys *s, bool timing, bool clear) {
  hipStream_t st = s->ctx->stream;
  const int n = s->n;
  // the histogram starts cleared (set-up, then each scan clears it)
  hipLaunchKernelGGL(k_bin, dim3(nblk(n, 256)), dim3(256), 0, st, n, P<double>(s->xorig), s->bin, P<uint32_t>(s->key),
                     P<double>(s->xwrap), P<int>(s->refcell), P<uint32_t>(s->hist),
                     clear ? P<int>(s->overflow) : nullptr);
  if (s->nbins <= kScanSingleMax) {
    hipLaunchKernelGGL(k_scan_columns, dim3(1), dim3(kScanBlock), 0, st, P<uint32_t>(s->hist), (int)s->nbins,
                       P<uint32_t>(s->start), P<uint32_t>(s->cursor), s->ncols, s->bin.nzb, n, s->nsuper,
                       P<int2>(s->sc_info), P<int>(s->sc_col), P<int>(s->colsc));
  } else {
    hipLaunchKernelGGL(k_scan_blocksums, dim3(s->nscanblocks), dim3(kScanBlock), 0, st, P<uint32_t>(s->hist),
                       s->nbins, P<uint32_t>(s->scansum));
    hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(kScanBlock), 0, st, P<uint32_t>(s->scansum), s->nscanblocks);
    hipLaunchKernelGGL(k_scan_final, dim3(s->nscanblocks), dim3(kScanBlock), 0, st, P<uint32_t>(s->hist), s->nbins,
                       P<uint32_t>(s->scansum), P<uint32_t>(s->start), P<uint32_t>(s->cursor));
    hipLaunchKernelGGL(k_columns, dim3(1), dim3(kScanBlock), 0, st, s->ncols, s->bin.nzb, n, P<uint32_t>(s->start),
                       s->nsuper, P<int2>(s->sc_info), P<int>(s->sc_col), P<int>(s->colsc));
  }
  hipLaunchKernelGGL(k_scatter, dim3(nblk(n, 256)), dim3(256), 0, st, n, P<uint32_t>(s->key), P<uint32_t>(s->cursor),
                     P<int>(s->perm));
  double4 *xbuild = s->md.on ? P<double4>(s->md.xbuild) : nullptr;
  if (s->mixed)
    hipLaunchKernelGGL(k_split_fill<float>, dim3(nblk((long long)s->nsuper * 64, 256)), dim3(256), 0, st, s->nsuper,
                       P<int2>(s->sc_info), sorted_bins(s), P<double>(s->xwrap), P<int>(s->permp), P<int>(s->slot),
                       P<double>(s->q_d), P<int>(s->type_d), P<float4>(s->xs), P<double4>(s->xs64), P<int>(s->ts),
                       P<double>(s->xorig), P<double>(s->md.minv), xbuild, P<float4>(s->sorg), P<float4>(s->ctr), P<float4>(s->half),
                       P<float4>(s->sctr), P<float4>(s->shalf), P<int>(s->nmaskwork), s->qpair, s->pme, pme_slots<float>(s));
  else
    hipLaunchKernelGGL(k_split_fill<double>, dim3(nblk((long long)s->nsuper * 64, 256)), dim3(256), 0, st, s->nsuper,
                       P<int2>(s->sc_info), sorted_bins(s), P<double>(s->xwrap), P<int>(s->permp), P<int>(s->slot),
                       P<double>(s->q_d), P<int>(s->type_d), P<double4>(s->xs), P<double4>(s->xs64), P<int>(s->ts),
                       P<double>(s->xorig), P<double>(s->md.minv), xbuild, P<float4>(s->sorg), P<float4>(s->ctr), P<float4>(s->half),
                       P<float4>(s->sctr), P<float4>(s->shalf), P<int>(s->nmaskwork), s->qpair, s->pme, pme_slots<double>(s));
  if (timing) hipEventRecord(s->ev[1], st);
  hipLaunchKernelGGL(k_build_list, dim3(s->nsuper), dim3(kListBlock), list_lds_bytes(s->cap), st, s->lp,
                     P<int>(s->sc_col), P<int>(s->colsc), P<float4>(s->sctr), P<float4>(s->shalf), P<float4>(s->ctr),
                     P<float4>(s->half), P<int4>(s->entries), P<int>(s->count), P<int>(s->ecost), P<int>(s->lcost),
                     mask_args(s), P<int>(s->nmaskwork), P<int>(s->overflow));
  make_runs(s, st);
  s->list_valid = true;
  s->prune_pending = true;
  if (timing) hipEventRecord(s->ev[2], st);
  return PMX_OK;
}

// Forces (and optionally energies) at the current positions with the
// current list: pair + boundary pairs, PME, correction, bonded terms, then
// the FP64 force array in the caller's atom order.
// next: the following MD step's kick (with next_dmax, its displacement
// record): the pass ends with that step's kick and drift fused into the
// force unsort.
// Clears the force accumulators and the pass counters.
void launch_zero(Sys *s) {
  const int npad = s->npad;
  ZeroRanges z{};
  int nr = 0;
  z.p[nr] = P<unsigned long long>(s->facc);
  z.n[nr++] = 3ll * npad;
  z.p[nr] = P<unsigned long long>(s->tilectr);
  z.n[nr++] = 1;
  z.p[nr] = P<unsigned long long>(s->nborder);
  z.n[nr++] = 1;
  z.p[nr] = P<unsigned long long>(s->border_acc);
  z.n[nr++] = 4;
  hipLaunchKernelGGL(k_zero, dim3(std::max(1u, nblk(3ll * npad, 256)), nr), dim3(256), 0, s->ctx->stream, z);
}

int forces(Sys *s, unsigned flags, bool energies, const Kick *next = nullptr, unsigned *next_dmax = nullptr,
           const ChunkEnd &end = {}) {
  hipStream_t st = s->ctx->stream;
  const bool timing = flags & PMX_EVAL_TIMING;
  const bool stats = flags & PMX_EVAL_PAIRSTATS;
  const int n = s->n, npad = s->npad;
  // A completed pass leaves the accumulators and the counters cleared
  // (k_unsort_forces, k_pair); only the first pass after (re)allocation or
  // after an interrupted pass clears them here.
  if (!s->acc_clean) launch_zero(s);
  s->acc_clean = false;
  s->staged = false;
  s->energies_at = energies ? Sys::kInResults : Sys::kInPartials;
  if (timing) hipEventRecord(s->ev[2], st);
  // fork: FFT, gather, exclusion correction and bonded terms on the second
  // stream beside the pair kernel; all add into the zeroed accumulators.
  // The spread runs before the fork on the main stream, or first on the
  // second stream (tuning knob).  The pair stage's start event is recorded
  // after the fork, right before the pair kernel.
  hipStream_t st2 = s->ctx->stream2;
  const bool spread = s->pme_on && (s->d.pme_terms & PMX_PME_RECIP);
  const bool spread2 = spread && s->tune_spread_stream2;
  // with the spread on the main stream go the correction and the bonded terms
  // that would follow the pair kernel there
  const bool terms_early = spread && !spread2 && s->tune_fixup_main && s->thr_z == 256;
  if (spread && !spread2) {
    if (s->mixed)
      run_spread<true>(s, st, terms_early);
    else
      run_spread<false>(s, st, terms_early);
  }
  HIPCHK(hipEventRecord(s->fork_ev, st));
  HIPCHK(hipStreamWaitEvent(st2, s->fork_ev, 0));
  if (spread2) {
    if (s->mixed)
      run_spread<true>(s, st2);
    else
      run_spread<false>(s, st2);
  }
  if (timing) hipEventRecord(s->ev[4], st);
  if (s->mixed)
    run_pair_phase<true>(s, stats, 0);
  else
    run_pair_phase<false>(s, stats, 0);
  if (timing) hipEventRecord(s->ev[3], st);
  if (s->pme_on) {
    int rc = s->mixed ? run_pme<true>(s, timing) : run_pme<false>(s, timing);
    if (rc) return rc;
  } else if (timing) {
    hipEventRecord(s->ev[5], st2);
    hipEventRecord(s->ev[6], st2);
  }
  // the exclusion correction and bonded terms (unless they went with the
  // spread) on the second stream (after the PME chain), or with the boundary
  // pairs on the main stream after the pair kernel (tuning knob)
  const int fix_phase = s->tune_fixup_main && !terms_early ? 3 : 1;
  if (!s->tune_fixup_main) {
    if (s->mixed)
      run_pair_phase<true>(s, stats, 2);
    else
      run_pair_phase<false>(s, stats, 2);
  }
  if (timing) hipEventRecord(s->ev[7], st2);
  HIPCHK(hipEventRecord(s->join_ev, st2));
  // boundary pairs after the pair kernel, then join
  if (s->mixed)
    run_pair_phase<true>(s, stats, fix_phase);
  else
    run_pair_phase<false>(s, stats, fix_phase);
  HIPCHK(hipStreamWaitEvent(st, s->join_ev, 0));
  if (next && s->mixed)
    hipLaunchKernelGGL((k_unsort_kick_drift<true, float>), dim3(nblk(npad, 256)), dim3(256), 0, st, npad, *next,
                       s->md.h, P<int>(s->permp), P<unsigned long long>(s->facc), P<int>(s->tilectr),
                       P<int>(s->nborder), P<double>(s->md.v), P<double>(s->xorig), P<double4>(s->md.xbuild),
                        P<float4>(s->xs), P<double4>(s->xs64),
                       P<float4>(s->sorg), next_dmax, s->pme, pme_slots<float>(s));
  else if (next)
    hipLaunchKernelGGL((k_unsort_kick_drift<false, double>), dim3(nblk(npad, 256)), dim3(256), 0, st, npad, *next,
                       s->md.h, P<int>(s->permp), P<double>(s->facc), P<int>(s->tilectr), P<int>(s->nborder),
                       P<double>(s->md.v), P<double>(s->xorig), P<double4>(s->md.xbuild), P<double4>(s->xs), P<double4>(s->xs64), P<float4>(s->sorg),
                       next_dmax, s->pme, pme_slots<double>(s));
  else if (energies && s->mixed)
    hipLaunchKernelGGL(k_unsort_energy<true>, dim3(1 + nblk(n, kEndBlock)), dim3(kEndBlock), 0, st, n, P<int>(s->slot),
                       P<unsigned long long>(s->facc), P<double>(s->fout), P<int>(s->tilectr), P<int>(s->nborder),
                       energy_args(s, stats));
  else if (energies)
    hipLaunchKernelGGL(k_unsort_energy<false>, dim3(1 + nblk(n, kEndBlock)), dim3(kEndBlock), 0, st, n,
                       P<int>(s->slot), P<double>(s->facc), P<double>(s->fout), P<int>(s->tilectr),
                       P<int>(s->nborder), energy_args(s, stats));
  else if (s->mixed)
    hipLaunchKernelGGL(k_unsort_forces<true>, dim3(nblk(n, 256)), dim3(256), 0, st, n, P<int>(s->slot),
                       P<unsigned long long>(s->facc), P<double>(s->fout), P<int>(s->tilectr),
                       P<int>(s->nborder), end);
  else
    hipLaunchKernelGGL(k_unsort_forces<false>, dim3(nblk(n, 256)), dim3(256), 0, st, n, P<int>(s->slot),
                       P<double>(s->facc), P<double>(s->fout), P<int>(s->tilectr), P<int>(s->nborder), end);
  s->acc_clean = true;
  if (timing) hipEventRecord(s->ev[8], st);
  HIPCHK(hipGetLastError());
  return PMX_OK;
}

int compute(Sys *s, unsigned flags) {
  const bool timing = flags & PMX_EVAL_TIMING;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s->ctx->stream, &cap) == hipSuccess && cap != hipStreamCaptureStatusNone) s->recorded = true;
  timing_begin_call(s, timing);
  int rc = rebuild(s, timing, true);
  if (rc) return rc;
  return forces(s, flags, true);
}

constexpr size_t kStageChunk = 1 << 20;
constexpr int kStageChunks = 4;
constexpr size_t kStageBytes = kStageChunk * kStageChunks;

int stage_get(Sys *s, size_t bytes) {
  s->staged = false;
  if (!host_get(s->stage, bytes)) return fail(s->ctx, PMX_ERR_OOM, "pinned host memory");
  if (bytes < kStageBytes || s->stage_ev[0]) return PMX_OK;
  RtLock lk(g_rt_mu);
  for (auto &e : s->stage_ev) HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  return PMX_OK;
}

// Device memory larger than the stage to the host: use(offset, data, bytes)
// for each chunk in order while the copies of the next ones run.
template <class F>
int fetch(Sys *s, const void *src, size_t bytes, F use) {
  hipStream_t st = s->ctx->stream;
  if (int rc = stage_get(s, kStageBytes)) return rc;
  unsigned char *const h = static_cast<unsigned char *>(s->stage.p);
  const size_t nc = (bytes + kStageChunk - 1) / kStageChunk;
  for (size_t k = 0; k < nc + kStageChunks - 1; ++k) {
    if (k < nc) {
      const size_t o = k * kStageChunk;
      HIPCHK(hipMemcpyAsync(h + k % kStageChunks * kStageChunk, static_cast<const unsigned char *>(src) + o,
                            std::min(kStageChunk, bytes - o), hipMemcpyDeviceToHost, st));
      HIPCHK(hipEventRecord(s->stage_ev[k % kStageChunks], st));
    }
    if (k + 1 < (size_t)kStageChunks) continue;
    const size_t c = k + 1 - kStageChunks, o = c * kStageChunk;
    HIPCHK(hipEventSynchronize(s->stage_ev[c % kStageChunks]));
    use(o, h + c % kStageChunks * kStageChunk, std::min(kStageChunk, bytes - o));
  }
  return PMX_OK;
}

// Host memory to the device in the stream's order; the source is free on
// return.  Large sources go through the stage in chunks (the runtime copies
// pageable memory one chunk after the other).
int send(Sys *s, void *dst, const void *src, size_t bytes) {
  hipStream_t st = s->ctx->stream;
  if (bytes <= kStageBytes) {
    HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st));
    return PMX_OK;
  }
  if (int rc = stage_get(s, kStageBytes)) return rc;
  unsigned char *const h = static_cast<unsigned char *>(s->stage.p);
  const size_t nc = (bytes + kStageChunk - 1) / kStageChunk;
  for (size_t k = 0; k < nc; ++k) {
    const size_t o = k * kStageChunk, len = std::min(kStageChunk, bytes - o);
    unsigned char *const c = h + k % kStageChunks * kStageChunk;
    if (k >= (size_t)kStageChunks) HIPCHK(hipEventSynchronize(s->stage_ev[k % kStageChunks]));
    std::memcpy(c, static_cast<const unsigned char *>(src) + o, len);
    HIPCHK(hipMemcpyAsync(static_cast<unsigned char *>(dst) + o, c, len, hipMemcpyHostToDevice, st));
    HIPCHK(hipEventRecord(s->stage_ev[k % kStageChunks], st));
  }
  for (auto &e : s->stage_ev) HIPCHK(hipEventSynchronize(e));
  return PMX_OK;
}

// The results of a pass, and then its forces, in the stage.
constexpr size_t kResultWords = sizeof(PassResults) / 8;
bool results_fit(const Sys *s) { return 8 * (kResultWords + 3 * (size_t)s->n) <= kStageBytes; }
// A batched pass brings this system's results to the host.
bool batch_stages(const Sys *s) { return results_fit(s) && !s->recorded; }

struct OutList {
  OutArgs a{};
  int k = 0;
  explicit OutList(void *dst) { a.dst = static_cast<unsigned long long *>(dst); }
  // words of 8 bytes from src on; returns where they arrive
  double *add(const void *src, size_t words) {
    const long long at = k ? a.end[k - 1] : 0;
    for (int i = k; i < 5; ++i) {
      a.src[i] = static_cast<const unsigned long long *>(src);
      a.end[i] = at + (long long)words;
    }
    if (words) ++k;
    return reinterpret_cast<double *>(a.dst + at);
  }
  unsigned blocks() const { return (unsigned)std::min<long long>(1024, std::max<long long>(1, (a.end[4] + 255) / 256)); }
  void launch(hipStream_t st) const { hipLaunchKernelGGL(k_out, dim3(blocks()), dim3(256), 0, st, a); }
};

int finish(Sys *s, unsigned flags, double *f_aos, double *energies) {
  hipStream_t st = s->ctx->stream;
  const size_t fb = f_aos ? 24 * (size_t)s->n : 0;
  const bool once = s->staged || !fb || results_fit(s);
  if (!s->staged) {
    if (int rc = stage_get(s, once ? sizeof(PassResults) + fb : kStageBytes)) return rc;
    OutList out(s->stage.p);
    out.add(s->eout.p, kResultWords);
    if (once) out.add(s->fout.p, fb / 8);
    out.launch(st);
  }
  HIPCHK(hipStreamSynchronize(st));
  const unsigned char *const h = static_cast<const unsigned char *>(s->stage.p);
  PassResults r;
  std::memcpy(&r, h, sizeof r);
  s->last_np = r.np[0];
  s->last_hash = r.hash[0];
  if (r.overflow[0]) return fail(s->ctx, PMX_ERR_OVERFLOW, "cluster pair list capacity exceeded");
  if ((flags & PMX_EVAL_TIMING) && s->ev)
    for (int k = 0; k < kStages; ++k)
      hipEventElapsedTime(&s->stage_ms[k], s->ev[kStageEv[k][0]], s->ev[kStageEv[k][1]]);
  auto add = [&](size_t o, const void *data, size_t bytes) {
    double *const to = f_aos + o / 8;
    const double *const from = static_cast<const double *>(data);
    for (size_t k = 0; k < bytes / 8; ++k) to[k] += from[k];
  };
  if (once && fb)
    add(0, h + sizeof(PassResults), fb);
  else if (fb)
    if (int rc = fetch(s, s->fout.p, fb, add)) return rc;
  if (energies) {
    double ec = r.e[0];
    if (s->pme_on) ec += r.e[2] + r.e[3] + s->self_e + s->charged_e;
    energies[PMX_E_COULOMB] += ec;
    energies[PMX_E_LENNARDJONES] += r.e[1];
  }
  return PMX_OK;
}

void drop_graphs(Sys *s) {
  for (auto &kv : s->md.gexec) hipGraphExecDestroy(kv.second);
  s->md.gexec.clear();
}

int grow_and_retry(Sys *s) {
  drop_graphs(s);  // captured chunks hold the old buffer addresses
  s->list_valid = false;
  // double the list capacity and the mask pool, then rebuild buffers
  s->cap = std::min(s->ncl + kTileEntries, 2 * s->cap);
  s->cap = (s->cap + kTileEntries - 1) / kTileEntries * kTileEntries;
  s->lp.cap = s->cap;
  s->ntiles_cap = kMaxRuns + 2 * s->nsuper;
  s->maxmaskwork *= 2;
  s->maxborder *= 2;
  if (int rc0 = dalloc(s, s->border, 8 * (size_t)s->maxborder)) return rc0;
  int rc;
  if ((rc = dalloc(s, s->entries, 16 * (size_t)s->nsuper * s->cap)) || (rc = dalloc(s, s->ecost, 4 * (size_t)s->nsuper * s->cap)) ||
      (rc = dalloc(s, s->pair_e, 16 * (size_t)s->ntiles_cap)) || (rc = dalloc(s, s->npairs, 8 * (size_t)s->ntiles_cap)) ||
      (rc = dalloc(s, s->hash, 8 * (size_t)s->ntiles_cap)) ||
      (rc = dalloc(s, s->masks, 16 * 8 * (size_t)s->maxmaskwork)))
    return rc;
  return PMX_OK;
}

}  // namespace

struct pmx_sys {
  Sys s;
};

extern "C" {

unsigned long long pmx_pair_hash(int i, int j) {
  if (i > j) std::swap(i, j);
  return pair_hash((uint32_t)i, (uint32_t)j);
}

int pmx_ctx_create(int device, pmx_ctx **out) {
  RtLock lk(g_rt_mu);
  if (!out) return PMX_ERR_ARG;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return PMX_ERR_NODEV;
  if (device < 0 || device >= ndev) return PMX_ERR_ARG;
  if (hipSetDevice(device) != hipSuccess) return PMX_ERR_HIP;
  // The code objects in this library are gfx950 only.
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) != hipSuccess) return PMX_ERR_HIP;
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) return PMX_ERR_NODEV;
  if (device >= kMaxDevices) return PMX_ERR_UNSUPPORTED;
  if (!g_scratch_addr[device]) {
    void *ptr = nullptr;
    if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return PMX_ERR_HIP;
    g_scratch_addr[device] = ptr;
  }
  pmx_ctx *c = new pmx_ctx();
  c->device = device;
  c->scratch = g_scratch_addr[device];
  c->cus = prop.multiProcessorCount > 0 ? prop.multiProcessorCount : 256;
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
    delete c;
    return PMX_ERR_HIP;
  }
  if (hipStreamCreateWithFlags(&c->stream2, hipStreamNonBlocking) != hipSuccess) {
    hipStreamDestroy(c->stream);
    delete c;
    return PMX_ERR_HIP;
  }
  ++g_contexts;
  *out = c;
  return PMX_OK;
}

int pmx_ctx_destroy(pmx_ctx *ctx) {
  RtLock lk(g_rt_mu);
  if (!ctx) return PMX_ERR_ARG;
  hipSetDevice(ctx->device);
  if (ctx->stream) hipStreamDestroy(ctx->stream);
  if (ctx->stream2) hipStreamDestroy(ctx->stream2);
  if (ctx->batch_host) hipHostFree(ctx->batch_host);
  if (--g_contexts == 0) {
    for (auto &kv : g_host_cache) hipHostFree(kv.second);
    g_host_cache.clear();
    g_host_cached = 0;
  }
  if (ctx->batch_fork) hipEventDestroy(ctx->batch_fork);
  if (ctx->batch_join) hipEventDestroy(ctx->batch_join);
  delete ctx;
  return PMX_OK;
}

const char *pmx_last_error(const pmx_ctx *ctx) { return ctx ? ctx->err.c_str() : "null context"; }

int pmx_sys_create(pmx_ctx *ctx, const pmx_sys_desc *desc, pmx_sys **out) {
  if (!ctx || !out) return PMX_ERR_ARG;
  *out = nullptr;
  int rc = validate(ctx, desc);
  if (rc) return rc;
  hipSetDevice(ctx->device);
  pmx_sys *ps = new pmx_sys();
  ps->s.ctx = ctx;
  ps->s.d = *desc;
  // below this size the PME chain (a fixed number of short dependent
  // launches) is the longer branch of a force pass
  ps->s.tune_fixup_main = desc->n < kFixupMainBelow ? 1 : 0;
  ps->s.tune_spread_stream2 = desc->n >= kSpread2From ? 1 : 0;
  rc = setup(&ps->s);
  if (rc) {
    pmx_sys_destroy(ps);
    return rc;
  }
  *out = ps;
  return PMX_OK;
}

int pmx_sys_destroy(pmx_sys *sys) {
  if (!sys) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  hipSetDevice(s->ctx->device);
  hipStreamSynchronize(s->ctx->stream);
  hipStreamSynchronize(s->ctx->stream2);
  RtLock lk(g_rt_mu);
  drop_graphs(s);
  for (DevBuf *b : s->all) block_put(s->ctx->device, b->p, b->bytes);
  if (s->fork_ev) hipEventDestroy(s->fork_ev);
  if (s->join_ev) hipEventDestroy(s->join_ev);
  for (auto &e : s->md.chunk_ev)
    if (e) hipEventDestroy(e);
  if (s->md.host) hipHostFree(s->md.host);
  for (auto &e : s->stage_ev)
    if (e) hipEventDestroy(e);
  host_put(s->stage);
  for (auto &set : s->evsets)
    for (auto &e : set) hipEventDestroy(e);
  delete sys;
  return PMX_OK;
}

int pmx_sys_uncache(pmx_sys *sys) {
  if (!sys) return PMX_ERR_ARG;
  sys->s.cached = false;
  return PMX_OK;
}

int pmx_sys_set_positions(pmx_sys *sys, const double *x_aos) {
  if (!sys || !x_aos) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  hipSetDevice(s->ctx->device);
  // an exponent of all ones carries into the sign bit (one branch in all: the loop vectorizes)
  unsigned long long bad = 0;
  for (size_t k = 0; k < 3 * (size_t)s->n; ++k) {
    unsigned long long u;
    std::memcpy(&u, x_aos + k, 8);
    bad |= (u & 0x7fffffffffffffffull) + 0x0010000000000000ull;
  }
  if (bad >> 63) return fail(s->ctx, PMX_ERR_ARG, "non-finite position");
  if (int rc = send(s, s->xorig.p, x_aos, 24 * (size_t)s->n)) return rc;
  s->have_positions = true;
  return PMX_OK;
}

int pmx_sys_compute(pmx_sys *sys, unsigned flags) {
  if (!sys) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  if (!s->have_positions) return fail(s->ctx, PMX_ERR_ARG, "positions not set");
  hipSetDevice(s->ctx->device);
  if (!s->cached) {
    int rc = setup(s);
    if (rc) return rc;
  }
  return compute(s, flags);
}

int pmx_sys_compute_noalloc(pmx_sys *sys, unsigned flags) {
  if (!sys) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  if (flags & PMX_EVAL_TIMING)
    return fail(s->ctx, PMX_ERR_ARG, "pmx_sys_compute_noalloc: PMX_EVAL_TIMING needs event creation");
  if (!s->have_positions) return fail(s->ctx, PMX_ERR_ARG, "positions not set");
  if (!s->cached)
    return fail(s->ctx, PMX_ERR_ARG,
                "pmx_sys_compute_noalloc: tables dropped by pmx_sys_uncache (pmx_sys_compute rebuilds them)");
  if (!s->ctx->scratch) return fail(s->ctx, PMX_ERR_NODEV, "no scratch address for this device");
  // layout: counters (tile counter, boundary count, 4 boundary sums), then
  // boundary records, per-tile energies, pair counts and hashes
  auto up = [](size_t v) { return (v + 255) / 256 * 256; };
  const size_t nb = (size_t)s->maxborder, nt = (size_t)s->ntiles_cap;
  const size_t o_border = 256, o_pe = up(o_border + 8 * nb), o_np = up(o_pe + 16 * nt), o_h = up(o_np + 8 * nt),
               end = o_h + 8 * nt;
  if (end > kScratchBytes)
    return fail(s->ctx, PMX_ERR_ARG,
                "pmx_sys_compute_noalloc: the pass needs " + std::to_string(end) + " bytes of scratch, the maximum is " +
                    std::to_string(kScratchBytes) + " (about 1,000,000 atoms at a 12 A list radius)");
  hipSetDevice(s->ctx->device);
  unsigned char *base = static_cast<unsigned char *>(s->ctx->scratch);
  DevBuf *bufs[7] = {&s->tilectr, &s->nborder, &s->border_acc, &s->border, &s->pair_e, &s->npairs, &s->hash};
  void *const addr[7] = {base, base + 8, base + 16, base + o_border, base + o_pe, base + o_np, base + o_h};
  void *saved[7];
  for (int k = 0; k < 7; ++k) {
    saved[k] = bufs[k]->p;
    bufs[k]->p = addr[k];
  }
  // the counters keep the last call's values (another system may have used
  // them): clear them with a fill kernel, which graph capture also records
  hipLaunchKernelGGL(k_fill_u64, dim3(1), dim3(64), 0, s->ctx->stream, reinterpret_cast<unsigned long long *>(base),
                     0ull, 6ll);
  const int rc = compute(s, flags);
  for (int k = 0; k < 7; ++k) bufs[k]->p = saved[k];
  return rc;
}

int pmx_sys_get_forces(pmx_sys *sys, double *f_aos, double *energies) {
  if (!sys) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  hipSetDevice(s->ctx->device);
  return finish(s, 0, f_aos, energies);
}

int pmx_sys_sync(pmx_sys *sys) {
  if (!sys) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  HIPCHK(hipStreamSynchronize(s->ctx->stream));
  return PMX_OK;
}

int pmx_sys_evaluate(pmx_sys *sys, const double *x_aos, double *f_aos, double *energies, unsigned flags) {
  if (!sys || !x_aos || !f_aos || !energies) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  int rc = pmx_sys_set_positions(sys, x_aos);
  if (rc) return rc;
  for (int attempt = 0; attempt < 6; ++attempt) {
    s->evused = 0;
    rc = pmx_sys_compute(sys, flags);
    if (rc) return rc;
    rc = finish(s, flags, f_aos, energies);
    if (rc != PMX_ERR_OVERFLOW) return rc;
    if ((rc = grow_and_retry(s))) return rc;
  }
  return fail(s->ctx, PMX_ERR_OVERFLOW, "cluster pair list capacity exceeded after retries");
}

int pmx_sys_alpha(const pmx_sys *sys, double *alpha) {
  if (!sys || !alpha) return PMX_ERR_ARG;
  *alpha = sys->s.alpha;
  return PMX_OK;
}

int pmx_sys_pair_stats(const pmx_sys *sys, long long *npairs, unsigned long long *hash) {
  if (!sys || !npairs || !hash) return PMX_ERR_ARG;
  *npairs = sys->s.last_np;
  *hash = sys->s.last_hash;
  return PMX_OK;
}

int pmx_sys_cells(pmx_sys *sys, int *cell_of_atom, int *dims) {
  if (!sys || !cell_of_atom || !dims) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  hipSetDevice(s->ctx->device);
  HIPCHK(hipMemcpyAsync(cell_of_atom, s->refcell.p, 4 * (size_t)s->n, hipMemcpyDeviceToHost, s->ctx->stream));
  HIPCHK(hipStreamSynchronize(s->ctx->stream));
  for (int k = 0; k < 3; ++k) dims[k] = s->bin.rc_n[k];
  return PMX_OK;
}

int pmx_sys_timing_begin(pmx_sys *sys) {
  if (!sys) return PMX_ERR_ARG;
  sys->s.evused = 0;
  sys->s.timing_active = true;
  return PMX_OK;
}

int pmx_sys_timing_end(pmx_sys *sys, float *avg_ms, int *ncalls) {
  if (!sys || !avg_ms || !ncalls) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  HIPCHK(hipStreamSynchronize(s->ctx->stream));
  for (int k = 0; k < kStages; ++k) avg_ms[k] = 0.f;
  const size_t m = s->evused;
  for (size_t c = 0; c < m; ++c)
    for (int k = 0; k < kStages; ++k) {
      float t = 0.f;
      HIPCHK(hipEventElapsedTime(&t, s->evsets[c][kStageEv[k][0]], s->evsets[c][kStageEv[k][1]]));
      avg_ms[k] += t;
    }
  for (int k = 0; k < kStages; ++k) avg_ms[k] = m ? avg_ms[k] / (float)m : 0.f;
  *ncalls = (int)m;
  s->evused = 0;
  s->timing_active = false;
  return PMX_OK;
}

int pmx_sys_time_pair(pmx_sys *sys, int reps, float *ms_per_launch) {
  if (!sys || reps < 1 || reps > 4096 || !ms_per_launch) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  if (!s->have_positions) return fail(s->ctx, PMX_ERR_ARG, "no positions set");
  hipSetDevice(s->ctx->device);
  hipStream_t st = s->ctx->stream;
  if (int rc = compute(s, 0)) return rc;
  // each launch gets its own zeroed tile counter and boundary-pair count
  int *ctrs = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  {
    RtLock lk(g_rt_mu);
    if (hipMalloc(&ctrs, 8 * (size_t)reps) != hipSuccess) return fail(s->ctx, PMX_ERR_OOM, "hipMalloc failed");
    if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
      if (e0) hipEventDestroy(e0);
      hipFree(ctrs);
      return fail(s->ctx, PMX_ERR_HIP, "hipEventCreate failed");
    }
  }
  hipLaunchKernelGGL(k_fill_i32, dim3(nblk(2ll * reps, 256)), dim3(256), 0, st, ctrs, 0, 2ll * reps);
  void *const tc = s->tilectr.p, *const nb = s->nborder.p;
  hipEventRecord(e0, st);
  for (int r = 0; r < reps; ++r) {
    s->tilectr.p = ctrs + r;
    s->nborder.p = ctrs + reps + r;
    if (s->mixed)
      run_pair_phase<true>(s, false, 0);
    else
      run_pair_phase<false>(s, false, 0);
  }
  s->tilectr.p = tc;
  s->nborder.p = nb;
  hipEventRecord(e1, st);
  const hipError_t e = hipEventSynchronize(e1);
  float t = 0.f;
  if (e == hipSuccess) hipEventElapsedTime(&t, e0, e1);
  {
    RtLock lk(g_rt_mu);
    hipEventDestroy(e0);
    hipEventDestroy(e1);
    hipFree(ctrs);
  }
  s->acc_clean = false;  // the repeated launches added into the accumulators
  if (e != hipSuccess) return fail(s->ctx, PMX_ERR_HIP, hipGetErrorString(e));
  *ms_per_launch = t / (float)reps;
  return PMX_OK;
}

int pmx_sys_set_tuning(pmx_sys *sys, int knob, int value) {
  if (!sys) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  switch (knob) {
    case PMX_TUNE_FFT_LINES:
      if (value < 1 || value > 64) return fail(s->ctx, PMX_ERR_ARG, "FFT lines per block must be 1..64");
      s->tune_fft_lines = value;
      break;
    case PMX_TUNE_PAIR_BLOCKS_PER_CU:
      if (value < -7 || value > 64) return fail(s->ctx, PMX_ERR_ARG, "pair blocks per CU must be -7..64");
      s->tune_pair_blocks = value;
      break;
    case PMX_TUNE_PAIR_SCHEDULE:
      if (value < 0 || value > 1) return fail(s->ctx, PMX_ERR_ARG, "pair schedule must be 0 or 1");
      s->tune_schedule = value;
      break;
    case PMX_TUNE_SPREAD_STREAM:
      if (value < 0 || value > 1) return fail(s->ctx, PMX_ERR_ARG, "spread stream must be 0 or 1");
      s->tune_spread_stream2 = value;
      break;
    case PMX_TUNE_LIST_PRUNE:
      if (value < 0 || value > 1) return fail(s->ctx, PMX_ERR_ARG, "list prune must be 0 or 1");
      s->tune_prune = value;
      break;
    case PMX_TUNE_FIXUP_STREAM:
      if (value < 0 || value > 1) return fail(s->ctx, PMX_ERR_ARG, "fixup stream must be 0 or 1");
      s->tune_fixup_main = value;
      break;
    case PMX_TUNE_FUSED_SPREAD:
      // kept for callers that set it: the spread has no launch of its own
      // that could be fused
      if (value < 0 || value > 1) return fail(s->ctx, PMX_ERR_ARG, "fused spread must be 0 or 1");
      break;
    case PMX_TUNE_FFT_PLANES:
      if (value < 0 || value > 1) return fail(s->ctx, PMX_ERR_ARG, "FFT planes must be 0 or 1");
      s->tune_fft_planes = value;
      break;
    default:
      return fail(s->ctx, PMX_ERR_ARG, "unknown tuning knob");
  }
  // captured chunks hold the old launch shapes; the tiles of the list and
  // the blocks of the x pass change, and with them the places of the energy
  // partials: those of the state at hand are added up before
  hipSetDevice(s->ctx->device);
  if (s->md.on && s->md.forces_valid) reduce_energies(s, true);
  HIPCHK(hipStreamSynchronize(s->ctx->stream));
  HIPCHK(hipStreamSynchronize(s->ctx->stream2));
  {
    RtLock lk(g_rt_mu);
    drop_graphs(s);
  }
  if (s->mixed)
    run_pair_phase<true>(s, false, -1);
  else
    run_pair_phase<false>(s, false, -1);
  // the runs follow the schedule and the grid: cut the current list again
  // (the next MD step may use it without a rebuild)
  if (s->list_valid) {
    make_runs(s, s->ctx->stream);
    HIPCHK(hipStreamSynchronize(s->ctx->stream));
  }
  return s->pme_on ? fft_blocking(s) : PMX_OK;
}

int pmx_sys_stage_times(const pmx_sys *sys, float *ms) {
  if (!sys || !ms) return PMX_ERR_ARG;
  for (int k = 0; k < kStages; ++k) ms[k] = sys->s.stage_ms[k];
  return PMX_OK;
}

// ---------------------------------------------------------------------------
// Device-resident MD

int pmx_md_init(pmx_sys *sys, const pmx_md_desc *d) {
  if (!sys || !d) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  hipSetDevice(s->ctx->device);
  if (d->nbonds < 0 || d->nangles < 0 || !d->mass || !(d->timestep_fs > 0) || d->skin < 0 || d->skin > 4.0 ||
      (d->nbonds > 0 && (!d->bonds || !d->bond_par)) || (d->nangles > 0 && (!d->angles || !d->angle_par)))
    return fail(s->ctx, PMX_ERR_ARG, "bad MD descriptor");
  if ((d->integrator != PMX_MD_LEAPFROG && d->integrator != PMX_MD_LANGEVIN) ||
      (d->integrator == PMX_MD_LANGEVIN && (!(d->temperature >= 0) || !(d->gamma >= 0))))
    return fail(s->ctx, PMX_ERR_ARG, "bad integrator parameters");
  for (int i = 0; i < s->n; ++i)
    if (!(d->mass[i] > 0)) return fail(s->ctx, PMX_ERR_ARG, "masses must be > 0");
  for (int b = 0; b < 2 * d->nbonds; ++b)
    if (d->bonds[b] < 0 || d->bonds[b] >= s->n) return fail(s->ctx, PMX_ERR_ARG, "bond atom out of range");
  for (int a = 0; a < 3 * d->nangles; ++a)
    if (d->angles[a] < 0 || d->angles[a] >= s->n) return fail(s->ctx, PMX_ERR_ARG, "angle atom out of range");
  double rcmax = std::max(s->pp.has_lj ? s->d.lj_rc : 0.0, s->d.coul_kind ? s->d.coul_rc : 0.0);
  for (int k = 0; k < 3; ++k)
    if (rcmax + d->skin > 0.5 * s->box.L[k])
      return fail(s->ctx, PMX_ERR_UNSUPPORTED, "cutoff + skin larger than half the box");
  Sys::Md &m = s->md;
  {
    RtLock lk(g_rt_mu);
    drop_graphs(s);
  }
  m.on = true;
  m.graphs = d->graphs != 0;
  m.nb = d->nbonds;
  m.na = d->nangles;
  m.h = d->timestep_fs * kInvTimeFactor;
  m.skin = d->skin;
  m.chunk = 16;
  m.steps = m.rebuilds = m.rollbacks = 0;
  m.forces_valid = false;
  m.integrator = d->integrator;
  m.seed = d->seed;
  if (d->integrator == PMX_MD_LANGEVIN) {
    // LangevinLeapfrogIntegrator.cpp:28 (gamma per internal time unit) and
    // :46-51; gamma = 0 takes the limits (plain leapfrog half kick, no noise)
    const double g = d->gamma / (1000.0 * kInvTimeFactor), dt = m.h;
    m.vdt = std::exp(-0.5 * g * dt);
    m.fdt = g > 0 ? (1.0 - std::exp(-0.5 * g * dt)) / g : 0.5 * dt;
    m.ndt = g > 0 ? std::sqrt((1.0 - std::exp(-g * dt)) / (2.0 * g)) : 0.0;
    m.fc = 2.0 * kBoltzmann * d->temperature * g;
  }
  const size_t N = s->n;
  // bonds and angles by atom, each listed for every atom it acts on
  std::vector<int2> mp(N + 1, make_int2(0, 0));
  for (int i = 0; i < 2 * m.nb; ++i) ++mp[d->bonds[i] + 1].x;
  for (int i = 0; i < 3 * m.na; ++i) ++mp[d->angles[i] + 1].y;
  for (size_t i = 0; i < N; ++i) mp[i + 1] = make_int2(mp[i + 1].x + mp[i].x, mp[i + 1].y + mp[i].y);
  std::vector<int> b(2 * (size_t)m.nb);
  std::vector<double2> bp(2 * (size_t)m.nb);
  std::vector<int4> a(3 * (size_t)m.na);
  std::vector<double2> ap(3 * (size_t)m.na);
  std::vector<int2> at(mp.begin(), mp.end() - 1);
  for (int i = 0; i < m.nb; ++i)
    for (int k = 0; k < 2; ++k) {
      const int t = at[d->bonds[2 * i + k]].x++;
      b[t] = d->bonds[2 * i + 1 - k];
      bp[t] = make_double2(d->bond_par[2 * i], d->bond_par[2 * i + 1]);
    }
  for (int i = 0; i < m.na; ++i)
    for (int k = 0; k < 3; ++k) {
      const int t = at[d->angles[3 * i + k]].y++;
      a[t] = make_int4(d->angles[3 * i], d->angles[3 * i + 1], d->angles[3 * i + 2], k);
      ap[t] = make_double2(d->angle_par[2 * i], d->angle_par[2 * i + 1]);
    }
  std::vector<double> minv(N);
  for (size_t i = 0; i < N; ++i) minv[i] = 1.0 / d->mass[i];
  int rc;
  if ((rc = dalloc(s, m.mptr, 8 * mp.size())) || (rc = dalloc(s, m.bonds, 4 * b.size())) || (rc = dalloc(s, m.bpar, 16 * bp.size())) ||
      (rc = dalloc(s, m.angles, 16 * a.size())) || (rc = dalloc(s, m.apar, 16 * ap.size())) ||
      (rc = dalloc(s, m.minv, 8 * N)) || (rc = dalloc(s, m.v, 24 * N)) || (rc = dalloc(s, m.xbuild, 32 * (size_t)s->npad)) ||
      (rc = dalloc(s, m.xbak, 2 * 24 * N)) || (rc = dalloc(s, m.vbak, 2 * 24 * N)) ||
      (rc = dalloc(s, m.fbak, 2 * 24 * N)) || (rc = dalloc(s, m.dmax, 4 * 2 * kMaxChunk)) ||
      (rc = dalloc(s, m.step_dev, 8)) || (rc = dalloc(s, m.bond_e, 16 * (size_t)s->term_blocks)) ||
      (rc = dalloc(s, m.ke_e, 8 * (size_t)nblk(N, 256))) || (rc = dalloc(s, m.held, sizeof(PassResults))))
    return rc;
  if (!m.host) {
    RtLock lk(g_rt_mu);
    HIPCHK(hipHostMalloc((void **)&m.host, 4 * 2 * (kMaxChunk + 1), hipHostMallocDefault));
    for (auto &e : m.chunk_ev) HIPCHK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  }
  hipStream_t st = s->ctx->stream;
  HIPCHK(hipMemcpyAsync(m.mptr.p, mp.data(), 8 * mp.size(), hipMemcpyHostToDevice, st));
  if (m.nb) HIPCHK(hipMemcpyAsync(m.bonds.p, b.data(), 4 * b.size(), hipMemcpyHostToDevice, st));
  if (m.nb) HIPCHK(hipMemcpyAsync(m.bpar.p, bp.data(), 16 * bp.size(), hipMemcpyHostToDevice, st));
  if (m.na) HIPCHK(hipMemcpyAsync(m.angles.p, a.data(), 16 * a.size(), hipMemcpyHostToDevice, st));
  if (m.na) HIPCHK(hipMemcpyAsync(m.apar.p, ap.data(), 16 * ap.size(), hipMemcpyHostToDevice, st));
  HIPCHK(hipMemcpyAsync(m.minv.p, minv.data(), 8 * N, hipMemcpyHostToDevice, st));
  HIPCHK(hipStreamSynchronize(st));
  // the pair-list radius includes the skin
  s->cached = false;
  return setup(s);
}

int pmx_md_set_state(pmx_sys *sys, const double *x, const double *v) {
  if (!sys || !x || !v) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  if (!s->md.on) return fail(s->ctx, PMX_ERR_ARG, "pmx_md_init first");
  int rc = pmx_sys_set_positions(sys, x);
  if (rc) return rc;
  if ((rc = send(s, s->md.v.p, v, 24 * (size_t)s->n))) return rc;
  s->md.forces_valid = false;
  return PMX_OK;
}

namespace {

// StandardIntegrator::initializeForces: forces at the current positions with
// a freshly built list.  A list capacity overflow grows the buffers and
// recomputes, so the forces the first step kicks with are complete.
int md_ensure_forces(Sys *s) {
  Sys::Md &m = s->md;
  if (m.forces_valid) return PMX_OK;
  hipStream_t st = s->ctx->stream;
  for (int tries = 0;; ++tries) {
    int rc = rebuild(s, false, true);
    if (rc) return rc;
    ++m.rebuilds;
    if ((rc = forces(s, 0, false))) return rc;
    int ovf = 0;
    HIPCHK(hipMemcpyAsync(&ovf, s->overflow.p, 4, hipMemcpyDeviceToHost, st));
    HIPCHK(hipStreamSynchronize(st));
    if (!ovf) break;
    if (tries >= 6) return fail(s->ctx, PMX_ERR_OVERFLOW, "pair list capacity exceeded");
    if ((rc = grow_and_retry(s))) return rc;
  }
  m.forces_valid = true;
  return PMX_OK;
}

int md_check_overflow(Sys *s) {
  int ovf = 0;
  HIPCHK(hipMemcpyAsync(&ovf, s->overflow.p, 4, hipMemcpyDeviceToHost, s->ctx->stream));
  HIPCHK(hipStreamSynchronize(s->ctx->stream));
  if (ovf) return fail(s->ctx, PMX_ERR_OVERFLOW, "pair list capacity exceeded during MD");
  return PMX_OK;
}

// One leapfrog step: kick + drift (+ optional list rebuild at the new
// positions) + forces.  dslot: per-step displacement slot.
// The kicks before the drift of global step `step`: the first step of a run
// gets one half kick (kick = 0.5), later steps the previous step's closing
// half kick and their own opening one (kick = 1).  Langevin half kicks are
// numbered 2 step (opening) and 2 step + 1 (closing).
// With step_dev, `step` is relative to the step index stored there.
Kick make_kick(const Sys::Md &m, double kick, long long step, const unsigned long long *step_dev = nullptr) {
  Kick kk{};
  kk.h_kick = kick * m.h;
  kk.langevin = m.integrator == PMX_MD_LANGEVIN;
  kk.nhalf = kick == 0.5 ? 1 : 2;
  kk.half0 = (unsigned long long)(kick == 0.5 ? 2 * step : 2 * step - 1);
  kk.seed = m.seed;
  kk.vdt = m.vdt;
  kk.fdt = m.fdt;
  kk.ndt = m.ndt;
  kk.fc = m.fc;
  kk.step_dev = step_dev;
  return kk;
}

// kicked: the previous step's force pass already did this step's kick and
// drift; next (with next_dslot): fuse the following step's into this one's.
int md_step(Sys *s, double kick, long long step, bool rebuild_here, int dslot,
            const unsigned long long *step_dev = nullptr, bool kicked = false, const Kick *next = nullptr,
            int next_dslot = 0, const ChunkEnd &end = {}) {
  hipStream_t st = s->ctx->stream;
  Sys::Md &m = s->md;
  const bool timing = s->timing_active;
  const Kick kk = make_kick(m, kick, step, step_dev);
  // stage 0 of a timed MD step is integrate (+ sort when the list is rebuilt)
  timing_begin_call(s, timing);
  if (kicked)
    ;
  else if (s->mixed)
    hipLaunchKernelGGL(k_kick_drift<float>, dim3(nblk(s->npad, 256)), dim3(256), 0, st, s->npad, kk, m.h,
                       P<int>(s->permp), P<double>(s->fout), P<double>(m.v), P<double>(s->xorig),
                       P<double4>(m.xbuild), P<float4>(s->xs), P<double4>(s->xs64),
                       P<float4>(s->sorg), P<unsigned>(m.dmax) + dslot, s->pme, pme_slots<float>(s));
  else
    hipLaunchKernelGGL(k_kick_drift<double>, dim3(nblk(s->npad, 256)), dim3(256), 0, st, s->npad, kk, m.h,
                       P<int>(s->permp), P<double>(s->fout), P<double>(m.v), P<double>(s->xorig),
                       P<double4>(m.xbuild), P<double4>(s->xs), P<double4>(s->xs64),
                       P<float4>(s->sorg), P<unsigned>(m.dmax) + dslot, s->pme, pme_slots<double>(s));
  if (rebuild_here) {
    int rc = rebuild(s, timing, false);
    if (rc) return rc;
  } else if (timing) {
    hipEventRecord(s->ev[1], st);
    hipEventRecord(s->ev[2], st);
  }
  return forces(s, timing ? PMX_EVAL_TIMING : 0u, false, next, next ? P<unsigned>(m.dmax) + next_dslot : nullptr,
                end);
}

// A chunk of K steps from the committed state: its state is backed up in
// slot `slot`, step 0 rebuilds the list, and the last pass writes the per-step
// displacements and the overflow flag to the slot's pinned host record, after
// which the slot's event fires.
struct Chunk {
  int K;
  long long step0;
  bool first;
  int slot;
};

// The work of a chunk.  rel: step indices relative to *step_dev (capture).
int chunk_body(Sys *s, const Chunk &c, bool rel) {
  Sys::Md &m = s->md;
  hipStream_t st = s->ctx->stream;
  const size_t n = s->n, off = c.slot * 3 * n;
  // backups of the committed state, cleared overflow flags and displacement
  // record, in one launch
  const long long m3 = 3ll * (long long)n;
  hipLaunchKernelGGL(k_chunk_begin, dim3(nblk(std::max<long long>(m3, kMaxChunk), 256)), dim3(256), 0, st, m3,
                     P<double>(s->xorig), P<double>(m.v), P<double>(s->fout), P<double>(m.xbak) + off,
                     P<double>(m.vbak) + off, P<double>(m.fbak) + off, P<int>(s->overflow),
                     P<unsigned>(m.dmax) + c.slot * kMaxChunk, kMaxChunk);
  const unsigned long long *sd = rel ? P<unsigned long long>(m.step_dev) : nullptr;
  // inside the chunk each force pass ends with the next step's kick and
  // drift (one launch instead of two); timed steps keep them apart
  const bool fuse = !s->timing_active;
  unsigned *const h = m.host + c.slot * (kMaxChunk + 1);
  const ChunkEnd end{P<unsigned>(m.dmax) + c.slot * kMaxChunk, c.K, P<int>(s->overflow), h, h + kMaxChunk};
  for (int k = 0; k < c.K; ++k) {
    Kick nk{};
    const bool nx = fuse && k + 1 < c.K;
    if (nx) nk = make_kick(m, 1.0, rel ? k + 1 : c.step0 + k + 1, sd);
    int rc = md_step(s, (c.first && k == 0) ? 0.5 : 1.0, rel ? k : c.step0 + k, k == 0 || m.skin == 0.0,
                     c.slot * kMaxChunk + k, sd, fuse && k > 0, nx ? &nk : nullptr, c.slot * kMaxChunk + k + 1,
                     k + 1 < c.K ? ChunkEnd{} : end);
    if (rc) return rc;
  }
  return PMX_OK;
}

constexpr size_t kMaxGraphs = 64;

// Queues a chunk: replays its captured graph (capturing it on first use), or
// launches its kernels one by one when graphs are off or stage timing is on.
int enqueue_chunk(Sys *s, const Chunk &c) {
  Sys::Md &m = s->md;
  hipStream_t st = s->ctx->stream;
  hipGraphExec_t x = nullptr;
  // only chunks whose length is a power of two are captured (the others are
  // launched kernel by kernel), so a system holds at most 2 x 2 x 8 graphs
  if (m.graphs && !s->timing_active && (c.K & (c.K - 1)) == 0) {
    const long long key = ((long long)c.K << 2) | ((long long)c.first << 1) | c.slot;
    auto it = m.gexec.find(key);
    if (it != m.gexec.end()) {
      x = it->second;
    } else {
      RtLock lk(g_rt_mu);
      if (m.gexec.size() >= kMaxGraphs) {
        // a launched graph may still run: wait before destroying
        HIPCHK(hipStreamSynchronize(st));
        drop_graphs(s);
      }
      hipGraph_t g = nullptr;
      bool ok = hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal) == hipSuccess;
      if (ok) {
        const int rc = chunk_body(s, c, true);
        ok = hipStreamEndCapture(st, &g) == hipSuccess && rc == PMX_OK && g;
      }
      if (ok) ok = hipGraphInstantiate(&x, g, nullptr, nullptr, 0) == hipSuccess;
      if (g) hipGraphDestroy(g);
      if (ok) {
        m.gexec.emplace(key, x);
      } else {
        // nothing captured runs: take this system off graphs and launch the
        // chunk's kernels one by one instead
        x = nullptr;
        m.graphs = false;
        (void)hipGetLastError();
      }
    }
  }
  s->staged = false;  // a replay runs no host code of the passes in it
  s->energies_at = Sys::kInPartials;
  if (x) {
    hipLaunchKernelGGL(k_set_u64, dim3(1), dim3(1), 0, st, P<unsigned long long>(m.step_dev),
                       (unsigned long long)c.step0);
    HIPCHK(hipGraphLaunch(x, st));
  } else if (int rc = chunk_body(s, c, false)) {
    return rc;
  }
  HIPCHK(hipEventRecord(m.chunk_ev[c.slot], st));
  return PMX_OK;
}

// Waits for everything queued (a speculative chunk included), then restores
// the state backed up in slot `slot`.
int restore_chunk(Sys *s, int slot) {
  Sys::Md &m = s->md;
  hipStream_t st = s->ctx->stream;
  HIPCHK(hipStreamSynchronize(st));
  const size_t n = s->n, off = slot * 3 * n;
  HIPCHK(hipMemcpyAsync(s->xorig.p, P<double>(m.xbak) + off, 24 * n, hipMemcpyDeviceToDevice, st));
  HIPCHK(hipMemcpyAsync(m.v.p, P<double>(m.vbak) + off, 24 * n, hipMemcpyDeviceToDevice, st));
  HIPCHK(hipMemcpyAsync(s->fout.p, P<double>(m.fbak) + off, 24 * n, hipMemcpyDeviceToDevice, st));
  return PMX_OK;
}

// Length of the next chunk from the largest squared displacement d2 that
// the last chunk reached at step k after its list build.  Displacement is
// taken to grow linearly with time (the fastest atoms move ballistically
// over a few steps; diffusive motion grows slower, so the estimate errs
// short): the list stays valid up to step L = k sqrt(lim2 / d2).  The chunk
// ends at 80 % of L, since a chunk that outlives its list is rolled back and
// the chunk queued behind it discarded, and grows at most 2x per chunk.
int next_chunk(int k, float d2, float lim2, int cur) {
  const int grow = std::min(kMaxChunk, 2 * std::max(1, cur));
  if (!(d2 > 0.f)) return grow;
  const double L = k * std::sqrt((double)lim2 / (double)d2);
  return std::max(1, std::min(grow, (int)std::floor(0.8 * L) + 1));
}

// Progress of one pmx_md_run on one system (see md_advance).
struct MdRun {
  int nsteps = 0;
  int done = 0;     // committed steps of this run
  int planned = 0;  // committed + queued
  int next_slot = 0;
  int overflow_retries = 0;
  std::deque<Chunk> inflight;
  bool finished = false;
};

int md_begin(Sys *s, MdRun &r, int nsteps) {
  Sys::Md &m = s->md;
  if (!m.on || !s->have_positions) return fail(s->ctx, PMX_ERR_ARG, "pmx_md_init and pmx_md_set_state first");
  r = MdRun{};
  r.nsteps = nsteps;
  hipSetDevice(s->ctx->device);
  if (nsteps == 0) {
    r.finished = true;
    return PMX_OK;
  }
  return md_ensure_forces(s);
}

// The steps run in chunks that each start with a list rebuild.  Two chunks
// are in flight: while the device runs chunk c + 1 (queued on the assumption
// that chunk c keeps every atom within half the skin of its build position),
// the host reads chunk c's displacements.  If chunk c crossed the limit at
// step b, the speculative chunk is discarded, the state of chunk c's start is
// restored and its first b steps (which used a valid list) are replayed; the
// trajectory is the same as with a rebuild at every step.  The device never
// waits for the host between chunks.
//
// One call queues chunks up to two in flight, then settles the oldest one if
// it has completed (waiting for it when `block`).  *progressed tells whether
// anything was queued or settled.  After the last step the closing half kick
// is queued and r.finished is set.
int md_advance(Sys *s, MdRun &r, bool block, bool *progressed) {
  Sys::Md &m = s->md;
  hipStream_t st = s->ctx->stream;
  const int n = s->n;
  const float lim2 = (float)(0.25 * m.skin * m.skin);
  *progressed = false;
  if (r.finished) return PMX_OK;
  while (r.inflight.size() < 2 && r.planned < r.nsteps) {
    Chunk c{std::min(m.chunk, r.nsteps - r.planned), m.steps + (r.planned - r.done), r.planned == 0, r.next_slot};
    if (int rc = enqueue_chunk(s, c)) return rc;
    r.inflight.push_back(c);
    r.planned += c.K;
    r.next_slot ^= 1;
    *progressed = true;
  }
  if (!r.inflight.empty()) {
    const Chunk c = r.inflight.front();
    if (block) {
      HIPCHK(hipEventSynchronize(m.chunk_ev[c.slot]));
    } else {
      const hipError_t q = hipEventQuery(m.chunk_ev[c.slot]);
      if (q == hipErrorNotReady) return PMX_OK;
      if (q != hipSuccess) return fail(s->ctx, PMX_ERR_HIP, hipGetErrorString(q));
    }
    r.inflight.pop_front();
    *progressed = true;
    const unsigned *h = m.host + c.slot * (kMaxChunk + 1);
    if (h[kMaxChunk]) {
      // a list or mask capacity was exceeded: grow, roll back, replay
      if (++r.overflow_retries > 6) return fail(s->ctx, PMX_ERR_OVERFLOW, "pair list capacity exceeded during MD");
      if (int rc = restore_chunk(s, c.slot)) return rc;
      if (int rc = grow_and_retry(s)) return rc;
      r.inflight.clear();
      r.planned = r.done;
      return PMX_OK;
    }
    int bad = -1;
    float worst = 0.f;
    for (int k = 1; k < c.K; ++k) {
      const float d = __builtin_bit_cast(float, h[k]);
      worst = std::max(worst, d);
      if (m.skin > 0 && d > lim2) {
        bad = k;
        break;
      }
    }
    if (bad < 0) {
      r.done += c.K;
      m.steps += c.K;
      m.rebuilds += m.skin > 0 ? 1 : c.K;
      if (m.skin > 0 && c.K > 1) m.chunk = next_chunk(c.K - 1, worst, lim2, m.chunk);
    } else {
      // roll back to the chunk's start and replay the steps that used a
      // valid list (deterministic: the replay reproduces them exactly)
      ++m.rollbacks;
      if (int rc = restore_chunk(s, c.slot)) return rc;
      r.inflight.clear();
      for (int k = 0; k < bad; ++k) {
        int rc = md_step(s, (c.first && k == 0) ? 0.5 : 1.0, c.step0 + k, k == 0, k);
        if (rc) return rc;
      }
      r.done += bad;
      m.steps += bad;
      m.rebuilds += 1;
      r.planned = r.done;
      m.chunk = next_chunk(bad, worst, lim2, m.chunk);
    }
  }
  if (r.done == r.nsteps && r.inflight.empty()) {
    // closing half kick of the last step (global index m.steps - 1)
    Kick kk = make_kick(m, 0.5, m.steps);
    kk.half0 = (unsigned long long)(2 * m.steps - 1);
    hipLaunchKernelGGL(k_half_kick, dim3(nblk(n, 256)), dim3(256), 0, st, n, kk, P<double>(s->fout),
                       P<double>(m.minv), P<double>(m.v));
    r.finished = true;
  }
  return PMX_OK;
}

int md_end(Sys *s) {
  HIPCHK(hipStreamSynchronize(s->ctx->stream));
  return md_check_overflow(s);
}

// ---- batched MD: every kernel of a step launched once for many systems ----
// (C++ linkage for the templates inside the C ABI's extern "C" block)
extern "C++" {

#define BHIPCHK(expr)                                                                                   \
  do {                                                                                                  \
    hipError_t _e = (expr);                                                                             \
    if (_e != hipSuccess) return fail(b.ctx, PMX_ERR_HIP, std::string(#expr ": ") + hipGetErrorString(_e)); \
  } while (0)

// A device block of the batch (from the block cache, given back at the end).
struct BatchBuf {
  int device = 0;
  void *p = nullptr;
  size_t cls = 0;
  BatchBuf() = default;
  BatchBuf(const BatchBuf &) = delete;
  BatchBuf &operator=(const BatchBuf &) = delete;
  ~BatchBuf() { release(); }
  void release() {
    if (!p) return;
    RtLock lk(g_rt_mu);
    block_put(device, p, cls);
    p = nullptr;
  }
  bool get(int dev, size_t bytes) {
    release();
    device = dev;
    cls = size_class(std::max<size_t>(bytes, 8));
    RtLock lk(g_rt_mu);
    p = block_get(dev, cls);
    return p != nullptr;
  }
};

// One batched launch: the argument table, each system's first block and the
// system of each block.
struct BatchLaunch {
  size_t tab_at = 0, first_at = 0, b2s_at = 0;  // in the batch's tables
  const void *tab = nullptr;
  const int *first = nullptr, *b2s = nullptr;
  unsigned blocks = 0;
  size_t lds = 0;
  int threads = 0;  // block size (0: the op's kBlock)
};

struct Batch {
  pmx_ctx *ctx = nullptr;
  std::vector<Sys *> sys;
  int nsys = 0;
  bool results = false;       // a force pass alone: its results go to the systems' stages with it
  bool first_forces = false;  // a force pass of a run's new systems: no energies, no results
  std::vector<Sys *> fresh;   // MD: systems that lack the forces at their positions
  BatchLaunch bin, scan, scatter, split, list, runs;
  BatchLaunch kick, spread, pair, yfwd, xconv, yinv, plane, gather, fixups, ukd, unsort, begin, half;
  BatchLaunch energy, out;
  BatchLaunch spreadL, yfwdL, xconvL, yinvL, gatherL;  // the systems with axes beyond kFftMax
  BatchBuf tables, bsys, need, base, flags, rebuilds;
  std::vector<unsigned char> image;    // the tables of every launch, uploaded in one copy
  std::vector<BatchLaunch *> launches;
  // slices of the context's pinned staging, and its events
  BatchSys *bsys_h = nullptr;
  unsigned long long *base_h = nullptr;
  int *flags_h = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
};

// The batch's device buffers, and its slices of the context's pinned staging
// (a batch that comes before another of the context shares them).
int batch_buffers(Batch &b) {
  pmx_ctx *ctx = b.ctx;
  const int dev = ctx->device, nsys = b.nsys;
  if (!b.bsys.get(dev, sizeof(BatchSys) * nsys) || !b.need.get(dev, nsys) || !b.base.get(dev, 8 * (size_t)nsys) ||
      !b.flags.get(dev, 4 * (size_t)nsys) || !b.rebuilds.get(dev, 8 * (size_t)nsys))
    return fail(ctx, PMX_ERR_OOM, "batch buffers");
  {
    RtLock lk(g_rt_mu);
    const size_t need = (sizeof(BatchSys) + 16) * (size_t)nsys;
    if (ctx->batch_host_bytes < need) {
      if (ctx->batch_host) hipHostFree(ctx->batch_host);
      ctx->batch_host = nullptr;
      ctx->batch_host_bytes = 0;
      if (hipHostMalloc(&ctx->batch_host, need, hipHostMallocDefault) != hipSuccess)
        return fail(ctx, PMX_ERR_HIP, "batch host buffers");
      ctx->batch_host_bytes = need;
    }
    if ((!ctx->batch_fork &&
         hipEventCreateWithFlags(&ctx->batch_fork, hipEventDisableTiming | hipEventDisableSystemFence) != hipSuccess) ||
        (!ctx->batch_join &&
         hipEventCreateWithFlags(&ctx->batch_join, hipEventDisableTiming | hipEventDisableSystemFence) != hipSuccess))
      return fail(ctx, PMX_ERR_HIP, "batch events");
  }
  b.bsys_h = static_cast<BatchSys *>(ctx->batch_host);
  b.base_h = reinterpret_cast<unsigned long long *>(b.bsys_h + nsys);
  b.flags_h = reinterpret_cast<int *>(b.base_h + nsys);
  b.fork = ctx->batch_fork;
  b.join = ctx->batch_join;
  return PMX_OK;
}

// Adds the table of one batched launch (args[s], nblocks[s] blocks of system
// s; dynamic LDS `lds`) to the batch's tables.
template <class Op>
int batch_table(Batch &b, BatchLaunch &L, const std::vector<typename Op::Args> &args,
                const std::vector<int> &nblocks, size_t lds = 0, int threads = 0) {
  L.lds = lds;
  L.threads = threads ? threads : Op::kBlock;
  auto room = [&](size_t bytes) {
    const size_t at = (b.image.size() + 255) / 256 * 256;
    b.image.resize(at + std::max<size_t>(bytes, 4));
    return at;
  };
  L.tab_at = room(sizeof(typename Op::Args) * args.size());
  std::memcpy(b.image.data() + L.tab_at, args.data(), sizeof(typename Op::Args) * args.size());
  L.first_at = room(4 * ((size_t)b.nsys + 1));
  int *first = reinterpret_cast<int *>(b.image.data() + L.first_at);
  first[0] = 0;
  for (int i = 0; i < b.nsys; ++i) first[i + 1] = first[i] + nblocks[i];
  L.blocks = (unsigned)first[b.nsys];
  L.b2s_at = room(4 * (size_t)L.blocks);
  int *b2s = reinterpret_cast<int *>(b.image.data() + L.b2s_at);
  for (int i = 0; i < b.nsys; ++i) b2s = std::fill_n(b2s, nblocks[i], i);
  b.launches.push_back(&L);
  return PMX_OK;
}

// Uploads the tables (nothing of an earlier upload may be in use).
int batch_upload(Batch &b) {
  if (!b.tables.get(b.ctx->device, b.image.size())) return fail(b.ctx, PMX_ERR_OOM, "batch tables");
  {
    RtLock lk(g_rt_mu);
    BHIPCHK(hipMemcpy(b.tables.p, b.image.data(), b.image.size(), hipMemcpyHostToDevice));
  }
  const unsigned char *d = static_cast<const unsigned char *>(b.tables.p);
  for (BatchLaunch *L : b.launches) {
    L->tab = d + L->tab_at;
    L->first = reinterpret_cast<const int *>(d + L->first_at);
    L->b2s = reinterpret_cast<const int *>(d + L->b2s_at);
  }
  b.image.clear();
  b.launches.clear();
  return PMX_OK;
}

template <class Op>
void batch_go(const BatchLaunch &L, hipStream_t st, const BatchStep &bs) {
  if (!L.blocks) return;
  hipLaunchKernelGGL(k_batch<Op>, dim3(L.blocks), dim3(L.threads), L.lds, st,
                     static_cast<const typename Op::Args *>(L.tab), L.b2s, L.first, bs);
}

// The batch's kernel case: the pair kernel's cases of run_pair_phase for PME
// systems (0: LJ C2 + Coulomb cutoff switch, 1: no LJ, 2: any switches, 3:
// LJ table beyond the kernel's LDS).
int batch_case(const Sys *s) {
  const int lj = s->d.lj_switch, cs = s->d.coul_switch;
  if (s->d.ntypes > kMaxTypes && lj != SW_NONE) return 3;
  if (lj == SW_C2 && cs == SW_CUTOFF) return 0;
  return lj == SW_NONE ? 1 : 2;
}

template <bool MIXED, int C, int LJ, int CS, bool BIGLJ, int ORDER>
using PairOp = OpPair<MIXED, C, LJ, CS, BIGLJ>;

// Fills every table of the batch from its systems (again after a system's
// buffers grow).
template <bool MIXED, int C, int LJ, int CS, bool BIGLJ, int ORDER>
int batch_tables(Batch &b) {
  using R = typename std::conditional<MIXED, float, double>::type;
  using R4 = typename Real4<R>::type;
  using T = R;
  using Acc = typename AccT<MIXED>::type;
  const int ns = b.nsys;
  const size_t cx = sizeof(Cx<T>);
  std::vector<int> nb(ns);
  int rc;
  {
    std::vector<OpBin::Args> args_bin(ns);
    std::vector<OpScanColumns::Args> args_scan(ns);
    std::vector<OpScatter::Args> args_scatter(ns);
    std::vector<typename OpSplitFill<R>::Args> args_split(ns);
    std::vector<OpBuildList::Args> args_list(ns);
    std::vector<OpRuns::Args> args_runs(ns);
    size_t list_lds = 0;
    for (int i = 0; i < ns; ++i) {
      Sys *s = b.sys[i];
      args_bin[i] = {s->n, P<double>(s->xorig), s->bin, P<uint32_t>(s->key), P<uint32_t>(s->hist),
                     P<double>(s->xwrap), P<int>(s->refcell)};
      args_scan[i] = {P<uint32_t>(s->hist), P<uint32_t>(s->start), P<uint32_t>(s->cursor), (int)s->nbins, s->ncols,
                      s->bin.nzb, s->n, s->nsuper, P<int2>(s->sc_info), P<int>(s->sc_col), P<int>(s->colsc)};
      args_scatter[i] = {s->n, P<uint32_t>(s->key), P<uint32_t>(s->cursor), P<int>(s->perm)};
      auto &sp = args_split[i];
      sp.nsuper = s->nsuper;
      sp.sc_info = P<int2>(s->sc_info);
      sp.sb = sorted_bins(s);
      sp.xwrap = P<double>(s->xwrap);
      sp.q = P<double>(s->q_d);
      sp.permp = P<int>(s->permp);
      sp.slot = P<int>(s->slot);
      sp.type = P<int>(s->type_d);
      sp.xs = P<R4>(s->xs);
      sp.xs64 = P<double4>(s->xs64);
      sp.ts = P<int>(s->ts);
      sp.xorig = P<double>(s->xorig);
      sp.minv = P<double>(s->md.minv);
      sp.xbuild = P<double4>(s->md.xbuild);
      sp.sorg = P<float4>(s->sorg);
      sp.ctr = P<float4>(s->ctr);
      sp.half = P<float4>(s->half);
      sp.sctr = P<float4>(s->sctr);
      sp.shalf = P<float4>(s->shalf);
      sp.nmaskwork = P<int>(s->nmaskwork);
      sp.qpair = s->qpair;
      sp.pme = s->pme;
      sp.rec = pme_slots<R>(s);
      args_list[i] = {s->lp, P<int>(s->sc_col), P<int>(s->colsc), P<float4>(s->sctr), P<float4>(s->shalf),
                      P<float4>(s->ctr), P<float4>(s->half), P<int4>(s->entries), P<int>(s->count),
                      P<int>(s->ecost), P<int>(s->lcost), mask_args(s), P<int>(s->nmaskwork), P<int>(s->overflow)};
      list_lds = std::max(list_lds, list_lds_bytes(s->cap));
      args_runs[i] = {s->nsuper, s->cap, P<int>(s->count), P<int>(s->lcost), P<int>(s->ecost),
                      P<int2>(s->runs), P<int>(s->ntiles)};
    }
    for (int i = 0; i < ns; ++i) nb[i] = (int)nblk(b.sys[i]->n, 256);
    if ((rc = batch_table<OpBin>(b, b.bin, args_bin, nb, 0))) return rc;
    if ((rc = batch_table<OpScatter>(b, b.scatter, args_scatter, nb, 0))) return rc;
    for (int i = 0; i < ns; ++i) nb[i] = 1;
    if ((rc = batch_table<OpScanColumns>(b, b.scan, args_scan, nb, 0))) return rc;
    for (int i = 0; i < ns; ++i) nb[i] = (int)runs_blocks(b.sys[i]);
    if ((rc = batch_table<OpRuns>(b, b.runs, args_runs, nb, 0))) return rc;
    for (int i = 0; i < ns; ++i) nb[i] = (int)nblk((long long)b.sys[i]->nsuper * 64, 256);
    if ((rc = batch_table<OpSplitFill<R>>(b, b.split, args_split, nb, 0))) return rc;
    for (int i = 0; i < ns; ++i) nb[i] = b.sys[i]->nsuper;
    if ((rc = batch_table<OpBuildList>(b, b.list, args_list, nb, list_lds))) return rc;
  }
  {
    std::vector<typename OpKickDrift<R>::Args> args_kick(ns);
    std::vector<typename OpPmeSpreadZ<MIXED, ORDER>::Args> args_spread(ns);
    std::vector<typename PairOp<MIXED, C, LJ, CS, BIGLJ, ORDER>::Args> args_pair(ns);
    std::vector<typename OpFftY<T>::Args> args_yfwd(ns), args_yinv(ns);
    std::vector<typename OpFftXConv<T>::Args> args_xconv(ns);
    std::vector<typename OpFftPlane<T>::Args> args_plane(ns);
    std::vector<typename OpPmeZGather<MIXED, ORDER>::Args> args_gather(ns);
    std::vector<FixupArgs<MIXED>> args_fixups(ns);
    std::vector<typename OpUnsortKickDrift<MIXED, R>::Args> args_ukd(ns);
    std::vector<typename OpUnsortForces<MIXED>::Args> args_unsort(ns);
    std::vector<OpChunkBegin::Args> args_begin(ns);
    std::vector<OpHalfKick::Args> args_half(ns);
    std::vector<typename OpUnsortEnergy<MIXED>::Args> args_energy(ns);
    std::vector<OutArgs> args_out(ns, OutArgs{});
    std::vector<int> nout(ns, 0);
    std::vector<int> nfix(ns);
    long long natoms = 0;
    // [1]: the LONG forms of the passes
    size_t lds_z[2] = {0, 0}, lds_g[2] = {0, 0}, lds_y[2] = {0, 0}, lds_x[2] = {0, 0}, lds_p = 0;
    int thr_z[2] = {256, 256}, thr_g[2] = {256, 256}, thr_y[2] = {256, 256}, thr_x[2] = {256, 256}, thr_p = 256;
    for (int i = 0; i < ns; ++i) {
      Sys *s = b.sys[i];
      Sys::Md &m = s->md;
      natoms += s->n;
      const Kick kk = make_kick(m, 1.0, 0, P<unsigned long long>(m.step_dev));
      Acc *facc = P<Acc>(s->facc);
      args_kick[i] = {s->npad, kk, m.h, P<int>(s->permp), P<double>(s->fout), P<double4>(m.xbuild),
                      P<double>(m.v), P<double>(s->xorig), P<R4>(s->xs), P<double4>(s->xs64), P<float4>(s->sorg),
                      P<unsigned>(m.dmax), s->pme, pme_slots<R>(s)};
      args_spread[i] = {s->pme, s->plz, P<int2>(s->tcol), P<int>(s->colsc), P<R4>(s->pmw), P<int2>(s->pmb),
                        P<Cx<T>>(s->twz), P<Cx<T>>(s->spec)};
      const R4 *ljt = MIXED ? reinterpret_cast<const R4 *>(s->ljt32.p) : reinterpret_cast<const R4 *>(s->ljtab.p);
      args_pair[i] = {s->pp, P<int2>(s->runs), P<int>(s->ntiles), P<int>(s->count), P<int>(s->tilectr),
                      P<int4>(s->entries), s->cap, P<unsigned short>(s->masks), P<R4>(s->xs), P<float4>(s->sorg),
                      P<int>(s->ts), P<int>(s->permp), P<double>(s->ljtab), ljt, facc,
                      PairOut{P<double>(s->pair_e), P<long long>(s->npairs), P<unsigned long long>(s->hash),
                              P<int2>(s->border), P<int>(s->nborder), s->maxborder, P<int>(s->overflow),
                              P<unsigned long long>(s->border_acc)}};
      const PmeParams &pm = s->pme;
      args_yfwd[i] = {pm, s->ply, s->ylog, false, P<Cx<T>>(s->twy), P<Cx<T>>(s->spec)};
      args_xconv[i] = {pm, s->plx, s->xlog, s->thr_x, P<Cx<T>>(s->twx), P<T>(s->theta), P<Cx<T>>(s->spec),
                       P<double>(s->recip_e)};
      args_yinv[i] = {pm, s->ply, s->ylog, true, P<Cx<T>>(s->twy), P<Cx<T>>(s->spec)};
      args_plane[i] = {pm, s->ply, s->plx, s->thr_pb, P<Cx<T>>(s->twy), P<Cx<T>>(s->twx), P<T>(s->theta), P<Cx<T>>(s->spec),
                       P<double>(s->recip_e)};
      args_gather[i] = {s->pme_g, s->plz, P<int2>(s->tcol) + pm.ntx + pm.nty, P<int>(s->colsc), P<R4>(s->pmw), P<int2>(s->pmb),
                        P<Cx<T>>(s->twz), P<Cx<T>>(s->spec), facc};
      args_fixups[i] = fixup_args<MIXED>(s, false, true, true, &nfix[i]);
      args_ukd[i] = {s->npad, kk, m.h, P<int>(s->permp), facc, P<int>(s->tilectr), P<int>(s->nborder),
                     P<double4>(m.xbuild), P<double>(m.v), P<double>(s->xorig),
                     P<R4>(s->xs), P<double4>(s->xs64), P<float4>(s->sorg), P<unsigned>(m.dmax), pm, pme_slots<R>(s)};
      args_unsort[i] = {s->n, P<int>(s->slot), facc, P<double>(s->fout), P<int>(s->tilectr), P<int>(s->nborder)};
      args_begin[i] = {3ll * s->n, P<double>(s->xorig), P<double>(m.v), P<double>(s->fout), P<double>(m.xbak),
                       P<double>(m.vbak), P<double>(m.fbak), P<int>(s->overflow), P<unsigned>(m.dmax), kMaxChunk};
      args_half[i] = {s->n, kk, m.h, P<double>(s->fout), P<double>(m.minv), P<double>(m.v)};
      args_energy[i] = {s->n, P<int>(s->slot), facc, P<double>(s->fout), P<int>(s->tilectr), P<int>(s->nborder),
                        energy_args(s, false)};
      if (b.results && batch_stages(s)) {
        if ((rc = stage_get(s, 8 * (kResultWords + 3 * (size_t)s->n)))) return rc;
        OutList out(s->stage.p);
        out.add(s->eout.p, kResultWords);
        out.add(s->fout.p, 3 * (size_t)s->n);
        args_out[i] = out.a;
        nout[i] = (int)out.blocks();
      }
      // dynamic LDS and block size of each launch: the largest of the
      // systems it serves
      auto most = [](auto &v, auto w) { v = std::max(v, w); };
      const int zl = pm.nz > kFftMax, yl = pm.ny > kFftMax, xl = pm.nx > kFftMax;
      most(thr_z[zl], s->thr_z);
      most(thr_g[zl], s->thr_gb);
      most(lds_g[zl], s->lds_g);
      most(lds_z[zl], s->lds_z);
      if (s->fft_plane) {
        most(lds_p, s->lds_p);
        most(thr_p, s->thr_pb);
      } else {
        most(lds_y[yl], s->lds_y);
        most(lds_x[xl], s->lds_x);
        most(thr_y[yl], s->thr_y);
        most(thr_x[xl], s->thr_x);
      }
    }
    for (int i = 0; i < ns; ++i) nb[i] = (int)nblk(b.sys[i]->npad, 256);
    if ((rc = batch_table<OpKickDrift<R>>(b, b.kick, args_kick, nb, 0))) return rc;
    if ((rc = batch_table<OpUnsortKickDrift<MIXED, R>>(b, b.ukd, args_ukd, nb, 0))) return rc;
    // blocks(s) of the systems of one form of a pass, none of the others
    auto of = [&](bool form, auto is, auto blocks) -> const std::vector<int> & {
      for (int i = 0; i < ns; ++i) nb[i] = (is(b.sys[i]) == form) ? blocks(b.sys[i]) : 0;
      return nb;
    };
    auto zlong = [](const Sys *s) { return s->pme.nz > kFftMax; };
    auto spread_blocks = [](const Sys *s) { return s->pme.ntx * s->pme.nty; };
    auto gather_blocks = [](const Sys *s) { return s->pme_g.ntx * s->pme_g.nty; };
    if ((rc = batch_table<OpPmeSpreadZ<MIXED, ORDER>>(b, b.spread, args_spread, of(false, zlong, spread_blocks),
                                                      lds_z[0], thr_z[0])) ||
        (rc = batch_table<OpPmeZGather<MIXED, ORDER>>(b, b.gather, args_gather, of(false, zlong, gather_blocks),
                                                      lds_g[0], thr_g[0])))
      return rc;
    // pair-kernel blocks in proportion to the atoms (a run's share of a
    // system's waves changes no result), about the device's resident blocks
    // in all
    static const int fit =
        pair_blocks_per_cu(reinterpret_cast<const void *>(k_batch<PairOp<MIXED, C, LJ, CS, BIGLJ, ORDER>>));
    const double pair_blocks = (double)b.ctx->cus * pair_blocks_of(fit, kMinRuns);
    for (int i = 0; i < ns; ++i)
      nb[i] = std::max(1, (int)std::lround(pair_blocks * b.sys[i]->n / (double)natoms));
    if ((rc = batch_table<PairOp<MIXED, C, LJ, CS, BIGLJ, ORDER>>(b, b.pair, args_pair, nb, 0))) return rc;
    // systems with small planes take the one-launch plane pass, the others
    // the three line passes
    auto ylong = [](const Sys *s) { return s->pme.ny > kFftMax; };
    auto xlong = [](const Sys *s) { return s->pme.nx > kFftMax; };
    auto y_blocks = [](const Sys *s) {
      return s->fft_plane ? 0 : s->pme.nzh * ((s->pme.nx + (1 << s->ylog) - 1) >> s->ylog);
    };
    auto x_blocks = [](const Sys *s) { return s->fft_plane ? 0 : s->recip_blocks; };
    of(false, ylong, y_blocks);
    if ((rc = batch_table<OpFftY<T>>(b, b.yfwd, args_yfwd, nb, lds_y[0], thr_y[0])) ||
        (rc = batch_table<OpFftY<T>>(b, b.yinv, args_yinv, nb, lds_y[0], thr_y[0])) ||
        (rc = batch_table<OpFftXConv<T>>(b, b.xconv, args_xconv, of(false, xlong, x_blocks), lds_x[0], thr_x[0])))
      return rc;
    if (std::any_of(b.sys.begin(), b.sys.end(), [&](const Sys *s) { return xlong(s) || ylong(s) || zlong(s); })) {
      if ((rc = batch_table<OpPmeSpreadZLong<MIXED, ORDER>>(b, b.spreadL, args_spread, of(true, zlong, spread_blocks),
                                                            lds_z[1], thr_z[1])) ||
          (rc = batch_table<OpPmeZGatherLong<MIXED, ORDER>>(b, b.gatherL, args_gather, of(true, zlong, gather_blocks),
                                                            lds_g[1], thr_g[1])))
        return rc;
      of(true, ylong, y_blocks);
      if ((rc = batch_table<OpFftYLong<T>>(b, b.yfwdL, args_yfwd, nb, lds_y[1], thr_y[1])) ||
          (rc = batch_table<OpFftYLong<T>>(b, b.yinvL, args_yinv, nb, lds_y[1], thr_y[1])) ||
          (rc = batch_table<OpFftXConvLong<T>>(b, b.xconvL, args_xconv, of(true, xlong, x_blocks), lds_x[1], thr_x[1])))
        return rc;
    }
    for (int i = 0; i < ns; ++i) nb[i] = b.sys[i]->fft_plane ? b.sys[i]->pme.nzh : 0;
    if ((rc = batch_table<OpFftPlane<T>>(b, b.plane, args_plane, nb, lds_p, thr_p))) return rc;
    if ((rc = batch_table<OpFixups<MIXED, C, LJ, CS>>(b, b.fixups, args_fixups, nfix, 0))) return rc;
    for (int i = 0; i < ns; ++i) nb[i] = (int)nblk(b.sys[i]->n, 256);
    if ((rc = batch_table<OpUnsortForces<MIXED>>(b, b.unsort, args_unsort, nb, 0))) return rc;
    if ((rc = batch_table<OpHalfKick>(b, b.half, args_half, nb, 0))) return rc;
    for (int i = 0; i < ns; ++i) nb[i] = 1 + (int)nblk(b.sys[i]->n, kEndBlock);
    if ((rc = batch_table<OpUnsortEnergy<MIXED>>(b, b.energy, args_energy, nb, 0))) return rc;
    if ((rc = batch_table<OpOut>(b, b.out, args_out, nout, 0))) return rc;
    for (int i = 0; i < ns; ++i) nb[i] = (int)nblk(std::max<long long>(3ll * b.sys[i]->n, kMaxChunk), 256);
    if ((rc = batch_table<OpChunkBegin>(b, b.begin, args_begin, nb, 0))) return rc;
  }
  // per-system bookkeeping
  for (int i = 0; i < ns; ++i) {
    Sys *s = b.sys[i];
    b.bsys_h[i] = BatchSys{P<unsigned>(s->md.dmax), s->md.skin > 0 ? (float)(0.25 * s->md.skin * s->md.skin) : -1.f, 0,
                           P<unsigned long long>(s->md.step_dev), P<int>(s->overflow),
                           reinterpret_cast<long long *>(b.rebuilds.p) + i};
  }
  return batch_upload(b);
}

// Queues one chunk of K steps of every system of the batch (the first step
// of each system's run when `opening`), then the gathering of the overflow
// flags into b.flags_h.  Step 0 kicks and drifts in a launch of its own; every
// later step's kick and drift run in the previous step's last launch.
template <bool MIXED, int C, int LJ, int CS, bool BIGLJ, int ORDER>
int batch_chunk(Batch &b, int K, bool opening) {
  using R = typename std::conditional<MIXED, float, double>::type;
  using T = R;
  hipStream_t st = b.ctx->stream, st2 = b.ctx->stream2;
  const int ns = b.nsys;
  BHIPCHK(hipMemcpyAsync(b.bsys.p, b.bsys_h, sizeof(BatchSys) * ns, hipMemcpyHostToDevice, st));
  BHIPCHK(hipMemcpyAsync(b.base.p, b.base_h, 8 * (size_t)ns, hipMemcpyHostToDevice, st));
  const BatchSys *bs = reinterpret_cast<const BatchSys *>(b.bsys.p);
  unsigned char *need = reinterpret_cast<unsigned char *>(b.need.p);
  hipLaunchKernelGGL(k_batch_steps, dim3(nblk(ns, 256)), dim3(256), 0, st, ns, bs,
                     reinterpret_cast<const unsigned long long *>(b.base.p));
  const BatchStep b0{0, opening ? 1 : 0, need};
  batch_go<OpChunkBegin>(b.begin, st, b0);
  for (int k = 0; k < K; ++k) {
    const BatchStep bk{k, opening ? 1 : 0, need};
    if (k == 0) batch_go<OpKickDrift<R>>(b.kick, st, bk);
    hipLaunchKernelGGL(k_batch_need, dim3(nblk(ns, 256)), dim3(256), 0, st, ns, bs, k, need);
    batch_go<OpBin>(b.bin, st, bk);
    batch_go<OpScanColumns>(b.scan, st, bk);
    batch_go<OpScatter>(b.scatter, st, bk);
    batch_go<OpSplitFill<R>>(b.split, st, bk);
    batch_go<OpBuildList>(b.list, st, bk);
    batch_go<OpRuns>(b.runs, st, bk);
    // the spread has the device to itself (beside the pair kernel a CU has
    // room for one of its blocks at a time: 0.51 ms instead of 0.1 for 64
    // systems of 331,000 atoms); fork: the rest of the PME chain beside the
    // pair kernel
    batch_go<OpPmeSpreadZ<MIXED, ORDER>>(b.spread, st, bk);
    batch_go<OpPmeSpreadZLong<MIXED, ORDER>>(b.spreadL, st, bk);
    BHIPCHK(hipEventRecord(b.fork, st));
    BHIPCHK(hipStreamWaitEvent(st2, b.fork, 0));
    batch_go<PairOp<MIXED, C, LJ, CS, BIGLJ, ORDER>>(b.pair, st, bk);
    batch_go<OpFftPlane<T>>(b.plane, st2, bk);
    batch_go<OpFftY<T>>(b.yfwd, st2, bk);
    batch_go<OpFftYLong<T>>(b.yfwdL, st2, bk);
    batch_go<OpFftXConv<T>>(b.xconv, st2, bk);
    batch_go<OpFftXConvLong<T>>(b.xconvL, st2, bk);
    batch_go<OpFftY<T>>(b.yinv, st2, bk);
    batch_go<OpFftYLong<T>>(b.yinvL, st2, bk);
    batch_go<OpPmeZGather<MIXED, ORDER>>(b.gather, st2, bk);
    batch_go<OpPmeZGatherLong<MIXED, ORDER>>(b.gatherL, st2, bk);
    BHIPCHK(hipEventRecord(b.join, st2));
    // boundary pairs, exclusion correction and bonded terms after the pair
    // kernel, then the join
    batch_go<OpFixups<MIXED, C, LJ, CS>>(b.fixups, st, bk);
    BHIPCHK(hipStreamWaitEvent(st, b.join, 0));
    if (k + 1 < K)
      batch_go<OpUnsortKickDrift<MIXED, R>>(b.ukd, st, bk);
    else
      batch_go<OpUnsortForces<MIXED>>(b.unsort, st, bk);
  }
  hipLaunchKernelGGL(k_batch_flags, dim3(nblk(ns, 256)), dim3(256), 0, st, ns, bs,
                     reinterpret_cast<int *>(b.flags.p));
  BHIPCHK(hipMemcpyAsync(b.flags_h, b.flags.p, 4 * (size_t)ns, hipMemcpyDeviceToHost, st));
  BHIPCHK(hipGetLastError());
  return PMX_OK;
}

// One force pass of every system of the batch at its set positions (list
// rebuilt for all): the work of compute() for each, or of md_ensure_forces
// (first_forces), which leaves the last evaluation's energies.  Where a list
// outgrew its buffers they are grown and the batch computed again: a system
// computed alone would get another cut of its list, and in the mixed form
// other last bits than without the growth.
template <bool MIXED, int C, int LJ, int CS, bool BIGLJ, int ORDER>
int batch_forces(Batch &b) {
  using R = typename std::conditional<MIXED, float, double>::type;
  using T = R;
  hipStream_t st = b.ctx->stream, st2 = b.ctx->stream2;
  const int ns = b.nsys;
  std::vector<unsigned char> all(ns, 1);
  for (int attempt = 0;; ++attempt) {
    for (Sys *s : b.sys)
      if (!s->acc_clean) launch_zero(s);
    BHIPCHK(hipMemcpyAsync(b.need.p, all.data(), ns, hipMemcpyHostToDevice, st));
    BHIPCHK(hipMemcpyAsync(b.bsys.p, b.bsys_h, sizeof(BatchSys) * ns, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_batch_clear, dim3(nblk(ns, 256)), dim3(256), 0, st, ns,
                       reinterpret_cast<const BatchSys *>(b.bsys.p));
    const BatchStep bk{0, 0, reinterpret_cast<unsigned char *>(b.need.p)};
    batch_go<OpBin>(b.bin, st, bk);
    batch_go<OpScanColumns>(b.scan, st, bk);
    batch_go<OpScatter>(b.scatter, st, bk);
    batch_go<OpSplitFill<R>>(b.split, st, bk);
    batch_go<OpBuildList>(b.list, st, bk);
    batch_go<OpRuns>(b.runs, st, bk);
    batch_go<OpPmeSpreadZ<MIXED, ORDER>>(b.spread, st, bk);
    batch_go<OpPmeSpreadZLong<MIXED, ORDER>>(b.spreadL, st, bk);
    BHIPCHK(hipEventRecord(b.fork, st));
    BHIPCHK(hipStreamWaitEvent(st2, b.fork, 0));
    batch_go<PairOp<MIXED, C, LJ, CS, BIGLJ, ORDER>>(b.pair, st, bk);
    batch_go<OpFftPlane<T>>(b.plane, st2, bk);
    batch_go<OpFftY<T>>(b.yfwd, st2, bk);
    batch_go<OpFftYLong<T>>(b.yfwdL, st2, bk);
    batch_go<OpFftXConv<T>>(b.xconv, st2, bk);
    batch_go<OpFftXConvLong<T>>(b.xconvL, st2, bk);
    batch_go<OpFftY<T>>(b.yinv, st2, bk);
    batch_go<OpFftYLong<T>>(b.yinvL, st2, bk);
    batch_go<OpPmeZGather<MIXED, ORDER>>(b.gather, st2, bk);
    batch_go<OpPmeZGatherLong<MIXED, ORDER>>(b.gatherL, st2, bk);
    BHIPCHK(hipEventRecord(b.join, st2));
    batch_go<OpFixups<MIXED, C, LJ, CS>>(b.fixups, st, bk);
    BHIPCHK(hipStreamWaitEvent(st, b.join, 0));
    if (b.first_forces)
      batch_go<OpUnsortForces<MIXED>>(b.unsort, st, bk);
    else
      batch_go<OpUnsortEnergy<MIXED>>(b.energy, st, bk);
    batch_go<OpOut>(b.out, st, bk);
    hipLaunchKernelGGL(k_batch_flags, dim3(nblk(ns, 256)), dim3(256), 0, st, ns,
                       reinterpret_cast<const BatchSys *>(b.bsys.p), reinterpret_cast<int *>(b.flags.p));
    BHIPCHK(hipMemcpyAsync(b.flags_h, b.flags.p, 4 * (size_t)ns, hipMemcpyDeviceToHost, st));
    BHIPCHK(hipGetLastError());
    BHIPCHK(hipStreamSynchronize(st));
    bool grown = false;
    for (int i = 0; i < ns; ++i) {
      b.sys[i]->acc_clean = true;
      if (!b.flags_h[i] || attempt >= 6) continue;
      grown = true;
      if (int rc = grow_and_retry(b.sys[i])) return rc;
    }
    if (!grown) break;
    if (int rc = batch_tables<MIXED, C, LJ, CS, BIGLJ, ORDER>(b)) return rc;
  }
  for (Sys *s : b.sys) {
    s->list_valid = true;
    s->prune_pending = false;
    s->staged = b.results && batch_stages(s);
    s->energies_at = b.results ? Sys::kInResults : Sys::kInPartials;
  }
  return PMX_OK;
}

constexpr int kBatchChunk = 64;  // steps between the host's checks of a batch

// nsteps MD steps of every system of the batch.  Chunks of up to
// kBatchChunk steps; after each the host reads the overflow flags, and a
// chunk in which a list outgrew its buffers is run again from its start
// (backups of every system) after those systems' buffers grow.
template <bool MIXED, int C, int LJ, int CS, bool BIGLJ, int ORDER>
int batch_run(Batch &b, int nsteps) {
  hipStream_t st = b.ctx->stream;
  int rc;
  // the first forces of the systems that lack them, in a batched pass of
  // their own: whatever the others of the batch, their lists get the same cut
  if (!b.fresh.empty()) {
    const bool every = b.fresh.size() == b.sys.size();
    Batch some;
    Batch &f = every ? b : some;
    if (!every) {
      some.ctx = b.ctx;
      some.sys = b.fresh;
      some.nsys = (int)b.fresh.size();
      if ((rc = batch_buffers(some))) return rc;
    }
    f.first_forces = true;
    if ((rc = batch_tables<MIXED, C, LJ, CS, BIGLJ, ORDER>(f)) || (rc = batch_forces<MIXED, C, LJ, CS, BIGLJ, ORDER>(f)))
      return rc;
    for (int i = 0; i < f.nsys; ++i) {
      if (f.flags_h[i]) return fail(b.ctx, PMX_ERR_OVERFLOW, "pair list capacity exceeded");
      ++f.sys[i]->md.rebuilds;
      f.sys[i]->md.forces_valid = true;
    }
  }
  if (b.fresh.size() < b.sys.size() && (rc = batch_tables<MIXED, C, LJ, CS, BIGLJ, ORDER>(b))) return rc;
  BHIPCHK(hipMemsetAsync(b.rebuilds.p, 0, 8 * (size_t)b.nsys, st));
  int done = 0, retries = 0, last = 0;
  while (done < nsteps) {
    const int K = std::min(kBatchChunk, nsteps - done);
    last = K;
    for (int i = 0; i < b.nsys; ++i) b.base_h[i] = (unsigned long long)(b.sys[i]->md.steps + done);
    if ((rc = batch_chunk<MIXED, C, LJ, CS, BIGLJ, ORDER>(b, K, done == 0))) return rc;
    BHIPCHK(hipStreamSynchronize(st));
    bool grown = false;
    for (int i = 0; i < b.nsys; ++i) {
      if (!b.flags_h[i]) continue;
      if (!grown && ++retries > 6) return fail(b.ctx, PMX_ERR_OVERFLOW, "pair list capacity exceeded during MD");
      if (!grown) {
        // every system back to the chunk's start
        for (Sys *s : b.sys)
          if ((rc = restore_chunk(s, 0))) return rc;
      }
      grown = true;
      if ((rc = grow_and_retry(b.sys[i]))) return rc;
    }
    if (grown) {
      if ((rc = batch_tables<MIXED, C, LJ, CS, BIGLJ, ORDER>(b))) return rc;
      for (int i = 0; i < b.nsys; ++i) b.bsys_h[i].force = 1;
      BHIPCHK(hipStreamSynchronize(st));
      continue;
    }
    for (int i = 0; i < b.nsys; ++i) b.bsys_h[i].force = 0;
    done += K;
  }
  // closing half kick of every system's last step
  const BatchStep bk{last, 0, nullptr};
  batch_go<OpHalfKick>(b.half, st, bk);
  std::vector<long long> nreb(b.nsys);
  BHIPCHK(hipMemcpyAsync(nreb.data(), b.rebuilds.p, 8 * (size_t)b.nsys, hipMemcpyDeviceToHost, st));
  BHIPCHK(hipStreamSynchronize(st));
  for (int i = 0; i < b.nsys; ++i) {
    Sys *s = b.sys[i];
    s->md.steps += nsteps;
    s->md.rebuilds += nreb[i];
    s->list_valid = true;
    s->energies_at = Sys::kInPartials;
    s->prune_pending = false;
    s->acc_clean = true;
  }
  return PMX_OK;
}

}  // extern "C++"


}  // namespace

int pmx_md_run(pmx_sys *sys, int nsteps) {
  if (!sys || nsteps < 0) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  MdRun r;
  if (int rc = md_begin(s, r, nsteps)) return rc;
  if (r.finished) return PMX_OK;
  bool progressed;
  while (!r.finished)
    if (int rc = md_advance(s, r, true, &progressed)) return rc;
  return md_end(s);
}

int pmx_md_run_many(pmx_sys *const *systems, int nsys, int nsteps) {
  if (!systems || nsys < 0 || nsteps < 0) return PMX_ERR_ARG;
  for (int i = 0; i < nsys; ++i) {
    if (!systems[i]) return PMX_ERR_ARG;
    for (int j = 0; j < i; ++j)
      if (systems[j] == systems[i]) return fail(systems[i]->s.ctx, PMX_ERR_ARG, "a system is listed twice");
  }
  // systems grouped by context; one host thread drives each group
  std::vector<pmx_ctx *> ctxs;
  std::vector<std::vector<Sys *>> groups;
  for (int i = 0; i < nsys; ++i) {
    Sys *s = &systems[i]->s;
    size_t g = std::find(ctxs.begin(), ctxs.end(), s->ctx) - ctxs.begin();
    if (g == ctxs.size()) {
      ctxs.push_back(s->ctx);
      groups.emplace_back();
    }
    groups[g].push_back(s);
  }
  std::vector<int> status(groups.size(), PMX_OK);
  auto drive = [&](size_t g) {
    std::vector<Sys *> &sys = groups[g];
    std::vector<MdRun> runs(sys.size());
    for (size_t i = 0; i < sys.size(); ++i)
      if (int rc = md_begin(sys[i], runs[i], nsteps)) {
        status[g] = rc;
        return;
      }
    for (;;) {
      bool any = false, progressed_any = false;
      for (size_t i = 0; i < sys.size(); ++i) {
        if (runs[i].finished) continue;
        any = true;
        bool p = false;
        if (int rc = md_advance(sys[i], runs[i], false, &p)) {
          status[g] = rc;
          return;
        }
        progressed_any |= p;
      }
      if (!any) break;
      if (!progressed_any) {
        // nothing completed: wait for the oldest chunk of the first
        // unfinished system
        for (size_t i = 0; i < sys.size(); ++i)
          if (!runs[i].finished) {
            bool p = false;
            if (int rc = md_advance(sys[i], runs[i], true, &p)) {
              status[g] = rc;
              return;
            }
            break;
          }
      }
    }
    for (Sys *s : sys)
      if (int rc = md_end(s)) {
        status[g] = rc;
        return;
      }
  };
  if (groups.size() == 1) {
    drive(0);
  } else {
    std::vector<std::thread> threads;
    for (size_t g = 0; g < groups.size(); ++g) threads.emplace_back(drive, g);
    for (auto &t : threads) t.join();
  }
  for (int rc : status)
    if (rc) return rc;
  return PMX_OK;
}

extern "C++" {
namespace {

// nsteps < 0: one force pass (batch_forces), else nsteps MD steps.
template <bool MIXED, int C, int LJ, int CS, bool BIG, int ORDER>
int batch_exec(Batch &b, int nsteps) {
  if (nsteps >= 0) return batch_run<MIXED, C, LJ, CS, BIG, ORDER>(b, nsteps);
  if (int rc = batch_tables<MIXED, C, LJ, CS, BIG, ORDER>(b)) return rc;
  return batch_forces<MIXED, C, LJ, CS, BIG, ORDER>(b);
}

template <bool MIXED, int CASE>
int batch_run_case(Batch &b, int order, int nsteps) {
  constexpr int LJ = CASE == 0 ? SW_C2 : (CASE == 1 ? SW_NONE : SW_ANY);
  constexpr int CS = CASE == 0 ? SW_CUTOFF : SW_ANY;
  constexpr bool BIG = CASE == 3;
  switch (order) {
    case 4: return batch_exec<MIXED, COUL_PME, LJ, CS, BIG, 4>(b, nsteps);
    case 6: return batch_exec<MIXED, COUL_PME, LJ, CS, BIG, 6>(b, nsteps);
    default: return batch_exec<MIXED, COUL_PME, LJ, CS, BIG, 8>(b, nsteps);
  }
}

template <bool MIXED>
int batch_run_form(Batch &b, int cs, int order, int nsteps) {
  switch (cs) {
    case 0: return batch_run_case<MIXED, 0>(b, order, nsteps);
    case 1: return batch_run_case<MIXED, 1>(b, order, nsteps);
    case 2: return batch_run_case<MIXED, 2>(b, order, nsteps);
    default: return batch_run_case<MIXED, 3>(b, order, nsteps);
  }
}

// Checks a batch's systems, makes the batch's buffers and runs it
// (nsteps < 0: one force pass).
int batch_entry(pmx_sys *const *systems, int nsys, int nsteps) {
  Sys *s0 = &systems[0]->s;
  pmx_ctx *ctx = s0->ctx;
  const bool md = nsteps >= 0;
  const int cs = batch_case(s0), order = s0->pme.order;
  std::set<const pmx_sys *> seen;
  for (int i = 0; i < nsys; ++i) {
    Sys *s = &systems[i]->s;
    if (!seen.insert(systems[i]).second) return fail(ctx, PMX_ERR_ARG, "a system is listed twice");
    if (s->ctx != ctx) return fail(ctx, PMX_ERR_ARG, "the systems of a batch share one context");
    if (md && !s->md.on) return fail(ctx, PMX_ERR_ARG, "pmx_md_init first (every system of the batch)");
    if (!s->have_positions) return fail(ctx, PMX_ERR_ARG, "positions not set (every system of the batch)");
    if (s->mixed != s0->mixed || batch_case(s) != cs)
      return fail(ctx, PMX_ERR_ARG, "the systems of a batch share the precision and the kinds of force");
    if (!s->pme_on || !(s->d.pme_terms & PMX_PME_RECIP) || s->pme.order < 4 || s->pme.order != order)
      return fail(ctx, PMX_ERR_UNSUPPORTED, "batched launches take PME systems of one stencil order (4, 6 or 8)");
    if (s->nbins > kScanSingleMax)
      return fail(ctx, PMX_ERR_UNSUPPORTED, "batched launches take systems of at most 65,536 cell bins");
  }
  if (nsteps == 0) return PMX_OK;
  hipSetDevice(ctx->device);
  Batch b;
  b.ctx = ctx;
  b.nsys = nsys;
  b.results = !md;
  for (int i = 0; i < nsys; ++i) {
    Sys *s = &systems[i]->s;
    s->staged = false;
    s->energies_at = Sys::kInPartials;
    b.sys.push_back(s);
    if (!s->cached)
      if (int rc = setup(s)) return rc;
    if (md && !s->md.forces_valid) b.fresh.push_back(s);
    if (md && !s->acc_clean) {
      launch_zero(s);
      s->acc_clean = true;
    }
  }
  if (int rc = batch_buffers(b)) return rc;
  // the batch runs on the context's two streams, idle from here on
  if (hipStreamSynchronize(ctx->stream) != hipSuccess || hipStreamSynchronize(ctx->stream2) != hipSuccess)
    return fail(ctx, PMX_ERR_HIP, "stream synchronize");
  return s0->mixed ? batch_run_form<true>(b, cs, order, nsteps) : batch_run_form<false>(b, cs, order, nsteps);
}

}  // namespace
}  // extern "C++"

int pmx_md_run_batch(pmx_sys *const *systems, int nsys, int nsteps) {
  if (!systems || nsys <= 0 || nsteps < 0) return PMX_ERR_ARG;
  for (int i = 0; i < nsys; ++i)
    if (!systems[i]) return PMX_ERR_ARG;
  return batch_entry(systems, nsys, nsteps);
}

int pmx_sys_compute_batch(pmx_sys *const *systems, int nsys, unsigned flags) {
  if (!systems || nsys <= 0) return PMX_ERR_ARG;
  for (int i = 0; i < nsys; ++i)
    if (!systems[i]) return PMX_ERR_ARG;
  if (flags) return fail(systems[0]->s.ctx, PMX_ERR_UNSUPPORTED, "batched force passes take no flags");
  return batch_entry(systems, nsys, -1);
}

int pmx_md_get_state(pmx_sys *sys, double *x, double *v, double *energies) {
  if (!sys) return PMX_ERR_ARG;
  Sys *s = &sys->s;
  Sys::Md &m = s->md;
  if (!m.on || !s->have_positions) return fail(s->ctx, PMX_ERR_ARG, "pmx_md_init and pmx_md_set_state first");
  hipSetDevice(s->ctx->device);
  hipStream_t st = s->ctx->stream;
  const int n = s->n;
  const bool bonded = m.nb + m.na > 0;
  const size_t nke = nblk(n, 256), nbe = bonded ? 2 * (size_t)s->term_blocks : 0, vec = 3 * (size_t)n;
  if (energies) {
    // potential energies at the current positions (computed first if the
    // state was just set) and kinetic energy of v
    if (int rc = md_ensure_forces(s)) return rc;
    reduce_energies(s, false);
    hipLaunchKernelGGL(k_kinetic, dim3(nblk(n, 256)), dim3(256), 0, st, n, P<double>(m.v), P<double>(m.minv),
                       P<double>(m.ke_e));
  }
  // everything in one go when it fits the stage, else positions and
  // velocities in chunks first
  size_t words = energies ? 4 + nke + nbe : 0;
  const bool once = 8 * (words + (x ? vec : 0) + (v ? vec : 0)) <= kStageBytes;
  for (int k = 0; k < 2 && !once; ++k) {
    double *const to = k ? v : x;
    if (!to) continue;
    const int rc = fetch(s, k ? m.v.p : s->xorig.p, 8 * vec, [&](size_t o, const void *data, size_t bytes) {
      std::memcpy(reinterpret_cast<unsigned char *>(to) + o, data, bytes);
    });
    if (rc) return rc;
  }
  if (once) words += (x ? vec : 0) + (v ? vec : 0);
  if (int rc = stage_get(s, 8 * words)) return rc;
  OutList out(s->stage.p);
  const double *const h = static_cast<double *>(s->stage.p);
  const double *ke = h, *be = h;
  if (energies) {
    out.add(s->energies_at == Sys::kInHeld ? s->md.held.p : s->eout.p, 4);
    ke = out.add(m.ke_e.p, nke);
    be = out.add(m.bond_e.p, nbe);
  }
  const double *const hx = out.add(s->xorig.p, once && x ? vec : 0);
  const double *const hv = out.add(m.v.p, once && v ? vec : 0);
  if (out.a.end[4]) out.launch(st);
  HIPCHK(hipStreamSynchronize(st));
  if (once && x) std::memcpy(x, hx, 8 * vec);
  if (once && v) std::memcpy(v, hv, 8 * vec);
  if (energies) {
    double eb = 0, ea = 0, ek = 0;
    for (size_t i = 0; i < nbe; i += 2) {
      eb += be[i];
      ea += be[i + 1];
    }
    for (size_t i = 0; i < nke; ++i) ek += ke[i];
    double ec = h[0];
    if (s->pme_on) ec += h[2] + h[3] + s->self_e + s->charged_e;
    energies[PMX_MD_E_COULOMB] = ec;
    energies[PMX_MD_E_LJ] = h[1];
    energies[PMX_MD_E_BOND] = eb;
    energies[PMX_MD_E_ANGLE] = ea;
    energies[PMX_MD_E_KINETIC] = ek;
  }
  return PMX_OK;
}

unsigned long long pmx_estimate_bytes(const pmx_sys_desc *desc, int kind) {
  if (!desc || validate(nullptr, desc) != PMX_OK) return 0;
  pmx_sys tmp;
  Sys *s = &tmp.s;
  s->d = *desc;
  s->dry = true;
  if (setup(s) != PMX_OK) return 0;
  unsigned long long b = s->dry_bytes;
  // device MD state: velocities, masses, build positions by slot, two chunk backups
  // of x, v and f, bonded tables (bonds and angles about one per atom in the
  // systems served)
  if (kind == 1)
    b += 176ull * (unsigned long long)desc->n + 32ull * (unsigned long long)s->npad + 132ull * (unsigned long long)desc->n + 8192;
  return b;
}

int pmx_sys_device_bytes(const pmx_sys *sys, unsigned long long *bytes) {
  if (!sys || !bytes) return PMX_ERR_ARG;
  unsigned long long b = 0;
  for (const DevBuf *d : sys->s.all)
    if (d->p) b += d->bytes;
  *bytes = b;
  return PMX_OK;
}

int pmx_langevin_noise(unsigned long long seed, unsigned long long half, int n, double *g) {
  if (n < 0 || (n > 0 && !g)) return PMX_ERR_ARG;
  for (int i = 0; i < n; ++i) langevin_gauss3(seed, half, (uint32_t)i, g + 3 * i);
  return PMX_OK;
}

int pmx_md_stats(const pmx_sys *sys, long long *steps, long long *rebuilds, long long *rollbacks) {
  if (!sys || !steps || !rebuilds || !rollbacks) return PMX_ERR_ARG;
  *steps = sys->s.md.steps;
  *rebuilds = sys->s.md.rebuilds;
  *rollbacks = sys->s.md.rollbacks;
  return PMX_OK;
}

}  // extern "C"
