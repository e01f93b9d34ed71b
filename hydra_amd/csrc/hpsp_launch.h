// Host-side launch interface between the C ABI (capi.hip) and the kernel
// translation units.  Internal to libhpsp.so.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "hpsp_device.h"

namespace hpsp {

constexpr int kAvgChunk = 4096;  // events per AverageOn reduction chunk
constexpr int kUwTile = 1024;    // events per Unweight tile (256 threads x 4)
constexpr int kXcds = 8;         // MI355X: workgroups are dealt to 8 XCDs in turn
constexpr uint64_t kRunMinRuns = 8192;  // 8 runs per SIMD of 256 CUs x 4 SIMDs

struct GenArgs {
  DecayK d;
  uint64_t first, n;
  void* cols;
  uint64_t ld;
  int out_f32;
  double* wt;
  double* evw;
  const double* mothers;  // FP64 mother columns (E,px,py,pz) or null
  uint64_t mld;
  int xcd_ranges;  // xcd_block's ranges (FP64)

  // the same call's events from off on, n of them
  GenArgs part(uint64_t off, uint64_t count) const {
    GenArgs c = *this;
    c.first += off;
    c.n = count;
    if (c.cols) c.cols = static_cast<char*>(c.cols) + off * (out_f32 ? 4 : 8);
    if (c.wt) c.wt += off;
    if (c.evw) c.evw += off;
    if (c.mothers) c.mothers += off;
    return c;
  }
};

// AverageOn arguments; FK is the functor: in the kernels a description
// (FunctorFastK, FunctorMixedK) or a user's callable in a translation unit that
// compiles its own kernels (hydra_amd/include/hydra/detail/UserKernels.h).
template <typename FK>
struct AvgArgsT {
  DecayK d;
  FK f;
  uint64_t first, n;
  const double* mothers;
  uint64_t mld;
  Stats* partials;  // one per kAvgChunk events
};
// A described functor in both forms, of which each launcher passes its own on.
struct AvgFunctor {
  FunctorFastK fast;
  FunctorMixedK mixed;
};
using AvgArgs = AvgArgsT<AvgFunctor>;
template <typename FK>
inline AvgArgsT<FK> with_functor(const AvgArgs& a, const FK& f) {
  return {a.d, f, a.first, a.n, a.mothers, a.mld, a.partials};
}

// Up to HPSP_MAX_EVAL_FUNCTORS described functors, evaluated one by one.
struct DescSet {
  FunctorK f[HPSP_MAX_EVAL_FUNCTORS];
  int nf;
  int pairs;  // some functor takes pair masses
};

// Evaluate arguments; FS is the set of functors whose values are written.
template <typename FS>
struct EvalArgsT {
  DecayK d;
  FS fs;
  uint64_t seed;            // Evaluate(mothers): the seed paired with each event index
  uint64_t first, n;
  const double* mothers;    // Evaluate(mothers): SoA mother columns
  uint64_t mld;
  double* out;              // 1 + nf columns of ld doubles
  uint64_t ld;

  EvalArgsT part(uint64_t off, uint64_t count) const {
    EvalArgsT c = *this;
    c.first += off;
    c.n = count;
    if (c.mothers) c.mothers += off;
    c.out += off;
    return c;
  }
};
using EvalArgs = EvalArgsT<DescSet>;

// Four-vectors of stored events: particle i, component c, event k at
// cols[i][c * ld[i] + k].
struct ParticlesK {
  const double* cols[HPSP_MAX_PARTICLES];
  uint64_t ld[HPSP_MAX_PARTICLES];
  int n;
};

// Reads the particles a functor asks for from memory (wave-uniform particle
// index, lane-contiguous events): only the columns in use are loaded.
struct MemAcc {
  const ParticlesK& p;
  uint64_t k;
  __device__ __forceinline__ void get(int i, double (&v)[4]) const {
    const double* c = p.cols[i] + k;
    const uint64_t ld = p.ld[i];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = c[(uint64_t)q * ld];
  }
  __device__ __forceinline__ const MemAcc& pairs() const { return *this; }
  __device__ __forceinline__ double pair(int a, int b) const {
    double u[4], v[4];
    get(a, u);
    get(b, v);
    return pair_mass2(u, v);
  }
  __device__ __forceinline__ void sum(int first, int last, double (&Pv)[4]) const {
#pragma clang fp contract(off)
    get(first, Pv);
    for (int i = first + 1; i < last; ++i) {
      double v[4];
      get(i, v);
#pragma unroll
      for (int q = 0; q < 4; ++q) Pv[q] = Pv[q] + v[q];
    }
  }
};

struct PartEvalArgs {
  ParticlesK p;
  FunctorK f[HPSP_MAX_EVAL_FUNCTORS];
  int nf;
  uint64_t n;
  double* out;  // nf columns of ld doubles
  uint64_t ld;
};

// Dense histogram geometry with the reference's derived quantities:
// delta = upper - lower, gridf = (double)grid, row-major strides.
struct HistK {
  int ndim;
  double lower[HPSP_HIST_MAX_DIM], delta[HPSP_HIST_MAX_DIM], gridf[HPSP_HIST_MAX_DIM];
  uint64_t stride[HPSP_HIST_MAX_DIM];
  uint64_t nbins;
};

constexpr int kHistBlock = 1024;

struct HistArgs {
  HistK h;
  const double* x;          // columns source: ndim value columns
  uint64_t ldx;
  DecayK d;                 // events source: masses and fMaxWeight (PhaseSpaceWeight)
  FunctorK axes[HPSP_HIST_MAX_DIM];
  const double* cols;       // events source: 4N momentum columns
  uint64_t ld;
  ParticlesK parts;         // particles source
  int weight_mode;          // hpsp_hist_weight (the launcher may add kByDaughter)
  const double* w;
  uint64_t n;
  double* contents;         // nbins + 2
  int use_lds;              // block-private bins in LDS
  uint64_t lds_slots;       // LDS capacity in doubles (launcher)
};

// phase_space_range: the DecayMother events of a minstd_rand stream.  Word j
// of element first + k is x_start * 48271^(k + j) mod (2^31 - 1), x_start
// being the engine's state after discard(first + 3N) and one step.
struct RangeArgs {
  DecayK d;            // key words unused
  uint32_t x_start;
  uint32_t run;        // consecutive groups of 64 elements per wave (set by the launcher)
  uint64_t n;
  double* cols;        // generate: 4N momentum columns of ld doubles
  uint64_t ld;
  double* wt;          // generate: weights or null
  HistK h;             // histogram fill
  FunctorK axes[HPSP_HIST_MAX_DIM];
  int weight_mode;
  double* contents;
  int use_lds;
  uint64_t lds_slots;
};

struct WeightArgs {
  DecayK d;
  FunctorK f;
  int use_f;
  const double* cols;
  uint64_t ld, n;
  double* w_out;       // values (event_weight; max_weight: null to skip)
};

struct UnweightArgs {
  DecayK d;
  FunctorK f;
  int use_f;
  double maxv;          // divisor of the acceptance test
  const double* maxv_dev;  // if non-null, divisor read from device memory
  uint64_t uw_key;      // splitmix64(seed) of the default engine
  const double* cols_in;
  uint64_t ld_in, n;
  const double* w_in;
  double* cols_out;
  uint64_t ld_out;
  uint64_t* idx_out;
  double* w_out;
  uint64_t* flags;      // one bit per event, 64 per word
  uint32_t* tile_count; // accepted per tile
  uint64_t* tile_off;   // exclusive prefix of tile_count
  uint64_t* run_sum;    // per-1024-tile sums, then their exclusive prefix
  uint64_t* n_acc;      // total accepted (device)
  int rule;             // 0: w / max > u (Decays::Unweight); 1: u * max <= w (RndFlag)
  uint64_t jump;        // counter offset of the uniforms (rule 1)
  int order;            // 0: both parts stable; 1: sequential swap partition
  uint64_t* tidx;       // order 1: original index of the r-th kept sample
  int regen;            // events regenerated at their destinations, not moved
  uint64_t gen_first;   // regen: generation index of the container's row 0
  int scan_here;        // the scatter sums the counts itself (use_scan_here): kScanTiles
                        // from tile_count, kScanBlocks from a 16-bit count per 256 events
                        // at tile_off (four in the place of one offset)
};
constexpr int kScanTiles = 1, kScanBlocks = 2;

// Up to kScanHereTiles tiles (2^20 events) the scatter's blocks sum the counts
// themselves, at most four per thread, instead of reading offsets that a kernel
// of its own wrote: a launch (about 4 us) less, for two shuffle sums per block.
// For calls with outputs; block 0 writes the accepted total.
constexpr uint64_t kScanHereTiles = 4 * kBlock;
inline bool use_scan_here(const UnweightArgs& a) {
  return (a.cols_out || a.idx_out || a.w_out) && a.order == 0 &&
         (a.n + kUwTile - 1) / kUwTile <= kScanHereTiles;
}

// Kernel launchers; each returns a hipError_t value.
int launch_generate_f64(int N, int engine, const GenArgs& a, hipStream_t s);
int launch_generate_mixed(int N, int engine, const GenArgs& a, hipStream_t s);
int launch_average_f64(int N, int engine, const AvgArgs& a, hipStream_t s);
int launch_average_mixed(int N, int engine, const AvgArgs& a, hipStream_t s);
int launch_evaluate_f64(int N, int engine, bool mothers, const EvalArgs& a, hipStream_t s);
// N = 0: value columns; N >= 2: events of N daughters; N = -1: particles
int launch_histogram_fill(int N, const HistArgs& a, hipStream_t s);
int launch_particles_evaluate(const PartEvalArgs& a, hipStream_t s);
void launch_zero(double* p, uint64_t n, hipStream_t s);
int launch_range_generate(int N, const RangeArgs& a, hipStream_t s);
int launch_range_histogram(int N, const RangeArgs& a, hipStream_t s);
int launch_stats_finalize(const Stats* partials, uint64_t m, Stats* out, hipStream_t s);
int launch_event_weight(int N, const WeightArgs& a, hipStream_t s);
// Exclusive scan of the tile counts into a.tile_off, the total into *a.n_acc
// (nothing where a.scan_here is set).
int launch_uw_scans(const UnweightArgs& a, hipStream_t s);
// Flags of Decays::Unweight for events a.gen_first.. of a Generate with decay
// a.d, decided from each event's generation weight where it is far enough
// from the boundary (generate_unweight.hip); dl_count and dl: a counter and a
// list of two words per group of 64 events (the groups with events left in
// doubt, decided by a second kernel); tab3: 2 kBin3 doubles, the 3-body
// bound's table (written and read by the call when N = 3); ck: the call's
// constants, formed on the host.
constexpr int kBin3Side = 8 + 28 * 8;  // bins per end of [0, 1]
constexpr int kBin3 = 2 * kBin3Side;
struct ChainK {
  double C;         // 2^64 (maxw / max)^2 / 4^(N-1)
  // N = 3, with A = invMas[2]:
  double C3;        // C / A^2
  double A2;        // A^2
  double sp2, sm2;  // (m1 + m0)^2, (m1 - m0)^2
  double ecm32;     // ecm / 2^32
  double ks_unit;   // eps S^2, S^2 bounding E^2 + p^2 of any subsystem
  double ks_fixed;  // (2K + 4) eps S^2 with the squares engines' K = 2^17 N
  double ic2_0;     // 1 / m0^2
  int fast_ok;      // max and maxw positive, 1/max and C (N = 3: the masses) in range
  double rmax;      // RN(1 / max) and whether it is normal (ratio_above)
  int rmax_ok;
};
// For few events with outputs (a.scan_here) instead: every event's momenta,
// PhaseSpaceWeight and test in one kernel (genbod_f64.hip; kScanBlocks).
int launch_flags_exact(int N, int engine, const UnweightArgs& a, hipStream_t s);
int launch_flags_chain(int N, int engine, const UnweightArgs& a, uint64_t* dl_count, uint64_t* dl,
                       double* tab3, const ChainK& ck, hipStream_t s);
// The mixed form: flags from each event's FP64 weight chain, the mixed
// Generate's weight column (generate_unweight.hip; tab3 and ck as for
// launch_flags_chain); then every event generated again at its place, FP32
// columns in a.cols_out, carried as a double pointer (genbod_mixed.hip).
// (for few events with outputs, a.scan_here, instead: every event's weight chain
// and test in one kernel, launch_flags_direct; kScanBlocks)
int launch_flags_direct(int N, int engine, const UnweightArgs& a, hipStream_t s);
int launch_flags_mixed(int N, int engine, const UnweightArgs& a, double* tab3, const ChainK& ck,
                       hipStream_t s);
int launch_unweight_regen_mixed(int N, int engine, const UnweightArgs& a, hipStream_t s);
int launch_max_weight(int N, const WeightArgs& a, double* block_max, uint64_t nblocks,
                      double* out, hipStream_t s);
int launch_unweight(int N, const UnweightArgs& a, hipStream_t s);
// order-independent checksum of n 64-bit words into *sum (device)
int launch_checksum(const uint64_t* w, uint64_t n, uint64_t* sum, hipStream_t s);
// largest of n values (max_element's value) into *out, through per-block maxima
int launch_max_column(const double* w, uint64_t n, double* block_max, uint64_t nblocks,
                      double* out, hipStream_t s);
// after launch_unweight with regen set: the stable partition of events
// gen_first .. gen_first + n - 1 of the generation stream, generated again
int launch_unweight_regen(int N, int engine, const UnweightArgs& a, hipStream_t s);
// hydra::unweight over ncols value columns and a weight column (rule 1).
int launch_unweight_sample(int ncols, const UnweightArgs& a, double* block_max,
                           uint64_t nblocks, double* max_dev, hipStream_t s);
int launch_rng_words(int engine, const uint64_t* key, uint64_t discard, uint64_t n,
                     uint64_t* out, hipStream_t s);

// The 256-event block of a workgroup, of those of n events.  Workgroups go to the
// XCDs in turn; with `ranges` each XCD takes a contiguous range of blocks, so that
// what one XCD's L2 sends to memory lies together.  Only stores that bound the
// kernel gain: FP64 events of 2 and 3 bodies from kXcdRangeBytes on (neighbouring
// blocks on different XCDs -> ranges: 3 bodies, 2^27 events 2505 -> 2340 us, their
// momenta alone 2270 -> 2126; 2^26 1280 -> 1247; 2 bodies, 2^27 1653 -> 1607).
// Below it results go either way (3 bodies, 2^22 -3 %, 2^24 +3 %), 4 and more
// bodies stay the same, mixed 5-body events of 2^25 lose 8 % (490 -> 527 us).
constexpr uint64_t kXcdRangeBytes = 4ull << 30;
__device__ __forceinline__ uint64_t xcd_block(uint64_t n, int ranges) {
  if (!ranges) return blockIdx.x;
  const uint64_t nblocks = (n + kBlock - 1) / kBlock;
  const uint64_t per_xcd = (nblocks + kXcds - 1) / kXcds;
  return (uint64_t)(blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
}

// One launch(args, blocks) of kBlock events per block (xcd_block; blocks a
// multiple of kXcds) for every 2^31 events (a dispatch holds fewer than 2^32
// work-items).
constexpr uint64_t kGridEvents = 1ULL << 31;
template <typename Args, typename Launch>
inline void over_grids(const Args& a, Launch&& launch) {
  for (uint64_t off = 0; off < a.n; off += kGridEvents) {
    const uint64_t n = a.n - off < kGridEvents ? a.n - off : kGridEvents;
    const uint64_t blocks = (n + kBlock - 1) / kBlock;
    launch(a.part(off, n), (unsigned)((blocks + kXcds - 1) / kXcds * kXcds));
  }
}

// Groups of 64 elements per wave in a run of k_range_generate: a longer run
// shares more engine words between consecutive groups, but the runs must still
// give every SIMD several waves; the longest power of two up to max_run that
// leaves kRunMinRuns runs.
inline uint32_t run_groups(uint64_t ngroups, uint64_t max_run) {
  uint64_t r = 1;
  while (r < max_run && ngroups >= 2 * r * kRunMinRuns) r *= 2;
  return (uint32_t)r;
}

// Blocks of four waves for the runs of ngroups groups, one run per wave; the runs
// are lengthened where they would be more than one launch can hold.
inline unsigned blocks_for_runs(uint64_t ngroups, uint32_t& run) {
  constexpr uint64_t kWavesPerBlock = kBlock / kWave, kMostRuns = kGridEvents / kWave;
  while ((ngroups + run - 1) / run > kMostRuns) run *= 2;
  const uint64_t nruns = (ngroups + run - 1) / run;
  return (unsigned)((nruns + kWavesPerBlock - 1) / kWavesPerBlock);
}

// AverageOn over n events: wide(blocks, threads), waves_wide waves per chunk,
// up to one chunk per CU, narrow(blocks), four waves per chunk, beyond.  At
// 2^20 events (256 chunks) wide took 24 us against 31 narrow for 3 bodies, 46
// against 66 for 6, 82 against 113 for 10, 26 against 37 for 5 in mixed
// precision; at 384 chunks, where some CUs get a second one, it lost (mixed:
// 104 against 95 for 10 bodies) or tied.
constexpr uint64_t kAvgWideChunks = 256;
template <typename Narrow, typename Wide>
inline void launch_avg(uint64_t n, int waves_wide, Narrow&& narrow, Wide&& wide) {
  const uint64_t nchunks = (n + kAvgChunk - 1) / kAvgChunk;
  if (nchunks <= kAvgWideChunks)
    wide((unsigned)(nchunks ? nchunks : 1), (unsigned)(waves_wide * kWave));
  else
    narrow((unsigned)(nchunks < 8192 ? nchunks : 8192));
}

// Blocks of the kernels that leave one maximum each to a last block: 8 waves
// per SIMD (65536 took that block 42 us).
constexpr unsigned kMaxBlocks = 2048;

// Blocks for a grid-stride launch over `items` work items of kBlock each.
inline unsigned grid_for(uint64_t items, unsigned cap = 65536u) {
  const uint64_t b = (items + kBlock - 1) / kBlock;
  return (unsigned)(b == 0 ? 1 : (b < cap ? b : cap));
}

}  // namespace hpsp
