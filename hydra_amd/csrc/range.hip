// hydra::phase_space_range on gfx950 (PhaseSpaceRange.inl:44-72): element k
// of the lazy range is GenerateDecay<N, minstd_rand>(mother, masses,
// seed)(k) = (weight, p_1, ..., p_N) (GenerateDecay.h:203-343), the GENBOD
// event of DecayMother with the engine discarded by k + 3N.  Built with
// -ffp-contract=off.
//
// Engine words.  minstd_rand's word j of element first + k is
// x_start * a^(k + j) mod m (a = 48271, m = 2^31 - 1).  A wave takes one run of
// consecutive groups of 64 elements, whose words it shares through LDS
// (WindowView): a lane evaluates the word 64 after its last one, one product
// with a^64, for each further group.  A run's first words cost one power of
// a, formed on the scalar unit, and a table lookup.
//
// Kernels:
//   k_range_generate<N>  elements into SoA momentum columns and a weight column
//   k_range_hist<N>      DenseHistogram::Fill(range | axes[, weights]) with
//                        the elements generated inside the fill: nothing but
//                        the bins touches memory.
#include <algorithm>
#include <array>
#include <utility>

#include "event_words.h"
#include "genbod_f64.h"
#include "hist_key.h"

namespace hpsp {

// a^l mod m for l = 0 .. 2 * kWave - 1
struct MinstdPowers {
  uint32_t v[2 * kWave];
};
constexpr MinstdPowers minstd_powers() {
  MinstdPowers t{};
  uint64_t x = 1;
  for (int l = 0; l < 2 * kWave; ++l) {
    t.v[l] = (uint32_t)x;
    x = x * kMinstdA % kMinstdM;
  }
  return t;
}
__constant__ MinstdPowers kPow = minstd_powers();

constexpr uint32_t kMinstdA64 = minstd_powers().v[kWave];  // a^64 mod m

// The words of a wave's groups of elements.
template <int N>
struct RangeWords {
  static constexpr int W = 3 * N - 4;
  using View = WindowView<uint32_t, 1, W>;
  using Window = typename View::Win;
  View v;
  uint32_t x;  // the lane's last word

  // the run's first group, whose first element is k0
  __device__ __forceinline__ void start(Window& win, uint32_t x_start, uint64_t k0, int lane) {
    const uint32_t xw = minstd_mul(x_start, minstd_pow(k0));
    const uint32_t lo[1] = {minstd_mul(xw, kPow.v[lane])};
    x = minstd_mul(lo[0], kMinstdA64);
    const uint32_t hi[1] = {x};
    v.start(win, lane, 0, lo, hi);
  }
  // the group after the last
  __device__ __forceinline__ void next() {
    x = minstd_mul(x, kMinstdA64);
    const uint32_t hi[1] = {x};
    v.shift(hi);
  }
  __device__ __forceinline__ uint64_t operator()(int j) const { return v.get(j); }
};

template <int N>
__device__ __forceinline__ double range_event(const DecayK& d, const RangeWords<N>& w,
                                              double (&p)[N][4]) {
  const double wt = genbod_f64<N, kMinstd>(d, w, p);
  if (d.do_boost) {
#pragma unroll
    for (int i = 0; i < N; ++i) boost_folded(p[i], d);
  }
  return wt;
}

template <int N>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(waves_for(N), 8)))
void k_range_generate(const RangeArgs a) {
  __shared__ typename RangeWords<N>::Window win[kBlock / kWave];
  const int lane = __lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint64_t ngroups = (a.n + kWave - 1) / kWave;
  const uint64_t g_first = ((uint64_t)blockIdx.x * (kBlock / kWave) + (uint64_t)wave) * a.run;
  if (g_first >= ngroups) return;  // wave-uniform
  const uint64_t g_end = (g_first + a.run < ngroups) ? g_first + a.run : ngroups;
  RangeWords<N> words;
  words.start(win[wave], a.x_start, g_first * kWave, lane);
  for (uint64_t g = g_first;;) {
    const uint64_t k0 = g * kWave;
    double p[N][4];
    const double wt = range_event<N>(a.d, words, p);
    if (k0 + (uint64_t)lane < a.n) {
      double* c = a.cols + k0;
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          st(uniform_ptr(c + (uint64_t)(4 * i + q) * a.ld) + lane, p[i][q]);
      if (a.wt) st(uniform_ptr(a.wt + k0) + lane, wt);
    }
    if (++g == g_end) break;
    words.next();
  }
}

// Most threads of a fill's block: every block adds its bins to the contents in
// the end, and those atomics, blocks times bins on few cache lines, not the
// elements set the time of smaller fills (1e6 elements into 100 bins: 2048
// blocks of 256 threads 53 us, 512 of them 31).  Fills of up to range_few_groups
// groups of 64 into few bins take blocks of 256: one wave on each SIMD, whose
// chains of dependent operations are the time (1001 8-body elements 15.4 us with
// 512 threads, 13.1 with 256; 2e4 3-body ones 10.6, 10.1).  With 5e4 elements
// 512 win up to 6 bodies (5: 12.3, 12.7) and lose beyond (8: 16.8, 14.7), and with
// 10^4 bins the blocks' merges are the time (1001 3-body elements 11.2, 12.5).
constexpr int kRangeHistBlock = 512;
constexpr uint64_t range_few_groups(int N) { return N <= 6 ? 512 : 1024; }
constexpr uint64_t kRangeFewSlots = 4096;

template <int N>
__global__ __launch_bounds__(kRangeHistBlock)
    __attribute__((amdgpu_waves_per_eu(N <= 4 ? 4 : (N <= 6 ? 3 : 2), 8)))
void k_range_hist(const RangeArgs a) {
  extern __shared__ double bins[];
  __shared__ typename RangeWords<N>::Window win[kRangeHistBlock / kWave];
  const uint64_t nslots = a.h.nbins + 2;
  if (a.use_lds) {
    for (uint64_t b = threadIdx.x; b < nslots; b += blockDim.x) bins[b] = 0.0;
    __syncthreads();
  }
  const int lane = __lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint64_t ngroups = (a.n + kWave - 1) / kWave;
  const uint64_t g_first =
      ((uint64_t)blockIdx.x * (blockDim.x / kWave) + (uint64_t)wave) * a.run;
  const uint64_t g_end = (g_first + a.run < ngroups) ? g_first + a.run : ngroups;
  if (g_first < ngroups) {  // wave-uniform
    RangeWords<N> words;
    words.start(win[wave], a.x_start, g_first * kWave, lane);
    for (uint64_t g = g_first;;) {
      const uint64_t k = g * kWave + (uint64_t)lane;
      double p[N][4];
      const double wt = range_event<N>(a.d, words, p);
      if (k < a.n) {
        double x[HPSP_HIST_MAX_DIM];
#pragma unroll
        for (int d = 0; d < HPSP_HIST_MAX_DIM; ++d)
          x[d] = (d < a.h.ndim) ? functor_late<true, true>(a.axes[d], p) : 0.0;
        const double w = a.weight_mode == HPSP_HIST_WEIGHT_GENERATION ? wt
                         : a.weight_mode == HPSP_HIST_WEIGHT_PHSP
                             ? event_weight_f64<N>(p, a.d.m, a.d.maxw)
                             : 1.0;
        const uint64_t key = hist_key(a.h, x);
        if (key != kDrop) {
          if (a.use_lds)
            atomicAdd(&bins[key], w);
          else
            unsafeAtomicAdd(&a.contents[key], w);
        }
      }
      if (++g == g_end) break;
      words.next();
    }
  }
  if (a.use_lds) {
    __syncthreads();
    for (uint64_t b = threadIdx.x; b < nslots; b += blockDim.x) {
      const double v = bins[b];
      if (v != 0.0) unsafeAtomicAdd(&a.contents[b], v);
    }
  }
}

// ---------------------------------------------------------------------------

// One run per wave, dispatched in order.  The longest runs: of 3 and 4 bodies, whose
// stores bound them, 1 up to 2^25 elements (4e6 3-body elements 72.7 us, runs of 2
// 78.4, of 4 81.5; 2e6 35.5, 34.0, 34.0; 2^25 620, of 4 621) and 4 or 16 beyond
// (2^27 K+ -> 3 pi 2595 us in runs of 1, 2059 of 4; 4 bodies 3583, 3159 of 16); 2
// for 2 bodies (4e6: 55.5, 43.3, 44.0); 4 for more than 4 (2e7 6-body elements in
// runs of 1, 2, 4 and 16: 774, 738, 723, 776 us).
constexpr uint64_t kRangeLongRuns = 1 << 25;  // elements
inline uint32_t range_run_max(int N, uint64_t n) {
  if (N == 2) return 2;
  if (N >= 5) return 4;
  return n <= kRangeLongRuns ? 1 : (N == 3 ? 4 : 16);
}

template <int N>
static void gen_one(RangeArgs a, hipStream_t s) {
  const uint64_t ngroups = (a.n + kWave - 1) / kWave;
  a.run = run_groups(ngroups, range_run_max(N, a.n));
  const unsigned g = blocks_for_runs(ngroups, a.run);
  hipLaunchKernelGGL(k_range_generate<N>, dim3(g), dim3(kBlock), 0, s, a);
}

template <int N>
static void hist_one(RangeArgs a, hipStream_t s) {
  const uint64_t nslots = a.h.nbins + 2;
  a.use_lds = nslots <= a.lds_slots ? 1 : 0;
  const size_t lds = a.use_lds ? nslots * sizeof(double) : 0;
  // 8 waves per SIMD while the private bins are small, at least four groups per
  // wave beyond one block per CU
  const uint64_t ngroups = (a.n + kWave - 1) / kWave;
  const uint64_t block_waves =
      ngroups <= range_few_groups(N) && nslots <= kRangeFewSlots ? kBlock / kWave
                                                                 : kRangeHistBlock / kWave;
  const uint64_t cap = (a.use_lds && lds > 32768) ? 256 : 1024;
  const uint64_t few = std::min<uint64_t>(256, (ngroups + block_waves - 1) / block_waves);
  const unsigned g = (unsigned)std::max(
      few, std::min<uint64_t>(cap, (ngroups + 4 * block_waves - 1) / (4 * block_waves)));
  const uint64_t nwaves = g * block_waves;
  a.run = (uint32_t)((ngroups + nwaves - 1) / nwaves);
  hipLaunchKernelGGL(k_range_hist<N>, dim3(g), dim3((unsigned)(block_waves * kWave)), lds, s, a);
}

template <int... I>
static constexpr auto gen_table(std::integer_sequence<int, I...>) {
  return std::array<void (*)(RangeArgs, hipStream_t), sizeof...(I)>{&gen_one<I + 2>...};
}
template <int... I>
static constexpr auto hist_table(std::integer_sequence<int, I...>) {
  return std::array<void (*)(RangeArgs, hipStream_t), sizeof...(I)>{&hist_one<I + 2>...};
}
static const auto kGen = gen_table(std::make_integer_sequence<int, HPSP_MAX_N - 1>{});
static const auto kHist = hist_table(std::make_integer_sequence<int, HPSP_MAX_N - 1>{});

int launch_range_generate(int N, const RangeArgs& a, hipStream_t s) {
  if (a.n == 0) return (int)hipSuccess;
  kGen[N - 2](a, s);
  return (int)hipGetLastError();
}

int launch_range_histogram(int N, const RangeArgs& a, hipStream_t s) {
  launch_zero(a.contents, a.h.nbins + 2, s);
  if (a.n == 0) return (int)hipGetLastError();
  kHist[N - 2](a, s);
  return (int)hipGetLastError();
}

}  // namespace hpsp
