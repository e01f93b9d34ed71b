// hydra::phase_space_range on gfx950 (PhaseSpaceRange.inl:44-72): element k
// of the lazy range is GenerateDecay<N, minstd_rand>(mother, masses,
// seed)(k) = (weight, p_1, ..., p_N) (GenerateDecay.h:203-343), the GENBOD
// event of DecayMother with the engine discarded by k + 3N.  Built with
// -ffp-contract=off.
//
// Engine words.  minstd_rand's word j of element first + k is
// x_start * a^(k + j) mod m (a = 48271, m = 2^31 - 1).  A wave takes runs of
// consecutive groups of 64 elements, whose words it shares through LDS
// (WindowView): a lane evaluates the word 64 after its last one, one product
// with a^64, for each further group.  A run's first words cost one power of
// a, formed on the scalar unit, and a table lookup; a wave's next run one
// product with a^(the events between).
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
  uint32_t x0;  // the lane's word at the run's first group
  uint32_t x;   // its last word

  // the first run, whose first element is k0
  __device__ __forceinline__ void first(uint32_t x_start, uint64_t k0, int lane) {
    const uint32_t xw = minstd_mul(x_start, minstd_pow(k0));
    x0 = minstd_mul(xw, kPow.v[lane]);
  }
  // the run's first group, or the group after the last
  __device__ __forceinline__ void next(Window& win, int lane, bool restart) {
    if (restart) {
      x = minstd_mul(x0, kMinstdA64);
      const uint32_t lo[1] = {x0}, hi[1] = {x};
      v.start(win, lane, 0, lo, hi);
    } else {
      x = minstd_mul(x, kMinstdA64);
      const uint32_t hi[1] = {x};
      v.shift(hi);
    }
  }
  // the wave's next run
  __device__ __forceinline__ void skip(uint32_t a_stride) { x0 = minstd_mul(x0, a_stride); }
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
  const uint64_t nruns = (ngroups + a.run - 1) / a.run;
  const uint64_t nwaves = (uint64_t)gridDim.x * (kBlock / kWave);
  uint64_t run = (uint64_t)blockIdx.x * (kBlock / kWave) + (uint64_t)wave;
  RangeWords<N> words;
  words.first(a.x_start, run * a.run * kWave, lane);
  for (; run < nruns; run += nwaves) {
    const uint64_t g_first = run * a.run;
    const uint64_t g_end = (g_first + a.run < ngroups) ? g_first + a.run : ngroups;
    for (uint64_t g = g_first; g < g_end; ++g) {
      const uint64_t k0 = g * kWave;
      words.next(win[wave], lane, g == g_first);
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
    }
    words.skip(a.a_stride);
  }
}

// Threads of a fill's block: every block adds its bins to the contents in the
// end, and those atomics, blocks times bins on few cache lines, not the
// elements set the time of smaller fills (1e6 elements into 100 bins: 2048
// blocks of 256 threads 53 us, 512 of them 31).
constexpr int kRangeHistBlock = 512;

template <int N>
__global__ __launch_bounds__(kRangeHistBlock)
    __attribute__((amdgpu_waves_per_eu(N <= 6 ? waves_for(N) : 2, 8)))
void k_range_hist(const RangeArgs a) {
  extern __shared__ double bins[];
  __shared__ typename RangeWords<N>::Window win[kRangeHistBlock / kWave];
  const uint64_t nslots = a.h.nbins + 2;
  if (a.use_lds) {
    for (uint64_t b = threadIdx.x; b < nslots; b += kRangeHistBlock) bins[b] = 0.0;
    __syncthreads();
  }
  const int lane = __lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint64_t ngroups = (a.n + kWave - 1) / kWave;
  const uint64_t nruns = (ngroups + a.run - 1) / a.run;
  const uint64_t nwaves = (uint64_t)gridDim.x * (kRangeHistBlock / kWave);
  uint64_t run = (uint64_t)blockIdx.x * (kRangeHistBlock / kWave) + (uint64_t)wave;
  RangeWords<N> words;
  words.first(a.x_start, run * a.run * kWave, lane);
  for (; run < nruns; run += nwaves) {
    const uint64_t g_first = run * a.run;
    const uint64_t g_end = (g_first + a.run < ngroups) ? g_first + a.run : ngroups;
    for (uint64_t g = g_first; g < g_end; ++g) {
      const uint64_t k = g * kWave + (uint64_t)lane;
      words.next(win[wave], lane, g == g_first);
      double p[N][4];
      const double wt = range_event<N>(a.d, words, p);
      if (k >= a.n) continue;
      double x[HPSP_HIST_MAX_DIM];
#pragma unroll
      for (int d = 0; d < HPSP_HIST_MAX_DIM; ++d)
        x[d] = (d < a.h.ndim) ? functor_eval<double>(a.axes[d], p) : 0.0;
      const double w = a.weight_mode == HPSP_HIST_WEIGHT_GENERATION ? wt
                       : a.weight_mode == HPSP_HIST_WEIGHT_PHSP
                           ? event_weight_f64<N>(p, a.d.m, a.d.maxw)
                           : 1.0;
      const uint64_t key = hist_key(a.h, x);
      if (key == kDrop) continue;
      if (a.use_lds)
        atomicAdd(&bins[key], w);
      else
        unsafeAtomicAdd(&a.contents[key], w);
    }
    words.skip(a.a_stride);
  }
  if (a.use_lds) {
    __syncthreads();
    for (uint64_t b = threadIdx.x; b < nslots; b += kRangeHistBlock) {
      const double v = bins[b];
      if (v != 0.0) unsafeAtomicAdd(&a.contents[b], v);
    }
  }
}

// ---------------------------------------------------------------------------

// Runs of the generation kernel as k_generate_f64's, dispatched in order
// (bound by its stores up to 3 daughters); the events from a wave's run to its
// next one are a power of a formed here.
template <int N>
static void gen_one(RangeArgs a, hipStream_t s) {
  const uint64_t ngroups = (a.n + kWave - 1) / kWave;
  a.run = run_groups(ngroups, N <= 3 ? kRunMaxStores : kRunMax);
  const unsigned g = grid_for_runs((ngroups + a.run - 1) / a.run);
  a.a_stride = minstd_pow((uint64_t)g * (kBlock / kWave) * a.run * kWave);
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
  constexpr uint64_t kWaves = kRangeHistBlock / kWave;
  const uint64_t cap = (a.use_lds && lds > 32768) ? 256 : 1024;
  const uint64_t few = std::min<uint64_t>(256, (ngroups + kWaves - 1) / kWaves);
  const unsigned g = (unsigned)std::max(
      few, std::min<uint64_t>(cap, (ngroups + 4 * kWaves - 1) / (4 * kWaves)));
  // one run per wave: nothing is stored on the way
  const uint64_t nwaves = g * kWaves;
  const uint64_t per = (ngroups + nwaves - 1) / nwaves;
  a.run = (uint32_t)(per < 1 ? 1 : (per < (1u << 20) ? per : (1u << 20)));
  a.a_stride = minstd_pow(nwaves * a.run * kWave);
  hipLaunchKernelGGL(k_range_hist<N>, dim3(g), dim3(kRangeHistBlock), lds, s, a);
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
