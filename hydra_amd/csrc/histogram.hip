// Dense histograms on gfx950: DenseHistogram<double, D>::Fill
// (DenseHistogram.inl:49-105, 174-222) for D = 1..HPSP_HIST_MAX_DIM.
//
// The reference computes every event's bin key (GetGlobalBin.h:41-209), sorts
// keys and weights, reduces by key and scatters the sums into nbins + 2
// contents.  Here each block keeps private bins in LDS and adds its events
// with FP64 LDS atomics, then adds its non-empty bins into the contents with
// device atomics; nothing is sorted.  Bin keys are computed with the
// reference's operations, so every event lands in the same bin; the order of
// the additions inside a bin differs (sums agree to rounding, unit-weight
// counts exactly).  Built with -ffp-contract=off.
//
// Sources of the axis values:
//   columns  D value columns (the reference's data range) and an optional
//            weight column;
//   events   the events of a Decays container in SoA columns, each axis a
//            functor of the event (the lazy `events | dalitz_calculator` of
//            phsp_basic.inl:196-214, fused into the fill), weights from a
//            column, the PhaseSpaceWeight of the event, or 1; the daughters
//            are filled from as particles where the axes read few of them;
//   particles  stored four-vectors given particle by particle (a melded
//            decay chain, phsp_chain.inl:244), read only where a functor
//            uses them; weights from a column or 1.
#include <algorithm>
#include <array>
#include <utility>

#include "hist_key.h"

namespace hpsp {

// s_waitcnt vmcnt(0) alone: export and LDS counters at their maxima.
constexpr int kWaitLoads = 0xF70;

// From here on an event with a PhaseSpaceWeight has its axes from memory, not from
// the daughters in registers, where they read fewer four-vectors than there are
// daughters (FEW): 4N momenta beside a functor's selections spilled, and what an
// axis reads is read again for the weight from L2 (1e7 events, two pair masses: 10
// bodies 795 -> 607 us; 9 bodies 541 -> 584, 8 bodies 480 -> 532).  Axes that read
// more stay with the registers (10 bodies, three Breit-Wigner terms and a helicity
// cosine: 794 us against 1057).
constexpr int kMemAxes = 10;

// Bound by the columns it reads: 3-body events with a weight column at 6.2 TB/s.
// Without a PhaseSpaceWeight to form, a wave of a large fill waits for each
// daughter's four columns before it asks for the next (kByDaughter beside the
// weight's mode): with all 12 or 13 columns asked for at once the same bytes came
// slower (2e7 3-body events 327 -> 306 us, 4-body ones 428 -> 412), and more bytes
// in flight from a look ahead at the next event gained nothing.  From kWaitEvents
// on: with 1e6 events both take the same time, and below, where a wave has one
// group of events or two, the waits are its time (1e5 3-body events 10.7 us
// against 10.3, 4-body ones 12.3 against 11.6); 5 and more bodies come here where
// the axes read as many, and wait at every size.  From 9 bodies on the selections
// bound it, and the waits cost; with a PhaseSpaceWeight they do at every size (2e7
// 3-body events 331 -> 337 us, 4-body ones 449 -> 457).
constexpr uint64_t kWaitEvents = 1 << 21;
constexpr int kByDaughter = 8;  // added to the mode

template <int N, bool FEW>
__device__ __forceinline__ void event_axes(const HistArgs& a, uint64_t k,
                                           double (&x)[HPSP_HIST_MAX_DIM], double& w) {
  if constexpr (FEW) {
    const MemAcc acc{a.parts, k};
#pragma unroll
    for (int d = 0; d < HPSP_HIST_MAX_DIM; ++d)
      x[d] = (d < a.h.ndim) ? functor_eval_acc<double, true>(a.axes[d], acc) : 0.0;
  }
  double p[N][4];
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (N >= 3 && N <= 8 && c == 0 && i > 0 &&
          (N <= 4 ? a.weight_mode >= kByDaughter : a.weight_mode != HPSP_HIST_WEIGHT_PHSP)) {
        __builtin_amdgcn_s_waitcnt(kWaitLoads);
        __builtin_amdgcn_sched_barrier(0);
      }
      p[i][c] = a.cols[(uint64_t)(4 * i + c) * a.ld + k];
    }
  if constexpr (!FEW) {
#pragma unroll
    for (int d = 0; d < HPSP_HIST_MAX_DIM; ++d) {
      // 4 bodies: the six pairs before the branch on the axis' kind cost registers
      // (122 against 111; 2e4 events 11.0 -> 10.8 us, 1e5 11.4 -> 11.1); 3 and 7
      // bodies with the weight lose by it (1e6 events 26 -> 27, 50 -> 52)
      if constexpr (N == 4) {
        x[d] = (d < a.h.ndim) ? functor_late<true, true>(a.axes[d], p) : 0.0;
      } else {
        const RegAcc<double, N, (N <= 8)> acc(p, wants_pairs(a.axes[d]));
        x[d] = (d < a.h.ndim) ? functor_eval_acc<double, true>(a.axes[d], acc) : 0.0;
      }
    }
  }
  if ((N <= 4 ? a.weight_mode % kByDaughter : a.weight_mode) == HPSP_HIST_WEIGHT_COLUMN)
    w = a.w[k];
  else if (a.weight_mode == HPSP_HIST_WEIGHT_PHSP)
    w = event_weight_f64<N>(p, a.d.m, a.d.maxw);
  else
    w = 1.0;
}

// N = 0: axis values from columns; N >= 2: from the events' momenta.
template <int N, bool FEW = false>
__global__ __launch_bounds__(kHistBlock) void k_hist_fill(const HistArgs a) {
  extern __shared__ double bins[];
  const uint64_t nslots = a.h.nbins + 2;
  if (a.use_lds) {
    for (uint64_t b = threadIdx.x; b < nslots; b += kHistBlock) bins[b] = 0.0;
    __syncthreads();
  }
  const uint64_t stride = (uint64_t)gridDim.x * kHistBlock;
  for (uint64_t k = (uint64_t)blockIdx.x * kHistBlock + threadIdx.x; k < a.n; k += stride) {
    double x[HPSP_HIST_MAX_DIM];
    double w;
    if constexpr (N == 0) {
#pragma unroll
      for (int d = 0; d < HPSP_HIST_MAX_DIM; ++d)
        x[d] = (d < a.h.ndim) ? a.x[(uint64_t)d * a.ldx + k] : 0.0;
      w = a.w ? a.w[k] : 1.0;
    } else if constexpr (N < 0) {
      const MemAcc acc{a.parts, k};
#pragma unroll
      for (int d = 0; d < HPSP_HIST_MAX_DIM; ++d)
        x[d] = (d < a.h.ndim) ? functor_eval_acc<double, true, true>(a.axes[d], acc) : 0.0;
      w = a.w ? a.w[k] : 1.0;
    } else {
      event_axes<N, FEW>(a, k, x, w);
    }
    const uint64_t key = hist_key(a.h, x);
    if (key == kDrop) continue;
    if (a.use_lds)
      atomicAdd(&bins[key], w);
    else
      unsafeAtomicAdd(&a.contents[key], w);
  }
  if (a.use_lds) {
    __syncthreads();
    for (uint64_t b = threadIdx.x; b < nslots; b += kHistBlock) {
      const double v = bins[b];
      if (v != 0.0) unsafeAtomicAdd(&a.contents[b], v);
    }
  }
}

__global__ void k_zero(double* p, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = 0.0;
}

void launch_zero(double* p, uint64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_zero, dim3((unsigned)std::min<uint64_t>((n + 255) / 256, 1024)),
                     dim3(256), 0, s, p, n);
}

// Four-vectors that an axis reads of an event.
static int axis_reads(const FunctorK& f) {
  switch (f.kind) {
    case HPSP_F_ONE: return 0;
    case HPSP_F_BW_SUM: return 2 * f.nterms;
    case HPSP_F_COS_HELICITY: return f.t[1].b + 2;
    default: return 2;
  }
}

template <int N>
static void hist_one(const HistArgs& a, unsigned grid, size_t lds, bool few, hipStream_t s) {
  if constexpr (N >= kMemAxes) {
    if (few) {
      hipLaunchKernelGGL((k_hist_fill<N, true>), dim3(grid), dim3(kHistBlock), lds, s, a);
      return;
    }
  }
  hipLaunchKernelGGL(k_hist_fill<N>, dim3(grid), dim3(kHistBlock), lds, s, a);
}

template <int... I>
static constexpr auto hist_table(std::integer_sequence<int, I...>) {
  return std::array<void (*)(const HistArgs&, unsigned, size_t, bool, hipStream_t), sizeof...(I)>{
      &hist_one<(I == 0 ? 0 : I + 1)>...};
}
// index 0: columns; index N - 1 (N = 2..HPSP_MAX_N): events of N daughters
static const auto kHist = hist_table(std::make_integer_sequence<int, HPSP_MAX_N>{});

int launch_histogram_fill(int N, const HistArgs& in, hipStream_t s) {
  HistArgs a = in;
  const uint64_t nslots = a.h.nbins + 2;
  launch_zero(a.contents, nslots, s);
  if (a.n == 0) return (int)hipGetLastError();
  bool few = false;
  if (N > 0) {  // the events' daughters as particles
    a.parts.n = N;
    for (int i = 0; i < N; ++i) {
      a.parts.cols[i] = a.cols + (uint64_t)(4 * i) * a.ld;
      a.parts.ld[i] = a.ld;
    }
    // Fewer four-vectors than daughters, and no weight that needs them all: the
    // particles' kernel reads those alone (1e7 events into two pair masses: 5
    // bodies 295 -> 233 us, 10 bodies 728 -> 230).  4 bodies read their four in
    // registers (4e7 events 869 us against 908), and so do axes that together
    // read a daughter twice.
    int reads = 0;
    for (int d = 0; d < a.h.ndim; ++d) reads += axis_reads(a.axes[d]);
    few = reads < N;
    if (a.weight_mode != HPSP_HIST_WEIGHT_PHSP) {
      if (N >= 5 && few) {
        if (a.weight_mode != HPSP_HIST_WEIGHT_COLUMN) a.w = nullptr;
        N = -1;
      } else if (N <= 4 && a.n >= kWaitEvents) {
        a.weight_mode += kByDaughter;
      }
    }
  }
  a.use_lds = nslots <= a.lds_slots ? 1 : 0;
  const size_t lds = a.use_lds ? nslots * sizeof(double) : 0;
  // one block per CU: each block's bins are added to the contents in the end, on
  // few cache lines where bins are few (400 bins, 2e6 3-body events: 1024 blocks
  // 54 us, 512 49, 256 43, 128 61; 10^4 bins: 512 66, 256 51, 128 65)
  const uint64_t want = (a.n + kHistBlock - 1) / kHistBlock;
  const uint64_t cap = a.use_lds ? 256 : 1024;
  const unsigned grid = (unsigned)std::min<uint64_t>(want, cap);
  if (N < 0)
    hist_one<-1>(a, grid, lds, few, s);
  else
    kHist[N == 0 ? 0 : N - 1](a, grid, lds, few, s);
  return (int)hipGetLastError();
}

// events | functors over stored particles: one event per lane, the functor
// columns written lane-contiguous.
__global__ __launch_bounds__(kBlock) void k_particles_eval(const PartEvalArgs a) {
  const uint64_t stride = (uint64_t)gridDim.x * kBlock;
  for (uint64_t k = (uint64_t)blockIdx.x * kBlock + threadIdx.x; k < a.n; k += stride) {
    const MemAcc acc{a.p, k};
    for (int j = 0; j < a.nf; ++j)
      a.out[(uint64_t)j * a.ld + k] = functor_eval_acc<double, true, true>(a.f[j], acc);
  }
}

int launch_particles_evaluate(const PartEvalArgs& a, hipStream_t s) {
  if (a.n == 0) return (int)hipSuccess;
  hipLaunchKernelGGL(k_particles_eval, dim3(grid_for(a.n, 1u << 16)), dim3(kBlock), 0, s, a);
  return (int)hipGetLastError();
}

}  // namespace hpsp
