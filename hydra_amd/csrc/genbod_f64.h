// FP64 GENBOD for one event, the engine-word sources it reads, and the
// AverageOn and Evaluate kernels, templated over the functor they evaluate:
// instantiated with described functors by the library (genbod_f64.hip,
// evaluate.hip) and with users' callables by translation units that include
// hydra_amd/include/hydra/detail/UserKernels.h.  Every function turns
// floating-point contraction off itself, so the operation sequence holds
// under any contraction flag that honours pragmas.  The weight chain (uniforms,
// invMas, pdk, the weight product) repeats the reference's double operations
// one for one with correctly rounded sqrt and division, so weights agree bit
// for bit (DecayMother.h:170-212).  The momenta (DecayMother.h:218-269) are
// formed with the same operations except: exactly-zero terms are dropped,
// products and sums are fused (one rounding instead of two), sin/cos and
// square roots outside the weight chain are evaluated to about one ulp, and
// the boost factors use gamma*beta = p/M, gamma = sqrt(1 + (p/M)^2).
//
// GENBOD is bound by its vector instructions.  The fused forms, the weight
// chain and PhaseSpaceWeight without a branch and a library path per square
// root, one reciprocal per invariant mass for the chain's division and the
// boost, and the decay's constants formed on the host took the 10-body
// Generate of 2^24 events from 1.89 to 1.57 ms, AverageOn of the 3-body Dalitz
// model over 2^24 events from 239 to 221 us, Evaluate of 10^7 events from 174 to
// 164 us.  gamma from gamma beta (one square root, no selects), the first
// boost's back-to-back pair formed once and no guard on the energies' square
// roots: AverageOn 208 -> 199 us, the 10-body Generate and Evaluate 2-5%
// in one run.  Now, in other runs, 1e6 3-body events 21-23 us, the 10-body Generate
// 1.50 ms, AverageOn 197 us, Evaluate 143 us.  The momenta's errors against extended
// precision did not grow (3 bodies: 2.28 -> 2.24e-16 E RMS; 10: 1.51 -> 1.47e-15).
#pragma once

#include <type_traits>

#include "event_words.h"
#include "hpsp_launch.h"

namespace hpsp {

// GENBOD for one event (DecayMother::process).  word(j) yields the j-th
// engine word of the event's stream (after discard(evt + 3N)).
template <int N, int ENGINE, typename WordFn>
__device__ __forceinline__ double genbod_f64(const DecayK& d, const WordFn& word,
                                             double (&p)[N][4]) {
#pragma clang fp contract(off)
  double rno[N];
  rno[0] = 0.0;
  rno[N - 1] = 1.0;
  if constexpr (N > 2) {
    using WT = std::conditional_t<narrow_words<ENGINE>(), uint32_t, uint64_t>;
    WT v[N - 2];
#pragma unroll
    for (int k = 0; k < N - 2; ++k) v[k] = (WT)word(k);
    sort_net(v);
#pragma unroll
    for (int k = 0; k < N - 2; ++k) rno[k + 1] = to_unit<ENGINE>(v[k]);
  }

  double invMas[N];
  invMas[0] = d.mas0;
  invMas[N - 1] = d.masN;
#pragma unroll
  for (int n = 1; n < N - 1; ++n) invMas[n] = rno[n] * d.ecm + d.msum[n];

  // The weight chain without a branch per square root: every radicand is
  // taken to lie in sqrt_core's range; the events of which one does not (a
  // pair of equal mass uniforms, masses out of the ordinary) repeat the chain
  // with the library's square root and division.  RN(s / (2 a)) =
  // RN(s / a) / 2, with the reciprocal of invMas[n] shared with the boost.  Two
  // bodies have the same momentum in every event, formed on the host (in the
  // event loops of AverageOn and the range the chain's branch kept it from being
  // formed once: 4e6 events 30.1 us against 25.6).
  double wt = d.maxw;
  double pd[N - 1];
  // gamma beta of the boost of step i = 1 .. N-2, pd[i] / invMas[i]
  [[maybe_unused]] double gb[N - 1];
  if constexpr (N == 2) {
    pd[0] = d.pd2;
    wt *= pd[0];
  } else {
    double ra = 0.0;  // 1 / invMas[n]
    bool ok = d.plain != 0;
#pragma unroll
    for (int n = 0; n < N - 1; ++n) {
      const double a = invMas[n + 1];
      const double x = pdk_radicand(a, invMas[n], d.m[n + 1]);
      ok = ok & sqrt_range(x);
      const double rn = n < N - 2 ? rcp_fast(a) : d.rmasN;
      pd[n] = 0.5 * div_core(sqrt_core(x), a, rn);
      wt *= pd[n];
      if (n > 0) gb[n] = pd[n] * ra;
      ra = rn;
    }
    if (__builtin_expect(!ok, 0)) {
      wt = d.maxw;
#pragma unroll
      for (int n = 0; n < N - 1; ++n) {
        pd[n] = __builtin_sqrt(pdk_radicand(invMas[n + 1], invMas[n], d.m[n + 1])) /
                (2 * invMas[n + 1]);
        wt *= pd[n];
        // for pd = 0 (beta = 0; NaN) the reference's boost does nothing
        if (n > 0) gb[n] = pd[n] > 0.0 ? pd[n] * rcp_fast(invMas[n]) : 0.0;
      }
    }
  }

  // Daughter 0 along +y; it is rotated for the first time at i = 1.
  p[0][0] = sqrt_pos(__builtin_fma(pd[0], pd[0], d.msq[0]));
  p[0][1] = 0.0;
  p[0][2] = pd[0];
  p[0][3] = 0.0;

  [[maybe_unused]] double y0 = 0.0, gy0 = 0.0;  // step 1: py of daughter 0, gamma py
#pragma unroll
  for (int i = 1; i < N; ++i) {
    // keep the scheduler from hoisting later steps' angles and boosts
    // above this one: their results would all be live at once
    if constexpr (N > 4) __builtin_amdgcn_sched_barrier(0);
    p[i][0] = sqrt_pos(__builtin_fma(pd[i - 1], pd[i - 1], d.msq[i]));
    p[i][1] = 0.0;
    p[i][2] = -pd[i - 1];
    p[i][3] = 0.0;

    const double cZ = to_cos<ENGINE>(word(N - 2 + 2 * (i - 1)));
    const double sZ = sqrt_fast(__builtin_fma(-cZ, cZ, 1.0));
    // sin/cos of angY = 2*pi*u
    double sY, cY;
    if constexpr (is_squares<ENGINE>())
      sincos_2pi_w32((uint32_t)word(N - 2 + 2 * (i - 1) + 1), sY, cY);
    else
      sincos_2pi(to_unit<ENGINE>(word(N - 2 + 2 * (i - 1) + 1)), sY, cY);

#pragma unroll
    for (int j = 0; j <= i; ++j) {
      const bool fresh = (j == i) || (i == 1);  // px = pz = 0 before this rotation
      if (i == 1 && j == 1) {  // back to back with daughter 0
        p[1][1] = -p[0][1];
        p[1][2] = -p[0][2];
        p[1][3] = -p[0][3];
      } else if (fresh) {
        const double y = p[j][2];
        const double t = -(sZ * y);  // cZ*0 - sZ*y
        p[j][2] = cZ * y;            // sZ*0 + cZ*y
        p[j][1] = cY * t;            // cY*t - sY*0
        p[j][3] = sY * t;            // sY*t + cY*0
      } else {
        double x = p[j][1];
        const double y = p[j][2];
        p[j][1] = __builtin_fma(cZ, x, -(sZ * y));
        p[j][2] = __builtin_fma(sZ, x, cZ * y);
        x = p[j][1];
        const double z = p[j][3];
        p[j][1] = __builtin_fma(cY, x, -(sY * z));
        p[j][3] = __builtin_fma(sY, x, cY * z);
      }
    }
    if (i == N - 1) break;

    // Boost along +y by beta = pd/sqrt(pd^2 + M^2) (Vector3R(0, beta, 0)):
    // only E and py change.  The reference's gamma = 1/sqrt(1 - beta^2) and
    // gamma*beta are sqrt(1 + (pd/M)^2) and pd/M; (gamma-1)/beta^2 * beta^2 is
    // gamma - 1.  The momenta are formed as E' = gamma E + gamma beta py and
    // py' = gamma beta E + gamma py: for gamma beta = 0 as they were (up to the
    // sign of a zero py).
    {
      const double gby = gb[i];
      const double gamma = sqrt_pos(__builtin_fma(gby, gby, 1.0));
#pragma unroll
      for (int j = 0; j <= i; ++j) {
        const double e2 = p[j][0], py2 = p[j][2];
        if (i == 1 && j == 1) {  // py2 = -p[0][2] before this boost: its product with gamma
          p[1][0] = __builtin_fma(-gby, y0, gamma * e2);
          p[1][2] = __builtin_fma(gby, e2, -gy0);
        } else {
          if (i == 1) {
            y0 = py2;
            gy0 = gamma * py2;
          }
          p[j][0] = __builtin_fma(gby, py2, gamma * e2);
          p[j][2] = __builtin_fma(gby, e2, i == 1 ? gy0 : gamma * py2);
        }
      }
    }
  }
  return wt;
}

// AverageOn's value of a described functor: divisions through reciprocals
// (the result is compared within a tolerance, not bit for bit).  A user's
// callable brings its own overload (found by argument-dependent lookup).
template <int P>
__device__ __forceinline__ double avg_value(const FunctorFastK& f, const double (&p)[P][4]) {
  if constexpr (P <= 4)
    return functor_late<false, true>(f, p);
  else
    return functor_eval<double, false>(f, p);
}

// AverageOn: chunks of kAvgChunk consecutive events, one partial per chunk.
// Within a chunk accumulating wave w folds its own run of consecutive groups
// of 64 events (groups 16w .. 16w+15), lane l event l of each, in order; the
// four wave results merge in a fixed tree, so a partial depends only on its
// event range.
//
// WAVES = 4: each wave generates the groups it folds, the engine words
// carrying from group to group.  With fewer chunks than the chip holds blocks,
// the 16 groups in series set the time (a 5-body chunk in mixed precision: 33
// us), so for those WAVES = 16 or 8 waves generate the chunk's groups, stage
// every event's functor value and weight in LDS, and four of them fold the
// staged values in the same order: the same partial, bit for bit.
constexpr int avg_wide_waves(int N) { return N <= 6 ? 16 : 8; }  // 128 or 256 registers

// Waves per SIMD asked for of the form with four waves per chunk: up to 3 bodies 5
// would spill over mothers, which hold one more four-vector and a boost, and for 2
// bodies beside Philox' products.
constexpr int avg_waves_for(int N, int engine, bool mothers) {
  const bool philox = engine == HPSP_PHILOX || engine == HPSP_PHILOX_LONG;
  return N <= 3 && (mothers || (N == 2 && philox)) ? 4 : waves_for(N);
}

template <int N, int ENGINE, bool MOTHERS, typename FK = FunctorFastK, int WAVES = kBlock / kWave>
__global__ __launch_bounds__(WAVES * kWave)
    __attribute__((amdgpu_waves_per_eu(WAVES == 4 ? avg_waves_for(N, ENGINE, MOTHERS) : WAVES / 4,
                                       8)))
void k_average_f64(const AvgArgsT<FK> a) {
  constexpr int kFold = kBlock / kWave;  // waves that fold
  constexpr bool kWide = WAVES > kFold;
  constexpr int kGroups = kAvgChunk / kWave;
  __shared__ Stats sh[kFold];
  __shared__ double staged[2][kWide ? kAvgChunk : 1];  // functor values, weights
  __shared__ typename EventWords<N, ENGINE>::Window win[WAVES];
  const int lane = __lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint64_t nchunks = (a.n + kAvgChunk - 1) / kAvgChunk;
  for (uint64_t c = blockIdx.x; c < nchunks; c += gridDim.x) {
    Stats acc = {0.0, 0.0, 0.0};
    // a chunk with few events spreads them over all its waves
    const uint64_t left = (a.n - c * kAvgChunk + kWave - 1) / kWave;
    const int groups = kWide && left < kGroups ? (int)left : kGroups;
    const int per_wave = (groups + WAVES - 1) / WAVES;
    EventWords<N, ENGINE> words;
    for (int it = 0; it < per_wave; ++it) {
      const int g = wave * per_wave + it;
      const uint64_t k0 = c * kAvgChunk + (uint64_t)g * kWave;
      const uint64_t k = k0 + (uint64_t)lane;
      const bool live = k < a.n;
      if (kWide && g >= groups) break;  // wave-uniform
      words.next(win[wave], a.d, a.first + k0, lane, it == 0);
      double p[N + (MOTHERS ? 1 : 0)][4];
      double f, wt;
      if constexpr (MOTHERS) {
        double q[N][4];
        wt = genbod_f64<N, ENGINE>(a.d, words, q);
        const uint64_t km = live ? k : 0;
        double m4[4];
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) m4[cc] = a.mothers[(uint64_t)cc * a.mld + km];
        const double bx = m4[1] / m4[0], by = m4[2] / m4[0], bz = m4[3] / m4[0];
#pragma unroll
        for (int i = 0; i < N; ++i) {
          boost_general(q[i], bx, by, bz);
#pragma unroll
          for (int cc = 0; cc < 4; ++cc) p[i + 1][cc] = q[i][cc];
        }
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) p[0][cc] = m4[cc];
      } else {
        wt = genbod_f64<N, ENGINE>(a.d, words, p);
        if (a.d.do_boost) {
#pragma unroll
          for (int i = 0; i < N; ++i) boost_folded(p[i], a.d);
        }
      }
      f = avg_value(a.f, p);
      if constexpr (kWide) {
        staged[0][g * kWave + lane] = f;
        staged[1][g * kWave + lane] = wt;
      } else {
        if (live) stats_push(acc, f, wt);
      }
    }
    if constexpr (kWide) __syncthreads();
    if (!kWide || wave < kFold) {
      if constexpr (kWide) {
        for (int it = 0; it < kGroups / kFold; ++it) {
          const int t = (wave * (kGroups / kFold) + it) * kWave + lane;
          if (c * kAvgChunk + (uint64_t)t < a.n) stats_push(acc, staged[0][t], staged[1][t]);
        }
      }
      acc = wave_reduce_stats(acc);
      if (lane == 0) sh[wave] = acc;
    }
    __syncthreads();
    if (threadIdx.x == 0)
      a.partials[c] =
          stats_or_zero(stats_merge(stats_merge(sh[0], sh[1]), stats_merge(sh[2], sh[3])));
    __syncthreads();
  }
}

// Evaluate's values of described functors, exact divisions (the values are
// compared with the reference's bit for bit); out(j, value) stores functor
// j's.  A user's set of callables brings its own overload.
template <int P, typename Out>
__device__ __forceinline__ void eval_set(const DescSet& s, const double (&p)[P][4], Out&& out) {
  const RegAcc<double, P> acc(p, s.pairs != 0);
  for (int j = 0; j < s.nf; ++j) out(j, functor_eval_acc<double, true>(s.f[j], acc));
}

// Words of an engine seeded per event and not discarded.
template <int N, int ENGINE>
struct LaneWords {
  static constexpr int W = 3 * N - 4;
  uint64_t key[4];
  uint64_t w[is_squares<ENGINE>() ? 1 : W];

  __device__ __forceinline__ void init(uint64_t seed) {
    engine_keys_dev<ENGINE>(seed, key);
    if constexpr (!is_squares<ENGINE>()) r123_words<ENGINE, W>(key, 0, w);
  }
  __device__ __forceinline__ uint64_t operator()(int j) const {
    if constexpr (is_squares<ENGINE>())
      return squares_word<ENGINE>(key[0], (uint64_t)j);
    else
      return w[j];
  }
};

// Evaluate (EvalMother.h:283-306, EvalMothers.h:145-273): one group of 64
// events per wave, as k_generate_f64; over one mother the block's events share
// their engine words.
template <int N, int ENGINE, bool MOTHERS, typename FS = DescSet>
__global__ __launch_bounds__(kBlock)
    __attribute__((amdgpu_waves_per_eu(MOTHERS ? waves_for(N) : eval_waves_for(N), 8)))
void k_evaluate_f64(const EvalArgsT<FS> a) {
  struct Nothing {};
  __shared__ std::conditional_t<MOTHERS, Nothing, typename BlockEventWords<N, ENGINE>::Store> sw;
  const int lane = __lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const uint64_t kb = (uint64_t)blockIdx.x * kBlock;
  [[maybe_unused]] BlockEventWords<N, ENGINE> bwords;
  if constexpr (!MOTHERS) bwords.fill(sw, a.d, a.first + kb);
  const uint64_t k0 = kb + (uint64_t)(wave * kWave);
  if (k0 >= a.n) return;  // wave-uniform
  const uint64_t k = k0 + (uint64_t)lane;
  const bool live = k < a.n;
  constexpr int P = N + (MOTHERS ? 1 : 0);
  double p[P][4];
  double wt;
  if constexpr (MOTHERS) {
    const uint64_t km = live ? k : 0;
    double m4[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) m4[c] = a.mothers[(uint64_t)c * a.mld + km];
    // fECM = mother.mass() - sum(m); maximum weight of this mother
    // (EvalMothers.h:151-176)
    DecayK d = a.d;
    {
#pragma clang fp contract(off)
      double te = mass_of(m4[0], m4[1], m4[2], m4[3]);
#pragma unroll
      for (int i = 0; i < N; ++i) te -= d.m[i];
      d.mas0 = 0.0 * te + d.msum[0];
      d.masN = 1.0 * te + d.msum[N - 1];
      d.rmasN = rcp_fast(d.masN);
      d.plain = d.plain_m && te >= 0.0 && te <= 0x1p+299;
      if constexpr (N == 2) d.pd2 = pdk(d.masN, d.mas0, d.m[1]);
      double emmax = te + d.m[0], emmin = 0.0, wtmax = 1.0;
#pragma unroll
      for (int i = 1; i < N; ++i) {
        emmin += d.m[i - 1];
        emmax += d.m[i];
        wtmax *= pdk(emmax, emmin, d.m[i]);
      }
      d.ecm = te;
      d.maxw = 1.0 / wtmax;
    }
    LaneWords<N, ENGINE> words;
    words.init(pair_hash(a.first + k, a.seed));
    double q[N][4];
    wt = genbod_f64<N, ENGINE>(d, words, q);
    const double bx = m4[1] / m4[0], by = m4[2] / m4[0], bz = m4[3] / m4[0];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      boost_general(q[i], bx, by, bz);
#pragma unroll
      for (int c = 0; c < 4; ++c) p[i + 1][c] = q[i][c];
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) p[0][c] = m4[c];
  } else {
    wt = genbod_f64<N, ENGINE>(a.d, bwords, p);
    if (a.d.do_boost) {
#pragma unroll
      for (int i = 0; i < N; ++i) boost_folded(p[i], a.d);
    }
  }
  if (live) {
    double* out = a.out + k0;
    st(uniform_ptr(out) + lane, wt);
    eval_set(a.fs, p, [&](int j, double v) {
      st(uniform_ptr(out + (uint64_t)(1 + j) * a.ld) + lane, v);
    });
  }
}

}  // namespace hpsp
