// Engine words of consecutive events, shared through LDS.
//
// Event e of a Generate reads the W = 3N - 4 words of its engine's stream
// after discard(e + 3N): with the squares engines the words of counters
// e + 3N .. e + 3N + W - 1, with the Random123 ones the words of the blocks
// (2 or 4 words) of counters e + 3N + 1 .. e + 3N + NB, NB = ceil(W / A).  So
// neighbouring events read all but one of the same words or blocks.  A wave
// (EventWords, in AverageOn and the flags kernels) or a block
// (BlockEventWords, in Generate and the regenerating scatters) evaluates each word or
// block once and puts it into LDS; the event in lane l reads word j at slot
// l + j / A, an immediate offset from one address.  The kernels that read them
// are bound by their vector instructions: evaluating every block in every lane
// (Random123) took Generate of 3e6 4-body Threefry events 118 us against 102,
// Evaluate of 6e5 8-body Threefry4x64 ones 52 against 42; one ds_bpermute, a
// select and its address per word (squares engines) took the 10-body Generate
// of 2^24 events 1.57 ms against 1.51, the mixed one 685 us against 659.
//
// The counter of a Random123 block is two 64-bit words: e + 3N wraps in 64
// bits, the steps from there carry into the second.  In the one group of
// events that wraps inside (first + n near 2^64) the lanes before and after
// the wrap need different blocks for the same slot: those after it read NB
// slots further on, where their own blocks are put.
#pragma once

#include "hpsp_launch.h"

namespace hpsp {

template <typename T>
using lptr = __attribute__((address_space(3))) T*;

template <int ENGINE>
using word_t = std::conditional_t<narrow_words<ENGINE>(), uint32_t, uint64_t>;

// Orders a wave's LDS stores before its later LDS loads and the other way
// round (the hardware runs a wave's LDS operations in order).
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Slots of consecutive words (A = 1) or blocks of A words for a wave's groups:
// a group's 64 + NB - 1 slots start at 0 or at 64 in turn, so that the 64
// slots after its first are the next group's first and stay where they are.
template <typename T, int A, int NB>
struct WordWindow {
  static constexpr int kSlots = 2 * kWave + NB - 1;
  T w[A][kSlots];
};

// A lane's view of its wave's window.
template <typename T, int A, int NB>
struct WindowView {
  using Win = WordWindow<T, A, NB>;
  lptr<T> p;  // word 0 of this lane's event
  lptr<T> w;  // the window
  int lane;
  bool odd;  // the group's slots start at 64

  // slots 0 .. 127; this lane's event starts at slot lane + shift
  __device__ __forceinline__ void start(Win& win, int l, int shift, const T (&lo)[A],
                                        const T (&hi)[A]) {
    lane = l;
    w = (lptr<T>)&win.w[0][0];
    odd = false;
    wave_lds_fence();
#pragma unroll
    for (int e = 0; e < A; ++e) {
      w[e * Win::kSlots + lane] = lo[e];
      w[e * Win::kSlots + kWave + lane] = hi[e];
    }
    wave_lds_fence();
    p = w + (lane + shift);
  }
  // the next group: its last 64 slots are hi
  __device__ __forceinline__ void shift(const T (&hi)[A]) {
    wave_lds_fence();
#pragma unroll
    for (int e = 0; e < A; ++e) {
      w[e * Win::kSlots + (odd ? kWave : 0) + lane] = hi[e];
      if (!odd && lane < NB - 1) w[e * Win::kSlots + 2 * kWave + lane] = hi[e];
    }
    wave_lds_fence();
    p += odd ? -kWave : kWave;
    odd = !odd;
  }
  __device__ __forceinline__ T get(int j) const { return p[(j % A) * Win::kSlots + j / A]; }
};

// Where the blocks of the events d0 + l (d0 the first one's e + 3N) lie: slot
// s holds the block of counter d0 + 1 + s, carried into the second word; where
// an event's own e + 3N wraps (l >= before) its slots are NB further on.
template <int NB>
struct BlockSlots {
  uint64_t d0;
  uint64_t before;  // events before the wrap; ~0 where none wraps
  __device__ __forceinline__ BlockSlots(uint64_t d0_, uint32_t events) : d0(d0_) {
    before = (d0 > ~0ULL - (events - 1)) ? 0 - d0 : ~0ULL;
  }
  __device__ __forceinline__ int shift(uint32_t l) const { return l < before ? 0 : NB; }
  template <int ENGINE, int A>
  __device__ __forceinline__ void eval(const uint64_t* key, uint32_t s, uint64_t (&out)[A]) const {
    const bool wrapped = s > before + (NB - 1) && before != ~0ULL;
    const uint64_t step = 1 + (uint64_t)(wrapped ? s - NB : s);
    uint64_t c[4] = {d0 + step, 0, 0, 0};
    c[1] = (!wrapped && c[0] < step) ? 1 : 0;
    uint64_t o[4];
    r123_block<ENGINE>(key, c, o);
#pragma unroll
    for (int e = 0; e < A; ++e) out[e] = o[e];
  }
};

// The one block of an event whose e + 3N is d.
template <int ENGINE, int A>
__device__ __forceinline__ void event_block(const uint64_t* key, uint64_t d, uint64_t (&out)[A]) {
  const uint64_t c[4] = {d + 1, d + 1 == 0 ? 1ULL : 0ULL, 0, 0};
  uint64_t o[4];
  r123_block<ENGINE>(key, c, o);
#pragma unroll
  for (int e = 0; e < A; ++e) out[e] = o[e];
}

// The first W words of each event of a wave's groups, taken in order.
template <int N, int ENGINE, int W = 3 * N - 4>
struct EventWords {
  using T = word_t<ENGINE>;
  static constexpr int A = engine_arity<ENGINE>();
  static constexpr int NB = (W + A - 1) / A;
  static constexpr bool kShared = NB > 1;  // else every lane evaluates its own
  using View = WindowView<T, A, kShared ? NB : 1>;
  struct Nothing {};
  using Window = std::conditional_t<kShared, typename View::Win, Nothing>;  // __shared__, per wave
  View v;
  T own[A];
  uint64_t y;  // squares: key * counter of the lane's last word
  bool again;  // Random123: the next group starts its window anew

  // The group of 64 events whose first is wave_first_evt; restart: not the
  // one that follows the last call's.
  __device__ __forceinline__ void next(Window& win, const DecayK& d, uint64_t wave_first_evt,
                                       int lane, bool restart) {
    const uint64_t d0 = wave_first_evt + 3 * (uint64_t)N;
    if constexpr (W == 0) {
    } else if constexpr (is_squares<ENGINE>()) {
      const uint64_t key = d.key[0];
      if (restart) {
        y = key * (d0 + (uint64_t)lane);
        own[0] = squares_word_y<ENGINE>(key, y);
        if constexpr (kShared) {
          y += key << 6;  // counter + 64
          const T hi[1] = {squares_word_y<ENGINE>(key, y)};
          v.start(win, lane, 0, own, hi);
        }
      } else {
        y += key << 6;
        own[0] = squares_word_y<ENGINE>(key, y);
        if constexpr (kShared) v.shift(own);
      }
    } else if constexpr (!kShared) {
      event_block<ENGINE>(d.key, d0 + (uint64_t)lane, own);
    } else {
      if (restart || again) {
        const BlockSlots<NB> b(d0, kWave);
        uint64_t o[2][A];
#pragma unroll
        for (int h = 0; h < 2; ++h) b.template eval<ENGINE, A>(d.key, lane + h * kWave, o[h]);
        v.start(win, lane, b.shift(lane), o[0], o[1]);
        again = d0 > ~0ULL - 4 * kWave;
      } else {
        // slot 64 + lane of a group away from the wrap
        uint64_t c[4] = {d0 + 1 + kWave + (uint64_t)lane, 0, 0, 0}, o[4];
        r123_block<ENGINE>(d.key, c, o);
        uint64_t hi[A];
#pragma unroll
        for (int e = 0; e < A; ++e) hi[e] = o[e];
        v.shift(hi);
        again = d0 > ~0ULL - 4 * kWave;
      }
    }
  }
  __device__ __forceinline__ uint64_t operator()(int j) const {
    if constexpr (kShared)
      return v.get(j);
    else
      return own[j];
  }
};

// The words of the kBlock consecutive events of a block, one per thread.  Events
// that need a single Random123 block (2 bodies) have none to share: each thread
// keeps its own (through LDS, 4e6 2-body events of Philox4x64 57 us against 47).
template <int N, int ENGINE>
struct BlockEventWords {
  using T = word_t<ENGINE>;
  static constexpr int W = 3 * N - 4;
  static constexpr int A = engine_arity<ENGINE>();
  static constexpr int NB = (W + A - 1) / A;
  static constexpr int kSlots = kBlock + (is_squares<ENGINE>() ? NB - 1 : 2 * NB);
  static constexpr bool kShared = NB > 1;
  struct Words {
    T w[A][kSlots];
  };
  struct Nothing {};
  using Store = std::conditional_t<kShared, Words, Nothing>;  // __shared__
  lptr<T> p;
  T own[kShared ? 1 : A];  // word 0; all of them

  // Event first + t in thread t; every thread of the block calls it.
  __device__ __forceinline__ void fill(Store& s, const DecayK& d, uint64_t first) {
    const uint32_t t = threadIdx.x;
    const uint64_t d0 = first + 3 * (uint64_t)N;
    if constexpr (is_squares<ENGINE>()) {
      const uint64_t key = d.key[0];
      own[0] = squares_word_y<ENGINE>(key, key * (d0 + t));
      s.w[0][t] = own[0];
      if (t < (uint32_t)(NB - 1))
        s.w[0][kBlock + t] = squares_word_y<ENGINE>(key, key * (d0 + kBlock + t));
      __syncthreads();
      p = (lptr<T>)&s.w[0][t];
    } else if constexpr (!kShared) {
      event_block<ENGINE>(d.key, d0 + t, own);
    } else {
      const BlockSlots<NB> b(d0, kBlock);
      const uint32_t slots = kBlock + (b.before == ~0ULL ? NB - 1 : 2 * NB);
      for (uint32_t k = t; k < slots; k += kBlock) {
        uint64_t o[A];
        b.template eval<ENGINE, A>(d.key, k, o);
#pragma unroll
        for (int e = 0; e < A; ++e) s.w[e][k] = o[e];
      }
      __syncthreads();
      p = (lptr<T>)&s.w[0][t + b.shift(t)];
      own[0] = p[0];
    }
  }
  __device__ __forceinline__ uint64_t operator()(int j) const {
    if constexpr (kShared)
      return j == 0 ? own[0] : p[(j % A) * kSlots + j / A];
    else
      return own[j];
  }
};

}  // namespace hpsp
