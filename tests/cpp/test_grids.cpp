// over_grids and the arguments' parts (hpsp_launch.h): calls of more events than
// one launch holds, their addresses checked on the host (nothing is launched).
#include <cstdint>
#include <cstdio>
#include <vector>

#include "hpsp_launch.h"

using namespace hpsp;

static int failures = 0;
#define CHECK(x)                                              \
  do {                                                        \
    if (!(x)) {                                               \
      std::printf("%s:%d: %s\n", __FILE__, __LINE__, #x);     \
      ++failures;                                             \
    }                                                         \
  } while (0)

template <typename T>
static uint64_t at(T* p) {
  return reinterpret_cast<uint64_t>(p);
}
template <typename T>
static T* address(uint64_t v) {
  return reinterpret_cast<T*>(v);
}

// the launches of a call, checked to cover its events in order
template <typename Args>
static std::vector<Args> parts_of(const Args& a) {
  std::vector<Args> parts;
  uint64_t done = 0;
  over_grids(a, [&](const Args& c, unsigned blocks) {
    CHECK(c.n > 0 && c.n <= kGridEvents);
    CHECK(c.first == a.first + done);
    CHECK(blocks % kXcds == 0);
    CHECK((uint64_t)blocks * kBlock >= c.n);
    CHECK((uint64_t)blocks * kBlock < c.n + (kXcds + 1) * (uint64_t)kBlock);
    CHECK((uint64_t)blocks * kBlock < 1ULL << 32);  // work-items of a dispatch
    parts.push_back(c);
    done += c.n;
  });
  CHECK(done == a.n);
  CHECK(parts.size() == (a.n + kGridEvents - 1) / kGridEvents);
  return parts;
}

int main() {
  const uint64_t sizes[] = {0,           1,           256,          257, kGridEvents - 1, kGridEvents,
                            kGridEvents + 1, 2 * kGridEvents, 5 * kGridEvents + 12345};
  for (uint64_t n : sizes) {
    for (int f32 = 0; f32 < 2; ++f32) {
      for (int given = 0; given < 16; ++given) {  // which of the pointers are given
        GenArgs a{};
        a.first = 77;
        a.n = n;
        a.out_f32 = f32;
        a.ld = n + 64;
        a.mld = n + 3;
        a.cols = given & 1 ? address<void>(1ULL << 44) : nullptr;
        a.wt = given & 2 ? address<double>(2ULL << 44) : nullptr;
        a.evw = given & 4 ? address<double>(3ULL << 44) : nullptr;
        a.mothers = given & 8 ? address<const double>(4ULL << 44) : nullptr;
        uint64_t off = 0;
        for (const GenArgs& c : parts_of(a)) {
          CHECK(at(c.cols) == (a.cols ? at(a.cols) + off * (f32 ? 4 : 8) : 0));
          CHECK(at(c.wt) == (a.wt ? at(a.wt) + 8 * off : 0));
          CHECK(at(c.evw) == (a.evw ? at(a.evw) + 8 * off : 0));
          CHECK(at(c.mothers) == (a.mothers ? at(a.mothers) + 8 * off : 0));
          CHECK(c.ld == a.ld && c.mld == a.mld && c.out_f32 == f32);
          off += c.n;
        }
      }
    }
    for (int mothers = 0; mothers < 2; ++mothers) {
      EvalArgs a{};
      a.first = 1ULL << 50;
      a.n = n;
      a.seed = 5;
      a.ld = n + 1;
      a.out = address<double>(5ULL << 44);
      a.mothers = mothers ? address<const double>(6ULL << 44) : nullptr;
      uint64_t off = 0;
      for (const EvalArgs& c : parts_of(a)) {
        CHECK(at(c.out) == at(a.out) + 8 * off);
        CHECK(at(c.mothers) == (a.mothers ? at(a.mothers) + 8 * off : 0));
        CHECK(c.ld == a.ld && c.seed == a.seed);
        off += c.n;
      }
    }
  }
  // the range's runs: one per wave, every group covered, few enough for a dispatch
  for (uint64_t ngroups : {1ULL, 3ULL, 4ULL, 5ULL, 1ULL << 25, (1ULL << 25) + 1, 1ULL << 42}) {
    for (uint32_t run : {1u, 2u, 4u}) {
      uint32_t r = run;
      const uint64_t waves = (uint64_t)blocks_for_runs(ngroups, r) * (kBlock / kWave);
      CHECK(r >= run);
      CHECK(waves * r >= ngroups && (waves - kBlock / kWave) * r < ngroups);
      CHECK(waves * kWave < 1ULL << 32);
    }
  }
  std::printf(failures ? "%d checks failed\n" : "ok\n", failures);
  return failures != 0;
}
