// The bounds of the quad rasteriser's lists, and the word that numbers their
// places: one 64-bit counter per shell, tests in its low 40 bits and records
// in its high 24, which workgroups add whole lots of quads to.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace meso {

constexpr uint32_t kWindow = 256u;  // tests per window
constexpr uint32_t kMaxWindows = 1u << 23;
constexpr uint32_t kMaxRecords = 1u << 22;
constexpr uint64_t kMaxTests = (uint64_t)kMaxWindows * kWindow;
constexpr uint64_t kTestsMask = (1ull << 40) - 1ull;
constexpr uint32_t kMaxLot = 1024u;         // quads of a lot
constexpr uint32_t kMaxQuadTests = 1u << 18;
constexpr uint32_t kMaxLotGroups = 2048u;   // workgroups that add lots

// What the lists hold: the constants, or less where a host lowers them.
struct ListLimits {
  uint32_t records;
  uint64_t tests;
};

// What a workgroup adds to the counter for a lot of n quads and `tests` tests;
// 0: nothing, it tests the lot itself.  full: a lot of this workgroup did not
// fit before.
// Neither field ever wraps, whatever the number of quads.  The lots that fit
// sum to the limits at most.  One that does not fit ends its workgroup's adds,
// so there is at most one per workgroup, of kMaxLot quads and an eighth of the
// tests' limit at most.
__host__ __device__ inline uint64_t lot_word(const ListLimits &l, uint32_t n, uint64_t tests,
                                             bool full) {
  return full || tests > l.tests / 8u ? 0ull : tests | ((uint64_t)n << 40);
}
static_assert(kMaxRecords + (uint64_t)kMaxLotGroups * kMaxLot < (1ull << 24), "records' field");
static_assert(kMaxTests + kMaxLotGroups * (kMaxTests / 8u) < (1ull << 40), "tests' field");

// How a quad's rectangle of w x h pixels is cut into tests: ws a row, test k of
// a row being the pixels k, k + ws, k + 2 ws, ... of it.
//  - A quad has at most kMaxQuadTests, so that every lot can be added.  (A pixel
//    a test, a few dozen quads that each covered a frame of 16384x16384 were
//    refused and tested by their one workgroup: 0.9 s, now 12 ms, 10 before there
//    were lists.)
//  - In frames above 2^26 pixels a test takes 2^spread pixels, so that the lists
//    hold as many layers of quads as there.  Fewer pixels a test are faster where
//    both fit: 16384x16384 with 4 of them 9.7 ms, with 32 of them 13.2.
__host__ __device__ inline uint32_t tests_per_row(uint32_t w, uint32_t h, uint32_t spread) {
  uint32_t ws = (w + (1u << spread) - 1u) >> spread;
  while (ws * h > kMaxQuadTests) ws = (ws + 1u) >> 1;  // ws * h < 2^28
  return ws;
}
static_assert((uint64_t)kMaxLot * kMaxQuadTests <= kMaxTests / 8u, "every lot can be added");
__host__ __device__ inline uint32_t test_spread(uint64_t pixels) {
  uint32_t s = 0;
  while ((pixels >> s) > (1u << 26)) s++;
  return s;
}

// Whether a lot added at counter value `at` lies within the lists.  Both fields
// only grow, so every lot added after one that does not fit does not fit either
// and the lots that fit fill the lists up to the lowest `at` that does not.
__host__ __device__ inline bool lot_fits(const ListLimits &l, uint64_t at, uint32_t n,
                                         uint64_t tests) {
  return (at >> 40) + n <= l.records && (at & kTestsMask) + tests <= l.tests;
}

}  // namespace meso
