// Replays the quad rasteriser's list counter (csrc/raster_lists.h) on the CPU:
// workgroups add lots in a random order, as many as 2^32 quads in a shell.
//   raster_lists_replay SEED QUADS GROUPS RECORDS WINDOWS MAX_AREA
//   raster_lists_replay cut SEED COUNT     rectangles cut into tests
#include "raster_lists.h"

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>

using namespace meso;

// every pixel of a rectangle is in exactly one test, and no quad has too many
static int cut(uint64_t rng, long count) {
  auto next = [&rng](uint32_t n) {
    rng = rng * 6364136223846793005ull + 1442695040888963407ull;
    return (uint32_t)(rng >> 33) % n;
  };
  std::vector<unsigned char> seen;
  for (; count; count--) {
    const uint32_t bits_w = next(15), bits_h = next(15);
    uint32_t w = 1u + next(1u << bits_w), h = 1u + next(1u << bits_h);
    if (next(16) == 0) w = 16384u, h = 16384u - next(3);
    const uint32_t spread = next(6), ws = tests_per_row(w, h, spread);
    if (ws < 1u || ws > w || (uint64_t)ws * h > kMaxQuadTests) return 1;
    if (spread == 0 && (uint64_t)w * h <= kMaxQuadTests && ws != w) return 1;
    seen.assign(w, 0);
    for (uint32_t k = 0; k < ws; k++)
      for (uint32_t x = k; x < w; x += ws) seen[x]++;
    for (unsigned char c : seen)
      if (c != 1) return 1;
  }
  if (test_spread(1) || test_spread(1u << 26) || test_spread((1u << 26) + 1u) != 1 ||
      test_spread(1u << 28) != 2)
    return 1;
  return 0;
}

int main(int argc, char **argv) {
  if (argc == 4 && argv[1][0] == 'c') return cut((uint64_t)std::atoll(argv[2]), std::atol(argv[3]));
  if (argc != 7) return 2;
  uint64_t rng = (uint64_t)std::atoll(argv[1]) * 2862933555777941757ull + 3037000493ull;
  uint64_t quads = (uint64_t)std::atoll(argv[2]);
  const uint32_t groups = (uint32_t)std::atoi(argv[3]);
  const ListLimits l{(uint32_t)std::atoll(argv[4]), (uint64_t)std::atoll(argv[5]) * kWindow};
  const uint64_t max_area = (uint64_t)std::atoll(argv[6]);
  auto next = [&rng] {
    rng = rng * 6364136223846793005ull + 1442695040888963407ull;
    return rng >> 33;
  };
  std::vector<char> full(groups, 0);
  uint64_t word = 0, lowest_full = ~0ull;       // counters kRasterTests, kRasterFull
  uint64_t records = 0, tests = 0, listed = 0, direct = 0;  // exact
  while (quads) {
    const uint32_t g = (uint32_t)(next() % groups);
    const uint32_t n = (uint32_t)std::min<uint64_t>(quads, 1u + next() % kMaxLot);
    quads -= n;
    const uint64_t all = n * (1u + next() % max_area);
    const uint64_t add = lot_word(l, n, all, full[g] != 0);
    if (!add) {
      direct += n;
      continue;
    }
    const uint64_t at = word;
    word += add;
    records += n;
    tests += all;
    if (word >> 40 != records || (word & kTestsMask) != tests) {
      std::printf("a field wrapped: %llu records, %llu tests\n", (unsigned long long)records,
                  (unsigned long long)tests);
      return 1;
    }
    if (lot_fits(l, at, n, all)) {
      listed += n;
      // places follow one another and lie inside the lists
      if (lowest_full != ~0ull || at >> 40 != records - n || records > l.records || tests > l.tests) {
        std::printf("a lot fits after one that did not, or outside the lists\n");
        return 1;
      }
    } else {
      direct += n;
      full[g] = 1;
      lowest_full = std::min(lowest_full, at);
    }
  }
  const uint64_t counted = std::min(word, lowest_full);
  std::printf("%llu listed, %llu tested directly, counter at %llu records\n",
              (unsigned long long)listed, (unsigned long long)direct, (unsigned long long)(word >> 40));
  return counted >> 40 == listed ? 0 : 1;
}
