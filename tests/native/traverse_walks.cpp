// The raymarcher's walks (csrc/traverse.h) built for the CPU and compared with
// the oracle, the scene's arrays held exactly (under AddressSanitizer a read
// outside one ends the run).  The header's few inline instructions are
// replaced by the same operations in C++ (tests/test_native_walks.py).
//
//   traverse_walks dense SEED PIXELS    small dense frames, four parts a ray
//   traverse_walks bricks SEED RAYS     secondary rays of brick scenes, from
//                                       origins in and far outside the scene
#define __umul24(a, b) (((a) & 0xFFFFFFu) * ((b) & 0xFFFFFFu))
#define __syncthreads() ((void)0)
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <algorithm>
#include <vector>
#include <hip/hip_runtime.h>
static const struct { uint32_t x, y, z; } threadIdx = {0, 0, 0}, blockIdx = {0, 0, 0},
                                          gridDim = {1, 1, 1};
#include "traverse_host.h"

#include "meso_oracle.h"

namespace {

struct Rng {
  uint64_t s;
  uint32_t next() {
    s = s * 6364136223846793005ull + 1442695040888963407ull;
    return (uint32_t)(s >> 33) * 2654435761u ^ (uint32_t)(s >> 40);
  }
  float u() { return (float)(next() >> 8) * (1.0f / 16777216.0f); }
};

int fail(const char *what, const float p[3], const float d[3], const int32_t start[3]) {
  std::printf("%s: o (%a %a %a) d (%a %a %a) start %d %d %d\n", what, p[0], p[1], p[2], d[0], d[1],
              d[2], start[0], start[1], start[2]);
  return 1;
}

// One dense ray by its parts; the first of them that hits.  Returns 1 on a
// hit, 0 on none, -1 when a part would start outside the grid.
int walk_parts(const meso::DevScene &s, const meso::Ray &r, const meso::WalkState &w0,
               meso::WalkState &hit) {
  int found = 0;
  for (uint32_t part = 0; part < (uint32_t)meso::kDenseParts; part++) {
    meso::WalkState w = w0;
    meso::DenseRay e;
    if (w.t < __builtin_inff() && e.setup(s, r)) {
      float tmax = __builtin_inff();
      meso::WalkState v = w;
      if (meso::dense_part(s, r, e, v, tmax, part))
        for (int a = 0; a < 3; a++)
          if (v.cell[a] < 0 || v.cell[a] >= s.n) return -1;
    }
    uint16_t m;
    if (meso::walk_part(s, r, w, __builtin_inff(), part, m) && !found) {
      found = 1;
      hit = w;
    }
  }
  return found;
}

int dense(uint64_t seed, int64_t pixels) {
  Rng rng{seed * 77u + 5u};
  long shadows = 0, outside = 0, hits = 0;
  while (pixels > 0) {
    const int32_t edges[] = {1, 5, 16, 33, 64};
    const int32_t n = edges[rng.next() % 5u];
    std::vector<uint8_t> grid((size_t)n * n * n);
    const float fill = rng.u() < 0.5f ? 0.3f : 0.01f;
    for (auto &v : grid) v = rng.u() < fill ? 3 : 0;
    meso::DevScene s{};
    s.n = n;
    s.dense = grid.data();
    mo_scene os{};
    os.kind = MO_SCENE_DENSE_U8;
    os.n = n;
    os.dense = grid.data();
    for (int a = 0; a < 3; a++) {
      s.lo[a] = 0, s.hi[a] = n, s.flo[a] = 0.0f, s.fhi[a] = (float)n;
      os.box_lo[a] = 0, os.box_hi[a] = n;
    }
    // an eye up to the walk's limit of 2^16 and beyond, most of them far off
    float dir[3], len = 0.0f;
    for (float &c : dir) c = rng.u() * 2.0f - 1.0f, len += c * c;
    len = std::sqrt(len);
    const float dists[] = {1.2f * n, 30.0f * n, 400.0f * n, 30000.0f, 60000.0f, 90000.0f};
    const float dist = dists[rng.next() % 6u], m = 0.5f * (float)n;
    float eye[3], target[3] = {m, m, m}, up[3] = {0.1f, 1.0f, 0.2f}, light[3];
    for (int a = 0; a < 3; a++) eye[a] = m + dir[a] / len * dist;
    for (int a = 0; a < 3; a++) light[a] = rng.next() % 4u ? rng.u() * 2.0f - 1.0f : 0.0f;
    if (light[0] == 0.0f && light[1] == 0.0f && light[2] == 0.0f) light[1] = 1.0f;
    len = std::sqrt(light[0] * light[0] + light[1] * light[1] + light[2] * light[2]);
    for (float &c : light) c = c / len;
    mo_camera cam;
    mo_camera_derive(eye, target, up, 60.0f * (float)n / (dist > n ? dist : (float)n), 96, 96, &cam);
    pixels -= 96 * 96;
    for (int py = 0; py < 96; py++)
      for (int px = 0; px < 96; px++) {
        float o[3], d[3];
        mo_primary_ray(&cam, px, py, o, d);
        meso::Ray r;
        meso::WalkState w, h{};
        mo_hit oh;
        mo_counters cnt{};
        const int want = mo_trace(&os, o, d, &oh, &cnt);
        int got = 0;
        if (meso::trace_begin(s, o, d, r, w)) got = walk_parts(s, r, w, h);
        if (got < 0) return fail("a primary ray's part starts outside the grid", o, d, w.cell);
        if (got != want) return fail("primary hit differs", o, d, w.cell);
        if (!got) continue;
        hits++;
        if (std::memcmp(h.cell, oh.cell, 12) || h.face != oh.face || std::memcmp(&h.t, &oh.t, 4))
          return fail("primary cell, face or t differs", o, d, h.cell);
        if (h.face >= 6) continue;
        meso::DevShading sh{};
        std::memcpy(sh.light, light, 12);
        meso::Secondary sc;
        meso::secondary_setup(sh, o, d, h.face, h.t, h.cell, sc);
        if (!(sc.lambert > 0.0f) || !meso::start_inside(s, sc.start)) continue;
        shadows++;
        for (int a = 0; a < 3; a++)
          if (sc.p[a] < 0.0f || sc.p[a] > (float)n) {
            outside++;
            break;
          }
        meso::occluded_begin(sc.p, light, sc.start, r, w);
        got = walk_parts(s, r, w, h);
        if (got < 0) return fail("a shadow ray's part starts outside the grid", sc.p, light, sc.start);
        if (got != mo_occluded(&os, sc.p, light, sc.start, __builtin_inff(), &cnt))
          return fail("shadow differs", sc.p, light, sc.start);
      }
  }
  std::printf("dense: %ld hits, %ld shadow rays, %ld of them from outside the grid\n", hits, shadows,
              outside);
  return shadows > 1000 && outside > 10 ? 0 : 1;
}

// A brick map (n a multiple of 8) or a two-level scene (of 128) of random
// bricks, with the derived levels of both sides.
struct Bricks {
  std::vector<uint32_t> slots, top, occ32, occ128;
  std::vector<uint64_t> masks, blocks, b32, groups;
  std::vector<uint16_t> voxels;
  meso::DevScene s{};
  mo_scene os{};
  Bricks(Rng &rng, int32_t n, bool two) {
    const int32_t nb = n / 8, nt = n / 128, n32 = (n + 31) / 32, n128 = (n + 127) / 128;
    const float fill = rng.u() * rng.u();
    size_t cells = (size_t)nb * nb * nb, nodes = 0;
    if (two) {
      top.resize((size_t)nt * nt * nt);
      for (auto &t : top) t = rng.next() % 3u ? (uint32_t)nodes++ : meso::kEmpty;
      cells = nodes * 4096;
    }
    slots.resize(cells);
    blocks.resize(cells);
    for (size_t i = 0; i < cells; i++) {
      slots[i] = meso::kEmpty;
      if (rng.u() >= fill) continue;
      slots[i] = (uint32_t)(masks.size() / 8);
      const float solid = rng.u() * rng.u();
      for (int z = 0; z < 8; z++) {
        uint64_t m = 0;
        for (int k = 0; k < 64; k++) {
          m |= (uint64_t)(rng.u() < solid) << k;
          voxels.push_back((m >> k) & 1 ? 5 : 0);
        }
        masks.push_back(m);
      }
      blocks[i] = meso::brick_blocks2(&masks[masks.size() - 8]);
    }
    os.kind = two ? MO_SCENE_TWO_LEVEL_U16 : MO_SCENE_BRICKMAP_U16;
    os.n = s.n = n;
    os.slots = s.slots = slots.data();
    os.masks = s.masks = masks.data();
    os.voxels = s.voxels = voxels.data();
    os.top = s.top = top.data();
    s.blocks = blocks.data();
    occ32.resize(((size_t)n32 * n32 * n32 + 31) / 32);
    occ128.resize(((size_t)n128 * n128 * n128 + 31) / 32);
    groups.resize(nodes);
    mo_build_coarse(&os, (int64_t)nodes, occ32.data(), occ128.data(), groups.data());
    os.occ32 = s.occ32 = occ32.data();
    os.occ128 = s.occ128 = occ128.data();
    os.groups = s.groups = groups.data();
    b32.resize((size_t)n32 * n32 * n32);
    for (int32_t z = 0; z < nb; z++)
      for (int32_t y = 0; y < nb; y++)
        for (int32_t x = 0; x < nb; x++) {
          size_t cell = (size_t)x + (size_t)nb * (y + (size_t)nb * z);
          if (two) {
            const uint32_t t = top[(x >> 4) + nt * ((y >> 4) + nt * (z >> 4))];
            if (t == meso::kEmpty) continue;
            cell = (size_t)t * 4096 + (x & 15) + 16 * (y & 15) + 256 * (z & 15);
          }
          if (slots[cell] != meso::kEmpty)
            b32[(x >> 2) + n32 * ((y >> 2) + n32 * (z >> 2))] |=
                1ull << ((x & 3) + 4 * (y & 3) + 16 * (z & 3));
        }
    s.bricks32 = b32.data();
    mo_scene_box(&os, os.box_lo, os.box_hi);
    for (int a = 0; a < 3; a++) {
      s.lo[a] = os.box_lo[a], s.hi[a] = os.box_hi[a];
      s.flo[a] = (float)s.lo[a], s.fhi[a] = (float)s.hi[a];
    }
  }
};

int bricks(uint64_t seed, int64_t rays) {
  Rng rng{seed * 99u + 1u};
  long compared = 0, dark = 0, far_off = 0;
  while (rays > 0) {
    const int32_t edges[] = {8, 24, 40, 136, 128, 256};
    const uint32_t k = rng.next() % 6u;
    const int32_t n = edges[k];
    Bricks b(rng, n, k >= 4u);
    if (b.s.lo[0] >= b.s.hi[0]) continue;
    for (int i = 0; i < 20000; i++, rays--) {
      // a start cell in the box; the origin in it, or off by up to 2^30 on an
      // axis, as hit points of eyes far away are; directions with zeros
      int32_t start[3];
      float p[3], d[3], len = 0.0f;
      bool comparable = true, off_still = false;
      for (int a = 0; a < 3; a++) {
        start[a] = b.s.lo[a] + (int32_t)(rng.next() % (uint32_t)(b.s.hi[a] - b.s.lo[a]));
        p[a] = (float)start[a] + rng.u();
        d[a] = rng.next() % 3u ? rng.u() * 2.0f - 1.0f : (rng.next() & 1u ? 0.0f : -0.0f);
        len += d[a] * d[a];
        const uint32_t scale = rng.next() % 64u;
        if (scale > 30u) continue;
        p[a] += (rng.u() * 2.0f - 1.0f) * (float)(1u << scale);
        // the oracle's float-to-integer conversions have to be in range
        if (d[a] != 0.0f && scale > 12u) comparable = false;
        off_still |= d[a] == 0.0f && scale > 18u;
      }
      if (len < 1e-4f) continue;
      len = std::sqrt(len);
      for (float &c : d) c = c / len;
      const float tmax = rng.next() & 1u ? __builtin_inff() : rng.u() * 40.0f;
      meso::StepCounts c;
      const int got = k >= 4u ? meso::occluded<3, false>(b.s, p, d, start, tmax, c)
                              : meso::occluded<2, false>(b.s, p, d, start, tmax, c);
      if (!comparable) continue;
      mo_counters cnt{};
      compared++;
      far_off += off_still;
      dark += got;
      if (got != mo_occluded(&b.os, p, d, start, tmax, &cnt))
        return fail("occlusion differs", p, d, start);
    }
  }
  std::printf("bricks: %ld rays compared, %ld dark, %ld from far off an axis they keep to\n", compared,
              dark, far_off);
  return dark > 1000 && far_off > 1000 ? 0 : 1;
}

}  // namespace

int main(int argc, char **argv) {
  if (argc == 4 && !std::strcmp(argv[1], "dense"))
    return dense((uint64_t)std::atoll(argv[2]), std::atoll(argv[3]));
  if (argc == 4 && !std::strcmp(argv[1], "bricks"))
    return bricks((uint64_t)std::atoll(argv[2]), std::atoll(argv[3]));
  return 2;
}
