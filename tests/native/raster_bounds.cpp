// The quad rasteriser's single-precision bounds (csrc/raster.hip: tight_rect,
// chunk_view, near_bound) against its own pixel test, on the CPU: whatever
// pixel's ray hits a quad lies in the quad's and in its chunk's bounds, at a t
// above their near bounds.  raster_bounds_host.h is cut from raster.hip by
// tests/test_native_raster_bounds.py.
//   raster_bounds SEED CAMERAS
#define __umul24(a, b) (((a) & 0xFFFFFFu) * ((b) & 0xFFFFFFu))
#define __syncthreads() ((void)0)
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <hip/hip_runtime.h>
static const struct { uint32_t x, y, z; } threadIdx = {0, 0, 0}, blockIdx = {0, 0, 0},
                                          gridDim = {1, 1, 1};
static uint64_t g_rng = 1;
static uint32_t next() {
  g_rng = g_rng * 6364136223846793005ull + 1442695040888963407ull;
  return (uint32_t)(g_rng >> 33) * 2654435761u ^ (uint32_t)(g_rng >> 40);
}
static float u01() { return (float)(next() >> 8) * (1.0f / 16777216.0f); }
// the reciprocal instruction: within one unit in the last place of the result
static float __builtin_amdgcn_rcpf(float x) {
  const float r = 1.0f / x;
  const uint32_t k = next() % 3u;
  return k == 0 ? r : std::nextafterf(r, k == 1 ? -FLT_MAX : FLT_MAX);
}
#include "traverse_host.h"
namespace meso {
#include "raster_bounds_host.h"
}
using namespace meso;

static void normalize(float v[3]) {
  const float l = std::sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
  for (int i = 0; i < 3; i++) v[i] = v[i] / l;
}
static void cross(const float a[3], const float b[3], float o[3]) {
  o[0] = a[1] * b[2] - a[2] * b[1];
  o[1] = a[2] * b[0] - a[0] * b[2];
  o[2] = a[0] * b[1] - a[1] * b[0];
}

int main(int argc, char **argv) {
  if (argc != 3) return 2;
  g_rng = (uint64_t)std::atoll(argv[1]) * 2862933555777941757ull + 3037000493ull;
  long hits = 0, tight = 0, loose = 0, near_eye = 0, edge = 0;
  for (long cams = std::atol(argv[2]); cams; cams--) {
    const int32_t n = 32 << (next() % 9u), nc = n / 32;  // 32 .. 8192
    DevCamera c{};
    const int32_t sizes[] = {1, 2, 7, 64, 333, 1080, 1920, 4096, 16384};
    c.width = sizes[next() % 9u];
    c.height = sizes[next() % 9u];
    const float fov = std::pow(10.0f, u01() * 2.9f - 0.65f);  // 0.2 .. 178 degrees
    // eyes in the scene, near a face, and up to 2^20 voxels away
    float target[3], dir[3], up[3];
    const float dist = next() % 2u ? u01() * 40.0f : std::exp2(u01() * 20.0f);
    for (int a = 0; a < 3; a++) {
      target[a] = u01() * (float)n;
      dir[a] = u01() * 2.0f - 1.0f;
      up[a] = u01() * 2.0f - 1.0f;
    }
    if (next() % 4u == 0) dir[next() % 3u] = 0.0f;
    normalize(dir);
    for (int a = 0; a < 3; a++) {
      c.eye[a] = target[a] - dir[a] * dist;
      if (next() % 8u == 0) c.eye[a] = std::floor(c.eye[a]);
      c.fwd[a] = dir[a] + (u01() - 0.5f) * 0.2f * fov / 60.0f;
    }
    normalize(c.fwd);
    cross(c.fwd, up, c.right);
    normalize(c.right);
    cross(c.right, c.fwd, c.up);
    const float th = (float)std::tan((double)fov * 3.14159265358979323846 / 360.0);
    c.sx = th * ((float)c.width / (float)c.height);
    c.sy = th;
    c.inv_w2 = 2.0f / (float)c.width;
    c.inv_h2 = 2.0f / (float)c.height;
    RasterView v;
    v.fx = (float)(0.5 * c.width / (double)c.sx);
    v.fy = (float)(0.5 * c.height / (double)c.sy);
    v.cx = (float)(0.5 * c.width - 0.5);
    v.cy = (float)(0.5 * c.height - 0.5);
    v.eye_sum = std::fabs(c.eye[0]) + std::fabs(c.eye[1]) + std::fabs(c.eye[2]);
    v.f_max = v.fx > v.fy ? v.fx : v.fy;
    v.s_one = 1.5f * (1.0f + (c.sx > c.sy ? c.sx : c.sy));
    v.ray_err = 8e-7f * v.f_max * (1.0f + c.sx * c.sx + c.sy * c.sy);
    for (int k = 0; k < 400; k++) {
      // a pixel, often on the frame's side, and a quad that its ray may just hit
      int32_t px = (int32_t)(next() % (uint32_t)c.width), py = (int32_t)(next() % (uint32_t)c.height);
      if (next() % 4u == 0) px = next() & 1u ? 0 : c.width - 1;
      if (next() % 4u == 0) py = next() & 1u ? 0 : c.height - 1;
      float o[3], d[3];
      primary_ray(c, px, py, o, d);
      const int axis = (int)(next() % 3u);
      if (!(std::fabs(d[axis]) > 1e-6f)) continue;
      const int32_t plane = (int32_t)(next() % (uint32_t)n);
      const bool pos = d[axis] < 0.0f;
      const float P = (float)(plane + (pos ? 1 : 0));
      const float t0 = (P - o[axis]) / d[axis];
      if (!(t0 > 0.0f)) continue;
      int32_t cell[3], lo[3];
      bool in = true;
      for (int a = 0; a < 3; a++) {
        cell[a] = a == axis ? plane : (int32_t)std::floor(o[a] + d[a] * t0);
        if (a != axis) cell[a] += (int32_t)(next() % 3u) - 1;  // on, beside and just past the hit
        in = in && cell[a] >= 0 && cell[a] < n;
        lo[a] = cell[a] & ~31;
      }
      if (!in) continue;
      QuadGeom g;
      g.a = axis;
      g.u = axis == 0 ? 1 : 0;
      g.v = axis == 2 ? 1 : 2;
      g.face = axis == 2 ? (pos ? 0 : 1) : (axis == 1 ? (pos ? 2 : 3) : (pos ? 4 : 5));
      g.pos = pos;
      g.slice = plane;
      g.P = P;
      g.U0 = cell[g.u];
      g.V0 = cell[g.v];
      g.W = 1 + (int32_t)(next() % (uint32_t)(32 - (g.U0 & 31)));
      g.H = 1 + (int32_t)(next() % (uint32_t)(32 - (g.V0 & 31)));
      if (next() & 1u) g.W = 1;
      if (next() & 1u) g.H = 1;
      const float t = quad_hit(g, pick3(o, g.a), pick3(o, g.u), pick3(o, g.v), pick3(d, g.a),
                               pick3(d, g.u), pick3(d, g.v));
      if (t < 0.0f) continue;
      hits++;
      int32_t r[4] = {0, 0, 0, 0}, cr[4] = {0, 0, 0, 0};
      bool large;
      const int kind = tight_rect(c, v, g, r, large);
      const int ck = chunk_view(c, v, lo, cr);
      const float qd[3] = {pick3(o, g.a) - g.P,
                           interval_gap(pick3(o, g.u), (float)g.U0, (float)(g.U0 + g.W)),
                           interval_gap(pick3(o, g.v), (float)g.V0, (float)(g.V0 + g.H))};
      float cd[3];
      for (int a = 0; a < 3; a++) cd[a] = interval_gap(o[a], (float)lo[a], (float)(lo[a] + 32));
      const bool in_q = kind < 0 || (kind == 1 && px >= r[0] && px < r[1] && py >= r[2] && py < r[3]);
      const bool in_c = ck == 1 || (ck == 2 && px >= cr[0] && px < cr[1] && py >= cr[2] && py < cr[3]);
      tight += kind == 1;
      loose += kind < 0;
      near_eye += ck == 1;
      edge += kind == 1 && (px == r[0] || px == r[1] - 1 || py == r[2] || py == r[3] - 1);
      if (!in_q || !in_c || !(near_bound(qd) < t) || !(near_bound(cd) < t)) {
        std::printf("pixel %d %d of %dx%d, fov %g, eye %a %a %a: kind %d rect %d %d %d %d, chunk %d "
                    "%d %d %d %d, t %a near %a %a, n %d\n",
                    px, py, c.width, c.height, fov, c.eye[0], c.eye[1], c.eye[2], kind, r[0], r[1],
                    r[2], r[3], ck, cr[0], cr[1], cr[2], cr[3], t, near_bound(qd), near_bound(cd), n);
        return 1;
      }
    }
  }
  std::printf("%ld hits: %ld in tight rectangles (%ld on their sides), %ld left to double precision, "
              "%ld with a chunk near the eye\n", hits, tight, edge, loose, near_eye);
  return hits > 10000 && tight > 10000 && edge > 1000 ? 0 : 1;
}
