// Quad visibility: the raster consumer of the meshes.  For every pixel of a
// camera, the nearest front-facing quad of a chunk pool's resident slots
// along the pixel's primary ray, written in the raymarcher's output format.
// It takes the place of the reference's per-cell imposter draw
// (Samples/SimpleVoxel.cpp:352-398, a 3-face fan per solid cell), drawing the
// packed quads of the mesher instead.
//
// What bounded it was work on hidden quads (a camera in the 2048^3 caves has
// 23 million resident quads and some 150 layers of them behind a pixel), lanes
// waiting for the one with the largest quad, and the pixels of loose
// rectangles.  So, on the device and without a host round trip:
//   raster_begin_kernel: clears the keys and writes every pixel's ray.
//   For each shell of chunks around the eye, nearest first (one shell for few
//   chunks or pixels):
//     raster_list_kernel: a lane per slot; slots of this shell whose box
//       projects into the frame and is not hidden by what the nearer shells
//       drew are listed, in items of a few dozen quads.
//     raster_quads_kernel: a wave per item, a lane per quad.  The lane culls
//       back faces, bounds the quad's pixels and drops a quad that is hidden.
//       The others become records that tile one range of pixel tests.
//     raster_pixels_kernel: a wave per kWindow tests of that range, a lane per
//       test, whatever the sizes of the quads they belong to.
//     raster_depth_kernel: the farthest t of each 8x8, 32x32 and 128x128
//       block of pixels so far, which the next shell is tested against.
//   raster_resolve_kernel: a lane per pixel turns the winning key into the
//     voxel index, face, t and shade.
// A hit is a 64-bit key (float bits of t << 32) | (slot * per_slot + k),
// combined with atomicMin, so the result does not depend on the order in
// which quads are tested, and leaving out a quad whose every t is above the
// keys of all its pixels does not change it.  The per-pixel test is written
// one FP32 operation at a time, as in the oracle, and uses the raymarcher's
// primary ray and its plane distance (p - o) * (1 / d), so t equals the DDA's
// entry t bit for bit when both find the same face.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "raster_lists.h"
#include "traverse.h"

namespace meso {

constexpr uint32_t kPoolNoSlot = 0xFFFFFFFFu;
constexpr int kSmall = 64;           // counted apart in the stats
constexpr uint32_t kMaxItems = 1u << 22;

__device__ __forceinline__ void chunk_origin(uint32_t chunk, uint32_t nc, int32_t o[3]) {
  o[0] = (int32_t)(chunk % nc) * 32;
  o[1] = (int32_t)((chunk / nc) % nc) * 32;
  o[2] = (int32_t)(chunk / (nc * nc)) * 32;
}

struct QuadGeom {
  int a, u, v;
  bool pos;
  float P;
  int32_t U0, V0, W, H, slice;
  int face;
};

__device__ __forceinline__ QuadGeom quad_decode(uint32_t q, const int32_t o[3]) {
  QuadGeom g;
  const int32_t x = o[0] + (int32_t)(q & 31u), y = o[1] + (int32_t)((q >> 5) & 31u),
                z = o[2] + (int32_t)((q >> 10) & 31u);
  g.W = (int32_t)((q >> 15) & 31u) + 1;
  g.H = (int32_t)((q >> 20) & 31u) + 1;
  g.face = (int)((q >> 25) & 7u);
  g.pos = (g.face & 1) == 0;
  if (g.face < 2) {
    g.a = 2; g.u = 0; g.v = 1; g.slice = z; g.U0 = x; g.V0 = y;
  } else if (g.face < 4) {
    g.a = 1; g.u = 0; g.v = 2; g.slice = y; g.U0 = x; g.V0 = z;
  } else {
    g.a = 0; g.u = 1; g.v = 2; g.slice = x; g.U0 = y; g.V0 = z;
  }
  g.P = (float)(g.slice + (g.pos ? 1 : 0));
  return g;
}

__device__ __forceinline__ float pick3(const float v[3], int i) {
  return i == 0 ? v[0] : (i == 1 ? v[1] : v[2]);
}

// t of the hit on the quad of the ray from the eye (ea, eu, ev on the quad's
// axes) with direction (da, du, dv), or -1
__device__ __forceinline__ float quad_hit(const QuadGeom &g, float ea, float eu, float ev, float da,
                                          float du, float dv) {
  if (g.pos ? !(da < 0.0f) : !(da > 0.0f)) return -1.0f;
  const float inv = 1.0f / da;
  const float q = g.P - ea;
  const float t = q * inv;
  if (!(t > 0.0f)) return -1.0f;
  const float tu = du * t, tv = dv * t;
  const float hu = eu + tu, hv = ev + tv;
  if (!(hu >= (float)g.U0 && hu < (float)(g.U0 + g.W))) return -1.0f;
  if (!(hv >= (float)g.V0 && hv < (float)(g.V0 + g.H))) return -1.0f;
  return t;
}

// conservative pixel rectangle [r0, r1) x [r2, r3); false when empty.  The
// quad is clipped at z >= 1e-3 in front of the eye (one Sutherland-Hodgman
// pass) and the projected vertices of the clipped polygon are bounded as
// they are found, so no vertex array is kept.
__device__ __forceinline__ void bound_point(const DevCamera &c, double x, double y, double z,
                                            double b[4]) {
  const double px = (x / z / c.sx + 1.0) * 0.5 * c.width - 0.5;
  const double py = (1.0 - y / z / c.sy) * 0.5 * c.height - 0.5;
  b[0] = px < b[0] ? px : b[0];
  b[1] = px > b[1] ? px : b[1];
  b[2] = py < b[2] ? py : b[2];
  b[3] = py > b[3] ? py : b[3];
}

// By four lanes per quad (g the same in each): lane k holds corner k, which
// keeps the kernel's registers low.  Every lane of the wave takes part.
__device__ __forceinline__ bool quad_rect(const DevCamera &c, const QuadGeom &g, int32_t r[4]) {
  const int k = (int)(threadIdx.x & 3u), next = (int)((threadIdx.x & 60u) | ((k + 1) & 3));
  const double pa = g.P, pu = g.U0 + ((k == 1 || k == 2) ? g.W : 0), pv = g.V0 + (k >= 2 ? g.H : 0);
  const double p0 = g.a == 0 ? pa : (g.u == 0 ? pu : pv);
  const double p1 = g.a == 1 ? pa : (g.u == 1 ? pu : pv);
  const double p2 = g.a == 2 ? pa : (g.u == 2 ? pu : pv);
  const double e0 = p0 - c.eye[0], e1 = p1 - c.eye[1], e2 = p2 - c.eye[2];
  const double cx = e0 * c.right[0] + e1 * c.right[1] + e2 * c.right[2];
  const double cy = e0 * c.up[0] + e1 * c.up[1] + e2 * c.up[2];
  const double cz = e0 * c.fwd[0] + e1 * c.fwd[1] + e2 * c.fwd[2];
  const double lx = __shfl(cx, next, 64), ly = __shfl(cy, next, 64), lz = __shfl(cz, next, 64);
  const double zn = 1e-3;
  double b[4] = {1e30, -1e30, 1e30, -1e30};
  bool any = false;
  const bool ia = cz >= zn, ib = lz >= zn;
  if (ia) {
    bound_point(c, cx, cy, cz, b);
    any = true;
  }
  if (ia != ib) {
    const double s = (zn - cz) / (lz - cz);
    bound_point(c, cx + (lx - cx) * s, cy + (ly - cy) * s, cz + (lz - cz) * s, b);
    any = true;
  }
#pragma unroll
  for (int off = 1; off < 4; off <<= 1) {
    const double o0 = __shfl_xor(b[0], off, 64), o1 = __shfl_xor(b[1], off, 64),
                 o2 = __shfl_xor(b[2], off, 64), o3 = __shfl_xor(b[3], off, 64);
    b[0] = o0 < b[0] ? o0 : b[0];
    b[1] = o1 > b[1] ? o1 : b[1];
    b[2] = o2 < b[2] ? o2 : b[2];
    b[3] = o3 > b[3] ? o3 : b[3];
  }
  if (((__ballot(any) >> (threadIdx.x & 60u)) & 0xFull) == 0ull) return false;
  double fx0 = floor(b[0]) - 1.0, fx1 = ceil(b[1]) + 2.0, fy0 = floor(b[2]) - 1.0,
         fy1 = ceil(b[3]) + 2.0;
  fx0 = fx0 < 0.0 ? 0.0 : fx0;
  fy0 = fy0 < 0.0 ? 0.0 : fy0;
  fx1 = fx1 > c.width ? (double)c.width : fx1;
  fy1 = fy1 > c.height ? (double)c.height : fy1;
  if (!(fx0 < fx1 && fy0 < fy1)) return false;
  r[0] = (int32_t)fx0;
  r[1] = (int32_t)fx1;
  r[2] = (int32_t)fy0;
  r[3] = (int32_t)fy1;
  return true;
}

// What the bounds of a quad's pixels need of the camera, from the host.
struct RasterView {
  float fx, fy, cx, cy;  // pixel = x / z * fx + cx, cy - y / z * fy
  float eye_sum;         // |eye| summed over the axes
  float f_max, s_one;    // max(fx, fy); 1.5 (1 + max(sx, sy))
  float ray_err;         // pixels that the rounding of a ray's direction can move it
};

// Tight pixel rectangle of a quad that lies at least 1/4 in front of the eye:
// every pixel whose ray passes quad_hit is in it, and it lies inside
// quad_rect's.  The margin m covers what rounding can move a hit by: the hit
// point's rounding (1e-7 of its coordinates and 4e-7 of its distance,
// projected at the nearest corner), the direction's, and the projection's own
// (1/8 pixel, ten times what frames of 16384 pixels need).  Where that comes
// near quad_rect's own margin of one pixel, and for quads that reach behind
// the eye, quad_rect decides (returns -1 here).  1: rectangle in r, 0: empty.
// large: quad_rect's rectangle has more than kSmall pixels (for the stats).
__device__ __forceinline__ int tight_rect(const DevCamera &c, const RasterView &v,
                                          const QuadGeom &g, int32_t r[4], bool &large) {
  const float e[3] = {(g.a == 0 ? g.P : (float)g.U0) - c.eye[0],
                      (g.a == 1 ? g.P : (g.u == 1 ? (float)g.U0 : (float)g.V0)) - c.eye[1],
                      (g.a == 2 ? g.P : (float)g.V0) - c.eye[2]};
  const float x0 = e[0] * c.right[0] + e[1] * c.right[1] + e[2] * c.right[2];
  const float y0 = e[0] * c.up[0] + e[1] * c.up[1] + e[2] * c.up[2];
  const float z0 = e[0] * c.fwd[0] + e[1] * c.fwd[1] + e[2] * c.fwd[2];
  const float w = (float)g.W, h = (float)g.H;
  const float xu = w * pick3(c.right, g.u), yu = w * pick3(c.up, g.u), zu = w * pick3(c.fwd, g.u);
  const float xv = h * pick3(c.right, g.v), yv = h * pick3(c.up, g.v), zv = h * pick3(c.fwd, g.v);
  const float z_min = z0 + (zu < 0.0f ? zu : 0.0f) + (zv < 0.0f ? zv : 0.0f);
  const float z_max = z0 + (zu > 0.0f ? zu : 0.0f) + (zv > 0.0f ? zv : 0.0f);
  if (z_max < -1.0f) return 0;
  if (z_min < 0.25f) return -1;
  const float dist = fabsf(e[0]) + fabsf(e[1]) + fabsf(e[2]) + 64.0f;
  const float m = 0.125f + v.ray_err +
                  (1e-7f * (v.eye_sum + dist) + 4e-7f * dist) * v.f_max / z_min * v.s_one;
  if (!(m < 0.8f)) return -1;
  float bx0 = 1e30f, bx1 = -1e30f, by0 = 1e30f, by1 = -1e30f;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const bool ku = k == 1 || k == 2, kv = k >= 2;
    const float x = x0 + (ku ? xu : 0.0f) + (kv ? xv : 0.0f);
    const float y = y0 + (ku ? yu : 0.0f) + (kv ? yv : 0.0f);
    const float z = z0 + (ku ? zu : 0.0f) + (kv ? zv : 0.0f);
    const float iz = __builtin_amdgcn_rcpf(z);
    const float px = x * iz * v.fx + v.cx, py = v.cy - y * iz * v.fy;
    bx0 = fminf(bx0, px);
    bx1 = fmaxf(bx1, px);
    by0 = fminf(by0, py);
    by1 = fmaxf(by1, py);
  }
  const float fx0 = fmaxf(ceilf(bx0 - m), 0.0f), fy0 = fmaxf(ceilf(by0 - m), 0.0f);
  const float fx1 = fminf(floorf(bx1 + m) + 1.0f, (float)c.width),
              fy1 = fminf(floorf(by1 + m) + 1.0f, (float)c.height);
  if (!(fx0 < fx1 && fy0 < fy1)) return 0;
  r[0] = (int32_t)fx0;
  r[1] = (int32_t)fx1;
  r[2] = (int32_t)fy0;
  r[3] = (int32_t)fy1;
  large = (fminf(ceilf(bx1) + 2.0f, (float)c.width) - fmaxf(floorf(bx0) - 1.0f, 0.0f)) *
              (fminf(ceilf(by1) + 2.0f, (float)c.height) - fmaxf(floorf(by0) - 1.0f, 0.0f)) >
          (float)kSmall;
  return 1;
}

// The 32^3 chunk at o: 0 when no part of it can reach a pixel (all of it lies
// behind the eye, or beyond one side of the frame), 2 when it lies at least 1
// in front of the eye and r bounds its pixels, 1 when it reaches nearer.  The
// frame and r have 4 pixels of margin; a quad's bounds have at most 2.
__device__ __forceinline__ int chunk_view(const DevCamera &c, const RasterView &v,
                                          const int32_t o[3], int32_t r[4]) {
  const float e0 = (float)o[0] - c.eye[0], e1 = (float)o[1] - c.eye[1], e2 = (float)o[2] - c.eye[2];
  const float sx = c.sx * (1.0f + 8.0f / (float)c.width), sy = c.sy * (1.0f + 8.0f / (float)c.height);
  float z_min = 1e30f, z_max = -1e30f, bx0 = 1e30f, bx1 = -1e30f, by0 = 1e30f, by1 = -1e30f;
  bool left = true, right = true, over = true, under = true;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const float a = e0 + ((k & 1) ? 32.0f : 0.0f), b = e1 + ((k & 2) ? 32.0f : 0.0f),
                d = e2 + ((k & 4) ? 32.0f : 0.0f);
    const float x = a * c.right[0] + b * c.right[1] + d * c.right[2];
    const float y = a * c.up[0] + b * c.up[1] + d * c.up[2];
    const float z = a * c.fwd[0] + b * c.fwd[1] + d * c.fwd[2];
    z_min = fminf(z_min, z);
    z_max = fmaxf(z_max, z);
    // beyond a side's plane, by more than the rounding of x and z
    right &= x > sx * z + 0.01f * (1.0f + sx);
    left &= x < -sx * z - 0.01f * (1.0f + sx);
    over &= y > sy * z + 0.01f * (1.0f + sy);
    under &= y < -sy * z - 0.01f * (1.0f + sy);
    const float iz = __builtin_amdgcn_rcpf(z);  // used where z >= 1
    const float px = x * iz * v.fx + v.cx, py = v.cy - y * iz * v.fy;
    bx0 = fminf(bx0, px);
    bx1 = fmaxf(bx1, px);
    by0 = fminf(by0, py);
    by1 = fmaxf(by1, py);
  }
  if (z_max < -1.0f || left || right || over || under) return 0;
  if (z_min < 1.0f) return 1;
  const float x1 = (float)(c.width - 1), y1 = (float)(c.height - 1);
  r[0] = (int32_t)fminf(fmaxf(floorf(bx0) - 4.0f, 0.0f), x1);
  r[1] = (int32_t)fminf(fmaxf(ceilf(bx1) + 4.0f, 0.0f), x1) + 1;
  r[2] = (int32_t)fminf(fmaxf(floorf(by0) - 4.0f, 0.0f), y1);
  r[3] = (int32_t)fminf(fmaxf(ceilf(by1) + 4.0f, 0.0f), y1) + 1;
  return 2;
}

// One shell's pixel tests are numbered through: record i owns the tests from
// its start to the next record's.  {start, quad id, x0 | y0 << 14, width |
// tests per row << 16} (tests_per_row) and
// {U0 | V0 << 13 | face << 26, slice | (W - 1) << 13 | (H - 1) << 18}.
struct RasterScratch {
  unsigned long long *keys;  // width * height
  float *rays;               // x, y and z of every pixel's ray, width * height each
  uint32_t *far_t;           // depth levels: 8x8, then 32x32, then 128x128 blocks
  uint32_t *items;           // slot | batch << 22
  uint4 *rec_a;              // kMaxRecords
  uint2 *rec_b;
  uint32_t *windows;         // the record that owns a window's first test
  // of the current shell: [0] tests | records << 40, [1] the items, [4] the
  // lowest [0] at which something did not fit; of the frame: [2] small | large
  // << 32 quads, [3] records | overflowed quads << 32
  unsigned long long *counters;
  ListLimits limits;
};
enum : int { kRasterTests = 0, kRasterItems = 1, kRasterDrawn = 2, kRasterRecords = 3, kRasterFull = 4, kRasterCounters = 5 };

// Farthest t (as float bits; ~0 where a pixel has no hit yet) of the blocks of
// 8, 32 and 128 pixels.
struct DepthLevels {
  const uint32_t *far_t;
  uint32_t w8, w32, w128, at32, at128;
};
__host__ __device__ inline DepthLevels depth_levels(const uint32_t *far_t, int32_t width,
                                                    int32_t height) {
  DepthLevels d;
  d.far_t = far_t;
  d.w8 = (uint32_t)(width + 7) / 8u;
  d.w32 = (uint32_t)(width + 31) / 32u;
  d.w128 = (uint32_t)(width + 127) / 128u;
  d.at32 = d.w8 * ((uint32_t)(height + 7) / 8u);
  d.at128 = d.at32 + d.w32 * ((uint32_t)(height + 31) / 32u);
  return d;
}

// True when every pixel of the rectangle already has a hit nearer than `near`
// (a bound below every t of the object): the object cannot win a pixel.
// Tested on the finest level where the rectangle touches at most 2x2 blocks.
__device__ __forceinline__ bool hidden(const DepthLevels &d, const int32_t r[4], float near) {
  if (!(near > 0.0f)) return false;
  const uint32_t x0 = (uint32_t)r[0], x1 = (uint32_t)r[1] - 1u, y0 = (uint32_t)r[2],
                 y1 = (uint32_t)r[3] - 1u;
  uint32_t sh = 3u, w = d.w8, at = 0u;
  if ((x1 >> 3) - (x0 >> 3) > 1u || (y1 >> 3) - (y0 >> 3) > 1u) sh = 5u, w = d.w32, at = d.at32;
  if ((x1 >> sh) - (x0 >> sh) > 1u || (y1 >> sh) - (y0 >> sh) > 1u)
    sh = 7u, w = d.w128, at = d.at128;
  if ((x1 >> sh) - (x0 >> sh) > 1u || (y1 >> sh) - (y0 >> sh) > 1u) return false;
  const uint32_t *p0 = d.far_t + at + w * (y0 >> sh), *p1 = d.far_t + at + w * (y1 >> sh);
  const uint32_t a = p0[x0 >> sh], b = p0[x1 >> sh], e = p1[x0 >> sh], f = p1[x1 >> sh];
  const uint32_t m = max(max(a, b), max(e, f));
  return __float_as_uint(near) > m;
}

// The squared distance, finite: an eye 2^64 voxels away, whose distance is a
// float but its square is not, counts as at the largest.
__device__ __forceinline__ float square_dist(const float d[3]) {
  return fminf(d[0] * d[0] + d[1] * d[1] + d[2] * d[2], 3.402823466e38f);
}
// A bound below the t of every hit on the box [lo, lo + size] from the eye:
// its distance, less what the hit's rounding and the unit ray's can take off.
__device__ __forceinline__ float near_bound(const float d[3]) {
  return __builtin_sqrtf(square_dist(d)) * 0.9999f - 0.01f;
}
__device__ __forceinline__ float interval_gap(float e, float lo, float hi) {
  return fmaxf(fmaxf(lo - e, e - hi), 0.0f);
}

__global__ void __launch_bounds__(256) raster_begin_kernel(DevCamera cam, RasterScratch s,
                                                           uint64_t npx) {
  const uint64_t i = block_id() * 256u + threadIdx.x;
  if (i < kRasterCounters) s.counters[i] = 0ull;
  if (i >= npx) return;
  s.keys[i] = ~0ull;
  float o[3], d[3];
  primary_ray(cam, (int32_t)(i % (uint32_t)cam.width), (int32_t)(i / (uint32_t)cam.width), o, d);
#pragma unroll
  for (int a = 0; a < 3; a++) s.rays[npx * a + i] = d[a];
}

// sum of the lower lanes' v
__device__ __forceinline__ uint32_t wave_exclusive(uint32_t v) {
  uint32_t inc = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t o = __shfl_up(inc, off, 64);
    if ((int)(threadIdx.x & 63u) >= off) inc += o;
  }
  return inc - v;
}

// The items of the chunks whose distance lies in [near2, far2) (squared): a
// lane per slot.  occlude: the depth levels hold the nearer shells.
__global__ void __launch_bounds__(1024) raster_list_kernel(
    DevCamera cam, RasterView view, const uint32_t *slot_chunk, const uint32_t *slot_count,
    uint32_t capacity, uint32_t per_slot, uint32_t nc, uint32_t batch, float near2, float far2, bool occlude,
    DepthLevels depth, RasterScratch s) {
  const uint32_t sl = blockIdx.x * 1024u + threadIdx.x;
  if (sl == 0u) {
    s.counters[kRasterTests] = 0ull;
    s.counters[kRasterFull] = ~0ull;
  }
  uint32_t n = 0;
  if (sl < capacity) {
    const uint32_t chunk = slot_chunk[sl];
    const uint32_t cnt = chunk == kPoolNoSlot ? 0u : min(slot_count[sl], per_slot);
    if (cnt) {
      int32_t o[3];
      chunk_origin(chunk, nc, o);
      float d[3];
#pragma unroll
      for (int a = 0; a < 3; a++)
        d[a] = interval_gap(cam.eye[a], (float)o[a], (float)(o[a] + 32));
      const float q = square_dist(d);
      if (q >= near2 && q < far2) {
        int32_t r[4];
        const int in = chunk_view(cam, view, o, r);
        if (in == 1 || (in == 2 && !(occlude && hidden(depth, r, near_bound(d)))))
          n = (cnt + batch - 1u) / batch;
      }
    }
  }
  // one counter add per workgroup; the lanes' places by prefix sums
  __shared__ uint32_t wave_sum[16], at;
  const uint32_t wave = threadIdx.x >> 6;
  uint32_t base = wave_exclusive(n);
  if ((threadIdx.x & 63u) == 63u) wave_sum[wave] = base + n;
  __syncthreads();
  uint32_t all = 0;
#pragma unroll
  for (uint32_t w = 0; w < 16u; w++) {
    base += w < wave ? wave_sum[w] : 0u;
    all += wave_sum[w];
  }
  if (threadIdx.x == 0u && all)
    at = (uint32_t)atomicAdd(&s.counters[kRasterItems], (unsigned long long)all);
  __syncthreads();
  base += at;
  for (uint32_t k = 0; k < n; k++) s.items[base + k] = sl | (k << 22);
}

// tests pixel (px, py) against a quad; e: the eye
__device__ __forceinline__ void test_pixel(const QuadGeom &g, const float e[3], uint64_t pix,
                                           uint64_t npx, uint32_t id, const RasterScratch &s) {
  const float da = s.rays[npx * (uint32_t)g.a + pix], du = s.rays[npx * (uint32_t)g.u + pix],
              dv = s.rays[npx * (uint32_t)g.v + pix];
  const float t = quad_hit(g, pick3(e, g.a), pick3(e, g.u), pick3(e, g.v), da, du, dv);
  if (t < 0.0f) return;
  atomicMin(&s.keys[pix], ((unsigned long long)__float_as_uint(t) << 32) | id);
}

// k / w for k < 2^28 and w <= 2^14, from iw = 1 / w: the float quotient is off
// by at most a few units (2^28 / 2^24, relative 2^-22 of it), which the
// remainder's own quotient corrects
__device__ __forceinline__ uint32_t div_pixels(uint32_t k, uint32_t w, float iw) {
  uint32_t q = (uint32_t)((float)k * iw);
  int32_t rem = (int32_t)(k - q * w);
  const int32_t c = (int32_t)floorf((float)rem * iw);
  q += (uint32_t)c;
  rem -= c * (int32_t)w;
  if (rem < 0) q--;
  else if (rem >= (int32_t)w) q++;
  return q;
}

__device__ __forceinline__ uint2 pack_geom(const QuadGeom &g) {
  return make_uint2((uint32_t)g.U0 | ((uint32_t)g.V0 << 13) | ((uint32_t)g.face << 26),
                    (uint32_t)g.slice | ((uint32_t)(g.W - 1) << 13) | ((uint32_t)(g.H - 1) << 18));
}
__device__ __forceinline__ QuadGeom unpack_geom(uint32_t b0, uint32_t b1) {
  QuadGeom g;
  g.U0 = (int32_t)(b0 & 0x1FFFu);
  g.V0 = (int32_t)((b0 >> 13) & 0x1FFFu);
  g.face = (int)(b0 >> 26);
  g.slice = (int32_t)(b1 & 0x1FFFu);
  g.W = (int32_t)((b1 >> 13) & 31u) + 1;
  g.H = (int32_t)((b1 >> 18) & 31u) + 1;
  g.a = g.face < 2 ? 2 : (g.face < 4 ? 1 : 0);
  g.u = g.face < 4 ? 0 : 1;
  g.v = g.face < 2 ? 1 : 2;
  g.pos = (g.face & 1) == 0;
  g.P = (float)(g.slice + (g.pos ? 1 : 0));
  return g;
}

// Quads that stay in the frame, collected per workgroup: every add to the
// shell's one counter takes 50 to 100 ns of the word's time, whoever adds, so
// a workgroup adds once per kCollect quads or more (an add per wave and 64
// quads took 0.79 ms for the far shell of 16,384 cave chunks, this 0.15 ms).
constexpr uint32_t kQuadThreads = 512u, kCollect = 512u;
static_assert(2u * kCollect <= kMaxLot, "a lot");
struct Collected {
  uint32_t id[2 * kCollect], xy[2 * kCollect], rw[2 * kCollect], area[2 * kCollect];
  uint2 geom[2 * kCollect];
  uint64_t wave_sum[kQuadThreads / 64];
  uint32_t n;
  bool full;  // a lot did not fit: the workgroup tests the rest of its quads itself
  unsigned long long at;
};

// Lists the collected quads (all threads; C.n of them, at most 2 * kCollect).
__device__ __forceinline__ void flush_quads(Collected &C, const DevCamera &cam,
                                            const RasterScratch &s, uint32_t &n_records,
                                            uint32_t &n_over) {
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6, n = C.n;
  // two neighbouring quads per thread; exclusive sums of their tests
  const uint32_t a0 = 2u * t < n ? C.area[2u * t] : 0u,
                 a1 = 2u * t + 1u < n ? C.area[2u * t + 1u] : 0u;
  uint64_t inc = (uint64_t)a0 + a1;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint64_t o = (uint64_t)__shfl_up((unsigned long long)inc, off, 64);
    if ((int)lane >= off) inc += o;
  }
  if (lane == 63u) C.wave_sum[wave] = inc;
  __syncthreads();
  uint64_t before = inc - a0 - a1, all = 0;
#pragma unroll
  for (uint32_t w = 0; w < kQuadThreads / 64u; w++) {
    before += w < wave ? C.wave_sum[w] : 0ull;
    all += C.wave_sum[w];
  }
  if (t == 0) {
    const uint64_t add = lot_word(s.limits, n, all, C.full);
    C.at = add ? atomicAdd(&s.counters[kRasterTests], (unsigned long long)add) : ~0ull;
  }
  __syncthreads();
  const unsigned long long at = C.at;
  const uint64_t rec0 = at >> 40, test0 = at & kTestsMask;
  if (at != ~0ull && lot_fits(s.limits, at, n, all)) {  // uniform
    uint64_t start = test0 + before;
#pragma unroll
    for (uint32_t j = 0; j < 2u; j++) {
      const uint32_t q = 2u * t + j, area = j ? a1 : a0;
      const uint32_t rec = (uint32_t)rec0 + q;
      const uint32_t w0 = (uint32_t)((start + kWindow - 1u) / kWindow),
                     w1 = (uint32_t)((start + area + kWindow - 1u) / kWindow);
      if (q < n) {
        s.rec_a[rec] = make_uint4((uint32_t)start, C.id[q], C.xy[q], C.rw[q]);
        s.rec_b[rec] = C.geom[q];
        if (w1 - w0 <= 4u)
          for (uint32_t w = w0; w < w1; w++) s.windows[w] = rec;
      }
      // the windows of a large quad by the whole wave
      for (uint64_t wide = __ballot(w1 - w0 > 4u); wide; wide &= wide - 1ull) {
        const int l = __ffsll((unsigned long long)wide) - 1;
        const uint32_t b0 = (uint32_t)__builtin_amdgcn_readlane((int)w0, l),
                       b1 = (uint32_t)__builtin_amdgcn_readlane((int)w1, l),
                       br = (uint32_t)__builtin_amdgcn_readlane((int)rec, l);
        for (uint32_t w = b0 + lane; w < b1; w += 64u) s.windows[w] = br;
      }
      start += area;
    }
    if (t == 0) n_records += n;
  } else {
    // no room: the workgroup tests its quads' pixels here, a wave per quad.
    // raster_pixels_kernel stops at the first lot that did not fit.
    if (t == 0) {
      if (at != ~0ull) {
        atomicMin(&s.counters[kRasterFull], at);
        C.full = true;
      }
      n_over += n;
    }
    const uint64_t npx = (uint64_t)cam.width * (uint32_t)cam.height;
    const float eye[3] = {cam.eye[0], cam.eye[1], cam.eye[2]};
    for (uint32_t q = wave; q < n; q += kQuadThreads / 64u) {
      const QuadGeom g = unpack_geom(C.geom[q].x, C.geom[q].y);
      const uint32_t xy = C.xy[q], w = C.rw[q] & 0xFFFFu, a = C.area[q] / (C.rw[q] >> 16) * w;
      for (uint32_t p = lane; p < a; p += 64u)
        test_pixel(g, eye, (uint64_t)((xy >> 14) + p / w) * (uint32_t)cam.width + (xy & 0x3FFFu) + p % w,
                   npx, C.id[q], s);
    }
  }
  __syncthreads();
  if (t == 0) C.n = 0u;
  __syncthreads();
}

// The quads of the shell's items, an item per wave, a lane per quad.  Bound to
// 5 waves per SIMD: the compiler's 141 registers allowed 3 and it ran 10%
// longer, at 6 and 8 the spills cost more than the waves gain.
__global__ void __launch_bounds__(kQuadThreads, 5) raster_quads_kernel(
    DevCamera cam, RasterView view, const uint32_t *slot_chunk, const uint32_t *slot_count,
    const uint32_t *quads, uint32_t per_slot, uint32_t nc, uint32_t batch, uint32_t spread,
    bool occlude, DepthLevels depth, RasterScratch s) {
  __shared__ Collected C;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  constexpr uint32_t kWaves = kQuadThreads / 64u;
  const uint32_t n_items = (uint32_t)s.counters[kRasterItems];
  const float eye[3] = {cam.eye[0], cam.eye[1], cam.eye[2]};
  uint32_t n_small = 0, n_large = 0, n_records = 0, n_over = 0;
  if (threadIdx.x == 0) {
    C.n = 0u;
    C.full = false;
  }
  __syncthreads();
  // every wave of the workgroup makes the same trips
  for (uint32_t it0 = blockIdx.x * kWaves; it0 < n_items; it0 += gridDim.x * kWaves) {
    uint32_t sl = 0, k0 = 0, cnt = 0;
    int32_t origin[3] = {0, 0, 0};
    if (it0 + wave < n_items) {
      const uint32_t item = s.items[it0 + wave];
      sl = item & 0x3FFFFFu;
      k0 = (item >> 22) * batch;
      chunk_origin(slot_chunk[sl], nc, origin);
      cnt = min(min(slot_count[sl], per_slot), k0 + batch);
    }
    for (uint32_t kb = 0; kb < batch; kb += 64u) {
      const uint32_t k = k0 + kb + lane;
      const uint32_t id = sl * per_slot + k;  // below 2^32 (checked by the caller)
      int32_t r[4] = {0, 0, 0, 0};
      int live = 0;
      bool large = false;
      const QuadGeom g = quad_decode(k < cnt ? quads[id] : 0u, origin);
      const float e = pick3(eye, g.a);
      // back-facing quads cannot be hit from this eye
      if (k < cnt && (g.pos ? e > g.P : e < g.P)) live = tight_rect(cam, view, g, r, large);
      const uint2 geom = pack_geom(g);
      // the few that quad_rect decides: 16 at a time, four lanes each
      for (uint64_t todo = __ballot(live < 0); todo;) {
        uint32_t src = lane;  // this lane's quad: the (lane / 4)-th of those left
        uint64_t rest = todo;
        for (uint32_t j = 0; j < 16u && rest; j++) {
          const uint32_t l = (uint32_t)__ffsll((unsigned long long)rest) - 1u;
          src = (lane >> 2) == j ? l : src;
          rest &= rest - 1ull;
        }
        const uint64_t taken = todo & ~rest;
        const QuadGeom n = unpack_geom((uint32_t)__shfl((int)geom.x, (int)src, 64),
                                       (uint32_t)__shfl((int)geom.y, (int)src, 64));
        int32_t rr[4] = {0, 0, 0, 0};
        const int any = quad_rect(cam, n, rr) ? 1 : 0;
        // back to the quad's lane: its place among those taken, four lanes each
        const int at = (int)(4u * (uint32_t)__popcll(taken & ((1ull << lane) - 1ull))) & 63;
        const int ra = __shfl(any, at, 64);
        const int r0 = __shfl(rr[0], at, 64), r1 = __shfl(rr[1], at, 64),
                  r2 = __shfl(rr[2], at, 64), r3 = __shfl(rr[3], at, 64);
        if ((taken >> lane) & 1ull) {
          live = ra;
          r[0] = r0, r[1] = r1, r[2] = r2, r[3] = r3;
          large = (r1 - r0) * (r3 - r2) > kSmall;
        }
        todo = rest;
      }
      if (live && occlude) {
        const float d[3] = {e - g.P,
                            interval_gap(pick3(eye, g.u), (float)g.U0, (float)(g.U0 + g.W)),
                            interval_gap(pick3(eye, g.v), (float)g.V0, (float)(g.V0 + g.H))};
        if (hidden(depth, r, near_bound(d))) live = 0;
      }
      const uint64_t lives = __ballot(live != 0);
      const uint32_t rw = (uint32_t)(r[1] - r[0]);
      n_small += live && !large ? 1u : 0u;
      n_large += live && large ? 1u : 0u;
      uint32_t at = 0;
      if (lane == 0 && lives) at = atomicAdd(&C.n, (uint32_t)__popcll(lives));  // LDS
      at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
      if (live) {
        at += (uint32_t)__popcll(lives & ((1ull << lane) - 1ull));
        C.id[at] = id;
        C.xy[at] = (uint32_t)r[0] | ((uint32_t)r[2] << 14);
        const uint32_t ws = tests_per_row(rw, (uint32_t)(r[3] - r[2]), spread);
        C.rw[at] = rw | (ws << 16);
        C.area[at] = ws * (uint32_t)(r[3] - r[2]);
        C.geom[at] = geom;
      }
      __syncthreads();
      const uint32_t held = C.n;
      __syncthreads();  // read by every wave before the next trip adds to it
      // room is left for one more trip (kQuadThreads quads) below kCollect
      if (held > kCollect) flush_quads(C, cam, s, n_records, n_over);  // uniform
    }
  }
  __syncthreads();
  if (C.n) flush_quads(C, cam, s, n_records, n_over);
  unsigned long long drawn = (unsigned long long)n_small | ((unsigned long long)n_large << 32);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) drawn += __shfl_xor(drawn, off, 64);
  if (lane == 0) C.wave_sum[wave] = drawn;
  __syncthreads();
  if (threadIdx.x == 0) {
    drawn = 0;
    for (uint32_t w = 0; w < kWaves; w++) drawn += C.wave_sum[w];
    if (drawn) {
      atomicAdd(&s.counters[kRasterDrawn], drawn);
      atomicAdd(&s.counters[kRasterRecords],
                (unsigned long long)n_records | ((unsigned long long)n_over << 32));
    }
  }
}

// Persistent waves over the windows of the shell's pixel tests.
__global__ void __launch_bounds__(64) raster_pixels_kernel(DevCamera cam, RasterScratch s) {
  __shared__ uint32_t owner_at[kWindow];
  const uint32_t lane = threadIdx.x;
  // the next shell's list is empty until its list kernel runs
  if (blockIdx.x == 0 && lane == 0) s.counters[kRasterItems] = 0ull;
  const uint64_t npx = (uint64_t)cam.width * (uint32_t)cam.height;
  const float eye[3] = {cam.eye[0], cam.eye[1], cam.eye[2]};
  // both fields of [0] only grow, so the smaller word is the earlier state
  const uint64_t counted = min((uint64_t)s.counters[kRasterTests], (uint64_t)s.counters[kRasterFull]);
  const uint32_t n_rec = (uint32_t)(counted >> 40);
  const uint64_t total = counted & kTestsMask;
  for (uint32_t k = lane; k < kWindow; k += 64u) owner_at[k] = 0u;
  for (uint64_t w = blockIdx.x; w * kWindow < total; w += gridDim.x) {
    const uint32_t base = (uint32_t)(w * kWindow);
    const uint32_t len = (uint32_t)min((uint64_t)kWindow, total - w * kWindow);
    uint32_t first = s.windows[w], done = 0;
    // 64 records at a time from the one that owns the next test; their starts
    // ascend, by at least one test each
    for (;;) {
      const uint32_t rec = first + lane;
      const bool in = rec < n_rec;
      const uint4 a = in ? s.rec_a[rec] : make_uint4(0u, 0u, 0u, 0u);
      const uint2 b = in ? s.rec_b[rec] : make_uint2(0u, 0u);
      const int32_t at = in ? (int32_t)(a.x - base) : (int32_t)kWindow;  // first test, from base
      const int32_t last = __builtin_amdgcn_readlane(at, 63);
      const uint32_t stop = last < (int32_t)len ? (uint32_t)last : len;  // tests these cover
      if (at >= (int32_t)done && at < (int32_t)stop) owner_at[at] = lane + 1u;
      const float iw = a.w ? 1.0f / (float)(a.w >> 16) : 0.0f;
      uint32_t carry = 0;
      __builtin_amdgcn_wave_barrier();
      for (uint32_t g0 = done; g0 < stop; g0 += 64u) {
        const uint32_t p = g0 + lane;
        uint32_t mark = 0;
        if (p < stop) {
          mark = owner_at[p];
          owner_at[p] = 0u;
        }
        // test p belongs to the last record that starts at or before it
        const uint64_t upto = __ballot(mark != 0u) & (~0ull >> (63u - lane));
        const uint32_t from = upto ? 63u - (uint32_t)__builtin_clzll(upto) : 0u;
        const uint32_t found = (uint32_t)__shfl((int)mark, (int)from, 64);
        const uint32_t own = upto ? found - 1u : carry;
        carry = (uint32_t)__builtin_amdgcn_readlane((int)own, 63);
        const uint32_t id = (uint32_t)__shfl((int)a.y, (int)own, 64);
        const uint32_t xy = (uint32_t)__shfl((int)a.z, (int)own, 64);
        const uint32_t ow = (uint32_t)__shfl((int)a.w, (int)own, 64);
        const int32_t oat = __shfl(at, (int)own, 64);
        const float oiw = __shfl(iw, (int)own, 64);
        const QuadGeom g = unpack_geom((uint32_t)__shfl((int)b.x, (int)own, 64),
                                       (uint32_t)__shfl((int)b.y, (int)own, 64));
        if (p < stop && ow) {
          const uint32_t k = (uint32_t)((int32_t)p - oat), ws = ow >> 16;
          const uint32_t py = div_pixels(k, ws, oiw);
          const uint64_t row = (uint64_t)((xy >> 14) + py) * (uint32_t)cam.width + (xy & 0x3FFFu);
          for (uint32_t x = k - py * ws; x < (ow & 0xFFFFu); x += ws)
            test_pixel(g, eye, row + x, npx, id, s);
        }
      }
      __builtin_amdgcn_wave_barrier();
      if (stop >= len) break;  // uniform
      done = stop;
      first += 63u;
    }
  }
}

// The depth levels from the keys: a workgroup per 128x128 block, a wave per
// 32x32 block, one 8x8 block at a time, a lane per pixel (pixels outside the
// frame count as nearest).
__global__ void __launch_bounds__(1024) raster_depth_kernel(const unsigned long long *keys,
                                                            int32_t width, int32_t height,
                                                            DepthLevels d, uint32_t *far_t) {
  __shared__ uint32_t far32[16];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t bx = blockIdx.x * 4u + (wave & 3u), by = blockIdx.y * 4u + (wave >> 2);
  uint32_t v[16];
#pragma unroll
  for (uint32_t b = 0; b < 16u; b++) {
    const uint32_t x = bx * 32u + (b & 3u) * 8u + (lane & 7u),
                   y = by * 32u + (b >> 2) * 8u + (lane >> 3);
    v[b] = x < (uint32_t)width && y < (uint32_t)height
               ? (uint32_t)(keys[(uint64_t)y * (uint32_t)width + x] >> 32)
               : 0u;
  }
  uint32_t all = 0;
#pragma unroll
  for (uint32_t b = 0; b < 16u; b++) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v[b] = max(v[b], (uint32_t)__shfl_xor((int)v[b], off, 64));
    const uint32_t x8 = bx * 4u + (b & 3u), y8 = by * 4u + (b >> 2);
    if (lane == b && x8 * 8u < (uint32_t)width && y8 * 8u < (uint32_t)height)
      far_t[y8 * d.w8 + x8] = v[b];
    all = max(all, v[b]);
  }
  if (lane == 0) {
    if (bx * 32u < (uint32_t)width && by * 32u < (uint32_t)height) far_t[d.at32 + by * d.w32 + bx] = all;
    far32[wave] = all;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t m = 0;
    for (int k = 0; k < 16; k++) m = max(m, far32[k]);
    far_t[d.at128 + blockIdx.y * d.w128 + blockIdx.x] = m;
  }
}

__global__ void __launch_bounds__(256) raster_resolve_kernel(DevCamera cam, DevShading sh,
                                                             const uint32_t *slot_chunk,
                                                             const uint32_t *quads,
                                                             uint32_t per_slot, uint32_t nc,
                                                             int32_t n, RayOut out,
                                                             RasterScratch s) {
  const uint64_t i = block_id() * 256u + threadIdx.x;
  const uint64_t npx = (uint64_t)cam.width * (uint32_t)cam.height;
  if (i >= npx) return;
  const unsigned long long key = s.keys[i];
  int64_t index = -1;
  int32_t face = kFaceMiss;
  float t = __builtin_inff(), shade = 0.0f;
  if (key != ~0ull) {
    const uint32_t id = (uint32_t)key;
    int32_t origin[3];
    chunk_origin(slot_chunk[id / per_slot], nc, origin);
    const QuadGeom g = quad_decode(quads[id], origin);
    t = __uint_as_float((uint32_t)(key >> 32));
    const float du = s.rays[npx * (uint32_t)g.u + i] * t, dv = s.rays[npx * (uint32_t)g.v + i] * t;
    const float hu = pick3(cam.eye, g.u) + du, hv = pick3(cam.eye, g.v) + dv;
    int32_t cu = (int32_t)__builtin_floorf(hu), cv = (int32_t)__builtin_floorf(hv);
    cu = cu < g.U0 ? g.U0 : (cu > g.U0 + g.W - 1 ? g.U0 + g.W - 1 : cu);
    cv = cv < g.V0 ? g.V0 : (cv > g.V0 + g.H - 1 ? g.V0 + g.H - 1 : cv);
    int32_t cell[3];
#pragma unroll
    for (int k = 0; k < 3; k++) cell[k] = k == g.a ? g.slice : (k == g.u ? cu : cv);
    index = lin3(cell[0], cell[1], cell[2], n);
    face = g.face;
    // the primary-only shade of the raymarcher: no shadow or AO rays
    const float lightc = pick3(sh.light, g.a);
    float lambert = g.pos ? lightc : -lightc;
    if (lambert < 0.0f) lambert = 0.0f;
    shade = shade_value(lambert, 1.0f, false, 0, 1);
  }
  if (out.index_bytes == 8)
    ((int64_t *)out.index)[i] = index;
  else
    ((int32_t *)out.index)[i] = (int32_t)index;
  if (out.face) out.face[i] = (uint8_t)face;
  if (out.t) out.t[i] = t;
  if (out.shade) out.shade[i] = shade;
}

}  // namespace meso

using namespace meso;

struct meso_raster {
  meso_context *ctx = nullptr;
  void *scratch = nullptr;  // holds the arrays of s
  uint64_t shell_line = 1ull << 32;  // chunks * pixels above which there are shells
  int32_t max_width = 0, max_height = 0;
  RasterScratch s{};
};

extern "C" {

meso_status meso_raster_create(meso_context *ctx, int32_t max_width, int32_t max_height,
                               meso_raster **out) {
  MESO_CHECK(ctx && out, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "NULL argument");
  *out = nullptr;
  MESO_CHECK(max_width >= 1 && max_height >= 1 && max_width <= 16384 && max_height <= 16384,
             MESO_ERR_ARGUMENT_OUT_OF_RANGE, "frame %dx%d outside 1..16384", max_width,
             max_height);
  meso_raster *r = new meso_raster;
  r->ctx = ctx;
  r->max_width = max_width;
  r->max_height = max_height;
  r->s.limits = ListLimits{kMaxRecords, kMaxTests};
  const uint64_t npx = (uint64_t)max_width * (uint64_t)max_height;
  const DepthLevels d = depth_levels(nullptr, max_width, max_height);
  const uint64_t depth = (uint64_t)d.at128 + (uint64_t)d.w128 * ((uint32_t)(max_height + 127) / 128u);
  // one allocation, each array from a multiple of 256 bytes (one for each took
  // 1.2 ms for frames of 1920x1080, this 0.29)
  const uint64_t bytes[] = {npx * 8, npx * 12, depth * 4, (uint64_t)kMaxItems * 4,
                            (uint64_t)kMaxRecords * 16, (uint64_t)kMaxRecords * 8,
                            (uint64_t)kMaxWindows * 4, kRasterCounters * 8};
  uint64_t total = 0;
  for (uint64_t b : bytes) total += (b + 255u) & ~255ull;
  if (hipMalloc(&r->scratch, total) != hipSuccess) {
    (void)hipGetLastError();
    delete r;
    return fail(MESO_ERR_OUT_OF_MEMORY, "raster: cannot allocate its scratch");
  }
  uint8_t *at = (uint8_t *)r->scratch;
  int k = 0;
  const auto take = [&](auto *&p) {
    p = (std::remove_reference_t<decltype(p)>)at;
    at += (bytes[k++] + 255u) & ~255ull;
  };
  take(r->s.keys);
  take(r->s.rays);
  take(r->s.far_t);
  take(r->s.items);
  take(r->s.rec_a);
  take(r->s.rec_b);
  take(r->s.windows);
  take(r->s.counters);
  *out = r;
  return MESO_OK;
}

meso_status meso_raster_set_list_limits(meso_raster *r, uint32_t records, uint32_t windows) {
  MESO_CHECK(r, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "NULL argument");
  r->s.limits = ListLimits{std::min(records, kMaxRecords),
                           (uint64_t)std::min(windows, kMaxWindows) * kWindow};
  return MESO_OK;
}

meso_status meso_raster_set_shell_line(meso_raster *r, uint64_t chunk_pixels) {
  MESO_CHECK(r, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "NULL argument");
  r->shell_line = chunk_pixels;
  return MESO_OK;
}

meso_status meso_raster_destroy(meso_raster *r) {
  if (!r) return MESO_OK;
  (void)hipDeviceSynchronize();
  (void)hipFree(r->scratch);
  delete r;
  return MESO_OK;
}

meso_status meso_raster_pool(meso_raster *r, meso_chunk_pool *pool, const meso_camera *cam,
                             const meso_shading *shading, const meso_ray_outputs *out,
                             meso_stream stream) {
  MESO_CHECK(r && pool && out, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "NULL argument");
  meso_status st = check_camera(cam);
  if (st != MESO_OK) return st;
  MESO_CHECK(cam->width <= r->max_width && cam->height <= r->max_height,
             MESO_ERR_ARGUMENT_OUT_OF_RANGE, "frame %dx%d larger than the raster's %dx%d",
             cam->width, cam->height, r->max_width, r->max_height);
  MESO_CHECK(out->size >= sizeof(meso_ray_outputs), MESO_ERR_ARGUMENT_OUT_OF_RANGE,
             "meso_ray_outputs.size too small");
  MESO_CHECK(out->hit_index, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "hit_index is NULL");
  MESO_CHECK(out->index_bytes == 4 || out->index_bytes == 8, MESO_ERR_ARGUMENT_OUT_OF_RANGE,
             "index_bytes must be 4 or 8");
  const PoolView pv = pool_view(pool);
  MESO_CHECK(pv.scene->ctx == r->ctx, MESO_ERR_ARGUMENT_OUT_OF_RANGE,
             "pool of another context");
  const uint64_t nvox = (uint64_t)pv.scene->n * pv.scene->n * pv.scene->n;
  MESO_CHECK(out->index_bytes == 8 || nvox <= 0x7FFFFFFFull, MESO_ERR_ARGUMENT_OUT_OF_RANGE,
             "scene of %llu voxels needs 8-byte hit indices", (unsigned long long)nvox);
  MESO_CHECK((uint64_t)pv.capacity * (uint64_t)pv.per_slot <= 0xFFFFFFFFull,
             MESO_ERR_NOT_SUPPORTED, "pool of more than 2^32 quad places");
  DevShading sh{};
  if (shading && shading->size >= sizeof(meso_shading) &&
      (shading->light[0] != 0.0f || shading->light[1] != 0.0f || shading->light[2] != 0.0f))
    derive_shading(shading, &sh);
  else
    sh.light[1] = 1.0f;
  DevCamera dc;
  derive_camera(cam, &dc);
  RayOut ro{out->hit_index, out->index_bytes, out->face, out->t, out->shade, nullptr};
  const hipStream_t s = stream_of(r->ctx, stream);
  const uint64_t npx = (uint64_t)cam->width * (uint64_t)cam->height;
  // quads per item: the fewest (a multiple of 64) whose items fit the list
  // whatever the slots hold
  const uint32_t cap = (uint32_t)pv.capacity, per = (uint32_t)pv.per_slot;
  uint32_t batch = 64u;
  while ((uint64_t)cap * ((per + batch - 1u) / batch) > kMaxItems ||
         (per + batch - 1u) / batch > 1024u)  // the batch's place in an item: 10 bits
    batch *= 2u;
  RasterView v;
  v.fx = (float)(0.5 * cam->width / (double)dc.sx);
  v.fy = (float)(0.5 * cam->height / (double)dc.sy);
  v.cx = (float)(0.5 * cam->width - 0.5);
  v.cy = (float)(0.5 * cam->height - 0.5);
  v.eye_sum = std::fabs(dc.eye[0]) + std::fabs(dc.eye[1]) + std::fabs(dc.eye[2]);
  v.f_max = v.fx > v.fy ? v.fx : v.fy;
  v.s_one = 1.5f * (1.0f + (dc.sx > dc.sy ? dc.sx : dc.sy));
  v.ray_err = 8e-7f * v.f_max * (1.0f + dc.sx * dc.sx + dc.sy * dc.sy);
  const DepthLevels depth = depth_levels(r->s.far_t, cam->width, cam->height);
  hipLaunchKernelGGL(raster_begin_kernel, grid_1d((npx + 255) / 256), dim3(256), 0, s, dc, r->s, npx);
  MESO_HIP(hipGetLastError());
  const uint32_t waves = (uint32_t)r->ctx->props.multiProcessorCount * 16u;
  // Shell bounds in voxels (3 and 8 chunks).  A shell costs 17 us of launches
  // and small kernels, 25 in frames of 3840x2160, and saves the quads hidden by
  // the nearer ones: two shells (at 112) took 355 us where three (64, 160) took
  // 318, (64, 160, 320) 262, and these 254 (16,384 cave chunks at 1920x1080).
  // What is saved grows with the chunks and with the pixels that a hidden quad
  // covers, so few chunks or small frames have one shell for all.  Cave chunks
  // with one shell and with three: 512 at 1920x1080 146 us and 183, at 3840x2160
  // 374 and 383; 2,048 at 640x360 96 and 146, at 1920x1080 247 and 233, at
  // 3840x2160 648 and 485; 16,384 at 320x180 134 and 167, at 640x360 186 and
  // 179, at 1920x1080 579 and 291.  The line lies where the two meet.
  constexpr int kShells = 3;
  constexpr float kBound[kShells + 1] = {0.0f, 96.0f, 256.0f, INFINITY};
  constexpr float kAll[2] = {0.0f, INFINITY};
  const bool many = pv.resident * npx > r->shell_line;
  const int shells = many ? kShells : 1;
  const float *bound = many ? kBound : kAll;
  for (int k = 0; k < shells; k++) {
    hipLaunchKernelGGL(raster_list_kernel, dim3((cap + 1023u) / 1024u), dim3(1024), 0, s, dc,
                       v, pv.slot_chunk, pv.slot_count, cap, per, (uint32_t)pv.nc, batch,
                       bound[k] * bound[k], bound[k + 1] * bound[k + 1], k > 0, depth, r->s);
    MESO_HIP(hipGetLastError());
    hipLaunchKernelGGL(raster_quads_kernel, dim3(std::min(waves / 8u, kMaxLotGroups)), dim3(kQuadThreads), 0, s, dc, v, pv.slot_chunk,
                       pv.slot_count, pv.quads, per, (uint32_t)pv.nc, batch, test_spread(npx), k > 0, depth, r->s);
    MESO_HIP(hipGetLastError());
    hipLaunchKernelGGL(raster_pixels_kernel, dim3(2u * waves), dim3(64), 0, s, dc, r->s);
    MESO_HIP(hipGetLastError());
    if (k + 1 < shells) {
      hipLaunchKernelGGL(raster_depth_kernel,
                         dim3(depth.w128, (uint32_t)(cam->height + 127) / 128u), dim3(1024), 0, s,
                         r->s.keys, cam->width, cam->height, depth, r->s.far_t);
      MESO_HIP(hipGetLastError());
    }
  }
  hipLaunchKernelGGL(raster_resolve_kernel, grid_1d((npx + 255) / 256), dim3(256), 0, s, dc, sh,
                     pv.slot_chunk, pv.quads, per, (uint32_t)pv.nc, pv.scene->n, ro, r->s);
  MESO_HIP(hipGetLastError());
  return MESO_OK;
}

meso_status meso_raster_stats_get(meso_raster *r, meso_raster_stats *out, meso_stream stream) {
  MESO_CHECK(r && out, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "NULL argument");
  MESO_CHECK(out->size >= sizeof(meso_raster_stats), MESO_ERR_ARGUMENT_OUT_OF_RANGE,
             "meso_raster_stats too small");
  const hipStream_t s = stream_of(r->ctx, stream);
  uint64_t c[kRasterCounters];
  MESO_HIP(hipMemcpyAsync(c, r->s.counters, sizeof(c), hipMemcpyDeviceToHost, s));
  MESO_HIP(hipStreamSynchronize(s));
  out->segments = (uint32_t)c[kRasterRecords];
  out->overflow_quads = (uint32_t)(c[kRasterRecords] >> 32);
  out->small_quads = (uint32_t)c[kRasterDrawn];
  out->large_quads = (uint32_t)(c[kRasterDrawn] >> 32);
  return MESO_OK;
}

}  // extern "C"
