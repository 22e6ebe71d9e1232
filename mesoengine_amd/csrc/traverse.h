// Device-side voxel traversal for gfx950: Amanatides & Woo (1987) DDA with
// hierarchical empty-space skipping over 128^3 blocks, 32^3 blocks, 8^3
// bricks, the 4^3 and 2^3 blocks inside a brick, and voxels.  Every float operation is written out in a fixed order
// and the library is compiled with -ffp-contract=off, so results are the IEEE
// binary32 results of these operations: the integer outputs (voxel index,
// face) and the float outputs (t, shade) are reproducible bit for bit by any
// scalar IEEE implementation of the same steps.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "meso_internal.h"

namespace meso {

constexpr uint32_t kEmpty = 0xFFFFFFFFu;
constexpr int kFaceInside = 6;
constexpr int kFaceMiss = 0xFF;

// Face ids follow Runtimes/Shape/Cube.h:25-54: 0:+Z 1:-Z 2:+Y 3:-Y 4:+X 5:-X.
// A ray stepping +x enters a voxel through its -X face.
__device__ __forceinline__ int entry_face(int axis, int step) {
  int base = axis == 2 ? 0 : (axis == 1 ? 2 : 4);
  return base + (step > 0 ? 1 : 0);
}
__device__ __forceinline__ int face_axis(int f) { return f < 2 ? 2 : (f < 4 ? 1 : 0); }

struct Ray {
  float o[3], d[3], inv[3];  // inv: +inf where d = 0
  int32_t step[3];
  // the exit plane of block b is b + pos: 1 where step > 0, 0 where step < 0,
  // and 2 where step = 0, so that plane lies beyond the origin and its t,
  // (plane - o) * inf, is +inf: an axis the ray does not move along is never
  // the nearest, with no select per step
  int32_t pos[3];
  uint32_t posmask;  // bit a: step[a] > 0
  uint32_t negmask;  // bit a: step[a] < 0 (the next cell is one below the plane)
  // the direction the cell can move in on axis a: step[a] > 0, or on an
  // axis the ray does not move along, floor(o[a]) above the start cell
  bool up[3];
};

__device__ __forceinline__ void ray_setup(Ray &r, const float o[3], const float d[3]) {
  r.posmask = 0u;
  r.negmask = 0u;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    r.o[a] = o[a];
    r.d[a] = d[a];
    // one division per axis, kept where d != 0: written per branch, the
    // divide sequence is emitted twice and lanes of both signs run both
    const float inv = 1.0f / d[a];
    const bool pos = d[a] > 0.0f, neg = d[a] < 0.0f;
    r.step[a] = pos ? 1 : (neg ? -1 : 0);
    r.inv[a] = (pos || neg) ? inv : __builtin_inff();
    r.pos[a] = pos ? 1 : (neg ? 0 : 2);
    r.up[a] = pos;
    r.posmask |= (r.step[a] > 0 ? 1u : 0u) << a;
    r.negmask |= (r.step[a] < 0 ? 1u : 0u) << a;
  }
}

__device__ __forceinline__ float plane_t(float o, float inv, float b) {
  float q = b - o;
  return q * inv;
}
// smallest t, ties to x then y
__device__ __forceinline__ int argmin3(float t0, float t1, float t2) {
  if (t0 <= t1 && t0 <= t2) return 0;
  return t1 <= t2 ? 1 : 2;
}

struct WalkState {
  int32_t cell[3];
  float t;
  int32_t face;
};

struct StepCounts {
  uint32_t n_vox, n_top, n_node, n_brickslot, n_brickmask, n_coarse, n_iter;
};

__device__ __forceinline__ int64_t lin3(int64_t x, int64_t y, int64_t z, int64_t n) {
  return x + y * n + z * n * n;
}
// Index of (x,y,z) in an n^3 grid of blocks or bricks, with 24-bit multiplies
// (full rate; a 32-bit multiply is quarter rate): scene edges are at most
// 8192, so n <= 1024 and x, y, z < n, and every operand stays below 2^24 and
// every product below 2^32.
__device__ __forceinline__ uint32_t lin3u(uint32_t x, uint32_t y, uint32_t z, uint32_t n) {
  return x + __umul24(y + __umul24(z, n), n);
}

// The median of a, b, c: for lo <= hi, med3_i32(x, lo, hi) clamps x into
// [lo, hi] in one instruction (the compiler cannot see lo <= hi).
__device__ __forceinline__ int32_t med3_i32(int32_t a, int32_t b, int32_t c) {
  int32_t m;
  asm("v_med3_i32 %0, %1, %2, %3" : "=v"(m) : "v"(a), "v"(b), "v"(c));
  return m;
}

// (int32_t)floor(x) in one instruction: on gfx950, v_cvt_flr_i32_f32 gives
// the same result as v_floor_f32 then v_cvt_i32_f32 for every finite float
// (checked on the device over every finite float by tests/native/floor_convert_probe.hip)
__device__ __forceinline__ int32_t floor_i32(float x) {
  int32_t r;
  asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
  return r;
}

// (1 << k) - 1 for k in [0, 31], one instruction
__device__ __forceinline__ int32_t low_mask(int32_t k) {
  int32_t m;
  asm("v_bfm_b32 %0, %1, 0" : "=v"(m) : "v"(k));
  return m;
}

// One step at level 2^sh (sh = 0 voxel, 3 brick, 5 and 7 empty blocks): leave
// the block holding the current cell through its nearest plane.  The other
// two coordinates come from the exit point, clamped into the block and the
// scene and never moving against the ray; at sh = 0 the block is the cell
// itself, so the clamp keeps them, which is the plain voxel step.  Written
// without branches (selects only), so that the lanes of a wave stepping at
// different levels stay converged.  Returns false when the step along the
// chosen axis leaves the scene's solid box (nothing solid lies beyond it);
// the step is computed all the same (no branch), and a walk that gets false
// ends without reading the cell.
template <bool LEVELS = true>
__device__ __forceinline__ bool advance(const Ray &r, const DevScene &s, int32_t sh, WalkState &w) {
  const int32_t n = s.n;
  float tb[3];
  int32_t bc[3], pl[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    bc[a] = w.cell[a] >> sh;
    pl[a] = (bc[a] + r.pos[a]) << sh;  // the exit plane on this axis
    // +inf where step = 0: pl is at least the cell + 2 there, and the
    // origin's coordinate stays below the cell + 2 (the cell is floor(o),
    // or for a secondary ray the hit cell, whose face holds o)
    tb[a] = plane_t(r.o[a], r.inv[a], (float)pl[a]);
  }
  // the chosen axis by selects and bit extracts only: an index into the
  // ray's arrays would move them out of registers
  const int ax = argmin3(tb[0], tb[1], tb[2]);
  const bool a0 = ax == 0, a1 = ax == 1;
  const float t = a0 ? tb[0] : (a1 ? tb[1] : tb[2]);
  const int32_t pax = a0 ? pl[0] : (a1 ? pl[1] : pl[2]);
  const int32_t na = pax - (int32_t)((r.negmask >> ax) & 1u);
  const int32_t face = 4 - 2 * ax + (int32_t)((r.posmask >> ax) & 1u);  // entry_face
  // compared with each axis' bounds (scalar operands; one unsigned compare
  // per axis) and the chosen axis' answer kept, combined as lane masks:
  // selecting the bounds per lane would hold them in vector registers for
  // the whole walk
  const bool out0 = (uint32_t)(na - s.lo[0]) >= (uint32_t)(s.hi[0] - s.lo[0]);
  const bool out1 = (uint32_t)(na - s.lo[1]) >= (uint32_t)(s.hi[1] - s.lo[1]);
  const bool out2 = (uint32_t)(na - s.lo[2]) >= (uint32_t)(s.hi[2] - s.lo[2]);
  const bool out = (a0 & out0) | (a1 & out1) | (!a0 & !a1 & out2);
  if constexpr (!LEVELS) {  // voxel steps only (dense grid): the other cells stay
#pragma unroll
    for (int b = 0; b < 3; b++) w.cell[b] = b == ax ? na : w.cell[b];
    w.t = t;
    w.face = face;
    return !out;
  }
  const int32_t span = low_mask(sh);
#pragma unroll
  for (int b = 0; b < 3; b++) {
    float dt = r.d[b] * t;
    float p = r.o[b] + dt;
    int32_t c = floor_i32(p);
    // clamp into the block [lo, hi], then not below the cell when stepping
    // up or above it when stepping down: the cell lies in [lo, hi], so that
    // is one clamp between the cell and one bound (a single med3).  On an
    // axis the ray does not move along, c is floor(o) on every step and
    // the cell only moves toward it, so the side up[] fixed at the start
    // holds for the whole walk and the same clamp gives clamp(c, lo, hi).
    const int32_t lo = bc[b] << sh;
    int32_t hi = lo + span;
    hi = hi > n - 1 ? n - 1 : hi;
    c = med3_i32(c, w.cell[b], r.up[b] ? hi : lo);
    w.cell[b] = b == ax ? na : c;
  }
  w.t = t;
  w.face = face;
  return !out;
}

// The 4x4 2^2 blocks of an 8x8 plane of a brick (bit x + 8 y) that hold a set
// bit, as 16 bits (bit cx + 4 cy): fold x and y pairs onto the even bits,
// then gather the 16 even bits.
__device__ __forceinline__ uint32_t plane_blocks2(uint64_t w) {
  w |= w >> 1;
  w |= w >> 8;
  w &= 0x0055005500550055ull;
  w = (w | (w >> 1)) & 0x0033003300330033ull;
  w = (w | (w >> 2)) & 0x000F000F000F000Full;
  w = (w | (w >> 12)) & 0x000000FF000000FFull;
  w = (w | (w >> 24)) & 0xFFFFull;
  return (uint32_t)w;
}

// One bit per aligned 2^3 block of a brick (bit cx + 4 cy + 16 cz), from its
// 64-byte mask (word z, bit x + 8 y): the planes of each z pair ORed, folded.
__device__ __forceinline__ uint64_t brick_blocks2(const uint64_t *mask) {
  uint64_t sub = 0;
#pragma unroll
  for (int p = 0; p < 4; p++)
    sub |= (uint64_t)plane_blocks2(mask[2 * p] | mask[2 * p + 1]) << (16 * p);
  return sub;
}

// A brick written by 512 lanes (lane = voxel x + 8 y + 64 z, each wave one z
// plane) whose plane bits are `b` (the wave's ballot of solid voxels): the
// brick's 2^3-block bits, returned to lane 0.  Every lane of the workgroup
// must call it (it synchronises the workgroup).
__device__ __forceinline__ uint64_t brick_blocks2_from_planes(uint64_t b) {
  __shared__ uint32_t plane[8];
  if ((threadIdx.x & 63u) == 0) plane[threadIdx.x >> 6] = plane_blocks2(b);
  __syncthreads();
  uint64_t sub = 0;
  if (threadIdx.x == 0) {
#pragma unroll
    for (int p = 0; p < 4; p++) sub |= (uint64_t)(plane[2 * p] | plane[2 * p + 1]) << (16 * p);
  }
  return sub;
}

__device__ __forceinline__ bool occ_bit(const uint32_t *bits, uint32_t i) {
  return (bits[i >> 5] >> (i & 31u)) & 1u;
}

// Cached answers of the coarse levels for the cell a walk is in.  The valid
// levels always form a prefix (the 128^3 block, then the 32^3 block, then
// the brick), and each valid level's block holds the walk's previous cell.
// So the cell is still in a valid level's block of edge 2^k exactly when dv,
// the previous step's (x ^ x') | (y ^ y') | (z ^ z'), is below 2^k, and
// max(dv, vmask) >= 2^k, with vmask one below the edge of the finest valid
// level (255: none valid), says that level k must be looked up.
struct WalkCache {
  uint32_t dv, vmask;
  bool e128, e32;
  uint32_t node, slot;
  uint64_t b32, sub;  // b32: allocated bricks of the 32^3 block; sub: 2^3-block bits of the brick
  __device__ __forceinline__ void reset() {
    dv = 0;
    vmask = 255u;
    e128 = e32 = false;
    node = slot = kEmpty;
    b32 = sub = 0;
  }
};

// KIND of a dense grid walked a few cells at a time, for a kernel of all scene
// kinds that has no registers for more
constexpr int kDenseShort = 4;

enum : int { kWalkOn = 0, kWalkHit = 1, kWalkOut = 2 };

// One step of a walk from a cell whose entry t is below tmax: kWalkHit when
// the cell is solid (material set), kWalkOut when the ray leaves the scene or
// the next cell's entry t reaches tmax, else kWalkOn after stepping to the
// next cell.  (Testing the next cell's t here, not at the top of the next
// step, saves a branch per step; walk tests the first cell's.)  KIND: 1 dense u8 (voxel
// steps only), 2 brick map, 3 two-level.  A brick scene steps at the coarsest
// empty level holding the cell: 128^3 block, 32^3 block (its word of
// allocated bricks, which also names the empty bricks without reading their
// slots), brick, the 4^3 and 2^3 blocks of a non-empty brick (from its 2^3-
// block bits, read once per brick), else the voxel (one 8-byte mask word).
// Brick scenes come here in launches that count steps; see walk_bricks().
template <int KIND, bool COUNT>
__device__ __forceinline__ int walk_step(const DevScene &s, const Ray &r, WalkState &w,
                                         WalkCache &c, float tmax, uint16_t &material,
                                         StepCounts &cnt) {
  const int32_t n = s.n;
  if (COUNT) cnt.n_iter++;
  if constexpr (KIND == 1 || KIND == kDenseShort) {
    if (COUNT) cnt.n_vox++;
    const uint8_t v = s.dense[lin3(w.cell[0], w.cell[1], w.cell[2], n)];
    if (v) {
      material = v;
      return kWalkHit;
    }
    return advance<false>(r, s, 0, w) && w.t < tmax ? kWalkOn : kWalkOut;
  } else {
    const uint32_t n128 = (uint32_t)(n + 127) >> 7, n32 = (uint32_t)(n + 31) >> 5;
    // one flat pass over the levels (no nesting, so a wave whose lanes sit
    // at different levels runs each piece once): refresh a level's cached
    // answer when the cell left its block, then step at the coarsest empty
    // level, or stop at a solid voxel
    const uint32_t x = (uint32_t)w.cell[0], y = (uint32_t)w.cell[1], z = (uint32_t)w.cell[2];
    const uint32_t q = c.dv > c.vmask ? c.dv : c.vmask;
    if (q >= 128u) {
      if constexpr (KIND == 3) {
        if (COUNT) cnt.n_top++;
        c.node = s.top[lin3u(x >> 7, y >> 7, z >> 7, n128)];
        c.e128 = c.node == kEmpty;
      } else {
        if (COUNT) cnt.n_coarse++;
        c.e128 = !occ_bit(s.occ128, lin3u(x >> 7, y >> 7, z >> 7, n128));
      }
    }
    if (!c.e128 && q >= 32u) {
      if (COUNT) cnt.n_coarse++;
      c.b32 = s.bricks32[lin3u(x >> 5, y >> 5, z >> 5, n32)];
      c.e32 = c.b32 == 0;
    }
    const bool coarse = c.e128 || c.e32;
    if (!coarse && q >= 8u) {
      if (COUNT) {
        if constexpr (KIND == 3)
          cnt.n_node++;
        else
          cnt.n_brickslot++;
      }
      c.slot = kEmpty;
      if ((c.b32 >> (((x >> 3) & 3u) + 4u * ((y >> 3) & 3u) + 16u * ((z >> 3) & 3u))) & 1ull) {
        // the slot and the 2^3-block word are both kept per brick cell, so
        // the two loads go out together (cells are below 2^30)
        const uint32_t cell =
            KIND == 3 ? c.node * 4096u + lin3u((x >> 3) & 15u, (y >> 3) & 15u, (z >> 3) & 15u, 16u)
                      : lin3u(x >> 3, y >> 3, z >> 3, (uint32_t)n >> 3);
        c.slot = s.slots[cell];
        c.sub = s.blocks[cell];
        if (COUNT) cnt.n_brickmask++;
      }
    }
    // inside a non-empty brick: step over its empty 4^3 and 2^3 blocks
    // (computed on every step without a branch: outside a brick c.sub is
    // stale and e4, e2 are not used)
    const bool in_brick = !coarse && c.slot != kEmpty;
    // bit of the cell's 2^3 block in sub ((x&7)>>1) + 4 ((y&7)>>1) + 16
    // ((z&7)>>1); its bits 1, 3 and 5 are the 4^3 block's corner bit
    const uint32_t i2 = ((x >> 1) & 3u) | ((y << 1) & 12u) | ((z << 3) & 48u);
    const bool e4 = ((uint32_t)(c.sub >> (i2 & 0x2Au)) & 0x00330033u) == 0;
    const bool e2 = ((c.sub >> i2) & 1ull) == 0;
    if (in_brick && !e4 && !e2) {
      if (COUNT) cnt.n_vox++;
      // 32-bit word index: a scene holds fewer than 2^29 bricks (checked
      // when it is generated or uploaded), so slot * 8 + 7 is below 2^32
      const uint32_t lz = z & 7u, lxy = (x & 7u) | ((y & 7u) << 3);
      const uint64_t m = s.masks[c.slot * 8u + lz];
      if ((m >> lxy) & 1ull) {
        material = s.voxels[(uint64_t)c.slot * 512u + lxy + 64u * lz];
        return kWalkHit;
      }
    }
    c.vmask = c.e128 ? 127u : (c.e32 ? 31u : 7u);
    const int32_t sh =
        c.e128 ? 7 : (c.e32 ? 5 : (!in_brick ? 3 : (e4 ? 2 : (e2 ? 1 : 0))));
    const bool on = advance(r, s, sh, w) && w.t < tmax;
    c.dv = (x ^ (uint32_t)w.cell[0]) | (y ^ (uint32_t)w.cell[1]) | (z ^ (uint32_t)w.cell[2]);
    return on ? kWalkOn : kWalkOut;
  }
}

// Dense grid: the cells a ray visits do not depend on what they hold, so a walk
// finds its next AHEAD cells first and then loads them together.  One
// voxel load at a time bounded it by latency: a 256x256 frame of a 256^3 grid
// has one wave per SIMD, and each of some 200 steps waited for its load (148
// us, now 53; 4 cells at a time 79, 8 70 and 16 68 before the steps below).
// Now the steps' own instructions bound it, so they are few: a cell's exit
// planes are kept as floats (whole numbers below 2^24, exact), each plane t is
// recomputed from its plane as advance() does, and a walk ends at t_out, the
// least t of the grid's far planes, which needs no count of the cells left (68
// us with one).  A step of t < t_out stays in the grid (t never falls from
// plane to plane of an axis), and the cells, t and faces are those of
// advance() to the bit.  (Taken back: one bit per voxel instead of a byte
// changed nothing; crossing empty 8^3 blocks in one step, with the exit cell
// made exact, was 5 times slower, lanes in blocks and lanes in steps running
// both ways in every trip.)
constexpr int kDenseAhead = 16;
// Rays that end within a few cells (solid scenes, eyes in them, occlusion rays of
// rough ones) would pay for 16 all the same, so a walk first looks at some cells
// one by one.  256^3 voxels at 1920x1080, primary rays, then with shadow and four
// AO rays: solid from within 34 us with batches alone, now 18 (17 where a lane
// steps through advance()); half of the voxels solid 38 and 183, now 28 and 152
// (25 and 129); a tenth of them 61 and 329 now (80 and 363 there).  4 cells: 31
// and 169 for the half, 62 and 314 for the tenth; a batch of 4 and then of 8
// instead: 30 and 137, but 323 us where hills take 261, the code of two sizes of
// batches taking registers.
constexpr int kDenseSingle = 8;
// where registers are short: the serving kernel has 131 with 16, which leaves 3
// waves a SIMD, and 96 with 4
constexpr int kDenseAheadShort = 4;
constexpr int32_t kDenseIndexed = 1625;  // 1625^3 < 2^32: 32-bit voxel indices

struct DenseRay {
  float t_out;  // least t of the grid's far planes
  int axis;     // its axis, of equal ones the first, which advance() takes
  // whether walk_dense() may take the ray: no plane t is NaN (the moving axes'
  // reciprocals are finite), and neighbouring planes differ in t (the origin
  // and the grid are within 2^16, so b - o keeps 2^-7)
  __device__ __forceinline__ bool setup(const DevScene &s, const Ray &r) {
    bool ok = s.n <= kDenseIndexed;
    float tb[3];
#pragma unroll
    for (int a = 0; a < 3; a++) {
      ok = ok && __builtin_fabsf(r.o[a]) < 65536.0f &&
           (r.step[a] == 0 || __builtin_fabsf(r.inv[a]) < __builtin_inff());
      const float t = plane_t(r.o[a], r.inv[a], r.step[a] > 0 ? (float)s.n : 0.0f);
      tb[a] = r.step[a] == 0 ? __builtin_inff() : t;
    }
    axis = argmin3(tb[0], tb[1], tb[2]);
    t_out = axis == 0 ? tb[0] : (axis == 1 ? tb[1] : tb[2]);
    return ok;
  }
  // Whether a plane of an axis before `axis` has the t t_out: its cell is
  // still entered before the ray leaves.  Such a plane is within 2^-6 of the
  // ray's point at t_out, so the nearest whole number is the only one to try.
  __device__ __forceinline__ bool ties(const Ray &r) const {
    bool tie = false;
#pragma unroll
    for (int a = 0; a < 2; a++) {
      const float dt = r.d[a] * t_out;
      const float t = plane_t(r.o[a], r.inv[a], __builtin_rintf(r.o[a] + dt));
      tie = tie || (a < axis && r.step[a] != 0 && t == t_out);
    }
    return tie;
  }
};

// The nearest exit plane: its t and axis, and the planes of the cell behind it.
__device__ __forceinline__ float dense_step(const Ray &r, float plane[3], int &ax) {
  const float t0 = plane_t(r.o[0], r.inv[0], plane[0]), t1 = plane_t(r.o[1], r.inv[1], plane[1]),
              t2 = plane_t(r.o[2], r.inv[2], plane[2]);
  const float t = fminf(fminf(t0, t1), t2);
  const bool a0 = t0 == t, a1 = !a0 && t1 == t;  // argmin3: no NaN here
  ax = a0 ? 0 : (a1 ? 1 : 2);
  plane[0] += a0 ? (float)r.step[0] : 0.0f;
  plane[1] += a1 ? (float)r.step[1] : 0.0f;
  plane[2] += a0 || a1 ? 0.0f : (float)r.step[2];
  return t;
}

// A walk of a dense grid, a batch of cells at a time.
struct DenseWalk {
  const DevScene &s;
  const Ray &r;
  const DenseRay &e;
  float tmax, t_lim;
  float plane[3], from[3];  // exit planes of the next cell, and of the batch's first
  uint32_t stride[3], idx, solid;
  bool on;

  __device__ __forceinline__ DenseWalk(const DevScene &s_, const Ray &r_, const DenseRay &e_,
                                       const WalkState &w, float tmax_)
      : s(s_), r(r_), e(e_), tmax(tmax_), solid(0), on(true) {
    const uint32_t n = (uint32_t)s.n;
    t_lim = tmax < e.t_out ? tmax : e.t_out;
#pragma unroll
    for (int a = 0; a < 3; a++) {
      plane[a] = from[a] = (float)(w.cell[a] + r.pos[a]);
      const uint32_t d = a == 0 ? 1u : (a == 1 ? n : n * n);
      stride[a] = r.step[a] < 0 ? 0u - d : d;
    }
    idx = (uint32_t)w.cell[0] + n * ((uint32_t)w.cell[1] + n * (uint32_t)w.cell[2]);
  }
  __device__ __forceinline__ int32_t face(int ax) const {  // entry_face
    return 4 - 2 * ax + (int32_t)((r.posmask >> ax) & 1u);
  }
  __device__ __forceinline__ int32_t cell(int a) const { return (int32_t)plane[a] - r.pos[a]; }

  // The next CELLS cells (0: one that is empty, unread): true when none is solid and
  // the walk goes on behind them (w.t and w.face then are the next cell's).
  template <int CELLS>
  __device__ __forceinline__ bool batch(WalkState &w) {
    constexpr int N = CELLS ? CELLS : 1;
    from[0] = plane[0], from[1] = plane[1], from[2] = plane[2];
    const uint32_t first = idx;
    uint32_t at[N];
    float t = 0.0f;
    int ax = 0;
#pragma unroll
    for (int i = 0; i < N; i++) {
      // cells past the walk's end are read as the batch's first cell, which is
      // its first solid one or empty
      at[i] = on ? idx : first;
      t = dense_step(r, plane, ax);
      idx += ax == 0 ? stride[0] : (ax == 1 ? stride[1] : stride[2]);
      on = on && t < t_lim;
    }
    uint8_t v[N];
#pragma unroll
    for (int i = 0; i < N; i++) v[i] = CELLS ? s.dense[at[i]] : 0;
    solid = 0;
#pragma unroll
    for (int i = 0; i < N; i++) solid |= (v[i] ? 1u : 0u) << i;
    if (solid != 0u || !on) return false;
    w.t = t;
    w.face = face(ax);
    return true;
  }

  // After the batch that ended the walk, its steps once more, to the first solid
  // cell for its t, face and cell, or to the planes that have the t the ray
  // leaves at.
  __device__ __forceinline__ bool finish(WalkState &w, uint16_t &material) {
    plane[0] = from[0], plane[1] = from[1], plane[2] = from[2];
    int ax = 0;
    if (solid) {
      for (uint32_t k = (uint32_t)__builtin_ctz(solid); k; k--) {
        w.t = dense_step(r, plane, ax);
        w.face = face(ax);
      }
    } else {
      if (!(e.t_out < tmax) || !e.ties(r)) return false;
      bool hit = false;
      while (!hit) {
        const float t_now = dense_step(r, plane, ax);
        if (t_now > e.t_out || (t_now == e.t_out && ax >= e.axis)) return false;
        if (t_now < e.t_out) continue;
        w.t = t_now;
        w.face = face(ax);
        hit = s.dense[lin3(cell(0), cell(1), cell(2), s.n)] != 0;
      }
    }
#pragma unroll
    for (int a = 0; a < 3; a++) w.cell[a] = cell(a);
    material = s.dense[lin3(w.cell[0], w.cell[1], w.cell[2], s.n)];
    return true;
  }
};

// SINGLE: cells looked at one by one first (see kDenseSingle), AHEAD: cells of
// a batch.  EMPTY: the start cell is known to be empty and not read again.
template <int SINGLE, int AHEAD, bool EMPTY>
__device__ __forceinline__ bool walk_dense(const DevScene &s, const Ray &r, const DenseRay &e,
                                           WalkState &w, float tmax, uint16_t &material) {
  DenseWalk d(s, r, e, w, tmax);
  bool more = true;
  if constexpr (EMPTY) more = d.batch<0>(w);
#pragma unroll 1
  for (int k = 0; k < SINGLE && more; k++) more = d.batch<1>(w);
  while (more) more = d.batch<AHEAD>(w);
  return d.finish(w, material);
}

// (a ^ -1) + b in one instruction
__device__ __forceinline__ int32_t not_add(int32_t a, int32_t b) {
  int32_t r;
  asm("v_xad_u32 %0, %1, -1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// The walk of a brick scene: walk_step() and advance() in one loop, the same
// cells, t and faces to the bit, for launches that count no steps.  The number
// of instructions bounds a frame (VALU issue above 90% of the time): 126 vector
// and 48 scalar ones a step, where walk_step() takes 144 and 52 (3840x2160
// caves with shadow and AO rays 1923 -> 1669 us, 1920x1080 hills with shadows
// 170 -> 146).
//  - b0, b1, b2, the end of the cell's block that the ray moves toward, are one
//    bit-select of the cell's low bits (all set where it moves up, else clear).
//    The exit plane, the clamp's bound and the next cell all come from them,
//    and a level is kept as its span of low bits.
//  - which levels are known is one value per lane, not lane masks, whose merges
//    at every branch are scalar work; and the loop has one exit.
//  - the next cell is computed on every axis and kept on the chosen one, which
//    takes fewer selects than selecting the plane and the direction.
//  - t_lim, the least t of the solid box's far planes (or tmax), replaces the
//    box test: a step of t < t_lim stays in the box on its axis, since t never
//    falls from plane to plane.  A step at or past it is tested as advance()
//    does, because blocks may reach past the box, and a cell may still be
//    entered at the t the ray leaves.
template <int KIND>
__device__ __forceinline__ bool walk_bricks(const DevScene &s, const Ray &r, WalkState &w,
                                            float tmax, uint16_t &material) {
  const int32_t n = s.n;
  const uint32_t n128 = (uint32_t)(n + 127) >> 7, n32 = (uint32_t)(n + 31) >> 5;
  int32_t um[3], beyond[3];
  float o[3], t_lim = tmax;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    um[a] = r.up[a] ? -1 : 0;
    asm("" : "+v"(um[a]));  // a value, not a select again at each use
    // An axis the ray does not move along: a plane 2^20 above the cell, and the
    // origin at most 2^19, so that its t is +inf.  (A hit point of an eye that
    // is 2^44 voxels away may lie farther off; cells are clamped to the scene,
    // 8192 at most, so the step sees no difference.)
    beyond[a] = r.step[a] > 0 ? 1 : (r.step[a] < 0 ? 0 : 1 << 20);
    o[a] = r.step[a] == 0 && r.o[a] > 524288.0f ? 524288.0f : r.o[a];
    const float far = r.step[a] > 0 ? s.fhi[a] : s.flo[a];
    const float t = plane_t(o[a], r.inv[a], r.step[a] == 0 ? __builtin_inff() : far);
    t_lim = fminf(t_lim, t);
  }
  int32_t cx = w.cell[0], cy = w.cell[1], cz = w.cell[2];
  // the cell's coarsest empty level: 127 for the 128^3 block, 31 for the 32^3
  // block, else 7; 255 none known.  slot: kEmpty outside a brick
  uint32_t dv = 0, level = 255u, node = kEmpty, slot = kEmpty;
  uint64_t b32 = 0, sub = 0;
  uint32_t hit = 0;
  for (;;) {
    const uint32_t x = (uint32_t)cx, y = (uint32_t)cy, z = (uint32_t)cz;
    const uint32_t q = dv > level ? dv : level;
    if (q >= 128u) {
      const uint32_t i = lin3u(x >> 7, y >> 7, z >> 7, n128);
      bool empty;
      if constexpr (KIND == 3) {
        node = s.top[i];
        empty = node == kEmpty;
      } else {
        empty = !occ_bit(s.occ128, i);
      }
      level = empty ? 127u : 7u;
      slot = kEmpty;
    }
    if (q >= 32u && level != 127u) {
      b32 = s.bricks32[lin3u(x >> 5, y >> 5, z >> 5, n32)];
      level = b32 == 0 ? 31u : 7u;
      slot = kEmpty;
    }
    if (q >= 8u && level == 7u) {
      slot = kEmpty;
      if ((b32 >> (((x >> 3) & 3u) + 4u * ((y >> 3) & 3u) + 16u * ((z >> 3) & 3u))) & 1ull) {
        const uint32_t cell =
            KIND == 3 ? node * 4096u + lin3u((x >> 3) & 15u, (y >> 3) & 15u, (z >> 3) & 15u, 16u)
                      : lin3u(x >> 3, y >> 3, z >> 3, (uint32_t)n >> 3);
        slot = s.slots[cell];
        sub = s.blocks[cell];
      }
    }
    const bool in_brick = slot != kEmpty;
    const uint32_t i2 = ((x >> 1) & 3u) | ((y << 1) & 12u) | ((z << 3) & 48u);
    const bool e4 = ((uint32_t)(sub >> (i2 & 0x2Au)) & 0x00330033u) == 0;
    const bool e2 = ((sub >> i2) & 1ull) == 0;
    if (in_brick && !e4 && !e2) {
      const uint32_t lz = z & 7u, lxy = (x & 7u) | ((y & 7u) << 3);
      const uint64_t m = s.masks[slot * 8u + lz];
      if ((m >> lxy) & 1ull) {
        hit = 1;
        break;
      }
    }
    const int32_t span = in_brick ? (e4 ? 3 : (e2 ? 1 : 0)) : (int32_t)level;
    const int32_t b0 = (um[0] & span) | (cx & ~span), b1 = (um[1] & span) | (cy & ~span),
                  b2 = (um[2] & span) | (cz & ~span);
    const int32_t p0 = b0 + beyond[0], p1 = b1 + beyond[1], p2 = b2 + beyond[2];
    const float t0 = plane_t(o[0], r.inv[0], (float)p0), t1 = plane_t(o[1], r.inv[1], (float)p1),
                t2 = plane_t(o[2], r.inv[2], (float)p2);
    const bool a0 = (t0 <= t1) & (t0 <= t2), a1 = !a0 & (t1 <= t2), a2 = !a0 & !a1;  // argmin3
    const float t = a0 ? t0 : (a1 ? t1 : t2);
    const float d0 = r.d[0] * t, d1 = r.d[1] * t, d2 = r.d[2] * t;
    const float q0 = o[0] + d0, q1 = o[1] + d1, q2 = o[2] + d2;
    const int32_t h0 = b0 > n - 1 ? n - 1 : b0, h1 = b1 > n - 1 ? n - 1 : b1,
                  h2 = b2 > n - 1 ? n - 1 : b2;
    const int32_t c0 = med3_i32(floor_i32(q0), cx, h0), c1 = med3_i32(floor_i32(q1), cy, h1),
                  c2 = med3_i32(floor_i32(q2), cz, h2);
    // (named first: a select does not move inline assembly into a branch)
    const int32_t n0 = not_add(um[0], p0), n1 = not_add(um[1], p1), n2 = not_add(um[2], p2);
    cx = a0 ? n0 : c0;
    cy = a1 ? n1 : c1;
    cz = a2 ? n2 : c2;
    w.t = t;
    w.face = a0 ? 4 + (int32_t)(r.posmask & 1u)
                : (a1 ? 2 + (int32_t)((r.posmask >> 1) & 1u) : (int32_t)((r.posmask >> 2) & 1u));
    bool on = t < t_lim;
    if (!on) {
      const bool out0 = (uint32_t)(cx - s.lo[0]) >= (uint32_t)(s.hi[0] - s.lo[0]);
      const bool out1 = (uint32_t)(cy - s.lo[1]) >= (uint32_t)(s.hi[1] - s.lo[1]);
      const bool out2 = (uint32_t)(cz - s.lo[2]) >= (uint32_t)(s.hi[2] - s.lo[2]);
      on = (t < tmax) & !((a0 & out0) | (a1 & out1) | (a2 & out2));
    }
    if (!on) break;
    dv = (x ^ (uint32_t)cx) | (y ^ (uint32_t)cy) | (z ^ (uint32_t)cz);
  }
  if (!hit) return false;
  w.cell[0] = cx, w.cell[1] = cy, w.cell[2] = cz;
  material = s.voxels[(uint64_t)slot * 512u + ((uint32_t)cx & 7u) + 8u * ((uint32_t)cy & 7u) +
                      64u * ((uint32_t)cz & 7u)];
  return true;
}

// Walk until a solid voxel is entered (true), the ray leaves the scene or the
// entry t reaches tmax (false).
// EMPTY: the start cell of a dense grid is known to be empty.
template <int KIND, bool COUNT, bool EMPTY = false>
__device__ __forceinline__ bool walk(const DevScene &s, const Ray &r, WalkState &w, float tmax,
                                     uint16_t &material, StepCounts &cnt) {
  if (!(w.t < tmax)) return false;
  if constexpr ((KIND == 1 || KIND == kDenseShort) && !COUNT) {
    constexpr int ahead = KIND == 1 ? kDenseAhead : kDenseAheadShort;
    DenseRay e;
    if (e.setup(s, r)) return walk_dense<kDenseSingle, ahead, EMPTY>(s, r, e, w, tmax, material);
  }
  if constexpr ((KIND == 2 || KIND == 3) && !COUNT) return walk_bricks<KIND>(s, r, w, tmax, material);
  WalkCache c;
  c.reset();
  for (;;) {
    const int st = walk_step<KIND, COUNT>(s, r, w, c, tmax, material, cnt);
    if (st != kWalkOn) return st == kWalkHit;
  }
}

// A dense ray walked in parts of its stretch of t, one by each of kDenseParts lanes.
constexpr int kDenseParts = 4;

// The part's start on a ray that walk_dense() takes: the cell after every plane
// with a t below `from` has been crossed, which is where the walk from w.cell
// would be then.  A plane at t is within 2^-5 of the ray's point at t, so the
// first plane with a t of at least `from` is one of four.
__device__ __forceinline__ void dense_skip(const Ray &r, WalkState &w, float from) {
#pragma unroll
  for (int a = 0; a < 3; a++) {
    if (r.step[a] == 0) continue;
    const float s = (float)r.step[a], first = (float)(w.cell[a] + r.pos[a]);
    const float dt = r.d[a] * from;
    const float mid = __builtin_rintf(r.o[a] + dt);
    float p = mid + 2.0f * s;
#pragma unroll
    for (int k = 1; k >= -1; k--) {
      const float c = mid + (float)k * s;
      p = plane_t(r.o[a], r.inv[a], c) >= from ? c : p;
    }
    p = (p - first) * s > 0.0f ? p : first;
    w.cell[a] = (int32_t)p - r.pos[a];
  }
}

// What the lane of a part walks of a ray that walk_dense() takes: its start in
// w and the t it ends at in tmax; false when that is nothing.
// The stretch may be empty or run backwards: the origin of a shadow ray is a
// hit point, which rounding can leave beyond the very side of the grid that
// the ray leaves by (t_out < 0), the more the farther the eye.  walk() then
// reads the start cell and ends, and so does the first lane; a part's `from`
// would lie past t_out, and its start cell past the grid.
__device__ __forceinline__ bool dense_part(const DevScene &s, const Ray &r, const DenseRay &e,
                                           WalkState &w, float &tmax, uint32_t part) {
  const float t_lim = tmax < e.t_out ? tmax : e.t_out;
  const float step = (t_lim - w.t) * (1.0f / kDenseParts);
  if (!(step > 0.0f)) return part == 0u;
  const float from = w.t + step * (float)part;  // at most t_lim: 3/4 of the stretch, rounded
  if (part + 1u < (uint32_t)kDenseParts) {
    const float to = w.t + step * (float)(part + 1u);
    tmax = to < tmax ? to : tmax;
  }
  if (part > 0u) dense_skip(r, w, from);
  // only planes with a t below t_out were crossed, so the cell is in the grid;
  // walk_dense() reads it without a test, so it is tested here
  bool in = true;
#pragma unroll
  for (int a = 0; a < 3; a++) in = in && (uint32_t)w.cell[a] < (uint32_t)s.n;
  return in;
}

// walk() by the four lanes of a pixel: true in the first of those that hit and
// perhaps in others.  The first kDenseTogether cells are looked at by all four,
// and most rays of solid or rough scenes end there.  A start cell of a part
// that is solid was the last cell of the part before, whose lane then has it.
constexpr int kDenseTogether = 8;
__device__ __forceinline__ bool walk_part(const DevScene &s, const Ray &r, WalkState &w, float tmax,
                                          uint32_t part, uint16_t &material) {
  if (!(w.t < tmax)) return false;
  DenseRay e;
  if (!e.setup(s, r)) {
    StepCounts cnt;
    return part == 0u && walk<1, false>(s, r, w, tmax, material, cnt);
  }
  DenseWalk d(s, r, e, w, tmax);
  if (!d.batch<kDenseTogether>(w)) return d.finish(w, material);
#pragma unroll
  for (int a = 0; a < 3; a++) w.cell[a] = d.cell(a);
  return dense_part(s, r, e, w, tmax, part) && walk_dense<0, kDenseAhead, false>(s, r, e, w, tmax, material);
}

__device__ __forceinline__ void primary_ray(const DevCamera &c, int32_t px, int32_t py, float o[3],
                                            float d[3]) {
  float a = (float)px + 0.5f;
  a = a * c.inv_w2;
  a = a - 1.0f;
  a = a * c.sx;
  float b = (float)py + 0.5f;
  b = b * c.inv_h2;
  b = 1.0f - b;
  b = b * c.sy;
  float v[3];
#pragma unroll
  for (int i = 0; i < 3; i++) {
    float ra = c.right[i] * a;
    float ub = c.up[i] * b;
    v[i] = c.fwd[i] + ra;
    v[i] = v[i] + ub;
    o[i] = c.eye[i];
  }
  float xx = v[0] * v[0], yy = v[1] * v[1], zz = v[2] * v[2];
  float s = xx + yy;
  s = s + zz;
  float len = __builtin_sqrtf(s);
#pragma unroll
  for (int i = 0; i < 3; i++) d[i] = v[i] / len;
}

struct Hit {
  int64_t index;
  int32_t face;
  float t;
  int32_t cell[3];
  uint16_t material;
};

// Set up the ray o + t d, clip it to the scene's solid box [lo, hi) and find
// its entry cell; false when it misses the box.
__device__ __forceinline__ bool trace_begin(const DevScene &s, const float o[3], const float d[3],
                                            Ray &r, WalkState &w) {
  ray_setup(r, o, d);
  float t_enter = 0.0f, t_exit = __builtin_inff();
  int ea = -1;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    if (s.lo[a] >= s.hi[a]) return false;  // nothing solid
    const float bl = s.flo[a], bh = s.fhi[a];
    if (r.step[a] == 0) {
      if (o[a] < bl || o[a] >= bh) return false;
      continue;
    }
    float lo = plane_t(r.o[a], r.inv[a], r.step[a] > 0 ? bl : bh);
    float hi = plane_t(r.o[a], r.inv[a], r.step[a] > 0 ? bh : bl);
    if (lo > t_enter) {
      t_enter = lo;
      ea = a;
    }
    if (hi < t_exit) t_exit = hi;
  }
  if (t_enter > t_exit) return false;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    if (a == ea) {
      w.cell[a] = r.step[a] > 0 ? s.lo[a] : s.hi[a] - 1;
    } else {
      float dt = d[a] * t_enter;
      float p = o[a] + dt;
      int32_t c = (int32_t)__builtin_floorf(p);
      c = c < s.lo[a] ? s.lo[a] : c;
      c = c > s.hi[a] - 1 ? s.hi[a] - 1 : c;
      w.cell[a] = c;
    }
  }
  w.t = t_enter;
  int est = 0;
#pragma unroll
  for (int a = 0; a < 3; a++)
    if (a == ea) est = r.step[a];
  w.face = ea >= 0 ? entry_face(ea, est) : kFaceInside;
  return true;
}

// The cell a primary ray of a dense grid enters first, looked at before the walk
// is set up: all there is to do where the grid's sides are solid or the eye is
// (see kDenseSingle).
__device__ __forceinline__ uint16_t dense_start(const DevScene &s, const WalkState &w) {
  return w.t < __builtin_inff() ? s.dense[lin3(w.cell[0], w.cell[1], w.cell[2], s.n)] : 0;
}

// Clip to [0,n]^3, find the entry cell and walk.
template <int KIND, bool COUNT>
__device__ __forceinline__ bool trace(const DevScene &s, const float o[3], const float d[3],
                                      Hit &hit, StepCounts &cnt) {
  hit.index = -1;
  hit.face = kFaceMiss;
  hit.t = __builtin_inff();
  hit.material = 0;
  Ray r;
  WalkState w;
  if (!trace_begin(s, o, d, r, w)) return false;
  const int32_t n = s.n;
  uint16_t m = 0;
  constexpr bool first = (KIND == 1 || KIND == kDenseShort) && !COUNT;
  if constexpr (first) m = dense_start(s, w);
  if (m == 0 && !walk<KIND, COUNT, first>(s, r, w, __builtin_inff(), m, cnt)) return false;
  hit.index = lin3(w.cell[0], w.cell[1], w.cell[2], n);
  hit.face = w.face;
  hit.t = w.t;
  hit.cell[0] = w.cell[0];
  hit.cell[1] = w.cell[1];
  hit.cell[2] = w.cell[2];
  hit.material = m;
  return true;
}

// true when a secondary ray can start in cell `start` (inside the scene's
// solid box).  A start outside it is the neighbour across a face of a voxel
// on the box's side, and the ray travels into that face's half-space, away
// from the box, so it is unoccluded.
__device__ __forceinline__ bool start_inside(const DevScene &s, const int32_t start[3]) {
  return start[0] >= s.lo[0] && start[0] < s.hi[0] && start[1] >= s.lo[1] && start[1] < s.hi[1] &&
         start[2] >= s.lo[2] && start[2] < s.hi[2];
}

// A secondary ray o + t d that walks from cell `start` at t = 0.
__device__ __forceinline__ void occluded_begin(const float o[3], const float d[3],
                                               const int32_t start[3], Ray &r, WalkState &w) {
  ray_setup(r, o, d);
  w.cell[0] = start[0];
  w.cell[1] = start[1];
  w.cell[2] = start[2];
  w.t = 0.0f;
  w.face = kFaceInside;
#pragma unroll
  for (int a = 0; a < 3; a++)
    r.up[a] = r.step[a] > 0 || (r.step[a] == 0 && (int32_t)__builtin_floorf(o[a]) > start[a]);
}

template <int KIND, bool COUNT>
__device__ __forceinline__ bool occluded(const DevScene &s, const float o[3], const float d[3],
                                         const int32_t start[3], float tmax, StepCounts &cnt) {
  if (!start_inside(s, start)) return false;
  Ray r;
  WalkState w;
  occluded_begin(o, d, start, r, w);
  uint16_t m;
  return walk<KIND, COUNT>(s, r, w, tmax, m, cnt);
}

// lowbias32 integer finaliser (C. Wellons, hash-prospector)
__device__ __forceinline__ uint32_t hash32(uint32_t x) {
  x ^= x >> 16;
  x *= 0x7feb352du;
  x ^= x >> 15;
  x *= 0x846ca68bu;
  x ^= x >> 16;
  return x;
}

// Cosine-weighted hemisphere direction about the face normal (Malley's
// method): a point uniform in the unit disk, found by rejection from
// counter-based hashes, lifted by z = sqrt(1 - r^2).
__device__ __forceinline__ void ao_direction(uint32_t seed, uint32_t pixel, uint32_t sample,
                                             int face, float dir[3]) {
  float a, b, r2;
  const uint32_t base = hash32(hash32(seed) ^ pixel);
  uint32_t k = 0;
  // one try a trip: the compiler made four at a time of the loop, with eight
  // quarter-rate multiplies, which cost more than the 3.6 trips that the
  // unluckiest lane of a wave needs on average (3840x2160 caves with four AO
  // rays 1672 us, now 1635)
#pragma clang loop vectorize(disable) interleave(disable) unroll(disable)
  do {
    uint32_t h = hash32(base ^ (sample * 16u + k));
    a = (float)(h & 0xFFFFu) * (1.0f / 32768.0f);
    a = a - 1.0f;
    b = (float)(h >> 16) * (1.0f / 32768.0f);
    b = b - 1.0f;
    float aa = a * a, bb = b * b;
    r2 = aa + bb;
    k++;
  } while (r2 >= 1.0f && k < 16u);
  if (r2 >= 1.0f) {
    a = 0.0f;
    b = 0.0f;
    r2 = 0.0f;
  }
  float z = __builtin_sqrtf(1.0f - r2);
  const int na = face_axis(face);
  const bool pos = (face & 1) == 0;
#pragma unroll
  for (int k = 0; k < 3; k++) {
    const int ua = na == 0 ? 1 : 0;
    const int va = na == 2 ? 1 : 2;
    if (k == na) dir[k] = pos ? z : -z;
    else if (k == ua) dir[k] = a;
    else if (k == va) dir[k] = b;
  }
}

struct PixelResult {
  int64_t index;
  int32_t face;
  float t;
  float shade;
};

// Where the secondary rays of a primary hit start: the hit point p = o + t d
// on entry face `face` (< 6) of voxel `cell`, the cell in front of that face,
// and the face's Lambert term max(0, n . light).
struct Secondary {
  float p[3];
  int32_t start[3];
  float lambert;
};

__device__ __forceinline__ void secondary_setup(const DevShading &sh, const float o[3],
                                                const float d[3], int32_t face, float t,
                                                const int32_t cell[3], Secondary &sc) {
  const int na = face_axis(face);
  const int sg = (face & 1) ? -1 : 1;
  float lightc = sh.light[0];
  sc.start[0] = cell[0];
  sc.start[1] = cell[1];
  sc.start[2] = cell[2];
#pragma unroll
  for (int k = 0; k < 3; k++)
    if (k == na) {
      lightc = sh.light[k];
      sc.start[k] += sg;
    }
  float lambert = sg > 0 ? lightc : -lightc;
  if (lambert < 0.0f) lambert = 0.0f;
  sc.lambert = lambert;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    float dt = d[i] * t;
    sc.p[i] = o[i] + dt;
  }
}

// (0.25 + 0.75 * lambert * visible) * (0.5 + 0.5 * unoccluded / samples),
// the second factor only with AO rays
__device__ __forceinline__ float shade_value(float lambert, float vis, bool ao_on, int32_t unocc,
                                             int32_t samples) {
  float ao = 1.0f;
  if (ao_on) {
    float frac = (float)unocc / (float)samples;
    frac = 0.5f * frac;
    ao = 0.5f + frac;
  }
  float l = lambert * vis;
  l = 0.75f * l;
  float shade = 0.25f + l;
  shade = shade * ao;
  return shade;
}

// The secondary rays of pixel `pix` whose primary ray hit face `face` (< 6),
// set up by secondary_setup: the shadow ray toward the light when the face is
// lit, the AO rays, and the shade.  With neither flag set it traces nothing.
template <int KIND, bool COUNT>
__device__ __forceinline__ float shade_secondary(const DevScene &s, uint32_t flags,
                                                 const DevShading &sh, uint32_t pix, int32_t face,
                                                 const Secondary &sc, StepCounts &cnt,
                                                 uint32_t &n_shadow, uint32_t &n_ao) {
  float vis = 1.0f;
  if ((flags & MESO_RAY_SHADOW) && sc.lambert > 0.0f) {
    n_shadow++;
    if (occluded<KIND, COUNT>(s, sc.p, sh.light, sc.start, __builtin_inff(), cnt)) vis = 0.0f;
  }
  int32_t unocc = 0;
  if (flags & MESO_RAY_AO) {
    for (int32_t k = 0; k < sh.ao_samples; k++) {
      float dir[3];
      ao_direction(sh.ao_seed, pix, (uint32_t)k, face, dir);
      n_ao++;
      if (!occluded<KIND, COUNT>(s, sc.p, dir, sc.start, sh.ao_radius, cnt)) unocc++;
    }
  }
  return shade_value(sc.lambert, vis, (flags & MESO_RAY_AO) != 0, unocc, sh.ao_samples);
}

// Secondary rays of a primary hit (voxel `cell`, entry face `face` < 6, at t
// along o + t d) and the shade.
template <int KIND, bool COUNT>
__device__ __forceinline__ float shade_hit(const DevScene &s, uint32_t flags, const DevShading &sh,
                                           uint32_t pix, const float o[3], const float d[3],
                                           int32_t face, float t, const int32_t cell[3],
                                           StepCounts &cnt, uint32_t &n_shadow, uint32_t &n_ao) {
  Secondary sc;
  secondary_setup(sh, o, d, face, t, cell, sc);
  return shade_secondary<KIND, COUNT>(s, flags, sh, pix, face, sc, cnt, n_shadow, n_ao);
}

// true when a primary hit on `face` needs secondary rays
__device__ __forceinline__ bool needs_secondary(uint32_t flags, const DevShading &sh, int32_t face) {
  if (face >= 6) return false;
  if (flags & MESO_RAY_AO) return true;
  if (!(flags & MESO_RAY_SHADOW)) return false;
  const int na = face_axis(face);
  const float lightc = na == 0 ? sh.light[0] : (na == 1 ? sh.light[1] : sh.light[2]);
  const float lambert = (face & 1) ? -lightc : lightc;
  return lambert > 0.0f;
}

// Primary ray of pixel (px,py), then its secondary rays and shade.
template <int KIND, bool COUNT>
__device__ __forceinline__ PixelResult shade_pixel(const DevScene &s, const DevCamera &cam,
                                                   uint32_t flags, const DevShading &sh,
                                                   int32_t px, int32_t py, StepCounts &cnt,
                                                   uint32_t &n_shadow, uint32_t &n_ao) {
  float o[3], d[3];
  primary_ray(cam, px, py, o, d);
  Hit h;
  PixelResult res;
  const bool hit = trace<KIND, COUNT>(s, o, d, h, cnt);
  float shade = 0.0f;
  if (hit) {
    if (h.face < 6)
      shade = shade_hit<KIND, COUNT>(s, flags, sh, (uint32_t)((int64_t)py * cam.width + px), o, d,
                                     h.face, h.t, h.cell, cnt, n_shadow, n_ao);
    else
      shade = 0.25f;
  }
  res.index = h.index;
  res.face = h.face;
  res.t = h.t;
  res.shade = shade;
  return res;
}

}  // namespace meso
