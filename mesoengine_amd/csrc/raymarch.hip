// Raymarch kernels: one lane per pixel, wave64 packets of 8x8 pixels so the
// rays of a wave fetch the same bricks (small dense frames: four lanes per
// pixel).  Tiled variants hand rows of tiles to the XCDs in turn; the
// persistent variant keeps every wave slot busy and pulls packets from
// per-band queues.
#include "traverse.h"

namespace meso {

// Hardware hands workgroup i to XCD i % 8.  XCD x takes every 8th group of
// `group` consecutive tiles, so neighbouring tiles share that XCD's L2 and all
// XCDs work all over the frame.  (A contiguous eighth of the frame each left
// the XCDs that had sky waiting for those that had ground: the slowest eighth
// bounded the frame.  1920x1080 rolling hills with shadows: 253 us, now 179
// with the same 16x16 tiles; 1800x1350 spheres with AO 396 us, now 232.)
__device__ __forceinline__ uint32_t xcd_remap(uint32_t bid, uint32_t group) {
  const uint32_t xcd = bid % 8u, local = bid / 8u, g = local / group;
  return (g * 8u + xcd) * group + (local - g * group);
}

template <int KIND, bool COUNT, int TW, int TH>
__global__ void __launch_bounds__(TW *TH) raymarch_kernel(DevScene s, DevCamera cam, uint32_t flags,
                                                          DevShading sh, RayOut out,
                                                          uint32_t tiles_x, uint32_t n_tiles,
                                                          uint32_t group) {
  // tile of TW x TH pixels made of 8x8 wave packets
  const uint32_t tile = xcd_remap(blockIdx.x, group);
  if (tile >= n_tiles) return;  // uniform: the last groups of some XCDs
  const uint32_t tx = tile % tiles_x, ty = tile / tiles_x;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  constexpr uint32_t waves_x = TW / 8;
  const int32_t px = (int32_t)(tx * TW + (wave % waves_x) * 8u + (lane & 7u));
  const int32_t py = (int32_t)(ty * TH + (wave / waves_x) * 8u + (lane >> 3));

  StepCounts cnt = {0, 0, 0, 0, 0, 0, 0};
  uint32_t n_shadow = 0, n_ao = 0;
  bool valid = px < cam.width && py < cam.height;
  PixelResult r{-1, kFaceMiss, 0.0f, 0.0f};
  if (valid) {
    r = shade_pixel<KIND, COUNT>(s, cam, flags, sh, px, py, cnt, n_shadow, n_ao);
    const int64_t pix = (int64_t)py * cam.width + px;
    if (out.index_bytes == 8)
      ((int64_t *)out.index)[pix] = r.index;
    else
      ((int32_t *)out.index)[pix] = (int32_t)r.index;
    if (out.face) out.face[pix] = (uint8_t)r.face;
    if (out.t) out.t[pix] = r.t;
    if (out.shade) out.shade[pix] = r.shade;
  }
  if constexpr (COUNT) {
    __shared__ unsigned long long acc[MESO_CNT_COUNT];
    if (threadIdx.x < MESO_CNT_COUNT) acc[threadIdx.x] = 0;
    __syncthreads();
    if (valid) {
      atomicAdd(&acc[MESO_CNT_N_VOX], (unsigned long long)cnt.n_vox);
      atomicAdd(&acc[MESO_CNT_N_TOP], (unsigned long long)cnt.n_top);
      atomicAdd(&acc[MESO_CNT_N_NODE], (unsigned long long)cnt.n_node);
      atomicAdd(&acc[MESO_CNT_N_BRICKSLOT], (unsigned long long)cnt.n_brickslot);
      atomicAdd(&acc[MESO_CNT_N_BRICKMASK], (unsigned long long)cnt.n_brickmask);
      atomicAdd(&acc[MESO_CNT_HITS], (unsigned long long)(r.index >= 0 ? 1 : 0));
      atomicAdd(&acc[MESO_CNT_RAYS], 1ull);
      atomicAdd(&acc[MESO_CNT_SHADOW_RAYS], (unsigned long long)n_shadow);
      atomicAdd(&acc[MESO_CNT_AO_RAYS], (unsigned long long)n_ao);
      atomicAdd(&acc[MESO_CNT_N_COARSE], (unsigned long long)cnt.n_coarse);
      atomicAdd(&acc[MESO_CNT_N_ITER], (unsigned long long)cnt.n_iter);
    }
    __syncthreads();
    if (threadIdx.x < MESO_CNT_COUNT && out.counters)
      atomicAdd(&out.counters[threadIdx.x], acc[threadIdx.x]);
  }
}

// Dense grid, small frames: four lanes per pixel.  A frame of few waves takes as
// long as its longest ray, a few hundred steps of one wave with a SIMD to
// itself.  Here a ray's stretch of t is cut into four, and each lane walks one
// of them; the first lane of the four that hits has the hit.  AO rays, which are
// short, are dealt out instead, one sample in four to a lane.  The rays' set-up
// is done four times.  256^3 voxels of spheres with shadows, a long view, a lane
// a ray and four: 200x200 119 and 52 us, 256x256 122 and 95, 400x225 121 and 51.
//
// The most 8x8 waves per SIMD of a frame that goes this way.  400x225, 1.4 a
// SIMD, gains as above and takes 5.8 us instead of 3.9 where all is solid; 512x512,
// 4 a SIMD, takes 124 instead of 119, and 11 instead of 4.8 where all is solid.
constexpr uint32_t kSmallWaves = 2;

__global__ void __launch_bounds__(64) raymarch_dense_small_kernel(DevScene s, DevCamera cam,
                                                                  uint32_t flags, DevShading sh,
                                                                  RayOut out, uint32_t tiles_x) {
  const uint32_t lane = threadIdx.x, part = lane & 3u, quad = lane & ~3u;
  // 4x4 pixels, by workgroup
  const int32_t px = (int32_t)((blockIdx.x % tiles_x) * 4u + ((lane >> 2) & 3u));
  const int32_t py = (int32_t)((blockIdx.x / tiles_x) * 4u + (lane >> 4));
  const bool valid = px < cam.width && py < cam.height;
  float o[3], d[3];
  primary_ray(cam, px, py, o, d);
  Ray r;
  WalkState w = {{0, 0, 0}, 0.0f, 0};
  uint16_t m = 0;
  bool hit = false;
  if (valid && trace_begin(s, o, d, r, w)) {
    m = dense_start(s, w);
    hit = m ? part == 0u : walk_part(s, r, w, __builtin_inff(), part, m);
  }
  // the first of the pixel's lanes that hit, in every lane of the pixel
  const uint32_t hits = (uint32_t)(__ballot(hit) >> quad) & 15u;
  const int src = (int)(quad + (hits ? (uint32_t)__builtin_ctz(hits) : 0u));
  const float t = __shfl(w.t, src, 64);
  const int32_t face = __shfl(w.face, src, 64);
  int32_t cell[3];
#pragma unroll
  for (int a = 0; a < 3; a++) cell[a] = __shfl(w.cell[a], src, 64);
  float shade = 0.0f;
  if (hits) {
    shade = 0.25f;
    if (face < 6) {
      Secondary sc;
      secondary_setup(sh, o, d, face, t, cell, sc);
      float vis = 1.0f;
      if ((flags & MESO_RAY_SHADOW) && sc.lambert > 0.0f) {
        bool dark = false;
        if (start_inside(s, sc.start)) {
          Ray q;
          WalkState v;
          occluded_begin(sc.p, sh.light, sc.start, q, v);
          uint16_t sm;
          dark = walk_part(s, q, v, __builtin_inff(), part, sm);
        }
        if ((__ballot(dark) >> quad) & 15ull) vis = 0.0f;
      }
      int32_t unocc = 0;
      if (flags & MESO_RAY_AO) {
        StepCounts cnt;
        const uint32_t pix = (uint32_t)((int64_t)py * cam.width + px);
        for (int32_t k = (int32_t)part; k < sh.ao_samples; k += kDenseParts) {
          float dir[3];
          ao_direction(sh.ao_seed, pix, (uint32_t)k, face, dir);
          if (!occluded<1, false>(s, sc.p, dir, sc.start, sh.ao_radius, cnt)) unocc++;
        }
        unocc += __shfl_xor(unocc, 1, 64);
        unocc += __shfl_xor(unocc, 2, 64);
      }
      shade = shade_value(sc.lambert, vis, (flags & MESO_RAY_AO) != 0, unocc, sh.ao_samples);
    }
  }
  if (valid && part == 0u) {
    const int64_t pix = (int64_t)py * cam.width + px;
    const int64_t index = hits ? lin3(cell[0], cell[1], cell[2], s.n) : -1;
    if (out.index_bytes == 8)
      ((int64_t *)out.index)[pix] = index;
    else
      ((int32_t *)out.index)[pix] = (int32_t)index;
    if (out.face) out.face[pix] = (uint8_t)(hits ? face : kFaceMiss);
    if (out.t) out.t[pix] = hits ? t : __builtin_inff();
    if (out.shade) out.shade[pix] = shade;
  }
}

// End of a persistent wave: add its counters, then leave.  The band counters
// persist per stream: the last wave to leave (queue[128] counts leavers) sets
// them back to zero, after every wave's last counter access has returned,
// for the next launch.
template <bool COUNT>
__device__ __forceinline__ void persistent_leave(const RayOut &out, unsigned int *queue,
                                                 const StepCounts &cnt, uint32_t n_hits,
                                                 uint32_t n_rays, uint32_t n_shadow,
                                                 uint32_t n_ao) {
  const uint32_t lane = threadIdx.x;
  if constexpr (COUNT) {
    unsigned long long v[MESO_CNT_COUNT] = {cnt.n_vox, cnt.n_top, cnt.n_node, cnt.n_brickslot,
                                            cnt.n_brickmask, n_hits, n_rays, n_shadow, n_ao,
                                            cnt.n_coarse, cnt.n_iter};
#pragma unroll
    for (int c = 0; c < MESO_CNT_COUNT; c++) {
      unsigned long long x = v[c];
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
      if (lane == 0 && out.counters && x) atomicAdd(&out.counters[c], x);
    }
  }
  if (lane == 0 && atomicAdd(&queue[128], 1u) == gridDim.x - 1u) {
#pragma unroll
    for (uint32_t b = 0; b < 8u; b++)
      __hip_atomic_store(&queue[b * 16u], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(&queue[128], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Persistent waves: one 64-lane workgroup per wave slot of the device.  The
// screen's PW x (64 / PW) packets (8x8, 16x4 or 32x2) are cut into 8 bands
// of rows; the waves of XCD x
// (workgroup i runs on XCD i % 8) take packets of band x from that band's
// counter, then help the other bands in turn.  A wave leaves once every
// counter has passed the end of its band, so the grid always drains; slots
// freed by short (sky) packets are refilled at once instead of waiting for
// the next workgroup dispatch.
template <int KIND, bool COUNT, int PW>
__global__ void __launch_bounds__(64) raymarch_persistent_kernel(
    DevScene s, DevCamera cam, uint32_t flags, DevShading sh, RayOut out, uint32_t packets_x,
    uint32_t n_packets, unsigned int *queue) {
  constexpr uint32_t PH = 64 / PW;  // packet of PW x PH pixels
  const uint32_t lane = threadIdx.x;
  const uint32_t home = blockIdx.x & 7u;
  StepCounts cnt = {0, 0, 0, 0, 0, 0, 0};
  uint32_t n_shadow = 0, n_ao = 0, n_hits = 0, n_rays = 0;
  for (uint32_t k = 0; k < 8u; k++) {
    const uint32_t band = (home + k) & 7u;
    const uint32_t lo = (uint32_t)(((uint64_t)n_packets * band) >> 3);
    const uint32_t hi = (uint32_t)(((uint64_t)n_packets * (band + 1u)) >> 3);
    for (;;) {
      uint32_t p = 0;
      if (lane == 0) p = atomicAdd(&queue[band * 16u], 1u);  // one counter per 64 B line
      p = lo + (uint32_t)__shfl((int)p, 0, 64);
      if (p >= hi) break;  // uniform over the wave
      const int32_t px = (int32_t)((p % packets_x) * (uint32_t)PW + lane % (uint32_t)PW);
      const int32_t py = (int32_t)((p / packets_x) * PH + lane / (uint32_t)PW);
      if (px < cam.width && py < cam.height) {
        const PixelResult r = shade_pixel<KIND, COUNT>(s, cam, flags, sh, px, py, cnt, n_shadow, n_ao);
        const int64_t pix = (int64_t)py * cam.width + px;
        if (out.index_bytes == 8)
          ((int64_t *)out.index)[pix] = r.index;
        else
          ((int32_t *)out.index)[pix] = (int32_t)r.index;
        if (out.face) out.face[pix] = (uint8_t)r.face;
        if (out.t) out.t[pix] = r.t;
        if (out.shade) out.shade[pix] = r.shade;
        n_hits += r.index >= 0 ? 1u : 0u;
        n_rays++;
      }
    }
  }
  persistent_leave<COUNT>(out, queue, cnt, n_hits, n_rays, n_shadow, n_ao);
}


// j-th (0-based) set bit of a 64-bit mask that has more than j set bits
__device__ __forceinline__ uint32_t select_bit64(uint64_t m, uint32_t j) {
  uint32_t pos = 0;
#pragma unroll
  for (uint32_t w = 32; w >= 1; w >>= 1) {
    const uint32_t c = (uint32_t)__popcll(m & ((1ull << w) - 1ull));
    if (j >= c) {
      j -= c;
      m >>= w;
      pos += w;
    }
  }
  return pos;
}

// A pixel's primary ray: writes index, face and t; returns true (and fills
// sc and face) when the pixel needs secondary rays, else writes the shade.
template <int KIND, bool COUNT>
__device__ __forceinline__ bool primary_pixel(const DevScene &s, const DevCamera &cam,
                                              uint32_t flags, const DevShading &sh, int32_t px,
                                              int32_t py, const RayOut &out, StepCounts &cnt,
                                              uint32_t &n_hits, Secondary &sc, int32_t &face) {
  float o[3], d[3];
  primary_ray(cam, px, py, o, d);
  Hit h;
  const bool hit = trace<KIND, COUNT>(s, o, d, h, cnt);
  const int64_t pix = (int64_t)py * cam.width + px;
  if (out.index_bytes == 8)
    ((int64_t *)out.index)[pix] = h.index;
  else
    ((int32_t *)out.index)[pix] = (int32_t)h.index;
  if (out.face) out.face[pix] = (uint8_t)h.face;
  if (out.t) out.t[pix] = h.t;
  n_hits += h.index >= 0 ? 1u : 0u;
  face = h.face;
  if (hit && h.face < 6) {
    secondary_setup(sh, o, d, h.face, h.t, h.cell, sc);
    if (needs_secondary(flags, sh, h.face)) return true;
    if (out.shade) out.shade[pix] = shade_value(sc.lambert, 1.0f, false, 0, sh.ao_samples);
    return false;
  }
  if (out.shade) out.shade[pix] = hit ? 0.25f : 0.0f;
  return false;
}

// Persistent waves over pairs of packets (variants 8 and 9).  The wave traces
// the primary rays of two packets, then shares out the pixels of both that
// need secondary rays (shadow, AO) over its 64 lanes, so that the secondary
// phase runs with up to twice the busy lanes of one packet.  A pixel's
// secondary state (hit point, start cell, Lambert term, face, pixel) moves to
// the lane that traces it by lane shuffles.  Every ray computes what
// shade_pixel computes, so the outputs are the same bits.  It holds more
// registers than the one-packet waves (5 waves/SIMD against 7), and pays off
// when issue, not latency, bounds the frame (for example with two frames in
// flight on the 1080p heightfield).
template <int KIND, bool COUNT, int PW>
__global__ void __launch_bounds__(64) raymarch_pair_kernel(
    DevScene s, DevCamera cam, uint32_t flags, DevShading sh, RayOut out, uint32_t packets_x,
    uint32_t n_packets, unsigned int *queue) {
  constexpr uint32_t PH = 64 / PW;
  const uint32_t lane = threadIdx.x;
  const uint32_t home = blockIdx.x & 7u;
  StepCounts cnt = {0, 0, 0, 0, 0, 0, 0};
  uint32_t n_shadow = 0, n_ao = 0, n_hits = 0, n_rays = 0;
  for (uint32_t k = 0; k < 8u; k++) {
    const uint32_t band = (home + k) & 7u;
    const uint32_t lo = (uint32_t)(((uint64_t)n_packets * band) >> 3);
    const uint32_t hi = (uint32_t)(((uint64_t)n_packets * (band + 1u)) >> 3);
    for (;;) {
      uint32_t p = 0;
      if (lane == 0) p = atomicAdd(&queue[band * 16u], 2u);  // two packets at a time
      p = lo + (uint32_t)__shfl((int)p, 0, 64);
      if (p >= hi) break;  // uniform over the wave
      Secondary sa = {{0.0f, 0.0f, 0.0f}, {0, 0, 0}, 0.0f}, sb = sa;
      int32_t fa = 0, fb = 0;
      uint32_t pa = 0, pb = 0;
      bool na = false, nb = false;
      {
        const int32_t px = (int32_t)((p % packets_x) * (uint32_t)PW + lane % (uint32_t)PW);
        const int32_t py = (int32_t)((p / packets_x) * PH + lane / (uint32_t)PW);
        if (px < cam.width && py < cam.height) {
          n_rays++;
          pa = (uint32_t)((int64_t)py * cam.width + px);
          na = primary_pixel<KIND, COUNT>(s, cam, flags, sh, px, py, out, cnt, n_hits, sa, fa);
        }
      }
      if (p + 1u < hi) {  // uniform
        const uint32_t q = p + 1u;
        const int32_t px = (int32_t)((q % packets_x) * (uint32_t)PW + lane % (uint32_t)PW);
        const int32_t py = (int32_t)((q / packets_x) * PH + lane / (uint32_t)PW);
        if (px < cam.width && py < cam.height) {
          n_rays++;
          pb = (uint32_t)((int64_t)py * cam.width + px);
          nb = primary_pixel<KIND, COUNT>(s, cam, flags, sh, px, py, out, cnt, n_hits, sb, fb);
        }
      }
      const uint64_t ma = __ballot(na), mb = __ballot(nb);
      const uint32_t ca = (uint32_t)__popcll(ma), total = ca + (uint32_t)__popcll(mb);
      for (uint32_t base = 0; base < total; base += 64u) {  // uniform
        const uint32_t j = base + lane;
        const bool from_a = j < ca;
        const uint32_t src = j < total ? (from_a ? select_bit64(ma, j) : select_bit64(mb, j - ca))
                                       : lane;
        // every lane takes part in every shuffle; the lane keeps A's or B's copy
        Secondary sc;
#pragma unroll
        for (int i = 0; i < 3; i++) {
          const float xa = __shfl(sa.p[i], (int)src, 64), xb = __shfl(sb.p[i], (int)src, 64);
          sc.p[i] = from_a ? xa : xb;
          const int32_t ia = __shfl(sa.start[i], (int)src, 64), ib = __shfl(sb.start[i], (int)src, 64);
          sc.start[i] = from_a ? ia : ib;
        }
        const float la = __shfl(sa.lambert, (int)src, 64), lb = __shfl(sb.lambert, (int)src, 64);
        sc.lambert = from_a ? la : lb;
        const int32_t ga = __shfl(fa, (int)src, 64), gb = __shfl(fb, (int)src, 64);
        const uint32_t qa = (uint32_t)__shfl((int)pa, (int)src, 64), qb = (uint32_t)__shfl((int)pb, (int)src, 64);
        const int32_t face = from_a ? ga : gb;
        const uint32_t pix = from_a ? qa : qb;
        if (j < total) {
          const float shade = shade_secondary<KIND, COUNT>(s, flags, sh, pix, face, sc, cnt,
                                                           n_shadow, n_ao);
          if (out.shade) out.shade[pix] = shade;
        }
      }
    }
  }
  persistent_leave<COUNT>(out, queue, cnt, n_hits, n_rays, n_shadow, n_ao);
}

template <int KIND, bool COUNT, int PW>
static meso_status launch_pair(meso_context *ctx, const meso_scene *scene, const DevCamera &cam,
                               uint32_t flags, const DevShading &sh, const RayOut &out,
                               hipStream_t stream, int grid) {
  constexpr int PH = 64 / PW;
  const uint32_t packets_x = (uint32_t)((cam.width + PW - 1) / PW);
  const uint32_t n_packets = packets_x * (uint32_t)((cam.height + PH - 1) / PH);
  if (grid <= 0) {
    int per_cu = 0;
    MESO_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &per_cu, raymarch_pair_kernel<KIND, COUNT, PW>, 64, 0));
    grid = (per_cu < 1 ? 1 : per_cu) * ctx->props.multiProcessorCount;
  }
  grid = (grid + 7) & ~7;
  unsigned int *queue = nullptr;
  const meso_status st = band_queue(ctx, stream, &queue);
  if (st != MESO_OK) return st;
  hipLaunchKernelGGL((raymarch_pair_kernel<KIND, COUNT, PW>), dim3((uint32_t)grid), dim3(64), 0,
                     stream, scene->dev(), cam, flags, sh, out, packets_x, n_packets, queue);
  MESO_HIP(hipGetLastError());
  return MESO_OK;
}

template <int KIND, bool COUNT, int PW>
static meso_status launch_persistent(meso_context *ctx, const meso_scene *scene,
                                     const DevCamera &cam, uint32_t flags, const DevShading &sh,
                                     const RayOut &out, hipStream_t stream, int grid) {
  constexpr int PH = 64 / PW;
  const uint32_t packets_x = (uint32_t)((cam.width + PW - 1) / PW);
  const uint32_t n_packets = packets_x * (uint32_t)((cam.height + PH - 1) / PH);
  if (grid <= 0) {
    int per_cu = 0;
    MESO_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
        &per_cu, raymarch_persistent_kernel<KIND, COUNT, PW>, 64, 0));
    grid = (per_cu < 1 ? 1 : per_cu) * ctx->props.multiProcessorCount;
  }
  grid = (grid + 7) & ~7;  // every XCD gets the same number of waves
  // one counter set per stream: launches on one stream are ordered, and
  // launches on different streams never share counters
  unsigned int *queue = nullptr;
  const meso_status st = band_queue(ctx, stream, &queue);
  if (st != MESO_OK) return st;
  hipLaunchKernelGGL((raymarch_persistent_kernel<KIND, COUNT, PW>), dim3((uint32_t)grid), dim3(64), 0,
                     stream, scene->dev(), cam, flags, sh, out, packets_x, n_packets, queue);
  MESO_HIP(hipGetLastError());
  return MESO_OK;
}

template <int KIND, bool COUNT, int TW, int TH>
static meso_status launch_shape(const meso_scene *scene, const DevCamera &cam, uint32_t flags,
                                const DevShading &sh, const RayOut &out, hipStream_t stream) {
  const uint32_t tiles_x = (uint32_t)((cam.width + TW - 1) / TW);
  const uint32_t tiles_y = (uint32_t)((cam.height + TH - 1) / TH);
  const uint32_t n_tiles = tiles_x * tiles_y;
  // Groups of one row of tiles: of a frame's 64 rows and more every XCD gets
  // its share of each part.  Shorter frames are cut finer, into an odd number
  // of groups per row, so that no XCD gets the same columns of every row
  // (3840x2160 caves: whole rows 1936 us, two rows a group 1938, quarter rows,
  // which give XCD x the same columns of every second row, 2312).
  const uint32_t per_row = tiles_y >= 64u ? 1u : (tiles_y >= 24u ? 3u : 7u);
  const uint32_t group = (tiles_x + per_row - 1u) / per_row;
  const uint32_t per_xcd = ((n_tiles + group - 1u) / group + 7u) / 8u * group;
  hipLaunchKernelGGL((raymarch_kernel<KIND, COUNT, TW, TH>), dim3(8u * per_xcd), dim3(TW * TH), 0,
                     stream, scene->dev(), cam, flags, sh, out, tiles_x, n_tiles, group);
  MESO_HIP(hipGetLastError());
  return MESO_OK;
}

template <int KIND, bool COUNT>
static meso_status launch_kind(meso_context *ctx, const meso_scene *scene, const DevCamera &cam,
                               uint32_t flags, const DevShading &sh, const RayOut &out,
                               hipStream_t stream, int variant, int grid) {
  switch (variant) {
    case 0: return launch_shape<KIND, COUNT, 16, 16>(scene, cam, flags, sh, out, stream);
    case 1: return launch_shape<KIND, COUNT, 32, 8>(scene, cam, flags, sh, out, stream);
    case 2:
      if constexpr (KIND == 1 && !COUNT) {
        // a dense frame of at most kSmallWaves waves of 8x8 pixels per SIMD
        const uint32_t tiles_x = (uint32_t)((cam.width + 3) / 4),
                       tiles_y = (uint32_t)((cam.height + 3) / 4);
        if (tiles_x * tiles_y <= kSmallWaves * 16u * (uint32_t)ctx->props.multiProcessorCount) {
          hipLaunchKernelGGL(raymarch_dense_small_kernel, dim3(tiles_x * tiles_y), dim3(64), 0,
                             stream, scene->dev(), cam, flags, sh, out, tiles_x);
          MESO_HIP(hipGetLastError());
          return MESO_OK;
        }
      }
      return launch_shape<KIND, COUNT, 8, 8>(scene, cam, flags, sh, out, stream);
    case 3: return launch_shape<KIND, COUNT, 16, 8>(scene, cam, flags, sh, out, stream);
    case 4: return launch_shape<KIND, COUNT, 32, 16>(scene, cam, flags, sh, out, stream);
    case 5: return launch_persistent<KIND, COUNT, 8>(ctx, scene, cam, flags, sh, out, stream, grid);
    case 6: return launch_persistent<KIND, COUNT, 16>(ctx, scene, cam, flags, sh, out, stream, grid);
    case 7: return launch_persistent<KIND, COUNT, 32>(ctx, scene, cam, flags, sh, out, stream, grid);
    case 8: return launch_pair<KIND, COUNT, 8>(ctx, scene, cam, flags, sh, out, stream, grid);
    case 9: return launch_pair<KIND, COUNT, 16>(ctx, scene, cam, flags, sh, out, stream, grid);
    default: return fail(MESO_ERR_ARGUMENT_OUT_OF_RANGE, "unknown raymarch variant %d", variant);
  }
}

// Where no shape was tuned: one wave a workgroup, so a slot is free again as
// soon as its own 8x8 pixels are done, not the slowest of four packets.
// 1920x1080 hills 170 us against 179 with 16x16 tiles, 3840x2160 caves 1936
// against 1950; persistent waves 2036 there, and some 200 us more on the
// smallest frames.  A launch that counts steps adds eleven counters to memory
// per workgroup, on words that all of them share, and keeps the four packets
// (1280x720 over 128^3 hills 228 us with 8x8 tiles, 119 with 16x16).
RayLaunch default_ray_launch(bool count) {
  return count ? RayLaunch{0, 256, 16, 16, 0} : RayLaunch{2, 64, 8, 8, 0};
}

meso_status launch_raymarch(meso_context *ctx, const meso_scene *scene, const DevCamera &cam,
                            uint32_t flags, const DevShading &sh, const RayOut &out,
                            hipStream_t stream, const RayLaunch *shape) {
  const bool count = (flags & MESO_RAY_COUNT) != 0;
  const int variant = shape ? shape->variant : default_ray_launch(count).variant;
  const int grid = shape ? shape->grid : 0;
  switch (scene->kind) {
    case MESO_SCENE_DENSE_U8:
      return count ? launch_kind<1, true>(ctx, scene, cam, flags, sh, out, stream, variant, grid)
                   : launch_kind<1, false>(ctx, scene, cam, flags, sh, out, stream, variant, grid);
    case MESO_SCENE_BRICKMAP_U16:
      return count ? launch_kind<2, true>(ctx, scene, cam, flags, sh, out, stream, variant, grid)
                   : launch_kind<2, false>(ctx, scene, cam, flags, sh, out, stream, variant, grid);
    case MESO_SCENE_TWO_LEVEL_U16:
      return count ? launch_kind<3, true>(ctx, scene, cam, flags, sh, out, stream, variant, grid)
                   : launch_kind<3, false>(ctx, scene, cam, flags, sh, out, stream, variant, grid);
    default: return fail(MESO_ERR_ARGUMENT_OUT_OF_RANGE, "unknown scene kind %d", scene->kind);
  }
}

}  // namespace meso
