// GPU voxelization: seeded scene generators into dense / brick-map /
// two-level layouts, the chunk batch for meshing, the reference sphere
// generator with its erosion mip chain, and brick edits.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "meso_internal.h"
#include "noise.h"
#include "traverse.h"

namespace meso {

// ------------------------------------------------------------------ scan
// Exclusive prefix sum of u32 flags (1024 elements per workgroup, recursive
// over block sums).  Used to assign brick and node slots in linear order.
__global__ void __launch_bounds__(256) scan_block_kernel(const uint32_t *in, uint32_t *out,
                                                         uint64_t n, uint32_t *block_sums) {
  __shared__ uint32_t s[256];
  const uint64_t base = (uint64_t)blockIdx.x * 1024u + threadIdx.x * 4u;
  uint32_t v[4];
  uint32_t sum = 0;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    v[k] = base + k < n ? in[base + k] : 0u;
    sum += v[k];
  }
  s[threadIdx.x] = sum;
  __syncthreads();
  for (uint32_t off = 1; off < 256; off <<= 1) {
    uint32_t add = threadIdx.x >= off ? s[threadIdx.x - off] : 0u;
    __syncthreads();
    s[threadIdx.x] += add;
    __syncthreads();
  }
  uint32_t run = s[threadIdx.x] - sum;  // exclusive
#pragma unroll
  for (int k = 0; k < 4; k++) {
    if (base + k < n) out[base + k] = run;
    run += v[k];
  }
  if (threadIdx.x == 255) block_sums[blockIdx.x] = s[255];
}

__global__ void scan_add_kernel(uint32_t *out, uint64_t n, const uint32_t *offsets) {
  const uint64_t i = (uint64_t)blockIdx.x * 1024u + threadIdx.x * 4u;
  const uint32_t add = offsets[blockIdx.x];
#pragma unroll
  for (int k = 0; k < 4; k++)
    if (i + k < n) out[i + k] += add;
}

// Workspace of scan_u32 over n elements: two words per 1024 elements and level.
static uint64_t scan_ws_words(uint64_t n) {
  uint64_t w = 0;
  while (n > 1) {
    n = (n + 1023) / 1024;
    w += 2 * n;
  }
  return w + 2;
}

// out[i] = sum(in[0..i)); the total goes to *total (device).  ws:
// scan_ws_words(n) words; no allocation and no wait.
static meso_status scan_u32(const uint32_t *in, uint32_t *out, uint64_t n, uint32_t *total,
                            uint32_t *ws, hipStream_t stream) {
  const uint64_t nb = (n + 1023) / 1024;
  uint32_t *sums = nb > 1 ? ws : total, *sums_scan = ws + nb;
  hipLaunchKernelGGL(scan_block_kernel, dim3((uint32_t)nb), dim3(256), 0, stream, in, out, n, sums);
  MESO_HIP(hipGetLastError());
  if (nb > 1) {
    meso_status st = scan_u32(sums, sums_scan, nb, total, ws + 2 * nb, stream);
    if (st != MESO_OK) return st;
    hipLaunchKernelGGL(scan_add_kernel, dim3((uint32_t)nb), dim3(256), 0, stream, out, n, sums_scan);
    MESO_HIP(hipGetLastError());
  }
  return MESO_OK;
}

// ------------------------------------------------------------------ dense spheres
constexpr int kMaxSpheres = 64;
struct SphereSet {
  int32_t count;
  int32_t p[4 * kMaxSpheres];  // cx, cy, cz, r in 1/256 voxel
};

// voxel centre (x + 1/2) against a sphere, exact integer arithmetic
__device__ __forceinline__ bool in_sphere_fp(const int32_t *s, int32_t x, int32_t y, int32_t z) {
  const int64_t dx = (int64_t)x * 256 + 128 - s[0];
  const int64_t dy = (int64_t)y * 256 + 128 - s[1];
  const int64_t dz = (int64_t)z * 256 + 128 - s[2];
  const int64_t r = s[3];
  return dx * dx + dy * dy + dz * dz <= r * r;
}

__global__ void spheres_dense_kernel(uint8_t *grid, int32_t n, SphereSet set,
                                     unsigned long long *solid) {
  const uint64_t total = (uint64_t)n * n * n;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  // grid-stride: every wave runs the same number of iterations
  const uint64_t rounds = (total + stride - 1) / stride;
  for (uint64_t it = 0; it < rounds; it++) {
    const uint64_t i = it * stride + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint8_t m = 0;
    if (i < total) {
      const int32_t x = (int32_t)(i % n), y = (int32_t)((i / n) % n),
                    z = (int32_t)(i / ((uint64_t)n * n));
      for (int k = 0; k < set.count; k++)
        if (in_sphere_fp(&set.p[4 * k], x, y, z)) {
          m = (uint8_t)(1 + k);
          break;
        }
      grid[i] = m;
    }
    const unsigned long long b = __ballot(m != 0);
    if ((threadIdx.x & 63u) == 0 && b) atomicAdd(solid, (unsigned long long)__popcll(b));
  }
}

// ------------------------------------------------------------------ brick scenes
__global__ void heights_kernel(int32_t *h, int32_t n, uint32_t seed, int32_t gen) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (uint64_t)n * n) return;
  const int32_t x = (int32_t)(i % n), z = (int32_t)(i / n);
  h[i] = gen == MESO_GEN_HEIGHTFIELD ? heightfield_height(x, z, n, seed)
                                     : terrain_height(x, z, n, seed);
}

// brick order: linear (brick map) or node-major (two-level: node * 4096 + local)
__device__ __forceinline__ void brick_of(uint64_t ordered, int32_t nb, bool two_level, int32_t &bx,
                                         int32_t &by, int32_t &bz) {
  if (!two_level) {
    bx = (int32_t)(ordered % nb);
    by = (int32_t)((ordered / nb) % nb);
    bz = (int32_t)(ordered / ((uint64_t)nb * nb));
  } else {
    const int32_t nt = nb / 16;
    const uint64_t node = ordered / 4096u;
    const uint32_t local = (uint32_t)(ordered % 4096u);
    const int32_t tx = (int32_t)(node % nt), ty = (int32_t)((node / nt) % nt),
                  tz = (int32_t)(node / ((uint64_t)nt * nt));
    bx = tx * 16 + (int32_t)(local & 15u);
    by = ty * 16 + (int32_t)((local >> 4) & 15u);
    bz = tz * 16 + (int32_t)(local >> 8);
  }
}

// What the brick kernels need of a generator.  [lo, hi]: the octave sums
// `sum` for which |fl(fl(sum / norm) - 1/2)| < threshold.  Both roundings are
// monotone, so these sums form an interval; its ends are found on the host
// (band_of_sums), and the kernels compare two floats per voxel instead of
// dividing.
struct BrickGen {
  int32_t gen, n;
  uint32_t seed;
  int32_t octaves;
  float base_freq, lo, hi;
  const int32_t *heights;
};

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __uint_as_float((uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(v), lane));
}
__device__ __forceinline__ float from_lane(float v, uint32_t lane) {
  return __uint_as_float(
      (uint32_t)__builtin_amdgcn_ds_bpermute((int)(lane * 4u), (int)__float_as_uint(v)));
}

// Octave sums of fbm3 over a brick by one wave: lane x + 8 y, sum[z] for the
// brick's 8 planes, each in fbm3's order of operations.
// What bounds it is instruction issue: hashing the 8 lattice corners of every
// voxel (14 hashes per octave, each with two quarter-rate multiplies) took
// most of the time.  A brick touches at most 3 lattice points per axis when a
// lattice cell is at least 8 voxels wide (f <= 1/8), so the 27 points of an
// octave are hashed by 27 lanes at once (two octaves per pass), and each lane
// fetches its corners by lane permutes.  The x and y interpolation is done
// once per column, since only the z weight changes along it.  At least 8
// voxels wide is every octave of scenes of 256 voxels and more; an octave with
// smaller cells hashes per voxel (value_noise3).
__device__ __forceinline__ void brick_fbm(const BrickGen &g, uint32_t seed, int32_t x0, int32_t y0,
                                          int32_t z0, float sum[8]) {
  const uint32_t lane = threadIdx.x & 63u;
  const float x = (float)(x0 + (int32_t)(lane & 7u)), y = (float)(y0 + (int32_t)(lane >> 3));
  // lane o * 8 + z: the z weight and lattice plane (relative to the brick's
  // first) of octave o at plane z
  const float fz_l = g.base_freq * (float)(1u << ((lane >> 3) & 3u));
  const float pz = (float)(z0 + (int32_t)(lane & 7u)) * fz_l;
  const float flz = __builtin_floorf(pz);
  const float uz_l = fade(pz - flz);
  const int32_t dz_l = (int32_t)flz - (int32_t)__builtin_floorf((float)z0 * fz_l);
  float lattice = 0.0f;
#pragma unroll
  for (int z = 0; z < 8; z++) sum[z] = 0.0f;
  float amp = 1.0f, f = g.base_freq;
#pragma unroll
  for (int o = 0; o < 4; o++) {
    if (o < g.octaves) {
      const uint32_t so = seed + (uint32_t)o * kOctaveSeedStep;
      if (f <= 0.125f) {
        if ((o & 1) == 0) {
          // lattice points of octaves o (lanes 0..26) and o + 1 (lanes 32..58)
          const float fl = lane < 32u ? f : f * 2.0f;
          const uint32_t sl = lane < 32u ? so : so + kOctaveSeedStep;
          const uint32_t r = lane & 31u, rz = r / 9u, ry = (r - rz * 9u) / 3u,
                         rx = r - rz * 9u - ry * 3u;
          const uint32_t ix = (uint32_t)(int32_t)__builtin_floorf((float)x0 * fl) + rx,
                         iy = (uint32_t)(int32_t)__builtin_floorf((float)y0 * fl) + ry,
                         iz = (uint32_t)(int32_t)__builtin_floorf((float)z0 * fl) + rz;
          lattice = hash_unit(nhash32(ix ^ nhash32(iy ^ nhash32(iz ^ sl))));
        }
        const float px = x * f, py = y * f;
        const float flx = __builtin_floorf(px), fly = __builtin_floorf(py);
        const float ux = fade(px - flx), uy = fade(py - fly);
        const uint32_t dx = (uint32_t)((int32_t)flx - (int32_t)__builtin_floorf((float)x0 * f)),
                       dy = (uint32_t)((int32_t)fly - (int32_t)__builtin_floorf((float)y0 * f));
        const uint32_t at = (uint32_t)(o & 1) * 32u + dx + 3u * dy;
        auto plane = [&](uint32_t level) {
          const uint32_t p = at + 9u * level;
          const float a = lerpf(from_lane(lattice, p), from_lane(lattice, p + 1u), ux);
          const float b = lerpf(from_lane(lattice, p + 3u), from_lane(lattice, p + 4u), ux);
          return lerpf(a, b, uy);
        };
        const float y0v = plane(0u), y1v = plane(1u);
        // the last plane of voxels lies in the second cell (uniform)
        const bool two = __builtin_amdgcn_readlane(dz_l, o * 8 + 7) != 0;
        const float y2v = two ? plane(2u) : y1v;
#pragma unroll
        for (int z = 0; z < 8; z++) {
          const bool second = __builtin_amdgcn_readlane(dz_l, o * 8 + z) != 0;
          const float n = lerpf(second ? y1v : y0v, second ? y2v : y1v, lane_value(uz_l, o * 8 + z));
          const float an = amp * n;
          sum[z] = sum[z] + an;
        }
      } else {
        for (int z = 0; z < 8; z++) {
          const float n = value_noise3(x * f, y * f, (float)(z0 + z) * f, so);
          const float an = amp * n;
          sum[z] = sum[z] + an;
        }
      }
      amp = amp * 0.5f;
      f = f * 2.0f;
    }
  }
}

// The occupancy words of brick (bx, by, bz) by one wave: m[z], bit x + 8 y.
// False when the brick is empty.
__device__ __forceinline__ bool brick_words(const BrickGen &g, int32_t bx, int32_t by, int32_t bz,
                                            uint64_t m[8]) {
  const uint32_t lane = threadIdx.x & 63u;
  const int32_t x0 = bx * 8, y0 = by * 8, z0 = bz * 8;
  int32_t h = 0;
  if (g.gen != MESO_GEN_CAVES) {
    // lane x + 8 z: the column's height; the whole brick lies above the
    // ground when no column reaches its lowest voxels
    h = g.heights[(int64_t)(z0 + (int32_t)(lane >> 3)) * g.n + x0 + (int32_t)(lane & 7u)];
    if (__ballot(h > y0) == 0ull) return false;
  }
  float sum[8];
  if (g.gen != MESO_GEN_HEIGHTFIELD)
    brick_fbm(g, g.gen == MESO_GEN_CAVES ? g.seed : g.seed ^ 0x5bd1e995u, x0, y0, z0, sum);
  const int32_t y = y0 + (int32_t)(lane >> 3);
  uint64_t any = 0;
#pragma unroll
  for (int z = 0; z < 8; z++) {
    bool solid;
    if (g.gen == MESO_GEN_CAVES) {
      solid = sum[z] >= g.lo && sum[z] <= g.hi;
    } else {
      solid = y < __shfl(h, (int)((lane & 7u) + 8u * (uint32_t)z), 64);
      if (g.gen == MESO_GEN_TERRAIN_CAVES) solid = solid && !(sum[z] >= g.lo && sum[z] <= g.hi);
    }
    m[z] = __ballot(solid);
    any |= m[z];
  }
  return any != 0ull;
}

// Which bricks hold a voxel, and how many voxels are solid: one wave per
// brick, `per` bricks in turn, so that a workgroup adds to the voxel count
// once (one add per brick kept the adds to that one word, at a few
// nanoseconds each, in the way).
__global__ void __launch_bounds__(256) brick_flags_kernel(BrickGen g, int32_t two_level,
                                                          uint32_t *flags,
                                                          unsigned long long *solid,
                                                          uint64_t n_bricks, uint32_t per) {
  __shared__ uint32_t wave_solid[4];
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint64_t first = (block_id() * 4u + wave) * per;
  const int32_t nb = g.n / 8;
  uint32_t count = 0;
  for (uint32_t k = 0; k < per && first + k < n_bricks; k++) {
    int32_t bx, by, bz;
    brick_of(first + k, nb, two_level != 0, bx, by, bz);
    uint64_t m[8];
    const bool any = brick_words(g, bx, by, bz, m);
    if (any) {
#pragma unroll
      for (int z = 0; z < 8; z++) count += (uint32_t)__popcll(m[z]);
    }
    if ((threadIdx.x & 63u) == 0) flags[first + k] = any ? 1u : 0u;
  }
  if ((threadIdx.x & 63u) == 0) wave_solid[wave] = count;
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t all = wave_solid[0] + wave_solid[1] + wave_solid[2] + wave_solid[3];
    if (all) atomicAdd(solid, (unsigned long long)all);
  }
}

// Writes the slots, and the masks and voxels of the bricks that hold a voxel:
// one wave per brick, `per` bricks in turn.  The words are computed again (a
// third of the bricks at most need it) rather than kept, which would take 64
// bytes per brick cell.  A voxel's material depends on its height alone, so a
// lane writes one row of 8 voxels (y, z) from its byte of the words: one
// 1 KiB store per brick.
__global__ void __launch_bounds__(256) brick_write_kernel(BrickGen g, int32_t two_level,
                                                          const uint32_t *flags,
                                                          const uint32_t *prefix,
                                                          const uint32_t *node_ids,
                                                          uint32_t *slots, uint64_t *masks,
                                                          uint16_t *voxels, uint64_t n_bricks,
                                                          uint32_t per) {
  const int32_t nb = g.n / 8;
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint64_t first = (block_id() * 4u + wave) * per;
  for (uint32_t k = 0; k < per && first + k < n_bricks; k++) {
    const uint64_t ordered = first + k;
    const bool live = flags[ordered] != 0u;
    uint64_t cell = ordered;
    if (two_level) {
      // bricks of empty nodes have no slot table
      const uint32_t node = node_ids[ordered / 4096u];
      if (node == kEmptySlot) continue;
      cell = (uint64_t)node * 4096u + ordered % 4096u;
    }
    if (lane == 0) slots[cell] = live ? prefix[ordered] : kEmptySlot;
    if (!live) continue;
    int32_t bx, by, bz;
    brick_of(ordered, nb, two_level != 0, bx, by, bz);
    uint64_t m[8];
    brick_words(g, bx, by, bz, m);
    uint64_t w = m[0];
#pragma unroll
    for (uint32_t z = 1; z < 8u; z++) w = (lane >> 3) == z ? m[z] : w;
    const uint64_t slot = prefix[ordered];
    if ((lane & 7u) == 0) masks[slot * 8u + (lane >> 3)] = w;
    const uint32_t row = (uint32_t)(w >> (8u * (lane & 7u))) & 0xFFu;
    const int32_t y = by * 8 + (int32_t)(lane & 7u);
    const uint32_t mat = g.gen == MESO_GEN_CAVES ? caves_material(y) : height_band(y, g.n);
    uint32_t v[4];
#pragma unroll
    for (int j = 0; j < 4; j++)
      v[j] = (((row >> (2 * j)) & 1u) | (((row >> (2 * j + 1)) & 1u) << 16)) * mat;
    *(uint4 *)(voxels + slot * 512u + 8u * lane) = make_uint4(v[0], v[1], v[2], v[3]);
  }
}

__global__ void node_flags_kernel(const uint32_t *brick_flags, uint32_t *node_flags) {
  __shared__ uint32_t any;
  if (threadIdx.x == 0) any = 0;
  __syncthreads();
  uint32_t a = 0;
  for (uint32_t i = threadIdx.x; i < 4096u; i += blockDim.x)
    a |= brick_flags[(uint64_t)blockIdx.x * 4096u + i];
  if (a) atomicOr(&any, 1u);
  __syncthreads();
  if (threadIdx.x == 0) node_flags[blockIdx.x] = any;
}

__global__ void node_ids_kernel(const uint32_t *node_flags, const uint32_t *node_prefix,
                                uint32_t *top, uint64_t n_top) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_top) top[i] = node_flags[i] ? node_prefix[i] : kEmptySlot;
}

// ------------------------------------------------------------------ chunk batch
struct ChunkParamsDev {
  uint32_t noise_seed;
  uint32_t target;       // solid voxels wanted from the noise
  int32_t n_spheres;
  int32_t sph[4][4];
};

__device__ __forceinline__ int32_t chunk_noise_q(int32_t x, int32_t y, int32_t z, uint32_t seed) {
  float v = fbm3((float)x, (float)y, (float)z, 2, 0.125f, seed);
  v = v * 256.0f;
  int32_t q = (int32_t)v;
  return q > 255 ? 255 : q;
}

// One workgroup per chunk: quantised noise into LDS with a 256-bin histogram,
// threshold at the fill quantile, spheres drawn over it.
__global__ void __launch_bounds__(1024) chunk_gen_kernel(const ChunkParamsDev *params,
                                                         uint16_t *out) {
  __shared__ uint8_t q[32768];
  __shared__ uint32_t hist[256];
  __shared__ uint32_t thr;
  const ChunkParamsDev p = params[blockIdx.x];
  if (threadIdx.x < 256) hist[threadIdx.x] = 0;
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < 32768u; i += 1024u) {
    const int32_t x = (int32_t)(i & 31u), y = (int32_t)((i >> 5) & 31u), z = (int32_t)(i >> 10);
    const int32_t v = chunk_noise_q(x, y, z, p.noise_seed);
    q[i] = (uint8_t)v;
    atomicAdd(&hist[v], 1u);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t t = 0, cum = 0;
    while (cum < p.target && t < 256u) {
      cum += hist[t];
      t++;
    }
    thr = t;
  }
  __syncthreads();
  const uint32_t T = thr;
  uint16_t *o = out + (uint64_t)blockIdx.x * 32768u;
  for (uint32_t i = threadIdx.x; i < 32768u; i += 1024u) {
    const int32_t x = (int32_t)(i & 31u), y = (int32_t)((i >> 5) & 31u), z = (int32_t)(i >> 10);
    uint16_t m = 0;
    for (int s = 0; s < p.n_spheres; s++)
      if (in_sphere_fp(p.sph[s], x, y, z)) {
        m = (uint16_t)(5 + s);
        break;
      }
    const uint32_t qi = q[i];
    if (!m && qi < T) m = (uint16_t)(1u + (qi * 4u) / T);
    o[i] = m;
  }
}

// ------------------------------------------------------------------ reference sphere + erosion
// FGeneratorHelper::GenerateSphere (Runtimes/Helper/GeneratorHelper.h:120-150)
// and FChunk::CalculateOccupancyErodeMipmaps (Runtimes/Voxel/Chunk/Chunk.h:73-94)
// with the 26-neighbour ErodeSingleVoxel rule (BinaryOccupancyVolume.h:76-99).
__global__ void __launch_bounds__(256) sphere_chunk_kernel(const int32_t *chunk_xyz, int32_t res,
                                                           double block_size, int32_t depth,
                                                           uint8_t *mips) {
  extern __shared__ uint8_t lds[];  // 2 * res^3
  const int32_t vol = res * res * res;
  uint8_t *cur = lds, *prev = lds + vol;
  const int32_t cx = chunk_xyz[3 * blockIdx.x], cy = chunk_xyz[3 * blockIdx.x + 1],
                cz = chunk_xyz[3 * blockIdx.x + 2];
  const double cr = (double)res;
  uint8_t *out = mips + (uint64_t)blockIdx.x * depth * vol;
  for (int32_t i = threadIdx.x; i < vol; i += blockDim.x) {
    const int32_t X = i % res, Y = (i / res) % res, Z = i / (res * res);
    double px = (double)cx * block_size * cr + (double)X * block_size;
    double py = (double)cy * block_size * cr + (double)Y * block_size;
    double pz = (double)cz * block_size * cr + (double)Z * block_size;
    double dx = px - 100.0, dy = py, dz = pz;
    double dd = dx * dx + dy * dy;
    dd = dd + dz * dz;
    double d = __builtin_sqrt(dd) - 50.0;
    const uint8_t s = d < 0.0 ? 1 : 0;
    prev[i] = s;
    out[i] = s;
  }
  __syncthreads();
  for (int32_t lvl = 1; lvl < depth; lvl++) {
    for (int32_t i = threadIdx.x; i < vol; i += blockDim.x) {
      const int32_t X = i % res, Y = (i / res) % res, Z = i / (res * res);
      uint8_t e = 0;
      if (out[i] && X >= 1 && Y >= 1 && Z >= 1 && X < res - 1 && Y < res - 1 && Z < res - 1) {
        e = 1;
        for (int dz = -1; dz <= 1; dz++)
          for (int dy = -1; dy <= 1; dy++)
            for (int dx = -1; dx <= 1; dx++) {
              if (!dx && !dy && !dz) continue;
              e &= prev[(X + dx) + (Y + dy) * res + (Z + dz) * res * res];
            }
      }
      cur[i] = e;
      out[(uint64_t)lvl * vol + i] = e;
    }
    __syncthreads();
    uint8_t *t = cur;
    cur = prev;
    prev = t;
  }
}

// ------------------------------------------------------------------ brick edits
__global__ void __launch_bounds__(512) brick_update_kernel(const uint32_t *edit_slots,
                                                           const uint16_t *edit_vox,
                                                           int64_t n_bricks, uint64_t *masks,
                                                           uint64_t *blocks,
                                                           const uint32_t *slot_cell,
                                                           uint16_t *voxels,
                                                           uint32_t *bad, uint64_t n_edit) {
  const uint64_t e = block_id();
  if (e >= n_edit) return;
  const uint32_t slot = edit_slots[e];
  if ((int64_t)slot >= n_bricks) {  // every lane takes the same branch
    if (threadIdx.x == 0 && bad) atomicAdd(bad, 1u);
    return;
  }
  const uint16_t v = edit_vox[e * 512u + threadIdx.x];
  const unsigned long long b = __ballot(v != 0);
  voxels[(uint64_t)slot * 512u + threadIdx.x] = v;
  if ((threadIdx.x & 63u) == 0) masks[(uint64_t)slot * 8u + (threadIdx.x >> 6)] = (uint64_t)b;
  const uint64_t sub = brick_blocks2_from_planes((uint64_t)b);
  if (threadIdx.x == 0 && slot_cell[slot] != 0u) blocks[slot_cell[slot] - 1u] = sub;
}

// ------------------------------------------------------------------ chunk edits
// cell (index into slots) of brick (bx,by,bz) in a brick map or two-level
// scene, or kEmptySlot outside the grid or in an empty node
__device__ __forceinline__ uint32_t scene_brick_cell(const DevScene &s, int32_t kind, int32_t bx,
                                                     int32_t by, int32_t bz) {
  const int32_t nb = s.n >> 3;
  if (bx < 0 || by < 0 || bz < 0 || bx >= nb || by >= nb || bz >= nb) return kEmptySlot;
  if (kind == MESO_SCENE_BRICKMAP_U16)
    return (uint32_t)bx + ((uint32_t)by + (uint32_t)bz * (uint32_t)nb) * (uint32_t)nb;
  const uint32_t nt = (uint32_t)s.n >> 7;
  const uint32_t node = s.top[((uint32_t)bx >> 4) + (((uint32_t)by >> 4) + ((uint32_t)bz >> 4) * nt) * nt];
  if (node == kEmptySlot) return kEmptySlot;
  return node * 4096u + ((uint32_t)bx & 15u) + 16u * ((uint32_t)by & 15u) +
         256u * ((uint32_t)bz & 15u);
}

// The mask words and the 2^3-block bits of a brick held by one wave, lane =
// row of 8 voxels (y + 8 z), from each row's bits: a row is a byte of the
// mask's 64, and four lanes' folded rows make the block bits of two z planes'
// y pair.
__device__ __forceinline__ void write_brick_bits(uint32_t row, uint64_t *mask, uint64_t *block) {
  const uint32_t lane = threadIdx.x & 63u;
  ((uint8_t *)mask)[lane] = (uint8_t)row;
  uint32_t f = row | (uint32_t)__shfl_xor((int)row, 1, 64);
  f |= (uint32_t)__shfl_xor((int)f, 8, 64);
  f |= f >> 1;  // bits 0, 2, 4, 6: the x pairs
  f = (f & 1u) | ((f >> 1) & 2u) | ((f >> 2) & 4u) | ((f >> 3) & 8u);
  f |= (uint32_t)__shfl_xor((int)f, 2, 64) << 4;  // used where y is 0 or 4: cy, cy + 1
  if ((lane & 0xBu) == 0u)  // y in {0, 4}, z even: byte 2 cz + cy / 2 of the word
    ((uint8_t *)block)[((lane >> 4) << 1) | ((lane >> 2) & 1u)] = (uint8_t)f;
}

// One workgroup of 8 waves per chunk, a wave per brick.  Its first wave looks
// up the 64 bricks' cells and slots at once (one lane each) and lists those to
// edit; a wave then holds a whole brick in one 16-byte load per lane, so bricks
// need no barrier and no LDS.  What bounds it is the latency of those few
// loads.  ALL: every allocated brick's mask follows its voxels, as it must
// where uploaded masks may differ from them; otherwise only the bricks that
// the sphere reaches can change, and the rest is not read.  (A workgroup per
// brick in turn, with the mask and block bits folded across waves, took 69 us
// for 2,621 chunks of the 2048^3 caves and 33 us for 40 terrain chunks; this
// takes 15 and 10 us or less.)
template <bool ALL>
__global__ void __launch_bounds__(512) edit_chunks_kernel(DevScene s, int32_t kind,
                                                          const int32_t *xyz, uint32_t seed,
                                                          uint64_t *masks, uint64_t *blocks,
                                                          uint16_t *voxels, uint64_t n_chunks) {
  __shared__ uint32_t live_b[64], live_cell[64], live_slot[64];
  __shared__ uint32_t n_live;
  const uint64_t chunk = block_id();
  if (chunk >= n_chunks) return;
  const int32_t nc = (s.n + 31) >> 5;  // a partial last chunk counts
  const int32_t cx = xyz[3 * chunk], cy = xyz[3 * chunk + 1], cz = xyz[3 * chunk + 2];
  if (cx < 0 || cy < 0 || cz < 0 || cx >= nc || cy >= nc || cz >= nc) return;
  const uint32_t h0 = nhash32(seed ^ nhash32((uint32_t)cx + ((uint32_t)cy + (uint32_t)cz * (uint32_t)nc) * (uint32_t)nc));
  const uint32_t h1 = nhash32(h0), h2 = nhash32(h1), h3 = nhash32(h2);
  // the sphere in the chunk's own coordinates, 1/256 voxel: every distance is
  // below 2^13 and every sum of squares below 2^28
  const int32_t sx = (int32_t)(h0 & 0x1FFFu), sy = (int32_t)(h1 & 0x1FFFu),
                sz = (int32_t)(h2 & 0x1FFFu);
  const int32_t r = 4 * 256 + (int32_t)(h3 % (8u * 256u)), r2 = r * r;
  if (threadIdx.x < 64u) {
    const uint32_t i = threadIdx.x;
    const int32_t lb[3] = {(int32_t)(i & 3u), (int32_t)((i >> 2) & 3u), (int32_t)(i >> 4)};
    const uint32_t cell = scene_brick_cell(s, kind, cx * 4 + lb[0], cy * 4 + lb[1], cz * 4 + lb[2]);
    const uint32_t slot = cell == kEmptySlot ? kEmptySlot : s.slots[cell];
    bool edit = slot != kEmptySlot;
    if (!ALL) {
      // the brick's voxel centre nearest to the sphere's
      const int32_t c[3] = {sx, sy, sz};
      int32_t q = 0;
#pragma unroll
      for (int a = 0; a < 3; a++) {
        int32_t v = c[a] >> 8;  // the voxel that holds the centre: its own centre is nearest
        v = v < lb[a] * 8 ? lb[a] * 8 : (v > lb[a] * 8 + 7 ? lb[a] * 8 + 7 : v);
        const int32_t d = v * 256 + 128 - c[a];
        q += d * d;
      }
      edit = edit && q <= r2;
    }
    const unsigned long long live = __ballot(edit);
    if (edit) {
      const uint32_t k = (uint32_t)__popcll(live & ((1ull << i) - 1ull));  // in brick order
      live_b[k] = i;
      live_cell[k] = cell;
      live_slot[k] = slot;
    }
    if (i == 0) n_live = (uint32_t)__popcll(live);
  }
  __syncthreads();
  const uint32_t n = n_live, lane = threadIdx.x & 63u;
  for (uint32_t k = threadIdx.x >> 6; k < n; k += 8u) {
    const uint32_t b = live_b[k], cell = live_cell[k], slot = live_slot[k];
    uint4 *row = (uint4 *)(voxels + (uint64_t)slot * 512u + 8u * lane);
    const uint4 v = *row;
    uint32_t w[4] = {v.x, v.y, v.z, v.w};
    const int32_t x0 = (int32_t)(b & 3u) * 2048 + 128 - sx;
    const int32_t dy = (int32_t)(((b >> 2) & 3u) * 8u + (lane & 7u)) * 256 + 128 - sy;
    const int32_t dz = (int32_t)((b >> 4) * 8u + (lane >> 3)) * 256 + 128 - sz;
    const int32_t left = r2 - dy * dy - dz * dz;  // what dx * dx may take
    uint32_t bits = 0, changed = 0;
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const int32_t dx = x0 + 256 * j;
      const uint32_t old = (w[j >> 1] >> (16 * (j & 1))) & 0xFFFFu;
      const bool in = dx * dx <= left;
      const uint32_t val = in ? (old ? 0u : 7u) : old;
      w[j >> 1] = (w[j >> 1] & (0xFFFFu << (16 * (1 - (j & 1))))) | (val << (16 * (j & 1)));
      bits |= (val ? 1u : 0u) << j;
      changed |= in ? 1u : 0u;
    }
    if (changed) *row = make_uint4(w[0], w[1], w[2], w[3]);
    write_brick_bits(bits, masks + (uint64_t)slot * 8u, blocks + cell);
  }
}

// *bad: whether some brick's mask is not that of its voxels.  A wave per brick.
__global__ void __launch_bounds__(256) mask_check_kernel(const uint64_t *masks,
                                                         const uint16_t *voxels, uint64_t n_bricks,
                                                         uint32_t *bad) {
  const uint64_t slot = block_id() * 4u + (threadIdx.x >> 6);
  if (slot >= n_bricks) return;  // uniform over the wave
  const uint32_t lane = threadIdx.x & 63u;
  const uint4 v = *(const uint4 *)(voxels + slot * 512u + 8u * lane);
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  uint32_t bits = 0;
#pragma unroll
  for (int j = 0; j < 8; j++) bits |= ((w[j >> 1] >> (16 * (j & 1))) & 0xFFFFu ? 1u : 0u) << j;
  const bool differs = bits != ((const uint8_t *)(masks + slot * 8u))[lane];
  if (__ballot(differs) && lane == 0) atomicOr(bad, 1u);
}

meso_status launch_mask_check(const meso_scene *sc, uint32_t *bad, hipStream_t stream) {
  if (sc->n_bricks == 0) return MESO_OK;
  hipLaunchKernelGGL(mask_check_kernel, grid_1d(((uint64_t)sc->n_bricks + 3) / 4), dim3(256), 0,
                     stream, sc->masks, sc->voxels, (uint64_t)sc->n_bricks, bad);
  MESO_HIP(hipGetLastError());
  return MESO_OK;
}

}  // namespace meso

using namespace meso;

// the sums whose noise value lies within `thr` of 1/2 (see BrickGen): the
// first and last positive float of the interval, found by bisection of the
// float's bits on both sides of the middle
static bool in_band(float sum, float norm, float thr) {
  float c = sum / norm;
  c = c - 0.5f;
  return std::fabs(c) < thr;
}
static float band_end(float norm, float thr, uint32_t outside) {
  float mid = 0.5f * norm;
  uint32_t in, out = outside;
  std::memcpy(&in, &mid, 4);
  while (in > out ? in - out > 1u : out - in > 1u) {
    const uint32_t probe = in > out ? out + (in - out) / 2u : in + (out - in) / 2u;
    float v;
    std::memcpy(&v, &probe, 4);
    if (in_band(v, norm, thr)) in = probe;
    else out = probe;
  }
  float r;
  std::memcpy(&r, &in, 4);
  return r;
}

// Fills sc's slots, masks and voxels (and top table) from the generator.
// scratch: the words meso_scene_generate counts out, first the totals.
static meso_status generate_bricks(meso_scene *sc, int32_t gen, uint32_t seed, uint32_t *scratch,
                                   hipStream_t stream) {
  const int32_t n = sc->n, nb = n / 8, nt = n / 128;
  const bool two = sc->kind == MESO_SCENE_TWO_LEVEL_U16;
  const uint64_t cells = (uint64_t)nb * nb * nb, n_top = two ? (uint64_t)nt * nt * nt : 0;
  uint32_t *totals = scratch;  // [0] bricks, [1] nodes, [2..3] solid voxels
  uint32_t *flags = totals + 4, *prefix = flags + cells;
  uint32_t *node_flags = prefix + cells, *node_prefix = node_flags + n_top;
  int32_t *heights = (int32_t *)(node_prefix + n_top);
  uint32_t *ws = (uint32_t *)heights + (gen != MESO_GEN_CAVES ? (uint64_t)n * n : 0);
  meso_status st = launch_zero(totals, 16, stream);
  if (st != MESO_OK) return st;
  if (gen != MESO_GEN_CAVES) {
    hipLaunchKernelGGL(heights_kernel, dim3((uint32_t)(((uint64_t)n * n + 255) / 256)), dim3(256),
                       0, stream, heights, n, seed, gen);
    MESO_HIP(hipGetLastError());
  }
  BrickGen g{};
  g.gen = gen;
  g.n = n;
  g.seed = seed;
  g.heights = heights;
  g.octaves = gen == MESO_GEN_CAVES ? 4 : 3;
  g.base_freq = gen == MESO_GEN_CAVES ? 1.0f / 64.0f : 8.0f / (float)n;
  const float norm = gen == MESO_GEN_CAVES ? 1.875f : 1.75f;  // 1 + 1/2 + 1/4 (+ 1/8)
  const float thr = gen == MESO_GEN_CAVES ? kCavesBand : kTunnelBand;
  g.lo = band_end(norm, thr, 0u);
  g.hi = band_end(norm, thr, 0x40000000u);
  // a wave takes several bricks once there are more than 16 waves per CU
  const uint32_t waves = (uint32_t)sc->ctx->props.multiProcessorCount * 16u;
  uint32_t per = (uint32_t)(cells / waves);
  per = per < 1u ? 1u : (per > 16u ? 16u : per);
  const dim3 grid = grid_1d((cells + 4u * per - 1) / (4u * per));
  hipLaunchKernelGGL(brick_flags_kernel, grid, dim3(256), 0, stream, g, two ? 1 : 0, flags,
                     (unsigned long long *)(totals + 2), cells, per);
  MESO_HIP(hipGetLastError());
  st = scan_u32(flags, prefix, cells, totals, ws, stream);
  if (st != MESO_OK) return st;
  if (two) {
    hipLaunchKernelGGL(node_flags_kernel, dim3((uint32_t)n_top), dim3(256), 0, stream, flags,
                       node_flags);
    MESO_HIP(hipGetLastError());
    st = scan_u32(node_flags, node_prefix, n_top, totals + 1, ws, stream);
    if (st != MESO_OK) return st;
  }
  uint32_t t[4];
  MESO_HIP(hipMemcpyAsync(t, totals, sizeof(t), hipMemcpyDeviceToHost, stream));
  MESO_HIP(hipStreamSynchronize(stream));
  const uint64_t n_bricks = t[0], n_nodes = t[1];
  sc->n_bricks = (int64_t)n_bricks;
  sc->n_nodes = (int64_t)n_nodes;
  sc->solid = (int64_t)((uint64_t)t[2] | ((uint64_t)t[3] << 32));
  MESO_CHECK(n_bricks < (1ull << 29), MESO_ERR_OUT_OF_MEMORY, "%llu bricks exceed 2^29",
             (unsigned long long)n_bricks);
  if (two) {
    MESO_HIP(hipMalloc((void **)&sc->top, n_top * 4));
    hipLaunchKernelGGL(node_ids_kernel, dim3((uint32_t)((n_top + 255) / 256)), dim3(256), 0,
                       stream, node_flags, node_prefix, sc->top, n_top);
    MESO_HIP(hipGetLastError());
    MESO_HIP(hipMalloc((void **)&sc->slots, std::max<uint64_t>(n_nodes, 1) * 4096 * 4));
    sc->bytes += n_top * 4 + n_nodes * 4096 * 4;
  } else {
    MESO_HIP(hipMalloc((void **)&sc->slots, cells * 4));
    sc->bytes += cells * 4;
  }
  MESO_HIP(hipMalloc((void **)&sc->masks, std::max<uint64_t>(n_bricks, 1) * 64));
  MESO_HIP(hipMalloc((void **)&sc->voxels, std::max<uint64_t>(n_bricks, 1) * 1024));
  sc->bytes += n_bricks * (64 + 1024);
  hipLaunchKernelGGL(brick_write_kernel, grid, dim3(256), 0, stream, g, two ? 1 : 0, flags, prefix,
                     sc->top, sc->slots, sc->masks, sc->voxels, cells, per);
  MESO_HIP(hipGetLastError());
  return MESO_OK;
}

static meso_status gen_free(meso_scene *sc, meso_status st) {
  if (sc) {
    hipSetDevice(sc->ctx->device);
    hipStreamSynchronize(sc->ctx->stream);
    free_scene_arrays(sc);
    delete sc;
  }
  return st;
}

#define GEN_TRY(expr)                      \
  do {                                     \
    meso_status st_ = (expr);              \
    if (st_ != MESO_OK) return gen_free(sc, st_); \
  } while (0)
#define GEN_HIP(call)                                                                  \
  do {                                                                                 \
    hipError_t e_ = (call);                                                            \
    if (e_ != hipSuccess)                                                              \
      return gen_free(sc, fail(e_ == hipErrorOutOfMemory ? MESO_ERR_OUT_OF_MEMORY      \
                                                         : MESO_ERR_RUNTIME,           \
                               "%s: %s", #call, hipGetErrorString(e_)));               \
  } while (0)

extern "C" {

meso_status meso_scene_generate(meso_context *ctx, const meso_generate_desc *d, meso_scene **out) {
  MESO_CHECK(ctx && d && out, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "NULL argument");
  MESO_CHECK(d->size >= sizeof(meso_generate_desc), MESO_ERR_ARGUMENT_OUT_OF_RANGE,
             "meso_generate_desc.size too small");
  *out = nullptr;
  const int32_t n = d->n;
  const uint32_t seed = (uint32_t)(d->seed ^ (d->seed >> 32));
  MESO_HIP(hipSetDevice(ctx->device));
  hipStream_t stream = ctx->stream;
  meso_scene *sc = nullptr;
  if (d->generator == MESO_GEN_SPHERES) {
    MESO_CHECK(d->layout == MESO_SCENE_DENSE_U8, MESO_ERR_NOT_SUPPORTED,
               "sphere scenes are generated as dense u8 grids");
    MESO_CHECK(n >= 1 && n <= 2048, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "dense edge %d", n);
    MESO_CHECK(d->n_spheres >= 1 && d->n_spheres <= kMaxSpheres && d->n_spheres < 256,
               MESO_ERR_ARGUMENT_OUT_OF_RANGE, "n_spheres %d not in 1..%d", d->n_spheres,
               kMaxSpheres);
    SphereSet set{};
    set.count = d->n_spheres;
    Pcg32 r;
    r.seed(d->seed);
    const uint32_t span = (uint32_t)n * 256u;
    for (int i = 0; i < d->n_spheres; i++) {
      set.p[4 * i + 0] = (int32_t)(r.next() % span);
      set.p[4 * i + 1] = (int32_t)(r.next() % span);
      set.p[4 * i + 2] = (int32_t)(r.next() % span);
      set.p[4 * i + 3] = (int32_t)(8 * 256 + r.next() % (24u * 256u + 1u));
    }
    sc = new meso_scene();
    sc->ctx = ctx;
    sc->kind = MESO_SCENE_DENSE_U8;
    sc->n = n;
    const uint64_t total = (uint64_t)n * n * n;
    GEN_HIP(hipMalloc((void **)&sc->dense, total));
    sc->bytes = total;
    unsigned long long *solid = nullptr;
    GEN_HIP(hipMallocAsync((void **)&solid, 8, stream));
    GEN_TRY(launch_zero(solid, 8, stream));
    hipLaunchKernelGGL(spheres_dense_kernel, dim3((uint32_t)std::min<uint64_t>((total + 255) / 256, 1u << 20)), dim3(256), 0,
                       stream, sc->dense, n, set, solid);
    GEN_HIP(hipGetLastError());
    unsigned long long s = 0;
    GEN_HIP(hipMemcpyAsync(&s, solid, 8, hipMemcpyDeviceToHost, stream));
    GEN_HIP(hipFreeAsync(solid, stream));
    GEN_HIP(hipStreamSynchronize(stream));
    sc->solid = (int64_t)s;
    *out = sc;
    return MESO_OK;
  }
  MESO_CHECK(d->generator == MESO_GEN_HEIGHTFIELD || d->generator == MESO_GEN_TERRAIN_CAVES ||
                 d->generator == MESO_GEN_CAVES,
             MESO_ERR_ARGUMENT_OUT_OF_RANGE, "unknown generator %d", d->generator);
  const bool two = d->layout == MESO_SCENE_TWO_LEVEL_U16;
  MESO_CHECK(d->layout == MESO_SCENE_BRICKMAP_U16 || two, MESO_ERR_NOT_SUPPORTED,
             "procedural scenes are built as brick maps or two-level maps");
  MESO_CHECK(two ? (n >= 128 && n % 128 == 0 && n <= 4096) : (n >= 8 && n % 8 == 0 && n <= 4096),
             MESO_ERR_ARGUMENT_OUT_OF_RANGE, "edge %d invalid for layout %d", n, d->layout);
  const int32_t nb = n / 8;
  const uint64_t n_brick_cells = (uint64_t)nb * nb * nb;
  MESO_CHECK(n_brick_cells < 0xFFFFFFFFull, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "too many bricks");
  sc = new meso_scene();
  sc->ctx = ctx;
  sc->kind = two ? MESO_SCENE_TWO_LEVEL_U16 : MESO_SCENE_BRICKMAP_U16;
  sc->n = n;
  const int32_t nt = n / 128;
  const uint64_t n_top = two ? (uint64_t)nt * nt * nt : 0;
  // one scratch allocation: totals (bricks, nodes, solid voxels), flags and
  // prefix per brick cell and per node, column heights, the scans' sums
  const uint64_t words = 4 + 2 * n_brick_cells + 2 * n_top +
                         (d->generator != MESO_GEN_CAVES ? (uint64_t)n * n : 0) +
                         scan_ws_words(n_brick_cells);
  uint32_t *scratch = nullptr;
  GEN_HIP(hipMallocAsync((void **)&scratch, words * 4, stream));
  const meso_status st = generate_bricks(sc, d->generator, seed, scratch, stream);
  // the stream is idle on success; after a failure gen_free waits for it
  (void)hipFreeAsync(scratch, stream);
  if (st != MESO_OK) return gen_free(sc, st);
  sc->masks_match = true;  // brick_write_kernel makes both from the same words
  GEN_TRY(build_coarse(sc, stream, false));
  *out = sc;
  return MESO_OK;
}

meso_status meso_generate_chunks(meso_context *ctx, uint64_t seed, int32_t n_chunks,
                                 uint16_t *d_out, meso_stream stream) {
  MESO_CHECK(ctx && d_out, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "NULL argument");
  MESO_CHECK(n_chunks >= 1 && n_chunks <= (1 << 20), MESO_ERR_ARGUMENT_OUT_OF_RANGE,
             "n_chunks %d not in 1..2^20", n_chunks);
  // Per-chunk parameters from PCG32: Beta(1/2,1/2) fill as cos^2 of a uniform
  // angle (a point uniform in the unit disk by rejection), noise seed, spheres.
  std::vector<ChunkParamsDev> host((size_t)n_chunks);
  Pcg32 r;
  r.seed(seed);
  for (int32_t c = 0; c < n_chunks; c++) {
    float a, b, r2;
    for (;;) {
      a = r.u01() * 2.0f;
      a = a - 1.0f;
      b = r.u01() * 2.0f;
      b = b - 1.0f;
      float aa = a * a, bb = b * b;
      r2 = aa + bb;
      if (r2 < 1.0f && r2 > 0.0f) break;
    }
    float aa = a * a;
    float fill = aa / r2;
    ChunkParamsDev &p = host[(size_t)c];
    p.noise_seed = r.next();
    p.n_spheres = 1 + (int32_t)(r.next() % 4u);
    for (int i = 0; i < 4; i++) {
      p.sph[i][0] = (int32_t)(r.next() % (32u * 256u));
      p.sph[i][1] = (int32_t)(r.next() % (32u * 256u));
      p.sph[i][2] = (int32_t)(r.next() % (32u * 256u));
      p.sph[i][3] = (int32_t)(3 * 256 + r.next() % (9u * 256u + 1u));
    }
    float tf = fill * 32768.0f;
    tf = tf + 0.5f;
    p.target = (uint32_t)tf;
  }
  hipStream_t s = stream_of(ctx, stream);
  MESO_HIP(hipSetDevice(ctx->device));
  ChunkParamsDev *dp = nullptr;
  MESO_HIP(hipMallocAsync((void **)&dp, host.size() * sizeof(ChunkParamsDev), s));
  MESO_HIP(hipMemcpyAsync(dp, host.data(), host.size() * sizeof(ChunkParamsDev),
                          hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(chunk_gen_kernel, dim3((uint32_t)n_chunks), dim3(1024), 0, s, dp, d_out);
  MESO_HIP(hipGetLastError());
  MESO_HIP(hipFreeAsync(dp, s));
  MESO_HIP(hipStreamSynchronize(s));
  return MESO_OK;
}

meso_status meso_generate_sphere_chunks(meso_context *ctx, const int32_t *d_chunk_xyz,
                                        int32_t n_chunks, int32_t res, float block_size,
                                        int32_t depth, uint8_t *d_mips, meso_stream stream) {
  MESO_CHECK(ctx && d_chunk_xyz && d_mips, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "NULL argument");
  MESO_CHECK(n_chunks >= 1 && n_chunks <= (1 << 20) && res >= 1 && res <= 32 && depth >= 1 &&
                 depth <= 8,
             MESO_ERR_ARGUMENT_OUT_OF_RANGE, "n_chunks %d, res %d (1..32), depth %d (1..8)",
             n_chunks, res, depth);
  hipStream_t s = stream_of(ctx, stream);
  MESO_HIP(hipSetDevice(ctx->device));
  const size_t lds = 2u * (size_t)res * res * res;
  hipLaunchKernelGGL(sphere_chunk_kernel, dim3((uint32_t)n_chunks), dim3(256), lds, s,
                     d_chunk_xyz, res, (double)block_size, depth, d_mips);
  MESO_HIP(hipGetLastError());
  return MESO_OK;
}

meso_status meso_scene_edit_chunks(meso_scene *scene, const int32_t *d_chunk_xyz, int32_t n_chunks,
                                   uint32_t seed, meso_stream stream) {
  MESO_CHECK(scene && d_chunk_xyz, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "NULL argument");
  MESO_CHECK(scene->kind != MESO_SCENE_DENSE_U8, MESO_ERR_NOT_SUPPORTED,
             "chunk edits need a brick map or two-level scene");
  MESO_CHECK(n_chunks >= 0 && n_chunks <= (1 << 24), MESO_ERR_ARGUMENT_OUT_OF_RANGE,
             "n_chunks %d out of range", n_chunks);
  if (n_chunks == 0) return MESO_OK;
  hipStream_t s = stream_of(scene->ctx, stream);
  MESO_HIP(hipSetDevice(scene->ctx->device));
  const auto kernel = scene->masks_match ? edit_chunks_kernel<false> : edit_chunks_kernel<true>;
  hipLaunchKernelGGL(kernel, grid_1d((uint64_t)n_chunks), dim3(512), 0, s, scene->dev(),
                     scene->kind, d_chunk_xyz, seed, scene->masks, scene->blocks, scene->voxels,
                     (uint64_t)n_chunks);
  MESO_HIP(hipGetLastError());
  return MESO_OK;
}

meso_status meso_scene_update_bricks(meso_scene *scene, const uint32_t *d_slots,
                                     const uint16_t *d_voxels, int32_t n_edit, meso_stream stream) {
  MESO_CHECK(scene && d_slots && d_voxels, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "NULL argument");
  MESO_CHECK(scene->kind != MESO_SCENE_DENSE_U8, MESO_ERR_NOT_SUPPORTED,
             "brick edits need a brick map or two-level scene");
  MESO_CHECK(n_edit >= 0, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "negative edit count");
  if (n_edit == 0) return MESO_OK;
  hipStream_t s = stream_of(scene->ctx, stream);
  MESO_HIP(hipSetDevice(scene->ctx->device));
  uint32_t *bad = nullptr;
  MESO_HIP(hipMallocAsync((void **)&bad, 16, s));
  meso_status st = launch_zero(bad, 16, s);
  if (st != MESO_OK) return st;
  hipLaunchKernelGGL(brick_update_kernel, grid_1d((uint64_t)n_edit), dim3(512), 0, s, d_slots,
                     d_voxels, scene->n_bricks, scene->masks, scene->blocks, scene->slot_cell,
                     scene->voxels, bad,
                     (uint64_t)n_edit);
  MESO_HIP(hipGetLastError());
  uint32_t nbad = 0;
  MESO_HIP(hipMemcpyAsync(&nbad, bad, 4, hipMemcpyDeviceToHost, s));
  MESO_HIP(hipFreeAsync(bad, s));
  MESO_HIP(hipStreamSynchronize(s));
  MESO_CHECK(nbad == 0, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "%u edits named a slot >= n_bricks", nbad);
  return MESO_OK;
}

meso_status meso_scene_update_bricks_async(meso_scene *scene, const uint32_t *d_slots,
                                           const uint16_t *d_voxels, int32_t n_edit,
                                           uint32_t *d_skipped, meso_stream stream) {
  MESO_CHECK(scene && d_slots && d_voxels, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "NULL argument");
  MESO_CHECK(scene->kind != MESO_SCENE_DENSE_U8, MESO_ERR_NOT_SUPPORTED,
             "brick edits need a brick map or two-level scene");
  MESO_CHECK(n_edit >= 0, MESO_ERR_ARGUMENT_OUT_OF_RANGE, "negative edit count");
  if (n_edit == 0) return MESO_OK;
  hipStream_t s = stream_of(scene->ctx, stream);
  MESO_HIP(hipSetDevice(scene->ctx->device));
  hipLaunchKernelGGL(brick_update_kernel, grid_1d((uint64_t)n_edit), dim3(512), 0, s, d_slots,
                     d_voxels, scene->n_bricks, scene->masks, scene->blocks, scene->slot_cell,
                     scene->voxels, d_skipped,
                     (uint64_t)n_edit);
  MESO_HIP(hipGetLastError());
  return MESO_OK;
}

}  // extern "C"
