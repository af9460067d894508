// raycast.hip -- fixed-step ray march over the hashed TSDF with regula-falsi
// refinement.
//
// Reference: visualization/ray_caster.cu:16-150 (CastKernel),
// geometry/isosurface_intersection.h:13-55 (LinearIntersection,
// BisectionIntersection), geometry/spatial_query.h:23-97 (trilinear value and
// gradient), geometry/voxel_query.h:102-129 (world-point voxel lookup).
//
// One lane per pixel, 8x8 pixels per wave (two or four lanes per pixel for
// small images).  Samples, the crossing test and
// the three regula-falsi steps follow the reference's FP32 expressions.  The
// march keeps the eight blocks around its current lowest-corner block
// (Octant) and shares block lookups, misses included, through a per-wave LDS
// table, so runs of samples in one block, or in one unallocated block, cost
// no hash probe; the neighbours come from a table filled before the march.
// The depth output is metric z (t * dir_c.z); the reference colour-maps it
// (ray_caster.cu:96-98) and keeps metric depth only in the vertex image.
#include <type_traits>

#include "mh_kernels.h"

namespace mh {

// Block lookups shared by the rays of a workgroup (one wave; four in the
// localiser's kernel of four lanes a point): a
// direct-mapped LDS table that a lane fills after a hash probe, so a block
// is probed about once per workgroup rather than once per ray.  An entry is one
// 64-bit word, read and written whole (relaxed atomics: single LDS
// instructions), so a reader always gets a block and its own index whatever
// order the divergent paths and the other waves run in: bits 0-23 hold the pool
// index + 3 (0 marks an empty slot),
// bits 24-63 the block coordinates minus the low bits that chose the slot
// (x, y: 3 bits, z: 2 bits), which makes (slot, entry) name one block.
// Blocks beyond +-2^15 on an axis bypass the table.  Of a wave's lanes that miss
// on one slot in the same instruction, only the one whose id survives in
// `owner` writes it.  That saves stores and decides nothing else: lanes of two
// waves may both write a slot, and any of the entries is a true one.
constexpr int kWaveTable = 256;
struct WaveTable {
  uint64_t e[kWaveTable];
  uint32_t owner[kWaveTable];
};
__device__ __forceinline__ void wave_table_init(WaveTable* t) {
  for (uint32_t i = threadIdx.x; i < (uint32_t)kWaveTable; i += 64u) t->e[i] = 0ull;
  __syncthreads();
}

// A block's pool index; kFreePtr if it is absent, kAbsentSuper if no block of
// its super-block was ever allocated either.  Both filters' words and the
// bucket's first slot are loaded together (one round trip in the usual cases).
constexpr int32_t kAbsentSuper = -1;
__device__ __forceinline__ int32_t ray_probe(const View& V, i3 b) {
  if (!coord_ok(b)) return kFreePtr;
  const uint64_t key = pack_key(b);
  const uint32_t bit = occ_bit(key), sbit = occ2_bit(super_key(b));
  const uint32_t first = hash_bucket(b, V.bucket_count) * V.bucket_size;
  const uint32_t word = V.occ[bit >> 5], sword = V.occ2[sbit >> 5];
  const Entry e0 = V.entries[first];
  if (!((word >> (bit & 31u)) & 1u)) return ((sword >> (sbit & 31u)) & 1u) ? kFreePtr : kAbsentSuper;
  if (e0.key == key) return e0.ptr;
  return hash_find_key<true>(V, b, key);
}

__device__ __forceinline__ int32_t table_find(const View& V, WaveTable* t, i3 b) {
  const int lim = 1 << 15;
  if (b.x < -lim || b.x >= lim || b.y < -lim || b.y >= lim || b.z < -lim || b.z >= lim) return ray_probe(V, b);
  const uint32_t slot = (uint32_t)(b.x & 7) | ((uint32_t)(b.y & 7) << 3) | ((uint32_t)(b.z & 3) << 6);
  const uint64_t tag = (uint64_t)((uint32_t)(b.x >> 3) & 0x1FFFu) |
                       ((uint64_t)((uint32_t)(b.y >> 3) & 0x1FFFu) << 13) |
                       ((uint64_t)((uint32_t)(b.z >> 2) & 0x3FFFu) << 26);
  const uint64_t e = __hip_atomic_load(&t->e[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  if (e != 0ull && (e >> 24) == tag) return (int32_t)(e & 0xFFFFFFu) - 3;
  const int32_t p = ray_probe(V, b);
  if (p >= (1 << 24) - 3) return p;  // does not fit the entry
  const uint32_t lane = threadIdx.x & 63u;
  volatile uint32_t* owner = t->owner;
  owner[slot] = lane;
  if (owner[slot] == lane)
    __hip_atomic_store(&t->e[slot], (tag << 24) | (uint64_t)(uint32_t)(p + 3), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_WORKGROUP);
  return p;
}

// The eight blocks around a lowest-corner block b: b + (i>>2 & 1, i>>1 & 1,
// i & 1) for entry i, kept while the march stays with b.  Entry 0 comes from
// the wave's table, the others from the block's row of V.oct (below) in two
// 16-byte loads.
struct Octant {
  int bx, by, bz;
  int32_t p[8];
};
__device__ __forceinline__ Octant empty_octant() {
  return Octant{INT32_MIN, INT32_MIN, INT32_MIN, {kFreePtr, -1, -1, -1, -1, -1, -1, -1}};
}
__device__ __forceinline__ void octant_move(const View& V, WaveTable* t, Octant& oc, int bx, int by, int bz) {
  if (bx == oc.bx && by == oc.by && bz == oc.bz) return;
  oc.bx = bx;
  oc.by = by;
  oc.bz = bz;
  oc.p[0] = table_find(V, t, i3{bx, by, bz});
  if (oc.p[0] < 0) return;
  const int4* row = reinterpret_cast<const int4*>(V.oct) + 2 * (size_t)oc.p[0];
  const int4 lo = row[0], hi = row[1];
  oc.p[1] = lo.y;
  oc.p[2] = lo.z;
  oc.p[3] = lo.w;
  oc.p[4] = hi.x;
  oc.p[5] = hi.y;
  oc.p[6] = hi.z;
  oc.p[7] = hi.w;
}

// One axis of a sample at coordinate p: the two corner voxels of its
// trilinear cell (rounded from p - vs/2 and p + vs/2, spatial_query.h:23-66;
// from a multiply by 1/vs when that is clear of a rounding tie, see
// corner_pair).
struct RCell {
  int x0, x1, y0, y1, z0, z1;
};
__device__ __forceinline__ RCell ray_cell(f3 pos, float vs, float inv_vs) {
  const float hv = 0.5f * vs;
  RCell c;
  // per axis, so that a wave runs the divisions only for the axes on which
  // some lane is near a tie
  corner_pair(pos.x - hv, vs, inv_vs, &c.x0, &c.x1);
  corner_pair(pos.y - hv, vs, inv_vs, &c.y0, &c.y1);
  corner_pair(pos.z - hv, vs, inv_vs, &c.z0, &c.z1);
  return c;
}
// The ratio frac(p / vs) of an axis.
__device__ __forceinline__ float ray_ratio(float p, float vs, float inv_vs) {
  const float q = quotient(p, vs, inv_vs);
  return q - floorf(q);
}
struct RAxis {
  int c0, c1;
  float r;
};
__device__ __forceinline__ RAxis ray_axis(float p, float vs, float inv_vs) {
  RAxis a;
  corner_pair(p - 0.5f * vs, vs, inv_vs, &a.c0, &a.c1);
  a.r = ray_ratio(p, vs, inv_vs);
  return a;
}

// Where the eight corner voxels of a cell lie in a voxel field (corner i: bit
// 2 x, bit 1 y, bit 0 z set); false if one of the blocks holding them is
// absent.  Offsets are in bytes and 32-bit, so that a load takes one address
// register beside the field's scalar base, unless the pool is larger than
// kNarrowCapacity blocks (kWide: 64-bit).
constexpr uint32_t kNarrowCapacity = 1u << 21;  // x 2 KiB a block
template <bool kWide>
struct RayOffset { using type = uint32_t; };
template <>
struct RayOffset<true> { using type = uint64_t; };
template <bool kWide>
using ray_offset = typename RayOffset<kWide>::type;
template <bool kWide>
__device__ __forceinline__ float field_at(const float* __restrict__ f, ray_offset<kWide> off) {
  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(f) + off);
}
template <bool kWide>
__device__ __forceinline__ bool cell_corners(const View& V, WaveTable* t, Octant& oc, const RCell& c,
                                             ray_offset<kWide> off[8]) {
  const int bx = voxel_to_block1(c.x0), by = voxel_to_block1(c.y0), bz = voxel_to_block1(c.z0);
  octant_move(V, t, oc, bx, by, bz);
  if (oc.p[0] < 0) {
    return false;
  }
  const bool xx = voxel_to_block1(c.x1) != bx, yy = voxel_to_block1(c.y1) != by, zz = voxel_to_block1(c.z1) != bz;
  if (V.ray_mark) {  // diagnostics: blocks sampled
    V.ray_mark[oc.p[0]] = V.ray_stamp;
#pragma unroll
    for (int i = 1; i < 8; ++i) {
      if (!((!(i & 4) || xx) && (!(i & 2) || yy) && (!(i & 1) || zz))) continue;
      if (oc.p[i] < 0) return false;
      V.ray_mark[oc.p[i]] = V.ray_stamp;
    }
  }
  // block of each corner, by selects
  const int32_t p0 = oc.p[0];
  const int32_t p1 = zz ? oc.p[1] : p0;
  const int32_t p2 = yy ? oc.p[2] : p0;
  const int32_t p3 = yy ? (zz ? oc.p[3] : oc.p[2]) : p1;
  const int32_t p4 = xx ? oc.p[4] : p0;
  const int32_t p5 = xx ? (zz ? oc.p[5] : oc.p[4]) : p1;
  const int32_t p6 = xx ? (yy ? oc.p[6] : oc.p[4]) : p2;
  const int32_t p7 = xx ? (yy ? (zz ? oc.p[7] : oc.p[6]) : (zz ? oc.p[5] : oc.p[4])) : p3;
  if (min(min(min(p1, p2), min(p3, p4)), min(min(p5, p6), p7)) < 0) return false;
  const uint32_t x0 = (uint32_t)(c.x0 & 7) * 4u, x1 = (uint32_t)(c.x1 & 7) * 4u;
  const uint32_t y0 = (uint32_t)(c.y0 & 7) * 32u, y1 = (uint32_t)(c.y1 & 7) * 32u;
  const uint32_t z0 = (uint32_t)(c.z0 & 7) * 256u, z1 = (uint32_t)(c.z1 & 7) * 256u;
  const int32_t pb[8] = {p0, p1, p2, p3, p4, p5, p6, p7};
#pragma unroll
  for (int i = 0; i < 8; ++i)
    off[i] = (ray_offset<kWide>)(uint32_t)pb[i] * (kBlockVoxels * 4u) +
             (((i & 4) ? x1 : x0) + ((i & 2) ? y1 : y0) + ((i & 1) ? z1 : z0));
  return true;
}

// The trilinear sum of GetSpatialValue (spatial_query.h:23-66), corner by
// corner in the reference's order.
__device__ __forceinline__ float trilinear(const float v[8], float rx, float ry, float rz) {
  float sdf = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float w = ((i & 4) ? rx : 1.0f - rx) * ((i & 2) ? ry : 1.0f - ry) * ((i & 1) ? rz : 1.0f - rz);
    sdf += w * v[i];
  }
  return sdf;
}

// GetSpatialValue's SDF at a point; false if a corner's block is absent (a
// missing lowest-corner block ends the sample after one compare while the
// octant is kept, which is how empty space inside the tile range costs
// little).  The ratios are the reference's quotients.
template <bool kWide>
__device__ __forceinline__ bool point_sample(const View& V, WaveTable* t, Octant& oc, f3 pos, float inv_vs,
                                             float* out) {
  const float vs = V.geo.voxel_size;
  ray_offset<kWide> off[8];
  if (!cell_corners<kWide>(V, t, oc, ray_cell(pos, vs, inv_vs), off)) return false;
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = field_at<kWide>(V.sdf, off[i]);
  *out = trilinear(v, ray_ratio(pos.x, vs, inv_vs), ray_ratio(pos.y, vs, inv_vs), ray_ratio(pos.z, vs, inv_vs));
  return true;
}

// GetSpatialSDFGradient's samples at p -+ vs/2 e_k (spatial_query.h:68-97):
// as central differences; false if any is invalid.  p -+ h e_k equals p off
// axis k (x - 0 = x), so the stencils take p's own axes there.  One sample site
// in a rolled loop: an axis's two samples loaded together need 128 registers
// (four waves a SIMD) and were slower, 640 x 480 of a 5 mm desk 175 against
// 165 us.
template <bool kWide>
__device__ __forceinline__ bool gradient_samples(const View& V, WaveTable* t, Octant& oc, f3 p, float inv_vs,
                                                 float* g0, float* g1, float* g2) {
  const float vs = V.geo.voxel_size;
  const float h = 0.5f * vs;
  const RAxis X = ray_axis(p.x, vs, inv_vs), Y = ray_axis(p.y, vs, inv_vs), Z = ray_axis(p.z, vs, inv_vs);
  bool valid = true;
  float last = 0.0f;
  *g0 = *g1 = *g2 = 0.0f;
  // x-, x+, y-, y+, z-, z+ from one sample site
#pragma unroll 1
  for (int j = 0; j < 6 && valid; ++j) {
    const int k = j >> 1;
    const float pk = k == 0 ? p.x : (k == 1 ? p.y : p.z);
    const RAxis S = ray_axis((j & 1) ? pk + h : pk - h, vs, inv_vs);
    RCell c{X.c0, X.c1, Y.c0, Y.c1, Z.c0, Z.c1};
    if (k == 0) { c.x0 = S.c0; c.x1 = S.c1; }
    if (k == 1) { c.y0 = S.c0; c.y1 = S.c1; }
    if (k == 2) { c.z0 = S.c0; c.z1 = S.c1; }
    ray_offset<kWide> off[8];
    valid = cell_corners<kWide>(V, t, oc, c, off);
    if (!valid) break;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = field_at<kWide>(V.sdf, off[i]);
    const float s = trilinear(v, k == 0 ? S.r : X.r, k == 1 ? S.r : Y.r, k == 2 ? S.r : Z.r);
    const float gk = (s - last) / vs;
    last = s;
    if (j == 1) *g0 = gk;
    if (j == 3) *g1 = gk;
    if (j == 5) *g2 = gk;
  }
  return valid;
}

// A ray parameter below which every sample position o + t dir lies more
// than 0.01 voxel inside the world box [b bs, (b + 1) bs)^3 of cell b, bs
// its side (8 voxels for a block, 32 for a super-block).  A sample's lowest
// corner voxel is vox1(pos - vs/2) per axis, so its lowest-corner block lies
// in cell b exactly on that box; the margin is 20 times the
// FP32 error of the reference's quotient (pos - vs/2) / vs at 16 m and
// covers the error of the position.  The box is shrunk by 0.02 voxel, so
// the approximate divisions (a few ulp of t, well under 1e-5 m) only
// lower the bound.
__device__ __forceinline__ float cell_exit_t(f3 o, f3 dir, int bx, int by, int bz, float bs, float vs) {
  const float eps = 0.02f * vs;
  const float ex = dir.x > 0.0f ? (float)(bx + 1) * bs - eps : (float)bx * bs + eps;
  const float ey = dir.y > 0.0f ? (float)(by + 1) * bs - eps : (float)by * bs + eps;
  const float ez = dir.z > 0.0f ? (float)(bz + 1) * bs - eps : (float)bz * bs + eps;
  float te = INFINITY;
  if (dir.x != 0.0f) te = fminf(te, __fdividef(ex - o.x, dir.x));
  if (dir.y != 0.0f) te = fminf(te, __fdividef(ey - o.y, dir.y));
  if (dir.z != 0.0f) te = fminf(te, __fdividef(ez - o.z, dir.z));
  return te;
}
__device__ __forceinline__ float block_exit_t(f3 o, f3 dir, int bx, int by, int bz, float vs) {
  return cell_exit_t(o, dir, bx, by, bz, (float)kBlockSide * vs, vs);
}
// The same for an absent block: over its super-block (4^3 blocks) when no
// block of that was ever allocated, every sample whose lowest-corner block
// lies in it being invalid.
__device__ __forceinline__ float absent_exit_t(int32_t found, f3 o, f3 dir, int bx, int by, int bz, float vs) {
  if (found != kAbsentSuper) return block_exit_t(o, dir, bx, by, bz, vs);
  return cell_exit_t(o, dir, bx >> kSuperShift, by >> kSuperShift, bz >> kSuperShift,
                     (float)(kBlockSide << kSuperShift) * vs, vs);
}

// The first element >= target of the FP32 sequence t, t + step, ...
// (t += step, t > 0, step > 0), without taking every step.  Inside a binade
// [lo, 2 lo) every sum rounds to the grid u = lo 2^-23, so once a step has
// been taken inside the binade the increment is constant (an exact tie
// rounds to an even multiple of u, after which the tie always resolves the
// same way): with t1, t2, t3 in one binade, d = t3 - t2 repeats for as long
// as each exact sum t + step stays 2u below the binade's top.  The jump is
// computed in FP64, where t3 + k d is exact.
__device__ __forceinline__ float advance_steps(float t, float step, float target) {
  while (t < target) {
    const float t1 = t + step;
    if (!(t1 < target)) return t1;
    const float t2 = t1 + step;
    if (!(t2 < target)) return t2;
    const float t3 = t2 + step;
    if (!(t3 < target)) return t3;
    const float lo = __uint_as_float(__float_as_uint(t3) & 0x7F800000u);
    if (t1 < lo) {
      t = t3;
      continue;
    }
    const double top = 2.0 * (double)lo, u = (double)lo * 0x1p-23;
    const double d = (double)t3 - (double)t2;
    const double room = (top - 2.0 * u - (double)step - (double)t3) / d;
    if (!(room >= 1.0)) {
      t = t3;
      continue;
    }
    const double k = fmin(floor(room) + 1.0, ceil(((double)target - (double)t3) / d));
    t = (float)((double)t3 + k * d);
  }
  return t;
}

// The accepted crossing of one ray
// and (t_k, s_k), and the last regula-falsi point m.
struct Hit {
  float tp, sp, tk, sk, m;
};

// The march of CastKernel (ray_caster.cu:56-92): fixed FP32 steps, a
// crossing between the previous valid sample and the current one, three
// regula-falsi steps (isosurface_intersection.h:24-55), then the acceptance
// test.  A failed refinement or test continues the march.
//
// [t_lo, t_hi] bounds the ray parameters at which a sample can be valid (the
// tile's block range): earlier samples are stepped over without sampling,
// so the sample sequence t_min, t_min + step, ... stays the reference's, and
// the march ends after t_hi.
template <bool kWide>
__device__ __forceinline__ bool find_surface(const View& V, const RayConst& R, f3 o, f3 dir, float t_min,
                                             float t_max, float t_lo, float t_hi, WaveTable* table,
                                             Octant& oc, Hit* hit, uint32_t* nsamp) {
  float prev_sdf = 0.0f, prev_t = 0.0f;
  bool prev_ok = false;
  if (!(t_lo < t_max) || t_hi < t_lo) return false;  // no block along this ray
  float t = advance_steps(t_min, R.step, t_lo);
  // The march stops at each crossing candidate and refines it outside the
  // stepping loop, so a wave runs the refinement once for all its lanes
  // rather than once per step at which some lane crosses.
  while (true) {
    float s = 0.0f;
    bool cross = false;
    for (; t < t_max && t <= t_hi; t += R.step) {
      float sv;
      if (!point_sample<kWide>(V, table, oc, mk3(o.x + t * dir.x, o.y + t * dir.y, o.z + t * dir.z), R.inv_vs,
                               &sv)) {
        // Lowest-corner block absent: the following samples inside its box
        // (its super-block's, if that never held a block) are invalid too
        // (an invalid sample changes nothing); step over them with the same
        // FP32 additions, so the t sequence is kept.
        if (oc.p[0] < 0) {
          const float t_out = absent_exit_t(oc.p[0], o, dir, oc.bx, oc.by, oc.bz, V.geo.voxel_size);
          for (float tn = t + R.step; tn < t_out && tn > t; tn = t + R.step) t = tn;
        }
        continue;
      }
      ++*nsamp;
      if (prev_ok && prev_sdf > 0.0f && sv < 0.0f) {
        s = sv;
        cross = true;
        break;
      }
      prev_sdf = sv;
      prev_t = t;
      prev_ok = true;
    }
    if (!cross) return false;
    // BisectionIntersection: three regula-falsi steps.
    float l = prev_t, r = t, m = (l + r) * 0.5f;
    float l_sdf = prev_sdf, r_sdf = s;
    bool found = true;
#pragma unroll 1
    for (int k = 0; k < 3; ++k) {
      m = l + (l_sdf / (l_sdf - r_sdf)) * (r - l);
      float m_sdf;
      if (!point_sample<kWide>(V, table, oc, mk3(o.x + m * dir.x, o.y + m * dir.y, o.z + m * dir.z), R.inv_vs,
                               &m_sdf)) {
        found = false;
        break;
      }
      if (l_sdf * m_sdf > 0.0f) {
        l = m;
        l_sdf = m_sdf;
      } else {
        r = m;
        r_sdf = m_sdf;
      }
    }
    if (found && fabsf(prev_sdf - s) < R.sample_sdf_threshold && fabsf(s) < R.sdf_threshold) {
      *hit = Hit{prev_t, prev_sdf, t, s, m};
      return true;
    }
    // not accepted: the march goes on, with this sample as the previous one
    prev_sdf = s;
    prev_t = t;
    prev_ok = true;
    t += R.step;
  }
}

// Lane j of the L lanes that share a ray, as seen by all of them (L: 2 or 4,
// neighbouring lanes; they run one path except inside a sample).
template <int L, int J>
__device__ __forceinline__ uint32_t ray_lane(uint32_t x) {
  constexpr int ctrl = L == 4 ? J * 0x55 : (J | (J << 2) | ((2 + J) << 4) | ((2 + J) << 6));
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, ctrl, 0xF, 0xF, true);
}
template <int L, int J>
__device__ __forceinline__ float ray_lane(float x) {
  return __uint_as_float(ray_lane<L, J>(__float_as_uint(x)));
}

// find_surface by L lanes a ray: lane q takes every L-th sample, from the q-th
// on; the samples of a round are then walked through in the ray's order by all
// of its lanes, so that the crossing, the acceptance and the count are
// find_surface's.  A round ends with the last lane's sample; where that lies
// in an absent block, the next round starts behind the block.
template <bool kWide, int L>
__device__ __forceinline__ bool find_surface_split(const View& V, const RayConst& R, f3 o, f3 dir, float t_min,
                                                   float t_max, float t_lo, float t_hi, WaveTable* table,
                                                   Octant& oc, Hit* hit, uint32_t* nsamp) {
  float prev_sdf = 0.0f, prev_t = 0.0f;
  bool prev_ok = false;
  if (!(t_lo < t_max) || t_hi < t_lo) return false;  // no block along this ray
  float t = advance_steps(t_min, R.step, t_lo);
  const uint32_t q = threadIdx.x & (L - 1);
  while (true) {
    float s = 0.0f, tc = 0.0f;
    bool cross = false;
    while (t < t_max && t <= t_hi) {
      float ts[L];
      ts[0] = t;
#pragma unroll
      for (int j = 1; j < L; ++j) ts[j] = ts[j - 1] + R.step;
      float tq = ts[0];
#pragma unroll
      for (int j = 1; j < L; ++j) tq = q == (uint32_t)j ? ts[j] : tq;
      float sv = 0.0f, t_out = 0.0f;
      bool ok = false;
      if (tq < t_max && tq <= t_hi) {
        ok = point_sample<kWide>(V, table, oc, mk3(o.x + tq * dir.x, o.y + tq * dir.y, o.z + tq * dir.z), R.inv_vs, &sv);
        if (!ok && oc.p[0] < 0) t_out = absent_exit_t(oc.p[0], o, dir, oc.bx, oc.by, oc.bz, V.geo.voxel_size);
      }
      const uint32_t oku = ok ? 1u : 0u;
      auto take = [&](float v, uint32_t k, float tj) {
        if (cross || !k) return;
        ++*nsamp;
        if (prev_ok && prev_sdf > 0.0f && v < 0.0f) {
          s = v;
          tc = tj;
          cross = true;
          return;
        }
        prev_sdf = v;
        prev_t = tj;
        prev_ok = true;
      };
      take(ray_lane<L, 0>(sv), ray_lane<L, 0>(oku), ts[0]);
      take(ray_lane<L, 1>(sv), ray_lane<L, 1>(oku), ts[1]);
      if constexpr (L == 4) {
        take(ray_lane<L, 2>(sv), ray_lane<L, 2>(oku), ts[2]);
        take(ray_lane<L, 3>(sv), ray_lane<L, 3>(oku), ts[3]);
      }
      if (cross) break;
      const float out = ray_lane<L, L - 1>(t_out);
      t = ts[L - 1];
      for (float tn = t + R.step; tn < out && tn > t; tn = t + R.step) t = tn;
      t += R.step;
    }
    if (!cross) return false;
    // BisectionIntersection: three regula-falsi steps.
    float l = prev_t, r = tc, m = (l + r) * 0.5f;
    float l_sdf = prev_sdf, r_sdf = s;
    bool found = true;
#pragma unroll 1
    for (int k = 0; k < 3; ++k) {
      m = l + (l_sdf / (l_sdf - r_sdf)) * (r - l);
      float m_sdf;
      if (!point_sample<kWide>(V, table, oc, mk3(o.x + m * dir.x, o.y + m * dir.y, o.z + m * dir.z), R.inv_vs,
                               &m_sdf)) {
        found = false;
        break;
      }
      if (l_sdf * m_sdf > 0.0f) {
        l = m;
        l_sdf = m_sdf;
      } else {
        r = m;
        r_sdf = m_sdf;
      }
    }
    if (found && fabsf(prev_sdf - s) < R.sample_sdf_threshold && fabsf(s) < R.sdf_threshold) {
      *hit = Hit{prev_t, prev_sdf, tc, s, m};
      return true;
    }
    prev_sdf = s;
    prev_t = tc;
    prev_ok = true;
    t = tc + R.step;
  }
}

// gradient_samples by L lanes a ray, each taking one stencil sample a round.
template <bool kWide, int L>
__device__ __forceinline__ bool gradient_samples_split(const View& V, WaveTable* t, Octant& oc, f3 p, float inv_vs,
                                                       float* g0, float* g1, float* g2) {
  const float vs = V.geo.voxel_size, h = 0.5f * vs;
  const uint32_t q = threadIdx.x & (L - 1);
  bool valid = true;
  *g0 = *g1 = *g2 = 0.0f;
#pragma unroll 1
  for (int j0 = 0; j0 < 6; j0 += L) {
    const int j = min(j0 + (int)q, 5), k = j >> 1;  // x-, x+, y-, y+, z-, z+
    const float d = (j & 1) ? h : -h;
    float s = 0.0f;
    // (p - 0 = p: the other two coordinates are p's)
    const bool ok = point_sample<kWide>(V, t, oc, mk3(k == 0 ? p.x + d : p.x, k == 1 ? p.y + d : p.y, k == 2 ? p.z + d : p.z),
                                        inv_vs, &s);
    const uint32_t oku = ok ? 1u : 0u;
    valid = valid && ray_lane<L, 0>(oku) && ray_lane<L, 1>(oku);
    const float ga = (ray_lane<L, 1>(s) - ray_lane<L, 0>(s)) / vs;
    if (j0 == 0) *g0 = ga;
    if (j0 == 2) *g1 = ga;
    if (j0 == 4) *g2 = ga;
    if constexpr (L == 4) {
      valid = valid && ray_lane<L, 2>(oku) && ray_lane<L, 3>(oku);
      const float gb = (ray_lane<L, 3>(s) - ray_lane<L, 2>(s)) / vs;
      if (j0 == 0) *g1 = gb;
    }
  }
  return valid;
}

// The ray parameters between which pixel (x, y) can meet an allocated block:
// the tile's camera-z range over dir_c.z, widened by 0.1 %.
__device__ __forceinline__ void ray_bounds(const RayConst& R, uint32_t x, uint32_t y, float dcz, float t_min,
                                           float t_max, float* t_lo, float* t_hi) {
  const uint32_t tile = (y >> 3) * R.tiles_x + (x >> 3);
  const float zmin = __uint_as_float(R.range[2 * tile]);
  const float zmax = __uint_as_float(R.range[2 * tile + 1]);
  *t_lo = fmaxf(t_min, 0.999f * (zmin / dcz));
  *t_hi = fminf(t_max, 1.001f * (zmax / dcz));
}

// March one pixel; returns the number of valid samples taken.
template <bool kWide, int L>
__device__ __forceinline__ uint32_t cast_pixel(const View& V, const RayConst& R, uint32_t x, uint32_t y,
                               WaveTable* table, float* res_d, f3* res_v, f3* res_n) {
  uint32_t nsamp = 0;
  float out_d = -INFINITY;
  f3 out_v = mk3(-INFINITY, -INFINITY, -INFINITY);
  f3 out_n = mk3(-INFINITY, -INFINITY, -INFINITY);

  const f3 dir_c = normalize(reproject(R.cam, x, y, 1.0f));
  const float t_min = R.min_depth / dir_c.z;
  const float t_max = R.max_depth / dir_c.z;
  const f3 o = xform(R.wTc, mk3(0.0f, 0.0f, 0.0f));
  const f3 dir = normalize(xform_dir(R.wTc, dir_c));

  Hit hit;
  float t_lo, t_hi;
  ray_bounds(R, x, y, dir_c.z, t_min, t_max, &t_lo, &t_hi);
  Octant oc = empty_octant();
  bool found;
  if constexpr (L == 1)
    found = find_surface<kWide>(V, R, o, dir, t_min, t_max, t_lo, t_hi, table, oc, &hit, &nsamp);
  else
    found = find_surface_split<kWide, L>(V, R, o, dir, t_min, t_max, t_lo, t_hi, table, oc, &hit, &nsamp);
  if (found) {
    const float m = hit.m;
    const float d = m * dir_c.z;
    out_d = d;
    out_v = reproject(R.cam, x, y, d);
    if (R.enable_gradients) {
      const f3 iso = mk3(o.x + m * dir.x, o.y + m * dir.y, o.z + m * dir.z);
      f3 grad;
      bool valid;
      if constexpr (L == 1)
        valid = gradient_samples<kWide>(V, table, oc, iso, R.inv_vs, &grad.x, &grad.y, &grad.z);
      else
        valid = gradient_samples_split<kWide, L>(V, table, oc, iso, R.inv_vs, &grad.x, &grad.y, &grad.z);
      const float l2 = length(grad);
      f3 nw = (l2 > 0.0f && valid) ? grad / l2 : mk3(0.0f, 0.0f, 0.0f);
      nw = -nw;
      out_n = xform_dir(R.cTw, nw);
    }
  }
  *res_d = out_d;
  *res_v = out_v;
  *res_n = out_n;
  return nsamp;
}

// ------------------------------------------------------------ adjoint
// GetSpatialValue's SDF (same corners, weights and summation order as
// point_sample, so the value is bit-identical) with the spatial gradient of the
// trilinear interpolant: each ratio frac(pos / vs) moves at 1 / vs.
template <bool kWide>
__device__ __forceinline__ bool ray_sdf_grad(const View& V, WaveTable* t, Octant& oc, f3 pos, float inv_vs, float* val,
                                             f3* grad) {
  const float vs = V.geo.voxel_size;
  const float rx = ray_ratio(pos.x, vs, inv_vs), ry = ray_ratio(pos.y, vs, inv_vs), rz = ray_ratio(pos.z, vs, inv_vs);
  ray_offset<kWide> off[8];
  if (!cell_corners<kWide>(V, t, oc, ray_cell(pos, vs, inv_vs), off)) return false;
  float v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = field_at<kWide>(V.sdf, off[i]);
  float sdf = 0.0f, gx = 0.0f, gy = 0.0f, gz = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int mx = (i >> 2) & 1, my = (i >> 1) & 1, mz = i & 1;
    const float c = v[i];
    const float wx = mx ? rx : 1.0f - rx, wy = my ? ry : 1.0f - ry, wz = mz ? rz : 1.0f - rz;
    sdf += wx * wy * wz * c;
    gx += (mx ? c : -c) * wy * wz;
    gy += (my ? c : -c) * wx * wz;
    gz += (mz ? c : -c) * wx * wy;
  }
  *val = sdf;
  *grad = mk3(gx / vs, gy / vs, gz / vs);
  return true;
}

// dL/dsdf of a wave's 64 pixels, summed in LDS before it goes to memory: the
// pixels of a tile and the five samples of each share most of their corner
// voxels (24 or so contributions a voxel at 640 x 480 over 1 cm voxels), and
// atomics on one address run one after another.  An open-addressed table of
// voxel offsets; a contribution that finds no place within kGradProbes slots
// goes to memory by itself.  640 x 480, 1 cm room: the pass takes 234 us so,
// 543 us with an atomic per contribution (157 us without dL/dsdf).
constexpr uint32_t kGradSlotsLds = 1024;
constexpr int kGradProbes = 8;
template <bool kWide>
struct GradTable {
  using key_t = typename std::conditional<kWide, unsigned long long, unsigned int>::type;
  key_t key[kGradSlotsLds];
  float val[kGradSlotsLds];
};
template <bool kWide>
__device__ __forceinline__ void grad_table_init(GradTable<kWide>& g) {
  for (uint32_t i = threadIdx.x; i < kGradSlotsLds; i += 64u) {
    g.key[i] = ~typename GradTable<kWide>::key_t(0);
    g.val[i] = 0.0f;
  }
  __syncthreads();
}
template <bool kWide>
__device__ __forceinline__ float* grad_at(float* grad_sdf, ray_offset<kWide> off) {
  return reinterpret_cast<float*>(reinterpret_cast<char*>(grad_sdf) + off);
}
template <bool kWide>
__device__ __forceinline__ void grad_add(GradTable<kWide>& g, float* grad_sdf, ray_offset<kWide> off, float x) {
  using key_t = typename GradTable<kWide>::key_t;
  uint32_t h = ((uint32_t)(off >> 2) * 2654435761u) >> 22;
  static_assert(kGradSlotsLds == 1u << 10, "hash");
  for (int k = 0; k < kGradProbes; ++k) {
    const key_t old = atomicCAS(&g.key[h], ~key_t(0), (key_t)off);
    if (old == ~key_t(0) || old == (key_t)off) {
      atomicAdd(&g.val[h], x);
      return;
    }
    h = (h + 1) & (kGradSlotsLds - 1);
  }
  atomicAdd(grad_at<kWide>(grad_sdf, off), x);
}
template <bool kWide>
__device__ __forceinline__ void grad_table_flush(GradTable<kWide>& g, float* grad_sdf) {
  __syncthreads();
  for (uint32_t i = threadIdx.x; i < kGradSlotsLds; i += 64u) {
    const auto k = g.key[i];
    if (k != ~typename GradTable<kWide>::key_t(0)) atomicAdd(grad_at<kWide>(grad_sdf, (ray_offset<kWide>)k), g.val[i]);
  }
}

// Adds coef * (trilinear weight of each corner) to the corners' gradient, for
// a sample that the forward pass accepted (all its blocks exist).
template <bool kWide>
__device__ __forceinline__ void scatter_sdf(const View& V, WaveTable* t, Octant& oc, f3 pos, float inv_vs, float coef,
                                            GradTable<kWide>& g, float* __restrict__ grad_sdf) {
  const float vs = V.geo.voxel_size;
  const float rx = ray_ratio(pos.x, vs, inv_vs), ry = ray_ratio(pos.y, vs, inv_vs), rz = ray_ratio(pos.z, vs, inv_vs);
  ray_offset<kWide> off[8];
  if (!cell_corners<kWide>(V, t, oc, ray_cell(pos, vs, inv_vs), off)) return;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int mx = (i >> 2) & 1, my = (i >> 1) & 1, mz = i & 1;
    const float w = (mx ? rx : 1.0f - rx) * (my ? ry : 1.0f - ry) * (mz ? rz : 1.0f - rz);
    grad_add<kWide>(g, grad_sdf, off[i], coef * w);
  }
}

// Tangents: d/d(omega_xyz, upsilon_xyz) of a pose perturbation
// wTc <- exp(xi^) wTc (a world point x moves by omega x x + upsilon), then
// d/d(eps_0..eps_4), a perturbation of the value of each of the five SDF
// evaluations the depth depends on (the two bracketing samples and the
// three regula-falsi points).
constexpr int kTan = 11;

__device__ __forceinline__ void sample_tangent(f3 x, f3 g, int slot, float* t) {
  const f3 c = mk3(x.y * g.z - x.z * g.y, x.z * g.x - x.x * g.z, x.x * g.y - x.y * g.x);  // x cross g
  t[0] = c.x; t[1] = c.y; t[2] = c.z;
  t[3] = g.x; t[4] = g.y; t[5] = g.z;
#pragma unroll
  for (int k = 6; k < kTan; ++k) t[k] = k == slot ? 1.0f : 0.0f;
}

// Differentiates the rendered depth of one pixel: recomputes the march
// (same decisions as the forward pass), then carries tangents through the
// three regula-falsi steps.  Returns false when the pixel has no hit.
template <bool kWide>
__device__ __forceinline__ bool depth_tangent(const View& V, const RayConst& R, uint32_t x, uint32_t y,
                                              WaveTable* table, Octant& oc, float* depth, float* dd, f3* X) {
  const f3 dir_c = normalize(reproject(R.cam, x, y, 1.0f));
  const float t_min = R.min_depth / dir_c.z;
  const float t_max = R.max_depth / dir_c.z;
  const f3 o = xform(R.wTc, mk3(0.0f, 0.0f, 0.0f));
  const f3 dir = normalize(xform_dir(R.wTc, dir_c));
  Hit hit;
  uint32_t ns = 0;
  float t_lo, t_hi;
  ray_bounds(R, x, y, dir_c.z, t_min, t_max, &t_lo, &t_hi);
  if (!find_surface<kWide>(V, R, o, dir, t_min, t_max, t_lo, t_hi, table, oc, &hit, &ns)) return false;
  float l = hit.tp, r = hit.tk, ls, rs;
  float dl[kTan], dr[kTan], dls[kTan], drs[kTan], dm[kTan];
  f3 g;
  X[0] = mk3(o.x + l * dir.x, o.y + l * dir.y, o.z + l * dir.z);
  X[1] = mk3(o.x + r * dir.x, o.y + r * dir.y, o.z + r * dir.z);
  ray_sdf_grad<kWide>(V, table, oc, X[0], R.inv_vs, &ls, &g);
  sample_tangent(X[0], g, 6, dls);
  ray_sdf_grad<kWide>(V, table, oc, X[1], R.inv_vs, &rs, &g);
  sample_tangent(X[1], g, 7, drs);
#pragma unroll
  for (int k = 0; k < kTan; ++k) dl[k] = dr[k] = 0.0f;
  float m = 0.0f;
#pragma unroll 1
  for (int j = 0; j < 3; ++j) {
    const float D = ls - rs;
    const float q = ls / D;
    m = l + (ls / (ls - rs)) * (r - l);
    const float inv_d2 = 1.0f / (D * D);
#pragma unroll
    for (int k = 0; k < kTan; ++k) {
      const float dq = (ls * drs[k] - rs * dls[k]) * inv_d2;
      dm[k] = dl[k] + dq * (r - l) + q * (dr[k] - dl[k]);
    }
    const f3 xm = mk3(o.x + m * dir.x, o.y + m * dir.y, o.z + m * dir.z);
#pragma unroll
    for (int q = 0; q < 3; ++q)
      if (j == q) X[2 + q] = xm;
    float ms;
    ray_sdf_grad<kWide>(V, table, oc, xm, R.inv_vs, &ms, &g);
    float dms[kTan];
    sample_tangent(xm, g, 8 + j, dms);
    const float gd = g.x * dir.x + g.y * dir.y + g.z * dir.z;
#pragma unroll
    for (int k = 0; k < kTan; ++k) dms[k] += gd * dm[k];
    if (ls * ms > 0.0f) {
      l = m;
      ls = ms;
#pragma unroll
      for (int k = 0; k < kTan; ++k) { dl[k] = dm[k]; dls[k] = dms[k]; }
    } else {
      r = m;
      rs = ms;
#pragma unroll
      for (int k = 0; k < kTan; ++k) { dr[k] = dm[k]; drs[k] = dms[k]; }
    }
  }
  *depth = m * dir_c.z;
#pragma unroll
  for (int k = 0; k < kTan; ++k) dd[k] = dm[k] * dir_c.z;
  return true;
}

// Per pixel: residual r = depth - observed depth (pixels with a hit, a
// finite positive observation and |r| <= max_residual; the others with a
// hit and an observation are counted as gated out), J = d depth / d xi.
// Every pixel with a finite positive observation is counted as observed,
// hit or not, so a caller can charge the pixels a pose loses.
// Pixels whose depth moves faster than max_slope times a camera translation
// (|d depth / d upsilon| on some axis; rays close to grazing the surface)
// are left out altogether.  Per workgroup (one
// wave): FP64 sums of r^2 / 2, r J, J J^T (upper triangle) and the pixel
// count, reduced in a fixed order by raycast_grad_reduce_kernel.  With
// grad_sdf, r * d depth / d sdf is scattered onto the voxels.
template <bool kWide>
__global__ __launch_bounds__(64) void raycast_backward_kernel(View V, RayConst R,
                                                              const float* __restrict__ obs,
                                                              float* __restrict__ grad_sdf,
                                                              double* __restrict__ partials,
                                                              float max_residual, float max_slope) {
  __shared__ WaveTable table;
  __shared__ GradTable<kWide> gtab;
  if (grad_sdf) grad_table_init<kWide>(gtab);
  wave_table_init(&table);
  const uint32_t x = blockIdx.x * 8 + (threadIdx.x & 7);
  const uint32_t y = blockIdx.y * 8 + (threadIdx.x >> 3);
  double acc[kGradSlots];
#pragma unroll
  for (int k = 0; k < kGradSlots; ++k) acc[k] = 0.0;
  if (x < R.cam.width && y < R.cam.height) {
    const float od = obs[y * R.cam.width + x];
    Octant oc = empty_octant();
    float d, dd[kTan];
    f3 X[5];
    acc[30] = od > 0.0f && od < INFINITY ? 1.0 : 0.0;
    if (od > 0.0f && od < INFINITY && depth_tangent<kWide>(V, R, x, y, &table, oc, &d, dd, X) &&
        fmaxf(fabsf(dd[3]), fmaxf(fabsf(dd[4]), fabsf(dd[5]))) <= max_slope) {
      const float res = d - od;
      if (!(fabsf(res) <= max_residual)) {
        acc[29] = 1.0;
      } else {
        acc[0] = 0.5 * (double)res * (double)res;
#pragma unroll
        for (int k = 0; k < 6; ++k) acc[1 + k] = (double)res * (double)dd[k];
        int t = 7;
#pragma unroll
        for (int i = 0; i < 6; ++i)
#pragma unroll
          for (int j = i; j < 6; ++j) acc[t++] = (double)dd[i] * (double)dd[j];
        acc[28] = 1.0;
        if (grad_sdf)
#pragma unroll 1
          for (int e = 0; e < 5; ++e) {
            f3 x = X[0];
            float c = dd[6];
#pragma unroll
            for (int q = 1; q < 5; ++q)
              if (e == q) {
                x = X[q];
                c = dd[6 + q];
              }
            scatter_sdf<kWide>(V, &table, oc, x, R.inv_vs, res * c, gtab, grad_sdf);
          }
      }
    }
  }
  if (grad_sdf) grad_table_flush<kWide>(gtab, grad_sdf);
#pragma unroll
  for (int k = 0; k < kGradSlots; ++k) {
    double v = acc[k];
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    acc[k] = v;
  }
  if (threadIdx.x == 0) {
    const size_t wg = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
#pragma unroll
    for (int k = 0; k < kGradSlots; ++k) partials[wg * kGradSlots + k] = acc[k];
  }
}

// Sums n rows of `slots` (<= 32) FP64 partials column by column into out, in
// an order fixed by n alone (deterministic).  A workgroup sums kReduceRows
// rows, eight of them at a time (32 lanes a row), and leaves the sum in the
// first of its rows; the workgroup that finishes last adds those up the same
// way.  A lane's chain is then kReduceRows / 8 loads rather than n: a lane
// per column walking every row took 1135 us for a 640 x 480 image's 4800 rows
// against 9 us here.  Up to kReduceOneRows rows go to one workgroup of 32 rows at
// a time, whose two round trips are less than the fence, the count and the
// second stage (a localiser's step with its 300 rows: 10.0 us by eights, 7.2 us).
constexpr uint32_t kReduceRows = 64;
constexpr uint32_t kReduceOneRows = 512;
template <uint32_t kGroups>
__device__ __forceinline__ double reduce_rows(const double* rows, uint32_t n, size_t stride,
                                              uint32_t slots, double (*red)[32]) {
  const uint32_t k = threadIdx.x & 31, g = threadIdx.x >> 5;
  double s = 0.0;
  if (k < slots)
#pragma unroll 8
    for (uint32_t i = g; i < n; i += kGroups) s += rows[i * stride + k];
  red[g][k] = s;
  __syncthreads();
  double all = 0.0;
#pragma unroll
  for (uint32_t j = 0; j < kGroups; ++j) all += red[j][k];
  __syncthreads();
  return all;
}
// (-> the whole sum in the first `slots` lanes of one workgroup, true there;
// kOne: the only workgroup, of 1024 lanes)
template <bool kOne>
__device__ __forceinline__ bool slot_reduce(double* partials, uint32_t n, uint32_t slots, uint32_t* done, double* sum) {
  constexpr uint32_t kGroups = kOne ? 32 : 8;
  __shared__ double red[kGroups][32];
  if (kOne) {
    *sum = reduce_rows<kGroups>(partials, n, slots, slots, red);
    return true;
  }
  __shared__ bool last;
  const uint32_t r0 = blockIdx.x * kReduceRows;
  double* const mine = partials + (size_t)r0 * slots;
  const double s = reduce_rows<kGroups>(mine, min(kReduceRows, n - r0), slots, slots, red);
  if (threadIdx.x < slots) mine[threadIdx.x] = s;
  __threadfence();  // the row before the count that announces it
  __syncthreads();
  if (threadIdx.x == 0) last = atomicAdd(done, 1u) == gridDim.x - 1;
  __syncthreads();
  if (!last) return false;
  __threadfence();  // the other workgroups' rows after their counts
  *sum = reduce_rows<kGroups>(partials, gridDim.x, (size_t)kReduceRows * slots, slots, red);
  if (threadIdx.x == 0) *done = 0u;  // for the next call
  return true;
}
inline uint32_t reduce_groups(uint32_t n) { return n <= kReduceOneRows ? 1 : (n + kReduceRows - 1) / kReduceRows; }
inline uint32_t reduce_lanes(uint32_t n) { return n <= kReduceOneRows ? 1024 : 256; }
template <bool kOne>
__global__ __launch_bounds__(kOne ? 1024 : 256) void slot_reduce_kernel(double* partials, uint32_t n, uint32_t slots,
                                                                         uint32_t* done, double* __restrict__ out) {
  double a;
  if (slot_reduce<kOne>(partials, n, slots, done, &a) && threadIdx.x < slots) out[threadIdx.x] = a;
}
void launch_slot_reduce(double* partials, uint32_t n, uint32_t slots, uint32_t* done, double* out, hipStream_t s) {
  const auto k = n <= kReduceOneRows ? slot_reduce_kernel<true> : slot_reduce_kernel<false>;
  k<<<reduce_groups(n), reduce_lanes(n), 0, s>>>(partials, n, slots, done, out);
}

// Lanes a ray: an image of few pixels leaves the chip nearly empty, a wave a
// SIMD at 333 x 251, and each wave's time is the latency of its rays' samples
// in a row; four (two) lanes a ray then take a quarter (half) of the rounds.
// Two as long as their waves fit the chip in one round; past that the extra lanes
// only add work.  Four an eighth past it, the first waves being done by then.
// Measured, whole call, us with 1 / 2 / 4 lanes (5 mm desk; 5 mm room; 2 cm room):
//   320 x 240    148 / 119 / 101    107 /  99 /  91    72 / 66 / 58
//   350 x 262    147 / 132 / 107    106 / 104 / 111    71 / 68 / 65  (just inside the four's line)
//   358 x 268    150 / 129 / 116    103 / 101 / 112    75 / 73 / 70  (just past it)
//   400 x 300    137 / 131 / 120    103 / 106 / 121    75 / 75 / 77
//   462 x 346    141 / 141 / 136    109 / 115 / 135    77 / 82 / 85  (just inside the two's)
//   480 x 360    140 / 144 / 138    113 / 136 / 149    76 / 88 / 92
// so that either line lies where the scenes' sums are about even.  beside: a
// meshing pass runs on the chip at the same time.  Two lanes then bring nothing
// (replayed frames: 2 cm room 400 x 300 183 us with one, 187 with two, 1 cm 249
// and 267; two 4 cm rooms of 320 x 240 134 and 144; 5 mm desk 400 x 300 293 and
// 312), and four still do where the march is the longer branch (2 cm room 160 x
// 120 178 and 130, 320 x 240 175 and 162, two of 237 x 177 208 and 180, four of
// 175 x 131 245 and 224) but cost time where the meshing pass is (5 mm desk
// 320 x 240 273 and 311; 1 cm room even, 241 and 237).
inline int ray_lanes(uint64_t pixels, int cus, bool beside) {
  const uint64_t waves = (pixels + 63) / 64, room = (uint64_t)kRayWavesPerSimd * 4 * (uint64_t)cus;
  return 4 * waves <= room + room / 8 ? 4 : (!beside && 2 * waves <= room ? 2 : 1);
}

// ------------------------------------------------------------ localisation
// PointToSurfaceKernel (localizing/point_to_psdf.cu:19-82): the odd pixels
// (both coordinates odd), 8 x 8 of them per workgroup, i.e.
// a 16 x 16 pixel tile as in the reference.  A depth that is -inf, 0 or at
// least sdf_upper_bound is skipped; the world point wTc * p, the SDF
// (GetSpatialValue) and its central difference at +-vs/2
// (GetSpatialSDFGradient, spatial_query.h:71-97) are the reference's FP32
// expressions.  J = (g, p x g) for the tangent (translation, rotation);
// `corrected` = 0 keeps the reference's g.x in J's third entry (:69-74).
// The per-pixel products J J^T, d J and d^2 are FP32, as the reference's
// mat6x6 arithmetic; they are summed in FP64 per wave and then per
// workgroup in a fixed order instead of float atomics.  Slots: A's upper
// triangle (21), b (6), err, count.
//
// L lanes a point (1 or 4; 64 L lanes a workgroup): a tracked frame's points are
// a wave or two a SIMD, and the pass then lasts as long as its seven samples in
// a row; four lanes take the gradient's six in two rounds, and add up eight
// slots each.  320 x 240 over a 2 cm room: 14 us with one, 10.3 with four.
template <bool kWide, int L>
__global__ __launch_bounds__(64 * L) void point_to_psdf_kernel(View V, M4 T0, float inv_vs, int corrected,
                                                               double* __restrict__ partials, LocalizeStep step) {
  if (step.st && !step.fresh && step.st->done) return;
  __shared__ WaveTable table;
  __shared__ double part[L][32];
  wave_table_init(&table);
  const uint32_t point = threadIdx.x / L;
  const uint32_t x = 2 * (blockIdx.x * 8 + (point & 7)) + 1;
  const uint32_t y = 2 * (blockIdx.y * 8 + (point >> 3)) + 1;
  M4 wTc = T0;
  if (step.st && !step.fresh)
#pragma unroll
    for (int k = 0; k < 16; ++k) wTc.m[k] = step.st->wTc[k];
  double acc[32];
#pragma unroll
  for (int k = 0; k < 32; ++k) acc[k] = 0.0;
  if (x < V.cam.width && y < V.cam.height) {
    const float depth = V.depth[(size_t)y * V.cam.width + x];
    if (!(depth == -INFINITY || depth == 0.0f || depth >= V.geo.sdf_upper_bound)) {
      const f3 pw = xform(wTc, reproject(V.cam, x, y, depth));
      Octant oc = empty_octant();
      float d;
      if (point_sample<kWide>(V, &table, oc, pw, inv_vs, &d)) {
        f3 g;
        bool valid;
        if constexpr (L == 1)
          valid = gradient_samples<kWide>(V, &table, oc, pw, inv_vs, &g.x, &g.y, &g.z);
        else
          valid = gradient_samples_split<kWide, L>(V, &table, oc, pw, inv_vs, &g.x, &g.y, &g.z);
        if (valid) {
          const float J[6] = {g.x, g.y, corrected ? g.z : g.x,
                              -g.y * pw.z + g.z * pw.y,
                              -g.z * pw.x + g.x * pw.z,
                              -g.x * pw.y + g.y * pw.x};
          int t = 0;
#pragma unroll
          for (int i = 0; i < 6; ++i)
#pragma unroll
            for (int j = i; j < 6; ++j) acc[t++] = (double)(J[i] * J[j]);
#pragma unroll
          for (int i = 0; i < 6; ++i) acc[21 + i] = (double)(d * J[i]);
          acc[27] = (double)(d * d);
          acc[28] = 1.0;
        }
      }
    }
  }
  // lane q of a point adds up slots [32 / L * q, 32 / L * (q + 1))
  constexpr int kOwn = 32 / L;
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = lane & (L - 1);
#pragma unroll
  for (int k = 0; k < (kOwn < kP2SSlots ? kOwn : kP2SSlots); ++k) {
    double v = acc[k];
#pragma unroll
    for (int j = 1; j < L; ++j) v = q == (uint32_t)j ? acc[kOwn * j + k] : v;
    for (int off = 32; off >= L; off >>= 1) v += __shfl_xor(v, off);
    if (lane < L) part[wave][kOwn * q + k] = v;
  }
  __syncthreads();
  if (threadIdx.x < kP2SSlots) {
    const size_t wg = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
    double s = part[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < L; ++w) s += part[w][threadIdx.x];
    partials[wg * kP2SSlots + threadIdx.x] = s;
  }
}

// SolveAndConvertDeltaXi (main_engine.cc:28-54) on the sums of one step, by one
// wave: (A + lambda I) dxi = -b, dT = exp(dxi) with dxi = (translation,
// rotation), wTc <- dT wTc.  Gaussian elimination with partial pivoting, an
// entry a lane; false if no point was in sight or the matrix is singular.
__device__ __forceinline__ bool localize_solve(const double* sums, double lambda, float* wTc) {
  __shared__ double A[6][8], E[16];
  const uint32_t lane = threadIdx.x, r = lane / 7, j = lane % 7;
  auto wave_sync = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
  if (sums[28] < 1.0) return false;
  if (r < 6) {
    if (j < 6) {
      const uint32_t lo = min(r, j), hi = max(r, j);
      const double h = sums[lo * 6 - lo * (lo - 1) / 2 + (hi - lo)] + (r == j ? lambda : 0.0);
      A[r][j] = h + (r == j ? 0.0 * h : 0.0);  // an infinite diagonal is singular
    } else {
      A[r][6] = -sums[21 + r];
    }
  }
  wave_sync();
  for (uint32_t c = 0; c < 6; ++c) {
    uint32_t piv = c;
    for (uint32_t i = c + 1; i < 6; ++i)
      if (fabs(A[i][c]) > fabs(A[piv][c])) piv = i;
    if (!(fabs(A[piv][c]) > 0.0)) return false;
    if (lane < 7) {
      const double a = A[c][lane], b = A[piv][lane];
      A[c][lane] = b;
      A[piv][lane] = a;
    }
    wave_sync();
    if (r > c && r < 6 && j >= c) {
      const double f = A[r][c] / A[c][c];
      const double v = A[r][j] - f * A[c][j];
      wave_sync();
      A[r][j] = v;
    }
    wave_sync();
  }
  double x[6];
#pragma unroll
  for (int i = 5; i >= 0; --i) {
    double s = A[i][6];
#pragma unroll
    for (int k = i + 1; k < 6; ++k) s -= A[i][k] * x[k];
    x[i] = s / A[i][i];
  }
  const double xi[6] = {x[3], x[4], x[5], x[0], x[1], x[2]};
  double e[16];
  se3_exp(xi, e);
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < 16; ++k) E[k] = e[k];
  wave_sync();
  if (lane < 16) {
    double s = 0.0;
#pragma unroll
    for (int k = 0; k < 4; ++k) s += E[4 * (lane >> 2) + k] * (double)wTc[4 * k + (lane & 3)];
    wave_sync();
    wTc[lane] = (float)s;
  }
  return true;
}
// The sums of a step and the step itself, by the workgroup that finishes them,
// so that the steps of a call follow each other without the host: 20 of them at
// 320 x 240 took 810 us with a copy, a wait and a launch from the host between
// two (17 us each), 417 us so.
template <bool kOne>
__global__ __launch_bounds__(kOne ? 1024 : 256) void localize_step_kernel(double* partials, uint32_t n, uint32_t* done, M4 T0,
                                                            LocalizeStep step) {
  LocalizeState* const st = step.st;
  if (!step.fresh && st->done) return;
  __shared__ double sums[32];
  __shared__ float wTc[16];
  double a;
  if (!slot_reduce<kOne>(partials, n, kP2SSlots, done, &a)) return;
  if (threadIdx.x < kP2SSlots) sums[threadIdx.x] = a;
  if (threadIdx.x < 16) wTc[threadIdx.x] = step.fresh ? T0.m[threadIdx.x] : st->wTc[threadIdx.x];
  __syncthreads();
  if (threadIdx.x >= 64) return;
  const bool ok = localize_solve(sums, step.lambda, wTc);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  if (threadIdx.x < 16) st->wTc[threadIdx.x] = wTc[threadIdx.x];
  if (threadIdx.x == 0) {
    st->err[step.slot] = sums[27];
    st->count[step.slot] = (uint32_t)sums[28];
    st->done = ok ? 0u : 1u;
    st->steps = step.slot + (ok ? 1u : 0u);
  }
}

uint32_t point_to_psdf_partials(const View& V) {
  return ((V.cam.width / 2 + 7) / 8) * ((V.cam.height / 2 + 7) / 8);
}

void launch_point_to_psdf(const View& V, const M4& wTc, int corrected, double* partials, double* out,
                          const LocalizeStep& step, hipStream_t s, int cus) {
  const dim3 grid((V.cam.width / 2 + 7) / 8, (V.cam.height / 2 + 7) / 8);
  const bool wide = V.capacity > kNarrowCapacity;
  // The march's line holds here too (20 steps in us, one / four lanes: 2 cm room
  // 320 x 240 543 / 396, 672 x 504 just inside it 630 / 596, 720 x 540 just past it
  // 645 / 623, 800 x 600 679 / 679, 1200 x 900 992 / 997; 5 mm desk 584 / 415, 698 /
  // 639, 741 / 690, 766 / 741, 1048 / 1148).
  const int lanes = !wide && ray_lanes((uint64_t)grid.x * grid.y * 64, cus, false) == 4 ? 4 : 1;
  const auto k = wide ? point_to_psdf_kernel<true, 1> : (lanes == 4 ? point_to_psdf_kernel<false, 4> : point_to_psdf_kernel<false, 1>);
  k<<<grid, 64 * lanes, 0, s>>>(V, wTc, 1.0f / V.geo.voxel_size, corrected, partials, step);
  const uint32_t n = grid.x * grid.y;
  const auto finish = n <= kReduceOneRows ? localize_step_kernel<true> : localize_step_kernel<false>;
  if (step.st)
    finish<<<reduce_groups(n), reduce_lanes(n), 0, s>>>(partials, n, &V.ctr->reduce_done, wTc, step);
  else
    launch_slot_reduce(partials, n, kP2SSlots, &V.ctr->reduce_done, out, s);
}

__device__ __forceinline__ const RayConst& ray_of(const One&, uint32_t, const RayConst& r) { return r; }
__device__ __forceinline__ const RayConst& ray_of(const Many& m, uint32_t s, const RayConst&) {
  return m.f[s].ray;
}

// Scene = blockIdx.z; a batch's outputs are scene-major (W*H per scene).
// At most 96 registers: five waves per SIMD hold a 640x480 frame's 4800
// tiles at once on 256 CUs (four would leave a partial second round).
// tw: log2 of the tile's width in pixels (the tile has 64; every shape gives
// the same per-pixel results, the autotuner picks the fastest).
// L lanes a ray (64 / L pixels a wave): see ray_lanes.
template <class Src, bool kWide, int L>
__global__ __launch_bounds__(64, kRayWavesPerSimd) void raycast_kernel(Src src_, const SceneFrame* __restrict__ tab, RayConst R1, int tw, float* __restrict__ depth_out,
                                                     float* __restrict__ vertex_out,
                                                     float* __restrict__ normal_out) {
  const Src src = with_table(src_, tab);
  __shared__ WaveTable table;
  wave_table_init(&table);
  const uint32_t scene = blockIdx.z;
  // copies, not references into the frame table: read once, and not
  // reloaded after the stores of the march (LDS table, outputs)
  const View V = src.view(scene);
  const RayConst R = ray_of(src, scene, R1);
  if (R.boost) __builtin_amdgcn_s_setprio(2);
  constexpr int kLog = L == 4 ? 2 : (L == 2 ? 1 : 0);
  const uint32_t ray = threadIdx.x >> kLog;
  const uint32_t x = (blockIdx.x << tw) + (ray & ((1u << tw) - 1u));
  const uint32_t y = (blockIdx.y << (6 - kLog - tw)) + (ray >> tw);
  uint32_t ns = 0;
  if (x < R.cam.width && y < R.cam.height) {
    const size_t pix = (size_t)scene * R.cam.width * R.cam.height + y * R.cam.width + x;
    float d;
    f3 vv, nn;
    ns = cast_pixel<kWide, L>(V, R, x, y, &table, &d, &vv, &nn);
    if (L == 1 || (threadIdx.x & (L - 1)) == 0) {
      if (depth_out) depth_out[pix] = d;
      if (vertex_out) {
        vertex_out[3 * pix + 0] = vv.x;
        vertex_out[3 * pix + 1] = vv.y;
        vertex_out[3 * pix + 2] = vv.z;
      }
      if (normal_out) {
        normal_out[3 * pix + 0] = nn.x;
        normal_out[3 * pix + 1] = nn.y;
        normal_out[3 * pix + 2] = nn.z;
      }
    } else {
      ns = 0;  // the ray's first lane has counted its samples
    }
  }
  wave_add_u64(&work_stripe(V.ctr).ray_samples, ns);
}

// ------------------------------------------------------------ block ranges
// Every valid sample lies in the box of the block holding its lowest
// trilinear corner, [8b, 8b + 8] voxels per axis; with one more voxel on each
// side the box bounds it beyond any rounding.  The part of each allocated
// block's box at z >= min_depth / 2 (every sample's z is at least min_depth) is
// projected and its camera-z extent merged into the 8 x 8 pixel tiles its
// projected rectangle, widened by a pixel, overlaps.  A ray then meets no valid
// sample outside its tile's [zmin, zmax].  A box that reaches through the plane
// z = min_depth / 2 is clipped there: a camera inside a room nearly always has
// such blocks beside it (a wall's, at the camera's own depth), and switching the
// ranges off for them (a pose that is not rigid has none: RayConst::whole) made every ray walk up to its surface from min_depth (5 mm
// room at 1237 x 931: the march 854 us, 499 us with the ranges).
//
// Before it, one launch clears the tile ranges (its first kClearGroups
// workgroups) and fills the blocks' rows of V.oct: the pool indices of the
// eight blocks b + {0, 1}^3 of every allocated block b, eight lanes a block.  A
// march sample then has its corners' blocks from two 16-byte loads instead of
// up to seven lookups that a wave's lanes ran one after another.
constexpr uint32_t kClearGroups = 8;
template <class Src>
__global__ __launch_bounds__(256) void ray_prepare_kernel(Src src_, const SceneFrame* __restrict__ tab, RayConst R1) {
  const Src src = with_table(src_, tab);
  if (blockIdx.x < kClearGroups) {
    const RayConst& R = ray_of(src, blockIdx.y, R1);
    if (!R.range) return;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < 2 * R.tiles; i += kClearGroups * blockDim.x)
      R.range[i] = ((i & 1u) != 0u) == (R.whole != 0) ? 0x7f800000u : 0u;  // zmin +inf, zmax 0; whole: 0, +inf
    return;
  }
  const View V = src.view(blockIdx.y);
  const size_t n = (size_t)V.ctr->block_hwm * 8;
  for (size_t i = (size_t)(blockIdx.x - kClearGroups) * blockDim.x + threadIdx.x; i < n;
       i += (size_t)(gridDim.x - kClearGroups) * blockDim.x) {
    const uint32_t p = (uint32_t)(i >> 3), e = (uint32_t)i & 7u;
    const uint64_t key = V.block_keys[p];
    if (key == kEmptyKey) continue;
    const i3 b = unpack_key(key);
    V.oct[i] = e == 0 ? (int32_t)p
                      : hash_find_eager(V, i3{b.x + (int)(e >> 2), b.y + (int)((e >> 1) & 1u), b.z + (int)(e & 1u)});
  }
}
template <class Src>
void launch_ray_prepare(Src src, const SceneFrame* tab, const RayConst& R, uint32_t nscenes, hipStream_t s) {
  ray_prepare_kernel<<<dim3(kClearGroups + (nscenes > 1 ? 64 : 1024), nscenes), 256, 0, s>>>(src, tab, R);
}

// The tiles that the part of block `key`'s box a ray can sample projects to,
// and its camera-z extent; false if there is none (a free slot, out of range,
// off the image).  Eight lanes a block, a corner each: a lane a block had its eight
// projections in a row, on a quarter of the chip at most, 10.7 us for the 5.8 k
// blocks of a 2 cm room at 320 x 240 (5.7 us so).
struct TileRect {
  int x0, x1, y0, y1;
  uint32_t zlo, zhi;
};
struct Extent {
  float lo, hi;
};
// (a value that is not a number counts as none)
__device__ __forceinline__ Extent eight_extent(float lo, float hi) {
  lo = fminf(lo, INFINITY);
  hi = fmaxf(hi, -INFINITY);
#pragma unroll
  for (int d = 1; d < 8; d <<= 1) {
    lo = fminf(lo, __shfl_xor(lo, d));
    hi = fmaxf(hi, __shfl_xor(hi, d));
  }
  return Extent{lo, hi};
}
__device__ __forceinline__ bool block_tiles(const RayConst& R, uint64_t key, float vs, TileRect* r) {
  const int c = (int)(threadIdx.x & 7u);
  const float zcut = 0.5f * R.min_depth;
  const i3 b = unpack_key(key);
  const float lo[3] = {(float)(8 * b.x - 1) * vs, (float)(8 * b.y - 1) * vs, (float)(8 * b.z - 1) * vs};
  const float hi[3] = {(float)(8 * b.x + 9) * vs, (float)(8 * b.y + 9) * vs, (float)(8 * b.z + 9) * vs};
  const f3 pc = xform(R.cTw, mk3((c & 1) ? hi[0] : lo[0], (c & 2) ? hi[1] : lo[1], (c & 4) ? hi[2] : lo[2]));
  const Extent z = eight_extent(pc.z, pc.z);
  float zmin = z.lo;
  const float zmax = z.hi;
  // no ray sample reaches it (the eight lanes agree)
  if (key == kEmptyKey || zmax < R.min_depth || zmin > R.max_depth) return false;
  float umin = INFINITY, umax = -INFINITY, vmin = INFINITY, vmax = -INFINITY;
  const bool before = !(pc.z >= zcut);
  if (!before) {
    umin = umax = R.cam.fx * pc.x / pc.z + R.cam.cx;
    vmin = vmax = R.cam.fy * pc.y / pc.z + R.cam.cy;
  }
  if ((__ballot(before) >> (threadIdx.x & 56u)) & 255u) {
    // the clipped box's other corners: where its twelve edges cross z = zcut
    zmin = zcut;
#pragma unroll 1
    for (int e = c; e < 12; e += 8) {
      // edge along axis e / 4 from the corner whose other two bits are e % 4
      const int ax = e >> 2, b0 = ax == 0 ? 2 : 1, b1 = ax == 2 ? 2 : 4;
      const int c0 = ((e & 1) ? b0 : 0) | ((e & 2) ? b1 : 0), c1 = c0 | (1 << ax);
      const f3 p0 = xform(R.cTw, mk3((c0 & 1) ? hi[0] : lo[0], (c0 & 2) ? hi[1] : lo[1], (c0 & 4) ? hi[2] : lo[2]));
      const f3 p1 = xform(R.cTw, mk3((c1 & 1) ? hi[0] : lo[0], (c1 & 2) ? hi[1] : lo[1], (c1 & 4) ? hi[2] : lo[2]));
      if ((p0.z >= zcut) == (p1.z >= zcut)) continue;
      const float s = (zcut - p0.z) / (p1.z - p0.z);
      const float u = R.cam.fx * (p0.x + s * (p1.x - p0.x)) / zcut + R.cam.cx;
      const float v = R.cam.fy * (p0.y + s * (p1.y - p0.y)) / zcut + R.cam.cy;
      umin = fminf(umin, u);
      umax = fmaxf(umax, u);
      vmin = fminf(vmin, v);
      vmax = fmaxf(vmax, v);
    }
  }
  const Extent ue = eight_extent(umin, umax), ve = eight_extent(vmin, vmax);
  umin = ue.lo;
  umax = ue.hi;
  vmin = ve.lo;
  vmax = ve.hi;
  const float W = (float)R.cam.width, H = (float)R.cam.height;
  if (!(umax >= -1.0f && umin <= W && vmax >= -1.0f && vmin <= H)) return false;  // off the image
  r->x0 = (int)fmaxf(floorf(umin) - 1.0f, 0.0f) >> 3;
  r->x1 = (int)fminf(ceilf(umax) + 1.0f, W - 1.0f) >> 3;
  r->y0 = (int)fmaxf(floorf(vmin) - 1.0f, 0.0f) >> 3;
  r->y1 = (int)fminf(ceilf(vmax) + 1.0f, H - 1.0f) >> 3;
  r->zlo = __float_as_uint(fmaxf(zmin, 0.0f));
  r->zhi = __float_as_uint(zmax);
  return true;
}
__device__ __forceinline__ void merge_tile(uint32_t* rng, uint32_t t, uint32_t zlo, uint32_t zhi) {
  atomicMin(&rng[2 * t], zlo);
  atomicMax(&rng[2 * t + 1], zhi);
}
// Tiles that a block's own lanes merge: a 16 cm block at a few metres covers at most
// 16 tiles of a 320 x 240 image.  With every rectangle left to its lane, a
// 2 cm probabilistic scan (outlier blocks in front of the camera) took 36-47 us
// a range pass at 333 x 251 (16 us so).
constexpr int kLaneTiles = 16;

// kLds: a workgroup first merges its blocks' ranges in an LDS copy of the
// tile table (up to kRangeLdsTiles tiles) and then sends each tile it
// touched to the global table with one atomic per bound, instead of one per
// block and tile.
constexpr uint32_t kRangeLdsTiles = 4800;  // 640 x 480 pixels
// Every workgroup sends its tiles once: twice as many of half the lanes took 10.2
// us for 31 k blocks at 640 x 480 (9.2 us so, 9.5 with half as many of 1024 lanes)
// and 31 us for 64 rooms (25 us, 26 us).
constexpr int kRangeLdsLanes = 512;
template <class Src, bool kLds>
__global__ __launch_bounds__(kLds ? kRangeLdsLanes : 256) void ray_range_kernel(Src src_, const SceneFrame* __restrict__ tab, RayConst R1) {
  const Src src = with_table(src_, tab);
  const uint32_t scene = blockIdx.y;
  const View& V = src.view(scene);
  const RayConst& R = ray_of(src, scene, R1);
  if (R.whole) return;
  const uint32_t n = V.ctr->block_hwm;
  const float vs = V.geo.voxel_size;
  __shared__ uint32_t lds_range[kLds ? 2 * kRangeLdsTiles : 1];
  uint32_t* const rng = kLds ? lds_range : R.range;
  if (kLds) {
    if (R.tiles > kRangeLdsTiles) return;  // not launched so
    for (uint32_t t = threadIdx.x; t < 2 * R.tiles; t += blockDim.x) lds_range[t] = (t & 1u) ? 0u : 0x7f800000u;
    __syncthreads();
  }
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t per = blockDim.x / 8, c = threadIdx.x & 7u;
  for (uint32_t p0 = blockIdx.x * per; p0 < n; p0 += gridDim.x * per) {
    const uint32_t p = p0 + (threadIdx.x >> 3);
    TileRect r;
    const bool on = block_tiles(R, p < n ? V.block_keys[p] : kEmptyKey, vs, &r);
    // a rectangle of a few tiles by its lanes, a larger one (a block close to
    // the camera: hundreds of tiles) by the whole wave, 8 x 8 tiles at a time
    const bool few = on && (r.x1 - r.x0 + 1) * (r.y1 - r.y0 + 1) <= kLaneTiles;
    if (few)
      for (int ty = r.y0 + (int)(c >> 2); ty <= r.y1; ty += 2)
        for (int tx = r.x0 + (int)(c & 3u); tx <= r.x1; tx += 4)
          merge_tile(rng, (uint32_t)ty * R.tiles_x + (uint32_t)tx, r.zlo, r.zhi);
    for (uint64_t big = __ballot(on && !few && c == 0); big; big &= big - 1) {
      const int l = __ffsll((unsigned long long)big) - 1;
      const int x0 = __builtin_amdgcn_readlane(r.x0, l), x1 = __builtin_amdgcn_readlane(r.x1, l);
      const int y0 = __builtin_amdgcn_readlane(r.y0, l), y1 = __builtin_amdgcn_readlane(r.y1, l);
      const uint32_t zlo = __builtin_amdgcn_readlane(r.zlo, l), zhi = __builtin_amdgcn_readlane(r.zhi, l);
      for (int ty = y0 + (int)(lane >> 3); ty <= y1; ty += 8)
        for (int tx = x0 + (int)(lane & 7u); tx <= x1; tx += 8)
          merge_tile(rng, (uint32_t)ty * R.tiles_x + (uint32_t)tx, zlo, zhi);
    }
  }
  if (kLds) {
    __syncthreads();
    for (uint32_t t = threadIdx.x; t < R.tiles; t += blockDim.x) {
      const uint32_t lo = lds_range[2 * t], hi = lds_range[2 * t + 1];
      if (lo != 0x7f800000u) atomicMin(&R.range[2 * t], lo);
      if (hi != 0u) atomicMax(&R.range[2 * t + 1], hi);
    }
  }
}

template <class Src>
void launch_ray_range(Src src, const SceneFrame* tab, const RayConst& R, uint32_t tiles, uint32_t nscenes,
                      hipStream_t s) {
  launch_ray_prepare(src, tab, R, nscenes, s);
  if (tiles <= kRangeLdsTiles) {
    ray_range_kernel<Src, true><<<dim3(nscenes > 1 ? 32 : 128, nscenes), kRangeLdsLanes, 0, s>>>(src, tab, R);
  } else {
    // the pool slots of a 118 k-block volume over the whole chip
    // (the projections are independent; 128 workgroups had left most CUs idle)
    ray_range_kernel<Src, false><<<dim3(nscenes > 1 ? 256 : 1024, nscenes), 256, 0, s>>>(src, tab, R);
  }
}

template <class Src>
void raycast_shaped(Src src, const SceneFrame* tab, const RayConst& p, uint32_t w, uint32_t h, uint32_t nscenes,
                    bool wide, bool marks, bool beside, int shape, int cus, float* depth, float* vertex,
                    float* normal, hipStream_t s) {
  // marks: the blocks of the samples are counted; several lanes a ray also
  // sample behind its crossing
  const int lanes = wide || marks || shape != 0 ? 1 : ray_lanes((uint64_t)w * h * nscenes, cus, beside);
  const int px = 64 / lanes;
  const int tw = lanes == 1 ? kRayTileWidths[shape] : (lanes == 2 ? 8 : 4), th = px / tw;
  const int log_tw = __builtin_ctz((unsigned)tw);
  const dim3 grid((w + tw - 1) / tw, (h + th - 1) / th, nscenes);
  const auto k = wide ? raycast_kernel<Src, true, 1>
                      : (lanes == 4 ? raycast_kernel<Src, false, 4>
                                    : (lanes == 2 ? raycast_kernel<Src, false, 2> : raycast_kernel<Src, false, 1>));
  k<<<grid, 64, 0, s>>>(src, tab, p, log_tw, depth, vertex, normal);
}

void launch_ray_rows(const View& V, hipStream_t s) { launch_ray_prepare(One{V}, nullptr, RayConst{}, 1, s); }

void launch_ray_range_one(const View& V, const RayConst& p, hipStream_t s) {
  launch_ray_range(One{V}, nullptr, p, p.tiles, 1, s);
}

void launch_raycast_march(const View& V, const RayConst& p, float* depth, float* vertex, float* normal,
                          hipStream_t s, int cus, int shape) {
  raycast_shaped(One{V}, nullptr, p, p.cam.width, p.cam.height, 1, V.capacity > kNarrowCapacity, V.ray_mark != nullptr,
                 false, shape, cus, depth, vertex, normal, s);
}

void launch_raycast(const View& V, const RayConst& p, float* depth, float* vertex, float* normal,
                    hipStream_t s, int cus, const KernelClock* kc, int shape) {
  tick(kc, s, "ray_range_kernel");
  launch_ray_range(One{V}, nullptr, p, p.tiles, 1, s);
  tick(kc, s, "raycast_kernel");
  raycast_shaped(One{V}, nullptr, p, p.cam.width, p.cam.height, 1, V.capacity > kNarrowCapacity, V.ray_mark != nullptr,
                 false, shape, cus, depth, vertex, normal, s);
  tick(kc, s, nullptr);
}

// Diagnostics: the distinct blocks the last raycast's lookups found (their
// ray_mark equals its stamp), added to the work counters.
__global__ __launch_bounds__(256) void ray_mark_count_kernel(View V) {
  const uint32_t n = V.ctr->block_hwm;
  uint32_t c = 0;
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < n; p += gridDim.x * blockDim.x)
    c += V.ray_mark[p] == V.ray_stamp;
  wave_add_u64(&work_stripe(V.ctr).ray_blocks, c);
}

void launch_ray_mark_count(const View& V, hipStream_t s, int grid) {
  ray_mark_count_kernel<<<grid, 256, 0, s>>>(V);
}

uint32_t raycast_grad_partials(const RayConst& p) {
  return ((p.cam.width + 7) / 8) * ((p.cam.height + 7) / 8);
}

void launch_raycast_backward(const View& V, const RayConst& p, const float* obs, float* grad_sdf,
                             double* partials, double* out, float max_residual, float max_slope,
                             hipStream_t s) {
  dim3 grid((p.cam.width + 7) / 8, (p.cam.height + 7) / 8);
  launch_ray_range(One{V}, nullptr, p, p.tiles, 1, s);
  if (V.capacity > kNarrowCapacity)
    raycast_backward_kernel<true><<<grid, 64, 0, s>>>(V, p, obs, grad_sdf, partials, max_residual, max_slope);
  else
    raycast_backward_kernel<false><<<grid, 64, 0, s>>>(V, p, obs, grad_sdf, partials, max_residual, max_slope);
  launch_slot_reduce(partials, grid.x * grid.y, kGradSlots, &V.ctr->reduce_done, out, s);
}

void launch_batch_raycast(const BatchDev& B, float* depth, float* vertex, float* normal,
                          hipStream_t s, int cus, int shape, bool beside) {
  launch_ray_range(B.src(), B.frames, RayConst{}, ((B.width + 7) / 8) * ((B.height + 7) / 8), B.nscenes, s);
  raycast_shaped(B.src(), B.frames, RayConst{}, B.width, B.height, B.nscenes, B.max_capacity > kNarrowCapacity, false,
                 beside, shape, cus, depth, vertex, normal, s);
}

}  // namespace mh
