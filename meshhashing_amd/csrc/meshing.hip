// meshing.hip -- incremental marching cubes over the worklist blocks.
//
// Reference: meshing/marching_cubes.cu:16-382 (SurfelExtractionKernel,
// TriangleExtractionKernel, RecycleTrianglesKernel, RecycleVerticesKernel),
// geometry/spatial_query.h:23-97 (trilinear value and gradient),
// core/mesh.h:53-107 (vertex/triangle pools and ref counts),
// visualization/color_util.h:13-37 (ValToRGB).
//
// MI355X layout: one workgroup per block, two cubes per lane.  The
// block and its 26 neighbours are staged once as an 11^3 voxel shell in LDS
// (local coordinates -1..9), which covers every corner, every trilinear
// sample and every gradient stencil of the block's cubes, so the 8 + 56
// hashed lookups per vertex of the reference become 26 lookups per block.
//
// Vertices are canonical: vertex (owner voxel o, axis a) is always computed
// from the endpoints o and o + e_a in that order, with the owner cube's
// corner positions.  In the reference up to four cubes write the same vertex
// with different endpoint orders and corner positions (last writer wins);
// here every writer stores the same bits.
#include "mh_kernels.h"
#include "mh_mc_tables.h"

namespace mh {

__constant__ McTables kMc = build_mc_tables();

constexpr int kShell = 11;
constexpr int kShellN = kShell * kShell * kShell;
constexpr int kShellWords = 48;  // 32 of its bits each, the whole waves that stage it

template <bool PSDF>
struct Shell {
  float sdf[kShellN];
  float w[kShellN];
  float a[PSDF ? kShellN : 1];
  float b[PSDF ? kShellN : 1];
  // Three bit strings over the shell's voxels (bit sidx): the SDF is negative;
  // the voxel passes the cube tests of a corner (|sdf| <= threshold,
  // rho >= rho_min, weight >= weight_min); it exists (its block is allocated).
  alignas(16) uint32_t bits[3][kShellWords];
};
enum ShellBits { kNeg = 0, kCorner = 1, kThere = 2 };

__device__ __forceinline__ int sidx(int x, int y, int z) {
  return (x + 1) + kShell * (y + 1) + kShell * kShell * (z + 1);
}
__device__ __forceinline__ int nb27(int dx, int dy, int dz) {
  return (dx + 1) + 3 * (dy + 1) + 9 * (dz + 1);
}

constexpr int kCfg = 9;  // local cube coordinates -1..7
// 32 bits of a shell bit string from bit `at` on.  A row of the shell is eleven
// of them, the next row (y + 1) follows, the next layer (z + 1) begins 121 on.
__device__ __forceinline__ uint32_t shell_bits(const uint32_t* b, uint32_t at) {
  const uint32_t w = at >> 5;
  return __builtin_amdgcn_alignbit(b[w + 1], b[w], at & 31u);
}

// The edge with owner offset (dx, dy, dz) and axis ax (a constant for
// constant arguments).
__host__ __device__ constexpr int edge_with(int dx, int dy, int dz, int ax) {
  int found = -1;
  for (int e = 0; e < 12; ++e)
    if (edge_owner_off(e, 0) == dx && edge_owner_off(e, 1) == dy && edge_owner_off(e, 2) == dz &&
        edge_axis(e) == ax)
      found = e;
  return found;
}
static_assert(edge_with(0, 0, 0, 0) >= 0 && edge_with(0, 1, 1, 0) >= 0 && edge_with(1, 0, 1, 1) >= 0 &&
                  edge_with(1, 1, 0, 2) >= 0,
              "every owner offset across an edge's axis names an edge");

// The 27 neighbours of every worklist block (x fastest, the block itself at
// 13) with their meshed-in-this-pass marks, one lane per (item, neighbour),
// before the surfel pass: the dependent worklist -> key -> occupancy ->
// bucket -> mark reads of a lookup then run with the whole grid's
// parallelism instead of on one workgroup's critical path.  Entry: the pool
// index, with bit 30 set when the neighbour is meshed in this pass; a
// negative value for an absent block.
__device__ __forceinline__ const McConst& mc_of(const One&, uint32_t, const McConst& mc) { return mc; }
__device__ __forceinline__ const McConst& mc_of(const Many& m, uint32_t s, const McConst&) {
  return m.f[s].mc;
}
// Surfel pass: 256 lanes a workgroup (two voxels a lane).  The next block's
// shell, cube words and vertex slots are loaded into registers while the
// current block is worked on, which takes 128 registers and spills seven a lane
// (three over a batch; none of a probabilistic volume's 168): four workgroups
// a CU, each a block at work and one on its way.  Bound by the instructions it
// issues where there are many blocks (64 rooms, 71 k blocks: 958 us, 673 of them
// VALU), by memory as well where most of them hold a fine surface (11 k blocks of a
// 5 mm frame: 155 us, 455 MB at 60 % of a device copy's rate), by the chain of a
// block's phases where there are few (1444 blocks: 50 us, two rounds of workgroups).  With eight lanes a vertex's payload and an item an
// edge of each cube, the replayed 640 x 480, 5 mm frame and a batch of 64 rooms took 358
// us and 2.87 ms so, 412 us and 3.35 ms with 512 lanes and two workgroups a CU, 466 us
// and 3.57 ms with 512 lanes, three workgroups and 80 registers (spills).
constexpr uint32_t kMcLanes = 256;
constexpr int kMcVox = kBlockVoxels / kMcLanes;
constexpr uint32_t kLookupLane = kMcLanes - 64;  // its last wave
// The surfel pass hands out its first items statically (workgroup g takes
// g, g + grid, ...) and the rest on demand from a counter, so workgroups
// whose blocks held little surface take more of them.  static_q quarters of
// the worklist (rounded down to whole rounds of the grid, at least one) are
// static.  The rest goes by kDynGroups counters (cleared by the neighbour-table
// pass), workgroup g taking every kDynGroups-th item from the one of its group:
// on one counter, workgroups that ask at the same time wait for each other.
__device__ __forceinline__ uint32_t mc_static_items(uint32_t n, uint32_t grid, uint32_t static_q) {
  const uint32_t k = (static_q * n / 4u) / grid;
  return (k ? k : 1u) * grid;
}
constexpr int32_t kMeshedBit = 1 << 30;
template <class Src>
__global__ __launch_bounds__(256) void mc_neighbours_kernel(Src src_, const SceneFrame* __restrict__ tab,
                                                             McConst mc1, int32_t* __restrict__ nbt) {
  const Src src = with_table(src_, tab);
  const uint32_t total = src.count() * 27u;
  // the surfel pass's counters of items handed out on demand (it runs next)
  if (blockIdx.x == 0 && threadIdx.x < kDynGroups) src.next_ctr()[64 * threadIdx.x] = 0u;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < total; i += gridDim.x * blockDim.x) {
    const uint32_t ci = i / 27u, t = i % 27u;
    uint32_t scene;
    const int32_t self = src.lane_item(ci, &scene);
    const View& V = src.view(scene);
    const i3 b = unpack_key(V.block_keys[self]);
    const int dx = (int)(t % 3) - 1, dy = (int)((t / 3) % 3) - 1, dz = (int)(t / 9) - 1;
    const int32_t p = (dx | dy | dz) == 0 ? self : hash_find_eager(V, i3{b.x + dx, b.y + dy, b.z + dz});
    int32_t e = kFreePtr;
    if (p >= 0) e = p | (V.block_mark[p] == mc_of(src, scene, mc1).pass ? kMeshedBit : 0);
    nbt[i] = e;
  }
}

// What a lane holds of a block on its way: its share of the shell, its two
// voxels' cube words and vertex slots.
constexpr int kShellPer = (kShellN + (int)kMcLanes - 1) / (int)kMcLanes;
template <bool PSDF>
struct BlockRegs {
  float sd[kShellPer], wt[kShellPer], va[PSDF ? kShellPer : 1], vb[PSDF ? kShellPer : 1];
  bool ok[kShellPer];
  int32_t vps[kMcVox][3];
  uint32_t word[kMcVox];
};
// Where shell voxel s lies: neighbour | local voxel << 5 | kCodeInner if it is a
// corner of a cube at local -1..7 (its coordinates are at most 8).
constexpr uint32_t kCodeInner = 1u << 14;
__device__ __forceinline__ uint32_t shell_code(int s) {
  const int lx = s % kShell - 1, ly = (s / kShell) % kShell - 1, lz = s / (kShell * kShell) - 1;
  const int dx = lx < 0 ? -1 : (lx >= 8 ? 1 : 0), dy = ly < 0 ? -1 : (ly >= 8 ? 1 : 0),
            dz = lz < 0 ? -1 : (lz >= 8 ? 1 : 0);
  return (uint32_t)nb27(dx, dy, dz) | ((uint32_t)((lx - 8 * dx) + 8 * (ly - 8 * dy) + 64 * (lz - 8 * dz)) << 5) |
         (lx <= 8 && ly <= 8 && lz <= 8 ? kCodeInner : 0u);
}
// A row entry's pool index (negative: absent) and mark.
__device__ __forceinline__ int32_t row_ptr(int32_t e) { return e < 0 ? e : (e & (kMeshedBit - 1)); }
__device__ __forceinline__ bool row_meshed(int32_t e) { return e >= 0 && (e & kMeshedBit) != 0; }

// Issues the loads of block ptr (row: its neighbours, code: shell_code's table).
template <bool PSDF>
__device__ __forceinline__ void load_block(const View& V, int32_t ptr, const int32_t* row, const uint16_t* code,
                                           BlockRegs<PSDF>& R) {
#pragma unroll
  for (int r = 0; r < kShellPer; ++r) {
    const int s = (int)(threadIdx.x + kMcLanes * r);
    R.ok[r] = false;
    R.sd[r] = R.wt[r] = 0.0f;
    if (PSDF) R.va[r] = R.vb[r] = 0.0f;
    if (s >= kShellN) continue;
    const uint32_t c = code[s];
    const int32_t p = row_ptr(row[c & 31u]);
    if (p < 0) continue;
    const size_t idx = (size_t)p * kBlockVoxels + ((c >> 5) & 511u);
    R.ok[r] = true;
    R.sd[r] = V.sdf[idx];
    R.wt[r] = V.weight[idx];
    if (PSDF) {
      R.va[r] = V.va[idx];
      R.vb[r] = V.vb[idx];
    }
  }
#pragma unroll
  for (int r = 0; r < kMcVox; ++r) {
    const size_t idx = (size_t)ptr * kBlockVoxels + threadIdx.x + kMcLanes * r;
    R.word[r] = V.cube[idx];
#pragma unroll
    for (int a = 0; a < 3; ++a) R.vps[r][a] = V.vptr[3 * idx + a];
  }
}

// Puts the lane's share of the shell into LDS.  Returns whether the block may
// hold a vertex or a triangle after this pass, or holds a vertex slot now, as
// far as this lane can see: a negative voxel around its own and its lower
// neighbours' cubes (local -1..8), a slot, or a lower neighbour that is not
// meshed in this pass (its stored configurations count then).  A block of
// which no lane says so is done: its cubes are all 0 and it has no surfels.
template <bool PSDF>
__device__ __forceinline__ bool stage_shell(const McConst& mc, const BlockRegs<PSDF>& R, const uint16_t* code,
                                            Shell<PSDF>& S) {
  bool keep = false;
#pragma unroll
  for (int r = 0; r < kShellPer; ++r) {
    const int s = (int)(threadIdx.x + kMcLanes * r);
    bool neg = false, corner = false, there = false;
    if (s < kShellN) {
      // the corner tests of IsValid (marching_cubes.cu:96-130), once per
      // voxel here instead of once per cube corner
      const float sd = R.sd[r], wt = R.wt[r];
      const float rho = PSDF ? R.va[r] / (R.va[r] + R.vb[r]) : 0.0f;
      const bool cube_ok = R.ok[r] && !(fabsf(sd) > mc.sdf_threshold) && (!PSDF || !(rho < mc.rho_min)) &&
                           !(wt < mc.weight_min);
      neg = sd < 0.0f;
      corner = cube_ok;
      there = R.ok[r];
      S.sdf[s] = R.ok[r] ? sd : NAN;  // a sample with an absent corner is none: NaN
      S.w[s] = wt;
      if (PSDF) {
        S.a[s] = R.va[r];
        S.b[s] = R.vb[r];
      }
      keep = keep || (neg && (code[s] & kCodeInner));
    }
    const uint64_t bn = __ballot(neg), bc = __ballot(corner), bt = __ballot(there);
    const uint32_t lane = threadIdx.x & 63u;
    if (lane < 3)
      reinterpret_cast<uint64_t*>(S.bits[lane])[kMcLanes / 64 * r + (threadIdx.x >> 6)] = lane == 0 ? bn : (lane == 1 ? bc : bt);
  }
#pragma unroll
  for (int r = 0; r < kMcVox; ++r) keep = keep || R.vps[r][0] >= 0 || R.vps[r][1] >= 0 || R.vps[r][2] >= 0;
  return keep;
}

// One axis of a GetSpatialValue sample (spatial_query.h:23-66) at world
// coordinate p: the two corner voxels (rounded from p - vs/2 and p + vs/2,
// exactly as the reference, so ties and negative coordinates pick the same
// voxels), local to the block origin base, and the ratio frac(p / vs).  A
// sample's axes are independent, so the gradient stencils p +- vs/2 e_k
// share two of their three axes with the centre sample.
struct SAxis {
  int c0, c1;
  float r;
};
__device__ __forceinline__ SAxis shell_axis(float p, float vs, float inv_vs, int base) {
  SAxis a;
  corner_pair(p - 0.5f * vs, vs, inv_vs, &a.c0, &a.c1);
  a.c0 -= base;
  a.c1 -= base;
  const float q = quotient(p, vs, inv_vs);
  a.r = q - floorf(q);
  return a;
}

// GetSpatialValue against a staged field, from the sample's three axes; `in`:
// its corners lie in the shell (local -1..9).
__device__ __forceinline__ bool axes_in(const SAxis& X, const SAxis& Y, const SAxis& Z) {
  return min(min(min(X.c0, X.c1), min(Y.c0, Y.c1)), min(Z.c0, Z.c1)) >= -1 &&
         max(max(max(X.c0, X.c1), max(Y.c0, Y.c1)), max(Z.c0, Z.c1)) <= 9;
}
__device__ __forceinline__ float shell_value(const float* f, const SAxis& X, const SAxis& Y, const SAxis& Z) {
  const int cx[2] = {X.c0, X.c1}, cy[2] = {Y.c0, Y.c1}, cz[2] = {Z.c0, Z.c1};
  float v = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int mx = (i >> 2) & 1, my = (i >> 1) & 1, mz = i & 1;
    const float w = (mx ? X.r : 1.0f - X.r) * (my ? Y.r : 1.0f - Y.r) * (mz ? Z.r : 1.0f - Z.r);
    v += w * f[sidx(cx[mx], cy[my], cz[mz])];
  }
  return v;
}

// ValToRGB (color_util.h:13-37); the 0.25/0.5/0.75 literals are doubles
// there, so the band tests and two of the channel formulas run in double.
__device__ __forceinline__ f3 val_to_rgb(float v, float vmin, float vmax) {
  f3 c = mk3(1.0f, 1.0f, 1.0f);
  if (v < vmin) v = vmin;
  if (v > vmax) v = vmax;
  const float dv = vmax - vmin;
  const double vd = v, mn = vmin, dd = dv;
  if (vd < mn + 0.25 * dd) {
    c.x = 0.0f;
    c.y = 4.0f * (v - vmin) / dv;
  } else if (vd < mn + 0.5 * dd) {
    c.x = 0.0f;
    c.z = (float)(1.0 + 4.0 * (mn + 0.25 * dd - vd) / dd);
  } else if (vd < mn + 0.75 * dd) {
    c.x = (float)(4.0 * (vd - mn - 0.5 * dd) / dd);
    c.z = 0.0f;
  } else {
    c.y = (float)(1.0 + 4.0 * (mn + 0.75 * dd - vd) / dd);
    c.z = 0.0f;
  }
  return c;
}

// ---------------------------------------------------------------- pass 1
// A cube of a block, from the shell's bits: `a` those of its layer from its own
// voxel on (0 and 1 its two corners there, 11 and 12 those of the next row), `b`
// those of the next layer.
constexpr uint32_t kCubeBits = 0x1803u;
__device__ __forceinline__ uint32_t cube_of(uint32_t a, uint32_t b) {
  // corners 0-7 (corner_off): 011 111 110 010 001 101 100 000
  const uint32_t swap = 0xD8u;  // two bits exchanged: 0, 2, 1, 3
  return ((b >> 11) & 3u) | ((swap >> (2 * ((a >> 11) & 3u))) & 3u) << 2 | (b & 3u) << 4 | ((swap >> (2 * (a & 3u))) & 3u) << 6;
}
constexpr bool corner_order_is(int i, int x, int y, int z) {
  return corner_off(i, 0) == x && corner_off(i, 1) == y && corner_off(i, 2) == z;
}
static_assert(corner_order_is(0, 0, 1, 1) && corner_order_is(1, 1, 1, 1) && corner_order_is(2, 1, 1, 0) &&
                  corner_order_is(3, 0, 1, 0) && corner_order_is(4, 0, 0, 1) && corner_order_is(5, 1, 0, 1) &&
                  corner_order_is(6, 1, 0, 0) && corner_order_is(7, 0, 0, 0),
              "cube_of");
// A configuration uses exactly the edges whose ends differ in sign.
constexpr bool edges_are_crossings() {
  const McTables t = build_mc_tables();
  for (int c = 0; c < 256; ++c)
    for (int e = 0; e < 12; ++e)
      if (((t.edges[c] >> e) & 1) != (((c >> edge_a(e)) ^ (c >> edge_b(e))) & 1)) return false;
  return true;
}
static_assert(edges_are_crossings(), "an edge is used where its ends differ in sign");

// Cubes at local coordinates -1..8: a row of ten bits for each y, z.
constexpr int kCubeHalo = 10;
__device__ __forceinline__ int crow(int y, int z) { return (y + 1) + kCubeHalo * (z + 1); }

// The surfel pass queues a block's vertex writes in LDS (a block with surface
// writes ~80): a round of slot claims adds at most one per lane, and the queue
// is worked off when another round might not fit.
constexpr uint32_t kQueue = 2 * kMcLanes;

// Payload of vertex (owner voxel at local (key & 15, key >> 4 & 15,
// key >> 8 & 15), axis key >> 12): VertexIntersection (marching_cubes.cu:16-28)
// in the canonical endpoint order, then AllocateVertexWithMutex's payload
// (:45-72).  Four lanes sample a vertex: lanes 0-2 the gradient stencils p -+ h e_k
// of an axis each, which share two axes with p, lane 3 the ratios of p itself
// (p -+ 0 = p), and each two of the eight corner radii of lane 3's cell.  What they
// found meets in LDS, a row a value (Payload), and one lane a vertex each then
// takes the normal from it (finish_normal) and the radius and colour
// (finish_sample).
//
// The pass is bound by the instructions it issues (VALU busy three quarters of
// the time), so the lanes that share a vertex are few and the record's end,
// with its divisions and square roots, has 64 vertices a wave.  Eight lanes a
// vertex, two of which also finished the record (eight vertices a wave there),
// took 9140 wave instructions a block of 64 rooms' pass (1385 us); 7940 so (1245
// us), and a 320 x 240 room's frame 62 us instead of 71.
constexpr uint32_t kPayRound = kMcLanes / 4;
constexpr uint32_t kPayPitch = kPayRound + 16;  // the four lanes' rows in other banks
enum PayRow { kPayS = 0, kPayR = 6, kPayRatio = 14, kPayPos = 17, kPayOk = 20, kPayA = 21, kPayB = 22 };
template <bool PSDF>
struct Payload {
  float v[PSDF ? 23 : 21][kPayPitch];
};
// The value of lane 3 of four.
__device__ __forceinline__ uint32_t quad_last(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xFF, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ uint32_t quad_swap(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xF, 0xF, true);
}
// The axes of the samples that lie at a voxel's coordinate, and half a voxel to
// either side: a vertex is off its voxel along its own axis only, so five of the
// eight axes of a lane's samples are among a block's 81 of these.  They are
// rounding ties, which shell_axis settles with divisions: 6850 wave instructions
// a block of 64 rooms without the table, 5780 with it (1033 and 946 us a pass).
struct AxisTable {
  uint32_t c[3][9][3];  // axis, voxel 0..8, -h / 0 / +h: c0 + 64 | c1 + 64 << 8
  float r[3][9][3];
};
constexpr uint32_t kAxisEntries = 81;
__device__ __forceinline__ void axis_table_fill(AxisTable& T, uint32_t e, float vs, float inv_vs, i3 base) {
  const uint32_t d = e % 3, o = e / 3 % 9, a = e / 27;
  const int b = a == 0 ? base.x : (a == 1 ? base.y : base.z);
  const float p = (float)(b + (int)o) * vs, h = 0.5f * vs;
  const SAxis A = shell_axis(d == 0 ? p - h : (d == 1 ? p : p + h), vs, inv_vs, b);
  auto byte = [](int c) { return (uint32_t)(min(max(c, -64), 191) + 64); };  // (out of the shell stays so)
  (&T.c[0][0][0])[e] = byte(A.c0) | byte(A.c1) << 8;
  (&T.r[0][0][0])[e] = A.r;
}
__device__ __forceinline__ SAxis axis_at(const AxisTable& T, int a, int o, int d) {
  const uint32_t c = T.c[a][o][d];
  return SAxis{(int)(c & 255u) - 64, (int)(c >> 8) - 64, T.r[a][o][d]};
}
// Lane sub's part for vertex j of the round; true if a sample lies outside the shell.
template <bool PSDF>
__device__ __forceinline__ bool payload_part(const Shell<PSDF>& S, const Geo& g, const McConst& mc, float inv_vs,
                                             const AxisTable& T, i3 base, uint32_t key, uint32_t sub, uint32_t j,
                                             Payload<PSDF>& P) {
  const float vs = g.voxel_size;
  const int ox = (int)(key & 15u), oy = (int)((key >> 4) & 15u), oz = (int)((key >> 8) & 15u);
  const int ax = (int)(key >> 12);
  const int sA = sidx(ox, oy, oz);
  const float vA = S.sdf[sA], vB = S.sdf[sA + (ax == 0 ? 1 : (ax == 1 ? kShell : kShell * kShell))];
  // the vertex's coordinate along its axis, from its voxel's to the next one's
  const int b = ax == 0 ? base.x : (ax == 1 ? base.y : base.z), o = (int)((key >> (4 * ax)) & 15u);
  const float pA = (float)(b + o) * vs, pB = pA + vs;
  float p;
  if ((double)fabsf(vA) < mc.snap) {
    p = pA;
  } else if ((double)fabsf(vB) < mc.snap) {
    p = pB;
  } else {
    const float mu = (0.0f - vA) / (vB - vA);
    p = pA + mu * (pB - pA);
  }
  const float h = 0.5f * vs;
  // the first stencil's axes (lane 3: p's), and the one that the second differs in
  const SAxis A = shell_axis((int)sub == ax ? p - h : p, vs, inv_vs, b);
  SAxis X = ax == 0 ? A : axis_at(T, 0, ox, sub == 0 ? 0 : 1);
  SAxis Y = ax == 1 ? A : axis_at(T, 1, oy, sub == 1 ? 0 : 1);
  SAxis Z = ax == 2 ? A : axis_at(T, 2, oz, sub == 2 ? 0 : 1);
  bool oob = !axes_in(X, Y, Z);
  // lane 3's cell, corner coordinates + 1 in 4 bits each (inside: all in 0..10)
  const uint32_t cell = (uint32_t)(X.c0 + 1) | ((uint32_t)(X.c1 + 1) << 4) | ((uint32_t)(Y.c0 + 1) << 8) |
                        ((uint32_t)(Y.c1 + 1) << 12) | ((uint32_t)(Z.c0 + 1) << 16) | ((uint32_t)(Z.c1 + 1) << 20);
  const uint32_t c3 = quad_last(oob ? ~0u : cell);
  uint32_t ok = c3 != ~0u ? 1u : 0u;
  if (c3 != ~0u) {
    const uint32_t cx = (c3 >> ((sub & 2u) ? 4 : 0)) & 15u, cy = (c3 >> ((sub & 1u) ? 12 : 8)) & 15u;
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) {  // corners 2 sub and 2 sub + 1
      const uint32_t s = cx + kShell * cy + kShell * kShell * ((c3 >> (i ? 20 : 16)) & 15u);
      ok &= S.bits[kThere][s >> 5] >> (s & 31u);
      P.v[kPayR + 2 * sub + i][j] = sqrtf(1.0f / S.w[s]);
    }
  }
  ok &= quad_swap<0xB1>(ok);
  ok &= quad_swap<0x4E>(ok);
  if (sub == 3) {
    P.v[kPayRatio][j] = X.r;
    P.v[kPayRatio + 1][j] = Y.r;
    P.v[kPayRatio + 2][j] = Z.r;
    P.v[kPayPos][j] = ax == 0 ? p : (float)(base.x + ox) * vs;
    P.v[kPayPos + 1][j] = ax == 1 ? p : (float)(base.y + oy) * vs;
    P.v[kPayPos + 2][j] = ax == 2 ? p : (float)(base.z + oz) * vs;
    P.v[kPayOk][j] = ok ? 1.0f : 0.0f;
    if (PSDF && ok) {
      P.v[kPayA][j] = shell_value(S.a, X, Y, Z);
      P.v[kPayB][j] = shell_value(S.b, X, Y, Z);
    }
  } else {
#pragma unroll 1
    for (uint32_t i = 0;; ++i) {
      P.v[kPayS + 2 * sub + i][j] = axes_in(X, Y, Z) ? shell_value(S.sdf, X, Y, Z) : NAN;
      if (i) break;
      SAxis A = axis_at(T, (int)sub, (int)((key >> (4 * sub)) & 15u), 2);
      if ((int)sub == ax) A = shell_axis(p + h, vs, inv_vs, b);
      if (sub == 0) X = A;
      if (sub == 1) Y = A;
      if (sub == 2) Z = A;
      oob = oob || !axes_in(X, Y, Z);
    }
  }
  return oob;
}

// Position, radius and colour of vertex j of the round.  An end that is no number
// (a NaN passes the corner tests) makes none of all three coordinates, the other
// axes' being pA + NaN * 0, and of its sample, in the cell of the voxel 0 that a
// NaN rounds to.
template <bool PSDF>
__device__ __forceinline__ void finish_sample(const Shell<PSDF>& S, const View& V, i3 base, int32_t vp, uint32_t j,
                                              const Payload<PSDF>& P) {
  float px = P.v[kPayPos][j], py = P.v[kPayPos + 1][j], pz = P.v[kPayPos + 2][j];
  bool ok = P.v[kPayOk][j] != 0.0f;
  const float sum = px + py + pz;
  const bool none = !(sum == sum);
  if (__builtin_expect(none, 0)) {
    px = py = pz = sum;
    ok = (uint32_t)-base.x <= 8u && (uint32_t)-base.y <= 8u && (uint32_t)-base.z <= 8u;
    if (ok) {
      const uint32_t s = (uint32_t)sidx(-base.x, -base.y, -base.z);
      ok = (S.bits[kThere][s >> 5] >> (s & 31u)) & 1u;
    } else {
      flag(V, MH_STATUS_STENCIL_RANGE);
    }
  }
  float radius = 0.0f, cr = 0.0f, cg = 0.0f, cb = 0.0f;  // the reference reads an uninitialised query here
  if (ok) {
    const float rx = P.v[kPayRatio][j], ry = P.v[kPayRatio + 1][j], rz = P.v[kPayRatio + 2][j];
    float rad = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float w = ((i & 4) ? rx : 1.0f - rx) * ((i & 2) ? ry : 1.0f - ry) * ((i & 1) ? rz : 1.0f - rz);
      rad += w * P.v[kPayR + i][j];
    }
    const float inv_sigma2 = 1.0f / (rad * rad);
    radius = sqrtf(1.0f / inv_sigma2);
    float a = PSDF ? P.v[PSDF ? kPayA : 0][j] : 0.0f, b = PSDF ? P.v[PSDF ? kPayB : 0][j] : 0.0f;
    if (PSDF && none) a = sum;
    const f3 c = val_to_rgb(a / (a + b), 0.4f, 1.0f);
    cr = c.x;
    cg = c.y;
    cb = c.z;
  }
  Vertex* dst = &V.vertices[vp];
  dst->px = px;
  dst->py = py;
  dst->pz = pz;
  dst->radius = radius;
  dst->cr = cr;
  dst->cg = cg;
  dst->cb = cb;
}

// GetSpatialSDFGradient's normal from the six stencil values of a vertex (-x,
// +x, -y, +y, -z, +z).  An invalid sample, which is NaN, zeroes it, which is what
// the reference's short-circuit produces.
template <bool PSDF>
__device__ __forceinline__ void finish_normal(const View& V, int32_t vp, uint32_t j, const Payload<PSDF>& P) {
  const float vs = V.geo.voxel_size;
  const f3 grad = mk3((P.v[1][j] - P.v[0][j]) / vs, (P.v[3][j] - P.v[2][j]) / vs, (P.v[5][j] - P.v[4][j]) / vs);
  const float l = length(grad);
  const f3 n = l > 0.0f ? grad / l : mk3(0.0f, 0.0f, 0.0f);
  Vertex* dst = &V.vertices[vp];
  dst->nx = n.x;
  dst->ny = n.y;
  dst->nz = n.z;
}

// SurfelExtractionKernel (marching_cubes.cu:75-170): cube index of every
// cube of the block, and the vertex of every active edge.  A vertex is
// shared by up to four cubes.  Its payload is written once per pass, by a
// designated cube: the first, in the order (0,0), (1,0), (0,1), (1,1) of
// the offsets across the edge, that is valid and belongs to a block meshed
// in this pass.  Every block can evaluate that rule from the staged shell (the
// halo's rows of valid cubes and the meshed flags of the 27 blocks), so
// no atomics are needed; the other cubes' blocks only make sure the vertex slot
// is allocated.  Any writer would store the same bits (canonical vertices).

// Work counts of a workgroup, kept by its first lane and added to the scene's
// counters when the scene changes.
struct McCounts {
  uint32_t writes = 0, assigned = 0, blocks = 0;
  int delta = 0;
  __device__ void flush(const View& V) {
    WorkStripe& w = work_stripe(V.ctr);
    if (writes) atomicAdd(&w.mc_vertex_writes, (unsigned long long)writes);
    if (assigned) atomicAdd(&w.mc_triangle_writes, (unsigned long long)assigned);
    if (blocks) atomicAdd(&w.mc_blocks, (unsigned long long)blocks);
    if (delta) atomicAdd(&w.tri_live, (unsigned long long)(long long)delta);
    *this = McCounts{};
  }
};

// Exclusive scan over the wave of values v whose set bits all lie in PLANES,
// one bit plane at a time (a ballot and a masked bit count per plane, no lane
// shuffles); *all gets the wave's sum.  Packed fields scan independently as
// long as no field's sum carries into the next one.
template <uint32_t PLANES>
__device__ __forceinline__ uint32_t wave_excl_scan(uint32_t v, uint32_t* all) {
  uint32_t before = 0, sum = 0;
#pragma unroll
  for (int k = 0; k < 32; ++k) {
    if (!((PLANES >> k) & 1u)) continue;
    const uint64_t m = __ballot((v >> k) & 1u);
    before += __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u)) << k;
    sum += (uint32_t)__popcll(m) << k;
  }
  *all = sum;
  return before;
}

// Exclusive scan of one value per lane over the workgroup (up to eight
// waves), its set bits in PLANES; *total gets the sum.  Every lane must call
// it; it synchronises the workgroup twice.
template <uint32_t PLANES>
__device__ __forceinline__ uint32_t block_excl_scan_planes(uint32_t v, uint32_t* wave_sums, uint32_t* total) {
  const uint32_t wave = threadIdx.x >> 6;
  uint32_t wsum;
  const uint32_t x = wave_excl_scan<PLANES>(v, &wsum);
  if ((threadIdx.x & 63u) == 0) wave_sums[wave] = wsum;
  __syncthreads();
  uint32_t before = 0, all = 0;
  const uint32_t nw = blockDim.x >> 6;
  for (uint32_t w = 0; w < nw; ++w) {
    const uint32_t ws = wave_sums[w];
    if (w < wave) before += ws;
    all += ws;
  }
  __syncthreads();
  *total = all;
  return before + x;
}
// The same for values v < 2^BITS.
template <int BITS>
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* wave_sums, uint32_t* total) {
  return block_excl_scan_planes<(1u << BITS) - 1u>(v, wave_sums, total);
}

template <bool PSDF, class Src>
__global__ __launch_bounds__(kMcLanes, PSDF ? 3 : 4) void mc_surfel_kernel(Src src_, const SceneFrame* __restrict__ tab, McConst mc1,
                                                                const int32_t* __restrict__ nbt, uint32_t static_q) {
  const Src src = with_table(src_, tab);
  __shared__ Shell<PSDF> S;
  __shared__ uint16_t code[kShellN];
  __shared__ int32_t row_[2][27];  // the neighbour-table rows of the block at work and of the next one
  // the halo's cubes that are valid and belong to a block meshed in this pass
  __shared__ uint16_t cv[kCubeHalo * kCubeHalo];
  __shared__ int surfels[2];
  __shared__ int tri_sum[2];  // the block's change of live triangles, and the triangles of its changed cubes
  // Flags of a block, three in turn: a block without surface ends without a
  // further barrier, so a fast wave may set the next block's while a slow one
  // still reads this one's; after a block's first barrier every wave is done
  // with the one before it, whose flags are then cleared for the one after next.
  __shared__ uint32_t busy_[3][3];
  __shared__ uint32_t next_[2];
  __shared__ uint32_t free_base;
  __shared__ int32_t qptr[kQueue];
  __shared__ uint16_t qkey[kQueue];
  __shared__ uint32_t qn;
  __shared__ uint32_t scan_wave[8];
  __shared__ int32_t pop_top;
  // One LDS region, two uses that never overlap in time: the slots that stored
  // configurations use, up to the recycling test; the item list from the item
  // scan to the end of the slot claims.  Barriers separate the uses.
  constexpr uint32_t kMaxItems = 3 * kBlockSide * (kBlockSide + 1) * (kBlockSide + 1);
  __shared__ uint32_t region[(kMaxItems + 1) / 2];
  uint16_t* const items = reinterpret_cast<uint16_t*>(region);
  uint32_t* const stored = region;  // axis, row (y + 8 z): a bit per x
  static_assert(sizeof(region) >= 3 * 64 * sizeof(uint32_t) && 3 * 64 <= kMcLanes, "region");
  __shared__ Payload<PSDF> pay;
  __shared__ AxisTable axes;
  __shared__ uint32_t nitems;
  // per-configuration crossed edges and triangle counts, read per lane with
  // divergent indices: from LDS rather than the constant tables
  __shared__ uint16_t etab[256];
  __shared__ uint8_t ntab[256];
  const uint32_t n = src.count();
  if (blockIdx.x >= n) return;
  for (uint32_t k = threadIdx.x; k < 256u; k += kMcLanes) {
    etab[k] = kMc.edges[k];
    ntab[k] = (uint8_t)kMc.ntri[k];
  }
  for (int s = (int)threadIdx.x; s < kShellN; s += (int)kMcLanes) code[s] = (uint16_t)shell_code(s);
  McCounts cnt;
  uint32_t cur_scene = ~0u, turns = 0;
  // items: ci at work, nx next (its loads under way), the one after it in
  // next_; lanes kLookupLane + t hold neighbour t's table entry of item nx
  const uint32_t nb_lane = threadIdx.x - kLookupLane;
  const uint32_t n_static = mc_static_items(n, gridDim.x, static_q);
  auto item_after = [&](uint32_t c) -> uint32_t {
    if (c + gridDim.x < n_static) return c + gridDim.x;
    if (n_static >= n) return n;
    const uint32_t groups = min(kDynGroups, gridDim.x), group = blockIdx.x % groups;
    return n_static + groups * atomicAdd(src.next_ctr() + 64 * group, 1u) + group;
  };
  uint32_t ci = blockIdx.x;
  if (threadIdx.x == 0) {
    next_[1] = item_after(ci);
    for (int k = 0; k < 3; ++k) busy_[k][0] = busy_[k][1] = busy_[k][2] = 0u;
  }
  if (nb_lane < 27) row_[0][nb_lane] = nbt[(size_t)ci * 27u + nb_lane];
  __syncthreads();
  uint32_t nx = next_[1];
  int32_t nbe = nb_lane < 27 && nx < n ? nbt[(size_t)nx * 27u + nb_lane] : kFreePtr;
  uint32_t scene, scene_n = 0;
  int32_t ptr = src.item(ci, &scene), ptr_n = 0;
  uint64_t key = src.view(scene).block_keys[ptr], key_n = 0;
  if (nx < n) {
    ptr_n = src.item(nx, &scene_n);
    key_n = src.view(scene_n).block_keys[ptr_n];
  }
  BlockRegs<PSDF> R;
  load_block<PSDF>(src.view(scene), ptr, row_[0], code, R);
  for (uint32_t turn = 0, third = 0; ci < n; turn ^= 1u, third = third == 2 ? 0 : third + 1) {
    // The lane's own places are worked out anew for each block: kept across them
    // they do not fit the registers (100 bytes a lane spilled).
    uint32_t tid = threadIdx.x;
    asm("" : "+v"(tid));
    if (scene != cur_scene) {
      if (cur_scene != ~0u && threadIdx.x == 0) cnt.flush(src.view(cur_scene));
      cur_scene = scene;
    }
    const View& V = src.view(scene);
    const McConst& mc = mc_of(src, scene, mc1);
    cnt.blocks += threadIdx.x == 0;
    const int32_t* const nb = row_[turn];
    if (threadIdx.x == 0) next_[turn] = nx < n ? item_after(nx) : n;
    if (nb_lane < 27) row_[turn ^ 1u][nb_lane] = nbe;
    bool lower = false;  // a lower neighbour that is not meshed in this pass
    if (nb_lane < 27 && nb_lane % 3 < 2 && (nb_lane / 3) % 3 < 2 && nb_lane / 9 < 2)
      lower = nb[nb_lane] >= 0 && !row_meshed(nb[nb_lane]);
    if (lower) busy_[third][2] = 1u;
    if (__any(stage_shell<PSDF>(mc, R, code, S) || lower) && (tid & 63u) == 0) busy_[third][0] = 1u;
    int32_t vps[kMcVox][3];
    uint32_t word[kMcVox];
#pragma unroll
    for (int r = 0; r < kMcVox; ++r) {
      word[r] = R.word[r];
#pragma unroll
      for (int a = 0; a < 3; ++a) vps[r][a] = R.vps[r][a];
    }
    __syncthreads();
    // every wave is past the previous block: its flags and counts can go, and
    // the next block's loads start
    if (threadIdx.x == 0) {
      const uint32_t before = third == 0 ? 2 : third - 1;
      busy_[before][0] = busy_[before][1] = busy_[before][2] = 0u;
      qn = 0;
      surfels[0] = surfels[1] = 0;
      tri_sum[0] = tri_sum[1] = 0;
    }
    const uint32_t nn = next_[turn];
    if (nx < n) load_block<PSDF>(src.view(scene_n), ptr_n, row_[turn ^ 1u], code, R);
    nbe = nb_lane < 27 && nn < n ? nbt[(size_t)nn * 27u + nb_lane] : kFreePtr;
    uint32_t scene_nn = 0;
    int32_t ptr_nn = 0;
    uint64_t key_nn = 0;
    if (nn < n) {
      ptr_nn = src.item(nn, &scene_nn);
      key_nn = src.view(scene_nn).block_keys[ptr_nn];
    }
    const int32_t self = ptr;
    const i3 b = unpack_key(key);
    auto advance = [&] {
      ci = nx;
      nx = nn;
      ptr = ptr_n;
      ptr_n = ptr_nn;
      scene = scene_n;
      scene_n = scene_nn;
      key = key_n;
      key_n = key_nn;
    };
    // A block that keeps and gets no vertex: its cubes' words, its counts.
    auto finish_empty = [&](const uint32_t* c) {
      int lost = 0;
#pragma unroll
      for (int r = 0; r < kMcVox; ++r) {
        const uint32_t prev = word[r] & 255u, nw = c[r] | (prev << 8);
        if (nw != word[r]) V.cube[(size_t)self * kBlockVoxels + tid + kMcLanes * r] = (uint16_t)nw;
        lost += ntab[prev];  // c is 0 or 255: no triangle
      }
      // (rare: a block that lost its surface)
      if (lost) atomicAdd(&work_stripe(V.ctr).tri_live, (unsigned long long)(long long)-lost);
      if (threadIdx.x == 0) V.surfel[2 * self] = V.surfel[2 * self + 1] = 0;
      advance();
    };
    uint32_t cube[kMcVox] = {};
    if (!busy_[third][0]) {  // uniform
      finish_empty(cube);
      continue;
    }
    // The block's own cubes, and the crossings of the edges it owns (cross: x, y,
    // z edges of a voxel whose ends differ in sign), from the shell's bits; the
    // halo's cubes, of which only the validity counts, as rows of bits.
    bool crossing = false;
    uint32_t cross[kMcVox];
#pragma unroll
    for (int r = 0; r < kMcVox; ++r) {
      const i3 o = devectorize(tid + kMcLanes * r);
      const uint32_t at = (uint32_t)sidx(o.x, o.y, o.z), up = at + kShell * kShell;
      const uint32_t na = shell_bits(S.bits[kNeg], at), nu = shell_bits(S.bits[kNeg], up);
      const uint32_t ca = shell_bits(S.bits[kCorner], at), cu = shell_bits(S.bits[kCorner], up);
      cube[r] = (ca & cu & kCubeBits) == kCubeBits ? cube_of(na, nu) : 0u;
      cross[r] = ((na ^ (na >> 1)) & 1u) | ((na ^ (na >> 11)) & 1u) << 1 | ((na ^ nu) & 1u) << 2;
      // an edge that a valid cube uses has ends that pass the corner tests
      cross[r] &= ca & 1u ? ((ca >> 1) & 1u) | ((ca >> 11) & 1u) << 1 | (cu & 1u) << 2 : 0u;
      crossing = crossing || (cube[r] != 0 && cube[r] != 255) || cross[r] != 0 || vps[r][0] >= 0 || vps[r][1] >= 0 || vps[r][2] >= 0;
    }
    // the halo's rows, and by the other two waves the block's axes
    const i3 base = i3{b.x * kBlockSide, b.y * kBlockSide, b.z * kBlockSide};
    const float inv_vs = 1.0f / V.geo.voxel_size;
    if (tid - (kMcLanes - 128) < kAxisEntries)
      axis_table_fill(axes, tid - (kMcLanes - 128), V.geo.voxel_size, inv_vs, base);
    if (tid < kCubeHalo * kCubeHalo) {
      const uint32_t y = tid % kCubeHalo, z = tid / kCubeHalo;
      const uint32_t at = kShell * y + kShell * kShell * z;
      uint32_t c = shell_bits(S.bits[kCorner], at) & shell_bits(S.bits[kCorner], at + kShell * kShell);
      c &= c >> kShell;
      c &= c >> 1;
      const int32_t* const q = nb + 3 * (y == 0 ? 0 : (y == 9 ? 2 : 1)) + 9 * (z == 0 ? 0 : (z == 9 ? 2 : 1));
      cv[tid] = (uint16_t)(c & ((row_meshed(q[0]) ? 1u : 0u) | (row_meshed(q[1]) ? 0x1FEu : 0u) |
                                        (row_meshed(q[2]) ? 0x200u : 0u)));
    }
    // Lower neighbours that are not meshed in this pass: the configurations that
    // their cubes beside this block hold count.
    const bool mixed = busy_[third][2] != 0;  // uniform
    if (mixed) {
      if (tid < 3 * 64) stored[tid] = 0u;
      __syncthreads();
      for (int s = (int)tid; s < kCfg * kCfg * kCfg; s += (int)kMcLanes) {
        const int x = s % kCfg - 1, y = (s / kCfg) % kCfg - 1, z = s / (kCfg * kCfg) - 1;
        const int dx = x < 0 ? -1 : 0, dy = y < 0 ? -1 : 0, dz = z < 0 ? -1 : 0;
        const int32_t q = nb[nb27(dx, dy, dz)];
        if (q < 0 || row_meshed(q)) continue;
        const uint32_t hc = V.cube[(size_t)q * kBlockVoxels + (x - 8 * dx) + 8 * (y - 8 * dy) + 64 * (z - 8 * dz)] & 255u;
        for (uint32_t m = etab[hc]; m; m &= m - 1u) {
          const int e = __ffs(m) - 1;
          const int ox = x + edge_owner_off(e, 0), oy = y + edge_owner_off(e, 1), oz = z + edge_owner_off(e, 2);
          if (min(min(ox, oy), oz) < 0 || max(max(ox, oy), oz) > 7) continue;
          atomicOr(&stored[64 * edge_axis(e) + oy + 8 * oz], 1u << ox);
          crossing = true;
        }
      }
    }
    if (__any(crossing) && (tid & 63u) == 0) busy_[third][1] = 1u;
    __syncthreads();
    if (!busy_[third][1]) {  // uniform: no crossed edge here or below, no slot held
      finish_empty(cube);
      continue;
    }
    // RecycleVerticesKernel on this block's own slots (marching_cubes.cu:
    // 303-321): a slot is referenced iff one of the four cubes around its edge
    // (this block and its lower neighbours, whose configurations are all
    // final above) crosses the edge: its ends differ and one of the cubes is
    // valid, or one that is not meshed here holds it.  Unreferenced allocated slots are freed
    // (to the free list; they go on the heap after the pass, so no pop of
    // this pass can take them).  The surfel counts are the slots allocated
    // once the pass's claims are done: allocated now, or referenced (a
    // referenced free slot is claimed in this pass, here or by a lower
    // neighbour).  No other workgroup touches an unreferenced slot.
    unsigned release = 0;
    {
      int inner = 0, boundary = 0;
#pragma unroll
      for (int r = 0; r < kMcVox; ++r) {
        const i3 o = devectorize(tid + kMcLanes * r);
        const bool is_inner = o.x >= 1 && o.y >= 1 && o.z >= 1 && o.x < 7 && o.y < 7 && o.z < 7;
        // the cubes at x - 1 (bit 0) and x of the rows y - {0, 1}, z - {0, 1}
        const int at = crow(o.y, o.z);
        const uint32_t m00 = cv[at] >> o.x, m10 = cv[at - 1] >> o.x, m01 = cv[at - kCubeHalo] >> o.x,
                       m11 = cv[at - kCubeHalo - 1] >> o.x;
        uint32_t used = cross[r] & (((m00 | m10 | m01 | m11) & 2u ? 1u : 0u) | ((m00 | m01) & 3u ? 2u : 0u) |
                                    ((m00 | m10) & 3u ? 4u : 0u));
        if (mixed)
#pragma unroll
          for (int a = 0; a < 3; ++a) used |= ((stored[64 * a + o.y + 8 * o.z] >> o.x) & 1u) << a;
        uint32_t held = 0;
#pragma unroll
        for (int a = 0; a < 3; ++a) held |= vps[r][a] >= 0 ? 1u << a : 0u;
        const int slots = __popc(held | used);
        if (is_inner) inner += slots;
        else boundary += slots;
        release |= (held & ~used) << (3 * r);
      }
      if (inner) atomicAdd(&surfels[0], inner);
      if (boundary) atomicAdd(&surfels[1], boundary);
    }
    {
      int delta = 0, assigned = 0;
#pragma unroll
      for (int r = 0; r < kMcVox; ++r) {
        const uint32_t prev = word[r] & 255u, nw = cube[r] | (prev << 8);
        if (nw != word[r]) V.cube[(size_t)self * kBlockVoxels + tid + kMcLanes * r] = (uint16_t)nw;
        // live triangles of a cube = its configuration's table row
        const int nt = ntab[cube[r]];
        delta += nt - ntab[prev];
        if (cube[r] != prev) assigned += nt;
      }
      if (delta) atomicAdd(&tri_sum[0], delta);
      if (assigned) atomicAdd(&tri_sum[1], assigned);
    }
    // The edges that the block's own valid cubes cross become a dense item list,
    // each once: a row of owner voxels (x 0..8 at some y, z in 0..8) has their x, y
    // and z edges from the rows of signs and of cubes.  (An item for each crossed
    // edge of each cube, four to a slot, took four times the claim rounds.)
    // The same scan ranks the freed slots (bits 13 and up: there are at most
    // 3 * 8 * 9 * 9 items).
    uint32_t free_rank, n_freed;
    {
      constexpr uint32_t kRows = kBlockSide + 1;
      static_assert(kRows * kRows <= 128 && kMcLanes >= 256, "the rows take the two waves that had no halo rows");
      const uint32_t row = tid - (kMcLanes - 128), ry = row % kRows, rz = row / kRows;
      uint32_t edges = 0;  // x edges in bits 0..7, y in 8..16, z in 17..25
      if (row < kRows * kRows) {
        const uint32_t at = (uint32_t)sidx(0, (int)ry, (int)rz);
        const uint32_t na = shell_bits(S.bits[kNeg], at), nu = shell_bits(S.bits[kNeg], at + kShell * kShell);
        // own valid cubes of the rows y - {0, 1}, z - {0, 1} (those outside the block count as none)
        const int c = crow((int)ry, (int)rz);
        const uint32_t y0 = ry < 8 ? 0xFFu : 0u, y1 = ry > 0 ? 0xFFu : 0u, z0 = rz < 8 ? 0xFFu : 0u, z1 = rz > 0 ? 0xFFu : 0u;
        const uint32_t v00 = (cv[c] >> 1) & y0 & z0, v10 = (cv[c - 1] >> 1) & y1 & z0,
                       v01 = (cv[c - kCubeHalo] >> 1) & y0 & z1, v11 = (cv[c - kCubeHalo - 1] >> 1) & y1 & z1;
        const uint32_t ey = v00 | v01, ez = v00 | v10;
        edges = ((na ^ (na >> 1)) & (ey | v10 | v11)) | ((na ^ (na >> kShell)) & (ey | ey << 1)) << 8 |
                ((na ^ nu) & (ez | ez << 1)) << 17;
      }
      static_assert(kMcVox <= 2, "at most 6 freed slots a lane");
      uint32_t total;
      const uint32_t at2 = block_excl_scan_planes<0x1Fu | (0x7u << 13)>((uint32_t)__popc(release) << 13 | (uint32_t)__popc(edges),
                                                                       scan_wave, &total);
      uint32_t at = at2 & 8191u;
      free_rank = at2 >> 13;
      for (; edges; edges &= edges - 1u) {
        const uint32_t k = (uint32_t)__ffs((int)edges) - 1u, ax = k >= 17 ? 2u : (k >= 8 ? 1u : 0u);
        items[at++] = (uint16_t)((k - (ax == 2 ? 17u : 8u * ax)) | (ry << 4) | (rz << 8) | (ax << 12));
      }
      if (threadIdx.x == 0) nitems = total & 8191u;
      n_freed = total >> 13;
    }
    // the freed slots' place on the list, waited for after the claims
    uint32_t base_got = 0;
    if (threadIdx.x == 0 && n_freed) base_got = atomicAdd(&V.ctr->vfree_count, n_freed);
    __syncthreads();
    const uint32_t n_items = nitems;
    if (threadIdx.x == 0) {
      V.surfel[2 * self + 0] = surfels[0];
      V.surfel[2 * self + 1] = surfels[1];
      cnt.delta += tri_sum[0];
      cnt.assigned += (uint32_t)tri_sum[1];
    }
    for (uint32_t c0 = 0;; c0 += kMcLanes) {
      // Vertex slot of each item: read it; claim it if free (CAS to the
      // lock value); pop fresh vertices for all claims of the workgroup
      // with one heap operation; publish them.
      const uint32_t jt = c0 + tid;
      const bool has = jt < n_items;
      uint32_t it = 0;  // a vertex's key: owner voxel and axis
      int32_t* slot = nullptr;
      int32_t cur = kFreePtr;
      bool claimed = false;
      if (has) {
        it = items[jt];
        const uint32_t x = it & 15u, y = (it >> 4) & 15u, z = (it >> 8) & 15u;
        const int32_t optr = row_ptr(nb[13 + (x >> 3) + 3 * (y >> 3) + 9 * (z >> 3)]);
        slot = &V.vptr[((size_t)optr * kBlockVoxels + ((x & 7u) | (y & 7u) << 3 | (z & 7u) << 6)) * 3 + (it >> 12)];
        cur = *slot;
        if (cur == kFreePtr) {
          const int32_t old = atomicCAS(slot, kFreePtr, kLockPtr);
          claimed = old == kFreePtr;
          if (!claimed) cur = old;
        }
      }
      uint32_t nclaims;
      const uint32_t rank = block_excl_scan<1>(claimed ? 1u : 0u, scan_wave, &nclaims);
      if (nclaims) {  // uniform
        if (threadIdx.x == 0) {
          const int32_t top = atomicSub(&V.ctr->vertex_top, (int32_t)nclaims);
          const int32_t avail = top + 1 > 0 ? top + 1 : 0;
          if (avail < (int32_t)nclaims) {
            atomicAdd(&V.ctr->vertex_top, (int32_t)nclaims - avail);
            atomicOr(&V.ctr->flags, MH_STATUS_VERTEX_HEAP_EXHAUSTED);
          }
          pop_top = top;
        }
        __syncthreads();
        if (claimed) {
          const int32_t hidx = pop_top - (int32_t)rank;
          const int32_t fresh = hidx >= 0 ? V.vertex_heap[hidx] : kFreePtr;
          atomicExch(slot, fresh);
          cur = fresh;
        }
      }
      if (has && cur >= 0) {
        // writer rule: of the four cubes around the edge, in the order (0, 0),
        // (1, 0), (0, 1), (1, 1) of the offsets in the two other axes, the first
        // that is valid and meshed in this pass; `first` is its bit, `own` those of
        // the cubes of this block
        const int x = (int)(it & 15u), y = (int)((it >> 4) & 15u), z = (int)((it >> 8) & 15u), ax = (int)(it >> 12);
        uint32_t first = 0, own = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int d1 = k & 1, d2 = k >> 1;
          const int qx = x - (ax != 0 ? d1 : 0), qy = y - (ax == 0 ? d1 : (ax == 2 ? d2 : 0)), qz = z - (ax != 2 ? d2 : 0);
          first |= (((uint32_t)cv[crow(qy, qz)] >> (qx + 1)) & 1u) << k;
          own |= ((qx | qy | qz) & ~7) == 0 ? 1u << k : 0u;
        }
        first &= 0u - first;
        // A slot claimed in this pass is also written by its claimer: the
        // designated cube may have read it while still locked and skipped it.
        const bool writer = claimed || (first & own) != 0;
        if (writer) {  // queue the payload; all lanes of the block work the queue
          const uint32_t q = atomicAdd(&qn, 1u);
          qptr[q] = cur;
          qkey[q] = (uint16_t)it;
        }
      }
      if (threadIdx.x == 0 && c0 == 0 && n_freed) free_base = base_got;
      __syncthreads();
      if (c0 == 0 && n_freed) {  // uniform
#pragma unroll
        for (int r = 0; r < kMcVox; ++r)
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            if (!((release >> (3 * r + a)) & 1u)) continue;
            const int32_t vp = vps[r][a];
            Vertex zv{};
            V.vertices[vp] = zv;
            V.vptr[3 * ((size_t)self * kBlockVoxels + tid + kMcLanes * r) + a] = kFreePtr;
            V.vfree[free_base + free_rank] = vp;
            ++free_rank;
          }
      }
      const bool last = c0 + kMcLanes >= n_items;  // uniform
      if (!last && qn + kMcLanes <= kQueue) continue;
      // payloads, four lanes per vertex, kPayRound vertices a round; then a wave
      // for their normals and one for the rest (other waves each time)
      const uint32_t nq = qn;
      cnt.writes += nq;
      const uint32_t jl = tid >> 2, lane = tid & 63u, wave = tid >> 6;
      for (uint32_t j0 = 0; j0 < nq; j0 += kPayRound, turns += 2) {  // uniform
        const uint32_t j = j0 + jl;
        if (j < nq &&  // the same for a vertex's four lanes
            payload_part<PSDF>(S, V.geo, mc, inv_vs, axes, base, qkey[j], tid & 3u, jl, pay))
          flag(V, MH_STATUS_STENCIL_RANGE);
        __syncthreads();
        const uint32_t role = (wave + turns) & 3u;
        if (j0 + lane < nq) {
          if (role == 0) finish_normal<PSDF>(V, qptr[j0 + lane], lane, pay);
          if (role == 1) finish_sample<PSDF>(S, V, base, qptr[j0 + lane], lane, pay);
        }
        __syncthreads();
      }
      if (last) break;
      if (threadIdx.x == 0) qn = 0;
      __syncthreads();
    }
    advance();
  }
  if (threadIdx.x == 0) cnt.flush(src.view(cur_scene));
}

// Meshed-in-this-pass marks for the writer rule.
template <class Src>
__global__ void mc_mark_kernel(Src src_, const SceneFrame* __restrict__ tab, McConst mc1) {
  const Src src = with_table(src_, tab);
  const uint32_t n = src.count();
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    uint32_t scene;
    const int32_t ptr = src.lane_item(i, &scene);
    src.view(scene).block_mark[ptr] = mc_of(src, scene, mc1).pass;
  }
}

// ---------------------------------------------------------------- pass 2
// The reference's TriangleExtractionKernel (marching_cubes.cu:180-275) and
// RecycleTrianglesKernel (:278-301) maintain a triangle pool: after a pass
// every processed cube holds exactly the triangles of its configuration's
// table row, over the vertices of its active edges, and keeps them until it
// is processed again.  That state is already held by the cube configuration
// and the per-voxel vertex slots, so the mesh is kept implicitly: no pool,
// no per-triangle writes, no reference-count atomics.  The triangle list
// is materialised only when the mesh is read out (dumps, compaction).  A
// vertex's reference count is likewise the sum over the four cubes around
// its edge of how many of their table triangles use that edge (edge_refs).
//
// RecycleVerticesKernel (marching_cubes.cu:303-321) frees a block's
// vertices with no references and produces its inner/boundary surfel counts
// (TriangleExtractionKernel counts the allocated vertex slots before
// recycling, :187-205).  The surfel pass does this for the blocks it meshes;
// this kernel does it for a list of other blocks (the garbage blocks, after
// their cubes lost their triangles).  Cube configurations of the block and of
// its -x/-y/-z neighbours (voxels -1..7) are staged in LDS.
template <class Src>
__global__ __launch_bounds__(256) void mc_recycle_vertices_kernel(Src src_, const SceneFrame* __restrict__ tab) {
  const Src src = with_table(src_, tab);
  __shared__ int32_t nb[8];  // blocks at offsets (dx, dy, dz) in {-1, 0}^3
  // edges used by the triangles of each staged cube's configuration
  __shared__ uint16_t cfg[kCfg * kCfg * kCfg];
  __shared__ uint16_t emask[256];
  __shared__ int counts[2];
  __shared__ uint32_t wave_sums[4];
  __shared__ int32_t push_top;
  const uint32_t n = src.count();
  static_assert(kBlockVoxels == 2 * 256, "two voxels per lane");
  // A configuration's table row uses exactly the edges of kMc.edges (its
  // crossed edges), so a vertex has references iff one of the four cubes
  // around its edge has that edge's bit set (edge_refs > 0).
  emask[threadIdx.x] = kMc.edges[threadIdx.x];
  for (uint32_t ci = blockIdx.x; ci < n; ci += gridDim.x) {
    uint32_t scene;
    const int32_t ptr = src.item(ci, &scene);
    const View V = src.view(scene);  // a copy: read once, not reloaded after stores
    // This lane's vertex slots (voxels threadIdx.x and threadIdx.x + 256);
    // a block without any is done at once (no slot to free, no surfels).
    int32_t vps[2][3];
    bool any = false;
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int ax = 0; ax < 3; ++ax) {
        vps[r][ax] = V.vptr[3 * ((size_t)ptr * kBlockVoxels + threadIdx.x + 256u * r) + ax];
        any = any || vps[r][ax] >= 0;
      }
    if (!__syncthreads_or(any)) {
      if (threadIdx.x == 0) {
        V.surfel[2 * ptr + 0] = 0;
        V.surfel[2 * ptr + 1] = 0;
      }
      continue;
    }
    if (threadIdx.x < 8) {
      const int t = (int)threadIdx.x;
      if (t == 0) {
        nb[t] = ptr;
      } else {
        const i3 b = unpack_key(V.block_keys[ptr]);
        nb[t] = hash_find(V, i3{b.x - (t & 1), b.y - ((t >> 1) & 1), b.z - ((t >> 2) & 1)});
      }
    }
    if (threadIdx.x == 0) { counts[0] = 0; counts[1] = 0; }
    __syncthreads();
    {  // all of a lane's loads in flight together (256 lanes)
      constexpr int kPer = (kCfg * kCfg * kCfg + 255) / 256;
      uint16_t cw[kPer];
#pragma unroll
      for (int r = 0; r < kPer; ++r) {
        const int s = (int)threadIdx.x + 256 * r;
        cw[r] = 0;
        if (s >= kCfg * kCfg * kCfg) continue;
        const int x = s % kCfg - 1, y = (s / kCfg) % kCfg - 1, z = s / (kCfg * kCfg) - 1;
        const int nx = x < 0, ny = y < 0, nz = z < 0;
        const int32_t cp = nb[nx + 2 * ny + 4 * nz];
        if (cp >= 0) cw[r] = V.cube[(size_t)cp * kBlockVoxels + (x + 8 * nx) + 8 * (y + 8 * ny) + 64 * (z + 8 * nz)];
      }
#pragma unroll
      for (int r = 0; r < kPer; ++r) {
        const int s = (int)threadIdx.x + 256 * r;
        if (s < kCfg * kCfg * kCfg) cfg[s] = emask[cw[r] & 255];
      }
    }
    __syncthreads();
    int inner = 0, boundary = 0;
    unsigned release = 0;  // bit 3r + ax: slot to free
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const uint32_t i = threadIdx.x + 256u * r;
      const i3 o = devectorize(i);
      const bool is_inner = o.x >= 1 && o.y >= 1 && o.z >= 1 && o.x < 7 && o.y < 7 && o.z < 7;
#pragma unroll
      for (int ax = 0; ax < 3; ++ax) {
        const int32_t vp = vps[r][ax];
        bool used = false;
        if (vp >= 0) {
          if (is_inner) ++inner; else ++boundary;
          const int b1 = ax == 0 ? 1 : 0, b2 = ax == 2 ? 1 : 2;
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            int d[3] = {0, 0, 0};
            d[b1] = k & 1;
            d[b2] = k >> 1;
            const unsigned m = cfg[(o.x - d[0] + 1) + kCfg * (o.y - d[1] + 1) + kCfg * kCfg * (o.z - d[2] + 1)];
            used |= ((m >> edge_with(d[0], d[1], d[2], ax)) & 1u) != 0;
          }
        }
        // (the reference count itself is not stored: readers derive it with
        // edge_refs)
        if (vp >= 0 && !used) release |= 1u << (3 * r + ax);
      }
    }
    // the block's freed slots go back to the heap with one counter update
    uint32_t nfree;
    uint32_t rank = block_excl_scan<3>((uint32_t)__popc(release), wave_sums, &nfree);  // <= 6
    if (nfree) {  // uniform
      if (threadIdx.x == 0) push_top = atomicAdd(&V.ctr->vertex_top, (int32_t)nfree);
      __syncthreads();
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
          if (!((release >> (3 * r + ax)) & 1u)) continue;
          const int32_t vp = vps[r][ax];
          Vertex z{};
          V.vertices[vp] = z;
          V.vptr[3 * ((size_t)ptr * kBlockVoxels + threadIdx.x + 256u * r) + ax] = kFreePtr;
          V.vertex_heap[push_top + 1 + (int32_t)rank] = vp;
          ++rank;
        }
    }
    if (inner) atomicAdd(&counts[0], inner);
    if (boundary) atomicAdd(&counts[1], boundary);
    __syncthreads();
    if (threadIdx.x == 0) {
      V.surfel[2 * ptr + 0] = counts[0];
      V.surfel[2 * ptr + 1] = counts[1];
    }
    __syncthreads();
  }
}

// The vertex slots the surfel pass freed go on the heap once the pass is over,
// so that no claim of the pass could pop one (pops and pushes of one stack
// cannot overlap).  Workgroups (x, scene y) copy strided parts of the scene's
// free list above the top; the last to finish moves the top.
template <class Src>
__global__ __launch_bounds__(256) void mc_push_freed_kernel(Src src_, const SceneFrame* __restrict__ tab) {
  const Src src = with_table(src_, tab);
  const View& V = src.view(blockIdx.y);
  // both unchanged until every workgroup of the scene has counted itself done
  const uint32_t n = V.ctr->vfree_count;
  const int32_t top = V.ctr->vertex_top;
  // no slot went back during the pass: the heap is at its lowest since the last
  if (blockIdx.x == 0 && threadIdx.x == 0) V.ctr->vertex_low = min(V.ctr->vertex_low, top);
  if (n == 0) return;  // the same for all of the scene's workgroups
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    V.vertex_heap[top + 1 + (int32_t)i] = V.vfree[i];
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence();
    if (atomicAdd(&V.ctr->vfree_done, 1u) == gridDim.x - 1) {
      V.ctr->vertex_top = top + (int32_t)n;
      V.ctr->vfree_count = 0;
      V.ctr->vfree_done = 0;
    }
  }
}
constexpr int kPushGrid = 64;  // workgroups per scene

// ---------------------------------------------------------------- recycling
// RecycleGarbageTrianglesKernel (mapping/recycle.cu:117-141): the garbage
// blocks' cubes lose their triangles (current configuration 0; the previous
// one stays in the high byte), so the reference counts of their vertices
// drop accordingly; RecycleGarbageVerticesKernel (:143-179) then frees the
// blocks' own vertex slots left without references (the MC recycle kernel
// over the garbage list).
__global__ __launch_bounds__(512) void gc_release_kernel(View V) {
  const uint32_t n = V.ctr->gc_count;
  int delta = 0;
  for (uint32_t ci = blockIdx.x; ci < n; ci += gridDim.x) {
    const size_t idx = (size_t)V.gc_list[ci] * kBlockVoxels + threadIdx.x;
    const uint32_t c = V.cube[idx] & 255u;
    V.cube[idx] = (uint16_t)(c << 8);
    delta -= (c == 0 || c == 255) ? 0 : kMc.ntri[c];
  }
  for (int off = 32; off > 0; off >>= 1) delta += __shfl_xor(delta, off);
  if ((threadIdx.x & 63u) == 0 && delta)
    atomicAdd(&work_stripe(V.ctr).tri_live, (unsigned long long)(long long)delta);
}

void launch_gc_release_triangles(const View& V, hipStream_t s, int grid) {
  gc_release_kernel<<<grid, 512, 0, s>>>(V);
}

// ---------------------------------------------------------------- compaction
// CompressMesh (visualization/compress_mesh.cu:10-172) over the implicit
// mesh: the live triangles of a worklist block are its cubes' table rows;
// a triangle is kept when all three vertex slots are allocated.  Pass 1
// counts triangles per block and marks the vertex slots they use; after
// exclusive scans (triangles over the worklist, used slots over the vertex
// pool) pass 2 writes triangles in worklist x voxel x slot order with the
// vertices renumbered in pool order, and the used vertices are gathered.

// Vertex pool index of edge e of the cube at local voxel o, -1 if its slot is
// not allocated.  nb holds the blocks at offsets {0, 1}^3 (x + 2y + 4z).
__device__ __forceinline__ int32_t cube_edge_vertex(const View& V, const int32_t* nb, i3 o, int e) {
  const int ox = o.x + edge_owner_off(e, 0), oy = o.y + edge_owner_off(e, 1), oz = o.z + edge_owner_off(e, 2);
  const int dx = ox >> 3, dy = oy >> 3, dz = oz >> 3;
  const int32_t bp = nb[dx + 2 * dy + 4 * dz];
  if (bp < 0) return -1;
  const uint32_t li = (uint32_t)((ox - 8 * dx) + 8 * (oy - 8 * dy) + 64 * (oz - 8 * dz));
  return V.vptr[((size_t)bp * kBlockVoxels + li) * 3 + edge_axis(e)];
}

template <bool EMIT>
__global__ __launch_bounds__(512) void compact_tris_kernel(View V, uint32_t n, uint32_t* __restrict__ used,
                                                           uint32_t* __restrict__ blk_tris,
                                                           const uint32_t* __restrict__ blk_off,
                                                           const uint32_t* __restrict__ remap,
                                                           int32_t* __restrict__ tri_out) {
  __shared__ int32_t nb[8];
  __shared__ uint32_t wave_sums[8];
  for (uint32_t ci = blockIdx.x; ci < n; ci += gridDim.x) {
    const int32_t ptr = V.cand[ci];
    const i3 b = unpack_key(V.block_keys[ptr]);
    if (threadIdx.x < 8) {
      const int t = (int)threadIdx.x;
      nb[t] = t == 0 ? ptr : hash_find(V, i3{b.x + (t & 1), b.y + ((t >> 1) & 1), b.z + ((t >> 2) & 1)});
    }
    __syncthreads();
    const uint32_t i = threadIdx.x;
    const i3 o = devectorize(i);
    const int c = V.cube[(size_t)ptr * kBlockVoxels + i] & 255;
    const int nt = (c == 0 || c == 255) ? 0 : kMc.ntri[c];
    uint32_t keep = 0;
    for (int t = 0; t < nt; ++t) {
      int32_t vp[3];
      bool ok = true;
      for (int k = 0; k < 3; ++k) {
        vp[k] = cube_edge_vertex(V, nb, o, kMc.tri[c][3 * t + k]);
        ok = ok && vp[k] >= 0;
      }
      if (!ok) continue;
      if (!EMIT) {
        for (int k = 0; k < 3; ++k) used[vp[k]] = 1u;
      } else {
        // slot within the block filled below after the scan
      }
      ++keep;
    }
    uint32_t total;
    const uint32_t excl = block_excl_scan<3>(keep, wave_sums, &total);  // keep <= 5
    if (!EMIT) {
      if (threadIdx.x == 0) blk_tris[ci] = total;
    } else {
      uint32_t at = blk_off[ci] + excl;
      for (int t = 0; t < nt; ++t) {
        int32_t vp[3];
        bool ok = true;
        for (int k = 0; k < 3; ++k) {
          vp[k] = cube_edge_vertex(V, nb, o, kMc.tri[c][3 * t + k]);
          ok = ok && vp[k] >= 0;
        }
        if (!ok) continue;
        for (int k = 0; k < 3; ++k) tri_out[3 * (size_t)at + k] = (int32_t)remap[vp[k]];
        ++at;
      }
    }
    __syncthreads();
  }
}

__global__ __launch_bounds__(256) void compact_vertices_kernel(View V, const uint32_t* __restrict__ used,
                                                               const uint32_t* __restrict__ remap,
                                                               float* __restrict__ pos, float* __restrict__ nrm,
                                                               float* __restrict__ col, uint32_t nv) {
  for (uint32_t vp = blockIdx.x * blockDim.x + threadIdx.x; vp < nv; vp += gridDim.x * blockDim.x) {
    if (!used[vp]) continue;
    const size_t j = remap[vp];
    const Vertex& x = V.vertices[vp];
    pos[3 * j + 0] = x.px; pos[3 * j + 1] = x.py; pos[3 * j + 2] = x.pz;
    nrm[3 * j + 0] = x.nx; nrm[3 * j + 1] = x.ny; nrm[3 * j + 2] = x.nz;
    col[3 * j + 0] = x.cr; col[3 * j + 1] = x.cg; col[3 * j + 2] = x.cb;
  }
}

// Exclusive scan of n uint32 (three launches: 1024-element chunks, the chunk
// sums in one workgroup, then the chunk offsets added back).
constexpr uint32_t kScanChunk = 1024;
__global__ __launch_bounds__(1024) void scan_chunks_kernel(const uint32_t* __restrict__ in,
                                                           uint32_t* __restrict__ out, uint32_t n,
                                                           uint32_t* __restrict__ chunk_sums) {
  __shared__ uint32_t ws[16];
  const uint32_t i = blockIdx.x * kScanChunk + threadIdx.x;
  const uint32_t v = i < n ? in[i] : 0u;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint32_t x = v;
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(x, off);
    if (lane >= (uint32_t)off) x += y;
  }
  if (lane == 63) ws[wave] = x;
  __syncthreads();
  uint32_t before = 0, all = 0;
  for (uint32_t w = 0; w < 16; ++w) {
    if (w < wave) before += ws[w];
    all += ws[w];
  }
  if (i < n) out[i] = before + x - v;
  if (threadIdx.x == 0) chunk_sums[blockIdx.x] = all;
}

__global__ __launch_bounds__(1024) void scan_sums_kernel(uint32_t* __restrict__ sums, uint32_t nchunks,
                                                         uint32_t* __restrict__ total) {
  __shared__ uint32_t ws[16];
  __shared__ uint32_t carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  for (uint32_t base = 0; base < nchunks; base += kScanChunk) {
    const uint32_t i = base + threadIdx.x;
    const uint32_t v = i < nchunks ? sums[i] : 0u;
    uint32_t x = v;
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t y = __shfl_up(x, off);
      if (lane >= (uint32_t)off) x += y;
    }
    if (lane == 63) ws[wave] = x;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (uint32_t w = 0; w < 16; ++w) {
      if (w < wave) before += ws[w];
      all += ws[w];
    }
    const uint32_t c = carry;
    if (i < nchunks) sums[i] = c + before + x - v;
    __syncthreads();
    if (threadIdx.x == 0) carry = c + all;
    __syncthreads();
  }
  if (threadIdx.x == 0) *total = carry;
}

__global__ __launch_bounds__(1024) void scan_add_kernel(uint32_t* __restrict__ out, uint32_t n,
                                                        const uint32_t* __restrict__ sums) {
  const uint32_t i = blockIdx.x * kScanChunk + threadIdx.x;
  if (i < n) out[i] += sums[blockIdx.x];
}

void launch_scan(const uint32_t* in, uint32_t* out, uint32_t n, uint32_t* chunk_sums,
                 uint32_t* total, hipStream_t s) {
  const uint32_t nchunks = n ? (n + kScanChunk - 1) / kScanChunk : 1;
  scan_chunks_kernel<<<nchunks, kScanChunk, 0, s>>>(in, out, n, chunk_sums);
  scan_sums_kernel<<<1, kScanChunk, 0, s>>>(chunk_sums, nchunks, total);
  scan_add_kernel<<<nchunks, kScanChunk, 0, s>>>(out, n, chunk_sums);
}

void launch_compact_count(const View& V, uint32_t n, uint32_t* used, uint32_t* blk_tris,
                          hipStream_t s, int grid) {
  compact_tris_kernel<false><<<grid, 512, 0, s>>>(V, n, used, blk_tris, nullptr, nullptr, nullptr);
}

void launch_compact_emit(const View& V, uint32_t n, const uint32_t* blk_off, const uint32_t* remap,
                         int32_t* tri_out, const uint32_t* used, float* pos, float* nrm, float* col,
                         hipStream_t s, int grid) {
  compact_tris_kernel<true><<<grid, 512, 0, s>>>(V, n, nullptr, nullptr, blk_off, remap, tri_out);
  compact_vertices_kernel<<<grid, 256, 0, s>>>(V, used, remap, pos, nrm, col, V.max_vertices);
}

// Workgroups of persistent kernel K (THREADS lanes) resident at once: cus x
// the occupancy the runtime reports for it (queried once per kernel).  A
// persistent grid of exactly that spreads its items over one round of
// workgroups; a larger one would run its surplus as a second, partial round.
template <auto K, int THREADS>
int resident_grid(int cus) {
  static const int per_cu = [] {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, K, THREADS, 0) != hipSuccess || n < 1) n = 1;
    return n;
  }();
  return per_cu * cus;
}

// Surfel-pass grid: shape.grid_per_cu workgroups per CU (0: as many as are
// resident), at most the resident count.
template <auto K>
int surfel_grid(int cus, const McShape& shape) {
  const int resident = resident_grid<K, (int)kMcLanes>(cus);
  const int g = shape.grid_per_cu > 0 ? shape.grid_per_cu * cus : resident;
  return g < resident ? g : resident;
}

void launch_marching_cubes(const View& V, const McConst& p, int32_t* nbt, hipStream_t s, int cus,
                           const KernelClock* kc, McShape shape) {
  const int grid = V.va ? surfel_grid<mc_surfel_kernel<true, One>>(cus, shape)
                        : surfel_grid<mc_surfel_kernel<false, One>>(cus, shape);
  const uint32_t q = (uint32_t)shape.static_quarters;
  tick(kc, s, "mc_mark_kernel");
  mc_mark_kernel<<<cus, 256, 0, s>>>(One{V}, nullptr, p);
  tick(kc, s, "mc_neighbours_kernel");
  mc_neighbours_kernel<<<cus * 8, 256, 0, s>>>(One{V}, nullptr, p, nbt);
  tick(kc, s, "mc_surfel_kernel");
  if (V.va)
    mc_surfel_kernel<true><<<grid, kMcLanes, 0, s>>>(One{V}, nullptr, p, nbt, q);
  else
    mc_surfel_kernel<false><<<grid, kMcLanes, 0, s>>>(One{V}, nullptr, p, nbt, q);
  tick(kc, s, "mc_push_freed_kernel");
  mc_push_freed_kernel<<<kPushGrid, 256, 0, s>>>(One{V}, nullptr);
  tick(kc, s, nullptr);
}

void launch_gc_recycle_vertices(const View& V, hipStream_t s, int cus) {
  mc_recycle_vertices_kernel<<<resident_grid<mc_recycle_vertices_kernel<Listed>, 256>(cus), 256, 0, s>>>(
      Listed{V, V.gc_list, &V.ctr->gc_count}, nullptr);
}

void launch_batch_marching_cubes(const BatchDev& B, int32_t* nbt, hipStream_t s, int cus, McShape shape,
                                 bool marks_stamped) {
  const McConst unused{};
  const int grid = B.psdf ? surfel_grid<mc_surfel_kernel<true, Many>>(cus, shape)
                          : surfel_grid<mc_surfel_kernel<false, Many>>(cus, shape);
  const uint32_t q = (uint32_t)shape.static_quarters;
  if (!marks_stamped) mc_mark_kernel<<<cus, 256, 0, s>>>(B.src(), B.frames, unused);
  mc_neighbours_kernel<<<cus * 8, 256, 0, s>>>(B.src(), B.frames, unused, nbt);
  if (B.psdf)
    mc_surfel_kernel<true><<<grid, kMcLanes, 0, s>>>(B.src(), B.frames, unused, nbt, q);
  else
    mc_surfel_kernel<false><<<grid, kMcLanes, 0, s>>>(B.src(), B.frames, unused, nbt, q);
  mc_push_freed_kernel<<<dim3(kPushGrid, B.nscenes), 256, 0, s>>>(B.src(), B.frames);
}

}  // namespace mh
