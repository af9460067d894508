// primal_dual.hip -- TV/Huber primal-dual denoising of the fused SDF.
//
// Reference: optimize/primal_dual.cu:10-223 (PrimalDualInitKernel,
// PrimalDualIteratePass1Kernel, PrimalDualIteratePass2Kernel, Huber),
// geometry/primal_dual_query.h:15-234 (forward-difference gradients,
// backward-difference divergence), core/voxel.h:62-82 (PrimalDualVariables).
//
// MI355X layout: the six face neighbours of every worklist block are looked
// up once per solve into a table (the block set does not change while
// iterating), so a stencil access outside the block is one table read plus a
// voxel read instead of a hash probe.  A fused model's blocks are sparse (of a
// 2 cm probabilistic room's 17.5 M voxels 23 % are observed and 17 % ever hold
// a dual variable, in 53 % and 19 % of the 64-byte sectors), so an iteration
// first packs the weights and masks into two bits a voxel; the passes take
// their stencils' validity from those, eight voxels at a time, and go over
// the voxels that matter only, one wave a block.  50 iterations of that room
// took 15.4 ms when each voxel's lane followed its own weights and masks
// (150 us a pass: 72 % of the lanes idle behind six dependent loads); 5.3 ms
// so (bits 16 us, pass 1 33 us, pass 2 53 us an iteration).
// Both passes are Jacobi steps; the energies are reduced per workgroup into
// FP64 partials and summed in a fixed order, so the whole iteration is
// deterministic.
#include <cmath>

#include "mh_kernels.h"

namespace mh {

// EPSILON is the double literal 1e-6 (core/common.h:60): float weights are
// widened before the comparison.
__device__ __forceinline__ bool below_eps(float w) { return (double)w < 1e-6; }
__device__ __forceinline__ bool above_eps(float w) { return (double)w > 1e-6; }

// A neighbour that is not on the worklist itself: its bits are not packed.
constexpr int32_t kPdOutside = 1 << 30;

// Where each block stands on the worklist.
__global__ __launch_bounds__(256) void pd_index_kernel(View V, uint32_t* index) {
  const uint32_t n = V.ctr->cand_count;
  for (uint32_t c = blockIdx.x * blockDim.x + threadIdx.x; c < n; c += gridDim.x * blockDim.x) index[V.cand[c]] = c;
}

// Face-neighbour table: nbr[6*c + k], k = +x, +y, +z, -x, -y, -z.
__global__ __launch_bounds__(256) void pd_neighbors_kernel(View V, int32_t* nbr, const uint32_t* index) {
  const uint32_t n = V.ctr->cand_count;
  const uint32_t gid = blockIdx.x * blockDim.x + threadIdx.x;
  for (uint32_t j = gid; j < 6 * n; j += gridDim.x * blockDim.x) {
    const uint32_t c = j / 6, k = j % 6;
    const i3 b = unpack_key(V.block_keys[V.cand[c]]);
    const int s = k < 3 ? 1 : -1;
    const int ax = (int)(k % 3);
    const i3 q = i3{b.x + (ax == 0 ? s : 0), b.y + (ax == 1 ? s : 0), b.z + (ax == 2 ? s : 0)};
    int32_t p = hash_find(V, q);
    if (p >= 0) {
      const uint32_t at = index[p];  // of an earlier worklist, if p is not on this one
      if (!(at < n && V.cand[at] == p)) p |= kPdOutside;
    }
    nbr[j] = p;
  }
}

// Address of the voxel at local offset o + d (d one of +-e_k), or -1 when
// its block is not allocated.
__device__ __forceinline__ int64_t nb_index(const int32_t* nbr6, int32_t self, i3 o, int ax,
                                            int s) {
  int c[3] = {o.x, o.y, o.z};
  c[ax] += s;
  int32_t p = self;
  if (c[ax] < 0 || c[ax] > 7) {
    p = nbr6[s > 0 ? ax : 3 + ax];
    c[ax] -= 8 * s;
    if (p < 0) return -1;
    p &= ~kPdOutside;
  }
  return (int64_t)p * kBlockVoxels + c[0] + 8 * c[1] + 64 * c[2];
}

// PrimalDualInitKernel (primal_dual.cu:15-43) with GetInitSDFGradient
// (primal_dual_query.h:44-86).
__global__ __launch_bounds__(256) void pd_init_kernel(View V, const int32_t* nbr, uint8_t* dual) {
  const uint32_t n = V.ctr->cand_count;
  const float vs = V.geo.voxel_size;
  for (uint32_t ci = blockIdx.x; ci < n; ci += gridDim.x) {
    const int32_t ptr = V.cand[ci];
    const int32_t* nb = nbr + 6 * ci;
    for (uint32_t i = threadIdx.x; i < (uint32_t)kBlockVoxels; i += blockDim.x) {
      const size_t idx = (size_t)ptr * kBlockVoxels + i;
      const bool live = !below_eps(V.weight[idx]);
      const uint64_t zeroed = __ballot(live);  // 64 consecutive voxels: eight rows
      if ((threadIdx.x & 63) == 0) reinterpret_cast<uint64_t*>(dual)[idx >> 6] &= ~zeroed;
      if (!live) continue;
      const i3 o = devectorize(i);
      const float c = V.sdf[idx];
      float g[3] = {0.0f, 0.0f, 0.0f};
      bool ok = true;
      for (int k = 0; k < 3 && ok; ++k) {
        const int64_t j = nb_index(nb, ptr, o, k, +1);
        if (j < 0 || below_eps(V.weight[j])) {
          ok = false;
          break;
        }
        g[k] = V.sdf[j];
      }
      const f3 grad = ok ? mk3(g[0] - c, g[1] - c, g[2] - c) : mk3(0.0f, 0.0f, 0.0f);
      V.pd_p[3 * idx + 0] = 0.0f;
      V.pd_p[3 * idx + 1] = 0.0f;
      V.pd_p[3 * idx + 2] = 0.0f;
      V.pd_sdf_bar[idx] = 0.0f;
      V.pd_w[idx] = expf(length(grad) / vs);
      V.pd_sdf0[idx] = c;
      V.pd_mask[idx] = 1;
    }
  }
}

__device__ __forceinline__ float huber(float x, float alpha) {
  return (fabsf(x) < alpha) ? 0.5f * (x * x) / alpha : (fabsf(x) - 0.5f * alpha);
}

__device__ __forceinline__ double block_sum(double v, double* red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < (int)(blockDim.x >> 6); ++w) s += red[w];
  __syncthreads();
  return s;
}

// A row is the eight voxels of one y and z of a block, a lane's share of a
// block: bit x of the low byte says that voxel x is observed, of the high byte
// that it is masked as well (a stencil may use it).
__device__ __forceinline__ uint32_t pd_row(const View& V, int32_t ptr, uint32_t row) {
  const size_t at = (size_t)ptr * kBlockVoxels + 8 * row;
  const float4 a = *reinterpret_cast<const float4*>(V.weight + at), b = *reinterpret_cast<const float4*>(V.weight + at + 4);
  const uint2 m = *reinterpret_cast<const uint2*>(V.pd_mask + at);
  const float w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  uint32_t live = 0, use = 0;
#pragma unroll
  for (int x = 0; x < 8; ++x) {
    live |= below_eps(w[x]) ? 0u : 1u << x;
    use |= (((x < 4 ? m.x : m.y) >> (8 * (x & 3))) & 255u) ? 1u << x : 0u;
  }
  return live | (live & use) << 8;
}
__global__ __launch_bounds__(256) void pd_bits_kernel(View V, uint16_t* bits) {
  const uint32_t n = V.ctr->cand_count, lane = threadIdx.x & 63;
  for (uint32_t c = blockIdx.x * 4 + (threadIdx.x >> 6); c < n; c += gridDim.x * 4) {
    const int32_t ptr = __builtin_amdgcn_readfirstlane(V.cand[c]);
    bits[(size_t)ptr * 64 + lane] = (uint16_t)pd_row(V, ptr, lane);
  }
}

// The usable voxels of row `row` of a neighbour (an entry of the table).
__device__ __forceinline__ uint32_t pd_face_row(const View& V, const uint16_t* bits, int32_t nb, uint32_t row) {
  if (nb < 0) return 0;
  if (nb & kPdOutside) return pd_row(V, nb & ~kPdOutside, row) >> 8;
  return (uint32_t)bits[(size_t)nb * 64 + row] >> 8;
}
// The voxels of a lane's row whose three neighbours at +S are usable, `use`
// being the row's own usable voxels and nb the neighbours on that side.
template <int S>
__device__ __forceinline__ uint32_t pd_stencils(const View& V, const uint16_t* bits, const int32_t nb[3], uint32_t use) {
  const uint32_t lane = threadIdx.x & 63, y = lane & 7, z = lane >> 3;
  const uint32_t fx = pd_face_row(V, bits, nb[0], lane);
  uint32_t my = (uint32_t)__shfl((int)use, (int)(lane + S) & 63), mz = (uint32_t)__shfl((int)use, (int)(lane + 8 * S) & 63);
  constexpr uint32_t kLast = S > 0 ? 7 : 0, kFirst = 7 - kLast;
  if (y == kLast) my = pd_face_row(V, bits, nb[1], 8 * z + kFirst);
  if (z == kLast) mz = pd_face_row(V, bits, nb[2], 8 * kFirst + y);
  const uint32_t mx = S > 0 ? (use >> 1) | (fx & 1u) << 7 : (use << 1) | (fx >> 7 & 1u);
  return mx & my & mz;
}
// The voxels `act` of a wave's block as a list in voxel order, those of `flag`
// with kPdFlag; returns their number.
constexpr uint32_t kPdFlag = 1u << 15;
__device__ __forceinline__ uint32_t pd_list(uint32_t act, uint32_t flag, uint16_t* list) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t own = (uint32_t)__popc(act);
  uint32_t end = own;
#pragma unroll
  for (uint32_t d = 1; d < 64; d <<= 1) {
    const uint32_t o = (uint32_t)__shfl_up((int)end, d);
    if (lane >= d) end += o;
  }
  uint32_t at = end - own;
  while (act) {
    const uint32_t x = (uint32_t)__ffs((int)act) - 1;
    list[at++] = (uint16_t)(lane * 8 + x | ((flag >> x) & 1u ? kPdFlag : 0u));
    act &= act - 1;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  return (uint32_t)__builtin_amdgcn_readlane((int)end, 63);
}
// The voxels next to voxel v of block ptr at +S (their blocks allocated).
template <int S>
__device__ __forceinline__ void pd_next(int32_t ptr, const int32_t nb[3], uint32_t v, size_t j[3]) {
  const uint32_t c[3] = {v & 7, (v >> 3) & 7, v >> 6}, stride[3] = {1, 8, 64};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const bool out = c[k] == (S > 0 ? 7u : 0u);
    const int32_t d = (int32_t)stride[k] * (out ? -7 * S : S);
    j[k] = (size_t)(out ? nb[k] & ~kPdOutside : ptr) * kBlockVoxels + (uint32_t)((int32_t)v + d);
  }
}

// PrimalDualIteratePass1Kernel (primal_dual.cu:45-109): energies, dual
// ascent p += sigma grad(sdf_bar), Huber shrink, projection onto |p| <= 1.
// The energies (ENERGY) are taken only when the caller asks for them: they
// need the field, its start and the field's three neighbours, which the dual
// step does not read.
//
// A voxel whose gradient is zeroed and whose dual variable is +0 keeps it, so
// only those with a valid stencil and those in `dual` are visited: bits of the
// voxels that have had a gradient since the solve began (`all`: a step size
// under which even +0 would change; then every observed voxel is).
template <bool ENERGY>
__global__ __launch_bounds__(256) void pd_pass1_kernel(View V, const int32_t* nbr, const uint16_t* __restrict__ bits,
                                                       uint8_t* __restrict__ dual, int all, float sigma, double* partials) {
  __shared__ double red[8];
  __shared__ uint16_t lists[4][kBlockVoxels];
  const float alpha = 0.02f;
  const uint32_t n = V.ctr->cand_count, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double e_data = 0.0, e_tv = 0.0;
  for (uint32_t c0 = blockIdx.x * 4 + wave; c0 < n; c0 += gridDim.x * 4) {
    const uint32_t ci = (uint32_t)__builtin_amdgcn_readfirstlane((int)c0);
    const int32_t ptr = V.cand[ci];
    const int32_t nb[3] = {nbr[6 * ci], nbr[6 * ci + 1], nbr[6 * ci + 2]};
    const size_t row = (size_t)ptr * 64 + lane;
    const uint32_t own = bits[row], had = dual[row];
    const uint32_t live = own & 255u;
    // GetSDFGradient (primal_dual_query.h:88-133) and GetPrimalGradient
    // (:189-234): forward differences; any missing, unobserved or
    // unmasked neighbour zeroes the whole gradient.
    const uint32_t ok = live & pd_stencils<1>(V, bits, nb, own >> 8);
    const uint32_t has = had | (all ? live : ok);
    if (has != had) dual[row] = (uint8_t)has;
    const uint32_t count = pd_list(ENERGY ? live : live & has, ok, lists[wave]);
    for (uint32_t t = lane; t < count; t += 64) {
      const uint32_t e = lists[wave][t], v = e & (kBlockVoxels - 1);
      const bool valid = (e & kPdFlag) != 0;
      const size_t idx = (size_t)ptr * kBlockVoxels + v;
      f3 p = mk3(V.pd_p[3 * idx], V.pd_p[3 * idx + 1], V.pd_p[3 * idx + 2]);
      f3 grad_b = mk3(0.0f, 0.0f, 0.0f), grad_s = grad_b;
      float sdf = 0.0f;
      if (ENERGY) sdf = V.sdf[idx];
      if (valid) {
        size_t j[3];
        pd_next<1>(ptr, nb, v, j);
        const float sb = V.pd_sdf_bar[idx];
        grad_b = mk3(V.pd_sdf_bar[j[0]] - sb, V.pd_sdf_bar[j[1]] - sb, V.pd_sdf_bar[j[2]] - sb);
        if (ENERGY) grad_s = mk3(V.sdf[j[0]] - sdf, V.sdf[j[1]] - sdf, V.sdf[j[2]] - sdf);
      }
      if (ENERGY) {
        float dd = fabsf(sdf - V.pd_sdf0[idx]);
        dd *= dd;
        if (above_eps(V.weight[idx])) e_data += (double)dd;
        e_tv += (double)huber(length(grad_s), alpha);
      }
      p = p + sigma * grad_b;
      p = p / (1.0f + sigma * alpha);
      const float len = fmaxf(1.0f, length(p));
      if (len > 1.0f) p = p / len;
      V.pd_p[3 * idx + 0] = p.x;
      V.pd_p[3 * idx + 1] = p.y;
      V.pd_p[3 * idx + 2] = p.z;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the list is read before the next one is written
  }
  if (ENERGY) {
    const double sd = block_sum(e_data, red);
    const double st = block_sum(e_tv, red);
    if (threadIdx.x == 0) {
      partials[2 * blockIdx.x + 0] = sd;
      partials[2 * blockIdx.x + 1] = st;
    }
  }
}

// PrimalDualIteratePass2Kernel (primal_dual.cu:111-151) with
// GetDualDivergence (primal_dual_query.h:135-187).  A field value that stays
// is not written (in that room 8 of 23 % of the voxels change none).
__global__ __launch_bounds__(256) void pd_pass2_kernel(View V, const int32_t* nbr, const uint16_t* __restrict__ bits,
                                                       float lambda, float tau) {
  __shared__ uint16_t lists[4][kBlockVoxels];
  const uint32_t n = V.ctr->cand_count, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (uint32_t c0 = blockIdx.x * 4 + wave; c0 < n; c0 += gridDim.x * 4) {
    const uint32_t ci = (uint32_t)__builtin_amdgcn_readfirstlane((int)c0);
    const int32_t ptr = V.cand[ci];
    const int32_t nb[3] = {nbr[6 * ci + 3], nbr[6 * ci + 4], nbr[6 * ci + 5]};
    const uint32_t own = bits[(size_t)ptr * 64 + lane];
    const uint32_t ok = (own >> 8) & pd_stencils<-1>(V, bits, nb, own >> 8);
    const uint32_t count = pd_list(own & 255u, ok, lists[wave]);
    for (uint32_t t = lane; t < count; t += 64) {
      const uint32_t e = lists[wave][t], v = e & (kBlockVoxels - 1);
      const size_t idx = (size_t)ptr * kBlockVoxels + v;
      const float prev = V.sdf[idx], w_pd = V.pd_w[idx], sdf0 = V.pd_sdf0[idx];
      float div = 0.0f;
      if (e & kPdFlag) {
        size_t j[3];
        pd_next<-1>(ptr, nb, v, j);
        const f3 pc = mk3(V.pd_p[3 * idx], V.pd_p[3 * idx + 1], V.pd_p[3 * idx + 2]);
        div = (V.pd_p[3 * j[0]] - pc.x) + (V.pd_p[3 * j[1] + 1] - pc.y) + (V.pd_p[3 * j[2] + 2] - pc.z);
      }
      const float lam = lambda * w_pd;
      float s = prev - tau * div;
      s = (s + lam * tau * sdf0) / (1.0f + lam * tau);
      if (w_pd > 2.0f) s = sdf0;
      if (__float_as_uint(s) != __float_as_uint(prev)) V.sdf[idx] = s;
      V.pd_sdf_bar[idx] = 2.0f * s - prev;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

// Sum of the per-workgroup partials, in an order fixed by n: a lane adds
// every 256th, then the lanes are added up in order.  (One lane adding all
// 2048 pairs was a chain of 183 us.)
__global__ __launch_bounds__(256) void pd_energy_kernel(const double* __restrict__ partials, uint32_t n, float lambda,
                                                        double* __restrict__ energy) {
  __shared__ double red[8];
  double d = 0.0, t = 0.0;
  for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
    d += partials[2 * i];
    t += partials[2 * i + 1];
  }
  d = block_sum(d, red);
  t = block_sum(t, red);
  if (threadIdx.x != 0) return;
  energy[0] = d;
  energy[1] = t;
  energy[2] = d * (double)lambda / 2.0 + t;
}

void launch_pd_init(const View& V, const PdTables& T, hipStream_t s, int grid) {
  pd_index_kernel<<<grid, 256, 0, s>>>(V, T.index);
  pd_neighbors_kernel<<<grid, 256, 0, s>>>(V, T.nbr, T.index);
  pd_init_kernel<<<grid, 256, 0, s>>>(V, T.nbr, T.dual);
}
// A wave's blocks hold from none to 512 observed voxels: four times the
// resident workgroups even that out (that room's 50 iterations 6.1 ms with one
// time, 5.3 with four and with eight, 5.5 with sixteen).
constexpr int kPdGroups = 4;
void launch_pd_iterate(const View& V, const PdTables& T, float lambda, float sigma, float tau,
                       double* partials, uint32_t npartials, double* energy, hipStream_t s,
                       int grid) {
  const int g = grid < (int)npartials ? grid : (int)npartials;
  const int all = !(std::isfinite(sigma) && 1.0f + sigma * 0.02f > 0.0f);
  pd_bits_kernel<<<kPdGroups * grid, 256, 0, s>>>(V, T.bits);
  if (energy) {
    pd_pass1_kernel<true><<<g, 256, 0, s>>>(V, T.nbr, T.bits, T.dual, all, sigma, partials);
    pd_energy_kernel<<<1, 256, 0, s>>>(partials, (uint32_t)g, lambda, energy);
  } else {
    pd_pass1_kernel<false><<<kPdGroups * grid, 256, 0, s>>>(V, T.nbr, T.bits, T.dual, all, sigma, nullptr);
  }
  pd_pass2_kernel<<<kPdGroups * grid, 256, 0, s>>>(V, T.nbr, T.bits, lambda, tau);
}

}  // namespace mh
