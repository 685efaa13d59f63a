// gvx_cost.hip -- differentiable clearance cost on the EDT (no reference counterpart).
//
//   c(traj) = sum over waypoints, links, spheres of  w * max(0, r + eps - d(x))^2
//   x = T_l(q) * c_local,  T_l = base * A_0(q_0) ... A_{l-1}(q_{l-1})
//   d(x) = trilinear interpolation of the metric EDT sampled at voxel centres.
// The adjoint is hand-written: dc/dx = -2 w h grad d; dc/dq_j = z_j . sum_{l>j}
// (M_l + (o_l - o_j) x G_l) for revolute joints (z_j . sum G_l for prismatic),
// where G_l = sum dc/dx and M_l = sum (x - o_l) x dc/dx over link l's spheres
// (moments about the link's own origin: short lever arms, no cancellation of
// large moments about the world origin) and (z_j, o_j) are the z axis and origin
// of frame T_j.  All reductions run in a fixed order, so results are
// deterministic.
//
// Layout: a block takes WB consecutive (trajectory, waypoint) pairs.  It builds their link
// frames together in LDS (DH matrices in parallel, one lane per waypoint chains them), then
// every wave takes one group of links: a link's spheres occupy a segment of 16, 32 or 64
// lanes (more spheres: several rounds), so a wave holds 4, 2 or 1 links and reduces each
// with lane shifts.  A second small kernel sums each trajectory's waypoint partials.
//
// What bounds it: the samples.  8192 random waypoints of 7 x 64 spheres on 512^3 miss L2
// 4.8 M times, 52 lines per ns, at a VALU load of a third; costs, gradient or both take the
// same 92-95 us.  So the costs and their gradient come from one pass where both are wanted
// (gvx_cost_forward_grad: an optimiser's step 341 -> 213 us with the host work of torch).  Loads past the L1
// (non-temporal) lose the lines that neighbouring spheres share: 129 us.
//
// Whole waves per link and a block per waypoint (as this file had it) left lanes idle and one
// lane's chain in everybody's way wherever the samples are not all there is; forward /
// backward call, host clock, 256^3, trajectories x waypoints x spheres per link:
//   256 x 32 x 16    57 /  72 -> 42 /  43 us      256 x 32 x 100  111 / 140 -> 76 /  85 us
//   512 x 64 x 32   204 / 245 -> 172 / 174        1024 x 64 x 64  462 / 532 -> 403 / 412
#include <type_traits>

#include "gvx_internal.hpp"

namespace gvx {

struct CostS {
  const float* grid = nullptr;
  uint32_t dims[3];
  float side, eps, w;
  uint32_t nl = 0, spl = 0;
  float* dh = nullptr;
  float* base = nullptr;
  float* spheres = nullptr;
  float* partial = nullptr;  // per (traj, wp)
  uint64_t cap = 0;          // (traj * wp) capacity
  std::recursive_mutex mu;
};

}  // namespace gvx

struct gvx_cost_s : gvx::CostS {};

namespace gvx {

// two neighbouring samples of an x row in one 8-byte load (rows are only 4-byte aligned)
struct __attribute__((packed, aligned(4))) SamplePair {
  float a, b;
};

// trilinear sample and gradient (samples at voxel centres, clamped at the border).  The
// eight samples are four pairs along x.  SMALL: the grid's bytes fit 32 bits, so the four
// loads share one lane offset from four uniform bases.
template <bool SMALL>
__device__ __forceinline__ float trilinear(const float* __restrict__ g, uint32_t dx, uint32_t dy, uint32_t dz, float side,
                                           float inv_side, float x, float y, float z, float& gx, float& gy, float& gz)
{
  const uint32_t d[3] = {dx, dy, dz};
  const float p[3] = {x, y, z};
  int i0[3];
  float t[3], s[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    float u = p[a] / side - 0.5f;
    s[a] = inv_side;
    const float hi = (float)(d[a] - 1);
    if (!(u >= 0.0f)) { u = 0.0f; s[a] = 0.0f; }
    if (u > hi) { u = hi; s[a] = 0.0f; }
    int i = (int)floorf(u);
    if (i > (int)d[a] - 2) i = (int)d[a] - 2;
    if (i < 0) i = 0;
    i0[a] = i;
    t[a] = u - (float)i;
  }
  const uint64_t sy = dx, sz = (uint64_t)dx * dy;
  SamplePair p00, p01, p10, p11;
  auto pair = [&](uint64_t row) {  // row: uniform offset of the pair's row from the first one
    if constexpr (SMALL) {
      const uint32_t o = (((uint32_t)i0[2] * dy + (uint32_t)i0[1]) * dx + (uint32_t)i0[0]) * 4u;
      return *reinterpret_cast<const SamplePair*>(reinterpret_cast<const char*>(g + row) + o);
    } else {
      const uint64_t o = (uint64_t)i0[2] * sz + (uint64_t)i0[1] * sy + (uint64_t)i0[0];
      return *reinterpret_cast<const SamplePair*>(g + row + o);
    }
  };
  p00 = pair(0);
  p01 = pair(sy);
  p10 = pair(sz);
  p11 = pair(sz + sy);
  const float c000 = p00.a, c001 = p00.b, c010 = p01.a, c011 = p01.b;
  const float c100 = p10.a, c101 = p10.b, c110 = p11.a, c111 = p11.b;
  const float tx = t[0], ty = t[1], tz = t[2];
  const float c00 = c000 * (1.f - tx) + c001 * tx, c01 = c010 * (1.f - tx) + c011 * tx;
  const float c10 = c100 * (1.f - tx) + c101 * tx, c11 = c110 * (1.f - tx) + c111 * tx;
  const float c0 = c00 * (1.f - ty) + c01 * ty, c1 = c10 * (1.f - ty) + c11 * ty;
  const float ddx0 = (c001 - c000) * (1.f - ty) + (c011 - c010) * ty;
  const float ddx1 = (c101 - c100) * (1.f - ty) + (c111 - c110) * ty;
  gx = (ddx0 * (1.f - tz) + ddx1 * tz) * s[0];
  gy = ((c01 - c00) * (1.f - tz) + (c11 - c10) * tz) * s[1];
  gz = (c1 - c0) * s[2];
  return c0 * (1.f - tz) + c1 * tz;
}

constexpr int CMAXW = 16;  // waves per block, at most

// What both kernels take.  seg: lanes per link (16, 32, 64); rounds: segments per link;
// groups: waves of links (64 / seg links each).
struct CostArgs {
  const float* grid;
  uint32_t dx, dy, dz;
  float side, inv_side;
  const float *dh, *base, *q, *spheres;
  uint32_t nl, spl, nwp;
  float eps, w;
  uint64_t n;  // (trajectory, waypoint) pairs
  uint32_t seg, rounds, groups;
};

// link frames of the block's waypoints into LDS: T[wp * nl + l] = base * A_0 ... A_{l-1}
// (KinematicChain::setConfiguration, robot/dh_robot/KinematicChain.cu:93-126).  The chain is
// serial: the block's waypoints walk theirs side by side, one lane each.
__device__ __forceinline__ void block_fk(const CostArgs& c, uint64_t tw0, uint32_t nw, float (*A)[12], float (*T)[12])
{
  for (uint32_t j = threadIdx.x; j < nw * c.nl; j += blockDim.x)  // rows of q are consecutive
    dh_matrix(c.dh + 5 * (j % c.nl), c.q[tw0 * c.nl + j], A[j]);
  __syncthreads();
  if (threadIdx.x < nw) {
    const uint32_t r = threadIdx.x * c.nl;
    float t[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) t[k] = c.base[k];
    for (uint32_t l = 0; l < c.nl; ++l) {
#pragma unroll
      for (int k = 0; k < 12; ++k) T[r + l][k] = t[k];
      affine_mul(t, A[r + l], t);
    }
  }
  __syncthreads();
}

// sums over the segments of seg lanes, in a fixed order: lane shifts inside the rows of 16,
// then the rows of a segment as a tree (a row's sum ends in its last lane)
__device__ __forceinline__ float row_fsum(float v)
{
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x111, 0xf, 0xf, true));  // row_shr:1
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x112, 0xf, 0xf, true));  // row_shr:2
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x114, 0xf, 0xf, true));  // row_shr:4
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x118, 0xf, 0xf, true));  // row_shr:8
  return v;
}
__device__ __forceinline__ float lane_value(float v, int lane)
{
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
// the sums of the wave's segments: s[0 .. 64 / seg), the same in every lane
__device__ __forceinline__ void segment_sums(float v, uint32_t seg, float (&s)[4])
{
  v = row_fsum(v);
  s[0] = lane_value(v, 15);
  s[1] = lane_value(v, 31);
  s[2] = lane_value(v, 47);
  s[3] = lane_value(v, 63);
  if (seg == 16) return;  // uniform
  s[0] += s[1];
  s[1] = s[2] + s[3];
  if (seg == 64) s[0] += s[1];
}

// forward: a lane's spheres of one link for all of the block's waypoints (the sphere is
// loaded once, the waypoints' samples overlap); the block's sum (waves in order) per
// waypoint is its partial
template <uint32_t WB, bool SMALL>
__global__ void __launch_bounds__(64 * CMAXW) k_cost_fwd(const CostArgs c, float* __restrict__ partial)
{
  extern __shared__ float cost_lds[];
  float(*A)[12] = reinterpret_cast<float(*)[12]>(cost_lds);
  float(*T)[12] = A + WB * c.nl;
  __shared__ float wsum[CMAXW][WB];
  const uint64_t tw0 = (uint64_t)blockIdx.x * WB;
  const uint32_t nw = c.n - tw0 < WB ? (uint32_t)(c.n - tw0) : WB;
  block_fk(c, tw0, nw, A, T);
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  float acc[WB];
#pragma unroll
  for (uint32_t p = 0; p < WB; ++p) acc[p] = 0.f;
  for (uint32_t g = wave; g < c.groups; g += waves) {
    const uint32_t l = g * (64 / c.seg) + lane / c.seg;
    for (uint32_t r = 0; r < c.rounds; ++r) {
      const uint32_t k = r * c.seg + lane % c.seg;
      if (l >= c.nl || k >= c.spl) continue;
      const float4 s4 = *reinterpret_cast<const float4*>(c.spheres + 4 * ((uint64_t)l * c.spl + k));
#pragma unroll
      for (uint32_t p = 0; p < WB; ++p) {
        if (p >= nw) continue;  // uniform
        float x, y, z, gx, gy, gz;
        transform(T[p * c.nl + l], s4.x, s4.y, s4.z, x, y, z);
        const float d = trilinear<SMALL>(c.grid, c.dx, c.dy, c.dz, c.side, c.inv_side, x, y, z, gx, gy, gz);
        const float h = s4.w + c.eps - d;
        if (h > 0.f) acc[p] += c.w * h * h;
      }
    }
  }
#pragma unroll
  for (uint32_t p = 0; p < WB; ++p) {
    float s[4];
    segment_sums(acc[p], 64, s);
    if (lane == 0) wsum[wave][p] = s[0];
  }
  __syncthreads();
  if (threadIdx.x < nw) {
    float s = 0.f;
    for (uint32_t i = 0; i < waves; ++i) s += wsum[i][threadIdx.x];
    partial[tw0 + threadIdx.x] = s;
  }
}

// per trajectory (one wave each): its waypoints' partials, lane l those at l, l + 64, ... in
// order, then the lanes in a fixed order
__global__ void __launch_bounds__(256) k_cost_sum(const float* __restrict__ partial, uint32_t ntraj, uint32_t nwp,
                                                  float* __restrict__ out)
{
  const uint32_t t = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (t >= ntraj) return;  // uniform over the wave
  float v = 0.f;
  for (uint32_t k = lane; k < nwp; k += 64) v += partial[(uint64_t)t * nwp + k];
  float s[4];
  segment_sums(v, 64, s);
  if (lane == 0) out[t] = s[0];
}

// backward: the same layout; per segment (one link's spheres) the six terms (G, M about the
// link origin) are reduced, then one lane per (waypoint, joint) forms dq, the upstream factor
// last.  partial: the forward sums as well, in k_cost_fwd's order (the same bits).
template <uint32_t WB, bool SMALL>
__global__ void __launch_bounds__(64 * CMAXW) k_cost_bwd(const CostArgs c, const float* __restrict__ upstream,
                                                         float* __restrict__ partial, float* __restrict__ dq,
                                                         float* __restrict__ dxo)
{
  extern __shared__ float cost_lds[];
  float(*A)[12] = reinterpret_cast<float(*)[12]>(cost_lds);
  float(*T)[12] = A + WB * c.nl;
  float(*lsum)[6] = reinterpret_cast<float(*)[6]>(A);  // the DH matrices are done with after the chain
  __shared__ float wsum[CMAXW][WB];
  const uint64_t tw0 = (uint64_t)blockIdx.x * WB;
  const uint32_t nw = c.n - tw0 < WB ? (uint32_t)(c.n - tw0) : WB;
  block_fk(c, tw0, nw, A, T);
  const uint32_t ns = c.nl * c.spl;
  const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  for (uint32_t p = 0; p < nw; ++p) {
    const float up = upstream && dxo ? upstream[(uint32_t)(tw0 + p) / c.nwp] : 1.0f;  // n < 2^31
    float acc = 0.f;
    for (uint32_t g = wave; g < c.groups; g += waves) {
      const uint32_t l = g * (64 / c.seg) + lane / c.seg;
      float c6[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (uint32_t r = 0; r < c.rounds; ++r) {
        const uint32_t k = r * c.seg + lane % c.seg;
        if (l >= c.nl || k >= c.spl) continue;
        const uint32_t ks = l * c.spl + k;
        const float4 s4 = *reinterpret_cast<const float4*>(c.spheres + 4 * (uint64_t)ks);
        const float* m = T[p * c.nl + l];
        float x, y, z, gx, gy, gz;
        transform(m, s4.x, s4.y, s4.z, x, y, z);
        const float d = trilinear<SMALL>(c.grid, c.dx, c.dy, c.dz, c.side, c.inv_side, x, y, z, gx, gy, gz);
        const float h = s4.w + c.eps - d;
        float ax = 0.f, ay = 0.f, az = 0.f;
        if (h > 0.f) {
          acc += c.w * h * h;
          const float f = -2.0f * c.w * h;
          ax = f * gx; ay = f * gy; az = f * gz;
        }
        if (dxo) {
          float* o = dxo + ((tw0 + p) * ns + ks) * 3;
          const bool on = h > 0.f;  // an idle sphere's zero stays one whatever the factor
          o[0] = on ? ax * up : 0.f; o[1] = on ? ay * up : 0.f; o[2] = on ? az * up : 0.f;
        }
        const float rx = x - m[3], ry = y - m[7], rz = z - m[11];
        c6[0] += ax; c6[1] += ay; c6[2] += az;
        c6[3] += ry * az - rz * ay; c6[4] += rz * ax - rx * az; c6[5] += rx * ay - ry * ax;
      }
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        float s[4];
        segment_sums(c6[i], c.seg, s);
        const uint32_t l0 = g * (64 / c.seg);  // lane j writes segment j's sum
        if (lane < 64 / c.seg && l0 + lane < c.nl)
          lsum[p * c.nl + l0 + lane][i] = lane == 0 ? s[0] : lane == 1 ? s[1] : lane == 2 ? s[2] : s[3];
      }
    }
    if (partial) {  // uniform
      float s[4];
      segment_sums(acc, 64, s);
      if (lane == 0) wsum[wave][p] = s[0];
    }
  }
  __syncthreads();
  // dq_j = z_j . sum_{l > j} (M_l + (o_l - o_j) x G_l)   (revolute), z_j . sum G_l (prismatic)
  for (uint32_t e = threadIdx.x; e < nw * c.nl; e += blockDim.x) {
    const uint32_t j = e % c.nl, r0 = e - j;
    const float* f = T[e];
    const float zx = f[2], zy = f[6], zz = f[10], ox = f[3], oy = f[7], oz = f[11];
    float r;
    if (c.dh[5 * j + 4] != 0.0f) {
      float Gx = 0.f, Gy = 0.f, Gz = 0.f;
      for (uint32_t l = j + 1; l < c.nl; ++l) {
        Gx += lsum[r0 + l][0]; Gy += lsum[r0 + l][1]; Gz += lsum[r0 + l][2];
      }
      r = zx * Gx + zy * Gy + zz * Gz;
    } else {
      float cx = 0.f, cy = 0.f, cz = 0.f;
      for (uint32_t l = j + 1; l < c.nl; ++l) {
        const float* g6 = lsum[r0 + l];
        const float* t = T[r0 + l];
        const float lx = t[3] - ox, ly = t[7] - oy, lz = t[11] - oz;
        cx += g6[3] + (ly * g6[2] - lz * g6[1]);
        cy += g6[4] + (lz * g6[0] - lx * g6[2]);
        cz += g6[5] + (lx * g6[1] - ly * g6[0]);
      }
      r = zx * cx + zy * cy + zz * cz;
    }
    // zero without contact, also where the factor is infinite (the root of a cost of zero)
    dq[tw0 * c.nl + e] = upstream && r != 0.f ? r * upstream[(uint32_t)(tw0 + e / c.nl) / c.nwp] : r;
  }
  if (partial && threadIdx.x < nw) {
    float s = 0.f;
    for (uint32_t i = 0; i < waves; ++i) s += wsum[i][threadIdx.x];
    partial[tw0 + threadIdx.x] = s;
  }
}

static int cost_reserve(CostS* c, uint64_t n)
{
  if (n <= c->cap) return GVX_OK;
  GVX_CHECK(sync());
  dfree(c->partial);
  c->partial = nullptr;
  c->cap = 0;
  GVX_CHECK(dalloc((void**)&c->partial, n * 4));
  c->cap = n;
  return GVX_OK;
}

// Layout for n waypoints: segments as long as a link's spheres need, a wave per group of
// links, and as many waypoints per block (up to 8) as leave 8 blocks per CU: fewer blocks
// end unevenly, smaller ones have more serial chains (forward / backward, 64 spheres:
// 8192 waypoints with 1, 2, 4, 8 in a block 76 / 90, 70 / 79, 71 / 75, 72 / 80 us; 65536:
// 443 / 568, 397 / 471, 397 / 420, 402 / 408).
struct CostShape {
  uint32_t wb, threads;
  size_t lds;
  bool small;
};
static CostShape cost_shape(const CostS* c, uint64_t n, const float* q, uint32_t nwp, CostArgs* a)
{
  const uint32_t seg = c->spl <= 16 ? 16 : c->spl <= 32 ? 32 : 64, lpw = 64 / seg;
  *a = CostArgs{c->grid, c->dims[0], c->dims[1], c->dims[2], c->side, 1.0f / c->side, c->dh, c->base, q, c->spheres,
                c->nl, c->spl, nwp, c->eps, c->w, n, seg, (c->spl + seg - 1) / seg, (c->nl + lpw - 1) / lpw};
  CostShape s;
  const uint64_t blocks = (uint64_t)(rt().num_cus > 0 ? rt().num_cus : 256) * 8;
  s.wb = n >= 8 * blocks ? 8 : n >= 4 * blocks ? 4 : n >= 2 * blocks ? 2 : 1;
  s.threads = 64 * (a->groups < (uint32_t)CMAXW ? a->groups : (uint32_t)CMAXW);
  s.lds = (size_t)s.wb * c->nl * 24 * sizeof(float);  // at most 8 x 64 x 96 B = 48 KiB
  s.small = (uint64_t)c->dims[0] * c->dims[1] * c->dims[2] < (1ull << 30);
  return s;
}

// out: the costs; dq: the gradient; or both from one pass
static int cost_run(CostS* c, const float* q, uint32_t ntraj, uint32_t nwp, float* out, const float* upstream, float* dq,
                    float* dxo)
{
  const uint64_t n = (uint64_t)ntraj * nwp;
  if (n > 0x7FFFFFFFull) return fail(GVX_ERR_BAD_ARG, "too many (trajectory, waypoint) pairs");
  std::lock_guard<std::recursive_mutex> g(c->mu);
  std::lock_guard<std::recursive_mutex> g2(rt().mu);
  if (n == 0) {  // a trajectory without waypoints costs nothing
    if (!out || ntraj == 0) return GVX_OK;
    hipLaunchKernelGGL(k_cost_sum, dim3((ntraj + 3) / 4), dim3(256), 0, rt().stream, c->partial, ntraj, nwp, out);
    GVX_HIP(hipGetLastError());
    return sync();
  }
  if (out) GVX_CHECK(cost_reserve(c, n));
  float* partial = out ? c->partial : nullptr;
  hipStream_t s = rt().stream;
  CostArgs a;
  const CostShape sh = cost_shape(c, n, q, nwp, &a);
  ProfScope ps(dq ? "cost_backward" : "cost_forward");
  const dim3 grid((unsigned)((n + sh.wb - 1) / sh.wb)), block(sh.threads);
  auto launch = [&](auto wb, auto small) {
    if (dq)
      hipLaunchKernelGGL((k_cost_bwd<wb(), small()>), grid, block, sh.lds, s, a, upstream, partial, dq, dxo);
    else
      hipLaunchKernelGGL((k_cost_fwd<wb(), small()>), grid, block, sh.lds, s, a, partial);
  };
  auto sized = [&](auto wb) {
    if (sh.small) launch(wb, std::true_type{});
    else launch(wb, std::false_type{});
  };
  switch (sh.wb) {
    case 8: sized(std::integral_constant<uint32_t, 8>{}); break;
    case 4: sized(std::integral_constant<uint32_t, 4>{}); break;
    case 2: sized(std::integral_constant<uint32_t, 2>{}); break;
    default: sized(std::integral_constant<uint32_t, 1>{}); break;
  }
  if (out) hipLaunchKernelGGL(k_cost_sum, dim3((ntraj + 3) / 4), dim3(256), 0, s, c->partial, ntraj, nwp, out);
  GVX_HIP(hipGetLastError());
  return sync();
}

}  // namespace gvx

using namespace gvx;

extern "C" {

int gvx_cost_create(const float* grid_dev, const uint32_t dims[3], float side, const float* dh, uint32_t n_links,
                    const float base[12], const float* spheres, uint32_t spl, float eps, float weight, gvx_cost* out)
{
  if (!out) return fail(GVX_ERR_BAD_ARG, "null out");
  *out = nullptr;
  GVX_CHECK(ensure_init());
  if (!grid_dev || !dims || !dh || !spheres) return fail(GVX_ERR_BAD_ARG, "null argument");
  if (dims[0] < 2 || dims[1] < 2 || dims[2] < 2 || !(side > 0.f)) return fail(GVX_ERR_BAD_ARG, "grid must be >= 2^3");
  if (n_links == 0 || n_links > 64 || spl == 0) return fail(GVX_ERR_BAD_ARG, "1..64 links and >= 1 sphere per link");
  gvx_cost c = new gvx_cost_s();
  c->grid = grid_dev;
  memcpy(c->dims, dims, 12);
  c->side = side;
  c->eps = eps;
  c->w = weight;
  c->nl = n_links;
  c->spl = spl;
  float ident[12] = {1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0};
  int s;
  if ((s = dalloc((void**)&c->dh, n_links * 20)) != GVX_OK ||
      (s = dalloc((void**)&c->base, 48)) != GVX_OK ||
      (s = dalloc((void**)&c->spheres, (uint64_t)n_links * spl * 16)) != GVX_OK) {
    gvx_cost_destroy(c);
    return s;
  }
  hipStream_t st = rt().stream;
  if (hipMemcpyAsync(c->dh, dh, n_links * 20, hipMemcpyHostToDevice, st) != hipSuccess ||
      hipMemcpyAsync(c->base, base ? base : ident, 48, hipMemcpyHostToDevice, st) != hipSuccess ||
      hipMemcpyAsync(c->spheres, spheres, (uint64_t)n_links * spl * 16, hipMemcpyHostToDevice, st) != hipSuccess) {
    gvx_cost_destroy(c);
    return fail(GVX_ERR_HIP, "copy cost description");
  }
  if ((s = sync()) != GVX_OK) {
    gvx_cost_destroy(c);
    return s;
  }
  *out = c;
  return GVX_OK;
}

int gvx_cost_destroy(gvx_cost c)
{
  if (!c) return GVX_OK;
  (void)sync();
  void* bufs[] = {c->dh, c->base, c->spheres, c->partial};
  for (auto p : bufs) dfree(p);
  delete c;
  return GVX_OK;
}

int gvx_cost_forward(gvx_cost c, const float* q, uint32_t ntraj, uint32_t nwp, float* out)
{
  if (!c || !q || !out) return fail(GVX_ERR_BAD_ARG, "null argument");
  return cost_run(c, q, ntraj, nwp, out, nullptr, nullptr, nullptr);
}

int gvx_cost_backward(gvx_cost c, const float* q, uint32_t ntraj, uint32_t nwp, const float* upstream, float* dq,
                      float* dxo)
{
  if (!c || !q || !dq) return fail(GVX_ERR_BAD_ARG, "null argument");
  return cost_run(c, q, ntraj, nwp, nullptr, upstream, dq, dxo);
}

int gvx_cost_forward_grad(gvx_cost c, const float* q, uint32_t ntraj, uint32_t nwp, float* out, float* dq)
{
  if (!c || !q || !out || !dq) return fail(GVX_ERR_BAD_ARG, "null argument");
  return cost_run(c, q, ntraj, nwp, out, nullptr, dq, nullptr);
}

}  // extern "C"
