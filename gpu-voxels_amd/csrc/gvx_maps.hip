// gvx_maps.hip -- dense voxel maps: create/clear, voxelization, map x map collision.
#include <algorithm>

#include "gvx_internal.hpp"

namespace gvx {

constexpr int TBIT = GVX_MT_BITVECTOR_VOXELMAP, TPROB = GVX_MT_PROBAB_VOXELMAP, TDIST = GVX_MT_DISTANCE_VOXELMAP;

// ---------------------------------------------------------------- voxel updates
template <int T>
__device__ __forceinline__ void voxel_insert(uint8_t* map, uint64_t idx, uint32_t x, uint32_t y, uint32_t z,
                                             uint32_t meaning, uint32_t uninit)
{
  if constexpr (T == TBIT) {
    // BitVoxel::insert = setBit (BitVoxel.hpp:60-65); atomic OR into the word holding the bit
    atomicOr(reinterpret_cast<uint32_t*>(map) + idx * 8 + (meaning >> 5), 1u << (meaning & 31));
  } else if constexpr (T == TPROB) {
    // ProbabilisticVoxel::insert (ProbabilisticVoxel.hpp:79-101) as a CAS on the 32-bit word
    uint32_t* w = reinterpret_cast<uint32_t*>(map + (idx & ~(uint64_t)3));
    const uint32_t sh = (uint32_t)(idx & 3) * 8;
    uint32_t old = __atomic_load_n(w, __ATOMIC_RELAXED);
    for (;;) {
      int cur = (int)(int8_t)((old >> sh) & 0xFF);
      int nv = prob_insert(cur, meaning);
      if (nv == cur) break;
      uint32_t neu = (old & ~(0xFFu << sh)) | ((uint32_t)(uint8_t)(int8_t)nv << sh);
      uint32_t prev = atomicCAS(w, old, neu);
      if (prev == old) break;
      old = prev;
    }
  } else {
    // DistanceVoxel::insert (DistanceVoxel.hpp:128-139)
    reinterpret_cast<uint32_t*>(map)[idx] = (meaning == M_OCCUPIED) ? (x | (y << 10) | (z << 20)) : uninit;
  }
}

// ProbabilisticVoxel::insert(meaning) updates on the four voxels of a 32-bit word, counts byte
// by byte, with one CAS (identical updates: any order gives the same byte)
__device__ __forceinline__ void prob_insert_word(uint32_t* w, uint32_t meaning, uint32_t counts)
{
  uint32_t old = __atomic_load_n(w, __ATOMIC_RELAXED);
  for (;;) {
    uint32_t neu = 0;
#pragma unroll
    for (int b = 0; b < 32; b += 8) {
      int v = (int)(int8_t)(old >> b);
      for (uint32_t k = (counts >> b) & 0xFFu; k; --k) {
        const int n = prob_insert(v, meaning);
        if (n == v) break;
        v = n;
      }
      neu |= (uint32_t)(uint8_t)(int8_t)v << b;
    }
    if (neu == old) return;
    const uint32_t prev = atomicCAS(w, old, neu);
    if (prev == old) return;
    old = prev;
  }
}

// points: kernelInsertGlobalPointCloud / kernelInsertMetaPointCloud (VoxelMapOperations.hpp:241-575).
// cloud_ends: inclusive prefix of the cloud sizes (n_clouds entries) or null.
template <int T>
__global__ void __launch_bounds__(256) k_insert_points(uint8_t* __restrict__ map, uint32_t dx, uint32_t dy, uint32_t dz,
                                                       float side, const float* __restrict__ pts, uint64_t n,
                                                       const uint32_t* __restrict__ cloud_ends, uint32_t n_clouds,
                                                       const uint32_t* __restrict__ meanings, uint32_t meaning,
                                                       uint32_t uninit, OutsideFlag outside)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    uint32_t m = meaning;
    if (cloud_ends) {
      uint32_t lo = 0, hi = n_clouds - 1;
      while (lo < hi) {
        uint32_t mid = (lo + hi) >> 1;
        if ((uint64_t)cloud_ends[mid] > i) hi = mid; else lo = mid + 1;
      }
      m = meanings[lo];
    }
    const uint32_t x = quantize(pts[3 * i], side), y = quantize(pts[3 * i + 1], side),
                   z = quantize(pts[3 * i + 2], side);
    const bool in = (x < dx) && (y < dy) && (z < dz);
    if constexpr (T == TPROB) {
      // neighbouring points often share a voxel or the word of four: a run of lanes on one
      // word updates it with one CAS, its points per voxel counted in the word's bytes (at
      // most 64).  A CAS per voxel had the lanes of a word wait for each other (304k points
      // of a depth image into 512^3, by scene: 16.5 -> 15.9 us, clear and insert 68 -> 63)
      const uint64_t idx = in ? ((uint64_t)z * dy + y) * dx + x : 0ull;
      const uint32_t lane = threadIdx.x & 63, own = in ? 1u << (8 * (uint32_t)(idx & 3)) : 0u;
      const uint32_t run = wave_run_head(in, idx >> 2, m);
      uint32_t sum = own;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t below = __shfl_up(sum, o);
        if (lane >= (uint32_t)o) sum += below;
      }
      const uint32_t counts = __shfl(sum, (int)(run ? lane + run - 1 : lane)) - (sum - own);
      if (run) prob_insert_word(reinterpret_cast<uint32_t*>(map) + (idx >> 2), m, counts);
    } else if constexpr (T == TBIT) {
      // setting a bit is idempotent: one lane per run on one (voxel, meaning) sets it
      const uint64_t idx = in ? ((uint64_t)z * dy + y) * dx + x : 0ull;
      if (wave_run_head(in, idx, m)) voxel_insert<T>(map, idx, x, y, z, m, uninit);
    } else {
      if (in) voxel_insert<T>(map, ((uint64_t)z * dy + y) * dx + x, x, y, z, m, uninit);
    }
    flag_outside(outside, !in);
  }
}

template <int T>
__global__ void __launch_bounds__(256) k_insert_coords(uint8_t* __restrict__ map, uint32_t dx, uint32_t dy, uint32_t dz,
                                                       const uint32_t* __restrict__ c, uint64_t n, uint32_t meaning,
                                                       uint32_t uninit, OutsideFlag outside)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const uint32_t x = c[3 * i], y = c[3 * i + 1], z = c[3 * i + 2];
    const bool in = (x < dx) && (y < dy) && (z < dz);
    if (in) voxel_insert<T>(map, ((uint64_t)z * dy + y) * dx + x, x, y, z, meaning, uninit);
    flag_outside(outside, !in);
  }
}

// ---------------------------------------------------------------- collision
template <int T>
__device__ __forceinline__ bool occupied(const uint8_t* __restrict__ m, uint64_t i, int thr)
{
  if constexpr (T == TBIT) {
    const uint4* p = reinterpret_cast<const uint4*>(m + i * 32);
    return bits_occupied(p[0], p[1]);
  } else {
    return (int)(int8_t)m[i] >= thr;
  }
}

template <int T>
__device__ __forceinline__ void mark_collision(uint8_t* __restrict__ m, uint64_t i)
{
  if constexpr (T == TBIT) {
    reinterpret_cast<uint32_t*>(m)[i * 8] |= (1u << M_COLLISION);
  } else {
    m[i] = (uint8_t)(int8_t)prob_update((int)(int8_t)m[i], SENSOR_OCC);
  }
}

// The voxels [lo, hi) of a BitVector map that hold one of the wanted bits (all of words
// 1..7, those of low in word 0): a wave reads kHalves x 1 KiB of consecutive memory with
// 16-byte loads, all issued before any is used; a voxel is two neighbouring lanes' halves,
// so one ballot per load says which of its 32 voxels hold something, and visit(i) runs on
// the lanes below 32 for those (voxel i; wave-uniform control otherwise).  HBM
// bound: a 512^3 map (4 GiB) in 685 us, 6.3 TB/s, a plain read's rate; one voxel per lane
// and iteration (two loads at a stride of 32 bytes) took 804 us.
constexpr int kHalves = 8;
template <typename Visit>
__device__ __forceinline__ void scan_bit_voxels(const uint8_t* __restrict__ m, uint64_t lo, uint64_t hi, uint32_t low,
                                                Visit&& visit)
{
  const uint4* __restrict__ h = reinterpret_cast<const uint4*>(m);
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t waves = (uint64_t)gridDim.x * (blockDim.x / 64);
  const uint32_t sel = lane & 1 ? 0xFFFFFFFFu : low;
  for (uint64_t h0 = 2 * lo + ((uint64_t)blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64) * (64 * kHalves); h0 < 2 * hi;
       h0 += waves * (64 * kHalves)) {
    uint4 v[kHalves];
#pragma unroll
    for (int u = 0; u < kHalves; ++u) {
      const uint64_t k = h0 + (uint64_t)(u * 64) + lane;
      v[u] = k < 2 * hi ? h[k] : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int u = 0; u < kHalves; ++u) {
      const uint64_t bal = wave_ballot(((v[u].x & sel) | v[u].y | v[u].z | v[u].w) != 0u);
      if (bal == 0ull) continue;
      if (lane < 32 && ((bal >> (2 * lane)) & 3ull)) visit(h0 / 2 + (uint64_t)(u * 32) + lane);
    }
  }
}

// kernelCollideVoxelMapsDebug (VoxelMapOperations.hpp:129-184) with DefaultCollider, both
// BitVector maps: a[i + off] against b[i] for i in [lo, hi); b is read whole, a only
// where b holds something.  64-bit count.
__global__ void __launch_bounds__(256) k_collide_bits(uint8_t* __restrict__ a, const uint8_t* __restrict__ b, uint64_t lo,
                                                      uint64_t hi, int64_t off, unsigned long long* __restrict__ count)
{
  uint64_t c = 0;
  scan_bit_voxels(b, lo, hi, ~1u, [&](uint64_t i) {
    const uint64_t j = (uint64_t)((int64_t)i + off);
    if (occupied<TBIT>(a, j, 0)) {
      mark_collision<TBIT>(a, j);
      ++c;
    }
  });
  add_count(c, count);
}

constexpr int kLoadsInFlight = 4;  // per lane, in the kernels that stream a ProbVoxelMap

// The passing voxels of a wave's 64 lanes x 16 voxels, spread over its lanes: each
// lane lists its own (offset lane * 16 + voxel) in the wave's LDS list at its prefix
// position, then lane t visits entries t, t + 64, ...  A lane whose 16 voxels all
// pass (a surface along x) would otherwise read the other side 16 times in a row.
// Called by every lane of the wave (wave-uniform control); sq holds 1024 entries.
template <typename Visit>
__device__ __forceinline__ void wave_spread(const uint32_t f[4], uint16_t* sq, Visit&& visit)
{
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t cnt = __popc(f[0]) + __popc(f[1]) + __popc(f[2]) + __popc(f[3]);
  uint32_t incl = cnt;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t t = __shfl_up(incl, d, 64);
    if (lane >= (uint32_t)d) incl += t;
  }
  const uint32_t total = __shfl(incl, 63, 64);
  uint32_t pos = incl - cnt;
  for (int q = 0; q < 4; ++q)
    for (uint32_t m = f[q]; m != 0u; m &= m - 1u) sq[pos++] = (uint16_t)(lane * 16 + q * 4 + (__builtin_ctz(m) >> 3));
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  for (uint32_t t = lane; t < total; t += 64) visit((uint32_t)sq[t]);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();  // the list is rewritten by the next call
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The same collision when one side is a ProbVoxelMap: a lane takes 16 consecutive
// Prob voxels with one 16-byte load and reads the other side's voxel only where
// the Prob voxel passes the threshold (a collision needs both), so a sparse
// environment costs 1 B per voxel instead of 33.  KEY_A: the Prob side is self
// (a[j], j = i + off), else other (b[i]).  Chunks are aligned on the Prob side;
// map allocations are padded to 256 B, and voxels outside the valid range are
// masked off.
template <int TA, int TB, bool KEY_A>
__global__ void __launch_bounds__(256) k_collide_prob(uint8_t* __restrict__ a, const uint8_t* __restrict__ b,
                                                      uint64_t lo, uint64_t hi, int64_t off, int thr,
                                                      unsigned long long* __restrict__ count)
{
  const uint8_t* key = KEY_A ? a : b;
  const int64_t shift = KEY_A ? off : 0;  // key index = i + shift
  const uint64_t klo = (uint64_t)((int64_t)lo + shift), khi = (uint64_t)((int64_t)hi + shift);
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint32_t lane = threadIdx.x & 63;
  __shared__ uint16_t sq[4][1024];
  uint64_t c = 0;
  // kLoadsInFlight 16-byte loads are issued before any is used; the loop runs while
  // the wave's first lane is in range, so control stays wave-uniform
  for (uint64_t k0 = klo / 16 + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; (k0 - lane) * 16 < khi;
       k0 += stride * kLoadsInFlight) {
    uint4 v[kLoadsInFlight];
#pragma unroll
    for (int u = 0; u < kLoadsInFlight; ++u) {
      const uint64_t k = k0 + (uint64_t)u * stride;
      v[u] = k * 16 < khi ? reinterpret_cast<const uint4*>(key)[k] : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int u = 0; u < kLoadsInFlight; ++u) {
      const uint64_t k = k0 + (uint64_t)u * stride, kw = (k - lane) * 16;  // the wave's first voxel
      if (kw >= khi) break;
      uint32_t f[4] = {0u, 0u, 0u, 0u};
      if (k * 16 < khi) prob_pass(v[u], thr, f);
      if (wave_ballot((f[0] | f[1] | f[2] | f[3]) != 0u) == 0ull) continue;
      wave_spread(f, sq[threadIdx.x >> 6], [&](uint32_t o) {
        const uint64_t kj = kw + o;
        if (kj < klo || kj >= khi) return;
        const uint64_t i = (uint64_t)((int64_t)kj - shift), j = (uint64_t)((int64_t)i + off);
        const bool hit = KEY_A ? occupied<TB>(b, i, thr) : occupied<TA>(a, j, thr);
        if (hit) {
          mark_collision<TA>(a, j);
          ++c;
        }
      });
    }
  }
  add_count(c, count);
}

// kernelCollideVoxelMapsBitvector (VoxelMapOperations.hpp:187-239) with SVCollider,
// Bit x Bit: bitMarginCollisionCheck with margin 0 = a & b restricted to bits 4..255,
// mask |= a & b.  Masks are ORed over all colliding voxels.  a is read whole, b only
// where a holds a bit that the AND can keep.
__global__ void __launch_bounds__(256) k_collide_types(uint8_t* __restrict__ a, const uint8_t* __restrict__ b, uint64_t n,
                                                       unsigned long long* __restrict__ count,
                                                       uint32_t* __restrict__ mask)
{
  uint64_t c = 0;
  uint32_t acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  scan_bit_voxels(a, 0, n, 0xFFFFFFF0u, [&](uint64_t i) {
    uint4* pa = reinterpret_cast<uint4*>(a + i * 32);
    const uint4* pb = reinterpret_cast<const uint4*>(b + i * 32);
    const uint4 a0 = pa[0], a1 = pa[1], b0 = pb[0], b1 = pb[1];
    const uint32_t r[8] = {a0.x & b0.x & 0xFFFFFFF0u, a0.y & b0.y, a0.z & b0.z, a0.w & b0.w,
                           a1.x & b1.x, a1.y & b1.y, a1.z & b1.z, a1.w & b1.w};
    if ((r[0] | r[1] | r[2] | r[3] | r[4] | r[5] | r[6] | r[7]) != 0u) {
#pragma unroll
      for (int k = 0; k < 8; ++k) acc[k] |= r[k];
      reinterpret_cast<uint32_t*>(pa)[0] = a0.x | (1u << M_COLLISION);
      ++c;
    }
  });
  add_hits(c, acc, count, mask);
}

// Bit x Prob of the above: prob >= thr and a occupied, mask |= a.  The Prob side
// is read 16 voxels per lane; the bit voxel only where the Prob voxel passes.
__global__ void __launch_bounds__(256) k_collide_types_prob(uint8_t* __restrict__ a, const uint8_t* __restrict__ b,
                                                            uint64_t n, int thr, unsigned long long* __restrict__ count,
                                                            uint32_t* __restrict__ mask)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  uint64_t c = 0;
  uint32_t acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  const uint32_t lane = threadIdx.x & 63;
  __shared__ uint16_t sq[4][1024];
  for (uint64_t k0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; (k0 - lane) * 16 < n;
       k0 += stride * kLoadsInFlight) {
    uint4 v[kLoadsInFlight];
#pragma unroll
    for (int u = 0; u < kLoadsInFlight; ++u) {
      const uint64_t k = k0 + (uint64_t)u * stride;
      v[u] = k * 16 < n ? reinterpret_cast<const uint4*>(b)[k] : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int u = 0; u < kLoadsInFlight; ++u) {
      const uint64_t k = k0 + (uint64_t)u * stride, kw = (k - lane) * 16;  // the wave's first voxel
      if (kw >= n) break;
      uint32_t f[4] = {0u, 0u, 0u, 0u};
      if (k * 16 < n) prob_pass(v[u], thr, f);
      if (wave_ballot((f[0] | f[1] | f[2] | f[3]) != 0u) == 0ull) continue;
      wave_spread(f, sq[threadIdx.x >> 6], [&](uint32_t o) {
        const uint64_t i = kw + o;
        if (i >= n) return;
        uint4* pa = reinterpret_cast<uint4*>(a + i * 32);
        const uint4 a0 = pa[0], a1 = pa[1];
        if (bits_occupied(a0, a1)) {
          acc[0] |= a0.x; acc[1] |= a0.y; acc[2] |= a0.z; acc[3] |= a0.w;
          acc[4] |= a1.x; acc[5] |= a1.y; acc[6] |= a1.z; acc[7] |= a1.w;
          reinterpret_cast<uint32_t*>(pa)[0] = a0.x | (1u << M_COLLISION);
          ++c;
        }
      });
    }
  }
  add_hits(c, acc, count, mask);
}

// insertMetaPointCloudWithSelfCollisionCheck, one sub-cloud
// (kernelInsertMetaPointCloudSelfCollCheck, VoxelMapOperations.hpp:582-638).  Test
// pass: every point reads its voxel as it was before the sub-cloud; masked = voxel
// & mask colliding (a bit other than eBVM_FREE) flags the point and is ORed, with
// the sub-cloud's meaning, into acc[0..7] (one atomic per word per wave); acc[8]
// is the points-outside flag.
__global__ void __launch_bounds__(256) k_selfcoll_test(const uint32_t* __restrict__ map, uint32_t dx, uint32_t dy,
                                                       uint32_t dz, float side, const float* __restrict__ pts,
                                                       uint64_t n, uint4 mlo, uint4 mhi, uint32_t meaning,
                                                       uint8_t* __restrict__ hit, uint32_t* __restrict__ acc)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  uint32_t a[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  bool any = false, outside = false;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const uint32_t x = quantize(pts[3 * i], side), y = quantize(pts[3 * i + 1], side),
                   z = quantize(pts[3 * i + 2], side);
    uint8_t h = 0;
    if (x < dx && y < dy && z < dz) {
      const uint4* v = reinterpret_cast<const uint4*>(map + (((uint64_t)z * dy + y) * dx + x) * 8);
      const uint4 v0 = v[0], v1 = v[1];
      const uint32_t m[8] = {v0.x & mlo.x, v0.y & mlo.y, v0.z & mlo.z, v0.w & mlo.w,
                             v1.x & mhi.x, v1.y & mhi.y, v1.z & mhi.z, v1.w & mhi.w};
      if (((m[0] & ~1u) | m[1] | m[2] | m[3] | m[4] | m[5] | m[6] | m[7]) != 0u) {  // BitVector::noneButEmpty
#pragma unroll
        for (int k = 0; k < 8; ++k) a[k] |= m[k];
        any = true;
        h = 1;
      }
    } else {
      outside = true;
    }
    hit[i] = h;
  }
  if (any) a[meaning >> 5] |= 1u << (meaning & 31);
#pragma unroll
  for (int k = 0; k < 8; ++k) a[k] = wave_or(a[k]);
  const bool out_w = wave_ballot(outside) != 0;
  if ((threadIdx.x & 63) == 0) {
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (a[k]) atomicOr(acc + k, a[k]);
    if (out_w) atomicOr(acc + 8, 1u);
  }
}

// insert pass of the sub-cloud: its meaning into every voxel it reaches,
// eBVM_COLLISION where the test pass flagged the point
__global__ void __launch_bounds__(256) k_selfcoll_insert(uint32_t* __restrict__ map, uint32_t dx, uint32_t dy,
                                                         uint32_t dz, float side, const float* __restrict__ pts,
                                                         uint64_t n, uint32_t meaning, const uint8_t* __restrict__ hit)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const uint32_t x = quantize(pts[3 * i], side), y = quantize(pts[3 * i + 1], side),
                   z = quantize(pts[3 * i + 2], side);
    if (x < dx && y < dy && z < dz) {
      uint32_t* v = map + (((uint64_t)z * dy + y) * dx + x) * 8;
      atomicOr(v + (meaning >> 5), 1u << (meaning & 31));
      if (hit[i]) atomicOr(v, 1u << M_COLLISION);
    }
  }
}

// kernelClearVoxelMap(bits), VoxelMapOperations.hpp:59-72
__global__ void k_clear_bits(uint32_t* __restrict__ m, uint64_t n, uint4 lo, uint4 hi)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    uint4* p = reinterpret_cast<uint4*>(m + i * 8);
    uint4 a = p[0], b = p[1];
    a.x &= ~lo.x; a.y &= ~lo.y; a.z &= ~lo.z; a.w &= ~lo.w;
    b.x &= ~hi.x; b.y &= ~hi.y; b.z &= ~hi.z; b.w &= ~hi.w;
    p[0] = a;
    p[1] = b;
  }
}

static unsigned stream_grid(uint64_t n)
{
  // enough waves to saturate HBM: ~2048 threads per CU, grid-stride beyond
  uint64_t cap = (uint64_t)(rt().num_cus > 0 ? rt().num_cus : 256) * 8;
  return grid_for(n, 256, (unsigned)cap);
}

// kernels that stream a ProbVoxelMap: one round of kLoadsInFlight chunks per lane, so that
// waves that wait for memory are replaced by others instead of looping (512^3: 31 us with
// 8 blocks per CU and 4 rounds each, 24 us).  Below 4 blocks per CU a lane takes fewer
// chunks, since a wave visits the passing voxels of its chunks one after another (a call on
// 64^3 21.2 -> 17.4 us, 128^3 20.9 -> 17.2, 200 x 200 x 150 19.2 -> 17.6, 256^3 equal; with 1
// or 2 blocks per CU the middle ones 18.5 to 19.2).
static unsigned prob_grid(uint64_t chunks)
{
  const unsigned rounds = grid_for((chunks + kLoadsInFlight - 1) / kLoadsInFlight, 256, 1u << 16);
  return std::max(rounds, grid_for(chunks, 256, (unsigned)(rt().num_cus > 0 ? rt().num_cus : 256) * 4));
}

// scan_bit_voxels: a block reads 32 kHalves x 4 voxels per iteration
static unsigned bits_grid(uint64_t voxels) { return grid_for((voxels + 32 * kHalves - 1) / (32 * kHalves) * 64, 256, 1u << 16); }

int map_clear_async(MapS* m)
{
  if (m->type == TBIT) return fill_u32(m->data, 0u, m->n * 8);
  if (m->type == TPROB) return fill_bytes(m->data, 0x80, m->n);
  return fill_u32(m->data, m->uninit, m->n);
}

// one cloud of a multi-cloud insert: points [ends[c-1], ends[c]) with meanings[c]
template <int T>
__global__ void __launch_bounds__(256) k_insert_cloud(uint8_t* __restrict__ map, uint32_t dx, uint32_t dy, uint32_t dz,
                                                      float side, const float* __restrict__ pts,
                                                      const uint32_t* __restrict__ cloud_ends, uint32_t c,
                                                      const uint32_t* __restrict__ meanings, uint32_t uninit,
                                                      OutsideFlag outside)
{
  const uint64_t lo = c ? cloud_ends[c - 1] : 0, hi = cloud_ends[c];
  const uint32_t m = meanings ? meanings[c] : 0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = lo + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < hi; i += stride) {
    const uint32_t x = quantize(pts[3 * i], side), y = quantize(pts[3 * i + 1], side),
                   z = quantize(pts[3 * i + 2], side);
    const bool in = (x < dx) && (y < dy) && (z < dz);
    if (in) voxel_insert<T>(map, ((uint64_t)z * dy + y) * dx + x, x, y, z, m, uninit);
    flag_outside(outside, !in);
  }
}

int insert_points_async(MapS* m, const float* pts_dev, uint64_t n, const uint32_t* ends_dev, uint32_t ncl,
                        const uint32_t* meanings_dev, uint32_t meaning, const OutsideFlag& outside)
{
  if (n == 0) return GVX_OK;
  unsigned g = grid_for(n, 256, 1u << 16);
  hipStream_t s = rt().stream;
  ProfScope ps("insert_points");
  // Prob and Distance voxels: updates with different meanings do not commute
  // (saturating log-odds of both signs; last-writer distance voxels), so a
  // multi-cloud insert runs cloud by cloud in order = the serial point order.
  // Within a cloud every update is the same and commutes.
  if (m->type != TBIT && ends_dev && meanings_dev && ncl > 1) {
    const unsigned gc = grid_for((n + ncl - 1) / ncl, 256, 1u << 16);
    for (uint32_t c = 0; c < ncl; ++c) {
      if (m->type == TPROB)
        hipLaunchKernelGGL(k_insert_cloud<TPROB>, dim3(gc), dim3(256), 0, s, (uint8_t*)m->data, m->dims[0],
                           m->dims[1], m->dims[2], m->side, pts_dev, ends_dev, c, meanings_dev, m->uninit, outside);
      else
        hipLaunchKernelGGL(k_insert_cloud<TDIST>, dim3(gc), dim3(256), 0, s, (uint8_t*)m->data, m->dims[0],
                           m->dims[1], m->dims[2], m->side, pts_dev, ends_dev, c, meanings_dev, m->uninit, outside);
    }
    GVX_HIP(hipGetLastError());
    return GVX_OK;
  }
#define LAUNCH(T)                                                                                           \
  hipLaunchKernelGGL(k_insert_points<T>, dim3(g), dim3(256), 0, s, (uint8_t*)m->data, m->dims[0], m->dims[1], \
                     m->dims[2], m->side, pts_dev, n, ends_dev, ncl, meanings_dev, meaning, m->uninit, outside)
  if (m->type == TBIT) LAUNCH(TBIT);
  else if (m->type == TPROB) LAUNCH(TPROB);
  else LAUNCH(TDIST);
#undef LAUNCH
  GVX_HIP(hipGetLastError());
  return GVX_OK;
}

// ---------------------------------------------------------------- sensor data
// insertSensorData (ProbVoxelMap.hpp:51-78, kernelInsertSensorData
// VoxelMapOperations.hpp:763-809).  The reference updates voxels with unguarded
// read-modify-writes from all rays at once; here one scan is deterministic: pass 1
// applies the FREE update (-10) to every cell of every ray, pass 2 the OCCUPIED
// update (+72) to every measured voxel.  Updates of one sign commute under the
// saturating rule, so each pass is order independent.

// point -> voxel if it is used: not NaN, point and sensor voxel inside the map,
// and (with a robot map) the robot does not occupy the voxel with robot_bit
__device__ __forceinline__ bool sensor_point(const float* __restrict__ p, float side, uint32_t dx, uint32_t dy,
                                             uint32_t dz, bool sensor_in, const uint8_t* __restrict__ robot,
                                             uint32_t robot_bit, uint32_t& x, uint32_t& y, uint32_t& z)
{
  const float px = p[0], py = p[1], pz = p[2];
  if (!sensor_in || px != px || py != py || pz != pz) return false;
  x = quantize(px, side);
  y = quantize(py, side);
  z = quantize(pz, side);
  if (!(x < dx && y < dy && z < dz)) return false;
  if (robot) {
    const uint8_t b = robot[(((uint64_t)z * dy + y) * dx + x) * 32 + (robot_bit >> 3)];
    if ((b >> (robot_bit & 7)) & 1u) return false;
  }
  return true;
}

// Points that fall into the same voxel cast the same ray (RayCaster::rayCast walks
// from the sensor voxel to the point's voxel) and add the same OCCUPIED update, so
// the scan runs once per distinct target voxel with its point count as a weight,
// which gives the same result (updates of one sign commute under the saturating
// rule).  The representative of a voxel is its lowest-indexed point, so the
// representatives keep the image order (neighbouring lanes walk neighbouring rays).
//
// counters of one scan: distinct targets, (ray, brick) pairs, chunks of pairs, bricks with
// several chunks; cleared by the tag kernel
struct SensorState {
  uint32_t targets, pairs, chunks, split;
};

// tag: hits[voxel] = max over its points of ~i (hits is zero at rest)
__global__ void __launch_bounds__(256) k_sensor_tag(uint32_t* __restrict__ hits, uint32_t dx, uint32_t dy, uint32_t dz,
                                                    float side, bool sensor_in, const float* __restrict__ pts,
                                                    uint64_t n, const uint8_t* __restrict__ robot, uint32_t robot_bit,
                                                    SensorState* __restrict__ st)
{
  if (blockIdx.x == 0 && threadIdx.x == 0) *st = SensorState{0u, 0u, 0u, 0u};
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    uint32_t x = 0, y = 0, z = 0;
    const bool in = sensor_point(pts + 3 * i, side, dx, dy, dz, sensor_in, robot, robot_bit, x, y, z);
    const uint64_t v = in ? ((uint64_t)z * dy + y) * dx + x : 0ull;
    // a run of consecutive points in one voxel: its first (lowest) index is the run's maximum ~i
    if (wave_run_head(in, v, 0u)) atomicMax(hits + v, ~(uint32_t)i);
  }
}

// the representatives, compacted: slot k holds a voxel (list), a weight to be counted and
// pos[representative] = k.  A block's slots are consecutive and in image order
// (neighbouring lanes walk neighbouring rays); blocks take theirs as they come (one
// atomic each), which changes no result.  A scan of flags took five launches.
constexpr int REP_BLOCK = 1024;
__global__ void __launch_bounds__(REP_BLOCK) k_sensor_rep(const uint32_t* __restrict__ hits, uint32_t dx, uint32_t dy,
                                                          uint32_t dz, float side, bool sensor_in,
                                                          const float* __restrict__ pts, uint64_t n,
                                                          const uint8_t* __restrict__ robot, uint32_t robot_bit,
                                                          SensorState* __restrict__ st, uint32_t* __restrict__ pos,
                                                          uint64_t* __restrict__ list, uint32_t* __restrict__ weight)
{
  __shared__ uint32_t wsum[REP_BLOCK / 64], wbase;
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  for (uint64_t i0 = (uint64_t)blockIdx.x * REP_BLOCK; i0 < n; i0 += (uint64_t)gridDim.x * REP_BLOCK) {  // uniform
    const uint64_t i = i0 + threadIdx.x;
    uint32_t x = 0, y = 0, z = 0;
    uint64_t v = 0;
    bool r = false;
    if (i < n && sensor_point(pts + 3 * i, side, dx, dy, dz, sensor_in, robot, robot_bit, x, y, z)) {
      v = ((uint64_t)z * dy + y) * dx + x;
      r = hits[v] == ~(uint32_t)i;
    }
    const uint64_t bal = wave_ballot(r);
    if (lane == 0) wsum[w] = (uint32_t)__popcll(bal);
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t t = 0;
      for (int k = 0; k < REP_BLOCK / 64; ++k) {
        const uint32_t c = wsum[k];
        wsum[k] = t;
        t += c;
      }
      wbase = t ? atomicAdd(&st->targets, t) : 0u;
    }
    __syncthreads();
    if (r) {
      const uint32_t k = wbase + wsum[w] + (uint32_t)__popcll(bal & ((1ull << lane) - 1ull));
      pos[i] = k;
      list[k] = v;
      weight[k] = 0u;
    }
    __syncthreads();  // wsum and wbase are free again
  }
}

// weight[pos[r]] += 1 for every point of representative r
__global__ void __launch_bounds__(256) k_sensor_weigh(const uint32_t* __restrict__ hits, uint32_t dx, uint32_t dy,
                                                      uint32_t dz, float side, bool sensor_in,
                                                      const float* __restrict__ pts, uint64_t n,
                                                      const uint8_t* __restrict__ robot, uint32_t robot_bit,
                                                      const uint32_t* __restrict__ pos, uint32_t* __restrict__ weight)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    uint32_t x = 0, y = 0, z = 0;
    const bool in = sensor_point(pts + 3 * i, side, dx, dy, dz, sensor_in, robot, robot_bit, x, y, z);
    const uint64_t v = in ? ((uint64_t)z * dy + y) * dx + x : 0ull;
    const uint32_t run = wave_run_head(in, v, 0u);  // consecutive points in one voxel add their count once
    if (run) atomicAdd(weight + pos[~hits[v]], run);
  }
}

// hits back to zero under the representatives' voxels
__global__ void __launch_bounds__(256) k_sensor_untag(uint32_t* __restrict__ hits, const uint64_t* __restrict__ list,
                                                      const SensorState* __restrict__ st)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x, m = st->targets;
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < m; k += stride) hits[list[k]] = 0u;
}

// ---- pass 1, by bricks.  Every cell of every distinct target's ray (RayCaster::rayCast's
// 3-D integer line, VoxelMapOperations.h:218-340) adds the target's weight to a counter.
// Added to counters in memory, even merged over runs of neighbouring lanes, these are 21 M
// device-scope atomics for a 640 x 480 depth image in a 512^3 map (0.6-1.1 ms), which bound
// the scan.  So the cells are counted where they lie: the map is cut into bricks of 16^3
// voxels; each ray is cut into its stretches inside bricks ((ray, entry cell) pairs, about
// one per 16 cells, found without walking), the pairs are sorted by brick, and
// a block walks a brick's pairs with the 4096 counters in LDS and updates the brick's
// voxels itself.  Bricks near the sensor hold most rays: their pairs are cut into chunks of
// SB_CHUNK, whose counters meet in memory (hits, zero at rest) before the voxels are
// updated.  That frame: count 23, place 6, pairs 39, cells 48, split 10 us; all of them
// half bound by instruction issue, half by latency.  Chunks of 1024 pairs, 512 threads
// each and 16 blocks per CU end more evenly than 2048, 256 and 8: cells 69 + split 6 us
// then (4096: 94 + 5; 1024 with 1024 threads 56).
//
// The line steps along x when tx < ty and tx < tz, else along y when ty < tz, else along z,
// where the i-th step of an axis of length d has the time t = (2i + 1) / (2d): the errors of
// the integer walk are these comparisons multiplied out.  So the steps of all axes are one
// sequence ordered by time (ties: z, then y, then x), and both the next brick boundary (the
// earliest of three steps) and the position on the other axes at that moment (steps earlier
// than it) have closed forms.
constexpr uint32_t SB = 16, SB_CELLS = SB * SB * SB;
constexpr uint32_t SB_CHUNK = 1024, SC_THREADS = 512;  // pairs per block at a time, its threads
constexpr uint32_t SB_EDGE = 4095;       // longest map edge: keeps products of step numbers and times in 32 bits
constexpr uint32_t SR_RAYS = 128, SR_THREADS = 1024;  // rays and threads of a block that cuts rays
constexpr uint32_t SH_SLOTS = 2048;      // bricks that such a block counts in LDS
constexpr uint32_t SH_NONE = 0xFFFFFFFFu;

struct SensorGeom {
  uint32_t s[3];       // sensor voxel
  UDiv dxd, dyd;       // map dimensions
  uint32_t bx, by;     // bricks along x and y
};

__device__ __forceinline__ void sensor_target(const SensorGeom& g, uint64_t v, uint32_t (&t)[3])
{
  t[2] = g.dyd.div(g.dxd.div((uint32_t)v, t[0]), t[1]);  // a map has at most 2^32 voxels
}

// floor(n / d) for n < 2^26 and quotients below 2^13 (edges up to SB_EDGE): the float
// quotient is within 1 of it (relative errors of 2^-24 and 2^-22), one step corrects it
__device__ __forceinline__ uint32_t sensor_div(uint32_t n, uint32_t d, float rcp)
{
  const uint32_t q = (uint32_t)((float)n * rcp);
  const int32_t r = (int32_t)(n - q * d);
  return r < 0 ? q - 1 : (uint32_t)r >= d ? q + 1 : q;
}

// a ray's steps per axis, and the step that leaves the sensor's brick along each
struct SensorRay {
  uint32_t d[3], e[3];
  bool up[3];
  __device__ __forceinline__ SensorRay(const SensorGeom& g, const uint32_t (&t)[3])
  {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      up[a] = t[a] > g.s[a];
      d[a] = up[a] ? t[a] - g.s[a] : g.s[a] - t[a];
      e[a] = up[a] ? SB - 1 - g.s[a] % SB : g.s[a] % SB;
    }
  }
  // brick faces crossed along axis a: steps e[a], e[a] + SB, ... below d[a]
  __device__ __forceinline__ uint32_t faces(int a) const { return e[a] < d[a] ? (d[a] - 1 - e[a]) / SB + 1 : 0u; }
  // k[] = steps of every axis up to and with axis ax's step i: those with a time (2j + 1) /
  // d[a] before (2i + 1) / d[ax], or equal to it when a comes first (a > ax)
  __device__ __forceinline__ void steps(int ax, uint32_t i, uint32_t (&k)[3]) const
  {
    const uint32_t ua = 2 * i + 1, da = ax == 0 ? d[0] : ax == 1 ? d[1] : d[2];
    const float rcp = __builtin_amdgcn_rcpf((float)da);
#pragma unroll
    for (int a = 0; a < 3; ++a)
      k[a] = a == ax ? i + 1 : d[a] == 0u ? 0u : (sensor_div(ua * d[a] - (a > ax ? 0u : 1u), da, rcp) + 1) / 2;
  }
  // the ray's f-th entry into a brick in no particular order (0: the sensor's), f below
  // 1 + the faces of all axes: steps taken by then
  __device__ __forceinline__ void entry(uint32_t f, uint32_t f0, uint32_t f1, uint32_t (&k)[3]) const
  {
    if (f == 0u) {
      k[0] = k[1] = k[2] = 0u;
      return;
    }
    --f;
    const int ax = f < f0 ? 0 : f < f0 + f1 ? 1 : 2;
    const uint32_t q = ax == 0 ? f : ax == 1 ? f - f0 : f - f0 - f1;
    steps(ax, (ax == 0 ? e[0] : ax == 1 ? e[1] : e[2]) + q * SB, k);
  }
  // cells from the one after k[] steps to the last one in its brick (both included): up to
  // the earliest of the three next faces, or the target
  __device__ __forceinline__ uint32_t stretch(const uint32_t (&k)[3]) const
  {
    uint32_t n[3];  // each axis's next step that crosses a face
    bool h[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      n[a] = k[a] <= e[a] ? e[a] : e[a] + (k[a] - e[a] + SB - 1) / SB * SB;
      h[a] = n[a] < d[a];
    }
    if (!(h[0] || h[1] || h[2])) return d[0] - k[0] + d[1] - k[1] + d[2] - k[2] + 1;
    const uint32_t u0 = 2 * n[0] + 1, u1 = 2 * n[1] + 1, u2 = 2 * n[2] + 1;
    const bool xy = h[0] && (!h[1] || u0 * d[1] < u1 * d[0]), xz = h[0] && (!h[2] || u0 * d[2] < u2 * d[0]);
    const bool yz = h[1] && (!h[2] || u1 * d[2] < u2 * d[1]);
    const int ax = xy && xz ? 0 : yz ? 1 : 2;
    uint32_t m[3];
    steps(ax, ax == 0 ? n[0] : ax == 1 ? n[1] : n[2], m);
    return m[0] - k[0] + m[1] - k[1] + m[2] - k[2];
  }
  __device__ __forceinline__ void cell(const SensorGeom& g, const uint32_t (&k)[3], uint32_t& brick, uint32_t& at) const
  {
    uint32_t c[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) c[a] = up[a] ? g.s[a] + k[a] : g.s[a] - k[a];
    brick = ((c[2] / SB) * g.by + c[1] / SB) * g.bx + c[0] / SB;
    at = ((c[2] % SB) * SB + c[1] % SB) * SB + c[0] % SB;
  }
};

// The entries of a block's rays, one thread each: the rays' targets and the prefix of
// their entry counts in LDS.  (A thread per ray, face after face, took as long as the
// longest ray: 43 + 77 us for the two kernels below, against 23 + 39 us.)
struct SensorCut {
  uint32_t t[3][SR_RAYS], pre[SR_RAYS + 1];
};
__device__ __forceinline__ void sensor_cut(const SensorGeom& g, const uint64_t* __restrict__ list, uint32_t m,
                                           SensorCut& c)
{
  const uint32_t r = threadIdx.x, k = blockIdx.x * SR_RAYS + r;
  uint32_t n = 0;
  if (r < SR_RAYS && k < m) {
    uint32_t t[3];
    sensor_target(g, list[k], t);
    const SensorRay ray(g, t);
    n = 1 + ray.faces(0) + ray.faces(1) + ray.faces(2);
#pragma unroll
    for (int a = 0; a < 3; ++a) c.t[a][r] = t[a];
  }
  static_assert(SR_RAYS == 128, "two waves");
  uint32_t incl = n;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(incl, o);
    if ((threadIdx.x & 63) >= (uint32_t)o) incl += y;
  }
  if (r < SR_RAYS) c.pre[r + 1] = incl;
  if (r == 0) c.pre[0] = 0u;
  __syncthreads();
  const uint32_t first = c.pre[64];
  __syncthreads();
  if (r >= 64 && r < SR_RAYS) c.pre[r + 1] += first;
  __syncthreads();
}
// the rays of the block's entries [i0, i0 + SP_BATCH), written by 8 threads per ray (a binary
// search of the prefix per entry instead: pairs 41 us, 39 now)
constexpr uint32_t SP_HELD = 4, SP_BATCH = SP_HELD * SR_THREADS;  // entries per thread and per block at a time
__device__ __forceinline__ void sensor_owners(const SensorCut& c, uint32_t i0, uint8_t* own)
{
  static_assert(SR_THREADS == 8 * SR_RAYS && SR_RAYS <= 256, "8 threads per ray, a byte per entry");
  const uint32_t r = threadIdx.x / 8, end = min(c.pre[r + 1], i0 + SP_BATCH);
  for (uint32_t i = max(c.pre[r], i0) + threadIdx.x % 8; i < end; i += 8) own[i - i0] = (uint8_t)r;
  __syncthreads();
}
// entry i of the block's ray r: f(its SensorRay, steps at the entry)
template <typename F>
__device__ __forceinline__ void sensor_entry(const SensorGeom& g, const SensorCut& c, uint32_t r, uint32_t i, F&& f)
{
  const uint32_t t[3] = {c.t[0][r], c.t[1][r], c.t[2][r]};
  const SensorRay ray(g, t);
  uint32_t k[3];
  ray.entry(i - c.pre[r], ray.faces(0), ray.faces(1), k);
  f(ray, k);
}

// a block's bricks with their pairs: slot of brick b, or SH_NONE when the table is full
__device__ __forceinline__ uint32_t sensor_slot(uint32_t* keys, uint32_t b)
{
  uint32_t h = (b * 2654435761u) >> 21;  // SH_SLOTS = 2^11
  for (int probe = 0; probe < 16; ++probe) {
    const uint32_t k = keys[h];
    if (k == b) return h;
    if (k == SH_NONE) {
      const uint32_t old = atomicCAS(&keys[h], SH_NONE, b);
      if (old == SH_NONE || old == b) return h;
    }
    h = (h + 1) % SH_SLOTS;
  }
  return SH_NONE;
}

// pairs per brick: counted per block first (neighbouring rays share bricks).  Also clears
// the targets' tags.
__global__ void __launch_bounds__(SR_THREADS) k_sensor_count(const SensorGeom g, const SensorState* __restrict__ st,
                                                             const uint64_t* __restrict__ list,
                                                             uint32_t* __restrict__ hits, uint32_t* __restrict__ cnt)
{
  __shared__ uint32_t keys[SH_SLOTS], num[SH_SLOTS];
  __shared__ uint8_t own[SP_BATCH];
  __shared__ SensorCut cut;
  const uint32_t m = st->targets;
  if (blockIdx.x * SR_RAYS >= m) return;  // uniform
  for (uint32_t i = threadIdx.x; i < SH_SLOTS; i += SR_THREADS) {
    keys[i] = SH_NONE;
    num[i] = 0u;
  }
  if (threadIdx.x < SR_RAYS && blockIdx.x * SR_RAYS + threadIdx.x < m) hits[list[blockIdx.x * SR_RAYS + threadIdx.x]] = 0u;
  sensor_cut(g, list, m, cut);
  const uint32_t total = cut.pre[SR_RAYS];
  for (uint32_t i0 = 0; i0 < total; i0 += SP_BATCH) {  // uniform
    sensor_owners(cut, i0, own);
    for (uint32_t i = i0 + threadIdx.x; i < min(total, i0 + SP_BATCH); i += SR_THREADS)
      sensor_entry(g, cut, own[i - i0], i, [&](const SensorRay& ray, const uint32_t (&k)[3]) {
        uint32_t b, at;
        ray.cell(g, k, b, at);
        const uint32_t h = sensor_slot(keys, b);
        if (h != SH_NONE) atomicAdd(&num[h], 1u);
        else atomicAdd(cnt + b, 1u);
      });
    __syncthreads();
  }
  for (uint32_t i = threadIdx.x; i < SH_SLOTS; i += SR_THREADS)
    if (num[i]) atomicAdd(cnt + keys[i], num[i]);
}

// places of the bricks' pairs (any order of bricks serves) and their chunks; counts back to
// zero.  Two device atomics per block of 1024 bricks: per wave they were 7.2 us of one address
// after the other (32768 bricks; 5.0 with the same chunks now).
__global__ void __launch_bounds__(1024) k_sensor_place(uint32_t nb, SensorState* __restrict__ st, uint32_t* __restrict__ cnt,
                                                       uint32_t* __restrict__ cursor, uint4* __restrict__ chunks,
                                                       uint32_t* __restrict__ split)
{
  __shared__ uint32_t wp[17], wk[17];
  const uint32_t b = blockIdx.x * 1024 + threadIdx.x, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t c = b < nb ? cnt[b] : 0u, cc = (c + SB_CHUNK - 1) / SB_CHUNK;
  uint32_t pc = c, pk = cc;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y0 = __shfl_up(pc, o), y1 = __shfl_up(pk, o);
    if (lane >= (uint32_t)o) {
      pc += y0;
      pk += y1;
    }
  }
  if (lane == 63) {
    wp[w + 1] = pc;
    wk[w + 1] = pk;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    uint32_t* s = threadIdx.x ? wk : wp;
    uint32_t sum = 0;
    for (int i = 1; i <= 16; ++i) sum += s[i];
    s[0] = sum ? atomicAdd(threadIdx.x ? &st->chunks : &st->pairs, sum) : 0u;
    for (int i = 1; i < 16; ++i) s[i] += s[i - 1];
  }
  __syncthreads();
  if (c == 0u) return;
  const uint32_t base = wp[w] + pc - c, kbase = wk[w] + pk - cc;
  cnt[b] = 0u;
  cursor[b] = base;
  for (uint32_t k = 0; k < cc; ++k)
    chunks[kbase + k] = make_uint4(b, base + k * SB_CHUNK, min(SB_CHUNK, c - k * SB_CHUNK), cc > 1 ? 1u : 0u);
  if (cc > 1) split[atomicAdd(&st->split, 1u)] = b;
}

// the pairs (ray; entry cell and number of cells), sorted by brick: a block takes SP_HELD
// entries per thread at a time, counts them per brick, takes a stretch per brick and fills
// it.  An entry's pair and place wait in registers for the stretch (cut twice instead: 60 us,
// 39 now; 512 threads 50).
__global__ void __launch_bounds__(SR_THREADS) k_sensor_pairs(const SensorGeom g, const SensorState* __restrict__ st,
                                                             const uint64_t* __restrict__ list,
                                                             uint32_t* __restrict__ cursor, uint2* __restrict__ pairs)
{
  __shared__ uint32_t keys[SH_SLOTS], num[SH_SLOTS];
  __shared__ uint8_t own[SP_BATCH];
  __shared__ SensorCut cut;
  const uint32_t m = st->targets;
  if (blockIdx.x * SR_RAYS >= m) return;  // uniform
  sensor_cut(g, list, m, cut);
  const uint32_t total = cut.pre[SR_RAYS];
  for (uint32_t i0 = 0; i0 < total; i0 += SP_BATCH) {  // uniform
    for (uint32_t i = threadIdx.x; i < SH_SLOTS; i += SR_THREADS) {
      keys[i] = SH_NONE;
      num[i] = 0u;
    }
    sensor_owners(cut, i0, own);
    uint32_t what[SP_HELD], slot[SP_HELD], nth[SP_HELD];
#pragma unroll
    for (uint32_t j = 0; j < SP_HELD; ++j) {
      const uint32_t i = i0 + j * SR_THREADS + threadIdx.x;
      slot[j] = SH_NONE;
      if (i < total) {
        const uint32_t r = own[i - i0];
        sensor_entry(g, cut, r, i, [&](const SensorRay& ray, const uint32_t (&k)[3]) {
          uint32_t b, at;
          ray.cell(g, k, b, at);
          what[j] = at | ray.stretch(k) << 12 | r << 18;  // at most 46 cells
          slot[j] = sensor_slot(keys, b);
          if (slot[j] != SH_NONE) nth[j] = atomicAdd(&num[slot[j]], 1u);
          else pairs[atomicAdd(cursor + b, 1u)] = make_uint2(blockIdx.x * SR_RAYS + r, what[j] & 0x3FFFFu);
        });
      }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < SH_SLOTS; i += SR_THREADS)
      if (num[i]) num[i] = atomicAdd(cursor + keys[i], num[i]);
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < SP_HELD; ++j)
      if (slot[j] != SH_NONE)
        pairs[num[slot[j]] + nth[j]] = make_uint2(blockIdx.x * SR_RAYS + (what[j] >> 18), what[j] & 0x3FFFFu);
    __syncthreads();
  }
}

// F free updates in a row on one voxel = max((unknown ? 0 : v) - 10 F, -127)
// (updateOccupancy saturates at MIN_PROBABILITY)
__device__ __forceinline__ uint8_t sensor_free(uint8_t old, uint32_t f)
{
  int v = (int)(int8_t)old;
  if (v == PROB_UNKNOWN) v = 0;
  return (uint8_t)(int8_t)max(v - 10 * (int)min(f, 64u), PROB_MIN);
}

__device__ __forceinline__ uint64_t sensor_voxel(const SensorGeom& g, uint32_t brick, uint32_t cell)
{
  const uint32_t x = brick % g.bx * SB + cell % SB, y = brick / g.bx % g.by * SB + cell / SB % SB,
                 z = brick / (g.bx * g.by) * SB + cell / (SB * SB);
  return ((uint64_t)z * g.dyd.d + y) * g.dxd.d + x;
}

__global__ void __launch_bounds__(SC_THREADS) k_sensor_cells(const SensorGeom g, const SensorState* __restrict__ st,
                                                      const uint4* __restrict__ chunks, const uint2* __restrict__ pairs,
                                                      const uint64_t* __restrict__ list,
                                                      const uint32_t* __restrict__ weight, uint8_t* __restrict__ map,
                                                      uint32_t* __restrict__ hits)
{
  __shared__ uint4 num4[SB_CELLS / 4];
  uint32_t* num = reinterpret_cast<uint32_t*>(num4);
  const uint32_t nc = st->chunks;
  for (uint32_t c = blockIdx.x; c < nc; c += gridDim.x) {  // uniform over the block
    const uint4 ch = chunks[c];
    for (uint32_t i = threadIdx.x; i < SB_CELLS / 4; i += SC_THREADS) num4[i] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
    const uint32_t o[3] = {ch.x % g.bx * SB, ch.x / g.bx % g.by * SB, ch.x / (g.bx * g.by) * SB};  // first voxel
    for (uint32_t i = threadIdx.x; i < ch.z; i += SC_THREADS) {
      const uint2 pr = pairs[ch.y + i];
      const uint32_t wgt = weight[pr.x];
      uint32_t t[3];
      sensor_target(g, list[pr.x], t);
      const SensorRay ray(g, t);
      uint32_t cell = pr.y % SB_CELLS, len = pr.y / SB_CELLS;
      // The axes' next times as integers, (2k + 1) d[b] d[c] for steps k taken and the other
      // axes' lengths (1 for 0), less the earliest so that they and the at most 46
      // increments 2 d[b] d[c] after it stay below 2^32 (differences are exact modulo 2^32).
      // An axis without steps never comes.
      uint32_t k[3], T[3], inc[3];
      const uint32_t l[3] = {cell % SB, cell / SB % SB, cell / (SB * SB)};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const uint32_t at = o[a] + l[a], p = max(ray.d[(a + 1) % 3], 1u) * max(ray.d[(a + 2) % 3], 1u);
        k[a] = ray.up[a] ? at - g.s[a] : g.s[a] - at;
        T[a] = (2 * k[a] + 1) * p;
        inc[a] = 2 * p;
      }
      uint32_t t0 = 0;
      bool none = true;
#pragma unroll
      for (int a = 0; a < 3; ++a)
        if (ray.d[a] != 0u && (none || (int32_t)(T[a] - t0) < 0)) {
          t0 = T[a];
          none = false;
        }
      uint32_t tx = ray.d[0] ? T[0] - t0 : 0xFFFFFFFFu, ty = ray.d[1] ? T[1] - t0 : 0xFFFFFFFFu,
               tz = ray.d[2] ? T[2] - t0 : 0xFFFFFFFFu;
      const uint32_t sx = ray.up[0] ? 1u : 0u - 1u, sy = ray.up[1] ? SB : 0u - SB, sz = ray.up[2] ? SB * SB : 0u - SB * SB;
      for (;;) {
        atomicAdd(&num[cell], wgt);
        if (--len == 0u) break;
        const bool x = tx < ty && tx < tz, y = !x && ty < tz;
        cell += x ? sx : y ? sy : sz;
        tx += x ? inc[0] : 0u;
        ty += y ? inc[1] : 0u;
        tz += x || y ? 0u : inc[2];
      }
    }
    __syncthreads();
    // 16 neighbouring lanes are 16 neighbouring voxels; bytes, since a word may belong to
    // two bricks
    for (uint32_t i = threadIdx.x; i < SB_CELLS; i += SC_THREADS) {
      const uint32_t f = num[i];
      if (!f) continue;
      const uint64_t v = sensor_voxel(g, ch.x, i);
      if (ch.w) atomicAdd(hits + v, f);
      else map[v] = sensor_free(map[v], f);
    }
    __syncthreads();
  }
}

// bricks whose pairs were cut into several chunks
__global__ void __launch_bounds__(1024) k_sensor_split(const SensorGeom g, const SensorState* __restrict__ st,
                                                      const uint32_t* __restrict__ split, uint32_t dz,
                                                      uint8_t* __restrict__ map, uint32_t* __restrict__ hits)
{
  const uint32_t n = st->split;
  for (uint32_t b = blockIdx.x; b < n; b += gridDim.x) {
    const uint32_t brick = split[b];
    const uint32_t x0 = brick % g.bx * SB, y0 = brick / g.bx % g.by * SB, z0 = brick / (g.bx * g.by) * SB;
    for (uint32_t i = threadIdx.x; i < SB_CELLS; i += 1024) {
      if (x0 + i % SB >= g.dxd.d || y0 + i / SB % SB >= g.dyd.d || z0 + i / (SB * SB) >= dz) continue;
      const uint64_t v = sensor_voxel(g, brick, i);
      const uint32_t f = hits[v];
      if (!f) continue;
      hits[v] = 0u;
      map[v] = sensor_free(map[v], f);
    }
  }
}

// pass 1 without bricks, for maps with an edge above SB_EDGE and for scans whose pairs
// would pass SB_PAIR_BYTES or find no memory: one lane per distinct target voxel walks the
// line from the sensor voxel to the target and adds the target's weight to the 32-bit
// counter of every cell it visits (atomics without a return value: the walk never waits).  Rays of neighbouring
// targets (consecutive lanes) share many cells, so at every step each run of
// consecutive lanes on one cell adds its summed weight once (a 640 x 480 depth
// image into a 512^3 map: 21.4 M atomics for 50.7 M cells walked).
__global__ void __launch_bounds__(256) k_sensor_rays(uint32_t* __restrict__ hits, uint32_t dx, uint32_t dy, uint32_t dz,
                                                     uint32_t sx, uint32_t sy, uint32_t sz,
                                                     const uint64_t* __restrict__ list,
                                                     const uint32_t* __restrict__ weight,
                                                     const SensorState* __restrict__ st)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t first = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t m = st->targets;
  const uint64_t rounds = (m + stride - 1) / stride;  // uniform trip count: every lane reaches the ballots
  const uint32_t lane = threadIdx.x & 63;
  const uint64_t plane = (uint64_t)dx * dy;
  for (uint64_t r = 0; r < rounds; ++r) {
    const uint64_t k = first + r * stride;
    const bool use = k < m;
    uint32_t wgt = 0;
    int32_t d[3] = {0, 0, 0}, inc[3] = {1, 1, 1};
    if (use) {
      const uint64_t v = list[k];
      wgt = weight[k];
      const uint32_t t[3] = {(uint32_t)(v % dx), (uint32_t)((v / dx) % dy), (uint32_t)(v / plane)};
      const uint32_t f[3] = {sx, sy, sz};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        if (t[a] > f[a]) { d[a] = (int32_t)(t[a] - f[a]); inc[a] = 1; }
        else { d[a] = (int32_t)(f[a] - t[a]); inc[a] = -1; }
      }
    }
    int64_t left = use ? 1 + (int64_t)d[0] + d[1] + d[2] : 0;
    int32_t exy = d[0] - d[1], exz = d[0] - d[2], eyz = d[1] - d[2];
    const int32_t dx2 = 2 * d[0], dy2 = 2 * d[1], dz2 = 2 * d[2];
    const int64_t sxs = inc[0], sys = inc[1] * (int64_t)dx, szs = inc[2] * (int64_t)plane;
    uint64_t idx = ((uint64_t)sz * dy + sy) * dx + sx;
    for (;;) {
      const bool active = left > 0;
      const uint64_t am = wave_ballot(active);
      if (am == 0) break;
      // consecutive lanes (neighbouring targets) on one cell form a run; the run's
      // first lane adds the run's summed weight with one atomic
      const uint32_t ilo = (uint32_t)idx, ihi = (uint32_t)(idx >> 32);
      const uint32_t plo = __shfl_up(ilo, 1, 64), phi = __shfl_up(ihi, 1, 64);
      const bool same = active && lane > 0 && ((am >> (lane - 1)) & 1ull) != 0ull && plo == ilo && phi == ihi;
      const uint64_t cont = wave_ballot(same);
      uint32_t v = active ? wgt : 0u;
      if (cont != 0ull) {  // uniform: segmented suffix sums of the weights
        const uint64_t above = lane == 63 ? 0ull : ~cont & (~0ull << (lane + 1));  // run starts after this lane
        const uint32_t end = above != 0ull ? (uint32_t)__builtin_ctzll(above) - 1u : 63u;
        for (uint32_t o = 1; o < 64; o <<= 1) {
          const uint32_t t = __shfl_down(v, o, 64);
          if (lane + o <= end) v += t;
        }
      }
      if (active && !same) atomicAdd(hits + idx, v);
      if (active) {
        if (exy > 0 && exz > 0) { idx += sxs; exy -= dy2; exz -= dz2; }
        else if (eyz > 0) { idx += sys; exy += dx2; eyz -= dz2; }
        else { idx += szs; exz += dx2; eyz += dy2; }
        --left;
      }
    }
  }
}

// pass 1b of that: the counters applied to the voxels and back to zero for the next scan.
// Four voxels per thread.
__global__ void __launch_bounds__(256) k_sensor_apply(uint8_t* __restrict__ map, uint32_t* __restrict__ hits, uint64_t n)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; 4 * q < n; q += stride) {
    const uint64_t i0 = 4 * q;
    if (i0 + 4 <= n) {
      const uint4 h = reinterpret_cast<const uint4*>(hits)[q];
      if ((h.x | h.y | h.z | h.w) == 0u) continue;
      uint32_t w = reinterpret_cast<const uint32_t*>(map)[q];
      const uint32_t hc[4] = {h.x, h.y, h.z, h.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (!hc[k]) continue;
        w = (w & ~(0xFFu << (8 * k))) | ((uint32_t)sensor_free((uint8_t)(w >> (8 * k)), hc[k]) << (8 * k));
      }
      reinterpret_cast<uint32_t*>(map)[q] = w;
      reinterpret_cast<uint4*>(hits)[q] = make_uint4(0u, 0u, 0u, 0u);
    } else {
      for (uint64_t i = i0; i < n; ++i) {
        const uint32_t c = hits[i];
        if (!c) continue;
        map[i] = sensor_free(map[i], c);
        hits[i] = 0u;
      }
    }
  }
}

// pass 2: the measured voxels, each with its point count.  Every voxel is listed once, so its
// byte has one writer (as a CAS on its word: 8.5 us for a depth image's 200 k voxels, 4.2 now).
__global__ void __launch_bounds__(256) k_sensor_hits(uint8_t* __restrict__ map, const uint64_t* __restrict__ list,
                                                     const uint32_t* __restrict__ weight,
                                                     const SensorState* __restrict__ st)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x, m = st->targets;
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < m; k += stride) {
    int8_t* v = reinterpret_cast<int8_t*>(map) + list[k];
    const int cur = *v;
    int nv = cur;
    for (uint32_t c = weight[k]; c; --c) {
      const int next = prob_update(nv, SENSOR_OCC);
      if (next == nv) break;
      nv = next;
    }
    if (nv != cur) *v = (int8_t)nv;
  }
}

// ---------------------------------------------------------------- swept volumes
// collisionCheckBitvector with SVCollider(thr, window) for Bit x Bit
// (BitVoxelMap.hpp:90-142, kernelCollideVoxelMapsBitvector
// VoxelMapOperations.hpp:186-239): bitMarginCollisionCheck per voxel, colliding
// voxels of self get eBVM_COLLISION, the mask ORs every colliding voxel's result.
__global__ void __launch_bounds__(256) k_collide_sv(uint8_t* __restrict__ a, const uint8_t* __restrict__ b, uint64_t n,
                                                    uint32_t margin, uint32_t sv_offset,
                                                    unsigned long long* __restrict__ count, uint32_t* __restrict__ mask)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  uint64_t c = 0;
  uint32_t acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    uint4* pa = reinterpret_cast<uint4*>(a + i * 32);
    const uint4* pb = reinterpret_cast<const uint4*>(b + i * 32);
    const uint4 a0 = pa[0], a1 = pa[1], b0 = pb[0], b1 = pb[1];
    const uint32_t va[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
    const uint32_t vb[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
    bool hit = false;
    // an empty side cannot collide: skip the byte loop for it
    if ((va[0] | va[1] | va[2] | va[3] | va[4] | va[5] | va[6] | va[7]) &&
        ((vb[0] & 0xFFFFFFF0u) | vb[1] | vb[2] | vb[3] | vb[4] | vb[5] | vb[6] | vb[7])) {
      uint32_t r[8];
      hit = bitmargin(va, vb, margin, sv_offset, r);
      if (hit) {
#pragma unroll
        for (int k = 0; k < 8; ++k) acc[k] |= r[k];
        reinterpret_cast<uint32_t*>(pa)[0] = a0.x | (1u << M_COLLISION);
      }
    }
    c += hit ? 1u : 0u;
  }
  add_hits(c, acc, count, mask);
}

// shiftLeftSweptVolumeIDs (BitVoxelMap.hpp:351-362 -> kernelShiftBitVector,
// VoxelMapOperations.hpp:815-823): performLeftShift on every 32-byte voxel
__global__ void __launch_bounds__(256) k_shift_sv(uint8_t* __restrict__ v, uint64_t n, uint32_t shift)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    uint4* p = reinterpret_cast<uint4*>(v + i * 32);
    const uint4 a0 = p[0], a1 = p[1];
    uint32_t w[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
    left_shift_sv(w, shift);
    p[0] = make_uint4(w[0], w[1], w[2], w[3]);
    p[1] = make_uint4(w[4], w[5], w[6], w[7]);
  }
}

// per-voxel words of insertSensorData (tags, then ray counters): allocated zeroed once
// per size and left zeroed by every scan, as are the bricks' counts below.  Open: taken by
// a scan that did not reach its end, and cleared before the next use.
static bool sensor_hits_open = false, sensor_bricks_open = false;
static int sensor_hits_buffer(uint64_t n, uint32_t** out)
{
  static uint32_t* buf = nullptr;
  static uint64_t cap = 0;
  if (cap < n) {
    GVX_CHECK(sync());
    dfree(buf);
    buf = nullptr;
    cap = 0;
    GVX_CHECK(dalloc((void**)&buf, ((n + 3) / 4) * 16));
    GVX_CHECK(fill_u32(buf, 0u, ((n + 3) / 4) * 4));
    cap = n;
  } else if (sensor_hits_open) {
    GVX_CHECK(fill_u32(buf, 0u, ((cap + 3) / 4) * 4));
  }
  sensor_hits_open = true;
  *out = buf;
  return GVX_OK;
}

// arrays of one scan (grown on demand, kept): representative slots and weights (n words
// each), target voxels (n u64)
struct SensorPoints {
  SensorState* st = nullptr;
  uint32_t *pos = nullptr, *weight = nullptr;
  uint64_t* list = nullptr;
};
static int sensor_points(uint64_t n, SensorPoints* out)
{
  static uint8_t* buf = nullptr;
  static uint64_t cap = 0;
  const auto al = [](uint64_t b) { return (b + 255) & ~(uint64_t)255; };
  if (cap < n) {
    GVX_CHECK(sync());
    dfree(buf);
    buf = nullptr;
    cap = 0;
    GVX_CHECK(dalloc((void**)&buf, 256 + al(4 * n) + al(4 * n) + al(8 * n)));
    cap = n;
  }
  out->st = (SensorState*)buf;
  out->pos = (uint32_t*)(buf + 256);
  out->weight = (uint32_t*)(buf + 256 + al(4 * cap));
  out->list = (uint64_t*)(buf + 256 + 2 * al(4 * cap));
  return GVX_OK;
}

// bricks and pairs of one scan: n rays enter at most bx + by + bz bricks each (236 MB for a
// 640 x 480 frame in 512^3); counts are zero between scans.  Without the memory for them
// (GVX_ERR_OOM) nothing is kept, and the scan goes without bricks.
constexpr uint64_t SB_PAIR_BYTES = 2ull << 30;
struct SensorBricks {
  uint32_t *cnt = nullptr, *cursor = nullptr, *split = nullptr;
  uint4* chunks = nullptr;
  uint2* pairs = nullptr;
};
static int sensor_bricks_buffers(uint64_t nb, uint64_t pairs, SensorBricks* out)
{
  static SensorBricks b;
  static uint64_t cap_b = 0, cap_p = 0;
  if (cap_b < nb || cap_p < pairs) {
    GVX_CHECK(sync());
    const auto drop = [] {
      dfree(b.cnt); dfree(b.cursor); dfree(b.split); dfree(b.chunks); dfree(b.pairs);
      b = SensorBricks();
      cap_b = cap_p = 0;
    };
    const uint64_t need_b = nb, need_p = pairs;
    nb = std::max(nb, cap_b);
    pairs = std::max(pairs, cap_p);
    int s;
    for (;;) {
      drop();
      if ((s = dalloc((void**)&b.cnt, nb * 4)) == GVX_OK && (s = dalloc((void**)&b.cursor, nb * 4)) == GVX_OK &&
          (s = dalloc((void**)&b.split, nb * 4)) == GVX_OK &&
          (s = dalloc((void**)&b.chunks, (nb + pairs / SB_CHUNK + 1) * 16)) == GVX_OK &&
          (s = dalloc((void**)&b.pairs, pairs * 8)) == GVX_OK)
        break;
      if (nb == need_b && pairs == need_p) {
        drop();
        return s;
      }
      nb = need_b;  // not the room of earlier scans too
      pairs = need_p;
    }
    GVX_CHECK(fill_u32(b.cnt, 0u, nb));
    cap_b = nb;
    cap_p = pairs;
  } else if (sensor_bricks_open) {
    GVX_CHECK(fill_u32(b.cnt, 0u, cap_b));
  }
  sensor_bricks_open = true;
  *out = b;
  return GVX_OK;
}

// per-point flags of the self-collision test (grown on demand, kept)
static int selfcoll_flags(uint64_t n, uint8_t** out)
{
  static uint8_t* buf = nullptr;
  static uint64_t cap = 0;
  if (cap < n) {
    GVX_CHECK(sync());
    dfree(buf);
    buf = nullptr;
    cap = 0;
    GVX_CHECK(dalloc((void**)&buf, (n + 255) & ~(uint64_t)255));
    cap = n;
  }
  *out = buf;
  return GVX_OK;
}

// insertMetaPointCloudWithSelfCollisionCheck on device points: sub-clouds in
// order, each a test launch and an insert launch.  acc_dev: 9 words (colliding
// meanings, points-outside flag), cleared here.  meanings / masks on the host,
// NULL for the defaults (BitVoxelMap.hpp:262-292).
int selfcoll_insert_async(MapS* m, const float* pts_dev, const uint32_t* sizes, uint32_t ncl,
                          const uint32_t* meanings, const uint8_t* masks, uint32_t* acc_dev)
{
  if (m->type != TBIT)
    return fail(GVX_ERR_UNSUPPORTED, "insertMetaPointCloudWithSelfCollisionCheck: BitVector maps only");
  uint64_t total = 0;
  for (uint32_t c = 0; c < ncl; ++c) {
    total += sizes[c];
    const uint32_t mc = meanings ? meanings[c] : M_SV_START + c;
    if (mc > 255) return fail(GVX_ERR_BAD_ARG, "meaning > 255");
  }
  uint8_t* hit = nullptr;
  GVX_CHECK(selfcoll_flags(total ? total : 1, &hit));
  GVX_CHECK(fill_u32(acc_dev, 0u, 12));
  hipStream_t s = rt().stream;
  uint64_t off = 0;
  for (uint32_t c = 0; c < ncl; ++c) {
    const uint32_t mc = meanings ? meanings[c] : M_SV_START + c;
    uint32_t w[8];
    if (masks) {
      memcpy(w, masks + (uint64_t)c * 32, 32);
    } else {
      for (int k = 0; k < 8; ++k) w[k] = 0xFFFFFFFFu;
      w[M_COLLISION >> 5] &= ~(1u << (M_COLLISION & 31));
      w[mc >> 5] &= ~(1u << (mc & 31));
    }
    const uint64_t n = sizes[c];
    if (n) {
      const unsigned g = grid_for(n, 256, 1u << 14);
      hipLaunchKernelGGL(k_selfcoll_test, dim3(g), dim3(256), 0, s, (const uint32_t*)m->data, m->dims[0], m->dims[1],
                         m->dims[2], m->side, pts_dev + 3 * off, n, make_uint4(w[0], w[1], w[2], w[3]),
                         make_uint4(w[4], w[5], w[6], w[7]), mc, hit + off, acc_dev);
      hipLaunchKernelGGL(k_selfcoll_insert, dim3(g), dim3(256), 0, s, (uint32_t*)m->data, m->dims[0], m->dims[1],
                         m->dims[2], m->side, pts_dev + 3 * off, n, mc, (const uint8_t*)(hit + off));
      GVX_HIP(hipGetLastError());
    }
    off += n;
  }
  return GVX_OK;
}

// colliding meanings and flags back from acc (after selfcoll_insert_async)
int selfcoll_finish(const uint32_t* acc_dev, uint8_t colliding[32], int* self_collision, int* points_outside)
{
  Runtime& r = rt();
  GVX_HIP(hipMemcpyAsync(r.host_small, acc_dev, 36, hipMemcpyDeviceToHost, r.stream));
  GVX_CHECK(sync());
  const uint32_t* h = (const uint32_t*)r.host_small;
  uint32_t any = 0;
  for (int k = 0; k < 8; ++k) any |= h[k];
  if (colliding) memcpy(colliding, h, 32);
  if (self_collision) *self_collision = any != 0u;
  if (points_outside) *points_outside = (int)h[8];
  return GVX_OK;
}

int shift_sv_async(uint8_t* voxels, uint64_t n, uint32_t shift)
{
  if (!n) return GVX_OK;
  hipLaunchKernelGGL(k_shift_sv, dim3(grid_for(n, 256, 1u << 16)), dim3(256), 0, rt().stream, voxels, n, shift);
  GVX_HIP(hipGetLastError());
  return GVX_OK;
}

}  // namespace gvx

using namespace gvx;

static int check_map(gvx_map m)
{
  if (!m || !m->data) return fail(GVX_ERR_BAD_ARG, "null map handle");
  return GVX_OK;
}

extern "C" {

int gvx_map_create(int type, uint32_t dx, uint32_t dy, uint32_t dz, float side, gvx_map* out)
{
  if (!out) return fail(GVX_ERR_BAD_ARG, "gvx_map_create: out is null");
  *out = nullptr;
  GVX_CHECK(ensure_init());
  if (type != TBIT && type != TPROB && type != TDIST)
    return fail(GVX_ERR_UNSUPPORTED, "THIS TYPE OF DATA STRUCTURE IS NOT YET IMPLEMENTED!");
  if (dx == 0 || dy == 0 || dz == 0 || !(side > 0.0f)) return fail(GVX_ERR_BAD_ARG, "gvx_map_create: bad dims/side");
  if (type == TDIST && (dx > 1024 || dy > 1024 || dz > 4094))
    return fail(GVX_ERR_UNSUPPORTED, "DistanceVoxelMap: x,y <= 1024 and z <= 4094 (10/10/12-bit packing)");
  uint64_t n = (uint64_t)dx * dy * dz;
  if (n > (1ull << 32)) return fail(GVX_ERR_UNSUPPORTED, "map larger than 2^32 voxels");
  gvx_map m = new gvx_map_s();
  m->type = type;
  m->dims[0] = dx; m->dims[1] = dy; m->dims[2] = dz;
  m->side = side;
  m->n = n;
  m->bytes = n * voxel_bytes(type);
  m->uninit = dist_uninit(m->dims);
  size_t alloc = (m->bytes + 255) & ~(size_t)255;
  int s = dalloc(&m->data, alloc);
  if (s != GVX_OK) { delete m; return s; }
  s = map_clear_async(m);
  if (s == GVX_OK) s = sync();
  if (s != GVX_OK) { dfree(m->data); delete m; return s; }
  *out = m;
  return GVX_OK;
}

int gvx_map_destroy(gvx_map m)
{
  if (!m) return GVX_OK;
  (void)sync();
  dfree(m->data);
  delete m;
  return GVX_OK;
}

int gvx_map_info(gvx_map m, int* type, uint32_t dims[3], float* side, uint64_t* bytes)
{
  GVX_CHECK(check_map(m));
  if (type) *type = m->type;
  if (dims) { dims[0] = m->dims[0]; dims[1] = m->dims[1]; dims[2] = m->dims[2]; }
  if (side) *side = m->side;
  if (bytes) *bytes = m->bytes;
  return GVX_OK;
}

int gvx_map_device_ptr(gvx_map m, void** ptr)
{
  GVX_CHECK(check_map(m));
  if (!ptr) return fail(GVX_ERR_BAD_ARG, "null");
  *ptr = m->data;
  return GVX_OK;
}

int gvx_map_clear(gvx_map m)
{
  GVX_CHECK(check_map(m));
  std::lock_guard<std::recursive_mutex> g(m->mu);
  {
    ProfScope ps("clear_map");
    GVX_CHECK(map_clear_async(m));
  }
  return sync();
}

int gvx_map_clear_bits(gvx_map m, const uint8_t bits[32])
{
  GVX_CHECK(check_map(m));
  if (m->type != TBIT) return fail(GVX_ERR_UNSUPPORTED, "clearBits needs a BitVector map");
  if (!bits) return fail(GVX_ERR_BAD_ARG, "null bits");
  std::lock_guard<std::recursive_mutex> g(m->mu);
  uint32_t w[8];
  memcpy(w, bits, 32);
  hipLaunchKernelGGL(k_clear_bits, dim3(stream_grid(m->n)), dim3(256), 0, rt().stream, (uint32_t*)m->data, m->n,
                     make_uint4(w[0], w[1], w[2], w[3]), make_uint4(w[4], w[5], w[6], w[7]));
  GVX_HIP(hipGetLastError());
  return sync();
}

int gvx_map_read(gvx_map m, void* dst, int mem)
{
  GVX_CHECK(check_map(m));
  if (!dst) return fail(GVX_ERR_BAD_ARG, "null dst");
  std::lock_guard<std::recursive_mutex> g(m->mu);
  GVX_CHECK(copy_out(dst, m->data, m->bytes, mem));
  return sync();
}

int gvx_map_write(gvx_map m, const void* src, int mem)
{
  GVX_CHECK(check_map(m));
  if (!src) return fail(GVX_ERR_BAD_ARG, "null src");
  std::lock_guard<std::recursive_mutex> g(m->mu);
  GVX_CHECK(copy_in(m->data, src, m->bytes, mem));
  return sync();
}

static int finish_outside(const OutsideFlag& f, int* points_outside)
{
  GVX_CHECK(sync());
  if (points_outside) *points_outside = f.raised() ? 1 : 0;
  return GVX_OK;
}

int gvx_map_insert_points(gvx_map m, const float* xyz, uint64_t n, uint32_t meaning, int mem, int* points_outside)
{
  GVX_CHECK(check_map(m));
  if (n && !xyz) return fail(GVX_ERR_BAD_ARG, "null points");
  if (meaning > 255) return fail(GVX_ERR_BAD_ARG, "meaning > 255");
  std::lock_guard<std::recursive_mutex> g(m->mu);
  std::lock_guard<std::recursive_mutex> g2(rt().mu);
  const void* d = nullptr;
  GVX_CHECK(stage_input(xyz, n * 12, mem, &d));
  const OutsideFlag f = outside_flag();
  GVX_CHECK(insert_points_async(m, (const float*)d, n, nullptr, 0, nullptr, meaning, f));
  return finish_outside(f, points_outside);
}

int gvx_map_insert_sensor(gvx_map m, const float* xyz, uint64_t n, const float sensor_pose[3], int enable_raycasting,
                          const void* robot_bits_dev, uint32_t robot_meaning, int mem)
{
  GVX_CHECK(check_map(m));
  if (m->type != TPROB) return fail(GVX_ERR_UNSUPPORTED, "insertSensorData needs a ProbVoxelMap");
  if (!sensor_pose) return fail(GVX_ERR_BAD_ARG, "null sensor pose");
  if (n && !xyz) return fail(GVX_ERR_BAD_ARG, "null points");
  if (robot_meaning > 255) return fail(GVX_ERR_BAD_ARG, "meaning > 255");
  if (n > m->n) n = m->n;  // the reference's loop also stops at the map size
  std::lock_guard<std::recursive_mutex> g(m->mu);
  std::lock_guard<std::recursive_mutex> g2(rt().mu);
  if (!n) return GVX_OK;
  const void* d = nullptr;
  GVX_CHECK(stage_input(xyz, n * 12, mem, &d));
  const float side = m->side;
  const uint32_t sx = quantize(sensor_pose[0], side), sy = quantize(sensor_pose[1], side),
                 sz = quantize(sensor_pose[2], side);
  const bool sin = sx < m->dims[0] && sy < m->dims[1] && sz < m->dims[2];
  const uint8_t* robot = (const uint8_t*)robot_bits_dev;
  hipStream_t s = rt().stream;
  if (n >= 0xFFFFFFFFull) return fail(GVX_ERR_UNSUPPORTED, "insertSensorData: more than 2^32 - 2 points");
  uint32_t* hits = nullptr;
  GVX_CHECK(sensor_hits_buffer(m->n, &hits));
  SensorPoints P;
  GVX_CHECK(sensor_points(n, &P));
  const uint32_t dx = m->dims[0], dy = m->dims[1], dz = m->dims[2];
  const uint32_t bx = (dx + SB - 1) / SB, by = (dy + SB - 1) / SB, bz = (dz + SB - 1) / SB;
  const uint64_t nb = (uint64_t)bx * by * bz, pairs = n * (uint64_t)(bx + by + bz);
  bool bricks = enable_raycasting && std::max(dx, std::max(dy, dz)) <= SB_EDGE && pairs * 8 <= SB_PAIR_BYTES;
  SensorBricks B;
  if (bricks) {
    const int e = sensor_bricks_buffers(nb, pairs, &B);
    if (e != GVX_OK && e != GVX_ERR_OOM) return e;
    bricks = e == GVX_OK;
  }
  const SensorGeom geom = {{sx, sy, sz}, udiv(dx), udiv(dy), bx, by};
  const unsigned gp = grid_for(n, 256, 1u << 14);
  {
    // distinct target voxels (in image order) and their point counts
    ProfScope ps("sensor_targets");
    const float* pts = (const float*)d;
    hipLaunchKernelGGL(k_sensor_tag, dim3(gp), dim3(256), 0, s, hits, dx, dy, dz, side, sin, pts, n, robot, robot_meaning,
                       P.st);
    hipLaunchKernelGGL(k_sensor_rep, dim3(grid_for(n, REP_BLOCK, 1u << 14)), dim3(REP_BLOCK), 0, s, hits, dx, dy, dz,
                       side, sin, pts, n, robot, robot_meaning, P.st, P.pos, P.list, P.weight);
    hipLaunchKernelGGL(k_sensor_weigh, dim3(gp), dim3(256), 0, s, hits, dx, dy, dz, side, sin, pts, n, robot,
                       robot_meaning, P.pos, P.weight);
    if (!bricks) hipLaunchKernelGGL(k_sensor_untag, dim3(gp), dim3(256), 0, s, hits, P.list, P.st);
    GVX_HIP(hipGetLastError());
  }
  if (bricks) {
    ProfScope ps("sensor_rays");
    const unsigned gr = (unsigned)((n + SR_RAYS - 1) / SR_RAYS);
    hipLaunchKernelGGL(k_sensor_count, dim3(gr), dim3(SR_THREADS), 0, s, geom, P.st, P.list, hits, B.cnt);
    hipLaunchKernelGGL(k_sensor_place, dim3((unsigned)((nb + 1023) / 1024)), dim3(1024), 0, s, (uint32_t)nb, P.st, B.cnt,
                       B.cursor, B.chunks, B.split);
    hipLaunchKernelGGL(k_sensor_pairs, dim3(gr), dim3(SR_THREADS), 0, s, geom, P.st, P.list, B.cursor, B.pairs);
    const unsigned gc = (unsigned)(rt().num_cus > 0 ? rt().num_cus : 256) * 16;
    hipLaunchKernelGGL(k_sensor_cells, dim3(gc), dim3(SC_THREADS), 0, s, geom, P.st, B.chunks, B.pairs, P.list, P.weight,
                       (uint8_t*)m->data, hits);
    hipLaunchKernelGGL(k_sensor_split, dim3(512), dim3(1024), 0, s, geom, P.st, B.split, dz, (uint8_t*)m->data, hits);
    GVX_HIP(hipGetLastError());
  } else if (enable_raycasting) {
    {
      ProfScope ps("sensor_rays");
      hipLaunchKernelGGL(k_sensor_rays, dim3(gp), dim3(256), 0, s, hits, dx, dy, dz, sx, sy, sz, P.list, P.weight, P.st);
      GVX_HIP(hipGetLastError());
    }
    {
      ProfScope ps("sensor_apply");
      hipLaunchKernelGGL(k_sensor_apply, dim3(grid_for((m->n + 3) / 4, 256, 1u << 16)), dim3(256), 0, s,
                         (uint8_t*)m->data, hits, m->n);
      GVX_HIP(hipGetLastError());
    }
  }
  {
    ProfScope ps("sensor_hits");
    hipLaunchKernelGGL(k_sensor_hits, dim3(grid_for(n, 256, 1u << 16)), dim3(256), 0, s, (uint8_t*)m->data, P.list,
                       P.weight, P.st);
    GVX_HIP(hipGetLastError());
  }
  GVX_CHECK(sync());
  sensor_hits_open = false;
  if (bricks) sensor_bricks_open = false;
  return GVX_OK;
}

int gvx_map_insert_coords(gvx_map m, const uint32_t* xyz, uint64_t n, uint32_t meaning, int mem, int* points_outside)
{
  GVX_CHECK(check_map(m));
  if (n && !xyz) return fail(GVX_ERR_BAD_ARG, "null coords");
  if (meaning > 255) return fail(GVX_ERR_BAD_ARG, "meaning > 255");
  std::lock_guard<std::recursive_mutex> g(m->mu);
  std::lock_guard<std::recursive_mutex> g2(rt().mu);
  const void* d = nullptr;
  GVX_CHECK(stage_input(xyz, n * 12, mem, &d));
  const OutsideFlag f = outside_flag();
  if (n) {
    unsigned gr = grid_for(n, 256, 1u << 16);
    hipStream_t s = rt().stream;
#define LAUNCH(T)                                                                                               \
  hipLaunchKernelGGL(k_insert_coords<T>, dim3(gr), dim3(256), 0, s, (uint8_t*)m->data, m->dims[0], m->dims[1], \
                     m->dims[2], (const uint32_t*)d, n, meaning, m->uninit, f)
    if (m->type == TBIT) LAUNCH(TBIT);
    else if (m->type == TPROB) LAUNCH(TPROB);
    else LAUNCH(TDIST);
#undef LAUNCH
    GVX_HIP(hipGetLastError());
  }
  return finish_outside(f, points_outside);
}

int gvx_map_insert_meta(gvx_map m, const float* xyz, const uint32_t* sizes, uint32_t ncl, const uint32_t* meanings,
                        uint32_t meaning, int mem, int* points_outside)
{
  GVX_CHECK(check_map(m));
  if (ncl == 0) {
    if (points_outside) *points_outside = 0;
    return GVX_OK;
  }
  if (!sizes) return fail(GVX_ERR_BAD_ARG, "null cloud sizes");
  std::vector<uint32_t> tab(2 * (size_t)ncl);
  uint64_t total = 0;
  for (uint32_t c = 0; c < ncl; ++c) {
    total += sizes[c];
    if (total > 0xFFFFFFFFull) return fail(GVX_ERR_UNSUPPORTED, "meta cloud larger than 2^32 points");
    tab[c] = (uint32_t)total;
    uint32_t mc = meanings ? meanings[c] : meaning;
    if (mc > 255) return fail(GVX_ERR_BAD_ARG, "meaning > 255");
    tab[ncl + c] = mc;
  }
  if (total && !xyz) return fail(GVX_ERR_BAD_ARG, "null points");
  std::lock_guard<std::recursive_mutex> g(m->mu);
  std::lock_guard<std::recursive_mutex> g2(rt().mu);
  // staging: [points | table]
  size_t pb = (total * 12 + 255) & ~(size_t)255;
  void* st = nullptr;
  GVX_CHECK(stage_reserve(pb + tab.size() * 4, &st));
  const float* dp = (const float*)xyz;
  if (mem == GVX_MEM_HOST) {
    GVX_HIP(hipMemcpyAsync(st, xyz, total * 12, hipMemcpyHostToDevice, rt().stream));
    dp = (const float*)st;
  }
  uint32_t* dtab = (uint32_t*)((char*)st + pb);
  GVX_HIP(hipMemcpyAsync(dtab, tab.data(), tab.size() * 4, hipMemcpyHostToDevice, rt().stream));
  const OutsideFlag f = outside_flag();
  GVX_CHECK(insert_points_async(m, dp, total, dtab, ncl, dtab + ncl, meaning, f));
  return finish_outside(f, points_outside);
}

int gvx_map_insert_meta_selfcoll(gvx_map m, const float* xyz, const uint32_t* cloud_sizes, uint32_t n_clouds,
                                 const uint32_t* meanings, const uint8_t* masks, int mem, uint8_t colliding[32],
                                 int* self_collision, int* points_outside)
{
  GVX_CHECK(check_map(m));
  if (n_clouds && !cloud_sizes) return fail(GVX_ERR_BAD_ARG, "null cloud sizes");
  uint64_t total = 0;
  for (uint32_t c = 0; c < n_clouds; ++c) total += cloud_sizes[c];
  if (total && !xyz) return fail(GVX_ERR_BAD_ARG, "null points");
  std::lock_guard<std::recursive_mutex> g(m->mu);
  std::lock_guard<std::recursive_mutex> g2(rt().mu);
  const void* d = nullptr;
  GVX_CHECK(stage_input(xyz, total * 12, mem, &d));
  uint32_t* acc = (uint32_t*)rt().dev_small + 64;
  GVX_CHECK(selfcoll_insert_async(m, (const float*)d, cloud_sizes, n_clouds, meanings, masks, acc));
  return selfcoll_finish(acc, colliding, self_collision, points_outside);
}

int gvx_map_collide(gvx_map self, gvx_map other, float threshold, const int32_t offset[3], uint64_t* count)
{
  GVX_CHECK(check_map(self));
  GVX_CHECK(check_map(other));
  if (!count) return fail(GVX_ERR_BAD_ARG, "null count");
  if (memcmp(self->dims, other->dims, sizeof(self->dims)) != 0)
    return fail(GVX_ERR_DIM_MISMATCH, "collideWith: map dimensions differ");
  if (self->type == TDIST || other->type == TDIST) {  // DefaultCollider: distance voxels never collide
    *count = 0;
    return GVX_OK;
  }
  std::unique_lock<std::recursive_mutex> g1(self->mu, std::defer_lock), g2(other->mu, std::defer_lock);
  if (self == other) g1.lock(); else std::lock(g1, g2);
  std::lock_guard<std::recursive_mutex> g3(rt().mu);
  const uint64_t n = self->n;
  int64_t off = 0;
  if (offset)
    off = (int64_t)offset[2] * (int64_t)self->dims[0] * (int64_t)self->dims[1] +
          (int64_t)offset[1] * (int64_t)self->dims[0] + (int64_t)offset[0];
  uint64_t lo = off < 0 ? (uint64_t)(-off) : 0, hi = off > 0 ? (off >= (int64_t)n ? 0 : n - (uint64_t)off) : n;
  if (lo > n) lo = n;
  const int thr = float_to_probability(threshold);
  if (hi <= lo) {
    *count = 0;
    return GVX_OK;
  }
  ResultDev res;
  GVX_CHECK(results_dev(&res));
  unsigned long long* dcount = res.count;
  {
    hipStream_t s = rt().stream;
    uint8_t* a = (uint8_t*)self->data;
    const uint8_t* b = (const uint8_t*)other->data;
    ProfScope ps("collide");
    const unsigned g16 = prob_grid((hi - lo + 15) / 16 + 1);
    if (self->type == TBIT && other->type == TBIT)
      hipLaunchKernelGGL(k_collide_bits, dim3(bits_grid(hi - lo)), dim3(256), 0, s, a, b, lo, hi, off, dcount);
    else if (self->type == TBIT && other->type == TPROB)
      hipLaunchKernelGGL((k_collide_prob<TBIT, TPROB, false>), dim3(g16), dim3(256), 0, s, a, b, lo, hi, off, thr,
                         dcount);
    else if (self->type == TPROB && other->type == TBIT)
      hipLaunchKernelGGL((k_collide_prob<TPROB, TBIT, true>), dim3(g16), dim3(256), 0, s, a, b, lo, hi, off, thr,
                         dcount);
    else
      hipLaunchKernelGGL((k_collide_prob<TPROB, TPROB, false>), dim3(g16), dim3(256), 0, s, a, b, lo, hi, off, thr,
                         dcount);
    GVX_HIP(hipGetLastError());
  }
  return results_fetch(count, nullptr);
}

int gvx_map_collide_types(gvx_map self, gvx_map other, float threshold, uint64_t* count, uint8_t mask[32])
{
  GVX_CHECK(check_map(self));
  GVX_CHECK(check_map(other));
  if (!count) return fail(GVX_ERR_BAD_ARG, "null count");
  if (self->type != TBIT) return fail(GVX_ERR_UNSUPPORTED, "collideWithTypes: self must be a BitVector map");
  if (other->type != TBIT && other->type != TPROB)
    return fail(GVX_ERR_UNSUPPORTED, "collideWithTypes: other must be a BitVector or Prob map");
  if (memcmp(self->dims, other->dims, sizeof(self->dims)) != 0)
    return fail(GVX_ERR_DIM_MISMATCH, "collideWithTypes: map dimensions differ");
  std::unique_lock<std::recursive_mutex> g1(self->mu, std::defer_lock), g2(other->mu, std::defer_lock);
  if (self == other) g1.lock(); else std::lock(g1, g2);
  std::lock_guard<std::recursive_mutex> g3(rt().mu);
  const int thr = sv_float_to_probability(threshold);
  ResultDev res;
  GVX_CHECK(results_dev(&res));
  {
    ProfScope ps("collide_types");
    if (other->type == TBIT)
      hipLaunchKernelGGL(k_collide_types, dim3(bits_grid(self->n)), dim3(256), 0, rt().stream, (uint8_t*)self->data,
                         (const uint8_t*)other->data, self->n, res.count, res.mask);
    else
      hipLaunchKernelGGL(k_collide_types_prob, dim3(prob_grid((self->n + 15) / 16)), dim3(256), 0, rt().stream,
                         (uint8_t*)self->data, (const uint8_t*)other->data, self->n, thr, res.count, res.mask);
    GVX_HIP(hipGetLastError());
  }
  return results_fetch(count, mask);
}

int gvx_map_collide_sv(gvx_map self, gvx_map other, float threshold, uint32_t window, uint32_t sv_offset,
                       uint64_t* count, uint8_t mask[32])
{
  GVX_CHECK(check_map(self));
  GVX_CHECK(check_map(other));
  if (!count) return fail(GVX_ERR_BAD_ARG, "null count");
  if (self->type != TBIT) return fail(GVX_ERR_UNSUPPORTED, "collisionCheckBitvector: self must be a BitVector map");
  if (other->type == TPROB) return gvx_map_collide_types(self, other, threshold, count, mask);  // window unused
  if (other->type != TBIT) return fail(GVX_ERR_UNSUPPORTED, "collisionCheckBitvector: other must be BitVector or Prob");
  if (window > 31 || sv_offset / 8 > 31 - window)
    return fail(GVX_ERR_BAD_ARG, "SV window must be <= 31 and sv_offset / 8 <= 31 - window");
  if (memcmp(self->dims, other->dims, sizeof(self->dims)) != 0)
    return fail(GVX_ERR_DIM_MISMATCH, "collisionCheckBitvector: map dimensions differ");
  std::unique_lock<std::recursive_mutex> g1(self->mu, std::defer_lock), g2(other->mu, std::defer_lock);
  if (self == other) g1.lock(); else std::lock(g1, g2);
  std::lock_guard<std::recursive_mutex> g3(rt().mu);
  ResultDev res;
  GVX_CHECK(results_dev(&res));
  {
    ProfScope ps("collide_sv");
    hipLaunchKernelGGL(k_collide_sv, dim3(stream_grid(self->n)), dim3(256), 0, rt().stream, (uint8_t*)self->data,
                       (const uint8_t*)other->data, self->n, window, sv_offset, res.count, res.mask);
    GVX_HIP(hipGetLastError());
  }
  return results_fetch(count, mask);
}

int gvx_map_shift_sv(gvx_map m, uint32_t shift)
{
  GVX_CHECK(check_map(m));
  if (m->type != TBIT) return fail(GVX_ERR_UNSUPPORTED, "shiftLeftSweptVolumeIDs needs a BitVector map");
  if (shift > 56) return fail(GVX_ERR_BAD_ARG, "Maximum shift size is 56");
  std::lock_guard<std::recursive_mutex> g(m->mu);
  ProfScope ps("shift_sv");
  GVX_CHECK(shift_sv_async((uint8_t*)m->data, m->n, shift));
  return sync();
}

}  // extern "C"
