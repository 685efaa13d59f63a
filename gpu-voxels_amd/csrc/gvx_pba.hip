// gvx_pba.hip -- DistanceVoxelMap: exact 3D EDT (PBA semantics), distance read-outs,
// mergeOccupied and the brute-force exactDistances3D.
//
// The EDT runs as three axis passes with no transposes of the map:
//   z pass  one thread per (x, y) column; the column's occupancy is held as a
//           register bitmask (all loads issued before any use), so each voxel is
//           read once and the nearest obstacle z (ties to the lower z) is written
//           as uint16.
//   y pass  on evenly filled x ranges a windowed search (k_pba_y_win): every voxel
//           takes the lowest key cost + k^2 within a radius that grows until the whole
//           wave has resolved, cut off where no result can need more, and stores its
//           site relative to itself in 2 bytes.  Other x ranges go to the
//           proximate-point stack kernel (k_pba_y: PBA phase 2 and phase 3 with
//           the stack's top entries in an LDS ring per line, spilled to a per-line
//           global array only when deeper), which writes packed DistanceVoxels.
//   x pass  a windowed search along x (k_pba_x_win), reading each slice's
//           y output in its format; rows it cannot resolve go to the stack kernel
//           (k_pba_x, 64 x 16 LDS tiles turning the per-lane walk into row loads,
//           final stacks to a global array) and the colouring kernel
//           (k_pba_x_colour: each position's owner as a prefix maximum of the
//           entries' first positions, whole row segments written).
// Small maps take one kernel each for y and x (k_pba_y_chunk, k_pba_x_chunk), which
// search outwards over chunks of a line whatever the field.
// All bisector tests compare whole numbers exactly.
#include "gvx_internal.hpp"

namespace gvx {

constexpr uint16_t ZNONE = 0xFFFF;

// ---------------------------------------------------------------- z pass
// Block = 64 columns (x range xr, row y; lanes = consecutive x) x W / ZWP waves; wave w
// takes the z range [32 ZWP w, 32 ZWP (w + 1)) of every column: its occupancy as ZWP
// register words (all loads issued before any is used).  The words of all waves meet in
// LDS, so each wave also knows the nearest obstacle below and above its range,
// and writes the nearest obstacle z (ties to the lower z) of its range as uint16.
// ZWP = 4 keeps 128 loads a lane in flight; small maps, whose few columns would leave
// most of the chip idle, take ZWP = 1 (four times the waves: 128^3 18 -> 7 us).
// FULL: dz == 32 * W, every load unconditional so the compiler keeps many in flight.
// flags (null: every column is stored and nothing is flagged):
// colm[(y / 32) * nxr + xr] gets bit y % 32 when the 64 columns of that row segment
// were stored (one of them holds an obstacle); the other segments are not stored.
// tflags[xr] gets bit y / tile_rows for every row holding an obstacle: the y pass skips
// (x range, row tile) blocks without one.  xcnt[xr] counts the obstacles of each x
// range and xcnt[16 + xr] its (row, 128 z) cells of 64 columns without one: few empty
// cells tell an evenly filled range from one whose obstacles sit on a few surfaces.
constexpr int ZCELL = 4;  // words (of 32 z) per cell
template <int W, bool FULL, int ZWP>
__global__ void __launch_bounds__(64 * (W / ZWP)) k_pba_z(const uint32_t* __restrict__ map,
                                                          uint16_t* __restrict__ zs, uint32_t* __restrict__ tflags,
                                                          uint32_t* __restrict__ colm, uint32_t* __restrict__ xcnt,
                                                          uint32_t tile_rows, uint32_t dx, uint32_t dy, uint32_t dz,
                                                          UDiv nxrd, uint32_t uninit)
{
  static_assert(W % ZWP == 0, "whole parts");
  __shared__ uint32_t sb[W][64];  // occupancy word w of the 64 columns
  const uint32_t lane = threadIdx.x & 63, part = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  uint32_t xr;
  const uint32_t cy = nxrd.div(blockIdx.x, xr), cx = xr * 64 + lane;
  const bool cin = cx < dx;
  const uint32_t col = cy * dx + (cin ? cx : dx - 1);  // dx dy <= 2^20: a lane offset from the layer's base
  const uint64_t layer = (uint64_t)dx * dy;
  uint32_t bits[ZWP];
#pragma unroll
  for (int i = 0; i < ZWP; ++i) {
    const int w = (int)part * ZWP + i;
    // layers past the map read the last one and are masked off, so that no load waits
    // behind a test (a test per load: 2.5 times the time on a 320^3 map)
    const uint32_t zn = FULL ? 32u : (uint32_t)(w * 32) < dz ? min(dz - (uint32_t)(w * 32), 32u) : 0u;  // uniform
    uint32_t word = 0;
    if (zn != 0u) {
      uint32_t v[32];
#pragma unroll
      for (int b = 0; b < 32; ++b)
        v[b] = (map + (uint64_t)((uint32_t)(w * 32) + (FULL ? (uint32_t)b : min((uint32_t)b, zn - 1u))) * layer)[col];
#pragma unroll
      for (int b = 0; b < 32; ++b) word |= (v[b] != uninit ? 1u : 0u) << b;
      if (zn < 32u) word &= (1u << zn) - 1u;
    }
    bits[i] = cin ? word : 0u;
    sb[w][lane] = bits[i];
  }
  __syncthreads();
  // nearest obstacle below this range (last set bit of the lower words) and above it
  // (first set bit of the higher words); 0xFFFF = none
  uint32_t last = 0xFFFFu, after = 0xFFFFu;
  for (int w = (int)part * ZWP - 1; w >= 0 && last == 0xFFFFu; --w) {
    const uint32_t m = sb[w][lane];
    if (m) last = (uint32_t)(w * 32 + 31 - __builtin_clz(m));
  }
  for (int w = ((int)part + 1) * ZWP; w < W && after == 0xFFFFu; ++w) {
    const uint32_t m = sb[w][lane];
    if (m) after = (uint32_t)(w * 32 + __builtin_ctz(m));
  }
  uint32_t any = last != 0xFFFFu || after != 0xFFFFu ? 1u : 0u;
#pragma unroll
  for (int i = 0; i < ZWP; ++i) any |= bits[i];
  // when none of the 64 columns holds an obstacle nothing is stored (the segment's bit
  // in colm stays clear and the y pass never reads it); with one, all 64 are, so stores
  // stay whole rows
  const bool wave_any = wave_ballot(any != 0u) != 0ull;
  if (cin && (!tflags || wave_any)) {
#pragma unroll
    for (int i = 0; i < ZWP; ++i) {
      const int w = (int)part * ZWP + i;
      // first set position in the words after this one (in this range, else above it)
      uint32_t nxt = after;
#pragma unroll
      for (int v = ZWP - 1; v > i; --v) nxt = bits[v] ? (uint32_t)(((int)part * ZWP + v) * 32 + __builtin_ctz(bits[v])) : nxt;
#pragma unroll
      for (int b = 0; b < 32; ++b) {
        const uint32_t z = (uint32_t)(w * 32 + b);
        if (FULL || z < dz) {
          if ((bits[i] >> b) & 1u) last = z;
          const uint32_t m = bits[i] & (0xFFFFFFFFu << b);
          const uint32_t hi = m ? (uint32_t)(w * 32 + __builtin_ctz(m)) : nxt;
          uint32_t pick;
          if (last == 0xFFFFu) pick = hi;
          else if (hi == 0xFFFFu) pick = last;
          else pick = (z - last <= hi - z) ? last : hi;
          (zs + (uint64_t)z * layer)[col] = (uint16_t)pick;
        }
      }
    }
  }
  if (part != 0 || !tflags) return;
  uint32_t nob = 0, empty = 0;
  for (int c = 0; c < W / ZCELL; ++c) {
    uint32_t m = 0;
    for (int i = 0; i < ZCELL; ++i) {
      const uint32_t v = sb[c * ZCELL + i][lane];
      nob += (uint32_t)__popc(v);
      m |= v;
    }
    if ((uint32_t)(c * ZCELL * 32) < dz && wave_ballot(m != 0u) == 0ull) ++empty;
  }
  // the block's 64 columns share one flag bit and one segment bit: one atomic each
  for (int o = 32; o > 0; o >>= 1) nob += (uint32_t)__shfl_xor((int)nob, o, 64);
  if (lane == 0) {
    if (wave_any) {
      atomicOr(tflags + xr, 1u << (cy / tile_rows));
      atomicOr(colm + (uint64_t)(cy >> 5) * nxrd.d + xr, 1u << (cy & 31));
      atomicAdd(xcnt + xr, nob);
    }
    if (empty) atomicAdd(xcnt + 16 + xr, empty);
  }
}

// columns longer than 1024: two sweeps through the uint16 buffer
__global__ void __launch_bounds__(256) k_pba_z_long(const uint32_t* __restrict__ map, uint16_t* __restrict__ zs,
                                                    uint32_t dx, uint32_t dy, uint32_t dz, uint32_t uninit)
{
  const uint64_t col = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= (uint64_t)dx * dy) return;
  const uint64_t layer = (uint64_t)dx * dy;
  uint32_t last = 0xFFFFu;
  for (uint32_t z = 0; z < dz; ++z) {
    if (map[z * layer + col] != uninit) last = z;
    zs[z * layer + col] = (uint16_t)last;
  }
  uint32_t next = 0xFFFFu;
  for (int64_t zz = (int64_t)dz - 1; zz >= 0; --zz) {
    const uint32_t z = (uint32_t)zz;
    if (map[z * layer + col] != uninit) next = z;
    const uint32_t lo = zs[z * layer + col];
    uint32_t pick;
    if (lo == 0xFFFFu) pick = next;
    else if (next == 0xFFFFu) pick = lo;
    else pick = (z - lo <= next - z) ? lo : next;
    zs[z * layer + col] = (uint16_t)pick;
  }
}

// ---------------------------------------------------------------- y and x passes
// One wave per block handles 64 lines (lanes = lines) and runs PBA's phase 2
// (proximate-point stack) and phase 3 (colouring, from the top of the line down).
// The stack of a line lives in an LDS ring of its RK topmost entries; entries
// pushed deeper spill to a per-line global array (stk[line * n + depth]) and come
// back RK - 1 at a time in one batch of independent loads when a pop reaches
// below the ring.  Short stacks therefore never touch global memory.  The input
// is staged through LDS tiles so global loads and stores are row-contiguous, and
// each lane walks only the positions of a tile that hold a site (a bit mask), so
// empty stretches of a line cost nothing.
//
// Bisector tests are exact.  For sites a < b on the line (positions pa, pb; squared
// off-line costs ca, cb), a is at least as close as b at position p exactly when
// 2 p D <= N with N = (pb^2 - pa^2) + cb - ca and D = pb - pa > 0; phase 2's comparison
// is N_ab * D_bc >= N_bc * D_ab (pop b, also on equality).  Positions are below 1024 and
// z below 4094, so costs reach 1023^2 + 4093^2 > 2^24: the numbers are floats where a
// whole diagonal stays below 2^24 (any map of up to 3832 layers) and integers beyond
// (bis_floats).
#ifndef GVX_PBA_TYR
#define GVX_PBA_TYR 32
#endif
#ifndef GVX_PBA_TX
#define GVX_PBA_TX 16
#endif
#ifndef GVX_PBA_RK
#define GVX_PBA_RK 16
#endif
constexpr int TB = 64;            // lines per wave
constexpr int TYR = GVX_PBA_TYR;  // y pass: positions per input tile
constexpr int TX = GVX_PBA_TX;    // x pass: positions per tile (4 TX-byte row segments)
constexpr int RK = GVX_PBA_RK;    // stack entries per line held in LDS
static_assert(RK >= 4 && (RK & (RK - 1)) == 0 && TX >= 4 && 64 % TX == 0 && TYR <= 32, "tile shape");

__device__ __forceinline__ void wave_lds_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ int32_t sq24(int32_t v) { return __mul24(v, v); }

// raw buffer loads over one z slice of a map or of the z-pass output (below
// 4 GiB): a per-lane byte offset plus a wave-uniform byte offset, so the tile
// loads need no per-load vector address arithmetic
__device__ __forceinline__ __amdgpu_buffer_rsrc_t slice_rsrc(const void* base, uint32_t bytes)
{
  const uint64_t b = reinterpret_cast<uint64_t>(base);  // the same for the whole wave: keep it scalar
  const uint64_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
  const uint64_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(hi << 32 | lo), (short)0,
                                           __builtin_amdgcn_readfirstlane((int)bytes), 0x00020000);
}

// Do costs, and with a line's squared positions every N, stay below 2^24?  Then they are
// floats (T of the kernels below), else integers.
static inline bool bis_floats(uint32_t dx, uint32_t dy, uint32_t dz)
{
  return (uint64_t)(dx - 1) * (dx - 1) + (uint64_t)(dy - 1) * (dy - 1) + (uint64_t)(dz - 1) * (dz - 1) < (1u << 24);
}
// bisector of sites a < b: a is at least as close as b at p  <=>  2 p D <= N
template <typename T>
struct Bis;
// whole numbers below 2^24 in floats, each step exact
template <>
struct Bis<float> {
  float N = 0.f, D = 1.f;
  __device__ __forceinline__ void set(float pa, float ca, float pb, float cb)
  {
    D = pb - pa;
    N = fmaf(D, pb + pa, cb - ca);
  }
  __device__ __forceinline__ bool a_wins(float p) const { return 2.0f * p * D <= N; }
};
// N below 2^25
template <>
struct Bis<int32_t> {
  int32_t N = 0, D = 1;
  __device__ __forceinline__ void set(int32_t pa, int32_t ca, int32_t pb, int32_t cb)
  {
    D = pb - pa;
    N = __mul24(D, pb + pa) + (cb - ca);
  }
  __device__ __forceinline__ bool a_wins(int32_t p) const { return 2 * __mul24(p, D) <= N; }
};
// b (the middle of a < b < c) owns no position: bisector(a, b) >= bisector(b, c), N_ab D_bc >=
// N_bc D_ab.  With p the rounded right side, its error is a whole number below 2^9 and a
// float, and the left side less p is a whole number that rounds only above 2^24: the two
// compare as the products do.  (In double precision the stack kernels of a 512^3 room took
// 313 and 112 us, this way 309 and 106: the chain of a line and its LDS round trips are longer.)
__device__ __forceinline__ bool middle_empty(const Bis<float>& ab, const Bis<float>& bc)
{
  const float p = bc.N * ab.D;
  return fmaf(ab.N, bc.D, -p) >= fmaf(bc.N, ab.D, -p);
}
__device__ __forceinline__ bool middle_empty(const Bis<int32_t>& ab, const Bis<int32_t>& bc)
{
  return (double)ab.N * (double)bc.D >= (double)bc.N * (double)ab.D;  // products below 2^35
}

// Per-lane stack of 32-bit entries: ring[depth % RK][lane] holds depths [lo, n);
// depths below lo are in g[0 .. lo).  The caller also keeps the top three
// entries in registers, so the only fetch is that of the new third entry after
// a pop.
struct LineStack {
  uint32_t (*ring)[TB];
  uint32_t* g;
  uint32_t lane, n, lo;

  __device__ __forceinline__ void push(uint32_t e)
  {
    if (n - lo == (uint32_t)RK) {  // ring full: the slot of depth n holds depth lo
      g[lo] = ring[lo % RK][lane];
      ++lo;
    }
    ring[n % RK][lane] = e;
    ++n;
  }
  __device__ __forceinline__ void pop() { --n; }  // lo <= n - 2 before a pop (see at3)
  // entry at depth d = n - 3 (any d <= n - 3 is harmless when n < 3: then
  // lo == 0 and nothing is reloaded): the caller keeps the top two entries in
  // registers and this third one too, fetching it right after a pop so the LDS
  // read is in flight while the next test runs.  Below the ring, depths
  // d+3-RK .. d come back in one batch of independent loads; the slots of
  // depths n - 2 and n - 1 are left alone (the ring always holds them: refills
  // happen as soon as d < lo, which keeps lo <= max(n - 2, 0)).
  __device__ __forceinline__ uint32_t at3(uint32_t d)
  {
    if (d < lo) {
      uint32_t v[RK - 2];  // all loads first, so they are in flight together
#pragma unroll
      for (int j = 0; j < RK - 2; ++j) v[j] = g[(uint32_t)j <= d ? d - (uint32_t)j : d];
#pragma unroll
      for (int j = 0; j < RK - 2; ++j) ring[((uint32_t)j <= d ? d - (uint32_t)j : d) % RK][lane] = v[j];
      lo = d + 3 >= (uint32_t)RK ? d + 3 - RK : 0;
    }
    return ring[d % RK][lane];
  }
};


// y pass: lines (x, z), lanes = consecutive x.  Stack entry = y | z_site << 10.
// Every lane touches only its own LDS columns, so no barriers are needed.
// Output: the packed DistanceVoxel (x, y_site, z_site) written into the map.
// Row tiles whose 64 x 32 block of columns holds no obstacle (tflags, from the z
// pass) are neither loaded nor walked: they hold no site.  xflags[z] gets bit
// x / TX for every line (x, z) left with a site, for the x pass.
template <typename T>
__global__ void __launch_bounds__(TB) k_pba_y(const uint16_t* __restrict__ zs, uint32_t* __restrict__ out,
                                              uint32_t* __restrict__ stk, const uint32_t* __restrict__ tflags,
                                              const uint32_t* __restrict__ colm,
                                              unsigned long long* __restrict__ xflags,
                                              uint32_t* __restrict__ yfs, uint32_t dx, uint32_t dy,
                                              uint32_t dz, uint32_t uninit, bool redo)
{
  static_assert(TYR == 32, "one column-mask word per row tile");
  __shared__ uint16_t ztile[TYR][TB];
  __shared__ uint32_t ring[RK][TB];
  const uint32_t ngroups = (dx + TB - 1) / TB * dz;
  if (!redo && blockIdx.x < dz) {
    // the format of slice z's y output for the x pass (yfs[dz + ngroups + z]): 0 =
    // relative sites, 1 = packed (each of its groups is done here), 2 = both
    const uint32_t zz = blockIdx.x, nxr = (dx + TB - 1) / TB, l = threadIdx.x;
    const uint64_t fm = wave_ballot(l < nxr && yfs[dz + l * dz + zz] != 0u);
    const uint64_t allc = nxr >= 64 ? ~0ull : (1ull << nxr) - 1ull;
    if (l == 0) yfs[dz + ngroups + zz] = fm == allc ? 1u : fm == 0ull ? 0u : 2u;
  }
  // first run: the groups that the window left to this kernel; second run (redo): the
  // others of slices whose cut-off window outputs the x pass could not use (yfs[z])
  const bool own = yfs[dz + blockIdx.x] != 0u;
  if (redo ? own || yfs[blockIdx.x % dz] == 0u : !own) return;
  // consecutive blocks take consecutive z with the same x range: workgroups are
  // dealt round-robin over the XCDs, so every XCD gets every x range (obstacles
  // clustered in a few x ranges would otherwise load a few XCDs only)
  const uint32_t z = blockIdx.x % dz, x0 = (blockIdx.x / dz) * TB;
  const uint32_t lane = threadIdx.x, x = x0 + lane;
  if (x >= dx) return;
  const int32_t zi = (int32_t)z;
  LineStack st{ring, stk + ((uint64_t)z * dx + x) * dy, lane, 0, 0};
  // top, second and third of the stack (entries; positions and costs of the first two);
  // bst = bisector(second, top)
  T ty = 0, tc = 0, sy = 0, sc = 0;
  uint32_t te = 0, se = 0, e3 = 0;
  Bis<T> bst;
  auto cost = [&](int32_t s) -> T { const T d = (T)(s - zi); return d * d; };
  // pop the top: second and third move up, the new third is fetched (when fewer
  // than two entries remain the moved values are never read)
  auto pop_y = [&]() {
    st.pop();
    ty = sy;
    tc = sc;
    te = se;
    se = e3;
    sy = (T)(e3 & 0x3FFu);
    sc = cost((int32_t)(e3 >> 10));
    bst.set(sy, sc, ty, tc);
    e3 = st.at3(st.n >= 3 ? st.n - 3 : 0);
  };
  // software pipeline: the next tile's values are loaded into registers (rows
  // clamped into the line) while the current tile is processed
  const __amdgpu_buffer_rsrc_t zr = slice_rsrc(zs + (uint64_t)z * dx * dy, dx * dy * 2);
  auto zload = [&](uint32_t yr) -> uint32_t {  // row yr of this lane's line, yr < dy
    return __builtin_amdgcn_raw_buffer_load_b16(zr, (int)(x * 2), (int)(yr * dx * 2), 0);
  };
  // row tiles with an obstacle column in this x range, in increasing y
  const uint32_t ntiles = (dy + TYR - 1) / TYR;
  uint32_t todo = tflags[x0 / 64] & (ntiles >= 32 ? 0xFFFFFFFFu : (1u << ntiles) - 1u);
  uint32_t pre[TYR], pre_cm = 0;
  auto load_rows = [&](uint32_t t) {  // past the end of the line: harmless reloads of the last row
    // rows of this tile whose 64-column segment was stored (TYR == 32)
    pre_cm = colm[(uint64_t)t * ((dx + 63) / 64) + x0 / 64];
#pragma unroll
    for (int r = 0; r < TYR; ++r) {
      const uint32_t yr = t * TYR + r;
      pre[r] = zload(yr < dy ? yr : dy - 1);
    }
  };
  if (todo) load_rows((uint32_t)__builtin_ctz(todo));
  while (todo) {
    const uint32_t t = (uint32_t)__builtin_ctz(todo);
    todo &= todo - 1u;
    const uint32_t y0 = t * TYR;
    const uint32_t rows = dy - y0 < (uint32_t)TYR ? dy - y0 : (uint32_t)TYR;
    const uint32_t cm = pre_cm;
    uint32_t m = 0;  // positions of this tile that hold a site
#pragma unroll
    for (int r = 0; r < TYR; ++r) {
      ztile[r][lane] = (uint16_t)pre[r];
      m |= (pre[r] != ZNONE ? 1u : 0u) << r;
    }
    m &= cm;  // a segment without an obstacle was not stored (its values are stale)
    if (rows < (uint32_t)TYR) m &= (1u << rows) - 1u;
    load_rows(todo ? (uint32_t)__builtin_ctz(todo) : t);  // the next tile (the last one reloads itself)
    // the next site's value is read from LDS while the current one is processed
    uint32_t r = m ? (uint32_t)__builtin_ctz(m) : 0u;
    int32_t s = ztile[r][lane];
    while (m) {
      m &= m - 1u;
      const uint32_t rn = m ? (uint32_t)__builtin_ctz(m) : r;
      const int32_t sn = ztile[rn][lane];
      const T y = (T)(y0 + r), c = cost(s);
      if (st.n >= 1) {
        Bis<T> btn;
        btn.set(ty, tc, y, c);
        while (st.n >= 2 && middle_empty(bst, btn)) {
          pop_y();
          btn.set(ty, tc, y, c);
        }
        bst = btn;
      }
      e3 = se;
      se = te;
      te = (y0 + r) | ((uint32_t)s << 10);
      st.push(te);
      sy = ty;
      sc = tc;
      ty = y;
      tc = c;
      r = rn;
      s = sn;
    }
  }
  // x tiles (TX lines each) of this slice that keep a site
  const uint64_t kept = wave_ballot(st.n > 0);
  {
    unsigned long long f = 0;
#pragma unroll
    for (int k = 0; k < TB / TX; ++k)
      if ((kept >> (k * TX)) & ((1ull << TX) - 1ull)) f |= 1ull << (x0 / TX + k);
    if (lane == 0 && f) atomicOr(xflags + z, f);
  }
  // a line whose x tile kept no site is never read again: the x pass skips the tile
  // and the colouring writes every voxel of every row, so its rows are not stored
  // (in a second run the window has announced every tile)
  if (!redo && ((kept >> ((lane / TX) * TX)) & ((1ull << TX) - 1ull)) == 0) return;
  // output rows through a descriptor over this z slice: lane offset x, row offset uniform
  const __amdgpu_buffer_rsrc_t orr = slice_rsrc(out + (uint64_t)z * dx * dy, dx * dy * 4);
  if (st.n == 0) {
    for (uint32_t y = 0; y < dy; ++y) __builtin_amdgcn_raw_buffer_store_b32(uninit, orr, (int)(x * 4), (int)(y * dx * 4), 0);
    return;
  }
  for (int32_t yy = (int32_t)dy - 1; yy >= 0; --yy) {
    while (st.n >= 2 && bst.a_wins((T)yy)) {
      pop_y();
    }
    __builtin_amdgcn_raw_buffer_store_b32(x | te << 10, orr, (int)(x * 4),
                                          (int)((uint32_t)yy * dx * 4), 0);
  }
}

// ---------------------------------------------------------------- windowed passes
// The three passes give every voxel its nearest obstacle with ties broken to the
// lowest coordinate along the pass's axis (z flood: lower z; the proximate-point
// stack pops on equality and colours ties to the lower entry), so the result is
// the nearest obstacle with ties to the lexicographically smallest (x, y, z).
//
// On fields where every voxel has a site within a few voxels, a search of the
// window |q - p| <= k finds a position's winner directly: every site outside the
// window costs more than k^2, so once the window's minimum is below (k + 1)^2
// nothing farther can reach or tie it.  Each site carries one 32-bit key,
//   cost << SH | position << (SH - 10) | payload,
// so the window minimum of key + (k^2 << SH) is the lowest minimum cost and,
// among equal costs, the lowest position (the tie rule) in one v_min3 per step;
// the payload rides along (positions are unique).  The x pass uses SH = 11 (a
// 20-bit cost, no payload), the y pass SH = 20 (an 11-bit cost and the site's z
// as payload, so the winner's key is its site).  Costs saturate at the field's
// maximum: a winner costs less than (WIN_R + 1)^2 = 1089, so a saturated site
// never resolves a voxel.  Lanes take consecutive
// positions of a line held in LDS and grow the radius together, one ds_read2 and
// one min3 per step, until every lane has resolved (or the radius reaches
// WIN_R).  An x-pass group with a voxel that does not resolve is flagged, and
// the proximate-point kernels redo it.  The output is the same either way.
constexpr int WIN_R = 32;                    // largest window radius
constexpr uint32_t KEY_NONE = 0x7FFFFFFFu;   // no site: at or above every real key, below 2^31
constexpr int WIN_CHECK = 4;                 // radius steps between the wave's all-resolved tests

// x-pass key (SH = 11): costs from 2^20 - 1 up saturate, so the key stays below 2^31
__device__ __forceinline__ uint32_t site_key(uint32_t cost, uint32_t pos)
{
  return ((cost < 0xFFFFFu ? cost : 0xFFFFFu) << 11) | (pos << 1);  // pos < 1024
}

// minimum over |q - p| <= k of kp[R + q - p] + ((q - p)^2 << SH), k growing until
// every active lane of the wave has resolved (its minimum cost below (k + 1)^2) or
// k = kmax (<= WIN_R); kp points at position p - WIN_R of a key array with kmax valid
// or KEY_NONE entries on each side.  ok: resolved.
template <int SH>
__device__ __forceinline__ uint32_t win_search(const uint32_t* kp, bool active, bool& ok, int kmax = WIN_R)
{
  // keys are below 2^31, so they compare the same as int32.  b = (minimum so far) -
  // (k^2 << SH): going from radius k - 1 to k subtracts (2k - 1) << SH and takes the
  // min with the two new keys, one subtract and one v_min3 per step (b stays above
  // -(WIN_R^2 << SH) >= -2^30).  A lane is resolved at radius k once its minimum is
  // below k^2 << SH, i.e. b < (2k - 1) << SH (it stays so as k grows); an inactive
  // lane starts resolved (key 0).
  const int32_t* ip = reinterpret_cast<const int32_t*>(kp);
  int32_t b = ip[WIN_R];  // kp is a valid address for every lane
  b = active ? b : 0;
  int k = 1;
#pragma unroll
  for (; k <= WIN_R; ++k) {
    // kmax: a multiple of WIN_CHECK
    if (k % WIN_CHECK == 1 && (k > kmax || __builtin_amdgcn_ballot_w64(b >= ((2 * k - 1) << SH)) == 0)) break;
    b = min(min(b - ((2 * k - 1) << SH), ip[WIN_R - k]), ip[WIN_R + k]);
  }
  // radius k - 1 was the last step; unsigned: with SH = 20 a saturated minimum plus k^2 passes 2^31
  const uint32_t best = (uint32_t)b + ((uint32_t)((k - 1) * (k - 1)) << SH);
  ok = best < ((uint32_t)((kmax + 1) * (kmax + 1)) << SH);
  return best;
}

// Growing windows of YG neighbouring outputs per lane: output i sits at row r0 + i of a
// column of keys (read(r): the key at row r, KEY_NONE outside the line) and starts with
// b[i] = its own key, or 0 when it is not wanted.  Step k looks at the rows r0 + i - k
// and r0 + i + k of every output; neighbouring outputs share all but one of them per
// side, so the two rows of YG keys live in registers that shift by one per step (the
// loop is unrolled by YG, so every register index is static) and a step costs two LDS
// reads, not 2 YG, beside its subtraction and v_min3 per output (see win_search for
// the relative minima).  Returns the radius K reached: kmax (a multiple of WIN_CHECK,
// at least the value passed) or the first multiple of WIN_CHECK at which the whole wave
// has resolved; output i is exact when b[i] + (K^2 << SH) < (K + 1)^2 << SH.
// One output at a time reads 2 keys per v_min3 and tests the wave's radius per output:
// the y window took 281 us at 512^3 with 1 % obstacles, this way 225 us (VALU bound).
constexpr int YG = 8;
template <int SH, typename Read>
__device__ __forceinline__ int grow_windows(Read&& read, int r0, int kmax, int32_t (&b)[YG])
{
  int32_t t[YG], u[YG];
#pragma unroll
  for (int i = 0; i < YG; ++i) t[i] = u[i] = (int32_t)read(r0 + i);
  for (int k = 0;; k += YG) {
#pragma unroll
    for (int s = 1; s <= YG; ++s) {
      t[(YG - s) % YG] = (int32_t)read(r0 - (k + s));          // output 0's row, the others' move on
      u[(YG - 1 + s) % YG] = (int32_t)read(r0 + YG - 1 + k + s);  // output YG - 1's
      const int32_t w = (2 * (k + s) - 1) << SH;
#pragma unroll
      for (int i = 0; i < YG; ++i) b[i] = min(min(b[i] - w, t[(i - s + YG) % YG]), u[(i + s) % YG]);
      if (s % WIN_CHECK == 0) {
        if (k + s >= kmax) return k + s;
        int32_t m = b[0];
#pragma unroll
        for (int i = 1; i < YG; ++i) m = max(m, b[i]);
        if (wave_ballot(m >= ((2 * (k + s) + 1) << SH)) == 0ull) return k + s;
      }
    }
  }
}
static_assert(YG % WIN_CHECK == 0, "the radius is tested inside the unrolled steps");

// y pass, windowed: a block takes 64 lines x0 .. x0+63 at one z and YBR output rows.
// The z-pass rows y0 - R .. y0 + YBR - 1 + R of the 64 columns are loaded with coalesced
// row loads into LDS keys (row-major: lane l reads line l's, one bank each); each wave
// searches YBR / YW_WAVES rows, YG at a time, with lanes = the 64 lines, so its winners,
// whose keys hold their sites, are whole rows and are stored directly.
//
// The window is cut off at a radius R that holds for the distances of the final result,
// not of this pass: a voxel at distance d from its nearest obstacle o takes it in the x
// pass from position (o.x, y, z), where o is at most d away in the (y, z) plane.  So a
// position with no site within R is marked (YREL_FAR: a cost above every window's) and
// the x pass checks that its winners cost less than (R + 1)^2; then no marked position,
// whose true cost is at least that, could have won or tied.  With obstacles spread
// evenly at density rho, P(no obstacle within r) = exp(-4/3 pi r^3 rho), an eighth of
// that ball in a corner of the map: R + 1 = 2.78 rho^(-1/3) (R = 12 at 1 %, 28 at 0.1 %,
// in steps of WIN_CHECK) leaves about 1 map of 512^3 in 1000 with a corner voxel beyond
// it and 10^-10 of the others.  (The whole-plane radius this pass would need is 2.5
// rho^(-1/2): 28 at 1 %, 79 at 0.1 %.)  A z slice holding marked positions that the x
// pass could not do with is redone by the stack kernel.
//
// x ranges that are not evenly filled, judged by their density (below 1/2048, where R
// would pass WIN_R) and by their share of empty 64 x 128 cells against the
// exp(-cell rho) of an even spread, go to the stack kernel at once.
// Blocks are dealt to the XCDs so that the blocks of one (x range, z) group run one
// after another on one XCD, where the overlapping halo rows are still in its L2.
constexpr int YBR = 128;               // output rows per block
constexpr int YNR = YBR + 2 * WIN_R;   // rows staged per block, at most
constexpr int YW_WAVES = 8;
constexpr uint32_t YREL_FAR = 0x3FFFu;  // relative site (63, 63): costs 7938
static_assert(YBR % (YW_WAVES * YG) == 0, "whole groups per wave");

// The windowed y pass writes each voxel's site relative to the voxel, 2 bytes:
// (y_site - y + 64) | (z_site - z + 64) << 7.  A window winner lies within WIN_R rows and
// at a cost below (WIN_R + 1)^2, so both offsets lie in [-WIN_R, WIN_R].  The stack
// kernel writes packed DistanceVoxels to the 4-byte buffer; the x pass reads a slice's
// rows in its one format, or leaves rows whose slice has both to the x stack kernels.
static_assert(WIN_R < 63, "relative sites hold offsets in [-64, 63], the last for YREL_FAR");
// For a window winner (key low bits y_site << 10 | z_site) neither field
// wraps, so the relative site is a sum: c = yrel_base(y, z)
__device__ __forceinline__ uint32_t yrel_base(uint32_t y, uint32_t z) { return (64u - y) + ((64u - z) << 7); }
__device__ __forceinline__ uint32_t yrel_win(uint32_t key, uint32_t c)
{
  return ((key >> 10) & 1023u) + ((key & 1023u) << 7) + c;
}
// the packed DistanceVoxel (x, y_site, z_site) of a relative site at (x, y, z)
__device__ __forceinline__ uint32_t yrel_site(uint32_t rel, uint32_t x, uint32_t y, uint32_t z)
{
  return x | ((y + (rel & 127u) - 64u) << 10) | ((z + (rel >> 7) - 64u) << 20);
}

// one block's rows with window radius R (a multiple of WIN_CHECK); returns whether this
// wave marked a position
template <int R>
__device__ __forceinline__ bool ywin_block(int32_t* kt, const uint16_t* __restrict__ zsl,
                                           const uint32_t* __restrict__ colm, const __amdgpu_buffer_rsrc_t orr,
                                           uint32_t x0, uint32_t y0, uint32_t z, uint32_t dx, uint32_t dy,
                                           uint32_t nxr, uint32_t lane, uint32_t w)
{
  constexpr int NR = YBR + 2 * R, RPW = NR / YW_WAVES;
  static_assert(NR % YW_WAVES == 0 && RPW <= 32 && R <= WIN_R && R % WIN_CHECK == 0, "whole rows per wave");
  const uint32_t x = x0 + lane, xl = x < dx ? x : dx - 1;
  const bool xin = x < dx;
  const int xoff = xin ? (int)(x * 2) : 0x7FFFFFF0;
  const int32_t ybase = (int32_t)y0 - R + (int32_t)w;
  // lane i looks up whether the wave's row i is inside the map and its 64-column segment
  // was stored: one load for all rows (a scalar load per row waits for each in turn)
  const int32_t yl = ybase + YW_WAVES * (int32_t)lane;
  uint32_t seg = 0;
  if (lane < (uint32_t)RPW && yl >= 0 && yl < (int32_t)dy) seg = colm[(uint32_t)(yl >> 5) * nxr + x0 / 64] >> (yl & 31);
  uint32_t v[RPW];
  // rows outside the map read a row inside it (their keys are KEY_NONE)
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    const int32_t yc = min(max(ybase + YW_WAVES * i, 0), (int32_t)dy - 1);
    v[i] = (zsl + (size_t)((uint32_t)yc * dx))[xl];  // uniform row, 32-bit lane offset
  }
  const uint32_t rows = (uint32_t)wave_ballot((seg & 1u) != 0u);
  const int32_t zc = (int32_t)(z & 1023u);  // z < 1024: tells the compiler dz fits a 24-bit product
#pragma unroll
  for (int i = 0; i < RPW; ++i) {
    const int32_t y = ybase + YW_WAVES * i;
    // key (SH = 20): min((z_site - z)^2, 2047) << 20 | y << 10 | z_site.  A column
    // without a site (ZNONE) costs 2047, above every cost that a window resolves.
    const int32_t dzv = (int32_t)v[i] - zc;
    const uint32_t c = min((uint32_t)__mul24(dzv, dzv), 2047u);
    const uint32_t key = (c << 20) | (((uint32_t)y << 10) & 0xFFC00u) | v[i];
    kt[(w + YW_WAVES * i) * TB + lane] = (int32_t)(key | ((rows >> i) & 1u ? 0u : KEY_NONE));
  }
  __syncthreads();
  bool cut = false;
#pragma unroll 1
  for (uint32_t g = 0; g < (uint32_t)(YBR / (YW_WAVES * YG)); ++g) {
    const uint32_t j = (g * YW_WAVES + w) * YG, yw = y0 + j;  // output rows yw .. yw + YG - 1
    if (yw >= dy) break;
    const int32_t* kl = kt + lane;
    int32_t b[YG];
#pragma unroll
    for (int i = 0; i < YG; ++i) {
      b[i] = kl[(R + j + i) * TB];
      if (!xin || yw + (uint32_t)i >= dy) b[i] = 0;
    }
    const int k = grow_windows<20>([&](int r) { return kl[r * TB]; }, R + (int)j, R, b);
    const uint32_t lim = (uint32_t)((k + 1) * (k + 1)) << 20, add = (uint32_t)(k * k) << 20;
    const uint32_t c = yrel_base(yw, z);
    // lanes and rows outside the map count as exact; the lanes' offset is beyond the
    // buffer, so nothing is stored for them
#pragma unroll
    for (int i = 0; i < YG; ++i) {
      const uint32_t res = (uint32_t)b[i] + add;
      const bool ok = res < lim;
      cut = cut || !ok;
      if (yw + (uint32_t)i < dy)  // uniform
        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(ok ? yrel_win(res, c - (uint32_t)i) : YREL_FAR), orr, xoff,
                                              (int)((yw + (uint32_t)i) * dx * 2), 0);
    }
  }
  return wave_ballot(cut) != 0ull;
}

__global__ void __launch_bounds__(TB * YW_WAVES, 6) k_pba_y_win(const uint16_t* __restrict__ zs,
                                                             uint16_t* __restrict__ out,
                                                             const uint32_t* __restrict__ tflags,
                                                             const uint32_t* __restrict__ colm,
                                                             unsigned long long* __restrict__ xflags,
                                                             uint32_t* __restrict__ yfs, uint32_t* __restrict__ ycut,
                                                             uint32_t* __restrict__ xcnt, uint32_t dx,
                                                             uint32_t dy, UDiv dzd, UDiv nybd, uint32_t ngroups)
{
  __shared__ int32_t kt[YNR * TB];
  const uint32_t xcd = blockIdx.x % 8, seq = blockIdx.x / 8;
  uint32_t jb, z;
  const uint32_t g = nybd.div(seq, jb) * 8 + xcd;
  if (g >= ngroups) return;  // uniform over the block
  const uint32_t dz = dzd.d, xr = dzd.div(g, z), x0 = xr * TB, y0 = jb * YBR;  // g = the stack kernel's block index
  const uint32_t lane = threadIdx.x % TB, w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / TB));
  const uint32_t ntl = (dy + TYR - 1) / TYR, nxr = (dx + TB - 1) / TB;
  const uint32_t tf = tflags[xr] & (ntl >= 32 ? 0xFFFFFFFFu : (1u << ntl) - 1u);
  if (tf == 0) return;  // no obstacle in these columns: no line keeps a site, nothing is read later
  // density and evenness of the x range (in float: they only pick the path)
  const float ncol = (float)(dx - x0 < (uint32_t)TB ? dx - x0 : (uint32_t)TB), nob = (float)xcnt[xr];
  const float rho = nob / (ncol * (float)dy * (float)dz);
  const uint32_t cz = 32 * ZCELL;
  const float cells = (float)dy * (float)((dz + cz - 1) / cz), zdepth = (float)(dz < cz ? dz : cz);
  const float even = __builtin_amdgcn_exp2f(-1.4427f * rho * ncol * zdepth);
  const float tail = dz > cz && dz % cz ? (float)dy : 0.0f;  // the last cells are shorter
  const bool sparse = rho * 2048.0f < 1.0f || (float)xcnt[16 + xr] > cells * fminf(1.0f, 1.5f * even + 0.03f) + tail;
  const float rf = 2.78f * __builtin_amdgcn_exp2f(-__builtin_amdgcn_logf(rho) * (1.0f / 3.0f)) - 1.0f;
  const int rr = (int)__builtin_ceilf(rf * (1.0f / WIN_CHECK)) * WIN_CHECK;
  const int r = __builtin_amdgcn_readfirstlane(rr < WIN_CHECK ? WIN_CHECK : rr > WIN_R ? WIN_R : rr);
  if (__builtin_amdgcn_readfirstlane((int)sparse)) {  // the same for every block of the x range
    if (threadIdx.x == 0) yfs[dz + g] = 1u;
    return;
  }
  const uint16_t* __restrict__ zsl = zs + (uint64_t)z * dx * dy;
  const __amdgpu_buffer_rsrc_t orr = slice_rsrc(out + (uint64_t)z * dx * dy, dx * dy * 2);
  bool cut;
  switch (r) {  // block-uniform
#define GVX_YWIN_CASE(RV) \
  case RV: cut = ywin_block<RV>(kt, zsl, colm, orr, x0, y0, z, dx, dy, nxr, lane, w); break;
    GVX_YWIN_CASE(4) GVX_YWIN_CASE(8) GVX_YWIN_CASE(12) GVX_YWIN_CASE(16)
    GVX_YWIN_CASE(20) GVX_YWIN_CASE(24) GVX_YWIN_CASE(28)
#undef GVX_YWIN_CASE
    default: cut = ywin_block<WIN_R>(kt, zsl, colm, orr, x0, y0, z, dx, dy, nxr, lane, w);
  }
  if (cut && lane == 0) ycut[z] = 1u;
  if (threadIdx.x == 0 && jb == 0) {
    if (z == 0) atomicMax(xcnt + 32, 64u - (uint32_t)r);  // the smallest radius used, as 64 - R
    // the x tiles of the range are read by the x pass
    unsigned long long f = 0;
#pragma unroll
    for (int k = 0; k < TB / TX; ++k)
      if (x0 + k * TX < dx) f |= 1ull << (x0 / TX + k);
    atomicOr(xflags + z, f);
  }
}

// ---------------------------------------------------------------- chunked search
// Where distances are large, windows that grow voxel by voxel look at many positions in
// vain.  A line's keys (SH = 10: cost << 10 | position, unsigned, NKEY_NONE without a
// site) are therefore kept in chunks of YG with each chunk's lowest key: YG outputs of
// one chunk take the sites of their own chunk, then look outwards chunk by chunk; a
// chunk whose lowest key plus the squared distance to it is no better than the worst of
// the outputs is passed over (one LDS read, an addition and a comparison for YG x YG
// pairs), and the search ends when the distance alone is no better.  The lower bound
// holds the tie rule too (key order: cost, then position).  On surface scenes (128^3 and
// 256^3) an x-pass wave visits 4 to 5 chunks of 8 and tests 7 to 15, a y-pass wave visits
// 6 to 9 (its 64 lines differ more) and tests 15 to 28.
// Dimensions up to 1024: costs stay below 3 * 1023^2, so keys stay below NKEY_NONE, and
// NKEY_NONE plus a squared distance inside the line below 2^32.
constexpr uint32_t NKEY_NONE = 0xC0000000u;
// the sites k[0 .. YG) of the chunk D positions after the outputs' (D: a multiple of YG,
// wave-uniform): output i takes the lowest of k[j] + ((D + j - i)^2 << 10)
__device__ __forceinline__ void chunk_visit(const uint32_t (&k)[YG], int D, uint32_t (&b)[YG])
{
  uint32_t c[2 * YG - 1];
#pragma unroll
  for (int m = 0; m < 2 * YG - 1; ++m) c[m] = (uint32_t)((D + m - (YG - 1)) * (D + m - (YG - 1))) << 10;
#pragma unroll
  for (int i = 0; i < YG; ++i)
#pragma unroll
    for (int j = 0; j < YG; j += 2)
      b[i] = min(min(b[i], k[j] + c[j - i + YG - 1]), k[j + 1] + c[j + 1 - i + YG - 1]);
}
__device__ __forceinline__ uint32_t chunk_max(const uint32_t (&b)[YG])
{
  uint32_t m = b[0];
#pragma unroll
  for (int i = 1; i < YG; ++i) m = max(m, b[i]);
  return m;
}
// squared distance (as a key) from any output to the nearest position of a chunk d >= 1 away
__device__ __forceinline__ uint32_t chunk_gap(int d) { return (uint32_t)((YG * (d - 1) + 1) * (YG * (d - 1) + 1)) << 10; }

// The y stack kernel walks a line per lane: a map with few lines leaves the chip idle and
// one walk's latency sets the pace (surface scenes: 60-130 us at 128^3, 80-250 us at
// 256^3, as at 512^3).  Maps of up to
// PBA_CHUNK_MAX voxels (and lines that fit LDS) search chunks instead.
// Both sides measured, whole EDT, box and depth-camera scenes / 1 % and 0.1 % uniform:
// 128^3 67, 68 / 59, 68 us against 202, 131 / 83, 88; 256^3 208, 199 / 146, 190 against
// 372, 264 / 144, 172; 320^3 488, 481 / 343, 420 against 563, 489 / 295, 358.
constexpr uint64_t PBA_CHUNK_MAX = 1ull << 24;
constexpr uint32_t PBA_CHUNK_EDGE = 512;  // longest y line: 64 x 4 bytes of LDS per row, and per chunk
static inline bool pba_chunk_suits(const uint32_t d[3])
{
  return (uint64_t)d[0] * d[1] * d[2] <= PBA_CHUNK_MAX && d[0] <= 1024 && d[1] <= PBA_CHUNK_EDGE && d[2] <= 1024;
}

// y pass: a block takes 64 lines (x range, z), lanes = the lines, a wave YG rows at a
// time; the winner's z is read again from the z pass (a 22-bit cost and two 10-bit
// coordinates do not fit one word).  Output: packed DistanceVoxels.
constexpr int YC_WAVES = 16;
static inline size_t yc_lds(uint32_t dy) { return (size_t)((dy + YG - 1) / YG) * (YG + 1) * TB * 4; }
__global__ void __launch_bounds__(TB * YC_WAVES) k_pba_y_chunk(const uint16_t* __restrict__ zs,
                                                               uint32_t* __restrict__ out, uint32_t dx, uint32_t dy,
                                                               UDiv dzd, uint32_t uninit)
{
  extern __shared__ uint32_t yc_keys[];  // rows up to a whole chunk x 64, then the chunks' lowest keys x 64
  __shared__ uint32_t yc_site[TB];       // the line holds a site
  uint32_t z;
  const uint32_t x0 = dzd.div(blockIdx.x, z) * TB;
  const uint32_t lane = threadIdx.x % TB, w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / TB));
  const uint32_t x = x0 + lane, xl = x < dx ? x : dx - 1;
  const uint32_t nch = (dy + YG - 1) / YG;
  uint32_t* low = yc_keys + nch * YG * TB;
  const uint16_t* __restrict__ zsl = zs + (uint64_t)z * dx * dy;
  if (w == 0) yc_site[lane] = 0u;
  __syncthreads();
  for (uint32_t g = w; g < nch; g += YC_WAVES) {  // a wave stages whole chunks
    uint32_t v[YG], lo = NKEY_NONE;
#pragma unroll
    for (int i = 0; i < YG; ++i) {
      const uint32_t y = g * YG + i;
      v[i] = (zsl + (size_t)((y < dy ? y : dy - 1) * dx))[xl];
    }
#pragma unroll
    for (int i = 0; i < YG; ++i) {
      const uint32_t y = g * YG + i;
      const uint32_t c = (uint32_t)sq24((int32_t)v[i] - (int32_t)z);
      const uint32_t key = v[i] == ZNONE || y >= dy ? NKEY_NONE : c << 10 | y;
      yc_keys[y * TB + lane] = key;
      lo = min(lo, key);
    }
    low[g * TB + lane] = lo;
    if (lo != NKEY_NONE) yc_site[lane] = 1u;
  }
  __syncthreads();
  // a line without a site would keep its wave searching to the end
  const bool want = x < dx && yc_site[lane] != 0u;
  for (uint32_t g = w; g < nch; g += YC_WAVES) {
    uint32_t b[YG], k[YG];
#pragma unroll
    for (int i = 0; i < YG; ++i) {
      b[i] = want && g * YG + i < dy ? 0xFFFFFFFFu : 0u;
      k[i] = yc_keys[(g * YG + i) * TB + lane];
    }
    chunk_visit(k, 0, b);
    uint32_t m = chunk_max(b);
    const int last = (int)max(g, nch - 1 - g);
    for (int d = 1; d <= last; ++d) {
      const uint32_t gap = chunk_gap(d);
      if (wave_ballot(m > gap) == 0ull) break;
#pragma unroll
      for (int side = 0; side < 2; ++side) {  // uniform
        const int gc = side ? (int)g + d : (int)g - d;
        if (gc < 0 || gc >= (int)nch || wave_ballot(low[gc * TB + lane] + gap < m) == 0ull) continue;
#pragma unroll
        for (int i = 0; i < YG; ++i) k[i] = yc_keys[(gc * YG + i) * TB + lane];
        chunk_visit(k, side ? d * YG : -d * YG, b);
        m = chunk_max(b);
      }
    }
    uint32_t ys[YG], zv[YG];
#pragma unroll
    for (int i = 0; i < YG; ++i) {
      ys[i] = b[i] & 1023u;
      zv[i] = zsl[(ys[i] < dy ? ys[i] : dy - 1) * dx + xl];
    }
#pragma unroll
    for (int i = 0; i < YG; ++i)
      if (x < dx && g * YG + i < dy)
        out[((uint64_t)z * dy + g * YG + i) * dx + x] = want ? x | (ys[i] << 10) | (zv[i] << 20) : uninit;
  }
}

// x pass: a block takes XN_ROWS rows (y, z), every wave XN_CH neighbouring chunks of all
// of them (lane = row + XN_ROWS * chunk), so the distances are wave-uniform; a chunk is
// read with two 16-byte LDS reads (row strides of 4 x odd words keep both arrays free of
// bank conflicts).  The winner's entry is read again from the y pass.
constexpr int XN_ROWS = 32, XN_CH = TB / XN_ROWS, XN_WAVES = 8;
static inline __host__ __device__ uint32_t xn_stride(uint32_t nch) { return nch * YG + 4; }            // 4 x odd
static inline __host__ __device__ uint32_t xn_lows(uint32_t nch) { return ((nch + 3) / 4 | 1u) * 4; }  // 4 x odd
static inline size_t xn_lds(uint32_t dx)
{
  const uint32_t nch = (dx + YG - 1) / YG;
  return (size_t)XN_ROWS * (xn_stride(nch) + xn_lows(nch)) * 4;
}
__global__ void __launch_bounds__(TB * XN_WAVES) k_pba_x_chunk(const uint32_t* __restrict__ yb,
                                                               uint32_t* __restrict__ map, uint32_t dx, UDiv dyd,
                                                               uint32_t dz, uint32_t uninit)
{
  extern __shared__ uint4 xn_lds4[];
  uint32_t* keys = reinterpret_cast<uint32_t*>(xn_lds4);
  const uint32_t lane = threadIdx.x % TB, w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / TB));
  const uint32_t nch = (dx + YG - 1) / YG, ks = xn_stride(nch), ls = xn_lows(nch);
  uint32_t* low = keys + XN_ROWS * ks;
  const uint32_t nlines = dyd.d * dz, line0 = blockIdx.x * XN_ROWS;
  constexpr int LD = 4;  // loads in flight
  for (uint32_t r = w; r < (uint32_t)XN_ROWS; r += XN_WAVES) {
    if (line0 + r >= nlines) break;
    uint32_t y;
    const uint32_t z = dyd.div(line0 + r, y);
    const uint32_t* __restrict__ prow = yb + (uint64_t)(line0 + r) * dx;
    for (uint32_t p0 = lane; p0 < nch * YG; p0 += TB * LD) {
      uint32_t v[LD];
#pragma unroll
      for (int j = 0; j < LD; ++j) {
        const uint32_t p = p0 + TB * j;
        v[j] = prow[p < dx ? p : dx - 1];
      }
#pragma unroll
      for (int j = 0; j < LD; ++j) {
        const uint32_t p = p0 + TB * j;
        const uint32_t c = (uint32_t)(sq24((int32_t)((v[j] >> 10) & 0x3FFu) - (int32_t)y) +
                                      sq24((int32_t)(v[j] >> 20) - (int32_t)z));
        if (p < nch * YG) keys[r * ks + p] = v[j] == uninit || p >= dx ? NKEY_NONE : c << 10 | p;
      }
    }
  }
  __syncthreads();
  auto chunk = [&](uint32_t r, uint32_t g, uint32_t (&k)[YG]) {
    const uint4* q = reinterpret_cast<const uint4*>(keys + r * ks + g * YG);
    const uint4 a = q[0], c = q[1];
    k[0] = a.x; k[1] = a.y; k[2] = a.z; k[3] = a.w;
    k[4] = c.x; k[5] = c.y; k[6] = c.z; k[7] = c.w;
  };
  for (uint32_t e = threadIdx.x; e < XN_ROWS * nch; e += TB * XN_WAVES) {
    const uint32_t r = e % XN_ROWS, g = e / XN_ROWS;
    uint32_t k[YG];
    chunk(r, g, k);  // rows past the map hold anything and are not used
    uint32_t lo = k[0];
#pragma unroll
    for (int i = 1; i < YG; ++i) lo = min(lo, k[i]);
    low[r * ls + g] = lo;
  }
  __syncthreads();
  const uint32_t row = lane % XN_ROWS, line = line0 + row;
  const bool act = line < nlines;
  for (uint32_t g0 = w * XN_CH; g0 < nch; g0 += XN_WAVES * XN_CH) {
    const int g = (int)(g0 + lane / XN_ROWS);
    const bool in = act && g < (int)nch;
    uint32_t b[YG], k[YG];
#pragma unroll
    for (int i = 0; i < YG; ++i) b[i] = in && (uint32_t)g * YG + i < dx ? 0xFFFFFFFFu : 0u;
    chunk(row, in ? (uint32_t)g : 0u, k);
    chunk_visit(k, 0, b);
    uint32_t m = chunk_max(b);
    const int last = max((int)g0 + XN_CH - 1, (int)nch - 1 - (int)g0);
    for (int d = 1; d <= last; ++d) {
      const uint32_t gap = chunk_gap(d);
      if (wave_ballot(m > gap) == 0ull) break;
#pragma unroll
      for (int side = 0; side < 2; ++side) {
        const int gc = side ? g + d : g - d;
        const bool there = gc >= 0 && gc < (int)nch;
        const bool better = there && low[row * ls + (there ? (uint32_t)gc : 0u)] + gap < m;
        if (wave_ballot(better) == 0ull) continue;
        if (there) {  // lanes whose line ends before: no sites (and squares beyond a key)
          chunk(row, (uint32_t)gc, k);
          chunk_visit(k, side ? d * YG : -d * YG, b);
        }
        m = chunk_max(b);
      }
    }
    if (!in) continue;
    uint32_t o[YG];
#pragma unroll
    for (int i = 0; i < YG; ++i) o[i] = b[i] >= NKEY_NONE ? uninit : yb[(uint64_t)line * dx + min(b[i] & 1023u, dx - 1)];
    uint32_t* __restrict__ dst = map + (uint64_t)line * dx + (uint32_t)g * YG;
    if ((dx & 3u) == 0) {  // rows of whole 16-byte quads
      *reinterpret_cast<uint4*>(dst) = make_uint4(o[0], o[1], o[2], o[3]);
      if ((uint32_t)g * YG + 4 < dx) *reinterpret_cast<uint4*>(dst + 4) = make_uint4(o[4], o[5], o[6], o[7]);
    } else {
#pragma unroll
      for (int i = 0; i < YG; ++i)
        if ((uint32_t)g * YG + i < dx) dst[i] = o[i];
    }
  }
}

// x pass, phase 2: lines (y, z), lanes = consecutive y.  Stack entry = x |
// (y_site | z_site << 10) << 10, i.e. the packed DistanceVoxel of the site.
// Tiles of 64 lines x TX positions move through LDS so global loads are
// contiguous row segments.
// Tiles of TX positions whose y lines of this slice kept no site (xflags, from the
// y pass) hold only uninitialised voxels: they are neither loaded nor walked.
template <typename T>
__global__ void __launch_bounds__(TB) k_pba_x(const uint32_t* __restrict__ map, const uint16_t* __restrict__ yr,
                                              const uint32_t* __restrict__ yfs, uint32_t* __restrict__ stk,
                                              uint32_t* __restrict__ cnt,
                                              const unsigned long long* __restrict__ xflags,
                                              const uint32_t* __restrict__ xfb, uint32_t dx,
                                              uint32_t dy, uint32_t dz, uint32_t uninit)
{
  constexpr int LPR = 64 / TX;  // loader: rows covered by one pass of the wave
  if (xfb[blockIdx.x] == 0u) return;  // the windowed kernel resolved this group
  constexpr int NLD = TB / LPR;   // loader passes per tile
  __shared__ uint32_t tile[TB][TX + 1];
  __shared__ uint32_t ring[RK][TB];
  __shared__ uint64_t occ[NLD];   // per loader pass: which loaded values hold a site
  // block coordinates as scalars (the buffer descriptor below must be wave-uniform)
  // consecutive blocks take consecutive z with the same y range (every XCD gets
  // every y range); block coordinates as scalars for the buffer descriptor
  const uint32_t z = (uint32_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x % dz));
  const uint32_t y0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)((blockIdx.x / dz) * TB));
  const uint32_t lane = threadIdx.x, y = y0 + lane;
  const bool active = y < dy;
  const int32_t yi = (int32_t)y, zi = (int32_t)z;
  auto cost = [&](uint32_t e) -> T {
    return (T)(sq24((int32_t)((e >> 10) & 0x3FFu) - yi) + sq24((int32_t)(e >> 20) - zi));
  };
  // loader mapping: pass k covers rows LPR k + lane / TX, column lane % TX
  const uint32_t lr = lane / TX, lc = lane % TX;
  const uint32_t ntiles = (dx + TX - 1) / TX;
  LineStack st{ring, stk + ((uint64_t)z * dy + (active ? y : 0)) * dx, lane, 0, 0};
  T tx = 0, tc = 0, sx = 0, sc = 0;
  uint32_t te = 0, se = 0, e3 = 0;  // top, second, third entry of the stack
  Bis<T> bst;
  uint32_t pre[NLD];
  const uint32_t* __restrict__ slice = map + (uint64_t)z * dy * dx;
  const uint16_t* __restrict__ rslice = yr + (uint64_t)z * dy * dx;
  // the tile's y lines went to the stack kernel (their slice, yfs[z], or their 64-column
  // group, yfs[dz + group]): packed sites in map, else relative sites in yr (uniform
  // over the block)
  const bool pks = yfs[z] != 0u;
  auto packed = [&](uint32_t x0) {  // uniform (a scalar branch keeps the tile loads together)
    return pks || __builtin_amdgcn_readfirstlane((int)yfs[dz + (x0 / 64) * dz + z]) != 0;
  };
  // one lane offset plus the row step; in the last block of a line
  // range (rows < TB) rows past dy read the next slice or, after the last slice, the
  // TB rows of padding behind both buffers (their lanes are inactive)
  auto load_tile = [&](uint32_t x0) {
    const uint32_t xc = x0 + lc < dx ? x0 + lc : dx - 1;
    const uint32_t vo = (y0 + lr) * dx + xc;
    if (!packed(x0)) {
      const __amdgpu_buffer_rsrc_t rr = slice_rsrc(rslice, (dx * dy + TB * dx) * 2);
#pragma unroll
      for (int k = 0; k < NLD; ++k)
        pre[k] = __builtin_amdgcn_raw_buffer_load_b16(rr, (int)((vo + LPR * k * dx) * 2), 0, 0);
    } else {
      const __amdgpu_buffer_rsrc_t mr = slice_rsrc(slice, (dx * dy + TB * dx) * 4);
#pragma unroll
      for (int k = 0; k < NLD; ++k)
        pre[k] = __builtin_amdgcn_raw_buffer_load_b32(mr, (int)((vo + LPR * k * dx) * 4), 0, 0);
    }
  };
  unsigned long long todo = xflags[z] & (ntiles >= 64 ? ~0ull : (1ull << ntiles) - 1ull);
  if (todo) load_tile((uint32_t)__builtin_ctzll(todo) * TX);
  while (todo) {
    const uint32_t t = (uint32_t)__builtin_ctzll(todo);
    todo &= todo - 1ull;
    const uint32_t x0 = t * TX;
    const uint32_t cols = dx - x0 < (uint32_t)TX ? dx - x0 : (uint32_t)TX;
    __syncthreads();
    if (!packed(x0)) {  // relative sites: every one is a site (rows >= dy: inactive lanes)
      const uint32_t xc = x0 + lc < dx ? x0 + lc : dx - 1;
#pragma unroll
      for (int k = 0; k < NLD; ++k) pre[k] = yrel_site(pre[k], xc, y0 + LPR * k + lr, z);
    }
#pragma unroll
    for (int k = 0; k < NLD; ++k) {
      tile[LPR * k + lr][lc] = pre[k];
      const uint64_t b = __ballot(pre[k] != uninit);
      if (lane == 0) occ[k] = b;
    }
    __syncthreads();
    load_tile(todo ? (uint32_t)__builtin_ctzll(todo) * TX : x0);  // the next tile (the last one reloads itself)
    if (active) {
      uint32_t m = (uint32_t)((occ[lane / LPR] >> (TX * (lane % LPR))) & ((1ull << TX) - 1ull));
      if (cols < (uint32_t)TX) m &= (1u << cols) - 1u;
      // the next site's value is read from LDS while the current one is processed
      uint32_t lx = m ? (uint32_t)__builtin_ctz(m) : 0u;
      uint32_t e = tile[lane][lx];
      while (m) {
        m &= m - 1u;
        const uint32_t lxn = m ? (uint32_t)__builtin_ctz(m) : lx;
        const uint32_t en = tile[lane][lxn];
        const T x = (T)(x0 + lx), c = cost(e);
        if (st.n >= 1) {
          Bis<T> btn;
          btn.set(tx, tc, x, c);
          while (st.n >= 2 && middle_empty(bst, btn)) {
            // pop the top: second and third move up, the new third is fetched
            st.pop();
            tx = sx;
            tc = sc;
            te = se;
            se = e3;
            sx = (T)(e3 & 0x3FFu);
            sc = cost(e3);
            bst.set(sx, sc, tx, tc);
            e3 = st.at3(st.n >= 3 ? st.n - 3 : 0);
            btn.set(tx, tc, x, c);
          }
          bst = btn;
        }
        e3 = se;
        se = te;
        te = (x0 + lx) | (e & ~0x3FFu);
        st.push(te);
        sx = tx;
        sc = tc;
        tx = x;
        tc = c;
        lx = lxn;
        e = en;
      }
    }
  }
  // the final stack goes to the line's global array (bottom first) for the colouring kernel
  if (active) {
    for (uint32_t d = st.lo; d < st.n; ++d) st.g[d] = ring[d % RK][lane];
    cnt[(uint64_t)z * dy + y] = st.n;
  }
}

// floor(N / D) for D > 0: a float quotient below 2^12 is within 1 of N / D (N and the
// division round to 2^-24 of it), and one integer step corrects its floor.  Larger ones
// (|N| up to 2^25) may be further off, but stay outside the line, which is all that counts.
__device__ __forceinline__ int32_t floor_div(int32_t N, int32_t D)
{
  int32_t q = (int32_t)floorf((float)N / (float)D);
  if (__mul24(q, D) > N) --q;
  else if (__mul24(q + 1, D) <= N) ++q;
  return q;
}

// inclusive prefix maximum over the 64 lanes of a wave: DPP row shifts inside
// each row of 16 lanes (lanes shifted in from outside the row read 0), then the
// totals of lanes 15, 31 and 47 carried into the rows above
__device__ __forceinline__ uint32_t wave_prefix_max(uint32_t v, uint32_t lane)
{
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true));  // row_shr:1
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true));  // row_shr:2
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true));  // row_shr:4
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true));  // row_shr:8
  const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)v, 15);
  if (lane >= 16) v = max(v, r0);
  const uint32_t r1 = (uint32_t)__builtin_amdgcn_readlane((int)v, 31);
  if (lane >= 32) v = max(v, r1);
  const uint32_t r2 = (uint32_t)__builtin_amdgcn_readlane((int)v, 47);
  if (lane >= 48) v = max(v, r2);
  return v;
}

// x pass, colouring: one wave per line (y, z), XC_LPW lines per wave one after
// another, XC_LINES waves per block; lane l takes positions 4 l .. 4 l + 3 of each
// 256-position chunk, so a wave stores 1 KiB of contiguous row per instruction.
// Stack entry k >= 1 owns the positions p with p * D_k > N_k, i.e. p >= start_k =
// floor(N_k / D_k) + 1, for the bisector (N_k, D_k) of entries k - 1 and k.  Phase
// 2 leaves these bisectors strictly increasing in k, so the owner of p is the
// largest k with start_k <= p (0 if none) -- the entry at which the sequential
// top-down colouring stops -- i.e. the prefix maximum over positions of
// mark[start_k] = k.  LDS per wave: mark and entries, dx rounded up to 256 each.
// Lines of groups the windowed kernel resolved are skipped (already written).
// Units of XC_LINES * XC_LPW consecutive lines are dealt to a bounded grid (unit
// u to block u % gridDim.x): a block reads the group flags of all its units with
// one load per lane first, so a field the windowed kernel resolved costs the
// dispatch of that grid and one load, not one block per unit.
constexpr int XC_LINES = 4;
constexpr int XC_LPW = 4;
__host__ __device__ constexpr uint32_t xc_pad(uint32_t dx) { return (dx + 255u) & ~255u; }
__global__ void __launch_bounds__(TB * XC_LINES) k_pba_x_colour(uint32_t* __restrict__ map,
                                                                const uint32_t* __restrict__ stk,
                                                                const uint32_t* __restrict__ cnt,
                                                                const uint32_t* __restrict__ xfb, uint32_t dx,
                                                                UDiv dyd, uint32_t dz, uint32_t uninit)
{
  extern __shared__ uint32_t xc_lds[];
  const uint32_t dy = dyd.d;
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / TB)), lane = threadIdx.x % TB;
  const uint32_t pad = xc_pad(dx);
  uint32_t* mark = xc_lds + (size_t)w * 2 * pad;
  uint32_t* ent = mark + pad;
  const bool vec = (dx & 3u) == 0;  // rows 16-byte aligned: whole uint4 stores
  constexpr uint32_t UL = XC_LINES * XC_LPW;  // lines per unit
  const uint32_t nlines = dy * dz, units = (nlines + UL - 1) / UL;  // dy <= 1024: below 2^32
  // this block's units u = blockIdx.x + i gridDim.x, i < 64 (the grid covers units / 64):
  // lane i tells whether unit i may hold a flagged line (with dy % UL == 0 a unit lies
  // in one group; otherwise every unit is walked and its lines checked one by one)
  unsigned long long todo;
  {
    const uint64_t u = blockIdx.x + (uint64_t)lane * gridDim.x;
    bool f = false;
    if (u < units) {
      uint32_t y0;
      const uint32_t z0 = dyd.div((uint32_t)u * UL, y0);
      f = dy % UL != 0 || xfb[(uint64_t)(y0 / TB) * dz + z0] != 0u;
    }
    todo = wave_ballot(f);  // the same in every wave of the block
  }
  while (todo) {  // no block-wide barrier in here
    const uint32_t ubase = (blockIdx.x + (uint32_t)__builtin_ctzll(todo) * gridDim.x) * UL;
    todo &= todo - 1ull;
    for (uint32_t li = 0; li < (uint32_t)XC_LPW; ++li) {
      const uint32_t ln = ubase + w * XC_LPW + li;
      if (ln >= nlines) return;
      uint32_t ly;
      const uint32_t lz = dyd.div(ln, ly);
      if (xfb[(uint64_t)(ly / TB) * dz + lz] == 0u) continue;
      const uint32_t* __restrict__ s = stk + (uint64_t)ln * dx;
      // the first 64 entries are loaded together with the count (slots past the
      // count hold stale values and are not used)
      const uint32_t n = cnt[ln];
      const uint32_t e0 = s[lane < dx ? lane : 0], a0 = s[lane >= 1 && lane <= dx ? lane - 1 : 0];
      uint32_t* __restrict__ row = map + (uint64_t)ln * dx;
      if (n == 0) {
        for (uint32_t p = lane; p < dx; p += TB) row[p] = uninit;
        continue;
      }
      wave_lds_sync();  // the previous line's reads of mark / ent are done
      for (uint32_t p = 4 * lane; p < pad; p += 4 * TB) *reinterpret_cast<uint4*>(mark + p) = make_uint4(0, 0, 0, 0);
      const int32_t yi = (int32_t)ly, zi = (int32_t)lz;
      auto cost = [&](uint32_t e) -> int32_t {
        return sq24((int32_t)((e >> 10) & 0x3FFu) - yi) + sq24((int32_t)(e >> 20) - zi);
      };
      wave_lds_sync();
      for (uint32_t k = lane; k < n; k += TB) {
        const uint32_t e = k == lane ? e0 : s[k];
        ent[k] = e;
        if (k >= 1) {
          const uint32_t a = k == lane ? a0 : s[k - 1];
          const int32_t pa = (int32_t)(a & 0x3FFu), pb = (int32_t)(e & 0x3FFu);
          const int32_t st = floor_div(__mul24(pb - pa, pb + pa) + cost(e) - cost(a), 2 * (pb - pa)) + 1;
          if (st < (int32_t)dx) atomicMax(&mark[st > 0 ? st : 0], k);
        }
      }
      wave_lds_sync();
      uint32_t carry = 0;
      for (uint32_t c0 = 0; c0 < dx; c0 += 4 * TB) {
        const uint32_t p = c0 + 4 * lane;
        const uint4 mk = *reinterpret_cast<const uint4*>(mark + p);
        uint32_t o0 = mk.x, o1 = max(o0, mk.y), o2 = max(o1, mk.z), o3 = max(o2, mk.w);
        const uint32_t incl = wave_prefix_max(o3, lane);
        uint32_t base = __shfl_up(incl, 1);
        base = max(lane == 0 ? 0u : base, carry);
        carry = max(carry, (uint32_t)__builtin_amdgcn_readlane((int)incl, TB - 1));
        o0 = max(o0, base);
        o1 = max(o1, base);
        o2 = max(o2, base);
        o3 = max(o3, base);
        const uint4 v = make_uint4(ent[o0], ent[o1], ent[o2], ent[o3]);
        if (vec) {
          if (p < dx) *reinterpret_cast<uint4*>(row + p) = v;
        } else {
          if (p < dx) row[p] = v.x;
          if (p + 1 < dx) row[p + 1] = v.y;
          if (p + 2 < dx) row[p + 2] = v.z;
          if (p + 3 < dx) row[p + 3] = v.w;
        }
      }
    }
  }
}

// x pass, windowed: a wave takes XW_RPW rows (y, z) one after another.  The row's
// y-pass entries (relative sites from yr, or packed ones from yb in the slices the y
// stack kernel redid) and their keys (cost (y - y_site)^2 + (z - z_site)^2, position x)
// are staged in LDS, the keys with WIN_R KEY_NONE entries on each side; lane l
// searches positions l + 64 j.  The output at p is the winner's entry, i.e. its
// packed obstacle.  Rows are written only when all of them resolved: a flagged
// group is redone from the untouched y-pass buffer by the proximate-point kernels.
constexpr int XW_WAVES = 4;
constexpr int XW_RPW = 8;  // rows per wave, one after another
// NJ: positions per lane (dx <= 64 NJ)
template <int NJ>
__global__ void __launch_bounds__(TB * XW_WAVES) k_pba_x_win(const uint32_t* __restrict__ yb,
                                                             const uint16_t* __restrict__ yr,
                                                             const uint32_t* __restrict__ yfmt,
                                                             uint32_t* __restrict__ map,
                                                             const unsigned long long* __restrict__ xflags,
                                                             const uint32_t* __restrict__ ycut,
                                                             const uint32_t* __restrict__ rinv,
                                                             uint32_t* __restrict__ xfb, uint32_t* __restrict__ yredo,
                                                             uint32_t dx, UDiv dyd, uint32_t dz, uint32_t uninit)
{
  extern __shared__ uint32_t xw_lds[];
  const uint32_t dy = dyd.d;
  const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / TB)), lane = threadIdx.x % TB;
  const uint32_t kstride = dx + 2 * WIN_R;
  uint32_t* key = xw_lds + (size_t)w * (kstride + dx);  // key[WIN_R + p]
  uint32_t* ent = key + kstride;                        // ent[p]
  const uint32_t ntiles = (dx + TX - 1) / TX;
  const unsigned long long allt = ntiles >= 64 ? ~0ull : (1ull << ntiles) - 1ull;
  const bool full = dx == (uint32_t)(TB * NJ);  // every lane's positions lie in the row
  if (lane < (uint32_t)WIN_R) {
    key[lane] = KEY_NONE;
    key[WIN_R + dx + lane] = KEY_NONE;
  }
  // lines (y, z) number below 2^32 (dy <= 1024); the wave's rows follow one another,
  // so (y, z) is divided out once and then stepped
  const uint32_t nlines = dy * dz, line0 = ((uint32_t)blockIdx.x * XW_WAVES + w) * XW_RPW;
  uint32_t y, yl;
  const uint32_t zf = dyd.div(line0 < nlines ? line0 : 0u, y);
  const uint32_t zl = dyd.div(line0 + XW_RPW - 1 < nlines ? line0 + XW_RPW - 1 : nlines - 1, yl);
  // the wave's rows lie in at most two slices: their x-tile masks are read before any
  // entry, so that no later wait for them also waits for a prefetch
  const unsigned long long tf = line0 < nlines ? xflags[zf] & allt : 0ull, tl = line0 < nlines ? xflags[zl] & allt : 0ull;
  // format of the y output of the wave's (at most two) slices, set by the y stack
  // kernel: 0 = relative sites in yr, 1 = packed sites in yb (every 64-column group of
  // the slice went to the y stack kernel), 2 = both (its rows are left to the x stack
  // kernels, which read each tile in its own format)
  const uint32_t fmtf = line0 < nlines ? yfmt[zf] : 0u, fmtl = line0 < nlines ? yfmt[zl] : 0u;
  // slices whose windowed y pass marked positions beyond its radius R: a winner counts
  // only up to R^2 (see the y pass); a group left over there has its slice's windowed y
  // lines redone by the stack kernel
  const uint32_t cutf = line0 < nlines ? ycut[zf] : 0u, cutl = line0 < nlines ? ycut[zl] : 0u;
  const uint32_t rcut = 64u - *rinv, lim = (rcut + 1u) * (rcut + 1u) << 11;
  if (line0 >= nlines) return;
  if (dy >= (uint32_t)XW_RPW && tf != 0 && tl != 0 && (tf != allt || fmtf == 2u) && (tl != allt || fmtl == 2u)) {
    // no row of this wave can be searched: leave them all (on a 512^3 depth-camera scene
    // every row; walking them one by one took 61 us, leaving them 10 us)
    const uint32_t line = line0 + lane;
    if (lane < (uint32_t)XW_RPW && line < nlines) {
      uint32_t yy;
      const uint32_t zz = dyd.div(line, yy);
      xfb[(uint64_t)(yy / TB) * dz + zz] = 1u;
      if ((zz == zf ? cutf : cutl) != 0u) yredo[zz] = 1u;
    }
    return;
  }
  // the next row's entries are loaded while the current one is searched (relative
  // sites are expanded once they have arrived); only rows that will be searched
  // (every x tile of their slice kept a site) are read: the others' loads get a
  // zero-size buffer and read nothing.  Lanes past dx read past the row (at most
  // into the padding behind the buffers) and are not used.
  auto fetch = [&](uint32_t ln, uint32_t yln, uint32_t zln, uint32_t* dst) {
    const uint32_t fmt = zln == zf ? fmtf : fmtl;
    const bool want = ln < nlines && ((zln == zf ? tf : tl) == allt) && fmt != 2u;  // uniform over the wave
    const uint64_t so = (uint64_t)zln * dx * dy;
    if (fmt == 1u) {
      const __amdgpu_buffer_rsrc_t r = slice_rsrc(yb + so, want ? (dx * dy + TB * dx) * 4 : 0u);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        dst[j] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)(lane * 4), (int)((yln * dx + TB * j) * 4), 0);
    } else {
      const __amdgpu_buffer_rsrc_t r = slice_rsrc(yr + so, want ? (dx * dy + TB * dx) * 2 : 0u);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        dst[j] = __builtin_amdgcn_raw_buffer_load_b16(r, (int)(lane * 2), (int)((yln * dx + TB * j) * 2), 0);
    }
  };
  uint32_t e[NJ], en[NJ];
  uint32_t z = zf;
  fetch(line0, y, z, en);
  for (uint32_t rr = 0; rr < (uint32_t)XW_RPW; ++rr) {  // no block-wide barrier in here
    const uint32_t line = line0 + rr;
    if (line >= nlines) return;
    if (rr > 0) {  // the next row: (y + 1, z) or (0, z + 1)
      const bool wrap = y + 1 == dy;
      y = wrap ? 0u : y + 1;
      z = wrap ? z + 1 : z;
    }
    const uint32_t fmt = z == zf ? fmtf : fmtl;
    const bool pk = fmt == 1u, cut = (z == zf ? cutf : cutl) != 0u;
#pragma unroll
    for (int j = 0; j < NJ; ++j)  // (waits for the prefetch) then the next row's
      e[j] = pk ? en[j] : yrel_site(en[j], lane + TB * j, y, z);
    fetch(rr + 1 < (uint32_t)XW_RPW ? line + 1 : nlines, y + 1 == dy ? 0u : y + 1, y + 1 == dy ? z + 1 : z, en);
    const unsigned long long tiles = z == zf ? tf : tl;
    const uint64_t grp = (uint64_t)(y / TB) * dz + z;
    uint32_t* __restrict__ row = map + (uint64_t)line * dx;
    bool search = false;
    if (tiles == 0) {  // no line of the slice kept a site
      for (uint32_t p = lane; p < dx; p += TB) row[p] = uninit;
    } else if (tiles != allt || fmt == 2u) {  // x ranges without a site (far voxels), or mixed formats
      if (lane == 0) {
        xfb[grp] = 1u;
        if (cut) yredo[z] = 1u;
      }
    } else {
      search = true;
    }
    if (search) {
      const int32_t yi = (int32_t)y, zi = (int32_t)z;
      // the previous row's reads of key / ent are complete before they are overwritten
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      bool any = false;
      if (!pk) {  // from relative sites: every position of a searched row holds one
        auto stage = [&](int j) {
          const uint32_t p = lane + TB * j;
          const int32_t ey = (int32_t)((e[j] >> 10) & 0x3FFu) - yi, ez = (int32_t)(e[j] >> 20) - zi;
          key[WIN_R + p] = site_key((uint32_t)(sq24(ey) + sq24(ez)), p);
          ent[p] = e[j];
        };
        if (full) {
#pragma unroll
          for (int j = 0; j < NJ; ++j) stage(j);
        } else {
#pragma unroll
          for (int j = 0; j < NJ; ++j)
            if (lane + TB * j < dx) stage(j);
        }
        any = true;
      } else {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const uint32_t p = lane + TB * j;
          if (p < dx) {
            const bool site = e[j] != uninit;
            const int32_t ey = (int32_t)((e[j] >> 10) & 0x3FFu) - yi, ez = (int32_t)(e[j] >> 20) - zi;
            key[WIN_R + p] = site ? site_key((uint32_t)(sq24(ey) + sq24(ez)), p) : KEY_NONE;
            ent[p] = e[j];
            any = any || site;
          }
        }
      }
      if (!wave_ballot(any)) {  // a row without a site stays uninitialised
        for (uint32_t p = lane; p < dx; p += TB) row[p] = uninit;
      } else {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        bool fail = false;
        uint32_t res[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          res[j] = 0;
          if ((uint32_t)(TB * j) < dx) {  // uniform over the wave
            const uint32_t p = lane + TB * j;
            bool ok = true;
            const uint32_t b = win_search<11>(key + (p < dx ? p : 0), p < dx, ok);
            fail = fail || !ok || (cut && p < dx && b >= lim);
            res[j] = (b >> 1) & 1023u;
          }
        }
        if (wave_ballot(fail)) {
          if (lane == 0) {
            xfb[grp] = 1u;
            if (cut) yredo[z] = 1u;
          }
        } else {
          if (full) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) row[lane + TB * j] = ent[res[j]];
          } else {
#pragma unroll
            for (int j = 0; j < NJ; ++j)
              if (lane + TB * j < dx) row[lane + TB * j] = ent[res[j]];
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------- read-outs
// DistanceVoxel::squaredObstacleDistance (DistanceVoxel.hpp:38-55)
__device__ __forceinline__ int32_t dist_sq(uint32_t raw, uint64_t id, uint32_t dx, uint32_t dy, uint32_t uninit)
{
  if (raw == uninit) return INT32_MAX;
  const int32_t x = (int32_t)(id % dx), y = (int32_t)((id / dx) % dy), z = (int32_t)(id / ((uint64_t)dx * dy));
  const int32_t ex = x - (int32_t)(raw & 0x3FF), ey = y - (int32_t)((raw >> 10) & 0x3FF), ez = z - (int32_t)(raw >> 20);
  return ex * ex + ey * ey + ez * ez;
}

__global__ void k_dist_sq(const uint32_t* __restrict__ map, const uint32_t* __restrict__ idx, uint64_t n, uint32_t dx,
                          uint32_t dy, uint32_t uninit, int32_t* __restrict__ out)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const uint64_t id = idx[i];
    out[i] = dist_sq(map[id], id, dx, dy, uninit);
  }
}

// The read-out of every voxel in index order: squared distances (int32) or metric
// ones (float).  A thread takes 4 consecutive voxels with one 16-byte load; the
// coordinates of the first come from two reciprocal divisions, the others step (the
// index fits 32 bits: a map has at most 2^32 voxels).  HBM bound: 8 bytes a voxel;
// one voxel per thread with two 64-bit divisions was VALU bound (1.5 instructions
// per byte moved).  vec: out is 16-byte aligned.
template <bool METRIC>
__global__ void __launch_bounds__(256) k_dist_all(const uint32_t* __restrict__ map, uint64_t n, UDiv dxd, UDiv dyd,
                                                  uint32_t uninit, float side, void* __restrict__ out, bool vec)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; 4 * q < n; q += stride) {
    uint32_t x, y;
    uint32_t z = dyd.div(dxd.div((uint32_t)(4 * q), x), y);
    const uint4 v = reinterpret_cast<const uint4*>(map)[q];  // allocations are padded to 256 bytes
    const uint32_t raw[4] = {v.x, v.y, v.z, v.w};
    uint32_t r[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int32_t ex = (int32_t)x - (int32_t)(raw[k] & 0x3FF), ey = (int32_t)y - (int32_t)((raw[k] >> 10) & 0x3FF),
                    ez = (int32_t)z - (int32_t)(raw[k] >> 20);
      const int32_t d = raw[k] == uninit ? INT32_MAX : ex * ex + ey * ey + ez * ez;
      if (METRIC) r[k] = __float_as_uint(d == INT32_MAX ? 3.402823466e+38f : sqrtf((float)d) * side);
      else r[k] = (uint32_t)d;
      if (++x == dxd.d) {
        x = 0;
        if (++y == dyd.d) {
          y = 0;
          ++z;
        }
      }
    }
    uint32_t* o = reinterpret_cast<uint32_t*>(out) + 4 * q;
    if (vec && 4 * q + 4 <= n) {
      *reinterpret_cast<uint4*>(o) = make_uint4(r[0], r[1], r[2], r[3]);
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (4 * q + k < n) o[k] = r[k];
    }
  }
}

// mergeOccupied (DistanceVoxelMap.hpp:109-136 / DistanceVoxelMap.h:92-134): log-odds
// at or above thr write their coordinates.  A lane tests 16 log-odds of one 16-byte
// load 4 bytes at a time and visits only the passing ones; the HBM bytes it needs are
// 1 per voxel and the written ones.  One voxel per thread with two 64-bit divisions
// was issue bound.
__global__ void __launch_bounds__(256) k_merge_occupied(uint32_t* __restrict__ dist, const uint8_t* __restrict__ prob,
                                                        uint64_t n, UDiv dxd, UDiv dyd, uint32_t ox, uint32_t oy,
                                                        uint32_t oz, int thr)
{
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; 16 * c < n; c += stride) {
    uint32_t f[4];
    prob_pass(reinterpret_cast<const uint4*>(prob)[c], thr, f);  // allocations are padded to 256 bytes
    if ((f[0] | f[1] | f[2] | f[3]) == 0u) continue;
    uint32_t x0, y0;
    const uint32_t z0 = dyd.div(dxd.div((uint32_t)(16 * c), x0), y0);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      for (uint32_t m = f[q]; m != 0u; m &= m - 1u) {
        const uint32_t o = (uint32_t)q * 4 + ((uint32_t)__builtin_ctz(m) >> 3);
        const uint64_t i = 16 * c + o;
        if (i >= n) break;
        uint32_t x = x0 + o, y = y0, z = z0;
        while (x >= dxd.d) {
          x -= dxd.d;
          if (++y == dyd.d) {
            y = 0;
            ++z;
          }
        }
        dist[i] = (x + ox) | ((y + oy) << 10) | ((z + oz) << 20);
      }
  }
}

// kernelExactDistances3D (VoxelMapOperations.hpp:896-990): obstacle list staged
// through LDS in tiles; strict < keeps the first minimum in list order.
constexpr int EX_BLOCK = 256;
__global__ void __launch_bounds__(EX_BLOCK) k_exact(uint32_t* __restrict__ map, uint64_t n, uint32_t dx, uint32_t dy,
                                                    uint32_t uninit, const float* __restrict__ obst, uint64_t no,
                                                    float side)
{
  __shared__ int32_t ob[EX_BLOCK][3];
  const uint64_t id = (uint64_t)blockIdx.x * EX_BLOCK + threadIdx.x;
  const bool active = id < n;
  int32_t x = 0, y = 0, z = 0, cur = 0, best = 0;
  int32_t bo[3] = {0, 0, 0};
  bool found = false;
  if (active) {
    x = (int32_t)(id % dx); y = (int32_t)((id / dx) % dy); z = (int32_t)(id / ((uint64_t)dx * dy));
    cur = dist_sq(map[id], id, dx, dy, uninit);
    best = cur;
  }
  for (uint64_t t = 0; t < no; t += EX_BLOCK) {
    __syncthreads();
    const uint64_t k = t + threadIdx.x;
    if (k < no) {
      ob[threadIdx.x][0] = quantize_signed(obst[3 * k], side);
      ob[threadIdx.x][1] = quantize_signed(obst[3 * k + 1], side);
      ob[threadIdx.x][2] = quantize_signed(obst[3 * k + 2], side);
    }
    __syncthreads();
    if (!active || cur == 0) continue;
    const int cnt = (int)((no - t) < (uint64_t)EX_BLOCK ? (no - t) : (uint64_t)EX_BLOCK);
    for (int s = 0; s < cnt; ++s) {
      const int32_t a = ob[s][0], b = ob[s][1], c = ob[s][2];
      if (a == x && b == y && c == z) continue;
      if (a == 1023 || b == 1023 || c == 1023) continue;
      const int32_t ex = x - a, ey = y - b, ez = z - c;
      const int32_t dd = ex * ex + ey * ey + ez * ez;
      if (dd < best) { best = dd; bo[0] = a; bo[1] = b; bo[2] = c; found = true; }
    }
  }
  if (active && found && best < cur) map[id] = (uint32_t)bo[0] | ((uint32_t)bo[1] << 10) | ((uint32_t)bo[2] << 20);
}

static unsigned dist_all_grid(uint64_t n) { return grid_for((n + 3) / 4, 256, 32768); }

struct PbaScratch {
  void* zs = nullptr;     // z pass output, uint16 per voxel
  void* ybuf = nullptr;   // y pass output of the stack kernel, the packed DistanceVoxel per voxel
  void* yrel = nullptr;   // y pass output of the windowed kernel, the relative site per voxel (uint16)
  void* node = nullptr;   // stack spills of the y pass, final stacks of the x pass
  void* cnt = nullptr;    // x pass: stack size per line
  void* flags = nullptr;  // z-pass block flags, x-tile masks per slice, stored row segments, group flags
  uint64_t n = 0, lines = 0, flag_words = 0;
};
static PbaScratch& pba_scratch()
{
  static PbaScratch s;
  return s;
}

// GVX_SYNC_CHECK=1 in the environment: every EDT launch is followed by a stream
// synchronisation, so an execution error is reported with the name of its kernel
static bool pba_sync_check()
{
  static const bool on = [] {
    const char* e = getenv("GVX_SYNC_CHECK");
    return e && e[0] == '1';
  }();
  return on;
}

static int pba_launched(const char* kernel)
{
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && pba_sync_check()) e = hipStreamSynchronize(rt().stream);
  if (e != hipSuccess) return fail(GVX_ERR_HIP, std::string("PBA kernel ") + kernel + ": " + hipGetErrorString(e));
  return GVX_OK;
}

// Elements of padding behind the y-pass outputs: the x stack kernel's tile loads of
// the last line block read up to TB rows of at most 1024 positions past a slice.
constexpr uint64_t PBA_ROW_PAD = (uint64_t)TB * 1024;

// Device buffers of one EDT run (sizes: pba_async, pba_carve).
struct PbaBufs {
  void* zs;     // z pass output, uint16 per voxel
  void* ybuf;   // y pass output of the stack kernel, the packed DistanceVoxel per voxel
  void* yrel;   // y pass output of the windowed kernel, the relative site per voxel (uint16)
  void* node;   // stack spills of the y pass, final stacks of the x pass
  void* cnt;    // x pass: stack size per line
  void* flags;  // z-pass block flags, x-tile masks per slice, stored row segments, group flags
};

// 32-bit words of the flag area for dims (dx, dy, dz)
static uint64_t pba_flag_words(uint32_t dx, uint32_t dy, uint32_t dz)
{
  const uint64_t cwords = (uint64_t)((dy + 31) / 32) * ((dx + 63) / 64);
  const uint64_t xgroups = (uint64_t)((dy + TB - 1) / TB) * dz;
  const uint64_t ygroups = (uint64_t)((dx + TB - 1) / TB) * dz;
  return 64 + 2 * (uint64_t)dz + cwords + dz + ygroups + dz + dz + xgroups + 64;  // the last 64: 2 + 33 used
}

static int pba_launch(MapS* m, const PbaBufs& sc, bool timed);

int pba_async(MapS* m)
{
  const uint32_t dx = m->dims[0], dy = m->dims[1], dz = m->dims[2];
  PbaScratch& sc = pba_scratch();
  {
    const hipError_t e = hipGetLastError();  // an error left by an earlier call is not this call's
    if (e != hipSuccess) return fail(GVX_ERR_HIP, std::string("PBA: pending error before the call: ") + hipGetErrorString(e));
  }
  if (dx > 64u * TX || dy > 32u * TYR) return fail(GVX_ERR_UNSUPPORTED, "PBA: x or y dimension above 1024");
  if (sc.n < m->n) {
    GVX_CHECK(sync());
    dfree(sc.zs);
    dfree(sc.ybuf);
    dfree(sc.yrel);
    dfree(sc.node);
    sc.zs = sc.ybuf = sc.yrel = sc.node = nullptr;
    sc.n = 0;
    GVX_CHECK(dalloc(&sc.zs, m->n * 2));
    GVX_CHECK(dalloc(&sc.ybuf, (m->n + PBA_ROW_PAD) * 4));
    GVX_CHECK(dalloc(&sc.yrel, (m->n + PBA_ROW_PAD) * 2));
    GVX_CHECK(dalloc(&sc.node, m->n * 4));
    sc.n = m->n;
  }
  const uint64_t lines = (uint64_t)dy * dz;
  if (sc.lines < lines) {
    GVX_CHECK(sync());
    dfree(sc.cnt);
    sc.cnt = nullptr;
    sc.lines = 0;
    GVX_CHECK(dalloc(&sc.cnt, lines * 4));
    sc.lines = lines;
  }
  const uint64_t fwords = pba_flag_words(dx, dy, dz);
  if (sc.flag_words < fwords) {
    GVX_CHECK(sync());
    dfree(sc.flags);
    sc.flags = nullptr;
    sc.flag_words = 0;
    GVX_CHECK(dalloc(&sc.flags, fwords * 4));
    sc.flag_words = fwords;
  }
  {
    const hipError_t e = hipGetLastError();  // from freeing or allocating the scratch
    if (e != hipSuccess) return fail(GVX_ERR_HIP, std::string("PBA scratch: ") + hipGetErrorString(e));
  }
  return pba_launch(m, PbaBufs{sc.zs, sc.ybuf, sc.yrel, sc.node, sc.cnt, sc.flags}, true);
}

// The three passes on the library stream over the buffers sc; no allocation.
// timed: named HIP-event scopes around the passes (when profiling is on).
static int pba_launch(MapS* m, const PbaBufs& sc, bool timed)
{
  const uint32_t dx = m->dims[0], dy = m->dims[1], dz = m->dims[2];
  // the skip masks hold 32 row tiles per x range and 64 x tiles per slice
  if (dx > 64u * TX || dy > 32u * TYR) return fail(GVX_ERR_UNSUPPORTED, "PBA: x or y dimension above 1024");
  const uint64_t lines = (uint64_t)dy * dz;
  const uint64_t cwords = (uint64_t)((dy + 31) / 32) * ((dx + 63) / 64);  // stored row segments
  const uint64_t ygroups = (uint64_t)((dx + TB - 1) / TB) * dz;          // y pass: 64 lines (x range, z)
  const uint64_t xgroups = (uint64_t)((dy + TB - 1) / TB) * dz;          // x pass: 64 lines (y range, z)
  const uint64_t fwords = pba_flag_words(dx, dy, dz);
  hipStream_t s = rt().stream;
  uint32_t* map = (uint32_t*)m->data;
  uint16_t* zs = (uint16_t*)sc.zs;
  uint32_t* yb = (uint32_t*)sc.ybuf;
  uint16_t* yr = (uint16_t*)sc.yrel;
  uint32_t* st = (uint32_t*)sc.node;
  uint32_t* tflags = (uint32_t*)sc.flags;
  unsigned long long* xflags = (unsigned long long*)((uint32_t*)sc.flags + 64);
  // 16-byte aligned for fill_u32, also where dz is odd (pba_flag_words' last 64 words have room)
  uint32_t* colm = (uint32_t*)sc.flags + 64 + 2 * ((uint64_t)dz + dz % 2);
  // y lines of the stack kernel: yfs[z] per slice (second run, see k_pba_y), then
  // yfs[dz + group] per 64-column group (ranges too sparse for the window), then per
  // slice the format of its y output (set by the first run for the x pass)
  uint32_t* yfs = colm + cwords;
  uint32_t* yfmt = yfs + dz + ygroups;
  uint32_t* ycut = yfmt + dz;  // slices with positions beyond the y window
  uint32_t* xfb = ycut + dz;   // x groups left to the stack kernels
  uint32_t* xcnt = xfb + xgroups;  // per x range: obstacles, empty cells (+ 16); smallest window radius (+ 32)
  const bool chunks = pba_chunk_suits(m->dims), floats = bis_floats(dx, dy, dz);
  const uint32_t nxr = (dx + TB - 1) / TB;
  const uint64_t cols = (uint64_t)dx * dy;
  const uint32_t u = m->uninit;
  {
    ProfScope ps(timed ? "pba_z" : nullptr);
    if (!chunks) {
      GVX_CHECK(fill_u32(sc.flags, 0u, fwords));
      GVX_CHECK(pba_launched("fill of the flags"));
    }
    const dim3 g(nxr * dy);
#define ZL(W, P)                                                                                               \
  if (dz == 32 * W)                                                                                            \
    hipLaunchKernelGGL((k_pba_z<W, true, P>), g, dim3(64 * (W / P)), 0, s, map, zs, chunks ? nullptr : tflags,    \
                       colm, xcnt, (uint32_t)TYR, dx, dy, dz, udiv(nxr), u);                                   \
  else hipLaunchKernelGGL((k_pba_z<W, false, P>), g, dim3(64 * (W / P)), 0, s, map, zs, chunks ? nullptr : tflags, \
                          colm, xcnt, (uint32_t)TYR, dx, dy, dz, udiv(nxr), u)
    if (chunks && dz <= 512) {
      if (dz <= 128) { ZL(4, 1); }
      else if (dz <= 256) { ZL(8, 1); }
      else { ZL(16, 1); }
    } else {
      if (dz <= 128) { ZL(4, 4); }
      else if (dz <= 256) { ZL(8, 4); }
      else if (dz <= 512) { ZL(16, 4); }
      else if (dz <= 1024) { ZL(32, 4); }
      else {
        hipLaunchKernelGGL(k_pba_z_long, dim3((unsigned)((cols + 255) / 256)), dim3(256), 0, s, map, zs, dx, dy, dz, u);
        GVX_CHECK(fill_u32(tflags, 0xFFFFFFFFu, 64));  // no block flags: every tile is walked
        GVX_CHECK(fill_u32(colm, 0xFFFFFFFFu, cwords));  // and every segment was stored
      }
    }
#undef ZL
    GVX_CHECK(pba_launched("k_pba_z"));
  }
  if (chunks) {
    {
      ProfScope ps(timed ? "pba_y" : nullptr);
      hipLaunchKernelGGL(k_pba_y_chunk, dim3(nxr * dz), dim3(TB * YC_WAVES), yc_lds(dy), s, zs, yb, dx, dy, udiv(dz), u);
      GVX_CHECK(pba_launched("k_pba_y_chunk"));
    }
    ProfScope ps(timed ? "pba_x" : nullptr);
    hipLaunchKernelGGL(k_pba_x_chunk, dim3((unsigned)((lines + XN_ROWS - 1) / XN_ROWS)), dim3(TB * XN_WAVES),
                       xn_lds(dx), s, yb, map, dx, udiv(dy), dz, u);
    return pba_launched("k_pba_x_chunk");
  }
  auto y_stack = [&](bool redo) {
    const auto k = floats ? k_pba_y<float> : k_pba_y<int32_t>;
    hipLaunchKernelGGL(k, dim3((unsigned)ygroups), dim3(TB), 0, s, zs, yb, st, tflags, colm, xflags, yfs, dx, dy, dz, u,
                       redo);
    return pba_launched("k_pba_y");
  };
  {
    ProfScope ps(timed ? "pba_y" : nullptr);
    const uint32_t nyb = (dy + YBR - 1) / YBR;             // blocks per group
    const uint64_t wblocks = (ygroups + 7) / 8 * 8 * nyb;  // blocks of 8 groups per XCD slot
    hipLaunchKernelGGL(k_pba_y_win, dim3((unsigned)wblocks), dim3(TB * YW_WAVES), 0, s, zs, yr, tflags, colm, xflags,
                       yfs, ycut, xcnt, dx, dy, udiv(dz), udiv(nyb), (uint32_t)ygroups);
    GVX_CHECK(pba_launched("k_pba_y_win"));
    GVX_CHECK(y_stack(false));
  }
  {
    ProfScope ps(timed ? "pba_x" : nullptr);
    uint32_t* cnt = (uint32_t*)sc.cnt;
    const uint64_t xrows = (uint64_t)XW_WAVES * XW_RPW;
    const dim3 xg((unsigned)((lines + xrows - 1) / xrows));
    const size_t xl = (size_t)(2 * dx + 2 * WIN_R) * 4 * XW_WAVES;
#define XL(NJ)                                                                                                  \
  hipLaunchKernelGGL(k_pba_x_win<NJ>, xg, dim3(TB * XW_WAVES), xl, s, yb, yr, yfmt, map, xflags, ycut, xcnt + 32, \
                     xfb, yfs, dx, udiv(dy), dz, u)
    if (dx <= 256) XL(4);
    else if (dx <= 512) XL(8);
    else XL(16);
#undef XL
    GVX_CHECK(pba_launched("k_pba_x_win"));
    GVX_CHECK(y_stack(true));
    const auto kx = floats ? k_pba_x<float> : k_pba_x<int32_t>;
    hipLaunchKernelGGL(kx, dim3((unsigned)xgroups), dim3(TB), 0, s, yb, yr, yfs, st, cnt, xflags, xfb, dx, dy, dz, u);
    GVX_CHECK(pba_launched("k_pba_x"));
    const uint64_t clines = (uint64_t)XC_LINES * XC_LPW, units = (lines + clines - 1) / clines;
    const uint64_t cgrid = std::max<uint64_t>((units + 63) / 64, std::min<uint64_t>(units, 4096));
    hipLaunchKernelGGL(k_pba_x_colour, dim3((unsigned)cgrid), dim3(TB * XC_LINES),
                       (size_t)xc_pad(dx) * 8 * XC_LINES, s, map, st, cnt, xfb, dx, udiv(dy), dz, u);
    GVX_CHECK(pba_launched("k_pba_x_colour"));
  }
  return GVX_OK;
}

// Workspace of gvx_dist_pba_noalloc: a fixed device array, so that call allocates
// nothing.  In host code `scratch` is only a symbol; its device address (one per
// device, taken once at gvx_init with the device current) is what kernels get.
constexpr size_t PBA_NOALLOC_BYTES = (size_t)32 << 20;
static __device__ __align__(256) uint8_t scratch[PBA_NOALLOC_BYTES];
static struct {
  int device = -1;         // device the address below belongs to
  void* ptr = nullptr;     // device address of scratch there
  std::string error;       // why it could not be taken, if it could not
} g_noalloc;

int pba_noalloc_setup(int device)
{
  void* ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || ptr == nullptr) {
    (void)hipGetLastError();
    g_noalloc.device = -1;
    g_noalloc.ptr = nullptr;
    g_noalloc.error = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
    return fail(GVX_ERR_HIP, g_noalloc.error);
  }
  g_noalloc.device = device;
  g_noalloc.ptr = ptr;
  g_noalloc.error.clear();
  return GVX_OK;
}

// Carves the run's buffers out of [base, base + cap); false when they do not fit.
static bool pba_carve(const MapS* m, uint8_t* base, size_t cap, PbaBufs* b, size_t* need)
{
  const uint32_t dx = m->dims[0], dy = m->dims[1], dz = m->dims[2];
  auto up = [](uint64_t v) { return (v + 255) & ~(uint64_t)255; };
  const uint64_t o_ybuf = up(m->n * 2), o_yrel = o_ybuf + up((m->n + PBA_ROW_PAD) * 4);
  const uint64_t o_node = o_yrel + up((m->n + PBA_ROW_PAD) * 2);
  const uint64_t o_cnt = o_node + up(m->n * 4);
  const uint64_t o_flags = o_cnt + up((uint64_t)dy * dz * 4);
  const uint64_t total = o_flags + up(pba_flag_words(dx, dy, dz) * 4);
  *need = (size_t)total;
  if (total > cap) return false;
  *b = PbaBufs{base, base + o_ybuf, base + o_yrel, base + o_node, base + o_cnt, base + o_flags};
  return true;
}

}  // namespace gvx

using namespace gvx;

static int check_dist(gvx_map m)
{
  if (!m || !m->data) return fail(GVX_ERR_BAD_ARG, "null map handle");
  if (m->type != GVX_MT_DISTANCE_VOXELMAP) return fail(GVX_ERR_UNSUPPORTED, "not a DistanceVoxelMap");
  return GVX_OK;
}

extern "C" {

int gvx_dist_pba(gvx_map m)
{
  GVX_CHECK(check_dist(m));
  std::lock_guard<std::recursive_mutex> g(m->mu);
  std::lock_guard<std::recursive_mutex> g2(rt().mu);
  {
    ProfScope ps("pba");
    GVX_CHECK(pba_async(m));
  }
  return sync();
}

int gvx_dist_pba_noalloc(gvx_map m)
{
  GVX_CHECK(check_dist(m));
  std::lock_guard<std::recursive_mutex> g(m->mu);
  std::lock_guard<std::recursive_mutex> g2(rt().mu);
  if (g_noalloc.ptr == nullptr || g_noalloc.device != rt().device)
    return fail(GVX_ERR_HIP, "gvx_dist_pba_noalloc: no workspace on this device (" +
                                 (g_noalloc.error.empty() ? std::string("gvx_init did not set it up") : g_noalloc.error) +
                                 ")");
  PbaBufs b;
  size_t need = 0;
  if (!pba_carve(m, (uint8_t*)g_noalloc.ptr, PBA_NOALLOC_BYTES, &b, &need))
    return fail(GVX_ERR_BAD_ARG, "gvx_dist_pba_noalloc: a " + std::to_string(m->dims[0]) + "x" +
                                     std::to_string(m->dims[1]) + "x" + std::to_string(m->dims[2]) + " map needs " +
                                     std::to_string(need) + " bytes of workspace, above the fixed " +
                                     std::to_string(PBA_NOALLOC_BYTES) + "; use gvx_dist_pba");
  {
    const hipError_t e = hipGetLastError();  // an error left by an earlier call is not this call's
    if (e != hipSuccess)
      return fail(GVX_ERR_HIP, std::string("PBA: pending error before the call: ") + hipGetErrorString(e));
  }
  GVX_CHECK(pba_launch(m, b, false));
  return sync();
}

int gvx_dist_merge_occupied(gvx_map dist, gvx_map prob, const uint32_t offset[3], float threshold)
{
  GVX_CHECK(check_dist(dist));
  if (!prob || prob->type != GVX_MT_PROBAB_VOXELMAP) return fail(GVX_ERR_BAD_ARG, "mergeOccupied needs a ProbVoxelMap");
  if (memcmp(dist->dims, prob->dims, sizeof(dist->dims)) != 0)
    return fail(GVX_ERR_DIM_MISMATCH, "mergeOccupied: map dimensions differ");
  std::unique_lock<std::recursive_mutex> g1(dist->mu, std::defer_lock), g2(prob->mu, std::defer_lock);
  std::lock(g1, g2);
  const int thr = (int)float_to_probability(threshold) + 1;  // strictly above the threshold
  if (thr <= PROB_MAX) {
    hipLaunchKernelGGL(k_merge_occupied, dim3(grid_for((dist->n + 15) / 16, 256, 16384)), dim3(256), 0, rt().stream,
                       (uint32_t*)dist->data, (const uint8_t*)prob->data, dist->n, udiv(dist->dims[0]),
                       udiv(dist->dims[1]), offset ? offset[0] : 0u, offset ? offset[1] : 0u, offset ? offset[2] : 0u,
                       thr);
    GVX_HIP(hipGetLastError());
  }
  return sync();
}

int gvx_dist_exact(gvx_map m, const float* obstacles, uint64_t n, int mem)
{
  GVX_CHECK(check_dist(m));
  if (n && !obstacles) return fail(GVX_ERR_BAD_ARG, "null obstacles");
  std::lock_guard<std::recursive_mutex> g(m->mu);
  std::lock_guard<std::recursive_mutex> g2(rt().mu);
  const void* d = nullptr;
  GVX_CHECK(stage_input(obstacles, n * 12, mem, &d));
  hipLaunchKernelGGL(k_exact, dim3((unsigned)((m->n + EX_BLOCK - 1) / EX_BLOCK)), dim3(EX_BLOCK), 0, rt().stream,
                     (uint32_t*)m->data, m->n, m->dims[0], m->dims[1], m->uninit, (const float*)d, n, m->side);
  GVX_HIP(hipGetLastError());
  return sync();
}

int gvx_dist_squared(gvx_map m, const uint32_t* idx, uint64_t n, int32_t* out, int mem)
{
  GVX_CHECK(check_dist(m));
  if (!out) return fail(GVX_ERR_BAD_ARG, "null out");
  if (!idx) n = m->n;
  if (n == 0) return GVX_OK;
  std::lock_guard<std::recursive_mutex> g(m->mu);
  std::lock_guard<std::recursive_mutex> g2(rt().mu);
  // indices staged in front, results behind
  size_t ib = idx ? ((n * 4 + 255) & ~(size_t)255) : 0;
  void* st = nullptr;
  const uint32_t* didx = nullptr;
  int32_t* dout = out;
  if (idx && mem == GVX_MEM_DEVICE) didx = idx;
  size_t need = (idx && mem == GVX_MEM_HOST ? ib : 0) + (mem == GVX_MEM_HOST ? n * 4 : 0);
  if (need) GVX_CHECK(stage_reserve(need, &st));
  if (idx && mem == GVX_MEM_HOST) {
    GVX_HIP(hipMemcpyAsync(st, idx, n * 4, hipMemcpyHostToDevice, rt().stream));
    didx = (const uint32_t*)st;
  }
  if (mem == GVX_MEM_HOST) dout = (int32_t*)((char*)st + (idx ? ib : 0));
  if (idx) {
    // bounds-check indices on the way: invalid ids are rejected before launch
    std::vector<uint32_t> host;
    const uint32_t* hp = idx;
    if (mem == GVX_MEM_DEVICE) {
      host.resize(n);
      GVX_HIP(hipMemcpyAsync(host.data(), idx, n * 4, hipMemcpyDeviceToHost, rt().stream));
      GVX_CHECK(sync());
      hp = host.data();
    }
    for (uint64_t i = 0; i < n; ++i)
      if (hp[i] >= m->n) return fail(GVX_ERR_BAD_ARG, "voxel index out of range");
  }
  if (didx)
    hipLaunchKernelGGL(k_dist_sq, dim3(grid_for(n, 256, 8192)), dim3(256), 0, rt().stream, (const uint32_t*)m->data,
                       didx, n, m->dims[0], m->dims[1], m->uninit, dout);
  else
    hipLaunchKernelGGL(k_dist_all<false>, dim3(dist_all_grid(n)), dim3(256), 0, rt().stream,
                       (const uint32_t*)m->data, n, udiv(m->dims[0]), udiv(m->dims[1]), m->uninit, m->side,
                       (void*)dout, ((uintptr_t)dout & 15) == 0);
  GVX_HIP(hipGetLastError());
  if (mem == GVX_MEM_HOST) GVX_HIP(hipMemcpyAsync(out, dout, n * 4, hipMemcpyDeviceToHost, rt().stream));
  return sync();
}

int gvx_dist_metric(gvx_map m, float* out, int mem)
{
  GVX_CHECK(check_dist(m));
  if (!out) return fail(GVX_ERR_BAD_ARG, "null out");
  std::lock_guard<std::recursive_mutex> g(m->mu);
  std::lock_guard<std::recursive_mutex> g2(rt().mu);
  float* dout = out;
  if (mem == GVX_MEM_HOST) {
    void* st = nullptr;
    GVX_CHECK(stage_reserve(m->n * 4, &st));
    dout = (float*)st;
  }
  hipLaunchKernelGGL(k_dist_all<true>, dim3(dist_all_grid(m->n)), dim3(256), 0, rt().stream,
                     (const uint32_t*)m->data, m->n, udiv(m->dims[0]), udiv(m->dims[1]), m->uninit, m->side,
                     (void*)dout, ((uintptr_t)dout & 15) == 0);
  GVX_HIP(hipGetLastError());
  if (mem == GVX_MEM_HOST) GVX_HIP(hipMemcpyAsync(out, dout, m->n * 4, hipMemcpyDeviceToHost, rt().stream));
  return sync();
}

}  // extern "C"
