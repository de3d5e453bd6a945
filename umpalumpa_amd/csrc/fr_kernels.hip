// FR insertion kernels for gfx950: voxel-owned gather.
//
// The reference scatters each rotated slice into the volume with three float atomics per voxel
// (fr_cuda_kernels.cu:266-365).  Here a wavefront owns a brick of 8 x 8 x D voxels (a z column
// of D per lane, D = 8, 4, 2 or 1 by distance from the centre) for the whole work item and
// keeps their running (complex, weight) sums in its LDS slot.  It culls the traverse spaces
// against the brick 64 at a time with one ballot and walks the surviving spaces in index
// order, so every voxel receives its per-space contributions in the order of the reference CPU
// loop over spaces (fr_cpu_kernels.hpp:254): no atomics, and no dependence on how bricks are
// scheduled.
//
// Per (brick, space) pair the wave
//   1. tests the reference's slab condition (q.z^2 <= r^2) for its voxels, an addition and a
//      compare each, and compacts the voxels that pass into its LDS queue;
//   2. runs the rest of the reference predicate and the gather over the queue with full lanes:
//      a branch-free NB x NB candidate loop over whole pixel rows in which a candidate the
//      reference skips reads the zero entry appended to the LDS blob table, adding +-0 (finite
//      slice values), so the sums are bit-identical to the reference's skip-the-pixel loop
//      while all table and pixel loads of an item issue back to back; each voxel appears once
//      per space, so its lane adds the contribution to the voxel's LDS sum directly.
// Workgroups are persistent (one per CU: 16 or 12 wavefronts sharing the blob table in LDS)
// and take bricks from a counter, most central (heaviest) first.
//
// Small volumes take the cell kernel (fr_cells.hip) instead; see use_cells().
//
// fr_insert_kernel covers every mode, precision and strategy; fr_insert_staged_kernel, for the
// exact FP32 lookup strategy, gathers the predicate's hits of several spaces together (see
// there).
#include "fr_cell.hpp"

#include <algorithm>

namespace umpa {

constexpr int kMaxLdsTable = kFrMaxLdsTable;  // floats next to the per-wave state; larger tables stay global
// Wavefronts per workgroup (they share the LDS table): 16 (4 per SIMD) in general; the exact
// FP32 lookup kernel runs faster with 12 (1.94 -> 1.86 ms per 1,000-slice chunk at box 256),
// the fast-math and FP16 kernels slower (1.46 -> 1.68 and 1.39 -> 1.60 ms).
constexpr int kMaxWaves = 16;
__host__ __device__ constexpr int fr_waves(int mode, bool half, bool fastMath)
{
  return (mode == kModeLookup && !half && !fastMath) ? 12 : kMaxWaves;
}
constexpr int kEdge = 8;             // brick edge: a wave owns 8 x 8 x 8 voxels, a z column per lane
constexpr int kVox = kEdge * kEdge * kEdge;

// Per-wave LDS state: running sums of the wave's 8 x 8 x 8 brick and the queue of voxels that
// pass the slab test for the current space.
struct alignas(16) WaveScratch {
  float accR[kVox];
  float accI[kVox];
  float accW[kVox];
  uint16_t queue[kVox];
};
// fr_insert_kernel's LDS with its largest table (and the words beside the per-wave state)
static_assert(kMaxWaves * (sizeof(WaveScratch) + sizeof(umpa_traverse_space)) + 16 +
                (kMaxLdsTable + 1) * sizeof(float) <= 160 * 1024, "one workgroup per CU");

// Element `index` (wave-uniform) of a buffer the kernels only read, through the constant
// address space: the compiler then reads it with scalar loads into SGPRs instead of 16-byte
// vector loads of one address.  The exact kernel with cross-space batches reads its space
// records this way (1.75 -> 1.62 ms per box-256 chunk).  In fr_insert_kernel the same change
// made the fast-math and FP16 kernels slower (1.46 -> 1.94 and 1.39 -> 1.87 ms; their SGPR
// count reached 100, with spills through VGPR lanes), so they keep the vector loads.
template <typename T>
__device__ __forceinline__ T uniform_load(const T *p, int index)
{
  static_assert(sizeof(T) % 4 == 0, "dword-sized records only");
  typedef __attribute__((address_space(4))) const int const_int;
  const const_int *src = (const const_int *)(p + index);
  int w[sizeof(T) / 4];
#pragma unroll
  for (int i = 0; i < (int)(sizeof(T) / 4); ++i) w[i] = src[i];
  T out;
  __builtin_memcpy(&out, w, sizeof(T));
  return out;
}

// The wavefront's number in the launch, workgroups first: consecutive numbers are different CUs.
__device__ __forceinline__ int wave_number()
{
  return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) * (int)gridDim.x + (int)blockIdx.x;
}

// Items are taken in order, heaviest first: a wavefront's first is its number, the others come
// from the counter, which counts on from the launch's `claimed` wavefronts.  (Every claim on the
// one counter holds up the others by about 8 ns: with the first ones counted too, a launch of 3,072
// wavefronts spent 25 us before its first brick; box 192, 333 spaces, exact 404 -> 373 us.)
// Each item taken makes one claim, so the last of the launch finds nItems - 1: it clears the
// counter for the next launch.
__device__ __forceinline__ int claim_item(const FrLaunch &l, int lane, int claimed)
{
  int next = 0;
  if (lane == 0) {
    next = atomicAdd(l.counter, 1);
    if (next == l.nItems - 1) atomicExch(l.counter, 0);
  }
  return __builtin_amdgcn_readfirstlane(next) + claimed;
}

// A wavefront's first brick where the first nCore of them begin with a cell of the core: the others
// start on the heaviest bricks, these on the lightest of the first ones.
__device__ __forceinline__ int first_after_core(const FrLaunch &l, int number, int claimed)
{
  const int core = l.nCore % claimed;
  return number >= core ? number - core : number + claimed - core;
}

// Bounded launches (l.waveItems items for each of a workgroup's wavefronts, the grid covering the
// items) need no global counter: workgroups go by groups of one per CU, a group takes the next
// items in order and deals them out across its workgroups, so that a workgroup's items cost about
// the same and the heaviest lie on different CUs.  (With the counter, a four-job serving tick of
// 63,000 items made 95,000 claims: 1737 -> 1635 us.)  A workgroup's wavefronts take its items in
// order from a count in LDS: its LDS comes free only with its last wavefront, and items of one
// estimated cost differ (the same tick, two items each: 1665 -> 1580 us).
struct DealtItems {
  int first, step, n;  // the workgroup's items: first + k step, k < n
};
__device__ __forceinline__ DealtItems deal_items(const FrLaunch &l, int waves)
{
  const int group = (int)blockIdx.x / l.numCUs, in = (int)blockIdx.x - group * l.numCUs;
  const int start = group * l.numCUs;
  const int size = min(l.numCUs, (int)gridDim.x - start);
  const int n = waves * l.waveItems;
  return { start * n + in, size, n };
}

// Item k of the workgroup's (nItems: none left).
__device__ __forceinline__ int dealt_item(const FrLaunch &l, const DealtItems &d, int k)
{
  return k < d.n ? min(d.first + k * d.step, l.nItems) : l.nItems;
}

__device__ __forceinline__ int next_dealt(const FrLaunch &l, const DealtItems &d, int *taken, int lane)
{
  int k = 0;
  if (lane == 0) k = atomicAdd(taken, 1);
  return dealt_item(l, d, __builtin_amdgcn_readfirstlane(k));
}

// ---- the brick's steps shared by the insertion kernels ----------------------------------------
constexpr float kHalfEdge = 0.5f * (kEdge - 1);
// |qz| <= r (1 + 1e-6) holds wherever the float qz * qz is at most the float r * r
constexpr float kSlabMargin = 1.f + 1e-6f;

// The slab test's bound for half width `r` and transforms of |t22| up to `t` (see slab_queue).  With
// u = 2^-24 and v the volume's depth: in either sum t22 pz rounds by at most u t v / 2, and a sum by
// u times its size, which is r where the voxel passes and at most r + 7 t at the up to eight levels
// that qz steps through: together less than u ((v + 56) t + 9 r), u = 6e-8.
__device__ __forceinline__ float slab_reach(float r, int v, float t)
{
  return r * kSlabMargin + 1e-7f * ((float)(v + 64) * t + 10.f * r);
}

// Brick of the work item and the lane's column of it.
struct BrickCtx {
  int x0, y0, z0;     // brick origin
  int nz;             // levels inside the volume (wave-uniform)
  int x, y;           // the lane's column
  bool colIn;         // the column lies inside the volume
  float px, py;       // the column in centred coordinates
  float bcx, bcy, bcz, hz, dmin, eps;  // brick centre, half depth and the cull's margins
};

__device__ __forceinline__ BrickCtx make_brick(const FrJob &a, const int4 &bo, int lane)
{
  BrickCtx b;
  const umpa_fr_constants &c = a.c;
  const int cxi = c.cMaxVolumeIndexX / 2, cyi = c.cMaxVolumeIndexYZ / 2;
  const int depth = bo.w & 15;
  b.x0 = bo.x;
  b.y0 = bo.y;
  b.z0 = bo.z & 0xffff;
  b.x = bo.x + (lane & (kEdge - 1));
  b.y = bo.y + lane / kEdge;
  b.colIn = b.x < a.vx && b.y < a.vy;
  b.nz = min(depth, a.vz - b.z0);
  b.px = (float)(b.x - cxi);
  b.py = (float)(b.y - cyi);
  // brick centre in centred volume coordinates, half extents (3.5, 3.5, (depth - 1) / 2)
  b.hz = 0.5f * (float)(depth - 1);
  b.bcx = (float)(bo.x - cxi) + kHalfEdge;
  b.bcy = (float)(bo.y - cyi) + kHalfEdge;
  b.bcz = (float)(b.z0 - cyi) + b.hz;
  const float bnorm = sqrtf(b.bcx * b.bcx + b.bcy * b.bcy + b.bcz * b.bcz);
  b.dmin = fmaxf(bnorm - sqrtf(2.f * kHalfEdge * kHalfEdge + b.hz * b.hz), 0.f);
  b.eps = 0.02f + 1e-5f * bnorm;
  return b;
}

// Do all of the brick's voxels pass the reference's sphere test (|p|^2 <= maxDistanceSqr; the
// farthest corner's squared distance is an exact integer in float, as is every voxel's) and lie
// in the space's traversal plane (the AABB extents orthogonal to `dir`)?  Wave-uniform.
__device__ __forceinline__ bool brick_inside(const BrickCtx &b, const umpa_traverse_space &sp,
                                             int cxi, int cyi)
{
  const int x1 = b.x0 + kEdge - 1, y1 = b.y0 + kEdge - 1, z1 = b.z0 + b.nz - 1;
  const int mx = max(abs(b.x0 - cxi), abs(x1 - cxi));
  const int my = max(abs(b.y0 - cyi), abs(y1 - cyi));
  const int mz = max(abs(b.z0 - cyi), abs(z1 - cyi));
  const bool sphere = (float)(mx * mx + my * my + mz * mz) <= sp.maxDistanceSqr;
  const bool inX = b.x0 >= sp.minX && x1 <= sp.maxX;
  const bool inY = b.y0 >= sp.minY && y1 <= sp.maxY;
  const bool inZ = b.z0 >= sp.minZ && z1 <= sp.maxZ;
  const int dir = sp.dir;
  const bool box = dir == 0 ? (inX && inY) : dir == 1 ? (inX && inZ) : (inY && inZ);
  return __builtin_amdgcn_readfirstlane((int)(sphere && box)) != 0;
}

// The brick's running sums start from the volume (or from zero for a split part).  Levels go
// four at a time, all their loads in flight before the first is written to LDS.
template <typename Scratch>
__device__ __forceinline__ void load_brick(Scratch &ws, const FrJob &a, const BrickCtx &b,
                                           int lane, bool fromZero)
{
  const int64_t plane = (int64_t)a.vy * a.vx;
  const int64_t g0 = ((int64_t)b.z0 * a.vy + b.y) * a.vx + b.x;
  const float2 *vol = reinterpret_cast<const float2 *>(a.volume);
  const bool read = !fromZero && b.colIn;
  for (int k0 = 0; k0 < b.nz; k0 += 4) {
    float2 v[4];
    float w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = make_float2(0.f, 0.f);
      w[k] = 0.f;
      if (read && k0 + k < b.nz) {
        v[k] = vol[g0 + (k0 + k) * plane];
        w[k] = a.weights[g0 + (k0 + k) * plane];
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int li = (k0 + k) * 64 + lane;
      if (k0 + k < b.nz) {
        ws.accR[li] = v[k].x;
        ws.accI[li] = v[k].y;
        ws.accW[li] = w[k];
      }
    }
  }
  wave_sync();
}

// The brick's sums back to the volume: stored, or added with atomics for a split part.
template <typename Scratch>
__device__ __forceinline__ void store_brick(const Scratch &ws, const FrJob &a,
                                            const BrickCtx &b, int lane, bool split)
{
  const int64_t plane = (int64_t)a.vy * a.vx;
  const int64_t g0 = ((int64_t)b.z0 * a.vy + b.y) * a.vx + b.x;
  if (b.colIn) {
    for (int k = 0; k < b.nz; ++k) {
      const int li = k * 64 + lane;
      const int64_t gi = g0 + k * plane;
      if (split) {
        float *vol = reinterpret_cast<float *>(a.volume);
        if (ws.accW[li] != 0.f || ws.accR[li] != 0.f || ws.accI[li] != 0.f) {
          atomicAdd(vol + 2 * gi, ws.accR[li]);
          atomicAdd(vol + 2 * gi + 1, ws.accI[li]);
          atomicAdd(a.weights + gi, ws.accW[li]);
        }
      } else {
        reinterpret_cast<float2 *>(a.volume)[gi] = make_float2(ws.accR[li], ws.accI[li]);
        a.weights[gi] = ws.accW[li];
      }
    }
  }
  wave_sync();
}

// Cull of space `si` (one per lane) against the brick: slab half-width, half-space and sphere
// with the brick's extents as margins; spaces naming a slice that does not exist never pass.
// Bricks this far from the centre (in voxels) exist only in volumes above box 256; there most
// spaces miss the brick's slab, so the cull rejects on the slab test before it loads the rest of
// the record (box 1024, D7: 141.5 -> 131.2 ms per 512-slice step), while closer bricks load every
// field at once (box 256: the early rejection would cost 1 to 3 %).
constexpr float kEarlyCullRadius = 128.f;
// `t22` is the record's |t22| (0 past the last space).
template <bool kEarly>
__device__ __forceinline__ bool cull_space(const FrJob &a, const BrickCtx &b, int si, int sEnd,
                                           float &t22)
{
  t22 = 0.f;
  if (si >= sEnd) return false;
  const umpa_traverse_space &sp = a.spaces[si];
  const float(*t)[3] = sp.transformInv;
  t22 = fabsf(t[2][2]);
  const float qz = t[2][0] * b.bcx + t[2][1] * b.bcy + t[2][2] * b.bcz;
  const float ez = kHalfEdge * (fabsf(t[2][0]) + fabsf(t[2][1])) + b.hz * fabsf(t[2][2]);
  const bool slab = fabsf(qz) <= a.cullHalfWidth + ez + b.eps;
  if (kEarly && !slab) return false;
  const float qx = t[0][0] * b.bcx + t[0][1] * b.bcy + t[0][2] * b.bcz;
  const float ex = kHalfEdge * (fabsf(t[0][0]) + fabsf(t[0][1])) + b.hz * fabsf(t[0][2]);
  // the (other) conditions are all evaluated (&, not &&), so their fields load together instead
  // of one after another behind the earlier tests
  const float mds = sp.maxDistanceSqr;
  const int proj = sp.projectionIndex, dir = sp.dir;
  return slab & (qx >= -a.cullHalfSpace - ex - b.eps) &
         (b.dmin * b.dmin <= mds * 1.0001f + b.eps) & (proj >= 0) & (proj < a.nProj) &
         (dir >= 0) & (dir <= 2);
}

// The column's limit in the slab tests of 64 spaces, `t22` from the lane's: `usual` where each is at
// most kUsualT22, as a rotation's is, else what the largest needs.  The five- and six-wide kernels
// (!kHold), which spill where one more register is held, compute it anew, for 4,096 or no limit at
// all.  (us, kUsualT22's only / held / anew: box 256, 1,000 slices, exact 1220 / 1224 / 1226, FP16 1039 /
// 1038 / 1044; four FP16 jobs, bounded 1306 / 1306 / 1338; box 256, 500, exact in a batch, r 2.5 1448
// / 1583 / 1461.)
constexpr float kUsualT22 = 2.f;
template <bool kHold>
__device__ __forceinline__ float slab_limit(float usual, const FrJob &a, const BrickCtx &b, float r,
                                            float t22)
{
  const bool large = __any(!(t22 <= kUsualT22));
  if constexpr (kHold) {
    if (!large) return usual;
    for (int d = 32; d > 0; d >>= 1) t22 = fmaxf(t22, __shfl_xor(t22, d));
    return b.colIn ? slab_reach(r, a.vz, fmaxf(t22, kUsualT22)) : -1.f;
  } else {
    const float t = !large ? kUsualT22 : __any(!(t22 <= 4096.f)) ? __builtin_inff() : 4096.f;
    return b.colIn ? slab_reach(r, a.vz, t) : -1.f;
  }
}

// Phase 1: the slab test of the column's nz voxels; the voxels that pass go to the wave's queue
// behind `pending` entries (index k * 64 + lane, plus `tag`), their number is returned.
// qz steps by t22 from level to level, one addition each where the reference's left-to-right sum
// (t20 px + t21 py) + t22 pz takes a conversion, a product and an addition; `lim` is above the
// slab's half width by what the two can differ (slab_reach), so that |qz| <= lim holds for every
// voxel that passes the reference's rounded q.z^2 <= r^2, which phase 2 tests: one compare per
// level, whose lane mask is the ballot.  (A column outside the volume compares against -1, which
// nothing passes.)  Box 256, 1,000 slices: fast math 1100 -> 1094 us, exact 1236 -> 1231; box 1024,
// D7, FP16 116.7 -> 114.9 ms; mixed batch 3710 -> 3671 us.
template <typename Scratch>
__device__ __forceinline__ int slab_queue(Scratch &ws, const FrJob &a, const BrickCtx &b,
                                          const umpa_traverse_space &sp, float lim, int lane,
                                          int pending = 0, uint32_t tag = 0)
{
  const int cyi = a.c.cMaxVolumeIndexYZ / 2;
  const float t20 = sp.transformInv[2][0], t21 = sp.transformInv[2][1],
              t22 = sp.transformInv[2][2];
  const float cz = t20 * b.px + t21 * b.py;
  uint32_t entry = (uint32_t)lane | tag;
  int end = pending;
  float qz = cz + t22 * (float)(b.z0 - cyi);
  for (int k = 0; k < b.nz; ++k, qz += t22) {
    const bool ok = !(fabsf(qz) > lim);
    const unsigned long long m = __ballot(ok);
    if (ok) ws.queue[lanes_below(m, (unsigned)end)] = (uint16_t)entry;
    end += __popcll(m);
    entry += 64;
  }
  return end - pending;
}

template <int kMode, int kOrder, int kNB, bool kHalf, bool kFastMath, bool kCount, bool kTableLds,
          bool kBatched, bool kShift>
__global__ __launch_bounds__(64 * fr_waves(kMode, kHalf, kFastMath)) void fr_insert_kernel(FrJob job0, FrLaunch l)
{
  constexpr int kWaves = fr_waves(kMode, kHalf, kFastMath);
  constexpr int kThreads = 64 * kWaves;
  extern __shared__ float s_table[];
  __shared__ WaveScratch s_wave[kWaves];
  __shared__ umpa_traverse_space s_space[kWaves];  // the space the wave works on
  __shared__ float s_blob[evaluates_blob(kMode) ? kWaves : 1][evaluates_blob(kMode) ? kBlobList : 1];
  const int nTable = l.nTable;
  if constexpr (kMode == kModeLookup && kTableLds) {
    stage_table<kThreads>(s_table, l.table, nTable);
  }
  const float *tbl = (kMode == kModeLookup && kTableLds) ? s_table : l.table;
  const int lane = threadIdx.x & 63;
  WaveScratch &ws = s_wave[threadIdx.x >> 6];
  constexpr int kPix = kHalf ? 4 : 8;
  // the workgroup's updates: one addition per item or cell to the launch's number, 8 ns each, was
  // longer than the work of a small volume (box 48, 16 spaces: 78 -> 54 us)
  __shared__ unsigned long long s_updates;
  if constexpr (kCount) {
    if (threadIdx.x == 0) s_updates = 0;
    __syncthreads();
  }
  static_assert(kBlobList <= kVox, "a cell's evaluations fit one of the wave's arrays of sums");

  const int number = wave_number(), claimed = kWaves * (int)gridDim.x;
  if constexpr (!kFastMath && !kBatched) {
    if (job0.spaceBegin >= job0.spaceEnd) return;
    // the volume's core, cell by cell, as in fr_insert_staged_kernel
    for (int b = number; b < l.nCore; b += claimed) {
      const int2 bo = make_uniform(reinterpret_cast<const int2 *>(l.core)[b]);
      const __amdgpu_buffer_rsrc_t all = __builtin_amdgcn_make_buffer_rsrc(
        (void *)job0.fft, 0, (int)((uint32_t)job0.nProj * (uint32_t)(job0.sliceElems * kPix)),
        kBufferConfig);
      unsigned long long n = 0;
      cell_item<kMode, kOrder, kNB, kMode == kModeLookup && kTableLds, kShift, kCount>(
        job0, bo.x & 0xffff, bo.x >> 16, bo.y, job0.spaceBegin, job0.spaceEnd,
        reinterpret_cast<uint32_t *>(ws.queue), ws.accR, ws.accI, nTable, all, tbl, lane, n);
      if constexpr (kCount) {
        if (lane == 0 && n) atomicAdd(&s_updates, n);
      }
    }
  }
  const bool bounded = kBatched && l.waveItems > 0;
  DealtItems dealt{};
  __shared__ int s_taken;  // bounded launches: items of the workgroup taken so far
  int begin = !kFastMath && !kBatched ? first_after_core(l, number, claimed) : number;
  if (bounded) {
    dealt = deal_items(l, kWaves);
    if (threadIdx.x == 0) s_taken = kWaves;
    __syncthreads();
    begin = dealt_item(l, dealt, __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)));
  }
  for (int b = begin; b < l.nItems;
       b = bounded ? next_dealt(l, dealt, &s_taken, lane) : claim_item(l, lane, claimed)) {
    const int4 bo = make_uniform(reinterpret_cast<const int4 *>(l.items)[b]);
    // work item: brick 8 x 8 x depth at (bo.x, bo.y, bo.z & 0xffff) of job bo.z >> 16; heavy
    // bricks run at raised wave priority; a brick split into `parts` slice ranges accumulates
    // its range from zero and merges the partial sums with atomics (fast-math schedules only)
    const FrJob a = kBatched ? global_pointers(make_uniform(l.jobs[bo.z >> 16])) : job0;
    const int s0 = a.spaceBegin, s1 = a.spaceEnd;
    if (s0 >= s1) continue;
    const bool heavy = (bo.w >> 4) & 1;
    const int parts = (bo.w >> 8) & 255, part = (bo.w >> 16) & 255;
    const bool split = parts > 1;
    const int sBegin = split ? s0 + (int)((int64_t)(s1 - s0) * part / parts) : s0;
    const int sEnd = split ? s0 + (int)((int64_t)(s1 - s0) * (part + 1) / parts) : s1;
    const umpa_fr_constants &c = a.c;
    const int cxi = c.cMaxVolumeIndexX / 2, cyi = c.cMaxVolumeIndexYZ / 2;
    // phase-1 filter on the slab coordinate: the reference's own test for blobs; for the
    // nearest-neighbour traversal the visited voxel lies within 1.5 of the plane
    const float slab = kMode == kModeNearest ? 1.6f : c.cBlobRadius;
    if (heavy) __builtin_amdgcn_s_setprio(2);
    // the lane owns the z column (x, y, z0 .. z0 + depth - 1) of the brick
    const BrickCtx bk = make_brick(a, bo, lane);
    const float usual = bk.colIn ? slab_reach(slab, a.vz, kUsualT22) : -1.f;
    const int bz = bk.z0;
    const float ox = (float)(bo.x - cxi), oy = (float)(bo.y - cyi), oz = (float)(bz - cyi);
    bool loaded = false;  // the sums are read when the first space reaches the brick
    // wave-uniform: the brick's distance from the centre
    const bool earlyCull = __builtin_amdgcn_readfirstlane((int)(bk.dmin > kEarlyCullRadius)) != 0;
    unsigned long long nupd = 0;
    for (int base = sBegin; base < sEnd; base += 64) {
      float t22;
      unsigned long long mask = earlyCull
                                  ? __ballot(cull_space<true>(a, bk, base + lane, sEnd, t22))
                                  : __ballot(cull_space<false>(a, bk, base + lane, sEnd, t22));
      const float lim = slab_limit<kNB <= 4>(usual, a, bk, slab, t22);
      if (mask && !loaded) {
        load_brick(ws, a, bk, lane, split);
        loaded = true;
      }
      // the space's record goes through the wave's LDS slot: one load of 28 dwords by 28
      // lanes, then broadcast reads, instead of seven 16-byte loads of one address by every
      // lane (its 28 SGPRs would not fit beside this kernel's other scalar state). The next
      // surviving space's dword is loaded while the current space is processed.
      constexpr int kRecDwords = (int)(sizeof(umpa_traverse_space) / 4);
      const bool recLane = lane < kRecDwords;
      int rec = 0;
      if (mask && recLane)
        rec = reinterpret_cast<const int *>(
          a.spaces + __builtin_amdgcn_readfirstlane(base + __builtin_ctzll(mask)))[lane];
      while (mask) {
        mask &= mask - 1;
        if (recLane) reinterpret_cast<int *>(&s_space[threadIdx.x >> 6])[lane] = rec;
        wave_sync();
        if (mask && recLane)
          rec = reinterpret_cast<const int *>(
            a.spaces + __builtin_amdgcn_readfirstlane(base + __builtin_ctzll(mask)))[lane];
        const umpa_traverse_space &sp = s_space[threadIdx.x >> 6];
        const int proj = __builtin_amdgcn_readfirstlane(sp.projectionIndex);
        const int64_t off = (int64_t)proj * a.sliceElems * kPix;
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
          (void *)((const char *)a.fft + off), 0, (int)(a.sliceElems * kPix), kBufferConfig);
        const float scale = kHalf ? a.scales[proj] : 1.f;

        // phase 1: slab test of the column's nz voxels (nz is wave-uniform: shallow bricks
        // run fewer levels)
        const int cnt = slab_queue(ws, a, bk, sp, lim, lane);
        if (cnt == 0) continue;
        wave_sync();
        const bool unit = sp.weight == 1.f;
        const bool inside = brick_inside(bk, sp, cxi, cyi);

        // phase 2: the rest of the predicate and the gather, with full lanes
        for (int t0 = 0; t0 < cnt; t0 += 64) {
          const int item = t0 + lane;
          const bool act = item < cnt;
          const int v = act ? (int)ws.queue[item] : 0;
          const int vl = v & 63, vk = v >> 6;
          const int xv = bo.x + (vl & (kEdge - 1)), yv = bo.y + vl / kEdge, zv = bz + vk;
          // small integers in float: exact however they are summed
          const float pxv = (float)(vl & (kEdge - 1)) + ox, pyv = (float)(vl / kEdge) + oy,
                      pzv = (float)vk + oz;
          float qx, qy, zs;
          bool hit;
          if constexpr (kMode == kModeNearest) {
            const float dsq = pxv * pxv + pyv * pyv + pzv * pzv;
            qx = sp.transformInv[0][0] * pxv + sp.transformInv[0][1] * pyv + sp.transformInv[0][2] * pzv;
            qy = sp.transformInv[1][0] * pxv + sp.transformInv[1][1] * pyv + sp.transformInv[1][2] * pzv;
            zs = 0.f;
            hit = act && !(dsq > sp.maxDistanceSqr) && !(qx < 0.f) && visited_nearest(sp, xv, yv, zv);
          } else {
            hit = act && blob_predicate<false>(sp, sp.transformInv, c, xv, yv, zv, pxv, pyv, pzv, inside, qx, qy, zs);
          }
          Contribution o;
          if constexpr (evaluates_blob(kMode))
            o = gather_evaluated<kMode, kOrder>(a, rsrc, s_blob[threadIdx.x >> 6], lane, hit, qx, qy,
                                                zs, sp.weight);
          if (hit) {
            if constexpr (evaluates_blob(kMode)) {
              // gathered above, by the whole wavefront
            } else if constexpr (kMode == kModeNearest) {
              o = gather_nearest<kHalf>(a, rsrc, qx, qy, sp.weight, scale);
            } else {
              o = gather_update<kMode, kOrder, kNB, kHalf, kFastMath, kTableLds, kShift, false>(
                a, nTable, rsrc, tbl, qx, qy, zs, sp.weight, unit, scale);
            }
            // volume += contribution, in space order (one item per voxel per space)
            ws.accR[v] = ws.accR[v] + o.re;
            ws.accI[v] = ws.accI[v] + o.im;
            ws.accW[v] = ws.accW[v] + o.w;
          }
          if constexpr (kCount) nupd += (unsigned long long)__popcll(__ballot(hit));
        }
        wave_sync();
      }
    }
    if (loaded) store_brick(ws, a, bk, lane, split);
    if (heavy) __builtin_amdgcn_s_setprio(0);
    if constexpr (kCount) {
      if (lane == 0 && nupd) atomicAdd(&s_updates, nupd);
    }
  }
  if constexpr (kCount) {
    __syncthreads();
    if (threadIdx.x == 0 && s_updates) atomicAdd(l.updates, s_updates);
  }
}

// ---- fast-math lookup insertion with queues carried across spaces ---------------------------
//
// fr_insert_kernel gathers each (brick, space) queue 64 voxels at a time, so the last batch of
// every pair runs partly empty.  This variant (fast math, FP32 or FP16 slices, table in LDS,
// 16 wavefronts per CU) lets the slab voxels of consecutive spaces share one queue: a space's
// voxels are appended behind the ones left from the previous spaces, every full batch of 64 is
// gathered as soon as it forms, and a partial batch runs only at the end of a brick or when a
// third space would be pending.  An entry carries the slot (0 / 1) of its space's record, so a
// batch holds at most two spaces; it adds their contributions space by space, the earlier one
// first (no voxel appears twice within one space), so every voxel still receives its spaces in
// index order and the sums are the ones fr_insert_kernel forms.  All slices of the chunk are
// read through one buffer resource (chunks up to 2 GiB of slices).
constexpr int kCarryQueue = kVox + 64;  // leftovers (< 64) plus one space's slab voxels

struct CarrySlot {
  umpa_traverse_space rec;
  uint32_t sliceOff;  // byte offset of the space's slice in the chunk
  float scale;        // FP16 dequantisation factor of that slice
  int inside;         // brick_inside() of the brick and this space
  uint32_t pad;
};
static_assert(sizeof(CarrySlot) == 128, "two slots per wave");

struct CarryScratch {
  float accR[kVox];
  float accI[kVox];
  float accW[kVox];
  uint16_t queue[kCarryQueue];  // voxel index (bits 0-8) | slot (bit 9)
};

// Largest blob table the carry kernel keeps in LDS beside its per-wave state (batched: and beside
// the count of taken items).
constexpr int carry_max_table(bool batched)
{
  return (160 * 1024 - kMaxWaves * (int)(sizeof(CarryScratch) + 2 * sizeof(CarrySlot)) -
          (batched ? 16 : 0)) / 4 - 1;
}

// One batch of `n` (1..64) queue entries from `start`: the rest of the predicate, the gather and
// the accumulation, space by space.
template <int kNB, bool kHalf, bool kCount, bool kShift>
__device__ __forceinline__ void carry_batch(CarryScratch &ws, const CarrySlot *slots,
                                            const FrJob &a, const int4 &bo, int bz, int nTable,
                                            __amdgpu_buffer_rsrc_t rsrc, const float *tbl,
                                            int lane, int start, int n,
                                            unsigned long long &nupd)
{
  const umpa_fr_constants &c = a.c;
  const int cxi = c.cMaxVolumeIndexX / 2, cyi = c.cMaxVolumeIndexYZ / 2;
  const bool act = lane < n;
  const uint32_t e = act ? (uint32_t)ws.queue[start + lane] : 0u;
  const int v = (int)(e & 511u), tag = (int)(e >> 9);
  const CarrySlot &slt = slots[tag];
  const umpa_traverse_space &sp = slt.rec;
  const int vl = v & 63, vk = v >> 6;
  const int xv = bo.x + (vl & (kEdge - 1)), yv = bo.y + vl / kEdge, zv = bz + vk;
  // small integers in float: exact however they are summed
  const float pxv = (float)(vl & (kEdge - 1)) + (float)(bo.x - cxi),
              pyv = (float)(vl / kEdge) + (float)(bo.y - cyi), pzv = (float)vk + (float)(bz - cyi);
  float qx, qy, zs;
  const bool hit =
    act && blob_predicate<false>(sp, sp.transformInv, c, xv, yv, zv, pxv, pyv, pzv, slt.inside != 0, qx, qy, zs);
  Contribution o{ 0.f, 0.f, 0.f };
  if (hit) {
    o = gather_update<kModeLookup, 0, kNB, kHalf, true, true, kShift, true>(
      a, nTable, rsrc, tbl, qx, qy, zs, sp.weight, false, slt.scale, slt.sliceOff);
  }
  // lane 0 holds the batch's oldest entry: its space is added first
  const int first = __builtin_amdgcn_readfirstlane(tag);
  if (hit && tag == first) {
    ws.accR[v] = ws.accR[v] + o.re;
    ws.accI[v] = ws.accI[v] + o.im;
    ws.accW[v] = ws.accW[v] + o.w;
  }
  if (__any(hit && tag != first)) {
    wave_sync();
    if (hit && tag != first) {
      ws.accR[v] = ws.accR[v] + o.re;
      ws.accI[v] = ws.accI[v] + o.im;
      ws.accW[v] = ws.accW[v] + o.w;
    }
  }
  if constexpr (kCount) nupd += (unsigned long long)__popcll(__ballot(hit));
}

template <int kNB, bool kHalf, bool kCount, bool kBatched, bool kShift>
__global__ __launch_bounds__(64 * kMaxWaves) void fr_insert_carry_kernel(FrJob job0, FrLaunch l)
{
  constexpr int kWaves = kMaxWaves;
  constexpr int kThreads = 64 * kWaves;
  constexpr int kPix = kHalf ? 4 : 8;
  extern __shared__ float s_table[];
  __shared__ CarryScratch s_wave[kWaves];
  __shared__ CarrySlot s_slot[kWaves][2];
  const int nTable = l.nTable;
  stage_table<kThreads>(s_table, l.table, nTable);
  const float *tbl = s_table;
  const int lane = threadIdx.x & 63;
  const int wv = threadIdx.x >> 6;
  CarryScratch &ws = s_wave[wv];
  CarrySlot *slots = s_slot[wv];

  const int number = wave_number(), claimed = kWaves * (int)gridDim.x;
  const bool bounded = kBatched && l.waveItems > 0;
  DealtItems dealt{};
  __shared__ int s_taken;  // bounded launches: items of the workgroup taken so far
  int begin = number;
  if (bounded) {
    dealt = deal_items(l, kWaves);
    if (threadIdx.x == 0) s_taken = kWaves;
    __syncthreads();
    begin = dealt_item(l, dealt, __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)));
  }
  for (int b = begin; b < l.nItems;
       b = bounded ? next_dealt(l, dealt, &s_taken, lane) : claim_item(l, lane, claimed)) {
    const int4 bo = make_uniform(reinterpret_cast<const int4 *>(l.items)[b]);
    const FrJob a = kBatched ? global_pointers(make_uniform(l.jobs[bo.z >> 16])) : job0;
    const int s0 = a.spaceBegin, s1 = a.spaceEnd;
    if (s0 >= s1) continue;
    const bool heavy = (bo.w >> 4) & 1;
    const int parts = (bo.w >> 8) & 255, part = (bo.w >> 16) & 255;
    const bool split = parts > 1;
    const int sBegin = split ? s0 + (int)((int64_t)(s1 - s0) * part / parts) : s0;
    const int sEnd = split ? s0 + (int)((int64_t)(s1 - s0) * (part + 1) / parts) : s1;
    const int cxi = a.c.cMaxVolumeIndexX / 2, cyi = a.c.cMaxVolumeIndexYZ / 2;
    if (heavy) __builtin_amdgcn_s_setprio(2);
    const BrickCtx bk = make_brick(a, bo, lane);
    const float usual = bk.colIn ? slab_reach(a.c.cBlobRadius, a.vz, kUsualT22) : -1.f;
    const int bz = bk.z0;
    // (read before the cull, reached or not; only a brick that a space reaches is written back)
    load_brick(ws, a, bk, lane, split);
    bool loaded = false;
    const uint32_t sliceBytes = (uint32_t)(a.sliceElems * kPix);
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void *)a.fft, 0, (int)((uint32_t)a.nProj * sliceBytes), kBufferConfig);
    const bool earlyCull = __builtin_amdgcn_readfirstlane((int)(bk.dmin > kEarlyCullRadius)) != 0;
    unsigned long long nupd = 0;
    int pending = 0;     // queue entries waiting, queue[0 .. pending)
    int pendSpaces = 0;  // spaces they come from (at most 2)
    int slot = 0;        // record slot of the next space
    for (int base = sBegin; base < sEnd; base += 64) {
      float t22;
      unsigned long long mask = earlyCull
                                  ? __ballot(cull_space<true>(a, bk, base + lane, sEnd, t22))
                                  : __ballot(cull_space<false>(a, bk, base + lane, sEnd, t22));
      const float lim = slab_limit<true>(usual, a, bk, a.c.cBlobRadius, t22);
      if (mask && !loaded) {
        loaded = true;
      }
      constexpr int kRecDwords = (int)(sizeof(umpa_traverse_space) / 4);
      const bool recLane = lane < kRecDwords;
      int rec = 0;
      if (mask && recLane)
        rec = reinterpret_cast<const int *>(
          a.spaces + __builtin_amdgcn_readfirstlane(base + __builtin_ctzll(mask)))[lane];
      while (mask) {
        mask &= mask - 1;
        if (pendSpaces == 2) {
          // the slot about to be rewritten still holds a pending space: gather everything
          wave_sync();
          carry_batch<kNB, kHalf, kCount, kShift>(ws, slots, a, bo, bz, nTable, rsrc, tbl, lane, 0,
                                          pending, nupd);
          pending = 0;
          pendSpaces = 0;
          wave_sync();
        }
        const int proj = __builtin_amdgcn_readlane(rec, 17);  // projectionIndex (byte 68)
        if (recLane) reinterpret_cast<int *>(&slots[slot])[lane] = rec;
        if (lane == kRecDwords) slots[slot].sliceOff = (uint32_t)proj * sliceBytes;
        if (lane == kRecDwords + 1) slots[slot].scale = kHalf ? a.scales[proj] : 1.f;
        wave_sync();
        if (mask && recLane)
          rec = reinterpret_cast<const int *>(
            a.spaces + __builtin_amdgcn_readfirstlane(base + __builtin_ctzll(mask)))[lane];
        const bool ins = brick_inside(bk, slots[slot].rec, cxi, cyi);
        if (lane == 0) slots[slot].inside = ins ? 1 : 0;
        const int cnt =
          slab_queue(ws, a, bk, slots[slot].rec, lim, lane, pending, (uint32_t)slot << 9);
        if (cnt == 0) continue;  // the slot stays free for the next space
        pending += cnt;
        ++pendSpaces;
        slot ^= 1;
        wave_sync();
        const int full = pending >> 6;
        if (full) {
          for (int t = 0; t < full; ++t)
            carry_batch<kNB, kHalf, kCount, kShift>(ws, slots, a, bo, bz, nTable, rsrc, tbl, lane,
                                            t * 64, 64, nupd);
          // the leftovers (< 64, all of the space just queued) move to the queue's front
          const int left = pending - (full << 6);
          const int x = lane < left ? (int)ws.queue[(full << 6) + lane] : 0;
          wave_sync();
          if (lane < left) ws.queue[lane] = (uint16_t)x;
          pending = left;
          pendSpaces = left ? 1 : 0;
        }
        wave_sync();
      }
    }
    if (pending) {
      carry_batch<kNB, kHalf, kCount, kShift>(ws, slots, a, bo, bz, nTable, rsrc, tbl, lane, 0, pending,
                                      nupd);
      wave_sync();
    }
    if (loaded) store_brick(ws, a, bk, lane, split);
    if (heavy) __builtin_amdgcn_s_setprio(0);
    if constexpr (kCount) {
      if (lane == 0 && nupd) atomicAdd(l.updates, nupd);
    }
  }
}

// ---- exact FP32 lookup insertion with cross-space gather batches -----------------------------
//
// In fr_insert_kernel a space's queue of slab voxels is gathered 64 at a time, so the last,
// partly filled batch of every (brick, space) pair leaves lanes idle: two thirds of the gather
// lanes do work at box 256.  This variant, for the exact strategy with the table in LDS (the
// one with LDS to spare at 12 wavefronts per CU), evaluates the predicate per space as before
// but appends the hits (voxel, space ordinal, q, slice offset, weight) to a per-wave ring in
// LDS and gathers whenever 64 are waiting, across spaces.  All slices are read through one
// buffer resource over the chunk.  A voxel still receives its contributions in space order:
// entries are appended in space order, and a batch adds its contributions space by space.
constexpr int kStagedWaves = 12;
constexpr int kStage = 128;  // ring entries per wave: a full batch plus one space's hits
// largest table the staged kernel's LDS holds beside its per-wave state (160 KiB in all)
constexpr int kStagedMaxTable =
  (160 * 1024 - kStagedWaves * (int)(sizeof(WaveScratch) + 6 * 4 * kStage)) / 4 - 1;

struct WaveStage {
  float qx[kStage], qy[kStage], zs[kStage], dw[kStage];
  uint32_t off[kStage];  // byte offset of the entry's slice in the chunk
  uint32_t key[kStage];  // voxel index in the brick (bits 0-15), space ordinal (bits 16-31)
};

template <int kNB, bool kShift>
__device__ __forceinline__ void staged_gather(const FrJob &a, int nTable,
                                              __amdgpu_buffer_rsrc_t rsrc, const float *tbl,
                                              WaveScratch &ws, const WaveStage &st, int lane,
                                              int head, int n)
{
  const int e = (head + lane) & (kStage - 1);
  const bool act = lane < n;
  const float qx = act ? st.qx[e] : 0.f, qy = act ? st.qy[e] : 0.f, zs = act ? st.zs[e] : 0.f;
  const float dw = act ? st.dw[e] : 1.f;
  const uint32_t off = act ? st.off[e] : 0u, key = act ? st.key[e] : 0u;
  Contribution o{ 0.f, 0.f, 0.f };
  if (act) {
    o = gather_update<kModeLookup, 0, kNB, false, false, true, kShift, true>(
      a, nTable, rsrc, tbl, qx, qy, zs, dw, __all(dw == 1.f), 1.f, off);
  }
  // add space by space (the lowest remaining lane holds the earliest space): within a space
  // every voxel appears once
  unsigned long long rem = __ballot(act);
  while (rem) {
    const int first = __builtin_ctzll(rem);
    const uint32_t ord = (uint32_t)__builtin_amdgcn_readlane((int)(key >> 16), first);
    const unsigned long long m = __ballot(act && (key >> 16) == ord) & rem;
    if ((m >> lane) & 1ull) {
      const int v = (int)(key & 0xffffu);
      ws.accR[v] = ws.accR[v] + o.re;
      ws.accI[v] = ws.accI[v] + o.im;
      ws.accW[v] = ws.accW[v] + o.w;
    }
    rem &= ~m;
  }
}

// kShift: the job's candidate boxes slide inside the slice (FrJob::shiftBox), a separate
// instantiation: decided per candidate at run time, the choice made the compiler reschedule the
// kernel (116 -> 83 VGPRs, 1.49 -> 1.92 ms per 1,000-slice chunk at box 256); as its own
// instantiation the sliding box takes the chunk from 1.502 to 1.445 ms, bit for bit the same.
template <int kNB, bool kShift>
__global__ __launch_bounds__(64 * kStagedWaves) void fr_insert_staged_kernel(FrJob a, FrLaunch l)
{
  constexpr int kWaves = kStagedWaves;
  constexpr int kThreads = 64 * kWaves;
  constexpr int kPix = 8;
  extern __shared__ float s_table[];
  __shared__ WaveScratch s_wave[kWaves];
  __shared__ WaveStage s_stage[kWaves];
  const int nTable = l.nTable;
  stage_table<kThreads>(s_table, l.table, nTable);
  const float *tbl = s_table;
  const int lane = threadIdx.x & 63;
  WaveScratch &ws = s_wave[threadIdx.x >> 6];
  WaveStage &st = s_stage[threadIdx.x >> 6];
  // one resource over the chunk's slices (the host keeps it under 2 GiB)
  const uint32_t sliceBytes = (uint32_t)(a.sliceElems * kPix);
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
    (void *)a.fft, 0, (int)((uint32_t)a.nProj * sliceBytes), kBufferConfig);
  const umpa_fr_constants &c = a.c;
  const int cxi = c.cMaxVolumeIndexX / 2, cyi = c.cMaxVolumeIndexYZ / 2;

  const int sBegin = a.spaceBegin, sEnd = a.spaceEnd;
  if (sBegin >= sEnd) return;
  const int number = wave_number(), claimed = kWaves * (int)gridDim.x;
  // the volume's core, cell by cell (a loop of its own: as a branch of the brick loop it cost that
  // loop's schedule 4 %)
  for (int b = number; b < l.nCore; b += claimed) {
    const int2 bo = uniform_load(reinterpret_cast<const int2 *>(l.core), b);
    unsigned long long none = 0;
    cell_item<kModeLookup, 0, kNB, true, kShift, false>(
      a, bo.x & 0xffff, bo.x >> 16, bo.y, sBegin, sEnd,
      reinterpret_cast<uint32_t *>(ws.queue), ws.accR, ws.accI, nTable, rsrc, tbl, lane, none);
  }

  // wavefronts with a cell of the core start on the lighter of the first bricks
  for (int b = first_after_core(l, number, claimed); b < l.nItems;) {
    const int4 bo = uniform_load(reinterpret_cast<const int4 *>(l.items), b);
    // work item: brick 8 x 8 x depth at (bo.x, bo.y, bo.z); the exact schedules never split
    const bool heavy = (bo.w >> 4) & 1;
    if (heavy) __builtin_amdgcn_s_setprio(2);
    const BrickCtx bk = make_brick(a, bo, lane);
    const float usual = bk.colIn ? slab_reach(c.cBlobRadius, a.vz, kUsualT22) : -1.f;
    const int bz = bk.z0;
    const float ox = (float)(bo.x - cxi), oy = (float)(bo.y - cyi), oz = (float)(bz - cyi);
    bool loaded = false;  // the sums are read when the first space reaches the brick
    // wave-uniform: the brick's distance from the centre
    const bool earlyCull = __builtin_amdgcn_readfirstlane((int)(bk.dmin > kEarlyCullRadius)) != 0;
    int head = 0, waiting = 0;  // the ring's oldest entry and its number of entries
    uint32_t ordinal = 0;       // spaces taken so far by this work item (mod 2^16)
    for (int base = sBegin; base < sEnd; base += 64) {
      float t22;
      unsigned long long mask = earlyCull
                                  ? __ballot(cull_space<true>(a, bk, base + lane, sEnd, t22))
                                  : __ballot(cull_space<false>(a, bk, base + lane, sEnd, t22));
      const float lim = slab_limit<true>(usual, a, bk, c.cBlobRadius, t22);
      if (mask && !loaded) {
        load_brick(ws, a, bk, lane, false);
        loaded = true;
      }
      while (mask) {
        const int k0 = __builtin_ctzll(mask);
        mask &= mask - 1;
        const umpa_traverse_space sp =
          uniform_load(a.spaces, __builtin_amdgcn_readfirstlane(base + k0));
        const uint32_t sliceOff =
          (uint32_t)__builtin_amdgcn_readfirstlane(sp.projectionIndex) * sliceBytes;
        // phase 1: the slab test, as in fr_insert_kernel
        const int cnt = slab_queue(ws, a, bk, sp, lim, lane);
        if (cnt == 0) continue;
        wave_sync();
        const bool inside = brick_inside(bk, sp, cxi, cyi);
        // phase 2: the rest of the predicate; hits go to the ring, gathered 64 at a time
        for (int t0 = 0; t0 < cnt; t0 += 64) {
          const int item = t0 + lane;
          const bool act = item < cnt;
          const int v = act ? (int)ws.queue[item] : 0;
          const int vl = v & 63, vk = v >> 6;
          const int xv = bo.x + (vl & (kEdge - 1)), yv = bo.y + vl / kEdge, zv = bz + vk;
          // small integers in float: exact however they are summed
          const float pxv = (float)(vl & (kEdge - 1)) + ox, pyv = (float)(vl / kEdge) + oy,
                      pzv = (float)vk + oz;
          float qx, qy, zs;
          const bool hit =
            act && blob_predicate<false>(sp, sp.transformInv, c, xv, yv, zv, pxv, pyv, pzv, inside, qx, qy, zs);
          const unsigned long long hm = __ballot(hit);
          if (hit) {
            const int e = (head + waiting + (int)lanes_below(hm)) & (kStage - 1);
            st.qx[e] = qx;
            st.qy[e] = qy;
            st.zs[e] = zs;
            st.dw[e] = sp.weight;
            st.off[e] = sliceOff;
            st.key[e] = (uint32_t)v | (ordinal << 16);
          }
          waiting += __popcll(hm);
          if (waiting >= 64) {
            wave_sync();
            staged_gather<kNB, kShift>(a, nTable, rsrc, tbl, ws, st, lane, head, 64);
            wave_sync();
            head = (head + 64) & (kStage - 1);
            waiting -= 64;
          }
        }
        ordinal = (ordinal + 1) & 0xffffu;
        wave_sync();
      }
    }
    if (waiting > 0) {
      wave_sync();
      staged_gather<kNB, kShift>(a, nTable, rsrc, tbl, ws, st, lane, head, waiting);
      wave_sync();
    }
    if (loaded) store_brick(ws, a, bk, lane, false);
    if (heavy) __builtin_amdgcn_s_setprio(0);
    b = claim_item(l, lane, claimed);
  }
}

// ---- host-side dispatch ------------------------------------------------------------------
// The kernel is instantiated per (mode, order, footprint width, FP16, fast math, counting, LDS
// table, batched); `visit` calls `f` with a pointer to the instantiation a variant selects.
template <int kMode, int kOrder, int kNB, bool kHalf, bool kFastMath, bool kCount, bool kShift>
static const void *pick_lds(bool lds, bool batched)
{
  // batches with a lookup table keep it in LDS (tables up to kMaxLdsTable samples)
  if constexpr (kMode == kModeLookup) {
    if (batched && !lds) return nullptr;
    if (batched) return (const void *)fr_insert_kernel<kMode, kOrder, kNB, kHalf, kFastMath, kCount, true, true, kShift>;
  }
  if (lds) return (const void *)fr_insert_kernel<kMode, kOrder, kNB, kHalf, kFastMath, kCount, true, false, kShift>;
  return batched ? (const void *)fr_insert_kernel<kMode, kOrder, kNB, kHalf, kFastMath, kCount, false, true, kShift>
                 : (const void *)fr_insert_kernel<kMode, kOrder, kNB, kHalf, kFastMath, kCount, false, false, kShift>;
}

// The sliding box (FrJob::shiftBox, every job of the launch) is an instantiation of its own for
// the fast-math kernels: tested per gather at run time, it cost 2-3 % (fast math 1.229 against
// 1.251 ms, FP16 1.189 against 1.222 ms per 1,000-slice chunk at box 256).
template <int kMode, int kOrder, int kNB, bool kHalf, bool kFastMath, bool kCount>
static const void *pick_shift(bool lds, bool batched, bool shift)
{
  if constexpr (kFastMath) {
    if (shift) return pick_lds<kMode, kOrder, kNB, kHalf, kFastMath, kCount, true>(lds, batched);
  }
  return pick_lds<kMode, kOrder, kNB, kHalf, kFastMath, kCount, false>(lds, batched);
}

template <int kMode, int kOrder, bool kHalf, bool kFastMath, bool kCount>
static const void *pick_nb(int nb, bool lds, bool batched, bool shift)
{
  switch (nb) {
  case 3: return pick_shift<kMode, kOrder, 3, kHalf, kFastMath, kCount>(lds, batched, shift);
  case 4: return pick_shift<kMode, kOrder, 4, kHalf, kFastMath, kCount>(lds, batched, shift);
  case 5: return pick_shift<kMode, kOrder, 5, kHalf, kFastMath, kCount>(lds, batched, shift);
  default: return pick_shift<kMode, kOrder, 6, kHalf, kFastMath, kCount>(lds, batched, shift);
  }
}

// Precise Kaiser (kDynamic, alpha > 15): one instantiation per blob order
// (fr_common_kernels.hpp:129-161); orders outside 0..4 are rejected at Init.
template <bool kCount>
static const void *pick_order(int order, bool batched)
{
  switch (order) {
  case 0: return pick_lds<kModePreciseKaiser, 0, 4, false, false, kCount, false>(false, batched);
  case 1: return pick_lds<kModePreciseKaiser, 1, 4, false, false, kCount, false>(false, batched);
  case 2: return pick_lds<kModePreciseKaiser, 2, 4, false, false, kCount, false>(false, batched);
  case 3: return pick_lds<kModePreciseKaiser, 3, 4, false, false, kCount, false>(false, batched);
  case 4: return pick_lds<kModePreciseKaiser, 4, 4, false, false, kCount, false>(false, batched);
  default: return nullptr;
  }
}

static bool table_in_lds(const FrVariant &v, int nTable)
{
  return v.mode == kModeLookup && nTable <= kMaxLdsTable && !(v.tableGlobal && !v.batched);
}

static const void *pick_kernel(const FrVariant &v, int nTable)
{
  const bool lds = table_in_lds(v, nTable);
  const bool b = v.batched;
  switch (v.mode) {
  case kModeLookup:
    if (v.count) {
      if (v.half) return pick_nb<kModeLookup, 0, true, true, true>(v.nb, lds, b, v.shift);
      return v.fastMath ? pick_nb<kModeLookup, 0, false, true, true>(v.nb, lds, b, v.shift)
                        : pick_nb<kModeLookup, 0, false, false, true>(v.nb, lds, b, v.shift);
    }
    if (v.half) return pick_nb<kModeLookup, 0, true, true, false>(v.nb, lds, b, v.shift);
    if (v.fastMath) return pick_nb<kModeLookup, 0, false, true, false>(v.nb, lds, b, v.shift);
    return pick_nb<kModeLookup, 0, false, false, false>(v.nb, lds, b, v.shift);
  case kModeFastKaiser:
    return v.count ? pick_lds<kModeFastKaiser, 0, 4, false, false, true, false>(false, b)
                   : pick_lds<kModeFastKaiser, 0, 4, false, false, false, false>(false, b);
  case kModeNearest:
    return v.count ? pick_lds<kModeNearest, 0, 4, false, false, true, false>(false, b)
                   : pick_lds<kModeNearest, 0, 4, false, false, false, false>(false, b);
  case kModePreciseKaiser:
    // the counting variant evaluates the same blob order as the plain one
    return v.count ? pick_order<true>(v.order, b) : pick_order<false>(v.order, b);
  default: return nullptr;
  }
}

// The exact FP32 lookup kernel with cross-space gather batches, for the variants it covers
// (the launch also needs the chunk's slices under 2 GiB, one buffer resource).
static const void *pick_staged(const FrVariant &v, int nTable, bool shift)
{
  if (v.mode != kModeLookup || v.half || v.fastMath || v.count || v.batched) return nullptr;
  if (!table_in_lds(v, nTable) || nTable > kStagedMaxTable) return nullptr;
  if (v.nb == 3) return shift ? (const void *)fr_insert_staged_kernel<3, true>
                              : (const void *)fr_insert_staged_kernel<3, false>;
  if (v.nb == 4) return shift ? (const void *)fr_insert_staged_kernel<4, true>
                              : (const void *)fr_insert_staged_kernel<4, false>;
  return nullptr;
}

static bool staged_fits(const FrJob &job)
{
  return (uint64_t)job.nProj * (uint64_t)job.sliceElems * 8u <= 0x7fff0000ull;
}

// The fast-math kernel with queues carried across spaces, for the variants it covers (the
// launch also needs the chunk's slices under 2 GiB, one buffer resource).
static const void *pick_carry(const FrVariant &v, int nTable)
{
  if (v.mode != kModeLookup || !v.fastMath) return nullptr;
  if (!table_in_lds(v, nTable) || nTable > carry_max_table(v.batched)) return nullptr;
  if (v.nb != 3 && v.nb != 4) return nullptr;
#define UMPA_CARRY(NB, H, B)                                                                 \
  (v.shift ? (v.count ? (const void *)fr_insert_carry_kernel<NB, H, true, B, true>           \
                      : (const void *)fr_insert_carry_kernel<NB, H, false, B, true>)         \
           : (v.count ? (const void *)fr_insert_carry_kernel<NB, H, true, B, false>          \
                      : (const void *)fr_insert_carry_kernel<NB, H, false, B, false>))
  if (v.batched) {
    if (v.half) return v.nb == 3 ? UMPA_CARRY(3, true, true) : UMPA_CARRY(4, true, true);
    return v.nb == 3 ? UMPA_CARRY(3, false, true) : UMPA_CARRY(4, false, true);
  }
  if (v.half) return v.nb == 3 ? UMPA_CARRY(3, true, false) : UMPA_CARRY(4, true, false);
  return v.nb == 3 ? UMPA_CARRY(3, false, false) : UMPA_CARRY(4, false, false);
#undef UMPA_CARRY
}

static bool carry_fits(const FrJob &job, bool half)
{
  return (uint64_t)job.nProj * (uint64_t)job.sliceElems * (half ? 4u : 8u) <= 0x7fff0000ull;
}

hipError_t prepare_fr_insert(const FrVariant &v, int nTable)
{
  if (!pick_kernel(v, nTable)) return hipErrorInvalidValue;
  if (!table_in_lds(v, nTable)) return hipSuccess;
  const int bytes = (int)((nTable + 1) * sizeof(float));
  hipError_t e = hipSuccess;
  // every kernel the launch may pick: either box form (a plain launch takes it from its job)
  for (bool shift : { false, true }) {
    FrVariant w = v;
    w.shift = shift;
    for (const void *k : { pick_kernel(w, nTable), pick_staged(w, nTable, shift),
                           pick_carry(w, nTable) })
      if (e == hipSuccess && k)
        e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  }
  return e;
}

// Does this launch run the small-problem kernel?  The brick kernels take a space per 0.3 to 1.2 us
// (their heaviest brick's chain) whatever the volume, the cell kernel a fixed 4 us per round of
// blocks and less per space.  Measured (us, bricks / cells at r 1.9, slices): exact, box 64 60
// 50 / 48, 150 92 / 63; 80 60 55 / 67, 150 87 / 78, 400 167 / 144, 1,200 442 / 365; 90 150 90 / 96,
// 400 149 / 171; 100 400 172 / 198; r 1.5 90 150 79 / 85, 1,200 368 / 330; 100 1,200 405 / 387, 112
// 390 / 464; r 2.5 100 150 228 / 186, 112 150 202 / 233, 1,200 1165 / 1101, 128 1218 / 1398.  Fast
// math: 64 60 73 / 47; 80 60 58 / 65, 150 89 / 75; 100 150 102 / 104, 400 188 / 179, 1,200 482 /
// 462; 112 400 189 / 211; FP16 100 1,200 554 / 433, 112 400 206 / 201, 1,200 541 / 514; 128 400 198 /
// 253, six columns 96 1,000 r 3.6 3667 / 3208, r 3 811 / 1035, 112 3618 / 3991, 776 / 1100, r 5 6819 /
// 9500.  Blob evaluated: 80 60 106 / 75, 100 60 114 / 117, 150 192 / 152; 112 60 127 / 146, 150 196 /
// 188, 400 392 / 334; 128 150 198 / 247.  Nearest: 64 150 62 / 54, 80 150 60 / 65, 1,200 485 / 351;
// 90 414 / 430.  So, with V the volume's mean extent: from (V - from) * slope spaces, up to a V.
bool use_cells(const FrJob &job, const FrLaunch &l, const FrVariant &v)
{
  if (l.nCells <= 0 || v.batched || v.count || v.kernel != kKernelAuto || v.tableGlobal) return false;
  if (v.mode == kModeLookup && l.nTable > kMaxLdsTable) return false;  // the table stays global
  if (!carry_fits(job, v.half)) return false;  // the chunk's slices need one buffer resource each
  struct Rule {
    int upTo;
    float from, slope;
  };
  const Rule rule = v.mode == kModeNearest  ? Rule{ 85, 45.f, 4.f }
                    : v.mode != kModeLookup ? Rule{ 121, 85.f, 5.f }
                    : v.half && v.nb == 6   ? Rule{ 97, 55.f, 5.f }
                    : v.half                ? Rule{ 115, 55.f, 5.f }
                    : v.fastMath            ? Rule{ 105, 55.f, 5.f }
                    : v.nb == 3             ? Rule{ 105, 45.f, 4.f }
                    : v.nb == 4             ? Rule{ 87, 45.f, 4.f }
                                            : Rule{ 121, 45.f, 3.f };
  const int64_t voxels = (int64_t)job.vx * job.vy * job.vz;
  if (voxels > (int64_t)rule.upTo * rule.upTo * rule.upTo) return false;
  const float spaces = (float)(job.spaceEnd - job.spaceBegin);
  return spaces >= (cbrtf((float)voxels) - rule.from) * rule.slope;
}

FrChoice choose_fr_insert(const FrJob &job, const FrLaunch &l, const FrVariant &v0, int numCUs)
{
  // a plain launch slides its boxes when its job does; a batch's host sets v.shift when every
  // job of the launch does
  FrVariant v = v0;
  if (!v.batched) v.shift = job.shiftBox != 0;
  if (use_cells(job, l, v)) return choose_fr_cells(l, v, numCUs);
  FrChoice ch{};
  ch.which = kKernelPair;
  ch.kernel = pick_kernel(v, l.nTable);
  if (!ch.kernel) return ch;
  ch.lds = table_in_lds(v, l.nTable) ? (size_t)(l.nTable + 1) * sizeof(float) : 0;
  // persistent workgroups: the per-wave LDS state allows one per CU
  int waves = fr_waves(v.mode, v.half, v.fastMath);
  // kKernelAuto: the staged kernel for the exact strategy, the carried queues for fast-math
  // FP32 slices (FP16 slices run faster on the per-pair kernel: 1.22 vs 1.26 ms per 1,000-slice
  // chunk at box 256); batches run the per-pair kernel unless they name the carried queues
  // (their host checks that every job's slices fit one buffer resource)
  const int want = v.kernel != kKernelAuto ? v.kernel
                   : v.batched            ? kKernelPair
                   : !v.fastMath          ? kKernelStaged
                   : v.half               ? kKernelPair
                                          : kKernelCarry;
  const void *staged = want == kKernelStaged ? pick_staged(v, l.nTable, v.shift) : nullptr;
  const void *carry = want == kKernelCarry ? pick_carry(v, l.nTable) : nullptr;
  if (staged && staged_fits(job)) {
    ch.kernel = staged;
    ch.which = kKernelStaged;
    waves = kStagedWaves;
  } else if (carry && carry_fits(job, v.half)) {
    ch.kernel = carry;
    ch.which = kKernelCarry;
  }
  ch.threads = 64 * waves;
  // persistent workgroups, one per CU, until the items run out; with l.waveItems, every workgroup
  // leaves after that many items for each of its waves and the grid covers the items (CUs come
  // free for other streams' launches as workgroups end)
  if (l.waveItems > 0) {
    const int64_t per = (int64_t)waves * l.waveItems;
    ch.blocks = (int)((l.nItems + per - 1) / per);
  } else {
    // (as many as the core has cells or the rest has bricks, whichever is more)
    ch.blocks = (std::max(l.nItems, l.nCore) + waves - 1) / waves;
    if (ch.blocks > numCUs) ch.blocks = numCUs;
    if (l.maxBlocks > 0 && ch.blocks > l.maxBlocks) ch.blocks = l.maxBlocks;
  }
  if (ch.blocks < 1) ch.blocks = 1;
  return ch;
}

hipError_t launch_fr_insert(const FrJob &job, const FrLaunch &l, const FrVariant &v, int numCUs,
                            hipStream_t st)
{
  const FrChoice ch = choose_fr_insert(job, l, v, numCUs);
  if (!ch.kernel) return hipErrorInvalidValue;
  FrJob j = job;
  FrLaunch ll = l;
  ll.numCUs = numCUs;
  const int waves = ch.threads / 64;
  if (l.waveItems > 0)  // (a workgroup's count of items stays an int)
    ll.waveItems = (int)std::min<int64_t>(l.waveItems, ((int64_t)l.nItems + waves - 1) / waves);
  void *args[] = { &j, &ll };
  return hipLaunchKernel(ch.kernel, dim3(ch.blocks), dim3(ch.threads), args, ch.lds, st);
}

}  // namespace umpa
