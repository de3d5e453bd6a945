// FR insertion for small problems on gfx950: eight spaces at a time into cells of 2 x 2 x 2 voxels.
//
// The brick kernels (fr_kernels.hip) take the spaces of a brick one after another: about 1 us
// per space and wavefront, whatever the brick's size, since a space's slab test, queue, gather
// and sums each wait for the one before.  A volume with few bricks then takes as long as its
// central brick, which every space reaches (box 100, 1,004 spaces, exact: 99 % of the
// wavefronts were done after 0.45 ms, the last after 1.06).  Here a lane is a (voxel, space)
// pair: a wavefront owns a cell of eight voxels and takes eight of its spaces at a time, so the
// chain is an eighth as long and a volume has 64 times the wavefronts' work items.
//
// A workgroup of eight wavefronts owns a block of 4 x 4 x 4 voxels (a cell per wavefront), or
// away from the centre, where few spaces reach a cell, of 8 x 8 x 8 (eight cells per wavefront),
// or at the centre of the smallest volumes of 4 x 2 x 2 (four wavefronts per cell, shared_cell).
// It culls a tile of spaces against the block, two per thread, into a list in index order; each
// wavefront culls the list further against its cell, 64 entries at a time, into a queue, and
// takes the queue eight spaces at a time: predicate and gather per lane (fr_gather.hpp), the
// contributions through LDS to 24 lanes, (component, voxel) each, which add the eight spaces'
// in order.  So every voxel receives its spaces in index order, the reference's order
// (fr_cpu_kernels.hpp:254), under every strategy: no atomics, and bit-identical sums under the
// exact one.  A pair that misses adds -0, which changes no float.
//
// The price is idle lanes and work per cell: about two thirds of a central cell's pairs hit,
// where the brick kernels compact the hits of 512 voxels, and away from the centre a step has
// fewer than eight spaces (VALU lane-instructions per voxel-update 520 to 950, against 360), so
// this kernel is for launches the brick kernels cannot fill the GPU with (use_cells() in
// fr_kernels.hip).  What bounds it is the chain of steps, about 1.5 us each, and between VALU
// busy 0.35 (box 64, 500 spaces) and 0.8.  us per pass, bricks -> cells: box 32, 16 slices
// 24.7 -> 15.3; box 64, 500, fast math 510 -> 120; box 100, 251, C4, r 1.5, exact 1004 -> 299;
// box 120, 400, blob evaluated 1224 -> 366.
#include "fr_cell.hpp"

namespace umpa {

constexpr int kCellWaves = 8;
constexpr int kCellThreads = 64 * kCellWaves;
constexpr int kCellTile = 2 * kCellThreads;  // spaces culled together

// A cell that four wavefronts share: each takes every fourth eight of the list's spaces, and the first
// of them adds the 32 spaces' contributions in order while the others gather the next.  `part` and
// `hit` are written in turn, so one barrier a round separates their uses.  Every wavefront of the
// workgroup makes the same rounds (the cell may lie outside the volume).
// The chain of the central cells' spaces is what a very small volume's launch waits for (about 1.5
// us per eight spaces; box 32, 500 slices, exact 97 -> 57 us, r 2.5 170 -> 110; rule: share_cells).
template <int kMode, int kOrder, int kNB, bool kHalf, bool kFastMath, bool kTableLds, bool kShift,
          int kRows>
__device__ __forceinline__ void shared_cell(const FrJob &a, int x0, int y0, int z0, int base,
                                            const uint16_t *list, int n,
                                            float (*part)[kCellWaves][3 * 64],
                                            int (*hits)[kCellWaves], float *blob, int nTable,
                                            __amdgpu_buffer_rsrc_t rsrc, const float *tbl,
                                            uint32_t sliceBytes, int wave, int lane)
{
  if (n == 0) return;
  Cell cell = make_cell(a, x0, y0, z0, lane);
  auto space_at = [&](int i) {
    const uint32_t e = list[i < n ? i : 0];
    return load_space<kHalf>(a, base + (int)(e & 0x7fffu), (e & 0x8000u) != 0, sliceBytes);
  };
  int turn = 0;
  int i = 8 * (wave & 3) + (lane & 7);
  CellSpace next = space_at(i);
  for (int r = 0; r < n; r += 32, i += 32, turn ^= 1) {
    const CellSpace sp = next;
    if (r + 32 < n) next = space_at(i + 32);
    float qx, qy, zs;
    const bool hit = cell_pair<kMode>(cell, a, sp, cell.valid && i < n, qx, qy, zs);
    const bool any = __any(hit);
    if (any) {
      const Contribution o =
        cell_gather<kMode, kOrder, kNB, kHalf, kFastMath, kTableLds, kShift, kRows>(
          a, sp, hit, qx, qy, zs, blob, nTable, rsrc, tbl, lane);
      float *mine = part[turn][wave];
      mine[lane] = o.re;
      mine[64 + lane] = o.im;
      mine[128 + lane] = o.w;
    }
    if (lane == 0) hits[turn][wave] = any;
    __syncthreads();
    if ((wave & 3) != 0) continue;
    for (int w = wave; w < wave + 4; ++w) {
      if (!__builtin_amdgcn_readfirstlane(hits[turn][w])) continue;
      if (!cell.loaded) {
        if (cell.owner) cell.acc = *cell.sum;
        cell.loaded = true;
      }
      if (lane < 24) cell_add(cell, part[turn][w], lane);
    }
  }
  if (cell.loaded && cell.owner) *cell.sum = cell.acc;
}

template <int kMode, int kOrder, int kNB, bool kHalf, bool kFastMath, bool kShift, bool kShared>
__global__ __launch_bounds__(kCellThreads, 4) void fr_insert_cell_kernel(FrJob a, FrLaunch l)
{
  constexpr bool kTableLds = kMode == kModeLookup;
  constexpr int kPix = kHalf ? 4 : 8;
  // rows of the gather in flight: what 128 registers hold beside two spaces' records (six columns:
  // two FP32 rows spilled up to 90; box 112, 400 slices, r 2.8, exact 803 -> 464 us with one)
  constexpr int kRows = kHalf ? (kNB <= 4 ? kNB : 3) : kNB <= 3 ? 3 : kNB <= 5 ? 2 : 1;
  extern __shared__ float s_table[];
  __shared__ __align__(16) float s_part[kShared ? 2 : 1][kCellWaves][3 * 64];
  __shared__ int s_hit[kShared ? 2 : 1][kCellWaves];
  __shared__ float s_blob[evaluates_blob(kMode) ? kCellWaves : 1][evaluates_blob(kMode) ? kBlobList : 1];
  __shared__ uint16_t s_list[kCellTile];
  __shared__ uint16_t s_queue[kCellWaves][kCellRing];
  __shared__ int s_count[kCellWaves];
  __shared__ int s_next[2];
  const int nTable = l.nTable;
  if constexpr (kTableLds) stage_table<kCellThreads>(s_table, l.table, nTable);
  const float *tbl = kTableLds ? s_table : l.table;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  float *part = s_part[0][wave], *blob = evaluates_blob(kMode) ? s_blob[wave] : nullptr;
  uint16_t *queue = s_queue[wave];
  const umpa_fr_constants &c = a.c;
  const int cxi = c.cMaxVolumeIndexX / 2, cyi = c.cMaxVolumeIndexYZ / 2;
  const uint32_t sliceBytes = (uint32_t)(a.sliceElems * kPix);
  const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
    (void *)a.fft, 0, (int)((uint32_t)a.nProj * sliceBytes), kBufferConfig);
  unsigned long long nupd = 0;

  // Blocks in turn, heaviest first: the first from the grid, the others from the counter.  Every
  // workgroup's last claim finds none; the one that makes the launch's last claim clears the
  // counter for the next launch.
  if (a.spaceBegin >= a.spaceEnd) return;
  int turn = 0;
  for (int b = blockIdx.x; b < l.nCells; turn ^= 1) {
    if (threadIdx.x == 0) {
      const int next = atomicAdd(l.cellCounter, 1);
      if (next == l.nCells - 1) atomicExch(l.cellCounter, 0);
      s_next[turn] = next + (int)gridDim.x;  // read after the block's barriers
    }
    const int2 item = reinterpret_cast<const int2 *>(l.cells)[b];
    const int x0 = item.x & 0xffff, y0 = (item.x >> 16) & 0xffff, z0 = item.y & 0xffff;
    // 2: two cells side by side, four wavefronts each; 4: a cell per wavefront; 8: eight cells
    const int edge = item.y >> 16;
    const int wide = kShared && edge == 2 ? 4 : edge;
    const int nMine = edge == 8 ? 8 : kShared && edge == 2 ? 0 : 1;  // the wavefront's own

    for (int base = a.spaceBegin; base < a.spaceEnd; base += kCellTile) {
      // cull the tile: wavefront w takes spaces base + 128 w ..., in index order
      const int s0 = base + wave * 128 + lane, s1 = s0 + 64;
      bool in0 = false, in1 = false;
      const unsigned long long m0 =
        __ballot(s0 < a.spaceEnd && cull_block(a, s0, x0, y0, z0, wide, edge, cxi, cyi, in0));
      const unsigned long long m1 =
        __ballot(s1 < a.spaceEnd && cull_block(a, s1, x0, y0, z0, wide, edge, cxi, cyi, in1));
      const int mine = __popcll(m0) + __popcll(m1);
      if (lane == 0) s_count[wave] = mine;
      __syncthreads();  // (also: every wavefront is done with the previous list)
      int n = 0, at = 0;
#pragma unroll
      for (int i = 0; i < kCellWaves; ++i) {
        at = i == wave ? n : at;
        n += __builtin_amdgcn_readfirstlane(s_count[i]);
      }
      if ((m0 >> lane) & 1ull)
        s_list[lanes_below(m0, (unsigned)at)] = (uint16_t)((s0 - base) | (in0 ? 0x8000 : 0));
      at += __popcll(m0);
      if ((m1 >> lane) & 1ull)
        s_list[lanes_below(m1, (unsigned)at)] = (uint16_t)((s1 - base) | (in1 ? 0x8000 : 0));
      __syncthreads();

      if constexpr (kShared) {
        if (edge == 2)
          shared_cell<kMode, kOrder, kNB, kHalf, kFastMath, kTableLds, kShift, kRows>(
            a, x0 + 2 * (wave >> 2), y0, z0, base, s_list, n, s_part, s_hit, blob, nTable, rsrc, tbl,
            sliceBytes, wave, lane);
      }
      for (int ci = 0; ci < nMine; ++ci) {
        // octant of the block = wave; in an octant of edge 4, cell ci
        const int step0 = edge >> 1;
        const int cellX = x0 + step0 * (wave & 1) + 2 * (ci & 1),
                  cellY = y0 + step0 * ((wave >> 1) & 1) + 2 * ((ci >> 1) & 1),
                  cellZ = z0 + step0 * (wave >> 2) + 2 * (ci >> 2);
        if (cellX >= a.vx || cellY >= a.vy || cellZ >= a.vz) continue;
        Cell cell = make_cell(a, cellX, cellY, cellZ, lane);
        int head = 0, pend = 0;
        for (int t0 = 0; t0 < n; t0 += 64) {
          const bool have = t0 + lane < n;
          const uint32_t e = have ? (uint32_t)s_list[t0 + lane] : 0u;
          const float *r2 = a.spaces[base + (int)(e & 0x7fffu)].transformInv[2];
          const float t20 = r2[0], t21 = r2[1], t22 = r2[2];
          const float qzc = t20 * cell.cx + t21 * cell.cy + t22 * cell.cz;
          const float ez = 0.5f * (fabsf(t20) + fabsf(t21) + fabsf(t22));
          const unsigned long long keep = __ballot(have && fabsf(qzc) <= cell.reach + ez);
          if ((keep >> lane) & 1ull)
            queue[lanes_below(keep, (unsigned)(head + pend)) & (kCellRing - 1)] = (uint16_t)e;
          pend += __popcll(keep);
          wave_sync();
          // the last entries also make a partial step
          cell_take<kMode, kOrder, kNB, kHalf, kFastMath, kTableLds, kShift, kRows, false>(
            cell, a, base, queue, part, blob, head, pend, t0 + 64 < n ? 8 : 1, nTable, rsrc, tbl,
            sliceBytes, lane, nupd);
        }
        if (cell.loaded && cell.owner) *cell.sum = cell.acc;
      }
    }
    b = __builtin_amdgcn_readfirstlane(s_next[turn]);
  }
}

// ---- host-side dispatch ------------------------------------------------------------------
template <int kNB, bool kShared>
static const void *pick_lookup(const FrVariant &v)
{
  if (v.half)
    return v.shift ? (const void *)fr_insert_cell_kernel<kModeLookup, 0, kNB, true, true, true, kShared>
                   : (const void *)fr_insert_cell_kernel<kModeLookup, 0, kNB, true, true, false, kShared>;
  if (v.fastMath)
    return v.shift ? (const void *)fr_insert_cell_kernel<kModeLookup, 0, kNB, false, true, true, kShared>
                   : (const void *)fr_insert_cell_kernel<kModeLookup, 0, kNB, false, true, false, kShared>;
  return v.shift ? (const void *)fr_insert_cell_kernel<kModeLookup, 0, kNB, false, false, true, kShared>
                 : (const void *)fr_insert_cell_kernel<kModeLookup, 0, kNB, false, false, false, kShared>;
}

template <bool kShared>
static const void *pick_cells(const FrVariant &v)
{
  switch (v.mode) {
  case kModeLookup:
    switch (v.nb) {
    case 3: return pick_lookup<3, kShared>(v);
    case 4: return pick_lookup<4, kShared>(v);
    case 5: return pick_lookup<5, kShared>(v);
    default: return pick_lookup<6, kShared>(v);
    }
  case kModeFastKaiser:
    return (const void *)fr_insert_cell_kernel<kModeFastKaiser, 0, 4, false, false, false, kShared>;
  case kModeNearest:
    return (const void *)fr_insert_cell_kernel<kModeNearest, 0, 4, false, false, false, kShared>;
  case kModePreciseKaiser:
    switch (v.order) {
    case 0: return (const void *)fr_insert_cell_kernel<kModePreciseKaiser, 0, 4, false, false, false, kShared>;
    case 1: return (const void *)fr_insert_cell_kernel<kModePreciseKaiser, 1, 4, false, false, false, kShared>;
    case 2: return (const void *)fr_insert_cell_kernel<kModePreciseKaiser, 2, 4, false, false, false, kShared>;
    case 3: return (const void *)fr_insert_cell_kernel<kModePreciseKaiser, 3, 4, false, false, false, kShared>;
    case 4: return (const void *)fr_insert_cell_kernel<kModePreciseKaiser, 4, 4, false, false, false, kShared>;
    }
  }
  return nullptr;
}

FrChoice choose_fr_cells(const FrLaunch &l, const FrVariant &v, int numCUs)
{
  FrChoice c{};
  c.which = kKernelCells;
  if (l.nCells <= 0) return c;
  // (an instantiation of its own: as a branch, shared cells cost the others 1 to 2 %)
  c.kernel = l.cellsShared ? pick_cells<true>(v) : pick_cells<false>(v);
  // two workgroups per CU: registers for 16 wavefronts, LDS for both tables (at most 47 KB each)
  c.blocks = l.nCells < 2 * numCUs ? l.nCells : 2 * numCUs;
  c.threads = kCellThreads;
  c.lds = v.mode == kModeLookup ? (size_t)(l.nTable + 1) * sizeof(float) : 0;
  return c;
}

}  // namespace umpa
