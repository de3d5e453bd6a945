// Cells: eight voxels (2 x 2 x 2) that a wavefront takes eight spaces at a time, one (voxel,
// space) pair per lane.  Used by the small-problem kernel (fr_cells.hip) for whole volumes and by
// the brick kernels (fr_kernels.hip) for the centre of larger ones under the exact strategy.
#pragma once

#include "fr_gather.hpp"

namespace umpa {

constexpr int kCellRing = 128;  // a wavefront's queue of spaces: 7 left over + 64 new

// What a lane needs of its space.
struct CellSpace {
  float t[3][3];
  float weight, scale;
  uint32_t off;  // byte offset of its slice in the chunk
  int index;
  bool inside;   // the cell lies inside the space's sphere and traversal plane
};

// A queue entry: the space's index (relative to the caller's base) and the `inside` flag on top.
template <typename Entry>
constexpr uint32_t kInsideBit = 1u << (8 * sizeof(Entry) - 1);

template <bool kHalf>
__device__ __forceinline__ CellSpace load_space(const FrJob &a, int index, bool inside,
                                                uint32_t sliceBytes)
{
  CellSpace s;
  const umpa_traverse_space &sp = a.spaces[index];
#pragma unroll
  for (int i = 0; i < 9; ++i) s.t[i / 3][i % 3] = sp.transformInv[i / 3][i % 3];
  s.weight = sp.weight;
  const int proj = sp.projectionIndex;
  s.off = (uint32_t)proj * sliceBytes;
  s.scale = 1.f;
  if constexpr (kHalf) s.scale = a.scales[proj];
  s.index = index;
  s.inside = inside;
  return s;
}

// Does space `si` reach the block of `wide` columns and edge `e` otherwise at (x0, y0, z0)?  As
// cull_space of the brick kernels; `inside` as brick_inside.
__device__ __forceinline__ bool cull_block(const FrJob &a, int si, int x0, int y0, int z0, int wide,
                                           int e, int cxi, int cyi, bool &inside)
{
  const umpa_traverse_space &sp = a.spaces[si];
  const float(*t)[3] = sp.transformInv;
  const float half = 0.5f * (float)(e - 1), halfX = 0.5f * (float)(wide - 1);
  const float cx = (float)(x0 - cxi) + halfX, cy = (float)(y0 - cyi) + half,
              cz = (float)(z0 - cyi) + half;
  const float norm = sqrtf(cx * cx + cy * cy + cz * cz);
  const float dmin = fmaxf(norm - 1.7321f * halfX, 0.f);  // (wide >= e)
  const float eps = 0.02f + 1e-5f * norm;
  const float qz = t[2][0] * cx + t[2][1] * cy + t[2][2] * cz;
  const float ez = halfX * fabsf(t[2][0]) + half * (fabsf(t[2][1]) + fabsf(t[2][2]));
  const float qx = t[0][0] * cx + t[0][1] * cy + t[0][2] * cz;
  const float ex = halfX * fabsf(t[0][0]) + half * (fabsf(t[0][1]) + fabsf(t[0][2]));
  const float mds = sp.maxDistanceSqr;
  const int proj = sp.projectionIndex, dir = sp.dir;
  const int x1 = x0 + wide - 1, y1 = y0 + e - 1, z1 = z0 + e - 1;
  const int mx = max(abs(x0 - cxi), abs(x1 - cxi));
  const int my = max(abs(y0 - cyi), abs(y1 - cyi));
  const int mz = max(abs(z0 - cyi), abs(z1 - cyi));
  const bool inX = (x0 >= sp.minX) & (x1 <= sp.maxX);
  const bool inY = (y0 >= sp.minY) & (y1 <= sp.maxY);
  const bool inZ = (z0 >= sp.minZ) & (z1 <= sp.maxZ);
  inside = ((float)(mx * mx + my * my + mz * mz) <= mds) &
           (dir == 0 ? (inX & inY) : dir == 1 ? (inX & inZ) : (inY & inZ));
  return (fabsf(qz) <= a.cullHalfWidth + ez + eps) & (qx >= -a.cullHalfSpace - ex - eps) &
         (dmin * dmin <= mds * 1.0001f + eps) & (proj >= 0) & (proj < a.nProj) & (dir >= 0) &
         (dir <= 2);
}

// A wavefront's cell: the lane's voxel (lane / 8 of the cell; lane % 8 is its space of eight), and
// for lanes 0..23 one of the cell's sums: component lane / 8 (re, im, weight) of voxel lane % 8.
struct Cell {
  int x, y, z;
  float px, py, pz;
  bool valid;           // the voxel lies in the volume
  float cx, cy, cz, reach;  // the cell's centre; slab half width and margin of its cull
  bool owner;
  float *sum;
  float acc;
  bool loaded;          // acc holds the sum (read when the first pair hits)
};

__device__ __forceinline__ Cell make_cell(const FrJob &a, int x0, int y0, int z0, int lane)
{
  Cell k;
  const umpa_fr_constants &c = a.c;
  const int cxi = c.cMaxVolumeIndexX / 2, cyi = c.cMaxVolumeIndexYZ / 2;
  const int v = lane >> 3;
  k.x = x0 + (v & 1);
  k.y = y0 + ((v >> 1) & 1);
  k.z = z0 + (v >> 2);
  k.valid = k.x < a.vx && k.y < a.vy && k.z < a.vz;
  k.px = (float)(k.x - cxi);
  k.py = (float)(k.y - cyi);
  k.pz = (float)(k.z - cyi);
  k.cx = (float)(x0 - cxi) + 0.5f;
  k.cy = (float)(y0 - cyi) + 0.5f;
  k.cz = (float)(z0 - cyi) + 0.5f;
  k.reach = 0.02f + 1e-5f * sqrtf(k.cx * k.cx + k.cy * k.cy + k.cz * k.cz) + a.cullHalfWidth;
  const int av = lane & 7, comp = lane >> 3;
  const int ax = x0 + (av & 1), ay = y0 + ((av >> 1) & 1), az = z0 + (av >> 2);
  k.owner = lane < 24 && ax < a.vx && ay < a.vy && az < a.vz;
  const int64_t gi = ((int64_t)az * a.vy + ay) * a.vx + ax;
  k.sum = comp == 2 ? a.weights + gi : reinterpret_cast<float *>(a.volume) + 2 * gi + comp;
  k.acc = 0.f;
  k.loaded = false;
  return k;
}

// The lane's pair: does space `sp` reach the cell's voxel, and where does it lie in the slice's frame?
template <int kMode>
__device__ __forceinline__ bool cell_pair(const Cell &k, const FrJob &a, const CellSpace &sp, bool act,
                                          float &qx, float &qy, float &zs)
{
  const umpa_traverse_space &rec = a.spaces[sp.index];
  bool hit;
  if constexpr (kMode == kModeNearest) {
    const float dsq = k.px * k.px + k.py * k.py + k.pz * k.pz;
    qx = sp.t[0][0] * k.px + sp.t[0][1] * k.py + sp.t[0][2] * k.pz;
    qy = sp.t[1][0] * k.px + sp.t[1][1] * k.py + sp.t[1][2] * k.pz;
    zs = 0.f;
    hit = act && !(dsq > rec.maxDistanceSqr) && !(qx < 0.f) && visited_nearest(rec, k.x, k.y, k.z);
  } else {
    hit = act && blob_predicate<false>(rec, sp.t, a.c, k.x, k.y, k.z, k.px, k.py, k.pz, sp.inside,
                                       qx, qy, zs);
  }
  return hit;
}

// Its contribution (-0, which changes no float, for a pair that misses); called by the whole
// wavefront.  `blob`: kBlobList floats of the wavefront's LDS for the evaluated blob modes.
template <int kMode, int kOrder, int kNB, bool kHalf, bool kFastMath, bool kTableLds, bool kShift,
          int kRows>
__device__ __forceinline__ Contribution cell_gather(const FrJob &a, const CellSpace &sp, bool hit,
                                                    float qx, float qy, float zs, float *blob,
                                                    int nTable, __amdgpu_buffer_rsrc_t rsrc,
                                                    const float *tbl, int lane)
{
  Contribution o{ -0.f, -0.f, -0.f };
  if constexpr (evaluates_blob(kMode)) {
    const Contribution got = gather_evaluated<kMode, kOrder>(a, rsrc, blob, lane, hit, qx, qy, zs,
                                                             sp.weight, sp.off);
    if (hit) o = got;
  } else if (hit) {
    if constexpr (kMode == kModeNearest) {
      o = gather_nearest<kHalf>(a, rsrc, qx, qy, sp.weight, sp.scale, sp.off);
    } else {
      // (a weight of 1 changes no product, so one copy of the gather serves all)
      o = gather_update<kMode, kOrder, kNB, kHalf, kFastMath, kTableLds, kShift, true, kRows>(
        a, nTable, rsrc, tbl, qx, qy, zs, sp.weight, false, sp.scale, sp.off);
    }
  }
  return o;
}

// Adds eight spaces' contributions (`part`, 192 floats: component, voxel, space) in order; lanes
// 0..23, each its sum.
__device__ __forceinline__ void cell_add(Cell &k, const float *part, int lane)
{
  const float4 p = reinterpret_cast<const float4 *>(part)[2 * lane],
               q = reinterpret_cast<const float4 *>(part)[2 * lane + 1];
  k.acc = k.acc + p.x;
  k.acc = k.acc + p.y;
  k.acc = k.acc + p.z;
  k.acc = k.acc + p.w;
  k.acc = k.acc + q.x;
  k.acc = k.acc + q.y;
  k.acc = k.acc + q.z;
  k.acc = k.acc + q.w;
}

// Takes the queue's spaces eight at a time while at least `least` are pending: predicate and
// gather per lane, the contributions through LDS (`part`, 192 floats) to the lanes that own the
// sums, which add the eight spaces' in order, so a voxel receives its spaces in index order.  A
// pair that misses adds -0, which changes no float.  Entry i of the queue names space base + i.
// `blob`: kBlobList floats of the wavefront's LDS for the evaluated blob modes.
template <int kMode, int kOrder, int kNB, bool kHalf, bool kFastMath, bool kTableLds, bool kShift,
          int kRows, bool kCount, typename Entry>
__device__ __forceinline__ void cell_take(Cell &k, const FrJob &a, int base, const Entry *queue,
                                          float *part, float *blob, int &head, int &pend, int least,
                                          int nTable,
                                          __amdgpu_buffer_rsrc_t rsrc, const float *tbl,
                                          uint32_t sliceBytes, int lane, unsigned long long &nupd)
{
  if (pend < least) return;
  const int s = lane & 7;
  auto space_at = [&](int from, int n) {
    const uint32_t q = queue[(from + (s < n ? s : 0)) & (kCellRing - 1)];
    return load_space<kHalf>(a, base + (int)(q & (kInsideBit<Entry> - 1u)),
                             (q & kInsideBit<Entry>) != 0, sliceBytes);
  };
  CellSpace next = space_at(head, pend);
  do {
    const CellSpace sp = next;
    const int n = pend < 8 ? pend : 8;
    // the next spaces' records load while these are gathered
    if (pend - n >= least) next = space_at(head + n, pend - n);
    head = (head + n) & (kCellRing - 1);
    pend -= n;

    float qx, qy, zs;
    const bool hit = cell_pair<kMode>(k, a, sp, k.valid && s < n, qx, qy, zs);
    if (!__any(hit)) continue;
    if constexpr (kCount) nupd += (unsigned long long)__popcll(__ballot(hit));
    if (!k.loaded) {
      if (k.owner) k.acc = *k.sum;
      k.loaded = true;
    }
    const Contribution o = cell_gather<kMode, kOrder, kNB, kHalf, kFastMath, kTableLds, kShift, kRows>(
      a, sp, hit, qx, qy, zs, blob, nTable, rsrc, tbl, lane);
    part[lane] = o.re;
    part[64 + lane] = o.im;
    part[128 + lane] = o.w;
    wave_sync();
    if (lane < 24) cell_add(k, part, lane);
    wave_sync();
  } while (pend >= least);
}

// A work item of the brick kernels that is one cell: culls the spaces 64 at a time and takes the
// survivors.  `queue`, `part` and `blob` are kCellRing, 192 and (evaluated blobs) kBlobList dwords
// of the wavefront's LDS.
template <int kMode, int kOrder, int kNB, bool kTableLds, bool kShift, bool kCount>
__device__ __forceinline__ void cell_item(const FrJob &a, int x0, int y0, int z0, int sBegin,
                                          int sEnd, uint32_t *queue, float *part, float *blob,
                                          int nTable,
                                          __amdgpu_buffer_rsrc_t rsrc, const float *tbl, int lane,
                                          unsigned long long &nupd)
{
  const umpa_fr_constants &c = a.c;
  const int cxi = c.cMaxVolumeIndexX / 2, cyi = c.cMaxVolumeIndexYZ / 2;
  const uint32_t sliceBytes = (uint32_t)(a.sliceElems * 8);
  Cell cell = make_cell(a, x0, y0, z0, lane);
  int head = 0, pend = 0;
  for (int base = sBegin; base < sEnd; base += 64) {
    const int si = base + lane;
    bool in = false;
    const unsigned long long m = __ballot(si < sEnd && cull_block(a, si, x0, y0, z0, 2, 2, cxi, cyi, in));
    if ((m >> lane) & 1ull)
      queue[lanes_below(m, (unsigned)(head + pend)) & (kCellRing - 1)] =
        (uint32_t)si | (in ? kInsideBit<uint32_t> : 0u);
    pend += __popcll(m);
    wave_sync();
    cell_take<kMode, kOrder, kNB, false, false, kTableLds, kShift, (kNB <= 5 ? 2 : 1), kCount>(
      cell, a, 0, queue, part, blob, head, pend, base + 64 < sEnd ? 8 : 1, nTable, rsrc, tbl, sliceBytes,
      lane, nupd);
  }
  if (cell.loaded && cell.owner) *cell.sum = cell.acc;
  wave_sync();
}

}  // namespace umpa
