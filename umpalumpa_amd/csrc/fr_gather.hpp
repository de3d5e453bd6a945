// Gather of one voxel-update: pixel loads through bounds-checked buffers, the blob-weighted sum
// over the candidate box, and the reference's per-voxel predicate.  Shared by the brick kernels
// (fr_kernels.hip) and the cell kernel (fr_cells.hip).
#pragma once

#include "fr_device.hpp"

namespace umpa {

constexpr uint32_t kOutOfRange = 0x7ffff000u;  // buffer offset past every slice: loads read 0
constexpr uint32_t kBufferConfig = 0x00020000u; // raw buffer descriptor word 3 on gfx9

__device__ __forceinline__ void wave_sync()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// `base` plus the number of lanes below this one in `mask` (the count's accumulator input)
__device__ __forceinline__ unsigned lanes_below(unsigned long long mask, unsigned base = 0u)
{
  return __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, base));
}

// Raw buffer loads through the LLVM intrinsics.  (The clang builtin for the 64-bit raw buffer
// load, __builtin_amdgcn_raw_buffer_load_b64, lowers to a single 32-bit load in this toolchain
// and returns that dword for both halves, so the vector forms are declared directly.)  Every
// byte offset travels in the vector offset, which the hardware range-checks together with the
// instruction's immediate offset; the scalar offset is not range-checked, and loads that
// differed only in it were observed to be merged into one by this compiler, so it stays 0.
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
__device__ f32x2_t raw_buffer_load_f32x2(__amdgpu_buffer_rsrc_t rsrc, uint32_t voffset,
                                        uint32_t soffset,
                                        int aux) __asm("llvm.amdgcn.raw.ptr.buffer.load.v2f32");
__device__ uint32_t raw_buffer_load_u32(__amdgpu_buffer_rsrc_t rsrc, uint32_t voffset,
                                        uint32_t soffset,
                                        int aux) __asm("llvm.amdgcn.raw.ptr.buffer.load.i32");
__device__ f32x4_t raw_buffer_load_f32x4(__amdgpu_buffer_rsrc_t rsrc, uint32_t voffset,
                                        uint32_t soffset,
                                        int aux) __asm("llvm.amdgcn.raw.ptr.buffer.load.v4f32");
__device__ u32x4_t raw_buffer_load_u32x4(__amdgpu_buffer_rsrc_t rsrc, uint32_t voffset,
                                        uint32_t soffset,
                                        int aux) __asm("llvm.amdgcn.raw.ptr.buffer.load.v4i32");

// Slice pixel at byte offset `byteOffset` through a bounds-checked buffer resource: offsets at
// or past the slice end return zero instead of faulting.
template <bool kHalf>
__device__ __forceinline__ float2 load_pixel(__amdgpu_buffer_rsrc_t rsrc, uint32_t byteOffset)
{
  if constexpr (kHalf) {
    const uint32_t v = raw_buffer_load_u32(rsrc, byteOffset, 0, 0);
    return __half22float2(__builtin_bit_cast(__half2, v));
  } else {
    const f32x2_t v = raw_buffer_load_f32x2(rsrc, byteOffset, 0, 0);
    return make_float2(v.x, v.y);
  }
}

// A slice pixel as loaded: complex float, or complex half packed in one dword (converted at
// the multiply-add, which the compiler fuses into a mixed-precision FMA).
template <bool kHalf> struct Pixel;
template <> struct Pixel<false> {
  float2 v;
  __device__ __forceinline__ float re() const { return v.x; }
  __device__ __forceinline__ float im() const { return v.y; }
};
template <> struct Pixel<true> {
  uint32_t v;
  __device__ __forceinline__ float re() const
  {
    return __half2float(__builtin_bit_cast(__half, (uint16_t)(v & 0xffffu)));
  }
  __device__ __forceinline__ float im() const
  {
    return __half2float(__builtin_bit_cast(__half, (uint16_t)(v >> 16)));
  }
};

template <bool kHalf>
__device__ __forceinline__ Pixel<kHalf> load_pixel_raw(__amdgpu_buffer_rsrc_t rsrc,
                                                       uint32_t byteOffset)
{
  Pixel<kHalf> p;
  if constexpr (kHalf) {
    p.v = raw_buffer_load_u32(rsrc, byteOffset, 0, 0);
  } else {
    const f32x2_t v = raw_buffer_load_f32x2(rsrc, byteOffset, 0, 0);
    p.v = make_float2(v.x, v.y);
  }
  return p;
}

// kNB consecutive pixels of a slice row starting at byte `voff`, with 16-byte loads (4 FP16 or
// 2 FP32 pixels each).  Dwords past the slice end read zero.  A load on the slice's last row
// can straddle the end; the raw buffer's range check then still returns its in-range dwords
// (the reference's 3 x 6 plane cases, where every last-row load straddles, are bit-exact).
template <bool kHalf, int kNB>
__device__ __forceinline__ void load_row(__amdgpu_buffer_rsrc_t rsrc, uint32_t voff,
                                         Pixel<kHalf> (&px)[kNB])
{
  constexpr int kPix = kHalf ? 4 : 8;
  constexpr int kPer = 16 / kPix;                  // pixels per 16-byte load
  constexpr int kLoads = (kNB + kPer - 1) / kPer;
  // (vector elements are named, never indexed by a loop variable: this compiler folded
  // v[e] in an unrolled loop over e to v[0] for every e, in the 16-byte loads here)
#pragma unroll
  for (int q = 0; q < kLoads; ++q) {
    if constexpr (kHalf) {
      const u32x4_t v = raw_buffer_load_u32x4(rsrc, voff + (uint32_t)(q * 16), 0, 0);
      const uint32_t w[4] = { v.x, v.y, v.z, v.w };
#pragma unroll
      for (int e = 0; e < kPer; ++e) {
        const int j = q * kPer + e;
        if (j < kNB) px[j].v = w[e];
      }
    } else {
      const f32x4_t v = raw_buffer_load_f32x4(rsrc, voff + (uint32_t)(q * 16), 0, 0);
      const float w[4] = { v.x, v.y, v.z, v.w };
#pragma unroll
      for (int e = 0; e < kPer; ++e) {
        const int j = q * kPer + e;
        if (j < kNB) px[j].v = make_float2(w[2 * e], w[2 * e + 1]);
      }
    }
  }
}

// Blob weight of one candidate pixel (kDynamic modes; kLookup reads the LDS table inline).
template <int kMode, int kOrder>
__device__ __forceinline__ float blob_weight(float d2, const umpa_fr_constants &c)
{
  if constexpr (kMode == kModeFastKaiser) {
    return kaiser_value_fast(d2, c);
  } else {
    return kaiser_value<kOrder>(sqrtf(d2), c.cBlobRadius, c) * c.cIw0;
  }
}

struct Contribution {
  float re, im, w;
};

// Reference-ordered gather of one voxel-update with generic loops (rows i ascending, columns j
// ascending, ProcessVoxelBlob fr_cpu_kernels.hpp:104-147).  Used for footprints wider than the
// unrolled NB x NB box, which only rounding at the blob edge can produce.
template <int kMode, int kOrder, bool kHalf, bool kFastMath>
__device__ inline Contribution gather_generic(const FrJob &a, int nTable, __amdgpu_buffer_rsrc_t rsrc,
                                       const float *tbl, float qx, float qy, float zSqr, float dw,
                                       uint32_t sliceOff = 0)
{
  const umpa_fr_constants &c = a.c;
  const float r = c.cBlobRadius, r2 = r * r;
  int minX = (int)ceilf(qx - r), maxX = (int)floorf(qx + r);
  int minY = (int)ceilf(qy - r), maxY = (int)floorf(qy + r);
  minX = minX < 0 ? 0 : minX;
  minY = minY < 0 ? 0 : minY;
  maxX = maxX > a.xSize - 1 ? a.xSize - 1 : maxX;
  maxY = maxY > a.ySize - 1 ? a.ySize - 1 : maxY;
  Contribution o{ 0.f, 0.f, 0.f };
  for (int i = minY; i <= maxY; ++i) {
    float dy = qy - (float)i;
    float yz = dy * dy + zSqr;
    if (yz > r2) continue;
    for (int j = minX; j <= maxX; ++j) {
      float xD = qx - (float)j;
      float d2 = xD * xD + yz;
      if (d2 > r2) continue;
      float wb;
      if constexpr (kMode == kModeLookup) {
        int aux = kFastMath ? (int)__builtin_fmaf(d2, c.cIDeltaSqrt, 0.5f)
                            : (int)(d2 * c.cIDeltaSqrt + 0.5f);
        aux = aux > nTable - 1 ? nTable - 1 : aux;
        wb = tbl[aux];
      } else {
        wb = blob_weight<kMode, kOrder>(d2, c);
      }
      float weight = wb * dw;
      float2 f = load_pixel<kHalf>(rsrc, sliceOff + (uint32_t)((i * a.xSize + j) * (kHalf ? 4 : 8)));
      o.w += weight;
      if constexpr (kFastMath) {
        o.re = __builtin_fmaf(f.x, weight, o.re);
        o.im = __builtin_fmaf(f.y, weight, o.im);
      } else {
        o.re += f.x * weight;
        o.im += f.y * weight;
      }
    }
  }
  return o;
}

// Blob weight of one candidate at squared distance d2, 0 for a candidate the reference skips
// (d2 > r^2, and d2 = +inf for box positions outside the slice).  Exact strategy: the
// reference's table position (int)(d2 * cIDeltaSqrt + 0.5); skipped candidates read the LDS
// copy's zero entry nTable.  Fast math with the table in LDS: a fused position, clamped into
// the zero entry, so +inf and every d2 past the blob edge weigh 0 without a test.
// kAlwaysRead: the global table is read for skipped candidates too.  A branch each, which spares
// their reads, is faster (box 64, 30 slices, r 1.9: 52 us, 84 without), but 36 of them, row by row,
// spill in the six-wide fast-math FP32 kernels (r 2.8, box 112, 60 slices: 437 us, 289 without).
template <int kMode, int kOrder, bool kFastMath, bool kTableLds, bool kAlwaysRead = false>
__device__ __forceinline__ float candidate_weight(float d2, float r2, int nTable, const float *tbl,
                                                  const umpa_fr_constants &c)
{
  if constexpr (kFastMath && kMode == kModeLookup && kTableLds) {
    // The reference's position (int)(d2 * cIDeltaSqrt + 0.5f): the product rounded to float,
    // then floor(t + 0.5), which v_cvt_rpi_i32_f32 computes in one instruction from the exact
    // sum; the reference's rounded sum truncates to the same integer for every t >= 0 outside
    // (0.5 - 2^-25, 0.5) (on the GPU: 2.16 M values, ties k + 0.5 and their neighbours).
    // Rounding the fused product to the nearest entry instead (one instruction less) moves
    // entries at rounding boundaries: 4.2e-5 rel-L2 from FRCPU at box 384 with 64 spaces,
    // whose central voxels carry most of the volume's norm.  Positions past the table and
    // +inf (saturated to INT_MAX) are clamped into the zero entry nTable, so candidates
    // outside the blob weigh 0 without a test.
    const float t = d2 * c.cIDeltaSqrt;
    int pos;
    asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(pos) : "v"(t));
    const uint32_t aux = (uint32_t)pos;
    typedef __attribute__((address_space(3))) const float lds_float;
    return ((lds_float *)tbl)[aux < (uint32_t)nTable ? aux : (uint32_t)nTable];
  } else {
    const bool in = d2 <= r2;
    if constexpr (kMode == kModeLookup) {
      int aux = kFastMath ? (int)__builtin_fmaf(d2, c.cIDeltaSqrt, 0.5f)
                          : (int)(d2 * c.cIDeltaSqrt + 0.5f);
      if constexpr (kTableLds) {
        return tbl[in ? aux : nTable];  // entry nTable of the LDS copy is 0
      } else {
        aux = aux > nTable - 1 ? nTable - 1 : aux;
        if constexpr (kAlwaysRead) {
          const float w = tbl[aux];
          return in ? w : 0.f;
        } else {
          return in ? tbl[aux] : 0.f;
        }
      }
    } else {
      return in ? blob_weight<kMode, kOrder>(d2, c) : 0.f;
    }
  }
}

// Branch-free gather of one voxel-update over the NB x NB candidate box around (qx, qy).
//
// Exact strategy: candidates the reference skips (outside the blob, outside the slice) read
// table[nTable] = 0, so with finite slice values they add +-0; the running sums start at +0
// and never hold -0, so the float results equal the reference's (footprints wider than 4 read
// skipped pixels past the buffer end, as zeros).  Fast-math strategy (finite slice values):
// the table index is clamped into the zero entry, so out-of-blob candidates weigh 0 without a
// test.  Rows are read whole; pixels past the slice end read 0 through the bounds-checked
// buffer.  With kShift (the caller's instantiation for jobs with FrJob::shiftBox) the box slides
// inside the slice (see below).  With kChunk the buffer covers a chunk of slices, where reading past
// one slice's end finds the next one, whose pixels (an Inf, a NaN) must not meet a weight of 0: a
// box that does not slide for its own sake then has its columns slid into the slice and its rows
// past the last not read (masking each pixel instead, FP16, r 3.2, box 64, 100 slices: 198 -> 330 us).
// Returns false when the footprint is wider than NB.
template <int kMode, int kOrder, int kNB, bool kHalf, bool kFastMath, bool kUnitWeight, bool kTableLds,
          bool kShift, bool kChunk, int kRows = 0>
__device__ __forceinline__ bool gather_box(const FrJob &a, int nTable,
                                           __amdgpu_buffer_rsrc_t rsrc, const float *tbl,
                                           float qx, float qy, float zSqr, float dw,
                                           Contribution &o, uint32_t sliceOff = 0)
{
  const umpa_fr_constants &c = a.c;
  const float r = c.cBlobRadius, r2 = r * r;
  const float inf = __builtin_inff();
  int minX = (int)ceilf(qx - r);
  int minY = (int)ceilf(qy - r);
  minX = minX < 0 ? 0 : minX;
  minY = minY < 0 ? 0 : minY;
  constexpr int kPix = kHalf ? 4 : 8;
  bool fits = true;
  float xd2[kNB], yz[kNB];
  if constexpr (kShift) {
    // The box slides inside the slice (slices of at least kNB x kNB pixels): it covers the
    // reference's bounding box [minX, maxX] x [minY, maxY] whenever that has at most kNB
    // columns and rows (the host sets shiftBox only where floor(2r) + 1 <= kNB, or 2r = kNB for
    // the widths that test for one column more), and every
    // other candidate in it lies farther than r from q, so it weighs 0 (the table's zero
    // entry; fast math: the clamp, or the last entry within 0.5 / cIDeltaSqrt of r^2), with no
    // per-candidate masking.
    minX = minX < a.xSize - kNB ? minX : a.xSize - kNB;
    minY = minY < a.ySize - kNB ? minY : a.ySize - kNB;
    // The reference's distance is the float nearest to q - j.  q - minX is exact for the radii
    // the host slides boxes for (r >= 0.5, box_can_shift): it is a multiple of q's last place
    // no larger than q, so (q - minX) - jj rounds once, to the same float.
    const float fx = qx - (float)minX, fy = qy - (float)minY;
    if constexpr (kNB == 3 || kNB == 5) {
      // where 2r = kNB: column (row) kNB of the box, if the slice has it, lies at distance
      // kNB - fx, beyond r unless fx >= kNB - r (= r: both edges exactly at distance r)
      const float edge = (float)kNB - r;
      fits = (fx < edge || minX >= a.xSize - kNB) & (fy < edge || minY >= a.ySize - kNB);
    }
#pragma unroll
    for (int jj = 0; jj < kNB; ++jj) {
      const float xD = fx - (float)jj;
      xd2[jj] = xD * xD;
    }
#pragma unroll
    for (int ii = 0; ii < kNB; ++ii) {
      const float dy = fy - (float)ii;
      yz[ii] = dy * dy + zSqr;
    }
  } else {
    int maxX = (int)floorf(qx + r), maxY = (int)floorf(qy + r);
    maxX = maxX > a.xSize - 1 ? a.xSize - 1 : maxX;
    maxY = maxY > a.ySize - 1 ? a.ySize - 1 : maxY;
    const int ny = maxY - minY;
    fits = (maxX - minX < kNB) && (ny < kNB);
    const int firstX = minX;
    if constexpr (kChunk) {
      fits = fits && a.xSize >= kNB;
      minX = minX < a.xSize - kNB ? minX : a.xSize - kNB;
    }
    const int nx = maxX - minX;
    // (float)j == (float)minX + jj exactly for slice indices
    const float fx0 = (float)minX, fy0 = (float)minY;
#pragma unroll
    for (int jj = 0; jj < kNB; ++jj) {
      const float xD = qx - (fx0 + (float)jj);
      const bool in = (jj <= nx) & (!kChunk || minX + jj >= firstX);
      xd2[jj] = in ? xD * xD : inf;
    }
#pragma unroll
    for (int ii = 0; ii < kNB; ++ii) {
      const float dy = qy - (fy0 + (float)ii);
      yz[ii] = (ii <= ny) ? dy * dy + zSqr : inf;
    }
  }
  const uint32_t rowStride = (uint32_t)(a.xSize * kPix);
  // sliceOff: the slice's byte offset within the buffer resource (0 when the resource covers
  // the slice alone)
  // (a 24-bit product where the host bounds the slice's extents, sliding boxes: a 32-bit one
  // takes four issue slots)
  uint32_t base = sliceOff + ((kShift ? __umul24((uint32_t)minY, (uint32_t)a.xSize)
                                      : (uint32_t)(minY * a.xSize)) + (uint32_t)minX) * kPix;
  // opaque, so that a row's offset is one addition and not a product of its own
  asm("" : "+v"(base));
  float w = 0.f, vr = 0.f, vi = 0.f;
  // Whole candidate rows, summed in the reference's order (rows, then columns).  Candidates
  // outside the blob or the slice weigh exactly 0 (the table's zero entry), so with finite slice
  // values they add +-0, which changes no running sum (the sums start at +0 and are never -0):
  // the result equals the reference's skip-the-pixel loop bit for bit.
  //
  // The rows go in groups of kGroup (kRows, or what the brick kernels' registers hold): all of a
  // group's pixel loads are issued, then its table reads, then its sums, each in a scheduling region
  // of its own.  Left to itself this compiler
  // orders the same code by what else the kernel holds in registers: a change elsewhere could
  // make it wait for every row before loading the next (1.42 -> 1.84 ms per 1,000-slice chunk
  // at box 256 under the exact strategy).
  constexpr int kVecs = (kNB * kPix + 15) / 16;          // 16-byte loads per row
  // Six FP32 columns go row by row: two rows' pixels and weights spilled up to 74 registers (r 2.8,
  // 500 slices, box 256: exact 5226 -> 1962 us, fast math 1463 -> 1441; r 3.6 13510 -> 8687), while
  // five columns want two (r 2.5, exact 1431 us, 1576 row by row).
  constexpr int kGroup =
    kRows ? kRows : kVecs == 1 ? kNB : kVecs == 2 ? (kNB <= 4 ? kNB : 3) : kNB == 5 ? 2 : 1;
  // wider boxes under the exact strategy mask skipped pixels, whatever their value
  constexpr bool kMask = kNB > 4 && !(kFastMath && kMode == kModeLookup && kTableLds);
  constexpr bool kSkipOutside = kChunk && !kShift;
  // The exact brick kernels' registers (12 wavefronts a CU) hold the next row's pixels beside the one
  // that is summed, so that a space's chain waits for one row, not six (r 2.8, us: a batch of one box
  // 176, 1,000 slices 3832 -> 2961, box 256, 500 slices 1962 -> 1661; fast math, with 16, spills: box
  // 256, 500 1441 -> 1486).
  constexpr bool kAhead = kGroup == 1 && kNB == 6 && kRows == 0 && !kFastMath && kTableLds;
  // fast-math FP32: a row wholly outside the blob (every candidate weighs 0) reads zeros from past
  // the slice end instead of its pixels, a quarter of the rows at r = 1.9
  constexpr bool kSkipRows = kFastMath && !kHalf;
  auto row_offset = [&](int k) {
    const bool read = kSkipRows ? yz[k] <= r2 : !kSkipOutside || yz[k] < inf;
    return read ? base + k * rowStride : kOutOfRange;
  };
  Pixel<kHalf> ahead[kNB];
  if constexpr (kAhead) load_row<kHalf, kNB>(rsrc, row_offset(0), ahead);
#pragma unroll
  for (int g = 0; g < kNB; g += kGroup) {
    Pixel<kHalf> px[kGroup][kNB];
    float wr[kGroup][kNB];
    if constexpr (kAhead) {
#pragma unroll
      for (int jj = 0; jj < kNB; ++jj) px[0][jj] = ahead[jj];
      if (g + 1 < kNB) load_row<kHalf, kNB>(rsrc, row_offset(g + 1), ahead);
    } else {
#pragma unroll
      for (int i = 0; i < kGroup; ++i) {
        if (g + i >= kNB) continue;
        load_row<kHalf, kNB>(rsrc, row_offset(g + i), px[i]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kGroup; ++i) {
      if (g + i >= kNB) continue;
#pragma unroll
      for (int jj = 0; jj < kNB; ++jj)
        wr[i][jj] = candidate_weight<kMode, kOrder, kFastMath, kTableLds,
                                     kNB == 6 && kFastMath && !kHalf>(xd2[jj] + yz[g + i], r2,
                                                                      nTable, tbl, c);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kGroup; ++i) {
      if (g + i >= kNB) continue;
#pragma unroll
      for (int jj = 0; jj < kNB; ++jj) {
        float fre = px[i][jj].re(), fim = px[i][jj].im();
        if constexpr (kMask) {
          const bool in = xd2[jj] + yz[g + i] <= r2;
          fre = in ? fre : 0.f;
          fim = in ? fim : 0.f;
        }
        const float weight = kUnitWeight ? wr[i][jj] : wr[i][jj] * dw;
        w += weight;
        if constexpr (kFastMath) {
          vr = __builtin_fmaf(fre, weight, vr);
          vi = __builtin_fmaf(fim, weight, vi);
        } else {
          vr += fre * weight;
          vi += fim * weight;
        }
      }
    }
  }
  o.re = vr;
  o.im = vi;
  o.w = w;
  return fits;
}

// The contribution of a voxel-update of a space with weight `dw`: the candidate box, or the
// general loop where the footprint is wider.  The exact strategy multiplies every candidate's
// weight by dw as the reference does (`unit`, wave-uniform: all weights are 1, which multiply
// nothing); fast math sums with unit weights and scales the three sums.
template <int kMode, int kOrder, int kNB, bool kHalf, bool kFastMath, bool kTableLds, bool kShift,
          bool kChunk, int kRows = 0>
__device__ __forceinline__ Contribution gather_update(const FrJob &a, int nTable,
                                                      __amdgpu_buffer_rsrc_t rsrc,
                                                      const float *tbl, float qx, float qy,
                                                      float zSqr, float dw, bool unit, float scale,
                                                      uint32_t sliceOff = 0)
{
  Contribution o;
  if constexpr (kFastMath) {
    if (!gather_box<kMode, kOrder, kNB, kHalf, kFastMath, true, kTableLds, kShift, kChunk, kRows>(
          a, nTable, rsrc, tbl, qx, qy, zSqr, 1.f, o, sliceOff))
      o = gather_generic<kMode, kOrder, kHalf, kFastMath>(a, nTable, rsrc, tbl, qx, qy, zSqr, 1.f,
                                                          sliceOff);
    const float s = kHalf ? dw * scale : dw;
    o.re *= s;
    o.im *= s;
    o.w *= dw;
  } else {
    bool fits;
    if (unit) {
      fits = gather_box<kMode, kOrder, kNB, kHalf, kFastMath, true, kTableLds, kShift, kChunk, kRows>(
        a, nTable, rsrc, tbl, qx, qy, zSqr, dw, o, sliceOff);
    } else {
      fits = gather_box<kMode, kOrder, kNB, kHalf, kFastMath, false, kTableLds, kShift, kChunk, kRows>(
        a, nTable, rsrc, tbl, qx, qy, zSqr, dw, o, sliceOff);
    }
    if (!fits)
      o = gather_generic<kMode, kOrder, kHalf, kFastMath>(a, nTable, rsrc, tbl, qx, qy, zSqr, dw,
                                                          sliceOff);
  }
  return o;
}

// The blob modes whose weights are evaluated (gather_evaluated), not read from a table.
__host__ __device__ constexpr bool evaluates_blob(int mode)
{
  return mode == kModeFastKaiser || mode == kModePreciseKaiser;
}
constexpr int kBlobRows = 2;                         // candidate rows evaluated together
constexpr int kBlobList = 64 * 4 * kBlobRows;        // floats of LDS a wavefront needs for them

// gather_update for the evaluated blob modes, called by the whole wavefront (lanes without a
// voxel-update: act false).  An evaluation is some 60 instructions (two divisions' and a square
// root's worth among them), and under half of the 4 x 4 candidates lie inside the blob, so a
// candidate per lane and step left most lanes idle.  Here the squared distances of two rows'
// candidates inside the blob go to `list` (kBlobList floats of the wavefront's LDS) one behind
// another, full wavefronts turn them into weights in place, and every lane reads its own back:
// the same float for each candidate, summed in the reference's order, 0 for the others.
// Box 128, 300 slices: 409 -> 366 us (bound by the spaces' chain through the heaviest bricks).
template <int kMode, int kOrder>
__device__ __forceinline__ Contribution gather_evaluated(const FrJob &a, __amdgpu_buffer_rsrc_t rsrc,
                                                         float *list, int lane, bool act, float qx,
                                                         float qy, float zSqr, float dw,
                                                         uint32_t sliceOff = 0)
{
  constexpr int kNB = 4, kPix = 8;
  const umpa_fr_constants &c = a.c;
  const float r = c.cBlobRadius, r2 = r * r;
  int minX = (int)ceilf(qx - r), maxX = (int)floorf(qx + r);
  int minY = (int)ceilf(qy - r), maxY = (int)floorf(qy + r);
  minX = minX < 0 ? 0 : minX;
  minY = minY < 0 ? 0 : minY;
  maxX = maxX > a.xSize - 1 ? a.xSize - 1 : maxX;
  maxY = maxY > a.ySize - 1 ? a.ySize - 1 : maxY;
  const int ny = maxY - minY;
  const bool fits = (maxX - minX < kNB) & (ny < kNB) & (a.xSize >= kNB);
  const bool box = act & fits;
  // The box's columns slide into the slice and its rows past the last are not read: the buffer may
  // hold other slices behind this one, whose pixels (an Inf, a NaN) must not meet a weight of 0.
  // (Box 128, 300 slices: 307 -> 309 us; masking each pixel instead, 329.)  A column before minX
  // needs no test: it lies farther than r from qx, by what qx - j, exact there, and its square keep.
  const int x0 = minX < a.xSize - kNB ? minX : a.xSize - kNB;
  const int nx = maxX - x0;
  const float fx0 = (float)x0, fy0 = (float)minY;
  const uint32_t rowStride = (uint32_t)(a.xSize * kPix);
  const uint32_t base = sliceOff + (uint32_t)(minY * a.xSize + x0) * kPix;
  Contribution o{ 0.f, 0.f, 0.f };
#pragma unroll
  for (int g = 0; g < kNB; g += kBlobRows) {
    Pixel<false> px[kBlobRows][kNB];
    int at[kBlobRows][kNB];
    bool in[kBlobRows][kNB];
#pragma unroll
    for (int i = 0; i < kBlobRows; ++i)
      load_row<false, kNB>(rsrc, (box & (g + i <= ny)) ? base + (g + i) * rowStride : kOutOfRange, px[i]);
    __builtin_amdgcn_sched_barrier(0);
    int total = 0;
#pragma unroll
    for (int i = 0; i < kBlobRows; ++i) {
      const float dy = qy - (fy0 + (float)(g + i));
      const float yz = dy * dy + zSqr;
#pragma unroll
      for (int j = 0; j < kNB; ++j) {
        const float xD = qx - (fx0 + (float)j);
        const float d2 = xD * xD + yz;
        in[i][j] = box & (g + i <= ny) & (j <= nx) & (d2 <= r2);
        const unsigned long long m = __ballot(in[i][j]);
        at[i][j] = (int)lanes_below(m, (unsigned)total);
        if (in[i][j]) list[at[i][j]] = d2;
        total += __popcll(m);
      }
    }
    wave_sync();
    for (int k = lane; k < total; k += 64) list[k] = blob_weight<kMode, kOrder>(list[k], c);
    wave_sync();
#pragma unroll
    for (int i = 0; i < kBlobRows; ++i)
#pragma unroll
      for (int j = 0; j < kNB; ++j) {
        const float wb = in[i][j] ? list[at[i][j]] : 0.f;
        const float weight = wb * dw;
        o.w += weight;
        o.re += px[i][j].re() * weight;
        o.im += px[i][j].im() * weight;
      }
    wave_sync();
  }
  if (act && !fits)
    o = gather_generic<kMode, kOrder, false, false>(a, 0, rsrc, nullptr, qx, qy, zSqr, dw, sliceOff);
  return o;
}

// ProcessVoxel (fr_cpu_kernels.hpp:50-67): the nearest pixel, weight = space weight.
template <bool kHalf>
__device__ __forceinline__ Contribution gather_nearest(const FrJob &a, __amdgpu_buffer_rsrc_t rsrc,
                                                       float qx, float qy, float dw, float scale,
                                                       uint32_t sliceOff = 0)
{
  int ix = (int)(qx + 0.5f);
  ix = ix > a.xSize - 1 ? a.xSize - 1 : ix;
  ix = ix < 0 ? 0 : ix;
  int iy = (int)(qy + 0.5f + (float)(a.c.cMaxVolumeIndexYZ / 2));
  iy = iy > a.ySize - 1 ? a.ySize - 1 : iy;
  iy = iy < 0 ? 0 : iy;
  const float wgt = 1.f * dw;
  float2 f = load_pixel<kHalf>(rsrc, sliceOff + (uint32_t)((iy * a.xSize + ix) * (kHalf ? 4 : 8)));
  if constexpr (kHalf) {
    f.x *= scale;
    f.y *= scale;
  }
  return { f.x * wgt, f.y * wgt, wgt };
}

// The reference's per-voxel predicate for one (voxel, space) pair in blob mode
// (ProcessVoxelBlob, fr_cpu_kernels.hpp:83-102) plus membership in the reference traversal of
// the space.  (qx, qy, zSqr) are returned for the gather, qy already shifted to slice rows.
// With kFma the rotation is evaluated with fused multiply-adds (fewer instructions; q moves by
// an ulp, which changes which nearly-zero-weight candidates at the blob edge are counted).  The
// kernels use the reference's separate products: fused, the weights of small volumes drift to
// about 1e-5 of FRCPU's, the edge of the fast-math strategy's tolerance.
template <bool kFma>
__device__ __forceinline__ bool blob_predicate(const umpa_traverse_space &s, const float (*t)[3],
                                               const umpa_fr_constants &c,
                                               int x, int y, int z, float px, float py, float pz,
                                               bool brickInside, float &qx, float &qy,
                                               float &zSqr)
{
  const float r = c.cBlobRadius;
  float qz;
  if constexpr (kFma) {
    qx = __builtin_fmaf(t[0][2], pz, __builtin_fmaf(t[0][1], py, t[0][0] * px));
    qy = __builtin_fmaf(t[1][2], pz, __builtin_fmaf(t[1][1], py, t[1][0] * px));
    qz = __builtin_fmaf(t[2][2], pz, __builtin_fmaf(t[2][1], py, t[2][0] * px));
  } else {
    qx = t[0][0] * px + t[0][1] * py + t[0][2] * pz;
    qy = t[1][0] * px + t[1][1] * py + t[1][2] * pz;
    qz = t[2][0] * px + t[2][1] * py + t[2][2] * pz;
  }
  zSqr = qz * qz;
  // & rather than &&: every test is evaluated, so the record's fields load together
  bool pass = !(qx < -r) & !(zSqr > r * r);
  qy += (float)(c.cMaxVolumeIndexYZ / 2);
  if (!brickInside) {
    // the sphere test, and the traversal: the column must lie in the AABB's plane orthogonal
    // to `dir` (both hold for every voxel of a brick that lies inside them: brick_inside)
    const float dsq = px * px + py * py + pz * pz;
    pass = pass & !(dsq > s.maxDistanceSqr);
    if (s.dir == 0) {
      pass = pass & (x >= s.minX) & (x <= s.maxX) & (y >= s.minY) & (y <= s.maxY);
    } else if (s.dir == 1) {
      pass = pass & (x >= s.minX) & (x <= s.maxX) & (z >= s.minZ) & (z <= s.maxZ);
    } else {
      pass = pass & (y >= s.minY) & (y <= s.maxY) & (z >= s.minZ) & (z <= s.maxZ);
    }
  }
  // ... and the voxel must lie in the column's slab between the two bounding planes.  A voxel
  // whose |qz| is at least 0.001 inside the blob radius is between the planes by at least that
  // much along the column (the axis of the normal's largest component), five times the float
  // error of the plane evaluation (about 2e-4 at coordinates up to 256), so the floor/ceil
  // range holds it; only voxels nearer the slab faces take the reference's exact test, whose
  // two IEEE divisions a wave runs whenever one lane needs it (a band of 0.01 sent about a
  // quarter of the batches there).
  if (pass && !(fabsf(qz) <= r - 0.001f)) {
    pass = visited_blob(s, x, y, z, c.cMaxVolumeIndexX, c.cMaxVolumeIndexYZ);
  }
  return pass;
}

// The blob table and its zero entry into LDS, eight loads of a thread in flight at a time (one
// at a time, a workgroup's 40 KB took as many round trips to L2 as it has rounds).
template <int kThreads>
__device__ __forceinline__ void stage_table(float *dst, const float *__restrict__ src, int n)
{
  for (int i0 = threadIdx.x; i0 < n; i0 += 8 * kThreads) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = i0 + k * kThreads < n ? src[i0 + k * kThreads] : 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (i0 + k * kThreads < n) dst[i0 + k * kThreads] = v[k];
  }
  if (threadIdx.x == 0) dst[n] = 0.f;
  __syncthreads();
}

// Copies a wave-uniform value into scalar registers, dword by dword: a job record read from
// memory at a uniform address then lives in SGPRs like a kernel argument.
template <typename T>
__device__ __forceinline__ T make_uniform(const T &v)
{
  static_assert(sizeof(T) % 4 == 0, "dword-sized records only");
  int w[sizeof(T) / 4];
  __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
  for (int i = 0; i < (int)(sizeof(T) / 4); ++i) w[i] = __builtin_amdgcn_readfirstlane(w[i]);
  T out;
  __builtin_memcpy(&out, w, sizeof(T));
  return out;
}

// The job with its pointers marked as global memory.  Pointers read from a record could name any
// address space, and a flat load counts as an LDS access too: every wait for LDS then also waited
// for the prefetch of the next space's record (seven mixed FP16 jobs 3873 -> 3710 us, four-job
// serving tick 1357 -> 1309).
__device__ __forceinline__ FrJob global_pointers(FrJob a)
{
#define UMPA_GLOBAL(p) p = (decltype(p))(__attribute__((address_space(1))) char *)(uintptr_t)(p)
  UMPA_GLOBAL(a.volume);
  UMPA_GLOBAL(a.weights);
  UMPA_GLOBAL(a.fft);
  UMPA_GLOBAL(a.scales);
  UMPA_GLOBAL(a.spaces);
#undef UMPA_GLOBAL
  return a;
}

}  // namespace umpa
