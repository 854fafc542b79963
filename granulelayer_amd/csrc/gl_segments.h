// The dX kernels' walk over the segment table of the input-major edges (gl_edges.hip): the segments of
// one feature range that lie in a wave's unit range, in chunks of up to 64 edges.  Plain arithmetic
// that compiles for the host too; opaque and wave_uniform are the includer's.
#pragma once

#include <stdint.h>

namespace gl {

// A wave's rows of the table: segment i (0 <= i < n) belongs to unit[i] and holds the edges
// [begin[i], begin[i + 1]).  The whole table can hold 2^31 segments (MAX_SLOTS slots of 16 edges each),
// past the reach of a 32-bit byte offset; a wave's rows are at most one per unit (at most MAX_SLOTS), so
// 32-bit offsets from their first row reach all of them.
struct DxSegs {
  const int32_t* unit;
  const uint32_t* begin;
  int n;
};

// first segment in [a, b) whose unit is at least u (b: none); units ascend
__host__ __device__ __forceinline__ uint32_t dx_seg_bound(const int32_t* seg_unit, uint32_t a, uint32_t b, int u) {
  while (a < b) {
    const uint32_t mid = a + (b - a) / 2;  // a + b passes 2^32 for the table's last rows
    if (seg_unit[mid] < u) a = mid + 1; else b = mid;
  }
  return a;
}

// the segments of feature range F with units in [u_lo, u_hi)
__host__ __device__ __forceinline__ DxSegs dx_segs(const uint32_t* seg_ptr, const int32_t* seg_unit,
                                                   const uint32_t* seg_begin, int F, int u_lo, int u_hi) {
  const uint32_t lo = dx_seg_bound(seg_unit, seg_ptr[F], seg_ptr[F + 1], u_lo);
  const uint32_t hi = dx_seg_bound(seg_unit, lo, seg_ptr[F + 1], u_hi);
  return DxSegs{seg_unit + lo, seg_begin + lo, (int)(hi - lo)};
}

struct DxChunk {
  int si;           // segment (row of the wave's DxSegs)
  unsigned e, end;  // chunk begin, segment end (edge positions)
  int u;            // unit of the segment
};

__host__ __device__ __forceinline__ DxChunk dx_first(const DxSegs& s) {
  return DxChunk{0, s.begin[0], s.begin[1], s.unit[0]};
}

__host__ __device__ __forceinline__ void dx_next(const DxSegs& s, DxChunk& c) {
  if (c.e + 64 < c.end) {
    c.e += 64;
  } else {
    c.si += 1;
    if (c.si < s.n) {
      c.e = c.end;
      c.end = s.begin[c.si + 1];
      c.u = s.unit[c.si];
    }
  }
}

// dx_next with the segment table read one step ahead: (pe, pu) hold the end and the unit of
// segment c.si + 1, loaded by the step that entered segment c.si; their loads land by the next
// loop-top wait, so no wait for them sits behind a chunk copy.  The opaque
// index keeps the offsets in vector registers: no 64-bit scalar address arithmetic.
__host__ __device__ __forceinline__ void dx_seg_ahead(const DxSegs& s, int si, unsigned& pe, unsigned& pu) {
  if (si + 1 < s.n) {
    const unsigned o = (unsigned)opaque(si) * 4u;
    pe = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(s.begin) + (o + 8u));
    pu = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(s.unit) + (o + 4u));
  }
}
__host__ __device__ __forceinline__ void dx_next_ahead(const DxSegs& s, DxChunk& c, unsigned& pe, unsigned& pu) {
  if (c.e + 64 < c.end) {
    c.e += 64;
  } else {
    c.si += 1;
    if (c.si < s.n) {
      c.e = c.end;
      c.end = wave_uniform(pe);
      c.u = (int)wave_uniform(pu);
      dx_seg_ahead(s, c.si, pe, pu);
    }
  }
}

}  // namespace gl
