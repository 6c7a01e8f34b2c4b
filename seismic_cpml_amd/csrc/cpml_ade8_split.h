// How a step of the ADE-PML RK4 kernels (cpml_ade8.hip) is cut into items: the box
// that takes two stages per pass, its strips and chunks, and the tiles of the
// frame around it.  Host code as well, so that the split and the addresses of
// the unchecked loads can be verified without a GPU.
#pragma once

#include <algorithm>

#include "cpml_internal.h"

namespace cpml {

// rows per 64-column block; measured at 4096^2 (float, full step): 1 row
// 8.84, 2 rows 9.00, 4 rows 8.91, 8 rows 8.32, 16 rows 8.13 Gcell/s
constexpr int ATY = 2;
constexpr int PG = 8;    // ring columns of a pair's strip (4 per stage)
constexpr int PW = 48;   // columns it owns

// The points whose ADE memories are updated (Fortran indices).
__host__ __device__ __forceinline__ bool ade_band(int I, int J, int nx, int ny, int npml) {
  return I <= npml + 2 || I >= nx - npml - 2 || J <= npml + 2 || J >= ny - npml - 2;
}

// Points [x0, x1) x [y0, y1) of the grid.
struct AdeBox {
  int x0, x1, y0, y1;
  __host__ __device__ bool in(int i, int j) const {
    return i >= x0 && i < x1 && j >= y0 && j < y1;
  }
};
// The same with `by` fewer points on each side (none if it is empty).
inline __host__ __device__ AdeBox shrink(AdeBox b, int by) {
  return b.x1 > b.x0 ? AdeBox{b.x0 + by, b.x1 - by, b.y0 + by, b.y1 - by} : b;
}

// Tiles of 64 x ATY points over the grid but for a box: below it, left and right
// of it, above it (whole rows).  An empty box leaves the whole grid.
struct AdeFrame {
  static constexpr int TX = 64;
  AdeBox below, above, left, right;
  static __host__ __device__ int count(AdeBox b) {
    return (b.x1 - b.x0 + TX - 1) / TX * ((b.y1 - b.y0 + ATY - 1) / ATY);
  }
  __host__ __device__ AdeFrame(int nx, int ny, AdeBox b) {
    const bool none = b.x1 <= b.x0;
    if (none) b = AdeBox{0, nx, 0, 0};
    below = AdeBox{0, nx, 0, b.y0};
    above = AdeBox{0, nx, b.y1, ny};
    left = AdeBox{0, b.x0, b.y0, b.y1};
    right = AdeBox{b.x1, nx, b.y0, b.y1};
  }
  __host__ __device__ int tiles() const {
    return count(below) + count(above) + count(left) + count(right);
  }
  // The part that tile t lies in; t becomes its number there.
  __host__ __device__ AdeBox part(int &t) const {
    const int n0 = count(below), n1 = n0 + count(left), n2 = n1 + count(right);
    const AdeBox b = t < n0 ? below : t < n1 ? left : t < n2 ? right : above;
    t -= t < n0 ? 0 : t < n1 ? n0 : t < n2 ? n1 : n2;
    return b;
  }
};

// The points whose two stages see neither band nor edges: the first stage's
// points (4 around them) lie outside the band, its stencil (8 around) off the
// edges; whole 64-byte sectors from the left.  Empty for grids whose step a
// march's length sets: 500 x 600 float 57 us with single stages, 96 with pairs,
// 1000 x 1200 135 and 127, 4096^2 1847 and 907; double 500 x 600 97 and 115, 1000 x
// 900 203 and 171, 2800^2 1960 and 943.
template <typename T>
inline AdeBox ade_pair_box(int nx, int ny, int npml) {
  const int lo = std::max(npml + 6, 9), sector = 64 / (int)sizeof(T);
  const AdeBox b{(lo + sector - 1) / sector * sector, std::min(nx - npml - 7, nx - 9), lo,
                 std::min(ny - npml - 7, ny - 9)};
  if (b.x1 - b.x0 < 64 || b.y1 - b.y0 < 64 ||
      (double)(b.x1 - b.x0) * (b.y1 - b.y0) * sizeof(T) < 4e6)
    return AdeBox{0, 0, 0, 0};
  return b;
}

// Items of the pairs: strips of PW columns x chunks of jc rows of the box.
struct AdePairs {
  AdeBox box;
  int jc;
  __host__ __device__ int strips() const { return (box.x1 - box.x0 + PW - 1) / PW; }
  __host__ __device__ int count() const { return strips() * ((box.y1 - box.y0 + jc - 1) / jc); }
  // columns [c0, c0 + PW) and rows [jb, je) of item t
  __host__ __device__ void item(int t, int &c0, int &jb, int &je) const {
    const int ns = strips();
    c0 = box.x0 + t % ns * PW;
    jb = box.y0 + t / ns * jc;
    je = jb + jc < box.y1 ? jb + jc : box.y1;
  }
};
// Rows of an item: as many items as fit in flight, 16 (its 16 ring rows cost as
// much) to 64 (4096^2 float 16, 32, 64 and 128 rows 1013, 951, 923 and 942 us per
// step; 2000 x 2400 365, 341, 350 and 570; 1000 x 900 double 203, 182, 292, 521).
template <typename T>
inline AdePairs ade_pairs(AdeBox box) {
  AdePairs p{box, 16};
  p.jc = std::clamp((int)((double)p.strips() * (box.y1 - box.y0) / (sizeof(T) == 4 ? 3000 : 600)),
                    16, 64);
  return p;
}

// Byte offset of column i in a row, for all 64 columns from c0 - PG of a strip
// (those past the grid read its last column; nothing uses them).
template <typename T>
__host__ __device__ __forceinline__ unsigned ade_pair_offset(int i, int nx) {
  return (unsigned)((i < nx - 1 ? i : nx - 1) * (int)sizeof(T));
}

}  // namespace cpml
