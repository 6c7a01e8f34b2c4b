// Items of the time-blocked marches (cpml_tb2d.h, cpml_tb3d.hip) and the
// addresses of one lane of them.  The marches read through plain pointers, without the range check of a
// buffer resource, and lanes beyond a tile's ring read too (nothing uses their
// values), so every coordinate is clamped here: the fields' to the zero ghost
// points around the grid, the memory variables' to the grid itself, since their
// rows have no ghost points.  Host code as well, so that the bounds can be
// checked without a GPU (tests/native/address_audit.cpp).
#pragma once

#include <algorithm>

#include "cpml_internal.h"

namespace cpml {

__host__ __device__ __forceinline__ int clamp_to(int v, int lo, int hi) {
  const int a = v < lo ? lo : v;
  return a < hi ? a : hi;
}
__host__ __device__ __forceinline__ int smaller(int a, int b) { return a < b ? a : b; }

// Item number `item` of one grid: strip ts, rows [jb, je), class (bit 0: it may
// touch the x slabs or faces, bit 1: y).  Items with C-PML code in chunks of js
// rows: those of the x slabs' strips (all rows), then those of the other strips
// (rows below y0, then from y1); they are few, with more code each, and shorter
// chunks end sooner.  Then the slab-free ones: strips [sx0, sx1) x chunks of jc
// rows of [y0, y1).
struct Tb2dItem {
  int ts, jb, je, cls;
};
template <typename T>
__host__ __device__ __forceinline__ Tb2dItem tb2d_item_at(const TB2D<T> &P, const Tb2dItems &n,
                                                          int item) {
  const int bx = P.sx1 - P.sx0, ny = P.a.ny;
  Tb2dItem o;
  if (item < n.edge) {
    const int wx = P.nstrips - bx, u = item % wx;
    o.ts = u < P.sx0 ? u : u + bx;
    o.jb = item / wx * P.js;
    o.je = smaller(o.jb + P.js, ny);
    o.cls = o.jb >= P.y0 && o.je <= P.y1 ? 1 : 3;
  } else if (item < n.edge + n.cap) {
    const int u = item - n.edge, c = u / bx, low = (P.y0 + P.js - 1) / P.js;
    const int end = c < low ? P.y0 : ny;
    o.ts = P.sx0 + u % bx;
    o.jb = c < low ? c * P.js : P.y1 + (c - low) * P.js;
    o.je = smaller(o.jb + P.js, end);
    o.cls = 2;
  } else {
    const int u = item - n.edge - n.cap;
    o.ts = P.sx0 + u % bx;
    o.jb = P.y0 + u / bx * P.jc;
    o.je = smaller(o.jb + P.jc, P.y1);
    o.cls = 0;
  }
  return o;
}

// The same items for a list of many grids, to emit(item), every class on its own
// rows (the batch: strips fastest).
template <typename T, typename F>
inline void tb2d_list(const TB2D<T> &P, F &&emit) {
  auto rows = [&](int cls, int j0, int j1, int step, int t0, int t1) {
    for (int r = j0; r < j1; r += step)
      for (int t = t0; t < t1; ++t) emit(Tb2dItem{t, r, std::min(r + step, j1), cls});
  };
  rows(0, P.y0, P.y1, P.jc, P.sx0, P.sx1);
  for (int r = 0; r < P.a.ny; r += P.js) {  // strips at the x slabs
    const int e = std::min(r + P.js, P.a.ny), cls = r >= P.y0 && e <= P.y1 ? 1 : 3;
    rows(cls, r, e, P.js, 0, P.sx0);
    rows(cls, r, e, P.js, P.sx1, P.nstrips);
  }
  rows(2, 0, P.y0, P.js, P.sx0, P.sx1);
  rows(2, P.y1, P.a.ny, P.js, P.sx0, P.sx1);
}

// Column i of a 2D item whose march reads rows from r0 up; SX, SY: the item may
// touch the x, y slabs or faces (else its rows lie strictly inside the grid).
template <typename T, bool SX, bool SY>
struct Tb2dLane {
  int ny, rl;          // rl: row of the corner
  long corner;         // element of the ghost corner (-1, rl), from the interior origin
  unsigned vo, ldb;    // byte offset of the column there, bytes per row
  unsigned mo;         // byte offset of the column in a row of a y memory variable
  bool inx;            // the column lies in the x slab
  long sxb;            // x memory variables: element of row 0 of the column, ...
  unsigned sxw;        // ... and elements from row to row

  __host__ __device__ __forceinline__ Tb2dLane(int i, int r0, int nx, int ny_, long ld,
                                               const Slab &sx)
      : ny(ny_) {
    constexpr unsigned es = sizeof(T);
    rl = r0 < -1 ? -1 : r0;
    corner = (long)rl * ld - 1;
    vo = (unsigned)(clamp_to(i, -1, nx) + 1) * es;
    ldb = (unsigned)ld * es;
    mo = (unsigned)clamp_to(i, 0, nx - 1) * es;
    inx = SX && sx.in(i);
    sxw = i < sx.wl ? sx.wl : sx.wr;
    sxb = inx ? sx.at(i, 0, ny) : 0;
  }
  // byte offset of row j of a field from the corner
  __host__ __device__ __forceinline__ unsigned at(int j) const {
    const int jj = SY ? clamp_to(j, -1, ny) : j;
    return (unsigned)(jj - rl) * ldb + vo;
  }
  // element of row j (inside the grid) of an x memory variable, where inx
  __host__ __device__ __forceinline__ long ox(int j) const {
    return sxb + (long)(sxw * (unsigned)j);
  }
};

struct Tb3dTile {
  int i0, j0, kb, ke, tx, ty;
};

// Index of the u-th tile of one axis' class: the clean tiles [c0, c1) when
// S is false, else the tiles outside them (below c0, then from c1).
template <bool S>
__host__ __device__ __forceinline__ int axis_tile(int u, int c0, int c1) {
  if (!S) return c0 + u;
  return u < c0 ? u : c1 + (u - c0);
}
template <bool S>
__host__ __device__ __forceinline__ int axis_count(int n, int c0, int c1) {
  return S ? n - (c1 - c0) : c1 - c0;
}

// Tile t of class (SX, SY, SZ).  Along each axis the tiles (z: chunks) whose
// points and ring avoid that axis' slabs form a range (box, zn); the
// class covers the product of the clean (flag false) or slab (flag true) tiles
// of each axis, x fastest, then y, then z.
template <bool SX, bool SY, bool SZ, typename P>
__host__ __device__ __forceinline__ Tb3dTile tb3d_tile_at(const P &Q, int t, int nx, int ny, int nz,
                                                          int kchunk) {
  const int ntx = (nx + Q.ow - 1) / Q.ow, nty = (ny + Q.ty - 1) / Q.ty;
  const int cx = axis_count<SX>(ntx, Q.box[0], Q.box[1]);
  const int cy = axis_count<SY>(nty, Q.box[2], Q.box[3]);
  Tb3dTile f;
  f.tx = axis_tile<SX>(t % cx, Q.box[0], Q.box[1]);
  f.ty = axis_tile<SY>((t / cx) % cy, Q.box[2], Q.box[3]);
  const int tz = axis_tile<SZ>(t / (cx * cy), Q.zn[0], Q.zn[0] + Q.zn[1]);
  f.i0 = f.tx * Q.ow;
  f.j0 = f.ty * Q.ty;
  if (tz < Q.zn[0]) {
    f.kb = tz * kchunk;
    f.ke = smaller(f.kb + kchunk, Q.z0);
  } else if (tz < Q.zn[0] + Q.zn[1]) {
    f.kb = Q.z0 + (tz - Q.zn[0]) * kchunk;
    f.ke = smaller(f.kb + kchunk, Q.z1);
  } else {
    f.kb = Q.z1 + (tz - Q.zn[0] - Q.zn[1]) * kchunk;
    f.ke = smaller(f.kb + kchunk, nz);
  }
  return f;
}

// Tiles along one axis (size B, extent n, slab widths wl, wr) whose points and
// ring of g avoid both slabs: [t0, t1), empty when t1 <= t0.
inline void clean_tiles(int n, int B, int g, int wl, int wr, int &t0, int &t1) {
  const int nt = (n + B - 1) / B;
  t0 = t1 = 0;
  bool seen = false;
  for (int t = 0; t < nt; ++t) {
    const int lo = t * B - g, hi = t * B + B - 1 + g;
    const bool clean = lo >= wl && hi < n - wr;
    if (clean && !seen) t0 = t, seen = true;
    if (clean) t1 = t + 1;
    else if (seen) break;
  }
}

// Fills P.ty, box, z0, z1, zn and ncls from a, ow (and the steps and wavefronts).
// Returns the tiles of the XCD that gets most.
template <typename T>
inline long tb3d_split(int nt, int nw, TB3D<T> &P) {
  const Step3D<T> &p = P.a;
  P.ty = nw - 2 * nt;
  // z regions: planes whose march (2 nt - 1 planes of ring) avoids the z slabs
  // and the first and last plane
  const int g = 2 * nt - 1, nz = p.nz, kc = p.kchunk;
  int z0 = std::max(p.sz.wl, 1) + g;
  int z1 = nz - std::max(p.sz.wr, 1) - g;
  if (z1 <= z0) z0 = z1 = 0;
  P.z0 = z0;
  P.z1 = z1;
  P.zn[0] = (z0 + kc - 1) / kc;
  P.zn[1] = (z1 - z0 + kc - 1) / kc;
  P.zn[2] = (nz - z1 + kc - 1) / kc;
  clean_tiles(p.nx, P.ow, nt, std::max(p.sx.wl, 1), std::max(p.sx.wr, 1), P.box[0], P.box[1]);
  clean_tiles(p.ny, P.ty, nt, std::max(p.sy.wl, 1), std::max(p.sy.wr, 1), P.box[2], P.box[3]);
  if (P.box[1] < P.box[0]) P.box[0] = P.box[1] = 0;
  if (P.box[3] < P.box[2]) P.box[2] = P.box[3] = 0;
  const int n[3] = {(p.nx + P.ow - 1) / P.ow, (p.ny + P.ty - 1) / P.ty,
                    P.zn[0] + P.zn[1] + P.zn[2]};
  long most = 0;  // tiles of the XCD that gets most
  for (int c = 0; c < 8; ++c) {
    const int cx = c & 1 ? n[0] - (P.box[1] - P.box[0]) : P.box[1] - P.box[0];
    const int cy = c & 2 ? n[1] - (P.box[3] - P.box[2]) : P.box[3] - P.box[2];
    const int cz = c & 4 ? n[2] - P.zn[1] : P.zn[1];
    P.ncls[c] = cx * cy * cz;
    most += (P.ncls[c] + 7) / 8;
  }
  return most;
}

// Column (i, j) of a 3D tile whose march reads planes from k0 up; SX, SY, SZ: the
// tile may touch that axis' slabs or faces.
template <typename T, bool SX, bool SY, bool SZ>
struct Tb3dLane {
  int nz, kl;              // kl: plane of the corner
  long corner;             // element of the ghost corner (-1, -1, kl)
  unsigned vo, psb;        // byte offset of the column there, bytes per plane
  bool inx, iny;           // the column lies in that axis' slab
  unsigned mxo, myo, mzo;  // byte offsets inside a plane of the memory variables
  long mxs, mys, mzs;      // elements of such a plane

  __host__ __device__ __forceinline__ Tb3dLane(int i, int j, int k0, const Step3D<T> &p)
      : nz(p.nz) {
    constexpr unsigned es = sizeof(T);
    const int ic = clamp_to(i, -1, p.nx), jc = clamp_to(j, -1, p.ny);
    const int im = clamp_to(i, 0, p.nx - 1), jm = clamp_to(j, 0, p.ny - 1);
    kl = k0 < -1 ? -1 : k0;
    corner = (long)kl * p.ps - p.ld - 1;
    vo = (unsigned)(((long)(jc + 1) * p.ld + (ic + 1)) * (long)es);
    psb = (unsigned)(p.ps * (long)es);
    inx = SX && p.sx.in(i);
    iny = SY && p.sy.in(j);
    mxo = inx ? (unsigned)p.sx.at(i, jm, p.ny) * es : 0u;
    myo = iny ? ((unsigned)im + (unsigned)p.mld * (unsigned)p.sy.s(j)) * es : 0u;
    mzo = ((unsigned)im + (unsigned)p.mld * (unsigned)jm) * es;
    mxs = (long)p.sx.w * p.ny;
    mys = p.mld * p.sy.w;
    mzs = p.mld * p.ny;
  }
  // byte offset of plane k of a field from the corner
  __host__ __device__ __forceinline__ unsigned at(int k) const {
    const int kk = SZ ? clamp_to(k, -1, nz) : k;
    return (unsigned)(kk - kl) * psb + vo;
  }
};

}  // namespace cpml
