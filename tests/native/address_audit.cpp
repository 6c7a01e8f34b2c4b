// Addresses of the marches that read through plain pointers, over random grids,
// slabs, strips and chunks, every item and every lane: time-blocked 2D and 3D
// (cpml_tb_geom.h) and the ADE-RK4 pairs of stages (cpml_ade8_split.h), the code that
// the kernels compile themselves:
//   * each point of the grid is stored by exactly one lane, at its own address;
//   * each field load lies in its padded array, without a wrap of the 32-bit offset;
//   * each load and store of a memory variable lies in its array (they are made
//     where the kernels' predicates say so), along y and z inside its row;
//   * Slab::at numbers an x slab's points without gaps;
//   * a pair's points and the first stage's points around them lie outside the band
//     and off the edges.
// usage: address_audit grids [ghost]   (ghost: the columns of the y and z memory
// variables clamped like the fields', to the ghost column nx: must be found)
// Prints the number of addresses checked; exit code 1 if one is out of bounds.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <set>
#include <string>
#include <vector>

#include "../../seismic_cpml_amd/csrc/cpml_ade8_split.h"
#include "../../seismic_cpml_amd/csrc/cpml_tb_geom.h"

using namespace cpml;

static std::mt19937 rng(7);
static int pick(int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); }
static bool ghost = false;
static long checked = 0, bad = 0;
static std::set<std::string> kinds;

static void expect(bool ok, const char *what, int a, int b, int c) {
  ++checked;
  if (ok) return;
  ++bad;
  if (kinds.insert(what).second) std::printf("%s (%d, %d, %d)\n", what, a, b, c);  // the first
}

static long round_up(long v, long m) { return (v + m - 1) / m * m; }
static Slab slab(int n) {
  Slab s;
  s.n = n;
  const int most = n / 2 < 24 ? n / 2 : 24;
  s.wl = pick(0, 2) ? pick(0, most) : 0;
  s.wr = pick(0, 2) ? pick(0, most) : 0;
  s.w = s.wl + s.wr;
  return s;
}
// Half of the extents are whole cache lines, where a row has no padding.
static int extent(int lo, int hi) {
  const int n = pick(lo, hi);
  return rng() & 1 ? (n + 63) / 64 * 64 : n;
}
// Element of a lane's column in a row without ghost points.
static long mem_column(unsigned byte_off, size_t es, int i, int nx) {
  return ghost ? clamp_to(i, -1, nx) : (long)(byte_off / es);
}

template <typename T, bool SX, bool SY>
static void item2(const TB2D<T> &P, int order, int nt, const Tb2dItem &it, std::vector<int> &owned) {
  const Step2D<T> &a = P.a;
  const int nx = a.nx, ny = a.ny, r = order / 2, G = nt * (order - 1);
  const long align = 256 / sizeof(T), xpad = align, base = xpad + r * a.ld;
  const long total = a.ld * (ny + 2 * r);
  const int s0 = it.jb - (2 * nt - 1) * r, s1 = it.je - 1 + (2 * nt - 1) * r;
  for (int lane = 0; lane < 64; ++lane) {
    const int i = it.ts * P.ow - G + lane;
    const Tb2dLane<T, SX, SY> L(i, s0 - r, nx, ny, a.ld, a.sx);
    for (int j = s0 - r; j <= s1 + r; ++j) {
      const int jj = SY ? clamp_to(j, -1, ny) : j;
      const long q = base + L.corner + (long)(L.at(j) / sizeof(T));
      expect((long)L.at(j) == (long)(jj - L.rl) * L.ldb + L.vo && q >= 0 && q < total, "field", i, j, P.ow);
      if (j > s1) continue;
      const bool row_in = !SY || (j >= 0 && j < ny), col_in = !SX || (i >= 0 && i < nx);
      if (SX && L.inx && row_in)
        expect(L.ox(j) >= 0 && L.ox(j) < (long)a.sx.w * ny, "x memory", i, j, P.ow);
      if (SY && col_in && a.sy.in(j)) {
        const long m = mem_column(L.mo, sizeof(T), i, nx);
        expect(m >= 0 && m < nx && a.mld * a.sy.s(j) + m < a.mld * a.sy.w, "y memory", i, j, P.ow);
      }
    }
    if (lane >= G && lane < G + P.ow && (!SX || i < nx))
      for (int j = it.jb; j < it.je; ++j) {
        const long q = L.corner + (long)(L.at(j) / sizeof(T));
        const bool in = i >= 0 && i < nx && j >= 0 && j < ny && q == i + j * a.ld;
        expect(in, "store", i, j, P.ow);
        if (in) ++owned[i + (size_t)nx * j];
        if (!SX) expect(!a.sx.in(i), "x slab in a class without it", i, j, P.ow);
        if (!SY) expect(!a.sy.in(j), "y slab in a class without it", i, j, P.ow);
      }
  }
}

template <typename T>
static void item2_any(const TB2D<T> &P, int order, int nt, const Tb2dItem &it, std::vector<int> &o) {
  if (it.cls == 0) item2<T, false, false>(P, order, nt, it, o);
  else if (it.cls == 1) item2<T, true, false>(P, order, nt, it, o);
  else if (it.cls == 2) item2<T, false, true>(P, order, nt, it, o);
  else item2<T, true, true>(P, order, nt, it, o);
}

static void once(const std::vector<int> &owned) {
  for (size_t q = 0; q < owned.size(); ++q) expect(owned[q] == 1, "owners", owned[q], (int)q, 0);
}

template <typename T>
static void grid2() {
  TB2D<T> P{};
  const int order = 2 << pick(0, 2), nt = pick(1, tb2d_max_nt(order, sizeof(T)));
  const int widest = 64 - 2 * nt * (order - 1);
  P.a.nx = extent(3, 330), P.a.ny = pick(3, 200);
  P.a.sx = slab(P.a.nx), P.a.sy = slab(P.a.ny);
  const long align = 256 / sizeof(T);
  P.a.ld = round_up(align + P.a.nx + order / 2, align);
  P.a.mld = round_up(P.a.nx, align);
  P.ow = pick(1, widest), P.jc = pick(1, 70), P.js = pick(0, 1) ? tb2d_slab_rows(P.jc) : pick(1, 30);
  tb2d_split(order, nt, P);
  const Tb2dItems n = tb2d_items(P);
  std::vector<int> one((size_t)P.a.nx * P.a.ny), list(one.size());
  for (int k = 0; k < n.clean + n.edge + n.cap; ++k)
    item2_any(P, order, nt, tb2d_item_at(P, n, k), one);
  tb2d_list(P, [&](const Tb2dItem &it) { item2_any(P, order, nt, it, list); });
  once(one);
  once(list);
}

template <typename T, int NT, int NW, bool SX, bool SY, bool SZ>
static void tiles3(const TB3D<T> &P, std::vector<int> &owned) {
  const Step3D<T> &p = P.a;
  const int nx = p.nx, ny = p.ny, nz = p.nz;
  const int n = P.ncls[(SX ? 1 : 0) | (SY ? 2 : 0) | (SZ ? 4 : 0)];
  const long base = p.xpad + p.R * p.ld + p.R * p.ps, total = p.ps * (nz + 2 * p.R);
  for (int t = 0; t < n; ++t) {
    const Tb3dTile f = tb3d_tile_at<SX, SY, SZ>(P, t, nx, ny, nz, p.kchunk);
    const int s0 = f.kb - (2 * NT - 1), s1 = f.ke - 1 + (2 * NT - 1);
    for (int w = 0; w < NW; ++w)
      for (int lane = 0; lane < 64; ++lane) {
        const int i = f.i0 - NT + lane, j = f.j0 - NT + w;
        const Tb3dLane<T, SX, SY, SZ> L(i, j, s0 - 1, p);
        const bool col_in = !SX || (i >= 0 && i < nx), row_in = !SY || (j >= 0 && j < ny);
        // planes s0 - 1 .. s1 + 1 of the fields, s0 - 1 .. s1 of the memory variables
        for (int k = s0 - 1; k <= s1 + 1; ++k) {
          const int kk = SZ ? clamp_to(k, -1, nz) : k;
          const long q = base + L.corner + (long)(L.at(k) / sizeof(T));
          expect((long)L.at(k) == (long)(kk - L.kl) * L.psb + L.vo && q >= 0 && q < total, "field", i, j, k);
          if (k > s1) continue;
          const bool kin = !SZ || (k >= 0 && k < nz);
          if (SX && L.inx && row_in && kin) {
            const long m = L.mxo / sizeof(T);
            expect(m < L.mxs && L.mxs * k + m < (long)p.sx.w * ny * nz, "x memory", i, j, k);
          }
          if (SY && L.iny && col_in && kin) {
            const long m = mem_column(L.myo, sizeof(T), i, nx) + (ghost ? p.mld * p.sy.s(j) : 0);
            expect(m % p.mld < nx && m < L.mys && L.mys * k + m < L.mys * nz, "y memory", i, j, k);
          }
          if (SZ && col_in && row_in && p.sz.in(k)) {
            const long m = mem_column(L.mzo, sizeof(T), i, nx) + (ghost ? p.mld * clamp_to(j, 0, ny - 1) : 0);
            expect(m % p.mld < nx && m < L.mzs && L.mzs * p.sz.s(k) + m < L.mzs * p.sz.w, "z memory", i, j, k);
          }
        }
        if (lane >= NT && lane < NT + P.ow && w >= NT && w < NT + P.ty && (!SX || i < nx) &&
            (!SY || j < ny))
          for (int k = f.kb; k < f.ke; ++k) {
            const long q = L.corner + (long)(L.at(k) / sizeof(T));
            const bool in = i >= 0 && i < nx && j >= 0 && j < ny && k >= 0 && k < nz &&
                            q == i + j * p.ld + k * p.ps;
            expect(in, "store", i, j, k);
            if (in) ++owned[i + (size_t)nx * (j + (size_t)ny * k)];
            if (!SX) expect(!p.sx.in(i), "x slab in a class without it", i, j, k);
            if (!SY) expect(!p.sy.in(j), "y slab in a class without it", i, j, k);
            if (!SZ) expect(!p.sz.in(k), "z slab in a class without it", i, j, k);
          }
      }
  }
}

template <typename T, int NT>
static void grid3() {
  constexpr int NW = sizeof(T) == 4 ? 16 : 8;
  TB3D<T> P{};
  Step3D<T> &p = P.a;
  p.nx = extent(3, 150), p.ny = pick(3, 60), p.nz = pick(3, 40), p.R = 2;
  p.sx = slab(p.nx), p.sy = slab(p.ny), p.sz = slab(p.nz);
  const long align = 256 / sizeof(T);
  p.xpad = align;
  p.ld = round_up(align + p.nx + p.R, align);
  p.ps = p.ld * (p.ny + 2 * p.R);
  p.mld = round_up(p.nx, align);
  p.kchunk = pick(1, 30);
  P.ow = pick(1, 64 - 2 * NT);
  tb3d_split(NT, NW, P);
  std::vector<int> owned((size_t)p.nx * p.ny * p.nz);
  tiles3<T, NT, NW, false, false, false>(P, owned);
  tiles3<T, NT, NW, true, false, false>(P, owned);
  tiles3<T, NT, NW, false, true, false>(P, owned);
  tiles3<T, NT, NW, true, true, false>(P, owned);
  tiles3<T, NT, NW, false, false, true>(P, owned);
  tiles3<T, NT, NW, true, false, true>(P, owned);
  tiles3<T, NT, NW, false, true, true>(P, owned);
  tiles3<T, NT, NW, true, true, true>(P, owned);
  once(owned);
}

// x-slab arrays: every point of the slab has its own element of [0, w * rows).
static void slab_layout() {
  const Slab s = slab(pick(2, 90));
  const int rows = pick(1, 50);
  std::vector<int> hit((size_t)s.w * rows);
  for (int i = 0; i < s.n; ++i)
    for (int j = 0; j < rows && s.in(i); ++j) {
      const long q = s.at(i, j, rows);
      expect(q >= 0 && q < (long)hit.size(), "slab layout", i, j, rows);
      if (q >= 0 && q < (long)hit.size()) ++hit[q];
    }
  once(hit);
}

// Points of the frame's tiles, each counted in `owned`.
static void frame(const AdeFrame &f, int nx, std::vector<int> &owned) {
  for (int h = 0; h < f.tiles(); ++h) {
    int t = h;
    const AdeBox b = f.part(t);
    const int ntx = (b.x1 - b.x0 + AdeFrame::TX - 1) / AdeFrame::TX;
    for (int y = 0; y < ATY; ++y)
      for (int x = 0; x < AdeFrame::TX; ++x) {
        const int i = b.x0 + (t % ntx) * AdeFrame::TX + x, j = b.y0 + (t / ntx) * ATY + y;
        if (i < b.x1 && j < b.y1) ++owned[i + (size_t)nx * j];
      }
  }
}

template <typename T>
static void ade() {
  const int npml = pick(0, 30), nx = extent(1100, 1500), ny = pick(1000, 1400);
  const long align = 256 / sizeof(T), ld = round_up(align + nx + 4, align);
  const long base = align + 4 * ld, total = ld * (ny + 8);
  const AdeBox box = ade_pair_box<T>(nx, ny, npml);
  std::vector<int> owned((size_t)nx * ny), first((size_t)nx * ny);
  frame(AdeFrame(nx, ny, box), nx, owned);
  if (box.x1 > 0) {
    const AdePairs pairs = ade_pairs<T>(box);
    for (int t = 0; t < pairs.count(); ++t) {
      int c0, jb, je;
      pairs.item(t, c0, jb, je);
      expect(jb - 8 >= 1 && je + 7 <= ny - 2, "pair rows", jb, je, npml);
      for (int lane = 0; lane < 64; ++lane) {
        const int i = c0 - PG + lane;
        const long o = ade_pair_offset<T>(i, nx) / sizeof(T);
        for (int j : {jb - 8, je + 7})
          expect(o < nx && base + j * ld + o >= 0 && base + j * ld + o < total, "pair load", i, j, npml);
        if (lane < PG || lane >= PG + PW || i >= box.x1) continue;
        expect(i - 8 >= 1 && i + 8 <= nx - 2, "pair columns", i, c0, npml);
        for (int j = jb; j < je; ++j) {
          ++owned[i + (size_t)nx * j];
          if (j > box.y0 && j < box.y1 - 1 && i > box.x0 && i < box.x1 - 1) continue;
          for (int di : {-4, 4})
            for (int dj : {-4, 4})
              expect(!ade_band(i + di + 1, j + dj + 1, nx, ny, npml), "pair in the band", i, j, npml);
        }
      }
    }
    // the first stage of the frame: all but the box less 4 points on each side
    const AdeBox in = shrink(box, 4);
    frame(AdeFrame(nx, ny, in), nx, first);
    for (int j = 0; j < ny; ++j)
      for (int i = 0; i < nx; ++i)
        expect(first[i + (size_t)nx * j] == (in.in(i, j) ? 0 : 1), "first stage", i, j, npml);
  }
  once(owned);
}

int main(int argc, char **argv) {
  const int grids = argc > 1 ? std::atoi(argv[1]) : 40;
  ghost = argc > 2 && std::strcmp(argv[2], "ghost") == 0;
  for (int g = 0; g < grids; ++g) {
    grid2<float>();
    grid2<double>();
    grid3<float, 1>();
    grid3<float, 2>();
    grid3<double, 1>();
    grid3<double, 2>();
    slab_layout();
    if (g % 20 == 0) ade<float>(), ade<double>();
  }
  std::printf("%ld addresses checked, %ld out of bounds\n", checked, bad);
  return bad ? 1 : 0;
}
