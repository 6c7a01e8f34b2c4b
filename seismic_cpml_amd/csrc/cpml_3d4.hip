// 3D 4th-order staggered C-PML step for gfx950: the elastic part of
// seismic_CPML_3D_viscoelastic_MPI.f90 (the program run with tau_epsilon =
// tau_sigma, where its attenuation memory variables stay zero):
//   stress    seismic_CPML_3D_viscoelastic_MPI.f90:977-1229
//   velocity  ...viscoelastic_MPI.f90:1244-1327, source 1329-1353,
//             Dirichlet 1355-1398 (planes 1 and N of every axis)
// on the whole grid of one device (no slab interfaces: the reference's MPI
// run reads zero ghost planes across each of its slab interfaces, which a
// single domain does not have).
//
// Difference operator, as written there:
//   (27 f(+1) - 27 f(0) - f(+2) + f(-1)) * ONE_OVER_DELTA / 24
// summed left to right, divided (not multiplied) by 24; the file is built
// with -ffp-contract=off, so float64 results equal the restatement bit for
// bit.  Lame coefficients per point with Mu_nu = 1 (3D-visco:981-985):
//   lambda_u = (lambda + (2/3) mu) - (2/3) mu,  lambda_u + 2 mu,  mu,
// and the stress increment is (sum of coefficient * derivative) * DELTAT.
//
// Mapping: a 64 x TY block (TY = 4, 8 or 16 rows, the handle's tile) covers
// 64 columns (tile3 says which); each (i, j) column marches through a chunk of z
// planes.  The column's own z neighbours are carried in registers from plane
// to plane (one new plane per field and step); the x and y neighbours are
// read from global memory and come from the same or adjacent rows of the
// block, so they hit in L1/L2.  Profile values of the column are loaded once.
//
// Bound by HBM, at a rate that the wavefronts in flight set: 6 per SIMD in float
// (79 registers), 3 in double (141).  A plane's loads, memory variables included,
// are issued together through buffers whose offsets the scalar unit adds.
// Loading the next plane ahead into a second register set leaves 4 and 2
// wavefronts and is slower: float 210 x 800 x 220 1606 us per step and 1531 without,
// 512^3 4353 and 4004, 768^3 13572 and 12794; double 512^3 9134 and 8773 (128^3 189 and
// 196).
#include <hip/hip_runtime.h>

#include "cpml_constdiv.h"
#include "cpml_device.h"
#include "cpml_internal.h"
#include "cpml_record.h"

namespace cpml {
namespace {

// Doubles number the columns through the plane (tile3).
template <typename T>
constexpr bool kFlat4 = sizeof(T) == 8;

// (27 fp - 27 f0 - fpp + fm) * od, in the reference's order; its callers divide
// by 24
template <typename T>
__device__ __forceinline__ T d4(T fp, T f0, T fpp, T fm, T od) {
  return (((T(27) * fp - T(27) * f0) - fpp) + fm) * od;
}

// The chunk's planes kb - 2 .. ke + 1 as buffers: per-lane 32-bit byte offset
// of the column, scalar offset of the plane and row, x shift in the
// instruction (the host keeps a chunk's planes and 8 more below 4 GiB).
template <typename T>
struct Chunk4 {
  unsigned v0, ldb, psb, bytes;
  long origin;
  __device__ Chunk4(const Step3D<T> &p, const Tile3 &c) {
    ldb = (unsigned)(p.ld * sizeof(T));
    psb = (unsigned)(p.ps * sizeof(T));
    bytes = (unsigned)((c.ke - c.kb + 4) * p.ps * sizeof(T));
    origin = (long)(c.kb - 2 + p.R) * p.ps;
    v0 = (unsigned)(((c.j - 2 + p.R) * p.ld + p.xpad + c.i - 2) * sizeof(T));
  }
  __device__ __amdgpu_buffer_rsrc_t rsrc(const T *interior_origin, long base) const {
    return make_rsrc(interior_origin - base + origin, bytes);
  }
  // f(i + dx, j + dy, k + dz) of buffer plane kk = k - kb + 2
  __device__ T ld(__amdgpu_buffer_rsrc_t r, int dx, int dy, int dz, int kk) const {
    return BufOp<T>::ld(r, v0 + (2 + dx) * (unsigned)sizeof(T),
                        (unsigned)(kk + dz) * psb + (unsigned)(2 + dy) * ldb);
  }
  __device__ void st(T x, __amdgpu_buffer_rsrc_t r, int kk) const {
    BufOp<T>::st(x, r, v0 + 2 * (unsigned)sizeof(T), (unsigned)kk * psb + 2 * ldb);
  }
};

// C-PML of one derivative of a point inside the axis' slab, with its memory
// variable m read with the plane: psi <- b*psi + a*d ; d <- d/K + psi
// where `in` (the update's loop range).
template <typename T>
__device__ __forceinline__ void pml4(bool in, T &d, T m, T *psi, T a, T b, T K) {
  if (!in) return;
  m = b * m + a * d;
  *psi = m;
  d = over_k(d, K) + m;
}

// Values the stress kernel reads at plane k.
template <typename T>
struct SPlane4 {
  T vx_zpp, vx_xp, vx_xpp, vx_xm, vx_yp, vx_ypp, vx_ym;
  T vy_zpp, vy_xm, vy_xp, vy_xmm, vy_ym, vy_yp, vy_ymm;
  T vz_zp, vz_xm, vz_xp, vz_xmm, vz_yp, vz_ypp, vz_ym;
  T mu, lam, xx, yy, zz, xy, xz, yz;
  T px[3], py[3], pz[3];  // memory variables, where the point lies in the axis' slab
};

template <typename T, int TY4>
__global__ __launch_bounds__(BX *TY4) void k_stress3d4(Step3D<T> p,
    Record<T> prev, int lead) {
  int h;
  if (lead_block(prev, lead, h)) return;
  const Tile3 c = tile3<TY4, kFlat4<T>>(p, h);
  if (!c.ok) return;
  const int i = c.i, j = c.j, nx = p.nx, ny = p.ny, nz = p.nz;
  const Chunk4<T> g(p, c);
  const auto rvx = g.rsrc(p.vx, p.base), rvy = g.rsrc(p.vy, p.base), rvz = g.rsrc(p.vz, p.base);
  const auto rla = g.rsrc(p.lam, p.base), rmu = g.rsrc(p.mu, p.base);
  const auto rxx = g.rsrc(p.sxx, p.base), ryy = g.rsrc(p.syy, p.base);
  const auto rzz = g.rsrc(p.szz, p.base), rxy = g.rsrc(p.sxy, p.base);
  const auto rxz = g.rsrc(p.sxz, p.base), ryz = g.rsrc(p.syz, p.base);
  const bool inx = p.sx.in(i), iny = p.sy.in(j);
  const long mxo = p.sx.at(i, j, ny), mxs = (long)p.sx.w * ny;
  const long myo = i + p.mld * p.sy.s(j), mys = p.mld * p.sy.w;
  const long mzo = i + p.mld * j, mzs = p.mld * ny;
  // loop ranges of 3D-visco:977-979, 1080-1082, 1141-1144, 1185-1186 (0-based)
  const bool r_n = i <= nx - 2 && j >= 1;
  const bool r_xy = i >= 1 && j <= ny - 2;
  const bool r_xz = i >= 1;
  const bool r_yz = j <= ny - 2;
  const T c23 = T(2) / T(3);  // 2.d0/DIM
  T xa = 0, xb = 0, xK = 1, xah = 0, xbh = 0, xKh = 1;
  T ya = 0, yb = 0, yK = 1, yah = 0, ybh = 0, yKh = 1;
  if (inx) {
    xa = p.px.a[i]; xb = p.px.b[i]; xK = p.px.K[i];
    xah = p.px.ah[i]; xbh = p.px.bh[i]; xKh = p.px.Kh[i];
  }
  if (iny) {
    ya = p.py.a[j]; yb = p.py.b[j]; yK = p.py.K[j];
    yah = p.py.ah[j]; ybh = p.py.bh[j]; yKh = p.py.Kh[j];
  }
  auto load = [&](SPlane4<T> &L, int k) {
    const auto Q = kernarg<Step3D<T>>();
    const int kk = k - c.kb + 2;
    L.vx_zpp = g.ld(rvx, 0, 0, 2, kk);
    L.vy_zpp = g.ld(rvy, 0, 0, 2, kk);
    L.vz_zp = g.ld(rvz, 0, 0, 1, kk);
    L.vx_xp = g.ld(rvx, 1, 0, 0, kk), L.vx_xpp = g.ld(rvx, 2, 0, 0, kk);
    L.vx_xm = g.ld(rvx, -1, 0, 0, kk);
    L.vx_yp = g.ld(rvx, 0, 1, 0, kk), L.vx_ypp = g.ld(rvx, 0, 2, 0, kk);
    L.vx_ym = g.ld(rvx, 0, -1, 0, kk);
    L.vy_xm = g.ld(rvy, -1, 0, 0, kk), L.vy_xp = g.ld(rvy, 1, 0, 0, kk);
    L.vy_xmm = g.ld(rvy, -2, 0, 0, kk);
    L.vy_ym = g.ld(rvy, 0, -1, 0, kk), L.vy_yp = g.ld(rvy, 0, 1, 0, kk);
    L.vy_ymm = g.ld(rvy, 0, -2, 0, kk);
    L.vz_xm = g.ld(rvz, -1, 0, 0, kk), L.vz_xp = g.ld(rvz, 1, 0, 0, kk);
    L.vz_xmm = g.ld(rvz, -2, 0, 0, kk);
    L.vz_yp = g.ld(rvz, 0, 1, 0, kk), L.vz_ypp = g.ld(rvz, 0, 2, 0, kk);
    L.vz_ym = g.ld(rvz, 0, -1, 0, kk);
    L.mu = g.ld(rmu, 0, 0, 0, kk), L.lam = g.ld(rla, 0, 0, 0, kk);
    L.xx = g.ld(rxx, 0, 0, 0, kk), L.yy = g.ld(ryy, 0, 0, 0, kk);
    L.zz = g.ld(rzz, 0, 0, 0, kk), L.xy = g.ld(rxy, 0, 0, 0, kk);
    L.xz = g.ld(rxz, 0, 0, 0, kk), L.yz = g.ld(ryz, 0, 0, 0, kk);
    if (inx) {
      const long m = mxo + k * mxs;
      L.px[0] = Q->mx[0][m], L.px[1] = Q->mx[1][m], L.px[2] = Q->mx[2][m];
    }
    if (iny) {
      const long m = myo + k * mys;
      L.py[0] = Q->my[0][m], L.py[1] = Q->my[1][m], L.py[2] = Q->my[2][m];
    }
    if (p.sz.in(k)) {
      const long m = mzo + p.sz.s(k) * mzs;
      L.pz[0] = Q->mz[0][m], L.pz[1] = Q->mz[1][m], L.pz[2] = Q->mz[2][m];
    }
  };
  // the column's own z neighbours, carried from plane to plane
  constexpr int k0 = 2;  // buffer plane of kb
  T vx_zm = g.ld(rvx, 0, 0, -1, k0), vx0 = g.ld(rvx, 0, 0, 0, k0), vx_zp = g.ld(rvx, 0, 0, 1, k0);
  T vy_zm = g.ld(rvy, 0, 0, -1, k0), vy0 = g.ld(rvy, 0, 0, 0, k0), vy_zp = g.ld(rvy, 0, 0, 1, k0);
  T vz_zmm = g.ld(rvz, 0, 0, -2, k0), vz_zm = g.ld(rvz, 0, 0, -1, k0);
  T vz0 = g.ld(rvz, 0, 0, 0, k0);
  for (int k = c.kb; k < c.ke; ++k) {
    const auto Q = kernarg<Step3D<T>>();
    const int kk = k - c.kb + 2;
    SPlane4<T> L;
    load(L, k);
    const T mu = L.mu, lam = L.lam;
    const bool inz = p.sz.in(k);
    const bool r_k1 = k >= 1, r_kn = k <= nz - 2;
    T dvx_dx = d4(L.vx_xp, vx0, L.vx_xpp, L.vx_xm, p.odx);
    T dvy_dy = d4(vy0, L.vy_ym, L.vy_yp, L.vy_ymm, p.ody);
    T dvz_dz = d4(vz0, vz_zm, L.vz_zp, vz_zmm, p.odz);
    T dvy_dx = d4(vy0, L.vy_xm, L.vy_xp, L.vy_xmm, p.odx);
    T dvx_dy = d4(L.vx_yp, vx0, L.vx_ypp, L.vx_ym, p.ody);
    T dvz_dx = d4(vz0, L.vz_xm, L.vz_xp, L.vz_xmm, p.odx);
    T dvx_dz = d4(vx_zp, vx0, L.vx_zpp, vx_zm, p.odz);
    T dvz_dy = d4(L.vz_yp, vz0, L.vz_ypp, L.vz_ym, p.ody);
    T dvy_dz = d4(vy_zp, vy0, L.vy_zpp, vy_zm, p.odz);
    const_divide(p.div24, dvx_dx, dvy_dy, dvz_dz);
    const_divide(p.div24, dvy_dx, dvx_dy, dvz_dx);
    const_divide(p.div24, dvx_dz, dvz_dy, dvy_dz);
    if (inx) {
      const long m = mxo + k * mxs;
      pml4(r_n && r_k1, dvx_dx, L.px[0], Q->mx[0] + m, xah, xbh, xKh);
      pml4(r_xy, dvy_dx, L.px[1], Q->mx[1] + m, xa, xb, xK);
      pml4(r_xz && r_kn, dvz_dx, L.px[2], Q->mx[2] + m, xa, xb, xK);
    }
    if (iny) {
      const long m = myo + k * mys;
      pml4(r_n && r_k1, dvy_dy, L.py[0], Q->my[0] + m, ya, yb, yK);
      pml4(r_xy, dvx_dy, L.py[1], Q->my[1] + m, yah, ybh, yKh);
      pml4(r_yz && r_kn, dvz_dy, L.py[2], Q->my[2] + m, yah, ybh, yKh);
    }
    if (inz) {
      const long m = mzo + p.sz.s(k) * mzs;
      const T zah = Q->pz.ah[k], zbh = Q->pz.bh[k], zKh = Q->pz.Kh[k];
      pml4(r_n && r_k1, dvz_dz, L.pz[0], Q->mz[0] + m, Q->pz.a[k], Q->pz.b[k], Q->pz.K[k]);
      pml4(r_xz && r_kn, dvx_dz, L.pz[1], Q->mz[1] + m, zah, zbh, zKh);
      pml4(r_yz && r_kn, dvy_dz, L.pz[2], Q->mz[2] + m, zah, zbh, zKh);
    }
    const T lu = (lam + c23 * mu) - c23 * mu;
    const T l2u = lu + T(2) * mu;
    if (r_n && r_k1) {
      g.st(L.xx + (l2u * dvx_dx + lu * dvy_dy + lu * dvz_dz) * p.dt, rxx, kk);
      g.st(L.yy + (lu * dvx_dx + l2u * dvy_dy + lu * dvz_dz) * p.dt, ryy, kk);
      g.st(L.zz + (lu * dvx_dx + lu * dvy_dy + l2u * dvz_dz) * p.dt, rzz, kk);
    }
    if (r_xy) g.st(L.xy + mu * (dvx_dy + dvy_dx) * p.dt, rxy, kk);
    if (r_xz && r_kn) g.st(L.xz + mu * (dvx_dz + dvz_dx) * p.dt, rxz, kk);
    if (r_yz && r_kn) g.st(L.yz + mu * (dvy_dz + dvz_dy) * p.dt, ryz, kk);
    vx_zm = vx0, vx0 = vx_zp, vx_zp = L.vx_zpp;
    vy_zm = vy0, vy0 = vy_zp, vy_zp = L.vy_zpp;
    vz_zmm = vz_zm, vz_zm = vz0, vz0 = L.vz_zp;
  }
}

// Values the velocity kernel reads at plane k.
template <typename T>
struct VPlane4 {
  T xx0, xx_xm, xx_xp, xx_xmm, xy0, xy_ym, xy_yp, xy_ymm, xy_xp, xy_xpp, xy_xm;
  T xz_zp, xz_xp, xz_xpp, xz_xm, yy0, yy_yp, yy_ypp, yy_ym, yz_zp, yz_ym, yz_yp, yz_ymm;
  T zz_zpp, cb, vx, vy, vz;
  T px[3], py[3], pz[3];
};

template <typename T, int TY4>
__global__ __launch_bounds__(BX *TY4) void k_velocity3d4(Step3D<T> p) {
  const Tile3 c = tile3<TY4, kFlat4<T>>(p, blockIdx.x);
  if (!c.ok) return;
  const int i = c.i, j = c.j, nx = p.nx, ny = p.ny, nz = p.nz;
  const Chunk4<T> g(p, c);
  const auto rvx = g.rsrc(p.vx, p.base), rvy = g.rsrc(p.vy, p.base), rvz = g.rsrc(p.vz, p.base);
  const auto rcb = g.rsrc(p.cbuoy, p.base);  // DELTAT_over_rho
  const auto rxx = g.rsrc(p.sxx, p.base), ryy = g.rsrc(p.syy, p.base);
  const auto rzz = g.rsrc(p.szz, p.base), rxy = g.rsrc(p.sxy, p.base);
  const auto rxz = g.rsrc(p.sxz, p.base), ryz = g.rsrc(p.syz, p.base);
  const bool inx = p.sx.in(i), iny = p.sy.in(j);
  const long mxo = p.sx.at(i, j, ny), mxs = (long)p.sx.w * ny;
  const long myo = i + p.mld * p.sy.s(j), mys = p.mld * p.sy.w;
  const long mzo = i + p.mld * j, mzs = p.mld * ny;
  // loop ranges of 3D-visco:1244-1246, 1266-1267, 1287-1289 (0-based)
  const bool r_vx = i >= 1 && j >= 1;
  const bool r_vy = i <= nx - 2 && j <= ny - 2;
  const bool r_vz = i <= nx - 2 && j >= 1;
  const bool edge_xy = i == 0 || i == nx - 1 || j == 0 || j == ny - 1;
  const bool src_col = i == p.isrc && j == p.jsrc;
  T xa = 0, xb = 0, xK = 1, xah = 0, xbh = 0, xKh = 1;
  T ya = 0, yb = 0, yK = 1, yah = 0, ybh = 0, yKh = 1;
  if (inx) {
    xa = p.px.a[i]; xb = p.px.b[i]; xK = p.px.K[i];
    xah = p.px.ah[i]; xbh = p.px.bh[i]; xKh = p.px.Kh[i];
  }
  if (iny) {
    ya = p.py.a[j]; yb = p.py.b[j]; yK = p.py.K[j];
    yah = p.py.ah[j]; ybh = p.py.bh[j]; yKh = p.py.Kh[j];
  }
  auto load = [&](VPlane4<T> &L, int k) {
    const auto Q = kernarg<Step3D<T>>();
    const int kk = k - c.kb + 2;
    L.zz_zpp = g.ld(rzz, 0, 0, 2, kk);
    L.xz_zp = g.ld(rxz, 0, 0, 1, kk), L.yz_zp = g.ld(ryz, 0, 0, 1, kk);
    L.xx0 = g.ld(rxx, 0, 0, 0, kk), L.xx_xm = g.ld(rxx, -1, 0, 0, kk);
    L.xx_xp = g.ld(rxx, 1, 0, 0, kk), L.xx_xmm = g.ld(rxx, -2, 0, 0, kk);
    L.xy0 = g.ld(rxy, 0, 0, 0, kk), L.xy_ym = g.ld(rxy, 0, -1, 0, kk);
    L.xy_yp = g.ld(rxy, 0, 1, 0, kk), L.xy_ymm = g.ld(rxy, 0, -2, 0, kk);
    L.xy_xp = g.ld(rxy, 1, 0, 0, kk), L.xy_xpp = g.ld(rxy, 2, 0, 0, kk);
    L.xy_xm = g.ld(rxy, -1, 0, 0, kk);
    L.xz_xp = g.ld(rxz, 1, 0, 0, kk), L.xz_xpp = g.ld(rxz, 2, 0, 0, kk);
    L.xz_xm = g.ld(rxz, -1, 0, 0, kk);
    L.yy0 = g.ld(ryy, 0, 0, 0, kk), L.yy_yp = g.ld(ryy, 0, 1, 0, kk);
    L.yy_ypp = g.ld(ryy, 0, 2, 0, kk), L.yy_ym = g.ld(ryy, 0, -1, 0, kk);
    L.yz_ym = g.ld(ryz, 0, -1, 0, kk), L.yz_yp = g.ld(ryz, 0, 1, 0, kk);
    L.yz_ymm = g.ld(ryz, 0, -2, 0, kk);
    L.cb = g.ld(rcb, 0, 0, 0, kk);
    L.vx = g.ld(rvx, 0, 0, 0, kk), L.vy = g.ld(rvy, 0, 0, 0, kk), L.vz = g.ld(rvz, 0, 0, 0, kk);
    if (inx) {
      const long m = mxo + k * mxs;
      L.px[0] = Q->mx[3][m], L.px[1] = Q->mx[4][m], L.px[2] = Q->mx[5][m];
    }
    if (iny) {
      const long m = myo + k * mys;
      L.py[0] = Q->my[3][m], L.py[1] = Q->my[4][m], L.py[2] = Q->my[5][m];
    }
    if (p.sz.in(k)) {
      const long m = mzo + p.sz.s(k) * mzs;
      L.pz[0] = Q->mz[3][m], L.pz[1] = Q->mz[4][m], L.pz[2] = Q->mz[5][m];
    }
  };
  constexpr int k0 = 2;  // buffer plane of kb
  T sxz_zmm = g.ld(rxz, 0, 0, -2, k0), sxz_zm = g.ld(rxz, 0, 0, -1, k0);
  T sxz0 = g.ld(rxz, 0, 0, 0, k0);
  T syz_zmm = g.ld(ryz, 0, 0, -2, k0), syz_zm = g.ld(ryz, 0, 0, -1, k0);
  T syz0 = g.ld(ryz, 0, 0, 0, k0);
  T szz_zm = g.ld(rzz, 0, 0, -1, k0), szz0 = g.ld(rzz, 0, 0, 0, k0);
  T szz_zp = g.ld(rzz, 0, 0, 1, k0);
  for (int k = c.kb; k < c.ke; ++k) {
    const auto Q = kernarg<Step3D<T>>();
    const int kk = k - c.kb + 2;
    VPlane4<T> L;
    load(L, k);
    const T cb = L.cb;
    T vxn = L.vx, vyn = L.vy, vzn = L.vz;
    const bool inz = p.sz.in(k);
    const bool r_k1 = k >= 1, r_kn = k <= nz - 2;
    T dsxx_dx = d4(L.xx0, L.xx_xm, L.xx_xp, L.xx_xmm, p.odx);
    T dsxy_dy = d4(L.xy0, L.xy_ym, L.xy_yp, L.xy_ymm, p.ody);
    T dsxz_dz = d4(sxz0, sxz_zm, L.xz_zp, sxz_zmm, p.odz);
    T dsxy_dx = d4(L.xy_xp, L.xy0, L.xy_xpp, L.xy_xm, p.odx);
    T dsyy_dy = d4(L.yy_yp, L.yy0, L.yy_ypp, L.yy_ym, p.ody);
    T dsyz_dz = d4(syz0, syz_zm, L.yz_zp, syz_zmm, p.odz);
    T dsxz_dx = d4(L.xz_xp, sxz0, L.xz_xpp, L.xz_xm, p.odx);
    T dsyz_dy = d4(syz0, L.yz_ym, L.yz_yp, L.yz_ymm, p.ody);
    T dszz_dz = d4(szz_zp, szz0, L.zz_zpp, szz_zm, p.odz);
    const_divide(p.div24, dsxx_dx, dsxy_dy, dsxz_dz);
    const_divide(p.div24, dsxy_dx, dsyy_dy, dsyz_dz);
    const_divide(p.div24, dsxz_dx, dsyz_dy, dszz_dz);
    if (inx) {
      const long m = mxo + k * mxs;
      pml4(r_vx && r_k1, dsxx_dx, L.px[0], Q->mx[3] + m, xa, xb, xK);
      pml4(r_vy && r_k1, dsxy_dx, L.px[1], Q->mx[4] + m, xah, xbh, xKh);
      pml4(r_vz && r_kn, dsxz_dx, L.px[2], Q->mx[5] + m, xah, xbh, xKh);
    }
    if (iny) {
      const long m = myo + k * mys;
      pml4(r_vx && r_k1, dsxy_dy, L.py[0], Q->my[3] + m, ya, yb, yK);
      pml4(r_vy && r_k1, dsyy_dy, L.py[1], Q->my[4] + m, yah, ybh, yKh);
      pml4(r_vz && r_kn, dsyz_dy, L.py[2], Q->my[5] + m, ya, yb, yK);
    }
    if (inz) {
      const long m = mzo + p.sz.s(k) * mzs;
      const T za = Q->pz.a[k], zb = Q->pz.b[k], zK = Q->pz.K[k];
      pml4(r_vx && r_k1, dsxz_dz, L.pz[0], Q->mz[3] + m, za, zb, zK);
      pml4(r_vy && r_k1, dsyz_dz, L.pz[1], Q->mz[4] + m, za, zb, zK);
      pml4(r_vz && r_kn, dszz_dz, L.pz[2], Q->mz[5] + m, Q->pz.ah[k], Q->pz.bh[k], Q->pz.Kh[k]);
    }
    if (r_vx && r_k1) vxn = cb * (dsxx_dx + dsxy_dy + dsxz_dz) + vxn;
    if (r_vy && r_k1) vyn = cb * (dsxy_dx + dsyy_dy + dsyz_dz) + vyn;
    if (r_vz && r_kn) vzn = cb * (dsxz_dx + dsyz_dy + dszz_dz) + vzn;
    // point force on the cut plane (3D-visco:1350-1352)
    if (src_col && k == p.ksrc) {
      const int it = *Q->step;
      const T rs = Q->rho[i + (long)j * p.ld + (long)k * p.ps];
      vxn = vxn + Q->fx[it - 1] * p.dt / rs;
      vyn = vyn + Q->fy[it - 1] * p.dt / rs;
    }
    // rigid faces: planes 1 and N of every axis (3D-visco:1355-1398)
    if (edge_xy || k == 0 || k == nz - 1) {
      vxn = T(0);
      vyn = T(0);
      vzn = T(0);
    }
    g.st(vxn, rvx, kk);
    g.st(vyn, rvy, kk);
    g.st(vzn, rvz, kk);
    sxz_zmm = sxz_zm, sxz_zm = sxz0, sxz0 = L.xz_zp;
    syz_zmm = syz_zm, syz_zm = syz0, syz0 = L.yz_zp;
    szz_zm = szz0, szz0 = szz_zp, szz_zp = L.zz_zpp;
  }
}

template <typename T>
unsigned ntiles4(const Step3D<T> &p, int ty) {
  return (unsigned)plane_tiles3<kFlat4<T>>(p.nx, p.ny, ty) *
         ((p.nz + p.kchunk - 1) / p.kchunk);
}

}  // namespace

// p.tile_y selects the rows per block (4, 8 or 16; double: at most 8, since the
// 128 registers that blocks of 16 wavefronts leave would spill)
template <typename T>
hipError_t launch_stress3d4(const Step3D<T> &p, const Record<T> *prev, hipStream_t s) {
  const int lead = prev ? kLead : 0;
  const Record<T> rec = prev ? *prev : Record<T>{};
  if (p.tile_y >= 8) {
    if (p.tile_y == 16 && sizeof(T) == 4)
      hipLaunchKernelGGL((k_stress3d4<T, 16>), dim3(lead + ntiles4(p, 16)), dim3(BX, 16), 0, s,
                         p, rec, lead);
    else
      hipLaunchKernelGGL((k_stress3d4<T, 8>), dim3(lead + ntiles4(p, 8)), dim3(BX, 8), 0, s, p, rec,
                       lead);
  } else
    hipLaunchKernelGGL((k_stress3d4<T, 4>), dim3(lead + ntiles4(p, 4)), dim3(BX, 4), 0, s, p, rec,
                       lead);
  return hipGetLastError();
}

template <typename T>
hipError_t launch_velocity3d4(const Step3D<T> &p, hipStream_t s) {
  if (p.tile_y >= 8) {
    if (p.tile_y == 16 && sizeof(T) == 4)
      hipLaunchKernelGGL((k_velocity3d4<T, 16>), dim3(ntiles4(p, 16)), dim3(BX, 16), 0, s, p);
    else
      hipLaunchKernelGGL((k_velocity3d4<T, 8>), dim3(ntiles4(p, 8)), dim3(BX, 8), 0, s, p);
  } else
    hipLaunchKernelGGL((k_velocity3d4<T, 4>), dim3(ntiles4(p, 4)), dim3(BX, 4), 0, s, p);
  return hipGetLastError();
}

template hipError_t launch_stress3d4<float>(const Step3D<float> &, const Record<float> *,
                                             hipStream_t);
template hipError_t launch_stress3d4<double>(const Step3D<double> &, const Record<double> *,
                                              hipStream_t);
template hipError_t launch_velocity3d4<float>(const Step3D<float> &, hipStream_t);
template hipError_t launch_velocity3d4<double>(const Step3D<double> &, hipStream_t);

}  // namespace cpml
