// ADE-PML RK4 step of seismic_ADEPML_2D_elastic_RK4_eighth_order.f90 (ADE8)
// for gfx950: the 8th-order (Holberg) staggered operator, four Runge-Kutta
// stages per time step and the auxiliary-differential-equation PML whose
// coefficients depend on the stage (ADE8:692-906).  Per stage one pass
// (k_ade_stage): velocity rates from the stage state's sigma, ADE memories in
// the PML band, force at t = (it-1 + rk41) * DELTAT, rate borders zeroed;
// stress rates from its v; then at once X += rk42 * rate * DELTAT, velocity
// borders 0, and the next stage's state X0 + rk41 * rate * DELTAT.  The
// rates stay in registers: 4 launches per step instead of the program's 13
// array sweeps.
//
// X ping-pongs between two state buffers: the step reads X0 (the program's
// d3, ADE8:697-703) from the buffer the step starts in, which it never
// writes, and accumulates into the other one.  Stage 1's state is
// X0 + rk41(1) * X * DELTAT with rk41(1) = 0, i.e. X0 itself bit for bit
// (x + 0 * x * dt == x for every finite x, signed zeros included), so stage
// 1 reads it from X0 and no copy of the state is made.
// Arithmetic statement by statement as there (8th-order difference divided
// by DELTA; -ffp-contract=off), so float64 results equal the reference.
// The ghost cells of every array stay zero, as the program's 4-cell borders do.
//
// Bound by HBM when every stage is a pass (one point per thread, k_ade_stage: 92
// words per point and step).  So away from the PML band and the rigid edges one
// pass does two stages (k_ade_pair: 41 words): a wavefront marches up the rows of
// a 64-column strip, keeps 9 rows of the stage's state and 8 of the next stage's
// in registers, and owns the 48 columns that two rings of 4 leave, whole 64-byte
// sectors.  Bound by the vector pipes (83% busy) and HBM (4.3 and 5.7 TB/s) about
// equally: 4096^2 float 1847 -> 907 us per step.  The frame around that box takes
// the stages one by one: with a pair runs the first of them, on 4 more points
// per side (the second one's stencil), and a small launch the second.
#include <hip/hip_runtime.h>

#include "cpml_ade8_split.h"
#include "cpml_constdiv.h"
#include "cpml_device.h"
#include "cpml_internal.h"

namespace cpml {
namespace {

// Tile h of nt in XCD-aware order: the hardware hands workgroup h to XCD h % 8;
// each XCD gets one contiguous band of tiles (x fastest), so the halo columns and
// rows that neighbouring tiles share are read through the same L2.
__device__ __forceinline__ int xcd_tile(int h, int nt) {
  const int xcd = h & 7, loc = h >> 3, q = nt >> 3, r = nt & 7;
  return xcd * q + min(xcd, r) + loc;
}
// Point of this thread in tile t of a box: false outside.
__device__ __forceinline__ bool tile_point(AdeBox b, int t, int &i, int &j) {
  const int ntx = (b.x1 - b.x0 + AdeFrame::TX - 1) / AdeFrame::TX;
  i = b.x0 + (t % ntx) * AdeFrame::TX + threadIdx.x;
  j = b.y0 + (t / ntx) * ATY + threadIdx.y;
  return i < b.x1 && j < b.y1;
}
__device__ __forceinline__ bool frame_point(const AdeFrame &f, int h, int &i, int &j) {
  int t = xcd_tile(h, f.tiles());
  const AdeBox b = f.part(t);
  return tile_point(b, t, i, j);
}

// c1 d1 + c2 d2 + c3 d3 + c4 d4, ADE8:263-266
template <typename T>
__device__ __forceinline__ T sum8(T d1, T d2, T d3, T d4) {
  return ((T(kHolberg1) * d1 + T(kHolberg2) * d2) + T(kHolberg3) * d3) + T(kHolberg4) * d4;
}
// the same over delta, ADE8:720-723
template <typename T>
__device__ __forceinline__ T h8(T d1, T d2, T d3, T d4, T del) {
  return sum8(d1, d2, d3, d4) / del;
}

template <typename T>
__device__ __forceinline__ T rk41(int inc) {
  return inc == 0 ? T(0) : inc == 3 ? T(1) : T(0.5);
}
template <typename T>
__device__ __forceinline__ T rk42(int inc) {
  return (inc == 0 || inc == 3) ? T(1) / T(6) : T(2) / T(6);
}

// One Runge-Kutta stage in one pass (ADE8:715-874): the rates of the stage
// state S (X0 in stage 1, else d[in]) at this point -- velocity rates from
// S's stresses with the ADE memories in the PML band and the stage-time
// force, rate borders zeroed (ADE8:718-810); stress rates from S's
// velocities, whose border values the program has zeroed by then
// (ADE8:803-861) -- and at once the accumulation X += rk42 * rate * DELTAT
// into the step's output buffer (stage 1 starts from X0) with the velocity
// borders zeroed, and the next stage's state d[out] =
// X0 + rk41(inc+1) * rate * DELTAT (ADE8:863-874; X0's velocity borders
// count as zero, as the program's d3 after ADE8:803-810).  The rates never
// go to memory, and S is read from one buffer while the next state goes to
// another, so neighbours always see the stage's own state.
//
// `own`: the point's X is accumulated (false: only the next stage's state is
// wanted).
template <typename T>
__device__ __forceinline__ void ade_point(const Ade8<T> &a, int inc, int in, int out, int i, int j,
                                          bool own) {
  const Step2D<T> &p = a.s;
  const long ld = p.ld, c = i + j * ld;
  const int nx = p.nx, ny = p.ny, I = i + 1, J = j + 1;
  const bool bd = ade_band(I, J, nx, ny, a.npml);
  const bool edge = i == 0 || i == nx - 1 || j == 0 || j == ny - 1;
  const T *const X0[5] = {p.vx, p.vy, p.sxx, p.syy, p.sxy};
  const T *const *st = inc == 0 ? X0 : a.d[in];
  const T *sxx = st[2], *syy = st[3], *sxy = st[4];
  const T *vxs = st[0], *vys = st[1];
  // everything that only this point reads, ahead of all stores
  T m[8], xo[5], x0[5];
  if (bd)
    for (int q = 0; q < 8; ++q) m[q] = a.mem[q][c];
  const bool next = inc < 3;
  for (int f = 0; f < 5; ++f) {
    // X0 is read only where used: stage 1 (accumulation base and next
    // state) and stages 2-3 (next state)
    xo[f] = inc == 0 ? X0[f][c] : a.xn[f][c];
    x0[f] = (f < 2 && edge) ? T(0) : inc == 0 ? xo[f] : next ? X0[f][c] : T(0);
  }
  T rate[5] = {T(0), T(0), T(0), T(0), T(0)};
  // vx rates: Fortran i = 2..NX, j = 2..NY (ADE8:718-744)
  if (i >= 1 && j >= 1) {
    T vx_ = h8(sxx[c] - sxx[c - 1], sxx[c + 1] - sxx[c - 2], sxx[c + 2] - sxx[c - 3],
               sxx[c + 3] - sxx[c - 4], a.dx);
    T vy_ = h8(sxy[c] - sxy[c - ld], sxy[c + ld] - sxy[c - 2 * ld], sxy[c + 2 * ld] - sxy[c - 3 * ld],
               sxy[c + 3 * ld] - sxy[c - 4 * ld], a.dy);
    if (bd) {
      a.mem[4][c] = m[4] = a.bx[inc * nx + i] * m[4] + a.ax[inc * nx + i] * vx_;
      a.mem[7][c] = m[7] = a.by[inc * ny + j] * m[7] + a.ay[inc * ny + j] * vy_;
      vx_ = vx_ / p.px.K[i] + m[4];
      vy_ = vy_ / p.py.K[j] + m[7];
    }
    rate[0] = (vx_ + vy_) / p.rho[c];
  }
  // vy rates: Fortran i = 1..NX-1, j = 1..NY-1 (ADE8:746-768)
  if (i <= nx - 2 && j <= ny - 2) {
    const T rh = T(0.25) * (p.rho[c] + p.rho[c + 1] + p.rho[c + 1 + ld] + p.rho[c + ld]);
    T sx_ = h8(sxy[c + 1] - sxy[c], sxy[c + 2] - sxy[c - 1], sxy[c + 3] - sxy[c - 2],
               sxy[c + 4] - sxy[c - 3], a.dx);
    T sy_ = h8(syy[c + ld] - syy[c], syy[c + 2 * ld] - syy[c - ld], syy[c + 3 * ld] - syy[c - 2 * ld],
               syy[c + 4 * ld] - syy[c - 3 * ld], a.dy);
    if (bd) {
      a.mem[6][c] = m[6] = a.bxh[inc * nx + i] * m[6] + a.axh[inc * nx + i] * sx_;
      a.mem[5][c] = m[5] = a.byh[inc * ny + j] * m[5] + a.ayh[inc * ny + j] * sy_;
      sx_ = sx_ / p.px.Kh[i] + m[6];
      sy_ = sy_ / p.py.Kh[j] + m[5];
    }
    rate[1] = (sx_ + sy_) / rh;
  }
  // force at the stage time (ADE8:786-802)
  if (i == p.isrc && j == p.jsrc) {
    const int it = *p.step;
    const T rh = T(0.25) * (p.rho[c] + p.rho[c + 1] + p.rho[c + 1 + ld] + p.rho[c + ld]);
    rate[0] = rate[0] + a.f4x[(long)(it - 1) * 4 + inc] / p.rho[c];
    rate[1] = rate[1] + a.f4y[(long)(it - 1) * 4 + inc] / rh;
  }
  if (edge) rate[0] = rate[1] = T(0);  // ADE8:803-810
  // S's velocities with the border points zero (ADE8:803-810 ran before)
  auto V = [&](const T *f, int di, int dj) -> T {
    const int ii = i + di, jj = j + dj;
    if (ii == 0 || ii == nx - 1 || jj == 0 || jj == ny - 1) return T(0);
    return f[c + di + (long)dj * ld];
  };
  // sigma_xx, sigma_yy rates: Fortran i = 1..NX-1, j = 2..NY (ADE8:811-834)
  if (i <= nx - 2 && j >= 1) {
    const T lh = T(0.5) * (p.lam[c + 1] + p.lam[c]);
    const T mh = T(0.5) * (p.mu[c + 1] + p.mu[c]);
    const T l2m = lh + T(2) * mh;
    T dvx_dx = h8(V(vxs, 1, 0) - V(vxs, 0, 0), V(vxs, 2, 0) - V(vxs, -1, 0),
                  V(vxs, 3, 0) - V(vxs, -2, 0), V(vxs, 4, 0) - V(vxs, -3, 0), a.dx);
    T dvy_dy = h8(V(vys, 0, 0) - V(vys, 0, -1), V(vys, 0, 1) - V(vys, 0, -2),
                  V(vys, 0, 2) - V(vys, 0, -3), V(vys, 0, 3) - V(vys, 0, -4), a.dy);
    if (bd) {
      a.mem[0][c] = m[0] = a.bxh[inc * nx + i] * m[0] + a.axh[inc * nx + i] * dvx_dx;
      a.mem[3][c] = m[3] = a.by[inc * ny + j] * m[3] + a.ay[inc * ny + j] * dvy_dy;
      dvx_dx = dvx_dx / p.px.Kh[i] + m[0];
      dvy_dy = dvy_dy / p.py.K[j] + m[3];
    }
    rate[2] = l2m * dvx_dx + lh * dvy_dy;
    rate[3] = lh * dvx_dx + l2m * dvy_dy;
  }
  // sigma_xy rate: Fortran i = 2..NX, j = 1..NY-1 (ADE8:836-861)
  if (i >= 1 && j <= ny - 2) {
    const T mhy = T(0.5) * (p.mu[c + ld] + p.mu[c]);
    T dvx_dy = h8(V(vxs, 0, 1) - V(vxs, 0, 0), V(vxs, 0, 2) - V(vxs, 0, -1),
                  V(vxs, 0, 3) - V(vxs, 0, -2), V(vxs, 0, 4) - V(vxs, 0, -3), a.dy);
    T dvy_dx = h8(V(vys, 0, 0) - V(vys, -1, 0), V(vys, 1, 0) - V(vys, -2, 0),
                  V(vys, 2, 0) - V(vys, -3, 0), V(vys, 3, 0) - V(vys, -4, 0), a.dx);
    if (bd) {
      a.mem[2][c] = m[2] = a.bx[inc * nx + i] * m[2] + a.ax[inc * nx + i] * dvy_dx;
      a.mem[1][c] = m[1] = a.byh[inc * ny + j] * m[1] + a.ayh[inc * ny + j] * dvx_dy;
      dvy_dx = dvy_dx / p.px.K[i] + m[2];
      dvx_dy = dvx_dy / p.py.Kh[j] + m[1];
    }
    rate[4] = mhy * (dvy_dx + dvx_dy);
  }
  // accumulation and the next stage's state (ADE8:863-874)
  const T r = rk42<T>(inc);
  const T rn = next ? rk41<T>(inc + 1) : T(0);
  for (int f = 0; f < 5; ++f) {
    const T d2 = rate[f];
    if (own) a.xn[f][c] = xo[f] + r * d2 * p.dt;
    if (next) a.d[out][f][c] = x0[f] + rn * d2 * p.dt;
  }
  if (edge && own) {
    a.xn[0][c] = T(0);
    a.xn[1][c] = T(0);
  }
}

// Stage inc on the grid but for `skip`; X is accumulated outside `box`.
template <typename T>
__device__ __forceinline__ void ade_frame(const Ade8<T> &a, int inc, AdeBox box, AdeBox skip, int h) {
  int i, j;
  if (frame_point(AdeFrame(a.s.nx, a.s.ny, skip), h, i, j))
    ade_point(a, inc, inc & 1, (inc & 1) ^ 1, i, j, !box.in(i, j));
}
template <typename T, bool WHOLE>
__global__ __launch_bounds__(BX *ATY) void k_ade_stage(Ade8<T> a, int inc, AdeBox box) {
  if (!WHOLE) {
    ade_frame(a, inc, box, box, blockIdx.x);
    return;
  }
  int i, j;
  if (tile_point(AdeBox{0, a.s.nx, 0, a.s.ny}, xcd_tile(blockIdx.x, gridDim.x), i, j))
    ade_point(a, inc, inc & 1, (inc & 1) ^ 1, i, j, true);
}

// Media of one row of a strip: values at the points and at their neighbours.
template <typename T>
struct AdeMedia {
  T l2m, lh, mhy, rho, rh;
  __device__ AdeMedia(T lam, T mu, T mu_up, T rho_, T rho_up) {
    lh = T(0.5) * (lane_next(lam) + lam);
    const T mh = T(0.5) * (lane_next(mu) + mu);
    l2m = lh + T(2) * mh;
    mhy = T(0.5) * (mu_up + mu);
    rho = rho_;
    rh = T(0.25) * (rho_ + lane_next(rho_) + lane_next(rho_up) + rho_up);
  }
};

// 8th-order sums along x of f at this lane: between columns i - 1 and i (back) and
// between i and i + 1 (forward).
template <typename T>
__device__ __forceinline__ T x_back(T f) {
  const T m1 = lane_prev(f), m2 = lane_prev(m1), m3 = lane_prev(m2), m4 = lane_prev(m3);
  const T n1 = lane_next(f), n2 = lane_next(n1), n3 = lane_next(n2);
  return sum8(f - m1, n1 - m2, n2 - m3, n3 - m4);
}
template <typename T>
__device__ __forceinline__ T x_fwd(T f) {
  const T m1 = lane_prev(f), m2 = lane_prev(m1), m3 = lane_prev(m2);
  const T n1 = lane_next(f), n2 = lane_next(n1), n3 = lane_next(n2), n4 = lane_next(n3);
  return sum8(n1 - f, n2 - m1, n3 - m2, n4 - m3);
}
// ... and along y of 8 rows w[0..7]: between w[3] and w[4].
template <typename T>
__device__ __forceinline__ T y_mid(const T *w) {
  return sum8(w[4] - w[3], w[5] - w[2], w[6] - w[1], w[7] - w[0]);
}

// Rates of one row away from band and edges (ADE8:718-861 as in ade_point): sxx
// of the row, 8 rows each of sxy and vy (from 4 below the row) and of syy and vx
// (from 3 below).
template <typename T>
__device__ __forceinline__ void ade_rates(const Step2D<T> &p, const AdeMedia<T> &m, T sxx,
                                          const T *sxy, const T *syy, const T *vx, const T *vy,
                                          T fx, T fy, bool src, T *rate) {
  T xx_x = x_back(sxx), xy_y = y_mid(sxy), xy_x = x_fwd(sxy[4]), yy_y = y_mid(syy);
  const_divide(xx_x, p.div_x, xy_y, p.div_y, xy_x, p.div_x, yy_y, p.div_y);
  rate[0] = (xx_x + xy_y) / m.rho;
  rate[1] = (xy_x + yy_y) / m.rh;
  if (src) {
    rate[0] = rate[0] + fx / m.rho;
    rate[1] = rate[1] + fy / m.rh;
  }
  T vx_x = x_fwd(vx[3]), vy_y = y_mid(vy), vx_y = y_mid(vx), vy_x = x_back(vy[4]);
  const_divide(vx_x, p.div_x, vy_y, p.div_y, vx_y, p.div_y, vy_x, p.div_x);
  rate[2] = m.l2m * vx_x + m.lh * vy_y;
  rate[3] = m.lh * vx_x + m.l2m * vy_y;
  rate[4] = m.mhy * (vy_x + vx_y);
}

// Stages 1 and 2 (FIRST) or 3 and 4 of the columns [c0, c0 + PW) and rows [jb, je)
// of the box.  Iteration p takes row p of the first stage and row p - 4 of the
// second.
template <typename T, bool FIRST>
__device__ __forceinline__ void ade_pair(const Ade8<T> &a, AdeBox box, int c0, int jb, int je,
                                         T (*delay)[4][BX]) {
  const Step2D<T> &p = a.s;
  const long ld = p.ld;
  const int lane = threadIdx.x, i = c0 - PG + lane;
  const bool own = lane >= PG && lane < PG + PW && i < box.x1;
  const unsigned o = ade_pair_offset<T>(i, p.nx);
  constexpr int inc = FIRST ? 0 : 2;
  const T r1 = rk42<T>(inc), r2 = rk42<T>(inc + 1);
  const T n1 = rk41<T>(inc + 1), n2 = FIRST ? rk41<T>(inc + 2) : T(0);
  const T *const *S = FIRST ? nullptr : a.d[0];
  const T *svx = FIRST ? p.vx : S[0], *svy = FIRST ? p.vy : S[1];
  const T *sxx = FIRST ? p.sxx : S[2], *syy = FIRST ? p.syy : S[3], *sxy = FIRST ? p.sxy : S[4];
  const T *const X0[5] = {p.vx, p.vy, p.sxx, p.syy, p.sxy};
  auto at = [&](const T *f, int row) { return ld_at(f + row * ld, o); };
  // the source's column and step
  const bool src_col = i == p.isrc;
  T f1x = 0, f1y = 0, f2x = 0, f2y = 0;
  if (p.jsrc >= jb - 4 && p.jsrc < je + 4) {
    const long q = (long)(*p.step - 1) * 4 + inc;
    f1x = a.f4x[q], f1y = a.f4y[q], f2x = a.f4x[q + 1], f2y = a.f4y[q + 1];
  }
  // first stage's windows: vx, syy rows p - 4 .. p + 4, vy, sxy rows p - 4 .. p + 3
  T VX[9], YY[9], VY[8], XY[8];
  // second stage's: vx, syy rows p - 7 .. p, vy, sxy rows p - 8 .. p - 1
  T VX2[8] = {}, YY2[8] = {}, VY2[8] = {}, XY2[8] = {};
  const int p0 = jb - 4, p1 = je + 4;
#pragma unroll
  for (int k = 1; k < 9; ++k) VX[k] = at(svx, p0 - 5 + k), YY[k] = at(syy, p0 - 5 + k);
#pragma unroll
  for (int k = 1; k < 8; ++k) VY[k] = at(svy, p0 - 5 + k), XY[k] = at(sxy, p0 - 5 + k);
  T mu1 = at(p.mu, p0), rho1 = at(p.rho, p0), mu2 = T(1), rho2 = T(1);
  struct Ahead {
    T vx, vy, xx, yy, xy, lam1, mu1, rho1, lam2, mu2, rho2, x0[5], xo[5];
  } A;
  // last rows again past the end: never beyond the rows the box's ring reaches
  auto load = [&](Ahead &L, int row) {
    const int q = min(row, p1 - 1);
    L.vx = at(svx, q + 4), L.yy = at(syy, q + 4), L.vy = at(svy, q + 3), L.xy = at(sxy, q + 3);
    L.xx = at(sxx, q);
    L.lam1 = at(p.lam, q), L.mu1 = at(p.mu, q + 1), L.rho1 = at(p.rho, q + 1);
    L.lam2 = at(p.lam, q - 4), L.mu2 = at(p.mu, q - 3), L.rho2 = at(p.rho, q - 3);
    if (!FIRST)
#pragma unroll
      for (int f = 0; f < 5; ++f) L.x0[f] = at(X0[f], q), L.xo[f] = at(a.xn[f], q);
  };
  auto row = [&](int j, const Ahead &L, Ahead &N) {
    load(N, j + 1);
#pragma unroll
    for (int k = 0; k < 8; ++k) VX[k] = VX[k + 1], YY[k] = YY[k + 1];
#pragma unroll
    for (int k = 0; k < 7; ++k) VY[k] = VY[k + 1], XY[k] = XY[k + 1];
    VX[8] = L.vx, YY[8] = L.yy, VY[7] = L.vy, XY[7] = L.xy;
    T k1[5], s1[5], xq[5], xx0q = T(0);
    const AdeMedia<T> m1(L.lam1, mu1, L.mu1, rho1, L.rho1);
    mu1 = L.mu1, rho1 = L.rho1;
    ade_rates(p, m1, L.xx, XY, YY + 1, VX + 1, VY, f1x, f1y, src_col && j == p.jsrc, k1);
    const T x0[5] = {FIRST ? VX[4] : L.x0[0], FIRST ? VY[4] : L.x0[1], FIRST ? L.xx : L.x0[2],
                     FIRST ? YY[4] : L.x0[3], FIRST ? XY[4] : L.x0[4]};
    const int slot = j & 3;
#pragma unroll
    for (int f = 0; f < 5; ++f) {
      s1[f] = x0[f] + n1 * k1[f] * p.dt;
      xq[f] = delay[f][slot][lane];
      delay[f][slot][lane] = (FIRST ? x0[f] : L.xo[f]) + r1 * k1[f] * p.dt;
    }
    const T xx1q = delay[5][slot][lane];
    delay[5][slot][lane] = s1[2];
    if (FIRST) {
      xx0q = delay[6][slot][lane];
      delay[6][slot][lane] = L.xx;
    }
#pragma unroll
    for (int k = 0; k < 7; ++k) VX2[k] = VX2[k + 1], YY2[k] = YY2[k + 1];
    VX2[7] = s1[0], YY2[7] = s1[3];
    const AdeMedia<T> m2(L.lam2, mu2, L.mu2, rho2, L.rho2);
    mu2 = L.mu2, rho2 = L.rho2;
    const int q = j - 4;
    if (q >= jb) {
      T k2[5];
      ade_rates(p, m2, xx1q, XY2, YY2, VX2, VY2, f2x, f2y, src_col && q == p.jsrc, k2);
      const T x0q[5] = {VX[0], VY[0], xx0q, YY[0], XY[0]};
      if (own)
#pragma unroll
        for (int f = 0; f < 5; ++f) {
          st_at(a.xn[f] + q * ld, o, xq[f] + r2 * k2[f] * p.dt);
          if (FIRST) st_at(a.d[0][f] + q * ld, o, x0q[f] + n2 * k2[f] * p.dt);
        }
    }
#pragma unroll
    for (int k = 0; k < 7; ++k) VY2[k] = VY2[k + 1], XY2[k] = XY2[k + 1];
    VY2[7] = s1[1], XY2[7] = s1[4];
  };
  Ahead B;
  load(A, p0);
  for (int j = p0; j < p1; j += 4) {  // 4 rows: the windows' moves merge
    row(j, A, B);
    if (j + 1 < p1) row(j + 1, B, A);
    if (j + 2 < p1) row(j + 2, A, B);
    if (j + 3 < p1) row(j + 3, B, A);
  }
}

// The pair's items (one wavefront each), then the frame's first stage.
template <typename T, bool FIRST>
__global__ __launch_bounds__(BX *ATY) void k_ade_pair(Ade8<T> a, AdePairs pairs, int nblocks) {
  __shared__ T delay[ATY][FIRST ? 7 : 6][4][BX];
  const int h = blockIdx.x;
  if (h >= nblocks) {
    ade_frame(a, FIRST ? 0 : 2, pairs.box, shrink(pairs.box, 4), h - nblocks);
    return;
  }
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.y);
  // each XCD gets one contiguous band of items (strips fastest)
  const int t = xcd_tile(h, nblocks) * ATY + w;
  if (t >= pairs.count()) return;
  int c0, jb, je;
  pairs.item(t, c0, jb, je);
  ade_pair<T, FIRST>(a, pairs.box, c0, jb, je, delay[w]);
}

}  // namespace

template <typename T>
hipError_t launch_ade8_step(const Ade8<T> &a, hipStream_t s) {
  const AdeBox box = ade_pair_box<T>(a.s.nx, a.s.ny, a.npml);
  const dim3 block(BX, ATY);
  const int frame = AdeFrame(a.s.nx, a.s.ny, box).tiles();
  if (box.x1 == 0) {
    // stage 1 reads X0; the states of stages 2..4 alternate between d[1] and d[0]
    for (int inc = 0; inc < 4; ++inc)
      hipLaunchKernelGGL((k_ade_stage<T, true>), dim3(frame), block, 0, s, a, inc, box);
    return hipGetLastError();
  }
  const AdePairs pairs = ade_pairs<T>(box);
  const int nblocks = (pairs.count() + ATY - 1) / ATY;
  const int first = AdeFrame(a.s.nx, a.s.ny, shrink(box, 4)).tiles();
  hipLaunchKernelGGL((k_ade_pair<T, true>), dim3(nblocks + first), block, 0, s, a, pairs, nblocks);
  hipLaunchKernelGGL((k_ade_stage<T, false>), dim3(frame), block, 0, s, a, 1, box);
  hipLaunchKernelGGL((k_ade_pair<T, false>), dim3(nblocks + first), block, 0, s, a, pairs, nblocks);
  hipLaunchKernelGGL((k_ade_stage<T, false>), dim3(frame), block, 0, s, a, 3, box);
  return hipGetLastError();
}

template hipError_t launch_ade8_step<float>(const Ade8<float> &, hipStream_t);
template hipError_t launch_ade8_step<double>(const Ade8<double> &, hipStream_t);

}  // namespace cpml
