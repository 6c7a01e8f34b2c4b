// Time-blocked 2D leapfrog: NT full time steps (stress + C-PML, velocity +
// C-PML, point force, rigid edges) per launch and per pass over HBM, for
// seismic_CPML_2D_isotropic_second_order.f90:550-686 and
// seismic_CPML_2D_isotropic_fourth_order.f90:551-687 (and the Holberg
// operator of seismic_ADEPML_2D_elastic_RK4_eighth_order.f90:263-266 in the
// same leapfrog).
//
// One 64-lane wavefront is one work item: lane l holds column
// i0 - G + l of a strip (G = NT (2r - 1) ring columns on each side, r = ORDER
// / 2) and the wave marches up the rows of one chunk.  At row iteration s the
// wave
//   * loads row s + r of v, row s of sigma and lambda, row s + 1 of mu and
//     row s - r + 1 of the density (one iteration ahead of their use),
//   * for each time level m = 1..NT computes sigma^m at row p = s - 2(m-1)r
//     from the row window of v^{m-1} (2r + 1 rows) and v^m at row p - r from
//     the row window of sigma^m, x neighbours moving across lanes,
//   * stores level NT (sigma at row s - 2(NT-1)r, v at s - (2NT-1)r) for the
//     owned lanes and rows, and records the receivers of every level.
// Every intermediate level stays in registers; the only HBM traffic is the
// state read once (v, sigma, lambda, mu, rho: 8 words per point) and written
// once (5 words) per NT steps.  Each level is valid on 2r - 1 fewer lanes on
// each side than the one before, so after NT levels lanes [G, 63 - G] hold
// correct values; the strip owns `ow` <= 64 - 2G of them.  Rows are handled
// the same way by starting (2NT - 1) r rows below the chunk and ending as far
// above it.  The state is read from one buffer and written to the other
// (ping-pong), so wavefronts never see each other's new values.
//
// The arithmetic of every point is the single-step kernels' (cpml_points2d.h),
// statement by statement, so results are bit-identical to them and to the
// reference association.
//
// Bound by issued instructions, then by HBM (4096^2, order 4, float, 2 steps:
// 13 words per point at 4.8 TB/s would be 185 us; the launch takes 280, of which
// the vector pipes are busy two thirds).  So the march is built to issue little
// beside the arithmetic: x neighbours move by DPP wave shifts instead of LDS
// permutes, the windows are renamed by unrolling the loop over their phases
// instead of being copied, loads run over the zeroed ghost rows and columns
// instead of being predicated, divisions by the launch's grid spacing take four
// instructions (cpml_constdiv.h), rows that only wait for a later level lie in
// LDS, and the owned columns are whole 64-byte sectors (a store of part of one
// reads it back).  Per launch of 2 steps, before and after: 4096^2 order 4
// float 410 -> 280 us; 1701 x 1403 order 2 double with the energy curve 207 ->
// 101; 32 uneven shots of up to 2048 points a side, order 4 float, 1577 -> 990.
#pragma once

#include <algorithm>

#include "cpml_device.h"
#include "cpml_energy.h"
#include "cpml_internal.h"
#include "cpml_tb_geom.h"

namespace cpml {
namespace {

// The description of the grid an item works on, in memory that no kernel
// writes while it runs: the kernel's argument block, or one entry of the
// batch's table.
template <typename T>
using GridPtr = const __attribute__((address_space(4))) TB2D<T> *;
// The same pointer, opaque to the compiler: what is read through it is read
// again instead of being kept (spilled) across rows.
template <typename T>
__device__ __forceinline__ GridPtr<T> reread(GridPtr<T> p) {
  asm volatile("" : "+s"(p));
  return p;
}
__device__ __forceinline__ Slab slab_copy(const __attribute__((address_space(4))) Slab &s) {
  Slab o;
  o.wl = s.wl, o.wr = s.wr, o.w = s.w, o.n = s.n, o.k1 = s.k1;
  return o;
}
template <typename T>
__device__ __forceinline__ ConstDiv<T> div_copy(
    const __attribute__((address_space(4))) ConstDiv<T> &s) {
  ConstDiv<T> o;
  o.d = s.d, o.c = s.c, o.cl = s.cl, o.ch = s.ch, o.hi = s.hi, o.lo = s.lo;
  return o;
}

template <typename T>
__device__ __forceinline__ T ld_el(const T *base, long element) {
  return *((const Glb<T> *)base + element);
}
template <typename T>
__device__ __forceinline__ void st_el(T *base, long element, T x) {
  *((Glb<T> *)base + element) = x;
}

// x difference of this row: DEL 0 between lanes l + 1 and l, 1 between l and
// l - 1; a27 = 27 * x (order 4).  Association as Op<T, ORDER>::d
// (cpml_points2d.h); x neighbours move by DPP wave shifts.
template <int ORDER, int DEL, typename T>
__device__ __forceinline__ T ddx(T x, T a27) {
  if constexpr (ORDER == 2) {
    return DEL ? x - lane_prev(x) : lane_next(x) - x;
  } else if constexpr (ORDER == 4) {
    if (DEL) return a27 - lane_prev(a27) - lane_next(x) + lane_prev(lane_prev(x));
    return lane_next(a27) - a27 - lane_next(lane_next(x)) + lane_prev(x);
  } else {
    const T p1 = lane_next(x), p2 = lane_next(p1), p3 = lane_next(p2);
    const T m1 = lane_prev(x), m2 = lane_prev(m1), m3 = lane_prev(m2);
    if (DEL) {
      const T m4 = lane_prev(m3);
      return T(kHolberg1) * (x - m1) + T(kHolberg2) * (p1 - m2) + T(kHolberg3) * (p2 - m3) +
             T(kHolberg4) * (p3 - m4);
    }
    const T p4 = lane_next(p3);
    return T(kHolberg1) * (p1 - x) + T(kHolberg2) * (p2 - m1) + T(kHolberg3) * (p3 - m2) +
           T(kHolberg4) * (p4 - m3);
  }
}

// y difference on a row window: g(k) = f[p + k rows]; g1, g0: 27 times the two
// middle rows (order 4).
template <int ORDER, typename T, typename G>
__device__ __forceinline__ T ddy(G g, T g1, T g0) {
  if constexpr (ORDER == 2) {
    return g(Int<1>{}) - g(Int<0>{});
  } else if constexpr (ORDER == 4) {
    return g1 - g0 - g(Int<2>{}) + g(Int<-1>{});
  } else {
    return T(kHolberg1) * (g(Int<1>{}) - g(Int<0>{})) + T(kHolberg2) * (g(Int<2>{}) - g(Int<-1>{})) +
           T(kHolberg3) * (g(Int<3>{}) - g(Int<-2>{})) + T(kHolberg4) * (g(Int<4>{}) - g(Int<-3>{}));
  }
}

// Words per lane of an item's delay lines in LDS (tb2d_item): the coefficients
// and, beside a slab, one axis' memory variables.
template <int ORDER, int NT, int CLS>
constexpr int tb2d_delay_words() {
  return (NT - 1) * ORDER * (CLS ? 9 : 5);
}

// One work item: strip ts (columns from ts * ow) and rows [jb, je) of the
// grid described by P, advanced NT steps.  EN: also the energy terms of every
// level at the item's owned points inside the energy window, summed over the
// wavefront and written to item slot `slot` of P.epart.
//
// The march is bound by instruction issue (4096^2, order 4, 2 steps per
// launch, float: 600 vector instructions per row before, 121 of them IEEE
// divisions by 24 DELTA and density and 129 register moves).  So: division by
// the launch constants in 4 instructions and a range test (cpml_constdiv.h); 27 f
// formed once per value and carried to the next row; half-point coefficients formed once
// and carried to the later levels; x neighbours by DPP, folded into the
// arithmetic; no predicates along an axis whose slabs and faces the class
// does not touch; unconditional loads (coordinates clamped to the zero ghost
// points); the rows unrolled by the window length, so windows do not move
// (orders 2 and 4 up to 2 steps: the others would not fit the instruction
// cache).
template <typename T, int ORDER, int NT, int CLS, bool EN = false>
__device__ __forceinline__ void tb2d_item(GridPtr<T> P, int ts, int jb, int je, T *delay,
                                          int ahead, int slot) {
  constexpr bool SX = (CLS & 1) != 0, SY = (CLS & 2) != 0;  // axes this class touches
  constexpr int r = ORDER / 2;
  constexpr int W = 2 * r + 1;                  // row window of one level
  constexpr int G = NT * (2 * r - 1);           // ring lanes on each side
  // rows unrolled by W (slab-free items: the C-PML code would not fit)
  constexpr bool UN = ORDER <= 4 && NT <= 2 && CLS == 0;
  constexpr int NPH = UN ? W : 1;
  constexpr int DC = 2 * (NT - 1) * r;          // rows from level 1 to level NT
  constexpr int DM = 2 * r;                     // rows from one level to the next
  constexpr int WE = EN ? (2 * NT - 1) * r + 1 : 1;  // lambda, mu rows for the energy
  constexpr int NL = NT > 1 ? NT - 1 : 1;       // memory-variable windows (levels 1..NT-1)
  const int nx = P->a.nx, ny = P->a.ny;
  const Slab sx = slab_copy(P->a.sx), sy = slab_copy(P->a.sy);
  const int lane = threadIdx.x & 63;
  const int i = ts * P->ow - G + lane;
  const bool col_in = !SX || (i >= 0 && i < nx);
  const bool xlo = !SX || (i >= 1 && i < nx), xhi = !SX || (i >= 0 && i <= nx - 2);
  const bool own_lane = lane >= G && lane < G + P->ow && (!SX || i < nx);
  auto row_in = [&](int j) { return !SY || (j >= 0 && j < ny); };
  auto ylo = [&](int j) { return !SY || (j >= 1 && j < ny); };
  auto yhi = [&](int j) { return !SY || (j >= 0 && j <= ny - 2); };

  const int s0 = jb - (2 * NT - 1) * r, s1 = je - 1 + (2 * NT - 1) * r;
  const Tb2dLane<T, SX, SY> L(i, s0 - r, nx, ny, P->a.ld, sx);
  const long corner = L.corner;
  const bool inx = L.inx, kx1 = sx.k1, ky1 = sy.k1;
  auto at = [&](int j) { return L.at(j); };
  auto ox = [&](int j) { return L.ox(j); };
  T pxa = T(0), pxb = T(0), pxah = T(0), pxbh = T(0);
  if (SX && inx) pxa = P->a.px.a[i], pxb = P->a.px.b[i], pxah = P->a.px.ah[i], pxbh = P->a.px.bh[i];

  // ---- row windows
  T V[NT][2][W];        // v^m, m = 0..NT-1: rows q_m - 2r .. q_m (q_0 = s + r)
  T S[NT][3][W];        // sigma^m, m = 1..NT: rows p_m - 2r .. p_m
  T El[WE], Em[WE];     // lambda, mu: rows s - (2NT-1)r .. s (energy)
  // Values a later level needs again a fixed number of rows on wait in this
  // lane's words of LDS (rings; no other lane touches them): the coefficients
  // of level 1 -- lambda and lambda+2mu at i+1/2, mu at j+1/2, density and its
  // mean at (i+1/2, j+1/2) -- and the memory variables of levels 1..NT-1 (x [0]
  // dvx_dx [1] dvy_dx [2] dsxx_dx [3] dsxy_dx, y [0] dvy_dy [1] dvx_dy
  // [2] dsxy_dy [3] dsyy_dy).  In registers they took 20 and 40 of them (order
  // 4) and as many moves per row.
  T *const dl = delay + lane;
  auto coef = [&](int q, int pos) -> T & { return dl[(q * DC + pos) * 64]; };
  auto slab_mem = [&](int m, int q, int pos) -> T & {
    return dl[(5 * DC + ((m - 1) * 4 + q) * DM + pos) * 64];
  };
  // corner items (both slabs): their y memory variables wait in registers, so
  // that all classes fit the same LDS
  T wy[NL][4][DM];
  if constexpr (SX && SY)
#pragma unroll
    for (int m = 0; m < NL; ++m)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int k = 0; k < DM; ++k) wy[m][q][k] = T(0);
  auto old_y = [&](int m, int q, int pos) -> T {
    if constexpr (SX) return wy[m - 1][q][0];
    else return slab_mem(m, q, pos);
  };
  for (int q = 0; q < tb2d_delay_words<ORDER, NT, CLS>(); ++q) dl[q * 64] = T(1);
  int pc = 0, pm = 0;   // this row's places in the rings (DC and DM rows long)
  // 27 f of the row that is a middle row of the next iteration's y differences
  T c_vx[NT], c_vy[NT], c_yy[NT], c_xy[NT];
#pragma unroll
  for (int m = 0; m < NT; ++m) {
    c_vx[m] = c_vy[m] = c_yy[m] = c_xy[m] = T(0);
#pragma unroll
    for (int k = 0; k < W; ++k) {
      V[m][0][k] = V[m][1][k] = T(0);
      S[m][0][k] = S[m][1][k] = S[m][2][k] = T(0);
    }
  }
#pragma unroll
  for (int k = 0; k < WE; ++k) El[k] = Em[k] = T(1);

  // rows to come: v row s + r, sigma and lambda row s, mu row s + 1, density
  // row s - r + 1, level-1 memory variables (sigma phase row s, velocity
  // phase row s - r)
  T nvx, nvy, nxx, nyy, nxy, nlam, nmu, nrho, lx[4], ly[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) lx[q] = ly[q] = T(0);
  auto load_v = [&](GridPtr<T> Q, int j) {
    const unsigned o = at(j);
    nvx = ld_at(Q->a.vx + corner, o), nvy = ld_at(Q->a.vy + corner, o);
  };
  auto load_s = [&](GridPtr<T> Q, int j) {
    const unsigned o = at(j);
    nxx = ld_at(Q->a.sxx + corner, o), nyy = ld_at(Q->a.syy + corner, o);
    nxy = ld_at(Q->a.sxy + corner, o), nlam = ld_at(Q->a.lam + corner, o);
    nmu = ld_at(Q->a.mu + corner, at(j + 1));
  };
  // memory variables [F, F + 2) of row j
  auto load_m = [&](GridPtr<T> Q, auto first, int j) {
    constexpr int F = decltype(first)::value;
    if (SX) {
      lx[F] = lx[F + 1] = T(0);
      if (inx && row_in(j)) {
        const long o = ox(j);
        lx[F] = ld_el(Q->a.mx[F], o), lx[F + 1] = ld_el(Q->a.mx[F + 1], o);
      }
    }
    if (SY) {
      ly[F] = ly[F + 1] = T(0);
      if (col_in && sy.in(j)) {
        const long b = Q->a.mld * sy.s(j);
        ly[F] = ld_at(Q->a.my[F] + b, L.mo);
        ly[F + 1] = ld_at(Q->a.my[F + 1] + b, L.mo);
      }
    }
  };
  // prologue: v rows s0 - r .. s0 + r - 1 (window places of phase 0)
#pragma unroll
  for (int k = 0; k < W - 1; ++k) {
    const unsigned o = at(s0 - r + k);
    V[0][0][k + 1] = ld_at(P->a.vx + corner, o);
    V[0][1][k + 1] = ld_at(P->a.vy + corner, o);
  }
  if constexpr (ORDER == 4) {
    c_vx[0] = T(27) * V[0][0][1 + r];
    c_vy[0] = T(27) * V[0][1][r];
  }
  T mu_c = ld_at(P->a.mu + corner, at(s0)), rho_c = ld_at(P->a.rho + corner, at(s0 - r));
  load_v(P, s0 + r);
  load_s(P, s0);
  nrho = ld_at(P->a.rho + corner, at(s0 - r + 1));
  if (SX || SY) {
    load_m(P, Int<0>{}, s0);
    load_m(P, Int<2>{}, s0 - r);
  }

  // receivers of this strip: a cursor per level (rows only increase), the row
  // of the next one held in a register
  constexpr int kNever = 0x7fffffff;
  int rc1 = 0, cur[NT], rk[NT];
#pragma unroll
  for (int m = 0; m < NT; ++m) cur[m] = 0, rk[m] = kNever;
  if (P->nrec > 0) {
    rc1 = __builtin_amdgcn_readfirstlane(P->rec_start[ts + 1]);
    const int c = first_from(P->rec_j, P->rec_start[ts], rc1, jb);
    const int j0 = c < rc1 ? __builtin_amdgcn_readfirstlane(P->rec_j[c]) : kNever;
#pragma unroll
    for (int m = 0; m < NT; ++m) cur[m] = c, rk[m] = j0;
  }
  const int it0 = *P->a.step + ahead;  // this launch's first step
  double ek[NT], ep[NT];  // energy terms per level (EN)
#pragma unroll
  for (int m = 0; m < NT; ++m) ek[m] = ep[m] = 0.0;
  const bool ecol = EN && own_lane && i >= P->ew[0] && i <= P->ew[1];

  auto row = [&](auto phase, int s) {
    constexpr int PH = decltype(phase)::value;
    // items with C-PML code have more pointers than fit in scalar registers:
    // re-read per row (scalar loads, cached)
    const GridPtr<T> Q = SX || SY ? reread(P) : P;
    const ConstDiv<T> div_x = div_copy(Q->a.div_x), div_y = div_copy(Q->a.div_y);
    const T dt = Q->a.dt;
    // place of row k of a window (k = W - 1: newest)
    auto wi = [](int k) { return UN ? (PH + 1 + k) % W : k; };
    auto push = [&](T(&w)[W], T x) {
      if constexpr (UN) {
        w[PH] = x;
      } else {
#pragma unroll
        for (int k = 0; k < W - 1; ++k) w[k] = w[k + 1];
        w[W - 1] = x;
      }
    };
    push(V[0][0], nvx);
    push(V[0][1], nvy);
    if (s < s1) load_v(Q, s + r + 1);
    // coefficients of stress row s and velocity row s - r, per level
    T cf[NT][5];
#pragma unroll
    for (int m = 1; m < NT; ++m) {
      const int ago = pc - m * DM, pos = ago < 0 ? ago + DC : ago;
#pragma unroll
      for (int q = 0; q < 5; ++q) cf[m][q] = coef(q, pos);
    }
    {
      cf[0][0] = T(0.5) * (lane_next(nlam) + nlam);
      const T mhx = T(0.5) * (lane_next(mu_c) + mu_c);
      cf[0][1] = cf[0][0] + T(2) * mhx;
      cf[0][2] = T(0.5) * (nmu + mu_c);
      cf[0][3] = rho_c;
      cf[0][4] = T(0.25) * (rho_c + lane_next(rho_c) + lane_next(nrho) + nrho);
      if (NT > 1)
#pragma unroll
        for (int q = 0; q < 5; ++q) coef(q, pc) = cf[0][q];
      if (EN) {
#pragma unroll
        for (int k = 0; k < WE - 1; ++k) El[k] = El[k + 1], Em[k] = Em[k + 1];
        El[WE - 1] = nlam, Em[WE - 1] = mu_c;
      }
      mu_c = nmu;
      rho_c = nrho;
    }

    T px[NL][4], py[NL][4];  // new memory variables of levels 1..NT-1
    auto level = [&](auto lev) {
      constexpr int m = decltype(lev)::value;
      constexpr int D = 2 * (m - 1) * r;
      const int pr = s - D;   // sigma row
      const int qr = pr - r;  // velocity row
      constexpr int mb = m >= 2 ? m - 2 : 0;  // previous level's windows
      // ---------------- sigma^m at row pr: 2D2:556-600 (2D4:557-601)
      T sxx = m == 1 ? nxx : S[mb][0][wi(0)];
      T syy = m == 1 ? nyy : S[mb][1][wi(0)];
      T sxy = m == 1 ? nxy : S[mb][2][wi(0)];
      T ox0 = lx[0], ox1 = lx[1], oy0 = ly[0], oy1 = ly[1];
      if (SX && m > 1) ox0 = slab_mem(m - 1, 0, pm), ox1 = slab_mem(m - 1, 1, pm);
      if (SY && m > 1) oy0 = old_y(m - 1, 0, pm), oy1 = old_y(m - 1, 1, pm);
      T npx0 = ox0, npx1 = ox1, npy0 = oy0, npy1 = oy1;
      {
        const T(&wx)[W] = V[m - 1][0];  // vx rows pr - r .. pr + r
        const T(&wy)[W] = V[m - 1][1];
        const T vxc = wx[wi(r)], vyc = wy[wi(r)];
        const T x27 = c_vx[m - 1], xn27 = T(27) * wx[wi(r + 1)];  // vx rows pr, pr + 1
        const T yp27 = c_vy[m - 1], y27 = T(27) * vyc;            // vy rows pr - 1, pr
        c_vx[m - 1] = xn27;
        c_vy[m - 1] = y27;
        T dvx_dx = ddx<ORDER, 0>(vxc, x27);
        T dvy_dx = ddx<ORDER, 1>(vyc, y27);
        T dvy_dy = ddy<ORDER>([&](auto k) { return wy[wi(r - 1 + decltype(k)::value)]; }, y27, yp27);
        T dvx_dy = ddy<ORDER>([&](auto k) { return wx[wi(r + decltype(k)::value)]; }, xn27, x27);
        const_divide(dvx_dx, div_x, dvy_dy, div_y, dvy_dx, div_x, dvx_dy, div_y);
        const bool iny = SY && sy.in(pr);
        T pya = T(0), pyb = T(0), pyah = T(0), pybh = T(0);
        if (SY && iny) pya = Q->a.py.a[pr], pyb = Q->a.py.b[pr], pyah = Q->a.py.ah[pr], pybh = Q->a.py.bh[pr];
        if (ylo(pr) && xhi) {
          const T lhx = cf[m - 1][0], lp2m = cf[m - 1][1];
          if (SX) dvx_dx = pml(inx, kx1, dvx_dx, ox0, npx0, pxah, pxbh, Q->a.px.Kh + i);
          if (SY) dvy_dy = pml(iny, ky1, dvy_dy, oy0, npy0, pya, pyb, Q->a.py.K + pr);
          sxx = sxx + (lp2m * dvx_dx + lhx * dvy_dy) * dt;
          syy = syy + (lhx * dvx_dx + lp2m * dvy_dy) * dt;
        }
        if (yhi(pr) && xlo) {
          if (SX) dvy_dx = pml(inx, kx1, dvy_dx, ox1, npx1, pxa, pxb, Q->a.px.K + i);
          // 2D4:596 divides by K_y(j) where 2D2:595 uses K_y_half(j)
          if (SY)
            dvx_dy = pml(iny, ky1, dvx_dy, oy1, npy1, pyah, pybh,
                         (ORDER == 4 ? Q->a.py.K : Q->a.py.Kh) + pr);
          sxy = sxy + cf[m - 1][2] * (dvy_dx + dvx_dy) * dt;
        }
      }
      push(S[m - 1][0], sxx);
      push(S[m - 1][1], syy);
      push(S[m - 1][2], sxy);
      if constexpr (m < NT) {
        if (SX) px[m - 1][0] = npx0, px[m - 1][1] = npx1;
        if (SY) py[m - 1][0] = npy0, py[m - 1][1] = npy1;
      }
      if (m == NT && pr >= jb && pr < je && own_lane) {
        const unsigned o = at(pr);
        st_at(Q->sxx + corner, o, sxx);
        st_at(Q->syy + corner, o, syy);
        st_at(Q->sxy + corner, o, sxy);
        if (SX && inx) {
          const long ob = ox(pr);
          st_el(Q->mx[0], ob, npx0);
          st_el(Q->mx[1], ob, npx1);
        }
        if (SY && sy.in(pr)) {
          const long b = Q->a.mld * sy.s(pr);
          st_at(Q->my[0] + b, L.mo, npy0);
          st_at(Q->my[1] + b, L.mo, npy1);
        }
      }
      if (m == 1 && s < s1) {
        load_s(Q, s + 1);
        nrho = ld_at(Q->a.rho + corner, at(s - r + 2));
        if (SX || SY) load_m(Q, Int<0>{}, s + 1);
      }
      // ---------------- v^m at row qr: 2D2:606-680 (2D4:607-681)
      T vxn = V[m - 1][0][wi(0)], vyn = V[m - 1][1][wi(0)];
      T ox2 = lx[2], ox3 = lx[3], oy2 = ly[2], oy3 = ly[3];
      if (SX && m > 1) ox2 = slab_mem(m - 1, 2, pm), ox3 = slab_mem(m - 1, 3, pm);
      if (SY && m > 1) oy2 = old_y(m - 1, 2, pm), oy3 = old_y(m - 1, 3, pm);
      T npx2 = ox2, npx3 = ox3, npy2 = oy2, npy3 = oy3;
      const T rho = cf[m - 1][3], rhh = cf[m - 1][4];
      {
        const T(&wxx)[W] = S[m - 1][0];  // rows qr - r .. qr + r
        const T(&wyy)[W] = S[m - 1][1];
        const T(&wxy)[W] = S[m - 1][2];
        const T sxxc = wxx[wi(r)], sxyc = wxy[wi(r)];
        const T y27 = c_yy[m - 1], yn27 = T(27) * wyy[wi(r + 1)];  // sigma_yy rows qr, qr + 1
        const T sp27 = c_xy[m - 1], s27 = T(27) * sxyc;            // sigma_xy rows qr - 1, qr
        c_yy[m - 1] = yn27;
        c_xy[m - 1] = s27;
        T dsxx_dx = ddx<ORDER, 1>(sxxc, T(27) * sxxc);
        T dsxy_dx = ddx<ORDER, 0>(sxyc, s27);
        T dsxy_dy = ddy<ORDER>([&](auto k) { return wxy[wi(r - 1 + decltype(k)::value)]; }, s27, sp27);
        T dsyy_dy = ddy<ORDER>([&](auto k) { return wyy[wi(r + decltype(k)::value)]; }, yn27, y27);
        const_divide(dsxx_dx, div_x, dsxy_dy, div_y, dsxy_dx, div_x, dsyy_dy, div_y);
        const bool iny = SY && sy.in(qr);
        T pya = T(0), pyb = T(0), pyah = T(0), pybh = T(0);
        if (SY && iny) pya = Q->a.py.a[qr], pyb = Q->a.py.b[qr], pyah = Q->a.py.ah[qr], pybh = Q->a.py.bh[qr];
        if (ylo(qr) && xlo) {
          if (SX) dsxx_dx = pml(inx, kx1, dsxx_dx, ox2, npx2, pxa, pxb, Q->a.px.K + i);
          if (SY) dsxy_dy = pml(iny, ky1, dsxy_dy, oy2, npy2, pya, pyb, Q->a.py.K + qr);
          vxn = vxn + (dsxx_dx + dsxy_dy) * dt / rho;
        }
        if (yhi(qr) && xhi) {
          if (SX) dsxy_dx = pml(inx, kx1, dsxy_dx, ox3, npx3, pxah, pxbh, Q->a.px.Kh + i);
          if (SY) dsyy_dy = pml(iny, ky1, dsyy_dy, oy3, npy3, pyah, pybh, Q->a.py.Kh + qr);
          vyn = vyn + (dsxy_dx + dsyy_dy) * dt / rhh;
        }
        // point force at step it0 + m - 1, after the update (2D2:660-667)
        if (qr == Q->a.jsrc && qr >= 0 && i == Q->a.isrc) {
          const int it = it0 + m - 1;
          vxn = vxn + Q->a.fx[it - 1] * dt / rho;
          vyn = vyn + Q->a.fy[it - 1] * dt / rhh;
        }
        // rigid edges (2D2:670-680), and nothing outside the grid
        if ((SX && (i <= 0 || i >= nx - 1)) || (SY && (qr <= 0 || qr >= ny - 1))) vxn = vyn = T(0);
        // energy of step it0 + m - 1 at (i, j): v^m, sigma^m of this row
        // (the middle of the sigma window) and the row's medium
        if (EN && qr >= jb && qr < je && qr >= Q->ew[2] && qr <= Q->ew[3] && ecol)
          point_energy2d(vxn, vyn, wxx[wi(r)], wyy[wi(r)], wxy[wi(r)],
                         El[EN ? WE - 1 - (2 * m - 1) * r : 0],
                         Em[EN ? WE - 1 - (2 * m - 1) * r : 0], rho, ek[m - 1], ep[m - 1]);
      }
      // receivers of step it0 + m - 1 on this row (owned rows only)
      if (qr == rk[m - 1] && qr < je) {
        int c = cur[m - 1], nk = qr;
        while (nk == qr) {
          if (Q->rec_i[c] == i && own_lane) {
            const long o = (long)(it0 + m - 2) * Q->nrec + Q->rec_slot[c];
            Q->sisx[o] = vxn;
            Q->sisy[o] = vyn;
          }
          ++c;
          nk = c < rc1 ? __builtin_amdgcn_readfirstlane(Q->rec_j[c]) : kNever;
        }
        cur[m - 1] = c;
        rk[m - 1] = nk;
      }
      if constexpr (m < NT) {
        push(V[m][0], vxn);
        push(V[m][1], vyn);
        if (SX) px[m - 1][2] = npx2, px[m - 1][3] = npx3;
        if (SY) py[m - 1][2] = npy2, py[m - 1][3] = npy3;
      } else if (qr >= jb && qr < je && own_lane) {
        const unsigned o = at(qr);
        st_at(Q->vx + corner, o, vxn);
        st_at(Q->vy + corner, o, vyn);
        if (SX && inx) {
          const long ob = ox(qr);
          st_el(Q->mx[2], ob, npx2);
          st_el(Q->mx[3], ob, npx3);
        }
        if (SY && sy.in(qr)) {
          const long b = Q->a.mld * sy.s(qr);
          st_at(Q->my[2] + b, L.mo, npy2);
          st_at(Q->my[3] + b, L.mo, npy3);
        }
      }
      if ((SX || SY) && m == 1 && s < s1) load_m(Q, Int<2>{}, s + 1 - r);
    };
    level(Int<1>{});
    if constexpr (NT > 1) level(Int<2>{});
    if constexpr (NT > 2) level(Int<3>{});
    if constexpr (NT > 3) level(Int<4>{});
    if constexpr (NT > 1 && (SX || SY)) {  // into the places the next levels have read
#pragma unroll
      for (int m = 1; m < NT; ++m)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          if (SX) slab_mem(m, q, pm) = px[m - 1][q];
          if constexpr (SX && SY) {
#pragma unroll
            for (int k = 0; k < DM - 1; ++k) wy[m - 1][q][k] = wy[m - 1][q][k + 1];
            wy[m - 1][q][DM - 1] = py[m - 1][q];
          } else if (SY) {
            slab_mem(m, q, pm) = py[m - 1][q];
          }
        }
    }
    if (NT > 1) {
      pc = pc == DC - 1 ? 0 : pc + 1;
      pm = pm == DM - 1 ? 0 : pm + 1;
    }
  };
  for (int s = s0;; s += NPH) {
    row(Int<0>{}, s);
    if (s == s1) break;
    if constexpr (NPH > 1) {
      row(Int<1>{}, s + 1);
      if (s + 1 == s1) break;
      row(Int<2>{}, s + 2);
      if (s + 2 == s1) break;
    }
    if constexpr (NPH > 3) {
      row(Int<3>{}, s + 3);
      if (s + 3 == s1) break;
      row(Int<4>{}, s + 4);
      if (s + 4 == s1) break;
    }
  }
  if (EN) {  // wavefront sums in a fixed order, lane 0 writes the item's slot
#pragma unroll
    for (int m = 0; m < NT; ++m) {
      double a = ek[m], b = ep[m];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        a += __shfl_xor(a, o, 64);
        b += __shfl_xor(b, o, 64);
      }
      if (lane == 0) {
        P->epart[((long)m * P->eslots + slot) * 2] = a;
        P->epart[((long)m * P->eslots + slot) * 2 + 1] = b;
      }
    }
  }
}

constexpr int WPB = 4;  // wavefronts (work items) per workgroup

// Waves per SIMD the kernels are built for: what the slab-free code's registers
// leave (orders 2 and 4 up to 2 steps; the C-PML code of the same kernel spills
// a little at the corners for it).
template <typename T, int ORDER, int NT>
constexpr int min_waves() {
  if (ORDER > 4 || NT > 2) return 1;
  return sizeof(T) == 4 ? 4 : 2;
}

// One item of class cls (bit 0: the x slabs' C-PML code and predicates, bit 1:
// the y slabs').  All classes are one kernel: a launch of its own per class
// costs a fork and a join of streams (20 us of 300 per launch at 4096^2), and
// the slab items, few and long, have to start before the slab-free ones fill
// the machine.
template <typename T, int ORDER, int NT, bool EN>
__device__ __forceinline__ void tb2d_any(GridPtr<T> P, int cls, int ts, int jb, int je, T *delay,
                                         int ahead, int slot) {
  if (cls == 0) tb2d_item<T, ORDER, NT, 0, EN>(P, ts, jb, je, delay, ahead, slot);
  else if (cls == 1) tb2d_item<T, ORDER, NT, 1, EN>(P, ts, jb, je, delay, ahead, slot);
  else if (cls == 2) tb2d_item<T, ORDER, NT, 2, EN>(P, ts, jb, je, delay, ahead, slot);
  else tb2d_item<T, ORDER, NT, 3, EN>(P, ts, jb, je, delay, ahead, slot);
}

// Item u of those XCD xcd gets: its contiguous share of the nslab items with
// C-PML code (the list's first), then of the nclean others; -1 past the end.
__device__ __forceinline__ int xcd_item(int xcd, int u, int nslab, int nclean) {
  const int qs = nslab >> 3, rs = nslab & 7, ns = qs + (xcd < rs ? 1 : 0);
  if (u < ns) return xcd * qs + min(xcd, rs) + u;
  const int qc = nclean >> 3, rc = nclean & 7, nc = qc + (xcd < rc ? 1 : 0);
  u -= ns;
  return u < nc ? nslab + xcd * qc + min(xcd, rc) + u : -1;
}
// Most items an XCD gets.
inline int xcd_items(int nslab, int nclean) { return (nslab + 7) / 8 + (nclean + 7) / 8; }

}  // namespace
}  // namespace cpml
