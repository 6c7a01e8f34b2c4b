// Time-blocked 3D leapfrog: NT full time steps (stress + C-PML, velocity +
// C-PML, point force, rigid faces) per launch and per pass over HBM, for
// seismic_CPML_3D_isotropic_MPI_OpenMP.f90:836-1121 (the two OpenMP phases of
// NT consecutive `do it` iterations).
//
// A workgroup is NW wavefronts; wave w holds grid row j0 - NT + w and lane l
// column i0 - NT + l, and the group marches through the z planes of one
// chunk.  At plane iteration s it
//   * for each time level m = 1..NT computes sigma^m at plane p = s - 2(m-1)
//     from the 3-plane column window of v^{m-1}, then v^m at plane p - 1
//     from the 3-plane window of sigma^m, and issues the loads of the next
//     iteration (v at s + 2, sigma and the coefficients at s + 1, the level-1
//     memory variables) as level 1 frees their registers; x neighbours move
//     across lanes, y neighbours through LDS (written the iteration before:
//     one barrier per plane, two buffers),
//   * stores level NT (sigma at s - 2(NT-1), v at s - 2NT + 1) for the owned
//     points and planes, and records the receivers of every level.
// Every intermediate level stays in registers and LDS; HBM sees the state
// read once (v 3, sigma 6, DELTAT*lambda, DELTAT*mu, DELTAT/rho: 12 words)
// and written once (9 words) per NT steps, plus the slab memory variables
// (read and written once per NT steps).  Each level is valid one lane and
// one row fewer on each side (the staggered differences reach one point),
// so a group owns 64 - 2NT columns (or fewer) x NW - 2NT rows; z is handled
// the same way by starting 2NT - 1 planes below the chunk and ending as far
// above it.  State is read from one buffer and written to the other.
//
// Per point the arithmetic is exactly the two-phase kernels' (same
// expressions, no FMA contraction), so results are bit-identical to them.
//
// Tiles are split by the axes along which their points and ring touch an
// absorbing slab or a grid face; each class has code with just the C-PML terms
// and the predicates of those axes.  All are one kernel, the classes with the
// most of them first: a launch per class on streams of their own cost 20 us per
// launch and 768^3 12.5 ms against 12.3.
#include "cpml_device.h"
#include "cpml_internal.h"
#include "cpml_tb_geom.h"

namespace cpml {
namespace {

// Plane slot of a 3-plane window in the iteration of phase PH (the march is
// unrolled by 3, so slots are compile-time constants and no window moves).
template <int PH, int K>
constexpr int slot_of() {
  return ((PH + K) % 3 + 3) % 3;
}
// What bounds the march (float, 2 steps, 768^3, milliseconds per launch; boxes
// differ by a few percent, pairs are from one box):
//  * stores of part of a cache line.  A copy of 12 arrays read and 9 written
//    in this tile pattern takes 12.9 ms with rows of 56 owned points (224
//    bytes, so tiles share lines and the memory must merge them), 8.5 with 48
//    (whole 64-byte sectors, non-temporal) and 7.6 with whole 128-byte lines;
//    re-reading the ring costs almost nothing beside that.  Hence strips of
//    whole sectors by default and non-temporal state stores: 15.1 -> 12.5.
//  * instruction issue: the first form had 523 scalar instructions of 816 per
//    plane (execution masks around every predicate and load, buffer resources
//    rebuilt from the argument block).  Now an axis without slab flag has no
//    predicates (its tiles and rings lie strictly inside the grid); loads are
//    unconditional (coordinates clamped to the zero ghost points once per
//    tile, planes once per iteration; a scalar base and one 32-bit lane
//    offset); x neighbours move by DPP wave shifts folded into the
//    subtractions; the march is unrolled by the window length, so windows do
//    not move: 455 instructions, and 3.9 ms for the slab-free class with all
//    loads hitting the L2, against 7.8 in earnest.
//  * register spills in the x-slab class wrote more than the fields (5.9 GB
//    per launch against 2.3 without): its updates are branches, not
//    selections, and K is read only where it is not 1.
// Loads two planes ahead (128 registers, 15 spilled): 16.8 against 15.1.
template <typename T, int NT, int NW, bool SX, bool SY, bool SZ>
__device__ __forceinline__ void tb3d_tile(const TB3D<T> &P, int t, T *xl) {
  constexpr bool SLAB = SX || SY || SZ;
  constexpr int NL = NT > 1 ? NT - 1 : 1;      // memory-variable windows (levels 1..NT-1)
  constexpr int NS = 6 * NT;                   // LDS slots per buffer
  const Step3D<T> &p = P.a;
  const int nx = p.nx, ny = p.ny, nz = p.nz;
  const Tb3dTile ft = tb3d_tile_at<SX, SY, SZ>(P, t, nx, ny, nz, p.kchunk);
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = ft.i0 - NT + lane, j = ft.j0 - NT + w;
  const bool col_in = !SX || (i >= 0 && i < nx), row_in = !SY || (j >= 0 && j < ny);
  const bool own = lane >= NT && lane < NT + P.ow && w >= NT && w < NT + P.ty &&
                   (!SX || i < nx) && (!SY || j < ny);
  const int kb = ft.kb, ke = ft.ke;
  // predicates of the update ranges: x per lane, y and z per wavefront
  const bool xlo = !SX || (i >= 1 && i < nx), xhi = !SX || (i >= 0 && i <= nx - 2);
  const bool ylo = !SY || (j >= 1 && j < ny), yhi = !SY || (j >= 0 && j <= ny - 2);
  auto zlo = [&](int k) { return !SZ || (k >= 1 && k < nz); };
  auto zhi = [&](int k) { return !SZ || (k >= 0 && k <= nz - 2); };

  const int s0 = kb - (2 * NT - 1), s1 = ke - 1 + (2 * NT - 1);
  const Tb3dLane<T, SX, SY, SZ> L(i, j, s0 - 1, p);
  const long corner = L.corner;
  auto pl = [&](int k) { return L.at(k); };
  const T *const ivx = p.vx + corner, *const ivy = p.vy + corner, *const ivz = p.vz + corner;
  const T *const ixx = p.sxx + corner, *const iyy = p.syy + corner, *const izz = p.szz + corner;
  const T *const ixy = p.sxy + corner, *const ixz = p.sxz + corner, *const iyz = p.syz + corner;
  const T *const icl = p.clam + corner, *const icm = p.cmu + corner, *const icb = p.cbuoy + corner;
  using KArgs = const __attribute__((address_space(4))) TB3D<T> *;
  auto args = [&]() -> KArgs { return kernarg<TB3D<T>>(); };

  // x/y slab membership and profiles (loop invariant)
  const bool inx = L.inx, iny = L.iny;
  T X[4] = {T(0), T(0), T(0), T(0)}, Y[4] = {T(0), T(0), T(0), T(0)};  // a, b, a_half, b_half
  if (SX && inx) X[0] = p.px.a[i], X[1] = p.px.b[i], X[2] = p.px.ah[i], X[3] = p.px.bh[i];
  if (SY && iny) Y[0] = p.py.a[j], Y[1] = p.py.b[j], Y[2] = p.py.ah[j], Y[3] = p.py.bh[j];
  const bool kx1 = p.sx.k1, ky1 = p.sy.k1, kz1 = p.sz.k1;
  const unsigned mxo = L.mxo, myo = L.myo, mzo = L.mzo;
  const bool mx_on = SX && inx && row_in, my_on = SY && iny && col_in, mz_on = col_in && row_in;
  const long mxs = L.mxs, mys = L.mys, mzs = L.mzs;

  // ---- column windows by plane (slot_of)
  T V[NT][3][3];    // v^m (m = 0..NT-1): vx vy vz
  T S[NT][6][3];    // sigma^m (m = 1..NT): xx yy zz xy xz yz
  T Cl[3], Cm[3], Cb[3];
  // memory variables of levels 1..NT-1 per slab axis: [0..2] the stress
  // phase's (x: dvx_dx dvy_dx dvz_dx, ...), [3..5] the velocity phase's
  T MX[NL][6][3], MY[NL][6][3], MZ[NL][6][3];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    Cl[k] = Cm[k] = Cb[k] = T(0);
#pragma unroll
    for (int m = 0; m < NT; ++m) {
#pragma unroll
      for (int f = 0; f < 3; ++f) V[m][f][k] = T(0);
#pragma unroll
      for (int f = 0; f < 6; ++f) S[m][f][k] = T(0);
    }
#pragma unroll
    for (int m = 0; m < NL; ++m)
#pragma unroll
      for (int f = 0; f < 6; ++f) MX[m][f][k] = MY[m][f][k] = MZ[m][f][k] = T(0);
  }

  // values in flight: sigma and DELTAT*lambda, DELTAT*mu of the plane to come,
  // DELTAT/rho of the plane below it, level-1 memory variables
  T so[6], ncl, ncm, ncb, nv0[3], lx[6], ly[6], lz[6];
#pragma unroll
  for (int f = 0; f < 6; ++f) lx[f] = ly[f] = lz[f] = T(0);
  auto load_s = [&](int k) {
    const unsigned o = pl(k);
    so[0] = ld_at(ixx, o), so[1] = ld_at(iyy, o), so[2] = ld_at(izz, o);
    so[3] = ld_at(ixy, o), so[4] = ld_at(ixz, o), so[5] = ld_at(iyz, o);
    ncl = ld_at(icl, o), ncm = ld_at(icm, o);
  };
  auto load_v = [&](int k) {  // v of plane k, buoyancy of plane k - 2
    const unsigned o = pl(k);
    nv0[0] = ld_at(ivx, o), nv0[1] = ld_at(ivy, o), nv0[2] = ld_at(ivz, o);
    ncb = ld_at(icb, pl(k - 2));
  };
  // memory variables of the stress (F = 0) or velocity (F = 3) phase, plane k
  auto load_m = [&](auto first, int k) {
    constexpr int F = decltype(first)::value;
    const KArgs Q = args();
    const bool kin = !SZ || (k >= 0 && k < nz);
    if (SX) {
#pragma unroll
      for (int f = F; f < F + 3; ++f) lx[f] = T(0);
      if (mx_on && kin)
#pragma unroll
        for (int f = F; f < F + 3; ++f) lx[f] = ld_at(Q->a.mx[f] + mxs * k, mxo);
    }
    if (SY) {
#pragma unroll
      for (int f = F; f < F + 3; ++f) ly[f] = T(0);
      if (my_on && kin)
#pragma unroll
        for (int f = F; f < F + 3; ++f) ly[f] = ld_at(Q->a.my[f] + mys * k, myo);
    }
    if (SZ) {
#pragma unroll
      for (int f = F; f < F + 3; ++f) lz[f] = T(0);
      if (mz_on && p.sz.in(k))
#pragma unroll
        for (int f = F; f < F + 3; ++f) lz[f] = ld_at(Q->a.mz[f] + mzs * p.sz.s(k), mzo);
    }
  };

  const int own_row = 64 + w * 64 + lane;  // this thread's word of LDS slot 0, buffer 0
  constexpr int SLOT = NW * 64, BUF = NS * SLOT;
  // prologue (phase 0): v planes s0 - 1 .. s0 + 1, sigma and coefficients of s0
  {
    V[0][0][slot_of<0, -1>()] = ld_at(ivx, pl(s0 - 1));
    V[0][1][slot_of<0, -1>()] = ld_at(ivy, pl(s0 - 1));
    V[0][2][slot_of<0, -1>()] = ld_at(ivz, pl(s0 - 1));
    V[0][0][slot_of<0, 0>()] = ld_at(ivx, pl(s0));
    V[0][1][slot_of<0, 0>()] = ld_at(ivy, pl(s0));
    V[0][2][slot_of<0, 0>()] = ld_at(ivz, pl(s0));
    load_s(s0);
    load_v(s0 + 1);
    if (SLAB) {
      load_m(Int<0>{}, s0);
      load_m(Int<3>{}, s0 - 1);
    }
    // LDS cleared, then the y neighbours of v at plane s0 for the first
    // iteration (which reads buffer 1)
    for (int q = threadIdx.x; q < 2 * BUF + 128; q += 64 * NW) xl[q] = T(0);
    __syncthreads();
    xl[BUF + own_row] = V[0][0][slot_of<0, 0>()];
    xl[BUF + own_row + SLOT] = V[0][1][slot_of<0, 0>()];
    xl[BUF + own_row + 2 * SLOT] = V[0][2][slot_of<0, 0>()];
  }
  __syncthreads();

  // receivers of this tile: a cursor per level (planes only increase), the
  // plane of the next one held in a register
  const int tix = ft.ty * ((nx + P.ow - 1) / P.ow) + ft.tx;
  constexpr int kNever = 0x7fffffff;
  int rc1 = 0, cur[NT], rk[NT];
#pragma unroll
  for (int m = 0; m < NT; ++m) cur[m] = 0, rk[m] = kNever;
  if (P.nrec > 0) {
    rc1 = __builtin_amdgcn_readfirstlane(P.rec_start[tix + 1]);
    const int c = first_from(P.rec_k, P.rec_start[tix], rc1, kb);
    const int k0 = c < rc1 ? __builtin_amdgcn_readfirstlane(P.rec_k[c]) : kNever;
#pragma unroll
    for (int m = 0; m < NT; ++m) cur[m] = c, rk[m] = k0;
  }
  const int it0 = *p.step + P.ahead;  // this launch's first step
  // the source's column: its plane if this wavefront holds its row
  const int ksrc = (j >= 0 && j == p.jsrc) ? p.ksrc : -1000;

  auto plane = [&](auto phase, int s, int bw) {
    constexpr int PH = decltype(phase)::value;
    T *const wr = xl + own_row + bw * BUF;          // written this iteration
    const T *const rd = xl + own_row + (bw ^ 1) * BUF;  // written the iteration before
    Cl[slot_of<PH, 0>()] = ncl;
    Cm[slot_of<PH, 0>()] = ncm;
    Cb[slot_of<PH, -1>()] = ncb;
#pragma unroll
    for (int f = 0; f < 3; ++f) V[0][f][slot_of<PH, 1>()] = nv0[f];
    // y neighbours of v at plane s + 1 for the next iteration
    wr[0 * SLOT] = V[0][0][slot_of<PH, 1>()];
    wr[1 * SLOT] = V[0][1][slot_of<PH, 1>()];
    wr[2 * SLOT] = V[0][2][slot_of<PH, 1>()];

    auto level = [&](auto lev) {
      constexpr int m = decltype(lev)::value;
      constexpr int D = 2 * (m - 1);
      const int pk = s - D;   // stress plane
      const int qk = pk - 1;  // velocity plane
      constexpr int mb = m >= 2 ? m - 2 : 0;
      constexpr int c0 = slot_of<PH, -D>(), cm1 = slot_of<PH, -D - 1>(),
                    cp1 = slot_of<PH, -D + 1>(), cm2 = slot_of<PH, -D - 2>();
      // LDS slots of this level's inputs: v^{m-1} at pk, sigma^m at qk
      constexpr int sv = m == 1 ? 0 : 3 + 6 * (m - 2) + 3;
      constexpr int ss = 3 + 6 * (m - 1);
      // ---------------- sigma^m at plane pk (3D:836-943)
      T sn[6];
#pragma unroll
      for (int f = 0; f < 6; ++f) sn[f] = m == 1 ? so[f] : S[mb][f][c0];
      T om[9] = {};  // old memory variables of the stress phase: x 0..2, y 3..5, z 6..8
      if (SLAB) {
#pragma unroll
        for (int f = 0; f < 3; ++f) {
          if (SX) om[f] = m == 1 ? lx[f] : MX[mb][f][c0];
          if (SY) om[3 + f] = m == 1 ? ly[f] : MY[mb][f][c0];
          if (SZ) om[6 + f] = m == 1 ? lz[f] : MZ[mb][f][c0];
        }
      }
      T nm[9];
#pragma unroll
      for (int f = 0; f < 9; ++f) nm[f] = om[f];
      {
        const T vxc = V[m - 1][0][c0], vyc = V[m - 1][1][c0], vzc = V[m - 1][2][c0];
        const T vx_yp = rd[(sv + 0) * SLOT + 64];
        const T vy_ym = rd[(sv + 1) * SLOT - 64];
        const T vz_yp = rd[(sv + 2) * SLOT + 64];
        const T dx_vx = lane_next(vxc) - vxc, dx_vy = vyc - lane_prev(vyc),
                dx_vz = vzc - lane_prev(vzc);
        const bool inz = SZ && p.sz.in(pk);
        T Zp[4] = {T(0), T(0), T(0), T(0)};
        if (SZ && inz)
          Zp[0] = p.pz.a[pk], Zp[1] = p.pz.b[pk], Zp[2] = p.pz.ah[pk], Zp[3] = p.pz.bh[pk];
        const T cl = Cl[c0], cm = Cm[c0];
        if (ylo && zlo(pk) && xhi) {
          T dvx_dx = dx_vx * p.odx;
          T dvy_dy = (vyc - vy_ym) * p.ody;
          T dvz_dz = (vzc - V[m - 1][2][cm1]) * p.odz;
          if (SX) dvx_dx = pml(inx, kx1, dvx_dx, om[0], nm[0], X[2], X[3], p.px.Kh + i);
          if (SY) dvy_dy = pml(iny, ky1, dvy_dy, om[3], nm[3], Y[0], Y[1], p.py.K + j);
          if (SZ) dvz_dz = pml(inz, kz1, dvz_dz, om[6], nm[6], Zp[0], Zp[1], p.pz.K + pk);
          const T lp2m = cl + T(2) * cm;
          sn[0] = lp2m * dvx_dx + cl * (dvy_dy + dvz_dz) + sn[0];
          sn[1] = cl * (dvx_dx + dvz_dz) + lp2m * dvy_dy + sn[1];
          sn[2] = cl * (dvx_dx + dvy_dy) + lp2m * dvz_dz + sn[2];
        }
        const bool zin = !SZ || (pk >= 0 && pk < nz);
        if (yhi && zin && xlo) {
          T dvy_dx = dx_vy * p.odx;
          T dvx_dy = (vx_yp - vxc) * p.ody;
          if (SX) dvy_dx = pml(inx, kx1, dvy_dx, om[1], nm[1], X[0], X[1], p.px.K + i);
          if (SY) dvx_dy = pml(iny, ky1, dvx_dy, om[4], nm[4], Y[2], Y[3], p.py.Kh + j);
          sn[3] = cm * (dvy_dx + dvx_dy) + sn[3];
        }
        if (row_in && zhi(pk) && xlo) {
          T dvz_dx = dx_vz * p.odx;
          T dvx_dz = (V[m - 1][0][cp1] - vxc) * p.odz;
          if (SX) dvz_dx = pml(inx, kx1, dvz_dx, om[2], nm[2], X[0], X[1], p.px.K + i);
          if (SZ) dvx_dz = pml(inz, kz1, dvx_dz, om[7], nm[7], Zp[2], Zp[3], p.pz.Kh + pk);
          sn[4] = cm * (dvz_dx + dvx_dz) + sn[4];
        }
        if (yhi && zhi(pk) && col_in) {
          T dvz_dy = (vz_yp - vzc) * p.ody;
          T dvy_dz = (V[m - 1][1][cp1] - vyc) * p.odz;
          if (SY) dvz_dy = pml(iny, ky1, dvz_dy, om[5], nm[5], Y[2], Y[3], p.py.Kh + j);
          if (SZ) dvy_dz = pml(inz, kz1, dvy_dz, om[8], nm[8], Zp[2], Zp[3], p.pz.Kh + pk);
          sn[5] = cm * (dvz_dy + dvy_dz) + sn[5];
        }
      }
#pragma unroll
      for (int f = 0; f < 6; ++f) S[m - 1][f][c0] = sn[f];
      if constexpr (SLAB && m < NT) {
#pragma unroll
        for (int f = 0; f < 3; ++f) {
          if (SX) MX[m - 1][f][c0] = nm[f];
          if (SY) MY[m - 1][f][c0] = nm[3 + f];
          if (SZ) MZ[m - 1][f][c0] = nm[6 + f];
        }
      }
      wr[(ss + 0) * SLOT] = sn[3];  // sigma_xy, sigma_yz, sigma_yy of plane pk
      wr[(ss + 1) * SLOT] = sn[5];
      wr[(ss + 2) * SLOT] = sn[1];
      if (m == NT && pk >= kb && pk < ke && own) {
        const unsigned o = pl(pk);
        st_stream_at(P.sxx + corner, o, sn[0]);
        st_stream_at(P.syy + corner, o, sn[1]);
        st_stream_at(P.szz + corner, o, sn[2]);
        st_stream_at(P.sxy + corner, o, sn[3]);
        st_stream_at(P.sxz + corner, o, sn[4]);
        st_stream_at(P.syz + corner, o, sn[5]);
        const KArgs Q = args();
        if (SX && inx)
#pragma unroll
          for (int f = 0; f < 3; ++f) st_at(Q->mx[f] + mxs * pk, mxo, nm[f]);
        if (SY && iny)
#pragma unroll
          for (int f = 0; f < 3; ++f) st_at(Q->my[f] + mys * pk, myo, nm[3 + f]);
        if (SZ && p.sz.in(pk))
#pragma unroll
          for (int f = 0; f < 3; ++f) st_at(Q->mz[f] + mzs * p.sz.s(pk), mzo, nm[6 + f]);
      }
      if (m == 1 && s < s1) {  // sigma and the coefficients of the next plane
        load_s(s + 1);
        if (SLAB) load_m(Int<0>{}, s + 1);
      }

      // ---------------- v^m at plane qk (3D:976-1121)
      T vn[3] = {V[m - 1][0][cm1], V[m - 1][1][cm1], V[m - 1][2][cm1]};
      T ov[9] = {};
      if (SLAB) {
#pragma unroll
        for (int f = 0; f < 3; ++f) {
          if (SX) ov[f] = m == 1 ? lx[3 + f] : MX[mb][3 + f][cm1];
          if (SY) ov[3 + f] = m == 1 ? ly[3 + f] : MY[mb][3 + f][cm1];
          if (SZ) ov[6 + f] = m == 1 ? lz[3 + f] : MZ[mb][3 + f][cm1];
        }
      }
      T nv[9];
#pragma unroll
      for (int f = 0; f < 9; ++f) nv[f] = ov[f];
      {
        const T(&sw)[6][3] = S[m - 1];
        const T xxc = sw[0][cm1], xyc = sw[3][cm1], xzc = sw[4][cm1], yzc = sw[5][cm1];
        const T sxy_ym = rd[(ss + 0) * SLOT - 64];
        const T syz_ym = rd[(ss + 1) * SLOT - 64];
        const T syy_yp = rd[(ss + 2) * SLOT + 64];
        const T dx_xx = xxc - lane_prev(xxc), dx_xy = lane_next(xyc) - xyc,
                dx_xz = lane_next(xzc) - xzc;
        const bool inz = SZ && p.sz.in(qk);
        T Zq[4] = {T(0), T(0), T(0), T(0)};
        if (SZ && inz)
          Zq[0] = p.pz.a[qk], Zq[1] = p.pz.b[qk], Zq[2] = p.pz.ah[qk], Zq[3] = p.pz.bh[qk];
        const T cb = Cb[cm1];
        if (ylo && zlo(qk) && xlo) {
          T dsxx_dx = dx_xx * p.odx;
          T dsxy_dy = (xyc - sxy_ym) * p.ody;
          T dsxz_dz = (xzc - sw[4][cm2]) * p.odz;
          if (SX) dsxx_dx = pml(inx, kx1, dsxx_dx, ov[0], nv[0], X[0], X[1], p.px.K + i);
          if (SY) dsxy_dy = pml(iny, ky1, dsxy_dy, ov[3], nv[3], Y[0], Y[1], p.py.K + j);
          if (SZ) dsxz_dz = pml(inz, kz1, dsxz_dz, ov[6], nv[6], Zq[0], Zq[1], p.pz.K + qk);
          vn[0] = cb * (dsxx_dx + dsxy_dy + dsxz_dz) + vn[0];
        }
        if (yhi && zlo(qk) && xhi) {
          T dsxy_dx = dx_xy * p.odx;
          T dsyy_dy = (syy_yp - sw[1][cm1]) * p.ody;
          T dsyz_dz = (yzc - sw[5][cm2]) * p.odz;
          if (SX) dsxy_dx = pml(inx, kx1, dsxy_dx, ov[1], nv[1], X[2], X[3], p.px.Kh + i);
          if (SY) dsyy_dy = pml(iny, ky1, dsyy_dy, ov[4], nv[4], Y[2], Y[3], p.py.Kh + j);
          if (SZ) dsyz_dz = pml(inz, kz1, dsyz_dz, ov[7], nv[7], Zq[0], Zq[1], p.pz.K + qk);
          vn[1] = cb * (dsxy_dx + dsyy_dy + dsyz_dz) + vn[1];
        }
        if (ylo && zhi(qk) && xhi) {
          T dsxz_dx = dx_xz * p.odx;
          T dsyz_dy = (yzc - syz_ym) * p.ody;
          T dszz_dz = (sw[2][c0] - sw[2][cm1]) * p.odz;
          if (SX) dsxz_dx = pml(inx, kx1, dsxz_dx, ov[2], nv[2], X[2], X[3], p.px.Kh + i);
          if (SY) dsyz_dy = pml(iny, ky1, dsyz_dy, ov[5], nv[5], Y[0], Y[1], p.py.K + j);
          if (SZ) dszz_dz = pml(inz, kz1, dszz_dz, ov[8], nv[8], Zq[2], Zq[3], p.pz.Kh + qk);
          vn[2] = cb * (dsxz_dx + dsyz_dy + dszz_dz) + vn[2];
        }
        // point force at step it0 + m - 1 (3D:1074-1082), rigid faces (3D:1087-1121)
        if (qk == ksrc && i == p.isrc) {
          const KArgs Q = args();
          const int it = it0 + m - 1;
          const T rsrc = Q->a.rho[i + (long)j * p.ld + (long)qk * p.ps];
          vn[0] = vn[0] + Q->a.fx[it - 1] * p.dt / rsrc;
          vn[1] = vn[1] + Q->a.fy[it - 1] * p.dt / rsrc;
        }
        if ((SX && (i == 0 || i == nx - 1)) || (SY && (j == 0 || j == ny - 1)) ||
            (SZ && (qk == 0 || qk == nz - 1)))
          vn[0] = vn[1] = vn[2] = T(0);
      }
      // receivers of step it0 + m - 1 on plane qk (owned points only)
      if (qk == rk[m - 1] && qk < ke) {
        const KArgs Q = args();
        int c = cur[m - 1], nk = qk;
        while (nk == qk) {
          if (Q->rec_i[c] == i && Q->rec_j[c] == j && own) {
            const long o = (long)(it0 + m - 2) * Q->nrec + Q->rec_slot[c];
            Q->sisx[o] = vn[0];
            Q->sisy[o] = vn[1];
            if (Q->sisz) Q->sisz[o] = vn[2];
          }
          ++c;
          nk = c < rc1 ? __builtin_amdgcn_readfirstlane(Q->rec_k[c]) : kNever;
        }
        cur[m - 1] = c;
        rk[m - 1] = nk;
      }
      if constexpr (m < NT) {
#pragma unroll
        for (int f = 0; f < 3; ++f) V[m][f][cm1] = vn[f];
        if (SLAB) {
#pragma unroll
          for (int f = 0; f < 3; ++f) {
            if (SX) MX[m - 1][3 + f][cm1] = nv[f];
            if (SY) MY[m - 1][3 + f][cm1] = nv[3 + f];
            if (SZ) MZ[m - 1][3 + f][cm1] = nv[6 + f];
          }
        }
        wr[(ss + 3) * SLOT] = vn[0];  // y neighbours of v^m at plane qk
        wr[(ss + 4) * SLOT] = vn[1];
        wr[(ss + 5) * SLOT] = vn[2];
      } else if (qk >= kb && qk < ke && own) {
        const unsigned o = pl(qk);
        st_stream_at(P.vx + corner, o, vn[0]);
        st_stream_at(P.vy + corner, o, vn[1]);
        st_stream_at(P.vz + corner, o, vn[2]);
        const KArgs Q = args();
        if (SX && inx)
#pragma unroll
          for (int f = 0; f < 3; ++f) st_at(Q->mx[3 + f] + mxs * qk, mxo, nv[f]);
        if (SY && iny)
#pragma unroll
          for (int f = 0; f < 3; ++f) st_at(Q->my[3 + f] + mys * qk, myo, nv[3 + f]);
        if (SZ && p.sz.in(qk))
#pragma unroll
          for (int f = 0; f < 3; ++f) st_at(Q->mz[3 + f] + mzs * p.sz.s(qk), mzo, nv[6 + f]);
      }
      if (m == 1 && s < s1) {  // v of the plane after the next, buoyancy of this one
        load_v(s + 2);
        if (SLAB) load_m(Int<3>{}, s);
      }
    };
    level(Int<1>{});
    if constexpr (NT > 1) level(Int<2>{});
    __syncthreads();
  };
  for (int s = s0, bw = 0;; s += 3, bw ^= 1) {
    plane(Int<0>{}, s, bw);
    if (s == s1) break;
    plane(Int<1>{}, s + 1, bw ^ 1);
    if (s + 1 == s1) break;
    plane(Int<2>{}, s + 2, bw);
    if (s + 2 == s1) break;
  }
}

// Every tile of the grid in one launch, class by class: all axes' slabs first
// (the most code), the slab-free tiles last; P.ncls[c] tiles of class c (bit 0
// x, bit 1 y, bit 2 z).  Each XCD gets one contiguous band of every class.  One
// launch, because a workgroup fills a CU whatever its class (LDS), and launches
// of single classes leave the machine idle at their ends: seven small ones in
// a row cost more than the step itself on small grids.
template <typename T, int NT, int NW>
__global__ __launch_bounds__(64 * NW) void k_tb3d(TB3D<T> P) {
  // one row of padding at both ends: the row below row 0 of slot 0 and above
  // the last row of the last slot are read (by ring rows only)
  __shared__ T xl[2 * 6 * NT * NW * 64 + 128];
  const int xcd = blockIdx.x & 7;
  int u = blockIdx.x >> 3;
#pragma unroll 1
  for (int c = 7; c >= 0; --c) {
    const int q = P.ncls[c] >> 3, r = P.ncls[c] & 7, n = q + (xcd < r ? 1 : 0);
    if (u >= n) {
      u -= n;
      continue;
    }
    const int t = xcd * q + min(xcd, r) + u;
    switch (c) {
      case 7: tb3d_tile<T, NT, NW, true, true, true>(P, t, xl); break;
      case 6: tb3d_tile<T, NT, NW, false, true, true>(P, t, xl); break;
      case 5: tb3d_tile<T, NT, NW, true, false, true>(P, t, xl); break;
      case 4: tb3d_tile<T, NT, NW, false, false, true>(P, t, xl); break;
      case 3: tb3d_tile<T, NT, NW, true, true, false>(P, t, xl); break;
      case 2: tb3d_tile<T, NT, NW, false, true, false>(P, t, xl); break;
      case 1: tb3d_tile<T, NT, NW, true, false, false>(P, t, xl); break;
      default: tb3d_tile<T, NT, NW, false, false, false>(P, t, xl);
    }
    return;
  }
}

template <typename T, int NT, int NW>
hipError_t tb3d_launch(const TB3D<T> &P0, hipStream_t s) {
  TB3D<T> P = P0;
  if (P.ow < 1 || P.ow > 64 - 2 * NT) return hipErrorInvalidValue;
  const long most = tb3d_split(NT, NW, P);
  hipLaunchKernelGGL((k_tb3d<T, NT, NW>), dim3((unsigned)(8 * most)), dim3(64 * NW), 0, s, P);
  return hipGetLastError();
}

}  // namespace

int tb3d_max_nt(int) { return 2; }

// rows per workgroup: 16 wavefronts in float, 8 in double (LDS: 6 NT values
// per point and buffer)
template <typename T>
hipError_t launch_tb3d(int nt, const TB3D<T> &p, hipStream_t s) {
  constexpr int NW = sizeof(T) == 4 ? 16 : 8;
  if (nt == 1) return tb3d_launch<T, 1, NW>(p, s);
  if (nt == 2) return tb3d_launch<T, 2, NW>(p, s);
  return hipErrorInvalidValue;
}

template hipError_t launch_tb3d<float>(int, const TB3D<float> &, hipStream_t);
template hipError_t launch_tb3d<double>(int, const TB3D<double> &, hipStream_t);

}  // namespace cpml
