// End of a time step: receivers, the step's energy from its partial sums, and
// the step counter.  One block's work; in the two-phase loop a block in front
// of the next step's stress launch does it (that launch changes neither the
// velocities nor the partial sums), so it costs no launch of its own: 101 x
// 641 double with the energy curve 16.6 us per step with the pass over the
// energy, its sum and the receivers in launches of their own, 10.6 now; 96 x 80 x 72
// float 41 and 30.
#pragma once

#include "cpml_device.h"
#include "cpml_internal.h"

namespace cpml {

// Blocks in front of a launch's tiles: one that works, and a count that keeps
// tile t on XCD t % 8.
constexpr int kLead = 8;

// Sums of a and b over the first 256 threads of the block (all call it), in
// every one of them.
__device__ __forceinline__ void block_sum2(int tid, double &a, double &b) {
  __shared__ double sa[256], sb[256];
  if (tid < 256) {
    sa[tid] = a;
    sb[tid] = b;
  }
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (tid < s) {
      sa[tid] += sa[tid + s];
      sb[tid] += sb[tid + s];
    }
    __syncthreads();
  }
  a = sa[0];
  b = sb[0];
}

// Sums of the partial pairs g, g + kEnergyGroups, ...
__device__ __forceinline__ void group_sum(const double *partial, int nparts, int g, double &kin,
                                          double &pot) {
  kin = pot = 0.0;
#pragma unroll 8
  for (int b = g; b < nparts; b += kEnergyGroups) {
    kin += partial[2 * b];
    pot += partial[2 * b + 1];
  }
}

// The kinetic and potential energy of step it from nparts partial sums, by the
// first 256 threads of a block, group by group (so that the sums of the groups can
// be formed by a launch of their own before).
template <typename E>
__device__ __forceinline__ void energy_final(const E &e, int tid, int it, int nparts, bool half) {
  double kin = 0.0, pot = 0.0;
  if (tid < 256)
    for (int g = tid; g < min(nparts, kEnergyGroups); g += 256) {
      double a, b;
      group_sum(e.partial, nparts, g, a, b);
      kin += a;
      pot += b;
    }
  block_sum2(tid, kin, pot);
  if (tid == 0) {
    e.out_kin[it - 1] = half ? 0.5 * kin : kin;
    e.out_pot[it - 1] = pot;
  }
}

template <typename T>
__device__ __forceinline__ void record_step(const Record<T> &p) {
  const int tid = threadIdx.x + threadIdx.y * blockDim.x, n = blockDim.x * blockDim.y;
  const int it = *p.step + p.skip;
  const long row = (long)(it - 1) * p.nrec;
  for (int r = tid; r < p.nrec; r += n) {
    const long q = p.idx[r];
    p.sx[row + r] = p.avg4 ? (p.vx[q] + p.vx[q + 1] + p.vx[q + p.ld] + p.vx[q + 1 + p.ld]) / T(4)
                           : p.vx[q];
    p.sy[row + r] = p.vy[q];
    if (p.sz) p.sz[row + r] = p.vz[q];
  }
  if (p.cadence > 0 && it % p.cadence == 0) energy_final(p, tid, it, p.nparts, !p.sz);
  __syncthreads();
  if (tid == 0) *p.step = it + 1;
}

// First blocks of a stress launch: true where this block is one of them (and
// done).  h: this block's tile number.
template <typename T>
__device__ __forceinline__ bool lead_block(const Record<T> &prev, int lead, int &h) {
  h = (int)blockIdx.x - lead;
  if (h >= 0) return false;
  if (blockIdx.x == 0) record_step(prev);
  return true;
}

}  // namespace cpml
