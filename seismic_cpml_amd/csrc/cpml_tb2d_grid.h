// Kernels and launcher of the time-blocked 2D step on one grid (cpml_tb2d.h),
// for the translation units that instantiate them in one precision each.
#pragma once

#include "cpml_tb2d.h"

namespace cpml {
namespace {

// One grid: an item (tb2d_item_at) per wavefront.
template <typename T, int ORDER, int NT, bool EN>
__global__ __launch_bounds__(64 * WPB, (min_waves<T, ORDER, NT>())) void k_tb2d(TB2D<T> P) {
  __shared__ T delay[WPB][tb2d_delay_words<ORDER, NT, 3>() * 64 + 1];
  const int wv = threadIdx.x >> 6;
  const Tb2dItems n = tb2d_items(P);
  const int item = __builtin_amdgcn_readfirstlane(
      xcd_item(blockIdx.x & 7, (blockIdx.x >> 3) * WPB + wv, n.edge + n.cap, n.clean));
  if (item < 0) return;
  const Tb2dItem it = tb2d_item_at(P, n, item);
  tb2d_any<T, ORDER, NT, EN>(kernarg<TB2D<T>>(), it.cls, it.ts, it.jb, it.je, delay[wv], P.ahead,
                           item);
}

// Energy of the levels of some launches: level b = blockIdx.x, step
// *e.step + b; the items' sums added in slot order, then as a tree.
constexpr int EBT = 256;
template <typename T>
__global__ __launch_bounds__(EBT) void k_tb2d_energy(Energy<T> e, const double *epart,
                                                     int eslots) {
  const int it = *e.step + (int)blockIdx.x;
  if (it % e.cadence != 0) return;
  const double *pp = epart + (long)blockIdx.x * eslots * 2;
  double kin = 0.0, pot = 0.0;
  for (int k = threadIdx.x; k < eslots; k += EBT) {
    kin += pp[2 * k];
    pot += pp[2 * k + 1];
  }
  __shared__ double sk[EBT], sp[EBT];
  sk[threadIdx.x] = kin;
  sp[threadIdx.x] = pot;
  __syncthreads();
  for (int h = EBT / 2; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) {
      sk[threadIdx.x] += sk[threadIdx.x + h];
      sp[threadIdx.x] += sp[threadIdx.x + h];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    e.out_kin[it - 1] = 0.5 * sk[0];  // 2D2:711: kinetic summed, then halved
    e.out_pot[it - 1] = sp[0];
  }
}

template <typename T, int ORDER, int NT>
hipError_t tb2d_launch(const TB2D<T> &P0, hipStream_t s) {
  constexpr int G = NT * (ORDER - 1);
  TB2D<T> P = P0;
  if (P.ow < 1 || P.ow > 64 - 2 * G) return hipErrorInvalidValue;
  tb2d_split(ORDER, NT, P);
  const Tb2dItems n = tb2d_items(P);
  const dim3 g(8 * ((xcd_items(n.edge + n.cap, n.clean) + WPB - 1) / WPB)), b(64 * WPB);
  if (P.epart) hipLaunchKernelGGL((k_tb2d<T, ORDER, NT, true>), g, b, 0, s, P);
  else hipLaunchKernelGGL((k_tb2d<T, ORDER, NT, false>), g, b, 0, s, P);
  return hipGetLastError();
}

}  // namespace

template <typename T>
hipError_t launch_tb2d(int order, int nt, const TB2D<T> &p, hipStream_t s) {
  if (nt < 1 || nt > tb2d_max_nt(order, sizeof(T))) return hipErrorInvalidValue;
  switch (order * 10 + nt) {
    case 21: return tb2d_launch<T, 2, 1>(p, s);
    case 22: return tb2d_launch<T, 2, 2>(p, s);
    case 41: return tb2d_launch<T, 4, 1>(p, s);
    case 42: return tb2d_launch<T, 4, 2>(p, s);
    case 81: return tb2d_launch<T, 8, 1>(p, s);
    case 82: return tb2d_launch<T, 8, 2>(p, s);
    default: break;
  }
  if constexpr (sizeof(T) == 4) {
    switch (order * 10 + nt) {
      case 23: return tb2d_launch<T, 2, 3>(p, s);
      case 24: return tb2d_launch<T, 2, 4>(p, s);
      case 43: return tb2d_launch<T, 4, 3>(p, s);
      default: break;
    }
  }
  return hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_tb2d_energy(const Energy<T> &e, const double *epart, int eslots, int nlevels,
                              hipStream_t s) {
  hipLaunchKernelGGL(k_tb2d_energy<T>, dim3(nlevels), dim3(EBT), 0, s, e, epart, eslots);
  return hipGetLastError();
}
}  // namespace cpml
