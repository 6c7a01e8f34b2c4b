// Kernels and launcher of the time-blocked 2D step on many grids (cpml_tb2d.h),
// for the translation units that instantiate them in one precision each.
#pragma once

#include "cpml_tb2d.h"

namespace cpml {
namespace {

// Many grids in one launch: items[k] = (grid, strip, first row, end row), the
// n3 of class 3 (both slabs) first, then n1 of class 1, n2 of class 2 and n0
// slab-free ones.  The wavefronts of the blocks an XCD receives stride through
// its share (one item each when the grid has one wavefront per item, several
// when it is a persistent grid).
template <typename T, int ORDER, int NT>
__global__ __launch_bounds__(64 * WPB, (min_waves<T, ORDER, NT>())) void k_tb2d_multi(
    const TB2D<T> *__restrict__ grids, const int4 *__restrict__ items, int n3, int n1, int n2,
    int n0, int ahead) {
  __shared__ T delay[WPB][tb2d_delay_words<ORDER, NT, 3>() * 64 + 1];
  const int G = gridDim.x, h = blockIdx.x;
  const int xcd = h & 7;
  const int nb = (G - xcd + 7) >> 3;  // blocks this XCD receives
  const int wv = threadIdx.x >> 6;
  for (int u = (h >> 3) * WPB + wv;; u += nb * WPB) {
    const int k = __builtin_amdgcn_readfirstlane(xcd_item(xcd, u, n3 + n1 + n2, n0));
    if (k < 0) return;
    const int4 e = items[k];
    const int cls = k < n3 ? 3 : k < n3 + n1 ? 1 : k < n3 + n1 + n2 ? 2 : 0;
    tb2d_any<T, ORDER, NT, false>((GridPtr<T>)(grids + __builtin_amdgcn_readfirstlane(e.x)), cls,
                                  __builtin_amdgcn_readfirstlane(e.y),
                                  __builtin_amdgcn_readfirstlane(e.z),
                                  __builtin_amdgcn_readfirstlane(e.w), delay[wv], ahead, 0);
  }
}

template <typename T, int ORDER, int NT>
hipError_t tb2d_multi(const TB2D<T> *grids, const int4 *items, const int (&n)[4], int waves,
                      int ahead, hipStream_t s) {
  // whole rounds of the 8 XCDs: each has its own share of the items
  const int blocks = std::min((xcd_items(n[1] + n[2] + n[3], n[0]) + WPB - 1) / WPB,
                              (waves + 8 * WPB - 1) / (8 * WPB));
  hipLaunchKernelGGL((k_tb2d_multi<T, ORDER, NT>), dim3(8 * std::max(blocks, 1)), dim3(64 * WPB), 0,
                     s, grids, items, n[3], n[1], n[2], n[0], ahead);
  return hipGetLastError();
}

}  // namespace

template <typename T>
hipError_t launch_tb2d_multi(int order, int nt, const TB2D<T> *grids, const int4 *items,
                             const int (&n)[4], int waves, int ahead, hipStream_t s) {
  if (nt < 1 || nt > tb2d_max_nt(order, sizeof(T)) || waves < 1) return hipErrorInvalidValue;
  switch (order * 10 + nt) {
    case 21: return tb2d_multi<T, 2, 1>(grids, items, n, waves, ahead, s);
    case 22: return tb2d_multi<T, 2, 2>(grids, items, n, waves, ahead, s);
    case 41: return tb2d_multi<T, 4, 1>(grids, items, n, waves, ahead, s);
    case 42: return tb2d_multi<T, 4, 2>(grids, items, n, waves, ahead, s);
    case 81: return tb2d_multi<T, 8, 1>(grids, items, n, waves, ahead, s);
    case 82: return tb2d_multi<T, 8, 2>(grids, items, n, waves, ahead, s);
    default: break;
  }
  if constexpr (sizeof(T) == 4) {
    switch (order * 10 + nt) {
      case 23: return tb2d_multi<T, 2, 3>(grids, items, n, waves, ahead, s);
      case 24: return tb2d_multi<T, 2, 4>(grids, items, n, waves, ahead, s);
      case 43: return tb2d_multi<T, 4, 3>(grids, items, n, waves, ahead, s);
      default: break;
    }
  }
  return hipErrorInvalidValue;
}

}  // namespace cpml
