// Device helpers shared by the kernel translation units of libcpml_gpu.
#pragma once

#include <hip/hip_runtime.h>

namespace cpml {

constexpr int BX = 64;  // points per wavefront row along x

// Position of a tile's z chunk in its XCD band -> z chunk.  When the chunks
// divide into 8 equal groups, band b holds the chunks c with c % 8 == b, so
// every XCD gets the same share of the (slower) absorbing z-slab planes
// instead of the first and last bands holding all of them.
__device__ __forceinline__ int zchunk_of(int band_pos, int ntz) {
  if (ntz & 7) return band_pos;
  const int m = ntz >> 3;
  return band_pos / m + 8 * (band_pos % m);
}

// Tile of the two-phase 3D kernels: 64 columns by TY rows (one wavefront per
// row) marching the z planes [kb, ke).
struct Tile3 {
  int i, j, kb, ke;
  bool ok;
};

// FLAT numbers the columns through the TY-row groups of a plane, one group after
// the other, and cuts them into wavefronts of 64, so that only a plane's last
// tile has idle lanes; otherwise each group of rows is cut by itself, so that
// every wavefront but a row's last stores whole cache lines.  Double, order 4: FLAT
// 3103 us per step at 210 x 800 x 220, by rows 3494; 65 x 300 x 300 578 and 862,
// 250 x 300 x 280 1680 and 1713, 700 x 500 x 100 2953 and 2912, alike where the
// columns are whole wavefronts.  Elsewhere the whole lines count for more: float,
// order 4, 210 x 800 x 220 1592 and 1531, 250 x 300 x 280 854 and 768; double, order 2,
// 101 columns 3068 and 2827.
template <bool FLAT>
inline __host__ __device__ int plane_tiles3(int nx, int ny, int ty) {
  const int groups = (ny + ty - 1) / ty;
  return FLAT ? (int)(((long)nx * groups + BX - 1) / BX) : (nx + BX - 1) / BX * groups;
}
// Tile number h of the launch.  Workgroups are dispatched round-robin over the
// 8 XCDs; each XCD gets one contiguous band of tiles (x fastest, then y, then z
// chunk) so the tiles that read each other's halo rows share its L2; the z chunks
// are interleaved over the bands (zchunk_of).
template <int TY, bool FLAT, typename P>
__device__ __forceinline__ Tile3 tile3(const P &p, int h) {
  const int nxy = plane_tiles3<FLAT>(p.nx, p.ny, TY);
  const int ntz = (p.nz + p.kchunk - 1) / p.kchunk;
  const int nt = nxy * ntz;
  const int xcd = h & 7, loc = h >> 3;
  const int q = nt >> 3, r = nt & 7;
  const int t = xcd * q + min(xcd, r) + loc, txy = t % nxy;
  Tile3 o;
  int group;
  if (FLAT) {
    const int col = txy * BX + threadIdx.x;
    group = col / p.nx;
    o.i = col - group * p.nx;
  } else {
    const int ntx = (p.nx + BX - 1) / BX;
    group = txy / ntx;
    o.i = (txy - group * ntx) * BX + threadIdx.x;
  }
  o.j = group * TY + threadIdx.y;
  o.kb = zchunk_of(t / nxy, ntz) * p.kchunk;
  o.ke = min(o.kb + p.kchunk, p.nz);
  o.ok = o.i < p.nx && o.j < p.ny;
  return o;
}

// d / K.  The reference profiles use K_MAX_PML = 1 (2D2:215), so K is 1 at
// every point and x / 1 == x exactly in IEEE arithmetic: the correctly
// rounded division (a dozen instructions) is only executed where K != 1.
template <typename T>
__device__ __forceinline__ T over_k(T d, T K) {
  return K == T(1) ? d : d / K;
}

// C-PML correction of a derivative: psi <- b*psi + a*d ; d <- d/K + psi
// (e.g. seismic_CPML_2D_isotropic_second_order.f90:567-571).
template <typename T>
__device__ __forceinline__ T cpml(T d, T *psi, T a, T b, T K) {
  const T m = b * *psi + a * d;
  *psi = m;
  return over_k(d, K) + m;
}

// Same recursion with the old value read from one array and the new one
// written to another (or not written when psi_new is null).
template <typename T>
__device__ __forceinline__ T cpml2(T d, const T *psi_old, T *psi_new, T a, T b, T K) {
  const T m = b * *psi_old + a * d;
  if (psi_new) *psi_new = m;
  return over_k(d, K) + m;
}

// The kernel's first argument, read through the kernel-argument segment with a
// pointer the compiler cannot prove loop-invariant.  Kernels whose argument
// block holds more pointers than fit in scalar registers re-read the ones
// they need inside their z loop (scalar loads, cached) instead of keeping
// them live across it (which spills scalar registers into vector lanes).
template <typename A>
__device__ __forceinline__ const __attribute__((address_space(4))) A *kernarg() {
  auto q = (const __attribute__((address_space(4))) A *)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(q));
  return q;
}

// x of the next / previous lane of the wavefront (0 past the ends): DPP wave
// shifts by one lane, which the compiler folds into the instruction that uses
// the value.
template <int CTRL>
__device__ __forceinline__ int dpp_shift(int x) {
  return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ float dpp_shift(float x) {
  return __builtin_bit_cast(float, dpp_shift<CTRL>(__builtin_bit_cast(int, x)));
}
template <int CTRL>
__device__ __forceinline__ double dpp_shift(double x) {
  typedef int i32x2 __attribute__((ext_vector_type(2)));
  i32x2 v = __builtin_bit_cast(i32x2, x);
  v.x = dpp_shift<CTRL>(v.x);
  v.y = dpp_shift<CTRL>(v.y);
  return __builtin_bit_cast(double, v);
}
template <typename T>
__device__ __forceinline__ T lane_next(T x) {
  return dpp_shift<0x130>(x);  // wave_shl:1
}
template <typename T>
__device__ __forceinline__ T lane_prev(T x) {
  return dpp_shift<0x138>(x);  // wave_shr:1
}

// First index in [lo, hi) whose (ascending) value is not below v; hi if none.
__device__ __forceinline__ int first_from(const int *a, int lo, int hi, int v) {
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (a[mid] < v) lo = mid + 1;
    else hi = mid;
  }
  return __builtin_amdgcn_readfirstlane(lo);
}

// psi <- b*psi + a*d ; d <- d/K + psi in an absorbing slab, with the old psi
// given and the new one returned through `out`.  k1: K is 1 all along the axis,
// so d / K == d; K: where to read it otherwise.
template <typename T>
__device__ __forceinline__ T pml(bool slab, bool k1, T d, T old, T &out, T a, T b, const T *K) {
  out = old;
  if (!slab) return d;
  out = b * old + a * d;
  if (!k1) d = over_k(d, *K);
  return d + out;
}

// Loads and stores through a scalar base and a 32-bit byte offset of the lane
// (explicitly global memory: the batch reads the bases from a table, where the
// compiler would otherwise emit flat accesses).
template <typename T>
using Glb = __attribute__((address_space(1))) T;
template <typename T>
__device__ __forceinline__ T ld_at(const T *base, unsigned byte_off) {
  return *reinterpret_cast<const Glb<T> *>(
      reinterpret_cast<const Glb<char> *>((const Glb<T> *)base) + byte_off);
}
template <typename T>
__device__ __forceinline__ void st_at(T *base, unsigned byte_off, T x) {
  *reinterpret_cast<Glb<T> *>(reinterpret_cast<Glb<char> *>((Glb<T> *)base) + byte_off) = x;
}

// The same store streamed past the caches: state that the next launch reads a
// whole grid later.  (Memory variables, whose rows are shorter than a cache line, merge
// in the L2 and take st_at.)
template <typename T>
__device__ __forceinline__ void st_stream_at(T *base, unsigned byte_off, T x) {
  __builtin_nontemporal_store(
      x, reinterpret_cast<Glb<T> *>(reinterpret_cast<Glb<char> *>((Glb<T> *)base) + byte_off));
}

// A number as a type, for phases and levels that the compiler has to know.
template <int V>
struct Int {
  static constexpr int value = V;
};

// Raw buffer resource over `bytes` bytes at p (gfx9 family word 3).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void *p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes,
                                           0x00020000);
}

template <typename T>
struct BufOp;

// Cache policy of accesses whose data no other thread touches (a point's own
// old stress, coefficients, results): when the state is much larger than the
// caches, the non-temporal hint (bit 1 of the policy operand on gfx950)
// streams them past the L2, which keeps its capacity for the halo rows and
// planes that neighbouring tiles re-read.  Grids whose state stays resident
// in the caches from one step to the next keep plain accesses (NT = false).
constexpr int kNonTemporal = 2;

template <bool NT, typename T>
__device__ __forceinline__ T ld_once(const T *p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}
template <bool NT, typename T>
__device__ __forceinline__ void st_once(T *p, T x) {
  if constexpr (NT) __builtin_nontemporal_store(x, p);
  else *p = x;
}

template <>
struct BufOp<float> {
  __device__ static float ld(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, v, s, 0));
  }
  __device__ static void st(float x, __amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), r, v, s, 0);
  }
  template <int POL>
  __device__ static float ldp(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, v, s, POL));
  }
  template <int POL>
  __device__ static void stp(float x, __amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, x), r, v, s, POL);
  }
};

template <>
struct BufOp<double> {
  typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
  __device__ static double ld(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, v, s, 0));
  }
  __device__ static void st(double x, __amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), r, v, s, 0);
  }
  template <int POL>
  __device__ static double ldp(__amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, v, s, POL));
  }
  template <int POL>
  __device__ static void stp(double x, __amdgpu_buffer_rsrc_t r, unsigned v, unsigned s) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, x), r, v, s, POL);
  }
};

}  // namespace cpml
