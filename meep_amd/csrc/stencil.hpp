// stencil.hpp — device helpers shared by the forward (kernels.hip) and reverse (adjoint.hip)
// step kernels, and the source terms of the forward ones.
#pragma once

#include "engine.hpp"

#include <hip/hip_runtime.h>

namespace mx {

constexpr int BLOCK = 256;

// logical block index, dealt to XCDs in contiguous runs (gridDim.x is a multiple of 8);
// rev walks them in descending order
__device__ __forceinline__ uint32_t xcd_block(int rev = 0) {
  const uint32_t nb = gridDim.x, b = blockIdx.x;
  const uint32_t lb = (b & 7u) * (nb >> 3) + (b >> 3);
  return rev ? nb - 1 - lb : lb;
}

// halo point along a folded axis fed by the owned point z of a component with Yee shift ysh
// there; -1 when z is not the wrapped end
__device__ __forceinline__ int zwrap_dst(int ysh, int z, int n) {
  if (ysh == 0) return z == n ? 0 : -1;
  return z == 0 ? n : -1;
}

// coordinate along loop axis k (a select over registers, never an indexed access)
__device__ __forceinline__ int asel(int j0, int j1, int j2, int k) { return k == 0 ? j0 : (k == 1 ? j1 : j2); }

__device__ __forceinline__ bool slot_owned(const AxisSlot &s, int j0, int j1, int j2) {
  return j0 >= s.lo[0] && j0 <= s.hi[0] && j1 >= s.lo[1] && j1 <= s.hi[1] && j2 >= s.lo[2] && j2 <= s.hi[2];
}
// on_metal_boundary for an owned point (src/boundaries.cpp:191-205)
__device__ __forceinline__ bool slot_metal(const AxisSlot &s, int j0, int j1, int j2) {
  return j0 == s.mhi[0] || j0 == s.mlo[0] || j1 == s.mhi[1] || j1 == s.mlo[1] || j2 == s.mhi[2] || j2 == s.mlo[2];
}

template <class R> __device__ __forceinline__ bool pml_on(const R *sig, const R *kap, int k) {
  return sig && (sig[k] != R(0) || kap[k] != R(1));
}

// ---- sources ----
// vrow: the step's row of source values
template <class R> __device__ __forceinline__ R apply_tab(const SrcTab &t, int c, uint32_t i, R v, const double *vrow) {
#pragma unroll
  for (int s = 0; s < SRC_TAB; ++s)
    if (s < t.n && t.comp[s] == c && t.idx[s] == int64_t(i)) v = R(double(v) - vrow[t.vbase + s]);
  return v;
}

// value of box source S at loop-axis indices (j0, j1, j2); contraction is off so the complex
// product rounds as the host's does
template <int S> __device__ __forceinline__ double box_value(const SrcBoxes &b, int cmp, int j0, int j1, int j2, const double *vrow) {
#pragma clang fp contract(off)
  const int64_t k = int64_t(j0 - b.lo[S][0]) * b.bst[S][0] + int64_t(j1 - b.lo[S][1]) * b.bst[S][1] +
                    int64_t(j2 - b.lo[S][2]) * b.bst[S][2];
  const double2 am = b.amp[S][k];
  const double sx = vrow[b.vbase + 2 * S], sy = vrow[b.vbase + 2 * S + 1];
  const double re = am.x * sx - am.y * sy, im = am.x * sy + am.y * sx;
  return cmp ? im * b.mult[S] : re * b.mult[S];
}
template <int S> __device__ __forceinline__ bool in_box(const SrcBoxes &b, int c, int j0, int j1, int j2) {
  return S < b.n && b.comp[S] == c && j0 >= b.lo[S][0] && j0 <= b.hi[S][0] && j1 >= b.lo[S][1] && j1 <= b.hi[S][1] &&
         j2 >= b.lo[S][2] && j2 <= b.hi[S][2];
}
template <class R>
__device__ __forceinline__ R apply_boxes(const SrcBoxes &b, int cmp, int c, int j0, int j1, int j2, R v, const double *vrow) {
  static_assert(SRC_BOX == 2, "one term per box");
  if (in_box<0>(b, c, j0, j1, j2)) v = R(double(v) - box_value<0>(b, cmp, j0, j1, j2, vrow));
  if (in_box<1>(b, c, j0, j1, j2)) v = R(double(v) - box_value<1>(b, cmp, j0, j1, j2, vrow));
  return v;
}
static inline unsigned nblocks(size_t n) { return unsigned((n + BLOCK - 1) / BLOCK); }
static inline unsigned nblocks8(size_t n) { return (nblocks(n) + 7u) / 8u * 8u; }

} // namespace mx
