// Triangular sweeps of one 8x8x8 tile by one wave64, in registers.
//
// Lane l owns the column (li, lj) = (l & 7, l >> 3) of the tile, eight points
// along k.  A forward step needs the results of (i-1), (j-1) and (k-1): with
// lane l starting its column s(l) = li + (lj & 1) + 3 (lj >> 1) steps late,
//   (k-1)            is the lane's own previous result,
//   (i-1)            is lane l-1's previous result (a DPP row shift),
//   (j-1), lj odd    is lane l-8's previous result (a DPP row shift by 8: the
//                    two columns j = 2r, 2r+1 share a 16-lane DPP row),
//   (j-1), lj even   crosses a DPP row: the result of two steps ago, passed
//                    through 64 LDS words, its read issued a step ahead.
// So no step waits for LDS: 25 steps of about 15 VALU instructions, against
// 22 steps that each wait for an LDS write, three dependent LDS reads and the
// per-point data when the hyperplanes i+j+k = h are swept out of an LDS box
// (measured there: about 450 cycles a step, here about 80).  The backward sweep
// is the same with every direction reversed; its step g handles register (-g) & 7.
//
// Registers are skewed so that a step's index is a constant: register u of a
// lane holds the column's point k = (u - s) & 7, and step h (k = h - s) uses
// register h & 7 in every lane.  Lanes whose step lies outside 0 <= h - s < 8
// compute on some other point of their column and keep nothing: their results
// only meet couplings that point out of the tile, which the caller has set to
// zero (it folds the neighbouring tiles' values into the right-hand side).  Zero
// times a NaN or an infinity is a NaN, so a tile that holds one ends as NaN
// whole and hands it to every neighbour.  Selects in place of the zeros would
// keep it to the points that depend on it: measured at 2.5 % of a two-system
// mixed solve (40x40x30+10), 7 % of an FP64 drop-in one, for a system that ends
// as a breakdown either way.
#pragma once

#include "mt_device.hpp"

namespace mt {

constexpr int kSwSteps = 25;

__device__ __forceinline__ int sw_skew(int lane) {
  const int lj = lane >> 3;
  return (lane & 7) + (lj & 1) + 3 * (lj >> 1);
}
// tile point of register u of a lane (k = (u - skew) & 7)
__device__ __forceinline__ int sw_point(int lane, int skew, int u) {
  return lane + 64 * ((u - skew) & 7);
}

// v moved across lanes by DPP control CTRL in the banks of BANK; `old` in the
// others (and, without BC, where the source lane is past the row's end)
template <int CTRL, int BANK, bool BC>
__device__ __forceinline__ float sw_dpp(float old, float v) {
  return __int_as_float(
      __builtin_amdgcn_update_dpp(__float_as_int(old), __float_as_int(v), CTRL, 0xf, BANK, BC));
}
template <int CTRL, int BANK, bool BC>
__device__ __forceinline__ double sw_dpp(double old, double v) {
  const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), CTRL, 0xf, BANK, BC);
  const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), CTRL, 0xf, BANK, BC);
  return __hiloint2double(hi, lo);
}
template <int CTRL, int BANK, bool BC, class T>
__device__ __forceinline__ C2<T> sw_dpp2(C2<T> old, C2<T> v) {
  return {sw_dpp<CTRL, BANK, BC>(old.x, v.x), sw_dpp<CTRL, BANK, BC>(old.y, v.y)};
}

// The wave's cross-row words: 64 entries, lane l's latest result.  A wave's
// LDS instructions execute in order, so the read after the write of the same
// step sees it; only the compiler must keep them so.
__device__ __forceinline__ void sw_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// step(u, i-, j-, k-neighbour, active) returns the value passed on.  UP: the
// backward direction (i+1, j+1, k+1).
template <bool UP, class T, class F>
__device__ __forceinline__ void sw_run(int lane, int skew, C2<T>* __restrict__ X, F&& step) {
  // UP: a lane's delay is 17 - skew (7+1+9 in all)
  const int s = UP ? 17 - skew : skew;
  const int xo = UP ? (lane < 48 ? lane + 8 : lane) : (lane >= 16 ? lane - 8 : lane);
  constexpr int C1 = UP ? 0x101 : 0x111;   // row_shl:1 / row_shr:1
  constexpr int C8 = UP ? 0x108 : 0x118;   // row_shl:8 / row_shr:8
  constexpr int B8 = UP ? 0x3 : 0xc;       // lanes 0-7 (j even) / 8-15 (j odd) of a row
  const C2<T> zero = {T(0), T(0)};
  C2<T> wp = zero, jn0 = zero, jn1 = zero;
#pragma unroll
  for (int h = 0; h < kSwSteps; ++h) {
    const int u = UP ? (-h) & 7 : h & 7;
    const C2<T> iv = sw_dpp2<C1, 0xf, true>(zero, wp);
    const C2<T> jv = sw_dpp2<C8, B8, false>(jn0, wp);
    const C2<T> w = step(u, iv, jv, wp, unsigned(h - s) < 8u);
    wp = w;
    jn0 = jn1;
    if (h + 2 < kSwSteps) {
      X[lane] = w;
      sw_order();
      jn1 = X[xo];
      sw_order();
    }
  }
}

}  // namespace mt
