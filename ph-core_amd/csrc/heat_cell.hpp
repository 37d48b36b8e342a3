// Device helpers shared by the heat kernels (heat.hip, heat_tile.hip): the
// cell update and the lane shifts that hand a lane its neighbours' columns.
#pragma once

#include "common.hpp"

namespace ph {
namespace heat {

// Fused multiply-add in the cell's own precision.
__device__ __forceinline__ float fma_t(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_t(double a, double b, double c) { return __builtin_fma(a, b, c); }

// Whole-wavefront lane shifts by one (DPP wave_shr:1 / wave_shl:1): lane i
// receives lane i-1's (shr) or lane i+1's (shl) value; the lane at the end
// receives 0.  One VALU move per 32 bits instead of an LDS-crossbar
// permute.  Only lanes 0 and 63 see the 0, and the stencil never stores them
// unless that 0 is the value outside the grid.
constexpr int kDppWaveShr1 = 0x138;
constexpr int kDppWaveShl1 = 0x130;
template <int kCtrl>
__device__ __forceinline__ float lane_shift(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xf, 0xf, true));
}
template <int kCtrl>
__device__ __forceinline__ double lane_shift(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffff), kCtrl, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), kCtrl, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// The cell update, in the operation order of examples/heat_equation.cr:47 and
// :50 extended to two axes:
//   d = (((uN - 4u) + uS) + uW) + uE;  u' = u + d * r
// kFused: the first operation as one fused multiply-add (the same rounding
// where 4u does not overflow).  Float32 rounds u + d * r once.
template <typename T, bool kFused>
__device__ __forceinline__ T minus_4c(T n, T c) {
  if constexpr (kFused) return fma_t(T(-4), c, n);
  else return n - T(4) * c;
}
template <typename T>
__device__ __forceinline__ T step_cell(T c, T d, T r) {
  if constexpr (sizeof(T) == 4) return fma_t(d, r, c);
  else return c + d * r;
}

// Compensated FP64 sum (Neumaier) and the combination of two of them.
struct D2 {
  double s, c;
};
__device__ __forceinline__ void d2_add(D2 &a, double v) {
  const double t = a.s + v;
  const double d = (fabs(a.s) >= fabs(v)) ? ((a.s - t) + v) : ((v - t) + a.s);
  a.c += d;
  a.s = t;
}
__device__ __forceinline__ D2 d2_comb(const D2 &a, const D2 &b) {
  const double t = a.s + b.s;
  const double bb = t - a.s;
  const double err = (a.s - (t - bb)) + (b.s - bb);
  D2 r;
  r.s = t;
  r.c = (a.c + b.c) + err;
  return r;
}

// A pass of steps over the grid (heat_tile.hip).
struct Pass {
  int tile;         // index into the tiles of heat_tile.hip
  int64_t passes;   // passes the span is cut into
  int64_t groups;   // workgroups of a pass (the number of tiles), at most
  bool one;         // one tile covers the grid: in and out may be the same buffer
  double us;        // predicted time of all the passes
};
// Most workgroups of a pass that leave the field's energy as one partial sum
// each (two sums of a pass fill the fixed array of ph_heat2d_noalloc).  Passes
// of more sum the field in a pass of its own.
constexpr int64_t kEnergyGroups = 8192;
// The tile, and the number of passes, for `span` steps (span >= 1) of a
// ny x nx grid with at most kmax steps per pass.  parity 0 or 1: a number of
// passes of the other parity costs one copy of the grid (copy_us) more.
// Passes of more than kEnergyGroups groups cost sum_us more (the energy at the
// span's end takes a pass of its own).  only >= 0: that tile alone, where it can take the grid.
template <typename T>
Pass plan(int64_t ny, int64_t nx, int64_t span, int64_t kmax, int parity, double copy_us, double sum_us,
          int only);
// One pass of `steps` steps, cur -> nxt.  part0 / part1, when given, receive
// one compensated sum per workgroup of the field before / after the pass
// (*groups of them, at most p.groups); a lone workgroup writes the sum itself,
// as one double.
template <typename T>
int launch(const Pass &p, bool fused, const T *cur, T *nxt, int64_t ny, int64_t nx, T r, int64_t steps, D2 *part0,
           D2 *part1, int64_t *groups);

}  // namespace heat
}  // namespace ph
