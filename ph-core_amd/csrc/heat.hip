// Explicit 2-D heat equation (5-point FTCS, Dirichlet zero outside the grid):
// the runs (ph_heat2d, ph_heat2d_noalloc), and the FP64 reductions around them
// (total energy, relative L2 distance).  The step kernel, and how a run is cut
// into passes of several steps, are in heat_tile.hip.
//
// The cell update keeps the operation order of examples/heat_equation.cr:47
// and :50 extended to two axes:
//   d = (((uN - 4u) + uS) + uW) + uE;  u' = u + d * r
// with one contraction that changes no result: 4u is exact unless it
// overflows, so uN - 4u rounds once whether it is computed as a multiply and
// a subtract or as one fused multiply-add.  The fused form runs only when the
// host has shown that 4u cannot overflow in the passes ahead (fused_safe).
// Float32 grids (the build's own variant of the workload; the reference's
// example is Float64) also compute u + d * r as one fused multiply-add,
// which rounds once instead of twice: one instruction less per cell and
// step, with the accuracy stated against the Float64 run.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>

#include "heat_cell.hpp"

namespace {

using namespace ph::heat;

// ---------------------------------------------------------------------------
// Deterministic FP64 sums: pass 1 gives each workgroup a fixed contiguous
// chunk (Neumaier-compensated per thread, ordered tree per group); pass 2
// folds the per-group partials in a fixed order in one workgroup.
// ---------------------------------------------------------------------------
template <int K>
__device__ __forceinline__ void block_fold(D2 (&v)[K], D2 (*sh)[256]) {
  for (int k = 0; k < K; ++k) sh[k][threadIdx.x] = v[k];
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    D2 o[K];
    for (int k = 0; k < K; ++k) {
      o[k] = sh[k][threadIdx.x];
      if ((threadIdx.x & (2 * off - 1)) == 0) o[k] = d2_comb(o[k], sh[k][threadIdx.x + off]);
    }
    __syncthreads();
    for (int k = 0; k < K; ++k) sh[k][threadIdx.x] = o[k];
    __syncthreads();
  }
  for (int k = 0; k < K; ++k) v[k] = sh[k][0];
}

// mode 0: K=1 sum of a; mode 1: K=2 sums of (a-b)^2 and b^2
template <typename TA, typename TB, int K>
__global__ __launch_bounds__(256) void k_sum_pass1(const TA *__restrict__ a,
                                                   const TB *__restrict__ b, int64_t n,
                                                   int64_t chunk, D2 *part) {
  __shared__ D2 sh[K][256];
  const int64_t lo = (int64_t)blockIdx.x * chunk;
  const int64_t hi = (lo + chunk < n) ? lo + chunk : n;
  D2 acc[K];
  for (int k = 0; k < K; ++k) acc[k] = D2{0.0, 0.0};
  // lane-strided (coalesced); the order is fixed, so the result is
  // deterministic
  for (int64_t i = lo + threadIdx.x; i < hi; i += 256) {
    const double x = (double)a[i];
    if constexpr (K == 1) {
      d2_add(acc[0], x);
    } else {
      const double y = (double)b[i];
      const double d = x - y;
      d2_add(acc[0], d * d);
      d2_add(acc[1], y * y);
    }
  }
  block_fold<K>(acc, sh);
  if (threadIdx.x == 0)
    for (int k = 0; k < K; ++k) part[(int64_t)blockIdx.x * K + k] = acc[k];
}

template <int K>
__global__ __launch_bounds__(256) void k_sum_pass2(const D2 *__restrict__ part, int64_t nparts,
                                                   double *out) {
  __shared__ D2 sh[K][256];
  D2 acc[K];
  for (int k = 0; k < K; ++k) acc[k] = D2{0.0, 0.0};
#pragma unroll 4
  for (int64_t i = threadIdx.x; i < nparts; i += 256)
    for (int k = 0; k < K; ++k) acc[k] = d2_comb(acc[k], part[i * K + k]);
  block_fold<K>(acc, sh);
  if (threadIdx.x == 0)
    for (int k = 0; k < K; ++k) out[k] = acc[k].s + acc[k].c;
}

// `part_buf` (cap bytes), when given, holds the per-group partials instead
// of library scratch: at most 2048 groups, so 2048 * K * 16 bytes cover any n.
template <typename TA, typename TB, int K>
int fp64_sum(const TA *a, const TB *b, int64_t n, double *out, void *part_buf = nullptr, size_t cap = 0) {
  const int64_t nparts_max = 2048;
  int64_t chunk = (n + nparts_max - 1) / nparts_max;
  if (chunk < 4096) chunk = 4096;
  const int64_t nparts = (n + chunk - 1) / chunk;
  const size_t need = (size_t)(nparts > 0 ? nparts : 1) * K * sizeof(D2);
  void *part = part_buf;
  int rc = PH_OK;
  if (part) {
    if (need > cap)
      return ph::set_error(PH_E_ARGUMENT, "fp64 sum: %zu bytes of partials exceed the fixed %zu", need, cap);
  } else {
    rc = ph::scratch(need, &part, 2);
    if (rc) return rc;
  }
  rc = ph::launch_gate("fp64 sum");
  if (rc) return rc;
  if (nparts > 0)
    hipLaunchKernelGGL((k_sum_pass1<TA, TB, K>), dim3((unsigned)nparts), dim3(256), 0, ph::stream(),
                       a, b, n, chunk, (D2 *)part);
  hipLaunchKernelGGL((k_sum_pass2<K>), dim3(1), dim3(256), 0, ph::stream(), (const D2 *)part,
                     nparts, out);
  return ph::check_launch("k_sum");
}

// Largest |u| of the grid as an ordered bit pattern: with the sign bit
// cleared, finite values order as their magnitudes, and infinities and NaN
// order above every finite value.
template <typename T> struct Bits;
template <> struct Bits<float> {
  typedef unsigned int U;
  static constexpr U kMag = 0x7fffffffu;
  static constexpr U kLimit = 251u << 23;  // 2^124
  static constexpr double kEps = 0x1p-24;
};
template <> struct Bits<double> {
  typedef unsigned long long U;
  static constexpr U kMag = 0x7fffffffffffffffull;
  static constexpr U kLimit = 2043ull << 52;  // 2^1020
  static constexpr double kEps = 0x1p-53;
};

template <typename T>
__global__ __launch_bounds__(256) void k_absmax_bits(const T *__restrict__ u, int64_t n, typename Bits<T>::U *out) {
  using U = typename Bits<T>::U;
  const U *b = reinterpret_cast<const U *>(u);
  U m = 0;
  const int64_t stride = (int64_t)gridDim.x * 256;
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  for (; i + 7 * stride < n; i += 8 * stride) {  // eight loads in flight
    U v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = b[i + k * stride] & Bits<T>::kMag;
#pragma unroll
    for (int k = 0; k < 8; ++k) m = v[k] > m ? v[k] : m;
  }
  for (; i < n; i += stride) {
    const U v = b[i] & Bits<T>::kMag;
    m = v > m ? v : m;
  }
  for (int off = 32; off > 0; off >>= 1) {
    const U o = __shfl_xor(m, off);
    m = o > m ? o : m;
  }
  // one atomic per workgroup: atomics on the one word serialise, and one per
  // wavefront of 2048 workgroups took 96 us on a grid of 833250 cells
  __shared__ U sh[4];
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) m = sh[w] > m ? sh[w] : m;
    atomicMax(out, m);
  }
}

// Whether the next passes may compute uN - 4u as one fused multiply-add:
// 4u must not overflow in any of them.  For 0 <= r <= 1/4 the update is a
// convex combination of a cell and its neighbours (weights 1 - 4r and r),
// so the largest |u| cannot grow beyond rounding: each step's roundings add
// at most 11 eps of it (d carries four roundings of terms summing to at most
// 8 max|u|, and the product and the final sum one each).  Starting from
// max|u| <= 2^124 (Float32) or 2^1020 (Float64), 4u stays finite for
// ln 4 / (11 eps) steps (about 2.1 million for Float32); *steps_ok returns
// a bound within that, after which the host checks again.  A grid holding
// an infinity, a NaN or a larger value, or r outside [0, 1/4], keeps the
// separate multiply and subtract.
template <typename T>
int fused_safe(const T *u, int64_t n, T r, bool *safe, int64_t *steps_ok) {
  using U = typename Bits<T>::U;
  *safe = false;
  *steps_ok = 0;
  if (!(r >= T(0) && r <= T(0.25))) return PH_OK;
  void *p;
  int rc = ph::scratch(64, &p, 2);
  if (rc) return rc;
  rc = ph::clear_i32((int *)p, 2);
  if (rc) return rc;
  rc = ph::launch_gate("heat max|u|");
  if (rc) return rc;
  const int64_t blocks = std::min<int64_t>(1024, (n + 2047) / 2048);
  hipLaunchKernelGGL(k_absmax_bits<T>, dim3((unsigned)std::max<int64_t>(1, blocks)), dim3(256), 0, ph::stream(), u,
                     n, (U *)p);
  rc = ph::check_launch("k_absmax_bits");
  if (rc) return rc;
  U m = 0;
  rc = ph::fetch(&m, p, sizeof(U));
  if (rc) return rc;
  *safe = m <= Bits<T>::kLimit;
  *steps_ok = (int64_t)(0.5 * std::log(4.0) / (11.0 * Bits<T>::kEps));
  return PH_OK;
}

// part_buf / part_cap: a fixed buffer for the energy partials (the
// allocation-free entry point); allow_fused: the fused first operation may
// be used (it needs one read-back of max|u|).
template <typename T>
int heat_run(T *u, T *tmp, int64_t ny, int64_t nx, double r, int64_t steps, int64_t every,
             double *energy, void *part_buf = nullptr, size_t part_cap = 0, bool allow_fused = true) {
  // The steps up to each energy checkpoint are cut into passes of equal
  // length by the tile and pass plan; PH_HEAT_K caps the steps of a pass.
  int64_t kmax = INT32_MAX;
  if (const char *e = std::getenv("PH_HEAT_K")) kmax = std::max<int64_t>(1, std::atol(e));
  int only = -1;
  if (const char *e = std::getenv("PH_HEAT_TILE")) only = std::atoi(e);  // tuning override: one tile of heat_tile.hip
  const T rr = (T)r;
  const bool sums = energy && every > 0;
  T *cur = u;
  int rc;
  if (sums && steps == 0) return fp64_sum<T, T, 1>(u, u, ny * nx, energy, part_buf, part_cap);
  // one grid copy, which an odd number of passes needs at the end
  const double copy_us = 4.0 + 2.0 * sizeof(T) * (double)ny * (double)nx / 5e6;
  // and the field's energy in a pass of its own
  const double sum_us = sums ? 6.0 + sizeof(T) * (double)ny * (double)nx / 3.1e6 : 0.0;
  bool fused = false, try_fused = false;
  int64_t fused_until = 0;
  Pass p{-1, 0, 0, false, 0.0};
  int64_t planned = 0;  // the span `p` is for
  int64_t t = 0;
  while (t < steps) {
    const int64_t until = sums ? std::min<int64_t>(steps, (t / every + 1) * every) : steps;
    const int64_t span = until - t;
    if (span != planned || until == steps) {
      // the last passes should leave the field in u
      p = plan<T>(ny, nx, span, kmax, until == steps ? (cur == u ? 0 : 1) : -1, copy_us, sum_us, only);
      planned = span;
      if (p.tile < 0) return ph::set_error(PH_E_UNSUPPORTED, "heat grid %lld x %lld", (long long)ny, (long long)nx);
    }
    // The fused form saves one instruction of six to eight and needs a
    // read-back of max|u| (some 25 us), so short runs keep the separate
    // multiply and subtract.
    if (t == 0) try_fused = allow_fused && steps >= 32 && p.us * ((double)steps / (double)span) > 300.0;
    if (try_fused && t >= fused_until) {
      int64_t ok = 0;
      rc = fused_safe<T>(cur, ny * nx, rr, &fused, &ok);
      if (rc) return rc;
      fused_until = fused ? t + ok : steps;
    }
    for (int64_t left = p.passes; left > 0; --left) {
      const int64_t k = (until - t + left - 1) / left;
      T *nxt = p.one ? u : (cur == u ? tmp : u);
      const bool e0 = sums && t == 0, e1 = sums && (t + k) % every == 0;
      // the field's energy before the first pass and after one that ends at a
      // checkpoint: summed by the pass itself from its registers
      const bool inside = p.groups <= kEnergyGroups;
      D2 *part0 = nullptr, *part1 = nullptr;
      if (e0 && !inside) {
        rc = fp64_sum<T, T, 1>(cur, cur, ny * nx, energy, part_buf, part_cap);
        if (rc) return rc;
      }
      const int64_t ei = sums ? (t + k) / every : 0;
      if ((e0 || e1) && inside) {
        if (p.groups == 1) {  // a lone workgroup writes the energy itself
          part0 = (D2 *)energy;
          part1 = (D2 *)(energy + ei);
        } else {
          void *base = part_buf;
          if (!base) {
            rc = ph::scratch(2 * kEnergyGroups * sizeof(D2), &base, 2);
            if (rc) return rc;
          } else if (part_cap < 2 * kEnergyGroups * sizeof(D2)) {
            return ph::set_error(PH_E_ARGUMENT, "heat energy: partials exceed the fixed %zu bytes", part_cap);
          }
          part0 = (D2 *)base;
          part1 = part0 + kEnergyGroups;
        }
      }
      rc = ph::launch_gate("heat step");
      if (rc) return rc;
      int64_t groups = 0;
      rc = launch<T>(p, fused, cur, nxt, ny, nx, rr, k, e0 ? part0 : nullptr, e1 ? part1 : nullptr, &groups);
      if (rc) return rc;
      cur = nxt;
      t += k;
      if ((e0 || e1) && inside && p.groups > 1) {
        rc = ph::launch_gate("heat energy");
        if (rc) return rc;
        if (e0) hipLaunchKernelGGL((k_sum_pass2<1>), dim3(1), dim3(256), 0, ph::stream(), part0, groups, energy);
        if (e1) hipLaunchKernelGGL((k_sum_pass2<1>), dim3(1), dim3(256), 0, ph::stream(), part1, groups, energy + ei);
        rc = ph::check_launch("k_sum");
        if (rc) return rc;
      } else if (e1 && !inside) {
        rc = fp64_sum<T, T, 1>(cur, cur, ny * nx, energy + ei, part_buf, part_cap);
        if (rc) return rc;
      }
    }
  }
  if (cur != u) PH_HIP(hipMemcpyAsync(u, cur, sizeof(T) * (size_t)(ny * nx), hipMemcpyDeviceToDevice, ph::stream()));
  return PH_OK;
}

}  // namespace

// ---------------------------------------------------------------------------
// The allocation-free heat run (ph_heat2d_noalloc) keeps its FP64 energy
// partials in this fixed device array instead of library scratch: the sums
// before and after a pass of at most kEnergyGroups groups, one compensated
// pair each (fp64_sum uses 2048 of them at most).  Its device
// address is looked up once per device when the library is initialised on
// it; host code uses that address, never the array's name.  Inside namespace
// ph the bare name would find the function ph::scratch (library scratch), so
// the lookup names the array as ::scratch.
// ---------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[2 * kEnergyGroups * sizeof(D2)];

namespace {
constexpr int kMaxDevices = 64;
void *g_noalloc_scratch[kMaxDevices] = {nullptr};
}  // namespace

namespace ph {

int heat_noalloc_setup(int device) {
  if (device < 0 || device >= kMaxDevices)
    return set_error(PH_E_ARGUMENT, "device %d beyond the %d the fixed heat scratch tracks", device, kMaxDevices);
  void *p = nullptr;
  const hipError_t e = hipGetSymbolAddress((void **)&p, HIP_SYMBOL(::scratch));
  if (e != hipSuccess || !p)
    return set_error(PH_E_HIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
  g_noalloc_scratch[device] = p;
  return PH_OK;
}

}  // namespace ph

extern "C" {

int ph_heat2d_noalloc(int32_t dtype, void *u, void *tmp, int64_t ny, int64_t nx, double r, int64_t steps,
                      int64_t energy_every, double *energy_out) {
  PH_GUARD();
  PH_REQUIRE_INIT();
  if (ny <= 0 || nx <= 0) return ph::set_error(PH_E_DIMENSION, "heat grid %lld x %lld", (long long)ny, (long long)nx);
  if (steps < 0) return ph::set_error(PH_E_ARGUMENT, "negative step count");
  if (!u || !tmp || u == tmp) return ph::set_error(PH_E_ARGUMENT, "heat2d needs two distinct buffers");
  if (energy_every > 0 && !energy_out) return ph::set_error(PH_E_ARGUMENT, "energy_out is null");
  const int dev = ph::device();
  void *sp = dev >= 0 && dev < kMaxDevices ? g_noalloc_scratch[dev] : nullptr;
  if (!sp) return ph::set_error(PH_E_NOINIT, "the fixed heat scratch of device %d was not set up", dev);
  const size_t cap = sizeof(::scratch);
  if (dtype == PH_F32)
    return heat_run<float>((float *)u, (float *)tmp, ny, nx, r, steps, energy_every, energy_out, sp, cap, false);
  if (dtype == PH_F64)
    return heat_run<double>((double *)u, (double *)tmp, ny, nx, r, steps, energy_every, energy_out, sp, cap, false);
  return ph::set_error(PH_E_ARGUMENT, "heat2d: dtype %d (F32 or F64)", dtype);
}

int ph_heat2d(int32_t dtype, void *u, void *tmp, int64_t ny, int64_t nx, double r, int64_t steps,
              int64_t energy_every, double *energy_out) {
  PH_GUARD();
  PH_REQUIRE_INIT();
  if (ny <= 0 || nx <= 0) return ph::set_error(PH_E_DIMENSION, "heat grid %lld x %lld", (long long)ny, (long long)nx);
  if (steps < 0) return ph::set_error(PH_E_ARGUMENT, "negative step count");
  if (!u || !tmp || u == tmp) return ph::set_error(PH_E_ARGUMENT, "heat2d needs two distinct buffers");
  if (energy_every > 0 && !energy_out) return ph::set_error(PH_E_ARGUMENT, "energy_out is null");
  if (dtype == PH_F32) return heat_run<float>((float *)u, (float *)tmp, ny, nx, r, steps, energy_every, energy_out);
  if (dtype == PH_F64) return heat_run<double>((double *)u, (double *)tmp, ny, nx, r, steps, energy_every, energy_out);
  return ph::set_error(PH_E_ARGUMENT, "heat2d: dtype %d (F32 or F64)", dtype);
}

int ph_l2_diff(int32_t dtype_a, const void *a, int32_t dtype_b, const void *b, int64_t n, double *out) {
  PH_GUARD();
  PH_REQUIRE_INIT();
  if (n < 0 || !out) return ph::set_error(PH_E_ARGUMENT, "ph_l2_diff arguments");
  if (dtype_a == PH_F32 && dtype_b == PH_F64) return fp64_sum<float, double, 2>((const float *)a, (const double *)b, n, out);
  if (dtype_a == PH_F64 && dtype_b == PH_F64) return fp64_sum<double, double, 2>((const double *)a, (const double *)b, n, out);
  if (dtype_a == PH_F32 && dtype_b == PH_F32) return fp64_sum<float, float, 2>((const float *)a, (const float *)b, n, out);
  if (dtype_a == PH_F64 && dtype_b == PH_F32) return fp64_sum<double, float, 2>((const double *)a, (const float *)b, n, out);
  return ph::set_error(PH_E_ARGUMENT, "ph_l2_diff: dtypes %d, %d", dtype_a, dtype_b);
}

}  // extern "C"
