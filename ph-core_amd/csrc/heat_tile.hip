// The heat step kernel: passes that keep a tile of the grid in registers.
//
// A workgroup of W wavefronts holds a tile of 64 V x W R cells (a lane: V
// consecutive columns; a wavefront: R consecutive rows) and advances it in
// place, any number of steps, before it writes the tile back: west and east
// neighbours come from the adjacent lane (DPP), north and south from the
// lane's own registers, and only the first and the last row of a wavefront
// pass through LDS (two buffers, one barrier a step).  A side of the tile
// that is not the grid's edge loses one ring of cells per step, so tiles
// overlap by `steps` cells there; a tile flush with the edge loses nothing
// (the zero beyond the wavefront's or the tile's end is the boundary value),
// and a grid that fits one tile runs all its steps in one launch.
//
// What bounds it, and why it took the place of a sweep that streamed rows
// through each wavefront (12 Float32 or 8 Float64 time levels in registers):
// the sweep makes every wavefront one long serial chain of rows, which left
// most of the chip idle below a few thousand rows (750 x 1111 Float64: 36 us
// for 8 steps), and its registers grow with the steps per pass.  Here the
// state is one value per cell whatever the steps, so their number is free:
// it balances the overlap against the launches (small grids) or the memory
// traffic (large ones).  The inner loop issues 5.1 vector instructions per
// cell and step at Float32 (five operations, the lane shifts folded into the
// additions) and 8.1 at Float64 (six, and two shifts of two words each per
// pair of cells).  At 8192^2 that keeps the vector ALUs 96% busy at Float32;
// the rest is the overlap (a third of the cells at 16 steps and 128 x 256).
// Time per step, the sweep's and this kernel's, over runs of 100 steps (and in
// passes of one step and of two: 8192^2 Float32 116 -> 102 and 59 -> 51 us, Float64
// 233 -> 196 and 119 -> 97):
//   8192^2     Float32 18.6 -> 13.9 us, Float64 36 -> 27.8 us
//   2048^2     Float32 3.9 -> 1.58, Float64 5.6 -> 3.0 us
//   1024^2     Float32 3.6 -> 0.89, Float64 3.9 -> 1.27 us
//   750 x 1111 Float32 6.1 -> 0.88, Float64 5.8 -> 1.18 us
//   64^2       Float64 2.7 -> 0.41 us (one workgroup)
//
// Every cell is computed with the single-step formula, so results are
// bit-identical to single steps.
#include <algorithm>
#include <cmath>

#include "heat_cell.hpp"

namespace {

using namespace ph::heat;

struct TileArgs {
  int64_t ny, nx;
  int64_t ux, uy;     // columns and rows a tile writes
  int32_t hx, hy;     // cells of overlap on each side (0 when one tile spans the axis)
  int32_t ntx;        // tiles along x
  int32_t steps;      // steps of this pass
  D2 *part0, *part1;  // sums of the cells each tile writes, before and after (may be null)
};

// kMask: the grid is narrower or lower than a tile, so the cells of the tile
// beyond the grid are held at zero after every step.
// Eight wavefronts to a SIMD are asked for in whole tiles of 16 wavefronts: the
// separate form of 128 x 256 Float32 took 65 registers, one too many for two
// workgroups on a CU (8192^2, 20 steps a pass: 477 us, and 340 with 64).
template <typename T, int V, int R, int W, bool kFused, bool kMask>
__global__ __launch_bounds__(64 * W, W == 16 && !kMask ? 8 : 0) void k_heat_tile(const T *u, T *out, TileArgs a, T r) {
  constexpr int TX = 64 * V, TY = W * R;
  typedef T Row __attribute__((ext_vector_type(V)));
  struct __attribute__((packed, aligned(sizeof(T)))) RowU {
    T v[V];
  };
  __shared__ D2 esh[W];
  // [buffer][wavefront + 1][first, last row]; the rows beyond the first and
  // last wavefront stay zero (a lone wavefront exchanges none)
  __shared__ T sh[2][W + 2][2][W > 1 ? TX : 1];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // Each XCD (workgroups are dealt to the eight in turn) takes an eighth of the
  // tiles in order, so that its L2 sees both writers of a line and the overlap
  // that neighbours read (8192^2 one step, with vector stores below, against
  // tiles dealt in turn: Float32 147 -> 114 us, Float64 254 -> 199; 16 and 10
  // steps a pass: 14.6 -> 14.2 and 28.1 -> 27.4 us a step, 1024^2 1.19 -> 0.89
  // and 1.51 -> 1.27).
  const int q8 = (int)gridDim.x >> 3, r8 = (int)gridDim.x & 7, xcd = (int)blockIdx.x & 7;
  const int tile = xcd * q8 + (xcd < r8 ? xcd : r8) + ((int)blockIdx.x >> 3);
  const int64_t tx = tile % a.ntx, ty = tile / a.ntx;
  // the tile's first cell: `h` before the cells it writes, moved inside the
  // grid (a tile flush with an edge needs no overlap there)
  const int64_t mx = a.nx > TX ? a.nx - TX : 0, my = a.ny > TY ? a.ny - TY : 0;
  int64_t xs = tx * a.ux - a.hx, ys = ty * a.uy - a.hy;
  xs = xs < 0 ? 0 : (xs > mx ? mx : xs);
  ys = ys < 0 ? 0 : (ys > my ? my : ys);
  // The wavefront's first row and the tile's first column are uniform, so
  // row addresses live in scalar registers and a lane adds a 32-bit offset:
  // 64-bit addresses per lane and row would cost a third of the vector
  // registers (128 x 256 cells of Float32: 114 instead of 64, half the
  // wavefronts, 2.1 ms for 100 steps of 8192^2 instead of 1.5).
  const int64_t y = ys + wave * R;
  const int lx = lane * V;
  const int nc = (int)(a.nx - xs < TX ? a.nx - xs : TX);        // columns of the tile inside the grid
  const int nr = (int)(a.ny - y < R ? (a.ny > y ? a.ny - y : 0) : R);  // rows of the wavefront inside it
  bool colok[V];
#pragma unroll
  for (int v = 0; v < V; ++v) colok[v] = !kMask || lx + v < nc;

  T c[R][V];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if constexpr (kMask) {
      const T *row = u + (i < nr ? y + i : a.ny - 1) * a.nx + xs;
      if (nc == TX) {  // rows alone are missing
        const RowU t = *(const RowU *)(row + (unsigned)lx);
#pragma unroll
        for (int v = 0; v < V; ++v) c[i][v] = i < nr ? t.v[v] : T(0);
      } else {
#pragma unroll
        for (int v = 0; v < V; ++v) {
          const T t = row[(unsigned)(colok[v] ? lx + v : 0)];
          c[i][v] = (colok[v] && i < nr) ? t : T(0);
        }
      }
    } else {
      const T *row = u + (y + i) * a.nx + xs;
      const RowU t = *(const RowU *)(row + (unsigned)lx);
#pragma unroll
      for (int v = 0; v < V; ++v) c[i][v] = t.v[v];
    }
  }
  auto put = [&](const T (&row)[V], T *dst) {
    Row t;
#pragma unroll
    for (int v = 0; v < V; ++v) t[v] = row[v];
    *(Row *)(dst + lane * V) = t;
  };
  auto get = [&](const T *src, T (&row)[V]) {
    const Row t = *(const Row *)(src + lane * V);
#pragma unroll
    for (int v = 0; v < V; ++v) row[v] = t[v];
  };
  // row i of the wavefront <- its next step: `n4` holds north - 4 centre of
  // its cells, s the old row south of it
  auto update = [&](int i, const T (&n4)[V], const T (&s)[V]) {
    const T wl = lane_shift<kDppWaveShr1>(c[i][V - 1]);
    const T er = lane_shift<kDppWaveShl1>(c[i][0]);
    T d[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const T w = v == 0 ? wl : c[i][v - 1];
      const T e = v == V - 1 ? er : c[i][v + 1];
      d[v] = ((n4[v] + s[v]) + w) + e;
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
      c[i][v] = step_cell(c[i][v], d[v], r);
      if constexpr (kMask) c[i][v] = (i < nr && colok[v]) ? c[i][v] : T(0);
    }
  };
  auto north = [&](const T (&n)[V], int i, T (&o)[V]) {
#pragma unroll
    for (int v = 0; v < V; ++v) o[v] = minus_4c<T, kFused>(n[v], c[i][v]);
  };
  // the cells this tile writes: columns [cx0, cx1) of the tile, rows
  // [ry0, ry1) of the wavefront
  const int64_t gx = tx * a.ux - xs, gy = ty * a.uy - y;
  const int cx0 = (int)gx, cx1 = (int)(gx + a.ux < nc ? gx + a.ux : nc);
  const int ry0 = (int)(gy > 0 ? (gy < R ? gy : R) : 0), ry1 = (int)(gy + a.uy < nr ? gy + a.uy : nr);
  bool own[V];
#pragma unroll
  for (int v = 0; v < V; ++v) own[v] = lx + v >= cx0 && lx + v < cx1;
  // their sum in FP64: per lane in row order, then a fixed tree
  auto sum_to = [&](D2 *part) {
    D2 e{0.0, 0.0};
#pragma unroll
    for (int i = 0; i < R; ++i)
      if (i >= ry0 && i < ry1) {
#pragma unroll
        for (int v = 0; v < V; ++v) d2_add(e, own[v] ? (double)c[i][v] : 0.0);
      }
    for (int off = 32; off > 0; off >>= 1) {
      D2 o;
      o.s = __shfl_down(e.s, off);
      o.c = __shfl_down(e.c, off);
      e = d2_comb(e, o);
    }
    if (lane == 0) esh[wave] = e;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < W; ++w) e = d2_comb(e, esh[w]);
      if (gridDim.x == 1) *(double *)part = e.s + e.c;
      else part[tile] = e;
    }
    __syncthreads();
  };
  if (a.part0) sum_to(a.part0);
  if constexpr (W > 1)
    for (int i = threadIdx.x; i < 2 * TX; i += 64 * W) sh[i / TX][0][1][i % TX] = sh[i / TX][W + 1][0][i % TX] = T(0);
  for (int s = 0; s < a.steps; ++s) {
    auto *b = sh[s & 1];
    T second[V], nn[V], nx4[V], up[V], dn[V];
    if constexpr (W > 1) {
      put(c[0], b[wave + 1][0]);
      put(c[R - 1], b[wave + 1][1]);
    } else {  // a lone wavefront holds all rows: beyond them is the boundary
#pragma unroll
      for (int v = 0; v < V; ++v) up[v] = dn[v] = T(0);
    }
#pragma unroll
    for (int v = 0; v < V; ++v) second[v] = R > 1 ? c[R > 1][v] : T(0);
    if constexpr (R > 1) north(c[0], 1, nn);
    // Rows are updated in place, top down: a row's north - 4 centre is taken
    // before the row above it changes.  Half of the inner rows run before the
    // barrier, half while the neighbours' rows are read; the first row, whose
    // north comes from another wavefront, is last.
    constexpr int kHalf = (R - 2) / 2;
#pragma unroll
    for (int i = 1; i < R; ++i) {
      if constexpr (W > 1)
        if (i == 1 + kHalf) {
          __syncthreads();
          get(b[wave][1], up);
          get(b[wave + 2][0], dn);
        }
      if (i < R - 1) {
        north(c[i], i + 1, nx4);
        update(i, nn, c[i + 1]);
#pragma unroll
        for (int v = 0; v < V; ++v) nn[v] = nx4[v];
      } else {
        update(i, nn, dn);
      }
    }
    north(up, 0, nn);
    update(0, nn, second);
  }
  if (a.part1) sum_to(a.part1);
#pragma unroll
  for (int i = 0; i < R; ++i)
    if (i >= ry0 && i < ry1) {
      T *row = out + (y + i) * a.nx + xs;
      if (own[0] && own[V - 1]) {
        RowU t;
#pragma unroll
        for (int v = 0; v < V; ++v) t.v[v] = c[i][v];
        *(RowU *)(row + (unsigned)lx) = t;
      } else {
#pragma unroll
        for (int v = 0; v < V; ++v)
          if (own[v]) row[(unsigned)(lx + v)] = c[i][v];
      }
    }
}

// The tiles, by dtype.  Measured over 24 grids from 33 x 47 to 8192^2 and 23
// tiles: the first eight leave the best of all 23 at most a few percent ahead
// (the last of them serve the large grids, 64 x 32 the small ones, the narrow
// rows of 64 x 48 and 64 x 64 a grid that fits one tile).  The other nine are
// for grids of few rows, where 32 rows and more would mostly hold cells beyond
// the grid, or 64 columns mostly overlap: up to 16 rows one wavefront spans them,
// without LDS or barrier, then two and four.  Per run of 100 steps (and of one), the
// sweep, the first eight tiles alone, and all:
//   1 x 10^7      Float32 2888 (68), 4119 (280),  127 (40) us, Float64 2650 (102), 6465 (321),  304 (59)
//   4 x 4 10^6    Float32 1555 (54), 2033 (148),  290 (51) us, Float64 1711 (94),  3236 (195),  482 (85)
//   16 x 10^6     Float32  949 (53),  660 (69),   342 (51) us, Float64 1211 (90),  1062 (97),   591 (85)
//   50 x 5 10^5   Float32  805 (73), 1139 (80),   731 (80) us, Float64 1545 (181), 1448 (168), 1362 (172)
struct Tile {
  int v, r, w;
};
template <typename T> struct Tiles;
template <> struct Tiles<double> {
  [[maybe_unused]] static constexpr Tile t[17] = {{1, 4, 8},  {1, 6, 8},  {1, 8, 8}, {2, 4, 8}, {2, 8, 8},  {2, 12, 8},
                                                  {2, 16, 8}, {2, 24, 8}, {4, 1, 1}, {4, 2, 1}, {4, 4, 1},  {4, 8, 1},
                                                  {2, 16, 1}, {2, 12, 2}, {2, 16, 2}, {2, 12, 4}, {2, 16, 4}};
};
template <> struct Tiles<float> {
  [[maybe_unused]] static constexpr Tile t[17] = {{1, 4, 8},   {1, 6, 8},   {1, 8, 8}, {2, 4, 8}, {2, 8, 16}, {2, 12, 8},
                                                  {2, 12, 16}, {2, 16, 16}, {4, 1, 1}, {4, 2, 1}, {4, 4, 1},  {4, 8, 1},
                                                  {2, 16, 1},  {2, 12, 2},  {2, 16, 2}, {2, 12, 4}, {2, 16, 4}};
};
constexpr int kTiles = 17;

struct Cut {
  int64_t ux, uy, ntx, nty;
};
// How tile t covers a ny x nx grid with k steps per pass; false when the
// overlap leaves too little of the tile.
template <typename T>
bool cut(const Tile &t, int64_t ny, int64_t nx, int64_t k, Cut *c) {
  const int64_t tx = 64 * t.v, ty = (int64_t)t.w * t.r;
  if (t.w == 1 && ny > ty) return false;  // (a lone wavefront spans the rows)
  c->ux = nx > tx ? tx - 2 * k : nx;
  c->uy = ny > ty ? ty - 2 * k : ny;
  if ((nx > tx && c->ux < tx / 8) || (ny > ty && c->uy < ty / 8)) return false;
  c->ntx = (nx + c->ux - 1) / c->ux;
  c->nty = (ny + c->uy - 1) / c->uy;
  return c->ntx * c->nty < (int64_t(1) << 30);
}

// Predicted time (us) of one pass of k steps: the launch, then per step
// either a workgroup's own latency (barrier and LDS exchange, and its work
// alone on a CU, of which a lone wavefront has one SIMD of four) or, with
// several workgroups to a CU, the CU's throughput, and the tiles' memory
// traffic.  The constants of the tiles of eight wavefronts and more are a fit to
// 7000 timings (17% rms over grids, tiles and steps), those of the smaller ones
// minimise the time of the tiles chosen for 65 grids of 1 to 100 rows and up
// to 10^6 columns and 20 others, 1 to 100 steps: on average within 3.7%
// (Float32) and 2.7% (Float64) of the best tile and number of steps, and 16%
// and 12% faster than with the first eight tiles alone.  A grid beyond the
// 256 MB MALL is streamed, at less in tall tiles, in rows of 256 bytes and in few
// rows (8192^2, one step: Float64 195 us in tiles of 4096 cells, 232 in 24576;
// Float32 101 us in 128 x 32, 114 in 64 x 32, 121 in 128 x 24); the Float32 rate
// is lower than the best measured, 5.3 TB/s, since four steps hide behind it in
// part only (109 us in 128 x 96 and 115 in 128 x 192, which the higher rate
// preferred).
struct Cost {
  double launch, fixed, alone, shared;  // a step alone: fixed + alone * work; with others: shared * work
};
template <typename T>
Cost cost(const Tile &t) {
  if constexpr (sizeof(T) == 8)
    return t.w == 1 ? Cost{2.3, 0.02, 1.4, 0.6} : t.w < 8 ? Cost{1.4, 0.7, 1.87, 1.07} : Cost{2.1, 0.129, 0.913, 0.805};
  else
    return t.w == 1 ? Cost{2.6, 0.1, 0.82, 0.69} : t.w < 8 ? Cost{2.3, 0.175, 0.76, 0.73} : Cost{t.w == 16 ? 0.7 : 2.5, 0.086, 0.831, 0.565};
}
template <typename T>
double pass_us(const Tile &t, int64_t ny, int64_t nx, int64_t k, const Cut &c) {
  constexpr bool f64 = sizeof(T) == 8;
  const bool mask = nx < 64 * t.v || ny < (int64_t)t.w * t.r;
  const double insn = (f64 ? 6 * t.v + 4 : 5 * t.v) + (mask ? (f64 ? 2 : 1) * t.v : 0);
  const double wave = (t.r * insn + 8) * 4 / 2400;  // of a step, of one wavefront
  const double work = t.w / 4.0 * wave;             // on a CU's four SIMDs
  const double traffic = 64.0 * t.v * t.w * t.r * sizeof(T) * 2 * 256 / 5e6;
  const double g = (double)(c.ntx * c.nty) / 256;
  const double per_cu = g <= 1 ? 1 : (g < 6 ? std::ceil(g) : g + 0.4);
  const Cost f = cost<T>(t);
  const double step = std::max(f.fixed + f.alone * std::max(wave, work), f.shared * work * per_cu);
  const double us = f.launch + k * step + (f64 ? (mask ? 0.38 : 0.486) : 0.685) * traffic * per_cu;
  const double bytes = 2.0 * sizeof(T) * (double)ny * (double)nx;
  if (bytes <= 256e6) return us;
  const double cells = t.v * t.w * t.r / 16.0;  // of a tile, in 1024
  const bool few = t.w < 8 && c.nty > 1;
  const double stream = f64 ? bytes / 5.65e6 * (1 + 0.009 * cells) * (t.v == 1 ? 1.02 : 1) * (few ? 1.08 : 1)
                            : bytes / 4.7e6 * (1 + 0.004 * cells) * (t.v == 1 ? 1.09 : 1) * (few ? 1.2 : 1);
  return std::max(us, stream);
}

template <typename T, int V, int R, int W>
int launch_tile(bool fused, bool mask, unsigned grid, const T *cur, T *nxt, const TileArgs &a, T r) {
  const dim3 g(grid), b(64 * W);
  if (fused && mask) hipLaunchKernelGGL((k_heat_tile<T, V, R, W, true, true>), g, b, 0, ph::stream(), cur, nxt, a, r);
  else if (fused) hipLaunchKernelGGL((k_heat_tile<T, V, R, W, true, false>), g, b, 0, ph::stream(), cur, nxt, a, r);
  else if (mask) hipLaunchKernelGGL((k_heat_tile<T, V, R, W, false, true>), g, b, 0, ph::stream(), cur, nxt, a, r);
  else hipLaunchKernelGGL((k_heat_tile<T, V, R, W, false, false>), g, b, 0, ph::stream(), cur, nxt, a, r);
  return ph::check_launch("k_heat_tile");
}

template <typename T, int I>
int launch_index(int i, bool fused, bool mask, unsigned grid, const T *cur, T *nxt, const TileArgs &a, T r) {
  if constexpr (I < kTiles) {
    constexpr Tile t = Tiles<T>::t[I];
    if (i == I) return launch_tile<T, t.v, t.r, t.w>(fused, mask, grid, cur, nxt, a, r);
    return launch_index<T, I + 1>(i, fused, mask, grid, cur, nxt, a, r);
  } else {
    return ph::set_error(PH_E_ARGUMENT, "heat tile %d", i);
  }
}

}  // namespace

namespace ph {
namespace heat {

template <typename T>
Pass plan(int64_t ny, int64_t nx, int64_t span, int64_t kmax, int parity, double copy_us, double sum_us, int only) {
  Pass best{-1, 0, 0, false, 0.0};
  for (int i = 0; i < kTiles; ++i) {
    const Tile &t = Tiles<T>::t[i];
    if (only >= 0 ? i != only : t.w < 8 && ny > 2 * t.w * t.r) continue;  // (low tiles are for low grids)
    const bool one = nx <= 64 * t.v && ny <= (int64_t)t.w * t.r;
    // a launch holds the device for some milliseconds at most
    const int64_t kcap = std::min(kmax, one ? int64_t(4096) : int64_t(48));
    int64_t seen = -1;
    for (int64_t k0 = one ? kcap : 1; k0 <= kcap; ++k0) {
      const int64_t passes = (span + k0 - 1) / k0;
      const int64_t k = (span + passes - 1) / passes;
      if (passes == seen && k0 < span) continue;
      seen = passes;
      Cut c;
      if (!cut<T>(t, ny, nx, k, &c)) break;  // more steps leave less of the tile
      double us = passes * pass_us<T>(t, ny, nx, k, c);
      if (!one && parity >= 0 && passes % 2 != parity) us += copy_us;
      if (c.ntx * c.nty > kEnergyGroups) us += sum_us;
      if (best.tile < 0 || us < best.us) best = Pass{i, passes, c.ntx * c.nty, one, us};
      if (k0 >= span) break;
    }
  }
  if (best.tile < 0 && only >= 0) return plan<T>(ny, nx, span, kmax, parity, copy_us, sum_us, -1);
  return best;
}

template <typename T>
int launch(const Pass &p, bool fused, const T *cur, T *nxt, int64_t ny, int64_t nx, T r, int64_t steps, D2 *part0,
           D2 *part1, int64_t *groups) {
  const Tile &t = Tiles<T>::t[p.tile];
  Cut c;
  if (p.tile < 0 || p.tile >= kTiles || steps < 1 || !cut<T>(t, ny, nx, steps, &c) || c.ntx * c.nty > p.groups ||
      (cur == nxt && c.ntx * c.nty != 1))
    return ph::set_error(PH_E_ARGUMENT, "heat pass of %lld steps", (long long)steps);
  TileArgs a;
  a.ny = ny;
  a.nx = nx;
  a.ux = c.ux;
  a.uy = c.uy;
  a.hx = c.ntx > 1 ? (int32_t)steps : 0;
  a.hy = c.nty > 1 ? (int32_t)steps : 0;
  a.ntx = (int32_t)c.ntx;
  a.steps = (int32_t)steps;
  a.part0 = part0;
  a.part1 = part1;
  *groups = c.ntx * c.nty;
  const bool mask = nx < 64 * t.v || ny < (int64_t)t.w * t.r;
  return launch_index<T, 0>(p.tile, fused, mask, (unsigned)(c.ntx * c.nty), cur, nxt, a, r);
}

#define PH_HEAT_INSTANCE(T)                                                                \
  template Pass plan<T>(int64_t, int64_t, int64_t, int64_t, int, double, double, int);      \
  template int launch<T>(const Pass &, bool, const T *, T *, int64_t, int64_t, T, int64_t, D2 *, D2 *, int64_t *);
// (the build compiles this file once per type, side by side)
#ifdef PH_HEAT_T
PH_HEAT_INSTANCE(PH_HEAT_T)
#else
PH_HEAT_INSTANCE(float)
PH_HEAT_INSTANCE(double)
#endif

}  // namespace heat
}  // namespace ph
