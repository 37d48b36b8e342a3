// Strided copies, fills and seeded random fills (hand-written, ahead-of-time).
//
// Layout of the work: a copy over a logical shape is first collapsed
// (ph::collapse) to `rows x cols` with the innermost axis as `cols`.  One
// 256-thread workgroup owns a tile of kTile consecutive columns of one row;
// lane t of the group handles columns tile0 + e*256 + t for e < EPT, so for
// every unrolled e the 64 lanes of a wavefront touch 64 consecutive elements
// of the destination (fully coalesced) and consecutive source elements
// `s_inner` apart (coalesced for |s_inner| <= 2 within 512-byte spans).  All
// EPT loads are issued before the stores, keeping EPT x 256 B per wavefront in
// flight.  Row offsets are decoded once per workgroup, in scalar registers.
#include <algorithm>
#include <cstring>
#include <type_traits>

#include "common.hpp"

namespace {

constexpr int kBlock = 256;
constexpr int64_t kStreamBytes = int64_t(100) << 20;

struct RowArgs {
  int64_t rows;
  int64_t cols;
  int64_t ntiles;
  int64_t nblocks;
  int32_t outer_rank;
  int32_t pad_;
  int64_t outer_shape[PH_MAX_RANK];
  int64_t d_off, s_off;
  int64_t d_outer[PH_MAX_RANK];
  int64_t s_outer[PH_MAX_RANK];
  int64_t d_inner, s_inner;
};

__device__ __forceinline__ void decode_row(const RowArgs &a, int64_t row, int64_t *d_base,
                                           int64_t *s_base) {
  int64_t d = a.d_off, s = a.s_off;
  for (int k = a.outer_rank - 1; k >= 0; --k) {
    int64_t n = a.outer_shape[k];
    int64_t q = row / n;
    int64_t c = row - q * n;
    row = q;
    d += c * a.d_outer[k];
    s += c * a.s_outer[k];
  }
  *d_base = d;
  *s_base = s;
}

// Index arithmetic runs in I (int32_t when every address of both operands fits
// in 31 bits, the common case: ph-core caps element counts at Int32::MAX), and
// a unit innermost stride is a compile-time constant (DCONT / SCONT), so the
// per-element work is one add and one address computation.
template <typename E, int EPT, typename I, bool DCONT, bool SCONT, bool STREAM>
__global__ __launch_bounds__(kBlock) void k_copy_rows(E *__restrict__ dst,
                                                      const E *__restrict__ src, RowArgs a) {
  constexpr int64_t kTile = (int64_t)kBlock * EPT;
  const I cols = (I)a.cols;
  const I di = (I)a.d_inner, si = (I)a.s_inner;
  for (int64_t b = blockIdx.x; b < a.nblocks; b += gridDim.x) {
    const int64_t row = b / a.ntiles;
    const int64_t tile = b - row * a.ntiles;
    int64_t db64, sb64;
    decode_row(a, row, &db64, &sb64);
    const I db = (I)db64, sb = (I)sb64;
    const I c0 = (I)(tile * kTile) + (I)threadIdx.x;
    E v[EPT];
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      const I c = c0 + (I)(e * kBlock);
      if (c < cols) v[e] = src[sb + (SCONT ? c : c * si)];
    }
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      const I c = c0 + (I)(e * kBlock);
      if (c < cols) {
        E *p = dst + db + (DCONT ? c : c * di);
        if constexpr (STREAM) __builtin_nontemporal_store(v[e], p);
        else *p = v[e];
      }
    }
  }
}

template <typename E, int EPT, typename I, bool DCONT>
__global__ __launch_bounds__(kBlock) void k_fill_rows(E *__restrict__ dst, E value, RowArgs a) {
  constexpr int64_t kTile = (int64_t)kBlock * EPT;
  const I cols = (I)a.cols;
  const I di = (I)a.d_inner;
  for (int64_t b = blockIdx.x; b < a.nblocks; b += gridDim.x) {
    const int64_t row = b / a.ntiles;
    const int64_t tile = b - row * a.ntiles;
    int64_t db64, sb64;
    decode_row(a, row, &db64, &sb64);
    const I db = (I)db64;
    const I c0 = (I)(tile * kTile) + (I)threadIdx.x;
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      const I c = c0 + (I)(e * kBlock);
      if (c < cols) dst[db + (DCONT ? c : c * di)] = value;
    }
  }
}

// Stores that bypass the caches are for destinations of more than kStreamBytes,
// which would only push each other out of the 256 MB MALL; a smaller result
// stays there for the kernel that reads it next.  Both ways, 8192^2 Int32: the
// transposing copy 79 us streamed, 110 not; the gather of a strided view and
// the fill+scatter that reads it 92 us streamed, 71 not (45 MB between them).
// (Of a loop that gathers alone, a smaller source then stays there in
// the destination's place: 5000^2 through every other column, 27 us streamed and
// 32 not for Int32, 44 and 50 for Float64; with a sum of the result after each
// gather 53 and 50, 87 and 82.)
// The choice is a template argument: of a run-time one the compiler makes a
// single store that is not streamed.
bool streams(int64_t bytes) { return bytes > kStreamBytes; }

// Both operands' addresses fit in 31 bits: [min, max] of every reachable
// index (the descriptors were validated against [0, extent)).
bool fits_i32(const ph_view_desc *a, const ph_view_desc *b) {
  return a->extent < (int64_t(1) << 31) && (!b || b->extent < (int64_t(1) << 31));
}

// Narrow rows (cols small): one element per thread, grid-stride, full decode.
template <typename E>
__global__ __launch_bounds__(kBlock) void k_copy_flat(E *__restrict__ dst,
                                                      const E *__restrict__ src, RowArgs a,
                                                      int64_t total, int has_src, E value) {
  for (int64_t g = (int64_t)blockIdx.x * kBlock + threadIdx.x; g < total;
       g += (int64_t)gridDim.x * kBlock) {
    const int64_t row = g / a.cols;
    const int64_t c = g - row * a.cols;
    int64_t db, sb;
    decode_row(a, row, &db, &sb);
    dst[db + c * a.d_inner] = has_src ? src[sb + c * a.s_inner] : value;
  }
}

// Granlund-Montgomery round-up divisor for 32-bit unsigned n < 2^32:
// l = ceil(log2 d), m = floor(2^32 (2^l - d) / d) + 1.
void magic_u32(uint32_t d, uint32_t *m, uint32_t *l) {
  uint32_t s = 0;
  while ((uint64_t(1) << s) < d) ++s;
  *l = s;
  *m = (uint32_t)(((uint64_t(1) << 32) * ((uint64_t(1) << s) - d)) / d + 1);
}

// 32-bit division by a run-time constant.
struct Div32 {
  uint32_t d, m, l;
};
__device__ __forceinline__ uint32_t div32(uint32_t n, const Div32 &v) {
  return (uint32_t)(((uint64_t)__umulhi(n, v.m) + n) >> v.l);
}

// Rows contiguous on both sides (a trimmed border, a slab of a concatenation,
// permuted outer axes), numbered through all rows: a lane takes 16 bytes of
// consecutive elements in lexicographic order, whichever row they fall in, so
// short and odd rows fill the lanes as long ones do.  A vector that crosses a
// row's end is copied element by element.  Vectors need element alignment
// only.  HBM-bound; the kernel that owned columns of one row (k_copy_rows) or,
// for short rows, one element per lane with 64-bit divisions took 26 us for a
// trimmed 6007 x 4001 BFloat16 (now 16), 33 for Int32 (28), 397 for
// [257, 1023, 515] Float32 permuted (1, 0, 2) (202).
struct FlatArgs {
  uint32_t total;   // elements
  Div32 cols;       // the innermost extent
  int32_t orank, s_inner;  // outer axes; source stride +1 or -1
  int32_t stream;          // every row of the destination is aligned: stores bypass the caches
  int32_t d_off, s_off;
  Div32 on[PH_MAX_RANK];   // outer extents
  int32_t o_d[PH_MAX_RANK], o_s[PH_MAX_RANK];
};

__device__ __forceinline__ void flat_row(const FlatArgs &a, uint32_t row, int32_t *d, int32_t *s) {
  *d = a.d_off;
  *s = a.s_off;
  for (int k = a.orank - 1; k > 0; --k) {
    const uint32_t q = div32(row, a.on[k]);
    const int32_t c = (int32_t)(row - q * a.on[k].d);
    row = q;
    *d += c * a.o_d[k];
    *s += c * a.o_s[k];
  }
  *d += (int32_t)row * a.o_d[0];
  *s += (int32_t)row * a.o_s[0];
}

template <typename E>
using Word = typename std::conditional<sizeof(E) == 8, uint64_t, uint32_t>::type;

template <typename E, int G, bool STREAM>
__global__ __launch_bounds__(kBlock) void k_copy_flat_vec(E *__restrict__ dst, const E *__restrict__ src, FlatArgs a) {
  constexpr uint32_t VW = 16 / sizeof(E);
  typedef E V __attribute__((ext_vector_type(VW)));
  typedef E VU __attribute__((ext_vector_type(VW), aligned(sizeof(E))));
  VU v[G];
  int32_t to[G];  // destination of a whole vector, -1: copied element by element
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const uint32_t i = ((blockIdx.x * (uint32_t)G + g) * kBlock + threadIdx.x) * VW;
    to[g] = -1;
    if (i >= a.total) continue;
    const uint32_t row = div32(i, a.cols), c = i - row * a.cols.d;
    int32_t d, s;
    flat_row(a, row, &d, &s);
    if (c + VW <= a.cols.d) {
      to[g] = d + (int32_t)c;
      if (a.s_inner > 0) {
        v[g] = *(const VU *)(src + s + (int32_t)c);
      } else {
        const VU w = *(const VU *)(src + s - (int32_t)(c + VW - 1));
#pragma unroll
        for (uint32_t k = 0; k < VW; ++k) v[g][k] = w[VW - 1 - k];
      }
    } else {
      // The part in row `row` and the part in the next row (rows of VW
      // elements or more; shorter ones step through their rows).  All loads
      // come before the stores, each into a register of its own: loads into
      // halves of one register would wait for each other.
      Word<E> t[VW];
      int32_t at[VW];
      int32_t d1 = d, s1 = s;
      const bool one = a.cols.d >= VW;
      if (one && i + (a.cols.d - c) < a.total) flat_row(a, row + 1, &d1, &s1);
      uint32_t r = row, cc = c;
#pragma unroll
      for (uint32_t k = 0; k < VW; ++k) {
        const bool in = i + k < a.total;
        if (cc == a.cols.d) {
          cc = 0;
          ++r;
          if (one) {
            d = d1;
            s = s1;
          } else if (in) {
            flat_row(a, r, &d, &s);
          }
        }
        at[k] = in ? d + (int32_t)cc : -1;
        t[k] = src[in ? s + (int32_t)cc * a.s_inner : a.s_off];
        ++cc;
      }
#pragma unroll
      for (uint32_t k = 0; k < VW; ++k)
        if (at[k] >= 0) dst[at[k]] = (E)t[k];
    }
  }
#pragma unroll
  for (int g = 0; g < G; ++g)
    if (to[g] >= 0) {
      if constexpr (STREAM) __builtin_nontemporal_store((V)v[g], (V *)(dst + to[g]));
      else *(VU *)(dst + to[g]) = v[g];
    }
}

// General path: descriptors with reshape/tile stages.  Element g of the
// common logical shape is decoded into a coordinate and mapped through each
// descriptor in full.
__device__ __forceinline__ int64_t map_index(const ph_view_desc &d, const int64_t *coord) {
  int64_t idx = d.view.offset;
  for (int i = 0; i < d.view.rank; ++i) idx += coord[i] * d.view.stride[i];
  for (int s = 0; s < d.nstage; ++s) {
    const ph_affine &st = d.stage[s];
    int64_t out = st.offset;
    for (int j = st.rank - 1; j >= 0; --j) {
      const int64_t n = st.shape[j];
      const int64_t q = idx / n;
      out += (idx - q * n) * st.stride[j];
      idx = q;
    }
    idx = out;
  }
  return idx;
}

template <typename E>
__global__ __launch_bounds__(kBlock) void k_copy_general(E *__restrict__ dst, ph_view_desc dd,
                                                         const E *__restrict__ src,
                                                         ph_view_desc sd, int64_t total,
                                                         int has_src, E value) {
  for (int64_t g = (int64_t)blockIdx.x * kBlock + threadIdx.x; g < total;
       g += (int64_t)gridDim.x * kBlock) {
    int64_t coord[PH_MAX_RANK];
    int64_t r = g;
    for (int i = dd.view.rank - 1; i >= 0; --i) {
      const int64_t n = dd.view.shape[i];
      const int64_t q = r / n;
      coord[i] = r - q * n;
      r = q;
    }
    const int64_t di = map_index(dd, coord);
    dst[di] = has_src ? src[map_index(sd, coord)] : value;
  }
}

// Buffer index of every coordinate of a view, lexicographic: out[g] = d(g).
__global__ __launch_bounds__(kBlock) void k_view_index(int64_t *__restrict__ out, ph_view_desc d, int64_t total) {
  for (int64_t g = (int64_t)blockIdx.x * kBlock + threadIdx.x; g < total; g += (int64_t)gridDim.x * kBlock) {
    int64_t coord[PH_MAX_RANK];
    int64_t r = g;
    for (int i = d.view.rank - 1; i >= 0; --i) {
      const int64_t n = d.view.shape[i];
      const int64_t q = r / n;
      coord[i] = r - q * n;
      r = q;
    }
    out[g] = map_index(d, coord);
  }
}

// Transposing copy through LDS: the source is contiguous along axis A and the
// destination along another axis B (a permuted view materialised, or a
// contiguous array scattered into a permuted MutableView).  A workgroup owns
// a TA x TB tile of (A, B) for one coordinate of the other axes.  A lane loads
// blocks of VW x VW elements (VW consecutive source rows of VW consecutive A
// elements: 16-byte loads, 8 and 4 bytes for 2- and 1-byte elements),
// transposes them in registers and stores VW vectors along B into LDS [A][B].
// The vector index within an LDS row is XOR-swizzled by (a / VW), so the lanes
// of a store and of the read that follows touch distinct banks.  The tile
// leaves LDS as vectors along B.  Either side moves runs of a tile's edge (256
// bytes in 64 x 64 tiles of 4-byte elements), every element read once and written
// once; vectors need element alignment only, so odd extents and row pitches
// run the same way, with single elements where a vector crosses the edge.
//
// What bounds it is HBM and, at odd pitches, the cache lines that neighbouring
// tiles share: a line written half by one XCD and half by another goes to
// memory twice.  So tiles are numbered for one XCD's L2 to see both halves:
// each XCD takes an eighth of the tiles in order (along A first).  On grids of
// 32 tiles or more both ways and over 20 million elements that made the XCDs
// start in step on pitches near a power of two (8192^2 Float64: 267 us, 246 in
// plain order); those deal patches of 2 x 8 tiles to the XCDs in turn (204).
// Vectors and numbering together, against single elements in plain order:
// [257, 1023, 515] Float32 permuted (2, 0, 1) 385 -> 221 us (4.9 TB/s),
// 4096 x 4100 27 -> 21, 8192^2 89 -> 80, 8193 x 8195 140 -> 117 (8191 x 8189, whose
// pitch falls the other way, 108 -> 115; patches of 8 x 2: 129 and 108); BFloat16
// 8192^2 82 -> 45.  Tiles of 64 x 64 measured
// as well as 128 x 128 or better (small arrays: 4.5 us against 7.7); a side of
// at most kNarrow elements takes tiles of 32 by 512 (8-byte: 128) instead
// ([1000, 2000, 24] Float32 (0, 2, 1): 204 -> 79 us).  8-byte copies take smaller
// tiles while 64 x 64 are too few for the CUs: 32 x 32 below 700000 elements, 32
// along A by 64 below 3 million (Float64, in 32 x 32, 32 x 64 and 64 x 64: 800 x 801
// 4.3, 4.5 and 5.1 us, 1023 x 1025 5.4, 5.2 and 5.9, 1600 x 1601 8.4, 7.5 and 8.8,
// 2000 x 1800 11.0, 10.6 and 10.3).
struct TileArgs {
  int64_t na, nb;    // extents along A and B
  uint32_t ta, tb;   // tiles along A and B
  int64_t nblocks;   // tiles in all
  int64_t per_xcd;   // tiles per XCD, or 0: patches of pa x pb tiles
  uint32_t pa, pb, npa, npb;  // (npa x npb patches a plane)
  int64_t s_a, s_b;  // source strides along A (+-1) and B
  int64_t d_a, d_b;  // destination strides along A and B (+-1)
  int64_t d_off, s_off;
  int32_t orank, stream;  // stream: the stores bypass the caches (aligned runs)
  int64_t o_shape[PH_MAX_RANK], o_dst[PH_MAX_RANK], o_src[PH_MAX_RANK];
};

constexpr int64_t kNarrow = 48;
// Sides shorter than 16 take a tile from 8 on where that measured faster than
// copying row by row: along A for 4- and 8-byte elements ([1000, 2000, 9] to
// (2, 0, 1): Float32 102 -> 59 us, Float64 205 -> 77, 2-byte 50 -> 62), along B
// up to 4 bytes ([9, 1000, 2000] to (1, 2, 0): 51 -> 45, Float64 78 -> 87).
constexpr int64_t tile_min_a(int esize) { return esize >= 4 ? 8 : 16; }
constexpr int64_t tile_min_b(int esize) { return esize <= 4 ? 8 : 16; }

template <typename E>
constexpr int tile_vec() { return sizeof(E) == 8 ? 2 : 4; }

template <typename E, int TA, int TB, bool STREAM>
__global__ __launch_bounds__(kBlock) void k_copy_tiled(E *__restrict__ dst, const E *__restrict__ src, TileArgs a) {
  constexpr int VW = tile_vec<E>();
  constexpr int GA = TA / VW, GB = TB / VW;  // vectors along A and B
  constexpr int NB = GA * GB / kBlock;       // blocks a lane loads
  constexpr int NW = TA * GB / kBlock;       // vectors a lane writes
  constexpr int kBankVecs = 128 / (VW * (int)sizeof(E));
  constexpr int kSwz = (GB < kBankVecs ? GB : kBankVecs) - 1;
  typedef E V __attribute__((ext_vector_type(VW)));
  typedef E VU __attribute__((ext_vector_type(VW), aligned(sizeof(E))));
  __shared__ __align__(16) E lds[TA * TB];  // [A][B]
  const int t = threadIdx.x;
  const uint32_t per = a.ta * a.tb;
  const uint32_t xcd = blockIdx.x & 7;  // workgroups are dealt to the XCDs in turn
  for (int64_t b = blockIdx.x >> 3;; b += gridDim.x >> 3) {
    // slot b of this XCD -> plane o, tile (ia, ib); every condition is
    // uniform over the workgroup
    int64_t o;
    uint32_t ia, ib;
    if (a.per_xcd) {
      const int64_t tile = xcd * a.per_xcd + b;
      if (b >= a.per_xcd || tile >= a.nblocks) break;
      o = tile < 0xffffffffll ? (uint32_t)tile / per : tile / per;
      const uint32_t rem = (uint32_t)(tile - o * per);
      ib = rem / a.ta;
      ia = rem - ib * a.ta;
    } else {
      const uint32_t pt = a.pa * a.pb, np = a.npa * a.npb;  // (16, and fewer than 2^32 patches in all)
      const uint32_t patch = (uint32_t)b / pt * 8 + xcd, w = (uint32_t)b % pt;
      o = patch / np;
      if (o * per >= a.nblocks) break;
      const uint32_t rem = patch - (uint32_t)o * np;
      const uint32_t jb = rem / a.npa, wb = w / a.pa;
      ia = (rem - jb * a.npa) * a.pa + (w - wb * a.pa);
      ib = jb * a.pb + wb;
      if (ia >= a.ta || ib >= a.tb) continue;
    }
    const int64_t a0 = (int64_t)ia * TA, b0 = (int64_t)ib * TB;
    int64_t db = a.d_off + a0 * a.d_a + b0 * a.d_b, sb = a.s_off + a0 * a.s_a + b0 * a.s_b;
    for (int k = a.orank - 1; k >= 0; --k) {
      const int64_t n = a.o_shape[k];
      const int64_t q = o / n;
      const int64_t c = o - q * n;
      o = q;
      db += c * a.o_dst[k];
      sb += c * a.o_src[k];
    }
    const int la = (int)(a.na - a0 < TA ? a.na - a0 : TA), lb_ = (int)(a.nb - b0 < TB ? a.nb - b0 : TB);
    V v[NB][VW];
#pragma unroll
    for (int m = 0; m < NB; ++m) {
      const int idx = t + kBlock * m, qa = idx % GA, rb = idx / GA;
#pragma unroll
      for (int j = 0; j < VW; ++j) {
        const int br = VW * rb + j;
        v[m][j] = V{};
        if (br >= lb_) continue;
        const E *p = src + sb + br * a.s_b + (int64_t)(VW * qa) * a.s_a;
        if (VW * qa + VW <= la) {
          const V w = *(const VU *)(a.s_a > 0 ? p : p - (VW - 1));
          if (a.s_a > 0) v[m][j] = w;
          else
#pragma unroll
            for (int i = 0; i < VW; ++i) v[m][j][i] = w[VW - 1 - i];
        } else {
#pragma unroll
          for (int i = 0; i < VW; ++i)
            if (VW * qa + i < la) v[m][j][i] = p[i * a.s_a];
        }
      }
    }
#pragma unroll
    for (int m = 0; m < NB; ++m) {
      const int idx = t + kBlock * m, qa = idx % GA, rb = idx / GA;
#pragma unroll
      for (int i = 0; i < VW; ++i) {
        V w;
#pragma unroll
        for (int j = 0; j < VW; ++j) w[j] = v[m][j][i];
        *(V *)&lds[(VW * qa + i) * TB + (rb ^ (qa & kSwz)) * VW] = w;
      }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NW; ++j) {
      const int idx = t + kBlock * j, q = idx % GB, al = idx / GB;
      if (al >= la || VW * q >= lb_) continue;
      V w = *(const V *)&lds[al * TB + (q ^ ((al / VW) & kSwz)) * VW];
      E *p = dst + db + al * a.d_a + (int64_t)(VW * q) * a.d_b;
      if (VW * q + VW <= lb_) {
        if (a.d_b < 0) {
          const V r = w;
#pragma unroll
          for (int i = 0; i < VW; ++i) w[i] = r[VW - 1 - i];
          p -= VW - 1;
        }
        if constexpr (STREAM) __builtin_nontemporal_store(w, (V *)p);
        else *(VU *)p = w;
      } else {
#pragma unroll
        for (int i = 0; i < VW; ++i)
          if (VW * q + i < lb_) p[i * a.d_b] = w[i];
      }
    }
    __syncthreads();  // the next tile reuses the LDS
  }
}

// Whether every vector of the destination starts on a vector boundary.
bool tiled_aligned(const TileArgs &t, const void *dst, int esize, int vw) {
  const int64_t vb = (int64_t)vw * esize;
  auto al = [&](int64_t elems) { return (elems * esize) % vb == 0; };
  if (t.d_b != 1 || (uintptr_t)dst % vb != 0 || !al(t.d_off) || !al(t.d_a)) return false;
  for (int k = 0; k < t.orank; ++k)
    if (!al(t.o_dst[k])) return false;
  return true;
}

// The (A, B) axes of a transposing copy over the collapsed layout (operand 0
// the destination, 1 the source), or false when the innermost axis already
// serves both operands or either operand has no unit-stride axis.  Both
// extents must fill a good part of a tile.
bool tiled_axes(const ph::Layout &L, int esize, int *A, int *B) {
  if (L.rank < 2) return false;
  auto unit = [](int64_t s) { return s == 1 || s == -1; };
  const int q = L.rank - 1;
  if (unit(L.stride[0][q]) && unit(L.stride[1][q])) return false;
  *A = *B = -1;
  for (int k = 0; k < L.rank; ++k) {
    if (unit(L.stride[1][k]) && *A < 0) *A = k;
    if (unit(L.stride[0][k]) && *B < 0) *B = k;
  }
  return *A >= 0 && *B >= 0 && *A != *B && L.shape[*A] >= tile_min_a(esize) && L.shape[*B] >= tile_min_b(esize);
}

void make_tile_args(const ph::Layout &L, int A, int B, int tile_a, int tile_b, TileArgs *t) {
  std::memset(t, 0, sizeof(*t));
  t->na = L.shape[A];
  t->nb = L.shape[B];
  t->ta = (uint32_t)((t->na + tile_a - 1) / tile_a);
  t->tb = (uint32_t)((t->nb + tile_b - 1) / tile_b);
  t->s_a = L.stride[1][A];
  t->s_b = L.stride[1][B];
  t->d_a = L.stride[0][A];
  t->d_b = L.stride[0][B];
  t->d_off = L.offset[0];
  t->s_off = L.offset[1];
  int64_t others = 1;
  for (int k = 0; k < L.rank; ++k) {
    if (k == A || k == B) continue;
    t->o_shape[t->orank] = L.shape[k];
    t->o_dst[t->orank] = L.stride[0][k];
    t->o_src[t->orank] = L.stride[1][k];
    ++t->orank;
    others *= L.shape[k];
  }
  t->nblocks = others * t->ta * t->tb;
}

int64_t grid_for(int64_t blocks) {
  const int64_t cap = 1 << 20;
  return blocks < 1 ? 1 : (blocks > cap ? cap : blocks);
}

void make_row_args(const ph::Layout &L, int d_op, int s_op, int ept, RowArgs *a) {
  std::memset(a, 0, sizeof(*a));
  if (L.rank == 0) {
    a->rows = 1;
    a->cols = 1;
    a->d_off = L.offset[d_op];
    a->s_off = s_op >= 0 ? L.offset[s_op] : 0;
  } else {
    a->cols = L.shape[L.rank - 1];
    a->d_inner = L.stride[d_op][L.rank - 1];
    a->s_inner = s_op >= 0 ? L.stride[s_op][L.rank - 1] : 0;
    a->outer_rank = L.rank - 1;
    a->rows = 1;
    for (int k = 0; k < L.rank - 1; ++k) {
      a->outer_shape[k] = L.shape[k];
      a->rows *= L.shape[k];
      a->d_outer[k] = L.stride[d_op][k];
      a->s_outer[k] = s_op >= 0 ? L.stride[s_op][k] : 0;
    }
    a->d_off = L.offset[d_op];
    a->s_off = s_op >= 0 ? L.offset[s_op] : 0;
  }
  const int64_t tile = (int64_t)kBlock * ept;
  a->ntiles = (a->cols + tile - 1) / tile;
  a->nblocks = a->rows * a->ntiles;
}

Div32 make_div(int64_t d) {
  Div32 v{(uint32_t)d, 0, 0};
  magic_u32(v.d, &v.m, &v.l);
  return v;
}

// Whether k_copy_flat_vec takes a copy: rows contiguous on both sides (the
// source also backwards), and 31-bit addresses.
bool flat_rows(const ph::Layout &L, const ph_view_desc *dd, const ph_view_desc *sd, int esize) {
  if (L.rank < 1 || !fits_i32(dd, sd) || ph::layout_count(L) > INT32_MAX) return false;
  const int q = L.rank - 1;
  if (L.stride[0][q] != 1 || (L.stride[1][q] != 1 && L.stride[1][q] != -1)) return false;
  // Long rows of 8-byte elements into a strided destination: a wavefront's
  // single elements already fill whole lines (rows of 4001 Float64 into a
  // larger array: 60 us against 69).
  return esize < 8 || L.shape[q] < 512 || L.rank == 1 || L.stride[0][q - 1] == L.shape[q];
}

void make_flat_args(const ph::Layout &L, const void *dst, int64_t d_extent, int esize, FlatArgs *f) {
  std::memset(f, 0, sizeof(*f));
  const int q = L.rank - 1;
  f->total = (uint32_t)ph::layout_count(L);
  f->cols = make_div(L.shape[q]);
  f->s_inner = (int32_t)L.stride[1][q];
  f->d_off = (int32_t)L.offset[0];
  f->s_off = (int32_t)L.offset[1];
  f->orank = q;
  for (int k = 0; k < q; ++k) {
    f->on[k] = make_div(L.shape[k]);
    f->o_d[k] = (int32_t)L.stride[0][k];
    f->o_s[k] = (int32_t)L.stride[1][k];
  }
  // (one run from end to end, or rows that all start on 16 bytes)
  bool run = true, rows = L.shape[q] * esize % 16 == 0;
  int64_t n = 1;
  for (int k = q; k >= 0; --k) {
    run = run && L.stride[0][k] == n;
    rows = rows && (k == q || L.stride[0][k] * esize % 16 == 0);
    n *= L.shape[k];
  }
  f->stream = streams(d_extent * esize) && (int64_t)f->total * esize >= (int64_t(4) << 20) && ((uintptr_t)dst + (uintptr_t)(L.offset[0] * esize)) % 16 == 0 && (run || rows);
}

template <typename E, int TA, int TB>
int launch_tile(const ph::Layout &L, int A, int B, void *dst, int64_t d_extent, const void *src) {
  TileArgs t;
  make_tile_args(L, A, B, TA, TB, &t);
  if ((t.na + TA - 1) / TA * ((t.nb + TB - 1) / TB) >= (int64_t(1) << 31)) return ph::set_error(PH_E_UNSUPPORTED, "copy of too many tiles");
  t.stream = streams(d_extent * (int64_t)sizeof(E)) && tiled_aligned(t, dst, (int)sizeof(E), tile_vec<E>());
  int64_t slots;  // per XCD
  if (t.ta >= 32 && t.tb >= 32 && ph::layout_count(L) > 20000000) {
    t.pa = 2;
    t.pb = 8;
    t.npa = (t.ta + t.pa - 1) / t.pa;
    t.npb = (t.tb + t.pb - 1) / t.pb;
    const int64_t patches = t.nblocks / ((int64_t)t.ta * t.tb) * t.npa * t.npb;
    slots = (patches + 7) / 8 * t.pa * t.pb;
  } else {
    slots = t.per_xcd = (t.nblocks + 7) / 8;
  }
  const int64_t grid = 8 * std::min<int64_t>(slots, int64_t(1) << 17);
  if (t.stream)
    hipLaunchKernelGGL((k_copy_tiled<E, TA, TB, true>), dim3((unsigned)grid), dim3(kBlock), 0, ph::stream(), (E *)dst,
                       (const E *)src, t);
  else
    hipLaunchKernelGGL((k_copy_tiled<E, TA, TB, false>), dim3((unsigned)grid), dim3(kBlock), 0, ph::stream(), (E *)dst,
                       (const E *)src, t);
  return ph::check_launch("k_copy_tiled");
}

template <typename E>
int launch_tiled(const ph::Layout &L, int A, int B, void *dst, int64_t d_extent, const void *src) {
  constexpr int W = sizeof(E) == 8 ? 128 : 512;
  if (L.shape[A] <= kNarrow) return launch_tile<E, 32, W>(L, A, B, dst, d_extent, src);
  if (L.shape[B] <= kNarrow) return launch_tile<E, W, 32>(L, A, B, dst, d_extent, src);
  if constexpr (sizeof(E) == 8) {
    if (ph::layout_count(L) < 700000) return launch_tile<E, 32, 32>(L, A, B, dst, d_extent, src);
    if (ph::layout_count(L) < 3000000) return launch_tile<E, 32, 64>(L, A, B, dst, d_extent, src);
  }
  return launch_tile<E, 64, 64>(L, A, B, dst, d_extent, src);
}

template <typename E>
int launch_copy(void *dst, const ph_view_desc *dd, const void *src, const ph_view_desc *sd,
                const void *value_bits) {
  E value{};
  if (value_bits) std::memcpy(&value, value_bits, sizeof(E));
  const int64_t total = ph::desc_count(dd);
  if (total == 0) return PH_OK;
  int rc = ph::launch_gate("strided copy");
  if (rc) return rc;
  hipStream_t st = ph::stream();
  const bool staged = dd->nstage > 0 || (src && sd->nstage > 0);
  if (staged) {
    const ph_view_desc &s_desc = src ? *sd : *dd;
    hipLaunchKernelGGL(k_copy_general<E>, dim3((unsigned)grid_for((total + kBlock - 1) / kBlock)),
                       dim3(kBlock), 0, st, (E *)dst, *dd, (const E *)src, s_desc, total,
                       src ? 1 : 0, value);
    return ph::check_launch("k_copy_general");
  }
  const ph_view_desc *descs[2] = {dd, src ? sd : dd};
  ph::Layout L;
  ph::collapse(descs, 2, &L);
  constexpr int EPT = sizeof(E) >= 8 ? 4 : 8;
  int ax_a, ax_b;
  if (src && tiled_axes(L, (int)sizeof(E), &ax_a, &ax_b)) {
    return launch_tiled<E>(L, ax_a, ax_b, dst, dd->extent, src);
  }
  if (src && flat_rows(L, dd, sd, (int)sizeof(E))) {
    FlatArgs f;
    make_flat_args(L, dst, dd->extent, (int)sizeof(E), &f);
    // two vectors a lane, one where that leaves few workgroups
    const int g = total * (int64_t)sizeof(E) < (int64_t(4) << 20) ? 1 : 2;
    const uint32_t per = kBlock * g * (16 / sizeof(E));
    const dim3 grid((f.total + per - 1) / per);
    if (f.stream)
      hipLaunchKernelGGL((k_copy_flat_vec<E, 2, true>), grid, dim3(kBlock), 0, st, (E *)dst, (const E *)src, f);
    else if (g == 2)
      hipLaunchKernelGGL((k_copy_flat_vec<E, 2, false>), grid, dim3(kBlock), 0, st, (E *)dst, (const E *)src, f);
    else
      hipLaunchKernelGGL((k_copy_flat_vec<E, 1, false>), grid, dim3(kBlock), 0, st, (E *)dst, (const E *)src, f);
    return ph::check_launch("k_copy_flat_vec");
  }
  RowArgs a;
  make_row_args(L, 0, src ? 1 : -1, EPT, &a);
  if (a.cols * 4 < (int64_t)kBlock * EPT && a.rows > 1) {
    hipLaunchKernelGGL(k_copy_flat<E>, dim3((unsigned)grid_for((total + kBlock - 1) / kBlock)),
                       dim3(kBlock), 0, st, (E *)dst, (const E *)src, a, total, src ? 1 : 0,
                       value);
    return ph::check_launch("k_copy_flat");
  }
  const dim3 grid((unsigned)grid_for(a.nblocks)), block(kBlock);
  const bool small = fits_i32(dd, src ? sd : nullptr);
  const bool dc = a.d_inner == 1, sc = a.s_inner == 1;
  if (src) {
#define PH_COPY_LAUNCH(I, D, S, NT) \
  hipLaunchKernelGGL((k_copy_rows<E, EPT, I, D, S, NT>), grid, block, 0, st, (E *)dst, (const E *)src, a)
    const bool nt = streams(dd->extent * (int64_t)sizeof(E));
    if (small) {
      constexpr bool both = sizeof(E) == 8;  // (flat_rows takes contiguous rows of smaller elements)
      if (both && dc && sc && nt) PH_COPY_LAUNCH(int32_t, true, both, true);
      else if (both && dc && sc) PH_COPY_LAUNCH(int32_t, true, both, false);
      else if (dc && nt) PH_COPY_LAUNCH(int32_t, true, false, true);
      else if (dc) PH_COPY_LAUNCH(int32_t, true, false, false);
      else if (sc) PH_COPY_LAUNCH(int32_t, false, true, false);
      else PH_COPY_LAUNCH(int32_t, false, false, false);
    } else {
      PH_COPY_LAUNCH(int64_t, false, false, false);
    }
#undef PH_COPY_LAUNCH
    return ph::check_launch("k_copy_rows");
  }
  if (small && dc)
    hipLaunchKernelGGL((k_fill_rows<E, EPT, int32_t, true>), grid, block, 0, st, (E *)dst, value, a);
  else if (small)
    hipLaunchKernelGGL((k_fill_rows<E, EPT, int32_t, false>), grid, block, 0, st, (E *)dst, value, a);
  else
    hipLaunchKernelGGL((k_fill_rows<E, EPT, int64_t, false>), grid, block, 0, st, (E *)dst, value, a);
  return ph::check_launch("k_fill_rows");
}

int dispatch_copy(void *dst, const ph_view_desc *dd, const void *src, const ph_view_desc *sd,
                  const void *value) {
  switch (ph::dtype_size(dd->dtype)) {
    case 1: return launch_copy<uint8_t>(dst, dd, src, sd, value);
    case 2: return launch_copy<uint16_t>(dst, dd, src, sd, value);
    case 4: return launch_copy<uint32_t>(dst, dd, src, sd, value);
    case 8: return launch_copy<uint64_t>(dst, dd, src, sd, value);
  }
  return ph::set_error(PH_E_ARGUMENT, "unsupported dtype %d", dd->dtype);
}

// ---------------------------------------------------------------------------
// Fused fill + scatter over a whole row-major destination buffer.
// ---------------------------------------------------------------------------
struct FillScatterArgs {
  int32_t rank;        // destination rank
  int32_t last_axis;   // view axis of the innermost destination axis, -1 fixed
  int64_t cols;        // innermost destination extent
  int64_t rows;        // product of the outer destination extents
  int64_t ntiles, nblocks;
  int64_t shape[PH_MAX_RANK];
  int64_t first[PH_MAX_RANK];
  int64_t step[PH_MAX_RANK];
  int64_t count[PH_MAX_RANK];
  int32_t axis[PH_MAX_RANK];
  int64_t src_stride[PH_MAX_RANK];  // per view axis
  int64_t src_off;
  // innermost axis: member iff (c - first) = q*step, 0 <= q < count
  int64_t in_first, in_step, in_count, in_src_stride;
};

// A lane owns 16 bytes of the flat destination, whichever rows they fall in, so
// every store is whole and aligned for any row length; all divisions are
// 32-bit.  A vector inside one row of a unit-step region loads its source as a
// vector.  HBM-bound; two vectors per lane: the gather and fill+scatter of
// 8192^2 Int32 through 1..3..-1, ..-2.. take 71 us with one, 74 with two and 79
// with four, a fill+scatter through ..2.. columns 70, 57 and 57.  The kernels before it owned 16 bytes of one row, four a
// lane, and took rows that are not whole vectors element by element with
// 64-bit divisions: 8192^2 Int32 50 us (now 40), 6007 x 4001 BFloat16 49 (18),
// 200000 x 33 Int32 304 (20).
constexpr int kScatterVecs = 2;

struct FlatScatterArgs {
  uint32_t total;
  Div32 cols;
  int32_t rank, src_off;
  int32_t vec_src;  // the innermost step and source stride are 1
  Div32 shape[PH_MAX_RANK], step[PH_MAX_RANK];  // |step|
  int32_t first[PH_MAX_RANK], sign[PH_MAX_RANK], src_stride[PH_MAX_RANK];  // sign 0: fixed axis
  uint32_t count[PH_MAX_RANK];
};

// coordinate x of axis k: whether it is in the region, and its index there
__device__ __forceinline__ bool fs_axis(const FlatScatterArgs &a, int k, uint32_t x, uint32_t *j) {
  int32_t u = (int32_t)x - a.first[k];
  if (a.sign[k] < 0) u = -u;
  const uint32_t q = div32((uint32_t)u, a.step[k]);
  *j = q;
  return u >= 0 && q * a.step[k].d == (uint32_t)u && q < a.count[k];
}

__device__ __forceinline__ bool fs_flat_row(const FlatScatterArgs &a, uint32_t row, int32_t *soff) {
  bool in = true;
  int32_t s = a.src_off;
  for (int k = a.rank - 2; k >= 0; --k) {
    const uint32_t q = div32(row, a.shape[k]);
    uint32_t j;
    in = fs_axis(a, k, row - q * a.shape[k].d, &j) && in;
    s += (int32_t)j * a.src_stride[k];
    row = q;
  }
  *soff = s;
  return in;
}

template <typename E>
__global__ __launch_bounds__(kBlock) void k_fill_scatter_flat(E *__restrict__ dst, const E *__restrict__ src,
                                                              FlatScatterArgs a, E fill) {
  constexpr uint32_t VW = 16 / sizeof(E);
  typedef E V __attribute__((ext_vector_type(VW)));
  typedef E VU __attribute__((ext_vector_type(VW), aligned(sizeof(E))));
  const int in = a.rank - 1;
  Word<E> v[kScatterVecs][VW];  // (one register an element, or the loads of a vector wait for each other)
#pragma unroll
  for (int g = 0; g < kScatterVecs; ++g) {
    const uint32_t i = ((blockIdx.x * (uint32_t)kScatterVecs + g) * kBlock + threadIdx.x) * VW;
#pragma unroll
    for (uint32_t k = 0; k < VW; ++k) v[g][k] = fill;
    if (i >= a.total) continue;
    uint32_t row = div32(i, a.cols), c = i - row * a.cols.d;
    int32_t soff;
    bool member = fs_flat_row(a, row, &soff);
    if (c + VW <= a.cols.d) {
      if (!member) continue;
      const int32_t rel = (int32_t)c - a.first[in];
      if (a.vec_src && rel >= 0 && (uint32_t)rel + VW <= a.count[in]) {
        const VU w = *(const VU *)(src + soff + rel);
#pragma unroll
        for (uint32_t k = 0; k < VW; ++k) v[g][k] = w[k];
        continue;
      }
#pragma unroll
      for (uint32_t k = 0; k < VW; ++k) {
        uint32_t j;
        if (fs_axis(a, in, c + k, &j)) v[g][k] = src[soff + (int32_t)j * a.src_stride[in]];
      }
    } else {  // the vector crosses the end of a row: of one, or of several short ones
      const bool one = a.cols.d >= VW;
      int32_t soff1 = 0;
      const bool member1 = one && i + (a.cols.d - c) < a.total && fs_flat_row(a, row + 1, &soff1);
#pragma unroll
      for (uint32_t k = 0; k < VW; ++k) {
        if (c == a.cols.d) {
          c = 0;
          ++row;
          if (one) {
            member = member1;
            soff = soff1;
          } else {
            member = i + k < a.total && fs_flat_row(a, row, &soff);
          }
        }
        uint32_t j;
        if (fs_axis(a, in, c, &j) && member) v[g][k] = src[soff + (int32_t)j * a.src_stride[in]];
        ++c;
      }
    }
  }
#pragma unroll
  for (int g = 0; g < kScatterVecs; ++g) {
    const uint32_t i = ((blockIdx.x * (uint32_t)kScatterVecs + g) * kBlock + threadIdx.x) * VW;
    V w;
#pragma unroll
    for (uint32_t k = 0; k < VW; ++k) w[k] = (E)v[g][k];
    if (i + VW <= a.total) {
      __builtin_nontemporal_store(w, (V *)(dst + i));
    } else {
#pragma unroll
      for (uint32_t k = 0; k < VW; ++k)
        if (i + k < a.total) dst[i + k] = w[k];
    }
  }
}

template <typename E, int EPT>
__global__ __launch_bounds__(kBlock) void k_fill_scatter(E *__restrict__ dst,
                                                         const E *__restrict__ src,
                                                         FillScatterArgs a, E fill) {
  constexpr int64_t kTile = (int64_t)kBlock * EPT;
  for (int64_t b = blockIdx.x; b < a.nblocks; b += gridDim.x) {
    const int64_t row = b / a.ntiles;
    const int64_t tile = b - row * a.ntiles;
    // decode the outer coordinate; decide row membership (uniform)
    bool member = true;
    int64_t soff = a.src_off;
    int64_t r = row;
    for (int k = a.rank - 2; k >= 0; --k) {
      const int64_t n = a.shape[k];
      const int64_t q = r / n;
      const int64_t x = r - q * n;
      r = q;
      const int64_t rel = x - a.first[k];
      const int64_t st = a.step[k];
      if (a.axis[k] < 0) {
        member = member && (rel == 0);
      } else {
        const int64_t j = rel / st;
        member = member && (j * st == rel) && j >= 0 && j < a.count[k];
        soff += j * a.src_stride[a.axis[k]];
      }
    }
    const int64_t dbase = row * a.cols;
    const int64_t c0 = tile * kTile + threadIdx.x;
    if (!member) {
#pragma unroll
      for (int e = 0; e < EPT; ++e) {
        const int64_t c = c0 + (int64_t)e * kBlock;
        if (c < a.cols) dst[dbase + c] = fill;
      }
      continue;
    }
    E v[EPT];
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      const int64_t c = c0 + (int64_t)e * kBlock;
      v[e] = fill;
      if (c < a.cols) {
        const int64_t rel = c - a.in_first;
        if (a.last_axis < 0) {
          if (rel == 0) v[e] = src[soff];
        } else {
          const int64_t j = rel / a.in_step;
          if (j * a.in_step == rel && j >= 0 && j < a.in_count) v[e] = src[soff + j * a.in_src_stride];
        }
      }
    }
#pragma unroll
    for (int e = 0; e < EPT; ++e) {
      const int64_t c = c0 + (int64_t)e * kBlock;
      if (c < a.cols) dst[dbase + c] = v[e];
    }
  }
}

// The 32-bit form of a fill+scatter, where sizes and alignment allow it.
bool make_flat_scatter(const FillScatterArgs &a, const void *dst, int64_t src_extent, FlatScatterArgs *f) {
  std::memset(f, 0, sizeof(*f));
  if ((uintptr_t)dst % 16 != 0 || src_extent > INT32_MAX || a.rows * a.cols > INT32_MAX - 65536) return false;
  f->total = (uint32_t)(a.rows * a.cols);
  if (f->total == 0) return true;
  f->cols = make_div(a.cols);
  f->rank = a.rank;
  f->src_off = (int32_t)a.src_off;
  for (int k = 0; k < a.rank; ++k) {
    f->shape[k] = make_div(a.shape[k]);
    f->first[k] = (int32_t)a.first[k];
    if (a.axis[k] < 0) {  // a fixed index: a region of one element
      f->step[k] = make_div(1);
      f->sign[k] = 1;
      f->count[k] = 1;
      continue;
    }
    const int64_t st = a.step[k] < 0 ? -a.step[k] : a.step[k];
    if (a.count[k] > INT32_MAX || (a.count[k] > 1 && st > INT32_MAX)) return false;
    f->step[k] = make_div(a.count[k] > 1 ? st : 1);
    f->sign[k] = a.step[k] < 0 ? -1 : 1;
    f->count[k] = (uint32_t)a.count[k];
    f->src_stride[k] = (int32_t)a.src_stride[a.axis[k]];
  }
  const int in = a.rank - 1;
  f->vec_src = a.axis[in] >= 0 && f->sign[in] > 0 && f->step[in].d == 1 && f->src_stride[in] == 1;
  return true;
}

template <typename E>
int launch_fill_scatter(void *dst, FillScatterArgs a, const void *src, int64_t src_extent, const void *fill_bits) {
  E fill{};
  std::memcpy(&fill, fill_bits, sizeof(E));
  constexpr int VEC = 16 / (int)sizeof(E);
  FlatScatterArgs f;
  if (make_flat_scatter(a, dst, src_extent, &f)) {
    const uint32_t per = kBlock * VEC * kScatterVecs;
    if (f.total == 0) return PH_OK;
    int rc = ph::launch_gate("fill scatter");
    if (rc) return rc;
    hipLaunchKernelGGL(k_fill_scatter_flat<E>, dim3((f.total + per - 1) / per), dim3(kBlock), 0, ph::stream(),
                       (E *)dst, (const E *)src, f, fill);
    return ph::check_launch("k_fill_scatter_flat");
  }
  constexpr int EPT = sizeof(E) >= 8 ? 4 : 8;
  const int64_t tile = (int64_t)kBlock * EPT;
  a.ntiles = (a.cols + tile - 1) / tile;
  a.nblocks = a.rows * a.ntiles;
  if (a.nblocks == 0) return PH_OK;
  int rc = ph::launch_gate("fill scatter");
  if (rc) return rc;
  hipLaunchKernelGGL((k_fill_scatter<E, EPT>), dim3((unsigned)grid_for(a.nblocks)), dim3(kBlock),
                     0, ph::stream(), (E *)dst, (const E *)src, a, fill);
  return ph::check_launch("k_fill_scatter");
}

// ---------------------------------------------------------------------------
// Seeded random fill (counter-based splitmix64)
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}
__device__ __forceinline__ uint64_t draw(uint64_t seed, uint64_t k) {
  return mix64(seed + (k + 1) * 0x9E3779B97F4A7C15ULL);
}

__device__ __forceinline__ uint16_t f32_to_bf16_rne(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

__global__ __launch_bounds__(kBlock) void k_random(void *buf, int dtype, int64_t n, uint64_t seed,
                                                   uint64_t offset, int dist, double a, double b) {
  const double two_pi = 6.283185307179586476925286766559;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kBlock) {
    const uint64_t k = offset + (uint64_t)i;
    double x = 0.0;
    int64_t xi = 0;
    if (dist == 0) {
      const uint64_t d = draw(seed, k);
      if (dtype == PH_I32) {
        const int64_t span = (int64_t)(b - a);
        xi = (int64_t)a + (int64_t)((d >> 11) % (uint64_t)span);
      } else {
        const double u = (double)(d >> 11) * 0x1.0p-53;
        x = __dadd_rn(a, __dmul_rn(__dsub_rn(b, a), u));
      }
    } else if (dist == 1) {
      const uint64_t kp = k & ~1ULL;
      const double u1 = (double)(draw(seed, kp) >> 11) * 0x1.0p-53;
      const double u2 = (double)(draw(seed, kp + 1) >> 11) * 0x1.0p-53;
      const double r = sqrt(-2.0 * log(1.0 - u1));
      const double t = __dmul_rn(two_pi, u2);
      const double z = (k & 1) ? __dmul_rn(r, sin(t)) : __dmul_rn(r, cos(t));
      x = __dadd_rn(a, __dmul_rn(b, z));
    } else {
      xi = (int64_t)(draw(seed, k) >> 33);
    }
    switch (dtype) {
      case PH_I32: ((int32_t *)buf)[i] = (int32_t)xi; break;
      case PH_F32: ((float *)buf)[i] = (float)x; break;
      case PH_F64: ((double *)buf)[i] = x; break;
      case PH_BF16: ((uint16_t *)buf)[i] = f32_to_bf16_rne((float)x); break;
    }
  }
}

__global__ void k_clear_i32(int *p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

}  // namespace

int ph::clear_i32(int *p, int n) {
  if (n <= 0) return PH_OK;
  hipLaunchKernelGGL(k_clear_i32, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, ph::stream(), p, n);
  return ph::check_launch("k_clear_i32");
}

extern "C" {

int ph_fill_random(void *buf, int32_t dtype, int64_t n, uint64_t seed, uint64_t offset,
                   int32_t dist, double a, double b) {
  PH_GUARD();
  PH_REQUIRE_INIT();
  if (n <= 0) return PH_OK;
  if (dtype == PH_BOOL || ph::dtype_size(dtype) == 0)
    return ph::set_error(PH_E_ARGUMENT, "ph_fill_random: unsupported dtype %d", dtype);
  if (dist < 0 || dist > 2) return ph::set_error(PH_E_ARGUMENT, "ph_fill_random: dist %d", dist);
  if (dist == 0 && dtype == PH_I32 && !(b > a))
    return ph::set_error(PH_E_ARGUMENT, "ph_fill_random: empty integer range");
  int rc = ph::launch_gate("random");
  if (rc) return rc;
  hipLaunchKernelGGL(k_random, dim3((unsigned)grid_for((n + kBlock - 1) / kBlock)), dim3(kBlock),
                     0, ph::stream(), buf, dtype, n, seed, offset, dist, a, b);
  return ph::check_launch("k_random");
}

int ph_fill(void *buf, const ph_view_desc *dst, const void *value) {
  PH_GUARD();
  PH_REQUIRE_INIT();
  int rc = ph::validate_desc(dst, "fill destination");
  if (rc) return rc;
  if (!value) return ph::set_error(PH_E_ARGUMENT, "ph_fill: null value");
  return dispatch_copy(buf, dst, nullptr, nullptr, value);
}

int ph_strided_copy(void *dst, const ph_view_desc *dd, const void *src, const ph_view_desc *sd,
                    int32_t flags) {
  PH_GUARD();
  PH_REQUIRE_INIT();
  int rc = ph::validate_desc(dd, "copy destination");
  if (rc) return rc;
  rc = ph::validate_desc(sd, "copy source");
  if (rc) return rc;
  if (dd->dtype != sd->dtype && ph::dtype_size(dd->dtype) != ph::dtype_size(sd->dtype))
    return ph::set_error(PH_E_ARGUMENT, "copy between dtypes %d and %d", sd->dtype, dd->dtype);
  if (dd->view.rank != sd->view.rank)
    return ph::set_error(PH_E_SHAPE, "copy between ranks %d and %d", sd->view.rank, dd->view.rank);
  for (int i = 0; i < dd->view.rank; ++i)
    if (dd->view.shape[i] != sd->view.shape[i])
      return ph::set_error(PH_E_SHAPE, "copy shapes differ on axis %d (%lld vs %lld)", i,
                           (long long)sd->view.shape[i], (long long)dd->view.shape[i]);
  if (flags != 0) return ph::set_error(PH_E_ARGUMENT, "ph_strided_copy: unknown flags %d", flags);
  if (ph::desc_count(dd) == 0) return PH_OK;
  const size_t es = ph::dtype_size(dd->dtype);
  if (src == dst) {
    // the reference's order decides what a source reading the destination
    // sees; the parallel kernels below are used when it cannot matter
    bool done = false;
    rc = ph::ordered_copy(dst, dd, src, sd, &done);
    if (rc || done) return rc;
  } else {
    const char *d0 = (const char *)dst, *s0 = (const char *)src;
    if (!(s0 + (size_t)sd->extent * es <= d0 || d0 + (size_t)dd->extent * es <= s0))
      return ph::set_error(PH_E_ARGUMENT, "copy source overlaps the destination through another base pointer");
  }
  return dispatch_copy(dst, dd, src, sd, nullptr);
}

int ph_view_index(int64_t *out, const ph_view_desc *d) {
  PH_GUARD();
  PH_REQUIRE_INIT();
  int rc = ph::validate_desc(d, "view_index");
  if (rc) return rc;
  const int64_t total = ph::desc_count(d);
  if (total == 0) return PH_OK;
  if (!out) return ph::set_error(PH_E_ARGUMENT, "ph_view_index: null output");
  rc = ph::launch_gate("view_index");
  if (rc) return rc;
  hipLaunchKernelGGL(k_view_index, dim3((unsigned)grid_for((total + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     ph::stream(), out, *d, total);
  return ph::check_launch("k_view_index");
}

int ph_fill_scatter(void *dst, int32_t dtype, const int64_t *dst_shape, int32_t rank,
                    const int64_t *first, const int64_t *step, const int64_t *count,
                    const int32_t *axis, const void *src, const ph_view_desc *sd,
                    const void *fill) {
  PH_GUARD();
  PH_REQUIRE_INIT();
  if (rank < 1 || rank > PH_MAX_RANK)
    return ph::set_error(PH_E_DIMENSION, "ph_fill_scatter: rank %d", rank);
  int rc = ph::validate_desc(sd, "fill_scatter source");
  if (rc) return rc;
  if (sd->nstage != 0)
    return ph::set_error(PH_E_UNSUPPORTED, "ph_fill_scatter: source must be affine");
  if (ph::dtype_size(dtype) != ph::dtype_size(sd->dtype))
    return ph::set_error(PH_E_ARGUMENT, "ph_fill_scatter: dtype mismatch");
  FillScatterArgs a;
  std::memset(&a, 0, sizeof(a));
  a.rank = rank;
  a.rows = 1;
  int used[PH_MAX_RANK] = {0};
  for (int k = 0; k < rank; ++k) {
    if (dst_shape[k] < 0) return ph::set_error(PH_E_DIMENSION, "negative extent");
    a.shape[k] = dst_shape[k];
    a.first[k] = first[k];
    a.step[k] = step[k];
    a.count[k] = count[k];
    a.axis[k] = axis[k];
    if (axis[k] >= 0) {
      if (axis[k] >= sd->view.rank || used[axis[k]])
        return ph::set_error(PH_E_ARGUMENT, "ph_fill_scatter: bad view axis %d", axis[k]);
      used[axis[k]] = 1;
      if (count[k] != sd->view.shape[axis[k]])
        return ph::set_error(PH_E_SHAPE, "ph_fill_scatter: axis %d count %lld vs source %lld", k,
                             (long long)count[k], (long long)sd->view.shape[axis[k]]);
      if (count[k] > 0) {
        if (step[k] == 0) return ph::set_error(PH_E_ARGUMENT, "ph_fill_scatter: zero step");
        const int64_t lastc = first[k] + (count[k] - 1) * step[k];
        if (first[k] < 0 || first[k] >= dst_shape[k] || lastc < 0 || lastc >= dst_shape[k])
          return ph::set_error(PH_E_INDEX, "ph_fill_scatter: region leaves axis %d", k);
      }
    } else if (first[k] < 0 || first[k] >= dst_shape[k]) {
      if (dst_shape[k] > 0) return ph::set_error(PH_E_INDEX, "ph_fill_scatter: fixed index outside axis %d", k);
    }
    if (k < rank - 1) a.rows *= dst_shape[k];
  }
  for (int i = 0; i < sd->view.rank; ++i) {
    if (!used[i] && sd->view.shape[i] != 1)
      return ph::set_error(PH_E_SHAPE, "ph_fill_scatter: source axis %d not mapped", i);
    a.src_stride[i] = sd->view.stride[i];
  }
  a.src_off = sd->view.offset;
  a.cols = dst_shape[rank - 1];
  a.last_axis = axis[rank - 1];
  a.in_first = first[rank - 1];
  a.in_step = step[rank - 1] == 0 ? 1 : step[rank - 1];
  a.in_count = count[rank - 1];
  a.in_src_stride = axis[rank - 1] >= 0 ? sd->view.stride[axis[rank - 1]] : 0;
  switch (ph::dtype_size(dtype)) {
    case 1: return launch_fill_scatter<uint8_t>(dst, a, src, sd->extent, fill);
    case 2: return launch_fill_scatter<uint16_t>(dst, a, src, sd->extent, fill);
    case 4: return launch_fill_scatter<uint32_t>(dst, a, src, sd->extent, fill);
    case 8: return launch_fill_scatter<uint64_t>(dst, a, src, sd->extent, fill);
  }
  return ph::set_error(PH_E_ARGUMENT, "ph_fill_scatter: dtype %d", dtype);
}

}  // extern "C"
