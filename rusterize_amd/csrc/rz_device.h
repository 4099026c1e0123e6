// rz_device.h -- device helpers shared by every kernel translation unit:
// Rust scalar rules, the crossing, wave-level synchronisation and
// reductions, the strip coverage of a polygon item and the seven pixel
// folds (plain and packed).
#pragma once

#include <hip/hip_runtime.h>
#include <limits.h>
#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "rz_kernels.h"

namespace rzk {

// ------------------------------------------------------ Rust scalar rules --

// `v as usize` (saturating, NaN -> 0), then clamped to `cap`.
__device__ inline int32_t sat_usize_cap(double v, int32_t cap) {
  if (!(v > 0.0)) return 0;
  if (v >= (double)cap) return cap;
  return (int32_t)v;
}
// `v as isize`: saturating, NaN -> 0.
__device__ inline int64_t sat_isize(double v) {
  if (v != v) return 0;
  if (v <= -9223372036854775808.0) return INT64_MIN;
  if (v >= 9223372036854775808.0) return INT64_MAX;
  return (int64_t)v;
}

// NaN results as the reference's x86 build produces them (SSE): an operation
// with a NaN operand returns that NaN, sign kept (the first one when both
// are NaN); an invalid operation (0 * inf, inf - inf, inf / inf) returns the
// default NaN, which is negative.  The GPU's default NaN is positive, and a
// compiled a - b may negate b first, NaN included, so the edge set-up picks
// every NaN explicitly.
__device__ inline double x86_nan(double r, double a, double b) {
  return isnan(a) ? a : (isnan(b) ? b : (isnan(r) ? -__builtin_nan("") : r));
}

// v / res, res the resolution of a raster and inv its exact reciprocal or 0
// (uniform).  Division by a power of two rounds as the product with its
// reciprocal does, and the product is one instruction where the division is
// twelve: 24 jobs of 82 M vertices take 3.77 ms where every edge divides 3.90.
__device__ inline double to_pixel(double v, double res, double inv) { return inv != 0.0 ? v * inv : v / res; }

// PolyEdge::intersect_at (rust/src/geo/edges.rs:50-55): x0 + ((r+0.5) - y0) * dxdy.
// k_prep leaves no NaN x0 or dxdy in a kept edge, so a NaN here comes from an
// invalid operation, which is negative on x86: span_col sends it to column 0
// like any NaN, which is where f64::total_cmp sorts a negative NaN.
__device__ inline double crossing(const PolyEdge& e, int32_t r) {
  return e.x0 + (((double)r + 0.5) - e.y0) * e.dxdy;
}

// PolyEdge of the ring segment (x0, y0) -> (x1, y1) in pixel coordinates
// (extract_ring + PolyEdge::new, edges.rs:27-46, 90-110), rows clamped to
// nrows; true when the edge crosses a row.  xb is its lower end's x.  `odd`
// is set when some row may end with an odd crossing count.  With `slope`
// false the slope of an edge of finite ends is left 0 (edge_slope sets it).
__device__ inline double edge_slope(double xt, double yt, double xb, double yb) {
  // (yb - yt is neither NaN nor zero here)
  const double dx = x86_nan(xb - xt, xb, xt);
  return x86_nan(dx / (yb - yt), dx, 0.0);
}
__device__ inline bool ring_edge(double x0, double y0, double x1, double y1, int32_t nrows, bool slope, PolyEdge& e,
                                 double& xb, double& yb, bool& odd) {
  e = PolyEdge{0.0, 0.0, 0.0, 0, 0};
  if (!(fabs(y0 - y1) >= 2.220446049250313e-16)) {  // edges.rs:100
    // a skipped segment whose end points straddle a pixel-centre row (or are
    // not numbers) leaves rows with an odd crossing count
    if (isnan(y0) || isnan(y1) || ceil(fmin(y0, y1) - 0.5) != ceil(fmax(y0, y1) - 0.5)) odd = true;
    return false;
  }
  if (!(fmin(y0, y1) < (double)nrows && fmax(y0, y1) >= 0.0)) return false;  // edges.rs:105
  const bool down = y0 < y1;
  e.x0 = down ? x0 : x1;
  e.y0 = down ? y0 : y1;
  xb = down ? x1 : x0;
  yb = down ? y1 : y0;
  e.ystart = sat_usize_cap(ceil(e.y0 - 0.5), nrows);
  e.yend = sat_usize_cap(ceil(yb - 0.5), nrows);
  const double inf = __builtin_inf();
  const bool finite = fabs(e.x0) < inf && fabs(xb) < inf && fabs(e.y0) < inf && fabs(yb) < inf;
  if (slope || !finite) {
    e.dxdy = edge_slope(e.x0, e.y0, xb, yb);
    // With a NaN x0 or slope, every crossing of the edge is NaN with that
    // NaN's sign (x0's when both are NaN).  The reference sorts a positive
    // NaN crossing last, where it closes an empty span or is the odd one out:
    // as if it were absent, so the edge is emptied.  A negative one sorts
    // first and spans from column 0, like -inf: the edge is pinned there.
    if (isnan(e.x0) || isnan(e.dxdy)) {
      if (signbit(isnan(e.x0) ? e.x0 : e.dxdy)) {
        e.x0 = -inf;
        e.y0 = 0.0;
        e.dxdy = 0.0;
      } else {
        if (e.ystart < e.yend) odd = true;  // its rows lose one crossing each
        e.ystart = e.yend = 0;
      }
    }
  }
  return e.ystart < e.yend;
}

// The wave's index in its workgroup, as a scalar (the compiler takes
// threadIdx.x >> 6 for a value per lane, and all addresses made of it too).
__device__ inline int wave_index() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// Orders a wave's LDS accesses around this point (wave-private buffers need
// no workgroup barrier).
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ----------------------------------------------------------- pixel folds --

template <typename T> __device__ inline bool isnan_t(T) { return false; }
template <> __device__ inline bool isnan_t<float>(float v) { return v != v; }
template <> __device__ inline bool isnan_t<double>(double v) { return v != v; }

template <typename T> struct Unsigned { using type = T; };
template <> struct Unsigned<int8_t> { using type = uint8_t; };
template <> struct Unsigned<int16_t> { using type = uint16_t; };
template <> struct Unsigned<int32_t> { using type = uint32_t; };
template <> struct Unsigned<int64_t> { using type = uint64_t; };

// Integer `+=` wraps (release profile); floats add in their own precision.
template <typename T> __device__ inline T add_wrap(T a, T b) {
  using U = typename Unsigned<T>::type;
  return (T)(U)((U)a + (U)b);
}
template <> __device__ inline float add_wrap<float>(float a, float b) { return a + b; }
template <> __device__ inline double add_wrap<double>(double a, double b) { return a + b; }

// The seven transitions of rust/src/rasterization/pixel_functions.rs:55-123,
// applied k >= 1 times with the same value (all writes of one geometry
// carry one value, so only their number matters; sum and count are the
// only non-idempotent transitions).
template <typename T, int FUN>
__device__ inline void fold(T& p, T v, T bg, uint32_t k) {
  if (FUN == 0) {  // sum
    for (uint32_t i = 0; i < k; ++i)
      p = (p == bg || isnan_t(p) || isnan_t(v)) ? v : add_wrap(p, v);
  } else if (FUN == 1) {  // first
    if (p == bg || isnan_t(p)) p = v;
  } else if (FUN == 2) {  // last
    p = v;
  } else if (FUN == 3) {  // min
    if (p == bg || isnan_t(p) || p > v) p = v;
  } else if (FUN == 4) {  // max
    if (p == bg || isnan_t(p) || p < v) p = v;
  } else if (FUN == 5) {  // count
    for (uint32_t i = 0; i < k; ++i) p = (p == bg || isnan_t(p)) ? (T)1 : add_wrap(p, (T)1);
  } else {  // any
    p = (T)1;
  }
}

// One write of value v, applied where `hit`: the same transitions as fold
// with k = 1, written as selects so the compiler emits no branch per pixel.
template <typename T, int FUN>
__device__ inline T fold_select(T p, T v, T bg, bool hit) {
  T n;
  if (FUN == 0) n = (p == bg || isnan_t(p) || isnan_t(v)) ? v : add_wrap(p, v);
  else if (FUN == 1) n = (p == bg || isnan_t(p)) ? v : p;
  else if (FUN == 2) n = v;
  else if (FUN == 3) n = (p == bg || isnan_t(p) || p > v) ? v : p;
  else if (FUN == 4) n = (p == bg || isnan_t(p) || p < v) ? v : p;
  else if (FUN == 5) n = (p == bg || isnan_t(p)) ? (T)1 : add_wrap(p, (T)1);
  else n = (T)1;
  return hit ? n : p;
}

// ---- packed folds for 1- and 2-byte outputs: the same transitions on the
// 4 (or 2) pixels of a 32-bit word at once, lane-wise on the word (SWAR).
// Equality and wrapping addition are bitwise, so signedness only matters for
// min / max.
template <int S> struct Lanes;
template <> struct Lanes<1> {
  static constexpr uint32_t lo7 = 0x7F7F7F7Fu, hi = 0x80808080u, one = 0x01010101u, full = 0xFFu;
  static constexpr int sh = 7;
};
template <> struct Lanes<2> {
  static constexpr uint32_t lo7 = 0x7FFF7FFFu, hi = 0x80008000u, one = 0x00010001u, full = 0xFFFFu;
  static constexpr int sh = 15;
};

// all-ones in each lane where a and b are equal
template <int S> __device__ inline uint32_t lane_eq(uint32_t a, uint32_t b) {
  using L = Lanes<S>;
  const uint32_t x = a ^ b;
  const uint32_t z = ~(((x & L::lo7) + L::lo7) | x | L::lo7);  // lane sign bit set iff the lane is 0
  return (z >> L::sh) * L::full;
}
// lane-wise wrapping a + b
template <int S> __device__ inline uint32_t lane_add(uint32_t a, uint32_t b) {
  using L = Lanes<S>;
  return ((a & L::lo7) + (b & L::lo7)) ^ ((a ^ b) & L::hi);
}
// 4 (or 2) pixel bits -> all-ones lanes
template <int S> __device__ inline uint32_t lane_mask(uint32_t bits) {
  if (S == 1) return ((bits * 0x00204081u) & 0x01010101u) * 0xFFu;
  return ((bits & 1u) * 0xFFFFu) | (((bits >> 1) & 1u) * 0xFFFF0000u);
}

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef short i16x2 __attribute__((ext_vector_type(2)));
template <typename V> __device__ inline V as_vec(uint32_t w) {
  V v;
  __builtin_memcpy(&v, &w, 4);
  return v;
}
template <typename V> __device__ inline uint32_t as_word(V v) {
  uint32_t w;
  __builtin_memcpy(&w, &v, 4);
  return w;
}
// lane-wise unsigned min / max of 16-bit lanes (packed 16-bit VALU)
__device__ inline uint32_t pk_min_u16(uint32_t a, uint32_t b) {
  return as_word(__builtin_elementwise_min(as_vec<u16x2>(a), as_vec<u16x2>(b)));
}
__device__ inline uint32_t pk_max_u16(uint32_t a, uint32_t b) {
  return as_word(__builtin_elementwise_max(as_vec<u16x2>(a), as_vec<u16x2>(b)));
}
// lane-wise min (MAX = false) or max of T lanes
template <typename T, bool MAX> __device__ inline uint32_t lane_minmax(uint32_t a, uint32_t b) {
  if (sizeof(T) == 2) {
    if (T(-1) < T(0)) {  // int16
      const i16x2 x = as_vec<i16x2>(a), y = as_vec<i16x2>(b);
      return as_word(MAX ? __builtin_elementwise_max(x, y) : __builtin_elementwise_min(x, y));
    }
    return MAX ? pk_max_u16(a, b) : pk_min_u16(a, b);
  }
  // bytes: the even and the odd bytes as two 16-bit lanes each; int8 lanes
  // are biased by 0x80 so that unsigned order is signed order
  const uint32_t bias = (T(-1) < T(0)) ? 0x80808080u : 0u;
  a ^= bias;
  b ^= bias;
  const uint32_t ae = a & 0x00FF00FFu, ao = (a >> 8) & 0x00FF00FFu;
  const uint32_t be = b & 0x00FF00FFu, bo = (b >> 8) & 0x00FF00FFu;
  const uint32_t e = MAX ? pk_max_u16(ae, be) : pk_min_u16(ae, be);
  const uint32_t o = MAX ? pk_max_u16(ao, bo) : pk_min_u16(ao, bo);
  return (e | (o << 8)) ^ bias;
}

// The transitions of fold_select on every lane of word p whose mask lane is
// set (vw, bgw: the value and background repeated in every lane).
template <typename T, int FUN>
__device__ inline uint32_t fold_word(uint32_t p, uint32_t vw, uint32_t bgw, uint32_t m) {
  constexpr int S = (int)sizeof(T);
  const uint32_t e = lane_eq<S>(p, bgw);  // `== bg` (integers: never NaN)
  uint32_t n;
  if (FUN == 0) n = (e & vw) | (~e & lane_add<S>(p, vw));  // sum
  else if (FUN == 1) n = (e & vw) | (~e & p);              // first
  else if (FUN == 2) n = vw;                               // last
  else if (FUN == 3) n = (e & vw) | (~e & lane_minmax<T, false>(p, vw));  // min: p > v -> v
  else if (FUN == 4) n = (e & vw) | (~e & lane_minmax<T, true>(p, vw));   // max: p < v -> v
  else if (FUN == 5) n = (e & Lanes<S>::one) | (~e & lane_add<S>(p, Lanes<S>::one));  // count
  else n = Lanes<S>::one;                                  // any
  return (m & n) | (~m & p);
}

// value bits repeated in every lane of a word
template <typename T> __device__ inline uint32_t lane_splat(uint64_t bits) {
  return sizeof(T) == 1 ? ((uint32_t)bits & 0xFFu) * 0x01010101u : ((uint32_t)bits & 0xFFFFu) * 0x00010001u;
}

template <typename T> __device__ inline T from_bits(uint64_t b) {
  T v;
  __builtin_memcpy(&v, &b, sizeof(T));
  return v;
}


// The new value of a pixel written once (the transitions of fold, k = 1).
template <typename T, int FUN>
__device__ inline T fold_value(T p, T v, T bg) {
  return fold_select<T, FUN>(p, v, bg, true);
}

// ~0 when bit r (a constant) of x is set, else 0.  (In asm: written out, the
// compiler turns the extract and the select below into a compare and a
// conditional move.)
__device__ __attribute__((always_inline)) inline int32_t bit_mask(uint32_t x, int r) {
  int32_t m;
  asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(m) : "v"(x), "n"(r));
  return m;
}

// p where mask is 0, n where it is ~0 (bit select, no compare).
template <typename T>
__device__ inline T bit_select(int32_t mask, T n, T p) {
  if constexpr (sizeof(T) == 8) {
    uint2 a, b;
    __builtin_memcpy(&a, &n, 8);
    __builtin_memcpy(&b, &p, 8);
    b.x = (a.x & (uint32_t)mask) | (b.x & ~(uint32_t)mask);
    b.y = (a.y & (uint32_t)mask) | (b.y & ~(uint32_t)mask);
    __builtin_memcpy(&p, &b, 8);
  } else {
    uint32_t a, b;
    __builtin_memcpy(&a, &n, 4);
    __builtin_memcpy(&b, &p, 4);
    b = (a & (uint32_t)mask) | (b & ~(uint32_t)mask);
    __builtin_memcpy(&p, &b, 4);
  }
  return p;
}

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Combine a value across groups of LANES (4 or 8) lanes with DPP quad
// permutations ([1,0,3,2] then [2,3,0,1]) and, for 8, a mirror of each half
// row (the quads hold one value each by then): VALU data movement, no LDS.
template <int LANES>
__device__ inline uint32_t group_xor(uint32_t x) {
  x ^= (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xF, 0xF, false);
  x ^= (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x4E, 0xF, 0xF, false);
  if constexpr (LANES == 8) x ^= (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x141, 0xF, 0xF, false);
  return x;
}
template <int LANES>
__device__ inline uint64_t group_xor64(uint64_t x) {
  return (uint64_t)group_xor<LANES>((uint32_t)x) | ((uint64_t)group_xor<LANES>((uint32_t)(x >> 32)) << 32);
}
template <int LANES>
__device__ inline int32_t group_max(int32_t x) {
  x = max(x, __builtin_amdgcn_mov_dpp(x, 0xB1, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_mov_dpp(x, 0x4E, 0xF, 0xF, false));
  if constexpr (LANES == 8) x = max(x, __builtin_amdgcn_mov_dpp(x, 0x141, 0xF, 0xF, false));
  return x;
}

// Transposes 16 x 16 bit blocks over 16 lanes' words: lane i (of each 16)
// gives row i of the low and of the high block and gets column i of each.
// Four exchanges with the lane 8, 4, 2 and 1 away, each a rotate and a bit
// select.
template <int S>
__device__ inline uint32_t exchange16(uint32_t x, int lane) {
  constexpr uint32_t M = S == 8 ? 0x00FF00FFu : (S == 4 ? 0x0F0F0F0Fu : (S == 2 ? 0x33333333u : 0x55555555u));
  int y;
  if constexpr (S == 8) {
    y = __builtin_amdgcn_update_dpp(0, (int)x, 0x128, 0xF, 0xF, false);  // row_ror:8
  } else if constexpr (S == 4) {
    y = __builtin_amdgcn_update_dpp(0, (int)x, 0x104, 0xF, 0x5, false);  // row_shl:4 into banks 0, 2
    y = __builtin_amdgcn_update_dpp(y, (int)x, 0x114, 0xF, 0xA, false);  // row_shr:4 into banks 1, 3
  } else {
    y = __builtin_amdgcn_update_dpp(0, (int)x, S == 2 ? 0x4E : 0xB1, 0xF, 0xF, false);  // quad_perm
  }
  const bool up = (lane & S) != 0;
  const uint32_t K = up ? ~M : M;
  const uint32_t r = __builtin_amdgcn_alignbit((uint32_t)y, (uint32_t)y, up ? (uint32_t)S : 32u - (uint32_t)S);
  return (x & K) | (r & ~K);
}
__device__ inline uint32_t transpose16x2(uint32_t x, int lane) {
  return exchange16<1>(exchange16<2>(exchange16<4>(exchange16<8>(x, lane), lane), lane), lane);
}

// A workgroup barrier that orders LDS accesses only: global loads and stores
// stay in flight across it (__syncthreads waits for all of them).
__device__ inline void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Inclusive prefix sum over the wave with DPP row shifts and broadcasts
// (VALU only: a shuffle of this chain waits on LDS at every step).
__device__ inline uint32_t wave_prefix_sum(uint32_t x) {
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xF, 0xF, true);   // row_shr:1
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xF, 0xF, true);   // row_shr:2
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xF, 0xF, true);   // row_shr:4
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xF, 0xF, true);   // row_shr:8
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1, 3
  x += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2, 3
  return x;
}

// The chunks of 64 vertices of an item's rings whose edges may meet rows
// [R0, R1), in order, those of numbers with a bit in `mine` (of number % 64):
// `rows` holds the row range of each (null: all chunks are taken), 64 of which
// are tested at a time (AHEAD: while the next 64 are loading; without it
// nothing is kept in vector registers).  A long ring is mostly local, so a
// window or strip reads about the edges it needs where it would read all of
// them (see k_cover and strip_coverage).  Every lane of the wave calls next().
template <bool AHEAD>
struct Chunks {
  const int2* rows;
  uint32_t n, sb;         // chunks; those of [sb, sb + 64) with a bit in m are still to come
  int32_t R0, R1;
  uint64_t mine, m;
  int2 ahead;
  int lane;

  __device__ Chunks(const int2* rows_, uint32_t n_, int32_t R0_, int32_t R1_, uint64_t mine_, int lane_)
      : rows(rows_), n(n_), sb(0), R0(R0_), R1(R1_), mine(mine_), ahead(make_int2(0, 0)), lane(lane_) {
    if (AHEAD && rows && (uint32_t)lane < n) ahead = rows[lane];
    test();
  }
  __device__ void test() {
    const uint32_t left = n - sb;
    m = left < 64u ? mine & ((1ull << left) - 1ull) : mine;
    if (rows) {
      if (!AHEAD) {
        ahead = make_int2(0, 0);
        if ((uint32_t)lane < left) ahead = rows[sb + (uint32_t)lane];
      }
      m &= __ballot(ahead.x < R1 && ahead.y > R0);
      if (AHEAD && left > 64u && (uint32_t)lane < left - 64u) ahead = rows[sb + 64u + (uint32_t)lane];
    }
  }
  __device__ bool next(uint32_t& c) {
    while (!m) {
      if (n - sb <= 64u) return false;
      sb += 64u;
      test();
    }
    c = sb + (uint32_t)__builtin_ctzll(m);
    m &= m - 1ull;
    return true;
  }
};

// One 64-byte descriptor from a read-only table (four 16-byte loads).
__device__ inline ItemDesc load_desc(const RZ_CONST ItemDesc* p) {
  const RZ_CONST u32x4* q = (const RZ_CONST u32x4*)p;
  const u32x4 w[4] = {q[0], q[1], q[2], q[3]};
  ItemDesc d;
  __builtin_memcpy(&d, w, sizeof(d));
  return d;
}

// The box (r0, r1, c0, c1) and kind | band word of a descriptor: its first
// 32 bytes (two 16-byte loads), all a box test needs.
struct BoxLayer {
  int32_t r0, r1, c0, c1;
  uint32_t kind_layer;
};
__device__ inline BoxLayer load_box(const RZ_CONST ItemDesc* p) {
  const RZ_CONST u32x4* q = (const RZ_CONST u32x4*)p;
  const u32x4 a = q[0], b = q[1];
  return BoxLayer{(int32_t)a[0], (int32_t)a[1], (int32_t)a[2], (int32_t)a[3], b[3]};
}

// First index of XCD x's contiguous share of n.
__device__ inline uint32_t xcd_unit_lo(uint32_t x, uint32_t n) {
  const uint32_t per = n / NUM_XCD, rem = n % NUM_XCD;
  return x * per + min(x, rem);
}

// Coverage of one polygon item over ROWS (16 or 8) rows from Rw on (rows from
// strip_r1 on excluded) and the columns [C0, C0 + 64 * NWORD): lane
// (rl = lane / LPR, q = lane % LPR, LPR = 64 / ROWS) returns word q of row
// Rw + rl's mask (lanes with q >= NWORD return 0).  Lane layout: the LPR lanes
// of a row take every LPR-th active edge; their crossing toggles are
// XOR-combined with DPP and the row mask follows from the note above
// row_coverage_word in rz_kernels.h.  The item's edges are edges[vbeg .. vbeg
// + n_e), in the chunks of 64 that meet the rows (chunk_rows: see Chunks).
// `stage` is 64 edges of wave-private LDS.
template <int NWORD, int ROWS>
__device__ inline uint64_t strip_coverage(const PolyEdge* edges, int64_t vbeg, uint32_t n_e, const int2* chunk_rows,
                                          int32_t Rw, int32_t strip_r1, int32_t C0, double ncols_f,
                                          PolyEdge* stage, int lane) {
  constexpr int LPR = 64 / ROWS;  // lanes per row
  static_assert(LPR == 4 || LPR == 8, "16 or 8 rows");
  const int rl = lane / LPR, q = lane % LPR;
  const int32_t r = Rw + rl;
  const bool row_ok = r < strip_r1;
  uint64_t tog[NWORD];
#pragma unroll
  for (int w = 0; w < NWORD; ++w) tog[w] = 0ull;
  uint32_t lp = 0;
  int32_t amax = -1;
  // (chunks start at multiples of 64 vertices of the batch)
  const bool local = chunk_rows && n_e > (uint32_t)kChunkNv;
  const uint32_t skew = local ? (uint32_t)vbeg & 63u : 0u;
  const PolyEdge* ebase = edges + vbeg;
  Chunks<false> chunks(local ? chunk_rows + (vbeg >> 6) : nullptr, (n_e + skew + 63u) >> 6, Rw, strip_r1, ~0ull, lane);
  uint32_t c;
  while (chunks.next(c)) {
    // stage the edges of this chunk that reach the strip, compacted
    // (two 16-byte vector loads and stores: no struct copy through scratch)
    const uint32_t e = c * 64u + (uint32_t)lane - skew;  // (those before the item wrap)
    uint4 e_lo = make_uint4(0u, 0u, 0u, 0u), e_hi = make_uint4(0u, 0u, 0u, 0u);
    bool act = false;
    if (e < n_e) {
      const uint4* src = reinterpret_cast<const uint4*>(ebase + e);
      e_lo = src[0];
      e_hi = src[1];  // dxdy, ystart (z), yend (w)
      const int32_t ys = (int32_t)e_hi.z, ye = (int32_t)e_hi.w;
      act = ys < strip_r1 && ye > Rw && ys < ye;
    }
    const uint64_t m = __ballot(act);
    if (act) {
      uint4* dst = reinterpret_cast<uint4*>(stage + __popcll(m & ((1ull << lane) - 1ull)));
      dst[0] = e_lo;
      dst[1] = e_hi;
    }
    wave_sync();
    const int n = __popcll(m);
    for (int k0 = 0; k0 < n; k0 += LPR) {  // uniform trip count, predicated lanes
      const int k = k0 + q;
      const PolyEdge ee = stage[k < n ? k : n - 1];
      const bool on = k < n && row_ok && ee.ystart <= r && r < ee.yend;
      const double x = crossing(ee, r);
      toggle_crossing_if<NWORD>(on, span_col(x, ncols_f), C0, tog, lp, amax);
    }
    wave_sync();
  }
  lp = group_xor<LPR>(lp);
  amax = group_max<LPR>(amax);
#pragma unroll
  for (int w = 0; w < NWORD; ++w) tog[w] = group_xor64<LPR>(tog[w]);
  return q < NWORD ? row_coverage_word<NWORD>(tog, lp, amax, C0, q) : 0ull;
}

}  // namespace rzk
