// rz_tile.hip -- the coverage pre-pass of the tile kernel (k_cover).
#pragma once

#include "rz_device.h"

namespace rzk {

// Inclusive prefix parity over the 64 columns of a mask block of toggles, its
// word i (columns 4 i .. 4 i + 3, 16 rows' bits each) in lane i of 16: `carry`
// holds the parities of the block's left neighbours (twice) and gets its own.
__device__ inline uint2 block_parity(uint2 x, uint32_t& carry) {
  x.x ^= x.x << 16;
  x.y ^= x.y << 16;
  x.y ^= __builtin_amdgcn_perm(x.x, x.x, 0x03020302u);  // (the high half, twice)
  uint32_t t = __builtin_amdgcn_perm(x.y, x.y, 0x03020302u);
  t ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)t, 0x111, 0xF, 0xF, true);  // row_shr:1, 2, 4, 8
  t ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)t, 0x112, 0xF, 0xF, true);
  t ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)t, 0x114, 0xF, 0xF, true);
  t ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)t, 0x118, 0xF, 0xF, true);
  const uint32_t left = carry ^ (uint32_t)__builtin_amdgcn_update_dpp(0, (int)t, 0x111, 0xF, 0xF, true);
  carry ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)t, 0x15F, 0xF, 0xF, true);  // row_newbcast:15
  return make_uint2(x.x ^ left, x.y ^ left);
}

// Row words keep column 4 i + j of 64 at bit 16 j + i, so that the transposition
// of 16 rows' words (below) leaves a mask block's word i in lane i.
// Inclusive prefix parity over a row word's columns, `carry` (0 or ~0) before
// them: that of the sums of four columns, then column by column.
__device__ inline uint64_t row_parity(uint64_t x, uint32_t& carry) {
  uint32_t lo = (uint32_t)x, hi = (uint32_t)(x >> 32);
  uint32_t t = lo ^ hi;
  t = (t ^ (t >> 16)) & 0xFFFFu;
  t ^= t << 1;
  t ^= t << 2;
  t ^= t << 4;
  t ^= t << 8;
  const uint32_t left = __builtin_amdgcn_perm(t << 1, t << 1, 0x01000100u) ^ carry;  // (the low half, twice)
  carry ^= 0u - ((t >> 15) & 1u);
  lo ^= lo << 16;
  hi ^= hi << 16;
  hi ^= __builtin_amdgcn_perm(lo, lo, 0x03020302u);
  return (uint64_t)(lo ^ left) | ((uint64_t)(hi ^ left) << 32);
}
// The columns below n of a row word.
__device__ inline uint64_t row_below(int64_t n) {
  uint64_t m = 0ull;
  for (int j = 0; j < 4; ++j) {
    const int64_t k = (n - j + 3) >> 2;
    m |= (uint64_t)(k <= 0 ? 0u : (k >= 16 ? 0xFFFFu : ((1u << k) - 1u))) << (16 * j);
  }
  return m;
}
// Row i's word in lane i of each 16: lane i gets word i of the mask block.
__device__ inline uint64_t block_word(uint64_t x, int lane) {
  return (uint64_t)transpose16x2((uint32_t)x, lane) | ((uint64_t)transpose16x2((uint32_t)(x >> 32), lane) << 32);
}

// An item (or a window of one) whose toggle words are in LDS.
struct __align__(16) CoverItem {
  uint32_t A;         // the words of strip (workgroups: row) r start at cover_word(A, r, stride)
  int32_t stride;
  int32_t W0, wid;    // first column and columns
  int32_t R0, R1;     // raster rows [R0, R1)
  int64_t lv;         // edge e of the unit starts at local vertex lv + e
  uint32_t mask;      // ItemDesc::mask
  uint32_t row0;      // rows of the unit's items before this one
  uint32_t base, pad; // word of its first strip
  // The windows of a whole item, its rows and LDS words.
  __device__ void set_box(int32_t r0, int32_t r1, int32_t c0, int32_t c1, uint32_t& rows, uint32_t& words) {
    const int32_t ww = mask_row_words(c0, c1);
    rows = (uint32_t)mask_strip_count(r0, r1) * 16u;
    stride = cover_stride(ww, false, false);
    words = (rows >> 4) * (uint32_t)stride;
    W0 = (c0 >> 6) * 64;
    wid = ww * 64;
    R0 = (r0 >> 4) * 16;
    R1 = R0 + (int32_t)rows;
  }
};

// A wave's share of the LDS of k_cover and k_items.
constexpr int kStartWords = 32;
struct CoverWave {
  uint64_t* tog;       // toggle words
  double (*edges)[4];  // [64] x0, y0, dxdy, (row offset, item)
  CoverItem* items;
  uint64_t* start;     // [kStartWords] start bits
  uint32_t base;       // the wave's first toggle word
  int lane;
  const int2* chunk_rows;  // (window<true> only)

  // Start bits up to and with this lane's, less one.
  __device__ static uint32_t rank_of(uint32_t lo, uint32_t hi) {
    const uint64_t s1 = (((uint64_t)hi << 32) | lo) >> 1;
    return (lo & 1u) - 1u +
           __builtin_amdgcn_mbcnt_hi((uint32_t)(s1 >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)s1, 0u));
  }

  // Owners (lanes with `own`) hold consecutive runs of positions, the lane's
  // from `first`.  Position c + lane belongs to owner number `before` plus
  // the value returned; `before` moves past the owners that start here.
  __device__ __attribute__((always_inline)) uint32_t owner(bool own, uint32_t first, uint32_t c, uint32_t& before) const {
    if (lane == 0) *start = 0ull;
    wave_sync();
    if (own && first >= c && first - c < 64u)
      __hip_atomic_fetch_or(start, 1ull << (first - c), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    wave_sync();
    const uint64_t v = *start;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    const uint32_t at = before + rank_of(lo, hi);
    before += (uint32_t)(__popc(lo) + __popc(hi));
    wave_sync();
    return at;
  }

  // The toggles of n_e edges, taken in chunks of 64.  MANY: of the items in
  // `items`, the lane's (own) from edge e0 of the one chunk on; else of `one`
  // (in scalar registers: a read of LDS less for every crossing).  AHEAD: those
  // chunks of it that `chunks` hands out, its first `skew` edges before the
  // item's.
  template <bool AHEAD, bool MANY>
  __device__ __attribute__((always_inline)) void toggles(const RZ_CONST JobDev& J, const CoverItem& one, bool own, uint32_t e0,
                                                         uint32_t n_e, Chunks<true>* chunks, uint32_t skew, bool odd) const {
    const double ncols_f = (double)J.ncols;
    auto px_x = [&](double X) { return isnan(X) ? X : to_pixel(X - J.xmin, J.xres, J.xinv); };
    auto px_y = [&](double Y) { return isnan(Y) ? Y : to_pixel(J.ymax - Y, J.yres, J.yinv); };
    // the crossing of row r by the edge x0, y0, dxdy of an item
    auto cross = [&](const CoverItem& it, int32_t r, double x0, double y0, double dxdy) __attribute__((always_inline)) {
      const int32_t W0 = it.W0, wid = it.wid;
      const double x = x0 + (((double)r + 0.5) - y0) * dxdy;
      const int32_t col = span_col(x, ncols_f);
      const int32_t rel = max(col - W0, 0);
      if constexpr (AHEAD) {
        // (row by row: the many short edges of a long ring would otherwise
        // flip bits of the same few words, one after the other: 24 jobs of
        // rings of up to 4,096 vertices 1.13 ms, row by row 1.06)
        uint32_t* row = reinterpret_cast<uint32_t*>(tog + cover_word(it.A, r, it.stride));
        if (rel < wid)
          __hip_atomic_fetch_xor(row + ((rel >> 6) * 2 + ((rel >> 1) & 1)), 1u << ((rel & 1) * 16 + ((rel >> 2) & 15)),
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        // the rightmost crossing of a row matters only with an odd count
        if (odd)
          __hip_atomic_fetch_max(row + (wid >> 5), (uint32_t)col + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        return;
      }
      uint32_t* strip = reinterpret_cast<uint32_t*>(tog + cover_word(it.A, r >> 4, it.stride));
      if (rel < wid)
        __hip_atomic_fetch_xor(strip + (rel >> 1), 1u << ((rel & 1) * 16 + (r & 15)), __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
      if (odd) {
        uint32_t* end = strip + (wid >> 1) + (r & 15) * 2;
        __hip_atomic_fetch_max(end, (uint32_t)col + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        __hip_atomic_fetch_xor(end + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      }
    };
    // (an item's next vertices are loaded while this chunk's edges are built)
    uint64_t vi = 0;
    double2 p{}, q{};
    auto load = [&](int64_t v) __attribute__((always_inline)) {
      const int64_t vn = min(v + 1, J.nv - 1);
      vi = J.vert_info[v];
      p = *reinterpret_cast<const double2*>(J.xy + 2 * v);
      q = *reinterpret_cast<const double2*>(J.xy + 2 * vn);
    };
    uint32_t cb = 0;  // the chunk's first edge (of a first chunk with edges before the item's it wraps)
    bool more = n_e > 0u;
    auto advance = [&]() __attribute__((always_inline)) {
      uint32_t c = 0;
      more = chunks->next(c);
      cb = c * 64u - skew;
      if (more && cb + (uint32_t)lane < n_e) load(one.lv + (int64_t)(cb + (uint32_t)lane));
    };
    if (AHEAD) advance();
    for (; AHEAD ? more : cb < n_e; cb += AHEAD ? 0u : 64u) {
      const uint32_t e = cb + (uint32_t)lane;
      uint32_t before = 0;
      const uint32_t k = MANY ? owner(own, e0, 0u, before) : 0u;
      const CoverItem& it = MANY ? items[k] : one;
      if (!AHEAD && e < n_e) load(it.lv + (int64_t)e);
      const uint64_t vi0 = vi;
      const double2 p0 = p, q0 = q;
      if (AHEAD) advance();
      PolyEdge ee{0.0, 0.0, 0.0, 0, 0};
      int32_t a0 = 0;
      uint32_t span = 0;
      if (e < n_e) {
        double xb, yb;
        bool o = false;
        if ((vi0 & VI_HAS_NEXT) && ring_edge(px_x(p0.x), px_y(p0.y), px_x(q0.x), px_y(q0.y), J.nrows, false, ee, xb, yb, o)) {
          a0 = max(ee.ystart, it.R0);
          span = (uint32_t)max(0, min(ee.yend, it.R1) - a0);
          // (an edge of an infinite or NaN end has its slope already: its
          // crossings are pinned or come from that slope)
          const double inf = __builtin_inf();
          if (span && fabs(ee.x0) < inf && fabs(xb) < inf && fabs(ee.y0) < inf && fabs(yb) < inf)
            ee.dxdy = edge_slope(ee.x0, ee.y0, xb, yb);
        }
      }
      const uint64_t act = __ballot(span != 0u);
      if (!act) continue;
      const uint32_t incl = wave_prefix_sum(span);
      const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
      const uint32_t excl = incl - span;
      if (span) {  // compacted: the crossing loop finds edges by their rank
        double* dst = edges[__popcll(act & ((1ull << lane) - 1ull))];
        dst[0] = ee.x0;
        dst[1] = ee.y0;
        dst[2] = ee.dxdy;
        const uint64_t rk = (uint64_t)(uint32_t)(a0 - (int32_t)excl) | ((uint64_t)k << 32);
        __builtin_memcpy(dst + 3, &rk, 8);
      }
      // Position c + lane of a block of 64 * kStartWords crossings belongs to
      // the edge whose start bit is the last one up to it: all start bits of
      // the block are set first and kept one word per lane, so a crossing's
      // edge is found without a trip through LDS.
      before = 0;
      for (uint32_t b0 = 0; b0 < total; b0 += 64u * kStartWords) {
        if (lane < kStartWords) start[lane] = 0ull;
        wave_sync();
        const uint32_t at0 = excl - b0;
        if (span && excl >= b0 && at0 < 64u * kStartWords)
          __hip_atomic_fetch_or(start + (at0 >> 6), 1ull << (at0 & 63u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        wave_sync();
        const uint64_t bits = start[lane & (kStartWords - 1)];
        const uint32_t top = min(total - b0, 64u * kStartWords);
        for (uint32_t c = 0; c < top; c += 64u) {
          const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)bits, (int)(c >> 6));
          const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(bits >> 32), (int)(c >> 6));
          const uint32_t at = before + rank_of(lo, hi);
          before += (uint32_t)(__popc(lo) + __popc(hi));
          if (c + (uint32_t)lane < top) {
            const double* src = edges[at];
            uint64_t rk;
            __builtin_memcpy(&rk, src + 3, 8);
            const int32_t r = (int32_t)(b0 + c + (uint32_t)lane) + (int32_t)(uint32_t)rk;
            cross(MANY ? items[rk >> 32] : one, r, src[0], src[1], src[2]);
          }
        }
        wave_sync();
      }
      wave_sync();
    }
  }

  // A strip's toggles (ww blocks of 16 words from `strip`, cleared as they are
  // read) into mask blocks out, out + 16, ..., by 16 neighbouring lanes, a word
  // of each block to a lane (k, of 16; out: the lane's word of a block).  odd:
  // each row's rightmost crossing + 1 and parity lie after its words; a row of
  // odd parity covers nothing from that crossing on, as if it were there twice
  // (W0: the strip's first column).
  __device__ __attribute__((always_inline)) void finish_strip(uint64_t* strip, int32_t k, int32_t ww, uint64_t* out,
                                                              bool odd, int32_t W0) const {
    if (odd) {
      const uint64_t end = strip[16 * ww + k];
      strip[16 * ww + k] = 0ull;
      const int32_t rel = max((int32_t)((uint32_t)end - 1u) - W0, 0);
      if ((end >> 32) && rel < 64 * ww)
        __hip_atomic_fetch_xor(reinterpret_cast<uint32_t*>(strip) + (rel >> 1), 1u << ((rel & 1) * 16 + k),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
      wave_sync();
    }
    uint2* p = reinterpret_cast<uint2*>(strip + k);
    uint32_t carry = 0u;
    for (int32_t w = 0; w < ww; ++w) {
      const uint2 x = block_parity(p[16 * w], carry);
      p[16 * w] = make_uint2(0u, 0u);
      reinterpret_cast<uint2*>(out)[16 * w] = x;
    }
  }

  // One row's toggles (ww words from `row`, cleared as they are read), the
  // rows of a strip in 16 neighbouring lanes, into mask blocks out, out + 16,
  // ... (out: the lane's word of a block); odd: the row's rightmost crossing + 1
  // lies after its words, W0 is its first column.
  __device__ __attribute__((always_inline)) void finish_row(uint64_t* row, int32_t ww, uint64_t* out, bool odd, int32_t W0) const {
    int64_t lim = INT_MAX;  // columns of the window left of the rightmost crossing
    if (odd) {
      lim = (int64_t)(uint32_t)row[ww] - 1 - (int64_t)W0;
      row[ww] = 0ull;
    }
    uint32_t carry = 0u;
    for (int32_t w = 0; w < ww; ++w) {
      uint64_t x = row_parity(row[w], carry);
      row[w] = 0ull;
      if (odd) x &= row_below(lim - 64 * (int64_t)w);
      out[(uint64_t)w * 16u] = block_word(x, lane);
    }
  }

  // The masks of small items, one per lane with `ok` (at most 64 edges and
  // kCoverWave LDS words each; it: all but A, base and row0): as many of them
  // as fit together form a unit.
  __device__ __attribute__((always_inline)) void small_items(const RZ_CONST JobDev* jobs_c, uint64_t* masks,
                                                             const CoverItem& it, bool ok, uint32_t job, uint32_t nv,
                                                             uint32_t words, uint32_t rows) const {
    uint64_t todo = __ballot(ok);
    while (todo) {
      // the unit: the next items of one job that fit together
      const uint32_t j = (uint32_t)__builtin_amdgcn_readlane((int)job, __builtin_ctzll(todo));
      const bool mine = (todo >> lane) & 1ull;
      const uint32_t ei = wave_prefix_sum(mine ? nv : 0u), wi = wave_prefix_sum(mine ? words : 0u);
      const uint64_t no = __ballot(mine && (job != j || ei > 64u || wi > (uint32_t)kCoverWave));
      const uint64_t unit = todo & (no ? ((1ull << __builtin_ctzll(no)) - 1ull) : ~0ull);
      todo &= ~unit;
      const bool own = (unit >> lane) & 1ull;
      const int last = 63 - __builtin_clzll(unit);
      const uint32_t n_e = (uint32_t)__builtin_amdgcn_readlane((int)ei, last);
      const uint32_t ri = wave_prefix_sum(own ? rows : 0u);
      const uint32_t n_rows = (uint32_t)__builtin_amdgcn_readlane((int)ri, 63);
      const RZ_CONST JobDev& J = jobs_c[j];
      if (own) {
        CoverItem x = it;
        x.base = base + wi - words;
        x.A = cover_origin(x.base, x.R0 >> 4, x.stride);
        x.R1 = min(x.R1, J.nrows);
        x.lv -= J.v_base + (int64_t)(ei - nv);
        x.row0 = ri - rows;
        items[__popcll(unit & ((1ull << lane) - 1ull))] = x;
      }
      wave_sync();
      toggles<false, true>(J, it, own, ei - nv, n_e, nullptr, 0u, false);
      uint32_t before = 0;
      for (uint32_t c = 0; c < n_rows; c += 64u) {
        const uint32_t at = owner(own, ri - rows, c, before);
        if (c + (uint32_t)lane < n_rows) {
          const CoverItem x = items[at];
          const uint32_t r = c + (uint32_t)lane - x.row0;
          finish_strip(tog + x.base + (r >> 4) * (uint32_t)x.stride, (int32_t)(r & 15u), x.wid >> 6,
                       masks + ((uint64_t)x.mask + (uint64_t)(r >> 4) * (uint64_t)(x.wid >> 6)) * 16u + (uint64_t)(r & 15u),
                       false, 0);
        }
      }
      wave_sync();
    }
  }

  // Window t of an item, by the wave or (BLOCK) the four of a workgroup.
  template <bool BLOCK>
  __device__ __attribute__((always_inline)) void window(const RZ_CONST JobDev& J, uint64_t* masks, int32_t r0, int32_t r1,
                                                        int32_t c0, int32_t c1, int64_t vbeg, uint32_t nv, bool odd,
                                                        uint32_t mask, int32_t t) const {
    const int32_t ns = mask_strip_count(r0, r1), nw = mask_row_words(c0, c1);
    const CoverWindows win = cover_windows(ns, nw, odd, BLOCK);
    const int32_t row = win.n == 1 ? 0 : t / win.ncw;
    const int32_t s0 = row * win.strips, w0 = (t - row * win.ncw) * win.ww;
    const int32_t ww = min(win.ww, nw - w0), n_rows = min(win.strips, ns - s0) * 16;
    const int32_t first = BLOCK ? 0 : (int32_t)base, R0 = ((r0 >> 4) + s0) * 16, W0 = ((c0 >> 6) + w0) * 64;
    CoverItem it{};
    it.stride = BLOCK ? win.stride >> 4 : win.stride;
    it.A = cover_origin((uint32_t)first, BLOCK ? R0 : R0 >> 4, it.stride);
    it.W0 = W0;
    it.wid = ww * 64;
    it.R0 = R0;
    it.R1 = min(R0 + n_rows, J.nrows);
    it.lv = vbeg - J.v_base;
    if constexpr (BLOCK) {  // the waves take the window's chunks in turn
      // (an item of one window needs them all, from its own first vertex on)
      const bool all = win.n == 1;
      const uint32_t skew = all ? 0u : (uint32_t)vbeg & 63u;
      static_assert(kCoverBlockWaves == 4, "every fourth chunk is a wave's");
      Chunks<true> chunks(all ? nullptr : chunk_rows + (vbeg >> 6), (nv + skew + 63u) >> 6, R0, R0 + n_rows,
                    0x1111111111111111ull << wave_index(), lane);
      toggles<true, false>(J, it, false, 0u, nv, &chunks, skew, odd);
    } else {
      toggles<false, false>(J, it, false, 0u, nv, nullptr, 0u, odd);
    }
    if (BLOCK) __syncthreads();
    else wave_sync();
    for (int32_t r = BLOCK ? (int32_t)threadIdx.x : lane; r < n_rows; r += BLOCK ? 64 * kCoverBlockWaves : 64) {
      uint64_t* out = masks + ((uint64_t)mask + (uint64_t)(s0 + (r >> 4)) * (uint64_t)nw + (uint64_t)w0) * 16u + (uint64_t)(r & 15);
      if (BLOCK) finish_row(tog + r * (win.stride >> 4), ww, out, odd, W0);
      else finish_strip(tog + first + (r >> 4) * win.stride, r & 15, ww, out, odd, W0);
    }
    if (BLOCK) __syncthreads();
    else wave_sync();
  }
};

// The coverage masks of the polygon items, each edge's crossings computed
// once (the tile kernels only read masks).
//
// Per unit (see CoverLists): lanes build the unit's edges from the world
// coordinates, 64 at a time; the (edge, row) crossings of those edges are
// then laid out one per lane (an edge of a few rows and one of hundreds cost
// what they cross, where a lane per edge would wait for the longest one);
// every crossing flips its toggle bit in LDS (order-free), in column 0 when it
// lies left of the window; and the 16 lanes of a strip turn its toggles into
// coverage (inclusive prefix parity across the columns, see the note above
// row_coverage_word) and store it as mask blocks.  A wave's toggles are in the
// blocks' own order, so a word of them (4 columns of 16 rows) takes about 20
// instructions (row by row, with a transposition, 66: 1.1 M small polygons on
// 40000 x 40000 took 0.83 ms, bound by vector issue, and take 0.65).  Small
// items are packed: as many as have at most 64 edges and a wave's LDS words
// together form one unit.
// Windows are bound by the latency of their dependent loads and LDS round
// trips (vector issue is busy about half of the time), so LDS is sized for 6
// waves per SIMD (4 of workgroups), the block list's next edges are loaded ahead and its entries handed
// out as workgroups finish (82 M vertices in rings of up to 4,096: 1.63 ms
// before, with the edges of crossings found through LDS, and 1.06 ms now).
// A window of the block list reads the chunks of its item's vertices that may
// meet its rows (Chunks): 200 rings of 50,000 vertices on 20000 x 20000 take
// 2.5 ms where reading whole rings in every window took 11.4.
// BLOCK: the block list, a workgroup per unit; else the wave and small lists.
template <bool BLOCK>
__global__ __launch_bounds__(64 * (BLOCK ? kCoverBlockWaves : 4)) void k_cover(CoverArgs a) {
  constexpr int NW = BLOCK ? kCoverBlockWaves : 4;  // waves
  constexpr int RUN = BLOCK ? 1 : kCoverRun;
  __shared__ uint64_t s_tog[BLOCK ? kCoverBlock : 4 * kCoverWave];
  __shared__ __align__(16) double s_edge[NW][64][4];  // x0, y0, dxdy, (row offset, item)
  __shared__ CoverItem s_item[NW][RUN];
  __shared__ uint64_t s_start[NW][kStartWords];
  const int wave = wave_index(), lane = threadIdx.x & 63;
  const RZ_CONST JobDev* jobs_c = as_const(a.jobs);
  const RZ_CONST ItemDesc* desc_c = as_const(a.desc);
  const CoverWave cw{s_tog, s_edge[wave], s_item[wave], s_start[wave], (uint32_t)(wave * kCoverWave), lane, a.chunk_rows};
  if (!BLOCK && !a.cover.ctr->n_wave && !a.cover.ctr->n_small) return;
  for (int k = threadIdx.x; k < (BLOCK ? kCoverBlock : 4 * kCoverWave); k += 64 * NW) s_tog[k] = 0ull;
  __syncthreads();

  auto window = [&](const uint2 en) __attribute__((always_inline)) {
    const ItemDesc d = load_desc(desc_c + (uint32_t)__builtin_amdgcn_readfirstlane((int)en.x));
    const int32_t t = __builtin_amdgcn_readfirstlane((int)en.y);
    if (d.flags & kItemMask)  // (not past a capacity)
      cw.window<BLOCK>(jobs_c[d.job], a.masks, d.r0, d.r1, d.c0, d.c1, d.vbeg, (uint32_t)d.nv,
                       (d.flags & kItemOddRows) != 0, d.mask, t);
  };

  if constexpr (BLOCK) {
    const uint32_t n_block = min(a.cover.ctr->n_block, a.cover.unit_cap);
    // (entries differ by their edges, so a workgroup takes the next one when
    // it is done; the counter's answer arrives during the window)
    __shared__ uint32_t s_next;
    for (uint32_t u = blockIdx.x; u < n_block;) {
      uint32_t next = 0;
      if (threadIdx.x == 0) next = gridDim.x + atomicAdd(&a.cover.ctr->next, 1u);
      window(a.cover.block[u]);
      if (threadIdx.x == 0) s_next = next;
      __syncthreads();
      u = s_next;
      __syncthreads();
    }
  } else {
    const uint32_t wid = blockIdx.x * 4u + (uint32_t)wave, n_wid = gridDim.x * 4u;
    const uint32_t n_wave = min(a.cover.ctr->n_wave, a.cover.unit_cap);
    for (uint32_t u = wid; u < n_wave; u += n_wid) window(a.cover.wave[u]);
    // Small items: runs of the list, one item per lane, fewer per run where
    // there are not enough to go round.
    const uint32_t n_small = a.cover.ctr->n_small;
    const uint32_t run = min((uint32_t)RUN, (n_small + n_wid - 1u) / n_wid);
    for (uint32_t b = wid * run; b < n_small; b += n_wid * run) {
      const uint32_t n = min(run, n_small - b);
      CoverItem it{};
      uint32_t nv = 0, words = 0, rows = 0, job = 0;
      bool ok = false;
      if ((uint32_t)lane < n) {
        const u32x4* q = reinterpret_cast<const u32x4*>(a.desc + a.cover.small[b + (uint32_t)lane]);
        const u32x4 box = q[0], vq = q[1], fq = q[3];
        ok = (fq[2] & kItemMask) != 0;
        job = fq[0];
        nv = vq[2];
        it.set_box((int32_t)box[0], (int32_t)box[1], (int32_t)box[2], (int32_t)box[3], rows, words);
        it.lv = (int64_t)((uint64_t)vq[0] | ((uint64_t)vq[1] << 32));
        it.mask = fq[3];
      }
      cw.small_items(jobs_c, a.masks, it, ok, job, nv, words, rows);
    }
  }
}

// k_prep, k_item_desc and most of k_cover in one launch, for calls of few
// items, all polygons, that do not wait for totals: a wave takes an item, a
// lane per edge for its box (as k_prep, but in LDS), hands out its masks, and
// covers it right away unless it has many windows.
// These calls are bound by the latency of dependent loads and by the launches
// between them, two of which fall away: 1,000 stars on 2048 x 2048 take 35 us
// in all, with k_prep, k_item_desc and k_cover apart 41.  With more items
// than waves the packed items of k_cover win (32,000 items: 54 us against 70).
__global__ __launch_bounds__(64 * kItemsWaves) void k_items(ItemsArgs a) {
  __shared__ uint64_t s_tog[kItemsWaves * kCoverWave];
  __shared__ __align__(16) double s_edge[kItemsWaves][64][4];
  __shared__ CoverItem s_item[kItemsWaves][1];
  __shared__ uint64_t s_start[kItemsWaves][kStartWords];
  __shared__ ItemBox s_box[kItemsWaves];
  const int wave = wave_index(), lane = threadIdx.x & 63;
  const uint32_t base = (uint32_t)(wave * kCoverWave);
  const CoverWave cw{s_tog, s_edge[wave], s_item[wave], s_start[wave], base, lane, nullptr};
  const int64_t i = (int64_t)blockIdx.x * kItemsWaves + wave;
  const bool item = i < a.d.n_items;  // (uniform)
  const int j = a.d.n_jobs == 1 || !item ? 0 : __builtin_amdgcn_readfirstlane(find_job(a.d.job_iend, a.d.n_jobs, i));
  const RZ_CONST JobDev& J = as_const(a.d.jobs)[j];
  ItemDesc d;
  __builtin_memset(&d, 0, sizeof(d));
  if (item) {
    if (lane == 0) s_box[wave] = ItemBox{INT_MAX, INT_MIN, INT_MAX, INT_MIN};
    for (int k = lane; k < kCoverWave; k += 64) s_tog[base + (uint32_t)k] = 0ull;
    wave_sync();
    const int64_t v0 = J.item_vbeg[i - J.i_base], v1 = J.item_vbeg[i - J.i_base + 1];
    bool odd = false;
    for (int64_t lv = v0 + lane; lv - lane < v1; lv += 64) {
      const bool active = lv < v1;
      ItemBox box{INT_MAX, INT_MIN, INT_MAX, INT_MIN};
      if (active) {
        const int64_t ln = min(lv + 1, J.nv - 1);
        const uint64_t vi = J.vert_info[lv];
        const double X0 = J.xy[2 * lv], Y0 = J.xy[2 * lv + 1], X1 = J.xy[2 * ln], Y1 = J.xy[2 * ln + 1];
        auto px_x = [&](double X) { return isnan(X) ? X : to_pixel(X - J.xmin, J.xres, J.xinv); };
        auto px_y = [&](double Y) { return isnan(Y) ? Y : to_pixel(J.ymax - Y, J.yres, J.yinv); };
        PolyEdge e;
        polygon_edge(vi, px_x(X0), px_y(Y0), px_x(X1), px_y(Y1), J, a.edges != nullptr, e, box, odd);
        if (a.edges) a.edges[J.v_base + lv] = e;
      }
      reduce_box(lv, 0, box, 0, &s_box[wave], nullptr, active);
    }
    odd = __any(odd);
    wave_sync();
    d = make_desc(a.d, i, s_box[wave], odd ? kItemOddBit : 0ull);
  }
  // (lane 0 stands for the item)
  const bool poly = item && lane == 0 && d.nv > 0 && d.r0 < d.r1 && d.c0 < d.c1;
  bool small, own;
  const bool ok = assign_cover<kItemsWaves, false>(a.d.cover, poly, d, i, d.mask, small, own);
  if (!item) return;
  if (ok) d.flags |= kItemMask;
  if (lane == 0) a.d.desc[i] = d;
  if (!__any(ok && (small || own))) return;
  const bool odd = (d.flags & kItemOddRows) != 0;
  const int32_t n_win = (int32_t)cover_windows(mask_strip_count(d.r0, d.r1), mask_row_words(d.c0, d.c1), odd, false).n;
  const uint32_t mask = (uint32_t)__builtin_amdgcn_readfirstlane((int)d.mask);
  for (int32_t t = 0; t < n_win; ++t)
    cw.window<false>(J, a.masks, d.r0, d.r1, d.c0, d.c1, d.vbeg, (uint32_t)d.nv, odd, mask, t);
}

}  // namespace rzk
