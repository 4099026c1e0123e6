// rz_tile_t.h -- the tile kernel templates (k_tile, k_tile_lp): burn folds
// and the write-once store of every output tile.
// Instantiated per output dtype in rz_tile_inst.hip.
#pragma once

#include <type_traits>

#include "rz_device.h"

namespace rzk {

// Persistent work queue of the tile kernels.  A unit of work is one 16-row
// strip of one output tile, and wave w of every workgroup takes strip w, so
// the waves working on one strip index walk neighbouring tiles together
// (their stores fill neighbouring lines).  Workgroup b runs on XCD b % 8;
// each XCD owns a contiguous eighth of the launch's tiles, so neighbouring
// tiles share cache lines and items in that XCD's L2.  A wave's first tile
// is its workgroup's slot in that range (no atomic); after the first `slots`
// tiles, queue (x, w) hands out blocks of a.chunk consecutive tiles.  A grab
// is issued one block ahead, so its latency overlaps the current block.  A
// wave whose own XCD range is used up reads all eight counters of its strip
// with one relaxed load (counters only grow: a range that reads as used up
// is used up) and continues on the next XCD range with work left; jobs of
// very uneven size still end together, and every wave leaves when all eight
// ranges of its strip are used up.  The waves of a workgroup never
// synchronise with each other.
struct TileQueue {
  uint32_t n_loc, xcd, slots, B, cur_x, pending, t_cur, t_end;
  uint32_t* qbase;  // queue (x, w) at qbase + 4x * kQueueStride
  int lane;

  __device__ TileQueue(const TileArgs& a, int wave, int lane_) : lane(lane_) {
    n_loc = a.t_hi - a.t_lo;
    xcd = blockIdx.x % NUM_XCD;
    const uint32_t slot = blockIdx.x / NUM_XCD;
    slots = gridDim.x / NUM_XCD;
    B = a.chunk;
    qbase = a.queue + (uint32_t)wave * kQueueStride;
    cur_x = xcd;
    pending = 0;  // lane 0: result of the grab in flight on cur_x
    t_cur = xcd_unit_lo(xcd, n_loc) + slot;  // current block [t_cur, t_end)
    t_end = t_cur + 1u;
  }
  __device__ void issue(uint32_t x) {
    if (lane == 0) pending = atomicAdd(qbase + x * 4u * kQueueStride, 1u);
  }
  // first tile handed out by queue x's grab number c
  __device__ uint64_t grab_tile(uint32_t x, uint32_t c) const {
    return (uint64_t)xcd_unit_lo(x, n_loc) + slots + (uint64_t)c * B;
  }
  __device__ bool take(uint32_t x) {
    const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)pending, 0);
    const uint64_t s = grab_tile(x, c), xhi = xcd_unit_lo(x + 1u, n_loc);
    if (s >= xhi) return false;
    t_cur = (uint32_t)s;
    t_end = (uint32_t)min(s + (uint64_t)B, xhi);
    return true;
  }
  // (a grab on cur_x is always in flight when next_block runs)
  __device__ bool next_block() {
    if (take(cur_x)) return true;
    for (;;) {
      bool avail = false;
      if (lane < NUM_XCD) {
        const uint32_t seen = __hip_atomic_load(qbase + (uint32_t)lane * 4u * kQueueStride,
                                                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        avail = grab_tile((uint32_t)lane, seen) < (uint64_t)xcd_unit_lo((uint32_t)lane + 1u, n_loc);
      }
      const uint32_t m = (uint32_t)__ballot(avail) & 0xFFu;
      if (m == 0u) return false;
      const uint32_t rot = ((m >> xcd) | (m << (NUM_XCD - xcd))) & 0xFFu;
      const uint32_t x = (xcd + (uint32_t)__builtin_ctz(rot)) % NUM_XCD;
      issue(x);
      if (take(x)) {
        cur_x = x;
        return true;
      }
    }
  }
  // Whether the wave has a first tile (t_cur).
  __device__ bool begin() {
    bool have = t_cur < xcd_unit_lo(xcd + 1u, n_loc);
    issue(xcd);  // the grab after the first tile (or the first block, if there is no first tile)
    if (!have) {
      have = next_block();
      if (have) issue(cur_x);
    }
    return have;
  }
  // Local index of the current tile; moves to the next one.
  __device__ uint32_t pop() { return t_cur++; }
  // Whether there is a next tile (t_cur), taking the next block when needed.
  __device__ bool advance() {
    if (t_cur != t_end) return true;
    const bool have = next_block();
    if (have) issue(cur_x);
    return have;
  }
};

// Geometry of one unit: job, band, tile and strip window.
struct StripUnit {
  const RZ_CONST JobDev* J;
  uint32_t layer;
  int32_t nrows, ncols, C0, Rw, strip_r1, tile_c1;
};

// (row0: the unit's first row in its tile; rows: its rows; job: the last
// unit's job, tried first, as a wave's tiles mostly follow each other)
__device__ inline StripUnit strip_unit(const TileArgs& a, uint32_t t, int32_t row0, int32_t rows, int tw, int& job) {
  StripUnit u;
  u.J = &as_const(a.jobs)[job];
  if (t - u.J->tile_base >= u.J->n_tiles) {
    job = find_job(as_const(a.job_tend), a.n_jobs, (int64_t)t);
    u.J = &as_const(a.jobs)[job];
  }
  u.nrows = u.J->nrows;
  u.ncols = u.J->ncols;
  const uint32_t tj = t - u.J->tile_base;
  u.layer = tj / u.J->tiles_per_layer;
  const uint32_t tl = tj - u.layer * u.J->tiles_per_layer;
  const int32_t ty = (int32_t)(tl / (uint32_t)u.J->ntx), tx = (int32_t)(tl % (uint32_t)u.J->ntx);
  u.C0 = tx * tw;
  u.Rw = ty * TILE_H + row0;  // first row of the strip
  u.strip_r1 = min(u.Rw + rows, u.nrows);
  u.tile_c1 = min(u.C0 + tw, u.ncols);
  return u;
}

// The row words of an item without masks in a unit of ROWS rows, from its
// edges: word w of row r in lane r * 64 / ROWS + w - wlo.  One reading of the
// edges for all the tile words it meets, and of the words only the one where
// it meets no other (a word less per crossing to toggle and combine).
template <int NWORD, int ROWS>
__device__ __attribute__((always_inline)) inline uint64_t edge_words(const TileArgs& a, const ItemDesc& d, const StripUnit& u,
                                                                     PolyEdge* stage, int lane, int& wlo) {
  const uint32_t n = (uint32_t)d.nv;
  const int w0 = max(0, (d.c0 >> 6) - (u.C0 >> 6));
  if (NWORD > 1 && w0 < min(NWORD - 1, ((d.c1 - 1) >> 6) - (u.C0 >> 6))) {
    wlo = 0;
    return strip_coverage<NWORD, ROWS>(a.edges, d.vbeg, n, a.chunk_rows, u.Rw, u.strip_r1, u.C0, (double)u.ncols, stage, lane);
  }
  wlo = w0;
  return strip_coverage<1, ROWS>(a.edges, d.vbeg, n, a.chunk_rows, u.Rw, u.strip_r1, u.C0 + 64 * w0, (double)u.ncols, stage,
                                 lane);
}

// The rows that edge_words' words number w (from wlo on) cover in column lane
// of it, as bits: each row's word goes to the lanes of its number (mod 16),
// where a 16 x 16 transposition turns the 16 columns of a lane's quarter into
// row bits (about 30 instructions, where reading the words back row by row
// took 100).
template <int ROWS>
__device__ inline uint32_t word_bits(uint64_t words, int w, int lane) {
  constexpr int LPR = 64 / ROWS;
  const int from = (lane & (ROWS - 1)) * LPR + w;
  const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * from, (int)(uint32_t)words);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * from, (int)(uint32_t)(words >> 32));
  const uint32_t half = lane < 32 ? lo : hi;
  uint32_t x = (lane & 16 ? half >> 16 : half) & 0xFFFFu;
  if (ROWS < 16 && (lane & 15) >= ROWS) x = 0u;
  return transpose16x2(x, lane) & 0xFFFFu;
}

// edge_words and word_bits for one word of a 16-row unit, as a function of its
// own: items without masks are rare in k_tile_lp, and inlined this took
// registers from all its calls (31 spilled of float's instead of 22, 2 waves
// per SIMD of double's instead of 3: 500,000 lines on 20000^2 float32 8.15 ms
// a call instead of 7.9, 7,000 on 2199 x 2923 float64 170 us in the kernel
// instead of 163).  Arguments arrive in vector registers; all but the lane are
// uniform.
__device__ __attribute__((noinline)) inline uint32_t edge_bits(const PolyEdge* edges, int64_t vbeg, int32_t nv,
                                                               const int2* chunk_rows, int32_t Rw, int32_t strip_r1,
                                                               int32_t C0, int32_t ncols, RZ_LDS PolyEdge* stage, int lane) {
  auto u32 = [](int32_t x) { return __builtin_amdgcn_readfirstlane(x); };
  auto u64 = [&](uint64_t x) {
    return (uint64_t)(uint32_t)u32((int32_t)x) | (uint64_t)(uint32_t)u32((int32_t)(x >> 32)) << 32;
  };
  const uint64_t cov = strip_coverage<1, WAVE_ROWS>((const PolyEdge*)u64((uint64_t)edges), (int64_t)u64((uint64_t)vbeg),
                                                    (uint32_t)u32(nv), (const int2*)u64((uint64_t)chunk_rows), u32(Rw),
                                                    u32(strip_r1), u32(C0), (double)u32(ncols), (PolyEdge*)stage, lane);
  return word_bits<WAVE_ROWS>(cov, 0, lane);
}

// The rows any polygon item covers in column lane of tile word w, for a unit
// of 16 rows (k_tile_lp).
__device__ inline uint32_t column_bits(const TileArgs& a, const ItemDesc& d, const StripUnit& u, int w, PolyEdge* stage,
                                       int lane) {
  const int32_t wi = (u.C0 >> 6) + w - (d.c0 >> 6), nw = mask_row_words(d.c0, d.c1);
  if (wi < 0 || wi >= nw) return 0u;
  if (!(d.flags & kItemMask))
    return edge_bits(a.edges, d.vbeg, d.nv, a.chunk_rows, u.Rw, u.strip_r1, u.C0 + 64 * w, u.ncols, (RZ_LDS PolyEdge*)stage, lane);
  const uint64_t* p = a.masks + ((uint64_t)d.mask + (uint64_t)((u.Rw >> 4) - (d.r0 >> 4)) * (uint64_t)nw + (uint64_t)wi) * 16u;
  return reinterpret_cast<const uint16_t*>(p)[lane];
}

// Writes a strip once: lane l's chunk of PPC pixels in rows
// srow + k * RSTEP (k < RPL) starting at column C0 + ccol, from `chunk(k)`
// (16 bytes); each store instruction covers RSTEP whole tile rows.
template <typename T, int PPC, int RPL, int RSTEP, typename F>
__device__ inline void store_strip(const StripUnit& u, int srow, int ccol, F&& chunk) {
  const int32_t c = u.C0 + ccol;
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    const int32_t row = u.Rw + srow + k * RSTEP;
    if (row < u.nrows) {
      T* orow = (T*)u.J->out + ((uint64_t)u.layer * (uint64_t)u.nrows + (uint64_t)row) * (uint64_t)u.ncols;
      const u32x4 vec = chunk(k);
      if (c + PPC <= u.ncols && ((uintptr_t)(orow + c) & 15u) == 0) {
        __builtin_nontemporal_store(vec, (u32x4*)(orow + c));
      } else {
        T px[PPC];
        __builtin_memcpy(px, &vec, 16);
#pragma unroll
        for (int j = 0; j < PPC; ++j)
          if (c + j < u.ncols) orow[c + j] = px[j];
      }
    }
  }
}

// A unit's pixels in registers: lane l owns column 64 w + l of every row.
// 4- and 8-byte pixels take a register (pair) each, px[w * ROWS + r]; 1- and
// 2-byte pixels are packed, RPW rows of one column to a word, and folded
// together.
template <typename T, int ROWS>
struct Pixels {
  static constexpr bool PACKED = sizeof(T) <= 2;
  static constexpr int RPW = PACKED ? 4 / (int)sizeof(T) : 1;
  static constexpr int NWORD = tile_w(sizeof(T)) / 64;
  using W = typename std::conditional<PACKED, uint32_t, T>::type;
  W px[NWORD * ROWS / RPW];
  __device__ void fill(const StripUnit& u) {
    W bg;
    if constexpr (PACKED) bg = lane_splat<T>(u.J->bg_bits);
    else bg = from_bits<T>(u.J->bg_bits);
#pragma unroll
    for (int j = 0; j < NWORD * ROWS / RPW; ++j) px[j] = bg;
  }
  // One write of the value bits v in the rows `bits` of tile word w (rows
  // outside [lo, hi) have none).  A packed sum or count over a background of
  // 0 is a plain addition of 0 or the value: the empty pixel's rule gives
  // the same.
  template <int FUN>
  __device__ __attribute__((always_inline)) void fold(int w, uint32_t bits, int lo, int hi, uint64_t v, uint64_t bg_bits) {
    if constexpr (PACKED) {
      const uint32_t bgw = lane_splat<T>(bg_bits);
      const uint32_t vw = FUN == 5 ? Lanes<sizeof(T)>::one : lane_splat<T>(v);
      const bool plain = bgw == 0u;
#pragma unroll
      for (int d = 0; d < ROWS / RPW; ++d)
        if (lo < (d + 1) * RPW && hi > d * RPW) {
          const uint32_t b = (bits >> (d * RPW)) & ((1u << RPW) - 1u);
          W& x = px[w * (ROWS / RPW) + d];
          const uint32_t m = lane_mask<(int)sizeof(T)>(b);
          if constexpr (FUN == 0 || FUN == 5) {
            uint32_t y = lane_add<sizeof(T)>(x, vw & m);
            if (!plain) {
              const uint32_t e = lane_eq<sizeof(T)>(x, bgw) & m;
              y = (e & vw) | (~e & y);
            }
            x = y;
          } else {
            x = fold_word<T, FUN>(x, vw, bgw, m);
          }
        }
    } else {
      const T val = from_bits<T>(v), bg = from_bits<T>(bg_bits);
#pragma unroll
      for (int r0 = 0; r0 < ROWS; r0 += 4)
        if (lo < r0 + 4 && hi > r0) {
#pragma unroll
          for (int r = r0; r < r0 + 4; ++r) {
            T& x = px[w * ROWS + r];
            x = bit_select(bit_mask(bits, r), fold_value<T, FUN>(x, val, bg), x);
          }
        }
    }
  }
};

// Packed pixels (1- and 2-byte outputs) as rows: f(r, v) with the dwords v of
// lane l's columns 4 l .. 4 l + 3 in row r, the rows of a dword at a time,
// exchanged across the lanes in LDS and transposed.  `x`: 256 words of
// wave-private LDS.
template <typename T, int ROWS, typename F>
__device__ inline void each_row(const uint32_t* px, uint32_t* x, int lane, F&& f) {
  constexpr int RPW = 4 / (int)sizeof(T);  // rows (pixels) per dword
  constexpr int ND = ROWS / RPW;
#pragma unroll
  for (int d = 0; d < ND; ++d) {
#pragma unroll
    for (int w = 0; w < 4; ++w) x[w * 64 + lane] = px[w * ND + d];
    wave_sync();
    const u32x4 c = *reinterpret_cast<const u32x4*>(x + 4 * lane);  // columns 4 lane .. + 3, RPW rows each
    wave_sync();
    uint32_t v[RPW][sizeof(T)];
    if constexpr (sizeof(T) == 1) {
      // 4 x 4 bytes transposed: pairs of columns, then of pairs
      const uint32_t a01 = __builtin_amdgcn_perm(c[1], c[0], 0x05010400u), a23 = __builtin_amdgcn_perm(c[3], c[2], 0x05010400u);
      const uint32_t b01 = __builtin_amdgcn_perm(c[1], c[0], 0x07030602u), b23 = __builtin_amdgcn_perm(c[3], c[2], 0x07030602u);
      v[0][0] = __builtin_amdgcn_perm(a23, a01, 0x05040100u);
      v[1][0] = __builtin_amdgcn_perm(a23, a01, 0x07060302u);
      v[2][0] = __builtin_amdgcn_perm(b23, b01, 0x05040100u);
      v[3][0] = __builtin_amdgcn_perm(b23, b01, 0x07060302u);
    } else {
      v[0][0] = __builtin_amdgcn_perm(c[1], c[0], 0x05040100u);
      v[0][1] = __builtin_amdgcn_perm(c[3], c[2], 0x05040100u);
      v[1][0] = __builtin_amdgcn_perm(c[1], c[0], 0x07060302u);
      v[1][1] = __builtin_amdgcn_perm(c[3], c[2], 0x07060302u);
    }
#pragma unroll
    for (int j = 0; j < RPW; ++j) f(d * RPW + j, v[j]);
  }
}

// The 4 (1-byte) or 8 bytes of a lane's four pixels.
template <typename T>
struct Quad {
  typedef uint32_t vec __attribute__((ext_vector_type(sizeof(T)), aligned(1)));
};
template <>
struct Quad<uint8_t> {
  typedef uint32_t vec __attribute__((aligned(1)));
};
template <>
struct Quad<int8_t> : Quad<uint8_t> {};

// Writes four neighbouring pixels of a row from column c on; `part`: those in
// [lo, hi) only.
template <typename T>
__device__ inline void put_quad(T* orow, int32_t c, bool part, int32_t lo, int32_t hi, const uint32_t (&v)[sizeof(T)]) {
  if (!part || (c >= lo && c + 4 <= hi)) {
    typename Quad<T>::vec y;
    __builtin_memcpy(&y, v, 4 * sizeof(T));
    __builtin_nontemporal_store(y, (typename Quad<T>::vec*)(orow + c));
  } else {
    T px[4];
    __builtin_memcpy(px, v, sizeof(px));
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (c + k >= lo && c + k < hi) orow[c + k] = px[k];
  }
}

// Writes a unit's rows (background + burns), each pixel once.
template <typename T, int ROWS>
__device__ inline void store_rows(const StripUnit& u, const Pixels<T, ROWS>& p, uint32_t* x, int lane) {
  T* out = (T*)u.J->out + ((uint64_t)u.layer * (uint64_t)u.nrows + (uint64_t)u.Rw) * (uint64_t)u.ncols;
  if constexpr (sizeof(T) >= 4) {
    if (u.C0 + lane < u.ncols) {
      // the address moves down a row in vector registers (the asm keeps it
      // there), and rows are only counted in a strip that ends the raster:
      // written as offsets from the first row, a row took up to 11 scalar
      // instructions, half of those of a strip that nothing meets
      T* at = out + u.C0 + lane;
      const uint64_t ncols = (uint64_t)u.ncols;
      const int n = u.nrows - u.Rw;
      if (n >= ROWS) {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
          __builtin_nontemporal_store(p.px[r], at);
          at += ncols;
          asm volatile("" : "+v"(at));
        }
      } else {
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
          if (r < n) __builtin_nontemporal_store(p.px[r], at);
          at += ncols;
          asm volatile("" : "+v"(at));
        }
      }
    }
  } else {
    const bool part = u.C0 + tile_w(sizeof(T)) > u.ncols;
    each_row<T, ROWS>(p.px, x, lane, [&](int r, const uint32_t (&v)[sizeof(T)]) {
      if (u.Rw + r < u.nrows) put_quad<T>(out + (uint64_t)r * (uint64_t)u.ncols, u.C0 + 4 * lane, part, 0, u.ncols, v);
    });
  }
}

// The strips of a wave's consecutive tiles, written in whole 128-byte lines
// wherever a row starts: a unit writes a row from the last line start at or
// before its first column on, with the columns before that from the unit to
// its left, which it left out.  (A 256-byte piece of a row that starts
// inside a line takes three lines, two of them in part: 2.3 times as long for
// float32 of 40,008 columns as of 40,000.)  A unit whose left neighbour was
// another wave's starts at its own first column, and one whose right
// neighbour is writes its last columns too.
template <typename T>
struct LineWriter {
  static constexpr int ROWS = WAVE_ROWS, TW = tile_w(sizeof(T));
  static constexpr int LINE = 128 / (int)sizeof(T);      // pixels of a line
  static constexpr bool NARROW = sizeof(T) <= 2;
  // the pixels left out, in LDS (registers would cost a wave per SIMD): the
  // last LINE pixels of every row, PITCH words apart; narrow ones are
  // followed by room for the row itself
  uint32_t* tail;
  static constexpr int PITCH = NARROW ? (LINE + TW) * (int)sizeof(T) / 4 + 1 : 32;

  __device__ static uint32_t skew(const T* p) { return ((uint32_t)(uintptr_t)p & 127u) / (uint32_t)sizeof(T); }

  // cont: the unit to the left left its last pixels out; more: the unit to
  // the right will write this one's.
  __device__ void store(const StripUnit& u, const Pixels<T, ROWS>& p, uint32_t* x, int lane, bool cont, bool more) {
    T* out = (T*)u.J->out + ((uint64_t)u.layer * (uint64_t)u.nrows + (uint64_t)u.Rw) * (uint64_t)u.ncols;
    if ((skew(out) | ((uint32_t)u.ncols % (uint32_t)LINE)) == 0u) {  // every row starts a line
      store_rows<T, ROWS>(u, p, x, lane);
      return;
    }
    if constexpr (!NARROW) {
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        if (u.Rw + r < u.nrows) {
          T* orow = out + (uint64_t)r * (uint64_t)u.ncols;
          const int32_t s = (int32_t)skew(orow + u.C0);
          // lane l: column C0 - s + l, from lane l - s of this unit or from the
          // last pixels of the one to the left
          T* last = reinterpret_cast<T*>(tail + r * PITCH);
          const T left = last[(LINE - s + lane) & (LINE - 1)];
          const T v = p.px[r];
          const int from = ((lane - s) & 63) * 4;
          T y;
          if constexpr (sizeof(T) == 8) {
            uint2 w;
            __builtin_memcpy(&w, &v, 8);
            w.x = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)w.x);
            w.y = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)w.y);
            __builtin_memcpy(&y, &w, 8);
          } else {
            int w;
            __builtin_memcpy(&w, &v, 4);
            w = __builtin_amdgcn_ds_bpermute(from, w);
            __builtin_memcpy(&y, &w, 4);
          }
          if (lane < s) y = left;
          const int32_t c = u.C0 - s + lane;
          if ((cont || lane >= s) && c < u.ncols) __builtin_nontemporal_store(y, orow + c);
          if (!more && lane >= 64 - s && u.C0 + lane < u.ncols) orow[u.C0 + lane] = p.px[r];
          wave_sync();
          if (lane >= 64 - LINE) last[lane - (64 - LINE)] = p.px[r];
        }
      }
    } else {
      constexpr int LW = LINE * (int)sizeof(T) / 4, NW = (int)sizeof(T);  // words of a line, of a lane's pixels
      each_row<T, ROWS>(p.px, x, lane, [&](int r, const uint32_t (&v)[sizeof(T)]) {
#pragma unroll
        for (int k = 0; k < NW; ++k) tail[r * PITCH + LW + lane * NW + k] = v[k];
      });
      wave_sync();
      const bool part = !cont || u.C0 + TW > u.ncols;
      const int n = min(ROWS, u.nrows - u.Rw);
      for (int r = 0; r < n; ++r) {
        T* orow = out + (uint64_t)r * (uint64_t)u.ncols;
        const int32_t s = (int32_t)skew(orow + u.C0);
        const int32_t b = LW * 4 + (4 * lane - s) * NW;  // byte of the row's buffer
        const uint32_t* t = tail + r * PITCH;
        uint32_t w[NW + 1], y[NW];
#pragma unroll
        for (int k = 0; k <= NW; ++k) w[k] = t[(b >> 2) + k];
#pragma unroll
        for (int k = 0; k < NW; ++k) y[k] = __builtin_amdgcn_alignbyte(w[k + 1], w[k], (uint32_t)b & 3u);
        put_quad<T>(orow, u.C0 - s + 4 * lane, part, cont ? 0 : u.C0, u.ncols, y);
      }
      for (int r = 0; r < n && !more; ++r) {
        T* orow = out + (uint64_t)r * (uint64_t)u.ncols;
        const int32_t s = (int32_t)skew(orow + u.C0);
        uint32_t y[NW];
#pragma unroll
        for (int k = 0; k < NW; ++k) y[k] = tail[r * PITCH + LW + lane * NW + k];
        if (4 * lane + 4 > TW - s) put_quad<T>(orow, u.C0 + 4 * lane, true, u.C0 + TW - s, u.ncols, y);
      }
      // the last line of every row is the next unit's first
      for (int k = lane; k < ROWS * LW; k += 64) {
        const int r = k / LW, j = k % LW;
        tail[r * PITCH + j] = tail[r * PITCH + TW * NW / 4 + j];
      }
      wave_sync();
    }
  }
};

// A lane's polygon item of a batch of up to 64: as loaded, then what the
// folds need of it in one unit.
struct RawItem {
  u32x4 box, fq;      // r0, r1, c0, c1; job, band, flags, mask
  uint32_t kl, v0, v1;  // kind | band, value
};
__device__ inline RawItem load_raw(const ItemDesc* d) {
  const u32x4* q = reinterpret_cast<const u32x4*>(d);
  const u32x4 a = q[1], b = q[2];
  return RawItem{q[0], q[3], a[3], b[0], b[1]};
}
// Up to 64 visits of a unit in order, visit k in lane k: an item (its value
// bits v0, v1) and a column of 64 it meets.
struct Visits {
  uint32_t blk;   // the mask block
  uint32_t v0, v1;
  uint32_t info;  // tile word, first row << 8, row end << 16, no masks << 31
  uint32_t item;  // lane of the item's descriptor in its batch
  uint32_t n;     // visits (uniform)
};

__device__ inline uint32_t push_lane(uint32_t v, uint32_t to) {
  return (uint32_t)__builtin_amdgcn_ds_permute((int)(to * 4u), (int)v);
}

// The visits of the batch's items q (lanes `cand`) that meet the unit.  At
// most 64: `left` returns the lanes whose items did not fit (0 with one word
// per row), to be passed as `cand` again.  `x`: 256 words of wave-private LDS
// (more than one word per row).  Every lane calls it.
template <int NWORD, int ROWS, bool WIDE_VALUE>
__device__ inline Visits visits_of(const RawItem& q, const StripUnit& u, bool cand, uint64_t& left, uint32_t* x) {
  const int lane = threadIdx.x & 63;
  const int32_t r0 = (int32_t)q.box[0], r1 = (int32_t)q.box[1], c0 = (int32_t)q.box[2], c1 = (int32_t)q.box[3];
  bool hit = cand && r0 < u.strip_r1 && r1 > u.Rw && c0 < u.tile_c1 && c1 > u.C0 && r0 < r1 && c0 < c1 &&
             (q.kl >> 2) == u.layer;
  const int32_t nw = mask_row_words(c0, c1);
  const int32_t wlo = max(0, (c0 >> 6) - (u.C0 >> 6)), whi = min(NWORD - 1, ((c1 - 1) >> 6) - (u.C0 >> 6));
  const int32_t wi = (u.C0 >> 6) + wlo - (c0 >> 6);  // the item's word in tile word wlo
  const bool bare = !(q.fq[2] & kItemMask);
  const uint32_t blk = bare ? 0u : q.fq[3] + (uint32_t)((u.Rw >> 4) - (r0 >> 4)) * (uint32_t)nw + (uint32_t)wi;
  const uint32_t info = (uint32_t)wlo | (uint32_t)min(max(r0 - u.Rw, 0), ROWS - 1) << 8 |
                        (uint32_t)min(max(r1 - u.Rw, 0), ROWS) << 16 | (bare ? 1u << 31 : 0u);
  Visits v{0u, 0u, 0u, 0u, 0u, 0u};
  left = 0ull;
  if constexpr (NWORD == 1) {
    const uint64_t m = __ballot(hit);
    v.n = (uint32_t)__popcll(m);
    // (a permutation of all lanes: the others go after the visits)
    const uint64_t below = (1ull << lane) - 1ull;
    const uint32_t to = hit ? (uint32_t)__popcll(m & below) : v.n + (uint32_t)__popcll(~m & below);
    v.blk = push_lane(blk, to);
    v.v0 = push_lane(q.v0, to);
    if (WIDE_VALUE) v.v1 = push_lane(q.v1, to);
    v.info = push_lane(info, to);
    v.item = push_lane((uint32_t)lane, to);
  } else {
    const uint32_t words = hit ? (uint32_t)(whi - wlo + 1) : 0u;
    const uint32_t end = wave_prefix_sum(words);
    const bool fits = end <= 64u;
    left = __ballot(hit && !fits);
    hit = hit && fits;
    const uint64_t m = __ballot(hit);
    if (m) v.n = (uint32_t)__builtin_amdgcn_readlane((int)end, 63 - __builtin_clzll(m));
    wave_sync();
    if (hit)
      for (uint32_t j = 0; j < words; ++j)
        *reinterpret_cast<uint4*>(x + 4u * (end - words + j)) = make_uint4(bare ? 0u : blk + j, q.v0, info + j, (uint32_t)lane);
    wave_sync();
    if ((uint32_t)lane < v.n) {
      const uint4 y = *reinterpret_cast<const uint4*>(x + 4 * lane);
      v.blk = y.x;
      v.v0 = y.y;
      v.info = y.z;
      v.item = y.w;
    }
    wave_sync();
  }
  return v;
}

// Visits whose mask blocks are loaded ahead of their folds (more cost waves;
// 4-byte pixels with 1 and 7 waves: 5.34 ms where 2 take 5.17).
template <typename T>
constexpr int kAhead = sizeof(T) == 8 ? 3 : 2;

// The column bits (16 rows) of visits k .. k + N - 1 (past the last one: the
// last one's again).
template <int N>
__device__ inline void load_bits(const TileArgs& a, const Visits& v, uint32_t k, uint32_t (&bits)[N], int lane) {
  const uint16_t* base = reinterpret_cast<const uint16_t*>(a.masks) + lane;
#pragma unroll
  for (int g = 0; g < N; ++g) {
    const uint32_t blk = (uint32_t)__builtin_amdgcn_readlane((int)v.blk, (int)min(k + (uint32_t)g, v.n - 1u));
    bits[g] = base[(uint64_t)blk * 64u];
  }
}

// Folds the visits in order; `bits` holds the first N ones' column bits
// (load_bits).  Lane l owns column 64 w + l of every row, so its 16 row bits
// come with one load and each row takes a bit extract, the fold (1 to 5
// instructions) and a bit select.  (Spreading a row over the lanes that
// store it took about 80 instructions per item and strip before the folds,
// and computing the coverage in the strip about 200.  Reading the masks as
// execution masks through scalar loads needs half the vector instructions,
// but the scalar cache's misses bound it.)
template <typename T, int FUN, int ROWS>
__device__ __attribute__((always_inline)) inline void fold_visit(const TileArgs& a, const StripUnit& u, Pixels<T, ROWS>& p,
                                                                 const Visits& v, uint32_t k, uint32_t y, uint32_t& burns) {
  constexpr int NWORD = Pixels<T, ROWS>::NWORD;
  const uint32_t info = (uint32_t)__builtin_amdgcn_readlane((int)v.info, (int)k);
  const uint32_t v0 = (uint32_t)__builtin_amdgcn_readlane((int)v.v0, (int)k);
  const uint32_t v1 = sizeof(T) == 8 ? (uint32_t)__builtin_amdgcn_readlane((int)v.v1, (int)k) : 0u;
  if (a.burns) burns += (uint32_t)__popc(y);
  const int lo = (int)((info >> 8) & 31u), hi = (int)((info >> 16) & 31u);
#pragma unroll
  for (int w = 0; w < NWORD; ++w)
    if (NWORD == 1 || (info & 3u) == (uint32_t)w) {  // (uniform)
      p.template fold<FUN>(w, y, lo, hi, (uint64_t)v0 | ((uint64_t)v1 << 32), u.J->bg_bits);
    }
}
// The unit's rows of a mask block's 16.
template <int ROWS>
__device__ inline uint32_t unit_rows(const StripUnit& u, uint32_t y) {
  return ROWS < 16 ? (y >> (u.Rw & 15)) & ((1u << ROWS) - 1u) : y;
}
template <typename T, int FUN, int ROWS, int N>
__device__ inline void fold_visits(const TileArgs& a, const StripUnit& u, Pixels<T, ROWS>& p, const Visits& v,
                                   uint32_t k0, uint32_t end, uint32_t (&bits)[N], int lane, uint32_t& burns) {
  constexpr int NWORD = Pixels<T, ROWS>::NWORD;
  const int shift = ROWS < 16 ? (u.Rw & 15) : 0;
  auto fold = [&](uint32_t k, uint32_t y) __attribute__((always_inline)) {
    const uint32_t info = (uint32_t)__builtin_amdgcn_readlane((int)v.info, (int)k);
    const uint32_t v0 = (uint32_t)__builtin_amdgcn_readlane((int)v.v0, (int)k);
    const uint32_t v1 = sizeof(T) == 8 ? (uint32_t)__builtin_amdgcn_readlane((int)v.v1, (int)k) : 0u;
    if (a.burns) burns += (uint32_t)__popc(y);
    const int lo = (int)((info >> 8) & 31u), hi = (int)((info >> 16) & 31u);
#pragma unroll
    for (int w = 0; w < NWORD; ++w)
      if (NWORD == 1 || (info & 3u) == (uint32_t)w) {  // (uniform)
        p.template fold<FUN>(w, y, lo, hi, (uint64_t)v0 | ((uint64_t)v1 << 32), u.J->bg_bits);
      }
  };
  auto rows = [&](uint32_t y) { return ROWS < 16 ? (y >> shift) & ((1u << ROWS) - 1u) : y; };
  for (uint32_t k = k0; k < end; k += (uint32_t)N) {
    uint32_t nxt[N] = {};
    const bool more = k + (uint32_t)N < end;
    if (more) load_bits(a, v, k + (uint32_t)N, nxt, lane);
#pragma unroll
    for (int g = 0; g < N; ++g)
      if (k + (uint32_t)g < end) fold(k + (uint32_t)g, rows(bits[g]));
    if (more) {
#pragma unroll
      for (int g = 0; g < N; ++g) bits[g] = nxt[g];
    }
  }
}

// Whether items without masks are among the visits.
__device__ inline bool any_bare(const Visits& v, int lane) { return __any((uint32_t)lane < v.n && (v.info >> 31)); }
// ... then fold(k, bits) for one visit after the other; desc_of: the
// descriptor of the item in a lane of the batch.
template <int NWORD, int ROWS, typename D, typename F>
__device__ __attribute__((always_inline)) inline void bare_visits(const TileArgs& a, const StripUnit& u, const Visits& v,
                                                                  PolyEdge* stage, int lane, D&& desc_of, F&& fold) {
  uint64_t words = 0ull;  // the row words of the item in lane `at`
  int at = -1, wlo = 0;
  for (uint32_t k = 0; k < v.n; ++k) {
    const uint32_t info = (uint32_t)__builtin_amdgcn_readlane((int)v.info, (int)k);
    // (what is computed of the lane alone is computed here each time: kept
    // from before the loop it would take 20 registers of all calls)
    int l = lane;
    asm volatile("" : "+v"(l));
    uint32_t y;
    if (info >> 31) {
      const int item = __builtin_amdgcn_readlane((int)v.item, (int)k);
      if (NWORD == 1 || item != at) words = edge_words<NWORD, ROWS>(a, desc_of(item), u, stage, l, wlo);
      at = item;
      y = word_bits<ROWS>(words, (int)(info & 3u) - wlo, l);
    } else {
      uint32_t one[1];
      load_bits(a, v, k, one, l);
      y = unit_rows<ROWS>(u, one[0]);
    }
    fold(k, y);
  }
}

// Waves per SIMD the register allocation of k_tile targets: 7 for 4-byte
// pixels (a million polygons on 40000^2 float32 in 8 bands, about one item to
// a tile: 10.9 ms a call, with 8 waves 11.5; with 5 waves and 6 visits ahead it
// was 14.3 where 7 took 12.1), 5 for 8-byte ones (24 uneven jobs 3.85 ms, with
// 4 waves 4.04), 3 for 2-byte ones (LineWriter's rows take the LDS of more); 4
// where more would spill.
template <typename T, bool BARE>
struct TileOccupancy {
  static constexpr int value = sizeof(T) == 2 ? 3 : (sizeof(T) == 1 || BARE ? 4 : (sizeof(T) == 4 ? 7 : 5));
};

// Tile kernel of polygon-only groups, one launch per pixel-function group of
// a batch (a single call is a batch of one job).
//
// Per unit (16 rows x TW columns of the job's output): the background fill
// of RasterInfo::build_raster (rust/src/geo/raster.rs:23-28) and every write
// of every item meeting the strip, folded in geometry order in registers
// (fold_visits), then written to HBM once.
//
// The masks and descriptors come from HBM, about 2 us away while the strips
// are written, and the loads of one strip depend on each other (range,
// descriptors, masks), so a wave works on four units at once: it folds one
// (A) while the masks of the next (B), the descriptors of the one after (C)
// and the range of the last (D) are loading.  A wait for a load waits for
// everything issued before it, stores included, so all loads of a step are
// issued at its start, arrive during the fold and are waited for once, after
// it; the strip is stored last, and its stores complete during the next fold.
// BARE: compiled with the path for items without masks (its registers would
// cost the other calls spills).
template <typename T, int FUN, bool BARE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(TileOccupancy<T, BARE>::value))) void k_tile(TileArgs a) {
  constexpr int TW = tile_w(sizeof(T));
  constexpr int NWORD = TW / 64;  // mask words per row
  __shared__ PolyEdge s_edge[BARE ? 4 : 1][64];
  __shared__ __align__(16) uint32_t s_x[4][NWORD > 1 ? 256 : 1];
  __shared__ __align__(16) uint32_t s_tail[4][WAVE_ROWS * LineWriter<T>::PITCH];

  const int wave = wave_index(), lane = threadIdx.x & 63;
  uint32_t burns = 0;
  TileQueue tq(a, wave, lane);
  const RZ_CONST uint32_t* toff_c = as_const(a.tile_off);
  int job = 0;

  // a unit's candidates: the tile's list (binned jobs) or the items of the job
  struct Range {
    const ItemDesc* list;
    int64_t ib, ie;
  };
  constexpr bool WIDE = sizeof(T) == 8;
  struct Unit {
    StripUnit u;
    Range g;
    bool have;
  };
  auto pop_unit = [&](bool have) {  // the next unit, its range loading
    Unit x{};
    x.have = have;
    if (have) {
      const uint32_t t = a.t_lo + tq.pop();
      uint32_t pb = 0, pe = 0;
      if (a.tile_off) {
        pb = toff_c[t];
        pe = toff_c[t + 1u];
      }
      x.u = strip_unit(a, t, wave * WAVE_ROWS, WAVE_ROWS, TW, job);
      x.g = x.u.J->scan ? Range{a.desc, x.u.J->i_base, x.u.J->i_base + x.u.J->ni}
                        : Range{a.pair_desc, (int64_t)pb, (int64_t)pe};
    }
    return x;
  };
  auto load_first = [&](const Unit& x) {
    RawItem q{};
    if (x.have && x.g.ib + lane < x.g.ie) q = load_raw(x.g.list + x.g.ib + lane);
    return q;
  };
  auto first_visits = [&](const Unit& x, const RawItem& q, uint64_t& left) {
    return visits_of<NWORD, WAVE_ROWS, WIDE>(q, x.u, x.have && x.g.ib + lane < x.g.ie, left, s_x[wave]);
  };

  // (batch: the first of the items whose lanes v.item names)
  auto fold = [&](const StripUnit& u, Pixels<T, WAVE_ROWS>& p, const Visits& v, uint32_t (&bits)[kAhead<T>],
                  const ItemDesc* batch) __attribute__((always_inline)) {
    if constexpr (BARE) {
      if (any_bare(v, lane)) {
        bare_visits<NWORD, WAVE_ROWS>(
            a, u, v, s_edge[wave], lane, [&](int b) { return load_desc(as_const(batch) + b); },
            [&](uint32_t k, uint32_t y) __attribute__((always_inline)) { fold_visit<T, FUN, WAVE_ROWS>(a, u, p, v, k, y, burns); });
        return;
      }
    }
    fold_visits<T, FUN, WAVE_ROWS>(a, u, p, v, 0u, v.n, bits, lane, burns);
  };

  Unit A = pop_unit(tq.begin()), B{}, C{};
  if (A.have) B = pop_unit(tq.advance());
  if (B.have) C = pop_unit(tq.advance());
  uint64_t left_a = 0, left_b = 0;  // lanes of the first batch whose visits are still to come
  uint32_t bits_a[kAhead<T>] = {};
  Visits va{}, vb{};
  if (A.have) {
    const RawItem qa = load_first(A), qb = load_first(B);
    va = first_visits(A, qa, left_a);
    vb = first_visits(B, qb, left_b);
    if (va.n) load_bits(a, va, 0u, bits_a, lane);
  }
  LineWriter<T> lines;
  lines.tail = s_tail[wave];
  bool cont = false;
  while (A.have) {
    uint32_t bits_b[kAhead<T>] = {};
    if (vb.n) load_bits(a, vb, 0u, bits_b, lane);
    const RawItem qc = load_first(C);
    const Unit D = pop_unit(C.have && tq.advance());

    Pixels<T, WAVE_ROWS> p;
    p.fill(A.u);
    if (va.n)
      fold(A.u, p, va, bits_a, A.g.list + A.g.ib);
    // the candidates past the first batch (64 items or visits), in order; scan
    // jobs of one band test the 8-byte boxes in strip and tile units first
    for (int64_t base = A.g.ib; left_a || base + 64 < A.g.ie;) {
      bool cand;
      if (NWORD > 1 && left_a) {
        cand = (left_a >> lane) & 1ull;
      } else {
        base += 64;
        cand = base + lane < A.g.ie;
        if (cand && A.u.J->scan && A.u.J->scan_compact && a.scan_box)
          cand = scan_box_meets(a.scan_box[base + lane], (uint32_t)A.u.Rw / WAVE_ROWS, (uint32_t)A.u.C0 / (uint32_t)TW);
      }
      RawItem q{};
      if (cand) q = load_raw(A.g.list + base + lane);
      const Visits v = visits_of<NWORD, WAVE_ROWS, WIDE>(q, A.u, cand, left_a, s_x[wave]);
      if (!v.n) continue;
      uint32_t bits[kAhead<T>];
      load_bits(a, v, 0u, bits, lane);
      fold(A.u, p, v, bits, A.g.list + base);
    }

    // everything loaded has arrived
#pragma unroll
    for (int g = 0; g < kAhead<T>; ++g) asm volatile("" : "+v"(bits_b[g]));
    asm volatile("" : "+v"(tq.pending));
    uint64_t left_c = 0;
    const Visits vc = first_visits(C, qc, left_c);
    // (neighbours: the next tile of the same rows)
    const bool more = B.have && B.u.J == A.u.J && B.u.layer == A.u.layer && B.u.Rw == A.u.Rw && B.u.C0 == A.u.C0 + TW;
    lines.store(A.u, p, s_x[wave], lane, cont, more);
    cont = more;
    A = B;
    B = C;
    C = D;
    va = vb;
    vb = vc;
    left_a = left_b;
    left_b = left_c;
#pragma unroll
    for (int g = 0; g < kAhead<T>; ++g) bits_a[g] = bits_b[g];
  }
  if (a.burns) {
    unsigned long long n = burns;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
    if (lane == 0 && n) atomicAdd(&a.burns[blockIdx.x % kBurnSlots], n);
  }
}

// The same for launches of few tiles, where latency counts: a workgroup per
// tile, 8 rows to a wave, so a dense tile's items are folded by twice the
// waves; the waves of a scan job's tile test 64 boxes each and share the list
// of those that meet the tile (every strip testing every box took half of the
// kernel's instructions on 1,000 items); and the pixel function is the job's,
// so one launch takes the groups of all functions (32 jobs of 256 to 1,024
// pixels square: 47 us, a launch per function one after the other 165).
// Bound by the chain from the job record over the boxes, the descriptors and
// the masks to the stores, so as many tiles as possible are resident: with 8
// waves 1,000 stars on 2048 x 2048 take 17.4 us, with 16 waves (4 rows each,
// half the tiles at a time) 23.5, with 4 waves 16.5 but 52 on the 32 jobs.
constexpr int kTileBlockWaves = 8;
template <typename F>
__device__ __attribute__((always_inline)) inline void with_fun(int32_t fun, F&& f) {
  switch (fun) {
    case 0: f(std::integral_constant<int, 0>{}); break;
    case 1: f(std::integral_constant<int, 1>{}); break;
    case 2: f(std::integral_constant<int, 2>{}); break;
    case 3: f(std::integral_constant<int, 3>{}); break;
    case 4: f(std::integral_constant<int, 4>{}); break;
    case 5: f(std::integral_constant<int, 5>{}); break;
    default: f(std::integral_constant<int, 6>{}); break;
  }
}
// BARE: whether items have no masks: 0 none, 1 some may, 2 all (calls too small
// for masks, the allocation-free entry point).  A variant each, as that path's
// registers and LDS cost the others 5 % on bytes (170 us against 163 for 10,000
// polygons on 3989 x 4013 x 3).  1 folds both kinds through one copy of the
// code, in at most 80 registers for 1-byte pixels, so that three workgroups
// fit a CU (1,800 stars on 3417 x 2960 uint8: 37.6 us a call; with a second
// copy of the folds 44.2); 2 needs no mask loads (95 stars on 827 x 1253
// float64: 19.4 us, through 1 20.2).
constexpr int kBlockMinWaves = 2;  // (what two waves of a workgroup per SIMD take anyway)
template <typename T, int BARE>
__global__ __launch_bounds__(64 * kTileBlockWaves)
    __attribute__((amdgpu_waves_per_eu(BARE == 1 && sizeof(T) == 1 ? 6 : kBlockMinWaves))) void k_tile_block(TileArgs a) {
  constexpr int TW = tile_w(sizeof(T));
  constexpr int NWORD = TW / 64;
  constexpr int ROWS = TILE_H / kTileBlockWaves;
  __shared__ PolyEdge s_edge[BARE ? kTileBlockWaves : 1][64];
  __shared__ __align__(16) uint32_t s_x[kTileBlockWaves][NWORD > 1 ? 256 : 1];
  __shared__ uint32_t s_list[64 * kTileBlockWaves], s_n[kTileBlockWaves];
  const int wave = wave_index(), lane = threadIdx.x & 63;
  uint32_t burns = 0;
  // neighbouring tiles on one XCD (workgroup b runs on XCD b % 8)
  const uint32_t n_tiles = a.t_hi - a.t_lo, xcd = blockIdx.x % NUM_XCD;
  const uint32_t tl = xcd_unit_lo(xcd, n_tiles) + blockIdx.x / NUM_XCD;
  if (tl >= xcd_unit_lo(xcd + 1u, n_tiles)) return;  // (the whole workgroup)
  int job = 0;
  const StripUnit u = strip_unit(a, a.t_lo + tl, wave * ROWS, ROWS, TW, job);
  const RZ_CONST JobDev& J = *u.J;
  Pixels<T, ROWS> p;
  p.fill(u);
  auto fold = [&](const ItemDesc* d, bool cand) __attribute__((always_inline)) {
    RawItem q{};
    if (cand) q = load_raw(d);
    uint64_t left = __ballot(cand);
    while (left) {
      const Visits v = visits_of<NWORD, ROWS, sizeof(T) == 8>(q, u, (left >> lane) & 1ull, left, s_x[wave]);
      if (!v.n) break;
      uint32_t bits[BARE == 2 ? 1 : kAhead<T>];
      if (BARE < 2) load_bits(a, v, 0u, bits, lane);
      // items without masks are folded one visit after the other, through the
      // same code (a second copy of it cost registers)
      const bool bare = BARE == 2 || (BARE && any_bare(v, lane));
      uint64_t words = 0ull;  // the row words of the item in lane `at`
      int at = -1, wlo = 0;
      uint32_t k = 0, end = v.n;
      do {
        if (bare) {
          int l = lane;
          asm volatile("" : "+v"(l));  // (what is computed of it is not kept in registers from before the loop)
          const uint32_t info = (uint32_t)__builtin_amdgcn_readlane((int)v.info, (int)k);
          if (BARE == 2 || info >> 31) {
            const int item = __builtin_amdgcn_readlane((int)v.item, (int)k);
            if (NWORD == 1 || item != at) {
              const uint64_t da = (uint64_t)d;
              const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)da, item);
              const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(da >> 32), item);
              words = edge_words<NWORD, ROWS>(a, load_desc((const RZ_CONST ItemDesc*)((uint64_t)lo | ((uint64_t)hi << 32))), u,
                                              s_edge[BARE ? wave : 0], l, wlo);
              at = item;
            }
            bits[0] = word_bits<ROWS>(words, (int)(info & 3u) - wlo, l) << (u.Rw & 15);
          } else {
            uint32_t one[1];
            load_bits(a, v, k, one, l);
            bits[0] = one[0];
          }
          end = k + 1u;
        }
        switch (J.fun) {
          case 0: fold_visits<T, 0, ROWS>(a, u, p, v, k, end, bits, lane, burns); break;
          case 1: fold_visits<T, 1, ROWS>(a, u, p, v, k, end, bits, lane, burns); break;
          case 2: fold_visits<T, 2, ROWS>(a, u, p, v, k, end, bits, lane, burns); break;
          case 3: fold_visits<T, 3, ROWS>(a, u, p, v, k, end, bits, lane, burns); break;
          case 4: fold_visits<T, 4, ROWS>(a, u, p, v, k, end, bits, lane, burns); break;
          case 5: fold_visits<T, 5, ROWS>(a, u, p, v, k, end, bits, lane, burns); break;
          default: fold_visits<T, 6, ROWS>(a, u, p, v, k, end, bits, lane, burns); break;
        }
        k = end;
      } while (k < v.n);
    }
  };
  if (!J.scan) {
    const uint32_t pb = as_const(a.tile_off)[a.t_lo + tl], pe = as_const(a.tile_off)[a.t_lo + tl + 1u];
    for (uint32_t i = pb; i < pe; i += 64u) fold(a.pair_desc + i + lane, (uint32_t)lane < pe - i);
  } else {
    const bool compact = J.scan_compact && a.scan_box;
    const int64_t ib = J.i_base;
    const int32_t T0 = u.Rw - wave * ROWS, T1 = min(T0 + TILE_H, u.nrows);  // the tile's rows
    for (int64_t base = 0; base < J.ni; base += 64 * kTileBlockWaves) {
      const int64_t i = base + wave * 64 + lane;
      bool meets = i < J.ni;
      if (meets) {
        if (compact) {
          const uint2 bx = a.scan_box[ib + i];
          const uint32_t tx = (uint32_t)u.C0 / (uint32_t)TW, s0 = (uint32_t)T0 / WAVE_ROWS;
          meets = (bx.x & 0xFFFFu) <= s0 + TILE_H / WAVE_ROWS - 1 && s0 <= (bx.x >> 16) && (bx.y & 0xFFFFu) <= tx &&
                  tx <= (bx.y >> 16);
        } else {
          const u32x4 q = *reinterpret_cast<const u32x4*>(a.desc + ib + i);
          meets = (int32_t)q[0] < T1 && (int32_t)q[1] > T0 && (int32_t)q[2] < u.tile_c1 && (int32_t)q[3] > u.C0;
        }
      }
      const uint64_t m = __ballot(meets);
      if (lane == 0) s_n[wave] = (uint32_t)__popcll(m);
      __syncthreads();
      uint32_t n = 0, at = 0;
      for (int w = 0; w < kTileBlockWaves; ++w) {
        if (w == wave) at = n;
        n += s_n[w];
      }
      if (meets) s_list[at + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = (uint32_t)(i - base);
      __syncthreads();
      for (uint32_t k = 0; k < n; k += 64u) {
        const bool cand = k + (uint32_t)lane < n;
        fold(a.desc + ib + base + (cand ? (int64_t)s_list[k + lane] : 0), cand);
      }
      __syncthreads();  // the next boxes overwrite the list
    }
  }
  store_rows<T, ROWS>(u, p, s_x[wave], lane);
  if (a.burns) {
    unsigned long long n = burns;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
    if (lane == 0 && n) atomicAdd(&a.burns[(blockIdx.x * kTileBlockWaves + wave) % kBurnSlots], n);
  }
}

// One line item of a group walked together in k_tile_lp: its records, the
// vertex range its end cell is tested against, kind | banded << 2.
struct GroupItem {
  const uint4* recs;
  int64_t vbeg;
  uint64_t last;
  uint32_t kb;
  uint32_t pad;
};

// Tile kernel of groups with lines or points (polygon items may be mixed
// in), one launch per pixel-function group.  Same work queue, strips, item
// order, background fill and write-once store as k_tile, but the strip's
// accumulator lives in wave-private LDS (16 x TW pixels), so a line or
// point write lands where it belongs instead of going through a per-item
// pass over the whole strip:
//  * first / last / min / max / any give the same result for one or several
//    writes of one value, so a line's cells set LDS mark bits (atomic OR,
//    not waited for) and after the line each lane folds its marked pixels
//    once.  A run of consecutive line items (up to 8 in a 64-wide strip,
//    with the one-vertex points between them) is walked together, its
//    records spread over the lanes and each line marking its own array; one
//    apply then folds each pixel's marks line by line, in item order (a line
//    meets a strip in a few short segments, so one item alone leaves most
//    lanes idle), and the points follow (a point whose cell a line of the
//    group also writes folds between the lines before and after it);
//  * sum and count depend on the number of writes: a line's cells are
//    counted in 16-bit LDS counters, and after the line each lane folds its
//    pixels k times.  Two lines of at most 255 segments each in the strip
//    (with the one-vertex points between them) are walked together, each
//    counting in its own 8-bit counters (a segment writes a pixel once),
//    and fold line 0, the points, then line 1.  With xres != yres
//    (LineWriter + PixelCache, burn_geometry.rs:179-185, 202-208) or
//    all-touched a pixel is written once per line: a mark bit, folded once;
//  * the unordered float sum adds every write with an LDS atomic;
//  * runs of one-vertex point items are folded in geometry order by one
//    lane each, from descriptors loaded 64 at a time (the point's cell is its
//    box, so its vertex is not read);
//  * polygon items fold their coverage masks into the LDS pixels; an
//    all-touched polygon folds its outline cells and its fill once each.
// Segments come as 16-byte records with floored end points (k_prep); a line
// item of many segments over several strips reads only its band of the strip.
// (Folding idempotent writes directly, lane by lane, measured 13 % slower
// than the marks: the read-modify-write per cell serialises the walk.)
template <typename T, int FUN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_tile_lp(TileArgs a) {
  constexpr int TW = tile_w(sizeof(T));
  constexpr int NWORD = TW / 64;
  constexpr int PPC = 16 / (int)sizeof(T);
  constexpr int LPR = TW / PPC;
  constexpr int RSTEP = 64 / LPR;
  constexpr int RPL = WAVE_ROWS / RSTEP;
  constexpr int NPIXS = WAVE_ROWS * TW;           // pixels of a strip
  constexpr bool COUNTED = FUN == 0 || FUN == 5;  // sum, count: the number of writes matters
  constexpr int PPL = NPIXS / 64;                      // pixels per lane in an apply (16 or 64)
  constexpr int MW = NPIXS / 32;                       // words of one mark array
  // line items walked together with marked writes (fewer in sum and count,
  // which group only their dedup lines this way: there the registers of
  // larger groups spill; 2, 4, 8 and 16 measured)
  constexpr int KGRP = TW == 64 ? (COUNTED ? 4 : 8) : 2;
  constexpr int CNT_WORDS = COUNTED ? NPIXS / 2 : 1;   // u16 counters of one item, 2 per word
  // counted line items walked together: CB-bit counters (NPIXS * CB / 32
  // words per item) in the counter words, for items of at most 2^CB - 1
  // records in the strip (a record writes a pixel at most once).  More
  // items measured slower, whether with more LDS, with the edge stage as
  // counters or with 4-bit counters (4 items): the kernel spills more.
  constexpr int CB = 8;
  constexpr int CW = NPIXS * CB / 32;                  // words of one item's counters
  constexpr int KCNT = COUNTED ? (CNT_WORDS / CW < KGRP ? CNT_WORDS / CW : KGRP) : 1;
  __shared__ PolyEdge s_edge[4][64];
  __shared__ __align__(16) T s_acc[4][NPIXS];
  __shared__ __align__(16) uint32_t s_cnt[4][CNT_WORDS];
  __shared__ uint32_t s_mark[4][KGRP * MW];
  __shared__ GroupItem s_grp[4][KGRP];
  // unordered float sum: the strip holds plain sums and s_wr which pixels have any
  constexpr bool FSUM = FUN == 0 && (sizeof(T) == 4 || sizeof(T) == 8) && (T)0.5 != (T)0;
  __shared__ uint32_t s_wr[4][FSUM ? NPIXS / 32 : 1];

  const int wave = wave_index(), lane = threadIdx.x & 63;
  const int srow = lane / LPR, ch = lane % LPR;
  const int ccol = ch * PPC;
  PolyEdge* stage = s_edge[wave];
  T* acc = s_acc[wave];
  uint32_t* cnt = s_cnt[wave];
  uint32_t* mark = s_mark[wave];
  uint32_t* wr = s_wr[wave];
  // (every apply leaves its counters and marks at zero)
  if (COUNTED)
    for (int w = lane; w < CNT_WORDS; w += 64) cnt[w] = 0u;
  for (int w = lane; w < KGRP * MW; w += 64) mark[w] = 0u;
  unsigned long long burns = 0;

  TileQueue tq(a, wave, lane);
  const RZ_CONST uint32_t* toff_c = as_const(a.tile_off);
  const RZ_CONST ItemDesc* pdesc_c = as_const(a.pair_desc);
  const RZ_CONST ItemDesc* desc_c = as_const(a.desc);
  uint32_t pb = 0, pe = 0;
  auto fetch_range = [&](uint32_t tl) {
    if (a.tile_off) {
      pb = toff_c[a.t_lo + tl];
      pe = toff_c[a.t_lo + tl + 1u];
    }
  };
  bool have = tq.begin();
  if (have) fetch_range(tq.t_cur);
  const int32_t strip = wave;
  int job = 0;

  while (have) {
    const uint32_t t = a.t_lo + tq.pop();
    const StripUnit u = strip_unit(a, t, strip * WAVE_ROWS, WAVE_ROWS, TW, job);
    const RZ_CONST JobDev& J = *u.J;
    const T bg = from_bits<T>(J.bg_bits);
    const bool dedup_job = J.dedup_lines != 0;
    const bool at_job = J.all_touched != 0;

    // unordered float sum (no dedup: a line's pixel counts once there):
    // lines and points add as they land (RZ_SUM_UNORDERED)
    const bool unord = FSUM && J.sum_unordered && !dedup_job && !at_job;
    // the strip starts as the background (unordered: as empty sums)
#pragma unroll
    for (int k = 0; k < RPL; ++k) {
      T* p = acc + (srow + k * RSTEP) * TW + ccol;
#pragma unroll
      for (int j = 0; j < PPC; ++j) p[j] = unord ? (T)0 : bg;
    }
    if (FSUM && unord)
      for (int w = lane; w < NPIXS / 32; w += 64) wr[w] = 0u;
    wave_sync();
    // an unordered write of v at strip pixel idx (any lane, any order)
    auto add1 = [&](uint32_t idx, T v) {
      if constexpr (FSUM) {
        atomicAdd(&acc[idx], v);
        atomicOr(&wr[idx >> 5], 1u << (idx & 31u));
      }
    };

    // one write of value v at strip pixel idx, by this lane alone
    auto fold1 = [&](uint32_t idx, T v) { fold<T, FUN>(acc[idx], v, bg, 1u); };

    // each lane folds its marked pixels once and clears their marks
    auto apply_marks = [&](T v) {
      wave_sync();
#pragma unroll
      for (int c0 = 0; c0 < PPL; c0 += 16) {
        const int base = lane * PPL + c0;
        const uint32_t bits = (mark[base >> 5] >> (base & 31)) & 0xFFFFu;
        if (bits) {
          burns += (unsigned long long)__popc(bits);
          T px[16];
          __builtin_memcpy(px, acc + base, sizeof(px));
#pragma unroll
          for (int j = 0; j < 16; ++j) px[j] = fold_select<T, FUN>(px[j], v, bg, (bits >> j) & 1u);
          __builtin_memcpy(acc + base, px, sizeof(px));
        }
      }
      wave_sync();
      for (int w = lane; w < NPIXS / 32; w += 64) mark[w] = 0u;
      wave_sync();
    };

    // all-touched: the cells of the kept segment from local vertex lv that
    // fall in this strip, as marks in mk (the walker stops past the strip)
    auto walk_at = [&](int64_t lv, uint32_t* mk) {
      double x0, y0, x1, y1;
      if (!kept_segment(J, lv, x0, y0, x1, y1)) return;
      // (cells lie within a pixel of the floors of the end points)
      if (floor(fmax(x0, x1)) + 1.0 < (double)u.C0 || floor(fmin(x0, x1)) - 1.0 >= (double)u.tile_c1 ||
          floor(fmax(y0, y1)) + 1.0 < (double)u.Rw || floor(fmin(y0, y1)) - 1.0 >= (double)u.strip_r1)
        return;
      const bool ok = walk_all_touched(x0, y0, x1, y1, J.ncols, J.nrows, u.C0, u.tile_c1, u.Rw, u.strip_r1,
                                       [&](int64_t x, int64_t y) {
                                         const uint32_t idx = (uint32_t)(y - u.Rw) * TW + (uint32_t)(x - u.C0);
                                         atomicOr(&mk[idx >> 5], 1u << (idx & 31u));
                                       });
      if (!ok) atomicOr(a.status, 64u);
    };

    // An all-touched polygon (burn_geometry.rs:219-238): its outline cells
    // and its fill, each pixel folded once.  Idempotent functions fold the
    // union; sum and count (LineWriter + FillWriter over the outline's
    // PixelCache) fold the outline cells once and the fill pixels the cache
    // does not contain: inside the cache window that is every fill pixel off
    // the outline, again the union; a fill pixel outside the window is
    // skipped when the cache bit its wrapped index lands on is set.
    auto polygon_at = [&](const ItemDesc& d) {
      const T v = from_bits<T>(d.value);
      for (int64_t e = lane; e < d.nv; e += 64) walk_at(d.vbeg + e - J.v_base, mark);
      wave_sync();
      // the fill's row words: word w of row `lane` in lanes 0 .. 15
      for (int w = 0; w < NWORD; ++w) {
        const uint32_t bits = column_bits(a, d, u, w, stage, lane);
        uint64_t m = 0ull;
        for (int r = 0; r < WAVE_ROWS; ++r) {
          const uint64_t row = __ballot((bits >> r) & 1u);
          if (lane == r) m = row;
        }
        if (lane < WAVE_ROWS) {
          if (COUNTED && (d.flags & kItemAtCache) && m && a.at_bits && a.at_base[d.last + 1] <= a.at_cap) {
            CacheWin cw;
            item_cache(a.item_win, (int64_t)d.last, cw);
            const uint64_t length = cw.cap / cw.width;
            const unsigned long long* cb = a.at_bits + a.at_base[d.last];
            const int64_t y = (int64_t)u.Rw + lane, xb = (int64_t)u.C0 + w * 64;
            for (uint64_t mm = m; mm; mm &= mm - 1) {
              const int b = __builtin_ctzll(mm);
              const int64_t x = xb + b;
              if ((uint64_t)x - (uint64_t)cw.x0 < cw.width && (uint64_t)y - (uint64_t)cw.y0 < length) continue;
              const uint64_t ci = cache_index(cw, x, y);
              if (ci < cw.cap && ((cb[ci >> 6] >> (ci & 63)) & 1ull)) m &= ~(1ull << b);
            }
          }
          const int idx = lane * TW + w * 64;
          mark[idx >> 5] |= (uint32_t)m;
          mark[(idx >> 5) + 1] |= (uint32_t)(m >> 32);
        }
      }
      apply_marks(v);
    };

    auto polygon = [&](const ItemDesc& d) {
      const T v = from_bits<T>(d.value);
      for (int w = 0; w < NWORD; ++w) {
        const uint32_t bits = column_bits(a, d, u, w, stage, lane);
        burns += (unsigned long long)__popc(bits);
        // (lane: a column; each row's pixels are one LDS access)
        for (int r = 0; r < WAVE_ROWS; ++r) {
          if (!__any((bits >> r) & 1u)) continue;
          if ((bits >> r) & 1u) {
            const int idx = r * TW + w * 64 + lane;
            if (FSUM && unord) {
              acc[idx] = acc[idx] + v;
              atomicOr(&wr[idx >> 5], 1u << (idx & 31));
            } else {
              acc[idx] = fold_select<T, FUN>(acc[idx], v, bg, true);
            }
          }
        }
      }
      wave_sync();
    };

    // a line or a multi-point item: its segment / cell records, lanes over
    // records (chunks of 65,535 records keep a pixel's count in 16 bits)
    // a line or a multi-point item: its records [recs, recs + n_r) (a line's
    // band of this strip, or the item's vertices), lanes over records; `pre`
    // is this lane's record of the first 64, already loaded (chunks of
    // 65,535 records keep a pixel's count in 16 bits)
    auto lines = [&](const ItemDesc& d, const uint4* recs, uint32_t n_r, bool banded, uint4 pre) {
      const int32_t kind = (int32_t)(d.kind_layer & 3u);
      const T v = from_bits<T>(d.value);
      const bool dedup = kind == 1 && (dedup_job || at_job);
      // a write is a mark (one fold per pixel: idempotent functions, or a
      // line's first write per pixel with xres != yres or all-touched) or a
      // count; both are LDS atomics whose result is not waited for
      const bool marked = !COUNTED || dedup;
      // a write at strip pixel idx (emit_idx: the clipped walk's cells,
      // inside by construction) or at a cell
      auto emit_idx = [&](uint32_t idx) {
        if (FSUM && unord) {
          ++burns;
          add1(idx, v);
        } else if (marked) {
          atomicOr(&mark[idx >> 5], 1u << (idx & 31u));
        } else {
          atomicAdd(&cnt[idx >> 1], 1u << ((idx & 1u) * 16u));
        }
      };
      auto emit = [&](auto cx, auto cy) {
        if (cx < u.C0 || cx >= u.tile_c1 || cy < u.Rw || cy >= u.strip_r1) return;
        emit_idx((uint32_t)(cy - u.Rw) * TW + (uint32_t)(cx - u.C0));
      };
      // end cell of the last kept edge of an open line (burners.rs:86-89)
      auto end_cell = [&](const uint4& r, uint32_t e) {
        return banded ? (r.w & kLsFlag) != 0
                      : ((uint64_t)(d.vbeg + (int64_t)e + 1) == d.last && !(r.w & kLsFlag));
      };
      for (uint32_t cs = 0; cs < n_r; cs += 65535u) {
        const uint32_t ce = min(n_r, cs + 65535u);
        bool far = false;
        for (uint32_t e = cs + (uint32_t)lane; e < ce; e += 64u) {
          const uint4 r = e < 64u ? pre : recs[e];
          if (r.x == kLsNone) continue;
          if (kind == 2) {  // a vertex of a multi-point: its cell
            emit((int32_t)r.x, (int32_t)r.y);
            continue;
          }
          if (at_job) {  // the all-touched walker, from the world coordinates
            walk_at(d.vbeg + (int64_t)e - J.v_base, mark);
            continue;
          }
          if (r.x == kLsFar) {
            far = true;
            continue;
          }
          const int32_t ix0 = (int32_t)((int64_t)r.x - kLsBias), iy0 = (int32_t)((int64_t)r.y - kLsBias);
          const int32_t ix1 = (int32_t)((int64_t)r.z - kLsBias);
          const int32_t iy1 = (int32_t)((int64_t)(r.w & ~kLsFlag) - kLsBias);
          walk_window32_idx(ix0, iy0, ix1, iy1, u.C0, u.tile_c1, u.Rw, u.strip_r1, TW, emit_idx);
          if (end_cell(r, e)) emit(ix1, iy1);
        }
        if (__any(far)) {
          // segments beyond +-2^30 pixels (never banded): the end points again
          // from the world coordinates (edges.rs:119-122), walked in 128 bits
          for (uint32_t e = cs + (uint32_t)lane; e < ce; e += 64u) {
            const uint4 r = recs[e];
            if (r.x != kLsFar) continue;
            const int64_t lv = d.vbeg + (int64_t)e - J.v_base;
            auto px_x = [&](double X) { return isnan(X) ? X : (X - J.xmin) / J.xres; };
            auto px_y = [&](double Y) { return isnan(Y) ? Y : (J.ymax - Y) / J.yres; };
            const int64_t ix0 = sat_isize(floor(px_x(J.xy[2 * lv]))), iy0 = sat_isize(floor(px_y(J.xy[2 * lv + 1])));
            const int64_t ix1 = sat_isize(floor(px_x(J.xy[2 * lv + 2]))), iy1 = sat_isize(floor(px_y(J.xy[2 * lv + 3])));
            const int64_t lim = (int64_t)1 << 60;
            if (ix0 > -lim && ix0 < lim && ix1 > -lim && ix1 < lim && iy0 > -lim && iy0 < lim &&
                iy1 > -lim && iy1 < lim)
              walk_window<__int128>(ix0, iy0, ix1, iy1, u.C0, u.tile_c1, u.Rw, u.strip_r1, emit);
            else
              atomicOr(a.status, 1u);  // pixel coordinates beyond +-2^60: unsupported
            if (end_cell(r, e)) emit(ix1, iy1);
          }
        }
        if (COUNTED && !marked && !unord) {
          // each lane folds its PPL pixels k times each and clears their counters
          wave_sync();
#pragma unroll
          for (int c0 = 0; c0 < PPL; c0 += 16) {
            const int base = lane * PPL + c0;
            uint32_t w[8];
            __builtin_memcpy(w, cnt + base / 2, 32);
            if (w[0] | w[1] | w[2] | w[3] | w[4] | w[5] | w[6] | w[7]) {
              T px[16];
              __builtin_memcpy(px, acc + base, sizeof(px));
#pragma unroll
              for (int j = 0; j < 16; ++j) {
                const uint32_t k = (w[j >> 1] >> ((j & 1) * 16)) & 0xFFFFu;
                burns += k;
                fold<T, FUN>(px[j], v, bg, k);
              }
              __builtin_memcpy(acc + base, px, sizeof(px));
              const uint32_t z[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
              __builtin_memcpy(cnt + base / 2, z, 32);
            }
          }
          wave_sync();
        }
      }
      if (marked && !unord) apply_marks(v);
    };

    // the records of a line or multi-point item in this strip: base, count,
    // whether they are the line's band (each lane may ask for its own item)
    auto records = [&](const ItemDesc& d, const uint4*& recs, uint32_t& n_r) -> bool {
      if ((d.kind_layer & 3u) == 1u && d.band) {
        const uint32_t bi = d.band - 1u + (uint32_t)(u.Rw / kBandRows - d.r0 / kBandRows);
        const uint64_t b0 = a.band_off[bi];
        recs = a.band_segs + b0;
        n_r = (uint32_t)(a.band_off[bi + 1u] - b0);
        return true;
      }
      recs = a.lseg + d.vbeg;
      n_r = (uint32_t)d.nv;
      return false;
    };
    auto first_chunk = [&](const uint4* recs, uint32_t n_r) {
      return (uint32_t)lane < n_r ? recs[lane] : make_uint4(kLsNone, 0u, 0u, 0u);
    };

    // The items of lanes G, consecutive in item order: the line items L (two
    // or more, at most 65,535 records each) and the one-vertex points
    // between them (cell pidx, value bits pv in their lanes).  Each lane's
    // own item is dl with records [rp, rp + rn).  The lanes take the lines'
    // records in turn, line k writing mark array k (cmode false) or CB-bit
    // counter array k (cmode: sum and count without dedup, at most
    // 2^CB - 1 records per line, and a record writes a pixel at most once);
    // then each lane folds its pixels' writes line by line, and the points
    // are folded in order after them, except that a point whose cell a line
    // of the group also writes is folded between the lines before it and
    // those after it.  A counted group (two lines) always folds line 0, the
    // points between them, then line 1.
    auto line_group = [&](uint64_t G, uint64_t L, const ItemDesc& dl, const uint4* rp, uint32_t rn, bool bnd,
                          bool cmode, uint32_t pidx, uint64_t pv) {
      GroupItem* gi = s_grp[wave];
      const int ng = __popcll(L);
      const uint64_t P = G & ~L;
      // the points of lanes pm, one at a time in item order
      auto fold_points = [&](uint64_t pm) {
        for (uint64_t m = pm; m; m &= m - 1ull) {
          const int b = __builtin_ctzll(m);
          const uint32_t idx = (uint32_t)__builtin_amdgcn_readlane((int)pidx, b);
          const uint64_t vb = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(pv >> 32), b) << 32) |
                              (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)pv, b);
          if (lane == 0) {
            ++burns;
            fold1(idx, from_bits<T>(vb));
          }
        }
      };
      if ((L >> lane) & 1ull) {
        GroupItem it;
        it.recs = rp;
        it.vbeg = dl.vbeg;
        it.last = dl.last;
        it.kb = (dl.kind_layer & 3u) | (bnd ? 4u : 0u);
        it.pad = 0u;
        gi[__popcll(L & ((1ull << lane) - 1ull))] = it;
      }
      // record offsets and values of the lines (uniform)
      uint32_t pre[KGRP];
      T vk[KGRP];
      uint32_t tot = 0;
      uint64_t g = L;
#pragma unroll
      for (int k = 0; k < KGRP; ++k) {
        pre[k] = tot;
        vk[k] = bg;
        if (g) {
          const int pk = __builtin_ctzll(g);
          g &= g - 1ull;
          tot += (uint32_t)__builtin_amdgcn_readlane((int)rn, pk);
          const uint64_t vb = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(dl.value >> 32), pk) << 32) |
                              (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)dl.value, pk);
          vk[k] = from_bits<T>(vb);
        }
      }
      // counter array of item k
      auto carr = [&](int k) { return cnt + k * CW; };
      wave_sync();
      // record e of the group: its item k and index ei in that item
      auto locate = [&](uint32_t e, int& k, uint32_t& ei) {
        uint32_t b = 0;
        k = 0;
#pragma unroll
        for (int j = 1; j < KGRP; ++j)
          if (e >= pre[j]) {
            k = j;
            b = pre[j];
          }
        ei = e - b;
      };
      bool far = false;
      for (uint32_t e = (uint32_t)lane; e < tot; e += 64u) {
        int k;
        uint32_t ei;
        locate(e, k, ei);
        const GroupItem it = gi[k];
        uint32_t* mk = mark + k * MW;
        uint32_t* ck = carr(k);
        auto emit_idx = [&](uint32_t idx) {
          if (COUNTED && cmode) atomicAdd(&ck[idx / (32 / CB)], 1u << ((idx % (32 / CB)) * CB));
          else atomicOr(&mk[idx >> 5], 1u << (idx & 31u));
        };
        auto emit = [&](auto cx, auto cy) {
          if (cx < u.C0 || cx >= u.tile_c1 || cy < u.Rw || cy >= u.strip_r1) return;
          emit_idx((uint32_t)(cy - u.Rw) * TW + (uint32_t)(cx - u.C0));
        };
        const uint4 r = it.recs[ei];
        if (r.x == kLsNone) continue;
        if ((it.kb & 3u) == 2u) {  // a vertex of a multi-point: its cell
          emit((int32_t)r.x, (int32_t)r.y);
          continue;
        }
        if (at_job) {
          walk_at(it.vbeg + (int64_t)ei - J.v_base, mk);
          continue;
        }
        if (r.x == kLsFar) {
          far = true;
          continue;
        }
        const int32_t ix0 = (int32_t)((int64_t)r.x - kLsBias), iy0 = (int32_t)((int64_t)r.y - kLsBias);
        const int32_t ix1 = (int32_t)((int64_t)r.z - kLsBias);
        const int32_t iy1 = (int32_t)((int64_t)(r.w & ~kLsFlag) - kLsBias);
        walk_window32_idx(ix0, iy0, ix1, iy1, u.C0, u.tile_c1, u.Rw, u.strip_r1, TW, emit_idx);
        const bool endc = (it.kb & 4u) ? (r.w & kLsFlag) != 0
                                       : ((uint64_t)(it.vbeg + (int64_t)ei + 1) == it.last && !(r.w & kLsFlag));
        if (endc) emit(ix1, iy1);
      }
      if (__any(far)) {
        for (uint32_t e = (uint32_t)lane; e < tot; e += 64u) {
          int k;
          uint32_t ei;
          locate(e, k, ei);
          const GroupItem it = gi[k];
          const uint4 r = it.recs[ei];
          if (r.x != kLsFar) continue;
          uint32_t* mk = mark + k * MW;
          uint32_t* ck = carr(k);
          auto emit = [&](auto cx, auto cy) {
            if (cx < u.C0 || cx >= u.tile_c1 || cy < u.Rw || cy >= u.strip_r1) return;
            const uint32_t idx = (uint32_t)(cy - u.Rw) * TW + (uint32_t)(cx - u.C0);
            if (COUNTED && cmode) atomicAdd(&ck[idx / (32 / CB)], 1u << ((idx % (32 / CB)) * CB));
            else atomicOr(&mk[idx >> 5], 1u << (idx & 31u));
          };
          const int64_t lv = it.vbeg + (int64_t)ei - J.v_base;
          auto px_x = [&](double X) { return isnan(X) ? X : (X - J.xmin) / J.xres; };
          auto px_y = [&](double Y) { return isnan(Y) ? Y : (J.ymax - Y) / J.yres; };
          const int64_t ix0 = sat_isize(floor(px_x(J.xy[2 * lv]))), iy0 = sat_isize(floor(px_y(J.xy[2 * lv + 1])));
          const int64_t ix1 = sat_isize(floor(px_x(J.xy[2 * lv + 2]))), iy1 = sat_isize(floor(px_y(J.xy[2 * lv + 3])));
          const int64_t lim = (int64_t)1 << 60;
          if (ix0 > -lim && ix0 < lim && ix1 > -lim && ix1 < lim && iy0 > -lim && iy0 < lim && iy1 > -lim &&
              iy1 < lim)
            walk_window<__int128>(ix0, iy0, ix1, iy1, u.C0, u.tile_c1, u.Rw, u.strip_r1, emit);
          else
            atomicOr(a.status, 1u);  // pixel coordinates beyond +-2^60: unsupported
          const bool endc = (it.kb & 4u) ? (r.w & kLsFlag) != 0
                                         : ((uint64_t)(it.vbeg + (int64_t)ei + 1) == it.last && !(r.w & kLsFlag));
          if (endc) emit(ix1, iy1);
        }
      }
      wave_sync();
      // the writes of line k (uniform) at this lane's pixels, folded
      auto apply_one = [&](int k) {
        T v = bg;
#pragma unroll
        for (int j = 0; j < KGRP; ++j)
          if (j == k) v = vk[j];
#pragma unroll
        for (int c0 = 0; c0 < PPL; c0 += 16) {
          const int base = lane * PPL + c0;
          if (COUNTED && cmode) {
            constexpr int NW = 16 * CB / 32;
            uint32_t w[NW];
            __builtin_memcpy(w, carr(k) + base / (32 / CB), sizeof(w));
            uint32_t any = 0u;
#pragma unroll
            for (int x = 0; x < NW; ++x) any |= w[x];
            if (any) {
              T px[16];
              __builtin_memcpy(px, acc + base, sizeof(px));
#pragma unroll
              for (int j = 0; j < 16; ++j) {
                const uint32_t c = (w[j / (32 / CB)] >> ((j % (32 / CB)) * CB)) & ((1u << CB) - 1u);
                burns += c;
                fold<T, FUN>(px[j], v, bg, c);
              }
              __builtin_memcpy(acc + base, px, sizeof(px));
            }
          } else {
            const uint32_t b = (mark[k * MW + (base >> 5)] >> (base & 31)) & 0xFFFFu;
            if (b) {
              T px[16];
              __builtin_memcpy(px, acc + base, sizeof(px));
              burns += (unsigned long long)__popc(b);
#pragma unroll
              for (int j = 0; j < 16; ++j) px[j] = fold_select<T, FUN>(px[j], v, bg, (b >> j) & 1u);
              __builtin_memcpy(acc + base, px, sizeof(px));
            }
          }
        }
      };
      if (COUNTED && cmode) {
        // two lines with the points between them: line 0, the points, line 1
        apply_one(0);
        wave_sync();
        fold_points(P);
        wave_sync();
        apply_one(1);
        wave_sync();
        for (int w = lane; w < ng * CW; w += 64) cnt[w] = 0u;
        wave_sync();
        return;
      }
      // the points whose cells a line of the group also writes (C): each is
      // folded after the lines before it and before those after it; the
      // others share no cell with a line and are folded last
      bool hit = false;
      if ((P >> lane) & 1ull) {
#pragma unroll
        for (int k = 0; k < KGRP; ++k) {
          if (k >= ng) break;
          hit |= ((mark[k * MW + (pidx >> 5)] >> (pidx & 31u)) & 1u) != 0u;
        }
      }
      const uint64_t C = __ballot(hit);
      // each lane folds its pixels' marks of lines [lo, hi), line by line (a
      // wave-wide loop over the lines would fold every line in every lane)
      auto apply_range = [&](int lo, int hi) {
#pragma unroll
        for (int c0 = 0; c0 < PPL; c0 += 16) {
          const int base = lane * PPL + c0;
          uint32_t bk[KGRP];
          uint32_t kmask = 0u;  // the lines with marks in this lane's pixels
#pragma unroll
          for (int k = 0; k < KGRP; ++k) {
            bk[k] = (k >= lo && k < hi) ? (mark[k * MW + (base >> 5)] >> (base & 31)) & 0xFFFFu : 0u;
            kmask |= bk[k] ? 1u << k : 0u;
          }
          if (kmask) {
            T px[16];
            __builtin_memcpy(px, acc + base, sizeof(px));
            while (kmask) {
              const int k = __builtin_ctz(kmask);
              kmask &= kmask - 1u;
              uint32_t b = 0u;
              T v = bg;
#pragma unroll
              for (int j = 0; j < KGRP; ++j)
                if (j == k) {
                  b = bk[j];
                  v = vk[j];
                }
              burns += (unsigned long long)__popc(b);
#pragma unroll
              for (int j = 0; j < 16; ++j) px[j] = fold_select<T, FUN>(px[j], v, bg, (b >> j) & 1u);
            }
            __builtin_memcpy(acc + base, px, sizeof(px));
          }
        }
      };
      int lo = 0;
      for (uint64_t m = C; m; m &= m - 1ull) {
        const int b = __builtin_ctzll(m);
        const int r = __popcll(L & ((1ull << b) - 1ull));  // the lines before the point
        if (r > lo) {
          apply_range(lo, r);
          wave_sync();
          lo = r;
        }
        fold_points(1ull << b);
        wave_sync();
      }
      apply_range(lo, ng);
      wave_sync();
      for (int w = lane; w < ng * MW; w += 64) mark[w] = 0u;
      wave_sync();
      fold_points(P & ~C);
    };

    auto process_item = [&](const ItemDesc& d) {
      if (d.r1 <= u.Rw || d.r0 >= u.strip_r1 || d.c1 <= u.C0 || d.c0 >= u.tile_c1) return;
      if ((d.kind_layer & 3u) == 0u) {
        if (at_job) polygon_at(d);
        else polygon(d);
      } else {
        const uint4* recs;
        uint32_t n_r;
        const bool banded = records(d, recs, n_r);
        lines(d, recs, n_r, banded, first_chunk(recs, n_r));
      }
    };

    if (!J.scan) {
      // descriptors 64 at a time, one per lane: which items meet the strip,
      // the cells and values of one-vertex points (their box), and the
      // record range of every line (its band bounds, loaded by all lanes at
      // once).  Items are then taken in order: a run of points is folded by
      // one lane from the lanes' copies, a polygon or line is reloaded
      // uniformly and processed by the wave, and the next line's first
      // records are loaded while the current one is walked.
      for (uint32_t i0 = pb; i0 < pe; i0 += 64u) {
        const uint32_t nb = min(64u, pe - i0);
        bool pt = false, ln = false, po = false, bnd = false, grp = false;
        uint32_t pidx = 0, rn = 0;
        uint64_t pv = 0;
        const uint4* rp = nullptr;
        ItemDesc dl;
        __builtin_memset(&dl, 0, sizeof(dl));
        if ((uint32_t)lane < nb) {
          dl = load_desc(pdesc_c + i0 + (uint32_t)lane);
          const uint32_t kind = dl.kind_layer & 3u;
          const bool vis = !(dl.r1 <= u.Rw || dl.r0 >= u.strip_r1 || dl.c1 <= u.C0 || dl.c0 >= u.tile_c1);
          pt = vis && kind == 2u && dl.nv == 1;
          po = vis && kind == 0u;
          ln = vis && !pt && !po;
          if (pt) {
            pidx = (uint32_t)(dl.r0 - u.Rw) * TW + (uint32_t)(dl.c0 - u.C0);
            pv = dl.value;
          }
          if (ln) bnd = records(dl, rp, rn);
          // lines walked in groups: those whose writes are marks, or counted
          // ones (sum, count without dedup) of at most 2^CB - 1 records here
          grp = ln && rn <= 0xFFFFu &&
                (!COUNTED ? true : (dedup_job || at_job) ? kind == 1u : (!unord && rn < (1u << CB)));
        }
        const uint64_t ptm = __ballot(pt), lnm = __ballot(ln), grm = __ballot(grp);
        uint64_t todo = ptm | lnm | __ballot(po);
        // the first records of line item q (a uniform lane index)
        auto prefetch = [&](int q) {
          const uint4* r = (const uint4*)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)((uint64_t)rp >> 32), q) << 32) |
                                          (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(uint64_t)rp, q));
          return first_chunk(r, (uint32_t)__builtin_amdgcn_readlane((int)rn, q));
        };
        uint64_t lrest = lnm;
        uint4 pre = make_uint4(kLsNone, 0u, 0u, 0u);
        if (lrest) pre = prefetch(__builtin_ctzll(lrest));
        while (todo) {
          const int p = __builtin_ctzll(todo);
          if ((ptm >> p) & 1ull) {
            // the run of points up to the next line or polygon, in order
            const uint64_t other = todo & ~ptm & (~0ull << p);
            const uint64_t run = todo & ptm & (other ? ((1ull << __builtin_ctzll(other)) - 1ull) : ~0ull);
            if (FSUM && unord) {
              if ((run >> lane) & 1ull) {
                ++burns;
                add1(pidx, from_bits<T>(pv));
              }
              todo &= ~run;
              continue;
            }
            uint64_t m = run;
            while (m) {
              const int b = __builtin_ctzll(m);
              m &= m - 1;
              const uint32_t idx = (uint32_t)__builtin_amdgcn_readlane((int)pidx, b);
              const uint64_t vb = ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(pv >> 32), b) << 32) |
                                  (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)pv, b);
              if (lane == 0) {
                ++burns;
                fold1(idx, from_bits<T>(vb));
              }
            }
            todo &= ~run;
            continue;
          }
          if ((grm >> p) & 1ull) {
            // the run of groupable lines and one-vertex points (not in dedup
            // groups of sum and count) up to the next other item, to its
            // KGRP-th line
            const uint64_t mem = (COUNTED && (dedup_job || at_job)) ? grm : (grm | ptm);
            const uint64_t other = todo & ~mem & (~0ull << p);
            const uint64_t run = todo & mem & (other ? ((1ull << __builtin_ctzll(other)) - 1ull) : ~0ull);
            const bool cmode = COUNTED && !dedup_job && !at_job;
            uint64_t lr = run & grm, L = 0;
#pragma unroll
            for (int k = 0; k < KGRP; ++k) {
              if (!cmode || k < KCNT) {
                L |= lr & (0ull - lr);
                lr &= lr - 1ull;
              }
            }
            if (L & (L - 1ull)) {
              const int hi = 63 - __builtin_clzll(L);
              const uint64_t G = run & (hi == 63 ? ~0ull : ((2ull << hi) - 1ull));
              line_group(G, L, dl, rp, rn, bnd, cmode, pidx, pv);
              todo &= ~G;
              lrest &= ~G;
              if (lrest) pre = prefetch(__builtin_ctzll(lrest));
              continue;
            }
          }
          todo &= todo - 1;
          // (reloaded with one uniform load: broadcasting lane p's copy kept
          // every descriptor word live across the loop, measured slower)
          const ItemDesc d = load_desc(pdesc_c + i0 + (uint32_t)p);
          if ((lnm >> p) & 1ull) {
            const uint4 cur = pre;
            lrest &= lrest - 1;
            if (lrest) pre = prefetch(__builtin_ctzll(lrest));
            const uint4* recs = (const uint4*)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)((uint64_t)rp >> 32), p) << 32) |
                                               (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(uint64_t)rp, p));
            const uint32_t n_r = (uint32_t)__builtin_amdgcn_readlane((int)rn, p);
            const bool banded = __builtin_amdgcn_readlane((int)bnd, p) != 0;
            lines(d, recs, n_r, banded, cur);
          } else if (at_job) {
            polygon_at(d);
          } else {
            polygon(d);
          }
        }
      }
    } else if (J.scan_compact && a.scan_box) {
      // scan job of one band: the 8-byte item boxes in strip and tile units,
      // 64 at a time, the next 64 loaded while this batch's hits are
      // processed
      const int64_t ib = J.i_base, ie = J.i_base + J.ni;
      const uint32_t sidx = (uint32_t)u.Rw / WAVE_ROWS, tx = (uint32_t)u.C0 / (uint32_t)TW;
      const uint2* sb = a.scan_box;
      uint2 nbx = ib + lane < ie ? sb[ib + lane] : make_uint2(0xFFFFu, 0u);
      for (int64_t base = ib; base < ie; base += 64) {
        const uint2 bx = nbx;
        const bool valid = base + lane < ie;
        if (base + 64 + lane < ie) nbx = sb[base + 64 + lane];
        uint64_t m = __ballot(valid && scan_box_meets(bx, sidx, tx));
        while (m) {
          const int bit = __builtin_ctzll(m);
          m &= m - 1;
          process_item(load_desc(desc_c + base + bit));
        }
      }
    } else {
      // scan job: test every item's box in order (small item counts), 64
      // boxes at a time, the next 64 loaded while this batch's hits are
      // processed
      const int64_t ib = J.i_base, ie = J.i_base + J.ni;
      BoxLayer nbx = ib + lane < ie ? load_box(desc_c + ib + lane) : BoxLayer{0, 0, 0, 0, 0u};
      for (int64_t base = ib; base < ie; base += 64) {
        const BoxLayer bx = nbx;
        const bool valid = base + lane < ie;
        if (base + 64 + lane < ie) nbx = load_box(desc_c + base + 64 + lane);
        const bool hit = valid && (bx.kind_layer >> 2) == u.layer && bx.r0 < u.strip_r1 && bx.r1 > u.Rw &&
                         bx.c0 < u.tile_c1 && bx.c1 > u.C0 && bx.r0 < bx.r1 && bx.c0 < bx.c1;
        uint64_t m = __ballot(hit);
        while (m) {
          const int bit = __builtin_ctzll(m);
          m &= m - 1;
          process_item(load_desc(desc_c + base + bit));
        }
      }
    }

    have = tq.advance();
    if (have) fetch_range(tq.t_cur);

    // ---- write the strip once from LDS
    wave_sync();
    store_strip<T, PPC, RPL, RSTEP>(u, srow, ccol, [&](int k) {
      const int idx = (srow + k * RSTEP) * TW + ccol;
      T px[PPC];
      __builtin_memcpy(px, acc + idx, 16);
      if (FSUM && unord) {  // pixels with no write keep the background
        const uint32_t w = wr[idx >> 5] >> (idx & 31);
#pragma unroll
        for (int j = 0; j < PPC; ++j) px[j] = ((w >> j) & 1u) ? px[j] : bg;
      }
      u32x4 vec;
      __builtin_memcpy(&vec, px, 16);
      return vec;
    });
    wave_sync();  // the next strip's background overwrites these pixels
  }
  if (a.burns) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) burns += __shfl_xor(burns, off, 64);
    if (lane == 0 && burns) atomicAdd(&a.burns[blockIdx.x % kBurnSlots], burns);
  }
}

}  // namespace rzk
