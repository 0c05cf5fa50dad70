// Per-thread work of the transpose kernels, written once for the device and
// for the host replay used by the CPU tests.
//
// Each kernel is a sequence of "rounds": every thread of a workgroup runs
// load(), the workgroup synchronises, every thread runs store(). The device
// kernels in kernels.hip wrap these with __syncthreads(); the host replay runs
// load() for all threads of a block, then store() for all threads, which is
// exactly the ordering the barrier guarantees.
#pragma once

#include "common.h"

namespace lrt {

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Opaque B-byte words: element moves never interpret the bits.
template <int BYTES> struct Word;
template <> struct Word<4> { using type = uint32_t; };
template <> struct Word<8> { using type = u32x2; };
template <> struct Word<16> { using type = u32x4; };

template <typename E, typename V>
__host__ __device__ inline E vget(const V& v, int k) {
  E e;
  __builtin_memcpy(&e, reinterpret_cast<const char*>(&v) + k * sizeof(E), sizeof(E));
  return e;
}

template <typename E, typename V>
__host__ __device__ inline void vset(V& v, int k, const E& e) {
  __builtin_memcpy(reinterpret_cast<char*>(&v) + k * sizeof(E), &e, sizeof(E));
}

// Global stores and loads of the transpose kernels. Every output byte is
// written once and never read back by the kernel, so stores are streaming
// (non-temporal): on MI355X they lift a plain 256 MiB copy from about 5.5 to
// about 7.1 TB/s. LRT_NT_STORES selects them at build time. Loads are
// streaming only where a kernel says so (STREAM): they help where whole lines
// are read once and the input is too large for the 256 MiB Infinity Cache,
// and cost where neighbouring work items share lines.
#ifndef LRT_NT_STORES
#define LRT_NT_STORES 1
#endif
// Host replay only: an observer that is told which work item and thread the
// replay is running and sees every global load and store it makes. The
// tests of the access counters compare these accesses with the counters'
// own enumeration. Null (the normal case) costs one test per access.
struct ReplayObserver {
  virtual void at(long long item, int thread) = 0;
  virtual void access(const void* p, int bytes, int store) = 0;
};
extern thread_local ReplayObserver* g_replay_observer;

template <typename V>
__host__ __device__ inline void st(V* p, const V& v) {
#if defined(__HIP_DEVICE_COMPILE__)
#if LRT_NT_STORES
  __builtin_nontemporal_store(v, p);
#else
  *p = v;
#endif
#else
  if (g_replay_observer) g_replay_observer->access(p, (int)sizeof(V), 1);
  *p = v;
#endif
}
template <bool STREAM = false, typename V>
__host__ __device__ inline V ld(const V* p) {
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (STREAM)
    return __builtin_nontemporal_load(p);
  else
    return *p;
#else
  if (g_replay_observer) g_replay_observer->access(p, (int)sizeof(V), 0);
  return *p;
#endif
}

// A V read from an address that is a multiple of AL bytes only (gfx950 loads
// 16 bytes from any 4-byte boundary in one instruction).
template <typename V, int AL, bool STREAM = false>
__host__ __device__ inline V ld_unaligned(const void* p) {
#if defined(__HIP_DEVICE_COMPILE__)
  typedef V U __attribute__((aligned(AL)));
  if constexpr (STREAM)
    return __builtin_nontemporal_load(static_cast<const U*>(p));
  else
    return *static_cast<const U*>(p);
#else
  if (g_replay_observer) g_replay_observer->access(p, (int)sizeof(V), 0);
  V v;
  __builtin_memcpy(&v, p, sizeof(V));
  return v;
#endif
}

// At both ends of a branch that loads non-temporally what the other branch loads
// temporally: without it the compiler merges the two into one temporal load
// (8192 x 8192 f32 93 us instead of 85).
__host__ __device__ inline void keep_branch() {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" ::: "memory");
#endif
}

// Elements between the last 128-byte line boundary and p (p a multiple of
// the element size).
template <typename E>
__host__ __device__ inline int line_phase(const E* p) {
  return (int)(((uintptr_t)p & 127) / sizeof(E));
}

struct TileCtx {
  int x0, y0;
  int off_in, off_out;
  bool full;
};

// Tile w of a Tiled plan with tiles of tx_size x ty_size elements.
template <class A>
__host__ __device__ inline TileCtx tile_item(const A& a, uint32_t w, int tx_size, int ty_size) {
  TileCtx c;
  const uint32_t mb = fdiv(w, a.ntiles_div);
  const uint32_t tile = w - mb * (uint32_t)a.ntiles;
  uint32_t tx, ty;
  if (a.group <= 1) {
    ty = fdiv(tile, a.ntx_div);
    tx = tile - ty * (uint32_t)a.ntx;
  } else {
    const uint32_t g = fdiv(tile, a.group_row_div);  // group index
    const uint32_t within = tile - g * a.group_row_div.d;
    const FastDiv& rows = (tile >= (uint32_t)a.last_group_start) ? a.last_div : a.group_div;
    tx = fdiv(within, rows);
    ty = g * (uint32_t)a.group + (within - tx * rows.d);
  }
  c.x0 = (int)tx * tx_size;
  c.y0 = (int)ty * ty_size;
  outer_offsets(a.outer, mb, c.off_in, c.off_out);
  c.full = (c.x0 + tx_size <= a.X) && (c.y0 + ty_size <= a.Y);
  return c;
}

// ---------------------------------------------------------------------------
// Tiled: a TX x TY tile of the (x, y) plane goes through LDS. Reads walk x
// (contiguous in the input) with VX elements per lane; writes walk y
// (contiguous in the output) with VY elements per lane. One LDS row of pitch
// TX + 1 per y keeps the column reads of the write phase spread over banks.
// When x or y is a group of dims, each row (column) finds its offset on the
// other side from the group's digits; a full tile of one-dim groups steps
// through memory by a fixed stride instead.
// Bound by HBM. One workgroup moves one tile and ends: a loop over tiles kept
// 106 SGPRs and up to 20 more VGPRs alive (34 SGPRs without it), and the
// dispatcher's order keeps neighbouring tiles closer in time than a stride
// over the grid does ([2, 8, 16, 32, 64, 128] f32 95 -> 88 us as 64 x 128 tiles,
// with the loads non-temporal too; a copy of the bytes takes 85 us, and the 64 x
// 64 tiles that librettPlan takes there 94 us, as before).
// Reference counterpart: transposeTiled, src/kernel.cpp:48-170.
// ---------------------------------------------------------------------------
// G = false compiles only the one-dim-group path (the kernel then needs no
// registers for group maps); G = true handles groups of several dims too.
template <int B, int TX, int TY, int VX, int VY, bool G = false>
struct TiledOps {
  using E = typename Word<B>::type;
  using VI = typename Word<B * VX>::type;
  using VO = typename Word<B * VY>::type;
  // 128 x 128 tiles take 512 threads: with 256, two workgroups of 66 KiB of LDS
  // leave a CU 8 waves (8192 x 8192 f32 on MI355X: 104 us; with 512, 95 us, and
  // 88 us with one tile per workgroup and non-temporal loads as well).
  static constexpr int NT = TX * TY >= 128 * 128 ? 512 : 256;
  static constexpr int LR = TX / VX;   // lanes per input row
  static constexpr int RP = NT / LR;   // input rows per pass
  static constexpr int NPR = TY / RP;  // read passes
  static constexpr int LW = TY / VY;   // lanes per output row
  static constexpr int WP = NT / LW;   // output rows (x) per pass
  static constexpr int NPW = TX / WP;  // write passes
  static constexpr int PITCH = TX + 1;
  // G: after the tile, TY input offsets of the tile's rows and TX output
  // offsets of its columns (ints), written once per tile by prepare().
  static constexpr int OFF_ELEMS = G ? ((TX + TY) * 4 + B - 1) / B : 0;
  static constexpr int LDS_ELEMS = TY * PITCH + OFF_ELEMS;
  static_assert(TX % VX == 0 && NT % LR == 0 && TY % RP == 0 && NPR >= 1, "read shape");
  static_assert(TY % VY == 0 && NT % LW == 0 && TX % WP == 0 && NPW >= 1, "write shape");
  static_assert(!G || TX + TY <= NT, "one thread per tile row and column");

  __host__ __device__ static int* offsets(E* lds) { return reinterpret_cast<int*>(lds + TY * PITCH); }
  __host__ __device__ static const int* offsets(const E* lds) {
    return reinterpret_cast<const int*>(lds + TY * PITCH);
  }

  // G only, before load(): thread t < TY finds the input offset of tile row
  // t, thread TY + i the output offset of tile column i (group digits, one
  // magic-number division each), so the load and store loops read them from
  // LDS instead of each thread dividing for every row it moves. A barrier
  // must separate prepare() from load().
  template <class A>
  __host__ __device__ static void prepare(const A& a, const TileCtx& c, int t, E* lds) {
    if constexpr (G) {
      int* o = offsets(lds);
      if (t < TY) {
        const int y = c.y0 + t;
        o[t] = y < a.Y ? tiled_in_y(a, (uint32_t)y) : 0;
      } else if (t < TY + TX) {
        const int x = c.x0 + (t - TY);
        o[t] = x < a.X ? tiled_out_x(a, (uint32_t)x) : 0;
      }
    }
  }

  template <class A>
  __host__ __device__ static TileCtx item(const A& a, uint32_t w) { return tile_item(a, w, TX, TY); }

  // LARGE: whole tiles are loaded non-temporally where the plan asks for it.
  template <bool LARGE = false, class A>
  __host__ __device__ static void load(const A& a, const TileCtx& c, int t,
                                       const E* __restrict__ in, E* lds) {
    VI r[NPR];
    const int lx = (t % LR) * VX;
    const int ly = t / LR;
    const int x = c.x0 + lx;
    if (c.full && (!G || a.yg.n == 1)) {
      const E* p = in + (c.off_in + x + (c.y0 + ly) * a.in_ys);
      const int step = RP * a.in_ys;
      if (LARGE && a.stream_in) {
        keep_branch();
#pragma unroll
        for (int j = 0; j < NPR; j++) r[j] = ld<true>(reinterpret_cast<const VI*>(p + j * step));
        keep_branch();
      } else {
#pragma unroll
        for (int j = 0; j < NPR; j++) r[j] = ld(reinterpret_cast<const VI*>(p + j * step));
      }
    } else if (G && LARGE && c.full && a.stream_in) {
      keep_branch();
      const E* p = in + (c.off_in + x);
#pragma unroll
      for (int j = 0; j < NPR; j++) r[j] = ld<true>(reinterpret_cast<const VI*>(p + offsets(lds)[ly + j * RP]));
      keep_branch();
    } else {
      const bool xin = x < a.X;
#pragma unroll
      for (int j = 0; j < NPR; j++) {
        const int y = c.y0 + ly + j * RP;
        const int yoff = G ? offsets(lds)[ly + j * RP] : y * a.in_ys;
        r[j] = VI{};
        if (xin && y < a.Y) r[j] = ld(reinterpret_cast<const VI*>(in + (c.off_in + x + yoff)));
      }
    }
    stash(t, r, lds);
  }

  // Rows and columns past the plane are stored too, and not read: no masks.
  __host__ __device__ static void stash(int t, const VI* r, E* lds) {
    const int lx = (t % LR) * VX;
    const int ly = t / LR;
#pragma unroll
    for (int j = 0; j < NPR; j++) {
#pragma unroll
      for (int e = 0; e < VX; e++) lds[(ly + j * RP) * PITCH + lx + e] = vget<E>(r[j], e);
    }
  }

  template <class A>
  __host__ __device__ static void store(const A& a, const TileCtx& c, int t,
                                        E* __restrict__ out, const E* lds) {
    const int ly = (t % LW) * VY;
    const int lx = t / LW;
    const int y = c.y0 + ly;
    VO r[NPW];
#pragma unroll
    for (int j = 0; j < NPW; j++)
#pragma unroll
      for (int e = 0; e < VY; e++) vset<E>(r[j], e, lds[(ly + e) * PITCH + lx + j * WP]);
    if (c.full && (!G || a.xg.n == 1)) {
      E* p = out + (c.off_out + y + (c.x0 + lx) * a.out_xs);
      const int step = WP * a.out_xs;
#pragma unroll
      for (int j = 0; j < NPW; j++) st(reinterpret_cast<VO*>(p + j * step), r[j]);
    } else {
      const bool yin = y < a.Y;
#pragma unroll
      for (int j = 0; j < NPW; j++) {
        const int x = c.x0 + lx + j * WP;
        const int xoff = G ? offsets(lds)[TY + lx + j * WP] : x * a.out_xs;
        if (yin && x < a.X) st(reinterpret_cast<VO*>(out + (c.off_out + y + xoff)), r[j]);
      }
    }
  }
};

// ---------------------------------------------------------------------------
// Skewed tiles, for planes whose output columns do not all start on 128-byte
// lines. Column x of a tile covers the TY rows that start at y0 - s(x), where
// s(x) is how far output row y0 of that column lies past a line boundary, so
// every store is an aligned 16-byte word and a tile writes whole lines; only
// a column's own first and last line are written in part. The tile's LDS holds
// LE (a line's elements) more rows than TY, of which each column uses its TY;
// each lane loads just the rows of its column, so no element is loaded twice.
// Bound by HBM. What it removes: lines written in two halves by two
// workgroups, which cost far more than their share of the bytes. What it costs:
// the input lines of the rows that a tile splits with its neighbours are read
// by both, in dispatch order into two L2s. (5, 97, 211, 331) f64 by the request
// counters: writes 1.063 -> 1.016, reads 1.002 -> 1.75 times the bytes, 129 ->
// 116 us. On MI355X, against unskewed tiles with their best lanes: (8191, 8193)
// f32 130 -> 94 us, (4097, 8191) f64 122 -> 94 us, (5, 97, 211, 331) f64 131 ->
// 107 us with 32 x 128 tiles (116 with the 32 x 64 that librettPlan takes); a
// copy of the bytes takes 85 us. That is among passes over three buffer pairs;
// where the input has just been written, (8191, 8193) goes from 97 to 91 us but
// (5, 97, 211, 331) from 115 to 117, and to 94-98 in the order across XCDs.
// One-element loads are as fast as 16-byte ones here (93-95 against 93 us,
// f32), and non-temporal loads slower (106 us), as neighbouring tiles share
// the lines of the rows they split. Tiles aligned to 64 bytes instead of 128
// cost 5-10%.
// ---------------------------------------------------------------------------
template <int B, int TX, int TY, int NTH, bool G>
struct SkewOps {
  using E = typename Word<B>::type;
  using V = typename Word<16>::type;
  static constexpr int NT = NTH;
  static constexpr int LE = 128 / B;               // elements per line
  static constexpr int PE = 16 / B;                // elements per output word
  static constexpr int R = TY + LE;                // tile rows held in LDS: row i is y0 - LE + i
  static constexpr int RP = NT / TX;               // rows per load pass
  static constexpr int NPR = (R + RP - 1) / RP;    // load passes
  static constexpr int LW = TY / PE;               // lanes per output column
  static constexpr int WP = NT / LW;               // columns per store pass
  static constexpr int NPW = TX / WP;              // store passes
  static constexpr int PITCH = TX + 1;
  // After the tile, ints: R input offsets of the rows (G), TX output offsets
  // of the columns (G).
  static constexpr int OFF_ELEMS = G ? ((R + TX) * 4 + B - 1) / B : 0;
  static constexpr int LDS_ELEMS = R * PITCH + OFF_ELEMS;
  static_assert(R + TX <= NT && NT % TX == 0 && TY % PE == 0 && NT % LW == 0 && TX % WP == 0 && NPW >= 1, "skew shape");

  __host__ __device__ static int* offsets(E* lds) { return reinterpret_cast<int*>(lds + R * PITCH); }
  __host__ __device__ static const int* offsets(const E* lds) {
    return reinterpret_cast<const int*>(lds + R * PITCH);
  }

  template <class A>
  __host__ __device__ static TileCtx item(const A& a, uint32_t w) { return tile_item(a, w, TX, TY); }

  // G only, as in TiledOps: prepare() with a barrier before load() where the y
  // group has several dims; else only the columns' output offsets are needed,
  // by store().
  template <class A>
  __host__ __device__ static bool early(const A& a) { return G && a.yg.n > 1; }
  template <class A>
  __host__ __device__ static void prepare(const A& a, const TileCtx& c, int t, E* lds) {
    int* o = offsets(lds);
    if (t < R) {
      const int y = c.y0 - LE + t;
      o[t] = y >= 0 && y < a.Y ? tiled_in_y(a, (uint32_t)y) : 0;
    } else if (t < R + TX) {
      const int x = c.x0 + (t - R);
      o[t] = x < a.X ? tiled_out_x(a, (uint32_t)x) : 0;
    }
  }

  // Output offset of tile column i, and its skew.
  template <class A>
  __host__ __device__ static int column(const A& a, const TileCtx& c, int i, const E* lds) {
    return c.off_out + (G ? offsets(lds)[R + i] : (c.x0 + i) * a.out_xs);
  }
  __host__ __device__ static int skew(int base, int phase) { return (base + phase) & (LE - 1); }

  // Tile rows [lo, hi) that a column with skew s covers.
  template <class A>
  __host__ __device__ static void rows(const A& a, const TileCtx& c, int s, int& lo, int& hi) {
    const int first = LE - c.y0, end = a.Y - c.y0 + LE;  // rows of y = 0 and y = Y
    lo = LE - s > first ? LE - s : first;
    hi = LE - s + TY < end ? LE - s + TY : end;
  }

  template <class A>
  __host__ __device__ static void load(const A& a, const TileCtx& c, int t, const E* __restrict__ in, E* lds,
                                       int phase) {
    const int lx = t % TX;
    const int ly = t / TX;
    int lo = 0, hi = 0;
    const int x = c.x0 + lx;
    if (x < a.X) rows(a, c, skew(c.off_out + (G ? tiled_out_x(a, (uint32_t)x) : x * a.out_xs), phase), lo, hi);
    const E* p = in + (c.off_in + c.x0 + lx);
    const int y = c.y0 - LE + ly;
    E r[NPR];
#pragma unroll
    for (int j = 0; j < NPR; j++) {
      const int i = ly + j * RP;
      r[j] = E{};
      if (i >= lo && i < hi) r[j] = ld(p + (early(a) ? offsets(lds)[i] : (y + j * RP) * a.in_ys));
    }
    if (G && !early(a) && t < TX && c.x0 + t < a.X) offsets(lds)[R + t] = tiled_out_x(a, (uint32_t)(c.x0 + t));
    // Rows of the tile that the column does not cover are stored too (and not
    // read): the lanes' masks then need no registers until here.
#pragma unroll
    for (int j = 0; j < NPR; j++) {
      const int i = ly + j * RP;
      if (RP * NPR == R || i < R) lds[i * PITCH + lx] = r[j];
    }
  }

  template <class A>
  __host__ __device__ static void store(const A& a, const TileCtx& c, int t, E* __restrict__ out,
                                        const E* lds, int phase) {
    const int ly = (t % LW) * PE;
    const int lx = t / LW;
#pragma unroll
    for (int j = 0; j < NPW; j++) {
      const int i = lx + j * WP;
      if (c.x0 + i >= a.X) continue;
      const int base = column(a, c, i, lds);
      const int s = skew(base, phase);
      const int y = c.y0 - s + ly;
      const E* q = lds + ((LE - s + ly) * PITCH + i);
      if (y >= 0 && y + PE <= a.Y) {
        V v;
#pragma unroll
        for (int k = 0; k < PE; k++) vset<E>(v, k, q[k * PITCH]);
        st(reinterpret_cast<V*>(out + (base + y)), v);
      } else {
#pragma unroll
        for (int k = 0; k < PE; k++)
          if (y + k >= 0 && y + k < a.Y) st(out + (base + y + k), q[k * PITCH]);
      }
    }
  }
};

// ---------------------------------------------------------------------------
// Narrow planes: X is at most kNarrowX columns and the rows lie back to back in
// the input (in_ys == X, y the input dim after x), as in an array of
// structures that becomes a structure of arrays. A tile is all X columns of TY
// rows: one contiguous stretch of the input, dealt to the threads element by
// element whatever X is, and X long runs of the output, skewed as in SkewOps.
// Bound by HBM. On MI355X, [7, 9587595] f32 takes 134 us as a Packed plan of
// 10381 elements, which writes its lines in parts, 92 us here; [5, 6710040]
// f64 118 -> 92 us, [2, 13107201] f64 288 -> 70 us; copies of the bytes take
// 85, 85 and 66 us. Tiles are small (8 to 16 KiB) for 7 workgroups on a CU: of
// 28 KiB with 512 threads, whose registers leave two, 113 us for the first.
// ---------------------------------------------------------------------------
template <int B, int NTH, int NL>
struct NarrowOps {
  using E = typename Word<B>::type;
  using V = typename Word<16>::type;
  static constexpr int NT = NTH;
  static constexpr int LE = 128 / B;
  static constexpr int PE = 16 / B;
  static constexpr int MAX = NT * NL;  // elements of a tile, with its line more of rows
  static constexpr int NW = (NL + PE - 1) / PE;  // store passes

  // LDS: rows of odd pitch, then X output offsets of the columns.
  template <class A>
  __host__ __device__ static int pitch(const A& a) { return a.X | 1; }
  template <class A>
  __host__ __device__ static int rows(const A& a) { return (PE << a.word_shift) + LE; }
  template <class A>
  __host__ __device__ static int* offsets(const A& a, E* lds) {
    return reinterpret_cast<int*>(lds + rows(a) * pitch(a));
  }
  template <class A>
  __host__ __device__ static const int* offsets(const A& a, const E* lds) {
    return reinterpret_cast<const int*>(lds + rows(a) * pitch(a));
  }

  template <class A>
  __host__ __device__ static TileCtx item(const A& a, uint32_t w) {
    return tile_item(a, w, a.X, PE << a.word_shift);
  }

  // Before load(), with a barrier between.
  template <class A>
  __host__ __device__ static constexpr bool early(const A&) { return true; }
  template <class A>
  __host__ __device__ static void prepare(const A& a, const TileCtx& c, int t, E* lds) {
    if (t < a.X) offsets(a, lds)[t] = c.off_out + tiled_out_x(a, (uint32_t)t);
  }

  template <class A>
  __host__ __device__ static void load(const A& a, const TileCtx& c, int t, const E* __restrict__ in, E* lds,
                                       int phase) {
    const int ty = PE << a.word_shift;
    const int n = (ty + LE) * a.X;
    // Element i of the tile lies i elements past row y0 - LE of the plane;
    // elements [lo, hi) are in the plane.
    const E* p = in + c.off_in;
    const int p0 = (c.y0 - LE) * a.X;
    const int lo = p0 < 0 ? -p0 : 0;
    const long long left = (long long)a.Y * a.X - p0;
    const int hi = n < left ? n : (int)left;
    E r[NL];
#pragma unroll
    for (int j = 0; j < NL; j++) {
      const int i = t + j * NT;
      r[j] = E{};
      bool use = i >= lo && i < hi;
      // Only the first and last line's elements of rows depend on the column's
      // skew.
      if (use && (i < LE * a.X || i >= ty * a.X)) {
        const int row = (int)fdiv((uint32_t)i, a.x_div);
        const int d = row - LE + ((offsets(a, lds)[i - row * a.X] + phase) & (LE - 1));
        use = d >= 0 && d < ty;
      }
      if (use) r[j] = ld(p + (p0 + i));
    }
    // An odd pitch X is the input's own layout.
    if (a.X & 1) {
#pragma unroll
      for (int j = 0; j < NL; j++)
        if (t + j * NT < n) lds[t + j * NT] = r[j];
    } else {
#pragma unroll
      for (int j = 0; j < NL; j++) {
        const int i = t + j * NT;
        if (i < n) lds[i + (int)fdiv((uint32_t)i, a.x_div)] = r[j];
      }
    }
  }

  template <class A>
  __host__ __device__ static void store(const A& a, const TileCtx& c, int t, E* __restrict__ out,
                                        const E* lds, int phase) {
    const int* off = offsets(a, lds);
    const int P = pitch(a);
    const int nw = a.X << a.word_shift;
#pragma unroll
    for (int j = 0; j < NW; j++) {
      const int i = t + j * NT;
      if (i >= nw) break;
      const int x = i >> a.word_shift;
      const int ly = (i - (x << a.word_shift)) * PE;
      const int base = off[x];
      const int s = (base + phase) & (LE - 1);
      const int y = c.y0 - s + ly;
      const E* q = lds + ((LE - s + ly) * P + x);
      if (y >= 0 && y + PE <= a.Y) {
        V v;
#pragma unroll
        for (int k = 0; k < PE; k++) vset<E>(v, k, q[k * P]);
        st(reinterpret_cast<V*>(out + (base + y)), v);
      } else {
#pragma unroll
        for (int k = 0; k < PE; k++)
          if (y + k >= 0 && y + k < a.Y) st(out + (base + y + k), q[k * P]);
      }
    }
  }
};

// ---------------------------------------------------------------------------
// Short columns: Y is at most kNarrowX elements and the columns lie back to back
// in the output (out_xs == Y, x the output dim after y), as in a structure of
// arrays that becomes an array of structures: NarrowOps the other way round. A
// tile is a stretch of CH output elements that starts on a line; it reads a run
// of each of the Y input rows and writes whole 16-byte words. Bound by HBM. On
// MI355X, against the best other plan: [26000000, 2] f32 455 -> 72 us,
// [13000000, 2] f64 315 -> 70 us; copies of the bytes take 66 us.
// ---------------------------------------------------------------------------
template <int B, int NTH, int NL>
struct ShortOps {
  using E = typename Word<B>::type;
  using V = typename Word<16>::type;
  static constexpr int NT = NTH;
  static constexpr int LE = 128 / B;
  static constexpr int PE = 16 / B;
  static constexpr int NW = NL / PE;        // 16-byte words per thread
  static constexpr int CH = NT * NW * PE;   // elements of a tile
  static_assert(NL % PE == 0 && CH % LE == 0, "short shape");
  // Columns of a tile whose first and last may be cut; loads per thread.
  __host__ __device__ static int columns(int Y) { return (CH + Y - 2) / Y + 1; }
  static constexpr int NLD = NL + 1;  // columns(Y) * Y <= CH + 2 * Y <= (NL + 1) * NT

  template <class A>
  __host__ __device__ static int pitch(const A& a) { return (int)a.nx_div.d | 1; }
  template <class A>
  __host__ __device__ static TileCtx item(const A& a, uint32_t w) {
    TileCtx c;
    const uint32_t mb = fdiv(w, a.ntiles_div);
    c.x0 = (int)(w - mb * (uint32_t)a.ntiles);  // tile of the plane
    c.y0 = 0;
    outer_offsets(a.outer, mb, c.off_in, c.off_out);
    c.full = false;
    return c;
  }
  // First element of the tile, counted from the plane's first output element.
  __host__ __device__ static int first(const TileCtx& c, int phase) {
    return c.x0 * CH - ((c.off_out + phase) & (LE - 1));
  }
  // Before load(), with a barrier between.
  template <class A>
  __host__ __device__ static constexpr bool early(const A&) { return true; }
  // After the tile's Y rows, their input offsets (ints).
  template <class A>
  __host__ __device__ static const int* offsets(const A& a, const E* lds) {
    return reinterpret_cast<const int*>(lds + a.Y * pitch(a));
  }
  template <class A>
  __host__ __device__ static void prepare(const A& a, const TileCtx&, int t, E* lds) {
    if (t < a.Y) const_cast<int*>(offsets(a, lds))[t] = tiled_in_y(a, (uint32_t)t);
  }

  template <class A>
  __host__ __device__ static void load(const A& a, const TileCtx& c, int t, const E* __restrict__ in, E* lds,
                                       int phase) {
    const int e0 = first(c, phase), n = a.X * a.Y;
    const uint32_t lo = e0 < 0 ? 0 : (uint32_t)e0;
    const uint32_t hi = (long long)n - e0 < CH ? (uint32_t)n : (uint32_t)(e0 + CH);
    const int xa = (int)fdiv(lo, a.x_div);
    const E* p = in + (c.off_in + xa);
    const int* off = offsets(a, lds);
    E r[NLD];
#pragma unroll
    for (int j = 0; j < NLD; j++) {
      const uint32_t i = (uint32_t)(t + j * NT);
      const int y = (int)fdiv(i, a.nx_div);
      const int xi = (int)(i - (uint32_t)y * a.nx_div.d);
      const uint32_t e = (uint32_t)(xa + xi) * (uint32_t)a.Y + (uint32_t)y;
      r[j] = E{};
      if (y < a.Y && e >= lo && e < hi) r[j] = ld(p + (xi + off[y]));
    }
#pragma unroll
    for (int j = 0; j < NLD; j++) {
      const uint32_t i = (uint32_t)(t + j * NT);
      const int y = (int)fdiv(i, a.nx_div);
      if (y < a.Y) lds[y * pitch(a) + (int)(i - (uint32_t)y * a.nx_div.d)] = r[j];
    }
  }

  template <class A>
  __host__ __device__ static void store(const A& a, const TileCtx& c, int t, E* __restrict__ out,
                                        const E* lds, int phase) {
    const int e0 = first(c, phase);
    const uint32_t n = (uint32_t)(a.X * a.Y);
    const int xa = (int)fdiv((uint32_t)(e0 < 0 ? 0 : e0), a.x_div);
    const int P = pitch(a);
#pragma unroll
    for (int j = 0; j < NW; j++) {
      // Elements before the plane wrap to values above any volume.
      const uint32_t e = (uint32_t)e0 + (uint32_t)((t + j * NT) * PE);
      if (e < n && n - e >= (uint32_t)PE) {
        int x = (int)fdiv(e, a.x_div);
        int y = (int)e - x * a.Y;
        V v;
#pragma unroll
        for (int k = 0; k < PE; k++) {
          vset<E>(v, k, lds[y * P + (x - xa)]);
          if (++y == a.Y) {
            y = 0;
            x++;
          }
        }
        st(reinterpret_cast<V*>(out + (c.off_out + (int)e)), v);
      } else {
#pragma unroll
        for (int k = 0; k < PE; k++)
          if (e + k < n) {
            const int x = (int)fdiv(e + k, a.x_div);
            st(out + (c.off_out + (int)(e + k)), lds[((int)(e + k) - x * a.Y) * P + (x - xa)]);
          }
      }
    }
  }
};

// ---------------------------------------------------------------------------
// TiledCopy: rows that are contiguous in both tensors (perm[0] == 0). The
// output is written front to back in 16-byte words that start on its 16-byte
// boundaries, so a wave stores 1024 consecutive bytes in whole lines whatever
// the row length; each thread finds its word's row and input offset by
// itself and loads the word from wherever the row starts (any element
// boundary). A word that crosses a row's end is loaded element by element.
// Bound by HBM. On MI355X a copy of [2307, 115, 126] f64 rows (18456 B, no
// row on a line boundary) takes 89 us against 128 us for row tiles of 8-byte
// words, whose lines are written in two parts by different workgroups, and
// [1024, 256, 256] f32 takes 86 us against 94 us; a plain copy of the bytes
// takes 85 us. Out of HBM one word per thread runs faster than two or four
// (85.8, 87.8, 90.3 us; in the batched engine 3.34 ms against 3.46 ms for
// four): more, shorter workgroups keep the open DRAM pages close together. Out
// of the Infinity Cache a workgroup's own time counts for more, and two words
// per thread are in flight at once (NP = 2; copy_words() in the planner).
// Reference counterpart: transposeTiledCopy, src/kernel.cpp:453-545.
// ---------------------------------------------------------------------------
template <int B, int NP = 1>
struct CopyOps {
  using E = typename Word<B>::type;
  using V = typename Word<16>::type;
  static constexpr int NT = 256;
  static constexpr int PE = 16 / B;         // elements per word
  static constexpr int PER = NP * NT * PE;  // elements per item

  // Words of item w start at element w * PER - phase: word boundaries are
  // 16-byte boundaries of the output's addresses, and items start on lines.
  template <class A>
  __host__ __device__ static void run(const A& a, uint32_t w, int t, const E* __restrict__ in,
                                      E* __restrict__ out) {
    if (a.stream_in) {
      keep_branch();
      move<true>(a, w, t, in, out);
      keep_branch();
    } else {
      move<false>(a, w, t, in, out);
    }
  }

  template <bool STREAM, class A>
  __host__ __device__ static void move(const A& a, uint32_t w, int t, const E* __restrict__ in,
                                       E* __restrict__ out) {
    const uint32_t first_e = first(w, t, line_phase(out));
    V r[NP];
#pragma unroll
    for (int j = 0; j < NP; j++) {
      const uint32_t e = first_e + (uint32_t)(j * NT * PE);
      if (!whole(a, e)) continue;
      const uint32_t row = fdiv(e, a.row_div);
      const int c = (int)(e - row * (uint32_t)a.X);
      if (PE == 1 || a.X - c >= PE) {
        r[j] = ld_unaligned<V, B, STREAM>(in + (copy_row_offset(a.rows, row) + c));
      } else {
#pragma unroll
        for (int k = 0; k < PE; k++) vset<E>(r[j], k, ld(in + source(a, e + k)));
      }
    }
#pragma unroll
    for (int j = 0; j < NP; j++) {
      const uint32_t e = first_e + (uint32_t)(j * NT * PE);
      if (whole(a, e)) {
        st(reinterpret_cast<V*>(out + e), r[j]);
      } else {
#pragma unroll
        for (int k = 0; k < PE; k++)
          if (e + k < (uint32_t)a.n) st(out + (e + k), ld(in + source(a, e + k)));
      }
    }
  }

  // First element of thread t's first word in item w. Unsigned: elements before the
  // tensor wrap to values above any volume, as do words past 2^31.
  __host__ __device__ static uint32_t first(uint32_t w, int t, int phase) {
    return w * (uint32_t)PER + (uint32_t)(t * PE) - (uint32_t)phase;
  }
  template <class A>
  __host__ __device__ static bool whole(const A& a, uint32_t e) {
    return e < (uint32_t)a.n && (uint32_t)a.n - e >= (uint32_t)PE;
  }
  // Input offset of output element e.
  template <class A>
  __host__ __device__ static int source(const A& a, uint32_t e) {
    const uint32_t row = fdiv(e, a.row_div);
    return copy_row_offset(a.rows, row) + (int)(e - row * (uint32_t)a.X);
  }
};

// ---------------------------------------------------------------------------
// Packed / PackedSplit: a whole on-chip sub-tensor (one chunk of the split dim
// for PackedSplit) goes through LDS per outer index. Each thread owns NREG
// positions of the staged volume and keeps their input offset, output offset
// and LDS read position in registers for all outer indices of its block.
// Reference counterparts: transposePacked (src/kernel.cpp:175-296) and
// transposePackedSplit (src/kernel.cpp:304-444).
// ---------------------------------------------------------------------------
template <int B, int NREG>
struct PackedOps {
  using E = typename Word<B>::type;

  struct Pre {
    int in[NREG];
    int out[NREG];
    int sh[NREG];
    int vol;
    int base_in, base_out;
    FastDiv pad;
  };

  __host__ __device__ static void prepare(const PackedArgs& a, int split, int t, int nt, Pre& p) {
    const int q0 = a.split_dim / a.num_split;
    const int c0 = (int)((long long)split * a.split_dim / a.num_split);
    const int c1 = (int)((long long)(split + 1) * a.split_dim / a.num_split);
    const int plus = (c1 - c0) - q0;
    const StagedShape& s = a.shape[plus];
    p.vol = s.vol;
    p.pad = s.pad;
    p.base_in = c0 * a.split_in_stride;
    p.base_out = c0 * a.split_out_stride;
#pragma unroll
    for (int r = 0; r < NREG; r++) {
      uint32_t k = (uint32_t)(t + r * nt);
      int oi = 0;
      for (int d = 0; d < s.n; d++) {
        uint32_t q = fdiv(k, s.din[d]);
        oi += (int)(k - q * s.din[d].d) * s.ct_in[d];
        k = q;
      }
      k = (uint32_t)(t + r * nt);
      int oo = 0, sh = 0;
      for (int d = 0; d < s.n; d++) {
        uint32_t q = fdiv(k, s.dout[d]);
        int digit = (int)(k - q * s.dout[d].d);
        oo += digit * s.ct_out[d];
        sh += digit * s.ct_sh[d];
        k = q;
      }
      p.in[r] = oi;
      p.out[r] = oo;
      p.sh[r] = sh;
    }
  }

  __host__ __device__ static void load(const Pre& p, int off_in, int t, int nt,
                                       const E* __restrict__ in, E* lds) {
    E r[NREG];
    fetch(p, off_in, t, nt, in, r);
    stash(p, t, nt, r, lds);
  }

  // The two halves of load(): global memory to registers, registers to LDS.
  __host__ __device__ static void fetch(const Pre& p, int off_in, int t, int nt, const E* __restrict__ in,
                                        E* r) {
    const E* base = in + (p.base_in + off_in);
#pragma unroll
    for (int j = 0; j < NREG; j++)
      if (t + j * nt < p.vol) r[j] = ld(base + p.in[j]);
  }
  __host__ __device__ static void stash(const Pre& p, int t, int nt, const E* r, E* lds) {
#pragma unroll
    for (int j = 0; j < NREG; j++)
      if (t + j * nt < p.vol) {
        const uint32_t q = (uint32_t)(t + j * nt);
        lds[q + fdiv(q, p.pad)] = r[j];
      }
  }

  __host__ __device__ static void store(const Pre& p, int off_out, int t, int nt,
                                        E* __restrict__ out, const E* lds) {
    E r[NREG];
#pragma unroll
    for (int j = 0; j < NREG; j++)
      if (t + j * nt < p.vol) r[j] = lds[p.sh[j]];
    E* base = out + (p.base_out + off_out);
#pragma unroll
    for (int j = 0; j < NREG; j++)
      if (t + j * nt < p.vol) st(base + p.out[j], r[j]);
  }
};

}  // namespace lrt
