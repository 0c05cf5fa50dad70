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

// ---------------------------------------------------------------------------
// Tiled: a TX x TY tile of the (x, y) plane goes through LDS. Reads walk x
// (contiguous in the input) with VX elements per lane; writes walk y
// (contiguous in the output) with VY elements per lane. One LDS row of pitch
// TX + 1 per y keeps the column reads of the write phase spread over banks.
// When x or y is a group of dims, each row (column) finds its offset on the
// other side from the group's digits; a full tile of one-dim groups steps
// through memory by a fixed stride instead.
// Reference counterpart: transposeTiled, src/kernel.cpp:48-170.
// ---------------------------------------------------------------------------
// G = false compiles only the one-dim-group path (the kernel then needs no
// registers for group maps); G = true handles groups of several dims too.
template <int B, int TX, int TY, int VX, int VY, bool G = false>
struct TiledOps {
  using E = typename Word<B>::type;
  using VI = typename Word<B * VX>::type;
  using VO = typename Word<B * VY>::type;
  static constexpr int NT = 256;
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
  __host__ __device__ static void prepare(const TiledArgs& a, const TileCtx& c, int t, E* lds) {
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

  __host__ __device__ static TileCtx item(const TiledArgs& a, uint32_t w) {
    TileCtx c;
    uint32_t mb = fdiv(w, a.ntiles_div);
    uint32_t tile = w - mb * (uint32_t)a.ntiles;
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
    c.x0 = (int)tx * TX;
    c.y0 = (int)ty * TY;
    outer_offsets(a.outer, mb, c.off_in, c.off_out);
    c.full = (c.x0 + TX <= a.X) && (c.y0 + TY <= a.Y);
    return c;
  }

  __host__ __device__ static void load(const TiledArgs& a, const TileCtx& c, int t,
                                       const E* __restrict__ in, E* lds) {
    VI r[NPR];
    fetch(a, c, t, in, r, lds);
    stash(a, c, t, r, lds);
  }

  // The two halves of load(): the tile's input rows into registers, then
  // registers into LDS (the pipelined kernel fetches the next tile between
  // them and the current tile's store phase).
  __host__ __device__ static void fetch(const TiledArgs& a, const TileCtx& c, int t, const E* __restrict__ in,
                                        VI* r, const E* lds) {
    const int lx = (t % LR) * VX;
    const int ly = t / LR;
    const int x = c.x0 + lx;
    if (c.full && (!G || a.yg.n == 1)) {
      const E* p = in + (c.off_in + x + (c.y0 + ly) * a.in_ys);
      const int step = RP * a.in_ys;
#pragma unroll
      for (int j = 0; j < NPR; j++) r[j] = ld(reinterpret_cast<const VI*>(p + j * step));
    } else {
      const bool xin = x < a.X;
#pragma unroll
      for (int j = 0; j < NPR; j++) {
        const int y = c.y0 + ly + j * RP;
        const int yoff = G ? offsets(lds)[ly + j * RP] : y * a.in_ys;
        if (xin && y < a.Y) r[j] = ld(reinterpret_cast<const VI*>(in + (c.off_in + x + yoff)));
      }
    }
  }
  __host__ __device__ static void stash(const TiledArgs& a, const TileCtx& c, int t, const VI* r, E* lds) {
    const int lx = (t % LR) * VX;
    const int ly = t / LR;
    const bool xin = c.x0 + lx < a.X;
#pragma unroll
    for (int j = 0; j < NPR; j++) {
      if (c.full || (xin && c.y0 + ly + j * RP < a.Y)) {
#pragma unroll
        for (int e = 0; e < VX; e++) lds[(ly + j * RP) * PITCH + lx + e] = vget<E>(r[j], e);
      }
    }
  }

  __host__ __device__ static void store(const TiledArgs& a, const TileCtx& c, int t,
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
// TiledCopy: rows that are contiguous in both tensors (perm[0] == 0). The
// output is written front to back in 16-byte words that start on its 16-byte
// boundaries, so a wave stores 1024 consecutive bytes in whole lines whatever
// the row length; each thread finds its word's row and input offset by
// itself and loads the word from wherever the row starts (any element
// boundary). A word that crosses a row's end is loaded element by element.
// Bound by HBM. On MI355X a copy of [2307, 115, 126] f64 rows (18456 B, no
// row on a line boundary) takes 86 us against 129 us for row tiles of 8-byte
// words, whose lines are written in two parts by different workgroups, and
// [1024, 256, 256] f32 takes 86 us against 94 us; a plain copy of the bytes
// takes 85 us. One word per thread runs faster than two or four (85.8, 87.8,
// 90.3 us; in the batched engine 3.34 ms against 3.46 ms for four): more,
// shorter workgroups keep the open DRAM pages close together.
// Reference counterpart: transposeTiledCopy, src/kernel.cpp:453-545.
// ---------------------------------------------------------------------------
template <int B>
struct CopyOps {
  using E = typename Word<B>::type;
  using V = typename Word<16>::type;
  static constexpr int NT = 256;
  static constexpr int PE = 16 / B;    // elements per word
  static constexpr int PER = NT * PE;  // elements per item

  // Words of item w start at element w * PER - phase: word boundaries are
  // 16-byte boundaries of the output's addresses, and items start on lines.
  __host__ __device__ static void run(const CopyArgs& a, uint32_t w, int t, const E* __restrict__ in,
                                      E* __restrict__ out) {
    if (a.stream_in)
      move<true>(a, w, t, in, out);
    else
      move<false>(a, w, t, in, out);
  }

  template <bool STREAM>
  __host__ __device__ static void move(const CopyArgs& a, uint32_t w, int t, const E* __restrict__ in,
                                       E* __restrict__ out) {
    const uint32_t e = first(w, t, line_phase(out));
    if (whole(a, e)) {
      V r;
      const uint32_t row = fdiv(e, a.row_div);
      const int c = (int)(e - row * (uint32_t)a.X);
      if (a.X - c >= PE) {
        r = ld_unaligned<V, B, STREAM>(in + (copy_row_offset(a.rows, row) + c));
      } else {
#pragma unroll
        for (int k = 0; k < PE; k++) vset<E>(r, k, ld(in + source(a, e + k)));
      }
      st(reinterpret_cast<V*>(out + e), r);
    } else {
#pragma unroll
      for (int k = 0; k < PE; k++)
        if (e + k < (uint32_t)a.n) st(out + (e + k), ld(in + source(a, e + k)));
    }
  }

  // First element of thread t in item w. Unsigned: elements before the
  // tensor wrap to values above any volume, as do words past 2^31.
  __host__ __device__ static uint32_t first(uint32_t w, int t, int phase) {
    return w * (uint32_t)PER + (uint32_t)(t * PE) - (uint32_t)phase;
  }
  __host__ __device__ static bool whole(const CopyArgs& a, uint32_t e) {
    return e < (uint32_t)a.n && (uint32_t)a.n - e >= (uint32_t)PE;
  }
  // Input offset of output element e.
  __host__ __device__ static int source(const CopyArgs& a, uint32_t e) {
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
