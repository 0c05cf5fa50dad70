// Kernel of the batched engine, its shape table and host replay.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "batch.h"

#include <cstdlib>
#include "kernel_ops.h"
#include "kernels.h"

namespace lrt {

namespace {

// Shape table: id, method, element bytes, four method parameters, group flag,
// tile form
//   Tiled:     tile_x, tile_y, vec_x, vec_y; group flag 1 for planes over
//              dim groups (rectangular tiles: their own family, so the one-dim
//              kernels keep their registers); narrow and short tiles size
//              themselves
//   TiledCopy: none
//   Packed:    nreg
#define LRT_BATCH_TABLE(X)                                                  \
  X(0, kTiled, 4, 64, 64, 1, 1, 0, kTileRect) X(1, kTiled, 4, 64, 64, 4, 1, 0, kTileRect)         \
  X(2, kTiled, 4, 64, 64, 1, 4, 0, kTileRect) X(3, kTiled, 4, 64, 64, 4, 4, 0, kTileRect)         \
  X(4, kTiled, 8, 32, 32, 1, 1, 0, kTileRect) X(5, kTiled, 8, 32, 32, 2, 1, 0, kTileRect)         \
  X(6, kTiled, 8, 32, 32, 1, 2, 0, kTileRect) X(7, kTiled, 8, 32, 32, 2, 2, 0, kTileRect)         \
  X(8, kTiled, 16, 32, 32, 1, 1, 0, kTileRect)                                         \
  X(9, kTiledCopy, 4, 0, 0, 0, 0, 0, kTileRect) X(10, kTiledCopy, 8, 0, 0, 0, 0, 0, kTileRect)    \
  X(11, kTiledCopy, 16, 0, 0, 0, 0, 0, kTileRect)                                      \
  X(12, kPacked, 4, 1, 0, 0, 0, 0, kTileRect) X(13, kPacked, 4, 2, 0, 0, 0, 0, kTileRect)         \
  X(14, kPacked, 4, 4, 0, 0, 0, 0, kTileRect) X(15, kPacked, 4, 8, 0, 0, 0, 0, kTileRect)         \
  X(16, kPacked, 8, 1, 0, 0, 0, 0, kTileRect) X(17, kPacked, 8, 2, 0, 0, 0, 0, kTileRect)         \
  X(18, kPacked, 8, 4, 0, 0, 0, 0, kTileRect) X(19, kPacked, 8, 8, 0, 0, 0, 0, kTileRect)         \
  X(20, kPacked, 16, 1, 0, 0, 0, 0, kTileRect) X(21, kPacked, 16, 2, 0, 0, 0, 0, kTileRect)       \
  X(22, kPacked, 16, 4, 0, 0, 0, 0, kTileRect)                                         \
  X(23, kTiled, 4, 64, 64, 1, 1, 1, kTileRect) X(24, kTiled, 4, 64, 64, 4, 1, 1, kTileRect)       \
  X(25, kTiled, 4, 64, 64, 1, 4, 1, kTileRect) X(26, kTiled, 4, 64, 64, 4, 4, 1, kTileRect)       \
  X(27, kTiled, 8, 32, 32, 1, 1, 1, kTileRect) X(28, kTiled, 8, 32, 32, 2, 1, 1, kTileRect)       \
  X(29, kTiled, 8, 32, 32, 1, 2, 1, kTileRect) X(30, kTiled, 8, 32, 32, 2, 2, 1, kTileRect)       \
  X(31, kTiled, 16, 32, 32, 1, 1, 1, kTileRect) \
  X(32, kTiled, 4, 32, 64, 1, 4, 0, kTileSkew) X(33, kTiled, 4, 32, 64, 1, 4, 1, kTileSkew)   \
  X(34, kTiled, 8, 32, 32, 1, 2, 0, kTileSkew) X(35, kTiled, 8, 32, 32, 1, 2, 1, kTileSkew)   \
  X(36, kTiled, 16, 16, 32, 1, 1, 0, kTileSkew) X(37, kTiled, 16, 16, 32, 1, 1, 1, kTileSkew) \
  X(38, kTiled, 4, 0, 0, 1, 4, 0, kTileNarrow) X(39, kTiled, 8, 0, 0, 1, 2, 0, kTileNarrow)   \
  X(40, kTiled, 16, 0, 0, 1, 1, 0, kTileNarrow) X(41, kTiled, 4, 0, 0, 1, 4, 0, kTileShort)   \
  X(42, kTiled, 8, 0, 0, 1, 2, 0, kTileShort) X(43, kTiled, 16, 0, 0, 1, 1, 0, kTileShort)

struct BatchShape {
  int id, method, b, p1, p2, p3, p4, g, form;
};
#define LRT_BATCH_ROW(ID, M, B, P1, P2, P3, P4, G, FORM) {ID, M, B, P1, P2, P3, P4, G, FORM},
const BatchShape kBatchShapes[] = {LRT_BATCH_TABLE(LRT_BATCH_ROW)};
#undef LRT_BATCH_ROW

// The problem owning unit u of nprob problems: the p with start[p] <= u <
// start[p + 1]. Each step the wave's lanes test 64 evenly spaced problems with
// one load and a ballot, so 4096 problems take two dependent loads (a binary
// search takes 12). hits(lo, n, step): how many of the lanes' problems lo,
// lo + step, ... below lo + n start at u or before (the first ones, as starts
// ascend, and start[lo] among them).
template <class HITS>
__host__ __device__ __forceinline__ int batch_find(int nprob, HITS&& hits) {
  int lo = 0, n = nprob;  // p is in [lo, lo + n)
  while (n > 1) {
    const int step = (n + 63) >> 6;
    const int last = hits(lo, n, step) - 1;
    lo += last * step;
    n = step < n - last * step ? step : n - last * step;
  }
  return lo;
}
__host__ __device__ __forceinline__ bool starts_by(const int* start, int u, int lo, int n, int step, int lane) {
  const int i = lane * step;
  return i < n && start[lo + i] <= u;
}

// The unit of workgroup (bx, by) of a grid gx wide, -1 past the last one.
__host__ __device__ __forceinline__ int unit_at(uint32_t bx, uint32_t by, uint32_t gx, int total) {
  const uint32_t u = by * gx + bx;
  return u < (uint32_t)total ? (int)u : -1;
}

template <int B, int TX, int TY, int VX, int VY, bool G = false>
__device__ __forceinline__ void dev_tiled(const BatchDesc& D, int lu, unsigned char* lds_raw) {
  using Ops = TiledOps<B, TX, TY, VX, VY, G>;
  using E = typename Ops::E;
  E* lds = reinterpret_cast<E*>(lds_raw);
  for (int w = lu; w < D.items; w += D.groups) {
    const TileCtx c = Ops::item(D.a.tiled, (uint32_t)w);
    if constexpr (G) {
      Ops::prepare(D.a.tiled, c, threadIdx.x, lds);
      __syncthreads();
    }
    Ops::load(D.a.tiled, c, threadIdx.x, static_cast<const E*>(D.in), lds);
    __syncthreads();
    Ops::store(D.a.tiled, c, threadIdx.x, static_cast<E*>(D.out), lds);
    __syncthreads();
  }
}

// Skewed, narrow and short tiles.
template <class Ops>
__device__ __forceinline__ void dev_lines(const BatchDesc& D, int lu, unsigned char* lds_raw) {
  using E = typename Ops::E;
  E* lds = reinterpret_cast<E*>(lds_raw);
  const TiledArgs& a = D.a.tiled;
  E* out = static_cast<E*>(D.out);
  const int phase = line_phase(out);
  for (int w = lu; w < D.items; w += D.groups) {
    const TileCtx c = Ops::item(a, (uint32_t)w);
    if (Ops::early(a)) {
      Ops::prepare(a, c, threadIdx.x, lds);
      __syncthreads();
    }
    Ops::load(a, c, threadIdx.x, static_cast<const E*>(D.in), lds, phase);
    __syncthreads();
    Ops::store(a, c, threadIdx.x, out, lds, phase);
    __syncthreads();
  }
}

template <int B>
__device__ __forceinline__ void dev_copy(const BatchDesc& D, int lu) {
  using Ops = CopyOps<B>;
  using E = typename Ops::E;
  for (int w = lu; w < D.items; w += D.groups)
    Ops::run(D.a.copy, (uint32_t)w, threadIdx.x, static_cast<const E*>(D.in), static_cast<E*>(D.out));
}

template <int B, int NREG>
__device__ __forceinline__ void dev_packed(const BatchDesc& D, int lu, unsigned char* lds_raw) {
  using Ops = PackedOps<B, NREG>;
  using E = typename Ops::E;
  E* lds = reinterpret_cast<E*>(lds_raw);
  const PackedArgs& a = D.a.packed;
  const uint32_t og = fdiv((uint32_t)lu, D.split_div);
  const int split = lu - (int)(og * D.split_div.d);
  typename Ops::Pre p;
  Ops::prepare(a, split, threadIdx.x, 256, p);
  for (int o = (int)og; o < a.vol_outer; o += D.groups) {
    int off_in, off_out;
    outer_offsets(a.outer, (uint32_t)o, off_in, off_out);
    Ops::load(p, off_in, threadIdx.x, 256, static_cast<const E*>(D.in), lds);
    __syncthreads();
    Ops::store(p, off_out, threadIdx.x, 256, static_cast<E*>(D.out), lds);
    __syncthreads();
  }
}

// Runs unit lu of descriptor D if its shape belongs to family FAM (the
// switch of each family kernel holds only that family's shapes, which keeps
// its register use to what those shapes need).
template <int FAM>
__device__ __forceinline__ void dev_unit(const BatchDesc& D, int lu, unsigned char* lds) {
  if constexpr (FAM == kFamTiled) {
    switch (D.variant) {
      case 0: dev_tiled<4, 64, 64, 1, 1>(D, lu, lds); break;
      case 1: dev_tiled<4, 64, 64, 4, 1>(D, lu, lds); break;
      case 2: dev_tiled<4, 64, 64, 1, 4>(D, lu, lds); break;
      case 3: dev_tiled<4, 64, 64, 4, 4>(D, lu, lds); break;
      case 4: dev_tiled<8, 32, 32, 1, 1>(D, lu, lds); break;
      case 5: dev_tiled<8, 32, 32, 2, 1>(D, lu, lds); break;
      case 6: dev_tiled<8, 32, 32, 1, 2>(D, lu, lds); break;
      case 7: dev_tiled<8, 32, 32, 2, 2>(D, lu, lds); break;
      case 8: dev_tiled<16, 32, 32, 1, 1>(D, lu, lds); break;
      default: break;
    }
  } else if constexpr (FAM == kFamTiledG) {
    switch (D.variant) {
      case 23: dev_tiled<4, 64, 64, 1, 1, true>(D, lu, lds); break;
      case 24: dev_tiled<4, 64, 64, 4, 1, true>(D, lu, lds); break;
      case 25: dev_tiled<4, 64, 64, 1, 4, true>(D, lu, lds); break;
      case 26: dev_tiled<4, 64, 64, 4, 4, true>(D, lu, lds); break;
      case 27: dev_tiled<8, 32, 32, 1, 1, true>(D, lu, lds); break;
      case 28: dev_tiled<8, 32, 32, 2, 1, true>(D, lu, lds); break;
      case 29: dev_tiled<8, 32, 32, 1, 2, true>(D, lu, lds); break;
      case 30: dev_tiled<8, 32, 32, 2, 2, true>(D, lu, lds); break;
      case 31: dev_tiled<16, 32, 32, 1, 1, true>(D, lu, lds); break;
      default: break;
    }
  } else if constexpr (FAM == kFamLines) {
    switch (D.variant) {
      case 9: dev_copy<4>(D, lu); break;
      case 10: dev_copy<8>(D, lu); break;
      case 11: dev_copy<16>(D, lu); break;
      case 32: dev_lines<SkewOps<4, 32, 64, 256, false>>(D, lu, lds); break;
      case 33: dev_lines<SkewOps<4, 32, 64, 256, true>>(D, lu, lds); break;
      case 34: dev_lines<SkewOps<8, 32, 32, 256, false>>(D, lu, lds); break;
      case 35: dev_lines<SkewOps<8, 32, 32, 256, true>>(D, lu, lds); break;
      case 36: dev_lines<SkewOps<16, 16, 32, 256, false>>(D, lu, lds); break;
      case 37: dev_lines<SkewOps<16, 16, 32, 256, true>>(D, lu, lds); break;
      case 38: dev_lines<NarrowOps<4, 256, 8>>(D, lu, lds); break;
      case 39: dev_lines<NarrowOps<8, 256, 6>>(D, lu, lds); break;
      case 40: dev_lines<NarrowOps<16, 256, 4>>(D, lu, lds); break;
      case 41: dev_lines<ShortOps<4, 256, 8>>(D, lu, lds); break;
      case 42: dev_lines<ShortOps<8, 256, 6>>(D, lu, lds); break;
      case 43: dev_lines<ShortOps<16, 256, 4>>(D, lu, lds); break;
      default: break;
    }
  } else {
    switch (D.variant) {
      case 12: dev_packed<4, 1>(D, lu, lds); break;
      case 13: dev_packed<4, 2>(D, lu, lds); break;
      case 14: dev_packed<4, 4>(D, lu, lds); break;
      case 15: dev_packed<4, 8>(D, lu, lds); break;
      case 16: dev_packed<8, 1>(D, lu, lds); break;
      case 17: dev_packed<8, 2>(D, lu, lds); break;
      case 18: dev_packed<8, 4>(D, lu, lds); break;
      case 19: dev_packed<8, 8>(D, lu, lds); break;
      case 20: dev_packed<16, 1>(D, lu, lds); break;
      case 21: dev_packed<16, 2>(D, lu, lds); break;
      case 22: dev_packed<16, 4>(D, lu, lds); break;
      default: break;
    }
  }
}

// One workgroup per unit of one family's `total` units of `nprob` descriptors.
// The dispatcher hands a unit to the next free slot: units differ (an edge
// tile, a short chunk, a long copy), and resident workgroups that walked a
// fixed share of them each finished far apart. It also needs fewer registers
// than a loop over units (48 to 68 VGPRs, no scratch; 58 to 85 with the loop),
// so 7 or 8 workgroups fit a CU where 5 or 6 did. On MI355X, 4096 problems of
// 13.8 GB 3335 -> 2981 us (2710 us with their kernels ranked by batch_cost), a
// burst of 128 served requests 775 -> 746 us (700 us). Bound by HBM; a copy of
// the bytes takes 2180 us. One kernel for all families (71 VGPRs, one launch
// instead of four) ran no faster: 2737 us and 688 us. Neither did units sorted
// by shape (3428 us against 3349 with the loop): problems of unlike kernels
// fill each other's waits.
template <int FAM>
__global__ __launch_bounds__(256) void k_batch(
    const BatchDesc* __restrict__ descs, const int* __restrict__ start, int nprob, int total) {
  __shared__ __attribute__((aligned(16))) unsigned char lds[kBatchLds];
  const int u = unit_at(blockIdx.x, blockIdx.y, gridDim.x, total);
  if (u < 0) return;
  const int lane = (int)(threadIdx.x & 63);
  const int p = batch_find(nprob, [&](int lo, int n, int step) {
    return __popcll(__ballot(starts_by(start, u, lo, n, step, lane)));
  });
  dev_unit<FAM>(descs[p], u - start[p], lds);
}

const void* batch_kernel(int fam) {
  switch (fam) {
    case kFamTiled: return reinterpret_cast<const void*>(&k_batch<kFamTiled>);
    case kFamTiledG: return reinterpret_cast<const void*>(&k_batch<kFamTiledG>);
    case kFamLines: return reinterpret_cast<const void*>(&k_batch<kFamLines>);
    default: return reinterpret_cast<const void*>(&k_batch<kFamPacked>);
  }
}

// ---------------------------------------------------------------------------
// Host replay: the same per-thread code, workgroup by workgroup.
// ---------------------------------------------------------------------------

template <int B, int TX, int TY, int VX, int VY, bool G = false>
void host_tiled(const BatchDesc& D, int lu, unsigned char* lds_raw) {
  using Ops = TiledOps<B, TX, TY, VX, VY, G>;
  using E = typename Ops::E;
  E* lds = reinterpret_cast<E*>(lds_raw);
  for (int w = lu; w < D.items; w += D.groups) {
    const TileCtx c = Ops::item(D.a.tiled, (uint32_t)w);
    for (int t = 0; t < 256; t++) Ops::prepare(D.a.tiled, c, t, lds);
    for (int t = 0; t < 256; t++) Ops::load(D.a.tiled, c, t, static_cast<const E*>(D.in), lds);
    for (int t = 0; t < 256; t++) Ops::store(D.a.tiled, c, t, static_cast<E*>(D.out), lds);
  }
}

template <class Ops>
void host_lines(const BatchDesc& D, int lu, unsigned char* lds_raw) {
  using E = typename Ops::E;
  E* lds = reinterpret_cast<E*>(lds_raw);
  const TiledArgs& a = D.a.tiled;
  E* out = static_cast<E*>(D.out);
  const int phase = line_phase(out);
  for (int w = lu; w < D.items; w += D.groups) {
    const TileCtx c = Ops::item(a, (uint32_t)w);
    if (Ops::early(a))
      for (int t = 0; t < Ops::NT; t++) Ops::prepare(a, c, t, lds);
    for (int t = 0; t < Ops::NT; t++) Ops::load(a, c, t, static_cast<const E*>(D.in), lds, phase);
    for (int t = 0; t < Ops::NT; t++) Ops::store(a, c, t, out, lds, phase);
  }
}

template <int B>
void host_copy(const BatchDesc& D, int lu) {
  using Ops = CopyOps<B>;
  using E = typename Ops::E;
  for (int w = lu; w < D.items; w += D.groups)
    for (int t = 0; t < Ops::NT; t++)
      Ops::run(D.a.copy, (uint32_t)w, t, static_cast<const E*>(D.in), static_cast<E*>(D.out));
}

template <int B, int NREG>
void host_packed(const BatchDesc& D, int lu, unsigned char* lds_raw) {
  using Ops = PackedOps<B, NREG>;
  using E = typename Ops::E;
  E* lds = reinterpret_cast<E*>(lds_raw);
  const PackedArgs& a = D.a.packed;
  const uint32_t og = fdiv((uint32_t)lu, D.split_div);
  const int split = lu - (int)(og * D.split_div.d);
  std::vector<typename Ops::Pre> pre(256);
  for (int t = 0; t < 256; t++) Ops::prepare(a, split, t, 256, pre[t]);
  for (int o = (int)og; o < a.vol_outer; o += D.groups) {
    int off_in, off_out;
    outer_offsets(a.outer, (uint32_t)o, off_in, off_out);
    for (int t = 0; t < 256; t++) Ops::load(pre[t], off_in, t, 256, static_cast<const E*>(D.in), lds);
    for (int t = 0; t < 256; t++) Ops::store(pre[t], off_out, t, 256, static_cast<E*>(D.out), lds);
  }
}

void host_unit(const BatchDesc& D, int lu, unsigned char* lds) {
  switch (D.variant) {
    case 0: host_tiled<4, 64, 64, 1, 1>(D, lu, lds); break;
    case 1: host_tiled<4, 64, 64, 4, 1>(D, lu, lds); break;
    case 2: host_tiled<4, 64, 64, 1, 4>(D, lu, lds); break;
    case 3: host_tiled<4, 64, 64, 4, 4>(D, lu, lds); break;
    case 4: host_tiled<8, 32, 32, 1, 1>(D, lu, lds); break;
    case 5: host_tiled<8, 32, 32, 2, 1>(D, lu, lds); break;
    case 6: host_tiled<8, 32, 32, 1, 2>(D, lu, lds); break;
    case 7: host_tiled<8, 32, 32, 2, 2>(D, lu, lds); break;
    case 8: host_tiled<16, 32, 32, 1, 1>(D, lu, lds); break;
    case 9: host_copy<4>(D, lu); break;
    case 10: host_copy<8>(D, lu); break;
    case 11: host_copy<16>(D, lu); break;
    case 12: host_packed<4, 1>(D, lu, lds); break;
    case 13: host_packed<4, 2>(D, lu, lds); break;
    case 14: host_packed<4, 4>(D, lu, lds); break;
    case 15: host_packed<4, 8>(D, lu, lds); break;
    case 16: host_packed<8, 1>(D, lu, lds); break;
    case 17: host_packed<8, 2>(D, lu, lds); break;
    case 18: host_packed<8, 4>(D, lu, lds); break;
    case 19: host_packed<8, 8>(D, lu, lds); break;
    case 20: host_packed<16, 1>(D, lu, lds); break;
    case 21: host_packed<16, 2>(D, lu, lds); break;
    case 22: host_packed<16, 4>(D, lu, lds); break;
    case 23: host_tiled<4, 64, 64, 1, 1, true>(D, lu, lds); break;
    case 24: host_tiled<4, 64, 64, 4, 1, true>(D, lu, lds); break;
    case 25: host_tiled<4, 64, 64, 1, 4, true>(D, lu, lds); break;
    case 26: host_tiled<4, 64, 64, 4, 4, true>(D, lu, lds); break;
    case 27: host_tiled<8, 32, 32, 1, 1, true>(D, lu, lds); break;
    case 28: host_tiled<8, 32, 32, 2, 1, true>(D, lu, lds); break;
    case 29: host_tiled<8, 32, 32, 1, 2, true>(D, lu, lds); break;
    case 30: host_tiled<8, 32, 32, 2, 2, true>(D, lu, lds); break;
    case 31: host_tiled<16, 32, 32, 1, 1, true>(D, lu, lds); break;
    case 32: host_lines<SkewOps<4, 32, 64, 256, false>>(D, lu, lds); break;
    case 33: host_lines<SkewOps<4, 32, 64, 256, true>>(D, lu, lds); break;
    case 34: host_lines<SkewOps<8, 32, 32, 256, false>>(D, lu, lds); break;
    case 35: host_lines<SkewOps<8, 32, 32, 256, true>>(D, lu, lds); break;
    case 36: host_lines<SkewOps<16, 16, 32, 256, false>>(D, lu, lds); break;
    case 37: host_lines<SkewOps<16, 16, 32, 256, true>>(D, lu, lds); break;
    case 38: host_lines<NarrowOps<4, 256, 8>>(D, lu, lds); break;
    case 39: host_lines<NarrowOps<8, 256, 6>>(D, lu, lds); break;
    case 40: host_lines<NarrowOps<16, 256, 4>>(D, lu, lds); break;
    case 41: host_lines<ShortOps<4, 256, 8>>(D, lu, lds); break;
    case 42: host_lines<ShortOps<8, 256, 6>>(D, lu, lds); break;
    case 43: host_lines<ShortOps<16, 256, 4>>(D, lu, lds); break;
    default: break;
  }
}

}  // namespace

bool batch_tiled_available(int elem, int tx, int ty, int vx, int vy, bool general) {
  for (const auto& s : kBatchShapes)
    if (s.method == kTiled && s.form == kTileRect && s.b == elem && s.p1 == tx && s.p2 == ty && s.p3 == vx &&
        s.p4 == vy && (s.g != 0) == general)
      return true;
  return false;
}

bool batch_skew_available(int elem, int tx, int ty) {
  for (const auto& s : kBatchShapes)
    if (s.form == kTileSkew && s.b == elem && s.p1 == tx && s.p2 == ty) return true;
  return false;
}

namespace {
// Bit nreg of the entry for elem / 4 (elements of 4, 8 and 16 bytes): the
// planner asks for every split it tries, so the table is indexed once.
struct PackedShapeBits {
  unsigned bits[5] = {0, 0, 0, 0, 0};
  PackedShapeBits() {
    for (const auto& s : kBatchShapes)
      if (s.method == kPacked && (s.b == 4 || s.b == 8 || s.b == 16) && s.p1 >= 0 && s.p1 < 32)
        bits[s.b / 4] |= 1u << s.p1;
  }
};
}  // namespace

bool batch_packed_available(int elem, int nreg) {
  static const PackedShapeBits t;
  if ((elem != 4 && elem != 8 && elem != 16) || nreg < 0 || nreg >= 32) return false;
  return (t.bits[elem / 4] >> nreg) & 1u;
}

int batch_variant(const Candidate& c) {
  for (const auto& s : kBatchShapes) {
    switch (c.method) {
      case kTiled:
        if (s.method == kTiled && s.b == c.elem && s.form == c.tiled.form &&
            (s.form >= kTileNarrow || (s.p1 == c.tile_x && s.p2 == c.tile_y && s.p3 == c.vec_x && s.p4 == c.vec_y &&
                                       (s.g != 0) == (c.xgroup > 1 || c.ygroup > 1))))
          return s.id;
        break;
      case kTiledCopy:
        if (s.method == kTiledCopy && s.b == c.elem) return s.id;
        break;
      case kPacked:
      case kPackedSplit:
        if (s.method == kPacked && s.b == c.elem && s.p1 == c.nreg && c.block == 256) return s.id;
        break;
      default:
        break;
    }
  }
  return -1;
}

bool batch_describe(const Candidate& c, BatchDesc& d) {
  d = BatchDesc();
  d.variant = batch_variant(c);
  if (d.variant < 0) return false;
  if (c.lds_bytes > kBatchLds) return false;
  d.split_div = make_fastdiv(1);
  switch (c.method) {
    case kTiled:
      d.a.tiled = c.tiled;
      d.items = c.tiled.items;
      d.item_bytes = 2 * c.elem * (c.tiled.form == kTileShort ? c.tile_x : c.tile_x * c.tile_y);
      break;
    case kTiledCopy:
      d.a.copy = c.copy;
      d.items = c.copy.items;
      d.item_bytes = 2 * c.copy.per * c.elem;
      break;
    default:
      d.a.packed = c.packed;
      d.items = c.packed.vol_outer;
      d.split_div = make_fastdiv((uint32_t)c.packed.num_split);
      d.item_bytes = std::max(1, 2 * std::max(1, c.packed.shape[0].vol) * c.elem / std::max(1, c.packed.num_split));
      break;
  }
  if (d.items <= 0) return false;
  batch_regroup(d, kBatchUnitBytes);
  return d.units > 0;
}

void batch_regroup(BatchDesc& d, long long unit_bytes) {
  const long long r = std::max<long long>(1, std::min<long long>(d.items, unit_bytes / std::max(1, d.item_bytes)));
  d.rounds = (int)r;
  d.groups = (int)((d.items + r - 1) / r);
  d.units = d.groups * (int)d.split_div.d;
}

long long batch_unit_bytes(long long total_bytes, int grid) {
  // LIBRETT_BATCH_UNIT_KB fixes the unit size; LIBRETT_BATCH_UNITS_PER_WG
  // sets the units for each workgroup that the device holds at a time (default 32).
  static const long long fixed = [] {
    const char* e = std::getenv("LIBRETT_BATCH_UNIT_KB");
    return e ? std::max(1LL, std::atoll(e)) << 10 : 0LL;
  }();
  static const long long per_wg = [] {
    const char* e = std::getenv("LIBRETT_BATCH_UNITS_PER_WG");
    return e ? std::max(1LL, std::atoll(e)) : 32LL;
  }();
  if (fixed) return fixed;
  const long long per = total_bytes / (per_wg * std::max(1, grid));
  return std::max<long long>(16 << 10, std::min<long long>(kBatchUnitBytes, per));
}

int batch_family(int variant) {
  return variant <= 8 ? kFamTiled : variant <= 11 ? kFamLines : variant <= 22 ? kFamPacked : variant <= 31 ? kFamTiledG : kFamLines;
}

hipError_t launch_batch(int fam, const BatchDesc* d_descs, const int* d_start, int nprob, int total,
                        hipStream_t stream) {
  if (total <= 0 || nprob <= 0) return hipSuccess;
  const int gx = std::min(total, kBatchGridRow);
  void* args[4] = {&d_descs, &d_start, &nprob, &total};
  return hipLaunchKernel(batch_kernel(fam), dim3(gx, (total - 1) / gx + 1), dim3(256), args, 0, stream);
}

int batch_occupancy(int fam) {
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, batch_kernel(fam), 256, 0) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return n;
}

void batch_layout(std::vector<BatchDesc>& descs, BatchLayout& L, std::vector<int>* order) {
  const int nd = (int)descs.size();
  std::vector<int> idx(nd);
  for (int k = 0; k < nd; k++) idx[k] = k;
  std::stable_sort(idx.begin(), idx.end(), [&](int a, int b) {
    return batch_family(descs[a].variant) < batch_family(descs[b].variant);
  });
  std::vector<BatchDesc> sorted(nd);
  for (int k = 0; k < nd; k++) sorted[k] = descs[idx[k]];
  descs.swap(sorted);
  if (order) *order = idx;
  L.start.assign(nd + kBatchFamilies, 0);
  int k = 0, off = 0;
  for (int f = 0; f < kBatchFamilies; f++) {
    L.first[f] = k;
    L.start_off[f] = off;
    long long tot = 0;
    int n = 0;
    while (k < nd && batch_family(descs[k].variant) == f) {
      L.start[off + n] = (int)std::min<long long>(tot, 0x7fffffff);
      tot += descs[k].units;
      n++;
      k++;
    }
    L.start[off + n] = (int)std::min<long long>(tot, 0x7fffffff);
    L.n[f] = n;
    L.total[f] = tot;
    off += n + 1;
  }
}

hipError_t launch_batch_all(const BatchDesc* d_descs, const int* d_start, const BatchLayout& L,
                            hipStream_t stream) {
  for (int f = 0; f < kBatchFamilies; f++) {
    if (L.n[f] == 0) continue;
    const hipError_t e =
        launch_batch(f, d_descs + L.first[f], d_start + L.start_off[f], L.n[f], (int)L.total[f], stream);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

bool replay_batch_all(const BatchDesc* descs, const BatchLayout& L, int row) {
  for (int f = 0; f < kBatchFamilies; f++) {
    if (L.n[f] == 0) continue;
    if (!replay_batch(descs + L.first[f], L.start.data() + L.start_off[f], L.n[f], (int)L.total[f], row))
      return false;
  }
  return true;
}

bool replay_batch(const BatchDesc* descs, const int* start, int nprob, int total, int row) {
  // The workgroup's LDS, followed by a guard band that no unit may touch.
  const size_t guard = 64 << 10;
  std::vector<unsigned char> lds(kBatchLds + guard, 0xC3);
  const int gx = std::min(total, row > 0 ? row : kBatchGridRow);
  for (int by = 0; gx > 0 && by < (total - 1) / gx + 1; by++)
    for (int bx = 0; bx < gx; bx++) {
      const int u = unit_at((uint32_t)bx, (uint32_t)by, (uint32_t)gx, total);
      if (u < 0) continue;
      const int p = batch_find(nprob, [&](int lo, int n, int step) {
        int hits = 0;
        for (int lane = 0; lane < 64; lane++) hits += starts_by(start, u, lo, n, step, lane);
        return hits;
      });
      host_unit(descs[p], u - start[p], lds.data());
    }
  for (size_t i = kBatchLds; i < lds.size(); i++)
    if (lds[i] != 0xC3) return false;
  return true;
}

}  // namespace lrt
