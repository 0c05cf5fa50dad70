// Batched engine: host side (planning, autotuning, descriptor arena, HIP
// graph) and its C-ABI entry points (librett_c.h). The reference has no
// batched mode; its per-call path is librettExecute (src/librett.cpp:372-385),
// which is the baseline this engine is measured against.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "devmem.h"
#include "../../include/librett_c.h"
#include "batch.h"
#include "kernels.h"
#include "lru_cache.h"
#include "planner.h"

namespace lrt {
namespace {

// Internal failures name their cause on stderr when LIBRETT_DEBUG is set.
int fail(const char* why, int code = LIBRETT_C_INTERNAL_ERROR) {
  static const bool on = std::getenv("LIBRETT_DEBUG") != nullptr;
  if (on) std::fprintf(stderr, "librett batch: %s\n", why);
  return code;
}

double now_s() {
  return std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
}

int check_problem(int rank, const int* dim, const int* perm, size_t elem) {
  if (elem != 4 && elem != 8 && elem != 16) return LIBRETT_C_INVALID_PARAMETER;
  if (rank < 1 || !dim || !perm) return LIBRETT_C_INVALID_PARAMETER;
  long long vol = 1;
  std::vector<char> seen(rank, 0);
  for (int i = 0; i < rank; i++) {
    if (dim[i] < 1) return LIBRETT_C_INVALID_PARAMETER;
    vol *= dim[i];
    if (vol >= (1LL << 31)) return LIBRETT_C_INVALID_PARAMETER;
    if (perm[i] < 0 || perm[i] >= rank || seen[perm[i]]++) return LIBRETT_C_INVALID_PARAMETER;
  }
  return LIBRETT_C_SUCCESS;
}

// A problem that reduces to a plain copy (the reference's Trivial method) as
// a TiledCopy candidate of one row.
Candidate flat_copy(const Problem& p) {
  Candidate c;
  c.method = kTiledCopy;
  c.elem = p.elem;
  c.word = 16;
  CopyArgs& a = c.copy;
  a.n = a.X = (int)p.vol;
  a.row_div = make_fastdiv((uint32_t)p.vol);
  a.per = 256 * (16 / p.elem);
  a.items = (int)((p.vol + 128 / p.elem - 1 + a.per - 1) / a.per);
  a.xcds = 1;
  a.stream_in = 0;
  a.rows.n = 0;
  for (int r = 0; r < kMaxRank; r++) {
    a.rows.div[r] = make_fastdiv(1);
    a.rows.ct_in[r] = a.rows.ct_out[r] = 0;
  }
  return c;
}

struct BatchObj {
  int device = 0;
  hipStream_t stream = nullptr;
  int nprob = 0;
  std::vector<Problem> probs;
  std::vector<Candidate> chosen;
  // Descriptors, one per problem, in family order.
  std::vector<BatchDesc> descs, fallback;
  std::vector<int> owner;               // problem of each descriptor
  BatchLayout layout;                   // descriptors grouped by kernel family
  long long total = 0;                  // units of all families
  int grid_max = 0;  // workgroups resident at a time, of the family that holds most
  long long unit_bytes = kBatchUnitBytes;
  BatchDesc* d_descs = nullptr;
  int* d_start = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  bool buffers_set = false;
  double plan_s = 0, tune_s = 0;
  int tuned = 0;

  ~BatchObj() {
    if (exec) (void)hipGraphExecDestroy(exec);
    if (graph) (void)hipGraphDestroy(graph);
    if (d_descs) (void)dev_free(d_descs);
    if (d_start) (void)dev_free(d_start);
  }
};

std::mutex g_batch_mu;
std::unordered_map<unsigned int, std::shared_ptr<BatchObj>> g_batches;
std::atomic<unsigned int> g_next_batch{1};

struct TuneValue {
  Candidate cand;
  double seconds;
};
LruCache<std::string, TuneValue> g_tune_cache(1 << 16);

std::string problem_key(const Problem& p) {
  std::string k = std::to_string(p.elem) + ":";
  for (int i = 0; i < p.rank; i++) k += std::to_string(p.dim[i]) + ",";
  k += "/";
  for (int i = 0; i < p.rank; i++) k += std::to_string(p.perm[i]) + ",";
  return k;
}


// Times candidate c of problem p inside its family's kernel, on enough
// clones of the problem to fill the device (scratch buffers `a`, `b`).
double time_in_batch(const Candidate& c, const Problem& p, void* a, void* b, size_t scratch, hipStream_t stream,
                     BatchDesc* d_desc, int* d_start, int max_clones, long long unit_bytes) {
  BatchDesc d;
  if (!batch_describe(c, d)) return -1;
  batch_regroup(d, unit_bytes);
  const int fam = batch_family(d.variant);
  const size_t bytes = (size_t)p.vol * p.elem;
  const size_t span = (bytes + 255) / 256 * 256;
  if (span > scratch) return -1;  // every clone must lie inside the scratch buffers
  int clones = (int)std::min<size_t>(max_clones, std::max<size_t>(1, scratch / span));
  clones = std::max(1, std::min(clones, (int)((64ull << 20) / std::max<size_t>(1, bytes)) + 1));
  std::vector<BatchDesc> ds(clones, d);
  std::vector<int> st(clones + 1);
  for (int k = 0; k < clones; k++) {
    ds[k].in = (const char*)a + k * span;
    ds[k].out = (char*)b + k * span;
    st[k] = k * d.units;
  }
  st[clones] = clones * d.units;
  if (hipMemcpyAsync(d_desc, ds.data(), clones * sizeof(BatchDesc), hipMemcpyHostToDevice, stream) != hipSuccess)
    return -1;
  if (hipMemcpyAsync(d_start, st.data(), (clones + 1) * sizeof(int), hipMemcpyHostToDevice, stream) != hipSuccess)
    return -1;
  hipEvent_t e0, e1;
  if (hipEventCreate(&e0) != hipSuccess) return -1;
  if (hipEventCreate(&e1) != hipSuccess) {
    (void)hipEventDestroy(e0);
    return -1;
  }
  bool ok = launch_batch(fam, d_desc, d_start, clones, st[clones], stream) == hipSuccess;
  float best = 1e30f;
  for (int r = 0; ok && r < 2; r++) {
    ok = hipEventRecord(e0, stream) == hipSuccess &&
         launch_batch(fam, d_desc, d_start, clones, st[clones], stream) == hipSuccess &&
         hipEventRecord(e1, stream) == hipSuccess && hipEventSynchronize(e1) == hipSuccess;
    float ms = 0;
    if (ok && hipEventElapsedTime(&ms, e0, e1) == hipSuccess) best = std::min(best, ms);
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (!ok) {
    (void)hipGetLastError();
    return -1;
  }
  return best * 1e-3 / clones;
}

int build_batch(BatchObj& B, const DeviceInfo& dev, int tune) {
  const double t0 = now_s();
  DeviceInfo bdev = dev;
  bdev.batch_mode = 1;
  B.chosen.resize(B.nprob);
  std::vector<std::vector<Candidate>> ranked(B.nprob);
  for (int i = 0; i < B.nprob; i++) {
    ranked[i] = batch_candidates(B.probs[i], bdev);
    if (ranked[i].empty()) return fail("no batch-mode candidate");
    B.chosen[i] = ranked[i][0];
  }
  B.plan_s = now_s() - t0;

  B.grid_max = 0;
  for (int f = 0; f < kBatchFamilies; f++) {
    const int occ = std::max(1, dev.has_gpu ? batch_occupancy(f) : 4);
    B.grid_max = std::max(B.grid_max, dev.cu_count * occ);
  }
  long long total_bytes = 0;
  for (const Problem& p : B.probs) total_bytes += 2LL * p.vol * p.elem;
  B.unit_bytes = batch_unit_bytes(total_bytes, B.grid_max);

  if (tune && dev.has_gpu) {
    // Autotuner: time the top candidates of each distinct problem inside their
    // family's kernel on clones of the problem, keep the fastest, and
    // remember it across batches.
    const double t1 = now_s();
    // Scratch for the clones: at least 256 MiB, and room for the largest
    // problem up to 4 GiB (larger problems keep the model's choice).
    size_t largest = 0;
    for (const Problem& p : B.probs) largest = std::max(largest, ((size_t)p.vol * p.elem + 255) / 256 * 256);
    const size_t scratch = std::max<size_t>(256ull << 20, std::min<size_t>(largest, 4ull << 30));
    void *a = nullptr, *b = nullptr;
    BatchDesc* d_desc = nullptr;
    int* d_start = nullptr;
    const int max_clones = 4096;
    bool ok = dev_malloc(&a, scratch) == hipSuccess && dev_malloc(&b, scratch) == hipSuccess &&
              dev_malloc((void**)&d_desc, max_clones * sizeof(BatchDesc)) == hipSuccess &&
              dev_malloc((void**)&d_start, (max_clones + 1) * sizeof(int)) == hipSuccess;
    if (ok) ok = hipMemsetAsync(a, 0, scratch, B.stream) == hipSuccess;
    const int topk = std::max(1, std::min(8, tune));
    for (int i = 0; ok && i < B.nprob; i++) {
      if (B.chosen[i].method == kTrivial) continue;
      const std::string key = problem_key(B.probs[i]);
      TuneValue tv;
      if (g_tune_cache.get(key, tv)) {
        B.chosen[i] = tv.cand;
        continue;
      }
      double best = 1e30;
      int bi = 0;
      for (int k = 0; k < (int)ranked[i].size() && k < topk; k++) {
        const double t = time_in_batch(ranked[i][k], B.probs[i], a, b, scratch, B.stream, d_desc, d_start,
                                       max_clones, B.unit_bytes);
        if (t > 0 && t < best) {
          best = t;
          bi = k;
        }
      }
      B.chosen[i] = ranked[i][bi];
      B.tuned++;
      g_tune_cache.put(key, TuneValue{B.chosen[i], best});
    }
    (void)hipStreamSynchronize(B.stream);
    if (a) (void)dev_free(a);
    if (b) (void)dev_free(b);
    if (d_desc) (void)dev_free(d_desc);
    if (d_start) (void)dev_free(d_start);
    if (!ok) return fail("autotuner HIP call failed");
    B.tune_s = now_s() - t1;
  }

  // Descriptors and the unit index space.
  B.descs.clear();
  B.fallback.clear();
  for (int i = 0; i < B.nprob; i++) {
    BatchDesc d, f;
    if (!describe_problem(B.probs[i], B.chosen[i], d, f)) return fail("no descriptor for the chosen plan");
    batch_regroup(d, B.unit_bytes);
    batch_regroup(f, B.unit_bytes);
    B.descs.push_back(d);
    B.fallback.push_back(f);
  }
  // Group by kernel family; the fallback descriptors follow the same order (a
  // fallback keeps its descriptor's family).
  batch_layout(B.descs, B.layout, &B.owner);
  std::vector<BatchDesc> fb(B.owner.size());
  for (size_t k = 0; k < B.owner.size(); k++) fb[k] = B.fallback[B.owner[k]];
  B.fallback.swap(fb);
  B.total = 0;
  for (int f = 0; f < kBatchFamilies; f++) {
    if (B.layout.total[f] >= (1LL << 31)) return LIBRETT_C_INVALID_PARAMETER;
    B.total += B.layout.total[f];
  }
  return LIBRETT_C_SUCCESS;
}

std::shared_ptr<BatchObj> find_batch(unsigned int h) {
  std::lock_guard<std::mutex> lock(g_batch_mu);
  auto it = g_batches.find(h);
  return it == g_batches.end() ? nullptr : it->second;
}

bool device_info_batch(DeviceInfo& d) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, dev) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  d.device_id = dev;
  d.cu_count = prop.multiProcessorCount;
  d.lds_per_block = (int)prop.sharedMemPerBlock;
  d.lds_per_cu = (int)std::max<size_t>(prop.sharedMemPerBlock, prop.maxSharedMemoryPerMultiProcessor);
  d.max_threads_per_block = prop.maxThreadsPerBlock;
  d.warp_size = prop.warpSize;
  d.max_waves_per_cu = std::max(1, prop.maxThreadsPerMultiProcessor / std::max(1, prop.warpSize));
  if (prop.l2CacheSize > 0) d.l2_bytes = (double)prop.l2CacheSize * std::max(1, d.cu_count / 32);
  d.has_gpu = 1;
  return true;
}

int read_problems(int count, const int* ranks, const int* dims, const int* perms, const size_t* elems,
                  std::vector<Problem>& out) {
  if (count < 1 || !ranks || !dims || !perms || !elems) return LIBRETT_C_INVALID_PARAMETER;
  out.clear();
  long long off = 0;
  for (int i = 0; i < count; i++) {
    const int r = check_problem(ranks[i], dims + off, perms + off, elems[i]);
    if (r != LIBRETT_C_SUCCESS) return r;
    out.push_back(canonicalize(ranks[i], dims + off, perms + off, (int)elems[i]));
    off += ranks[i];
  }
  return LIBRETT_C_SUCCESS;
}

}  // namespace

// Modelled device time of a candidate in a batch, microseconds. Workgroups of
// other problems fill the chip, so a kernel is bound by its memory lines
// (t_stream) or, where tiles are mostly empty or chunks small, by the time
// its items take however little they move: barriers, address decoding, the
// wait for the first line. Both sides are measured, every candidate of 2200
// random problems on enough clones to fill the device: ns is the mean time
// between finished items, and `lines` corrects t_stream. Against ranking by
// t_stream alone, the sum of the chosen kernels' times fell from 1.13 to 1.02
// of that of the best ones (f64 and c128 of up to 1e6 elements) and from
// 1.25 to 1.02 (all types up to 64 MiB). Example: [4,41,10,40,18] to
// (1,4,0,3,2) f64 as 4800 tiles an eighth full 20.7 us, as chunks 4.7 us.
static double batch_cost(const Candidate& c) {
  const int e = c.elem == 4 ? 0 : c.elem == 8 ? 1 : 2;
  double lines = 1.0, ns = 2.0;
  if (c.method == kPacked || c.method == kPackedSplit) {
    static const double t[3][4] = {{0.5, 1.0, 2.0, 4.0}, {1.1, 1.4, 3.1, 11.0}, {1.2, 1.9, 6.2, 12.0}};
    ns = t[e][c.nreg <= 1 ? 0 : c.nreg <= 2 ? 1 : c.nreg <= 4 ? 2 : 3];
  } else if (c.method == kTiled) {
    const bool general = c.xgroup > 1 || c.ygroup > 1;
    static const double rect[2][3] = {{2.5, 2.0, 3.0}, {2.0, 3.0, 3.4}};
    static const double skew[2][3] = {{2.1, 1.9, 2.5}, {3.0, 2.5, 3.0}};
    if (c.tiled.form == kTileRect) {
      lines = general ? 1.0 : 1.07;
      ns = rect[general][e];
    } else if (c.tiled.form == kTileSkew) {
      lines = general ? 0.8 : 0.86;
      ns = skew[general][e];
    } else {
      lines = 0.7;
      ns = e == 1 ? 2.7 : 2.0;
    }
  }
  return std::max(lines * c.model.t_stream * 1e6, ns * 1e-3 * c.model.items);
}

std::vector<Candidate> batch_candidates(const Problem& p, const DeviceInfo& dev) {
  DeviceInfo bdev = dev;
  bdev.batch_mode = 1;
  std::vector<Candidate> cands = make_candidates(p, bdev);
  std::vector<Candidate> ok;
  for (auto& c : cands)
    if (c.method == kTrivial || (batch_variant(c) >= 0 && !copy_beats(cands, c))) ok.push_back(c);
  std::stable_sort(ok.begin(), ok.end(), [](const Candidate& a, const Candidate& b) {
    return batch_cost(a) < batch_cost(b);
  });
  return ok;
}

int batch_alignment(const Problem& p, const Candidate& c) {
  return c.method == kTrivial ? p.elem : needed_alignment(c);
}

bool describe_problem(const Problem& p, const Candidate& c, BatchDesc& desc, BatchDesc& fallback) {
  if (!batch_describe(c.method == kTrivial ? flat_copy(p) : c, desc)) return false;
  if (batch_alignment(p, c) == p.elem || !batch_describe(unaligned_fallback(c), fallback)) fallback = desc;
  return true;
}

}  // namespace lrt

using namespace lrt;

extern "C" {

int librett_c_batch_plan(unsigned int* handle, int count, const int* ranks, const int* dims, const int* perms,
                         const size_t* elems, void* stream, int tune) {
  if (!handle) return LIBRETT_C_INVALID_PARAMETER;
  try {
    auto B = std::make_shared<BatchObj>();
    int r = read_problems(count, ranks, dims, perms, elems, B->probs);
    if (r != LIBRETT_C_SUCCESS) return r;
    B->nprob = count;
    B->stream = (hipStream_t)stream;
    DeviceInfo dev;
    if (!device_info_batch(dev)) return fail("device query failed");
    B->device = dev.device_id;
    r = build_batch(*B, dev, tune);
    if (r != LIBRETT_C_SUCCESS) return r;
    const size_t nd = B->descs.size();
    if (dev_malloc((void**)&B->d_descs, nd * sizeof(BatchDesc)) != hipSuccess ||
        dev_malloc((void**)&B->d_start, B->layout.start.size() * sizeof(int)) != hipSuccess) {
      (void)hipGetLastError();
      return fail("descriptor allocation failed");
    }
    if (hipMemcpy(B->d_start, B->layout.start.data(), B->layout.start.size() * sizeof(int), hipMemcpyHostToDevice) !=
        hipSuccess)
      return fail("descriptor upload failed");
    const unsigned int h = g_next_batch.fetch_add(1);
    {
      std::lock_guard<std::mutex> lock(g_batch_mu);
      g_batches[h] = B;
    }
    *handle = h;
    return LIBRETT_C_SUCCESS;
  } catch (const std::exception& e) {
    return fail(e.what());
  } catch (...) {
    return fail("unknown exception");
  }
}

int librett_c_batch_set_buffers(unsigned int handle, const void* const* idata, void* const* odata) {
  auto B = find_batch(handle);
  if (!B) return LIBRETT_C_INVALID_PLAN;
  if (!idata || !odata) return LIBRETT_C_INVALID_PARAMETER;
  std::vector<BatchDesc> up(B->descs.size());
  for (size_t k = 0; k < B->descs.size(); k++) {
    const int i = B->owner[k];
    if (!idata[i] || !odata[i] || idata[i] == odata[i]) return LIBRETT_C_INVALID_PARAMETER;
    const int align = batch_alignment(B->probs[i], B->chosen[i]);
    const bool mis = (((uintptr_t)idata[i] | (uintptr_t)odata[i]) & (uintptr_t)(align - 1)) != 0;
    up[k] = mis ? B->fallback[k] : B->descs[k];
    up[k].in = idata[i];
    up[k].out = odata[i];
  }
  // A fallback descriptor may have another unit count: rebuild the index
  // space and re-capture the graph when it changes. The descriptors are
  // already in family order, and a fallback keeps its family, so the
  // layout keeps that order.
  BatchLayout L;
  std::vector<BatchDesc> tmp = up;
  batch_layout(tmp, L, nullptr);
  long long total = 0;
  for (int f = 0; f < kBatchFamilies; f++) {
    if (L.total[f] >= (1LL << 31)) return LIBRETT_C_INVALID_PARAMETER;
    total += L.total[f];
  }
  if (L.start != B->layout.start) {
    B->layout = L;
    B->total = total;
    if (hipMemcpyAsync(B->d_start, L.start.data(), L.start.size() * sizeof(int), hipMemcpyHostToDevice,
                       B->stream) != hipSuccess)
      return LIBRETT_C_INTERNAL_ERROR;
    if (B->exec) {
      (void)hipGraphExecDestroy(B->exec);
      B->exec = nullptr;
    }
    if (B->graph) {
      (void)hipGraphDestroy(B->graph);
      B->graph = nullptr;
    }
  }
  if (hipMemcpyAsync(B->d_descs, up.data(), up.size() * sizeof(BatchDesc), hipMemcpyHostToDevice, B->stream) !=
          hipSuccess ||
      hipStreamSynchronize(B->stream) != hipSuccess) {
    (void)hipGetLastError();
    return LIBRETT_C_INTERNAL_ERROR;
  }
  B->buffers_set = true;
  return LIBRETT_C_SUCCESS;
}

int librett_c_batch_execute(unsigned int handle, int use_graph) {
  auto B = find_batch(handle);
  if (!B) return LIBRETT_C_INVALID_PLAN;
  if (!B->buffers_set) return LIBRETT_C_INVALID_PARAMETER;
  if (!use_graph) {
    return launch_batch_all(B->d_descs, B->d_start, B->layout, B->stream) == hipSuccess
               ? LIBRETT_C_SUCCESS
               : LIBRETT_C_INTERNAL_ERROR;
  }
  if (!B->exec) {
    if (hipStreamBeginCapture(B->stream, hipStreamCaptureModeThreadLocal) != hipSuccess) {
      (void)hipGetLastError();
      return LIBRETT_C_INTERNAL_ERROR;
    }
    const hipError_t le = launch_batch_all(B->d_descs, B->d_start, B->layout, B->stream);
    hipGraph_t g = nullptr;
    const hipError_t ce = hipStreamEndCapture(B->stream, &g);
    if (le != hipSuccess || ce != hipSuccess || !g) {
      (void)hipGetLastError();
      if (g) (void)hipGraphDestroy(g);
      return LIBRETT_C_INTERNAL_ERROR;
    }
    hipGraphExec_t ex = nullptr;
    if (hipGraphInstantiate(&ex, g, nullptr, nullptr, 0) != hipSuccess) {
      (void)hipGetLastError();
      (void)hipGraphDestroy(g);
      return LIBRETT_C_INTERNAL_ERROR;
    }
    B->graph = g;
    B->exec = ex;
  }
  return hipGraphLaunch(B->exec, B->stream) == hipSuccess ? LIBRETT_C_SUCCESS : LIBRETT_C_INTERNAL_ERROR;
}

int librett_c_batch_destroy(unsigned int handle) {
  std::lock_guard<std::mutex> lock(g_batch_mu);
  auto it = g_batches.find(handle);
  if (it == g_batches.end()) return LIBRETT_C_INVALID_PLAN;
  g_batches.erase(it);
  return LIBRETT_C_SUCCESS;
}

int librett_c_batch_info_get(unsigned int handle, librett_c_batch_info* info) {
  auto B = find_batch(handle);
  if (!B) return LIBRETT_C_INVALID_PLAN;
  if (!info) return LIBRETT_C_INVALID_PARAMETER;
  std::memset(info, 0, sizeof(*info));
  info->count = B->nprob;
  info->descriptors = (int)B->descs.size();
  info->total_units = (int)std::min<long long>(B->total, 0x7fffffff);
  info->grid = B->grid_max;
  info->tuned = B->tuned;
  info->plan_seconds = B->plan_s;
  info->tune_seconds = B->tune_s;
  for (const auto& c : B->chosen)
    if (c.method >= 0 && c.method < 6) info->method_count[c.method]++;
  for (int i = 0; i < B->nprob; i++) info->bytes += B->chosen[i].bytes;
  return LIBRETT_C_SUCCESS;
}

int librett_c_batch_host_replay(int count, const int* ranks, const int* dims, const int* perms, const size_t* elems,
                                const librett_c_device* d, const void* const* idata, void* const* odata, int grid) {
  try {
    BatchObj B;
    int r = read_problems(count, ranks, dims, perms, elems, B.probs);
    if (r != LIBRETT_C_SUCCESS) return r;
    B.nprob = count;
    DeviceInfo dev;
    if (d) {
      dev.cu_count = d->cu_count;
      dev.lds_per_block = d->lds_per_block;
      dev.lds_per_cu = d->lds_per_cu;
      dev.max_threads_per_block = d->max_threads_per_block;
      dev.max_waves_per_cu = d->max_waves_per_cu;
      dev.hbm_bytes_per_s = d->hbm_bytes_per_s;
    }
    dev.has_gpu = 0;
    r = build_batch(B, dev, 0);
    if (r != LIBRETT_C_SUCCESS) return r;
    // Every problem runs between guard bands; a stray store changes a
    // guard, a stray load brings guard bytes into an output.
    const size_t g = 4096;
    std::vector<std::vector<unsigned char>> gin(count), gout(count);
    for (int i = 0; i < count; i++) {
      const size_t n = (size_t)B.probs[i].vol * B.probs[i].elem;
      gin[i].assign(n + 2 * g, 0xA5);
      gout[i].assign(n + 2 * g, 0x5A);
      std::memcpy(gin[i].data() + g, idata[i], n);
    }
    std::vector<BatchDesc> ds = B.descs;
    for (size_t k = 0; k < ds.size(); k++) {
      const int i = B.owner[k];
      ds[k].in = gin[i].data() + g;
      ds[k].out = gout[i].data() + g;
    }
    if (!replay_batch_all(ds.data(), B.layout, grid)) return LIBRETT_C_UNDEFINED_ERROR;
    for (int i = 0; i < count; i++) {
      const size_t n = (size_t)B.probs[i].vol * B.probs[i].elem;
      for (size_t j = 0; j < g; j++)
        if (gout[i][j] != 0x5A || gout[i][g + n + j] != 0x5A) return LIBRETT_C_UNDEFINED_ERROR;
      std::memcpy(odata[i], gout[i].data() + g, n);
    }
    return LIBRETT_C_SUCCESS;
  } catch (...) {
    return LIBRETT_C_INTERNAL_ERROR;
  }
}

int librett_c_batch_host_candidate(int rank, const int* dim, const int* permutation, size_t sizeofType,
                                   const librett_c_device* d, int index, int fallback, long long unit_bytes,
                                   int grid, const void* idata, void* odata, int* count) {
  try {
    std::vector<Problem> probs;
    const size_t elems[1] = {sizeofType};
    int r = read_problems(1, &rank, dim, permutation, elems, probs);
    if (r != LIBRETT_C_SUCCESS) return r;
    DeviceInfo dev;
    if (d) {
      dev.cu_count = d->cu_count;
      dev.lds_per_block = d->lds_per_block;
      dev.lds_per_cu = d->lds_per_cu;
      dev.max_threads_per_block = d->max_threads_per_block;
      dev.max_waves_per_cu = d->max_waves_per_cu;
      dev.hbm_bytes_per_s = d->hbm_bytes_per_s;
    }
    dev.has_gpu = 0;
    const Problem& p = probs[0];
    const std::vector<Candidate> ranked = batch_candidates(p, dev);
    if (count) *count = (int)ranked.size();
    if (!idata && !odata) return LIBRETT_C_SUCCESS;
    if (!idata || !odata || index < 0 || index >= (int)ranked.size()) return LIBRETT_C_INVALID_PARAMETER;
    BatchDesc d0, f0;
    if (!describe_problem(p, ranked[index], d0, f0)) return LIBRETT_C_INTERNAL_ERROR;
    BatchDesc& run = fallback ? f0 : d0;
    const long long ub = unit_bytes > 0 ? unit_bytes : kBatchUnitBytes;
    const size_t n = (size_t)p.vol * p.elem;
    const int align = fallback ? p.elem : batch_alignment(p, ranked[index]);
    GuardedBuffer gin(n, idata, align, 0xA5), gout(n, odata, align, 0x5A);
    std::memcpy(gin.data(), idata, n);
    batch_regroup(run, ub);
    run.in = gin.data();
    run.out = gout.data();
    const int start[2] = {0, run.units};
    if (!replay_batch(&run, start, 1, run.units, grid)) return LIBRETT_C_UNDEFINED_ERROR;
    if (!gout.intact()) return LIBRETT_C_UNDEFINED_ERROR;
    std::memcpy(odata, gout.data(), n);
    return LIBRETT_C_SUCCESS;
  } catch (...) {
    return LIBRETT_C_INTERNAL_ERROR;
  }
}

}  // extern "C"
