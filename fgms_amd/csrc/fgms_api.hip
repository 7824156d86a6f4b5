// extern "C" entry points of libfgms_hip.so: argument checks, kernel selection,
// workspace bookkeeping.  The host-side counterpart of backend/spconv.cu:23-571.
#include <stdarg.h>
#include <stdio.h>

#include <algorithm>
#include <atomic>
#include <initializer_list>
#include <map>
#include <mutex>
#include <utility>
#include <vector>
#include <string.h>

#include "fgms_internal.h"

namespace fgms {

static thread_local char g_error[512] = "";
static int g_policy = 0;
int kernel_policy() { return g_policy; }

void set_error(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_error, sizeof(g_error), fmt, ap);
  va_end(ap);
}

// ---- workspace: one growable buffer per (device, stream, slot) --------------
namespace {
struct WsKey {
  int device;
  hipStream_t stream;
  int slot;
  bool operator<(const WsKey &o) const {
    if (device != o.device) return device < o.device;
    if (stream != o.stream) return stream < o.stream;
    return slot < o.slot;
  }
};
struct WsBuf {
  void *ptr = nullptr;
  size_t bytes = 0;
  bool captured = false;      // a call under stream capture was given it: a graph points at it
};
std::mutex g_ws_mutex;
std::map<WsKey, WsBuf> g_ws;
}  // namespace

bool is_capturing(hipStream_t stream) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return stream && hipStreamIsCapturing(stream, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

size_t workspace_bytes(hipStream_t stream, int slot) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 0;
  std::lock_guard<std::mutex> lock(g_ws_mutex);
  auto it = g_ws.find(WsKey{dev, stream, slot});
  return it == g_ws.end() ? 0 : it->second.bytes;
}

// Device / pinned allocations the library has made since it was loaded (fgms_allocation_count).
std::atomic<long long> g_allocations{0};
void note_allocation() { g_allocations.fetch_add(1, std::memory_order_relaxed); }

int workspace_get(hipStream_t stream, int slot, size_t bytes, void **ptr, bool *fresh) {
  if (fresh) *fresh = false;
  int dev = 0;
  FGMS_HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_ws_mutex);
  WsBuf &b = g_ws[WsKey{dev, stream, slot}];
  const bool capturing = is_capturing(stream);
  if (b.bytes < bytes) {
    if (capturing) {
      // (an allocation cannot be recorded)
      set_error("a workspace of %zu bytes is needed while the stream is being captured: run the call once "
                "outside the capture first", bytes);
      return FGMS_E_INVALID;
    }
    const size_t want = bytes + bytes / 4 + 4096;
    void *p = nullptr;
    const int rc = pool_alloc(&p, want, stream);
    if (rc != FGMS_OK) return rc;
    // The old buffer goes back to the pool, to be handed out again behind the work queued on this stream;
    // one that a capture was given is kept for good: a replay of the graph may come at any time, and nothing
    // says when the graph is gone.  (Buffers grow by a quarter and more, so all that is kept of one is less
    // than four times its latest size.)
    if (b.ptr && !b.captured) pool_free(b.ptr, stream, false);
    b = WsBuf{p, want, false};
    if (fresh) *fresh = true;
  }
  b.captured |= capturing;
  *ptr = b.ptr;
  return FGMS_OK;
}

// ---- re-laid copies of pinned weights -----------------------------------------
// Some kernels read the weights from a re-laid copy, made by a small launch in front of the
// main one (4-9 us where the main launch takes 90).  A caller that promises that a weight
// tensor's bytes stay as they are (fgms_weights_pin: inference, or between two optimizer
// steps) lets the library keep those copies, per (address, layout), until fgms_weights_unpin
// or the next fgms_weights_pin of the address.
namespace {
struct RelaidCopy {
  const void *w;
  int device;
  unsigned layout;
  int k_vol, c_in, c_out;
  size_t bytes;
  void *ptr;
  hipStream_t made_on;
  hipEvent_t ready;                  // nullptr: the fill has not been queued (yet)
  std::vector<hipStream_t> users;    // streams other than made_on that wait for `ready` already
};
std::mutex g_pin_mutex;
std::vector<std::pair<int, const void *>> g_pinned;
std::vector<RelaidCopy> g_relaid;
std::atomic<int> g_pinned_count{0};
std::atomic<long long> g_relaid_hits{0};

bool is_pinned_locked(int dev, const void *w) {
  for (const auto &e : g_pinned)
    if (e.first == dev && e.second == w) return true;
  return false;
}

// Hands a copy's block back to the pool once every stream that read it has passed this point.
void retire_locked(RelaidCopy &c) {
  for (hipStream_t s : c.users) {
    hipEvent_t ev = nullptr;
    if (hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) continue;
    if (hipEventRecord(ev, s) == hipSuccess) (void)hipStreamWaitEvent(c.made_on, ev, 0);
    (void)hipEventDestroy(ev);
  }
  if (c.ready) (void)hipEventDestroy(c.ready);
  pool_free(c.ptr, c.made_on, false);
}

void drop_copies_locked(int dev, const void *w) {
  for (size_t i = 0; i < g_relaid.size();) {
    if (g_relaid[i].device == dev && g_relaid[i].w == w) {
      retire_locked(g_relaid[i]);
      g_relaid.erase(g_relaid.begin() + i);
    } else {
      ++i;
    }
  }
}
}  // namespace

bool weights_pinned(const void *w) {
  if (g_pinned_count.load(std::memory_order_relaxed) == 0) return false;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  std::lock_guard<std::mutex> lock(g_pin_mutex);
  return is_pinned_locked(dev, w);
}

int relaid_weights_buffer(const GmsArgs &a, unsigned layout, size_t bytes, void **ptr, bool *fill) {
  *fill = true;
  if (g_pinned_count.load(std::memory_order_relaxed) > 0) {
    int dev = 0;
    FGMS_HIP_TRY(hipGetDevice(&dev));
    const bool capturing = is_capturing(a.stream);
    std::lock_guard<std::mutex> lock(g_pin_mutex);
    if (!capturing && is_pinned_locked(dev, a.w)) {
      for (RelaidCopy &c : g_relaid) {
        if (c.w != a.w || c.device != dev || c.layout != layout || c.k_vol != a.k_vol || c.c_in != a.c_in ||
            c.c_out != a.c_out || c.bytes != bytes)
          continue;
        *ptr = c.ptr;
        if (!c.ready) {           // an earlier call failed between the buffer and its fill
          c.made_on = a.stream;
          c.users.clear();
          return FGMS_OK;
        }
        if (a.stream != c.made_on && std::find(c.users.begin(), c.users.end(), a.stream) == c.users.end()) {
          FGMS_HIP_TRY(hipStreamWaitEvent(a.stream, c.ready, 0));
          c.users.push_back(a.stream);
        }
        *fill = false;
        g_relaid_hits.fetch_add(1, std::memory_order_relaxed);
        return FGMS_OK;
      }
      void *p = nullptr;
      int rc = pool_alloc(&p, bytes, a.stream);
      if (rc != FGMS_OK) return rc;
      g_relaid.push_back(RelaidCopy{a.w, dev, layout, a.k_vol, a.c_in, a.c_out, bytes, p, a.stream, nullptr, {}});
      *ptr = p;
      return FGMS_OK;
    }
  }
  return workspace_get(a.stream, 0, bytes, ptr);
}

void relaid_weights_filled(const GmsArgs &a, void *ptr) {
  if (g_pinned_count.load(std::memory_order_relaxed) == 0) return;
  std::lock_guard<std::mutex> lock(g_pin_mutex);
  for (RelaidCopy &c : g_relaid) {
    if (c.ptr != ptr || c.ready) continue;
    hipEvent_t ev = nullptr;
    if (hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) return;
    if (hipEventRecord(ev, a.stream) != hipSuccess) {
      (void)hipEventDestroy(ev);
      return;
    }
    c.ready = ev;
    return;
  }
}

extern "C" int fgms_weights_pin(const void *kernel) {
  if (!kernel) {
    set_error("fgms_weights_pin: null pointer");
    return FGMS_E_INVALID;
  }
  int dev = 0;
  FGMS_HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_pin_mutex);
  if (is_pinned_locked(dev, kernel)) {
    drop_copies_locked(dev, kernel);       // pinned again: the bytes have changed since
  } else {
    g_pinned.emplace_back(dev, kernel);
    g_pinned_count.store((int)g_pinned.size(), std::memory_order_relaxed);
  }
  return FGMS_OK;
}

extern "C" int fgms_weights_unpin(const void *kernel) {
  int dev = 0;
  FGMS_HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_pin_mutex);
  for (size_t i = 0; i < g_pinned.size();) {
    if (g_pinned[i].first == dev && (!kernel || g_pinned[i].second == kernel)) {
      drop_copies_locked(dev, g_pinned[i].second);
      g_pinned.erase(g_pinned.begin() + i);
    } else {
      ++i;
    }
  }
  g_pinned_count.store((int)g_pinned.size(), std::memory_order_relaxed);
  return FGMS_OK;
}

extern "C" long long fgms_relaid_weights_hits(void) { return g_relaid_hits.load(std::memory_order_relaxed); }

// ---- dynamic-LDS limits already granted, per (device, kernel) ------------------
namespace {
std::mutex g_lds_mutex;
std::map<std::pair<int, const void *>, size_t> g_lds_granted;
}  // namespace

int allow_dynamic_lds(const void *kernel, size_t bytes) {
  int dev = 0;
  FGMS_HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(g_lds_mutex);
  size_t &granted = g_lds_granted[{dev, kernel}];
  if (granted >= bytes) return FGMS_OK;
  FGMS_HIP_TRY(hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
  granted = bytes;
  return FGMS_OK;
}

// ---- block pool: device memory of plans and of the map builder's temporaries --
// hipMalloc / hipFree cost 50-100 us each and a plan needs a dozen blocks, which
// made building a plan (once per kernel map, i.e. several times per training
// step) three times as expensive as its kernels.  Freed blocks are kept per
// device and handed out again to requests of similar size.  A block that may
// still be read by queued work carries an event recorded on the stream that used
// it last; whoever gets the block next makes its own stream wait for that event.
namespace {
struct PoolBlock {
  void *ptr;
  size_t bytes;
  int device;
  hipEvent_t ready;    // nullptr: idle
};
std::mutex g_pool_mutex;
std::vector<PoolBlock> g_pool_free;
std::map<void *, std::pair<size_t, int>> g_pool_live;   // ptr -> (bytes, device)
size_t g_pool_cached = 0;
constexpr size_t kPoolMaxCached = (size_t)2 << 30;

// Events for blocks on their way back, and for plans: kept per device, a few dozen at most.
std::mutex g_event_mutex;
std::vector<std::pair<int, hipEvent_t>> g_events;
}  // namespace

hipEvent_t event_get(int device) {
  {
    std::lock_guard<std::mutex> lock(g_event_mutex);
    for (size_t i = g_events.size(); i-- > 0;)
      if (g_events[i].first == device) {
        hipEvent_t ev = g_events[i].second;
        g_events.erase(g_events.begin() + i);
        return ev;
      }
  }
  hipEvent_t ev = nullptr;
  return hipEventCreateWithFlags(&ev, hipEventDisableTiming) == hipSuccess ? ev : nullptr;
}

void event_put(hipEvent_t ev, int device) {
  {
    std::lock_guard<std::mutex> lock(g_event_mutex);
    if (g_events.size() < 64) {
      g_events.emplace_back(device, ev);
      return;
    }
  }
  (void)hipEventDestroy(ev);
}

int pool_alloc(void **ptr, size_t bytes, hipStream_t user) {
  *ptr = nullptr;
  if (bytes == 0) bytes = 256;
  bytes = (bytes + 255) & ~(size_t)255;
  int dev = 0;
  FGMS_HIP_TRY(hipGetDevice(&dev));
  PoolBlock got{};
  {
    std::lock_guard<std::mutex> lock(g_pool_mutex);
    int best = -1;
    for (int i = 0; i < (int)g_pool_free.size(); ++i) {
      const PoolBlock &b = g_pool_free[i];
      if (b.device != dev || b.bytes < bytes || b.bytes > 2 * bytes + 4096) continue;
      if (best < 0 || b.bytes < g_pool_free[best].bytes) best = i;
    }
    if (best >= 0) {
      got = g_pool_free[best];
      g_pool_free.erase(g_pool_free.begin() + best);
      g_pool_cached -= got.bytes;
      g_pool_live[got.ptr] = {got.bytes, dev};
    }
  }
  if (got.ptr) {
    if (got.ready) {
      hipError_t e = hipStreamWaitEvent(user, got.ready, 0);
      event_put(got.ready, got.device);
      if (e != hipSuccess) {
        set_error("pool_alloc: hipStreamWaitEvent: %s", hipGetErrorString(e));
        return FGMS_E_HIP;
      }
    }
    *ptr = got.ptr;
    return FGMS_OK;
  }
  void *q = nullptr;
  note_allocation();
  if (hipMalloc(&q, bytes) != hipSuccess) {
    // give cached blocks back to the driver and try once more
    pool_trim(0);
    if (hipMalloc(&q, bytes) != hipSuccess) {
      set_error("device allocation of %zu bytes failed", bytes);
      return FGMS_E_NOMEM;
    }
  }
  std::lock_guard<std::mutex> lock(g_pool_mutex);
  g_pool_live[q] = {bytes, dev};
  *ptr = q;
  return FGMS_OK;
}

void pool_free(void *ptr, hipStream_t last_user, bool idle) {
  if (!ptr) return;
  PoolBlock b{};
  {
    std::lock_guard<std::mutex> lock(g_pool_mutex);
    auto it = g_pool_live.find(ptr);
    if (it == g_pool_live.end()) return;
    b = PoolBlock{ptr, it->second.first, it->second.second, nullptr};
    g_pool_live.erase(it);
  }
  if (!idle) {
    // queued work may still read the block: mark the point after which it is free
    hipEvent_t ev = event_get(b.device);
    if (!ev || hipEventRecord(ev, last_user) != hipSuccess) {
      if (ev) (void)hipEventDestroy(ev);
      (void)hipFree(ptr);     // synchronises; also the path taken while the runtime shuts down
      return;
    }
    b.ready = ev;
  }
  std::lock_guard<std::mutex> lock(g_pool_mutex);
  g_pool_free.push_back(b);
  g_pool_cached += b.bytes;
  while (g_pool_cached > kPoolMaxCached && !g_pool_free.empty()) {
    PoolBlock old = g_pool_free.front();
    g_pool_free.erase(g_pool_free.begin());
    g_pool_cached -= old.bytes;
    if (old.ready) (void)hipEventDestroy(old.ready);
    (void)hipFree(old.ptr);
  }
}

void pool_trim(size_t keep_bytes) {
  std::lock_guard<std::mutex> lock(g_pool_mutex);
  while (g_pool_cached > keep_bytes && !g_pool_free.empty()) {
    PoolBlock old = g_pool_free.front();
    g_pool_free.erase(g_pool_free.begin());
    g_pool_cached -= old.bytes;
    if (old.ready) (void)hipEventDestroy(old.ready);
    (void)hipFree(old.ptr);
  }
}

// ---- profiling records -------------------------------------------------------
namespace {
struct ProfRec {
  const char *name;
  hipEvent_t start, stop;
};
std::mutex g_prof_mutex;
std::vector<ProfRec> g_prof;
bool g_prof_on = false;
}  // namespace

ProfileScope::ProfileScope(const char *name, hipStream_t s) : slot(-1), stream(s) {
  if (!g_prof_on) return;
  std::lock_guard<std::mutex> lock(g_prof_mutex);
  ProfRec r{name, nullptr, nullptr};
  if (hipEventCreate(&r.start) != hipSuccess || hipEventCreate(&r.stop) != hipSuccess) return;
  (void)hipEventRecord(r.start, stream);
  g_prof.push_back(r);
  slot = (int)g_prof.size() - 1;
}

ProfileScope::~ProfileScope() {
  if (slot < 0) return;
  std::lock_guard<std::mutex> lock(g_prof_mutex);
  if (slot < (int)g_prof.size()) (void)hipEventRecord(g_prof[slot].stop, stream);
}

namespace {

int check_common(const void *a, const void *b, const void *c, const int32_t *kpos,
                 const int32_t *imap, const int32_t *omap, int64_t n_in, int64_t n_out, int c_in,
                 int c_out, int k_vol, int64_t n_pairs, int dtype) {
  if (dtype != FGMS_F32 && dtype != FGMS_F16) {
    set_error("dtype must be FGMS_F32 (0) or FGMS_F16 (1), got %d", dtype);
    return FGMS_E_INVALID;
  }
  if (n_in < 0 || n_out < 0 || c_in <= 0 || c_out <= 0 || k_vol <= 0 || n_pairs < 0) {
    set_error("bad sizes: n_in=%lld n_out=%lld c_in=%d c_out=%d k_vol=%d n_pairs=%lld",
              (long long)n_in, (long long)n_out, c_in, c_out, k_vol, (long long)n_pairs);
    return FGMS_E_INVALID;
  }
  if (n_in > INT32_MAX || n_out > INT32_MAX || n_pairs > INT32_MAX - 65536) {
    set_error("row and pair counts must fit int32 (the maps are int32)");
    return FGMS_E_INVALID;
  }
  if (!kpos || (n_pairs > 0 && (!imap || !omap)) ||
      ((n_in > 0 || n_out > 0) && (!a || !b || !c))) {
    set_error("null pointer argument");
    return FGMS_E_INVALID;
  }
  return FGMS_OK;
}

// The output-stationary kernel multiplies every (64-row block, offset) combination in
// use, 64 row slots each, whether or not a row has a pair there; the pair-stationary
// kernels multiply pairs only and pay with an atomic per result element.  Which one wins
// depends on the row slots per pair of the map (1.0 .. 1.2 for surface-like clouds at full
// density, 2 .. 3 for random subsamples of them) and on the channel count.  Measured on
// MI355X over subsamples of a 200 k-voxel indoor-like cloud (35 k .. 200 k voxels, 32 .. 256
// channels), the slots per pair at which both take the same time:
//   fp16: 2.25 .. 2.5 at every channel count (2.2 + 16 / c);
//   fp32 MFMAs: 2.35 / 1.76 / 1.3 at 32 / 64 / 128 channels, about 1 + 45 / c.
// The kernel without atomics, whose results do not depend on the run, gets 5 % on top.
// fp32 tensors in bf16 parts, beyond that line: products cost so little that the output-stationary kernel's chain of stages counts (a
// stage: an offset and a slab of 32 channels; a tile waits for one after the other), and what the (64-row block, offset)
// combinations of all its tiles come to, against the pair view's atomics and gathers.  Fitted to either kernel over 17 channel counts from
// 32 x 32 to 256 x 256 on indoor, LiDAR and scattered clouds of 500 .. 150 k voxels, sorted and in scan order (half of the
// estimates are within 9 %, nine in ten within 21 .. 32 %; the choice costs 0.3 .. 1.4 % over the better of the two in the mean).
// Pair view / output-stationary, fp32: 64 -> 64 forward over 20 k scattered voxels 32 / 55 us, LiDAR 60 k 97 / 74; 96 -> 96 over that
// 140 / 207; 128 -> 128 input gradient over 50 k scattered 117 / 239; with its weight gradient, which the output-stationary
// kernel's grid hides, 64 -> 64 over 50 k 130 / 101, 128 -> 128 225 / 253.
double rows_us(const GmsArgs &a, const Plan *plan) {
  const int c_src = a.transpose_w ? a.c_out : a.c_in, c_dst = a.transpose_w ? a.c_in : a.c_out;
  const int slabs = (c_src + 31) / 32, cols = (c_dst + 31) / 32;
  const double blocks = (double)(a.transpose_w ? plan->stages_in : plan->stages_out) * cols / num_cus() *
                        (cols % 2 == 0 || cols == 1 ? 1 : a.reduced ? 1.66 : 1.36);      // (32 columns a tile: rows gathered once for each)
  const double chain = a.k_vol * (a.transpose_w && cols % 2 == 0 ? 1.3 : 1.0);           // (64; small forward launches take 32)
  return a.reduced ? 9.6 + slabs * (0.293 * chain + 0.139 * blocks) : 9.8 + slabs * (0.41 * chain + 0.271 * blocks);
}
double pair_view_us(const GmsArgs &a, double pairs) {
  const int c_src = a.transpose_w ? a.c_out : a.c_in, c_dst = a.transpose_w ? a.c_in : a.c_out;
  return a.reduced ? 14.1 + 3.4e-4 * c_src * c_dst + 1e-6 * pairs * c_dst * (2.8 + 0.0046 * c_src)
                   : 14.6 + 6.1e-4 * c_src * c_dst + 1e-6 * pairs * c_dst * (2.7 + 0.0104 * c_src);
}
// `masked`: the channels' rest would be masked (else counts that are no multiple of 32 stay on fp32 MFMAs, which the first rule is for).
bool sparse_rows(const GmsArgs &a, const Plan *plan, bool masked = false) {
  const int stages = a.transpose_w ? plan->stages_in : plan->stages_out;
  if (stages <= 0 || plan->pairs_counted <= 0) return false;   // (the plan's own pair count: a.n_pairs is a bound)
  const double slots_per_pair = (double)stages * 64.0 / (double)plan->pairs_counted;
  const double c_src = a.transpose_w ? a.c_out : a.c_in;
  const double even = a.dtype == FGMS_F16 ? 2.2 + 16.0 / c_src : 1.0 + 45.0 / c_src;
  // (no break-even point was measured below 1.3: denser maps stay output-stationary)
  const double need = 1.05 * even;
  if (slots_per_pair <= (need > 1.4 ? need : 1.4)) return false;
  return a.dtype == FGMS_F16 || !split_bf16_enabled() || ((int)c_src % 32 != 0 && !masked) ||
         rows_us(a, plan) > pair_view_us(a, (double)plan->pairs_counted) + a.beside_us;
}

enum class Route { kNarrow, kSkinny, kRows, kPairView, kWide, kPairs, kGeneric };

// Which kernel a forward / input-gradient pass takes.  (A question only, asked for estimates too: a pair view that is not there yet is
// built by the call that walks it.  with_view = false: it could not be had.)
Route route_of(const GmsArgs &a, const Plan *plan, bool with_view = true) {
  const bool dense = a.dense_k >= 0;
  if (g_policy == 1) return Route::kGeneric;
  const bool pair_view = !dense && with_view && pair_view_gms_supported(a, plan);
  if (g_policy == 5 && pair_view) return Route::kPairView;
  // (16 -> 64 channels fill the output-stationary kernel's tiles: 150 k voxels 20 us, 39 us here; the others 1.1 .. 3 times
  // faster than on the vector ALUs from 2 k to 150 k voxels)
  if (!dense && (g_policy == 0 || g_policy == 4) && narrow_gms_supported(a, plan) &&
      !(a.c_in == 16 && a.c_out > 32 && planned_gms_supported(a, plan) && !sparse_rows(a, plan)))
    return Route::kNarrow;
  if (!dense && (g_policy == 0 || g_policy == 4) && small_gms_supported(a, plan)) return Route::kSkinny;
  if (g_policy == 7 && wide_gms_supported(a)) return Route::kWide;
  if (!dense && g_policy != 2 && planned_gms_supported(a, plan) &&
      !(g_policy != 4 && sparse_rows(a, plan) && mfma_gms_supported(a)))
    return Route::kRows;
  // Which pair-stationary kernel: the output-stationary kernel's body over the plan's pair
  // view streams the weights of a stage through LDS where gms_pairs_kernel holds a column
  // block's weights of one offset.  Measured (same clouds): fp32 a tie up to 128 channels,
  // 245 against 341 us at 256 -> 256 over 50 k voxels; fp16 14.2 against 18.3 us at 64
  // channels over 35 k voxels, a tie from 128 channels on (96.6 against 96.3 us at 256).
  if (g_policy == 0 && pair_view && (a.dtype == FGMS_F32 || (a.transpose_w ? a.c_out : a.c_in) <= 64))
    return Route::kPairView;
  if (g_policy == 0 && wide_gms_supported(a)) return Route::kWide;
  return mfma_gms_supported(a) ? Route::kPairs : Route::kGeneric;
}

int run_gms(GmsArgs a, const Plan *plan);
int run_gms_one(GmsArgs a, const Plan *plan);

// ---- channel counts no tuned kernel takes: padded copies (fgms_pad.hip) -----------------------
// Workspace slots of the copies (slots 0 .. 3: see fgms_internal.h).
constexpr int kSlotPadIn = 4, kSlotPadOut = 5, kSlotPadWeights = 6, kSlotPadResult = 7;

// May the call grow the stream's workspaces?  (Not under stream capture: the shape-agnostic
// kernels, which need none, then serve it unless an earlier call has left them big enough.)
bool workspaces_fit(hipStream_t s, std::initializer_list<std::pair<int, size_t>> wanted) {
  if (!is_capturing(s)) return true;
  for (const auto &w : wanted)
    if (workspace_bytes(s, w.first) < w.second) return false;
  return true;
}

int up_to_power_of_two(int c, int least) {
  int p = least;
  while (p < c) p *= 2;
  return p;
}
int up_to_32(int c) { return (c + 31) / 32 * 32; }

size_t elem_size(int dtype) { return dtype == FGMS_F16 ? 2 : 4; }

// `a` as it would look over padded copies (aligned, so any address will do).
GmsArgs with_channels(GmsArgs a, int c_in, int c_out) {
  a.c_in = c_in;
  a.c_out = c_out;
  a.src = a.w = (const void *)4096;
  a.dst = (void *)4096;
  return a;
}

// Route of a pass over all offsets (of its first group, for plans over more than 64).
Route first_route(const GmsArgs &a, const Plan *plan) {
  if (plan && !plan->groups.empty() && a.dense_k < 0) {
    GmsArgs g = a;
    g.k_vol = plan->groups.front()->k_vol;
    return route_of(g, plan->groups.front());
  }
  return route_of(a, plan);
}
bool tuned_gms(const GmsArgs &a, const Plan *plan) { return first_route(a, plan) != Route::kGeneric; }

// fp32 passes: padded copies, or the vector ALUs' kernel on the channels as they are.  The copies are two
// more launches in front (three where the weights are re-laid) and one behind, and on small clouds a tile's
// chain of fp32 products is all there is to the main launch, where the shape-agnostic kernel spreads single
// 32-pair pieces over the chip.  The functions below estimate either side in microseconds, fitted to 22 channel
// counts from 3 x 32 to 96 x 100 and 48 x 200 over 500 .. 60 k voxels, dense, LiDAR and thinned clouds, with and without a
// plan (4 500 pairs of times; half of the estimates are within 8 % and nine in ten within 20 %).  Forward,
// copies / vector ALUs: 32 -> 20 over 2 k dense voxels 32 / 16 us, 10 k 32 / 25, 14 k 32 / 31, 40 k 42 / 72;
// 48 -> 48 over 2 k 49 / 18, 20 k 76 / 64, 40 k 98 / 120; over 20 k thinned ones (pair view, atomics) 44 / 30.
double pairs_of(const GmsArgs &a, const Plan *plan) {
  return (double)(a.dense_k >= 0 ? a.n_dense : plan && plan->pairs_counted > 0 ? plan->pairs_counted : a.n_pairs);
}
int group_count(const GmsArgs &a, const Plan *plan) {
  return plan && !plan->groups.empty() && a.dense_k < 0 ? (int)plan->groups.size() : 1;
}
// Products (pieces of 32 source and 64 destination channels), atomics, gathered channels.
double vector_alu_us(const GmsArgs &a, const Plan *plan) {
  const int c_src = a.transpose_w ? a.c_out : a.c_in, c_dst = a.transpose_w ? a.c_in : a.c_out;
  const double base = (a.overwrite ? 13 : 11) * group_count(a, plan);       // (fill and) launch
  return base + 1e-6 * pairs_of(a, plan) * (0.043 * up_to_32(c_src) * ((c_dst + 63) / 64 * 64) + 1.4 * c_dst + c_src);
}
// `p`: the pass over the copies.  What a small launch takes is its launches and a tile's chain of (offset,
// 32-channel slab) stages, more of it once there is more than a tile to a CU; the routes with atomics add what these cost.
double padded_us(const GmsArgs &p, const Plan *plan) {
  const int c_src = p.transpose_w ? p.c_out : p.c_in, c_dst = p.transpose_w ? p.c_in : p.c_out;
  const double slabs = (c_src + 31) / 32, wide = c_dst % 64 == 0 ? 1 : 0;
  switch (first_route(p, plan)) {
    case Route::kNarrow:
    case Route::kSkinny: return 17 * group_count(p, plan) + (p.transpose_w ? 1.5 : c_src * c_dst / 45.0);
    case Route::kRows: return 6 + rows_us(p, plan);      // (copies in front, crop behind)
    default:
      return 20 + 1.5 * slabs * (1 + wide) + 1e-6 * pairs_of(p, plan) * (p.dense_k >= 0 ? 2.0 * c_dst : 3.4 * c_dst + 0.4 * c_src);
  }
}
// The same over the masked tiles (fp32: no copies, nothing to crop), with the weight gradient beside the input's if there is one.
// Forward, measured (estimated), fp32 and tf32 mode: 24 -> 32 over 4 k dense voxels 24.1 us (21.7) and 18.6 (18.2), 48 -> 48 over 30 k
// 56 (58) and 34 (39), LiDAR 60 k 77 (76) and 42 (49).  On the vector ALUs 24 -> 32 over 4 k 15, 48 -> 48 over 30 k 93.  Both gradients:
// 24 -> 32 over 4 k 22.6 (22.4) and 19.6 (18.9), 48 -> 48 45 (44) and 34 (35), over 60 k 127 (129) and 86 (98).
double masked_us(const GmsArgs &a, const Plan *plan) {
  return rows_us(a, plan) + (a.transpose_w ? 16e-6 * pairs_of(a, plan) * (up_to_32(a.c_in) / 32) * (up_to_32(a.c_out) / 32) : 0);
}
bool takes_ragged(const GmsArgs &a, const Plan *plan);
bool padding_pays(const GmsArgs &a, const Plan *plan, int c_in, int c_out) {
  if (a.dtype != FGMS_F16 && takes_ragged(a, plan) && ragged_gms_supported(a, plan)) return masked_us(a, plan) < vector_alu_us(a, plan);
  // (fp16 adds on the vector ALUs cost ten times as much: 32 -> 20 over 500 voxels 17 us over copies, 24 without.
  // The copies' fp32 kernels mostly do without atomics: a near tie goes to them.)
  return a.dtype == FGMS_F16 || padded_us(with_channels(a, c_in, c_out), plan) < 1.05 * vector_alu_us(a, plan);
}

// Widened channels of a forward / input-gradient pass that no tuned kernel takes as it is: the
// skinny kernel's where its products are no more than the padded MFMA tile's eighth (it runs on
// the vector ALUs), else multiples of the MFMA kernels' 32.
bool padded_gms_channels(const GmsArgs &a, const Plan *plan, int *c_in, int *c_out) {
  if (g_policy != 0 || tuned_gms(a, plan)) return false;
  const int si = up_to_power_of_two(a.c_in, 4), so = up_to_power_of_two(a.c_out, 4);
  if (si * so <= 256 && tuned_gms(with_channels(a, si, so), plan)) {
    *c_in = si; *c_out = so;
  } else {
    *c_in = up_to_32(a.c_in); *c_out = up_to_32(a.c_out);
    if (!tuned_gms(with_channels(a, *c_in, *c_out), plan)) return false;
  }
  return padding_pays(a, plan, *c_in, *c_out);
}

// Layers whose channels fill no whole tile go straight to kernels that mask the rest, where the map
// is dense enough for the output-stationary kernel (else the pair-stationary kernels over padded copies).
bool takes_ragged(const GmsArgs &a, const Plan *plan) {
  return g_policy == 0 && plan && a.n_pairs > 0 && a.dense_k < 0 && !narrow_gms_supported(a, plan) &&
         !small_gms_supported(a, plan) && !sparse_rows(a, plan, true);
}

// fp32 counts that are no multiple of 32: over the masked tiles where another matrix kernel takes them as they are or the
// vector ALUs are slower.  (Not for 16 channels forward in fp32: half of every slab of 32 is empty, and eight products (then six)
// each make it more than 61 us for 16 -> 64 over 120 k voxels where slabs of 16 on fp32 MFMAs took 47; in tf32 mode 36.)
bool ragged_pays(const GmsArgs &a, const Plan *plan) {
  int pi, po;
  if (a.dtype == FGMS_F16) return true;
  const size_t parts = (size_t)a.k_vol * up_to_32(a.c_in) * up_to_32(a.c_out) * (a.reduced ? 4 : 6);
  if (parts > 0xfffffff0u || !workspaces_fit(a.stream, {{0, parts}})) return false;     // (the re-laid weights)
  if (tuned_gms(a, plan)) return a.reduced || a.transpose_w || a.c_in > 16;
  return padded_gms_channels(a, plan, &pi, &po);
}

// A pass over all offsets: one walk for plans of up to 64 offsets (or none), one per group of 64
// offsets for larger kernels (the groups' results add up in the destination rows).
int run_gms_padded(const GmsArgs &a, const Plan *plan, int c_in, int c_out, bool *done);

// Does the output-stationary kernel take the centre offset along with the others?  (One launch instead of a fill, a
// re-layout, an atomic pass over all rows and a main launch that reads its result back: 48 -> 96 fp16 over 90 k voxels,
// a forward and a backward call, 125 -> 98 us.)
bool centre_rides(const GmsArgs &a, const Plan *plan) {
  if (!plan || a.n_pairs == 0 || !plan->groups.empty() || !plan->centre_line || a.centre - 1 != a.k_vol / 2 || a.n_src != a.n_dst) return false;
  if (brief_gms_pays(a, plan) || held_gms_pays(a, plan)) return true;
  if (takes_ragged(a, plan) && ragged_gms_supported(a, plan) && ragged_pays(a, plan)) return true;
  int pi, po;
  return route_of(padded_gms_channels(a, plan, &pi, &po) ? with_channels(a, pi, po) : a, plan) == Route::kRows;
}

// The centre offset by itself.
int run_centre(GmsArgs a) {
  a.gmap = a.smap = nullptr;
  a.dense_k = a.centre - 1;
  a.n_dense = a.n_dst;
  a.centre = 0;
  a.side = SideJob{};
  return run_gms(a, nullptr);
}

int run_gms(GmsArgs a, const Plan *plan) {
  if (a.centre && !centre_rides(a, plan)) {
    const int rc = run_centre(a);
    if (rc != FGMS_OK) return rc;
    a.centre = 0;
    a.overwrite = false;
  }
  int pi, po;
  if (brief_gms_pays(a, plan)) {
    plan_touch(plan, a.stream);
    return launch_brief_gms(a, plan);
  }
  if (held_gms_pays(a, plan)) {
    plan_touch(plan, a.stream);
    return launch_held_gms(a, plan);
  }
  if (takes_ragged(a, plan) && ragged_gms_supported(a, plan) && ragged_pays(a, plan)) {
    plan_touch(plan, a.stream);
    return launch_ragged_gms(a, plan);
  }
  if ((a.dense_k >= 0 ? a.n_dense : a.n_pairs) > 0 && padded_gms_channels(a, plan, &pi, &po)) {
    bool done = false;
    const int rc = run_gms_padded(a, plan, pi, po, &done);
    if (rc != FGMS_OK || done) return rc;
  }
  if (!plan || plan->groups.empty() || a.dense_k >= 0) return run_gms_one(a, plan);
  plan_touch(plan, a.stream);
  const size_t esz = a.dtype == FGMS_F16 ? 2 : 4;
  int k0 = 0;
  for (const Plan *g : plan->groups) {
    GmsArgs ga = a;
    ga.w = (const char *)a.w + (size_t)k0 * a.c_in * a.c_out * esz;
    ga.kpos = a.kpos + k0;
    ga.k_vol = g->k_vol;
    ga.overwrite = a.overwrite && k0 == 0;      // (the later groups add to the first one's sums)
    int rc = run_gms_one(ga, g);
    if (rc != FGMS_OK) return rc;
    k0 += g->k_vol;
  }
  return FGMS_OK;
}

// Is the list of an offset that meets every row once worth a launch of its own, in front of the other pairs'?  It saves that launch
// the fill and an atomic per result element (a sixth to a third of a thin map's) and costs a tile's chain of slabs.  Fitted over
// 2 k .. 50 k scattered voxels; all pairs with atomics over zeros / the middle offset's list first: 128 -> 128 over 16 k 25.3 / 27.8 us, 50 k
// 50.8 / 47.6, 256 -> 128 over 50 k 62.6 / 60.6, 40 k 44.2 / 45.6,
// 256 -> 256 over 6 k 32.4 / 44.5, 16 k 45.2 / 51.3, 32 k 72.5 / 71.9, 50 k 100.9 / 88.3, 128 -> 256 over 30 k 63.3 / 59.6.
bool full_offset_pays(const GmsArgs &a, Route route) {
  if (a.dtype != FGMS_F16) return false;
  const int c_src = a.transpose_w ? a.c_out : a.c_in, c_dst = a.transpose_w ? a.c_in : a.c_out;
  const double saved = 1e-6 * (double)a.n_dst * c_dst * (route == Route::kWide ? 2.05 : 1.25);
  const double costs = route == Route::kWide ? 10.4 + 0.0125 * c_src : 3.3 + 0.0145 * c_src;
  return saved > costs + 2.5;
}

// That offset, or -1.  (A plan of another map, which the kernels that walk the lists do without, says nothing about these lists.)
int full_offset_of(const GmsArgs &a, const Plan *plan) {
  if (!plan || a.k_vol != plan->k_vol) return -1;
  if (a.transpose_w) return a.n_dst == plan->n_in && a.n_src == plan->n_out ? plan->full_in : -1;
  return a.n_dst == plan->n_out && a.n_src == plan->n_in ? plan->full_out : -1;
}

int run_gms_one(GmsArgs a, const Plan *plan) {
  if (plan) plan_touch(plan, a.stream);
  const bool dense = a.dense_k >= 0;
  auto zero_result = [&]() {
    return launch_fill_zero(a.dst, (size_t)a.n_dst * (a.transpose_w ? a.c_in : a.c_out) * elem_size(a.dtype), a.stream);
  };
  if ((!dense && a.n_pairs == 0) || (dense && a.n_dense == 0)) return a.overwrite ? zero_result() : FGMS_OK;
  Route route = route_of(a, plan);
  if (route == Route::kPairView && !plan_pair_view(plan, a)) route = route_of(a, plan, false);
  if (a.centre && route != Route::kRows) {      // (the copies it was to run over could not be had)
    const int rc = run_centre(a);
    if (rc != FGMS_OK) return rc;
    a.centre = 0;
    a.overwrite = false;
  }
  // (these kernels add with atomics, several workgroups to a row.  Where the identity map, or the list of one offset, meets
  // every row once, its products are written in the place of the zeros.)
  const bool pairs = route == Route::kWide || route == Route::kPairs;
  if (pairs && a.overwrite && !dense && full_offset_pays(a, route)) a.first_offset = full_offset_of(a, plan) + 1;
  const bool written = pairs && a.overwrite && (a.first_offset || (dense && a.n_dense == a.n_dst));
  if (a.overwrite && !written && (pairs || route == Route::kGeneric)) {
    const int rc = zero_result();
    if (rc != FGMS_OK) return rc;
  }
  // (a pending fingerprint check of the plan rides along as the launch's side job)
  if (plan && !a.side.kind && route != Route::kGeneric) (void)plan_take_check(plan, &a.side);
  switch (route) {
    case Route::kNarrow: return launch_narrow_gms(a, plan);
    case Route::kSkinny: return launch_small_gms(a, plan);
    case Route::kRows: return launch_planned_gms(a, plan);
    case Route::kPairView: return launch_pair_view_gms(a, plan);
    case Route::kWide: return launch_wide_gms(a);
    case Route::kPairs: return launch_mfma_gms(a);
    default: return launch_generic_gms(a);
  }
}

// The pass over copies padded to c_in x c_out channels; *done = false (and nothing launched)
// where their workspaces cannot be had now.
int run_gms_padded(const GmsArgs &a, const Plan *plan, int c_in, int c_out, bool *done) {
  const size_t esz = elem_size(a.dtype);
  const int c_src = a.transpose_w ? a.c_out : a.c_in, c_dst = a.transpose_w ? a.c_in : a.c_out;
  const int p_src = a.transpose_w ? c_out : c_in, p_dst = a.transpose_w ? c_in : c_out;
  const size_t src_bytes = (size_t)a.n_src * p_src * esz, w_bytes = (size_t)a.k_vol * c_in * c_out * esz,
               dst_bytes = (size_t)a.n_dst * p_dst * esz;
  const int src_slot = a.transpose_w ? kSlotPadOut : kSlotPadIn;
  // (rows that fill whole tiles as they are need no copy, nor do results)
  const bool copy_src = p_src != c_src || reinterpret_cast<uintptr_t>(a.src) % 16;
  const bool crop = p_dst != c_dst || reinterpret_cast<uintptr_t>(a.dst) % 16;
  *done = workspaces_fit(a.stream, {{src_slot, copy_src ? src_bytes : 0}, {kSlotPadWeights, w_bytes}, {kSlotPadResult, crop ? dst_bytes : 0}});
  if (!*done) return FGMS_OK;
  GmsArgs p = a;
  p.c_in = c_in;
  p.c_out = c_out;
  void *src = nullptr, *w = nullptr, *dst = nullptr;
  int rc;
  if ((copy_src && (rc = workspace_get(a.stream, src_slot, src_bytes, &src))) || (rc = workspace_get(a.stream, kSlotPadWeights, w_bytes, &w)) ||
      (crop && (rc = workspace_get(a.stream, kSlotPadResult, dst_bytes, &dst))))
    return rc;
  PadBatch pads{};
  if (copy_src) {
    pads.add(a.src, src, (size_t)a.n_src, 1, 1, c_src, p_src, (int)esz);
    p.src = src;
  }
  pads.add(a.w, w, (size_t)a.k_vol, a.c_in, c_in, a.c_out, c_out, (int)esz);
  if ((rc = launch_pad(pads, a.dtype, a.stream))) return rc;
  p.w = w;
  if (crop) {
    p.dst = dst;
    p.overwrite = true;
  }
  if ((rc = run_gms(p, plan)) || !crop) return rc;
  return launch_crop(dst, a.dst, (size_t)a.n_dst, c_dst, p_dst, a.overwrite, a.dtype, a.stream);
}

// Widened channels of a weight gradient no MFMA / skinny kernel takes as it is.
bool padded_wgrad_channels(const WgradArgs &a, int *c_in, int *c_out) {
  if (g_policy != 0 || mfma_wgrad_supported(a)) return false;
  WgradArgs p = a;
  p.in = p.gout = (const void *)4096;
  if (a.c_in <= 16 && a.c_out <= 64) {
    p.c_in = up_to_power_of_two(a.c_in, 4);
    p.c_out = up_to_power_of_two(a.c_out, 16);
  } else {
    p.c_in = up_to_32(a.c_in);
    p.c_out = up_to_32(a.c_out);
  }
  *c_in = p.c_in; *c_out = p.c_out;
  p.crop_in = a.c_in; p.crop_out = a.c_out;      // (what will run, and at what price)
  return mfma_wgrad_supported(p) && (a.dtype == FGMS_F16 || padded_wgrad_us(p) < vector_alu_wgrad_us(a));
}

// The weight gradient over padded copies of the rows (as above); its fp32 sums are cropped when
// they are added to the caller's tensor.
int run_wgrad_padded(const WgradArgs &a, int c_in, int c_out, bool *done) {
  const size_t esz = elem_size(a.dtype);
  const bool copy_in = c_in != a.c_in || reinterpret_cast<uintptr_t>(a.in) % 16;
  const bool copy_gout = c_out != a.c_out || reinterpret_cast<uintptr_t>(a.gout) % 16;
  const size_t in_bytes = copy_in ? (size_t)a.n_in * c_in * esz : 0, gout_bytes = copy_gout ? (size_t)a.n_out * c_out * esz : 0;
  *done = workspaces_fit(a.stream, {{kSlotPadIn, in_bytes}, {kSlotPadOut, gout_bytes}, {1, (size_t)a.k_vol * c_in * c_out * sizeof(float)}});
  if (!*done) return FGMS_OK;
  void *in = nullptr, *gout = nullptr;
  int rc;
  if ((copy_in && (rc = workspace_get(a.stream, kSlotPadIn, in_bytes, &in))) ||
      (copy_gout && (rc = workspace_get(a.stream, kSlotPadOut, gout_bytes, &gout))))
    return rc;
  WgradArgs p = a;
  PadBatch pads{};
  if (copy_in) {
    pads.add(a.in, in, (size_t)a.n_in, 1, 1, a.c_in, c_in, (int)esz);
    p.in = in;
  }
  if (copy_gout) {
    pads.add(a.gout, gout, (size_t)a.n_out, 1, 1, a.c_out, c_out, (int)esz);
    p.gout = gout;
  }
  if ((rc = launch_pad(pads, a.dtype, a.stream))) return rc;
  p.c_in = c_in;
  p.c_out = c_out;
  p.crop_in = a.c_in;
  p.crop_out = a.c_out;
  return launch_mfma_wgrad(p);
}

int run_wgrad(const WgradArgs &a) {
  const size_t gw_bytes = (size_t)a.k_vol * a.c_in * a.c_out * elem_size(a.dtype);
  if (a.n_pairs == 0) return a.overwrite ? launch_fill_zero(a.gw, gw_bytes, a.stream) : FGMS_OK;
  if (a.plan) plan_touch(a.plan, a.stream);
  int pi, po;
  if (padded_wgrad_channels(a, &pi, &po)) {
    bool done = false;
    const int rc = run_wgrad_padded(a, pi, po, &done);
    if (rc != FGMS_OK || done) return rc;
  }
  if (g_policy != 1 && mfma_wgrad_supported(a)) return launch_mfma_wgrad(a);
  if (a.overwrite) {
    const int rc = launch_fill_zero(a.gw, gw_bytes, a.stream);
    if (rc != FGMS_OK) return rc;
  }
  return launch_generic_wgrad(a);
}

// Both gradients.
int run_bwd(GmsArgs d, const Plan *p, WgradArgs w) {
  int rc;
  // Both gradients through their main kernels: two launches instead of four.  The weight
  // gradient goes first and its launch also re-lays the weights for the input gradient,
  // whose launch in turn also rounds the weight gradient's fp32 sums into the caller's
  // fp16 tensor.  (The two gradients do not depend on each other.)
  if (d.n_pairs > 0 && (!p || p->groups.empty()) && route_of(d, p) == Route::kRows && g_policy != 1 && mfma_wgrad_supported(w)) {
    plan_touch(p, d.stream);
    // one launch for both where the shapes allow (and a small one that rounds an fp16
    // weight gradient), else two
    bool fused = false;
    if ((rc = launch_fused_bwd(d, p, w, &fused))) return rc;
    if (fused) return FGMS_OK;
    SideJob pack{}, flush{};
    const void *packed = nullptr;
    if ((rc = planned_pack_job(d, &pack, &packed))) return rc;
    w.side = pack;
    w.deferred_flush = &flush;
    if ((rc = launch_mfma_wgrad(w))) return rc;
    d.prepacked = packed;
    d.side = flush;
    if ((rc = launch_planned_gms(d, p))) {
      (void)launch_side_job(flush, d.stream);   // the accumulator must not stay filled
      return rc;
    }
    return FGMS_OK;
  }
  if ((rc = run_gms(d, p))) return rc;
  return run_wgrad(w);
}

// fp32: both gradients over shared copies in one grid (`pd`, `pw`), or each on its better side in a call of its own?
// The grid overlaps the shorter of the two with the longer.  (48 -> 48 over 2 k voxels: 55 us together, 19 and 20
// apart; 20 -> 128 over 10 k: 69 together, 69 and 50 apart.)
bool together_pays(const GmsArgs &d, const Plan *p, const WgradArgs &w, const GmsArgs &pd, const WgradArgs &pw) {
  const double in_us = padded_us(pd, p), w_us = padded_wgrad_us(pw);
  const double in_alone = tuned_gms(d, p) ? padded_us(d, p) : std::min(in_us, vector_alu_us(d, p));
  return std::max(in_us, w_us) + 0.4 * std::min(in_us, w_us) < 1.1 * (in_alone + std::min(w_us, vector_alu_wgrad_us(w)));
}

// fp32: both gradients over the masked tiles, or each on its better side?  The weights' hide behind the tiles; on their own they
// take three launches and what the copies' kernel adds (48 x 48: 15 us over 9 k pairs, 23 over 39 k, 74 over 69 k of 20 k scattered
// voxels, whose cells wait for more rows).  Masked / apart: 48 -> 48 over 4 k voxels 45 / 44 us, 20 k scattered ones 72 / 104; 24 -> 32
// over 1 k 22 / 28.  Maps too thin for the output-stationary kernel at the copies' channel counts stay with the copies.
bool masked_bwd_pays(const GmsArgs &d, const Plan *p, const WgradArgs &w) {
  if (d.dtype == FGMS_F16 || (tuned_gms(d, p) && mfma_wgrad_supported(w))) return true;
  const GmsArgs pd = with_channels(d, up_to_32(d.c_in), up_to_32(d.c_out));
  if (sparse_rows(pd, p)) return false;
  const double in_alone = tuned_gms(d, p) ? padded_us(d, p) : std::min(padded_us(pd, p), vector_alu_us(d, p));
  const double cells = (double)(pd.c_in / 32) * (pd.c_out / 32);
  const double w_alone = 12.3 + 6e-4 * (double)w.n_out + 1e-3 * (double)w.n_pairs * (0.045 + 0.05 * std::min(cells, 4.0));
  return masked_us(d, p) < 0.95 * (in_alone + w_alone);
}

// Widened channels for a backward pass one of whose gradients no tuned kernel takes as it is: the
// narrow layers' kernels up to 16 x 64, else multiples of 32 for both, which the one-grid launch takes.
bool padded_bwd_channels(const GmsArgs &d, const Plan *p, const WgradArgs &w, int *c_in, int *c_out) {
  if (g_policy != 0 || (tuned_gms(d, p) && mfma_wgrad_supported(w))) return false;
  for (int narrow = w.c_in <= 16 && w.c_out <= 64 ? 1 : 0; narrow >= 0; --narrow) {
    *c_in = narrow ? up_to_power_of_two(w.c_in, 4) : up_to_32(w.c_in);
    *c_out = narrow ? up_to_power_of_two(w.c_out, 16) : up_to_32(w.c_out);
    WgradArgs pw = w;
    pw.in = pw.gout = (const void *)4096;
    pw.c_in = *c_in;
    pw.c_out = *c_out;
    pw.crop_in = w.c_in;
    pw.crop_out = w.c_out;
    if (!tuned_gms(with_channels(d, *c_in, *c_out), p) || !mfma_wgrad_supported(pw)) continue;
    return d.dtype == FGMS_F16 || together_pays(d, p, w, with_channels(d, *c_in, *c_out), pw);
  }
  return false;
}

// The backward pass over padded copies; the copies of the output gradient's rows serve both gradients.
int run_bwd_padded(const GmsArgs &d, const Plan *p, const WgradArgs &w, int c_in, int c_out, bool *done) {
  const size_t esz = elem_size(d.dtype);
  const size_t in_bytes = (size_t)w.n_in * c_in * esz, gout_bytes = (size_t)w.n_out * c_out * esz,
               w_bytes = (size_t)w.k_vol * c_in * c_out * esz;
  *done = workspaces_fit(d.stream, {{kSlotPadIn, in_bytes}, {kSlotPadOut, gout_bytes}, {kSlotPadWeights, w_bytes},
                                    {kSlotPadResult, in_bytes}, {1, (size_t)w.k_vol * c_in * c_out * sizeof(float)}});
  if (!*done) return FGMS_OK;
  GmsArgs pd = d;
  WgradArgs pw = w;
  pd.c_in = pw.c_in = c_in;
  pd.c_out = pw.c_out = c_out;
  pw.crop_in = w.c_in;
  pw.crop_out = w.c_out;
  void *in = nullptr, *gout = nullptr, *weights = nullptr, *gin = nullptr;
  hipStream_t s = d.stream;
  int rc;
  PadBatch pads{};
  if ((rc = workspace_get(s, kSlotPadWeights, w_bytes, &weights))) return rc;
  pads.add(d.w, weights, (size_t)d.k_vol, d.c_in, c_in, d.c_out, c_out, (int)esz);
  pd.w = weights;
  if (c_out != d.c_out || reinterpret_cast<uintptr_t>(d.src) % 16) {
    if ((rc = workspace_get(s, kSlotPadOut, gout_bytes, &gout))) return rc;
    pads.add(d.src, gout, (size_t)w.n_out, 1, 1, d.c_out, c_out, (int)esz);
    pd.src = pw.gout = gout;
  }
  if (c_in != d.c_in || reinterpret_cast<uintptr_t>(w.in) % 16) {
    if ((rc = workspace_get(s, kSlotPadIn, in_bytes, &in))) return rc;
    pads.add(w.in, in, (size_t)w.n_in, 1, 1, d.c_in, c_in, (int)esz);
    pw.in = in;
  }
  const bool crop_result = c_in != d.c_in || reinterpret_cast<uintptr_t>(d.dst) % 16;
  if (crop_result) {
    if ((rc = workspace_get(s, kSlotPadResult, in_bytes, &gin))) return rc;
    pd.dst = gin;
    pd.overwrite = true;
  }
  if ((rc = launch_pad(pads, d.dtype, s))) return rc;
  if ((rc = run_bwd(pd, p, pw))) return rc;
  return crop_result ? launch_crop(gin, d.dst, (size_t)w.n_in, d.c_in, c_in, d.overwrite, d.dtype, s) : FGMS_OK;
}

int mid_of(int k_vol) { return (k_vol % 2 == 1) ? k_vol / 2 : 0; }

GmsArgs fwd_args(const void *in, const void *w, void *out, const int32_t *kpos,
                 const int32_t *imap, const int32_t *omap, int64_t n_in, int64_t n_out, int c_in,
                 int c_out, int k_vol, int64_t n_pairs, int dtype, hipStream_t s) {
  GmsArgs a{};
  a.src = in; a.w = w; a.dst = out; a.kpos = kpos; a.gmap = imap; a.smap = omap;
  a.n_src = n_in; a.n_dst = n_out; a.c_in = c_in; a.c_out = c_out; a.k_vol = k_vol;
  a.n_pairs = n_pairs; a.transpose_w = false; a.dense_k = -1; a.n_dense = 0; a.dtype = dtype;
  a.stream = s;
  return a;
}

int check_mid(int separate_mid, int64_t n_in, int64_t n_out) {
  if (separate_mid && n_in != n_out) {
    set_error("separate_mid needs n_in == n_out (got %lld, %lld)", (long long)n_in, (long long)n_out);
    return FGMS_E_INVALID;
  }
  return FGMS_OK;
}

}  // namespace
}  // namespace fgms

using namespace fgms;

// A fingerprint check of the plan that none of the call's launches carried as a side job goes
// out as a launch of its own when the entry point returns.
namespace {
struct CheckFlush {
  const Plan *p;
  hipStream_t s;
  ~CheckFlush() { if (p) (void)plan_flush_check(p, s); }
};

// One or both gradients, added to what the tensors hold or written over it.
int backward(const void *out_feats_grad, const void *in_feats, const void *kernel, void *in_feats_grad,
             void *kernel_grad, const int32_t *kpos, const int32_t *in_map, const int32_t *out_map, int arch80,
             int64_t n_in, int64_t n_out, int c_in, int c_out, int k_vol, int64_t n_pairs, int dtype,
             fgms_plan_t *plan, hipStream_t stream, bool want_in, bool want_kernel, bool overwrite) {
  int rc;
  if (want_in && (rc = check_common(out_feats_grad, kernel, in_feats_grad, kpos, in_map, out_map, n_in, n_out, c_in, c_out,
                                    k_vol, n_pairs, dtype)))
    return rc;
  if (want_kernel && (rc = check_common(in_feats, out_feats_grad, kernel_grad, kpos, in_map, out_map, n_in, n_out, c_in,
                                        c_out, k_vol, n_pairs, dtype)))
    return rc;
  const Plan *p = plan_resolve(plan, stream, &rc);
  CheckFlush flush{p, stream};
  if (rc) return rc;
  GmsArgs d{};
  d.src = out_feats_grad; d.w = kernel; d.dst = in_feats_grad; d.kpos = kpos;
  d.gmap = out_map; d.smap = in_map;   // roles swap, as at backend/spconv.cu:460,559
  d.n_src = n_out; d.n_dst = n_in; d.c_in = c_in; d.c_out = c_out; d.k_vol = k_vol;
  d.n_pairs = n_pairs; d.transpose_w = true; d.dense_k = -1; d.n_dense = 0; d.dtype = dtype;
  d.stream = stream;
  d.reduced = arch80 != 0 && dtype == FGMS_F32;     // (the reference's backward is tf32 whenever the tensors are fp32)
  d.overwrite = overwrite;
  WgradArgs w{};
  w.in = in_feats; w.gout = out_feats_grad; w.gw = kernel_grad; w.kpos = kpos;
  w.imap = in_map; w.omap = out_map; w.n_in = n_in; w.n_out = n_out; w.c_in = c_in;
  w.c_out = c_out; w.k_vol = k_vol; w.n_pairs = n_pairs; w.dtype = dtype;
  w.stream = stream;
  w.plan = p;
  w.reduced = d.reduced;
  w.overwrite = overwrite;
  if (!want_kernel) return want_in ? run_gms(d, p) : FGMS_OK;
  if (!want_in) return run_wgrad(w);
  // (a weight gradient of its own: 64 x 64 over 20 k scattered voxels 60 us, 128 x 128 66; half of it vanishes in the other's
  // grid.  Next to masked tiles more: on its own it needs padded copies.  48 x 48 over 20 k: masked tiles 60 us, copies and pair view 104.)
  if (dtype != FGMS_F16)
    d.beside_us = (c_in % 32 || c_out % 32 ? 0.8 : 0.5) * (d.reduced ? 0.75 : 1) *
                  (25 + 1e-3 * (double)n_out + 18e-6 * pairs_of(d, p) * (up_to_32(c_in) / 32) * (up_to_32(c_out) / 32));
  int pi, po;
  if (takes_ragged(d, p) && masked_bwd_pays(d, p, w)) {
    bool done = false;
    plan_touch(p, stream);
    rc = launch_ragged_bwd(d, p, w, &done);
    if (rc || done) return rc;
  }
  if (n_pairs > 0 && padded_bwd_channels(d, p, w, &pi, &po)) {
    bool done = false;
    rc = run_bwd_padded(d, p, w, pi, po, &done);
    if (rc || done) return rc;
  }
  return run_bwd(d, p, w);
}
}  // namespace

extern "C" {

const char *fgms_version(void) { return "fgms-hip 0.1 (gfx950)"; }
const char *fgms_last_error(void) { return g_error; }
void fgms_set_kernel_policy(int policy) { g_policy = policy; }

void fgms_profile_enable(int on) { g_prof_on = on != 0; }
long long fgms_allocation_count(void) { return g_allocations.load(std::memory_order_relaxed); }

void fgms_profile_reset(void) {
  std::lock_guard<std::mutex> lock(g_prof_mutex);
  for (auto &r : g_prof) {
    (void)hipEventSynchronize(r.stop);
    (void)hipEventDestroy(r.start);
    (void)hipEventDestroy(r.stop);
  }
  g_prof.clear();
}

int fgms_profile_read(int index, char *name, int name_len, float *ms) {
  std::lock_guard<std::mutex> lock(g_prof_mutex);
  if (index < 0 || index >= (int)g_prof.size() || !ms) return FGMS_E_INVALID;
  FGMS_HIP_TRY(hipEventSynchronize(g_prof[index].stop));
  FGMS_HIP_TRY(hipEventElapsedTime(ms, g_prof[index].start, g_prof[index].stop));
  if (name && name_len > 0) {
    strncpy(name, g_prof[index].name, (size_t)name_len - 1);
    name[name_len - 1] = 0;
  }
  return FGMS_OK;
}

int fgms_fusion_fwd(const void *in_feats, const void *kernel, int sum_nnz, void *out_feats,
                    const int32_t *kpos, const int32_t *qkpos, const int32_t *in_map,
                    const int32_t *out_map, int separate_mid, int arch80, int64_t n_in,
                    int64_t n_out, int c_in, int c_out, int k_vol, int64_t n_pairs, int dtype,
                    fgms_plan_t *plan, void *stream) {
  (void)sum_nnz; (void)qkpos;
  int rc = check_common(in_feats, kernel, out_feats, kpos, in_map, out_map, n_in, n_out, c_in,
                        c_out, k_vol, n_pairs, dtype);
  if (rc) return rc;
  if ((rc = check_mid(separate_mid, n_in, n_out))) return rc;
  hipStream_t s = (hipStream_t)stream;
  GmsArgs a = fwd_args(in_feats, kernel, out_feats, kpos, in_map, out_map, n_in, n_out, c_in,
                       c_out, k_vol, n_pairs, dtype, s);
  a.reduced = arch80 != 0 && dtype == FGMS_F32;
  if (separate_mid) {
    // the centre product overwrites, as the beta = 0 GEMM of the reference
    a.centre = mid_of(k_vol) + 1;
    a.overwrite = true;
  }
  const Plan *p = plan_resolve(plan, s, &rc);
  CheckFlush flush{p, s};
  if (rc) return rc;
  return run_gms(a, p);
}

int fgms_fwd(const void *in_feats, const void *kernel, int sum_nnz, void *out_feats,
             const int32_t *kernel_nnz, const int32_t *kernel_pos, const int32_t *in_map,
             const int32_t *out_map, int separate_mid, int arch80, int64_t n_in, int64_t n_out,
             int c_in, int c_out, int k_vol, int64_t n_pairs, int dtype, fgms_plan_t *plan,
             void *stream) {
  (void)sum_nnz;
  int rc = check_common(in_feats, kernel, out_feats, kernel_pos, in_map, out_map, n_in, n_out,
                        c_in, c_out, k_vol, n_pairs, dtype);
  if (rc) return rc;
  if ((rc = check_mid(separate_mid, n_in, n_out))) return rc;
  if (!kernel_nnz) {
    set_error("kernel_nnz (host int32[k_vol]) is null");
    return FGMS_E_INVALID;
  }
  // The host-side counts bound the pair range exactly (the reference walks them
  // to slice the maps, backend/spconv.cu:307-324).
  int64_t total = 0;
  for (int k = 0; k < k_vol; ++k) {
    if (kernel_nnz[k] < 0) {
      set_error("kernel_nnz[%d] is negative", k);
      return FGMS_E_INVALID;
    }
    total += kernel_nnz[k];
  }
  if (total > n_pairs) {
    set_error("kernel_nnz sums to %lld but the maps hold %lld pairs", (long long)total,
              (long long)n_pairs);
    return FGMS_E_INVALID;
  }
  hipStream_t s = (hipStream_t)stream;
  GmsArgs a = fwd_args(in_feats, kernel, out_feats, kernel_pos, in_map, out_map, n_in, n_out,
                       c_in, c_out, k_vol, total, dtype, s);
  a.reduced = arch80 != 0 && dtype == FGMS_F32;
  const Plan *p = plan_resolve(plan, s, &rc);
  CheckFlush flush{p, s};
  if (rc) return rc;
  if (separate_mid) a.centre = mid_of(k_vol) + 1;
  return run_gms(a, p);
}

int fgms_dgrad(const void *out_feats_grad, const void *kernel, void *in_feats_grad,
               const int32_t *kpos, const int32_t *in_map, const int32_t *out_map, int64_t n_in,
               int64_t n_out, int c_in, int c_out, int k_vol, int64_t n_pairs, int dtype,
               fgms_plan_t *plan, void *stream) {
  int rc = check_common(out_feats_grad, kernel, in_feats_grad, kpos, in_map, out_map, n_in, n_out,
                        c_in, c_out, k_vol, n_pairs, dtype);
  if (rc) return rc;
  GmsArgs a{};
  a.src = out_feats_grad; a.w = kernel; a.dst = in_feats_grad; a.kpos = kpos;
  a.gmap = out_map; a.smap = in_map;   // roles swap, as at backend/spconv.cu:460,559
  a.n_src = n_out; a.n_dst = n_in; a.c_in = c_in; a.c_out = c_out; a.k_vol = k_vol;
  a.n_pairs = n_pairs; a.transpose_w = true; a.dense_k = -1; a.n_dense = 0; a.dtype = dtype;
  a.stream = (hipStream_t)stream;
  const Plan *p = plan_resolve(plan, a.stream, &rc);
  CheckFlush flush{p, a.stream};
  if (rc) return rc;
  return run_gms(a, p);
}

int fgms_wgrad(const void *in_feats, const void *out_feats_grad, void *kernel_grad,
               const int32_t *kpos, const int32_t *in_map, const int32_t *out_map, int64_t n_in,
               int64_t n_out, int c_in, int c_out, int k_vol, int64_t n_pairs, int dtype,
               fgms_plan_t *plan, void *stream) {
  int rc = check_common(in_feats, out_feats_grad, kernel_grad, kpos, in_map, out_map, n_in, n_out,
                        c_in, c_out, k_vol, n_pairs, dtype);
  if (rc) return rc;
  WgradArgs a{};
  a.in = in_feats; a.gout = out_feats_grad; a.gw = kernel_grad; a.kpos = kpos;
  a.imap = in_map; a.omap = out_map; a.n_in = n_in; a.n_out = n_out; a.c_in = c_in;
  a.c_out = c_out; a.k_vol = k_vol; a.n_pairs = n_pairs; a.dtype = dtype;
  a.stream = (hipStream_t)stream;
  a.plan = plan_resolve(plan, a.stream, &rc);
  CheckFlush flush{a.plan, a.stream};
  if (rc) return rc;
  return run_wgrad(a);
}

int fgms_wgrad_static(const void *in_feats, const void *out_feats_grad, void *kernel_grad,
                      const int32_t *kpos, const int32_t *in_map, const int32_t *out_map, int64_t n_in,
                      int64_t n_out, int c_in, int c_out, int k_vol, int64_t n_pairs, int dtype,
                      fgms_plan_t *plan, void *stream) {
  int rc = check_common(in_feats, out_feats_grad, kernel_grad, kpos, in_map, out_map, n_in, n_out,
                        c_in, c_out, k_vol, n_pairs, dtype);
  if (rc) return rc;
  WgradArgs a{};
  a.in = in_feats; a.gout = out_feats_grad; a.gw = kernel_grad; a.kpos = kpos;
  a.imap = in_map; a.omap = out_map; a.n_in = n_in; a.n_out = n_out; a.c_in = c_in;
  a.c_out = c_out; a.k_vol = k_vol; a.n_pairs = n_pairs; a.dtype = dtype;
  a.stream = (hipStream_t)stream;
  // (resolving a plan on its first use waits for the build and may allocate the pair view: this
  // entry point does neither, it takes the plan's row bands only if they are known already)
  a.plan = plan_if_resolved(plan);
  return wgrad_static(a);
}

int fgms_bwd(const void *out_feats_grad, const void *in_feats, const void *kernel, int sum_nnz,
             void *in_feats_grad, void *kernel_grad, const int32_t *kpos, const int32_t *qkpos,
             const int32_t *in_map, const int32_t *out_map, int separate_mid, int arch80,
             int64_t n_in, int64_t n_out, int c_in, int c_out, int k_vol, int64_t n_pairs,
             int dtype, fgms_plan_t *plan, void *stream) {
  (void)sum_nnz; (void)qkpos; (void)separate_mid;
  return backward(out_feats_grad, in_feats, kernel, in_feats_grad, kernel_grad, kpos, in_map, out_map, arch80, n_in,
                  n_out, c_in, c_out, k_vol, n_pairs, dtype, plan, (hipStream_t)stream, true, true, false);
}

int fgms_conv_fwd(const void *in_feats, const void *kernel, void *out_feats, const int32_t *kpos, const int32_t *in_map,
                  const int32_t *out_map, int arch80, int64_t n_in, int64_t n_out, int c_in, int c_out, int k_vol,
                  int64_t n_pairs, int dtype, fgms_plan_t *plan, void *stream) {
  int rc = check_common(in_feats, kernel, out_feats, kpos, in_map, out_map, n_in, n_out, c_in,
                        c_out, k_vol, n_pairs, dtype);
  if (rc) return rc;
  hipStream_t s = (hipStream_t)stream;
  GmsArgs a = fwd_args(in_feats, kernel, out_feats, kpos, in_map, out_map, n_in, n_out, c_in,
                       c_out, k_vol, n_pairs, dtype, s);
  a.reduced = arch80 != 0 && dtype == FGMS_F32;
  a.overwrite = true;
  const Plan *p = plan_resolve(plan, s, &rc);
  CheckFlush flush{p, s};
  if (rc) return rc;
  return run_gms(a, p);
}

int fgms_conv_bwd(const void *out_feats_grad, const void *in_feats, const void *kernel, void *in_feats_grad,
                  void *kernel_grad, const int32_t *kpos, const int32_t *in_map, const int32_t *out_map, int arch80,
                  int64_t n_in, int64_t n_out, int c_in, int c_out, int k_vol, int64_t n_pairs, int dtype,
                  fgms_plan_t *plan, void *stream) {
  return backward(out_feats_grad, in_feats, kernel, in_feats_grad, kernel_grad, kpos, in_map, out_map, arch80, n_in,
                  n_out, c_in, c_out, k_vol, n_pairs, dtype, plan, (hipStream_t)stream, in_feats_grad != nullptr,
                  kernel_grad != nullptr, true);
}

int fgms_build_kernel_map(const int32_t *in_coords, int64_t n_in, const int32_t *out_coords,
                          int64_t n_out, const int32_t *offsets, int k_vol, int stride,
                          int skip_offset, int32_t *in_map, int32_t *out_map, int64_t capacity,
                          int32_t *kernel_nnz, int32_t *kpos, int64_t *n_pairs, void *stream) {
  if (!n_pairs) {
    set_error("fgms_build_kernel_map: bad argument");
    return FGMS_E_INVALID;
  }
  fgms_map_build_t *build = nullptr;
  const int rc = fgms_build_map_begin(&build, in_coords, n_in, out_coords, n_out, offsets, k_vol, stride, skip_offset, in_map,
                                      out_map, capacity, kernel_nnz, kpos, nullptr, 0, stream);
  return rc != FGMS_OK ? rc : fgms_build_map_end(build, nullptr, n_pairs, nullptr);
}

int fgms_build_map_begin(fgms_map_build_t **build, const int32_t *in_coords, int64_t n_in, const int32_t *out_coords,
                         int64_t n_out, const int32_t *offsets, int k_vol, int stride, int skip_offset, int32_t *in_map,
                         int32_t *out_map, int64_t capacity, int32_t *kernel_nnz, int32_t *kpos, int32_t *qkpos,
                         int want_plan, void *stream) {
  if (!build || n_in < 0 || n_out < 0 || k_vol <= 0 || stride <= 0 || capacity < 0 || !offsets || !kernel_nnz ||
      !kpos || (n_in > 0 && !in_coords) || (n_out > 0 && !out_coords) ||
      (capacity > 0 && (!in_map || !out_map)) || n_in > INT32_MAX ||
      (int64_t)k_vol * n_out > INT32_MAX - 65536) {
    set_error("fgms_build_kernel_map: bad argument");
    return FGMS_E_INVALID;
  }
  return map_build_begin((MapBuild **)build, in_coords, n_in, out_coords, n_out, offsets, k_vol, stride, skip_offset, in_map,
                         out_map, capacity, kernel_nnz, kpos, qkpos, want_plan != 0, true, (hipStream_t)stream);
}

int fgms_build_map_end(fgms_map_build_t *build, int32_t *host_nnz, int64_t *n_pairs, fgms_plan_t **plan) {
  if (!build || !n_pairs) {
    set_error("fgms_build_map_end: bad argument");
    return FGMS_E_INVALID;
  }
  return map_build_end((MapBuild *)build, host_nnz, n_pairs, plan);
}

int fgms_probe_gather(const void *feats, int c_src, int dtype, int for_dgrad, fgms_plan_t *plan,
                      void *stream) {
  int prc = FGMS_OK;
  const Plan *p = plan_resolve(plan, (hipStream_t)stream, &prc);
  if (!p || !feats || c_src <= 0 || (dtype != FGMS_F16 && dtype != FGMS_F32)) {
    if (!prc) set_error("fgms_probe_gather: bad argument");
    return FGMS_E_INVALID;
  }
  plan_touch(p, (hipStream_t)stream);
  void *sink = nullptr;
  int rc = workspace_get((hipStream_t)stream, 3, 256, &sink);
  if (rc) return rc;
  return launch_gather_probe(p, feats, c_src, dtype, for_dgrad != 0, sink, (hipStream_t)stream);
}

}  // extern "C"
