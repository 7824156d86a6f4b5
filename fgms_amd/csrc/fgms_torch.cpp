// Python module FGMS.backend: the three functions hkeee21/FGMS exports
// (backend/pybind_cuda.cpp:7-11) with the same names and positional arguments
// (backend/spconv.h:10-49), over the C ABI of libfgms_hip.so.
//
// Differences a caller can observe, all deliberate:
//  * work is queued on torch's current HIP stream, not on stream 0
//    (the reference uses bare <<<>>> launches, backend/spconv.cu:112);
//  * a kernel-map plan is built on first use of a (kpos, in_map, out_map)
//    triple (asynchronously: the call queues the build and goes on) and kept in a
//    small cache; an entry holds references to the three tensors, so their storage
//    cannot be recycled while it is cached, and is dropped when one of them is
//    modified in place (version counter).  Writes through raw pointers do not bump
//    it, and tensors made under inference mode have none: every cache hit therefore
//    queues a fingerprint check of the lists (fgms_plan_check), and the call after
//    a rewrite raises RuntimeError and drops the plan.  A call with in_map and out_map exchanged (the
//    transposed convolution over the same pairs) shares the cached plan's tables;
//  * fgms_weights_pin(kernel) lets the library keep the re-laid copies of a weight tensor that
//    some kernels read (inference); a forward call that finds the tensor's version counter
//    moved drops them;
//  * HIP errors raise RuntimeError instead of passing silently.
//
// sparse_conv is FGMS.nn's layer as one native autograd node: a python autograd.Function around the
// functions above costs 20-40 us of host time per pass on top of the launches (a small layer's
// kernels take 10), zero-fills outputs that are then read back to be added to, and computes the
// input gradient of a first layer that nobody asked for.
#include <torch/extension.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/library.h>

#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <cstdlib>
#include <list>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <utility>
#include <vector>

#include "fgms.h"
#include "fgms_diag.h"

namespace {

// A call holds the plan it was given until its launches are queued: another thread's call may drop the
// entry from the cache meanwhile (autograd's threads run without the GIL).
using PlanRef = std::shared_ptr<fgms_plan_t>;
PlanRef own(fgms_plan_t *plan) { return PlanRef(plan, fgms_plan_destroy); }

struct CacheEntry {
  at::Tensor kpos, in_map, out_map;       // keeps the storage alive
  int64_t v_kpos, v_in, v_out;            // version counters at build time
  int64_t n_in, n_out;
  int device;
  PlanRef plan;
  bool view;                              // a transposed view of another entry's plan
  bool captured = false;                  // a call under stream capture used it
};

// Inference tensors track no version.
int64_t version_of(const at::Tensor &t) { return t.is_inference() ? 0 : (int64_t)t._version(); }

size_t g_views_made = 0;

std::mutex g_mutex;
std::list<CacheEntry> g_cache;            // most recently used first
size_t g_cache_cap = 8;
bool g_cache_enabled = true;

// Kernels recorded into a HIP graph point at a plan's tables and at the lists they were made from, and
// nothing says when the graph is gone: an entry that a capture used does not count towards the cache's
// capacity, and once it has to leave (its map was rewritten, the cache cleared) it is kept here for good.
std::list<CacheEntry> g_captured;

bool is_capturing(hipStream_t stream) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return stream && hipStreamIsCapturing(stream, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}

// Entries leave the cache by way of a list that its owner destroys after g_mutex is released: the
// last reference to a tensor may need the GIL, which another thread can hold while it waits for
// g_mutex (calls come from python with the GIL and from autograd's threads without).
struct Dropped {
  std::list<CacheEntry> entries;
};

void drop(std::list<CacheEntry>::iterator it, Dropped &dropped) {
  std::list<CacheEntry> &to = it->captured ? g_captured : dropped.entries;
  to.splice(to.begin(), g_cache, it);
}

// Leaves the `capacity` entries used last, and those of captures.
void shrink_cache(size_t capacity, Dropped &dropped) {
  size_t seen = 0;
  for (auto it = g_cache.begin(); it != g_cache.end();) {
    const auto entry = it++;
    if (!entry->captured && ++seen > capacity) drop(entry, dropped);
  }
}

void clear_cache() {
  Dropped dropped;
  std::lock_guard<std::mutex> lock(g_mutex);
  while (!g_cache.empty()) drop(g_cache.begin(), dropped);
}

void set_cache(bool enabled, int64_t capacity) {
  clear_cache();
  std::lock_guard<std::mutex> lock(g_mutex);
  g_cache_enabled = enabled;
  if (capacity > 0) g_cache_cap = (size_t)capacity;
}

size_t cache_size() {
  std::lock_guard<std::mutex> lock(g_mutex);
  return g_cache.size();
}

void check(int rc) {
  if (rc == FGMS_OK) return;
  if (rc == FGMS_E_INVALID) throw std::invalid_argument(fgms_last_error());
  throw std::runtime_error(fgms_last_error());
}

const int32_t *i32(const at::Tensor &t) { return t.numel() ? t.data_ptr<int>() : nullptr; }

int dtype_of(const at::Tensor &t) {
  if (t.scalar_type() == at::ScalarType::Half) return FGMS_F16;
  if (t.scalar_type() == at::ScalarType::Float) return FGMS_F32;
  throw std::invalid_argument("FGMS handles float32 and float16 tensors");
}

void same_dtype(const at::Tensor &a, const at::Tensor &b, const char *what) {
  if (a.scalar_type() != b.scalar_type())
    throw std::invalid_argument(std::string(what) + " must have the dtype of the features");
}

void need_contiguous_cuda(const at::Tensor &t, const char *name) {
  if (!t.is_cuda()) throw std::invalid_argument(std::string(name) + " must be a GPU tensor");
  if (!t.is_contiguous()) throw std::invalid_argument(std::string(name) + " must be contiguous");
}

// Finds or builds the plan for this map.  Returns nullptr when caching is off.
PlanRef plan_for(const at::Tensor &kpos, const at::Tensor &in_map, const at::Tensor &out_map,
                 int64_t n_in, int64_t n_out, int k_vol, hipStream_t stream) {
  Dropped dropped;
  std::lock_guard<std::mutex> lock(g_mutex);
  if (!g_cache_enabled) return nullptr;
  const int dev = in_map.get_device();
  for (auto it = g_cache.begin(); it != g_cache.end(); ++it) {
    if (it->in_map.is_same(in_map) && it->out_map.is_same(out_map) && it->kpos.is_same(kpos) &&
        it->n_in == n_in && it->n_out == n_out && it->device == dev) {
      if (it->v_in == version_of(in_map) && it->v_out == version_of(out_map) &&
          it->v_kpos == version_of(kpos)) {
        // The version counters do not see writes through raw pointers (a map builder filling a
        // pre-allocated tensor, this library's own included).  Every hit queues a check of the
        // lists against the fingerprint the plan was built with; what it finds reaches the host
        // a call later: that call drops the plan and raises.
        const int rc = fgms_plan_check(it->plan.get(), stream, 1);      // (rides along with this call's launch)
        if (rc == FGMS_E_STALE) {
          drop(it, dropped);
          throw std::runtime_error(
              "FGMS: the kernel map tensors were rewritten in place after their plan was cached "
              "(a write through data_ptr() does not bump the version counter); the previous call on this "
              "map used the old neighbour tables.  Call fgms_plan_cache_clear() after rewriting a map.");
        }
        check(rc);
        if (is_capturing(stream)) it->captured = true;
        g_cache.splice(g_cache.begin(), g_cache, it);
        return g_cache.front().plan;
      }
      drop(it, dropped);  // modified in place since the plan was built
      break;
    }
  }
  // a map first seen while the stream is being captured into a graph: no plan is built (the build
  // allocates, and its kernels would be recorded); the call records the kernels that need none
  if (is_capturing(stream)) return nullptr;
  fgms_plan_t *made = nullptr;
  bool view = false;
  // the same pairs with the sides exchanged: share that plan's tables
  for (auto it = g_cache.begin(); it != g_cache.end(); ++it) {
    if (!it->view && it->in_map.is_same(out_map) && it->out_map.is_same(in_map) && it->kpos.is_same(kpos) &&
        it->n_in == n_out && it->n_out == n_in && it->device == dev && it->v_in == version_of(out_map) &&
        it->v_out == version_of(in_map) && it->v_kpos == version_of(kpos)) {
      check(fgms_plan_transposed(&made, it->plan.get()));
      view = true;
      ++g_views_made;
      break;
    }
  }
  if (!made)
    check(fgms_plan_create(&made, i32(kpos), i32(in_map), i32(out_map), n_in, n_out, k_vol,
                           in_map.numel(), stream));
  PlanRef plan = own(made);
  g_cache.push_front(CacheEntry{kpos, in_map, out_map, version_of(kpos), version_of(in_map),
                                version_of(out_map), n_in, n_out, dev, plan, view});
  shrink_cache(g_cache_cap, dropped);
  return plan;
}

// Weight tensors whose re-laid copies the library may keep (fgms_weights_pin): the entry holds
// the tensor, so that its address cannot go to another tensor meanwhile, and its version counter;
// a forward call that finds the counter moved pins the address again, which drops the copies.
struct PinnedWeights {
  at::Tensor kernel;
  int64_t version;
};
std::vector<PinnedWeights> g_pins;

void pin_weights(const at::Tensor &kernel) {
  need_contiguous_cuda(kernel, "kernel");
  c10::hip::HIPGuardMasqueradingAsCUDA guard(kernel.device());
  std::lock_guard<std::mutex> lock(g_mutex);
  for (auto &p : g_pins)
    if (p.kernel.is_same(kernel)) {
      p.version = version_of(kernel);
      check(fgms_weights_pin(kernel.data_ptr()));
      return;
    }
  check(fgms_weights_pin(kernel.data_ptr()));
  g_pins.push_back(PinnedWeights{kernel, version_of(kernel)});
}

void unpin_weights(const at::Tensor &kernel) {
  c10::hip::HIPGuardMasqueradingAsCUDA guard(kernel.device());
  std::lock_guard<std::mutex> lock(g_mutex);
  for (size_t i = 0; i < g_pins.size(); ++i)
    if (g_pins[i].kernel.is_same(kernel)) {
      check(fgms_weights_unpin(kernel.data_ptr()));
      g_pins.erase(g_pins.begin() + i);
      return;
    }
}

// (with the device guard of the call in place)
void refresh_pin(const at::Tensor &kernel) {
  if (g_pins.empty()) return;
  std::lock_guard<std::mutex> lock(g_mutex);
  for (auto &p : g_pins)
    if (p.kernel.is_same(kernel)) {
      const int64_t v = version_of(kernel);
      if (v != p.version) {
        check(fgms_weights_pin(kernel.data_ptr()));
        p.version = v;
      }
      return;
    }
}

void check_channels(const at::Tensor &in_feats, const at::Tensor &kernel) {
  // the reference's one argument check, backend/spconv.cu:39-43
  if (in_feats.size(1) != kernel.size(1))
    throw std::invalid_argument("Input feature size and kernel size mismatch");
}

}  // namespace

void ConvolutionForwardFused(const at::Tensor in_feats, const at::Tensor kernel, const int sum_nnz,
                             at::Tensor out_feats, const at::Tensor kpos, const at::Tensor qkpos,
                             const at::Tensor in_map, const at::Tensor out_map,
                             const bool separate_mid, const bool arch80) {
  check_channels(in_feats, kernel);
  need_contiguous_cuda(in_feats, "in_feats"); need_contiguous_cuda(kernel, "kernel");
  need_contiguous_cuda(out_feats, "out_feats"); need_contiguous_cuda(kpos, "kpos");
  need_contiguous_cuda(in_map, "in_map"); need_contiguous_cuda(out_map, "out_map");
  same_dtype(in_feats, kernel, "kernel"); same_dtype(in_feats, out_feats, "out_feats");
  c10::hip::HIPGuardMasqueradingAsCUDA guard(in_feats.device());
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
  const int k_vol = (int)kernel.size(0);
  refresh_pin(kernel);
  const PlanRef plan = plan_for(kpos, in_map, out_map, in_feats.size(0), out_feats.size(0), k_vol, stream);
  check(fgms_fusion_fwd(in_feats.data_ptr(), kernel.data_ptr(), sum_nnz, out_feats.data_ptr(),
                        i32(kpos), qkpos.defined() && qkpos.numel() ? i32(qkpos) : nullptr,
                        i32(in_map), i32(out_map), separate_mid, arch80, in_feats.size(0),
                        out_feats.size(0), (int)kernel.size(1), (int)kernel.size(2), k_vol,
                        in_map.numel(), dtype_of(in_feats), plan.get(), stream));
}

void ConvolutionForward(const at::Tensor in_feats, const at::Tensor kernel, const int sum_nnz,
                        at::Tensor out_feats, const at::Tensor kernel_nnz,
                        const at::Tensor kernel_pos, const at::Tensor in_map,
                        const at::Tensor out_map, const bool separate_mid, const bool arch80) {
  check_channels(in_feats, kernel);
  need_contiguous_cuda(in_feats, "in_feats"); need_contiguous_cuda(kernel, "kernel");
  need_contiguous_cuda(out_feats, "out_feats"); need_contiguous_cuda(kernel_pos, "kernel_pos");
  need_contiguous_cuda(in_map, "in_map"); need_contiguous_cuda(out_map, "out_map");
  same_dtype(in_feats, kernel, "kernel"); same_dtype(in_feats, out_feats, "out_feats");
  if (kernel_nnz.is_cuda())
    throw std::invalid_argument("kernel_nnz must be a CPU int32 tensor (it is read on the host)");
  const int k_vol = (int)kernel.size(0);
  if (kernel_nnz.numel() < k_vol) throw std::invalid_argument("kernel_nnz is shorter than k_vol");
  at::Tensor knnz = kernel_nnz.contiguous();
  c10::hip::HIPGuardMasqueradingAsCUDA guard(in_feats.device());
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
  refresh_pin(kernel);
  const PlanRef plan = plan_for(kernel_pos, in_map, out_map, in_feats.size(0), out_feats.size(0), k_vol, stream);
  check(fgms_fwd(in_feats.data_ptr(), kernel.data_ptr(), sum_nnz, out_feats.data_ptr(),
                 knnz.data_ptr<int>(), i32(kernel_pos), i32(in_map), i32(out_map), separate_mid,
                 arch80, in_feats.size(0), out_feats.size(0), (int)kernel.size(1),
                 (int)kernel.size(2), k_vol, in_map.numel(), dtype_of(in_feats), plan.get(), stream));
}

void ConvolutionBackward(const at::Tensor out_feats_grad, const at::Tensor in_feats,
                         const at::Tensor kernel, const int sum_nnz, at::Tensor in_feats_grad,
                         at::Tensor kernel_grad, const at::Tensor kpos, const at::Tensor qkpos,
                         const at::Tensor in_map, const at::Tensor out_map,
                         const bool separate_mid, const bool arch80) {
  check_channels(in_feats, kernel);
  need_contiguous_cuda(out_feats_grad, "out_feats_grad"); need_contiguous_cuda(in_feats, "in_feats");
  need_contiguous_cuda(kernel, "kernel"); need_contiguous_cuda(in_feats_grad, "in_feats_grad");
  need_contiguous_cuda(kernel_grad, "kernel_grad"); need_contiguous_cuda(kpos, "kpos");
  need_contiguous_cuda(in_map, "in_map"); need_contiguous_cuda(out_map, "out_map");
  same_dtype(in_feats, kernel, "kernel"); same_dtype(in_feats, out_feats_grad, "out_feats_grad");
  same_dtype(in_feats, in_feats_grad, "in_feats_grad"); same_dtype(in_feats, kernel_grad, "kernel_grad");
  c10::hip::HIPGuardMasqueradingAsCUDA guard(in_feats.device());
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
  const int k_vol = (int)kernel.size(0);
  const PlanRef plan = plan_for(kpos, in_map, out_map, in_feats.size(0), out_feats_grad.size(0), k_vol, stream);
  check(fgms_bwd(out_feats_grad.data_ptr(), in_feats.data_ptr(), kernel.data_ptr(), sum_nnz,
                 in_feats_grad.data_ptr(), kernel_grad.data_ptr(), i32(kpos),
                 qkpos.defined() && qkpos.numel() ? i32(qkpos) : nullptr, i32(in_map),
                 i32(out_map), separate_mid, arch80, in_feats.size(0), out_feats_grad.size(0),
                 (int)kernel.size(1), (int)kernel.size(2), k_vol, in_map.numel(),
                 dtype_of(in_feats), plan.get(), stream));
}

namespace {

// The layer has no formula for tangents: an input that carries one is refused, as torch refuses it for a
// python autograd.Function without jvp (the kernels read the primal values alone, and an output without a
// tangent stands for a derivative of zero).
void refuse_tangent(const at::Tensor &t, const char *name) {
  TORCH_CHECK_NOT_IMPLEMENTED(!torch::autograd::isFwGradDefined(t), "sparse_conv has no forward-mode derivative, but ",
                              name, " carries a tangent");
}

// One kernel map as a layer uses it.
struct LayerMap {
  at::Tensor kpos, in_map, out_map;
  int64_t n_in, n_out;
};

at::Tensor layer_forward(const at::Tensor &feats, const at::Tensor &weight, const LayerMap &map, bool tf32) {
  const int k_vol = (int)weight.size(0);
  c10::hip::HIPGuardMasqueradingAsCUDA guard(feats.device());
  hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
  at::Tensor out = at::empty({map.n_out, weight.size(2)}, feats.options().requires_grad(false));
  refresh_pin(weight);
  const PlanRef plan = plan_for(map.kpos, map.in_map, map.out_map, map.n_in, map.n_out, k_vol, stream);
  check(fgms_conv_fwd(feats.data_ptr(), weight.data_ptr(), out.data_ptr(), i32(map.kpos), i32(map.in_map), i32(map.out_map),
                      tf32, map.n_in, map.n_out, (int)weight.size(1), (int)weight.size(2), k_vol, map.in_map.numel(),
                      dtype_of(feats), plan.get(), stream));
  return out;
}

struct SparseConvBackward final : public torch::autograd::Node {
  torch::autograd::SavedVariable feats, weight;
  std::vector<int64_t> feats_shape, weight_shape;
  at::TensorOptions options;               // dtype and device of both
  LayerMap map;
  bool tf32 = false;

  // A saved tensor as the forward pass had it.  Saved-tensor hooks (offloading, compression) may hand back
  // any tensor for it, and the kernels go by its pointer and the forward pass's sizes.
  at::Tensor unpacked(torch::autograd::SavedVariable &saved, const std::vector<int64_t> &shape, const char *name) {
    const at::Tensor t = saved.unpack(shared_from_this());
    TORCH_CHECK_VALUE(t.sizes() == at::IntArrayRef(shape) && t.dtype() == options.dtype() && t.device() == options.device(),
                      "sparse_conv: the saved ", name, " came back with another shape, dtype or device than it was saved with");
    refuse_tangent(t, name);
    return t;
  }

  torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    if (!grads[0].defined()) return {at::Tensor(), at::Tensor()};
    at::Tensor x = unpacked(feats, feats_shape, "feats"), w = unpacked(weight, weight_shape, "weight");
    refuse_tangent(grads[0], "the output gradient");
    at::NoGradGuard no_grad;
    x = x.contiguous();
    w = w.contiguous();
    at::Tensor g = grads[0].contiguous();
    same_dtype(x, g, "the output gradient");
    const int k_vol = (int)w.size(0);
    c10::hip::HIPGuardMasqueradingAsCUDA guard(x.device());
    hipStream_t stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
    at::Tensor gx, gw;
    if (task_should_compute_output(0)) gx = at::empty(x.sizes(), x.options().requires_grad(false));
    if (task_should_compute_output(1)) gw = at::empty(w.sizes(), w.options().requires_grad(false));
    const PlanRef plan = plan_for(map.kpos, map.in_map, map.out_map, map.n_in, map.n_out, k_vol, stream);
    check(fgms_conv_bwd(g.data_ptr(), x.data_ptr(), w.data_ptr(), gx.defined() ? gx.data_ptr() : nullptr,
                        gw.defined() ? gw.data_ptr() : nullptr, i32(map.kpos), i32(map.in_map), i32(map.out_map), tf32,
                        map.n_in, map.n_out, (int)w.size(1), (int)w.size(2), k_vol, map.in_map.numel(), dtype_of(x), plan.get(),
                        stream));
    return {gx, gw};
  }

  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    feats.reset_data();
    weight.reset_data();
  }

  std::string name() const override { return "SparseConvBackward"; }
};

// out[out_map[j]] += feats[in_map[j]] @ weight[k] over a zero output; differentiable in feats and weight.
at::Tensor sparse_conv_node(const at::Tensor &feats, const at::Tensor &weight, const at::Tensor &kpos, const at::Tensor &in_map,
                       const at::Tensor &out_map, int64_t n_in, int64_t n_out, bool tf32) {
  if (feats.dim() != 2 || weight.dim() != 3 || weight.size(0) != kpos.numel() - 1)
    throw std::invalid_argument("expected feats [N, Cin] and weight [K, Cin, Cout] with K = the map's offsets");
  if (feats.size(0) != n_in)
    throw std::invalid_argument("feats has " + std::to_string(feats.size(0)) + " rows, the kernel map expects " +
                                std::to_string(n_in));
  check_channels(feats, weight);
  refuse_tangent(feats, "feats");
  refuse_tangent(weight, "weight");
  const LayerMap map{kpos, in_map, out_map, n_in, n_out};
  at::Tensor x, w, out;
  {
    at::AutoGradMode no_grad(false);
    x = feats.contiguous();
    w = weight.contiguous();
    need_contiguous_cuda(x, "in_feats"); need_contiguous_cuda(w, "kernel"); need_contiguous_cuda(kpos, "kpos");
    need_contiguous_cuda(in_map, "in_map"); need_contiguous_cuda(out_map, "out_map");
    same_dtype(x, w, "kernel");
    out = layer_forward(x, w, map, tf32);
  }
  if (at::GradMode::is_enabled() && (feats.requires_grad() || weight.requires_grad())) {
    auto node = std::shared_ptr<SparseConvBackward>(new SparseConvBackward(), torch::autograd::deleteNode);
    node->set_next_edges(torch::autograd::collect_next_edges(feats, weight));
    node->feats = torch::autograd::SavedVariable(x, false);
    node->weight = torch::autograd::SavedVariable(w, false);
    node->feats_shape = x.sizes().vec();
    node->weight_shape = w.sizes().vec();
    node->options = x.options();
    node->map = map;
    node->tf32 = tf32;
    torch::autograd::set_history(out, node);
  }
  return out;
}

// Under torch.jit.trace the layer goes through torch's dispatcher, as operator fgms::sparse_conv, whose
// calls the tracer records; a plain function's result would stand in the graph as a constant.  (Only there:
// the dispatcher costs a small layer host time and gives it nothing.)
at::Tensor sparse_conv(const at::Tensor &feats, const at::Tensor &weight, const at::Tensor &kpos, const at::Tensor &in_map,
                       const at::Tensor &out_map, int64_t n_in, int64_t n_out, bool tf32) {
  if (!torch::jit::tracer::isTracing()) return sparse_conv_node(feats, weight, kpos, in_map, out_map, n_in, n_out, tf32);
  static const auto op =
      c10::Dispatcher::singleton().findSchemaOrThrow("fgms::sparse_conv", "").typed<decltype(sparse_conv)>();
  return op.call(feats, weight, kpos, in_map, out_map, n_in, n_out, tf32);
}

}  // namespace

TORCH_LIBRARY(fgms, m) {
  m.def("sparse_conv(Tensor feats, Tensor weight, Tensor kpos, Tensor in_map, Tensor out_map, int n_in, int n_out, bool tf32) -> Tensor",
        &sparse_conv_node);
}

namespace {

void need_coords(const at::Tensor &t, const char *name) {
  if (t.scalar_type() != at::ScalarType::Int || !t.is_cuda() || !t.is_contiguous() || t.dim() != 2 || t.size(1) != 3)
    throw std::invalid_argument(std::string(name) + " must be a contiguous int32 [N, 3] tensor on the GPU");
}

// A kernel map from voxel coordinates on its way: everything is queued, the sizes are not known yet.
struct MapOnItsWay {
  at::Tensor in_coords, out_coords;        // (read by the queued build: kept until its sizes are there)
  at::Tensor in_map, out_map, sizes, nnz;
  int64_t n_in = 0, n_out = 0, k_vol = 0;
  fgms_map_build_t *build = nullptr;
  hipStream_t stream = nullptr;

  MapOnItsWay(const at::Tensor &in_coords_, const at::Tensor &out_coords_, const at::Tensor &offsets, int64_t stride)
      : in_coords(in_coords_), out_coords(out_coords_) {
    need_coords(in_coords, "in_coords");
    need_coords(out_coords, "out_coords");
    if (offsets.scalar_type() != at::ScalarType::Int || offsets.is_cuda() || !offsets.is_contiguous() || offsets.dim() != 2 ||
        offsets.size(1) != 3)
      throw std::invalid_argument("offsets must be a contiguous int32 [K, 3] tensor on the host");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(in_coords.device());
    stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
    k_vol = offsets.size(0), n_in = in_coords.size(0), n_out = out_coords.size(0);
    const int64_t capacity = std::max<int64_t>(k_vol * n_out, 1);
    const auto opts = in_coords.options().requires_grad(false);
    in_map = at::empty({capacity}, opts);
    out_map = at::empty({capacity}, opts);
    sizes = at::empty({3 * k_vol + 2}, opts);         // kernel_nnz, kpos, qkpos
    nnz = at::empty({k_vol}, offsets.options());
    int *base = sizes.data_ptr<int>();
    bool want_plan;
    {
      std::lock_guard<std::mutex> lock(g_mutex);
      want_plan = g_cache_enabled;
    }
    check(fgms_build_map_begin(&build, i32(in_coords), n_in, i32(out_coords), n_out, offsets.data_ptr<int>(), (int)k_vol,
                               (int)stride, -1, in_map.data_ptr<int>(), out_map.data_ptr<int>(), k_vol * n_out, base,
                               base + k_vol, base + 2 * k_vol + 1, want_plan, stream));
  }

  ~MapOnItsWay() {
    if (!build) return;
    int64_t pairs;
    (void)fgms_build_map_end(build, nullptr, &pairs, nullptr);
  }

  // (in_map, out_map, kernel_nnz on the host, kpos, qkpos, sum of the padded sizes); its plan goes to the cache.
  std::tuple<at::Tensor, at::Tensor, at::Tensor, at::Tensor, at::Tensor, int64_t> finish() {
    fgms_map_build_t *b = std::exchange(build, nullptr);
    if (!b) throw std::runtime_error("FGMS: this kernel map has been taken already");
    c10::hip::HIPGuardMasqueradingAsCUDA guard(in_coords.device());
    int64_t pairs = 0;
    fgms_plan_t *plan = nullptr;
    check(fgms_build_map_end(b, nnz.data_ptr<int>(), &pairs, &plan));
    at::Tensor im = in_map.narrow(0, 0, pairs), om = out_map.narrow(0, 0, pairs);
    at::Tensor kpos = sizes.narrow(0, k_vol, k_vol + 1), qkpos = sizes.narrow(0, 2 * k_vol + 1, k_vol + 1);
    int64_t qsum = 0;
    for (int64_t k = 0; k < k_vol; ++k) qsum += (nnz.data_ptr<int>()[k] + 255) / 256 * 256;
    if (plan) {
      Dropped dropped;
      std::lock_guard<std::mutex> lock(g_mutex);
      g_cache.push_front(CacheEntry{kpos, im, om, version_of(kpos), version_of(im), version_of(om), n_in, n_out,
                                    (int)in_coords.get_device(), own(plan), false});
      shrink_cache(g_cache_enabled ? g_cache_cap : 0, dropped);
    }
    return {im, om, nnz, kpos, qkpos, qsum};
  }
};

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  pybind11::class_<MapOnItsWay>(m, "MapOnItsWay")
      .def(pybind11::init<const at::Tensor &, const at::Tensor &, const at::Tensor &, int64_t>(),
           pybind11::call_guard<pybind11::gil_scoped_release>())
      .def("finish", &MapOnItsWay::finish, pybind11::call_guard<pybind11::gil_scoped_release>());
  m.def("sparse_conv", &sparse_conv);
  m.def("fgms_fusion_fwd_cuda", &ConvolutionForwardFused);
  m.def("fgms_fwd_cuda", &ConvolutionForward);
  m.def("fgms_bwd_cuda", &ConvolutionBackward);
  // additions (not in the reference): plan-cache control and library identity
  m.def("fgms_plan_cache", &set_cache, pybind11::arg("enabled"), pybind11::arg("capacity") = 8);
  m.def("fgms_plan_cache_clear", &clear_cache);
  m.def("fgms_plan_cache_size", &cache_size);
  m.def("fgms_plan_cache_views", []() { std::lock_guard<std::mutex> lock(g_mutex); return g_views_made; });
  m.def("fgms_weights_pin", &pin_weights, pybind11::arg("kernel"));
  m.def("fgms_weights_unpin", &unpin_weights, pybind11::arg("kernel"));
  m.def("fgms_version", []() { return std::string(fgms_version()); });
  m.def("fgms_set_kernel_policy", &fgms_set_kernel_policy);
}
