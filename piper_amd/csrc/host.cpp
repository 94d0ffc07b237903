// The host path of the operators in native code: argument checks, allocation, the launch sequences of
// the C ABI and the autograd nodes.  One forward and backward of the expert region is about thirty
// launches of 2 us each on the host; with a Python call, a ctypes call and one to three tensor
// allocations in front of every one of them it was 370 us, more than the GPU needs below about a
// thousand tokens.  Here a node allocates one block of memory for what the weight gradients read, one
// for what else it saves and one for what it does not, and issues its launches back to back.
//
// Python keeps what it is the better place for: the torch.library definitions (functional.py), the
// modules, and every decision that depends on Python state.  Functions that may meet something else
// than ordinary GPU tensors (fake tensors, tracing modes) return None and leave the call to the
// dispatcher.
#include <ATen/record_function.h>
#include <c10/hip/HIPStream.h>
#include <c10/hip/HIPGuard.h>
#include <hip/hip_runtime.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/extension.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <functional>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "../../include/piper_amd.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

namespace {

// ------------------------------------------------------------------------------ small helpers
void ok(int rc, const char* name) {
  TORCH_CHECK(rc == 0, name, " failed with status ", rc, ": ", pk_status_string(rc));
}
#define PK_CALL(fn, ...) ok(fn(__VA_ARGS__), #fn)

int dtype_code(const Tensor& t) {
  if (t.scalar_type() == at::kFloat) return PK_F32;
  if (t.scalar_type() == at::kBFloat16) return PK_BF16;
  TORCH_CHECK_TYPE(false, "piper_amd kernels support float32 and bfloat16, got ", t.scalar_type());
}

void require_gpu(const Tensor& t) {
  TORCH_CHECK(t.is_cuda(), "piper_amd kernels run on the GPU only; got a tensor on ", t.device(), " (there is no CPU fallback)");
}

void same_device(const Tensor& first, std::initializer_list<const Tensor*> others) {
  for (const Tensor* t : others)
    TORCH_CHECK_VALUE(!t->defined() || t->device() == first.device(), "all tensors of a call must be on one device");
}

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
const float* fptr(const Tensor& t) { return t.defined() ? t.data_ptr<float>() : nullptr; }
Tensor contig(const Tensor& t) { return t.defined() && !t.is_contiguous() ? t.contiguous() : t; }
Tensor opt(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }
bool aligned16(const Tensor& t) { return (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0; }
bool aligned16_all(std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (t->defined() && !aligned16(*t)) return false;
  return true;
}

// The stream of the current context on t's device; pk_init runs once per device before its first
// launch, so that the launch may already sit inside a HIP graph capture.
pk_stream_t stream_of(const Tensor& t) {
  static std::atomic<uint64_t> ready{0};
  const int dev = t.get_device();
  const uint64_t bit = 1ull << (dev & 63);
  if (!(ready.load(std::memory_order_acquire) & bit)) {
    c10::hip::HIPGuard device((c10::DeviceIndex)dev);      // it prepares the current one
    PK_CALL(pk_init);
    ready.fetch_or(bit, std::memory_order_release);
  }
  return reinterpret_cast<pk_stream_t>(c10::hip::getCurrentHIPStream(dev).stream());
}

// Ordinary tensors outside every tracing or dispatch mode: the kernels may be launched directly.  (In a
// call that torch.jit.trace records only the dispatcher leaves a node behind.)
bool plain(std::initializer_list<const Tensor*> ts) {
  for (const c10::DispatchKey mode : {c10::DispatchKey::Python, c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::Tracer})
    if (c10::impl::tls_is_dispatch_key_included(mode)) return false;
  for (const Tensor* t : ts) {
    if (!t->defined()) continue;
    if (!t->is_cuda() || t->key_set().has(c10::DispatchKey::Python)) return false;
  }
  return true;
}
// The operators have a backward and no rule for other transforms: a tensor that carries a forward-mode
// tangent (it would be dropped on the way, whether or not a backward is wanted) or that is a functorch
// wrapper (it has no memory of its own) is refused.
void refuse_transforms(std::initializer_list<const Tensor*> ts, const char* what) {
  constexpr c10::DispatchKeySet wrappers({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper});
  for (const Tensor* t : ts) {
    if (!t->defined()) continue;
    TORCH_CHECK_NOT_IMPLEMENTED(!t->_fw_grad(/*level=*/0).defined(), what, " has no forward-mode derivative");
    TORCH_CHECK(!t->key_set().has_any(wrappers), what, " does not support functorch transforms");
  }
}
// A direct call under its operator's name in the profiler (the dispatcher records its own calls)
struct RecordDirect {
  std::optional<at::RecordFunction> record;
  RecordDirect(bool direct, const char* name) {
    if (!direct) return;
    record.emplace(at::RecordScope::FUNCTION);
    if (record->isActive()) record->before(name);
  }
};
bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}

// Several buffers in one allocation, each on a 256-byte boundary.
class Block {
 public:
  // returns the position of a buffer of `bytes`
  size_t add(int64_t bytes) {
    const size_t at = size_;
    size_ += ((size_t)(bytes > 0 ? bytes : 0) + 255) / 256 * 256;
    return at;
  }
  void allocate(const Tensor& like) {
    mem_ = at::empty({(int64_t)(size_ ? size_ : 256)}, like.options().dtype(at::kByte));
    base_ = static_cast<char*>(mem_.data_ptr());
  }
  // this block and another one in a single allocation: where both live equally long
  void allocate_with(Block& other, const Tensor& like) {
    const size_t mine = size_;
    size_ += other.size_;
    allocate(like);
    size_ = mine;
    other.mem_ = mem_;
    other.base_ = base_ + mine;
  }
  void adopt(Tensor mem) {
    mem_ = std::move(mem);
    base_ = static_cast<char*>(mem_.data_ptr());
  }
  void* at_(size_t pos) const { return base_ + pos; }
  int32_t* i32(size_t pos) const { return reinterpret_cast<int32_t*>(base_ + pos); }
  float* f32(size_t pos) const { return reinterpret_cast<float*>(base_ + pos); }
  const Tensor& memory() const { return mem_; }

 private:
  size_t size_ = 0;
  Tensor mem_;
  char* base_ = nullptr;
};

// ------------------------------------------------------------------------------ Python-side switches
std::atomic<bool> g_accumulate{false};       // functional.accumulate_weight_grads
std::atomic<bool> g_overlap{false};          // functional.set_overlap_wgrad
PyObject* g_queue = nullptr;                 // functional.defer_weight_grads: a WeightGradQueue or null
std::atomic<bool> g_deferring{false};

void push_deferred(std::function<void()> fn) {
  py::gil_scoped_acquire gil;
  py::handle(g_queue).attr("push")(py::cpp_function(std::move(fn)));
}
bool leaf(const Tensor& p) { return p.defined() && p.is_leaf() && p.requires_grad(); }
// The parameters of a node, kept beside its saved variables: those that are leaves, undefined in the other
// places.  What get_saved_variables() returns is for reading values only -- under saved-tensor hooks
// (checkpointing, offload) it is a new leaf without a .grad -- while postponed and accumulated weight
// gradients belong to the tensors that the caller handed in.
void keep_parameters(AutogradContext* ctx, std::initializer_list<const Tensor*> ps) {
  std::vector<Tensor> kept;
  kept.reserve(ps.size());
  for (const Tensor* p : ps) kept.push_back(leaf(*p) ? *p : Tensor());
  ctx->saved_data["parameters"] = std::move(kept);
}
variable_list parameters_of(AutogradContext* ctx) { return ctx->saved_data["parameters"].toTensorVector(); }

// A leaf whose existing .grad the kernels can add to directly.
bool accumulates_in_place(const Tensor& p) {
  if (!leaf(p)) return false;
  const Tensor& g = p.grad();
  return g.defined() && g.scalar_type() == p.scalar_type() && g.sizes() == p.sizes() && g.is_contiguous() && g.device() == p.device();
}
void add_or_set_grad(const Tensor& p, const Tensor& g) {
  Tensor& slot = const_cast<Tensor&>(p).mutable_grad();
  if (slot.defined()) {
    at::NoGradGuard no_grad;
    slot.add_(g);
  } else {
    slot = g;
  }
}

// ------------------------------------------------------------------------------ router gate backward
// d_x (fp32, may be null) and the gate weight / bias gradients of d_logits.
void gate_bwd(const float* d_logits, const void* x, int x_dtype, const Tensor& w_gate, float* d_x32, const Tensor& d_w, const Tensor& d_b,
              bool accumulate, int64_t T, int64_t H, int64_t E) {
  Tensor ws;
  if (d_w.defined()) {
    const int64_t bytes = pk_gate_bwd_workspace_bytes(T, H, E);
    if (bytes > 0) ws = at::empty({bytes}, w_gate.options().dtype(at::kByte));
  }
  PK_CALL(pk_gate_logits_bwd, d_logits, x, x_dtype, fptr(w_gate), d_x32, static_cast<float*>(ptr(d_w)),
          static_cast<float*>(ptr(d_b)), accumulate ? 1 : 0, T, H, E, ptr(ws), ws.defined() ? ws.numel() : 0, stream_of(w_gate));
}
// d_w_gate (and d_gate_bias) added to / stored as the parameters' .grad: inside the kernel, which writes
// contiguous fp32 and has one flag for both, where every .grad is such a buffer; a gradient that is
// strided, or missing for one of the two only, is added to (or set) here.
void router_weight_grads(const Tensor& p_gate, const Tensor& p_bias, const float* d_logits, const void* x, int x_dtype, const Tensor& w_gate,
                         int64_t T, int64_t H, int64_t E) {
  if (accumulates_in_place(p_gate) && (!p_bias.defined() || accumulates_in_place(p_bias))) {
    gate_bwd(d_logits, x, x_dtype, w_gate, nullptr, p_gate.grad(), p_bias.defined() ? p_bias.grad() : Tensor(), true, T, H, E);
    return;
  }
  const auto f32 = w_gate.options();
  Tensor gw = at::empty({E, H}, f32), gb = p_bias.defined() ? at::empty({E}, f32) : Tensor();
  gate_bwd(d_logits, x, x_dtype, w_gate, nullptr, gw, gb, false, T, H, E);
  add_or_set_grad(p_gate, gw);
  if (gb.defined()) add_or_set_grad(p_bias, gb);
}

// ------------------------------------------------------------------------------ the fused region
struct Shape {
  int64_t T, H, E, I, K, A;
  int dtype;
  int64_t es;
  double route_scale, eps;
  bool route_norm;
};

Shape region_shape(const Tensor& x, const Tensor& w_gate, const Tensor& bias, const Tensor& w1, const Tensor& w2, const Tensor& w3,
                   int64_t top_k, bool route_norm, double route_scale, double eps, const Tensor& residual, const Tensor& norm_w) {
  require_gpu(x);
  TORCH_CHECK_VALUE(x.dim() == 2 && w_gate.dim() == 2 && x.size(1) == w_gate.size(1), "gate_logits: x [T,H], w_gate [E,H]");
  TORCH_CHECK_VALUE(w_gate.scalar_type() == at::kFloat, "gate_logits: the router gate is kept in float32");
  TORCH_CHECK_VALUE(w1.dim() == 3 && w2.dim() == 3 && w3.dim() == 3, "expert weights must be [E,I,H], [E,H,I], [E,I,H]");
  Shape s;
  s.T = x.size(0); s.H = x.size(1); s.E = w1.size(0); s.I = w1.size(1); s.K = top_k; s.A = s.T * top_k;
  TORCH_CHECK_VALUE(w_gate.size(0) == s.E && w1.size(2) == s.H && w3.sizes() == w1.sizes() && w2.size(0) == s.E && w2.size(1) == s.H &&
                        w2.size(2) == s.I, "expert weight shapes disagree");
  TORCH_CHECK_VALUE(w1.scalar_type() == x.scalar_type() && w2.scalar_type() == x.scalar_type() && w3.scalar_type() == x.scalar_type(),
                    "expert weights and activations must share a dtype");
  TORCH_CHECK_VALUE(!bias.defined() || (bias.scalar_type() == at::kFloat && bias.dim() == 1 && bias.size(0) == s.E),
                    "gate_logits: bias must be float32 [E]");
  TORCH_CHECK_VALUE(!residual.defined() || (residual.sizes() == x.sizes() && residual.scalar_type() == x.scalar_type()),
                    "combine_fwd: residual must be [T,H] in the dtype of y");
  TORCH_CHECK_VALUE(!norm_w.defined() || (norm_w.dim() == 1 && norm_w.size(0) == s.H && norm_w.scalar_type() == x.scalar_type()),
                    "rmsnorm_fwd: x [T,H], weight [H] in the dtype of x");
  same_device(x, {&w_gate, &bias, &w1, &w2, &w3, &residual, &norm_w});
  s.dtype = dtype_code(x);
  s.es = s.dtype == PK_BF16 ? 2 : 4;
  s.route_norm = route_norm; s.route_scale = route_scale; s.eps = eps;
  return s;
}

// What a forward leaves for its backward: `rows` is read by the weight gradients as well, which may be
// postponed past the rest of the backward, `mem` by the input pass only.
struct Saved {
  Block rows, mem;
  size_t starts, perm, order, xn;                     // in rows
  size_t logits, scores, idx, inv, rstd, g, u;        // in mem
  // grads: g and u are kept, and with a norm its output and 1/rms
  Saved(const Shape& s, bool grads, bool norm) {
    const int64_t es = s.es;
    starts = rows.add((s.E + 1) * 4);
    perm = rows.add(s.A * 4);
    order = rows.add(s.E * 4);
    xn = rows.add(norm ? s.T * s.H * es : 0);
    logits = mem.add(s.T * s.E * 4);
    scores = mem.add(s.A * 4);
    idx = mem.add(s.A * 4);
    inv = mem.add(s.A * 4);
    rstd = mem.add(norm ? s.T * 4 : 0);
    g = mem.add(grads ? s.A * s.I * es : 0);
    u = mem.add(grads ? s.A * s.I * es : 0);
  }
};

// The routing step through a Python callable (a replaced ops.route_topk: somebody records or forces the
// choice): logits -> (scores, expert indices), copied to where the kernels expect them.
void route_in_python(PyObject* route, const Shape& s, const Saved& sv, const Tensor& like) {
  py::gil_scoped_acquire gil;
  const auto keep = [mem = sv.mem.memory()](void*) {};
  const auto f32 = like.options().dtype(at::kFloat);
  Tensor logits = at::from_blob(sv.mem.at_(sv.logits), {s.T, s.E}, keep, f32);
  py::tuple r = py::handle(route)(logits, s.K, s.route_norm, s.route_scale);
  at::from_blob(sv.mem.at_(sv.scores), {s.T, s.K}, keep, f32).copy_(r[0].cast<Tensor>());
  at::from_blob(sv.mem.at_(sv.idx), {s.T, s.K}, keep, f32.dtype(at::kInt)).copy_(r[1].cast<Tensor>());
}

// out = [residual +] region([norm](x)); every input contiguous
// for_backward: what is in sv outlives the call
Tensor region_forward(const Shape& s, PyObject* route, Saved& sv, bool keep_gu, bool for_backward, const Tensor& x, const Tensor& w_gate, const Tensor& bias, const Tensor& w1,
                      const Tensor& w2, const Tensor& w3, const Tensor& residual, const Tensor& norm_w) {
  Tensor out = at::empty({s.T, s.H}, x.options());
  if (for_backward) {
    sv.rows.allocate(x);
    sv.mem.allocate(x);
  } else {
    sv.rows.allocate_with(sv.mem, x);
  }
  Block tmp;
  const int64_t ws_bytes = pk_gate_route_sort_workspace_bytes(s.T, s.H, s.E, s.K);
  TORCH_CHECK(ws_bytes >= 0, "pk_gate_route_sort_workspace_bytes failed: ", pk_status_string((int)ws_bytes));
  const size_t ws = tmp.add(ws_bytes);
  const size_t h = tmp.add(s.A * s.I * s.es), y = tmp.add(s.A * s.H * s.es);
  tmp.allocate(x);
  const pk_stream_t st = stream_of(x);
  const Block &m = sv.mem, &r = sv.rows;
  int32_t *const starts = r.i32(sv.starts), *const perm = r.i32(sv.perm);
  int32_t* const order = for_backward ? r.i32(sv.order) : nullptr;      // only the weight gradient asks for it
  const void* xin = x.data_ptr();
  if (route) {
    if (norm_w.defined()) {
      PK_CALL(pk_rmsnorm_fwd, xin, s.dtype, ptr(norm_w), (float)s.eps, r.at_(sv.xn), m.f32(sv.rstd), s.T, s.H, st);
      xin = r.at_(sv.xn);
    }
    PK_CALL(pk_gate_logits, xin, s.dtype, fptr(w_gate), fptr(bias), m.f32(sv.logits), s.T, s.H, s.E, tmp.at_(ws), ws_bytes, st);
    route_in_python(route, s, sv, x);
    PK_CALL(pk_sort_by_expert, m.i32(sv.idx), s.A, s.E, nullptr, starts, perm, m.i32(sv.inv), order, tmp.at_(ws), ws_bytes, st);
  } else if (norm_w.defined()) {
    PK_CALL(pk_norm_gate_route_sort, xin, s.dtype, ptr(norm_w), (float)s.eps, r.at_(sv.xn), m.f32(sv.rstd), fptr(w_gate), fptr(bias), s.T, s.H,
            s.E, s.K, s.route_norm, (float)s.route_scale, m.f32(sv.logits), m.f32(sv.scores), m.i32(sv.idx), nullptr, starts, perm,
            m.i32(sv.inv), order, tmp.at_(ws), ws_bytes, st);
    xin = r.at_(sv.xn);
  } else {
    PK_CALL(pk_gate_route_sort, xin, s.dtype, fptr(w_gate), fptr(bias), s.T, s.H, s.E, s.K, s.route_norm, (float)s.route_scale, m.f32(sv.logits),
            m.f32(sv.scores), m.i32(sv.idx), nullptr, starts, perm, m.i32(sv.inv), order, tmp.at_(ws), ws_bytes, st);
  }
  PK_CALL(pk_grouped_swiglu_fwd, xin, perm, s.K, ptr(w1), ptr(w2), ptr(w3), starts, keep_gu ? m.at_(sv.g) : nullptr,
          keep_gu ? m.at_(sv.u) : nullptr, tmp.at_(h), tmp.at_(y), s.A, s.H, s.I, s.E, s.dtype, st);
  PK_CALL(pk_combine_fwd, tmp.at_(y), s.dtype, m.i32(sv.inv), m.f32(sv.scores), ptr(residual), ptr(out), s.T, s.H, s.K, st);
  return out;
}

// Weight-gradient kernels of the fused region with everything they read.
struct RegionWgrad {
  Shape s;
  Tensor d_out, x, rows, grads;           // owners of the memory below (x: undefined where the rows are a norm's output)
  const void *x_rows, *d_g, *d_u, *hs;    // row-major, or
  const void *d_gT, *d_uT, *hsT;          // the transposed copies
  int64_t ldt;
  const int32_t *perm, *starts, *order;
  void operator()(const Tensor& dw1, const Tensor& dw2, const Tensor& dw3, bool accumulate) const {
    const pk_stream_t st = stream_of(d_out);
    if (ldt > 0)
      PK_CALL(pk_grouped_swiglu_wgrad_scaled_t, ptr(d_out), hsT, d_gT, d_uT, ldt, x_rows, perm, s.K, starts, order, ptr(dw1), ptr(dw2),
              ptr(dw3), accumulate, s.A, s.H, s.I, s.E, s.dtype, st);
    else
      PK_CALL(pk_grouped_swiglu_wgrad_scaled, ptr(d_out), hs, d_g, d_u, x_rows, perm, s.K, starts, order, ptr(dw1), ptr(dw2), ptr(dw3),
              accumulate, s.A, s.H, s.I, s.E, s.dtype, st);
  }
};
// `wgrad` into the three parameters' .grad: inside the kernels where all three are buffers that they can
// write (contiguous, of the parameter's type), added or set here otherwise
template <typename F>
void weight_grads_into_params(const Tensor& p1, const Tensor& p2, const Tensor& p3, const F& wgrad) {
  if (accumulates_in_place(p1) && accumulates_in_place(p2) && accumulates_in_place(p3)) {
    wgrad(p1.grad(), p2.grad(), p3.grad(), true);
    return;
  }
  Tensor g1 = at::empty_like(p1, at::MemoryFormat::Contiguous), g2 = at::empty_like(p2, at::MemoryFormat::Contiguous),
         g3 = at::empty_like(p3, at::MemoryFormat::Contiguous);
  wgrad(g1, g2, g3, false);
  add_or_set_grad(p1, g1);
  add_or_set_grad(p2, g2);
  add_or_set_grad(p3, g3);
}

c10::hip::HIPStream side_stream(int dev) {
  static std::mutex mu;
  static std::vector<std::optional<c10::hip::HIPStream>> streams(64);
  std::lock_guard<std::mutex> lock(mu);
  if (!streams[dev]) streams[dev] = c10::hip::getStreamFromPool(false, dev);
  return *streams[dev];
}
// ROCm tensors call their device type CUDA, and record_stream wants a stream of that type
c10::Stream as_cuda(const c10::hip::HIPStream& s) {
  return c10::Stream(c10::Stream::UNSAFE, c10::Device(c10::DeviceType::CUDA, s.device_index()), s.id());
}
// A stream as Python hands it over: (stream_id, device_index, device_type)
typedef std::tuple<int64_t, int64_t, int64_t> StreamKey;
c10::hip::HIPStream hip_stream(const StreamKey& k) {
  return c10::hip::HIPStream(
      c10::Stream(c10::Stream::UNSAFE, c10::Device(c10::DeviceType::HIP, (c10::DeviceIndex)std::get<1>(k)), std::get<0>(k)));
}
// `with torch.cuda.stream(s)` without its Python (about ten calls on the way in and out): makes a stream,
// and its device, the current one.
class StreamScope {
 public:
  StreamScope(int64_t id, int64_t device, int64_t type) : stream_(hip_stream({id, device, type})) {}
  void enter() {
    device_ = c10::hip::current_device();
    if (device_ != stream_.device_index()) c10::hip::set_device(stream_.device_index());
    before_ = c10::hip::getCurrentHIPStream(stream_.device_index());
    c10::hip::setCurrentHIPStream(stream_);
  }
  void exit() {
    c10::hip::setCurrentHIPStream(*before_);
    if (device_ != stream_.device_index()) c10::hip::set_device(device_);
  }

 private:
  c10::hip::HIPStream stream_;
  std::optional<c10::hip::HIPStream> before_;
  c10::DeviceIndex device_ = 0;
};

// `waiter` waits for everything queued on `other` so far.  An event belongs to the device that is current
// when it is created, and only a stream of that device can record it.
void wait_stream(const c10::hip::HIPStream& waiter, const c10::hip::HIPStream& other) {
  hipEvent_t e;
  c10::hip::HIPGuard device(other.device_index());
  TORCH_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess, "hipEventCreate failed");
  bool fine = hipEventRecord(e, other.stream()) == hipSuccess;
  device.set_index(waiter.device_index());
  fine = fine && hipStreamWaitEvent(waiter.stream(), e, 0) == hipSuccess;
  (void)hipEventDestroy(e);
  TORCH_CHECK(fine, "event between two streams failed");
}

// x [T,H] -> out [T,H]; with norm_w the norm in front of the region belongs to the node and x is its
// own residual (h + moe(ffn_norm(h))): the backward then adds the residual branch's gradient inside the
// norm's backward kernel.
struct RegionFn : public torch::autograd::Function<RegionFn> {
  enum { X, W_GATE, BIAS, W1, W2, W3, RESIDUAL, NORM_W, N_TENSORS };

  // (tensors that are absent are passed as empty optionals: autograd gives them no edge)
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w_gate, const OptTensor& bias_, const Tensor& w1, const Tensor& w2,
                        const Tensor& w3, const OptTensor& residual_, const OptTensor& norm_w_, int64_t top_k, bool route_norm,
                        double route_scale, double eps, PyObject* route) {
    const Tensor bias = opt(bias_), residual = opt(residual_), norm_w = opt(norm_w_);
    const Shape s = region_shape(x, w_gate, bias, w1, w2, w3, top_k, route_norm, route_scale, eps, residual, norm_w);
    const bool norm = norm_w.defined();
    Saved sv(s, true, norm);
    const Tensor xc = contig(x);
    Tensor out = region_forward(s, route, sv, true, true, xc, contig(w_gate), contig(bias), contig(w1), contig(w2), contig(w3),
                                norm ? xc : contig(residual), contig(norm_w));
    ctx->save_for_backward({x, w_gate, bias, w1, w2, w3, norm_w, sv.rows.memory(), sv.mem.memory()});
    keep_parameters(ctx, {&w_gate, &bias, &w1, &w2, &w3});
    ctx->saved_data["k"] = top_k;
    ctx->saved_data["norm"] = route_norm;
    ctx->saved_data["scale"] = route_scale;
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["residual"] = residual.defined();
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &bias = saved[2], &norm_w = saved[6];
    const bool norm = norm_w.defined();
    const Shape s = region_shape(x, saved[1], bias, saved[3], saved[4], saved[5], ctx->saved_data["k"].toInt(), ctx->saved_data["norm"].toBool(),
                                 ctx->saved_data["scale"].toDouble(), ctx->saved_data["eps"].toDouble(), Tensor(), norm_w);
    Saved sv(s, true, norm);
    sv.rows.adopt(saved[7]);
    sv.mem.adopt(saved[8]);
    const Block &m = sv.mem, &r = sv.rows;
    bool need[N_TENSORS];
    const bool present[N_TENSORS] = {true, true, bias.defined(), true, true, true, ctx->saved_data["residual"].toBool(), norm};
    for (int i = 0, edge = 0; i < N_TENSORS; ++i) need[i] = present[i] && ctx->needs_input_grad(edge++);
    const bool need_xn = need[X] || (norm && need[NORM_W]);      // the gradient of what the router and the experts read
    const Tensor d_out = contig(grads[0]);
    const Tensor xc = contig(x), w1 = contig(saved[3]), w2 = contig(saved[4]), w3 = contig(saved[5]);
    Tensor w_gate = contig(saved[1]);
    if (!aligned16(w_gate)) w_gate = w_gate.clone();
    const void* x_rows = norm ? r.at_(sv.xn) : xc.data_ptr();
    const int32_t *perm = r.i32(sv.perm), *starts = r.i32(sv.starts);
    // what the gradients are put into where this node does it itself (undefined: not a leaf)
    const variable_list params = parameters_of(ctx);
    const Tensor &p_gate = params[0], &p_bias = params[1], &p1 = params[2], &p2 = params[3], &p3 = params[4];
    const bool any_w = need[W1] || need[W2] || need[W3], all_w = need[W1] && need[W2] && need[W3];
    // backward-input pass: the weight gradients of the experts and of the router gate are queued with the
    // tensors they need and computed by the weight pass
    const bool postpone = g_deferring.load() && all_w && need[W_GATE] && leaf(p_gate) && (!bias.defined() || leaf(p_bias)) && leaf(p1) && leaf(p2) &&
                          leaf(p3);

    // Shapes where the K-contiguous weight-gradient path pays get d_g, d_u and score*h transposed; with long
    // experts the d_x GEMM reads its A operand from the same blocks and the row-major pair is left out.
    // With few rows an expert the transposed copies are mostly padding, and d_h without them runs on smaller tiles.  d_h and the
    // weight gradients, us, with -> without, even / counts ~ 1 / sqrt(rank):
    //   128 experts 2048 x  768, 8 rows 328 -> 296 / 328 -> 290, 32 rows 340 -> 326 / 335 -> 344, 36 rows 329 -> 334 / 338 -> 359
    //   128 experts 2048 x  512, 32 rows 225 -> 228 / 256 -> 227      64 experts 1024 x 512, 32 rows 98 -> 67 / 89 -> 68
    //    64 experts 2048 x 1024, 16 rows 207 -> 209 / 216 -> 212, 32 rows 217 -> 229 / 246 -> 232, 40 rows 214 -> 239 / 251 -> 232
    //    16 experts 2048 x 1024, 40 rows  86 ->  80 /  90 ->  81       4 experts 2048 x 1024, 32 and 40 rows 59 -> 39
    // Where d_h's persistent units (128 x 256) outnumber the 256 CUs they lose less, hence the lower line.  (One expert per
    // token: the order of the sums behind the score's gradient stays, see pk_tile::launch_ragged_m.)
    const int64_t dh_units = (s.A / 128 + std::min(s.A, s.E) / 2) * ((s.I + 255) / 256);
    const bool few_rows = s.K > 1 && s.A <= (dh_units > 256 ? 32 : 40) * s.E;
    const int64_t ldt = !few_rows && pk_region_transposed_pays(s.A, s.H, s.I, s.E, s.dtype) ? pk_grouped_swiglu_transposed_ld(s.A, s.H, s.I, s.E, s.dtype) : 0;
    const bool blocks_only = ldt > 0 && pk_grouped_swiglu_dx_from_transposed_pays(s.A, s.H, s.I, s.E, s.dtype);
    // w: what the weight gradients read, t: the rest
    Block w, t;
    const int64_t ai = s.A * s.I * s.es, ait = ldt * s.I * s.es;
    const int64_t ds_ws = std::max<int64_t>(pk_region_dgrad_dh_workspace_bytes(s.A, s.I), 4);
    int64_t n_part = (s.I + 63) / 64;      // rows of partial score gradients; 0: d_scores is written
    Block& gu = ldt > 0 ? t : w;           // the row-major pair: beside transposed copies only the d_x GEMM reads it
    const size_t d_g = gu.add(blocks_only ? 0 : ai), d_u = gu.add(blocks_only ? 0 : ai), hs = w.add(ldt > 0 ? 0 : ai);
    const size_t d_gT = w.add(ait), d_uT = w.add(ait), hsT = w.add(ait), d_logits = w.add(s.T * s.E * 4);
    const size_t d_scores = t.add(ldt > 0 ? 0 : s.A * 4), part = t.add(ds_ws);
    const size_t d_xs = t.add(need_xn ? s.A * s.H * s.es : 0);
    const int64_t router_ws_bytes = norm ? pk_region_router_norm_bwd_workspace_bytes(s.T, s.H, s.E, s.dtype)
                                         : pk_region_router_bwd_workspace_bytes(s.T, s.H, s.E, s.dtype);
    const size_t router_ws = t.add(router_ws_bytes);
    const size_t d_xn = t.add(norm && need_xn ? s.T * s.H * s.es : 0);
    if (postpone) {
      w.allocate(x);
      t.allocate(x);
    } else {
      w.allocate_with(t, x);
    }
    const pk_stream_t st = stream_of(x);
    void *dg = blocks_only ? nullptr : gu.at_(d_g), *du = blocks_only ? nullptr : gu.at_(d_u);
    // the combine backward is folded into the d_h GEMM: d_out rows are gathered per routed row, the score
    // is applied in the epilogue
    if (ldt > 0)
      PK_CALL(pk_grouped_swiglu_dgrad_dh_scaled_t, ptr(d_out), perm, s.K, m.f32(sv.scores), ptr(w2), m.at_(sv.g), m.at_(sv.u), starts, dg, du,
              w.at_(d_gT), w.at_(d_uT), w.at_(hsT), ldt, nullptr, t.at_(part), ds_ws, s.A, s.H, s.I, s.E, s.dtype, st);
    else
      PK_CALL(pk_region_dgrad_dh, ptr(d_out), perm, s.K, m.f32(sv.scores), ptr(w2), m.at_(sv.g), m.at_(sv.u), starts, dg, du,
              w.at_(hs), t.f32(d_scores), &n_part, t.at_(part), ds_ws, s.A, s.H, s.I, s.E, s.dtype, st);

    const RegionWgrad wgrad{s, d_out, norm ? Tensor() : xc, r.memory(), w.memory(), x_rows, ldt > 0 ? nullptr : dg, ldt > 0 ? nullptr : du,
                            w.at_(hs), w.at_(d_gT), w.at_(d_uT), w.at_(hsT), ldt, perm, starts, r.i32(sv.order)};
    const auto input_grad = [&] {
      if (!need_xn) return;
      if (blocks_only)
        PK_CALL(pk_grouped_swiglu_dgrad_dx_t, w.at_(d_gT), w.at_(d_uT), ldt, ptr(w1), ptr(w3), starts, t.at_(d_xs), s.A, s.H, s.I, s.E, s.dtype, st);
      else if (s.K > 1)
        PK_CALL(pk_region_dgrad_dx_any_order, dg, du, ptr(w1), ptr(w3), starts, t.at_(d_xs), s.A, s.H, s.I, s.E, s.dtype, st);
      else
        PK_CALL(pk_region_dgrad_dx, dg, du, ptr(w1), ptr(w3), starts, t.at_(d_xs), s.A, s.H, s.I, s.E, s.dtype, st);
    };
    // The router's backward and the gradient of the region's input; with a norm in front its backward
    // follows and adds the residual branch's gradient.
    Tensor d_x, d_norm_w;
    const auto router_and_input = [&](const Tensor& d_wg, const Tensor& d_b) {
      if (need_xn) d_x = at::empty({s.T, s.H}, x.options());
      const float *const d_s = n_part > 0 ? nullptr : t.f32(d_scores), *const parts = t.f32(part);
      float *const dwg = static_cast<float*>(ptr(d_wg)), *const db = static_cast<float*>(ptr(d_b));
      if (!norm || !need_xn) {
        PK_CALL(pk_region_router_bwd, m.f32(sv.logits), m.i32(sv.idx), d_s, parts, n_part, m.i32(sv.inv), s.route_norm, (float)s.route_scale,
                x_rows, s.dtype, fptr(w_gate), t.at_(d_xs), need_xn ? ptr(d_x) : nullptr, dwg, db, 0, w.f32(d_logits), s.T, s.H, s.E, s.K,
                t.at_(router_ws), router_ws_bytes, st);
        return;
      }
      if (need[NORM_W]) d_norm_w = at::empty({s.H}, norm_w.options());
      PK_CALL(pk_region_router_norm_bwd, m.f32(sv.logits), m.i32(sv.idx), d_s, parts, n_part, m.i32(sv.inv), s.route_norm, (float)s.route_scale,
              x_rows, s.dtype, fptr(w_gate), t.at_(d_xs), t.at_(d_xn), dwg, db, 0, w.f32(d_logits), ptr(xc), ptr(contig(norm_w)), m.f32(sv.rstd),
              ptr(d_out), ptr(d_x), ptr(d_norm_w), s.T, s.H, s.E, s.K, t.at_(router_ws), router_ws_bytes, st);
      if (!need[X]) d_x = Tensor();
    };
    Tensor d_w1, d_w2, d_w3, d_wg, d_b;
    const Tensor d_res = !norm && need[RESIDUAL] ? d_out : Tensor();

    if (postpone) {
      push_deferred([wgrad, p1, p2, p3] { weight_grads_into_params(p1, p2, p3, wgrad); });
      input_grad();
      router_and_input(Tensor(), Tensor());
      push_deferred([s, p_gate, p_bias, w_gate, x_rows, dl = w.f32(d_logits), keep = std::array<Tensor, 3>{wgrad.x, wgrad.rows, wgrad.grads}] {
        router_weight_grads(p_gate, p_bias, dl, x_rows, s.dtype, w_gate, s.T, s.H, s.E);
      });
      return {d_x, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), d_res, d_norm_w, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
    // backward into .grad with gradients already there (a later microbatch of an iteration): the
    // weight-gradient kernels add to them in their epilogues and autograd gets nothing to add
    const bool acc = g_accumulate.load();
    const bool experts_in_place = acc && all_w && accumulates_in_place(p1) && accumulates_in_place(p2) && accumulates_in_place(p3);
    const bool gate_in_place = acc && need[W_GATE] && accumulates_in_place(p_gate) && (!bias.defined() || (need[BIAS] && leaf(p_bias)));
    const bool overlap = any_w && g_overlap.load() && !experts_in_place;
    const auto cur = c10::hip::getCurrentHIPStream(x.get_device());
    if (experts_in_place) {
      wgrad(p1.grad(), p2.grad(), p3.grad(), true);
    } else if (any_w) {
      const auto fresh = [&] {
        d_w1 = at::empty({s.E, s.I, s.H}, x.options());
        d_w2 = at::empty({s.E, s.H, s.I}, x.options());
        d_w3 = at::empty({s.E, s.I, s.H}, x.options());
        wgrad(d_w1, d_w2, d_w3, false);
      };
      if (overlap) {
        const auto side = side_stream(x.get_device());
        wait_stream(side, cur);
        c10::hip::HIPStreamGuard guard(side);
        fresh();
      } else {
        fresh();
      }
    }
    input_grad();
    if (!gate_in_place) {
      if (need[W_GATE]) d_wg = at::empty({s.E, s.H}, w_gate.options());
      if (bias.defined() && need[BIAS]) d_b = at::empty({s.E}, w_gate.options());
    }
    router_and_input(d_wg, d_b);
    if (gate_in_place) router_weight_grads(p_gate, p_bias, w.f32(d_logits), x_rows, s.dtype, w_gate, s.T, s.H, s.E);
    if (overlap) {
      const auto side = side_stream(x.get_device());
      wait_stream(cur, side);
      for (const Tensor* b : {&d_out, &xc, &r.memory(), &w.memory()}) b->record_stream(as_cuda(side));
      for (const Tensor* b : {&d_w1, &d_w2, &d_w3}) b->record_stream(as_cuda(cur));
    }
    return {d_x, d_wg, d_b, d_w1, d_w2, d_w3, d_res, d_norm_w, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// None (with `direct`): not ordinary GPU tensors, or a tracing mode is on
std::optional<Tensor> expert_region(const Tensor& x, const Tensor& w_gate, const OptTensor& bias_, const Tensor& w1, const Tensor& w2,
                                    const Tensor& w3, int64_t top_k, bool route_norm, double route_scale, const OptTensor& residual_,
                                    const OptTensor& norm_w_, double eps, const py::object& route_, bool direct) {
  PyObject* const route = route_.ptr() == Py_None ? nullptr : route_.ptr();
  const Tensor bias = opt(bias_), residual = opt(residual_), norm_w = opt(norm_w_);
  if (direct && !plain({&x, &w_gate, &bias, &w1, &w2, &w3, &residual, &norm_w})) return std::nullopt;
  refuse_transforms({&x, &w_gate, &bias, &w1, &w2, &w3, &residual, &norm_w}, "expert_region");
  const RecordDirect record(direct, "piper_amd::expert_region");
  require_gpu(x);
  c10::hip::HIPGuard device(x.device().index());
  if (wants_grad({&x, &w_gate, &bias, &w1, &w2, &w3, &residual, &norm_w}))
    return RegionFn::apply(x, w_gate, bias_, w1, w2, w3, residual_, norm_w_, top_k, route_norm, route_scale, eps, route);
  const Shape s = region_shape(x, w_gate, bias, w1, w2, w3, top_k, route_norm, route_scale, eps, residual, norm_w);
  const Tensor xc = contig(x), w1c = contig(w1), w2c = contig(w2), w3c = contig(w3);
  const Tensor gc = contig(w_gate), bc = contig(bias), rc = norm_w.defined() ? xc : contig(residual), nc = contig(norm_w);
  // a decode step: three launches of its own, nothing sorted
  const int64_t decode_ws = route || !pk_region_decode_pays(s.T, s.H, s.E, s.I, s.K) ? 0 : pk_region_decode_workspace_bytes(s.T, s.H, s.E, s.I, s.K, s.dtype);
  if (decode_ws > 0 && aligned16_all({&xc, &gc, &bc, &w1c, &w2c, &w3c, &rc, &nc})) {
    Tensor out = at::empty({s.T, s.H}, x.options());
    const Tensor ws = at::empty({decode_ws}, x.options().dtype(at::kByte));
    PK_CALL(pk_region_decode, ptr(xc), s.dtype, ptr(nc), (float)s.eps, fptr(gc), fptr(bc), ptr(w1c), ptr(w2c), ptr(w3c), s.route_norm,
            (float)s.route_scale, ptr(rc), ptr(out), s.T, s.H, s.E, s.I, s.K, ptr(ws), decode_ws, stream_of(x));
    return out;
  }
  // without a backward the pre-activations need not be written, except by the any-width kernels
  const int64_t piece = 16 / s.es;
  const bool keep_gu = s.H % piece != 0 || s.I % piece != 0 || !aligned16(xc) || !aligned16(w1c) || !aligned16(w2c) || !aligned16(w3c);
  Saved sv(s, keep_gu, norm_w.defined());
  return region_forward(s, route, sv, keep_gu, false, xc, gc, bc, w1c, w2c, w3c, rc, nc);
}

// ------------------------------------------------------------------------------ RMSNorm
struct NormFn : public torch::autograd::Function<NormFn> {
  static Tensor run(const Tensor& x, const Tensor& w, double eps, const Tensor& rstd) {
    TORCH_CHECK_VALUE(x.dim() == 2 && w.dim() == 1 && w.size(0) == x.size(1) && w.scalar_type() == x.scalar_type(),
                      "rmsnorm_fwd: x [T,H], weight [H] in the dtype of x");
    const Tensor xc = contig(x);
    Tensor y = at::empty({x.size(0), x.size(1)}, x.options());
    PK_CALL(pk_rmsnorm_fwd, ptr(xc), dtype_code(x), ptr(contig(w)), (float)eps, ptr(y), static_cast<float*>(ptr(rstd)), x.size(0), x.size(1),
            stream_of(x));
    return y;
  }
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, double eps) {
    require_gpu(x);
    Tensor rstd = at::empty({x.size(0)}, x.options().dtype(at::kFloat));
    Tensor y = run(x, w, eps, rstd);
    ctx->save_for_backward({x, w, rstd});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list sv = ctx->get_saved_variables();
    const Tensor x = contig(sv[0]), w = contig(sv[1]), d_y = contig(grads[0]);
    const int64_t T = x.size(0), H = x.size(1);
    Tensor d_x = at::empty_like(x), d_w, ws;
    if (ctx->needs_input_grad(1)) {
      d_w = at::empty_like(w);
      ws = at::empty({pk_rmsnorm_bwd_workspace_bytes(T, H)}, x.options().dtype(at::kByte));
    }
    PK_CALL(pk_rmsnorm_bwd, ptr(d_y), ptr(x), dtype_code(x), ptr(w), fptr(sv[2]), nullptr, ptr(d_x), ptr(d_w), 0, T, H, ptr(ws),
            ws.defined() ? ws.numel() : 0, stream_of(x));
    if (!ctx->needs_input_grad(0)) d_x = Tensor();
    return {d_x, d_w, Tensor()};
  }
};
std::optional<Tensor> rmsnorm(const Tensor& x, const Tensor& w, double eps, bool direct) {
  if (direct && !plain({&x, &w})) return std::nullopt;
  refuse_transforms({&x, &w}, "rmsnorm");
  const RecordDirect record(direct, "piper_amd::rmsnorm");
  require_gpu(x);
  same_device(x, {&w});
  c10::hip::HIPGuard device(x.device().index());
  return wants_grad({&x, &w}) ? NormFn::apply(x, w, eps) : NormFn::run(x, w, eps, Tensor());
}

// ------------------------------------------------------------------------------ piecewise operators
// (counts [E], starts [E+1], perm [A], inv_perm [A]) of the stable counting sort of top_idx
std::vector<Tensor> sort_by_expert(const Tensor& top_idx, int64_t E) {
  require_gpu(top_idx);
  TORCH_CHECK_VALUE(top_idx.scalar_type() == at::kInt, "sort_by_expert: top_idx must be int32");
  c10::hip::HIPGuard device(top_idx.device().index());
  const Tensor flat = contig(top_idx);
  const int64_t A = flat.numel(), ws_bytes = pk_sort_workspace_bytes(A, E);
  TORCH_CHECK(ws_bytes >= 0, "pk_sort_workspace_bytes failed: ", pk_status_string((int)ws_bytes));
  const auto i32 = flat.options();
  Tensor counts = at::empty({E}, i32), starts = at::empty({E + 1}, i32), perm = at::empty({A}, i32), inv = at::empty({A}, i32);
  Tensor ws = at::empty({std::max<int64_t>(ws_bytes, 4)}, i32.dtype(at::kByte));
  PK_CALL(pk_sort_by_expert, flat.data_ptr<int32_t>(), A, E, counts.data_ptr<int32_t>(), starts.data_ptr<int32_t>(), perm.data_ptr<int32_t>(),
          inv.data_ptr<int32_t>(), nullptr, ptr(ws), ws.numel(), stream_of(flat));
  return {counts, starts, perm, inv};
}

struct RouterFn : public torch::autograd::Function<RouterFn> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& w_gate, const OptTensor& bias_, int64_t top_k, bool route_norm,
                               double route_scale, PyObject* route) {
    require_gpu(x);
    const Tensor bias = opt(bias_);
    TORCH_CHECK_VALUE(x.dim() == 2 && w_gate.dim() == 2 && x.size(1) == w_gate.size(1), "gate_logits: x [T,H], w_gate [E,H]");
    TORCH_CHECK_VALUE(w_gate.scalar_type() == at::kFloat, "gate_logits: the router gate is kept in float32");
    const int64_t T = x.size(0), H = x.size(1), E = w_gate.size(0);
    TORCH_CHECK_VALUE(!bias.defined() || (bias.scalar_type() == at::kFloat && bias.dim() == 1 && bias.size(0) == E),
                      "gate_logits: bias must be float32 [E]");
    const auto f32 = x.options().dtype(at::kFloat);
    Tensor logits = at::empty({T, E}, f32), scores = at::empty({T, top_k}, f32), idx = at::empty({T, top_k}, f32.dtype(at::kInt));
    const int64_t ws_bytes = pk_gate_workspace_bytes(T, H, E);
    Tensor ws = ws_bytes > 0 ? at::empty({ws_bytes}, f32.dtype(at::kByte)) : Tensor();
    const pk_stream_t st = stream_of(x);
    const Tensor xc = contig(x), wc = contig(w_gate), bc = contig(bias);
    const int64_t bytes = ws.defined() ? ws_bytes : 0;
    if (route) {
      PK_CALL(pk_gate_logits, ptr(xc), dtype_code(x), fptr(wc), fptr(bc), logits.data_ptr<float>(), T, H, E, ptr(ws), bytes, st);
      py::gil_scoped_acquire gil;
      py::tuple r = py::handle(route)(logits, top_k, route_norm, route_scale);
      scores.copy_(r[0].cast<Tensor>());
      idx.copy_(r[1].cast<Tensor>());
    } else {
      PK_CALL(pk_gate_route, ptr(xc), dtype_code(x), fptr(wc), fptr(bc), T, H, E, top_k, route_norm, (float)route_scale, logits.data_ptr<float>(),
              scores.data_ptr<float>(), idx.data_ptr<int32_t>(), ptr(ws), bytes, st);
    }
    ctx->save_for_backward({x, w_gate, bias, logits, idx});
    ctx->saved_data["norm"] = route_norm;
    ctx->saved_data["scale"] = route_scale;
    ctx->mark_non_differentiable({idx});
    return {scores, idx};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list sv = ctx->get_saved_variables();
    const Tensor x = contig(sv[0]), w_gate = contig(sv[1]), logits = sv[3], idx = sv[4];
    const int64_t T = x.size(0), H = x.size(1), E = w_gate.size(0), K = idx.size(1);
    Tensor d_s = grads[0].defined() ? contig(grads[0]).to(at::kFloat) : at::zeros({T, K}, logits.options());
    Tensor d_logits = at::empty_like(logits);
    PK_CALL(pk_route_topk_bwd, fptr(logits), idx.data_ptr<int32_t>(), fptr(d_s), T, E, K, ctx->saved_data["norm"].toBool(),
            (float)ctx->saved_data["scale"].toDouble(), d_logits.data_ptr<float>(), stream_of(x));
    Tensor d_x32, d_w, d_b;
    if (ctx->needs_input_grad(0)) d_x32 = at::empty({T, H}, logits.options());
    if (ctx->needs_input_grad(1)) d_w = at::empty({E, H}, logits.options());
    if (sv[2].defined() && ctx->needs_input_grad(2)) d_b = at::empty({E}, logits.options());
    gate_bwd(fptr(d_logits), ptr(x), dtype_code(x), w_gate, static_cast<float*>(ptr(d_x32)), d_w, d_b, false, T, H, E);
    return {d_x32.defined() ? d_x32.to(x.scalar_type()) : Tensor(), d_w, d_b, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};
std::pair<Tensor, Tensor> router(const Tensor& x, const Tensor& w_gate, const OptTensor& bias, int64_t top_k, bool route_norm, double route_scale,
                                 const py::object& route) {
  const Tensor b = opt(bias);
  refuse_transforms({&x, &w_gate, &b}, "router");
  require_gpu(x);
  same_device(x, {&w_gate, &b});
  c10::hip::HIPGuard device(x.device().index());
  auto r = RouterFn::apply(x, w_gate, bias, top_k, route_norm, route_scale, route.ptr() == Py_None ? nullptr : route.ptr());
  return {r[0], r[1]};
}

struct PermuteFn : public torch::autograd::Function<PermuteFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& perm, const Tensor& inv, int64_t top_k) {
    require_gpu(x);
    const int64_t H = x.size(1), A = perm.numel();
    Tensor routed = at::empty({A, H}, x.options());
    PK_CALL(pk_permute_fwd, ptr(contig(x)), dtype_code(x), contig(perm).data_ptr<int32_t>(), ptr(routed), A, H, top_k, stream_of(x));
    ctx->save_for_backward({inv});
    ctx->saved_data["k"] = top_k;
    return routed;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const Tensor d = contig(grads[0]), inv = ctx->get_saved_variables()[0];
    const int64_t K = ctx->saved_data["k"].toInt(), T = d.size(0) / K, H = d.size(1);
    Tensor d_x = at::empty({T, H}, d.options());
    PK_CALL(pk_permute_bwd, ptr(d), dtype_code(d), inv.data_ptr<int32_t>(), nullptr, ptr(d_x), T, H, K, stream_of(d));
    return {d_x, Tensor(), Tensor(), Tensor()};
  }
};
Tensor permute(const Tensor& x, const Tensor& perm, const Tensor& inv, int64_t top_k) {
  refuse_transforms({&x, &perm, &inv}, "permute");
  require_gpu(x);
  same_device(x, {&perm, &inv});
  TORCH_CHECK_VALUE(x.dim() == 2, "permute: x [T,H]");
  c10::hip::HIPGuard device(x.device().index());
  return PermuteFn::apply(x, perm, inv, top_k);
}

struct CombineFn : public torch::autograd::Function<CombineFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& y, const Tensor& perm, const Tensor& inv, const Tensor& scores) {
    require_gpu(y);
    const int64_t A = y.size(0), H = y.size(1), T = scores.size(0), K = scores.size(1);
    TORCH_CHECK_VALUE(A == T * K, "combine_fwd: y_sorted rows must equal T*K");
    Tensor out = at::empty({T, H}, y.options());
    PK_CALL(pk_combine_fwd, ptr(contig(y)), dtype_code(y), contig(inv).data_ptr<int32_t>(), fptr(contig(scores)), nullptr, ptr(out), T, H, K, stream_of(y));
    ctx->save_for_backward({y, perm, scores});
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list sv = ctx->get_saved_variables();
    const Tensor y = contig(sv[0]), perm = contig(sv[1]), scores = contig(sv[2]), d_out = contig(grads[0]);
    const int64_t A = y.size(0), H = y.size(1), K = scores.size(1);
    Tensor d_y = at::empty({A, H}, y.options()), d_s = at::empty({scores.size(0), K}, scores.options());
    PK_CALL(pk_combine_bwd, ptr(d_out), ptr(y), dtype_code(y), perm.data_ptr<int32_t>(), fptr(scores), ptr(d_y), d_s.data_ptr<float>(), A, H, K, stream_of(y));
    return {d_y, Tensor(), Tensor(), d_s};
  }
};
Tensor combine(const Tensor& y, const Tensor& perm, const Tensor& inv, const Tensor& scores) {
  refuse_transforms({&y, &perm, &inv, &scores}, "combine");
  require_gpu(y);
  same_device(y, {&perm, &inv, &scores});
  TORCH_CHECK_VALUE(y.dim() == 2 && scores.dim() == 2 && perm.numel() >= y.size(0) && inv.numel() >= y.size(0),
                    "combine_fwd: y_sorted [A,H], scores [T,K] and a permutation of A slots");
  c10::hip::HIPGuard device(y.device().index());
  return CombineFn::apply(y, perm, inv, scores);
}

// ------------------------------------------------------------------------------ bmm_experts
struct ExpertsFn : public torch::autograd::Function<ExpertsFn> {
  static Tensor counts_to_starts(const Tensor& counts) {
    TORCH_CHECK_VALUE(counts.scalar_type() == at::kInt || counts.scalar_type() == at::kLong, "counts must be int32 or int64");
    Tensor starts = at::empty({counts.numel() + 1}, counts.options().dtype(at::kInt));
    PK_CALL(pk_counts_to_starts, ptr(contig(counts)), counts.scalar_type() == at::kLong, counts.numel(), starts.data_ptr<int32_t>(), stream_of(counts));
    return starts;
  }
  // rows past sum(num_tokens_per_expert) belong to no expert: zeros, as in the reference
  // (qwen3_bmm_experts_patch.py:43); the kernels only write rows below starts[E]
  static void zero_tail(const Tensor& buf, const Tensor& starts) {
    PK_CALL(pk_zero_rows_from, ptr(buf), dtype_code(buf), starts.data_ptr<int32_t>() + starts.numel() - 1, buf.size(0), buf.size(1), stream_of(buf));
  }
  // y [A,H]; the pre-activations are left in gu [2,A,I], and h [A,I], which the weight gradients read as well.
  // Without a backward (gu and h null) they share one allocation.
  static Tensor run(const Tensor& w1, const Tensor& w2, const Tensor& w3, const Tensor& x, const Tensor& starts, Tensor* gu, Tensor* h) {
    TORCH_CHECK_VALUE(x.dim() == 2 && w1.dim() == 3 && x.size(1) == w1.size(2) && starts.numel() > w1.size(0),
                      "bmm_experts: x [A,H] and a row count for every expert");
    TORCH_CHECK_VALUE(w1.dim() == 3 && w2.dim() == 3 && w3.dim() == 3, "expert weights must be [E,I,H], [E,H,I], [E,I,H]");
    const int64_t E = w1.size(0), I = w1.size(1), H = w1.size(2), A = x.size(0);
    TORCH_CHECK_VALUE(w3.sizes() == w1.sizes() && w2.size(0) == E && w2.size(1) == H && w2.size(2) == I, "expert weight shapes disagree");
    TORCH_CHECK_VALUE(w1.scalar_type() == x.scalar_type() && w2.scalar_type() == x.scalar_type() && w3.scalar_type() == x.scalar_type(),
                      "expert weights and activations must share a dtype");
    const Tensor guh = at::empty({gu ? 2 : 3, A, I}, x.options());
    Tensor y = at::empty({A, H}, x.options());
    char* const g = static_cast<char*>(guh.data_ptr());
    const int64_t step = A * I * x.element_size();
    void* hp = g + 2 * step;
    if (gu) {
      *gu = guh;
      *h = at::empty({A, I}, x.options());
      hp = h->data_ptr();
    }
    PK_CALL(pk_grouped_swiglu_fwd, ptr(contig(x)), nullptr, 1, ptr(contig(w1)), ptr(contig(w2)), ptr(contig(w3)), starts.data_ptr<int32_t>(), g,
            g + step, hp, ptr(y), A, H, I, E, dtype_code(x), stream_of(x));
    zero_tail(y, starts);
    return y;
  }
  static Tensor forward(AutogradContext* ctx, const Tensor& w1, const Tensor& w2, const Tensor& w3, const Tensor& x, const Tensor& counts) {
    require_gpu(x);
    Tensor starts = counts_to_starts(counts), gu, h;
    Tensor y = run(w1, w2, w3, x, starts, &gu, &h);
    ctx->save_for_backward({w1, w2, w3, x, starts, gu, h});
    keep_parameters(ctx, {&w1, &w2, &w3});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list sv = ctx->get_saved_variables();
    const variable_list params = parameters_of(ctx);
    const Tensor &p1 = params[0], &p2 = params[1], &p3 = params[2], starts = sv[4], gu = sv[5], h = sv[6];
    const Tensor w1 = contig(sv[0]), w2 = contig(sv[1]), w3 = contig(sv[2]), x = contig(sv[3]), d_y = contig(grads[0]);
    const int64_t E = w1.size(0), I = w1.size(1), H = w1.size(2), A = x.size(0);
    const int code = dtype_code(x);
    const pk_stream_t st = stream_of(x);
    const int64_t step = A * I * x.element_size();
    char* const g = static_cast<char*>(gu.data_ptr());
    Tensor dgu = at::empty({2, A, I}, x.options()), d_x = at::empty({A, H}, x.options());
    char* const dg = static_cast<char*>(dgu.data_ptr());
    PK_CALL(pk_grouped_swiglu_dgrad, ptr(d_y), ptr(w1), ptr(w2), ptr(w3), g, g + step, starts.data_ptr<int32_t>(), dg, dg + step, ptr(d_x), A, H, I, E, code, st);
    zero_tail(d_x, starts);
    const auto wgrad = [d_y, h, dgu, x, starts, A, H, I, E, code, step](const Tensor& d1, const Tensor& d2, const Tensor& d3, bool accumulate) {
      char* const ds = static_cast<char*>(dgu.data_ptr());
      PK_CALL(pk_grouped_swiglu_wgrad, ptr(d_y), ptr(h), ds, ds + step, ptr(x), nullptr, 1, starts.data_ptr<int32_t>(), nullptr, ptr(d1),
              ptr(d2), ptr(d3), accumulate, A, H, I, E, code, stream_of(x));
    };
    Tensor d1, d2, d3;
    const bool n1 = ctx->needs_input_grad(0), n2 = ctx->needs_input_grad(1), n3 = ctx->needs_input_grad(2);
    if (n1 && n2 && n3 && g_deferring.load() && leaf(p1) && leaf(p2) && leaf(p3)) {
      push_deferred([wgrad, p1, p2, p3] { weight_grads_into_params(p1, p2, p3, wgrad); });
    } else if (n1 && n2 && n3 && g_accumulate.load() && accumulates_in_place(p1) && accumulates_in_place(p2) && accumulates_in_place(p3)) {
      wgrad(p1.grad(), p2.grad(), p3.grad(), true);
    } else if (n1 || n2 || n3) {
      d1 = at::empty({E, I, H}, x.options());
      d2 = at::empty({E, H, I}, x.options());
      d3 = at::empty({E, I, H}, x.options());
      wgrad(d1, d2, d3, false);
    }
    return {d1, d2, d3, d_x, Tensor()};
  }
};
std::optional<Tensor> bmm_experts(const Tensor& w1, const Tensor& w2, const Tensor& w3, const Tensor& x, const Tensor& counts, bool direct) {
  if (direct && !plain({&w1, &w2, &w3, &x, &counts})) return std::nullopt;
  refuse_transforms({&w1, &w2, &w3, &x, &counts}, "bmm_experts");
  const RecordDirect record(direct, "piper_artifact::bmm_experts");
  require_gpu(x);
  require_gpu(counts);
  same_device(x, {&w1, &w2, &w3, &counts});
  c10::hip::HIPGuard device(x.device().index());
  if (wants_grad({&w1, &w2, &w3, &x})) return ExpertsFn::apply(w1, w2, w3, x, counts);
  return ExpertsFn::run(w1, w2, w3, x, ExpertsFn::counts_to_starts(counts), nullptr, nullptr);
}

// ------------------------------------------------------------------------------ bucket path
// A bucket's tensors with their places, as BucketState.param_view_specs lists them:
// (parameter, element offset, element count, shape).
PyObject* spec_item(PyObject* spec, int i) {
  TORCH_CHECK_TYPE(PyTuple_Check(spec) && PyTuple_GET_SIZE(spec) > i, "param_view_specs: tuples (param, offset, numel, shape)");
  return PyTuple_GET_ITEM(spec, i);
}
const Tensor& spec_param(PyObject* spec) {
  PyObject* const p = spec_item(spec, 0);
  TORCH_CHECK_TYPE(THPVariable_Check(p), "param_view_specs: tuples (param, offset, numel, shape)");
  return THPVariable_Unpack(p);
}
int64_t spec_int(PyObject* spec, int i) { return PyLong_AsLongLong(spec_item(spec, i)); }

std::optional<c10::Stream> unpack_stream(const std::optional<StreamKey>& s) {
  if (!s) return std::nullopt;
  return c10::Stream::unpack3(std::get<0>(*s), (c10::DeviceIndex)std::get<1>(*s), (c10::DeviceType)std::get<2>(*s));
}

// The gradients of a bucket's parameters (undefined where there is none), which still have them.
struct ParamGrads {
  std::vector<const Tensor*> params;      // (the list owns them)
  std::vector<Tensor> grads;
  explicit ParamGrads(const py::list& specs) {
    params.reserve(specs.size());
    grads.reserve(specs.size());
    for (const py::handle spec : specs) {
      params.push_back(&spec_param(spec.ptr()));
      const Tensor& g = params.back()->grad();
      grads.push_back(g.defined() && g.requires_grad() ? g.detach() : g);
    }
  }
  // p.grad = None.  With a stream the memory is marked as used on it.
  void drop(const std::optional<c10::Stream>& stream) {
    for (size_t i = 0; i < grads.size(); ++i) {
      if (!grads[i].defined()) continue;
      if (stream) grads[i].record_stream(*stream);
      params[i]->mutable_grad().reset();
    }
  }
};
// flat[off : off + n] += grad.to(flat.dtype) for the bucket's gradients, one launch per gradient dtype;
// the parameters end without gradients.  Where one of them cannot be packed none is, and all are kept.
void pack_param_grads(const py::list& specs, const Tensor& flat, const std::optional<StreamKey>& stream) {
  require_gpu(flat);
  TORCH_CHECK_VALUE(flat.is_contiguous(), "bucket_pack: the flat bucket must be contiguous");
  c10::hip::HIPGuard device(flat.device().index());
  ParamGrads pg(specs);
  struct Launch {
    std::vector<const void*> ptrs;
    std::vector<int64_t> offs, nums;
  } launches[2];
  std::vector<Tensor> keep;
  for (size_t i = 0; i < pg.grads.size(); ++i) {
    if (!pg.grads[i].defined()) continue;
    Launch& l = launches[dtype_code(pg.grads[i]) == PK_F32];
    Tensor g = contig(pg.grads[i]);
    const int64_t off = spec_int(PyList_GET_ITEM(specs.ptr(), i), 1);
    TORCH_CHECK_VALUE(off >= 0 && off + g.numel() <= flat.numel(), "bucket_pack: tensor outside the bucket");
    same_device(flat, {&g});
    l.ptrs.push_back(g.data_ptr());
    l.offs.push_back(off);
    l.nums.push_back(g.numel());
    if (!g.is_same(pg.grads[i])) keep.push_back(std::move(g));
  }
  for (int f32 = 0; f32 < 2; ++f32) {
    const Launch& l = launches[f32];
    if (!l.ptrs.empty())
      PK_CALL(pk_bucket_pack, l.ptrs.data(), l.offs.data(), l.nums.data(), (int64_t)l.ptrs.size(), f32 ? PK_F32 : PK_BF16, flat.data_ptr(),
              dtype_code(flat), 1, stream_of(flat));
  }
  pg.drop(unpack_stream(stream));
}
std::vector<Tensor> hold_param_grads(const py::list& specs, const std::optional<StreamKey>& stream) {
  ParamGrads pg(specs);
  pg.drop(unpack_stream(stream));
  return std::move(pg.grads);
}
void clear_param_grads(const py::list& specs) {
  for (const py::handle spec : specs) {
    spec_param(spec.ptr()).mutable_grad().reset();
  }
}

void adamw_packed(const Tensor& master, const Tensor& exp_avg, const Tensor& exp_avg_sq, const Tensor& flat_grad, const std::vector<OptTensor>& grads,
                  const std::vector<int64_t>& offsets, const std::vector<int64_t>& numels, int64_t step, double lr, double beta1, double beta2,
                  double eps, double weight_decay, const Tensor& shadow, double grad_scale, bool zero_grad) {
  require_gpu(master);
  c10::hip::HIPGuard device(master.device().index());
  const size_t n = grads.size();
  TORCH_CHECK_VALUE(offsets.size() == n && numels.size() == n, "adamw_fused_packed: one offset and element count per tensor");
  const int64_t total = master.numel();
  for (const Tensor* t : {&master, &exp_avg, &exp_avg_sq})
    TORCH_CHECK_VALUE(t->scalar_type() == at::kFloat && t->numel() == total && t->is_contiguous(), "adamw_fused_packed: fp32 contiguous buffers of equal size");
  TORCH_CHECK_VALUE(!flat_grad.defined() || (flat_grad.scalar_type() == at::kFloat && flat_grad.numel() == total && flat_grad.is_contiguous()),
                    "adamw_fused_packed: flat_grad must match the bucket");
  TORCH_CHECK_VALUE(!shadow.defined() || (shadow.scalar_type() == at::kBFloat16 && shadow.numel() == total && shadow.is_contiguous()),
                    "adamw_fused_packed: bf16 shadow of the bucket's size");
  same_device(master, {&exp_avg, &exp_avg_sq, &flat_grad, &shadow});
  std::vector<const void*> ptrs(std::max<size_t>(n, 1), nullptr);
  std::vector<Tensor> keep;
  std::optional<at::ScalarType> dtype;
  for (size_t i = 0; i < n; ++i) {
    TORCH_CHECK_VALUE(offsets[i] >= 0 && offsets[i] + numels[i] <= total, "adamw_fused_packed: tensor outside the bucket");
    if (!grads[i].has_value() || !grads[i]->defined()) continue;
    const Tensor& g = *grads[i];
    TORCH_CHECK_VALUE(g.numel() == numels[i], "adamw_fused_packed: gradient size differs from the tensor's");
    same_device(master, {&g});
    TORCH_CHECK_VALUE(!dtype || *dtype == g.scalar_type(), "adamw_fused_packed: gradients of one call must share a dtype");
    dtype = g.scalar_type();
    if (g.is_contiguous()) {
      ptrs[i] = g.data_ptr();
    } else {
      keep.push_back(g.contiguous());
      ptrs[i] = keep.back().data_ptr();
    }
  }
  int code = PK_BF16;
  if (dtype) { code = *dtype == at::kBFloat16 ? PK_BF16 : PK_F32; TORCH_CHECK_TYPE(*dtype == at::kBFloat16 || *dtype == at::kFloat, "piper_amd kernels support float32 and bfloat16"); }
  PK_CALL(pk_adamw_fused_packed, master.data_ptr<float>(), exp_avg.data_ptr<float>(), exp_avg_sq.data_ptr<float>(), static_cast<float*>(ptr(flat_grad)),
          ptrs.data(), offsets.data(), numels.data(), (int64_t)n, code, ptr(shadow), PK_BF16, (float)lr, (float)beta1, (float)beta2, (float)eps,
          (float)weight_decay, step, (float)grad_scale, zero_grad, stream_of(master));
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  const auto nogil = py::call_guard<py::gil_scoped_release>();
  m.def("expert_region", &expert_region, nogil);
  m.def("rmsnorm", &rmsnorm, nogil);
  m.def("sort_by_expert", &sort_by_expert, nogil);
  m.def("router", &router, nogil);
  m.def("permute", &permute, nogil);
  m.def("combine", &combine, nogil);
  m.def("bmm_experts", &bmm_experts, nogil);
  m.def("pack_param_grads", &pack_param_grads);
  m.def("hold_param_grads", &hold_param_grads);
  m.def("clear_param_grads", &clear_param_grads);
  m.def("adamw_packed", [](const Tensor& master, const Tensor& exp_avg, const Tensor& exp_avg_sq, const OptTensor& flat_grad,
                           const std::vector<OptTensor>& grads, const std::vector<int64_t>& offsets, const std::vector<int64_t>& numels, int64_t step,
                           double lr, double beta1, double beta2, double eps, double weight_decay, const OptTensor& shadow, double grad_scale,
                           bool zero_grad) {
    adamw_packed(master, exp_avg, exp_avg_sq, opt(flat_grad), grads, offsets, numels, step, lr, beta1, beta2, eps, weight_decay, opt(shadow),
                 grad_scale, zero_grad);
  });
  py::class_<StreamScope>(m, "StreamScope")
      .def(py::init<int64_t, int64_t, int64_t>())
      .def("__enter__", &StreamScope::enter)
      .def("__exit__", [](StreamScope& s, const py::args&) { s.exit(); });
  // everything queued on `other` so far happens before what `waiter` gets from now on
  m.def("wait_stream", [](const StreamKey& waiter, const StreamKey& other) { wait_stream(hip_stream(waiter), hip_stream(other)); }, nogil);
  m.def("set_accumulate", [](bool on) { return g_accumulate.exchange(on); });
  m.def("set_overlap", [](bool on) { return g_overlap.exchange(on); });
  // the WeightGradQueue that backward passes hand their weight gradients to (None: they run them)
  m.def("set_queue", [](py::object q) {
    PyObject* const old = g_queue;
    g_queue = q.is_none() ? nullptr : q.inc_ref().ptr();
    g_deferring.store(g_queue != nullptr);
    Py_XDECREF(old);
  });
}
