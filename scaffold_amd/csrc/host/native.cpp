// The host path of the eager ops in C++: gates, allocations, launches through the C ABI, and the autograd nodes.
//
// A train step of the U-Net is a few hundred launches of 3 to 60 us.  Issued from Python -- argument checks, ctypes, one
// torch.autograd.Function per op, whose backward runs in the engine's thread and takes the interpreter lock -- an op cost
// 25 us of host time in the forward pass and 40 us in the backward pass, which is what a step on a volume of 64^3 or less
// took.  Here a forward op is one call into this module and a backward node runs without the interpreter.
//
// Every function either serves a call or returns None with nothing launched; the Python layer then takes the call apart
// and raises what the contract says.  Nothing is kept from call to call but sizes derived from a problem's shape.
#include <torch/extension.h>

#include <ATen/autocast_mode.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/Event.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/engine.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <string>
#include <unordered_map>

#include "../../../include/scaffold_hip.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;
constexpr auto kCL3D = at::MemoryFormat::ChannelsLast3d;
using MaybeTensor = std::optional<Tensor>;

// ---- the Python side -----------------------------------------------------------------------------------------------------
PyObject* g_kernel_error = nullptr;    // scaffold_amd._lib.ScaffoldKernelError
PyObject* g_note_device = nullptr;     // scaffold_amd._lib._note_device(device)
PyObject* g_send_early = nullptr;      // scaffold_amd.modules._send_early(batch)
PyObject* g_join_early = nullptr;      // scaffold_amd.modules._join_early(batch)

// A status code as the exception the entry points raise (the interpreter lock is taken if this thread does not hold it).
void check(int rc, const char* what) {
  if (rc == SFH_OK) return;
  const char* said = sfh_last_error();
  const std::string text = std::string(what) + ": " + (said != nullptr && *said ? said : "unknown error");
  const bool called_from_python = PyGILState_Check() != 0;
  py::gil_scoped_acquire gil;
  PyObject* cls = rc == SFH_ERR_UNSUPPORTED ? PyExc_NotImplementedError
                  : rc == SFH_ERR_INVALID || rc == SFH_ERR_WORKSPACE ? PyExc_ValueError
                  : g_kernel_error != nullptr ? g_kernel_error : PyExc_RuntimeError;
  PyErr_SetString(cls, text.c_str());
  if (called_from_python) throw py::error_already_set();
  python_error e;  // in a backward node: the engine carries it to the thread that called backward()
  e.persist();
  throw std::move(e);
}

std::atomic<uint64_t> g_devices_seen{0};

// The stream torch is issuing work to on the tensor's device; the first call per device has Python look the device over.
void* stream_of(const Tensor& t) {
  const auto index = t.device().index();
  const uint64_t bit = 1ull << (index & 63);
  if (!(g_devices_seen.load(std::memory_order_relaxed) & bit)) {
    g_devices_seen.fetch_or(bit);
    if (g_note_device != nullptr) {
      py::gil_scoped_acquire gil;
      py::reinterpret_borrow<py::function>(g_note_device)(py::cast(t.device()));
    }
  }
  return (void*)c10::hip::getCurrentHIPStream(index).stream();
}

c10::Stream stream_on(c10::Device device) { return c10::impl::VirtualGuardImpl(c10::DeviceType::CUDA).getStream(device); }

int code_of(at::ScalarType t) {
  return t == at::kBFloat16 ? SFH_BF16 : t == at::kHalf ? SFH_FP16 : t == at::kFloat ? SFH_FP32 : -1;
}

bool on_gpu(const Tensor& t) { return t.is_cuda() && t.layout() == at::kStrided; }
const void* ptr(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }
void* out_ptr(const Tensor& t) { return t.defined() ? t.mutable_data_ptr() : nullptr; }
Tensor dense(const Tensor& t) { return t.is_contiguous(kCL3D) ? t : t.contiguous(kCL3D); }
// (the backend's own factory: a pass allocates a few hundred tensors, and the dispatcher is a third of what that costs)
Tensor plain(at::IntArrayRef sizes, const Tensor& like, at::ScalarType dtype) {
  return Tensor(at::detail::empty_cuda(sizes, dtype, like.device(), std::nullopt));
}
Tensor volume(at::IntArrayRef sizes, const Tensor& like, at::ScalarType dtype) {
  return Tensor(at::detail::empty_cuda(sizes, dtype, like.device(), kCL3D));
}
Tensor bytes(size_t n, const Tensor& like) { return n == 0 ? Tensor() : plain({(int64_t)n}, like, at::kByte); }

// An int or three ints, as the Python layer has it (subclasses of int, no bool); false for any other spelling (the Python
// layer then says what is wrong with it).
bool three(py::handle h, int32_t v[3]) {
  auto one = [](PyObject* o, int32_t& to) {
    if (!PyLong_Check(o) || PyBool_Check(o)) return false;
    int overflow = 0;
    const long x = PyLong_AsLongAndOverflow(o, &overflow);
    if (overflow || x < INT32_MIN || x > INT32_MAX) return false;
    to = (int32_t)x;
    return true;
  };
  if (PyLong_Check(h.ptr())) return one(h.ptr(), v[0]) && (v[1] = v[2] = v[0], true);
  if (!PyTuple_Check(h.ptr()) && !PyList_CheckExact(h.ptr())) return false;
  if (PySequence_Fast_GET_SIZE(h.ptr()) != 3) return false;
  for (int i = 0; i < 3; ++i)
    if (!one(PySequence_Fast_GET_ITEM(h.ptr(), i), v[i])) return false;
  return true;
}

// ---- convolution problems ------------------------------------------------------------------------------------------------
// What the library says about a problem, asked once per shape and thread.
struct Sizes {
  size_t packed[2];           // bytes of the packed weight each direction reads
  size_t work[3];             // workspace bytes: forward, data gradient, weight gradient
  size_t work_bias;           // weight gradient with the bias gradient in the same pass (0: not offered)
  int32_t groups = -1, records = 0;  // GroupNorm records for the last group count asked for
};

struct ProblemKey {
  sfh_conv3d_desc d;
  int32_t code;
  bool operator==(const ProblemKey& o) const { return std::memcmp(this, &o, sizeof(ProblemKey)) == 0; }
};
static_assert(sizeof(ProblemKey) == 19 * sizeof(int32_t), "no padding in the key");
struct ProblemHash {
  size_t operator()(const ProblemKey& k) const {
    const auto* p = reinterpret_cast<const uint32_t*>(&k);
    uint64_t h = 1469598103934665603ull;
    for (size_t i = 0; i < sizeof(ProblemKey) / 4; ++i) h = (h ^ p[i]) * 1099511628211ull;
    return (size_t)(h ^ h >> 29);
  }
};

struct Problem {
  ProblemKey key;
  int32_t out[3];
  Sizes* sizes;
  const sfh_conv3d_desc* desc() const { return &key.d; }
  int32_t records(int groups) const {
    if (sizes->groups != groups) {
      sizes->records = sfh_conv3d_fwd_gn_records(&key.d, key.code, groups);
      sizes->groups = groups;
    }
    return sizes->records;
  }
};

Sizes* sizes_of(const ProblemKey& k) {
  thread_local std::unordered_map<ProblemKey, Sizes, ProblemHash> known;
  auto it = known.find(k);
  if (it == known.end()) {
    if (known.size() > 4096) known.clear();
    Sizes s;
    for (int dir = 0; dir < 2; ++dir) s.packed[dir] = sfh_conv3d_packed_weight_bytes(&k.d, k.code, dir);
    s.work[0] = sfh_conv3d_fwd_workspace_bytes(&k.d, k.code);
    s.work[1] = sfh_conv3d_dgrad_workspace_bytes(&k.d, k.code);
    s.work[2] = sfh_conv3d_wgrad_workspace_bytes(&k.d, k.code);
    s.work_bias = sfh_conv3d_wgrad_bias_workspace_bytes(&k.d, k.code);
    it = known.emplace(k, s).first;
  }
  return &it->second;
}

// Geometry of conv3d(in, w) with (N, C, D, H, W) and (Cout, Cin, kd, kh, kw) sizes. False: not a problem the library has.
bool make_problem(at::IntArrayRef in, at::IntArrayRef w, const int32_t s[3], const int32_t p[3], const int32_t d[3], int code, Problem& r) {
  if (in.size() != 5 || w.size() != 5 || code < 0) return false;
  for (auto v : in) if (v < 1 || v > INT32_MAX) return false;
  for (auto v : w) if (v < 1 || v > INT32_MAX) return false;
  for (int i = 0; i < 3; ++i) {
    if (s[i] < 1 || d[i] < 1 || p[i] < 0) return false;
    const int64_t span = in[2 + i] + 2 * (int64_t)p[i] - (int64_t)d[i] * (w[2 + i] - 1) - 1;
    if (span < 0) return false;
    r.out[i] = (int32_t)(span / s[i] + 1);
  }
  r.key.d = sfh_conv3d_desc{(int32_t)in[0], (int32_t)in[1], (int32_t)in[2], (int32_t)in[3], (int32_t)in[4], (int32_t)w[0],
                            (int32_t)w[2], (int32_t)w[3], (int32_t)w[4], s[0], s[1], s[2], p[0], p[1], p[2], d[0], d[1], d[2]};
  r.key.code = code;
  r.sizes = sizes_of(r.key);
  return true;
}

bool bias_fits(const MaybeTensor& b, const Tensor& x, int64_t channels) {
  return !b.has_value() || (b->dim() == 1 && b->size(0) == channels && b->scalar_type() == x.scalar_type() && b->device() == x.device() &&
                            b->stride(0) == 1);
}

// The gate of the forward (conv3d.is_supported), and with `all` of both gradients too (is_supported_all).  `packed`: the
// caller has made packed forms of x's dtype from w, so an fp32 master may stand in w's place (nothing else may: packed forms
// of bf16 and fp16 weights have the same size).
bool conv_gate(const Tensor& x, const Tensor& w, const MaybeTensor& bias, const int32_t s[3], const int32_t p[3], const int32_t d[3],
               bool all, Problem& prob, int64_t more_channels = 0, bool packed = false) {
  if (x.dim() != 5 || w.dim() != 5 || !on_gpu(x) || !on_gpu(w) || x.device() != w.device()) return false;
  if ((x.scalar_type() != w.scalar_type() && !(packed && w.scalar_type() == at::kFloat)) || x.size(1) + more_channels != w.size(1)) return false;
  if (!bias_fits(bias, x, w.size(0))) return false;
  const int64_t in[5] = {x.size(0), w.size(1), x.size(2), x.size(3), x.size(4)};
  if (!make_problem(in, w.sizes(), s, p, d, code_of(x.scalar_type()), prob)) return false;
  if (all)
    for (int i = 0; i < 3; ++i)
      if (s[i] != 1 || p[i] > d[i] * ((int32_t)w.size(2 + i) - 1)) return false;
  return true;
}

bool packed_fits(const Tensor& packed, size_t want, const Tensor& like) {
  return want != 0 && packed.scalar_type() == at::kByte && packed.dim() == 1 && packed.is_contiguous() && packed.device() == like.device() &&
         (size_t)packed.numel() == want;
}

struct ConvResult {
  Tensor y, partials;
  int32_t records = 0;
};

// x (and second: the channels after x's), dense channels-last, gated.
ConvResult launch_conv(const Problem& prob, const Tensor& x, const Tensor& second, const Tensor& w, const Tensor& bias, const Tensor& packed,
                       int groups) {
  c10::OptionalDeviceGuard guard(x.device());
  ConvResult r;
  r.y = volume({prob.key.d.n, prob.key.d.cout, prob.out[0], prob.out[1], prob.out[2]}, x, x.scalar_type());
  const Tensor ws = bytes(prob.sizes->work[0] - (packed.defined() ? prob.sizes->packed[0] : 0), x);
  const size_t ws_bytes = ws.defined() ? (size_t)ws.numel() : 0;
  const uint32_t flags = packed.defined() ? SFH_FLAG_WEIGHT_PACKED : 0;
  const void* wp = packed.defined() ? ptr(packed) : ptr(w);
  const int64_t* strides = packed.defined() ? nullptr : w.strides().data();
  void* st = stream_of(x);
  int rc = SFH_ERR_UNSUPPORTED;
  r.records = groups > 0 ? prob.records(groups) : 0;
  if (r.records > 0) {
    r.partials = plain({(int64_t)prob.key.d.n * r.records * groups * 4}, x, at::kFloat);
    rc = second.defined()
             ? sfh_conv3d_fwd_pair(prob.desc(), prob.key.code, ptr(x), ptr(second), (int32_t)x.size(1), wp, strides, ptr(bias), out_ptr(r.y),
                                   out_ptr(ws), ws_bytes, flags, groups, (float*)out_ptr(r.partials), (size_t)r.partials.numel() * 4, st)
             : sfh_conv3d_fwd_gn(prob.desc(), prob.key.code, ptr(x), wp, strides, ptr(bias), out_ptr(r.y), out_ptr(ws), ws_bytes, flags, groups,
                                 (float*)out_ptr(r.partials), (size_t)r.partials.numel() * 4, st);
  }
  if (rc == SFH_ERR_UNSUPPORTED) {  // no statistics asked for, or not offered: the plain launch
    r.records = 0;
    rc = second.defined() ? sfh_conv3d_fwd_pair(prob.desc(), prob.key.code, ptr(x), ptr(second), (int32_t)x.size(1), wp, strides, ptr(bias),
                                                out_ptr(r.y), out_ptr(ws), ws_bytes, flags, 0, nullptr, 0, st)
                          : sfh_conv3d_fwd(prob.desc(), prob.key.code, ptr(x), wp, strides, ptr(bias), out_ptr(r.y), out_ptr(ws), ws_bytes, flags, st);
  }
  check(rc, "conv3d_forward");
  return r;
}

// The groups whose records a module asks a convolution for. Those of a batch of 32 channels are left by walking its samples apart, sums in another
// order than the statistics pass's; a network's bits stay with that pass (a step of two samples of 44x60x75: 24 of 1560 us). The operator
// leaves them to whoever asks.
int module_groups(const Problem& prob, int64_t groups) { return prob.key.d.n > 1 && prob.key.d.cin == 32 ? 0 : (int)groups; }

// The data gradient; `first` > 0: as two tensors cut at that channel.
std::pair<Tensor, Tensor> launch_dgrad(const Problem& prob, const Tensor& gy, const Tensor& w, const Tensor& packed, int64_t first) {
  c10::OptionalDeviceGuard guard(gy.device());
  const auto& d = prob.key.d;
  const int64_t c1 = first > 0 ? first : d.cin;
  Tensor gx = volume({d.n, c1, d.in_d, d.in_h, d.in_w}, gy, gy.scalar_type()), gx2;
  if (first > 0) gx2 = volume({d.n, d.cin - first, d.in_d, d.in_h, d.in_w}, gy, gy.scalar_type());
  const Tensor ws = bytes(prob.sizes->work[1] - (packed.defined() ? prob.sizes->packed[1] : 0), gy);
  const size_t ws_bytes = ws.defined() ? (size_t)ws.numel() : 0;
  const uint32_t flags = packed.defined() ? SFH_FLAG_WEIGHT_PACKED : 0;
  const void* wp = packed.defined() ? ptr(packed) : ptr(w);
  const int64_t* strides = packed.defined() ? nullptr : w.strides().data();
  const int rc = first > 0 ? sfh_conv3d_dgrad_pair(prob.desc(), prob.key.code, ptr(gy), wp, strides, out_ptr(gx), out_ptr(gx2), (int32_t)first,
                                                   out_ptr(ws), ws_bytes, flags, stream_of(gy))
                           : sfh_conv3d_dgrad(prob.desc(), prob.key.code, ptr(gy), wp, strides, out_ptr(gx), out_ptr(ws), ws_bytes, flags, stream_of(gy));
  check(rc, "conv3d_backward_data");
  return {gx, gx2};
}

// The weight gradient in the operands' dtype or, with `fp32`, unrounded where the kernel that serves the problem has that
// form (else widened afterwards: what autocast's cast node would have done).
Tensor launch_wgrad(const Problem& prob, const Tensor& x, const Tensor& second, const Tensor& gy, bool fp32) {
  c10::OptionalDeviceGuard guard(gy.device());
  const auto& d = prob.key.d;
  const bool widen = fp32 && gy.scalar_type() != at::kFloat;
  const Tensor ws = bytes(prob.sizes->work[2], gy);
  const size_t ws_bytes = ws.defined() ? (size_t)ws.numel() : 0;
  for (int attempt = widen ? 0 : 1; attempt < 2; ++attempt) {
    Tensor gw = volume({d.cout, d.cin, d.kd, d.kh, d.kw}, gy, attempt == 0 ? at::kFloat : gy.scalar_type());
    const uint32_t flags = attempt == 0 ? SFH_FLAG_GRAD_FP32 : 0;
    const int rc = second.defined() ? sfh_conv3d_wgrad_pair(prob.desc(), prob.key.code, ptr(x), ptr(second), (int32_t)x.size(1), ptr(gy), out_ptr(gw),
                                                            out_ptr(ws), ws_bytes, flags, stream_of(gy))
                                    : sfh_conv3d_wgrad(prob.desc(), prob.key.code, ptr(x), ptr(gy), out_ptr(gw), out_ptr(ws), ws_bytes, flags, stream_of(gy));
    if (attempt == 0 && rc == SFH_ERR_UNSUPPORTED) continue;
    check(rc, "conv3d_backward_weight");
    return widen && attempt == 1 ? gw.to(at::kFloat) : gw;
  }
  return Tensor();
}

// grad_output.sum((0, 2, 3, 4)) in a fixed order
Tensor launch_bias_grad(const Tensor& gy, at::ScalarType dtype) {
  c10::OptionalDeviceGuard guard(gy.device());
  const int64_t c = gy.size(1), rows = gy.numel() / c;
  Tensor gb = plain({c}, gy, dtype);
  const Tensor ws = bytes(sfh_bias_grad_workspace_bytes(rows, (int32_t)c), gy);
  check(sfh_bias_grad(code_of(gy.scalar_type()), code_of(dtype), ptr(gy), rows, (int32_t)c, out_ptr(gb), out_ptr(ws),
                      ws.defined() ? (size_t)ws.numel() : 0, stream_of(gy)), "bias_grad");
  return gb;
}

// ---- autograd ------------------------------------------------------------------------------------------------------------
// A node whose gradients are computed by launches: under create_graph its results refuse to be differentiated again.
struct LaunchNode : public Node {
  virtual variable_list backward(variable_list& grads) = 0;
  variable_list apply(variable_list&& grads) override {
    bool twice = false;
    if (at::GradMode::is_enabled())
      for (const auto& g : grads) twice = twice || (g.defined() && g.requires_grad());
    variable_list outs;
    {
      at::AutoGradMode no_grad(false);
      outs = backward(grads);
    }
    if (!twice) return outs;
    variable_list marked;
    for (const auto& o : outs) {
      if (!o.defined()) {
        marked.push_back(o);
        continue;
      }
      auto refuse = std::make_shared<torch::autograd::DelayedError>("trying to differentiate twice a function that was marked with @once_differentiable", 1);
      marked.push_back((*refuse)({o.detach().set_requires_grad(true)})[0]);
    }
    return marked;
  }
};

template <typename N> std::shared_ptr<N> new_node() { return {new N(), torch::autograd::deleteNode}; }

// A tensor kept for the backward pass.  Saved-tensor hooks decide what comes back: save_on_cpu returns the values in the
// default layout, whatever the layout was.  The kernels read plain pointers, so the layout they take is restored here, and
// anything that is not the tensor that was kept (a hook that left it on the host, say) is refused.
struct Kept {
  SavedVariable saved;
  c10::DimVector sizes;
  at::ScalarType dtype = at::kFloat;
  c10::Device device{c10::DeviceType::CPU};
  void keep(const Tensor& t) {
    saved = SavedVariable(t, false);
    if (!t.defined()) return;
    sizes.assign(t.sizes().begin(), t.sizes().end());
    dtype = t.scalar_type();
    device = t.device();
  }
  void reset() { saved.reset_data(); }
  Tensor get() const {  // in any layout
    const Tensor t = saved.unpack();
    TORCH_CHECK(!t.defined() || (t.sizes() == c10::IntArrayRef(sizes) && t.scalar_type() == dtype && t.device() == device && t.layout() == at::kStrided),
                "a saved tensor came back as ", t.sizes(), " ", t.scalar_type(), " on ", t.device(), "; it was ", c10::IntArrayRef(sizes), " ", dtype,
                " on ", device);
    return t;
  }
  Tensor volume() const { const Tensor t = get(); return t.defined() ? dense(t) : t; }
  Tensor flat() const { const Tensor t = get(); return t.defined() ? t.contiguous() : t; }
};

bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t != nullptr && t->defined() && t->requires_grad()) return true;
  return false;
}

Tensor or_none(const MaybeTensor& t) { return t.has_value() ? *t : Tensor(); }

// ---- weight gradients of a backward pass in one launch ---------------------------------------------------------------------
// See scaffold_amd/modules.py: a convolution whose module defers leaves (parameter, operands) here instead of computing its
// weight gradient; when the pass ends -- still inside backward() -- all that the pass queued are computed by one batched
// call and added to the parameters' .grad.  The queue is kept per backward pass (graph task), so passes that run at the
// same time on other threads or streams never take each other's entries, and it ends with its pass: what a pass that
// raised has queued is dropped with it.
struct QueuedWeight {
  Tensor param, x, second, gy;
  c10::Stream stream;  // the one they are ready on
  int32_t p[3];
  bool master = false, early = false;
  int family = 1;  // the launch of the batch that takes it (1: large rows, 2: small volumes)
};

struct WeightBatch {
  std::vector<QueuedWeight> items;
  std::vector<Tensor> grads;
  std::optional<c10::Stream> beside;  // the pass's stream, while the launches run on a side stream of it
  c10::Event done{c10::DeviceType::CUDA};  // behind those launches
  size_t size() const { return items.size(); }
};

struct PassQueue {
  std::vector<QueuedWeight> items;
  std::vector<std::shared_ptr<WeightBatch>> sent;  // on their way on a side stream
};

std::mutex g_pass_lock;
auto& g_passes = *new std::unordered_map<int, PassQueue>;  // never destroyed: a thread may still be in a pass at exit

Problem problem_of(const QueuedWeight& q, int code) {
  int64_t in[5];
  std::copy(q.x.sizes().begin(), q.x.sizes().end(), in);
  if (q.second.defined()) in[1] += q.second.size(1);
  const int32_t one[3] = {1, 1, 1};
  Problem prob;
  TORCH_INTERNAL_ASSERT(make_problem(in, q.param.sizes(), one, q.p, one, code, prob));
  return prob;
}

// Where the gradients of `batch` (one device, operand dtype and gradient dtype) go: memory of the current stream.
void allocate_grads(WeightBatch& batch) {
  for (const QueuedWeight& q : batch.items) batch.grads.push_back(volume(q.param.sizes(), q.gy, q.master ? at::kFloat : q.gy.scalar_type()));
}

// Computes them on the current stream, in calls of at most SFH_WGRAD_BATCH_MAX problems filled family by family.
void launch_batch(WeightBatch& batch, bool share_device) {
  if (batch.items.empty()) return;
  const Tensor& like = batch.items[0].gy;
  c10::OptionalDeviceGuard guard(like.device());
  const int code = code_of(like.scalar_type());
  const uint32_t flags = (batch.items[0].master ? SFH_FLAG_GRAD_FP32 : 0) | (share_device ? SFH_FLAG_SHARE_DEVICE : 0);
  if (batch.grads.empty()) allocate_grads(batch);
  std::vector<sfh_conv3d_wgrad_item> work(batch.items.size());
  for (size_t i = 0; i < batch.items.size(); ++i) {
    const QueuedWeight& q = batch.items[i];
    work[i] = sfh_conv3d_wgrad_item{problem_of(q, code).key.d, ptr(q.x), ptr(q.second), q.second.defined() ? (int32_t)q.x.size(1) : 0, ptr(q.gy),
                                    out_ptr(batch.grads[i])};
  }
  for (int family = 1; family <= 2; ++family) {
    std::vector<sfh_conv3d_wgrad_item> call;
    auto send = [&] {
      if (call.empty()) return;
      const size_t need = sfh_conv3d_wgrad_batch_workspace_bytes(call.data(), (int32_t)call.size(), code, flags);
      const Tensor ws = bytes(need, like);
      check(sfh_conv3d_wgrad_batch(call.data(), (int32_t)call.size(), code, out_ptr(ws), need, flags, stream_of(like)), "conv3d_backward_weight_batch");
      call.clear();
    };
    for (size_t i = 0; i < work.size(); ++i) {
      if (batch.items[i].family != family) continue;
      call.push_back(work[i]);
      if (call.size() == SFH_WGRAD_BATCH_MAX) send();
    }
    send();
  }
}

// A pass computes on the stream of whoever called backward(), and its nodes ran on the streams of their forward ops: what
// came from another stream is waited for, and its memory is not handed out before this stream has read it.
void take_over(WeightBatch& batch) {
  if (batch.items.empty()) return;
  const c10::Stream here = stream_on(batch.items[0].gy.device());
  std::vector<c10::Stream> met;
  for (size_t i = 0; i < batch.items.size(); ++i) {
    const QueuedWeight& q = batch.items[i];
    if (q.stream == here) continue;
    if (std::find(met.begin(), met.end(), q.stream) == met.end()) {
      met.push_back(q.stream);
      c10::Event ready(c10::DeviceType::CUDA);
      ready.record(q.stream);
      ready.block(here);
    }
    for (const Tensor& t : {q.x, q.second, q.gy, batch.grads.empty() ? Tensor() : batch.grads[i]})
      if (t.defined()) t.record_stream(here);
  }
}

// Passes of several threads may meet in one parameter: its .grad is written by one at a time, on the device as well (the
// additions of a pass on another stream come first).  Inside a capture the recorded order is all there is.
std::mutex g_add_lock;
struct LastAddition {
  c10::Stream stream;
  c10::Event done{c10::DeviceType::CUDA};
};
auto& g_last_addition = *new std::unordered_map<int, LastAddition>;  // by device (never destroyed: the runtime may be gone before)

void add_to_grads(WeightBatch& batch) {
  if (batch.items.empty()) return;
  const c10::Device device = batch.items[0].gy.device();
  c10::OptionalDeviceGuard guard(device);
  const c10::Stream here = stream_on(device);
  const bool eager = c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None;
  std::lock_guard<std::mutex> hold(g_add_lock);
  auto last = g_last_addition.try_emplace(device.index(), LastAddition{here}).first;
  if (eager && last->second.stream != here) last->second.done.block(here);
  for (size_t i = 0; i < batch.items.size(); ++i) {
    const Tensor &param = batch.items[i].param, &gw = batch.grads[i];
    Tensor& grad = param.mutable_grad();
    if (grad.defined()) grad.add_(gw);
    else grad = gw.strides() == param.strides() ? gw : at::empty_like(param).copy_(gw);  // the parameter's own layout, as the engine leaves it
  }
  if (eager) {
    last->second.stream = here;
    last->second.done.record(here);
  }
}

// Sends the batch to `side`, behind what the current stream has been given so far (modules._send_early).
void launch_beside(WeightBatch& batch, const c10::Stream& side) {
  const c10::Stream main = stream_on(side.device());
  const auto behind = [](const c10::Stream& waits, const c10::Stream& for_) {
    c10::Event reached(c10::DeviceType::CUDA);
    reached.record(for_);
    reached.block(waits);
  };
  behind(side, main);
  try {
    c10::StreamGuard on_side(side);
    at::AutoGradMode no_grad(false);
    launch_batch(batch, true);
  } catch (...) {
    behind(main, side);
    throw;
  }
  batch.beside = main;
  batch.done.record(side);
}

// Makes the pass's stream, and the current one, wait for a batch sent to a side stream.
void join_beside(WeightBatch& batch) {
  const c10::Stream here = stream_on(batch.beside.value().device());
  batch.done.block(*batch.beside);
  if (here != *batch.beside) batch.done.block(here);
}

PassQueue take_pass(int id) {
  std::lock_guard<std::mutex> hold(g_pass_lock);
  PassQueue pass;
  auto it = g_passes.find(id);
  if (it != g_passes.end()) {
    pass = std::move(it->second);
    g_passes.erase(it);
  }
  return pass;
}

void join_sent(const PassQueue& pass) {
  if (pass.sent.empty()) return;
  py::gil_scoped_acquire gil;
  for (const auto& batch : pass.sent) py::reinterpret_borrow<py::function>(g_join_early)(batch);
}

// Computes what a pass has queued and adds it (no entry: nothing to do).
void finish_pass(int id) {
  PassQueue pass = take_pass(id);
  at::AutoGradMode no_grad(false);
  join_sent(pass);
  for (auto& batch : pass.sent) {
    take_over(*batch);
    add_to_grads(*batch);
  }
  while (!pass.items.empty()) {
    WeightBatch batch;
    std::vector<QueuedWeight> rest;
    for (auto& q : pass.items) {
      const bool same = batch.items.empty() || (q.gy.device() == batch.items[0].gy.device() && q.gy.scalar_type() == batch.items[0].gy.scalar_type() &&
                                                q.master == batch.items[0].master);
      (same ? batch.items : rest).push_back(std::move(q));
    }
    pass.items = std::move(rest);
    take_over(batch);
    launch_batch(batch, false);
    add_to_grads(batch);
  }
}

// Lives as long as the pass whose final callback holds it.  A pass that raises runs no callback: its entry is dropped here,
// after the launches already sent to a side stream have been joined (they read the operands that are let go).
struct PassEnd {
  const int id;
  explicit PassEnd(int pass) : id(pass) {}
  PassEnd(const PassEnd&) = delete;
  ~PassEnd() {
    try {
      join_sent(take_pass(id));
    } catch (const std::exception& e) {
      TORCH_WARN("weight gradients of a backward pass that raised: ", e.what());
    }
  }
};

// What the pass this thread is in has queued so far (outside of a pass nothing waits).
void finish_current_pass() { finish_pass(torch::autograd::get_current_graph_task_id()); }

size_t waiting_weight_gradients() {
  std::lock_guard<std::mutex> hold(g_pass_lock);
  size_t n = 0;
  for (const auto& kv : g_passes) {
    n += kv.second.items.size();
    for (const auto& batch : kv.second.sent) n += batch->size();
  }
  return n;
}

void queue_weight(QueuedWeight&& q) {
  const int id = torch::autograd::get_current_graph_task_id();
  std::shared_ptr<WeightBatch> leave;
  {
    std::lock_guard<std::mutex> hold(g_pass_lock);
    auto found = g_passes.find(id);
    if (found == g_passes.end()) {
      torch::autograd::Engine::get_default_engine().queue_callback([end = std::make_shared<PassEnd>(id)] { finish_pass(end->id); });
      found = g_passes.emplace(id, PassQueue{}).first;
    }
    auto& items = found->second.items;
    if (q.early && q.family == 2) {
      // The pass has reached a small volume: the deep levels, whose kernels are bound by latency and leave most of the
      // device idle.  The large-row gradients queued so far (the decoder's upper levels) go out now, on a stream of their
      // own and on half of the compute units, beside the rest of the pass.
      auto goes = [&](const QueuedWeight& o) {
        return o.family == 1 && o.early && o.stream == q.stream && o.gy.scalar_type() == q.gy.scalar_type() && o.master == q.master;
      };
      if (std::count_if(items.begin(), items.end(), goes) >= 2) {
        leave = std::make_shared<WeightBatch>();
        std::vector<QueuedWeight> rest;
        for (auto& o : items) (goes(o) ? leave->items : rest).push_back(std::move(o));
        items = std::move(rest);
      }
    }
    items.push_back(std::move(q));
  }
  if (leave) {
    allocate_grads(*leave);  // here and not on the side stream: the pass and the optimizer read them on this one
    {
      py::gil_scoped_acquire gil;
      py::reinterpret_borrow<py::function>(g_send_early)(leave);
    }
    std::lock_guard<std::mutex> hold(g_pass_lock);
    g_passes[id].sent.push_back(leave);
  }
}

// What the backward of a convolution over x, or over the pair (x, second), needs.  In the depth-shard form the tensors that
// are saved are slabs of which x and second are the depth interiors.
struct ConvSaved {
  Kept x, second, w, packed_dgrad;  // w undefined: an fp32 master of which only the packed forms are read
  c10::DimVector w_sizes;
  Tensor param;             // the parameter whose weight gradient waits for the end of the pass (undefined: computed here)
  int family = 0;
  bool early = false, pair = false, has_bias = false, master = false;
  at::ScalarType bias_dtype = at::kFloat;
  int32_t s[3], p[3], d[3];
  int64_t halo = 0, depth = 0, first_channels = 0;
  std::vector<int64_t> in_sizes;

  void release() {
    x.reset(); second.reset(); w.reset(); packed_dgrad.reset();
    param.reset();
  }
  // out: the gradients of x, weight, bias and second that are wanted (gy dense)
  void backward(const Tensor& gy, bool need_x, bool need_w, bool need_b, bool need_2, Tensor out[4]) {
    const Tensor xs = x.volume(), x2 = second.volume(), wt = w.get(), packed = packed_dgrad.flat();
    Problem prob;
    TORCH_INTERNAL_ASSERT(make_problem(in_sizes, w_sizes, s, p, d, code_of(gy.scalar_type()), prob));
    if (need_x || need_2) {
      // The faces of a slab are zeros that the module put there: nobody receives their gradients.  The planes between them
      // are the data gradient of the padded problem, whose launch has no planes to drop (on 8 planes a fifth of the work) and
      // no workgroups past a round for them; a voxel's products are the same, added in the order of the kernel that serves
      // the padded problem.  Where that is not one the gradient serves (a halo wider than the kernel reaches) the slab's is cut.
      Problem inner = prob;
      int64_t cut = halo;
      if (halo > 0 && p[0] + halo <= (int64_t)d[0] * (w_sizes[2] - 1)) {
        std::vector<int64_t> in = in_sizes;
        in[2] = depth;
        const int32_t padding[3] = {p[0] + (int32_t)halo, p[1], p[2]};
        Problem padded;
        if (make_problem(in, w_sizes, s, padding, d, prob.key.code, padded) && padded.sizes->packed[1] == prob.sizes->packed[1] &&
            (!pair || sfh_conv3d_pair_supported(padded.desc(), prob.key.code, (int32_t)first_channels, 1))) {
          inner = padded;
          cut = 0;
        }
      }
      auto gx = launch_dgrad(inner, gy, wt, packed, pair ? first_channels : 0);
      if (cut > 0) {
        gx.first = gx.first.narrow(2, cut, depth);
        if (pair) gx.second = gx.second.narrow(2, cut, depth);
      }
      if (need_x) out[0] = gx.first;
      if (need_2) out[3] = gx.second;
    }
    if (need_w && need_b && !pair && prob.sizes->work_bias > 0) {
      // both parameter gradients from one pass over the output gradient (the 1x1x1 head)
      c10::OptionalDeviceGuard guard(gy.device());
      const auto& pd = prob.key.d;
      const auto dtype = master ? at::kFloat : gy.scalar_type();
      Tensor gw = volume({pd.cout, pd.cin, pd.kd, pd.kh, pd.kw}, gy, dtype), gb = plain({pd.cout}, gy, dtype);
      const Tensor ws = bytes(prob.sizes->work_bias, gy);
      const int rc = sfh_conv3d_wgrad_bias(prob.desc(), prob.key.code, ptr(xs), ptr(gy), out_ptr(gw), out_ptr(gb), out_ptr(ws), prob.sizes->work_bias,
                                           dtype != gy.scalar_type() ? SFH_FLAG_GRAD_FP32 : 0, stream_of(gy));
      if (rc != SFH_ERR_UNSUPPORTED) {
        check(rc, "conv3d_backward_weight_bias");
        out[1] = gw;
        out[2] = gb.scalar_type() == bias_dtype ? gb : gb.to(bias_dtype);
        return;
      }
    }
    if (need_w && param.defined()) {
      queue_weight(QueuedWeight{param, xs, x2, gy, stream_on(gy.device()), {p[0], p[1], p[2]}, master, early, family});
    } else if (need_w) {
      out[1] = launch_wgrad(prob, xs, x2, gy, master);
    }
    if (need_b) out[2] = launch_bias_grad(gy, bias_dtype);
  }
};

struct ConvNode : public LaunchNode {  // edges: x, weight, bias, second
  ConvSaved saved;
  std::string name() const override { return "ScaffoldConv3dBackward"; }
  void release_variables() override { saved.release(); }
  variable_list backward(variable_list& grads) override {
    variable_list out(4);
    if (grads[0].defined())
      saved.backward(dense(grads[0]), task_should_compute_output(0), task_should_compute_output(1), saved.has_bias && task_should_compute_output(2),
                     saved.pair && task_should_compute_output(3), out.data());
    return out;
  }
};

// The weight a node keeps: one that was packed from an fp32 master is not read again, and a program may step the master
// between forward and backward, as it may where autocast has cast it.
Tensor unless_packed_master(const Tensor& w, const Tensor& x) { return w.scalar_type() == x.scalar_type() ? w : Tensor(); }

void save_conv(ConvSaved& c, const Tensor& x, const Tensor& x_read, const Tensor& w, const Tensor& packed_dgrad, int64_t halo, bool master,
               const Tensor& param, int family, bool early) {
  c.x.keep(x_read);
  c.w.keep(unless_packed_master(w, x_read));
  c.w_sizes.assign(w.sizes().begin(), w.sizes().end());
  c.packed_dgrad.keep(packed_dgrad);
  c.halo = halo;
  c.depth = x.size(2);
  c.first_channels = x_read.size(1);
  c.in_sizes = x_read.sizes().vec();
  c.master = master;
  c.param = param;
  c.family = family;
  c.early = early;
}

// Records the node of y = conv(x[, second]) that a launch has just produced.  `x_read` / `second_read`: the tensors the
// kernels read (slabs in the depth-shard form, halo > 0; else x and second themselves).
void record_conv(Tensor y, const Tensor& x, const Tensor& weight, const MaybeTensor& bias, const MaybeTensor& second, const Tensor& x_read,
                 const MaybeTensor& second_read, const Tensor& w, const MaybeTensor& packed_dgrad, int64_t halo, py::handle stride,
                 py::handle padding, py::handle dilation, bool master, int family, bool early) {
  const Tensor b = or_none(bias), x2 = or_none(second);
  if (!wants_grad({&x, &weight, &b, &x2})) return;
  auto node = new_node<ConvNode>();
  ConvSaved& c = node->saved;
  TORCH_CHECK_VALUE(three(stride, c.s) && three(padding, c.p) && three(dilation, c.d), "stride, padding and dilation are ints or three ints");
  node->set_next_edges(torch::autograd::collect_next_edges(x, weight, b, x2));
  const Tensor read2 = or_none(second_read);
  save_conv(c, x, x_read, w, or_none(packed_dgrad), halo, master, family > 0 ? weight : Tensor(), family, early);
  c.second.keep(read2);
  c.pair = x2.defined();
  if (read2.defined()) c.in_sizes[1] += read2.size(1);
  c.has_bias = b.defined();
  if (b.defined()) c.bias_dtype = b.scalar_type();
  torch::autograd::set_history(y, node);
}

py::object tensor_or_none(const Tensor& t) { return t.defined() ? py::cast(t) : py::none(); }

// conv3d.conv3d_forward / conv3d_forward_pair: (y, partials, records), or None for a call that is not served as it stands.
// `master`: w may be the fp32 master that `packed` was made from.
py::object conv_forward(const Tensor& x, const Tensor& w, const MaybeTensor& bias, py::handle stride, py::handle padding, py::handle dilation,
                        const MaybeTensor& packed, int gn_groups, const MaybeTensor& second, bool master) {
  int32_t s[3], p[3], d[3];
  if (!three(stride, s) || !three(padding, p) || !three(dilation, d)) return py::none();
  Problem prob;
  if (!conv_gate(x, w, bias, s, p, d, false, prob, second.has_value() && second->dim() == 5 ? second->size(1) : 0, master && packed.has_value())) return py::none();
  if (packed.has_value() && !packed_fits(*packed, prob.sizes->packed[0], x)) return py::none();
  if (second.has_value() && (second->dim() != 5 || !on_gpu(*second) || second->device() != x.device() || second->scalar_type() != x.scalar_type() ||
                             second->size(0) != x.size(0) || second->size(2) != x.size(2) || second->size(3) != x.size(3) || second->size(4) != x.size(4)))
    return py::none();
  const ConvResult r = launch_conv(prob, dense(x), second.has_value() ? dense(*second) : Tensor(), w, or_none(bias), or_none(packed), gn_groups);
  return py::make_tuple(r.y, tensor_or_none(r.records > 0 ? r.partials : Tensor()), r.records);
}

// conv3d.is_supported_all for exact argument kinds (False also where the Python gate has to look closer)
// `packed`: the kernels read packed forms, w may be the fp32 master they were made from
bool conv_supported(const Tensor& x, const Tensor& w, const MaybeTensor& bias, py::handle stride, py::handle padding, py::handle dilation, bool all,
                    bool packed) {
  int32_t s[3], p[3], d[3];
  Problem prob;
  return three(stride, s) && three(padding, p) && three(dilation, d) && conv_gate(x, w, bias, s, p, d, all, prob, 0, packed);
}

// conv3d.conv3d_backward_data
py::object conv_backward_data(const Tensor& grad_output, const Tensor& w, at::IntArrayRef in_sizes, py::handle stride, py::handle padding,
                              py::handle dilation, const MaybeTensor& packed) {
  int32_t s[3], p[3], d[3];
  if (!three(stride, s) || !three(padding, p) || !three(dilation, d)) return py::none();
  if (grad_output.dim() != 5 || w.dim() != 5 || in_sizes.size() != 5 || !on_gpu(grad_output) || !on_gpu(w)) return py::none();
  if (grad_output.device() != w.device() || grad_output.scalar_type() != w.scalar_type() || in_sizes[1] != w.size(1)) return py::none();
  for (int i = 0; i < 3; ++i)
    if (s[i] != 1 || p[i] > d[i] * ((int32_t)w.size(2 + i) - 1)) return py::none();
  Problem prob;
  if (!make_problem(in_sizes, w.sizes(), s, p, d, code_of(w.scalar_type()), prob)) return py::none();
  if (grad_output.size(0) != prob.key.d.n || grad_output.size(1) != prob.key.d.cout) return py::none();
  for (int i = 0; i < 3; ++i)
    if (grad_output.size(2 + i) != prob.out[i]) return py::none();
  if (packed.has_value() && !packed_fits(*packed, prob.sizes->packed[1], grad_output)) return py::none();
  return py::cast(launch_dgrad(prob, dense(grad_output), w, or_none(packed), 0).first);
}

// conv3d.conv3d_backward_weight in the operands' dtype
py::object conv_backward_weight(const Tensor& x, at::IntArrayRef w_sizes, const Tensor& grad_output, py::handle stride, py::handle padding,
                                py::handle dilation) {
  int32_t s[3], p[3], d[3];
  if (!three(stride, s) || !three(padding, p) || !three(dilation, d)) return py::none();
  if (x.dim() != 5 || grad_output.dim() != 5 || w_sizes.size() != 5 || !on_gpu(x) || !on_gpu(grad_output)) return py::none();
  if (x.device() != grad_output.device() || x.scalar_type() != grad_output.scalar_type() || x.size(1) != w_sizes[1]) return py::none();
  Problem prob;
  if (!make_problem(x.sizes(), w_sizes, s, p, d, code_of(x.scalar_type()), prob)) return py::none();
  if (grad_output.size(0) != prob.key.d.n || grad_output.size(1) != prob.key.d.cout) return py::none();
  for (int i = 0; i < 3; ++i)
    if (grad_output.size(2 + i) != prob.out[i]) return py::none();
  return py::cast(launch_wgrad(prob, dense(x), Tensor(), dense(grad_output), false));
}

// The packed forms of an fp32 master weight for a 16-bit convolution of an input of `in_sizes`, in one launch:
// (packed_fwd, packed_dgrad, complete).  A form is None when that direction does not read one or (data gradient) was not
// asked for; `complete`: every direction asked for has its form, so nobody reads the weight itself.  Nothing is packed for
// an input whose channels are not the weight's.
py::object pack_master(const Tensor& weight, at::ScalarType dtype, at::IntArrayRef in_sizes, py::handle stride, py::handle padding, py::handle dilation,
                       bool want_dgrad) {
  int32_t s[3], p[3], d[3];
  Problem prob;
  if (!three(stride, s) || !three(padding, p) || !three(dilation, d) || weight.scalar_type() != at::kFloat || !on_gpu(weight) ||
      weight.dim() != 5 || in_sizes.size() != 5 || in_sizes[1] != weight.size(1) || !make_problem(in_sizes, weight.sizes(), s, p, d, code_of(dtype), prob))
    return py::make_tuple(py::none(), py::none(), false);
  c10::OptionalDeviceGuard guard(weight.device());
  const Tensor pf = bytes(prob.sizes->packed[0], weight), pd = want_dgrad ? bytes(prob.sizes->packed[1], weight) : Tensor();
  if (pf.defined() || pd.defined())
    check(sfh_conv3d_pack_master_weights(prob.desc(), prob.key.code, (const float*)ptr(weight), weight.strides().data(), out_ptr(pf), out_ptr(pd),
                                         stream_of(weight)), "pack_weights");
  return py::make_tuple(tensor_or_none(pf), tensor_or_none(pd), pf.defined() && (pd.defined() || !want_dgrad));
}

// ---- the 2x2x2-like transposed convolution (kernel == stride) ------------------------------------------------------------
struct ConvTransposeNode : public LaunchNode {  // edges: x, weight, bias
  Kept x, w, packed_fwd;  // w as in ConvSaved
  c10::DimVector w_sizes;
  int32_t k[3];
  bool has_bias = false, master = false;
  at::ScalarType bias_dtype = at::kFloat;
  std::string name() const override { return "ScaffoldConvTranspose3dBackward"; }
  void release_variables() override { x.reset(); w.reset(); packed_fwd.reset(); }
  variable_list backward(variable_list& grads) override {
    variable_list out(3);
    if (!grads[0].defined()) return out;
    const Tensor xs = x.volume(), wt = w.get(), packed = packed_fwd.flat();
    const Tensor gy = dense(grads[0]);
    if (gy.numel() == 0) {
      const auto dtype = master ? at::kFloat : gy.scalar_type();
      out[0] = volume(xs.sizes(), gy, gy.scalar_type());
      out[1] = volume(w_sizes, gy, dtype).zero_();
      if (has_bias) out[2] = at::zeros({w_sizes[1]}, gy.options().dtype(bias_dtype));
      return out;
    }
    // the stride-k convolution over gy whose forward is the data gradient and whose weight gradient is this one's
    const int32_t zero[3] = {0, 0, 0}, one[3] = {1, 1, 1};
    Problem prob;
    TORCH_INTERNAL_ASSERT(make_problem(gy.sizes(), w_sizes, k, zero, one, code_of(gy.scalar_type()), prob));
    const bool need_w = task_should_compute_output(1), need_b = has_bias && task_should_compute_output(2);
    if (task_should_compute_output(0)) out[0] = launch_conv(prob, gy, Tensor(), wt, Tensor(), packed, 0).y;
    // a result padded at the end: what is past the input's patches belongs to nobody
    int32_t extents[3];
    bool padded = false;
    for (int i = 0; i < 3; ++i) {
      extents[i] = (int32_t)gy.size(2 + i);
      padded = padded || gy.size(2 + i) != xs.size(2 + i) * k[i];
    }
    if (need_w && need_b) {
      c10::OptionalDeviceGuard guard(gy.device());
      const sfh_convT3d_desc td{(int32_t)xs.size(0), (int32_t)xs.size(1), (int32_t)xs.size(2), (int32_t)xs.size(3), (int32_t)xs.size(4),
                                (int32_t)w_sizes[1], k[0], k[1], k[2]};
      const size_t need = sfh_convT3d_wgrad_bias_workspace_bytes(&td, prob.key.code);
      if (need > 0) {
        const auto dtype = master ? at::kFloat : gy.scalar_type();
        Tensor gw = volume(w_sizes, gy, dtype), gb = plain({w_sizes[1]}, gy, dtype);
        const Tensor ws = bytes(need, gy);
        const int rc = sfh_convT3d_wgrad_bias_padded(&td, extents, prob.key.code, ptr(xs), ptr(gy), out_ptr(gw), out_ptr(gb), out_ptr(ws), need,
                                                     dtype != gy.scalar_type() ? SFH_FLAG_GRAD_FP32 : 0, stream_of(gy));
        if (rc != SFH_ERR_UNSUPPORTED) {
          check(rc, "conv_transpose3d_backward_weight_bias");
          out[1] = gw;
          out[2] = gb.scalar_type() == bias_dtype ? gb : gb.to(bias_dtype);
          return out;
        }
      }
    }
    if (need_w) out[1] = launch_wgrad(prob, gy, Tensor(), xs, master);
    if (need_b) {
      Tensor under = gy;
      for (int i = 0; i < 3 && padded; ++i) under = under.narrow(2 + i, 0, xs.size(2 + i) * k[i]);
      out[2] = launch_bias_grad(dense(under), bias_dtype);
    }
    return out;
  }
};

// FastConvTranspose3d: y (and the slab it lies in, or None), or None for a call that is not served as it stands.  `weight` /
// `bias` receive gradients, `w` / `b` are what the kernels read; the packed forms are those of the stride-k convolution.  `extents`:
// y is padded with zeros at the end to these (and lies in no slab); the problems that do that themselves only.
py::object conv_transpose(const Tensor& x_in, const Tensor& weight, const MaybeTensor& bias, const Tensor& w, const MaybeTensor& b, py::handle stride,
                          const MaybeTensor& packed_fwd, const MaybeTensor& packed_dgrad, int64_t halo, bool master,
                          const std::optional<std::vector<int64_t>>& extents) {
  int32_t k[3];
  if (!three(stride, k) || x_in.dim() != 5 || w.dim() != 5 || !on_gpu(x_in) || !on_gpu(w) || x_in.device() != w.device()) return py::none();
  // an fp32 master that nobody reads: both packed forms were made from it in x's dtype
  const bool all_packed = master && w.scalar_type() == at::kFloat && packed_fwd.has_value() && packed_dgrad.has_value();
  if ((x_in.scalar_type() != w.scalar_type() && !all_packed) || x_in.size(1) != w.size(0) || !bias_fits(b, x_in, w.size(1))) return py::none();
  int64_t big[5] = {x_in.size(0), w.size(1), 0, 0, 0};
  for (int i = 0; i < 3; ++i) {
    if (k[i] < 1 || w.size(2 + i) != k[i] || x_in.size(2 + i) < 1) return py::none();
    big[2 + i] = x_in.size(2 + i) * k[i];
  }
  const int32_t zero[3] = {0, 0, 0}, one[3] = {1, 1, 1};
  Problem prob;
  const bool empty = big[0] == 0;  // a batch of no samples: an empty result, zero parameter gradients
  if (empty && code_of(x_in.scalar_type()) < 0) return py::none();
  if (!empty && !make_problem(big, w.sizes(), k, zero, one, code_of(x_in.scalar_type()), prob)) return py::none();
  if (!empty && packed_dgrad.has_value() && !packed_fits(*packed_dgrad, prob.sizes->packed[1], x_in)) return py::none();
  if (!empty && packed_fwd.has_value() && !packed_fits(*packed_fwd, prob.sizes->packed[0], x_in)) return py::none();
  int32_t padded[3] = {0, 0, 0};
  if (extents.has_value()) {
    if (empty || extents->size() != 3 || k[0] != 2 || k[1] != 2 || k[2] != 2) return py::none();
    std::vector<int64_t> sizes{big[0], big[1]};
    for (int i = 0; i < 3; ++i) {
      if ((*extents)[i] < big[2 + i] || (*extents)[i] > INT32_MAX) return py::none();
      sizes.push_back(padded[i] = (int32_t)(*extents)[i]);
    }
    // both gradients of the padded problem are served, from the same packed forms
    const sfh_convT3d_desc td{(int32_t)x_in.size(0), (int32_t)x_in.size(1), (int32_t)x_in.size(2), (int32_t)x_in.size(3), (int32_t)x_in.size(4),
                              (int32_t)w.size(1), k[0], k[1], k[2]};
    Problem around;
    if (sfh_convT3d_wgrad_bias_workspace_bytes(&td, prob.key.code) == 0 || !make_problem(sizes, w.sizes(), k, zero, one, prob.key.code, around) ||
        around.sizes->packed[0] != prob.sizes->packed[0])
      return py::none();
  }
  const Tensor weight_b = or_none(bias);
  const bool graph = wants_grad({&x_in, &weight, &weight_b});
  Tensor x = x_in, y, slab;
  if (empty) {
    y = volume(big, x, x.scalar_type());
  } else {
    at::AutoGradMode no_grad(false);
    x = dense(x_in);
    c10::OptionalDeviceGuard guard(x.device());
    const sfh_convT3d_desc td{(int32_t)x.size(0), (int32_t)x.size(1), (int32_t)x.size(2), (int32_t)x.size(3), (int32_t)x.size(4),
                              (int32_t)w.size(1), k[0], k[1], k[2]};
    const int code = prob.key.code;
    const Tensor ws = packed_dgrad.has_value() ? Tensor() : bytes(sfh_convT3d_fwd_workspace_bytes(&td, code), x);
    const size_t ws_bytes = ws.defined() ? (size_t)ws.numel() : 0;
    const void* wp = packed_dgrad.has_value() ? ptr(*packed_dgrad) : ptr(w);
    const int64_t* strides = packed_dgrad.has_value() ? nullptr : w.strides().data();
    const uint32_t flags = packed_dgrad.has_value() ? SFH_FLAG_WEIGHT_PACKED : 0;
    int rc = SFH_ERR_UNSUPPORTED;
    if (extents.has_value()) {
      y = volume({big[0], big[1], padded[0], padded[1], padded[2]}, x, x.scalar_type());
      rc = sfh_convT3d_fwd_padded(&td, padded, code, ptr(x), wp, strides, ptr(or_none(b)), out_ptr(y), out_ptr(ws), ws_bytes, flags, stream_of(x));
      if (rc == SFH_ERR_UNSUPPORTED) return py::none();
    } else if (halo > 0 && x.size(0) == 1) {
      slab = volume({1, big[1], big[2] + 2 * halo, big[3], big[4]}, x, x.scalar_type());
      rc = sfh_convT3d_fwd_slab(&td, code, ptr(x), wp, strides, ptr(or_none(b)), out_ptr(slab), halo * big[3] * big[4] * big[1], out_ptr(ws), ws_bytes,
                                flags, stream_of(x));
      if (rc != SFH_ERR_UNSUPPORTED) y = slab.narrow(2, halo, big[2]);
    }
    if (rc == SFH_ERR_UNSUPPORTED) {
      slab = Tensor();
      y = volume(big, x, x.scalar_type());
      rc = sfh_convT3d_fwd(&td, code, ptr(x), wp, strides, ptr(or_none(b)), out_ptr(y), out_ptr(ws), ws_bytes, flags, stream_of(x));
    }
    check(rc, "conv_transpose3d_forward");
  }
  if (graph) {
    auto node = new_node<ConvTransposeNode>();
    node->set_next_edges(torch::autograd::collect_next_edges(x_in, weight, weight_b));
    node->x.keep(x);
    node->w.keep(unless_packed_master(w, x));
    node->w_sizes.assign(w.sizes().begin(), w.sizes().end());
    node->packed_fwd.keep(or_none(packed_fwd));
    std::memcpy(node->k, k, sizeof(k));
    node->has_bias = weight_b.defined();
    if (weight_b.defined()) node->bias_dtype = weight_b.scalar_type();
    node->master = master;
    if (slab.defined()) y = y.detach();  // a tensor of its own: a view would keep the slab as its differentiable base
    torch::autograd::set_history(y, node);
  }
  return py::make_tuple(y, tensor_or_none(slab));
}

// ---- GroupNorm -----------------------------------------------------------------------------------------------------------
// What the backward of GroupNorm (+ ReLU) needs.
struct NormSaved {
  Kept input, weight, bias, stats, idx;  // idx: where the pooled result's maxima lie (undefined: the result was not pooled)
  int groups = 1;
  bool relu = false;
  void release() { input.reset(); weight.reset(); bias.reset(); stats.reset(); idx.reset(); }
  // grad / pooled: of the result and of what the same launch pooled from it (either may be undefined)
  void backward(const Tensor& grad, const Tensor& pooled, Tensor& dx, Tensor& dw, Tensor& db) {
    const Tensor x = input.volume(), st = stats.flat(), ix = pooled.defined() ? idx.flat() : Tensor();
    Tensor w = weight.flat(), b = bias.flat();
    Tensor gy = grad.defined() ? dense(grad) : Tensor(), gp = pooled.defined() ? dense(pooled) : Tensor();
    if (gp.defined() && gp.scalar_type() != x.scalar_type()) gp = gp.to(x.scalar_type());
    if (gy.defined() && gy.scalar_type() != x.scalar_type() && (gp.defined() || gy.scalar_type() != at::kFloat)) gy = gy.to(x.scalar_type());
    const Tensor w_in = w, b_in = b;
    if (w.defined() && b.defined() && w.scalar_type() != b.scalar_type()) b = b.to(w.scalar_type());
    c10::OptionalDeviceGuard guard(x.device());
    const int64_t c = x.size(1), n = x.size(0);
    const sfh_groupnorm_desc d{(int32_t)n, (int32_t)c, groups, relu ? 1 : 0, x.numel() / (n * c), 0.f};
    const int code = code_of(x.scalar_type());
    dx = volume(x.sizes(), x, x.scalar_type());
    if (w.defined()) dw = plain({c}, x, at::kFloat);
    if (b.defined()) db = plain({c}, x, at::kFloat);
    const Tensor ws = bytes(sfh_groupnorm_bwd_workspace_bytes(&d, code), x);
    const size_t ws_bytes = ws.defined() ? (size_t)ws.numel() : 0;
    const float* mean = (const float*)ptr(st);
    const int pcode = code_of(w.defined() ? w.scalar_type() : b.defined() ? b.scalar_type() : x.scalar_type());
    int rc = SFH_ERR_UNSUPPORTED;
    if (gp.defined() && gy.defined()) {
      const int32_t extents[3] = {(int32_t)x.size(2), (int32_t)x.size(3), (int32_t)x.size(4)};
      rc = sfh_groupnorm_bwd_pool(&d, extents, code, pcode, ptr(gy), ptr(gp), (const uint8_t*)ptr(ix), ptr(x), ptr(w), ptr(b), mean, mean + n * groups,
                                  out_ptr(dx), (float*)out_ptr(dw), (float*)out_ptr(db), out_ptr(ws), ws_bytes, stream_of(x));
    }
    if (rc == SFH_ERR_UNSUPPORTED) {
      if (gp.defined()) {  // the sum of the two gradients in a launch of its own
        const sfh_pool_desc pd{(int32_t)n, (int32_t)c, (int32_t)x.size(2), (int32_t)x.size(3), (int32_t)x.size(4)};
        Tensor sum = volume(x.sizes(), x, x.scalar_type());
        check(gy.defined() ? sfh_maxpool2_bwd_add(&pd, code, ptr(gp), (const uint8_t*)ptr(ix), ptr(gy), out_ptr(sum), stream_of(x))
                           : sfh_maxpool2_bwd(&pd, code, ptr(gp), (const uint8_t*)ptr(ix), out_ptr(sum), stream_of(x)), "max_pool3d_2x backward");
        gy = sum;
      }
      rc = sfh_groupnorm_bwd(&d, code, code_of(gy.scalar_type()), pcode, ptr(gy), ptr(x), ptr(w), ptr(b), mean, mean + n * groups, out_ptr(dx),
                             (float*)out_ptr(dw), (float*)out_ptr(db), out_ptr(ws), ws_bytes, stream_of(x));
    }
    check(rc, "group_norm_backward");
    if (dw.defined() && dw.scalar_type() != w_in.scalar_type()) dw = dw.to(w_in.scalar_type());
    if (db.defined() && db.scalar_type() != b_in.scalar_type()) db = db.to(b_in.scalar_type());
  }
};

struct NormResult {
  Tensor y, slab, stats;  // stats: mean and rstd
};

// The gate of the forward (groupnorm.is_supported) for an input of this description.
bool norm_gate(const Tensor& like, int64_t n, int64_t c, int64_t spatial, int64_t groups, const MaybeTensor& weight, const MaybeTensor& bias) {
  if (code_of(like.scalar_type()) < 0 || groups < 1 || c % groups != 0 || n * c * spatial == 0) return false;
  if ((c == groups && n * spatial == 1) || n > INT32_MAX || c > INT32_MAX) return false;
  for (const MaybeTensor* t : {&weight, &bias}) {
    if (!t->has_value()) continue;
    if ((*t)->dim() != 1 || (*t)->numel() != c || (*t)->device() != like.device()) return false;
    if ((*t)->scalar_type() != like.scalar_type() && ((*t)->scalar_type() != at::kFloat || !at::autocast::is_autocast_enabled(at::kCUDA))) return false;
  }
  return true;
}

NormResult launch_norm(const Tensor& input, int64_t groups, const Tensor& weight, const Tensor& bias, double eps, bool relu, at::ScalarType odt, int64_t halo,
                       const Tensor& partials, int32_t records) {
  c10::OptionalDeviceGuard guard(input.device());
  const int64_t n = input.size(0), c = input.size(1);
  const int code = code_of(input.scalar_type());
  NormResult r;
  Tensor w = weight.defined() ? weight.contiguous() : weight, b = bias.defined() ? bias.contiguous() : bias;
  if (w.defined() && b.defined() && w.scalar_type() != b.scalar_type()) b = b.to(w.scalar_type());
  const int pcode = code_of(w.defined() ? w.scalar_type() : b.defined() ? b.scalar_type() : input.scalar_type());
  r.stats = plain({2, n, groups}, input, at::kFloat);
  float* mean = (float*)out_ptr(r.stats);
  float* rstd = mean + n * groups;
  const sfh_groupnorm_desc d{(int32_t)n, (int32_t)c, (int32_t)groups, relu ? 1 : 0, input.numel() / (n * c), (float)eps};
  void* st = stream_of(input);
  int64_t halo_rows = 0;
  if (halo > 0 && n == 1 && (int64_t)c10::elementSize(odt) == (int64_t)input.element_size()) {
    r.slab = volume({1, c, input.size(2) + 2 * halo, input.size(3), input.size(4)}, input, odt);
    r.y = r.slab.narrow(2, halo, input.size(2));
    halo_rows = halo * input.size(3) * input.size(4);
  } else {
    r.y = volume(input.sizes(), input, odt);
  }
  int rc = SFH_ERR_UNSUPPORTED;
  if (partials.defined())
    rc = sfh_groupnorm_fwd_from_partials(&d, code, code_of(odt), pcode, ptr(input), ptr(w), ptr(b), out_ptr(r.slab.defined() ? r.slab : r.y), halo_rows, mean,
                                         rstd, (const float*)ptr(partials), (size_t)partials.numel() * 4, records, st);
  if (rc == SFH_ERR_UNSUPPORTED) {
    const Tensor ws = bytes(sfh_groupnorm_fwd_workspace_bytes(&d, code), input);
    const size_t ws_bytes = ws.defined() ? (size_t)ws.numel() : 0;
    if (r.slab.defined()) {
      rc = sfh_groupnorm_fwd_slab(&d, code, code_of(odt), pcode, ptr(input), ptr(w), ptr(b), out_ptr(r.slab), halo_rows, mean, rstd, out_ptr(ws), ws_bytes, st);
      if (rc == SFH_ERR_UNSUPPORTED) {  // channel counts off the vector path: the plain form
        r.slab = Tensor();
        r.y = volume(input.sizes(), input, odt);
      }
    }
    if (rc == SFH_ERR_UNSUPPORTED)
      rc = sfh_groupnorm_fwd(&d, code, code_of(odt), pcode, ptr(input), ptr(w), ptr(b), out_ptr(r.y), mean, rstd, out_ptr(ws), ws_bytes, st);
  }
  check(rc, "group_norm");
  return r;
}

// The normalisation with the pooling that follows it, from the records the producer of `input` left, in one launch.
struct PooledResult {
  Tensor pooled, slab, idx;  // idx: undefined where no gradient is wanted
};
bool launch_norm_pool(const Tensor& input, int64_t groups, const Tensor& weight, const Tensor& bias, double eps, bool relu, int64_t halo,
                      const Tensor& partials, int32_t records, int64_t pool_halo, bool want_idx, NormResult& r, PooledResult& out) {
  const int64_t n = input.size(0), c = input.size(1), d2 = input.size(2) / 2, h2 = input.size(3) / 2, w2 = input.size(4) / 2;
  if (d2 < 1 || h2 < 1 || w2 < 1 || n < 1 || c % 8 != 0 || input.scalar_type() == at::kFloat || (pool_halo > 0 && n != 1)) return false;
  c10::OptionalDeviceGuard guard(input.device());
  Tensor w = weight.contiguous(), b = bias.contiguous();
  if (w.scalar_type() != b.scalar_type()) b = b.to(w.scalar_type());
  NormResult made;
  PooledResult pool;
  made.stats = plain({2, n, groups}, input, at::kFloat);
  float* mean = (float*)out_ptr(made.stats);
  int64_t halo_rows = 0;
  if (halo > 0 && n == 1) {
    made.slab = volume({1, c, input.size(2) + 2 * halo, input.size(3), input.size(4)}, input, input.scalar_type());
    made.y = made.slab.narrow(2, halo, input.size(2));
    halo_rows = halo * input.size(3) * input.size(4);
  } else {
    made.y = volume(input.sizes(), input, input.scalar_type());
  }
  if (pool_halo > 0) {
    pool.slab = volume({1, c, d2 + 2 * pool_halo, h2, w2}, input, input.scalar_type());
    pool.pooled = pool.slab.narrow(2, pool_halo, d2);
  } else {
    pool.pooled = volume({n, c, d2, h2, w2}, input, input.scalar_type());
  }
  if (want_idx) pool.idx = plain({n, d2, h2, w2, c}, input, at::kByte);
  const int32_t extents[3] = {(int32_t)input.size(2), (int32_t)input.size(3), (int32_t)input.size(4)};
  const sfh_groupnorm_desc d{(int32_t)n, (int32_t)c, (int32_t)groups, relu ? 1 : 0, input.numel() / (n * c), (float)eps};
  const int rc = sfh_groupnorm_fwd_pool(&d, extents, code_of(input.scalar_type()), code_of(w.scalar_type()), ptr(input), ptr(w), ptr(b),
                                        out_ptr(made.slab.defined() ? made.slab : made.y), halo_rows, mean, mean + n * groups, (const float*)ptr(partials),
                                        (size_t)partials.numel() * 4, records, out_ptr(pool.slab.defined() ? pool.slab : pool.pooled),
                                        pool_halo > 0 ? pool_halo * h2 * w2 * c : 0, (uint8_t*)out_ptr(pool.idx), stream_of(input));
  if (rc == SFH_ERR_UNSUPPORTED) return false;
  check(rc, "group_norm with pooling");
  r = std::move(made);
  out = std::move(pool);
  return true;
}

void save_norm(NormSaved& s, const Tensor& input, const Tensor& weight, const Tensor& bias, const Tensor& stats, int64_t groups, bool relu) {
  s.input.keep(input);
  s.weight.keep(weight);
  s.bias.keep(bias);
  s.stats.keep(stats);
  s.groups = (int)groups;
  s.relu = relu;
}

struct GroupNormNode : public LaunchNode {  // edges: input, weight, bias
  NormSaved saved;
  std::string name() const override { return "ScaffoldGroupNormBackward"; }
  void release_variables() override { saved.release(); }
  variable_list backward(variable_list& grads) override {
    variable_list out(3);
    if (grads[0].defined()) saved.backward(grads[0], Tensor(), out[0], out[1], out[2]);
    return out;
  }
};

// groupnorm.group_norm outside torch.compile: (y, slab or None), or None for a call that is not served as it stands.
// `out_dtype`: None or "stock" (what F.group_norm would return: fp32 inside autocast); `partials`: Welford records the
// producer of `input` left for these very bits, `records` per sample.
py::object group_norm(const Tensor& input, int64_t groups, const MaybeTensor& weight, const MaybeTensor& bias, double eps, bool relu,
                      std::optional<at::ScalarType> out_dtype, bool stock_dtype, int64_t halo, const MaybeTensor& partials, int32_t records) {
  if (input.dim() != 5 || !on_gpu(input) || input.numel() == 0 || !input.is_contiguous(kCL3D)) return py::none();
  if (!norm_gate(input, input.size(0), input.size(1), input.numel() / (input.size(0) * input.size(1)), groups, weight, bias)) return py::none();
  at::ScalarType odt = out_dtype.value_or(input.scalar_type());
  if (stock_dtype) odt = input.scalar_type() != at::kFloat && at::autocast::is_autocast_enabled(at::kCUDA) ? at::kFloat : input.scalar_type();
  if (code_of(odt) < 0) return py::none();
  const Tensor w = or_none(weight), b = or_none(bias);
  const bool graph = wants_grad({&input, &w, &b});
  NormResult r;
  {
    at::AutoGradMode no_grad(false);
    r = launch_norm(input, groups, w, b, eps, relu, odt, halo, or_none(partials), records);
    if (graph && r.slab.defined()) r.y = r.y.detach();  // a tensor of its own: a view would keep the slab as its differentiable base
  }
  if (graph) {
    auto node = new_node<GroupNormNode>();
    node->set_next_edges(torch::autograd::collect_next_edges(input, w, b));
    save_norm(node->saved, input, w, b, r.stats, groups, relu);
    torch::autograd::set_history(r.y, node);
  }
  return py::make_tuple(r.y, tensor_or_none(r.slab));
}

// ---- a convolution and the GroupNorm that reads it -----------------------------------------------------------------------
// One call and one node for the pair every block of the U-Net is made of (bias-free convolution): half of the module calls
// and of the nodes of a pass.
struct ConvNormNode : public LaunchNode {  // edges: x, convolution weight, norm weight, norm bias; the second output, if any: what was pooled
  ConvSaved conv;
  NormSaved norm;
  std::string name() const override { return "ScaffoldConvGroupNormBackward"; }
  void release_variables() override { conv.release(); norm.release(); }
  variable_list backward(variable_list& grads) override {
    variable_list out(4);
    const Tensor pooled = grads.size() > 1 ? grads[1] : Tensor();
    if (!grads[0].defined() && !pooled.defined()) return out;
    Tensor gy, c[4];
    norm.backward(grads[0], pooled, gy, out[2], out[3]);
    conv.backward(gy, task_should_compute_output(0), task_should_compute_output(1), false, false, c);
    out[0] = c[0];
    out[1] = c[1];
    return out;
  }
};

// modules.conv_then_norm: (y, slab or None, pooled), or None (nothing launched) for a call that is not served as it stands.
// x / x_read, weight / w, packed forms, halo, master, family and early as in record_conv.  `pool_halo` >= 0: a MaxPool3d(2) with that
// halo follows; pooled is its result (tensor, slab or None), differentiable as y is, or None where this launch does not make it.
py::object conv_norm(const Tensor& x, const Tensor& x_read, const Tensor& weight, const Tensor& w, const MaybeTensor& packed_fwd, const MaybeTensor& packed_dgrad,
                     int64_t halo, py::handle stride, py::handle padding, py::handle dilation, bool master, int family, bool early, int64_t groups,
                     const Tensor& norm_weight, const Tensor& norm_bias, double eps, bool relu, int64_t out_halo, int64_t pool_halo) {
  int32_t s[3], p[3], d[3];
  if (!three(stride, s) || !three(padding, p) || !three(dilation, d) || !x_read.is_contiguous(kCL3D)) return py::none();
  const bool graph = wants_grad({&x, &weight, &norm_weight, &norm_bias});
  Problem prob;
  if (!conv_gate(x_read, w, std::nullopt, s, p, d, graph, prob, 0, master && packed_fwd.has_value())) return py::none();
  if (packed_fwd.has_value() && !packed_fits(*packed_fwd, prob.sizes->packed[0], x_read)) return py::none();
  if (packed_dgrad.has_value() && !packed_fits(*packed_dgrad, prob.sizes->packed[1], x_read)) return py::none();
  if (!norm_gate(x_read, prob.key.d.n, prob.key.d.cout, (int64_t)prob.out[0] * prob.out[1] * prob.out[2], groups, norm_weight, norm_bias)) return py::none();
  ConvResult c;
  NormResult r;
  PooledResult pool;
  {
    at::AutoGradMode no_grad(false);
    c = launch_conv(prob, x_read, Tensor(), w, Tensor(), or_none(packed_fwd), module_groups(prob, groups));
    if (pool_halo < 0 || c.records < 1 ||
        !launch_norm_pool(c.y, groups, norm_weight, norm_bias, eps, relu, out_halo, c.partials, c.records, pool_halo, graph, r, pool))
      r = launch_norm(c.y, groups, norm_weight, norm_bias, eps, relu, c.y.scalar_type(), out_halo, c.records > 0 ? c.partials : Tensor(), c.records);
    if (graph && r.slab.defined()) r.y = r.y.detach();
    if (graph && pool.slab.defined()) pool.pooled = pool.pooled.detach();
  }
  if (graph) {
    auto node = new_node<ConvNormNode>();
    node->set_next_edges(torch::autograd::collect_next_edges(x, weight, norm_weight, norm_bias));
    std::memcpy(node->conv.s, s, sizeof(s));
    std::memcpy(node->conv.p, p, sizeof(p));
    std::memcpy(node->conv.d, d, sizeof(d));
    save_conv(node->conv, x, x_read, w, or_none(packed_dgrad), halo, master, family > 0 ? weight : Tensor(), family, early);
    save_norm(node->norm, c.y, norm_weight, norm_bias, r.stats, groups, relu);
    node->norm.idx.keep(pool.idx);
    torch::autograd::set_history(r.y, node);
    if (pool.pooled.defined()) torch::autograd::set_history(pool.pooled, node);
  }
  const py::object pooled = pool.pooled.defined() ? py::object(py::make_tuple(pool.pooled, tensor_or_none(pool.slab))) : py::none();
  return py::make_tuple(r.y, tensor_or_none(r.slab), pooled);
}

// ---- MaxPool3d(2) --------------------------------------------------------------------------------------------------------
struct MaxPoolNode : public LaunchNode {  // edge: x; the second output, where there is one, is an alias of x (the skip connection)
  Kept idx;
  std::vector<int64_t> sizes;
  std::string name() const override { return "ScaffoldMaxPool3dBackward"; }
  void release_variables() override { idx.reset(); }
  variable_list backward(variable_list& grads) override {
    variable_list out(1);
    const Tensor skip = grads.size() > 1 ? grads[1] : Tensor();
    if (!grads[0].defined()) {
      out[0] = skip;
      return out;
    }
    const Tensor gy = dense(grads[0]), ix = idx.flat();
    c10::OptionalDeviceGuard guard(gy.device());
    Tensor gx = volume(sizes, gy, gy.scalar_type());
    const sfh_pool_desc d{(int32_t)sizes[0], (int32_t)sizes[1], (int32_t)sizes[2], (int32_t)sizes[3], (int32_t)sizes[4]};
    const int code = code_of(gy.scalar_type());
    if (skip.defined()) {
      Tensor gs = dense(skip);
      if (gs.scalar_type() != gy.scalar_type()) gs = gs.to(gy.scalar_type());
      check(sfh_maxpool2_bwd_add(&d, code, ptr(gy), (const uint8_t*)ptr(ix), ptr(gs), out_ptr(gx), stream_of(gy)), "max_pool3d_2x backward");
    } else {
      check(sfh_maxpool2_bwd(&d, code, ptr(gy), (const uint8_t*)ptr(ix), out_ptr(gx), stream_of(gy)), "max_pool3d_2x backward");
    }
    out[0] = gx;
    return out;
  }
};

// pooling.max_pool3d_2x: (y, slab or None[, alias of x]), or None for a call that is not served.
py::object max_pool(const Tensor& x_in, int64_t halo, bool with_skip) {
  if (x_in.dim() != 5 || !on_gpu(x_in) || code_of(x_in.scalar_type()) < 0 || x_in.size(1) < 1) return py::none();
  for (int i = 2; i < 5; ++i)
    if (x_in.size(i) < 1) return py::none();
  const bool graph = wants_grad({&x_in});
  Tensor y, slab, idx, skip;
  const auto z = x_in.sizes();
  {
    at::AutoGradMode no_grad(false);
    const Tensor x = dense(x_in);
    c10::OptionalDeviceGuard guard(x.device());
    const int64_t n = z[0], c = z[1], d2 = z[2] / 2, h2 = z[3] / 2, w2 = z[4] / 2;
    idx = plain({n, d2, h2, w2, c}, x, at::kByte);
    const sfh_pool_desc d{(int32_t)n, (int32_t)c, (int32_t)z[2], (int32_t)z[3], (int32_t)z[4]};
    const int code = code_of(x.scalar_type());
    int rc = SFH_ERR_UNSUPPORTED;
    if (halo > 0 && n == 1 && d2 > 0 && h2 > 0 && w2 > 0) {
      slab = volume({1, c, d2 + 2 * halo, h2, w2}, x, x.scalar_type());
      rc = sfh_maxpool2_fwd_slab(&d, code, ptr(x), out_ptr(slab), halo * h2 * w2 * c, (uint8_t*)out_ptr(idx), stream_of(x));
      if (rc != SFH_ERR_UNSUPPORTED) y = slab.narrow(2, halo, d2);
    }
    if (rc == SFH_ERR_UNSUPPORTED) {
      slab = Tensor();
      y = volume({n, c, d2, h2, w2}, x, x.scalar_type());
      rc = sfh_maxpool2_fwd(&d, code, ptr(x), out_ptr(y), (uint8_t*)out_ptr(idx), stream_of(x));
    }
    check(rc, "max_pool3d_2x");
    // (a view made without a graph: what is written into it would also change x_in, whose other uses autograd could not tell)
    if (with_skip) skip = graph ? x_in.view_as(x_in) : x_in.detach();
    if (graph && slab.defined()) y = y.detach();
  }
  if (graph) {
    auto node = new_node<MaxPoolNode>();
    node->set_next_edges(torch::autograd::collect_next_edges(x_in));
    node->idx.keep(idx);
    node->sizes = z.vec();
    torch::autograd::set_history(y, node);
    if (with_skip) torch::autograd::set_history(skip, node);
  }
  return with_skip ? py::make_tuple(y, tensor_or_none(slab), skip) : py::make_tuple(y, tensor_or_none(slab));
}

// ---- loss head -----------------------------------------------------------------------------------------------------------
struct LossNode : public LaunchNode {  // edge: logits
  Kept logits, labels, stats, class_weight;
  sfh_loss_desc d{};
  std::string name() const override { return "ScaffoldCeDiceBackward"; }
  void release_variables() override { logits.reset(); labels.reset(); stats.reset(); class_weight.reset(); }
  variable_list backward(variable_list& grads) override {
    variable_list out(1);
    if (!grads[0].defined()) return out;
    const Tensor x = logits.volume(), lab = labels.flat(), st = stats.flat(), cw = class_weight.flat();
    c10::OptionalDeviceGuard guard(x.device());
    const Tensor g = grads[0].to(x.device(), at::kFloat).reshape({1}).contiguous();
    Tensor dx = volume(x.sizes(), x, x.scalar_type());
    check(sfh_ce_dice_bwd(&d, code_of(x.scalar_type()), ptr(x), (const int64_t*)ptr(lab), (const float*)ptr(cw), (const float*)ptr(st), (const float*)ptr(g),
                          out_ptr(dx), stream_of(x)), "ce_dice_loss backward");
    out[0] = dx;
    return out;
  }
};

// losses.ce_dice_loss: the 0-dim loss, or None for a call that is not served.
py::object ce_dice_loss(const Tensor& logits, const Tensor& labels, const MaybeTensor& class_weight, double eps) {
  if (logits.dim() != 5 || labels.dim() != 4 || !on_gpu(logits) || labels.device() != logits.device() || labels.scalar_type() != at::kLong) return py::none();
  const int code = code_of(logits.scalar_type());
  const int64_t n = logits.size(0), c = logits.size(1);
  if (code < 0 || c < 2 || c > 32 || logits.numel() == 0 || labels.size(0) != n) return py::none();
  for (int i = 0; i < 3; ++i)
    if (labels.size(1 + i) != logits.size(2 + i)) return py::none();
  if (class_weight.has_value() && (class_weight->device() != logits.device() || class_weight->dim() != 1 || class_weight->size(0) != c ||
                                   !at::isFloatingType(class_weight->scalar_type())))
    return py::none();
  const bool graph = wants_grad({&logits});
  Tensor x, lab, cw, loss, stats;
  const sfh_loss_desc d{(int32_t)n, (int32_t)c, logits.numel() / (n * c), (float)eps};
  {
    at::AutoGradMode no_grad(false);
    c10::OptionalDeviceGuard guard(logits.device());
    x = dense(logits);
    lab = labels.contiguous();
    if (class_weight.has_value()) cw = class_weight->detach().to(at::kFloat).contiguous();
    loss = plain({}, x, at::kFloat);
    stats = plain({n * 3 * c + 2}, x, at::kFloat);
    const Tensor ws = bytes(sfh_ce_dice_workspace_bytes(&d), x);
    check(sfh_ce_dice_fwd(&d, code, ptr(x), (const int64_t*)ptr(lab), (const float*)ptr(cw), (float*)out_ptr(loss), (float*)out_ptr(stats), out_ptr(ws),
                          ws.defined() ? (size_t)ws.numel() : 0, stream_of(x)), "ce_dice_loss");
  }
  if (graph) {
    auto node = new_node<LossNode>();
    node->set_next_edges(torch::autograd::collect_next_edges(logits));
    node->logits.keep(x);
    node->labels.keep(lab);
    node->stats.keep(stats);
    node->class_weight.keep(cw);
    node->d = d;
    torch::autograd::set_history(loss, node);
  }
  return py::cast(loss);
}

void set_callbacks(py::object kernel_error, py::object note_device) {
  g_kernel_error = kernel_error.release().ptr();
  g_note_device = note_device.release().ptr();
}
void set_early_callbacks(py::object send, py::object join) {
  g_send_early = send.release().ptr();
  g_join_early = join.release().ptr();
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("set_callbacks", &set_callbacks);
  m.def("set_early_callbacks", &set_early_callbacks);
  py::class_<WeightBatch, std::shared_ptr<WeightBatch>>(m, "WeightBatch").def("__len__", &WeightBatch::size);
  m.def("launch_beside", [](WeightBatch& batch, int64_t stream_id, int64_t device_index) {
    launch_beside(batch, c10::Stream::unpack3(stream_id, (c10::DeviceIndex)device_index, c10::DeviceType::CUDA));
  });
  m.def("join_beside", &join_beside);
  m.def("batch_device", [](const WeightBatch& batch) { return batch.items.at(0).gy.device(); });
  m.def("finish_current_pass", &finish_current_pass, py::call_guard<py::gil_scoped_release>());
  m.def("waiting_weight_gradients", &waiting_weight_gradients);
  m.def("conv_forward", &conv_forward);
  m.def("conv_supported", &conv_supported);
  m.def("pack_master", &pack_master);
  m.def("conv_backward_data", &conv_backward_data);
  m.def("conv_backward_weight", &conv_backward_weight);
  m.def("record_conv", &record_conv);
  m.def("conv_transpose", &conv_transpose);
  m.def("group_norm", &group_norm);
  m.def("conv_norm", &conv_norm);
  m.def("max_pool", &max_pool);
  m.def("ce_dice_loss", &ce_dice_loss);
}
