// The ops of flash_pop_amd as a CPython extension over the C ABI: argument checks, output and workspace allocation, launches and
// autograd nodes in native code.  With these in Python, behind ctypes, a call of a few microseconds of kernels was bound by its host
// work: 16 us a forward, 100 us and more a backward, which the autograd thread ran under the interpreter lock.  Before and
// after, per pass: decode layer step B1 H12 64 x 128 (three calls) 53 -> 21 us, forward B1 H4 T512 64 x 64 28 -> 17 us in three
// launches (12.5 us in the one it is now), forward + backward B32 H4 T2048 64 x 64 148 -> 118 us (now its kernels).
//
// Functions return NotImplemented when an argument is not what they take, or the call is being traced; the Python wrappers then
// raise the exception that says what is wrong, or make the call one that can be traced (flash_pop_amd/_ops.py).  Errors of the C ABI become RuntimeError.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/TracerMode.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <ATen/ops/zeros.h>
#include <c10/core/DeviceGuard.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>

#include <algorithm>
#include <initializer_list>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/flashpop_hip.h"
#include <torch_device.h>

namespace {

using at::Tensor;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// ---- calls of the C ABI -------------------------------------------------------------------------------------------------

void check(int rc) {
  if (rc != 0) throw std::runtime_error("flashpop_hip error " + std::to_string(rc) + ": " + fp_last_error());
}

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
using fpt::stream;

// The pass kernels must not be recorded into a HIP graph: instantiating a graph that holds them has crashed the host process
// (a segmentation fault inside the runtime, after every launch had been recorded without error).
void refuse_capture(const char* what) {
  if (fpt::capturing())
    throw std::runtime_error(std::string(what) +
                             " cannot be captured into a HIP graph with this ROCm / PyTorch build (graph instantiation crashes "
                             "the process); call it eagerly, outside torch.cuda.graph");
}

struct Shape {
  int B, T, H, dk, dv;
};
using Decays = std::vector<double>;

Tensor bytes_like(size_t n, const Tensor& t) { return at::empty({(int64_t)n}, t.options().dtype(at::kByte)); }
Tensor state_like(const Tensor& t, const Shape& s) { return at::empty({s.B, s.H, s.dk, s.dv}, t.options()); }
Tensor values_like(const Tensor& t, const Shape& s) { return at::empty({s.B, s.T, s.H, s.dv}, t.options()); }

// What a forward leaves for its backward: states every `every` tokens, or (every = 0), where the backward is cut too, the workspace
// of a forward that cut its sequences into segments, which holds the state at the start of every segment.
struct Kept {
  Tensor t;
  int every = 0;
};

void retention_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& s, const Decays& g, const Shape& n,
                   bool for_backward, Tensor& o, Tensor& s_out, Kept& kept) {
  c10::DeviceGuard guard(q.device());
  refuse_capture("retention_fwd");
  o = values_like(q, n);
  s_out = state_like(q, n);
  if (const size_t bytes = fp_retention_workspace_bytes(n.B, n.T, n.H, n.dk, n.dv)) {
    Tensor ws = bytes_like(bytes, q);   // (from a stream-ordered allocator: handing it back right after the call is safe)
    check(fp_retention_fwd_split(ptr(q), ptr(k), ptr(v), ptr(s), g.data(), ptr(o), ptr(s_out), n.B, n.T, n.H, n.dk, n.dv, ptr(ws),
                                 bytes, stream()));
    if (for_backward && fp_retention_backward_workspace_bytes(n.B, n.T, n.H, n.dk, n.dv)) kept.t = ws;
    return;
  }
  int every = 0;
  if (for_backward && fp_retention_checkpoint_bytes(n.B, n.T, n.H, n.dk, n.dv, &every)) {
    kept.every = every;
    kept.t = at::empty({n.B, n.T / every, n.H, n.dk, n.dv}, q.options());
    check(fp_retention_fwd_ckpt(ptr(q), ptr(k), ptr(v), ptr(s), g.data(), ptr(o), ptr(s_out), ptr(kept.t), every, n.B, n.T, n.H,
                                n.dk, n.dv, stream()));
    return;
  }
  check(fp_retention_fwd(ptr(q), ptr(k), ptr(v), ptr(s), g.data(), ptr(o), ptr(s_out), n.B, n.T, n.H, n.dk, n.dv, stream()));
}

void pop_retention_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& s, const Decays& g, int block,
                       const Shape& n, bool for_backward, Tensor& o, Tensor& states, Kept& kept) {
  c10::DeviceGuard guard(q.device());
  refuse_capture("pop_retention_fwd");
  o = values_like(q, n);
  states = at::empty({n.B, n.T / block, n.H, n.dk, n.dv}, q.options());
  if (const size_t bytes = fp_pop_retention_workspace_bytes(n.B, n.T, n.H, n.dk, n.dv, block)) {
    Tensor ws = bytes_like(bytes, q);
    check(fp_pop_retention_fwd_split(ptr(q), ptr(k), ptr(v), ptr(s), g.data(), ptr(o), ptr(states), n.B, n.T, n.H, n.dk, n.dv, block,
                                     ptr(ws), bytes, stream()));
    if (for_backward && fp_pop_retention_backward_workspace_bytes(n.B, n.T, n.H, n.dk, n.dv, block)) kept.t = ws;
    return;
  }
  check(fp_pop_retention_fwd(ptr(q), ptr(k), ptr(v), ptr(s), g.data(), ptr(o), states.numel() ? ptr(states) : nullptr, n.B, n.T,
                             n.H, n.dk, n.dv, block, stream()));
}

struct Grads {
  Tensor dq, dk, dv, ds0;
};

// block = 0: the plain op.  states_kept: the workspace in `kept` still holds the forward's segment states.
Grads retention_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& s, const Decays& g, const Shape& n,
                    const Tensor& d_o, const Tensor& d_s_out, const Tensor& d_blocks, int block, bool want_ds0, const Kept& kept,
                    bool states_kept) {
  c10::DeviceGuard guard(q.device());
  refuse_capture("retention_bwd");
  Grads r{at::empty_like(q), at::empty_like(k), at::empty_like(v), want_ds0 ? state_like(q, n) : Tensor()};
  if (block > 0) {
    const void* const d_states = d_blocks.defined() && d_blocks.numel() ? ptr(d_blocks) : nullptr;
    Tensor ws = kept.t;
    if (!ws.defined()) {
      if (const size_t bytes = fp_pop_retention_backward_workspace_bytes(n.B, n.T, n.H, n.dk, n.dv, block)) ws = bytes_like(bytes, q);
    }
    if (ws.defined())
      check(fp_pop_retention_bwd_split(ptr(q), ptr(k), ptr(v), ptr(s), g.data(), ptr(d_o), d_states, ptr(r.dq), ptr(r.dk), ptr(r.dv),
                                       ptr(r.ds0), n.B, n.T, n.H, n.dk, n.dv, block, ptr(ws), (size_t)ws.numel(),
                                       kept.t.defined() && states_kept, stream()));
    else
      check(fp_pop_retention_bwd(ptr(q), ptr(k), ptr(v), ptr(s), g.data(), ptr(d_o), d_states, ptr(r.dq), ptr(r.dk), ptr(r.dv),
                                 ptr(r.ds0), n.B, n.T, n.H, n.dk, n.dv, block, stream()));
    return r;
  }
  if (kept.t.defined() && kept.every > 0) {
    check(fp_retention_bwd_ckpt(ptr(q), ptr(k), ptr(v), ptr(s), g.data(), ptr(d_o), ptr(d_s_out), ptr(kept.t), kept.every,
                                ptr(r.dq), ptr(r.dk), ptr(r.dv), ptr(r.ds0), n.B, n.T, n.H, n.dk, n.dv, stream()));
    return r;
  }
  Tensor ws = kept.t;
  if (!ws.defined()) {
    if (const size_t bytes = fp_retention_backward_workspace_bytes(n.B, n.T, n.H, n.dk, n.dv)) ws = bytes_like(bytes, q);
  }
  if (ws.defined())
    check(fp_retention_bwd_split(ptr(q), ptr(k), ptr(v), ptr(s), g.data(), ptr(d_o), ptr(d_s_out), ptr(r.dq), ptr(r.dk), ptr(r.dv),
                                 ptr(r.ds0), n.B, n.T, n.H, n.dk, n.dv, ptr(ws), (size_t)ws.numel(),
                                 kept.t.defined() && states_kept, stream()));
  else
    check(fp_retention_bwd(ptr(q), ptr(k), ptr(v), ptr(s), g.data(), ptr(d_o), ptr(d_s_out), ptr(r.dq), ptr(r.dk), ptr(r.dv),
                           ptr(r.ds0), n.B, n.T, n.H, n.dk, n.dv, stream()));
  return r;
}

struct Suffixes {
  Tensor q, k, v;
};

void pop_fused_fwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& s, const Suffixes& x, const Decays& g, int block,
                   const Shape& n, Tensor& o, Tensor& o_sfx, Tensor& s_out) {
  c10::DeviceGuard guard(q.device());
  refuse_capture("pop_fused_fwd");
  o = values_like(q, n);
  o_sfx = at::empty_like(x.v);
  s_out = state_like(q, n);
  check(fp_pop_fused_fwd(ptr(q), ptr(k), ptr(v), ptr(s), ptr(x.q), ptr(x.k), ptr(x.v), g.data(), ptr(o), ptr(o_sfx), ptr(s_out), n.B,
                         n.T, n.H, n.dk, n.dv, block, (int)x.q.size(1), stream()));
}

Grads pop_fused_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& s, const Suffixes& x, const Decays& g, int block,
                    const Shape& n, const Tensor& d_o, const Tensor& d_o_sfx, const Tensor& d_s_out, bool want_ds0, Suffixes& dx) {
  c10::DeviceGuard guard(q.device());
  refuse_capture("pop_fused_bwd");
  Grads r{at::empty_like(q), at::empty_like(k), at::empty_like(v), want_ds0 ? state_like(q, n) : Tensor()};
  dx = Suffixes{at::empty_like(x.q), at::empty_like(x.k), at::empty_like(x.v)};
  check(fp_pop_fused_bwd(ptr(q), ptr(k), ptr(v), ptr(s), ptr(x.q), ptr(x.k), ptr(x.v), g.data(), ptr(d_o), ptr(d_o_sfx), ptr(d_s_out),
                         ptr(r.dq), ptr(r.dk), ptr(r.dv), ptr(dx.q), ptr(dx.k), ptr(dx.v), ptr(r.ds0), n.B, n.T, n.H, n.dk, n.dv,
                         block, (int)x.q.size(1), stream()));
  return r;
}

// start: one position per sequence, or undefined (start0)
void rotary(const Tensor& q, const Tensor& k, const Tensor& theta, const Tensor& start, int64_t start0, bool inverse, Tensor& q_out,
            Tensor& k_out) {
  c10::DeviceGuard guard(q.device());
  q_out = at::empty_like(q);
  if (k.defined()) k_out = at::empty_like(k);
  if (q.numel() == 0) return;
  check(fp_rotary_qk(ptr(q), ptr(k), ptr(q_out), ptr(k_out), theta.data_ptr<float>(),
                     start.defined() ? reinterpret_cast<const long long*>(start.data_ptr<int64_t>()) : nullptr, start0,
                     (int)q.size(0), (int)q.size(1), (int)q.size(2), (int)q.size(3), inverse, stream()));
}

Tensor gated_norm_fwd(const Tensor& r, const Tensor& g, double eps) {
  c10::DeviceGuard guard(r.device());
  Tensor out = at::empty_like(g);
  const int64_t H = r.size(-2), dv = r.size(-1);
  if (r.numel() == 0) return out;
  check(fp_gated_group_norm_fwd(ptr(r), ptr(g), ptr(out), r.numel() / (H * dv), (int)H, (int)dv, eps, stream()));
  return out;
}

void gated_norm_bwd(const Tensor& r, const Tensor& g, const Tensor& d_out, double eps, Tensor& d_r, Tensor& d_g) {
  c10::DeviceGuard guard(r.device());
  d_r = at::empty_like(r);
  d_g = at::empty_like(g);
  const int64_t H = r.size(-2), dv = r.size(-1);
  if (r.numel() == 0) return;
  check(fp_gated_group_norm_bwd(ptr(r), ptr(g), ptr(d_out), ptr(d_r), ptr(d_g), r.numel() / (H * dv), (int)H, (int)dv, eps, stream()));
}

// ---- autograd nodes -----------------------------------------------------------------------------------------------------

// The gradients that a backward returns.  The ops have no second derivative: under create_graph, where gradients without a history
// would count as constants, they get one that raises when it is differentiated.  `inputs`: what the gradients depend on.
template <typename... Inputs>
variable_list once_differentiable(variable_list&& gradients, bool create_graph, const Inputs&... inputs) {
  at::AutoGradMode grad_mode(create_graph);
  if (create_graph && torch::autograd::compute_requires_grad(inputs...)) {
    std::shared_ptr<torch::autograd::Node> error(
        new torch::autograd::Error("flash_pop_amd's ops can be differentiated once only", torch::autograd::collect_next_edges(inputs...)),
        torch::autograd::deleteNode);
    for (Tensor& g : gradients) {
      if (g.defined()) torch::autograd::set_history(g, error);
    }
  }
  return std::move(gradients);
}

// q, k, v, s and the decays of a retention op, saved for its backward
struct RetentionNode : public torch::autograd::Node {
  SavedVariable q, k, v, s;
  Decays decays;
  Shape n{};
  std::mutex mutex;

  void save(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& s_, Decays g, const Shape& shape) {
    q = SavedVariable(q_, false);
    k = SavedVariable(k_, false);
    v = SavedVariable(v_, false);
    s = SavedVariable(s_, false);
    decays = std::move(g);
    n = shape;
  }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex);
    q.reset_data();
    k.reset_data();
    v.reset_data();
    s.reset_data();
  }
  // a gradient as the kernels take it; an output that nobody differentiates contributes zeros (`shape`), or nothing (empty)
  static Tensor incoming(const Tensor& g, at::IntArrayRef shape, const Tensor& like) {
    if (g.defined()) return g.contiguous();
    return shape.empty() ? Tensor() : at::zeros(shape, like.options());
  }
};

// What a forward left (Kept) goes through SavedVariable like the inputs, so that saved-tensor hooks see all that a node holds.
struct KeepingNode : public RetentionNode {
  SavedVariable kept_tensor;
  int every = 0;

  void keep(const Kept& kept) {
    kept_tensor = SavedVariable(kept.t, false);
    every = kept.every;
  }
  void release_variables() override {
    RetentionNode::release_variables();
    std::lock_guard<std::mutex> lock(mutex);
    kept_tensor.reset_data();
  }
};

struct PlainBackward : public KeepingNode {
  bool spent = false;   // the kept workspace has been overwritten by a backward
  std::string name() const override { return "FusedChunkRetentionBackward"; }
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex);
    const bool create_graph = at::GradMode::is_enabled();
    at::AutoGradMode no_grad(false);
    const Tensor q_ = q.unpack(), k_ = k.unpack(), v_ = v.unpack(), s_ = s.unpack();
    const Tensor d_o = incoming(grads[0], {n.B, n.T, n.H, n.dv}, q_), d_s = incoming(grads[1], {}, q_);
    const Kept kept{kept_tensor.unpack(), every};
    // a forward that cut its sequences leaves its workspace: the first backward starts from the states in it and overwrites them,
    // a second one (retain_graph) recomputes them
    Grads r = retention_bwd(q_, k_, v_, s_, decays, n, d_o, d_s, Tensor(), 0, s_.defined() && task_should_compute_output(3), kept, !spent);
    spent = spent || (kept.t.defined() && kept.every == 0);
    return once_differentiable({r.dq, r.dk, r.dv, r.ds0}, create_graph, grads, q_, k_, v_, s_);
  }
};

struct PopBackward : public KeepingNode {
  int block = 0;
  bool spent = false;   // as in PlainBackward
  std::string name() const override { return "FlashPOPRetentionBackward"; }
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex);
    const bool create_graph = at::GradMode::is_enabled();
    at::AutoGradMode no_grad(false);
    const Tensor q_ = q.unpack(), k_ = k.unpack(), v_ = v.unpack(), s_ = s.unpack();
    const Tensor d_o = incoming(grads[0], {n.B, n.T, n.H, n.dv}, q_), d_b = incoming(grads[1], {}, q_);
    const Kept kept{kept_tensor.unpack(), 0};
    Grads r = retention_bwd(q_, k_, v_, s_, decays, n, d_o, Tensor(), d_b, block, s_.defined() && task_should_compute_output(3), kept, !spent);
    spent = spent || kept.t.defined();
    return once_differentiable({r.dq, r.dk, r.dv, r.ds0}, create_graph, grads, q_, k_, v_, s_);
  }
};

struct PopFusedBackward : public RetentionNode {
  SavedVariable qs, ks, vs;
  int block = 0;
  std::string name() const override { return "FlashPOPRetentionWithSuffixesBackward"; }
  void release_variables() override {
    RetentionNode::release_variables();
    std::lock_guard<std::mutex> lock(mutex);
    qs.reset_data();
    ks.reset_data();
    vs.reset_data();
  }
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex);
    const bool create_graph = at::GradMode::is_enabled();
    at::AutoGradMode no_grad(false);
    const Tensor q_ = q.unpack(), k_ = k.unpack(), v_ = v.unpack(), s_ = s.unpack();
    const Suffixes x{qs.unpack(), ks.unpack(), vs.unpack()};
    const Tensor d_o = incoming(grads[0], {n.B, n.T, n.H, n.dv}, q_), d_os = incoming(grads[1], x.v.sizes(), q_),
                 d_s = incoming(grads[2], {}, q_);
    Suffixes dx;
    Grads r = pop_fused_bwd(q_, k_, v_, s_, x, decays, block, n, d_o, d_os, d_s, s_.defined() && task_should_compute_output(3), dx);
    return once_differentiable({r.dq, r.dk, r.dv, r.ds0, dx.q, dx.k, dx.v}, create_graph, grads, q_, k_, v_, s_, x.q, x.k, x.v);
  }
};

// (This node and the next give an input whose output nobody differentiates a gradient of zeros, as the retention nodes do.)
struct RotaryBackward : public torch::autograd::Node {
  Tensor theta;          // a table of the module's own
  SavedVariable start;   // a tensor of the caller's, which may advance it in place before the backward runs: that is an error then
  std::mutex mutex;
  std::vector<int64_t> shape;   // of q and of k
  at::TensorOptions options;
  int64_t start0 = 0;
  bool inverse = false;
  std::string name() const override { return "RotaryQKBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex);
    start.reset_data();
  }
  variable_list apply(variable_list&& grads) override {
    const bool create_graph = at::GradMode::is_enabled();
    at::AutoGradMode no_grad(false);
    std::lock_guard<std::mutex> lock(mutex);
    const Tensor start_ = start.unpack();
    Tensor in[2], out[2], none;
    for (int i = 0; i < 2; ++i) {
      if (i < (int)grads.size() && grads[i].defined()) in[i] = grads[i].contiguous();
    }
    if (in[0].defined()) rotary(in[0], in[1], theta, start_, start0, !inverse, out[0], out[1]);
    else if (in[1].defined()) rotary(in[1], none, theta, start_, start0, !inverse, out[1], none);
    for (int i = 0; i < 2; ++i) {
      if (!out[i].defined() && task_should_compute_output(i)) out[i] = at::zeros(shape, options);
    }
    return once_differentiable({out[0], out[1]}, create_graph, grads);
  }
};

struct GatedNormBackward : public torch::autograd::Node {
  SavedVariable r, g;
  double eps = 0;
  std::mutex mutex;
  std::string name() const override { return "GatedGroupNormBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex);
    r.reset_data();
    g.reset_data();
  }
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex);
    const bool create_graph = at::GradMode::is_enabled();
    at::AutoGradMode no_grad(false);
    const Tensor r_ = r.unpack(), g_ = g.unpack();
    if (!grads[0].defined()) return {at::zeros(r_.sizes(), r_.options()), at::zeros(g_.sizes(), g_.options())};
    Tensor d_r, d_g;
    gated_norm_bwd(r_, g_, grads[0].contiguous(), eps, d_r, d_g);
    return once_differentiable({d_r, d_g}, create_graph, grads, r_, g_);
  }
};

template <typename N, typename... Inputs>
std::shared_ptr<N> make_node(const Inputs&... inputs) {
  std::shared_ptr<N> node(new N(), torch::autograd::deleteNode);
  node->set_next_edges(torch::autograd::collect_next_edges(inputs...));
  return node;
}

template <typename... Inputs>
bool differentiates(const Inputs&... inputs) {
  return at::GradMode::is_enabled() && torch::autograd::compute_requires_grad(inputs...);
}

// ---- Python arguments ---------------------------------------------------------------------------------------------------

// an optional tensor: None gives an undefined one
bool as_tensor(PyObject* o, Tensor& t) {
  if (o == Py_None) {
    t = Tensor();
    return true;
  }
  if (!THPVariable_Check(o)) return false;
  t = THPVariable_Unpack(o);
  return true;
}

// what has a length and gives, item by item, something that float() takes
void as_decays(PyObject* o, Decays& g) {
  if (PyObject_Length(o) < 0) throw python_error();   // (an iterator would be spent by the first look at it)
  PyObject* fast = PySequence_Fast(o, "head decays: a sequence of numbers expected");
  if (!fast) throw python_error();
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(fast);
  g.resize((size_t)n);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* item = PySequence_Fast_GET_ITEM(fast, i);
    if (PyFloat_CheckExact(item)) {
      g[(size_t)i] = PyFloat_AS_DOUBLE(item);
      continue;
    }
    PyObject* number = PyNumber_Float(item);
    if (!number) {
      Py_DECREF(fast);
      throw python_error();
    }
    g[(size_t)i] = PyFloat_AS_DOUBLE(number);
    Py_DECREF(number);
  }
  Py_DECREF(fast);
}

int64_t as_int(PyObject* o) {
  PyObject* i = PyNumber_Long(o);
  if (!i) throw python_error();
  const long long v = PyLong_AsLongLong(i);
  Py_DECREF(i);
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}
int64_t as_index(PyObject* o) { return PyLong_CheckExact(o) ? PyLong_AsLongLong(o) : as_int(o); }

// The ops have no forward-mode rule: a call with a tangent is refused, as an autograd Function without a jvp refuses it.
void refuse_tangents(std::initializer_list<const Tensor*> inputs) {
  for (const Tensor* t : inputs)
    TORCH_CHECK_NOT_IMPLEMENTED(!t->defined() || !t->_fw_grad(0).defined(), "flash_pop_amd's ops do not support forward mode AD");
}

// a block size as the C ABI takes it, whose sums stay below 2^31; any size beyond the sequence means no block
int64_t as_block(PyObject* o) { return std::min<int64_t>(as_int(o), 1 << 30); }

bool is_bf16(const Tensor& t) { return !t.defined() || (t.scalar_type() == at::kBFloat16 && fpt::on_device(t)); }

// q, k [B,T,H,dk], v [B,T,H,dv], s [B,H,dk,dv] or none, H decays: what _ops.check_retention asks for; makes them contiguous
bool retention_args(PyObject* const* a, Tensor& q, Tensor& k, Tensor& v, Tensor& s, Decays& g, Shape& n) {
  if (!as_tensor(a[0], q) || !as_tensor(a[1], k) || !as_tensor(a[2], v) || !as_tensor(a[3], s) || !q.defined() || !k.defined() || !v.defined())
    return false;
  if (q.dim() != 4 || !k.sizes().equals(q.sizes()) || v.dim() != 4 || !v.sizes().slice(0, 3).equals(q.sizes().slice(0, 3))) return false;
  as_decays(a[4], g);
  n = Shape{(int)q.size(0), (int)q.size(1), (int)q.size(2), (int)q.size(3), (int)v.size(3)};
  if ((int64_t)g.size() != n.H || !is_bf16(q) || !is_bf16(k) || !is_bf16(v) || !is_bf16(s)) return false;
  if (s.defined() && !s.sizes().equals({n.B, n.H, n.dk, n.dv})) return false;
  refuse_tangents({&q, &k, &v, &s});
  q = q.contiguous();
  k = k.contiguous();
  v = v.contiguous();
  if (s.defined()) s = s.contiguous();
  return true;
}

bool suffix_args(PyObject* const* a, const Shape& n, int block, Suffixes& x) {
  if (!as_tensor(a[0], x.q) || !as_tensor(a[1], x.k) || !as_tensor(a[2], x.v) || !x.q.defined() || !x.k.defined() || !x.v.defined())
    return false;
  if (x.q.dim() != 4 || !x.k.sizes().equals(x.q.sizes()) || x.v.dim() != 4 || !x.v.sizes().slice(0, 3).equals(x.q.sizes().slice(0, 3)))
    return false;
  if (x.q.size(0) != (int64_t)n.B * (n.T / block + 1) || x.q.size(2) != n.H || x.q.size(3) != n.dk || x.v.size(3) != n.dv) return false;
  if (!is_bf16(x.q) || !is_bf16(x.k) || !is_bf16(x.v)) return false;
  refuse_tangents({&x.q, &x.k, &x.v});
  x = Suffixes{x.q.contiguous(), x.k.contiguous(), x.v.contiguous()};
  return true;
}

PyObject* wrap(const Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}
template <typename... T>
PyObject* tuple_of(const T&... t) {
  PyObject* items[] = {wrap(t)...};
  PyObject* out = PyTuple_New(sizeof...(t));
  for (size_t i = 0; i < sizeof...(t); ++i) {
    if (!items[i] || !out) throw python_error();
    PyTuple_SET_ITEM(out, (Py_ssize_t)i, items[i]);
  }
  return out;
}

PyObject* not_implemented() { Py_RETURN_NOTIMPLEMENTED; }
// torch.jit.trace cannot see native ops and would keep their results as constants: the wrappers then call them through an autograd
// Function (flash_pop_amd/_ops.py), which it records.
bool traced() { return at::tracer::impl::is_dispatch_enabled(); }
bool count(Py_ssize_t n, Py_ssize_t want) {
  if (n == want) return true;
  PyErr_Format(PyExc_TypeError, "%zd arguments expected, got %zd", want, n);
  return false;
}
// lets go of the interpreter while native code runs
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

// ---- the ops ------------------------------------------------------------------------------------------------------------

// fused_chunk_retention(q, k, v, s, head_decays) -> (o, s_out)
PyObject* py_fused_chunk_retention(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (!count(nargs, 5)) return nullptr;
  if (traced()) return not_implemented();
  Tensor q, k, v, s, o, s_out;
  Decays g;
  Shape n;
  if (!retention_args(a, q, k, v, s, g, n)) return not_implemented();
  {
    NoGil free;
    const bool grad = differentiates(q, k, v, s);
    Kept kept;
    {
      at::AutoGradMode no_grad(false);
      retention_fwd(q, k, v, s, g, n, grad, o, s_out, kept);
    }
    if (grad) {
      auto node = make_node<PlainBackward>(q, k, v, s);
      node->save(q, k, v, s, std::move(g), n);
      node->keep(kept);
      torch::autograd::set_history(o, node);
      torch::autograd::set_history(s_out, node);
    }
  }
  return tuple_of(o, s_out);
  END_HANDLE_TH_ERRORS
}

// flash_pop_retention(q, k, v, s, head_decays, block_size) -> (o, block_states)
PyObject* py_flash_pop_retention(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (!count(nargs, 6)) return nullptr;
  if (traced()) return not_implemented();
  Tensor q, k, v, s, o, states;
  Kept kept;
  Decays g;
  Shape n;
  const int64_t block = as_block(a[5]);
  if (block < 1 || !retention_args(a, q, k, v, s, g, n)) return not_implemented();
  {
    NoGil free;
    const bool grad = differentiates(q, k, v, s);
    {
      at::AutoGradMode no_grad(false);
      pop_retention_fwd(q, k, v, s, g, (int)block, n, grad, o, states, kept);
    }
    if (grad) {
      auto node = make_node<PopBackward>(q, k, v, s);
      node->save(q, k, v, s, std::move(g), n);
      node->block = (int)block;
      node->keep(kept);
      torch::autograd::set_history(o, node);
      torch::autograd::set_history(states, node);
    }
  }
  return tuple_of(o, states);
  END_HANDLE_TH_ERRORS
}

// flash_pop_retention_with_suffixes(q, k, v, s, head_decays, block_size, q_sfx, k_sfx, v_sfx) -> (o, o_sfx, last_state)
PyObject* py_pop_with_suffixes(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (!count(nargs, 9)) return nullptr;
  if (traced()) return not_implemented();
  Tensor q, k, v, s, o, o_sfx, last;
  Suffixes x;
  Decays g;
  Shape n;
  const int64_t block = as_block(a[5]);
  if (block < 1 || !retention_args(a, q, k, v, s, g, n) || !suffix_args(a + 6, n, (int)block, x)) return not_implemented();
  {
    NoGil free;
    const bool grad = differentiates(q, k, v, s, x.q, x.k, x.v);
    {
      at::AutoGradMode no_grad(false);
      pop_fused_fwd(q, k, v, s, x, g, (int)block, n, o, o_sfx, last);
    }
    if (grad) {
      auto node = make_node<PopFusedBackward>(q, k, v, s, x.q, x.k, x.v);
      node->save(q, k, v, s, std::move(g), n);
      node->qs = SavedVariable(x.q, false);
      node->ks = SavedVariable(x.k, false);
      node->vs = SavedVariable(x.v, false);
      node->block = (int)block;
      torch::autograd::set_history(o, node);
      torch::autograd::set_history(o_sfx, node);
      torch::autograd::set_history(last, node);
    }
  }
  return tuple_of(o, o_sfx, last);
  END_HANDLE_TH_ERRORS
}

// decode_step(q, k, v, s, head_decays, in_place) -> (o, new state): q, k [B,H,dk], v [B,H,dv], s [B,H,dk,dv] or none
PyObject* py_decode_step(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (!count(nargs, 6)) return nullptr;
  if (traced()) return not_implemented();
  Tensor q, k, v, s, o, s_out;
  Decays g;
  if (!as_tensor(a[0], q) || !as_tensor(a[1], k) || !as_tensor(a[2], v) || !as_tensor(a[3], s) || !q.defined() || !k.defined() || !v.defined())
    return not_implemented();
  if (q.dim() != 3 || !k.sizes().equals(q.sizes()) || v.dim() != 3 || !v.sizes().slice(0, 2).equals(q.sizes().slice(0, 2)))
    return not_implemented();
  as_decays(a[4], g);
  const int B = (int)q.size(0), H = (int)q.size(1), dk = (int)q.size(2), dv = (int)v.size(2);
  const int in_place = PyObject_IsTrue(a[5]);
  if (in_place < 0) throw python_error();
  if ((int64_t)g.size() != H || !is_bf16(q) || !is_bf16(k) || !is_bf16(v) || !is_bf16(s)) return not_implemented();
  if (s.defined() && !s.sizes().equals({B, H, dk, dv})) return not_implemented();
  if (in_place && (!s.defined() || !s.is_contiguous())) return not_implemented();
  {
    NoGil free;
    at::AutoGradMode no_grad(false);
    c10::DeviceGuard guard(q.device());
    q = q.contiguous();
    k = k.contiguous();
    v = v.contiguous();
    if (s.defined()) s = s.contiguous();
    s_out = in_place ? s : at::empty({B, H, dk, dv}, q.options());
    o = at::empty({B, H, dv}, q.options());
    check(fp_retention_decode_step(ptr(q), ptr(k), ptr(v), ptr(s), g.data(), ptr(o), ptr(s_out), B, H, dk, dv, stream()));
    if (in_place && !s.is_inference()) s.unsafeGetTensorImpl()->bump_version();   // a graph node that saved this state must notice
  }
  return tuple_of(o, s_out);
  END_HANDLE_TH_ERRORS
}

// rotary_qk(q, k or None, theta, start, inverse) -> (q, k): q, k [B,T,H,d]; start a number or an integer tensor [B]
PyObject* py_rotary_qk(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (!count(nargs, 5)) return nullptr;
  if (traced()) return not_implemented();
  Tensor q, k, theta, start, q_out, k_out;
  int64_t start0 = 0;
  if (!as_tensor(a[0], q) || !as_tensor(a[1], k) || !as_tensor(a[2], theta) || !q.defined() || !theta.defined()) return not_implemented();
  if (!is_bf16(q) || !is_bf16(k) || q.dim() != 4 || (k.defined() && !k.sizes().equals(q.sizes()))) return not_implemented();
  if (theta.dim() != 1 || theta.size(0) != q.size(3) / 2 || theta.scalar_type() != at::kFloat || theta.device() != q.device())
    return not_implemented();
  if (THPVariable_Check(a[3])) {
    start = THPVariable_Unpack(a[3]);
    if (start.dim() != 1 || start.size(0) != q.size(0)) return not_implemented();
  } else {
    start0 = as_index(a[3]);
    if (start0 == -1 && PyErr_Occurred()) throw python_error();
  }
  const int inverse = PyObject_IsTrue(a[4]);
  if (inverse < 0) throw python_error();
  refuse_tangents({&q, &k});
  {
    NoGil free;
    q = q.contiguous();
    if (k.defined()) k = k.contiguous();
    theta = theta.contiguous();
    const bool grad = differentiates(q, k);
    {
      at::AutoGradMode no_grad(false);
      if (start.defined()) start = start.to(q.device(), at::kLong).contiguous();
      rotary(q, k, theta, start, start0, inverse, q_out, k_out);
    }
    if (grad) {
      auto node = make_node<RotaryBackward>(q, k);
      node->theta = theta;
      node->shape = q.sizes().vec();
      node->options = q.options();
      if (start.defined() && start.is_inference()) start = start.clone();   // (cannot be saved as it is)
      node->start = SavedVariable(start, false);
      node->start0 = start0;
      node->inverse = inverse;
      torch::autograd::set_history(q_out, node);
      if (k.defined()) torch::autograd::set_history(k_out, node);
    }
  }
  return tuple_of(q_out, k_out);
  END_HANDLE_TH_ERRORS
}

// gated_group_norm(r, g, eps) -> out: r [..., H, dv], g and out [..., H * dv]
PyObject* py_gated_group_norm(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (!count(nargs, 3)) return nullptr;
  if (traced()) return not_implemented();
  Tensor r, g, out;
  if (!as_tensor(a[0], r) || !as_tensor(a[1], g) || !r.defined() || !g.defined() || !is_bf16(r) || !is_bf16(g)) return not_implemented();
  if (r.dim() < 2 || g.dim() < 1 || g.numel() != r.numel() || g.size(-1) != r.size(-2) * r.size(-1)) return not_implemented();
  const double eps = PyFloat_AsDouble(a[2]);
  if (eps == -1.0 && PyErr_Occurred()) throw python_error();
  refuse_tangents({&r, &g});
  {
    NoGil free;
    r = r.contiguous();
    g = g.contiguous();
    const bool grad = differentiates(r, g);
    {
      at::AutoGradMode no_grad(false);
      out = gated_norm_fwd(r, g, eps);
    }
    if (grad) {
      auto node = make_node<GatedNormBackward>(r, g);
      node->r = SavedVariable(r, false);
      node->g = SavedVariable(g, false);
      node->eps = eps;
      torch::autograd::set_history(out, node);
    }
  }
  return wrap(out);
  END_HANDLE_TH_ERRORS
}

#define FP_METHOD(name, fn) \
  { name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(fn)), METH_FASTCALL, nullptr }
PyMethodDef methods[] = {
    FP_METHOD("fused_chunk_retention", py_fused_chunk_retention),
    FP_METHOD("flash_pop_retention", py_flash_pop_retention),
    FP_METHOD("flash_pop_retention_with_suffixes", py_pop_with_suffixes),
    FP_METHOD("decode_step", py_decode_step),
    FP_METHOD("rotary_qk", py_rotary_qk),
    FP_METHOD("gated_group_norm", py_gated_group_norm),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_native", "flash_pop_amd's ops over libflashpop_hip", -1, methods,
                          nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module_def); }
