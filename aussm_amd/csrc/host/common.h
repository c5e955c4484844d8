// Shared pieces of the native host path: the Python extension module _aussm_host (torch C++ API over the C ABI of
// libaussm_hip.so).  It holds what a call of the package does between Python and the kernel launches - argument
// checks, output and workspace allocation, the autograd graph node - so that a small call costs a few microseconds
// of host time.  (Python autograd functions over ctypes took 60-100 us per forward + backward.)
#pragma once
#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>

#include <optional>
#include <sstream>
#include <stdexcept>
#include <string>

#include "../../../include/aussm_hip.h"

namespace aussm_host {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;
typedef std::optional<Tensor> OptTensor;

// raised in Python as aussm_amd._lib.AussmError
struct AussmError : std::runtime_error {
  using std::runtime_error::runtime_error;
};
// raised in Python as RuntimeError, without the C++ call stack that TORCH_CHECK appends
struct ArgError : std::runtime_error {
  using std::runtime_error::runtime_error;
};

template <typename... T>
std::string cat(const T&... v) {
  std::ostringstream s;
  (s << ... << v);
  return s.str();
}
template <typename... T>
[[noreturn]] void fail(const T&... v) { throw ArgError(cat(v...)); }

inline std::string shape_str(at::IntArrayRef v) {
  std::ostringstream s;
  s << '(';
  for (size_t i = 0; i < v.size(); ++i) s << (i ? ", " : "") << v[i];
  if (v.size() == 1) s << ',';
  s << ')';
  return s.str();
}

inline void check(int code, const char* what) {
  if (code != 0) throw AussmError(cat(what, " failed with code ", code, ": ", aussm_error_string(code)));
}

template <typename T = float>
T* ptr(const Tensor& t) { return t.defined() ? static_cast<T*>(t.data_ptr()) : nullptr; }

inline void* cur_stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

inline Tensor opt(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }

// a tensor whose data pointer can be handed to a kernel: dense, no lazy conjugation or negation.
// (Called with gradient recording off: the graph node keeps the edges of the tensor it was given.)
inline Tensor dense(const Tensor& t) {
  if (!t.defined()) return t;
  Tensor r = t;
  if (r.is_conj()) r = r.resolve_conj();
  if (r.is_neg()) r = r.resolve_neg();
  return r.contiguous();
}

inline bool wants_grad(const Tensor& t) { return t.defined() && t.requires_grad(); }

inline Tensor empty_f32(at::IntArrayRef shape, const Tensor& like) {
  return at::empty(shape, at::TensorOptions().dtype(at::kFloat).device(like.device()));
}

// float32 (optional) tensor of a given shape
inline Tensor f32(const Tensor& t, const char* name, at::IntArrayRef shape) {
  if (!t.defined()) return t;
  if (t.scalar_type() != at::kFloat) fail("expected ", name, " to be float32, got torch.", t.scalar_type());
  if (t.sizes() != shape) fail("expected ", name, " of shape ", shape_str(shape), ", got ", shape_str(t.sizes()));
  return dense(t);
}

// every tensor of a call lies on one device (a kernel must not be handed an address of another)
inline bool same_device(const Tensor& ref, at::ArrayRef<Tensor> ts) {
  for (const Tensor& t : ts)
    if (t.defined() && t.device() != ref.device()) return false;
  return true;
}
inline void check_devices(const Tensor& ref, at::ArrayRef<Tensor> ts) {
  for (const Tensor& t : ts)
    if (t.defined() && t.device() != ref.device()) fail("expected all tensors of the call on ", ref.device(), ", got one on ", t.device());
}

// Buffers that kernels add into, cleared by one launch: own() is an allocation of its own, part() a piece of one that the
// parameter gradients of the call share (they are small and go together; a view takes half the time of an allocation).
// What a caller keeps so holds no gradient of an activation's size but itself.
struct Cleared {
  std::vector<float*> p;
  std::vector<size_t> n;
  Tensor parts;
  std::vector<int64_t> at;
  int64_t total = 0;
  void entry(const Tensor& t, int64_t floats) { p.push_back(ptr(t)); n.push_back((size_t)floats); }
  Tensor own(const Tensor& like, at::IntArrayRef shape, at::ScalarType type = at::kFloat) {
    const Tensor t = at::empty(shape, at::TensorOptions().dtype(type).device(like.device()));
    entry(t, t.numel() * (type == at::kComplexFloat ? 2 : 1));
    return t;
  }
  int part(int64_t floats) {
    at.push_back(total);
    total += (floats + 3) / 4 * 4;              // every part starts on 16 bytes
    return (int)at.size() - 1;
  }
  void clear(const Tensor& like) {
    if (total) {
      parts = empty_f32({total}, like);
      entry(parts, total);
    }
    if (!p.empty()) check(aussm_zero_many(p.data(), n.data(), (int)p.size(), cur_stream()), "aussm_zero_many");
  }
  float* data(int i) const { return ptr(parts) + at[i]; }
  Tensor view(int i, at::IntArrayRef shape) const {
    std::vector<int64_t> strides(shape.size());
    int64_t s = 1;
    for (size_t k = shape.size(); k-- > 0;) { strides[k] = s; s *= shape[k]; }
    return parts.as_strided(shape, strides, at[i]);
  }
};

// tensors that stand for others: wrapped by a function transform, or handled by Python
constexpr c10::DispatchKeySet WRAPPED{c10::DispatchKey::Batched, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                      c10::DispatchKey::Functionalize, c10::DispatchKey::Python};

// A graph node over saved tensors: `saved` are released together, and unpacking them after that raises torch's
// usual error about a second backward pass.
struct SavingNode : Node {
  std::vector<SavedVariable> saved;
  void save(std::initializer_list<Tensor> ts) {
    saved.reserve(ts.size());
    for (const Tensor& t : ts) saved.emplace_back(t, false);
  }
  // hooks stood between the forward pass and what `saved` hands out: it need not be what was saved, nor lie where it lay
  bool hooked() const {
    for (const auto& s : saved)
      if (s.has_hooks()) return true;
    return false;
  }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    for (auto& s : saved) s.reset_data();
  }
  variable_list apply(variable_list&& g) override {
    bool more = at::GradMode::is_enabled();            // create_graph
    for (const Tensor& t : g) more = more || (t.defined() && (t._fw_grad(0).defined() || t.key_set().has_any(WRAPPED)));
    return more ? composed(std::move(g)) : launched(g);
  }
  // gradients of the inputs from the kernels, called with gradient recording off
  virtual variable_list gradients(const variable_list& g) = 0;
  variable_list launched(const variable_list& g) {
    std::lock_guard<std::mutex> lock(mutex_);
    at::NoGradGuard no_grad;
    return gradients(g);
  }
  // ... and for a backward pass that is recorded itself (create_graph).  The kernels' gradients carry no graph: they can
  // be used, and differentiating them raises.  (The error hangs on the edges of this node and of the gradients
  // it got, so that every derivative that should pass through it does.)  Tangents and batches have no kernel.
  virtual variable_list composed(variable_list&& g) {
    for (const Tensor& t : g)
      if (t.defined() && t._fw_grad(0).defined()) fail(name(), ": forward-mode derivatives of this operator are not implemented");
    variable_list out = launched(g);
    if (!at::GradMode::is_enabled()) return out;
    torch::autograd::edge_list edges = torch::autograd::collect_next_edges(g);
    edges.insert(edges.end(), next_edges().begin(), next_edges().end());
    std::shared_ptr<Node> refusal(new torch::autograd::Error(cat(name(), ": second derivatives of this operator are not implemented"),
                                                             std::move(edges)),
                                  torch::autograd::deleteNode);
    for (Tensor& t : out)
      if (t.defined()) {
        t = t.detach();
        torch::autograd::set_history(t, refusal);
      }
    return out;
  }
};

template <typename N>
std::shared_ptr<N> make_node() { return std::shared_ptr<N>(new N(), torch::autograd::deleteNode); }

}  // namespace aussm_host
