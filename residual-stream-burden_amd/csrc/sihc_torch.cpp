// Native dispatch of the eager `sihc::` ops.
//
// The Python custom ops (sihc_hip/sublayer_kernels.py, event_ops.py, indexed.py, kernels.py)
// cost 50-120 us of interpreter and dispatcher time per forward and backward pair, more than
// the kernels of a small or ordinary call take. Each function here takes the arguments of one
// of those ops and, where the call is plain, allocates the outputs, enqueues the C-ABI call on
// the current stream and records one C++ autograd node whose backward does the same.
//
// Plain means: exactly the tensors and shapes that the op accepts, all packed, dense, on one
// GPU and not empty, of type torch.Tensor or torch.nn.Parameter, and nothing in force that has
// to see the op: no dispatch or function mode (tracing, fake tensors, selective checkpointing),
// no functorch transform, no forward-mode tangent, and no kernel or autocast rule that the
// program registered for the op itself. Anything else returns NotImplemented and
// the caller runs the Python op, which validates, raises and composes as it always did. The
// same holds in a backward: under create_graph, or where a mode or a wrapped tensor shows up
// there, the node calls the registered ops through the dispatcher. Inputs are kept with
// save_for_backward, so saved-tensor hooks and version checks apply, and undefined output
// gradients are materialised as zeros, as for the Python ops. An unpack hook may return another
// type, shape, layout or device than was saved, so every backward repeats the forward's checks on
// what it got, and leaves operands that do not fit to the registered ops, which raise.

#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstring>
#include <optional>
#include <string>
#include <tuple>
#include <vector>

#include "sihc_hip.h"

namespace {

using at::Tensor;
using at::TensorList;
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;

PyObject* parameter_type = nullptr;  // torch.nn.Parameter

struct Failure {};  // a C-ABI call returned an error in a forward: the Python op repeats and reports it

// ------------------------------------------------------------------ what may run here
bool plain_mode() {
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  if (!(tls.included_ - c10::default_included_set).empty()) return false;
  return !at::impl::torch_function_mode_enabled();
}
bool plain(const Tensor& t) {
  static const c10::DispatchKeySet special({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot,
                                            c10::DispatchKey::FuncTorchBatched,
                                            c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                            c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                            c10::DispatchKey::ZeroTensor});
  return t.defined() && t.is_cuda() && t.layout() == c10::kStrided && !t.is_quantized() && !t.is_nested() &&
         !t.key_set().has_any(special) && t.is_contiguous() && !t._fw_grad(0).defined();
}
bool below_autograd() {
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  return tls.excluded_.has(c10::DispatchKey::AutogradCUDA);
}
int dtype_code(const Tensor& t) {
  if (t.scalar_type() == at::kFloat) return SIHC_DTYPE_F32;
  return t.scalar_type() == at::kBFloat16 ? SIHC_DTYPE_BF16 : -1;
}
bool unwrap(PyObject* o, Tensor& t) {
  PyObject* type = reinterpret_cast<PyObject*>(Py_TYPE(o));
  if (type != THPVariableClass && type != parameter_type) return false;
  t = THPVariable_Unpack(o);
  return true;
}
bool unwrap_list(PyObject* o, std::vector<Tensor>& out) {
  if (!PyList_CheckExact(o) && !PyTuple_CheckExact(o)) return false;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
  out.resize(size_t(n));
  for (Py_ssize_t i = 0; i < n; ++i)
    if (!unwrap(PySequence_Fast_GET_ITEM(o, i), out[size_t(i)])) return false;
  return true;
}

struct Shape {
  int64_t batch, grid, cell, channels, slots;
};
// A square NHWC carrier of whole cells and weights whose last dimensions are [channels, slots].
bool carrier_shape(const Tensor& x, const Tensor& w, Shape& s) {
  if (x.dim() != 4 || w.dim() < 2 || x.numel() == 0 || dtype_code(x) < 0) return false;
  s.slots = w.size(-1);
  if (s.slots != 4 && s.slots != 16) return false;
  s.cell = s.slots == 4 ? 2 : 4;
  s.batch = x.size(0);
  s.channels = x.size(3);
  s.grid = x.size(1) / s.cell;
  return x.size(1) == x.size(2) && x.size(1) % s.cell == 0 && w.size(-2) == s.channels &&
         w.scalar_type() == x.scalar_type() && w.device() == x.device() && s.channels < (int64_t(1) << 31) &&
         s.grid < (int64_t(1) << 15);
}
bool token_shape(const Tensor& z, const Tensor& x, const Shape& s) {
  return z.dim() == 3 && z.size(0) == s.batch && z.size(1) == s.grid * s.grid && z.size(2) == s.channels &&
         z.scalar_type() == x.scalar_type() && z.device() == x.device();
}
bool index_shape(const Tensor& index, const Tensor& x, const Shape& s) {
  return index.scalar_type() == at::kInt && index.dim() == 2 && index.size(0) == s.batch &&
         index.size(1) == s.grid * s.grid && index.device() == x.device();
}

// Everything the launches below take for granted about their operands: asked by the Python
// entries of the arguments and by the backward nodes of the gradients and unpacked tensors.
bool read_fits(const Tensor& x, const Tensor& alpha, const Tensor& index, Shape& s) {
  return plain(x) && plain(alpha) && alpha.dim() == 3 && alpha.size(0) >= 1 && alpha.size(0) <= SIHC_MAX_EVENTS &&
         carrier_shape(x, alpha, s) && (!index.defined() || (plain(index) && index_shape(index, x, s)));
}
// (also the adjoint of the read, whose gradients have the updates' shape)
bool write_fits(const Tensor& x, TensorList updates, const Tensor& beta, const Tensor& index, Shape& s) {
  if (!read_fits(x, beta, index, s) || beta.size(0) != int64_t(updates.size())) return false;
  for (const Tensor& u : updates)
    if (!plain(u) || !token_shape(u, x, s)) return false;
  return true;
}
bool triangular_fits(const Tensor& base, TensorList updates, const Tensor& gamma) {
  if (!plain(base) || !plain(gamma) || base.dim() < 1 || base.numel() == 0 || dtype_code(base) < 0 ||
      updates.empty() || updates.size() > SIHC_MAX_EVENTS || gamma.dim() != 2 ||
      gamma.size(0) != int64_t(updates.size()) || gamma.size(1) != base.size(-1) ||
      gamma.device() != base.device() ||
      (gamma.scalar_type() != base.scalar_type() && gamma.scalar_type() != at::kFloat))
    return false;
  for (const Tensor& u : updates)
    if (!plain(u) || !u.sizes().equals(base.sizes()) || u.scalar_type() != base.scalar_type() ||
        u.device() != base.device())
      return false;
  return true;
}
bool event_fits(const Tensor& x, const Tensor& dz, const Tensor& beta, const Tensor& alpha) {
  Shape s{};
  return plain(x) && plain(dz) && plain(beta) && plain(alpha) && beta.dim() == 2 && carrier_shape(x, beta, s) &&
         token_shape(dz, x, s) && alpha.sizes().equals(beta.sizes()) && alpha.scalar_type() == x.scalar_type() &&
         alpha.device() == x.device();
}
bool gather_fits(const Tensor& x, const Tensor& index, int64_t slots) {
  if (!plain(x) || !plain(index)) return false;
  const int64_t k = slots == 4 ? 2 : 4;
  if (x.dim() != 4 || x.numel() == 0 || dtype_code(x) < 0 || (slots != 4 && slots != 16) ||
      x.size(1) != x.size(2) || x.size(1) % k != 0 || x.size(3) >= (int64_t(1) << 31))
    return false;
  const Shape s{x.size(0), x.size(1) / k, k, x.size(3), slots};
  // (the adjoint holds a batch row of the index in LDS: 16384 cells)
  return index_shape(index, x, s) && s.grid <= 128;
}
bool scatter_fits(const Tensor& cells, const Tensor& index) {
  if (!plain(cells) || !plain(index) || cells.dim() != 4 || cells.numel() == 0 || dtype_code(cells) < 0 ||
      (cells.size(2) != 4 && cells.size(2) != 16) || cells.size(1) > 16384 || cells.size(3) >= (int64_t(1) << 31))
    return false;
  Shape s{cells.size(0), 1, cells.size(2) == 4 ? 2 : 4, cells.size(3), cells.size(2)};
  while (s.grid * s.grid < cells.size(1)) ++s.grid;
  return s.grid * s.grid == cells.size(1) && index_shape(index, cells, s);
}

// ----------------------------------------------------------------------- the C-ABI calls
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream(); }
void check(int rc, bool forward) {
  if (rc == SIHC_OK) return;
  if (forward) throw Failure{};
  TORCH_CHECK(false, sihc_last_error());
}
struct Ptrs {
  void* p[SIHC_MAX_EVENTS] = {};
  explicit Ptrs(TensorList ts) {
    for (size_t i = 0; i < ts.size(); ++i) p[i] = ts[i].data_ptr();
  }
  const void* const* in() const { return const_cast<const void* const*>(p); }
};
const int32_t* index_ptr(const Tensor& index) { return index.defined() ? index.const_data_ptr<int32_t>() : nullptr; }
Tensor workspace(size_t bytes, const Tensor& like) {
  return at::empty({int64_t((std::max<size_t>(bytes, 4) + 63) / 64 * 16)}, like.options().dtype(at::kFloat));
}
Shape shape_of(const Tensor& x, const Tensor& w) {
  Shape s{};
  s.slots = w.size(-1);
  s.cell = s.slots == 4 ? 2 : 4;
  s.batch = x.size(0);
  s.channels = x.size(3);
  s.grid = x.size(1) / s.cell;
  return s;
}

variable_list run_read(const Tensor& x, const Tensor& alpha, const Tensor& index) {
  const c10::DeviceGuard guard(x.device());
  const Shape s = shape_of(x, alpha);
  variable_list out;
  out.reserve(size_t(alpha.size(0)));
  for (int64_t e = 0; e < alpha.size(0); ++e)
    out.push_back(at::empty({s.batch, s.grid * s.grid, s.channels}, x.options()));
  check(sihc_read(x.const_data_ptr(), alpha.const_data_ptr(), Ptrs(out).p, int(out.size()), s.batch, int(s.grid),
                  int(s.cell), int(s.channels), index_ptr(index), dtype_code(x), stream_of(x)),
        true);
  return out;
}
Tensor run_write(const Tensor& x, TensorList updates, const Tensor& beta, const Tensor& index) {
  const c10::DeviceGuard guard(x.device());
  const Shape s = shape_of(x, beta);
  Tensor out = at::empty_like(x);
  check(sihc_write(x.const_data_ptr(), Ptrs(updates).in(), beta.const_data_ptr(), out.data_ptr(), int(updates.size()),
                   s.batch, int(s.grid), int(s.cell), int(s.channels), 1, index_ptr(index), dtype_code(x),
                   dtype_code(beta), stream_of(x)),
        true);
  return out;
}
std::tuple<Tensor, Tensor> run_read_backward(const Tensor& x, TensorList grads, const Tensor& alpha,
                                             const Tensor& index) {
  const c10::DeviceGuard guard(x.device());
  const Shape s = shape_of(x, alpha);
  Tensor dx = at::empty_like(x), da = at::empty_like(alpha);
  const int events = int(grads.size());
  Tensor ws = workspace(
      sihc_weight_grad_workspace_size(events, s.batch, int(s.grid), int(s.cell), int(s.channels)), x);
  check(sihc_read_backward(x.const_data_ptr(), Ptrs(grads).in(), alpha.const_data_ptr(), dx.data_ptr(), da.data_ptr(),
                           events, s.batch, int(s.grid), int(s.cell), int(s.channels), index_ptr(index),
                           dtype_code(x), dtype_code(da), ws.data_ptr(), size_t(ws.numel()) * 4, stream_of(x)),
        false);
  return {dx, da};
}
std::tuple<variable_list, Tensor> run_write_backward(const Tensor& grad, TensorList updates, const Tensor& beta,
                                                     const Tensor& index) {
  const c10::DeviceGuard guard(grad.device());
  const Shape s = shape_of(grad, beta);
  variable_list dz;
  for (const Tensor& u : updates) dz.push_back(at::empty_like(u));
  Tensor db = at::empty_like(beta);
  const int events = int(updates.size());
  Tensor ws = workspace(
      sihc_weight_grad_workspace_size(events, s.batch, int(s.grid), int(s.cell), int(s.channels)), grad);
  check(sihc_write_backward(grad.const_data_ptr(), Ptrs(updates).in(), beta.const_data_ptr(), Ptrs(dz).p,
                            db.data_ptr(), events, s.batch, int(s.grid), int(s.cell), int(s.channels),
                            index_ptr(index), dtype_code(grad), dtype_code(db), ws.data_ptr(),
                            size_t(ws.numel()) * 4, stream_of(grad)),
        false);
  return {dz, db};
}

// --------------------------------------------------------------------------- dispatcher
template <typename Sig>
auto registered(const char* name) {
  return c10::Dispatcher::singleton().findSchemaOrThrow(name, "").typed<Sig>();
}
// A backward may launch directly: nothing recorded or in force (its operands are asked apart).
bool direct() { return !at::GradMode::is_enabled() && plain_mode(); }

// What a profiler sees of a call: the op's name and its arguments (made only if one looks).
using Args = std::vector<c10::IValue>;
Args listed(const Tensor& x, TensorList ts, const Tensor& w, const Tensor& index) {
  Args args{x, ts.vec(), w};
  if (index.defined()) args.emplace_back(index);
  return args;
}
// ------------------------------------------------------------------------ autograd nodes
struct ReadFn : torch::autograd::Function<ReadFn> {
  static constexpr bool is_traceable = true;
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& alpha,
                               const std::optional<Tensor>& index) {
    const Tensor idx = index.value_or(Tensor());
    ctx->save_for_backward({x, alpha, idx});
    return run_read(x, alpha, idx);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &alpha = saved[1], &index = saved[2];
    for (Tensor& g : grads) g = g.contiguous();
    std::tuple<Tensor, Tensor> r;
    Shape s{};
    if (direct() && write_fits(x, grads, alpha, index, s)) {
      RECORD_FUNCTION(index.defined() ? "sihc::indexed_read_backward" : "sihc::sublayer_read_backward",
                      listed(x, grads, alpha, index));
      r = run_read_backward(x, grads, alpha, index);
    } else if (index.defined()) {
      static auto op = registered<std::tuple<Tensor, Tensor>(const Tensor&, TensorList, const Tensor&,
                                                             const Tensor&)>("sihc::indexed_read_backward");
      r = op.call(x, grads, alpha, index);
    } else {
      static auto op = registered<std::tuple<Tensor, Tensor>(const Tensor&, TensorList, const Tensor&)>(
          "sihc::sublayer_read_backward");
      r = op.call(x, grads, alpha);
    }
    return {std::get<0>(r), std::get<1>(r), Tensor()};
  }
};

struct WriteFn : torch::autograd::Function<WriteFn> {
  static constexpr bool is_traceable = true;
  static Tensor forward(AutogradContext* ctx, const Tensor& x, TensorList updates, const Tensor& beta,
                        const std::optional<Tensor>& index) {
    const Tensor idx = index.value_or(Tensor());
    variable_list keep{beta, idx};
    keep.insert(keep.end(), updates.begin(), updates.end());
    ctx->save_for_backward(keep);
    return run_write(x, updates, beta, idx);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &beta = saved[0], &index = saved[1];
    const variable_list updates(saved.begin() + 2, saved.end());
    const Tensor grad = grads[0].contiguous();
    variable_list dz;
    Tensor db;
    Shape s{};
    if (direct() && write_fits(grad, updates, beta, index, s)) {
      RECORD_FUNCTION(index.defined() ? "sihc::indexed_write_backward" : "sihc::sublayer_write_backward",
                      listed(grad, updates, beta, index));
      std::tie(dz, db) = run_write_backward(grad, updates, beta, index);
    } else if (index.defined()) {
      static auto read =
          registered<std::vector<Tensor>(const Tensor&, const Tensor&, const Tensor&)>("sihc::indexed_read");
      static auto wgrad = registered<Tensor(const Tensor&, TensorList, const Tensor&, const Tensor&)>(
          "sihc::indexed_weight_grad");
      dz = read.call(grad, beta, index);
      db = wgrad.call(grad, updates, beta, index);
    } else {
      static auto read = registered<std::vector<Tensor>(const Tensor&, const Tensor&)>("sihc::sublayer_read");
      static auto wgrad =
          registered<Tensor(const Tensor&, TensorList, const Tensor&)>("sihc::sublayer_weight_grad");
      dz = read.call(grad, beta);
      db = wgrad.call(grad, updates, beta);
    }
    variable_list out{grad};
    out.insert(out.end(), dz.begin(), dz.end());
    out.push_back(db);
    out.emplace_back();
    return out;
  }
};

Tensor run_triangular(const Tensor& base, TensorList updates, const Tensor& gamma) {
  const c10::DeviceGuard guard(base.device());
  const int64_t c = base.size(-1);
  Tensor out = at::empty_like(base);
  check(sihc_triangular(base.const_data_ptr(), Ptrs(updates).in(), gamma.const_data_ptr(), out.data_ptr(),
                        int(updates.size()), base.numel() / c, int(c), dtype_code(base), dtype_code(gamma),
                        stream_of(base)),
        true);
  return out;
}
struct TriangularFn : torch::autograd::Function<TriangularFn> {
  static constexpr bool is_traceable = true;
  static Tensor forward(AutogradContext* ctx, const Tensor& base, TensorList updates, const Tensor& gamma) {
    variable_list keep{gamma};
    keep.insert(keep.end(), updates.begin(), updates.end());
    ctx->save_for_backward(keep);
    return run_triangular(base, updates, gamma);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor& gamma = saved[0];
    const variable_list updates(saved.begin() + 1, saved.end());
    const Tensor grad = grads[0].contiguous();
    variable_list out{grad};
    if (direct() && triangular_fits(grad, updates, gamma)) {
      RECORD_FUNCTION("sihc::sublayer_triangular_backward", listed(grad, updates, gamma, Tensor()));
      const c10::DeviceGuard device(grad.device());
      const int64_t c = grad.size(-1), rows = grad.numel() / c;
      const int active = int(updates.size());
      // one allocation, as the Python op's stacked result
      const Tensor stack = at::empty(
          [&] {
            std::vector<int64_t> sizes{active};
            sizes.insert(sizes.end(), grad.sizes().begin(), grad.sizes().end());
            return sizes;
          }(),
          grad.options());
      const variable_list dz = stack.unbind(0);
      const Tensor dg = at::empty_like(gamma);
      const Tensor ws = workspace(sihc_triangular_gamma_grad_workspace_size(active, rows, int(c)), grad);
      check(sihc_triangular_backward(grad.const_data_ptr(), Ptrs(updates).in(), gamma.const_data_ptr(), Ptrs(dz).p,
                                     dg.data_ptr(), active, rows, int(c), dtype_code(grad), dtype_code(gamma),
                                     dtype_code(dg), ws.data_ptr(), size_t(ws.numel()) * 4, stream_of(grad)),
            false);
      out.insert(out.end(), dz.begin(), dz.end());
      out.push_back(dg);
    } else {
      static auto op = registered<std::tuple<Tensor, Tensor>(const Tensor&, TensorList, const Tensor&)>(
          "sihc::sublayer_triangular_backward");
      const auto [stack, dg] = op.call(grad, updates, gamma);
      for (const Tensor& t : stack.unbind(0)) out.push_back(t);
      out.push_back(dg);
    }
    return out;
  }
};

variable_list run_event(const Tensor& x, const Tensor& dz, const Tensor& beta, const Tensor& alpha) {
  const c10::DeviceGuard guard(x.device());
  const Shape s = shape_of(x, beta);
  Tensor xo = at::empty_like(x), zo = at::empty_like(dz);
  check(sihc_event_forward(x.const_data_ptr(), dz.const_data_ptr(), beta.const_data_ptr(), alpha.const_data_ptr(),
                           xo.data_ptr(), zo.data_ptr(), s.batch, int(s.grid), int(s.cell), int(s.channels), nullptr,
                           dtype_code(x), stream_of(x)),
        true);
  return {xo, zo};
}
struct EventFn : torch::autograd::Function<EventFn> {
  static constexpr bool is_traceable = true;
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& dz, const Tensor& beta,
                               const Tensor& alpha) {
    variable_list out = run_event(x, dz, beta, alpha);
    ctx->save_for_backward({out[0], dz, beta, alpha});
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &xo = saved[0], &dz = saved[1], &beta = saved[2], &alpha = saved[3];
    const Tensor gx = grads[0].contiguous(), gz = grads[1].contiguous();
    if (!direct() || !event_fits(xo, dz, beta, alpha) || !event_fits(gx, gz, beta, alpha) ||
        !gx.sizes().equals(xo.sizes()) || gx.scalar_type() != xo.scalar_type()) {
      static auto op = registered<std::tuple<Tensor, Tensor, Tensor, Tensor>(
          const std::optional<Tensor>&, const std::optional<Tensor>&, const Tensor&, const Tensor&, const Tensor&,
          const Tensor&)>("sihc::event_write_read_backward");
      const auto [a, b, c, d] = op.call(gx, gz, xo, dz, beta, alpha);
      return {a, b, c, d};
    }
    RECORD_FUNCTION("sihc::event_write_read_backward", (Args{gx, gz, xo, dz, beta, alpha}));
    const c10::DeviceGuard device(xo.device());
    const Shape s = shape_of(xo, beta);
    Tensor dx = at::empty_like(xo), ddz = at::empty_like(dz), db = at::empty_like(beta), da = at::empty_like(alpha);
    const Tensor ws = workspace(
        sihc_event_backward_workspace_size(s.batch, int(s.grid), int(s.cell), int(s.channels)), xo);
    check(sihc_event_backward(gx.const_data_ptr(), gz.const_data_ptr(), xo.const_data_ptr(), dz.const_data_ptr(),
                              beta.const_data_ptr(), alpha.const_data_ptr(), dx.data_ptr(), ddz.data_ptr(),
                              db.data_ptr(), da.data_ptr(), s.batch, int(s.grid), int(s.cell), int(s.channels),
                              nullptr, dtype_code(xo), dtype_code(beta), ws.data_ptr(), size_t(ws.numel()) * 4,
                              stream_of(xo)),
          false);
    return {dx, ddz, db, da};
  }
};

// The block-wise stage-end write: one weight tensor per block, stacked for the C ABI; their
// gradients are rows of one [E, C, S] result in the weights' type.
struct BlockWriteFn : torch::autograd::Function<BlockWriteFn> {
  static constexpr bool is_traceable = true;
  static Tensor forward(AutogradContext* ctx, const Tensor& x, TensorList updates, TensorList betas,
                        const std::string& name) {
    ctx->saved_data["name"] = name;
    variable_list keep(updates.begin(), updates.end());
    keep.insert(keep.end(), betas.begin(), betas.end());
    ctx->save_for_backward(keep);
    return run_write(x, updates, at::stack(betas), Tensor());
  }
  // Updates and one [C, S] weight tensor each, of one type, for a carrier of 16 x 16 cells.
  static bool fits(const Tensor& x, const variable_list& updates, const variable_list& betas) {
    Shape s{};
    if (!plain(x)) return false;
    for (size_t i = 0; i < updates.size(); ++i) {
      const Tensor &u = updates[i], &w = betas[i];
      if (!plain(u) || !plain(w) || w.dim() != 2 || w.size(1) != betas[0].size(1) || !carrier_shape(x, w, s) ||
          s.grid != 16 || !token_shape(u, x, s))
        return false;
    }
    return true;
  }
  static variable_list finish(variable_list out) {
    out.emplace_back();  // the op's name
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const size_t n = saved.size() / 2;
    const variable_list updates(saved.begin(), saved.begin() + long(n)), betas(saved.begin() + long(n), saved.end());
    const Tensor grad = grads[0].contiguous();
    if (direct() && fits(grad, updates, betas)) {
      const Tensor beta = at::stack(betas);
      RECORD_FUNCTION("sihc::sublayer_write_backward", listed(grad, updates, beta, Tensor()));
      const auto [dz, db] = run_write_backward(grad, updates, beta, Tensor());
      variable_list out{grad};
      out.insert(out.end(), dz.begin(), dz.end());
      for (const Tensor& t : db.unbind(0)) out.push_back(t);
      return finish(std::move(out));
    }
    // the gradient ops of the legacy family, which widen bf16 updates and weights to fp32
    std::string name = ctx->saved_data["name"].toStringRef();  // sihc::final_accumulate_<tag>_traceable
    name.resize(name.rfind("_traceable"));
    auto gradient_op = [&](const char* which, const variable_list& rest) {
      const auto op = c10::Dispatcher::singleton().findSchemaOrThrow((name + which).c_str(), "");
      torch::jit::Stack stack{grad};
      for (const Tensor& t : rest) stack.emplace_back(t);
      op.callBoxed(stack);
      return stack.back().toTensor();
    };
    variable_list out{grad};
    for (const Tensor& t : gradient_op("_grad_dz_ptr", betas).unbind(0)) out.push_back(t);
    const variable_list db = gradient_op("_grad_beta_ptr", updates).unbind(0);
    for (size_t i = 0; i < n; ++i) out.push_back(db[i].to(betas[i].scalar_type()));
    return finish(std::move(out));
  }
};

Tensor run_gather(const Tensor& x, const Tensor& index, int64_t slots) {
  const c10::DeviceGuard guard(x.device());
  const int64_t k = slots == 4 ? 2 : 4, g = x.size(1) / k, c = x.size(3);
  Tensor cells = at::empty({x.size(0), g * g, slots, c}, x.options());
  check(sihc_gather_cells(x.const_data_ptr(), index_ptr(index), cells.data_ptr(), x.size(0), int(g), int(k), int(c),
                          dtype_code(x), stream_of(x)),
        true);
  return cells;
}
using CellsCall = int (*)(const void*, const int32_t*, void*, int64_t, int, int, int, int, void*);
Tensor run_scatter(CellsCall call, const Tensor& cells, const Tensor& index, bool forward) {
  const c10::DeviceGuard guard(cells.device());
  const int64_t k = cells.size(2) == 4 ? 2 : 4, c = cells.size(3), g = index.size(1);
  int64_t edge = 1;
  while (edge * edge < g) ++edge;
  Tensor x = at::empty({cells.size(0), edge * k, edge * k, c}, cells.options());
  check(call(cells.const_data_ptr(), index_ptr(index), x.data_ptr(), cells.size(0), int(edge), int(k), int(c),
             dtype_code(cells), stream_of(cells)),
        forward);
  return x;
}
struct GatherFn : torch::autograd::Function<GatherFn> {
  static constexpr bool is_traceable = true;
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& index, int64_t slots) {
    ctx->save_for_backward({index});
    return run_gather(x, index, slots);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const Tensor index = ctx->get_saved_variables()[0], grad = grads[0].contiguous();
    if (direct() && scatter_fits(grad, index)) {
      RECORD_FUNCTION("sihc::scatter_add_cells", (Args{grad, index}));
      return {run_scatter(sihc_scatter_add_cells, grad, index, false), Tensor(), Tensor()};
    }
    static auto op = registered<Tensor(const Tensor&, const Tensor&)>("sihc::scatter_add_cells");
    return {op.call(grad, index), Tensor(), Tensor()};
  }
};
struct ScatterFn : torch::autograd::Function<ScatterFn> {
  static constexpr bool is_traceable = true;
  static Tensor forward(AutogradContext* ctx, const Tensor& cells, const Tensor& index) {
    ctx->save_for_backward({index});
    ctx->saved_data["slots"] = cells.size(2);
    return run_scatter(sihc_scatter_cells, cells, index, true);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const Tensor index = ctx->get_saved_variables()[0], grad = grads[0].contiguous();
    const int64_t slots = ctx->saved_data["slots"].toInt();
    if (direct() && gather_fits(grad, index, slots)) {
      RECORD_FUNCTION("sihc::gather_cells", (Args{grad, index, slots}));
      return {run_gather(grad, index, slots), Tensor()};
    }
    static auto op = registered<Tensor(const Tensor&, const Tensor&, int64_t)>("sihc::gather_cells");
    return {op.call(grad, index, slots), Tensor()};
  }
};

// ------------------------------------------------------------------------ Python entries
PyObject* to_list(const variable_list& ts) {
  PyObject* out = PyList_New(Py_ssize_t(ts.size()));
  for (size_t i = 0; out && i < ts.size(); ++i) PyList_SET_ITEM(out, Py_ssize_t(i), THPVariable_Wrap(ts[i]));
  return out;
}
PyObject* not_implemented() { Py_RETURN_NOTIMPLEMENTED; }

// One Python entry: the op that it stands for.
struct Entry {
  c10::OperatorHandle op;
  const char* name() const { return op.operator_name().name.c_str(); }
  // A custom op has kernels under alias keys only: one under these is the program's own.
  bool overridden() const {
    return op.hasKernelForDispatchKey(c10::DispatchKey::CUDA) ||
           op.hasKernelForDispatchKey(c10::DispatchKey::AutogradCUDA) ||
           op.hasKernelForDispatchKey(c10::DispatchKey::AutocastCUDA);
  }
};
constexpr const char* ENTRY = "sihc_entry";
const Entry& entry_of(PyObject* self) { return *static_cast<Entry*>(PyCapsule_GetPointer(self, ENTRY)); }

// Run `f`; a C-ABI error, or a C++ exception, hands the call to the Python op, which repeats
// the checks and raises what it always raised. A Python exception comes from the caller's own
// code (a saved-tensor hook) and goes on to the caller: checkpointing ends its recomputation
// by raising from such a hook, which must not run again for the same call.
template <typename F>
PyObject* guarded(PyObject* self, F&& f) {
  try {
    const Entry& entry = entry_of(self);
    if (!plain_mode() || entry.overridden()) return not_implemented();
    return f();
  } catch (const Failure&) {
    return not_implemented();
  } catch (python_error& e) {
    e.restore();
    return nullptr;
  } catch (const std::exception&) {
    PyErr_Clear();
    return not_implemented();
  }
}
// f() as a call of the op of `self`, with the GIL released: a launch waits where the queue is full,
// and an allocation may wait for the device. (The registered ops release it around every dispatch
// and launch.) Saved-tensor hooks take it again for their own calls.
template <typename A, typename F>
auto call(PyObject* self, A&& args, F&& f) {
  RECORD_FUNCTION(entry_of(self).name(), args());
  struct Released {
    PyThreadState* state = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(state); }
  } released;
  return f();
}
// Below autograd (a custom op's own body, inference mode) and under no_grad nothing is recorded.
bool unrecorded() { return !at::GradMode::is_enabled() || below_autograd(); }
std::optional<Tensor> maybe(const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; }

PyObject* read_impl(PyObject* self, PyObject* const* args, bool indexed) {
  return guarded(self, [&]() -> PyObject* {
    Tensor x, alpha, index;
    Shape s{};
    if (!unwrap(args[0], x) || !unwrap(args[1], alpha) || (indexed && !unwrap(args[2], index))) return not_implemented();
    if ((indexed && !index.defined()) || !read_fits(x, alpha, index, s)) return not_implemented();
    return to_list(call(
        self, [&] { return index.defined() ? Args{x, alpha, index} : Args{x, alpha}; },
        [&] { return unrecorded() ? run_read(x, alpha, index) : ReadFn::apply(x, alpha, maybe(index)); }));
  });
}
PyObject* write_impl(PyObject* self, PyObject* const* args, bool indexed) {
  return guarded(self, [&]() -> PyObject* {
    Tensor x, beta, index;
    std::vector<Tensor> updates;
    Shape s{};
    if (!unwrap(args[0], x) || !unwrap_list(args[1], updates) || !unwrap(args[2], beta) ||
        (indexed && !unwrap(args[3], index)))
      return not_implemented();
    if ((indexed && !index.defined()) || !write_fits(x, updates, beta, index, s)) return not_implemented();
    return THPVariable_Wrap(call(self, [&] { return listed(x, updates, beta, index); }, [&] {
      return unrecorded() ? run_write(x, updates, beta, index)
                          : WriteFn::apply(x, TensorList(updates), beta, maybe(index));
    }));
  });
}

PyObject* py_read(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  return n == 2 ? read_impl(self, args, false) : not_implemented();
}
PyObject* py_indexed_read(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  return n == 3 ? read_impl(self, args, true) : not_implemented();
}
PyObject* py_write(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  return n == 3 ? write_impl(self, args, false) : not_implemented();
}
PyObject* py_indexed_write(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  return n == 4 ? write_impl(self, args, true) : not_implemented();
}
PyObject* py_triangular(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  if (n != 3) return not_implemented();
  return guarded(self, [&]() -> PyObject* {
    Tensor base, gamma;
    std::vector<Tensor> updates;
    if (!unwrap(args[0], base) || !unwrap_list(args[1], updates) || !unwrap(args[2], gamma)) return not_implemented();
    if (!triangular_fits(base, updates, gamma)) return not_implemented();
    return THPVariable_Wrap(call(self, [&] { return listed(base, updates, gamma, Tensor()); }, [&] {
      return unrecorded() ? run_triangular(base, updates, gamma)
                          : TriangularFn::apply(base, TensorList(updates), gamma);
    }));
  });
}
PyObject* py_event(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  if (n != 4) return not_implemented();
  return guarded(self, [&]() -> PyObject* {
    Tensor x, dz, beta, alpha;
    if (!unwrap(args[0], x) || !unwrap(args[1], dz) || !unwrap(args[2], beta) || !unwrap(args[3], alpha))
      return not_implemented();
    if (!event_fits(x, dz, beta, alpha)) return not_implemented();
    const variable_list out = call(
        self, [&] { return Args{x, dz, beta, alpha}; },
        [&] { return unrecorded() ? run_event(x, dz, beta, alpha) : EventFn::apply(x, dz, beta, alpha); });
    PyObject* pair = PyTuple_New(2);
    for (int i = 0; pair && i < 2; ++i) PyTuple_SET_ITEM(pair, i, THPVariable_Wrap(out[size_t(i)]));
    return pair;
  });
}

// (carrier edge, blocks, slots, x0, dz_0.., beta_0..)
PyObject* py_block_write(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  if (n < 4) return not_implemented();
  const long edge = PyLong_AsLong(args[0]), blocks = PyLong_AsLong(args[1]), slots = PyLong_AsLong(args[2]);
  if (n != 4 + 2 * blocks) return not_implemented();
  return guarded(self, [&]() -> PyObject* {
    Tensor x;
    std::vector<Tensor> updates(static_cast<size_t>(blocks)), betas(static_cast<size_t>(blocks));
    if (!unwrap(args[3], x)) return not_implemented();
    for (long i = 0; i < blocks; ++i)
      if (!unwrap(args[4 + i], updates[size_t(i)]) || !unwrap(args[4 + blocks + i], betas[size_t(i)]))
        return not_implemented();
    if (!BlockWriteFn::fits(x, updates, betas) || x.size(1) != edge || betas[0].size(1) != slots)
      return not_implemented();
    auto listing = [&] {
      Args all{x};
      for (const auto* ts : {&updates, &betas})
        for (const Tensor& t : *ts) all.emplace_back(t);
      return all;
    };
    return THPVariable_Wrap(call(self, listing, [&] {
      return unrecorded() ? run_write(x, updates, at::stack(betas), Tensor())
                          : BlockWriteFn::apply(x, TensorList(updates), TensorList(betas),
                                                std::string(entry_of(self).name()));
    }));
  });
}
PyObject* py_gather(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  if (n != 3 || !PyLong_CheckExact(args[2])) return not_implemented();
  const long slots = PyLong_AsLong(args[2]);
  return guarded(self, [&]() -> PyObject* {
    Tensor x, index;
    if (!unwrap(args[0], x) || !unwrap(args[1], index) || !gather_fits(x, index, slots)) return not_implemented();
    return THPVariable_Wrap(call(
        self, [&] { return Args{x, index, int64_t(slots)}; },
        [&] { return unrecorded() ? run_gather(x, index, slots) : GatherFn::apply(x, index, int64_t(slots)); }));
  });
}
PyObject* py_scatter(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  if (n != 2) return not_implemented();
  return guarded(self, [&]() -> PyObject* {
    Tensor cells, index;
    if (!unwrap(args[0], cells) || !unwrap(args[1], index) || !scatter_fits(cells, index)) return not_implemented();
    return THPVariable_Wrap(call(self, [&] { return Args{cells, index}; }, [&] {
      return unrecorded() ? run_scatter(sihc_scatter_cells, cells, index, true) : ScatterFn::apply(cells, index);
    }));
  });
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyMethodDef define(const char* name) {
  return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)), METH_FASTCALL, nullptr};
}
PyMethodDef entries[] = {
    define<py_read>("sublayer_read"),        define<py_write>("sublayer_write"),
    define<py_triangular>("sublayer_triangular"), define<py_event>("event_write_read"),
    define<py_indexed_read>("indexed_read"), define<py_indexed_write>("indexed_write"),
    define<py_block_write>("block_write"),   define<py_gather>("gather_cells"),
    define<py_scatter>("scatter_cells"),
};
// entry(name, op): the native entry `name` for the registered op `op` ("namespace::name")
PyObject* py_entry(PyObject*, PyObject* args) {
  const char *name, *op;
  if (!PyArg_ParseTuple(args, "ss", &name, &op)) return nullptr;
  for (PyMethodDef& def : entries) {
    if (std::strcmp(def.ml_name, name) != 0) continue;
    const auto handle = c10::Dispatcher::singleton().findSchema({op, ""});
    if (!handle) return PyErr_Format(PyExc_ValueError, "no registered op %s", op);
    PyObject* self = PyCapsule_New(new Entry{*handle}, ENTRY, [](PyObject* capsule) {
      delete static_cast<Entry*>(PyCapsule_GetPointer(capsule, ENTRY));
    });
    if (!self) return nullptr;
    PyObject* function = PyCFunction_New(&def, self);
    Py_DECREF(self);
    return function;
  }
  return PyErr_Format(PyExc_AttributeError, "no native entry %s", name);
}
PyMethodDef methods[] = {{"entry", py_entry, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_sihc_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__sihc_torch(void) {
  if (sihc_abi_version() != SIHC_ABI_VERSION)
    return PyErr_Format(PyExc_ImportError, "libsihc_hip.so has ABI %d, expected %d: rebuild it", sihc_abi_version(),
                        SIHC_ABI_VERSION);
  PyObject* nn = PyImport_ImportModule("torch.nn");
  if (!nn) return nullptr;
  parameter_type = PyObject_GetAttrString(nn, "Parameter");
  Py_DECREF(nn);
  if (!parameter_type) return nullptr;
  return PyModule_Create(&module);
}
