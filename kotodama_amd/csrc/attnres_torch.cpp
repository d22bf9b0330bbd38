// Native call path of the eager PyTorch layer: a CPython extension that takes
// torch tensors, allocates the outputs on torch's caching allocator and calls
// the C ABI (include/attnres.h) on the current HIP stream.
//
// Every function handles the plain case only: dense contiguous ROCm tensors on
// one device in the kernels' dtypes, no dispatch or function mode, no functorch
// transform, no tracing.  For any other call it returns None with nothing done,
// and the Python layer (ops.py) takes the call through its own implementation
// or the registered op, which also report the errors.  A call the C ABI rejects
// is likewise left to that layer.
//
// Why: a routing call through the Python layer cost 11.4 us of host time (the
// launch itself about 3), several times a decode kernel's 2.7 us, and one
// under autograd through the op's Python forward and backward about 100 us.

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <c10/util/SmallVector.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <optional>
#include <vector>

#include "attnres.h"
#include "attnres_params.h"

namespace {

using at::Tensor;
using c10::DispatchKey;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ------------------------------------------------------------ plain calls --

// Dispatch keys whose tensors are not plain device memory (subclasses, functorch
// wrappers, lazy conjugation and the like).
constexpr c10::DispatchKeySet kOddKeys({DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::Functionalize,
                                        DispatchKey::FuncTorchBatched, DispatchKey::BatchedNestedTensor,
                                        DispatchKey::FuncTorchGradWrapper, DispatchKey::Batched,
                                        DispatchKey::Conjugate, DispatchKey::Negative, DispatchKey::ZeroTensor,
                                        DispatchKey::Tracer});

bool dtype_ok(at::ScalarType t) { return t == at::kBFloat16 || t == at::kFloat; }
int code(at::ScalarType t) { return t == at::kBFloat16 ? ATTNRES_DTYPE_BF16 : ATTNRES_DTYPE_F32; }

bool dense(const Tensor& t) { return t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(kOddKeys); }
bool plain(const Tensor& t) { return dense(t) && dtype_ok(t.scalar_type()) && t.is_contiguous(); }

// Nothing is watching the calls of this thread: no dispatch mode, no function
// mode, no functorch transform, no tracer.
bool unwatched() {
  if (c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled()) return false;
  const auto tls = c10::impl::tls_local_dispatch_key_set();
  if (tls.included_.has(DispatchKey::FuncTorchDynamicLayerFrontMode) ||
      tls.included_.has(DispatchKey::FuncTorchDynamicLayerBackMode) || tls.included_.has(DispatchKey::Functionalize) ||
      tls.included_.has(DispatchKey::Python) || tls.included_.has(DispatchKey::FuncTorchVmapMode))
    return false;
  return !torch::jit::tracer::isTracing();
}

// Makes the tensors' device current for the C-ABI call; `stream` is its current stream.
struct OnDevice {
  c10::OptionalDeviceGuard guard;
  void* stream;
  explicit OnDevice(const Tensor& t) {
    const c10::Device dev = t.device();
    if (c10::hip::current_device() != dev.index()) guard.reset_device(dev);
    stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  }
};

Tensor empty(at::IntArrayRef size, at::ScalarType dtype, c10::Device device) {
  return Tensor(at::detail::empty_cuda(size, dtype, device, std::nullopt));
}

using Dims = c10::SmallVector<int64_t, 6>;

// The parameters of one call: query (D,) or (Q, D), gain (D,) or undefined.
struct Fold {
  int64_t nq = 1;
  bool ok = false;
  Fold(const Tensor& query, const Tensor& gain, int64_t d, const Tensor& ref) {
    if (!plain(query) || query.get_device() != ref.get_device()) return;
    if (query.dim() != 1 && query.dim() != 2) return;
    if (query.size(-1) != d) return;
    nq = query.dim() == 1 ? 1 : query.size(0);
    if (gain.defined() && (!plain(gain) || gain.get_device() != ref.get_device() ||
                           gain.scalar_type() != query.scalar_type() || gain.dim() != 1 || gain.size(0) != d))
      return;
    ok = nq >= 1;
  }
};

const void* ptr(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }
template <typename T>
T* out_ptr(const Tensor& t) {
  return t.defined() && t.numel() ? static_cast<T*>(t.mutable_data_ptr()) : nullptr;
}

// A list of S row blocks (..., D) of one shape and dtype: the slots of a stacked
// buffer or separate tensors.
struct Sources {
  const void* ptrs[ATTNRES_MAX_SOURCES];
  int s = 0;
  int64_t n = 1, d = 0;
  at::ScalarType dtype = at::kFloat;
  Dims batch;
  Tensor ref;
  bool ok = false;

  static Sources stacked(const Tensor& buf, int64_t num) {
    Sources r;
    if (!plain(buf) || buf.dim() < 2 || num < 0 || num > buf.size(0) || num > ATTNRES_MAX_SOURCES) return r;
    r.shape(buf, 1);
    const int64_t slot = r.n * r.d * (int64_t)buf.element_size();
    const char* base = static_cast<const char*>(buf.const_data_ptr());
    for (int64_t i = 0; i < num; ++i) r.ptrs[i] = base + i * slot;
    r.s = (int)num;
    r.ok = r.d > 0;
    return r;
  }
  static Sources list(const std::vector<Tensor>& srcs) {
    Sources r;
    if (srcs.empty() || srcs.size() > ATTNRES_MAX_SOURCES || srcs[0].dim() < 1) return r;
    const Tensor& a = srcs[0];
    for (const Tensor& t : srcs) {
      if (!plain(t) || t.scalar_type() != a.scalar_type() || t.get_device() != a.get_device() || t.sizes() != a.sizes())
        return r;
      r.ptrs[r.s++] = t.const_data_ptr();
    }
    r.shape(a, 0);
    r.ok = r.d > 0;
    return r;
  }

 private:
  void shape(const Tensor& t, int64_t first) {
    ref = t;
    dtype = t.scalar_type();
    d = t.size(-1);
    for (int64_t i = first; i < t.dim() - 1; ++i) {
      batch.push_back(t.size(i));
      n *= t.size(i);
    }
  }
};

// A profiler's event of a launch that does not pass the dispatcher, under the op's name.
#define ATTNRES_RECORD(name) RECORD_FUNCTION(name, c10::ArrayRef<const c10::IValue>{})

// ---------------------------------------------------------------- routing --

struct Routed {
  Tensor out, weights, lse, inv_rms, logits;
};

// One attnres_route_fwd call, `op` in a profiler; false when the call is not for this path.
// `squeeze`: one query's rows without the leading query dimension.
bool route_rows(const char* op, const Sources& src, const Tensor& query, const Tensor& gain, double eps,
                at::ScalarType out_dtype, bool want_weights, bool want_lse, bool want_aux, bool squeeze, Routed* r) {
  if (!src.ok || !dtype_ok(out_dtype)) return false;
  const Fold fold(query, gain, src.d, src.ref);
  if (!fold.ok) return false;
  ATTNRES_RECORD(op);
  const c10::Device dev = src.ref.device();
  const int64_t nq = fold.nq;
  Dims size;
  if (!(squeeze && nq == 1)) size.push_back(nq);
  size.append(src.batch.begin(), src.batch.end());
  size.push_back(src.d);
  r->out = empty(size, out_dtype, dev);
  Dims q_batch{nq};
  q_batch.append(src.batch.begin(), src.batch.end());
  if (want_weights) {
    Dims w{nq, src.s};
    w.append(src.batch.begin(), src.batch.end());
    r->weights = empty(w, at::kFloat, dev);
  }
  if (want_lse) r->lse = empty(q_batch, at::kFloat, dev);
  if (want_aux) {
    Dims a(src.batch.begin(), src.batch.end());
    a.push_back(src.s);
    r->inv_rms = empty(a, at::kFloat, dev);
    Dims l(q_batch.begin(), q_batch.end());
    l.push_back(src.s);
    r->logits = empty(l, at::kFloat, dev);
  }
  const OnDevice on(src.ref);
  return attnres_route_fwd(src.ptrs, src.s, src.n, (int)src.d, src.d, code(src.dtype), ptr(query), ptr(gain), (int)nq,
                           code(query.scalar_type()), (float)eps, out_ptr<void>(r->out), code(out_dtype), src.d,
                           src.n * src.d, out_ptr<float>(r->weights), out_ptr<float>(r->lse),
                           out_ptr<float>(r->inv_rms), out_ptr<float>(r->logits), on.stream) == ATTNRES_OK;
}

Tensor workspace(int64_t bytes, c10::Device dev) {
  return empty({std::max<int64_t>(1, (bytes + 3) / 4)}, at::kFloat, dev);
}

// Backward over contiguous sources into `grads` (attnres_route_bwd, or
// attnres_route_bwd_queries for Q > 1); false when not for this path.
bool route_rows_bwd(const Sources& src, void* const* grads, const Tensor& query, const Tensor& gain, double eps,
                    Tensor g_out, Tensor g_lse, const void* const* adds, Tensor* dq, Tensor* dg) {
  if (!src.ok || src.s < 1 || src.n < 1) return false;
  const Fold fold(query, gain, src.d, src.ref);
  if (!fold.ok || !dense(g_out) || !dtype_ok(g_out.scalar_type()) || g_out.get_device() != src.ref.get_device() ||
      g_out.numel() != fold.nq * src.n * src.d)
    return false;
  if (g_lse.defined() &&
      (!dense(g_lse) || g_lse.get_device() != src.ref.get_device() || g_lse.numel() != fold.nq * src.n))
    return false;
  g_out = g_out.contiguous();
  if (g_lse.defined()) g_lse = g_lse.to(at::kFloat).contiguous();
  const c10::Device dev = src.ref.device();
  *dq = empty(query.sizes(), query.scalar_type(), dev);
  if (gain.defined()) *dg = empty(gain.sizes(), gain.scalar_type(), dev);
  const OnDevice on(src.ref);
  int64_t bytes = 0;
  if (fold.nq > 1) {
    if (adds != nullptr ||
        attnres_route_bwd_queries_workspace_size(src.n, (int)src.d, src.s, (int)fold.nq, &bytes) != ATTNRES_OK)
      return false;
    const Tensor ws = workspace(bytes, dev);
    return attnres_route_bwd_queries(src.ptrs, src.s, src.n, (int)src.d, src.d, code(src.dtype), ptr(query), ptr(gain),
                                     (int)fold.nq, code(query.scalar_type()), (float)eps, ptr(g_out),
                                     code(g_out.scalar_type()), src.d, src.n * src.d,
                                     static_cast<const float*>(ptr(g_lse)), grads, src.d, out_ptr<void>(ws),
                                     ws.numel() * 4, out_ptr<void>(*dq), out_ptr<void>(*dg), on.stream) == ATTNRES_OK;
  }
  if (attnres_route_bwd_workspace_size(src.n, (int)src.d, &bytes) != ATTNRES_OK) return false;
  const Tensor ws = workspace(bytes, dev);
  if (adds != nullptr)
    return attnres_route_bwd_add(src.ptrs, src.s, src.n, (int)src.d, src.d, code(src.dtype), ptr(query), ptr(gain),
                                 code(query.scalar_type()), (float)eps, ptr(g_out), code(g_out.scalar_type()), src.d,
                                 static_cast<const float*>(ptr(g_lse)), grads, adds, src.d, out_ptr<void>(ws),
                                 ws.numel() * 4, out_ptr<void>(*dq), out_ptr<void>(*dg), on.stream) == ATTNRES_OK;
  return attnres_route_bwd(src.ptrs, src.s, src.n, (int)src.d, src.d, code(src.dtype), ptr(query), ptr(gain),
                           code(query.scalar_type()), (float)eps, ptr(g_out), code(g_out.scalar_type()), src.d,
                           static_cast<const float*>(ptr(g_lse)), grads, src.d, out_ptr<void>(ws), ws.numel() * 4,
                           out_ptr<void>(*dq), out_ptr<void>(*dg), on.stream) == ATTNRES_OK;
}

// The registered op, called through the dispatcher (the cases the direct
// launches leave out, and backward passes that are themselves recorded).
template <typename... Args>
std::vector<c10::IValue> call_op(const char* name, Args&&... args) {
  const auto op = c10::Dispatcher::singleton().findSchemaOrThrow(name, "");
  std::vector<c10::IValue> stack{c10::IValue(std::forward<Args>(args))...};
  op.callBoxed(&stack);
  return stack;
}
std::optional<Tensor> opt(const Tensor& t) { return t.defined() ? std::optional<Tensor>(t) : std::nullopt; }

// route over a stacked buffer under autograd: the registered op's formula
// (ops.py: _route_backward, route_bwd) without its Python.  Only differentiable
// outputs (the rows, the lse) pass through the function: compiled autograd
// takes no function with others.  is_traceable: the backward is made of calls
// that compiled autograd can trace (under it no call is plain and the ops run).
struct RouteStacked : public torch::autograd::Function<RouteStacked> {
  static constexpr bool is_traceable = true;
  static variable_list forward(AutogradContext* ctx, const Tensor& buf, const Tensor& query,
                               const std::optional<Tensor>& gain_opt, const Routed* r, int64_t num, double eps,
                               bool zero_inactive) {
    const Tensor gain = gain_opt.value_or(Tensor());
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({buf, query, gain});
    ctx->saved_data["num"] = num;
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["zero"] = zero_inactive;
    ctx->saved_data["dtype"] = (int64_t)r->out.scalar_type();
    ctx->saved_data["shape"] = r->out.sizes().vec();
    ctx->saved_data["has_lse"] = r->lse.defined();
    variable_list out{r->out};
    if (r->lse.defined()) out.push_back(r->lse);
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list g) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &buf = saved[0], &query = saved[1], &gain = saved[2];
    const bool has_gain = gain.defined();
    variable_list res(7);
    Tensor g_out = g[0], g_lse = ctx->saved_data["has_lse"].toBool() ? g[1] : Tensor();
    if (!g_out.defined() && !g_lse.defined()) return res;
    if (!g_out.defined())
      g_out = at::zeros(ctx->saved_data["shape"].toIntVector(),
                        buf.options().dtype((at::ScalarType)ctx->saved_data["dtype"].toInt()));
    const int64_t num = ctx->saved_data["num"].toInt();
    const double eps = ctx->saved_data["eps"].toDouble();
    const bool zero = ctx->saved_data["zero"].toBool();
    Tensor gb, dq, dg;
    bool done = false;
    if (!at::GradMode::is_enabled() && unwatched()) {
      const Sources src = Sources::stacked(buf, num);
      if (src.ok && src.s >= 1 && src.n >= 1) {
        ATTNRES_RECORD("attnres_hip::route_bwd");
        gb = empty(buf.sizes(), buf.scalar_type(), buf.device());
        const int64_t slot = src.n * src.d * (int64_t)buf.element_size();
        void* grads[ATTNRES_MAX_SOURCES];
        for (int i = 0; i < src.s; ++i) grads[i] = static_cast<char*>(gb.mutable_data_ptr()) + i * slot;
        if (zero && num < buf.size(0)) gb.slice(0, num).zero_();
        done = route_rows_bwd(src, grads, query, gain, eps, g_out, g_lse, nullptr, &dq, &dg);
      }
    }
    if (!done) {
      const auto st = call_op("attnres_hip::route_bwd", buf, num, query, opt(gain), eps, g_out, opt(g_lse), zero);
      gb = st[0].toTensor();
      dq = st[1].toTensor();
      dg = has_gain ? st[2].toTensor() : Tensor();
    }
    // edges of the tensor inputs: buf, query and, where given, gain
    if (ctx->needs_input_grad(0)) res[0] = gb;
    if (ctx->needs_input_grad(1)) res[1] = dq;
    if (has_gain && ctx->needs_input_grad(2)) res[2] = dg;
    return res;
  }
};

// The same over a list of separate blocks (ops.py: _route_list_backward, route_list_bwd).
struct RouteList : public torch::autograd::Function<RouteList> {
  static constexpr bool is_traceable = true;
  static variable_list forward(AutogradContext* ctx, at::TensorList blocks, const Tensor& query,
                               const std::optional<Tensor>& gain_opt, const Routed* r, double eps) {
    const Tensor gain = gain_opt.value_or(Tensor());
    ctx->set_materialize_grads(false);
    variable_list keep(blocks.begin(), blocks.end());
    keep.push_back(query);
    keep.push_back(gain);
    ctx->save_for_backward(keep);
    ctx->saved_data["eps"] = eps;
    ctx->saved_data["dtype"] = (int64_t)r->out.scalar_type();
    ctx->saved_data["shape"] = r->out.sizes().vec();
    ctx->saved_data["has_lse"] = r->lse.defined();
    variable_list out{r->out};
    if (r->lse.defined()) out.push_back(r->lse);
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list g) {
    auto saved = ctx->get_saved_variables();
    const Tensor gain = saved.back(), query = saved[saved.size() - 2];
    saved.resize(saved.size() - 2);
    const size_t s = saved.size();
    variable_list res(s + 4);
    Tensor g_out = g[0], g_lse = ctx->saved_data["has_lse"].toBool() ? g[1] : Tensor();
    if (!g_out.defined() && !g_lse.defined()) return res;
    if (!g_out.defined())
      g_out = at::zeros(ctx->saved_data["shape"].toIntVector(),
                        query.options().dtype((at::ScalarType)ctx->saved_data["dtype"].toInt()));
    const double eps = ctx->saved_data["eps"].toDouble();
    Tensor dq, dg;
    std::vector<Tensor> grads;
    bool done = false;
    if (!at::GradMode::is_enabled() && unwatched()) {
      const Sources src = Sources::list(saved);
      if (src.ok && src.n >= 1) {
        ATTNRES_RECORD("attnres_hip::route_list_bwd");
        void* ptrs[ATTNRES_MAX_SOURCES];
        for (size_t i = 0; i < s; ++i) {
          grads.push_back(empty(saved[i].sizes(), saved[i].scalar_type(), saved[i].device()));
          ptrs[i] = grads[i].mutable_data_ptr();
        }
        done = route_rows_bwd(src, ptrs, query, gain, eps, g_out, g_lse, nullptr, &dq, &dg);
      }
    }
    if (!done) {
      const auto st = call_op("attnres_hip::route_list_bwd", saved, query, opt(gain), eps, g_out, opt(g_lse));
      grads = st[0].toTensorVector();
      dq = st[1].toTensor();
      dg = gain.defined() ? st[2].toTensor() : Tensor();
    }
    for (size_t i = 0; i < s; ++i) {
      if (ctx->needs_input_grad(i)) res[i] = grads[i];
    }
    if (ctx->needs_input_grad(s)) res[s] = dq;
    if (gain.defined() && ctx->needs_input_grad(s + 1)) res[s + 1] = dg;
    return res;
  }
};

// ------------------------------------------------------------------ merge --

bool merge_rows(const Tensor& p, const Tensor& query, const Tensor& inter, const Tensor& lse, double eps, Tensor* out) {
  if (!plain(p) || !plain(inter) || !plain(query) || !plain(lse) || p.dim() < 1) return false;
  const int64_t d = p.size(-1);
  if (d < 1 || inter.sizes() != p.sizes() || query.dim() != 1 || query.size(0) != d ||
      lse.scalar_type() != at::kFloat || lse.sizes() != p.sizes().slice(0, p.dim() - 1))
    return false;
  for (const Tensor* t : {&query, &inter, &lse})
    if (t->get_device() != p.get_device()) return false;
  ATTNRES_RECORD("attnres_hip::merge");
  *out = empty(inter.sizes(), inter.scalar_type(), inter.device());
  const OnDevice on(p);
  return attnres_merge_fwd(ptr(p), p.numel() / d, (int)d, code(p.scalar_type()), ptr(query), code(query.scalar_type()),
                           ptr(inter), code(inter.scalar_type()), static_cast<const float*>(ptr(lse)), (float)eps,
                           out_ptr<void>(*out), nullptr, nullptr, on.stream) == ATTNRES_OK;
}

struct Merge : public torch::autograd::Function<Merge> {
  static constexpr bool is_traceable = true;
  static Tensor forward(AutogradContext* ctx, const Tensor& p, const Tensor& query, const Tensor& inter,
                        const Tensor& lse, const Tensor* out, double eps) {
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({p, query, inter, lse});
    ctx->saved_data["eps"] = eps;
    return *out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list g) {
    variable_list res(6);
    if (!g[0].defined()) return res;
    const auto saved = ctx->get_saved_variables();
    const Tensor &p = saved[0], &query = saved[1], &inter = saved[2], &lse = saved[3];
    const double eps = ctx->saved_data["eps"].toDouble();
    const int64_t d = p.size(-1), n = p.numel() / d;
    Tensor gp, gq, gi, gl, go = g[0];
    bool done = false;
    if (!at::GradMode::is_enabled() && unwatched() && n >= 1 && plain(p) && plain(query) && plain(inter) &&
        plain(lse) && dense(go) && go.get_device() == p.get_device() && go.sizes() == inter.sizes()) {
      ATTNRES_RECORD("attnres_hip::merge_bwd");
      const c10::Device dev = p.device();
      go = go.to(inter.scalar_type()).contiguous();
      gp = empty(p.sizes(), p.scalar_type(), dev);
      gi = empty(inter.sizes(), inter.scalar_type(), dev);
      gl = empty(lse.sizes(), at::kFloat, dev);
      gq = empty(query.sizes(), query.scalar_type(), dev);
      const OnDevice on(p);
      int64_t bytes = 0;
      if (attnres_route_bwd_workspace_size(n, (int)d, &bytes) == ATTNRES_OK) {
        const Tensor ws = workspace(bytes, dev);
        done = attnres_merge_bwd(ptr(p), n, (int)d, code(p.scalar_type()), ptr(query), code(query.scalar_type()),
                                 ptr(inter), code(inter.scalar_type()), static_cast<const float*>(ptr(lse)), (float)eps,
                                 ptr(go), out_ptr<void>(gp), out_ptr<void>(gi), out_ptr<float>(gl), out_ptr<void>(ws),
                                 ws.numel() * 4, out_ptr<void>(gq), on.stream) == ATTNRES_OK;
      }
    }
    if (!done) {
      const auto st = call_op("attnres_hip::merge_bwd", p, query, inter, lse, eps, g[0]);
      gp = st[0].toTensor(), gq = st[1].toTensor(), gi = st[2].toTensor(), gl = st[3].toTensor();
    }
    if (ctx->needs_input_grad(0)) res[0] = gp;
    if (ctx->needs_input_grad(1)) res[1] = gq;
    if (ctx->needs_input_grad(2)) res[2] = gi;
    if (ctx->needs_input_grad(3)) res[3] = gl;
    return res;
  }
};

// ---------------------------------------------------------- Python entries --

// How a routing call's result is handed back.
enum Form : int64_t {
  kRows = 1,          // the routed rows alone, one query's without its dimension
  kTuple = 2,         // (out, weights, lse, inv_rms, logits), None where not requested
  kPlaceholders = 3,  // the same with empty fp32 tensors there (what the op returns)
};

// The tensor behind an argument of exactly type Tensor or Parameter; undefined
// for None; false for anything else.
bool take(PyObject* o, bool none_ok, Tensor* t) {
  if (o == Py_None) {
    *t = Tensor();
    return none_ok;
  }
  if (!THPVariable_CheckExact(o)) return false;
  *t = THPVariable_Unpack(o);
  return true;
}
bool take(PyObject* o, double* v) {
  *v = PyFloat_AsDouble(o);
  if (*v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}
bool take(PyObject* o, int64_t* v) {
  if (!PyLong_Check(o)) return false;
  *v = PyLong_AsLongLong(o);
  if (*v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}
// exactly True or False (another truthy value is left to Python)
bool take(PyObject* o, bool* v) {
  *v = o == Py_True;
  return PyBool_Check(o);
}
// out_dtype: a torch.dtype; with the rows form and a gain None too, for the promotion of the sources' and
// the parameters' dtypes (the other forms stand for the op, which takes no None, and the drop-ins need a gain)
bool take_dtype(PyObject* o, int64_t form, const Tensor& src, const Tensor& query, const Tensor& gain,
                at::ScalarType* t) {
  if (THPDtype_Check(o)) {
    *t = reinterpret_cast<THPDtype*>(o)->scalar_type;
    return true;
  }
  if (o != Py_None || form != kRows || !gain.defined()) return false;
  *t = at::promote_types(src.scalar_type(), at::promote_types(query.scalar_type(), gain.scalar_type()));
  return true;
}
bool take_list(PyObject* o, std::vector<Tensor>* v) {
  if (!PyList_CheckExact(o) && !PyTuple_CheckExact(o)) return false;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
  PyObject** items = PySequence_Fast_ITEMS(o);
  v->reserve((size_t)n);
  for (Py_ssize_t i = 0; i < n; ++i) {
    Tensor t;
    if (!take(items[i], false, &t)) return false;
    v->push_back(std::move(t));
  }
  return true;
}

// Whether autograd would record a call on these tensors.
bool recorded(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->defined() && t->requires_grad()) return true;
  return false;
}
bool recorded(const std::vector<Tensor>& ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor& t : ts)
    if (t.requires_grad()) return true;
  return false;
}
// No tensor carries a forward-mode tangent (the autograd functions here have no forward-mode rule: the op reports it).
bool no_tangent(const Tensor& t) { return !t.defined() || !t._fw_grad(0).defined(); }

PyObject* none() { Py_RETURN_NONE; }
PyObject* wrap(const Tensor& t) {
  if (!t.defined()) return none();
  return THPVariable_Wrap(t);
}
PyObject* pack(const Routed& r, int64_t form) {
  if (form == kRows) return wrap(r.out);
  PyObject* tup = PyTuple_New(5);
  if (tup == nullptr) return nullptr;
  const Tensor* ts[] = {&r.out, &r.weights, &r.lse, &r.inv_rms, &r.logits};
  for (int i = 0; i < 5; ++i)
    PyTuple_SET_ITEM(tup, i,
                     !ts[i]->defined() && form == kPlaceholders ? wrap(empty({0}, at::kFloat, r.out.device()))
                                                                : wrap(*ts[i]));
  return tup;
}

// route(buf, num_sources, query, gain, eps, out_dtype, want_weights, want_lse, want_aux, form, zero_inactive)
//   zero_inactive: None (a call that autograd records is left alone) or whether
//   the gradient's inactive slots are cleared.
PyObject* py_route(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor buf, query, gain;
  bool ww, wl, wa;
  int64_t num = 0, form = 0;
  double eps = 0;
  at::ScalarType dt;
  if (n != 11 || !take(a[0], false, &buf) || !take(a[1], &num) || !take(a[2], false, &query) ||
      !take(a[3], true, &gain) || !take(a[4], &eps) || !take(a[9], &form) ||
      !take_dtype(a[5], form, buf, query, gain, &dt) || !take(a[6], &ww) || !take(a[7], &wl) || !take(a[8], &wa) ||
      !unwatched())
    return none();
  const bool rec = recorded({&buf, &query, &gain});
  if (rec && (a[10] == Py_None || num < 1 || !no_tangent(buf) || !no_tangent(query) || !no_tangent(gain)))
    return none();
  Routed r;
  {
    pybind11::gil_scoped_release nogil;
    if (!route_rows("attnres_hip::route", Sources::stacked(buf, num), query, gain, eps, dt, ww, wl, wa, form == kRows,
                    &r))
      r.out = Tensor();
  }
  if (!r.out.defined()) return none();
  if (rec) {
    const variable_list o = RouteStacked::apply(buf, query, opt(gain), &r, num, eps, a[10] == Py_True);
    r.out = o[0];
    if (r.lse.defined()) r.lse = o[1];
  }
  return pack(r, form);
  END_HANDLE_TH_ERRORS
}

// route_list(sources, query, gain, eps, out_dtype, want_weights, want_lse, want_aux, form, grad)
//   grad: whether a call that autograd records is taken (without weights and aux outputs)
PyObject* py_route_list(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  std::vector<Tensor> srcs;
  Tensor query, gain;
  bool ww, wl, wa;
  double eps = 0;
  int64_t form = 0;
  at::ScalarType dt;
  if (n != 10 || !take_list(a[0], &srcs) || srcs.empty() || !take(a[1], false, &query) || !take(a[2], true, &gain) ||
      !take(a[3], &eps) || !take(a[8], &form) || !take_dtype(a[4], form, srcs[0], query, gain, &dt) ||
      !take(a[5], &ww) || !take(a[6], &wl) || !take(a[7], &wa) || !unwatched())
    return none();
  const bool rec = recorded(srcs) || recorded({&query, &gain});
  if (rec) {
    if (a[9] != Py_True || ww || wa || !no_tangent(query) || !no_tangent(gain)) return none();
    for (const Tensor& t : srcs)
      if (!no_tangent(t)) return none();
  }
  Routed r;
  {
    pybind11::gil_scoped_release nogil;
    if (!route_rows("attnres_hip::route_list", Sources::list(srcs), query, gain, eps, dt, ww, wl, wa, form == kRows,
                    &r))
      r.out = Tensor();
  }
  if (!r.out.defined()) return none();
  if (rec) {
    const variable_list o = RouteList::apply(at::TensorList(srcs), query, opt(gain), &r, eps);
    r.out = o[0];
    if (r.lse.defined()) r.lse = o[1];
  }
  return pack(r, form);
  END_HANDLE_TH_ERRORS
}

// merge(partial, query, inter, lse, eps) -> merged rows
PyObject* py_merge(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor p, q, inter, lse, out;
  double eps = 0;
  if (n != 5 || !take(a[0], false, &p) || !take(a[1], false, &q) || !take(a[2], false, &inter) ||
      !take(a[3], false, &lse) || !take(a[4], &eps) || !unwatched())
    return none();
  const bool rec = recorded({&p, &q, &inter, &lse});
  if (rec && !(no_tangent(p) && no_tangent(q) && no_tangent(inter) && no_tangent(lse))) return none();
  bool ok = false;
  {
    pybind11::gil_scoped_release nogil;
    ok = merge_rows(p, q, inter, lse, eps, &out);
  }
  if (!ok) return none();
  if (rec) out = Merge::apply(p, q, inter, lse, &out, eps);
  return wrap(out);
  END_HANDLE_TH_ERRORS
}

// block_step(arena, n_committed, commit, delta, query, gain, eps, want_weights) -> (out, weights, lse); no autograd
PyObject* py_block_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor arena, delta, query, gain;
  int64_t nc = 0;
  double eps = 0;
  bool commit, ww;
  if (n != 8 || !take(a[0], false, &arena) || !take(a[1], &nc) || !take(a[2], &commit) || !take(a[3], true, &delta) ||
      !take(a[4], false, &query) || !take(a[5], true, &gain) || !take(a[6], &eps) || !take(a[7], &ww) || !unwatched() ||
      recorded({&arena, &delta, &query, &gain}))
    return none();
  const int64_t s = nc + (commit ? 1 : 0) + 1;
  const Sources src = Sources::stacked(arena, std::min<int64_t>(s, arena.dim() > 0 ? arena.size(0) : 0));
  if (!src.ok || s < 1 || s > arena.size(0) || query.dim() != 1) return none();
  if (delta.defined() && (!plain(delta) || delta.scalar_type() != src.dtype ||
                          delta.get_device() != arena.get_device() || delta.sizes() != arena.sizes().slice(1)))
    return none();
  const Fold fold(query, gain, src.d, arena);
  if (!fold.ok) return none();
  Tensor out, weights, lse;
  bool ok = false;
  {
    pybind11::gil_scoped_release nogil;
    out = empty(arena.sizes().slice(1), src.dtype, arena.device());
    if (ww) {
      Dims w{s};
      w.append(src.batch.begin(), src.batch.end());
      weights = empty(w, at::kFloat, arena.device());
      lse = empty(src.batch, at::kFloat, arena.device());
    }
    const OnDevice on(arena);
    ok = attnres_block_step(arena.mutable_data_ptr(), (int)arena.size(0), src.n * src.d, (int)nc, commit ? 1 : 0,
                            ptr(delta), src.n, (int)src.d, code(src.dtype), ptr(query), ptr(gain),
                            code(query.scalar_type()), (float)eps, out_ptr<void>(out), out_ptr<float>(weights),
                            out_ptr<float>(lse), on.stream) == ATTNRES_OK;
  }
  if (!ok) return none();
  PyObject* tup = PyTuple_New(3);
  if (tup == nullptr) return nullptr;
  PyTuple_SET_ITEM(tup, 0, wrap(out));
  PyTuple_SET_ITEM(tup, 1, wrap(weights));
  PyTuple_SET_ITEM(tup, 2, wrap(lse));
  return tup;
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------- training points --
//
// The launches of ops.py's _RoutePoint and GradSegments (run inside a Python
// autograd function: nothing is recorded here).

// step(committed, partial, delta, query, gain, eps, out_dtype) -> (routed rows, partial + delta)
PyObject* py_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  std::vector<Tensor> srcs;
  Tensor partial, delta, query, gain, out, next;
  double eps = 0;
  at::ScalarType dt;
  if (n != 7 || !take_list(a[0], &srcs) || !take(a[1], false, &partial) || !take(a[2], false, &delta) ||
      !take(a[3], false, &query) || !take(a[4], true, &gain) || !take(a[5], &eps) ||
      !take_dtype(a[6], kTuple, partial, query, gain, &dt) || !unwatched())
    return none();
  const int k = (int)srcs.size();
  srcs.push_back(partial);
  const Sources src = Sources::list(srcs);
  if (!src.ok || dt != src.dtype || !plain(delta) || delta.scalar_type() != src.dtype ||
      delta.sizes() != partial.sizes() || delta.get_device() != partial.get_device())
    return none();
  const Fold fold(query, gain, src.d, partial);
  if (!fold.ok || fold.nq != 1) return none();
  bool ok = false;
  {
    pybind11::gil_scoped_release nogil;
    next = empty(partial.sizes(), src.dtype, partial.device());
    out = empty(partial.sizes(), dt, partial.device());
    const OnDevice on(partial);
    ok = attnres_route_step(src.ptrs, k, ptr(partial), ptr(delta), out_ptr<void>(next), src.n, (int)src.d,
                            code(src.dtype), ptr(query), ptr(gain), code(query.scalar_type()), (float)eps,
                            out_ptr<void>(out), nullptr, nullptr, on.stream) == ATTNRES_OK;
  }
  if (!ok) return none();
  PyObject* o = wrap(out);
  PyObject* p = wrap(next);
  return o != nullptr && p != nullptr ? Py_BuildValue("(NN)", o, p) : nullptr;
  END_HANDLE_TH_ERRORS
}

// bwd_rows(sources, grads, adds, query, gain, eps, grad_out) -> (dquery, dgain): attnres_route_bwd_add into
// `grads`, adds[s] None or the rows added to source s's gradient
PyObject* py_bwd_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  std::vector<Tensor> srcs, grads;
  Tensor query, gain, go, dq, dg;
  double eps = 0;
  if (n != 7 || !take_list(a[0], &srcs) || !take_list(a[1], &grads) || !PyList_CheckExact(a[2]) ||
      !take(a[3], false, &query) || !take(a[4], true, &gain) || !take(a[5], &eps) || !take(a[6], false, &go) ||
      grads.size() != srcs.size() || PyList_GET_SIZE(a[2]) != (Py_ssize_t)srcs.size() || !unwatched())
    return none();
  const Sources src = Sources::list(srcs);
  if (!src.ok || query.numel() != src.d) return none();
  void* gp[ATTNRES_MAX_SOURCES];
  const void* ap[ATTNRES_MAX_SOURCES];
  bool any = false;
  for (size_t i = 0; i < srcs.size(); ++i) {
    Tensor add;
    if (!take(PyList_GET_ITEM(a[2], (Py_ssize_t)i), true, &add)) return none();
    for (const Tensor* t : {&grads[i], &add}) {
      if (t->defined() && (!plain(*t) || t->scalar_type() != src.dtype || t->numel() != srcs[i].numel() ||
                           t->get_device() != srcs[i].get_device()))
        return none();
    }
    gp[i] = grads[i].mutable_data_ptr();
    ap[i] = ptr(add);
    any = any || add.defined();
  }
  bool ok = false;
  {
    pybind11::gil_scoped_release nogil;
    ok = route_rows_bwd(src, gp, query, gain, eps, go, Tensor(), any ? ap : nullptr, &dq, &dg);
  }
  return ok ? Py_BuildValue("(NN)", wrap(dq), wrap(dg)) : none();
  END_HANDLE_TH_ERRORS
}

// bwd_defer(sources, query, gain, eps, grad_out, grad_add)
//   -> (partial's gradient, records, folded query, grad_out rows, dquery, dgain)
PyObject* py_bwd_defer(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  std::vector<Tensor> srcs;
  Tensor query, gain, go, add, gp, coef, qfold, dq, dg;
  double eps = 0;
  if (n != 6 || !take_list(a[0], &srcs) || !take(a[1], false, &query) || !take(a[2], true, &gain) ||
      !take(a[3], &eps) || !take(a[4], false, &go) || !take(a[5], true, &add) || !unwatched())
    return none();
  const Sources src = Sources::list(srcs);
  if (!src.ok || src.s < 2 || src.n < 1 || src.dtype != at::kBFloat16) return none();
  const Tensor& p = srcs.back();
  const Fold fold(query, gain, src.d, p);
  if (!fold.ok || fold.nq != 1 || query.scalar_type() != at::kBFloat16 || !dense(go) ||
      go.scalar_type() != at::kBFloat16 || go.get_device() != p.get_device() || go.numel() != src.n * src.d)
    return none();
  if (add.defined() && (!plain(add) || add.scalar_type() != src.dtype || add.numel() != p.numel() ||
                        add.get_device() != p.get_device()))
    return none();
  bool ok = false;
  {
    pybind11::gil_scoped_release nogil;
    go = go.reshape({src.n, src.d}).contiguous();
    const c10::Device dev = p.device();
    gp = empty(p.sizes(), src.dtype, dev);
    coef = empty({src.n, src.s - 1, 4}, at::kFloat, dev);
    qfold = empty({src.d}, query.scalar_type(), dev);
    dq = empty(query.sizes(), query.scalar_type(), dev);
    if (gain.defined()) dg = empty(gain.sizes(), gain.scalar_type(), dev);
    const OnDevice on(p);
    int64_t bytes = 0;
    if (attnres_route_bwd_workspace_size(src.n, (int)src.d, &bytes) == ATTNRES_OK) {
      const Tensor ws = workspace(bytes, dev);
      ok = attnres_route_bwd_defer(src.ptrs, src.s, src.n, (int)src.d, src.d, code(src.dtype), ptr(query), ptr(gain),
                                   code(query.scalar_type()), (float)eps, ptr(go), code(go.scalar_type()), src.d,
                                   nullptr, out_ptr<void>(gp), ptr(add), src.d, out_ptr<float>(coef),
                                   out_ptr<void>(qfold), out_ptr<void>(ws), ws.numel() * 4, out_ptr<void>(dq),
                                   out_ptr<void>(dg), on.stream) == ATTNRES_OK;
    }
  }
  return ok ? Py_BuildValue("(NNNNNN)", wrap(gp), wrap(coef), wrap(qfold), wrap(go), wrap(dq), wrap(dg)) : none();
  END_HANDLE_TH_ERRORS
}

// gather_seg(terms, part_in, csum_in, x, addend) -> (gradient, running sums, x-coefficient sums): one
// attnres_route_bwd_gather_seg over the blocks of part_in / csum_in (Tensor or None each, the last block's too);
// terms: (grad_out, records, folded query, blocks) per point.  Running sums are updated in place or, where None,
// new; the gradient goes to `addend` or a new tensor.
PyObject* py_gather_seg(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor x, addend;
  if (n != 5 || !PyList_CheckExact(a[0]) || !PyList_CheckExact(a[1]) || !PyList_CheckExact(a[2]) ||
      !take(a[3], false, &x) || !take(a[4], true, &addend) || !unwatched())
    return none();
  const Py_ssize_t nt = PyList_GET_SIZE(a[0]), nb = PyList_GET_SIZE(a[1]);
  constexpr Py_ssize_t kMaxBlocks = ATTNRES_SEG_MAX_BLOCKS, kMaxTerms = ATTNRES_SEG_MAX_TERMS;  // one launch
  if (nb < 1 || nb > kMaxBlocks || PyList_GET_SIZE(a[2]) != nb || nt < 1 || nt > kMaxTerms || !plain(x) || x.dim() < 1)
    return none();
  const int64_t d = x.size(-1), rows = d > 0 ? x.numel() / d : 0;
  if (rows < 1 || (addend.defined() && (!plain(addend) || addend.scalar_type() != x.scalar_type() ||
                                        addend.numel() != x.numel() || addend.get_device() != x.get_device())))
    return none();
  auto same = [&](const Tensor& t, at::ScalarType dt, int64_t numel) {
    return plain(t) && t.scalar_type() == dt && t.numel() == numel && t.get_device() == x.get_device();
  };
  Tensor keep[kMaxTerms][3], part[kMaxBlocks], csum[kMaxBlocks];
  const void *go[kMaxTerms], *qf[kMaxTerms];
  const float* coef[kMaxTerms];
  int64_t coef_ld[kMaxTerms];
  for (Py_ssize_t j = 0; j < nt; ++j) {
    PyObject* t = PyList_GET_ITEM(a[0], j);
    if (!PyTuple_CheckExact(t) || PyTuple_GET_SIZE(t) != 4) return none();
    for (int i = 0; i < 3; ++i)
      if (!take(PyTuple_GET_ITEM(t, i), false, &keep[j][i])) return none();
    const Tensor &g = keep[j][0], &c = keep[j][1], &q = keep[j][2];
    if (!same(g, x.scalar_type(), x.numel()) || !same(q, x.scalar_type(), d) || c.dim() != 3 || c.size(1) < nb ||
        c.size(2) != 4 || !same(c, at::kFloat, rows * c.size(1) * 4))
      return none();
    go[j] = ptr(g), qf[j] = ptr(q), coef[j] = static_cast<const float*>(ptr(c)), coef_ld[j] = 4 * c.size(1);
  }
  const void *pin[kMaxBlocks];
  const float* cin[kMaxBlocks];
  for (Py_ssize_t j = 0; j < nb; ++j) {
    if (!take(PyList_GET_ITEM(a[1], j), true, &part[j]) || !take(PyList_GET_ITEM(a[2], j), true, &csum[j]))
      return none();
    if ((part[j].defined() && !same(part[j], x.scalar_type(), x.numel())) ||
        (csum[j].defined() && !same(csum[j], at::kFloat, rows)))
      return none();
    pin[j] = ptr(part[j]), cin[j] = static_cast<const float*>(ptr(csum[j]));
  }
  Tensor out = addend;
  bool ok = false;
  {
    pybind11::gil_scoped_release nogil;
    const c10::Device dev = x.device();
    void* pout[kMaxBlocks];
    float* cout[kMaxBlocks];
    for (Py_ssize_t j = 0; j < nb - 1; ++j) {
      if (!part[j].defined()) part[j] = empty({rows, d}, x.scalar_type(), dev);
      if (!csum[j].defined()) csum[j] = empty({rows}, at::kFloat, dev);
      pout[j] = out_ptr<void>(part[j]), cout[j] = out_ptr<float>(csum[j]);
    }
    if (!out.defined()) out = empty(x.sizes(), x.scalar_type(), dev);
    pout[nb - 1] = out_ptr<void>(out), cout[nb - 1] = nullptr;
    const OnDevice on(x);
    ok = attnres_route_bwd_gather_seg((int)nb, rows, (int)d, code(x.scalar_type()), (int)nt, go, d, coef, coef_ld, qf,
                                      pin, cin, pout, cout, ptr(x), d, ptr(addend), d, on.stream) == ATTNRES_OK;
  }
  if (!ok) return none();
  PyObject* parts = PyList_New(nb - 1);
  PyObject* csums = PyList_New(nb - 1);
  if (parts == nullptr || csums == nullptr) return nullptr;
  for (Py_ssize_t j = 0; j < nb - 1; ++j) {
    PyList_SET_ITEM(parts, j, wrap(part[j]));
    PyList_SET_ITEM(csums, j, wrap(csum[j]));
  }
  return Py_BuildValue("(NNN)", wrap(out), parts, csums);
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"gather_seg", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_gather_seg)), METH_FASTCALL, nullptr},
    {"step", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_step)), METH_FASTCALL, nullptr},
    {"bwd_rows", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_bwd_rows)), METH_FASTCALL, nullptr},
    {"bwd_defer", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_bwd_defer)), METH_FASTCALL, nullptr},
    {"route", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_route)), METH_FASTCALL, nullptr},
    {"route_list", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_route_list)), METH_FASTCALL, nullptr},
    {"merge", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_merge)), METH_FASTCALL, nullptr},
    {"block_step", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_block_step)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_attnres_torch", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__attnres_torch() {
  PyObject* mod = PyModule_Create(&kModule);
  // the torch this was compiled for: the loader takes no other (_native.py)
  if (mod != nullptr && PyModule_AddStringConstant(mod, "torch_version", ATTNRES_TORCH_VERSION) != 0) Py_CLEAR(mod);
  return mod;
}
