// Eager calls of the normalisation without Python on the way: checks, allocations, the C ABI call and the autograd node
// of GN_NHWC.forward and group_norm_nhwc.  What bounds the small and middle sizes is host time, not kernels: a forward +
// backward through a Python autograd.Function costs about 130 us of interpreter, engine hand-over and ctypes around two
// kernels of 8 us each.
//
// group_norm() takes ordinary eager calls only -- plain device tensors in one of the two dense layouts, no mode, transform,
// tracer or tangent that would want to see the individual torch operations -- and answers NotImplemented to everything
// else, errors included; the caller then runs the Python implementation, which remains the general one.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/gnnhwc.h"

namespace {

using at::Tensor;
using std::optional;

// The C ABI's entry points, handed over by address: the Python binding decides which library is loaded.
struct Entry {
  decltype(&gnnhwc_last_error) last_error;
  decltype(&gnnhwc_fwd_workspace_bytes) fwd_workspace_bytes;
  decltype(&gnnhwc_bwd_workspace_bytes) bwd_workspace_bytes;
  decltype(&gnnhwc_nchw_workspace_bytes) nchw_workspace_bytes;
  decltype(&gnnhwc_fwd_cast) fwd_cast;
  decltype(&gnnhwc_bwd_cast) bwd_cast;
  decltype(&gnnhwc_fwd_add) fwd_add;
  decltype(&gnnhwc_fwd_nchw) fwd_nchw;
  decltype(&gnnhwc_bwd_nchw) bwd_nchw;
} abi = {};

int code_of(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return GNNHWC_F32;
    case at::kDouble: return GNNHWC_F64;
    case at::kHalf: return GNNHWC_F16;
    case at::kBFloat16: return GNNHWC_BF16;
    default: return -1;
  }
}
bool is_half(at::ScalarType t) { return t == at::kHalf || t == at::kBFloat16; }
// 16-bit data keep their statistics in float32
at::ScalarType stats_type(at::ScalarType t) { return is_half(t) ? at::kFloat : t; }

// Channels fastest, the other dimensions contiguous in their logical order (strides of dimensions of size 1 are free).
bool channels_last(const Tensor &t) {
  const auto sizes = t.sizes(), strides = t.strides();
  const int64_t nd = t.dim();
  int64_t expect = 1;
  if (sizes[1] != 1 && strides[1] != 1) return false;
  expect = sizes[1];
  for (int64_t d = nd - 1; d >= 2; --d) {
    if (sizes[d] != 1 && strides[d] != expect) return false;
    expect *= sizes[d];
  }
  return sizes[0] == 1 || strides[0] == expect;
}
Tensor empty_channels_last(const Tensor &like, at::ScalarType type) {
  const auto sizes = like.sizes();
  c10::SmallVector<int64_t, 6> strides(sizes.size());
  strides[1] = 1;
  int64_t s = sizes[1];
  for (int64_t d = (int64_t)sizes.size() - 1; d >= 2; --d) {
    strides[d] = s;
    s *= sizes[d];
  }
  strides[0] = s;
  return at::empty_strided(sizes, strides, like.options().dtype(type));
}

struct Shape {
  int64_t N, C, R;
};
Shape shape_of(const Tensor &x) {
  Shape s = {x.size(0), x.size(1), 1};
  for (int64_t d = 2; d < x.dim(); ++d) s.R *= x.size(d);
  return s;
}
void *stream_of(const Tensor &x) { return (void *)c10::hip::getCurrentHIPStream(x.device().index()).stream(); }
// Scratch memory of one call, from the caching allocator: in stream order, and part of a graph's own pool under capture.
Tensor workspace(size_t bytes, const Tensor &x, const char *what) {
  TORCH_CHECK(bytes != 0, what, ": ", abi.last_error());
  return at::empty({(int64_t)bytes}, x.options().dtype(at::kByte));
}
void *ptr(const optional<Tensor> &t) { return t.has_value() && t->defined() ? t->data_ptr() : nullptr; }
void check(int rc, const char *what) { TORCH_CHECK(rc == 0, what, " failed (code ", rc, "): ", abi.last_error()); }

// A tensor the kernels may read: memory of x's device.
void require_device(const Tensor &t, const Tensor &x, const char *name) {
  TORCH_CHECK(t.defined() && t.is_cuda() && t.layout() == at::kStrided, name, " must be a CUDA tensor");
  TORCH_CHECK(t.device() == x.device(), name, " is on ", t.device(), ", the other tensors on ", x.device());
}
// Dimension orders that take the channels of an nd-dimensional tensor behind the spatial dimensions, and back.
struct Orders {
  c10::SmallVector<int64_t, 6> last, back;
};
Orders orders_of(int64_t nd) {
  Orders o = {c10::SmallVector<int64_t, 6>(nd), c10::SmallVector<int64_t, 6>(nd)};
  o.last[0] = o.back[0] = 0;
  for (int64_t d = 2; d < nd; ++d) o.last[d - 1] = d;
  o.last[nd - 1] = 1;
  o.back[1] = nd - 1;
  for (int64_t d = 2; d < nd; ++d) o.back[d] = d - 1;
  return o;
}
Tensor resolved(const Tensor &t) { return t.is_neg() ? t.resolve_neg() : t; }
// t in the layout of the kernels -- `first`: contiguous, else channels-last --; t itself where it already is.
Tensor in_layout(const Tensor &t, bool first) {
  if (first) return t.contiguous();
  if (t.dim() < 3 || channels_last(t)) return t;
  const Orders o = orders_of(t.dim());
  return t.permute(o.last).contiguous().permute(o.back);
}

// The operator's name in torch's profiler, around one call.
class OperatorRange {
 public:
  explicit OperatorRange(const char *what) : range_(at::RecordScope::FUNCTION) {
    if (range_.isActive()) range_.before(what);
  }

 private:
  at::RecordFunction range_;
};

struct Added {  // pre-additions of the forward (group_norm_nhwc)
  optional<Tensor> residual, channel_bias;
  Tensor sum;  // where x + residual + channel_bias goes (undefined: nowhere)
  bool any = false;
};
// One forward call on checked arguments; stats (null: nobody will ask for them) comes back as (2, N, G): mean, 1 / sqrt(var + eps).
Tensor run_forward(const Tensor &x, const optional<Tensor> &weight, const optional<Tensor> &bias, int64_t G, double eps, int act,
                   bool first, at::ScalarType out, const Added &add, Tensor *stats) {
  const c10::DeviceGuard guard(x.device());
  const at::AutoDispatchBelowADInplaceOrView below;
  const Shape s = shape_of(x);
  const int dt = code_of(x.scalar_type()), pdt = ptr(weight) ? code_of(weight->scalar_type()) : dt;
  const at::ScalarType st = stats_type(x.scalar_type());
  Tensor y = first ? at::empty(x.sizes(), x.options()) : empty_channels_last(x, out);
  char *mean = nullptr, *rstd = nullptr;
  if (stats) {
    *stats = at::empty({2, s.N, G}, x.options().dtype(st));
    mean = (char *)stats->data_ptr();
    rstd = mean + s.N * G * stats->element_size();
  }
  const size_t bytes = first ? abi.nchw_workspace_bytes(s.N, s.C, s.R, G, dt, 0) : abi.fwd_workspace_bytes(s.N, s.R, s.C, G, dt);
  const char *what = first ? "gnop::fwd_nchw" : add.any ? "gnop::fwd_add" : out != x.scalar_type() ? "gnop::fwd_cast" : "gnop::fwd";
  const OperatorRange range(what);
  const Tensor ws = workspace(bytes, x, what);
  int rc;
  if (first)
    rc = abi.fwd_nchw(x.data_ptr(), ptr(weight), ptr(bias), y.data_ptr(), mean, rstd, s.N, s.C, s.R, G, eps, act, dt, pdt,
                      code_of(st), ws.data_ptr(), bytes, stream_of(x));
  else if (add.any)
    rc = abi.fwd_add(x.data_ptr(), ptr(add.residual), ptr(add.channel_bias), add.sum.defined() ? add.sum.data_ptr() : nullptr,
                     ptr(weight), ptr(bias), y.data_ptr(), mean, rstd, s.N, s.R, s.C, G, eps, act, dt, pdt, code_of(st),
                     ptr(add.channel_bias) ? code_of(add.channel_bias->scalar_type()) : dt, ws.data_ptr(), bytes, stream_of(x));
  else
    rc = abi.fwd_cast(x.data_ptr(), ptr(weight), ptr(bias), y.data_ptr(), mean, rstd, s.N, s.R, s.C, G, eps, act, dt, pdt,
                      code_of(st), code_of(out), ws.data_ptr(), bytes, stream_of(x));
  check(rc, what);
  return y;
}

// Dispatch keys of a plain device tensor; any other key (a subclass, a transform's wrapper, a lazy conjugate ...) declines.
const c10::DispatchKeySet &plain_keys() {
  static const c10::DispatchKeySet keys = c10::DispatchKeySet(c10::DispatchKey::CUDA) |
                                          c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA) |
                                          c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) |
                                          c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA);
  return keys;
}
// Keys that are switched on for every thread, or by autocast (which has no rule for this operation).
const c10::DispatchKeySet &plain_tls() {
  static const c10::DispatchKeySet keys =
      c10::default_included_set | c10::autocast_dispatch_keyset | c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView);
  return keys;
}
// (by the bits: the sets' difference keeps the bits of the backends)
bool only(c10::DispatchKeySet keys, c10::DispatchKeySet allowed) { return (keys.raw_repr() & ~allowed.raw_repr()) == 0; }
bool ordinary_dispatch() {
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() && only(c10::impl::tls_local_dispatch_key_set().included_, plain_tls());
}
bool ordinary_thread() { return at::impl::PythonTorchFunctionTLS::stack_len() == 0 && ordinary_dispatch(); }
bool plain(const Tensor &t, const c10::Device &device) {
  return t.defined() && t.is_cuda() && t.device() == device && t.layout() == at::kStrided && only(t.key_set(), plain_keys()) &&
         !t._fw_grad(0).defined();
}

// Memory the kernels can be given, whatever else the tensor carries.
bool readable(const Tensor &t) { return t.has_storage() && !t.key_set().has(c10::DispatchKey::Python); }

// The backward through the dispatcher, as the operators' registered formula calls it: for gradients and saved tensors that are
// no plain device tensors (batched gradients, subclasses), and where something on this thread is to see the operator.
torch::autograd::variable_list backward_operator(const Tensor &dy, const Tensor &x, const Tensor &weight, const Tensor &bias,
                                                 const Tensor &stats, int64_t G, int64_t act, bool first) {
  const char *what = first ? "gnop::bwd_nchw" : "gnop::bwd";
  TORCH_CHECK(weight.defined(), what, " of a normalisation without parameters takes plain device tensors only");
  TORCH_CHECK(x.dim() >= 3 && dy.sizes() == x.sizes(), what, " expects dy and X of the same shape, got ", dy.sizes(), " and ", x.sizes());
  using Signature = std::tuple<Tensor, Tensor, Tensor>(const Tensor &, const Tensor &, const Tensor &, const Tensor &,
                                                       const Tensor &, const Tensor &, int64_t, int64_t);
  const auto op = c10::Dispatcher::singleton().findSchemaOrThrow(what, "").typed<Signature>();
  const Orders o = orders_of(x.dim());
  const Shape s = shape_of(x);
  const auto flat = [&](const Tensor &t) {  // (N, C, R), channels-last unless `first`
    if (first) return t.contiguous().view({s.N, s.C, s.R});
    return t.permute(o.last).contiguous().view({s.N, s.R, s.C}).permute({0, 2, 1});
  };
  const Tensor mean = stats.select(0, 0), rstd = stats.select(0, 1);
  const auto [dx, dw, db] = op.call(flat(dy), flat(x), weight, bias, mean, rstd, G, act);
  if (first) return {dx.reshape(x.sizes()), dw, db, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  c10::SmallVector<int64_t, 6> sizes(x.dim());
  for (int64_t d = 0; d < x.dim(); ++d) sizes[d] = x.size(o.last[d]);
  return {dx.permute({0, 2, 1}).reshape(sizes).permute(o.back), dw, db, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
}

// The derivative of the normalisation (no pre-additions), either layout.
struct GroupNormNode : public torch::autograd::Function<GroupNormNode> {
  static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &x, const optional<Tensor> &weight,
                        const optional<Tensor> &bias, int64_t G, double eps, int64_t act, bool first, int64_t out,
                        bool functional) {
    Tensor stats;
    Tensor y = run_forward(x, weight, bias, G, eps, (int)act, first, (at::ScalarType)out, Added{}, &stats);
    ctx->save_for_backward({x, weight.value_or(Tensor()), bias.value_or(Tensor()), stats});
    ctx->saved_data["call"] = std::vector<int64_t>{G, act, first ? 1 : 0, functional ? 1 : 0};
    // a view, as the Python function returns: an in-place change of y is refused the same way
    return y.view(y.sizes());
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const auto call = ctx->saved_data["call"].toIntVector();
    const int64_t G = call[0], act = call[1];
    const bool first = call[2] != 0, functional = call[3] != 0;
    const char *what = first ? "gnop::bwd_nchw" : "gnop::bwd";
    // The saved tensors are what the caller's saved-tensor hooks return, which need not be what the forward saved: offloading
    // hooks give back contiguous copies, others may leave a tensor on the host.
    require_device(grads[0], grads[0], "dy");
    require_device(saved[0], grads[0], "X");
    require_device(saved[3], grads[0], "means");
    if (saved[1].defined()) {
      require_device(saved[1], grads[0], "weight");
      require_device(saved[2], grads[0], "bias");
    }
    const c10::Device device = grads[0].device();
    const c10::DeviceGuard guard(device);
    // (the module's own autograd function never recorded a graph of its backward; the functional form went through the operator)
    const at::AutoGradMode graph(functional && at::GradMode::is_enabled());
    Tensor dy = resolved(grads[0]), x = resolved(saved[0]);
    const bool formula = functional && saved[1].defined();  // (without parameters there is no operator to go through)
    const auto kernels_take = [&](const Tensor &t) { return !t.defined() || (formula ? plain(t, device) : readable(t)); };
    if ((formula && (at::GradMode::is_enabled() || !ordinary_dispatch())) || !kernels_take(dy) || !kernels_take(x) ||
        !kernels_take(saved[1]) || !kernels_take(saved[2]) || !kernels_take(saved[3]))
      return backward_operator(dy, x, saved[1], saved[2], saved[3], G, act, first);
    const at::AutoGradMode no_graph(false);
    dy = in_layout(dy, first);
    x = in_layout(x, first);
    const Tensor stats = saved[3].contiguous();
    TORCH_CHECK(x.dim() >= 3 && dy.sizes() == x.sizes(), what, " expects dy and X of the same shape, got ", dy.sizes(), " and ",
                x.sizes());
    const bool dy16 = !first && x.scalar_type() == at::kFloat && is_half(dy.scalar_type());
    TORCH_CHECK(dy.scalar_type() == x.scalar_type() || dy16,
                "dy and X must have the same dtype, or dy float16 / bfloat16 with float32 X (", dy.scalar_type(), " vs ",
                x.scalar_type(), ")");
    TORCH_CHECK(stats.numel() == 2 * x.size(0) * G, "means and rstds must have N*G = ", x.size(0) * G, " elements");
    Tensor weight, bias;
    if (saved[1].defined()) {
      weight = saved[1].contiguous();
      bias = saved[2].contiguous();
      TORCH_CHECK(bias.scalar_type() == weight.scalar_type(), "weight and bias must have the same dtype (", weight.scalar_type(),
                  " vs ", bias.scalar_type(), ")");
      TORCH_CHECK(weight.numel() == x.size(1) && bias.numel() == x.size(1), "weight and bias must have ", x.size(1), " elements");
    }
    const at::AutoDispatchBelowADInplaceOrView below;
    const Shape s = shape_of(x);
    const int dt = code_of(x.scalar_type()), pdt = weight.defined() ? code_of(weight.scalar_type()) : dt;
    const int sdt = code_of(stats.scalar_type());
    Tensor dx = first ? at::empty(x.sizes(), x.options()) : empty_channels_last(x, x.scalar_type());
    // a normalisation without parameters has no parameter gradients: nothing is allocated or computed for them
    Tensor dw, db;
    if (weight.defined()) {
      dw = at::empty({s.C}, weight.options());
      db = at::empty({s.C}, bias.options());
    }
    const char *mean = (const char *)stats.data_ptr(), *rstd = mean + s.N * G * stats.element_size();
    const size_t bytes = first ? abi.nchw_workspace_bytes(s.N, s.C, s.R, G, dt, 1) : abi.bwd_workspace_bytes(s.N, s.R, s.C, G, dt);
    const OperatorRange range(what);
    const Tensor ws = workspace(bytes, x, what);
    void *const wp = weight.defined() ? weight.data_ptr() : nullptr, *const bp = bias.defined() ? bias.data_ptr() : nullptr;
    void *const dwp = dw.defined() ? dw.data_ptr() : nullptr, *const dbp = db.defined() ? db.data_ptr() : nullptr;
    const int rc = first ? abi.bwd_nchw(dy.data_ptr(), x.data_ptr(), wp, bp, mean, rstd, dx.data_ptr(), dwp, dbp, s.N, s.C, s.R, G,
                                        (int)act, dt, pdt, sdt, ws.data_ptr(), bytes, stream_of(x))
                         : abi.bwd_cast(dy.data_ptr(), x.data_ptr(), wp, bp, mean, rstd, dx.data_ptr(), dwp, dbp, s.N, s.R, s.C, G,
                                        (int)act, dt, pdt, sdt, code_of(dy.scalar_type()), ws.data_ptr(), bytes, stream_of(x));
    check(rc, what);
    return {dx, dw, db, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// ---- what group_norm() takes -----------------------------------------------------------------------------------------
// While it lives, other Python threads run: allocations may have to wait for the device, launches for a full queue or for
// another thread's.  (Saved-tensor hooks and operators implemented in Python take the lock again by themselves.)
class WithoutGil {
 public:
  WithoutGil() : state_(PyEval_SaveThread()) {}
  ~WithoutGil() { PyEval_RestoreThread(state_); }
  WithoutGil(const WithoutGil &) = delete;
  WithoutGil &operator=(const WithoutGil &) = delete;

 private:
  PyThreadState *state_;
};
bool needs_grad(const optional<Tensor> &t) { return t.has_value() && t->requires_grad(); }

// None -> no value; an exact torch.Tensor / Parameter -> its tensor; anything else -> false.
bool tensor_or_none(PyObject *o, optional<Tensor> &t) {
  if (o == Py_None) return true;
  if (!THPVariable_CheckExact(o)) return false;
  t = THPVariable_Unpack(o);
  return true;
}

// group_norm(x, weight, bias, num_groups, eps, act_code, out_dtype, residual, channel_bias, return_sum[, functional])
//   -> y, (y, sum), or NotImplemented.  functional: on behalf of group_norm_nhwc, whose derivative is the operators' own.
PyObject *group_norm(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(nargs == 10 || nargs == 11, "group_norm takes 10 or 11 arguments");
  constexpr int kX = 0, kW = 1, kB = 2, kG = 3, kEps = 4, kAct = 5, kOut = 6, kRes = 7, kCb = 8, kSum = 9, kFunctional = 10;
  auto decline = []() { Py_RETURN_NOTIMPLEMENTED; };
  if (!THPVariable_CheckExact(args[kX]) || !ordinary_thread()) return decline();
  const Tensor x = THPVariable_Unpack(args[kX]);
  optional<Tensor> weight, bias;
  Added add;
  if (!tensor_or_none(args[kW], weight) || !tensor_or_none(args[kB], bias) || !tensor_or_none(args[kRes], add.residual) ||
      !tensor_or_none(args[kCb], add.channel_bias))
    return decline();
  if (!PyLong_CheckExact(args[kG]) || !PyFloat_CheckExact(args[kEps]) || !PyLong_CheckExact(args[kAct]) || !PyBool_Check(args[kSum]))
    return decline();
  const int64_t G = PyLong_AsLongLong(args[kG]);
  const int64_t act = PyLong_AsLongLong(args[kAct]);
  const double eps = PyFloat_AS_DOUBLE(args[kEps]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return decline();
  }
  const bool want_sum = args[kSum] == Py_True;
  add.any = add.residual.has_value() || add.channel_bias.has_value() || want_sum;

  const c10::Device device = x.device();
  if (!plain(x, device) || x.dim() < 3 || x.numel() == 0 || code_of(x.scalar_type()) < 0) return decline();
  const int64_t N = x.size(0), C = x.size(1);
  if (G <= 0 || C % G != 0 || act < 0 || act > 4) return decline();
  if (weight.has_value() != bias.has_value()) return decline();
  if (weight.has_value()) {
    const at::ScalarType pt = weight->scalar_type();
    if (!plain(*weight, device) || !plain(*bias, device) || weight->numel() != C || bias->numel() != C || weight->dim() != 1 ||
        bias->dim() != 1 || !weight->is_contiguous() || !bias->is_contiguous() || bias->scalar_type() != pt ||
        !(pt == x.scalar_type() || (is_half(x.scalar_type()) && pt == at::kFloat)))
      return decline();
  }
  const bool first = x.stride(1) != 1;  // contiguous channels-first input has kernels of its own
  if (first ? !x.is_contiguous() : !channels_last(x)) return decline();
  at::ScalarType out = x.scalar_type();
  if (args[kOut] != Py_None) {
    if (!THPDtype_Check(args[kOut])) return decline();
    out = reinterpret_cast<THPDtype *>(args[kOut])->scalar_type;
    if (out != x.scalar_type() && (first || x.scalar_type() != at::kFloat || !is_half(out))) return decline();
  }
  const bool grad = at::GradMode::is_enabled() && (x.requires_grad() || needs_grad(weight) || needs_grad(bias) ||
                                                   needs_grad(add.residual) || needs_grad(add.channel_bias));
  if (add.any) {
    if (grad || first || !weight.has_value() || out != x.scalar_type()) return decline();
    if (add.residual.has_value() && (!plain(*add.residual, device) || add.residual->sizes() != x.sizes() ||
                                     add.residual->scalar_type() != x.scalar_type() || !channels_last(*add.residual)))
      return decline();
    if (add.channel_bias.has_value()) {
      const Tensor &cb = *add.channel_bias;
      if (!plain(cb, device) || cb.dim() != 2 || cb.size(0) != N || cb.size(1) != C || !cb.is_contiguous() ||
          !(cb.scalar_type() == x.scalar_type() || (is_half(x.scalar_type()) && cb.scalar_type() == at::kFloat)))
        return decline();
    }
  }
  Tensor y;
  {
    const WithoutGil released;
    if (grad) {
      // (the module goes through the functional form where the result leaves in another type)
      const bool functional = (nargs == 11 && args[kFunctional] == Py_True) || out != x.scalar_type();
      y = GroupNormNode::apply(x, weight, bias, G, eps, act, first, (int64_t)out, functional);
    } else {
      if (want_sum) {
        const c10::DeviceGuard guard(device);
        const at::AutoDispatchBelowADInplaceOrView below;
        add.sum = empty_channels_last(x, x.scalar_type());
      }
      y = run_forward(x, weight, bias, G, eps, (int)act, first, out, add, nullptr);
    }
  }
  if (!want_sum) return THPVariable_Wrap(y);
  PyObject *yo = THPVariable_Wrap(y);
  PyObject *so = yo ? THPVariable_Wrap(add.sum) : nullptr;
  PyObject *both = so ? PyTuple_Pack(2, yo, so) : nullptr;
  Py_XDECREF(yo);
  Py_XDECREF(so);
  return both;
  END_HANDLE_TH_ERRORS
}

// bind(address, ...): the C ABI's functions in the order of Entry.
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  void **slot = reinterpret_cast<void **>(&abi);
  constexpr Py_ssize_t kSlots = sizeof(Entry) / sizeof(void *);
  if (nargs != kSlots) {
    PyErr_SetString(PyExc_TypeError, "bind: one address per entry point");
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < kSlots; ++i) {
    slot[i] = PyLong_AsVoidPtr(args[i]);
    if (!slot[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null address");
      return nullptr;
    }
  }
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"group_norm", (PyCFunction)(void (*)(void))group_norm, METH_FASTCALL,
     "group_norm(x, weight, bias, num_groups, eps, act_code, out_dtype, residual, channel_bias, return_sum[, functional]) -> y, (y, sum) "
     "or NotImplemented"},
    {"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, "bind(*addresses): the C ABI's entry points"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
