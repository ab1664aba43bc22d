// The small calls of core_scheduler_amd.ops in native code: outputs and workspace from torch's allocator, then the
// library call on the current stream.
//
// A step's small ops cost more host than device time, and most of that was Python's: 1.3 us for an allocation,
// 3-4 us of argument checks and ctypes conversions for a call, against 2.8 us for a launch, which stays.  One norm of
// 77 rows, forward and backward: 30.7 -> 16.7 us (11.4 since its backward is one launch and its outputs are made
// directly); the 25 calls of two short blocks 237 -> 115 (91-99 with fewer launches and cheaper outputs); embedding forward
// and backward of 4000 tokens 23 -> 17.7 (device time again).
//
// Every function takes the arguments of its counterpart in ops.py by position and returns NotImplemented for
// anything but the plain case: exact torch tensors, contiguous, on the current device, of exactly matching shapes and
// supported types, exact ints and floats, no torch mode active.  ops.py then goes its own way, which checks, raises
// or runs as ever; nothing is refused here.
#define PY_SSIZE_T_CLEAN
#include <ATen/Context.h>
#include <ATen/EmptyTensor.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <ATen/record_function.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <array>

#include "cs_hip_kernels.h"

namespace {

// ---------------------------------------------------------------- arguments
// What is not plain is not refused by an exception: one costs 2.5 us and more, on top of the Python body's call.
#define CS_PLAIN(condition) \
  if (!(condition)) Py_RETURN_NOTIMPLEMENTED

constexpr int kNoCode = -1;
int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return CS_F32;
    case at::kDouble: return CS_F64;
    case at::kHalf: return CS_F16;
    case at::kBFloat16: return CS_BF16;
    default: return kNoCode;
  }
}
int index_code(at::ScalarType t) { return t == at::kInt ? CS_I32 : t == at::kLong ? CS_I64 : kNoCode; }
template <typename... Codes>
bool supported(Codes... codes) {
  return ((codes != kNoCode) && ...);
}

// The arguments of one call; `device` is that of its first tensor, `plain` whether every one looked at is (what is
// not reads as nothing, zero or an undefined tensor).
struct Args {
  PyObject *const *items;
  Py_ssize_t n;
  int device = -1;
  bool plain = true;

  PyObject *at(Py_ssize_t i) const { return items[i]; }
  bool is(bool ok) {
    plain = plain && ok;
    return ok;
  }
  const at::Tensor &tensor(Py_ssize_t i) {
    static const at::Tensor none;
    PyObject *o = items[i];
    if (!is(THPVariable_CheckExact(o))) return none;
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!is(t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() && t.is_contiguous())) return none;
    if (device < 0) {
      device = t.get_device();
      is(device == c10::hip::current_device());
    }
    is(t.get_device() == device);
    return t;
  }
  const at::Tensor *optional(Py_ssize_t i) { return items[i] == Py_None ? nullptr : &tensor(i); }
  at::ScalarType dtype_or(Py_ssize_t i, at::ScalarType otherwise) {
    if (items[i] == Py_None || !is(THPDtype_Check(items[i]))) return otherwise;
    return reinterpret_cast<THPDtype *>(items[i])->scalar_type;
  }
  int64_t integer(Py_ssize_t i) {
    if (!is(PyLong_CheckExact(items[i]))) return 0;
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(items[i], &overflow);
    is(overflow == 0);
    return v;
  }
  double real(Py_ssize_t i) { return is(PyFloat_CheckExact(items[i])) ? PyFloat_AS_DOUBLE(items[i]) : 0.; }
  bool flag(Py_ssize_t i) {
    is(items[i] == Py_True || items[i] == Py_False);
    return items[i] == Py_True;
  }
  // the code of a text argument among `names`, in order from 0
  template <size_t N>
  int choice(Py_ssize_t i, const std::array<const char *, N> &names) {
    if (is(PyUnicode_CheckExact(items[i])))
      for (size_t k = 0; k < N; ++k)
        if (PyUnicode_CompareWithASCIIString(items[i], names[k]) == 0) return (int)k;
    is(false);
    return 0;
  }
};

const std::array<const char *, 2> kGelu = {"none", "tanh"};                // CS_GELU_*
const std::array<const char *, 3> kReductions = {"none", "mean", "sum"};  // CS_REDUCTION_*
static_assert(CS_GELU_ERF == 0 && CS_GELU_TANH == 1, "the order of kGelu");
static_assert(CS_REDUCTION_NONE == 0 && CS_REDUCTION_MEAN == 1 && CS_REDUCTION_SUM == 2, "the order of kReductions");

// ---------------------------------------------------------------- one call
// An output costs more host time than it should: of 0.70 us, torch's allocator takes 0.22 and the tensor object 0.1; the
// rest is the way there through the dispatcher, its device guard and its factory's options.  Where no dispatch key, no
// deterministic fill and no profiler has a part in that way the tensor is made directly (0.34 us; a norm, forward and
// backward, 13.2 -> 11.4).  The device is the current one (Args::tensor).
bool nothing_listens() {
  const auto expected = c10::default_included_set | c10::autocast_dispatch_keyset;
  return (c10::impl::tls_local_dispatch_key_set().included_ - expected).empty() &&
         !at::globalContext().deterministicAlgorithms() &&  // which fills new tensors
         !at::hasCallbacks();                               // that see every call of the dispatcher
}
thread_local bool direct_outputs;  // of the call under way (unlocked): asked once, the callbacks take a lock of 25 ns
at::Tensor empty(at::IntArrayRef sizes, at::ScalarType t, const at::Tensor &like) {
  c10::Allocator *const device_memory = c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::get();
  if (!direct_outputs) return at::empty(sizes, at::TensorOptions().dtype(t).device(like.device()));
  return at::detail::empty_generic(sizes, device_memory, c10::DispatchKeySet(c10::DispatchKey::CUDA), t, std::nullopt);
}
// (a dimension of one element may have any stride, which empty_like keeps)
bool rows_follow(const at::Tensor &t) {
  int64_t stride = 1;
  for (int64_t d = t.dim() - 1; d >= 0; stride *= t.size(d--))
    if (t.stride(d) != stride) return false;
  return true;
}
at::Tensor output_like(const at::Tensor &x) {
  return rows_follow(x) && !x.has_names() ? empty(x.sizes(), x.scalar_type(), x) : at::empty_like(x);
}
at::Tensor workspace(size_t bytes, const at::Tensor &like) {
  return empty({(int64_t)(bytes < 256 ? 256 : bytes)}, at::kByte, like);
}
void *ptr(const at::Tensor &t) { return t.data_ptr(); }
void *ptr(const at::Tensor *t) { return t ? t->data_ptr() : nullptr; }

bool aligned16(const at::Tensor &t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

PyObject *wrap(const at::Tensor &t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}
template <typename... Ts>
PyObject *tuple(const Ts &...ts) {
  PyObject *out = PyTuple_New(sizeof...(Ts));
  if (!out) throw python_error();
  Py_ssize_t i = 0;
  auto put = [&](const at::Tensor &t) {
    PyObject *o = wrap(t);
    if (!o) {
      Py_DECREF(out);
      throw python_error();
    }
    PyTuple_SET_ITEM(out, i++, o);
  };
  (put(ts), ...);
  return out;
}

// ops.py's way to an exception: core_scheduler_amd._capi.check(name, code)
void raise_for(const char *name, int code) {
  py::module_::import("core_scheduler_amd._capi").attr("check")(name, code);
}

// Allocations and the launch, without the interpreter's lock (a launch waits while the queue is full).
template <typename Body>
int unlocked(int device, Body &&body) {
  pybind11::gil_scoped_release release;
  direct_outputs = nothing_listens();
  return body(static_cast<void *>(c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream()));
}

// the rows of a norm; not plain without any
struct Ln {
  const at::Tensor &x;
  int64_t C = 0, rows = 0;
  explicit Ln(const at::Tensor &x_) : x(x_) {
    if (x.dim() == 0 || x.numel() == 0) return;
    C = x.size(-1);
    rows = x.numel() / C;
  }
  at::ScalarType stat() const { return x.scalar_type() == at::kDouble ? at::kDouble : at::kFloat; }
  bool params(const at::Tensor &gamma, const at::Tensor *beta) const {
    return rows > 0 && gamma.numel() == C &&
           (!beta || (beta->numel() == C && beta->scalar_type() == gamma.scalar_type()));
  }
  // what a backward call reads: dy as x, the statistics by row, gamma by column
  bool backward(const at::Tensor &dy, const at::Tensor &mean, const at::Tensor &rstd, const at::Tensor &gamma) const {
    return rows > 0 && dy.numel() == x.numel() && gamma.numel() == C && mean.numel() == rows && rstd.numel() == rows &&
           mean.scalar_type() == stat() && rstd.scalar_type() == stat();
  }
};
bool same(const at::Tensor &a, const at::Tensor &b) {
  return a.sizes() == b.sizes() && a.scalar_type() == b.scalar_type();
}
bool residual_of(const at::Tensor *dres, const at::Tensor &x, at::ScalarType t) {
  return !dres || (dres->sizes() == x.sizes() && dres->scalar_type() == t);
}

// ---------------------------------------------------------------------- ops
PyObject *gelu_forward(Args a) {  // x, approximate
  const at::Tensor &x = a.tensor(0);
  const int mode = a.choice(1, kGelu);
  CS_PLAIN(a.plain);
  const int dt = dtype_code(x.scalar_type());
  CS_PLAIN(supported(dt));
  at::Tensor y;
  const int code = unlocked(a.device, [&](void *s) {
    y = output_like(x);
    return cs_gelu_forward(ptr(x), ptr(y), x.numel(), dt, mode, s);
  });
  if (code != CS_OK) raise_for("cs_gelu_forward", code);
  return wrap(y);
}

PyObject *gelu_backward(Args a) {  // dy, x, approximate
  const at::Tensor &dy = a.tensor(0), &x = a.tensor(1);
  const int mode = a.choice(2, kGelu);
  CS_PLAIN(a.plain && dy.scalar_type() == x.scalar_type() && dy.numel() == x.numel());
  const int dt = dtype_code(x.scalar_type());
  CS_PLAIN(supported(dt));
  at::Tensor dx;
  const int code = unlocked(a.device, [&](void *s) {
    dx = output_like(x);
    return cs_gelu_backward(ptr(dy), ptr(x), ptr(dx), x.numel(), dt, mode, s);
  });
  if (code != CS_OK) raise_for("cs_gelu_backward", code);
  return wrap(dx);
}

PyObject *layernorm_forward(Args a) {  // x, gamma, beta, eps, out_dtype
  const at::Tensor &x = a.tensor(0), &gamma = a.tensor(1);
  const at::Tensor *beta = a.optional(2);
  const double eps = a.real(3);
  CS_PLAIN(a.plain);
  const at::ScalarType out = a.dtype_or(4, x.scalar_type());
  const Ln ln(x);
  const int dx = dtype_code(x.scalar_type()), dy = dtype_code(out), dg = dtype_code(gamma.scalar_type());
  CS_PLAIN(a.plain && ln.params(gamma, beta) && supported(dx, dy, dg));
  at::Tensor y, mean, rstd;
  const int code = unlocked(a.device, [&](void *s) {
    y = empty(x.sizes(), out, x);
    mean = empty({ln.rows}, ln.stat(), x);
    rstd = empty({ln.rows}, ln.stat(), x);
    return cs_layernorm_forward(ptr(x), ptr(gamma), ptr(beta), ptr(y), ptr(mean), ptr(rstd), ln.rows, ln.C, eps, dx, dy,
                                dg, s);
  });
  if (code != CS_OK) raise_for("cs_layernorm_forward", code);
  return tuple(y, mean, rstd);
}

PyObject *add_layernorm_forward(Args a) {  // x, residual, gamma, beta, eps, out_dtype; a new sum
  const at::Tensor &x = a.tensor(0), &residual = a.tensor(1), &gamma = a.tensor(2);
  const at::Tensor *beta = a.optional(3);
  const double eps = a.real(4);
  CS_PLAIN(a.plain);
  const at::ScalarType out = a.dtype_or(5, x.scalar_type());
  const Ln ln(x);
  const int dx = dtype_code(x.scalar_type()), dy = dtype_code(out), dg = dtype_code(gamma.scalar_type());
  CS_PLAIN(a.plain && same(x, residual) && ln.params(gamma, beta) && supported(dx, dy, dg));
  at::Tensor total, y, mean, rstd;
  const int code = unlocked(a.device, [&](void *s) {
    total = output_like(x);
    y = empty(x.sizes(), out, x);
    mean = empty({ln.rows}, ln.stat(), x);
    rstd = empty({ln.rows}, ln.stat(), x);
    return cs_add_layernorm_forward(ptr(x), ptr(residual), ptr(total), ptr(gamma), ptr(beta), ptr(y), ptr(mean), ptr(rstd),
                                    ln.rows, ln.C, eps, dx, dy, dg, s);
  });
  if (code != CS_OK) raise_for("cs_add_layernorm_forward", code);
  return tuple(total, y, mean, rstd);
}

// dy, x, mean, rstd, gamma, dx_dtype, dresidual: every gradient, none added to
PyObject *layernorm_backward(Args a) {
  const at::Tensor &dy = a.tensor(0), &x = a.tensor(1), &mean = a.tensor(2), &rstd = a.tensor(3), &gamma = a.tensor(4);
  const at::Tensor *dres = a.optional(6);
  CS_PLAIN(a.plain);
  const at::ScalarType out = a.dtype_or(5, x.scalar_type());
  const Ln ln(x);
  const int cdy = dtype_code(dy.scalar_type()), cx = dtype_code(x.scalar_type()), cdx = dtype_code(out);
  const int cg = dtype_code(gamma.scalar_type());
  CS_PLAIN(a.plain && residual_of(dres, x, out) && ln.backward(dy, mean, rstd, gamma) && supported(cdy, cx, cdx, cg));
  at::Tensor dx, dgamma, dbeta, ws;
  const int code = unlocked(a.device, [&](void *s) {
    dx = empty(x.sizes(), out, x);
    dgamma = empty({ln.C}, gamma.scalar_type(), x);
    dbeta = empty({ln.C}, gamma.scalar_type(), x);
    const size_t bytes = cs_layernorm_backward_workspace_bytes(ln.rows, ln.C);
    if (bytes) ws = workspace(bytes, x);
    void *w = bytes ? ptr(ws) : nullptr;
    if (dres)
      return cs_layernorm_backward_add(ptr(dy), ptr(x), ptr(mean), ptr(rstd), ptr(gamma), ptr(dres), ptr(dx), ptr(dgamma),
                                       ptr(dbeta), w, bytes, ln.rows, ln.C, cdy, cx, cdx, cg, 0, s);
    return cs_layernorm_backward(ptr(dy), ptr(x), ptr(mean), ptr(rstd), ptr(gamma), ptr(dx), ptr(dgamma), ptr(dbeta), w,
                                 bytes, ln.rows, ln.C, cdy, cx, cdx, cg, 0, s);
  });
  if (code != CS_OK) raise_for(dres ? "cs_layernorm_backward_add" : "cs_layernorm_backward", code);
  return tuple(dx, dgamma, dbeta);
}

// One call of a LayerNormBackwardChain that adds up what the call before it left, if any, in its own launch.
// dy, x, mean, rstd, gamma, dresidual, dx_dtype, pending partials, pending dgamma, pending dbeta, pending accumulate;
// the pending sums are of x's width and type.  Returns (dx, dgamma, dbeta, partials), partials None where the sums
// were taken at once.
PyObject *layernorm_backward_chained(Args a) {
  const at::Tensor &dy = a.tensor(0), &x = a.tensor(1), &mean = a.tensor(2), &rstd = a.tensor(3), &gamma = a.tensor(4);
  const at::Tensor *dres = a.optional(5);
  const at::Tensor *pend = a.optional(7), *pend_dgamma = a.optional(8), *pend_dbeta = a.optional(9);
  const bool pend_acc = a.flag(10);
  CS_PLAIN(a.plain);
  const at::ScalarType out = a.dtype_or(6, x.scalar_type());
  const Ln ln(x);
  const int cdy = dtype_code(dy.scalar_type()), cx = dtype_code(x.scalar_type()), cdx = dtype_code(out);
  const int cg = dtype_code(gamma.scalar_type());
  CS_PLAIN(a.plain && residual_of(dres, x, out) && ln.backward(dy, mean, rstd, gamma) && supported(cdy, cx, cdx, cg));
  const int64_t n = cs_layernorm_backward_partial_rows(ln.rows, ln.C, cx);
  CS_PLAIN(n > 0);
  const bool at_once = cs_layernorm_backward_one_launch(ln.rows, ln.C, cx) && aligned16(dy) && aligned16(x) &&
                       aligned16(gamma) && (!dres || aligned16(*dres));
  CS_PLAIN(!at_once || !pend);  // the earlier sums first, in a launch of their own
  at::Tensor dx, dgamma, dbeta, partials;
  const int code = unlocked(a.device, [&](void *s) {
    dx = empty(x.sizes(), out, x);
    dgamma = empty({ln.C}, gamma.scalar_type(), x);
    dbeta = empty({ln.C}, gamma.scalar_type(), x);
    if (at_once) {
      const size_t bytes = cs_layernorm_backward_workspace_bytes(ln.rows, ln.C);
      const at::Tensor ws = workspace(bytes, x);
      if (dres)
        return cs_layernorm_backward_add(ptr(dy), ptr(x), ptr(mean), ptr(rstd), ptr(gamma), ptr(dres), ptr(dx), ptr(dgamma),
                                         ptr(dbeta), ptr(ws), bytes, ln.rows, ln.C, cdy, cx, cdx, cg, 0, s);
      return cs_layernorm_backward(ptr(dy), ptr(x), ptr(mean), ptr(rstd), ptr(gamma), ptr(dx), ptr(dgamma), ptr(dbeta),
                                   ptr(ws), bytes, ln.rows, ln.C, cdy, cx, cdx, cg, 0, s);
    }
    partials = empty({n, 2, ln.C}, at::kFloat, x);
    return cs_layernorm_backward_rows_pending(
        ptr(dy), ptr(x), ptr(mean), ptr(rstd), ptr(gamma), ptr(dres), ptr(dx), (float *)ptr(partials),
        (size_t)partials.numel() * 4, (float *)ptr(pend), pend ? pend->size(0) : 0, ptr(pend_dgamma), ptr(pend_dbeta),
        pend_acc ? 1 : 0, ln.rows, ln.C, cdy, cx, cdx, cg, s);
  });
  if (code != CS_OK) raise_for(at_once ? "cs_layernorm_backward" : "cs_layernorm_backward_rows_pending", code);
  return tuple(dx, dgamma, dbeta, partials);
}

PyObject *embedding_forward(Args a) {  // weight, indices
  const at::Tensor &w = a.tensor(0), &ids = a.tensor(1);
  CS_PLAIN(a.plain && w.dim() == 2);
  const int dt = dtype_code(w.scalar_type()), it = index_code(ids.scalar_type());
  CS_PLAIN(supported(dt, it));
  std::vector<int64_t> shape(ids.sizes().begin(), ids.sizes().end());
  shape.push_back(w.size(1));
  at::Tensor out;
  const int code = unlocked(a.device, [&](void *s) {
    out = empty(shape, w.scalar_type(), w);
    return cs_embedding_forward(ptr(w), ptr(ids), ptr(out), ids.numel(), w.size(1), w.size(0), dt, it, s);
  });
  if (code != CS_OK) raise_for("cs_embedding_forward", code);
  return wrap(out);
}

PyObject *embedding_forward_add(Args a) {  // wte, wpe, indices
  const at::Tensor &w = a.tensor(0), &p = a.tensor(1), &ids = a.tensor(2);
  CS_PLAIN(a.plain && w.dim() == 2 && p.dim() == 2 && ids.dim() == 2);
  const int64_t B = ids.size(0), T = ids.size(1), C = w.size(1);
  const int dt = dtype_code(w.scalar_type()), it = index_code(ids.scalar_type());
  CS_PLAIN(p.size(0) >= T && p.size(1) == C && p.scalar_type() == w.scalar_type() && supported(dt, it));
  at::Tensor out;
  const int code = unlocked(a.device, [&](void *s) {
    out = empty({B, T, C}, w.scalar_type(), w);
    return cs_embedding_forward_add(ptr(w), ptr(p), ptr(ids), ptr(out), B, T, C, w.size(0), dt, it, s);
  });
  if (code != CS_OK) raise_for("cs_embedding_forward_add", code);
  return wrap(out);
}

PyObject *embedding_backward(Args a) {  // dout, indices, num_weights, padding_idx, scale_grad_by_freq; a new dweight
  const at::Tensor &dout = a.tensor(0), &ids = a.tensor(1);
  const int64_t V = a.integer(2), pad = a.integer(3);
  const bool by_freq = a.flag(4);
  CS_PLAIN(a.plain && dout.dim() > 0 && V >= 0);
  const int64_t n = ids.numel(), C = dout.size(-1);
  const int dt = dtype_code(dout.scalar_type()), it = index_code(ids.scalar_type());
  CS_PLAIN(dout.numel() == n * C && supported(dt, it));
  at::Tensor dw, ws;
  const int code = unlocked(a.device, [&](void *s) {
    dw = empty({V, C}, dout.scalar_type(), dout);
    const size_t bytes = cs_embedding_backward_workspace_bytes(n, C, V);
    ws = workspace(bytes, dout);
    return (by_freq ? cs_embedding_backward_scaled : cs_embedding_backward)(ptr(dout), ptr(ids), ptr(dw), ptr(ws), bytes, n,
                                                                           C, V, pad, dt, it, 0, s);
  });
  if (code != CS_OK) raise_for(by_freq ? "cs_embedding_backward_scaled" : "cs_embedding_backward", code);
  return wrap(dw);
}

PyObject *embedding_backward_fused(Args a) {  // dout, indices, num_weights; new dwte and dwpe
  const at::Tensor &dout = a.tensor(0), &ids = a.tensor(1);
  const int64_t V = a.integer(2);
  CS_PLAIN(a.plain && dout.dim() == 3 && V >= 0);
  const int64_t B = dout.size(0), T = dout.size(1), C = dout.size(2);
  const int dt = dtype_code(dout.scalar_type()), it = index_code(ids.scalar_type());
  CS_PLAIN(ids.numel() == B * T && supported(dt, it));
  at::Tensor dwte, dwpe, ws;
  const int code = unlocked(a.device, [&](void *s) {
    dwte = empty({V, C}, dout.scalar_type(), dout);
    dwpe = empty({T, C}, dout.scalar_type(), dout);
    const size_t bytes = cs_embedding_backward_workspace_bytes(B * T, C, V);
    ws = workspace(bytes, dout);
    return cs_embedding_backward_fused(ptr(dout), ptr(ids), ptr(dwte), ptr(dwpe), ptr(ws), bytes, B, T, C, V, dt, it, 0, s);
  });
  if (code != CS_OK) raise_for("cs_embedding_backward_fused", code);
  return tuple(dwte, dwpe);
}

// logits, targets, num_classes, ignore_index, reduction, dloss, want_dlogits, dlogits_dtype, class_weight;
// a new dlogits.  Returns (loss, row_loss, dlogits, total_weight).
PyObject *fused_classifier(Args a) {
  const at::Tensor &logits = a.tensor(0), &targets = a.tensor(1);
  const at::Tensor *weight = a.optional(8);
  CS_PLAIN(a.plain && logits.dim() == 2);
  const int64_t N = logits.size(0), stride = logits.size(1);
  const int64_t V = a.at(2) == Py_None ? stride : a.integer(2), ignore = a.integer(3);
  const int reduction = a.choice(4, kReductions);
  const float dloss = (float)a.real(5);
  const bool want = a.flag(6);
  const at::ScalarType out = want ? a.dtype_or(7, logits.scalar_type()) : logits.scalar_type();
  const int dl = dtype_code(logits.scalar_type()), dd = dtype_code(out);
  CS_PLAIN(a.plain && targets.scalar_type() == at::kLong && targets.numel() == N && supported(dl, dd));
  CS_PLAIN(!weight || (weight->scalar_type() == at::kFloat && weight->numel() == V));
  at::Tensor row_loss, loss, total, d, ws;
  const int code = unlocked(a.device, [&](void *s) {
    row_loss = empty({N}, at::kFloat, logits);
    loss = empty({}, at::kFloat, logits);
    total = empty({}, at::kFloat, logits);
    if (want) d = empty(logits.sizes(), out, logits);
    const size_t bytes = cs_fused_classifier_workspace_bytes(N);
    ws = workspace(bytes, logits);
    void *pd = want ? ptr(d) : nullptr;
    if (weight)
      return cs_fused_classifier_weighted(ptr(logits), pd, (const int64_t *)ptr(targets), (const float *)ptr(weight),
                                          (float *)ptr(row_loss), (float *)ptr(loss), (float *)ptr(total), ptr(ws), bytes, N,
                                          V, stride, ignore, reduction, dloss, dl, dd, s);
    return cs_fused_classifier(ptr(logits), pd, (const int64_t *)ptr(targets), (float *)ptr(row_loss), (float *)ptr(loss),
                               (float *)ptr(total), ptr(ws), bytes, N, V, stride, ignore, reduction, dloss, dl, dd, s);
  });
  if (code != CS_OK) raise_for(weight ? "cs_fused_classifier_weighted" : "cs_fused_classifier", code);
  return tuple(reduction == CS_REDUCTION_NONE ? row_loss : loss, row_loss, d, total);
}

// -------------------------------------------------------------------- module
template <PyObject *(*FN)(Args), Py_ssize_t COUNT>
PyObject *entry(PyObject *, PyObject *const *items, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  // a torch mode sees the calls that ops.py makes
  if (n != COUNT || at::impl::torch_function_mode_enabled() || c10::impl::dispatch_mode_enabled())
    Py_RETURN_NOTIMPLEMENTED;
  try {
    return FN(Args{items, n});
  } catch (py::error_already_set &e) {
    e.restore();
    return nullptr;
  }
  END_HANDLE_TH_ERRORS
}
#define CS_ENTRY(fn, count) \
  {#fn, (PyCFunction)(void (*)(void))entry<fn, count>, METH_FASTCALL, nullptr}

PyMethodDef methods[] = {CS_ENTRY(gelu_forward, 2),
                         CS_ENTRY(gelu_backward, 3),
                         CS_ENTRY(layernorm_forward, 5),
                         CS_ENTRY(add_layernorm_forward, 6),
                         CS_ENTRY(layernorm_backward, 7),
                         CS_ENTRY(layernorm_backward_chained, 11),
                         CS_ENTRY(embedding_forward, 2),
                         CS_ENTRY(embedding_forward_add, 3),
                         CS_ENTRY(embedding_backward, 5),
                         CS_ENTRY(embedding_backward_fused, 3),
                         CS_ENTRY(fused_classifier, 9),
                         {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_cs_calls", "Native forms of the small calls of ops.py.", -1, methods};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject *PyInit__cs_calls(void) {
  if (cs_hip_abi_version() != 1) {  // _capi.load() says so to whoever calls an op
    PyErr_SetString(PyExc_ImportError, "libcs_hip_kernels.so has another ABI version");
    return nullptr;
  }
  return PyModule_Create(&module);
}
