// The host path between torch tensors and the C ABI of include/ttt_mi355x.h, as a CPython extension (_ttt_torch.so):
// argument checks, output allocation and the library call of every function in inner.py.
//
// Why native: a call of a few tokens is one kernel of about 10 us, and the same work in Python (ctypes conversions,
// torch.empty, shape tuples, slices) took 17 us in front of it, 25 - 110 us for the calls that allocate more outputs or
// launch several kernels.  Here tensors are unpacked, checked and allocated through torch's C++ interface: a decode
// call costs the host about as long as its kernel runs.  Nothing is kept between calls.
//
// Plain host code (g++), linked against libttt_mi355x.so and torch.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <cstdarg>
#include <cstdio>
#include <string>
#include <vector>

#include "../../include/ttt_mi355x.h"

namespace {

PyObject* g_error = nullptr;  // TttError(code, message), given by the package when it loads the module

struct TttFailure {
  int code;
  std::string msg;
};
struct PyFailure {};  // a Python exception is already set

[[noreturn]] void fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  throw TttFailure{code, buf};
}
void check(int rc) {
  if (rc != TTT_OK) throw TttFailure{rc, ttt_last_error()};
}

// ---- arguments -------------------------------------------------------------------------------
using Shape = at::IntArrayRef;

std::string text(Shape s) {
  std::string r = "(";
  for (size_t i = 0; i < s.size(); ++i) r += (i ? ", " : "") + std::to_string(s[i]);
  return r + (s.size() == 1 ? ",)" : ")");
}

const at::Tensor& tensor(PyObject* o, const char* name) {
  if (!THPVariable_Check(o)) {
    PyErr_Format(PyExc_TypeError, "%s: a torch tensor is needed, got %s", name, Py_TYPE(o)->tp_name);
    throw PyFailure{};
  }
  return THPVariable_Unpack(o);
}
int64_t integer(PyObject* o) {
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw PyFailure{};
  return v;
}
float real(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw PyFailure{};
  return (float)v;
}
int io_of(const at::Tensor& t) {
  if (t.scalar_type() == at::kFloat) return TTT_F32;
  if (t.scalar_type() == at::kBFloat16) return TTT_BF16;
  fail(TTT_ERR_UNSUPPORTED, "activation dtype %s (f32 or bf16 only)", c10::toString(t.scalar_type()));
}

// Tensors that a call made itself (packed copies, scratch): alive until its work is enqueued; the allocator hands their
// memory to later work of the same stream only.
using Keep = std::vector<at::Tensor>;

void must_be(const at::Tensor& t, Shape shape, at::ScalarType dtype, const char* name) {
  if (t.sizes() != shape) fail(TTT_ERR_SHAPE, "%s: shape %s != %s", name, text(t.sizes()).c_str(), text(shape).c_str());
  if (t.scalar_type() != dtype)
    fail(TTT_ERR_SHAPE, "%s: dtype %s != %s", name, c10::toString(t.scalar_type()), c10::toString(dtype));
  if (!t.is_cuda()) fail(TTT_ERR_NULL, "%s is not a device tensor", name);
}
void* packed(const at::Tensor& t, Keep& keep) {
  if (t.is_contiguous()) return t.data_ptr();
  keep.push_back(t.contiguous());
  return keep.back().data_ptr();
}
void* need(const at::Tensor& t, Shape shape, at::ScalarType dtype, const char* name, Keep& keep) {
  must_be(t, shape, dtype, name);
  return packed(t, keep);
}
void* need(PyObject* o, Shape shape, at::ScalarType dtype, const char* name, Keep& keep) {
  return need(tensor(o, name), shape, dtype, name, keep);
}
float* need_f32(PyObject* o, Shape shape, const char* name, Keep& keep) {
  return static_cast<float*>(need(o, shape, at::kFloat, name, keep));
}
// token_eta: the first n entries are read; any dtype
const float* eta_of(PyObject* o, int64_t n, Keep& keep) {
  const at::Tensor& t = tensor(o, "token_eta");
  if (t.numel() < n) fail(TTT_ERR_SHAPE, "token_eta shorter than mini_batch");
  if (!t.is_cuda()) fail(TTT_ERR_NULL, "token_eta is not a device tensor");
  if (t.scalar_type() == at::kFloat) return static_cast<const float*>(packed(t, keep));
  keep.push_back(t.to(at::kFloat).contiguous());
  return static_cast<const float*>(keep.back().data_ptr());
}

// ---- outputs, stream, call -------------------------------------------------------------------
at::Tensor empty(Shape shape, at::ScalarType dtype, c10::Device dev) {
  return at::Tensor(at::detail::empty_cuda(shape, dtype, dev, std::nullopt));
}
template <class T = float>
T* ptr(const at::Tensor& t) {
  return static_cast<T*>(t.data_ptr());
}

// The library call of one function: on the current stream of the tensors' device, that device current meanwhile, the
// interpreter lock released (launching waits when the queue is full).
template <class F>
void enqueue(c10::Device dev, F&& call) {
  struct Scope {
    c10::DeviceIndex want, had;
    PyThreadState* py;
    explicit Scope(c10::DeviceIndex d) : want(d), had(c10::hip::ExchangeDevice(d)), py(PyEval_SaveThread()) {}
    ~Scope() {
      PyEval_RestoreThread(py);
      if (had != want) c10::hip::ExchangeDevice(had);
    }
  };
  void* stream = static_cast<void*>(c10::hip::getCurrentHIPStream(dev.index()).stream());
  int rc;
  {
    const Scope scope(dev.index());
    rc = call(stream);
  }
  check(rc);
}

PyObject* wrap(at::Tensor&& t) {
  PyObject* o = THPVariable_Wrap(std::move(t));
  if (o == nullptr) throw PyFailure{};
  return o;
}
PyObject* wrap_tuple(std::initializer_list<at::Tensor*> ts) {
  PyObject* r = PyTuple_New((Py_ssize_t)ts.size());
  if (r == nullptr) throw PyFailure{};
  Py_ssize_t i = 0;
  for (at::Tensor* t : ts) PyTuple_SET_ITEM(r, i++, THPVariable_Wrap(std::move(*t)));
  return r;
}
void put(PyObject* dict, const char* key, at::Tensor&& t) {
  PyObject* o = wrap(std::move(t));
  const int rc = PyDict_SetItemString(dict, key, o);
  Py_DECREF(o);
  if (rc != 0) throw PyFailure{};
}

ttt_desc desc_of(int64_t B, int64_t H, int64_t seq, int64_t d, int64_t K, float eps, int64_t ci, int io, bool per_batch,
                 int64_t stride, int64_t format, int64_t hint) {
  ttt_desc r;
  r.batch = (int32_t)B; r.heads = (int32_t)H; r.seq = (int32_t)seq; r.head_dim = (int32_t)d;
  r.mini_batch = (int32_t)K; r.eps = eps; r.checkpoint_interval = (int32_t)ci; r.io_dtype = io;
  r.state_per_batch = per_batch ? 1 : 0; r.seq_stride = (int32_t)stride; r.checkpoint_format = (int32_t)format;
  r.kernel_hint = (int32_t)hint;
  return r;
}
struct Rows {  // xq [B,H,seq,d], which sets the shape and dtype of the others
  const at::Tensor& t;
  int64_t B, H, seq, d;
  at::ScalarType dtype;
  c10::Device dev;
  explicit Rows(PyObject* o) : t(tensor(o, "xq")), dtype(t.scalar_type()), dev(t.device()) {
    if (t.dim() != 4) fail(TTT_ERR_SHAPE, "xq: four dimensions are needed, got %s", text(t.sizes()).c_str());
    B = t.size(0); H = t.size(1); seq = t.size(2); d = t.size(3);
  }
  std::array<int64_t, 4> shape() const { return {B, H, seq, d}; }
};

// ---- TTT-Linear forward ----------------------------------------------------------------------
// Tokens between consecutive (batch, head) units if t ([B,H,seq,d] or [B,H,seq]) is a window along seq of a dense
// tensor, else -1.
int64_t seq_pitch(const at::Tensor& t) {
  const auto st = t.strides();
  const int64_t trail = t.dim() == 4 ? t.size(3) : 1;
  if (t.dim() == 4 ? (st[3] != 1 || st[2] != trail) : st[2] != 1) return -1;
  if (st[1] % trail != 0 || st[0] != t.size(1) * st[1]) return -1;
  const int64_t pitch = st[1] / trail;
  return pitch >= t.size(2) ? pitch : -1;
}

// (xq, xk, xv, weight, bias, token_eta, lr, ln_weight, ln_bias, mini_batch, eps, checkpoint_interval, want_checkpoints,
//  out or None, checkpoint_format, kernel_hint)
PyObject* linear_forward(PyObject* const* a) {
  Keep keep;
  const Rows q(a[0]);
  const int64_t B = q.B, H = q.H, seq = q.seq, d = q.d, K = integer(a[9]);
  const std::array<int64_t, 4> rows = q.shape();
  const std::array<int64_t, 3> gates = {B, H, seq};
  const at::Tensor &xk = tensor(a[1], "xk"), &xv = tensor(a[2], "xv"), &lr = tensor(a[6], "ttt_lr_eta");
  must_be(q.t, rows, q.dtype, "xq");
  must_be(xk, rows, q.dtype, "xk");
  must_be(xv, rows, q.dtype, "xv");
  must_be(lr, gates, q.dtype, "ttt_lr_eta");
  // sequence windows of dense tensors are processed in place (desc.seq_stride) when inputs and the caller's output
  // window share one pitch; anything else is packed first
  const at::Tensor* given = a[13] == Py_None ? nullptr : &tensor(a[13], "out");
  int64_t pitch = 0;
  if (given != nullptr && given->dim() == 4) {
    const int64_t p = seq_pitch(*given);
    if (p > 0 && p != seq && seq_pitch(q.t) == p && seq_pitch(xk) == p && seq_pitch(xv) == p && seq_pitch(lr) == p) pitch = p;
  }
  auto src = [&](const at::Tensor& t) { return pitch ? t.data_ptr() : packed(t, keep); };
  void *pq = src(q.t), *pk = src(xk), *pv = src(xv), *pl = src(lr);
  const bool per_batch = tensor(a[3], "weight").dim() == 4;
  const std::array<int64_t, 4> W4 = {B, H, d, d};
  const std::array<int64_t, 3> b3 = {B, H, d};
  const std::array<int64_t, 2> hd = {H, d};
  const float* W0 = need_f32(a[3], per_batch ? Shape(W4) : Shape(W4).slice(1), "weight", keep);
  const float* b0 = need_f32(a[4], per_batch ? Shape(b3) : Shape(b3).slice(1), "bias", keep);
  const float* gam = need_f32(a[7], hd, "ln_weight", keep);
  const float* bet = need_f32(a[8], hd, "ln_bias", keep);
  const float* te = eta_of(a[5], K, keep);
  const ttt_desc desc = desc_of(B, H, seq, d, K, real(a[10]), integer(a[11]), io_of(q.t), per_batch, pitch, integer(a[14]),
                                integer(a[15]));
  check(ttt_linear_supported(&desc));
  const bool in_place = given != nullptr && (pitch != 0 || given->is_contiguous());
  if (in_place) must_be(*given, rows, q.dtype, "out");
  at::Tensor out = in_place ? *given : empty(rows, q.dtype, q.dev);
  at::Tensor W = empty(W4, at::kFloat, q.dev), b = empty(b3, at::kFloat, q.dev), Wc, bc;
  const bool want = PyObject_IsTrue(a[12]) == 1;
  if (want) {
    const int64_t n = ttt_linear_num_checkpoints(&desc);
    Wc = empty({B, H, n, d, d}, at::kFloat, q.dev);
    bc = empty({B, H, n, d}, at::kFloat, q.dev);
  }
  enqueue(q.dev, [&](void* s) {
    return ttt_linear_fwd(&desc, pq, pk, pv, W0, b0, te, pl, gam, bet, out.data_ptr(), ptr(W), ptr(b),
                          want ? ptr(Wc) : nullptr, want ? ptr(bc) : nullptr, s);
  });
  if (given != nullptr && !in_place) {
    given->copy_(out);
    out = *given;
  }
  return want ? wrap_tuple({&out, &W, &b, &Wc, &bc}) : wrap_tuple({&out, &W, &b});
}

// A layer's pass over the tokens start .. stop of its inputs: whole mini-batches in one launch, a remainder as one
// short mini-batch in the same launch where the library has one, or behind it.  (xq, xk, xv, weight, bias, token_eta, lr, ln_weight, ln_bias, mini_batch, eps,
// checkpoint_interval, start, stop) -> (out, weight, bias); of token_eta the first K entries from start on are read, and
// those of a remainder; the state goes in shared over the batch ([H,d,d], [H,d]) or per
// batch element and comes out per batch element.
PyObject* linear_layer_forward(PyObject* const* a) {
  Keep keep;
  const Rows q(a[0]);
  const int64_t B = q.B, H = q.H, d = q.d, K = integer(a[9]), start = integer(a[12]), stop = integer(a[13]);
  const int64_t n = stop - start;
  if (start < 0 || n <= 0 || stop > q.seq)
    fail(TTT_ERR_SHAPE, "tokens %lld .. %lld of a sequence of %lld", (long long)start, (long long)stop, (long long)q.seq);
  if (K < 1) fail(TTT_ERR_SHAPE, "mini_batch %lld", (long long)K);
  const std::array<int64_t, 4> whole = q.shape(), rows = {B, H, n, d};
  const std::array<int64_t, 3> gates = {B, H, q.seq};
  const at::Tensor &xk = tensor(a[1], "xk"), &xv = tensor(a[2], "xv"), &lr = tensor(a[6], "ttt_lr_eta");
  must_be(q.t, whole, q.dtype, "xq");
  must_be(xk, whole, q.dtype, "xk");
  must_be(xv, whole, q.dtype, "xv");
  must_be(lr, gates, q.dtype, "ttt_lr_eta");
  // a window of the sequence is packed (the output is dense and the kernels take one pitch for both)
  auto src = [&](const at::Tensor& t) {
    return static_cast<char*>(n == q.seq ? packed(t, keep) : packed(t.slice(2, start, stop), keep));
  };
  // t.slice() is a temporary: a contiguous one is its parent's memory (kept by the caller), any other was copied
  char *pq = src(q.t), *pk = src(xk), *pv = src(xv), *pl = src(lr);
  const std::array<int64_t, 4> W4 = {B, H, d, d};
  const std::array<int64_t, 3> b3 = {B, H, d};
  const std::array<int64_t, 2> hd = {H, d};
  const bool per_batch = tensor(a[3], "weight").dim() == 4;
  const float* W0 = need_f32(a[3], per_batch ? Shape(W4) : Shape(W4).slice(1), "weight", keep);
  const float* b0 = need_f32(a[4], per_batch ? Shape(b3) : Shape(b3).slice(1), "bias", keep);
  const float* gam = need_f32(a[7], hd, "ln_weight", keep);
  const float* bet = need_f32(a[8], hd, "ln_bias", keep);
  const int io = io_of(q.t);
  const int64_t size = io == TTT_F32 ? 4 : 2, full = n / K * K, rest = n - full;
  // a launch reads as many entries as a mini-batch of it has tokens
  const float* te = eta_of(a[5], rest > 0 ? stop : start + K, keep) + start;
  const float eps = real(a[10]);
  const int64_t ci = integer(a[11]);
  // both launches' descs before anything is allocated or enqueued
  ttt_desc desc[2];
  int calls = 0;
  if (full > 0) desc[calls++] = desc_of(B, H, full, d, K, eps, ci, io, per_batch, rest > 0 ? n : 0, 0, 0);
  if (rest > 0) desc[calls++] = desc_of(B, H, rest, d, rest, eps, ci, io, per_batch || full > 0, full > 0 ? n : 0, 0, 0);
  for (int i = 0; i < calls; ++i) check(ttt_linear_supported(&desc[i]));
  at::Tensor out = empty(rows, q.dtype, q.dev), W[2], b[2];
  char* po = static_cast<char*>(out.data_ptr());
  W[0] = empty(W4, at::kFloat, q.dev);
  b[0] = empty(b3, at::kFloat, q.dev);
  if (calls == 2) {  // in one launch where there is one
    bool one = true;
    enqueue(q.dev, [&](void* s) {
      one = ttt_linear_fwd_takes_rest(&desc[0], (int32_t)rest) == 1;
      return one ? ttt_linear_fwd_with_rest(&desc[0], (int32_t)rest, pq, pk, pv, W0, b0, te, pl, gam, bet, po, ptr(W[0]), ptr(b[0]), s)
                 : (int)TTT_OK;
    });
    if (one) return wrap_tuple({&out, &W[0], &b[0]});
    W[1] = empty(W4, at::kFloat, q.dev);
    b[1] = empty(b3, at::kFloat, q.dev);
  }
  enqueue(q.dev, [&](void* s) {
    for (int i = 0; i < calls; ++i) {
      const int64_t at = i == 0 ? 0 : full, rb = at * d * size;
      const int rc = ttt_linear_fwd(&desc[i], pq + rb, pk + rb, pv + rb, i == 0 ? W0 : ptr(W[0]), i == 0 ? b0 : ptr(b[0]),
                                    te + at, pl + at * size, gam, bet, po + rb, ptr(W[i]), ptr(b[i]), nullptr, nullptr, s);
      if (rc != TTT_OK) return rc;
    }
    return (int)TTT_OK;
  });
  return wrap_tuple({&out, &W[calls - 1], &b[calls - 1]});
}

// (xq, xk, xv, weight, bias, token_eta, lr, ln_weight, ln_bias, mini_batch, beta1, beta2, adam_eps, adam_lr,
//  moments or None, step, eps)
PyObject* linear_adam_forward(PyObject* const* a) {
  Keep keep;
  const Rows q(a[0]);
  const int64_t B = q.B, H = q.H, seq = q.seq, d = q.d, K = integer(a[9]);
  const std::array<int64_t, 4> rows = q.shape(), W4 = {B, H, d, d};
  const std::array<int64_t, 3> gates = {B, H, seq}, b3 = {B, H, d};
  const std::array<int64_t, 2> hd = {H, d};
  void* pq = need(q.t, rows, q.dtype, "xq", keep);
  void* pk = need(a[1], rows, q.dtype, "xk", keep);
  void* pv = need(a[2], rows, q.dtype, "xv", keep);
  const bool per_batch = tensor(a[3], "weight").dim() == 4;
  const float* W0 = need_f32(a[3], per_batch ? Shape(W4) : Shape(W4).slice(1), "weight", keep);
  const float* b0 = need_f32(a[4], per_batch ? Shape(b3) : Shape(b3).slice(1), "bias", keep);
  const at::Tensor& eta = tensor(a[5], "token_eta");
  if (eta.dim() != 1 || eta.size(0) < K || eta.scalar_type() != at::kFloat)
    fail(TTT_ERR_SHAPE, "token_eta: %lld f32 entries are needed", (long long)K);
  const float* te = eta_of(a[5], K, keep);
  void* pl = need(a[6], gates, q.dtype, "ttt_lr_eta", keep);
  const float* gam = need_f32(a[7], hd, "ln_weight", keep);
  const float* bet = need_f32(a[8], hd, "ln_bias", keep);
  const float* m_in[4] = {nullptr, nullptr, nullptr, nullptr};
  if (a[14] != Py_None) {
    PyObject* seqm = PySequence_Fast(a[14], "moments: a sequence of four tensors is needed");
    if (seqm == nullptr) throw PyFailure{};
    keep.reserve(keep.size() + 8);
    const Py_ssize_t n = PySequence_Fast_GET_SIZE(seqm);
    try {
      for (Py_ssize_t i = 0; i < 4 && i < n; ++i)
        m_in[i] = need_f32(PySequence_Fast_GET_ITEM(seqm, i), i % 2 == 0 ? Shape(W4) : Shape(b3), "moment", keep);
    } catch (...) {
      Py_DECREF(seqm);
      throw;
    }
    Py_DECREF(seqm);
  }
  const ttt_desc desc = desc_of(B, H, seq, d, K, real(a[16]), 1, io_of(q.t), per_batch, 0, 0, 0);
  check(ttt_linear_adam_supported(&desc));
  const float beta1 = real(a[10]), beta2 = real(a[11]), aeps = real(a[12]), alr = real(a[13]);
  const int64_t step = integer(a[15]);
  at::Tensor out = empty(rows, q.dtype, q.dev), W = empty(W4, at::kFloat, q.dev), b = empty(b3, at::kFloat, q.dev);
  at::Tensor m[4] = {empty(W4, at::kFloat, q.dev), empty(b3, at::kFloat, q.dev), empty(W4, at::kFloat, q.dev),
                     empty(b3, at::kFloat, q.dev)};
  enqueue(q.dev, [&](void* s) {
    return ttt_linear_adam_fwd(&desc, pq, pk, pv, W0, b0, m_in[0], m_in[1], m_in[2], m_in[3], (int)step, beta1, beta2, aeps,
                               alr, te, pl, gam, bet, out.data_ptr(), ptr(W), ptr(b), ptr(m[0]), ptr(m[1]), ptr(m[2]),
                               ptr(m[3]), s);
  });
  PyObject* r = PyTuple_New(5);
  if (r == nullptr) throw PyFailure{};
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(out)));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(std::move(W)));
  PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(std::move(b)));
  PyTuple_SET_ITEM(r, 3, wrap_tuple({&m[0], &m[1], &m[2], &m[3]}));
  PyTuple_SET_ITEM(r, 4, PyLong_FromLongLong(step + seq / K));
  return r;
}

// ---- TTT-Linear backward ---------------------------------------------------------------------
// (xq, xk, xv, weight, bias, token_eta, lr, ln_weight, ln_bias, weight_ckpt, bias_ckpt, grad_output, mini_batch, eps,
//  checkpoint_interval, grad_weight_out or None, grad_bias_out or None, checkpoint_format, kernel_hint,
//  workspace: a tensor, None or True to allocate one, False for the entry point without) -> dict
PyObject* linear_backward(PyObject* const* a) {
  Keep keep;
  const Rows q(a[0]);
  const int64_t B = q.B, H = q.H, seq = q.seq, d = q.d, K = integer(a[12]);
  const std::array<int64_t, 4> rows = q.shape(), W4 = {B, H, d, d};
  const std::array<int64_t, 3> gates = {B, H, seq}, b3 = {B, H, d};
  const std::array<int64_t, 2> hd = {H, d};
  void* pq = need(q.t, rows, q.dtype, "xq", keep);
  void* pk = need(a[1], rows, q.dtype, "xk", keep);
  void* pv = need(a[2], rows, q.dtype, "xv", keep);
  void* pg = need(a[11], rows, q.dtype, "grad_output", keep);
  void* pl = need(a[6], gates, q.dtype, "ttt_lr_eta", keep);
  const bool per_batch = tensor(a[3], "weight").dim() == 4;
  const float* W0 = need_f32(a[3], per_batch ? Shape(W4) : Shape(W4).slice(1), "weight", keep);
  const float* b0 = need_f32(a[4], per_batch ? Shape(b3) : Shape(b3).slice(1), "bias", keep);
  const float* gam = need_f32(a[7], hd, "ln_weight", keep);
  const float* bet = need_f32(a[8], hd, "ln_bias", keep);
  const float* te = eta_of(a[5], K, keep);
  const ttt_desc desc = desc_of(B, H, seq, d, K, real(a[13]), integer(a[14]), io_of(q.t), per_batch, 0, integer(a[17]),
                                integer(a[18]));
  check(ttt_linear_bwd_supported(&desc));
  const int64_t n = ttt_linear_num_checkpoints(&desc);
  const float* Wc = need_f32(a[9], {B, H, n, d, d}, "weight_ckpt", keep);
  const float* bc = need_f32(a[10], {B, H, n, d}, "bias_ckpt", keep);
  const float* gW = a[15] == Py_None ? nullptr : need_f32(a[15], W4, "grad_weight_out", keep);
  const float* gb = a[16] == Py_None ? nullptr : need_f32(a[16], b3, "grad_bias_out", keep);
  at::Tensor dq = empty(rows, q.dtype, q.dev), dk = empty(rows, q.dtype, q.dev), dv = empty(rows, q.dtype, q.dev),
             dW = empty(W4, at::kFloat, q.dev), db = empty(b3, at::kFloat, q.dev), dl = empty(gates, q.dtype, q.dev),
             dt = empty({seq}, at::kFloat, q.dev), dg = empty(hd, at::kFloat, q.dev), de = empty(hd, at::kFloat, q.dev);
  // a desc whose backward can use a workspace gets one
  const int64_t bytes = ttt_linear_bwd_workspace_bytes(&desc);
  if (bytes < 0) check((int)bytes);
  void* ws = nullptr;
  if (bytes > 0 && a[19] != Py_False) {
    if (a[19] == Py_None || a[19] == Py_True) {
      keep.push_back(empty({bytes}, at::kByte, q.dev));
      ws = keep.back().data_ptr();
    } else {
      const at::Tensor& t = tensor(a[19], "workspace");
      if ((int64_t)t.nbytes() < bytes) fail(TTT_ERR_SHAPE, "workspace holds fewer than %lld bytes", (long long)bytes);
      ws = t.data_ptr();
    }
  }
  enqueue(q.dev, [&](void* s) {
    return ttt_linear_bwd_ws(&desc, pq, pk, pv, W0, b0, te, pl, gam, bet, Wc, bc, pg, gW, gb, dq.data_ptr(), dk.data_ptr(),
                             dv.data_ptr(), ptr(dW), ptr(db), dl.data_ptr(), ptr(dt), ptr(dg), ptr(de), ws, s);
  });
  PyObject* r = PyDict_New();
  if (r == nullptr) throw PyFailure{};
  put(r, "grad_xq", std::move(dq));
  put(r, "grad_xk", std::move(dk));
  put(r, "grad_xv", std::move(dv));
  put(r, "grad_weight", std::move(dW));
  put(r, "grad_bias", std::move(db));
  put(r, "grad_ttt_lr_eta", std::move(dl));
  put(r, "grad_token_eta", std::move(dt));
  put(r, "grad_ln_weight", std::move(dg));
  put(r, "grad_ln_bias", std::move(de));
  return r;
}

// ---- TTT-MLP ---------------------------------------------------------------------------------
struct MlpArgs {  // (xq, xk, xv, w1, b1, w2, b2, token_eta, lr, ln_weight, ln_bias) of a forward or backward
  Rows q;
  int64_t m;
  bool per_batch;
  void *pq, *pk, *pv, *pl;
  const float *w1, *b1, *w2, *b2, *te, *gam, *bet;
  std::array<int64_t, 4> rows, s1, s3;
  std::array<int64_t, 3> gates, s2, s4;
  std::array<int64_t, 2> hd;
  MlpArgs(PyObject* const* a, int64_t K, Keep& keep) : q(a[0]) {
    const at::Tensor& W = tensor(a[3], "w1");
    m = W.dim() > 0 ? W.size(-1) : 0;
    per_batch = W.dim() == 4;
    rows = q.shape();
    gates = {q.B, q.H, q.seq};
    hd = {q.H, q.d};
    s1 = {q.B, q.H, q.d, m};
    s2 = {q.B, q.H, m};
    s3 = {q.B, q.H, m, q.d};
    s4 = {q.B, q.H, q.d};
    pq = need(q.t, rows, q.dtype, "xq", keep);
    pk = need(a[1], rows, q.dtype, "xk", keep);
    pv = need(a[2], rows, q.dtype, "xv", keep);
    pl = need(a[8], gates, q.dtype, "ttt_lr_eta", keep);
    if (m != 4 * q.d)
      fail(TTT_ERR_UNSUPPORTED, "mlp_dim %lld != 4*head_dim (only expansion 4)", (long long)m);
    auto lead = [&](Shape s) { return per_batch ? s : s.slice(1); };
    w1 = need_f32(a[3], lead(s1), "w1", keep);
    b1 = need_f32(a[4], lead(s2), "b1", keep);
    w2 = need_f32(a[5], lead(s3), "w2", keep);
    b2 = need_f32(a[6], lead(s4), "b2", keep);
    gam = need_f32(a[9], hd, "ln_weight", keep);
    bet = need_f32(a[10], hd, "ln_bias", keep);
    te = eta_of(a[7], K, keep);
  }
};

int64_t mlp_bwd_bytes(const ttt_desc& desc) {
  const int64_t n = ttt_mlp_bwd_workspace_bytes(&desc);
  if (n < 0) fail(TTT_ERR_SHAPE, "ttt_mlp_bwd_workspace_bytes failed");
  return n;
}

// (the eleven of MlpArgs, mini_batch, eps, kernel_hint, save_for_backward)
PyObject* mlp_forward(PyObject* const* a) {
  Keep keep;
  const int64_t K = integer(a[11]);
  const MlpArgs x(a, K, keep);
  const c10::Device dev = x.q.dev;
  const ttt_desc desc = desc_of(x.q.B, x.q.H, x.q.seq, x.q.d, K, real(a[12]), 1, io_of(x.q.t), x.per_batch, 0, 0, integer(a[13]));
  check(ttt_mlp_supported(&desc));
  const bool save = PyObject_IsTrue(a[14]) == 1;
  if (save) check(ttt_mlp_fwd_saving_supported(&desc));
  at::Tensor out = empty(x.rows, x.q.dtype, dev), W1 = empty(x.s1, at::kFloat, dev), b1 = empty(x.s2, at::kFloat, dev),
             W2 = empty(x.s3, at::kFloat, dev), b2 = empty(x.s4, at::kFloat, dev), saved;
  if (save) saved = empty({(mlp_bwd_bytes(desc) + 3) / 4}, at::kFloat, dev);
  enqueue(dev, [&](void* s) {
    if (save)
      return ttt_mlp_fwd_saving(&desc, x.pq, x.pk, x.pv, x.w1, x.b1, x.w2, x.b2, x.te, x.pl, x.gam, x.bet, out.data_ptr(),
                                ptr(W1), ptr(b1), ptr(W2), ptr(b2), ptr(saved), s);
    return ttt_mlp_fwd(&desc, x.pq, x.pk, x.pv, x.w1, x.b1, x.w2, x.b2, x.te, x.pl, x.gam, x.bet, out.data_ptr(), ptr(W1),
                       ptr(b1), ptr(W2), ptr(b2), s);
  });
  return save ? wrap_tuple({&out, &W1, &b1, &W2, &b2, &saved}) : wrap_tuple({&out, &W1, &b1, &W2, &b2});
}

// (the eleven of MlpArgs, d_out, mini_batch, eps, d_state_out or None, static_scratch, into or None, kernel_hint,
//  saved or None) -> dict
PyObject* mlp_backward(PyObject* const* a) {
  static const char* const names[11] = {"d_xq", "d_xk", "d_xv", "d_W1", "d_b1", "d_W2", "d_b2", "d_lr", "d_token_eta",
                                        "d_gamma", "d_beta"};
  Keep keep;
  keep.reserve(16);
  const int64_t K = integer(a[12]);
  const MlpArgs x(a, K, keep);
  const c10::Device dev = x.q.dev;
  void* po = need(a[11], x.rows, x.q.dtype, "d_out", keep);
  const ttt_desc desc = desc_of(x.q.B, x.q.H, x.q.seq, x.q.d, K, real(a[13]), 1, io_of(x.q.t), x.per_batch, 0, 0, integer(a[17]));
  check(ttt_mlp_supported(&desc));
  const Shape states[4] = {x.s1, x.s2, x.s3, x.s4};
  const float* up[4] = {nullptr, nullptr, nullptr, nullptr};
  if (a[14] != Py_None) {
    PyObject* g = PySequence_Tuple(a[14]);
    if (g == nullptr) throw PyFailure{};
    const Py_ssize_t n = PyTuple_GET_SIZE(g);
    try {
      for (Py_ssize_t i = 0; i < 4 && i < n; ++i) {
        up[i] = need_f32(PyTuple_GET_ITEM(g, i), states[i], "d_state_out", keep);
        keep.push_back(tensor(PyTuple_GET_ITEM(g, i), "d_state_out"));
      }
    } catch (...) {
      Py_DECREF(g);
      throw;
    }
    Py_DECREF(g);
  }
  const int64_t seq1[1] = {x.q.seq};
  const Shape shapes[11] = {x.rows, x.rows, x.rows, x.s1, x.s2, x.s3, x.s4, x.gates, seq1, x.hd, x.hd};
  at::Tensor g[11];
  for (int i = 0; i < 11; ++i) {
    const at::ScalarType dt = i < 3 || i == 7 ? x.q.dtype : at::kFloat;
    if (a[16] == Py_None) {
      g[i] = empty(shapes[i], dt, dev);
      continue;
    }
    PyObject* o = PyDict_Check(a[16]) ? PyDict_GetItemString(a[16], names[i]) : nullptr;
    if (o == nullptr) {
      PyErr_SetString(PyExc_KeyError, names[i]);
      throw PyFailure{};
    }
    g[i] = tensor(o, names[i]);
    if (g[i].sizes() != shapes[i] || g[i].scalar_type() != dt || !g[i].is_contiguous() || !g[i].is_cuda())
      fail(TTT_ERR_SHAPE, "into: a gradient tensor has the wrong shape or layout");
  }
  float *saved = nullptr, *ws = nullptr;
  const bool stat = a[18] == Py_None && PyObject_IsTrue(a[15]) == 1;
  if (a[18] != Py_None) {
    const at::Tensor& t = tensor(a[18], "saved");
    if ((int64_t)t.nbytes() < mlp_bwd_bytes(desc))
      fail(TTT_ERR_SHAPE, "saved is smaller than this desc's workspace (a forward with another kernel_hint?)");
    saved = ptr(t);
  } else if (!stat) {
    keep.push_back(empty({(mlp_bwd_bytes(desc) + 3) / 4}, at::kFloat, dev));
    ws = ptr(keep.back());
  }
  enqueue(dev, [&](void* s) {
    if (stat)
      return ttt_mlp_bwd_static(&desc, x.pq, x.pk, x.pv, x.w1, x.b1, x.w2, x.b2, x.te, x.pl, x.gam, x.bet, po, up[0], up[1],
                                up[2], up[3], g[0].data_ptr(), g[1].data_ptr(), g[2].data_ptr(), ptr(g[3]), ptr(g[4]),
                                ptr(g[5]), ptr(g[6]), g[7].data_ptr(), ptr(g[8]), ptr(g[9]), ptr(g[10]), s);
    const auto call = saved != nullptr ? ttt_mlp_bwd_saved : ttt_mlp_bwd;
    return call(&desc, x.pq, x.pk, x.pv, x.w1, x.b1, x.w2, x.b2, x.te, x.pl, x.gam, x.bet, po, up[0], up[1], up[2], up[3],
                g[0].data_ptr(), g[1].data_ptr(), g[2].data_ptr(), ptr(g[3]), ptr(g[4]), ptr(g[5]), ptr(g[6]),
                g[7].data_ptr(), ptr(g[8]), ptr(g[9]), ptr(g[10]), saved != nullptr ? saved : ws, s);
  });
  PyObject* r = PyDict_New();
  if (r == nullptr) throw PyFailure{};
  for (int i = 0; i < 11; ++i) put(r, names[i], std::move(g[i]));
  return r;
}

// (xq, xk, xv, weights list, biases list, token_eta, lr, ln_weight, ln_bias, mini_batch, eps, kernel_hint)
PyObject* mlpn_forward(PyObject* const* a) {
  Keep keep;
  keep.reserve(24);
  const Rows q(a[0]);
  const int64_t B = q.B, H = q.H, seq = q.seq, d = q.d, K = integer(a[9]);
  if (!PyList_Check(a[3]) || !PyList_Check(a[4])) {
    PyErr_SetString(PyExc_TypeError, "weights and biases: lists of tensors are needed");
    throw PyFailure{};
  }
  const int layers = (int)PyList_GET_SIZE(a[3]), hidden = layers - 1;
  if (layers < 1 || layers > 8 || PyList_GET_SIZE(a[4]) != layers)
    fail(TTT_ERR_UNSUPPORTED, "weights and biases: one of each per layer, of 2, 3 or 4 hidden layers");
  const std::array<int64_t, 4> rows = q.shape();
  const std::array<int64_t, 3> gates = {B, H, seq};
  const std::array<int64_t, 2> hd = {H, d};
  void* pq = need(q.t, rows, q.dtype, "xq", keep);
  void* pk = need(a[1], rows, q.dtype, "xk", keep);
  void* pv = need(a[2], rows, q.dtype, "xv", keep);
  const bool per_batch = tensor(PyList_GET_ITEM(a[3], 0), "weights[0]").dim() == 4;
  auto dim = [&](int i) { return i == 0 || i == layers ? d : 4 * d; };
  const float *Wi[8], *bi[8];
  float *Wo[8], *bo[8];
  for (int i = 0; i < layers; ++i) {
    const std::array<int64_t, 4> W4 = {B, H, dim(i), dim(i + 1)};
    const std::array<int64_t, 3> b3 = {B, H, dim(i + 1)};
    Wi[i] = need_f32(PyList_GET_ITEM(a[3], i), per_batch ? Shape(W4) : Shape(W4).slice(1), "weights", keep);
    bi[i] = need_f32(PyList_GET_ITEM(a[4], i), per_batch ? Shape(b3) : Shape(b3).slice(1), "biases", keep);
  }
  const at::Tensor& eta = tensor(a[5], "token_eta");
  if (eta.dim() != 1 || eta.size(0) < K || eta.scalar_type() != at::kFloat)
    fail(TTT_ERR_SHAPE, "token_eta: %lld f32 entries are needed", (long long)K);
  const float* te = eta_of(a[5], K, keep);
  void* pl = need(a[6], gates, q.dtype, "ttt_lr_eta", keep);
  const float* gam = need_f32(a[7], hd, "ln_weight", keep);
  const float* bet = need_f32(a[8], hd, "ln_bias", keep);
  const ttt_desc desc = desc_of(B, H, seq, d, K, real(a[10]), 1, io_of(q.t), per_batch, 0, 0, integer(a[11]));
  check(ttt_mlpn_supported(&desc, hidden));
  at::Tensor out = empty(rows, q.dtype, q.dev), W[8], b[8];
  for (int i = 0; i < layers; ++i) {
    W[i] = empty({B, H, dim(i), dim(i + 1)}, at::kFloat, q.dev);
    b[i] = empty({B, H, dim(i + 1)}, at::kFloat, q.dev);
    Wo[i] = ptr(W[i]);
    bo[i] = ptr(b[i]);
  }
  enqueue(q.dev, [&](void* s) {
    return ttt_mlpn_fwd(&desc, hidden, pq, pk, pv, Wi, bi, te, pl, gam, bet, out.data_ptr(), Wo, bo, s);
  });
  PyObject *r = PyTuple_New(3), *lw = PyList_New(layers), *lb = PyList_New(layers);
  if (r == nullptr || lw == nullptr || lb == nullptr) throw PyFailure{};
  for (int i = 0; i < layers; ++i) {
    PyList_SET_ITEM(lw, i, THPVariable_Wrap(std::move(W[i])));
    PyList_SET_ITEM(lb, i, THPVariable_Wrap(std::move(b[i])));
  }
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(out)));
  PyTuple_SET_ITEM(r, 1, lw);
  PyTuple_SET_ITEM(r, 2, lb);
  return r;
}

// ---- a stack of layers -----------------------------------------------------------------------
// (layers: list of dicts, token_eta, mini_batch, eps, kernel_hint, workspace or None, chunk_tokens, aux stream handle,
//  check_lost: 0 or 1) -> (out, states)
PyObject* stack_forward(PyObject* const* a) {
  if (!PyList_Check(a[0]) && !PyTuple_Check(a[0])) {
    PyErr_SetString(PyExc_TypeError, "layers: a list of dicts is needed");
    throw PyFailure{};
  }
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(a[0]);
  auto at_key = [&](PyObject* L, const char* key) {
    PyObject* o = PyDict_Check(L) ? PyDict_GetItemString(L, key) : nullptr;
    if (o == nullptr) {
      PyErr_SetString(PyExc_KeyError, key);
      throw PyFailure{};
    }
    return o;
  };
  if (n == 0) {
    PyErr_SetString(PyExc_IndexError, "layers: at least one layer is needed");
    throw PyFailure{};
  }
  Keep keep;
  keep.reserve(12 * (size_t)n + 4);
  const Rows q(at_key(PySequence_Fast_GET_ITEM(a[0], 0), "pq"));
  const int64_t B = q.B, H = q.H, seq = q.seq, d = q.d, m = 4 * d, K = integer(a[2]), hint = integer(a[4]), chunk = integer(a[6]);
  const std::array<int64_t, 4> rows = q.shape();
  const std::array<int64_t, 3> gates = {B, H, seq};
  const std::array<int64_t, 2> hd = {H, d};
  const ttt_desc desc = desc_of(B, H, seq, d, K, real(a[3]), 1, io_of(q.t), false, 0, 0, hint);
  const float* te = eta_of(a[1], K, keep);
  std::vector<ttt_stack_layer> layers((size_t)n);
  std::vector<std::vector<at::Tensor>> states((size_t)n);
  bool any_mlp = false;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* L = PySequence_Fast_GET_ITEM(a[0], i);
    if (!PyDict_Check(L)) at_key(L, "pq");
    ttt_stack_layer& l = layers[(size_t)i];
    std::vector<at::Tensor>& st = states[(size_t)i];
    const bool mlp = PyDict_GetItemString(L, "W2") != nullptr;
    any_mlp |= mlp;
    l.kind = mlp ? TTT_LAYER_MLP : TTT_LAYER_LINEAR;
    l.pq = need(at_key(L, "pq"), rows, q.dtype, "pq", keep);
    l.pk = need(at_key(L, "pk"), rows, q.dtype, "pk", keep);
    l.pv = need(at_key(L, "pv"), rows, q.dtype, "pv", keep);
    l.lr = need(at_key(L, "lr"), gates, q.dtype, "lr", keep);
    l.gamma = need_f32(at_key(L, "gamma"), hd, "gamma", keep);
    l.beta = need_f32(at_key(L, "beta"), hd, "beta", keep);
    l.W2 = l.b2 = nullptr;
    l.W2_out = l.b2_out = nullptr;
    if (mlp) {
      l.W1 = need_f32(at_key(L, "W1"), {H, d, m}, "W1", keep);
      l.b1 = need_f32(at_key(L, "b1"), {H, m}, "b1", keep);
      l.W2 = need_f32(at_key(L, "W2"), {H, m, d}, "W2", keep);
      l.b2 = need_f32(at_key(L, "b2"), {H, d}, "b2", keep);
      st = {empty({B, H, d, m}, at::kFloat, q.dev), empty({B, H, m}, at::kFloat, q.dev), empty({B, H, m, d}, at::kFloat, q.dev),
            empty({B, H, d}, at::kFloat, q.dev)};
      l.W2_out = ptr(st[2]);
      l.b2_out = ptr(st[3]);
    } else {
      l.W1 = need_f32(at_key(L, "W0"), {H, d, d}, "W0", keep);
      l.b1 = need_f32(at_key(L, "b0"), {H, d}, "b0", keep);
      st = {empty({B, H, d, d}, at::kFloat, q.dev), empty({B, H, d}, at::kFloat, q.dev)};
    }
    l.W1_out = ptr(st[0]);
    l.b1_out = ptr(st[1]);
  }
  const int64_t bytes = ttt_stack_fwd_workspace_bytes(&desc, (int32_t)n, layers.data(), (int32_t)chunk);
  if (bytes < 0) fail(TTT_ERR_SHAPE, "%s", ttt_last_error());
  void* ws;
  if (a[5] == Py_None) {
    keep.push_back(empty({bytes}, at::kByte, q.dev));
    ws = keep.back().data_ptr();
  } else {
    const at::Tensor& t = tensor(a[5], "workspace");
    if ((int64_t)t.nbytes() < bytes) fail(TTT_ERR_SHAPE, "workspace too small");
    ws = t.data_ptr();
  }
  at::Tensor out = empty(rows, q.dtype, q.dev);
  void* aux = PyLong_AsVoidPtr(a[7]);
  if (aux == nullptr && PyErr_Occurred()) throw PyFailure{};
  const bool two_cu = (d == 128 || (d == 96 && (hint & TTT_HINT_TWO_CU) != 0)) && q.dtype == at::kBFloat16 && any_mlp &&
                      (hint & TTT_HINT_LDS_TILES) == 0;
  const bool guard = two_cu && integer(a[8]) != 0;
  int64_t before = 0, after = 0;
  enqueue(q.dev, [&](void* s) {
    int rc = TTT_OK;
    if (guard) {
      c10::hip::device_synchronize();
      rc = ttt_mlp_fwd_lost_workgroups(&before);
    }
    if (rc == TTT_OK) rc = ttt_stack_fwd(&desc, (int32_t)n, layers.data(), te, out.data_ptr(), ws, (int32_t)chunk, aux, s);
    if (rc == TTT_OK && guard) {
      c10::hip::device_synchronize();
      rc = ttt_mlp_fwd_lost_workgroups(&after);
    }
    return rc;
  });
  if (after != before && (hint & TTT_HINT_TEST_LOST_PARTNER) == 0)
    fail(TTT_ERR_HIP, "ttt_stack_fwd: %lld workgroups of the two-CU TTT-MLP kernel waited for their partner in vain; the "
         "outputs of their units are NaN", (long long)(after - before));
  PyObject *r = PyTuple_New(2), *ls = PyList_New(n);
  if (r == nullptr || ls == nullptr) throw PyFailure{};
  for (Py_ssize_t i = 0; i < n; ++i) {
    std::vector<at::Tensor>& st = states[(size_t)i];
    PyObject* l = PyList_New((Py_ssize_t)st.size());
    if (l == nullptr) throw PyFailure{};
    for (size_t j = 0; j < st.size(); ++j) PyList_SET_ITEM(l, (Py_ssize_t)j, THPVariable_Wrap(std::move(st[j])));
    PyList_SET_ITEM(ls, i, l);
  }
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(out)));
  PyTuple_SET_ITEM(r, 1, ls);
  return r;
}

// ---- either side of the inner loop -----------------------------------------------------------
struct Projections {  // xq, xk, xv [B,seq,H,d] and the lr gate's operands, rotary tables
  const at::Tensor& t;
  int64_t B, seq, H, d, K;
  at::ScalarType dtype;
  c10::Device dev;
  void *pq, *pk, *pv, *lg;
  const float *lb, *ti, *lti, *cos = nullptr, *sin = nullptr;
  // (xq, xk, xv, lr_logits, lr_bias, token_idx, learnable_token_idx, cos or None, sin or None, pos_offset, pos_wrap)
  Projections(PyObject* const* a, int64_t mini_batch, Keep& keep) : t(tensor(a[0], "xq")), K(mini_batch), dtype(t.scalar_type()), dev(t.device()) {
    if (t.dim() != 4) fail(TTT_ERR_SHAPE, "xq: four dimensions are needed, got %s", text(t.sizes()).c_str());
    B = t.size(0); seq = t.size(1); H = t.size(2); d = t.size(3);
    const std::array<int64_t, 4> rows = {B, seq, H, d};
    pq = need(t, rows, dtype, "xq", keep);
    pk = need(a[1], rows, dtype, "xk", keep);
    pv = need(a[2], rows, dtype, "xv", keep);
    lg = need(a[3], {B, seq, H}, dtype, "lr_logits", keep);
    const at::Tensor& bias = tensor(a[4], "lr_bias");
    if (bias.dim() != 1) keep.push_back(bias.reshape({-1}));
    lb = static_cast<float*>(need(bias.dim() != 1 ? at::Tensor(keep.back()) : bias, {H}, at::kFloat, "lr_bias", keep));
    ti = need_f32(a[5], {K}, "token_idx", keep);
    lti = need_f32(a[6], {K}, "learnable_token_idx", keep);
    if (a[7] != Py_None) {
      const at::Tensor& c = tensor(a[7], "rope cos");
      const int64_t npos = c.dim() > 0 ? c.size(0) : 0, off = integer(a[9]), wrap = integer(a[10]);
      cos = need_f32(a[7], {npos, d / 2}, "rope cos", keep);
      sin = need_f32(a[8], {npos, d / 2}, "rope sin", keep);
      const int64_t end = off + seq - 1, last = wrap == 0 || end < wrap - 1 ? end : wrap - 1;
      if (last >= npos) fail(TTT_ERR_SHAPE, "rope table shorter than the positions used");
    }
  }
};

// (the eleven of Projections, mini_batch, base_lr) -> (xq, xk, xv, lr, token_eta)
PyObject* inner_inputs(PyObject* const* a) {
  Keep keep;
  keep.reserve(16);
  const Projections p(a, integer(a[11]), keep);
  const ttt_desc desc = desc_of(p.B, p.H, p.seq, p.d, p.K, 0.f, 1, io_of(p.t), false, 0, 0, 0);
  const std::array<int64_t, 4> rows = {p.B, p.H, p.seq, p.d};
  at::Tensor q = empty(rows, p.dtype, p.dev), k = empty(rows, p.dtype, p.dev), v = empty(rows, p.dtype, p.dev),
             lr = empty({p.B, p.H, p.seq}, p.dtype, p.dev), te = empty({p.seq}, at::kFloat, p.dev);
  const int off = (int)integer(a[9]), wrp = (int)integer(a[10]);
  const float base = real(a[12]);
  enqueue(p.dev, [&](void* s) {
    return ttt_inner_inputs(&desc, p.pq, p.pk, p.pv, p.lg, p.lb, base, p.ti, p.lti, p.cos, p.sin, off, wrp, q.data_ptr(),
                            k.data_ptr(), v.data_ptr(), lr.data_ptr(), ptr(te), s);
  });
  return wrap_tuple({&q, &k, &v, &lr, &te});
}

// (the eleven of Projections, mini_batch, base_lr, weight, bias, ln_weight, ln_bias, eps, checkpoint_interval,
//  want_checkpoints, checkpoint_format, save_inputs) -> (out, W, b[, W_ckpt, b_ckpt][, xq, xk, xv, lr, token_eta])
PyObject* linear_forward_fused_inputs(PyObject* const* a) {
  Keep keep;
  keep.reserve(24);
  const Projections p(a, integer(a[11]), keep);
  const int64_t B = p.B, H = p.H, seq = p.seq, d = p.d;
  const bool per_batch = tensor(a[13], "weight").dim() == 4;
  const std::array<int64_t, 4> rows = {B, H, seq, d}, W4 = {B, H, d, d};
  const std::array<int64_t, 3> b3 = {B, H, d};
  const std::array<int64_t, 2> hd = {H, d};
  const float* W0 = need_f32(a[13], per_batch ? Shape(W4) : Shape(W4).slice(1), "weight", keep);
  const float* b0 = need_f32(a[14], per_batch ? Shape(b3) : Shape(b3).slice(1), "bias", keep);
  const float* gam = need_f32(a[15], hd, "ln_weight", keep);
  const float* bet = need_f32(a[16], hd, "ln_bias", keep);
  const ttt_desc desc = desc_of(B, H, seq, d, p.K, real(a[17]), integer(a[18]), io_of(p.t), per_batch, 0, integer(a[20]), 0);
  const int off = (int)integer(a[9]), wrp = (int)integer(a[10]);
  check(ttt_linear_fwd_fused_inputs_supported(&desc, wrp, p.cos != nullptr ? 1 : 0));
  at::Tensor out = empty(rows, p.dtype, p.dev), W = empty(W4, at::kFloat, p.dev), b = empty(b3, at::kFloat, p.dev);
  at::Tensor Wc, bc, q, k, v, lr, te;
  const bool want = PyObject_IsTrue(a[19]) == 1, save = PyObject_IsTrue(a[21]) == 1;
  if (want) {
    const int64_t n = ttt_linear_num_checkpoints(&desc);
    Wc = empty({B, H, n, d, d}, at::kFloat, p.dev);
    bc = empty({B, H, n, d}, at::kFloat, p.dev);
  }
  if (save) {
    q = empty(rows, p.dtype, p.dev);
    k = empty(rows, p.dtype, p.dev);
    v = empty(rows, p.dtype, p.dev);
    lr = empty({B, H, seq}, p.dtype, p.dev);
    te = empty({seq}, at::kFloat, p.dev);
  }
  auto opt = [](const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; };
  const float base = real(a[12]);
  enqueue(p.dev, [&](void* s) {
    return ttt_linear_fwd_fused_inputs(&desc, p.pq, p.pk, p.pv, p.lg, p.lb, base, p.ti, p.lti, p.cos, p.sin, off, wrp, W0, b0,
                                       gam, bet, out.data_ptr(), ptr(W), ptr(b), static_cast<float*>(opt(Wc)),
                                       static_cast<float*>(opt(bc)), opt(q), opt(k), opt(v), opt(lr),
                                       static_cast<float*>(opt(te)), s);
  });
  if (want && save) return wrap_tuple({&out, &W, &b, &Wc, &bc, &q, &k, &v, &lr, &te});
  if (want) return wrap_tuple({&out, &W, &b, &Wc, &bc});
  if (save) return wrap_tuple({&out, &W, &b, &q, &k, &v, &lr, &te});
  return wrap_tuple({&out, &W, &b});
}

// (inner_out, weight, bias, gate or None, eps)
PyObject* layer_epilogue(PyObject* const* a) {
  Keep keep;
  const at::Tensor& x = tensor(a[0], "inner_out");
  if (x.dim() != 4) fail(TTT_ERR_SHAPE, "inner_out: four dimensions are needed, got %s", text(x.sizes()).c_str());
  const int64_t B = x.size(0), H = x.size(1), seq = x.size(2), d = x.size(3);
  const c10::Device dev = x.device();
  void* px = need(x, {B, H, seq, d}, x.scalar_type(), "inner_out", keep);
  const float* g = need_f32(a[1], {H * d}, "post_norm_weight", keep);
  const float* b = need_f32(a[2], {H * d}, "post_norm_bias", keep);
  void* gate = a[3] == Py_None ? nullptr : need(a[3], {B, seq, H * d}, x.scalar_type(), "gate", keep);
  const float eps = real(a[4]);
  const ttt_desc desc = desc_of(B, H, seq, d, 1, eps, 1, io_of(x), false, 0, 0, 0);
  at::Tensor out = empty({B, seq, H * d}, x.scalar_type(), dev);
  enqueue(dev, [&](void* s) { return ttt_layer_epilogue(&desc, px, g, b, eps, gate, out.data_ptr(), s); });
  return wrap(std::move(out));
}

// ---- module ----------------------------------------------------------------------------------
template <PyObject* (*F)(PyObject* const*), Py_ssize_t N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != N) {
    PyErr_Format(PyExc_TypeError, "%zd arguments are needed, got %zd", N, nargs);
    return nullptr;
  }
  try {
    return F(args);
  } catch (const PyFailure&) {
  } catch (const TttFailure& e) {
    PyObject* v = g_error == nullptr ? nullptr : PyObject_CallFunction(g_error, "is", e.code, e.msg.c_str());
    if (v != nullptr) {
      PyErr_SetObject(g_error, v);
      Py_DECREF(v);
    } else if (!PyErr_Occurred()) {
      PyErr_SetString(PyExc_RuntimeError, e.msg.c_str());
    }
  } catch (...) {  // torch's own: out of memory and the like
    torch::translate_exception_to_python(std::current_exception());
  }
  return nullptr;
}

PyObject* set_error(PyObject*, PyObject* cls) {
  Py_INCREF(cls);
  Py_XSETREF(g_error, cls);
  Py_RETURN_NONE;
}

#define ENTRY(f, n) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<f, n>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    ENTRY(linear_forward, 16),
    ENTRY(linear_layer_forward, 14),
    ENTRY(linear_adam_forward, 17),
    ENTRY(linear_backward, 20),
    ENTRY(mlp_forward, 15),
    ENTRY(mlp_backward, 19),
    ENTRY(mlpn_forward, 12),
    ENTRY(stack_forward, 9),
    ENTRY(inner_inputs, 13),
    ENTRY(linear_forward_fused_inputs, 22),
    ENTRY(layer_epilogue, 5),
    {"set_error", set_error, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ttt_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ttt_torch() { return PyModule_Create(&module); }
