// The launch path of the torch-facing wrappers (w8a8/ops.py, fused.py, attention.py) in native code:
// what a call of these wrappers costs is host time, 8-16 us of attribute checks, allocations and foreign-call
// conversion around a launch of 2-3 us, more than the kernel runs for at one token or one short prompt.
//
// Every function takes the wrapper's tensors, checks the plain case (exact torch.Tensor, GPU, dtype,
// rank, contiguous rows, one device, matching shapes), allocates the outputs, calls the C ABI on
// torch's current stream of that device with the GIL released, and returns the outputs.  Anything else
// -- another type, a mismatch, an allocation that fails, a status that the C entry decides before its
// outputs are touched -- returns None, and the wrapper's own code then runs the call or raises its error:
// this path accepts nothing that the wrapper refuses.  W8A8_EHIP comes from after a launch, or clears an
// earlier call's error, so it is raised here as the wrappers raise it, and nothing is run again.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <string>

#include "w8a8.h"

namespace {

using at::ScalarType;
using at::Tensor;

// A call that this path does not take.
struct Decline {};

void need(bool ok) {
  if (!ok) throw Decline{};
}

// A C entry that failed with its work possibly queued.
struct Failed {
  std::string fn;
  int rc;
  std::string msg;
};

// The device of a call, fixed by its first tensor; every other one must be on it.
struct Call {
  int device = -1;

  const Tensor& tensor(PyObject* o, ScalarType dt, int64_t dim) {
    need(THPVariable_CheckExact(o));
    const Tensor& t = THPVariable_Unpack(o);
    need(t.is_cuda() && t.layout() == at::kStrided && t.scalar_type() == dt && t.dim() == dim);
    need(t.has_storage());  // not so inside torch.func's transforms
    if (device < 0) device = t.get_device();
    need(t.get_device() == device);
    return t;
  }
  // [M, K] with contiguous rows.
  const Tensor& rows(PyObject* o, ScalarType dt) {
    const Tensor& t = tensor(o, dt, 2);
    need(t.size(1) <= 1 || t.stride(1) == 1);
    return t;
  }
  const Tensor& vec(PyObject* o, ScalarType dt) {
    const Tensor& t = tensor(o, dt, 1);
    need(t.size(0) <= 1 || t.stride(0) == 1);
    return t;
  }
  // A bf16 weight vector of n, or none.
  const uint16_t* weight(PyObject* o, int64_t n) {
    if (o == Py_None) return nullptr;
    const Tensor& t = vec(o, at::kBFloat16);
    need(t.size(0) == n);
    return static_cast<const uint16_t*>(t.data_ptr());
  }
  Tensor make(at::IntArrayRef size, ScalarType dt) const {
    return at::empty(size, at::TensorOptions(dt).device(at::Device(at::kCUDA, static_cast<c10::DeviceIndex>(device))));
  }
  hipStream_t stream() const {
    return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(static_cast<c10::DeviceIndex>(device)).stream();
  }
};

int64_t ld(const Tensor& t) { return t.size(0) > 1 ? t.stride(0) : std::max<int64_t>(t.size(1), 1); }
const uint16_t* bf(const Tensor& t) { return static_cast<const uint16_t*>(t.data_ptr()); }
uint16_t* bfo(const Tensor& t) { return static_cast<uint16_t*>(t.data_ptr()); }
int8_t* i8(const Tensor& t) { return static_cast<int8_t*>(t.data_ptr()); }
float* f32(const Tensor& t) { return static_cast<float*>(t.data_ptr()); }

// Whole numbers and floats as the wrappers pass them: exact Python ints, floats and bools.
int64_t integer(PyObject* o) {
  need(PyLong_Check(o));
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    throw Decline{};
  }
  return v;
}
float real(PyObject* o) {
  need(PyFloat_CheckExact(o) || PyLong_CheckExact(o));
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    throw Decline{};
  }
  return static_cast<float>(v);
}

// Without the GIL for its lifetime, whichever way its block is left.
struct Released {
  PyThreadState* state = PyEval_SaveThread();
  ~Released() { PyEval_RestoreThread(state); }
};

// Runs the C entry `fn` with the GIL released.
template <class F>
void launch(const char* fn, F&& f) {
  int rc;
  {
    Released gil;
    rc = f();
  }
  if (rc == W8A8_EINVAL || rc == W8A8_EALIGN || rc == W8A8_ENOTSUP) throw Decline{};
  if (rc != W8A8_OK) throw Failed{fn, rc, w8a8_last_error()};
}

// Raises w8a8._lib.W8A8Error, as _lib.call does.
PyObject* raise_failed(const Failed& e) {
  PyObject* m = PyImport_ImportModule("w8a8._lib");
  PyObject* cls = m ? PyObject_GetAttrString(m, "W8A8Error") : nullptr;
  PyObject* err = cls ? PyObject_CallFunction(cls, "sis", e.fn.c_str(), e.rc, e.msg.c_str()) : nullptr;
  if (err) PyErr_SetObject(cls, err);
  Py_XDECREF(err);
  Py_XDECREF(cls);
  Py_XDECREF(m);
  return nullptr;
}

PyObject* none() { Py_RETURN_NONE; }
PyObject* wrap(const Tensor& t) { return THPVariable_Wrap(t); }
template <class... T>
PyObject* tuple(const T&... ts) {
  PyObject* r = PyTuple_New(sizeof...(T));
  if (!r) return nullptr;
  Py_ssize_t i = 0;
  for (const Tensor* t : {&ts...}) PyTuple_SET_ITEM(r, i++, wrap(*t));
  return r;
}

// The output: given, with these sizes, or a new one.
Tensor output(Call& c, PyObject* o, int64_t M, int64_t N, ScalarType dt) {
  if (o == Py_None) return c.make({M, N}, dt);
  const Tensor& t = c.rows(o, dt);
  need(t.size(0) == M && t.size(1) == N);
  return t;
}

// x, w.data, w.N, w.K, s, out
PyObject* gemv(PyObject* const* a) {
  Call c;
  const Tensor& x = c.rows(a[0], at::kBFloat16);
  const Tensor& w = c.tensor(a[1], at::kChar, 1);
  const int64_t N = integer(a[2]), K = integer(a[3]), M = x.size(0);
  need(x.size(1) == K && THPVariable_CheckExact(a[4]));
  const ScalarType sd = THPVariable_Unpack(a[4]).scalar_type();
  need(sd == at::kBFloat16 || sd == at::kFloat);
  const Tensor& s = c.vec(a[4], sd);
  need(s.size(0) == N);
  const Tensor y = output(c, a[5], M, N, at::kBFloat16);
  const hipStream_t st = c.stream();
  launch("w8a8_gemv_packed_bf16", [&] {
    return w8a8_gemv_packed_bf16(bf(x), ld(x), M, i8(w), N, K, s.data_ptr(), sd == at::kFloat ? 1 : 0, bfo(y), ld(y), st);
  });
  return wrap(y);
}

// x, w.data, sw, N, K, interleave, epilogue, residual, rms_w, eps, out, workspace
PyObject* linear(PyObject* const* a) {
  Call c;
  const Tensor& x = c.rows(a[0], at::kBFloat16);
  const Tensor& w = c.tensor(a[1], at::kChar, 1);
  const Tensor& sw = c.vec(a[2], at::kFloat);
  const int64_t N = integer(a[3]), K = integer(a[4]), I = integer(a[5]), epi = integer(a[6]), M = x.size(0);
  need(x.size(1) == K && sw.size(0) == N);
  const uint16_t* res = nullptr;
  int64_t ldr = 0;
  if (epi == 2 || epi == 3) {
    const Tensor& r = c.rows(a[7], at::kBFloat16);
    need(r.size(0) == M && r.size(1) == N);
    res = bf(r);
    ldr = ld(r);
  } else {
    need(a[7] == Py_None);
  }
  const uint16_t* rw = nullptr;
  if (a[8] != Py_None) {
    const Tensor& r = c.vec(a[8], at::kBFloat16);
    need(epi != 3 || r.size(0) >= N);
    rw = bf(r);
  }
  const float eps = real(a[9]);
  const Tensor y = output(c, a[10], M, epi == 1 ? I : N, at::kBFloat16);
  // the C entry checks a given workspace's size
  const Tensor ws = a[11] != Py_None ? c.vec(a[11], at::kByte)
                                     : c.make({std::max<int64_t>(w8a8_linear_workspace_bytes(M, N, K), 256)}, at::kByte);
  const hipStream_t st = c.stream();
  launch("w8a8_linear_bf16", [&] {
    return w8a8_linear_bf16(bf(x), ld(x), i8(w), f32(sw), M, N, K, int(epi), I, res, ldr, rw, eps, bfo(y), ld(y),
                            ws.data_ptr(), ws.numel(), st);
  });
  return wrap(y);
}

// The A operand: (tensor, M, K) of a PackedActivation's data, or M = -1 for row-major rows.
struct Operand {
  const int8_t* p;
  int64_t lda, M, K;
  int packed;
};
Operand operand(Call& c, PyObject* o, PyObject* m, PyObject* k) {
  const int64_t M = integer(m);
  if (M < 0) {
    const Tensor& t = c.rows(o, at::kChar);
    return {i8(t), ld(t), t.size(0), t.size(1), 0};
  }
  return {i8(c.tensor(o, at::kChar, 1)), 0, M, integer(k), 1};
}

// a, M, K, w.data, w.N, w.K, c
PyObject* gemm_i32(PyObject* const* a) {
  Call c;
  const Operand A = operand(c, a[0], a[1], a[2]);
  const Tensor& w = c.tensor(a[3], at::kChar, 1);
  const int64_t N = integer(a[4]);
  need(A.K == integer(a[5]));
  const Tensor y = output(c, a[6], A.M, N, at::kInt);
  const hipStream_t st = c.stream();
  launch("w8a8_gemm_i32_ex", [&] {
    return w8a8_gemm_i32_ex(A.p, A.lda, A.packed, i8(w), A.M, N, A.K, static_cast<int32_t*>(y.data_ptr()), ld(y), -1, 0,
                            nullptr, 0, st);
  });
  return wrap(y);
}

// a, M, K, sx, w.data, sw, w.N, w.K, interleave, epilogue, residual, out
PyObject* gemm_bf16(PyObject* const* a) {
  Call c;
  const Operand A = operand(c, a[0], a[1], a[2]);
  const Tensor& sx = c.vec(a[3], at::kFloat);
  const Tensor& w = c.tensor(a[4], at::kChar, 1);
  const Tensor& sw = c.vec(a[5], at::kFloat);
  const int64_t N = integer(a[6]), I = integer(a[8]), epi = integer(a[9]);
  need(A.K == integer(a[7]) && sx.size(0) == A.M && sw.size(0) == N && epi >= 0 && epi <= 2);
  const uint16_t* res = nullptr;
  int64_t ldr = 0;
  if (epi == 2) {
    const Tensor& r = c.rows(a[10], at::kBFloat16);
    need(r.size(0) == A.M && r.size(1) == N);
    res = bf(r);
    ldr = ld(r);
  } else {
    need(a[10] == Py_None);
  }
  const Tensor y = output(c, a[11], A.M, epi == 1 ? I : N, at::kBFloat16);
  const hipStream_t st = c.stream();
  launch("w8a8_gemm_bf16_ex", [&] {
    return w8a8_gemm_bf16_ex(A.p, A.lda, A.packed, f32(sx), i8(w), f32(sw), A.M, N, A.K, int(epi), I, res, ldr, bfo(y),
                             ld(y), -1, 0, nullptr, 0, st);
  });
  return wrap(y);
}

Tensor packed_rows(const Call& c, int64_t M, int64_t K) {
  const int64_t n = w8a8_packed_act_bytes(M, K);
  need(n >= 0);
  return c.make({std::max<int64_t>(n, 1)}, at::kChar);
}

// x -> (packed data, scales)
PyObject* quant_packed(PyObject* const* a) {
  Call c;
  const Tensor& x = c.rows(a[0], at::kBFloat16);
  const int64_t M = x.size(0), K = x.size(1);
  const Tensor q = packed_rows(c, M, K), s = c.make({M}, at::kFloat);
  const hipStream_t st = c.stream();
  launch("w8a8_quant_rows_packed_bf16", [&] { return w8a8_quant_rows_packed_bf16(bf(x), ld(x), M, K, i8(q), f32(s), st); });
  return tuple(q, s);
}

// h, w, eps -> (packed data, scales)
PyObject* k_in(PyObject* const* a) {
  Call c;
  const Tensor& h = c.rows(a[0], at::kBFloat16);
  const int64_t M = h.size(0), N = h.size(1);
  const uint16_t* w = c.weight(a[1], N);
  const float eps = real(a[2]);
  const Tensor q = packed_rows(c, M, N), s = c.make({M}, at::kFloat);
  const hipStream_t st = c.stream();
  launch("w8a8_k_in", [&] { return w8a8_k_in(bf(h), ld(h), w, eps, M, N, i8(q), 0, 1, f32(s), st); });
  return tuple(q, s);
}

// The GEMM result that a fused kernel starts from: bf16 rows, or int32 with its scales.
struct Acc {
  bool y;
  const Tensor* t;
  const float *sx = nullptr, *sw = nullptr;
  const uint16_t* rows() const { return bf(*t); }
  const int32_t* i32() const { return static_cast<const int32_t*>(t->data_ptr()); }
  int64_t stride() const { return ld(*t); }
};
Acc acc_in(Call& c, PyObject* acc, PyObject* sx, PyObject* sw, int64_t ncols) {
  need(THPVariable_CheckExact(acc));
  Acc r;
  r.y = THPVariable_Unpack(acc).scalar_type() == at::kBFloat16;
  r.t = &c.rows(acc, r.y ? at::kBFloat16 : at::kInt);
  need(r.t->size(1) >= ncols);
  if (!r.y) {
    const Tensor &x = c.vec(sx, at::kFloat), &w = c.vec(sw, at::kFloat);
    need(x.size(0) == r.t->size(0) && w.size(0) >= ncols);
    r.sx = f32(x);
    r.sw = f32(w);
  }
  return r;
}

// acc, sx, sw, res, w_post, w_pre_ff, eps -> (h, packed data, scales)
PyObject* k_post_attn(PyObject* const* a) {
  Call c;
  const Tensor& res = c.rows(a[3], at::kBFloat16);
  const int64_t M = res.size(0), N = res.size(1);
  const Acc acc = acc_in(c, a[0], a[1], a[2], N);
  need(acc.t->size(0) == M);
  const uint16_t *w1 = c.weight(a[4], N), *w2 = c.weight(a[5], N);
  const float eps = real(a[6]);
  const Tensor h = c.make({M, N}, at::kBFloat16), q = packed_rows(c, M, N), s = c.make({M}, at::kFloat);
  const hipStream_t st = c.stream();
  launch(acc.y ? "w8a8_k_post_attn_y" : "w8a8_k_post_attn", [&] {
    return acc.y ? w8a8_k_post_attn_y(acc.rows(), acc.stride(), bf(res), ld(res), w1, w2, eps, M, N, bfo(h), N, i8(q), 0, 1,
                                      f32(s), st)
                 : w8a8_k_post_attn(acc.i32(), acc.stride(), acc.sx, acc.sw, bf(res), ld(res), w1, w2, eps, M, N, bfo(h), N,
                                    i8(q), 0, 1, f32(s), st);
  });
  return tuple(h, q, s);
}

// acc, sx, sw, res, w_post_ff, eps -> (h, packed data, scales)
PyObject* k_post_ff(PyObject* const* a) {
  Call c;
  const Tensor& res = c.rows(a[3], at::kBFloat16);
  const int64_t M = res.size(0), N = res.size(1);
  const Acc acc = acc_in(c, a[0], a[1], a[2], N);
  need(acc.t->size(0) == M);
  const uint16_t* w = c.weight(a[4], N);
  const float eps = real(a[5]);
  const Tensor h = c.make({M, N}, at::kBFloat16), q = packed_rows(c, M, N), s = c.make({M}, at::kFloat);
  const hipStream_t st = c.stream();
  launch(acc.y ? "w8a8_k_post_ff_y" : "w8a8_k_post_ff", [&] {
    return acc.y ? w8a8_k_post_ff_y(acc.rows(), acc.stride(), bf(res), ld(res), w, eps, M, N, bfo(h), N, i8(q), 0, 1, f32(s),
                                    st)
                 : w8a8_k_post_ff(acc.i32(), acc.stride(), acc.sx, acc.sw, bf(res), ld(res), w, eps, M, N, bfo(h), N, i8(q),
                                  0, 1, f32(s), st);
  });
  return tuple(h, q, s);
}

// acc, sx, sw, ple -> (packed data, scales)
PyObject* k_ple_gate(PyObject* const* a) {
  Call c;
  const Tensor& ple = c.rows(a[3], at::kBFloat16);
  const int64_t M = ple.size(0), N = ple.size(1);
  const Acc acc = acc_in(c, a[0], a[1], a[2], N);
  need(acc.t->size(0) == M);
  const Tensor q = packed_rows(c, M, N), s = c.make({M}, at::kFloat);
  const hipStream_t st = c.stream();
  launch(acc.y ? "w8a8_k_ple_gate_y" : "w8a8_k_ple_gate", [&] {
    return acc.y ? w8a8_k_ple_gate_y(acc.rows(), acc.stride(), bf(ple), ld(ple), M, N, i8(q), 0, 1, f32(s), st)
                 : w8a8_k_ple_gate(acc.i32(), acc.stride(), acc.sx, acc.sw, bf(ple), ld(ple), M, N, i8(q), 0, 1, f32(s), st);
  });
  return tuple(q, s);
}

// acc, sx, sw, h, w_post_ple, scalar, eps, norm_next -> (out, packed data, scales)
PyObject* k_ple_out_k_in(PyObject* const* a) {
  Call c;
  const Tensor& h = c.rows(a[3], at::kBFloat16);
  const int64_t M = h.size(0), N = h.size(1);
  const Acc acc = acc_in(c, a[0], a[1], a[2], N);
  need(acc.t->size(0) == M);
  const uint16_t *w = c.weight(a[4], N), *wn = c.weight(a[7], N);
  const Tensor& sc = c.vec(a[5], at::kBFloat16);
  need(sc.size(0) == 1 && wn);
  const float eps = real(a[6]);
  const Tensor o = c.make({M, N}, at::kBFloat16), q = packed_rows(c, M, N), s = c.make({M}, at::kFloat);
  const hipStream_t st = c.stream();
  launch(acc.y ? "w8a8_k_ple_out_k_in_y" : "w8a8_k_ple_out_k_in", [&] {
    return acc.y ? w8a8_k_ple_out_k_in_y(acc.rows(), acc.stride(), bf(h), ld(h), w, bf(sc), wn, eps, M, N, bfo(o), N, i8(q), 0,
                                         1, f32(s), st)
                 : w8a8_k_ple_out_k_in(acc.i32(), acc.stride(), acc.sx, acc.sw, bf(h), ld(h), w, bf(sc), wn, eps, M, N,
                                       bfo(o), N, i8(q), 0, 1, f32(s), st);
  });
  return tuple(o, q, s);
}

// acc, sx, sw, cos, sin, qw, kw, eps, H, KV, D, shared -> (q, k, v), or (q,) when shared
PyObject* k_qkv(PyObject* const* a) {
  Call c;
  const int64_t H = integer(a[8]), KV = integer(a[9]), D = integer(a[10]);
  const bool shared = PyObject_IsTrue(a[11]) == 1;
  const Acc acc = acc_in(c, a[0], a[1], a[2], (shared ? H : H + 2 * KV) * D);
  const int64_t T = acc.t->size(0);
  const Tensor &cs = c.rows(a[3], at::kBFloat16), &sn = c.rows(a[4], at::kBFloat16);
  need(cs.size(0) == T && cs.size(1) == D && sn.size(0) == T && sn.size(1) == D && cs.stride(0) == sn.stride(0));
  const uint16_t *qw = c.weight(a[5], D), *kw = shared ? nullptr : c.weight(a[6], D);
  const float eps = real(a[7]);
  const Tensor q = c.make({H, T, D}, at::kBFloat16);
  Tensor k, v;
  if (!shared) {
    k = c.make({KV, T, D}, at::kBFloat16);
    v = c.make({KV, T, D}, at::kBFloat16);
  }
  uint16_t *kp = shared ? nullptr : bfo(k), *vp = shared ? nullptr : bfo(v);
  const hipStream_t st = c.stream();
  launch(acc.y ? "w8a8_k_qkv_y" : "w8a8_k_qkv", [&] {
    return acc.y ? w8a8_k_qkv_y(acc.rows(), acc.stride(), bf(cs), bf(sn), ld(cs), qw, kw, eps, T, H, KV, D, shared ? 1 : 0,
                                bfo(q), kp, vp, st)
                 : w8a8_k_qkv(acc.i32(), acc.stride(), acc.sx, acc.sw, bf(cs), bf(sn), ld(cs), qw, kw, eps, T, H, KV, D,
                              shared ? 1 : 0, bfo(q), kp, vp, st);
  });
  return shared ? tuple(q) : tuple(q, k, v);
}

// [heads, rows, head_dim] with a contiguous last dimension, and its strides (sizes of 1 take the natural one).
struct Heads {
  const Tensor* t;
  int64_t hs, rs;
};
Heads heads(Call& c, PyObject* o) {
  const Tensor& t = c.tensor(o, at::kBFloat16, 3);
  need(t.size(2) <= 1 || t.stride(2) == 1);
  const int64_t rs = t.size(1) > 1 ? t.stride(1) : t.size(2);
  return {&t, t.size(0) > 1 ? t.stride(0) : std::max<int64_t>(t.size(1), 1) * rs, rs};
}

// The stream's cached workspace of at least n bytes, from the wrapper's dict {(device, stream): uint8 tensor}.
// Missing or too small: declined, and the wrapper grows it.
const Tensor* cached(const Call& c, PyObject* dict, hipStream_t st, int64_t n) {
  if (n == 0) return nullptr;
  need(n > 0 && PyDict_CheckExact(dict));
  PyObject* key = Py_BuildValue("(iK)", c.device, static_cast<unsigned long long>(reinterpret_cast<uintptr_t>(st)));
  need(key);
  PyObject* o = PyDict_GetItemWithError(dict, key);
  Py_DECREF(key);
  if (!o) PyErr_Clear();
  need(o && THPVariable_CheckExact(o));
  const Tensor& t = THPVariable_Unpack(o);
  need(t.is_cuda() && t.get_device() == c.device && t.scalar_type() == at::kByte && t.dim() == 1 && t.numel() >= n);
  return &t;
}

// q, k, v, q_start, window, scale, workspaces -> o
PyObject* attention(PyObject* const* a) {
  Call c;
  const Heads q = heads(c, a[0]), k = heads(c, a[1]), v = heads(c, a[2]);
  const int64_t H = q.t->size(0), Tq = q.t->size(1), D = q.t->size(2), KV = k.t->size(0), Tk = k.t->size(1);
  need(k.t->size(2) == D && v.t->sizes() == k.t->sizes());
  const int64_t start = integer(a[3]), window = integer(a[4]);
  const float scale = real(a[5]);
  const Tensor o = c.make({H, Tq, D}, at::kBFloat16);
  const hipStream_t st = c.stream();
  const Tensor* w = cached(c, a[6], st, w8a8_attention_workspace_bytes(H, KV, Tq, Tk, D, start, window));
  const Tensor ws = w ? *w : Tensor();  // held while the GIL is released
  launch("w8a8_attention_ws_bf16", [&] {
    return w8a8_attention_ws_bf16(bf(*q.t), q.hs, q.rs, bf(*k.t), k.hs, k.rs, bf(*v.t), v.hs, v.rs, H, KV, Tq, Tk, D, start,
                                  window, scale, bfo(o), std::max<int64_t>(Tq, 1) * D, D, nullptr,
                                  w ? ws.data_ptr() : nullptr, w ? ws.numel() : 0, st);
  });
  return wrap(o);
}

// q, k, v, q_start, window, scale, workspaces -> (packed data, scales)
PyObject* attention_quant(PyObject* const* a) {
  Call c;
  const Heads q = heads(c, a[0]), k = heads(c, a[1]), v = heads(c, a[2]);
  const int64_t H = q.t->size(0), Tq = q.t->size(1), D = q.t->size(2), KV = k.t->size(0), Tk = k.t->size(1);
  need(k.t->size(2) == D && v.t->sizes() == k.t->sizes());
  const int64_t start = integer(a[3]), window = integer(a[4]);
  const float scale = real(a[5]);
  need(Tq > 0 && w8a8_attention_quant_supported(H, KV, Tq, Tk, D, start, window) == 1);
  const Tensor x = packed_rows(c, Tq, H * D), s = c.make({Tq}, at::kFloat);
  const hipStream_t st = c.stream();
  const Tensor* w = cached(c, a[6], st, w8a8_attention_workspace_bytes(H, KV, Tq, Tk, D, start, window));
  const Tensor ws = w ? *w : Tensor();
  launch("w8a8_attention_quant_bf16", [&] {
    return w8a8_attention_quant_bf16(bf(*q.t), q.hs, q.rs, bf(*k.t), k.hs, k.rs, bf(*v.t), v.hs, v.rs, H, KV, Tq, Tk, D,
                                     start, window, scale, i8(x), f32(s), w ? ws.data_ptr() : nullptr, w ? ws.numel() : 0,
                                     st);
  });
  return tuple(x, s);
}

// q [H, D], k, v, q_pos, window, scale, workspaces -> o [H, D]
PyObject* decode(PyObject* const* a) {
  Call c;
  const Tensor& q = c.rows(a[0], at::kBFloat16);
  const Heads k = heads(c, a[1]), v = heads(c, a[2]);
  const int64_t H = q.size(0), D = q.size(1), KV = k.t->size(0), Tk = k.t->size(1);
  need(k.t->size(2) == D && v.t->sizes() == k.t->sizes());
  const int64_t pos = a[3] == Py_None ? Tk - 1 : integer(a[3]), window = integer(a[4]);
  const float scale = real(a[5]);
  const Tensor o = c.make({H, D}, at::kBFloat16);
  const hipStream_t st = c.stream();
  const int64_t bytes = w8a8_attention_decode_workspace_bytes(H, KV, Tk, D, pos, window);
  need(bytes > 0);
  const Tensor ws = *cached(c, a[6], st, bytes);
  launch("w8a8_attention_decode_bf16", [&] {
    return w8a8_attention_decode_bf16(bf(q), H > 1 ? q.stride(0) : D, bf(*k.t), k.hs, k.rs, bf(*v.t), v.hs, v.rs, H, KV, Tk,
                                      D, pos, window, scale, bfo(o), D, nullptr, ws.data_ptr(), ws.numel(), st);
  });
  return wrap(o);
}

// Waits for torch's current stream of tensor t's device; True when it is done, None without waiting if t is
// no GPU tensor.
PyObject* wait_stream(PyObject* const* a) {
  need(THPVariable_CheckExact(a[0]));
  const Tensor& t = THPVariable_Unpack(a[0]);
  need(t.is_cuda());
  Call c;
  c.device = t.get_device();
  const hipStream_t st = c.stream();
  hipError_t e;
  {
    Released gil;
    e = hipStreamSynchronize(st);
  }
  if (e != hipSuccess) throw Failed{"hipStreamSynchronize", W8A8_EHIP, hipGetErrorString(e)};
  Py_RETURN_TRUE;
}

// (C entry's name, status) -> what a call whose entry returned it comes to: True, None (declined) or the
// error raised.  A negative status throws in the entry's place.
PyObject* settle(PyObject* const* a) {
  const char* fn = PyUnicode_AsUTF8(a[0]);
  need(fn);
  const int rc = static_cast<int>(integer(a[1]));
  launch(fn, [&] {
    if (rc < 0) throw std::string("thrown");
    return rc;
  });
  Py_RETURN_TRUE;
}

// A METH_FASTCALL entry of `n` arguments around `f`: every refusal and every C++ exception is None, a
// failed launch is raised.
template <PyObject* (*f)(PyObject* const*), int n>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != n) return none();
  try {
    return f(args);
  } catch (const Failed& e) {
    return raise_failed(e);
  } catch (...) {  // Decline, or torch's: no storage, out of memory, a Python mode's error, ...
    PyErr_Clear();
    return none();
  }
}

#define W8A8_ENTRY(name, n) \
  {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<name, n>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    W8A8_ENTRY(gemv, 6),        W8A8_ENTRY(linear, 12),         W8A8_ENTRY(gemm_i32, 7),  W8A8_ENTRY(gemm_bf16, 12),
    W8A8_ENTRY(quant_packed, 1), W8A8_ENTRY(k_in, 3),           W8A8_ENTRY(k_post_attn, 7), W8A8_ENTRY(k_post_ff, 6),
    W8A8_ENTRY(k_ple_gate, 4),  W8A8_ENTRY(k_ple_out_k_in, 8),  W8A8_ENTRY(k_qkv, 12),    W8A8_ENTRY(attention, 7),
    W8A8_ENTRY(attention_quant, 7), W8A8_ENTRY(decode, 7),      W8A8_ENTRY(wait_stream, 1),
    W8A8_ENTRY(settle, 2),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launch", "The wrappers' launch path in native code.", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

// What the module fits, compared by _lib.launch_module before anything here is called.
PyMODINIT_FUNC PyInit__launch() {
  PyObject* m = PyModule_Create(&module);
  if (m && (PyModule_AddStringConstant(m, "torch_build", W8A8_TORCH) < 0 ||
            PyModule_AddStringConstant(m, "sources", W8A8_SOURCES) < 0)) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
