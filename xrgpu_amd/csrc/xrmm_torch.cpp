// Native front end of the zero-copy entry points: the argument checks, output
// allocations and calls of xrgpu_amd/ops.py for ordinary arguments. In Python they
// cost more than a decode kernel runs (Qkv at four rows: 16.8 us a call for an 8 us
// kernel; 27 ctypes arguments, four allocations, ten tensors' properties).
//
// Every function returns None, having done nothing, for whatever it does not take: a
// tensor that is not a plain torch.Tensor on one GPU (subclasses, wrappers, CPU), any
// mode that intercepts calls, a dtype, shape or layout that does not match, an empty
// batch. ops.py then runs its own checks, which raise or accept as they always did.
// Nothing is kept between calls. Measured, among other passes: Qkv 4 x 4096 x (4096 + 2 x
// 1024) 17.8 -> 7.6 us a call, MatMulNBits 1 x 4096 x 14336 8.4 -> 6.9.
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/version.h>

#include <cstdint>
#include <initializer_list>

namespace {

constexpr int F32 = 0, F16 = 1, U8 = 6, UNSPECIFIED = 9;  // xrmm_dtype

using MatmulFn = int (*)(const void*, const void*, const void*, const void*, int32_t, const void*, void*, int64_t, int64_t,
                         int64_t, int32_t, int32_t, int32_t, void*);
using MatmulWsFn = int64_t (*)(int64_t, int64_t, int64_t, int32_t, int32_t, int32_t);
using FusedWsFn = int64_t (*)(int32_t, int64_t, int64_t, int64_t, int64_t, int32_t, int32_t, int32_t, int32_t, int32_t);
using QkvFn = int (*)(const void*, const void*, const void*, const void*, const void*, const void*, const void*, const void*,
                      const void*, const void*, const void*, const void*, int32_t, void*, void*, void*, void*, int64_t,
                      int64_t, int64_t, int64_t, int32_t, int32_t, float, int32_t, void*, int64_t, void*);
using MlpFn = int (*)(const void*, const void*, const void*, const void*, const void*, const void*, const void*, const void*,
                      const void*, const void*, const void*, int32_t, void*, void*, int64_t, int64_t, int64_t, int32_t,
                      int32_t, float, int32_t, int32_t, void*, int64_t, void*);
using BnbFn = int (*)(const void*, const void*, const void*, void*, int64_t, int64_t, int64_t, int32_t, int32_t, int32_t,
                      int32_t, void*);
using GatherFn = int (*)(const void*, const void*, int32_t, const void*, const void*, void*, void*, int64_t, int64_t,
                         int64_t, int32_t, int32_t, void*);

// the library's entry points, the current stream's raw handle and the error check, from ops.py
MatmulFn g_matmul;
MatmulWsFn g_matmul_ws;
FusedWsFn g_fused_ws;
QkvFn g_qkv;
MlpFn g_mlp;
BnbFn g_bnb;
GatherFn g_gather;
PyObject *g_stream, *g_check;

struct Decline {};  // ops.py takes the call

// a plain tensor on one GPU, contiguous; `dev` is the call's device (-1: not known yet)
const at::Tensor& plain(PyObject* o, int& dev) {
  if (!THPVariable_CheckExact(o)) throw Decline{};
  const at::Tensor& t = THPVariable_Unpack(o);
  const auto ks = t.key_set();
  if (!t.is_cuda() || t.layout() != at::kStrided || ks.has(c10::DispatchKey::Python) ||
      ks.has_any(c10::functorch_transforms_ks) || t.is_conj() || t.is_neg() || !t.is_contiguous() || t.numel() == 0)
    throw Decline{};
  const int d = t.get_device();
  if (dev < 0) dev = d;
  if (d != dev) throw Decline{};
  return t;
}

bool none(PyObject* o) { return o == Py_None; }

int64_t integer(PyObject* o) {
  if (!PyLong_CheckExact(o)) throw Decline{};
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    throw Decline{};
  }
  return v;
}

double real(PyObject* o) {
  if (!PyFloat_CheckExact(o)) throw Decline{};
  return PyFloat_AS_DOUBLE(o);
}

void want(bool ok) {
  if (!ok) throw Decline{};
}

bool shape(const at::Tensor& t, std::initializer_list<int64_t> s) { return t.sizes() == at::IntArrayRef(s.begin(), s.size()); }

int t1(const at::Tensor& a) {
  if (a.scalar_type() == at::kHalf) return F16;
  want(a.scalar_type() == at::kFloat);
  return F32;
}

void* stream_of(int dev) {
  PyObject* i = PyLong_FromLong(dev);
  PyObject* r = i ? PyObject_CallOneArg(g_stream, i) : nullptr;
  Py_XDECREF(i);
  if (!r) {
    PyErr_Clear();
    throw Decline{};
  }
  void* s = PyLong_AsVoidPtr(r);
  Py_DECREF(r);
  if (s == nullptr && PyErr_Occurred()) {
    PyErr_Clear();
    throw Decline{};
  }
  return s;
}

// rows, K and the leading axes of the activations
struct Act {
  const at::Tensor& A;
  int64_t K, M;
  int dt;
  at::DimVector lead;
  Act(const at::Tensor& a, PyObject* k) : A(a), K(0), M(0), dt(t1(a)) {
    want(a.dim() >= 1);
    K = a.size(-1);
    want(none(k) || integer(k) == K);
    M = a.numel() / K;
    lead = at::DimVector(a.sizes().slice(0, a.dim() - 1));
  }
  at::Tensor out(int64_t n) const {
    at::DimVector s = lead;
    s.push_back(n);
    return at::empty(s, A.options());
  }
};

struct Quant {
  int bits, bs;
  int64_t kb, blob, zrow;
  Quant(PyObject* b, PyObject* s, int64_t K) {
    const int64_t bb = integer(b), ss = integer(s);
    want((bb == 2 || bb == 4 || bb == 8) && ss > 0 && ss <= (1 << 20));
    bits = static_cast<int>(bb);
    bs = static_cast<int>(ss);
    kb = (K + bs - 1) / bs;
    blob = (static_cast<int64_t>(bs) * bits + 7) / 8;
    zrow = (kb * bits + 7) / 8;
  }
};

struct Weights {
  const void *B, *S, *Z;
  int zdt;
  int64_t N;
};

Weights weights(PyObject* b, PyObject* s, PyObject* z, PyObject* n, const Act& a, const Quant& q, int& dev) {
  const at::Tensor &B = plain(b, dev), &S = plain(s, dev);
  want(B.scalar_type() == at::kByte && B.dim() == 3);
  const int64_t N = B.size(0);
  want((none(n) || integer(n) == N) && shape(B, {N, q.kb, q.blob}) && S.scalar_type() == a.A.scalar_type() && shape(S, {N, q.kb}));
  Weights w{B.data_ptr(), S.data_ptr(), nullptr, UNSPECIFIED, N};
  if (!none(z)) {
    const at::Tensor& Z = plain(z, dev);
    const bool packed = Z.scalar_type() == at::kByte;
    w.zdt = packed ? U8 : t1(Z);
    want(shape(Z, {N, packed ? q.zrow : q.kb}));
    w.Z = Z.data_ptr();
  }
  return w;
}

// an optional tensor of A's dtype with n elements (vec: one-dimensional)
const void* aux(PyObject* o, const Act& a, int64_t n, bool vec, int& dev) {
  if (none(o)) return nullptr;
  const at::Tensor& t = plain(o, dev);
  want(t.scalar_type() == a.A.scalar_type() && t.numel() == n && (!vec || t.dim() == 1));
  return t.data_ptr();
}

// the projections' common zero-point dtype
int one_zdt(std::initializer_list<const Weights*> ws) {
  int dt = UNSPECIFIED;
  for (const Weights* w : ws)
    if (w->Z) {
      want(dt == UNSPECIFIED || dt == w->zdt);
      dt = w->zdt;
    }
  return dt;
}

bool checked(int rc) {  // false: the Python error is set
  if (rc == 0) return true;
  PyObject* i = PyLong_FromLong(rc);
  PyObject* r = i ? PyObject_CallOneArg(g_check, i) : nullptr;
  Py_XDECREF(i);
  Py_XDECREF(r);
  return r != nullptr;
}

// Other Python threads run while a call allocates and launches.
struct NoGil {
  PyThreadState* state = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(state); }
};

PyObject* optional(const at::Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}

template <typename F>
PyObject* guarded(Py_ssize_t n, Py_ssize_t expected, F&& f) {
  if (n != expected || c10::impl::dispatch_mode_enabled() || at::impl::torch_function_mode_enabled()) Py_RETURN_NONE;
  try {
    return f();
  } catch (const Decline&) {
    Py_RETURN_NONE;
  } catch (const std::exception& e) {  // an allocation that failed, say: ops.py meets it again
    Py_RETURN_NONE;
  }
}

// (A, B, scales, zero_points, bias, K, N, bits, block_size)
PyObject* matmul(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 9, [&]() -> PyObject* {
    int dev = -1;
    const Act a(plain(v[0], dev), v[5]);
    const Quant q(v[7], v[8], a.K);
    const Weights w = weights(v[1], v[2], v[3], v[6], a, q, dev);
    const void* bias = aux(v[4], a, w.N, true, dev);
    // calls on a workspace stay with ops.py, which keeps one per stream
    if (a.M > 4 && g_matmul_ws(a.M, a.K, w.N, q.bits, q.bs, a.dt) > 0) throw Decline{};
    void* st = stream_of(dev);
    at::Tensor y;
    int rc;
    {
      NoGil ng;
      y = a.out(w.N);
      rc = g_matmul(a.A.data_ptr(), w.B, w.S, w.Z, w.zdt, bias, y.data_ptr(), a.M, a.K, w.N, q.bits, q.bs, a.dt, st);
    }
    if (!checked(rc)) return nullptr;
    return THPVariable_Wrap(y);
  });
}

at::Tensor scratch(int op, const Act& a, int64_t N, int64_t Nkv, const Quant& q, bool skip, bool norm, int64_t& bytes) {
  bytes = g_fused_ws(op, a.M, a.K, N, Nkv, q.bits, q.bs, a.dt, skip, norm);
  if (bytes <= 0) {
    bytes = 0;
    return {};
  }
  return at::empty({bytes}, a.A.options().dtype(at::kByte));
}

// (A, q_B, q_scales, k_B, k_scales, v_B, v_scales, norm_scale, skip, K, Nq, Nkv, bits,
//  block_size, epsilon, q_zero_points, k_zero_points, v_zero_points, want_residual)
PyObject* qkv(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 19, [&]() -> PyObject* {
    int dev = -1;
    const Act a(plain(v[0], dev), v[9]);
    const Quant q(v[12], v[13], a.K);
    const Weights wq = weights(v[1], v[2], v[15], v[10], a, q, dev);
    const Weights wk = weights(v[3], v[4], v[16], v[11], a, q, dev);
    const Weights wv = weights(v[5], v[6], v[17], v[11], a, q, dev);
    want(wk.N == wv.N && !none(v[7]));
    const int zdt = one_zdt({&wq, &wk, &wv});
    const void* gamma = aux(v[7], a, a.K, true, dev);
    const void* skip = aux(v[8], a, a.M * a.K, false, dev);
    const float eps = static_cast<float>(real(v[14]));
    want(PyBool_Check(v[18]));
    void* st = stream_of(dev);
    const bool residual = v[18] == Py_True;
    at::Tensor Q, Ko, V, R;
    int rc;
    {
      NoGil ng;
      Q = a.out(wq.N), Ko = a.out(wk.N), V = a.out(wv.N);
      if (residual) R = a.out(a.K);
      int64_t nws = 0;
      const at::Tensor ws = scratch(1, a, wq.N, wk.N, q, skip != nullptr, true, nws);
      rc = g_qkv(a.A.data_ptr(), skip, gamma, wq.B, wq.S, wq.Z, wk.B, wk.S, wk.Z, wv.B, wv.S, wv.Z, zdt, Q.data_ptr(),
                 Ko.data_ptr(), V.data_ptr(), residual ? R.data_ptr() : nullptr, a.M, a.K, wq.N, wk.N, q.bits, q.bs, eps, a.dt,
                 nws ? ws.data_ptr() : nullptr, nws, st);
    }
    if (!checked(rc)) return nullptr;
    PyObject *o0 = THPVariable_Wrap(Q), *o1 = THPVariable_Wrap(Ko), *o2 = THPVariable_Wrap(V), *o3 = optional(R);
    return Py_BuildValue("(NNNN)", o0, o1, o2, o3);
  });
}

// (A, gate_B, gate_scales, up_B, up_scales, skip, norm_scale, gate_bias, up_bias, K, N, bits,
//  block_size, epsilon, activation code, gate_zero_points, up_zero_points, want_residual)
PyObject* mlp(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 18, [&]() -> PyObject* {
    int dev = -1;
    const Act a(plain(v[0], dev), v[9]);
    const Quant q(v[11], v[12], a.K);
    const Weights g = weights(v[1], v[2], v[15], v[10], a, q, dev), u = weights(v[3], v[4], v[16], v[10], a, q, dev);
    want(g.N == u.N);
    const int zdt = one_zdt({&g, &u});
    const void* skip = aux(v[5], a, a.M * a.K, false, dev);
    const void* gamma = aux(v[6], a, a.K, true, dev);
    const void *gb = aux(v[7], a, g.N, true, dev), *ub = aux(v[8], a, g.N, true, dev);
    const float eps = static_cast<float>(real(v[13]));
    const int act = static_cast<int>(integer(v[14]));
    want(PyBool_Check(v[17]));
    void* st = stream_of(dev);
    const bool residual = v[17] == Py_True;
    at::Tensor Y, R;
    int rc;
    {
      NoGil ng;
      Y = a.out(g.N);
      if (residual) R = a.out(a.K);
      int64_t nws = 0;
      const at::Tensor ws = scratch(2, a, g.N, 0, q, skip != nullptr, gamma != nullptr, nws);
      rc = g_mlp(a.A.data_ptr(), skip, gamma, g.B, g.S, g.Z, gb, u.B, u.S, u.Z, ub, zdt, Y.data_ptr(),
                 residual ? R.data_ptr() : nullptr, a.M, a.K, g.N, q.bits, q.bs, eps, act, a.dt,
                 nws ? ws.data_ptr() : nullptr, nws, st);
    }
    if (!checked(rc)) return nullptr;
    PyObject *o0 = THPVariable_Wrap(Y), *o1 = optional(R);
    return Py_BuildValue("(NN)", o0, o1);
  });
}

// (A, B, absmax, K, N, block_size, quant_type, trans_b)
PyObject* bnb4(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 8, [&]() -> PyObject* {
    int dev = -1;
    const Act a(plain(v[0], dev), v[3]);
    const at::Tensor &B = plain(v[1], dev), &S = plain(v[2], dev);
    const int64_t N = integer(v[4]), bs = integer(v[5]), qt = integer(v[6]), tb = integer(v[7]);
    want(a.A.dim() == 2 && N > 0 && N < (int64_t(1) << 31) && a.K < (int64_t(1) << 31) && bs > 0 && bs <= (1 << 20) && B.scalar_type() == at::kByte &&
         S.scalar_type() == a.A.scalar_type() && B.numel() >= (N * a.K + 1) / 2 && S.numel() >= (N * a.K + bs - 1) / bs &&
         (qt == 0 || qt == 1) && (tb == 0 || tb == 1));
    void* st = stream_of(dev);
    at::Tensor y;
    int rc;
    {
      NoGil ng;
      y = a.out(N);
      rc = g_bnb(a.A.data_ptr(), B.data_ptr(), S.data_ptr(), y.data_ptr(), a.M, a.K, N, static_cast<int32_t>(bs),
                 static_cast<int32_t>(qt), static_cast<int32_t>(tb), a.dt, st);
    }
    if (!checked(rc)) return nullptr;
    return THPVariable_Wrap(y);
  });
}

// (data, indices, scales, zero_points, status, bits, block_size)
PyObject* gather(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 7, [&]() -> PyObject* {
    int dev = -1;
    const at::Tensor &D = plain(v[0], dev), &I = plain(v[1], dev), &S = plain(v[2], dev), &st_t = plain(v[4], dev);
    const int64_t bits = integer(v[5]), bs = integer(v[6]);
    want((bits == 4 || bits == 8) && bs > 0 && bs <= (1 << 20) && D.scalar_type() == at::kByte && D.dim() == 2 && I.dim() == 1 &&
         S.scalar_type() == at::kFloat && st_t.scalar_type() == at::kInt);
    const bool i64 = I.scalar_type() == at::kLong;
    want(i64 || I.scalar_type() == at::kInt);
    const int64_t rows = D.size(0), pcols = D.size(1), width = pcols * (8 / bits), blocks = (width + bs - 1) / bs;
    want(shape(S, {rows, blocks}));
    const void* z = nullptr;
    if (!none(v[3])) {
      const at::Tensor& Z = plain(v[3], dev);
      want(Z.scalar_type() == at::kByte && shape(Z, {rows, (blocks * bits + 7) / 8}));
      z = Z.data_ptr();
    }
    void* st = stream_of(dev);
    at::Tensor y;
    int rc;
    {
      NoGil ng;
      y = at::empty({I.size(0), width}, S.options());
      rc = g_gather(D.data_ptr(), I.data_ptr(), i64 ? 7 : 2, S.data_ptr(), z, y.data_ptr(), st_t.data_ptr(), rows, pcols,
                    I.size(0), static_cast<int32_t>(bits), static_cast<int32_t>(bs), st);
    }
    if (!checked(rc)) return nullptr;
    return THPVariable_Wrap(y);
  });
}

// (raw stream function, check function, addresses of the seven entry points)
PyObject* bind(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (n != 9) {
    PyErr_SetString(PyExc_TypeError, "bind takes nine arguments");
    return nullptr;
  }
  void* f[7];
  for (int i = 0; i < 7; ++i) {
    f[i] = PyLong_AsVoidPtr(v[2 + i]);
    if (f[i] == nullptr) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point");
      return nullptr;
    }
  }
  Py_INCREF(v[0]);
  Py_INCREF(v[1]);
  Py_XDECREF(g_stream);
  Py_XDECREF(g_check);
  g_stream = v[0];
  g_check = v[1];
  g_matmul = reinterpret_cast<MatmulFn>(f[0]);
  g_matmul_ws = reinterpret_cast<MatmulWsFn>(f[1]);
  g_fused_ws = reinterpret_cast<FusedWsFn>(f[2]);
  g_qkv = reinterpret_cast<QkvFn>(f[3]);
  g_mlp = reinterpret_cast<MlpFn>(f[4]);
  g_bnb = reinterpret_cast<BnbFn>(f[5]);
  g_gather = reinterpret_cast<GatherFn>(f[6]);
  Py_RETURN_NONE;
}

#define XRMM_FN(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {XRMM_FN(bind), XRMM_FN(matmul), XRMM_FN(qkv), XRMM_FN(mlp),
                          XRMM_FN(bnb4), XRMM_FN(gather), {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_xrmm_torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__xrmm_torch() {
  PyObject* m = PyModule_Create(&kModule);
  if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) != 0) Py_CLEAR(m);
  return m;
}
