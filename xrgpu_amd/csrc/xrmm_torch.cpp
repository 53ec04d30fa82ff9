// Native front end of the zero-copy entry points: the argument checks, output
// allocations and calls of xrgpu_amd/ops.py for ordinary arguments. In Python they
// cost more than a decode kernel runs (Qkv at four rows: 16.8 us a call for an 8 us
// kernel; 27 ctypes arguments, four allocations, ten tensors' properties).
//
// Every function returns None, having done nothing, for whatever it does not take: a
// tensor that is not a plain torch.Tensor on one GPU (subclasses, wrappers, CPU), any
// mode that intercepts calls, a dtype, shape or layout that does not match, an empty
// batch. ops.py then runs its own checks, which raise or accept as they always did. A
// MatMulNBits call that runs on a workspace comes back checked, as the workspace's
// bytes (an int): ops.py, which keeps one per stream, makes the call. Declines are
// return values and no exceptions: a throw costs 4 us, more than the checks (a float32
// call on a workspace 17 x 1024 x 1024 took 18.7 us on the host with throws and every
// check made twice, 15.8 without a front end).
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

// Helpers return false where ops.py takes the call.

// A plain tensor on one GPU, contiguous; `dev` is the call's device (-1: not known yet).
bool plain(PyObject* o, int& dev, const at::Tensor*& out) {
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  const auto ks = t.key_set();
  if (!t.is_cuda() || t.layout() != at::kStrided || ks.has(c10::DispatchKey::Python) ||
      ks.has_any(c10::functorch_transforms_ks) || t.is_conj() || t.is_neg() || !t.is_contiguous() || t.numel() == 0)
    return false;
  const int d = t.get_device();
  if (dev < 0) dev = d;
  out = &t;
  return d == dev;
}

bool none(PyObject* o) { return o == Py_None; }

bool integer(PyObject* o, int64_t& v) {
  if (!PyLong_CheckExact(o)) return false;
  int over = 0;
  v = PyLong_AsLongLongAndOverflow(o, &over);
  return over == 0;
}

bool real(PyObject* o, float& v) {
  if (PyFloat_CheckExact(o)) {
    v = static_cast<float>(PyFloat_AS_DOUBLE(o));
    return true;
  }
  int64_t i = 0;
  if (!integer(o, i)) return false;
  v = static_cast<float>(static_cast<double>(i));
  return true;
}

// None or the integer n
bool none_or(PyObject* o, int64_t n) {
  int64_t v = 0;
  return none(o) || (integer(o, v) && v == n);
}

bool shape(const at::Tensor& t, std::initializer_list<int64_t> s) { return t.sizes() == at::IntArrayRef(s.begin(), s.size()); }

bool t1(const at::Tensor& a, int& dt) {
  dt = a.scalar_type() == at::kHalf ? F16 : F32;
  return dt == F16 || a.scalar_type() == at::kFloat;
}

bool stream_of(int dev, void*& s) {
  PyObject* i = PyLong_FromLong(dev);
  PyObject* r = i ? PyObject_CallOneArg(g_stream, i) : nullptr;
  Py_XDECREF(i);
  s = r ? PyLong_AsVoidPtr(r) : nullptr;
  Py_XDECREF(r);
  if (s == nullptr && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

// rows, K and the leading axes of the activations
struct Act {
  const at::Tensor* A = nullptr;
  int64_t K = 0, M = 0;
  int dt = F32;
  bool set(PyObject* a, PyObject* k, int& dev) {
    if (!plain(a, dev, A) || !t1(*A, dt) || A->dim() < 1) return false;
    K = A->size(-1);
    M = A->numel() / K;
    return none_or(k, K);
  }
  const void* data() const { return A->data_ptr(); }
  at::Tensor out(int64_t n) const {
    at::DimVector s(A->sizes().slice(0, A->dim() - 1));
    s.push_back(n);
    return at::empty(s, A->options());
  }
};

struct Quant {
  int bits = 0, bs = 0;
  int64_t kb = 0, blob = 0, zrow = 0;
  bool set(PyObject* b, PyObject* s, int64_t K) {
    int64_t bb = 0, ss = 0;
    if (!integer(b, bb) || !integer(s, ss) || !(bb == 2 || bb == 4 || bb == 8) || ss <= 0 || ss > (1 << 20)) return false;
    bits = static_cast<int>(bb);
    bs = static_cast<int>(ss);
    kb = (K + bs - 1) / bs;
    blob = (static_cast<int64_t>(bs) * bits + 7) / 8;
    zrow = (kb * bits + 7) / 8;
    return true;
  }
};

struct Weights {
  const void *B = nullptr, *S = nullptr, *Z = nullptr;
  int zdt = UNSPECIFIED;
  int64_t N = 0;
  bool set(PyObject* b, PyObject* s, PyObject* z, PyObject* n, const Act& a, const Quant& q, int& dev) {
    const at::Tensor *tb, *ts, *tz;
    if (!plain(b, dev, tb) || !plain(s, dev, ts) || tb->scalar_type() != at::kByte || tb->dim() != 3) return false;
    N = tb->size(0);
    if (!none_or(n, N) || !shape(*tb, {N, q.kb, q.blob}) || ts->scalar_type() != a.A->scalar_type() || !shape(*ts, {N, q.kb}))
      return false;
    B = tb->data_ptr();
    S = ts->data_ptr();
    if (none(z)) return true;
    if (!plain(z, dev, tz)) return false;
    const bool packed = tz->scalar_type() == at::kByte;
    if (packed) zdt = U8;
    else if (!t1(*tz, zdt)) return false;
    Z = tz->data_ptr();
    return shape(*tz, {N, packed ? q.zrow : q.kb});
  }
};

// an optional tensor of A's dtype with n elements (vec: one-dimensional)
bool aux(PyObject* o, const Act& a, int64_t n, bool vec, int& dev, const void*& p) {
  p = nullptr;
  if (none(o)) return true;
  const at::Tensor* t;
  if (!plain(o, dev, t) || t->scalar_type() != a.A->scalar_type() || t->numel() != n || (vec && t->dim() != 1)) return false;
  p = t->data_ptr();
  return true;
}

// the projections' common zero-point dtype
bool one_zdt(std::initializer_list<const Weights*> ws, int& dt) {
  dt = UNSPECIFIED;
  for (const Weights* w : ws)
    if (w->Z) {
      if (dt != UNSPECIFIED && dt != w->zdt) return false;
      dt = w->zdt;
    }
  return true;
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
  } catch (const std::exception& e) {  // an allocation that failed, say: ops.py meets it again
    Py_RETURN_NONE;
  }
}

// (A, B, scales, zero_points, bias, K, N, bits, block_size); an int: checked, needs a
// workspace of that many bytes
PyObject* matmul(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 9, [&]() -> PyObject* {
    int dev = -1;
    Act a;
    Quant q;
    Weights w;
    const void* bias;
    if (!a.set(v[0], v[5], dev) || !q.set(v[7], v[8], a.K) || !w.set(v[1], v[2], v[3], v[6], a, q, dev) ||
        !aux(v[4], a, w.N, true, dev, bias))
      Py_RETURN_NONE;
    if (a.M > 4) {
      const int64_t need = g_matmul_ws(a.M, a.K, w.N, q.bits, q.bs, a.dt);
      if (need > 0) return PyLong_FromLongLong(need);
    }
    void* st;
    if (!stream_of(dev, st)) Py_RETURN_NONE;
    at::Tensor y;
    int rc;
    {
      NoGil ng;
      y = a.out(w.N);
      rc = g_matmul(a.data(), w.B, w.S, w.Z, w.zdt, bias, y.data_ptr(), a.M, a.K, w.N, q.bits, q.bs, a.dt, st);
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
  return at::empty({bytes}, a.A->options().dtype(at::kByte));
}

// (A, q_B, q_scales, k_B, k_scales, v_B, v_scales, norm_scale, skip, K, Nq, Nkv, bits,
//  block_size, epsilon, q_zero_points, k_zero_points, v_zero_points, want_residual)
PyObject* qkv(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 19, [&]() -> PyObject* {
    int dev = -1, zdt;
    Act a;
    Quant q;
    Weights wq, wk, wv;
    const void *gamma, *skip;
    void* st;
    float eps;
    if (!real(v[14], eps) || !PyBool_Check(v[18]) || none(v[7]) || !a.set(v[0], v[9], dev) || !q.set(v[12], v[13], a.K) || !wq.set(v[1], v[2], v[15], v[10], a, q, dev) ||
        !wk.set(v[3], v[4], v[16], v[11], a, q, dev) || !wv.set(v[5], v[6], v[17], v[11], a, q, dev) || wk.N != wv.N ||
        !one_zdt({&wq, &wk, &wv}, zdt) || !aux(v[7], a, a.K, true, dev, gamma) ||
        !aux(v[8], a, a.M * a.K, false, dev, skip) || !stream_of(dev, st))
      Py_RETURN_NONE;
    const bool residual = v[18] == Py_True;
    at::Tensor Q, Ko, V, R;
    int rc;
    {
      NoGil ng;
      Q = a.out(wq.N), Ko = a.out(wk.N), V = a.out(wv.N);
      if (residual) R = a.out(a.K);
      int64_t nws = 0;
      const at::Tensor ws = scratch(1, a, wq.N, wk.N, q, skip != nullptr, true, nws);
      rc = g_qkv(a.data(), skip, gamma, wq.B, wq.S, wq.Z, wk.B, wk.S, wk.Z, wv.B, wv.S, wv.Z, zdt, Q.data_ptr(),
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
    int dev = -1, zdt;
    Act a;
    Quant q;
    Weights g, u;
    const void *skip, *gamma, *gb, *ub;
    int64_t act = 0;
    void* st;
    float eps;
    if (!real(v[13], eps) || !integer(v[14], act) || !PyBool_Check(v[17]) || !a.set(v[0], v[9], dev) || !q.set(v[11], v[12], a.K) || !g.set(v[1], v[2], v[15], v[10], a, q, dev) ||
        !u.set(v[3], v[4], v[16], v[10], a, q, dev) || g.N != u.N || !one_zdt({&g, &u}, zdt) ||
        !aux(v[5], a, a.M * a.K, false, dev, skip) || !aux(v[6], a, a.K, true, dev, gamma) || !aux(v[7], a, g.N, true, dev, gb) ||
        !aux(v[8], a, g.N, true, dev, ub) || !stream_of(dev, st))
      Py_RETURN_NONE;
    const bool residual = v[17] == Py_True;
    at::Tensor Y, R;
    int rc;
    {
      NoGil ng;
      Y = a.out(g.N);
      if (residual) R = a.out(a.K);
      int64_t nws = 0;
      const at::Tensor ws = scratch(2, a, g.N, 0, q, skip != nullptr, gamma != nullptr, nws);
      rc = g_mlp(a.data(), skip, gamma, g.B, g.S, g.Z, gb, u.B, u.S, u.Z, ub, zdt, Y.data_ptr(),
                 residual ? R.data_ptr() : nullptr, a.M, a.K, g.N, q.bits, q.bs, eps, static_cast<int>(act), a.dt,
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
    Act a;
    const at::Tensor *B, *S;
    int64_t N = 0, bs = 0, qt = 0, tb = 0;
    void* st;
    if (!a.set(v[0], v[3], dev) || !plain(v[1], dev, B) || !plain(v[2], dev, S) || !integer(v[4], N) || !integer(v[5], bs) ||
        !integer(v[6], qt) || !integer(v[7], tb))
      Py_RETURN_NONE;
    const int64_t lim = int64_t(1) << 31;
    if (a.A->dim() != 2 || N <= 0 || N >= lim || a.K >= lim || bs <= 0 || bs > (1 << 20) || B->scalar_type() != at::kByte ||
        S->scalar_type() != a.A->scalar_type() || B->numel() < (N * a.K + 1) / 2 || S->numel() < (N * a.K + bs - 1) / bs ||
        !(qt == 0 || qt == 1) || !(tb == 0 || tb == 1) || !stream_of(dev, st))
      Py_RETURN_NONE;
    at::Tensor y;
    int rc;
    {
      NoGil ng;
      y = a.out(N);
      rc = g_bnb(a.data(), B->data_ptr(), S->data_ptr(), y.data_ptr(), a.M, a.K, N, static_cast<int32_t>(bs),
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
    const at::Tensor *D, *I, *S, *T, *Z;
    int64_t bits = 0, bs = 0;
    if (!plain(v[0], dev, D) || !plain(v[1], dev, I) || !plain(v[2], dev, S) || !plain(v[4], dev, T) || !integer(v[5], bits) ||
        !integer(v[6], bs) || !(bits == 4 || bits == 8) || bs <= 0 || bs > (1 << 20) || D->scalar_type() != at::kByte ||
        D->dim() != 2 || I->dim() != 1 || S->scalar_type() != at::kFloat ||
        !(T->scalar_type() == at::kInt || T->scalar_type() == at::kUInt32))
      Py_RETURN_NONE;
    const bool i64 = I->scalar_type() == at::kLong;
    const int64_t rows = D->size(0), pcols = D->size(1), width = pcols * (8 / bits), blocks = (width + bs - 1) / bs;
    if (!(i64 || I->scalar_type() == at::kInt) || !shape(*S, {rows, blocks})) Py_RETURN_NONE;
    const void* z = nullptr;
    if (!none(v[3])) {
      if (!plain(v[3], dev, Z) || Z->scalar_type() != at::kByte || !shape(*Z, {rows, (blocks * bits + 7) / 8})) Py_RETURN_NONE;
      z = Z->data_ptr();
    }
    void* st;
    if (!stream_of(dev, st)) Py_RETURN_NONE;
    at::Tensor y;
    int rc;
    {
      NoGil ng;
      y = at::empty({I->size(0), width}, S->options());
      rc = g_gather(D->data_ptr(), I->data_ptr(), i64 ? 7 : 2, S->data_ptr(), z, y.data_ptr(), T->data_ptr(), rows, pcols,
                    I->size(0), static_cast<int32_t>(bits), static_cast<int32_t>(bs), st);
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
