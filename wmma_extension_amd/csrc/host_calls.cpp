// The calls of wmma_extension_amd/tcec.py that a program makes often, from Python
// straight to the C entry points of libwmmae_tcec.so: argument checks, pointers and
// output allocation in native code instead of Python and ctypes.
//
// A small product takes the GPU 4.3 us, and issuing it from Python took 7.1
// (tcec.sgemm) and 10.3 (tcec.matmul_tn, with its output): the host bound every
// call below about 10 us.  Now 5.3 and 8.0, of which 1.2 went with OneDeviceCall
// (capi_common.hpp): 4.1 and 6.6; a pack and gemm_packed of a small product 13.2 ->
// 7.4, primitive_tiles with its six outputs 12.9 -> 8.7.
//
// Only the plain case is taken here: exact torch tensors on the GPU, contiguous and
// long enough, ordinary numbers, no torch-function or dispatch mode active.  For
// anything else a function returns kNotTaken, having done nothing, and the caller
// goes on in Python, where every error has its message.  No exception leaves a
// function here: torch's own (a tensor without storage) are a reason not to take the
// call.
#include <Python.h>
// (after Python.h)
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/python_variable.h>

namespace {
constexpr long kNotTaken = 1; // the entry points' statuses are <= 0

// ---- the C entry points, as addresses from whoever loaded the library
typedef int (*sgemm_t)(char, char, int, int, int, const float *, const float *,
                       int, const float *, int, const float *, float *, int,
                       int, int, void *, size_t, void *);
typedef int (*strided_t)(char, char, int, int, int, const float *,
                         const float *, int, long long, const float *, int,
                         long long, const float *, float *, int, long long, int,
                         int, int, void *, size_t, void *);
typedef int (*batched_t)(char, char, int, int, int, const float *,
                         const float *const *, int, const float *const *, int,
                         const float *, float *const *, int, int, int, int,
                         void *, size_t, void *);
typedef int (*pack_bytes_t)(int, int, int, int, size_t *);
typedef int (*pack_t)(int, int, int, const float *, long long, long long,
                      long long, int, void *, size_t, void *);
typedef int (*gemm_packed_t)(int, int, int, int, const float *, const void *,
                             const void *, const float *, float *, int,
                             long long, int, int, void *, size_t, void *);
typedef int (*api_gemm_t)(int, int, int, int, int, const float *, const float *,
                          int, const float *, int, const float *, float *, int,
                          void *);
typedef int (*tiles_t)(const float *, long long, void *, void *, void *, void *,
                       float *, float *, void *);
struct Entries {
  sgemm_t sgemm;
  strided_t strided;
  batched_t batched;
  pack_bytes_t pack_bytes;
  pack_t pack;
  gemm_packed_t gemm_packed;
  api_gemm_t api_gemm;
  tiles_t tiles;
} entries = {};

PyObject *not_taken() { return PyLong_FromLong(kNotTaken); }
// An exact torch.Tensor (or Parameter) on the GPU, else nullptr
const at::Tensor *gpu_tensor(PyObject *const o) {
  if (!THPVariable_CheckExact(o))
    return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o);
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided ? &t : nullptr;
}
bool integer(PyObject *const o, long long &out) {
  if (!PyLong_Check(o))
    return false;
  out = PyLong_AsLongLong(o);
  if (out == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}
bool integer(PyObject *const o, int &out) {
  long long v;
  if (!integer(o, v) || v < INT32_MIN || v > INT32_MAX)
    return false;
  out = static_cast<int>(v);
  return true;
}
bool number(PyObject *const o, float &out) {
  if (PyFloat_CheckExact(o)) {
    out = static_cast<float>(PyFloat_AS_DOUBLE(o));
    return true;
  }
  int v;
  if (!PyLong_CheckExact(o) || !integer(o, v))
    return false;
  out = static_cast<float>(v);
  return true;
}
bool letter(PyObject *const o, char &out) {
  if (!PyUnicode_Check(o) || PyUnicode_GET_LENGTH(o) != 1)
    return false;
  const Py_UCS4 c = PyUnicode_READ_CHAR(o, 0);
  out = static_cast<char>(c);
  return c < 128;
}
bool is_n(const char c) { return c == 'N' || c == 'n'; }
// a column-major rows x cols matrix of leading dimension ld, `batch` of them
// `stride` apart, inside a contiguous fp32 tensor
bool holds(const at::Tensor &t, const long long rows, const long long cols,
           const long long ld, const long long batch, const long long stride) {
  return t.scalar_type() == at::kFloat && rows > 0 && cols > 0 && batch > 0 &&
         ld >= rows && stride >= 0 && t.is_contiguous() &&
         t.numel() >= static_cast<__int128>(batch - 1) * stride +
                          static_cast<__int128>(cols - 1) * ld + rows;
}
struct Room {
  void *data = nullptr;
  size_t bytes = 0;
};
bool room(PyObject *const o, Room &out) {
  if (o == Py_None)
    return true;
  const at::Tensor *const t = gpu_tensor(o);
  if (t == nullptr)
    return false;
  out.data = t->data_ptr();
  out.bytes = static_cast<size_t>(t->numel()) * t->element_size();
  return true;
}
size_t bytes_of(const at::Tensor &t) {
  return static_cast<size_t>(t.numel()) * t.element_size();
}
bool stream_of(PyObject *const o, void *&out) {
  long long v;
  if (!integer(o, v))
    return false;
  out = reinterpret_cast<void *>(static_cast<uintptr_t>(v));
  return true;
}
bool torch_modes() {
  return c10::impl::TorchDispatchModeTLS::any_modes_set() ||
         at::impl::torch_function_mode_enabled();
}
// f() without the interpreter lock, as ctypes calls
template <class F> long unlocked(F f) {
  long st;
  Py_BEGIN_ALLOW_THREADS st = f();
  Py_END_ALLOW_THREADS return st;
}
template <class F> PyObject *guarded(F f) {
  try {
    return f();
  } catch (...) {
    PyErr_Clear();
    return not_taken();
  }
}
#define WMMAE_ARGS PyObject *, PyObject *const *const a, const Py_ssize_t na

// (transa, transb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, policy, flags,
//  workspace, stream)
PyObject *sgemm(WMMAE_ARGS) {
  return guarded([&]() -> PyObject * {
    char ta, tb;
    int m, n, k, lda, ldb, ldc, policy, flags;
    float alpha, beta;
    Room ws;
    void *stream;
    if (na != 17 || !entries.sgemm || !letter(a[0], ta) || !letter(a[1], tb) ||
        !integer(a[2], m) || !integer(a[3], n) || !integer(a[4], k) ||
        !number(a[5], alpha) || !integer(a[7], lda) || !integer(a[9], ldb) ||
        !number(a[10], beta) || !integer(a[12], ldc) || !integer(a[13], policy) ||
        !integer(a[14], flags) || !room(a[15], ws) || !stream_of(a[16], stream))
      return not_taken();
    const at::Tensor *const A = gpu_tensor(a[6]), *const B = gpu_tensor(a[8]),
                            *const C = gpu_tensor(a[11]);
    if (!A || !B || !C || A->get_device() != C->get_device() ||
        B->get_device() != C->get_device() ||
        !holds(*A, is_n(ta) ? m : k, is_n(ta) ? k : m, lda, 1, 0) ||
        !holds(*B, is_n(tb) ? k : n, is_n(tb) ? n : k, ldb, 1, 0) ||
        !holds(*C, m, n, ldc, 1, 0))
      return not_taken();
    const auto *const pa = static_cast<const float *>(A->data_ptr());
    const auto *const pb = static_cast<const float *>(B->data_ptr());
    auto *const pc = static_cast<float *>(C->data_ptr());
    return PyLong_FromLong(unlocked([&] {
      return entries.sgemm(ta, tb, m, n, k, &alpha, pa, lda, pb, ldb, &beta, pc,
                           ldc, policy, flags, ws.data, ws.bytes, stream);
    }));
  });
}

// (transa, transb, m, n, k, alpha, A, lda, stride_a, B, ldb, stride_b, beta, C,
//  ldc, stride_c, batch, policy, flags, workspace, stream)
PyObject *sgemm_strided_batched(WMMAE_ARGS) {
  return guarded([&]() -> PyObject * {
    char ta, tb;
    int m, n, k, lda, ldb, ldc, batch, policy, flags;
    long long sa, sb, sc;
    float alpha, beta;
    Room ws;
    void *stream;
    if (na != 21 || !entries.strided || !letter(a[0], ta) ||
        !letter(a[1], tb) || !integer(a[2], m) || !integer(a[3], n) ||
        !integer(a[4], k) || !number(a[5], alpha) || !integer(a[7], lda) ||
        !integer(a[8], sa) || !integer(a[10], ldb) || !integer(a[11], sb) ||
        !number(a[12], beta) || !integer(a[14], ldc) || !integer(a[15], sc) ||
        !integer(a[16], batch) || !integer(a[17], policy) ||
        !integer(a[18], flags) || !room(a[19], ws) || !stream_of(a[20], stream))
      return not_taken();
    const at::Tensor *const A = gpu_tensor(a[6]), *const B = gpu_tensor(a[9]),
                            *const C = gpu_tensor(a[13]);
    if (!A || !B || !C || A->get_device() != C->get_device() ||
        B->get_device() != C->get_device() ||
        !holds(*A, is_n(ta) ? m : k, is_n(ta) ? k : m, lda, batch, sa) ||
        !holds(*B, is_n(tb) ? k : n, is_n(tb) ? n : k, ldb, batch, sb) ||
        !holds(*C, m, n, ldc, batch, sc))
      return not_taken();
    const auto *const pa = static_cast<const float *>(A->data_ptr());
    const auto *const pb = static_cast<const float *>(B->data_ptr());
    auto *const pc = static_cast<float *>(C->data_ptr());
    return PyLong_FromLong(unlocked([&] {
      return entries.strided(ta, tb, m, n, k, &alpha, pa, lda, sa, pb, ldb, sb,
                             &beta, pc, ldc, sc, batch, policy, flags, ws.data,
                             ws.bytes, stream);
    }));
  });
}

// (transa, transb, m, n, k, alpha, A_array, lda, B_array, ldb, beta, C_array, ldc,
//  batch, policy, flags, workspace, stream)
PyObject *sgemm_batched(WMMAE_ARGS) {
  return guarded([&]() -> PyObject * {
    char ta, tb;
    int m, n, k, lda, ldb, ldc, batch, policy, flags;
    float alpha, beta;
    Room ws;
    void *stream;
    if (na != 18 || !entries.batched || !letter(a[0], ta) ||
        !letter(a[1], tb) || !integer(a[2], m) || !integer(a[3], n) ||
        !integer(a[4], k) || !number(a[5], alpha) || !integer(a[7], lda) ||
        !integer(a[9], ldb) || !number(a[10], beta) || !integer(a[12], ldc) ||
        !integer(a[13], batch) || !integer(a[14], policy) ||
        !integer(a[15], flags) || !room(a[16], ws) || !stream_of(a[17], stream))
      return not_taken();
    void *p[3];
    for (int i = 0; i < 3; i++) {
      const at::Tensor *const t = gpu_tensor(a[i == 0 ? 6 : i == 1 ? 8 : 11]);
      if (!t || t->scalar_type() != at::kLong || t->numel() < batch)
        return not_taken();
      p[i] = t->data_ptr();
    }
    return PyLong_FromLong(unlocked([&] {
      return entries.batched(ta, tb, m, n, k, &alpha,
                             static_cast<const float *const *>(p[0]), lda,
                             static_cast<const float *const *>(p[1]), ldb, &beta,
                             static_cast<float *const *>(p[2]), ldc, batch,
                             policy, flags, ws.data, ws.bytes, stream);
    }));
  });
}

// (A, B, policy, flags, workspace, stream) -> the output, or a status
PyObject *matmul_tn(WMMAE_ARGS) {
  return guarded([&]() -> PyObject * {
    int policy, flags;
    Room ws;
    void *stream;
    if (na != 6 || !entries.sgemm || !integer(a[2], policy) ||
        !integer(a[3], flags) || !room(a[4], ws) || !stream_of(a[5], stream) ||
        torch_modes())
      return not_taken();
    const at::Tensor *const A = gpu_tensor(a[0]), *const B = gpu_tensor(a[1]);
    if (!A || !B || A->dim() != 2 || B->dim() != 2 ||
        A->get_device() != B->get_device() || A->size(1) != B->size(1) ||
        A->numel() == 0 || B->numel() == 0 || A->size(0) > INT32_MAX ||
        B->size(0) > INT32_MAX || A->size(1) > INT32_MAX ||
        A->scalar_type() != at::kFloat || B->scalar_type() != at::kFloat ||
        !A->is_contiguous() || !B->is_contiguous())
      return not_taken();
    const int m = static_cast<int>(A->size(0)), n = static_cast<int>(B->size(0)),
              k = static_cast<int>(A->size(1));
    at::Tensor out = at::empty({n, m}, A->options());
    const float one = 1.f, zero = 0.f;
    const auto *const pa = static_cast<const float *>(A->data_ptr());
    const auto *const pb = static_cast<const float *>(B->data_ptr());
    auto *const pc = static_cast<float *>(out.data_ptr());
    const long st = unlocked([&] {
      return entries.sgemm('T', 'N', m, n, k, &one, pa, k, pb, k, &zero, pc, m,
                           policy, flags, ws.data, ws.bytes, stream);
    });
    return st != 0 ? PyLong_FromLong(st) : THPVariable_Wrap(std::move(out));
  });
}

// (policy, rows, k, X, row_stride, k_stride, packed, batch, batch_stride, stream)
PyObject *pack(WMMAE_ARGS) {
  return guarded([&]() -> PyObject * {
    int policy, rows, k, batch;
    long long rs, ks, bs;
    void *stream;
    if (na != 10 || !entries.pack || !integer(a[0], policy) ||
        !integer(a[1], rows) || !integer(a[2], k) || !integer(a[4], rs) ||
        !integer(a[5], ks) || !integer(a[7], batch) || !integer(a[8], bs) ||
        !stream_of(a[9], stream))
      return not_taken();
    const at::Tensor *const X = gpu_tensor(a[3]), *const P = gpu_tensor(a[6]);
    if (!X || !P || X->scalar_type() != at::kFloat || rows <= 0 || k <= 0 ||
        batch <= 0 || rs < 0 || ks < 0 || bs < 0 ||
        X->get_device() != P->get_device() || !X->is_contiguous() ||
        X->numel() < static_cast<__int128>(batch - 1) * bs +
                         static_cast<__int128>(rows - 1) * rs +
                         static_cast<__int128>(k - 1) * ks + 1)
      return not_taken();
    const auto *const px = static_cast<const float *>(X->data_ptr());
    void *const pp = P->data_ptr();
    const size_t bytes = bytes_of(*P);
    return PyLong_FromLong(unlocked([&] {
      return entries.pack(policy, rows, k, px, rs, ks, bs, batch, pp, bytes,
                          stream);
    }));
  });
}

// (policy, m, n, k, alpha, packed_a, packed_b, beta, C, ldc, batch, stride_c, flags,
//  workspace, stream)
PyObject *gemm_packed(WMMAE_ARGS) {
  return guarded([&]() -> PyObject * {
    int policy, m, n, k, ldc, batch, flags;
    long long sc;
    float alpha, beta;
    Room ws;
    void *stream;
    if (na != 15 || !entries.gemm_packed || !entries.pack_bytes ||
        !integer(a[0], policy) || !integer(a[1], m) || !integer(a[2], n) ||
        !integer(a[3], k) || !number(a[4], alpha) || !number(a[7], beta) ||
        !integer(a[9], ldc) || !integer(a[10], batch) || !integer(a[11], sc) ||
        !integer(a[12], flags) || !room(a[13], ws) || !stream_of(a[14], stream))
      return not_taken();
    const at::Tensor *const A = gpu_tensor(a[5]), *const B = gpu_tensor(a[6]),
                            *const C = gpu_tensor(a[8]);
    size_t need_a = 0, need_b = 0;
    if (!A || !B || !C || k <= 0 ||
        !holds(*C, m, n, ldc, batch, sc) ||
        A->get_device() != C->get_device() || B->get_device() != C->get_device() ||
        !A->is_contiguous() || !B->is_contiguous() ||
        entries.pack_bytes(m, k, batch, policy, &need_a) != 0 ||
        entries.pack_bytes(n, k, batch, policy, &need_b) != 0 ||
        bytes_of(*A) < need_a || bytes_of(*B) < need_b)
      return not_taken();
    const void *const pa = A->data_ptr(), *const pb = B->data_ptr();
    auto *const pc = static_cast<float *>(C->data_ptr());
    return PyLong_FromLong(unlocked([&] {
      return entries.gemm_packed(policy, m, n, k, &alpha, pa, pb, &beta, pc, ldc,
                                 sc, batch, flags, ws.data, ws.bytes, stream);
    }));
  });
}

// (type, ec, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, stream)
PyObject *api_gemm(WMMAE_ARGS) {
  return guarded([&]() -> PyObject * {
    int type, ec, m, n, k, lda, ldb, ldc;
    float alpha, beta;
    void *stream;
    if (na != 14 || !entries.api_gemm || !integer(a[0], type) ||
        !integer(a[1], ec) || !integer(a[2], m) || !integer(a[3], n) ||
        !integer(a[4], k) || !number(a[5], alpha) || !integer(a[7], lda) ||
        !integer(a[9], ldb) || !number(a[10], beta) || !integer(a[12], ldc) ||
        !stream_of(a[13], stream))
      return not_taken();
    const at::Tensor *const A = gpu_tensor(a[6]), *const B = gpu_tensor(a[8]),
                            *const C = gpu_tensor(a[11]);
    if (!A || !B || !C || A->get_device() != C->get_device() ||
        B->get_device() != C->get_device() || !holds(*A, k, m, lda, 1, 0) ||
        !holds(*B, k, n, ldb, 1, 0) || !holds(*C, m, n, ldc, 1, 0))
      return not_taken();
    const auto *const pa = static_cast<const float *>(A->data_ptr());
    const auto *const pb = static_cast<const float *>(B->data_ptr());
    auto *const pc = static_cast<float *>(C->data_ptr());
    return PyLong_FromLong(unlocked([&] {
      return entries.api_gemm(type, ec, m, n, k, &alpha, pa, lda, pb, ldb, &beta,
                              pc, ldc, stream);
    }));
  });
}

// (tiles, stream) -> dict of the outputs, or a status
PyObject *primitive_tiles(WMMAE_ARGS) {
  return guarded([&]() -> PyObject * {
    void *stream;
    if (na != 2 || !entries.tiles || !stream_of(a[1], stream) || torch_modes())
      return not_taken();
    const at::Tensor *const t = gpu_tensor(a[0]);
    if (!t || t->dim() != 2 || t->size(1) != 256 || t->size(0) == 0 ||
        t->scalar_type() != at::kFloat || !t->is_contiguous())
      return not_taken();
    const long long T = t->size(0);
    static const char *const names[6] = {"a_row", "a_col", "b_row",
                                         "b_col", "acc",   "vec"};
    at::Tensor out[6];
    void *p[6];
    const auto half = t->options().dtype(at::kHalf);
    for (int i = 0; i < 6; i++) {
      out[i] = i < 4    ? at::empty({T, 64, 4}, half)
               : i == 4 ? at::empty({T, 256}, t->options())
                        : at::empty({T, 32}, t->options());
      p[i] = out[i].data_ptr();
    }
    const auto *const pt = static_cast<const float *>(t->data_ptr());
    const long st = unlocked([&] {
      return entries.tiles(pt, T, p[0], p[1], p[2], p[3],
                           static_cast<float *>(p[4]),
                           static_cast<float *>(p[5]), stream);
    });
    if (st != 0)
      return PyLong_FromLong(st);
    PyObject *const d = PyDict_New();
    for (int i = 0; d != nullptr && i < 6; i++) {
      PyObject *const v = THPVariable_Wrap(std::move(out[i]));
      if (v == nullptr || PyDict_SetItemString(d, names[i], v) != 0) {
        Py_XDECREF(v);
        Py_DECREF(d);
        return nullptr;
      }
      Py_DECREF(v);
    }
    return d;
  });
}

// bind(name, address): an entry point of the loaded library
PyObject *bind(PyObject *, PyObject *const args) {
  const char *name;
  unsigned long long address;
  if (!PyArg_ParseTuple(args, "sK", &name, &address))
    return nullptr;
  const struct {
    const char *name;
    void *slot;
  } slots[] = {{"wmmae_tcec_sgemm", &entries.sgemm},
               {"wmmae_tcec_sgemm_strided_batched", &entries.strided},
               {"wmmae_tcec_sgemm_batched", &entries.batched},
               {"wmmae_tcec_pack_bytes", &entries.pack_bytes},
               {"wmmae_tcec_pack", &entries.pack},
               {"wmmae_tcec_gemm_packed", &entries.gemm_packed},
               {"wmmae_tcec_api_gemm", &entries.api_gemm},
               {"wmmae_primitive_tiles", &entries.tiles}};
  for (const auto &s : slots)
    if (__builtin_strcmp(s.name, name) == 0) {
      *static_cast<void **>(s.slot) = reinterpret_cast<void *>(address);
      Py_RETURN_TRUE;
    }
  Py_RETURN_FALSE;
}

#define WMMAE_FAST(f)                                                          \
  {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)),          \
   METH_FASTCALL, nullptr}
PyMethodDef methods[] = {WMMAE_FAST(sgemm),
                         WMMAE_FAST(sgemm_strided_batched),
                         WMMAE_FAST(sgemm_batched),
                         WMMAE_FAST(matmul_tn),
                         WMMAE_FAST(pack),
                         WMMAE_FAST(gemm_packed),
                         WMMAE_FAST(api_gemm),
                         WMMAE_FAST(primitive_tiles),
                         {"bind", bind, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_wmmae_host_calls", nullptr, -1,
                      methods};
} // namespace

PyMODINIT_FUNC PyInit__wmmae_host_calls() { return PyModule_Create(&module); }
