// The host path of the ordinary calls, in native code: flash_maxsim_amd._native.
//
// A call on floating-point GPU tensors of the current device with int32 lengths
// is checked, given its outputs and workspace and launched here; operands that
// the kernels do not read as they are (float32, mixed types, rows off the
// alignment that include/fmx.h asks for) go through fmx_convert_rows first, one
// pass each. Every other call (other types and devices, inner strides, empty
// sizes, wrong shapes) gets None and takes the Python path, which has the asserts and the
// error messages. In Python and ctypes an ordinary call's checks, allocations
// and the conversion of twenty arguments took longer than the kernels of a
// rerank: 100 docs of up to 300 x 128 under 32 tokens
// 14.3 -> 4.8 us a call, 1000 docs with 16 tokens each 12.8 -> 9.1. (A training
// step's host time depends more on where autograd's thread runs: 85 or 150 us
// before, 105 after, for 32 x 32 tokens over 256 docs of up to 180.)
//
// The library is reached through its C ABI alone.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>

#include "../../include/fmx.h"

namespace {

using at::Tensor;

// A tensor that nothing wraps (no subclass, no function transform) on the GPU, or null.
const Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet watched({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                         c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::BatchedNestedTensor,
                                         c10::DispatchKey::Functionalize, c10::DispatchKey::Negative,
                                         c10::DispatchKey::Conjugate, c10::DispatchKey::ZeroTensor});
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return nullptr;
  if (t.key_set().has_any(watched)) return nullptr;
  return &t;
}

// Operand rows that the kernels read in place: unit inner stride, rows at
// least d apart, every other stride a multiple of 8 (fp32: 4), 16-byte aligned.
bool rows_ready(const Tensor& t) {
  const int64_t n = t.dim();
  if (n < 2 || t.stride(n - 1) != 1 || t.stride(n - 2) < t.size(n - 1)) return false;
  const int64_t m = t.scalar_type() == at::kFloat ? 3 : 7;
  for (int64_t i = 0; i + 1 < n; ++i)
    if (t.stride(i) & m) return false;
  return (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15u) == 0;
}

// The library's code of a floating-point type, or -1.
int code_of(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kHalf: return FMX_DTYPE_F16;
    case at::kBFloat16: return FMX_DTYPE_BF16;
    case at::kFloat: return FMX_DTYPE_F32;
    default: return -1;
  }
}

// The type the kernels run Q and D in: bf16 when both are, else fp16; -1 for types cast elsewhere.
int kernel_dtype(const Tensor& Q, const Tensor& D) {
  const int q = code_of(Q), x = code_of(D);
  if (q < 0 || x < 0) return -1;
  return q == FMX_DTYPE_BF16 && x == FMX_DTYPE_BF16 ? FMX_DTYPE_BF16 : FMX_DTYPE_F16;
}

// Whether n fp32 rows of t and `slack` more span less than 2 GiB, as the library's
// checks ask of a query (slack 128) and of a document (16).
bool f32_in_range(const Tensor& t, int64_t n, int64_t slack) {
  return t.stride(t.dim() - 2) <= (((int64_t)1 << 29) - 1) / (n + slack);
}

// The same for one query of Lq tokens (or Lq tokens a doc) over docs of up to Ld:
// float32 operands that the kernels read in place stay so. Rows too far apart for
// that (views of token-major storage), or too many of them, are cast like other
// layouts: the fp16 copy is contiguous and half the size.
int scoring_dtype(const Tensor& Q, const Tensor& D, int64_t Lq, int64_t Ld, int64_t d) {
  if (code_of(Q) == FMX_DTYPE_F32 && code_of(D) == FMX_DTYPE_F32 && fmx_fwd_reads_f32(Lq, d) && rows_ready(Q) &&
      rows_ready(D) && f32_in_range(Q, std::max(Lq, Q.size(0)), 128) && f32_in_range(D, Ld, 16))
    return FMX_DTYPE_F32;
  return kernel_dtype(Q, D);
}

// Whether `ready` can make t an operand.
bool convertible(const Tensor& t) {
  const int64_t n = t.dim(), d = t.size(n - 1);
  return (n == 2 || n == 3) && t.stride(n - 1) == 1 && d >= 1 && t.numel() > 0 &&
         t.size(n - 2) <= (INT32_MAX - 4096) / (2 * (d / 8 + 1));
}

bool is_row_of(const Tensor* t, at::ScalarType type, int64_t n) {
  return t->scalar_type() == type && t->numel() == n && t->is_contiguous();
}

// Document lengths: None, or n int32 values. False: not such a tensor.
bool take_lengths(PyObject* o, int64_t n, const Tensor& like, const int32_t** out) {
  *out = nullptr;
  if (o == Py_None) return true;
  const Tensor* t = plain(o);
  if (!t || t->device() != like.device() || !is_row_of(t, at::kInt, n)) return false;
  *out = t->const_data_ptr<int32_t>();
  return true;
}

// Nothing but a launch between the caller and the GPU: the operand's device is
// current and no dispatch mode watches the allocations.
bool here(const Tensor& t) {
  return t.device().index() == c10::hip::current_device() && !c10::impl::TorchDispatchModeTLS::any_modes_set();
}

void* stream_of(const Tensor& t);

// t as the kernels read it in type `dtype`: itself, or a converted copy with its
// rows padded to a multiple of 8 elements (of documents, the rows within `lengths`,
// where given: nothing reads the others). Undefined, with *rc set: the conversion failed.
Tensor ready(const Tensor& t, int dtype, const int32_t* lengths, int* rc) {
  if (code_of(t) == dtype && rows_ready(t)) return t;
  const int64_t n = t.dim(), d = t.size(n - 1), dp = (d + 7) / 8 * 8, rows = t.size(n - 2);
  // Docs of fewer than 1024 elements are converted whole: by lengths each takes a
  // workgroup of its own, without them they are cut like one long doc (16666 docs of 5
  // x 48 15.9 -> 4.6 us, 78125 of 8 x 64 60 -> 35; 146484 of 8 x 128 by lengths 121, whole 142).
  if (rows * dp < 1024) lengths = nullptr;
  auto sizes = t.sizes().vec();
  sizes[n - 1] = dp;
  Tensor out = at::empty(sizes, t.options().dtype(dtype == FMX_DTYPE_BF16 ? at::kBFloat16 : at::kHalf));
  *rc = fmx_convert_rows(code_of(t), t.const_data_ptr(), n == 3 ? t.stride(0) : 0, t.stride(n - 2),
                         n == 3 ? t.size(0) : 1, rows, d, lengths, dtype, out.data_ptr(), dp, stream_of(t));
  return *rc ? Tensor() : out;
}

// Q and D as operands, in place of their originals.
#define FMX_READY(Q, D, lengths)                       \
  int prc = 0;                                         \
  const Tensor Qk = ready(*Q, dtype, nullptr, &prc);   \
  if (prc) return failed(prc);                         \
  const Tensor Dk = ready(*D, dtype, lengths, &prc);   \
  if (prc) return failed(prc)

PyObject* failed(int rc);

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// Scratch of n bytes, or an undefined tensor for none.
Tensor scratch(size_t n, const Tensor& like) {
  return n ? at::empty({(int64_t)((n + 3) / 4)}, like.options().dtype(at::kFloat)) : Tensor();
}
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

PyObject* failed(int rc) {
  PyErr_Format(PyExc_RuntimeError, "flash_maxsim_amd: %s (code %d)", fmx_last_error(), rc);
  return nullptr;
}

// Runs a library call without the GIL. The error text is this thread's, so it is read after.
template <typename F>
int unlocked(F&& f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  Py_END_ALLOW_THREADS
  return rc;
}

#define FMX_ARGS(n) \
  if (nargs != n) return PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", n, nargs)
#define FMX_ORDINARY(cond) \
  if (!(cond)) Py_RETURN_NONE

// score(Q [Lq, d], D [B, Ld, d], lengths): float32 [B]
PyObject* score(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  FMX_ARGS(3);
  const Tensor *Q = plain(args[0]), *D = plain(args[1]);
  FMX_ORDINARY(Q && D && Q->dim() == 2 && D->dim() == 3 && Q->size(1) == D->size(2));
  const int64_t Lq = Q->size(0), d = Q->size(1), B = D->size(0), Ld = D->size(1);
  const int dtype = scoring_dtype(*Q, *D, Lq, Ld, d);
  const int32_t* lengths;
  FMX_ORDINARY(dtype >= 0 && B > 0 && Lq > 0 && convertible(*Q) && convertible(*D) && Q->device() == D->device() &&
               take_lengths(args[2], B, *D, &lengths) && here(*Q));
  Tensor out = at::empty({B}, D->options().dtype(at::kFloat));
  const size_t n = fmx_fwd_workspace_bytes(1, B, Lq, Ld, d);
  const Tensor ws = scratch(n, *D);
  FMX_READY(Q, D, lengths);
  void* s = stream_of(*Q);
  const int rc = unlocked([&] {
    return fmx_fwd(dtype, Qk.const_data_ptr(), 0, Qk.stride(0), Dk.const_data_ptr(), Dk.stride(0), Dk.stride(1),
                   lengths, out.data_ptr<float>(), B, 1, nullptr, 1, B, Lq, Ld, d, 1, ptr(ws), n, s);
  });
  return rc ? failed(rc) : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// batched(Q [Nq, Lq, d], D [B, Ld, d] or [Nq, B, Ld, d], lengths, shared_docs): float32 [Nq, B]
PyObject* batched(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  FMX_ARGS(4);
  const Tensor *Q = plain(args[0]), *D = plain(args[1]);
  const int shared = PyObject_IsTrue(args[3]);
  if (shared < 0) return nullptr;
  FMX_ORDINARY(Q && D && Q->dim() == 3 && D->dim() == (shared ? 3 : 4));
  const int64_t Nq = Q->size(0), Lq = Q->size(1), d = Q->size(2), k = shared ? 0 : 1;
  const int64_t B = D->size(k), Ld = D->size(k + 1);
  const int dtype = kernel_dtype(*Q, *D);
  const int32_t* lengths;
  FMX_ORDINARY(D->size(k + 2) == d && (shared || (D->size(0) == Nq && D->stride(0) == B * D->stride(1))));
  FMX_ORDINARY(dtype >= 0 && Nq > 0 && B > 0 && Lq > 0 && convertible(*Q) &&
               (shared ? convertible(*D) : code_of(*D) == dtype && rows_ready(*D)) &&
               Q->device() == D->device() && take_lengths(args[2], shared ? B : Nq * B, *D, &lengths) && here(*Q));
  Tensor out = at::empty({Nq, B}, D->options().dtype(at::kFloat));
  const size_t n = fmx_fwd_workspace_bytes(Nq, B, Lq, Ld, d);
  const Tensor ws = scratch(n, *D);
  FMX_READY(Q, D, lengths);
  void* s = stream_of(*Q);
  const int rc = unlocked([&] {
    return fmx_fwd(dtype, Qk.const_data_ptr(), Qk.stride(0), Qk.stride(1), Dk.const_data_ptr(), Dk.stride(k),
                   Dk.stride(k + 1), lengths, out.data_ptr<float>(), B, 1, nullptr, Nq, B, Lq, Ld, d, shared, ptr(ws),
                   n, s);
  });
  return rc ? failed(rc) : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// sparse(Q [Lq, d], D [B, Ld, d], indices [B, K] int32, lengths): float32 [B]
PyObject* sparse(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  FMX_ARGS(4);
  const Tensor *Q = plain(args[0]), *D = plain(args[1]), *idx = plain(args[2]);
  FMX_ORDINARY(Q && D && idx && Q->dim() == 2 && D->dim() == 3 && idx->dim() == 2 && Q->size(1) == D->size(2));
  const int64_t Lq = Q->size(0), d = Q->size(1), B = D->size(0), Ld = D->size(1), K = idx->size(1);
  const int dtype = scoring_dtype(*Q, *D, K, Ld, d);
  const int32_t* lengths;
  FMX_ORDINARY(dtype >= 0 && B > 0 && Lq > 0 && K > 0 && idx->size(0) == B && is_row_of(idx, at::kInt, B * K));
  FMX_ORDINARY(convertible(*Q) && convertible(*D) && Q->device() == D->device() && idx->device() == D->device() &&
               take_lengths(args[3], B, *D, &lengths) && here(*Q));
  Tensor out = at::empty({B}, D->options().dtype(at::kFloat));
  const size_t n = fmx_fwd_sparse_workspace_bytes(B, K, Ld, d);
  const Tensor ws = scratch(n, *D);
  FMX_READY(Q, D, lengths);
  void* s = stream_of(*Q);
  const int rc = unlocked([&] {
    return fmx_fwd_sparse(dtype, Qk.const_data_ptr(), Qk.stride(0), Lq, Dk.const_data_ptr(), Dk.stride(0), Dk.stride(1),
                          idx->const_data_ptr<int32_t>(), K, 1, K, lengths, out.data_ptr<float>(), B, Ld, d, ptr(ws), n,
                          s);
  });
  return rc ? failed(rc) : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// topk(Q [Lq, d], D [B, Ld, d], k, lengths): (float32 [k], int64 [k])
PyObject* topk(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  FMX_ARGS(4);
  const Tensor *Q = plain(args[0]), *D = plain(args[1]);
  FMX_ORDINARY(PyLong_CheckExact(args[2]));
  FMX_ORDINARY(Q && D && Q->dim() == 2 && D->dim() == 3 && Q->size(1) == D->size(2));
  const long long k = PyLong_AsLongLong(args[2]);
  if (k == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const int64_t Lq = Q->size(0), d = Q->size(1), B = D->size(0), Ld = D->size(1);
  const int dtype = scoring_dtype(*Q, *D, Lq, Ld, d);
  const int32_t* lengths;
  FMX_ORDINARY(dtype >= 0 && Lq > 0 && k > 0 && k <= B && convertible(*Q) && convertible(*D) &&
               Q->device() == D->device() && take_lengths(args[3], B, *D, &lengths) && here(*Q));
  const auto f32 = D->options().dtype(at::kFloat);
  const Tensor scores = at::empty({B}, f32);
  Tensor values = at::empty({k}, f32), indices = at::empty({k}, D->options().dtype(at::kLong));
  const size_t n = fmx_fwd_topk_workspace_bytes(B, Lq, Ld, d, k);
  const Tensor ws = scratch(n, *D);
  FMX_READY(Q, D, lengths);
  void* s = stream_of(*Q);
  const int rc = unlocked([&] {
    return fmx_fwd_topk(dtype, Qk.const_data_ptr(), Qk.stride(0), Dk.const_data_ptr(), Dk.stride(0), Dk.stride(1),
                        lengths, B, Lq, Ld, d, k, scores.data_ptr<float>(), values.data_ptr<float>(),
                        indices.data_ptr<int64_t>(), ptr(ws), n, s);
  });
  if (rc) return failed(rc);
  return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(values)), THPVariable_Wrap(std::move(indices)));
  END_HANDLE_TH_ERRORS
}

// int8(Q [Lq, d] fp16, codes [B, Ld, d] uint8, scales and mins [B, Ld(, 1)] fp16, lengths): float32 [B]
PyObject* int8(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  FMX_ARGS(5);
  const Tensor *Q = plain(args[0]), *D = plain(args[1]), *sc = plain(args[2]), *mn = plain(args[3]);
  FMX_ORDINARY(Q && D && sc && mn && Q->dim() == 2 && D->dim() == 3 && Q->size(1) == D->size(2));
  FMX_ORDINARY(Q->scalar_type() == at::kHalf && D->scalar_type() == at::kByte);
  const int64_t Lq = Q->size(0), d = Q->size(1), B = D->size(0), Ld = D->size(1);
  for (const Tensor* t : {sc, mn}) {
    FMX_ORDINARY(t->scalar_type() == at::kHalf && (t->dim() == 2 || (t->dim() == 3 && t->size(2) == 1)));
    FMX_ORDINARY(t->size(0) == B && t->size(1) == Ld && t->stride(1) == 1 && t->stride(0) >= Ld &&
                 t->device() == D->device());
  }
  const int32_t* lengths;
  FMX_ORDINARY(B > 0 && Lq > 0 && sc->stride(0) == mn->stride(0) && rows_ready(*Q) && rows_ready(*D) &&
               Q->device() == D->device() && take_lengths(args[4], B, *D, &lengths) && here(*Q));
  Tensor out = at::empty({B}, D->options().dtype(at::kFloat));
  const size_t n = fmx_fwd_int8_workspace_bytes(B, Lq, Ld, d);
  const Tensor ws = scratch(n, *D);
  void* s = stream_of(*Q);
  const int rc = unlocked([&] {
    return fmx_fwd_int8(Q->const_data_ptr(), Q->stride(0), D->const_data_ptr<uint8_t>(), D->stride(0), D->stride(1),
                        sc->const_data_ptr(), mn->const_data_ptr(), sc->stride(0), lengths, out.data_ptr<float>(), B,
                        Lq, Ld, d, ptr(ws), n, s);
  });
  return rc ? failed(rc) : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// The slots of packed docs: tok_group int64, lengths int32 and doc_ids int32 or None, of B docs.
bool take_slots(PyObject* group, PyObject* len, PyObject* ids, const Tensor& like, int64_t* B, const int64_t** g,
                const int32_t** l, const int32_t** i) {
  const Tensor *tg = plain(group), *tl = plain(len);
  if (!tg || !tl || tg->device() != like.device()) return false;
  *B = tl->numel();
  if (!is_row_of(tg, at::kLong, *B)) return false;
  *g = tg->const_data_ptr<int64_t>();
  return len != Py_None && take_lengths(len, *B, like, l) && take_lengths(ids, *B, like, i);
}

// packed(Q [Lq, d], tokens [T, d], tok_group, lengths, max_len, doc_ids): float32 [B]
PyObject* packed(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  FMX_ARGS(6);
  const Tensor *Q = plain(args[0]), *D = plain(args[1]);
  FMX_ORDINARY(Q && D && Q->dim() == 2 && D->dim() == 2 && Q->size(1) == D->size(1) && PyLong_CheckExact(args[4]));
  const int64_t Lq = Q->size(0), d = Q->size(1), T = D->size(0);
  const long max_len = PyLong_AsLong(args[4]);
  if (max_len == -1 && PyErr_Occurred()) return nullptr;
  const int64_t Ld = max_len > 1 ? max_len : 1;
  const int dtype = scoring_dtype(*Q, *D, Lq, Ld, d);
  int64_t B;
  const int64_t* group;
  const int32_t *lengths, *ids;
  FMX_ORDINARY(dtype >= 0 && Q->device() == D->device() && convertible(*Q) && convertible(*D) &&
               take_slots(args[2], args[3], args[5], *D, &B, &group, &lengths, &ids) && B > 0 && Lq > 0 && T > 0 &&
               here(*Q));
  Tensor out = at::empty({B}, D->options().dtype(at::kFloat));
  const size_t n = fmx_fwd_packed_workspace_bytes(B, Lq, Ld, d);
  const Tensor ws = scratch(n, *D);
  FMX_READY(Q, D, nullptr);
  void* s = stream_of(*Q);
  const int rc = unlocked([&] {
    return fmx_fwd_packed(dtype, Qk.const_data_ptr(), Qk.stride(0), Lq, Dk.const_data_ptr(), Dk.stride(0), T, group,
                          lengths, ids, out.data_ptr<float>(), B, Ld, d, ptr(ws), n, s);
  });
  return rc ? failed(rc) : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// int8_packed(Q [Lq, d] fp16, codes [T, d] uint8, scales [T], mins [T] fp16, tok_group, lengths, max_len, doc_ids)
PyObject* int8_packed(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  FMX_ARGS(8);
  const Tensor *Q = plain(args[0]), *D = plain(args[1]), *sc = plain(args[2]), *mn = plain(args[3]);
  FMX_ORDINARY(Q && D && sc && mn && Q->dim() == 2 && D->dim() == 2 && Q->size(1) == D->size(1) &&
               PyLong_CheckExact(args[6]));
  const int64_t Lq = Q->size(0), d = Q->size(1), T = D->size(0);
  const long max_len = PyLong_AsLong(args[6]);
  if (max_len == -1 && PyErr_Occurred()) return nullptr;
  FMX_ORDINARY(Q->scalar_type() == at::kHalf && D->scalar_type() == at::kByte && is_row_of(sc, at::kHalf, T) &&
               is_row_of(mn, at::kHalf, T) && sc->device() == D->device() && mn->device() == D->device());
  int64_t B;
  const int64_t* group;
  const int32_t *lengths, *ids;
  FMX_ORDINARY(Q->device() == D->device() && rows_ready(*Q) && rows_ready(*D) &&
               take_slots(args[4], args[5], args[7], *D, &B, &group, &lengths, &ids) && B > 0 && Lq > 0 && T > 0 &&
               here(*Q));
  const int64_t Ld = max_len > 1 ? max_len : 1;
  Tensor out = at::empty({B}, D->options().dtype(at::kFloat));
  const size_t n = fmx_fwd_int8_packed_workspace_bytes(B, Lq, Ld, d);
  const Tensor ws = scratch(n, *D);
  void* s = stream_of(*Q);
  const int rc = unlocked([&] {
    return fmx_fwd_int8_packed(Q->const_data_ptr(), Q->stride(0), Lq, D->const_data_ptr<uint8_t>(), D->stride(0),
                               sc->const_data_ptr(), mn->const_data_ptr(), T, group, lengths, ids,
                               out.data_ptr<float>(), B, Ld, d, ptr(ws), n, s);
  });
  return rc ? failed(rc) : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// forward(Q [Nq, Lq, d], D [B, Ld, d], lengths): (scores [Nq, B], argmax [Nq * B, Lq] int32, and Q and D as the
// kernels read them), of training
PyObject* forward(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  FMX_ARGS(3);
  const Tensor *Q = plain(args[0]), *D = plain(args[1]);
  FMX_ORDINARY(Q && D && Q->dim() == 3 && D->dim() == 3 && Q->size(2) == D->size(2));
  const int64_t Nq = Q->size(0), Lq = Q->size(1), d = Q->size(2), B = D->size(0), Ld = D->size(1);
  const int dtype = kernel_dtype(*Q, *D);
  const int32_t* lengths;
  FMX_ORDINARY(dtype >= 0 && Nq > 0 && B > 0 && Lq > 0 && convertible(*Q) && convertible(*D) &&
               Q->device() == D->device() && take_lengths(args[2], B, *D, &lengths) && here(*Q));
  Tensor scores = at::empty({Nq, B}, D->options().dtype(at::kFloat));
  Tensor argmax = at::empty({Nq * B, Lq}, D->options().dtype(at::kInt));
  const size_t n = fmx_fwd_workspace_bytes(Nq, B, Lq, Ld, d);
  const Tensor ws = scratch(n, *D);
  FMX_READY(Q, D, lengths);
  void* s = stream_of(*Q);
  const int rc = unlocked([&] {
    return fmx_fwd(dtype, Qk.const_data_ptr(), Qk.stride(0), Qk.stride(1), Dk.const_data_ptr(), Dk.stride(0),
                   Dk.stride(1), lengths, scores.data_ptr<float>(), B, 1, argmax.data_ptr<int32_t>(), Nq, B, Lq, Ld, d,
                   1, ptr(ws), n, s);
  });
  if (rc) return failed(rc);
  return Py_BuildValue("(NNNN)", THPVariable_Wrap(std::move(scores)), THPVariable_Wrap(std::move(argmax)),
                       THPVariable_Wrap(Qk), THPVariable_Wrap(Dk));
  END_HANDLE_TH_ERRORS
}

// backward(Q, D, lengths, argmax, grad [Nq, B] float32, d, need_q, need_d, f32): (dQ [Nq, Lq, d] or None,
// dD [B, Ld, d] or None), float32 when f32 and the operands are fp16, else in their type
PyObject* backward(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  FMX_ARGS(9);
  const Tensor *Q = plain(args[0]), *D = plain(args[1]), *am = plain(args[3]), *g = plain(args[4]);
  FMX_ORDINARY(Q && D && am && g && Q->dim() == 3 && D->dim() == 3 && g->dim() == 2 && PyLong_CheckExact(args[5]));
  const int64_t d = PyLong_AsLongLong(args[5]);
  const int need_q = PyObject_IsTrue(args[6]), need_d = PyObject_IsTrue(args[7]);
  const int want_f32 = PyObject_IsTrue(args[8]);
  if (PyErr_Occurred()) return nullptr;
  const int64_t Nq = Q->size(0), Lq = Q->size(1), B = D->size(0), Ld = D->size(1);
  const int dtype = kernel_dtype(*Q, *D);
  const int32_t* lengths;
  FMX_ORDINARY(dtype >= 0 && code_of(*Q) == dtype && code_of(*D) == dtype && Nq > 0 && Lq > 0 && B > 0 && Ld > 0 &&
               d > 0 && d <= Q->size(2) && d <= D->size(2) &&
               (need_q || need_d) && rows_ready(*Q) && rows_ready(*D) && is_row_of(am, at::kInt, Nq * B * Lq));
  FMX_ORDINARY(g->scalar_type() == at::kFloat && g->size(0) == Nq && g->size(1) == B && g->stride(0) >= 0 &&
               g->stride(1) >= 0 && Q->device() == D->device() && am->device() == D->device() &&
               g->device() == D->device() && take_lengths(args[2], B, *D, &lengths) && here(*Q));
  Tensor dQ, dD;
  const bool f32 = want_f32 && dtype == FMX_DTYPE_F16;
  const auto options = f32 ? Q->options().dtype(at::kFloat) : Q->options();
  if (need_q) dQ = at::empty({Nq, Lq, d}, options);
  if (need_d) dD = at::empty({B, Ld, d}, options);
  const size_t n = fmx_bwd_batched_workspace_bytes(Nq, B, Lq, Ld, d);
  const Tensor ws = scratch(n, *D);
  void* s = stream_of(*Q);
  const int rc = unlocked([&] {
    if (f32)
      return fmx_bwd_batched_f32(Q->const_data_ptr(), Q->stride(0), Q->stride(1), D->const_data_ptr(), D->stride(0),
                                 D->stride(1), lengths, am->const_data_ptr<int32_t>(), g->const_data_ptr<float>(),
                                 g->stride(0), g->stride(1), static_cast<float*>(ptr(dQ)), static_cast<float*>(ptr(dD)),
                                 Nq, B, Lq, Ld, d, ptr(ws), n, s);
    return fmx_bwd_batched(dtype, Q->const_data_ptr(), Q->stride(0), Q->stride(1), D->const_data_ptr(), D->stride(0),
                           D->stride(1), lengths, am->const_data_ptr<int32_t>(), g->const_data_ptr<float>(),
                           g->stride(0), g->stride(1), ptr(dQ), ptr(dD), Nq, B, Lq, Ld, d, ptr(ws), n, s);
  });
  if (rc) return failed(rc);
  return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(dQ)), THPVariable_Wrap(std::move(dD)));  // undefined: None
  END_HANDLE_TH_ERRORS
}

#define FMX_METHOD(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FMX_METHOD(score),   FMX_METHOD(batched), FMX_METHOD(sparse),
                         FMX_METHOD(topk),    FMX_METHOD(int8),    FMX_METHOD(packed),
                         FMX_METHOD(int8_packed), FMX_METHOD(forward), FMX_METHOD(backward),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
