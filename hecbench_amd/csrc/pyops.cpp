// The operators' host path: checks every tensor against the problem sizes (the C ABI sees raw pointers and
// cannot), allocates what the caller did not pass, makes one library call on the current stream.
//
// What bounds it: nothing but instructions.  Most calls of the library are shorter on the GPU than they used to
// be in Python - 10.5 to 14 us of interpreter and ctypes per call (tensor attribute look-ups 3, stream object 2.8,
// argument conversion 1.5, ...) in front of kernels of 3 to 12 us - so a program that makes one call after the other
// ran at the host's pace.  Here the tensors' own fields are read, and a call costs the launch (2.65 us in the HIP
// runtime, for a kernel of two to four packed arguments), the allocation of its result and 0.3 us.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <climits>
#include <cstdint>
#include <string>

#include "../../include/hq.h"

namespace {

using at::ScalarType;

// ---- errors: a Python exception is set, then python_error unwinds to the method wrapper ---------------------------
[[noreturn]] void raise(PyObject* type, const std::string& text) {
  PyErr_SetString(type, text.c_str());
  throw python_error();
}
[[noreturn]] void value_error(const std::string& text) { raise(PyExc_ValueError, text); }

// hecbench_amd._lib.check(code, where) raises the package's own exception for a library return code
void check_code(int code, const char* where) {
  if (code == HQ_OK) return;
  THPObjectPtr mod(PyImport_ImportModule("hecbench_amd._lib"));
  if (!mod) throw python_error();
  THPObjectPtr r(PyObject_CallMethod(mod.get(), "check", "is", code, where));
  throw python_error();
}

std::string text_of(PyObject* o) {  // steals the reference; an empty text if it cannot be had
  THPObjectPtr obj(o);
  if (!obj) { PyErr_Clear(); return ""; }
  THPObjectPtr s(PyObject_Str(obj.get()));
  const char* c = s ? PyUnicode_AsUTF8(s.get()) : nullptr;
  if (!c) { PyErr_Clear(); return ""; }
  return c;
}

// ---- argument checks -----------------------------------------------------------------------------------------------
constexpr unsigned dt(ScalarType t) { return 1u << (unsigned)t; }
constexpr unsigned kF32 = dt(ScalarType::Float), kF16 = dt(ScalarType::Half), kBF16 = dt(ScalarType::BFloat16),
                   kU8 = dt(ScalarType::Byte), kI8 = dt(ScalarType::Char), kI16 = dt(ScalarType::Short),
                   kI32 = dt(ScalarType::Int), kU32 = dt(ScalarType::UInt32);
static_assert((unsigned)ScalarType::UInt32 < 32, "a dtype set is a 32-bit mask");

std::string names_of(unsigned dtypes) {
  const struct { unsigned bit; const char* name; } all[] = {
      {kF32, "float32"}, {kF16, "float16"}, {kBF16, "bfloat16"}, {kU8, "uint8"},
      {kI8, "int8"},     {kI16, "int16"},   {kI32, "int32"},     {kU32, "uint32"}};
  std::string s;
  for (const auto& d : all)
    if (dtypes & d.bit) s += (s.empty() ? "" : " or ") + std::string(d.name);
  return s;
}

// One tensor argument; null for an optional one that is None.
const at::Tensor* tensor(PyObject* o, const char* name, unsigned dtypes, int64_t numel = -1, bool optional = false) {
  if (o == Py_None) {
    if (optional) return nullptr;
    value_error(std::string(name) + " is required");
  }
  if (!THPVariable_Check(o)) value_error(std::string(name) + " must be a torch tensor");
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!(dtypes & ((unsigned)t.scalar_type() < 32 ? 1u << (unsigned)t.scalar_type() : 0u))) {
    std::string got = text_of(PyObject_GetAttrString(o, "dtype"));
    if (got.rfind("torch.", 0) == 0) got = got.substr(6);
    value_error(std::string(name) + " must be " + names_of(dtypes) + ", got " + got);
  }
  if (numel >= 0 && t.numel() != numel)
    value_error(std::string(name) + " must hold " + std::to_string(numel) + " elements, got " +
                std::to_string(t.numel()) + " (shape " + text_of(PySequence_Tuple(THPObjectPtr(PyObject_GetAttrString(o, "shape")).get())) + ")");
  if (!t.is_contiguous()) value_error(std::string(name) + " must be contiguous");
  return &t;
}

// All tensors on one GPU, which must be the current device (the library launches there).
template <typename... T>
void same_device(const at::Tensor* first, T... rest) {
  const at::Tensor* const ts[] = {first, rest...};
  const c10::Device dev = first->device();
  for (const at::Tensor* t : ts) {
    if (!t) continue;
    if (!t->is_cuda()) value_error("hecbench_amd operators take device tensors only (no CPU path)");
    if (t->device() != dev)
      value_error("tensors on different devices (" + dev.str() + " and " + t->device().str() + ")");
  }
  const int cur = c10::hip::current_device();
  if (dev.index() != cur)
    value_error("tensors live on " + dev.str() + " but the current device is cuda:" + std::to_string(cur));
}

int64_t integer(PyObject* o) {
  int overflow = 0;
  const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
  if (overflow) value_error("an integer argument is out of range");
  if (v == -1 && PyErr_Occurred()) throw python_error();
  return v;
}
int small_integer(PyObject* o, const char* name) {
  const int64_t v = integer(o);
  if (v < INT_MIN || v > INT_MAX) value_error(std::string(name) + " is out of range");
  return (int)v;
}
// A 32-bit value by its low bits, as a C cast takes it: any integer is accepted.
int low_bits(PyObject* o) {
  const unsigned long long v = PyLong_AsUnsignedLongLongMask(o);
  if (v == (unsigned long long)-1 && PyErr_Occurred()) throw python_error();
  return (int)(unsigned)v;
}
// A bound that is compared with 32-bit numbers: beyond their range the nearest of them compares alike.
int bound(PyObject* o) {
  int overflow = 0;
  const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
  if (v == -1 && !overflow && PyErr_Occurred()) throw python_error();
  if (overflow > 0 || v > INT_MAX) return INT_MAX;
  if (overflow < 0 || v < INT_MIN) return INT_MIN;
  return (int)v;
}
// problem sizes are C ints at the boundary
int size_of(int64_t v) {
  if (v > INT_MAX) check_code(HQ_ERR_TOO_LARGE, "hecbench_amd");
  return (int)v;
}
float real(PyObject* o) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) throw python_error();
  return (float)v;
}

int act_dtype(const at::Tensor& t) {
  return t.scalar_type() == ScalarType::Float ? HQ_DTYPE_F32
         : t.scalar_type() == ScalarType::Half ? HQ_DTYPE_F16 : HQ_DTYPE_BF16;
}

const void* ptr(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }
template <typename T> const T* in(const at::Tensor* t) { return static_cast<const T*>(ptr(t)); }
template <typename T> T* to(const at::Tensor& t) { return static_cast<T*>(t.data_ptr()); }

void* stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

// The result tensor: the caller's own (returned as the same object) or a new one on the device of `like`.
struct Result {
  PyObject* given;
  at::Tensor t;
  Result(PyObject* o, const at::Tensor* checked, const at::Tensor& like, at::IntArrayRef shape, ScalarType type)
      : given(checked ? o : nullptr),
        t(checked ? *checked : at::Tensor(at::detail::empty_cuda(shape, type, like.device(), std::nullopt))) {}
  PyObject* release() {
    if (given) { Py_INCREF(given); return given; }
    return THPVariable_Wrap(std::move(t));
  }
};

at::Tensor fresh(at::IntArrayRef shape, ScalarType type, const at::Tensor& like) {
  return at::Tensor(at::detail::empty_cuda(shape, type, like.device(), std::nullopt));
}

// The library call without the interpreter lock, as other threads may issue work on their own streams meanwhile.
template <typename F>
void call(const char* where, F f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  Py_END_ALLOW_THREADS
  check_code(rc, where);
}

// ---- operators (positional arguments; names and defaults live in ops.py) ----------------------------------------------
PyObject* q3_matvec(PyObject* const* a) {  // x, qweight, scales, zeros, out, accumulate
  const at::Tensor* x = tensor(a[0], "x", kF32 | kF16);
  const at::Tensor* w = tensor(a[1], "qweight", kI32);
  if (w->dim() != 2) value_error("qweight must be [3*K/32][N]");
  const int64_t K = x->numel(), N = w->size(1);
  if (w->size(0) * 32 != 3 * K) value_error("qweight must have 3*K/32 packed rows");
  const at::Tensor* s = tensor(a[2], "scales", kF32, N);
  const at::Tensor* z = tensor(a[3], "zeros", kF32, N);
  const at::Tensor* o = tensor(a[4], "out", kF32, N, true);
  same_device(x, w, s, z, o);
  const int accumulate = PyObject_IsTrue(a[5]);
  if (accumulate < 0) throw python_error();
  Result r(a[4], o, *x, {N}, ScalarType::Float);
  const int k = size_of(K), n = size_of(N);
  void* st = stream();
  call("hq_q3_matvec", [&] {
    return hq_q3_matvec(ptr(x), act_dtype(*x), in<int32_t>(w), in<float>(s), in<float>(z), to<float>(r.t), k, n, 1,
                        accumulate ? HQ_FLAG_ACCUMULATE : 0u, st);
  });
  return r.release();
}

PyObject* q3_gemm(PyObject* const* a) {  // A, qweight, scales, zeros, out
  const at::Tensor* x = tensor(a[0], "A", kF16);
  const at::Tensor* w = tensor(a[1], "qweight", kI32);
  if (x->dim() != 2 || w->dim() != 2) value_error("A must be [M][K] and qweight [3*K/32][N]");
  const int64_t M = x->size(0), K = x->size(1), N = w->size(1);
  if (w->size(0) * 32 != 3 * K) value_error("qweight must have 3*K/32 packed rows");
  const at::Tensor* s = tensor(a[2], "scales", kF32, N);
  const at::Tensor* z = tensor(a[3], "zeros", kF32, N);
  const at::Tensor* o = tensor(a[4], "out", kF32, M * N, true);
  same_device(x, w, s, z, o);
  Result r(a[4], o, *x, {M, N}, ScalarType::Float);
  const int m = size_of(M), k = size_of(K), n = size_of(N);
  void* st = stream();
  call("hq_q3_matvec(batch)", [&] {
    return hq_q3_matvec(ptr(x), HQ_DTYPE_F16, in<int32_t>(w), in<float>(s), in<float>(z), to<float>(r.t), k, n, m, 0u, st);
  });
  return r.release();
}

PyObject* dequant_4bit(PyObject* const* a) {  // packed, absmax, n_elems, blocksize, table, out
  const int64_t n = integer(a[2]);
  const int bs = small_integer(a[3], "blocksize"), table = low_bits(a[4]);
  if (n < 0 || bs <= 0) value_error("n_elems must be >= 0 and blocksize > 0");
  const at::Tensor* p = tensor(a[0], "packed", kU8, n / 2 + (n & 1));
  const at::Tensor* am = tensor(a[1], "absmax", kF32, n / bs + (n % bs != 0));
  const at::Tensor* o = tensor(a[5], "out", kF16, n, true);
  same_device(p, am, o);
  Result r(a[5], o, *p, {n}, ScalarType::Half);
  void* st = stream();
  call("hq_dequant_nf4", [&] { return hq_dequant_nf4(in<uint8_t>(p), in<float>(am), r.t.data_ptr(), n, bs, table, st); });
  return r.release();
}

PyObject* quantize_4bit(PyObject* const* a) {  // x, blocksize, table
  const at::Tensor* x = tensor(a[0], "x", kF32 | kF16);
  const int bs = small_integer(a[1], "blocksize"), table = low_bits(a[2]);
  if (bs <= 0) value_error("blocksize must be > 0");
  same_device(x);
  const int64_t n = x->numel();
  at::Tensor packed = fresh({n / 2 + (n & 1)}, ScalarType::Byte, *x);
  at::Tensor absmax = fresh({n / bs + (n % bs != 0)}, ScalarType::Float, *x);
  void* st = stream();
  call("hq_quantize_4bit", [&] {
    return hq_quantize_4bit(ptr(x), act_dtype(*x), to<uint8_t>(packed), to<float>(absmax), n, bs, table, st);
  });
  THPObjectPtr p(THPVariable_Wrap(std::move(packed))), m(THPVariable_Wrap(std::move(absmax)));
  return PyTuple_Pack(2, p.get(), m.get());
}

PyObject* quantize_dynamic8(PyObject* const* a) {  // code, A, out
  const at::Tensor* code = tensor(a[0], "code", kF32, 256);
  const at::Tensor* x = tensor(a[1], "A", kF32);
  const at::Tensor* o = tensor(a[2], "out", kU8, x->numel(), true);
  same_device(code, x, o);
  Result r(a[2], o, *x, {x->numel()}, ScalarType::Byte);
  void* st = stream();
  call("hq_quantize_dynamic8",
       [&] { return hq_quantize_dynamic8(in<float>(code), in<float>(x), to<uint8_t>(r.t), x->numel(), st); });
  return r.release();
}

PyObject* lut_matmul(PyObject* const* a) {  // x, bW, alpha, q_bias, group_size, out
  const at::Tensor* x = tensor(a[0], "x", kF16);
  const at::Tensor* w = tensor(a[1], "bW", kI32 | kU32);
  if (w->dim() != 3) value_error("bW must be [K/32][nbits][N]");
  const int64_t K = x->numel(), nb = w->size(1), N = w->size(2), G = integer(a[4]);
  if (G <= 0 || K % G || w->size(0) * 32 != K) value_error("bW must have K/32 packed rows and group_size must divide K");
  const at::Tensor* al = tensor(a[2], "alpha", kF16, K / G * nb * N);
  const at::Tensor* qb = tensor(a[3], "q_bias", kF16, K / G * N, true);
  const at::Tensor* o = tensor(a[5], "out", kF16, N, true);
  same_device(x, w, al, qb, o);
  Result r(a[5], o, *x, {N}, ScalarType::Half);
  const int k = size_of(K), n = size_of(N), b = size_of(nb), g = size_of(G);
  void* st = stream();
  call("hq_lut_gemv",
       [&] { return hq_lut_gemv(in<uint32_t>(w), ptr(al), ptr(qb), ptr(x), r.t.data_ptr(), k, n, b, g, st); });
  return r.release();
}

PyObject* code1x16_matvec(PyObject* const* a) {  // codes, x, codebooks, codebook_a_sizes, codebook_stride_int4, scales, out
  const at::Tensor* c = tensor(a[0], "codes", kI16);
  const at::Tensor* x = tensor(a[1], "x", kF16);
  if (c->dim() != 2) value_error("codes must be [M][K/8]");
  const int64_t M = c->size(0), K = x->numel();
  if (c->size(1) * 8 != K) value_error("codes must hold K/8 codes per row");
  THPObjectPtr bounds(PySequence_Fast(a[3], "codebook_a_sizes must be a sequence"));
  if (!bounds) throw python_error();
  if (PySequence_Fast_GET_SIZE(bounds.get()) != 4) value_error("codebook_a_sizes must hold four row bounds");
  int sizes[4];
  for (int j = 0; j < 4; ++j) sizes[j] = bound(PySequence_Fast_GET_ITEM(bounds.get(), j));
  int ncb = 0;  // code book of the last row: the first j with M-1 < codebook_a_sizes[j], the fifth where there is none
  while (ncb < 4 && M - 1 >= sizes[ncb]) ++ncb;
  ++ncb;
  // one code book: no row goes by the stride
  const int stride = ncb == 1 ? low_bits(a[4]) : small_integer(a[4], "codebook_stride_int4");
  const at::Tensor* cb = tensor(a[2], "codebooks", kF16);
  if (cb->numel() < (int64_t)(ncb - 1) * stride * 8 + 65536 * 8)
    value_error("codebooks too small for " + std::to_string(ncb) + " code book(s) of 65536 x 8 halves at the given stride");
  const at::Tensor* s = tensor(a[5], "scales", kF16, M, true);
  const at::Tensor* o = tensor(a[6], "out", kF16, M, true);
  same_device(c, x, cb, s, o);
  Result r(a[6], o, *x, {M}, ScalarType::Half);
  const int m = size_of(M), k = size_of(K);
  void* st = stream();
  call("hq_aqlm_matvec", [&] {
    return hq_aqlm_matvec(in<int16_t>(c), ptr(cb), ptr(s), ptr(x), r.t.data_ptr(), m, k, sizes, stride, st);
  });
  return r.release();
}

PyObject* q3_pack(PyObject* const* a) {  // codes
  const at::Tensor* c = tensor(a[0], "codes", kU8);
  if (c->dim() != 2 || c->size(0) % 32) value_error("codes must be [K][N] with K a multiple of 32");
  same_device(c);
  const int64_t K = c->size(0), N = c->size(1);
  at::Tensor w = fresh({3 * K / 32, N}, ScalarType::Int, *c);
  const int k = size_of(K), n = size_of(N);
  void* st = stream();
  call("hq_q3_pack", [&] { return hq_q3_pack(in<uint8_t>(c), to<int32_t>(w), k, n, st); });
  return THPVariable_Wrap(std::move(w));
}

PyObject* bcq_pack(PyObject* const* a) {  // signs
  const at::Tensor* s = tensor(a[0], "signs", kI8);
  if (s->dim() != 3 || s->size(0) % 32) value_error("signs must be [K][nbits][N] with K a multiple of 32");
  same_device(s);
  const int64_t K = s->size(0), nb = s->size(1), N = s->size(2);
  at::Tensor w = fresh({K / 32, nb, N}, ScalarType::Int, *s);
  const int k = size_of(K), n = size_of(N), b = size_of(nb);
  void* st = stream();
  call("hq_bcq_pack", [&] { return hq_bcq_pack(in<int8_t>(s), reinterpret_cast<uint32_t*>(to<int32_t>(w)), k, n, b, st); });
  return THPVariable_Wrap(std::move(w));
}

PyObject* int8_quant_static(PyObject* const* a) {  // x, scale, azp, out
  const at::Tensor* x = tensor(a[0], "x", kF32 | kF16 | kBF16);
  if (x->dim() != 2) value_error("x must be [tokens][hidden]");
  const at::Tensor* o = tensor(a[3], "out", kI8, x->numel(), true);
  same_device(x, o);
  const float scale = real(a[1]);
  const bool has_azp = a[2] != Py_None;
  const int azp = has_azp ? low_bits(a[2]) : 0;
  const int64_t tokens = x->size(0), hidden = x->size(1);
  Result r(a[3], o, *x, {tokens, hidden}, ScalarType::Char);
  const int h = size_of(hidden);
  void* st = stream();
  call("hq_int8_quant_static",
       [&] { return hq_int8_quant_static(ptr(x), act_dtype(*x), to<int8_t>(r.t), tokens, h, scale, has_azp, azp, st); });
  return r.release();
}

PyObject* int8_quant_dynamic(PyObject* const* a) {  // x, with_azp, out
  const at::Tensor* x = tensor(a[0], "x", kF32 | kF16 | kBF16);
  if (x->dim() != 2) value_error("x must be [tokens][hidden]");
  const at::Tensor* o = tensor(a[2], "out", kI8, x->numel(), true);
  same_device(x, o);
  const int with_azp = PyObject_IsTrue(a[1]);
  if (with_azp < 0) throw python_error();
  const int64_t tokens = x->size(0), hidden = x->size(1);
  Result r(a[2], o, *x, {tokens, hidden}, ScalarType::Char);
  at::Tensor scales = fresh({tokens}, ScalarType::Float, *x), azp;
  if (with_azp) azp = fresh({tokens}, ScalarType::Int, *x);
  const int h = size_of(hidden);
  void* st = stream();
  call("hq_int8_quant_dynamic", [&] {
    return hq_int8_quant_dynamic(ptr(x), act_dtype(*x), to<int8_t>(r.t), to<float>(scales),
                                 with_azp ? to<int32_t>(azp) : nullptr, tokens, h, st);
  });
  THPObjectPtr q(r.release()), s(THPVariable_Wrap(std::move(scales))), z;
  if (with_azp) z = THPVariable_Wrap(std::move(azp));
  return PyTuple_Pack(3, q.get(), s.get(), with_azp ? z.get() : Py_None);
}

PyObject* gemv_fp16(PyObject* const* a) {  // mat, vec, out
  const at::Tensor* m = tensor(a[0], "mat", kF16);
  if (m->dim() != 2) value_error("mat must be [rows][n]");
  const int64_t rows = m->size(0), n = m->size(1);
  const at::Tensor* v = tensor(a[1], "vec", kF16, n);
  const at::Tensor* o = tensor(a[2], "out", kF16, rows, true);
  same_device(m, v, o);
  Result r(a[2], o, *m, {rows}, ScalarType::Half);
  const int ri = size_of(rows), ni = size_of(n);
  void* st = stream();
  call("hq_gemv_fp16", [&] { return hq_gemv_fp16(ptr(m), ptr(v), r.t.data_ptr(), ri, ni, st); });
  return r.release();
}

template <bool INT4>
PyObject* gemv_int(PyObject* const* a) {  // mat, vec, scale, zero_point, out
  const at::Tensor* m = tensor(a[0], "mat", INT4 ? kU8 : kI8);
  if (m->dim() != 2) value_error(INT4 ? "mat must be [rows][n/2]" : "mat must be [rows][n]");
  const int64_t rows = m->size(0), n = m->size(1) * (INT4 ? 2 : 1);
  const at::Tensor* v = tensor(a[1], "vec", kF16, n);
  const at::Tensor* o = tensor(a[4], "out", kF16, rows, true);
  same_device(m, v, o);
  const float scale = real(a[2]), zero = real(a[3]);
  Result r(a[4], o, *m, {rows}, ScalarType::Half);
  const int ri = size_of(rows), ni = size_of(n);
  void* st = stream();
  call(INT4 ? "hq_gemv_int4" : "hq_gemv_int8", [&] {
    return INT4 ? hq_gemv_int4(in<uint8_t>(m), ptr(v), r.t.data_ptr(), ri, ni, scale, zero, st)
                : hq_gemv_int8(in<int8_t>(m), ptr(v), r.t.data_ptr(), ri, ni, scale, zero, st);
  });
  return r.release();
}

PyObject* mxfp4_qdq(PyObject* const* a) {  // x, out
  if (THPVariable_Check(a[0])) {
    const ScalarType t = THPVariable_Unpack(a[0]).scalar_type();
    if (t != ScalarType::Half && t != ScalarType::BFloat16) raise(PyExc_TypeError, "mxfp4_qdq takes fp16 or bf16 tensors");
  }
  const at::Tensor* x = tensor(a[0], "x", kF16 | kBF16);
  const at::Tensor* o = tensor(a[1], "out", dt(x->scalar_type()), x->numel(), true);
  same_device(x, o);
  Result r(a[1], o, *x, x->sizes(), x->scalar_type());
  void* st = stream();
  call("hq_mxfp4_qdq", [&] { return hq_mxfp4_qdq(ptr(x), r.t.data_ptr(), x->numel(), act_dtype(*x), st); });
  return r.release();
}

// ---- the module ------------------------------------------------------------------------------------------------------
template <PyObject* (*F)(PyObject* const*), int NARGS>
PyObject* method(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != NARGS) raise(PyExc_TypeError, "wrong number of arguments (the wrappers in hecbench_amd/ops.py are the interface)");
  return F(args);
  END_HANDLE_TH_ERRORS
}
#define HQ_METHOD(name, fn, nargs) {name, (PyCFunction)(void (*)(void)) & method<fn, nargs>, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    HQ_METHOD("q3_matvec", q3_matvec, 6),
    HQ_METHOD("q3_gemm", q3_gemm, 5),
    HQ_METHOD("dequant_4bit", dequant_4bit, 6),
    HQ_METHOD("quantize_4bit", quantize_4bit, 3),
    HQ_METHOD("quantize_dynamic8", quantize_dynamic8, 3),
    HQ_METHOD("lut_matmul", lut_matmul, 6),
    HQ_METHOD("code1x16_matvec", code1x16_matvec, 7),
    HQ_METHOD("q3_pack", q3_pack, 1),
    HQ_METHOD("bcq_pack", bcq_pack, 1),
    HQ_METHOD("int8_quant_static", int8_quant_static, 4),
    HQ_METHOD("int8_quant_dynamic", int8_quant_dynamic, 3),
    HQ_METHOD("gemv_fp16", gemv_fp16, 3),
    HQ_METHOD("gemv_int8", gemv_int<false>, 5),
    HQ_METHOD("gemv_int4", gemv_int<true>, 5),
    HQ_METHOD("mxfp4_qdq", mxfp4_qdq, 2),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_ops", "Host path of the operators over libhq.", -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__ops(void) { return PyModule_Create(&kModule); }
