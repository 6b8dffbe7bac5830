// Native call path of the Python entry points (CPython extension dsl_fast).
//
// At decode sizes a layer's kernels take about 10 us while each Python
// wrapper (shape checks, output allocation, device context, stream lookup,
// ctypes marshalling) took about 12 us a call, so the GPU waited for the
// host.  These functions do the same work natively for well-formed calls:
// they check that the operands are exactly what the C ABI reads in place,
// allocate the outputs, and call it on the current stream.  Anything else --
// another dtype, layout, device mix, shape mismatch, tensor subclass, empty
// operand -- returns None, and the Python function goes on with its own
// checks, copies and errors; a status from the C ABI also returns None, so the
// Python path repeats the call and raises it.  Nothing is kept between calls.
// A call costs about 1.5 us beside its launches (ctypes path: about 9).
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include "dsl_gemm.h"

namespace {

using at::ScalarType;
using at::Tensor;

// the plain tensor of a Python object (exactly torch.Tensor or Parameter), on
// a GPU, or nullptr
const Tensor *gpu_tensor(PyObject *o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor &t = THPVariable_Unpack(o);
  if (!t.defined() || t.device().type() != at::DeviceType::CUDA || t.layout() != at::kStrided)
    return nullptr;
  return &t;
}

bool aligned16(const Tensor &t) { return (reinterpret_cast<uintptr_t>(t.const_data_ptr()) & 15) == 0; }

// contiguous, 16-byte aligned, not empty
bool plain(const Tensor &t, int64_t dim) {
  return t.dim() == dim && t.numel() > 0 && t.is_contiguous() && aligned16(t);
}

bool is_codes(const Tensor &t) {
  return t.scalar_type() == ScalarType::Byte || t.scalar_type() == ScalarType::Float8_e4m3fn;
}

bool is_scales(const Tensor &t, ScalarType dt) {
  return t.scalar_type() == dt && t.numel() > 0 && t.is_contiguous();
}

// bf16 rows with unit column stride and a row stride of whole 16-byte chunks
bool bf16_rows(const Tensor &t) {
  return t.dim() == 2 && t.numel() > 0 && t.scalar_type() == ScalarType::BFloat16 &&
         t.stride(1) == 1 && t.stride(0) >= t.size(1) && t.stride(0) % 8 == 0 && aligned16(t);
}

// output dtype code of a torch.dtype, or -1
int out_code(PyObject *o) {
  if (!THPDtype_Check(o)) return -1;
  const ScalarType s = reinterpret_cast<THPDtype *>(o)->scalar_type;
  return s == ScalarType::BFloat16 ? DSL_OUT_BF16 : (s == ScalarType::Float ? DSL_OUT_F32 : -1);
}

Tensor empty(at::IntArrayRef shape, ScalarType dt, const Tensor &like) {
  return at::empty(shape, at::TensorOptions().dtype(dt).device(like.device()));
}
Tensor bytes(int64_t n, const Tensor &like) { return empty({n}, ScalarType::Byte, like); }
Tensor out_matrix(int64_t m, int64_t n, int code, const Tensor &like) {
  return empty({m, n}, code == DSL_OUT_F32 ? ScalarType::Float : ScalarType::BFloat16, like);
}

void *stream_of(const Tensor &t) {
  return c10::hip::getCurrentHIPStream(t.device().index()).stream();
}

template <class T = void>
T *ptr(const Tensor &t) {
  return static_cast<T *>(t.data_ptr());
}

PyObject *none() { Py_RETURN_NONE; }

PyObject *pack(std::initializer_list<Tensor> ts) {
  PyObject *r = PyTuple_New((Py_ssize_t)ts.size());
  if (!r) return nullptr;
  Py_ssize_t i = 0;
  for (const Tensor &t : ts) PyTuple_SET_ITEM(r, i++, THPVariable_Wrap(t));
  return r;
}

// Work without the GIL on `dev`'s device; false: leave the call to Python.
template <class F>
bool on_device(const Tensor &dev, F &&f) {
  pybind11::gil_scoped_release no_gil;
  const c10::DeviceGuard guard(dev.device());
  return f();
}

// ------------------------------------------------------------- quantize --
// bf16 / fp32 matrix with positive strides, not empty
const Tensor *quant_source(PyObject *o, int *dt) {
  const Tensor *x = gpu_tensor(o);
  if (!x || x->dim() != 2 || x->numel() == 0 || x->stride(0) <= 0 || x->stride(1) <= 0) return nullptr;
  if (x->scalar_type() == ScalarType::BFloat16) *dt = DSL_IN_BF16;
  else if (x->scalar_type() == ScalarType::Float) *dt = DSL_IN_F32;
  else return nullptr;
  return x;
}

PyObject *quant_fp8_tensor(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int dt;
  const Tensor *x = n == 1 ? quant_source(a[0], &dt) : nullptr;
  if (!x) return none();
  Tensor q, s;
  const bool ok = on_device(*x, [&] {
    const int64_t r = x->size(0), c = x->size(1);
    const size_t nb = dsl_quant_workspace_bytes(r, c);
    q = empty({r, c}, ScalarType::Byte, *x);
    s = empty({1}, ScalarType::Float, *x);
    const Tensor ws = bytes((int64_t)nb, *x);
    return dsl_quant_fp8_tensor(ptr(*x), r, c, x->stride(0), x->stride(1), dt, ptr<uint8_t>(q),
                                ptr<float>(s), ptr(ws), nb, stream_of(*x)) == DSL_OK;
  });
  return ok ? pack({q, s}) : none();
  END_HANDLE_TH_ERRORS
}

PyObject *quant_fp8_blocks(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int dt;
  const Tensor *x = n == 3 && PyLong_CheckExact(a[1]) && PyLong_CheckExact(a[2]) ? quant_source(a[0], &dt)
                                                                                 : nullptr;
  if (!x) return none();
  int over1 = 0, over2 = 0;
  const long long gr = PyLong_AsLongLongAndOverflow(a[1], &over1);
  const long long gc = PyLong_AsLongLongAndOverflow(a[2], &over2);
  if (over1 || over2 || gr <= 0 || gc <= 0) return none();
  Tensor q, s;
  const bool ok = on_device(*x, [&] {
    const int64_t r = x->size(0), c = x->size(1);
    q = empty({r, c}, ScalarType::Byte, *x);
    s = empty({(r - 1) / gr + 1, (c - 1) / gc + 1}, ScalarType::Float, *x);
    return dsl_quant_fp8_blocks(ptr(*x), r, c, x->stride(0), x->stride(1), dt, gr, gc, ptr<uint8_t>(q),
                                ptr<float>(s), stream_of(*x)) == DSL_OK;
  });
  return ok ? pack({q, s}) : none();
  END_HANDLE_TH_ERRORS
}

// the view of [G, K, N] storage as [G, N, K], one scale per row
PyObject *quant_fp8_rows_batched(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Tensor *w = n == 1 ? gpu_tensor(a[0]) : nullptr;
  if (!w || w->dim() != 3 || w->numel() == 0 || w->stride(1) != 1 || w->stride(2) < w->size(1) ||
      w->stride(0) <= 0 || w->size(0) > 65535)
    return none();
  const bool bf16 = w->scalar_type() == ScalarType::BFloat16;
  if (!bf16 && w->scalar_type() != ScalarType::Float) return none();
  Tensor q, s;
  const bool ok = on_device(*w, [&] {
    const int64_t g = w->size(0), r = w->size(1), c = w->size(2);
    q = empty({g * r, c}, ScalarType::Byte, *w);
    s = empty({g * r, 1}, ScalarType::Float, *w);
    return dsl_quant_fp8_rows_batched(ptr(*w), g, r, c, w->stride(0), w->stride(2),
                                      bf16 ? DSL_IN_BF16 : DSL_IN_F32, ptr<uint8_t>(q), ptr<float>(s),
                                      stream_of(*w)) == DSL_OK;
  });
  return ok ? pack({q, s}) : none();
  END_HANDLE_TH_ERRORS
}

PyObject *quant_mxfp4(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int dt;
  const Tensor *x = n == 1 ? quant_source(a[0], &dt) : nullptr;
  if (!x || x->size(1) % 32 != 0) return none();
  Tensor q, s;
  const bool ok = on_device(*x, [&] {
    const int64_t r = x->size(0), c = x->size(1);
    q = empty({r, c / 2}, ScalarType::Byte, *x);
    s = empty({r, c / 32}, ScalarType::Byte, *x);
    return dsl_quant_mxfp4(ptr(*x), r, c, x->stride(0), x->stride(1), dt, ptr<uint8_t>(q),
                           ptr<uint8_t>(s), stream_of(*x)) == DSL_OK;
  });
  return ok ? pack({q, s}) : none();
  END_HANDLE_TH_ERRORS
}

PyObject *quant_nvfp4(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int dt;
  const Tensor *x = n == 1 ? quant_source(a[0], &dt) : nullptr;
  if (!x || x->size(1) % 16 != 0) return none();
  Tensor q, s, g;
  const bool ok = on_device(*x, [&] {
    const int64_t r = x->size(0), c = x->size(1);
    const size_t nb = dsl_quant_workspace_bytes(r, c);
    q = empty({r, c / 2}, ScalarType::Byte, *x);
    s = empty({r, c / 16}, ScalarType::Byte, *x);
    g = empty({1}, ScalarType::Float, *x);
    const Tensor ws = bytes((int64_t)nb, *x);
    return dsl_quant_nvfp4(ptr(*x), r, c, x->stride(0), x->stride(1), dt, ptr<uint8_t>(q),
                           ptr<uint8_t>(s), ptr<float>(g), ptr(ws), nb, stream_of(*x)) == DSL_OK;
  });
  return ok ? pack({q, s, g}) : none();
  END_HANDLE_TH_ERRORS
}

// ----------------------------------------------------------------- GEMM --
// fp8_gemm(qa, qw, scale_a, scale_b, scale_mode, out_dtype)
PyObject *fp8_gemm(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) return none();
  const Tensor *qa = gpu_tensor(a[0]), *qw = gpu_tensor(a[1]), *sa = gpu_tensor(a[2]), *sb = gpu_tensor(a[3]);
  const int code = out_code(a[5]);
  if (!qa || !qw || !sa || !sb || code < 0 || !PyLong_CheckExact(a[4])) return none();
  const int mode = (int)PyLong_AsLong(a[4]);
  if (!is_codes(*qa) || !is_codes(*qw) || !plain(*qa, 2) || !plain(*qw, 2) ||
      qa->size(1) != qw->size(1) || !is_scales(*sa, ScalarType::Float) ||
      !is_scales(*sb, ScalarType::Float) || qw->device() != qa->device() ||
      sa->device() != qa->device() || sb->device() != qa->device())
    return none();
  const int64_t m = qa->size(0), nn = qw->size(0), k = qa->size(1), g = (k + 127) / 128;
  if (mode == DSL_SCALE_TENSOR) {
    if (sa->numel() != 1 || sb->numel() != 1) return none();
  } else {
    if (sa->dim() != 2 || sb->dim() != 2 || sa->size(0) != m || sa->size(1) != g) return none();
    const bool block = mode == DSL_SCALE_BLOCK128;
    if (sb->size(0) != (block ? (nn + 127) / 128 : g) || sb->size(1) != (block ? g : nn)) return none();
  }
  Tensor c;
  const bool ok = on_device(*qa, [&] {
    const size_t nb = dsl_gemm_workspace_bytes(DSL_OP_FP8, m, nn, k);
    c = out_matrix(m, nn, code, *qa);
    Tensor ws;
    if (nb) ws = bytes((int64_t)nb, *qa);
    return dsl_fp8_gemm(ptr<uint8_t>(*qa), ptr<uint8_t>(*qw), ptr(c), m, nn, k, nn, code, mode,
                        ptr<float>(*sa), ptr<float>(*sb), nb ? ptr(ws) : nullptr, nb,
                        stream_of(*qa)) == DSL_OK;
  });
  return ok ? THPVariable_Wrap(c) : none();
  END_HANDLE_TH_ERRORS
}

// fp4_gemm(qa, sa, qw, sw, fmt, global_a, global_w, out_dtype); the globals
// 1-element fp32 tensors (NVFP4) or None
PyObject *fp4_gemm(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8 || !PyLong_CheckExact(a[4])) return none();
  const Tensor *qa = gpu_tensor(a[0]), *sa = gpu_tensor(a[1]), *qw = gpu_tensor(a[2]), *sw = gpu_tensor(a[3]);
  const int code = out_code(a[7]), fmt = (int)PyLong_AsLong(a[4]);
  if (!qa || !qw || !sa || !sw || code < 0) return none();
  const int64_t blk = fmt == DSL_FMT_MXFP4 ? 32 : 16;
  if (qa->scalar_type() != ScalarType::Byte || qw->scalar_type() != ScalarType::Byte || !plain(*qa, 2) ||
      !plain(*qw, 2) || qa->size(1) != qw->size(1) || !is_scales(*sa, ScalarType::Byte) ||
      !is_scales(*sw, ScalarType::Byte) || sa->dim() != 2 || sw->dim() != 2 ||
      qw->device() != qa->device() || sa->device() != qa->device() || sw->device() != qa->device())
    return none();
  const int64_t m = qa->size(0), nn = qw->size(0), k = 2 * qa->size(1);
  if (sa->size(0) != m || sw->size(0) != nn || sa->size(1) != k / blk || sw->size(1) != k / blk) return none();
  const Tensor *ga = nullptr, *gw = nullptr;
  if (fmt == DSL_FMT_NVFP4) {
    ga = gpu_tensor(a[5]);
    gw = gpu_tensor(a[6]);
    if (!ga || !gw || !is_scales(*ga, ScalarType::Float) || !is_scales(*gw, ScalarType::Float) ||
        ga->numel() != 1 || gw->numel() != 1 || ga->device() != qa->device() || gw->device() != qa->device())
      return none();
  } else if (a[5] != Py_None || a[6] != Py_None) {
    return none();
  }
  Tensor c;
  const bool ok = on_device(*qa, [&] {
    const size_t nb = dsl_gemm_workspace_bytes(DSL_OP_FP4, m, nn, k);
    c = out_matrix(m, nn, code, *qa);
    Tensor ws;
    if (nb) ws = bytes((int64_t)nb, *qa);
    return dsl_fp4_gemm(ptr<uint8_t>(*qa), ptr<uint8_t>(*qw), ptr(c), m, nn, k, nn, code, fmt,
                        ptr<uint8_t>(*sa), ptr<uint8_t>(*sw), ga ? ptr<float>(*ga) : nullptr,
                        gw ? ptr<float>(*gw) : nullptr, nb ? ptr(ws) : nullptr, nb,
                        stream_of(*qa)) == DSL_OK;
  });
  return ok ? THPVariable_Wrap(c) : none();
  END_HANDLE_TH_ERRORS
}

// b [K, N] is the transpose view of contiguous, aligned [N, K] storage
bool k_major_view(const Tensor &b) {
  return b.dim() == 2 && b.numel() > 0 && aligned16(b) && b.t().is_contiguous();
}

// bf16_gemm(A, B, out_dtype)
PyObject *bf16_gemm(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) return none();
  const Tensor *x = gpu_tensor(a[0]), *b = gpu_tensor(a[1]);
  const int code = out_code(a[2]);
  if (!x || !b || code < 0 || x->scalar_type() != ScalarType::BFloat16 ||
      b->scalar_type() != ScalarType::BFloat16 || !plain(*x, 2) || !k_major_view(*b) ||
      x->size(1) != b->size(0) || b->device() != x->device())
    return none();
  const int64_t m = x->size(0), k = x->size(1), nn = b->size(1);
  Tensor c;
  const bool ok = on_device(*x, [&] {
    const size_t nb = dsl_gemm_workspace_bytes(DSL_OP_BF16, m, nn, k);
    c = out_matrix(m, nn, code, *x);
    Tensor ws;
    if (nb) ws = bytes((int64_t)nb, *x);
    return dsl_bf16_gemm(ptr(*x), ptr(*b), ptr(c), m, nn, k, nn, code, nb ? ptr(ws) : nullptr, nb,
                         stream_of(*x)) == DSL_OK;
  });
  return ok ? THPVariable_Wrap(c) : none();
  END_HANDLE_TH_ERRORS
}

// grouped_fp8_gemm(qx, sx, qw, sw, offsets, out_dtype)
PyObject *grouped_fp8_gemm(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 6) return none();
  const Tensor *qx = gpu_tensor(a[0]), *sx = gpu_tensor(a[1]), *qw = gpu_tensor(a[2]),
               *sw = gpu_tensor(a[3]), *off = gpu_tensor(a[4]);
  const int code = out_code(a[5]);
  if (!qx || !sx || !qw || !sw || !off || code < 0) return none();
  if (!is_codes(*qx) || !is_codes(*qw) || !plain(*qx, 2) || !plain(*qw, 3) ||
      qx->size(1) != qw->size(2) || !is_scales(*sx, ScalarType::Float) ||
      !is_scales(*sw, ScalarType::Float) || !is_scales(*off, ScalarType::Int) || off->dim() != 1)
    return none();
  const at::Device d = qx->device();
  if (sx->device() != d || qw->device() != d || sw->device() != d || off->device() != d) return none();
  const int64_t t = qx->size(0), k = qx->size(1), g = qw->size(0), nn = qw->size(1);
  if (off->numel() != g + 1 || sx->numel() != t || sw->numel() != g * nn) return none();
  Tensor y;
  const bool ok = on_device(*qx, [&] {
    y = out_matrix(t, nn, code, *qx);
    return dsl_grouped_fp8_gemm(ptr<uint8_t>(*qx), ptr<uint8_t>(*qw), ptr(y), ptr<int32_t>(*off), g, t,
                                nn, k, nn, code, ptr<float>(*sx), ptr<float>(*sw),
                                stream_of(*qx)) == DSL_OK;
  });
  return ok ? THPVariable_Wrap(y) : none();
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------ producers --
void producer_outputs(int64_t r, int64_t c, int qfmt, const Tensor &x, Tensor *q, Tensor *s) {
  if (qfmt == DSL_QFMT_FP8_G128) {
    *q = empty({r, c}, ScalarType::Byte, x);
    *s = empty({r, (c + 127) / 128}, ScalarType::Float, x);
  } else {
    *q = empty({r, c / 2}, ScalarType::Byte, x);
    *s = empty({r, c / 32}, ScalarType::Byte, x);
  }
}

// rmsnorm_quant(x, weight, eps, qfmt)
PyObject *rmsnorm_quant(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4 || !PyFloat_CheckExact(a[2]) || !PyLong_CheckExact(a[3])) return none();
  const Tensor *x = gpu_tensor(a[0]), *w = gpu_tensor(a[1]);
  const float eps = (float)PyFloat_AS_DOUBLE(a[2]);
  const int qfmt = (int)PyLong_AsLong(a[3]);
  if (!x || !w || !bf16_rows(*x) || !plain(*w, 1) || w->size(0) != x->size(1) || w->device() != x->device())
    return none();
  const int64_t r = x->size(0), c = x->size(1);
  int wd;
  if (w->scalar_type() == ScalarType::BFloat16) wd = DSL_W_BF16;
  else if (w->scalar_type() == ScalarType::Float) wd = DSL_W_F32;
  else return none();
  if (qfmt == DSL_QFMT_MXFP4 && c % 32 != 0) return none();
  Tensor q, s;
  const bool ok = on_device(*x, [&] {
    producer_outputs(r, c, qfmt, *x, &q, &s);
    return dsl_rmsnorm_quant(ptr(*x), r, c, x->stride(0), ptr(*w), wd, eps, qfmt, ptr(q), ptr(s), nullptr,
                             0, stream_of(*x)) == DSL_OK;
  });
  return ok ? pack({q, s}) : none();
  END_HANDLE_TH_ERRORS
}

// swiglu_quant(input, qfmt)
PyObject *swiglu_quant(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !PyLong_CheckExact(a[1])) return none();
  const Tensor *x = gpu_tensor(a[0]);
  const int qfmt = (int)PyLong_AsLong(a[1]);
  if (!x || !bf16_rows(*x) || x->size(1) % 2 != 0) return none();
  const int64_t r = x->size(0), h = x->size(1) / 2;
  if (qfmt == DSL_QFMT_MXFP4 && h % 32 != 0) return none();
  Tensor q, s;
  const bool ok = on_device(*x, [&] {
    producer_outputs(r, h, qfmt, *x, &q, &s);
    return dsl_swiglu_quant(ptr(*x), r, h, x->stride(0), qfmt, ptr(q), ptr(s), nullptr, 0,
                            stream_of(*x)) == DSL_OK;
  });
  return ok ? pack({q, s}) : none();
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------ MoE --
// moe_projection(x, topk_ids, topk_weights, qw, sw, one_launch, out_dtype):
// route + per-token E4M3, the grouped GEMM through the row map, combine.
PyObject *moe_projection(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 7) return none();
  const Tensor *x = gpu_tensor(a[0]), *ids = gpu_tensor(a[1]), *tw = gpu_tensor(a[2]),
               *qw = gpu_tensor(a[3]), *sw = gpu_tensor(a[4]);
  const bool one_launch = a[5] == Py_True;
  const int code = out_code(a[6]);
  if (!x || !ids || !tw || !qw || !sw || code < 0) return none();
  if (!bf16_rows(*x) || !is_scales(*ids, ScalarType::Int) || ids->dim() != 2 ||
      !is_scales(*tw, ScalarType::Float) || tw->sizes() != ids->sizes() || !is_codes(*qw) ||
      !plain(*qw, 3) || !is_scales(*sw, ScalarType::Float))
    return none();
  const at::Device d = x->device();
  if (ids->device() != d || tw->device() != d || qw->device() != d || sw->device() != d) return none();
  const int64_t t = x->size(0), k = x->size(1), topk = ids->size(1), e = qw->size(0), nn = qw->size(1);
  if (ids->size(0) != t || qw->size(2) != k || sw->numel() != e * nn) return none();
  const int64_t rows = t * topk;
  Tensor out;
  const bool ok = on_device(*x, [&] {
    void *st = stream_of(*x);
    // offsets, dest, src_token and the rows' scales in one allocation
    const int64_t o1 = (e + 1 + 3) / 4 * 4, o2 = o1 + (rows + 3) / 4 * 4, o3 = o2 + (rows + 3) / 4 * 4;
    const Tensor tab = empty({o3 + rows}, ScalarType::Int, *x);
    int32_t *off = ptr<int32_t>(tab), *dest = off + o1, *src = off + o2;
    float *sx = reinterpret_cast<float *>(off + o3);
    const Tensor qx = empty({t, k}, ScalarType::Byte, *x);
    if (one_launch) {
      if (dsl_moe_route_quant_tokens(ptr<int32_t>(*ids), t, topk, e, ptr(*x), k, x->stride(0), off, dest,
                                     src, ptr<uint8_t>(qx), sx, st) != DSL_OK)
        return false;
    } else {
      const size_t nb = dsl_moe_route_workspace_bytes(t, topk, e);
      const Tensor ws = bytes((int64_t)(nb > 4 ? nb : 4), *x);
      if (dsl_moe_route(ptr<int32_t>(*ids), t, topk, e, off, dest, src, ptr(ws), (size_t)ws.numel(), st) != DSL_OK ||
          dsl_moe_quant_tokens(ptr(*x), t, k, x->stride(0), dest, topk, rows, ptr<uint8_t>(qx), sx, st) != DSL_OK)
        return false;
    }
    const Tensor y = out_matrix(rows, nn, DSL_OUT_BF16, *x);
    if (dsl_moe_grouped_fp8_gemm(ptr<uint8_t>(qx), t, src, ptr<uint8_t>(*qw), ptr(y), off, e, rows, nn, k,
                                 nn, DSL_OUT_BF16, sx, ptr<float>(*sw), st) != DSL_OK)
      return false;
    out = out_matrix(t, nn, code, *x);
    return dsl_moe_combine(ptr(y), rows, nn, nn, dest, ptr<float>(*tw), t, topk, ptr(out), nn, code, st) ==
           DSL_OK;
  });
  return ok ? THPVariable_Wrap(out) : none();
  END_HANDLE_TH_ERRORS
}

// ----------------------------------------------------------------- LoRA --
// lora_gemm(X, W, loraA, loraB, scales): W the view of K-major storage
PyObject *lora_gemm(PyObject *, PyObject *const *a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 5) return none();
  const Tensor *x = gpu_tensor(a[0]), *w = gpu_tensor(a[1]), *la = gpu_tensor(a[2]),
               *lb = gpu_tensor(a[3]), *sc = gpu_tensor(a[4]);
  if (!x || !w || !la || !lb || !sc) return none();
  for (const Tensor *t : {x, w, la, lb})
    if (t->scalar_type() != ScalarType::BFloat16 || t->device() != x->device()) return none();
  if (!plain(*x, 2) || !k_major_view(*w) || la->dim() != 3 || lb->dim() != 3 || la->numel() == 0 ||
      lb->numel() == 0 || !is_scales(*sc, ScalarType::Float) || sc->device() != x->device())
    return none();
  const int64_t m = x->size(0), k = x->size(1), nn = w->size(1), l = la->size(0), r = la->size(2);
  if (w->size(0) != k || la->size(1) != k || lb->size(0) != l || lb->size(1) != r || lb->size(2) != nn ||
      sc->numel() != l)
    return none();
  Tensor y;
  const bool ok = on_device(*x, [&] {
    if (la->is_contiguous() && lb->is_contiguous()) {   // packed by the call itself
      const size_t nb = dsl_lora_gemm_ab_workspace_bytes(m, nn, k, r, l);
      const Tensor ws = bytes((int64_t)(nb > 256 ? nb : 256), *x);
      y = empty({m, nn}, ScalarType::Float, *x);
      return dsl_lora_gemm_ab(ptr(*x), ptr(*w), ptr(*la), ptr(*lb), ptr<float>(*sc), ptr<float>(y), m, nn, k, r,
                              l, nn, ptr(ws), (size_t)ws.numel(), stream_of(*x)) == DSL_OK;
    }
    const Tensor at = la->detach().permute({0, 2, 1}).reshape({l * r, k}).contiguous();
    const Tensor bt = lb->detach().permute({2, 0, 1}).reshape({nn, l * r}).contiguous();
    if (!aligned16(at) || !aligned16(bt)) return false;
    const size_t nb = dsl_lora_gemm_workspace_bytes(m, nn, k, r, l);
    const Tensor ws = bytes((int64_t)(nb > 256 ? nb : 256), *x);
    y = empty({m, nn}, ScalarType::Float, *x);
    return dsl_lora_gemm(ptr(*x), ptr(*w), ptr(at), ptr(bt), ptr<float>(*sc), ptr<float>(y), m, nn, k, r, l,
                         nn, ptr(ws), (size_t)ws.numel(), stream_of(*x)) == DSL_OK;
  });
  return ok ? THPVariable_Wrap(y) : none();
  END_HANDLE_TH_ERRORS
}

#define DSL_FN(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {DSL_FN(quant_fp8_tensor), DSL_FN(quant_fp8_blocks), DSL_FN(quant_mxfp4),
                         DSL_FN(quant_nvfp4),      DSL_FN(fp8_gemm),         DSL_FN(fp4_gemm),
                         DSL_FN(bf16_gemm),        DSL_FN(grouped_fp8_gemm), DSL_FN(rmsnorm_quant),
                         DSL_FN(swiglu_quant),     DSL_FN(moe_projection),   DSL_FN(lora_gemm),
                         DSL_FN(quant_fp8_rows_batched),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "dsl_fast", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_dsl_fast() { return PyModule_Create(&module); }
