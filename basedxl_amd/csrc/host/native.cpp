// The host path of an ordinary eager call in one C++ function: checks, result tensor, stream, workspace and the call
// into libcascmm.so.
//
// A UNet step makes some 500 of these calls, most of them on kernels of 5 - 15 us; issued from Python (argument checks,
// views, torch.empty, a ctypes call of twenty arguments) each took 13 - 21 us of host time, so the GPU waited for the
// host.  Everything here is a short cut: a function returns None whenever a call is not the ordinary case (another
// device, unusual strides, a workspace that has to grow, a status other than 0, ...) and the Python code, which holds
// all rules and raises all errors, takes it from the start.  Nothing is remembered about a tensor.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <tuple>
#include <unordered_map>

#include "../../../include/cascmm.h"

namespace {

PyObject* g_scales = nullptr;       // the dict {(device index, stream handle): int32[2] tensor} of the fp8 scale searches' scratch
PyObject* g_workspaces = nullptr;   // the dict {(device index, stream handle): uint8 tensor} of the Python wrapper

struct Need {
  int64_t M, N, K;
  int dt, fmt, terms, products;
  bool operator==(const Need& o) const {
    return M == o.M && N == o.N && K == o.K && dt == o.dt && fmt == o.fmt && terms == o.terms && products == o.products;
  }
};
struct NeedHash {
  size_t operator()(const Need& n) const {
    uint64_t h = 1469598103934665603ull;
    for (uint64_t v : {(uint64_t)n.M, (uint64_t)n.N, (uint64_t)n.K, (uint64_t)(n.dt | n.fmt << 8 | n.terms << 16 | n.products << 24)})
      h = (h ^ v) * 1099511628211ull;
    return (size_t)h;
  }
};
// cascmm_workspace_bytes per problem (it walks the whole variant table); guarded by the interpreter lock
size_t workspace_need(const Need& n) {
  static std::unordered_map<Need, size_t, NeedHash> memo;
  auto it = memo.find(n);
  if (it != memo.end()) return it->second;
  if (memo.size() >= 4096) memo.clear();
  return memo[n] = cascmm_workspace_bytes(n.M, n.N, n.K, n.dt, n.fmt, n.terms, n.products);
}

int dtype_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return CASCMM_DT_F32;
    case at::kHalf: return CASCMM_DT_F16;
    case at::kBFloat16: return CASCMM_DT_BF16;
    default: return -1;
  }
}
int format_code(PyObject* s) {
  if (!PyUnicode_Check(s)) return -1;
  if (PyUnicode_CompareWithASCIIString(s, "bf16") == 0) return CASCMM_FMT_BF16;
  if (PyUnicode_CompareWithASCIIString(s, "fp16") == 0) return CASCMM_FMT_FP16;
  return -1;   // (fp8 products find scales first: a function of their own)
}
int products_code(PyObject* s) {
  if (!PyUnicode_Check(s)) return -1;
  if (PyUnicode_CompareWithASCIIString(s, "tri") == 0) return CASCMM_PROD_TRI;
  if (PyUnicode_CompareWithASCIIString(s, "full") == 0) return CASCMM_PROD_FULL;
  return -1;
}

// a plain torch.Tensor or Parameter on the current GPU (no subclass: those may not own memory)
const at::Tensor* gpu_tensor(PyObject* o, int device) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.is_cuda() && t.get_device() == device && t.has_storage() ? &t : nullptr;
}
// the left operand as rows of K elements: false where it is not a view of such rows
bool rows_of(const at::Tensor& a, int64_t& M, int64_t& K, int64_t& lda) {
  if (a.dim() < 1) return false;
  K = a.size(-1);
  if (K <= 0 || a.numel() == 0) return false;
  M = a.numel() / K;
  if (a.is_contiguous()) lda = K;
  else if (a.dim() == 2 && a.stride(1) == 1 && a.stride(0) >= K) lda = a.stride(0);
  else return false;
  if (M == 1) lda = K;
  return true;
}
// a bias the kernels can read (None: no bias); false: not the ordinary case
bool bias_of(PyObject* o, const at::Tensor& a, int64_t n, int device, const void*& ptr) {
  ptr = nullptr;
  if (o == Py_None) return true;
  const at::Tensor* b = gpu_tensor(o, device);
  if (!b || b->dim() != 1 || b->size(0) != n || b->scalar_type() != a.scalar_type() || !b->is_contiguous()) return false;
  ptr = b->const_data_ptr();
  return true;
}
// the stream's workspace if it holds `need` bytes already (eager launches: a recorded one takes the Python path).
// `hold` keeps it until the launch: another thread may replace the dict's entry while this one has given up the lock, and
// memory freed before the launch could be written by work that was enqueued in between
bool workspace_of(size_t need, int device, hipStream_t stream, at::Tensor& hold, void*& ptr, size_t& bytes) {
  ptr = nullptr;
  bytes = 0;
  if (need == 0) return true;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) return false;
  PyObject* key = Py_BuildValue("(iK)", device, (unsigned long long)(uintptr_t)stream);
  if (!key) { PyErr_Clear(); return false; }
  PyObject* ws = PyDict_GetItem(g_workspaces, key);   // borrowed
  Py_DECREF(key);
  if (!ws || !THPVariable_Check(ws)) return false;
  hold = THPVariable_Unpack(ws);
  if ((size_t)hold.numel() < need) return false;
  ptr = hold.data_ptr();
  bytes = (size_t)hold.numel();
  return true;
}
// the stream's scratch of the scale searches, if it exists already and nothing is being recorded; `hold` as above
bool scale_scratch_of(int device, hipStream_t stream, at::Tensor& hold, int32_t*& ptr) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (!g_scales || hipStreamIsCapturing(stream, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) return false;
  PyObject* key = Py_BuildValue("(iK)", device, (unsigned long long)(uintptr_t)stream);
  if (!key) { PyErr_Clear(); return false; }
  PyObject* t = PyDict_GetItem(g_scales, key);   // borrowed
  Py_DECREF(key);
  if (!t || !THPVariable_Check(t)) return false;
  hold = THPVariable_Unpack(t);
  if (hold.numel() != 2 || hold.scalar_type() != at::kInt) return false;
  ptr = (int32_t*)hold.data_ptr();
  return true;
}
at::Tensor result_like(const at::Tensor& a, int64_t n) {
  c10::SmallVector<int64_t, 6> sizes(a.sizes().begin(), a.sizes().end());
  sizes.back() = n;
  return at::empty(sizes, at::TensorOptions().dtype(a.scalar_type()).device(a.device()));
}

// matmul(a, b, bias | None, lowp | None, terms | None, products) -> Tensor | None: b a raw [K, N] tensor
PyObject* matmul(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 6) Py_RETURN_NONE;
  try {
    const int device = c10::hip::current_device();
    const at::Tensor *a = gpu_tensor(args[0], device), *b = gpu_tensor(args[1], device);
    if (!a || !b || b->dim() != 2 || b->scalar_type() != a->scalar_type() || !b->is_contiguous()) Py_RETURN_NONE;
    const int dt = dtype_code(*a);
    // the default cascade: two bf16 terms for fp32, one term of their own format for 16-bit tensors
    const int fmt = args[3] != Py_None ? format_code(args[3]) : dt == CASCMM_DT_F16 ? CASCMM_FMT_FP16 : CASCMM_FMT_BF16;
    const int terms = args[4] != Py_None ? (PyLong_Check(args[4]) ? (int)PyLong_AsLong(args[4]) : -1) : dt == CASCMM_DT_F32 ? 2 : 1;
    const int products = products_code(args[5]);
    int64_t M, K, lda;
    const void* bias;
    if (PyErr_Occurred()) { PyErr_Clear(); Py_RETURN_NONE; }
    if (dt < 0 || fmt < 0 || terms < 1 || products < 0 || !rows_of(*a, M, K, lda) || b->size(0) != K || b->size(1) <= 0) Py_RETURN_NONE;
    const int64_t N = b->size(1);
    if (!bias_of(args[2], *a, N, device, bias)) Py_RETURN_NONE;
    const hipStream_t stream = c10::hip::getCurrentHIPStream(device).stream();
    at::Tensor hold;
    void* ws;
    size_t ws_bytes;
    if (!workspace_of(workspace_need({M, N, K, dt, fmt, terms, products}), device, stream, hold, ws, ws_bytes)) Py_RETURN_NONE;
    at::Tensor out = result_like(*a, N);
    const void *ap = a->const_data_ptr(), *bp = b->const_data_ptr();
    void* cp = out.data_ptr();
    int st;
    Py_BEGIN_ALLOW_THREADS
    st = cascmm_gemm_variant(ap, bp, cp, bias, M, N, K, lda, N, N, dt, fmt, terms, products, nullptr, ws, ws_bytes, stream, -1);
    Py_END_ALLOW_THREADS
    if (st != CASCMM_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
  } catch (...) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

// prepared(a, slots, bias | None, K, N, fmt, terms, products, dtype of the weight, glu, min_rows) -> Tensor | None: the
// operand slots of a PreparedWeight (not fp8); fp32 problems of fewer than min_rows rows are left to the caller
PyObject* prepared(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 11) Py_RETURN_NONE;
  try {
    const int device = c10::hip::current_device();
    const at::Tensor *a = gpu_tensor(args[0], device), *slots = gpu_tensor(args[1], device);
    if (!a || !slots) Py_RETURN_NONE;
    const int64_t wk = PyLong_AsLongLong(args[3]), N = PyLong_AsLongLong(args[4]);
    const int fmt = (int)PyLong_AsLong(args[5]), terms = (int)PyLong_AsLong(args[6]), products = products_code(args[7]);
    const int w_dt = (int)PyLong_AsLong(args[8]), glu = PyObject_IsTrue(args[9]);
    const int64_t min_rows = PyLong_AsLongLong(args[10]);
    if (PyErr_Occurred()) { PyErr_Clear(); Py_RETURN_NONE; }
    const int dt = dtype_code(*a);
    int64_t M, K, lda;
    const void* bias;
    if (dt < 0 || fmt == CASCMM_FMT_FP8 || products < 0 || N <= 0 || !rows_of(*a, M, K, lda) || K != wk) Py_RETURN_NONE;
    if (!bias_of(args[2], *a, N, device, bias)) Py_RETURN_NONE;
    const size_t slot_bytes = cascmm_prepared_bytes(wk, N, fmt, terms);
    if (slots->nbytes() != (slot_bytes > 16 ? slot_bytes : 16)) Py_RETURN_NONE;   // (not this layout: the wrapper raises)
    const uintptr_t at0 = (uintptr_t)a->const_data_ptr();
    if (at0 % 16 != 0 || (size_t)lda * a->element_size() % 16 != 0) Py_RETURN_NONE;   // (the wrapper copies such rows)
    if (dt == CASCMM_DT_F32) {
      const bool any_rows = fmt == CASCMM_FMT_BF16 && terms == 2 && !glu && K % 8 == 0;
      if (M < min_rows || (!any_rows && (K % 64 != 0 || N % 4 != 0))) Py_RETURN_NONE;
    } else if (dt != w_dt || terms != 1 || K % 8 != 0) {
      Py_RETURN_NONE;
    }
    const hipStream_t stream = c10::hip::getCurrentHIPStream(device).stream();
    at::Tensor hold;
    void* ws = nullptr;
    size_t ws_bytes = 0;
    if (!glu &&
        !workspace_of(workspace_need({M, N, K, dt, fmt, terms, products}), device, stream, hold, ws, ws_bytes))
      Py_RETURN_NONE;
    const int64_t NO = glu ? N / 2 : N;
    at::Tensor out = result_like(*a, NO);
    const void *ap = (const void*)at0, *bp = slots->const_data_ptr();
    void* cp = out.data_ptr();
    int st;
    Py_BEGIN_ALLOW_THREADS
    st = glu ? cascmm_gemm_prepared_glu(1, &ap, &bp, &cp, bias ? &bias : nullptr, M, N, K, lda, NO, dt, fmt, terms, products, nullptr, stream, -1)
             : cascmm_gemm_prepared(1, &ap, &bp, &cp, bias ? &bias : nullptr, M, N, K, lda, NO, dt, fmt, terms, products, nullptr, ws, ws_bytes,
                                    stream, -1);
    Py_END_ALLOW_THREADS
    if (st != CASCMM_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
  } catch (...) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

// fp8(a, b, bias | None, b_exp | None, K, N, terms, products, b is slots) -> Tensor | None: fp8 terms of fp32 tensors, the scale of a found
// in the call; b a raw [K, N] tensor or the operand slots of a PreparedWeight, b_exp its scale exponent (None, raw only: found too)
PyObject* fp8(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 9) Py_RETURN_NONE;
  try {
    const int device = c10::hip::current_device();
    const at::Tensor *a = gpu_tensor(args[0], device), *b = gpu_tensor(args[1], device);
    if (!a || !b) Py_RETURN_NONE;
    int64_t wk = PyLong_AsLongLong(args[4]), N = PyLong_AsLongLong(args[5]);   // (of slots)
    const int terms = PyLong_Check(args[6]) ? (int)PyLong_AsLong(args[6]) : -1, products = products_code(args[7]), slots = PyObject_IsTrue(args[8]);
    if (PyErr_Occurred()) { PyErr_Clear(); Py_RETURN_NONE; }
    if (!slots) {
      if (b->dim() != 2 || b->scalar_type() != at::kFloat || !b->is_contiguous()) Py_RETURN_NONE;
      wk = b->size(0);
      N = b->size(1);
    }
    const at::Tensor* exp = args[3] == Py_None ? nullptr : gpu_tensor(args[3], device);
    if ((args[3] != Py_None || slots) && (!exp || exp->scalar_type() != at::kInt || exp->numel() != 1)) Py_RETURN_NONE;
    int64_t M, K, lda;
    const void* bias;
    if (a->scalar_type() != at::kFloat || terms < 1 || products < 0 || N <= 0 || !rows_of(*a, M, K, lda) || K != wk) Py_RETURN_NONE;
    if (!bias_of(args[2], *a, N, device, bias)) Py_RETURN_NONE;
    if (slots) {
      const size_t bytes = cascmm_prepared_bytes(wk, N, CASCMM_FMT_FP8, terms);
      if (b->nbytes() != (bytes > 16 ? bytes : 16)) Py_RETURN_NONE;                                    // (not this layout: the wrapper raises)
      if ((uintptr_t)a->const_data_ptr() % 16 != 0 || lda % 4 != 0 || K % 64 != 0 || N % 4 != 0) Py_RETURN_NONE;   // (the wrapper copies such rows)
    }
    const hipStream_t stream = c10::hip::getCurrentHIPStream(device).stream();
    at::Tensor hold, hold_scratch;
    void* ws;
    size_t ws_bytes;
    int32_t* scratch;
    if (!scale_scratch_of(device, stream, hold_scratch, scratch) ||
        !workspace_of(workspace_need({M, N, K, CASCMM_DT_F32, CASCMM_FMT_FP8, terms, products}), device, stream, hold, ws, ws_bytes))
      Py_RETURN_NONE;
    at::Tensor out = result_like(*a, N);
    at::Tensor exps = at::empty({2}, at::TensorOptions().dtype(at::kInt).device(a->device()));
    const void *ap = a->const_data_ptr(), *bp = b->const_data_ptr();
    const int32_t* b_exp = exp ? (const int32_t*)exp->const_data_ptr() : nullptr;
    void* cp = out.data_ptr();
    int32_t* ep = (int32_t*)exps.data_ptr();
    int st;
    Py_BEGIN_ALLOW_THREADS
    if (b_exp) {
      st = cascmm_gemm_fp8_autoscale(ap, bp, slots, cp, bias, M, N, K, lda, N, N, terms, products, b_exp, ep, scratch, ws, ws_bytes, stream);
    } else {
      st = cascmm_tensor_exps(ap, M, K, lda, CASCMM_DT_F32, nullptr, ep, scratch, stream);
      if (st == CASCMM_OK) st = cascmm_tensor_exps(bp, K, N, N, CASCMM_DT_F32, nullptr, ep + 1, scratch, stream);
      if (st == CASCMM_OK) st = cascmm_gemm_variant(ap, bp, cp, bias, M, N, K, lda, N, N, CASCMM_DT_F32, CASCMM_FMT_FP8, terms, products, ep, ws, ws_bytes, stream, -1);
    }
    Py_END_ALLOW_THREADS
    if (st != CASCMM_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
  } catch (...) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
}

// init_scales(scratch): the dict to look the scale searches' scratch up in
PyObject* init_scales(PyObject*, PyObject* d) {
  if (!PyDict_Check(d)) {
    PyErr_SetString(PyExc_TypeError, "init_scales takes the dict of scale scratch");
    return nullptr;
  }
  Py_INCREF(d);
  Py_XDECREF(g_scales);
  g_scales = d;
  Py_RETURN_NONE;
}

// init(workspaces): the dict to look workspaces up in
PyObject* init(PyObject*, PyObject* d) {
  if (!PyDict_Check(d)) {
    PyErr_SetString(PyExc_TypeError, "init takes the dict of workspaces");
    return nullptr;
  }
  Py_INCREF(d);
  Py_XDECREF(g_workspaces);
  g_workspaces = d;
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"matmul", (PyCFunction)(void (*)(void))matmul, METH_FASTCALL, "raw operands; None: not the ordinary case"},
    {"prepared", (PyCFunction)(void (*)(void))prepared, METH_FASTCALL, "prepared weight; None: not the ordinary case"},
    {"fp8", (PyCFunction)(void (*)(void))fp8, METH_FASTCALL, "fp8 terms, scale found in the call; None: not the ordinary case"},
    {"init_scales", init_scales, METH_O, "hands over the dict of the scale searches' scratch"},
    {"init", init, METH_O, "hands over the workspaces' dict"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_native", "host path of ordinary eager calls", -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&kModule); }
