// The calls of the operators, from Python arguments to the C entry points of libtlq, in native code.
//
// What a small operator costs is the host: a decode GEMV runs 6 us on the GPU, and checking its arguments, allocating its
// output and workspace and making the call took 23 us in Python (torch's own one-launch operators take 4.0 us).
// Here the same steps are one extension call of 4 - 5 us with one launch (1 x 11008 x 4096: 22.5 -> 6.1 us a call, which is the
// kernel): a Plan is built once per kernel object from its parameter list, and calling it checks the tensors, allocates
// outputs (and the workspace the entry point asks for) from torch's caching allocator on the current stream, releases the
// interpreter lock and calls the entry point.
//
// A Plan does the ordinary call only.  Whatever its checks do not let through -- a wrong type or shape, a tensor on another
// device, an allocation that fails -- comes back as NotImplemented with nothing done, and the Python path of the caller takes
// over: it names the error, or runs the call on the other device.  What passes the checks is called once: where the entry point refuses it, the entry point's
// message is raised from here, as that path would.  Nothing here keeps state between calls, so any number of threads and streams may
// use one Plan.
#include <Python.h>
#include <structmember.h>

#include <string>
#include <vector>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "tlq.h"

namespace {

// ---- the entry points, as loaded by the Python side (which may be told to load another library) -----------------------
#define TLQ_ENTRIES(X)                                                                                              \
  X(tlq_last_error) X(tlq_gemm_w4a16_layout_ws) X(tlq_w4a16_workspace_bytes_for) X(tlq_gemm_w8a8_ws) X(tlq_w8a8_workspace_bytes) \
  X(tlq_act_quant_i8) X(tlq_gemm_w4a8_ws) X(tlq_gemm_w4a8) X(tlq_gemm_i8) X(tlq_gemm_f16_ws) X(tlq_f16_workspace_bytes)          \
  X(tlq_gemm_f16_batched) X(tlq_gemv) X(tlq_gemm_f16_splitk) X(tlq_dequant_w4_layout) X(tlq_unpack_int4) X(tlq_pack_int4)        \
  X(tlq_quantize_sym4)
struct Entries {
#define X(name) decltype(&::name) name = nullptr;
  TLQ_ENTRIES(X)
#undef X
};
Entries lib;

enum Kind { kW4A16, kW8A8, kActQuant, kW4A8Ws, kW4A8, kI8, kF16, kF16Batched, kGemv, kSplitK };
struct KindName {
  const char* name;
  Kind kind;
  int ints, tensors;  // how many integers the kind's call takes, how many tensors its parameter list holds at least
};
const KindName kKinds[] = {{"w4a16", kW4A16, 10, 3}, {"w8a8", kW8A8, 8, 4},  {"act_quant", kActQuant, 3, 3}, {"w4a8_ws", kW4A8Ws, 4, 4},
                           {"w4a8", kW4A8, 4, 3},    {"i8", kI8, 3, 3},      {"f16", kF16, 3, 3},            {"f16_batched", kF16Batched, 5, 3},
                           {"gemv", kGemv, 3, 3},    {"splitk", kSplitK, 5, 3}};

const int kMaxDims = 4, kMaxParams = 8, kMaxSymbols = 4;
enum Role { kInput, kOutput, kWorkspace };
struct Param {
  int ndim = 0;
  int64_t dim[kMaxDims];  // a size, or -1 - (number of a symbol)
  at::ScalarType type = at::kByte;
  Role role = kInput;
};
struct PlanObject {
  PyObject_HEAD
  vectorcallfunc vectorcall;
  Kind kind;
  int n_params, n_inputs, n_outputs;
  int64_t v[12];
  float zero;
  Param param[kMaxParams];
};

bool scalar_type(int code, at::ScalarType& t) {  // the type codes of tlq.h, and 5 for uint8
  switch (code) {
    case TLQ_F16: t = at::kHalf; return true;
    case TLQ_BF16: t = at::kBFloat16; return true;
    case TLQ_F32: t = at::kFloat; return true;
    case TLQ_I8: t = at::kChar; return true;
    case TLQ_I32: t = at::kInt; return true;
    case 5: t = at::kByte; return true;
    default: return false;
  }
}

at::Tensor new_tensor(at::IntArrayRef shape, at::ScalarType type, int device) {
  return at::Tensor(at::detail::empty_cuda(shape, type, at::Device(at::kCUDA, (at::DeviceIndex)device), std::nullopt));
}

struct Released {  // the interpreter lock is free inside (a launch can wait for room in the queue)
  PyThreadState* s = PyEval_SaveThread();
  ~Released() { PyEval_RestoreThread(s); }
};

PyObject* not_ordinary() { Py_RETURN_NOTIMPLEMENTED; }

int raise_for(int rc) {
  const char* msg = lib.tlq_last_error();
  if (msg && *msg)
    PyErr_SetString(PyExc_RuntimeError, msg);
  else
    PyErr_Format(PyExc_RuntimeError, "libtlq call failed with code %d", rc);
  return -1;
}

void* ptr(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }

// The entry point of a plan on its tensors (in parameter order; null where there is none), on `stream` of `device`.
// other_stream: not the stream that is current to torch; a workspace is then kept from reuse until that stream is done.
int launch(const PlanObject& p, const at::Tensor* const* t, int device, hipStream_t stream, bool other_stream) {
  const int64_t* const v = p.v;
  int64_t ws_bytes = 0;
  if (p.kind == kW4A16) {
    ws_bytes = lib.tlq_w4a16_workspace_bytes_for(v[0], v[1], v[2], (int)v[6]);
    // interleaved words have no entry of their own in that size: the two passes may want the dequantised matrix
    if (v[7] != TLQ_W_PLAIN && v[6] == TLQ_ALGO_AUTO && v[0] > 256) ws_bytes = std::max(ws_bytes, v[1] * v[2] * 2);
  } else if (p.kind == kW8A8) {
    ws_bytes = lib.tlq_w8a8_workspace_bytes(v[0], v[1] < 0 ? t[0]->size(0) : v[1], v[2], v[3]);
  } else if (p.kind == kF16) {
    ws_bytes = lib.tlq_f16_workspace_bytes(1, v[0], v[1], v[2]);
  }
  c10::DataPtr ws;  // the allocator's block alone: no tensor around it
  if (ws_bytes > 0) {
    ws = c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::get()->allocate((size_t)ws_bytes);
    if (other_stream)
      c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::recordStreamMasqueradingAsCUDA(ws, c10::hip::getStreamFromExternalMasqueradingAsCUDA(stream, (c10::DeviceIndex)device));
  }
  void* const w = ws.get();
  Released free_lock;
  switch (p.kind) {
    case kW4A16: {
      int i = 2;
      const at::Tensor* s = v[8] ? t[i++] : nullptr;
      const at::Tensor* z = v[9] ? t[i++] : nullptr;
      return lib.tlq_gemm_w4a16_layout_ws(ptr(t[0]), ptr(t[1]), ptr(s), ptr(z), ptr(t[i]), v[0], v[1], v[2], v[3], p.zero, (int)v[4], (int)v[5],
                                          (int)v[6], (int)v[7], w, ws_bytes, stream);
    }
    case kW8A8: {
      const int i = v[7] ? 3 : 2;
      return lib.tlq_gemm_w8a8_ws(ptr(t[0]), ptr(t[1]), v[7] ? ptr(t[2]) : nullptr, ptr(t[i]), ptr(t[i + 1]), w, ws_bytes, v[0],
                                  v[1] < 0 ? t[0]->size(0) : v[1], v[2], v[3], v[4], (int)v[5], (int)v[6], stream);
    }
    case kActQuant: return lib.tlq_act_quant_i8(ptr(t[0]), ptr(t[1]), ptr(t[2]), t[0]->size(0), v[0], (int)v[1], (int)v[2], stream);
    case kW4A8Ws: return lib.tlq_gemm_w4a8_ws(ptr(t[0]), ptr(t[1]), ptr(t[2]), t[2] ? (int64_t)t[2]->nbytes() : 0, ptr(t[3]), v[0], v[1], v[2], (int)v[3], stream);
    case kW4A8: return lib.tlq_gemm_w4a8(ptr(t[0]), ptr(t[1]), ptr(t[2]), v[0], v[1], v[2], (int)v[3], stream);
    case kI8: return lib.tlq_gemm_i8(ptr(t[0]), ptr(t[1]), ptr(t[2]), 1, v[0], v[1], v[2], TLQ_B_KN, stream);
    case kF16: return lib.tlq_gemm_f16_ws(ptr(t[0]), ptr(t[1]), ptr(t[2]), w, ws_bytes, 1, v[0], v[1], v[2], TLQ_F16, TLQ_F16, TLQ_B_KN, stream);
    case kF16Batched: return lib.tlq_gemm_f16_batched(ptr(t[0]), ptr(t[1]), ptr(t[2]), v[0], v[1], v[2], v[3], (int)v[4], (int)v[4], TLQ_B_KN, stream);
    case kGemv: return lib.tlq_gemv(ptr(t[0]), ptr(t[1]), ptr(t[2]), v[0], v[1], (int)v[2], (int)v[2], stream);
    case kSplitK: return lib.tlq_gemm_f16_splitk(ptr(t[0]), ptr(t[1]), ptr(t[2]), v[0], v[1], v[2], v[3], (int)v[4], TLQ_B_KN, stream);
  }
  return 1;
}

// A tensor that the ordinary call takes: a plain contiguous one on the current device.
const at::Tensor* plain_tensor(PyObject* o, int device) {
  if (!THPVariable_Check(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.get_device() != device || t.layout() != at::kStrided || !t.has_storage() || !t.is_contiguous() ||
      t.key_set().has(c10::DispatchKey::Python))
    return nullptr;
  return &t;
}

PyObject* plan_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
  const PlanObject& p = *(const PlanObject*)self;
  const Py_ssize_t nargs = PyVectorcall_NARGS(nargsf);
  if (nargs < p.n_inputs || (kwnames && PyTuple_GET_SIZE(kwnames))) return not_ordinary();  // (surplus positionals are ignored)
  try {
    const int device = c10::hip::current_device();
    const at::Tensor* t[kMaxParams] = {};
    at::Tensor made[kMaxParams];
    int64_t symbol[kMaxSymbols] = {-1, -1, -1, -1};
    int next = 0;
    for (int i = 0; i < p.n_params; ++i) {
      const Param& q = p.param[i];
      if (q.role != kInput) continue;
      const at::Tensor* x = plain_tensor(args[next++], device);
      if (!x || x->scalar_type() != q.type || x->dim() != q.ndim) return not_ordinary();
      for (int d = 0; d < q.ndim; ++d) {
        const int64_t have = x->size(d);
        int64_t want = q.dim[d];
        if (want < 0) {
          int64_t& s = symbol[-1 - want];
          if (s < 0) s = have;
          want = s;
        }
        if (have != want) return not_ordinary();
      }
      t[i] = x;
    }
    for (int i = 0; i < p.n_params; ++i) {
      const Param& q = p.param[i];
      if (q.role != kOutput) continue;
      int64_t shape[kMaxDims];
      for (int d = 0; d < q.ndim; ++d) {
        shape[d] = q.dim[d] < 0 ? symbol[-1 - q.dim[d]] : q.dim[d];
        if (shape[d] < 0) return not_ordinary();
      }
      made[i] = new_tensor(at::IntArrayRef(shape, (size_t)q.ndim), q.type, device);
      t[i] = &made[i];
    }
    const int rc = launch(p, t, device, c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(), false);
    if (rc != 0) {
      raise_for(rc);
      return nullptr;
    }
    PyObject* list = p.n_outputs == 1 ? nullptr : PyList_New(p.n_outputs);
    if (p.n_outputs != 1 && !list) return nullptr;
    int k = 0;
    for (int i = 0; i < p.n_params; ++i) {
      if (p.param[i].role != kOutput) continue;
      PyObject* o = THPVariable_Wrap(std::move(made[i]));
      if (!list) return o;
      if (!o) {
        Py_DECREF(list);
        return nullptr;
      }
      PyList_SET_ITEM(list, k++, o);
    }
    return list;
  } catch (const std::exception&) {
    // (the Python path meets the same condition and names it: an allocation that failed, for instance)
    PyErr_Clear();
    return not_ordinary();
  }
}

// Plan.launch(tensors, stream): the call alone, for the Python path, which has checked and allocated everything and made the
// tensors' device the current one.  tensors: one per parameter, None for the reference's workspace parameters.
PyObject* plan_launch(PyObject* self, PyObject* args) {
  const PlanObject& p = *(const PlanObject*)self;
  PyObject* list;
  unsigned long long stream;
  if (!PyArg_ParseTuple(args, "O!K", &PyList_Type, &list, &stream)) return nullptr;
  if (PyList_GET_SIZE(list) != p.n_params) {
    PyErr_SetString(PyExc_ValueError, "one tensor per parameter is wanted");
    return nullptr;
  }
  try {
    const at::Tensor* t[kMaxParams] = {};
    for (int i = 0; i < p.n_params; ++i) {
      PyObject* o = PyList_GET_ITEM(list, i);
      if (o == Py_None && p.param[i].role == kWorkspace) continue;
      if (!THPVariable_Check(o)) {
        PyErr_SetString(PyExc_ValueError, "one tensor per parameter is wanted");
        return nullptr;
      }
      t[i] = &THPVariable_Unpack(o);
    }
    const int device = c10::hip::current_device();
    hipStream_t st = (hipStream_t)stream;
    const bool other = st && st != c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
    const int rc = launch(p, t, device, st, other);
    if (rc != 0) {
      raise_for(rc);
      return nullptr;
    }
    Py_RETURN_NONE;
  } catch (const c10::OutOfMemoryError& e) {
    PyObject* torch = PyImport_ImportModule("torch");
    PyObject* type = torch ? PyObject_GetAttrString(torch, "OutOfMemoryError") : nullptr;
    if (type) PyErr_SetString(type, e.what_without_backtrace());
    Py_XDECREF(type);
    Py_XDECREF(torch);
    return nullptr;
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// Plan(kind, params, ints, zero): params is a sequence of (shape, type code, role) with sizes or symbol names as the shape.
PyObject* plan_new(PyTypeObject* type, PyObject* args, PyObject*) {
  const char* kind;
  PyObject *params, *ints;
  double zero;
  if (!PyArg_ParseTuple(args, "sO!O!d", &kind, &PyTuple_Type, &params, &PyTuple_Type, &ints, &zero)) return nullptr;
  PlanObject* p = (PlanObject*)type->tp_alloc(type, 0);
  if (!p) return nullptr;
  p->vectorcall = plan_call;
  p->zero = (float)zero;
  const KindName* kn = nullptr;
  for (const KindName& k : kKinds)
    if (!strcmp(k.name, kind)) kn = &k;
  auto bad = [&](const char* what) -> PyObject* {
    if (!PyErr_Occurred()) PyErr_Format(PyExc_ValueError, "%s: %s", kind, what);
    Py_DECREF(p);
    return nullptr;
  };
  if (!kn) return bad("no such kind of call");
  p->kind = kn->kind;
  if (PyTuple_GET_SIZE(ints) != kn->ints) return bad("wrong number of integers");
  for (int i = 0; i < kn->ints; ++i) {
    p->v[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(ints, i));
    if (PyErr_Occurred()) return bad("");
  }
  const Py_ssize_t n = PyTuple_GET_SIZE(params);
  int least = kn->tensors;
  if (kn->kind == kW4A16) least += (p->v[8] != 0) + (p->v[9] != 0);
  if (kn->kind == kW8A8) least += p->v[7] != 0;
  if (n > kMaxParams || n < least) return bad("wrong number of parameters");
  p->n_params = (int)n;
  std::vector<std::string> names;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* shape;
    int code, role;
    if (!PyArg_ParseTuple(PyTuple_GET_ITEM(params, i), "O!ii", &PyTuple_Type, &shape, &code, &role)) return bad("");
    Param& q = p->param[i];
    const Py_ssize_t nd = PyTuple_GET_SIZE(shape);
    if (nd > kMaxDims || !scalar_type(code, q.type) || role < kInput || role > kWorkspace) return bad("bad parameter");
    q.ndim = (int)nd;
    q.role = (Role)role;
    p->n_inputs += role == kInput, p->n_outputs += role == kOutput;
    for (Py_ssize_t d = 0; d < nd; ++d) {
      PyObject* s = PyTuple_GET_ITEM(shape, d);
      if (PyUnicode_Check(s)) {
        const char* name = PyUnicode_AsUTF8(s);
        if (!name) return bad("");
        size_t k = 0;
        while (k < names.size() && names[k] != name) ++k;
        if (k == names.size()) names.push_back(name);
        if (names.size() > (size_t)kMaxSymbols) return bad("too many symbols");
        q.dim[d] = -1 - (int64_t)k;
      } else {
        q.dim[d] = PyLong_AsLongLong(s);
        if (PyErr_Occurred()) return bad("");
        if (q.dim[d] < 0) return bad("negative size");
      }
    }
  }
  return (PyObject*)p;
}

void plan_dealloc(PyObject* self) { Py_TYPE(self)->tp_free(self); }

PyMethodDef plan_methods[] = {{"launch", plan_launch, METH_VARARGS, "launch(tensors, stream): the entry point on checked tensors"},
                              {nullptr, nullptr, 0, nullptr}};

PyTypeObject PlanType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---- the helpers that are functions, not kernel objects: the same rule (NotImplemented with nothing done) -----------------
PyObject* wrap_or_raise(int rc, at::Tensor&& a) {
  if (rc != 0) {
    raise_for(rc);
    return nullptr;
  }
  return THPVariable_Wrap(std::move(a));
}
int64_t as_int(PyObject* o) { return PyLong_Check(o) ? PyLong_AsLongLong(o) : -1; }
hipStream_t current_stream(int device) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

// dequantize(packed, scales | None, zeros | None, zero, group, type code, layout)
PyObject* fn_dequantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 7) return not_ordinary();
  const double zero = PyFloat_AsDouble(a[3]);
  const int64_t group = as_int(a[4]), code = as_int(a[5]), layout = as_int(a[6]);
  at::ScalarType type;
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return not_ordinary();
  }
  if (group <= 0 || !scalar_type((int)code, type)) return not_ordinary();
  try {
    const int device = c10::hip::current_device();
    const at::Tensor* w = plain_tensor(a[0], device);
    if (!w || w->dim() != 2 || w->element_size() != 1) return not_ordinary();
    const int64_t N = w->size(0), K = 2 * w->size(1);
    const at::Tensor* g[2] = {nullptr, nullptr};
    for (int i = 0; i < 2; ++i) {
      if (a[1 + i] == Py_None) continue;
      g[i] = plain_tensor(a[1 + i], device);
      if (!g[i] || g[i]->scalar_type() != type || g[i]->dim() != 2 || g[i]->size(0) != N || g[i]->size(1) != K / group) return not_ordinary();
    }
    const int64_t shape[2] = {N, K};
    at::Tensor out = new_tensor(shape, type, device);
    int rc;
    {
      Released free_lock;
      rc = lib.tlq_dequant_w4_layout(ptr(w), ptr(g[0]), ptr(g[1]), out.data_ptr(), N, K, group, (float)zero, (int)code, (int)layout, current_stream(device));
    }
    return wrap_or_raise(rc, std::move(out));
  } catch (const std::exception&) {
    return not_ordinary();
  }
}

// unpack(packed, type code, sign mode)
PyObject* fn_unpack(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3) return not_ordinary();
  const int64_t code = as_int(a[1]), mode = as_int(a[2]);
  at::ScalarType type;
  if (!scalar_type((int)code, type)) return not_ordinary();
  try {
    const int device = c10::hip::current_device();
    const at::Tensor* w = plain_tensor(a[0], device);
    if (!w || w->dim() != 2 || w->scalar_type() != at::kByte) return not_ordinary();
    const int64_t shape[2] = {w->size(0), 2 * w->size(1)};
    at::Tensor out = new_tensor(shape, type, device);
    int rc;
    {
      Released free_lock;
      rc = lib.tlq_unpack_int4(ptr(w), out.data_ptr(), shape[0], shape[1], (int)code, (int)mode, current_stream(device));
    }
    return wrap_or_raise(rc, std::move(out));
  } catch (const std::exception&) {
    return not_ordinary();
  }
}

// pack(values, interleave code, type code of the result)
PyObject* fn_pack(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 3) return not_ordinary();
  const int64_t interleave = as_int(a[1]), code = as_int(a[2]);
  at::ScalarType type;
  if (!scalar_type((int)code, type)) return not_ordinary();
  try {
    const int device = c10::hip::current_device();
    const at::Tensor* v = plain_tensor(a[0], device);
    if (!v || v->dim() != 2 || (v->scalar_type() != at::kChar && v->scalar_type() != at::kByte)) return not_ordinary();
    const int64_t shape[2] = {v->size(0), v->size(1) / 2};
    at::Tensor out = new_tensor(shape, type, device);
    int rc;
    {
      Released free_lock;
      rc = lib.tlq_pack_int4(ptr(v), out.data_ptr(), v->size(0), v->size(1), (int)interleave, current_stream(device));
    }
    return wrap_or_raise(rc, std::move(out));
  } catch (const std::exception&) {
    return not_ordinary();
  }
}

// quantize(weights, group) -> (q - 8, scales)
PyObject* fn_quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2) return not_ordinary();
  const int64_t group = as_int(a[1]);
  if (group <= 0) return not_ordinary();
  try {
    const int device = c10::hip::current_device();
    const at::Tensor* w = plain_tensor(a[0], device);
    if (!w || w->dim() != 2 || (w->scalar_type() != at::kHalf && w->scalar_type() != at::kBFloat16)) return not_ordinary();
    const int64_t N = w->size(0), K = w->size(1);
    const int64_t shape_q[2] = {N, K}, shape_s[2] = {N, K / group};
    at::Tensor q = new_tensor(shape_q, at::kChar, device), s = new_tensor(shape_s, w->scalar_type(), device);
    int rc;
    {
      Released free_lock;
      rc = lib.tlq_quantize_sym4(ptr(w), q.data_ptr(), s.data_ptr(), N, K, group, w->scalar_type() == at::kHalf ? TLQ_F16 : TLQ_BF16, current_stream(device));
    }
    PyObject* first = wrap_or_raise(rc, std::move(q));
    PyObject* second = first ? THPVariable_Wrap(std::move(s)) : nullptr;
    if (!second) {
      Py_XDECREF(first);
      return nullptr;
    }
    PyObject* both = PyTuple_New(2);
    if (!both) {
      Py_DECREF(first), Py_DECREF(second);
      return nullptr;
    }
    PyTuple_SET_ITEM(both, 0, first), PyTuple_SET_ITEM(both, 1, second);
    return both;
  } catch (const std::exception&) {
    return not_ordinary();
  }
}

// bind({name: address}): the entry points of the loaded libtlq
PyObject* fn_bind(PyObject*, PyObject* dict) {
  if (!PyDict_Check(dict)) {
    PyErr_SetString(PyExc_TypeError, "a dict of addresses is wanted");
    return nullptr;
  }
  Entries e;
#define X(name)                                                                     \
  {                                                                                 \
    PyObject* o = PyDict_GetItemString(dict, #name);                                \
    e.name = o ? (decltype(e.name))PyLong_AsVoidPtr(o) : nullptr;                   \
    if (!e.name) {                                                                  \
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, #name);                \
      return nullptr;                                                               \
    }                                                                               \
  }
  TLQ_ENTRIES(X)
#undef X
  lib = e;
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"bind", fn_bind, METH_O, "bind({name: address}): the entry points to call"},
                         {"dequantize", (PyCFunction)(void (*)(void))fn_dequantize, METH_FASTCALL, "tlq_dequant_w4_layout"},
                         {"unpack", (PyCFunction)(void (*)(void))fn_unpack, METH_FASTCALL, "tlq_unpack_int4"},
                         {"pack", (PyCFunction)(void (*)(void))fn_pack, METH_FASTCALL, "tlq_pack_int4"},
                         {"quantize", (PyCFunction)(void (*)(void))fn_quantize, METH_FASTCALL, "tlq_quantize_sym4"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "tlq_host", "Native calls of the operators", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_tlq_host(void) {
  PlanType.tp_name = "tlq_host.Plan";
  PlanType.tp_basicsize = sizeof(PlanObject);
  PlanType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  PlanType.tp_vectorcall_offset = offsetof(PlanObject, vectorcall);
  PlanType.tp_call = PyVectorcall_Call;
  PlanType.tp_new = plan_new;
  PlanType.tp_dealloc = plan_dealloc;
  PlanType.tp_methods = plan_methods;
  if (PyType_Ready(&PlanType) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module);
  if (!m) return nullptr;
  Py_INCREF(&PlanType);
  if (PyModule_AddObject(m, "Plan", (PyObject*)&PlanType) < 0) {
    Py_DECREF(&PlanType), Py_DECREF(m);
    return nullptr;
  }
  return m;
}
