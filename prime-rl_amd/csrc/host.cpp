// The Python entry points' everyday call, in one native step: argument checks, output allocation, workspace
// lookup and the C-ABI call.  A decode-sized layer takes 10-35 us on the GPU; the same steps in Python took
// 17-39 us of host time per call, i.e. more than the kernels they launch.
//
// Every function returns the result tensor(s); None when anything about the call is out of the ordinary (a
// type, shape, device or layout it does not expect, no workspace large enough, a capture in progress), in
// which case the caller runs the Python path, which handles or names it; or a negative int, the C-ABI's error
// code.  Nothing is launched before all checks are done, so None always means nothing has happened yet.
//
// The interpreter lock is held while arguments are read and given up around every call that may block (the output's
// allocation, the launches, the capture query): a launch waits where the queue is full, and what it waits for may be
// a host callback that needs the lock.  Whatever the launches use is therefore read, or kept alive, beforehand.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <utility>
#include <vector>

#include "../../include/moe_i8.h"

namespace {

// The interpreter lock given up for a scope.
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};

// Default workspaces the Python side has made, by (device, stream); it withdraws an entry when it lets go of the
// tensor.  A call holds a reference of its own until its launches are in the stream: another thread may replace the
// entry meanwhile.  Guarded by the interpreter lock.
struct Workspace {
  int device;
  hipStream_t stream;
  at::Tensor tensor;
};
constexpr size_t kMaxWorkspaces = 64;
std::vector<Workspace>& workspaces() {
  static auto* all = new std::vector<Workspace>();  // never destroyed: the allocator may be gone by then
  return *all;
}

Workspace* find_workspace(int device, hipStream_t stream) {
  for (Workspace& w : workspaces())
    if (w.device == device && w.stream == stream) return &w;
  return nullptr;
}

// The device and stream a call runs on; false: leave it to the Python path.
struct Where {
  int device;
  hipStream_t stream;
  bool init(const at::Tensor& t) {
    device = t.get_device();
    if (device != c10::hip::current_device()) return false;
    stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    const Unlocked unlocked;
    if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    return status == hipStreamCaptureStatusNone;
  }
};

// A tensor argument: contiguous, of the type, on the GPU (of `where`, once that is known).
bool plain(PyObject* o, at::ScalarType type, const at::Tensor** out) {
  if (!THPVariable_Check(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.is_cuda() || t.scalar_type() != type || !t.is_contiguous()) return false;
  *out = &t;
  return true;
}

at::Tensor make(at::IntArrayRef sizes, at::ScalarType type, const Where& at) {
  return at::empty(sizes, at::TensorOptions().dtype(type).device(at::Device(at::kCUDA, (c10::DeviceIndex)at.device)));
}

// A caller's workspace, or the default one of the stream.
struct Scratch {
  at::Tensor keep;
  char* data;
  int64_t bytes;
  bool init(PyObject* o, const Where& at, int64_t need) {
    if (o == Py_None) {
      const Workspace* w = find_workspace(at.device, at.stream);
      if (!w) return false;
      keep = w->tensor;
    } else {
      if (!THPVariable_Check(o)) return false;
      keep = THPVariable_Unpack(o);
      if (!keep.is_cuda() || keep.get_device() != at.device || !keep.is_contiguous()) return false;
    }
    bytes = (int64_t)keep.nbytes();
    if (bytes < need) return false;
    data = static_cast<char*>(keep.data_ptr());
    return true;
  }
};

template <class T>
T* data(const at::Tensor* t) {
  return t ? static_cast<T*>(t->data_ptr()) : nullptr;
}

// An int that the C-ABI's 32 bits hold.
bool as_int(PyObject* o, int64_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return !overflow && *v >= INT32_MIN && *v <= INT32_MAX;
}

// A switch that is True or False; any other value's truth is for the Python path to ask.
bool as_bool(PyObject* o, bool* v) {
  *v = o == Py_True;
  return PyBool_Check(o);
}

// [N, K] int8 weights, contiguous or as the transposed [K, N] view of such a tensor, with N scales.
bool dense_weight(PyObject* wo, PyObject* so, const at::Tensor** w, const at::Tensor** s, int64_t* n, int64_t* k) {
  if (!THPVariable_Check(wo)) return false;
  const at::Tensor& t = THPVariable_Unpack(wo);
  if (!t.is_cuda() || t.scalar_type() != at::kChar || t.dim() != 2) return false;
  if (t.is_contiguous()) {
    *n = t.size(0), *k = t.size(1);
  } else if (t.stride(0) == 1 && t.stride(1) == t.size(0)) {
    *n = t.size(1), *k = t.size(0);
  } else {
    return false;
  }
  *w = &t;
  return plain(so, at::kFloat, s) && (*s)->numel() == *n;
}

#define MOE_I8_ARGS(count) \
  if (nargs != count) { PyErr_SetString(PyExc_TypeError, "wrong number of arguments"); return nullptr; }

PyObject* wrap_guarded(PyObject* (*fn)(PyObject* const*, Py_ssize_t), PyObject* const* args, Py_ssize_t nargs) {
  try {
    return fn(args, nargs);
  } catch (const std::exception&) {  // as torch's own bindings raise it: an allocation that fails is an OutOfMemoryError
    torch::translate_exception_to_python(std::current_exception());
    return nullptr;
  }
}
template <PyObject* (*fn)(PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  return wrap_guarded(fn, args, nargs);
}

// remember(device, stream, tensor): the default workspace of (device, stream) is now this one.
PyObject* remember(PyObject* const* args, Py_ssize_t nargs) {
  MOE_I8_ARGS(3);
  const long long d = PyLong_AsLongLong(args[0]);
  void* s = PyLong_AsVoidPtr(args[1]);
  if (PyErr_Occurred()) return nullptr;
  if (!THPVariable_Check(args[2])) {
    PyErr_SetString(PyExc_TypeError, "a workspace is a tensor");
    return nullptr;
  }
  const at::Tensor& t = THPVariable_Unpack(args[2]);
  if (Workspace* w = find_workspace((int)d, (hipStream_t)s)) {
    w->tensor = t;
  } else if (workspaces().size() < kMaxWorkspaces) {
    workspaces().push_back({(int)d, (hipStream_t)s, t});
  }
  Py_RETURN_NONE;
}

// forget(device, stream)
PyObject* forget(PyObject* const* args, Py_ssize_t nargs) {
  MOE_I8_ARGS(2);
  const long long d = PyLong_AsLongLong(args[0]);
  void* s = PyLong_AsVoidPtr(args[1]);
  if (PyErr_Occurred()) return nullptr;
  if (Workspace* w = find_workspace((int)d, (hipStream_t)s)) {
    std::swap(*w, workspaces().back());
    const at::Tensor last = std::move(workspaces().back().tensor);  // let go of once the table is in order again
    workspaces().pop_back();
  }
  Py_RETURN_NONE;
}

// linear(input, weight, weight_scale, variant, workspace)
PyObject* linear(PyObject* const* args, Py_ssize_t nargs) {
  MOE_I8_ARGS(5);
  const at::Tensor *x, *w, *s;
  int64_t n, k, variant;
  Where at;
  Scratch ws;
  if (!plain(args[0], at::kBFloat16, &x) || !dense_weight(args[1], args[2], &w, &s, &n, &k) || !as_int(args[3], &variant) ||
      x->dim() < 1 || x->size(-1) != k || k == 0 || n > INT32_MAX || k > INT32_MAX || !at.init(*x) ||
      w->get_device() != at.device || s->get_device() != at.device)
    Py_RETURN_NONE;
  const int64_t m = x->numel() / k;
  if (m == 0 || !ws.init(args[4], at, moe_i8_dense_workspace_bytes(m, (int)k, 0))) Py_RETURN_NONE;
  c10::SmallVector<int64_t, 4> shape(x->sizes().begin(), x->sizes().end());
  shape.back() = n;
  const void* xp = data<void>(x);
  const int8_t* wp = data<int8_t>(w);
  const float* sp = data<float>(s);
  at::Tensor out;
  int rc;
  {
    const Unlocked unlocked;
    out = make(shape, at::kBFloat16, at);
    rc = moe_i8_w8a8_linear(xp, wp, sp, out.data_ptr(), m, (int)n, (int)k, ws.data, ws.bytes, (int)variant, at.stream);
  }
  return rc ? PyLong_FromLong(rc) : THPVariable_Wrap(std::move(out));
}

// mlp(x, w13, w13_scale, w2, w2_scale, variant, workspace)
PyObject* mlp(PyObject* const* args, Py_ssize_t nargs) {
  MOE_I8_ARGS(7);
  const at::Tensor *x, *w13, *s13, *w2, *s2;
  int64_t two_i, h, h2, i, variant;
  Where at;
  Scratch ws;
  if (!plain(args[0], at::kBFloat16, &x) || !dense_weight(args[1], args[2], &w13, &s13, &two_i, &h) ||
      !dense_weight(args[3], args[4], &w2, &s2, &h2, &i) || !as_int(args[5], &variant) || x->dim() < 1 || two_i != 2 * i ||
      h2 != h || h == 0 || x->size(-1) != h || h > INT32_MAX || two_i > INT32_MAX || !at.init(*x) ||
      w13->get_device() != at.device || s13->get_device() != at.device || w2->get_device() != at.device ||
      s2->get_device() != at.device)
    Py_RETURN_NONE;
  const int64_t m = x->numel() / h;
  if (m == 0 || !ws.init(args[6], at, moe_i8_dense_workspace_bytes(m, (int)h, (int)i))) Py_RETURN_NONE;
  const c10::SmallVector<int64_t, 4> shape(x->sizes().begin(), x->sizes().end());
  const void* xp = data<void>(x);
  const int8_t *w13p = data<int8_t>(w13), *w2p = data<int8_t>(w2);
  const float *s13p = data<float>(s13), *s2p = data<float>(s2);
  at::Tensor out;
  int rc;
  {
    const Unlocked unlocked;
    out = make(shape, at::kBFloat16, at);
    rc = moe_i8_w8a8_mlp(xp, w13p, s13p, w2p, s2p, out.data_ptr(), m, (int)h, (int)i, ws.data, ws.bytes, (int)variant, at.stream);
  }
  return rc ? PyLong_FromLong(rc) : THPVariable_Wrap(std::move(out));
}

// The layer's tensors, checked against each other.
struct Layer {
  const at::Tensor *x, *w1, *w2, *s1, *s2;
  int64_t m, e, h, i;
  Where at;
  bool init(PyObject* xo, PyObject* w1o, PyObject* w2o, PyObject* s1o, PyObject* s2o) {
    if (!plain(xo, at::kBFloat16, &x) || !plain(w1o, at::kChar, &w1) || !plain(w2o, at::kChar, &w2) ||
        !plain(s1o, at::kFloat, &s1) || !plain(s2o, at::kFloat, &s2) || x->dim() != 2 || w1->dim() != 3 || w2->dim() != 3)
      return false;
    m = x->size(0), h = x->size(1), e = w1->size(0), i = w1->size(1) / 2;
    if (m == 0 || w1->size(1) % 2 || w1->size(2) != h || w2->size(0) != e || w2->size(1) != h || w2->size(2) != i ||
        s1->numel() != e * 2 * i || s2->numel() != e * h || e < 1 || e > MOE_I8_MAX_EXPERTS || h % 64 || i % 64 || h > INT32_MAX ||
        i > INT32_MAX / 2 || !at.init(*x))
      return false;
    for (const at::Tensor* t : {w1, w2, s1, s2})
      if (t->get_device() != at.device) return false;
    return true;
  }
  // `out`: None (a new tensor, made with the launches; the input itself if `inplace`) or the tensor to write
  bool output(PyObject* o, bool inplace, at::Tensor* out) const {
    if (o == Py_None) {
      if (inplace) *out = *x;
      return true;
    }
    const at::Tensor* t;
    if (!plain(o, at::kBFloat16, &t) || t->sizes() != x->sizes() || t->get_device() != at.device) return false;
    *out = *t;
    return true;
  }
};

// experts(hidden, w1, w2, topk_weights, topk_ids, w1_scale, w2_scale, block, variant, inplace, out, workspace)
PyObject* experts(PyObject* const* args, Py_ssize_t nargs) {
  MOE_I8_ARGS(12);
  Layer l;
  const at::Tensor *tw, *ids;
  int64_t block, variant;
  bool inplace;
  Scratch ws;
  at::Tensor out;
  if (!l.init(args[0], args[1], args[2], args[5], args[6]) || !plain(args[3], at::kFloat, &tw) || !plain(args[4], at::kInt, &ids) ||
      !as_int(args[7], &block) || !as_int(args[8], &variant) || !as_bool(args[9], &inplace) || ids->dim() != 2 ||
      ids->size(0) != l.m || tw->sizes() != ids->sizes() || tw->get_device() != l.at.device || ids->get_device() != l.at.device ||
      ids->size(1) < 1 || ids->size(1) > l.e)
    Py_RETURN_NONE;
  const int k = (int)ids->size(1);
  const int64_t need = moe_i8_workspace_bytes(l.m, k, (int)l.e, (int)l.h, (int)l.i, (int)block);
  if (need < 0 || !ws.init(args[11], l.at, need) || !l.output(args[10], inplace, &out)) Py_RETURN_NONE;
  const void* xp = data<void>(l.x);
  const int8_t *w1 = data<int8_t>(l.w1), *w2 = data<int8_t>(l.w2);
  const float *twp = data<float>(tw), *s1 = data<float>(l.s1), *s2 = data<float>(l.s2);
  const int32_t* idp = data<int32_t>(ids);
  int rc;
  {
    const Unlocked unlocked;
    if (!out.defined()) out = make({l.m, l.h}, at::kBFloat16, l.at);
    rc = moe_i8_fused_experts(xp, w1, w2, twp, idp, s1, s2, out.data_ptr(), l.m, k, (int)l.e, (int)l.h, (int)l.i, (int)block,
                              ws.data, ws.bytes, (int)variant, l.at.stream);
  }
  return rc ? PyLong_FromLong(rc) : THPVariable_Wrap(std::move(out));
}

// The router's arguments: (logits, top_k, score_func, renormalize, scale, bias, groups, topk_groups, top2,
// record, layer), in this order from `a` on.
struct Router {
  const at::Tensor* logits;
  const at::Tensor* bias = nullptr;
  const at::Tensor* record = nullptr;
  int64_t m, e, k, score, renormalize, groups, topk_groups, top2, layer = 0;
  double scale;
  bool init(PyObject* const* a) {
    if (!plain(a[0], at::kFloat, &logits) || logits->dim() != 2 || !as_int(a[1], &k) || !as_int(a[2], &score) ||
        !as_int(a[3], &renormalize) || !PyFloat_CheckExact(a[4]) || !as_int(a[6], &groups) || !as_int(a[7], &topk_groups) ||
        !as_int(a[8], &top2) || k < 1 || k > 64)
      return false;
    scale = PyFloat_AS_DOUBLE(a[4]);
    m = logits->size(0), e = logits->size(1);
    if (m == 0 || e < 1 || e > MOE_I8_MAX_EXPERTS || k > e || groups > e || topk_groups > e) return false;
    if (a[5] != Py_None && (!plain(a[5], at::kFloat, &bias) || bias->numel() != e || bias->get_device() != logits->get_device()))
      return false;
    if (a[9] != Py_None) {
      if (!THPVariable_Check(a[9]) || !as_int(a[10], &layer)) return false;
      record = &THPVariable_Unpack(a[9]);
      if (!record->is_cuda() || !record->is_contiguous() || record->get_device() != logits->get_device() ||
          (record->scalar_type() != at::kByte && record->scalar_type() != at::kUInt16) || record->dim() != 3 ||
          record->size(0) != m || record->size(2) != k || layer < 0 || layer >= record->size(1))
        return false;
    }
    return true;
  }
  int record_dtype() const { return record ? (record->scalar_type() == at::kByte ? 1 : 2) : 0; }
  int64_t record_stride() const { return record ? record->size(1) * k : 0; }
  int64_t record_offset() const { return record ? layer * k : 0; }
};

// route(<router>) -> (weights, ids)
PyObject* route(PyObject* const* args, Py_ssize_t nargs) {
  MOE_I8_ARGS(11);
  Router r;
  Where at;
  if (!r.init(args) || !at.init(*r.logits)) Py_RETURN_NONE;
  const float *logits = data<float>(r.logits), *bias = data<float>(r.bias);
  void* record = data<void>(r.record);
  const int record_dtype = r.record_dtype();
  const int64_t stride = r.record_stride(), offset = r.record_offset();
  at::Tensor weights, ids;
  int rc;
  {
    const Unlocked unlocked;
    weights = make({r.m, r.k}, at::kFloat, at);
    ids = make({r.m, r.k}, at::kInt, at);
    rc = moe_i8_route_topk(logits, r.m, (int)r.e, (int)r.k, (int)r.score, bias, (int)r.groups, (int)r.topk_groups, (int)r.top2,
                           (int)r.renormalize, (float)r.scale, static_cast<float*>(weights.data_ptr()),
                           static_cast<int32_t*>(ids.data_ptr()), record, record_dtype, stride, offset, at.stream);
  }
  if (rc) return PyLong_FromLong(rc);
  PyObject* w = THPVariable_Wrap(std::move(weights));
  PyObject* i = THPVariable_Wrap(std::move(ids));
  PyObject* both = w && i ? PyTuple_Pack(2, w, i) : nullptr;
  Py_XDECREF(w);
  Py_XDECREF(i);
  return both;
}

// moe(hidden, w1, w2, w1_scale, w2_scale, block, variant, inplace, workspace, <router>): router, then experts.
// The routing stays in the workspace, behind what the layer needs.  False: only a default workspace of that
// size is missing.
PyObject* moe(PyObject* const* args, Py_ssize_t nargs) {
  MOE_I8_ARGS(20);
  Layer l;
  Router r;
  int64_t block, variant;
  bool inplace;
  Scratch ws;
  at::Tensor out;
  if (!l.init(args[0], args[1], args[2], args[3], args[4]) || !as_int(args[5], &block) || !as_int(args[6], &variant) ||
      !as_bool(args[7], &inplace) ||
      !r.init(args + 9) || r.m != l.m || r.e != l.e || r.logits->get_device() != l.at.device)
    Py_RETURN_NONE;
  const int64_t need = moe_i8_workspace_bytes(l.m, (int)r.k, (int)l.e, (int)l.h, (int)l.i, (int)block);
  if (need < 0) Py_RETURN_NONE;
  if (!ws.init(args[8], l.at, need + 8 * l.m * r.k)) {
    if (args[8] == Py_None) Py_RETURN_FALSE;
    Py_RETURN_NONE;
  }
  if (!l.output(Py_None, inplace, &out)) Py_RETURN_NONE;
  float* weights = reinterpret_cast<float*>(ws.data + need);
  int32_t* ids = reinterpret_cast<int32_t*>(weights + l.m * r.k);
  const void* xp = data<void>(l.x);
  const int8_t *w1 = data<int8_t>(l.w1), *w2 = data<int8_t>(l.w2);
  const float *s1 = data<float>(l.s1), *s2 = data<float>(l.s2), *logits = data<float>(r.logits), *bias = data<float>(r.bias);
  void* record = data<void>(r.record);
  const int record_dtype = r.record_dtype();
  const int64_t stride = r.record_stride(), offset = r.record_offset();
  int rc;
  {
    const Unlocked unlocked;
    if (!out.defined()) out = make({l.m, l.h}, at::kBFloat16, l.at);
    rc = moe_i8_fused_moe(xp, logits, w1, w2, s1, s2, out.data_ptr(), l.m, (int)r.k, (int)l.e, (int)l.h, (int)l.i, (int)block,
                          (int)r.score, bias, (int)r.groups, (int)r.topk_groups, (int)r.top2, (int)r.renormalize, (float)r.scale,
                          weights, ids, record, record_dtype, stride, offset, ws.data, ws.bytes, (int)variant, l.at.stream);
  }
  return rc ? PyLong_FromLong(rc) : THPVariable_Wrap(std::move(out));
}

// requantise(gate, up, down, w13, w13_scale, w2, w2_scale) -> True
PyObject* requantise(PyObject* const* args, Py_ssize_t nargs) {
  MOE_I8_ARGS(7);
  const at::Tensor *g, *u, *d, *w13, *s13, *w2, *s2;
  Where at;
  if (!plain(args[0], at::kBFloat16, &g) || !plain(args[1], at::kBFloat16, &u) || !plain(args[2], at::kBFloat16, &d) ||
      !plain(args[3], at::kChar, &w13) || !plain(args[4], at::kFloat, &s13) || !plain(args[5], at::kChar, &w2) ||
      !plain(args[6], at::kFloat, &s2) || g->dim() != 3 || d->dim() != 3 || w13->dim() != 3 || u->sizes() != g->sizes())
    Py_RETURN_NONE;
  const int64_t e = g->size(0), i = g->size(1), h = g->size(2);
  if (e == 0 || i == 0 || h == 0 || h % 8 || i % 8 || d->size(0) != e || d->size(1) != h || d->size(2) != i || w13->size(0) != e ||
      w13->size(1) != 2 * i || w13->size(2) != h || w2->sizes() != d->sizes() || s13->numel() != e * 2 * i || s2->numel() != e * h ||
      !at.init(*g))
    Py_RETURN_NONE;
  for (const at::Tensor* t : {u, d, w13, s13, w2, s2})
    if (t->get_device() != at.device) Py_RETURN_NONE;
  const void *gp = data<void>(g), *up = data<void>(u), *dp = data<void>(d);
  int8_t *w13p = data<int8_t>(w13), *w2p = data<int8_t>(w2);
  float *s13p = data<float>(s13), *s2p = data<float>(s2);
  int rc;
  {
    const Unlocked unlocked;
    rc = moe_i8_quant_expert_weights(gp, up, dp, MOE_I8_DTYPE_BF16, e, i, h, w13p, s13p, w2p, s2p, at.stream);
  }
  if (rc) return PyLong_FromLong(rc);
  Py_RETURN_TRUE;
}

PyMethodDef kMethods[] = {
    {"remember", (PyCFunction)(void*)guarded<remember>, METH_FASTCALL, nullptr},
    {"forget", (PyCFunction)(void*)guarded<forget>, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void*)guarded<linear>, METH_FASTCALL, nullptr},
    {"mlp", (PyCFunction)(void*)guarded<mlp>, METH_FASTCALL, nullptr},
    {"experts", (PyCFunction)(void*)guarded<experts>, METH_FASTCALL, nullptr},
    {"route", (PyCFunction)(void*)guarded<route>, METH_FASTCALL, nullptr},
    {"moe", (PyCFunction)(void*)guarded<moe>, METH_FASTCALL, nullptr},
    {"requantise", (PyCFunction)(void*)guarded<requantise>, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
  PyObject* m = PyModule_Create(&kModule);
  if (m && PyModule_AddStringConstant(m, "torch_version", MOE_I8_TORCH_VERSION) == 0) return m;
  Py_XDECREF(m);
  return nullptr;
}
