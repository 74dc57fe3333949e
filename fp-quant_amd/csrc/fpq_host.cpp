// The eager calls of the quantized layers without the interpreter between their one to three launches.
//
// What bounds a decode step is the host: one layer is 8 us of kernels behind 25 us of Python (attribute lookups on the
// module, tensor constructors, two foreign calls of eleven to fourteen arguments, the checks of every cached constant),
// a fused decoder block of one token 52 us of kernels behind 170, a quantize operator 6 us behind 18 (most of it
// operator dispatch).  On this path they take 8.7, 36 and 6.9 us from call to call: a layer of few rows is one launch
// (fpq_linear_rows, 4.8 us), the rest of its time three allocations, what publish() makes and the module call around
// them; with more rows it is two launches of 3.3 us (32 rows, 14336 -> 4096: 13.2 us).  Here the same sequence -- checks,
// allocations, launches, the hand-over of quantized activations between layers that share an input -- runs as native code
// on constants that the Python path has worked out once and left in plans (module/host.py):
//
//   QuantPlan   on a rotation matrix: its kind, norm and size, the activation scale as fp32
//   LinearPlan  on a layer's code tensor: its packed operands, alpha, bias and split-K workspace size
//   GroupPlan   on a WeightGroup: the same for layers whose packed weights lie end to end
//
// A plan states the tensors it was made from (object, address, modification counter), and every call compares them.
// Every function here returns None (False where a plan is missing or outdated and may be made), having launched nothing
// that is not repeated, whenever a call is not the plain one (tracing, gradients, tensor subclasses, modes, another
// device, strides): the caller then takes the Python path, which is the definition of the result and makes the plans anew.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/InferenceMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <structmember.h>

#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../include/fpq.h"

namespace {

// ---- the library: the entry points of the build that the ctypes binding has loaded
#define FPQ_ENTRIES(X)                                                                                       \
  X(fpq_stream_capture_id) X(fpq_quantize_mx) X(fpq_quantize_mx_quest) X(fpq_quantize_nv) X(fpq_pack_padded)          \
  X(fpq_gemm_mxf4) X(fpq_gemm_nvf4) X(fpq_linear_rows)                                                                          \
  X(fpq_quantize_mx_packed_padded) X(fpq_quantize_nv_packed_padded)                 \
  X(fpq_gemm_mxf4_packed) X(fpq_gemm_mxf4_packed_residual) X(fpq_gemm_mxf4_packed_splitk)                    \
  X(fpq_gemm_mxf4_packed_multi) X(fpq_gemm_nvf4_packed) X(fpq_gemm_nvf4_packed_residual)                     \
  X(fpq_gemm_nvf4_packed_splitk) X(fpq_gemm_nvf4_packed_multi) X(fpq_rmsnorm_rows_quantize_mx_packed)        \
  X(fpq_rmsnorm_tile_quantize_mx_packed) X(fpq_rmsnorm_rows_quantize_nv_packed)                              \
  X(fpq_rmsnorm_tile_quantize_nv_packed) X(fpq_silu_mul_quantize_mx_packed) X(fpq_silu_mul_quantize_nv_packed) \
  X(fpq_gemm_packed_gated) X(fpq_gemm_packed_gated_takes) X(fpq_norm_rows_multi)
enum Entry {
#define X(name) E_##name,
  FPQ_ENTRIES(X)
#undef X
  kEntries
};
const char* const kEntryNames[kEntries] = {
#define X(name) #name,
    FPQ_ENTRIES(X)
#undef X
};
void* g_fn[kEntries];
PyObject* g_entry_name[kEntries];
PyObject* g_entry_object[kEntries];   // the binding's function objects as they were at start-up
PyObject* g_binding;                  // the binding's attributes
#define FPQ_CALL(name) reinterpret_cast<decltype(&name)>(g_fn[E_##name])

// A binding whose entry has been replaced (instrumented) is called through Python.
bool plain_entry(int e) { return PyDict_GetItem(g_binding, g_entry_name[e]) == g_entry_object[e]; }

PyObject* g_shared;           // device index -> the activations of the latest call (eager._shared_activations)
PyObject* g_workspaces;       // device index -> {stream: workspace} (hip_ops._stream_workspaces)
PyObject* g_eager_globals;    // eager.SHARE_ACT_QUANT is read from here on every call
PyTypeObject* g_activations;  // eager.QuantizedActivations
int g_policy, g_packed_rows_mx, g_packed_rows_nv, g_linear_rows_mx;

PyObject *s_qweight, *s_scales, *s_wgs, *s_ags, *s_h, *s_bias, *s_plan, *s_qplan, *s_alpha, *s_packed, *s_share,
    *s_parameters, *s_buffers, *s_weight, *s_eps, *s_rotation, *s_splitk;

// ---- tensors
const at::Tensor* tensor_of(PyObject* o) { return o && THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

// A dense tensor on a GPU without anything wrapped around it (batching, functionalization, Python dispatch).
bool plain_cuda(const at::Tensor& t) {
  if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || !t.has_storage() || t.is_neg() || t.is_conj())
    return false;
  const auto ks = t.key_set();
  return !ks.has(c10::DispatchKey::Python) && !ks.has(c10::DispatchKey::FuncTorchBatched) &&
         !ks.has(c10::DispatchKey::FuncTorchGradWrapper) && !ks.has(c10::DispatchKey::Functionalize);
}

struct Key {   // a tensor as it was when a plan was made
  const void* impl = nullptr;
  const void* ptr = nullptr;
  uint32_t version = 0;
  at::Tensor held;   // keeps the object (not for the tensor that the plan hangs on)
  bool take(PyObject* o, bool hold) {
    if (o == Py_None) return true;
    const at::Tensor* t = tensor_of(o);
    if (!t || !plain_cuda(*t) || t->is_inference()) return false;
    impl = t->unsafeGetTensorImpl();
    ptr = t->const_data_ptr();
    version = (uint32_t)t->_version();
    if (hold) held = *t;
    return true;
  }
  bool is(PyObject* o) const {
    if (!o || o == Py_None) return impl == nullptr;
    const at::Tensor* t = tensor_of(o);
    return t && t->unsafeGetTensorImpl() == impl && t->const_data_ptr() == ptr && (uint32_t)t->_version() == version;
  }
};

PyObject* attribute(PyObject* tensor, PyObject* name) {   // borrowed, or null
  PyObject** d = _PyObject_GetDictPtr(tensor);
  return d && *d ? PyDict_GetItem(*d, name) : nullptr;
}

PyObject* member(PyObject* params, PyObject* buffers, PyObject* name) {   // borrowed, or null
  PyObject* o = PyDict_GetItem(params, name);
  return o ? o : PyDict_GetItem(buffers, name);
}

at::Tensor empty(at::IntArrayRef sizes, at::ScalarType type, c10::Device dev) {
  return at::Tensor(at::detail::empty_cuda(sizes, type, dev, std::nullopt));
}

// ---- plans
struct QuantPlan {
  PyObject_HEAD
  struct Body {
    Key h, ags;
    int kind, g;
    float norm;
    bool nvfp4, usable;
    at::Tensor gs;
    PyObject *rot, *gs_host;
  }* b;
};
struct LinearPlan {
  PyObject_HEAD
  struct Body {
    Key qweight, scales, wgs, ags, bias;
    PyObject *packed, *alpha_obj;
    at::Tensor wp, wsp, alpha;
    int64_t n, k, kp, need, split_rows, min_rows;
    bool nvfp4, packed_only, usable;
  }* b;
};
struct GroupPlan {
  PyObject_HEAD
  struct Body {
    std::vector<Key> members;   // qweight, scales, bias of each
    std::vector<int64_t> splits;
    Key wgs, ags;
    PyObject* alpha_obj;
    at::Tensor wp, wsp, alpha, bias;
    int64_t k, kp;
    bool nvfp4, usable;
  }* b;
};

template <class P>
PyObject* plan_new(PyTypeObject* type, PyObject*, PyObject*) {
  P* self = (P*)type->tp_alloc(type, 0);
  if (self) self->b = new (typename std::remove_pointer<decltype(self->b)>::type)();
  return (PyObject*)self;
}
PyObject* plan_reduce(PyObject*, PyObject*) { return Py_BuildValue("(O())", (PyObject*)Py_TYPE(Py_None)); }
PyMethodDef plan_methods[] = {{"__reduce__", plan_reduce, METH_NOARGS, "plans are not copied or stored"},
                              {nullptr, nullptr, 0, nullptr}};

void quant_dealloc(PyObject* o) {
  auto* b = ((QuantPlan*)o)->b;
  if (b) { Py_XDECREF(b->rot); Py_XDECREF(b->gs_host); delete b; }
  Py_TYPE(o)->tp_free(o);
}
void linear_dealloc(PyObject* o) {
  auto* b = ((LinearPlan*)o)->b;
  if (b) { Py_XDECREF(b->packed); Py_XDECREF(b->alpha_obj); delete b; }
  Py_TYPE(o)->tp_free(o);
}
void group_dealloc(PyObject* o) {
  auto* b = ((GroupPlan*)o)->b;
  if (b) { Py_XDECREF(b->alpha_obj); delete b; }
  Py_TYPE(o)->tp_free(o);
}
PyTypeObject QuantPlanType = {PyVarObject_HEAD_INIT(nullptr, 0) "fp_quant._lib._fpq_host.QuantPlan"};
PyTypeObject LinearPlanType = {PyVarObject_HEAD_INIT(nullptr, 0) "fp_quant._lib._fpq_host.LinearPlan"};
PyTypeObject GroupPlanType = {PyVarObject_HEAD_INIT(nullptr, 0) "fp_quant._lib._fpq_host.GroupPlan"};

bool take_tensor(PyObject* o, at::Tensor& out) {
  if (o == Py_None) return true;
  const at::Tensor* t = tensor_of(o);
  if (!t || !plain_cuda(*t) || !t->is_contiguous()) return false;
  out = *t;
  return true;
}

// ---- quantized activations of one [m, k] tensor (the base of eager.QuantizedActivations, which documents them)
struct Activations {
  PyObject_HEAD
  PyObject *m, *k, *nvfp4, *ref, *version, *key, *keep, *mx_packed, *row_major, *nv_packed;
};
PyMemberDef activation_members[] = {
#define X(name) {#name, T_OBJECT, offsetof(Activations, name), 0, nullptr}
    X(m), X(k), X(nvfp4), X(ref), X(version), X(key), X(keep), X(mx_packed), X(row_major), X(nv_packed),
#undef X
    {nullptr, 0, 0, 0, nullptr}};
void activations_dealloc(PyObject* o) {
  auto* a = (Activations*)o;
  Py_CLEAR(a->m); Py_CLEAR(a->k); Py_CLEAR(a->nvfp4); Py_CLEAR(a->ref); Py_CLEAR(a->version); Py_CLEAR(a->key);
  Py_CLEAR(a->keep); Py_CLEAR(a->mx_packed); Py_CLEAR(a->row_major); Py_CLEAR(a->nv_packed);
  Py_TYPE(o)->tp_free(o);
}
PyTypeObject ActivationsType = {PyVarObject_HEAD_INIT(nullptr, 0) "fp_quant._lib._fpq_host.Activations"};

// Codes and scales in the packed layout, held for the length of a call.
struct Packed {
  at::Tensor codes, scales;
};

// The source of a shared quantization died: nobody can ask for it any more.
PyObject* source_died(PyObject* device, PyObject* ref) {
  PyObject* slot = PyDict_GetItem(g_shared, device);
  if (slot && PyObject_TypeCheck(slot, &ActivationsType) && ((Activations*)slot)->ref == ref)
    if (PyDict_DelItem(g_shared, device) < 0) PyErr_Clear();
  Py_RETURN_NONE;
}
PyMethodDef source_died_def = {"source_died", source_died, METH_O, nullptr};

struct Call {   // where a call runs
  c10::DeviceIndex dev;
  hipStream_t stream;
  unsigned long long capture;   // of the graph being recorded, 0: none
};

// Whether `x` is an input that the plain path takes; fills `call`.
bool plain_call(const at::Tensor& x, Call& call, at::ScalarType type = at::kBFloat16) {
  if (!g_binding || !plain_cuda(x) || x.scalar_type() != type || !x.is_contiguous() || x.dim() < 1 || x.numel() == 0 ||
      x.requires_grad() || (x.is_inference() && !c10::InferenceMode::is_enabled()))
    return false;
  if (at::impl::PythonTorchFunctionTLS::stack_len() > 0 || c10::impl::TorchDispatchModeTLS::stack_len() > 0) return false;
  if (c10::impl::tls_local_dispatch_key_set().included_.has(c10::DispatchKey::Tracer)) return false;   // (torch.jit.trace)
  call.dev = x.device().index();
  if (c10::hip::current_device() != call.dev) return false;
  call.stream = c10::hip::getCurrentHIPStream(call.dev).stream();
  call.capture = 0;
  return plain_entry(E_fpq_stream_capture_id) && FPQ_CALL(fpq_stream_capture_id)(call.stream, &call.capture) == 0;
}

QuantPlan::Body* quant_plan(PyObject* h, PyObject* ags, bool nvfp4) {   // whatever is current, usable or not
  PyObject* p = attribute(h, s_qplan);
  if (!p || Py_TYPE(p) != &QuantPlanType) return nullptr;
  auto* b = ((QuantPlan*)p)->b;
  return b->nvfp4 == nvfp4 && b->h.is(h) && (!nvfp4 || b->ags.is(ags)) ? b : nullptr;
}

// What two calls must agree on to share quantized activations, as eager._sharing_key states it; null: error.
PyObject* sharing_key(const QuantPlan::Body& q, int64_t m, int64_t k, const Call& call, bool quest) {
  return Py_BuildValue("(OOKK(LL)O)", q.rot, q.nvfp4 ? q.gs_host : Py_None, (unsigned long long)(uintptr_t)call.stream,
                       call.capture, (long long)m, (long long)k, quest ? Py_True : Py_False);
}
bool sharing_enabled(const QuantPlan::Body& q, bool& declined) {
  PyObject* on = PyDict_GetItem(g_eager_globals, s_share);
  if (on != Py_True) return false;
  if (c10::InferenceMode::is_enabled()) return false;
  if (q.nvfp4 && q.gs_host == Py_None) declined = true;   // (the plan was made while sharing was off)
  return true;
}

// Steals `key`.
bool publish(PyObject* src, const at::Tensor& t, PyObject* key, PyObject* keep, const Packed& p, int64_t m, int64_t k,
             bool nvfp4, const Call& call) {
  PyObject* dev = PyLong_FromLong(call.dev);
  auto* a = (Activations*)g_activations->tp_alloc(g_activations, 0);
  PyObject* died = dev ? PyCFunction_New(&source_died_def, dev) : nullptr;
  bool ok = a && died;
  if (ok) {
    a->key = key;
    a->m = PyLong_FromLongLong(m);
    a->k = PyLong_FromLongLong(k);
    a->nvfp4 = Py_NewRef(nvfp4 ? Py_True : Py_False);
    a->version = PyLong_FromUnsignedLong((unsigned long)t._version());
    a->keep = Py_NewRef(keep);
    a->ref = PyWeakref_NewRef(src, died);
    (nvfp4 ? a->nv_packed : a->mx_packed) = Py_BuildValue("(NN)", THPVariable_Wrap(p.codes), THPVariable_Wrap(p.scales));
    ok = a->m && a->k && a->version && a->ref && (nvfp4 ? a->nv_packed : a->mx_packed) &&
         PyDict_SetItem(g_shared, dev, (PyObject*)a) == 0;
  } else {
    Py_DECREF(key);
  }
  Py_XDECREF(a);
  Py_XDECREF(died);
  Py_XDECREF(dev);
  return ok;
}

// The quantized buffers that publish() hands on hold rows of a whole 32-row tile.
Packed packed_buffers(int64_t m, int64_t k, bool nvfp4, c10::DeviceIndex dev) {
  const int64_t rows = (m + 31) / 32 * 32, kp = (k + 255) / 256 * 256;
  const c10::Device d(c10::kCUDA, dev);
  return Packed{empty({rows * kp / 2}, at::kByte, d), empty({rows * kp / (nvfp4 ? 16 : 32)}, at::kByte, d)};
}

struct NoGil {
  PyThreadState* s = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(s); }
};

// The quantized form of `src` that an earlier call left: 1 found, 2 none (`key`, if set: what to publish one under),
// 0 not the plain path, -1 Python error
int shared_activations(QuantPlan::Body& q, PyObject* src, const at::Tensor& x, int64_t m, int64_t k, bool quest,
                       const Call& call, Packed& out, PyObject*& key) {
  bool declined = false;
  key = nullptr;
  if (sharing_enabled(q, declined)) {
    if (declined) return 0;
    key = sharing_key(q, m, k, call, quest);
    if (!key) return -1;
    PyObject* dev = PyLong_FromLong(call.dev);
    PyObject* slot = dev ? PyDict_GetItem(g_shared, dev) : nullptr;
    Py_XDECREF(dev);
    if (slot && PyObject_TypeCheck(slot, &ActivationsType)) {
      auto* a = (Activations*)slot;
      if (a->ref && PyWeakref_CheckRef(a->ref) && PyWeakref_GET_OBJECT(a->ref) == src && a->version && a->key &&
          PyLong_Check(a->version) && PyLong_AsUnsignedLong(a->version) == (unsigned long)x._version()) {
        const int same = PyObject_RichCompareBool(a->key, key, Py_EQ);
        if (same < 0) { Py_CLEAR(key); return -1; }
        if (same) {
          PyObject* form = q.nvfp4 ? a->nv_packed : a->mx_packed;
          Py_CLEAR(key);
          if (!form || !PyTuple_Check(form) || PyTuple_GET_SIZE(form) != 2) return 0;   // (row-major: re-tiled there)
          const at::Tensor *c = tensor_of(PyTuple_GET_ITEM(form, 0)), *s = tensor_of(PyTuple_GET_ITEM(form, 1));
          if (!c || !s) return 0;
          out = Packed{*c, *s};
          return 1;
        }
      }
      if (PyErr_Occurred()) PyErr_Clear();
    }
  }
  return 2;
}

// Steals `key`.  1: done, 0: not the plain path, -1: Python error
int quantize(QuantPlan::Body& q, PyObject* src, const at::Tensor& x, PyObject* h, int64_t m, int64_t k, bool quest,
             const Call& call, Packed& out, PyObject* key) {
  if (!plain_entry(E_fpq_quantize_nv_packed_padded) || !plain_entry(E_fpq_quantize_mx_packed_padded) || (quest && q.nvfp4)) {
    Py_XDECREF(key);
    return 0;
  }
  out = packed_buffers(m, k, q.nvfp4, call.dev);
  const at::Tensor gs = q.gs, rotation = *tensor_of(h);
  const int kind = q.kind, g = q.g;
  const float norm = q.norm;
  const bool nv = q.nvfp4;
  const void* const xd = x.const_data_ptr();
  int st;
  {
    NoGil nogil;
    void *pc = out.codes.mutable_data_ptr(), *ps = out.scales.mutable_data_ptr();
    st = nv ? FPQ_CALL(fpq_quantize_nv_packed_padded)(xd, m, k, kind, g, norm, (const float*)gs.const_data_ptr(), pc, ps,
                                                      g_policy, call.stream)
            : FPQ_CALL(fpq_quantize_mx_packed_padded)(xd, m, k, quest ? 1 : 0, kind, g, norm, pc, ps, g_policy, call.stream);
  }
  if (st == FPQ_E_UNSUPPORTED) {   // a rotation the packed quantizers do not take: row-major codes, re-tiled
    const int64_t groups = k / (nv ? 16 : 32);
    const c10::Device d(c10::kCUDA, call.dev);
    const at::Tensor codes = empty({m * (k / 2)}, at::kByte, d), scales = empty({m * groups}, at::kByte, d);
    NoGil nogil;
    void *c = codes.mutable_data_ptr(), *s = scales.mutable_data_ptr();
    const void* const hd = rotation.const_data_ptr();
    st = nv ? FPQ_CALL(fpq_quantize_nv)(xd, m, k, kind, g, norm, hd, (const float*)gs.const_data_ptr(), c, s, m, groups,
                                        g_policy, call.stream)
         : quest ? FPQ_CALL(fpq_quantize_mx_quest)(xd, m, k, kind, g, norm, hd, c, s, m, groups, nullptr, g_policy, call.stream)
                 : FPQ_CALL(fpq_quantize_mx)(xd, m, k, kind, g, norm, hd, c, s, m, groups, g_policy, call.stream);
    if (st == FPQ_OK)
      st = FPQ_CALL(fpq_pack_padded)(nv, c, s, groups, m, k, out.codes.mutable_data_ptr(), out.scales.mutable_data_ptr(),
                                     call.stream);
  }
  if (st != FPQ_OK) { Py_XDECREF(key); return 0; }
  if (key && !publish(src, x, key, h, out, m, k, nv, call)) return -1;
  return 1;
}

int activations(QuantPlan::Body& q, PyObject* src, const at::Tensor& x, PyObject* h, int64_t m, int64_t k, bool quest,
                const Call& call, Packed& out) {
  PyObject* key;
  const int rc = shared_activations(q, src, x, m, k, quest, call, out, key);
  return rc == 2 ? quantize(q, src, x, h, m, k, quest, call, out, key) : rc;
}

bool packed_weights_enabled() {
  const char* v = getenv("FPQ_PACKED_WEIGHTS");
  return !v || strcmp(v, "0") != 0;
}

// Whether operands with this K have a packed form (hip_ops.packable_k).
bool packable_k(int64_t k) {
  if (k < 256 || k % 32 != 0) return false;
  const char* v = k % 256 != 0 ? getenv("FPQ_SINGLE_WEIGHT_COPY") : nullptr;
  return !v || strcmp(v, "1") != 0;
}

bool is_alpha(PyObject* wgs, PyObject* alpha_obj) {   // what eager.linear_alpha holds for this layer is still that tensor
  PyObject* c = attribute(wgs, s_alpha);
  return c && PyTuple_Check(c) && PyTuple_GET_SIZE(c) == 2 && PyTuple_GET_ITEM(c, 1) == alpha_obj;
}

struct LayerTensors {
  PyObject *qweight, *scales, *wgs, *ags, *h, *bias;
};
bool layer_tensors(PyObject* params, PyObject* buffers, LayerTensors& t) {
  if (!PyDict_Check(params) || !PyDict_Check(buffers)) return false;
  t.qweight = member(params, buffers, s_qweight);
  t.scales = member(params, buffers, s_scales);
  t.wgs = member(params, buffers, s_wgs);
  t.ags = member(params, buffers, s_ags);
  t.h = member(params, buffers, s_h);
  t.bias = member(params, buffers, s_bias);
  return t.qweight && t.scales && t.wgs && t.ags && t.h && t.qweight != Py_None && t.scales != Py_None;
}

// The parameter and buffer dictionaries of a module (borrowed: the module holds them).
bool module_dicts(PyObject* module, PyObject** params, PyObject** buffers) {
  PyObject** d = _PyObject_GetDictPtr(module);
  *params = d && *d ? PyDict_GetItem(*d, s_parameters) : nullptr;
  *buffers = d && *d ? PyDict_GetItem(*d, s_buffers) : nullptr;
  return *params && *buffers && PyDict_Check(*params) && PyDict_Check(*buffers);
}
bool module_tensors(PyObject* module, LayerTensors& t) {
  PyObject *params, *buffers;
  return module_dicts(module, &params, &buffers) && layer_tensors(params, buffers, t);
}

// What to answer for want of a plan: False (one may be made), or None where a tensor cannot be in one -- an inference
// tensor has no modification counter, a subclass may be more than its data.
bool may_be_planned(PyObject* o) {
  const at::Tensor* t = tensor_of(o);
  return t && plain_cuda(*t) && !t->is_inference();
}
PyObject* no_plan(const LayerTensors& t) {
  for (PyObject* o : {t.qweight, t.scales, t.wgs, t.ags, t.h})
    if (!may_be_planned(o)) Py_RETURN_NONE;
  if (t.bias && t.bias != Py_None && !may_be_planned(t.bias)) Py_RETURN_NONE;
  Py_RETURN_FALSE;
}
PyObject* no_quant_plan(PyObject* h, PyObject* ags) {
  return Py_NewRef(may_be_planned(h) && may_be_planned(ags) ? Py_False : Py_None);
}

// Whether a layer without a plan would run on packed weights, as every plan has it.
bool may_pack(const LayerTensors& t, bool nvfp4, int64_t m) {
  const at::Tensor* q = tensor_of(t.qweight);
  if (q && q->dim() == 2 && !packable_k(q->size(1) * 2)) return false;
  return packed_weights_enabled() && (nvfp4 || m >= g_linear_rows_mx || (q && q->dim() == 1));
}

LinearPlan::Body* linear_plan(const LayerTensors& t) {   // whatever is current, usable or not
  PyObject* p = attribute(t.qweight, s_plan);
  if (!p || Py_TYPE(p) != &LinearPlanType) return nullptr;
  auto* b = ((LinearPlan*)p)->b;
  if (!b->qweight.is(t.qweight) || !b->scales.is(t.scales) || !b->wgs.is(t.wgs) || !b->ags.is(t.ags) || !b->bias.is(t.bias))
    return nullptr;
  if (b->usable) {
    if (!is_alpha(t.wgs, b->alpha_obj)) return nullptr;
    if (!b->packed_only && attribute(t.qweight, s_packed) != b->packed) return nullptr;
  }
  return b;
}

bool serves(const LinearPlan::Body* p, bool nvfp4, int64_t m, int64_t k) {
  return p && p->usable && p->nvfp4 == nvfp4 && p->k == k && (p->packed_only || (m >= p->min_rows && packed_weights_enabled()));
}

// The residual as the GEMMs take it: None (null pointer), or bf16 [m, n], contiguous.  False: not the plain path.
bool residual_of(PyObject* o, int64_t m, int64_t n, const Call& call, const at::Tensor** out) {
  *out = nullptr;
  if (o == Py_None) return true;
  const at::Tensor* t = tensor_of(o);
  if (!t || !plain_cuda(*t) || t->scalar_type() != at::kBFloat16 || !t->is_contiguous() || t->numel() != m * n ||
      t->device().index() != call.dev || t->requires_grad())
    return false;
  *out = t;
  return true;
}

// The split-K workspace of a call, left undefined where none is used: the stream's own, which the Python path makes on
// the stream's first call that needs it, or, in a capture, the layer's.  False: not there.
bool splitk_workspace(const LinearPlan::Body& p, PyObject* qweight, int64_t m, const Call& call, at::Tensor& workspace) {
  if (p.need == 0 || m > p.split_rows) return true;
  const at::Tensor* w = nullptr;
  if (call.capture) {
    w = tensor_of(attribute(qweight, s_splitk));
  } else {
    PyObject* dev = PyLong_FromLong(call.dev);
    PyObject* stream = PyLong_FromUnsignedLongLong((unsigned long long)(uintptr_t)call.stream);
    PyObject* per = dev ? PyDict_GetItem(g_workspaces, dev) : nullptr;
    w = per && stream && PyDict_Check(per) ? tensor_of(PyDict_GetItem(per, stream)) : nullptr;
    Py_XDECREF(dev);
    Py_XDECREF(stream);
  }
  if (!w || !w->is_cuda() || w->device().index() != call.dev || w->numel() < p.need) return false;
  workspace = *w;
  return true;
}

// A few rows in one launch, quantization included (fpq_linear_rows); `out`, if its tensors are there, receives the
// quantized rows.  1: launched, 0: the kernel does not take them
int linear_rows(const LinearPlan::Body& p, const QuantPlan::Body& q, const LayerTensors& t, const at::Tensor& x,
                const at::Tensor* up, const at::Tensor* residual, const Packed& out, at::Tensor& y, int64_t m,
                const Call& call) {
  if (m > 16 || q.kind > 1 || !plain_entry(E_fpq_linear_rows)) return 0;
  for (int e : {E_fpq_gemm_mxf4_packed, E_fpq_gemm_nvf4_packed, E_fpq_gemm_mxf4_packed_splitk, E_fpq_gemm_nvf4_packed_splitk,
                E_fpq_gemm_mxf4_packed_residual, E_fpq_gemm_nvf4_packed_residual})
    if (!plain_entry(e)) return 0;   // (whoever instruments the GEMMs sees every one of them)
  at::Tensor workspace;
  if (!splitk_workspace(p, t.qweight, m, call, workspace)) return 0;
  const at::Tensor wp = p.packed_only ? *tensor_of(t.qweight) : p.wp, wsp = p.packed_only ? *tensor_of(t.scales) : p.wsp;
  const at::Tensor alpha = p.alpha, bias = p.bias.held, gs = q.gs;
  const int64_t n = p.n, k = p.k;
  const int kind = q.kind, g = q.g;
  const float norm = q.norm;
  const bool nv = p.nvfp4;
  NoGil nogil;
  auto data = [](const at::Tensor& v) -> void* { return v.defined() ? v.data_ptr() : nullptr; };
  return FPQ_CALL(fpq_linear_rows)(nv, x.const_data_ptr(), up ? up->const_data_ptr() : nullptr, m, k, kind, g, norm,
                                   (const float*)data(gs), wp.const_data_ptr(), wsp.const_data_ptr(),
                                   (const float*)alpha.const_data_ptr(), data(bias),
                                   residual ? residual->const_data_ptr() : nullptr, y.mutable_data_ptr(), n, data(out.codes),
                                   data(out.scales), data(workspace), workspace.defined() ? workspace.numel() : 0, g_policy,
                                   call.stream) == FPQ_OK;
}

// 1: launched, 0: not the plain path
int gemm(const LinearPlan::Body& p, const LayerTensors& t, const Packed& x, const at::Tensor* residual, at::Tensor& y,
         int64_t m, const Call& call) {
  at::Tensor workspace;
  if (!splitk_workspace(p, t.qweight, m, call, workspace)) return 0;
  const bool nv = p.nvfp4, split = workspace.defined();
  const int entry = split ? (nv ? E_fpq_gemm_nvf4_packed_splitk : E_fpq_gemm_mxf4_packed_splitk)
                    : residual ? (nv ? E_fpq_gemm_nvf4_packed_residual : E_fpq_gemm_mxf4_packed_residual)
                               : (nv ? E_fpq_gemm_nvf4_packed : E_fpq_gemm_mxf4_packed);
  if (!plain_entry(entry)) return 0;
  // (held while the interpreter lock is released)
  const at::Tensor wp = p.packed_only ? *tensor_of(t.qweight) : p.wp, wsp = p.packed_only ? *tensor_of(t.scales) : p.wsp;
  const at::Tensor alpha = p.alpha, bias = p.bias.held, res = residual ? *residual : at::Tensor();
  const int64_t n = p.n, kp = p.kp;
  const void* const b = bias.defined() ? bias.const_data_ptr() : nullptr;
  const float* const a = (const float*)alpha.const_data_ptr();
  int st;
  {
    NoGil nogil;
    const void *xq = x.codes.const_data_ptr(), *xs = x.scales.const_data_ptr(), *wq = wp.const_data_ptr(),
               *ws = wsp.const_data_ptr(), *r = res.defined() ? res.const_data_ptr() : nullptr;
    void* out = y.mutable_data_ptr();
    if (split)
      st = nv ? FPQ_CALL(fpq_gemm_nvf4_packed_splitk)(xq, xs, wq, ws, a, b, r, out, m, n, kp, workspace.mutable_data_ptr(),
                                                      workspace.numel(), call.stream)
              : FPQ_CALL(fpq_gemm_mxf4_packed_splitk)(xq, xs, wq, ws, a, b, r, out, m, n, kp, workspace.mutable_data_ptr(),
                                                      workspace.numel(), call.stream);
    else if (r)
      st = nv ? FPQ_CALL(fpq_gemm_nvf4_packed_residual)(xq, xs, wq, ws, a, b, r, out, m, n, kp, call.stream)
              : FPQ_CALL(fpq_gemm_mxf4_packed_residual)(xq, xs, wq, ws, a, b, r, out, m, n, kp, call.stream);
    else
      st = nv ? FPQ_CALL(fpq_gemm_nvf4_packed)(xq, xs, wq, ws, a, b, out, m, n, kp, call.stream)
              : FPQ_CALL(fpq_gemm_mxf4_packed)(xq, xs, wq, ws, a, b, out, m, n, kp, call.stream);
  }
  return st == FPQ_OK;
}

at::Tensor output_like(const at::Tensor& x, int64_t n, const Call& call) {   // bf16 [*x.shape[:-1], n]
  c10::SmallVector<int64_t, 6> sizes(x.sizes().begin(), x.sizes().end());
  sizes.back() = n;
  return empty(sizes, at::kBFloat16, c10::Device(c10::kCUDA, call.dev));
}

// linear(layer, x, residual, nvfp4, method): FPQuantLinear.forward
PyObject* host_linear(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 5) Py_RETURN_NONE;
  LayerTensors t;
  const at::Tensor* xp = tensor_of(args[1]);
  Call call;
  if (!xp || !module_tensors(args[0], t) || !plain_call(*xp, call)) Py_RETURN_NONE;
  const bool nvfp4 = args[3] == Py_True;
  if (!PyUnicode_Check(args[4])) Py_RETURN_NONE;
  const bool quest = !nvfp4 && PyUnicode_CompareWithASCIIString(args[4], "quest") == 0;
  if (!quest && PyUnicode_CompareWithASCIIString(args[4], "abs_max") != 0) Py_RETURN_NONE;
  const at::Tensor x = *xp;
  const int64_t k = x.size(-1), m = x.numel() / k;
  LinearPlan::Body* p = linear_plan(t);
  QuantPlan::Body* q = quant_plan(t.h, t.ags, nvfp4);
  const at::Tensor* residual;
  if (!p && !may_pack(t, nvfp4, m)) Py_RETURN_NONE;
  if (!p || !q) return no_plan(t);
  if (x.dim() < 2 || !serves(p, nvfp4, m, k) || !q->usable || tensor_of(t.qweight)->device().index() != call.dev ||
      !residual_of(args[2], m, p->n, call, &residual))
    Py_RETURN_NONE;
  // (the plans stay while the interpreter lock is given up around a launch)
  const THPObjectPtr hold_p(Py_NewRef(attribute(t.qweight, s_plan))), hold_q(Py_NewRef(attribute(t.h, s_qplan)));
  const THPObjectPtr hold_w(Py_NewRef(t.qweight)), hold_s(Py_NewRef(t.scales)), hold_h(Py_NewRef(t.h));
  Packed packed;
  PyObject* key;
  int rc = shared_activations(*q, args[1], x, m, k, quest, call, packed, key);
  if (rc < 0) return nullptr;
  if (rc == 0) Py_RETURN_NONE;
  at::Tensor y = output_like(x, p->n, call);
  if (rc == 2) {
    if (!quest && m <= 16 && q->kind <= 1) {
      if (key) packed = packed_buffers(m, k, nvfp4, call.dev);
      if (linear_rows(*p, *q, t, x, nullptr, residual, packed, y, m, call)) {
        if (key && !publish(args[1], x, key, t.h, packed, m, k, nvfp4, call)) return nullptr;
        return THPVariable_Wrap(std::move(y));
      }
    }
    rc = quantize(*q, args[1], x, t.h, m, k, quest, call, packed, key);
    if (rc < 0) return nullptr;
    if (rc == 0) Py_RETURN_NONE;
  }
  if (!gemm(*p, t, packed, residual, y, m, call)) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// The weight and epsilon of an RMSNorm module over `cols` columns, if the fused kernels take them.
bool norm_of(PyObject* norm, int64_t cols, const Call& call, at::Tensor& weight, float& eps) {
  PyObject *params, *buffers;
  if (!module_dicts(norm, &params, &buffers)) return false;
  PyObject* eps_obj = PyDict_GetItem(*_PyObject_GetDictPtr(norm), s_eps);
  const at::Tensor* w = tensor_of(member(params, buffers, s_weight));
  if (!eps_obj || !PyFloat_Check(eps_obj) || !w || !plain_cuda(*w) || w->scalar_type() != at::kBFloat16 ||
      !w->is_contiguous() || w->numel() != cols || w->device().index() != call.dev || cols > 16384 || !packable_k(cols) ||
      !packed_weights_enabled())
    return false;
  weight = *w;
  eps = (float)PyFloat_AS_DOUBLE(eps_obj);
  return true;
}
// (fused producers take Hadamard (0) and identity (1) rotations)
bool norm_rotation(const QuantPlan::Body& q, int64_t cols) {
  return q.usable && q.kind <= 1 && cols % (q.g > 32 ? q.g : 32) == 0;
}
bool norm_few(int64_t rows, int64_t cols) { return rows <= 64 && cols % 256 == 0; }
bool norm_in_two_launches(int64_t rows, int64_t cols) {   // (eager._norm_in_two_launches)
  return !norm_few(rows, cols) && rows <= 640 && cols > 8192 && cols % 256 == 0 && rows * cols <= (1 << 23);
}
int norm_entry(int64_t rows, int64_t cols, bool nvfp4) {
  return norm_few(rows, cols) ? (nvfp4 ? E_fpq_rmsnorm_rows_quantize_nv_packed : E_fpq_rmsnorm_rows_quantize_mx_packed)
                              : (nvfp4 ? E_fpq_rmsnorm_tile_quantize_nv_packed : E_fpq_rmsnorm_tile_quantize_mx_packed);
}
// `y`: receives the norm's bf16 result, if it is wanted.  The status of the launch.
int norm_quantize(const QuantPlan::Body& q, const at::Tensor& x, const at::Tensor& w, float eps, at::Tensor* y, Packed& out,
                  int64_t rows, int64_t cols, bool nvfp4, const Call& call) {
  const bool few = norm_few(rows, cols);
  const at::Tensor gs = q.gs;
  const int kind = q.kind, g = q.g;
  const float norm = q.norm;
  NoGil nogil;
  const void *xd = x.const_data_ptr(), *wd = w.const_data_ptr();
  void *yd = y ? y->mutable_data_ptr() : nullptr, *pc = out.codes.mutable_data_ptr(), *ps = out.scales.mutable_data_ptr();
  if (nvfp4) {
    const float* g_s = (const float*)gs.const_data_ptr();
    return few ? FPQ_CALL(fpq_rmsnorm_rows_quantize_nv_packed)(xd, cols, wd, rows, cols, eps, kind, g, norm, g_s, nullptr, yd,
                                                               pc, ps, g_policy, call.stream)
               : FPQ_CALL(fpq_rmsnorm_tile_quantize_nv_packed)(xd, cols, wd, rows, cols, eps, kind, g, norm, g_s, nullptr, yd,
                                                               pc, ps, g_policy, call.stream);
  }
  return few ? FPQ_CALL(fpq_rmsnorm_rows_quantize_mx_packed)(xd, cols, wd, rows, cols, eps, kind, g, norm, nullptr, yd, pc, ps,
                                                             g_policy, call.stream)
             : FPQ_CALL(fpq_rmsnorm_tile_quantize_mx_packed)(xd, cols, wd, rows, cols, eps, kind, g, norm, nullptr, yd, pc, ps,
                                                             g_policy, call.stream);
}

// rmsnorm(norm, layer, x, nvfp4): eager.rmsnorm_quantize with the rotation and activation scale of `layer`
PyObject* host_rmsnorm(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  LayerTensors t;
  if (n_args != 4 || !module_tensors(args[1], t)) Py_RETURN_NONE;
  const at::Tensor* xp = tensor_of(args[2]);
  Call call;
  if (!xp || !plain_call(*xp, call)) Py_RETURN_NONE;
  const bool nvfp4 = args[3] == Py_True;
  const at::Tensor x = *xp;
  at::Tensor w;
  float eps;
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  if (!norm_of(args[0], cols, call, w, eps)) Py_RETURN_NONE;
  QuantPlan::Body* q = quant_plan(t.h, t.ags, nvfp4);
  if (!q) return no_quant_plan(t.h, t.ags);
  if (!norm_rotation(*q, cols) || norm_in_two_launches(rows, cols)) Py_RETURN_NONE;
  bool declined = false;
  const bool share = sharing_enabled(*q, declined);
  if (!plain_entry(norm_entry(rows, cols, nvfp4)) || declined) Py_RETURN_NONE;
  THPObjectPtr hold_h(Py_NewRef(t.h));
  const THPObjectPtr hold_q(Py_NewRef(attribute(t.h, s_qplan)));
  THPObjectPtr key(share ? sharing_key(*q, rows, cols, call, false) : nullptr);
  if (share && !key) return nullptr;
  at::Tensor y = output_like(x, cols, call);
  Packed out = packed_buffers(rows, cols, nvfp4, call.dev);
  if (norm_quantize(*q, x, w, eps, &y, out, rows, cols, nvfp4, call) != FPQ_OK) Py_RETURN_NONE;
  THPObjectPtr result(THPVariable_Wrap(y));
  if (!result) return nullptr;
  if (share && !publish(result.get(), y, key.release(), hold_h.get(), out, rows, cols, nvfp4, call)) return nullptr;
  return result.release();
  END_HANDLE_TH_ERRORS
}

// Whether the layers' tensors are those of a group's plan: null, with the first layer's rotation and activation scale, or
// what to answer (None, False).
PyObject* group_members(const GroupPlan::Body& p, PyObject* layers, THPObjectPtr& h, PyObject*& first_ags) {
  const size_t count = PyTuple_GET_SIZE(layers);
  if (count * 3 != p.members.size() || count > 4) Py_RETURN_NONE;
  for (size_t i = 0; i < count; ++i) {
    LayerTensors t;
    if (!module_tensors(PyTuple_GET_ITEM(layers, i), t)) Py_RETURN_NONE;
    if (!p.members[3 * i].is(t.qweight) || !p.members[3 * i + 1].is(t.scales) || !p.members[3 * i + 2].is(t.bias))
      return no_plan(t);
    if (i == 0 && p.usable) {
      if (!p.wgs.is(t.wgs) || !p.ags.is(t.ags) || !is_alpha(t.wgs, p.alpha_obj)) return no_plan(t);
      h = THPObjectPtr(Py_NewRef(t.h));
      first_ags = t.ags;
    }
  }
  return nullptr;
}

// What a norm in front of a group does to the group's call: rows that one launch takes together with the GEMM, rows whose
// norm is a launch of its own but need not leave its bf16 result, or neither (the caller runs the norm module first; it asks
// for these two only, fuse._norm_bounds).  Without the bf16 result the kernel of 8192 x 4096 takes 23.9 us instead of 30.2, a
// decoder block of 8192 / 4096 tokens 956.7 / 471.8 instead of 967.2 / 477.2; from 65 to 2048 rows the GPU's time is the
// same within 0.3 %, and the host has one call and two allocations less (128 rows of 2048 features: 53.4 -> 48.5).
constexpr int64_t kNormInGemmRows = 4, kNormAloneRows = 64;

// The quantized output of `norm` on x where that is a launch of its own.  1: done, 0: not the plain path
int norm_activations(const QuantPlan::Body& q, PyObject* norm, const at::Tensor& x, int64_t m, int64_t k, bool nvfp4,
                     const Call& call, Packed& out) {
  at::Tensor w;
  float eps;
  if (m <= kNormAloneRows || !norm_of(norm, k, call, w, eps) || !norm_rotation(q, k) || norm_in_two_launches(m, k) ||
      !plain_entry(norm_entry(m, k, nvfp4)))
    return 0;
  out = packed_buffers(m, k, nvfp4, call.dev);
  return norm_quantize(q, x, w, eps, nullptr, out, m, k, nvfp4, call) == FPQ_OK;
}

// group(plan, layers, x): the outputs of layers whose packed weights lie end to end (eager.linear_cat)
// norm_group(plan, layers, x, norm): ... on norm(x)
PyObject* host_group(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if ((n_args != 3 && n_args != 4) || !PyTuple_Check(args[1])) Py_RETURN_NONE;
  PyObject* const norm = n_args == 4 ? args[3] : nullptr;
  if (Py_TYPE(args[0]) != &GroupPlanType) {   // no plan yet, if the call is a plain one
    const at::Tensor* t = tensor_of(args[2]);
    Call c;
    if (!t || !plain_call(*t, c)) Py_RETURN_NONE;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(args[1]); ++i) {
      LayerTensors l;
      if (!module_tensors(PyTuple_GET_ITEM(args[1], i), l)) Py_RETURN_NONE;
      PyObject* answer = no_plan(l);
      if (answer == Py_None) return answer;
      Py_DECREF(answer);
    }
    Py_RETURN_FALSE;
  }
  const THPObjectPtr hold(Py_NewRef(args[0]));
  auto* p = ((GroupPlan*)args[0])->b;
  const at::Tensor* xp = tensor_of(args[2]);
  Call call;
  if (!xp || !plain_call(*xp, call)) Py_RETURN_NONE;
  const size_t count = PyTuple_GET_SIZE(args[1]);
  THPObjectPtr h;
  PyObject* first_ags = nullptr;
  if (PyObject* answer = group_members(*p, args[1], h, first_ags)) return answer;
  if (!p->usable) Py_RETURN_NONE;
  const at::Tensor x = *xp;
  const int64_t k = x.size(-1), m = x.numel() / k;
  QuantPlan::Body* q = quant_plan(h.get(), first_ags, p->nvfp4);
  const int entry = p->nvfp4 ? E_fpq_gemm_nvf4_packed_multi : E_fpq_gemm_mxf4_packed_multi;
  if (!q) return no_quant_plan(h.get(), first_ags);
  if (!q->usable || k != p->k || x.dim() < 2 || p->wp.device().index() != call.dev || !plain_entry(entry)) Py_RETURN_NONE;
  const THPObjectPtr hold_q(Py_NewRef(attribute(h.get(), s_qplan)));
  const bool one_launch = norm && m <= kNormInGemmRows;
  Packed packed;
  at::Tensor w;
  float eps = 0.0f;
  if (one_launch) {
    if (!norm_of(norm, k, call, w, eps) || !norm_rotation(*q, k) || !plain_entry(norm_entry(m, k, p->nvfp4)) ||
        !plain_entry(E_fpq_norm_rows_multi))
      Py_RETURN_NONE;
  } else {
    const int rc = norm ? norm_activations(*q, norm, x, m, k, p->nvfp4, call, packed)
                        : activations(*q, args[2], x, h.get(), m, k, false, call, packed);
    if (rc < 0) return nullptr;
    if (rc == 0) Py_RETURN_NONE;
  }
  at::Tensor ys[4];
  void* y_ptr[4];
  for (size_t i = 0; i < count; ++i) {
    ys[i] = output_like(x, p->splits[i], call);
    y_ptr[i] = ys[i].mutable_data_ptr();
  }
  int st;
  if (one_launch) {
    const at::Tensor gs = q->gs;
    const int kind = q->kind, g = q->g;
    const float h_norm = q->norm;
    NoGil nogil;
    st = FPQ_CALL(fpq_norm_rows_multi)(p->nvfp4, x.const_data_ptr(), w.const_data_ptr(), eps, m, k, kind, g, h_norm,
                                       gs.defined() ? (const float*)gs.const_data_ptr() : nullptr, p->wp.const_data_ptr(),
                                       p->wsp.const_data_ptr(), (const float*)p->alpha.const_data_ptr(),
                                       p->bias.defined() ? p->bias.const_data_ptr() : nullptr, y_ptr, p->splits.data(),
                                       (int64_t)count, g_policy, call.stream);
  } else {
    NoGil nogil;   // (the plan, and with it every operand, is held)
    auto fn = p->nvfp4 ? FPQ_CALL(fpq_gemm_nvf4_packed_multi) : FPQ_CALL(fpq_gemm_mxf4_packed_multi);
    st = fn(packed.codes.const_data_ptr(), packed.scales.const_data_ptr(), p->wp.const_data_ptr(), p->wsp.const_data_ptr(),
            (const float*)p->alpha.const_data_ptr(), p->bias.defined() ? p->bias.const_data_ptr() : nullptr, y_ptr,
            p->splits.data(), (int64_t)count, m, p->kp, call.stream);
  }
  if (st != FPQ_OK) Py_RETURN_NONE;
  THPObjectPtr out(PyList_New((Py_ssize_t)count));
  if (!out) return nullptr;
  for (size_t i = 0; i < count; ++i) PyList_SET_ITEM(out.get(), i, THPVariable_Wrap(std::move(ys[i])));
  return out.release();
  END_HANDLE_TH_ERRORS
}

// gated_down(layer, gate, up, residual, nvfp4): down(bf16(silu(gate)) * up) + residual, the product
// quantized as it is formed (eager.silu_mul_quantize, FPQuantLinear.forward_quantized)
PyObject* host_gated_down(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if (n_args != 5) Py_RETURN_NONE;
  LayerTensors t;
  const at::Tensor *gp = tensor_of(args[1]), *up = tensor_of(args[2]);
  Call call;
  if (!gp || !up || !module_tensors(args[0], t) || !plain_call(*gp, call)) Py_RETURN_NONE;
  const at::Tensor gate = *gp, u = *up;
  const bool nvfp4 = args[4] == Py_True;
  if (!plain_cuda(u) || u.scalar_type() != at::kBFloat16 || !u.is_contiguous() || u.sizes() != gate.sizes() ||
      u.device() != gate.device() || u.requires_grad() || gate.dim() < 2)
    Py_RETURN_NONE;
  const int64_t k = gate.size(-1), m = gate.numel() / k;
  LinearPlan::Body* p = linear_plan(t);
  QuantPlan::Body* q = quant_plan(t.h, t.ags, nvfp4);
  const at::Tensor* residual;
  if (!p && !may_pack(t, nvfp4, m)) Py_RETURN_NONE;
  if (!p || !q) return no_plan(t);
  if (!serves(p, nvfp4, m, k) || !q->usable || q->kind > 1 || k % (q->g > 32 ? q->g : 32) != 0 || !packed_weights_enabled() ||
      ((uintptr_t)gate.const_data_ptr() & 15) || ((uintptr_t)u.const_data_ptr() & 15) ||
      tensor_of(t.qweight)->device().index() != call.dev || !residual_of(args[3], m, p->n, call, &residual))
    Py_RETURN_NONE;
  const int entry = nvfp4 ? E_fpq_silu_mul_quantize_nv_packed : E_fpq_silu_mul_quantize_mx_packed;
  if (!plain_entry(entry)) Py_RETURN_NONE;
  const THPObjectPtr hold_p(Py_NewRef(attribute(t.qweight, s_plan))), hold_q(Py_NewRef(attribute(t.h, s_qplan)));
  const THPObjectPtr hold_w(Py_NewRef(t.qweight)), hold_s(Py_NewRef(t.scales));
  at::Tensor y = output_like(gate, p->n, call);
  if (linear_rows(*p, *q, t, gate, &u, residual, Packed{}, y, m, call)) return THPVariable_Wrap(std::move(y));
  Packed out = packed_buffers(m, k, nvfp4, call.dev);
  int st;
  {
    const at::Tensor gs = q->gs;
    const int kind = q->kind, g = q->g;
    const float norm = q->norm;
    NoGil nogil;
    void *pc = out.codes.mutable_data_ptr(), *ps = out.scales.mutable_data_ptr();
    st = nvfp4 ? FPQ_CALL(fpq_silu_mul_quantize_nv_packed)(gate.const_data_ptr(), k, u.const_data_ptr(), k, m, k, kind, g, norm,
                                                           (const float*)gs.const_data_ptr(), nullptr, pc, ps, g_policy,
                                                           call.stream)
               : FPQ_CALL(fpq_silu_mul_quantize_mx_packed)(gate.const_data_ptr(), k, u.const_data_ptr(), k, m, k, kind, g, norm,
                                                           nullptr, pc, ps, g_policy, call.stream);
  }
  if (st != FPQ_OK) Py_RETURN_NONE;
  if (!gemm(*p, t, out, residual, y, m, call)) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// gated_mlp(plan, (gate, up), down, x, residual, norm): norm (unless it is None), group() and gated_down() of its outputs where
// one GEMM forms and quantizes the product in its epilogue (fpq_gemm_packed_gated: many rows); None for any other call.
PyObject* host_gated_mlp(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  if ((n_args != 5 && n_args != 6) || Py_TYPE(args[0]) != &GroupPlanType || !PyTuple_Check(args[1])) Py_RETURN_NONE;
  PyObject* const norm = n_args == 6 && args[5] != Py_None ? args[5] : nullptr;
  const THPObjectPtr hold(Py_NewRef(args[0]));
  auto* p = ((GroupPlan*)args[0])->b;
  const at::Tensor* xp = tensor_of(args[3]);
  Call call;
  LayerTensors t;
  if (!xp || !plain_call(*xp, call) || xp->dim() < 2 || !p->usable || p->splits.size() != 2 || p->splits[0] != p->splits[1] ||
      p->bias.defined() || !module_tensors(args[2], t))
    Py_RETURN_NONE;
  const at::Tensor x = *xp;
  const int64_t k = x.size(-1), m = x.numel() / k, inner = p->splits[0];
  const bool nvfp4 = p->nvfp4;
  if (k != p->k || p->wp.device().index() != call.dev ||
      !FPQ_CALL(fpq_gemm_packed_gated_takes)(nvfp4, m, inner, p->kp))
    Py_RETURN_NONE;
  THPObjectPtr h;
  PyObject* first_ags = nullptr;
  if (PyObject* answer = group_members(*p, args[1], h, first_ags)) {
    Py_DECREF(answer);
    Py_RETURN_NONE;
  }
  QuantPlan::Body* q = quant_plan(h.get(), first_ags, nvfp4);
  LinearPlan::Body* d = linear_plan(t);
  QuantPlan::Body* dq = quant_plan(t.h, t.ags, nvfp4);
  const at::Tensor* residual;
  if (!q || !q->usable || !serves(d, nvfp4, m, inner) || !dq || !dq->usable || dq->kind > 1 || !packed_weights_enabled() ||
      inner % (dq->g > 32 ? dq->g : 32) != 0 || tensor_of(t.qweight)->device().index() != call.dev ||
      !residual_of(args[4], m, d->n, call, &residual))
    Py_RETURN_NONE;
  for (int e : {E_fpq_gemm_nvf4_packed_multi, E_fpq_gemm_mxf4_packed_multi, E_fpq_silu_mul_quantize_nv_packed,
                E_fpq_silu_mul_quantize_mx_packed, E_fpq_gemm_packed_gated})
    if (!plain_entry(e)) Py_RETURN_NONE;   // (whoever instruments either kernel sees both)
  const THPObjectPtr hold_q(Py_NewRef(attribute(h.get(), s_qplan)));
  const THPObjectPtr hold_d(Py_NewRef(attribute(t.qweight, s_plan))), hold_dq(Py_NewRef(attribute(t.h, s_qplan)));
  const THPObjectPtr hold_w(Py_NewRef(t.qweight)), hold_s(Py_NewRef(t.scales));
  Packed in;
  const int rc = norm ? norm_activations(*q, norm, x, m, k, nvfp4, call, in)
                      : activations(*q, args[3], x, h.get(), m, k, false, call, in);
  if (rc < 0) return nullptr;
  if (rc == 0) Py_RETURN_NONE;
  const Packed product = packed_buffers(m, inner, nvfp4, call.dev);
  at::Tensor y = output_like(x, d->n, call);
  int st;
  {
    const at::Tensor gs = dq->gs;
    const int kind = dq->kind, g = dq->g;
    const float norm = dq->norm;
    NoGil nogil;   // (the plans, and with them every operand, are held)
    st = FPQ_CALL(fpq_gemm_packed_gated)(nvfp4, in.codes.const_data_ptr(), in.scales.const_data_ptr(), p->wp.const_data_ptr(),
                                         p->wsp.const_data_ptr(), (const float*)p->alpha.const_data_ptr(), m, inner, p->kp,
                                         kind, g, norm, gs.defined() ? (const float*)gs.const_data_ptr() : nullptr,
                                         product.codes.mutable_data_ptr(), product.scales.mutable_data_ptr(), g_policy,
                                         call.stream);
  }
  if (st != FPQ_OK || !gemm(*d, t, product, residual, y, m, call)) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// ---- the quantize and matmul operators, called outside any tracing: the bodies of hip_ops' custom operators
// without the operator dispatch (10 us of host time per call)
// (an operand of such a call)
const at::Tensor* operand(PyObject* o, const Call& call) {
  const at::Tensor* t = tensor_of(o);
  return t && plain_cuda(*t) && t->is_contiguous() && !t->requires_grad() && t->device().index() == call.dev
             ? t
             : nullptr;
}

bool is_number(PyObject* o, unsigned long long v) {
  return o && PyLong_Check(o) && PyLong_AsUnsignedLongLongMask(o) == v;
}

// Kind and norm of a bf16 rotation matrix that classify_rotation has seen in its present state.
bool rotation_of(PyObject* h, const at::Tensor& t, int& kind, float& norm) {
  if (t.scalar_type() != at::kBFloat16 || t.dim() != 2) return false;
  PyObject* c = t.is_inference() ? nullptr : attribute(h, s_rotation);
  if (!c || !PyTuple_Check(c) || PyTuple_GET_SIZE(c) != 3) return false;
  PyObject* key = PyTuple_GET_ITEM(c, 0);
  if (!PyTuple_Check(key) || PyTuple_GET_SIZE(key) != 2 ||
      !is_number(PyTuple_GET_ITEM(key, 0), (unsigned long long)(uintptr_t)t.const_data_ptr()) ||
      !is_number(PyTuple_GET_ITEM(key, 1), (unsigned long long)t._version()))
    return false;
  kind = (int)PyLong_AsLong(PyTuple_GET_ITEM(c, 1));
  norm = (float)PyFloat_AsDouble(PyTuple_GET_ITEM(c, 2));
  if (PyErr_Occurred()) { PyErr_Clear(); return false; }
  return true;
}

// quantize_mx(x, rotation, method, return_mask), quantize_nv(x, rotation, global_scale)
template <bool NV>
PyObject* host_quantize(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  const at::Tensor* xp = n_args == (NV ? 3 : 4) ? tensor_of(args[0]) : nullptr;
  Call call;
  if (!xp || !plain_call(*xp, call)) Py_RETURN_NONE;
  const at::Tensor x = *xp;
  const at::Tensor *hp = operand(args[1], call), *gsp = NV ? operand(args[2], call) : nullptr;
  int kind;
  float norm;
  if (!hp || !rotation_of(args[1], *hp, kind, norm)) Py_RETURN_NONE;
  bool quest = false;
  if (NV) {
    if (!gsp || gsp->scalar_type() != at::kFloat || gsp->numel() != 1) Py_RETURN_NONE;
  } else {
    if (x.dim() != 2 || args[3] != Py_False || !PyUnicode_Check(args[2])) Py_RETURN_NONE;
    quest = PyUnicode_CompareWithASCIIString(args[2], "quest") == 0;
    if (!quest && PyUnicode_CompareWithASCIIString(args[2], "abs_max") != 0) Py_RETURN_NONE;
  }
  const int entry = NV ? E_fpq_quantize_nv : quest ? E_fpq_quantize_mx_quest : E_fpq_quantize_mx;
  if (!plain_entry(entry)) Py_RETURN_NONE;
  const int64_t cols = x.size(-1), rows = x.numel() / cols;
  const int64_t prow = (rows + 127) / 128 * 128, pcol = (cols / (NV ? 16 : 32) + 3) / 4 * 4;
  if (pcol == 0 || cols % 2 != 0) Py_RETURN_NONE;
  const c10::Device d(c10::kCUDA, call.dev);
  c10::SmallVector<int64_t, 6> sizes(x.sizes().begin(), x.sizes().end());
  sizes.back() = cols / 2;
  at::Tensor codes = empty(sizes, at::kByte, d), scales = empty({prow, pcol}, NV ? at::kFloat8_e4m3fn : at::kFloat8_e8m0fnu, d);
  const at::Tensor h = *hp, gs = gsp ? *gsp : at::Tensor();
  const int g = (int)h.size(0);
  int st;
  {
    NoGil nogil;
    const void *xd = x.const_data_ptr(), *hd = h.const_data_ptr();
    void *c = codes.mutable_data_ptr(), *s = scales.mutable_data_ptr();
    st = NV ? FPQ_CALL(fpq_quantize_nv)(xd, rows, cols, kind, g, norm, hd, (const float*)gs.const_data_ptr(), c, s, prow, pcol,
                                        g_policy, call.stream)
         : quest ? FPQ_CALL(fpq_quantize_mx_quest)(xd, rows, cols, kind, g, norm, hd, c, s, prow, pcol, nullptr, g_policy,
                                                   call.stream)
                 : FPQ_CALL(fpq_quantize_mx)(xd, rows, cols, kind, g, norm, hd, c, s, prow, pcol, g_policy, call.stream);
  }
  if (st != FPQ_OK) Py_RETURN_NONE;
  if (NV) return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(codes)), THPVariable_Wrap(std::move(scales)));
  return Py_BuildValue("(NNO)", THPVariable_Wrap(std::move(codes)), THPVariable_Wrap(std::move(scales)), Py_None);
  END_HANDLE_TH_ERRORS
}

// The packed copy that hip_ops.packed_weight holds for a row-major weight in its present state.
bool packed_copy(PyObject* wo, const at::Tensor& w, const at::Tensor& ws, bool nvfp4, at::Tensor& wp, at::Tensor& wsp) {
  PyObject* c = w.is_inference() || ws.is_inference() ? nullptr : attribute(wo, s_packed);
  if (!c || !PyTuple_Check(c) || PyTuple_GET_SIZE(c) != 3) return false;
  PyObject* key = PyTuple_GET_ITEM(c, 0);
  if (!PyTuple_Check(key) || PyTuple_GET_SIZE(key) != 6) return false;
  PyObject* shape = PyTuple_GET_ITEM(key, 4);
  if (!is_number(PyTuple_GET_ITEM(key, 0), (unsigned long long)(uintptr_t)w.const_data_ptr()) ||
      !is_number(PyTuple_GET_ITEM(key, 1), (unsigned long long)w._version()) ||
      !is_number(PyTuple_GET_ITEM(key, 2), (unsigned long long)(uintptr_t)ws.const_data_ptr()) ||
      !is_number(PyTuple_GET_ITEM(key, 3), (unsigned long long)ws._version()) || !PyTuple_Check(shape) ||
      PyTuple_GET_SIZE(shape) != 2 || !is_number(PyTuple_GET_ITEM(shape, 0), (unsigned long long)w.size(0)) ||
      !is_number(PyTuple_GET_ITEM(shape, 1), (unsigned long long)w.size(1)) ||
      PyTuple_GET_ITEM(key, 5) != (nvfp4 ? Py_True : Py_False))
    return false;
  const at::Tensor *a = tensor_of(PyTuple_GET_ITEM(c, 1)), *b = tensor_of(PyTuple_GET_ITEM(c, 2));
  if (!a || !b) return false;
  wp = *a;
  wsp = *b;
  return true;
}

// matmul_mx / matmul_nv(x, w, x_scales, w_scales, alpha[, bias])
template <bool NV>
PyObject* host_matmul(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  const at::Tensor* xp = n_args == 5 || n_args == 6 ? tensor_of(args[0]) : nullptr;
  Call call;
  if (!xp || !plain_call(*xp, call, at::kByte)) Py_RETURN_NONE;
  const at::Tensor *wp = operand(args[1], call), *xsp = operand(args[2], call), *wsp = operand(args[3], call),
                   *ap = operand(args[4], call), *bp = n_args == 6 ? operand(args[5], call) : nullptr;
  if (!wp || !xsp || !wsp || !ap || (n_args == 6 && !bp)) Py_RETURN_NONE;
  const at::Tensor x = *xp, w = *wp, xs = *xsp, ws = *wsp, alpha = *ap, bias = bp ? *bp : at::Tensor();
  if (w.scalar_type() != at::kByte || w.dim() != 2 || x.dim() < 2 || xs.element_size() != 1 || ws.element_size() != 1 ||
      xs.dim() < 2 || ws.dim() < 2 || xs.numel() == 0 || ws.numel() == 0 || alpha.scalar_type() != at::kFloat ||
      alpha.numel() != 1)
    Py_RETURN_NONE;
  const int64_t kb = x.size(-1), m = x.numel() / kb, k = kb * 2, n = w.size(0), groups = k / (NV ? 16 : 32);
  const int64_t ldx = xs.size(-1), ldw = ws.size(-1);
  if (w.size(1) != kb || n == 0 || xs.numel() / ldx < m || ldx < groups || ws.numel() / ldw < n || ldw < groups ||
      (bias.defined() && (bias.scalar_type() != at::kBFloat16 || bias.numel() != n)))
    Py_RETURN_NONE;
  const bool packed = m >= (NV ? g_packed_rows_nv : g_packed_rows_mx) && packable_k(k) && packed_weights_enabled();
  if (!plain_entry(E_fpq_gemm_mxf4) || !plain_entry(E_fpq_gemm_nvf4) || !plain_entry(E_fpq_gemm_mxf4_packed) ||
      !plain_entry(E_fpq_gemm_nvf4_packed) || !plain_entry(E_fpq_pack_padded))
    Py_RETURN_NONE;
  at::Tensor pw, pws;
  if (packed && !packed_copy(args[1], w, ws, NV, pw, pws)) Py_RETURN_NONE;
  c10::SmallVector<int64_t, 6> sizes(x.sizes().begin(), x.sizes().end());
  sizes.back() = n;
  at::Tensor y = empty(sizes, at::kBFloat16, c10::Device(c10::kCUDA, call.dev));
  const Packed px = packed ? packed_buffers(m, k, NV, call.dev) : Packed{};
  int st;
  {
    NoGil nogil;
    const void *xd = x.const_data_ptr(), *xsd = xs.const_data_ptr(), *wd = w.const_data_ptr(), *wsd = ws.const_data_ptr(),
               *b = bias.defined() ? bias.const_data_ptr() : nullptr;
    const float* a = (const float*)alpha.const_data_ptr();
    void* out = y.mutable_data_ptr();
    if (packed) {
      void *pc = px.codes.mutable_data_ptr(), *ps = px.scales.mutable_data_ptr();
      const int64_t kp = (k + 255) / 256 * 256;
      st = FPQ_CALL(fpq_pack_padded)(NV, xd, xsd, ldx, m, k, pc, ps, call.stream);
      if (st == FPQ_OK)
        st = NV ? FPQ_CALL(fpq_gemm_nvf4_packed)(pc, ps, pw.const_data_ptr(), pws.const_data_ptr(), a, b, out, m, n, kp, call.stream)
                : FPQ_CALL(fpq_gemm_mxf4_packed)(pc, ps, pw.const_data_ptr(), pws.const_data_ptr(), a, b, out, m, n, kp, call.stream);
    } else {
      st = NV ? FPQ_CALL(fpq_gemm_nvf4)(xd, xsd, ldx, wd, wsd, ldw, a, b, out, m, n, k, call.stream)
              : FPQ_CALL(fpq_gemm_mxf4)(xd, xsd, ldx, wd, wsd, ldw, a, b, out, m, n, k, call.stream);
    }
  }
  if (st != FPQ_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// ---- making plans (module/host.py)
// linear_plan_current(layer): whether the layer's plan, usable or not, matches its tensors
PyObject* host_linear_plan_current(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject* layer;
  if (!PyArg_ParseTuple(args, "O", &layer)) return nullptr;
  LayerTensors t;
  return PyBool_FromLong(module_tensors(layer, t) && linear_plan(t) != nullptr);
  END_HANDLE_TH_ERRORS
}
// quant_plan_current(rotation, act_global_scale, nvfp4): likewise
PyObject* host_quant_plan_current(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *h, *ags;
  int nvfp4;
  if (!PyArg_ParseTuple(args, "OOp", &h, &ags, &nvfp4)) return nullptr;
  PyObject* p = attribute(h, s_qplan);
  if (!p || Py_TYPE(p) != &QuantPlanType) Py_RETURN_FALSE;
  auto* b = ((QuantPlan*)p)->b;
  return PyBool_FromLong(b->nvfp4 == (bool)nvfp4 && b->h.is(h) && (!nvfp4 || b->ags.is(ags)));
  END_HANDLE_TH_ERRORS
}
// quant_plan(rotation, act_global_scale, nvfp4, kind, norm, g, gs, rot, gs_host) -> plan or None; kind < 0: a marker that
// there is none
PyObject* host_quant_plan(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *h, *ags, *gs, *rot, *gs_host;
  int nvfp4, kind, g;
  float norm;
  if (!PyArg_ParseTuple(args, "OOpifiOOO", &h, &ags, &nvfp4, &kind, &norm, &g, &gs, &rot, &gs_host)) return nullptr;
  THPObjectPtr o(plan_new<QuantPlan>(&QuantPlanType, nullptr, nullptr));
  if (!o) return nullptr;
  auto* b = ((QuantPlan*)o.get())->b;
  b->rot = Py_NewRef(rot);
  b->gs_host = Py_NewRef(gs_host);
  b->kind = kind;
  b->norm = norm;
  b->g = g;
  b->nvfp4 = nvfp4;
  b->usable = kind >= 0;
  if (!b->h.take(h, false) || !b->ags.take(ags, true) || h == Py_None || ags == Py_None || !take_tensor(gs, b->gs)) Py_RETURN_NONE;
  if (b->usable && nvfp4 && (!b->gs.defined() || b->gs.scalar_type() != at::kFloat)) Py_RETURN_NONE;
  return o.release();
  END_HANDLE_TH_ERRORS
}
// linear_plan(qweight, scales, wgs, ags, bias, alpha, packed, n, k, need, split_rows, min_rows, nvfp4, packed_only, usable)
PyObject* host_linear_plan(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *q, *s, *wgs, *ags, *bias, *alpha, *packed;
  long long n, k, need, split_rows, min_rows;
  int nvfp4, packed_only, usable;
  if (!PyArg_ParseTuple(args, "OOOOOOOLLLLLppp", &q, &s, &wgs, &ags, &bias, &alpha, &packed, &n, &k, &need, &split_rows,
                        &min_rows, &nvfp4, &packed_only, &usable))
    return nullptr;
  THPObjectPtr o(plan_new<LinearPlan>(&LinearPlanType, nullptr, nullptr));
  if (!o) return nullptr;
  auto* b = ((LinearPlan*)o.get())->b;
  if (!b->qweight.take(q, false) || !b->scales.take(s, true) || !b->wgs.take(wgs, true) || !b->ags.take(ags, true) ||
      !b->bias.take(bias, true))
    Py_RETURN_NONE;
  b->n = n; b->k = k; b->kp = (k + 255) / 256 * 256;
  b->need = need; b->split_rows = split_rows; b->min_rows = min_rows;
  b->nvfp4 = nvfp4; b->packed_only = packed_only; b->usable = usable;
  if (usable) {
    const at::Tensor* a = tensor_of(alpha);
    if (!a || !plain_cuda(*a) || a->scalar_type() != at::kFloat || a->numel() != 1) Py_RETURN_NONE;
    b->alpha = *a;
    b->alpha_obj = Py_NewRef(alpha);
    const at::Tensor *wp = tensor_of(q), *wsp = tensor_of(s);
    if (!packed_only) {
      if (!PyTuple_Check(packed) || PyTuple_GET_SIZE(packed) != 3 || !take_tensor(PyTuple_GET_ITEM(packed, 1), b->wp) ||
          !take_tensor(PyTuple_GET_ITEM(packed, 2), b->wsp))
        Py_RETURN_NONE;
      b->packed = Py_NewRef(packed);
      wp = &b->wp;
      wsp = &b->wsp;
    }
    const int64_t rows = (n + 31) / 32 * 32;
    if (!wp->defined() || !wsp->defined() || !wp->is_contiguous() || !wsp->is_contiguous() ||
        wp->numel() < rows * b->kp / 2 || wsp->numel() < rows * b->kp / (nvfp4 ? 16 : 32))
      Py_RETURN_NONE;
    if (b->bias.impl && (b->bias.held.scalar_type() != at::kBFloat16 || !b->bias.held.is_contiguous() || b->bias.held.numel() != n))
      Py_RETURN_NONE;
  }
  return o.release();
  END_HANDLE_TH_ERRORS
}
// group_plan(members, splits, wgs, ags, alpha, wp, wsp, bias, k, nvfp4, usable) -> plan or None; not usable: a marker for
// these members
PyObject* host_group_plan(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *members, *splits, *wgs, *ags, *alpha, *wp, *wsp, *bias;
  long long k;
  int nvfp4, usable;
  if (!PyArg_ParseTuple(args, "O!O!OOOOOOLpp", &PyTuple_Type, &members, &PyTuple_Type, &splits, &wgs, &ags, &alpha, &wp, &wsp,
                        &bias, &k, &nvfp4, &usable))
    return nullptr;
  THPObjectPtr o(plan_new<GroupPlan>(&GroupPlanType, nullptr, nullptr));
  if (!o) return nullptr;
  auto* b = ((GroupPlan*)o.get())->b;
  const Py_ssize_t count = PyTuple_GET_SIZE(splits);
  if (PyTuple_GET_SIZE(members) != 3 * count || count < 1 || count > 4) Py_RETURN_NONE;
  for (Py_ssize_t i = 0; i < 3 * count; ++i) {
    b->members.emplace_back();
    if (!b->members.back().take(PyTuple_GET_ITEM(members, i), false)) Py_RETURN_NONE;
  }
  b->usable = usable;
  if (!usable) return o.release();
  int64_t n = 0;
  for (Py_ssize_t i = 0; i < count; ++i) {
    const long long s = PyLong_AsLongLong(PyTuple_GET_ITEM(splits, i));
    if (PyErr_Occurred()) return nullptr;
    if (s < 1 || s % 256 != 0) Py_RETURN_NONE;
    b->splits.push_back(s);
    n += s;
  }
  const at::Tensor* a = tensor_of(alpha);
  if (!b->wgs.take(wgs, true) || !b->ags.take(ags, true) || !a || !plain_cuda(*a) || a->scalar_type() != at::kFloat ||
      a->numel() != 1 || !take_tensor(wp, b->wp) || !take_tensor(wsp, b->wsp) || !take_tensor(bias, b->bias) || !b->wp.defined() || !b->wsp.defined())
    Py_RETURN_NONE;
  b->alpha = *a;
  b->k = k;
  b->kp = (k + 255) / 256 * 256;
  b->nvfp4 = nvfp4;
  if (b->wp.numel() * 2 != n * b->kp || b->wsp.numel() != n * b->kp / (nvfp4 ? 16 : 32) || (b->bias.defined() && b->bias.numel() != n))
    Py_RETURN_NONE;
  b->alpha_obj = Py_NewRef(alpha);
  return o.release();
  END_HANDLE_TH_ERRORS
}

// configure(library path, binding attributes, shared slot, workspaces, eager globals, QuantizedActivations, policy,
// activation rows from which the MXFP4 and NVFP4 matmul operators re-tile their operands, and from which MXFP4 layers
// run on packed weights)
PyObject* host_configure(PyObject*, PyObject* args) {
  const char* path;
  PyObject *binding, *shared, *workspaces, *globals, *type;
  int policy;
  if (!PyArg_ParseTuple(args, "sO!O!O!O!O!iiii", &path, &PyDict_Type, &binding, &PyDict_Type, &shared, &PyDict_Type, &workspaces,
                        &PyDict_Type, &globals, &PyType_Type, &type, &policy, &g_packed_rows_mx, &g_packed_rows_nv,
                        &g_linear_rows_mx))
    return nullptr;
  if (!PyType_IsSubtype((PyTypeObject*)type, &ActivationsType)) {
    PyErr_SetString(PyExc_TypeError, "the activations type must derive from Activations");
    return nullptr;
  }
  void* lib = dlopen(path, RTLD_NOW | RTLD_LOCAL);   // (stays open: the entry points are used until the process ends)
  if (!lib) {
    PyErr_SetString(PyExc_RuntimeError, dlerror());
    return nullptr;
  }
  for (int e = 0; e < kEntries; ++e) {
    g_fn[e] = dlsym(lib, kEntryNames[e]);
    g_entry_name[e] = PyUnicode_InternFromString(kEntryNames[e]);
    PyObject* fn = g_entry_name[e] ? PyDict_GetItem(binding, g_entry_name[e]) : nullptr;
    if (!g_fn[e] || !fn) {
      PyErr_Format(PyExc_RuntimeError, "%s has no entry point %s", path, kEntryNames[e]);
      return nullptr;
    }
    g_entry_object[e] = Py_NewRef(fn);
  }
  g_shared = Py_NewRef(shared);
  g_workspaces = Py_NewRef(workspaces);
  g_eager_globals = Py_NewRef(globals);
  g_activations = (PyTypeObject*)Py_NewRef(type);
  g_policy = policy;
  g_binding = Py_NewRef(binding);   // (last: calls before this take the Python path)
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"linear", (PyCFunction)(void (*)())host_linear, METH_FASTCALL, nullptr},
    {"rmsnorm", (PyCFunction)(void (*)())host_rmsnorm, METH_FASTCALL, nullptr},
    {"group", (PyCFunction)(void (*)())host_group, METH_FASTCALL, nullptr},
    {"norm_group", (PyCFunction)(void (*)())host_group, METH_FASTCALL, nullptr},
    {"gated_mlp", (PyCFunction)(void (*)())host_gated_mlp, METH_FASTCALL, nullptr},
    {"gated_down", (PyCFunction)(void (*)())host_gated_down, METH_FASTCALL, nullptr},
    {"quantize_mx", (PyCFunction)(void (*)())host_quantize<false>, METH_FASTCALL, nullptr},
    {"quantize_nv", (PyCFunction)(void (*)())host_quantize<true>, METH_FASTCALL, nullptr},
    {"matmul_mx", (PyCFunction)(void (*)())host_matmul<false>, METH_FASTCALL, nullptr},
    {"matmul_nv", (PyCFunction)(void (*)())host_matmul<true>, METH_FASTCALL, nullptr},
    {"linear_plan_current", host_linear_plan_current, METH_VARARGS, nullptr},
    {"quant_plan_current", host_quant_plan_current, METH_VARARGS, nullptr},
    {"quant_plan", host_quant_plan, METH_VARARGS, nullptr},
    {"linear_plan", host_linear_plan, METH_VARARGS, nullptr},
    {"group_plan", host_group_plan, METH_VARARGS, nullptr},
    {"configure", host_configure, METH_VARARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_fpq_host", "Native host path of the eager layers", -1, methods,
                          nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fpq_host() {
  struct {
    PyObject** slot;
    const char* text;
  } names[] = {{&s_qweight, "qweight"}, {&s_scales, "scales"}, {&s_wgs, "weight_global_scale"}, {&s_ags, "act_global_scale"},
               {&s_h, "forward_hadamard_matrix"}, {&s_bias, "bias"}, {&s_plan, "_fpq_plan"}, {&s_qplan, "_fpq_qplan"},
               {&s_alpha, "_fpq_alpha"}, {&s_packed, "_fpq_packed"}, {&s_share, "SHARE_ACT_QUANT"},
               {&s_parameters, "_parameters"}, {&s_buffers, "_buffers"}, {&s_weight, "weight"},
               {&s_eps, "variance_epsilon"}, {&s_rotation, "_fpq_rotation"},
               {&s_splitk, "_fpq_splitk"}};
  for (auto& n : names)
    if (!(*n.slot = PyUnicode_InternFromString(n.text))) return nullptr;
  struct {
    PyTypeObject* type;
    size_t size;
    destructor dealloc;
  } plans[] = {{&QuantPlanType, sizeof(QuantPlan), quant_dealloc},
               {&LinearPlanType, sizeof(LinearPlan), linear_dealloc},
               {&GroupPlanType, sizeof(GroupPlan), group_dealloc}};
  for (auto& p : plans) {
    p.type->tp_basicsize = (Py_ssize_t)p.size;
    p.type->tp_dealloc = p.dealloc;
    p.type->tp_flags = Py_TPFLAGS_DEFAULT;
    p.type->tp_methods = plan_methods;
    if (PyType_Ready(p.type) < 0) return nullptr;
  }
  ActivationsType.tp_basicsize = sizeof(Activations);
  ActivationsType.tp_dealloc = activations_dealloc;
  ActivationsType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE;
  ActivationsType.tp_members = activation_members;
  ActivationsType.tp_new = PyType_GenericNew;
  if (PyType_Ready(&ActivationsType) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  if (PyModule_AddObjectRef(m, "Activations", (PyObject*)&ActivationsType) < 0) return nullptr;
  return m;
}
