// The host work of a layer call in its usual form: what moe.py does with the arguments, in native code.
//
// A small call waits for the host: in Python, taking a layer's arguments apart (fourteen tensors checked, two allocations, forty
// fields of a struct filled through ctypes) took 10 to 17 us beside 2.8 us a launch.  Here the same checks take 1 to 2 us.
//   A function of this module returns None for whatever it does not take as it is -- tensors of other types, layouts or
// subclasses, plain or per-row weights, wrong shapes, active modes and transforms -- and touches nothing; moe.py then
// goes the general way, which converts or refuses.  So nothing here raises an error of its own.
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/headeronly/version.h>

#include <climits>

#include "moe_hip.h"

namespace {

// the library's functions, and moe.py's
struct Bound {
  decltype(&moe_forward_workspace_bytes) workspace_bytes;
  decltype(&moe_forward) forward, forward_f32;
  decltype(&moe_forward_selected) selected;
  decltype(&moe_router_workspace_bytes) router_workspace_bytes;
  decltype(&moe_routing) routing;
  PyObject *check, *router_weight, *device, *raw_stream;
} bound = {};
PyObject *k_w, *k_scale_inv, *k_gate, *k_up, *k_down, *k_shared_gate, *k_shared_up, *k_shared_down, *k_router, *k_shared_router;

// A tensor that its data pointer stands for: contiguous, on the GPU, with no subclass, transform or lazy form around it.
const at::Tensor* usable(PyObject* o, at::ScalarType type, int64_t dim) {
  if (!o || !THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::Functionalize, c10::DispatchKey::FuncTorchBatched,
                                         c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched, c10::DispatchKey::Conjugate,
                                         c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.key_set().has_any(wrapped) || !t.has_storage()) return nullptr;
  return t.scalar_type() == type && t.dim() == dim && t.is_contiguous() ? &t : nullptr;
}
bool plain_int(PyObject* o, int* v) {
  if (!PyLong_Check(o)) return false;
  int overflow = 0;
  const long n = PyLong_AsLongAndOverflow(o, &overflow);
  if (overflow || n < INT_MIN || n > INT_MAX) return false;
  *v = (int)n;
  return true;
}
bool plain_float(PyObject* o, float* v) {
  if (!PyFloat_CheckExact(o)) return false;
  *v = (float)PyFloat_AS_DOUBLE(o);
  return true;
}
PyObject* item(PyObject* dict, PyObject* key) { return PyDict_GetItemWithError(dict, key); }   // borrowed

// One call: the struct, and the tensors that it points into (another thread may drop the caller's while this one runs).
struct Call {
  MoeForwardArgs a{};
  at::Tensor held[20];
  int n_held = 0;
  const void* hold(const at::Tensor& t) {
    held[n_held++] = t;
    return t.data_ptr();
  }
  // a block-scaled fp8 projection of `groups` x n x k (0: as the tensor says)
  bool weight(PyObject* d, int& groups, int& n, int& k, const uint8_t** w, const float** s) {
    if (!d || !PyDict_CheckExact(d)) return false;
    const at::Tensor *q = usable(item(d, k_w), at::kFloat8_e4m3fn, 3), *sc = usable(item(d, k_scale_inv), at::kFloat, 3);
    if (!q || !sc) return false;
    for (int i = 0; i < 3; ++i)
      if (q->size(i) > INT_MAX || sc->size(i) != (i ? q->size(i) / 128 : q->size(i))) return false;
    if (!groups) groups = (int)q->size(0);
    if (!n) n = (int)q->size(1);
    if (!k) k = (int)q->size(2);
    if (q->size(0) != groups || q->size(1) != n || q->size(2) != k) return false;
    *w = (const uint8_t*)hold(*q);
    *s = (const float*)hold(*sc);
    return true;
  }
};
bool modes_active() { return at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set(); }

bool current_stream(moe_stream_t* s) {
  PyObject* dev = PyObject_CallNoArgs(bound.device);
  if (!dev) return false;
  PyObject* raw = PyObject_CallOneArg(bound.raw_stream, dev);
  Py_DECREF(dev);
  if (!raw) return false;
  *s = (moe_stream_t)PyLong_AsVoidPtr(raw);
  Py_DECREF(raw);
  return !PyErr_Occurred();
}
// moe.py's (E, D) bf16 form of a router weight, cached there; false: see the error state, or none is set and it is not usable
bool router_weight(PyObject* w, const char* name, at::Tensor* out) {
  if (!THPVariable_CheckExact(w)) return false;
  PyObject* n = PyUnicode_FromString(name);
  if (!n) return false;
  PyObject* r = PyObject_CallFunctionObjArgs(bound.router_weight, w, n, nullptr);
  Py_DECREF(n);
  if (!r) return false;
  const at::Tensor* t = usable(r, at::kBFloat16, 2);
  if (t) *out = *t;
  Py_DECREF(r);
  return t != nullptr;
}
PyObject* general_way() {
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

// What the entry points below have in common.  experts / shared: the six projections' dicts (shared[0] null: no shared expert).
struct Inputs {
  PyObject *x, *logits, *experts[3], *shared[3], *router, *shared_router, *bias, *norm_weight, *idx, *w;
  int rank, io_f32;
};
PyObject* run(Call& c, const Inputs& in) {
  MoeForwardArgs& a = c.a;
  // (the caller's dict alone may hold these two, and router_weight runs Python code, which lets other threads at it)
  Py_XINCREF(in.router);
  Py_XINCREF(in.shared_router);
  const THPObjectPtr router(in.router), shared_router(in.shared_router);
  const at::Tensor* x = usable(in.x, in.io_f32 ? at::kFloat : at::kBFloat16, in.rank);
  if (!x || modes_active()) return general_way();
  const int64_t rows = in.rank == 2 ? x->size(0) : x->size(0) * x->size(1), D = x->size(in.rank - 1);
  if (rows > INT_MAX || D > INT_MAX || D == 0) return general_way();
  a.M = (int)rows, a.D = (int)D;
  a.x = c.hold(*x);
  if (!c.weight(in.experts[0], a.E, a.I, a.D, &a.w_gate, &a.sw_gate) || !a.E || !a.I || !c.weight(in.experts[1], a.E, a.I, a.D, &a.w_up, &a.sw_up) ||
      !c.weight(in.experts[2], a.E, a.D, a.I, &a.w_down, &a.sw_down))
    return general_way();
  if (in.shared[0]) {
    int one = 1;
    if (!c.weight(in.shared[0], one, a.SI, a.D, &a.ws_gate, &a.sws_gate) || !a.SI || !c.weight(in.shared[1], one, a.SI, a.D, &a.ws_up, &a.sws_up) ||
        !c.weight(in.shared[2], one, a.D, a.SI, &a.ws_down, &a.sws_down))
      return general_way();
  }
  if (in.bias) {
    const at::Tensor* b = usable(in.bias, at::kFloat, 1);
    if (!b || b->size(0) < a.E) return general_way();
    a.bias = (const float*)c.hold(*b);
  }
  if (in.norm_weight) {
    const at::Tensor* n = usable(in.norm_weight, at::kFloat, 1);
    if (!n || n->size(0) != D) return general_way();
    a.norm_weight = (const float*)c.hold(*n);
  }
  const at::Tensor *idx = nullptr, *w = nullptr;
  if (in.idx) {
    idx = usable(in.idx, at::kInt, 2), w = usable(in.w, at::kFloat, 2);
    if (!idx || !w || idx->size(0) != rows || w->sizes() != idx->sizes() || idx->size(1) != a.k) return general_way();
    c.hold(*idx), c.hold(*w);
  } else if (in.logits) {
    const at::Tensor* l = usable(in.logits, at::kFloat, 2);
    if (!l || in.router || l->size(0) != rows || l->size(1) != a.E) return general_way();
    a.logits = (const float*)c.hold(*l);
  } else if (!in.router) {
    return general_way();
  }
  if (in.shared_router && (!in.router || !in.shared[0])) return general_way();
  if (in.router) {
    at::Tensor wr;
    if (!router_weight(in.router, "gate_weight", &wr) || wr.size(0) != a.E || wr.size(1) != D) return general_way();
    a.w_router = c.hold(wr);
  }
  if (in.shared_router) {
    at::Tensor wsg;
    if (!router_weight(in.shared_router, "shared_expert_gate_weight", &wsg) || wsg.size(0) != 1 || wsg.size(1) != D) return general_way();
    a.w_shared_gate = c.hold(wsg);
  }
  at::Tensor out = at::empty_like(*x);
  a.out = out.data_ptr();
  const size_t bytes = bound.workspace_bytes(a.M, a.D, a.E, a.k, a.I, a.SI);
  const at::Tensor ws = at::empty({(int64_t)(bytes > 16 ? bytes : 16)}, at::TensorOptions().dtype(at::kByte).device(x->device()));
  moe_stream_t stream;
  if (!current_stream(&stream)) return nullptr;
  PyThreadState* state = PyEval_SaveThread();
  const int code = idx ? bound.selected(&a, (const int32_t*)idx->data_ptr(), (const float*)w->data_ptr(), ws.data_ptr(), bytes, stream)
                       : (in.io_f32 ? bound.forward_f32 : bound.forward)(&a, ws.data_ptr(), bytes, stream);
  PyEval_RestoreThread(state);
  if (code) {   // (moe.py's check raises it, with the library's message for this thread)
    PyObject* n = PyLong_FromLong(code);
    PyObject* r = n ? PyObject_CallOneArg(bound.check, n) : nullptr;
    Py_XDECREF(n);
    Py_XDECREF(r);
    return general_way();
  }
  return THPVariable_Wrap(out);
}
PyObject* or_null(PyObject* o) { return o == Py_None ? nullptr : o; }
void three(PyObject* d, PyObject* const (&keys)[3], PyObject* (&out)[3]) {
  for (int i = 0; i < 3; ++i) out[i] = item(d, keys[i]);
}

// experts(x, logits, top_k, experts, routing code, bias, n_group, topk_group, renorm, routed_scale, shared, gate_weight,
//         shared_expert_gate_weight, norm_weight, norm_eps, add_residual, io_f32, selected, rank)
PyObject* experts(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 19) return general_way();
  Call c;
  Inputs in{};
  MoeForwardArgs& a = c.a;
  PyObject* const names[3] = {k_gate, k_up, k_down};
  int residual;
  if (!plain_int(v[2], &a.k) || !PyDict_CheckExact(v[3]) || !plain_int(v[4], &a.routing) || !plain_int(v[6], &a.n_group) ||
      !plain_int(v[7], &a.topk_group) || !plain_int(v[8], &a.renorm) || !plain_float(v[9], &a.routed_scale) ||
      !plain_float(v[14], &a.norm_eps) || !plain_int(v[15], &residual) || !plain_int(v[16], &in.io_f32) || !plain_int(v[18], &in.rank) ||
      (in.rank != 2 && in.rank != 3) || (v[10] != Py_None && !PyDict_CheckExact(v[10])))
    return general_way();
  a.add_residual = residual != 0;
  in.x = v[0], in.logits = or_null(v[1]), in.bias = or_null(v[5]), in.router = or_null(v[11]), in.shared_router = or_null(v[12]);
  in.norm_weight = or_null(v[13]);
  if (!in.norm_weight) a.norm_eps = 0.f;
  three(v[3], names, in.experts);
  if (v[10] != Py_None) {
    three(v[10], names, in.shared);
    if (!in.shared[0]) return general_way();
  }
  if (v[17] != Py_None) {
    if (!PyTuple_CheckExact(v[17]) || PyTuple_GET_SIZE(v[17]) != 2 || in.router || in.logits) return general_way();
    in.idx = PyTuple_GET_ITEM(v[17], 0), in.w = PyTuple_GET_ITEM(v[17], 1);
  }
  return run(c, in);
  END_HANDLE_TH_ERRORS
}

// layer(x, params, top_k, norm_weight, norm_eps, add_residual)
PyObject* layer(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Call c;
  Inputs in{};
  MoeForwardArgs& a = c.a;
  int residual;
  if (n != 6 || !THPVariable_CheckExact(v[0]) || !PyDict_CheckExact(v[1]) || !plain_int(v[2], &a.k) || !plain_float(v[4], &a.norm_eps) ||
      !plain_int(v[5], &residual))
    return general_way();
  a.add_residual = residual != 0;
  a.routing = MOE_ROUTING_SOFTMAX, a.n_group = a.topk_group = a.renorm = 1, a.routed_scale = 1.f;
  in.x = v[0], in.rank = 3;
  in.io_f32 = THPVariable_Unpack(v[0]).scalar_type() == at::kFloat;
  in.norm_weight = or_null(v[3]);
  if (!in.norm_weight) a.norm_eps = 0.f;
  in.router = item(v[1], k_router);
  if (!in.router || in.router == Py_None) return general_way();
  three(v[1], {k_gate, k_up, k_down}, in.experts);
  PyObject* shared = item(v[1], k_shared_gate);
  if (shared && shared != Py_None) {
    three(v[1], {k_shared_gate, k_shared_up, k_shared_down}, in.shared);
    in.shared_router = item(v[1], k_shared_router);
    if (in.shared_router == Py_None) in.shared_router = nullptr;
  }
  const at::Tensor* x = usable(in.x, in.io_f32 ? at::kFloat : at::kBFloat16, 3);
  if (!x || (in.io_f32 && (uintptr_t)x->data_ptr() % 16)) return general_way();   // (moe.py copies such a view)
  return run(c, in);
  END_HANDLE_TH_ERRORS
}

// routing(x, gate_weight, top_k) -> (indices, weights)
PyObject* routing(PyObject*, PyObject* const* v, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int k;
  if (n != 3 || !plain_int(v[2], &k) || k < 0) return general_way();
  const at::Tensor* seen = usable(v[0], at::kBFloat16, 2);
  if (!seen || modes_active() || seen->size(0) > INT_MAX || seen->size(1) > INT_MAX) return general_way();
  const at::Tensor x = *seen;
  at::Tensor wr;
  if (!router_weight(v[1], "gate_weight", &wr) || wr.size(1) != x.size(1) || wr.size(0) > INT_MAX) return general_way();
  const int M = (int)x.size(0), D = (int)x.size(1), E = (int)wr.size(0);
  const at::Tensor idx = at::empty({M, k}, x.options().dtype(at::kInt).requires_grad(false));
  const at::Tensor w = at::empty({M, k}, x.options().dtype(at::kFloat).requires_grad(false));
  const size_t bytes = bound.router_workspace_bytes(M, D, E);
  const at::Tensor ws = at::empty({(int64_t)(bytes > 16 ? bytes : 16)}, at::TensorOptions().dtype(at::kByte).device(x.device()));
  moe_stream_t stream;
  if (!current_stream(&stream)) return nullptr;
  PyThreadState* state = PyEval_SaveThread();
  const int code = bound.routing(x.data_ptr(), M, D, wr.data_ptr(), E, k, 1, (int32_t*)idx.data_ptr(), (float*)w.data_ptr(), ws.data_ptr(),
                                 bytes, stream);
  PyEval_RestoreThread(state);
  if (code) {
    PyObject* c = PyLong_FromLong(code);
    PyObject* r = c ? PyObject_CallOneArg(bound.check, c) : nullptr;
    Py_XDECREF(c);
    Py_XDECREF(r);
    return general_way();
  }
  PyObject *pi = THPVariable_Wrap(idx), *pw = THPVariable_Wrap(w);
  PyObject* pair = pi && pw ? PyTuple_Pack(2, pi, pw) : nullptr;
  Py_XDECREF(pi);
  Py_XDECREF(pw);
  return pair;
  END_HANDLE_TH_ERRORS
}

// bind(addresses of the library's six functions, in the order of Bound; moe.py's check and router_weight; the current device, a device's current stream)
PyObject* bind(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (n != 10) {
    PyErr_SetString(PyExc_TypeError, "bind: ten arguments");
    return nullptr;
  }
  void* at[6];
  for (int i = 0; i < 6; ++i)
    if (!(at[i] = PyLong_AsVoidPtr(v[i]))) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null address");
      return nullptr;
    }
  for (int i = 6; i < 10; ++i) Py_INCREF(v[i]);   // (held until the process ends)
  bound = Bound{(decltype(bound.workspace_bytes))at[0], (decltype(bound.forward))at[1], (decltype(bound.forward_f32))at[2],
                (decltype(bound.selected))at[3], (decltype(bound.router_workspace_bytes))at[4], (decltype(bound.routing))at[5],
                v[6], v[7], v[8], v[9]};
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"bind", (PyCFunction)(void (*)())bind, METH_FASTCALL, nullptr},
                         {"experts", (PyCFunction)(void (*)())experts, METH_FASTCALL, nullptr},
                         {"layer", (PyCFunction)(void (*)())layer, METH_FASTCALL, nullptr},
                         {"routing", (PyCFunction)(void (*)())routing, METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "moe_call", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_moe_call() {
  struct { PyObject** at; const char* name; } const keys[] = {
      {&k_w, "w"}, {&k_scale_inv, "scale_inv"}, {&k_gate, "gate_proj"}, {&k_up, "up_proj"}, {&k_down, "down_proj"},
      {&k_shared_gate, "shared_gate_proj"}, {&k_shared_up, "shared_up_proj"}, {&k_shared_down, "shared_down_proj"},
      {&k_router, "gate_weight"}, {&k_shared_router, "shared_expert_gate_weight"}};
  for (const auto& k : keys)
    if (!(*k.at = PyUnicode_InternFromString(k.name))) return nullptr;
  PyObject* m = PyModule_Create(&module);
  // (what this was compiled against: moe.py compares it with what there is)
  if (!m || PyModule_AddIntConstant(m, "args_bytes", (long)sizeof(MoeForwardArgs)) || PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION)) {
    Py_XDECREF(m);
    return nullptr;
  }
  return m;
}
