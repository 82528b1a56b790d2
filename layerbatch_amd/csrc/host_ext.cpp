// CPython extension layerbatch_amd._host: the host side of the modules' forward calls in C++.
//
// A forward call of moe.py checks every tensor it hands to the C ABI, allocates the outputs and the
// workspace and enqueues three to eight kernels. In Python that took about 40 us, while the kernels
// of a one-token Qwen3-30B-A3B layer take 25 us and those of a router or a dense MLP 10-20 us, so
// eager calls of small batches were bound by it. Here one call does the same in a few microseconds
// plus the launches. Nothing is kept between calls: every call reads the module's tensors and checks
// them anew.
//
// Each entry takes the plain case only: modules and tensors of exactly the expected types, with the
// attributes that moe.py's constructors and load_fp8_ leave, no packed weights, no torch modes (but a
// default device) or transforms in effect. It returns None for anything else (a wrong shape, dtype
// or device included) before any allocation or launch, and moe.py's general path then runs the call
// or raises.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/PyInterpreter.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/csrc/utils/pybind.h>
#include <torch/headeronly/version.h>

#include <cstring>
#include <optional>

#include "../../include/lbmoe.h"

namespace {

// Entry points of liblbmoe.so, bound once by _lib.lib() (which has loaded the library).
struct Abi {
  decltype(&lbmoe_status_string) status_string;
  decltype(&lbmoe_workspace_size) workspace_size;
  decltype(&lbmoe_forward) forward;
  decltype(&lbmoe_forward_norm) forward_norm;
  decltype(&lbmoe_router_logits) router_logits;
  decltype(&lbmoe_route) route;
  decltype(&lbmoe_experts) experts;
  decltype(&lbmoe_dense_mlp_workspace_size) dense_mlp_workspace_size;
  decltype(&lbmoe_dense_mlp) dense_mlp;
};
Abi abi{};

// The module classes and torch's default-device mode, set by bind (strong references).
PyTypeObject *t_router, *t_experts, *t_mlp, *t_block, *t_linear, *t_device_context;

struct Names {
  PyObject *parameters, *modules, *weight, *bias, *gate, *experts, *shared_expert,
      *shared_expert_gate, *gate_proj, *up_proj, *down_proj, *gate_up_proj, *top_k, *num_experts,
      *hidden_size, *intermediate_size, *logit_bias, *weight_dtype, *gate_up_q, *gate_up_scale,
      *down_q, *down_scale, *gate_up_tiled, *q, *up, *down, *eps;
} nm;

// Borrowed reference, or null.
PyObject* get(PyObject* dict, PyObject* name) { return PyDict_GetItemWithError(dict, name); }

PyObject* instance_dict(PyObject* obj) {
  PyObject** d = _PyObject_GetDictPtr(obj);
  return d && *d && PyDict_CheckExact(*d) ? *d : nullptr;
}

bool int_attr(PyObject* dict, PyObject* name, int64_t* out) {
  PyObject* o = get(dict, name);
  if (!o || !PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *out = PyLong_AsLongLongAndOverflow(o, &overflow);
  return !overflow && *out >= 0 && *out <= INT32_MAX;
}

// The parameters or submodules of a module whose table holds exactly n entries.
PyObject* table(PyObject* dict, PyObject* name, Py_ssize_t n) {
  PyObject* t = get(dict, name);
  return t && PyDict_CheckExact(t) && PyDict_GET_SIZE(t) == n ? t : nullptr;
}

constexpr int kMaxTensors = 24;
// The tensors of one call, held for its length (another thread may replace a module's weight while
// the launches run without the interpreter lock), all on one device.
struct Tensors {
  at::Tensor t[kMaxTensors];
  int n = 0;
  c10::Device device{c10::DeviceType::CPU};

  // A plain strided GPU tensor on the call's device (the first one sets it), or null.
  const at::Tensor* add(PyObject* o) {
    if (!o || n == kMaxTensors || !THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& v = THPVariable_Unpack(o);
    if (!v.defined() || !v.is_cuda() || !v.has_storage() || v.layout() != c10::kStrided)
      return nullptr;
    constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python,
                                           c10::DispatchKey::PythonTLSSnapshot,
                                           c10::DispatchKey::Functionalize,
                                           c10::DispatchKey::FuncTorchBatched,
                                           c10::DispatchKey::FuncTorchGradWrapper});
    if (v.key_set().has_any(wrapped)) return nullptr;
    if (n == 0) device = v.device();
    else if (v.device() != device) return nullptr;
    t[n] = v;
    return &t[n++];
  }
  const at::Tensor* add(PyObject* o, c10::ScalarType dtype, int64_t ndim) {
    const at::Tensor* v = add(o);
    return v && v->scalar_type() == dtype && v->dim() == ndim && v->is_contiguous() ? v : nullptr;
  }
  template <class... D>
  const void* shaped(PyObject* o, c10::ScalarType dtype, D... dims) {
    const at::Tensor* v = add(o, dtype, sizeof...(dims));
    if (!v || v->sizes() != at::IntArrayRef{static_cast<int64_t>(dims)...}) return nullptr;
    return v->const_data_ptr();
  }
};

// Torch function or dispatch modes, functorch transforms: the general path's business. A default
// device is let through: torch.set_default_device leaves its mode on the stack for good (an engine's
// model runner sets one), and it only gives a device to calls that name none, which no allocation
// here or in the general path is.
bool plain_torch() {
  using Modes = at::impl::PythonTorchFunctionTLS;
  for (int64_t i = 0, n = Modes::stack_len(); i < n; ++i)
    if (Py_TYPE(Modes::get_stack_at(i)->ptr(getPyInterpreter())) != t_device_context) return false;
  if (c10::impl::TorchDispatchModeTLS::any_modes_set()) return false;
  constexpr c10::DispatchKeySet special({c10::DispatchKey::Python,
                                         c10::DispatchKey::PythonTLSSnapshot,
                                         c10::DispatchKey::Functionalize,
                                         c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
                                         c10::DispatchKey::FuncTorchDynamicLayerBackMode});
  return !c10::impl::tls_local_dispatch_key_set().included_.has_any(special);
}

// An nn.Linear without bias: its weight, or null.
PyObject* linear_weight(PyObject* mod) {
  if (!mod || Py_TYPE(mod) != t_linear) return nullptr;
  PyObject* d = instance_dict(mod);
  if (!d || get(d, nm.weight) || !table(d, nm.modules, 0)) return nullptr;
  PyObject* p = table(d, nm.parameters, 2);
  if (!p || get(p, nm.bias) != Py_None) return nullptr;
  return get(p, nm.weight);
}

constexpr auto kBf16 = c10::ScalarType::BFloat16;
constexpr auto kF32 = c10::ScalarType::Float;

bool fill_router(PyObject* mod, Tensors& ts, lbmoe_layer* L) {
  if (!mod || Py_TYPE(mod) != t_router) return false;
  PyObject* d = instance_dict(mod);
  int64_t E, k;
  if (!d || get(d, nm.weight) || !table(d, nm.modules, 0) || !int_attr(d, nm.num_experts, &E) ||
      !int_attr(d, nm.top_k, &k))
    return false;
  PyObject* p = table(d, nm.parameters, 1);
  PyObject* bias = get(d, nm.logit_bias);
  if (!p || !bias) return false;
  const at::Tensor* w = ts.add(get(p, nm.weight), kBf16, 2);
  if (!w || w->size(0) != E || w->size(1) > INT32_MAX) return false;
  L->hidden_size = static_cast<int32_t>(w->size(1));
  L->num_experts = static_cast<int32_t>(E);
  L->top_k = static_cast<int32_t>(k);
  L->gate_weight = w->const_data_ptr();
  if (bias != Py_None) {
    L->logit_bias = static_cast<const float*>(ts.shaped(bias, kF32, E));
    if (!L->logit_bias) return false;
  }
  return true;
}

bool fill_experts(PyObject* mod, Tensors& ts, lbmoe_layer* L) {
  if (!mod || Py_TYPE(mod) != t_experts) return false;
  PyObject* d = instance_dict(mod);
  int64_t E, H, I, dt;
  if (!d || get(d, nm.gate_up_proj) || get(d, nm.down_proj) || !table(d, nm.modules, 0) ||
      !int_attr(d, nm.num_experts, &E) || !int_attr(d, nm.hidden_size, &H) ||
      !int_attr(d, nm.intermediate_size, &I) || !int_attr(d, nm.weight_dtype, &dt))
    return false;
  PyObject* p = table(d, nm.parameters, 2);
  if (!p) return false;
  L->hidden_size = static_cast<int32_t>(H);
  L->num_experts = static_cast<int32_t>(E);
  L->moe_intermediate_size = static_cast<int32_t>(I);
  L->weight_dtype = static_cast<int32_t>(dt);
  PyObject *gu = get(p, nm.gate_up_proj), *dn = get(p, nm.down_proj);
  if (dt == LBMOE_W_BF16) {
    if (get(d, nm.gate_up_tiled) != Py_None) return false;
    L->gate_up_proj = ts.shaped(gu, kBf16, E, 2 * I, H);
    L->down_proj = ts.shaped(dn, kBf16, E, H, I);
    // every tensor that _same_device looks at: fp8 leftovers are None here
    for (PyObject* n : {nm.gate_up_q, nm.gate_up_scale, nm.down_q, nm.down_scale})
      if (get(d, n) != Py_None) return false;
    return L->gate_up_proj && L->down_proj;
  }
  if (dt != LBMOE_W_FP8_E4M3 || !ts.add(gu) || !ts.add(dn)) return false;
  const at::Tensor *q0 = ts.add(get(d, nm.gate_up_q)), *s0 = ts.add(get(d, nm.gate_up_scale));
  const at::Tensor *q1 = ts.add(get(d, nm.down_q)), *s1 = ts.add(get(d, nm.down_scale));
  if (!q0 || !s0 || !q1 || !s1 || s0->scalar_type() != kF32 || s1->scalar_type() != kF32)
    return false;
  L->gate_up_proj = q0->const_data_ptr();
  L->down_proj = q1->const_data_ptr();
  L->gate_up_scale = static_cast<const float*>(s0->const_data_ptr());
  L->down_scale = static_cast<const float*>(s1->const_data_ptr());
  return true;
}

// The shared-expert fields of L, and H (the gate projection's width).
bool fill_mlp(PyObject* mod, Tensors& ts, lbmoe_layer* L, int64_t* H, int64_t* dtype) {
  if (!mod || Py_TYPE(mod) != t_mlp) return false;
  PyObject* d = instance_dict(mod);
  if (!d || !table(d, nm.parameters, 0) || !int_attr(d, nm.weight_dtype, dtype)) return false;
  PyObject* m = table(d, nm.modules, 3);
  if (!m || get(d, nm.gate_proj) || get(d, nm.up_proj) || get(d, nm.down_proj)) return false;
  PyObject* w[3] = {linear_weight(get(m, nm.gate_proj)), linear_weight(get(m, nm.up_proj)),
                    linear_weight(get(m, nm.down_proj))};
  const at::Tensor* g = ts.add(w[0]);
  if (!g || g->dim() != 2 || g->size(0) > INT32_MAX || g->size(1) > INT32_MAX) return false;
  const int64_t Is = g->size(0);
  *H = g->size(1);
  L->shared_intermediate_size = static_cast<int32_t>(Is);
  PyObject* q = get(d, nm.q);
  if (*dtype == LBMOE_W_BF16) {
    if (get(d, nm.gate_up_tiled) != Py_None || q != Py_None) return false;
    if (g->scalar_type() != kBf16 || !g->is_contiguous()) return false;
    L->shared_gate_proj = g->const_data_ptr();
    L->shared_up_proj = ts.shaped(w[1], kBf16, Is, *H);
    L->shared_down_proj = ts.shaped(w[2], kBf16, *H, Is);
    return L->shared_up_proj && L->shared_down_proj;
  }
  if (*dtype != LBMOE_W_FP8_E4M3 || !ts.add(w[1]) || !ts.add(w[2])) return false;
  if (!q || !PyDict_CheckExact(q) || PyDict_GET_SIZE(q) != 3) return false;
  const void* c[3];
  const float* s[3];
  PyObject* names[3] = {nm.gate, nm.up, nm.down};
  for (int i = 0; i < 3; ++i) {
    PyObject* pair = get(q, names[i]);
    if (!pair || !PyTuple_CheckExact(pair) || PyTuple_GET_SIZE(pair) != 2) return false;
    const at::Tensor *qc = ts.add(PyTuple_GET_ITEM(pair, 0)), *qs = ts.add(PyTuple_GET_ITEM(pair, 1));
    if (!qc || !qs || qs->scalar_type() != kF32) return false;
    c[i] = qc->const_data_ptr();
    s[i] = static_cast<const float*>(qs->const_data_ptr());
  }
  L->shared_gate_proj = c[0], L->shared_up_proj = c[1], L->shared_down_proj = c[2];
  L->shared_gate_scale = s[0], L->shared_up_scale = s[1], L->shared_down_scale = s[2];
  return true;
}

bool fill_block(PyObject* mod, Tensors& ts, lbmoe_layer* L) {
  if (Py_TYPE(mod) != t_block) return false;
  PyObject* d = instance_dict(mod);
  if (!d || !table(d, nm.parameters, 0) || get(d, nm.gate) || get(d, nm.experts)) return false;
  PyObject* se = get(d, nm.shared_expert);
  const bool shared = se == nullptr;                 // else the attribute is None
  if (!shared && (se != Py_None || get(d, nm.shared_expert_gate) != Py_None)) return false;
  if (shared && get(d, nm.shared_expert_gate)) return false;
  PyObject* m = table(d, nm.modules, shared ? 4 : 2);
  if (!m || !fill_router(get(m, nm.gate), ts, L)) return false;
  const int32_t H = L->hidden_size, E = L->num_experts;
  if (!fill_experts(get(m, nm.experts), ts, L)) return false;
  if (L->hidden_size != H || L->num_experts != E) return false;
  if (!shared) return true;
  int64_t Hs, dtype;
  if (!fill_mlp(get(m, nm.shared_expert), ts, L, &Hs, &dtype)) return false;
  if (Hs != H || dtype != L->weight_dtype) return false;
  L->shared_expert_gate = ts.shaped(linear_weight(get(m, nm.shared_expert_gate)), kBf16, 1, H);
  return L->shared_expert_gate != nullptr;
}

at::Tensor empty_bytes(size_t n, c10::Device dev) {
  return at::empty({static_cast<int64_t>(n)}, at::TensorOptions().dtype(at::kByte).device(dev));
}

void* stream_of(c10::Device dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }

void check(int32_t status, const char* what) {
  if (status != LBMOE_OK) {
    char buf[256];
    snprintf(buf, sizeof(buf), "%s failed: %s (status %d)", what, abi.status_string(status), status);
    throw std::runtime_error(buf);
  }
}

// block(module, hidden_states, workspace) or, with residual and norm, forward_norm's call.
PyObject* run_block(PyObject* mod, PyObject* px, PyObject* pres, PyObject* pnorm, PyObject* pws) {
  HANDLE_TH_ERRORS
  if (!abi.forward || !plain_torch()) Py_RETURN_NONE;
  Tensors ts;
  lbmoe_layer L{};
  const at::Tensor* x = ts.add(px, kBf16, 2);
  if (!x || !fill_block(mod, ts, &L) || x->size(1) != L.hidden_size) Py_RETURN_NONE;
  const at::Tensor* res = nullptr;
  const void* norm_w = nullptr;
  float eps = 0.f;
  if (pres) {
    res = ts.add(pres, kBf16, 2);
    if (!res || res->sizes() != x->sizes()) Py_RETURN_NONE;
    THPObjectPtr w(PyObject_GetAttr(pnorm, nm.weight));
    if (!w) { PyErr_Clear(); Py_RETURN_NONE; }
    norm_w = ts.shaped(w.get(), kBf16, x->size(1));
    if (!norm_w) Py_RETURN_NONE;
    THPObjectPtr e(PyObject_GetAttr(pnorm, nm.eps));
    if (!e || !PyFloat_CheckExact(e.get())) { PyErr_Clear(); Py_RETURN_NONE; }
    eps = static_cast<float>(PyFloat_AS_DOUBLE(e.get()));
  }
  at::Tensor ws;
  if (pws != Py_None) {
    const at::Tensor* w = ts.add(pws);
    if (!w || w->scalar_type() != at::kByte || !w->is_contiguous() ||
        (reinterpret_cast<uintptr_t>(w->const_data_ptr()) & 3) != 0)
      Py_RETURN_NONE;
    ws = *w;
  }
  at::Tensor y, res_out;
  {
    pybind11::gil_scoped_release nogil;
    const int64_t T = x->size(0);
    if (!ws.defined()) {
      size_t n = 0;
      check(abi.workspace_size(&L, T, &n), "lbmoe_workspace_size");
      ws = empty_bytes(n, ts.device);
    }
    y = at::empty_like(*x);
    if (res) res_out = at::empty_like(*res);
    const c10::DeviceGuard guard(ts.device);
    if (res)
      check(abi.forward_norm(&L, x->const_data_ptr(), res->const_data_ptr(), norm_w, eps, T,
                             y.mutable_data_ptr(), res_out.mutable_data_ptr(),
                             ws.mutable_data_ptr(), static_cast<size_t>(ws.numel()),
                             stream_of(ts.device)),
            "lbmoe_forward_norm");
    else
      check(abi.forward(&L, x->const_data_ptr(), T, y.mutable_data_ptr(), ws.mutable_data_ptr(),
                        static_cast<size_t>(ws.numel()), stream_of(ts.device)),
            "lbmoe_forward");
  }
  if (!res) return THPVariable_Wrap(std::move(y));
  THPObjectPtr a(THPVariable_Wrap(std::move(y))), b(THPVariable_Wrap(std::move(res_out)));
  if (!a || !b) return nullptr;
  return PyTuple_Pack(2, a.get(), b.get());
  END_HANDLE_TH_ERRORS
}

PyObject* block(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 3) Py_RETURN_NONE;
  return run_block(args[0], args[1], nullptr, nullptr, args[2]);
}

PyObject* block_norm(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 5) Py_RETURN_NONE;
  return run_block(args[0], args[1], args[2], args[3], args[4]);
}

// router(module, hidden_states) -> (weights bf16 [T, k], indices int64 [T, k])
PyObject* router(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !abi.forward || !plain_torch()) Py_RETURN_NONE;
  Tensors ts;
  lbmoe_layer L{};
  const at::Tensor* x = ts.add(args[1], kBf16, 2);
  if (!x || !fill_router(args[0], ts, &L) || x->size(1) != L.hidden_size) Py_RETURN_NONE;
  L.moe_intermediate_size = 256;                     // unused by the router
  at::Tensor w, idx;
  {
    pybind11::gil_scoped_release nogil;
    const int64_t T = x->size(0);
    const auto opt = at::TensorOptions().device(ts.device);
    at::Tensor logits = at::empty({T, L.num_experts}, opt.dtype(kBf16));
    const c10::DeviceGuard guard(ts.device);
    void* stream = stream_of(ts.device);
    check(abi.router_logits(&L, x->const_data_ptr(), T, logits.mutable_data_ptr(), stream),
          "lbmoe_router_logits");
    w = at::empty({T, L.top_k}, opt.dtype(kBf16));
    idx = at::empty({T, L.top_k}, opt.dtype(at::kLong));
    check(abi.route(&L, logits.const_data_ptr(), nullptr, T, idx.mutable_data_ptr(), 8,
                    w.mutable_data_ptr(), nullptr, stream),
          "lbmoe_route");
  }
  THPObjectPtr a(THPVariable_Wrap(std::move(w))), b(THPVariable_Wrap(std::move(idx)));
  if (!a || !b) return nullptr;
  return PyTuple_Pack(2, a.get(), b.get());
  END_HANDLE_TH_ERRORS
}

// experts(module, hidden_states, top_k_indices, top_k_weights)
PyObject* experts(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4 || !abi.forward || !plain_torch()) Py_RETURN_NONE;
  Tensors ts;
  lbmoe_layer L{};
  const at::Tensor* x = ts.add(args[1], kBf16, 2);
  if (!x || !fill_experts(args[0], ts, &L) || x->size(1) != L.hidden_size) Py_RETURN_NONE;
  const at::Tensor* idx = ts.add(args[2]);
  if (!idx || idx->dim() != 2 || !idx->is_contiguous() || idx->size(0) != x->size(0) ||
      idx->size(1) > INT32_MAX ||
      (idx->scalar_type() != at::kLong && idx->scalar_type() != at::kInt))
    Py_RETURN_NONE;
  const at::Tensor* tw = ts.add(args[3], kBf16, 2);
  if (!tw || tw->sizes() != idx->sizes()) Py_RETURN_NONE;
  L.top_k = static_cast<int32_t>(idx->size(1));
  at::Tensor y;
  {
    pybind11::gil_scoped_release nogil;
    const int64_t T = x->size(0);
    y = at::empty_like(*x);
    size_t bytes = 0;
    check(abi.workspace_size(&L, T, &bytes), "lbmoe_workspace_size");
    at::Tensor ws = empty_bytes(bytes, ts.device);
    const c10::DeviceGuard guard(ts.device);
    check(abi.experts(&L, x->const_data_ptr(), idx->const_data_ptr(),
                      static_cast<int32_t>(idx->element_size()), tw->const_data_ptr(), T,
                      y.mutable_data_ptr(), ws.mutable_data_ptr(), bytes, stream_of(ts.device)),
          "lbmoe_experts");
  }
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// mlp(module, x)
PyObject* mlp(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !abi.forward || !plain_torch()) Py_RETURN_NONE;
  Tensors ts;
  lbmoe_layer L{};
  int64_t H, dtype;
  const at::Tensor* x = ts.add(args[1], kBf16, 2);
  if (!x || !fill_mlp(args[0], ts, &L, &H, &dtype) || x->size(1) != H) Py_RETURN_NONE;
  at::Tensor out;
  {
    pybind11::gil_scoped_release nogil;
    const int64_t T = x->size(0);
    const int32_t h = static_cast<int32_t>(H), Is = L.shared_intermediate_size;
    const int32_t dt = static_cast<int32_t>(dtype);
    size_t bytes = 0;
    check(abi.dense_mlp_workspace_size(h, Is, dt, T, &bytes), "lbmoe_dense_mlp_workspace_size");
    at::Tensor ws = empty_bytes(bytes, ts.device);
    out = at::empty_like(*x);
    const c10::DeviceGuard guard(ts.device);
    check(abi.dense_mlp(L.shared_gate_proj, L.shared_up_proj, L.shared_down_proj,
                        L.shared_gate_scale, L.shared_up_scale, L.shared_down_scale, h, Is, dt,
                        x->const_data_ptr(), T, out.mutable_data_ptr(), ws.mutable_data_ptr(),
                        bytes, stream_of(ts.device)),
          "lbmoe_dense_mlp");
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// Whether the modes and transforms in effect leave a call to this extension.
PyObject* plain(PyObject*, PyObject*) {
  HANDLE_TH_ERRORS
  return PyBool_FromLong(plain_torch());
  END_HANDLE_TH_ERRORS
}

// bind(addresses, classes): addresses of the entry points in Abi's order; (router, experts, mlp,
// block, nn.Linear, DeviceContext) classes.
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  constexpr Py_ssize_t kFns = sizeof(Abi) / sizeof(void*);
  PyTypeObject** types[] = {&t_router, &t_experts, &t_mlp, &t_block, &t_linear, &t_device_context};
  constexpr Py_ssize_t kTypes = sizeof(types) / sizeof(*types);
  if (n != 2 || !PyTuple_CheckExact(args[0]) || PyTuple_GET_SIZE(args[0]) != kFns ||
      !PyTuple_CheckExact(args[1]) || PyTuple_GET_SIZE(args[1]) != kTypes) {
    PyErr_SetString(PyExc_TypeError, "bind(entry point addresses, module classes)");
    return nullptr;
  }
  void* fn[kFns];
  for (Py_ssize_t i = 0; i < kFns; ++i) {
    fn[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(args[0], i));
    if (!fn[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point");
      return nullptr;
    }
  }
  for (Py_ssize_t i = 0; i < kTypes; ++i)
    if (!PyType_Check(PyTuple_GET_ITEM(args[1], i))) {
      PyErr_SetString(PyExc_TypeError, "bind: classes expected");
      return nullptr;
    }
  for (Py_ssize_t i = 0; i < kTypes; ++i) {
    PyObject* old = reinterpret_cast<PyObject*>(*types[i]);
    *types[i] = reinterpret_cast<PyTypeObject*>(Py_NewRef(PyTuple_GET_ITEM(args[1], i)));
    Py_XDECREF(old);
  }
  std::memcpy(&abi, fn, sizeof(fn));
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", reinterpret_cast<PyCFunction>(bind), METH_FASTCALL, nullptr},
    {"block", reinterpret_cast<PyCFunction>(block), METH_FASTCALL, nullptr},
    {"block_norm", reinterpret_cast<PyCFunction>(block_norm), METH_FASTCALL, nullptr},
    {"router", reinterpret_cast<PyCFunction>(router), METH_FASTCALL, nullptr},
    {"experts", reinterpret_cast<PyCFunction>(experts), METH_FASTCALL, nullptr},
    {"mlp", reinterpret_cast<PyCFunction>(mlp), METH_FASTCALL, nullptr},
    {"plain", plain, METH_NOARGS, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods,
                          nullptr, nullptr, nullptr, nullptr};

}  // namespace

#define LBMOE_STR1(x) #x
#define LBMOE_STR(x) LBMOE_STR1(x)

PyMODINIT_FUNC PyInit__host(void) {
  PyObject** names[] = {&nm.parameters, &nm.modules, &nm.weight, &nm.bias, &nm.gate, &nm.experts,
                        &nm.shared_expert, &nm.shared_expert_gate, &nm.gate_proj, &nm.up_proj,
                        &nm.down_proj, &nm.gate_up_proj, &nm.top_k, &nm.num_experts,
                        &nm.hidden_size, &nm.intermediate_size, &nm.logit_bias, &nm.weight_dtype,
                        &nm.gate_up_q, &nm.gate_up_scale, &nm.down_q, &nm.down_scale,
                        &nm.gate_up_tiled, &nm.q, &nm.up, &nm.down, &nm.eps};
  const char* text[] = {"_parameters", "_modules", "weight", "bias", "gate", "experts",
                        "shared_expert", "shared_expert_gate", "gate_proj", "up_proj",
                        "down_proj", "gate_up_proj", "top_k", "num_experts",
                        "hidden_size", "intermediate_size", "logit_bias", "weight_dtype",
                        "gate_up_q", "gate_up_scale", "down_q", "down_scale",
                        "gate_up_tiled", "q", "up", "down", "eps"};
  static_assert(sizeof(names) / sizeof(*names) == sizeof(text) / sizeof(*text));
  for (size_t i = 0; i < sizeof(text) / sizeof(*text); ++i) {
    *names[i] = PyUnicode_InternFromString(text[i]);
    if (!*names[i]) return nullptr;
  }
  PyObject* m = PyModule_Create(&module_def);
  // the torch whose headers this was compiled with: _lib.py loads no other
  constexpr const char* kTorch =
      LBMOE_STR(TORCH_VERSION_MAJOR) "." LBMOE_STR(TORCH_VERSION_MINOR);
  if (m && PyModule_AddStringConstant(m, "torch_version", kTorch) < 0) Py_CLEAR(m);
  return m;
}
