// Host side of the layers' generation step (_layer_step.py): what every step does besides launching, natively.
//
// A step is 15 us of launches and 25 us of kernels for one sequence of the 340M geometry; comparing the layer with its plan, checking
// the cache's tensors, allocating the step's tensors and filling the call's structure took another 25 us as Python, and the host was
// what a token waited for: 48 us a token, 33 with this.  Nothing here outlives a call but what make_watch() and make_step() are given:
// names, types, options, addresses and sizes, never a tensor.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros.h>

#include <vector>

#include "../../../include/natsl.h"
#include "layer_core.h"

namespace {

// ---- a layer as its plans saw it -----------------------------------------------------------------------------------------
struct Weight {
  PyTypeObject* type;     // (held by Watch::keep)
  bool none;
  const void* data;
  at::ScalarType dtype;
  bool contiguous;
  std::vector<int64_t> sizes;
};
struct Part {
  PyObject* name;
  PyTypeObject* type;
  std::vector<PyObject*> params, options, values;
};
struct Watch {
  std::vector<PyObject*> keep;   // everything below that is a Python object (names, types, option values)
  std::vector<Part> parts;
  std::vector<PyObject*> own, absent, options, values;
  std::vector<Weight> weights;
  PyObject *modules, *parameters, *forward, *hooks[4];
};

const char* const WATCH = "natsl.watch";
const char* const STEP = "natsl.step";

PyObject* kept(Watch& w, PyObject* o) {
  Py_INCREF(o);
  w.keep.push_back(o);
  return o;
}

std::vector<PyObject*> list_of(Watch& w, PyObject* seq) {
  std::vector<PyObject*> out;
  THPObjectPtr fast(PySequence_Fast(seq, "a sequence"));
  if (!fast) throw python_error();
  for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(fast.get()); ++i) out.push_back(kept(w, PySequence_Fast_GET_ITEM(fast.get(), i)));
  return out;
}

// whether the dict's entries under the names equal the values, entry by entry; false when one is gone
bool options_hold(PyObject* dict, const std::vector<PyObject*>& names, const std::vector<PyObject*>& values) {
  for (size_t i = 0; i < names.size(); ++i) {
    PyObject* have = PyDict_GetItemWithError(dict, names[i]);
    if (!have) {
      if (PyErr_Occurred()) throw python_error();
      return false;
    }
    if (have == values[i]) continue;
    const int eq = PyObject_RichCompareBool(have, values[i], Py_EQ);
    if (eq < 0) throw python_error();
    if (!eq) return false;
  }
  return true;
}

PyObject* entry(PyObject* dict, PyObject* name) {   // borrowed; null when it is not there
  PyObject* o = PyDict_GetItemWithError(dict, name);
  if (!o && PyErr_Occurred()) throw python_error();
  return o;
}

PyObject* dict_of(PyObject* o) {
  PyObject** d = _PyObject_GetDictPtr(o);
  return d && *d && PyDict_Check(*d) ? *d : nullptr;
}

bool weight_holds(const Weight& w, PyObject* o) {
  if (Py_TYPE(o) != w.type) return false;
  if (w.none) return true;
  const at::Tensor& t = THPVariable_Unpack(o);
  return t.data_ptr() == w.data && t.scalar_type() == w.dtype && t.is_contiguous() == w.contiguous && t.sizes() == at::IntArrayRef(w.sizes);
}

void free_watch(PyObject* capsule) {
  auto* w = static_cast<Watch*>(PyCapsule_GetPointer(capsule, WATCH));
  for (PyObject* o : w->keep) Py_DECREF(o);
  delete w;
}

// make_watch(parts, own, absent, option names, option values, weights): parts as (name, type, parameter names, option names, option
// values); weights in the order own parameters, then the parts' parameters
PyObject* make_watch(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *parts, *own, *absent, *options, *values, *weights;
  if (!PyArg_ParseTuple(args, "OOOOOO", &parts, &own, &absent, &options, &values, &weights)) return nullptr;
  auto* w = new Watch;
  THPObjectPtr capsule(PyCapsule_New(w, WATCH, free_watch));
  if (!capsule) {
    delete w;
    return nullptr;
  }
  w->own = list_of(*w, own);
  w->absent = list_of(*w, absent);
  w->options = list_of(*w, options);
  w->values = list_of(*w, values);
  for (PyObject* p : list_of(*w, parts)) {
    PyObject *name, *type, *params, *names, *vals;
    if (!PyArg_ParseTuple(p, "OO!OOO", &name, &PyType_Type, &type, &params, &names, &vals)) return nullptr;
    Part part;
    part.name = kept(*w, name);
    part.type = reinterpret_cast<PyTypeObject*>(kept(*w, type));
    part.params = list_of(*w, params);
    part.options = list_of(*w, names);
    part.values = list_of(*w, vals);
    w->parts.push_back(std::move(part));
  }
  THPObjectPtr fast(PySequence_Fast(weights, "a sequence of weights"));
  if (!fast) return nullptr;
  for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(fast.get()); ++i) {
    PyObject* o = PySequence_Fast_GET_ITEM(fast.get(), i);
    Weight r{};
    r.type = reinterpret_cast<PyTypeObject*>(kept(*w, reinterpret_cast<PyObject*>(Py_TYPE(o))));
    r.none = o == Py_None;
    if (!r.none) {
      if (!THPVariable_Check(o)) {
        PyErr_SetString(PyExc_TypeError, "a weight must be a tensor or None");
        return nullptr;
      }
      const at::Tensor& t = THPVariable_Unpack(o);
      r.data = t.data_ptr();
      r.dtype = t.scalar_type();
      r.contiguous = t.is_contiguous();
      r.sizes = t.sizes().vec();
    }
    w->weights.push_back(std::move(r));
  }
  static const char* const names[7] = {"_modules", "_parameters", "forward", "_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks"};
  PyObject** at[7] = {&w->modules, &w->parameters, &w->forward, &w->hooks[0], &w->hooks[1], &w->hooks[2], &w->hooks[3]};
  for (int i = 0; i < 7; ++i) {
    *at[i] = PyUnicode_InternFromString(names[i]);
    if (!*at[i]) return nullptr;
    w->keep.push_back(*at[i]);
  }
  return capsule.release();
  END_HANDLE_TH_ERRORS
}

// -> 0: something has changed; 1: everything is as it was; 2: it is, and a submodule has a hook or a forward of its own
int watch_holds(const Watch& w, PyObject* layer) {
  PyObject* ld = dict_of(layer);
  PyObject* mods = ld ? entry(ld, w.modules) : nullptr;
  PyObject* own = ld ? entry(ld, w.parameters) : nullptr;
  if (!mods || !own) return 0;
  size_t at = 0;
  bool hooked = false;
  for (PyObject* n : w.own) {
    PyObject* o = entry(own, n);
    if (!o || !weight_holds(w.weights[at++], o)) return 0;
  }
  for (const Part& p : w.parts) {
    PyObject* m = entry(mods, p.name);
    if (!m || Py_TYPE(m) != p.type) return 0;
    PyObject* d = dict_of(m);
    PyObject* params = d ? entry(d, w.parameters) : nullptr;
    if (!params) return 0;
    for (PyObject* n : p.params) {
      PyObject* o = entry(params, n);
      if (!o || !weight_holds(w.weights[at++], o)) return 0;
    }
    for (PyObject* n : w.hooks) {
      PyObject* h = entry(d, n);
      if (!h) return 0;
      const int any = PyObject_IsTrue(h);
      if (any < 0) throw python_error();
      hooked |= any != 0;
    }
    hooked |= entry(d, w.forward) != nullptr;
    if (!options_hold(d, p.options, p.values)) return 0;
  }
  if (!options_hold(ld, w.options, w.values)) return 0;
  for (PyObject* n : w.absent) {
    PyObject* m = entry(mods, n);
    if (m && m != Py_None) return 0;
  }
  return hooked ? 2 : 1;
}

PyObject* holds(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2) {
    PyErr_SetString(PyExc_TypeError, "holds(watch, layer)");
    return nullptr;
  }
  auto* w = static_cast<Watch*>(PyCapsule_GetPointer(args[0], WATCH));
  if (!w) return nullptr;
  return PyLong_FromLong(watch_holds(*w, args[1]));
  END_HANDLE_TH_ERRORS
}

// ---- the step ----------------------------------------------------------------------------------------------------------
struct Step {
  natsl_layer_step fixed;
  decltype(&natsl_layer_step_sync_fwd) fwd;
  decltype(&natsl_layer_step_sync_bytes) sync_bytes;
  unsigned long long max_wait_us;
  decltype(&natsl_layer_step_workspace_bytes) workspace_bytes;
  int device;
};

void free_step(PyObject* capsule) { delete static_cast<Step*>(PyCapsule_GetPointer(capsule, STEP)); }

// make_step(address of the structure with everything that stays the same, its size, addresses of the three entry points, the longest wait, device index)
PyObject* make_step(PyObject*, PyObject* args) {
  unsigned long long fixed, size, fwd, bytes, sync_bytes, max_wait_us;
  int device;
  if (!PyArg_ParseTuple(args, "KKKKKKi", &fixed, &size, &fwd, &bytes, &sync_bytes, &max_wait_us, &device)) return nullptr;
  if (size != sizeof(natsl_layer_step)) {
    PyErr_SetString(PyExc_ValueError, "the step's structure has another size than the library's");
    return nullptr;
  }
  auto* s = new Step;
  s->fixed = *reinterpret_cast<const natsl_layer_step*>(fixed);
  s->fwd = reinterpret_cast<decltype(s->fwd)>(fwd);
  s->workspace_bytes = reinterpret_cast<decltype(s->workspace_bytes)>(bytes);
  s->sync_bytes = reinterpret_cast<decltype(s->sync_bytes)>(sync_bytes);
  s->max_wait_us = max_wait_us;
  s->device = device;
  PyObject* capsule = PyCapsule_New(s, STEP, free_step);
  if (!capsule) delete s;
  return capsule;
}

// the cache's tensors, in the order the calls below take them
struct CacheTensors {
  at::Tensor conv[3], state, l_k, l_v, l_g, hidden, beta, k, v, valid, start, g_sum;
};
constexpr int CACHE_ARGS = 12;   // conv states, state, l_k, l_v, l_g, hidden, beta, k, v, valid, block start, g sum

bool fits(const at::Tensor& t, const int device, const at::ScalarType dtype, const at::IntArrayRef sizes) {
  return t.scalar_type() == dtype && t.sizes() == sizes && t.is_contiguous() && t.get_device() == device;
}

// Whether the cache's tensors have the types, shapes and layouts that the kernels read and write (a cache filled under autocast or by
// other code can hold others: the layers' general path converts).
bool take_cache(const Step& step, const int64_t B, PyObject* const* a, CacheTensors& c) {
  const natsl_layer_step& f = step.fixed;
  THPObjectPtr conv(PySequence_Fast(a[0], "the convolution states"));
  if (!conv) {
    PyErr_Clear();
    return false;
  }
  if (PySequence_Fast_GET_SIZE(conv.get()) != 3) return false;
  auto take = [](PyObject* o, at::Tensor& t) {
    if (!THPVariable_Check(o)) return false;
    t = THPVariable_Unpack(o);
    return true;
  };
  for (int i = 0; i < 3; ++i)
    if (!take(PySequence_Fast_GET_ITEM(conv.get(), i), c.conv[i])) return false;
  if (!take(a[1], c.state) || !take(a[2], c.l_k) || !take(a[3], c.l_v) || !take(a[4], c.l_g) || !take(a[5], c.hidden) ||
      (f.is_delta && !take(a[6], c.beta)) || !take(a[7], c.k) || !take(a[8], c.v) || !take(a[9], c.valid))
    return false;
  if (!f.is_delta) take(a[6], c.beta);
  if (a[10] != Py_None && !take(a[10], c.start)) return false;
  if (a[11] != Py_None && !take(a[11], c.g_sum)) return false;
  const int64_t H = f.H, K = f.K, V = f.V, W = f.conv_width, bs = f.block, HQ = f.HQ;
  if (c.k.dim() != 4) return false;
  const int64_t cap = c.k.size(1);
  const auto bf16 = at::kBFloat16, f32 = at::kFloat;
  const int d = step.device;
  return fits(c.conv[0], d, bf16, {B, H * K, W}) && fits(c.conv[1], d, bf16, {B, H * K, W}) && fits(c.conv[2], d, bf16, {B, H * V, W}) &&
         fits(c.state, d, f32, {B, H, K, V}) && fits(c.l_k, d, bf16, {B, bs, H, K}) && fits(c.l_v, d, bf16, {B, bs, H, V}) &&
         fits(c.l_g, d, f32, {B, bs, H}) && fits(c.hidden, d, bf16, {B, bs, f.D}) && (!f.is_delta || fits(c.beta, d, bf16, {B, bs, H})) &&
         fits(c.k, d, bf16, {B, cap, HQ, H * K / HQ}) && fits(c.v, d, bf16, {B, cap, HQ, H * V / HQ}) &&
         fits(c.valid, d, at::kBool, {B, cap / bs, f.HN}) && cap % bs == 0 && (!c.start.defined() || fits(c.start, d, f32, {B, H, K, V})) &&
         (!c.g_sum.defined() || (c.g_sum.numel() == B * H && c.g_sum.get_device() == d));
}

// takes(step, B, the cache's tensors ...) -> bool
PyObject* takes(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 + CACHE_ARGS) {
    PyErr_SetString(PyExc_TypeError, "takes(step, B, the cache's tensors ...)");
    return nullptr;
  }
  auto* step = static_cast<Step*>(PyCapsule_GetPointer(args[0], STEP));
  if (!step) return nullptr;
  CacheTensors c;
  const int64_t B = PyLong_AsLongLong(args[1]);
  return PyBool_FromLong(take_cache(*step, B, args + 2, c));
  END_HANDLE_TH_ERRORS
}

// run(step, x, n_in, n_kept, stream, types or None, their code, the cache's tensors ..., what its steps in one launch share or None)
// -> None: the cache's tensors do not fit; a number: the entry point's error; else (out, state, block start, conv states, g sum, what they share)
PyObject* run(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 8 + CACHE_ARGS || !THPVariable_Check(args[1])) {
    PyErr_SetString(PyExc_TypeError, "run(step, x, n_in, n_kept, stream, types, types' code, the cache's tensors ..., shared)");
    return nullptr;
  }
  auto* step = static_cast<Step*>(PyCapsule_GetPointer(args[0], STEP));
  if (!step) return nullptr;
  const at::Tensor x = THPVariable_Unpack(args[1]).contiguous();
  const int64_t B = x.size(0), T = x.size(1);
  const long n_in = PyLong_AsLong(args[2]), n_kept = PyLong_AsLong(args[3]), code = PyLong_AsLong(args[6]);
  const natsl_stream_t stream = static_cast<natsl_stream_t>(PyLong_AsVoidPtr(args[4]));
  if (PyErr_Occurred()) return nullptr;
  CacheTensors c;
  if (!take_cache(*step, B, args + 7, c)) Py_RETURN_NONE;
  at::Tensor types;
  if (args[5] != Py_None) types = THPVariable_Unpack(args[5]);

  natsl_layer_step s = step->fixed;
  s.B = (int32_t)B;
  s.T = (int32_t)T;
  s.n_in = (int32_t)n_in;
  s.n_kept = (int32_t)n_kept;
  s.cache_tokens = (int32_t)c.k.size(1);
  const auto f32 = c.state.options(), bf16 = x.options();
  at::Tensor conv_out[3];
  for (int i = 0; i < 3; ++i) conv_out[i] = at::empty(c.conv[i].sizes(), bf16);
  at::Tensor state_out = at::empty(c.state.sizes(), f32);
  if (!c.start.defined()) {
    c.start = at::empty(c.state.sizes(), f32);
    s.flags |= NATSL_STEP_FRESH_START;
  }
  if (c.g_sum.defined() && (c.g_sum.scalar_type() != at::kFloat || !c.g_sum.is_contiguous())) c.g_sum = c.g_sum.to(at::kFloat).contiguous();
  at::Tensor g_out = at::empty({B, 1, s.H}, f32);
  at::Tensor out = at::empty({B, T, s.D}, bf16);
  s.x = x.data_ptr();
  s.out = out.data_ptr();
  s.state = static_cast<const float*>(c.state.data_ptr());
  s.state_out = static_cast<float*>(state_out.data_ptr());
  s.block_start = static_cast<float*>(c.start.data_ptr());
  s.conv_state_q = c.conv[0].data_ptr();
  s.conv_state_k = c.conv[1].data_ptr();
  s.conv_state_v = c.conv[2].data_ptr();
  s.conv_out_q = conv_out[0].data_ptr();
  s.conv_out_k = conv_out[1].data_ptr();
  s.conv_out_v = conv_out[2].data_ptr();
  s.g_cumsum = c.g_sum.defined() ? static_cast<const float*>(c.g_sum.data_ptr()) : nullptr;
  s.g_cumsum_out = static_cast<float*>(g_out.data_ptr());
  s.cache_k = c.k.data_ptr();
  s.cache_v = c.v.data_ptr();
  s.cache_valid = static_cast<uint8_t*>(c.valid.data_ptr());
  s.block_k = c.l_k.data_ptr();
  s.block_v = c.l_v.data_ptr();
  s.block_g = static_cast<float*>(c.l_g.data_ptr());
  if (c.beta.defined()) s.block_beta = c.beta.data_ptr();
  if (types.defined()) {
    s.types = types.data_ptr();
    s.types_dtype = (int32_t)code;
  } else {
    s.block_hidden = c.hidden.data_ptr();
  }
  const size_t bytes = step->workspace_bytes(&s);
  at::Tensor ws = at::empty({(int64_t)bytes}, f32.dtype(at::kByte));
  void* const ws_ptr = ws.data_ptr();
  // What the parts of a step in one launch meet on belongs to the cache, whose steps follow one another; it holds something from step to step and
  // is made anew for another number of sequences, but for the word that says that a step has failed.  Steps of several launches look at that, too.
  const size_t shared_bytes = step->sync_bytes(&s);
  at::Tensor shared;
  if (args[7 + CACHE_ARGS] != Py_None && THPVariable_Check(args[7 + CACHE_ARGS])) shared = THPVariable_Unpack(args[7 + CACHE_ARGS]);
  if (shared.defined() && (shared.get_device() != step->device || !shared.is_contiguous() || shared.scalar_type() != at::kInt)) shared = at::Tensor();
  if (shared_bytes && (!shared.defined() || shared.nbytes() != shared_bytes)) {
    const at::Tensor before = shared;
    shared = at::zeros({(int64_t)(shared_bytes / 4)}, f32.dtype(at::kInt));
    if (before.defined()) shared.narrow(0, NATSL_STEP_SYNC_FAILED, 1).copy_(before.narrow(0, NATSL_STEP_SYNC_FAILED, 1));
  }
  const size_t given = shared.defined() ? shared.nbytes() : 0;
  void* const shared_ptr = given ? shared.data_ptr() : nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = step->fwd(&s, ws_ptr, bytes, shared_ptr, given, step->max_wait_us, stream);
  Py_END_ALLOW_THREADS
  if (rc) return PyLong_FromLong(rc);
  THPObjectPtr conv(PyTuple_New(3));
  if (!conv) return nullptr;
  for (int i = 0; i < 3; ++i) {
    PyObject* t = THPVariable_Wrap(conv_out[i]);
    if (!t) return nullptr;
    PyTuple_SET_ITEM(conv.get(), i, t);
  }
  THPObjectPtr o(THPVariable_Wrap(out)), so(THPVariable_Wrap(state_out)), st(THPVariable_Wrap(c.start)), g(THPVariable_Wrap(g_out)), kept(shared.defined() ? THPVariable_Wrap(shared) : Py_NewRef(Py_None));
  if (!o || !so || !st || !g || !kept) return nullptr;
  return PyTuple_Pack(6, o.get(), so.get(), st.get(), conv.get(), g.get(), kept.get());
  END_HANDLE_TH_ERRORS
}

template <class F>
PyCFunction fast(F f) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)); }

PyMethodDef methods[] = {
    {"make_watch", make_watch, METH_VARARGS, nullptr},
    {"holds", fast(holds), METH_FASTCALL, nullptr},
    {"make_step", make_step, METH_VARARGS, nullptr},
    {"takes", fast(takes), METH_FASTCALL, nullptr},
    {"run", fast(run), METH_FASTCALL, nullptr},
    {"make_layer", natsl_make_layer, METH_VARARGS, nullptr},
    {"layer_train", fast(natsl_layer_train), METH_FASTCALL, nullptr},
    {"layer_backward", fast(natsl_layer_backward), METH_FASTCALL, nullptr},
    {"layer_front", fast(natsl_layer_prompt_front), METH_FASTCALL, nullptr},
    {"layer_rest", fast(natsl_layer_prompt_rest), METH_FASTCALL, nullptr},
    {"make_entries", natsl_make_entries, METH_VARARGS, nullptr},
    {"mixed_plain", fast(natsl_mixed_plain), METH_FASTCALL, nullptr},
    {"hard_select", fast(natsl_hard_select_plain), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_step_core", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__step_core() { return PyModule_Create(&module); }
