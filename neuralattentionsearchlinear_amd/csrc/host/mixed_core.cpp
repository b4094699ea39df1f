// Host side of the mixed operators' forward and of the selector's hard choice (_mixed_common.py, nats_util.py) for calls that need nothing out of the
// ordinary: no gradient, no packed sequences, tensors of the types and shapes that go together.  What a call does besides launching took twice as
// long as its launches when it was Python: the host has 42 us with B1 T256 H4 128/128 and 57 with fp32 B1 T256 H2 64/64, 25 and 30 with this, and the call then
// takes what its kernels take: 32 and 33 (the second 27 since the routing launch is gone and the branches' first kernels are one).  Everything else is
// declined (None) and runs, or is refused, there.  Nothing outlives a call.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <ATen/ATen.h>
#include <c10/core/GradMode.h>

#include <dlfcn.h>

#include "../../../include/natsl.h"
#include "layer_core.h"

namespace {

using T = at::Tensor;

struct Entries {
  decltype(&natsl_mixed_fwd) mixed_fwd;
  decltype(&natsl_mixed_workspace_bytes) workspace_bytes;
  decltype(&natsl_hard_select) hard_select;
};
const char* const ENTRIES = "natsl.entries";

const Entries* entries_of(PyObject* o) { return static_cast<const Entries*>(PyCapsule_GetPointer(o, ENTRIES)); }

// A plain tensor on a GPU, of a type that the kernels take or convert, with no interpreter or transform behind it
bool take(PyObject* o, T& t, const int64_t dims) {
  if (!THPVariable_CheckExact(o)) return false;
  t = THPVariable_Unpack(o);
  static const c10::DispatchKeySet others({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched,
                                           c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize, c10::DispatchKey::BatchedNestedTensor,
                                           c10::DispatchKey::Conjugate, c10::DispatchKey::Negative});
  return !t.key_set().has_any(others) && t.is_cuda() && t.layout() == at::kStrided && t.dim() == dims && t.numel() > 0 &&
         (t.scalar_type() == at::kBFloat16 || t.scalar_type() == at::kFloat);
}
bool sized(const T& t, const at::IntArrayRef sizes, const T& like) { return t.sizes() == sizes && t.device() == like.device(); }
int32_t code(const T& t) { return t.scalar_type() == at::kFloat ? NATSL_F32 : NATSL_BF16; }

// A call's own memory: places in one allocation
struct Scratch {
  size_t total = 0;
  size_t place(const size_t bytes) {
    const size_t at = total;
    total += (bytes + 255) / 256 * 256;
    return at;
  }
};

struct Conversion { const void* src; at::IntArrayRef sizes; size_t at; };

}  // namespace

// make_entries(the library's handle)
PyObject* natsl_make_entries(PyObject*, PyObject* args) {
  unsigned long long handle;
  if (!PyArg_ParseTuple(args, "K", &handle)) return nullptr;
  void* const lib = reinterpret_cast<void*>(handle);
  Entries e{reinterpret_cast<decltype(e.mixed_fwd)>(dlsym(lib, "natsl_mixed_fwd")),
            reinterpret_cast<decltype(e.workspace_bytes)>(dlsym(lib, "natsl_mixed_workspace_bytes")),
            reinterpret_cast<decltype(e.hard_select)>(dlsym(lib, "natsl_hard_select"))};
  if (!e.mixed_fwd || !e.workspace_bytes || !e.hard_select) {
    PyErr_SetString(PyExc_RuntimeError, "the library does not export what the operators call");
    return nullptr;
  }
  auto* own = new Entries(e);
  PyObject* capsule = PyCapsule_New(own, ENTRIES, [](PyObject* c) { delete static_cast<Entries*>(PyCapsule_GetPointer(c, ENTRIES)); });
  if (!capsule) delete own;
  return capsule;
}

// mixed_plain(entries, options, block, scale_attn, scale_linear, stream, the softmax branch's stream, q, k, v of the softmax branch, q, k, v of the
// linear branch, initial state or None, g, beta or None, types); options: 1 the delta rule, 2 decay, 4 l2 norm, 8 intra, 16 own block, 32 final state
// -> None: not a plain call; a number: the entry point's error; else (o_linear, o_attn, final state or None)
PyObject* natsl_mixed_plain(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 17) {
    PyErr_SetString(PyExc_TypeError, "mixed_plain: 17 arguments");
    return nullptr;
  }
  const Entries* e = entries_of(a[0]);
  if (!e) return nullptr;
  const long options = PyLong_AsLong(a[1]), block = PyLong_AsLong(a[2]);
  const double scale_attn = PyFloat_AsDouble(a[3]), scale_linear = PyFloat_AsDouble(a[4]);
  const natsl_stream_t stream = static_cast<natsl_stream_t>(PyLong_AsVoidPtr(a[5])), side = static_cast<natsl_stream_t>(PyLong_AsVoidPtr(a[6]));
  if (PyErr_Occurred()) return nullptr;
  const bool delta = options & 1;
  T t[7], h0, g, types;                                   // q, k, v twice and beta
  for (int i = 0; i < 6; ++i)
    if (!take(a[7 + i], t[i], 4)) Py_RETURN_NONE;
  if (!take(a[14], g, 3) || (delta ? !take(a[15], t[6], 3) : a[15] != Py_None) || !take(a[16], types, 4)) Py_RETURN_NONE;
  const int64_t B = t[3].size(0), Tn = t[3].size(1), H = t[3].size(2), K = t[3].size(3), V = t[5].size(3);
  const int64_t HQ = t[0].size(2), KA = t[0].size(3), HKV = t[1].size(2), VA = t[2].size(3), TN = types.size(1), HN = types.size(2);
  if (a[13] != Py_None && (!take(a[13], h0, 4) || h0.scalar_type() != at::kFloat || !sized(h0, {B, H, K, V}, t[3]))) Py_RETURN_NONE;
  if (block < 64 || block % 64 || TN != (Tn + block - 1) / block || B * Tn > 0x7fffffff || !sized(t[0], {B, Tn, HQ, KA}, t[3]) || !sized(t[1], {B, Tn, HKV, KA}, t[3]) ||
      !sized(t[2], {B, Tn, HKV, VA}, t[3]) || !sized(t[4], {B, Tn, H, K}, t[3]) || !sized(t[5], {B, Tn, H, V}, t[3]) || !sized(g, {B, Tn, H}, t[3]) ||
      (delta && !sized(t[6], {B, Tn, H}, t[3])) || !sized(types, {B, TN, HN, 2}, t[3]))
    Py_RETURN_NONE;
  c10::NoGradGuard no_grad;
  const auto io = t[3].options().requires_grad(false), f32 = io.dtype(at::kFloat), bf16 = io.dtype(at::kBFloat16);
  natsl_mixed m{};
  Scratch scratch;
  Conversion made[NATSL_MIXED_CASTS];
  const void** const field[7] = {&m.q_attn, &m.k_attn, &m.v_attn, &m.q, &m.k, &m.v, &m.beta};
  int from[7];                                            // which conversion a tensor comes from, -1: none
  for (int i = 0; i < 7; ++i) {
    from[i] = -1;
    if (!t[i].defined()) continue;
    if (t[i].scalar_type() == at::kFloat) {
      t[i] = t[i].contiguous();
      const void* src = t[i].data_ptr();
      if (!(reinterpret_cast<uintptr_t>(src) & 15)) {
        int j = 0;
        while (j < m.n_cast_in && !(made[j].src == src && made[j].sizes == t[i].sizes())) ++j;
        if (j == m.n_cast_in) {
          made[j] = {src, t[i].sizes(), scratch.place((size_t)t[i].numel() * 2)};
          m.cast_in[j].src = src;
          m.cast_in[j].n = t[i].numel();
          ++m.n_cast_in;
        }
        from[i] = j;
        continue;
      }
      t[i] = t[i].to(at::kBFloat16);
    }
    t[i] = t[i].contiguous();
    *field[i] = t[i].data_ptr();
  }
  g = g.to(at::kFloat).contiguous();
  types = types.contiguous();
  if (h0.defined()) h0 = h0.contiguous();
  const int64_t chunks = B * ((Tn + 63) / 64);
  const size_t ws_bytes = e->workspace_bytes(chunks, (int)H);
  const size_t idx = scratch.place((size_t)(B * TN * HN * 2) * 4), nblk = scratch.place((size_t)(B * HN * 2) * 4), lse = scratch.place((size_t)(B * Tn * HQ) * 4),
               ws = scratch.place(ws_bytes);
  const T o_attn = at::empty({B, Tn, HQ, VA}, io), o_lin = at::empty({B, Tn, H, V}, io);
  const bool wide = io.dtype() == at::kFloat;
  size_t out[2] = {0, 0};
  if (wide) {
    out[0] = scratch.place((size_t)o_attn.numel() * 2);
    out[1] = scratch.place((size_t)o_lin.numel() * 2);
  }
  T ht;
  if (options & 32) ht = at::empty({B, H, K, V}, f32);
  const T memory = at::empty({(int64_t)scratch.total}, io.dtype(at::kByte));
  char* const base = static_cast<char*>(memory.data_ptr());
  for (int j = 0; j < m.n_cast_in; ++j) m.cast_in[j].dst = base + made[j].at;
  for (int i = 0; i < 7; ++i)
    if (from[i] >= 0) *field[i] = base + made[from[i]].at;
  m.o_attn = o_attn.data_ptr();
  m.o = o_lin.data_ptr();
  if (wide) {
    void** const to[2] = {&m.o_attn, &m.o};
    const T* const last[2] = {&o_attn, &o_lin};
    for (int i = 0; i < 2; ++i) {
      m.cast_out[i].src = base + out[i];
      m.cast_out[i].dst = last[i]->data_ptr();
      m.cast_out[i].n = last[i]->numel();
      *to[i] = base + out[i];
    }
    m.n_cast_out = 2;
  }
  m.is_delta = delta;
  m.private_tables = 1;
  m.B = (int32_t)B; m.T = m.T_attn = (int32_t)Tn; m.H = (int32_t)H; m.HN = (int32_t)HN; m.K = (int32_t)K; m.V = (int32_t)V; m.TN = m.TN_attn = (int32_t)TN;
  m.block = (int32_t)block; m.HQ = (int32_t)HQ; m.HKV = (int32_t)HKV; m.KA = (int32_t)KA; m.VA = (int32_t)VA;
  m.flags = (options & 2 ? NATSL_DECAY_NON_LINEAR : 0) | (options & 4 ? NATSL_QK_L2NORM : 0) | (options & 8 ? NATSL_INTRA_CHUNK : 0);
  m.same_block_visible = (options & 16) != 0;
  m.types_dtype = code(types);
  m.scale_attn = (float)scale_attn;
  m.scale_linear = (float)scale_linear;
  m.types = m.types_attn = types.data_ptr();
  m.g = static_cast<const float*>(g.data_ptr());
  m.h0 = h0.defined() ? static_cast<const float*>(h0.data_ptr()) : nullptr;
  m.ht = ht.defined() ? static_cast<float*>(ht.data_ptr()) : nullptr;
  m.block_indices = reinterpret_cast<int32_t*>(base + idx);
  m.n_blocks = reinterpret_cast<int32_t*>(base + nblk);
  m.lse = reinterpret_cast<float*>(base + lse);
  m.workspace = base + ws;
  m.workspace_bytes = ws_bytes;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = e->mixed_fwd(&m, NATSL_MIXED_CONVERT | NATSL_MIXED_ROUTE | NATSL_MIXED_SOFTMAX | NATSL_MIXED_LINEAR | NATSL_MIXED_JOIN, stream, side);
  Py_END_ALLOW_THREADS
  if (rc) return PyLong_FromLong(rc);
  THPObjectPtr ol(THPVariable_Wrap(o_lin)), oa(THPVariable_Wrap(o_attn)), state(ht.defined() ? THPVariable_Wrap(ht) : Py_NewRef(Py_None));
  if (!ol || !oa || !state) return nullptr;
  return PyTuple_Pack(3, ol.get(), oa.get(), state.get());
  END_HANDLE_TH_ERRORS
}

// hard_select(entries, logits, whether the last block is forced, stream) -> None: not a plain call; a number: the entry point's error; else
// (types, n_nats_blocks)
PyObject* natsl_hard_select_plain(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4) {
    PyErr_SetString(PyExc_TypeError, "hard_select: 4 arguments");
    return nullptr;
  }
  const Entries* e = entries_of(a[0]);
  if (!e) return nullptr;
  T logits;
  if (!take(a[1], logits, 4) || logits.size(3) != 2) Py_RETURN_NONE;
  const int force = PyObject_IsTrue(a[2]);
  const natsl_stream_t stream = static_cast<natsl_stream_t>(PyLong_AsVoidPtr(a[3]));
  if (PyErr_Occurred()) return nullptr;
  c10::NoGradGuard no_grad;
  logits = logits.contiguous();
  const auto options = logits.options().requires_grad(false);
  const T types = at::empty(logits.sizes(), options), counts = at::empty({logits.size(0), logits.size(2), 2}, options.dtype(at::kInt));
  const int rc = e->hard_select(logits.data_ptr(), types.data_ptr(), static_cast<int32_t*>(counts.data_ptr()), (int)logits.size(0), (int)logits.size(1),
                                (int)logits.size(2), code(logits), force, nullptr, 0, 0, stream);
  if (rc) return PyLong_FromLong(rc);
  THPObjectPtr ty(THPVariable_Wrap(types)), nb(THPVariable_Wrap(counts));
  if (!ty || !nb) return nullptr;
  return PyTuple_Pack(2, ty.get(), nb.get());
  END_HANDLE_TH_ERRORS
}
