// Host side of a whole layer's forward and backward (_front.py): the layers' fast path as one call each way, natively.
//
// A training step of a layer is some 45 launches; as Python (seven autograd functions, forty allocations and as many ctypes calls each way) its
// host time was what small steps took: 760M geometry 1 x 256 tokens 1021 us, 635 with this, a Mamba layer 1 x 256 1057 and 603; a prompt of 777
// tokens 380 and 193, about its kernels' time.
// What is launched, and in which order, is what _front.py and _mixed_common.py describe.  Nothing here outlives a call but what make_layer()
// is given: names of entry points, options and sizes, never a tensor.
#include <algorithm>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <ATen/ATen.h>
#include <c10/core/GradMode.h>

#include <dlfcn.h>

#include <string>
#include <vector>

#include "../../../include/natsl.h"
#include "layer_core.h"

namespace {

#define NATSL_ENTRIES(X)                                                                                                                   \
  X(layer_front) X(project) X(project_bwd) X(layer_select) X(conv_norm_fwd) X(conv_norm_bwd) X(conv_norm_bwd_workspace_bytes) \
  X(mixed_fwd) X(mixed_workspace_bytes) X(norm_gate_logits_fwd) X(norm_gate_logits_bwd) X(norm_gate_bwd_workspace_bytes) X(wgrad)           \
  X(wgrad_workspace_bytes) X(narrow_linear_bwd) X(narrow_wgrad) X(narrow_wgrad_workspace_bytes) X(narrow_wgrad_split) X(gates_bwd) X(gates_bwd_workspace_bytes) X(dx_init) X(softmax_sparse_bwd)  \
  X(softmax_bwd_workspace_bytes) X(linear_workspace_bytes) X(linear_chunk_states) X(linear_chunk_bwd_steps)            \
  X(block_grads_logits) X(order_streams) X(narrow_fwd_pays) X(narrow_linear_bwd_pays) X(narrow_wgrad_pays) X(project_bwd_takes)

struct Layer {
#define X(n) decltype(&natsl_##n) n;
  NATSL_ENTRIES(X)
#undef X
  PyObject* check;             // raises for an entry point's code
  int device, delta, D, H, K, V, HQ, KA, VA, HN, NL, W, act, norm_width, norm_dtype, gate_dtype, out_dtype, neg, decay, same_block, intra;
  float front_eps, out_eps, scale_attn, scale_linear;
};

const char* const LAYER = "natsl.layer";

enum Weight { WQ, WK, WV, WG, WA, WB, W_MIX, WO, CONV_WQ, CONV_WK, CONV_WV, CONV_BQ, CONV_BK, CONV_BV, NORM_Q, NORM_K, A_LOG, DT_BIAS, OUT_NORM1, OUT_NORM2, WN, WEIGHTS };

typedef at::Tensor T;
typedef std::vector<T> Ts;

// Which parts of the backward run for gradients of x and of the weights (in that order): what nobody wants is neither computed nor kept for, as in
// a graph of one node for each (340M geometry, 8 x 4096 tokens, only o_proj trains: 2711 -> 1164 us a step).
struct Needs {
  std::vector<bool> of;        // empty: nothing
  bool conv, gates, op, tail;  // convolutions, gates, operator (conv and gates are in front of it), norm-gate (the operator is in front of it)
  Needs(const std::vector<bool>& need, const bool delta) : of(need) {
    auto any = [&](std::initializer_list<Weight> ws) { return std::any_of(ws.begin(), ws.end(), [&](const Weight w) { return want(w); }); };
    gates = x() || any({WA, WB, A_LOG, DT_BIAS});
    conv = x() || any({WQ, WK, WV, CONV_WQ, CONV_WK, CONV_WV, CONV_BQ, CONV_BK, CONV_BV, NORM_Q, NORM_K}) || (!delta && any({WA, DT_BIAS}));
    op = conv || gates || want(WN);
    tail = op || any({W_MIX, WG, OUT_NORM1, OUT_NORM2});
  }
  bool x() const { return !of.empty() && of[0]; }
  bool want(const Weight w) const { return !of.empty() && of[1 + w]; }
};

struct Failed {                // an entry point's code
  int rc;
  const char* what;
};
void must(const int rc, const char* what) {
  if (rc) throw Failed{rc, what};
}

void* at_(const T& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* f_(const T& t) { return t.defined() ? static_cast<float*>(t.data_ptr()) : nullptr; }
int32_t* i_(const T& t) { return t.defined() ? static_cast<int32_t*>(t.data_ptr()) : nullptr; }
// Tensors that nothing reads any more: what a call allocates next may take their memory (a step at the 340M geometry, 8 x 4096 tokens, has a peak
// of 1.8 GB so, and of 2.2 GB where all live to its end).  What the side stream works on is dropped behind its join.
template <class... Dropped>
void drop(Dropped&... t) { (t.reset(), ...); }
T like(const T& t) { return at::empty(t.sizes(), t.options()); }
int64_t up(const int64_t n, const int64_t m) { return (n + m - 1) / m * m; }
int64_t blocks_of(const int64_t t) { return (t + 63) / 64; }
bool on16(const T& t) { return !(reinterpret_cast<uintptr_t>(t.data_ptr()) & 15); }

// one call's surroundings
struct Call {
  const Layer& l;
  const T x;
  const Ts& w;
  natsl_stream_t stream;
  natsl_stream_t side;         // the softmax branch's stream, or `stream`
  int64_t B, T_, rows;
  at::TensorOptions bf16, f32, i32, u8;

  Call(const Layer& layer, const T& input, const Ts& weights, natsl_stream_t s, natsl_stream_t beside)
      : l(layer), x(input), w(weights), stream(s), side(beside), B(input.size(0)), T_(input.size(1)), rows(B * T_), bf16(input.options()),
        f32(bf16.dtype(at::kFloat)), i32(bf16.dtype(at::kInt)), u8(bf16.dtype(at::kByte)) {}
  T sized(const int64_t columns) const { return at::empty({B, T_, columns}, bf16); }
  T bytes(const size_t n) const { return at::empty({(int64_t)n}, u8); }
};

// ---- forward ----------------------------------------------------------------------------------------------------------------
struct Front {
  T g, beta, dt, logits, ab, wab, pooled, types, raw, counts, fraction;
};

Front front(const Call& c, const Needs& needs, const bool want_raw) {
  const Layer& l = c.l;
  Front o;
  natsl_front a{};
  const int64_t nb = blocks_of(c.T_);
  o.g = at::empty({c.B, c.T_, l.H}, c.f32);
  if (l.delta) o.beta = at::empty({c.B, c.T_, l.H}, c.bf16);
  else o.dt = like(o.g);
  o.logits = at::empty({c.B, nb, l.HN, 2}, c.bf16);
  a.NA = l.H; a.NB = l.delta ? l.H : 0; a.NL = l.NL;
  const int32_t ld = (int32_t)up(a.NA + a.NB, 32);
  if (needs.want(WN)) o.pooled = at::empty({c.B * nb, l.D}, c.bf16);
  if (needs.gates) o.ab = c.sized(a.ld = ld);
  if (needs.x()) o.wab = at::empty({a.wab_rows = ld, l.D}, c.bf16);
  a.x = at_(c.x); a.wa = at_(c.w[WA]); a.wb = l.delta ? at_(c.w[WB]) : nullptr; a.wn = at_(c.w[WN]); a.a_log = at_(c.w[A_LOG]); a.dt_bias = at_(c.w[DT_BIAS]);
  a.ab = at_(o.ab); a.pooled = at_(o.pooled); a.logits = at_(o.logits); a.beta = at_(o.beta); a.wab = at_(o.wab); a.g = f_(o.g); a.dt = f_(o.dt);
  a.B = (int32_t)c.B; a.T = (int32_t)c.T_; a.D = l.D; a.neg_eigval = l.neg; a.param_dtype = l.gate_dtype;
  must(l.layer_front(&a, c.stream), "natsl_layer_front");
  o.types = like(o.logits);
  if (want_raw) o.raw = like(o.logits);
  o.counts = at::empty({c.B, l.HN, 2}, c.i32);
  o.fraction = at::empty({l.HN}, c.f32);
  must(l.layer_select(at_(o.logits), at_(o.types), at_(o.raw), i_(o.counts), f_(o.fraction), (int)c.B, (int)nb, l.HN, NATSL_BF16, c.stream), "natsl_layer_select");
  return o;
}

void project(const Call& c, const bool joint, T (&y)[4]) {
  natsl_project_seg segs[4];
  for (int i = 0; i < 4; ++i) {
    const T& w = c.w[WQ + i];
    if (!joint) {
      y[i] = at::linear(c.x, w);
      continue;
    }
    y[i] = at::empty({c.B, c.T_, w.size(0)}, c.bf16);
    segs[i] = {at_(y[i]), at_(w), (int32_t)w.size(0), (int32_t)w.size(0)};
  }
  if (joint) must(c.l.project(segs, 4, at_(c.x), c.rows, c.l.D, c.l.D, c.stream), "natsl_project");
}

void conv_segs(const Call& c, const T* raw, const T& dt, natsl_conv_seg (&s)[3]) {
  const Layer& l = c.l;
  for (int i = 0; i < 3; ++i) {
    s[i] = natsl_conv_seg{};
    s[i].x = at_(raw[i]); s[i].D = (int32_t)raw[i].size(2); s[i].weight = at_(c.w[CONV_WQ + i]); s[i].bias = at_(c.w[CONV_BQ + i]);
    if (i < 2) {
      s[i].norm_lanes = l.norm_width / 8; s[i].norm_l2 = !l.delta; s[i].norm_eps = l.front_eps;
      s[i].norm_weight = l.delta ? at_(c.w[NORM_Q + i]) : nullptr;
    } else if (dt.defined()) {
      s[i].norm_lanes = l.V / 8; s[i].scale = f_(dt);
    }
  }
}

T mix_logits(const Call& c, const T& yq) {
  const T& w = c.w[W_MIX];
  const int64_t n = w.size(0), d = w.size(1);
  if (!c.l.narrow_fwd_pays(c.rows, (int)d, (int)n) || !on16(w)) return at::linear(yq, w);
  T y = at::empty({c.B, c.T_, n}, c.bf16);
  natsl_front a{};
  a.x = at_(yq); a.wa = at_(w); a.ab = at_(y);
  a.B = 1; a.T = (int32_t)c.rows; a.D = (int32_t)d; a.NA = (int32_t)n; a.ld = (int32_t)n; a.param_dtype = NATSL_BF16;
  must(c.l.layer_front(&a, c.stream), "natsl_layer_front");
  return y;
}

struct Mixed {
  T q_a, k_a, v_a, q_l, k_l, v_l;                       // the operators' inputs
  T o_lin, o_attn, lse, idx, nblk, states, v_new, ws, ht, hs, gs;
};

void mixed(const Call& c, const Front& f, const bool keep, const bool keep_states, const bool final_state, Mixed& m) {
  const Layer& l = c.l;
  const int64_t nb = blocks_of(c.T_), chunks = c.B * nb;
  natsl_mixed a{};
  const size_t ws = l.mixed_workspace_bytes(chunks, l.H);
  m.o_attn = at::empty({c.B, c.T_, l.HQ, l.VA}, c.bf16);
  m.o_lin = at::empty({c.B, c.T_, l.H, l.V}, c.bf16);
  T scratch;
  if (keep) {
    m.idx = at::empty({c.B, nb, l.HN, 2}, c.i32);
    m.nblk = at::empty({c.B, l.HN, 2}, c.i32);
    m.lse = at::empty({c.B, c.T_, l.HQ}, c.f32);
    m.ws = c.bytes(ws);
    a.block_indices = i_(m.idx); a.n_blocks = i_(m.nblk); a.lse = f_(m.lse); a.workspace = at_(m.ws);
  } else {                                               // (nobody sees them afterwards: one piece of memory)
    const int64_t idx = up(c.B * nb * l.HN * 8, 256), nblk = up(c.B * l.HN * 8, 256), lse = up(c.rows * l.HQ * 4, 256);
    scratch = c.bytes((size_t)(idx + nblk + lse) + ws);
    char* p = static_cast<char*>(scratch.data_ptr());
    a.private_tables = 1;
    a.block_indices = reinterpret_cast<int32_t*>(p); a.n_blocks = reinterpret_cast<int32_t*>(p + idx); a.lse = reinterpret_cast<float*>(p + idx + nblk);
    a.workspace = p + idx + nblk + lse;
  }
  if (keep_states) {
    m.states = at::empty({chunks, l.H, l.V, l.K}, c.bf16);
    if (l.delta) m.v_new = like(m.v_l);
  }
  if (final_state) {
    m.ht = at::empty({c.B, l.H, l.K, l.V}, c.f32);
    m.hs = like(m.ht);
    m.gs = at::empty({c.B, l.H}, c.f32);
  }
  a.is_delta = l.delta; a.B = (int32_t)c.B; a.T = a.T_attn = (int32_t)c.T_; a.H = l.H; a.HN = l.HN; a.K = l.K; a.V = l.V; a.TN = a.TN_attn = (int32_t)nb; a.block = 64;
  a.flags = (l.decay ? NATSL_DECAY_NON_LINEAR : 0) | (l.delta ? NATSL_QK_L2NORM : 0) | (l.intra ? NATSL_INTRA_CHUNK : 0);
  a.HQ = a.HKV = l.HQ; a.KA = l.KA; a.VA = l.VA; a.same_block_visible = l.same_block; a.types_dtype = NATSL_BF16;
  a.scale_attn = l.scale_attn; a.scale_linear = l.scale_linear;
  a.q_attn = at_(m.q_a); a.k_attn = at_(m.k_a); a.v_attn = at_(m.v_a); a.types_attn = a.types = at_(f.types); a.o_attn = at_(m.o_attn);
  a.q = at_(m.q_l); a.k = at_(m.k_l); a.v = at_(m.v_l); a.g = f_(f.g); a.beta = at_(f.beta); a.o = at_(m.o_lin);
  a.ht = f_(m.ht); a.h_block_start = f_(m.hs); a.g_block_sum = f_(m.gs); a.chunk_states = at_(m.states); a.chunk_v_new = at_(m.v_new);
  a.workspace_bytes = ws;
  must(l.mixed_fwd(&a, NATSL_MIXED_ROUTE | NATSL_MIXED_SOFTMAX | NATSL_MIXED_LINEAR | NATSL_MIXED_JOIN, c.stream, c.side), "natsl_mixed_fwd");
}

struct Rest {
  T raw[4], y[3], n[2], conv[3], mix, tail, out;         // projections, convolutions, what follows them, new states, mixing logits, norm-gate, output
  Mixed m;
};

void rest(const Call& c, const Front& f, const bool joint, const Needs& needs, const bool keep_states, const bool cache, Rest& r) {
  const Layer& l = c.l;
  project(c, joint, r.raw);
  natsl_conv_seg s[3];
  conv_segs(c, r.raw, f.dt, s);
  for (int i = 0; i < 3; ++i) {
    if (!(i == 1 && !l.delta)) r.y[i] = like(r.raw[i]);
    if (i < 2) {
      r.n[i] = like(r.raw[i]);
      s[i].y = at_(r.y[i]);
      s[i].y_norm = at_(r.n[i]);
    } else {
      (l.delta ? s[i].y : s[i].y_norm) = at_(r.y[i]);
    }
    if (cache) {
      r.conv[i] = at::empty({c.B, r.raw[i].size(2), l.W}, c.bf16);
      s[i].state_out = at_(r.conv[i]);
    }
  }
  must(l.conv_norm_fwd(s, 3, (int)c.B, (int)c.T_, l.W, l.act, l.norm_dtype, c.stream), "natsl_conv_norm_fwd");
  r.mix = mix_logits(c, r.y[0]);
  if (l.delta && !needs.conv) drop(r.raw[0], r.raw[1], r.raw[2]);
  if (!l.delta && !needs.want(W_MIX)) drop(r.y[0]);
  Mixed& m = r.m;
  if (l.delta) {
    m.q_a = r.n[0]; m.k_a = r.n[1]; m.v_a = r.y[2];
    m.q_l = r.y[0]; m.k_l = r.y[1]; m.v_l = r.y[2];
  } else {
    m.q_a = r.raw[0]; m.k_a = r.raw[1]; m.v_a = r.raw[2];
    m.q_l = r.n[0]; m.k_l = r.n[1]; m.v_l = r.y[2];
  }
  mixed(c, f, needs.op, keep_states, cache, m);
  drop(m.q_a, m.q_l);
  if (!keep_states) drop(m.ws);
  if (!cache) drop(m.k_a, m.v_a, m.k_l, m.v_l);
  if (!needs.op) {
    if (!needs.want(W_MIX)) drop(r.y[0]);
    drop(r.raw[0], r.raw[1], r.raw[2], r.y[1], r.y[2], r.n[0], r.n[1]);
  }
  r.tail = like(m.o_attn);
  must(l.norm_gate_logits_fwd(at_(m.o_lin), at_(m.o_attn), at_(r.raw[3]), at_(r.mix), at_(c.w[OUT_NORM1]), at_(c.w[OUT_NORM2]), at_(r.tail), c.rows * l.HQ, l.VA,
                              NATSL_BF16, l.out_eps, l.out_dtype, c.stream), "natsl_norm_gate_logits_fwd");
  if (!needs.tail) drop(m.o_lin, m.o_attn, r.raw[3], r.mix);
  r.out = at::linear(r.tail.view({c.B, c.T_, l.H * l.V}), c.w[WO]);
}

// ---- backward ----------------------------------------------------------------------------------------------------------------
// what the forward keeps, in this order behind x and the weights: each only where a part that runs reads it
enum Kept { AB, WAB, POOLED, LOGITS, TYPES, RAW_Q, RAW_K, RAW_V, GATE, Y_Q, Y_K, Y_V, N_Q, N_K, MIX, G, BETA, DT, O_LIN, O_ATTN, LSE, IDX, NBLK, TAIL, STATES, V_NEW, WS, KEPT };

// dy_i [rows, n_i]^T x [rows, D], one launch for those whose widths are multiples of 8; a narrow one that is not, or that is alone, by itself.  On
// the stream `on`; what is only used there is kept in `hold`.
void wgrads(const Call& c, const T& x, const std::vector<T>& dys, std::vector<T>& out, natsl_stream_t on, Ts& hold) {
  const int64_t rows = x.size(0), D = x.size(1);
  out.assign(dys.size(), T());
  std::vector<natsl_wgrad_seg> segs;
  const bool alone = std::count_if(dys.begin(), dys.end(), [](const T& t) { return t.defined(); }) == 1;
  for (size_t i = 0; i < dys.size(); ++i) {
    const T& dy = dys[i];
    if (!dy.defined()) continue;
    const int64_t N = dy.size(1);
    if (c.l.narrow_wgrad_pays(rows, (int)D, (int)N, 0, alone) && !(reinterpret_cast<uintptr_t>(x.data_ptr()) & 3)) {
      out[i] = at::empty({N, D}, c.bf16);
      const size_t n = c.l.narrow_wgrad_workspace_bytes(rows, (int)D, (int)N);
      const T ws = c.bytes(n);
      hold.push_back(ws);
      must(c.l.narrow_wgrad_split(at_(dy), at_(x), at_(out[i]), rows, (int)D, (int)N, at_(ws), n, on), "natsl_narrow_wgrad_split");
      continue;
    }
    if (dy.size(1) % 8 || D % 8 || !on16(x) || !on16(dy)) {
      out[i] = at::mm(dy.t(), x);
      continue;
    }
    out[i] = at::empty({dy.size(1), D}, c.bf16);
    segs.push_back({at_(dy), at_(out[i]), (int32_t)dy.size(1), (int32_t)dy.size(1)});
  }
  if (segs.empty()) return;
  const size_t n = c.l.wgrad_workspace_bytes(segs.data(), (int)segs.size(), rows, (int)D);
  const T ws = c.bytes(n);
  hold.push_back(ws);
  must(c.l.wgrad(segs.data(), (int)segs.size(), at_(x), rows, (int)D, (int)D, at_(ws), n, on), "natsl_wgrad");
}
T wgrad(const Call& c, const T& x, const T& dy, natsl_stream_t on, Ts& hold) {
  std::vector<T> out;
  wgrads(c, x, {dy}, out, on, hold);
  return out[0];
}
T wgrad(const Call& c, const T& x, const T& dy) {
  Ts hold;
  return wgrad(c, x, dy, c.stream, hold);
}

bool narrow_bwd_takes(const Call& c, const T& dy, const T& w, const bool few) {
  return c.l.narrow_linear_bwd_pays(dy.size(0), (int)w.size(1), (int)w.size(0), few) && on16(dy) && on16(w);
}
T narrow_bwd(const Call& c, const T& dy, const T& w, const bool few, natsl_stream_t on, T dx = T()) {
  const int64_t N = w.size(0), D = w.size(1);
  if (!narrow_bwd_takes(c, dy, w, few)) return at::mm(dy, w);
  if (!dx.defined()) dx = at::empty({dy.size(0), D}, c.bf16);
  must(c.l.narrow_linear_bwd(at_(dy), at_(w), at_(dx), dy.size(0), (int)D, (int)N, on), "natsl_narrow_linear_bwd");
  return dx;
}

// joins the streams on the way out, errors included: what the other one works on may be freed then
struct Fork {
  const Call& c;
  bool open = false;
  explicit Fork(const Call& call) : c(call) {}
  void join() {
    if (!open) return;
    open = false;
    must(c.l.order_streams(c.side, c.stream), "natsl_order_streams");
  }
  ~Fork() {
    if (open) (void)c.l.order_streams(c.side, c.stream);
  }
};

struct MixedGrads {
  T q_a, k_a, v_a, q_l, k_l, v_l, g, beta, logits;                // logits: the selector's
};

// behind: what else may run behind the softmax branch, on the stream that it is given: beside the linear branch's last kernel, where there are two.
template <class Behind>
MixedGrads mixed_bwd(const Call& c, const Ts& s, const T& do_lin, const T& do_attn, const int invalid_attn, const int invalid_linear, Behind behind) {
  const Layer& l = c.l;
  const int64_t nb = blocks_of(c.T_), chunks = c.B * nb;
  const bool delta = l.delta, beside = c.side != c.stream, saved = s[STATES].defined();
  const T q_a = delta ? s[N_Q] : s[RAW_Q], k_a = delta ? s[N_K] : s[RAW_K], v_a = delta ? s[Y_V] : s[RAW_V];
  const T q_l = delta ? s[Y_Q] : s[N_Q], k_l = delta ? s[Y_K] : s[N_K], v_l = s[Y_V];
  const int flags = (l.decay ? NATSL_DECAY_NON_LINEAR : 0) | (delta ? NATSL_QK_L2NORM : 0) | (l.intra ? NATSL_INTRA_CHUNK : 0);
  const int B = (int)c.B, Tn = (int)c.T_, TN = (int)nb;
  MixedGrads r;
  // The softmax branch's tensors are made first, on this stream, and live until this stream has its kernels behind it.
  r.q_a = like(q_a); r.k_a = like(k_a); r.v_a = like(v_a);
  const T dnats = at::empty({c.B, nb, l.HQ}, c.f32);
  const size_t sb = l.softmax_bwd_workspace_bytes(B, Tn, l.HQ);
  const T sws = c.bytes(sb);
  auto softmax = [&](natsl_stream_t on) {
    must(l.softmax_sparse_bwd(at_(q_a), at_(k_a), at_(v_a), at_(s[O_ATTN]), f_(s[LSE]), at_(do_attn), at_(r.q_a), at_(r.k_a), at_(r.v_a), f_(dnats), at_(s[TYPES]),
                              NATSL_BF16, i_(s[IDX]), i_(s[NBLK]), B, Tn, l.HQ, l.HQ, l.HN, l.KA, l.VA, TN, 64, l.scale_attn,
                              (l.same_block ? 1 : 0) | (invalid_attn ? 2 : 0), NATSL_BF16, at_(sws), sb, nullptr, 0, 0, 0, on), "natsl_softmax_sparse_bwd");
  };
  Fork fork(c);
  if (!beside) {
    softmax(c.stream);
  } else if (saved) {
    must(l.order_streams(c.stream, c.side), "natsl_order_streams");
    fork.open = true;
  }
  // side by side both scans are enqueued first, with the softmax branch behind the kernel in front of the first
  T states = s[STATES], v_new = delta ? s[V_NEW] : v_l, ws = s[WS];
  if (!saved) {
    states = at::empty({chunks, l.H, l.V, l.K}, c.bf16);
    if (delta) v_new = like(v_l);
    const size_t n = l.linear_workspace_bytes(chunks, l.H);
    ws = c.bytes(n);
    fork.open = beside;
    must(l.linear_chunk_states(delta, at_(q_l), at_(k_l), at_(v_l), f_(s[G]), at_(s[BETA]), nullptr, nullptr, at_(states), delta ? at_(v_new) : nullptr, at_(s[TYPES]),
                               NATSL_BF16, B, Tn, l.H, l.HN, l.K, l.V, TN, 64, l.scale_linear, flags, at_(ws), n, NATSL_BF16, nullptr, 0, (int)chunks, c.stream,
                               beside ? c.side : nullptr), "natsl_linear_chunk_states");
  }
  const T d_states = like(states);
  r.q_l = like(q_l); r.k_l = like(k_l); r.v_l = like(v_l);
  r.g = at::empty({c.B, c.T_, l.H}, c.f32);
  T parts;
  if (delta) {
    r.beta = at::empty({c.B, c.T_, l.H}, c.bf16);
    parts = at::empty({c.B, c.T_, l.H, l.V / 16}, c.f32);
  }
  const T gate = at::empty({chunks, l.H}, c.f32), rb = like(gate);
  must(l.linear_chunk_bwd_steps(3 + (beside ? 4 : 0) + (delta ? 8 : 0), 0, nullptr, delta, at_(q_l), at_(k_l), at_(v_new), f_(s[G]), at_(s[BETA]), at_(do_lin), nullptr,
                                at_(states), at_(s[TYPES]), NATSL_BF16, nullptr, at_(ws), at_(d_states), f_(parts), at_(r.q_l), at_(r.k_l), at_(r.v_l), f_(r.g),
                                at_(r.beta), nullptr, f_(gate), f_(rb), B, Tn, l.H, l.HN, l.K, l.V, TN, 64, l.scale_linear, flags, NATSL_BF16, nullptr, 0, (int)chunks,
                                c.stream), "natsl_linear_chunk_bwd_steps");
  if (beside) {
    softmax(c.side);
    behind(c.side);
    fork.join();
  } else {
    behind(c.stream);
  }
  r.logits = like(s[LOGITS]);
  must(l.block_grads_logits(at_(s[TYPES]), at_(s[LOGITS]), NATSL_BF16, f_(gate), l.decay ? f_(rb) : nullptr, f_(dnats), l.HQ, f_(r.g), at_(r.logits), invalid_linear,
                            B, Tn, l.H, l.HN, TN, 64, c.stream), "natsl_block_grads_logits");
  return r;
}

// dout: c.x; s: what the forward kept, dropped on the way; grads: x, then the weights
void backward(const Call& c, const T& x, Ts& s, const Needs& need, const int invalid_attn, const int invalid_linear, Ts& grads) {
  const Layer& l = c.l;
  const Ts& w = c.w;
  grads.assign(1 + WEIGHTS, T());
  auto want = [&](const Weight i) { return need.want(i); };
  const int64_t rows = c.rows, vd = l.H * l.V;
  const T d2 = c.x.reshape({rows, l.D}).contiguous();
  if (want(WO)) grads[1 + WO] = wgrad(c, s[TAIL].view({rows, vd}), d2);
  drop(s[TAIL]);
  if (!need.tail) return;
  T dy = at::mm(d2, w[WO]);
  // norm-gate
  T do_lin = like(s[O_LIN]), do_attn = like(s[O_ATTN]), dgate = like(s[GATE]), dmix = like(s[MIX]), dwn = at::empty({2, l.VA}, c.f32);
  {
    const size_t n = l.norm_gate_bwd_workspace_bytes(rows * l.HQ, l.VA);
    const T ws = c.bytes(n);
    must(l.norm_gate_logits_bwd(at_(s[O_LIN]), at_(s[O_ATTN]), at_(s[GATE]), at_(s[MIX]), at_(w[OUT_NORM1]), at_(w[OUT_NORM2]), at_(dy), at_(do_lin), at_(do_attn),
                                at_(dgate), at_(dmix), f_(dwn), f_(dwn) + l.VA, at_(ws), n, rows * l.HQ, l.VA, NATSL_BF16, l.out_eps, l.out_dtype, c.stream),
         "natsl_norm_gate_logits_bwd");
    if (want(OUT_NORM1) || want(OUT_NORM2)) {
      const T d = dwn.to(w[OUT_NORM1].scalar_type());
      grads[1 + OUT_NORM1] = d.select(0, 0);
      grads[1 + OUT_NORM2] = d.select(0, 1);
    }
  }
  drop(dy, s[O_LIN], s[GATE], s[MIX]);
  // mixing logits: they need the norm-gate only, and the softmax branch's stream is done 75 to 160 us before the linear branch's (a layer's training
  // step at 340M 8 x 4096 3 202 -> 3 184 us, 760M 2 x 3000 1 468 -> 1 446; o_proj's weight gradient there as well: 3 223 and 1 485 for 3 266 and 1 503)
  Ts hold;                                               // (what that stream uses lives until it is joined)
  T dq_mix;
  dmix = dmix.view({rows, -1});
  auto mixing = [&](natsl_stream_t on) {
    if (want(W_MIX)) grads[1 + W_MIX] = wgrad(c, s[Y_Q].view({rows, -1}), dmix, on, hold);
    // (its place is the softmax branch's output gradient, which only that branch reads; where that is too small it waits)
    if (!need.op || !need.conv) return;
    const int64_t n = rows * w[W_MIX].size(1);
    if (n <= do_attn.numel() && narrow_bwd_takes(c, dmix, w[W_MIX], false))
      dq_mix = narrow_bwd(c, dmix, w[W_MIX], false, on, do_attn.view({-1}).narrow(0, 0, n).view({rows, -1}));
  };
  MixedGrads m;
  if (need.op) m = mixed_bwd(c, s, do_lin, do_attn, invalid_attn, invalid_linear, mixing);
  else mixing(c.stream);
  drop(do_lin, do_attn, s[Y_Q]);
  hold.clear();
  for (const Kept i : {O_ATTN, LSE, IDX, NBLK, TYPES, LOGITS, G, BETA, N_Q, N_K, Y_K, Y_V, STATES, V_NEW, WS}) drop(s[i]);
  // convolutions
  T dx[4], ddt;
  dx[3] = std::move(dgate);
  if (need.conv) {
    if (!dq_mix.defined()) dq_mix = narrow_bwd(c, dmix, w[W_MIX], false, c.stream);
    drop(dmix);
    natsl_conv_seg g[3];
    conv_segs(c, &s[RAW_Q], s[DT], g);
    for (int i = 0; i < 3; ++i) {
      dx[i] = like(s[RAW_Q + i]);
      const T dw = like(w[CONV_WQ + i]);
      g[i].dx = at_(dx[i]);
      g[i].dweight = at_(dw);
      grads[1 + CONV_WQ + i] = dw;
      if (w[CONV_BQ + i].defined()) {
        grads[1 + CONV_BQ + i] = like(w[CONV_BQ + i]);
        g[i].dbias = at_(grads[1 + CONV_BQ + i]);
      }
    }
    g[0].dy_b = at_(dq_mix);
    if (l.delta) {
      g[0].dy_a = at_(m.q_l); g[1].dy_a = at_(m.k_l); g[2].dy_a = at_(m.v_l);
      g[2].dy_b = at_(m.v_a);
      g[0].dy_norm = at_(m.q_a); g[1].dy_norm = at_(m.k_a);
      for (int i = 0; i < 2; ++i) {
        grads[1 + NORM_Q + i] = like(w[NORM_Q + i]);
        g[i].dnorm_weight = at_(grads[1 + NORM_Q + i]);
      }
    } else {
      g[0].dy_norm = at_(m.q_l); g[1].dy_norm = at_(m.k_l); g[2].dy_norm = at_(m.v_l);
      g[0].dx_add = at_(m.q_a); g[1].dx_add = at_(m.k_a); g[2].dx_add = at_(m.v_a);
      ddt = like(s[DT]);
      g[2].dscale = f_(ddt);
    }
    const size_t n = l.conv_norm_bwd_workspace_bytes(g, 3, (int)c.B, (int)c.T_, l.W);
    const T ws = c.bytes(n);
    must(l.conv_norm_bwd(g, 3, (int)c.B, (int)c.T_, l.W, l.act, l.norm_dtype, at_(ws), n, c.stream), "natsl_conv_norm_bwd");
  }
  drop(dmix, dq_mix, m.q_a, m.k_a, m.v_a, m.q_l, m.k_l, m.v_l, s[RAW_Q], s[RAW_K], s[RAW_V], s[DT]);
  // gates
  T dab;
  if (need.gates) {
    dab = like(s[AB]);
    grads[1 + A_LOG] = like(w[A_LOG]);
    grads[1 + DT_BIAS] = like(w[DT_BIAS]);
    const size_t n = l.gates_bwd_workspace_bytes(rows, l.H);
    const T ws = c.bytes(n);
    must(l.gates_bwd(at_(s[AB]), at_(w[A_LOG]), at_(w[DT_BIAS]), f_(m.g), at_(m.beta), f_(ddt), l.delta, at_(dab), at_(grads[1 + A_LOG]), at_(grads[1 + DT_BIAS]), at_(ws), n,
                     rows, l.H, (int)s[AB].size(2), l.neg, l.gate_dtype, c.stream), "natsl_gates_bwd");
  }
  drop(m.g, m.beta, ddt, s[AB]);
  // selector
  T dl2;
  if (need.op) dl2 = m.logits.view({-1, l.NL});
  if (want(WN)) {
    const int64_t r = dl2.size(0), n = l.NL;
    if (!l.narrow_wgrad_pays(r, l.D, (int)n, 1, 0)) {
      grads[1 + WN] = at::mm(dl2.t(), s[POOLED]);
    } else {
      grads[1 + WN] = at::empty({n, l.D}, c.bf16);
      must(l.narrow_wgrad(at_(dl2), at_(s[POOLED]), at_(grads[1 + WN]), r, l.D, (int)n, c.stream), "natsl_narrow_wgrad");
    }
  }
  std::vector<T> dys(5);
  for (int i = 0; i < 4; ++i)
    if (dx[i].defined()) dys[i] = dx[i].view({rows, -1});
  drop(dx[0], dx[1], dx[2], dx[3]);
  if (dab.defined()) dys[4] = dab.view({rows, -1});
  if (need.x()) {
    const int64_t ld = dab.size(2);
    const T dpool = narrow_bwd(c, dl2, w[WN], true, c.stream), dX = c.sized(l.D);
    natsl_project_seg segs[5];
    for (int i = 0; i < 5; ++i) {
      const T& ww = i < 4 ? w[WQ + i] : s[WAB];
      segs[i] = {at_(dys[i]), at_(ww), (int32_t)ww.size(0), (int32_t)ww.size(0)};
    }
    if (l.project_bwd_takes(segs, 5, at_(dpool), at_(dX))) {
      must(l.project_bwd(segs, 5, at_(dpool), at_(dX), (int)c.B, (int)c.T_, l.D, 64, c.stream), "natsl_project_bwd");
    } else {
      must(l.dx_init(at_(dys[4]), at_(s[WAB]), at_(dpool), at_(dX), (int)c.B, (int)c.T_, l.D, (int)ld, (int)ld, 64, c.stream), "natsl_dx_init");
      T flat = dX.view({rows, l.D});
      for (int i = 0; i < 4; ++i) flat.addmm_(dys[i], w[WQ + i]);
    }
    grads[0] = dX;
  }
  for (int i = 0; i < 4; ++i)
    if (!want(Weight(WQ + i))) dys[i] = T();
  if (!want(WA) && !want(WB)) dys[4] = T();
  if (std::none_of(dys.begin(), dys.end(), [](const T& t) { return t.defined(); })) return;
  std::vector<T> dws;
  wgrads(c, x.view({rows, l.D}), dys, dws, c.stream, hold);
  for (int i = 0; i < 4; ++i) grads[1 + WQ + i] = dws[i];
  if (dws[4].defined()) {
    grads[1 + WA] = dws[4].slice(0, 0, l.H);
    if (l.delta) grads[1 + WB] = dws[4].slice(0, l.H, 2 * l.H);
  }
}

// ---- Python ------------------------------------------------------------------------------------------------------------------
void free_layer(PyObject* capsule) {
  auto* l = static_cast<Layer*>(PyCapsule_GetPointer(capsule, LAYER));
  Py_DECREF(l->check);
  delete l;
}

Layer* layer_of(PyObject* o) { return static_cast<Layer*>(PyCapsule_GetPointer(o, LAYER)); }

PyObject* wrap(const T& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}
PyObject* tuple_of(const Ts& ts) {
  THPObjectPtr out(PyTuple_New((Py_ssize_t)ts.size()));
  if (!out) return nullptr;
  for (size_t i = 0; i < ts.size(); ++i) {
    PyObject* o = wrap(ts[i]);
    if (!o) return nullptr;
    PyTuple_SET_ITEM(out.get(), (Py_ssize_t)i, o);
  }
  return out.release();
}
bool tensors_of(PyObject* seq, Ts& out) {
  THPObjectPtr fast(PySequence_Fast(seq, "a sequence of tensors"));
  if (!fast) return false;
  const Py_ssize_t n = PySequence_Fast_GET_SIZE(fast.get());
  out.resize((size_t)n);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = PySequence_Fast_GET_ITEM(fast.get(), i);
    if (o == Py_None) continue;
    if (!THPVariable_Check(o)) {
      PyErr_SetString(PyExc_TypeError, "tensors or None");
      return false;
    }
    out[(size_t)i] = THPVariable_Unpack(o);
  }
  return true;
}
bool weights_of(PyObject* seq, Ts& out) {
  if (!tensors_of(seq, out)) return false;
  if ((int)out.size() == WEIGHTS) return true;
  PyErr_Format(PyExc_ValueError, "%d weights, got %d", (int)WEIGHTS, (int)out.size());
  return false;
}
// body() without the interpreter's lock; an entry point's failure becomes the exception that `check` raises
template <class F>
bool run_free(const Layer& l, F body) {
  Failed failed{0, nullptr};
  {
    struct Unlock {
      PyThreadState* s = PyEval_SaveThread();
      ~Unlock() { PyEval_RestoreThread(s); }
    } unlocked;
    c10::NoGradGuard no_grad;
    try {
      body();
    } catch (const Failed& f) {
      failed = f;
    }
  }
  if (!failed.rc) return true;
  THPObjectPtr r(PyObject_CallFunction(l.check, "is", failed.rc, failed.what));
  if (r) PyErr_SetString(PyExc_RuntimeError, failed.what);
  return false;
}
natsl_stream_t stream_of(PyObject* o) { return static_cast<natsl_stream_t>(PyLong_AsVoidPtr(o)); }

}  // namespace

// make_layer(the library's handle, check, the integers and the numbers of Layer in its order)
PyObject* natsl_make_layer(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  unsigned long long handle;
  PyObject* check;
  Layer l{};
  if (!PyArg_ParseTuple(args, "KO(iiiiiiiiiiiiiiiiiiiii)(ffff)", &handle, &check, &l.device, &l.delta, &l.D, &l.H, &l.K, &l.V, &l.HQ, &l.KA, &l.VA, &l.HN, &l.NL, &l.W, &l.act,
                        &l.norm_width, &l.norm_dtype, &l.gate_dtype, &l.out_dtype, &l.neg, &l.decay, &l.same_block, &l.intra, &l.front_eps, &l.out_eps, &l.scale_attn,
                        &l.scale_linear))
    return nullptr;
  void* const lib = reinterpret_cast<void*>(handle);
#define X(n)                                                                        \
  if (!(l.n = reinterpret_cast<decltype(l.n)>(dlsym(lib, "natsl_" #n)))) {           \
    PyErr_SetString(PyExc_RuntimeError, "the library does not export natsl_" #n);    \
    return nullptr;                                                                  \
  }
  NATSL_ENTRIES(X)
#undef X
  l.check = check;
  auto* own = new Layer(l);
  Py_INCREF(check);
  PyObject* capsule = PyCapsule_New(own, LAYER, free_layer);
  if (!capsule) {
    Py_DECREF(check);
    delete own;
  }
  return capsule;
  END_HANDLE_TH_ERRORS
}

bool needs_of(PyObject* seq, std::vector<bool>& need) {
  THPObjectPtr fast(PySequence_Fast(seq, "what wants a gradient"));
  if (!fast) return false;
  if (PySequence_Fast_GET_SIZE(fast.get()) != 1 + WEIGHTS) {
    PyErr_SetString(PyExc_ValueError, "what wants a gradient: x, then the weights");
    return false;
  }
  need.resize(1 + WEIGHTS);
  for (int i = 0; i <= WEIGHTS; ++i) need[(size_t)i] = PyObject_IsTrue(PySequence_Fast_GET_ITEM(fast.get(), i)) > 0;
  return true;
}

// layer_train(layer, x, weights, stream, side, joint, what wants a gradient (x, then the weights) or None, keep states) -> (out, attention's share per
// head, what the backward needs: x, the weights and KEPT tensors, None for those that it does not read; or None)
PyObject* natsl_layer_train(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Ts w;
  std::vector<bool> of;
  if (n != 8 || !THPVariable_Check(a[1])) {
    PyErr_SetString(PyExc_TypeError, "layer_train(layer, x, weights, stream, side, joint, needs, keep states)");
    return nullptr;
  }
  Layer* l = layer_of(a[0]);
  if (!l || !weights_of(a[2], w) || (a[6] != Py_None && !needs_of(a[6], of))) return nullptr;
  const Needs need(of, l->delta);
  const Call c(*l, THPVariable_Unpack(a[1]), w, stream_of(a[3]), stream_of(a[4]));
  const bool joint = PyObject_IsTrue(a[5]) > 0, states = need.op && PyObject_IsTrue(a[7]) > 0;
  Front f;
  Rest r;
  if (!run_free(*l, [&] {
        f = front(c, need, false);
        rest(c, f, joint, need, states, false, r);
      }))
    return nullptr;
  const Mixed& m = r.m;
  THPObjectPtr kept;
  if (!of.empty()) {
    Ts all(1 + WEIGHTS + KEPT);
    T* const s = all.data() + 1 + WEIGHTS;
    auto weights = [&](std::initializer_list<Weight> ws) {
      for (const Weight i : ws) all[1 + i] = w[i];
    };
    if (need.want(WO)) s[TAIL] = r.tail;
    if (need.tail) {
      weights({WO, OUT_NORM1, OUT_NORM2});
      s[GATE] = r.raw[3]; s[MIX] = r.mix; s[O_LIN] = m.o_lin; s[O_ATTN] = m.o_attn;
    }
    if (need.want(W_MIX)) s[Y_Q] = r.y[0];
    if (need.op) {
      for (int i = 0; i < 3; ++i) {
        if (i > 0 || l->delta) s[Y_Q + i] = r.y[i];
        if (need.conv || !l->delta) s[RAW_Q + i] = r.raw[i];
      }
      s[LOGITS] = f.logits; s[TYPES] = f.types; s[G] = f.g; s[BETA] = f.beta; s[N_Q] = r.n[0]; s[N_K] = r.n[1]; s[LSE] = m.lse; s[IDX] = m.idx; s[NBLK] = m.nblk;
    }
    if (states) { s[STATES] = m.states; s[V_NEW] = m.v_new; s[WS] = m.ws; }
    if (need.conv) {
      weights({W_MIX, CONV_WQ, CONV_WK, CONV_WV, CONV_BQ, CONV_BK, CONV_BV, NORM_Q, NORM_K});
      s[DT] = f.dt;
    }
    if (need.gates) {
      weights({A_LOG, DT_BIAS});
      s[AB] = f.ab;
    }
    if (need.x()) {
      weights({WQ, WK, WV, WG, WN});
      s[WAB] = f.wab;
    }
    if (need.x() || need.want(WA) || need.want(WB)) weights({WA, WB});          // (read as WAB, which was made of them)
    s[POOLED] = f.pooled;
    for (const Weight i : {WQ, WK, WV, WG, WA, WB})
      if (need.want(i)) all[0] = c.x;
    kept = tuple_of(all);
  } else {
    Py_INCREF(Py_None);
    kept = Py_None;
  }
  THPObjectPtr o(wrap(r.out)), fr(wrap(f.fraction));
  if (!kept || !o || !fr) return nullptr;
  return PyTuple_Pack(3, o.get(), fr.get(), kept.get());
  END_HANDLE_TH_ERRORS
}

// layer_backward(layer, dout, what the forward kept (a list, emptied: its tensors are dropped after their last use), what wants a gradient (x, then the weights), stream, side, invalid attention, invalid linear)
// -> gradients of x, then of the weights
PyObject* natsl_layer_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Ts kept, grads;
  std::vector<bool> of;
  if (n != 8 || !THPVariable_Check(a[1]) || !PyList_Check(a[2])) {
    PyErr_SetString(PyExc_TypeError, "layer_backward(layer, dout, kept, needs, stream, side, invalid attention, invalid linear)");
    return nullptr;
  }
  Layer* l = layer_of(a[0]);
  if (!l || !tensors_of(a[2], kept) || !needs_of(a[3], of)) return nullptr;
  if ((int)kept.size() != 1 + WEIGHTS + KEPT) {
    PyErr_SetString(PyExc_ValueError, "layer_backward: another number of tensors than the forward gave");
    return nullptr;
  }
  if (PyList_SetSlice(a[2], 0, PyList_GET_SIZE(a[2]), nullptr) < 0) return nullptr;
  const Needs need(of, l->delta);
  const T x = kept[0];
  const Ts w(kept.begin() + 1, kept.begin() + 1 + WEIGHTS);
  Ts s(kept.begin() + 1 + WEIGHTS, kept.end());
  kept.clear();
  const Call c(*l, THPVariable_Unpack(a[1]), w, stream_of(a[4]), stream_of(a[5]));
  const int ia = PyObject_IsTrue(a[6]) > 0, il = PyObject_IsTrue(a[7]) > 0;
  if (!run_free(*l, [&] { backward(c, x, s, need, ia, il, grads); })) return nullptr;
  for (int i = 0; i <= WEIGHTS; ++i)
    if (!of[(size_t)i]) grads[(size_t)i] = T();
  return tuple_of(grads);
  END_HANDLE_TH_ERRORS
}

// layer_front(layer, x, weights, stream) -> (g, beta, dt, logits, types, raw types, counts, attention's share per head)
PyObject* natsl_layer_prompt_front(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Ts w;
  if (n != 4 || !THPVariable_Check(a[1])) {
    PyErr_SetString(PyExc_TypeError, "layer_front(layer, x, weights, stream)");
    return nullptr;
  }
  Layer* l = layer_of(a[0]);
  if (!l || !weights_of(a[2], w)) return nullptr;
  const Call c(*l, THPVariable_Unpack(a[1]), w, stream_of(a[3]), nullptr);
  Front f;
  if (!run_free(*l, [&] { f = front(c, Needs({}, l->delta), true); })) return nullptr;
  return tuple_of({f.g, f.beta, f.dt, f.logits, f.types, f.raw, f.counts, f.fraction});
  END_HANDLE_TH_ERRORS
}

// layer_rest(layer, x, weights, what layer_front gave, stream, side, joint, cache) -> (out, keys and values of attention, of the linear branch, the convolutions' states,
// final state, the state that entered the last block, sum of g over it): what a cache keeps is None without `cache`
PyObject* natsl_layer_prompt_rest(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Ts w, fr;
  if (n != 8 || !THPVariable_Check(a[1])) {
    PyErr_SetString(PyExc_TypeError, "layer_rest(layer, x, weights, front, stream, side, joint, cache)");
    return nullptr;
  }
  Layer* l = layer_of(a[0]);
  if (!l || !weights_of(a[2], w) || !tensors_of(a[3], fr)) return nullptr;
  if (fr.size() != 8) {
    PyErr_SetString(PyExc_ValueError, "layer_rest: what layer_front gave");
    return nullptr;
  }
  const Call c(*l, THPVariable_Unpack(a[1]), w, stream_of(a[4]), stream_of(a[5]));
  const bool joint = PyObject_IsTrue(a[6]) > 0, cache = PyObject_IsTrue(a[7]) > 0;
  Front f;
  f.g = fr[0]; f.beta = fr[1]; f.dt = fr[2]; f.types = fr[4];
  Rest r;
  Ts out(11);
  if (!run_free(*l, [&] {
        rest(c, f, joint, Needs({}, l->delta), false, cache, r);
        out[0] = r.out;
        if (cache) {
          const Mixed& m = r.m;
          out[1] = m.k_a.view({c.B, c.T_, l->HQ, l->KA}); out[2] = m.v_a.view({c.B, c.T_, l->HQ, l->VA});
          out[3] = m.k_l.view({c.B, c.T_, l->H, l->K}); out[4] = m.v_l.view({c.B, c.T_, l->H, l->V});
          for (int i = 0; i < 3; ++i) out[5 + i] = r.conv[i];
          out[8] = m.ht; out[9] = m.hs; out[10] = m.gs;
        }
      }))
    return nullptr;
  return tuple_of(out);
  END_HANDLE_TH_ERRORS
}
