// A generation step of a whole hybrid layer: a few new tokens of each cached sequence, from the hidden states to the layer's
// output, in one launch for one token of few sequences, three for one token a sequence and five for several.  At this size a step is bound by launches and by the
// host that issues them (the same step as separate operations was 40 launches, 0.2 ms of kernels and 0.57 ms of host time for one
// 340M-geometry layer), so each kernel takes as much of the step as its data dependences allow:
//   rows_gemm_kernel     q, k, v, gate, a (and beta) projections as one pass over all their weights; the output projection
//   step_one_kernel      one token a sequence: all that the other three do
//   step_all_kernel      ... and both products
//   step_mix_kernel      short convolutions, activations, row norms, gates; the new rows of every cache, written in place
//   attend_and_recur     attention over the cached keys next to the token recurrence (natsl_decode.hip)
//   step_tail_kernel     join of the attention's splits, mixing weights, two-input norm and gate
// Roundings to bf16 are where the layer's separate operations round (projections, convolutions, norms, gates, branch outputs).
#include <algorithm>
#include <atomic>
#include <mutex>

#include "natsl_decode_device.h"
#include "natsl_host.h"

namespace natsl {

constexpr int STEP_MAX_ROWS = 64;

// ---- out[m][col] = x[m] . w[n] for a few rows x and several weight matrices ---------------------------------------------
// Bound by reading the weights once.  A workgroup owns 16 weight rows; its eight waves split the contraction (each takes every
// eighth 32-wide step, all loads of up to four steps in flight) so that even a 1024-wide output has 512 waves requesting; the
// partial tiles are added in LDS in a fixed order.  Weights are the A operand, straight from memory to registers: no reuse, no LDS.
struct GemmSeg { const bf16_t* w; int rows, tile0, col0; };
constexpr int GEMM_SEGS = 6;
struct RowsGemm {
  const bf16_t* x; bf16_t* out;
  int M, D, ldo, n_seg;
  GemmSeg seg[GEMM_SEGS];
  unsigned* zero; int n_zero;   // cleared for a later launch of the step
  const unsigned* failed;       // null, or where a step says that it has failed: then the rows are NaN
};

// FAILED: p.failed is looked at.  (For all launches, and through an argument that may be null, it was 0.5 us of eight sequences' step on 16 heads of 128/64.)
template <int MT, bool FAILED>
__global__ __launch_bounds__(512) void rows_gemm_kernel(const RowsGemm p) {
  constexpr int NW = 8, U = 4;
  __shared__ f32x4 red[NW][MT][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < p.n_zero; i += 512) p.zero[i] = 0u;
  // (by steps before this one, whose launches are over.  The lanes' load, waited for with the weights': a scalar one holds up the first use of an argument)
  unsigned failed = 0u;
  if constexpr (FAILED) failed = __hip_atomic_load(p.failed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  int si = 0;
#pragma unroll
  for (int i = 1; i < GEMM_SEGS; ++i) si = i < p.n_seg && (int)blockIdx.x >= p.seg[i].tile0 ? i : si;
  const GemmSeg sg = p.seg[si];
  const int n0 = 16 * ((int)blockIdx.x - sg.tile0);
  const int r16 = lane & 15, kg = lane >> 4;
  const bf16_t* wp = sg.w + (size_t)min(n0 + r16, sg.rows - 1) * p.D + 8 * kg;
  const bf16_t* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xp[t] = p.x + (size_t)min(16 * t + r16, p.M - 1) * p.D + 8 * kg;
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const int steps = p.D / 32;
  int s = wave;
  for (; s + (U - 1) * NW < steps; s += U * NW) {
    bf16x8 a[U], b[U][MT];
#pragma unroll
    for (int u = 0; u < U; ++u) a[u] = ld8(wp + 32 * (s + u * NW));
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < MT; ++t) b[u][t] = ld8(xp[t] + 32 * (s + u * NW));
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[t] = mfma16(a[u], b[u][t], acc[t]);
  }
  for (; s < steps; s += NW) {
    const bf16x8 a = ld8(wp + 32 * s);
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = mfma16(a, ld8(xp[t] + 32 * s), acc[t]);
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) red[wave][t][lane] = acc[t];
  __syncthreads();
  if (wave >= MT) return;
  f32x4 sum = red[0][wave][lane];
#pragma unroll
  for (int w = 1; w < NW; ++w) sum += red[w][wave][lane];
  if (FAILED && failed != 0u) sum = (f32x4){NAN, NAN, NAN, NAN};
  // lane: row m = lane%16 of the tile, columns 4*(lane/16)..
  const int m = 16 * wave + r16, n = n0 + 4 * kg;
  if (m >= p.M) return;
  bf16_t* dst = p.out + (size_t)m * p.ldo + sg.col0 + n;
  if (n + 4 <= sg.rows) {
    *reinterpret_cast<u32x2*>(dst) = (u32x2){pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3])};
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (n + j < sg.rows) dst[j] = f32_to_bf16(sum[j]);
  }
}

// ---- convolutions, norms, gates, cache rows -------------------------------------------------------------------------------
struct StepMix {
  natsl_layer_step s;
  const bf16_t* proj; int ldp, cq, ck, cv, ca, cb;   // projections [M][ldp] and where each starts in a row
  bf16_t *q_conv, *q_lin, *q_attn;                    // [M][H*K]; q_lin == q_conv without L2-normalised rows
};

template <int W>
struct ConvWindow {
  float e[W], w[W], b;      // e: the last W inputs
  NATSL_DEVICE void init(const bf16_t* state, const bf16_t* weight, const bf16_t* bias, const size_t d, const size_t sd) {
    b = bias ? bf16_to_f32(bias[d]) : 0.f;
#pragma unroll
    for (int j = 0; j < W; ++j) {
      e[j] = bf16_to_f32(state[sd * W + j]);
      w[j] = bf16_to_f32(weight[d * W + j]);
    }
  }
  NATSL_DEVICE float next(const float x, const bool silu) {
#pragma unroll
    for (int j = 0; j + 1 < W; ++j) e[j] = e[j + 1];
    e[W - 1] = x;
    float a = b;
#pragma unroll
    for (int j = 0; j < W; ++j) a += w[j] * e[j];
    if (silu) a = a / (1.f + __expf(-a));
    return bf16_to_f32(f32_to_bf16(a));
  }
  NATSL_DEVICE void save(bf16_t* state, const size_t sd) {
#pragma unroll
    for (int j = 0; j < W; ++j) state[sd * W + j] = f32_to_bf16(e[j]);
  }
};

// What one token needs from memory, as it was loaded: a launch that does little else asks for all of it before it looks at any of it.  A
// load behind a branch, or converted where it stands, is waited for on the spot, so nothing here depends on which form an input has: the
// absent one is read from another tensor's place and dropped.  (An attending wave made four to seven round trips one behind another before
// its first keys, three are left: arguments, windows and flags, keys.  step_one_kernel, 340M geometry, one sequence of 800 tokens: 10.9 -> 9.6 us;
// 16 heads of 128/64, eight sequences of 2000: 17.3 -> 16.7.)
struct AnyRaw {             // an element of either type
  bf16_t lo, hi;
  NATSL_DEVICE void load(const void* p, const int dtype, const size_t i) {
    const int size = dtype == NATSL_F32 ? 4 : 2;
    const char* at = reinterpret_cast<const char*>(p) + i * size;
    lo = *reinterpret_cast<const bf16_t*>(at);
    hi = *reinterpret_cast<const bf16_t*>(at + size - 2);
  }
  NATSL_DEVICE float get(const int dtype) const { return __uint_as_float((unsigned)hi << 16 | (dtype == NATSL_F32 ? (unsigned)lo : 0u)); }
};
// A number that crosses from one workgroup to another inside a launch (StepAll): a bf16 and, in the word's lower half, the launch's tag, so that
// it is its own flag.  Written through and read past the reader's L2.
NATSL_DEVICE unsigned tagged(const bf16_t x, const unsigned tag) { return (unsigned)x << 16 | tag; }
NATSL_DEVICE unsigned ld_word(const unsigned* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
struct StepWindow {         // a convolution of width 4 at one channel, every pointer on 8 bytes; x: the new input
  u32x2 e, w;
  bf16_t b, x;
  // (channel d of sequence row `seq`, the same in every lane: offsets of 32 bits a lane on scalar bases)
  // fixed(): what was there before the launch; input(): from the projections, word(): from those of this launch, `late` where it is not there yet.
  NATSL_DEVICE void fixed(const void* state, const void* weight, const void* bias, const unsigned d, const size_t seq) {
    auto at = [](const void* p, const unsigned bytes) __attribute__((always_inline)) -> const char* { return reinterpret_cast<const char*>(p) + bytes; };
    e = *reinterpret_cast<const u32x2*>(at(reinterpret_cast<const u32x2*>(state) + seq, 8u * d));
    w = *reinterpret_cast<const u32x2*>(at(weight, 8u * d));
    b = *reinterpret_cast<const bf16_t*>(at(bias ? bias : weight, 2u * d));
  }
  NATSL_DEVICE void input(const bf16_t* proj, const unsigned d) { x = proj[d]; }
  NATSL_DEVICE void word(const unsigned w, const unsigned tag, unsigned& late) {
    x = (bf16_t)(w >> 16);
    late |= (w & 0xffffu) ^ tag;
  }
  NATSL_DEVICE float next(const bool bias, const bool silu) const {
    float a = bias ? bf16_to_f32(b) : 0.f;
    a += __uint_as_float(w[0] << 16) * __uint_as_float(e[0] & 0xffff0000u);
    a += __uint_as_float(w[0] & 0xffff0000u) * __uint_as_float(e[1] << 16);
    a += __uint_as_float(w[1] << 16) * __uint_as_float(e[1] & 0xffff0000u);
    a += __uint_as_float(w[1] & 0xffff0000u) * bf16_to_f32(x);
    if (silu) a = a / (1.f + __expf(-a));
    return bf16_to_f32(f32_to_bf16(a));
  }
  NATSL_DEVICE void save(void* state, const size_t sd) const {
    reinterpret_cast<u32x2*>(state)[sd] = (u32x2){e[0] >> 16 | e[1] << 16, e[1] >> 16 | (unsigned)x << 16};
  }
};

// Workgroups: one per (sequence, q head), (sequence, k head), (sequence, v head); the rest copy the hidden states.  A thread
// owns a channel (several for v) and walks the step's tokens.
template <int W>
__global__ __launch_bounds__(256) void step_mix_kernel(const StepMix p) {
  const natsl_layer_step& s = p.s;
  __shared__ float red[2][4];
  const int tid = threadIdx.x, b = blockIdx.y, T = s.T, H = s.H, K = s.K, V = s.V;
  const int role = (int)blockIdx.x / H, h = (int)blockIdx.x % H;
  const bool silu = s.flags & NATSL_STEP_SILU, from_conv = s.flags & NATSL_STEP_ATTN_FROM_CONV;
  const size_t cache_row = (size_t)b * s.cache_tokens + (size_t)s.n_kept * s.block + s.n_in;   // of the first new token
  const size_t block_row = (size_t)b * s.block + s.n_in;
  if (role < 2) {
    const bool is_q = role == 0;
    const int KD = H * K, KA = KD / s.HQ, d = h * K + min(tid, K - 1);
    const bool on = tid < K;
    const size_t sd = (size_t)b * KD + d;
    ConvWindow<W> win;
    win.init((const bf16_t*)(is_q ? s.conv_state_q : s.conv_state_k), (const bf16_t*)(is_q ? s.conv_wq : s.conv_wk),
             (const bf16_t*)(is_q ? s.conv_bq : s.conv_bk), d, sd);
    const bool l2 = s.flags & NATSL_STEP_L2_ROWS, norm = s.flags & NATSL_STEP_ATTN_NORM;
    const float nw = norm ? ld_any(is_q ? s.norm_q : s.norm_k, s.norm_dtype, d % KA) : 1.f;
    for (int t = 0; t < T; ++t) {
      const size_t row = (size_t)b * T + t;
      const float x = bf16_to_f32(p.proj[row * p.ldp + (is_q ? p.cq : p.ck) + d]);
      const float y = win.next(x, silu);
      float lin = y, at = from_conv ? y : x;
      if (l2 || norm) {
        float a2 = on ? at * at : 0.f, y2 = on ? y * y : 0.f;
        a2 = wave_sum(a2);
        y2 = wave_sum(y2);
        __syncthreads();                               // the previous token's sums have been read
        if ((tid & 63) == 0) { red[0][tid >> 6] = a2; red[1][tid >> 6] = y2; }
        __syncthreads();
        if (l2) {
          float ss = 0.f;
          for (int w = 0; w < K / 64; ++w) ss += red[1][w];
          lin = y * rsqrtf(ss + s.l2_eps);
        }
        if (norm) {
          float ss = 0.f;
          const int w0 = min(tid, K - 1) / KA * (KA / 64);
          for (int w = 0; w < KA / 64; ++w) ss += red[0][w0 + w];
          at = at * rsqrtf(ss / KA + s.norm_eps) * nw;
        }
      }
      if (on) {
        const bf16_t lb = f32_to_bf16(lin), ab = f32_to_bf16(at);
        if (is_q) {
          p.q_conv[row * KD + d] = f32_to_bf16(y);
          if (l2) p.q_lin[row * KD + d] = lb;
          p.q_attn[row * KD + d] = ab;
        } else {
          ((bf16_t*)s.block_k)[(block_row + t) * KD + d] = lb;
          ((bf16_t*)s.cache_k)[(cache_row + t) * KD + d] = ab;
        }
      }
    }
    if (on) win.save((bf16_t*)(is_q ? s.conv_out_q : s.conv_out_k), sd);
    return;
  }
  if (role == 2) {
    const int VD = H * V;
    const float A = expf(ld_any(s.a_log, s.gate_dtype, h)), bias = ld_any(s.dt_bias, s.gate_dtype, h);
    for (int t = tid; t < T; t += 256) {
      const size_t row = (size_t)b * T + t;
      const float dt = softplus_gate(bf16_to_f32(p.proj[row * p.ldp + p.ca + h]) + bias);
      s.block_g[(block_row + t) * H + h] = -A * dt;
      if (s.is_delta) {
        const float be = bf16_to_f32(p.proj[row * p.ldp + p.cb + h]);
        float sg = bf16_to_f32(f32_to_bf16(sigmoid_gate(be)));
        if (s.flags & NATSL_STEP_NEG_EIGVAL) sg *= 2.f;
        ((bf16_t*)s.block_beta)[(block_row + t) * H + h] = f32_to_bf16(sg);
      }
    }
    if (h == 0)
      for (int i = tid; i < s.HN; i += 256) s.cache_valid[((size_t)b * (s.cache_tokens / s.block) + s.n_kept) * s.HN + i] = 1;
    for (int c = tid; c < V; c += 256) {
      const int d = h * V + c;
      const size_t sd = (size_t)b * VD + d;
      ConvWindow<W> win;
      win.init((const bf16_t*)s.conv_state_v, (const bf16_t*)s.conv_wv, (const bf16_t*)s.conv_bv, d, sd);
      for (int t = 0; t < T; ++t) {
        const size_t row = (size_t)b * T + t;
        const float x = bf16_to_f32(p.proj[row * p.ldp + p.cv + d]);
        const float y = win.next(x, silu);
        float lin = y;
        if (!s.is_delta) lin = y * softplus_gate(bf16_to_f32(p.proj[row * p.ldp + p.ca + h]) + bias);
        ((bf16_t*)s.block_v)[(block_row + t) * VD + d] = f32_to_bf16(lin);
        ((bf16_t*)s.cache_v)[(cache_row + t) * VD + d] = f32_to_bf16(from_conv ? y : x);
      }
      win.save((bf16_t*)s.conv_out_v, sd);
    }
    return;
  }
  const int c = ((int)blockIdx.x - 3 * H) * 256 + tid;
  if (c >= s.D) return;
  for (int t = 0; t < T; ++t) ((bf16_t*)s.block_hidden)[(block_row + t) * s.D + c] = ((const bf16_t*)s.x)[((size_t)b * T + t) * s.D + c];
}

// ---- join, mixing weights, norms, gate: one wave per (row, attention head) ---------------------------------------------
struct StepTail {
  const float* partials; int nsplit;
  const bf16_t *o_lin, *q_conv, *proj, *w_mix;
  const void *w1, *w2; int w_dtype;
  bf16_t* y;
  int rows, HQ, KD, ldp, cg;
  float eps;
};

// the part of one wave: d0, d1 the head's two mixing logits, at the attention's columns CPL*lane.., x1 the linear branch's
template <int VA>
struct TailRow {
  static constexpr int CPL = VA / 64;
  bf16_t gate[CPL];
  AnyRaw w1[CPL], w2[CPL];
  NATSL_DEVICE void load(const StepTail& p, const int row, const int hq, const bool gates = true) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int j = 0; j < CPL; ++j) {
      if (gates) gate[j] = p.proj[(size_t)row * p.ldp + p.cg + hq * VA + CPL * lane + j];
      w1[j].load(p.w1, p.w_dtype, CPL * lane + j);
      w2[j].load(p.w2, p.w_dtype, CPL * lane + j);
    }
  }
  NATSL_DEVICE void finish(const StepTail& p, const int row, const int hq, float d0, float d1, const float* at, const float* x1, unsigned* words = nullptr,
                           unsigned tag = 0) const;
};

template <int VA>
NATSL_DEVICE void TailRow<VA>::finish(const StepTail& p, const int row, const int hq, float d0, float d1, const float* at, const float* x1, unsigned* words,
                               const unsigned tag) const {
  const int lane = threadIdx.x & 63;
  float x2[CPL], sa = 0.f, sb = 0.f;
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    x2[j] = bf16_to_f32(f32_to_bf16(at[j]));
    sa += x1[j] * x1[j];
    sb += x2[j] * x2[j];
  }
  sa = wave_sum(sa);
  sb = wave_sum(sb);
  d0 = bf16_to_f32(f32_to_bf16(wave_sum(d0)));         // (as the projection's output is)
  d1 = bf16_to_f32(f32_to_bf16(wave_sum(d1)));
  mix_softmax(d0, d1);
  const float ra = rsqrtf(sa / VA + p.eps) * d0, rb = rsqrtf(sb / VA + p.eps) * d1;
  const size_t base = ((size_t)row * p.HQ + hq) * VA + CPL * lane;
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    const float mix = x1[j] * ra * w1[j].get(p.w_dtype) + x2[j] * rb * w2[j].get(p.w_dtype), g = bf16_to_f32(gate[j]);
    const bf16_t y = f32_to_bf16(mix * g / (1.f + __expf(-g)));
    if (words) __hip_atomic_store(words + base + j, tagged(y, tag), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else p.y[base + j] = y;
  }
}

template <int VA>
__global__ __launch_bounds__(256) void step_tail_kernel(const StepTail p) {
  constexpr int CPL = VA / 64;
  const int lane = threadIdx.x & 63;
  const int rh = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (rh >= p.rows * p.HQ) return;
  const int row = rh / p.HQ, hq = rh % p.HQ;
  TailRow<VA> out;
  out.load(p, row, hq);
  float d0 = 0.f, d1 = 0.f;                            // the lane's share of the two logits
  for (int i = 8 * lane; i < p.KD; i += 512) {
    const u32x4 qv = *reinterpret_cast<const u32x4*>(p.q_conv + (size_t)row * p.KD + i);
    const u32x4 a = *reinterpret_cast<const u32x4*>(p.w_mix + (size_t)(2 * hq) * p.KD + i);
    const u32x4 c = *reinterpret_cast<const u32x4*>(p.w_mix + (size_t)(2 * hq + 1) * p.KD + i);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float lo = __uint_as_float(qv[j] << 16), hi = __uint_as_float(qv[j] & 0xffff0000u);
      d0 += lo * __uint_as_float(a[j] << 16) + hi * __uint_as_float(a[j] & 0xffff0000u);
      d1 += lo * __uint_as_float(c[j] << 16) + hi * __uint_as_float(c[j] & 0xffff0000u);
    }
  }
  float at[CPL], x1[CPL];
  join_splits<VA>(p.partials + (size_t)rh * p.nsplit * (2 + VA), p.nsplit, at);
#pragma unroll
  for (int j = 0; j < CPL; ++j) x1[j] = bf16_to_f32(p.o_lin[(size_t)rh * VA + CPL * lane + j]);
  out.finish(p, row, hq, d0, d1, at, x1);
}

// ---- one token a sequence: everything between the two products in one launch --------------------------------------------
// For one token the convolutions, norms and gates are a few operations on a few kilobytes, so every wave forms the ones that it
// needs itself, and the tail of a (sequence, head) is done by whichever wave is the last to have written something for it: they
// count themselves in on arrived[], which the projections' launch has cleared.  No wave waits for another.  Bound by round trips to
// memory one behind another (arguments, windows and flags, keys, the count, the others' results); with many keys by their bytes.
// Against the three launches: 340M geometry, one sequence of 800 tokens, 9.6 us for 4.3 + 5.4 + 4.8 and two gaps of 3.5; 16 heads of
// 128/64 and eight sequences of 2000 tokens, 16.7 us for 5 + 13.6 + 5.3 (the three before the changes noted at AnyRaw and wave_sum).  Of the
// 9.6 us: 2.2 until the first keys are asked for, 1.6 - 2.4 for a chunk and the join of the waves, 0.8 to hand a result over and count it,
// 1.4 for the tail, 2 - 3 before and behind the waves.  Workgroups:
//   mixing logits   (sequence, 256 channels of q): their convolution, and their share of all heads' two logits
//   recurrence      (sequence, head, 64 state columns), as in attend_and_recur
//   attention       (sequence, head, split), as in attend_and_recur; the wave with the last chunk makes the new key and value
//                   and writes them to the cache, which nothing else of the launch reads there
// What leaves the launch besides y is written by one wave each: conv_out_q and block_hidden, cache_valid by the logits' waves,
// conv_out_k, block_k, g and beta by the head's first recurrence wave, conv_out_v and block_v by the columns' own.
struct StepOne {
  StepMix m;
  AttnParams a;
  RecurrentParams r;
  StepTail t;
  float *o_lin, *logits;      // [B][H*V] rounded to bf16; [B][n_chunks][HQ][2]
  unsigned* arrived;          // [B][HQ]
  int n_chunks, n_logits, n_rec;
  // with HERE (StepAll): what the launch's parts meet on (StepSync), the projections and the tail's rows as tagged words, like proj and y
  unsigned *sync, *proj_words, *y_words;
  unsigned long long max_wait;
  unsigned long long *started, ticket;   // what the host reads (StepsUnderWay; behind it the last one that failed), and what the launch leaves there
};
constexpr int LOGIT_CHUNK = 256;

// Everything that the wave handed over (stores that write through) has arrived before the lane with `on` counts it in.  What orders the two
// is this machine, not the language: the atomics are relaxed, s_waitcnt vmcnt(0) holds the count back until every lane's
// write-through store has been acknowledged by the memory that all XCDs see, the empty asm statements keep the compiler from moving
// accesses across, and the last arriver's loads (ld_agent) go past its own L2.  Release and acquire would write back and drop whole L2s.
// The returned mask has the lanes that were their counter's last.
NATSL_DEVICE unsigned long long arrive(const StepOne& p, const int b, const int hq, const bool on, const int expected) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  unsigned before = 0u;
  if (on) before = __hip_atomic_fetch_add(p.arrived + (size_t)b * p.a.HQ + hq, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const unsigned long long last = __ballot(on && before + 1u == (unsigned)expected);
  asm volatile("" ::: "memory");
  return last;
}

// What the parts of a launch with the products in it (HERE) meet on, in lines of their own.  Zeros at first; a launch leaves the epoch, which its
// words' tags come from, one higher, and everything else as it was, but FAILED when it did.
struct StepSync {
  static constexpr int LINE = 32, LEFT = 0, FAILED = LINE, EPOCH = 2 * LINE, STARTED = 3 * LINE, ARRIVED = 4 * LINE;
};
static_assert(StepSync::FAILED == NATSL_STEP_SYNC_FAILED, "what the header says");
NATSL_DEVICE unsigned step_tag(const StepOne& p) { return (ld_word(p.sync + StepSync::EPOCH) + 1u) & 0xffffu; }

// Until ask(), which requests words, finds that none of any lane's is late, or the time is over: then the step has failed, its outputs become
// NaN, and every wave still ends.  The workgroups that a wave waits for come before its own in the grid, and wait for nothing or for others before
// them; each XCD starts its share of the grid in order.  So a launch always ends next to others that do: of what an XCD has not started, the first
// is waited for by none that would have to end before it.  Two launches that have not started all of their workgroups can keep each other's
// out, one on this XCD and the other on that, unless both fit: see step_may_wait and StepsUnderWay.
template <class Ask>
NATSL_DEVICE void wait_for(const StepOne& p, Ask ask) {
  if (!__ballot(ask() != 0u)) return;
  const unsigned long long since = __builtin_amdgcn_s_memrealtime();
  for (unsigned n = 1;; ++n) {
    __builtin_amdgcn_s_sleep(2);
    if (!__ballot(ask() != 0u)) return;
    if (n % 64u == 0u && ld_word(p.sync + StepSync::FAILED)) return;
    if (__builtin_amdgcn_s_memrealtime() - since > p.max_wait) {
      if ((threadIdx.x & 63) == 0) __hip_atomic_store(p.sync + StepSync::FAILED, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // (seen before whatever the wave makes of what it has: see arrive())
      if ((threadIdx.x & 63) == 0) __hip_atomic_store(p.started + 1, p.ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      return;
    }
  }
}

template <int VA, bool HERE>
NATSL_DEVICE void step_tail(const StepOne& p, const int b, const int hq) {
  constexpr int CPL = VA / 64;
  const int lane = threadIdx.x & 63;
  const size_t rh = (size_t)b * p.a.HQ + hq;
  TailRow<VA> out;
  out.load(p.t, b, hq, !HERE);
  unsigned tag = 0;
  if constexpr (HERE) tag = step_tag(p);
  float at[CPL], x1[CPL];
#pragma unroll
  for (int j = 0; j < CPL; ++j) x1[j] = ld_agent(p.o_lin + rh * VA + CPL * lane + j);
  const float* lg = p.logits + (((size_t)b * p.n_chunks + min(lane, p.n_chunks - 1)) * p.a.HQ + hq) * 2;
  const float d0 = ld_agent(lg), d1 = ld_agent(lg + 1);
  join_splits<VA, true>(p.a.partials + rh * p.a.nsplit * (2 + VA), p.a.nsplit, at);
  if constexpr (HERE) {
    const unsigned* gates = p.proj_words + (size_t)b * p.t.ldp + p.t.cg + hq * VA + CPL * lane;
    wait_for(p, [&]() __attribute__((always_inline)) {
      unsigned late = 0;
#pragma unroll
      for (int j = 0; j < CPL; ++j) {
        const unsigned w = ld_word(gates + j);
        out.gate[j] = (bf16_t)(w >> 16);
        late |= (w & 0xffffu) ^ tag;
      }
      return late;
    });
  }
  out.finish(p.t, b, hq, lane < p.n_chunks ? d0 : 0.f, lane < p.n_chunks ? d1 : 0.f, at, x1, HERE ? p.y_words : nullptr, tag);
}

template <int VA, bool HERE>
NATSL_DEVICE void step_logits(const StepOne& p, const int b, const int chunk, const int expected) {
  __shared__ __align__(16) bf16_t qs[LOGIT_CHUNK];
  const natsl_layer_step& s = p.m.s;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int KD = s.H * s.K, d = LOGIT_CHUNK * chunk + tid;
  constexpr int U = 4;                                  // four channels a lane, waves over the heads, four heads' rows in flight
  const int c = LOGIT_CHUNK * chunk + 4 * lane;
  const bf16_t* w = p.t.w_mix + min(c, KD - 4);
  u32x2 r[2 * U];
  auto load = [&](const int h0) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 2 * U; ++u) r[u] = *reinterpret_cast<const u32x2*>(w + (size_t)(2 * min(h0 + 4 * (u >> 1), s.HQ - 1) + (u & 1)) * KD);
  };
  const size_t sd = (size_t)b * KD;
  StepWindow win;
  win.fixed(s.conv_state_q, s.conv_wq, s.conv_bq, min(d, KD - 1), sd);
  load(wave);
  if constexpr (HERE) {
    const unsigned tag = step_tag(p);
    const unsigned* w = p.proj_words + (size_t)b * p.m.ldp + p.m.cq + min(d, KD - 1);
    wait_for(p, [&]() __attribute__((always_inline)) {
      unsigned late = 0;
      win.word(ld_word(w), tag, late);
      return late;
    });
  } else {
    win.input(p.m.proj + (size_t)b * p.m.ldp + p.m.cq, min(d, KD - 1));
  }
  const bf16_t y = f32_to_bf16(win.next(s.conv_bq != nullptr, s.flags & NATSL_STEP_SILU));
  if (d < KD) win.save(s.conv_out_q, sd + d);
  qs[tid] = d < KD ? y : (bf16_t)0;
  if (s.block_hidden) {
    const bf16_t* x = (const bf16_t*)s.x + (size_t)b * s.D;
    bf16_t* to = (bf16_t*)s.block_hidden + ((size_t)b * s.block + s.n_in) * s.D;
    for (int i = d; i < s.D; i += LOGIT_CHUNK * p.n_chunks) to[i] = x[i];
  }
  if (chunk == 0)
    for (int i = tid; i < s.HN; i += 256) s.cache_valid[((size_t)b * (s.cache_tokens / s.block) + s.n_kept) * s.HN + i] = 1;
  __syncthreads();
  const u32x2 qv = *reinterpret_cast<const u32x2*>(qs + 4 * lane);
  const float q0 = __uint_as_float(qv[0] << 16), q1 = __uint_as_float(qv[0] & 0xffff0000u), q2 = __uint_as_float(qv[1] << 16),
              q3 = __uint_as_float(qv[1] & 0xffff0000u);
  float* dst = p.logits + ((size_t)b * p.n_chunks + chunk) * s.HQ * 2;
  for (int h0 = wave; h0 < s.HQ; h0 += 4 * U) {
    if (h0 != wave) load(h0);
#pragma unroll
    for (int u = 0; u < 2 * U; ++u) {
      float x = q0 * __uint_as_float(r[u][0] << 16) + q1 * __uint_as_float(r[u][0] & 0xffff0000u) + q2 * __uint_as_float(r[u][1] << 16) +
                q3 * __uint_as_float(r[u][1] & 0xffff0000u);
      x = wave_sum(c < KD ? x : 0.f);
      const int h = h0 + 4 * (u >> 1);
      if (lane == 0 && h < s.HQ) st_agent(dst + 2 * h + (u & 1), x);
    }
  }
  for (int h0 = wave; h0 < s.HQ; h0 += 256) {           // lane i counts in for the wave's i-th head
    const int h = h0 + 4 * lane;
    for (unsigned long long last = arrive(p, b, h, h < s.HQ, expected); last; last &= last - 1) step_tail<VA, HERE>(p, b, h0 + 4 * __builtin_ctzll(last));
  }
}

// The recurrence's token: q and k of the head go through the wave's own piece of LDS, the rest stays in registers.
template <int DK, bool HERE>
struct StepToken {
  const StepOne& p;
  bf16_t* rows;               // [2][DK], this wave's
  const bool first;           // the head's first wave
  const int expected, VA;
  bool last = false;          // whether this wave is the one to do the tail
  template <bool DELTA>
  NATSL_DEVICE void token(const RecurrentParams& r, const int n, int, const int h, const int kq, const int vc, float* kk, float* qq, float& gt,
                          float& bt, float& vt) const {
    constexpr int R = DK / 4, C = DK / 64;
    const natsl_layer_step& s = p.m.s;
    const int lane = threadIdx.x & 63, KD = s.H * DK, VD = s.H * s.V;
    const bool silu = s.flags & NATSL_STEP_SILU;
    const bf16_t* proj = p.m.proj + (size_t)n * p.m.ldp;
    const size_t block_row = (size_t)n * s.block + s.n_in;
    StepWindow wq[C], wk[C], wv;
    float xq[C], xk[C];
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int d = h * DK + 64 * i + lane;
      wq[i].fixed(s.conv_state_q, s.conv_wq, s.conv_bq, d, (size_t)n * KD);
      wk[i].fixed(s.conv_state_k, s.conv_wk, s.conv_bk, d, (size_t)n * KD);
    }
    const int dv = h * s.V + vc;
    wv.fixed(s.conv_state_v, s.conv_wv, s.conv_bv, dv, (size_t)n * VD);
    AnyRaw a_log, dt_bias;
    a_log.load(s.a_log, s.gate_dtype, h);
    dt_bias.load(s.dt_bias, s.gate_dtype, h);
    bf16_t xa, xb = 0;
    if constexpr (HERE) {
      const unsigned tag = step_tag(p);
      const unsigned* w = p.proj_words + (size_t)n * p.m.ldp;
      wait_for(p, [&]() __attribute__((always_inline)) {
        unsigned late = 0, words[2 * C + 3];
#pragma unroll
        for (int i = 0; i < C; ++i) {
          words[2 * i] = ld_word(w + p.m.cq + h * DK + 64 * i + lane);
          words[2 * i + 1] = ld_word(w + p.m.ck + h * DK + 64 * i + lane);
        }
        words[2 * C] = ld_word(w + p.m.cv + dv);
        words[2 * C + 1] = ld_word(w + p.m.ca + h);
        words[2 * C + 2] = ld_word(w + (DELTA ? p.m.cb : p.m.ca) + h);
#pragma unroll
        for (int i = 0; i < C; ++i) {
          wq[i].word(words[2 * i], tag, late);
          wk[i].word(words[2 * i + 1], tag, late);
        }
        wv.word(words[2 * C], tag, late);
        xa = (bf16_t)(words[2 * C + 1] >> 16);
        if (DELTA) xb = (bf16_t)(words[2 * C + 2] >> 16);
        return late | ((words[2 * C + 1] & 0xffffu) ^ tag) | ((words[2 * C + 2] & 0xffffu) ^ tag);
      });
    } else {
#pragma unroll
      for (int i = 0; i < C; ++i) {
        wq[i].input(proj + p.m.cq, h * DK + 64 * i + lane);
        wk[i].input(proj + p.m.ck, h * DK + 64 * i + lane);
      }
      wv.input(proj + p.m.cv, dv);
      xa = proj[p.m.ca + h];
      if (DELTA) xb = proj[p.m.cb + h];
    }
    const float A = expf(a_log.get(s.gate_dtype));
    const float dt = softplus_gate(bf16_to_f32(xa) + dt_bias.get(s.gate_dtype));
    gt = -A * dt;
    bt = 1.f;
    if (DELTA) {
      float sg = bf16_to_f32(f32_to_bf16(sigmoid_gate(bf16_to_f32(xb))));
      if (s.flags & NATSL_STEP_NEG_EIGVAL) sg *= 2.f;
      bt = bf16_to_f32(f32_to_bf16(sg));
    }
    float ssq = 0.f, ssk = 0.f;
    const bool l2 = s.flags & NATSL_STEP_L2_ROWS;
#pragma unroll
    for (int i = 0; i < C; ++i) {
      xq[i] = wq[i].next(s.conv_bq != nullptr, silu);
      xk[i] = wk[i].next(s.conv_bk != nullptr, silu);
      if (l2) {
        ssq += wave_sum(xq[i] * xq[i]);
        ssk += wave_sum(xk[i] * xk[i]);
      }
    }
    const float rq = l2 ? rsqrtf(ssq + s.l2_eps) : 1.f, rk = l2 ? rsqrtf(ssk + s.l2_eps) : 1.f;
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const bf16_t kb = f32_to_bf16(xk[i] * rk);
      rows[64 * i + lane] = f32_to_bf16(xq[i] * rq);
      rows[DK + 64 * i + lane] = kb;
      if (first) {
        const int d = h * DK + 64 * i + lane;
        ((bf16_t*)s.block_k)[block_row * KD + d] = kb;
        wk[i].save(s.conv_out_k, (size_t)n * KD + d);
      }
    }
    if (first && lane == 0) {
      s.block_g[block_row * s.H + h] = gt;
      if (DELTA) ((bf16_t*)s.block_beta)[block_row * s.H + h] = f32_to_bf16(bt);
    }
    float y = wv.next(s.conv_bv != nullptr, silu);
    if (!DELTA) y = bf16_to_f32(f32_to_bf16(y * dt));
    vt = y;
    if (kq == 0) {
      ((bf16_t*)s.block_v)[block_row * VD + dv] = f32_to_bf16(y);
      wv.save(s.conv_out_v, (size_t)n * VD + dv);
    }
    __builtin_amdgcn_wave_barrier();
    ld_row<R>(rows, NATSL_BF16, true, kq * R, qq);
    ld_row<R>(rows + DK, NATSL_BF16, true, kq * R, kk);
  }
  NATSL_DEVICE void out(const RecurrentParams& r, const int n, int, const int h, const int vc, const float x) const {
    st_agent(p.o_lin + ((size_t)n * r.H + h) * r.V + vc, bf16_to_f32(f32_to_bf16(x)));
  }
  NATSL_DEVICE void done(const int n, const int h, const int vc) {   // (counted in before the states' stores are waited for)
    last = arrive(p, n, (h * p.m.s.V + vc) / VA, (threadIdx.x & 63) == 0, expected) != 0;
  }
};

// One head's row of the attention view of q, k or v (N channels), 64 i + lane in a lane: requested, then formed.
template <int N>
struct StepRow {
  static constexpr int C = N / 64;
  StepWindow win[C];
  AnyRaw nw[C];
  NATSL_DEVICE void request(const natsl_layer_step& s, const void* state, const void* weight, const void* bias, const void* norm, const size_t seq,
                            const int d0) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < C; ++i) {
      win[i].fixed(state, weight, bias, d0 + 64 * i + lane, seq);
      nw[i].load(norm ? norm : weight, s.norm_dtype, 64 * i + lane);
    }
  }
  NATSL_DEVICE void input(const bf16_t* proj, const int d0) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int i = 0; i < C; ++i) win[i].input(proj, d0 + 64 * i + lane);
  }
  NATSL_DEVICE void words(const unsigned* proj, const int d0, const unsigned tag, unsigned& late) {
    const int lane = threadIdx.x & 63;
    unsigned w[C];
#pragma unroll
    for (int i = 0; i < C; ++i) w[i] = ld_word(proj + d0 + 64 * i + lane);
#pragma unroll
    for (int i = 0; i < C; ++i) win[i].word(w[i], tag, late);
  }
  NATSL_DEVICE void form(const natsl_layer_step& s, const bool bias, const bool norm, bf16_t* dst, bf16_t* also) const {
    const int lane = threadIdx.x & 63;
    float x[C], ss = 0.f, r = 1.f;
    AnyRaw m[C];
#pragma unroll
    for (int i = 0; i < C; ++i) {
      // (a row is formed once, but inside a loop: without this the conversions move in front of it, and their waits with them)
      StepWindow c = win[i];
      m[i].lo = nw[i].lo;
      m[i].hi = nw[i].hi;
      asm volatile("" : "+v"(c.x), "+v"(c.b), "+v"(c.e), "+v"(c.w), "+v"(m[i].lo), "+v"(m[i].hi));
      x[i] = s.flags & NATSL_STEP_ATTN_FROM_CONV ? c.next(bias, s.flags & NATSL_STEP_SILU) : bf16_to_f32(c.x);
    }
    if (norm) {
#pragma unroll
      for (int i = 0; i < C; ++i) ss += wave_sum(x[i] * x[i]);
      r = rsqrtf(ss / N + s.norm_eps);
    }
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const bf16_t y = f32_to_bf16(norm ? x[i] * r * m[i].get(s.norm_dtype) : x[i]);
      dst[64 * i + lane] = y;
      if (also) also[64 * i + lane] = y;
    }
  }
};

// What an attending wave of the step makes itself: its query, and in the wave with the last chunk (`mine`) the new key and value.  All
// inputs are requested (request()) before the first chunk is, and used when that is on its way.
template <int KA, int VA, bool HERE>
struct StepKeys {
  static constexpr bool STEP = true;
  const StepOne& p;
  bf16_t *q, *k, *v;             // LDS
  const int b, hq, first;        // first: the new key's index
  const bool mine;
  bool done = false;
  StepRow<KA> rq, rk;
  StepRow<VA> rv;
  NATSL_DEVICE StepKeys(const StepOne& p, bf16_t* q, bf16_t* k, bf16_t* v, const int b, const int hq, const bool mine)
      : p(p), q(q), k(k), v(v), b(b), hq(hq), first(p.a.TK - 1), mine(mine) {}
  NATSL_DEVICE void request() {
    const natsl_layer_step& s = p.m.s;
    const size_t KD = (size_t)s.H * s.K, VD = (size_t)s.H * s.V;
    const bool norm = s.flags & NATSL_STEP_ATTN_NORM;
    rq.request(s, s.conv_state_q, s.conv_wq, s.conv_bq, norm ? s.norm_q : nullptr, b * KD, hq * KA);
    if (mine) {
      rk.request(s, s.conv_state_k, s.conv_wk, s.conv_bk, norm ? s.norm_k : nullptr, b * KD, hq * KA);
      rv.request(s, s.conv_state_v, s.conv_wv, s.conv_bv, nullptr, b * VD, hq * VA);
    }
    if constexpr (!HERE) {
      const bf16_t* proj = p.m.proj + (size_t)b * p.m.ldp;
      rq.input(proj + p.m.cq, hq * KA);
      if (mine) {
        rk.input(proj + p.m.ck, hq * KA);
        rv.input(proj + p.m.cv, hq * VA);
      }
    }
  }
  NATSL_DEVICE void ready(AttnRow<KA, VA, false>& row) {
    if (done) return;
    done = true;
    if constexpr (HERE) {        // (the first chunk's keys are on their way by now)
      const unsigned tag = step_tag(p);
      const unsigned* w = p.proj_words + (size_t)b * p.m.ldp;
      wait_for(p, [&]() __attribute__((always_inline)) {
        unsigned late = 0;
        rq.words(w + p.m.cq, hq * KA, tag, late);
        if (mine) {
          rk.words(w + p.m.ck, hq * KA, tag, late);
          rv.words(w + p.m.cv, hq * VA, tag, late);
        }
        return late;
      });
    }
    const natsl_layer_step& s = p.m.s;
    const bool norm = s.flags & NATSL_STEP_ATTN_NORM;
    rq.form(s, s.conv_bq != nullptr, norm, q, nullptr);
    if (mine) {
      const size_t at = ((size_t)b * s.cache_tokens + first) * s.HQ + hq;
      rk.form(s, s.conv_bk != nullptr, norm, k, (bf16_t*)s.cache_k + at * KA);
      rv.form(s, s.conv_bv != nullptr, false, v, (bf16_t*)s.cache_v + at * VA);
    }
    __builtin_amdgcn_wave_barrier();
    row.query(q, 0, p.a.scale_log2);
  }
};

// The launch's only argument.  Read through a pointer that the optimiser cannot see through, so that each role loads the fields that it
// needs where it needs them: as a plain argument the roles' fields are all loaded at the kernel's start and spill (70 scalar registers).
NATSL_DEVICE const StepOne& step_one_args() {
  typedef __attribute__((address_space(4))) const StepOne* arg_ptr;
  unsigned long long at = (unsigned long long)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(at));
  return *(const StepOne*)(arg_ptr)at;
}

// The roles of the workgroups between the products; id: which of them
template <int KA, int VA, int K, bool DELTA, bool HERE>
NATSL_DEVICE void step_roles(const StepOne& p, int id) {
  __shared__ __align__(16) bf16_t rows[4][2 * K > KA ? 2 * K : KA], own_k[KA], own_v[VA];
  const natsl_layer_step& s = p.m.s;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int expected = p.a.nsplit + VA / 16 + p.n_chunks;
  int b, hq;
  if (id < p.n_logits) {
    step_logits<VA, HERE>(p, id / p.n_chunks, id % p.n_chunks, expected);
    return;
  }
  id -= p.n_logits;
  if (id < p.n_rec) {
    const int per = (s.V + 63) / 64, col16 = (id % per) * 4 + wave, nh = id / per;
    if (col16 * 16 >= s.V) return;
    StepToken<K, HERE> token{p, rows[wave], col16 == 0, expected, VA};
    recurrent_columns<K, DELTA>(p.r, nh, col16, token);
    if (!token.last) return;
    b = nh / s.H;
    hq = (nh % s.H * s.V + 16 * col16) / VA;
  } else {
    id -= p.n_rec;
    const int split = id % p.a.nsplit;
    hq = id / p.a.nsplit % s.HQ;
    b = id / p.a.nsplit / s.HQ;
    const bool mine = (p.a.TK - 1) / KEYS_PER_CHUNK % (4 * p.a.nsplit) == 4 * split + wave;
    attend<KA, VA, false, 4>(p.a, b, 0, hq, split, StepKeys<KA, VA, HERE>(p, rows[wave], own_k, own_v, b, hq, mine));
    if (wave != 0 || !arrive(p, b, hq, lane == 0, expected)) return;
  }
  step_tail<VA, HERE>(p, b, hq);
}

template <int KA, int VA, int K, bool DELTA>
__global__ __launch_bounds__(256) void step_one_kernel(const StepOne) {
  step_roles<KA, VA, K, DELTA, false>(step_one_args(), blockIdx.x);
}

// ---- ... and the products in the same launch ----------------------------------------------------------------------------
// One sequence's step is bound by the host, which takes 22 us for a token and its three launches (18 of kernels, each of which begins with a trip
// to memory for its arguments and one for its first operands).  Here the workgroups of the projections come first, those between the products
// ask for windows, states and keys before they wait for them, and those of the output projection hold their weights when the rows come.
// What crosses is words that are their own flags: counters behind the stores cost two trips more at each crossing, and with a few hundred
// waves looking at the same ones far more (340M geometry 20.5 us, 760M 30).  A token with its host work, one sequence of 777: 340M geometry 22.1 ->
// 15.9 us, 760M 22.4 -> 17.3, 16 heads of 128/64 21.9 -> 15.5; four of 500 (340M) 27.4 -> 23.1.
// The sums are those of rows_gemm_kernel, in its order: a wave is two of its eight (accumulators 0 and 1).
struct StepAll {
  StepOne one;
  RowsGemm in, out;
  int in_tiles, out_tiles;
};
constexpr int STEP_ROWS = 8192;       // numbers of the rows that a workgroup of the output projection keeps: 16 KiB

NATSL_DEVICE const StepAll& step_all_args() {
  typedef __attribute__((address_space(4))) const StepAll* arg_ptr;
  unsigned long long at = (unsigned long long)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(at));
  return *(const StepAll*)(arg_ptr)at;
}

// One tile of 16 weight rows; OUT: of the output projection, behind everything else, else of the projections in front.  U: steps of 32 that a
// wave has on their way at once.
template <bool OUT, int U>
NATSL_DEVICE void step_product(const StepAll& all, const int tile) {
  extern __shared__ __align__(16) bf16_t step_rows[];   // OUT: [M][D]
  __shared__ f32x4 red[8][64];
  const RowsGemm& p = OUT ? all.out : all.in;
  const StepOne& one = all.one;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int si = 0;
  if constexpr (!OUT) {
#pragma unroll
    for (int i = 1; i < GEMM_SEGS; ++i) si = i < p.n_seg && tile >= p.seg[i].tile0 ? i : si;
  }
  const GemmSeg sg = p.seg[si];
  const int n0 = 16 * (tile - sg.tile0), r16 = lane & 15, kg = lane >> 4, steps = p.D / 32;
  const bf16_t* wp = sg.w + (size_t)min(n0 + r16, sg.rows - 1) * p.D + 8 * kg;
  const size_t x_at = (size_t)min(r16, p.M - 1) * p.D + 8 * kg;
  f32x4 acc[2] = {(f32x4){0.f, 0.f, 0.f, 0.f}, (f32x4){0.f, 0.f, 0.f, 0.f}};
  unsigned tag = 0;
  for (int s0 = wave; s0 < steps; s0 += 4 * U) {
    bf16x8 a[U], b[U];
#pragma unroll
    for (int u = 0; u < U; ++u) a[u] = ld8(wp + 32 * min(s0 + 4 * u, steps - 1));
    if constexpr (OUT) {
      // (these workgroups are the grid's last on every XCD, and have time until the rows come: told at the launch's end, a token took 1.7 us more)
      if (s0 == 0 && lane == 0 && __hip_atomic_fetch_add(one.sync + StepSync::STARTED, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u == (unsigned)all.out_tiles) {
        __hip_atomic_store(one.sync + StepSync::STARTED, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(one.started, one.ticket, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
      // the rows go through LDS: a thread brings its share of their words, two at a time
      if (s0 == wave) {
        constexpr int N = 8;
        const auto* y = reinterpret_cast<const unsigned long long*>(one.y_words);
        unsigned* to = reinterpret_cast<unsigned*>(step_rows);
        const int pairs = p.M * p.D / 2;
        tag = step_tag(one);
        for (int i0 = threadIdx.x; i0 < pairs; i0 += 256 * N) {
          unsigned long long w[N];
          wait_for(one, [&]() __attribute__((always_inline)) {
            unsigned late = 0;
#pragma unroll
            for (int j = 0; j < N; ++j) w[j] = __hip_atomic_load(y + min(i0 + 256 * j, pairs - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int j = 0; j < N; ++j) late |= (((unsigned)w[j] & 0xffffu) ^ tag) | (((unsigned)(w[j] >> 32) & 0xffffu) ^ tag);
            return late;
          });
#pragma unroll
          for (int j = 0; j < N; ++j)
            if (i0 + 256 * j < pairs) to[i0 + 256 * j] = __builtin_amdgcn_perm((unsigned)(w[j] >> 32), (unsigned)w[j], 0x07060302);
        }
        __syncthreads();
      }
    } else {
      if (s0 == wave) tag = step_tag(one);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) b[u] = OUT ? *reinterpret_cast<const bf16x8*>(step_rows + x_at + 32 * min(s0 + 4 * u, steps - 1)) : ld8(p.x + x_at + 32 * min(s0 + 4 * u, steps - 1));
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s0 + 4 * u < steps) acc[u & 1] = mfma16(a[u], b[u], acc[u & 1]);
  }
  red[wave][lane] = acc[0];
  red[wave + 4][lane] = acc[1];
  __syncthreads();
  if (wave != 0) return;
  f32x4 sum = red[0][lane];
#pragma unroll
  for (int w = 1; w < 8; ++w) sum += red[w][lane];
  const int n = n0 + 4 * kg;
  if constexpr (!OUT) {
    if (r16 < p.M) {
      unsigned* dst = one.proj_words + (size_t)r16 * p.ldo + sg.col0 + n;    // (a row's tiles are whole in the words)
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        const unsigned long long lo = tagged(f32_to_bf16(sum[j]), tag), hi = tagged(f32_to_bf16(sum[j + 1]), tag);
        __hip_atomic_store(reinterpret_cast<unsigned long long*>(dst + j), lo | hi << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    return;
  }
  unsigned left = 0u;
  if (lane == 0) left = __hip_atomic_fetch_add(one.sync + StepSync::LEFT, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // (a step that has failed leaves no numbers)
  if (ld_word(one.sync + StepSync::FAILED)) sum = (f32x4){NAN, NAN, NAN, NAN};
  if (r16 < p.M) {
    bf16_t* dst = p.out + (size_t)r16 * p.ldo + n;
    if (n + 4 <= sg.rows) {
      *reinterpret_cast<u32x2*>(dst) = (u32x2){pack_bf16x2(sum[0], sum[1]), pack_bf16x2(sum[2], sum[3])};
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (n + j < sg.rows) dst[j] = f32_to_bf16(sum[j]);
    }
  }
  if (__builtin_amdgcn_readfirstlane(left) + 1u == (unsigned)all.out_tiles) {       // all tails are written: nobody counts or looks any more
    for (int i = lane; i < one.m.s.B * one.a.HQ; i += 64) __hip_atomic_store(one.arrived + i, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (lane == 0) {
      __hip_atomic_store(one.sync + StepSync::LEFT, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(one.sync + StepSync::EPOCH, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// (as many workgroups a CU as step_one_kernel's registers allow: the splits count on them.  For that the delta rule with 128-wide linear keys, other than on
// 128/128 heads, keeps 4 vector registers of a lane (20 bytes) in scratch; the other forms none.)
template <int KA, int VA, int K, bool DELTA>
__global__ __launch_bounds__(256, K == 192 || KA + VA == 256 ? 2 : KA + VA + K == 192 ? 4 : 3) void step_all_kernel(const StepAll) {
  const StepAll& all = step_all_args();
  constexpr int U = K == 192 ? 18 : KA + VA + K == 192 ? 8 : 12;
  int id = blockIdx.x;
  if (id < all.in_tiles) return step_product<false, 12>(all, id);
  id -= all.in_tiles;
  const int roles = (int)gridDim.x - all.in_tiles - all.out_tiles;
  if (id < roles) step_roles<KA, VA, K, DELTA, true>(all.one, id);
  else step_product<true, U>(all, id - roles);
}

// all: the products of the launch, or null where they are launches of their own
static int launch_step_one(const char* what, const StepOne& p, const StepAll* all, const int K, const int KA, const int VA, hipStream_t st) {
  const natsl_layer_step& s = p.m.s;
  const unsigned roles = (unsigned)(p.n_logits + p.n_rec + s.B * s.HQ * p.a.nsplit), grid = all ? all->in_tiles + roles + all->out_tiles : roles;
  const size_t rows = all ? (size_t)s.B * s.H * s.V * sizeof(bf16_t) : 0;
#define NATSL_S1(KK, VV, KL, DD)                                                                            \
  if (KA == KK && VA == VV && K == KL && (s.is_delta != 0) == DD) {                                         \
    if (all) hipLaunchKernelGGL((step_all_kernel<KK, VV, KL, DD>), dim3(grid), dim3(256), rows, st, *all);  \
    else hipLaunchKernelGGL((step_one_kernel<KK, VV, KL, DD>), dim3(grid), dim3(256), 0, st, p);            \
    return check_launch(what);                                                                              \
  }
#define NATSL_S3(KK, VV)                                                                                                     \
  NATSL_S1(KK, VV, 64, true) NATSL_S1(KK, VV, 128, true) NATSL_S1(KK, VV, 192, true) NATSL_S1(KK, VV, 64, false)             \
  NATSL_S1(KK, VV, 128, false) NATSL_S1(KK, VV, 192, false)
  NATSL_S3(64, 64) NATSL_S3(64, 128) NATSL_S3(128, 64) NATSL_S3(128, 128)
#undef NATSL_S3
#undef NATSL_S1
  return fail(NATSL_ERR_UNSUPPORTED, "%s: head dims %d (linear), %d / %d (attention) not built", what, K, KA, VA);
}

struct StepLayout {
  int ldp, cq, ck, cv, cg, ca, cb, tiles, nsplit, n_chunks;
  bool one;
  bool all;                   // ... and the products can be in it
  size_t proj, q_conv, q_lin, q_attn, o_lin, y, partials, logits, arrived, bytes;
  size_t proj_words, y_words, sync_bytes;   // in the caller's memory behind StepSync
};

// Workgroups of step_one_kernel that fit on the chip at once, less those of the logits and the recurrence: what its registers allow a CU
// (236 with 192-wide states: two; 104 with 64-wide everything: four; else 129 - 168: three.  128-wide keys and values are counted as two, which
// the splits below were measured with).
static int step_one_per_cu(const natsl_layer_step& s) {
  const int KA = s.H * s.K / s.HQ, VA = s.H * s.V / s.HQ;
  return s.K == 192 || KA + VA == 256 ? 2 : KA + VA + s.K == 192 ? 4 : 3;
}
static int step_one_slots(const natsl_layer_step& s, const int n_chunks) {
  return step_one_per_cu(s) * 256 - s.B * (n_chunks + s.H * cdiv(s.V, 64));
}

// Workgroups that wait when the products are in the launch too: those between the products and those behind them.  At most half of what fits on
// the chip, so that those of two launches (of two processes: StepsUnderWay) leave room for one that is waited for, and no more than this: with 268 of the
// 340M geometry (four sequences of 500 tokens) a token is 0.87 of the three launches' time, with 304 and 352 of 16 heads of 128/64 (six of 300, four of
// 1200) 1.02, where the host is no longer what a step waits for.
constexpr int STEP_WAITERS = 280;
static bool step_may_wait(const natsl_layer_step& s, const int n_chunks, const int nsplit, const int cus) {
  const int n = s.B * (n_chunks + s.H * cdiv(s.V, 64) + s.HQ * nsplit) + cdiv(s.D, 16);
  return n <= STEP_WAITERS && 2 * n <= step_one_per_cu(s) * cus;
}

// The launches whose workgroups wait for each other, by device: of a process's, one at a time has workgroups that have not started, or several of one
// stream, which follow one another.  Steps on another stream (of another cache: another thread's, another request's) are several launches, which wait for
// nothing, until the last has started all of its workgroups, which it writes into pinned memory that the host looks at; so are those that are
// captured, whose replays nobody counts.  Held from the look to the launch, so that tickets are in the order of their launches.
struct StepsUnderWay {
  std::mutex mu;
  unsigned long long issued = 0;
  std::atomic<unsigned long long*> words{nullptr};   // the last launch that has started, the last that gave up
  hipStream_t on = nullptr;
  std::atomic<int> cus{0};
};
static StepsUnderWay steps_of[64];
static StepsUnderWay* steps_under_way() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
  StepsUnderWay& u = steps_of[dev];
  if (u.cus.load(std::memory_order_relaxed) == 0 && hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess)
    u.cus.store(n, std::memory_order_relaxed);
  return &u;
}
// The next launch's ticket, or 0: not now.
static unsigned long long step_ticket(StepsUnderWay& u, hipStream_t st) {
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &capturing) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  if (capturing != hipStreamCaptureStatusNone) return 0;
  unsigned long long* words = u.words.load(std::memory_order_relaxed);
  if (!words) {
    void* p = nullptr;
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;                // (another thread may be capturing: this is none of its graph's)
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    const hipError_t e = hipHostMalloc(&p, 64, hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent);    // one line a device, for as long as the process lives
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      return 0;
    }
    words = static_cast<unsigned long long*>(p);
    __atomic_store_n(words, 0ull, __ATOMIC_RELAXED);
    __atomic_store_n(words + 1, 0ull, __ATOMIC_RELAXED);
    u.words.store(words, std::memory_order_release);
  }
  // (every thread's own default stream has the same name)
  if ((st != u.on || st == hipStreamPerThread) && __atomic_load_n(words, __ATOMIC_ACQUIRE) < u.issued) return 0;
  u.on = st;
  return ++u.issued;
}

// One token a sequence: one launch between the two products.  That kernel is built for the layers' own convolution width and reads windows
// and mixing rows 8 bytes at a time; a wave's lanes are its chunks of logits.  With 128-wide attention values and more logits and
// recurrence workgroups than fit at once the several launches are faster (340M geometry from 29 sequences, 760M from 13: mostly 0.89 - 1.0
// of the time that the one launch takes at its best split, 1.09 at most, up to 64 sequences of 600 to 5000 cached tokens); with 64-wide
// values the one launch is (0.89 - 1.0 of theirs, up to 64 sequences).
static bool step_is_one(const natsl_layer_step& s, const int n_chunks) {
  if (s.H * s.V == 128 * s.HQ && step_one_slots(s, n_chunks) < 0) return false;
  const uintptr_t at8 = (uintptr_t)s.conv_state_q | (uintptr_t)s.conv_state_k | (uintptr_t)s.conv_state_v | (uintptr_t)s.conv_out_q |
                        (uintptr_t)s.conv_out_k | (uintptr_t)s.conv_out_v | (uintptr_t)s.conv_wq | (uintptr_t)s.conv_wk | (uintptr_t)s.conv_wv |
                        (uintptr_t)s.w_mix;
  return s.T == 1 && s.conv_width == 4 && n_chunks <= 64 && at8 % 8 == 0;
}

// As many splits as leave all of the launch's workgroups resident at once, of 256 keys or more (two chunks a wave: 760M, one sequence,
// 1333 tokens: a step of 24.5 us with 6 - 8 splits, 33 with 11).  Where that leaves fewer than four there is no one round to keep, and
// what counts is that a wave walks few chunks one after the other: up to five splits of 768 keys (a step of 16 sequences of the 340M
// geometry with 5421 cached tokens: 91 us with one split, 83 with five; 32 of the Mamba geometry with 3113: 129 and 113; five rather
// than four or eight, which spread the heads worse over the XCDs).  Over seven geometries, 1 - 64 sequences and 400 - 10000 cached
// tokens a step takes 1.015 times the best split's (geometric mean; 1.14 at most).
static int step_one_splits(const natsl_layer_step& s, const int n_chunks) {
  const int keys = s.n_kept * s.block + s.n_in + s.T, queries = s.B * s.HQ;
  const int one_round = std::min({attend_splits(queries, keys), cdiv(keys, 256), step_one_slots(s, n_chunks) / queries});
  return one_round >= 4 ? one_round : std::max({1, one_round, std::min(5, cdiv(keys, 768))});
}

static StepLayout step_layout(const natsl_layer_step& s) {
  StepLayout l;
  const int KD = s.H * s.K, VD = s.H * s.V, M = s.B * s.T;
  auto up16 = [](int x) { return (x + 15) / 16 * 16; };
  l.cq = 0; l.ck = l.cq + up16(KD); l.cv = l.ck + up16(KD); l.cg = l.cv + up16(VD); l.ca = l.cg + up16(VD);
  l.cb = l.ca + up16(s.H);
  l.ldp = l.cb + (s.is_delta ? up16(s.H) : 0);
  l.tiles = l.ldp / 16;
  l.n_chunks = cdiv(KD, LOGIT_CHUNK);
  l.one = step_is_one(s, l.n_chunks);
  l.nsplit = l.one ? step_one_splits(s, l.n_chunks) : attend_splits(M * s.HQ, s.n_kept * s.block + s.n_in + s.T);
  size_t at = 0;
  auto take = [&](size_t n) { const size_t r = at; at += (n + 255) / 256 * 256; return r; };
  l.proj = take((size_t)M * l.ldp * 2);
  l.q_conv = take((size_t)M * KD * 2);
  l.q_lin = s.flags & NATSL_STEP_L2_ROWS ? take((size_t)M * KD * 2) : l.q_conv;
  l.q_attn = take((size_t)M * KD * 2);
  l.o_lin = take((size_t)M * VD * 4);
  l.y = take((size_t)M * VD * 2);
  l.partials = take((size_t)M * s.HQ * ATTEND_MAX_SPLITS * (2 + VD / s.HQ) * 4);   // (the size does not follow the cache's)
  l.logits = take((size_t)M * l.n_chunks * s.HQ * 2 * 4);
  l.arrived = take((size_t)M * s.HQ * 4);
  l.bytes = at;
  // The products in the launch: a row tile of tokens, whose rows fit the output projection's workgroups (each of its waves has a part of a row), and
  // no more workgroups that wait than may, and some of the last ones on each of eight XCDs (StepSync::STARTED); whether they do at this step's number of
  // keys, and on this device, is step_fwd's to see, so that a cache's steps all want the same memory.
  l.all = l.one && M <= 16 && M * VD <= STEP_ROWS && VD >= 128 && s.D >= 128 && step_may_wait(s, l.n_chunks, 1, 256);
  at = 0;
  take((StepSync::ARRIVED + (size_t)M * s.HQ) * 4);
  l.proj_words = take((size_t)M * l.ldp * 4);
  l.y_words = take((size_t)M * VD * 4);
  l.sync_bytes = l.all ? at : 0;
  return l;
}

static int step_check(const natsl_layer_step& s, const char* what) {
  if (s.B <= 0 || s.T <= 0 || s.D <= 0 || s.H <= 0 || s.K <= 0 || s.V <= 0 || s.HQ <= 0 || s.HN <= 0 || s.block <= 0)
    return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  const int KD = s.H * s.K, VD = s.H * s.V;
  if ((long long)s.B * s.T > STEP_MAX_ROWS) return fail(NATSL_ERR_UNSUPPORTED, "%s: at most %d new tokens in all", what, STEP_MAX_ROWS);
  if (s.n_in < 0 || s.n_in + s.T > s.block) return fail(NATSL_ERR_INVALID, "%s: the new tokens must stay inside the selector block", what);
  if (s.n_kept < 0 || s.block % 64 || s.cache_tokens % s.block || (long long)s.n_kept * s.block + s.n_in + s.T > s.cache_tokens)
    return fail(NATSL_ERR_INVALID, "%s: the cache does not hold the new tokens", what);
  if (s.HQ % s.H || s.HQ % s.HN || s.H % s.HN) return fail(NATSL_ERR_UNSUPPORTED, "%s: head counts %d / %d / %d", what, s.HQ, s.H, s.HN);
  const int KA = KD / s.HQ, VA = VD / s.HQ;
  if ((s.K != 64 && s.K != 128 && s.K != 192) || (KA != 64 && KA != 128) || (VA != 64 && VA != 128) || s.K % KA)
    return fail(NATSL_ERR_UNSUPPORTED, "%s: head dims %d (linear), %d / %d (attention) not built", what, s.K, KA, VA);
  if (s.V % 16 || s.D % 32 || VD % 32 || s.conv_width < 2 || s.conv_width > 4) return fail(NATSL_ERR_UNSUPPORTED, "%s: widths", what);
  return NATSL_OK;
}

}  // namespace natsl

using namespace natsl;

extern "C" size_t natsl_layer_step_workspace_bytes(const natsl_layer_step* step) {
  return step && step_check(*step, "natsl_layer_step") == NATSL_OK ? step_layout(*step).bytes : 0;
}

static int step_fwd(const char* what, const natsl_layer_step* step, void* workspace, size_t workspace_bytes, unsigned* sync, size_t sync_bytes,
                    unsigned long long max_wait_us, natsl_stream_t stream) {
  if (!step || !workspace) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  const natsl_layer_step& s = *step;
  int rc = step_check(s, what);
  if (rc != NATSL_OK) return rc;
  if (!s.x || !s.wq || !s.wk || !s.wv || !s.wg || !s.wa || (s.is_delta && !s.wb) || !s.w_mix || !s.wo || !s.conv_wq || !s.conv_wk || !s.conv_wv ||
      !s.a_log || !s.dt_bias || !s.out_norm1 || !s.out_norm2 || ((s.flags & NATSL_STEP_ATTN_NORM) && (!s.norm_q || !s.norm_k)) ||
      !s.conv_state_q || !s.conv_state_k || !s.conv_state_v || !s.conv_out_q || !s.conv_out_k || !s.conv_out_v || !s.state || !s.block_start ||
      !s.state_out || !s.cache_k || !s.cache_v || !s.cache_valid || !s.block_k || !s.block_v || !s.block_g || (s.is_delta && !s.block_beta) || !s.out ||
      (s.n_in + s.T == s.block && !s.types))
    return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  const StepLayout l = step_layout(s);
  if (workspace_bytes < l.bytes) return fail(NATSL_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", what, l.bytes, workspace_bytes);
  const size_t sync_needed = std::max(l.sync_bytes, (size_t)StepSync::ARRIVED * 4);
  if (sync && ((uintptr_t)sync % 8 || sync_bytes < sync_needed))
    return fail(NATSL_ERR_INVALID, "%s: %zu bytes of the step's own memory needed, %zu given", what, sync_needed, sync_bytes);
  const int KD = s.H * s.K, VD = s.H * s.V, KA = KD / s.HQ, VA = VD / s.HQ, M = s.B * s.T;
  const int out_tiles = cdiv(s.D, 16);
  StepsUnderWay* const under_way = sync && l.all ? steps_under_way() : nullptr;
  std::unique_lock<std::mutex> turn;
  unsigned long long ticket = 0;
  if (under_way && step_may_wait(s, l.n_chunks, l.nsplit, under_way->cus.load(std::memory_order_relaxed))) {
    turn = std::unique_lock<std::mutex>(under_way->mu);
    if ((ticket = step_ticket(*under_way, reinterpret_cast<hipStream_t>(stream))) == 0) turn.unlock();
  }
  const bool in_one = ticket != 0;
  char* ws = reinterpret_cast<char*>(workspace);
  bf16_t *proj = (bf16_t*)(ws + l.proj), *q_conv = (bf16_t*)(ws + l.q_conv), *q_lin = (bf16_t*)(ws + l.q_lin), *q_attn = (bf16_t*)(ws + l.q_attn),
         *o_lin = (bf16_t*)(ws + l.o_lin), *y = (bf16_t*)(ws + l.y);
  float* partials = (float*)(ws + l.partials);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);

  auto gemm = [&](const RowsGemm& g, int tiles) {
    auto kernel = g.failed ? (M <= 16 ? rows_gemm_kernel<1, true> : M <= 32 ? rows_gemm_kernel<2, true> : rows_gemm_kernel<4, true>)
                           : (M <= 16 ? rows_gemm_kernel<1, false> : M <= 32 ? rows_gemm_kernel<2, false> : rows_gemm_kernel<4, false>);
    hipLaunchKernelGGL(kernel, dim3(tiles), dim3(512), 0, st, g);
    return check_launch(what);
  };
  RowsGemm g;
  g.x = (const bf16_t*)s.x; g.out = proj; g.M = M; g.D = s.D; g.ldo = l.ldp;
  const GemmSeg segs[GEMM_SEGS] = {{(const bf16_t*)s.wq, KD, 0, l.cq}, {(const bf16_t*)s.wk, KD, 0, l.ck}, {(const bf16_t*)s.wv, VD, 0, l.cv},
                                   {(const bf16_t*)s.wg, VD, 0, l.cg}, {(const bf16_t*)s.wa, s.H, 0, l.ca}, {(const bf16_t*)s.wb, s.H, 0, l.cb}};
  g.n_seg = s.is_delta ? 6 : 5; g.failed = nullptr;
  unsigned* arrived = in_one ? sync + StepSync::ARRIVED : (unsigned*)(ws + l.arrived);
  g.zero = arrived; g.n_zero = l.one && !in_one ? M * s.HQ : 0;
  for (int i = 0; i < GEMM_SEGS; ++i) {
    g.seg[i] = segs[i];
    g.seg[i].tile0 = segs[i].col0 / 16;
  }
  if (!in_one && (rc = gemm(g, l.tiles)) != NATSL_OK) return rc;

  StepMix m;
  m.s = s; m.proj = proj; m.ldp = l.ldp; m.cq = l.cq; m.ck = l.ck; m.cv = l.cv; m.ca = l.ca; m.cb = l.cb;
  m.q_conv = q_conv; m.q_lin = q_lin; m.q_attn = q_attn;
  AttnParams a;
  a.q = q_attn; a.k = s.cache_k; a.v = s.cache_v; a.mask = nullptr; a.o = nullptr;
  a.B = s.B; a.TQ = s.T; a.TK = s.n_kept * s.block + s.n_in + s.T; a.HQ = a.HKV = s.HQ; a.HM = s.HN; a.dtype = NATSL_BF16;
  a.scale_log2 = s.scale_attn * 1.4426950408889634f;
  a.nsplit = l.nsplit; a.partials = partials;
  a.k_bs = (size_t)s.cache_tokens * KD; a.v_bs = (size_t)s.cache_tokens * VD;
  a.valid = s.cache_valid; a.valid_bs = s.cache_tokens / s.block * s.HN; a.n_kept = s.n_kept; a.block = s.block; a.n_in = s.n_in;
  a.own_visible = (s.flags & NATSL_STEP_ATTN_OWN_BLOCK) != 0;
  RecurrentParams r;
  r.q = q_lin; r.k = s.block_k; r.v = s.block_v; r.g = s.block_g; r.g_cumsum = s.g_cumsum; r.beta = s.block_beta;
  r.h0 = s.state; r.hcur = s.block_start; r.o = o_lin; r.ht = s.state_out;
  r.types = s.types; r.types_dtype = s.types_dtype; r.n_in_block = nullptr; r.n_in_block_scalar = s.n_in;
  r.N = s.B; r.T = s.T; r.H = s.H; r.HN = s.HN; r.V = s.V; r.block = s.block; r.dtype = NATSL_BF16; r.scale = s.scale_linear;
  r.decay = (s.flags & NATSL_STEP_DECAY) != 0; r.l2norm = s.is_delta; r.query_only = 0;
  r.kv_stride = s.block; r.kv_first = s.n_in; r.fresh_start = (s.flags & NATSL_STEP_FRESH_START) != 0; r.aligned = 1;
  r.g_cumsum_out = s.g_cumsum_out;
  StepTail t;
  t.partials = partials; t.nsplit = l.nsplit; t.o_lin = o_lin; t.q_conv = q_conv; t.proj = proj; t.w_mix = (const bf16_t*)s.w_mix;
  t.w1 = s.out_norm1; t.w2 = s.out_norm2; t.w_dtype = s.out_norm_dtype; t.y = y; t.rows = M; t.HQ = s.HQ; t.KD = KD; t.ldp = l.ldp; t.cg = l.cg;
  t.eps = s.out_norm_eps;
  RowsGemm o;
  o.x = y; o.out = (bf16_t*)s.out; o.M = M; o.D = VD; o.ldo = s.D; o.n_seg = 1; o.zero = nullptr; o.n_zero = 0;
  o.failed = sync ? sync + StepSync::FAILED : nullptr;    // (what a failed step left in the cache is nothing to go on from, in however many launches)
  for (int i = 0; i < GEMM_SEGS; ++i) o.seg[i] = {(const bf16_t*)s.wo, s.D, 0, 0};
  if (l.one) {
    StepOne f;
    f.m = m; f.a = a; f.r = r; f.t = t;
    f.o_lin = (float*)(ws + l.o_lin); f.logits = (float*)(ws + l.logits); f.arrived = arrived;
    f.n_chunks = l.n_chunks; f.n_logits = s.B * l.n_chunks; f.n_rec = s.B * s.H * cdiv(s.V, 64);
    if (in_one) {
      char* mem = reinterpret_cast<char*>(sync);
      f.sync = sync; f.proj_words = reinterpret_cast<unsigned*>(mem + l.proj_words); f.y_words = reinterpret_cast<unsigned*>(mem + l.y_words);
      f.started = under_way->words.load(std::memory_order_relaxed); f.ticket = ticket;
      f.max_wait = 100 * max_wait_us;                     // (the counter behind s_memrealtime runs at 100 MHz)
      const StepAll all = {f, g, o, l.tiles, out_tiles};
      return launch_step_one(what, f, &all, s.K, KA, VA, st);
    }
    if ((rc = launch_step_one(what, f, nullptr, s.K, KA, VA, st)) != NATSL_OK) return rc;
    return gemm(o, out_tiles);
  }

  const dim3 mgrid(3 * s.H + (s.block_hidden ? cdiv(s.D, 256) : 0), s.B);
  if (s.conv_width == 4) hipLaunchKernelGGL((step_mix_kernel<4>), mgrid, dim3(256), 0, st, m);
  else if (s.conv_width == 3) hipLaunchKernelGGL((step_mix_kernel<3>), mgrid, dim3(256), 0, st, m);
  else hipLaunchKernelGGL((step_mix_kernel<2>), mgrid, dim3(256), 0, st, m);
  if ((rc = check_launch(what)) != NATSL_OK) return rc;
  if ((rc = launch_attend_and_recur(what, a, r, s.is_delta != 0, s.K, KA, VA, st)) != NATSL_OK) return rc;

  const dim3 tgrid(cdiv(M * s.HQ, 4));
  if (VA == 128) hipLaunchKernelGGL((step_tail_kernel<128>), tgrid, dim3(256), 0, st, t);
  else hipLaunchKernelGGL((step_tail_kernel<64>), tgrid, dim3(256), 0, st, t);
  if ((rc = check_launch(what)) != NATSL_OK) return rc;
  return gemm(o, cdiv(s.D, 16));
}

extern "C" int natsl_layer_step_fwd(const natsl_layer_step* step, void* workspace, size_t workspace_bytes, natsl_stream_t stream) {
  return step_fwd("natsl_layer_step_fwd", step, workspace, workspace_bytes, nullptr, 0, 0, stream);
}

extern "C" size_t natsl_layer_step_sync_bytes(const natsl_layer_step* step) {
  return step && step_check(*step, "natsl_layer_step") == NATSL_OK ? step_layout(*step).sync_bytes : 0;
}

extern "C" int natsl_layer_step_sync_fwd(const natsl_layer_step* step, void* workspace, size_t workspace_bytes, void* shared, size_t shared_bytes,
                                         uint64_t max_wait_us, natsl_stream_t stream) {
  return step_fwd("natsl_layer_step_sync_fwd", step, workspace, workspace_bytes, reinterpret_cast<unsigned*>(shared), shared_bytes, max_wait_us, stream);
}

extern "C" uint64_t natsl_layer_step_gave_up(int device) {
  const unsigned long long* words = device >= 0 && device < 64 ? steps_of[device].words.load(std::memory_order_acquire) : nullptr;
  return words ? __atomic_load_n(words + 1, __ATOMIC_ACQUIRE) : 0;
}
