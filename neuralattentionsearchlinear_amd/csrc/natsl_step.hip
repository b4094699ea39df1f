// A generation step of a whole hybrid layer: a few new tokens of each cached sequence, from the hidden states to the layer's
// output, in five launches.  At this size a step is bound by launches and by the host that issues them (the same step as
// separate operations was 40 launches, 0.2 ms of kernels and 0.57 ms of host time for one 340M-geometry layer), so each kernel
// takes as much of the step as its data dependences allow:
//   rows_gemm_kernel     q, k, v, gate, a (and beta) projections as one pass over all their weights; the output projection
//   step_mix_kernel      short convolutions, activations, row norms, gates; the new rows of every cache, written in place
//   attend_and_recur     attention over the cached keys next to the token recurrence (natsl_decode.hip)
//   step_tail_kernel     join of the attention's splits, mixing weights, two-input norm and gate
// Roundings to bf16 are where the layer's separate operations round (projections, convolutions, norms, gates, branch outputs).
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
};

template <int MT>
__global__ __launch_bounds__(512) void rows_gemm_kernel(const RowsGemm p) {
  constexpr int NW = 8, U = 4;
  __shared__ f32x4 red[NW][MT][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
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
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          a2 += __shfl_xor(a2, o);
          y2 += __shfl_xor(y2, o);
        }
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

template <int VA>
__global__ __launch_bounds__(256) void step_tail_kernel(const StepTail p) {
  constexpr int CPL = VA / 64;
  const int lane = threadIdx.x & 63;
  const int rh = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (rh >= p.rows * p.HQ) return;
  const int row = rh / p.HQ, hq = rh % p.HQ;
  // the head's two mixing logits (rounded to bf16 as the projection's output is), their softmax
  float d0 = 0.f, d1 = 0.f;
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
  float at[CPL];
  join_splits<VA>(p.partials + (size_t)rh * p.nsplit * (2 + VA), p.nsplit, at);
  float x1[CPL], x2[CPL], sa = 0.f, sb = 0.f;
  const size_t base = (size_t)rh * VA + CPL * lane;
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    x1[j] = bf16_to_f32(p.o_lin[base + j]);
    x2[j] = bf16_to_f32(f32_to_bf16(at[j]));
    sa += x1[j] * x1[j];
    sb += x2[j] * x2[j];
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    d0 += __shfl_xor(d0, o);
    d1 += __shfl_xor(d1, o);
    sa += __shfl_xor(sa, o);
    sb += __shfl_xor(sb, o);
  }
  d0 = bf16_to_f32(f32_to_bf16(d0));
  d1 = bf16_to_f32(f32_to_bf16(d1));
  mix_softmax(d0, d1);
  const float ra = rsqrtf(sa / VA + p.eps) * d0, rb = rsqrtf(sb / VA + p.eps) * d1;
#pragma unroll
  for (int j = 0; j < CPL; ++j) {
    const float g = bf16_to_f32(p.proj[(size_t)row * p.ldp + p.cg + hq * VA + CPL * lane + j]);
    const float mix = x1[j] * ra * ld_any(p.w1, p.w_dtype, CPL * lane + j) + x2[j] * rb * ld_any(p.w2, p.w_dtype, CPL * lane + j);
    p.y[base + j] = f32_to_bf16(mix * g / (1.f + __expf(-g)));
  }
}

struct StepLayout {
  int ldp, cq, ck, cv, cg, ca, cb, tiles, nsplit;
  size_t proj, q_conv, q_lin, q_attn, o_lin, y, partials, bytes;
};

static StepLayout step_layout(const natsl_layer_step& s) {
  StepLayout l;
  const int KD = s.H * s.K, VD = s.H * s.V, M = s.B * s.T;
  auto up16 = [](int x) { return (x + 15) / 16 * 16; };
  l.cq = 0; l.ck = l.cq + up16(KD); l.cv = l.ck + up16(KD); l.cg = l.cv + up16(VD); l.ca = l.cg + up16(VD);
  l.cb = l.ca + up16(s.H);
  l.ldp = l.cb + (s.is_delta ? up16(s.H) : 0);
  l.tiles = l.ldp / 16;
  l.nsplit = attend_splits(M * s.HQ, s.n_kept * s.block + s.n_in + s.T);
  size_t at = 0;
  auto take = [&](size_t n) { const size_t r = at; at += (n + 255) / 256 * 256; return r; };
  l.proj = take((size_t)M * l.ldp * 2);
  l.q_conv = take((size_t)M * KD * 2);
  l.q_lin = s.flags & NATSL_STEP_L2_ROWS ? take((size_t)M * KD * 2) : l.q_conv;
  l.q_attn = take((size_t)M * KD * 2);
  l.o_lin = take((size_t)M * VD * 2);
  l.y = take((size_t)M * VD * 2);
  l.partials = take((size_t)M * s.HQ * ATTEND_MAX_SPLITS * (2 + VD / s.HQ) * 4);   // (the size does not follow the cache's)
  l.bytes = at;
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

extern "C" int natsl_layer_step_fwd(const natsl_layer_step* step, void* workspace, size_t workspace_bytes, natsl_stream_t stream) {
  const char* what = "natsl_layer_step_fwd";
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
  const int KD = s.H * s.K, VD = s.H * s.V, KA = KD / s.HQ, VA = VD / s.HQ, M = s.B * s.T;
  char* ws = reinterpret_cast<char*>(workspace);
  bf16_t *proj = (bf16_t*)(ws + l.proj), *q_conv = (bf16_t*)(ws + l.q_conv), *q_lin = (bf16_t*)(ws + l.q_lin), *q_attn = (bf16_t*)(ws + l.q_attn),
         *o_lin = (bf16_t*)(ws + l.o_lin), *y = (bf16_t*)(ws + l.y);
  float* partials = (float*)(ws + l.partials);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);

  auto gemm = [&](const RowsGemm& g, int tiles) {
    if (M <= 16) hipLaunchKernelGGL((rows_gemm_kernel<1>), dim3(tiles), dim3(512), 0, st, g);
    else if (M <= 32) hipLaunchKernelGGL((rows_gemm_kernel<2>), dim3(tiles), dim3(512), 0, st, g);
    else hipLaunchKernelGGL((rows_gemm_kernel<4>), dim3(tiles), dim3(512), 0, st, g);
    return check_launch(what);
  };
  RowsGemm g;
  g.x = (const bf16_t*)s.x; g.out = proj; g.M = M; g.D = s.D; g.ldo = l.ldp;
  const GemmSeg segs[GEMM_SEGS] = {{(const bf16_t*)s.wq, KD, 0, l.cq}, {(const bf16_t*)s.wk, KD, 0, l.ck}, {(const bf16_t*)s.wv, VD, 0, l.cv},
                                   {(const bf16_t*)s.wg, VD, 0, l.cg}, {(const bf16_t*)s.wa, s.H, 0, l.ca}, {(const bf16_t*)s.wb, s.H, 0, l.cb}};
  g.n_seg = s.is_delta ? 6 : 5;
  for (int i = 0; i < GEMM_SEGS; ++i) {
    g.seg[i] = segs[i];
    g.seg[i].tile0 = segs[i].col0 / 16;
  }
  if ((rc = gemm(g, l.tiles)) != NATSL_OK) return rc;

  StepMix m;
  m.s = s; m.proj = proj; m.ldp = l.ldp; m.cq = l.cq; m.ck = l.ck; m.cv = l.cv; m.ca = l.ca; m.cb = l.cb;
  m.q_conv = q_conv; m.q_lin = q_lin; m.q_attn = q_attn;
  const dim3 mgrid(3 * s.H + (s.block_hidden ? cdiv(s.D, 256) : 0), s.B);
  if (s.conv_width == 4) hipLaunchKernelGGL((step_mix_kernel<4>), mgrid, dim3(256), 0, st, m);
  else if (s.conv_width == 3) hipLaunchKernelGGL((step_mix_kernel<3>), mgrid, dim3(256), 0, st, m);
  else hipLaunchKernelGGL((step_mix_kernel<2>), mgrid, dim3(256), 0, st, m);
  if ((rc = check_launch(what)) != NATSL_OK) return rc;

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
  if ((rc = launch_attend_and_recur(what, a, r, s.is_delta != 0, s.K, KA, VA, st)) != NATSL_OK) return rc;

  StepTail t;
  t.partials = partials; t.nsplit = l.nsplit; t.o_lin = o_lin; t.q_conv = q_conv; t.proj = proj; t.w_mix = (const bf16_t*)s.w_mix;
  t.w1 = s.out_norm1; t.w2 = s.out_norm2; t.w_dtype = s.out_norm_dtype; t.y = y; t.rows = M; t.HQ = s.HQ; t.KD = KD; t.ldp = l.ldp; t.cg = l.cg;
  t.eps = s.out_norm_eps;
  const dim3 tgrid(cdiv(M * s.HQ, 4));
  if (VA == 128) hipLaunchKernelGGL((step_tail_kernel<128>), tgrid, dim3(256), 0, st, t);
  else hipLaunchKernelGGL((step_tail_kernel<64>), tgrid, dim3(256), 0, st, t);
  if ((rc = check_launch(what)) != NATSL_OK) return rc;

  RowsGemm o;
  o.x = y; o.out = (bf16_t*)s.out; o.M = M; o.D = VD; o.ldo = s.D; o.n_seg = 1;
  for (int i = 0; i < GEMM_SEGS; ++i) o.seg[i] = {(const bf16_t*)s.wo, s.D, 0, 0};
  return gemm(o, cdiv(s.D, 16));
}
