// The front of the hybrid layers around their projections: short convolutions with the row norms that follow them, the gates, the
// input gradient's first terms, and the selector's straight-through gradient.  All of it is bound by HBM traffic (and, for short
// inputs, by launches), so what touches the same rows is one pass and q, k, v share a launch:
//   conv_norm_kernel      y = act(conv(x)) and, per head, rms(y) w, l2(y) or y times a number: one read, two writes
//   conv_norm_bwd_kernel  the gradients that meet at y (linear branch, mixing logits, through the norm or the number) are added in registers, then
//                         the convolution's backward; weight sums per run of tokens, added up in a fixed order afterwards
//   gates_kernel          g = -exp(A_log) softplus(a + dt_bias), beta = sigmoid(b) (GDN) / dt (Mamba), and its backward
//   dx_init_kernel        block mean's gradient spread over its tokens + the narrow projections' share of dx: what the four wide
//                         products then accumulate onto
#include <type_traits>

#include "natsl_device.h"
#include "natsl_host.h"

namespace natsl {

NATSL_DEVICE float ldf(const void* p, int dtype, size_t i) {
  return dtype == NATSL_F32 ? reinterpret_cast<const float*>(p)[i] : bf16_to_f32(reinterpret_cast<const bf16_t*>(p)[i]);
}
NATSL_DEVICE void stf(void* p, int dtype, size_t i, float x) {
  if (dtype == NATSL_F32) reinterpret_cast<float*>(p)[i] = x;
  else reinterpret_cast<bf16_t*>(p)[i] = f32_to_bf16(x);
}
NATSL_DEVICE void up8(const u32x4 w, float* f) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f[2 * j] = __uint_as_float(w[j] << 16);
    f[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
  }
}
NATSL_DEVICE u32x4 down8(const float* f) {
  u32x4 w;
#pragma unroll
  for (int j = 0; j < 4; ++j) w[j] = pack_bf16x2(f[2 * j], f[2 * j + 1]);
  return w;
}
NATSL_DEVICE const u32x4* row8(const void* p, const size_t elem) { return reinterpret_cast<const u32x4*>(reinterpret_cast<const bf16_t*>(p) + elem); }

// CH adjacent channels as they lie in memory, and as fp32
template <int CH> struct Piece;
template <> struct Piece<8> {
  typedef u32x4 type;
  static NATSL_DEVICE type at(const void* p, const size_t elem) { return *row8(p, elem); }
  static NATSL_DEVICE void up(const type w, float* f) { up8(w, f); }
  static NATSL_DEVICE type down(const float* f) { return down8(f); }
};
template <> struct Piece<4> {
  typedef u32x2 type;
  static NATSL_DEVICE type at(const void* p, const size_t elem) { return *reinterpret_cast<const u32x2*>(reinterpret_cast<const bf16_t*>(p) + elem); }
  static NATSL_DEVICE void up(const type w, float* f) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      f[2 * j] = __uint_as_float(w[j] << 16);
      f[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
    }
  }
  static NATSL_DEVICE type down(const float* f) { return (u32x2){pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3])}; }
};

struct ConvNormParams {
  natsl_conv_seg seg[NATSL_CONV_SEGS];
  int first[NATSL_CONV_SEGS + 1];     // the segments' first workgroups
  int n_seg, B, T, run, silu, norm_dtype, ch;   // ch: channels of a thread
  float* part[NATSL_CONV_SEGS];        // backward: [run id][W+2][D] sums (taps, bias, norm weight)
};

NATSL_DEVICE int conv_segment(const ConvNormParams& p) {
  int s = 0;
#pragma unroll
  for (int i = 1; i < NATSL_CONV_SEGS; ++i) s = i < p.n_seg && (int)blockIdx.x >= p.first[i] ? i : s;
  return s;
}

// A thread owns 8 adjacent channels for a run of consecutive tokens and slides the last W-1 rows through registers; eight rows
// are requested before the first is used.  The lanes of a head's row are adjacent, so its norm is a few lane shuffles.
template <int W>
__global__ __launch_bounds__(256) void conv_norm_kernel(const ConvNormParams p) {
  const int si = conv_segment(p);
  const natsl_conv_seg& s = p.seg[si];
  const int D = s.D, T = p.T, groups = D / 8, runs = (T + p.run - 1) / p.run;
  const long long gid = (long long)((int)blockIdx.x - p.first[si]) * 256 + threadIdx.x;
  if (gid >= (long long)p.B * runs * groups) return;
  const int cg = (int)(gid % groups), r = (int)((gid / groups) % runs), b = (int)(gid / ((long long)groups * runs));
  const int d0 = 8 * cg, t0 = r * p.run, t1 = min(T, t0 + p.run);
  const bf16_t* w = reinterpret_cast<const bf16_t*>(s.weight);
  const bf16_t* st = reinterpret_cast<const bf16_t*>(s.state);
  float wt[W][8], bs[8], win[W][8], nw[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) {
#pragma unroll
    for (int j = 0; j < W; ++j) wt[j][c] = bf16_to_f32(w[(size_t)(d0 + c) * W + j]);
    bs[c] = s.bias ? bf16_to_f32(reinterpret_cast<const bf16_t*>(s.bias)[d0 + c]) : 0.f;
    nw[c] = s.norm_weight ? ldf(s.norm_weight, p.norm_dtype, (d0 + c) % (8 * s.norm_lanes)) : 1.f;
  }
  const size_t base = (size_t)b * T * D + d0;
#pragma unroll
  for (int j = 0; j < W - 1; ++j) {
    const int q = t0 - (W - 1) + j;
    if (q >= 0) {
      up8(*row8(s.x, base + (size_t)q * D), win[j]);
    } else {
#pragma unroll
      for (int c = 0; c < 8; ++c) win[j][c] = st ? bf16_to_f32(st[((size_t)b * D + d0 + c) * W + (W + q)]) : 0.f;
    }
  }
  if (s.state_out && r == runs - 1) {
    bf16_t* so = reinterpret_cast<bf16_t*>(s.state_out);
#pragma unroll
    for (int j = 0; j < W; ++j) {
      const int q = T - W + j;
      float e[8];
      if (q >= 0) {
        up8(*row8(s.x, base + (size_t)q * D), e);
      } else {
#pragma unroll
        for (int c = 0; c < 8; ++c) e[c] = st ? bf16_to_f32(st[((size_t)b * D + d0 + c) * W + (W + q)]) : 0.f;
      }
#pragma unroll
      for (int c = 0; c < 8; ++c) so[((size_t)b * D + d0 + c) * W + j] = f32_to_bf16(e[c]);
    }
  }
  auto number = [&](const int t) __attribute__((always_inline)) { return s.scale ? s.scale[((size_t)b * T + t) * (groups / s.norm_lanes) + cg / s.norm_lanes] : 0.f; };
  auto one_row = [&](const u32x4 in, const float num, const int t) __attribute__((always_inline)) {
    float y[8], ss = 0.f, none = 0.f;
    up8(in, win[W - 1]);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      float acc = bs[c];
#pragma unroll
      for (int j = 0; j < W; ++j) acc += wt[j][c] * win[j][c];
      y[c] = p.silu ? acc / (1.f + __expf(-acc)) : acc;
    }
    const u32x4 packed = down8(y);
    const size_t at = base + (size_t)t * D;
    if (s.y) *reinterpret_cast<u32x4*>(reinterpret_cast<bf16_t*>(s.y) + at) = packed;
    if (s.y_norm) {
      up8(packed, y);
      float rs = num;
      if (!s.scale) {                                   // (nw is one where it is)
#pragma unroll
        for (int c = 0; c < 8; ++c) ss += y[c] * y[c];
        group_sum2(ss, none, s.norm_lanes);
        rs = rsqrtf((s.norm_l2 ? ss : ss / (8 * s.norm_lanes)) + s.norm_eps);
      }
#pragma unroll
      for (int c = 0; c < 8; ++c) y[c] *= rs * nw[c];
      *reinterpret_cast<u32x4*>(reinterpret_cast<bf16_t*>(s.y_norm) + at) = down8(y);
    }
#pragma unroll
    for (int j = 0; j < W - 1; ++j)
#pragma unroll
      for (int c = 0; c < 8; ++c) win[j][c] = win[j + 1][c];
  };
  constexpr int AHEAD = 8;
  int tb = t0;
  for (; tb + AHEAD <= t1; tb += AHEAD) {   // (no way out between a batch's loads and their use: they all go out together)
    u32x4 rows[AHEAD];
    float num[AHEAD];
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) {
      rows[a] = *row8(s.x, base + (size_t)(tb + a) * D);
      num[a] = number(tb + a);
    }
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) one_row(rows[a], num[a], tb + a);
  }
  for (; tb < t1; ++tb) one_row(*row8(s.x, base + (size_t)tb * D), number(tb), tb);
}

// Backward: dy = dy_a + dy_b + (backward of the norm, or of the number, of dy_norm), then dpre = dy act'(pre), dx[s] = sum_i w[W-1-i] dpre[s+i] +
// dx_add[s], dw[j] = sum dpre[t] x[t-(W-1)+j].  pre and y are recomputed from x; a few rows of every input are requested at a time.  A thread
// reads W-1 rows past its run (for dx of the run's last tokens) without adding them to its sums.
// Bound by vector issue and the bytes alike (340M geometry 0.86 GB, a Mamba layer 1.48 GB at 8 x 4096): 215 -> 199 and 475 -> 385 us, 760M 2 x 3000
// 76 -> 63, against a branch around every channel's activation, the head sums through LDS, dx_add requested where it is used and eight channels a
// thread.  The activation's division is eight per cent of that (189, 357 and 58 with the hardware's reciprocal, which is off by an ulp).  Four
// channels with two rows ahead 4 - 5 % slower, with four 10 - 24 % (175 registers: two waves a SIMD).
// A thread has CH channels: four (eight hold 229 - 262 registers, two waves a SIMD or one), eight for heads of 512, which have to fit a wave.
template <int W, bool SILU, int CH>
__global__ __launch_bounds__(256) void conv_norm_bwd_kernel(const ConvNormParams p) {
  typedef Piece<CH> Pc;
  const int si = conv_segment(p);
  const natsl_conv_seg& s = p.seg[si];
  const int D = s.D, T = p.T, groups = D / CH, runs = (T + p.run - 1) / p.run;
  const long long gid = (long long)((int)blockIdx.x - p.first[si]) * 256 + threadIdx.x;
  if (gid >= (long long)p.B * runs * groups) return;
  const int cg = (int)(gid % groups), r = (int)((gid / groups) % runs), b = (int)(gid / ((long long)groups * runs));
  const int d0 = CH * cg, t0 = r * p.run, t1 = min(T, t0 + p.run);
  const bf16_t* w = reinterpret_cast<const bf16_t*>(s.weight);
  const bf16_t* st = reinterpret_cast<const bf16_t*>(s.state);
  float wt[W][CH], bs[CH], win[W][CH], dwin[W][CH], dws[W + 2][CH], nw[CH];
#pragma unroll
  for (int c = 0; c < CH; ++c) {
#pragma unroll
    for (int j = 0; j < W; ++j) { wt[j][c] = bf16_to_f32(w[(size_t)(d0 + c) * W + j]); dwin[j][c] = 0.f; }
#pragma unroll
    for (int j = 0; j < W + 2; ++j) dws[j][c] = 0.f;
    bs[c] = s.bias ? bf16_to_f32(reinterpret_cast<const bf16_t*>(s.bias)[d0 + c]) : 0.f;
    nw[c] = s.norm_weight ? ldf(s.norm_weight, p.norm_dtype, (d0 + c) % (8 * s.norm_lanes)) : 1.f;
  }
  const size_t base = (size_t)b * T * D + d0;
  const int lanes = s.norm_lanes * (8 / CH), heads = groups / lanes, head = cg / lanes;
  const float inv_n = s.norm_l2 ? 1.f : 1.f / (CH * lanes), eps = s.norm_eps;
#pragma unroll
  for (int j = 0; j < W - 1; ++j) {
    const int q = t0 - (W - 1) + j;
    if (q >= 0) {
      Pc::up(Pc::at(s.x, base + (size_t)q * D), win[j]);
    } else {
#pragma unroll
      for (int c = 0; c < CH; ++c) win[j][c] = st ? bf16_to_f32(st[((size_t)b * D + d0 + c) * W + (W + q)]) : 0.f;
    }
  }
  struct Row { typename Pc::type x, a, b, n, add; float scale; };
  const typename Pc::type zero = {};
  // row t of every input (rows behind the end repeat the last one), and dx_add of the row that t completes
  auto load = [&](const int t) __attribute__((always_inline)) -> Row {
    const int tc = min(t, T - 1);
    const size_t at = base + (size_t)tc * D;
    Row q;
    q.x = Pc::at(s.x, at);
    q.a = s.dy_a ? Pc::at(s.dy_a, at) : zero;
    q.b = s.dy_b ? Pc::at(s.dy_b, at) : zero;
    q.n = s.dy_norm ? Pc::at(s.dy_norm, at) : zero;
    q.add = s.dx_add ? Pc::at(s.dx_add, base + (size_t)max(t - (W - 1), t0) * D) : zero;
    q.scale = s.scale ? s.scale[((size_t)b * T + tc) * heads + head] : 0.f;
    return q;
  };
  // row t: its gradient at y, its sums (rows of the next run, t >= t1, have none), and dx of row t - (W-1)
  auto one_row = [&](const Row& q, const int t, const bool own) __attribute__((always_inline)) {
    float dp[CH], g[CH], g2[CH], y[CH], da[CH];
    Pc::up(q.x, win[W - 1]);
    Pc::up(q.a, g);
    Pc::up(q.b, g2);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      float acc = bs[c];
#pragma unroll
      for (int j = 0; j < W; ++j) acc += wt[j][c] * win[j][c];
      if constexpr (SILU) {
        const float sg = 1.f / (1.f + __expf(-acc));
        y[c] = acc * sg;
        da[c] = sg * (1.f + acc * (1.f - sg));
      } else {
        y[c] = acc;
        da[c] = 1.f;
      }
      g[c] += g2[c];
    }
    if (s.dy_norm) {
      float dn[CH], ss = 0.f, an = 0.f;
      Pc::up(Pc::down(y), y);                                 // the rounded activation, as the forward normalised it
      Pc::up(q.n, dn);
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        ss += y[c] * y[c];
        an += dn[c] * nw[c] * y[c];
      }
      group_sum2(ss, an, lanes);
      if (s.scale) {                                    // y times its head's number: an is that number's gradient
        if (s.dscale && own && cg == head * lanes) s.dscale[((size_t)b * T + t) * heads + head] = an;
#pragma unroll
        for (int c = 0; c < CH; ++c) g[c] += q.scale * dn[c];
      } else {
        const float rs = rsqrtf(ss * inv_n + eps);
        const float m = an * rs * inv_n;                // mean (sum) of a n
#pragma unroll
        for (int c = 0; c < CH; ++c) {
          const float n = y[c] * rs;
          g[c] += rs * (dn[c] * nw[c] - n * m);
          if (own) dws[W + 1][c] += dn[c] * n;
        }
      }
    } else if (s.dscale && own && cg == head * lanes) {
      s.dscale[((size_t)b * T + t) * heads + head] = 0.f;
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      dp[c] = own || t < T ? g[c] * da[c] : 0.f;
      if (own) {
#pragma unroll
        for (int j = 0; j < W; ++j) dws[j][c] += dp[c] * win[j][c];
        dws[W][c] += dp[c];
      }
      dwin[W - 1][c] = dp[c];
    }
    const int sx = t - (W - 1);
    if (sx >= t0) {
      float o[CH];
      Pc::up(q.add, o);
#pragma unroll
      for (int c = 0; c < CH; ++c)
#pragma unroll
        for (int i = 0; i < W; ++i) o[c] += wt[W - 1 - i][c] * dwin[i][c];
      *reinterpret_cast<typename Pc::type*>(reinterpret_cast<bf16_t*>(s.dx) + base + (size_t)sx * D) = Pc::down(o);
    }
#pragma unroll
    for (int j = 0; j < W - 1; ++j)
#pragma unroll
      for (int c = 0; c < CH; ++c) { win[j][c] = win[j + 1][c]; dwin[j][c] = dwin[j + 1][c]; }
  };
  constexpr int AHEAD = CH == 4 ? 3 : 1;   // (three replace the whole window: no moves; eight channels leave room for one)
  int tb = t0;
  for (; tb + AHEAD <= t1; tb += AHEAD) {
    Row q[AHEAD];
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) q[a] = load(tb + a);
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) one_row(q[a], tb + a, true);
  }
#pragma unroll 1
  for (; tb < t1 + W - 1; ++tb) one_row(load(tb), tb, tb < t1);   // the run's odd row, and the W-1 rows behind it that its dx needs
  float* pr = p.part[si] + ((size_t)(b * runs + r) * (W + 2)) * D + d0;
#pragma unroll
  for (int j = 0; j < W + 2; ++j) {
#pragma unroll
    for (int c = 0; c < CH; c += 4) *reinterpret_cast<f32x4*>(pr + (size_t)j * D + c) = (f32x4){dws[j][c], dws[j][c + 1], dws[j][c + 2], dws[j][c + 3]};
  }
}

// Sums of the runs' partial rows in a fixed order: a workgroup takes 64 adjacent columns of one segment, 16 thread rows each add
// every 16th run (eight loads in flight).  Taps and bias leave in bf16; the norm weight's sums (per channel) in fp32.
struct ConvReduce {
  const float* part[NATSL_CONV_SEGS];
  bf16_t* dw[NATSL_CONV_SEGS];
  bf16_t* db[NATSL_CONV_SEGS];
  float* dn[NATSL_CONV_SEGS];
  int D[NATSL_CONV_SEGS], first[NATSL_CONV_SEGS + 1];
  int n_seg, n_part, W;
};
__global__ __launch_bounds__(1024) void conv_norm_reduce_kernel(const ConvReduce p) {
  __shared__ float sums[16][64];
  int si = 0;
#pragma unroll
  for (int i = 1; i < NATSL_CONV_SEGS; ++i) si = i < p.n_seg && (int)blockIdx.x >= p.first[i] ? i : si;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6, D = p.D[si];
  const int i = ((int)blockIdx.x - p.first[si]) * 64 + tx, n_col = (p.W + 2) * D;
  float acc = 0.f;
  if (i < n_col) {
    const float* src = p.part[si] + i;
    int k = ty;
    for (; k + 7 * 16 < p.n_part; k += 8 * 16) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = src[(size_t)(k + 16 * u) * n_col];
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += v[u];
    }
    for (; k < p.n_part; k += 16) acc += src[(size_t)k * n_col];
  }
  sums[ty][tx] = acc;
  __syncthreads();
  if (ty != 0 || i >= n_col) return;
  float t = 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) t += sums[r][tx];
  const int j = i / D, d = i % D;
  if (j < p.W) p.dw[si][(size_t)d * p.W + j] = f32_to_bf16(t);
  else if (j == p.W) { if (p.db[si]) p.db[si][d] = f32_to_bf16(t); }
  else if (p.dn[si]) p.dn[si][d] = t;
}
// norm weights: the channels' sums over the heads
struct NormReduce { const float* dn[NATSL_CONV_SEGS]; void* out[NATSL_CONV_SEGS]; int D[NATSL_CONV_SEGS], width[NATSL_CONV_SEGS]; int dtype; };
__global__ __launch_bounds__(256) void norm_head_sum_kernel(const NormReduce p) {
  const int si = blockIdx.x;
  if (!p.out[si]) return;
  for (int c = threadIdx.x; c < p.width[si]; c += 256) {
    float t = 0.f;
    for (int d = c; d < p.D[si]; d += p.width[si]) t += p.dn[si][d];
    stf(p.out[si], p.dtype, c, t);
  }
}

// ---- gates ------------------------------------------------------------------------------------------------------------------
struct GatesParams {
  const bf16_t* ab; const void *a_log, *dt_bias;   // ab [rows][ld]: a in columns 0..H-1, b behind them (GDN)
  float* g; bf16_t* beta; float* dt;
  const float* dg; const bf16_t* dbeta; const float* ddt;
  bf16_t* dab; float* part;
  long long rows;
  int H, ld, dtype, neg, iters;                    // iters: batches of rows of a backward workgroup
};

__global__ __launch_bounds__(256) void gates_kernel(const GatesParams p) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= p.rows * p.H) return;
  const long long row = i / p.H;
  const int h = (int)(i - row * p.H);
  const float dt = softplus_gate(bf16_to_f32(p.ab[row * p.ld + h]) + ldf(p.dt_bias, p.dtype, h));
  p.g[i] = -expf(ldf(p.a_log, p.dtype, h)) * dt;
  if (p.dt) p.dt[i] = dt;
  if (p.beta) {
    float s = bf16_to_f32(f32_to_bf16(sigmoid_gate(bf16_to_f32(p.ab[row * p.ld + p.H + h]))));
    p.beta[i] = f32_to_bf16(p.neg ? 2.f * s : s);
  }
}

// Batches of 256 / H rows of a backward workgroup: two, so that the launch fills the chip, and more where that makes more than GATES_WGS
// workgroups, each of which leaves 2 H sums to be written and read again (32768 rows of 256 heads: 33 MB from two batches each; with at most
// 1024, 2048, 4096 workgroups 67, 58, 58 us, 65536 rows of 64 heads 37, 33, 34).
constexpr int GATES_WGS = 2048;
// thread = (row of the workgroup's batch, head); the rows' shares of the two parameter gradients are added through LDS in order
__global__ __launch_bounds__(256) void gates_bwd_kernel(const GatesParams p) {
  __shared__ float red[2][256];
  const int in = 256 / p.H, h = threadIdx.x % p.H, ri = threadIdx.x / p.H;
  float sa = 0.f, sb = 0.f;
  const float A = expf(ldf(p.a_log, p.dtype, h)), bias = ldf(p.dt_bias, p.dtype, h);
  if (ri < in) {
    for (int it = 0; it < p.iters; ++it) {
      const long long row = ((long long)blockIdx.x * p.iters + it) * in + ri;
      if (row >= p.rows) break;
      const float x = bf16_to_f32(p.ab[row * p.ld + h]) + bias;
      const float dt = softplus_gate(x), sg = x > 20.f ? 1.f : sigmoid_gate(x);
      const float dg = p.dg ? p.dg[row * p.H + h] : 0.f;
      const float ddt = (p.ddt ? p.ddt[row * p.H + h] : 0.f) - A * dg;
      const float da = ddt * sg;
      sa += dg * -A * dt;
      sb += da;
      bf16_t* o = p.dab + row * p.ld;
      o[h] = f32_to_bf16(da);
      int used = p.H;
      if (p.beta || p.dbeta) {
        const float s = bf16_to_f32(f32_to_bf16(sigmoid_gate(bf16_to_f32(p.ab[row * p.ld + p.H + h]))));
        const float db = p.dbeta ? bf16_to_f32(p.dbeta[row * p.H + h]) : 0.f;
        o[p.H + h] = f32_to_bf16((p.neg ? 2.f : 1.f) * db * s * (1.f - s));
        used = 2 * p.H;
      }
      for (int c = used + h; c < p.ld; c += p.H) o[c] = 0;
    }
  }
  red[0][threadIdx.x] = ri < in ? sa : 0.f;
  red[1][threadIdx.x] = ri < in ? sb : 0.f;
  __syncthreads();
  if ((int)threadIdx.x < p.H) {
    float ta = 0.f, tb = 0.f;
    for (int r = 0; r < in; ++r) {
      ta += red[0][r * p.H + threadIdx.x];
      tb += red[1][r * p.H + threadIdx.x];
    }
    p.part[(size_t)blockIdx.x * 2 * p.H + threadIdx.x] = ta;
    p.part[(size_t)blockIdx.x * 2 * p.H + p.H + threadIdx.x] = tb;
  }
}
// 16 adjacent columns (sums for A_log, then for dt_bias) per workgroup, 64 thread rows.  With one workgroup for all columns and a load at a
// time it is this kernel that decides from 16 heads on (both kernels, 32768 rows, such a one / this one, us: 6 heads 8.9 / 8.9, 16 15.3 / 9.7,
// 32 41.5 / 13.1, 256 2276 / 58; 65536 rows of 64 heads 300 / 32).
constexpr int GATES_COLS = 16;
__global__ __launch_bounds__(1024) void gates_reduce_kernel(const float* part, void* da_log, void* ddt_bias, const int n_part, const int H, const int dtype) {
  constexpr int TY = 1024 / GATES_COLS;
  __shared__ float sums[16][GATES_COLS];
  const int tx = threadIdx.x % GATES_COLS, ty = threadIdx.x / GATES_COLS, c = blockIdx.x * GATES_COLS + tx;
  float t = c < 2 * H ? column_share<TY>(part, c, ty, n_part, 2 * H) : 0.f;
  t += __shfl_xor(t, 16);                          // (a wave holds four thread rows)
  t += __shfl_xor(t, 32);
  if ((threadIdx.x & 63) < GATES_COLS) sums[threadIdx.x >> 6][tx] = t;
  __syncthreads();
  if (ty == 0 && c < 2 * H) {
    t = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) t += sums[r][tx];
    if (c < H) stf(da_log, dtype, c, t);
    else stf(ddt_bias, dtype, c - H, t);
  }
}

// ---- dx = (block gradient / block length of every token) + dn W: 32 tokens x 64 columns per wave ------------------------------
// W^T is the A operand (a lane's 8 contraction slots are 8 rows of the narrow weight, gathered once), the narrow gradient the B
// operand straight from memory; a lane then holds one token's columns in groups of four.
struct DxInit {
  const bf16_t *dn, *w, *dpool;
  bf16_t* dx;
  long long rows;
  int D, N, ld, T, block, nb;     // dn [rows][ld], w [N][D] (N a multiple of 16, or 0); dpool [B][nb][D] or null
};
constexpr int DX_TILES = 4;
// columns d0.. (one per lane%32) of rows k.. of the narrow weight, as the A operand of W^T
NATSL_DEVICE bf16x8 dx_operand(const DxInit& p, const int k, const int d0) {
  const int lane = threadIdx.x & 63;
  bf16_t wv[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) wv[j] = p.w[(size_t)(k + 8 * (lane >> 5) + j) * p.D + min(d0 + (lane & 31), p.D - 1)];
  u32x4 a;
#pragma unroll
  for (int j = 0; j < 4; ++j) a[j] = (unsigned)wv[2 * j] | ((unsigned)wv[2 * j + 1] << 16);
  return __builtin_bit_cast(bf16x8, a);
}
__global__ __launch_bounds__(256) void dx_init_kernel(const DxInit p) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int half = lane >> 5;
  // a wave keeps its 64 columns for DX_TILES tiles of tokens: the first 16 rows of W^T stay in registers
  bf16x8 w0[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) w0[u] = p.N > 0 ? dx_operand(p, 0, ((int)blockIdx.y * 4 + wave) * 64 + 32 * u) : zero8();
#pragma unroll 1
  for (int it = 0; it < DX_TILES; ++it) {
  const long long t = ((long long)blockIdx.x * DX_TILES + it) * 32 + (lane & 31);
  const long long tc = t < p.rows ? t : p.rows - 1;
  const int b = (int)(tc / p.T), tt = (int)(tc - (long long)b * p.T);
  const int blk = tt / p.block;
  const float inv = 1.f / (float)(min(p.T, (blk + 1) * p.block) - blk * p.block);
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int d0 = ((int)blockIdx.y * 4 + wave) * 64 + 32 * u;
    if (d0 >= p.D) break;
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = 0.f;
    if (p.N > 0) acc = mfma32(w0[u], ld8(p.dn + tc * p.ld + 8 * half), acc);
    for (int k = 16; k < p.N; k += 16) acc = mfma32(dx_operand(p, k, d0), ld8(p.dn + tc * p.ld + k + 8 * half), acc);
    if (t >= p.rows) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int d = d0 + 8 * q + 4 * half;
      if (d >= p.D) continue;                                 // (D is a multiple of 8: whole groups of four)
      float o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = acc[4 * q + r];
      if (p.dpool) {
        const u32x2 w2 = *reinterpret_cast<const u32x2*>(p.dpool + ((size_t)b * p.nb + blk) * p.D + d);
        o[0] += inv * __uint_as_float(w2[0] << 16);
        o[1] += inv * __uint_as_float(w2[0] & 0xffff0000u);
        o[2] += inv * __uint_as_float(w2[1] << 16);
        o[3] += inv * __uint_as_float(w2[1] & 0xffff0000u);
      }
      *reinterpret_cast<u32x2*>(p.dx + (size_t)t * p.D + d) = (u32x2){pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
    }
  }
  }
}

// ---- selector: gradient of the softmax behind the hard selection ---------------------------------------------------------------
__global__ __launch_bounds__(256) void select_bwd_kernel(const void* logits, const void* dtypes, void* dlogits, const long long n, const int TN,
                                                         const int HN, const int dtype, const int last_forced) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float x0 = ldf(logits, dtype, 2 * i), x1 = ldf(logits, dtype, 2 * i + 1);
  float d0 = ldf(dtypes, dtype, 2 * i), d1 = ldf(dtypes, dtype, 2 * i + 1);
  if (last_forced && (i / HN) % TN == TN - 1) d0 = d1 = 0.f;   // the last block's type is a constant there
  select_grad(x0, x1, dtype == NATSL_BF16, d0, d1);
  stf(dlogits, dtype, 2 * i, d0);
  stf(dlogits, dtype, 2 * i + 1, d1);
}

static int conv_cus() {
  static std::atomic<int> cached{0};
  int n = cached.load();
  if (n == 0) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached.store(n);
  }
  return n;
}

// Tokens per thread: long runs read the fewest rows twice (and leave the fewest partial sums), but what counts first is that the
// workgroups fill whole rounds of the chip -- registers admit three of them on a CU forward (150) and backward with four channels a thread
// (165), two with eight (247).  340M geometry, 8 x 4096: forward 32 -> 64 tokens 100 -> 94 us; backward, with eight channels, runs of 64 in 1.5
// rounds 233 us, of 98 in one 208.
static int conv_run(int B, int T, int W, int groups, bool bwd, int ch) {
  const long long slots = (long long)conv_cus() * (bwd && ch == 8 ? 2 : 3);
  int best = 8;
  double best_cost = 1e300;
  for (int run = 8; run <= (bwd ? 128 : 64); run += bwd ? 2 : 8) {
    const long long wgs = ((long long)B * cdiv(T, run) * groups + 255) / 256;
    const double cost = (double)((wgs + slots - 1) / slots) * (run + W - 1 + (bwd ? 5 : 1));
    if (cost <= best_cost) { best_cost = cost; best = run; }
  }
  return best;
}

static int conv_plan(ConvNormParams& p, const natsl_conv_seg* seg, int n_seg, int B, int T, int W, int silu, int norm_dtype, bool bwd, const char* what) {
  if (!seg || n_seg <= 0 || n_seg > NATSL_CONV_SEGS) return fail(NATSL_ERR_INVALID, "%s: 1 to %d tensors", what, NATSL_CONV_SEGS);
  if (B <= 0 || T <= 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  if (W < 2 || W > 4) return fail(NATSL_ERR_UNSUPPORTED, "%s: kernel size %d not built (2, 3, 4)", what, W);
  long long all = 0;
  bool wide = false;                           // (heads of 512 need eight channels a lane to fit a wave)
  for (int i = 0; i < n_seg; ++i) {
    const natsl_conv_seg& s = seg[i];
    if (s.D <= 0 || s.D % 8) return fail(NATSL_ERR_UNSUPPORTED, "%s: D=%d must be a positive multiple of 8", what, s.D);
    if (!s.x || !s.weight || (bwd ? !s.dx || !s.dweight : !s.y && !s.y_norm)) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
    if (s.y_norm || s.dy_norm || (bwd && s.scale && s.dscale)) {
      const int l = s.norm_lanes;
      if (l <= 0 || l > 64 || (l & (l - 1)) || (s.D / 8) % l) return fail(NATSL_ERR_UNSUPPORTED, "%s: norm width %d", what, 8 * l);
      wide |= l == 64;
      if (bwd && s.norm_weight && !s.dnorm_weight) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
      if (s.scale && s.norm_weight) return fail(NATSL_ERR_INVALID, "%s: a norm or a number", what);
    }
    all += s.D;
  }
  const int ch = bwd && !wide ? 4 : 8, run = conv_run(B, T, W, all / ch, bwd, ch);
  p.ch = ch; p.n_seg = n_seg; p.B = B; p.T = T; p.run = run; p.silu = silu; p.norm_dtype = norm_dtype;
  long long wgs = 0;
  for (int i = 0; i < NATSL_CONV_SEGS; ++i) {
    p.part[i] = nullptr;
    p.first[i] = (int)wgs;
    if (i >= n_seg) continue;
    natsl_conv_seg& s = p.seg[i] = seg[i];
    // (numbers that nothing is multiplied by are not read: without a tensor that follows them norm_lanes says nothing about their rows)
    if (!bwd || !s.scale) s.dscale = nullptr;
    if (bwd ? !s.dy_norm && !s.dscale : !s.y_norm) s.scale = nullptr;
    if (!s.y_norm && !s.dy_norm && !s.dscale) s.norm_lanes = 1;
    wgs += ((long long)B * cdiv(T, run) * (seg[i].D / ch) + 255) / 256;
    if (wgs > 0x7fffffffll) return fail(NATSL_ERR_UNSUPPORTED, "%s: problem too large", what);
  }
  p.first[NATSL_CONV_SEGS] = (int)wgs;
  return NATSL_OK;
}

}  // namespace natsl

using namespace natsl;

extern "C" int natsl_conv_norm_fwd(const natsl_conv_seg* seg, int n_seg, int B, int T, int W, int activation, int norm_dtype, natsl_stream_t stream) {
  const char* what = "natsl_conv_norm_fwd";
  ConvNormParams p;
  const int rc = conv_plan(p, seg, n_seg, B, T, W, activation, norm_dtype, false, what);
  if (rc != NATSL_OK) return rc;
  for (int i = 0; i < n_seg; ++i)
    if (seg[i].state_out && seg[i].state_out == seg[i].state) return fail(NATSL_ERR_INVALID, "%s: state_out must not alias state", what);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)p.first[NATSL_CONV_SEGS]);
  if (W == 4) hipLaunchKernelGGL((conv_norm_kernel<4>), grid, dim3(256), 0, s, p);
  else if (W == 3) hipLaunchKernelGGL((conv_norm_kernel<3>), grid, dim3(256), 0, s, p);
  else hipLaunchKernelGGL((conv_norm_kernel<2>), grid, dim3(256), 0, s, p);
  return check_launch(what);
}

static size_t conv_part_bytes(const ConvNormParams& p, int i, int W) {
  return (size_t)p.B * cdiv(p.T, p.run) * (W + 2) * p.seg[i].D * sizeof(float);
}
extern "C" size_t natsl_conv_norm_bwd_workspace_bytes(const natsl_conv_seg* seg, int n_seg, int B, int T, int W) {
  ConvNormParams p;
  if (conv_plan(p, seg, n_seg, B, T, W, 0, 0, true, "natsl_conv_norm_bwd") != NATSL_OK) return 0;
  size_t n = 0;
  for (int i = 0; i < n_seg; ++i) n += conv_part_bytes(p, i, W) + (size_t)p.seg[i].D * sizeof(float);
  return n;
}

extern "C" int natsl_conv_norm_bwd(const natsl_conv_seg* seg, int n_seg, int B, int T, int W, int activation, int norm_dtype, void* workspace,
                                   size_t workspace_bytes, natsl_stream_t stream) {
  const char* what = "natsl_conv_norm_bwd";
  ConvNormParams p;
  int rc = conv_plan(p, seg, n_seg, B, T, W, activation, norm_dtype, true, what);
  if (rc != NATSL_OK) return rc;
  const size_t need = natsl_conv_norm_bwd_workspace_bytes(seg, n_seg, B, T, W);
  if (!workspace || workspace_bytes < need) return fail(NATSL_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", what, need, workspace_bytes);
  if ((uintptr_t)workspace & 15) return fail(NATSL_ERR_INVALID, "%s: workspace must be 16-byte aligned", what);
  ConvReduce r;
  NormReduce nr;
  r.n_seg = n_seg; r.n_part = B * cdiv(T, p.run); r.W = W;
  nr.dtype = norm_dtype;
  char* at = reinterpret_cast<char*>(workspace);
  int wgs = 0;
  bool norms = false;
  for (int i = 0; i < NATSL_CONV_SEGS; ++i) {
    r.first[i] = wgs;
    r.part[i] = nullptr; r.dw[i] = r.db[i] = nullptr; r.dn[i] = nullptr; r.D[i] = 0;
    nr.out[i] = nullptr; nr.dn[i] = nullptr; nr.D[i] = nr.width[i] = 0;
    if (i >= n_seg) continue;
    p.part[i] = reinterpret_cast<float*>(at);
    at += conv_part_bytes(p, i, W);
    r.part[i] = p.part[i]; r.dw[i] = (bf16_t*)seg[i].dweight; r.db[i] = (bf16_t*)seg[i].dbias; r.D[i] = seg[i].D;
    wgs += cdiv((W + 2) * seg[i].D, 64);
  }
  r.first[NATSL_CONV_SEGS] = wgs;
  for (int i = 0; i < n_seg; ++i) {
    if (seg[i].dy_norm && seg[i].dnorm_weight) {
      r.dn[i] = reinterpret_cast<float*>(at);
      nr.dn[i] = r.dn[i]; nr.out[i] = seg[i].dnorm_weight; nr.D[i] = seg[i].D; nr.width[i] = 8 * seg[i].norm_lanes;
      norms = true;
    }
    at += (size_t)seg[i].D * sizeof(float);
  }
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)p.first[NATSL_CONV_SEGS]);
  auto launch = [&](auto w_c) {
    constexpr int WC = decltype(w_c)::value;
    if (p.ch == 4) {
      if (activation) hipLaunchKernelGGL((conv_norm_bwd_kernel<WC, true, 4>), grid, dim3(256), 0, s, p);
      else hipLaunchKernelGGL((conv_norm_bwd_kernel<WC, false, 4>), grid, dim3(256), 0, s, p);
    } else {
      if (activation) hipLaunchKernelGGL((conv_norm_bwd_kernel<WC, true, 8>), grid, dim3(256), 0, s, p);
      else hipLaunchKernelGGL((conv_norm_bwd_kernel<WC, false, 8>), grid, dim3(256), 0, s, p);
    }
  };
  if (W == 4) launch(std::integral_constant<int, 4>{});
  else if (W == 3) launch(std::integral_constant<int, 3>{});
  else launch(std::integral_constant<int, 2>{});
  if ((rc = check_launch(what)) != NATSL_OK) return rc;
  hipLaunchKernelGGL(conv_norm_reduce_kernel, dim3((unsigned)wgs), dim3(1024), 0, s, r);
  if ((rc = check_launch(what)) != NATSL_OK || !norms) return rc;
  hipLaunchKernelGGL(norm_head_sum_kernel, dim3((unsigned)n_seg), dim3(256), 0, s, nr);
  return check_launch(what);
}

static int gates_check(const void* ab, const void* a_log, const void* dt_bias, int64_t rows, int H, int ld, int delta, int dtype, const char* what) {
  if (!ab || !a_log || !dt_bias) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (rows <= 0 || H <= 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  if (H > 256 || ld < (delta ? 2 * H : H)) return fail(NATSL_ERR_UNSUPPORTED, "%s: %d heads in rows of %d", what, H, ld);
  if (dtype != NATSL_BF16 && dtype != NATSL_F32) return fail(NATSL_ERR_UNSUPPORTED, "%s: parameters must be f32 or bf16", what);
  return NATSL_OK;
}

extern "C" int natsl_gates_fwd(const void* ab, const void* a_log, const void* dt_bias, float* g, void* beta, float* dt, int64_t rows, int H, int ld,
                               int neg_eigval, int param_dtype, natsl_stream_t stream) {
  const char* what = "natsl_gates_fwd";
  const int rc = gates_check(ab, a_log, dt_bias, rows, H, ld, beta != nullptr, param_dtype, what);
  if (rc != NATSL_OK) return rc;
  if (!g) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  GatesParams p{};
  p.ab = (const bf16_t*)ab; p.a_log = a_log; p.dt_bias = dt_bias; p.g = g; p.beta = (bf16_t*)beta; p.dt = dt; p.rows = rows; p.H = H; p.ld = ld;
  p.dtype = param_dtype; p.neg = neg_eigval;
  hipLaunchKernelGGL(gates_kernel, dim3((unsigned)((rows * H + 255) / 256)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), p);
  return check_launch(what);
}

static int gates_iters(int64_t rows, int H) {
  const long long batches = (rows + 256 / H - 1) / (256 / H), per = (batches + GATES_WGS - 1) / GATES_WGS;
  return (int)(per < 2 ? 2 : per);
}
static long long gates_wgs(int64_t rows, int H) { const long long n = (long long)(256 / H) * gates_iters(rows, H); return (rows + n - 1) / n; }
extern "C" size_t natsl_gates_bwd_workspace_bytes(int64_t rows, int H) {
  return rows > 0 && H > 0 && H <= 256 ? (size_t)gates_wgs(rows, H) * 2 * H * sizeof(float) : 0;
}
extern "C" int natsl_gates_bwd(const void* ab, const void* a_log, const void* dt_bias, const float* dg, const void* dbeta, const float* ddt, int delta,
                               void* dab, void* da_log, void* ddt_bias, void* workspace, size_t workspace_bytes, int64_t rows, int H, int ld,
                               int neg_eigval, int param_dtype, natsl_stream_t stream) {
  const char* what = "natsl_gates_bwd";
  int rc = gates_check(ab, a_log, dt_bias, rows, H, ld, delta, param_dtype, what);
  if (rc != NATSL_OK) return rc;
  if (!dab || !da_log || !ddt_bias) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (!workspace || workspace_bytes < natsl_gates_bwd_workspace_bytes(rows, H)) return fail(NATSL_ERR_WORKSPACE, "%s: workspace too small", what);
  GatesParams p{};
  p.ab = (const bf16_t*)ab; p.a_log = a_log; p.dt_bias = dt_bias; p.dg = dg; p.dbeta = (const bf16_t*)dbeta; p.ddt = ddt; p.dab = (bf16_t*)dab;
  p.beta = delta ? (bf16_t*)dab : nullptr;      // (only tells the kernel that the rows hold b)
  p.part = reinterpret_cast<float*>(workspace); p.rows = rows; p.H = H; p.ld = ld; p.dtype = param_dtype; p.neg = neg_eigval;
  p.iters = gates_iters(rows, H);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const long long wgs = gates_wgs(rows, H);
  hipLaunchKernelGGL(gates_bwd_kernel, dim3((unsigned)wgs), dim3(256), 0, s, p);
  if ((rc = check_launch(what)) != NATSL_OK) return rc;
  hipLaunchKernelGGL(gates_reduce_kernel, dim3((unsigned)cdiv(2 * H, GATES_COLS)), dim3(1024), 0, s, p.part, da_log, ddt_bias, (int)wgs, H, param_dtype);
  return check_launch(what);
}

extern "C" int natsl_dx_init(const void* dn, const void* w, const void* dpool, void* dx, int B, int T, int D, int N, int ld, int block, natsl_stream_t stream) {
  const char* what = "natsl_dx_init";
  if (!dx || (N > 0 && (!dn || !w))) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (B <= 0 || T <= 0 || D <= 0 || block <= 0 || N < 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  if (D % 8 || N % 16 || ld % 8 || ld < N) return fail(NATSL_ERR_UNSUPPORTED, "%s: D=%d must be a multiple of 8, N=%d of 16", what, D, N);
  DxInit p;
  p.dn = (const bf16_t*)dn; p.w = (const bf16_t*)w; p.dpool = (const bf16_t*)dpool; p.dx = (bf16_t*)dx; p.rows = (long long)B * T; p.D = D; p.N = N;
  p.ld = ld; p.T = T; p.block = block; p.nb = cdiv(T, block);
  hipLaunchKernelGGL(dx_init_kernel, dim3((unsigned)((p.rows + 32 * DX_TILES - 1) / (32 * DX_TILES)), (unsigned)cdiv(D, 256)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), p);
  return check_launch(what);
}

extern "C" int natsl_hard_select_bwd(const void* logits, const void* dtypes, void* dlogits, int B, int TN, int HN, int dtype, int last_forced,
                                     natsl_stream_t stream) {
  const char* what = "natsl_hard_select_bwd";
  if (!logits || !dtypes || !dlogits) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (B <= 0 || TN <= 0 || HN <= 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  if (dtype != NATSL_BF16 && dtype != NATSL_F32) return fail(NATSL_ERR_UNSUPPORTED, "%s: dtype %d", what, dtype);
  const long long n = (long long)B * TN * HN;
  hipLaunchKernelGGL(select_bwd_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), logits, dtypes, dlogits, n,
                     TN, HN, dtype, last_forced);
  return check_launch(what);
}
