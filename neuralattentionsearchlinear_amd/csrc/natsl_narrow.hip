// The layers' narrow products (weights of a few dozen rows), bound by the wide tensor's bytes:
//   forward   Y[t][n] = sum_d X[t][d] W[n][d], in the same pass over X the means of its 64-token blocks, their selector logits and the
//             gates behind Y
//   backward  X'[t][d] = sum_n Y'[t][n] W[n][d]   writes X' once
// bf16 operands, fp32 sums, one rounding.  Where the contraction is no multiple of 32 a library product takes two to three times as long as for
// one that is (36 rows of 1152 over 32768 tokens 36 us, 32 rows of 1024 19).
#include <algorithm>
#include <type_traits>

#include "natsl_device.h"
#include "natsl_host.h"

namespace natsl {

// ---- forward -------------------------------------------------------------------------------------------------------------------------
// A workgroup takes 64 tokens (a selector block); its waves share the contraction, 64 columns at a time in turn, and add up through LDS in
// a fixed order.  A lane's operands are 16-byte pieces of rows as they lie in memory, requested a step ahead: nothing is staged.  The block's
// mean is formed from the same registers (four rows a lane, then across the 16 lanes of a row group) and is the operand of the logits.
// Against four launches (block means, two library products, gates), us: 32768 tokens of 1024, 12 rows and 12 logits 36 -> 24 (13 at the rate of a
// copy: a workgroup has its 64 columns' share requested at once and little to overlap it with; two workgroups a CU spill, 28 - 40), 16 rows and 32
// logits 39 -> 27; 6000 of 1536 26 -> 13; 777 of 1024 25 -> 9.
struct FrontParams {
  natsl_front f;
  int nb;
};

template <int NT, int NL>
struct FrontLds {
  static constexpr int TILES = 4 * NT + NL, NW = 8, RED = NW * TILES * 1024, TOTAL = RED + 64 * 16 * NT * 2;
};

// the sum over the 16 lanes that share lane / 16, in all of them
NATSL_DEVICE float row_sum16(float x) {
  auto ror = [](const float v, auto c) __attribute__((always_inline)) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(v), 0x120 + decltype(c)::value, 0xf, 0xf, true));
  };
  x += ror(x, std::integral_constant<int, 8>{});
  x += ror(x, std::integral_constant<int, 4>{});
  x += ror(x, std::integral_constant<int, 2>{});
  return x + ror(x, std::integral_constant<int, 1>{});
}

template <int NT, int NL>
__global__ __launch_bounds__((64 * FrontLds<NT, NL>::NW)) void narrow_front_kernel(const FrontParams p) {
  using L = FrontLds<NT, NL>;
  constexpr int NW = L::NW, TILES = L::TILES, NLA = NL > 0 ? NL : 1;
  extern __shared__ __align__(16) unsigned char smem[];
  const natsl_front& f = p.f;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i16 = lane & 15, g4 = lane >> 4;
  const int b = (int)blockIdx.x / p.nb, t0 = ((int)blockIdx.x - b * p.nb) * 64, len = min(64, f.T - t0), D = f.D, N = f.NA + f.NB;
  const size_t row0 = (size_t)b * f.T + t0;
  const bf16_t* x = reinterpret_cast<const bf16_t*>(f.x) + row0 * D + 8 * g4;
  const bf16_t *xr[4], *wr[NT], *nr[NLA];
#pragma unroll
  for (int t = 0; t < 4; ++t) xr[t] = x + (size_t)min(16 * t + i16, len - 1) * D;
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int r = min(16 * n + i16, N - 1);
    wr[n] = reinterpret_cast<const bf16_t*>(r < f.NA ? f.wa : f.wb) + (size_t)(r < f.NA ? r : r - f.NA) * D + 8 * g4;
  }
#pragma unroll
  for (int n = 0; n < NL; ++n) nr[n] = reinterpret_cast<const bf16_t*>(f.wn) + (size_t)min(16 * n + i16, f.NL - 1) * D + 8 * g4;

  f32x4 acc[4][NT], lacc[NLA];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t][n] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int n = 0; n < NLA; ++n) lacc[n] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const float inv = 1.f / (float)len;
  struct Step { u32x4 x[2][4], w[2][NT], n[2][NLA]; };
  const int pairs = (D + 63) >> 6;
  auto load = [&](Step& s, const int pr) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = min(64 * pr + 32 * h, D - 32);
#pragma unroll
      for (int t = 0; t < 4; ++t) s.x[h][t] = *reinterpret_cast<const u32x4*>(xr[t] + k);
#pragma unroll
      for (int n = 0; n < NT; ++n) s.w[h][n] = *reinterpret_cast<const u32x4*>(wr[n] + k);
#pragma unroll
      for (int n = 0; n < NL; ++n) s.n[h][n] = *reinterpret_cast<const u32x4*>(nr[n] + k);
    }
  };
  auto use = [&](Step& s, const int pr) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = 64 * pr + 32 * h;
      if (h == 1 && k >= D) break;                  // (the width's odd 32 columns)
      if (len < 64) {                               // rows past the end count for nothing
#pragma unroll
        for (int t = 0; t < 4; ++t)
          if (16 * t + i16 >= len) s.x[h][t] = (u32x4){0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t][n] = mfma16(__builtin_bit_cast(bf16x8, s.x[h][t]), __builtin_bit_cast(bf16x8, s.w[h][n]), acc[t][n]);
      if constexpr (NL > 0) {
        float m[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float lo = 0.f, hi = 0.f;
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            lo += __uint_as_float(s.x[h][t][j] << 16);
            hi += __uint_as_float(s.x[h][t][j] & 0xffff0000u);
          }
          m[2 * j] = row_sum16(lo) * inv;
          m[2 * j + 1] = row_sum16(hi) * inv;
        }
        u32x4 a;
#pragma unroll
        for (int j = 0; j < 4; ++j) a[j] = pack_bf16x2(m[2 * j], m[2 * j + 1]);
        if (f.pooled && i16 == 0) *reinterpret_cast<u32x4*>(reinterpret_cast<bf16_t*>(f.pooled) + (size_t)blockIdx.x * D + k + 8 * g4) = a;
#pragma unroll
        for (int n = 0; n < NL; ++n) lacc[n] = mfma16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, s.n[h][n]), lacc[n]);
      }
    }
  };
  Step s0, s1;
  int pr = wave;
  if (pr < pairs) load(s0, pr);
  for (; pr < pairs; pr += 2 * NW) {
    if (pr + NW < pairs) load(s1, pr + NW);
    use(s0, pr);
    if (pr + NW >= pairs) break;
    if (pr + 2 * NW < pairs) load(s0, pr + 2 * NW);
    use(s1, pr + NW);
  }
  // ---- the waves' shares are added in order; rounded rows wait in LDS for the stores and the gates
  f32x4* red = reinterpret_cast<f32x4*>(smem);
  bf16_t* rows = reinterpret_cast<bf16_t*>(smem + L::RED);
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int t = 0; t < 4; ++t) red[(wave * TILES + 4 * n + t) * 64 + lane] = acc[t][n];
#pragma unroll
  for (int n = 0; n < NL; ++n) red[(wave * TILES + 4 * NT + n) * 64 + lane] = lacc[n];
  __syncthreads();
  for (int j = wave; j < TILES; j += NW) {
    f32x4 sum = red[j * 64 + lane];
#pragma unroll
    for (int w = 1; w < NW; ++w) sum += red[(w * TILES + j) * 64 + lane];
    if (j < 4 * NT) {
      const int n = j >> 2, t = j & 3;
#pragma unroll
      for (int r = 0; r < 4; ++r) rows[(16 * t + 4 * g4 + r) * (16 * NT) + 16 * n + i16] = f32_to_bf16(sum[r]);
    } else {
      const int col = 16 * (j - 4 * NT) + i16;      // (all rows of a logits tile are the block's)
      if (g4 == 0 && col < f.NL) reinterpret_cast<bf16_t*>(f.logits)[(size_t)blockIdx.x * f.NL + col] = f32_to_bf16(sum[0]);
    }
  }
  __syncthreads();
  if (f.ab) {
    unsigned* out = reinterpret_cast<unsigned*>(reinterpret_cast<bf16_t*>(f.ab) + row0 * f.ld);
    const int half = f.ld >> 1;
    for (int e = threadIdx.x; e < len * half; e += 64 * NW) {
      const int r = e / half, c = 2 * (e - r * half);
      const unsigned lo = c < N ? rows[r * (16 * NT) + c] : 0u, hi = c + 1 < N ? rows[r * (16 * NT) + c + 1] : 0u;
      out[e] = lo | (hi << 16);
    }
  }
  if (f.g) {
    auto param = [&](const void* q, const int h) __attribute__((always_inline)) {
      return f.param_dtype == NATSL_F32 ? reinterpret_cast<const float*>(q)[h] : bf16_to_f32(reinterpret_cast<const bf16_t*>(q)[h]);
    };
    for (int e = threadIdx.x; e < len * f.NA; e += 64 * NW) {
      const int r = e / f.NA, h = e - r * f.NA;
      const float dt = softplus_gate(bf16_to_f32(rows[r * (16 * NT) + h]) + param(f.dt_bias, h));
      f.g[row0 * f.NA + e] = -expf(param(f.a_log, h)) * dt;
      if (f.dt) f.dt[row0 * f.NA + e] = dt;
      if (f.beta) {
        const float s = bf16_to_f32(f32_to_bf16(sigmoid_gate(bf16_to_f32(rows[r * (16 * NT) + f.NA + h]))));
        reinterpret_cast<bf16_t*>(f.beta)[row0 * f.NA + e] = f32_to_bf16(f.neg_eigval ? 2.f * s : s);
      }
    }
  }
  if (f.wab) {   // both weights behind each other and zeros up to wab_rows, for the products of the backward
    for (int r = blockIdx.x; r < f.wab_rows; r += gridDim.x) {
      const bf16_t* src = r < f.NA ? reinterpret_cast<const bf16_t*>(f.wa) + (size_t)r * D : reinterpret_cast<const bf16_t*>(f.wb) + (size_t)(r - f.NA) * D;
      for (int c = 8 * threadIdx.x; c < D; c += 8 * 64 * NW)
        *reinterpret_cast<u32x4*>(reinterpret_cast<bf16_t*>(f.wab) + (size_t)r * D + c) =
            r < N ? *reinterpret_cast<const u32x4*>(src + c) : (u32x4){0u, 0u, 0u, 0u};
    }
  }
}

template <int NT, int NL>
static int launch_front(const FrontParams& p, hipStream_t s, const char* what) {
  using L = FrontLds<NT, NL>;
  auto kern = narrow_front_kernel<NT, NL>;
  static std::atomic<unsigned long long> reserved{0};
  if (const int rc = reserve_lds(reinterpret_cast<const void*>(kern), reserved, L::TOTAL, what)) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.f.B * p.nb)), dim3(64 * L::NW), L::TOTAL, s, p);
  return check_launch(what);
}

// ---- backward ------------------------------------------------------------------------------------------------------------------------
constexpr int NARROW_MAX = 48;                 // rows of the weight

struct NarrowParams {
  const bf16_t *dy, *w;
  bf16_t* dx;
  long long rows;
  int D, N;
};

// A wave keeps the weight's share of 64 columns as A operands and walks NARROW_TILES tiles of 32 tokens; the results leave through LDS as
// whole 128-byte lines.
constexpr int NARROW_TILES = 4;
template <int NS>                              // steps of 16 rows of the weight
__global__ __launch_bounds__(256) void narrow_bwd_kernel(const NarrowParams p) {
  __shared__ __align__(16) unsigned char out[4][4096];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31, hf = lane >> 5;
  const int d0 = ((int)blockIdx.y * 4 + wave) * 64;
  if (d0 >= p.D) return;
  bf16x8 A[2][NS];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      bf16_t wv[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int n = 16 * s + 8 * hf + j;
        wv[j] = n < p.N ? p.w[(size_t)n * p.D + min(d0 + 32 * u + l32, p.D - 1)] : 0;
      }
      u32x4 a;
#pragma unroll
      for (int j = 0; j < 4; ++j) a[j] = (unsigned)wv[2 * j] | ((unsigned)wv[2 * j + 1] << 16);
      A[u][s] = __builtin_bit_cast(bf16x8, a);
    }
  unsigned char* st = out[wave];
#pragma unroll 1
  for (int it = 0; it < NARROW_TILES; ++it) {
    const long long t0 = ((long long)blockIdx.x * NARROW_TILES + it) * 32;
    if (t0 >= p.rows) return;
    const long long t = t0 + l32 < p.rows ? t0 + l32 : p.rows - 1;
    bf16x8 B[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      u32x2 h[2];                              // (a row starts on 8 bytes; slots behind the weight's rows are zero on both sides)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int n = 16 * s + 8 * hf + 4 * i;
        h[i] = n < p.N ? *reinterpret_cast<const u32x2*>(p.dy + t * p.N + n) : (u32x2){0u, 0u};
      }
      B[s] = __builtin_bit_cast(bf16x8, (u32x4){h[0][0], h[0][1], h[1][0], h[1][1]});
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      f32x16 acc;
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
      for (int s = 0; s < NS; ++s) acc = mfma32(A[u][s], B[s], acc);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<u32x2*>(st + l32 * 128 + (((4 * u + q) ^ (l32 & 7)) * 16) + 8 * hf) = (u32x2){pack_bf16x2(acc[4 * q], acc[4 * q + 1]), pack_bf16x2(acc[4 * q + 2], acc[4 * q + 3])};
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    const int s = lane & 7, r0 = lane >> 3, col = d0 + 8 * s;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = 8 * u + r0;
      const u32x4 w = *reinterpret_cast<const u32x4*>(st + r * 128 + ((s ^ (r & 7)) * 16));
      if (t0 + r < p.rows && col < p.D) *reinterpret_cast<u32x4*>(p.dx + (size_t)(t0 + r) * p.D + col) = w;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// dW[n][d] = sum_t dY[t][n] X[t][d] for a narrow weight over few rows (the block means behind the selector's).  A workgroup takes 32 columns and
// every row of the weight, its eight waves the tokens, 32 at a time in turn; both operands have the tokens along the contraction and are
// gathered from the rows as they lie (X two columns a word: one product for the even, one for the odd ones).  Added up through LDS in order.
// SPLIT, for many rows (the mixing logits' weight): gridDim.x workgroups share a column group's tokens and leave partial sums for
// narrow_wgrad_sum_kernel.  Their number is a multiple of eight and their index the faster one: an XCD then takes every column of its tokens, and
// reads the lines of X, which two column groups share, and of dY, which all do, once.  Bound by that reading, for few rows by two launches: a library product over so many rows
// for so few outputs leaves most of the chip idle.  us, library / this: 36 x 1152 over 6000 tokens 42 / 12, 32768 112 / 36; 24 x 768 over 6000 42 / 7.2,
// 32768 108 / 14 (natsl_wgrad 21 and 28).  A step asks for all its pieces before it uses one: left to itself the compiler had half of them in flight
// (32768 tokens, 36 x 1152: 69 us).
constexpr int NWG_WAVES = 8;
template <int NT, bool SPLIT>
__global__ __launch_bounds__(64 * NWG_WAVES) void narrow_wgrad_kernel(const bf16_t* dy, const bf16_t* x, bf16_t* dw, float* parts, const int rows, const int D,
                                                                      const int N) {
  __shared__ f32x4 sums[NWG_WAVES][2 * NT][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), i16 = lane & 15, g4 = lane >> 4;
  const int d = 32 * (int)(SPLIT ? blockIdx.y : blockIdx.x) + 2 * i16, part = SPLIT ? (int)blockIdx.x : 0, n_parts = SPLIT ? (int)gridDim.x : 1;
  f32x4 acc[2][NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[0][n] = acc[1][n] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const int dc = min(d, D - 2);
  int nc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) nc[n] = min(16 * n + i16, N - 1);
  // 32 tokens, `left` of them there; everything is requested before any of it is looked at
  auto step = [&](const int t0, auto whole_c, const int left) __attribute__((always_inline)) {
    constexpr bool WHOLE = decltype(whole_c)::value;
    const bf16_t *xr = x + (size_t)t0 * D, *yr = dy + (size_t)t0 * N;
    unsigned xv[8];
    bf16_t yv[NT][8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      // (whole steps: a row's distance from the lane's first is the same in every lane)
      xv[j] = WHOLE ? *reinterpret_cast<const unsigned*>(xr + (size_t)j * D + (unsigned)(8 * g4 * D + dc))
                    : *reinterpret_cast<const unsigned*>(xr + (unsigned)(min(8 * g4 + j, left - 1) * D + dc));
#pragma unroll
      for (int n = 0; n < NT; ++n)
        yv[n][j] = WHOLE ? yr[(size_t)j * N + (unsigned)(8 * g4 * N + nc[n])] : yr[(unsigned)(min(8 * g4 + j, left - 1) * N + nc[n])];
    }
    __builtin_amdgcn_sched_barrier(0);
    if (!WHOLE) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {                // (both sides: nothing that a row behind the end holds enters a product)
        const bool on = 8 * g4 + j < left;
        xv[j] = on ? xv[j] : 0u;
#pragma unroll
        for (int n = 0; n < NT; ++n) yv[n][j] = on ? yv[n][j] : (bf16_t)0;
      }
    }
    u32x4 be, bo;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      be[j] = (xv[2 * j] & 0xffffu) | (xv[2 * j + 1] << 16);
      bo[j] = (xv[2 * j] >> 16) | (xv[2 * j + 1] & 0xffff0000u);
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      u32x4 a;
#pragma unroll
      for (int j = 0; j < 4; ++j) a[j] = (unsigned)yv[n][2 * j] | ((unsigned)yv[n][2 * j + 1] << 16);
      acc[0][n] = mfma16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, be), acc[0][n]);
      acc[1][n] = mfma16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, bo), acc[1][n]);
    }
  };
#pragma unroll 1
  for (int t0 = 32 * (NWG_WAVES * part + wave); t0 < rows; t0 += 32 * NWG_WAVES * n_parts) {
    if (t0 + 32 <= rows) step(t0, std::true_type{}, 32);
    else step(t0, std::false_type{}, rows - t0);
  }
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    sums[wave][2 * n][lane] = acc[0][n];
    sums[wave][2 * n + 1][lane] = acc[1][n];
  }
  __syncthreads();
  if (wave >= NT || d >= D) return;                // wave n ends 16 rows of the weight
  f32x4 e = {0.f, 0.f, 0.f, 0.f}, o = e;
#pragma unroll
  for (int w = 0; w < NWG_WAVES; ++w) {
    e += sums[w][2 * wave][lane];
    o += sums[w][2 * wave + 1][lane];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = 16 * wave + 4 * g4 + r;
    if (n >= N) continue;
    if (SPLIT) *reinterpret_cast<f32x2*>(parts + ((size_t)part * N + n) * D + d) = (f32x2){e[r], o[r]};
    else *reinterpret_cast<unsigned*>(dw + (size_t)n * D + d) = pack_bf16x2(e[r], o[r]);
  }
}

// 128 elements of dW a workgroup; its four waves take every fourth part each, added up through LDS in order.
__global__ __launch_bounds__(256) void narrow_wgrad_sum_kernel(const float* parts, bf16_t* dw, const int n_parts, const int elements) {
  __shared__ f32x2 sums[4][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int e = 128 * (int)blockIdx.x + 2 * lane;
  const float* src = parts + min(e, elements - 2);
  f32x2 a = {0.f, 0.f};
#pragma unroll 8
  for (int i = wave; i < n_parts; i += 4) a += *reinterpret_cast<const f32x2*>(src + (size_t)i * elements);
  sums[wave][lane] = a;
  __syncthreads();
  if (wave != 0 || e >= elements) return;
#pragma unroll
  for (int w = 1; w < 4; ++w) a += sums[w][lane];
  *reinterpret_cast<unsigned*>(dw + e) = pack_bf16x2(a[0], a[1]);
}

// Parts of the rows: eight (one an XCD) until the bytes of X count for more than the partial sums and the rounds of workgroups do.  us with 8 / 16 / 32:
// 6000 tokens 36 x 1152 11.6 / 14.4 / 15.9, 24 x 768 7.2 / 8.4 / 9.8; 16000 19.1 / 18.5 / 20.8, 10.6 / 11.5 / 10.7; 32768 38.8 / 33.6 / 35.6,
// 15.7 / 16.8 / 14.1; 65536 73 / 60 / 59, 39 / 42 / 33.
static int narrow_wgrad_parts(const int64_t rows) {
  const int64_t steps = (rows + 32 * NWG_WAVES - 1) / (32 * NWG_WAVES);
  return (int)std::min<int64_t>(rows <= 16384 ? 8 : 32, (steps + 7) / 8 * 8);
}

}  // namespace natsl

using namespace natsl;

// The one-pass kernel up to 32 rows of the weight (24 x 768 over 32768 tokens 20 -> 16 us, 32 x 2048 over 16000 24 -> 21), and for a few thousand
// tokens of more, where it takes 3 us more than the library's kernel but 30 less of the host's time.
extern "C" int natsl_narrow_fwd_pays(const int64_t rows, const int D, const int N) {
  return N > 0 && N <= 64 && N % 2 == 0 && D > 0 && D % 32 == 0 && rows > 0 && rows < 1ll << 30 && (N <= 32 || rows <= 4096);
}

// Measured (library / natsl_narrow_linear_bwd, us, tensors in the cache): 8 x 512 over 16000 10.3 / 7.2, 24 x 768 over 2048 6.5 / 6.8, 6000 12.5 / 7.7,
// 32768 26.1 / 14.2, 36 x 1152 over 2048 7.3 / 7.9, 6000 11.1 / 9.2, 40 x 1024 over 6000 9.9 / 9.4 (from memory 10.2 / 10.7), 48 x 768 over 65536
// 39 / 29.  The library's kernels for 32 and 64 rows are as good or better (32 x 512 over 6000 5.5 / 7.5, 64 x 1024 over 32768 20 / 27), 52 to 60
// rows lose below 2^24 elements.  few: a library product of the selector's size is 4 to 8 us against 3 to 7, and 40 us of the host's time against 5.
extern "C" int natsl_narrow_linear_bwd_pays(const int64_t rows, const int D, const int N, const int few) {
  if (N <= 0 || N % 4 || N > NARROW_MAX || D <= 0 || D % 128 || rows <= 0) return 0;
  return few || (N % 32 != 0 && rows * D >= (N < 32 ? 4 << 20 : 6 << 20));
}

// few, over the block means (library / natsl_narrow_wgrad, us): 12 x 1536 over 94 6.7 / 2.7, 512 8.1 / 3.2, 2048 7.0 / 5.1, 4096 9.6 / 7.6;
// 32 x 1024 over 512 7.3 / 3.6, 2048 8.6 / 6.5; 64 x 2048 over 2048 15.5 / 9.0.
// Else the split product (the other way / it, us): widths that are no multiple of 8, which leaves the library, 36 x 1152 over 2000 19 / 8.5, 6000 42 / 12,
// 32768 112 / 36; natsl_wgrad 24 x 768 over 2000 14 / 5.7, 32768 28 / 14, 32 x 2048 over 2000 16 / 7.3, 16000 24 / 21, 32768 39 / 46, 48 x 1536 over
// 16000 25 / 20, 32768 37 / 49, 64 x 2048 over 6000 20 / 24.
extern "C" int natsl_narrow_wgrad_pays(const int64_t rows, const int D, const int N, const int few, const int alone) {
  if (N <= 0 || N > 64 || D <= 0 || D % 2 || rows <= 0 || rows > 0x7fffff00ll) return 0;
  if (few) return rows <= 2048;
  return N % 8 != 0 || (alone && N <= 48 && rows * D <= 1ll << 25) ? 2 : 0;
}

static int narrow_wgrad(const char* what, const void* dy, const void* x, void* dw, const int64_t rows, const int D, const int N, float* parts, hipStream_t s) {
  if (!dy || !x || !dw) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (rows <= 0 || D <= 0 || N <= 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  if (N > 64 || D % 2 || rows > 0x7fffff00ll) return fail(NATSL_ERR_UNSUPPORTED, "%s: N=%d (up to 64), D=%d (even)", what, N, D);
  if (((uintptr_t)x | (uintptr_t)dw) & 3) return fail(NATSL_ERR_INVALID, "%s: tensors must start on 4 bytes", what);
  const int n_parts = narrow_wgrad_parts(rows);
  const dim3 grid(parts ? (unsigned)n_parts : (unsigned)cdiv(D, 32), parts ? (unsigned)cdiv(D, 32) : 1u), wg(64 * NWG_WAVES);
  const bf16_t *y = (const bf16_t*)dy, *xx = (const bf16_t*)x;
#define NATSL_NW(NT)                                                                                                                          \
  if (parts) hipLaunchKernelGGL((narrow_wgrad_kernel<NT, true>), grid, wg, 0, s, y, xx, (bf16_t*)dw, parts, (int)rows, D, N);                 \
  else hipLaunchKernelGGL((narrow_wgrad_kernel<NT, false>), grid, wg, 0, s, y, xx, (bf16_t*)dw, parts, (int)rows, D, N);                      \
  break
  switch (cdiv(N, 16)) {
    case 1: NATSL_NW(1);
    case 2: NATSL_NW(2);
    case 3: NATSL_NW(3);
    default: NATSL_NW(4);
  }
#undef NATSL_NW
  const int rc = check_launch(what);
  if (rc != NATSL_OK || !parts) return rc;
  hipLaunchKernelGGL(narrow_wgrad_sum_kernel, dim3((unsigned)cdiv(N * D, 128)), dim3(256), 0, s, parts, (bf16_t*)dw, n_parts, N * D);
  return check_launch(what);
}

extern "C" int natsl_narrow_wgrad(const void* dy, const void* x, void* dw, int64_t rows, int D, int N, natsl_stream_t stream) {
  return narrow_wgrad("natsl_narrow_wgrad", dy, x, dw, rows, D, N, nullptr, reinterpret_cast<hipStream_t>(stream));
}

extern "C" size_t natsl_narrow_wgrad_workspace_bytes(int64_t rows, int D, int N) {
  return rows > 0 && D > 0 && N > 0 ? (size_t)narrow_wgrad_parts(rows) * N * D * sizeof(float) : 0;
}

extern "C" int natsl_narrow_wgrad_split(const void* dy, const void* x, void* dw, int64_t rows, int D, int N, void* workspace, size_t workspace_bytes,
                                        natsl_stream_t stream) {
  const char* what = "natsl_narrow_wgrad_split";
  const size_t need = natsl_narrow_wgrad_workspace_bytes(rows, D, N);
  if (!workspace || (uintptr_t)workspace & 7) return fail(NATSL_ERR_INVALID, "%s: the workspace must start on 8 bytes", what);
  if (workspace_bytes < need) return fail(NATSL_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", what, need, workspace_bytes);
  return narrow_wgrad(what, dy, x, dw, rows, D, N, (float*)workspace, reinterpret_cast<hipStream_t>(stream));
}

extern "C" int natsl_narrow_linear_bwd(const void* dy, const void* w, void* dx, int64_t rows, int D, int N, natsl_stream_t stream) {
  const char* what = "natsl_narrow_linear_bwd";
  if (!dy || !w || !dx) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (rows <= 0 || D <= 0 || N <= 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  if (N > NARROW_MAX || N % 4 || D % 128 || rows > (1ll << 32))
    return fail(NATSL_ERR_UNSUPPORTED, "%s: N=%d (a multiple of 4 up to %d), D=%d (a multiple of 128)", what, N, NARROW_MAX, D);
  if (((uintptr_t)dy | (uintptr_t)w | (uintptr_t)dx) & 15) return fail(NATSL_ERR_INVALID, "%s: tensors must start on 16 bytes", what);
  const NarrowParams p{(const bf16_t*)dy, (const bf16_t*)w, (bf16_t*)dx, rows, D, N};
  const dim3 grid((unsigned)((rows + 32 * NARROW_TILES - 1) / (32 * NARROW_TILES)), (unsigned)cdiv(D, 256));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  switch (cdiv(N, 16)) {
    case 1: hipLaunchKernelGGL(narrow_bwd_kernel<1>, grid, dim3(256), 0, s, p); break;
    case 2: hipLaunchKernelGGL(narrow_bwd_kernel<2>, grid, dim3(256), 0, s, p); break;
    default: hipLaunchKernelGGL(narrow_bwd_kernel<3>, grid, dim3(256), 0, s, p); break;
  }
  return check_launch(what);
}

extern "C" int natsl_layer_front(const natsl_front* a, natsl_stream_t stream) {
  const char* what = "natsl_layer_front";
  if (!a || !a->x || !a->wa || (a->NB > 0 && !a->wb) || (a->NL > 0 && (!a->wn || !a->logits)) || (a->g && (!a->a_log || !a->dt_bias)) || (!a->ab && !a->g))
    return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (a->B <= 0 || a->T <= 0 || a->D <= 0 || a->NA <= 0 || a->NB < 0 || a->NL < 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  const int N = a->NA + a->NB;
  if (a->D % 32 || N > 64 || a->NL > 64 || (a->NL > 0 && N > 32))
    return fail(NATSL_ERR_UNSUPPORTED, "%s: D=%d (a multiple of 32), %d rows (up to 64, 32 next to logits), %d logits (up to 64)", what, a->D, N, a->NL);
  if ((a->ab && (a->ld < N || a->ld % 2)) || (a->beta && (!a->g || a->NB < a->NA)) || (a->dt && !a->g))
    return fail(NATSL_ERR_UNSUPPORTED, "%s: rows of %d for %d columns, or gates that do not belong together", what, a->ld, N);
  if (a->param_dtype != NATSL_BF16 && a->param_dtype != NATSL_F32) return fail(NATSL_ERR_UNSUPPORTED, "%s: parameters must be f32 or bf16", what);
  if (((uintptr_t)a->x | (uintptr_t)a->wa | (uintptr_t)a->wb | (uintptr_t)a->wn | (uintptr_t)a->pooled | (uintptr_t)a->wab) & 15 || (uintptr_t)a->ab & 3)
    return fail(NATSL_ERR_INVALID, "%s: tensors must start on 16 bytes", what);
  FrontParams p{*a, cdiv(a->T, 64)};
  if ((long long)a->B * p.nb > 0x7fffffffll) return fail(NATSL_ERR_UNSUPPORTED, "%s: problem too large", what);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int nt = cdiv(N, 16), nl = cdiv(a->NL, 16);
  if (nt == 4) return launch_front<4, 0>(p, s, what);
  if (nt == 3) return launch_front<3, 0>(p, s, what);
  if (nt == 2) return nl == 0 ? launch_front<2, 0>(p, s, what) : nl == 1 ? launch_front<2, 1>(p, s, what) : nl == 2 ? launch_front<2, 2>(p, s, what) : launch_front<2, 4>(p, s, what);
  return nl == 0 ? launch_front<1, 0>(p, s, what) : nl == 1 ? launch_front<1, 1>(p, s, what) : nl == 2 ? launch_front<1, 2>(p, s, what) : launch_front<1, 4>(p, s, what);
}
