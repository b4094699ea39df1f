// Products with a narrow weight (the mixing logits' layer: a few dozen rows), bound by the wide tensor's bytes:
//   narrow_fwd_kernel   Y[t][n] = sum_d X[t][d] W[n][d]     reads X once
//   narrow_bwd_kernel   X'[t][d] = sum_n Y'[t][n] W[n][d]   writes X' once
// bf16 operands, fp32 sums, one rounding.  A library product takes 256 x 16 tiles for the first (23 us for 24 x 768 over 32768 tokens, 50 MB)
// and 192 x 256 tiles with a contraction of 24 for the second (36 us).
#include "natsl_device.h"
#include "natsl_host.h"

namespace natsl {

constexpr int NARROW_MAX = 64;                 // rows of the weight
constexpr int NARROW_LDS = 160 * 1024;

struct NarrowParams {
  const bf16_t *x, *w;                         // x: the wide tensor (forward) or the narrow gradient (backward)
  bf16_t* y;
  long long rows;
  int D, N;
};

// Two waves take 32 tokens, half of the contraction each; the weight lies in LDS, row n's 16-byte segment s at s ^ (n % 16), so that the 32
// rows that an operand read names meet all banks.  A wave requests up to 24 of a token's segments before the first is used.
template <int NB>
__global__ __launch_bounds__(256) void narrow_fwd_kernel(const NarrowParams p) {
  extern __shared__ __align__(1024) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l32 = lane & 31, hf = lane >> 5;
  const long long t = (long long)blockIdx.x * 64 + 32 * (wave >> 1) + l32;
  const bf16_t* xr = p.x + (size_t)(t < p.rows ? t : p.rows - 1) * p.D + 8 * hf;
  constexpr int AHEAD = 24;
  bf16x8 xb[AHEAD];
  const int half = p.D / 32, first = (wave & 1) * half, steps = first + half;   // this wave's steps of 16 (a multiple of 4)
  auto load = [&](const int s0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) xb[i] = ld8(xr + 16 * min(s0 + i, steps - 1));
  };
  load(first);
  const int segs = p.D / 8;
  for (int i = threadIdx.x; i < p.N * segs; i += 256) {
    const int n = i / segs, s = i - n * segs;
    *reinterpret_cast<u32x4*>(smem + (size_t)n * p.D * 2 + 16 * (s ^ (n & 15))) = *reinterpret_cast<const u32x4*>(p.w + (size_t)i * 8);
  }
  __syncthreads();
  f32x16 acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[b][r] = 0.f;
  for (int s0 = first; s0 < steps; s0 += AHEAD) {
    if (s0 > first) load(s0);
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      if (s0 + i >= steps) break;
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int n = min(32 * b + l32, p.N - 1);   // (rows behind the weight: the last one again, never stored)
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(smem + (size_t)n * p.D * 2 + 16 * ((2 * (s0 + i) + hf) ^ (n & 15)));
        acc[b] = mfma32(a, xb[i], acc[b]);
      }
    }
  }
  __syncthreads();                             // (the weight has been read: its place takes the second halves' sums)
  f32x16* sums = reinterpret_cast<f32x16*>(smem) + (wave >> 1) * NB * 64;
  if (wave & 1)
#pragma unroll
    for (int b = 0; b < NB; ++b) sums[b * 64 + lane] = acc[b];
  __syncthreads();
  if ((wave & 1) || t >= p.rows) return;
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b] += sums[b * 64 + lane];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int n = 32 * b + 8 * q + 4 * hf;
      if (n < p.N)                             // (N is a multiple of 4)
        *reinterpret_cast<u32x2*>(p.y + t * p.N + n) = (u32x2){pack_bf16x2(acc[b][4 * q], acc[b][4 * q + 1]), pack_bf16x2(acc[b][4 * q + 2], acc[b][4 * q + 3])};
    }
}

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
        h[i] = n < p.N ? *reinterpret_cast<const u32x2*>(p.x + t * p.N + n) : (u32x2){0u, 0u};
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
      if (t0 + r < p.rows && col < p.D) *reinterpret_cast<u32x4*>(p.y + (size_t)(t0 + r) * p.D + col) = w;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

static int narrow_check(NarrowParams& p, const void* x, const void* w, void* y, int64_t rows, int D, int N, const char* what) {
  if (!x || !w || !y) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (rows <= 0 || D <= 0 || N <= 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  if (N > NARROW_MAX || N % 4 || D % 128 || (long long)N * D * 2 > NARROW_LDS || rows > (1ll << 32))
    return fail(NATSL_ERR_UNSUPPORTED, "%s: N=%d (a multiple of 4 up to %d), D=%d (a multiple of 128, N D up to %d)", what, N, NARROW_MAX, D, NARROW_LDS / 2);
  if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)y) & 15) return fail(NATSL_ERR_INVALID, "%s: tensors must start on 16 bytes", what);
  p.x = (const bf16_t*)x; p.w = (const bf16_t*)w; p.y = (bf16_t*)y; p.rows = rows; p.D = D; p.N = N;
  return NATSL_OK;
}

}  // namespace natsl

using namespace natsl;

extern "C" int natsl_narrow_linear(const void* x, const void* w, void* y, int64_t rows, int D, int N, natsl_stream_t stream) {
  const char* what = "natsl_narrow_linear";
  NarrowParams p;
  int rc = narrow_check(p, x, w, y, rows, D, N, what);
  if (rc != NATSL_OK) return rc;
  auto kern = N > 32 ? narrow_fwd_kernel<2> : narrow_fwd_kernel<1>;
  const size_t sums = (size_t)(N > 32 ? 2 : 1) * 2 * 64 * 64, lds = (size_t)N * D * 2 > sums ? (size_t)N * D * 2 : sums;
  static std::atomic<unsigned long long> reserved[2];
  if ((rc = reserve_lds(reinterpret_cast<const void*>(kern), reserved[N > 32], NARROW_LDS, what)) != NATSL_OK) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)((rows + 63) / 64)), dim3(256), lds, reinterpret_cast<hipStream_t>(stream), p);
  return check_launch(what);
}

extern "C" int natsl_narrow_linear_bwd(const void* dy, const void* w, void* dx, int64_t rows, int D, int N, natsl_stream_t stream) {
  const char* what = "natsl_narrow_linear_bwd";
  NarrowParams p;
  int rc = narrow_check(p, dy, w, dx, rows, D, N, what);
  if (rc != NATSL_OK) return rc;
  const dim3 grid((unsigned)((rows + 32 * NARROW_TILES - 1) / (32 * NARROW_TILES)), (unsigned)cdiv(D, 256));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  switch (cdiv(N, 16)) {
    case 1: hipLaunchKernelGGL(narrow_bwd_kernel<1>, grid, dim3(256), 0, s, p); break;
    case 2: hipLaunchKernelGGL(narrow_bwd_kernel<2>, grid, dim3(256), 0, s, p); break;
    case 3: hipLaunchKernelGGL(narrow_bwd_kernel<3>, grid, dim3(256), 0, s, p); break;
    default: hipLaunchKernelGGL(narrow_bwd_kernel<4>, grid, dim3(256), 0, s, p); break;
  }
  return check_launch(what);
}
