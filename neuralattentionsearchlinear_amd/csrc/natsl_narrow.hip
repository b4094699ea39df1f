// The gradient behind a narrow weight (the mixing logits' layer: a few dozen rows), bound by the wide tensor's bytes:
//   X'[t][d] = sum_n Y'[t][n] W[n][d]   writes X' once
// bf16 operands, fp32 sums, one rounding.  Where the contraction is no multiple of 32 a library product takes two to three times as long as for
// one that is (36 rows of 1152 over 32768 tokens 36 us, 32 rows of 1024 19).
#include "natsl_device.h"
#include "natsl_host.h"

namespace natsl {

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

}  // namespace natsl

using namespace natsl;

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
