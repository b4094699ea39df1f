// Device-side helpers shared by the gfx950 kernels: bf16 packing, MFMA wrappers and
// LDS operand loads.  wave = 64 lanes throughout.
//
// MFMA operand layouts used here (verified on hardware against a CPU matmul):
//   v_mfma_f32_16x16x32_bf16  A: lane l holds row (l%16),  k = 8*(l/16)+j   j<8
//                             B: lane l holds col (l%16),  k = 8*(l/16)+j
//                             C: lane l holds col (l%16),  rows 4*(l/16)+r  r<4
//   v_mfma_f32_32x32x16_bf16  A: lane l holds row (l%32),  k = 8*(l/32)+j
//                             B: lane l holds col (l%32),  k = 8*(l/32)+j
//                             C: lane l holds col (l%32),  rows 8*(r/4)+4*(l/32)+(r%4)  r<16
//   ds_read_b64_tr_b16        within each group of 16 lanes, lane i supplies the address of
//                             a 4-element row R_i; lane i receives { R_{4j + i/4}[i%4] : j<4 }.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace natsl {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;

typedef uint16_t bf16_t;  // raw bits

#define NATSL_DEVICE __device__ __forceinline__

NATSL_DEVICE float bf16_to_f32(bf16_t b) { return __uint_as_float(((unsigned)b) << 16); }

// round-to-nearest-even through the hardware conversion (v_cvt_pk_bf16_f32)
NATSL_DEVICE unsigned pack_bf16x2(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
  f32x2 v = {lo, hi};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2_t));
}

NATSL_DEVICE bf16_t f32_to_bf16(float f) { return (bf16_t)(pack_bf16x2(f, 0.f) & 0xffffu); }

// 8 fp32 -> one bf16x8 operand: slots 0..3 from a, 4..7 from b
NATSL_DEVICE bf16x8 pack8(const f32x4 a, const f32x4 b) {
  u32x4 w;
  w[0] = pack_bf16x2(a[0], a[1]);
  w[1] = pack_bf16x2(a[2], a[3]);
  w[2] = pack_bf16x2(b[0], b[1]);
  w[3] = pack_bf16x2(b[2], b[3]);
  return __builtin_bit_cast(bf16x8, w);
}

NATSL_DEVICE f32x4 mfma16(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
NATSL_DEVICE f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// 16-byte LDS / global loads of 8 bf16 as an MFMA operand
NATSL_DEVICE bf16x8 ld8(const bf16_t* p) { return *reinterpret_cast<const bf16x8*>(p); }

NATSL_DEVICE bf16x8 zero8() {
  u32x4 z = {0u, 0u, 0u, 0u};
  return __builtin_bit_cast(bf16x8, z);
}

// Transposing LDS read: see the layout note at the top of this file.
NATSL_DEVICE s16x4 lds_tr4(const bf16_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)(p));
}

NATSL_DEVICE bf16x8 join4(s16x4 lo, s16x4 hi) {
  typedef __attribute__((ext_vector_type(8))) short s16x8;
  s16x8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return __builtin_bit_cast(bf16x8, v);
}

// x[lane ^ 32] combined symmetrically: both returned words together hold {own, partner}.
NATSL_DEVICE float xhalf_max(float x) {
  u32x2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
NATSL_DEVICE float xhalf_sum(float x) {
  u32x2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The same for x[lane ^ 16].
NATSL_DEVICE float xrow_max(float x) {
  u32x2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
NATSL_DEVICE float xrow_sum(float x) {
  u32x2 r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// sums over the `lanes` adjacent lanes (a power of two, the same for the wave) that share a head row
NATSL_DEVICE void group_sum2(float& a, float& b, const int lanes) {
  auto add = [&](auto c) __attribute__((always_inline)) {
    a += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(a), decltype(c)::value, 0xf, 0xf, true));
    b += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(b), decltype(c)::value, 0xf, 0xf, true));
  };
  auto first = [&]() __attribute__((always_inline)) {
    add(std::integral_constant<int, 0xb1>{});    // lane ^ 1
    add(std::integral_constant<int, 0x4e>{});    // lane ^ 2
    add(std::integral_constant<int, 0x141>{});   // 7 - lane: the other four, which all hold their sum
  };
  if (lanes == 8) {
    first();
  } else if (lanes >= 16) {
    first();
    add(std::integral_constant<int, 0x140>{});   // 15 - lane
    if (lanes >= 32) {
      auto both = [](const u32x2 r) __attribute__((always_inline)) { return __uint_as_float(r[0]) + __uint_as_float(r[1]); };
      a = both(__builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(a), false, false));
      b = both(__builtin_amdgcn_permlane16_swap(__float_as_uint(b), __float_as_uint(b), false, false));
      if (lanes == 64) {
        a = xhalf_sum(a);
        b = xhalf_sum(b);
      }
    }
  } else {
    for (int d = 1; d < lanes; d <<= 1) {
      a += __shfl_xor(a, d);
      b += __shfl_xor(b, d);
    }
  }
}

// The layers' gates, shared by whole sequences and single steps: both write rows of the same cache, so both take the library's
// exponential (the hardware's differs from it by up to its argument in ulps, and g is kept and summed up in fp32).
NATSL_DEVICE float softplus_gate(const float x) { return x > 20.f ? x : log1pf(expf(x)); }
NATSL_DEVICE float sigmoid_gate(const float x) { return 1.f / (1.f + expf(-x)); }
// the selector's straight-through gradient: d0, d1 of the two types -> of their logits, through the softmax (rounded: as bf16 tensors hold it)
NATSL_DEVICE void select_grad(const float x0, const float x1, const bool rounded, float& d0, float& d1) {
  const float mx = fmaxf(x0, x1), e0 = expf(x0 - mx), e1 = expf(x1 - mx);
  float y0 = e0 / (e0 + e1), y1 = e1 / (e0 + e1);
  if (rounded) { y0 = bf16_to_f32(f32_to_bf16(y0)); y1 = bf16_to_f32(f32_to_bf16(y1)); }
  const float m = d0 * y0 + d1 * y1;
  d0 = y0 * (d0 - m);
  d1 = y1 * (d1 - m);
}

// The softmax of a head's two mixing logits, rounded to bf16: what the mixing layer's separate softmax returns
NATSL_DEVICE void mix_softmax(float& a, float& b) {
  const float mx = fmaxf(a, b), e0 = expf(a - mx), e1 = expf(b - mx);
  a = __uint_as_float(pack_bf16x2(e0 / (e0 + e1), 0.f) << 16);
  b = __uint_as_float(pack_bf16x2(e1 / (e0 + e1), 0.f) << 16);
}

// The sum of part[k][col] (n_col columns) over every TY-th k from `first` on, sixteen loads in flight: a thread's share of a column's sum.
template <int TY>
NATSL_DEVICE float column_share(const float* part, const int col, const int first, const int n_part, const int n_col) {
  const float* src = part + col;
  float acc = 0.f;
  int k = first;
  for (; k + 15 * TY < n_part; k += 16 * TY) {
    float v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = src[(size_t)(k + TY * u) * n_col];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 16; ++u) acc += v[u];
  }
  for (; k + 3 * TY < n_part; k += 4 * TY) {
    float v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = src[(size_t)(k + TY * u) * n_col];
#pragma unroll
    for (int u = 0; u < 4; ++u) acc += v[u];
  }
  for (; k < n_part; k += TY) acc += src[(size_t)k * n_col];
  return acc;
}

// Per-sequence descriptor for packed (variable-length) input; one row per sequence.
struct SeqRow {
  int bos;        // first token (flat index)
  int eos;        // one past the last token
  int bos_nats;   // first selector block (flat index)
  int chunk_off;  // number of 64-token chunks in earlier sequences
  int qtile_off;  // number of softmax query tiles in earlier sequences
  int pad0, pad1, pad2;
};

}  // namespace natsl
