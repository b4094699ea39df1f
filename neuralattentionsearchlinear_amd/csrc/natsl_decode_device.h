// Device pieces of the decode-time kernels, shared by the operator entries (natsl_decode.hip) and the whole layer step
// (natsl_step.hip): attention of one query row over cached keys, and the linear branch's token recurrence.
#pragma once
#include <type_traits>

#include "natsl_device.h"
#include "../../include/natsl.h"

namespace natsl {

NATSL_DEVICE float ld_any(const void* p, int dtype, size_t i) {
  return dtype == NATSL_F32 ? reinterpret_cast<const float*>(p)[i] : bf16_to_f32(reinterpret_cast<const bf16_t*>(p)[i]);
}
NATSL_DEVICE void st_any(void* p, int dtype, size_t i, float x) {
  if (dtype == NATSL_F32) reinterpret_cast<float*>(p)[i] = x;
  else reinterpret_cast<bf16_t*>(p)[i] = f32_to_bf16(x);
}

// Sum over the 16 lanes of a row (every lane gets it): rotations inside the row ride on the additions, no LDS.
NATSL_DEVICE float row16_sum(float x) {
#define NATSL_ROR(n) x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x120 + n, 0xf, 0xf, false))
  NATSL_ROR(8); NATSL_ROR(4); NATSL_ROR(2); NATSL_ROR(1);
#undef NATSL_ROR
  return x;
}
NATSL_DEVICE float row16_max(float x) {
#define NATSL_ROR(n) x = fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x120 + n, 0xf, 0xf, false)))
  NATSL_ROR(8); NATSL_ROR(4); NATSL_ROR(2); NATSL_ROR(1);
#undef NATSL_ROR
  return x;
}

// Sum over the wave, in every lane: lanes 1, 2, 4, 8, 16, 32 apart are added in turn (the quad's permutations, the two mirrors, which by
// then hold the same as lanes 4 and 8 apart, and the swaps of rows and halves).  All of it on the vector unit: a step of one token is
// bound by what depends on what, and a shuffle through LDS has the latency of a dozen of these.  With the joins below done the same way
// step_one_kernel takes 10.9 us for 12.2 (340M geometry, one sequence of 800 tokens) and 17.3 for 18.4 (16 heads of 128/64, eight of 2000).
NATSL_DEVICE float wave_sum(float x) {
#define NATSL_DPP(c) x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), c, 0xf, 0xf, false))
  NATSL_DPP(0xb1); NATSL_DPP(0x4e); NATSL_DPP(0x141); NATSL_DPP(0x140);
#undef NATSL_DPP
  return xhalf_sum(xrow_sum(x));
}

// Values that waves of one launch hand to each other: stores that write through the XCD's own L2 and loads that do not trust it.
NATSL_DEVICE void st_agent(float* p, const float x) { __hip_atomic_store(p, x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
NATSL_DEVICE float ld_agent(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// ---------------------------------------------------------------------------------------------
// attention of one query row over cached keys
// ---------------------------------------------------------------------------------------------
// Bound by the bytes of K and V.  A wave takes chunks of KEYS_PER_CHUNK keys: 16 lanes share a row (16 or 8 bytes each in
// bf16), four rows per instruction, and ALL loads of a chunk, keys and values, are issued before the first is used (16 KiB in
// flight per wave at 128-wide bf16 heads).  8 sequences x 16 heads x 2066 keys with the recurrence beside it, 161 MB from HBM:
// 36 us = 4.5 TB/s a decode step, against 57 us when four rows were requested at a time and the values only after the softmax.
// A key row's four lane groups never meet until the end: the score of key (pass, group) sits in all 16 lanes of its group,
// which are the lanes that hold that key's value row, so neither scores nor probabilities go through LDS.  A chunk without a
// visible key is not loaded.
constexpr int KEYS_PER_CHUNK = 32;
constexpr int KEY_PASSES = KEYS_PER_CHUNK / 4;

template <int E, bool F32> struct RowPiece;             // E adjacent elements of a row, as loaded
template <> struct RowPiece<8, false> {
  u32x4 w;
  NATSL_DEVICE void load(const void* p, const size_t i) { w = *reinterpret_cast<const u32x4*>(reinterpret_cast<const bf16_t*>(p) + i); }
  NATSL_DEVICE float at(const int e) const { return __uint_as_float(e & 1 ? w[e >> 1] & 0xffff0000u : w[e >> 1] << 16); }
};
template <> struct RowPiece<4, false> {
  u32x2 w;
  NATSL_DEVICE void load(const void* p, const size_t i) { w = *reinterpret_cast<const u32x2*>(reinterpret_cast<const bf16_t*>(p) + i); }
  NATSL_DEVICE float at(const int e) const { return __uint_as_float(e & 1 ? w[e >> 1] & 0xffff0000u : w[e >> 1] << 16); }
};
template <int E> struct RowPiece<E, true> {
  f32x4 w[E / 4];
  NATSL_DEVICE void load(const void* p, const size_t i) {
#pragma unroll
    for (int j = 0; j < E / 4; ++j) w[j] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(p) + i + 4 * j);
  }
  NATSL_DEVICE float at(const int e) const { return w[e >> 2][e & 3]; }
};

template <int DK, int DV, bool F32>
struct AttnRow {
  static constexpr int EK = DK / 16, EV = DV / 16;      // elements of a key / value row per lane
  float q[EK], acc[EV], m, l;                            // m: running maximum (log2 units, the same in every lane); l, acc: this lane group's share

  NATSL_DEVICE void query(const void* qs, const size_t row, const float scale_log2) {
    const int sub = threadIdx.x & 15;
#pragma unroll
    for (int e = 0; e < EK; ++e) q[e] = ld_any(qs, F32 ? NATSL_F32 : NATSL_BF16, row * DK + EK * sub + e) * scale_log2;
  }
  NATSL_DEVICE void clear() {
#pragma unroll
    for (int e = 0; e < EV; ++e) acc[e] = 0.f;
    m = -INFINITY;
    l = 0.f;
  }
  NATSL_DEVICE void init(const void* qs, const size_t row, const float scale_log2) {
    query(qs, row, scale_log2);
    clear();
  }

  // keys k0 .. k0+31, rows of k_row / v_row elements behind element k_at / v_at; rows from n_keys on are not read (`vis` hides
  // them); vis: bit i = key k0+i visible, not all zero
  // Own::STEP: own.ready() is called between the requests and their use; keys from own.first on are the row in own.k / own.v instead
  // (a key that this launch itself adds to the cache).
  template <class Own>
  NATSL_DEVICE void chunk(const void* k, const void* v, const size_t k_at, const size_t v_at, const size_t k_row, const size_t v_row,
                          const int k0, const int n_keys, const unsigned vis, Own& own) {
    const int sub = threadIdx.x & 15, grp = (threadIdx.x & 63) >> 4;
    RowPiece<EK, F32> kr[KEY_PASSES];
    RowPiece<EV, F32> vr[KEY_PASSES];
#pragma unroll
    for (int i = 0; i < KEY_PASSES; ++i) kr[i].load(k, k_at + (size_t)min(k0 + 4 * i + grp, n_keys - 1) * k_row + EK * sub);
#pragma unroll
    for (int i = 0; i < KEY_PASSES; ++i) vr[i].load(v, v_at + (size_t)min(k0 + 4 * i + grp, n_keys - 1) * v_row + EV * sub);
    if constexpr (Own::STEP) {
      own.ready(*this);
      if (k0 + KEYS_PER_CHUNK > own.first) {
#pragma unroll
        for (int i = 0; i < KEY_PASSES; ++i)
          if (k0 + 4 * i + grp >= own.first) {
            kr[i].load(own.k, EK * sub);
            vr[i].load(own.v, EV * sub);
          }
      }
    }
    float s[KEY_PASSES];
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < KEY_PASSES; ++i) {
      float d = 0.f;
#pragma unroll
      for (int e = 0; e < EK; ++e) d += q[e] * kr[i].at(e);
      s[i] = row16_sum(d);
    }
    if (vis != 0xffffffffu) {
      const unsigned mine = vis >> grp;
#pragma unroll
      for (int i = 0; i < KEY_PASSES; ++i) s[i] = ((mine >> (4 * i)) & 1u) ? s[i] : -INFINITY;
    }
#pragma unroll
    for (int i = 0; i < KEY_PASSES; ++i) mx = fmaxf(mx, s[i]);
    mx = xhalf_max(xrow_max(mx));
    // Scores can be -inf for keys that are visible (infinite entries, an overflow of q.k): such keys weigh 0.  While there is no
    // other key the exponents are taken from 0, as -inf minus -inf would make NaN of everything that follows.
    const float mn = fmaxf(m, mx), ref = mn == -INFINITY ? 0.f : mn;
    const float alpha = __builtin_amdgcn_exp2f(m - ref);
    m = mn;
    l *= alpha;
#pragma unroll
    for (int e = 0; e < EV; ++e) acc[e] *= alpha;
#pragma unroll
    for (int i = 0; i < KEY_PASSES; ++i) {
      const float p = __builtin_amdgcn_exp2f(s[i] - ref);
      l += p;
#pragma unroll
      for (int e = 0; e < EV; ++e) acc[e] += p * vr[i].at(e);
    }
  }

  // the lane groups' shares together, in every lane
  NATSL_DEVICE void join_groups() {
    l = xhalf_sum(xrow_sum(l));
#pragma unroll
    for (int e = 0; e < EV; ++e) acc[e] = xhalf_sum(xrow_sum(acc[e]));
  }
};

// What a query may see: a byte per key, or (mask == null) the generation cache's own bookkeeping -- the first n_kept blocks of
// `block` keys where the (sequence, block, mask head) flag is set, then the incomplete block's keys up to the query's own.
struct AttnParams {
  const void* q; const void* k; const void* v; const uint8_t* mask; void* o;
  int B, TQ, TK, HQ, HKV, HM, dtype;
  float scale_log2;
  int nsplit;        // workgroups per query, each owning every nsplit-th group of chunks (one per wave)
  float* partials;   // [B, TQ, HQ, nsplit, 2 + DV] running (max, sum, accumulator) of each split; null: one split, o is written
  size_t k_bs, v_bs; // elements from one sequence's keys / values to the next (TK * HKV * D when dense)
  const uint8_t* valid; int valid_bs, n_kept, block, n_in, own_visible;   // valid[b][block][HM], valid_bs bytes per sequence
};

struct CachedRows { static constexpr bool STEP = false; };   // query and keys are all in memory

// One workgroup of NW waves works on split `split` of query (b, tq, hq); wave 0 writes the result.  Own::STEP (above): the query comes
// from own.ready(), called once with or without a visible chunk, memory holds the keys before own.first only, and the result goes to
// the partials for another wave of this launch.
template <int DK, int DV, bool F32, int NW, class Own>
NATSL_DEVICE void attend(const AttnParams& p, const int b, const int tq, const int hq, const int split, Own&& own) {
  constexpr bool STEP = std::remove_reference_t<Own>::STEP;
  constexpr int CPL = DV / 64, EV = DV / 16;
  __shared__ float sm_m[NW], sm_l[NW], sm_acc[NW][DV];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hkv = STEP ? hq : hq / (p.HQ / p.HKV), hm = hq / (p.HQ / p.HM);
  const size_t row = ((size_t)b * p.TQ + tq) * p.HQ + hq;
  AttnRow<DK, DV, F32> r;
  if constexpr (STEP) r.clear();
  else r.init(p.q, row, p.scale_log2);
  const uint8_t* mrow = !STEP && p.mask ? p.mask + (((size_t)b * p.HM + hm) * p.TQ + tq) * p.TK : nullptr;
  const size_t k_at = (size_t)b * p.k_bs + (size_t)hkv * DK, v_at = (size_t)b * p.v_bs + (size_t)hkv * DV;
  const int first = KEYS_PER_CHUNK * (split * NW + wave), stride = KEYS_PER_CHUNK * NW * p.nsplit;   // the wave's chunks
  auto chunk = [&](const int k0, const unsigned vis) __attribute__((always_inline)) {
    r.chunk(p.k, p.v, k_at, v_at, (size_t)p.HKV * DK, (size_t)p.HKV * DV, k0, STEP ? max(p.TK - 1, 1) : p.TK, vis, own);
  };
  if (mrow) {
    for (int k0 = first; k0 < p.TK; k0 += stride) {
      const int key = k0 + (lane & 31);
      const unsigned vis = (unsigned)__ballot(key < p.TK && mrow[min(key, p.TK - 1)] != 0);
      if (vis != 0u) chunk(k0, vis);                     // (wave-uniform)
    }
  } else {
    // lane i looks at the i-th of the wave's next 64 chunks, so that their flags are one round trip
    const int own_at = p.n_kept * p.block;              // the incomplete block's first key
    const int end = min(own_at + p.n_in + tq + 1, p.TK);  // behind the last key that the query may see there
    // (the flag is read without a branch, a wave's further ones at the end of the loop: what the wave asks for itself, own.request(), goes
    // out behind the first ones and ahead of the wait for them: step_one_kernel 10.4 -> 9.9 us, 340M geometry, one sequence of 800 tokens, and
    // 17.2 -> 16.7, 16 heads of 128/64, eight of 2000)
    const uint8_t* valid = p.valid + (size_t)b * p.valid_bs + hm;
    auto flag_of = [&](const int base) __attribute__((always_inline)) -> uint8_t {
      return valid[(size_t)((unsigned)min(base + lane * stride, max(own_at - 1, 0)) / (unsigned)p.block) * p.HM];
    };
    uint8_t flag = flag_of(first);
    if constexpr (STEP) own.request();
    for (int base = first; base < p.TK;) {
      const int mine = base + lane * stride;
      for (unsigned long long todo = __ballot(mine < own_at ? flag != 0 : p.own_visible && mine < end); todo; todo &= todo - 1) {
        const int k0 = base + __builtin_ctzll(todo) * stride, n = end - k0;
        chunk(k0, k0 < own_at || n >= 32 ? 0xffffffffu : (1u << n) - 1u);
      }
      base += 64 * stride;
      if (base < p.TK) flag = flag_of(base);
    }
  }
  if constexpr (STEP) own.ready(r);
  // the waves' shares together
  r.join_groups();
  if (lane == 0) { sm_m[wave] = r.m; sm_l[wave] = r.l; }
  if (lane < 16) {
#pragma unroll
    for (int e = 0; e < EV; ++e) sm_acc[wave][EV * lane + e] = r.acc[e];
  }
  __syncthreads();
  if (wave != 0) return;
  float m = -INFINITY, l = 0.f, o[CPL];
#pragma unroll
  for (int j = 0; j < CPL; ++j) o[j] = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) m = fmaxf(m, sm_m[w]);
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float f = sm_m[w] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(sm_m[w] - m);
    l += f * sm_l[w];
#pragma unroll
    for (int j = 0; j < CPL; ++j) o[j] += f * sm_acc[w][CPL * lane + j];
  }
  if (p.partials) {
    float* dst = p.partials + (row * p.nsplit + split) * (2 + DV);
    if constexpr (STEP) {
      if (lane == 0) { st_agent(dst, m); st_agent(dst + 1, l); }
#pragma unroll
      for (int j = 0; j < CPL; ++j) st_agent(dst + 2 + CPL * lane + j, o[j]);
      return;
    }
    if (lane == 0) { dst[0] = m; dst[1] = l; }
#pragma unroll
    for (int j = 0; j < CPL; ++j) dst[2 + CPL * lane + j] = o[j];
    return;
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int j = 0; j < CPL; ++j) st_any(p.o, F32 ? NATSL_F32 : NATSL_BF16, row * DV + CPL * lane + j, o[j] * inv);
}

// (m, l, acc) of the splits (at most 64) of one query row, written by one workgroup each as [2 + DV] floats: the joined, normalised
// columns CPL*lane.. of the row; a row that saw no key gives 0.  Lane s holds split s's weight, so that the maxima are one round
// trip to memory and the partial rows another.
// The first rows are requested with the maxima.  AGENT: the partials come from this launch.
template <int DV, bool AGENT = false>
NATSL_DEVICE void join_splits(const float* src, const int nsplit, float* o) {
  constexpr int CPL = DV / 64, U = AGENT ? 8 : 4;
  const int lane = threadIdx.x & 63;
  auto ld = [](const float* p) __attribute__((always_inline)) { return AGENT ? ld_agent(p) : *p; };
  const float ms = lane < nsplit ? ld(src + lane * (2 + DV)) : -INFINITY, ls = lane < nsplit ? ld(src + lane * (2 + DV) + 1) : 0.f;
  float v[U][CPL];
  auto rows = [&](const int s) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < CPL; ++j) v[u][j] = ld(src + min(s + u, nsplit - 1) * (2 + DV) + 2 + CPL * lane + j);
  };
  rows(0);
  float m = ms;
  m = row16_max(xrow_max(xhalf_max(m)));
  const float f = ms == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ms - m);
  float l = f * ls;
  l = row16_sum(xrow_sum(xhalf_sum(l)));
#pragma unroll
  for (int j = 0; j < CPL; ++j) o[j] = 0.f;
  for (int s = 0; s < nsplit; s += U) {
    if (s > 0) rows(s);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float fu = s + u < nsplit ? __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), s + u)) : 0.f;
#pragma unroll
      for (int j = 0; j < CPL; ++j) o[j] += fu * v[u][j];
    }
  }
  const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
  for (int j = 0; j < CPL; ++j) o[j] *= inv;
}

// ---------------------------------------------------------------------------------------------
// the linear branch token by token on a cached state
// ---------------------------------------------------------------------------------------------
struct RecurrentParams {
  const void* q; const void* k; const void* v; const float* g; const float* g_cumsum; const void* beta;
  const float* h0; float* hcur; void* o; float* ht;
  const void* types; int types_dtype; const int32_t* n_in_block;
  int N, T, H, HN, V, block, dtype;
  float scale; int decay, l2norm, n_in_block_scalar;
  int query_only;          // outputs from the decayed block-start state, no state update (the 'attn' mode of decode)
  int kv_stride, kv_first; // token t of sequence n is row n * kv_stride + kv_first + t of k, v, g, beta (q, o: n * T + t)
  int fresh_start;         // hcur is write-only: the block starts from h0
  int aligned;             // q and k start on 16 bytes
  float* g_cumsum_out;     // g_cumsum + sum of the tokens' g, or null
};

// R consecutive elements of a row as floats, 16 bytes per load where every row starts on 16 bytes
template <int R>
NATSL_DEVICE void ld_row(const void* p, const int dtype, const bool aligned, const size_t i, float* f) {
  if (!aligned) {
#pragma unroll
    for (int r = 0; r < R; ++r) f[r] = ld_any(p, dtype, i + r);
  } else if (dtype == NATSL_BF16) {
    const bf16_t* s = reinterpret_cast<const bf16_t*>(p) + i;
#pragma unroll
    for (int j = 0; j < R / 8; ++j) {
      const u32x4 w = *reinterpret_cast<const u32x4*>(s + 8 * j);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f[8 * j + 2 * e] = __uint_as_float(w[e] << 16);
        f[8 * j + 2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
      }
    }
  } else {
    const float* s = reinterpret_cast<const float*>(p) + i;
#pragma unroll
    for (int j = 0; j < R / 4; ++j) {
      const f32x4 w = *reinterpret_cast<const f32x4*>(s + 4 * j);
#pragma unroll
      for (int e = 0; e < 4; ++e) f[4 * j + e] = w[e];
    }
  }
}

// Where recurrent_columns takes a token from and puts its output: the tensors of the parameters.
template <int DK>
struct TokenRows {
  static constexpr int R = DK / 4;
  template <bool DELTA>
  NATSL_DEVICE void token(const RecurrentParams& p, const int n, const int t, const int h, const int kq, const int vc, float* kk, float* qq, float& gt,
                          float& bt, float& vt) const {
    const size_t tok = (size_t)n * p.T + t, row = (size_t)n * p.kv_stride + p.kv_first + t;
    ld_row<R>(p.k, p.dtype, p.aligned, (row * p.H + h) * DK + kq * R, kk);
    ld_row<R>(p.q, p.dtype, p.aligned, (tok * p.H + h) * DK + kq * R, qq);
    gt = p.g[row * p.H + h];
    bt = DELTA ? ld_any(p.beta, p.dtype, row * p.H + h) : 1.f;
    vt = ld_any(p.v, p.dtype, (row * p.H + h) * p.V + vc);
  }
  NATSL_DEVICE void out(const RecurrentParams& p, const int n, const int t, const int h, const int vc, const float x) const {
    st_any(p.o, p.dtype, (((size_t)n * p.T + t) * p.H + h) * p.V + vc, x);
  }
  NATSL_DEVICE void done(int, int, int) const {}          // all outputs are written, the states are not
};

// One wave owns the state slice S[0:K][16 columns] of one (sequence, head): lane = (kq, col) with kq = lane/16 the quarter of
// the K rows it keeps in registers (K/4 floats) and col = lane%16.  Sums over K are K/4 in-lane terms plus two cross-lane
// steps; no LDS, no barriers.  Bound by the state's bytes (read and written once); the block-start state is only read by the
// step that completes a block.  All of a lane's state loads are in flight before the token's k and q arrive.
// DELTA = false is the Mamba form (src/nats/ops/mamba/fused_recurrent.py:150-178): S += k v^T, no beta, no norms.
template <int DK, bool DELTA, class Tokens = TokenRows<DK>>
NATSL_DEVICE void recurrent_columns(const RecurrentParams& p, const int nh, const int col16, Tokens&& tokens = Tokens()) {
  constexpr int R = DK / 4;  // state rows per lane
  const int lane = threadIdx.x & 63;
  const int kq = lane >> 4, col = lane & 15;
  const int n = nh / p.H, h = nh % p.H;
  const int vc = col16 * 16 + col;
  const int hn = h / (p.H / p.HN);
  const size_t s_at = ((size_t)nh * DK + kq * R) * p.V + vc;

  float S[R];
  {
    const float* src = p.query_only ? p.hcur : p.h0;
    if (src) {
#pragma unroll
      for (int r = 0; r < R; ++r) S[r] = src[s_at + (size_t)r * p.V];
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) S[r] = 0.f;
    }
  }
  float gcum = p.g_cumsum ? p.g_cumsum[nh] : 0.f;
  const int n_in = p.n_in_block ? p.n_in_block[n] : p.n_in_block_scalar;
  const int n_tok = min(p.T, p.block - n_in);  // fused_recurrent.py:144
  const bool completes = n_in + p.T >= p.block;
  if (p.query_only) {
    // The mode in which the linear operator does not run on the incomplete block: a token reads the state that entered
    // the block, decayed by the block's g up to and including itself (what the chunked forward without its intra-chunk
    // term gives, and what the reference's UPDATE_HS_FOR_EACH_ITER = False branch gives for a one-token step,
    // fused_recurrent.py:156-201 as called at mixed_attn_gdn.py:510-527); nothing is written back.
    const float e0 = __expf(gcum);
#pragma unroll
    for (int r = 0; r < R; ++r) S[r] *= e0;
    for (int t = 0; t < n_tok; ++t) {
      const size_t tok = (size_t)n * p.T + t;
      float qq[R];
      ld_row<R>(p.q, p.dtype, p.aligned, (tok * p.H + h) * DK + kq * R, qq);
      float rq = 1.f;
      if (DELTA && p.l2norm) {
        float sq = 0.f;
#pragma unroll
        for (int r = 0; r < R; ++r) sq += qq[r] * qq[r];
        sq = xhalf_sum(xrow_sum(sq));
        rq = 1.f / sqrtf(sq + 1e-6f);
      }
      const float eg = __expf(p.g[((size_t)n * p.kv_stride + p.kv_first + t) * p.H + h]);
      float hq = 0.f;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        S[r] *= eg;
        hq += S[r] * qq[r];
      }
      hq = xhalf_sum(xrow_sum(hq));
      if (kq == 0) st_any(p.o, p.dtype, (tok * p.H + h) * p.V + vc, hq * rq * p.scale);
    }
    return;
  }
  if (p.fresh_start && !completes) {
#pragma unroll
    for (int r = 0; r < R; ++r) p.hcur[s_at + (size_t)r * p.V] = S[r];
  }

  for (int t = 0; t < n_tok; ++t) {
    float kk[R], qq[R], gt, bt, vt;
    tokens.template token<DELTA>(p, n, t, h, kq, vc, kk, qq, gt, bt, vt);
    if (DELTA && p.l2norm) {
      float sk = 0.f, sq = 0.f;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        sk += kk[r] * kk[r];
        sq += qq[r] * qq[r];
      }
      sk = xhalf_sum(xrow_sum(sk));
      sq = xhalf_sum(xrow_sum(sq));
      const float rk = 1.f / sqrtf(sk + 1e-6f), rq = 1.f / sqrtf(sq + 1e-6f);  // :165-169
#pragma unroll
      for (int r = 0; r < R; ++r) { kk[r] *= rk; qq[r] *= rq; }
    }
    const float eg = __expf(gt);
    if (p.decay || p.g_cumsum_out) gcum += gt;                  // :183-184
    float hk = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      S[r] *= eg;                                               // :182
      hk += S[r] * kk[r];
    }
    hk = xhalf_sum(xrow_sum(hk));
    const float dv = DELTA ? bt * (vt - hk) : vt;               // :195
    float hq = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      S[r] += kk[r] * dv;                                       // :196
      hq += S[r] * qq[r];
    }
    hq = xhalf_sum(xrow_sum(hq));
    if (kq == 0) tokens.out(p, n, t, h, vc, hq * p.scale);      // :199-201
  }
  tokens.done(n, h, vc);
  if (p.g_cumsum_out && vc == 0 && kq == 0) p.g_cumsum_out[nh] = gcum;
  // the selector block is complete: a block not typed linear restores the state it started from
  // (times the block's total decay when asked), and that becomes the next block's start (:343-352)
  if (completes) {
    const size_t ti = ((size_t)n * p.HN + hn) * 2 + 1;
    const bool is_delta = rintf(ld_any(p.types, p.types_dtype, ti)) == 1.0f;
    if (!is_delta) {
      const float f = p.decay ? __expf(gcum) : 1.f;
      const float* start = p.fresh_start ? p.h0 : p.hcur;
#pragma unroll
      for (int r = 0; r < R; ++r) S[r] = start ? start[s_at + (size_t)r * p.V] * f : 0.f;
    }
#pragma unroll
    for (int r = 0; r < R; ++r) p.hcur[s_at + (size_t)r * p.V] = S[r];
  }
  if (p.ht) {
#pragma unroll
    for (int r = 0; r < R; ++r) p.ht[s_at + (size_t)r * p.V] = S[r];
  }
}

// Both halves of a decode step in one launch (natsl_decode.hip); K, V: the linear branch's widths in r, KA, VA the attention's.
int launch_attend_and_recur(const char* what, const AttnParams& a, const RecurrentParams& r, bool delta, int K, int KA, int VA, hipStream_t s);
constexpr int ATTEND_MAX_SPLITS = 16;
int attend_splits(int queries, int TK);   // splits per query of that launch, at most ATTEND_MAX_SPLITS

}  // namespace natsl
