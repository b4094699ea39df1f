// The linear branches' work per 64-token chunk that does not depend on the running state, as device code of 256 threads: of kernels of their own
// (natsl_linear.hip, whose head says what they leave for the scan) and, in small calls, of the softmax tiles' launch (natsl_softmax.hip).
#pragma once
#include "../../include/natsl.h"
#include "natsl_device.h"

namespace natsl {

struct LinearParams {
  const bf16_t* q;
  const bf16_t* k;
  const bf16_t* v;
  const float* g;
  const bf16_t* beta;
  const float* h0;
  bf16_t* o;
  float* ht;
  float* hs;      // state entering each sequence's last selector block (optional)
  float* gs;      // sum of g over that block, [N,H] (optional)
  bf16_t* s_out;  // the state entering every chunk, transposed: [chunk][H][V][K] bf16 (optional; for the backward)
  bf16_t* vn_out; // v_new of every token, [tokens][H][V] bf16 (optional, delta rule only; for the backward)
  const void* types;
  int types_dtype;
  const SeqRow* seqs;
  int n_seqs;
  int B, T, H, HN, K, V, TN, block;
  int nt;            // chunks per sequence (regular batch)
  int total_chunks;
  float scale;
  int flags;
  bf16_t* ws_tm;
  bf16_t* ws_p;
  float* ws_sc;
};

constexpr int C = 64;

// =============================================================================================
// prep
// =============================================================================================
// acc + the squares of two bf16
NATSL_DEVICE float sum_squares(const unsigned w, const float acc) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  const bf16x2 x = __builtin_bit_cast(bf16x2, w);
  return __builtin_amdgcn_fdot2_f32_bf16(x, x, acc, false);
}

// PF ("P formed by the scan"): the kernel reads k only -- no q tile, no q k^T product, no P -- and leaves TmB and six scale
// vectors; the two extra ones (in the first 512 bytes of the unit's P area) are the exponents the scan needs to form
// P_ij = rq_i (q_i . k_j) exp2(gq_i - gk_j):   gk = gamma log2(e) - log2 rk,   gq = gamma log2(e) + log2 scale,
// and sq comes without its 1/|q| factor (the scan takes the row norms of q from the tile it holds anyway).
//
// Bound by the instructions of its phases and by the barriers between them (63 % of the wave cycles wait; 2.2 TB/s), so what counts is
// their number and how many workgroups share a CU: six with PF (26 KB of LDS, 78 registers).  B8 T8192 H16 d128: 124 us; with row
// norms by separate conversions, branches around the exponentials, the substitution in 16 lanes of every wave and five workgroups a
// CU 137.  A loop over units with the next rows requested ahead takes registers from it: 150 us at four workgroups.  The gates' and the type's
// round trips behind the tiles' instead of beside them, and gamma formed by one wave before the first barrier instead of by the idle one
// behind it: 46.5 us for 42.4 (B4 T4096 H16, without PF), 122 for 117 (B8 T8192 H16, with).
// LDS: region0, PREP_REGION bytes (the q, k tiles are dead once the Gram products are done; the solve reuses their space), and four rows of C floats, all
// aligned to 16 bytes.
template <int DK, bool DELTA, bool PF>
constexpr int PREP_REGION = DELTA && 20 * 16 * 20 * 4 > (PF ? 1 : 2) * C * (DK + 8) * 2 ? 20 * 16 * 20 * 4 : (PF ? 1 : 2) * C * (DK + 8) * 2;   // bytes
template <int DK, bool DELTA, bool PF>
__device__ __attribute__((always_inline)) inline void linear_prep(const LinearParams& p, const unsigned wg, unsigned char* region0, float* gam, float* rq, float* rk,
                                                                  float* bet) {
  static_assert(DELTA || !PF, "the Mamba form has its own prep");
  constexpr int KP = DK + 8;   // bf16 row pitch
  constexpr int KL = DK / 32;  // 16-byte loads per thread per tile
  // The 64x64 fp32 matrices of the solve are kept as their lower 16x16 blocks, rows of BP floats.  A = strictly lower system matrix, ten
  // blocks, (i, k) at index i(i+1)/2 + k; its diagonal blocks are replaced by those of X = (I+A)^-1.  Xb = the six others of X,
  // (i, k) at i(i-1)/2 + k.  Xt = the diagonal blocks of X transposed (an MFMA B operand with one 16-byte read).
  constexpr int BP = 20, BLK = 16 * BP, NBLK = 10, NOFF = 6;
  constexpr int TILE_BYTES = (PF ? 1 : 2) * C * KP * 2, SOLVE_BYTES = (NBLK + NOFF + 4) * BLK * 4;
  static_assert(PREP_REGION<DK, DELTA, PF> >= TILE_BYTES && (!DELTA || PREP_REGION<DK, DELTA, PF> >= SOLVE_BYTES), "the tiles, and in their place the solve");
  bf16_t* Qs = reinterpret_cast<bf16_t*>(region0);
  bf16_t* Ks = PF ? Qs : Qs + C * KP;   // (no q tile with PF)
  float* Ab = reinterpret_cast<float*>(region0);
  float* Xb = Ab + NBLK * BLK;
  float* Xt = Xb + NOFF * BLK;
  auto bidx = [](int i, int k) { return i * (i + 1) / 2 + k; };
  auto xblk = [&](int i, int k) { return i == k ? Ab + bidx(i, i) * BLK : Xb + (i * (i - 1) / 2 + k) * BLK; };

  // the waves' shares differ: workgroups that are on a CU together give a share to different SIMDs
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = ((__builtin_amdgcn_readfirstlane(tid >> 6)) + (int)(wg >> 8)) & 3;
  const int gc = wg / p.H, h = wg % p.H;
  int bos, len, c, bos_nats;
  if (p.seqs == nullptr) {
    const int n = gc / p.nt;
    c = gc - n * p.nt;
    bos = n * p.T;
    len = p.T;
    bos_nats = n * p.TN;
  } else {
    int n = 0;
    for (int i = 1; i < p.n_seqs; ++i)
      if (p.seqs[i].chunk_off <= gc) n = i;
    c = gc - p.seqs[n].chunk_off;
    bos = p.seqs[n].bos;
    len = p.seqs[n].eos - bos;
    bos_nats = p.seqs[n].bos_nats;
  }
  const int t0 = c * C;
  const bool l2 = (p.flags & NATSL_QK_L2NORM) != 0;

  // ---- the per-token inputs and the chunk's type, which one wave each uses further down: asked for here, in every wave and as they lie, so that
  // their round trips to memory are the tiles' own
  const bool tok_ok = t0 + lane < len;
  const size_t gi = (size_t)(bos + min(t0 + lane, len - 1)) * p.H + h;
  const float g_tok = p.g[gi];
  const bf16_t b_tok = DELTA ? p.beta[gi] : (bf16_t)0;
  bf16_t type_lo, type_hi;

  // ---- load q, k tiles; row sums of squares from the registers just loaded -----------------
  {
    const int row = tid >> 2, seg = tid & 3;
    const bool ok = t0 + row < len;
    const size_t off = ((size_t)(bos + t0 + row) * p.H + h) * DK;
    const u32x4* qr = reinterpret_cast<const u32x4*>(p.q + off);
    const u32x4* kr = reinterpret_cast<const u32x4*>(p.k + off);
    const u32x4 z = {0u, 0u, 0u, 0u};
    float sq = 0.f, sk = 0.f;
    u32x4 qa[KL], kb[KL];
#pragma unroll
    for (int i = 0; i < KL; ++i) {
      qa[i] = (ok && !PF) ? qr[seg + 4 * i] : z;
      kb[i] = ok ? kr[seg + 4 * i] : z;
    }
    const int type_size = p.types_dtype == NATSL_F32 ? 4 : 2;
    const char* type_at = reinterpret_cast<const char*>(p.types) + (((size_t)(bos_nats + t0 / p.block) * p.HN + h / (p.H / p.HN)) * 2 + 1) * type_size;
    type_lo = *reinterpret_cast<const bf16_t*>(type_at);
    type_hi = *reinterpret_cast<const bf16_t*>(type_at + type_size - 2);
#pragma unroll
    for (int i = 0; i < KL; ++i) {
      const u32x4 a = qa[i], b = kb[i];
      if (!PF) *reinterpret_cast<u32x4*>(Qs + row * KP + (seg + 4 * i) * 8) = a;
      *reinterpret_cast<u32x4*>(Ks + row * KP + (seg + 4 * i) * 8) = b;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (!PF) sq = sum_squares(a[j], sq);
        sk = sum_squares(b[j], sk);
      }
    }
    // (lanes 1 and 2 apart, by the quad's permutations)
    auto quad_sum = [](float x) __attribute__((always_inline)) -> float {
      x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xb1, 0xf, 0xf, false));
      return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4e, 0xf, 0xf, false));
    };
    sq = quad_sum(sq);
    sk = quad_sum(sk);
    if (seg == 0) {
      rq[row] = (l2 && !PF) ? rsqrtf(sq + 1e-6f) : 1.f;
      rk[row] = l2 ? rsqrtf(sk + 1e-6f) : 1.f;
    }
  }
  __syncthreads();

  const size_t unit = (size_t)gc * p.H + h;
  bf16_t* Pout = p.ws_p + unit * (C * C);
  bf16_t* Tout = p.ws_tm + unit * (C * C);
  float* Sout = p.ws_sc + unit * (4 * C);

  // ---- Gram products on the matrix cores: wave w owns the 32x32 tile (w/2, w%2) ------------
  // P and TmB are stored as the scan kernel's MFMA A operands (16x16x32: 16 rows x 32 contraction tokens), 1 KiB each,
  // operand (t, s) = rows 16t.., tokens 32s.. at index 2t + s; in it, scan-lane (row i%16, group g) finds its 16 bytes
  // at (16 g + i%16) * 16.  The scan feeds the other operand from accumulator registers, where lane group g holds
  // tokens 4g..4g+3 of a 16-token tile, so slot j of group g stands for token 32s + 16(j/4) + 4g + j%4.
  // Operands (0,1) and (1,1) lie above the diagonal: never written, never read.
  {
    const int ti = wave >> 1, tj = wave & 1, l32 = lane & 31, hf = lane >> 5;
    const int i = 32 * ti + l32;  // P row owned by this lane
    bf16_t* prow = Pout + ((size_t)((2 * (i >> 4) + tj) * 64 + (i & 15))) * 8;
    f32x16 gk, gq;
    if (ti >= tj) {
#pragma unroll
      for (int r = 0; r < 16; ++r) gk[r] = gq[r] = 0.f;
#pragma unroll
      for (int s = 0; s < DK / 16; ++s) {
        const bf16x8 kb = ld8(Ks + (32 * tj + l32) * KP + 16 * s + 8 * hf);
        if (!PF) {
          const bf16x8 qa = ld8(Qs + (32 * ti + l32) * KP + 16 * s + 8 * hf);
          gq = mfma32(kb, qa, gq);  // transposed: lane = query row i, registers = key tokens j
        }
        if (DELTA) {
          const bf16x8 ka = ld8(Ks + (32 * ti + l32) * KP + 16 * s + 8 * hf);
          gk = mfma32(ka, kb, gk);  // lane = column j, registers = rows i
        }
      }
    } else {
      // meanwhile, the wave above the diagonal: gamma = inclusive cumsum of g over the chunk; beta
      float x = tok_ok ? g_tok : 0.f;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const float y = __shfl_up(x, d);
        if (lane >= d) x += y;
      }
      gam[lane] = x;
      if (DELTA) bet[lane] = tok_ok ? bf16_to_f32(b_tok) : 0.f;
    }
    // all waves are done reading the q, k tiles before the A blocks overwrite them
    __syncthreads();
    if (ti >= tj) {
      if (!PF) {
        // this lane's 16 key tokens are four runs of four: 16-byte reads of their gamma and 1/|k|
        const float gi = gam[i], fi = p.scale * rq[i];
        // this lane holds tokens 8 q4 + 4 hf + e of the tile: q4 = 0, 2 are the two halves of group hf's slots,
        // q4 = 1, 3 those of group 2 + hf
        u32x4 w[2];
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const int j0 = 32 * tj + 8 * q4 + 4 * hf;
          const f32x4 gj = *reinterpret_cast<const f32x4*>(gam + j0), rj = *reinterpret_cast<const f32x4*>(rk + j0);
          float pv[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            float a = fi * rj[e] * gq[4 * q4 + e] * __expf(gi - gj[e]);
            asm volatile("" : "+v"(a));                  // (a select, no branch around the exponential)
            pv[e] = i >= j0 + e ? a : 0.f;
          }
          w[q4 & 1][2 * (q4 >> 1)] = pack_bf16x2(pv[0], pv[1]);
          w[q4 & 1][2 * (q4 >> 1) + 1] = pack_bf16x2(pv[2], pv[3]);
        }
        *reinterpret_cast<u32x4*>(prow + hf * 128) = w[0];
        *reinterpret_cast<u32x4*>(prow + (2 + hf) * 128) = w[1];
      }
    }
    if (DELTA) {
      if (ti >= tj) {
        const int j = 32 * tj + l32;
        const float gj = gam[j], rkj = rk[j];
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          const int i0 = 32 * ti + 8 * q4 + 4 * hf;  // rows i0..i0+3, all in one 16-row block
          const f32x4 gi4 = *reinterpret_cast<const f32x4*>(gam + i0), ri4 = *reinterpret_cast<const f32x4*>(rk + i0),
                      bi4 = *reinterpret_cast<const f32x4*>(bet + i0);
          if ((i0 >> 4) >= (j >> 4)) {
            float* dst = Ab + bidx(i0 >> 4, j >> 4) * BLK + (i0 & 15) * BP + (j & 15);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              float a = bi4[e] * ri4[e] * rkj * gk[4 * q4 + e] * __expf(gi4[e] - gj);
              asm volatile("" : "+v"(a));               // (a select, no branch around the exponential)
              dst[e * BP] = i0 + e > j ? a : 0.f;
            }
          }
        }
      }
    }
  }
  // ---- per-token scale vectors -------------------------------------------------------------
  if (wave == 1) {
    const float gl = gam[C - 1], gt = gam[lane], eg = __expf(gt);
    float dk = gl - gt;
    if (!DELTA) dk = fminf(dk, 0.f);  // src/nats/ops/mamba/chunk_h.py:177
    Sout[lane] = eg * rk[lane];
    Sout[C + lane] = p.scale * rq[lane] * eg;
    Sout[2 * C + lane] = rk[lane] * __expf(dk);
    if (PF) {
      float* Eout = reinterpret_cast<float*>(Pout);
      Eout[lane] = gt * 1.4426950408889634f - __builtin_amdgcn_logf(rk[lane]);
      Eout[C + lane] = gt * 1.4426950408889634f + __builtin_amdgcn_logf(p.scale);
    }
    if (lane == 0) Sout[3 * C] = __expf(gl);
    if (lane == 1) Sout[3 * C + 1] = gl;
    if (lane == 2) {
      // is this chunk's selector block typed linear?  (kept next to the decay so the scan finds it
      // in the cache line it prefetches anyway)
      Sout[3 * C + 2] = rintf(__uint_as_float((unsigned)type_hi << 16 | (p.types_dtype == NATSL_F32 ? (unsigned)type_lo : 0u))) == 1.0f ? 1.f : 0.f;
    }
  }
  if (!DELTA) return;
  __syncthreads();

  // ---- X = (I + A)^-1 in fp32, 4x4 blocks of 16x16 ------------------------------------------
  // diagonal blocks by forward substitution: one wave, 16 lanes a block, one column per lane (16 lanes of each of the four waves
  // cost the SIMDs four times the issue slots)
  const int x16 = lane & 15, g4 = lane >> 4;
  if (wave == 3) {
    float* Ad = Ab + bidx(g4, g4) * BLK;
    f32x4 arow[16][4];
#pragma unroll
    for (int r = 1; r < 16; ++r)
#pragma unroll
      for (int j4 = 0; j4 < (r + 3) / 4; ++j4) arow[r][j4] = *reinterpret_cast<const f32x4*>(Ad + r * BP + 4 * j4);
    float x[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float acc = r == x16 ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < r; ++j) acc -= arow[r][j >> 2][j & 3] * x[j];
      x[r] = acc;
    }
    float* Xtd = Xt + g4 * BLK;
#pragma unroll
    for (int r = 0; r < 16; ++r) Ad[r * BP + x16] = x[r];
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4)
      *reinterpret_cast<f32x4*>(Xtd + x16 * BP + 4 * r4) = (f32x4){x[4 * r4], x[4 * r4 + 1], x[4 * r4 + 2], x[4 * r4 + 3]};
  }
  __syncthreads();
  // off-diagonal blocks on the fp32 matrix cores, wave k down its own block column:
  //   X_ik = -X_ii * sum_{j=k}^{i-1} A_ij X_jk        (i = k+1 .. 3)
  // MFMA 16x16x4: lane (x, g) supplies A[x][kk] and B[kk][x].  With kk = 4g + s in step s, the A operand of all four
  // steps is one 16-byte row read, and an accumulator (lane = column x, registers = rows 4g..4g+3) is already a B
  // operand: the X_jk of the column stay in registers (only the diagonal block comes from LDS), and the inner sum feeds
  // the second product from registers too.  Nothing a wave reads here was written by another wave after the barrier above,
  // so the column needs no barrier of its own.
  {
    const int k = wave;
    f32x4 Xcol[4];
#pragma unroll
    for (int i = 1; i < 4; ++i) {
      Xcol[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
      if (i > k) {
        f32x4 M = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < i; ++j) {
          if (j >= k) {
            const f32x4 a4 = *reinterpret_cast<const f32x4*>(Ab + bidx(i, j) * BLK + x16 * BP + 4 * g4);
            f32x4 b4 = Xcol[j];
            if (j == k) b4 = *reinterpret_cast<const f32x4*>(Xt + k * BLK + x16 * BP + 4 * g4);
#pragma unroll
            for (int st = 0; st < 4; ++st) M = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[st], b4[st], M, 0, 0, 0);
          }
        }
        const f32x4 d4 = *reinterpret_cast<const f32x4*>(xblk(i, i) + x16 * BP + 4 * g4);
        f32x4 Xa = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st < 4; ++st) Xa = __builtin_amdgcn_mfma_f32_16x16x4f32(d4[st], M[st], Xa, 0, 0, 0);
        Xcol[i] = (f32x4){-Xa[0], -Xa[1], -Xa[2], -Xa[3]};
        float* Xo = Xb + (i * (i - 1) / 2 + k) * BLK;
#pragma unroll
        for (int r = 0; r < 4; ++r) Xo[(4 * g4 + r) * BP + x16] = Xcol[i][r];
      }
    }
  }
  __syncthreads();
  // TmB = Tm * diag(beta), bf16, in the scan kernel's A-operand order (see above): this thread's 16 columns are one
  // half (cb % 2) of the 32 tokens of operand (row / 16, cb / 2); columns 4g..4g+3 of them are the lower (upper) 8 bytes
  // of scan-lane group g.  Blocks above the diagonal are zero; operands (0,1), (1,1) are not stored at all.
  {
    const int row = tid >> 2, cb = tid & 3;
    if (!((row >> 4) < 2 && cb >= 2)) {
      float x[16];
#pragma unroll
      for (int e4 = 0; e4 < 4; ++e4) {
        const f32x4 xv = cb <= (row >> 4) ? *reinterpret_cast<const f32x4*>(xblk(row >> 4, cb) + (row & 15) * BP + 4 * e4)
                                          : (f32x4){0.f, 0.f, 0.f, 0.f};
        const f32x4 bv = *reinterpret_cast<const f32x4*>(bet + 16 * cb + 4 * e4);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[4 * e4 + e] = xv[e] * bv[e];
      }
      bf16_t* trow = Tout + ((size_t)((2 * (row >> 4) + (cb >> 1)) * 64 + (row & 15))) * 8 + 4 * (cb & 1);
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        u32x2 w;
        w[0] = pack_bf16x2(x[4 * g], x[4 * g + 1]);
        w[1] = pack_bf16x2(x[4 * g + 2], x[4 * g + 3]);
        *reinterpret_cast<u32x2*>(trow + g * 128) = w;
      }
    }
  }
}

// The Mamba form needs no Gram products ahead of the scan (its intra-chunk matrix is formed in the scan from the k, q tiles
// that are in LDS anyway): what is left of the prep is the chunk's scale vectors, one wave per chunk and four heads, nothing read
// but g and the block type:  sc = { gamma log2(e), scale e^{gamma}, e^{min(gamma_last - gamma, 0)}, {e^{gamma_last}, gamma_last, is_linear} }.
constexpr int MS_HEADS = 4;   // of a wave: their running sums hide each other's shuffles, and the lines of g, all heads of a token, are read by one
                              // workgroup in sixteens instead of fours (B4 T8192 H32: 11.7 -> 8.0 us)
__device__ __attribute__((always_inline)) inline void mamba_scale(const LinearParams& p, const unsigned wg) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int groups = (p.H + 4 * MS_HEADS - 1) / (4 * MS_HEADS);
  const int gc = (int)(wg / (unsigned)groups), h0 = ((int)(wg % (unsigned)groups) * 4 + wave) * MS_HEADS;
  if (h0 >= p.H) return;
  int bos, len, c, bos_nats;
  if (p.seqs == nullptr) {
    const int n = gc / p.nt;
    c = gc - n * p.nt;
    bos = n * p.T;
    len = p.T;
    bos_nats = n * p.TN;
  } else {
    int n = 0;
    for (int i = 1; i < p.n_seqs; ++i)
      if (p.seqs[i].chunk_off <= gc) n = i;
    c = gc - p.seqs[n].chunk_off;
    bos = p.seqs[n].bos;
    len = p.seqs[n].eos - bos;
    bos_nats = p.seqs[n].bos_nats;
  }
  const int t0 = c * C;
  const float* g = p.g + (size_t)(bos + min(t0 + lane, len - 1)) * p.H;
  float x[MS_HEADS];
#pragma unroll
  for (int u = 0; u < MS_HEADS; ++u) x[u] = g[min(h0 + u, p.H - 1)];
  // lane u: the type of head h0 + u
  const int type_size = p.types_dtype == NATSL_F32 ? 4 : 2, ht = min(h0 + (lane & (MS_HEADS - 1)), p.H - 1);
  const char* type_at = reinterpret_cast<const char*>(p.types) + (((size_t)(bos_nats + t0 / p.block) * p.HN + ht / (p.H / p.HN)) * 2 + 1) * type_size;
  const bf16_t type_lo = *reinterpret_cast<const bf16_t*>(type_at), type_hi = *reinterpret_cast<const bf16_t*>(type_at + type_size - 2);
#pragma unroll
  for (int u = 0; u < MS_HEADS; ++u) x[u] = t0 + lane < len ? x[u] : 0.f;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1)
#pragma unroll
    for (int u = 0; u < MS_HEADS; ++u) {
      const float y = __shfl_up(x[u], d);
      if (lane >= d) x[u] += y;
    }
  const float type = rintf(__uint_as_float((unsigned)type_hi << 16 | (p.types_dtype == NATSL_F32 ? (unsigned)type_lo : 0u))) == 1.0f ? 1.f : 0.f;
#pragma unroll
  for (int u = 0; u < MS_HEADS; ++u) {
    if (h0 + u >= p.H) return;
    const float gl = __shfl(x[u], C - 1), linear = __shfl(type, u);
    float* Sout = p.ws_sc + ((size_t)gc * p.H + h0 + u) * (4 * C);
    Sout[lane] = x[u] * 1.4426950408889634f;   // in log2 units: the scan forms e^{gamma_i - gamma_j} with one exp2 per element
    Sout[C + lane] = p.scale * __expf(x[u]);
    Sout[2 * C + lane] = __expf(fminf(gl - x[u], 0.f));  // src/nats/ops/mamba/chunk_h.py:177
    const float tail = lane == 0 ? __expf(gl) : lane == 1 ? gl : linear;
    if (lane < 3) Sout[3 * C + lane] = tail;
  }
}

// The workgroups of either form.
inline long long linear_prep_wgs(const bool delta, const long long chunks, const int H) {
  return chunks * (delta ? H : (H + 4 * MS_HEADS - 1) / (4 * MS_HEADS));
}

}  // namespace natsl
