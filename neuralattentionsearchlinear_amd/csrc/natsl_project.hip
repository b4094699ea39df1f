// The wide products of a layer's projections, one launch for all that share an input:
//   forward   Y_s[t][n]  = sum_d X[t][d] W_s[n][d]                           for every projection s
//   backward  dX[t][d]   = sum_s sum_n dY_s[t][n] W_s[n][d] + the block mean's gradient
// bf16 operands, fp32 sums, one rounding.
//
// Why not a library product each: a projection of 768 or 1152 columns leaves part of its last round of tiles idle, four products of a
// short prompt are four launches, and the gradients of one input accumulate, so that dX is read and written once per projection.  Here the
// tiles of all projections (forward) or the contraction over all of them (backward) follow each other in one launch.  340M geometry, 8 x 4096
// tokens: backward 342 us (four accumulating products and the block mean's pass) -> 237, 1.3 PFLOP/s; forward 267 -> 260.
//
// A tile is 256 tokens (or 192, 128) x 256 columns, four waves with 128 x 128 of it each: 256 accumulator registers, a wave per SIMD; an
// operand pair from LDS serves 16 matrix instructions.  Stages of 32 contraction elements come by LDS-DMA into a ring of four; the
// operands of the next 16 elements are requested while the current ones multiply, and the one barrier of a stage sits in its middle, where
// the next stage's operands are about to be read.  A workgroup walks its tiles with the requests running on into the next one, so a tile
// has no prologue.  1 190 - 1 220 cycles a stage against 1 024 of matrix time, 6 500 for a tile's way out (its stores: held back and
// spread over the next tile's stages they cost the same there).  What bounds it then is the power limit: 1.75 - 1.9 GHz in a training step,
// where the passes around it run at 2.4, 1.25 - 1.7 back to back.
#include <type_traits>

#include "natsl_device.h"
#include "natsl_host.h"

namespace natsl {

constexpr int PJ_K = 32;                       // contraction elements per stage
constexpr int PJ_N = 256;                      // output columns of a tile
constexpr int PJ_W = PJ_N * PJ_K * 2;          // 16 KiB of W per stage
constexpr int PJ_STAGES = 4;
constexpr int PJ_GROUP = 8;                    // row tiles that are walked together
constexpr int PJ_OUT = 4096;                   // bytes a wave's output passes through: 32 tokens x 64 columns

struct ProjSeg { const bf16_t* y; const bf16_t* w; int n, ld, tile0; };   // y: the output, or the gradient; tile0: its first column tile
struct ProjParams {
  const bf16_t* x;                             // forward: the input
  bf16_t* dx;                                  // backward: the output
  const bf16_t* dpool;
  int rows, D, ldx, n_seg, stages;
  int tiles_m, tiles_n, tiles, per, wgs;       // per: tiles of an XCD; wgs: its workgroups
  int T, block, nb;
  ProjSeg seg[NATSL_PROJECT_SEGS];
};

NATSL_DEVICE void pj_dma(const void* base, const unsigned voff, const unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(lds) : "memory", "m0");
}

template <int MB>
struct ProjLds {
  static constexpr int X = 64 * MB * PJ_K * 2, STAGE = X + PJ_W, OUT = PJ_STAGES * STAGE, TOTAL = OUT + 4 * PJ_OUT;
};

// Four waves, each 32 MB tokens x 128 columns of the tile (64 MB tokens x 256 columns).  Workgroup ids go round the XCDs; an XCD's
// workgroups take consecutive tiles, eight rows of tiles by columns, so that what they read together stays in its L2.
template <int MB, bool BWD, bool POOL>
__global__ __launch_bounds__(256, 1) void project_kernel(const ProjParams p) {
  using L = ProjLds<MB>;
  constexpr int PER = MB + 4, HALF = 4;        // requests of a wave per stage, and those of them that go out in the second half of a stage
  extern __shared__ __align__(1024) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, hf = lane >> 5;
  const int xcd = (int)blockIdx.x & 7, slot = (int)blockIdx.x >> 3;
  const int end = min(p.tiles, (xcd + 1) * p.per);
  int cur = xcd * p.per + slot;
  if (cur >= end) return;
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;

  struct Tile { int m0, tn; };
  auto tile_of = [&](const int o) __attribute__((always_inline)) -> Tile {
    const int span = PJ_GROUP * p.tiles_n, grp = o / span, r = o - grp * span;
    const int gm = min(PJ_GROUP, p.tiles_m - grp * PJ_GROUP), tn = r / gm;
    return {(grp * PJ_GROUP + r - tn * gm) * 64 * MB, tn};
  };
  auto seg_of = [&](const int tn) __attribute__((always_inline)) -> int {
    int si = 0;
#pragma unroll
    for (int i = 1; i < NATSL_PROJECT_SEGS; ++i) si = i < p.n_seg && tn >= p.seg[i].tile0 ? i : si;
    return si;
  };

  // ---- requests, three stages ahead of the products and on into the workgroup's next tile
  int rq_tile = cur, rq_k = 0, rq_seg = 0, rq_n = 0, rq_f = 0;
  Tile rq = tile_of(cur);
  const bf16_t *ra = nullptr, *rb = nullptr;
  unsigned va[MB], vb[4];
  auto offsets = [&]() __attribute__((always_inline)) {
    const ProjSeg& sg = p.seg[rq_seg];
    const int ld = BWD ? sg.ld : p.ldx;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int row = 16 * (MB * wave + i) + (lane >> 2), s = (lane & 3) ^ ((row >> 2) & 3);
      va[i] = (unsigned)(min(row, p.rows - rq.m0 - 1) * ld * 2 + s * 16);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (BWD) {
        const int row = 8 * wave + 2 * i + hf, s = l32 ^ (4 * (row & 3));
        vb[i] = (unsigned)(row * p.D * 2 + min(rq.tn * (PJ_N / 8) + s, p.D / 8 - 1) * 16);
      } else {
        const int row = 16 * (4 * wave + i) + (lane >> 2), s = (lane & 3) ^ ((row >> 2) & 3);
        vb[i] = (unsigned)(min(row, sg.n - (rq.tn - sg.tile0) * PJ_N - 1) * p.D * 2 + s * 16);
      }
    }
  };
  auto begin = [&]() __attribute__((always_inline)) {
    rq_k = 0;
    const ProjSeg& sg = p.seg[rq_seg];
    if constexpr (BWD) {
      ra = sg.y + (size_t)rq.m0 * sg.ld;
      rb = sg.w;
      rq_n = sg.n;
    } else {
      ra = p.x + (size_t)rq.m0 * p.ldx;
      rb = sg.w + (size_t)(rq.tn - sg.tile0) * PJ_N * p.D;
      rq_n = p.D;
    }
    offsets();
  };
  auto advance = [&]() __attribute__((always_inline)) {
    ++rq_f;
    ra += PJ_K;
    rb += BWD ? (size_t)PJ_K * p.D : (size_t)PJ_K;
    rq_k += PJ_K;
    if (rq_k >= rq_n) {
      if (BWD && rq_seg + 1 < p.n_seg) {
        ++rq_seg;
        begin();
      } else {
        rq_tile = rq_tile + p.wgs < end ? rq_tile + p.wgs : rq_tile;   // (behind the last tile: its first stages again, for nobody)
        rq = tile_of(rq_tile);
        rq_seg = BWD ? 0 : seg_of(rq.tn);
        begin();
      }
    }
  };
  // request j of the stage: four of W, then MB of X
  auto request = [&](const int j) __attribute__((always_inline)) {
    const unsigned l = lds0 + (unsigned)(rq_f & (PJ_STAGES - 1)) * L::STAGE;
    if (j < 4) pj_dma(rb, vb[j], l + L::X + 1024 * (4 * wave + j));
    else pj_dma(ra, va[j - 4], l + 1024 * (MB * wave + j - 4));
  };
  // ---- operands.  X (and W forward): rows of 64 bytes, 16-byte segment s at slot s ^ (row / 4) % 4.  W backward: rows of 512 bytes, segment s
  // at slot s ^ 4 (row % 4), read with the transposing read.
  const int wm = wave >> 1, wn = wave & 1;
  const unsigned row_lane = (unsigned)(l32 * 64 + 16 * (hf ^ ((l32 >> 2) & 3)));
  const unsigned am = lds0 + wm * MB * 2048 + row_lane;
  unsigned an[BWD ? 4 : 1];
  if constexpr (BWD) {
    const int g = lane >> 4, j = (lane & 15) >> 2, c = lane & 3;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      an[i] = lds0 + L::X + (8 * (g >> 1) + j) * 512 + (2 * (g & 1) + (c >> 1)) * 16 + (c & 1) * 8 + (4 * wn + (i ^ j)) * 64;
  } else {
    an[0] = lds0 + L::X + wn * 8192 + row_lane;
  }
  typedef s16x4 __attribute__((address_space(3))) * lds_s4_t;
  typedef bf16x8 __attribute__((address_space(3))) * lds_b128_t;
  typedef u32x2 __attribute__((address_space(3))) * lds_w2_t;
  typedef u32x4 __attribute__((address_space(3))) * lds_w4_t;
  auto m_operand = [&](const unsigned at, const int kk, const int b) __attribute__((always_inline)) -> bf16x8 {
    return *(lds_b128_t)(uintptr_t)((kk ? am ^ 32u : am) + at + 2048 * b);
  };
  auto n_operand = [&](const unsigned at, const int kk, const int i) __attribute__((always_inline)) -> bf16x8 {
    if constexpr (BWD) {
      const unsigned a = an[i] + at + kk * 16 * 512;
      return join4(__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t)(uintptr_t)a), __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t)(uintptr_t)(a + 4 * 512)));
    } else {
      return *(lds_b128_t)(uintptr_t)((kk ? an[0] ^ 32u : an[0]) + at + 2048 * i);
    }
  };

  rq_seg = BWD ? 0 : seg_of(rq.tn);
  begin();
#pragma unroll 1
  for (int s = 0; s < 3; ++s) {                // (a tile has at least four stages)
#pragma unroll
    for (int j = 0; j < PER; ++j) request(j);
    advance();
  }
#pragma unroll
  for (int j = 0; j < HALF; ++j) request(j);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * PER + HALF) : "memory");
  __syncthreads();

  f32x16 acc[4][MB];
  bf16x8 N[2][4], M[2][MB];
#pragma unroll
  for (int i = 0; i < 4; ++i) N[0][i] = n_operand(0, 0, i);
#pragma unroll
  for (int b = 0; b < MB; ++b) M[0][b] = m_operand(0, 0, b);

  unsigned f = 0;                              // the stage among all of the workgroup's
  // One stage's products; FIRST: a tile's first.
  auto stage = [&](auto first_c) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first_c)::value;
    const unsigned here = (f & (PJ_STAGES - 1)) * L::STAGE, next = ((f + 1) & (PJ_STAGES - 1)) * L::STAGE;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      if (kk == 1) {
        // stage f + 1 has landed for every wave, and nobody reads stage f any more
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * PER) : "memory");
        __syncthreads();
        advance();
      }
      const unsigned at = kk == 0 ? here : next;   // (behind the last stage: a buffer that nobody writes any more; the values are not used)
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        N[kk ^ 1][a] = n_operand(at, kk ^ 1, a);
        if (a < MB) M[kk ^ 1][a] = m_operand(at, kk ^ 1, a);
#pragma unroll
        for (int b = 0; b < MB; ++b) {
          if (FIRST && kk == 0) {
            f32x16 z;
#pragma unroll
            for (int r = 0; r < 16; ++r) z[r] = 0.f;
            acc[a][b] = mfma32(N[kk][a], M[kk][b], z);
          } else {
            acc[a][b] = mfma32(N[kk][a], M[kk][b], acc[a][b]);
          }
        }
#pragma unroll
        for (int b = 0; b < MB; ++b) {
          __builtin_amdgcn_sched_group_barrier(0x100, MB == 2 ? 2 : 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        if (kk == 0 && HALF + a < PER) request(HALF + a);   // the rest of stage f + 3 ..
        if (kk == 1 && a < HALF) request(a);                // .. and the first requests of stage f + 4, into the buffer of stage f
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    ++f;
  };

  for (; cur < end; cur += p.wgs) {
    const Tile t = tile_of(cur);
    stage(std::true_type{});
#pragma unroll 1
    for (int s = 1; s < p.stages; ++s) {
      stage(std::false_type{});
    }
    // ---- the tile leaves: lane = token, registers = 8 q + 4 hf + r of 32 columns; through LDS as whole 128-byte lines
    const int si = BWD ? 0 : seg_of(t.tn);
    const int n0 = BWD ? t.tn * PJ_N : (t.tn - p.seg[si].tile0) * PJ_N;
    const int n_end = BWD ? p.D : p.seg[si].n, ldo = BWD ? p.D : p.seg[si].ld;
    bf16_t* out = BWD ? p.dx : const_cast<bf16_t*>(p.seg[si].y);
    int el = lane;
    asm volatile("" : "+v"(el));               // (its addresses are formed here and not kept through the products)
    const int e32 = el & 31, ehf = el >> 5;
    const unsigned ew = lds0 + L::OUT + wave * PJ_OUT + e32 * 128 + 8 * ehf;          // written: token e32, 8 bytes of segment q at slot q ^ e32 % 8
    const unsigned er = lds0 + L::OUT + wave * PJ_OUT + (el >> 3) * 128 + ((el & 7) ^ (el >> 3)) * 16;   // read: token el / 8 (+ 8 u), segment el % 8
    const int c_st = n0 + wn * 128 + 8 * (el & 7), r_st = t.m0 + wm * MB * 32 + (el >> 3);
    bf16_t* o_st = out + (size_t)r_st * ldo + c_st;
    const bool in0 = c_st < n_end, in1 = c_st + 64 < n_end;
    u32x2 pw[8];
    float inv = 0.f;
    auto pool = [&](const int c) __attribute__((always_inline)) {     // the block means' gradients of chunk c (32 tokens x 64 columns)
      if constexpr (POOL) {
        const int row = min(t.m0 + (wm * MB + (c >> 1)) * 32 + e32, p.rows - 1), n = (int)((unsigned)row / (unsigned)p.T), tt = row - n * p.T;
        const int blk = (int)((unsigned)tt / (unsigned)p.block);
        inv = 1.f / (float)(min(p.T, (blk + 1) * p.block) - blk * p.block);
        const bf16_t* src = p.dpool + ((size_t)n * p.nb + blk) * p.D;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int col = n0 + wn * 128 + 64 * (c & 1) + 8 * i + 4 * ehf;
          pw[i] = *reinterpret_cast<const u32x2*>(src + min(col, p.D - 4));
        }
      }
    };
    pool(0);
#pragma unroll
    for (int c = 0; c < 2 * MB; ++c) {
      const int b = c >> 1, ip = c & 1;
      asm volatile("" : "+a"(acc[2 * ip][b]), "+a"(acc[2 * ip + 1][b]));   // (read out here: all at once they do not fit)
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = acc[2 * ip + (i >> 2)][b][4 * (i & 3) + r];
        if constexpr (POOL) {
          const u32x2 w2 = pw[i];
          o[0] += inv * __uint_as_float(w2[0] << 16);
          o[1] += inv * __uint_as_float(w2[0] & 0xffff0000u);
          o[2] += inv * __uint_as_float(w2[1] << 16);
          o[3] += inv * __uint_as_float(w2[1] & 0xffff0000u);
        }
        *(lds_w2_t)(uintptr_t)(ew + 16 * (i ^ (e32 & 7))) = (u32x2){pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
      }
      if (c + 1 < 2 * MB) pool(c + 1);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      u32x4 w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = *(lds_w4_t)(uintptr_t)(er + 1024 * u);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (r_st + 32 * b + 8 * u < p.rows && (ip ? in1 : in0)) *reinterpret_cast<u32x4*>(o_st + (size_t)(32 * b + 8 * u) * ldo + 64 * ip) = w[u];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (the requests behind the last tile: not into memory that is another workgroup's by then)
}

static int project_cus() {
  static std::atomic<int> cached{0};
  int n = cached.load();
  if (n == 0) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached.store(n);
  }
  return n;
}

template <int MB, bool BWD, bool POOL>
static int launch_project(ProjParams& p, const int cus, hipStream_t stream, const char* what) {
  using L = ProjLds<MB>;
  p.tiles_m = cdiv(p.rows, 64 * MB);
  p.tiles = p.tiles_m * p.tiles_n;
  p.per = cdiv(p.tiles, 8);
  p.wgs = p.per < cus / 8 ? p.per : cus / 8;
  auto kern = project_kernel<MB, BWD, POOL>;
  static std::atomic<unsigned long long> reserved{0};
  if (const int rc = reserve_lds(reinterpret_cast<const void*>(kern), reserved, L::TOTAL, what)) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)(8 * p.wgs)), dim3(256), L::TOTAL, stream, p);
  return check_launch(what);
}

// Tokens of a tile: the height whose rounds over the CUs take least.  A tile of 192 or 128 tokens takes 0.72-0.81 or 0.55-0.64 of one of 256
// (measured, 32 to 217 stages); the shorter ones read W more often and lose a little more where the power limit decides.
// Backward, 256 / 192 / 128 tokens, us: 340M geometry 8 x 4096 260 / 281 / 287, 1 x 4000 82 / 70 / 54; 760M 2 x 3000 141 / 121 / 158.
template <bool BWD, bool POOL>
static int launch_project_any(ProjParams& p, hipStream_t stream, const char* what) {
  const int cus = project_cus() < 8 ? 8 : project_cus();
  constexpr double COST[3] = {0.62, 0.75, 1.};
  int best = 4;
  double best_cost = 1e300;
  for (int mb = 4; mb >= 2; --mb) {
    const long long tiles = (long long)cdiv(p.rows, 64 * mb) * p.tiles_n, per = (tiles + 7) / 8;
    const double cost = (double)((per + cus / 8 - 1) / (cus / 8)) * COST[mb - 2];
    if (cost < best_cost) { best_cost = cost; best = mb; }
  }
  if ((long long)cdiv(p.rows, 64 * best) * p.tiles_n > (1 << 28)) return fail(NATSL_ERR_UNSUPPORTED, "%s: problem too large", what);
  if (best == 4) return launch_project<4, BWD, POOL>(p, cus, stream, what);
  if (best == 3) return launch_project<3, BWD, POOL>(p, cus, stream, what);
  return launch_project<2, BWD, POOL>(p, cus, stream, what);
}

static int project_segs(ProjParams& p, const natsl_project_seg* segs, int n_seg, int64_t rows, int D, const char* what) {
  if (!segs || n_seg <= 0 || n_seg > NATSL_PROJECT_SEGS) return fail(NATSL_ERR_INVALID, "%s: 1 to %d projections", what, NATSL_PROJECT_SEGS);
  if (rows <= 0 || D <= 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  if (rows > (1ll << 30) || D % 8) return fail(NATSL_ERR_UNSUPPORTED, "%s: the width must be a multiple of 8", what);
  uintptr_t low = 0;
  for (int i = 0; i < NATSL_PROJECT_SEGS; ++i) {
    if (i >= n_seg) { p.seg[i] = {nullptr, nullptr, 0, 0, 1 << 30}; continue; }
    const natsl_project_seg& s = segs[i];
    if (!s.y || !s.w) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
    if (s.n <= 0 || s.ld < s.n || s.n % 8 || s.ld % 8) return fail(NATSL_ERR_UNSUPPORTED, "%s: widths and row strides must be multiples of 8", what);
    if (256ll * s.ld * 2 > 0x7fffffffll || 256ll * D * 2 > 0x7fffffffll) return fail(NATSL_ERR_UNSUPPORTED, "%s: rows too long", what);
    low |= (uintptr_t)s.y | (uintptr_t)s.w;
    p.seg[i] = {(const bf16_t*)s.y, (const bf16_t*)s.w, s.n, s.ld, 0};
  }
  if (low & 15) return fail(NATSL_ERR_INVALID, "%s: tensors must start on 16 bytes", what);
  p.rows = (int)rows; p.D = D; p.n_seg = n_seg;
  return NATSL_OK;
}

}  // namespace natsl

using namespace natsl;

extern "C" int natsl_project(const natsl_project_seg* segs, int n_seg, const void* x, int64_t rows, int D, int ldx, natsl_stream_t stream) {
  const char* what = "natsl_project";
  ProjParams p{};
  int rc = project_segs(p, segs, n_seg, rows, D, what);
  if (rc != NATSL_OK) return rc;
  if (!x || ((uintptr_t)x & 15)) return fail(NATSL_ERR_INVALID, "%s: the input must start on 16 bytes", what);
  if (D % PJ_K || D < 4 * PJ_K || ldx % 8 || ldx < D || 256ll * ldx * 2 > 0x7fffffffll)
    return fail(NATSL_ERR_UNSUPPORTED, "%s: the input's width must be a multiple of %d from %d on", what, PJ_K, 4 * PJ_K);
  p.x = (const bf16_t*)x; p.ldx = ldx; p.stages = D / PJ_K;
  for (int i = 0; i < n_seg; ++i) {
    p.seg[i].tile0 = p.tiles_n;
    p.tiles_n += cdiv(p.seg[i].n, PJ_N);
  }
  return launch_project_any<false, false>(p, reinterpret_cast<hipStream_t>(stream), what);
}

// (as the whole of natsl_project_bwd's conditions on these: it refuses what this does not take)
extern "C" int natsl_project_bwd_takes(const natsl_project_seg* segs, const int n_seg, const void* dpool, const void* dx) {
  if (!segs || n_seg <= 0 || n_seg > NATSL_PROJECT_SEGS) return 0;
  uintptr_t low = (uintptr_t)dpool | (uintptr_t)dx;
  long long columns = 0;
  for (int i = 0; i < n_seg; ++i) {
    const natsl_project_seg& s = segs[i];
    if (s.n <= 0 || s.n % PJ_K || s.ld < s.n || s.ld % 8) return 0;
    columns += s.n;
    low |= (uintptr_t)s.y | (uintptr_t)s.w;
  }
  return columns >= 4 * PJ_K && low % 16 == 0;
}

extern "C" int natsl_project_bwd(const natsl_project_seg* segs, int n_seg, const void* dpool, void* dx, int B, int T, int D, int block, natsl_stream_t stream) {
  const char* what = "natsl_project_bwd";
  if (B <= 0 || T <= 0 || block <= 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  ProjParams p{};
  int rc = project_segs(p, segs, n_seg, (int64_t)B * T, D, what);
  if (rc != NATSL_OK) return rc;
  if (!dx || (((uintptr_t)dx | (uintptr_t)dpool) & 15)) return fail(NATSL_ERR_INVALID, "%s: tensors must start on 16 bytes", what);
  for (int i = 0; i < n_seg; ++i) {
    if (p.seg[i].n % PJ_K) return fail(NATSL_ERR_UNSUPPORTED, "%s: widths must be multiples of %d", what, PJ_K);
    p.stages += p.seg[i].n / PJ_K;
  }
  if (p.stages < 4) return fail(NATSL_ERR_UNSUPPORTED, "%s: fewer than four stages of %d columns", what, PJ_K);
  p.dx = (bf16_t*)dx; p.dpool = (const bf16_t*)dpool; p.T = T; p.block = block; p.nb = cdiv(T, block);
  p.tiles_n = cdiv(D, PJ_N);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  return dpool ? launch_project_any<true, true>(p, st, what) : launch_project_any<true, false>(p, st, what);
}
