// Weight gradients of projections that share their input: dW_s[n][d] = sum over tokens t of dY_s[t][n] X[t][d], bf16 operands,
// fp32 sums, one launch for all of them.
//
// The output is small (a weight) and the contraction long (the tokens), so a library product with one workgroup per output tile
// leaves most of the chip idle: 24 to 48 tiles on 256 CUs (308 us for 1536 x 1024 over 32768 tokens, a third of the rate large
// products reach).  Here the tokens are split as well: a unit is (slice of the tokens, 256 x 256 output tile), partial tiles go to
// a workspace in fp32 and wgrad_reduce_kernel adds them in a fixed order.
//
// (WG_N rows of dY by 64 NB columns of X, NB 3 or 4: 256 or 192.)
// Both operands have the contraction index as their slow dimension in memory and the matrix instruction wants it inside a lane:
// tiles of 32 tokens x 256 columns go to LDS row by row (LDS-DMA, no staging registers) and operands are fetched with the
// transposing read ds_read_b64_tr_b16.  What fixes the tile is the LDS: a wave that owns 128 x 128 of the output reads 8 operands
// (8 KiB) per 16 matrix instructions (512 cycles), 64 B/clk for the CU's four waves, which the transposing read sustains; with
// 64 x 64 per wave it would need twice that.  256 accumulator registers, one wave per SIMD; the operands of the next 16 tokens are
// requested while the current ones multiply, and tiles two and three stages ahead are on their way (ring of four, 128 KiB).
#include <type_traits>

#include "natsl_device.h"
#include "natsl_host.h"

namespace natsl {

constexpr int WG_T = 32;                       // tokens per stage
constexpr int WG_N = 256;                      // output tile edge
constexpr int WG_ROW = WG_N * 2;               // bytes of a tile row
constexpr int WG_TILE = WG_T * WG_ROW;         // 16 KiB per operand
constexpr int WG_STAGE = 2 * WG_TILE;
constexpr int WG_STAGES = 4;
constexpr double WG_TOKEN_US = 0.0213, WG_TOKEN_US_3 = 0.0187;   // a unit's time a token, by tile width (at the power limit)

struct WgradSeg { const bf16_t* dy; bf16_t* out; int n, ld, tile0, block0; };   // tile0, block0: first row of tiles, of 32-row blocks
struct WgradParams {
  const bf16_t* x;
  float* part;
  int ldx, D, n_seg, tiles_d, tiles, blocks, splits, units, nb;   // blocks: 32-row blocks of all weights; nb: the kernel's NB
  long long T, slice;                          // tokens; tokens per slice (a multiple of WG_T)
  WgradSeg seg[NATSL_WGRAD_SEGS];
};

NATSL_DEVICE void wg_dma(const void* base, const unsigned voff, const unsigned lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(lds) : "memory", "m0");
}

// Partial sums lie as strips of 32 rows x a tile's columns (wg_strip), those that the weights have and no others: whole tiles of a 24-row weight
// would be eight times as much (24 x 768 over 32768 tokens: 59 MiB, 7.4 as strips).
// A tile has 64 NB columns of x: 256, or 192 where that leaves fewer CUs without work.
constexpr int wg_strip_size(const int nb) { return 32 * 64 * nb; }
template <int NB>
NATSL_DEVICE size_t wg_strip(const WgradParams& p, const int split, const int td, const int block) {
  return (((size_t)split * p.tiles_d + td) * p.blocks + block) * wg_strip_size(NB);
}

template <int NB>
__global__ __launch_bounds__(256, 1) void wgrad_kernel(const WgradParams p) {
  extern __shared__ __align__(256) unsigned char wg_smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // consecutive units share a token slice, and an XCD (block index mod 8) takes consecutive units: its CUs walk the same tokens
  const int per = (p.units + 7) / 8, u = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
  if (((int)blockIdx.x >> 3) >= per || u >= p.units) return;
  const int split = u / p.tiles, tile = u - split * p.tiles;
  const int tn = tile / p.tiles_d, td = tile - tn * p.tiles_d;
  int si = 0;
#pragma unroll
  for (int i = 1; i < NATSL_WGRAD_SEGS; ++i) si = i < p.n_seg && tn >= p.seg[i].tile0 ? i : si;
  const WgradSeg sg = p.seg[si];
  const int n0 = (tn - sg.tile0) * WG_N, d0 = td * 64 * NB;
  const long long t_first = (long long)split * p.slice;
  const int n_tok = (int)(p.T - t_first < p.slice ? p.T - t_first : p.slice);
  const int n_st = (n_tok + WG_T - 1) / WG_T;
  // 32-row blocks of this wave's 128 that the weight has: a narrow weight's others are neither multiplied nor stored
  const int blocks = min(4, max(0, (sg.n - n0 - 128 * (wave >> 1) + 31) / 32));

  // what this wave requests of a stage: rows 8*wave .. +7 of either tile, two rows per instruction.  16-byte segment s of row r
  // sits at slot s ^ 4*(r%4): the four rows of a transposing read then meet four different quarters of the banks.  Columns past
  // the matrix repeat its last segment (their products are never stored).
  unsigned va[4], vb[4];
  const int r2 = lane >> 5, slot = lane & 31;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 8 * wave + 2 * i + r2, seg = slot ^ (4 * (row & 3));
    va[i] = (unsigned)(row * sg.ld * 2 + min(n0 / 8 + seg, sg.n / 8 - 1) * 16);
    vb[i] = (unsigned)(row * p.ldx * 2 + min(d0 / 8 + min(seg, 8 * NB - 1), p.D / 8 - 1) * 16);   // (rows are 256 columns apart in LDS)
  }
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)wg_smem;
  auto request = [&](const int st) __attribute__((always_inline)) {
    const long long t = t_first + (long long)st * WG_T;
    const bf16_t* a = sg.dy + t * sg.ld;
    const bf16_t* b = p.x + t * p.ldx;
    const unsigned l = lds0 + (unsigned)(st & (WG_STAGES - 1)) * WG_STAGE + wave * 8 * WG_ROW;
    const int left = n_tok - st * WG_T;
    if (left >= WG_T) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        wg_dma(a, va[i], l + 2 * i * WG_ROW);
        wg_dma(b, vb[i], l + WG_TILE + 2 * i * WG_ROW);
      }
    } else {
      // the slice's last tokens: rows past the end repeat the last one (zeroed in LDS before use)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 8 * wave + 2 * i + r2, back = row - min(row, left - 1);
        wg_dma(a, va[i] - (unsigned)(back * sg.ld * 2), l + 2 * i * WG_ROW);
        wg_dma(b, vb[i] - (unsigned)(back * p.ldx * 2), l + WG_TILE + 2 * i * WG_ROW);
      }
    }
  };
  // stage st has landed for every wave; a partial one gets zero rows in the dY tile
  auto finish_partial = [&](const int st) __attribute__((always_inline)) {
    const int left = n_tok - st * WG_T;
    if (st == n_st - 1 && left < WG_T) {
      u32x4* z = reinterpret_cast<u32x4*>(wg_smem + (st & (WG_STAGES - 1)) * WG_STAGE + left * WG_ROW);
      for (int i = threadIdx.x; i < (WG_T - left) * (WG_ROW / 16); i += 256) z[i] = (u32x4){0u, 0u, 0u, 0u};
      __syncthreads();
    }
  };

  // operand addresses: 16-lane group g, supplier (j, c) of the transposing read; column block cb of 32 columns
  const int g = lane >> 4, j = (lane & 15) >> 2, c = lane & 3;
  const int wn = wave >> 1, wd = wave & 1;
  unsigned oa[4], ob[NB];
  const unsigned row = (8 * (g >> 1) + j) * WG_ROW + (2 * (g & 1) + (c >> 1)) * 16 + (c & 1) * 8;
#pragma unroll
  for (int i = 0; i < 4; ++i) oa[i] = lds0 + row + (4 * wn + (i ^ j)) * 64;
#pragma unroll
  for (int i = 0; i < NB; ++i) ob[i] = lds0 + WG_TILE + row + ((NB * wd + i) ^ j) * 64;
  typedef s16x4 __attribute__((address_space(3))) * lds_s4_t;
  auto operand = [&](const unsigned at) __attribute__((always_inline)) {
    return join4(__builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t)(uintptr_t)at), __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t)(uintptr_t)(at + 4 * WG_ROW)));
  };

  f32x16 acc[4][NB];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.f;

  request(0);
  if (n_st > 1) request(1);
  if (n_st > 2) {
    request(2);
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  __syncthreads();
  finish_partial(0);
  finish_partial(1);
  bf16x8 A[2][4], B[2][NB];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    A[0][i] = operand(oa[i]);
    if (i < NB) B[0][i] = operand(ob[i]);
  }
  // One stage's products.  AHEAD: stage st + 3 is a whole one, and its eight requests go out one behind every four products (issued
  // together they took 290 cycles in which the matrix cores had nothing: 4608 + 2 x 6 rows x 1024 columns over 32768 tokens 321 -> 264 us,
  // 1.2 PFLOP/s); else they are all in front, if there are any.
  auto stage = [&](auto ahead, auto whole, const int st) __attribute__((always_inline)) {
    constexpr bool AHEAD = decltype(ahead)::value, WHOLE = decltype(whole)::value;
    const unsigned here = (unsigned)(st & (WG_STAGES - 1)) * WG_STAGE, next = (unsigned)((st + 1) & (WG_STAGES - 1)) * WG_STAGE;
    const bool more = AHEAD || st + 3 < n_st;
    if (!AHEAD && more) request(st + 3);       // into the buffer of stage st-1, which every wave has read
    const long long t = t_first + (long long)(st + 3) * WG_T;
    const bf16_t *ra = sg.dy + t * sg.ld, *rb = p.x + t * p.ldx;
    const unsigned rl = lds0 + (unsigned)((st + 3) & (WG_STAGES - 1)) * WG_STAGE + wave * 8 * WG_ROW;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      // (behind the last stage the reads fetch a buffer nobody writes any more; the values are not used)
      const unsigned at = kk == 0 ? here + 16 * WG_ROW : next;
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        A[kk ^ 1][a] = operand(oa[a] + at);
        if (a < NB) B[kk ^ 1][a] = operand(ob[a] + at);
        if (WHOLE || a < blocks) {
#pragma unroll
          for (int b = 0; b < NB; ++b) acc[a][b] = mfma32(A[kk][a], B[kk][b], acc[a][b]);
        }
        // one read next to each product: the scheduler otherwise saves registers by reading an operand right before its use
        if constexpr (NB == 3) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        }
        if (AHEAD) {
          const int i = 2 * kk + (a >> 1);
          if (a & 1) wg_dma(rb, vb[i], rl + WG_TILE + 2 * i * WG_ROW);
          else wg_dma(ra, va[i], rl + 2 * i * WG_ROW);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (more) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (!AHEAD) finish_partial(st + 2);
  };
  int st = 0;
  if (sg.n - n0 > WG_N / 2)
    for (; (st + 4) * WG_T <= n_tok; ++st) stage(std::true_type{}, std::true_type{}, st);
  else
    for (; (st + 4) * WG_T <= n_tok; ++st) stage(std::true_type{}, std::false_type{}, st);
  for (; st < n_st; ++st) stage(std::false_type{}, std::false_type{}, st);

  // lane: column d = lane%32 of each 32x32 tile, rows 8*(r/4) + 4*(lane/32) + r%4: four rows of a column per 16-byte store
  float* dst = p.part + wg_strip<NB>(p, split, td, sg.block0 + (tn - sg.tile0) * 8 + 4 * (wave >> 1)) + (wave & 1) * (1024 * NB) + lane * 4;
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (a < blocks) *reinterpret_cast<f32x4*>(dst + a * wg_strip_size(NB) + (b * 4 + q) * 256) = (f32x4){acc[a][b][4 * q], acc[a][b][4 * q + 1], acc[a][b][4 * q + 2], acc[a][b][4 * q + 3]};
}

// Adds the slices' partial tiles in order and writes the gradient: a workgroup takes one 32 x 32 block of a tile per wave.
template <int NB>
__global__ __launch_bounds__(256) void wgrad_reduce_kernel(const WgradParams p) {
  const int lane = threadIdx.x & 63;
  const int id = (int)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int tile = id / (16 * NB), wave = id / (4 * NB) & 3, ab = id % (4 * NB);   // tile, wave of the tile, 32x32 block of the wave
  const int tn = tile / p.tiles_d, td = tile - tn * p.tiles_d;
  int si = 0;
#pragma unroll
  for (int i = 1; i < NATSL_WGRAD_SEGS; ++i) si = i < p.n_seg && tn >= p.seg[i].tile0 ? i : si;
  const WgradSeg sg = p.seg[si];
  const int n = (tn - sg.tile0) * WG_N + 128 * (wave >> 1) + 32 * (ab / NB), d = td * 64 * NB + 32 * NB * (wave & 1) + 32 * (ab % NB) + (lane & 31);
  if (n >= sg.n || d - (lane & 31) >= p.D) return;
  f32x4 sum[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) sum[q] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const float* src = p.part + wg_strip<NB>(p, 0, td, sg.block0 + (tn - sg.tile0) * 8 + 4 * (wave >> 1) + ab / NB) + (wave & 1) * (1024 * NB) + (ab % NB) * 1024 + lane * 4;
  const size_t step = (size_t)p.tiles_d * p.blocks * wg_strip_size(NB);
  int s = 0;
  for (; s + 6 <= p.splits; s += 6) {          // (six slices on their way at a time; one by one a slice takes a round trip, 0.4 us)
    f32x4 v[6][4];
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) v[i][q] = *reinterpret_cast<const f32x4*>(src + (s + i) * step + q * 256);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 6; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) sum[q] += v[i][q];
  }
  for (; s < p.splits; ++s)
#pragma unroll
    for (int q = 0; q < 4; ++q) sum[q] += *reinterpret_cast<const f32x4*>(src + s * step + q * 256);
  if (d >= p.D) return;
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = n + 8 * q + 4 * (lane >> 5) + r;
      if (row < sg.n) sg.out[(size_t)row * p.D + d] = f32_to_bf16(sum[q][r]);
    }
}

static int wgrad_cus() {
  static std::atomic<int> cached{0};
  int n = cached.load();
  if (n == 0) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached.store(n);
  }
  return n;
}

// Slices of the tokens and width of the tiles: a CU holds one unit at a time, so the launch takes ceil(tiles * slices / CUs) rounds of T / slices tokens,
// and every slice writes and reads its partial sums once more (0.1 us a whole tile; full_rows: whole tiles' worth of rows.  24 rows x 768 columns over
// 32768 tokens: 37 us with 32 slices of whole tiles, 27 with 85 of the strips that there are).  A tile of 192 columns takes 0.88 of the time of
// one of 256 for 0.75 of its work and is taken where such tiles fill the CUs better: 6944 rows x 1536 columns over 6000 tokens, 232 units for 174, 155 -> 139
// us; 1536 x 2304 over 6000 56 -> 53, 1024 x 1536 over 8192 41 -> 39; over 24000 tokens four slices of the first in tiles of 256 stay (461, 493 in 192).
// The slices for tiles of 256 go by 17 ns a token, what a unit takes on a chip that is not full, the choice of the width by what units take at the power limit: with
// that for the slices too, 6176 rows x 1024 columns over 18688 tokens went from two slices, 200 units in one round, to five in two (88 -> 109 us a launch and 11 -> 17 of sums).
struct WgradSplit { int nb, splits; };
static WgradSplit wgrad_splits(long long T, int tile_rows, int D, double full_rows) {
  const int cus = wgrad_cus();
  auto cost = [&](const int nb, const int s, const double token_us) {
    const double rounds = (double)(((long long)tile_rows * cdiv(D, 64 * nb) * s + cus - 1) / cus);
    return rounds * (4.0 + token_us * (double)T / s) + 0.1 * full_rows * (cdiv(D, 64 * nb) * nb / 4.) * s;
  };
  auto slices = [&](const int nb, const double token_us) {
    int best = 1;
    double best_cost = 1e300;
    for (int s = 1; s <= 128 && (s == 1 || T >= 64ll * s); ++s)
      if (const double c = cost(nb, s, token_us); c < best_cost) { best_cost = c; best = s; }
    return best;
  };
  const int s4 = slices(4, 0.017), s3 = slices(3, WG_TOKEN_US_3);
  // (two per cent nearer than they look: 6944 rows x 1536 columns over 18688 tokens 385 us in tiles of 192, 368 in four slices of 256)
  return 1.02 * cost(3, s3, WG_TOKEN_US_3) < cost(4, s4, WG_TOKEN_US) ? WgradSplit{3, s3} : WgradSplit{4, s4};
}

static int wgrad_plan(WgradParams& p, const natsl_wgrad_seg* segs, int n_seg, const void* x, int64_t T, int D, int ldx, const char* what) {
  if (!segs || n_seg <= 0 || n_seg > NATSL_WGRAD_SEGS) return fail(NATSL_ERR_INVALID, "%s: 1 to %d weights", what, NATSL_WGRAD_SEGS);
  if (T <= 0 || D <= 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  if (D % 8 || ldx % 8 || ldx < D) return fail(NATSL_ERR_UNSUPPORTED, "%s: the input's width and row stride must be multiples of 8", what);
  p.x = (const bf16_t*)x; p.ldx = ldx; p.D = D; p.n_seg = n_seg; p.T = T;
  int rows = 0;
  long long blocks = 0;
  for (int i = 0; i < NATSL_WGRAD_SEGS; ++i) {
    if (i >= n_seg) { p.seg[i] = {nullptr, nullptr, 0, 0, 1 << 30, 0}; continue; }
    const natsl_wgrad_seg& s = segs[i];
    if (s.n <= 0 || s.ld < s.n || s.n % 8 || s.ld % 8) return fail(NATSL_ERR_UNSUPPORTED, "%s: a gradient's width and row stride must be multiples of 8", what);
    if ((long long)WG_T * s.ld * 2 > 0x7fffffffll || (long long)WG_T * ldx * 2 > 0x7fffffffll) return fail(NATSL_ERR_UNSUPPORTED, "%s: rows too long", what);
    p.seg[i] = {(const bf16_t*)s.dy, (bf16_t*)s.out, s.n, s.ld, rows, (int)blocks};
    rows += cdiv(s.n, WG_N);
    blocks += cdiv(s.n, 32);
  }
  p.blocks = (int)blocks;
  const WgradSplit how = wgrad_splits(T, rows, D, blocks / 8.);
  const int splits = how.splits;
  p.nb = how.nb;
  p.tiles_d = cdiv(D, 64 * p.nb);
  p.tiles = rows * p.tiles_d;
  p.slice = (T + splits - 1) / splits;
  p.slice = (p.slice + WG_T - 1) / WG_T * WG_T;
  p.splits = (int)((T + p.slice - 1) / p.slice);
  if ((long long)p.tiles * p.splits > (1 << 24) || p.slice > (1ll << 30)) return fail(NATSL_ERR_UNSUPPORTED, "%s: problem too large", what);
  p.units = p.tiles * p.splits;
  return NATSL_OK;
}

static size_t wgrad_bytes(const WgradParams& p) { return (size_t)p.splits * p.tiles_d * p.blocks * wg_strip_size(p.nb) * sizeof(float); }

}  // namespace natsl

using namespace natsl;

extern "C" size_t natsl_wgrad_workspace_bytes(const natsl_wgrad_seg* segs, int n_seg, int64_t T, int D) {
  WgradParams p;
  if (wgrad_plan(p, segs, n_seg, nullptr, T, D, D, "natsl_wgrad") != NATSL_OK) return 0;
  return wgrad_bytes(p);
}

extern "C" int natsl_wgrad(const natsl_wgrad_seg* segs, int n_seg, const void* x, int64_t T, int D, int ldx, void* workspace,
                           size_t workspace_bytes, natsl_stream_t stream) {
  const char* what = "natsl_wgrad";
  WgradParams p;
  int rc = wgrad_plan(p, segs, n_seg, x, T, D, ldx, what);
  if (rc != NATSL_OK) return rc;
  if (!x || !workspace) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  uintptr_t low = (uintptr_t)x | (uintptr_t)workspace;
  for (int i = 0; i < n_seg; ++i) {
    if (!segs[i].dy || !segs[i].out) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
    low |= (uintptr_t)segs[i].dy;
  }
  if (low & 15) return fail(NATSL_ERR_INVALID, "%s: tensors must start on 16 bytes", what);
  if (workspace_bytes < wgrad_bytes(p)) return fail(NATSL_ERR_WORKSPACE, "%s: workspace too small", what);
  p.part = reinterpret_cast<float*>(workspace);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  auto launch = [&](auto nb) -> int {
    constexpr int NB = decltype(nb)::value;
    static std::atomic<unsigned long long> reserved{0};
    if (const int r = reserve_lds(reinterpret_cast<const void*>(wgrad_kernel<NB>), reserved, WG_STAGES * WG_STAGE, what)) return r;
    hipLaunchKernelGGL(wgrad_kernel<NB>, dim3((unsigned)(cdiv(p.units, 8) * 8)), dim3(256), WG_STAGES * WG_STAGE, s, p);
    if (const int r = check_launch(what)) return r;
    hipLaunchKernelGGL(wgrad_reduce_kernel<NB>, dim3((unsigned)(p.tiles * 4 * NB)), dim3(256), 0, s, p);
    return check_launch(what);
  };
  return p.nb == 4 ? launch(std::integral_constant<int, 4>{}) : launch(std::integral_constant<int, 3>{});
}
