// Compaction of the softmax branch's K/V cache for gfx950.
//
// After a forward pass the selector has typed every completed block of new tokens.  Only blocks typed
// "attention" are ever read again by later queries, and every (sequence, selector head) keeps a different
// subset.  The cache therefore stores, per (sequence, kv head), its attention-typed blocks back to back from
// block 0, and the tokens of the current incomplete block at one block index shared by all heads (the
// largest count of kept blocks), so that one [B, tokens, heads, D] tensor plus a per-block validity flag
// describes the whole cache (src/nats/models/utils.py:509-588 does this with advanced indexing on a clone).
//
// This is byte movement, bound by HBM: a 16-byte lane (token in block, segment of the head row) is owned by
// one thread for all blocks of its (sequence, head), which walks the region in order.  A kept block only
// moves towards the front (its destination is never behind its source), so walking in order makes the move
// safe in place without a second buffer; the kept blocks are moved NATSL_KV_BATCH at a time, all loads of a batch
// ahead of its stores, which stays safe because the stores of a batch only reach positions in front of every
// source not yet loaded.  Which blocks are kept is scanned once per workgroup into a bit mask in LDS.
#include "natsl_device.h"
#include "natsl_host.h"
#include "../../include/natsl.h"

namespace natsl {

#define NATSL_KV_BATCH 8
#define NATSL_KV_SCAN 1024   // blocks typed per scan round (a multiple of 256)

struct KvCompactParams {
  const char* src[2]; char* dst[2];       // K and V: [B, cap, HKV, row] with row bytes below
  int row[2];
  long src_cap, dst_cap;                  // tokens per sequence in the source / destination tensors
  const void* types; int types_dtype;     // [B, NB, HN, 2]; column 0 == 1 marks an attention-typed block
  const int64_t* n_before;                // [B, HN] blocks already kept per (sequence, selector head); may be null
  int B, HKV, HN, block;
  int src_block0;                         // block index of the region's first block in the source
  int NB, n_complete;                     // blocks in the region / how many of them are complete
  int tail_dst, tail_tokens;              // destination block of the incomplete block (-1: none), tokens in it
  int wgs[2];                             // workgroups per (sequence, head) for K and for V
  int zero_rest;                          // the destination is new memory: blocks that hold nothing get zeros
};

NATSL_DEVICE bool kv_is_attn(const KvCompactParams& p, int b, int s, int hn) {
  size_t i = (((size_t)b * p.NB + s) * p.HN + hn) * 2;
  float t = p.types_dtype == NATSL_F32 ? reinterpret_cast<const float*>(p.types)[i]
                                       : bf16_to_f32(reinterpret_cast<const bf16_t*>(p.types)[i]);
  return rintf(t) == 1.0f;   // the predicate of the router and of both branches (mixed_attn_gdn.py:88 rounds the types)
}

__global__ __launch_bounds__(256) void kv_compact_kernel(KvCompactParams p) {
  // which blocks of the region this (sequence, selector head) keeps: one bit per block, NATSL_KV_SCAN blocks at a time
  __shared__ unsigned long long keep[NATSL_KV_SCAN / 64];
  const int bh = blockIdx.y, b = bh / p.HKV, h = bh % p.HKV, hn = h / (p.HKV / p.HN);
  int wg = blockIdx.x;
  const int which = wg >= p.wgs[0] ? 1 : 0;
  if (which) wg -= p.wgs[0];
  const int row = p.row[which], segs = row / 16;
  const int tid = (int)threadIdx.x, lane = wg * 256 + tid;
  const bool active = lane < p.block * segs;            // idle lanes still take part in the scan and its barriers
  const int tok = lane / segs, seg = lane % segs;
  const size_t tok_stride = (size_t)p.HKV * row;
  const char* sbase = p.src[which] + (size_t)b * p.src_cap * tok_stride + (size_t)h * row + seg * 16;
  char* dbase = p.dst[which] + (size_t)b * p.dst_cap * tok_stride + (size_t)h * row + seg * 16;
  auto saddr = [&](long blk) { return reinterpret_cast<const u32x4*>(sbase + ((size_t)blk * p.block + tok) * tok_stride); };
  auto daddr = [&](long blk) { return reinterpret_cast<u32x4*>(dbase + ((size_t)blk * p.block + tok) * tok_stride); };
  const bool in_place = p.src[which] == p.dst[which];

  long dst = p.n_before ? (long)p.n_before[b * p.HN + hn] : 0;
  for (int base = 0; base < p.n_complete; base += NATSL_KV_SCAN) {
    __syncthreads();
#pragma unroll
    for (int r = 0; r < NATSL_KV_SCAN / 256; ++r) {
      const int s = base + r * 256 + tid;
      const unsigned long long m = __ballot(s < p.n_complete && kv_is_attn(p, b, s, hn));
      if ((tid & 63) == 0) keep[r * 4 + (tid >> 6)] = m;
    }
    __syncthreads();
    // walk the kept blocks NATSL_KV_BATCH at a time: all loads of a batch are in flight before its stores
    unsigned long long m = 0;
    int word = -1;
    auto next = [&]() -> int {
      while (m == 0) {
        if (word + 1 >= NATSL_KV_SCAN / 64) return -1;
        m = keep[++word];
      }
      const int bit = __builtin_ctzll(m);
      m &= m - 1;
      return base + word * 64 + bit;
    };
    for (;;) {
      int s[NATSL_KV_BATCH];
#pragma unroll
      for (int j = 0; j < NATSL_KV_BATCH; ++j) s[j] = next();
      if (s[0] < 0) break;
      u32x4 buf[NATSL_KV_BATCH];
#pragma unroll
      for (int j = 0; j < NATSL_KV_BATCH; ++j)
        if (s[j] >= 0 && active) buf[j] = *saddr(p.src_block0 + s[j]);
#pragma unroll
      for (int j = 0; j < NATSL_KV_BATCH; ++j) {
        if (s[j] < 0) continue;
        // the bound only guards against counts the caller did not size the destination for
        if (active && !(in_place && dst == p.src_block0 + s[j]) && (dst + 1) * p.block <= p.dst_cap) *daddr(dst) = buf[j];
        ++dst;
      }
    }
  }
  if (p.tail_dst >= 0 && active) {
    const long sblk = p.src_block0 + p.NB - 1;
    if (!(in_place && sblk == p.tail_dst)) {
      u32x4 x = {0u, 0u, 0u, 0u};
      if (tok < p.tail_tokens) x = *saddr(sblk);
      *daddr(p.tail_dst) = x;
    }
  }
  // (a cache made in one go costs its bytes once; zeroed as a whole before, the kept blocks' bytes were written twice)
  if (p.zero_rest && active)
    for (long blk = dst; blk < p.dst_cap / p.block; ++blk)
      if (blk != p.tail_dst) *daddr(blk) = (u32x4){0u, 0u, 0u, 0u};
}

// ---- bookkeeping of the kept blocks ----------------------------------------------------------------------------------------
// after[b][hn] = before + attention-typed blocks among the first n_complete, and the largest of them to *host_max (host memory the
// GPU can write: the host needs that one number to size the cache and would otherwise wait for everything enqueued before it asks).
// One workgroup; a wave takes a (sequence, head) pair at a time, its lanes the blocks.
__global__ __launch_bounds__(1024) void kv_counts_kernel(const void* types, const int dtype, const int64_t* before, int64_t* after, int* host_max,
                                                         const int pairs, const int HN, const int NB, const int n_complete) {
  __shared__ int top[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int most = 0;
  for (int i = wave; i < pairs; i += 16) {
    const int b = i / HN, hn = i % HN;
    int n = 0;
    for (int c = lane; c < n_complete; c += 64) {
      const size_t at = (((size_t)b * NB + c) * HN + hn) * 2;
      const float t = dtype == NATSL_F32 ? reinterpret_cast<const float*>(types)[at] : bf16_to_f32(reinterpret_cast<const bf16_t*>(types)[at]);
      n += rintf(t) == 1.f;
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) n += __shfl_xor(n, d);
    const int64_t total = n + (before ? before[i] : 0);
    if (lane == 0) after[i] = total;
    most = max(most, (int)total);
  }
  if (lane == 0) top[wave] = most;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 16; ++w) most = max(most, top[w]);
    *host_max = most;
    __threadfence_system();
  }
}
// valid[b][i][hn]: kept blocks, and the incomplete block at `tail` (-1: none).  The workgroups behind those of the flags, a wave per
// (sequence, head) each, leave the sum of g [B, T, H] over the incomplete block's tokens (the last `rest`; 0 where there are none).
__global__ __launch_bounds__(256) void kv_flags_kernel(const int64_t* after, uint8_t* valid, const long long n, const int HN, const int blocks, const int tail,
                                                       const unsigned flag_wgs, const float* g, float* g_sum, const int B, const int T, const int H,
                                                       const int rest) {
  if (blockIdx.x < flag_wgs) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int hn = (int)(i % HN), blk = (int)(i / HN % blocks), b = (int)(i / ((long long)HN * blocks));
    valid[i] = blk < after[(size_t)b * HN + hn] || blk == tail;
    return;
  }
  const long long pair = (long long)(blockIdx.x - flag_wgs) * 4 + (threadIdx.x >> 6);
  if (pair >= (long long)B * H) return;
  const int b = (int)(pair / H), h = (int)(pair % H);
  float s = 0.f;
  for (int t = threadIdx.x & 63; t < rest; t += 64) s += g[((size_t)b * T + T - rest + t) * H + h];
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) s += __shfl_xor(s, d);
  if ((threadIdx.x & 63) == 0) g_sum[pair] = s;
}

// ---- a cache's first prompt -------------------------------------------------------------------------------------------------
// dst [B, block, row] = the last `rest` tokens of src [B, T, row], zeros behind them, for several tensors in one launch: the incomplete
// block's rows of a cache that was empty before.  Fills and strided copies of their own were eleven launches of a prompt (six where it
// ends on a block's end), 4.7 us each where the GPU is the limit and about 10 us of host time.  `unit`: bytes a thread moves, what the
// row's length and the addresses allow.
struct TailParams {
  natsl_tail_seg seg[NATSL_TAIL_SEGS];
  int unit[NATSL_TAIL_SEGS];
  unsigned first[NATSL_TAIL_SEGS + 1];   // the segments' first workgroups
  int n, B, T, block, rest;
};
template <typename U>
NATSL_DEVICE void tail_unit(const natsl_tail_seg& s, const long long i, const TailParams& p) {
  const int per_row = (int)(s.row_bytes / sizeof(U));
  const long long token = i / per_row;
  const int at = (int)(i - token * per_row), b = (int)(token / p.block), t = (int)(token - (long long)b * p.block);
  if (b >= p.B) return;
  U x{};
  if (t < p.rest) x = reinterpret_cast<const U*>(s.src)[((size_t)b * p.T + p.T - p.rest + t) * per_row + at];
  reinterpret_cast<U*>(s.dst)[i] = x;
}
__global__ __launch_bounds__(256) void block_tails_kernel(const TailParams p) {
  int k = 0;
  while (k + 1 < p.n && blockIdx.x >= p.first[k + 1]) ++k;
  const long long i = (long long)(blockIdx.x - p.first[k]) * 256 + threadIdx.x;
  if (p.unit[k] == 16) tail_unit<u32x4>(p.seg[k], i, p);
  else if (p.unit[k] == 4) tail_unit<unsigned>(p.seg[k], i, p);
  else tail_unit<uint16_t>(p.seg[k], i, p);
}

// The state that the next block starts from where a prompt ends on a block's end: the final state where the last block's own type is
// linear, else the state that entered it, decayed by the block's g where asked for (src/nats/ops/gated_delta_rule/chunk_fwd.py:178-206).
__global__ __launch_bounds__(256) void roll_state_kernel(const float* ht, const float* hs, const float* gs, const void* last, const int dtype,
                                                         const long long stride_b, const long long stride_h, float* out, const int H, const int HN,
                                                         const int n4) {
  const int b = blockIdx.y / H, h = blockIdx.y % H;
  const long long at = b * stride_b + (h / (H / HN)) * stride_h + 1;
  const float t = dtype == NATSL_F32 ? reinterpret_cast<const float*>(last)[at] : bf16_to_f32(reinterpret_cast<const bf16_t*>(last)[at]);
  const bool linear = t > 0.f;
  const float f = linear || !gs ? 1.f : expf(gs[blockIdx.y]);
  const f32x4* src = reinterpret_cast<const f32x4*>(linear ? ht : hs) + (size_t)blockIdx.y * n4;
  f32x4* dst = reinterpret_cast<f32x4*>(out) + (size_t)blockIdx.y * n4;
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n4; i += gridDim.x * 256) {
    f32x4 x = src[i];
    x *= f;
    dst[i] = x;
  }
}

}  // namespace natsl

using namespace natsl;

static int kv_compact(const char* what, bool zero_rest, const void* src_k, const void* src_v, long long src_tokens, int src_block0, void* dst_k,
                      void* dst_v, long long dst_tokens, const void* types, int types_dtype, const int64_t* n_before, int B, int HKV, int HN, int K,
                      int V, int dtype, int block, int NB, int n_complete, int tail_dst, int tail_tokens, natsl_stream_t stream) {
  if (!src_k || !src_v || !dst_k || !dst_v || !types) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (dtype != NATSL_BF16 && dtype != NATSL_F32) return fail(NATSL_ERR_UNSUPPORTED, "%s: tensors must be f32 or bf16", what);
  if (types_dtype != NATSL_BF16 && types_dtype != NATSL_F32) return fail(NATSL_ERR_UNSUPPORTED, "%s: block types must be f32 or bf16", what);
  if (B <= 0 || HKV <= 0 || HN <= 0 || K <= 0 || V <= 0 || block <= 0 || NB <= 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  if (HKV % HN) return fail(NATSL_ERR_INVALID, "%s: HKV=%d must be a multiple of HN=%d", what, HKV, HN);
  const int esize = dtype == NATSL_BF16 ? 2 : 4;
  if ((K * esize) % 16 || (V * esize) % 16) return fail(NATSL_ERR_UNSUPPORTED, "%s: head rows must be multiples of 16 bytes (K=%d, V=%d)", what, K, V);
  if (n_complete < 0 || n_complete > NB || (tail_dst >= 0 && n_complete != NB - 1) || (tail_dst < 0 && n_complete != NB))
    return fail(NATSL_ERR_INVALID, "%s: n_complete=%d does not fit NB=%d with%s an incomplete block", what, n_complete, NB, tail_dst >= 0 ? "" : "out");
  if (tail_dst >= 0 && (tail_tokens <= 0 || tail_tokens >= block)) return fail(NATSL_ERR_INVALID, "%s: tail_tokens=%d outside (0, %d)", what, tail_tokens, block);
  if (src_block0 < 0) return fail(NATSL_ERR_INVALID, "%s: negative source block", what);
  // the source must hold the region's complete blocks and the tokens of the incomplete one
  const long long src_need = ((long long)src_block0 + n_complete) * block + (tail_dst >= 0 ? tail_tokens : 0);
  if (src_tokens < src_need) return fail(NATSL_ERR_INVALID, "%s: source holds %lld tokens per sequence, the region needs %lld", what, src_tokens, src_need);
  // the destination must hold every block that can be written: at most n_complete more than the largest count the
  // caller has (which it bounds by tail_dst or by dst_tokens itself); the in-place case never moves a block backwards
  if (tail_dst >= 0 && ((long long)tail_dst + 1) * block > dst_tokens) return fail(NATSL_ERR_INVALID, "%s: destination too small for the incomplete block at %d", what, tail_dst);
  if ((src_k == dst_k) != (src_v == dst_v)) return fail(NATSL_ERR_INVALID, "%s: K and V must both be in place or both not", what);
  if (src_k == dst_k && src_tokens != dst_tokens) return fail(NATSL_ERR_INVALID, "%s: in place, source and destination sizes must agree", what);
  if ((long long)B * HKV > 65535) return fail(NATSL_ERR_UNSUPPORTED, "%s: B*HKV=%lld above 65535", what, (long long)B * HKV);
  KvCompactParams p;
  p.src[0] = (const char*)src_k; p.src[1] = (const char*)src_v; p.dst[0] = (char*)dst_k; p.dst[1] = (char*)dst_v;
  p.row[0] = K * esize; p.row[1] = V * esize;
  p.src_cap = (long)src_tokens; p.dst_cap = (long)dst_tokens;
  p.types = types; p.types_dtype = types_dtype; p.n_before = n_before;
  p.B = B; p.HKV = HKV; p.HN = HN; p.block = block; p.src_block0 = src_block0; p.NB = NB; p.n_complete = n_complete;
  p.tail_dst = tail_dst; p.tail_tokens = tail_tokens;
  p.zero_rest = zero_rest ? 1 : 0;
  p.wgs[0] = cdiv(block * (p.row[0] / 16), 256); p.wgs[1] = cdiv(block * (p.row[1] / 16), 256);
  hipLaunchKernelGGL(kv_compact_kernel, dim3(p.wgs[0] + p.wgs[1], B * HKV), dim3(256), 0, (hipStream_t)stream, p);
  return check_launch(what);
}

extern "C" int natsl_kv_compact(const void* src_k, const void* src_v, long long src_tokens, int src_block0, void* dst_k,
                                void* dst_v, long long dst_tokens, const void* types, int types_dtype,
                                const int64_t* n_before, int B, int HKV, int HN, int K, int V, int dtype, int block,
                                int NB, int n_complete, int tail_dst, int tail_tokens, natsl_stream_t stream) {
  return kv_compact("natsl_kv_compact", false, src_k, src_v, src_tokens, src_block0, dst_k, dst_v, dst_tokens, types, types_dtype, n_before, B, HKV, HN,
                    K, V, dtype, block, NB, n_complete, tail_dst, tail_tokens, stream);
}

extern "C" int natsl_kv_collect(const void* src_k, const void* src_v, long long src_tokens, void* dst_k, void* dst_v, long long dst_tokens,
                                const void* types, int types_dtype, int B, int HKV, int HN, int K, int V, int dtype, int block, int NB, int n_complete,
                                int tail_dst, int tail_tokens, natsl_stream_t stream) {
  const char* what = "natsl_kv_collect";
  if (src_k == dst_k || src_v == dst_v) return fail(NATSL_ERR_INVALID, "%s: the cache must be new memory", what);
  if (block <= 0 || dst_tokens <= 0 || dst_tokens % block) return fail(NATSL_ERR_INVALID, "%s: the cache must hold whole blocks", what);
  return kv_compact(what, true, src_k, src_v, src_tokens, 0, dst_k, dst_v, dst_tokens, types, types_dtype, nullptr, B, HKV, HN, K, V, dtype, block, NB,
                    n_complete, tail_dst, tail_tokens, stream);
}

extern "C" int natsl_kv_counts(const void* types, int types_dtype, const int64_t* n_before, int64_t* n_after, int32_t* host_max, int B, int HN, int NB,
                               int n_complete, natsl_stream_t stream) {
  const char* what = "natsl_kv_counts";
  if (!types || !n_after || !host_max) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (B <= 0 || HN <= 0 || NB <= 0 || n_complete < 0 || n_complete > NB) return fail(NATSL_ERR_INVALID, "%s: bad dimension", what);
  if (types_dtype != NATSL_BF16 && types_dtype != NATSL_F32) return fail(NATSL_ERR_UNSUPPORTED, "%s: block types must be f32 or bf16", what);
  hipLaunchKernelGGL(kv_counts_kernel, dim3(1), dim3(1024), 0, reinterpret_cast<hipStream_t>(stream), types, types_dtype, n_before, n_after, host_max,
                     B * HN, HN, NB, n_complete);
  return check_launch(what);
}

static int kv_flags(const char* what, const int64_t* n_after, uint8_t* valid, int B, int blocks, int HN, int tail_block, const float* g, float* g_sum,
                    int T, int H, int rest, natsl_stream_t stream) {
  if (!n_after || !valid) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (B <= 0 || HN <= 0 || blocks <= 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  const long long n = (long long)B * blocks * HN;
  const unsigned flag_wgs = (unsigned)((n + 255) / 256), sum_wgs = g_sum ? (unsigned)(((long long)B * H + 3) / 4) : 0u;
  hipLaunchKernelGGL(kv_flags_kernel, dim3(flag_wgs + sum_wgs), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), n_after, valid, n, HN, blocks,
                     tail_block, flag_wgs, g, g_sum, B, T, H, rest);
  return check_launch(what);
}

extern "C" int natsl_kv_flags(const int64_t* n_after, uint8_t* valid, int B, int blocks, int HN, int tail_block, natsl_stream_t stream) {
  return kv_flags("natsl_kv_flags", n_after, valid, B, blocks, HN, tail_block, nullptr, nullptr, 0, 0, 0, stream);
}

extern "C" int natsl_kv_note(const int64_t* n_after, uint8_t* valid, int B, int blocks, int HN, int tail_block, const float* g, float* g_sum, int T, int H,
                             int rest, natsl_stream_t stream) {
  const char* what = "natsl_kv_note";
  if (!g || !g_sum) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (T <= 0 || H <= 0 || rest < 0 || rest > T) return fail(NATSL_ERR_INVALID, "%s: %d of %d tokens, %d heads", what, rest, T, H);
  return kv_flags(what, n_after, valid, B, blocks, HN, tail_block, g, g_sum, T, H, rest, stream);
}

extern "C" int natsl_block_tails(const natsl_tail_seg* segs, int n, int B, int T, int block, int rest, natsl_stream_t stream) {
  const char* what = "natsl_block_tails";
  if (!segs) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (n <= 0 || n > NATSL_TAIL_SEGS) return fail(NATSL_ERR_INVALID, "%s: %d tensors (1 to %d)", what, n, NATSL_TAIL_SEGS);
  if (B <= 0 || T <= 0 || block <= 0 || rest < 0 || rest > T || rest > block)
    return fail(NATSL_ERR_INVALID, "%s: B=%d T=%d block=%d rest=%d", what, B, T, block, rest);
  TailParams p{};
  long long wgs = 0;
  for (int i = 0; i < n; ++i) {
    const natsl_tail_seg& s = segs[i];
    if (!s.src || !s.dst) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
    const size_t bits = (size_t)s.src | (size_t)s.dst | (size_t)s.row_bytes;
    if (s.row_bytes <= 0 || s.row_bytes > (1ll << 30) || bits % 2)
      return fail(NATSL_ERR_UNSUPPORTED, "%s: rows of %lld bytes at odd places", what, (long long)s.row_bytes);
    p.seg[i] = s;
    p.unit[i] = bits % 16 == 0 ? 16 : bits % 4 == 0 ? 4 : 2;
    p.first[i] = (unsigned)wgs;
    wgs += ((long long)B * block * (s.row_bytes / p.unit[i]) + 255) / 256;
    if (wgs >= (1ll << 31)) return fail(NATSL_ERR_UNSUPPORTED, "%s: too many rows", what);
  }
  p.first[n] = (unsigned)wgs;
  p.n = n; p.B = B; p.T = T; p.block = block; p.rest = rest;
  hipLaunchKernelGGL(block_tails_kernel, dim3((unsigned)wgs), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), p);
  return check_launch(what);
}

extern "C" int natsl_roll_state(const float* ht, const float* hs, const float* gs, const void* last_types, int types_dtype, int64_t stride_b,
                                int64_t stride_h, float* out, int B, int H, int HN, int64_t state_elems, natsl_stream_t stream) {
  const char* what = "natsl_roll_state";
  if (!ht || !hs || !last_types || !out) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (B <= 0 || H <= 0 || HN <= 0 || H % HN || state_elems <= 0 || (long long)B * H > 65535)
    return fail(NATSL_ERR_INVALID, "%s: B=%d H=%d HN=%d", what, B, H, HN);
  if (types_dtype != NATSL_BF16 && types_dtype != NATSL_F32) return fail(NATSL_ERR_UNSUPPORTED, "%s: block types must be f32 or bf16", what);
  if (state_elems % 4 || state_elems >= (1ll << 31) || ((size_t)ht | (size_t)hs | (size_t)out) % 16)
    return fail(NATSL_ERR_UNSUPPORTED, "%s: states must be multiples of four elements, aligned to 16 bytes", what);
  const int n4 = (int)(state_elems / 4);
  hipLaunchKernelGGL(roll_state_kernel, dim3((unsigned)cdiv(n4, 256 * 8), (unsigned)(B * H)), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), ht, hs, gs,
                     last_types, types_dtype, (long long)stride_b, (long long)stride_h, out, H, HN, n4);
  return check_launch(what);
}
