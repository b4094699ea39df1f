// Decode-time kernels of the NAtS-L hybrid layer for gfx950: tokens that continue the current
// (incomplete) selector block of a sequence whose state is cached.
//
//   gdn_recurrent_kernel   the gated delta rule token by token on a cached state
//                          (src/nats/ops/gated_delta_rule/fused_recurrent.py:28-358, the branch the
//                          reference takes at decode: UPDATE_HS_FOR_EACH_ITER with one selector block)
//   attn_masked_kernel     softmax attention of a few queries over cached keys/values under an explicit
//                          visibility mask (the scaled_dot_product_attention call at
//                          src/nats/ops/mixed_ops/mixed_attn_gdn.py:475-481)
//
// Both are memory-bound: the first reads and writes the fp32 state once, the second reads K and V once per
// query.  No matrix cores: per token the delta rule is two K-long dot products and one rank-1 update.
#include "natsl_decode_device.h"
#include "natsl_host.h"

namespace natsl {

// the gated delta rule / SSD recurrence: a workgroup is four waves of 16 state columns each
template <int DK, bool DELTA>
__global__ __launch_bounds__(256) void gdn_recurrent_kernel(const RecurrentParams p) {
  const int col16 = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (col16 * 16 >= p.V) return;  // V is a multiple of 16: whole waves leave together
  recurrent_columns<DK, DELTA>(p, blockIdx.y, col16);
}

// attention of a few queries over cached keys: one workgroup of NW waves per (split, query head, query row)
constexpr int MASKED_WAVES = 8;

template <int DK, int DV, bool F32, int NW>
__global__ __launch_bounds__(64 * NW) void attn_masked_kernel(const AttnParams p) {
  attend<DK, DV, F32, NW>(p, blockIdx.z / p.nsplit, blockIdx.x, blockIdx.y, blockIdx.z % p.nsplit, CachedRows());
}

// joins the splits of one query: one wave per (sequence, query, head)
template <int DV>
__global__ __launch_bounds__(64) void attn_masked_join_kernel(const AttnParams p) {
  constexpr int CPL = DV / 64;
  const size_t row = ((size_t)blockIdx.z * p.TQ + blockIdx.x) * p.HQ + blockIdx.y;
  float o[CPL];
  join_splits<DV>(p.partials + row * p.nsplit * (2 + DV), p.nsplit, o);
#pragma unroll
  for (int j = 0; j < CPL; ++j) st_any(p.o, p.dtype, row * DV + CPL * threadIdx.x + j, o[j]);
}

// The two halves of a decode step side by side: the first workgroups attend (4 waves each), the rest run the recurrence (4
// waves of 16 state columns).  Both are bound by memory and neither fills the chip at small batches; one launch less, and the
// state's traffic overlaps the keys'.
template <int DKA, int DVA, int DK, bool DELTA>
__global__ __launch_bounds__(256) void attend_and_recur_kernel(const AttnParams a, const RecurrentParams r, const int n_attn) {
  int id = blockIdx.x;
  if (id < n_attn) {
    const int split = id % a.nsplit;
    id /= a.nsplit;
    const int hq = id % a.HQ;
    id /= a.HQ;
    attend<DKA, DVA, false, 4>(a, id / a.TQ, id % a.TQ, hq, split, CachedRows());
    return;
  }
  id -= n_attn;
  const int per = (r.V + 63) / 64, col16 = (id % per) * 4 + (threadIdx.x >> 6);
  if (col16 * 16 >= r.V) return;
  recurrent_columns<DK, DELTA>(r, id / per, col16);
}

// Enough splits for 1024 attending workgroups (16 waves per CU keep ~256 KiB of loads in flight), no wave without a chunk.
int attend_splits(int queries, int TK) {
  int want = cdiv(1024, queries), most = cdiv(TK, 4 * KEYS_PER_CHUNK);
  if (want > most) want = most;
  return want < 1 ? 1 : want > ATTEND_MAX_SPLITS ? ATTEND_MAX_SPLITS : want;
}

int launch_attend_and_recur(const char* what, const AttnParams& a, const RecurrentParams& r, bool delta, int K, int KA, int VA, hipStream_t s) {
  const long long n_attn = (long long)a.B * a.TQ * a.HQ * a.nsplit, n_rec = (long long)r.N * r.H * cdiv(r.V, 64);
  if (n_attn + n_rec > 0x7fffffffll) return fail(NATSL_ERR_UNSUPPORTED, "%s: too many workgroups", what);
  const dim3 grid((unsigned)(n_attn + n_rec));
#define NATSL_AR(KK, VV, KL, DD)                                                                                             \
  if (KA == KK && VA == VV && K == KL && delta == DD) {                                                                      \
    hipLaunchKernelGGL((attend_and_recur_kernel<KK, VV, KL, DD>), grid, dim3(256), 0, s, a, r, (int)n_attn);                 \
    return check_launch(what);                                                                                               \
  }
#define NATSL_AR3(KK, VV)                                                                                                    \
  NATSL_AR(KK, VV, 64, true) NATSL_AR(KK, VV, 128, true) NATSL_AR(KK, VV, 192, true) NATSL_AR(KK, VV, 64, false)             \
  NATSL_AR(KK, VV, 128, false) NATSL_AR(KK, VV, 192, false)
  NATSL_AR3(64, 64) NATSL_AR3(64, 128) NATSL_AR3(128, 64) NATSL_AR3(128, 128)
#undef NATSL_AR3
#undef NATSL_AR
  return fail(NATSL_ERR_UNSUPPORTED, "%s: head dims %d (linear), %d / %d (attention) not built", what, K, KA, VA);
}

}  // namespace natsl

using namespace natsl;

// checks and fills in what both the recurrent entries and the joint decode entry need
static int recurrent_params(RecurrentParams& p, bool delta, const char* what, const void* q, const void* k, const void* v, const float* g,
                         const float* g_cumsum, const void* beta, const float* h0, float* h_block_start, void* o, float* ht,
                         const void* types, int types_dtype, const int32_t* n_tokens_in_block, int n_tokens_in_block_scalar,
                         int N, int T, int H, int HN, int K, int V, int block, float scale, int flags, int dtype) {
  const bool query_only = (flags & NATSL_QUERY_ONLY) != 0;
  if (!q || !g || !h_block_start || !o || !types || (!query_only && (!k || !v || (delta && !beta))))
    return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (dtype != NATSL_BF16 && dtype != NATSL_F32) return fail(NATSL_ERR_UNSUPPORTED, "%s: tensors must be f32 or bf16", what);
  if (types_dtype != NATSL_BF16 && types_dtype != NATSL_F32) return fail(NATSL_ERR_UNSUPPORTED, "%s: block types must be f32 or bf16", what);
  if (N <= 0 || T <= 0 || H <= 0 || HN <= 0 || block <= 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  if (H % HN) return fail(NATSL_ERR_INVALID, "%s: H=%d must be a multiple of HN=%d", what, H, HN);
  if (V <= 0 || V % 16) return fail(NATSL_ERR_UNSUPPORTED, "%s: V=%d must be a multiple of 16", what, V);
  if ((long long)N * H > 65535) return fail(NATSL_ERR_UNSUPPORTED, "%s: N*H=%lld above 65535", what, (long long)N * H);
  if (!n_tokens_in_block && (n_tokens_in_block_scalar < 0 || n_tokens_in_block_scalar >= block))
    return fail(NATSL_ERR_INVALID, "%s: n_tokens_in_current_block=%d outside [0, %d)", what, n_tokens_in_block_scalar, block);
  p.q = q; p.k = k; p.v = v; p.g = g; p.g_cumsum = g_cumsum; p.beta = beta; p.h0 = h0; p.hcur = h_block_start; p.o = o; p.ht = ht;
  p.types = types; p.types_dtype = types_dtype; p.n_in_block = n_tokens_in_block; p.n_in_block_scalar = n_tokens_in_block_scalar;
  p.N = N; p.T = T; p.H = H; p.HN = HN; p.V = V; p.block = block; p.dtype = dtype; p.scale = scale;
  p.decay = (flags & NATSL_DECAY_NON_LINEAR) != 0; p.l2norm = (flags & NATSL_QK_L2NORM) != 0; p.query_only = query_only ? 1 : 0;
  p.kv_stride = T; p.kv_first = 0; p.fresh_start = (flags & NATSL_FRESH_BLOCK_START) != 0; p.g_cumsum_out = nullptr;
  p.aligned = (((uintptr_t)q | (uintptr_t)k) & 15) == 0;
  if (p.fresh_start && query_only) return fail(NATSL_ERR_INVALID, "%s: the query-only form reads the block-start state", what);
  if (K != 64 && K != 128 && K != 192) return fail(NATSL_ERR_UNSUPPORTED, "%s: K=%d not built (supported: 64, 128, 192)", what, K);
  return NATSL_OK;
}

static int recurrent_fwd(const RecurrentParams& p, bool delta, const char* what, int K, natsl_stream_t stream) {
  const dim3 grid(cdiv(p.V, 64), p.N * p.H);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (K == 128 && delta) hipLaunchKernelGGL((gdn_recurrent_kernel<128, true>), grid, dim3(256), 0, s, p);
  else if (K == 64 && delta) hipLaunchKernelGGL((gdn_recurrent_kernel<64, true>), grid, dim3(256), 0, s, p);
  else if (K == 128) hipLaunchKernelGGL((gdn_recurrent_kernel<128, false>), grid, dim3(256), 0, s, p);
  else if (K == 64) hipLaunchKernelGGL((gdn_recurrent_kernel<64, false>), grid, dim3(256), 0, s, p);
  else if (delta) hipLaunchKernelGGL((gdn_recurrent_kernel<192, true>), grid, dim3(256), 0, s, p);
  else hipLaunchKernelGGL((gdn_recurrent_kernel<192, false>), grid, dim3(256), 0, s, p);
  return check_launch(what);
}

extern "C" int natsl_gdn_recurrent_fwd(const void* q, const void* k, const void* v, const float* g, const float* g_cumsum,
                                       const void* beta, const float* h0, float* h_block_start, void* o, float* ht,
                                       const void* types, int types_dtype, const int32_t* n_tokens_in_block,
                                       int n_tokens_in_block_scalar, int N, int T, int H, int HN, int K, int V, int block,
                                       float scale, int flags, int dtype, natsl_stream_t stream) {
  RecurrentParams p;
  const int rc = recurrent_params(p, true, "natsl_gdn_recurrent_fwd", q, k, v, g, g_cumsum, beta, h0, h_block_start, o, ht, types, types_dtype,
                                  n_tokens_in_block, n_tokens_in_block_scalar, N, T, H, HN, K, V, block, scale, flags, dtype);
  return rc != NATSL_OK ? rc : recurrent_fwd(p, true, "natsl_gdn_recurrent_fwd", K, stream);
}

extern "C" int natsl_mamba_recurrent_fwd(const void* q, const void* k, const void* v, const float* g, const float* g_cumsum,
                                         const float* h0, float* h_block_start, void* o, float* ht, const void* types,
                                         int types_dtype, const int32_t* n_tokens_in_block, int n_tokens_in_block_scalar, int N,
                                         int T, int H, int HN, int K, int V, int block, float scale, int flags, int dtype,
                                         natsl_stream_t stream) {
  RecurrentParams p;
  const int rc = recurrent_params(p, false, "natsl_mamba_recurrent_fwd", q, k, v, g, g_cumsum, nullptr, h0, h_block_start, o, ht, types,
                                  types_dtype, n_tokens_in_block, n_tokens_in_block_scalar, N, T, H, HN, K, V, block, scale, flags, dtype);
  return rc != NATSL_OK ? rc : recurrent_fwd(p, false, "natsl_mamba_recurrent_fwd", K, stream);
}

// splits per query: enough workgroups to cover the CUs twice, at least two chunk groups per split
static int attn_masked_splits(int B, int TQ, int TK, int HQ) {
  const long long queries = (long long)B * TQ * HQ;
  const int groups = cdiv(TK, 1024);
  long long want = cdiv(512, (int)(queries < 512 ? queries : 512));
  if (want > groups) want = groups;
  if (want > 16) want = 16;
  return want < 1 ? 1 : (int)want;
}

extern "C" size_t natsl_attn_masked_workspace_bytes(int B, int TQ, int TK, int HQ, int V) {
  const int ns = attn_masked_splits(B, TQ, TK, HQ);
  return ns > 1 ? (size_t)B * TQ * HQ * ns * (2 + V) * sizeof(float) : 0;
}

static int attn_params(AttnParams& p, const char* what, const void* q, const void* k, const void* v, const uint8_t* mask, void* o, int B, int TQ,
                       int TK, int HQ, int HKV, int HM, int K, int V, float scale, int dtype, long long k_batch_stride,
                       long long v_batch_stride) {
  if (!q || !k || !v || !mask || !o) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (dtype != NATSL_BF16 && dtype != NATSL_F32) return fail(NATSL_ERR_UNSUPPORTED, "%s: tensors must be f32 or bf16", what);
  if (B <= 0 || TQ <= 0 || TK <= 0 || HQ <= 0 || HKV <= 0 || HM <= 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  if (HQ % HKV || HQ % HM) return fail(NATSL_ERR_INVALID, "%s: HQ=%d must be a multiple of HKV=%d and of the mask heads %d", what, HQ, HKV, HM);
  if ((K != 64 && K != 128) || (V != 64 && V != 128))
    return fail(NATSL_ERR_UNSUPPORTED, "%s: head dims K=%d, V=%d not built (supported: 64/128 x 64/128)", what, K, V);
  if ((k_batch_stride && k_batch_stride < (long long)TK * HKV * K) || (v_batch_stride && v_batch_stride < (long long)TK * HKV * V) ||
      k_batch_stride % 8 || v_batch_stride % 8)
    return fail(NATSL_ERR_INVALID, "%s: a batch stride must be 0 (dense) or at least TK*HKV*D, and a multiple of 8 elements", what);
  p.q = q; p.k = k; p.v = v; p.mask = mask; p.o = o;
  p.B = B; p.TQ = TQ; p.TK = TK; p.HQ = HQ; p.HKV = HKV; p.HM = HM; p.dtype = dtype;
  p.scale_log2 = scale * 1.4426950408889634f;
  p.k_bs = k_batch_stride ? (size_t)k_batch_stride : (size_t)TK * HKV * K;
  p.v_bs = v_batch_stride ? (size_t)v_batch_stride : (size_t)TK * HKV * V;
  p.valid = nullptr; p.valid_bs = p.n_kept = p.n_in = p.own_visible = 0; p.block = 64;
  return NATSL_OK;
}

static int join_if_split(const char* what, const AttnParams& p, int V, hipStream_t s) {
  if (!p.partials) return NATSL_OK;
  const dim3 grid(p.TQ, p.HQ, p.B);
  if (V == 128) hipLaunchKernelGGL((attn_masked_join_kernel<128>), grid, dim3(64), 0, s, p);
  else hipLaunchKernelGGL((attn_masked_join_kernel<64>), grid, dim3(64), 0, s, p);
  return check_launch(what);
}

// The one implementation behind both entry points.  `strict`: a workspace smaller than the split needs is an error
// instead of a silent fall-back to one workgroup per query.
static int attn_masked_run(const char* what, const void* q, const void* k, const void* v, const uint8_t* mask, void* o, int B, int TQ,
                           int TK, int HQ, int HKV, int HM, int K, int V, float scale, int dtype, void* workspace,
                           size_t workspace_bytes, bool strict, long long k_batch_stride, long long v_batch_stride,
                           natsl_stream_t stream) {
  AttnParams p;
  int rc = attn_params(p, what, q, k, v, mask, o, B, TQ, TK, HQ, HKV, HM, K, V, scale, dtype, k_batch_stride, v_batch_stride);
  if (rc != NATSL_OK) return rc;
  // without a workspace (or with one that is too small) every query is handled by one workgroup
  p.nsplit = attn_masked_splits(B, TQ, TK, HQ);
  const size_t need = natsl_attn_masked_workspace_bytes(B, TQ, TK, HQ, V);
  if (!workspace || workspace_bytes < need) {
    if (strict && need > 0)
      return fail(NATSL_ERR_WORKSPACE, "%s: this shape needs %zu bytes of split scratch, the built-in buffer holds %zu", what, need, workspace_bytes);
    p.nsplit = 1;
  }
  p.partials = p.nsplit > 1 ? reinterpret_cast<float*>(workspace) : nullptr;
  if (TQ > 65535 || HQ > 65535 || (long long)B * p.nsplit > 65535) return fail(NATSL_ERR_UNSUPPORTED, "%s: grid dimension above 65535", what);
  const dim3 grid(TQ, HQ, B * p.nsplit);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
#define NATSL_MA(KK, VV, FF)                                                                                        \
  if (K == KK && V == VV && (dtype == NATSL_F32) == FF)                                                             \
    hipLaunchKernelGGL((attn_masked_kernel<KK, VV, FF, MASKED_WAVES>), grid, dim3(64 * MASKED_WAVES), 0, s, p);
  NATSL_MA(128, 128, false) NATSL_MA(64, 64, false) NATSL_MA(64, 128, false) NATSL_MA(128, 64, false)
  NATSL_MA(128, 128, true) NATSL_MA(64, 64, true) NATSL_MA(64, 128, true) NATSL_MA(128, 64, true)
#undef NATSL_MA
  rc = check_launch(what);
  return rc != NATSL_OK ? rc : join_if_split(what, p, V, s);
}

extern "C" int natsl_attn_masked_fwd(const void* q, const void* k, const void* v, const uint8_t* mask, void* o, int B, int TQ,
                                     int TK, int HQ, int HKV, int HM, int K, int V, float scale, int dtype, void* workspace,
                                     size_t workspace_bytes, int64_t k_batch_stride, int64_t v_batch_stride,
                                     natsl_stream_t stream) {
  return attn_masked_run("natsl_attn_masked_fwd", q, k, v, mask, o, B, TQ, TK, HQ, HKV, HM, K, V, scale, dtype, workspace,
                         workspace_bytes, false, k_batch_stride, v_batch_stride, stream);
}

// ---- the variant that allocates nothing -----------------------------------------------------------------------------
// The split scratch (per query and split: running maximum, sum and DV partial outputs, fp32) lives in a device array
// of this library instead of a caller's workspace.  Every GPU holds its own copy at its own address until the process
// ends; the array's name is a host-side handle, so its device address is looked up once per device and only that
// pointer is ever handed to a kernel.  Nothing in it has to start at zero: every (query, split) slot that the join
// kernel reads is written by the split kernel of the same call.  Calls that overlap on one GPU share the array and race.
#define NATSL_ATTN_STATIC_SCRATCH_BYTES (256u << 10)
static __device__ __align__(256) unsigned char scratch[NATSL_ATTN_STATIC_SCRATCH_BYTES];

#include <mutex>
static void* scratch_device_address(const char* what, int* rc) {
  constexpr int MAX_DEVICES = 64;
  static void* ptr[MAX_DEVICES];
  static std::mutex mu;
  *rc = NATSL_OK;
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
    *rc = fail(NATSL_ERR_LAUNCH, "%s: cannot name the current device (%s)", what, hipGetErrorString(e));
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr[dev]) {
    void* a = nullptr;
    e = hipGetSymbolAddress(&a, HIP_SYMBOL(scratch));   // with device `dev` current: that device's copy
    if (e != hipSuccess || !a) {
      *rc = fail(NATSL_ERR_LAUNCH, "%s: hipGetSymbolAddress failed on device %d (%s)", what, dev, hipGetErrorString(e));
      return nullptr;
    }
    ptr[dev] = a;
  }
  return ptr[dev];
}

extern "C" size_t natsl_attn_masked_static_scratch_bytes(void) { return NATSL_ATTN_STATIC_SCRATCH_BYTES; }

extern "C" int natsl_attn_masked_fwd_static(const void* q, const void* k, const void* v, const uint8_t* mask, void* o, int B,
                                            int TQ, int TK, int HQ, int HKV, int HM, int K, int V, float scale, int dtype,
                                            natsl_stream_t stream) {
  const char* what = "natsl_attn_masked_fwd_static";
  int rc;
  void* ws = scratch_device_address(what, &rc);
  if (!ws) return rc;
  return attn_masked_run(what, q, k, v, mask, o, B, TQ, TK, HQ, HKV, HM, K, V, scale, dtype, ws, NATSL_ATTN_STATIC_SCRATCH_BYTES,
                         true, 0, 0, stream);
}

// ---- a whole decode step of the mixed operators: two launches ---------------------------------------------------------
extern "C" size_t natsl_decode_workspace_bytes(int B, int T, int TK, int HQ, int VA) {
  const int ns = B > 0 && T > 0 && TK > 0 && HQ > 0 ? attend_splits(B * T * HQ, TK) : 1;
  return ns > 1 ? (size_t)B * T * HQ * ns * (2 + VA) * sizeof(float) : 0;
}

extern "C" int natsl_decode_fwd(int is_delta, const void* q_attn, const void* k_attn, const void* v_attn, const uint8_t* mask, void* o_attn,
                                int B, int T, int TK, int HQ, int HKV, int HM, int KA, int VA, float scale_attn, int64_t k_batch_stride,
                                int64_t v_batch_stride, void* workspace, size_t workspace_bytes, const void* q, const void* k,
                                const void* v, const float* g, const float* g_cumsum, const void* beta, const float* h0,
                                float* h_block_start, void* o, float* ht, const void* types, int types_dtype,
                                const int32_t* n_tokens_in_block, int n_tokens_in_block_scalar, int H, int HN, int K, int V, int block,
                                float scale, int flags, natsl_stream_t stream) {
  const char* what = "natsl_decode_fwd";
  AttnParams a;
  int rc = attn_params(a, what, q_attn, k_attn, v_attn, mask, o_attn, B, T, TK, HQ, HKV, HM, KA, VA, scale_attn, NATSL_BF16, k_batch_stride,
                       v_batch_stride);
  if (rc != NATSL_OK) return rc;
  RecurrentParams r;
  rc = recurrent_params(r, is_delta != 0, what, q, k, v, g, g_cumsum, beta, h0, h_block_start, o, ht, types, types_dtype, n_tokens_in_block,
                        n_tokens_in_block_scalar, B, T, H, HN, K, V, block, scale, flags, NATSL_BF16);
  if (rc != NATSL_OK) return rc;
  a.nsplit = attend_splits(B * T * HQ, TK);
  if (a.nsplit > 1 && (!workspace || workspace_bytes < natsl_decode_workspace_bytes(B, T, TK, HQ, VA)))
    return fail(NATSL_ERR_WORKSPACE, "%s: workspace of %zu bytes needed, %zu given", what, natsl_decode_workspace_bytes(B, T, TK, HQ, VA), workspace_bytes);
  a.partials = a.nsplit > 1 ? reinterpret_cast<float*>(workspace) : nullptr;
  if (T > 65535 || HQ > 65535 || B > 65535) return fail(NATSL_ERR_UNSUPPORTED, "%s: grid dimension above 65535", what);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  rc = launch_attend_and_recur(what, a, r, is_delta != 0, K, KA, VA, s);
  return rc != NATSL_OK ? rc : join_if_split(what, a, VA, s);
}
