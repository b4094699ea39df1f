// The mixed operator's forward as one native call: dtype conversions, routing, the softmax branch and the linear branch, on one
// stream or with the softmax branch on a second one.  At small sizes the operator's cost is launches and the host that issues
// them (fp32 B1 T256 H2: 60 us of kernels behind 200 us of host time as separate calls with torch conversions), so all tensor
// conversions of a side go out as one launch and nothing returns to the interpreter in between.
#include <cstring>
#include <mutex>

#include "natsl_host.h"
#include "natsl_linear_prep.h"

namespace natsl {

// ---- fp32 <-> bf16 copies of several tensors in one launch: 2048 elements per workgroup, 8 per thread -----------------------
struct CastSet {
  natsl_cast seg[NATSL_MIXED_CASTS];
  unsigned first[NATSL_MIXED_CASTS + 1];   // the segments' first workgroups
  int n;
};

template <bool TO_BF16>
__global__ __launch_bounds__(256) void cast_kernel(const CastSet p) {
  int s = 0;
#pragma unroll
  for (int i = 1; i < NATSL_MIXED_CASTS; ++i) s = i < p.n && blockIdx.x >= p.first[i] ? i : s;
  const natsl_cast c = p.seg[s];
  const long long at = (long long)(blockIdx.x - p.first[s]) * 2048 + 8 * threadIdx.x;
  if (at >= c.n) return;
  if (at + 8 <= c.n) {
    if constexpr (TO_BF16) {
      const float* src = reinterpret_cast<const float*>(c.src) + at;
      const f32x4 a = *reinterpret_cast<const f32x4*>(src), b = *reinterpret_cast<const f32x4*>(src + 4);
      *reinterpret_cast<bf16x8*>(reinterpret_cast<bf16_t*>(c.dst) + at) = pack8(a, b);
    } else {
      const u32x4 w = *reinterpret_cast<const u32x4*>(reinterpret_cast<const bf16_t*>(c.src) + at);
      float* dst = reinterpret_cast<float*>(c.dst) + at;
      *reinterpret_cast<f32x4*>(dst) = (f32x4){__uint_as_float(w[0] << 16), __uint_as_float(w[0] & 0xffff0000u), __uint_as_float(w[1] << 16), __uint_as_float(w[1] & 0xffff0000u)};
      *reinterpret_cast<f32x4*>(dst + 4) = (f32x4){__uint_as_float(w[2] << 16), __uint_as_float(w[2] & 0xffff0000u), __uint_as_float(w[3] << 16), __uint_as_float(w[3] & 0xffff0000u)};
    }
  } else {
    for (long long i = at; i < c.n; ++i) {
      if constexpr (TO_BF16) reinterpret_cast<bf16_t*>(c.dst)[i] = f32_to_bf16(reinterpret_cast<const float*>(c.src)[i]);
      else reinterpret_cast<float*>(c.dst)[i] = bf16_to_f32(reinterpret_cast<const bf16_t*>(c.src)[i]);
    }
  }
}

template <bool TO_BF16>
static int cast_all(const natsl_cast* seg, int n, hipStream_t s, const char* what) {
  if (n <= 0) return NATSL_OK;
  CastSet p;
  p.n = n;
  long long wgs = 0;
  for (int i = 0; i < NATSL_MIXED_CASTS; ++i) {
    if (i < n) {
      if (!seg[i].src || !seg[i].dst || seg[i].n <= 0) return fail(NATSL_ERR_INVALID, "%s: bad conversion segment", what);
      if (((uintptr_t)seg[i].src | (uintptr_t)seg[i].dst) & 15) return fail(NATSL_ERR_INVALID, "%s: converted tensors must start on 16 bytes", what);
      p.seg[i] = seg[i];
    }
    p.first[i] = (unsigned)wgs;
    if (i < n) wgs += (seg[i].n + 2047) / 2048;
  }
  p.first[NATSL_MIXED_CASTS] = (unsigned)wgs;
  if (wgs > 0x7fffffffll) return fail(NATSL_ERR_UNSUPPORTED, "%s: too much to convert", what);
  hipLaunchKernelGGL((cast_kernel<TO_BF16>), dim3((unsigned)wgs), dim3(256), 0, s, p);
  return check_launch(what);
}

// Rows of the table of packed sequences travel as arguments of the launch that stores them: a copy from host memory makes the host wait
// (40 us in front of an operator, 5 for the launch).  64 rows are 2 KiB of arguments.
struct SeqTableArgs {
  int4 part[NATSL_SEQ_TABLE_ROWS * 2];   // (a row is 32 bytes)
};
__global__ __launch_bounds__(NATSL_SEQ_TABLE_ROWS * 2) void seq_table_kernel(const SeqTableArgs a, int4* table, const int parts) {
  const int i = threadIdx.x;
  if (i < parts) table[i] = a.part[i];
}

// The streams' device is the current one while a call runs: events, kernel attributes and null handles go by the current device, and
// the caller's may be another.
class OnDeviceOf {
  int before = -1;

 public:
  int enter(const hipStream_t a, const hipStream_t b, const char* what) {
    int now = 0, dev = 0, other = 0;
    hipError_t e = hipGetDevice(&now);
    dev = now;
    if (e == hipSuccess && (a || b)) e = hipStreamGetDevice(a ? a : b, &dev);
    other = dev;
    if (e == hipSuccess && a && b) e = hipStreamGetDevice(b, &other);
    if (e == hipSuccess && other != dev) return fail(NATSL_ERR_INVALID, "%s: streams of devices %d and %d", what, dev, other);
    if (e == hipSuccess && dev != now && (e = hipSetDevice(dev)) == hipSuccess) before = now;
    return e == hipSuccess ? NATSL_OK : fail(NATSL_ERR_LAUNCH, "%s: cannot enter the streams' device (%s)", what, hipGetErrorString(e));
  }
  ~OnDeviceOf() {
    if (before >= 0) (void)hipSetDevice(before);
  }
};

// `to` waits for what `from` holds so far (both of the current device).  One event per device; a wait takes the event's state at the
// call, so the pair is made under a lock and the event can serve the next pair at once.
static int order_streams(hipStream_t from, hipStream_t to, const char* what) {
  constexpr int MAX_DEVICES = 64;
  static hipEvent_t events[MAX_DEVICES];
  static std::mutex mu;
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= MAX_DEVICES) return fail(NATSL_ERR_LAUNCH, "%s: cannot name the current device (%s)", what, hipGetErrorString(e));
  std::lock_guard<std::mutex> lock(mu);
  if (!events[dev]) e = hipEventCreateWithFlags(&events[dev], hipEventDisableTiming);
  if (e == hipSuccess) e = hipEventRecord(events[dev], from);
  if (e == hipSuccess) e = hipStreamWaitEvent(to, events[dev], 0);
  return e == hipSuccess ? NATSL_OK : fail(NATSL_ERR_LAUNCH, "%s: cannot order the streams (%s)", what, hipGetErrorString(e));
}

}  // namespace natsl

using namespace natsl;

// What natsl_mixed_fwd enqueues, on the streams' device; forked: the side stream may hold work that nothing waits for yet.
static int mixed_phases(const natsl_mixed* m, const int phases, natsl_stream_t stream, natsl_stream_t attn_stream, bool& forked, const char* what) {
  hipStream_t s = reinterpret_cast<hipStream_t>(stream), side = reinterpret_cast<hipStream_t>(attn_stream);
  const bool fork = side != s;
  // (a table that nobody reads afterwards is not made where the softmax kernel does not need it)
  const bool no_tables = m->private_tables && softmax_reads_types(m->B, m->T_attn, m->HQ, m->HKV, m->TN_attn, m->block, m->seqs, SOFTMAX_OPERATOR);
  int rc = NATSL_OK;
  if ((phases & NATSL_MIXED_CONVERT) && (rc = cast_all<true>(m->cast_in, m->n_cast_in, s, what)) != NATSL_OK) return rc;
  if (phases & NATSL_MIXED_ROUTE) {
    if (fork && (rc = order_streams(s, side, what)) != NATSL_OK) return rc;
    forked = fork;
    rc = no_tables ? NATSL_OK : natsl_route(m->types_attn, m->types_dtype, m->B, m->TN_attn, m->HN, m->T_attn, m->block, m->block_indices, m->n_blocks, nullptr, nullptr,
                     nullptr, nullptr, m->seqs, m->n_seqs, 0, attn_stream);
    if (rc != NATSL_OK) return rc;
  }
  auto softmax = [&](const LinearParams* prep, unsigned prep_wgs) {
    // the work queues lie behind the linear branch's part of the workspace
    const long long chunks = m->seqs ? m->total_chunks : (long long)m->B * cdiv(m->T, 64);
    const size_t at = natsl_linear_workspace_bytes(chunks, m->H);
    unsigned* queue = nullptr;
    if (m->workspace && m->workspace_bytes >= at + SOFTMAX_QUEUE_BYTES) queue = reinterpret_cast<unsigned*>(reinterpret_cast<char*>(m->workspace) + at);
    return softmax_fwd(m->q_attn, m->k_attn, m->v_attn, m->o_attn, m->lse, m->types_attn, m->types_dtype, no_tables ? nullptr : m->block_indices,
                       no_tables ? nullptr : m->n_blocks, m->B, m->T_attn, m->HQ, m->HKV, m->HN, m->KA, m->VA, m->TN_attn, m->block, m->scale_attn, m->same_block_visible, NATSL_BF16,
                       m->seqs, m->n_seqs, m->total_qtiles, attn_stream, SOFTMAX_OPERATOR, queue, prep, prep_wgs);
  };
  // Side by side, the scan comes first and the softmax kernel right behind the prep kernel: its workgroups take a CU each for as long
  // as there are tiles, so it has to find the scan's in place and fill the CUs they leave (the other way round the scan waits
  // for it).
  const bool both = fork && (phases & NATSL_MIXED_SOFTMAX) && (phases & NATSL_MIXED_LINEAR);
  // One after the other: the softmax tiles and the prep in one launch where the tiles are the small ones.
  const bool joined = !fork && (phases & NATSL_MIXED_SOFTMAX) && (phases & NATSL_MIXED_LINEAR) && !(m->flags & NATSL_STATES_ONLY) && m->B > 0 && m->T > 0 && m->H > 0 &&
                      softmax_takes_prep(m->B, m->T_attn, m->HQ, m->HKV, m->KA, m->VA, m->block, m->seqs, m->is_delta != 0, m->K,
                                         linear_prep_wgs(m->is_delta != 0, (long long)m->B * cdiv(m->T, 64), m->H));
  if ((phases & NATSL_MIXED_SOFTMAX) && !both && !joined && (rc = softmax(nullptr, 0)) != NATSL_OK) return rc;
  if (phases & NATSL_MIXED_LINEAR) {
    const BesideScan beside{order_streams, side};
    const PrepWith with{[](void* call, const LinearParams* p, unsigned wgs) { return (*static_cast<decltype(softmax)*>(call))(p, wgs); }, &softmax};
    rc = linear_fwd(m->is_delta != 0, m->q, m->k, m->v, m->g, m->is_delta ? m->beta : nullptr, m->h0, m->o, m->ht, m->h_block_start, m->g_block_sum,
                    m->chunk_states, m->is_delta ? m->chunk_v_new : nullptr, m->types, m->types_dtype, m->B, m->T, m->H, m->HN, m->K, m->V, m->TN,
                    m->block, m->scale_linear, m->is_delta ? m->flags : m->flags & ~NATSL_QK_L2NORM, m->workspace, m->workspace_bytes, NATSL_BF16,
                    m->seqs, m->n_seqs, m->total_chunks, stream, both ? &beside : nullptr, joined ? &with : nullptr);
    if (rc != NATSL_OK) return rc;
  }
  if (both && (rc = softmax(nullptr, 0)) != NATSL_OK) return rc;
  if (phases & NATSL_MIXED_JOIN) {
    if (fork && (rc = order_streams(side, s, what)) != NATSL_OK) return rc;
    forked = false;
    rc = cast_all<false>(m->cast_out, m->n_cast_out, s, what);
  }
  return rc;
}

// The linear branch's chunk states for a backward, next to whose scan the caller puts the softmax branch's backward: the other stream goes
// on behind the prep kernel, for the reason given above.  Forward and backward of an operator against the dQ kernel free to start at
// once and the scan behind its workgroups: B4 T4096 H12 128/128 1034 -> 969 us, B1 T32768 H2 4586 -> 3964 (50 % attention); the Mamba
// operators, where the softmax branch is the longer one anyway, within 1 %.  Behind the whole scan instead, so that the reverse scan
// follows at once as well: 1799 -> 1581 at B1 T16384 H8, where the linear branch is the longer one, but 1158 -> 1247 at B1 T8192 H16 with
// 50 % attention and 1022 -> 1109 for Mamba B2 T8192 H16: which one it is the routing decides, on the GPU.
extern "C" int natsl_linear_chunk_states(int is_delta, const void* q, const void* k, const void* v, const float* g, const void* beta, const float* h0,
                                         float* ht, void* chunk_states, void* chunk_v_new, const void* types, int types_dtype, int B, int T, int H, int HN, int K,
                                         int V, int TN, int block, float scale, int flags, void* workspace, size_t workspace_bytes, int dtype,
                                         const natsl_seq_row* seqs, int n_seqs, int total_units, natsl_stream_t stream, natsl_stream_t beside) {
  const char* what = "natsl_linear_chunk_states";
  hipStream_t s = reinterpret_cast<hipStream_t>(stream), other = reinterpret_cast<hipStream_t>(beside);
  OnDeviceOf device;
  if (const int rc = device.enter(s, other, what)) return rc;
  const BesideScan side{order_streams, other};
  flags |= NATSL_STATES_ONLY;
  return linear_fwd(is_delta != 0, q, k, v, g, is_delta ? beta : nullptr, h0, nullptr, ht, nullptr, nullptr, chunk_states, is_delta ? chunk_v_new : nullptr,
                    types, types_dtype, B, T, H, HN, K, V, TN, block, scale, is_delta ? flags : flags & ~NATSL_QK_L2NORM, workspace, workspace_bytes,
                    dtype, seqs, n_seqs, total_units, stream, other ? &side : nullptr);
}

extern "C" int natsl_order_streams(natsl_stream_t from, natsl_stream_t to) {
  const char* what = "natsl_order_streams";
  hipStream_t a = reinterpret_cast<hipStream_t>(from), b = reinterpret_cast<hipStream_t>(to);
  OnDeviceOf device;
  if (const int rc = device.enter(a, b, what)) return rc;
  return order_streams(a, b, what);
}

extern "C" int natsl_seq_table(const natsl_seq_row* rows, int n, natsl_seq_row* table, natsl_stream_t stream) {
  const char* what = "natsl_seq_table";
  static_assert(sizeof(natsl_seq_row) == 32, "a row is two pieces of 16 bytes");
  if (!rows || !table) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (n <= 0) return fail(NATSL_ERR_INVALID, "%s: non-positive dimension", what);
  if (reinterpret_cast<uintptr_t>(table) & 15) return fail(NATSL_ERR_INVALID, "%s: the table must start on 16 bytes", what);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  OnDeviceOf device;
  int rc = device.enter(s, nullptr, what);
  for (int at = 0; rc == NATSL_OK && at < n; at += NATSL_SEQ_TABLE_ROWS) {
    const int here = n - at < NATSL_SEQ_TABLE_ROWS ? n - at : NATSL_SEQ_TABLE_ROWS;
    SeqTableArgs a = {};
    memcpy(a.part, rows + at, (size_t)here * sizeof(natsl_seq_row));
    hipLaunchKernelGGL(seq_table_kernel, dim3(1), dim3(NATSL_SEQ_TABLE_ROWS * 2), 0, s, a, reinterpret_cast<int4*>(table + at), 2 * here);
    rc = check_launch(what);
  }
  return rc;
}

extern "C" size_t natsl_mixed_workspace_bytes(int64_t total_chunks, int H) {
  return natsl_linear_workspace_bytes(total_chunks, H) + SOFTMAX_QUEUE_BYTES;
}

extern "C" int natsl_mixed_fwd(const natsl_mixed* m, int phases, natsl_stream_t stream, natsl_stream_t attn_stream) {
  const char* what = "natsl_mixed_fwd";
  if (!m) return fail(NATSL_ERR_INVALID, "%s: null pointer argument", what);
  if (m->n_cast_in < 0 || m->n_cast_in > NATSL_MIXED_CASTS || m->n_cast_out < 0 || m->n_cast_out > NATSL_MIXED_CASTS)
    return fail(NATSL_ERR_INVALID, "%s: conversion counts", what);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream), side = reinterpret_cast<hipStream_t>(attn_stream);
  OnDeviceOf device;
  int rc = device.enter(s, side, what);
  if (rc != NATSL_OK) return rc;
  bool forked = side != s && !(phases & NATSL_MIXED_ROUTE);      // (by an earlier call)
  rc = mixed_phases(m, phases, stream, attn_stream, forked, what);
  // after an error too the caller may free what the side stream works on, as soon as its own stream allows
  if (rc != NATSL_OK && forked) (void)order_streams(side, s, what);
  return rc;
}
