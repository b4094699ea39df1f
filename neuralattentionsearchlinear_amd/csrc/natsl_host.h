// Host-side helpers shared by the C-ABI entry points.
#pragma once
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdio.h>
#include <atomic>

#include "../../include/natsl.h"

namespace natsl {

char* error_buffer();  // thread-local, 512 bytes (defined in natsl_route.hip)

inline int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(error_buffer(), 512, fmt, ap);
  va_end(ap);
  return code;
}

inline int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(NATSL_ERR_LAUNCH, "%s: %s", what, hipGetErrorString(e));
  return NATSL_OK;
}

// The LDS reservation of a kernel is an attribute of the function per device: set when a device first runs it.
inline int reserve_lds(const void* kern, std::atomic<unsigned long long>& done, size_t lds, const char* what) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(NATSL_ERR_LAUNCH, "%s: cannot name the current device (%s)", what, hipGetErrorString(e));
  const unsigned long long bit = 1ull << (dev & 63);
  if (dev < 64 && (done.load(std::memory_order_acquire) & bit)) return NATSL_OK;
  e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return fail(NATSL_ERR_LAUNCH, "%s: cannot reserve %zu bytes of LDS: %s", what, lds, hipGetErrorString(e));
  if (dev < 64) done.fetch_or(bit, std::memory_order_release);
  return NATSL_OK;
}

// Work on another stream that runs next to the linear branch's scan: ready(stream, other, what) is called between what the whole chip
// does (the prep kernel) and the scan.
struct BesideScan {
  int (*ready)(hipStream_t, hipStream_t, const char*);
  hipStream_t other;
};
// The softmax branch in the launch of the prep kernel, or before it: softmax(call, p, wgs) enqueues it, together with the prep's `wgs` workgroups
// unless p is null.
struct LinearParams;
struct PrepWith {
  int (*softmax)(void* call, const LinearParams* p, unsigned wgs);
  void* call;
};
// The two chunked linear branches behind their C entries (natsl_linear.hip); beside: null, or what the scan shares the chip with; with: null, or
// what goes with the prep kernel.
int linear_fwd(bool delta, const void* q, const void* k, const void* v, const float* g, const void* beta, const float* h0, void* o, float* ht,
               float* hs, float* gs, void* chunk_states, void* chunk_v_new, const void* types, int types_dtype, int B, int T, int H, int HN, int K,
               int V, int TN, int block, float scale, int flags, void* workspace, size_t workspace_bytes, int dtype, const natsl_seq_row* seqs,
               int n_seqs, int total_units, natsl_stream_t stream, const BesideScan* beside, const PrepWith* with = nullptr);

// The softmax branch behind its C entries (natsl_softmax.hip); queue: SOFTMAX_QUEUE_BYTES of this call's own for the persistent kernel's
// work queues, or null (see launch_softmax_stream).
constexpr size_t SOFTMAX_QUEUE_BYTES = 64;
enum SoftmaxUse { SOFTMAX_PER_TILE, SOFTMAX_ENTRY, SOFTMAX_OPERATOR };   // who calls: which kernel runs depends on it (see softmax_variant)
int softmax_fwd(const void* q, const void* k, const void* v, void* o, float* lse, const void* types, int types_dtype,
                const int32_t* nats_block_indices, const int32_t* n_nats_blocks, int B, int T, int HQ, int HKV, int HN, int K, int V, int TN,
                int block, float scale, int same_block_visible, int dtype, const natsl_seq_row* seqs, int n_seqs, int total_units,
                natsl_stream_t stream, SoftmaxUse use, unsigned* queue, const LinearParams* prep = nullptr, unsigned prep_wgs = 0);

// Whether softmax_fwd can take the linear branch's prep into its launch (`prep`, `prep_wgs`: see PrepWith): see softmax_prep_kernel.
bool softmax_takes_prep(int B, int T, int HQ, int HKV, int KA, int VA, int block, const natsl_seq_row* seqs, bool delta, int K, long long prep_wgs);

// Whether the kernel that such a call takes finds a tile's blocks in the types as well as in a routing table, which may be null then: the kernels of
// one workgroup a tile, unpacked, up to 256 selector blocks.
bool softmax_reads_types(int B, int T, int HQ, int HKV, int TN, int block, const natsl_seq_row* seqs, SoftmaxUse use);

inline int cdiv(int a, int b) { return (a + b - 1) / b; }

}  // namespace natsl
