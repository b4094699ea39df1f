/*
 * natsl.h -- C ABI of the MI355X (gfx950) implementation of the NAtS-L token-level hybrid
 * attention forward path.
 *
 * Plain pointers and sizes only: every pointer is DEVICE memory owned by the caller unless a
 * comment says "host"; tensors are dense, token-major [B,T,H,D] as in the reference
 * (src/nats/ops/mixed_ops/mixed_attn_gdn.py:49-50 makes its inputs contiguous).  Nothing here
 * allocates or synchronises with the host; work is enqueued on `stream`.  Two pieces of device
 * memory belong to the library and are shared by all calls on one GPU: the ticket counters of
 * natsl_softmax_sparse_fwd's persistent kernel on whole tiles (64 slots used in rotation, each zeroed
 * on the caller's stream ahead of the launch that uses it) and the scratch of
 * natsl_attn_masked_fwd_static; their comments say what that means for overlapping calls.
 * Each function returns NATSL_OK or a negative natsl_status; natsl_last_error() gives the
 * message for the calling thread.
 *
 * Each entry point names the reference interface it replaces (paths relative to the
 * reference repository root).
 */
#ifndef NATSL_H
#define NATSL_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct ihipStream_t* natsl_stream_t; /* a hipStream_t */

enum natsl_dtype { NATSL_F32 = 0, NATSL_BF16 = 1 };

enum natsl_status {
  NATSL_OK = 0,
  NATSL_ERR_INVALID = -1,     /* inconsistent shapes / null pointers */
  NATSL_ERR_UNSUPPORTED = -2, /* a shape or dtype this build has no kernel for */
  NATSL_ERR_WORKSPACE = -3,   /* workspace too small */
  NATSL_ERR_LAUNCH = -4       /* the HIP runtime refused the launch */
};

/* flags for the linear-recurrent branches */
enum natsl_flags {
  NATSL_DECAY_NON_LINEAR = 1, /* decay_for_non_gdn_blocks / decay_for_non_mamba_blocks */
  NATSL_QK_L2NORM = 2,        /* lattn_use_qk_l2norm_in_kernel */
  NATSL_INTRA_CHUNK = 4,      /* the linear op also scores its own incomplete block ('all', 'gated_delta_net', 'mamba') */
  NATSL_QUERY_ONLY = 8,       /* recurrent entries: outputs from the decayed block-start state, nothing updated ('attn') */
  NATSL_FRESH_BLOCK_START = 16, /* recurrent entries: h_block_start is written only; the block starts from h0 (zeros if NULL) */
  NATSL_STATES_ONLY = 32      /* chunked entries: no outputs (o is NULL), for a backward that forms chunk_states and chunk_v_new again */
};

/* One row per packed sequence (cu_seqlens / cu_seqlens_nats of the reference, plus prefix
 * counts the kernels would otherwise have to scan for).  Pass seqs = NULL, n_seqs = 0 for a
 * regular [B,T,...] batch.  With a table, B must be 1, T is the packed length, TN the packed
 * number of selector blocks, and `total_units` is the sum over sequences of the entry point's
 * work unit (ceil(len/64) chunks for the linear branches and the router, ceil(len/256) query
 * tiles for the softmax branch); it is ignored for regular batches. */
typedef struct natsl_seq_row {
  int32_t bos;       /* first token of the sequence (flat token index) */
  int32_t eos;       /* one past its last token */
  int32_t bos_nats;  /* first selector block of the sequence (flat block index) */
  int32_t chunk_off; /* number of 64-token chunks in earlier sequences */
  int32_t qtile_off; /* number of 256-row softmax query tiles in earlier sequences */
  int32_t pad[3];
} natsl_seq_row;

/* Stores n rows of host memory into a table on the stream's device, in ceil(n / NATSL_SEQ_TABLE_ROWS) launches: the rows are read before the
 * call returns, and it does not wait for the device.  table starts on 16 bytes. */
#define NATSL_SEQ_TABLE_ROWS 64
int natsl_seq_table(const natsl_seq_row* rows, int n, natsl_seq_row* table, natsl_stream_t stream);

int natsl_version(void);
const char* natsl_last_error(void);

/* Block mean of hidden [B,T,D] -> pooled [B,ceil(T/block),D] (same dtype), divisor
 * min(block, T - c*block).
 * Replaces mean_pooling (src/nats/ops/utils/pooling.py:26-57,190-207) as called by the layer at
 * src/nats/layers/natsl_attn_gdn.py:412-417. */
int natsl_mean_pool(const void* hidden, void* pooled, int B, int T, int D, int block, int dtype,
                    const natsl_seq_row* seqs, int n_seqs, int total_units, natsl_stream_t stream);

/* Selector: logits [B,TN,HN,2] -> types [B,TN,HN,2] in the same dtype with values exactly {0,1}
 * (softmax evaluated in fp32, rounded to the logits dtype, first maximum wins), optionally
 * forcing the last block of every sequence to 1 for both ops, and n_nats_blocks [B,HN,2] int32.
 * Replaces hard_softmax (src/nats/layers/natsl_attn_gdn.py:47-61) and the two statements at
 * src/nats/layers/natsl_attn_gdn.py:553-554. n_nats_blocks may be NULL. */
int natsl_hard_select(const void* logits, void* types, int32_t* n_nats_blocks, int B, int TN, int HN,
                      int dtype, int force_last, const natsl_seq_row* seqs, int n_seqs,
                      int total_units, natsl_stream_t stream);

/* What a layer's forward takes from its logits [B,TN,HN,2], in one launch: natsl_hard_select's types with the last block of every
 * sequence forced, the types before that (raw_types, or NULL), n_nats_blocks [B,HN,2], and attn_fraction [HN] fp32, the attention
 * blocks' share of all blocks (src/nats/layers/natsl_attn_gdn.py:553-554). */
int natsl_layer_select(const void* logits, void* types, void* raw_types, int32_t* n_nats_blocks, float* attn_fraction, int B, int TN, int HN,
                       int dtype, natsl_stream_t stream);

/* Routing tables derived from types [B,TN,HN,2] (values rounded as the reference does at
 * src/nats/ops/mixed_ops/mixed_attn_gdn.py:88).  Any output may be NULL.
 *   nats_block_indices   int32 [B,TN,HN,2]   ascending ids of selected blocks, padded with TN
 *                                            (mixed_attn_gdn.py:93-97)
 *   n_nats_blocks        int32 [B,HN,2]      (mixed_attn_gdn.py:99-100)
 *   linear_chunk_offsets int64 [B*HN+1]      prepare_nats_chunk_offsets (src/nats/ops/nats_util.py:35-64)
 *   chunk_indices_linear int32 [cap,2]       prepare_nats_block_indices (nats_util.py:6-32); cap must be
 *                                            >= B*HN*TN*(block/64); rows beyond the total are untouched
 *   starting_h_idx       int64 [B,ceil(T/64),HN]   compute_starting_idx_for_chunks (nats_util.py:124-162)
 *   attn_n_iters         int64 [B,ceil(T/128),HN]  compute_attn_n_iters_per_block (nats_util.py:67-121)
 * The last two are defined for regular batches only (seqs == NULL). */
int natsl_route(const void* types, int types_dtype, int B, int TN, int HN, int T, int block,
                int32_t* nats_block_indices, int32_t* n_nats_blocks, int64_t* linear_chunk_offsets,
                int32_t* chunk_indices_linear, int64_t* starting_h_idx, int64_t* attn_n_iters,
                const natsl_seq_row* seqs, int n_seqs, int total_units, natsl_stream_t stream);

/* Softmax branch: causal attention in which a query sees its own block and every earlier block
 * typed "attention" (same_block_visible = 1), or only earlier attention blocks (= 0).
 * q [B,T,HQ,K], k [B,T,HKV,K], v [B,T,HKV,V] -> o [B,T,HQ,V] (same dtype), lse [B,T,HQ] fp32 in
 * log2 units; rows that see no key give o = 0, lse = 0.
 * Replaces parallel_attn_nats_fwd (src/nats/ops/attns/attns.py:1421-1531, kernel :62-353) as
 * called at src/nats/ops/mixed_ops/mixed_attn_gdn.py:111-117.
 * K, V in {64, 128}.  Problems with tiles enough for every compute unit (natsl_softmax_fwd_variant says which;
 * T <= 65536, block <= 2048, at most 64 packed sequences) run as a persistent kernel.  On batches with T a multiple of 256 its work
 * queues are ticket counters in device memory owned by the library: 64 slots used in rotation, the launch's slot zeroed by a small
 * fill kernel enqueued on `stream` right before it (both kernels can be captured into a HIP graph).  Such launches may overlap across
 * streams as long as fewer than 64 of them are in flight on one GPU; a captured one keeps the slot it drew at capture, so replay it
 * on the stream that also carries the eager launches.  Packed sequences and other lengths use no device memory but what the
 * arguments name, and may overlap and be replayed in any way. */
int natsl_softmax_sparse_fwd(const void* q, const void* k, const void* v, void* o, float* lse,
                             const void* types, int types_dtype, const int32_t* nats_block_indices,
                             const int32_t* n_nats_blocks, int B, int T, int HQ, int HKV, int HN, int K,
                             int V, int TN, int block, float scale, int same_block_visible, int dtype,
                             const natsl_seq_row* seqs, int n_seqs, int total_units, natsl_stream_t stream);

/* The same operation, always as one workgroup per query tile (what natsl_softmax_sparse_fwd itself runs for small
 * problems, short sequences and more than 64 packed sequences): for callers that want no library-owned device state in the launch, and the regression
 * check of the persistent kernel.  The same results bit for bit, except for the queries of a sequence's last 256-row
 * tile where its length is no multiple of 64: there the two take other reference maxima, so the probabilities round differently.
 * Same reference interface as natsl_softmax_sparse_fwd. */
int natsl_softmax_sparse_fwd_per_tile(const void* q, const void* k, const void* v, void* o, float* lse,
                             const void* types, int types_dtype, const int32_t* nats_block_indices,
                             const int32_t* n_nats_blocks, int B, int T, int HQ, int HKV, int HN, int K,
                             int V, int TN, int block, float scale, int same_block_visible, int dtype,
                             const natsl_seq_row* seqs, int n_seqs, int total_units, natsl_stream_t stream);

/* Which kernel natsl_softmax_sparse_fwd runs for a problem on the current device (host-side query, no launch; packed: the
 * number of packed sequences, 0 for a batch;
 * the choice that src/nats/ops/attns/attns.py:1497-1512 leaves to Triton's autotuner). */
enum natsl_softmax_variant { NATSL_SOFTMAX_TILE_128 = 0, NATSL_SOFTMAX_TILE_256 = 1, NATSL_SOFTMAX_PERSISTENT = 2 };
int natsl_softmax_fwd_variant(int B, int T, int HQ, int HKV, int block, int packed);


/* Backward of the softmax branch: dq [B,T,HQ,K], dk [B,T,HKV,K], dv [B,T,HKV,V] (bf16, summed over the query heads of
 * a kv head) and dnats fp32 [B,TN,HQ] (written whole): per block typed "attention" and query head, the sum
 * of the score gradients dS = P (dP - delta) over (keys of the block) x (queries of later blocks), i.e. the gradient
 * with respect to a bias on that block's scores as later blocks see them; blocks not typed attention keep 0 unless
 * flags bit 1 is set (the reference's compute_dnats_for_invalid_blocks_attn, attns.py:1318-1325): then they get
 * sum min(exp2(s - lse), 1) (dP - delta) over the same (keys) x (later queries), what their keys would contribute if
 * they were visible.  flags bit 0: same_block_visible, as in the forward.  The caller sums dnats over the query heads
 * of a selector head.  o, lse are the forward's outputs, d_o the gradient of o.  workspace: natsl_softmax_bwd_workspace_bytes()
 * bytes (delta = rowsum(d_o * o), then the work-queue counters of the dk/dv kernel; nothing to initialise: every call resets
 * them, so calls that share a workspace must not overlap).  T * HQ * max(K, V) * 2 must stay below 2^32 (32-bit row offsets
 * within the input).  Packed sequences: B = 1 and `seqs` as in the forward, with total_qtiles the table's count of
 * 256-query tiles and total_chunks its count of 64-token chunks (n_nats_blocks is [n_seqs,HN,2]); else null, 0, 0, 0.
 * Replaces parallel_attn_nats_bwd (src/nats/ops/attns/attns.py:1562-1759; kernels :357-372, :383-708, :719-983) as
 * called at src/nats/ops/mixed_ops/mixed_attn_gdn.py:226-243. */
size_t natsl_softmax_bwd_workspace_bytes(int B, int T, int HQ);
int natsl_softmax_sparse_bwd(const void* q, const void* k, const void* v, const void* o, const float* lse, const void* d_o,
                             void* dq, void* dk, void* dv, float* dnats, const void* types, int types_dtype,
                             const int32_t* nats_block_indices, const int32_t* n_nats_blocks, int B, int T, int HQ, int HKV,
                             int HN, int K, int V, int TN, int block, float scale, int flags, int dtype,
                             void* workspace, size_t workspace_bytes, const natsl_seq_row* seqs, int n_seqs,
                             int total_qtiles, int total_chunks, natsl_stream_t stream);

/* Bytes of scratch the two linear-branch entry points need for `total_chunks` 64-token chunks
 * (sum over sequences of ceil(len/64)) and H heads. */
size_t natsl_linear_workspace_bytes(int64_t total_chunks, int H);

/* Gated DeltaNet branch, chunked forward.
 * q,k [B,T,H,K], v [B,T,H,V], beta [B,T,H] in `dtype`; g [B,T,H] fp32 log-decay; h0 / ht
 * [N,H,K,V] fp32 (either may be NULL) -> o [B,T,H,V] in `dtype`.
 * Optional prefill hand-off outputs: h_block_start [N,H,K,V] fp32 = the state that entered each
 * sequence's last selector block, g_block_sum [N,H] fp32 = the sum of g over that block (the two
 * quantities chunk_gated_delta_rule_nats_inference_fwd derives at
 * src/nats/ops/gated_delta_rule/chunk_fwd.py:178-206); pass NULL for both in training.
 * chunk_states (optional, for a backward): the state ENTERING every 64-token chunk, transposed and rounded as the kernel
 * uses it, bf16 [total_chunks][H][V][K] (total_chunks as for natsl_linear_workspace_bytes; the reference keeps the same
 * per-chunk states as `h`, src/nats/ops/common/chunk_delta_h.py:681-683); NULL = not stored.
 * chunk_v_new (optional, for a backward): the delta rule's corrected values v_new of every token, bf16 [B*T][H][V] (the
 * reference's `v_new`, chunk_delta_h.py:684); NULL = not stored.  With NATSL_STATES_ONLY o is NULL and chunk_states is not: q is read
 * for the workspace only (the delta rule's P and norms).
 * The workspace is scratch between the entry's two kernels and its contents are the entry's own business, except after a call
 * with chunk_states: then it holds what natsl_linear_chunk_bwd reads (per chunk and head TmB, P and four scale vectors).  A
 * call without chunk_states may leave P out (a launch that fills the GPU forms it inside its second kernel).
 * Replaces l2norm_fwd + chunk_gated_delta_rule_nats_fwd
 * (src/nats/ops/mixed_ops/mixed_attn_gdn.py:119-164, src/nats/ops/gated_delta_rule/chunk.py:22-167). */
int natsl_gdn_chunk_fwd(const void* q, const void* k, const void* v, const float* g, const void* beta,
                        const float* h0, void* o, float* ht, float* h_block_start, float* g_block_sum,
                        void* chunk_states, void* chunk_v_new, const void* types, int types_dtype, int B,
                        int T, int H, int HN, int K, int V, int TN, int block, float scale, int flags,
                        void* workspace, size_t workspace_bytes, int dtype, const natsl_seq_row* seqs,
                        int n_seqs, int total_units, natsl_stream_t stream);

/* Mamba2-style SSD branch, chunked forward (q = C, k = B, v = X*dt, g = A*dt).
 * h_block_start / g_block_sum / chunk_states as for the Gated DeltaNet entry (src/nats/ops/mamba/chunk_fwd.py:22-157).
 * Replaces chunk_mamba2_fwd (src/nats/ops/mamba/chunk.py:21-109) as called at
 * src/nats/ops/mixed_ops/mixed_attn_mamba.py:140-161. */
int natsl_mamba_chunk_fwd(const void* q, const void* k, const void* v, const float* g, const float* h0,
                          void* o, float* ht, float* h_block_start, float* g_block_sum, void* chunk_states, const void* types,
                          int types_dtype, int B, int T, int H,
                          int HN, int K, int V, int TN, int block, float scale, int flags, void* workspace,
                          size_t workspace_bytes, int dtype, const natsl_seq_row* seqs, int n_seqs,
                          int total_units, natsl_stream_t stream);

/* Backward of the two chunked linear branches (delta_rule != 0: Gated DeltaNet, else Mamba2-style SSD); packed input as for the
 * forward (B = 1, the sequence table, TN = all blocks; dht, dh0 then hold one state per sequence).  Call the forward entry first with chunk_states and (delta rule) chunk_v_new and
 * keep its workspace (both forms: the reverse scan reads the scale vectors from it and, for the delta rule, the triangular solves
 * and the intra-chunk matrices).  Inputs as for the forward, plus
 *   v_new [B*T][H][V] (Mamba: v itself), d_o [B*T][H][V] bf16, dht [B][H][K][V] f32 or NULL,
 *   g_block_sums [B][TN][H] f32 = sum of g over every selector block (packed: flat over the sequences' blocks); NULL where these are the
 *   chunks' (block 64, not packed): then the workspace's.
 * Outputs: dq, dk [B*T][H][K], dv [B*T][H][V] bf16; dg, dbeta (delta rule) [B*T][H] f32; dh0 [B][H][K][V] f32 or NULL;
 *   d_gate [chunks][H] f32 = derivative with respect to a gate on every chunk's state update (the selector's
 *   straight-through gradient for the linear operator, src/nats/ops/common/chunk_o.py:438-443, :487-492, before the sum over
 *   a block's chunks and a selector head's heads);
 *   d_rollback [chunks][H] f32 = what the decay of a rolled-back block adds to dg of each of its tokens (non-zero behind
 *   the last chunk of blocks that are not typed linear, NATSL_DECAY_NON_LINEAR only);
 *   d_chunk_states: scratch, bf16 [chunks][H][V][K] (the gradient of the state behind every chunk);
 *   dbeta_parts: scratch, f32 [B*T][H][V/16] (delta rule only).
 * K in {64, 128, 192}, V a multiple of 64.
 * Replaces chunk_gated_delta_rule_nats_bwd (src/nats/ops/gated_delta_rule/chunk.py:170-332) and the Mamba counterpart
 * (src/nats/ops/mamba/chunk.py:112-260). */
int natsl_linear_chunk_bwd(int delta_rule, const void* q, const void* k, const void* v_new, const float* g, const void* beta,
                           const void* d_o, const float* dht, const void* chunk_states, const void* types, int types_dtype,
                           const float* g_block_sums, const void* workspace, void* d_chunk_states, float* dbeta_parts,
                           void* dq, void* dk, void* dv, float* dg, float* dbeta, float* dh0, float* d_gate, float* d_rollback, int B, int T,
                           int H, int HN, int K, int V, int TN, int block, float scale, int flags, int dtype,
                           const natsl_seq_row* seqs, int n_seqs, int total_chunks, natsl_stream_t stream);

/* natsl_linear_chunk_bwd in its two steps, so that something can run next to the scan or be ready before the second step: steps 1 = the
 * reverse scan (dv, d_chunk_states, dbeta_parts, dh0), 2 = the per-chunk gradients (dq, dk, dg, dbeta, d_gate, d_rollback), 3 = both; + 4: another
 * kernel shares the chip with the scan (wider workgroups on fewer CUs); + 8: dbeta is bf16.
 * add (second step): 1, 2 = dq, dk are added to what is there; dv_sum, when given, [B*T][H][V]: dv is added to what is there.  (A tensor
 * that another operator takes as well has one gradient; the sum is rounded as an elementwise bf16 addition would.) */
int natsl_linear_chunk_bwd_steps(int steps, int add, void* dv_sum, int delta_rule, const void* q, const void* k, const void* v_new, const float* g,
                                 const void* beta, const void* d_o, const float* dht, const void* chunk_states, const void* types,
                                 int types_dtype, const float* g_block_sums, const void* workspace, void* d_chunk_states, float* dbeta_parts,
                                 void* dq, void* dk, void* dv, float* dg, void* dbeta, float* dh0, float* d_gate, float* d_rollback, int B, int T,
                                 int H, int HN, int K, int V, int TN, int block, float scale, int flags, int dtype,
                                 const natsl_seq_row* seqs, int n_seqs, int total_chunks, natsl_stream_t stream);

/* What is per selector block around natsl_linear_chunk_bwd.  natsl_linear_block_sums fills its g_block_sums from the forward's
 * workspace.  natsl_block_grads, after it: d_types [B,TN,HN,2] (f32 or bf16) = the selector's straight-through gradients --
 * [..., 1] d_gate summed over a block's chunks and a selector head's heads where the block is typed linear (others: 0, or with
 * `invalid` their last chunk's), [..., 0] dnats [B,TN,HQ] f32 of natsl_softmax_sparse_bwd summed over the query heads (NULL: 0) --
 * and, where d_rollback is given, dg [B*T][H] += the rolled-back decay's share. */
int natsl_linear_block_sums(const void* workspace, float* g_block_sums, int B, int T, int H, int TN, int block, const natsl_seq_row* seqs, int n_seqs,
                            int total_chunks, natsl_stream_t stream);
int natsl_block_grads(const void* types, int types_dtype, const float* d_gate, const float* d_rollback, const float* dnats, int HQ, float* dg,
                      void* d_types, int d_types_dtype, int invalid, int B, int T, int H, int HN, int TN, int block, const natsl_seq_row* seqs,
                      int n_seqs, natsl_stream_t stream);
/* natsl_block_grads and natsl_hard_select_bwd (last_forced) of its d_types in one launch: dlogits [B,TN,HN,2]; logits, types and dlogits in `dtype`. */
int natsl_block_grads_logits(const void* types, const void* logits, int dtype, const float* d_gate, const float* d_rollback, const float* dnats, int HQ,
                             float* dg, void* dlogits, int invalid, int B, int T, int H, int HN, int TN, int block, natsl_stream_t stream);

/* Layer tail: y = (rms(x1)*w1*xw[...,0] + rms(x2)*w2*xw[...,1]) * gate*sigmoid(gate) with
 * rms(x) = x*rsqrt(mean(x^2)+eps); x1, x2, gate, y [rows, D] and x_weights [rows, 2] in `dtype`,
 * w1, w2 [D] in `w_dtype`.  D in {32, 64, 96, 128, 192, 256, 384, 512}.
 * Replaces the forward of FusedMultiInputRMSNormGated (src/nats/modules/fused_norm_gate.py:38-182)
 * as called at src/nats/layers/natsl_attn_gdn.py:652-661. */
int natsl_norm_gate_fwd(const void* x1, const void* x2, const void* gate, const void* x_weights, const void* w1,
                        const void* w2, void* y, int64_t rows, int D, int dtype, float eps, int w_dtype,
                        natsl_stream_t stream);

/* Backward of natsl_norm_gate_fwd: dx1, dx2, dgate [rows, D] in `dtype`; dx_weights [rows, 2] f32; dw1, dw2 [D] f32, the two
 * rows of ONE [2][D] tensor (dw2 == dw1 + D).  The weight gradients are summed over the rows in a fixed order (partial sums
 * per 128 rows in the workspace, then one reduction): the same bits on every run.
 * Replaces the backward of FusedMultiInputRMSNormGated (src/nats/modules/fused_norm_gate.py:185-420). */
size_t natsl_norm_gate_bwd_workspace_bytes(int64_t rows, int D);
int natsl_norm_gate_bwd(const void* x1, const void* x2, const void* gate, const void* x_weights, const void* w1,
                        const void* w2, const void* dy, void* dx1, void* dx2, void* dgate, float* dx_weights, float* dw1,
                        float* dw2, void* workspace, size_t workspace_bytes, int64_t rows, int D, int dtype, float eps,
                        int w_dtype, natsl_stream_t stream);

/* The same with the two mixing weights of a row given as logits (bf16): x_weights = softmax(x_logits) rounded to bf16, and the
 * gradient comes back for the logits (bf16) -- the mixing layer's softmax (src/nats/layers/natsl_attn_gdn.py:492-494) without a pass
 * of its own. */
int natsl_norm_gate_logits_fwd(const void* x1, const void* x2, const void* gate, const void* x_logits, const void* w1, const void* w2, void* y,
                               int64_t rows, int D, int dtype, float eps, int w_dtype, natsl_stream_t stream);
int natsl_norm_gate_logits_bwd(const void* x1, const void* x2, const void* gate, const void* x_logits, const void* w1, const void* w2,
                               const void* dy, void* dx1, void* dx2, void* dgate, void* dx_logits, float* dw1, float* dw2, void* workspace,
                               size_t workspace_bytes, int64_t rows, int D, int dtype, float eps, int w_dtype, natsl_stream_t stream);

/* Layer glue, depthwise causal short convolution with its activation, on the layer's token-major tensors:
 * y[b,t,d] = act(bias[d] + sum_j w[d,j] e[b, t-(W-1)+j, d]) where e is x preceded by the W-1 inputs before it: the last
 * W-1 entries of `state` [B,D,W] (the cache of a previous call, in `state_dtype`), or zeros when state is NULL.
 * x, y [B,T,D] in `dtype` (f32 or bf16; sums in f32, one rounding); weight [D,W] (the [D,1,W] of a Conv1d), bias [D] or NULL
 * in `w_dtype`; activation 0 = none, 1 = silu; W in {2, 3, 4}; D % 8 == 0.  state_out [B,D,W] in `dtype`, or NULL: the
 * last W inputs of (state ++ x), what the next call takes as `state`; it must not alias `state`.
 * Replaces the forward of flash-linear-attention's ShortConvolution as called at
 * src/nats/layers/natsl_attn_gdn.py:425-491 and src/nats/layers/natsl_attn_mamba2.py:368-425. */
int natsl_short_conv_fwd(const void* x, const void* weight, const void* bias, const void* state, void* y, void* state_out,
                         int B, int T, int D, int W, int activation, int dtype, int w_dtype, int state_dtype,
                         natsl_stream_t stream);

/* Backward of natsl_short_conv_fwd: dx [B,T,D] in `dtype` (gradient of x; the cached state gets none), dweight fp32 [D,W],
 * dbias fp32 [D] or NULL, from x, weight, bias, state as given to the forward and dy [B,T,D] in `dtype`.  The pre-activation
 * is recomputed; the weight sums are reduced in a fixed order through the workspace
 * (natsl_short_conv_bwd_workspace_bytes(), fp32 partial sums per run of tokens): no atomics, repeatable bits.
 * Replaces the backward of flash-linear-attention's ShortConvolution under the same call sites. */
size_t natsl_short_conv_bwd_workspace_bytes(int B, int T, int D, int W);
int natsl_short_conv_bwd(const void* x, const void* weight, const void* bias, const void* state, const void* dy, void* dx,
                         float* dweight, float* dbias, void* workspace, size_t workspace_bytes, int B, int T, int D, int W,
                         int activation, int dtype, int w_dtype, int state_dtype, natsl_stream_t stream);

/* Layer glue, row normalisation: y = x * rsqrt(mean(x^2) + eps) * weight (l2 = 0, RMSNorm; weight [D] in `w_dtype` or NULL
 * for none) or y = x * rsqrt(sum(x^2) + eps) (l2 = 1).  x, y [rows, D] in `dtype` (f32 or bf16), arithmetic in f32.
 * D in {32, 64, 96, 128, 192, 256, 384, 512}.
 * Replaces the RMSNorm of the attention view's q and k (flash-linear-attention's, called at
 * src/nats/layers/natsl_attn_gdn.py:504-505) and the L2 normalisation of the Mamba layer's B and C
 * (src/nats/layers/natsl_attn_mamba2.py:469-470). */
int natsl_row_norm_fwd(const void* x, const void* weight, void* y, int64_t rows, int D, float eps, int l2, int dtype,
                       int w_dtype, natsl_stream_t stream);

/* Backward of natsl_row_norm_fwd: dx [rows, D] in `dtype`; dweight [D] f32 when a weight is given (summed over the rows in a
 * fixed order: partial sums per 128 rows in the workspace, then one reduction; no weight: workspace may be NULL).
 * Replaces the backward of the reference's RMSNorm / l2norm modules (fla.modules, as used at
 * src/nats/layers/natsl_attn_gdn.py:275-330). */
size_t natsl_row_norm_bwd_workspace_bytes(int64_t rows, int D);
int natsl_row_norm_bwd(const void* x, const void* weight, const void* dy, void* dx, float* dweight, void* workspace,
                       size_t workspace_bytes, int64_t rows, int D, float eps, int l2, int dtype, int w_dtype,
                       natsl_stream_t stream);

/* Decode: T tokens that continue the current (incomplete) selector block of N cached sequences, token by
 * token.  Per token: S *= e^g; d = beta (v - S^T k); S += k d^T; o = scale S^T q (k, q L2-normalised with
 * NATSL_QK_L2NORM).  Only the first min(T, block - n_tokens_in_block) tokens are processed.  If they
 * complete the block (n_tokens_in_block + T >= block) and the block is not typed linear, S is restored to
 * h_block_start (times e^(g_cumsum + sum of g) with NATSL_DECAY_NON_LINEAR), and in either case
 * h_block_start <- S.  q,k [N,T,H,K], v,o [N,T,H,V], beta [N,T,H] in `dtype`; g fp32 [N,T,H];
 * g_cumsum fp32 [N,H] or NULL (0): sum of g over the tokens already in the block; h0 fp32 [N,H,K,V] or NULL
 * (zeros); h_block_start fp32 [N,H,K,V] in/out; ht fp32 [N,H,K,V] or NULL; types [N,1,HN,2] (op 1 = linear);
 * n_tokens_in_block int32 [N] or NULL (then the scalar is used for every sequence).  K in {64, 128, 192}, V % 16 == 0.
 * With NATSL_QUERY_ONLY (the mode in which the linear operator skips the incomplete block, ops_for_incomplete_chunks = 'attn'):
 * o_t = scale q_t^T (e^(g_cumsum + g_1 + .. + g_t) h_block_start), no state is read from h0 or written; k, v, beta may be NULL
 * (the reference's branch without UPDATE_HS_FOR_EACH_ITER, fused_recurrent.py:156-201, as called for one-token steps at
 * src/nats/ops/mixed_ops/mixed_attn_gdn.py:510-527).
 * Replaces fused_recurrent_gated_delta_rule_nats_fwd, src/nats/ops/gated_delta_rule/fused_recurrent.py:360-470
 * (kernel :28-358) as called with update_hs_for_each_iter=True at
 * src/nats/ops/mixed_ops/mixed_attn_gdn.py:485-503. */
int natsl_gdn_recurrent_fwd(const void* q, const void* k, const void* v, const float* g, const float* g_cumsum,
                            const void* beta, const float* h0, float* h_block_start, void* o, float* ht,
                            const void* types, int types_dtype, const int32_t* n_tokens_in_block,
                            int n_tokens_in_block_scalar, int N, int T, int H, int HN, int K, int V, int block,
                            float scale, int flags, int dtype, natsl_stream_t stream);

/* The same for the Mamba2 (SSD) branch: S *= e^g; S += k v^T; o = scale S^T q (q = C, k = B, v = x*dt); no beta,
 * no normalisation (NATSL_QK_L2NORM is ignored).
 * Replaces fused_recurrent_mamba_nats_fwd (src/nats/ops/mamba/fused_recurrent.py, kernel :150-300) as called
 * at src/nats/ops/mixed_ops/mixed_attn_mamba.py:498-514. */
int natsl_mamba_recurrent_fwd(const void* q, const void* k, const void* v, const float* g, const float* g_cumsum,
                              const float* h0, float* h_block_start, void* o, float* ht, const void* types,
                              int types_dtype, const int32_t* n_tokens_in_block, int n_tokens_in_block_scalar, int N,
                              int T, int H, int HN, int K, int V, int block, float scale, int flags, int dtype,
                              natsl_stream_t stream);

/* Decode: softmax attention of TQ queries over TK cached keys under an explicit visibility mask.
 * q [B,TQ,HQ,K], k [B,TK,HKV,K], v [B,TK,HKV,V], o [B,TQ,HQ,V] in `dtype`; mask uint8 [B,HM,TQ,TK], non-zero =
 * visible, HM divides HQ; query head hq uses kv head hq/(HQ/HKV) and mask head hq/(HQ/HM).  A query that sees
 * no key gives 0.  With a workspace of natsl_attn_masked_workspace_bytes() the keys of one query are split over
 * several workgroups (needed to fill the GPU when B*TQ*HQ is small); with workspace = NULL one workgroup
 * handles a query.  k_batch_stride / v_batch_stride: elements from one sequence's keys / values to the next, for keys that
 * are the front part of a larger cache buffer [B,capacity,HKV,D] (a multiple of 8, at least TK*HKV*D); 0 = dense.
 * Replaces repeat_masks + torch.nn.functional.scaled_dot_product_attention at
 * src/nats/ops/mixed_ops/mixed_attn_gdn.py:475-481. */
size_t natsl_attn_masked_workspace_bytes(int B, int TQ, int TK, int HQ, int V);
int natsl_attn_masked_fwd(const void* q, const void* k, const void* v, const uint8_t* mask, void* o, int B, int TQ,
                          int TK, int HQ, int HKV, int HM, int K, int V, float scale, int dtype, void* workspace,
                          size_t workspace_bytes, int64_t k_batch_stride, int64_t v_batch_stride, natsl_stream_t stream);

/* natsl_attn_masked_fwd for callers that cannot allocate (code under HIP graph capture, tight serving loops, harnesses
 * that forbid hipMalloc): the same kernels with the split scratch in a device array of the library itself, so the caller
 * passes inputs and outputs only and the call allocates nothing.  It has no counterpart in the reference.  The array
 * holds natsl_attn_masked_static_scratch_bytes() = 256 KiB per GPU for the life of the process; a shape whose splits need
 * more (natsl_attn_masked_workspace_bytes() above that limit) is refused with NATSL_ERR_WORKSPACE.  Results are
 * identical to natsl_attn_masked_fwd with a workspace.  All calls on one GPU share the array: calls that overlap on
 * one GPU (different streams or threads) race. */
size_t natsl_attn_masked_static_scratch_bytes(void);
int natsl_attn_masked_fwd_static(const void* q, const void* k, const void* v, const uint8_t* mask, void* o, int B, int TQ,
                                 int TK, int HQ, int HKV, int HM, int K, int V, float scale, int dtype,
                                 natsl_stream_t stream);

/* KV cache of the softmax branch: keep the attention-typed blocks of a region of new tokens, per (sequence, kv
 * head), back to back behind the blocks already kept, and put the tokens of the incomplete last block at block
 * index tail_dst (the same for every head; pass -1 when the region ends on a block boundary).
 * src_k/src_v [B, src_tokens, HKV, K|V] hold the region from block src_block0 on: NB blocks of `block` tokens,
 * the first n_complete complete (n_complete = NB, or NB-1 with an incomplete block of tail_tokens tokens).
 * dst_k/dst_v [B, dst_tokens, HKV, K|V] is the cache; it may be the source itself (in place: same pointers and
 * sizes), since a kept block never moves towards the back.  types [B, NB, HN, 2] (f32 or bf16): column 0 equal to
 * 1 marks an attention-typed block; kv head h follows selector head h/(HKV/HN).  n_before int64 [B, HN] = blocks
 * already kept per (sequence, selector head), NULL = none.  The caller sizes the destination for the largest new
 * count (stores past dst_tokens are dropped, never issued).  The rest of the block at tail_dst is zero filled when
 * the block is moved or copied.
 * Replaces the gather/scatter at src/nats/models/utils.py:509-588 (NAtSLayerCache.update). */
int natsl_kv_compact(const void* src_k, const void* src_v, long long src_tokens, int src_block0, void* dst_k, void* dst_v,
                     long long dst_tokens, const void* types, int types_dtype, const int64_t* n_before, int B, int HKV,
                     int HN, int K, int V, int dtype, int block, int NB, int n_complete, int tail_dst, int tail_tokens,
                     natsl_stream_t stream);

/* natsl_kv_compact into a cache that is new (uninitialised) memory of whole blocks: the first region of a sequence, nothing kept
 * before; every block of the cache that holds nothing is zeroed. */
int natsl_kv_collect(const void* src_k, const void* src_v, long long src_tokens, void* dst_k, void* dst_v, long long dst_tokens, const void* types,
                     int types_dtype, int B, int HKV, int HN, int K, int V, int dtype, int block, int NB, int n_complete, int tail_dst,
                     int tail_tokens, natsl_stream_t stream);

/* The cache's bookkeeping around natsl_kv_compact: n_after [B, HN] = n_before (or 0) + the attention-typed blocks among the first
 * n_complete of types [B, NB, HN, 2], with the largest of them written to *host_max (HOST memory that the GPU can write); and the
 * validity flags valid [B, blocks, HN] of n_after kept blocks plus the incomplete block at tail_block (-1 = none).
 * src/nats/models/utils.py:509-588. */
int natsl_kv_counts(const void* types, int types_dtype, const int64_t* n_before, int64_t* n_after, int32_t* host_max, int B, int HN, int NB,
                    int n_complete, natsl_stream_t stream);
int natsl_kv_flags(const int64_t* n_after, uint8_t* valid, int B, int blocks, int HN, int tail_block, natsl_stream_t stream);
/* natsl_kv_flags, and g_sum [B, H] = the sum of g [B, T, H] over the last `rest` tokens (fp32; 0 for none). */
int natsl_kv_note(const int64_t* n_after, uint8_t* valid, int B, int blocks, int HN, int tail_block, const float* g, float* g_sum, int T, int H,
                  int rest, natsl_stream_t stream);

/* The incomplete block's rows of a cache that was empty: for each of n tensors, dst [B, block, row] = the last `rest` tokens of
 * src [B, T, row] and zeros behind them (dense, row_bytes a token). */
#define NATSL_TAIL_SEGS 8
typedef struct natsl_tail_seg {
  const void* src;
  void* dst;
  int64_t row_bytes;
} natsl_tail_seg;
int natsl_block_tails(const natsl_tail_seg* segs, int n, int B, int T, int block, int rest, natsl_stream_t stream);

/* out [B, H, state_elems] = ht where the last block's type is linear (last_types: element [b, hn, 1] at b * stride_b + hn * stride_h + 1),
 * else hs, times exp(gs [B, H]) unless gs is NULL: the state the next block starts from when the input ends on a block's end
 * (src/nats/ops/gated_delta_rule/chunk_fwd.py:178-206). */
int natsl_roll_state(const float* ht, const float* hs, const float* gs, const void* last_types, int types_dtype, int64_t stride_b, int64_t stride_h,
                     float* out, int B, int H, int HN, int64_t state_elems, natsl_stream_t stream);

/* The layers' short convolutions with what follows them, for up to NATSL_CONV_SEGS bf16 tensors [B, T, D_i] in one launch:
 *   y = act(conv(x)) (as natsl_short_conv_fwd; bf16 weights [D, W]), and, when y_norm is given, its rows of 8 * norm_lanes
 *   channels (a power of two of lanes) normalised: y rsqrt(mean y^2 + eps) norm_weight, or y rsqrt(sum y^2 + eps) (norm_l2); or,
 *   where scale [B, T, D / (8 norm_lanes)] is given, multiplied by its number (then without norm_weight; dscale: its gradient, zeros without dy_norm; may be NULL).
 * The backward takes the gradients that meet at y (dy_a, dy_b, and dy_norm through the norm; each may be NULL) and one that
 * meets at x (dx_add), and gives dx, dweight, dbias (bf16) and dnorm_weight (norm_dtype); sums in a fixed order.
 * Takes the place of natsl_short_conv_* and natsl_row_norm_* inside the layers (src/nats/layers/natsl_attn_gdn.py:425-505). */
#define NATSL_CONV_SEGS 3
typedef struct natsl_conv_seg {
  const void *x, *weight, *bias, *state, *norm_weight;
  void *y, *y_norm, *state_out;
  const void *dy_a, *dy_b, *dy_norm, *dx_add;
  void *dx, *dweight, *dbias, *dnorm_weight;
  int32_t D, norm_lanes, norm_l2;
  float norm_eps;
  const float* scale;
  float* dscale;
} natsl_conv_seg;
int natsl_conv_norm_fwd(const natsl_conv_seg* seg, int n_seg, int B, int T, int W, int activation, int norm_dtype, natsl_stream_t stream);
size_t natsl_conv_norm_bwd_workspace_bytes(const natsl_conv_seg* seg, int n_seg, int B, int T, int W);
int natsl_conv_norm_bwd(const natsl_conv_seg* seg, int n_seg, int B, int T, int W, int activation, int norm_dtype, void* workspace,
                        size_t workspace_bytes, natsl_stream_t stream);

/* The narrow products of one input in one pass over it (bf16): ab [B T, ld] = x [wa; wb]^T (columns behind NA + NB are zero), and, where asked
 * for: wn -> the means of x over blocks of 64 tokens (pooled [B, cdiv(T,64), D]; may be NULL) and logits [B, cdiv(T,64), NL] = means wn^T; g -> the
 * gates of natsl_gates_fwd from ab's rounded values (NA heads; ab itself may then be NULL); wab [wab_rows, D] = [wa; wb; zeros].  D a multiple of 32,
 * NA + NB <= 64 (32 with logits), NL <= 64.  src/nats/layers/natsl_attn_gdn.py:411-420, 507-512, src/nats/layers/natsl_attn_mamba2.py:391-393. */
typedef struct natsl_front {
  const void *x, *wa, *wb, *wn, *a_log, *dt_bias;
  void *ab, *pooled, *logits, *beta, *wab;
  float *g, *dt;
  int32_t B, T, D, NA, NB, NL, ld, neg_eigval, param_dtype, wab_rows;
} natsl_front;
int natsl_layer_front(const natsl_front* a, natsl_stream_t stream);
/* dw [N, D] = dy [rows, N]^T x [rows, D] (bf16, N up to 64, D even) for a narrow weight over few rows: the selector's over the block means. */
int natsl_narrow_wgrad(const void* dy, const void* x, void* dw, int64_t rows, int D, int N, natsl_stream_t stream);
/* The same over many rows, through partial sums in a workspace: the mixing logits' weight. */
size_t natsl_narrow_wgrad_workspace_bytes(int64_t rows, int D, int N);
int natsl_narrow_wgrad_split(const void* dy, const void* x, void* dw, int64_t rows, int D, int N, void* workspace, size_t workspace_bytes, natsl_stream_t stream);

/* The layers' gates from one projection ab [rows, ld] (bf16; a in columns 0..H-1, b in H..2H-1 for the delta rule):
 * g = -exp(a_log) softplus(a + dt_bias) fp32 [rows, H], beta = sigmoid(b) bf16 (doubled with neg_eigval; NULL for Mamba),
 * dt = softplus(a + dt_bias) fp32 (or NULL); and the gradients (dab has zeros behind the used columns).
 * src/nats/layers/natsl_attn_gdn.py:507-512, src/nats/layers/natsl_attn_mamba2.py:391-393. */
int natsl_gates_fwd(const void* ab, const void* a_log, const void* dt_bias, float* g, void* beta, float* dt, int64_t rows, int H, int ld,
                    int neg_eigval, int param_dtype, natsl_stream_t stream);
size_t natsl_gates_bwd_workspace_bytes(int64_t rows, int H);
int natsl_gates_bwd(const void* ab, const void* a_log, const void* dt_bias, const float* dg, const void* dbeta, const float* ddt, int delta,
                    void* dab, void* da_log, void* ddt_bias, void* workspace, size_t workspace_bytes, int64_t rows, int H, int ld,
                    int neg_eigval, int param_dtype, natsl_stream_t stream);

/* dx [B, T, D] = dn [B*T, ld] w [N, D] (N a multiple of 16, 0 = none) + the block mean's gradient dpool [B, ceil(T/block), D] (or
 * NULL) over the block's length, bf16: the terms of a layer's input gradient that are no wide product. */
int natsl_dx_init(const void* dn, const void* w, const void* dpool, void* dx, int B, int T, int D, int N, int ld, int block,
                  natsl_stream_t stream);

/* Straight-through gradient of natsl_hard_select: the softmax's backward of dtypes, [B, TN, HN, 2] in one dtype; last_forced:
 * the last block's types were constants (src/nats/layers/natsl_attn_gdn.py:47-61, :553-554). */
int natsl_hard_select_bwd(const void* logits, const void* dtypes, void* dlogits, int B, int TN, int HN, int dtype, int last_forced,
                          natsl_stream_t stream);

/* Weight gradients of up to NATSL_WGRAD_SEGS projections that share their input: out_i [n_i, D] = dy_i^T x, bf16, sums in fp32;
 * dy_i [T, ld_i] (n_i columns used), x [T, ldx] (D columns used); widths and row strides are multiples of 8, dy and x start on
 * 16 bytes.  Deterministic.  Takes the place of the library products in the backward of the layers' projections
 * (src/nats/layers/natsl_attn_gdn.py:425-491). */
#define NATSL_WGRAD_SEGS 8
typedef struct natsl_wgrad_seg { const void* dy; void* out; int32_t n, ld; } natsl_wgrad_seg;
size_t natsl_wgrad_workspace_bytes(const natsl_wgrad_seg* segs, int n_seg, int64_t T, int D);
int natsl_wgrad(const natsl_wgrad_seg* segs, int n_seg, const void* x, int64_t T, int D, int ldx, void* workspace,
                size_t workspace_bytes, natsl_stream_t stream);

/* The wide products of up to NATSL_PROJECT_SEGS projections that share their input, one launch, bf16 with fp32 sums and one rounding.
 * natsl_project: y_i [rows, ld_i] (n_i columns written) = x [rows, ldx] w_i^T, w_i [n_i, D] contiguous; D a multiple of 32 from 128 on.
 * natsl_project_bwd: dx [B*T, D] = sum_i dy_i w_i + the block mean's gradient dpool [B, ceil(T/block), D] (or NULL) over the block's
 * length; every n_i a multiple of 32, 128 or more in all.  Widths and row strides are multiples of
 * 8, tensors start on 16 bytes; nothing else is taken.  (src/nats/layers/natsl_attn_gdn.py:425-491) */
#define NATSL_PROJECT_SEGS 8
typedef struct natsl_project_seg { const void* y; const void* w; int32_t n, ld; } natsl_project_seg;
int natsl_project(const natsl_project_seg* segs, int n_seg, const void* x, int64_t rows, int D, int ldx, natsl_stream_t stream);
int natsl_project_bwd(const natsl_project_seg* segs, int n_seg, const void* dpool, void* dx, int B, int T, int D, int block,
                      natsl_stream_t stream);

/* dx [rows, D] = dy [rows, N] w for a narrow weight w [N, D] (N a multiple of 4 up to 48, D of 128), bf16 with fp32 sums.  Contiguous, on 16
 * bytes.  (The mixing logits' layer, src/nats/layers/natsl_attn_gdn.py:425-491.) */
int natsl_narrow_linear_bwd(const void* dy, const void* w, void* dx, int64_t rows, int D, int N, natsl_stream_t stream);

/* Which of several ways to the same product the layers take: rules on sizes, on the host, for every caller the same.  Alignments are the caller's.
 * natsl_narrow_fwd_pays: the mixing logits [rows, N] = x [rows, D] w^T by natsl_layer_front.  natsl_narrow_linear_bwd_pays: dx by
 * natsl_narrow_linear_bwd; few != 0: the selector's, over the block means.  natsl_narrow_wgrad_pays: dw [N, D] = dy [rows, N]^T x by natsl_narrow_wgrad
 * (1; few only) or natsl_narrow_wgrad_split (2); alone: no other weight's gradient shares its launch of natsl_wgrad.  0: the other way (natsl_wgrad, the library). */
int natsl_narrow_fwd_pays(int64_t rows, int D, int N);
int natsl_narrow_linear_bwd_pays(int64_t rows, int D, int N, int few);
int natsl_narrow_wgrad_pays(int64_t rows, int D, int N, int few, int alone);
/* Whether natsl_project_bwd takes the projections' widths and the tensors' alignment; else dx is natsl_dx_init's and the wide products accumulate onto it. */
int natsl_project_bwd_takes(const natsl_project_seg* segs, int n_seg, const void* dpool, const void* dx);

/* natsl_gdn_chunk_fwd (is_delta) or natsl_mamba_chunk_fwd with NATSL_STATES_ONLY and no state of the last block.  beside: NULL, or
 * another stream of the same device that is made to wait for `stream` up to the kernel in front of the scan, for work that shares the
 * GPU with the scan. */
int natsl_linear_chunk_states(int is_delta, const void* q, const void* k, const void* v, const float* g, const void* beta, const float* h0, float* ht,
                              void* chunk_states, void* chunk_v_new, const void* types, int types_dtype, int B, int T, int H, int HN, int K, int V,
                              int TN, int block, float scale, int flags, void* workspace, size_t workspace_bytes, int dtype, const natsl_seq_row* seqs,
                              int n_seqs, int total_units, natsl_stream_t stream, natsl_stream_t beside);

/* The mixed operator's forward (src/nats/ops/mixed_ops/mixed_attn_gdn.py:47-191, src/nats/ops/mixed_ops/mixed_attn_mamba.py:51-192)
 * in one call: natsl_route, natsl_softmax_sparse_fwd and natsl_gdn_chunk_fwd (is_delta) or natsl_mamba_chunk_fwd with the
 * arguments those take, in bf16, and in front of and behind them the conversions of fp32 tensors (cast_in: fp32 -> bf16,
 * cast_out: bf16 -> fp32; tensors on 16 bytes).  `phases` says which steps to enqueue, so that a caller can time them one by
 * one.  attn_stream carries routing and the softmax branch: the same stream, or another one, which is then made to wait for
 * `stream` before (at ROUTE) and waited for after (at JOIN).  Both belong to one device, which need not be the caller's current one.
 * The attention view may hold other lengths (a prefix of cached
 * keys): T_attn tokens in TN_attn blocks.
 * workspace: natsl_mixed_workspace_bytes(), for total_chunks as for natsl_linear_workspace_bytes; of the bytes behind the linear
 * branch's the softmax branch makes its work queues, so that calls with workspaces of their own may overlap and be replayed in any way.
 * With natsl_linear_workspace_bytes() alone it has the queues that natsl_softmax_sparse_fwd has.  (That entry takes the persistent kernel for
 * smaller problems than this one.) */
#define NATSL_MIXED_CASTS 8
enum natsl_mixed_phases { NATSL_MIXED_CONVERT = 1, NATSL_MIXED_ROUTE = 2, NATSL_MIXED_SOFTMAX = 4, NATSL_MIXED_LINEAR = 8, NATSL_MIXED_JOIN = 16 };
typedef struct natsl_cast { const void* src; void* dst; int64_t n; } natsl_cast;
typedef struct natsl_mixed {
  int32_t is_delta, B, T, H, HN, K, V, TN, block, flags;
  int32_t T_attn, TN_attn, HQ, HKV, KA, VA, same_block_visible, types_dtype;
  int32_t n_seqs, total_chunks, total_qtiles, n_cast_in, n_cast_out;
  int32_t private_tables;   /* block_indices and n_blocks are room for this call only: nobody reads them afterwards, they need not be written */
  float scale_attn, scale_linear;
  const void *q_attn, *k_attn, *v_attn, *types_attn;
  void* o_attn;
  float* lse;
  int32_t *block_indices, *n_blocks;
  const void *q, *k, *v;
  const float* g;
  const void* beta;
  const float* h0;
  void* o;
  float *ht, *h_block_start, *g_block_sum;
  void *chunk_states, *chunk_v_new;
  const void* types;
  void* workspace;
  size_t workspace_bytes;
  const natsl_seq_row* seqs;
  natsl_cast cast_in[NATSL_MIXED_CASTS], cast_out[NATSL_MIXED_CASTS];
} natsl_mixed;
size_t natsl_mixed_workspace_bytes(int64_t total_chunks, int H);
/* `to` waits for what `from` holds so far (two streams of one device). */
int natsl_order_streams(natsl_stream_t from, natsl_stream_t to);
int natsl_mixed_softmax_variant(int B, int T, int HQ, int HKV, int block, int packed);   /* natsl_softmax_fwd_variant of its softmax branch */
int natsl_mixed_fwd(const natsl_mixed* m, int phases, natsl_stream_t stream, natsl_stream_t attn_stream);

/* Decode: both operators of a step in one call and two launches -- what natsl_attn_masked_fwd and natsl_gdn_recurrent_fwd
 * (is_delta) or natsl_mamba_recurrent_fwd give on the same arguments, bf16, without the query-only form.  The attention runs
 * next to the recurrence and splits its keys over more workgroups; workspace of natsl_decode_workspace_bytes().
 * Replaces the pair of calls at src/nats/ops/mixed_ops/mixed_attn_gdn.py:475-503. */
size_t natsl_decode_workspace_bytes(int B, int T, int TK, int HQ, int VA);
int natsl_decode_fwd(int is_delta, const void* q_attn, const void* k_attn, const void* v_attn, const uint8_t* mask, void* o_attn,
                     int B, int T, int TK, int HQ, int HKV, int HM, int KA, int VA, float scale_attn, int64_t k_batch_stride,
                     int64_t v_batch_stride, void* workspace, size_t workspace_bytes, const void* q, const void* k,
                     const void* v, const float* g, const float* g_cumsum, const void* beta, const float* h0,
                     float* h_block_start, void* o, float* ht, const void* types, int types_dtype,
                     const int32_t* n_tokens_in_block, int n_tokens_in_block_scalar, int H, int HN, int K, int V, int block,
                     float scale, int flags, natsl_stream_t stream);

/* A generation step of a whole hybrid layer (bf16): T new tokens for each of B cached sequences, all inside the current
 * selector block, from the hidden states to the layer's output.  Replaces the decode path of the layers' forward
 * (src/nats/layers/natsl_attn_gdn.py:387-666, src/nats/layers/natsl_attn_mamba2.py:328-599) together with what their cache
 * does with the new tokens (src/nats/models/utils.py:178-457) when no block is compacted.
 * Weights are the layers' own (row-major [out, in], bf16; convolutions [channels, conv_width]); H linear heads of K / V, HQ
 * attention heads that divide them evenly, HN selector heads; B*T <= 64.  The cache rows of the new tokens are written in
 * place: cache_k / cache_v [B, cache_tokens, HQ, *] at token n_kept*block + n_in, cache_valid (a byte per (sequence, block,
 * selector head)) for the incomplete block, block_k / block_v / block_g / block_beta / block_hidden [B, block, ...] at n_in
 * (block_hidden may be NULL).  States and convolution states are read from one tensor and written to another. */
enum natsl_step_flags {
  NATSL_STEP_DECAY = 1,          /* decay_for_non_*_blocks */
  NATSL_STEP_SILU = 2,           /* the convolutions' activation */
  NATSL_STEP_ATTN_FROM_CONV = 4, /* the attention view takes the convolved q, k, v (else the projections) */
  NATSL_STEP_ATTN_NORM = 8,      /* RMSNorm of the attention view's q and k rows */
  NATSL_STEP_L2_ROWS = 16,       /* the linear view's q and k rows are L2-normalised (and rounded) first (Mamba layer) */
  NATSL_STEP_ATTN_OWN_BLOCK = 32,/* the softmax operator runs on the incomplete block */
  NATSL_STEP_NEG_EIGVAL = 64,    /* beta doubled */
  NATSL_STEP_FRESH_START = 128   /* block_start is written only: the block starts from `state` */
};
typedef struct natsl_layer_step {
  int32_t B, T, D, H, K, V, HQ, HN, block, conv_width, is_delta, flags;
  int32_t n_in, n_kept, cache_tokens, types_dtype, norm_dtype, gate_dtype, out_norm_dtype, reserved;
  float scale_attn, scale_linear, norm_eps, l2_eps, out_norm_eps, reserved_f;
  const void *wq, *wk, *wv, *wg, *wa, *wb, *w_mix, *wo;
  const void *conv_wq, *conv_wk, *conv_wv, *conv_bq, *conv_bk, *conv_bv;
  const void *norm_q, *norm_k, *a_log, *dt_bias, *out_norm1, *out_norm2;
  const void *x, *types;
  const void *conv_state_q, *conv_state_k, *conv_state_v;
  void *conv_out_q, *conv_out_k, *conv_out_v;
  const float *state, *g_cumsum;
  float *block_start, *state_out, *g_cumsum_out;
  void *cache_k, *cache_v;
  uint8_t* cache_valid;
  void *block_k, *block_v;
  float* block_g;
  void *block_beta, *block_hidden;
  void* out;
} natsl_layer_step;
size_t natsl_layer_step_workspace_bytes(const natsl_layer_step* step);
int natsl_layer_step_fwd(const natsl_layer_step* step, void* workspace, size_t workspace_bytes, natsl_stream_t stream);
/* The same with memory that the caller keeps from step to step, natsl_layer_step_sync_bytes of it on the device, zeros before the first step and
 * not touched between steps: a step of one token of few sequences is one launch then instead of three.  0 bytes: such a step meets nowhere, but it is given
 * the memory of the cache's other steps, where there is any, to know whether one of them failed.
 * Steps that may run at the same time, or of other numbers of sequences, have memory of their own.  A process has one launch at a time on a device whose
 * parts wait for each other and have not all started, or several on one stream: steps on another stream meanwhile, and captured ones, are several
 * launches.  Those of two processes fit on a device side by side; where more processes step on one, they can keep each other waiting.  A part of the launch that waits
 * longer than max_wait_us for another gives up: the step's output, and that of every later step with this memory, in one launch or in several, is NaN.
 * Word NATSL_STEP_SYNC_FAILED of the memory is not 0 from then on. */
enum { NATSL_STEP_SYNC_FAILED = 32 };
size_t natsl_layer_step_sync_bytes(const natsl_layer_step* step);
int natsl_layer_step_sync_fwd(const natsl_layer_step* step, void* workspace, size_t workspace_bytes, void* shared, size_t shared_bytes,
                              uint64_t max_wait_us, natsl_stream_t stream);
/* A number that changes with every such launch of this process on the device that gives up, 0 before the first: by when the host sees it, the launch's memory
 * says so, too. */
uint64_t natsl_layer_step_gave_up(int device);

#ifdef __cplusplus
}
#endif
#endif /* NATSL_H */
