/*
 * gstar_evict — C ABI of the MI355X (gfx950) KV-cache eviction hot path.
 *
 * Every entry point takes caller-owned device buffers as plain pointers with
 * element strides, sizes as integers, and the HIP stream to launch on as the
 * last argument. Entry points return GSE_OK or an error code; the message of
 * the last error on the calling thread is available from gse_last_error().
 * Kernels never allocate; buffers the kernels need beyond inputs and outputs
 * come in through a caller-provided workspace.
 *
 * Reference paths below are relative to the tonghuikang/cache-eviction
 * repository: R = code/cache_eviction/sglang_evict_runtime.py,
 * C = code/cache_eviction/core.py, T = code/tests/test_sglang_evict.py, TEX = source.tex (the
 * reference report, which describes the block variant that the reference ships no code for).
 *
 * Layouts (the reference's, R:89-110):
 *   K/V pool of one layer   bf16 [slots, kv_heads, head_dim], head_dim contiguous
 *   scores                  fp32 [full layers, kv_heads, slots] with explicit strides; the
 *                           runtime keeps the KV heads of a slot adjacent (strides
 *                           slots*kv_heads, 1, kv_heads), so one page's scores fill whole lines
 *   table / req_to_token    int32 [rows, width]
 *   frontier / count / mode int32 [rows]; a mode word (mode_by_row[row], and the `mode`
 *                           of gse_prefill_scores) holds the score kind in bits 0-3 (1 sum,
 *                           2 max over a KV head's query heads, 4 block counters
 *                           (GSE_SCORE_KIND_BLOCK_STEP), else no scores), log2 of the
 *                           block size in bits 4-7 (kind 4 only) and the score delay in
 *                           bits 8-30 (GSE_SCORE_DELAY_SHIFT)
 *   pos (per row)           int32 [full layers, kv_heads, count]
 */
#ifndef GSTAR_EVICT_H
#define GSTAR_EVICT_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef struct ihipStream_t* gse_stream_t; /* hipStream_t */

enum { GSE_OK = 0, GSE_EINVAL = 1, GSE_ESHAPE = 2, GSE_ELAUNCH = 3, GSE_EWORKSPACE = 4 };
enum { GSE_I32 = 0, GSE_I64 = 1 };  /* dtype codes of index arrays */
enum { GSE_F32 = 0, GSE_BF16 = 1 }; /* dtype codes of float arrays */

/* Policy ids of the boundary selector (names of R:45-46). */
enum {
  GSE_POLICY_HEAD_SUM = 1,         /* head_sum_2048: scores gathered from the score table */
  GSE_POLICY_HEAD_MAX_SUM = 2,     /* head_max_sum_2048: same gather                   */
  GSE_POLICY_RANDOM = 3,           /* random_2048: caller-drawn float64 scores          */
  GSE_POLICY_RESERVOIR = 4,        /* random_reservoir_2048: splitmix64 in-kernel       */
  GSE_POLICY_PREFIX_SLIDING = 5,   /* prefix_sliding_2048: protected set only           */
  GSE_POLICY_BLOCK_SUM = 6,        /* block_sum_2048 (no reference counterpart): a block's
                                      score is the sum of its table scores              */
  GSE_POLICY_BLOCK_MAX = 7         /* block_max_2048 (no reference counterpart): the max */
};

/* Decode score modes of gse_decode. */
enum {
  GSE_SCORE_NONE = 0,  /* attention only                                                */
  GSE_SCORE_EAGER = 1, /* this step's scores are added before the call returns (second K */
                       /* pass, the reference's per-step update)                         */
  GSE_SCORE_QUEUE = 2  /* this step's query is queued; gse_score_flush adds the queued   */
                       /* queries' scores (one K pass per queue)                         */
};

/*
 * Score delay (block policies; no reference counterpart, the reference report's ARC-AGI-3 runs
 * count a block's attention only after 128 tokens, TEX:197): with delay d = word >> 8, a query
 * at list length lim (its own key being entry lim - 1) adds scores to entries c < lim - d only.
 * A block-policy boundary leaves the row's newest positions at the end of its table (the
 * protected recent region after the kept middle), so with d <= recent these are exactly the
 * keys at least d positions older than the query. d = 0 is the reference's update.
 */
#define GSE_SCORE_DELAY_SHIFT 8

/*
 * Block counters (score kind 4; no reference code: the reference report's ARC-AGI-3 block score,
 * TEX:197, "a counter per block, scored by the maximum post-softmax attention over its four
 * tokens and all query heads, counted after a delay of 128 tokens"). A block is 2^s aligned
 * entries of the row's list (s = bits 4-7 of the word, 0..6); a block-policy boundary keeps
 * whole position blocks in position order, so list blocks are position blocks. A query at list
 * length lim credits the whole blocks of entries c < lim - d (d the delay): each such block's
 * counter, KV head 0's score of the block's first slot, grows by the maximum over the block's
 * keys and all query heads of the query's probability. The other slots of the block keep 0, so
 * a block policy's sum or max over the block's scores is the counter.
 */
#define GSE_SCORE_KIND_BLOCK_STEP 4
#define GSE_SCORE_BLOCK_SHIFT 4

/* Boundary outcome written to device memory by gse_boundary. */
enum {
  GSE_BOUNDARY_EVICTED = 0,
  GSE_BOUNDARY_DEFERRED = 2,       /* protected count > budget (R:390-391, R:438-441)       */
  GSE_BOUNDARY_ERR_HEADS = 3,      /* heads protect different counts (R:388-389)             */
  GSE_BOUNDARY_ERR_SWA = 4,        /* a leftover slot still holds a sliding-window entry (R:477-479) */
  GSE_BOUNDARY_ERR_PACKED = 5,     /* packed ownership overlaps the sliding-window region (R:487-489) */
  GSE_BOUNDARY_ERR_RELOCATE = 6    /* the single-pass relocation's grid barrier timed out after its
                                      first phase (no reference counterpart; not seen in practice:
                                      a wait that times out in the first phase abandons the single
                                      pass before any store, and the relocation runs through scratch) */
};

/* gse_boundary_status.relocation: how the survivors' K/V/score rows were moved. */
enum {
  GSE_RELOCATION_SINGLE_PASS = 0,  /* one kernel with grid barriers, or no move needed            */
  GSE_RELOCATION_SCRATCH = 1       /* through scratch: chosen by the host (widths past the single
                                      pass's capacity, GSE_RELOCATE_SCRATCH=1) or taken after the
                                      single pass found its workgroups not all resident           */
};

typedef struct {
  int32_t state;            /* GSE_BOUNDARY_*                                   */
  int32_t protected_count;  /* protected columns of head (0, 0)                 */
  int32_t width;            /* kept middle columns per head                     */
  int32_t count;            /* new table length = protected_count + width       */
  int32_t leftover;         /* slots handed back (candidates beyond width)      */
  int32_t packed;           /* owned slots packed at the start of req_to_token  */
  int32_t min_protected;    /* smallest per-head protected count                */
  int32_t max_protected;    /* largest per-head protected count                 */
  int32_t relocation;       /* GSE_RELOCATION_*                                 */
} gse_boundary_status;

/* Library version (major * 10000 + minor * 100 + patch) and last error text. */
int gse_version(void);
const char* gse_last_error(void);

/*
 * fill — full-layer CSR of resident slots. Replaces R:136-152 (`fill`, with
 * SGLang's create_flashinfer_kv_indices_triton called twice, R:147-151):
 *   kv_indptr[b+1] = sum_{i<=b} (seq_lens[i] - frontier[rows[i]] + count[rows[i]])
 *   kv_indices     = table[row, :count] ++ req_to_token[row, frontier:seq_len]   per b
 * max_len bounds every entry's list length (e.g. req_to_token's width); the grid is
 * (bs, max_len / 2048 + 1) and reads nothing on the host: capturable in a HIP graph.
 */
int gse_fill(const int32_t* table, int64_t table_stride, const int32_t* req_to_token, int64_t r2t_stride,
             const void* rows, int rows_dtype, const void* seq_lens, int lens_dtype,
             const int32_t* frontier, const int32_t* count, int bs, int64_t max_len,
             int32_t* kv_indptr, void* kv_indices, int indices_dtype, gse_stream_t stream);

/*
 * zero_slots — scores[l, g, slots[i]] = 0 for every full layer l and KV head g.
 * Replaces R:211-212 / R:293-294 (`st.scores.index_fill_(2, out_cache_loc, 0.0)`).
 */
int gse_zero_slots(float* scores, int layers, int64_t layer_stride, int kv_heads, int64_t head_stride,
                   int64_t slot_stride, const void* slots, int slots_dtype, int64_t n, gse_stream_t stream);

/* A key list of two parts as int32 slots: out[0..n) = first, out[n..n+m) = second (each int32
 * or int64, contiguous). */
int gse_join_slots(const void* first, int first_dtype, int64_t n, const void* second, int second_dtype, int64_t m,
                   int32_t* out, gse_stream_t stream);

/* Workspace bytes gse_decode needs for bs sequences. */
int64_t gse_decode_workspace_bytes(int bs, int q_heads, int head_dim);

/* Extra workspace bytes of a gse_decode call that folds n_fold queues over lists of at most
 * max_len entries (0 when n_fold is 0); see gse_decode. */
int64_t gse_decode_fold_bytes(int n_fold, int kv_heads, int max_len);

/*
 * decode — one full-attention layer's decode step: attention with the learned
 * sink folded into the softmax normaliser, plus the H2O score of the step's
 * query. Replaces SGLang's decode_attention_fwd (the attention before the
 * reference's after_decode hook, O:35-41) together with `_decode_scores` /
 * `after_decode` (R:155-224):
 *   o[b, h]       = sum_s softmax([q_h.k_s*scale, sink_h])_s v_s  (sink column dropped)
 *   norm_out[b,h] = log(exp(sink_h) + sum_s exp(q_h.k_s*scale))    (may be null)
 *   scores[g, slot_s] += sum_{h in g} p_hs  (mode 1)  or  max_{h in g} p_hs  (mode 2)
 * where mode = mode_by_row[rows[b]] & 0xff, for the list's entries s < len - delay (the
 * word's score delay); rows whose mode is not 1 or 2 get no score.
 * score_mode GSE_SCORE_EAGER adds the scores before returning (max_len bounds
 * every sequence's list length); GSE_SCORE_QUEUE appends the step to the row's
 * queue instead: queue_count[row] = n + 1 for n = queue_count[row], and if n < queue_cap
 *   entry n receives queue_q[row, n] = q[b] ([q_heads, 64] bf16), queue_norm[row, n] =
 *   norm (natural log, [q_heads]) and queue_lim[row, n] = the list length;
 * gse_score_flush adds the queued scores. The caller flushes a row before its queue is
 * full (a count above queue_cap records dropped steps) and before the row's list changes
 * other than by appending (boundaries). Shapes: q_heads = 8 * kv_heads, kv_heads <= 8,
 * head_dim = 64; a slot's K and V head rows lie within one slot row (kv_stride_s elements)
 * of under 16 KiB, read as one record of a buffer resource (GSE_ESHAPE otherwise). The
 * attention kernel runs one workgroup per CU over an equal share of the batch's keys, or one
 * per 64 of the bs * max_len keys when that is fewer (max_len, the upper bound of the list
 * lengths, also sizes the grid); fixed grid, no host reads: capturable in a HIP graph. rows[b] must
 * index mode_by_row and the queue buffers (as SGLang's req_pool_indices index
 * req_to_token): the kernels do not check it.
 * Kept logits (logits may be null): for a sequence whose row has
 *   k = logit_index[rows[b]] in [0, logit_rows), the fp32 products q_h.k_c (unscaled) of its
 *   list entries c < min(list length, logit_cap) are written to logits[((k * kv_heads + g) *
 *   logit_cap + c) * 8 + j] for query head h = 8 * g + j (a plane per KV head);
 *   gse_score_flush_logits then adds a one-step queue's scores from them instead of reading K
 *   again. Entries of other sequences, and c >= logit_cap, are not written.
 * Queue folds (GSE_SCORE_QUEUE; fold_seq may be null when n_fold is 0): for each batch index
 *   b in fold_seq[0..n_fold) whose row has score kind 1 or 2, the launch also adds the row's
 *   queued steps (entries [0, queue_count[row])) to scores, as gse_score_flush would for this
 *   layer, in extra workgroups beside the attention (the fold is bound by its exponentials,
 *   the attention by HBM); the step's own entry then restarts the queue (entry 0, count 1).
 *   fold_seq is device memory. Call it for every full layer of the step, with the same list.
 *   fold_workgroups (in [0, CUs / 2]) of the launch's one-per-CU workgroups fold, the rest
 *   attend; 0 leaves the count to the library (32 per folded row, up to a third of the CUs).
 *   The workspace then needs gse_decode_workspace_bytes rounded up to 256 plus
 *   gse_decode_fold_bytes(n_fold, kv_heads, max_len) bytes: the fold workgroups write their
 *   totals there and the launch's merge adds them to scores after the attention has read K and
 *   V (random score writes during the attention's stream slowed it).
 */
int gse_decode(const void* q, int64_t q_stride_b, int64_t q_stride_h,
               const void* k_pool, const void* v_pool, int64_t kv_stride_s, int64_t kv_stride_h,
               const int32_t* kv_indptr, const void* kv_indices, int indices_dtype,
               const void* sinks, int sinks_dtype, const int32_t* mode_by_row, const void* rows, int rows_dtype,
               float* scores, int64_t scores_stride_g, int64_t scores_stride_s,
               void* o, int64_t o_stride_b, int64_t o_stride_h, float* norm_out,
               void* queue_q, float* queue_norm, int32_t* queue_lim, int32_t* queue_count, int queue_cap,
               int bs, int q_heads, int kv_heads, int head_dim, float sm_scale, int max_len,
               int score_mode, float* logits, const int32_t* logit_index, int logit_rows, int logit_cap,
               const int32_t* fold_seq, int n_fold, int fold_workgroups, void* workspace, int64_t workspace_bytes,
               gse_stream_t stream);

/* Bytes of the library's own scratch for gse_decode_noalloc on each GPU (9 MiB: bs <= 256 at
 * 64 query heads on 256 CUs). */
#define GSE_DECODE_NOALLOC_SCRATCH_BYTES (9 * 1024 * 1024)

/*
 * decode_noalloc — gse_decode without a workspace argument, allocating nothing: no counterpart
 * in the reference. For callers that cannot call hipMalloc (code under HIP graph capture, tight
 * serving loops, harnesses that forbid allocation). Same arguments (less the workspace), result
 * and kernels as gse_decode; the partials live in a static device array of
 * GSE_DECODE_NOALLOC_SCRATCH_BYTES per GPU, held until the process ends, whose address is looked
 * up once per device on its first call there. Returns GSE_EWORKSPACE (no launch) when
 * gse_decode_workspace_bytes(bs, q_heads, head_dim) exceeds that size. Every call on one GPU
 * shares its array: calls that overlap on one GPU (other streams, other threads) race, so
 * order them on one stream.
 */
int gse_decode_noalloc(const void* q, int64_t q_stride_b, int64_t q_stride_h,
                       const void* k_pool, const void* v_pool, int64_t kv_stride_s, int64_t kv_stride_h,
                       const int32_t* kv_indptr, const void* kv_indices, int indices_dtype,
                       const void* sinks, int sinks_dtype, const int32_t* mode_by_row, const void* rows,
                       int rows_dtype, float* scores, int64_t scores_stride_g, int64_t scores_stride_s,
                       void* o, int64_t o_stride_b, int64_t o_stride_h, float* norm_out,
                       void* queue_q, float* queue_norm, int32_t* queue_lim, int32_t* queue_count, int queue_cap,
                       int bs, int q_heads, int kv_heads, int head_dim, float sm_scale, int max_len,
                       int score_mode, float* logits, const int32_t* logit_index, int logit_rows, int logit_cap,
                       const int32_t* fold_seq, int n_fold, int fold_workgroups, gse_stream_t stream);

/*
 * score_flush — add the queued decode scores of the listed rows, for every full
 * layer, and empty their queues. No reference counterpart as an entry point: the
 * reference adds each step's scores eagerly (R:189-200, R:218-224); this applies
 * the same update for all queued steps at once:
 *   scores[l, g, slot(c)] += sum_i [c < lim_i - delay] (sum | max)_{h in g} exp(q_ih . k_cg * scale - norm_ih)
 * with slot(c) = table[row, c] for c < count[row], else req_to_token[row, frontier[row] + c - count[row]]
 * (the list of `fill`). k_pools is a device array of `layers` pointers; the queue
 * buffers are those of gse_decode for layer 0, each layer's `rows_total` rows after
 * the previous layer's. max_len bounds every listed row's list length. If a flushed
 * count exceeds queue_cap (steps that were dropped), *overflow (may be null) is set to 1.
 * A slot's row of K (kv_stride_s bf16 elements, the KV heads at kv_stride_h apart within
 * it) must be under 16 KiB: the kernels read it through a buffer resource of that record
 * size; GSE_ESHAPE otherwise.
 */
int gse_score_flush(void* const* k_pools, int layers, int64_t kv_stride_s, int64_t kv_stride_h,
                    float* scores, int64_t scores_stride_l, int64_t scores_stride_g, int64_t scores_stride_s,
                    const int32_t* table, int64_t table_stride, const int32_t* req_to_token, int64_t r2t_stride,
                    const int32_t* frontier, const int32_t* count, const int32_t* mode_by_row,
                    const void* rows, int rows_dtype, int n_rows, int64_t max_len,
                    const void* queue_q, const float* queue_norm, const int32_t* queue_lim, int32_t* queue_count,
                    int rows_total, int queue_cap, int q_heads, int kv_heads, int head_dim, float sm_scale,
                    int32_t* overflow, gse_stream_t stream);

/*
 * score_flush_short — gse_score_flush for short queues (a few steps per row, e.g. rows that
 * evict at every step): same arguments, result and queue handling. No reference counterpart
 * (the reference adds each step eagerly, R:189-200). Each workgroup reads every KV head of its
 * keys at once and writes a slot's score row with one read-modify-write (no atomics); up to 8
 * queued steps per row are read once, longer queues again per 128 keys, so for full queues
 * gse_score_flush is the faster choice.
 */
int gse_score_flush_short(void* const* k_pools, int layers, int64_t kv_stride_s, int64_t kv_stride_h,
                          float* scores, int64_t scores_stride_l, int64_t scores_stride_g,
                          int64_t scores_stride_s, const int32_t* table, int64_t table_stride,
                          const int32_t* req_to_token, int64_t r2t_stride, const int32_t* frontier,
                          const int32_t* count, const int32_t* mode_by_row, const void* rows, int rows_dtype,
                          int n_rows, int64_t max_len, const void* queue_q, const float* queue_norm,
                          const int32_t* queue_lim, int32_t* queue_count, int rows_total, int queue_cap,
                          int q_heads, int kv_heads, int head_dim, float sm_scale, int32_t* overflow,
                          gse_stream_t stream);

/*
 * score_flush_blocks — gse_score_flush for rows of score kind 4 (block counters,
 * GSE_SCORE_KIND_BLOCK_STEP; no reference code, TEX:197): per queued step in queue order,
 * each whole block of entries c < lim_i - delay adds to its counter (KV head 0's score of
 * the block's first slot) the maximum over its keys and all query heads of
 * exp(q_ih . k_c,g(h) * scale - norm_ih). Same arguments and queue semantics as
 * gse_score_flush; each entry point folds only rows of its own kinds and empties the
 * queues of every listed row, so a caller lists each row with the one that matches it.
 */
int gse_score_flush_blocks(void* const* k_pools, int layers, int64_t kv_stride_s, int64_t kv_stride_h,
                           float* scores, int64_t scores_stride_l, int64_t scores_stride_g,
                           int64_t scores_stride_s, const int32_t* table, int64_t table_stride,
                           const int32_t* req_to_token, int64_t r2t_stride, const int32_t* frontier,
                           const int32_t* count, const int32_t* mode_by_row, const void* rows, int rows_dtype,
                           int n_rows, int64_t max_len, const void* queue_q, const float* queue_norm,
                           const int32_t* queue_lim, int32_t* queue_count, int rows_total, int queue_cap,
                           int q_heads, int kv_heads, int head_dim, float sm_scale, int32_t* overflow,
                           gse_stream_t stream);

/*
 * score_flush_logits — gse_score_flush for rows whose queue holds exactly one step whose
 * products gse_decode kept (rows that evict at every step): same arguments and result, with
 * q_h.k_c read from `logits` (layer l's at logits + l * logits_layer_stride floats, laid out as
 * gse_decode writes them; logit_index, logit_rows and logit_cap as given to it) instead of
 * recomputed from K, 256 bytes per list entry read instead of 1024. K is not read. Rows of
 * score kinds 1 and 2 whose queue count is 1 and whose logit_index is in range are folded, for
 * entries c < min(lim - delay, logit_cap); the queues of every listed row are emptied. For
 * such a row the scores equal gse_score_flush_short's bit for bit. No reference counterpart
 * (R:189-200 adds each step eagerly).
 */
int gse_score_flush_logits(void* const* k_pools, int layers, int64_t kv_stride_s, int64_t kv_stride_h,
                           float* scores, int64_t scores_stride_l, int64_t scores_stride_g,
                           int64_t scores_stride_s, const int32_t* table, int64_t table_stride,
                           const int32_t* req_to_token, int64_t r2t_stride, const int32_t* frontier,
                           const int32_t* count, const int32_t* mode_by_row, const void* rows, int rows_dtype,
                           int n_rows, int64_t max_len, const void* queue_q, const float* queue_norm,
                           const int32_t* queue_lim, int32_t* queue_count, int rows_total, int queue_cap,
                           int q_heads, int kv_heads, int head_dim, float sm_scale, const float* logits,
                           int64_t logits_layer_stride, const int32_t* logit_index, int logit_rows, int logit_cap,
                           int32_t* overflow, gse_stream_t stream);

/*
 * decode_scores_from_lse —the reference's score update given an external
 * decode kernel's split log-sum-exps. Replaces `_decode_scores` + `after_decode`
 * (R:155-224) exactly: the normaliser is rebuilt from attn_lse [bs, q_heads,
 * max_kv_splits] (strides in elements) over the valid splits of SGLang's layout
 * per = cdiv(cdiv(len, num_kv_splits[b]), min_block_kv) * min_block_kv, started
 * at (sink, 1) (R:180-188), then every resident key's probability is added.
 * max_len bounds every sequence's list length (it sizes the grid). The pass forms the normalisers
 * itself: workspace is not used and may be null.
 */
int gse_decode_scores_from_lse(const void* q, int64_t q_stride_b, int64_t q_stride_h,
                               const void* k_pool, int64_t kv_stride_s, int64_t kv_stride_h,
                               const int32_t* kv_indptr, const void* kv_indices, int indices_dtype,
                               const float* attn_lse, int64_t lse_stride_b, int64_t lse_stride_h,
                               const int32_t* num_kv_splits, int max_kv_splits, int min_block_kv,
                               const void* sinks, int sinks_dtype, const int32_t* mode_by_row,
                               const void* rows, int rows_dtype, float* scores, int64_t scores_stride_g,
                               int64_t scores_stride_s,
                               int bs, int q_heads, int kv_heads, int head_dim, float sm_scale,
                               int max_len, void* workspace, int64_t workspace_bytes,
                               gse_stream_t stream);

/*
 * reservoir_scores — out[l, g, i] = (splitmix64 of (seed, layer_ids[l], head_ids[g], pos[l, g, i])) >> 11, / 2^53.
 * Replaces R:358-373 (and C:23-30). pos is int32 or int64 [L, G, N] contiguous;
 * null layer_ids / head_ids mean 0..L-1 / 0..G-1.
 */
int gse_reservoir_scores(const void* pos, int pos_dtype, const int64_t* layer_ids, const int64_t* head_ids,
                         int layers, int kv_heads, int64_t n, int64_t seed, double* out, gse_stream_t stream);

/*
 * select_kept — per (layer, KV head) row of pos [L, G, N] (int32) and float64
 * keys (score [L, G, N]; protected entries are ranked first), mark the kept
 * columns: protected ∪ top-(budget - protected) by (score desc, position desc).
 * Replaces the ranking of `choose` (R:376-397); kept_mask is uint8 [L, G, N],
 * prot_count int32 [L, G]. prefix_sliding keeps only the protected set.
 */
int gse_select_kept(const int32_t* pos, const double* score, int layers, int kv_heads, int64_t n_cols,
                    int64_t n, int64_t budget, int64_t prefix, int64_t recent, int64_t cursor, int has_cursor,
                    int prefix_sliding, uint8_t* kept_mask, int32_t* prot_count, void* workspace,
                    int64_t workspace_bytes, gse_stream_t stream);

/* Workspace bytes gse_boundary needs (n_cols = N columns, n = logical length; policy and
 * block as passed to gse_boundary). */
int64_t gse_boundary_workspace_bytes(int layers, int kv_heads, int head_dim, int64_t n_cols, int64_t n,
                                     int64_t budget, int policy, int block);

/*
 * boundary — ranking half of one row's eviction boundary at logical length n.
 * Replaces `choose`/`_scores` (R:376-412) and R:415-475 of `_boundary`:
 *   slots  = table[row, :count] ++ req_to_token[row, frontier:n]            (R:428)
 *   pos    = pos_old[l, g, :count] ++ arange(frontier, n)                    (R:429-431)
 *   keep   = protected ∪ top-k by (score desc, position desc) per head       (R:376-397)
 *   middle = each head's kept non-protected columns sorted by position       (R:444-446)
 *   targets/leftover = non-protected slots in column order split at width    (R:447-451)
 *   K, V, score of (middle[l,g,j], g) -> (targets[j], g) for every full layer (R:455-463)
 *   table[row] = slots[protected cols] ++ targets; count; frontier = n        (R:468-473)
 *   (block policies: slots[protected cols before the recent region] ++ targets ++ slots[the
 *   recent region's protected cols], the region starting at the first block of min(n - recent,
 *   cursor); pos_new in the same column order)
 * k_pools / v_pools are device arrays of `layers` device pointers. pos_old rows
 * are pos_old_stride elements apart. Writes pos_new [L, G, budget] (first
 * `count` columns valid), leftover slots (int64, N - count of them) and
 * *status. Deferred or invalid boundaries (status.state != EVICTED) change no
 * state. Call only when N = row_count + n - row_frontier > budget (R:433-435).
 * block / shared: 1 / 0 except for the block policies (no reference counterpart;
 * the block-granular, layer-shared variant of the reference report's ARC-AGI-3
 * runs), which keep whole blocks of `block` positions (1..2048): a block is
 * protected if any of its positions is, the kept width is budget - protected
 * rounded down to whole blocks, and each column ranks by its block's float64
 * score, the sum (GSE_POLICY_BLOCK_SUM) or max (GSE_POLICY_BLOCK_MAX) of the
 * table scores of the block's positions ascending and, if shared, of every KV
 * head of the layer ascending (then all heads of a layer keep the same blocks).
 */
int gse_boundary(void* const* k_pools, void* const* v_pools, int layers, int64_t kv_stride_s, int64_t kv_stride_h,
                 int kv_heads, int head_dim, float* scores, int64_t scores_stride_l, int64_t scores_stride_g,
                 int64_t scores_stride_s,
                 int32_t* table, int64_t table_stride, const int32_t* req_to_token, int64_t r2t_stride,
                 int32_t* frontier, int32_t* count, int row, int64_t row_count, int64_t row_frontier,
                 const int32_t* pos_old, int64_t pos_old_stride, int64_t n, int64_t budget, int64_t prefix,
                 int64_t recent, int64_t cursor, int has_cursor, int policy, int64_t seed, int block, int shared,
                 const double* random_scores, int32_t* pos_new, int64_t* leftover, gse_boundary_status* status,
                 void* workspace, int64_t workspace_bytes, gse_stream_t stream);

/*
 * One row of a boundary batch: gse_boundary's per-row arguments. The array is read on the host
 * during the call; the pointers in it are device memory.
 */
typedef struct {
  int32_t row;                  /* table / req_to_token row (distinct within a batch)            */
  int32_t has_cursor;           /* 1: `cursor` is the sliding-window guard (R:384-386)           */
  int64_t row_count;            /* the row's retained columns before the boundary                */
  int64_t row_frontier;         /* its frontier before the boundary                              */
  int64_t n;                    /* logical length at the boundary                                */
  int64_t cursor;
  const int32_t* pos_old;       /* [L, G, >= row_count] retained positions, rows pos_old_stride
                                   elements apart; null when row_count is 0                      */
  int64_t pos_old_stride;
  const double* random_scores;  /* random_2048: [L, G, N] draws; else null                      */
  int32_t* pos_new;             /* out: [L, G, budget]                                           */
  int64_t* leftover;            /* out: N slots (status.leftover of them valid)                  */
  gse_boundary_status* status;  /* out                                                           */
} gse_boundary_row;

/* Workspace bytes gse_boundary_batch needs for these rows. */
int64_t gse_boundary_batch_workspace_bytes(int layers, int kv_heads, int head_dim, const gse_boundary_row* rows,
                                           int n_rows, int64_t budget, int policy, int block);

/*
 * boundary_batch — gse_boundary for n_rows rows that share a policy and budget, each row's
 * result as if it ran alone (R:415-475 per row). No reference counterpart as an entry point: the
 * reference evicts one request at a time (R:704-710); when several rows reach a boundary at one
 * decode step (SGLang calls on_decode once per batch), their selections, column splits and
 * protected positions run as one launch each (up to 8 rows per launch) and their relocations one
 * row after another. Each row must satisfy gse_boundary's conditions (N > budget).
 */
int gse_boundary_batch(void* const* k_pools, void* const* v_pools, int layers, int64_t kv_stride_s,
                       int64_t kv_stride_h, int kv_heads, int head_dim, float* scores, int64_t scores_stride_l,
                       int64_t scores_stride_g, int64_t scores_stride_s, int32_t* table, int64_t table_stride,
                       const int32_t* req_to_token, int64_t r2t_stride, int32_t* frontier, int32_t* count,
                       const gse_boundary_row* rows, int n_rows, int64_t budget, int64_t prefix, int64_t recent,
                       int policy, int64_t seed, int block, int shared, void* workspace, int64_t workspace_bytes,
                       gse_stream_t stream);

/* Workspace bytes gse_boundary_live needs for a pool of num_slots slots. */
int64_t gse_boundary_live_workspace_bytes(int64_t num_slots);

/*
 * boundary_live — compaction half of a live boundary (R:476-491), after
 * gse_boundary reported EVICTED in *status:
 *   ERR_SWA if swa_mapping[leftover[i]] != 0 for any leftover slot (R:477-479), else
 *   scores[:, :, leftover] = 0                                            (R:481)
 *   true = min(n - recent, cursor or n); real = req_to_token[row, true:n]  (R:485-486)
 *   packed = table[row, :count] entries not in real, in order             (R:487)
 *   ERR_PACKED if len(packed) > true (R:488-489), else
 *   req_to_token[row, :true] = 0; req_to_token[row, :len(packed)] = packed (R:490-491)
 * swa_mapping (int32/int64 [num_slots]) may be null. The caller frees the
 * leftover slots (status.leftover of them) once the stream completes.
 */
int gse_boundary_live(float* scores, int layers, int64_t scores_stride_l, int kv_heads, int64_t scores_stride_g,
                      int64_t scores_stride_s,
                      const int32_t* table, int64_t table_stride, int32_t* req_to_token, int64_t r2t_stride,
                      int row, int64_t n, int64_t true_len, const int64_t* leftover, const void* swa_mapping,
                      int swa_dtype, int64_t num_slots, gse_boundary_status* status, void* workspace,
                      int64_t workspace_bytes, gse_stream_t stream);

/* One row of a live-compaction batch: gse_boundary_live's per-row arguments (host array). */
typedef struct {
  int32_t row;
  int64_t n;
  int64_t true_len;
  const int64_t* leftover;       /* the row's gse_boundary leftover output */
  gse_boundary_status* status;   /* the row's gse_boundary status          */
} gse_live_row;

/* Workspace bytes gse_boundary_live_batch needs for n_rows rows. */
int64_t gse_boundary_live_batch_workspace_bytes(int64_t num_slots, int n_rows);

/*
 * boundary_live_batch — gse_boundary_live for n_rows rows after their gse_boundary_batch (R:476-491
 * per row); its kernels run once for all rows (up to 8 rows per launch). No reference counterpart
 * as an entry point, for the same reason as gse_boundary_batch.
 */
int gse_boundary_live_batch(float* scores, int layers, int64_t scores_stride_l, int kv_heads,
                            int64_t scores_stride_g, int64_t scores_stride_s, const int32_t* table,
                            int64_t table_stride, int32_t* req_to_token, int64_t r2t_stride, const gse_live_row* rows,
                            int n_rows, const void* swa_mapping, int swa_dtype, int64_t num_slots, void* workspace,
                            int64_t workspace_bytes, gse_stream_t stream);

/*
 * prefill_scores — one extend chunk's exact per-KV-head column sums, added to
 * the score table (R:314-340, `_probabilities` + `_prefill_scores`):
 *   p[h, i, k] = exp(q_i,h . k_k * scale - logaddexp(logsumexp_k'(...), sink_h)),  k <= prefix_len + i
 *   scores[g, slots[k]] += sum_i (sum_{h in g} | max_{h in g}) p[h, i, k] [k <= prefix_len + i - delay]
 * with mode & 0xf (1 sum, 2 max) and the score delay of the mode word (the normaliser still
 * covers every key k <= prefix_len + i). Kind 4 (block counters, GSE_SCORE_KIND_BLOCK_STEP)
 * instead adds, per query i and whole block of keys < prefix_len + i + 1 - delay, the block's
 * maximum over its keys and all query heads of p to the block's counter (KV head 0's score of
 * the block's first slot); kv_heads <= 8. total must be below 2^31 keys.
 * q [count, q_heads, head_dim] bf16, keys gathered through slots (int64 or
 * int32, prefix slots then the chunk's own) from the pool. head_dim = 64,
 * q_heads = 8 * kv_heads. MFMA 16x16x32 bf16 tiles, two passes (row
 * log-sum-exp, then column sums). The workspace holds the row normalisers
 * (count * q_heads floats, rounded up to 256 bytes: the least that is accepted)
 * and pass 1's (reference, sum) pairs of each row and key range; one smaller
 * than gse_prefill_workspace_bytes takes fewer key ranges.
 */
int64_t gse_prefill_workspace_bytes(int64_t count, int q_heads);
int gse_prefill_scores(const void* q, int64_t q_stride_t, int64_t q_stride_h, int64_t count,
                       const void* k_pool, int64_t kv_stride_s, int64_t kv_stride_h,
                       const void* slots, int slots_dtype, int64_t total, int64_t prefix_len,
                       const void* sinks, int sinks_dtype, int mode, float* scores, int64_t scores_stride_g,
                       int64_t scores_stride_s,
                       int q_heads, int kv_heads, int head_dim, float sm_scale,
                       void* workspace, int64_t workspace_bytes, gse_stream_t stream);

/*
 * diagnose_chunk — one full layer of one prefill chunk of a static regret
 * diagnostic (R:587-615, `_diagnose`), with the row normalisers of
 * prefill_scores' first pass:
 *   score_sum[g, k] += sum_i sum_{h in g} p[h, i, k]      (k = CSR position 0..total-1)
 *   score_max[g, k] += sum_i max_{h in g} p[h, i, k]
 *   lost[s, i]      += lost_scale * sum_g sum_k [evicted(s, g, k)] sum_{h in g} p[h, i, k]
 * evicted: bit k%32 of word k/32 of row (s, g) (rows evicted_stride_g words,
 * covering total rounded up to 64); lost points at the chunk's first query
 * column; lost_scale = 1 / (q_heads * full layers). n_specs <= 8; same shape
 * limits, key limit and workspace as prefill_scores.
 */
int gse_diagnose_chunk(const void* q, int64_t q_stride_t, int64_t q_stride_h, int64_t count,
                       const void* k_pool, int64_t kv_stride_s, int64_t kv_stride_h,
                       const void* slots, int slots_dtype, int64_t total, int64_t prefix_len,
                       const void* sinks, int sinks_dtype, float* score_sum, float* score_max,
                       int64_t scores_stride_g, int64_t scores_stride_s, const uint32_t* evicted, int n_specs,
                       int64_t evicted_stride_s, int64_t evicted_stride_g, float* lost, int64_t lost_stride_s,
                       float lost_scale, int q_heads, int kv_heads, int head_dim, float sm_scale,
                       void* workspace, int64_t workspace_bytes, gse_stream_t stream);
/* A diagnostic's bit masks: words[(s * kv_heads + g) * n_words + k/32], bit k%32 set when
 * resident[s, g, k] (bytes, unit stride over k < n) is zero; 0 past n. n_words (even)
 * covers n rounded up to 64. */
int gse_pack_evicted(const void* resident, int64_t resident_stride_s, int64_t resident_stride_g, int n_specs,
                     int kv_heads, int64_t n, uint32_t* words, int64_t n_words, gse_stream_t stream);

/*
 * replay_layer_difference — static replay's per-query error of the first full
 * layer for one prefill chunk (R:520-546, `_replay_layer_difference`):
 *   a_i = attention of query start+i over positions 0..start+i (all unevicted keys)
 *   b_i = the same over each KV head's survivors: retained[g][0..retained_count)
 *         then positions frontier..start+i
 *   error[i] = |b_i - a_i| / max(|a_i|, 1e-12)   (norm over q_heads x head_dim)
 * Both with the sink in the normaliser. k_shadow / v_shadow hold the layer's
 * unevicted keys and values by position ([shadow_rows, kv_heads, head_dim]
 * bf16, shadow_rows >= start + count); retained positions (int32, rows
 * retained_stride_g apart) lie below frontier <= start. retained_count = 0
 * (nothing evicted yet) gives error 0. head_dim = 64, q_heads = 8 * kv_heads.
 * MFMA 16x16x32 bf16 tiles with a single-pass online softmax; probabilities
 * enter the value product as bf16 hi + lo parts. retained_count + start + count
 * must be below 2^31. The workspace holds both outputs, per key range where a
 * short chunk's keys are split; a smaller one than gse_replay_workspace_bytes
 * takes fewer ranges, down to the two outputs alone.
 */
int64_t gse_replay_workspace_bytes(int64_t count, int q_heads);
int gse_replay_layer_difference(const void* q, int64_t q_stride_t, int64_t q_stride_h, int64_t count,
                                const void* k_shadow, const void* v_shadow, int64_t kv_stride_s,
                                int64_t kv_stride_h, int64_t shadow_rows, int64_t start, const int32_t* retained,
                                int64_t retained_stride_g, int64_t retained_count, int64_t frontier,
                                const void* sinks, int sinks_dtype, int q_heads, int kv_heads, int head_dim,
                                float sm_scale, float* error, void* workspace, int64_t workspace_bytes,
                                gse_stream_t stream);

#ifdef __cplusplus
}
#endif

#endif /* GSTAR_EVICT_H */
