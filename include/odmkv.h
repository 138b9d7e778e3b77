/* odmkv.h - C ABI of libodmkv.so: ODM-KV compression-and-decode kernels for AMD MI355X (gfx950).
 *
 * Every pointer named "device" is HIP device memory owned by the caller (the Python host
 * side hands over torch tensors' data pointers).  The library allocates nothing that outlives
 * a call; scratch space is passed in as a workspace whose size the matching *_workspace_bytes
 * function returns.  All kernels are enqueued on the caller's stream (a hipStream_t passed as
 * void*); no entry point synchronises the device.  Every entry point returns 0 on success or
 * a negative ODMKV_E* code, and odmkv_last_error() then holds a message (thread local).
 *
 * Citations name the reference code (yiiwang118/ODM-KV) that each entry point stands in for.
 */
#ifndef ODMKV_H
#define ODMKV_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define ODMKV_VERSION 1

#define ODMKV_EINVAL   (-1)   /* bad argument: shape, level set, null pointer, unsupported head_dim */
#define ODMKV_ENOSPACE (-2)   /* workspace too small */
#define ODMKV_EHIP     (-3)   /* a HIP runtime call failed */
#define ODMKV_ENOMEM   (-4)   /* out of host memory */

/* element types of K/V/Q tensors */
#define ODMKV_F16  0
#define ODMKV_BF16 1
#define ODMKV_F32  2

#define ODMKV_HEAD_DIM   128  /* the only head_dim the kernels are written for */
#define ODMKV_TILE       64   /* tokens per packed tile = one wavefront */
#define ODMKV_NQ         4    /* quantised widths, in this order: 2, 3, 4, 8 bits */
#define ODMKV_MAX_LEVELS 8    /* candidate bit levels of the allocator */
#define ODMKV_MAX_GROUP  8    /* query heads per KV head (GQA group) */

int odmkv_version(void);
const char* odmkv_last_error(void);

/* ---------------------------------------------------------------------------------------------
 * Scorer.  Replaces RiskScorer.score_prefill after the mean query is known
 * (kvquant/scorer.py:285-325, 385-404) and RiskScorer.score_with_attn (kvquant/scorer.py:406-416).
 *
 *   p[h,t]  = mean over the G query heads of kv-head h of softmax_t( mu[q] . K[h,t] / sqrt(d) ),  t >= n_sink
 *   obar[h] = sum_t p[h,t] V[h,t] / max(sum_t p[h,t], 1e-8)
 *   s[h,t]  = (p[h,t] + eps)^2 * ( |V[h,t]|^2 + |K[h,t]|^2 / d * |V[h,t] - obar[h]|^2 )
 *   s[h, 0..n_sink) = max over all (h, t >= n_sink) of s
 *
 * K, V: [Hkv, T, 128] of `dtype`, element strides (stride_h, stride_t), innermost contiguous.
 * mu: device fp32 [Hq, 128], 16-byte aligned (the RoPE-averaged mean query; Hq = G * Hkv).
 * attn: NULL, or device fp32 [Hkv, T] attention weights to use instead of computing p from mu
 *       (then n_sink must be 0 and no sink padding happens: score_with_attn).
 * scores: device fp32 [Hkv, T] out.
 * Arithmetic: every sum is accumulated in fp32 in a fixed order.  With fp16 / bf16 keys the products mu . k run on
 * the matrix cores: the keys as they are, mu as 16-bit pieces whose sum is the fp32 vector (fp16: high + low of the
 * vector scaled by a power of two; bf16: three pieces), so that no bit of mu is dropped; fp32 keys take fp32 products.
 */
size_t odmkv_score_workspace_bytes(int Hkv, int Hq, int T);
int odmkv_score(const void* K, const void* V, int dtype, int Hkv, int T,
                int64_t stride_h, int64_t stride_t,
                const float* mu, int Hq, const float* attn, int n_sink, float eps,
                float* scores, void* workspace, size_t workspace_bytes, void* stream);

/* The same score as a model of 16-bit dtype computes it in the reference: the mean-query logits are rounded
 * to round_dtype (ODMKV_F16 / ODMKV_BF16) after the product and again after the division by sqrt(d), every
 * query head's softmax and the mean over the GQA group are rounded to it (kvquant/scorer.py:309-315, where
 * these tensors have the module's dtype), and so are eps, p + eps and its square (kvquant/scorer.py:403); the
 * rest is fp32 as in odmkv_score.  round_dtype = -1 is odmkv_score.  mu holds values of that dtype, widened to fp32. */
int odmkv_score_model_dtype(const void* K, const void* V, int dtype, int Hkv, int T,
                            int64_t stride_h, int64_t stride_t,
                            const float* mu, int Hq, const float* attn, int n_sink, float eps,
                            int round_dtype, float* scores, void* workspace, size_t workspace_bytes,
                            void* stream);

/* The mean query (kvquant/scorer.py:204-227, kvquant/attention_utils.py:57-115), around the layer's own projection:
 * odmkv_token_mean: out [batch, cols] = mean over the tokens of x [batch, rows, cols] (`dtype`, element strides; rows of whole
 * 16-byte pieces), summed in fp32 and rounded to dtype; workspace odmkv_token_mean_workspace_bytes (room for any call with at most that many rows).
 * odmkv_average_rope: out fp32 [heads, 128] = c * mu + s * rotate_half(mu) with c, s the means over the positions of cosine,
 * sine [positions, 128]; mu [heads, 128], all contiguous and of `dtype`; every product, sum and mean is rounded to dtype. */
size_t odmkv_token_mean_workspace_bytes(int batch, int rows, int cols);
int odmkv_token_mean(const void* x, int dtype, int batch, int rows, int cols, int64_t stride_b, int64_t stride_t,
                     void* out, void* workspace, size_t workspace_bytes, void* stream);
int odmkv_average_rope(const void* mu, const void* cosine, const void* sine, int dtype, int heads, int positions,
                       float* out, void* stream);

/* out [batch, rows] = x [batch, cols] . weight [rows, cols]^T + bias, weight and x of `dtype` (float16 / bfloat16), summed in
 * fp32 and rounded to dtype; out_dtype: dtype, or float32 for the rounded values widened. */
int odmkv_project_rows(const void* weight, int64_t ld, const void* bias, const void* x, int dtype, int batch, int rows,
                       int cols, void* out, int out_dtype, void* stream);

/* A prompt's risk scores from its hidden states (kvquant/scorer.py:285-325, 385-416), all sequences of the batch in one call:
 * token mean behind the sinks, projection, averaged RoPE, odmkv_score_model_dtype.  hidden_states [B, T, hidden], weight
 * [Hq * 128, hidden] and bias of `dtype` (float16 / bfloat16); cosine, sine [positions, 128] of dtype, or both NULL; K, V of
 * kv_dtype with element strides; scores fp32 [B, Hkv, T].  Long batches go in turns: the workspace stays within 64 MB, or what one
 * sequence takes. */
typedef struct odmkv_prompt {
    const void* hidden_states; int64_t h_stride_b, h_stride_t;
    const void* weight; int64_t ld_weight;
    const void* bias;
    const void* cosine; const void* sine;
    const void* K; const void* V; int64_t stride_b, stride_h, stride_t;
    float* scores;
    void* workspace; size_t workspace_bytes;
    int32_t dtype, kv_dtype, B, T, hidden, Hq, Hkv, positions, n_sink, round_dtype;
    float eps;
} odmkv_prompt_t;
size_t odmkv_prompt_scores_workspace_bytes(int B, int T, int hidden, int Hq, int Hkv);
int odmkv_prompt_scores(const odmkv_prompt_t* p, void* stream);

/* Mean and covariance of the queries of every head, through the averaged RoPE (kvquant/scorer.py:204-257,
 * kvquant/attention_utils.py:57-115): q float16 / bfloat16, head h and token t at element h * stride_h + t * stride_t; cosine,
 * sine fp32 [positions, 128] or NULL (no RoPE); mu fp32 [heads, 128], cov fp32 [heads, 128, 128]. */
size_t odmkv_query_covariance_workspace_bytes(int heads, int tokens);
int odmkv_query_covariance(const void* q, int dtype, int heads, int tokens, int64_t stride_h, int64_t stride_t,
                           const float* cosine, const float* sine, int positions, float* mu, float* cov,
                           void* workspace, size_t workspace_bytes, void* stream);

/* RoPE of a window's queries: q [heads, tokens, 128] (element strides) with cosine, sine [tokens, 128] of the same type, out
 * contiguous; every product and sum is rounded to the type. */
int odmkv_rotate_queries(const void* q, int dtype, int heads, int tokens, int64_t stride_h, int64_t stride_t,
                         const void* cosine, const void* sine, void* out, void* stream);

/* scores fp32 [rows, cols] -> out [rows, pad + cols]: the first pad columns are the largest score, and with scale != 0
 * everything is normalised to [0, 1] over the whole tensor (0.5 everywhere if max - min < 1e-8; kvquant/scorer.py:36-66). */
size_t odmkv_normalize_workspace_bytes(void);
int odmkv_normalize_scores(const float* scores, int64_t rows, int64_t cols, int pad, int scale, float* out,
                           void* workspace, size_t workspace_bytes, void* stream);

/* Expected-attention score.  Replaces ExpectedAttentionScorer.score_prefill after the query
 * statistics are known (kvquant/scorer.py:204-257):
 *
 *   logit[q,t] = mu[q] . K[h,t] / sqrt(d) + K[h,t]^T cov[q] K[h,t] / (2 d),   t >= n_sink, h = q / G
 *   p[h,t]     = mean over the G query heads of softmax_t(logit[q,:])
 *   s[h,t]     = use_vnorm ? (p[h,t] + eps) * |V[h,t]| : p[h,t]
 *   s[h, 0..n_sink) = max over all (h, t >= n_sink) of s
 *
 * mu: device fp32 [Hq, 128]; cov: device fp32 [Hq, 128, 128] (the RoPE-averaged query covariance),
 * or NULL for the mean-query term alone (use_covariance=False).  The quadratic form runs on the
 * matrix cores: 16-bit keys with cov split into two fp16 / three bf16 pieces (exact products, fp32
 * sums), fp32 keys on the fp32 matrix instructions.  K, V, strides, scores and the workspace (odmkv_score_workspace_bytes) are
 * those of odmkv_score.
 */
int odmkv_score_expected(const void* K, const void* V, int dtype, int Hkv, int T,
                         int64_t stride_h, int64_t stride_t,
                         const float* mu, const float* cov, int Hq, int n_sink, float eps,
                         int use_vnorm, float* scores, void* workspace, size_t workspace_bytes,
                         void* stream);

/* Observation-window attention mass (the per-query form of the scorer's attention estimate; the
 * reference scores with one query per head, the mean query: kvquant/scorer.py:285-318, and has no
 * counterpart of this entry point):
 *
 *   p[h,t] = mean over the W window queries and the G heads of kv-head h of
 *            softmax_t( Q[q,w] . K[h,t] * scaling ),  t >= n_sink,
 *   causal inside the window: query w stands at position q_pos0 + w and sees keys at positions <= its own.
 *
 * K: [Hkv, T, 128] float16 or bfloat16 (strides as for odmkv_score); Q: [Hq, W, 128] of the same type,
 * contiguous, already rotated to their positions (post-RoPE); q_pos0 >= n_sink.  p: device fp32
 * [Hkv, T - n_sink] out; it can be handed to odmkv_score as `attn` over the core tokens.  Runs on the
 * 16-bit matrix cores, two passes over K, logits are not stored.
 */
size_t odmkv_window_attention_workspace_bytes(int Hkv, int Hq, int W, int T);
int odmkv_window_attention(const void* K, int dtype, int Hkv, int T, int64_t stride_h, int64_t stride_t,
                           const void* Q, int Hq, int W, int q_pos0, int n_sink, float scaling,
                           float* p, void* workspace, size_t workspace_bytes, void* stream);
/* The same, and |k|^2 of the core tokens, fp32 [Hkv, T - n_sink], which the first pass over K leaves by the way. */
int odmkv_window_attention_norms(const void* K, int dtype, int Hkv, int T, int64_t stride_h, int64_t stride_t,
                                 const void* Q, int Hq, int W, int q_pos0, int n_sink, float scaling,
                                 float* p, float* kn2, void* workspace, size_t workspace_bytes, void* stream);
/* odmkv_score with attention weights attn [Hkv, T] (n_sink 0) where |k|^2 [Hkv, T] is known: K is not read.  Workspace:
 * odmkv_score_workspace_bytes(Hkv, Hkv, T). */
int odmkv_score_given(const void* K, const void* V, int dtype, int Hkv, int T, int64_t stride_h, int64_t stride_t,
                      const float* attn, const float* kn2, float eps, float* scores, void* workspace, size_t workspace_bytes,
                      void* stream);

/* ---------------------------------------------------------------------------------------------
 * Allocator.  Replaces optimal_scores_to_bits (kvquant/allocator.py:459-663) for a batch of
 * independent rows (one row = one (layer, sequence): the flattened [Hkv, T] scores).
 *
 * scores: device fp32 [rows, n].  sink_mask: device uint8 [rows, n] (non-zero = sink, gets
 * sink_bits and is left out of the budget) or NULL, in which case token i of a row is a sink
 * iff (i % period) < n_sink.  levels: n_levels ascending bit widths (host).  eps: host fp64
 * table, eps[k] for levels[k], already multiplied by eviction_cost / blended for
 * above_target_alpha as the reference does on the host (allocator.py:549-569).
 * target: device fp64 [rows], one budget per row (clamped into the level range on the device).
 * bits_out: device int32 [rows, n].
 * level_counts: device int32 [rows, n_levels] count of non-sink tokens per level, or NULL.
 * lambda_out: device fp64 [rows] the multiplier found, or NULL.
 * The workspace is about 6 bytes a score (5 of them the list of undecided scores, 1 the repair's candidates) and 4 KB a row, for
 * the first 2048 rows at most: a call of more rows runs in turns.
 */
size_t odmkv_allocate_workspace_bytes(int rows, int n);
int odmkv_allocate(const float* scores, int rows, int n,
                   const uint8_t* sink_mask, int period, int n_sink, int sink_bits,
                   const int32_t* levels, int n_levels, const double* eps,
                   const double* target,
                   int32_t* bits_out, int32_t* level_counts, double* lambda_out,
                   void* workspace, size_t workspace_bytes, void* stream);

/* ---------------------------------------------------------------------------------------------
 * Packed mixed-width KV store.  Replaces the banks of TurboQuantAdaptiveKVCacheState
 * (kvquant/tq_adaptive_backend.py:74-243, 346-374) with TurboQuantMSE.quantize / _pack_indices
 * (kvquant/tq_backend.py:185-197, 103-125) as the quantiser.
 *
 * Tokens of one (sequence b, kv-head h) stored at one bit level form a segment; a segment is a
 * whole number of 64-token tiles, tokens in ascending position ("slot" s = 0..63 of a tile), the tail
 * of the last tile padded (pos = -1, norm = 0).  Level index li = 0..3 means 2, 3, 4, 8 bits; "exact"
 * tokens (16 bits) are fp16/bf16 rows.  The code and row buffers of a tile are laid out for the
 * 16x16x32 matrix instructions of the decode kernel: every buffer is C chunks of 16 bytes per lane
 * l = 0..63 (C = w for codes of width w, C = 16 for exact rows), chunk c of lane l at byte
 * (c*64 + l)*16 of the tile, and with l = 16*j + n the lane's 16*C bytes hold
 *   K codes:  128 codes as one little-endian bit stream (code i at bits [i*w, i*w + w));
 *             code 32*b + i  is dim 32*j + i  of slot key_slot(n, b)    (b = 0..3, i = 0..31),
 *             key_slot(n, b) = 32*(b>>1) + 8*(n>>2) + 2*(n&3) + (b&1): the bytes of blocks 0, 1 hold slots 0..31
 *   V codes:  128 codes likewise; code 64*k + 8*m + e  is slot 32*k + 8*j + e  of dim 16*m + n
 *                                                                        (k = 0..1, m = 0..7, e = 0..7)
 *   exact K:  chunk 4*b + k  = the 8 elements  dims 32*j + 8*k .. + 7  of slot key_slot(n, b)
 *   exact V:  chunk 8*k + m  = the 8 elements  slots 32*k + 8*j .. + 7 of dim 16*m + n
 *   norms fp32 [64], pos int32 [64] per tile, in slot order.
 */
typedef struct odmkv_packed {
    int32_t B, Hkv;                      /* segments are indexed bh = b*Hkv + h */
    int32_t exact_dtype;                 /* ODMKV_F16 or ODMKV_BF16 */
    int32_t n_tiles[ODMKV_NQ + 1];       /* tiles allocated per level; index 4 = exact */
    uint8_t* kcodes[ODMKV_NQ];           /* device, n_tiles[li] * 1024*w bytes */
    uint8_t* vcodes[ODMKV_NQ];           /* device, n_tiles[li] * 1024*w bytes */
    float*   knorm[ODMKV_NQ];            /* device, n_tiles[li] * 64 */
    float*   vnorm[ODMKV_NQ];
    int32_t* pos[ODMKV_NQ + 1];          /* device, n_tiles * 64 token positions, -1 = padding */
    int32_t* seg_tile[ODMKV_NQ + 1];     /* device [B*Hkv + 1] first tile of each segment */
    int32_t* seg_count[ODMKV_NQ + 1];    /* device [B*Hkv] tokens stored in each segment */
    uint16_t* kexact;                    /* device, n_tiles[4] * 64*128 elements */
    uint16_t* vexact;
} odmkv_packed_t;

/* Count tokens per (b, h, level): bits is device int32 [B, Hkv, T] with values in
 * {0, 2, 3, 4, 8, 16}; counts is device int32 [B*Hkv, 6] in the order 0, 2, 3, 4, 8, 16.
 * (The per-level mask / nonzero of tq_adaptive_backend.py:355-361.) */
int odmkv_level_counts(const int32_t* bits, int B, int Hkv, int T, int32_t* counts, void* stream);

/* A layer's levels between the allocation and the store, in one pass over bits (device int32 [rows, T];
 * rows = B*Hkv): the tokens from tail_begin on are set to 16 bits (in bits too), the levels are written down as bytes
 * (device uint8 [rows, stride], T levels followed by 16s: what the store's level map reads behind the last token), and
 * they are counted: counts int32 [rows, odmkv_finish_levels_chunks(stride), 2, 6], device memory or page-locked host
 * memory, holds for every chunk of 4096 tokens the tokens of [count_begin, count_end) per level as they came (evicted, 2, 3,
 * 4, 8, 16 bits) and all tokens as they are stored; a value that is no level is counted nowhere.  (The reference counts the
 * prefill's level shares and sets the window in tensor operations: kvquant/adaptive_backend_press.py:292-325.) */
int odmkv_finish_levels_chunks(int64_t stride);
int odmkv_finish_levels(int32_t* bits, int rows, int T, int count_begin, int count_end, int tail_begin,
                        uint8_t* levels, int64_t stride, int32_t* counts, void* stream);

/* The evicted (0-bit) positions of a level map (device uint8 [B*Hkv, stride], T levels per row) in the order (sequence,
 * head, token): out device int64 [3, n], n the caller's own count of them (masked_key_indices,
 * kvquant/tq_adaptive_backend.py:499-505).  workspace: odmkv_evicted_workspace_bytes. */
size_t odmkv_evicted_workspace_bytes(int B, int Hkv, int T);
int odmkv_evicted_indices(const uint8_t* levels, int B, int Hkv, int T, int64_t stride, int64_t n, int64_t* out,
                          void* workspace, size_t workspace_bytes, void* stream);
/* The same for `layers` level maps one behind the other ([layers, B*Hkv, stride]) in one pass: n host int64 [layers], out the
 * layers' [3, n] lists one behind the other. */
size_t odmkv_evicted_layers_workspace_bytes(int layers, int B, int Hkv, int T);
int odmkv_evicted_indices_layers(const uint8_t* levels, int layers, int B, int Hkv, int T, int64_t stride, const int64_t* n,
                                 int64_t* out, void* workspace, size_t workspace_bytes, void* stream);

/* Host arithmetic for callers that keep a store in ONE device allocation: where its 33 buffers lie, given the
 * segments' first tiles (seg_tile: host int32 [5][nseg + 1], the last entry of a row = tiles of the level).
 * Order: seg_tile[5], seg_count[5], (knorm, vnorm)[4], kexact, vexact, pos[5], (kcodes, vcodes)[4]; offsets and
 * sizes in bytes (host uint64 [33] each), every buffer on a multiple of 256; marks (host uint64 [5]): end of the
 * tables, of the counts, of what odmkv_store_init clears, of the positions, and the bytes in all.
 * odmkv_store_bind fills the descriptor over such an allocation.  (The reference keeps a Python object per
 * bank with a tensor per field: kvquant/tq_adaptive_backend.py:31-44, 75-98.) */
int odmkv_store_layout(const int32_t* seg_tile, int nseg, uint64_t* offsets, uint64_t* sizes, uint64_t* marks);
int odmkv_store_bind(void* arena, const uint64_t* offsets, const int32_t* seg_tile, int nseg, int B, int Hkv,
                     int exact_dtype, odmkv_packed_t* out);

/* Prepare a store's buffers, laid out by the caller inside one device allocation `arena` (16-byte
 * aligned), in one launch: the five seg_tile tables (tables_host: host int32 [5][words_per_table], table
 * li written at byte table_offsets[li] of the arena), bytes [zero_begin, zero_end) cleared (segment
 * counts, norms, exact rows) and bytes [zero_end, fill_end) set to 0xff (positions: int32 -1).  Offsets
 * are multiples of 16.  It stands for the empty banks the reference starts from (ExactBank / QuantizedBank
 * __post_init__, kvquant/tq_adaptive_backend.py:39-40, 97-98), for the packed layout. */
int odmkv_store_init(void* arena, const int32_t* tables_host, int n_tables, int words_per_table,
                     const uint64_t* table_offsets, uint64_t zero_begin, uint64_t zero_end, uint64_t fill_end,
                     void* stream);

/* Move what a staging store holds into `store`: for every level and segment the tiles that hold tokens
 * (codes, norms, positions, exact rows), and the segment counts.  A staging store is a store whose
 * segments are laid out for the worst case (every token of a call at every level), so that
 * odmkv_quant_pack can fill it before the host has read the level counts back; `store` is laid out for
 * the counts, prepared by odmkv_store_init and still empty.  No counterpart in the reference, whose
 * banks grow by torch.cat (kvquant/tq_adaptive_backend.py:46-52, 149-174). */
int odmkv_store_gather(const odmkv_packed_t* staging, const odmkv_packed_t* store, void* stream);

/* The other half of a staged first fill, in one call, once counts_event has arrived: the chunk counts (host memory,
 * as odmkv_quant_pack_staged delivered them) are added up into counts (host int32 [B*Hkv, 6]); every segment gets a
 * tile per 64 tokens, the exact segments `exact_slack` tokens of room to grow and, if `quant_headroom` is not 0, every
 * quantised segment a sixteenth more tiles (two at least) for the tokens that decode-time flushes add, so that the
 * first of them need not move the store (seg_tile: host int32 [5][B*Hkv + 1], written); the store is laid out in `arena` (offsets, sizes, marks as odmkv_store_layout gives them), prepared
 * (odmkv_store_init), described (odmkv_store_bind into `store`) and filled from the staging store
 * (odmkv_store_gather).  need_bytes receives the size of the layout; if `arena` is NULL or smaller, nothing is
 * launched and ODMKV_ENOSPACE returned: allocate and call again.  `staging` may be NULL: the store is laid out and prepared
 * and stays empty (for callers that know the counts and quantise straight into it).  Counts that do not add up to B*Hkv*T (a value that
 * is no level) give ODMKV_EINVAL.  No counterpart in the reference. */
int odmkv_store_finish_staged(const int32_t* chunk_counts, int n_chunks, int B, int Hkv, int T,
                              int exact_slack, int quant_headroom, int exact_dtype, void* arena, uint64_t arena_bytes,
                              const odmkv_packed_t* staging, int32_t* counts, int32_t* seg_tile,
                              uint64_t* offsets, uint64_t* sizes, uint64_t* marks,
                              odmkv_packed_t* store, uint64_t* need_bytes, void* stream);

/* The part of a store's first fill that does not depend on the level counts, in one call: the staging store emptied
 * (its tables as odmkv_store_layout gave them: staging_tables_host, staging_offsets, tables_end, counts_end), then
 * odmkv_quant_pack into it, whose first kernel counts the levels of every 2048-token chunk anyway: those counts go to
 * counts_dev (device int32 [B*Hkv, odmkv_pack_count_chunks(T), 6]: evicted, then 2, 3, 4, 8, 16 bits; a value that is
 * no level is counted nowhere) and from there, asynchronously, to counts_host (page-locked host memory of the same
 * size), with counts_event (a hipEvent_t) recorded behind the copy.  The caller waits for the event alone, adds up the
 * chunks, lays out the store proper and calls odmkv_store_gather.  No counterpart in the reference. */
int odmkv_pack_count_chunks(int T);
int odmkv_quant_pack_staged(const void* K, const void* V, int dtype, int B, int Hkv, int T,
                            int64_t stride_b, int64_t stride_h, int64_t stride_t,
                            const int32_t* bits, int pos_offset,
                            const float* pi_k, const float* pi_v, const float* codebooks,
                            const odmkv_packed_t* staging, void* staging_arena, const int32_t* staging_tables_host,
                            const uint64_t* staging_offsets, uint64_t tables_end, uint64_t counts_end,
                            int32_t* counts_dev, int32_t* counts_host, void* counts_event,
                            void* workspace, size_t workspace_bytes, void* stream);

/* Quantise and pack T new tokens per (b, h) into a store whose seg_tile tables are filled in
 * and whose seg_count hold the tokens already present (0 after a reset); new tokens are
 * appended behind them and seg_count is advanced.  K, V: [B, Hkv, T, 128] of `dtype` with
 * element strides (stride_b, stride_h, stride_t).  bits: device int32 [B, Hkv, T].
 * pos_offset is added to the token index to form the stored position.
 * pi_k, pi_v: device fp32 [128,128] row-major rotations; codebooks: device fp32, the 4+8+16+256
 * centroids of widths 2, 3, 4, 8 back to back.
 * The arithmetic per token is, in this order and in fp32:
 *   ss = fma(x_j, x_j, ss) j=0..127; norm = sqrt(ss); u_j = x_j / (norm + 1e-10);
 *   y_i = fma(u_j, Pi[i][j], y_i) j=0..127; code_i = nearer of the two centroids bracketing y_i
 *   (lower index on a tie).
 * fp16 and bf16 tensors take a shorter route to the same bytes (widths 2, 3, 4): y_i is first estimated on
 * the 16-bit matrix cores, and only values next to a decision threshold are recomputed by the chain above.
 * The workspace (odmkv_pack_workspace_bytes(B, Hkv, T) bytes, device) holds per-call scratch only. */
size_t odmkv_pack_workspace_bytes(int B, int Hkv, int T);
int odmkv_quant_pack(const void* K, const void* V, int dtype, int B, int Hkv, int T,
                     int64_t stride_b, int64_t stride_h, int64_t stride_t,
                     const int32_t* bits, int pos_offset,
                     const float* pi_k, const float* pi_v, const float* codebooks,
                     const odmkv_packed_t* store, void* workspace, size_t workspace_bytes,
                     void* stream);

/* Lloyd-Max codebook of 2 <= k <= 256 levels for the coordinate density of a randomly rotated unit vector in
 * d >= 100 dimensions, N(0, 1/d): the reference's offline routine (codebook.py:75-113 compute_codebook with
 * :36-72 lloyd_max_iteration: 10 000 grid points over +-x_range / sqrt(d), at most n_iter rounds, stop when no
 * centroid moves by tol) run by one workgroup in fp64.  centroids: device fp64 [k], ascending; rounds: device
 * int (rounds run) or NULL.  Agrees with the host routine to about 1e-16 relative (only the order inside a
 * cell's sums differs), i.e. gives the same fp32 tables. */
int odmkv_lloyd_max(int k, int d, int n_iter, double tol, double x_range, double* centroids, int* rounds,
                    void* stream);

/* Row-wise quantiser without the packed store: x [N, 128] of `dtype` with element stride
 * `stride_n` -> codes uint8 [N, 128] (one code per byte) and norms fp32 [N], same arithmetic as
 * odmkv_quant_pack.  `bits` is 2, 3, 4 or 8; cb the 2^bits centroids (device).  This is
 * TurboQuantMSE.quantize before _pack_indices (kvquant/tq_backend.py:185-196). */
int odmkv_quantize_rows(const void* x, int dtype, int64_t N, int64_t stride_n, int bits,
                        const float* pi, const float* cb, uint8_t* codes, float* norms, void* stream);

/* out[n] = (cb[codes[n]] @ Pi) * norms[n], fp32 [N, 128] (TurboQuantMSE.dequantize,
 * kvquant/tq_backend.py:199-203). */
int odmkv_dequantize_rows(const uint8_t* codes, const float* norms, int64_t N, int bits,
                          const float* pi, const float* cb, float* out, void* stream);

/* The same with the codes in the reference's container bytes (_pack_indices, kvquant/tq_backend.py:103-125: 2-bit codes four
 * to a byte, 3- and 4-bit codes two to a byte, 8-bit codes as they are). */
int odmkv_quantize_rows_packed(const void* x, int dtype, int64_t N, int64_t stride_n, int bits,
                               const float* pi, const float* cb, uint8_t* indices, float* norms, void* stream);
int odmkv_dequantize_rows_packed(const uint8_t* indices, const float* norms, int64_t N, int bits,
                                 const float* pi, const float* cb, float* out, void* stream);

/* Rows of K and V quantised and dequantised in place (float16 / bfloat16): groups x group_rows rows each, row (g, t) at
 * element g * stride_group + t * stride_row of both (what the uniform-width press does to the model's cache,
 * kvquant/backend_press.py:94-148).  workspace: odmkv_round_trip_workspace_bytes(groups * group_rows) where bits_k or bits_v
 * is 8; the narrower widths need none (workspace may be NULL).  No two rows may share memory. */
size_t odmkv_round_trip_workspace_bytes(int64_t n);
int odmkv_round_trip_rows(void* K, void* V, int dtype, int64_t groups, int64_t group_rows, int64_t stride_group,
                          int64_t stride_row, int bits_k, int bits_v, const float* pi_k, const float* pi_v,
                          const float* cb_k, const float* cb_v, void* workspace, size_t workspace_bytes, void* stream);

/* Dequantise the store into dense [B, Hkv, T, 128] tensors of `dtype` (strides as above):
 * x_hat = (centroids[code] @ Pi) * norm, cast to dtype, written at the stored positions
 * (TurboQuantMSE.dequantize, kvquant/tq_backend.py:199-203, and the scatter of
 * QuantizedBank.materialize_into, kvquant/tq_adaptive_backend.py:205-242).
 * include_exact != 0 also writes the exact tokens (ExactBank.materialize_into, :66-70);
 * positions not stored are left untouched. */
int odmkv_dequant(const odmkv_packed_t* store, void* K, void* V, int dtype, int T,
                  int64_t stride_b, int64_t stride_h, int64_t stride_t,
                  const float* pi_k, const float* pi_v, const float* codebooks,
                  int include_exact, void* stream);
/* The same for the quantised tokens at positions t_min <= t < T only (include_exact must be 0 when t_min > 0):
 * after a decode-time flush only the re-stored tokens have new values in the dense copy
 * (materialize_quantized_into, kvquant/tq_adaptive_backend.py:452-464, restricted to what changed). */
int odmkv_dequant_from(const odmkv_packed_t* store, void* K, void* V, int dtype, int t_min, int T,
                       int64_t stride_b, int64_t stride_h, int64_t stride_t,
                       const float* pi_k, const float* pi_v, const float* codebooks,
                       int include_exact, void* stream);


/* Append one fp16/bf16 token per (b, h) to the exact segments (append_all_exact,
 * kvquant/tq_adaptive_backend.py:380-425, for one decode step).  k, v: [B, Hkv, 128] of the
 * store's exact dtype with batch and head strides in elements (the same for k and v; the 128
 * values of a row are contiguous), so the newest token of a [B, Hkv, T, 128] cache is passed as
 * it lies.  Fails with ODMKV_ENOSPACE semantics on the device side by leaving seg_count
 * untouched when a segment is full; the caller sizes segments. */
int odmkv_append_exact(const odmkv_packed_t* store, const void* k, const void* v, int64_t stride_b,
                       int64_t stride_h, int pos, void* stream);
/* T tokens per (b, h) at positions pos, pos + 1, ...: k, v [B, Hkv, T, 128] with token strides of their own (a question of
 * several tokens, append_all_exact with T > 1). */
int odmkv_append_exact_rows(const odmkv_packed_t* store, const void* k, const void* v, int T, int64_t stride_b,
                            int64_t stride_h, int64_t stride_tk, int64_t stride_tv, int pos, void* stream);
/* Forget the newest n tokens of every exact segment (a flush stores them again at other levels). */
int odmkv_drop_exact_tail(const odmkv_packed_t* store, int n, void* stream);
/* Forget every token at a position >= length (truncate, kvquant/tq_adaptive_backend.py:499-541).  counts: int32
 * [5][B*Hkv], device or page-locked host memory, receives the segments' new counts. */
int odmkv_truncate(const odmkv_packed_t* store, int length, int32_t* counts, void* stream);

/* ---------------------------------------------------------------------------------------------
 * Decode-time flush of the exact token buffer on the device.  Stands where the reference scores the
 * buffered tokens with the current query and ranks them with a chain of torch operations
 * (kvquant/adaptive_backend_press.py:464-665).
 *
 * odmkv_exact_tail: the newest n_tail tokens of every exact segment as dense rows K, V [B*Hkv, n_tail, 128]
 * of the store's exact type, oldest first (get_buffer_tokens, kvquant/tq_adaptive_backend.py:466-497, when
 * every head buffers the same positions).  A segment holding fewer tokens yields zero rows in front.
 *
 * odmkv_flush_score: per (sequence, kv-head) bh, with its n buffered rows K, V [BH, n, 128] of `dtype` and one
 * query q fp32 [BH, 128] (the GQA group's mean query at the last position, post-RoPE):
 *   a_t = softmax_t(q . k_t * scaling)                                  (_flush_attention, :602-665)
 *   mode 0: s_t = (a_t + eps)^2 * (|v_t|^2 + |k_t|^2/128 * |v_t - o|^2), o = sum_t a_t v_t / max(sum a, 1e-8)
 *           (RiskScorer.score_with_attn, kvquant/scorer.py:406-416);  mode 1: s_t = a_t^2 |v_t|^2 (no scorer).
 * attn (fp32 [BH, n], may be NULL), scores fp32 [BH, n], minmax fp32 [BH, 2] (min and max score of each bh).
 * n <= 2048.  Arithmetic in fp32 on the 16-bit inputs.
 *
 * odmkv_flush_rank: scores [B, H, n] are min-max normalised over the whole flush as the press does
 * ((x - lo) / max(hi - lo, 1e-30); 0.5 everywhere when hi - lo <= 1e-8; lo, hi from minmax), then each
 * kv-head's B*n tokens (sequence after sequence) are sorted ascending, equal values in index order, and the token
 * of rank r gets by_rank[h][r] (device int32 [H, B*n]: the head's level shares cached at prefill, expanded to
 * levels by rank on the host, _allocate_bits_via_cached_ratios :198-241).  bits: device int32 [B, H, n] out.
 * B*n <= 4096. */
int odmkv_exact_tail(const odmkv_packed_t* store, int n_tail, void* K, void* V, void* stream);
int odmkv_flush_score(const void* K, const void* V, int dtype, int BH, int n, const float* q, float scaling,
                      float eps, int mode, float* attn, float* scores, float* minmax, void* stream);
int odmkv_flush_rank(const float* scores, const float* minmax, int B, int H, int n, const int32_t* by_rank,
                     int32_t* bits, void* stream);

/* ---------------------------------------------------------------------------------------------
 * Fused LUT decode attention over the packed store: one query token per sequence.
 * Stands where the reference runs the HF attention function over the re-materialised fp16
 * cache (kvquant/attention_patch.py:30-55 on the tensors of tq_adaptive_backend.py:439-464):
 *   out[b,q] = sum_t softmax_t( scaling * q[b,q] . Khat[b,q/G,t] ) Vhat[b,q/G,t]
 * over the stored (non-evicted) tokens.  Evicted tokens are simply absent.
 *
 * q: device [B, Hq, 128] of q_dtype (ODMKV_F16 / ODMKV_BF16 / ODMKV_F32), contiguous and 16-byte
 * aligned: the model's query states are passed as they are.  work: the work list (below), built by the caller once per
 * change of the store.
 * out: device [B, Hq, 128] of out_dtype (accumulated in fp32, rounded once on the store);
 * lse: device fp32 [B, Hq] or NULL (log-sum-exp of the scaled logits).
 * pi_k_ops is the key rotation as the operand table odmkv_rotation_operands writes (the kernel rotates the query on the
 * matrix cores: q' = Pi_k q, keys are never un-rotated), pi_v the value rotation as is (row-major fp32 [128,128]).
 * The query is rounded to fp16 on entry (the attention being replaced receives it in the model's
 * fp16/bf16); bf16 and fp32 values beyond fp16's range saturate at +-65504.  The centroid tables live in
 * LDS as fp16; to keep their rounding out of the result,
 * `codebooks` here holds the centroids of each width times a per-width scale chosen on the host
 * so that the scaled values are (nearly) exact in fp16, codebooks_host a host copy of the same 284
 * floats (the small tables travel as kernel arguments), and inv_scales (host, 4 floats) the
 * reciprocals of those scales.  Exact rows are multiplied in their own type (fp16, or bf16 with the
 * query and the softmax weights split into two bf16 pieces each): nothing is narrowed.
 *
 * Work list.  items: device int32 [n_items, 8], sorted by bh: (bh, level index 0..4, first tile,
 * tile count, tokens held by those tiles, first tile of the segment, items that follow in the same workgroup,
 * 1 if the item belongs to an earlier item's workgroup: 0 and 0 without n_workgroups); for the exact level
 * (index 4) the token count is read from seg_count instead, so that tokens appended since the list
 * was built are seen.  item_range: device int32 [B*Hkv + 1] first item of each bh (any number of
 * items per bh; one item per compute unit is what performs best; a bh without items gets zeros and
 * lse = -inf).  One workgroup of the main kernel runs one item.
 * dispatch_order: NULL (workgroup k takes item k), or device int32 [n_items], a permutation of the
 * items in the order the workgroups should take them (longest first, when there are more items than
 * compute units).
 * wavefronts: wavefronts of the workgroup that runs an item: 8 (0 means 8), 12, or 16 (runs as 12).  Eight start and finish
 * faster and suit short items of 3 bits and wider; twelve stream long items, and short ones of 2 bits, 2 to 12 % faster.
 * Two launches per call (main kernel, merge); the workspace holds the per-item partial results.
 */
typedef struct odmkv_worklist {
    const int32_t* items;            /* device [n_items, 8] */
    const int32_t* item_range;       /* device [B*Hkv + 1] */
    const int32_t* dispatch_order;   /* device [n_items] or NULL */
    int32_t n_items;
    int32_t wavefronts;              /* 0, 8, 12 or 16 */
    int32_t n_workgroups;            /* 0 or n_items: a workgroup per item.  Fewer: workgroup k starts at item
                                      * dispatch_order[k] and also takes the items[.][6] items behind it (further quantised
                                      * levels of the same (sequence, kv-head): one query rotation, one result); those
                                      * items carry items[.][7] = 1 */
    int32_t two_per_cu;              /* 1: the workgroups (eight wavefronts; needs dispatch_order) are the build that keeps to
                                      * 128 registers a wavefront and half a compute unit's LDS, so that two of them share a
                                      * compute unit and one streams while the other starts or finishes: for lists with more
                                      * items than compute units (a batch of sequences, many levels).  0: one per compute unit */
    int32_t covers_exact;            /* 1: the exact items cover every tile the exact segments have room in (as
                                      * odmkv_worklist_cut makes them): a decode step's new token is then stored by the workgroup
                                      * that attends over its tile.  0: by a launch of its own */
} odmkv_worklist_t;

/* Cut the work list of a store on the host: every (segment, level) run of tiles into items of about equal cost (what the
 * kernel was measured to need per tile of each level, plus a fixed part per item).  counts: host int64 [5][nseg] tokens per
 * level and segment; seg_tile: host int64 [5][nseg + 1]; n_cu: compute units.  target_items > 0: the coarsest cut with at
 * most that many items; 0: a few cuts are compared by the time a longest-first assignment of their items to the compute
 * units would take, and `choice` keeps the winner, which is cut again without a comparison until the store has grown by
 * 5 %.  A list with more items than compute units is cut for two eight-wavefront workgroups per compute unit, as chains
 * of a pair's levels where the runs alone are many more than those places.  chains, pairs: -1 by these rules, 0 never,
 * 1 always; waves: 0 by the items' length and widths, or 8, 12, 16.
 * table (host int32, `capacity` integers) receives the items, the ranges at shape->range_at and, where shape->ordered, the
 * dispatch order at shape->order_at; too small a table gives ODMKV_ENOSPACE with shape->need set, a list that does not
 * fit host memory ODMKV_ENOMEM.  No counterpart in the
 * reference. */
typedef struct odmkv_worklist_choice {
    double multiple;                 /* items (or workgroups) per compute unit of the winning cut */
    int64_t total_bytes;             /* packed bytes it was chosen at */
    int32_t valid, chained, paired;
} odmkv_worklist_choice_t;
typedef struct odmkv_worklist_shape {
    uint64_t need, range_at, order_at;               /* in integers of the table */
    int32_t n_items, ordered, n_workgroups, two_per_cu, wavefronts;
} odmkv_worklist_shape_t;
int odmkv_worklist_cut(const int64_t* counts, const int64_t* seg_tile, int nseg, int n_cu, int64_t target_items,
                       int64_t min_item_bytes, int chains, int pairs, int waves, odmkv_worklist_choice_t* choice,
                       int32_t* table, uint64_t capacity, odmkv_worklist_shape_t* shape);

size_t odmkv_decode_workspace_bytes(int B, int Hq, int n_items);
/* The key rotation (random_rotation, kvquant/tq_backend.py:25-36, as TurboQuantMSE.dequantize applies it,
 * tq_backend.py:199-203) in the form the decode kernel multiplies the query by: pi_k device fp32 row-major [128,128];
 * ops device uint16 [32768] (64 KB): block (rb, kk, part), rb < 8, kk < 4, part < 2, at ((rb*4 + kk)*2 + part) * 512
 * elements, holds for lane l = 16 j + n its 8 fp16 values e < 8 of row 16 rb + n, columns 32 kk + 8 j + e: part 0 = the
 * entries rounded to fp16, part 1 = 4096 times what the rounding left, as fp16.  Once per rotation (per layer). */
int odmkv_rotation_operands(const float* pi_k, uint16_t* ops, void* stream);
int odmkv_decode_attn(const void* q, int q_dtype, int B, int Hq, float scaling,
                      const odmkv_packed_t* store, const odmkv_worklist_t* work,
                      const uint16_t* pi_k_ops, const float* pi_v, const float* codebooks,
                      const float* codebooks_host, const float* inv_scales,
                      void* out, int out_dtype, float* lse, void* workspace, size_t workspace_bytes,
                      void* stream);

/* One decode step of a layer in one call, for a serving loop whose host time per layer matters: the step's new token
 * of every (sequence, kv-head) is stored exact behind the others (odmkv_append_exact: k_new, v_new, strides, pos as
 * there, a full segment's count stays; both NULL = the store already holds it), then odmkv_decode_attn runs for the step's query over the store, the
 * new token included.  Stands where the reference's forward hook appends the token to its state and the model then
 * attends over the re-materialised cache (kvquant/adaptive_backend_press.py:221-262; append_all_exact,
 * kvquant/tq_adaptive_backend.py:412-440).  What does not change from step to step sits in a block the caller fills
 * once per store and work list (the pointers in it are those of odmkv_decode_attn and must stay valid); q, out and lse
 * as in odmkv_decode_attn.  Two launches on `stream` (three where the work list does not cover the exact segments). */
typedef struct odmkv_step {
    const odmkv_packed_t* store;
    const odmkv_worklist_t* work;
    const uint16_t* pi_k_ops;
    const float* pi_v;
    const float* codebooks;
    const float* codebooks_host;
    const float* inv_scales;
    void* workspace;
    size_t workspace_bytes;
    int32_t B, Hq;
    int32_t q_dtype, out_dtype;
    float scaling;
} odmkv_step_t;
int odmkv_decode_step(const odmkv_step_t* step, const void* q, const void* k_new, const void* v_new,
                      int64_t stride_b, int64_t stride_h, int pos, void* out, float* lse, void* stream);

/* A block of L query tokens per sequence that all see the whole store (the question after a prefill): q [B, Hq, L, 128] with
 * element strides, out fp32 [B, Hq, L, 128] and lse fp32 [B, Hq, L] contiguous.  The L tokens of a kv-head's G query heads
 * are handed over as further heads of it, 8 / G tokens per pass over the store, the passes in one launch.  step: as for
 * odmkv_decode_step (out_dtype is not looked at); its workspace: odmkv_decode_block_workspace_bytes. */
size_t odmkv_decode_block_workspace_bytes(int B, int Hq, int Hkv, int L, int n_items);
int odmkv_decode_block(const odmkv_step_t* step, const void* q, int64_t stride_b, int64_t stride_h, int64_t stride_l,
                       int L, float* out, float* lse, void* stream);
/* The rest of such a block's attention: every token over the block's own tokens k, v [B, Hkv, L, 128] (kv_dtype) up to its
 * position, or where mask (uint8 [B, L, L] with strides mask_sb, mask_sl; NULL: causal) is not 0, merged by log-sum-exp
 * with the store's part (out_store, lse_store as odmkv_decode_block left them); out [B, L, Hq, 128] of q_dtype.
 * (kvquant/attention_patch.py:38-48 runs such a call over the re-materialised cache.) */
int odmkv_block_merge(const void* q, int q_dtype, int64_t q_sb, int64_t q_sh, int64_t q_sl, const void* k, int64_t k_sb,
                      int64_t k_sh, int64_t k_sl, const void* v, int64_t v_sb, int64_t v_sh, int64_t v_sl, int kv_dtype,
                      const uint8_t* mask, int64_t mask_sb, int64_t mask_sl, int B, int Hq, int Hkv, int L, float scaling,
                      const float* out_store, const float* lse_store, void* out, void* stream);

/* odmkv_decode_attn without a workspace, for callers that cannot allocate device memory and have none
 * to hand over (code under HIP graph capture, tight serving loops, harnesses that forbid hipMalloc).
 * No counterpart in the reference.  The per-item partial results live in
 * a fixed array of ODMKV_STATIC_SCRATCH_BYTES inside the library's device image (held by every GPU
 * the library runs on until the process ends); a call whose odmkv_decode_workspace_bytes(B, Hq,
 * n_items) exceeds it fails with ODMKV_ENOSPACE and launches nothing.  The call allocates and
 * frees nothing.  All calls on one GPU share that GPU's array: calls that overlap on one GPU (two
 * streams, two threads) race; calls on one stream do not.  The first call on a device looks the
 * array's address up (no stream work); make it outside graph capture.  Everything else is
 * odmkv_decode_attn. */
#define ODMKV_STATIC_SCRATCH_BYTES (8u << 20)
int odmkv_decode_attn_static(const void* q, int q_dtype, int B, int Hq, float scaling,
                             const odmkv_packed_t* store, const odmkv_worklist_t* work,
                             const uint16_t* pi_k_ops, const float* pi_v, const float* codebooks,
                             const float* codebooks_host, const float* inv_scales,
                             void* out, int out_dtype, float* lse, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* ODMKV_H */
