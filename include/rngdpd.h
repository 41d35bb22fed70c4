/*
 * rngdpd.h -- C ABI of the MI355X (gfx950) prefill->decode KV handoff and
 * decode-attention library (librngdpd.so).
 *
 * Every entry point is `extern "C"`, takes plain pointers and sizes, and
 * returns an int status: PDK_OK (0) on success, a negative errno-style code
 * otherwise, with a message readable through pdk_last_error() on the calling
 * thread. Streams and events travel as uintptr_t (a hipStream_t / hipEvent_t
 * value; 0 is the null stream). Compute entry points enqueue work on the given
 * stream and return without synchronising the host; they allocate nothing.
 * Allocation, stream, event and IPC entry points are explicit set-up calls.
 *
 * Tensor conventions (all element types are bf16 carried as uint16 bits):
 *   prefill KV, per request   K/V [L][T][Hkv][D] with free layer and token
 *                             strides (elements); [Hkv][D] contiguous per token
 *   transport frame           [L][2][F], F = Hkv*D*S: the K frame [Hkv][D][S]
 *                             then the V frame [Hkv][S][D], columns >= P zero.
 *                             This is byte for byte the bf16 payload of the
 *                             reference's shm wire for one layer's (k, v).
 *   paged decode cache        K [L][num_blocks][Hkv][16*D]    (tiled, below)
 *                             V [L][num_blocks][Hkv][D][16]   (dim rows)
 *                             block table int32 [n_table], block j holds
 *                             tokens 16j .. 16j+15 of the request.
 *                             A K block is 16-byte units of 8 consecutive
 *                             dims of one token; token `slot` (0..15), dims
 *                             d0..d0+7 (d0 % 8 == 0) is unit
 *                               ((t*(D/32) + d0/32)*4 + (d0/8)%4)*8 + j8,
 *                             t = (slot>>2)&1, j8 = (slot>>3)*4 + (slot&3):
 *                             the order decode attention's QK tiles read, so
 *                             each of those loads covers whole 128-byte lines.
 *                             D % 32 == 0.
 *
 * Reference citations are file:line in ai-computing/rngd-pd.
 */
#ifndef RNGDPD_H
#define RNGDPD_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define PDK_OK 0
#define PDK_EHIP (-5)      /* EIO: the HIP runtime reported an error         */
#define PDK_EAGAIN (-11)   /* event or stream not complete yet               */
#define PDK_ENOMEM (-12)   /* allocation failed                              */
#define PDK_EINVAL (-22)   /* bad argument: shape, alignment, null pointer   */
#define PDK_ENOTSUP (-95)  /* shape the kernels do not implement             */

#define PDK_BLOCK_SIZE 16     /* tokens per paged cache block                  */
#define PDK_MAX_BATCH 16      /* requests per batched pack/scatter launch      */
#define PDK_IPC_HANDLE_BYTES 64

/* ---- library state ------------------------------------------------------ */

/* ABI version (major*100 + minor). */
int pdk_version(void);

/* Message of the last failing call on this thread ("" if none). */
const char* pdk_last_error(void);

/* Number of visible devices / select the calling thread's device. */
int pdk_device_count(int* out);
int pdk_set_device(int device);

/* ---- pack: prefill KV -> transport frame --------------------------------
 * Replaces the per-layer-group frame step of FullPrefillEngine.prefill_stream
 * (engines/prefill_full.py:366-384: zero-pad columns >= P to S at :378-379,
 * download at :381-382) and the bf16 encode of ser()
 * (connector/transport.py:29-37: f32 bits >> 16). The frame written here is
 * the u16 payload ser() would pickle for the same bf16 K and V.
 */
typedef struct pdk_pack_req {
  const uint16_t* src_k;   /* K of layer 0, token 0                         */
  const uint16_t* src_v;   /* V of layer 0, token 0                         */
  uint16_t* frame;         /* [L][2][Hkv*D*S]                               */
  int64_t layer_stride;    /* elements between layers (both K and V)        */
  int64_t tok_stride;      /* elements between tokens; a multiple of 8      */
  int32_t P;               /* valid tokens, 0 <= P <= S                     */
  int32_t flags;           /* 0 or PDK_PACK_NARROW                          */
} pdk_pack_req;

/* Leave the frame's zero tail unwritten: K columns >= min(64 * ceil(P / 64), S)
 * (K is written in whole 64-token tiles, zeros past P inside the last one, so
 * every K row ends on a 128-byte line) and V rows >= P. For consumers that
 * read only the first P columns (the same-GPU scatter), and for frames in
 * pinned host memory whose tail the host writes (pdk_host_zero_frame_tail). */
#define PDK_PACK_NARROW 1

/* One request: all L layers in one launch. Requires D % 64 == 0, S % 16 == 0,
 * 16-byte aligned pointers. */
int pdk_pack_kv(const uint16_t* src_k, const uint16_t* src_v,
                int64_t layer_stride, int64_t tok_stride, int n_layers, int P,
                int S, int n_kv_heads, int head_dim, uint16_t* frame,
                uintptr_t stream);

/* Up to PDK_MAX_BATCH requests of the same (L, S, Hkv, D) in one launch. */
int pdk_pack_kv_batch(const pdk_pack_req* reqs, int n_reqs, int n_layers,
                      int S, int n_kv_heads, int head_dim, uintptr_t stream);

/* ---- scatter: transport frame -> paged decode cache ----------------------
 * Replaces the decode-side placement of a delivered layer
 * (connector/rngd_kv.py:160-165), the f32->bf16 stage, lane stack and upload
 * (engines/decode_batch.py:305-351) and the in-place lane write
 * (engines/decode_batch.py:357-377). Writes blocks 0 .. ceil(P/16)-1 of the
 * request; token slots >= P inside the last block are written as zero, as
 * the reference's one-hot injection needs a zero slot
 * (connector/rngd_kv.py:155-159). A block id outside [0, num_blocks) among
 * a request's first ceil(P/16) table entries is skipped: nothing is written
 * for its 16 tokens and the call still returns 0. The Python wrappers check
 * host tables before the call; pdk_scatter_paged_batch_counted reports the
 * skipped ids of device tables without a host synchronisation.
 */
typedef struct pdk_scatter_req {
  const uint16_t* frame;   /* [L][2][Hkv*D*S]                               */
  const int32_t* table;    /* device int32 [n_table]                        */
  int32_t P;               /* tokens to place                               */
  int32_t n_table;         /* >= ceil(P/16)                                 */
} pdk_scatter_req;

int pdk_scatter_paged(const uint16_t* frame, const int32_t* block_table,
                      int n_table, int n_layers, int P, int S, int n_kv_heads,
                      int head_dim, uint16_t* cache_k, uint16_t* cache_v,
                      int64_t cache_layer_stride, int num_blocks,
                      uintptr_t stream);

int pdk_scatter_paged_batch(const pdk_scatter_req* reqs, int n_reqs,
                            int n_layers, int S, int n_kv_heads, int head_dim,
                            uint16_t* cache_k, uint16_t* cache_v,
                            int64_t cache_layer_stride, int num_blocks,
                            uintptr_t stream);

/* pdk_scatter_paged_batch that also adds to *skipped (device int32, zeroed by
 * the caller, e.g. once before a run of calls) the number of (request, block)
 * ids it skipped because they lie outside [0, num_blocks): each such id once
 * per call. Read it after the stream has passed the call (an event, or the
 * request's own fence): a nonzero count means KV was not placed. No
 * reference counterpart: the reference writes dense per-lane caches with no
 * block table (engines/decode_batch.py:357-377). */
int pdk_scatter_paged_batch_counted(const pdk_scatter_req* reqs, int n_reqs,
                                    int n_layers, int S, int n_kv_heads,
                                    int head_dim, uint16_t* cache_k,
                                    uint16_t* cache_v, int64_t cache_layer_stride,
                                    int num_blocks, int32_t* skipped,
                                    uintptr_t stream);

/* ---- gather: paged decode cache -> transport frame -----------------------
 * Inverse of the scatter (the frame is written S-wide, zero for t >= P).
 * Replaces the resident-cache export BatchDecodeEngine.download_kv
 * (engines/decode_batch.py:379-390) and ResidentSession.export_kv
 * (engines/decode_resident.py:222-225).
 */
int pdk_gather_paged(const uint16_t* cache_k, const uint16_t* cache_v,
                     int64_t cache_layer_stride, int num_blocks,
                     const int32_t* block_table, int n_table, int n_layers,
                     int P, int S, int n_kv_heads, int head_dim,
                     uint16_t* frame, uintptr_t stream);

/* ---- decode attention -----------------------------------------------------
 * GQA decode attention for one layer over the paged cache. Replaces the
 * attention slice of DecodeLayer.forward (kernels/decode_batch.py:83-85)
 * and softmax_dsl (kernels/dsl_batch.py:73-86); the fp32 reference it must
 * match is cpu_layer (kernels/decode_batch.py:151-156).
 *   q      [B][Hq][D] bf16; query head qh reads KV head qh / (Hq/Hkv)
 *   ctx    device int32 [B]: stream b attends to tokens 0 .. ctx[b]-1
 *          (the reference's slots 0..pos inclusive, pos = ctx-1)
 *   tables device int32 [B][max_blocks]. A block id outside [0, num_blocks)
 *          inside a stream's context masks that block's 16 tokens: they
 *          take no part in the softmax, as slots past the context do (a
 *          stream with no token left gets a zero output). The reference's
 *          dense per-lane cache has no block ids; this is the paged cache's
 *          counterpart of its -1e4 mask (engines/decode_batch.py:246-261).
 *   scale  multiplies q.k (1.0 when the scale is folded into q, as the
 *          reference folds 1/sqrt(D) into wq, kernels/decode_batch.py:204)
 *   max_ctx  host upper bound of ctx[] used for the launch grid (tokens
 *          past max_ctx, rounded up to the split size, are not read)
 *   workspace  scratch of pdk_decode_attn_workspace_bytes() bytes (0 means
 *          none is needed) holding the per-split partial maxima, sums and
 *          outputs when the context is split across workgroups. Every
 *          entry read is written earlier in the same call, so it needs no
 *          clearing. One workspace serves one stream at a time: calls that
 *          overlap on one workspace race.
 *   Splitting: the context is split across workgroups (splits of at least
 *          128 tokens, about 256 workgroups in all) while B * Hkv is below
 *          128, and for contexts of 1024 tokens or more above that; results
 *          agree with the unsplit path to fp32 rounding.
 *   out    [B][Hq][D] bf16
 * Requires D == 128, Hq/Hkv in {1, 2, 4, 8, 16}, max_ctx <= 16384.
 */
size_t pdk_decode_attn_workspace_bytes(int B, int n_q_heads, int max_ctx,
                                       int head_dim);

int pdk_decode_attn(const uint16_t* q, const uint16_t* cache_k,
                    const uint16_t* cache_v, int num_blocks,
                    const int32_t* block_tables, int max_blocks,
                    const int32_t* ctx_lens, int max_ctx, int B,
                    int n_q_heads, int n_kv_heads, int head_dim, float scale,
                    void* workspace, size_t workspace_bytes, uint16_t* out,
                    uintptr_t stream);

/* pdk_cache_append followed by pdk_decode_attn with the same results, bit for
 * bit: the new token's k_new and v_new [B][n_kv_heads][head_dim] (16-byte
 * aligned) go to slot ctx_lens[b] - 1 of the cache and take part in the
 * attention, also in that of other streams whose tables hold the slot's block.
 * Two streams with one and the same slot leave either's token there, and each
 * attends over its own. One launch for up to 64 streams; two for more, for more
 * than 256 (stream, KV head) pairs at contexts where two are faster, and for an
 * out that overlaps k_new or v_new. */
int pdk_decode_attn_append(const uint16_t* q, const uint16_t* k_new,
                           const uint16_t* v_new, uint16_t* cache_k,
                           uint16_t* cache_v, int num_blocks,
                           const int32_t* block_tables, int max_blocks,
                           const int32_t* ctx_lens, int max_ctx, int B,
                           int n_q_heads, int n_kv_heads, int head_dim,
                           float scale, void* workspace,
                           size_t workspace_bytes, uint16_t* out,
                           uintptr_t stream);

/* pdk_decode_attn without the workspace argument, for callers that cannot
 * allocate device memory (code under HIP graph capture, tight serving loops,
 * harnesses that forbid hipMalloc). No counterpart in the reference. The split
 * partials live in a file-scope device array of PDK_NOALLOC_SCRATCH_BYTES per
 * GPU, held until the process ends; a launch whose plan needs more than that
 * (pdk_decode_attn_workspace_bytes) is refused with PDK_ENOMEM. The call
 * allocates nothing. Every call on one GPU shares that GPU's array: calls that
 * overlap on one GPU (other streams, other threads) race and must be ordered
 * by the caller. Results are bit-identical to pdk_decode_attn's. Llama-3.1-8B
 * shapes (32 query heads over 8 KV heads) need at most about 1 MiB. */
#define PDK_NOALLOC_SCRATCH_BYTES (4u << 20)
int pdk_decode_attn_noalloc(const uint16_t* q, const uint16_t* cache_k,
                            const uint16_t* cache_v, int num_blocks,
                            const int32_t* block_tables, int max_blocks,
                            const int32_t* ctx_lens, int max_ctx, int B,
                            int n_q_heads, int n_kv_heads, int head_dim,
                            float scale, uint16_t* out, uintptr_t stream);

/* pdk_rope_cache_append_partials followed by pdk_decode_attn, in one launch:
 * q, k and v of the new token come as split-K partial sums of the q|k|v
 * projection (qkv_partials [splits][B][(n_q_heads + 2 n_kv_heads) head_dim]
 * fp32, splits in {1, 2, 4}; inv_freq fp32 [head_dim/2]). Each workgroup adds
 * the partials of its KV head's group in split order, rounds once to bf16,
 * rotates q and k (RoPE at position ctx[b]-1), uses them for the new token in
 * place of the cache's old contents, and the workgroup holding that position
 * writes the new k and v into its cache slot. Outputs and cache contents are
 * bit-identical to the two calls. Replaces the RoPE rotation, the one-hot
 * cache injection and the attention of DecodeLayer.forward
 * (kernels/decode_batch.py:69-85) as one step. Other arguments and limits as
 * pdk_decode_attn (same workspace size).
 * plan_batch (0: B; else >= B) is the batch size the launch plan (how the
 * context is split across workgroups, hence the order of the fp32 sums) is
 * chosen for. A decoder that passes the same plan_batch at every step makes
 * each stream's result independent of how many other streams share the step. */
int pdk_decode_attn_rope(const float* qkv_partials, int splits,
                         const float* inv_freq, uint16_t* cache_k,
                         uint16_t* cache_v, int num_blocks,
                         const int32_t* block_tables, int max_blocks,
                         const int32_t* ctx_lens, int max_ctx, int B,
                         int n_q_heads, int n_kv_heads, int head_dim,
                         float scale, void* workspace, size_t workspace_bytes,
                         uint16_t* out, int plan_batch, uintptr_t stream);

/* pdk_decode_attn_rope for a q|k|v projection whose input was the
 * un-normalised residual and whose weights carry the pre-attention RMSNorm's
 * gain (rms_dsl, kernels/dsl_batch.py:22-41, folded): each stream's summed
 * partials are scaled by r_b = rsqrt(sum_t ssq[b][t] / (16 n_ssq) + eps)
 * before the one rounding, ssq [B][n_ssq] fp32 holding the residual's per
 * 16-column tile sums of squares (pdk_linear_splitk_final, pdk_row_ssq). The
 * row scale is summed in a fixed order, so a stream's value does not depend
 * on B. head_dim 128. */
int pdk_decode_attn_rope_rms(const float* qkv_partials, int splits,
                             const float* ssq, int n_ssq, float eps,
                             const float* inv_freq, uint16_t* cache_k,
                             uint16_t* cache_v, int num_blocks,
                             const int32_t* block_tables, int max_blocks,
                             const int32_t* ctx_lens, int max_ctx, int B,
                             int n_q_heads, int n_kv_heads, int head_dim,
                             float scale, void* workspace, size_t workspace_bytes,
                             uint16_t* out, int plan_batch, uintptr_t stream);

/* Write one new token's k and v per stream at slot ctx[b]-1 of the paged
 * cache: the one-hot cache injection Kf = Kp + k*oh, Vf = Vp + v*oh
 * (kernels/decode_batch.py:81-82), done as a store.
 *   k_new, v_new [B][Hkv][D] bf16. */
int pdk_cache_append(const uint16_t* k_new, const uint16_t* v_new,
                     uint16_t* cache_k, uint16_t* cache_v, int num_blocks,
                     const int32_t* block_tables, int max_blocks,
                     const int32_t* ctx_lens, int B, int n_kv_heads,
                     int head_dim, uintptr_t stream);

/* ---- greedy sampling -------------------------------------------------------
 * First-maximum argmax per row of bf16 logits [B][ld] over V columns
 * (greedy_tokens, engines/decode_batch.py:162-171: torch.argmax semantics,
 * NaN counts as the maximum). out: device int32 [B]. */
int pdk_greedy_argmax(const uint16_t* logits, int B, int V, int64_t ld,
                      int32_t* out, uintptr_t stream);

/* ---- decode step: the non-GEMM operations of one Llama layer ----------------
 * The rest of the reference's DecodeLayer.forward (kernels/decode_batch.py:73-91)
 * around the attention above; the projections and the lm_head are plain GEMMs
 * for the caller's BLAS. bf16 in and out, fp32 inside. */

/* RMSNorm of B rows of H (H % 8 == 0, H <= 8192): out = x * rsqrt(mean(x^2) +
 * eps) * weight (rms_dsl, kernels/dsl_batch.py:22-41, engines/model.py:53-54).
 * With add != NULL the residual add comes first and is written back:
 * x = bf16(x + add) (zipadd_dsl, kernels/dsl_batch.py:43-53). */
int pdk_rmsnorm(uint16_t* x, const uint16_t* add, const uint16_t* weight, int B,
                int H, float eps, uint16_t* out, uintptr_t stream);

/* pdk_rmsnorm with the residual of a split-K projection (pdk_linear_splitk):
 * x = bf16(x + sum over s < splits of partials[s] [B][H]) (fp32, summed in
 * order s = 0, 1, ...), written back, then out = rmsnorm(x) * weight. The
 * residual add of the down projection folded into the next layer's norm. */
int pdk_rmsnorm_partials(uint16_t* x, const float* partials, int splits,
                         const uint16_t* weight, int B, int H, float eps,
                         uint16_t* out, uintptr_t stream);

/* RoPE at position ctx[b]-1 and the new token's cache write, from one
 * projection row per stream: qkv [B][qkv_ld] holds q (n_q_heads heads), k and
 * v (n_kv_heads each) of head_dim. Rotate-half with angle pos*inv_freq[i]
 * (inv_freq fp32 [head_dim/2]; engines/model.py:32-48,57-65, the llama3
 * scaling applied by the caller). Writes rotated q to q_out [B][n_q_heads]
 * [head_dim], and the rotated k and v into slot ctx[b]-1 of the paged cache
 * (one layer, block_tables [B][max_blocks]): the one-hot injection of
 * kernels/decode_batch.py:81-82 as a store. head_dim % 32 == 0. */
int pdk_rope_cache_append(const uint16_t* qkv, int64_t qkv_ld, uint16_t* q_out,
                          const float* inv_freq, const int32_t* ctx_lens,
                          const int32_t* block_tables, int max_blocks,
                          uint16_t* cache_k, uint16_t* cache_v, int num_blocks,
                          int B, int n_q_heads, int n_kv_heads, int head_dim,
                          uintptr_t stream);

/* The same from the split-K q|k|v projection: partials [splits][B][N] fp32
 * (pdk_linear_splitk's output, N = (n_q_heads + 2 n_kv_heads) head_dim) are
 * added in split order and rounded to bf16 once per element, the value the
 * unsplit projection writes, then RoPE and the cache write as above.
 * splits in {1, 2, 4}. */
int pdk_rope_cache_append_partials(const float* partials, int splits, int N,
                                   uint16_t* q_out, const float* inv_freq,
                                   const int32_t* ctx_lens,
                                   const int32_t* block_tables, int max_blocks,
                                   uint16_t* cache_k, uint16_t* cache_v,
                                   int num_blocks, int B, int n_q_heads,
                                   int n_kv_heads, int head_dim,
                                   uintptr_t stream);

/* The same with the folded pre-attention norm's row scale (as
 * pdk_decode_attn_rope_rms; head_dim >= 64): the two calls' outputs and cache
 * contents are bit-identical to pdk_decode_attn_rope_rms's. */
int pdk_rope_cache_append_partials_rms(const float* partials, int splits, int N,
                                       const float* ssq, int n_ssq, float eps,
                                       uint16_t* q_out, const float* inv_freq,
                                       const int32_t* ctx_lens,
                                       const int32_t* block_tables, int max_blocks,
                                       uint16_t* cache_k, uint16_t* cache_v,
                                       int num_blocks, int B, int n_q_heads,
                                       int n_kv_heads, int head_dim,
                                       uintptr_t stream);

/* ssq [B][H/16] fp32: per 16-column tile t, the sum of x[b][16t..16t+15]^2
 * (bf16 x [B][H], H % 16 == 0): the row-scale input of the folded norms when
 * no GEMM produced x (the embedding rows before the first layer). */
int pdk_row_ssq(const uint16_t* x, int B, int H, float* ssq, uintptr_t stream);

/* The decode step's embedding lookup with pdk_row_ssq fused: x [B][H] (bf16)
 * = table[tokens[b]] (table [vocab][H], the reference's embed_tokens gather of
 * engines/decode_batch.py:422-442) and ssq [B][H/16] exactly as pdk_row_ssq
 * computes it from x. tokens are int32 (tok_bytes 4) or int64 (8) on the
 * device; a token outside [0, vocab) gives a zero row. */
int pdk_embed_ssq(const uint16_t* table, int64_t vocab, const void* tokens, int tok_bytes,
                  int B, int H, uint16_t* x, float* ssq, uintptr_t stream);

/* out [B][M] = silu(g) * u for gate_up [B][2M] = [g | u] (swiglu_dsl,
 * kernels/dsl_batch.py:55-71). M % 8 == 0. */
int pdk_swiglu(const uint16_t* gate_up, int B, int M, uint16_t* out,
               uintptr_t stream);

/* ---- decode step: weight-streaming GEMMs ------------------------------------
 * The projections of the reference's DecodeLayer.forward (kernels/decode_batch.py:
 * 73-91: q/k/v, o, gate/up and down matmuls, each followed there by a bf16
 * result) and the batched lm_head (engines/decode_batch.py:162-171), for the
 * decode batch sizes where every weight is read once per step:
 *   y [B][N] = x [B][K] . w [N][K]^T (+ residual [B][N]),  1 <= B <= 64,
 * w in [out][in] layout, K % 128 == 0, N >= 1, fp32 accumulation, one
 * bf16 rounding. With residual != NULL the sum is y = residual + x.w^T
 * (zipadd_dsl, kernels/dsl_batch.py:43-53, fused); residual may alias y. */
int pdk_linear(const uint16_t* x, const uint16_t* w, int B, int K, int N,
               const uint16_t* residual, uint16_t* y, uintptr_t stream);

/* The same product split over K: partials [splits][B][N] fp32, partial s
 * holding the sum over its share of K (no rounding). For a large K with a
 * small N (the down projection, K = 14336, N = 4096) the split restores the
 * workgroup count that wide column tiles take away. 1 <= splits <= 16, K/128. */
int pdk_linear_splitk(const uint16_t* x, const uint16_t* w, int B, int K, int N,
                      int splits, float* partials, uintptr_t stream);

/* y [B][M] = silu(x . wg^T) * (x . wu^T), w_gate_up = [wg; wu] as [2M][K]
 * (the gate and up matmuls and swiglu_dsl, kernels/dsl_batch.py:55-71, in one
 * pass over the weights). M >= 1, K % 128 == 0, 1 <= B <= 64. */
int pdk_linear_swiglu(const uint16_t* x, const uint16_t* w_gate_up, int B, int K,
                      int M, uint16_t* y, uintptr_t stream);

/* The lm_head GEMM with greedy sampling fused: logits = x . w^T as in
 * pdk_linear (written to `logits` [B][N] unless it is NULL), and tokens[b] =
 * the first-maximum argmax of row b of the bf16 logits, NaN ranking first
 * (the same result as pdk_greedy_argmax on those logits; greedy_tokens,
 * engines/decode_batch.py:162-171). keys: device uint64 [B] scratch that
 * must read zero before the first call; every call leaves it zero. Calls
 * sharing one keys array must not overlap. */
int pdk_linear_argmax(const uint16_t* x, const uint16_t* w, int B, int K, int N,
                      uint16_t* logits, uint64_t* keys, int32_t* tokens,
                      uintptr_t stream);

/* Tiled weights: the four GEMMs above also take w as a tiled copy, written
 * once (at weight load) by pdk_weight_tile, in which every 16-row x 128-column
 * block is contiguous in the order the kernels' load instructions read it,
 * and the blocks are step-major (the first 128 columns of every 16-row tile,
 * then the next 128), so that the workgroups running together read one
 * region of memory. The copy holds
 * pdk_weight_tiled_elems(N, K) = ceil(N/16)*16*K bf16 (rows >= N zero):
 * element ((c*4 + kg)*16 + col)*8 + e of block (t, s), which starts at
 * (s*ceil(N/16) + t)*2048, is w[16t + col][128s + 32c + 8kg + e]. A gate|up
 * weight [2M][K] is tiled as one matrix and needs M % 16 == 0. Results are
 * bit-identical to the [out][in] entry points. No reference counterpart: the
 * reference's weights stay in their torch layout (engines/decode_batch.py:
 * 458-460); this is a load-time relayout of the same values.
 * pdk_weight_tiled_elems returns 0 for an invalid shape. */
int64_t pdk_weight_tiled_elems(int N, int K);
int pdk_weight_tile(const uint16_t* w, int N, int K, uint16_t* wt, uintptr_t stream);
int pdk_linear_tiled(const uint16_t* x, const uint16_t* wt, int B, int K, int N,
                     const uint16_t* residual, uint16_t* y, uintptr_t stream);
int pdk_linear_splitk_tiled(const uint16_t* x, const uint16_t* wt, int B, int K,
                            int N, int splits, float* partials, uintptr_t stream);
int pdk_linear_swiglu_tiled(const uint16_t* x, const uint16_t* wt_gate_up, int B,
                            int K, int M, uint16_t* y, uintptr_t stream);
int pdk_linear_argmax_tiled(const uint16_t* x, const uint16_t* wt, int B, int K,
                            int N, uint16_t* logits, uint64_t* keys,
                            int32_t* tokens, uintptr_t stream);

/* The post-attention RMSNorm folded into its neighbours (rms_dsl,
 * kernels/dsl_batch.py:22-41, between the o and gate/up matmuls of
 * kernels/decode_batch.py:73-91):
 * pdk_linear_ssq is pdk_linear with a residual (y = residual + x.w^T, residual
 *   may alias y) that also writes ssq [B][N/16] fp32: ssq[b][t] = the sum over
 *   columns 16t..16t+15 of y[b][.]^2, y as rounded to bf16. N % 16 == 0.
 * pdk_linear_swiglu_rms is pdk_linear_swiglu on the un-normalised x with the
 *   norm's gain folded into the weights (w_gate_up[n][k] = bf16(w[n][k] g[k]),
 *   made once at weight load): row b's two sums are scaled by
 *   r_b = rsqrt(sum_t ssq[b][t] / K + eps) (t in a fixed order) before silu,
 *   i.e. silu(r x.wg^T) * (r x.wu^T) = the gate/up of rmsnorm(x) g, with one
 *   bf16 rounding (of the weights' product with g) in place of the rounding of
 *   the normalised activations. n_ssq = K / 16 (the tiles of the producing
 *   pdk_linear_ssq call, with the same B). No launch between the two GEMMs. */
int pdk_linear_ssq(const uint16_t* x, const uint16_t* w, int B, int K, int N,
                   const uint16_t* residual, uint16_t* y, float* ssq, uintptr_t stream);
int pdk_linear_ssq_tiled(const uint16_t* x, const uint16_t* wt, int B, int K, int N,
                         const uint16_t* residual, uint16_t* y, float* ssq,
                         uintptr_t stream);
int pdk_linear_swiglu_rms(const uint16_t* x, const uint16_t* w_gate_up, int B, int K,
                          int M, const float* ssq, int n_ssq, float eps, uint16_t* y,
                          uintptr_t stream);
int pdk_linear_swiglu_rms_tiled(const uint16_t* x, const uint16_t* wt_gate_up, int B,
                                int K, int M, const float* ssq, int n_ssq, float eps,
                                uint16_t* y, uintptr_t stream);

/* pdk_linear_splitk on weights carrying an RMSNorm's gain, x the
 * un-normalised residual: each row's partials are scaled by its r (ssq
 * [B][K/16], as pdk_linear_swiglu_rms), so the splits' sum is the projection
 * of the normalised row (the q|k|v projection after the pre-attention norm,
 * kernels/decode_batch.py:73-80 with rms_dsl folded). */
int pdk_linear_splitk_rms(const uint16_t* x, const uint16_t* w, int B, int K, int N,
                          int splits, const float* ssq, int n_ssq, float eps,
                          float* partials, uintptr_t stream);
int pdk_linear_splitk_rms_tiled(const uint16_t* x, const uint16_t* wt, int B, int K, int N,
                                int splits, const float* ssq, int n_ssq, float eps,
                                float* partials, uintptr_t stream);

/* The down projection and the next RMSNorm's residual add in one launch:
 * pdk_linear_splitk whose last split to finish, per group of columns, adds the
 * splits' partials in split order to `residual` in place (residual =
 * bf16(residual + sum), the update pdk_rmsnorm_partials makes) and writes
 * ssq [B][N/16] as pdk_linear_ssq does. Workgroups never wait for each other:
 * each counts itself in on counters (int32, >= N/16 of them, zero before the
 * first call; every call leaves them zero) after its partials are stored, and
 * the one that completes a group finishes it. Calls sharing counters must not
 * overlap. N % 16 == 0, 1 <= splits <= 16. */
int pdk_linear_splitk_final(const uint16_t* x, const uint16_t* w, int B, int K, int N,
                            int splits, float* partials, uint16_t* residual, float* ssq,
                            int* counters, uintptr_t stream);
int pdk_linear_splitk_final_tiled(const uint16_t* x, const uint16_t* wt, int B, int K,
                                  int N, int splits, float* partials, uint16_t* residual,
                                  float* ssq, int* counters, uintptr_t stream);

/* The lm_head with greedy sampling (pdk_linear_argmax) on weights carrying
 * the final norm's gain, x the un-normalised residual: each row's logits are
 * scaled by its r (ssq [B][K/16], as pdk_linear_swiglu_rms) before the bf16
 * rounding the argmax ranks. */
int pdk_linear_argmax_rms(const uint16_t* x, const uint16_t* w, int B, int K, int N,
                          const float* ssq, int n_ssq, float eps, uint16_t* logits,
                          uint64_t* keys, int32_t* tokens, uintptr_t stream);
int pdk_linear_argmax_rms_tiled(const uint16_t* x, const uint16_t* wt, int B, int K, int N,
                                const float* ssq, int n_ssq, float eps, uint16_t* logits,
                                uint64_t* keys, int32_t* tokens, uintptr_t stream);

/* ---- decode step on tiled activations -----------------------------------------
 * The step's bf16 activations (the residual stream, attention's output and
 * SwiGLU's output) in the order the GEMMs read their MFMA operand: for an
 * operand of K columns (K % 128 == 0) and rows padded to a multiple of 16,
 * element (m, n) is at
 *   ((m/16)*(K/128) + n/128)*2048 + (((n%128)/8)*16 + m%16)*8 + n%8,
 * i.e. each 16-row x 128-column block is contiguous and, inside it, the 8
 * columns 8j..8j+7 of the 16 rows are 16 rows of 16 bytes (the weights'
 * tiling with rows and columns exchanged). Buffers hold 16 ceil(B/16) rows;
 * rows past B are never read. Each _xt entry point is its _tiled (or plain)
 * namesake with x, residual, y (and attention's out) in this layout; fp32
 * partials, logits, ssq and q|k|v partials stay row-major. Results are
 * bit-identical to the row-major entry points. No reference counterpart: a
 * relayout of the same values (engines/decode_batch.py:422-442 keeps them as
 * torch [B][H] tensors). */
int pdk_embed_ssq_xt(const uint16_t* table, int64_t vocab, const void* tokens, int tok_bytes,
                     int B, int H, uint16_t* x, float* ssq, uintptr_t stream);
int pdk_linear_splitk_rms_xt(const uint16_t* x, const uint16_t* wt, int B, int K, int N,
                             int splits, const float* ssq, int n_ssq, float eps,
                             float* partials, uintptr_t stream);
int pdk_decode_attn_rope_xt(const float* qkv_partials, int splits,
                            const float* inv_freq, uint16_t* cache_k,
                            uint16_t* cache_v, int num_blocks,
                            const int32_t* block_tables, int max_blocks,
                            const int32_t* ctx_lens, int max_ctx, int B,
                            int n_q_heads, int n_kv_heads, int head_dim,
                            float scale, void* workspace, size_t workspace_bytes,
                            uint16_t* out, int plan_batch, uintptr_t stream);
int pdk_linear_ssq_xt(const uint16_t* x, const uint16_t* wt, int B, int K, int N,
                      const uint16_t* residual, uint16_t* y, float* ssq, uintptr_t stream);
/* pdk_linear_ssq_xt's result, bit for bit, with a workspace that lets it split
 * K over workgroups: pdk_linear_ssq_ws_bytes(B, K, N) bytes (0: none needed),
 * 16-byte aligned, zeroed once before its first use and used by one stream at
 * a time; the call leaves its counters zero again. One workspace serves calls
 * of any shapes whose bytes it holds. */
int64_t pdk_linear_ssq_ws_bytes(int B, int K, int N);
int pdk_linear_ssq_ws_xt(const uint16_t* x, const uint16_t* wt, int B, int K,
                         int N, const uint16_t* residual, uint16_t* y,
                         float* ssq, void* workspace, int64_t workspace_bytes,
                         uintptr_t stream);
int pdk_linear_swiglu_rms_xt(const uint16_t* x, const uint16_t* wt_gate_up, int B, int K,
                             int M, const float* ssq, int n_ssq, float eps, uint16_t* y,
                             uintptr_t stream);
int pdk_linear_splitk_final_xt(const uint16_t* x, const uint16_t* wt, int B, int K, int N,
                               int splits, float* partials, uint16_t* residual, float* ssq,
                               int* counters, uintptr_t stream);
int pdk_linear_argmax_rms_xt(const uint16_t* x, const uint16_t* wt, int B, int K, int N,
                             const float* ssq, int n_ssq, float eps, uint16_t* logits,
                             uint64_t* keys, int32_t* tokens, uintptr_t stream);

/* ---- KONI token blocks (second frame format) --------------------------------
 * The Furiosa native connector's KV payload (native_v4/kv.py:1-20): units of
 * one token of one tensor (t = 2*layer + 0 for K, 1 for V), each [Hkv][D] bf16,
 * uploaded as received. index [n_tensors][n_tokens]: the unit of token tok of
 * tensor t in `units`, or -1 when this batch does not carry it. Writes every
 * carried token into the request's paged cache blocks (block_table, as for
 * pdk_scatter_paged): K in the tiled block order, V as [D][16]; other slots
 * are left alone. Replaces the placement of KVReceiver.accept
 * (native_v4/kv.py:100-118, 122-155), which writes host ATOM buffers.
 * Hkv * head_dim <= 1024, head_dim % 32 == 0. */
int pdk_scatter_koni(const uint16_t* units, int64_t n_units, const int32_t* index,
                     int n_tensors, int n_tokens, const int32_t* block_table,
                     int max_blocks, uint16_t* cache_k, uint16_t* cache_v,
                     int64_t layer_stride, int num_blocks, int n_kv_heads,
                     int head_dim, uintptr_t stream);

/* ---- staging and device memory ----------------------------------------------
 * Pinned host staging replaces the synchronous .cpu() download
 * (engines/prefill_full.py:381-382) and .to(dev) upload
 * (engines/decode_batch.py:343-351). Pinned memory is allocated here
 * (hipHostMalloc); existing memory is never registered. */
int pdk_host_alloc(size_t bytes, void** out);
int pdk_host_free(void* p);
int pdk_dev_alloc(size_t bytes, void** out);
int pdk_dev_free(void* p);
int pdk_memcpy_d2h(void* host_dst, const void* dev_src, size_t bytes,
                   uintptr_t stream);
int pdk_memcpy_h2d(void* dev_dst, const void* host_src, size_t bytes,
                   uintptr_t stream);
int pdk_memcpy_d2d(void* dev_dst, const void* dev_src, size_t bytes,
                   uintptr_t stream);
/* A plain streaming copy kernel (16-byte vectors; bytes % 16 == 0), used to
 * calibrate HBM traffic counters against a known byte count. */
int pdk_copy_kernel(void* dev_dst, const void* dev_src, size_t bytes,
                    uintptr_t stream);
/* Streaming probes for the HBM ceilings the handoff kernels are compared with:
 * kind PDK_STREAM_READ reads `bytes` of dev_src, PDK_STREAM_WRITE writes `key`
 * to every word of dev_dst, PDK_STREAM_COPY copies dev_src to dev_dst; 16-byte
 * vectors (bytes % 16 == 0). blocks == 0: one-shot, one vector per lane and
 * one 256-lane workgroup per 4 KiB (bytes <= 32 GiB); blocks > 0: a grid-stride
 * loop over that many 256-lane workgroups, four vectors in flight per lane.
 * PDK_STREAM_NONTEMPORAL
 * asks for streaming (non-temporal) accesses. A read folds what it loads and
 * stores into dev_sink[0..255] only where a fold equals `key` (pick a key no
 * fold is expected to take). No counterpart in the reference: measurement only. */
#define PDK_STREAM_READ 0
#define PDK_STREAM_WRITE 1
#define PDK_STREAM_COPY 2
#define PDK_STREAM_NONTEMPORAL 1
int pdk_stream_probe(int kind, void* dev_dst, const void* dev_src, size_t bytes, int flags,
                     int blocks, uint32_t key, uint32_t* dev_sink, uintptr_t stream);

/* Decode attention's reads without its arithmetic: the launch pdk_decode_attn
 * makes for the same arguments (grid, split plan, block-id reads, every K/V
 * load), with the loaded words folded into one register per lane and stored
 * into out ([B][n_q_heads][head_dim] bf16, contents meaningless). It measures
 * what a kernel with attention's access pattern costs before any compute. No
 * counterpart in the reference: measurement only. */
int pdk_attn_read_probe(const uint16_t* cache_k, const uint16_t* cache_v, int num_blocks,
                        const int32_t* block_tables, int max_blocks, const int32_t* ctx_lens,
                        int max_ctx, int B, int n_q_heads, int n_kv_heads, int head_dim,
                        uint16_t* out, uintptr_t stream);

/* ---- layer-wise staging pipeline ---------------------------------------------
 * The reference hands each layer group to the writer while the next computes
 * (engines/prefill_full.py:337-388, serving/cluster.py:187-218) and loads
 * layer by layer on the decode side (serving/cluster.py:458-459). These calls
 * enqueue all layers of one request in a native loop, chaining stages on
 * different streams through per-layer events (arrays of n_layers events made
 * by pdk_event_create; a null array means no dependency). */
#define PDK_COPY_D2H 0
#define PDK_COPY_H2D 1
#define PDK_COPY_D2D 2

/* Per layer l: one pack launch of layer l of all n_reqs requests (1..16;
 * each request's frame slice l), then done_events[l]. */
int pdk_pack_kv_layerwise(const pdk_pack_req* reqs, int n_reqs, int n_layers,
                          int S, int n_kv_heads, int head_dim,
                          const uintptr_t* done_events, uintptr_t stream);

/* n_layers copies of layer_bytes at offsets l*layer_bytes: wait
 * wait_events[l], copy, record done_events[l]. Host memory must be pinned
 * (pdk_host_alloc) for the copies to run asynchronously. */
int pdk_copy_layers(void* dst, const void* src, size_t layer_bytes,
                    int n_layers, int direction, const uintptr_t* wait_events,
                    const uintptr_t* done_events, uintptr_t stream);

/* The valid columns of frame layers [layer0, layer0 + n_layers) -- K rows'
 * columns [0, min(round16(P), S)) and V rows [0, P) -- copied by the DMA
 * engines between a device frame and a pinned host frame (dst and src are
 * frame bases, layer 0): one rectangular copy for each part in `parts`
 * (PDK_FRAME_K, PDK_FRAME_V or both); direction PDK_COPY_D2H or
 * PDK_COPY_H2D. The device->host and host->device legs of the reference's
 * download / upload (engines/prefill_full.py:378-384, engines/decode_batch.py:
 * 305-351) for the bytes that are not padding. P = 0 copies nothing. */
#define PDK_FRAME_K 1
#define PDK_FRAME_V 2
#define PDK_FRAME_KV 3
int pdk_copy_frame_valid(void* dst, const void* src, int layer0, int n_layers,
                         int n_kv_heads, int head_dim, int S, int P,
                         int direction, int parts, uintptr_t stream);

/* Host side of a pinned frame whose valid columns the device wrote: zero what
 * it left unwritten -- per layer, K rows' columns [round_k(P), S) and V rows
 * [P, S) -- with `threads` host threads (1..64), so the frame becomes the
 * S-wide wire payload while the host link carries only the valid columns.
 * k_round: 64 after a PDK_PACK_NARROW pack into the frame (whole 64-token
 * tiles of K), 16 after pdk_copy_frame_valid. Host memory only; no stream, no
 * device work. Replaces the device-side zero padding of
 * engines/prefill_full.py:378-379 for frames staged through the host. */
int pdk_host_zero_frame_tail(uint16_t* frame, int n_layers, int n_kv_heads,
                             int head_dim, int S, int P, int k_round,
                             int threads);

/* Per layer l: wait wait_events[l], then one scatter launch of frame slice l
 * of all n_reqs requests (1..16) into cache layer l. */
int pdk_scatter_paged_layerwise(const pdk_scatter_req* reqs, int n_reqs,
                                int n_layers, int S, int n_kv_heads, int head_dim,
                                uint16_t* cache_k, uint16_t* cache_v,
                                int64_t cache_layer_stride, int num_blocks,
                                const uintptr_t* wait_events,
                                uintptr_t stream);

/* ---- prefill -------------------------------------------------------------------
 * The non-GEMM part of one prompt's prefill (engines/prefill_full.py:337-388),
 * head_dim 128. table [T][half] (cos, sin) fp32 pairs of t * inv_freq[i]. */
int pdk_rope_table(const float* inv_freq, int T, int half, float* table,
                   uintptr_t stream);

/* Elements of each of the two operand buffers kt and vt below. */
int64_t pdk_prefill_kv_tile_elems(int T, int n_kv_heads);

/* qkv [T][(Hq + 2 Hkv) * 128] bf16, contiguous: q is rotated in place, the
 * rotated k and the v go to k_out and v_out ([T] rows of [Hkv][128], the given
 * token strides in elements, multiples of 8) and, as pdk_prefill_attn reads
 * them, to kt and vt. table is pdk_rope_table's with half = 64. */
int pdk_prefill_rope_kv(uint16_t* qkv, const float* table, int T, int n_q_heads,
                        int n_kv_heads, int head_dim, uint16_t* k_out,
                        int64_t k_tok_stride, uint16_t* v_out,
                        int64_t v_tok_stride, uint16_t* kt, uint16_t* vt,
                        uintptr_t stream);

/* The projections of prompts of up to 256 tokens (512 where N is small enough
 * that the library's tiles would leave the chip idle): W [N][K] bf16 as the
 * model holds it, K split over workgroups. pdk_prefill_gemm_splits: how many
 * splits T, K, N give, 0 where pdk_prefill_gemm does not take them (K % 64, N %
 * 4, K >= 256, or a shape the library is faster at). pdk_prefill_gemm writes
 * that many fp32 partial sums, partials [splits][T][N], for
 * pdk_prefill_rope_kv_partials or pdk_prefill_rmsnorm_partials.
 * pdk_prefill_gemm_swiglu (where pdk_prefill_gemm_swiglu_takes is 1): y [T][M]
 * = silu(x . Wg^T) * (x . Wu^T) from w_gate_up = [Wg; Wu] [2M][K], rounded once. */
int pdk_prefill_gemm_splits(int T, int K, int N);
int pdk_prefill_gemm(const uint16_t* x, const uint16_t* w, int T, int K, int N,
                     float* partials, uintptr_t stream);
int pdk_prefill_gemm_swiglu_takes(int T, int K, int M);
int pdk_prefill_gemm_swiglu(const uint16_t* x, const uint16_t* w_gate_up, int T,
                            int K, int M, uint16_t* y, uintptr_t stream);

/* pdk_prefill_rope_kv on the projection's partial sums (added in order, rounded
 * to bf16 once); the rotated q goes to q_out [T][Hq][128]. */
int pdk_prefill_rope_kv_partials(const float* partials, int splits,
                                 const float* table, int T, int n_q_heads,
                                 int n_kv_heads, int head_dim, uint16_t* q_out,
                                 uint16_t* k_out, int64_t k_tok_stride,
                                 uint16_t* v_out, int64_t v_tok_stride,
                                 uint16_t* kt, uint16_t* vt, uintptr_t stream);

/* pdk_rmsnorm_partials with split s at partials + s * split_stride elements (a
 * multiple of 4), so that it can take some rows of a larger projection. */
int pdk_prefill_rmsnorm_partials(uint16_t* x, const float* partials,
                                 int64_t split_stride, int splits,
                                 const uint16_t* weight, int B, int H, float eps,
                                 uint16_t* out, uintptr_t stream);

/* The greedy token of one row of logits given as partial sums [splits][1][N]
 * (pdk_prefill_gemm's at T = 1): keys[i], i < ceil(N / 1024), is the best key of
 * columns 1024 i .. (as pdk_linear_argmax's: the value in an order-preserving
 * code above the complement of the column), so the token is 0xffffffff minus the
 * low 32 bits of the largest. */
int pdk_prefill_argmax(const float* partials, int splits, int N, uint64_t* keys,
                       uintptr_t stream);

/* Causal GQA attention of the prompt: out [T][Hq][128] bf16 from q (rows of
 * q_tok_stride elements, Hq * 128 of them used) and pdk_prefill_rope_kv's kt
 * and vt. Query head h reads KV head h / (Hq / Hkv). Weights stay fp32. */
int pdk_prefill_attn(const uint16_t* q, int64_t q_tok_stride, const uint16_t* kt,
                     const uint16_t* vt, int T, int n_q_heads, int n_kv_heads,
                     int head_dim, float scale, uint16_t* out, uintptr_t stream);

/* ---- streams and events ------------------------------------------------------
 * Fences for the side-stream staging and for wait_for_save()
 * (connector/rngd_kv.py:129-131), which becomes a real barrier once saves
 * are asynchronous. Streams are created at the default priority. */
int pdk_stream_create(uintptr_t* out);
int pdk_stream_destroy(uintptr_t stream);
int pdk_stream_sync(uintptr_t stream);
#define PDK_EVENT_TIMING 0
#define PDK_EVENT_INTERPROCESS 1   /* hipEventInterprocess | DisableTiming */
#define PDK_EVENT_SYNC 2           /* hipEventDisableTiming: dependencies only */
int pdk_event_create(uintptr_t* out, int flags);
int pdk_event_destroy(uintptr_t event);
int pdk_event_record(uintptr_t event, uintptr_t stream);
int pdk_event_query(uintptr_t event);   /* PDK_OK done, PDK_EAGAIN pending */
int pdk_event_sync(uintptr_t event);
int pdk_stream_wait_event(uintptr_t stream, uintptr_t event);
int pdk_event_elapsed_ms(uintptr_t start, uintptr_t stop, float* ms);

/* ---- same-GPU inter-process handoff --------------------------------------------
 * The /dev/shm file handoff between the prefill and decode processes
 * (connector/transport.py:80-101) becomes, on one GPU, an IPC handle to the
 * producer's device frame pool plus an IPC event as the publish fence (the
 * reference's tmp+fsync+rename, :90-94). Handles are PDK_IPC_HANDLE_BYTES
 * opaque bytes. The producer owns the memory until the consumer acknowledges;
 * the consumer closes what it opened. Exported allocations must come from
 * pdk_dev_alloc and stay below 2 GiB each. */
int pdk_ipc_export_mem(const void* dev_ptr, void* handle_out);
int pdk_ipc_open_mem(const void* handle, void** dev_ptr_out);
int pdk_ipc_close_mem(void* dev_ptr);
int pdk_ipc_export_event(uintptr_t event, void* handle_out);
int pdk_ipc_open_event(const void* handle, uintptr_t* event_out);

#ifdef __cplusplus
}
#endif

#endif /* RNGDPD_H */
