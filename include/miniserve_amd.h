/*
 * miniserve_amd -- C ABI of the MI355X (gfx950) kernels for MiniServe's per-step hot path.
 *
 * Every entry point takes plain device pointers, sizes and a HIP stream (hipStream_t passed as
 * void*, NULL = the default stream), launches asynchronously on that stream, allocates nothing,
 * never synchronizes, and returns MSA_OK or an error code; msa_last_error() then holds a message.
 * bf16 tensors are passed as uint16_t bit patterns. All tensors are row-major.
 *
 * The reference is pure Python + PyTorch (no FFI of its own); each declaration names the
 * reference function (file:line, paths relative to the reference repository) whose GPU work it
 * replaces. The Python host mirror in miniserve_amd/ binds these through ctypes.
 */
#ifndef MINISERVE_AMD_H
#define MINISERVE_AMD_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef void* msa_stream_t;

enum {
  MSA_OK = 0,
  MSA_ERR_INVALID = 1,     /* bad shape, pointer, alignment or argument            */
  MSA_ERR_UNSUPPORTED = 2, /* valid but not implemented (e.g. head_dim != 128)       */
  MSA_ERR_LAUNCH = 3,      /* the HIP runtime reported an error for a launch         */
  MSA_ERR_WORKSPACE = 4    /* workspace missing or smaller than the *_workspace_size */
};

/* Message of the last failing call on the calling host thread ("" if none). */
const char* msa_last_error(void);
/* ABI version: bumped whenever a signature below changes. */
int msa_abi_version(void);

/* ---- int8 weight-only linears (quant/int8.py) ----------------------------------------------- */

/* Int8Linear.__init__ (quant/int8.py:25-33): per-row scale32 = max(max|w|, 1e-8) / 127 (IEEE
 * division), qweight = round_half_even(w / scale32) clamped to [-127, 127], scale = bf16(scale32).
 * weight_dtype: 0 = bf16, 1 = float32. weight [rows, cols], qweight [rows, cols], scale [rows]. */
int msa_int8_quantize(const void* weight, int weight_dtype, int64_t rows, int64_t cols,
                      int8_t* qweight, uint16_t* scale, msa_stream_t stream);

enum {
  MSA_EPI_NONE = 0,     /* y = bf16(x @ W^T)                                                   */
  MSA_EPI_SILU_MUL = 1, /* rows [gate | up] (layers.py:77-78): y = bf16(silu(g) * u), n/2 cols  */
  MSA_EPI_RESIDUAL = 2  /* y = bf16(residual + bf16(x @ W^T))  (model/qwen3.py:122)             */
};

/* Bytes of float32 workspace msa_int8_linear may use for this shape (0 if none). With less (or no)
 * workspace the call still succeeds, without splitting K across workgroups. */
size_t msa_int8_linear_workspace_size(int64_t m, int64_t n, int64_t k);
/* The same of msa_int8_linear_add_rmsnorm and of msa_int8_gemm_qk_norm_rope_cache (n its qkv columns). */
size_t msa_int8_linear_add_rmsnorm_workspace_size(int64_t m, int64_t n, int64_t k);
size_t msa_int8_gemm_qk_norm_rope_cache_workspace_size(int64_t m, int64_t n, int64_t k);
/* What a caller should hold for any of the three before it captures them in a graph (0 if nothing):
 * without it a call leaves much of the chip idle. The sizes above can be larger, or nonzero where this is 0;
 * a call without the difference is served by another kernel at a smaller loss. */
size_t msa_int8_linear_min_workspace_size(int64_t m, int64_t n, int64_t k);

/* Int8Linear.forward (quant/int8.py:35-37) without materializing W: y[m, :] from x [m, k] (row
 * stride ldx), qweight [n, k] int8, scale [n] bf16. Each weight is dequantized in registers to
 * bf16(q * s) -- the same value the reference's whole-matrix dequantization produces -- then
 * multiplied on bf16 MFMA tiles with float32 accumulation. k % 16 == 0; x, qweight 16-byte
 * aligned. y has n columns (n/2 for MSA_EPI_SILU_MUL) with row stride ldy; residual (row stride
 * ldr) is read only for MSA_EPI_RESIDUAL and may alias y. When K is split across workgroups the
 * splits meet in the workspace and a second kernel sums them in a fixed order (deterministic).
 * Batches of 128 or more rows with k % 64 == 0 run msa_int8_gemm (its split-K partials in the
 * workspace). Smaller ones with k in {1024, 2048, 3072, 4096} run msa_int8_linear_dec (no norm prologue),
 * those whose activation tile fits in LDS (k % 64 == 0, k <= 4544) msa_int8_linear_rows (neither uses
 * the workspace), the rest a split-K kernel. Over weights of n * k >= 12 MiB with k % 64 == 0, where it is
 * faster, 65 or more rows run the GEMM and fewer a kernel that reads the weights once for all of them
 * (with a long k in splits whose partials meet in the workspace). Without a workspace nothing is split. */
int msa_int8_linear(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                    const uint16_t* scale, int64_t n, uint16_t* y, int64_t ldy, int epilogue,
                    const uint16_t* residual, int64_t ldr, void* workspace, size_t workspace_bytes,
                    msa_stream_t stream);

/* Int8Linear.forward (quant/int8.py:35-37) for prefill-sized batches: an LDS-tiled MFMA GEMM over
 * 128-token x 128-row tiles; each int8 weight tile is dequantized once per token tile to the same
 * bf16(q * s) value as the reference, float32 accumulation, then the epilogue of msa_int8_linear
 * (MSA_EPI_RESIDUAL may write y in place over residual). k % 64 == 0; x, qweight 16-byte aligned.
 * msa_int8_linear routes batches of 128 or more rows here (65 or more over large weights, where it is faster). */
int msa_int8_gemm(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                  const uint16_t* scale, int64_t n, uint16_t* y, int64_t ldy, int epilogue,
                  const uint16_t* residual, int64_t ldr, msa_stream_t stream);

/* The split-K half of Int8Linear.forward (quant/int8.py:35-37) for callers that fuse the
 * reduction into the next kernel: partials[s][m][n] (float32, k_split * m * n elements) holds the
 * product over the s-th of k_split equal ranges of 64-aligned K chunks (ranges past k hold zeros);
 * bf16(sum over s in order) is what msa_int8_linear returns. 1 <= k_split <= ceil(k / 64). */
int msa_int8_linear_splitk(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                           const uint16_t* scale, int64_t n, int k_split, float* partials,
                           msa_stream_t stream);

/* Int8Linear.forward (quant/int8.py:35-37) for decode-sized batches, split over tokens instead of
 * K: a workgroup owns up to 16 tokens x a block of weight rows over the whole of K, so there are
 * no float32 partials. Epilogues as msa_int8_linear (MSA_EPI_RESIDUAL may write y in place over
 * residual). With MSA_EPI_SILU_MUL an RMSNorm prologue may be applied to the activations (norm_w
 * non-NULL; model/layers.py:18-22 with eps), as when gate_up consumes post_attention_layernorm
 * (model/qwen3.py:122); other epilogues take norm_w = NULL. k % 64 == 0 and
 * 16 * (k + 8) * 2 bytes + 16 KiB <= 160 KiB (k <= 4416); x, qweight, norm_w 16-byte aligned. */
int msa_int8_linear_rows(const uint16_t* x, int64_t ldx, int64_t m, int64_t k, const uint16_t* norm_w, float eps,
                         const int8_t* qweight, const uint16_t* scale, int64_t n, int epilogue, uint16_t* y,
                         int64_t ldy, const uint16_t* residual, int64_t ldr, msa_stream_t stream);

/* Int8Linear.forward (quant/int8.py:35-37) for decode-sized batches with the neighbouring ops of
 * the layer fused: activations read straight into MFMA operand registers, each workgroup owning
 * up to 32 tokens x 16-64 weight rows over the whole of K (no float32 partials). Activation rows
 * are x[gather_rows[t]] (indices clamped into [0, x_rows); the embedding lookup of
 * model/qwen3.py:148, then also copied to x_copy: the residual stream) when gather_rows is
 * non-NULL, else x[t]. norm_w non-NULL applies RMSNorm(x) first (model/layers.py:18-22 with eps;
 * the input_layernorm / post_attention_layernorm of model/qwen3.py:121-122). Rounded where the
 * reference rounds: weights dequantized to bf16(q * s), the norm as bf16(w * bf16(x * r)),
 * float32 accumulation, bf16 output. Epilogues as msa_int8_linear (MSA_EPI_RESIDUAL may write y in place over
 * residual); gather_rows takes MSA_EPI_NONE and needs norm_w. k in {1024, 2048, 3072, 4096}; x,
 * qweight, norm_w, x_copy 16-byte aligned with row strides % 8 == 0. */
int msa_int8_linear_dec(const uint16_t* x, int64_t ldx, int64_t x_rows, const int64_t* gather_rows,
                        uint16_t* x_copy, int64_t ld_copy, int64_t m, int64_t k, const uint16_t* norm_w,
                        float eps, const int8_t* qweight, const uint16_t* scale, int64_t n, int epilogue,
                        uint16_t* y, int64_t ldy, const uint16_t* residual, int64_t ldr, msa_stream_t stream);

/* The front half of Qwen3Attention.forward (model/qwen3.py:94-98) plus the cache write of
 * paged_attention (attention/backends.py:159-160), fused with the layer's input RMSNorm
 * (model/qwen3.py:121) and, for the first layer, the embedding lookup (model/qwen3.py:148):
 * activation rows are x[gather_rows[t]] when gather_rows is non-NULL (then also copied to x_copy:
 * the residual stream; indices are clamped into [0, x_rows)) else x[t]; RMSNorm with norm_w when non-NULL; int8 qkv projection (rows
 * [q | k | v], model/loader.py:22-28); per-head RMSNorm of q and k (q_norm_w / k_norm_w, qk_eps);
 * RoPE at positions[t] from the float32 tables [max_positions, 128] (model/layers.py:43-65);
 * q -> q_out [tokens, heads, 128]; k, v -> k_cache / v_cache [num_slots, kv_heads, 128] at
 * slot_mapping[t] (slots outside [0, num_slots) are not written). head_dim == 128. */
int msa_qkv_rope_cache_rows(const uint16_t* x, int64_t ldx, int64_t x_rows, const int64_t* gather_rows,
                            const uint16_t* norm_w,
                            float eps, uint16_t* x_copy, int64_t ld_copy, int64_t tokens, int64_t hidden,
                            const int8_t* qweight, const uint16_t* scale, int heads, int kv_heads, int head_dim,
                            const uint16_t* q_norm_w, const uint16_t* k_norm_w, float qk_eps,
                            const int64_t* positions, const float* cos_table, const float* sin_table,
                            int64_t max_positions, const int64_t* slot_mapping, uint16_t* q_out,
                            uint16_t* k_cache, uint16_t* v_cache, int64_t num_slots, msa_stream_t stream);

/* Bytes of workspace msa_lm_head_argmax needs for num_rows rows of width k over a vocabulary of
 * vocab entries (per-block argmax candidates; with many rows at a large k also the normalized
 * rows of the GEMM route). */
size_t msa_lm_head_argmax_workspace_size(int64_t num_rows, int64_t k, int64_t vocab);

/* Final norm + LM head + greedy sampling (model/qwen3.py:152-158, runner/model_runner.py:217,
 * runner/sampler.py:59) without materializing logits: for each i < num_rows,
 * out_ids[i] = argmax_v bf16(RMSNorm(hidden[rows[i]]) . weight[v]) (rows[i] clamped into
 * [0, hidden_rows)) with the first index winning
 * ties -- the argmax of the reference's bf16 logits cast to float32. norm_w NULL: the rows are
 * taken as already normalized. weight [vocab, k] bf16 (the tied embedding or the LM head).
 * k % 32 == 0. Up to 64 rows (fewer at large k) stream the weight once with the rows in LDS;
 * more rows (k % 64 == 0) normalize into the workspace and run an MFMA GEMM whose tiles keep
 * only each row's best entry. */
int msa_lm_head_argmax(const uint16_t* hidden, int64_t ld_hidden, int64_t hidden_rows, const int64_t* rows,
                       int64_t num_rows, int64_t k,
                       const uint16_t* norm_w, float eps, const uint16_t* weight, int64_t vocab, int64_t* out_ids,
                       void* workspace, size_t workspace_bytes, msa_stream_t stream);

/* Bytes of workspace msa_lm_head_logits needs (the normalized rows of the GEMM route; 0 when the
 * rows take the streaming route). */
size_t msa_lm_head_logits_workspace_size(int64_t num_rows, int64_t k, int64_t vocab);

/* Final norm + LM head for the sampled rows (model/qwen3.py:152-158 with the row selection of
 * runner/model_runner.py:214-217): logits[i][v] = float(bf16(RMSNorm(hidden[rows[i]]) . weight[v]))
 * for i < num_rows, v < vocab -- compute_logits' bf16 product cast to float32 -- into logits
 * [num_rows, ld_logits] (ld_logits >= vocab). norm_w NULL: the rows are taken as already
 * normalized. Shapes, routes and alignment as msa_lm_head_argmax. */
int msa_lm_head_logits(const uint16_t* hidden, int64_t ld_hidden, int64_t hidden_rows, const int64_t* rows,
                       int64_t num_rows, int64_t k, const uint16_t* norm_w, float eps, const uint16_t* weight,
                       int64_t vocab, float* logits, int64_t ld_logits, void* workspace, size_t workspace_bytes,
                       msa_stream_t stream);

/* ---- norms, RoPE and the KV-cache write (model/layers.py, model/qwen3.py) -------------------- */

/* The embedding rows embed[ids[t]] (bf16 [vocab, hidden]) into x [tokens, hidden] and the rotary rows of
 * positions[t] (float32 tables [max_positions, 128]; a negative position counts from the end, as in an
 * index) into cos_rows / sin_rows [tokens, 128]: model/qwen3.py:147-148 in one launch. An id or position
 * out of range aborts, as torch's own kernels do. */
int msa_embed_rope_rows(const int64_t* ids, const int64_t* positions, int64_t tokens, const uint16_t* embed,
                        int64_t vocab, int64_t hidden, const float* cos_table, const float* sin_table,
                        int64_t max_positions, uint16_t* x, float* cos_rows, float* sin_rows, msa_stream_t stream);

/* RMSNorm.forward (model/layers.py:18-22): out = bf16(w * bf16(x * rsqrt(mean(x^2) + eps))). */
int msa_rmsnorm(const uint16_t* x, int64_t ldx, const uint16_t* weight, uint16_t* out, int64_t ldo,
                int64_t rows, int64_t dim, float eps, msa_stream_t stream);

/* The residual add then RMSNorm of Qwen3DecoderLayer.forward (model/qwen3.py:121-122):
 * residual_out = bf16(residual + delta) (residual_out may alias residual), out =
 * RMSNorm(residual_out). Rows are contiguous [rows, dim]. */
int msa_add_rmsnorm(const uint16_t* residual, const uint16_t* delta, uint16_t* residual_out,
                    const uint16_t* weight, uint16_t* out, int64_t rows, int64_t dim, float eps,
                    msa_stream_t stream);

/* msa_add_rmsnorm whose delta is the bf16 sum of k_split float32 partials [k_split][rows][dim]
 * from msa_int8_linear_splitk -- the o_proj / down_proj output, residual add and the following
 * RMSNorm of Qwen3DecoderLayer.forward (model/qwen3.py:121-122) in one kernel. dim % 4 == 0. */
/* The o / down projection of a layer with the next RMSNorm (model/qwen3.py:121-122 then
 * model/layers.py:18-22): residual = bf16(residual + bf16(x @ bf16(q * s)^T)) in place, then
 * out = RMSNorm(residual) with norm_w, eps. x [m, k] (row stride ldx), qweight [n, k], residual and
 * out [m, n] contiguous, n % 8 == 0, 16-byte aligned. When the GEMM splits K (128+ rows, few
 * output tiles) the float32 partials go to workspace (msa_int8_linear_add_rmsnorm_workspace_size
 * bytes) and one kernel merges them, adds the residual and normalizes -- the split-K merge and the
 * norm launch of the unfused sequence become one pass. */
int msa_int8_linear_add_rmsnorm(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                                const uint16_t* scale, int64_t n, uint16_t* residual, const uint16_t* norm_w,
                                float eps, uint16_t* out, void* workspace, size_t workspace_bytes,
                                msa_stream_t stream);

int msa_splitk_add_rmsnorm(const float* partials, int k_split, const uint16_t* residual,
                           uint16_t* residual_out, const uint16_t* weight, uint16_t* out, int64_t rows,
                           int64_t dim, float eps, msa_stream_t stream);

/* Qwen3Attention.forward after qkv_proj (model/qwen3.py:94-98) plus the cache write of
 * paged_attention (attention/backends.py:159-160): split qkv [tokens, (H + 2 KVH) * D] (row stride
 * ldqkv) into q | k | v; per-head RMSNorm of q and k with q_norm_w / k_norm_w [D]; RoPE with the
 * float32 rows cos, sin [tokens, D] (cast to bf16 as layers.py:63-64 does); q -> q_out [tokens,
 * H, D]; k, v -> k_cache, v_cache [num_slots, KVH, D] at slot_mapping[t]. Slots outside
 * [0, num_slots) are not written. D even, D <= 256. */
int msa_qk_norm_rope_cache(const uint16_t* qkv, int64_t ldqkv, int64_t tokens, int heads, int kv_heads,
                           int head_dim, const uint16_t* q_norm_w, const uint16_t* k_norm_w, float eps,
                           const float* cos, const float* sin, const int64_t* slot_mapping,
                           uint16_t* q_out, uint16_t* k_cache, uint16_t* v_cache, int64_t num_slots,
                           msa_stream_t stream);

/* msa_qk_norm_rope_cache reading the qkv rows as k_split float32 partials
 * [k_split][tokens][(H + 2 KVH) * D] from msa_int8_linear_splitk (summed in order, rounded to bf16). */
int msa_qk_norm_rope_cache_splitk(const float* partials, int k_split, int64_t tokens, int heads, int kv_heads,
                                  int head_dim, const uint16_t* q_norm_w, const uint16_t* k_norm_w, float eps,
                                  const float* cos, const float* sin, const int64_t* slot_mapping,
                                  uint16_t* q_out, uint16_t* k_cache, uint16_t* v_cache, int64_t num_slots,
                                  msa_stream_t stream);

/* k_cache.index_copy_(0, slot_mapping, k) and the same for v (attention/backends.py:159-160).
 * k, v [tokens, KVH, D] with row strides ldk, ldv (elements per token). */
int msa_reshape_and_cache(const uint16_t* k, int64_t ldk, const uint16_t* v, int64_t ldv, int64_t tokens,
                          int kv_heads, int head_dim, const int64_t* slot_mapping, uint16_t* k_cache,
                          uint16_t* v_cache, int64_t num_slots, msa_stream_t stream);

/* ---- paged attention (attention/backends.py:145-197) ----------------------------------------- */

size_t msa_paged_attention_decode_workspace_size(int num_seqs, int heads, int head_dim, int max_partitions);

/* The batched short-query path of paged_attention (attention/backends.py:165-180) for one new
 * token per sequence, reading K/V blocks in place instead of gathering them: sequence i's query
 * is row q_rows[i] of q [*, H, D] (row stride ldq), its keys are positions 0..context_lens[i]-1
 * through block_tables[i, :] (int32, row stride max_blocks), query head h reads KV head
 * h / (H / KVH); out row q_rows[i] (row stride ldo). A workgroup of wavefronts covers
 * partition_tokens keys of one (sequence, KV head) with an online softmax; with max_partitions > 1
 * the partitions meet in the workspace (msa_paged_attention_decode_workspace_size bytes) and a
 * second kernel merges them. partition_tokens % 16 == 0 and partition_tokens * max_partitions >=
 * 16 * max_blocks. D == 128, block_size == 16, H / KVH in {1, 2, 4, 8}. */
int msa_paged_attention_decode(const uint16_t* q, int64_t ldq, const uint16_t* k_cache,
                               const uint16_t* v_cache, int64_t num_slots, int heads, int kv_heads,
                               int head_dim, int block_size, const int32_t* block_tables, int max_blocks,
                               const int32_t* context_lens, const int32_t* q_rows, int num_seqs,
                               int partition_tokens, int max_partitions, float scale, uint16_t* out,
                               int64_t ldo, void* workspace, size_t workspace_bytes, msa_stream_t stream);

/* msa_paged_attention_decode with four-wavefront workgroups at every partition size (the plain
 * entry point takes eight for partitions of 1024+ keys with heads / kv_heads <= 2), for decode rows
 * attended while another kernel runs on another stream: the decode rows of a mixed batch beside
 * the prefill chunk's attention (the call of attention/backends.py:165-196 with both kinds of rows),
 * whose workgroups leave each CU room for one four-wavefront workgroup but not for eight. Same
 * arguments, partitions and workspace as msa_paged_attention_decode; results equal its results up to
 * the order in which a workgroup's wavefronts are merged (float32 sums). */
int msa_paged_attention_decode_narrow(const uint16_t* q, int64_t ldq, const uint16_t* k_cache,
                                      const uint16_t* v_cache, int64_t num_slots, int heads, int kv_heads,
                                      int head_dim, int block_size, const int32_t* block_tables, int max_blocks,
                                      const int32_t* context_lens, const int32_t* q_rows, int num_seqs,
                                      int partition_tokens, int max_partitions, float scale, uint16_t* out,
                                      int64_t ldo, void* workspace, size_t workspace_bytes, msa_stream_t stream);

/* Largest split-partials size (msa_paged_attention_decode_workspace_size) that
 * msa_paged_attention_decode_noalloc serves: 16 MiB. */
#define MSA_DECODE_NOALLOC_MAX_BYTES ((size_t)16 << 20)

/* msa_paged_attention_decode without a workspace argument, for callers that cannot allocate device
 * memory (code under HIP graph capture, tight serving loops, harnesses that forbid hipMalloc). No
 * counterpart in the reference. The split partials live in a scratch array inside the library, one
 * per GPU, held until the process ends; calls whose partials need more than
 * MSA_DECODE_NOALLOC_MAX_BYTES fail with MSA_ERR_WORKSPACE, and the call allocates nothing. Every
 * call on one GPU shares that GPU's scratch: calls that overlap in time on one GPU (different
 * streams) race and must be ordered by the caller. Results are bit-identical to
 * msa_paged_attention_decode's for the same arguments. */
int msa_paged_attention_decode_noalloc(const uint16_t* q, int64_t ldq, const uint16_t* k_cache,
                                       const uint16_t* v_cache, int64_t num_slots, int heads, int kv_heads,
                                       int head_dim, int block_size, const int32_t* block_tables, int max_blocks,
                                       const int32_t* context_lens, const int32_t* q_rows, int num_seqs,
                                       int partition_tokens, int max_partitions, float scale, uint16_t* out,
                                       int64_t ldo, msa_stream_t stream);

/* The decode rows of Qwen3Attention.forward from the projection onward (model/qwen3.py:95-99 with
 * the cache write of attention/backends.py:159-160) in one launch: qkv [*, (H + 2 KVH) * 128]
 * holds the int8 qkv projection rows [q | k | v] (row stride ldqkv, model/loader.py:22-28). For
 * sequence i (row q_rows[i]) the new token sits at position p = context_lens[i] - 1
 * (runner/model_runner.py:186-189): each workgroup applies the per-head RMSNorm (q_norm_w /
 * k_norm_w, qk_eps) and RoPE at p (float32 tables [max_positions, 128], model/layers.py:43-65) to
 * its query heads and its KV head's key, writes the key and value into k_cache / v_cache at slot
 * slot_mapping[q_rows[i]] (int64; slots outside [0, num_slots) are not written -- the runner's
 * slot is block_tables[i, p / 16] * 16 + p % 16), and attends to keys 0..p-1 from the cache and to
 * key p from registers. Otherwise as msa_paged_attention_decode (same partitions and workspace);
 * out has H * 128 columns. */
int msa_paged_attention_decode_qkv(const uint16_t* qkv, int64_t ldqkv, const uint16_t* q_norm_w,
                                   const uint16_t* k_norm_w, float qk_eps, const float* cos_table,
                                   const float* sin_table, int64_t max_positions, const int64_t* slot_mapping,
                                   uint16_t* k_cache,
                                   uint16_t* v_cache, int64_t num_slots, int heads, int kv_heads, int head_dim,
                                   int block_size, const int32_t* block_tables, int max_blocks,
                                   const int32_t* context_lens, const int32_t* q_rows, int num_seqs,
                                   int partition_tokens, int max_partitions, float scale, uint16_t* out,
                                   int64_t ldo, void* workspace, size_t workspace_bytes, msa_stream_t stream);
/* The same with the rotary rows gathered by the caller: sequence i is rotated by row q_rows[i] of the
 * float32 [rows, 128] cos_rows / sin_rows (one per row of qkv), whatever its context length. */
int msa_paged_attention_decode_qkv_rows(const uint16_t* qkv, int64_t ldqkv, const uint16_t* q_norm_w,
                                        const uint16_t* k_norm_w, float qk_eps, const float* cos_rows,
                                        const float* sin_rows, int64_t rows, const int64_t* slot_mapping,
                                        uint16_t* k_cache,
                                        uint16_t* v_cache, int64_t num_slots, int heads, int kv_heads, int head_dim,
                                        int block_size, const int32_t* block_tables, int max_blocks,
                                        const int32_t* context_lens, const int32_t* q_rows, int num_seqs,
                                        int partition_tokens, int max_partitions, float scale, uint16_t* out,
                                        int64_t ldo, void* workspace, size_t workspace_bytes, msa_stream_t stream);

/* The qkv projection of a prefill-sized batch with the per-head q/k RMSNorm, RoPE and KV-cache
 * write of msa_qk_norm_rope_cache in its epilogue (model/qwen3.py:94-98, then the cache write of
 * attention/backends.py:159-160): y = x @ bf16(q * s)^T as msa_int8_gemm computes it
 * (float32 sums rounded to bf16), n = (heads + 2 kv_heads) * 128 weight rows
 * whose 128-row blocks are the head slots (q heads, k heads, v heads); then the same rounding
 * steps as msa_qk_norm_rope_cache, bit for bit: q_out [m, heads, 128] gets the normed, rotated
 * queries, k_cache / v_cache [num_slots, kv_heads, 128] the normed, rotated keys and the values at
 * slot_mapping[t] (slots outside [0, num_slots) are skipped). cos / sin are [m, 128] float32.
 * head_dim must be 128; x, the norm weights, cos / sin, q_out and the caches 16-byte aligned.
 * When the GEMM would split K (few output tiles) and the workspace holds
 * msa_int8_gemm_qk_norm_rope_cache_workspace_size(m, n, k) bytes, the split-K partials go there and
 * msa_qk_norm_rope_cache_splitk sums them (the same values); otherwise the epilogue does it. */
int msa_int8_gemm_qk_norm_rope_cache(const uint16_t* x, int64_t m, int64_t k, int64_t ldx, const int8_t* qweight,
                                     const uint16_t* scale, int heads, int kv_heads, int head_dim,
                                     const uint16_t* q_norm_w, const uint16_t* k_norm_w, float eps,
                                     const float* cos, const float* sin, const int64_t* slot_mapping,
                                     uint16_t* q_out, uint16_t* k_cache, uint16_t* v_cache, int64_t num_slots,
                                     void* workspace, size_t workspace_bytes, msa_stream_t stream);

/* The prefill path of paged_attention (attention/backends.py:182-196) for chunks of any length,
 * fresh or continuing from cached keys: causal attention of each new token over positions
 * 0..its own, keys and values read through the block table from the caches (which already hold
 * this step's tokens). seq_info [num_seqs, 3] int32 = (first flat row, num_new, num_cached);
 * work [num_work, 2] int32 = (sequence index, first new-token index of a 64 / (H / KVH)-token
 * tile). D == 128, block_size == 16, H / KVH in {1, 2, 4}. */
int msa_paged_attention_prefill(const uint16_t* q, int64_t ldq, const uint16_t* k_cache,
                                const uint16_t* v_cache, int64_t num_slots, int heads, int kv_heads,
                                int head_dim, int block_size, const int32_t* block_tables, int max_blocks,
                                const int32_t* seq_info, const int32_t* work, int num_work, float scale,
                                uint16_t* out, int64_t ldo, msa_stream_t stream);
/* The same on query tiles of twice the tokens (work lists of 128 / (heads / kv_heads) tokens): for
 * batches with enough tiles to fill the chip. */
int msa_paged_attention_prefill_wide(const uint16_t* q, int64_t ldq, const uint16_t* k_cache,
                                     const uint16_t* v_cache, int64_t num_slots, int heads, int kv_heads,
                                     int head_dim, int block_size, const int32_t* block_tables, int max_blocks,
                                     const int32_t* seq_info, const int32_t* work, int num_work, float scale,
                                     uint16_t* out, int64_t ldo, msa_stream_t stream);

/* ---- sampling (runner/sampler.py) ------------------------------------------------------------ */

/* apply_top_k_top_p (runner/sampler.py:12-27) without a sort: out[r] = logits[r] where the entry
 * is among the row's top_k[r] largest (ties with the k-th kept) and inside its top_p[r] nucleus
 * (the smallest-value entries are dropped while their cumulative softmax probability stays
 * <= 1 - p; the largest entry is always kept), -inf elsewhere. top_k[r] outside (0, vocab) or a
 * NULL top_k: no top-k; top_p[r] >= 1 or a NULL top_p: no top-p. logits / out float32, row
 * strides ld / ldo. */
int msa_top_k_top_p_mask(const float* logits, int64_t ld, int64_t rows, int64_t vocab, const int32_t* top_k,
                         const float* top_p, float* out, int64_t ldo, msa_stream_t stream);

/* compute_probs (runner/sampler.py:30-40): probs[r] = softmax over the kept entries of
 * logits[r] / temperature[r] (temperature already clamped to >= 1e-5 by the caller; NULL: 1),
 * with top-k / top-p applied to the scaled logits as in msa_top_k_top_p_mask; 0 elsewhere. */
int msa_sampling_probs(const float* logits, int64_t ld, int64_t rows, int64_t vocab, const float* temperature,
                       const int32_t* top_k, const float* top_p, float* probs, int64_t ldp, msa_stream_t stream);

/* sample (runner/sampler.py:55-69): out_ids[r] = argmax(logits[r]) (first index) where
 * greedy[r] != 0, else the exponential race argmax_i probs[r][i] / max(noise[r][i], FLT_MIN) with
 * probs as msa_sampling_probs and noise ~ Exp(1) [rows, ldn] drawn by the caller (the reference
 * draws it with torch's exponential_, per-row generators for seeded requests). With a workspace
 * of msa_sample_workspace_size(rows, vocab) bytes (rows <= 65535), greedy rows and rows with
 * 0 < top_k <= 256 are spread over vocabulary chunks (two launches); a NULL workspace takes one
 * workgroup per row. */
size_t msa_sample_workspace_size(int64_t rows, int64_t vocab);
int msa_sample(const float* logits, int64_t ld, int64_t rows, int64_t vocab, const float* temperature,
               const int32_t* top_k, const float* top_p, const uint8_t* greedy, const float* noise, int64_t ldn,
               int64_t* out_ids, void* workspace, size_t workspace_bytes, msa_stream_t stream);
/* msa_sample for a batch with rows without top-k: they are spread over the chunks too (four launches;
 * the workspace 8-byte aligned, else one workgroup each as above). */
int msa_sample_wide(const float* logits, int64_t ld, int64_t rows, int64_t vocab, const float* temperature,
                    const int32_t* top_k, const float* top_p, const uint8_t* greedy, const float* noise, int64_t ldn,
                    int64_t* out_ids, void* workspace, size_t workspace_bytes, msa_stream_t stream);

/* ---- speculative-decoding verification (spec/rejection.py) ----------------------------------- */

/* verify_greedy (spec/rejection.py:27-40) from the target's per-position argmax target_ids
 * [batch, k + 1] (int64; msa_sample with every row greedy computes them from logits): accepted[i] =
 * leading run of drafts[i, j] == target_ids[i, j] over j < num_drafts[i]; next_token[i] =
 * target_ids[i, accepted[i]]. drafts [batch, k] int64. */
int msa_verify_greedy(const int64_t* target_ids, int64_t batch, int64_t k, const int64_t* drafts,
                      const int64_t* num_drafts, int64_t* accepted, int64_t* next_token, msa_stream_t stream);

/* verify_sampled (spec/rejection.py:43-79): target_probs [batch, k + 1, vocab], drafts [batch, k],
 * num_drafts [batch], draft_probs [batch, k, vocab] or NULL (a deterministic proposer), uniform
 * [batch, k] ~ U(0, 1), noise [batch, vocab] ~ Exp(1); float32 tensors contiguous. Accepts draft j
 * while uniform < min(1, p_j(d_j) / q_j(d_j)); next_token samples normalize(max(0, p_a - q_a)) after
 * a rejection (p_a with the draft zeroed when q is NULL), else p_a, as argmax(dist / noise). k >= 1. */
int msa_verify_sampled(const float* target_probs, int64_t batch, int64_t k, int64_t vocab, const int64_t* drafts,
                       const int64_t* num_drafts, const float* draft_probs, const float* uniform, const float* noise,
                       int64_t* accepted, int64_t* next_token, msa_stream_t stream);

#ifdef __cplusplus
}
#endif

#endif /* MINISERVE_AMD_H */
