/*
 * kvfp8.h - C ABI of the MI355X (gfx950) FP8 paged KV-cache library `libkvfp8.so`.
 *
 * Every pointer argument named *_dev is a device pointer owned by the caller.
 * Work is enqueued on `stream` (a hipStream_t, passed as void*) and never
 * synchronizes with the host. Return value: 0 on success, a negative KVFP8_E*
 * code for an argument rejected on the host (shapes and dtypes only, no device
 * values are read), or a positive hipError_t from the launch.
 * kvfp8_strerror() names every code.
 *
 * The Python mirror of the reference API (aiproj_amd.kernals.*) binds these
 * entry points with ctypes (aiproj_amd/_native.py holds the signatures).
 */
#ifndef KVFP8_H
#define KVFP8_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Element types understood by the library. */
enum kvfp8_dtype {
    KVFP8_F32 = 0,
    KVFP8_F16 = 1,
    KVFP8_BF16 = 2,
    KVFP8_E4M3FN = 3, /* OCP float8_e4m3fn */
    KVFP8_I32 = 4,
    KVFP8_I64 = 5,
};

/* Host-side argument errors (negative return codes). */
enum kvfp8_status {
    KVFP8_OK = 0,
    KVFP8_EDTYPE = -1,     /* unsupported dtype for this argument */
    KVFP8_ESHAPE = -2,     /* inconsistent or non-positive sizes */
    KVFP8_ESTRIDE = -3,    /* unsupported stride / alignment */
    KVFP8_ENULL = -4,      /* required pointer is NULL */
    KVFP8_EWORKSPACE = -5, /* workspace too small */
    KVFP8_ELIMIT = -6,     /* size beyond what the kernels support */
};

/*
 * Quantize-and-scatter append of T new tokens into an FP8 paged cache.
 *
 * Replaces `quantize_append_wrapper` + the Triton `quantize_append` kernel,
 * reference src/torch_llm/kernals/kv_cache/quantized_append.py:35-133.
 * For each (token t, kv head h), separately for K and V:
 *     amax  = max_d |x[t,h,d]|               (float32, NaN-propagating)
 *     scale = amax > 0 ? amax / 448 : 1       (IEEE float32 division)
 *     code  = e4m3fn_rne(clamp(x / scale, -448, 448))
 * stores code at cache[blocks[t], offsets[t], h, :] and scale at
 * scales[blocks[t], offsets[t], h]. Caches are [num_blocks, block_size, H_kv, D]
 * uint8 (e4m3fn bits); scales are [num_blocks, block_size, H_kv] float32.
 * Rows whose (block, offset) lies outside the pool are skipped.
 *
 * k/v: [T, H_kv, D] with element strides (stride_t, stride_h, 1), dtype
 * f32/f16/bf16. blocks/offsets: [T] int32 or int64.
 */
int kvfp8_quantize_append(const void* k_dev, const void* v_dev, int in_dtype,
                          int64_t k_stride_t, int64_t k_stride_h,
                          int64_t v_stride_t, int64_t v_stride_h,
                          const void* blocks_dev, int blocks_dtype,
                          const void* offsets_dev, int offsets_dtype,
                          int64_t num_tokens, int32_t num_kv_heads, int32_t head_dim,
                          int64_t num_blocks, int32_t block_size,
                          void* k_cache_dev, void* v_cache_dev,
                          float* k_scales_dev, float* v_scales_dev,
                          void* stream);

/*
 * Unquantized scatter append: cache[blocks[t], offsets[t]] = x[t].to(cache dtype).
 *
 * Replaces the indexed store of reference
 * src/torch_llm/inference/paged_kv_cache.py:77-79 for device storage.
 * cache_dtype is f32/f16/bf16 (round-to-nearest-even narrowing, as torch's .to()).
 */
int kvfp8_store_append(const void* k_dev, const void* v_dev, int in_dtype,
                       int64_t k_stride_t, int64_t k_stride_h,
                       int64_t v_stride_t, int64_t v_stride_h,
                       const void* blocks_dev, int blocks_dtype,
                       const void* offsets_dev, int offsets_dtype,
                       int64_t num_tokens, int32_t num_kv_heads, int32_t head_dim,
                       int64_t num_blocks, int32_t block_size,
                       void* k_cache_dev, void* v_cache_dev, int cache_dtype,
                       void* stream);

/*
 * Bytes of device workspace kvfp8_paged_decode needs for these shapes
 * (split-K partial softmax states). Depends on shapes only.
 */
int64_t kvfp8_decode_workspace_bytes(int32_t batch, int32_t num_q_heads, int32_t num_kv_heads,
                                     int32_t head_dim, int64_t bt_width, int32_t block_size,
                                     int kv_dtype);

/*
 * Paged decode attention over a (quantized or plain) paged cache.
 *
 * Replaces `decode_attention_wrapper` and the Triton split and reduction kernels,
 * reference src/torch_llm/kernals/decode_attention.py:39-550:
 *   out[b, hq, :] = softmax_t( q[b,hq,:] . khat[t,:] * sm_scale ) @ vhat
 * over t < context_lengths[b], where khat/vhat are the cache rows of kv head
 * hq / (Hq / Hkv) gathered through block_table[slots[b], t / block_size] at
 * offset t % block_size, dequantized as code * scale when kv_dtype is e4m3fn.
 * A sequence with no context (or no valid page) yields zeros.
 *
 * q: [B, Hq, D], element strides (q_stride_b, q_stride_h, 1), dtype f32/f16/bf16.
 * out: [B, Hq, D] contiguous, same dtype as q.
 * k/v cache: [num_blocks, block_size, Hkv, D] of kv_dtype (e4m3fn/bf16/f16/f32).
 * k/v scales: [num_blocks, block_size, Hkv] float32, NULL unless e4m3fn.
 * block_table: [bt_rows, bt_width] int32, entries outside [0, num_blocks) skipped.
 * slots: [B] int32/int64 rows of block_table; context_lengths: [B] int32/int64.
 * workspace: at least kvfp8_decode_workspace_bytes(...) bytes, any contents.
 */
int kvfp8_paged_decode(const void* q_dev, int q_dtype, int64_t q_stride_b, int64_t q_stride_h,
                       int32_t batch, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                       const void* k_cache_dev, const void* v_cache_dev, int kv_dtype,
                       const float* k_scales_dev, const float* v_scales_dev,
                       int64_t num_blocks, int32_t block_size,
                       const int32_t* block_table_dev, int64_t bt_rows, int64_t bt_width,
                       const void* slots_dev, int slots_dtype,
                       const void* context_lengths_dev, int ctx_dtype,
                       float sm_scale, void* out_dev,
                       void* workspace_dev, int64_t workspace_bytes,
                       void* stream);

/*
 * The two launches of kvfp8_paged_decode as separate calls (same arguments; the
 * same workspace must reach both, and nothing may write it in between):
 *
 * kvfp8_paged_decode_split enqueues the split kernel, reference
 * `decode_attention_split_kernel` (src/torch_llm/kernals/decode_attention.py:194-434):
 * it writes the output rows of the sequences it finishes whole and a partial
 * softmax state (m, l, acc) per piece of every other sequence into the workspace.
 *
 * kvfp8_paged_decode_reduce enqueues the merge, reference
 * `decode_attention_reduction_kernel` (decode_attention.py:437-550): out =
 * sum_i 2^(m_i - M) acc_i / sum_i 2^(m_i - M) l_i over the pieces, zeros for empty
 * sequences.
 *
 * Callers that combine pieces from elsewhere (a sequence split across devices) or
 * time the split kernel alone use these; split followed by reduce on one stream
 * equals kvfp8_paged_decode bit for bit.
 */
int kvfp8_paged_decode_split(const void* q_dev, int q_dtype, int64_t q_stride_b, int64_t q_stride_h,
                             int32_t batch, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                             const void* k_cache_dev, const void* v_cache_dev, int kv_dtype,
                             const float* k_scales_dev, const float* v_scales_dev,
                             int64_t num_blocks, int32_t block_size,
                             const int32_t* block_table_dev, int64_t bt_rows, int64_t bt_width,
                             const void* slots_dev, int slots_dtype,
                             const void* context_lengths_dev, int ctx_dtype,
                             float sm_scale, void* out_dev,
                             void* workspace_dev, int64_t workspace_bytes,
                             void* stream);
int kvfp8_paged_decode_reduce(const void* q_dev, int q_dtype, int64_t q_stride_b, int64_t q_stride_h,
                              int32_t batch, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                              const void* k_cache_dev, const void* v_cache_dev, int kv_dtype,
                              const float* k_scales_dev, const float* v_scales_dev,
                              int64_t num_blocks, int32_t block_size,
                              const int32_t* block_table_dev, int64_t bt_rows, int64_t bt_width,
                              const void* slots_dev, int slots_dtype,
                              const void* context_lengths_dev, int ctx_dtype,
                              float sm_scale, void* out_dev,
                              void* workspace_dev, int64_t workspace_bytes,
                              void* stream);

/*
 * kvfp8_paged_decode for callers that cannot allocate device memory: code under HIP
 * graph capture, serving loops and harnesses that forbid hipMalloc. It has no
 * counterpart in the reference. Same arguments, computation and results as
 * kvfp8_paged_decode, bit for bit, minus the workspace: the split-K plan and partial
 * states live in a static device array of KVFP8_NOALLOC_SCRATCH_BYTES that the
 * library holds on every device it runs on until the process ends. Shapes whose
 * workspace would exceed it return KVFP8_ELIMIT before anything is launched. The call
 * allocates nothing (no hipMalloc/hipFree, no allocating library routine); its first
 * call on a device looks up that device's array address (hipGetSymbolAddress), so a
 * caller that captures graphs makes one call on each device before capturing.
 * Every call on one device uses the same array: calls that overlap on one device
 * (concurrent streams, or a graph replay concurrent with an eager call) race on it.
 * Calls ordered on one stream do not.
 */
#define KVFP8_NOALLOC_SCRATCH_BYTES (32ll << 20)
int kvfp8_paged_decode_noalloc(const void* q_dev, int q_dtype, int64_t q_stride_b, int64_t q_stride_h,
                               int32_t batch, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                               const void* k_cache_dev, const void* v_cache_dev, int kv_dtype,
                               const float* k_scales_dev, const float* v_scales_dev,
                               int64_t num_blocks, int32_t block_size,
                               const int32_t* block_table_dev, int64_t bt_rows, int64_t bt_width,
                               const void* slots_dev, int slots_dtype,
                               const void* context_lengths_dev, int ctx_dtype,
                               float sm_scale, void* out_dev, void* stream);

/*
 * RMSNorm forward over rows of x [rows, d_model] (row stride x_stride elements):
 *   inv_rms[r] = 1 / sqrt(mean_d x[r,d]^2 + eps); out[r,d] = (x[r,d] * inv_rms[r]) * weight[d]
 * in float32, out stored in x's dtype (f32/f16/bf16); weight f32/f16/bf16; inv_rms
 * (float32 [rows]) may be NULL.
 * Replaces `triton_rmsnorm` + `rmsnorm_kernal`, reference
 * src/torch_llm/model/rmsnorm.py:60-113.
 */
int kvfp8_rmsnorm_forward(const void* x_dev, int dtype, int64_t x_stride, int64_t rows, int32_t d_model,
                          const void* weight_dev, int w_dtype, float eps,
                          void* out_dev, int64_t out_stride, float* inv_rms_dev, void* stream);

/*
 * Residual add fused with the RMSNorm that follows it:
 *   state_out = x + update (rounded to x's dtype), out = rmsnorm(state_out).
 * Replaces `residual.write` + the next sublayer's norm, reference
 * src/torch_llm/model/decoder_block.py:60-66 and model/residual.py:33-35.
 */
int kvfp8_add_rmsnorm_forward(const void* x_dev, const void* update_dev, int dtype,
                              int64_t x_stride, int64_t update_stride, int64_t rows, int32_t d_model,
                              const void* weight_dev, int w_dtype, float eps,
                              void* state_out_dev, int64_t state_stride,
                              void* out_dev, int64_t out_stride, float* inv_rms_dev, void* stream);

/*
 * Backward of kvfp8_rmsnorm_forward in float32: dx (x's dtype) and dw (weight's dtype) from
 * x, the forward's inv_rms and the gradient of its output (x's dtype). d_model: multiples of
 * 8 up to 4096 (KVFP8_ELIMIT otherwise), rows 16-byte aligned. The workspace holds
 * kvfp8_rmsnorm_backward_workspace_bytes(...) bytes, any contents. Sums are added in a fixed
 * order. No reference counterpart on this path (training).
 */
int64_t kvfp8_rmsnorm_backward_workspace_bytes(int64_t rows, int32_t d_model);
int kvfp8_rmsnorm_backward(const void* x_dev, const void* grad_dev, int dtype, int64_t x_stride, int64_t grad_stride,
                           int64_t rows, int32_t d_model, const void* weight_dev, int w_dtype,
                           const float* inv_rms_dev, void* dx_dev, int64_t dx_stride, void* dw_dev,
                           void* workspace_dev, int64_t workspace_bytes, void* stream);

/*
 * Varlen causal attention over packed prompts (prefill):
 *   q [T, Hq, D], k and v [T, Hkv, D] contiguous, one dtype (f32/f16/bf16);
 *   cu_seqlens [batch + 1] (int32/int64): sequence b is tokens
 *   [cu_seqlens[b], cu_seqlens[b + 1]); query row i of it attends keys 0..i of it;
 *   q head h reads KV head h / (Hq / Hkv).
 *   out [T, Hq, D] (q's dtype) and lse [T, Hq] float32 = m + log(sum exp(s - m)) of
 *   the scaled scores s = scale * q.k. Rows outside every sequence are not written;
 *   only the first max_seq_len rows of each sequence are computed.
 *   head_dim 1..512: multiples of 8 up to 128 run on the matrix cores (pointers
 *   16-byte aligned), every other size on a vector-ALU kernel (pointers aligned to
 *   the element size).
 * Replaces the forward of reference src/torch_llm/kernals/flash_attention.py:51-211
 * (flash_attention_forward and flash_attention_forward_kernal).
 */
int kvfp8_prefill_attention(const void* q_dev, const void* k_dev, const void* v_dev, int dtype,
                            int64_t total_tokens, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                            const void* cu_seqlens_dev, int cu_dtype, int32_t batch, int32_t max_seq_len,
                            float scale, void* out_dev, float* lse_dev, void* stream);

/*
 * Backward of kvfp8_prefill_attention: dq [T, Hq, D], dk and dv [T, Hkv, D] (the inputs'
 * dtype) from q, k, v, the forward's out and lse, and grad_out [T, Hq, D], all contiguous
 * and of one dtype. Products have float32 accuracy and the results one rounding; dk and
 * dv are summed over the q heads of a KV head. Rows of no sequence, or past the first
 * max_seq_len of theirs, get zeros. head_dim 1..128. Results do not depend on timing.
 *   workspace: kvfp8_prefill_backward_workspace_bytes(...) bytes, 16-byte aligned, any
 *   contents; `aligned`: q, k, v and grad_out are 16-byte aligned (fewer bytes then). dq, dk and dv are 16-byte aligned.
 * Both return KVFP8_ELIMIT where a launch would take 2^32 threads or more.
 * Replaces the backward of reference src/torch_llm/kernals/flash_attention.py:213 onwards.
 */
int64_t kvfp8_prefill_backward_workspace_bytes(int dtype, int64_t total_tokens, int32_t num_q_heads,
                                               int32_t num_kv_heads, int32_t head_dim, int32_t batch,
                                               int32_t max_seq_len, int aligned);
int kvfp8_prefill_attention_backward(const void* q_dev, const void* k_dev, const void* v_dev, const void* out_dev,
                                     const float* lse_dev, const void* grad_out_dev, int dtype, int64_t total_tokens,
                                     int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                     const void* cu_seqlens_dev, int cu_dtype, int32_t batch, int32_t max_seq_len,
                                     float scale, void* dq_dev, void* dk_dev, void* dv_dev,
                                     void* workspace_dev, int64_t workspace_bytes, void* stream);

/*
 * Fused append + decode: the quantize-and-scatter write of every sequence's new
 * token and the paged decode attention over the context that includes it, in the
 * decode kernel's launches (no separate append launch).
 *
 * Replaces the two calls the reference makes back to back in its decode step,
 * reference src/torch_llm/model/attention.py:86-99 (PagedKVCache.append_kv, then
 * decode_attention_wrapper). The new token of sequence b is its last attended
 * position L - 1 (L = context_lengths[b]), page block_table[slots[b], (L - 1) /
 * block_size] at offset (L - 1) % block_size. The wave that serves KV head h over
 * the sequence's last tile quantizes head h of row b of k_new/v_new with the
 * kvfp8_quantize_append rule and stores it at (new_blocks[b], new_offsets[b])
 * before it reads that tile; no other wave reads that row. Results (cache codes and
 * scales, and outputs) equal the two calls bit for bit.
 *
 * The kernel checks every write location on the device against the block table.
 * A location that is not the sequence's last attended position, or a sequence that
 * attends no new token (L = 0, L beyond the table, a slot outside it), is refused:
 * nothing is stored for it, 1 is stored to *refused_dev (when not NULL; the call
 * never clears it, so the caller zeroes it before), and its output is that of
 * kvfp8_paged_decode on the cache as it is. So the write never races with a read.
 * A matching location outside the pool is skipped, as in kvfp8_quantize_append.
 *
 * Takes the kvfp8_paged_decode arguments (the same workspace size), then the new
 * rows: k_new/v_new [batch, H_kv, D] (f32/f16/bf16, one dtype) with element strides
 * (stride_b, stride_h, 1), stride_h == D and stride_b below 2^31, then the write locations
 * new_blocks/new_offsets [batch] (int32/int64), then refused_dev (int32, may be
 * NULL). e4m3fn caches on the MFMA kernel only: other shapes return KVFP8_ESHAPE
 * before launching anything (kvfp8_append_decode_supported says which).
 */
int kvfp8_append_paged_decode(const void* q_dev, int q_dtype, int64_t q_stride_b, int64_t q_stride_h,
                              int32_t batch, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                              const void* k_cache_dev, const void* v_cache_dev, int kv_dtype,
                              const float* k_scales_dev, const float* v_scales_dev,
                              int64_t num_blocks, int32_t block_size,
                              const int32_t* block_table_dev, int64_t bt_rows, int64_t bt_width,
                              const void* slots_dev, int slots_dtype,
                              const void* context_lengths_dev, int ctx_dtype,
                              float sm_scale, void* out_dev,
                              void* workspace_dev, int64_t workspace_bytes, void* stream,
                              const void* k_new_dev, const void* v_new_dev, int new_dtype,
                              int64_t k_new_stride_b, int64_t k_new_stride_h,
                              int64_t v_new_stride_b, int64_t v_new_stride_h,
                              const void* new_blocks_dev, int new_blocks_dtype,
                              const void* new_offsets_dev, int new_offsets_dtype,
                              int32_t* refused_dev);

/* 1 when kvfp8_append_paged_decode handles these shapes (e4m3fn cache on the MFMA
 * kernel), else 0. Shapes only; pointer alignment is checked by the call. */
int kvfp8_append_decode_supported(int32_t batch, int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                  int64_t bt_rows, int64_t bt_width, int32_t block_size, int kv_dtype);

/*
 * Interleaved-pair rotary embedding in place on heads [0, heads) of every row of x
 * (element strides row_stride, head_stride; pairs (2i, 2i+1) of head_dim):
 *   x0' = c x0 - s x1, x1' = s x0 + c x1,  c/s = cos/sin_table[positions[r], i]
 * with each operation rounded to x's dtype (f32/f16/bf16) and the table values
 * ([table_rows, head_dim / 2], table_dtype f32/f16/bf16) cast to it first. Rows
 * whose position is outside the tables are left unchanged. positions: [rows]
 * int32/int64.
 * Replaces the RoPE op sequence of reference src/torch_llm/model/rope.py:46-55.
 */
int kvfp8_rope_inplace(void* x_dev, int dtype, int64_t rows, int32_t heads, int32_t head_dim,
                       int64_t row_stride, int64_t head_stride, const void* positions_dev, int pos_dtype,
                       const void* cos_table_dev, const void* sin_table_dev, int table_dtype,
                       int64_t table_rows, void* stream);

/*
 * kvfp8_rope_inplace's rotation of the fused projection rows [q heads | k heads | v heads]
 * (head_dim elements each), written to packed q [rows, num_q_heads, head_dim], k and v
 * [rows, num_kv_heads, head_dim]; v is copied. head_dim a multiple of 8, rows, tables and
 * outputs aligned for 16-byte accesses (KVFP8_ESTRIDE otherwise).
 */
int kvfp8_rope_split(const void* x_dev, int dtype, int64_t rows, int32_t num_q_heads, int32_t num_kv_heads,
                     int32_t head_dim, int64_t row_stride, const void* positions_dev, int pos_dtype,
                     const void* cos_table_dev, const void* sin_table_dev, int table_dtype, int64_t table_rows,
                     void* q_out_dev, void* k_out_dev, void* v_out_dev, void* stream);

/*
 * SwiGLU activation: out[r, j] = silu(g) * u with g = x[r, j], u = x[r, n + j] and
 * silu(g) = g * (1 / (1 + exp(-g))), in float32 with one rounding to the dtype
 * (f32/f16/bf16). x rows hold gate then up (row stride >= 2 n elements); out rows
 * n elements (row stride >= n).
 * Replaces the activation of reference src/torch_llm/kernals/moe/grouped_swiglu_up.py:239
 * (applied there to the float32 accumulators of the fused gate/up product).
 */
int kvfp8_silu_mul(const void* x_dev, int dtype, int64_t rows, int32_t n, int64_t x_row_stride,
                   void* out_dev, int64_t out_row_stride, void* stream);

/*
 * Kernel timing hook for benchmarks (not part of the reference interface).
 * kvfp8_timing_enable(n) arms start/stop HIP events on the dispatch packets of
 * the next n decode-kernel launches (hipExtLaunchKernel, on the stream each launch
 * uses); kvfp8_timing_read() waits for those events and returns the summed kernel
 * milliseconds and the number of timed launches, then disarms. n <= 0 disarms.
 */
int kvfp8_timing_enable(int32_t max_launches);
int kvfp8_timing_read(double* total_ms, int64_t* launches);

/*
 * out [rows, n] = x [rows, k] weight^T for the few rows of a decode step: weight [n, k]
 * row-major, everything one dtype (f16/bf16), float32 sums, one rounding. rows 0..64, k a
 * multiple of 32, n of 16; x and weight rows 16-byte aligned. Strides in elements. The
 * projections of reference src/torch_llm/model/attention.py:57-122 and its FFN at M <= 64.
 */
int kvfp8_skinny_linear(const void* x_dev, int dtype, int64_t x_stride, int32_t rows, int32_t k,
                        const void* weight_dev, int64_t w_stride, int32_t n, void* out_dev, int64_t out_stride,
                        void* stream);

/*
 * out [rows, n] = silu(x G^T) * (x U^T) with weight [2 n, k] the rows of G then those of U:
 * kvfp8_skinny_linear followed by kvfp8_silu_mul, bit for bit, in one launch. n a multiple of
 * 8, the rest as kvfp8_skinny_linear.
 */
int kvfp8_skinny_linear_swiglu(const void* x_dev, int dtype, int64_t x_stride, int32_t rows, int32_t k,
                               const void* weight_dev, int64_t w_stride, int32_t n, void* out_dev,
                               int64_t out_stride, void* stream);

/*
 * kvfp8_skinny_linear followed by kvfp8_rope_inplace over the first `heads` heads of head_dim
 * columns, bit for bit, in one launch. heads * head_dim at most n; positions, tables and rows
 * outside them as kvfp8_rope_inplace.
 */
int kvfp8_skinny_linear_rope(const void* x_dev, int dtype, int64_t x_stride, int32_t rows, int32_t k,
                             const void* weight_dev, int64_t w_stride, int32_t n, int32_t heads, int32_t head_dim,
                             const void* positions_dev, int pos_dtype, const void* cos_table_dev,
                             const void* sin_table_dev, int table_dtype, int64_t table_rows, void* out_dev,
                             int64_t out_stride, void* stream);

/* Human-readable name of a return code (negative KVFP8_E* or positive hipError_t). */
const char* kvfp8_strerror(int code);

/* Library version string, e.g. "kvfp8 1 gfx950". */
const char* kvfp8_version(void);

/*
 * Host-side helpers that run the exact device encoding routines on the CPU
 * (shared __host__ __device__ code), so the CPU test suite can check them
 * against the oracle without a GPU. Not part of the reference interface.
 */
void kvfp8_host_encode_e4m3fn(const float* x, uint8_t* codes, int64_t n);
void kvfp8_host_quantize_rows(const float* x, int64_t rows, int32_t head_dim,
                              uint8_t* codes, float* scales);
/* x / scale of every element with its row's scale, by the device's division routine. */
void kvfp8_host_row_quotients(const float* x, int64_t rows, int32_t head_dim, float* q);

/*
 * GPU self-test of the hardware float32 -> e4m3fn converter the append kernel uses
 * for finite rows: adds to *mismatches_dev the number of float32 values with
 * |x| <= 448 (1 + 2^-19) (both signs) whose hardware code differs from the
 * software round-to-nearest-even encoder (which the CPU tests pin to the oracle).
 * Not part of the reference interface.
 */
int kvfp8_selftest_fp8_encoder(unsigned long long* mismatches_dev, void* stream);

#ifdef __cplusplus
}
#endif

#endif /* KVFP8_H */
