/*
 * mynn_hip.h -- C ABI of the MI355X (gfx950) implementation of my-nn-engine's quantized-LLM
 * inference hot path.  Plain pointers and sizes only; every pointer named "device" is HIP
 * device memory owned by the caller unless stated.  One process drives one GPU.
 *
 * Two seams of the reference engine (kcvlex/my-nn-engine) are replaced:
 *
 *  (1) the per-session model library that `SessionCUDA` dlopens -- `model_init`, `model`,
 *      `model_destroy`, `model_device_sync`, `model_memcpy`, `alloc_pinned`, `free_pinned`
 *      (generated by src/codegen/cuda.rs:2727-2825, bound in src/session/cuda.rs:53-56,323-335,
 *      src/codegen/cuda/cpp/common.cu:4-13).  Here it is a fixed Llama decoder executor
 *      configured once with `mynn_model_configure`.
 *  (2) the CUDA kernel templates of src/codegen/cuda/cpp/ (.cuh) together with the kernel
 *      choice made in src/codegen/cuda.rs; one `mynn_*` launcher per kernel, operands in the
 *      template's order, stream passed explicitly.
 *
 * Process-wide state, all of it: (a) the configuration that `mynn_model_configure` leaves for the
 * next `model_init` (the reference ABI has no other way to say it; `mynn_model_create` takes the
 * configuration as an argument and touches nothing global); (b) the scratch memory of the entry
 * points that need some and are not given any: `mynn_dequant_matmul` (M >= 2), `mynn_quantized_matmul`
 * (M >= 3), `mynn_attention` (a cache split over workgroups) and `mynn_attention_streaming`.  Each of
 * these three groups keeps one grown-on-demand block PER STREAM, locked until the call's launches are
 * made, so calls on different streams never share one and several host threads may call on one stream.
 * Growing synchronises that stream and cannot happen while the stream is being captured: a captured call
 * that needs a larger block than there is fails with MYNN_ERR_STATE (make it once before the capture).
 * A block that a captured call was given stays valid for the graph's life, also when a later call makes
 * the stream's block grow; it is shared with that stream's other calls, so replays have to be ordered
 * with those.  Products that only split K (no weight is dequantised: see the calls) use no library
 * memory at all while being captured, and one that would dequantise its weight, for which the block is
 * too small, takes the int8 weights instead; their graphs may be replayed anywhere.  The `_ws` variants take
 * the caller's block instead and touch nothing global; `mynn_attention_noalloc` uses a fixed
 * device array of the library.  Executors (seam 1) own everything they use: nothing an executor
 * launches touches library-global memory.
 *
 * Return value of every `int` function: 0 on success, a negative MYNN_ERR_* for a rejected
 * argument, or a positive hipError_t.  Nothing here calls exit().
 */
#ifndef MYNN_HIP_H_
#define MYNN_HIP_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* element types; 0/1 match the reference's FType (src/codegen/cpu/kernels/ftype.rs:4-9) */
enum { MYNN_F32 = 0, MYNN_BF16 = 1, MYNN_F16 = 2, MYNN_I8 = 3 /* only reported by the checkpoint reader */ };

enum {
    MYNN_OK = 0,
    MYNN_ERR_INVALID = -1,      /* null pointer, non-positive size, misaligned operand */
    MYNN_ERR_UNSUPPORTED = -2,  /* shape/dtype combination with no kernel */
    MYNN_ERR_STATE = -3,        /* call order (e.g. model_init before mynn_model_configure) */
    MYNN_ERR_TOO_LONG = -4,     /* prompt does not fit max_seq (LlmError::PromptTooLong) */
    MYNN_ERR_NO_PAGES = -5      /* paged KV cache: the pool has too few free pages for the rows asked for */
};

typedef void *mynn_stream; /* hipStream_t; NULL = the default stream */

const char *mynn_last_error(void);   /* text for the last failure on this thread */
int mynn_version(void);
/* device facts read once with hipGetDeviceProperties: CU count, wavefront size, LDS bytes */
int mynn_device_info(int *cu_count, int *wave_size, int *lds_bytes, char *arch, size_t arch_len);

/* ===================================================================== seam 2: kernels */

/* DequantizeLinear axis 0 -- dequantize.cuh:5-19 `dequantize_linear<Tin,Tout>`.
 * out[r,c] = (T)((f32)x[r,c] * scale[r]); x int8 [rows,cols], scale/out dtype. */
int mynn_dequantize_linear(void *out, const int8_t *x, const void *scale,
                           size_t rows, size_t cols, int dtype, mynn_stream s);

/* DequantMatMul, M == 1 -- dequant_gemv.cuh:12-59 `dequant_gemv<TAct,TOut>(out,act,wq,scale,N,K)`.
 * out[n] = (TOut)(scale[n] * sum_k (f32)act[k] * (f32)wq[n,k]); wq int8 [N,K] row-major,
 * K % 16 == 0, wq 16-byte aligned.  scale and out share out_dtype. */
int mynn_dequant_gemv(void *out, const void *act, const int8_t *wq, const void *scale,
                      int N, int K, int act_dtype, int out_dtype, mynn_stream s);

/* DequantMatMul, any M -- the kernel choice of cuda.rs:1518-1652:
 *   M >= 16, 16-bit act+scale, K % 8 == 0 -> matrix-core GEMM with W dequantised to the 16-bit
 *        type (scale folded in, one rounding) before the MMA (dequant_matmul_wmma.cuh:87-192);
 *   otherwise scale-after-sum per (m,n) (dequant_gemv.cuh / dequant_matmul.cuh:12-51).
 * act [M,K], out [M,N].
 * For M >= 16 the f32 sum of an output may run over several ranges of K, each summed up from zero and added in their
 * order.  Their number is a function of M, N, K and the type alone: this call, the same call captured into a graph,
 * mynn_dequant_matmul_ws with any tile and mynn_dequant_matmul_prepared give the same bits.  (Another M may be summed up
 * in another number of ranges, so a row's last bits can depend on how many rows it is multiplied with.) */
int mynn_dequant_matmul(void *out, const void *act, const int8_t *wq, const void *scale,
                        int M, int N, int K, int act_dtype, int out_dtype, mynn_stream s);

/* The same with the caller's scratch memory: for M >= 16 (16-bit operands) `workspace`
 * (mynn_dequant_matmul_workspace_bytes(...) bytes, 16-byte aligned, 0 = none needed) takes the dequantised weight of a
 * large product or the partial sums of a small one; nothing global is touched, so the call can be captured into a graph and calls on several streams
 * may overlap when their workspaces differ.  gemm_tile forces the workgroup tile of the matrix-core GEMM:
 * 0 = chosen per shape, 1 = 256x128, 2 = 256x256 with operands staged through registers, 3 = 256x256 and
 * 4 = 256x320 with operands loaded straight into LDS (3 and 4 fall back to 1 when K % 64 != 0, and every forced tile
 * is 1 where the sum runs over several ranges of K). */
size_t mynn_dequant_matmul_workspace_bytes(int M, int N, int K, int act_dtype, int out_dtype);
int mynn_dequant_matmul_ws(void *out, const void *act, const int8_t *wq, const void *scale,
                           int M, int N, int K, int act_dtype, int out_dtype,
                           void *workspace, size_t workspace_bytes, int gemm_tile, mynn_stream s);

/* Prepare once, multiply many (M >= 16, 16-bit types): `wt` (mynn_dequant_weight_bytes(N, K) bytes,
 * 16-byte aligned, caller-owned) receives W dequantised to `dtype` with the scale folded in -- the values
 * every call of mynn_dequant_matmul computes again -- and mynn_dequant_matmul_prepared multiplies by it:
 * out[M,N] = act[M,K] . wt^T, bit-identical to mynn_dequant_matmul on the same operands. */
size_t mynn_dequant_weight_bytes(int N, int K);
int mynn_dequant_weight_prepare(void *wt, const int8_t *wq, const void *scale, int N, int K, int dtype,
                                mynn_stream s);
int mynn_dequant_matmul_prepared(void *out, const void *act, const void *wt, int M, int N, int K,
                                 int dtype, int gemm_tile, mynn_stream s);

/* Measurement aid, no counterpart in the reference, process-wide: 1 = the few-row gate/up GEMM (M <= 32, 768 row
 * blocks of 32 and more) of a batched decode step runs its loads alone (no LDS, no conversion, no MFMA, no barrier), 2 = everything but the MFMAs,
 * 0 = the product kernel.  The ablated launches compute garbage; only their duration means anything
 * (bench.py --workload decode_batch --skinny-ablation). */
void mynn_skinny_set_ablation(int mode);

/* Measurement aid, no counterpart in the reference: the weight stream of the batch-1 decode GEMV alone -- the
 * grid, row groups and per-lane 16-byte non-temporal loads mynn_dequant_gemv issues for a 16-bit [N,K] product,
 * without activation, arithmetic or store.  Launched the way a decode step launches its GEMVs (one after the other
 * on a stream, a different matrix each time) its duration is the floor of such a launch; empty != 0 launches the
 * same grid with nothing to read (the cost of the dispatch itself).  sink: 4 bytes of device memory, never
 * written in practice.  bench.py --workload gemv and the default line's roofline.floor use it. */
int mynn_gemv_read_probe(const int8_t *wq, void *sink, int N, int K, int empty, mynn_stream s);

/* QuantizedMatMul -- quantized_gemv_int8.cuh:13-51, quantized_matmul_int8.cuh:112-269,
 * CPU twin src/codegen/cpu/kernels/qgemv_i8i8.rs:38-80.
 * acc[m,n] = sum_k lhs[m,k]*rhs[n,k] in exact int32;
 * out[m,n] = (T)((f32)acc * lhs_scale[m] * rhs_scale[n]).  K % 32 == 0.
 * `acc_out` (device int32 [M,N]) may be NULL; `out` may be NULL when only acc is wanted. */
int mynn_quantized_matmul(void *out, int32_t *acc_out, const int8_t *lhs, const void *lhs_scale,
                          const int8_t *rhs, const void *rhs_scale,
                          int M, int N, int K, int dtype, mynn_stream s);

/* DynamicQuantizeLinear -- dynamic_quantize_linear.cuh:39-153
 * `dynamic_quantize_linear_kernel(y,y_scale,y_zero_point,x,axis_dim,inner_size)`.
 * symmetric: int8, scale = amax/127 (1 for an all-zero slice), y = clamp(round_half_away(x*(1/s)),
 *   -127,127) -- the CPU backend's rule (cpu/kernels/dynquant_i8.rs:13-37), zero_point 0;
 * asymmetric: ONNX uint8 form, round-half-even.  y_zero_point may be NULL when symmetric. */
int mynn_dynamic_quantize_linear(void *y, void *y_scale, void *y_zero_point, const void *x,
                                 int axis_dim, int inner_size, int dtype, int symmetric,
                                 mynn_stream s);

/* Attention -- attention.cuh:495-606 `attention_decode`, :45-314 `attention_tc`, :316-489
 * `attention`, chosen as cuda.rs:1194-1403 does (seq_q == 1 -> decode kernel).
 * Q,out [B,Hq,Sq,D]; K,V [B,Hkv,cache_seq_len,D]; kv head = q head / (Hq/Hkv).
 * Keys visited for query row sq: [0, min(active, q_pos_offset + sq + 1 if causal, cache_seq_len)).
 * `active_seq_kv` is the host scalar the reference reads at launch time; when `d_active`
 * (device int32[1]) is non-NULL it is read on the device instead (graph-replay safe) and
 * q_pos_offset becomes *d_active - Sq.
 * kv_int8 != 0: K,V are int8 with per-token scales k_scale,v_scale [B,Hkv,cache_seq_len]. */
int mynn_attention(void *out, const void *Q, const void *K, const void *V,
                   const void *k_scale, const void *v_scale, float scale, int is_causal,
                   int B, int Sq, int active_seq_kv, const int32_t *d_active, int cache_seq_len,
                   int q_pos_offset, int num_q_heads, int num_kv_heads, int head_dim,
                   int dtype, int kv_int8, mynn_stream s);

/* The same with the additive mask of operator slot 3 (src/graph/operator.rs:1024-1042) and with the
 * caller's scratch memory.  mask (dtype, may be NULL): score(b, h, sq, key) = q.k * scale
 * + mask[(b * Hq + h) * mask_outer_stride + sq * mask_row_stride + key], added before the softmax to the
 * keys that the length and causal rules admit; a stride of 0 broadcasts that dimension
 * (src/codegen/cuda.rs:1297-1323, attention.cuh:436-451).  workspace: mynn_attention_workspace_bytes(...)
 * bytes -- enough for every active length up to cache_seq_len --, 16-byte aligned (0 = none needed: the call
 * then accepts NULL); nothing global is touched. */
size_t mynn_attention_workspace_bytes(int B, int Sq, int cache_seq_len, int num_q_heads, int num_kv_heads,
                                      int head_dim, int dtype, int kv_int8);
int mynn_attention_ws(void *out, const void *Q, const void *K, const void *V,
                      const void *mask, long mask_outer_stride, long mask_row_stride,
                      const void *k_scale, const void *v_scale, float scale, int is_causal,
                      int B, int Sq, int active_seq_kv, const int32_t *d_active, int cache_seq_len,
                      int q_pos_offset, int num_q_heads, int num_kv_heads, int head_dim,
                      int dtype, int kv_int8, void *workspace, size_t workspace_bytes, mynn_stream s);

/* mynn_attention for callers that cannot allocate device memory (code under HIP graph capture, tight serving
 * loops, harnesses that forbid hipMalloc).  No counterpart in the reference.  Same operands and results as
 * mynn_attention, bit for bit; the partial results of a cache that several workgroups share go to a fixed
 * 8 MiB device array of the library (one per GPU, held until the process ends) instead of grown-on-demand
 * memory, and the call makes no hipMalloc / hipFree.  A shape whose partial results exceed the array is refused
 * with MYNN_ERR_UNSUPPORTED (mynn_attention_workspace_bytes says how much a shape needs).  All calls on one GPU
 * share the array: calls that overlap on one GPU (different streams) race. */
int mynn_attention_noalloc(void *out, const void *Q, const void *K, const void *V,
                           const void *k_scale, const void *v_scale, float scale, int is_causal,
                           int B, int Sq, int active_seq_kv, const int32_t *d_active, int cache_seq_len,
                           int q_pos_offset, int num_q_heads, int num_kv_heads, int head_dim,
                           int dtype, int kv_int8, mynn_stream s);

/* Paged K/V.  No counterpart in the reference, whose caches are contiguous [B,Hkv,max_seq,D] buffers reserved in
 * full per session (crates/llm/src/session.rs:284-394).  K_pool, V_pool: [n_pages, Hkv, page_rows, D] (an int8
 * cache: scale pools [n_pages, Hkv, page_rows]); page_rows a power of two >= 32.  page_table (device
 * int32 [B, pages_per_seq]): cache row r of sequence b is row r % page_rows of pool page
 * page_table[b * pages_per_seq + r / page_rows]; the entries of every page with a row below the active
 * length must name pages of the pool (they are addresses: the call cannot check device memory), the rest
 * are not read.  Same arithmetic as mynn_attention on the rows gathered into a contiguous cache of
 * pages_per_seq * page_rows rows, and the same bits whenever that call takes the same kernel.
 * Sq == 1: 16-bit or int8 K/V, head_dim 64 / 128, 1 / 2 / 4 / 8 query heads per kv head.  Sq > 1 (prefill,
 * matrix cores): 16-bit K/V, head_dim 64 / 128, page_rows >= 64, pages_per_seq <= 64.
 * A key range of the Sq == 1 kernel spans at most 62 pages; longer contexts are cut into more ranges.
 * workspace: mynn_attention_paged_workspace_bytes(...) bytes -- enough for every active length up to
 * pages_per_seq * page_rows --, 16-byte aligned (0 = none needed). */
size_t mynn_attention_paged_workspace_bytes(int B, int Sq, int pages_per_seq, int page_rows,
                                            int num_q_heads, int num_kv_heads, int head_dim);
int mynn_attention_paged(void *out, const void *Q, const void *K_pool, const void *V_pool,
                         const void *k_scale_pool, const void *v_scale_pool,
                         const int32_t *page_table, int pages_per_seq, int page_rows,
                         float scale, int is_causal, int B, int Sq, int active_seq_kv,
                         const int32_t *d_active, int q_pos_offset, int num_q_heads, int num_kv_heads,
                         int head_dim, int dtype, int kv_int8, void *workspace, size_t workspace_bytes,
                         mynn_stream s);
/* KVCacheUpdate into a pool: row offset+t of (b, kv head) <- new_kv[b, kv head, t, :] through the table. */
int mynn_kvcache_update_paged(void *pool, const void *new_kv, int offset, int B, int Hkv, int S_new,
                              int D, int dtype, const int32_t *page_table, int pages_per_seq,
                              int page_rows, mynn_stream s);

/* The pages themselves: a pool is a free list of page numbers (host memory only -- the pool BUFFERS are the
 * caller's, one K and one V buffer per layer, all indexed by the same page numbers), a page set is the
 * table of the `batch` sequences of one session (its prefill and its decode executor share it), kept in
 * host memory and mirrored on the device.  Sets on one pool share its pages: a set takes pages when its
 * sequences reach them (mynn_kv_pages_reserve; the executors call it themselves before every step) and
 * gives them back with mynn_kv_pages_release.  Thread-safe across sets; one set is used by one thread
 * at a time.  reserve / release copy the table synchronously: no launch that reads it may be in flight.
 * Lifetimes: a pool outlives its page sets (mynn_kv_pool_destroy refuses otherwise), a page set outlives the
 * models made with it (they keep the pointer; model_destroy does not touch the set). */
typedef struct mynn_kv_pool mynn_kv_pool;
typedef struct mynn_kv_pages mynn_kv_pages;
mynn_kv_pool *mynn_kv_pool_create(int n_pages, int page_rows);
int mynn_kv_pool_free_pages(const mynn_kv_pool *pool);
int mynn_kv_pool_destroy(mynn_kv_pool *pool);              /* MYNN_ERR_STATE while a set still uses it */
mynn_kv_pages *mynn_kv_pages_create(mynn_kv_pool *pool, int batch, int max_seq /* multiple of page_rows */);
/* pages for rows [0, rows) of every sequence: MYNN_ERR_TOO_LONG beyond max_seq, MYNN_ERR_NO_PAGES when
 * the pool has too few left (nothing is taken then) */
int mynn_kv_pages_reserve(mynn_kv_pages *pages, int64_t rows);
int mynn_kv_pages_release(mynn_kv_pages *pages);           /* every page back to the pool; the set stays usable */
int mynn_kv_pages_mapped_rows(const mynn_kv_pages *pages);
int mynn_kv_pages_per_seq(const mynn_kv_pages *pages);
const int32_t *mynn_kv_pages_table(const mynn_kv_pages *pages);          /* device int32 [batch, pages_per_seq], -1 = unmapped */
int mynn_kv_pages_table_host(const mynn_kv_pages *pages, int32_t *out);  /* the same, copied to host memory */
int mynn_kv_pages_destroy(mynn_kv_pages *pages);

/* KVCacheUpdate -- kvcache_update.cuh:6-26: cache[bh, offset+t, :] = new[bh, t, :] in place. */
int mynn_kvcache_update(void *cache, const void *new_kv, int offset, int BH, int S_new,
                        int max_seq, int D, int dtype, mynn_stream s);

/* QuantizingKVCacheUpdate -- quantizing_kvcache_update.cuh:16-70 with the CPU backend's rounding
 * (translator.rs:4090-4372): s = amax/127, q = clamp(trunc(x*(127/amax) +/- 0.5), -128, 127). */
int mynn_quantizing_kvcache_update(int8_t *cache, void *scale, const void *new_kv, int offset,
                                   int BH, int S_new, int max_seq, int D, int dtype,
                                   mynn_stream s);

/* Streaming KV (sink + ring cache), the kernel-level operators -- common.cuh:55-60 `ring_phys_index`:
 * the key of recency rank r lives in cache row r for r < ring_sink, else in row
 * ring_sink + (ring_start + r - ring_sink) % ring_window; ring_window == 0 switches the map off.
 *
 * KVCacheUpdate with the ring inputs (kvcache_update.cuh:12-26, operator slots 3-5 of
 * builder.rs:304-321): cache[bh, ring_phys_index(offset + t), :] = new[bh, t, :], rows in increasing t. */
int mynn_kvcache_update_streaming(void *cache, const void *new_kv, int offset, int BH, int S_new,
                                  int max_seq, int D, int ring_sink, int ring_window, int ring_start,
                                  int dtype, mynn_stream s);

/* QuantizingKVCacheUpdate with the ring inputs (quantizing_kvcache_update.cuh:24-36, builder.rs:324-342):
 * the quantised row and its scale go to row ring_phys_index(offset + t). */
int mynn_quantizing_kvcache_update_streaming(int8_t *cache, void *scale, const void *new_kv, int offset,
                                             int BH, int S_new, int max_seq, int D, int ring_sink,
                                             int ring_window, int ring_start, int dtype, mynn_stream s);

/* Attention with the ring inputs (operator slots 7-9, attention.cuh:386-404, 436-438, 548-550): keys are
 * enumerated by recency rank 0..active_seq_kv-1, rank r is read from cache row ring_phys_index(r), the
 * causal rule compares query positions with ranks.  Other arguments as mynn_attention; the length is
 * the host scalar.
 * cos_t, sin_t ([rows, head_dim], dtype) and kv_position (device int64, one entry per rank) -- slots
 * 10-12, all three or none: K is rotated inside the operator (attention.cuh:407-420, 559-570): the
 * dequantised key of rank r is rotated half-split by table row kv_position[r], in f32, and scores,
 * softmax and P.V stay in f32; the result is rounded once. */
int mynn_attention_streaming(void *out, const void *Q, const void *K, const void *V,
                             const void *k_scale, const void *v_scale, float scale, int is_causal,
                             int B, int Sq, int active_seq_kv, int cache_seq_len, int q_pos_offset,
                             int num_q_heads, int num_kv_heads, int head_dim, int dtype, int kv_int8,
                             int ring_sink, int ring_window, int ring_start,
                             const void *cos_t, const void *sin_t, const int64_t *kv_position,
                             mynn_stream s);
/* The same with the caller's scratch memory (the rank-ordered rows and the partial results behind them):
 * mynn_attention_streaming_workspace_bytes(...) bytes -- enough for every active length and ring up to the
 * cache length; rope_on = whether cos_t / sin_t / kv_position will be given --, 256-byte aligned.  Nothing
 * global is touched and nothing is allocated. */
size_t mynn_attention_streaming_workspace_bytes(int B, int Sq, int cache_seq_len, int num_q_heads,
                                                int num_kv_heads, int head_dim, int dtype, int kv_int8,
                                                int rope_on);
int mynn_attention_streaming_ws(void *out, const void *Q, const void *K, const void *V,
                                const void *k_scale, const void *v_scale, float scale, int is_causal,
                                int B, int Sq, int active_seq_kv, int cache_seq_len, int q_pos_offset,
                                int num_q_heads, int num_kv_heads, int head_dim, int dtype, int kv_int8,
                                int ring_sink, int ring_window, int ring_start,
                                const void *cos_t, const void *sin_t, const int64_t *kv_position,
                                void *workspace, size_t workspace_bytes, mynn_stream s);

/* RMSNormalization -- rms_norm.cuh:9-59: y = (x * (1/sqrt(mean(x^2)+eps))) * w per row. */
int mynn_rms_norm(void *out, const void *x, const void *w, int rows, int dim, float eps,
                  int dtype, mynn_stream s);

/* Rope -- rope.cuh:18-46: half-split rotation, table row chosen by position[s] (device int64).
 * x,out [outer,S,D]; cos,sin [max_seq,D]. */
int mynn_rope(void *out, const void *x, const void *cos_t, const void *sin_t,
              const int64_t *position, int outer, int S, int D, int dtype, mynn_stream s);

/* Gather axis 0 -- gather.cuh:5-21: out[i,:] = data[idx[i] (+rows if negative), :]. */
int mynn_gather_rows(void *out, const void *data, const int64_t *idx, int n_idx, int rows,
                     size_t row_bytes, mynn_stream s);

/* fused elementwise groups (generated by cuda/kernel.rs:723-957 in the reference): f32 compute,
 * one rounding.  swiglu = silu(gate)*up, add = a+b. */
int mynn_swiglu(void *out, const void *gate, const void *up, size_t n, int dtype, mynn_stream s);
int mynn_add(void *out, const void *a, const void *b, size_t n, int dtype, mynn_stream s);

/* greedy argmax with the reference's tie rule (crates/llm/src/session.rs:683-690, the LAST
 * maximum wins); result is a device int32[1]. */
int mynn_argmax_last(int32_t *out_index, const void *logits, int n, int dtype, mynn_stream s);

/* ===================================================================== seam 1: model library */

typedef struct {
    int n_layers, hidden, n_heads, n_kv_heads, head_dim, ffn, vocab, max_seq;
    float eps;
    float rope_theta;
    int dtype;        /* activation / scale / KV type: MYNN_F16 or MYNN_BF16 (MYNN_F32 unsupported) */
    int seq_q;        /* 1 = decode graph, >1 = prefill graph of that length (Mode::Prefill{len}) */
    int batch;        /* sequences per step; the reference's crates/llm is batch 1 */
    int weights_int8; /* 1: linear weights + embed table are int8 [N,K] with per-row scales
                         (model.int8.safetensors); 0: plain cfg.dtype matrices, the scale slots of
                         `initializer` are ignored (the reference's bf16 checkpoints) */
    int quant_kv_cache; /* BuildOptions::quant_kv_cache (crates/llm/src/decoder.rs:672, 405-470): the KV
                         cache is int8 with one scale per token row; `session_state` then holds four
                         buffers per layer: past_key i8 [B,Hkv,max_seq,D], past_value, past_key_scale
                         cfg.dtype [B,Hkv,max_seq], past_value_scale */
    int quantize_activations; /* Options::quantize_activations (src/options.rs:76, the pass
                         src/transform/optimize/quantize_activations.rs): every int8 linear with
                         K % 32 == 0 runs as DynamicQuantizeLinear (per row, symmetric) +
                         QuantizedMatMul (int8 x int8 -> exact int32) instead of DequantMatMul */
    int streaming_kv; /* BuildOptions::streaming_kv (crates/llm/src/decoder.rs:673, 281-347, 472-487): the
                         graph takes four more inputs [ring_sink, ring_window, ring_start, kv_position] and
                         keeps K UN-ROTATED in the cache (written through the sink + ring slot map); the
                         cached keys are rotated by kv_position before every attention.  Batch 1.  past_len
                         is the session's unbounded stream position and may lie past ring_sink +
                         ring_window (and past max_seq): the operators then do exactly what the reference's
                         CUDA kernels do with those inputs -- the update writes row
                         ring_phys_index(past_len + t) with the session's ring_start (kvcache_update.cuh:21),
                         the attention enumerates ranks 0 .. active-1 through the same map
                         (attention.cuh:397, 549), and with an int8 cache rotates the key of RANK r by
                         kv_position[r] (attention.cuh:416, 560) although the session fills that table by
                         slot (session.rs:604-635) */
    /* ---- executor options with no counterpart in the reference; 0 = the library's choice */
    int gemm_tile;      /* workgroup tile of this model's matrix-core GEMMs, as mynn_dequant_matmul_ws */
    int unfused_decode; /* 1: every op of a batch-1 decode step is a launch of its own (5 per layer + 3).
                         0: dependent ops share launches where the shape allows (int8 weights, head_dim
                         64 / 128, max_seq <= 2048 / 1024, hidden <= 4096): a layer's q|k|v projection,
                         attention and o projection are one launch, the first makes the embedding row
                         itself, the lm_head launch finds the greedy token and moves the loop state on --
                         3 launches per layer + 1, with a 16-bit and with an int8 KV cache (the new row is
                         then quantised inside the launch, as QuantizingKVCacheUpdate does it).  Bit-identical
                         logits and tokens with a 16-bit cache; with an int8 cache the two forms agree as
                         closely as either agrees with the reference.  With
                         quantize_activations a linear's RMSNorm, quantiser, int8 product and residual / SwiGLU
                         are one launch (5 per layer + 3 instead of 16 per layer + 5; the same operators, but the
                         row's sum of squares is taken in another order, so results agree within the path's
                         quantisation noise, not bit for bit). */
    int handover_spin_limit; /* polls a workgroup of a shared launch makes for its producer's output before
                         it gives up: 0 = 400000; n > 0 = n; -1 = none beyond the first two looks (test
                         knob: forces the recovery described at mynn_model_step) */
    int weight_arena;   /* 1: model_init copies every int8 linear weight and scale (the caller's o / down / lm_head
                         included) into ONE device allocation in the order a step reads them, instead of keeping
                         the caller's buffers and separate repacked copies (1 byte per weight of extra memory) */
    int kv_page_rows;   /* > 0: paged KV cache with this many rows per page (a power of two >= 64, dividing max_seq;
                         at most 64 pages per sequence for a prefill model).  `session_state` then holds per
                         layer the K pool and the V pool, [n_pages, Hkv, kv_page_rows, D] in cfg.dtype, and after
                         the last layer ONE more entry: the session's mynn_kv_pages (made with this batch and
                         max_seq over a pool of the same page size).  Every step reserves the pages its rows need
                         before it launches (MYNN_ERR_NO_PAGES when the pool is exhausted: nothing ran).
                         head_dim 64 / 128, 1 / 2 / 4 / 8 query heads per kv head; not with streaming_kv.  With
                         quant_kv_cache (decode models only, seq_q == 1): four pools per layer -- K codes, V codes
                         (int8), K scales, V scales [n_pages, Hkv, kv_page_rows] in cfg.dtype -- then the page set.
                         Batched decode attention runs in the kernel made for large batch x context products; a
                         batch-1 decode model takes the same single-launch layer as with contiguous caches (up to
                         64 pages per sequence; beyond that 6 launches per layer + 3).  Where the executor
                         with contiguous caches takes the same kernels (prefill, batched decode) the results are
                         the same bits: the same rows are walked in the same order. */
    int qkv_bias;       /* 1: the q, k and v projections have a bias (model_type "qwen2",
                         crates/llm/src/decoder.rs:542-600): `initializer` holds it behind each of the three
                         weights (q_w,q_s,q_b, k_w,k_s,k_b, v_w,v_s,v_b; [N] in cfg.dtype, 19 entries per layer)
                         and the executor adds it to the stored projection, rounding once more, as the graph's
                         Add node does (decoder.rs:167-184).  The q|k|v projection then keeps a launch of its
                         own in every executor. */
} mynn_model_config;

/* Describes the graph the next `model_init` instantiates (the reference bakes this into the
 * generated library; a fixed library needs it said once).  crates/llm/src/decoder.rs:667-865.
 * Process-wide: callers serialise configure + model_init as the reference serialises session
 * creation (CUDA_LOCK, src/session/cuda.rs:36-40). */
int mynn_model_configure(const mynn_model_config *cfg);
/* mynn_model_configure + model_init in one call that touches no process-wide state. */
void *mynn_model_create(const mynn_model_config *cfg, void **initializer, void **session_state);

/* One set of derived weight copies for all executors of a session.  No counterpart in the reference, whose sessions
 * share the checkpoint's device buffers by name (PersistentBuffers, src/session.rs:284-394) and derive nothing from
 * them.  Here an executor derives copies at init -- q|k|v rows concatenated and gate/up rows interleaved (decode),
 * every weight dequantised once to the 16-bit type (prefill, matrix cores), an int8 copy tiled for streaming
 * (2..64 rows), int8 gate/up interleaved in groups of 32 (quantize_activations prefill) -- and a prefill, a decode
 * and a batched executor made by mynn_model_create each derive their own.  mynn_weight_set_create makes the holder
 * (cfg: the shapes, dtype, weights_int8 and qkv_bias are what matters; initializer as mynn_model_create), and
 * mynn_model_create_shared builds an executor on it: each kind of copy is made by the first executor that needs it
 * and reused by the rest.  The set lives until its handle is destroyed AND every executor built on it is.
 * mynn_weight_set_stats: bytes[4] = {decode repacks, 16-bit resident copy, tiled int8 copy, W8A8 gate/up interleave},
 * holders = the handle + executors still alive. */
typedef struct mynn_weight_set mynn_weight_set;
mynn_weight_set *mynn_weight_set_create(const mynn_model_config *cfg, void **initializer);
void *mynn_model_create_shared(const mynn_model_config *cfg, mynn_weight_set *set, void **session_state);
int mynn_weight_set_stats(mynn_weight_set *set, size_t *bytes, int *holders);
void mynn_weight_set_destroy(mynn_weight_set *set);

/* Reference ABI (cuda.rs:2727-2773).  `initializer` = device pointers in this order:
 *   [0] embed_tokens int8 [vocab,hidden]   [1] its scale [vocab]
 *   per layer l, base 2+16*l: input_layernorm, q_w,q_s, k_w,k_s, v_w,v_s, o_w,o_s,
 *                             post_attention_layernorm, gate_w,gate_s, up_w,up_s, down_w,down_s
 *   then final norm, lm_head int8 [vocab,hidden], lm_head scale.
 * `session_state` = per layer: past_key, past_value, each [batch,Hkv,max_seq,D] in cfg.dtype,
 * zero-initialised by the caller (src/session.rs:284-394) and shared between a prefill and a
 * decode model.  The library makes its own repacked copies of q/k/v and gate/up; the caller's
 * buffers are only read.  Returns NULL on failure (see mynn_last_error).
 * Two differences from the generated library, which a fixed one cannot avoid: the order above is
 * this library's own (the reference passes the graph's initializers in graph order, which depends
 * on how the graph was built), and the RoPE tables, which the reference passes as two more
 * initializers (crates/llm/src/builder.rs:359-393), are computed inside from head_dim, max_seq and
 * rope_theta with the same arithmetic (mynn_rope_table). */
void *model_init(void **initializer, void **session_state);
/* input  = HOST pointers [input_ids i64[batch,seq_q], position_id i64[seq_q], past_len i64,
 *                         active_seq_kv i64]  (crates/llm/src/session.rs:508-519); a streaming_kv
 *          model takes four more: [ring_sink i64, ring_window i64, ring_start i64,
 *          kv_position i64[max_seq]] (session.rs:572-597)
 * output = HOST pointer  [logits cfg.dtype [batch,seq_q,vocab]].  Synchronous.
 * The reference's `model` is void and exits the process on a device error; this one returns, prints
 * the failure on stderr, and keeps the status of the state's last `model` call (0, MYNN_ERR_* or a
 * hipError_t) for mynn_model_last_status -- which a SessionHIP::run checks after the void call --
 * with the text in mynn_last_error(). */
void model(void *state, void **output, void **input);
int mynn_model_last_status(void *state);
void model_destroy(void *state);
void model_device_sync(void);
int  model_memcpy(void *dst, const void *src, size_t n, int kind /* hipMemcpyKind 0..3 */);
void *alloc_pinned(size_t n);
void free_pinned(void *p);

/* `model` with a status code and no logits copy: runs the step and leaves the greedy token
 * (argmax, last maximum) of the last row of each sequence in `next_token` (host int32[batch]).
 * `logits_host` may be NULL.
 * Shared launches (see unfused_decode) hand data between workgroups of one grid through memory,
 * with bounded waits.  If a wait runs out (the device is shared or serialised so that a producer
 * was not running), the step's results are discarded, the executor switches to one op per launch
 * -- the same arithmetic, bit-identical results, no workgroup waits for another --, captures its
 * step again and repeats the step from the host-side inputs; the call still returns 0.  After 256
 * steps without a give-up it goes back to the shared launches (whatever held a producer up has
 * usually gone by then); every further give-up doubles that number.
 * mynn_model_set_handover_rearm changes it (0: stay with one op per launch for good),
 * mynn_model_handover_failures reports how often a step gave up. */
int mynn_model_step(void *state, const int64_t *input_ids, const int64_t *position_id,
                    int64_t past_len, int64_t active_seq_kv, int32_t *next_token, void *logits_host);
/* the same for a streaming_kv model: the four ring inputs of session.rs:572-597 (kv_position: host
 * int64[max_seq]) */
int mynn_model_step_streaming(void *state, const int64_t *input_ids, const int64_t *position_id,
                              int64_t past_len, int64_t active_seq_kv, int64_t ring_sink, int64_t ring_window,
                              int64_t ring_start, const int64_t *kv_position, int32_t *next_token,
                              void *logits_host);
int mynn_model_handover_failures(void *state);
int mynn_model_set_handover_rearm(void *state, int clean_steps);
/* paged KV cache: every page of the model's page set back to the pool (mynn_kv_pages_release; the prefill and the
 * decode model of a session share the set); 0 and nothing done for a model with contiguous caches.  mynn_llm_reset
 * calls it. */
int mynn_model_release_kv_pages(void *state);
/* greedy token (last maximum) of logits row `row` (0 <= row < batch*seq_q) of the last step */
int mynn_model_argmax_row(void *state, int row, int32_t *token);
/* device pointer of the last step's logits [batch,seq_q,vocab] (valid until the next step) */
const void *mynn_model_logits_device(void *state);
/* rebuilds nothing, only reports: activation-arena bytes, kernel launches per step, whether
 * the step replays a captured hipGraph */
int mynn_model_stats(void *state, size_t *arena_bytes, int *launches_per_step, int *graph);
/* decode loop kept on the device: feeds `token` at `past_len`, then `n_steps-1` further greedy
 * tokens without a host round trip per step; writes the n_steps produced ids to out_tokens (host).
 * Same result as n_steps calls of mynn_model_step.  A batch-1 model replays graphs of 32 steps
 * where n_steps allows (a graph launch costs the device a few microseconds of its own). */
int mynn_model_decode_loop(void *state, int32_t token, int64_t past_len, int n_steps,
                           int32_t *out_tokens);
/* per-launch timing of one step with HIP events on the executor's stream (no graph): fills up to
 * `cap` entries of name / milliseconds / algorithmic bytes / flops (0 where not a contraction);
 * returns the number of launches.  profile_step: batch-1 decode model, one token at past_len;
 * profile: any model, same operands as mynn_model_step. */
typedef struct { const char *name; float ms; double bytes; double flops; } mynn_kernel_time;
int mynn_model_profile_step(void *state, int32_t token, int64_t past_len,
                            mynn_kernel_time *out, int cap);
int mynn_model_profile(void *state, const int64_t *input_ids, const int64_t *position_id,
                       int64_t past_len, int64_t active_seq_kv, mynn_kernel_time *out, int cap);

/* ===================================================================== host side of crates/llm */

/* per-output-channel int8 quantiser (crates/llm/src/quantize.rs:124-169), host memory:
 * scale = amax/127 (1 for a zero row), q = clamp(round_half_away(w/scale), -128, 127). */
int mynn_quantize_per_channel(int8_t *q, void *scale, const float *w, size_t rows, size_t cols,
                              int scale_dtype);
/* RoPE tables (crates/llm/src/builder.rs:359-393), host memory [max_seq, head_dim]. */
int mynn_rope_table(void *cos_t, void *sin_t, int max_seq, int head_dim, float base, int dtype);

/* LlmSession (crates/llm/src/session.rs:311-537): decode session + optional prefill session
 * over shared weights and KV buffers, greedy generate loop, past_len bookkeeping. */
typedef struct mynn_llm mynn_llm;
/* decode_state / prefill_state come from model_init (prefill_state may be NULL: the prompt is
 * then fed token by token, session.rs:376-381). */
mynn_llm *mynn_llm_create(void *decode_state, void *prefill_state, int prefill_len, int max_seq,
                          int64_t eos_token_id);
void mynn_llm_destroy(mynn_llm *llm);
void mynn_llm_reset(mynn_llm *llm);                       /* past_len = 0; a paged cache gives its pages back */
int64_t mynn_llm_past_len(const mynn_llm *llm);
void mynn_llm_set_past_len(mynn_llm *llm, int64_t past_len); /* stop-string rewind, session.rs:411-424 */
/* DecodeKind::LlamaStreaming { sink, window } (session.rs:87-91, 176-241): the sessions' models were built
 * with streaming_kv; every step gets the ring inputs of streaming_decode_inputs / streaming_prefill_inputs
 * (session.rs:539-635), and the max_seq checks of the generate loop are off (session.rs:352-370).
 * Needs window > 0, sink + window <= max_seq, prefill_len <= window. */
int mynn_llm_set_streaming(mynn_llm *llm, int sink, int window);
/* generate_ids without tokenizer: returns the number of new ids written to out (<= max_new),
 * MYNN_ERR_TOO_LONG when the prompt does not fit, another negative MYNN_ERR_*, or -1000-e for
 * hipError_t e.  After the prompt the decode steps run in runs of mynn_model_decode_loop (32 steps
 * when an end-of-sequence id is set, up to 256 otherwise) where the decode model has that loop: ids,
 * the stop at the end-of-sequence id and past_len are those of one mynn_model_step per token
 * (session.rs:508-537); cache rows a run computed past the stop lie beyond past_len and are
 * overwritten by the next turn. */
int mynn_llm_generate_ids(mynn_llm *llm, const int64_t *prompt_ids, size_t n_prompt,
                          size_t max_new_tokens, int64_t *out);
/* the same loop over a caller-supplied step function (token, past_len) -> next token, for
 * sessions that are not a Llama graph (DecodeKind::Mock, session.rs:508-513) */
typedef int64_t (*mynn_step_fn)(void *user, int64_t token, int64_t past_len);
mynn_llm *mynn_llm_create_with_step(mynn_step_fn step, void *user, int max_seq, int64_t eos_token_id);

/* ===================================================================== checkpoints (host) */

/* HfWeights (crates/llm/src/hf_weights.rs:65-159): `path` is a .safetensors file or a model
 * directory, searched in the reference's order: model.int8.safetensors, then the shards named by
 * model.safetensors.index.json, then model.safetensors.  Shards are memory-mapped; `data` pointers
 * stay valid until close.  NULL + mynn_last_error() on failure. */
typedef struct mynn_weights mynn_weights;
mynn_weights *mynn_weights_open(const char *path);
void mynn_weights_close(mynn_weights *w);
int mynn_weights_count(const mynn_weights *w);
const char *mynn_weights_name(const mynn_weights *w, int i);          /* file order */
/* dtype: MYNN_F32 / MYNN_BF16 / MYNN_F16 / MYNN_I8; shape holds up to 8 extents; any out may be NULL */
int mynn_weights_find(const mynn_weights *w, const char *name, int *dtype, int64_t *shape, int *ndim,
                      const void **data, size_t *nbytes);

/* quantize_safetensors_int8 / _dir (crates/llm/src/quantize.rs:28-42, 249-337): tensors whose name ends
 * in one of q/k/v/o/gate/up/down_proj.weight, lm_head.weight, embed_tokens.weight become int8 [out,in]
 * plus "<name>.scale" (bf16 [out]); fp16 tensors that are not quantised are stored as bf16, everything
 * else is copied.  `src` is a file or a model directory (its fp shards, never model.int8.safetensors). */
int mynn_quantize_safetensors_int8(const char *src, const char *dst, int *quantized, int *passthrough);

/* Device copy of a Llama checkpoint in the order `initializer` wants (tensor names as
 * ModelSpec::from_hf, crates/llm/src/decoder.rs:570-660); float tensors are converted to cfg->dtype,
 * int8 weights and their scales are uploaded as they are.  The result owns the device memory. */
typedef struct mynn_device_weights mynn_device_weights;
mynn_device_weights *mynn_weights_upload(const mynn_weights *w, const mynn_model_config *cfg);
void **mynn_device_weights_initializer(mynn_device_weights *dw);
int mynn_device_weights_int8(const mynn_device_weights *dw);   /* 1: int8 linears (set cfg->weights_int8) */
void mynn_device_weights_free(mynn_device_weights *dw);

#ifdef __cplusplus
}
#endif
#endif /* MYNN_HIP_H_ */
