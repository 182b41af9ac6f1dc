/*
 * arctic_embed.h -- C ABI of the MI355X-native W8A8 arctic-embed-s engine.
 *
 * Drop-in for the public API of mdlockyer/snowflake-arctic-embed-s-rust
 * (crate `arctic-embed-s-int8`).  Every entry point names the reference item it
 * replaces (path:line in the reference tree).  Plain C types only: pointers,
 * sizes, status codes.  Streams are passed as `void*` (a hipStream_t; NULL is
 * the workspace's own stream for workspace calls, the null stream otherwise).
 *
 * Threading: an engine is immutable after open and may be shared by any number
 * of threads (the reference's `ArcticEmbedS` is shared `&self`).  A workspace
 * is single-threaded, one per caller thread (the reference's `&mut Workspace`).
 */
#ifndef ARCTIC_EMBED_H
#define ARCTIC_EMBED_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* ---- model dimensions: src/quantize.rs:9-18 ----------------------------- */
#define AE_HIDDEN_SIZE 384
#define AE_INTERMEDIATE_SIZE 1536
#define AE_NUM_HEADS 12
#define AE_HEAD_DIM 32
#define AE_NUM_LAYERS 12
#define AE_VOCAB_SIZE 30522
#define AE_MAX_POSITIONS 512

/* ---- status codes -------------------------------------------------------
 * The reference returns io::Result / panics; here every failure is a code.
 *   AE_ERR_NOT_FOUND      io::ErrorKind::NotFound (fs::read, src/quantize.rs:77)
 *   AE_ERR_INVALID_DATA   bad `.ae8` magic (src/quantize.rs:81-86) or malformed pack
 *   AE_ERR_EOF            truncated pack (read_exact -> UnexpectedEof)
 *   AE_ERR_INVALID_ARG    empty ids (the panic at src/model.rs:192), bad sizes, id >= vocab
 *   AE_ERR_UNSUPPORTED    no usable gfx950 device (src/lib.rs:53-61 analogue)
 *   AE_ERR_CAPACITY       request exceeds the workspace capacity
 *   AE_ERR_HIP            a HIP runtime call failed (message in ae_last_error)
 */
#define AE_OK 0
#define AE_ERR_NOT_FOUND (-1)
#define AE_ERR_INVALID_DATA (-2)
#define AE_ERR_EOF (-3)
#define AE_ERR_INVALID_ARG (-4)
#define AE_ERR_UNSUPPORTED (-5)
#define AE_ERR_CAPACITY (-6)
#define AE_ERR_HIP (-7)

typedef struct ae_engine ae_engine;       /* ArcticEmbedS, src/lib.rs:34-38 */
typedef struct ae_workspace ae_workspace; /* Workspace, src/model.rs:123-173 */
typedef struct ae_linear ae_linear;       /* PackedLinearInt8, src/gemm.rs:165-181 */
typedef struct ae_tokenizer ae_tokenizer; /* BertTokenizer, src/tokenizer.rs:26-31 */
typedef struct ae_parallel_context ae_parallel_context; /* ParallelContext, src/parallel.rs:137-142 */

/* Human-readable text of the last error raised on the calling thread. */
const char* ae_last_error(void);
/* Library version string. */
const char* ae_version(void);

/* ---- engine ------------------------------------------------------------- */
/* ArcticEmbedS::from_dir(dir) (src/lib.rs:46-48): reads dir/vocab.txt and
 * dir/model.ae8 (MODEL_FILE / VOCAB_FILE, src/lib.rs:18-20), uploads the weights
 * to the current HIP device once.  A NULL dir means default_model_dir()
 * ($ARCTIC_EMBED_MODEL_DIR or ./model, src/lib.rs:22-31). */
int ae_engine_open(const char* dir, ae_engine** out);
/* Same as ae_engine_open with explicit file paths; vocab_path may be NULL for an
 * ids-only engine (ae_embed_query/_document/_batch then return AE_ERR_INVALID_ARG). */
int ae_engine_open_files(const char* ae8_path, const char* vocab_path, ae_engine** out);
void ae_engine_close(ae_engine* e);
/* ArcticEmbedS::raw_size_bytes = PackedModel::size_bytes (src/lib.rs:65, src/model.rs:87-119),
 * counted for the device image (weights + scales + biases + smoothing vectors). */
size_t ae_engine_size_bytes(const ae_engine* e);
/* QuantizedModelRaw::size_bytes (src/quantize.rs:140-165) of the pack as read. */
size_t ae_engine_raw_size_bytes(const ae_engine* e);
/* default_model_dir() (src/lib.rs:26-31) into buf; returns the needed length. */
size_t ae_default_model_dir(char* buf, size_t cap);

/* ---- workspace ---------------------------------------------------------- */
/* Workspace::new() (src/model.rs:147-172).  Owns a HIP stream, device activations
 * sized for max_tokens packed tokens and max_seqs sequences per call, and pinned
 * host staging.  0 selects the defaults (512 tokens, 64 sequences, as the
 * reference's Workspace).  The embedding calls below grow it on demand (once,
 * up to 2^18 tokens and 8192 sequences per device batch; a larger request runs
 * as several batches); ae_forward_packed_device and the operators return
 * AE_ERR_CAPACITY past it.  512 <= max_tokens <= 2^26, max_seqs <= max_tokens
 * and max_seqs < 2^24, else AE_ERR_INVALID_ARG. */
int ae_workspace_create(const ae_engine* e, size_t max_tokens, size_t max_seqs, ae_workspace** out);
void ae_workspace_destroy(ae_workspace* ws);
/* the workspace's hipStream_t */
void* ae_workspace_stream(ae_workspace* ws);

/* ---- embedding API ------------------------------------------------------ */
/* Every call here takes a workspace or NULL: NULL selects the engine's own
 * (created on first use, grown on demand and kept; calls that share it take
 * turns), as the reference's embed_batch(&self, ...) owns its scratch.  The
 * calls are synchronous: they return with the embeddings in host memory. */
/* ArcticEmbedS::embed_tokens (src/lib.rs:98-102) -> PackedModel::forward_cls
 * (src/model.rs:185-513): ids truncated to 512, out = L2-normalized [CLS] f32[384].
 * n == 0 returns AE_ERR_INVALID_ARG (the reference panics, src/model.rs:192). */
int ae_embed_tokens(const ae_engine* e, ae_workspace* ws, const uint16_t* ids, size_t n, float* out384);
/* ArcticEmbedS::embed_query / embed_document (src/lib.rs:76-94). */
int ae_embed_query(const ae_engine* e, ae_workspace* ws, const char* utf8, float* out384);
int ae_embed_document(const ae_engine* e, ae_workspace* ws, const char* utf8, float* out384);
/* ArcticEmbedS::embed_batch (src/lib.rs:138-260): out is n*384 floats in input
 * order; n == 0 is a no-op.  Sequences are length-sorted and packed into as few
 * device batches as the (grown) workspace holds, all queued on its stream with
 * their copies and one synchronization at the end; batches of at most 16384
 * tokens are padded with dummy sequences to a bucketed shape (max length to a
 * power of two, tokens to a quarter binade, sequences to a multiple of 8) and
 * replay that shape's captured graph.  num_threads drives host tokenization only; all
 * sequences run as token-packed device batches. */
int ae_embed_batch(const ae_engine* e, ae_workspace* ws, const char* const* texts, size_t n,
                   int is_query, int num_threads, float* out);
/* embed_batch over pre-tokenized ids: sequence i is ids[offsets[i] .. offsets[i+1]). */
int ae_embed_batch_tokens(const ae_engine* e, ae_workspace* ws, const uint16_t* ids,
                          const uint32_t* offsets, size_t n, float* out);
/* PackedModel::forward_ragged_cls (src/model.rs:521-914) with device-resident
 * inputs: ids_dev[total_tokens] u16, cu_seqlens_dev[n_seqs+1] i32 (each sequence
 * 1..max_seq_len tokens; max_seq_len <= 512, 0 means 512), out_dev[n_seqs*384]
 * f32.  A max_seq_len below 512 is taken for the batch's longest length where the
 * attention kernels are chosen (the same bits by any).  Asynchronous on `stream`; no host copies.  Used when the caller keeps
 * token ids in HBM.  The device checks cu_seqlens (cu[0] = 0, cu[n_seqs] =
 * total_tokens, every segment 1..max_seq_len tokens); a batch that fails is
 * reported as AE_ERR_INVALID_ARG by the next ae_workspace_synchronize.  Its
 * outputs are then unspecified, but no kernel reads or writes outside the
 * batch's rows: the first kernel writes a checked copy of cu_seqlens (n_seqs
 * one-token segments when it fails) and every later kernel reads that copy. */
int ae_forward_packed_device(const ae_engine* e, ae_workspace* ws, const uint16_t* ids_dev,
                             const int32_t* cu_seqlens_dev, int n_seqs, int total_tokens,
                             int max_seq_len, float* out_dev, void* stream);
/* Waits for the workspace's work on `stream` (NULL: its own stream) and reports
 * the device-side batch checks of the asynchronous calls since the last one:
 * AE_OK, or AE_ERR_INVALID_ARG (and the check is reset).  No counterpart in the
 * reference, whose calls are all synchronous and panic on bad input. */
int ae_workspace_synchronize(ae_workspace* ws, void* stream);

/* ---- latency mode: one sequence at a time ------------------------------- */
/* ParallelContext::new(n_threads) (src/parallel.rs:144-160): n_threads is clamped
 * to 1..8 as there and only recorded; the device parallelizes the sequence.  The
 * context holds a single-sequence workspace for `e` (512 tokens, own stream,
 * graph replay per length); use it from one thread at a time. */
int ae_parallel_context_create(const ae_engine* e, int n_threads, ae_parallel_context** out);
void ae_parallel_context_destroy(ae_parallel_context* c);
/* the clamped thread count */
int ae_parallel_context_threads(const ae_parallel_context* c);
/* ArcticEmbedS::embed_tokens_parallel / embed_query_parallel /
 * embed_document_parallel (src/lib.rs:104-133): same results as ae_embed_tokens /
 * ae_embed_query / ae_embed_document, bit for bit. */
int ae_embed_tokens_parallel(const ae_engine* e, ae_parallel_context* c, const uint16_t* ids, size_t n,
                             float* out384);
int ae_embed_query_parallel(const ae_engine* e, ae_parallel_context* c, const char* utf8, float* out384);
int ae_embed_document_parallel(const ae_engine* e, ae_parallel_context* c, const char* utf8, float* out384);

/* ---- tokenizer (host only) ---------------------------------------------- */
/* BertTokenizer::from_vocab_file (src/tokenizer.rs:34-37). */
int ae_tokenizer_open(const char* vocab_path, ae_tokenizer** out);
void ae_tokenizer_close(ae_tokenizer* t);
/* BertTokenizer::encode / encode_query (src/tokenizer.rs:75-89): writes up to cap
 * ids ([CLS] (+ query prefix) ... [SEP], at most 512) and the count to *n_out. */
int ae_tokenizer_encode(const ae_tokenizer* t, const char* utf8, int is_query, uint16_t* ids, size_t cap,
                        size_t* n_out);
/* BertTokenizer::vocab_size (src/tokenizer.rs:69-71). */
size_t ae_tokenizer_vocab_size(const ae_tokenizer* t);

/* cosine_similarity (src/lib.rs:265-271): dot product of two f32[384]. */
float ae_cosine_similarity(const float* a, const float* b);

/* ---- operator level (device pointers, asynchronous on `stream`) ---------- */
/* PackedLinearInt8::from_raw_row_major (src/gemm.rs:186-246): w_q [n_out,k_in]
 * row-major int8, w_scale/bias [n_out], inv_smooth [k_in] (host pointers).
 * Requires n_out % 384 == 0 and k_in % 64 == 0. */
int ae_linear_create(int n_out, int k_in, const int8_t* w_q, const float* w_scale,
                     const float* bias, const float* inv_smooth, ae_linear** out);
void ae_linear_destroy(ae_linear* l);
/* gemm_int8_fused (src/gemm.rs:630-671):
 * out[m,n] = fma(f32(sum_k a[m,k]*w[n,k]), a_scale[m]*w_scale[n], bias[n] + res[m,n]).
 * a_dev [m,k_in] int8 row-major, a_scale_dev [m], res_dev [m,n_out] or NULL. */
int ae_gemm_w8a8(const ae_linear* l, int m, const int8_t* a_dev, const float* a_scale_dev,
                 const float* res_dev, float* out_dev, void* stream);
/* layernorm_smooth_quantize_row (src/simd_math.rs:181-247) over m rows of width 384:
 * x_dev updated in place, q_dev [m,384] int8, scale_dev [m]. */
int ae_layernorm_smooth_quantize(int m, float* x_dev, const float* gamma_dev, const float* beta_dev,
                                 const float* inv_smooth_dev, int8_t* q_dev, float* scale_dev,
                                 void* stream);
/* smooth_quantize_row (src/simd_math.rs:501-531) over m rows of width n (n % 64 == 0). */
int ae_smooth_quantize(int m, int n, const float* x_dev, const float* inv_smooth_dev, int8_t* q_dev,
                       float* scale_dev, void* stream);
/* gelu_smooth_quantize_batch (src/simd_math.rs:655-674, 1283-1313) over m rows of
 * width n (n % 64 == 0): x_dev <- GELU(x)*inv_smooth in place, q_dev, scale_dev. */
int ae_gelu_smooth_quantize(int m, int n, float* x_dev, const float* inv_smooth_dev, int8_t* q_dev,
                            float* scale_dev, void* stream);
/* Segment-bounded multi-head attention of one layer (src/model.rs:663-694):
 * qkv_dev [T,1152] f32 (Q|K|V, head h at column h*32), cu_seqlens_dev [n_seqs+1],
 * ctx_dev [T,384] f32.  Synchronous: reads cu_seqlens back to size the work
 * (0 <= cu[0], non-decreasing, cu[n_seqs] <= total_tokens, else
 * AE_ERR_INVALID_ARG); segments longer than 512 are cut to their first 512
 * rows.  Its scratch is one device buffer per GPU, kept and reused by later
 * calls (allocated only when a call needs more than any before it); concurrent
 * calls on one GPU take turns.  For a per-layer loop prefer
 * ae_workspace_attention_varlen, which neither copies to the host nor waits. */
int ae_attention_varlen(const float* qkv_dev, const int32_t* cu_seqlens_dev, int n_seqs,
                        int total_tokens, float* ctx_dev, void* stream);
/* The same attention as the reference's ArmSme backend computes it over a
 * packed batch (attention_multihead_sme with segment ranges, src/model.rs:607-621,
 * src/simd_math.rs:1933-2192): int8 Q and K per token and head, int8 V per head
 * column over all total_tokens rows, integer scores, the exact-range int16
 * softmax (round(16383 * 2^(s - max)), exp2 in log2 units) and integer P @ V.
 * Bit-identical to that path; within a cosine budget of ae_attention_varlen.
 * Same arguments and synchronization as ae_attention_varlen, except that the V
 * scales span every row: cu_seqlens must be an exact prefix sum (cu[0] = 0,
 * cu[n_seqs] = total_tokens) of segments of at most 512 tokens, and
 * n_seqs < 2^24, else AE_ERR_INVALID_ARG. */
int ae_attention_varlen_quantized(const float* qkv_dev, const int32_t* cu_seqlens_dev, int n_seqs,
                                  int total_tokens, float* ctx_dev, void* stream);
/* No counterpart in the reference: ae_attention_varlen for callers that cannot
 * allocate device memory (code under HIP graph capture, tight serving loops,
 * harnesses that forbid hipMalloc).  It allocates nothing, copies nothing to the
 * host and does not synchronize: the caller states max_seq_len (1..512; below 512
 * taken for the longest segment where the kernels are chosen), and
 * cu_seqlens must lie in [0, total_tokens] with segments of 0..max_seq_len
 * tokens.  A cu_seqlens that breaks this gives unspecified values (the call
 * cannot report it) but no access outside the batch's rows: a checked copy of
 * cu_seqlens (n_seqs one-token segments when it fails) is what the kernels read.
 * The only scratch, the tile plan and that copy, is a static device array of
 * 524288 16-byte records (8 MiB, held by each GPU the library runs on until the
 * process ends): 2 (4 + 12 (total_tokens / 32 + n_seqs + 1)) + (n_seqs + 4) / 4
 * records at most, else AE_ERR_CAPACITY (checked before any pointer is used).
 * All calls on one GPU share that array, so calls that overlap on one GPU race.
 * The first call on a device (current) resolves the array's address there and
 * must not be inside a stream capture. */
int ae_attention_varlen_noalloc(const float* qkv_dev, const int32_t* cu_seqlens_dev, int n_seqs,
                                int total_tokens, int max_seq_len, float* ctx_dev, void* stream);
/* ae_attention_varlen / ae_attention_varlen_quantized on a workspace's scratch,
 * for callers that run the operator per layer (the reference's per-layer
 * attention call, src/model.rs:607-694): asynchronous on `stream` (NULL: the
 * workspace's), no host copy, no synchronization, no allocation (the quantized
 * variant allocates its scratch on its first call, as
 * ae_workspace_set_attention_mode does).  The caller states max_seq_len
 * (1..512), the longest segment (512 also where it is not known: kernels that need
 * it are then not chosen); n_seqs and total_tokens within the workspace
 * capacity (AE_ERR_CAPACITY otherwise).  A cu_seqlens that is not an exact
 * prefix sum of segments of 1..max_seq_len tokens is reported by the next
 * ae_workspace_synchronize (its values are then unspecified; every access stays
 * inside the batch's rows).  These calls use the workspace's plan and checked
 * cu_seqlens scratch, which its forward passes use too: work on one workspace
 * must not overlap (a call on another stream must be ordered after the
 * workspace's earlier work, and the workspace's later work after it). */
int ae_workspace_attention_varlen(ae_workspace* ws, const float* qkv_dev, const int32_t* cu_seqlens_dev,
                                  int n_seqs, int total_tokens, int max_seq_len, float* ctx_dev, void* stream);
int ae_workspace_attention_varlen_quantized(ae_workspace* ws, const float* qkv_dev, const int32_t* cu_seqlens_dev,
                                            int n_seqs, int total_tokens, int max_seq_len, float* ctx_dev,
                                            void* stream);

/* ---- tools and test hooks (no counterpart in the reference) -------------- */
/* Writes a seeded synthetic model in `.ae8` layout (fp32
 * N(0,0.02) embeddings stored per-row int8, int8 weights U{-127..127}, scales
 * 0.05/127*U(0.5,1.5), SmoothQuant 1/U(0.5,2), biases N(0,0.02), LN gamma
 * 1+N(0,0.05), beta N(0,0.02); layer 11 carries the Q / KV split).  Host only. */
int ae_write_synthetic_ae8(const char* path, uint64_t seed);
/* Per-kernel device timing of the workspace's forward passes (hipEvents around
 * every launch).  Kinds: see AE_KERNEL_* below.  ms_out/counts have AE_KERNEL_KINDS
 * entries; times cover the passes since timing was enabled and require the
 * passes to have completed (synchronize first). */
#define AE_KERNEL_EMBED_LN 0
#define AE_KERNEL_GEMM_QKV 1
#define AE_KERNEL_ATTENTION 2
#define AE_KERNEL_GEMM_ATTN_OUT 3
#define AE_KERNEL_LN1 4 /* unused (count 0): LN1 runs in the kernel of GEMM_ATTN_OUT or GEMM_FFN_UP */
#define AE_KERNEL_GEMM_FFN_UP 5 /* the whole fused FFN block when a pass has more than 1024 tokens (with LN2 while its
                                  16-row workgroups run in one round, 4096 tokens) */
#define AE_KERNEL_GEMM_FFN_DOWN 6 /* unused (count 0) when the FFN block is fused */
#define AE_KERNEL_LN2 7
#define AE_KERNEL_LAYER11_TAIL 8
#define AE_KERNEL_KINDS 9
int ae_workspace_set_timing(ae_workspace* ws, int enabled);
/* Graph replay of repeated forward passes (on by default): the second call with
 * the same buffers, stream and batch shape captures the pass into a hipGraph and
 * later calls replay it.  Disabled while timing is on.  0 forces eager launches. */
int ae_workspace_set_graphs(ae_workspace* ws, int enabled);
/* Attention of layers 0-10 in this workspace's forward passes.
 * AE_ATTENTION_EXACT (default): the reference's scalar order, bit-exact.
 * AE_ATTENTION_QUANTIZED: each sequence as the reference's forward_cls runs it
 * on its ArmSme backend (src/model.rs:223-259): from 16 tokens on the quantized
 * attention (int8 Q, K, V and int16 P, see ae_attention_varlen_quantized) with
 * V scales over that sequence alone, below 16 tokens the exact path.  A
 * sequence's result is therefore the same alone or in any batch.  Setting it
 * the first time allocates the mode's scratch for the workspace capacity. */
#define AE_ATTENTION_EXACT 0
#define AE_ATTENTION_QUANTIZED 1
int ae_workspace_set_attention_mode(ae_workspace* ws, int mode);
int ae_workspace_kernel_times(ae_workspace* ws, double* ms_out, int* counts);
/* The fused GEMM variants of the forward pass, exposed for parity tests:
 * A given as f32 rows quantized on load with q = round((x*s_k)*(127/rowmax[m]))
 * (s = smooth_dev, or 1 when NULL) and scale rowmax[m]/127 (rowmax as f32 bits). */
int ae_debug_gemm_quant_a(const ae_linear* l, int m, const float* x_dev, const uint32_t* rowmax_dev,
                          const float* smooth_dev, const float* res_dev, float* out_dev, void* stream);
/* The attention output projection and LN1 as the forward pass runs them (one
 * kernel; src/model.rs:695-724): out = the smoothed quantize-on-load GEMM of
 * ae_debug_gemm_quant_a with residual res_dev (N = K = 384), then dst = the
 * LayerNorm of out (gamma, beta, eps 1e-12) and q / scale its SmoothQuant int8
 * rows with ln_smooth_dev.  out itself is not stored; dst may equal res_dev. */
int ae_debug_gemm_ln(const ae_linear* l, int m, const float* x_dev, const uint32_t* rowmax_dev,
                     const float* smooth_dev, const float* res_dev, const float* gamma_dev, const float* beta_dev,
                     const float* ln_smooth_dev, float* dst_dev, int8_t* q_dev, float* scale_dev, void* stream);
/* int8 A; epilogue g = GELU(out) * g_smooth[n] stored as f32, and
 * rowmax[m] = max(rowmax[m], max_n |g|) on f32 bits (caller pre-sets rowmax). */
int ae_debug_gemm_gelu(const ae_linear* l, int m, const int8_t* a_dev, const float* a_scale_dev,
                       const float* g_smooth_dev, float* out_dev, uint32_t* rowmax_dev, void* stream);
/* The FFN block of src/model.rs:725-755 as the forward pass runs it beyond 1,024
 * tokens (one kernel, no [m,1536] intermediate in memory):
 * out = gemm_int8_fused(ffn_out, gelu_smooth_quantize(gemm_int8_fused(ffn_inter, a)), res).
 * up: 384 -> 1536 linear, down: 1536 -> 384 linear (its inv_smooth smooths the
 * GELU output).  out may equal res. */
int ae_debug_ffn(const ae_linear* up, const ae_linear* down, int m, const int8_t* a_dev, const float* a_scale_dev,
                 const float* res_dev, float* out_dev, void* stream);
/* ae_debug_ffn with the LayerNorm + SmoothQuant of its output rows in the same
 * kernel (src/model.rs:756-767), as a pass of 1,025 to 4,096 tokens runs it:
 * dst = LayerNorm(out), q / scale its int8 rows.  AE_ERR_INVALID_ARG if m rows are
 * more than one round of 16-row workgroups (4,096 on 256 compute units). */
int ae_debug_ffn_ln(const ae_linear* up, const ae_linear* down, int m, const int8_t* a_dev, const float* a_scale_dev,
                    const float* res_dev, float* out_dev, const float* gamma_dev, const float* beta_dev,
                    const float* ln_smooth_dev, float* dst_dev, int8_t* q_dev, float* scale_dev, void* stream);
/* Embedding + the first `layers` (0..11) encoder layers over one packed batch of n
 * sequences (given order, each 1..512 ids); copies back hidden [T,384] f32,
 * act_q [T,384] int8 and act_scale [T] (T = offsets[n]), the state that
 * src/model.rs:593-768 leaves after those layers. */
int ae_debug_forward_prefix(const ae_engine* e, ae_workspace* ws, const uint16_t* ids, const uint32_t* offsets,
                            size_t n, int layers, float* hidden, int8_t* act_q, float* act_scale);
/* Device GELU (the reference's scalar_gelu, src/simd_math.rs:15-23) over n floats. */
int ae_debug_gelu_map(const float* x_dev, float* y_dev, size_t n, void* stream);
/* The attention kernels' multiplier: v_mfma_f32_16x16x1_4b_f32 with a zero
 * accumulator over n_sets sets of 64 operand pairs (a_dev, b_dev: n_sets*64
 * floats).  out_dev[(set*64 + lane)*16 + r] = a[set*64 + blk*16 + m] *
 * b[set*64 + blk*16 + n] with blk = r/4, m = 4*(lane/16) + r%4, n = lane%16. */
int ae_debug_mfma_products(const float* a_dev, const float* b_dev, float* out_dev, int n_sets, void* stream);
/* Which exact-attention kernels the library launches, process-wide (a test
 * hook, no reference counterpart): 0 by the batch's shape (the default), 1 the
 * tiled and register-row kernels only, 2 the latency form only.  Every form
 * gives the same bits.  AE_ERR_INVALID_ARG for another value. */
int ae_debug_set_attention_form(int form);
/* The kernels of the exact attention for a batch of n_seqs segments, total_tokens
 * tokens and rows of at most max_seq_len, the longest of them of `longest` tokens
 * (0: not known), on a GPU of `cus` compute units (a test hook, no reference
 * counterpart, no device access): 0 tiles of 32 queries (rows
 * in registers up to 64 keys), 1 tiles of 16 queries, 2 the kernel of batches so
 * small that each of its workgroups has a compute unit to itself. */
int ae_debug_attention_choice(int n_seqs, int total_tokens, int max_seq_len, int longest, int cus);
/* Whether ae_gemm_w8a8 of m > 1024 rows, with or without a residual, takes the
 * 16-row workgroups on a GPU of `cus` compute units (a test hook, no reference
 * counterpart, no device access): 1 or 0.  Either form gives the same bits. */
int ae_debug_gemm_int8_rows16(int m, int n, int k, int residual, int cus);
/* Token rows per workgroup of the fused FFN kernel, process-wide (a test hook,
 * no reference counterpart): 0 by the batch's size (the default), 16, 32 or 64,
 * or -m (m a multiple of 64): the first m rows in 64-row workgroups and the rest
 * in a second launch of 32-row ones.  Every plan gives the same bits.
 * AE_ERR_INVALID_ARG for another value. */
int ae_debug_set_ffn_rows(int rows);
/* The fused FFN kernel's GELU, process-wide (a test hook, no reference
 * counterpart): 0 (the default) evaluates it with a fast approximation whose
 * distance from the reference's f32 GELU is certified on all 2^32 inputs and
 * evaluates exactly the values that decide a row maximum and every value whose
 * int8 quantization that distance leaves undecided; nonzero evaluates the reference's GELU on every
 * element.  Both give the same bits. */
int ae_debug_set_ffn_exact_gelu(int exact);
/* Counters of the fast FFN kernel's exact recomputations on the current device
 * (a test hook): *tiles = tiles of 16 rows x 16 columns recomputed for an undecided
 * quantized value, *rows = the 16-row groups (one or two) of each pass that
 * evaluated more candidates for its row maxima than it has rows; reset != 0 clears them after reading. */
int ae_debug_ffn_repairs(uint64_t* tiles, uint64_t* rows, int reset);
/* The certification of the fused FFN kernel's fast GELU (a test hook,
 * synchronous, a few seconds): evaluates it and the reference's GELU on all
 * 2^32 f32 inputs on the current device, both as the kernel does (the fast one
 * on 4 and on 8 values at once), and writes 6 counters: [0] inputs outside the
 * certified bound or whose two fast values differ, [1] NaN results for a non-NaN, finite input,
 * [2] / [3] inputs in the saturated ranges where the reference's GELU is not
 * exactly v / 0, [4] inputs outside the bound with half its absolute term (must
 * be nonzero: the check can fail), [5] inputs checked (2^32). */
int ae_debug_gelu_fast_certify(uint64_t* out6);

#ifdef __cplusplus
}
#endif
#endif
