// kernels.hpp -- host-side launch interface of the gfx950 kernels (kernels.hip).
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

namespace aek {

// GEMM A-operand modes
constexpr int kAI8 = 0;          // int8 rows + per-row scale
constexpr int kAF32Q = 1;        // f32 rows quantized on load: q = round(x * (127/max))
constexpr int kAF32QSmooth = 2;  // f32 rows quantized on load: q = round((x * s_k) * (127/max))
constexpr int kALn = 3;          // f32 rows (K = 384) put through the LayerNorm + SmoothQuant of an LnArgs
constexpr int kAPreLn = 4;       // kALn whose f32 rows come from an N = 384 GEMM of a PreArgs in the same kernel
                                 // first (launch_gemm_ln_prologue, few rows only)
// GEMM epilogues
constexpr int kEpiF32 = 0;   // out = fma(f32(acc), sa*ws, bias (+res))
constexpr int kEpiGelu = 1;  // out = GELU(that) * g_smooth[n]; g_rowmax[m] = max |out|

struct GemmArgs {
  int M, N, K;
  const void* A;              // int8 [M,K] or f32 [M,K]
  const float* a_scale;       // kAI8: [M]
  const uint32_t* a_rowmax;   // kAF32Q*: [M] bits of max_abs (>= 1e-8)
  const float* a_smooth;      // kAF32QSmooth: inv_smooth [K]
  const int8_t* w;            // pre-swizzled by swizzle_weights
  const float* w_scale;       // [N]
  const float* bias;          // [N]
  const float* res;           // [M,N] or null
  float* out;                 // [M,N]
  const float* g_smooth;      // kEpiGelu: next layer inv_smooth [N]
  uint32_t* g_rowmax;         // kEpiGelu: [M], pre-set to bits(1e-8f)
  int col_fast;               // set by launch_gemm: workgroup order (column tile fastest)
  // launch_gemm_ln only: res holds a LayerNorm's input rows, and the residual is that LayerNorm's output, recomputed as ((res - mean) * rstd) * res_gamma +
  // res_beta from its (mean, rstd) per row
  const float2* res_stats = nullptr;
  const float* res_gamma = nullptr;
  const float* res_beta = nullptr;
  int stream_cols = 0;        // output columns [0, stream_cols) are stored nontemporally (read once later)
};
// N % 384 == 0, K % 64 == 0
void launch_gemm(const GemmArgs& p, int amode, int emode, hipStream_t st);
// host: [N,K] row-major int8 -> the GEMM's fragment order [K/64][N/16][64][16] (out has N*K bytes)
void swizzle_weights(int n, int k, const int8_t* w, int8_t* out);

// The FFN block of one layer in one kernel (hidden 384, intermediate 1536):
// out = FFN-down(quant(GELU(FFN-up(A)) * g_smooth)) + b2 + res, with the
// arithmetic of launch_gemm's kAI8/kEpiGelu and kAF32Q/kEpiF32 variants.
struct FfnArgs {
  int M;
  const int8_t* A;         // [M,384]
  const float* a_scale;    // [M]
  const int8_t* w1;        // FFN-up, swizzled [1536,384]
  const float* w1_scale;   // [1536]
  const float* b1;         // [1536]
  const float* g_smooth;   // FFN-down inv_smooth [1536]
  const int8_t* w2;        // FFN-down, swizzled [384,1536]
  const float* w2_scale;   // [384]
  const float* b2;         // [384]
  const float* res;        // [M,384] (may equal out)
  float* out;              // [M,384]
  // the FFN-up GELU through gelu_fast with exact repair (same bits); needs every
  // g_smooth entry finite (else the exact-GELU kernel runs)
  bool fast_gelu = false;
};
// side (optional, with fork and join events): a second stream on which a mixed
// plan's launch of short workgroups runs beside the 64-row one (forked after the
// work queued on st, joined before st continues), so its partial round of
// workgroups fills CUs as the 64-row rounds free them instead of running alone
// at the end
// ln (optional): the LayerNorm + SmoothQuant of the output rows in the same kernel
// where its workgroups are 16 rows high (ln->src is ignored, ln->rowmax_init2 not
// written; ln->q may be p.A, ln->scale p.a_scale and ln->dst p.res: a workgroup has
// read its rows before it writes them).  Returns whether the launch includes it;
// if not, it is the caller's to launch.
struct LnArgs;
bool launch_ffn(const FfnArgs& p, hipStream_t st, hipStream_t side = nullptr, hipEvent_t fork = nullptr,
                hipEvent_t join = nullptr, const LnArgs* ln = nullptr);
// test hooks: the exact-GELU kernel for every launch (process-wide); the fast
// kernel's repair counters on the current device ([0] 16 x 16 tiles recomputed for
// an undecided quantized value, [1] the 16-row groups of passes with more candidates
// for the row maxima than rows), optionally reset
void set_ffn_exact_gelu(bool exact);
bool ffn_exact_gelu();
hipError_t ffn_repair_counts(unsigned long long counts[2], bool reset);
// the exhaustive check of gelu_fast against gelu_exact (6 counters at out_dev, device memory)
hipError_t gelu_fast_certify(unsigned long long* out_dev, hipStream_t st);
// token rows per FFN workgroup, process-wide (a test hook): 0 by the batch (default), 16, 32, 64 or -m
void set_ffn_rows(int rows);
int ffn_rows();  // the current setting
// compute units of the current device (cached per device)
int device_cu_count();

constexpr int kLnSrcF32 = 0;
constexpr int kLnSrcEmb = 1;
struct LnArgs {
  int T;
  // kLnSrcEmb
  const uint16_t* ids;
  const int* cu;
  int B;
  const int8_t* word_q;
  const float* word_s;
  const int8_t* pos_q;
  const float* pos_s;
  const float* type0;
  // kLnSrcF32
  const float* src;
  const float* gamma;
  const float* beta;
  const float* smooth;
  float* dst;       // LayerNorm output (f32 residual stream), may alias src; may be null (stats instead)
  float2* stats;    // optional: (mean, rstd) per row, from which a consumer recomputes the output exactly
  int8_t* q;        // [T,384]
  float* scale;     // [T]
  uint32_t* rowmax_init;   // optional: set to bits(1e-8f) for each row
  uint32_t* rowmax_init2;  // optional second buffer
  // kLnSrcEmb, optional: set to bits(1e-8f) for rows < n_c (the layer-11 [CLS] rows' buffers)
  uint32_t* rowmax_c;
  uint32_t* rowmax_c2;
  int n_c;
  // kLnSrcEmb, optional: the first workgroup writes cu_safe[0..B], the segment
  // bounds the later kernels of the pass read: cu when it is a prefix sum of T
  // with every segment 1..max_len tokens long, else B one-token segments, and
  // then it sets bit 0 of *err (launch_sanitize_segments, strict)
  int max_len;
  int* err;
  int* cu_safe;
};
void launch_ln_quant(const LnArgs& p, int src_mode, hipStream_t st);
// cs[0..B] = cu[0..B] when valid, else cs[b] = b (needs B <= T) and bit 0 of *err
// (err may be null).  Valid, strict: cu[0] = 0, cu[B] = T, segments of 1..max_len
// tokens; loose: 0 <= cu[0], cu[B] <= T, segments of 0..max_len tokens.  Kernels
// given cs index rows inside [0, T) whatever cu held.
void launch_sanitize_segments(const int* cu, int B, int T, int max_len, bool strict, int* err, int* cs,
                              hipStream_t st);
// The attention output GEMM (kAF32QSmooth, N = K = 384, with residual) and the
// LayerNorm + SmoothQuant of its output rows in one kernel (ln.src is ignored, p.out
// is not written).
void launch_gemm_ln(const GemmArgs& p, const LnArgs& ln, hipStream_t st);
// Few rows (gemm_small_path): a GEMM whose A operand is the LayerNorm + SmoothQuant
// of the f32 rows p.A (K = 384) under `ln` (gamma, beta, smooth), applied in each
// workgroup's prologue; the workgroups of the first column tile also store the
// LayerNorm's outputs (ln.dst, and ln.q / ln.scale / ln.rowmax_init* when set).
// ln.dst must not alias p.A.
void launch_gemm_ln_prologue(const GemmArgs& p, const LnArgs& ln, hipStream_t st);
// The GEMM in front of such a LayerNorm (kAPreLn): x = fma(f32(q(A) . W^T), sa * ws,
// bias + res) with A [M,384] f32 quantized on load as kAF32QSmooth does (sa =
// max_abs / 127 from a_rowmax), W [384,384] pre-swizzled.
struct PreArgs {
  const float* A;
  const uint32_t* a_rowmax;
  const float* a_smooth;
  const int8_t* w;
  const float* w_scale;
  const float* bias;
  const float* res;
};
// Few rows: launch_gemm_ln_prologue with the LayerNorm's input rows computed in
// every workgroup by `pre` (the attention-output GEMM in front of LN1, then the
// FFN-up GEMM): one kernel instead of two.  ln.dst must not alias pre.res or pre.A.
void launch_gemm_pre_ln(const GemmArgs& p, const PreArgs& pre, const LnArgs& ln, hipStream_t st);
// whether launch_gemm takes the few-rows kernels for m rows (and the prologue form applies)
constexpr int kSmallM = 1024;
inline bool gemm_small_path(int m) { return m > 0 && m <= kSmallM; }
// whether an int8-A GEMM (kEpiF32, m rows beyond the few-rows path, K = k) keeps the
// 16-row workgroups on a GPU of cus compute units
bool gemm_int8_rows16(int m, int n, int k, bool res, int cus);

void launch_row_quant(int m, int n, float* x, const float* smooth, int8_t* q, float* scale, bool gelu,
                      hipStream_t st);

struct AttnArgs {
  const float* qkv;        // [T,1152]
  const int* cu;           // [B+1]
  int B;
  int* plan;               // scratch: attention_plan_ints(B, T) ints, 16-byte aligned
  float* ctx;              // [T,384]
  const float* smooth;     // attn_out inv_smooth [384] or null
  uint32_t* rowmax;        // [T] or null
  int s_pitch;             // score row pitch: attention_pitch(bound of the sequence lengths)
  int skip_from = 0;       // attention_rows_kernel: segments of at least this many tokens are left out (0: none)
  int len1 = 0;            // B == 1 and cu_seqlens = {0, len1} known on the host: the latency form needs no load
  int longest = 0;         // the longest segment, where the host knows it (it chooses the kernels; 0: not known)
};
int attention_pitch(int max_len);
size_t attention_lds_bytes(int s_pitch);
// tiles of 32 queries: max_tiles >= sum_b ceil(L_b / 32); T/32 + B + 1 is one
inline int attention_max_tiles(int B, int T) { return T / 32 + B + 1; }
// a plan list: kPlanHdr header records (each XCD's item count and first item),
// then one 4-int record per (tile, head)
constexpr int kPlanHdr = 4;
// an item record carries its segment's index in the high 24 bits of its last int
constexpr int kPlanMaxSegs = 1 << 24;
inline size_t attention_plan_list_records(int B, int T) { return kPlanHdr + 12 * (size_t)attention_max_tiles(B, T); }
// ints of `plan` scratch for B segments and T tokens: two lists
inline size_t attention_plan_ints(int B, int T) { return 8 * attention_plan_list_records(B, T); }
// items of one list on one XCD: at most the average (12 max_tiles / 8) plus one
// (segment, head) group of up to 16 tiles; a launch runs 8 times this many workgroups
constexpr int attention_plan_cap(int max_tiles) { return (12 * max_tiles + 7) / 8 + 16; }
void init_attention_kernels();  // once per device before the first launch (not during capture)
// ae_attention_varlen_noalloc: the tile plan and the checked copy of cu_seqlens in
// a static device array of this many 16-byte records (8 MiB), so
// 2 attention_plan_list_records(B, T) + ceil((B + 1) / 4) <= kNoAllocPlanRecords
constexpr int kNoAllocPlanRecords = 524288;
// the current device's address of that array (resolved on the first call per
// device, with the device current; not during a stream capture)
hipError_t noalloc_plan_scratch(int** plan);
// T = total tokens of the batch; plan = false reuses the plan already in p.plan
// (launch_attention_plan, which depends only on cu, B and s_pitch)
void launch_attention(const AttnArgs& p, int T, hipStream_t st, bool plan = true);
// the exact attention's kernels for B segments, T tokens and rows of at most max_len
// keys, the longest of them of `longest` (0: not known), on a GPU of cus compute units:
// 32-query tiles (register rows up to 64 keys), 16-query tiles, or
// attention_lat_kernel.  Every choice gives the same bits.
enum AttnChoice { kAttnTiles32 = 0, kAttnTiles16 = 1, kAttnLat = 2 };
int attention_choice(int B, int T, int max_len, int longest, int cus);
// split = 1: rows of more than 400 keys in the plan's second list
void launch_attention_plan(const AttnArgs& p, hipStream_t st, int split, int max_tiles);
// exact-attention kernel choice for later launches: 0 by the batch, 1 tiled (32 queries) /
// register rows only, 2 the latency form only (a test hook; same bits)
void set_attention_form(int form);
int attention_form();  // the current setting
// Quantized attention (the reference's ArmSme backend): scratch for the int8 Q
// and K of every token and head, their scales and the per-column |V| maximum.
struct SmeArgs {
  int8_t* q8;       // [T,384]
  int8_t* k8;       // [T,384]
  float* qs;        // [T,12]
  float* ks;        // [T,12]
  uint32_t* vmax;   // [384], f32 bits
  int8_t* vt;       // [384][sme_vt_len(T, B)]: int8 V per head column, keys contiguous; segment b
                    // starts at round8(cu[b] + 7b), so every 8-key group is 8-byte aligned
  int* tseg;        // [T]: each token's segment index (sme_pack_kernel, for sme_vquant_kernel)
  // 0: V column scales over the whole packed batch (vmax [384]), every segment
  // quantized; 1: per sequence as forward_cls runs it (vmax [B][384]), segments
  // of fewer than 16 tokens left to the exact attention (launch_attention_short)
  int per_seq = 0;
};
inline size_t sme_vt_len(int T, int B) { return ((size_t)T + 7 * (size_t)B + 64 + 7) & ~(size_t)7; }
// the packing, the plan (plan = true) and the attention; p.smooth / p.rowmax as launch_attention
void launch_attention_sme(const AttnArgs& p, const SmeArgs& s, int T, hipStream_t st, bool plan = true);
void init_attention_sme_kernels();  // once per device before the first launch
// the exact attention of the segments shorter than 16 tokens only (the rest untouched)
void launch_attention_short(const AttnArgs& p, hipStream_t st);
// test hook: raw results of the exact-product MFMA (16 floats per lane per set of 64 pairs)
void launch_mfma_products(const float* a, const float* b, float* out, int n_sets, hipStream_t st);

struct ClsArgs {
  int B;
  const int* cu;
  const float* hidden;     // [T,384]
  const int8_t* act_q;     // [T,384] (the layer input, quantized)
  const float* act_scale;  // [T]
  float* hidden_c;         // [B,384]: the [CLS] rows of hidden, gathered
  const int8_t* wq;        // q_only linear: swizzled [384,384] int8, w_scale, bias
  const float* wq_scale;
  const float* wq_bias;
  const float* kv;         // [T,768]
  float* ctx_c;            // [B,384]
  const float* smooth;     // attn_out inv_smooth
  uint32_t* rowmax_ctx_c;  // [B], pre-set to bits(1e-8f)
  int max_len = 512;       // keys attended per sequence (<= 512): sizes the V tile in LDS
  // optional: hidden holds a LayerNorm's input rows and hidden_c gets that
  // LayerNorm's output, ((x - mean) * rstd) * ln_gamma + ln_beta per row
  const float2* hidden_stats = nullptr;
  const float* ln_gamma = nullptr;
  const float* ln_beta = nullptr;
};
// the layer-11 [CLS] attention: per (sequence, head) the [CLS] row's q (the q_only
// GEMM for that row and head), its attention over the segment's K/V rows, ctx_c
// and its row absmax; the head-0 workgroups also gather hidden_c
void launch_cls(const ClsArgs& p, hipStream_t st);
void launch_final_ln_l2(int B, const float* src, const float* gamma, const float* beta, float* out, hipStream_t st);
void launch_fill_u32(uint32_t* dst, int n, uint32_t v, hipStream_t st);
void launch_gelu_map(const float* x, float* y, size_t n, hipStream_t st);

}  // namespace aek
