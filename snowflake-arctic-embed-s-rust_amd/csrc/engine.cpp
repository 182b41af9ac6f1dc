// engine.cpp -- host runtime of the MI355X W8A8 arctic-embed-s engine and the
// C ABI declared in include/arctic_embed.h.
//
// Mirrors the reference's API layer (src/lib.rs) and model driver
// (src/model.rs): one engine holds the device-resident weights, one workspace
// per caller thread holds a HIP stream and device activations; a forward pass is
// one token-packed device batch of any number of sequences.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <numeric>
#include <string>
#include <vector>

#include "../../include/arctic_embed.h"
#include "ae8.hpp"
#include "kernels.hpp"
#include "tokenizer.hpp"

namespace {

thread_local std::string g_last_error;

// Graph captures and the calls that could disturb another thread's capture
// (allocation and freeing, stream and event creation, synchronous copies, device
// synchronization) take turns process-wide: a workspace captures its forward
// pass on its own stream, and another thread growing, creating or destroying a
// workspace meanwhile would otherwise invalidate that capture.  Recursive: the
// guarded helpers call each other.  Lock order: an engine's own-workspace mutex
// or the operator scratch mutex first, then this one.
std::recursive_mutex g_dev_mu;
typedef std::lock_guard<std::recursive_mutex> DevLock;

int fail(int code, const std::string& msg) {
  g_last_error = msg;
  return code;
}

#define HIP_TRY(expr)                                                                   \
  do {                                                                                  \
    hipError_t e_ = (expr);                                                             \
    if (e_ != hipSuccess)                                                               \
      return fail(AE_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));       \
  } while (0)

template <class T>
int dalloc(T** p, size_t count) {
  void* v = nullptr;
  DevLock lock(g_dev_mu);
  hipError_t e = hipMalloc(&v, count * sizeof(T) > 0 ? count * sizeof(T) : 16);
  if (e != hipSuccess) return fail(AE_ERR_HIP, std::string("hipMalloc: ") + hipGetErrorString(e));
  *p = static_cast<T*>(v);
  return AE_OK;
}

template <class T>
int dupload(T** p, const T* src, size_t count) {
  DevLock lock(g_dev_mu);
  if (int rc = dalloc(p, count)) return rc;
  if (count) HIP_TRY(hipMemcpy(*p, src, count * sizeof(T), hipMemcpyHostToDevice));
  return AE_OK;
}

int check_device(int* dev_out) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return fail(AE_ERR_UNSUPPORTED, "no HIP device available");
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  hipDeviceProp_t prop;
  HIP_TRY(hipGetDeviceProperties(&prop, dev));
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0)
    return fail(AE_ERR_UNSUPPORTED, std::string("device is ") + prop.gcnArchName + ", this build targets gfx950");
  *dev_out = dev;
  return AE_OK;
}

void free_all(std::vector<void*>& ptrs) {
  DevLock lock(g_dev_mu);
  for (void* p : ptrs)
    if (p) (void)hipFree(p);
  ptrs.clear();
}

// pinned host memory that grows on demand (kept across calls; freed with its owner)
struct PinnedBuf {
  void* p = nullptr;
  size_t bytes = 0;
  int ensure(size_t b) {
    if (b <= bytes) return AE_OK;
    DevLock lock(g_dev_mu);
    if (p) (void)hipHostFree(p);
    p = nullptr;
    bytes = 0;
    HIP_TRY(hipHostMalloc(&p, b, hipHostMallocDefault));
    bytes = b;
    return AE_OK;
  }
  template <class T>
  T* as() const { return static_cast<T*>(p); }
  PinnedBuf() = default;
  PinnedBuf(const PinnedBuf&) = delete;
  PinnedBuf& operator=(const PinnedBuf&) = delete;
  ~PinnedBuf() {
    DevLock lock(g_dev_mu);
    if (p) (void)hipHostFree(p);
  }
};

}  // namespace

// PackedLinearInt8 (src/gemm.rs:165-181) on the device
struct ae_linear {
  int n = 0, k = 0;
  int8_t* w = nullptr;  // swizzled
  float* w_scale = nullptr;
  float* bias = nullptr;
  float* inv_smooth = nullptr;
  bool smooth_finite = false;  // every inv_smooth entry finite (the fused FFN's fast GELU needs it of FFN-down's)
  bool owns = false;
  ~ae_linear() {
    DevLock lock(g_dev_mu);
    if (owns) {
      (void)hipFree(w);
      (void)hipFree(w_scale);
      (void)hipFree(bias);
      (void)hipFree(inv_smooth);
    }
  }
};

namespace {
int make_linear(int n, int k, const int8_t* w_q, const float* w_scale, const float* bias, const float* inv_smooth,
                ae_linear* l) {
  if (n <= 0 || k <= 0 || n % 384 || k % 64) return fail(AE_ERR_INVALID_ARG, "linear shape must be n%384==0, k%64==0");
  l->n = n;
  l->k = k;
  l->owns = true;
  std::vector<int8_t> sw(size_t(n) * k);
  aek::swizzle_weights(n, k, w_q, sw.data());
  if (int rc = dupload(&l->w, sw.data(), sw.size())) return rc;
  if (int rc = dupload(&l->w_scale, w_scale, size_t(n))) return rc;
  if (int rc = dupload(&l->bias, bias, size_t(n))) return rc;
  if (int rc = dupload(&l->inv_smooth, inv_smooth, size_t(k))) return rc;
  l->smooth_finite = std::all_of(inv_smooth, inv_smooth + k, [](float v) { return std::isfinite(v); });
  return AE_OK;
}
size_t linear_bytes(const ae_linear& l) { return size_t(l.n) * l.k + (size_t(l.n) * 2 + l.k) * 4; }
}  // namespace

struct DevLayer {
  ae_linear qkv, q_only, kv_only, attn_out, ffn_inter, ffn_out;
  float* qkv_smooth = nullptr;  // layer's qkv.inv_smooth (kept for layer 11 where qkv has no weights)
  float *ln1_w = nullptr, *ln1_b = nullptr, *ln2_w = nullptr, *ln2_b = nullptr;
};

// ArcticEmbedS (src/lib.rs:34-38): immutable after open
struct ae_engine {
  int device = 0;
  int8_t* word_q = nullptr;
  float* word_s = nullptr;
  int8_t* pos_q = nullptr;
  float* pos_s = nullptr;
  float* type0 = nullptr;  // pre-dequantized token_type row 0 (src/model.rs:50-54)
  float* emb_ln_w = nullptr;
  float* emb_ln_b = nullptr;
  DevLayer layers[ae::kLayers];
  std::vector<void*> extra;  // plain device allocations owned by the engine
  size_t size_bytes = 0, raw_size_bytes = 0;
  std::unique_ptr<ae::Tokenizer> tokenizer;
  // the workspace of the embedding calls made without one (ws == NULL: the
  // reference's embed_batch(&self, ...) owns its scratch), created on first use
  // and grown on demand; one call at a time
  mutable std::mutex own_mu;
  mutable ae_workspace* own_ws = nullptr;
  ~ae_engine();
};

// Workspace (src/model.rs:123-173): per-thread device scratch + stream
struct ae_workspace {
  const ae_engine* e = nullptr;
  hipStream_t stream = nullptr;
  // a second stream and its fork / join events: the fused FFN's launch of short
  // workgroups in a mixed plan runs there beside the 64-row one (aek::launch_ffn)
  hipStream_t side = nullptr;
  hipEvent_t fork_ev = nullptr, join_ev = nullptr;
  int max_tokens = 0, max_seqs = 0;
  uint16_t* ids = nullptr;
  int* cu = nullptr;
  int* cu_safe = nullptr;    // [max_seqs + 1]: the checked segment bounds every kernel after the first reads
  int* attn_plan = nullptr;  // attention work plan, attention_plan_ints(max_seqs, max_tokens)
  // AE_ATTENTION_QUANTIZED (ae_workspace_set_attention_mode): the reference's
  // ArmSme attention in layers 0-10; its scratch is allocated when the mode is set
  int attention_mode = AE_ATTENTION_EXACT;
  aek::SmeArgs sme{};
  int* err = nullptr;        // device error word: bit 0 = a packed batch with a bad segment (ae_workspace_synchronize)
  float *hidden = nullptr, *tmp = nullptr, *qkv = nullptr, *ctx = nullptr;
  float* g = nullptr;        // [min(max_tokens, kSmallM), 1536]: the FFN's intermediate of the few-row path (and rowmax_g)
  int8_t* act_q = nullptr;
  float* act_scale = nullptr;
  uint32_t *rowmax_ctx = nullptr, *rowmax_g = nullptr;
  float2* ln2_stats = nullptr;  // [T]: LN2's (mean, rstd) per row, when the next layer recomputes its output
  float *hidden_c = nullptr, *tmp_c = nullptr, *ctx_c = nullptr, *g_c = nullptr, *out_c = nullptr;
  int8_t* act_q_c = nullptr;
  float* act_scale_c = nullptr;
  uint32_t *rowmax_ctx_c = nullptr, *rowmax_g_c = nullptr;
  // pinned host staging of the embedding calls (all device batches of one call), grown on demand
  PinnedBuf st_ids, st_cu, st_out;
  std::vector<void*> dev;  // the device buffers sized by the capacity (max_tokens, max_seqs)
  // per-kernel timing (ae_workspace_set_timing): event pairs around launches
  bool timing = false;
  std::vector<hipEvent_t> ev_pool;
  std::vector<std::pair<int, int>> ev_marks;  // (kind, index of the start event)
  size_t ev_used = 0;
  double kind_ms[AE_KERNEL_KINDS] = {};
  int kind_count[AE_KERNEL_KINDS] = {};
  // replay of captured forward passes (hipGraph), keyed by the launch parameters;
  // a key is captured on its second use, so one-off batch shapes stay eager
  // (the process-wide kernel-choice hooks are part of the key: a graph holds the
  // kernels chosen when it was captured)
  struct GraphKey {
    const void *ids, *cu, *out;
    hipStream_t st;
    int B, T, max_len;
    int attention_mode, attention_choice;
    int attention_form, ffn_rows, ffn_exact_gelu;
    bool operator==(const GraphKey& o) const {
      return ids == o.ids && cu == o.cu && out == o.out && st == o.st && B == o.B && T == o.T && max_len == o.max_len &&
             attention_mode == o.attention_mode && attention_choice == o.attention_choice && attention_form == o.attention_form && ffn_rows == o.ffn_rows &&
             ffn_exact_gelu == o.ffn_exact_gelu;
    }
  };
  struct GraphEntry {
    GraphKey key;
    hipGraphExec_t exec;  // null: seen once, not captured yet
    uint64_t last_use;
  };
  bool graphs = true;
  std::vector<GraphEntry> graph_cache;
  uint64_t graph_tick = 0;
  static constexpr size_t kGraphCacheSize = 8;
  ~ae_workspace() {
    DevLock lock(g_dev_mu);
    if (stream) (void)hipStreamSynchronize(stream);
    if (side) (void)hipStreamSynchronize(side);
    if (fork_ev) (void)hipEventDestroy(fork_ev);
    if (join_ev) (void)hipEventDestroy(join_ev);
    if (side) (void)hipStreamDestroy(side);
    for (GraphEntry& g : graph_cache)
      if (g.exec) (void)hipGraphExecDestroy(g.exec);
    for (hipEvent_t ev : ev_pool) (void)hipEventDestroy(ev);
    free_all(dev);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

ae_engine::~ae_engine() {
  delete own_ws;  // (its destructor waits for its stream: kernels still reading the weights below)
  free_all(extra);
}

namespace {

int upload_model(const ae::ModelRaw& m, ae_engine* e) {
  auto up_i8 = [&](int8_t** p, const std::vector<int8_t>& v) {
    int rc = dupload(p, v.data(), v.size());
    e->extra.push_back(*p);
    return rc;
  };
  auto up_f = [&](float** p, const float* v, size_t n) {
    int rc = dupload(p, v, n);
    e->extra.push_back(*p);
    return rc;
  };
  int rc;
  if ((rc = up_i8(&e->word_q, m.word_q)) || (rc = up_f(&e->word_s, m.word_s.data(), m.word_s.size())) ||
      (rc = up_i8(&e->pos_q, m.pos_q)) || (rc = up_f(&e->pos_s, m.pos_s.data(), m.pos_s.size())) ||
      (rc = up_f(&e->emb_ln_w, m.emb_ln_w.data(), ae::kHidden)) ||
      (rc = up_f(&e->emb_ln_b, m.emb_ln_b.data(), ae::kHidden)))
    return rc;
  std::vector<float> type0(ae::kHidden);
  for (int j = 0; j < ae::kHidden; j++) type0[j] = float(m.type_q[j]) * m.type_s[0];
  if ((rc = up_f(&e->type0, type0.data(), type0.size()))) return rc;
  size_t bytes = m.word_q.size() + m.pos_q.size() + (m.word_s.size() + m.pos_s.size() + 3 * ae::kHidden) * 4;
  for (int i = 0; i < ae::kLayers; i++) {
    const ae::LayerRaw& L = m.layers[i];
    DevLayer& D = e->layers[i];
    auto lin = [&](const ae::LinearRaw& r, ae_linear& d) {
      int c = make_linear(int(r.n_out), int(r.k_in), r.w_q.data(), r.w_scale.data(), r.bias.data(),
                          r.inv_smooth.data(), &d);
      bytes += linear_bytes(d);
      return c;
    };
    if (i < ae::kLayers - 1) {
      if ((rc = lin(L.qkv, D.qkv))) return rc;
    } else {
      if ((rc = lin(L.q_only, D.q_only)) || (rc = lin(L.kv_only, D.kv_only))) return rc;
    }
    if ((rc = lin(L.attn_out, D.attn_out)) || (rc = lin(L.ffn_inter, D.ffn_inter)) || (rc = lin(L.ffn_out, D.ffn_out)))
      return rc;
    if ((rc = up_f(&D.qkv_smooth, L.qkv.inv_smooth.data(), ae::kHidden)) ||
        (rc = up_f(&D.ln1_w, L.ln1_w.data(), ae::kHidden)) || (rc = up_f(&D.ln1_b, L.ln1_b.data(), ae::kHidden)) ||
        (rc = up_f(&D.ln2_w, L.ln2_w.data(), ae::kHidden)) || (rc = up_f(&D.ln2_b, L.ln2_b.data(), ae::kHidden)))
      return rc;
    bytes += ae::kHidden * 4 * 5;
  }
  e->size_bytes = bytes;
  return AE_OK;
}

// folds completed event pairs into the per-kind totals
void drain_timing(ae_workspace* ws) {
  for (const auto& m : ws->ev_marks) {
    float ms = 0.f;
    if (hipEventElapsedTime(&ms, ws->ev_pool[m.second], ws->ev_pool[m.second + 1]) == hipSuccess) {
      ws->kind_ms[m.first] += ms;
      ws->kind_count[m.first] += 1;
    }
  }
  ws->ev_marks.clear();
  ws->ev_used = 0;
}

// RAII event pair around the launches of one kernel kind (no-op unless timing)
struct KernelTimer {
  ae_workspace* ws;
  hipStream_t st;
  int idx = -1;
  KernelTimer(ae_workspace* w, hipStream_t s, int kind) : ws(w), st(s) {
    if (!ws->timing) return;
    if (ws->ev_used + 2 > ws->ev_pool.size()) return;
    idx = int(ws->ev_used);
    ws->ev_used += 2;
    ws->ev_marks.push_back({kind, idx});
    (void)hipEventRecord(ws->ev_pool[idx], st);
  }
  ~KernelTimer() {
    if (idx >= 0) (void)hipEventRecord(ws->ev_pool[idx + 1], st);
  }
};

static aek::FfnArgs ffn_args(const ae_linear& up, const ae_linear& down, int m, const int8_t* a, const float* a_scale,
                             const float* res, float* out) {
  aek::FfnArgs f{};
  f.M = m;
  f.A = a;
  f.a_scale = a_scale;
  f.w1 = up.w;
  f.w1_scale = up.w_scale;
  f.b1 = up.bias;
  f.g_smooth = down.inv_smooth;
  f.w2 = down.w;
  f.w2_scale = down.w_scale;
  f.b2 = down.bias;
  f.res = res;
  f.out = out;
  f.fast_gelu = down.smooth_finite;
  return f;
}

// one forward pass over a token-packed batch already resident on the device
// (PackedModel::forward_ragged_cls, src/model.rs:521-914, without its 64-sequence /
// 512-token limits).  ids/cu may be the workspace's or the caller's buffers;
// max_len bounds every sequence length (it sizes the attention score rows);
// longest is the longest of them, where it is known (0: not), and chooses kernels.
// stop_layers >= 0 stops after the embedding and that many encoder layers
// (a test hook that leaves hidden / act_q / act_scale in the workspace).
int run_forward(ae_workspace* ws, const uint16_t* ids, const int* cu, int B, int T, int max_len, int longest,
                float* out, hipStream_t st, int stop_layers = -1) {
  const ae_engine* E = ws->e;
  using namespace aek;
  if (ws->timing && ws->ev_used + 2 * 80 > ws->ev_pool.size()) {
    // pool exhausted by passes not yet folded in: wait for them and fold
    (void)hipStreamSynchronize(st);
    drain_timing(ws);
  }
  auto gemm_args = [&](const ae_linear& L, int M, const void* A, const float* a_scale, const uint32_t* a_rowmax,
                       const float* a_smooth, const float* res, float* o, const float* g_smooth, uint32_t* g_rowmax) {
    GemmArgs p{};
    p.M = M;
    p.N = L.n;
    p.K = L.k;
    p.A = A;
    p.a_scale = a_scale;
    p.a_rowmax = a_rowmax;
    p.a_smooth = a_smooth;
    p.w = L.w;
    p.w_scale = L.w_scale;
    p.bias = L.bias;
    p.res = res;
    p.out = o;
    p.g_smooth = g_smooth;
    p.g_rowmax = g_rowmax;
    return p;
  };
  auto gemm = [&](const ae_linear& L, int M, const void* A, int amode, const float* a_scale, const uint32_t* a_rowmax,
                  const float* a_smooth, const float* res, float* o, int emode, const float* g_smooth,
                  uint32_t* g_rowmax) {
    launch_gemm(gemm_args(L, M, A, a_scale, a_rowmax, a_smooth, res, o, g_smooth, g_rowmax), amode, emode, st);
  };
  auto ln_args = [&](const float* src, float* dst, const float* gw, const float* gb, const float* smooth, int8_t* q,
                     float* scale, uint32_t* rowmax_init, int rows, uint32_t* rowmax_init2 = nullptr) {
    LnArgs p{};
    p.T = rows;
    p.src = src;
    p.dst = dst;
    p.gamma = gw;
    p.beta = gb;
    p.smooth = smooth;
    p.q = q;
    p.scale = scale;
    p.rowmax_init = rowmax_init;
    p.rowmax_init2 = rowmax_init2;
    return p;
  };
  {  // embeddings + LayerNorm + SmoothQuant (src/model.rs:549-586)
    KernelTimer kt(ws, st, AE_KERNEL_EMBED_LN);
    LnArgs p{};
    p.T = T;
    p.ids = ids;
    p.cu = cu;
    p.B = B;
    p.word_q = E->word_q;
    p.word_s = E->word_s;
    p.pos_q = E->pos_q;
    p.pos_s = E->pos_s;
    p.type0 = E->type0;
    p.gamma = E->emb_ln_w;
    p.beta = E->emb_ln_b;
    p.smooth = E->layers[0].qkv_smooth;
    p.dst = ws->hidden;
    p.q = ws->act_q;
    p.scale = ws->act_scale;
    p.rowmax_init = ws->rowmax_ctx;
    p.rowmax_init2 = gemm_small_path(T) ? ws->rowmax_g : nullptr;
    p.rowmax_c = ws->rowmax_ctx_c;  // the layer-11 [CLS] rows' targets (row b < B)
    p.rowmax_c2 = ws->rowmax_g_c;
    p.n_c = B;
    p.max_len = max_len;
    p.err = ws->err;
    p.cu_safe = ws->cu_safe;
    launch_ln_quant(p, kLnSrcEmb, st);
  }
  // every later kernel reads the checked copy of cu written by the embedding
  // kernel: a malformed device-resident cu_seqlens then gives wrong values (and
  // the error word), never an access outside the batch's rows
  cu = ws->cu_safe;
  const int s_pitch = attention_pitch(max_len);
  // AE_ATTENTION_QUANTIZED: every sequence as forward_cls runs it on the
  // reference's ArmSme backend (src/model.rs:244-259): the quantized attention
  // with that sequence's own V scales from 16 tokens on, the exact one below,
  // so a sequence's result does not depend on its batch mates
  const bool sme = ws->attention_mode == AE_ATTENTION_QUANTIZED && max_len >= 16;
  if (sme && !ws->sme.vt) return fail(AE_ERR_INVALID_ARG, "quantized attention scratch missing");
  SmeArgs sme_args = ws->sme;
  sme_args.per_seq = 1;
  // Few rows (gemm_small_path): every LayerNorm runs in the prologue of the GEMM
  // that consumes it (QKV, FFN-up, the layer-11 K/V), whose column-tile-0
  // workgroups also store its outputs; the attention output GEMM runs inside the
  // FFN-up kernel, in front of LN1 (each workgroup for its 16 rows), and LN1's
  // output (the FFN-down residual, updated in place) lives in tmp.  The
  // row-absmax targets of a layer (attention -> rowmax_ctx, GELU -> rowmax_g)
  // are reset by the LayerNorm that precedes the layer.
  const bool small = gemm_small_path(T);
  const float* ln2_w = nullptr;  // small: the previous layer's LN2, applied by the next QKV prologue
  const float* ln2_b = nullptr;
  // Many rows (every other batch): the FFN block is one kernel (launch_ffn).  It
  // starts where the few-row path ends because a launch takes 18 us with any
  // number of 16-row workgroups up to one per CU, while the FFN-up and FFN-down
  // GEMMs took 16 + 30 us at 1,280 rows and 18 + 30 at 3,776 (few workgroups,
  // 24 dependent K steps each in FFN-down).  LN2 then writes its (mean, rstd) per
  // row instead of its f32 output: the next attention-output kernel, its only
  // reader, recomputes that output from LN2's input rows (tmp) as LN2 forms it,
  // and the [CLS] gather of layer 11 does so for its rows.  This saves LN2's f32
  // store (T x 1536 bytes per layer).  The last layer of a truncated pass
  // (stop_layers) still stores it: it is the state returned.
  const bool ln2_stats = !small;
  for (int l = 0; l < ae::kLayers - 1; l++) {  // src/model.rs:593-768
    if (stop_layers >= 0 && l >= stop_layers) break;
    const DevLayer& D = E->layers[l];
    {
      KernelTimer kt(ws, st, AE_KERNEL_GEMM_QKV);
      if (small && ln2_w) {
        launch_gemm_ln_prologue(gemm_args(D.qkv, T, ws->tmp, nullptr, nullptr, nullptr, nullptr, ws->qkv, nullptr,
                                          nullptr),
                                ln_args(ws->tmp, ws->hidden, ln2_w, ln2_b, D.qkv_smooth, nullptr, nullptr,
                                        ws->rowmax_ctx, T, ws->rowmax_g),
                                st);
      } else {
        GemmArgs g = gemm_args(D.qkv, T, ws->act_q, ws->act_scale, nullptr, nullptr, nullptr, ws->qkv, nullptr, nullptr);
        // Q is read once by the attention; K and V many times: only K and V
        // are left in the Infinity Cache
        g.stream_cols = 384;
        launch_gemm(g, kAI8, kEpiF32, st);
      }
    }
    {
      KernelTimer kt(ws, st, AE_KERNEL_ATTENTION);
      AttnArgs a{ws->qkv, cu, B, ws->attn_plan, ws->ctx, D.attn_out.inv_smooth, ws->rowmax_ctx, s_pitch};
      // one sequence: its only segment is [0, T) (a cu_seqlens saying otherwise sets the error word)
      if (B == 1) a.len1 = T;
      a.longest = longest;
      if (sme) {
        launch_attention_sme(a, sme_args, T, st, /*plan=*/l == 0);
        launch_attention_short(a, st);
      } else {
        launch_attention(a, T, st, /*plan=*/l == 0);  // the tile plan depends only on cu: built once
      }
    }
    if (small) {
      {  // attention output GEMM + LN1 + FFN-up/GELU in one kernel; LN1's output goes to tmp
        KernelTimer kt(ws, st, AE_KERNEL_GEMM_FFN_UP);
        const PreArgs pre{ws->ctx, ws->rowmax_ctx, D.attn_out.inv_smooth, D.attn_out.w, D.attn_out.w_scale,
                          D.attn_out.bias, ws->hidden};
        launch_gemm_pre_ln(gemm_args(D.ffn_inter, T, nullptr, nullptr, nullptr, nullptr, nullptr, ws->g,
                                     D.ffn_out.inv_smooth, ws->rowmax_g),
                           pre,
                           ln_args(nullptr, ws->tmp, D.ln1_w, D.ln1_b, D.ffn_inter.inv_smooth, nullptr, nullptr,
                                   nullptr, T),
                           st);
      }
      {  // residual LN1(h) in tmp, written in place
        KernelTimer kt(ws, st, AE_KERNEL_GEMM_FFN_DOWN);
        gemm(D.ffn_out, T, ws->g, kAF32Q, nullptr, ws->rowmax_g, nullptr, ws->tmp, ws->tmp, kEpiF32, nullptr,
             nullptr);
      }
      ln2_w = D.ln2_w;
      ln2_b = D.ln2_b;
      continue;
    }
    {
      GemmArgs g = gemm_args(D.attn_out, T, ws->ctx, nullptr, ws->rowmax_ctx, D.attn_out.inv_smooth, ws->hidden,
                             ws->tmp, nullptr, nullptr);
      if (ln2_stats && l > 0) {  // the residual: the previous layer's LN2 of tmp, recomputed
        g.res = ws->tmp;
        g.res_stats = ws->ln2_stats;
        g.res_gamma = E->layers[l - 1].ln2_w;
        g.res_beta = E->layers[l - 1].ln2_b;
      }
      KernelTimer kt(ws, st, AE_KERNEL_GEMM_ATTN_OUT);  // and LN1, in the same kernel
      launch_gemm_ln(g,
                     ln_args(ws->tmp, ws->hidden, D.ln1_w, D.ln1_b, D.ffn_inter.inv_smooth, ws->act_q, ws->act_scale,
                             nullptr, T),
                     st);
    }
    LnArgs ln2 = ln_args(ws->tmp, ws->hidden, D.ln2_w, D.ln2_b, E->layers[l + 1].qkv_smooth, ws->act_q,
                         ws->act_scale, ws->rowmax_ctx, T);
    if (ln2_stats) {
      ln2.stats = ws->ln2_stats;
      if (!(stop_layers >= 0 && l + 1 == stop_layers)) ln2.dst = nullptr;
    }
    const FfnArgs ffn = ffn_args(D.ffn_inter, D.ffn_out, T, ws->act_q, ws->act_scale, ws->hidden, ws->tmp);
    {  // FFN-up, GELU, quantize and FFN-down in one kernel (up to 4,096 rows, LN2 too)
      KernelTimer kt(ws, st, AE_KERNEL_GEMM_FFN_UP);
      if (launch_ffn(ffn, st, ws->side, ws->fork_ev, ws->join_ev, &ln2)) continue;
    }
    KernelTimer kt(ws, st, AE_KERNEL_LN2);
    launch_ln_quant(ln2, kLnSrcF32, st);
  }
  if (stop_layers >= 0) {
    if (small && ln2_w) {  // the state after the last layer run: its LN2, as the next QKV would apply it
      const int s = std::min(stop_layers, ae::kLayers - 1);
      launch_ln_quant(ln_args(ws->tmp, ws->hidden, ln2_w, ln2_b, E->layers[s].qkv_smooth, ws->act_q, ws->act_scale,
                              ws->rowmax_ctx, T),
                      kLnSrcF32, st);
    }
    hipError_t err = hipGetLastError();
    return err == hipSuccess ? AE_OK : fail(AE_ERR_HIP, std::string("kernel launch: ") + hipGetErrorString(err));
  }
  // layer 11: [CLS] pruning (src/model.rs:770-913)
  KernelTimer kt(ws, st, AE_KERNEL_LAYER11_TAIL);
  const DevLayer& D = E->layers[ae::kLayers - 1];
  float* kv = ws->qkv;  // [T,768]
  if (small) {  // layer 10's LN2 in the K/V GEMM's prologue; the [CLS] gather reads its act_q / act_scale
    launch_gemm_ln_prologue(gemm_args(D.kv_only, T, ws->tmp, nullptr, nullptr, nullptr, nullptr, kv, nullptr, nullptr),
                            ln_args(ws->tmp, ws->hidden, ln2_w, ln2_b, D.qkv_smooth, ws->act_q, ws->act_scale, nullptr,
                                    T),
                            st);
  } else {
    gemm(D.kv_only, T, ws->act_q, kAI8, ws->act_scale, nullptr, nullptr, nullptr, kv, kEpiF32, nullptr, nullptr);
  }
  const bool small_tail = gemm_small_path(B);
  ClsArgs c{};
  c.B = B;
  c.cu = cu;
  c.hidden = ws->hidden;
  c.act_q = ws->act_q;
  c.act_scale = ws->act_scale;
  c.hidden_c = ws->hidden_c;
  c.wq = D.q_only.w;
  c.wq_scale = D.q_only.w_scale;
  c.wq_bias = D.q_only.bias;
  c.kv = kv;
  c.ctx_c = ws->ctx_c;
  c.smooth = D.attn_out.inv_smooth;
  c.rowmax_ctx_c = ws->rowmax_ctx_c;  // reset by the embedding kernel
  c.max_len = std::min(max_len, ae::kMaxPos);
  if (ln2_stats) {  // layer 10's LN2 output for the [CLS] rows, recomputed from tmp
    c.hidden = ws->tmp;
    c.hidden_stats = ws->ln2_stats;
    c.ln_gamma = E->layers[ae::kLayers - 2].ln2_w;
    c.ln_beta = E->layers[ae::kLayers - 2].ln2_b;
  }
  launch_cls(c, st);
  if (small_tail) {  // attention output + LN1 + FFN-up in one kernel (rowmax_g_c reset by the embedding kernel)
    const PreArgs pre{ws->ctx_c, ws->rowmax_ctx_c, D.attn_out.inv_smooth, D.attn_out.w, D.attn_out.w_scale,
                      D.attn_out.bias, ws->hidden_c};
    launch_gemm_pre_ln(gemm_args(D.ffn_inter, B, nullptr, nullptr, nullptr, nullptr, nullptr, ws->g_c,
                                 D.ffn_out.inv_smooth, ws->rowmax_g_c),
                       pre,
                       ln_args(nullptr, ws->tmp_c, D.ln1_w, D.ln1_b, D.ffn_inter.inv_smooth, nullptr, nullptr, nullptr,
                               B),
                       st);
    gemm(D.ffn_out, B, ws->g_c, kAF32Q, nullptr, ws->rowmax_g_c, nullptr, ws->tmp_c, ws->tmp_c, kEpiF32, nullptr,
         nullptr);
    launch_final_ln_l2(B, ws->tmp_c, D.ln2_w, D.ln2_b, out, st);
  } else {
    {
      const GemmArgs g = gemm_args(D.attn_out, B, ws->ctx_c, nullptr, ws->rowmax_ctx_c, D.attn_out.inv_smooth,
                                   ws->hidden_c, ws->tmp_c, nullptr, nullptr);
      const LnArgs l = ln_args(ws->tmp_c, ws->tmp_c, D.ln1_w, D.ln1_b, D.ffn_inter.inv_smooth, ws->act_q_c,
                               ws->act_scale_c, ws->rowmax_g_c, B);
      launch_gemm_ln(g, l, st);
    }
    gemm(D.ffn_inter, B, ws->act_q_c, kAI8, ws->act_scale_c, nullptr, nullptr, nullptr, ws->g_c, kEpiGelu,
         D.ffn_out.inv_smooth, ws->rowmax_g_c);
    gemm(D.ffn_out, B, ws->g_c, kAF32Q, nullptr, ws->rowmax_g_c, nullptr, ws->tmp_c, ws->hidden_c, kEpiF32, nullptr,
         nullptr);
    launch_final_ln_l2(B, ws->hidden_c, D.ln2_w, D.ln2_b, out, st);
  }
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return fail(AE_ERR_HIP, std::string("kernel launch: ") + hipGetErrorString(err));
  return AE_OK;
}

// run_forward through the workspace's graph cache: the same launch parameters a
// second time are captured into a hipGraph, later calls replay it (one launch
// instead of ~90).  Eager when timing is on or the stream is already capturing.
int run_forward_replay(ae_workspace* ws, const uint16_t* ids, const int* cu, int B, int T, int max_len, int longest,
                       float* out, hipStream_t st) {
  if (!ws->graphs || ws->timing) return run_forward(ws, ids, cu, B, T, max_len, longest, out, st);
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone)
    return run_forward(ws, ids, cu, B, T, max_len, longest, out, st);
  // (of longest, a graph holds only the attention kernels that it chose)
  const int choice = ws->attention_mode == AE_ATTENTION_EXACT
                         ? aek::attention_choice(B, T, aek::attention_pitch(max_len) - 4, longest, aek::device_cu_count())
                         : 0;
  const ae_workspace::GraphKey key{ids, cu, out, st, B, T, max_len, ws->attention_mode, choice, aek::attention_form(),
                                   aek::ffn_rows(), aek::ffn_exact_gelu() ? 1 : 0};
  ws->graph_tick++;
  ae_workspace::GraphEntry* hit = nullptr;
  for (auto& g : ws->graph_cache)
    if (g.key == key) hit = &g;
  if (hit && hit->exec) {
    hit->last_use = ws->graph_tick;
    HIP_TRY(hipGraphLaunch(hit->exec, st));
    return AE_OK;
  }
  if (!hit) {  // first use: remember the key, run eagerly
    if (ws->graph_cache.size() >= ae_workspace::kGraphCacheSize) {
      auto lru = std::min_element(ws->graph_cache.begin(), ws->graph_cache.end(),
                                  [](const auto& a, const auto& b) { return a.last_use < b.last_use; });
      if (lru->exec) {
        DevLock lock(g_dev_mu);
        (void)hipGraphExecDestroy(lru->exec);
      }
      ws->graph_cache.erase(lru);
    }
    ws->graph_cache.push_back({key, nullptr, ws->graph_tick});
    return run_forward(ws, ids, cu, B, T, max_len, longest, out, st);
  }
  // second use: capture, instantiate, launch
  DevLock lock(g_dev_mu);
  HIP_TRY(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
  const int rc = run_forward(ws, ids, cu, B, T, max_len, longest, out, st);
  hipGraph_t graph = nullptr;
  const hipError_t end = hipStreamEndCapture(st, &graph);
  if (rc != AE_OK) {
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  if (end != hipSuccess || !graph) return fail(AE_ERR_HIP, std::string("graph capture: ") + hipGetErrorString(end));
  hipGraphExec_t exec = nullptr;
  const hipError_t inst = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  if (inst != hipSuccess) return fail(AE_ERR_HIP, std::string("graph instantiate: ") + hipGetErrorString(inst));
  hit->exec = exec;
  hit->last_use = ws->graph_tick;
  HIP_TRY(hipGraphLaunch(exec, st));
  return AE_OK;
}

int grow_workspace(ae_workspace* ws, size_t T, size_t B);

// An embedding call grows the workspace (once) so that the whole request runs in
// as few device batches as these bounds allow (10 KB of device memory per token).
constexpr size_t kGrowTokens = size_t(1) << 18;
constexpr size_t kGrowSeqs = 8192;
// Batches of at most this many tokens are padded to a bucketed shape (below),
// so that ragged batches of similar size replay one captured graph: below a few
// thousand tokens a pass is bound by its ~90 launches rather than by the GPU.
constexpr int kBucketMaxTokens = 16384;

// The bucketed shape of a batch of B sequences, T tokens, longest max_len:
// max_len up to a power of two (32 .. 512), T up to a multiple of a quarter of
// its binade (at least 256), B up to a multiple of 8, with the extra tokens in
// extra (dummy) sequences of 1 .. Lp tokens each.  Sequences are independent
// (every operation is row-local or bounded by its segment), so the dummies
// change no real sequence's result.  False if it does not fit the capacity.
bool bucket_shape(int B, int T, int max_len, int cap_T, int cap_B, int* Bp, int* Tp, int* Lp) {
  int L = 32;
  while (L < max_len) L *= 2;
  int q = 256;
  while (q * 8 <= T) q *= 2;
  auto up = [](int x, int m) { return (x + m - 1) / m * m; };
  int tp = up(T + 1, q);
  for (int it = 0; it < 4; it++) {
    const int P = tp - T;
    const int bp = up(B + (P + L - 1) / L, 8);  // room for P tokens of at most L each
    if (bp - B <= P) {                           // and at least one token per dummy
      *Bp = bp;
      *Tp = tp;
      *Lp = L;
      return bp <= cap_B && tp <= cap_T;
    }
    tp = up(T + (bp - B), q);
  }
  return false;
}

struct DevBatch {
  size_t first;      // first sequence (in length order)
  int B, T;          // real sequences and tokens
  int Bp, Tp, Lp;    // the launched shape (bucketed, or the real one)
  int longest;       // its longest sequence, the dummies of a bucketed shape included
  size_t ids_off, cu_off;
};

// Runs `n` pre-tokenized sequences (already validated and truncated) through as
// few device batches as the workspace capacity allows, growing the workspace
// first where the request needs more.  Sequences are length-sorted so each
// batch packs similar lengths (length-bucketed packing); small batches are
// padded to a bucketed shape and replay its captured graph.  Every batch's ids
// are staged in pinned memory and all batches are queued on the workspace
// stream with their copies (no host synchronization until the last batch's
// embeddings are back); the results are then scattered to input order.
int run_sequences(const ae_engine* e, ae_workspace* ws, const std::vector<const uint16_t*>& seqs,
                  const std::vector<int>& lens, float* out) {
  (void)e;
  const size_t n = seqs.size();
  std::vector<size_t> order(n);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) { return lens[a] < lens[b]; });
  size_t total = 0;
  for (int L : lens) total += size_t(L);
  if (n > 1) {  // (single sequences keep the caller's capacity: the latency mode's workspace)
    const size_t want_T = std::min(total <= size_t(kBucketMaxTokens) ? total + total / 4 + 512 : total, kGrowTokens);
    const size_t want_B = std::min(n + 16, kGrowSeqs);
    if (size_t(ws->max_tokens) < want_T || size_t(ws->max_seqs) < want_B)
      if (int rc = grow_workspace(ws, want_T, want_B)) return rc;
  }
  std::vector<DevBatch> plan;
  size_t ids_total = 0, cu_total = 0;
  for (size_t i = 0; i < n;) {
    DevBatch d{};
    d.first = i;
    size_t j = i;
    while (j < n && d.B < ws->max_seqs && d.T + lens[order[j]] <= ws->max_tokens) {
      d.T += lens[order[j]];
      d.B++;
      j++;
    }
    if (d.B == 0) return fail(AE_ERR_CAPACITY, "sequence longer than the workspace token capacity");
    const int max_len = lens[order[j - 1]];  // length-sorted: the last is the longest
    if (!(d.B >= 2 && d.T <= kBucketMaxTokens &&
          bucket_shape(d.B, d.T, max_len, ws->max_tokens, ws->max_seqs, &d.Bp, &d.Tp, &d.Lp))) {
      d.Bp = d.B;
      d.Tp = d.T;
      d.Lp = max_len;
    }
    const int D = d.Bp - d.B;
    d.longest = D ? std::max(max_len, (d.Tp - d.T + D - 1) / D) : max_len;
    d.ids_off = ids_total;
    d.cu_off = cu_total;
    ids_total += size_t(d.Tp);
    cu_total += size_t(d.Bp) + 1;
    plan.push_back(d);
    i = j;
  }
  // pinned staging for the whole request (the stream may still read the old buffers)
  if (ws->st_ids.bytes < ids_total * 2 || ws->st_cu.bytes < cu_total * 4 || ws->st_out.bytes < n * ae::kHidden * 4)
    HIP_TRY(hipStreamSynchronize(ws->stream));
  if (int rc = ws->st_ids.ensure(ids_total * sizeof(uint16_t))) return rc;
  if (int rc = ws->st_cu.ensure(cu_total * sizeof(int))) return rc;
  if (int rc = ws->st_out.ensure(n * ae::kHidden * sizeof(float))) return rc;
  uint16_t* h_ids = ws->st_ids.as<uint16_t>();
  int* h_cu = ws->st_cu.as<int>();
  float* h_out = ws->st_out.as<float>();
  for (const DevBatch& d : plan) {
    uint16_t* bi = h_ids + d.ids_off;
    int* bc = h_cu + d.cu_off;
    bc[0] = 0;
    for (int b = 0; b < d.B; b++) {
      const size_t s = order[d.first + b];
      std::memcpy(bi + bc[b], seqs[s], size_t(lens[s]) * sizeof(uint16_t));
      bc[b + 1] = bc[b] + lens[s];
    }
    const int D = d.Bp - d.B, P = d.Tp - d.T;  // dummy sequences: [PAD] ids, 1 .. Lp tokens each
    for (int k = 0; k < D; k++) bc[d.B + k + 1] = bc[d.B + k] + P / D + (k < P % D ? 1 : 0);
    std::memset(bi + d.T, 0, size_t(P) * sizeof(uint16_t));
    HIP_TRY(hipMemcpyAsync(ws->ids, bi, size_t(d.Tp) * sizeof(uint16_t), hipMemcpyHostToDevice, ws->stream));
    HIP_TRY(hipMemcpyAsync(ws->cu, bc, size_t(d.Bp + 1) * sizeof(int), hipMemcpyHostToDevice, ws->stream));
    if (int rc = run_forward_replay(ws, ws->ids, ws->cu, d.Bp, d.Tp, d.Lp, d.longest, ws->out_c, ws->stream))
      return rc;
    HIP_TRY(hipMemcpyAsync(h_out + d.first * ae::kHidden, ws->out_c, size_t(d.B) * ae::kHidden * sizeof(float),
                           hipMemcpyDeviceToHost, ws->stream));
  }
  HIP_TRY(hipStreamSynchronize(ws->stream));
  for (size_t k = 0; k < n; k++)
    std::memcpy(out + order[k] * ae::kHidden, h_out + k * ae::kHidden, ae::kHidden * sizeof(float));
  return AE_OK;
}

int check_ids(const uint16_t* ids, size_t n) {
  for (size_t i = 0; i < n; i++)
    if (ids[i] >= ae::kVocab) return fail(AE_ERR_INVALID_ARG, "token id " + std::to_string(ids[i]) + " >= vocab size");
  return AE_OK;
}

// the longest sequence by the max_seq_len that a caller states: a program that
// gives the model's limit says nothing about its batch
int stated_longest(int max_seq_len) { return max_seq_len < ae::kMaxPos ? max_seq_len : 0; }

hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

// The quantized attention's scratch for the workspace capacity (int8 Q and K,
// their scales, the |V| column maxima per sequence and the transposed int8 V),
// allocated once.  All-or-nothing: on a failed allocation the ones already made
// are freed and ws->sme stays empty.
int alloc_sme_scratch(ae_workspace* ws) {
  if (ws->sme.vt) return AE_OK;
  HIP_TRY(hipSetDevice(ws->e->device));
  DevLock lock(g_dev_mu);
  const size_t T = size_t(ws->max_tokens), B = size_t(ws->max_seqs);
  const size_t bytes[7] = {T * 384, T * 384, T * 12 * 4, T * 12 * 4, B * 384 * 4,
                           384 * aek::sme_vt_len(ws->max_tokens, ws->max_seqs), T * 4};
  void* p[7] = {};
  for (int i = 0; i < 7; i++) {
    const hipError_t e = hipMalloc(&p[i], bytes[i]);
    if (e != hipSuccess) {
      for (int j = 0; j < i; j++) (void)hipFree(p[j]);
      return fail(AE_ERR_HIP, std::string("quantized attention scratch: ") + hipGetErrorString(e));
    }
  }
  for (void* q : p) ws->dev.push_back(q);
  aek::SmeArgs s{};
  s.q8 = static_cast<int8_t*>(p[0]);
  s.k8 = static_cast<int8_t*>(p[1]);
  s.qs = static_cast<float*>(p[2]);
  s.ks = static_cast<float*>(p[3]);
  s.vmax = static_cast<uint32_t*>(p[4]);
  s.vt = static_cast<int8_t*>(p[5]);
  s.tseg = static_cast<int*>(p[6]);
  aek::init_attention_sme_kernels();
  ws->sme = s;
  return AE_OK;
}

// The device buffers sized by a workspace's capacity (T tokens, B sequences),
// replacing any it held (the quantized attention's scratch included: the caller
// allocates it again where the mode needs it).
int alloc_capacity(ae_workspace* ws, size_t T, size_t B) {
  DevLock lock(g_dev_mu);
  free_all(ws->dev);
  ws->sme = aek::SmeArgs{};
  ws->max_tokens = ws->max_seqs = 0;
  auto A = [&](auto** p, size_t count) {
    int rc = dalloc(p, count);
    if (rc == AE_OK) ws->dev.push_back(*p);
    return rc;
  };
  const size_t Ts = std::min(T, size_t(aek::kSmallM));  // only the few-row path holds the FFN's intermediate
  int rc;
  if ((rc = A(&ws->ids, T)) || (rc = A(&ws->cu, B + 1)) || (rc = A(&ws->cu_safe, B + 1)) ||
      (rc = A(&ws->err, size_t(1))) || (rc = A(&ws->attn_plan, aek::attention_plan_ints(int(B), int(T)))) ||
      (rc = A(&ws->hidden, T * 384)) || (rc = A(&ws->tmp, T * 384)) || (rc = A(&ws->qkv, T * 1152)) ||
      (rc = A(&ws->ctx, T * 384)) || (rc = A(&ws->g, Ts * 1536)) || (rc = A(&ws->act_q, T * 384)) ||
      (rc = A(&ws->act_scale, T)) || (rc = A(&ws->rowmax_ctx, T)) || (rc = A(&ws->rowmax_g, Ts)) ||
      (rc = A(&ws->ln2_stats, T)) ||
      (rc = A(&ws->hidden_c, B * 384)) || (rc = A(&ws->tmp_c, B * 384)) ||
      (rc = A(&ws->ctx_c, B * 384)) || (rc = A(&ws->g_c, B * 1536)) || (rc = A(&ws->out_c, B * 384)) ||
      (rc = A(&ws->act_q_c, B * 384)) || (rc = A(&ws->act_scale_c, B)) || (rc = A(&ws->rowmax_ctx_c, B)) ||
      (rc = A(&ws->rowmax_g_c, B))) {
    free_all(ws->dev);
    return rc;
  }
  HIP_TRY(hipMemsetAsync(ws->err, 0, sizeof(int), ws->stream));
  HIP_TRY(hipStreamSynchronize(ws->stream));
  ws->max_tokens = int(T);
  ws->max_seqs = int(B);
  return AE_OK;
}

// Grows a workspace to at least (T tokens, B sequences): waits for its stream,
// drops its captured graphs (they name the old buffers), allocates the new
// capacity and carries the device error word and the quantized attention's
// scratch over.  If the larger allocation fails the old capacity is restored.
int grow_workspace(ae_workspace* ws, size_t T, size_t B) {
  T = std::max(T, size_t(ws->max_tokens));
  B = std::max(B, size_t(ws->max_seqs));
  HIP_TRY(hipSetDevice(ws->e->device));
  DevLock lock(g_dev_mu);
  int err = 0;
  HIP_TRY(hipMemcpyAsync(&err, ws->err, sizeof(int), hipMemcpyDeviceToHost, ws->stream));
  HIP_TRY(hipStreamSynchronize(ws->stream));
  for (auto& g : ws->graph_cache)
    if (g.exec) (void)hipGraphExecDestroy(g.exec);
  ws->graph_cache.clear();
  const size_t T0 = size_t(ws->max_tokens), B0 = size_t(ws->max_seqs);
  int rc = alloc_capacity(ws, T, B);
  if (rc != AE_OK) {
    const std::string msg = g_last_error;
    if (alloc_capacity(ws, T0, B0) == AE_OK && ws->attention_mode == AE_ATTENTION_QUANTIZED) (void)alloc_sme_scratch(ws);
    return fail(rc, msg);
  }
  if (err) {
    HIP_TRY(hipMemcpyAsync(ws->err, &err, sizeof(int), hipMemcpyHostToDevice, ws->stream));
    HIP_TRY(hipStreamSynchronize(ws->stream));
  }
  if (ws->attention_mode == AE_ATTENTION_QUANTIZED)
    if (int rc2 = alloc_sme_scratch(ws)) return rc2;
  return AE_OK;
}

}  // namespace

extern "C" {

const char* ae_last_error(void) { return g_last_error.c_str(); }
const char* ae_version(void) { return "arctic-embed-amd 0.1.0 (gfx950)"; }

size_t ae_default_model_dir(char* buf, size_t cap) {
  const char* env = std::getenv("ARCTIC_EMBED_MODEL_DIR");  // MODEL_DIR_ENV_VAR, src/lib.rs:22
  std::string d = env ? env : "model";
  if (buf && cap) {
    std::strncpy(buf, d.c_str(), cap - 1);
    buf[cap - 1] = 0;
  }
  return d.size() + 1;
}

int ae_engine_open_files(const char* ae8_path, const char* vocab_path, ae_engine** out) {
  if (!out || !ae8_path) return fail(AE_ERR_INVALID_ARG, "null argument");
  *out = nullptr;
  std::unique_ptr<ae_engine> e(new ae_engine());
  std::string err;
  if (vocab_path) {  // BertTokenizer::from_vocab_file (src/tokenizer.rs:34-37) is read first
    e->tokenizer.reset(new ae::Tokenizer());
    if (int rc = e->tokenizer->load_vocab_file(vocab_path, err)) return fail(rc, err);
  }
  ae::ModelRaw m;
  if (int rc = ae::load_ae8(ae8_path, m, err)) return fail(rc, err);
  if (int rc = ae::validate_model(m, err)) return fail(rc, err);
  e->raw_size_bytes = m.size_bytes();
  if (int rc = check_device(&e->device)) return rc;
  if (int rc = upload_model(m, e.get())) return rc;
  aek::init_attention_kernels();
  *out = e.release();
  return AE_OK;
}

int ae_engine_open(const char* dir, ae_engine** out) {
  std::string d;
  if (dir) {
    d = dir;
  } else {
    std::vector<char> buf(ae_default_model_dir(nullptr, 0));
    ae_default_model_dir(buf.data(), buf.size());
    d = buf.data();
  }
  const std::string vocab = d + "/vocab.txt", pack = d + "/model.ae8";  // VOCAB_FILE / MODEL_FILE
  return ae_engine_open_files(pack.c_str(), vocab.c_str(), out);
}

void ae_engine_close(ae_engine* e) {
  DevLock lock(g_dev_mu);
  if (e) (void)hipDeviceSynchronize();
  delete e;
}

size_t ae_engine_size_bytes(const ae_engine* e) { return e ? e->size_bytes : 0; }
size_t ae_engine_raw_size_bytes(const ae_engine* e) { return e ? e->raw_size_bytes : 0; }

int ae_workspace_create(const ae_engine* e, size_t max_tokens, size_t max_seqs, ae_workspace** out) {
  if (!e || !out) return fail(AE_ERR_INVALID_ARG, "null argument");
  *out = nullptr;
  if (max_tokens == 0) max_tokens = ae::kMaxPos;
  if (max_seqs == 0) max_seqs = 64;
  if (max_tokens < size_t(ae::kMaxPos) || max_tokens > (size_t(1) << 26) || max_seqs > max_tokens ||
      max_seqs >= size_t(aek::kPlanMaxSegs))
    return fail(AE_ERR_INVALID_ARG, "workspace needs 512 <= max_tokens <= 2^26 and max_seqs <= max_tokens, < 2^24");
  HIP_TRY(hipSetDevice(e->device));
  DevLock lock(g_dev_mu);
  std::unique_ptr<ae_workspace> ws(new ae_workspace());
  ws->e = e;
  ws->max_tokens = int(max_tokens);
  ws->max_seqs = int(max_seqs);
  HIP_TRY(hipStreamCreateWithFlags(&ws->stream, hipStreamNonBlocking));
  HIP_TRY(hipStreamCreateWithFlags(&ws->side, hipStreamNonBlocking));
  HIP_TRY(hipEventCreateWithFlags(&ws->fork_ev, hipEventDisableTiming));
  HIP_TRY(hipEventCreateWithFlags(&ws->join_ev, hipEventDisableTiming));
  if (int rc = alloc_capacity(ws.get(), max_tokens, max_seqs)) return rc;
  *out = ws.release();
  return AE_OK;
}

void ae_workspace_destroy(ae_workspace* ws) { delete ws; }
void* ae_workspace_stream(ae_workspace* ws) { return ws ? reinterpret_cast<void*>(ws->stream) : nullptr; }

int ae_embed_batch_tokens(const ae_engine* e, ae_workspace* ws, const uint16_t* ids, const uint32_t* offsets, size_t n,
                          float* out) {
  if (e && !ws) {  // the engine's own workspace (created on first use), one call at a time
    std::lock_guard<std::mutex> lock(e->own_mu);
    if (!e->own_ws)
      if (int rc = ae_workspace_create(e, 0, 0, &e->own_ws)) return rc;
    return ae_embed_batch_tokens(e, e->own_ws, ids, offsets, n, out);
  }
  if (!e || !ws || ws->e != e) return fail(AE_ERR_INVALID_ARG, "engine/workspace mismatch");
  if (n == 0) return AE_OK;  // src/lib.rs:145-147
  if (!ids || !offsets || !out) return fail(AE_ERR_INVALID_ARG, "null argument");
  std::vector<const uint16_t*> seqs(n);
  std::vector<int> lens(n);
  for (size_t i = 0; i < n; i++) {
    if (offsets[i + 1] < offsets[i]) return fail(AE_ERR_INVALID_ARG, "offsets must be non-decreasing");
    const size_t len = offsets[i + 1] - offsets[i];
    if (len == 0) return fail(AE_ERR_INVALID_ARG, "input_ids must not be empty");  // src/model.rs:192
    seqs[i] = ids + offsets[i];
    lens[i] = int(std::min<size_t>(len, ae::kMaxPos));  // src/model.rs:191
    if (int rc = check_ids(seqs[i], size_t(lens[i]))) return rc;
  }
  HIP_TRY(hipSetDevice(e->device));
  return run_sequences(e, ws, seqs, lens, out);
}

int ae_embed_tokens(const ae_engine* e, ae_workspace* ws, const uint16_t* ids, size_t n, float* out384) {
  if (n == 0) return fail(AE_ERR_INVALID_ARG, "input_ids must not be empty");
  uint32_t off[2] = {0, uint32_t(n)};
  return ae_embed_batch_tokens(e, ws, ids, off, 1, out384);
}

static int embed_texts(const ae_engine* e, ae_workspace* ws, const char* const* texts, size_t n, bool is_query,
                       int num_threads, float* out) {
  if (!e) return fail(AE_ERR_INVALID_ARG, "null argument");
  if (!e->tokenizer) return fail(AE_ERR_INVALID_ARG, "engine opened without vocab.txt");
  if (n == 0) return AE_OK;
  std::vector<std::vector<uint16_t>> toks;
  e->tokenizer->encode_batch(texts, n, is_query, num_threads, toks);
  std::vector<uint16_t> flat;
  std::vector<uint32_t> offs(n + 1, 0);
  for (size_t i = 0; i < n; i++) {
    flat.insert(flat.end(), toks[i].begin(), toks[i].end());
    offs[i + 1] = uint32_t(flat.size());
  }
  return ae_embed_batch_tokens(e, ws, flat.data(), offs.data(), n, out);
}

int ae_embed_query(const ae_engine* e, ae_workspace* ws, const char* utf8, float* out384) {
  if (!utf8) return fail(AE_ERR_INVALID_ARG, "null text");
  return embed_texts(e, ws, &utf8, 1, true, 1, out384);
}

int ae_embed_document(const ae_engine* e, ae_workspace* ws, const char* utf8, float* out384) {
  if (!utf8) return fail(AE_ERR_INVALID_ARG, "null text");
  return embed_texts(e, ws, &utf8, 1, false, 1, out384);
}

int ae_embed_batch(const ae_engine* e, ae_workspace* ws, const char* const* texts, size_t n, int is_query,
                   int num_threads, float* out) {
  if (n && !texts) return fail(AE_ERR_INVALID_ARG, "null texts");
  return embed_texts(e, ws, texts, n, is_query != 0, num_threads, out);
}

// ParallelContext (src/parallel.rs:137-253): the reference's latency mode, which
// spreads the forward pass of one sequence over 1..8 host threads.  On the
// device the parallelism comes from the kernels themselves, so the context is a
// single-sequence workspace (512 tokens, its own stream, one captured hipGraph
// per sequence length) and the thread count is recorded only.  Results equal the
// workspace path bit for bit (the same kernels on the same batch of one).
struct ae_parallel_context {
  int n_threads = 1;
  ae_workspace* ws = nullptr;
  ~ae_parallel_context() { ae_workspace_destroy(ws); }
};

int ae_parallel_context_create(const ae_engine* e, int n_threads, ae_parallel_context** out) {
  if (!e || !out) return fail(AE_ERR_INVALID_ARG, "null argument");
  *out = nullptr;
  std::unique_ptr<ae_parallel_context> c(new ae_parallel_context());
  c->n_threads = std::min(std::max(n_threads, 1), 8);  // ParallelContext::new clamps to 1..8 (src/parallel.rs:146)
  if (int rc = ae_workspace_create(e, ae::kMaxPos, 1, &c->ws)) return rc;
  *out = c.release();
  return AE_OK;
}

void ae_parallel_context_destroy(ae_parallel_context* c) { delete c; }

int ae_parallel_context_threads(const ae_parallel_context* c) { return c ? c->n_threads : 0; }

int ae_embed_tokens_parallel(const ae_engine* e, ae_parallel_context* c, const uint16_t* ids, size_t n, float* out384) {
  if (!c) return fail(AE_ERR_INVALID_ARG, "null parallel context");
  return ae_embed_tokens(e, c->ws, ids, n, out384);
}

int ae_embed_query_parallel(const ae_engine* e, ae_parallel_context* c, const char* utf8, float* out384) {
  if (!c) return fail(AE_ERR_INVALID_ARG, "null parallel context");
  return ae_embed_query(e, c->ws, utf8, out384);
}

int ae_embed_document_parallel(const ae_engine* e, ae_parallel_context* c, const char* utf8, float* out384) {
  if (!c) return fail(AE_ERR_INVALID_ARG, "null parallel context");
  return ae_embed_document(e, c->ws, utf8, out384);
}

int ae_forward_packed_device(const ae_engine* e, ae_workspace* ws, const uint16_t* ids_dev, const int32_t* cu_seqlens_dev,
                             int n_seqs, int total_tokens, int max_seq_len, float* out_dev, void* stream) {
  if (!e || !ws || ws->e != e) return fail(AE_ERR_INVALID_ARG, "engine/workspace mismatch");
  if (n_seqs <= 0 || total_tokens < n_seqs || !ids_dev || !cu_seqlens_dev || !out_dev || max_seq_len < 0 ||
      max_seq_len > ae::kMaxPos)
    return fail(AE_ERR_INVALID_ARG, "bad packed batch");
  if (n_seqs > ws->max_seqs || total_tokens > ws->max_tokens)
    return fail(AE_ERR_CAPACITY, "packed batch exceeds workspace capacity");
  hipStream_t st = stream ? as_stream(stream) : ws->stream;
  return run_forward_replay(ws, ids_dev, cu_seqlens_dev, n_seqs, total_tokens,
                            max_seq_len ? max_seq_len : ae::kMaxPos, stated_longest(max_seq_len), out_dev, st);
}

float ae_cosine_similarity(const float* a, const float* b) {  // src/lib.rs:265-271
  float sum = 0.0f;
  for (int i = 0; i < ae::kHidden; i++) sum += a[i] * b[i];
  return sum;
}

int ae_linear_create(int n_out, int k_in, const int8_t* w_q, const float* w_scale, const float* bias,
                     const float* inv_smooth, ae_linear** out) {
  if (!out || !w_q || !w_scale || !bias || !inv_smooth) return fail(AE_ERR_INVALID_ARG, "null argument");
  *out = nullptr;
  int dev;
  if (int rc = check_device(&dev)) return rc;
  std::unique_ptr<ae_linear> l(new ae_linear());
  if (int rc = make_linear(n_out, k_in, w_q, w_scale, bias, inv_smooth, l.get())) return rc;
  *out = l.release();
  return AE_OK;
}

void ae_linear_destroy(ae_linear* l) { delete l; }

int ae_gemm_w8a8(const ae_linear* l, int m, const int8_t* a_dev, const float* a_scale_dev, const float* res_dev,
                 float* out_dev, void* stream) {
  if (!l || !a_dev || !a_scale_dev || !out_dev || m < 0) return fail(AE_ERR_INVALID_ARG, "bad gemm arguments");
  if (m == 0) return AE_OK;  // src/gemm.rs:639-641
  aek::GemmArgs p{};
  p.M = m;
  p.N = l->n;
  p.K = l->k;
  p.A = a_dev;
  p.a_scale = a_scale_dev;
  p.w = l->w;
  p.w_scale = l->w_scale;
  p.bias = l->bias;
  p.res = res_dev;
  p.out = out_dev;
  aek::launch_gemm(p, aek::kAI8, aek::kEpiF32, as_stream(stream));
  HIP_TRY(hipGetLastError());
  return AE_OK;
}

int ae_layernorm_smooth_quantize(int m, float* x_dev, const float* gamma_dev, const float* beta_dev,
                                 const float* inv_smooth_dev, int8_t* q_dev, float* scale_dev, void* stream) {
  if (m < 0 || !x_dev || !gamma_dev || !beta_dev || !inv_smooth_dev || !q_dev || !scale_dev)
    return fail(AE_ERR_INVALID_ARG, "bad layernorm arguments");
  if (m == 0) return AE_OK;
  aek::LnArgs p{};
  p.T = m;
  p.src = x_dev;
  p.dst = x_dev;
  p.gamma = gamma_dev;
  p.beta = beta_dev;
  p.smooth = inv_smooth_dev;
  p.q = q_dev;
  p.scale = scale_dev;
  aek::launch_ln_quant(p, aek::kLnSrcF32, as_stream(stream));
  HIP_TRY(hipGetLastError());
  return AE_OK;
}

int ae_smooth_quantize(int m, int n, const float* x_dev, const float* inv_smooth_dev, int8_t* q_dev, float* scale_dev,
                       void* stream) {
  if (m < 0 || n <= 0 || n % 64 || !x_dev || !inv_smooth_dev || !q_dev || !scale_dev)
    return fail(AE_ERR_INVALID_ARG, "bad smooth_quantize arguments");
  if (m == 0) return AE_OK;
  aek::launch_row_quant(m, n, const_cast<float*>(x_dev), inv_smooth_dev, q_dev, scale_dev, false, as_stream(stream));
  HIP_TRY(hipGetLastError());
  return AE_OK;
}

int ae_gelu_smooth_quantize(int m, int n, float* x_dev, const float* inv_smooth_dev, int8_t* q_dev, float* scale_dev,
                            void* stream) {
  if (m < 0 || n <= 0 || n % 64 || !x_dev || !inv_smooth_dev || !q_dev || !scale_dev)
    return fail(AE_ERR_INVALID_ARG, "bad gelu_smooth_quantize arguments");
  if (m == 0) return AE_OK;
  aek::launch_row_quant(m, n, x_dev, inv_smooth_dev, q_dev, scale_dev, true, as_stream(stream));
  HIP_TRY(hipGetLastError());
  return AE_OK;
}

static int attention_varlen(const float* qkv_dev, const int32_t* cu_seqlens_dev, int n_seqs, int total_tokens,
                            float* ctx_dev, void* stream, bool quantized);

int ae_attention_varlen(const float* qkv_dev, const int32_t* cu_seqlens_dev, int n_seqs, int total_tokens,
                        float* ctx_dev, void* stream) {
  return attention_varlen(qkv_dev, cu_seqlens_dev, n_seqs, total_tokens, ctx_dev, stream, false);
}

int ae_attention_varlen_quantized(const float* qkv_dev, const int32_t* cu_seqlens_dev, int n_seqs, int total_tokens,
                                  float* ctx_dev, void* stream) {
  return attention_varlen(qkv_dev, cu_seqlens_dev, n_seqs, total_tokens, ctx_dev, stream, true);
}

// Scratch of the synchronous operators ae_attention_varlen{,_quantized}: one
// grow-only device buffer per GPU, reused by every later call on that GPU (a
// call allocates only when it needs more than any call before it).  The calls
// synchronize before they return, and a mutex per GPU keeps concurrent callers
// from sharing the buffer while a call is in flight.
namespace {
constexpr int kOpScratchDevices = 64;
struct OpScratch {
  std::mutex mu;
  void* p = nullptr;
  size_t bytes = 0;
};
OpScratch g_op_scratch[kOpScratchDevices];
}  // namespace

static int attention_varlen(const float* qkv_dev, const int32_t* cu_seqlens_dev, int n_seqs, int total_tokens,
                            float* ctx_dev, void* stream, bool quantized) {
  if (!qkv_dev || !cu_seqlens_dev || !ctx_dev || n_seqs < 0 || total_tokens < 0)
    return fail(AE_ERR_INVALID_ARG, "bad attention arguments");
  if (n_seqs == 0) return AE_OK;
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= kOpScratchDevices) return fail(AE_ERR_HIP, "device ordinal beyond the operator scratch table");
  // the longest segment sizes the score rows and picks the kernel variant
  std::vector<int32_t> cu(size_t(n_seqs) + 1);
  HIP_TRY(hipMemcpyAsync(cu.data(), cu_seqlens_dev, cu.size() * sizeof(int32_t), hipMemcpyDeviceToHost,
                         as_stream(stream)));
  HIP_TRY(hipStreamSynchronize(as_stream(stream)));
  int max_len = 1;
  if (cu[0] < 0) return fail(AE_ERR_INVALID_ARG, "cu_seqlens is not a prefix sum of total_tokens");
  for (int b = 0; b < n_seqs; b++) {
    const long long L = (long long)cu[b + 1] - cu[b];
    if (L < 0 || cu[b + 1] > total_tokens) return fail(AE_ERR_INVALID_ARG, "cu_seqlens is not a prefix sum of total_tokens");
    max_len = std::max(max_len, int(L));
  }
  // The quantized path takes its V column scales over every row of the batch,
  // so a row outside the segments, or cut from one, would still change them:
  // it takes exact prefix sums of segments of at most 512 tokens.
  if (quantized && (cu[0] != 0 || cu[n_seqs] != total_tokens || max_len > ae::kMaxPos || n_seqs >= aek::kPlanMaxSegs))
    return fail(AE_ERR_INVALID_ARG, "quantized attention needs cu_seqlens[0] = 0, cu_seqlens[n_seqs] = total_tokens, "
                                    "segments of at most 512 tokens and fewer than 2^24 of them");
  const size_t T = size_t(total_tokens), vt = aek::sme_vt_len(total_tokens, n_seqs);
  const size_t plan_bytes = (aek::attention_plan_ints(n_seqs, total_tokens) * sizeof(int) + 255) & ~size_t(255);
  const size_t need = plan_bytes + (quantized ? T * 384 * 2 + T * 12 * 4 * 2 + 384 * 4 + 384 * vt + T * 4 : 0);
  OpScratch& sc = g_op_scratch[dev];
  std::lock_guard<std::mutex> lock(sc.mu);
  if (sc.bytes < need) {
    DevLock dlock(g_dev_mu);
    if (sc.p) {
      HIP_TRY(hipDeviceSynchronize());  // an earlier caller's stream may still read it
      (void)hipFree(sc.p);
      sc.p = nullptr;
      sc.bytes = 0;
    }
    const hipError_t e = hipMalloc(&sc.p, need);
    if (e != hipSuccess) return fail(AE_ERR_HIP, std::string("attention scratch: ") + hipGetErrorString(e));
    sc.bytes = need;
  }
  int* plan = static_cast<int*>(sc.p);
  aek::init_attention_kernels();
  aek::AttnArgs a{qkv_dev, cu_seqlens_dev, n_seqs, plan, ctx_dev, nullptr, nullptr,
                  aek::attention_pitch(std::min(max_len, ae::kMaxPos))};
  if (quantized) {  // int8 Q, K [T,384] each, their scales [T,12] each, the |V| column max [384],
                    // int8 V^T [384][vt], the tokens' segment indexes [T]
    char* b = static_cast<char*>(sc.p) + plan_bytes;
    aek::SmeArgs sa{reinterpret_cast<int8_t*>(b), reinterpret_cast<int8_t*>(b + T * 384),
                    reinterpret_cast<float*>(b + T * 768), reinterpret_cast<float*>(b + T * 768 + T * 48),
                    reinterpret_cast<uint32_t*>(b + T * 768 + T * 96),
                    reinterpret_cast<int8_t*>(b + T * 768 + T * 96 + 384 * 4),
                    reinterpret_cast<int*>(b + T * 768 + T * 96 + 384 * 4 + 384 * vt)};
    aek::init_attention_sme_kernels();
    aek::launch_attention_sme(a, sa, total_tokens, as_stream(stream));
  } else {
    a.longest = std::min(max_len, ae::kMaxPos);
    aek::launch_attention(a, total_tokens, as_stream(stream));
  }
  const hipError_t err = hipStreamSynchronize(as_stream(stream));
  if (err != hipSuccess) return fail(AE_ERR_HIP, std::string("attention: ") + hipGetErrorString(err));
  return AE_OK;
}

// ae_attention_varlen for callers that cannot allocate: the tile plan lives in
// a static device array (aek::noalloc_plan_scratch), the caller states
// max_seq_len, and nothing is allocated, copied to the host or synchronized.
int ae_attention_varlen_noalloc(const float* qkv_dev, const int32_t* cu_seqlens_dev, int n_seqs, int total_tokens,
                                int max_seq_len, float* ctx_dev, void* stream) {
  if (n_seqs < 0 || total_tokens < n_seqs || max_seq_len < 1 || max_seq_len > ae::kMaxPos)
    return fail(AE_ERR_INVALID_ARG, "bad attention arguments (max_seq_len must be 1..512)");
  if (n_seqs == 0) return AE_OK;
  // the plan's two lists, then the checked copy of cu_seqlens (n_seqs + 1 ints)
  const size_t plan_records = 2 * aek::attention_plan_list_records(n_seqs, total_tokens);
  const size_t records = plan_records + (size_t(n_seqs) + 1 + 3) / 4;
  if (records > (size_t)aek::kNoAllocPlanRecords)
    return fail(AE_ERR_CAPACITY, "ae_attention_varlen_noalloc: 2 (4 + 12 (total_tokens / 32 + n_seqs + 1)) + "
                                 "(n_seqs + 4) / 4 = " + std::to_string(records) +
                                     " records exceed its static scratch of " +
                                     std::to_string(aek::kNoAllocPlanRecords));
  if (!qkv_dev || !cu_seqlens_dev || !ctx_dev) return fail(AE_ERR_INVALID_ARG, "bad attention arguments");
  int* plan = nullptr;
  const hipError_t e = aek::noalloc_plan_scratch(&plan);
  if (e != hipSuccess) return fail(AE_ERR_HIP, std::string("no-allocation attention scratch: ") + hipGetErrorString(e));
  int* cs = plan + 4 * plan_records;
  hipStream_t st = as_stream(stream);
  // a cu_seqlens outside [0, total_tokens] or with a segment longer than
  // max_seq_len gives unspecified values, never an access outside the rows
  aek::launch_sanitize_segments(cu_seqlens_dev, n_seqs, total_tokens, max_seq_len, /*strict=*/false, nullptr, cs, st);
  aek::AttnArgs a{qkv_dev, cs, n_seqs, plan, ctx_dev, nullptr, nullptr, aek::attention_pitch(max_seq_len)};
  a.longest = stated_longest(max_seq_len);
  aek::launch_attention(a, total_tokens, st);
  HIP_TRY(hipGetLastError());
  return AE_OK;
}

// The same operators on the workspace's scratch: no allocation after the first
// quantized call, no host copy, no synchronization.  The caller bounds the
// segment lengths (max_seq_len, 1..512); a batch that breaks the bound, or whose
// cu_seqlens is not a prefix sum of total_tokens, is reported by the next
// ae_workspace_synchronize.
static int workspace_attention(ae_workspace* ws, const float* qkv_dev, const int32_t* cu_dev, int n_seqs,
                               int total_tokens, int max_seq_len, float* ctx_dev, void* stream, bool quantized) {
  if (!ws || !qkv_dev || !cu_dev || !ctx_dev || n_seqs < 0 || total_tokens < n_seqs || max_seq_len < 1 ||
      max_seq_len > ae::kMaxPos)
    return fail(AE_ERR_INVALID_ARG, "bad attention arguments");
  if (n_seqs == 0) return AE_OK;
  if (n_seqs > ws->max_seqs || total_tokens > ws->max_tokens)
    return fail(AE_ERR_CAPACITY, "attention batch exceeds workspace capacity");
  HIP_TRY(hipSetDevice(ws->e->device));
  if (quantized)
    if (int rc = alloc_sme_scratch(ws)) return rc;
  hipStream_t st = stream ? as_stream(stream) : ws->stream;
  aek::launch_sanitize_segments(cu_dev, n_seqs, total_tokens, max_seq_len, /*strict=*/true, ws->err, ws->cu_safe, st);
  aek::AttnArgs a{qkv_dev, ws->cu_safe, n_seqs, ws->attn_plan, ctx_dev, nullptr, nullptr,
                  aek::attention_pitch(max_seq_len)};
  a.longest = stated_longest(max_seq_len);
  if (quantized) aek::launch_attention_sme(a, ws->sme, total_tokens, st);  // per_seq = 0: the batch's V scales
  else aek::launch_attention(a, total_tokens, st);
  HIP_TRY(hipGetLastError());
  return AE_OK;
}

int ae_workspace_attention_varlen(ae_workspace* ws, const float* qkv_dev, const int32_t* cu_seqlens_dev, int n_seqs,
                                  int total_tokens, int max_seq_len, float* ctx_dev, void* stream) {
  return workspace_attention(ws, qkv_dev, cu_seqlens_dev, n_seqs, total_tokens, max_seq_len, ctx_dev, stream, false);
}

int ae_workspace_attention_varlen_quantized(ae_workspace* ws, const float* qkv_dev, const int32_t* cu_seqlens_dev,
                                            int n_seqs, int total_tokens, int max_seq_len, float* ctx_dev,
                                            void* stream) {
  return workspace_attention(ws, qkv_dev, cu_seqlens_dev, n_seqs, total_tokens, max_seq_len, ctx_dev, stream, true);
}

int ae_workspace_synchronize(ae_workspace* ws, void* stream) {
  if (!ws) return fail(AE_ERR_INVALID_ARG, "null workspace");
  HIP_TRY(hipSetDevice(ws->e->device));
  hipStream_t st = stream ? as_stream(stream) : ws->stream;
  HIP_TRY(hipStreamSynchronize(st));
  if (st != ws->stream) HIP_TRY(hipStreamSynchronize(ws->stream));
  int err = 0;
  HIP_TRY(hipMemcpyAsync(&err, ws->err, sizeof(int), hipMemcpyDeviceToHost, ws->stream));
  HIP_TRY(hipStreamSynchronize(ws->stream));
  if (err) {
    HIP_TRY(hipMemsetAsync(ws->err, 0, sizeof(int), ws->stream));
    HIP_TRY(hipStreamSynchronize(ws->stream));
    return fail(AE_ERR_INVALID_ARG, "a packed batch had a segment outside 1..max_seq_len tokens or cu_seqlens that "
                                    "is not a prefix sum of total_tokens");
  }
  return AE_OK;
}

struct ae_tokenizer {
  ae::Tokenizer tok;
};

int ae_tokenizer_open(const char* vocab_path, ae_tokenizer** out) {
  if (!vocab_path || !out) return fail(AE_ERR_INVALID_ARG, "null argument");
  *out = nullptr;
  std::unique_ptr<ae_tokenizer> t(new ae_tokenizer());
  std::string err;
  if (int rc = t->tok.load_vocab_file(vocab_path, err)) return fail(rc, err);
  *out = t.release();
  return AE_OK;
}

void ae_tokenizer_close(ae_tokenizer* t) { delete t; }

int ae_tokenizer_encode(const ae_tokenizer* t, const char* utf8, int is_query, uint16_t* ids, size_t cap,
                        size_t* n_out) {
  if (!t || !utf8 || !n_out) return fail(AE_ERR_INVALID_ARG, "null argument");
  std::vector<uint16_t> v;
  t->tok.encode(utf8, is_query != 0, v);
  *n_out = v.size();
  if (v.size() > cap || (!ids && !v.empty())) return fail(AE_ERR_CAPACITY, "id buffer too small");
  std::memcpy(ids, v.data(), v.size() * sizeof(uint16_t));
  return AE_OK;
}

size_t ae_tokenizer_vocab_size(const ae_tokenizer* t) { return t ? t->tok.vocab_size() : 0; }

int ae_write_synthetic_ae8(const char* path, uint64_t seed) {
  if (!path) return fail(AE_ERR_INVALID_ARG, "null path");
  std::string err;
  if (int rc = ae::write_synthetic_ae8(path, seed, err)) return fail(rc, err);
  return AE_OK;
}

int ae_workspace_set_attention_mode(ae_workspace* ws, int mode) {
  if (!ws) return fail(AE_ERR_INVALID_ARG, "null workspace");
  if (mode != AE_ATTENTION_EXACT && mode != AE_ATTENTION_QUANTIZED)
    return fail(AE_ERR_INVALID_ARG, "unknown attention mode");
  if (mode == AE_ATTENTION_QUANTIZED)
    if (int rc = alloc_sme_scratch(ws)) return rc;
  ws->attention_mode = mode;
  return AE_OK;
}

int ae_workspace_set_graphs(ae_workspace* ws, int enabled) {
  if (!ws) return fail(AE_ERR_INVALID_ARG, "null workspace");
  ws->graphs = enabled != 0;
  return AE_OK;
}

int ae_workspace_set_timing(ae_workspace* ws, int enabled) {
  if (!ws) return fail(AE_ERR_INVALID_ARG, "null workspace");
  HIP_TRY(hipStreamSynchronize(ws->stream));
  if (enabled && ws->ev_pool.empty()) {
    DevLock lock(g_dev_mu);
    ws->ev_pool.resize(4096);
    for (auto& ev : ws->ev_pool) HIP_TRY(hipEventCreate(&ev));
  }
  ws->ev_marks.clear();
  ws->ev_used = 0;
  for (int k = 0; k < AE_KERNEL_KINDS; k++) {
    ws->kind_ms[k] = 0.0;
    ws->kind_count[k] = 0;
  }
  ws->timing = enabled != 0;
  return AE_OK;
}

int ae_workspace_kernel_times(ae_workspace* ws, double* ms_out, int* counts) {
  if (!ws) return fail(AE_ERR_INVALID_ARG, "null workspace");
  drain_timing(ws);
  for (int k = 0; k < AE_KERNEL_KINDS; k++) {
    if (ms_out) ms_out[k] = ws->kind_ms[k];
    if (counts) counts[k] = ws->kind_count[k];
  }
  return AE_OK;
}

int ae_debug_gemm_quant_a(const ae_linear* l, int m, const float* x_dev, const uint32_t* rowmax_dev,
                          const float* smooth_dev, const float* res_dev, float* out_dev, void* stream) {
  if (!l || m <= 0 || !x_dev || !rowmax_dev || !out_dev) return fail(AE_ERR_INVALID_ARG, "bad arguments");
  aek::GemmArgs p{};
  p.M = m;
  p.N = l->n;
  p.K = l->k;
  p.A = x_dev;
  p.a_rowmax = rowmax_dev;
  p.a_smooth = smooth_dev;
  p.w = l->w;
  p.w_scale = l->w_scale;
  p.bias = l->bias;
  p.res = res_dev;
  p.out = out_dev;
  aek::launch_gemm(p, smooth_dev ? aek::kAF32QSmooth : aek::kAF32Q, aek::kEpiF32, as_stream(stream));
  HIP_TRY(hipGetLastError());
  return AE_OK;
}

int ae_debug_gemm_ln(const ae_linear* l, int m, const float* x_dev, const uint32_t* rowmax_dev,
                     const float* smooth_dev, const float* res_dev, const float* gamma_dev, const float* beta_dev,
                     const float* ln_smooth_dev, float* dst_dev, int8_t* q_dev, float* scale_dev, void* stream) {
  if (!l || m <= 0 || !x_dev || !rowmax_dev || !smooth_dev || !res_dev || !gamma_dev || !beta_dev || !ln_smooth_dev ||
      !dst_dev || !q_dev || !scale_dev)
    return fail(AE_ERR_INVALID_ARG, "bad arguments");
  if (l->n != 384 || l->k != 384) return fail(AE_ERR_INVALID_ARG, "ae_debug_gemm_ln: a 384 x 384 linear");
  aek::GemmArgs p{};
  p.M = m;
  p.N = l->n;
  p.K = l->k;
  p.A = x_dev;
  p.a_rowmax = rowmax_dev;
  p.a_smooth = smooth_dev;
  p.w = l->w;
  p.w_scale = l->w_scale;
  p.bias = l->bias;
  p.res = res_dev;
  aek::LnArgs ln{};
  ln.T = m;
  ln.gamma = gamma_dev;
  ln.beta = beta_dev;
  ln.smooth = ln_smooth_dev;
  ln.dst = dst_dev;
  ln.q = q_dev;
  ln.scale = scale_dev;
  aek::launch_gemm_ln(p, ln, as_stream(stream));
  HIP_TRY(hipGetLastError());
  return AE_OK;
}

int ae_debug_gemm_gelu(const ae_linear* l, int m, const int8_t* a_dev, const float* a_scale_dev,
                       const float* g_smooth_dev, float* out_dev, uint32_t* rowmax_dev, void* stream) {
  if (!l || m <= 0 || !a_dev || !a_scale_dev || !g_smooth_dev || !out_dev || !rowmax_dev)
    return fail(AE_ERR_INVALID_ARG, "bad arguments");
  aek::GemmArgs p{};
  p.M = m;
  p.N = l->n;
  p.K = l->k;
  p.A = a_dev;
  p.a_scale = a_scale_dev;
  p.w = l->w;
  p.w_scale = l->w_scale;
  p.bias = l->bias;
  p.out = out_dev;
  p.g_smooth = g_smooth_dev;
  p.g_rowmax = rowmax_dev;
  aek::launch_gemm(p, aek::kAI8, aek::kEpiGelu, as_stream(stream));
  HIP_TRY(hipGetLastError());
  return AE_OK;
}

int ae_debug_ffn(const ae_linear* up, const ae_linear* down, int m, const int8_t* a_dev, const float* a_scale_dev,
                 const float* res_dev, float* out_dev, void* stream) {
  if (!up || !down || m <= 0 || !a_dev || !a_scale_dev || !res_dev || !out_dev)
    return fail(AE_ERR_INVALID_ARG, "bad arguments");
  if (up->k != ae::kHidden || up->n != ae::kInter || down->k != ae::kInter || down->n != ae::kHidden)
    return fail(AE_ERR_INVALID_ARG, "ffn: expects a 384->1536 and a 1536->384 linear");
  aek::launch_ffn(ffn_args(*up, *down, m, a_dev, a_scale_dev, res_dev, out_dev), as_stream(stream));
  HIP_TRY(hipGetLastError());
  return AE_OK;
}

// test hook: the FFN with the LayerNorm + SmoothQuant of its rows in the same kernel (16-row workgroups)
int ae_debug_ffn_ln(const ae_linear* up, const ae_linear* down, int m, const int8_t* a_dev, const float* a_scale_dev,
                    const float* res_dev, float* out_dev, const float* gamma_dev, const float* beta_dev,
                    const float* ln_smooth_dev, float* dst_dev, int8_t* q_dev, float* scale_dev, void* stream) {
  if (!up || !down || m <= 0 || !a_dev || !a_scale_dev || !res_dev || !out_dev || !gamma_dev || !beta_dev ||
      !ln_smooth_dev || !dst_dev || !q_dev || !scale_dev)
    return fail(AE_ERR_INVALID_ARG, "bad arguments");
  if (up->k != ae::kHidden || up->n != ae::kInter || down->k != ae::kInter || down->n != ae::kHidden)
    return fail(AE_ERR_INVALID_ARG, "ffn: expects a 384->1536 and a 1536->384 linear");
  aek::LnArgs ln{};
  ln.T = m;
  ln.gamma = gamma_dev;
  ln.beta = beta_dev;
  ln.smooth = ln_smooth_dev;
  ln.dst = dst_dev;
  ln.q = q_dev;
  ln.scale = scale_dev;
  const bool fused = aek::launch_ffn(ffn_args(*up, *down, m, a_dev, a_scale_dev, res_dev, out_dev),
                                     as_stream(stream), nullptr, nullptr, nullptr, &ln);
  HIP_TRY(hipGetLastError());
  if (!fused) return fail(AE_ERR_INVALID_ARG, "ae_debug_ffn_ln: more rows than one round of 16-row workgroups");
  return AE_OK;
}

// test hook: embedding + the first `layers` encoder layers over one packed batch
// (in the given order); copies hidden [T,384], act_q [T,384], act_scale [T] back
int ae_debug_forward_prefix(const ae_engine* e, ae_workspace* ws, const uint16_t* ids, const uint32_t* offsets,
                            size_t n, int layers, float* hidden, int8_t* act_q, float* act_scale) {
  if (!e || !ws || n == 0 || layers < 0 || layers > ae::kLayers - 1) return fail(AE_ERR_INVALID_ARG, "bad args");
  const int T = int(offsets[n]);
  if (int(n) > ws->max_seqs || T > ws->max_tokens) return fail(AE_ERR_CAPACITY, "too large");
  int max_len = 0;
  HIP_TRY(hipStreamSynchronize(ws->stream));
  if (int rc = ws->st_cu.ensure((n + 1) * sizeof(int))) return rc;
  if (int rc = ws->st_ids.ensure(size_t(T) * sizeof(uint16_t))) return rc;
  int* h_cu = ws->st_cu.as<int>();
  uint16_t* h_ids = ws->st_ids.as<uint16_t>();
  for (size_t i = 0; i <= n; i++) h_cu[i] = int(offsets[i]);
  for (size_t i = 0; i < n; i++) {
    const int len = int(offsets[i + 1] - offsets[i]);
    if (len < 1 || len > ae::kMaxPos) return fail(AE_ERR_INVALID_ARG, "sequence lengths must be 1..512");
    max_len = std::max(max_len, len);
  }
  std::memcpy(h_ids, ids, size_t(T) * sizeof(uint16_t));
  HIP_TRY(hipMemcpyAsync(ws->ids, h_ids, size_t(T) * sizeof(uint16_t), hipMemcpyHostToDevice, ws->stream));
  HIP_TRY(hipMemcpyAsync(ws->cu, h_cu, (n + 1) * sizeof(int), hipMemcpyHostToDevice, ws->stream));
  if (int rc = run_forward(ws, ws->ids, ws->cu, int(n), T, max_len, max_len, nullptr, ws->stream, layers)) return rc;
  HIP_TRY(hipMemcpyAsync(hidden, ws->hidden, size_t(T) * 384 * 4, hipMemcpyDeviceToHost, ws->stream));
  HIP_TRY(hipMemcpyAsync(act_q, ws->act_q, size_t(T) * 384, hipMemcpyDeviceToHost, ws->stream));
  HIP_TRY(hipMemcpyAsync(act_scale, ws->act_scale, size_t(T) * 4, hipMemcpyDeviceToHost, ws->stream));
  HIP_TRY(hipStreamSynchronize(ws->stream));
  return AE_OK;
}

// test hook: exact GELU over n floats on the device (exhaustive parity checks)
int ae_debug_gelu_map(const float* x_dev, float* y_dev, size_t n, void* stream) {
  aek::launch_gelu_map(x_dev, y_dev, n, as_stream(stream));
  HIP_TRY(hipGetLastError());
  return AE_OK;
}

// test hook: the attention kernels' exact-product MFMA
int ae_debug_set_attention_form(int form) {
  if (form < 0 || form > 2) return fail(AE_ERR_INVALID_ARG, "attention form must be 0, 1 or 2");
  aek::set_attention_form(form);
  return AE_OK;
}

// test hook: the exact attention's kernels by the batch (no device access)
int ae_debug_attention_choice(int n_seqs, int total_tokens, int max_seq_len, int longest, int cus) {
  return aek::attention_choice(n_seqs, total_tokens, aek::attention_pitch(max_seq_len) - 4, longest, cus);
}

// test hook: the rule that keeps the 16-row workgroups of the int8 GEMM (no device access)
int ae_debug_gemm_int8_rows16(int m, int n, int k, int residual, int cus) {
  return aek::gemm_int8_rows16(m, n, k, residual != 0, cus) ? 1 : 0;
}

// test hook: the FFN kernel's workgroup height
int ae_debug_set_ffn_rows(int rows) {
  if (rows != 0 && rows != 16 && rows != 32 && rows != 64 && !(rows < 0 && rows % 64 == 0))
    return fail(AE_ERR_INVALID_ARG, "FFN rows must be 0, 16, 32, 64 or a negative multiple of 64");
  aek::set_ffn_rows(rows);
  return AE_OK;
}

// test hooks: the fused FFN's exact-GELU kernel for every launch; the fast kernel's repair counters
int ae_debug_set_ffn_exact_gelu(int exact) {
  aek::set_ffn_exact_gelu(exact != 0);
  return AE_OK;
}

int ae_debug_ffn_repairs(uint64_t* tiles, uint64_t* rows, int reset) {
  unsigned long long c[2] = {0, 0};
  HIP_TRY(aek::ffn_repair_counts(c, reset != 0));
  if (tiles) *tiles = c[0];
  if (rows) *rows = c[1];
  return AE_OK;
}

int ae_debug_gelu_fast_certify(uint64_t* out6) {
  if (!out6) return fail(AE_ERR_INVALID_ARG, "null output");
  DevLock lock(g_dev_mu);
  unsigned long long* d = nullptr;
  HIP_TRY(hipMalloc(reinterpret_cast<void**>(&d), 6 * sizeof(unsigned long long)));
  hipError_t e = aek::gelu_fast_certify(d, nullptr);
  if (e == hipSuccess) e = hipMemcpy(out6, d, 6 * sizeof(unsigned long long), hipMemcpyDeviceToHost);
  (void)hipFree(d);
  if (e != hipSuccess) return fail(AE_ERR_HIP, std::string("gelu certification: ") + hipGetErrorString(e));
  return AE_OK;
}

int ae_debug_mfma_products(const float* a_dev, const float* b_dev, float* out_dev, int n_sets, void* stream) {
  if (!a_dev || !b_dev || !out_dev || n_sets < 0) return fail(AE_ERR_INVALID_ARG, "bad mfma_products arguments");
  aek::launch_mfma_products(a_dev, b_dev, out_dev, n_sets, as_stream(stream));
  HIP_TRY(hipGetLastError());
  return AE_OK;
}

}  // extern "C"
