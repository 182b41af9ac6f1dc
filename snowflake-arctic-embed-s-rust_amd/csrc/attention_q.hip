// attention_q.hip -- the reference's quantized attention (its ArmSme backend,
// attention_multihead_sme with segment ranges: src/model.rs:607-621,
// src/simd_math.rs:1933-2192), on int8 MFMA:
//   Q, K: int8 per token and head (quantize_head32_row_neon, :2482-2526), K's
//         scale also carrying log2(e)/sqrt(32);
//   V:    int8 per head column over every token of the packed batch
//         (pack_qkv_head_int8_neon, :2564-2640; quantize_v_row_neon, :2530-2559);
//   s   = (f32(q.k) * k_scale) * q_scale   (log2 units);
//   p   = round(16383 * 2^(s - max)) per segment row: exp2_q_neon's cubic for
//         the row's 8-aligned part, glibc exp2f for its last len % 8 keys
//         (softmax_quantize_i16_from_acc_neon / softmax_exp2_quantize_pass_i16_neon,
//         :2291-2410), p_scale = 1 / max(sum p, 1);
//   ctx = f32(sum_t p_t * v_t) * (v_scale * p_scale).
// Every step is integer or one rounded f32 / f64 operation in the reference's
// order, so the result is bit-identical to the reference's path on the same qkv.
#include <hip/hip_runtime.h>

#include "device_common.hpp"
#include "kernels.hpp"

namespace aek {

namespace {
constexpr int kSmeQ = 32;  // queries per workgroup (the exact kernel's tile plan)
// P tile, as two int8 planes (p = 256 hi + lo, split_p4): row pitch round16(max length) +
// 8 bytes (s_pitch = round16 + 4), a multiple of 8 so that every 8-key group is
// one aligned 8-byte LDS read of each plane
__host__ __device__ inline int sme_p_pitch(int s_pitch) { return s_pitch + 4; }
inline size_t sme_p_bytes(int s_pitch) { return (size_t)kSmeQ * sme_p_pitch(s_pitch) * 2; }
typedef long v_i64;

// vcvtnq_s32_f32 on in-range values: round to nearest, ties to even
__device__ __forceinline__ int cvtn(float x) {
  const float r = __builtin_rintf(x);
  int q;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(q) : "v"(r));  // NaN -> 0
  return q;
}
__device__ __forceinline__ int sat8(int v) { return min(127, max(-128, v)); }
// f32::round (half away from zero), then `as i32` on an in-range value
__device__ __forceinline__ int cvtn_away(float x) {
  const float r = roundf(x);
  int q;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(q) : "v"(r));
  return q;
}
// vmaxq_f32 over non-NaN values
__device__ __forceinline__ float vmax(float a, float b) { return b > a ? b : a; }

// quantize_head32_row_neon over one 32-float row: int8 values into q (8-byte
// aligned), returns (max_abs / 127) * mul
__device__ __forceinline__ float quant_row32(const float* src, float mul, int8_t* q) {
  float4 v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) v[i] = reinterpret_cast<const float4*>(src)[i];
  float m = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; i++) m = vmax(vmax(vmax(vmax(m, fabsf(v[i].x)), fabsf(v[i].y)), fabsf(v[i].z)), fabsf(v[i].w));
  const float max_abs = m > 1e-8f ? m : 1e-8f;
  const float inv_s = 127.0f / max_abs;
  uint32_t w[8];
#pragma unroll
  for (int i = 0; i < 8; i++)
    w[i] = pack4(sat8(cvtn(v[i].x * inv_s)), sat8(cvtn(v[i].y * inv_s)), sat8(cvtn(v[i].z * inv_s)),
                 sat8(cvtn(v[i].w * inv_s)));
#pragma unroll
  for (int i = 0; i < 2; i++)
    reinterpret_cast<uint4*>(q)[i] = make_uint4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
  return (max_abs / 127.0f) * mul;
}

// exp2_q_neon (src/simd_math.rs:2353-2370) for one lane: round(scale * 2^x),
// x clamped at x_min; the coefficients are f32 products with the scale, as the
// reference forms them.  Returned as the f32 bits of kQBias + q: scaled lies in
// [0.24, 16382) (x <= 0 is a score minus its row maximum, f in [0, 1),
// n >= -16), so the f32 sum with 1.5 * 2^23 + 128 rounds it to the nearest
// integer, ties to even (the spacing there is 1 and the bias is even), which is
// the reference's vcvtnq_s32_f32, and its low 16 bits are q + 128.  A NaN x
// meets the clamp's fmaxf and gives q = 0, as a NaN through the reference's
// vmaxq_f32 and vcvtnq_s32_f32 does.
constexpr uint32_t kQBias = 0x4B400080u;  // bits of 1.5 * 2^23 + 128
__device__ __forceinline__ uint32_t exp2_q16_biased(float x) {
  constexpr float S = 16383.0f;
  x = fmaxf(x, -16.0f);
  const float fl = floorf(x);
  const int n = (int)fl;
  const float f = x - fl;
  float p = __builtin_fmaf(f, 0.07842169f * S, 0.22511937f * S);
  p = __builtin_fmaf(f, p, 0.6963853f * S);
  p = __builtin_fmaf(f, p, 0.999857f * S);
  const float scaled = __int_as_float(__float_as_int(p) + (int)((uint32_t)n << 23));
  return __float_as_uint(scaled + 12583040.0f);
}

// Four biased p values (kQBias + p, p < 2^14) as the two int8 MFMA operands of
// p = 256 hi + lo: hi = (p + 128) >> 8 in [0, 64] (byte 1 of the biased
// value) and lo = ((p + 128) & 255) - 128 (byte 0 with its top bit flipped),
// key r in byte r of each.
__device__ __forceinline__ void split_p4(const uint32_t (&b)[4], uint32_t& hi, uint32_t& lo) {
  const uint32_t t01 = __builtin_amdgcn_perm(b[1], b[0], 0x05010400u);  // b0.0 b1.0 b0.1 b1.1
  const uint32_t t23 = __builtin_amdgcn_perm(b[3], b[2], 0x05010400u);
  lo = __builtin_amdgcn_perm(t23, t01, 0x05040100u) ^ 0x80808080u;
  hi = __builtin_amdgcn_perm(t23, t01, 0x07060302u);
}
}  // namespace

// Q and K of every token and head to int8 with their scales, and the per-column
// |V| maximum folded into s.vmax (atomicMax on f32 bits; the buffer is preset to
// bits(1e-8f), the reference's starting value): one maximum per column over the
// whole batch, or (s.per_seq) one per sequence and column, vmax[b][c].
// 64 tokens per workgroup of 12 waves.
__global__ __launch_bounds__(768) void sme_pack_kernel(const float* qkv, const int* cu, int B, int T, SmeArgs s) {
  const int tid = threadIdx.x, t0 = blockIdx.x * 64;
  if (tid < 64 && t0 + tid < T) s.tseg[t0 + tid] = find_segment(cu, B, t0 + tid);  // for sme_vquant_kernel
  const float k_mul = kInvSqrtD * 1.44269504088896340736f;  // inv_sqrt_d * LOG2_E in f32
  for (int it = tid; it < 64 * 12; it += 768) {  // one (token, head) per thread
    const int t = t0 + it / 12, h = it % 12;
    if (t < T) {
      const float* row = qkv + (size_t)t * HQKV + h * 32;
      s.qs[t * 12 + h] = quant_row32(row, 1.0f, s.q8 + (size_t)t * H + h * 32);
      s.ks[t * 12 + h] = quant_row32(row + H, k_mul, s.k8 + (size_t)t * H + h * 32);
    }
  }
  __shared__ float s_m[12][H];
  // The block's tokens in runs that share one V scale group: the whole block,
  // or (per_seq) its run inside each segment.  Wave w: tokens a + w + 12i of a
  // run; lane: columns lane + 64k (row-contiguous loads).  Block-uniform loop.
  const int w = tid >> 6, lane = tid & 63, t1 = min(T, t0 + 64);
  int a = t0, g = s.per_seq ? find_segment(cu, B, t0) : 0;
  while (a < t1 && g < (s.per_seq ? B : 1)) {
    const int e = s.per_seq ? max(a, min(t1, cu[g + 1])) : t1;
    float m[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    for (int t = a + w; t < e; t += 12) {
      const float* vr = qkv + (size_t)t * HQKV + 2 * H + lane;
#pragma unroll
      for (int k = 0; k < 6; k++) m[k] = vmax(m[k], fabsf(vr[64 * k]));
    }
#pragma unroll
    for (int k = 0; k < 6; k++) s_m[w][lane + 64 * k] = m[k];
    __syncthreads();
    if (e > a) {
      for (int c = tid; c < H; c += 768) {
        float mm = s_m[0][c];
#pragma unroll
        for (int v = 1; v < 12; v++) mm = vmax(mm, s_m[v][c]);
        atomicMax(&s.vmax[(size_t)g * H + c], __float_as_uint(mm));
      }
    }
    __syncthreads();
    a = e;
    g++;
  }
}

// V to int8 with its group's per-column scales (quantize_v_row_neon: v *
// (127 / vmax), the scale group being the batch or, per_seq, the sequence),
// stored transposed: s.vt[c][round8(cu[b] + 7b) + (t - cu[b])] for token t of
// segment b.  Workgroup (64-token block, head): the block's V columns are staged
// in LDS so that both the f32 reads and the int8 writes are row-contiguous.
__global__ __launch_bounds__(256) void sme_vquant_kernel(const float* qkv, const int* cu, int B, int T, SmeArgs s,
                                                         size_t vt_len) {
  __shared__ float sv[64][33];
  __shared__ size_t s_pos[64];
  __shared__ int s_grp[64];
  const int tid = threadIdx.x, t0 = blockIdx.x * 64, h = blockIdx.y;
  // the tile's loads first, then the tokens' segments (from sme_pack_kernel)
  float v[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int i = tid + 256 * k, r = i >> 5, c = i & 31;
    v[k] = t0 + r < T ? qkv[(size_t)(t0 + r) * HQKV + 2 * H + h * 32 + c] : 0.0f;
  }
  if (tid < 64) {
    const int t = min(t0 + tid, T - 1), b = s.tseg[t], cb = cu[b];
    s_pos[tid] = (size_t)((cb + 7 * b + 7) & ~7) + (size_t)(t - cb);
    s_grp[tid] = s.per_seq ? b : 0;
  }
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const int i = tid + 256 * k;
    sv[i >> 5][i & 31] = v[k];
  }
  __syncthreads();
  for (int i = tid; i < 64 * 32; i += 256) {
    const int c = i >> 6, r = i & 63, t = t0 + r;
    if (t < T) {
      const float inv = 127.0f / __uint_as_float(s.vmax[(size_t)s_grp[r] * H + h * 32 + c]);
      s.vt[(size_t)(h * 32 + c) * vt_len + s_pos[r]] = (int8_t)sat8(cvtn(sv[r][c] * inv));
    }
  }
}

// One workgroup per (head, tile of 32 queries of one segment), the exact
// kernel's tile records and numbering (plan_item).  The only LDS tile is P as
// two int8 planes [32][pitch16] (33 KB at 512 keys): several workgroups per CU.
__global__ __launch_bounds__(256) void sme_attention_kernel(AttnArgs p, SmeArgs sa, size_t vt_len) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  __shared__ float s_maxw[4][kSmeQ];
  __shared__ float s_max[kSmeQ], s_pscale[kSmeQ], s_vscale[32];
  __shared__ int s_isum[kSmeQ];
  __shared__ uint64_t s_tab[32];
  int h, b;
  int4 rec;
  if (!plan_item(reinterpret_cast<const int4*>(p.plan), blockIdx.x >> 3, h, b, rec)) return;  // a surplus workgroup (list 0)
  const int nq = rec.w;
  const int s0 = rec.x, L = rec.y, q0 = rec.z;
  // per_seq: sequences under 16 tokens take the exact attention (forward_cls,
  // src/model.rs:244-259), launched separately
  if (nq == 0 || (sa.per_seq && L < 16)) return;
  const int pitch16 = sme_p_pitch(p.s_pitch);
  int8_t* Phi = reinterpret_cast<int8_t*>(smem);  // (p + 128) >> 8
  int8_t* Plo = Phi + kSmeQ * pitch16;            // ((p + 128) & 255) - 128
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  exp_tab_fill(s_tab, tid);  // ordered before the exp phase by the row-max barriers
  const ExpTabLds tb{s_tab};
  if (tid < 32) {
    const float vm = __uint_as_float(sa.vmax[(size_t)(sa.per_seq ? b : 0) * H + h * 32 + tid]);
    s_vscale[tid] = vm * (1.0f / 127.0f);
    s_isum[tid] = 0;
  }

  // phase 1: integer scores, A = K (16 keys x 32 dims), B = Q (32 dims x 16
  // queries), one v_mfma_i32_16x16x32_i8 per (key block, query half); lane l
  // supplies row l % 16 and dims 8(l/16)..+7 of both, and ends with keys
  // 16kb + 4(l/16) + r of the block for query l % 16 of the half: four
  // consecutive keys of one query row per lane.  Rows past the segment are
  // clamped (a clamped key repeats key L - 1's score, which cannot change the max).
  const int nqh = (nq + 15) >> 4, nkb = (L + 15) >> 4;
  v_i64 qa[2];
  float qsc[2];
#pragma unroll
  for (int qh = 0; qh < 2; qh++) {
    const int qrow = s0 + min(q0 + 16 * qh + lr, L - 1);
    qa[qh] = *reinterpret_cast<const v_i64*>(sa.q8 + (size_t)qrow * H + h * 32 + 8 * lg);
    qsc[qh] = sa.qs[qrow * 12 + h];
  }
  // all of this wave's K blocks (kb = wave + 4i, at most 8) are loaded up front;
  // lane l holds key 16kb + l % 16's operands and scale
  v_i64 kvs[8];
  float kss[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int key = min(16 * (wave + 4 * i) + lr, L - 1);
    if (wave + 4 * i < nkb) {
      kvs[i] = *reinterpret_cast<const v_i64*>(sa.k8 + (size_t)(s0 + key) * H + h * 32 + 8 * lg);
      kss[i] = sa.ks[(s0 + key) * 12 + h];
    }
  }
  // this lane's int8 V for phase 3, issued once Q and K have arrived and left
  // in flight through phases 1 and 2.  The explicit wait is what lets it stay in
  // flight: the memory counter drains in issue order, and past the joins of the
  // conditional loads above the compiler's count makes the first uses of the Q
  // and K scales wait for everything issued before them.  Keys 32k + 8(l/16) ..
  // +7 of column c = 16(w % 2) + l % 16, one aligned 8-byte load per 32-key
  // chunk k (keys past the segment meet p = 0)
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0)
  const int nch = (L + 31) >> 5;
  v_i64 vb[16];
  {
    const int8_t* vrow =
        sa.vt + (size_t)(h * 32 + 16 * (wave & 1) + lr) * vt_len + ((s0 + 7 * b + 7) & ~7) + 8 * lg;  // s0 = cu[b]
#pragma unroll
    for (int k = 0; k < 16; k++)
      vb[k] = k < nch ? *reinterpret_cast<const v_i64*>(vrow + 32 * k) : 0;  // zero past the row (phase 3's groups)
  }
  // the scale of this lane's key 16kb + 4(l/16) + r, from the lane that loaded it
  auto key_scales = [&](int i, float (&ksc)[4]) {
#pragma unroll
    for (int r = 0; r < 4; r++) ksc[r] = __shfl(kss[i], 4 * lg + r, 64);
  };
  // the row maxima of f32(acc) * k_scale; the q_scale product follows on the
  // maximum: q_scale > 0, so x -> RN(x * q_scale) is non-decreasing and the
  // maximum of the products is the product of the maximum.  fmaxf ignores a NaN
  // operand, as the reference's maximum over finite scores needs no NaN rule.
  float mrow[2] = {-INFINITY, -INFINITY};
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int kb = wave + 4 * i;
    if (kb >= nkb) break;  // wave-uniform
    float ksc[4];
    key_scales(i, ksc);
#pragma unroll
    for (int qh = 0; qh < 2; qh++) {
      if (qh >= nqh) break;  // wave-uniform
      const v4i acc = __builtin_amdgcn_mfma_i32_16x16x32_i8(kvs[i], qa[qh], v4i{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; r++) mrow[qh] = fmaxf(mrow[qh], (float)acc[r] * ksc[r]);
    }
  }
#pragma unroll
  for (int qh = 0; qh < 2; qh++) {
    float m = mrow[qh];  // -inf where a wave had no block
    m = fmaxf(m, __shfl_xor(m, 16, 64));
    m = fmaxf(m, __shfl_xor(m, 32, 64));
    if (lane < 16) s_maxw[wave][16 * qh + lr] = m * qsc[qh];
  }
  __syncthreads();
  if (tid < kSmeQ) s_max[tid] = fmaxf(fmaxf(s_maxw[0][tid], s_maxw[1][tid]), fmaxf(s_maxw[2][tid], s_maxw[3][tid]));
  __syncthreads();

  // phase 2: the same scores again (the int8 MFMAs are cheap; recomputing
  // them is bit-identical and keeps the tile small), p = round(16383 *
  // 2^(s - max)) < 2^14 into the P planes, a lane's four keys as one 4-byte
  // store to each: the cubic for keys below nv = L & ~7, glibc exp2f
  // (half-away rounding) for the last L - nv, 0 for the padding keys of the last
  // block.  Keys from nv on all lie in block nv / 16, the only block that
  // takes the masked form.  The p values are carried biased (kQBias + p); the
  // integer row sums are order-free and drop the bias at the end (mod 2^32).
  {
    const int nv = L & ~7;
    float mq[2];
#pragma unroll
    for (int qh = 0; qh < 2; qh++) mq[qh] = s_max[16 * qh + lr];
    uint32_t isum[2] = {0, 0};
    int nblk = 0;  // blocks of this wave (wave-uniform)
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int kb = wave + 4 * i;
      if (kb >= nkb) break;  // wave-uniform
      nblk++;
      const int key0 = 16 * kb + 4 * lg;
      const bool masked = kb == (nv >> 4);  // wave-uniform
      float ksc[4];
      key_scales(i, ksc);
#pragma unroll
      for (int qh = 0; qh < 2; qh++) {
        if (qh >= nqh) break;  // wave-uniform
        const v4i acc = __builtin_amdgcn_mfma_i32_16x16x32_i8(kvs[i], qa[qh], v4i{0, 0, 0, 0}, 0, 0, 0);
        uint32_t b[4];
        if (!masked) {
#pragma unroll
          for (int r = 0; r < 4; r++) b[r] = exp2_q16_biased(((float)acc[r] * ksc[r]) * qsc[qh] - mq[qh]);
        } else {
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const float x = ((float)acc[r] * ksc[r]) * qsc[qh] - mq[qh];
            b[r] = exp2_q16_biased(key0 + r < nv ? x : -16.0f);  // keys from nv on: p = 0 here
            if (nv < L) {  // wave-uniform
              const bool in = key0 + r >= nv && key0 + r < L;
              const float e = exp2f_libm(in ? x : 0.0f, tb);  // every lane evaluates (the table lookup)
              if (in) b[r] = kQBias + (uint32_t)min(16383, max(0, cvtn_away(e * 16383.0f)));
            }
          }
        }
        uint32_t hi, lo;
        split_p4(b, hi, lo);
        // key0 + 3 < round16(L) <= pitch16 - 8; the offset is a multiple of 4 keys
        const int off = (16 * qh + lr) * pitch16 + key0;
        *reinterpret_cast<uint32_t*>(Phi + off) = hi;
        *reinterpret_cast<uint32_t*>(Plo + off) = lo;
        isum[qh] += (b[0] + b[1]) + (b[2] + b[3]);
      }
    }
#pragma unroll
    for (int qh = 0; qh < 2; qh++) {
      uint32_t v = isum[qh] - (qh < nqh ? (uint32_t)(4 * nblk) * kQBias : 0u);  // sum of p over this lane's keys
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      if (lane < 16) atomicAdd(&s_isum[16 * qh + lr], (int)v);
    }
  }
  __syncthreads();
  if (tid < kSmeQ) s_pscale[tid] = 1.0f / (float)max(s_isum[tid], 1);
  __syncthreads();

  // phase 3: ctx = P @ V over chunks of 32 keys.  Wave w owns the 16 x 16
  // (query, dim) quadrant (w / 2, w % 2).  p < 2^14 is held as 256 p_hi + p_lo
  // (p_hi in [0, 64], p_lo in [-128, 127]) so the int8 MFMA takes it: the
  // planes' 8 bytes of a lane's keys are its A operands.  The integer sums are
  // exact (|256 acc_hi| <= 2^30), so ctx = f32(256 acc_hi + acc_lo) * (v_scale * p_scale).
  const int qh = wave >> 1, dh = wave & 1;
  if (qh < nqh) {
    const int c = 16 * dh + lr;
    const int8_t* hrow = Phi + (16 * qh + lr) * pitch16;
    const int8_t* lrow = Plo + (16 * qh + lr) * pitch16;
    v4i acc_hi = {0, 0, 0, 0}, acc_lo = {0, 0, 0, 0};
    // chunks in groups of 4 (a constant trip count: a break at nch would leave
    // the loop rolled), each group's 8 LDS reads before its MFMAs; the chunks of
    // a group past the row read clamped addresses and meet p = 0 and v = 0
    const int last8 = ((L + 7) & ~7) - 8;  // the last 8-key group phase 2 wrote
#pragma unroll
    for (int g = 0; g < 4; g++) {
      if (4 * g >= nch) continue;  // wave-uniform
      v_i64 ah[4], al[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int tb8 = 32 * (4 * g + j) + 8 * lg;  // this lane's 8 keys
        // groups from L on (not written when round16(L) <= tb8) take p = 0,
        // their reads clamped onto the last written group; keys from L to
        // round8(L) - 1 hold p = 0
        const int off = min(tb8, last8);
        const v_i64 h8 = *reinterpret_cast<const v_i64*>(hrow + off);
        const v_i64 l8 = *reinterpret_cast<const v_i64*>(lrow + off);
        ah[j] = tb8 < L ? h8 : 0;
        al[j] = tb8 < L ? l8 : 0;
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        acc_hi = __builtin_amdgcn_mfma_i32_16x16x32_i8(ah[j], vb[4 * g + j], acc_hi, 0, 0, 0);
        acc_lo = __builtin_amdgcn_mfma_i32_16x16x32_i8(al[j], vb[4 * g + j], acc_lo, 0, 0, 0);
      }
    }
    const int qb = 16 * qh + 4 * lg;
    const float vsc = s_vscale[c];
    const float sm = p.rowmax ? p.smooth[h * 32 + c] : 0.0f;
    float out[4], a[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      out[i] = (float)(acc_hi[i] * 256 + acc_lo[i]) * (vsc * s_pscale[qb + i]);
      a[i] = p.rowmax ? row16_max(nanless_max(0.0f, fabsf(out[i] * sm))) : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (qb + i < nq) p.ctx[(size_t)(s0 + q0 + qb + i) * H + h * 32 + c] = out[i];
    if (p.rowmax && lr == 0) {
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (qb + i < nq) atomicMax(&p.rowmax[s0 + q0 + qb + i], __float_as_uint(a[i]));
    }
  }
}

void launch_attention_sme(const AttnArgs& p, const SmeArgs& s, int T, hipStream_t st, bool plan) {
  if (T <= 0 || p.B <= 0) return;
  launch_fill_u32(s.vmax, H * (s.per_seq ? p.B : 1), 0x322bcc77u, st);  // bits of 1e-8f
  hipLaunchKernelGGL(sme_pack_kernel, dim3((T + 63) / 64), dim3(768), 0, st, p.qkv, p.cu, p.B, T, s);
  const size_t vt_len = sme_vt_len(T, p.B);
  hipLaunchKernelGGL(sme_vquant_kernel, dim3((T + 63) / 64, 12), dim3(256), 0, st, p.qkv, p.cu, p.B, T, s, vt_len);
  const int max_tiles = attention_max_tiles(p.B, T);
  if (plan) launch_attention_plan(p, st, 0, max_tiles);  // every tile in list 0
  hipLaunchKernelGGL(sme_attention_kernel, dim3(8 * attention_plan_cap(max_tiles)), dim3(256), sme_p_bytes(p.s_pitch),
                     st, p, s, vt_len);
}

void init_attention_sme_kernels() {
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(sme_attention_kernel),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)sme_p_bytes(attention_pitch(512)));
}

}  // namespace aek
