// attention.hip -- varlen multi-head attention (head_dim 32) and the layer-11
// [CLS]-only attention, both in the reference's exact scalar evaluation order.
#include <hip/hip_runtime.h>
#include <type_traits>

#include <mutex>

#include "device_common.hpp"
#include "kernels.hpp"

namespace aek {

// ---------------------------------------------------------------------------
// Varlen attention, head_dim 32, bit-exact with the reference's scalar path
// (src/model.rs:663-694 with compute_scores_head32 / softmax_inplace /
// weighted_sum_head32 scalar branches, src/simd_math.rs:1461-1821):
//   s_t  = (sum_{i=0..31, in order} q_i*k_t,i) * (1/sqrt(32))
//   e_t  = expf(s_t - max_t s_t)            (glibc expf: expf_libm, device_common.hpp)
//   sum  = sum_{t in order} e_t ; inv = 1/sum ; p_t = e_t * inv
//   ctx_d = sum_{t in order} p_t * v_t,d
// every sum left to right with separately rounded products.
//
// A workgroup (tile, head) owns kAttnQ queries of one sequence.  Scores for all
// keys of the sequence stay in LDS (row pitch = padded max length); the score,
// exp and PV phases use all 256 lanes, only the in-order softmax denominator is
// one lane per query.  The kernel also folds the SmoothQuant row absmax of its
// output (|ctx_j * inv_smooth_j|) into `rowmax` (atomicMax on non-negative f32
// bits), which the attn_out GEMM prologue consumes.
// ---------------------------------------------------------------------------
constexpr int kAttnQ = 32;     // queries per workgroup
// In batches of mostly shorter rows (launch_attention), the tiles of rows of at
// most kAttnLongL keys and those of longer rows go to two launches: score tiles
// of at most 32 x (kAttnLongL + 4) floats (51.7 KB, three workgroups per CU) in
// the first, up to 32 x 516 floats (66 KB, two per CU) in the second.  (At 416
// keys, 53.8 KB, C3 ran 6 % slower, as with two workgroups per CU.)
constexpr int kAttnLongL = 400;

// Work plan, built on the device from cu_seqlens (attention_plan_kernel).  An
// item is kAttnQ queries of one segment and one head; its 16-byte record is
// {s0, L, q0 | h << 16, nq | b << 8}: the segment's first token, its length, the
// first query, the head, the number of queries and the segment's index, so a
// workgroup learns its whole assignment from two scalar loads (plan_item).  The hardware deals a launch's
// workgroups to the 8 XCDs round-robin (workgroup p to XCD p % 8), so the plan
// gives each XCD a list of its own, which its workgroups x, x + 8, x + 16, ...
// take in order.  The items of one (segment, head), which share its K and V
// rows, are dealt together: they run on one XCD and hit in its L2.  Groups are
// dealt longest first (by tile count), one per XCD per round, in snake order
// (rounds alternate XCDs 0..7 and 7..0), so every XCD runs its longest tiles
// first and ends on short ones.  An XCD receives at most the average plus one
// group (16 items at 512 keys): each of its groups is at most its round's
// first, and the average is at least the sum of the full rounds' last groups,
// which telescopes (attention_plan_cap).
//
// A plan holds two lists of kPlanHdr + 12 max_tiles records: int2 x of records
// 0..3 is XCD x's (item count, first item), the items follow.  split = 0: every
// row in list 0; split = 1: rows of at most kAttnLongL keys in list 0, longer
// rows in list 1.  Rows are clamped to lmax keys (the score row length).  A list
// whose segments would need more than max_tiles tiles (cu_seqlens not a prefix
// sum of at most T tokens) gets no items.
constexpr int kPlanBuckets = 17;  // tiles per segment 0..16 (rows of at most 512 keys)

__global__ __launch_bounds__(256) void attention_plan_kernel(const int* cu, int B, int lmax, int max_tiles, int split,
                                                             int4* plan) {
  // cnt[l][n][t]: thread t's segments of list l with n tiles, then their
  // exclusive prefix over the threads (the ranks of thread t's first ones)
  __shared__ __attribute__((aligned(16))) int cnt[2][kPlanBuckets][256];
  // part[l][x][t]: items of XCD x in thread t's chunk of rounds, then the
  // exclusive prefix over the chunks
  __shared__ __attribute__((aligned(16))) int part[2][8][256];
  __shared__ int tot[2][kPlanBuckets], first[2][kPlanBuckets], xoff[2][8], bad[2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // exclusive prefix sum of a 256-int LDS row, by one whole wave (4 entries per
  // lane, then a shuffle scan over the lanes); *total gets the row's sum
  auto scan_row = [&](int* row, int* total) {
    const int4 v = reinterpret_cast<const int4*>(row)[lane];
    const int sum = v.x + v.y + v.z + v.w;
    int incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(incl, o, 64);
      if (lane >= o) incl += t;
    }
    const int ex = incl - sum;
    reinterpret_cast<int4*>(row)[lane] = make_int4(ex, ex + v.x, ex + v.x + v.y, ex + v.x + v.y + v.z);
    if (lane == 63) *total = incl;
  };
  const int per = (B + 255) / 256;
  const int b0 = min(B, tid * per), b1 = min(B, b0 + per);
  const int lcap = min(lmax, 16 * kAttnQ);
  auto seg_len = [&](int b) { return max(0, min(cu[b + 1] - cu[b], lcap)); };
  auto list_of = [&](int L) { return split && L > kAttnLongL ? 1 : 0; };
  for (int l = 0; l < 2; l++) {
    for (int n = 0; n < kPlanBuckets; n++) cnt[l][n][tid] = 0;
    for (int x = 0; x < 8; x++) part[l][x][tid] = 0;
  }
  for (int b = b0; b < b1; b++) {
    const int L = seg_len(b);
    cnt[list_of(L)][(L + kAttnQ - 1) / kAttnQ][tid]++;
  }
  __syncthreads();
  for (int r = wave; r < 2 * kPlanBuckets; r += 4)  // wave-uniform
    scan_row(cnt[r / kPlanBuckets][r % kPlanBuckets], &tot[r / kPlanBuckets][r % kPlanBuckets]);
  __syncthreads();
  if (tid < 2) {  // first rank of each tile count, longest first; first[l][0] = segments with tiles
    int acc = 0;
    for (int n = kPlanBuckets - 1; n >= 1; n--) {
      first[tid][n] = acc;
      acc += tot[tid][n];
    }
    first[tid][0] = acc;
  }
  __syncthreads();
  // tile count of the segment of rank r < first[l][0] in list l: 1 + the
  // number of buckets n >= 2 whose ranks end after r (ranks run longest first),
  // from the bucket ends held in registers
  int bend[2][kPlanBuckets - 2];
#pragma unroll
  for (int l = 0; l < 2; l++)
#pragma unroll
    for (int m = 0; m < kPlanBuckets - 2; m++) bend[l][m] = first[l][m + 2] + tot[l][m + 2];
  auto tiles_of_rank = [&](int l, int r) {
    int n = 1;
#pragma unroll
    for (int m = 0; m < kPlanBuckets - 2; m++) n += r < (l ? bend[1][m] : bend[0][m]) ? 1 : 0;
    return n;
  };
  int G[2], RC[2];  // groups (segment, head) and rounds per thread chunk
#pragma unroll
  for (int l = 0; l < 2; l++) {
    G[l] = 12 * first[l][0];
    RC[l] = (((G[l] + 7) >> 3) + 255) / 256;
    const int j1 = min((G[l] + 7) >> 3, (tid + 1) * RC[l]);
    for (int j = tid * RC[l]; j < j1; j++)
      for (int pos = 0; pos < 8; pos++) {
        const int k = 8 * j + pos;
        if (k < G[l]) part[l][(j & 1) ? 7 - pos : pos][tid] += tiles_of_rank(l, k / 12);
      }
  }
  __syncthreads();
  for (int r = wave; r < 16; r += 4) scan_row(part[r >> 3][r & 7], &xoff[r >> 3][r & 7]);  // XCD counts, then firsts
  __syncthreads();
  const size_t list_records = kPlanHdr + 12 * (size_t)max_tiles;
  if (tid < 2) {
    const int l = tid;
    int tiles = 0;
    for (int n = 1; n < kPlanBuckets; n++) tiles += n * tot[l][n];
    bool ok = tiles <= max_tiles;
    for (int x = 0; x < 8; x++) ok = ok && xoff[l][x] <= attention_plan_cap(max_tiles);
    bad[l] = ok ? 0 : 1;
    int2* hdr = reinterpret_cast<int2*>(plan + l * list_records);
    int acc = 0;
    for (int x = 0; x < 8; x++) {
      const int c = xoff[l][x];
      hdr[x] = make_int2(ok ? c : 0, acc);
      xoff[l][x] = acc;
      acc += c;
    }
  }
  __syncthreads();
  for (int b = b0; b < b1; b++) {
    const int s0 = cu[b], L = seg_len(b), l = list_of(L), n = (L + kAttnQ - 1) / kAttnQ;
    if (n == 0) continue;
    const int rank = first[l][n] + cnt[l][n][tid]++;
    if (bad[l]) continue;
    const int Gl = l ? G[1] : G[0], RCl = l ? RC[1] : RC[0];  // (static register indexes)
    int4* items = plan + l * list_records + kPlanHdr;
    for (int h = 0; h < 12; h++) {
      const int k = 12 * rank + h, j = k >> 3, pos = k & 7, x = (j & 1) ? 7 - pos : pos;
      const int c = j / RCl;  // the thread chunk that counted round j
      int off = xoff[l][x] + part[l][x][c];
      for (int jj = c * RCl; jj < j; jj++) {  // XCD x's groups in the chunk's earlier rounds
        const int kk = 8 * jj + ((jj & 1) ? 7 - x : x);
        if (kk < Gl) off += tiles_of_rank(l, kk / 12);
      }
      for (int t = 0; t < n; t++)
        items[off + t] = make_int4(s0, L, (t * kAttnQ) | (h << 16), min(kAttnQ, L - t * kAttnQ) | (int)((uint32_t)b << 8));
    }
  }
}

// MFMA as an exact multiplier.  v_mfma_f32_16x16x1_4b_f32 with a zero
// accumulator returns the correctly rounded f32 product a*b for each of its
// 4 x 16 x 16 outputs (K = 1: one product per output, rounded once), i.e. the
// same value as the VALU's v_mul_f32, up to the sign of an exact zero, which
// cannot change a sum that starts at +0.  The matrix core thus takes every
// multiply of QK^T and PV; the VALU keeps the separately rounded, in-order
// additions the reference's scalar loops perform.  Operand/result layout (lane l,
// result register r): A[m][blk] from lane blk*16 + m, B[n][blk] from lane
// blk*16 + n; result r holds block r/4, row m = 4*(l/16) + r%4, column n = l%16.
typedef float v16f __attribute__((ext_vector_type(16)));

// Element loads from this workgroup's rows of the packed qkv buffer through a
// buffer resource: the row offset (wave-uniform) is a scalar and the lane's
// column offset one VGPR shared by every load, so a load costs no vector
// address arithmetic.  Raw buffer, gfx9 descriptor word 3 (32-bit data format).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_rsrc(const float* base, int rows) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, rows * HQKV * 4, 0x00020000);
}
__device__ __forceinline__ float row_load(__amdgpu_buffer_rsrc_t r, uint32_t lane_bytes, uint32_t row) {
  return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, lane_bytes, row * (uint32_t)(HQKV * 4), 0));
}

__device__ __forceinline__ v16f mfma_products(float a, float b) {
  const v16f zero = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, zero, 0, 0, 0);
}

// acc[i] += blocks 0..3 of `pr` in block order (the blocks are consecutive
// terms of the reference's sums)
__device__ __forceinline__ void add_blocks(float (&acc)[4], const v16f& pr) {
#pragma unroll
  for (int blk = 0; blk < 4; blk++)
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = acc[i] + pr[4 * blk + i];
}

// The item of a workgroup of the latency form for a batch of at most kHalfMaxSegs
// segments, found from cu_seqlens by the workgroup itself where the plan kernel
// would cost a launch.  Returns false for a surplus workgroup.
//
// tps > 0 (16-query tiles of the longest segment; all workgroups are resident at
// once, so their order does not matter): workgroup (segment, tile, head), heads
// fastest, which spreads every batch evenly over the CUs (dealt by (segment, head)
// to XCDs instead, four XCDs get two of a row's 12 heads and the others one: 320
// keys 16.4 us, against 13.0).  The bounds are two scalar loads, or known (len1).
//
// tps = 0, the plan's dealing in short, for XCD x = blockIdx % 8 and its slot
// blockIdx / 8: segments longest first (lane b holds segment b), the 12 heads of
// the one of rank r to XCDs (12 r + h) % 8, so XCD x has two of its heads when
// (x < 4) == (r even) and one otherwise; a slot counts through its XCD's tiles in
// that order.
constexpr int kHalfMaxSegs = 16;
__device__ __forceinline__ bool half_item(const AttnArgs& p, int tps, int& h, int4& rec) {
  const int lmax = p.s_pitch - 4;
  if (tps > 0) {
    const int u = blockIdx.x / 12, b = u / tps, q0 = 16 * (u - b * tps);
    h = blockIdx.x - 12 * u;
    int s0 = 0, len = p.len1;
    if (p.len1 <= 0) {
      s0 = p.cu[b];
      len = p.cu[b + 1] - s0;
    }
    len = min(len, lmax);
    rec = make_int4(s0, len, q0, len - q0);
    return true;
  }
  const int x = blockIdx.x & 7, slot = blockIdx.x >> 3, lane = threadIdx.x & 63;
  const int s0 = p.cu[min(lane, p.B)], s1 = p.cu[min(lane + 1, p.B)];  // (lanes past the last segment: length 0)
  const int L = max(0, min(s1 - s0, lmax)), key = (L << 6) - lane;
  int rank = 0;
#pragma unroll
  for (int j = 0; j < kHalfMaxSegs; j++) rank += __builtin_amdgcn_readlane(key, j) > key ? 1 : 0;
  // lane r: the segment of rank r, its tiles on this XCD and their inclusive prefix over the ranks (one DPP row)
  const int seg = __builtin_amdgcn_ds_permute(4 * (lane < kHalfMaxSegs ? rank : lane), (L << 6) | lane);
  const int tiles = ((seg >> 6) + 15) >> 4;
  const bool two = (x < 4) == ((lane & 1) == 0);
  const int mine = two ? 2 * tiles : tiles;
  int incl = mine;
  incl += __builtin_amdgcn_update_dpp(0, incl, 0x111, 0xf, 0xf, true);  // row_shr:1, 2, 4, 8
  incl += __builtin_amdgcn_update_dpp(0, incl, 0x112, 0xf, 0xf, true);
  incl += __builtin_amdgcn_update_dpp(0, incl, 0x114, 0xf, 0xf, true);
  incl += __builtin_amdgcn_update_dpp(0, incl, 0x118, 0xf, 0xf, true);
  const uint64_t owner = __ballot(lane < kHalfMaxSegs && slot < incl);
  if (owner == 0) return false;
  const int r = __builtin_ctzll(owner);
  const int e = __builtin_amdgcn_readlane(seg, r), n = __builtin_amdgcn_readlane(tiles, r);
  const int len = e >> 6;
  int k = slot - __builtin_amdgcn_readlane(incl - mine, r);
  h = (x + 4 * (r & 1)) & 7;
  if (k >= n) {
    k -= n;
    h += 8;
  }
  rec = make_int4(__builtin_amdgcn_readlane(s0, e & 63), len, 16 * k, len - 16 * k);
  return true;
}

// dynamic LDS: S[kAttnQ][pitch] scores -> exps, per tile: pitch = round16(L) + 4
// (at most the launch's s_pitch, or kAttnLongL + 4 in the short-row launch)
// The tiles of one (sequence, head) share that head's K and V: the plan deals
// them to one XCD, where they hit in its L2.
// grid: 8 attention_plan_cap(max_tiles) workgroups (a bound); plan_item maps
// them to the plan's items (the surplus workgroups leave at once)
//
// kWide: operands in float4 groups with four MFMA results live at a time (one
// float4 load of K per 16 dims, one float4 LDS read of P per 16 keys, and four
// back-to-back MFMAs before their adds), 156 VGPRs.  Otherwise one MFMA result
// at a time with scalar operands, 92 VGPRs: for short rows, where the score
// tile leaves room for more waves than the wide variant's registers do.
//
// kHalf > 0 (wide only; the latency form): tiles of 16 queries with half the LDS,
// for batches whose 32-query tiles leave CUs idle (launch_attention), 116 VGPRs.
// kHalf = 1: each item of the plan is taken by two workgroups; kHalf = 2: the tiles
// come from half_item.
//
// kWaves = 8 for the smallest batches: the score and exp phases of a tile are
// split over twice the waves (the in-order sums of a tile occupy one wave, or two,
// either way).
template <bool kWide, int kHalf, int kWaves>
__global__ __launch_bounds__(64 * kWaves) void attention_kernel(AttnArgs p, int list_records, int list) {
  extern __shared__ __attribute__((aligned(16))) float smem[];
  __shared__ float s_maxw[kWaves][kAttnQ];
  __shared__ float s_max[kAttnQ], s_inv[kAttnQ];
  __shared__ uint64_t s_tab[32];
  int h;
  int4 rec;
  if constexpr (kHalf == 2) {
    if (!half_item(p, /*tps=*/list_records, h, rec)) return;  // surplus
  } else {
    // workgroups x, x + 8, .. run on XCD x: with kHalf every second one takes an item's other half
    const int slot = blockIdx.x >> 3, half = kHalf ? slot & 1 : 0;
    if (!plan_item(reinterpret_cast<const int4*>(p.plan) + (size_t)list * list_records, kHalf ? slot >> 1 : slot, h, rec))
      return;
    rec.z += 16 * half;
    rec.w -= 16 * half;
  }
  const int nq = kHalf ? min(rec.w, 16) : rec.w;
  if (nq <= 0) return;
  const int s0 = rec.x, L = rec.y, q0 = rec.z;  // L <= s_pitch - 4 (the plan clamps it)
  const int pitch = ((L + 15) & ~15) + 4;        // this tile's score row pitch
  const int nqh = kHalf ? 1 : (nq + 15) >> 4;  // query halves with at least one query
  float* S = smem;                 // [kAttnQ][pitch]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: per-wave loop bounds stay scalar
  const int lr = lane & 15, lg = lane >> 4;  // fragment row / block of this lane
  exp_tab_fill(s_tab, tid);  // ordered before phase 3 by the row-max barriers
  const ExpTabLds tb{s_tab};
  const float* qkv = p.qkv + (size_t)s0 * HQKV + h * 32;

  // Dims of the score products (MFMA j, block b): kWide: dim 16(j/4) + 4b + j%4,
  // so each lane's operands for MFMAs 4c..4c+3 are one float4 (dims 16c + 4lg ..
  // +3) and four consecutive MFMA results hold 16 consecutive dims; otherwise
  // dim 4j + b.  load_dims gives a lane its 8 operands of one row.
  constexpr int G = kWide ? 4 : 1;  // MFMA results live at a time
  auto load_dims = [&](const float* row, float (&f)[8]) {
    if constexpr (kWide) {
      const float4* src = reinterpret_cast<const float4*>(row + 4 * lg);
#pragma unroll
      for (int c = 0; c < 2; c++) {
        const float4 v = src[4 * c];
        f[4 * c] = v.x; f[4 * c + 1] = v.y; f[4 * c + 2] = v.z; f[4 * c + 3] = v.w;
      }
    } else {
#pragma unroll
      for (int j = 0; j < 8; j++) f[j] = row[4 * j + lg];
    }
  };
  // qf[qh] = the Q operands of query q0 + 16qh + lr (rows past the segment clamped)
  float qf[2][8];
#pragma unroll
  for (int qh = 0; qh < 2; qh++) load_dims(qkv + (size_t)min(q0 + 16 * qh + lr, L - 1) * HQKV, qf[qh]);

  // phase 1: scores (dot32_f32 scalar order) and the row max.  Wave w takes the
  // 16-key blocks kb = w, w + kWaves, ... with both query halves; A = K block, B = Q
  // half, so lane l ends with the scores of query 16qh + lr for keys
  // 16kb + 4lg + i.  K fragments come straight from global memory (L2), one
  // block ahead, into ping-pong registers (rows clamped to the segment).
  // The row max uses v_max_f32 (fmaxf): it ignores NaN like the reference's
  // `if s > max` scan, and the sign it gives an all-zero max cannot change
  // expf(s - max).
  float mrow[2] = {-INFINITY, -INFINITY};
  const int nkb = (L + 15) >> 4;
  auto load_kf = [&](int kb, float (&kf)[8]) { load_dims(qkv + H + (size_t)min(16 * kb + lr, L - 1) * HQKV, kf); };
  // The dot product starts from its first product instead of 0 + p_0: the two
  // differ only in the sign of a zero sum, and a score's zero sign cannot change
  // expf(s - max) (the row max is then a zero too, or s - max = -max).
  auto score_half = [&](int t, const float (&kf)[8], const float (&q)[8], float* srow, float& m) {
    float acc[4];
#pragma unroll
    for (int c = 0; c < 8 / G; c++) {
      v16f pr[G];
#pragma unroll
      for (int u = 0; u < G; u++) pr[u] = mfma_products(kf[G * c + u], q[G * c + u]);
#pragma unroll
      for (int blk = 0; blk < 4; blk++)  // dims 4Gc + G*blk + u, in order
#pragma unroll
        for (int u = 0; u < G; u++)
#pragma unroll
          for (int i = 0; i < 4; i++)
            acc[i] = (c == 0 && blk == 0 && u == 0) ? pr[0][i] : acc[i] + pr[u][4 * blk + i];
    }
    float4 sc;
    sc.x = acc[0] * kInvSqrtD;
    sc.y = acc[1] * kInvSqrtD;
    sc.z = acc[2] * kInvSqrtD;
    sc.w = acc[3] * kInvSqrtD;
    *reinterpret_cast<float4*>(srow + t) = sc;  // t + 3 < round16(L) = pitch - 4
    // a key t >= L was computed from K row L - 1 (clamped), so its score repeats
    // key L - 1's bit for bit and cannot change the max: no mask needed.  (The
    // narrow layout keeps the masked form: without it the compiler schedules its
    // loop into 145 VGPRs instead of 90.)
    if (kWide || t + 3 < L) {
      m = fmaxf(fmaxf(m, fmaxf(sc.x, sc.y)), fmaxf(sc.z, sc.w));
    } else {
      if (t < L) m = fmaxf(m, sc.x);
      if (t + 1 < L) m = fmaxf(m, sc.y);
      if (t + 2 < L) m = fmaxf(m, sc.z);
    }
  };
  float* srow0 = &S[lr * pitch];
  float* srow1 = &S[(16 + lr) * pitch];
  auto score_block = [&](int kb, const float (&kf)[8]) {
    const int t = 16 * kb + 4 * lg;
    score_half(t, kf, qf[0], srow0, mrow[0]);
    if (nqh > 1) score_half(t, kf, qf[1], srow1, mrow[1]);  // wave-uniform
  };
  {
    float ka[8], kb8[8];
    if (wave < nkb) load_kf(wave, ka);
    for (int kb = wave; kb < nkb; kb += 2 * kWaves) {  // wave-uniform
      load_kf(kb + kWaves, kb8);
      score_block(kb, ka);
      if (kb + kWaves >= nkb) break;
      load_kf(kb + 2 * kWaves, ka);
      score_block(kb + kWaves, kb8);
    }
  }
  // PV set-up (phase 6), and the V fragments of its first three key groups and
  // of the masked tail group, issued now: their latency hides behind the max,
  // exp and denominator phases instead of opening the PV loop.  Wave w owns the
  // 16 x 16 output quadrant (query half w/2, dim half w%2).  Group g's V rows are
  // clamped to the last full group (wave-uniform), so every load is unconditional.
  const int qh = wave >> 1, dh = wave & 1;
  const bool has_item = qh < nqh;
  const int vcol = 2 * H + 16 * dh + lr;
  // lane part of the V fragment offset (32-bit, from the segment's base)
  const uint32_t voff = (uint32_t)((kWide ? 4 * lg : lg) * HQKV + vcol);
  const int Lf = L & ~15, ng = Lf >> 4;
  const __amdgpu_buffer_rsrc_t vbuf = rows_rsrc(qkv, L);
  auto load_v = [&](int g, float (&v)[4]) {
    const uint32_t t0 = (uint32_t)(16 * min(g, ng - 1));
#pragma unroll
    for (int u = 0; u < 4; u++) v[u] = row_load(vbuf, 4 * voff, t0 + (kWide ? u : 4 * u));
  };
  // The last L - Lf (< 16) keys form one more group, masked in phase 6; tail_key(u)
  // is this lane's key of MFMA u there, its V row clamped per lane.
  const bool tail = L > Lf;  // wave-uniform
  auto tail_key = [&](int u) { return Lf + (kWide ? 4 * lg + u : 4 * u + lg); };
  float v0[4], v1[4], v2[4], vt[4];
  if (has_item) {
    if (ng > 0) {
      load_v(0, v0);
      load_v(1, v1);
      load_v(2, v2);
    }
    if (tail) {
#pragma unroll
      for (int u = 0; u < 4; u++)
        vt[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
            vbuf, (uint32_t)(min(tail_key(u), L - 1) * HQKV + vcol) * 4u, 0, 0));
    }
  }
#pragma unroll
  for (int qh = 0; qh < 2; qh++) {
    float m = mrow[qh];
    m = fmaxf(m, __shfl_xor(m, 16, 64));
    m = fmaxf(m, __shfl_xor(m, 32, 64));
    if (lane < 16) s_maxw[wave][16 * qh + lane] = m;
  }
  __syncthreads();
  if (tid < kAttnQ) {
    float m = s_maxw[0][tid];
#pragma unroll
    for (int w = 1; w < kWaves; w++) m = fmaxf(m, s_maxw[w][tid]);
    s_max[tid] = m;
  }
  __syncthreads();

  // phase 3: e_t = expf(s_t - max) over the nq x ceil(L/4) float4s of the tile,
  // spread over all lanes (entries past L are padding and never summed)
  {
    const int cols4 = (L + 3) >> 2;
    // q = u / cols4 as floor((u + 0.5) * (1/cols4)) in f32: exact for u < 2^13 and
    // cols4 <= 128 (the quotient stays >= 0.5/cols4 away from an integer, far
    // above the rounding error)
    const float rcols = 1.0f / (float)cols4;
    const int units = nq * cols4;
    // two float4 units per lane and step (eight independent exps in flight);
    // wave-uniform trip count (expf_libm needs all lanes).  kHalf: one unit in a
    // last step of at most one per lane.
    auto exps = [&](int u0, auto n) {
      float* e[n];
      float4 v[n];
      float m[n];
#pragma unroll
      for (int k = 0; k < n; k++) {
        const int u = min(u0 + 64 * kWaves * k + tid, units - 1);
        const int q = (int)(((float)u + 0.5f) * rcols);
        const int c4 = u - q * cols4;
        e[k] = &S[q * pitch + 4 * c4];
        v[k] = *reinterpret_cast<const float4*>(e[k]);
        m[k] = s_max[q];
      }
#pragma unroll
      for (int k = 0; k < n; k++) {
        v[k].x = expf_libm(v[k].x - m[k], tb);
        v[k].y = expf_libm(v[k].y - m[k], tb);
        v[k].z = expf_libm(v[k].z - m[k], tb);
        v[k].w = expf_libm(v[k].w - m[k], tb);
      }
#pragma unroll
      for (int k = 0; k < n; k++)
        if (u0 + 64 * kWaves * k + tid < units) *reinterpret_cast<float4*>(e[k]) = v[k];
    };
    int u0 = 0;
    for (; u0 + (kHalf ? 64 * kWaves : 0) < units; u0 += 128 * kWaves) exps(u0, std::integral_constant<int, 2>{});
    if (kHalf && u0 < units) exps(u0, std::integral_constant<int, 1>{});
  }
  __syncthreads();
  // phase 4: in-order denominator, one lane per query
  if (tid < kAttnQ) {
    float inv = 0.0f;
    if (tid < nq) {
      const float* e = &S[tid * pitch];
      float sum = 0.0f;
      // batches of 32 keys, each read while the previous one is added (reads past
      // the last full batch are clamped to it and not added)
      const int nb = L >> 5;
      auto ld = [&](int bi, float4 (&v)[8]) {
        const float4* src = reinterpret_cast<const float4*>(e + 32 * min(bi, nb - 1));
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = src[i];
      };
      auto add = [&](const float4 (&v)[8]) {
#pragma unroll
        for (int i = 0; i < 8; i++) {
          sum += v[i].x; sum += v[i].y; sum += v[i].z; sum += v[i].w;
        }
      };
      if (nb > 0) {
        float4 va[8], vb[8];
        ld(0, va);
        int bi = 0;
        for (; bi + 2 <= nb; bi += 2) {  // va holds batch bi
          ld(bi + 1, vb);
          add(va);
          ld(bi + 2, va);
          add(vb);
        }
        if (bi < nb) add(va);
      }
      int t = 32 * nb;
      for (; t + 4 <= L; t += 4) {
        const float4 v = *reinterpret_cast<const float4*>(e + t);
        sum += v.x; sum += v.y; sum += v.z; sum += v.w;
      }
      for (; t < L; t++) sum += e[t];
      inv = 1.0f / sum;
    }
    s_inv[tid] = inv;
  }

  // phase 6: ctx[q][d] = sum_t p_t * v_t,d in order, p_t = e_t * inv.  Wave w
  // owns the 16 x 16 quadrant (query half w/2, dim half w%2): A = P (query x
  // key), B = V (key x dim).  In a group of 16 keys from t0, MFMA u, block b
  // multiplies key t0 + 4b + u (kWide: each lane reads its four p operands as
  // one float4, keys t0 + 4lg .. +3, and the four results are added key by key)
  // or key t0 + 4u + b (one MFMA result at a time).
  // Lane l ends with queries 16qh + 4lg + i at dim 16dh + lr.  V fragments come
  // from global memory through a register ring.
  __syncthreads();  // publishes s_inv
  float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  if (has_item) {
    // the output's inv_smooth, loaded ahead of the PV loop
    const float sm = p.rowmax ? p.smooth[h * 32 + 16 * dh + lr] : 0.0f;
    const float* prow = &S[(16 * qh + lr) * pitch];
    const float inv = s_inv[16 * qh + lr];
    // full groups of 16 keys: no masking.  Group g's V goes to a 4-deep register
    // ring three groups ahead and its P one group ahead (groups 0-2 were loaded
    // before phase 3), so the main loop has no early exit.
    auto load_p = [&](int g) {
      const float* e = prow + 16 * min(g, ng - 1);
      if constexpr (kWide) {
        return *reinterpret_cast<const float4*>(e + 4 * lg);  // keys t0 + 4lg .. +3
      } else {
        return float4{e[lg], e[4 + lg], e[8 + lg], e[12 + lg]};  // keys t0 + 4u + lg
      }
    };
    // one group of 16 keys: p[u] and v[u] are the operands of MFMA u
    auto pv_add = [&](const float (&pu)[4], const float (&v)[4]) {
      if constexpr (kWide) {
        v16f pr[4];
#pragma unroll
        for (int u = 0; u < 4; u++) pr[u] = mfma_products(pu[u], v[u]);
#pragma unroll
        for (int blk = 0; blk < 4; blk++)
#pragma unroll
          for (int u = 0; u < 4; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) acc[i] = acc[i] + pr[u][4 * blk + i];
      } else {
#pragma unroll
        for (int u = 0; u < 4; u++) add_blocks(acc, mfma_products(pu[u], v[u]));
      }
    };
    auto pv_group = [&](const float4& e4, const float (&v)[4]) {
      const float pu[4] = {e4.x * inv, e4.y * inv, e4.z * inv, e4.w * inv};
      pv_add(pu, v);
    };
    // The tail group (keys Lf .. L - 1) is masked: keys past the segment get
    // p = v = +0, whose +0 products leave the sum unchanged (it starts at +0, so
    // it is never -0).
    if (!kWide) {
      // one group per step through the ring (fewer registers, for short rows)
      auto pv_narrow = [&](int g, const float (&v)[4]) {  // P read as the MFMAs go
#pragma unroll
        for (int u = 0; u < 4; u++) add_blocks(acc, mfma_products(prow[16 * g + 4 * u + lg] * inv, v[u]));
      };
      float v3[4];
      for (int g = 0; g < ng; g += 4) {
        load_v(g + 3, v3);
        pv_narrow(g, v0);
        if (g + 1 >= ng) break;
        load_v(g + 4, v0);
        pv_narrow(g + 1, v1);
        if (g + 2 >= ng) break;
        load_v(g + 5, v1);
        pv_narrow(g + 2, v2);
        if (g + 3 >= ng) break;
        load_v(g + 6, v2);
        pv_narrow(g + 3, v3);
      }
    } else if (ng > 0) {
      float v3[4];
      float4 pa, pb;
      pa = load_p(0);
      int g = 0;
      for (; g + 4 <= ng; g += 4) {
        load_v(g + 3, v3);
        pb = load_p(g + 1);
        pv_group(pa, v0);
        load_v(g + 4, v0);
        pa = load_p(g + 2);
        pv_group(pb, v1);
        load_v(g + 5, v1);
        pb = load_p(g + 3);
        pv_group(pa, v2);
        load_v(g + 6, v2);
        pa = load_p(g + 4);
        pv_group(pb, v3);
      }
      // the last ng - g < 4 groups: V already in v0, v1, v2, P of the first in pa
      if (g < ng) {
        pb = load_p(g + 1);
        pv_group(pa, v0);
      }
      if (g + 1 < ng) {
        pa = load_p(g + 2);
        pv_group(pb, v1);
      }
      if (g + 2 < ng) pv_group(pa, v2);
    }
    if (tail) {
      // keys up to Lf + 15 < round16(L) <= pitch - 4 stay inside the score row
      float pu[4], vu[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int t = tail_key(u);
        pu[u] = t < L ? prow[t] * inv : 0.0f;
        vu[u] = t < L ? vt[u] : 0.0f;
      }
      pv_add(pu, vu);
    }

    // Lane l holds queries qb .. qb + 3 at dim d.  With `rowmax`, each query's
    // max |ctx * inv_smooth| over this wave's 16 dims (one DPP row; every value
    // is a non-NaN >= +0, where fmaxf is the reference's `if a > max` scan) goes
    // to rowmax by atomicMax on its f32 bits.  The maxima are formed before any
    // store is issued (a wait for the inv_smooth load placed after the stores
    // would also wait for them), and the stores go out last with no wait between.
    const int qb = 16 * qh + 4 * lg, d = 16 * dh + lr;
    float a[4];
    if (p.rowmax) {
#pragma unroll
      for (int i = 0; i < 4; i++) a[i] = row16_max(nanless_max(0.0f, fabsf(acc[i] * sm)));
    }
    float* out = p.ctx + (size_t)(s0 + q0 + qb) * H + h * 32 + d;
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (qb + i < nq) out[(size_t)i * H] = acc[i];
    if (p.rowmax) {
      if (lr == 0) {
#pragma unroll
        for (int i = 0; i < 4; i++)
          if (qb + i < nq) atomicMax(&p.rowmax[s0 + q0 + qb + i], __float_as_uint(a[i]));
      }
    }
  }
}

// ---------------------------------------------------------------------------
// A few tokens (single sequences above all): one workgroup of 8 waves per
// (sequence, 8 queries, head), with the arithmetic of attention_kernel<true> in
// the same order, laid out for a short critical path rather than for throughput,
// and taken while its workgroups fit the compute units one to one
// (attention_choice).  kB = 1 or 2: sequences of at most 128 kB tokens.
//  * every global load (the Q operands, the K operands of the wave's key
//    blocks, the head's V rows into LDS) is issued at the start;
//  * scores: wave w takes the 16-key blocks w and w + 8: MFMA products and
//    in-order adds exactly as attention_kernel<true>'s phase 1;
//  * exp and the in-order denominator as there;
//  * p_t = e_t * inv in place (the reference's `s[i] * inv`), then PV on the
//    VALU, one output (query, dim) per thread: p_t * v_t,d rounded, added in
//    key order from LDS.
// ---------------------------------------------------------------------------
constexpr int kLatQ = 8;  // queries per workgroup (MFMA rows 8-15 repeat a query and are not used)

template <int kB>
__global__ __launch_bounds__(512) void attention_lat_kernel(AttnArgs p, int tiles_per_seq) {
  constexpr int kLatL = 128 * kB;  // keys: kB 16-key blocks per wave
  __shared__ float s_maxw[8][kLatQ];
  __shared__ float s_max[kLatQ], s_inv[kLatQ];
  __shared__ uint64_t s_tab[32];
  constexpr int pitch = kLatL + 4;
  __shared__ __attribute__((aligned(16))) float S[kLatQ * pitch];  // scores -> exps -> probabilities
  __shared__ __attribute__((aligned(16))) float sV[kLatL * 32];
  const int h = blockIdx.x % 12, bt = blockIdx.x / 12, b = bt / tiles_per_seq;
  const int q0 = (bt - b * tiles_per_seq) * kLatQ;
  // bounds that the host knows (p.len1 > 0): no cu_seqlens load
  const int s0 = p.len1 > 0 ? 0 : p.cu[b], L = min(p.len1 > 0 ? p.len1 : p.cu[b + 1] - s0, min(p.s_pitch - 4, kLatL));
  if (q0 >= L) return;  // workgroup-uniform
  const int nq = min(kLatQ, L - q0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  exp_tab_fill(s_tab, tid);  // ordered before the exp phase by the row-max barriers
  const ExpTabLds tb{s_tab};
  const float* qkv = p.qkv + (size_t)s0 * HQKV + h * 32;

  // operands of one row in the wide layout: f[4c + i] = dim 16c + 4lg + i
  auto load_dims = [&](const float* row, float (&f)[8]) {
    const float4* src = reinterpret_cast<const float4*>(row + 4 * lg);
#pragma unroll
    for (int c = 0; c < 2; c++) {
      const float4 v = src[4 * c];
      f[4 * c] = v.x; f[4 * c + 1] = v.y; f[4 * c + 2] = v.z; f[4 * c + 3] = v.w;
    }
  };
  // V rows (this head) first, then Q and K; V goes to LDS as soon as it has
  // arrived, which waits for V only (the memory counter drains in issue order),
  // so the V and Q/K latencies overlap.  Float4 f = tid + 512 i is key f / 8,
  // dims 4 (f % 8) .. +3.  Every load up to the stores is unconditional (lanes
  // past the segment load its last float4 and store it again; K blocks past it
  // load row L - 1 and are not used) and a scheduling barrier separates the
  // loads from the stores: otherwise the compiler sank each V load to its store
  // and waited for it there, one at a time (or, with a load under a per-lane
  // branch, kept the array in scratch memory).
  constexpr int kVF = 8 * kLatL / 512;  // float4s per thread
  typedef float f4 __attribute__((ext_vector_type(4)));
  f4 vr[kVF];
#pragma unroll
  for (int i = 0; i < kVF; i++) {
    const int f = min(tid + 512 * i, 8 * L - 1);
    vr[i] = *reinterpret_cast<const f4*>(qkv + (size_t)(f >> 3) * HQKV + 2 * H + (f & 7) * 4);
  }
  float qf[8];  // query q0 + lr (rows past the segment, and lr >= kLatQ, clamped)
  load_dims(qkv + (size_t)min(q0 + min(lr, kLatQ - 1), L - 1) * HQKV, qf);
  float kf[kB][8];
#pragma unroll
  for (int j = 0; j < kB; j++) load_dims(qkv + H + (size_t)min(16 * (wave + 8 * j) + lr, L - 1) * HQKV, kf[j]);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < kVF; i++)  // lanes past the segment rewrite its last float4
    *reinterpret_cast<f4*>(&sV[4 * min(tid + 512 * i, 8 * L - 1)]) = vr[i];

  // scores of query lr for keys 16kb + 4lg + i (dot32_f32 order) and the row max;
  // keys >= L repeat key L - 1 (clamped rows) and cannot change the max
  float m = -INFINITY;
#pragma unroll
  for (int j = 0; j < kB; j++) {
    const int kb = wave + 8 * j;
    if (16 * kb < L) {  // wave-uniform
      float acc[4];
#pragma unroll
      for (int c = 0; c < 2; c++) {
        v16f pr[4];
#pragma unroll
        for (int u = 0; u < 4; u++) pr[u] = mfma_products(kf[j][4 * c + u], qf[4 * c + u]);
#pragma unroll
        for (int blk = 0; blk < 4; blk++)  // dims 16c + 4blk + u, in order
#pragma unroll
          for (int u = 0; u < 4; u++)
#pragma unroll
            for (int i = 0; i < 4; i++)
              acc[i] = (c == 0 && blk == 0 && u == 0) ? pr[0][i] : acc[i] + pr[u][4 * blk + i];
      }
      float4 sc;
      sc.x = acc[0] * kInvSqrtD;
      sc.y = acc[1] * kInvSqrtD;
      sc.z = acc[2] * kInvSqrtD;
      sc.w = acc[3] * kInvSqrtD;
      if (lr < kLatQ) {
        *reinterpret_cast<float4*>(&S[lr * pitch + 16 * kb + 4 * lg]) = sc;
        m = fmaxf(fmaxf(m, fmaxf(sc.x, sc.y)), fmaxf(sc.z, sc.w));
      }
    }
  }
  m = fmaxf(m, __shfl_xor(m, 16, 64));
  m = fmaxf(m, __shfl_xor(m, 32, 64));
  if (lane < kLatQ) s_maxw[wave][lane] = m;
  __syncthreads();
  if (tid < kLatQ) {
    float mm = s_maxw[0][tid];
#pragma unroll
    for (int w = 1; w < 8; w++) mm = fmaxf(mm, s_maxw[w][tid]);
    s_max[tid] = mm;
  }
  __syncthreads();

  // e_t = expf(s_t - max) over the nq x ceil(L/4) float4s (as attention_kernel's phase 3)
  {
    const int cols4 = (L + 3) >> 2;
    const float rcols = 1.0f / (float)cols4;  // q = floor((u + 0.5) / cols4): exact for u < 2^13
    const int units = nq * cols4;
    static_assert(kLatQ * kLatL / 4 <= 512, "one float4 per thread");
    if (64 * wave < units) {  // wave-uniform (expf_libm needs all lanes)
      const int u = min(tid, units - 1);
      const int q = (int)(((float)u + 0.5f) * rcols);
      float* e = &S[q * pitch + 4 * (u - q * cols4)];
      float4 v = *reinterpret_cast<const float4*>(e);
      const float mq = s_max[q];
      v.x = expf_libm(v.x - mq, tb);
      v.y = expf_libm(v.y - mq, tb);
      v.z = expf_libm(v.z - mq, tb);
      v.w = expf_libm(v.w - mq, tb);
      if (tid < units) *reinterpret_cast<float4*>(e) = v;
    }
  }
  __syncthreads();
  if (tid < kLatQ) {  // in-order denominator, one lane per query
    float inv = 0.0f;
    if (tid < nq) {
      const float* e = &S[tid * pitch];
      float sum = 0.0f;
      // batches of 16 keys, each read while the previous one is added (reads past
      // the last full batch are clamped to it and not added)
      const int nb = L >> 4;
      float4 ea[4], eb[4];
      auto ld = [&](int bi, float4 (&v)[4]) {
        const float4* src = reinterpret_cast<const float4*>(e + 16 * min(bi, nb - 1));
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = src[i];
      };
      auto add = [&](const float4 (&v)[4]) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
          sum += v[i].x; sum += v[i].y; sum += v[i].z; sum += v[i].w;
        }
      };
      if (nb > 0) {
        ld(0, ea);
        int bi = 0;
        for (; bi + 2 <= nb; bi += 2) {
          ld(bi + 1, eb);
          __builtin_amdgcn_sched_barrier(0);
          add(ea);
          __builtin_amdgcn_sched_barrier(0);
          ld(bi + 2, ea);
          __builtin_amdgcn_sched_barrier(0);
          add(eb);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (bi < nb) add(ea);
      }
      for (int t = 16 * nb; t < L; t++) sum += e[t];
      inv = 1.0f / sum;
    }
    s_inv[tid] = inv;
  }
  __syncthreads();
  // p_t = e_t * inv in place (the reference's normalization), one float4 per thread
  {
    const int cols4 = (L + 3) >> 2;
    const float rcols = 1.0f / (float)cols4;
    const int units = nq * cols4;
    if (tid < units) {
      const int q = (int)(((float)tid + 0.5f) * rcols);
      float4* e = reinterpret_cast<float4*>(&S[q * pitch + 4 * (tid - q * cols4)]);
      const float inv = s_inv[q];
      float4 v = *e;
      v.x = v.x * inv; v.y = v.y * inv; v.z = v.z * inv; v.w = v.w * inv;
      *e = v;
    }
  }
  __syncthreads();

  // PV: thread (q, d) = (tid / 32, tid % 32), p_t * v_t,d added in key order
  const int q = tid >> 5, d = tid & 31;
  float o = 0.0f;
  if (q < nq) {  // uniform per half-wave
    const float* pr = &S[q * pitch];
    // batches of 8 keys: the next batch's LDS reads go out before this batch's
    // chain of adds (reads past the last full batch are clamped to it, not used)
    const int nb = L >> 3;
    float4 pa[2], pb[2];
    float va[8], vb[8];
    auto ld = [&](int bi, float4 (&pp)[2], float (&v)[8]) {
      const int t0 = 8 * min(bi, nb - 1);
      pp[0] = *reinterpret_cast<const float4*>(pr + t0);
      pp[1] = *reinterpret_cast<const float4*>(pr + t0 + 4);
#pragma unroll
      for (int k = 0; k < 8; k++) v[k] = sV[32 * (t0 + k) + d];
    };
    auto add = [&](const float4 (&pp)[2], const float (&v)[8]) {
      o = o + pp[0].x * v[0];
      o = o + pp[0].y * v[1];
      o = o + pp[0].z * v[2];
      o = o + pp[0].w * v[3];
      o = o + pp[1].x * v[4];
      o = o + pp[1].y * v[5];
      o = o + pp[1].z * v[6];
      o = o + pp[1].w * v[7];
    };
    if (nb > 0) {
      ld(0, pa, va);
      int bi = 0;
      for (; bi + 2 <= nb; bi += 2) {
        ld(bi + 1, pb, vb);
        __builtin_amdgcn_sched_barrier(0);
        add(pa, va);
        __builtin_amdgcn_sched_barrier(0);
        ld(bi + 2, pa, va);
        __builtin_amdgcn_sched_barrier(0);
        add(pb, vb);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (bi < nb) add(pa, va);
    }
    for (int t = 8 * nb; t < L; t++) o = o + pr[t] * sV[32 * t + d];
    p.ctx[(size_t)(s0 + q0 + q) * H + h * 32 + d] = o;
  }
  if (p.rowmax) {
    // max |ctx * inv_smooth| over the head's 32 dims (one half-wave; every value
    // is a non-NaN >= +0 where fmaxf is the reference's scan), by atomicMax on
    // the f32 bits
    float a = q < nq ? nanless_max(0.0f, fabsf(o * p.smooth[h * 32 + d])) : 0.0f;
    a = lanes32_max(a);
    if (d == 0 && q < nq) atomicMax(&p.rowmax[s0 + q0 + q], __float_as_uint(a));
  }
}

// Short rows (every sequence of the batch at most 16 * NKB <= 64 keys): one
// workgroup per (sequence, head), one wave per 16 queries, the whole score row
// in registers (NKB blocks of 16 keys, 4 scores per lane and block).  Same
// arithmetic, in the same order, as attention_kernel:
//  * scores: A = K block with its rows permuted so that lane (lg, lr) ends with
//    query lr and keys 16kb + lg + 4i in result register i, B = Q (dims 4j + b);
//  * the in-order denominator: each lane gathers the 16 exps of its query and
//    block (key 16kb + lg' + 4i from lane lr + 16lg', register i) and adds them
//    in key order (padding keys hold exact +0);
//  * PV: MFMA i of block kb multiplies keys 16kb + 4i + j (block j), so register
//    i is directly its A operand; lane (lg, lr) ends with queries 4lg + r at
//    dims lr and 16 + lr.
// The workgroup first stages the segment's K and V rows of the head in LDS
// with float4 loads (one 128-byte row section per 8 lanes), and the MFMA
// operands are then read from there: the operands' own layout (4 bytes per
// lane from 16 rows) read from global memory by every wave kept the address
// unit busy 90 % of the time.  (Each wave still loads its own Q operands, once:
// without a Q tile the LDS admits 8 workgroups per CU, as the 64 registers do.)
// Batches of short sequences spend most of a tiled workgroup on set-up and
// partial tiles; this form keeps 8 waves per SIMD busy instead.
template <int NKB>
__global__ __launch_bounds__(256, 8) void attention_rows_kernel(AttnArgs p) {
  constexpr int kRows = 16 * NKB, kP = 33;  // staged rows; row pitch in floats (conflict-free reads)
  __shared__ float sK[kRows * kP], sV[kRows * kP];
  const int item = xcd_contiguous(blockIdx.x, p.B * 12);
  const int b = item / 12, h = item - b * 12;
  const int s0 = p.cu[b];
  if (p.skip_from > 0 && p.cu[b + 1] - s0 >= p.skip_from) return;  // another kernel's segment (uniform)
  const int L = min(p.cu[b + 1] - s0, kRows);
  // this lane's Q operands (query q0 + lr, rows past the segment clamped):
  // loaded before the K/V staging below where NKB > 1, so that their latency
  // overlaps it (at NKB = 1 that placement spilled)
  float qf[8];
  auto load_q = [&]() {
    const int l = threadIdx.x & 63, qq = (threadIdx.x >> 6) * 16 + (l & 15);
    const float* qrow = p.qkv + (size_t)(s0 + min(qq, L - 1)) * HQKV + h * 32 + (l >> 4);
#pragma unroll
    for (int j = 0; j < 8; j++) qf[j] = qrow[4 * j];
  };
  if constexpr (NKB > 1) load_q();
  // this thread's NKB float4s of rows [0, L) of the head's K and V sections
  // (16 float4s per row; float4 c = tid + 256 i, its row clamped to the segment
  // and stored only when c < 16 L), every load issued before the first store
  // (a loop with a load and its store per trip waited for each load in turn).
  // NKB = 1 keeps that loop (one trip): the other form spilled there.
  typedef float f4 __attribute__((ext_vector_type(4)));
  if constexpr (NKB == 1) {
    const float* src = p.qkv + (size_t)s0 * HQKV + H + h * 32;
    for (int c = threadIdx.x; c < 16 * L; c += blockDim.x) {
      const int r = c >> 4, sec = (c >> 3) & 1, f = 4 * (c & 7);
      const float4 v = *reinterpret_cast<const float4*>(src + (size_t)r * HQKV + sec * H + f);
      float* dst = (sec == 0 ? sK : sV) + r * kP + f;
      dst[0] = v.x; dst[1] = v.y; dst[2] = v.z; dst[3] = v.w;
    }
  } else {
    const float* src = p.qkv + (size_t)s0 * HQKV + H + h * 32;
    f4 kv[NKB];
#pragma unroll
    for (int i = 0; i < NKB; i++) {
      const int c = threadIdx.x + 256 * i, r = min(c >> 4, L - 1), sec = (c >> 3) & 1, f = 4 * (c & 7);
      kv[i] = *reinterpret_cast<const f4*>(src + (size_t)r * HQKV + sec * H + f);
    }
#pragma unroll
    for (int i = 0; i < NKB; i++) {
      const int c = threadIdx.x + 256 * i, r = c >> 4, sec = (c >> 3) & 1, f = 4 * (c & 7);
      if (c < 16 * L) {
        float* dst = (sec == 0 ? sK : sV) + r * kP + f;
        dst[0] = kv[i].x; dst[1] = kv[i].y; dst[2] = kv[i].z; dst[3] = kv[i].w;
      }
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, q0 = (threadIdx.x >> 6) * 16;
  if (q0 >= L) return;  // wave-uniform; nothing below synchronizes across waves
  const int lr = lane & 15, lg = lane >> 4;
  // the exp table in registers (ExpTab): at 8 waves per SIMD this kernel is
  // VALU-bound, and the LDS table's index arithmetic measured 0.35 % slower
  const ExpTab tb = exp_tab_regs();
  const int nkb = (L + 15) >> 4;

  if constexpr (NKB == 1) load_q();
  const int kperm = 4 * (lr & 3) + (lr >> 2);  // key of A row lr within a block
  auto load_kf = [&](int kb, float (&kf)[8]) {
    const float* src = sK + min(16 * kb + kperm, L - 1) * kP + lg;
#pragma unroll
    for (int j = 0; j < 8; j++) kf[j] = src[4 * j];
  };
  float s[NKB][4];
  float mx = -INFINITY;
  {
    float kf[2][8];
    load_kf(0, kf[0]);
#pragma unroll
    for (int kb = 0; kb < NKB; kb++) {
      if (kb < nkb) {  // wave-uniform
        if (kb + 1 < nkb) load_kf(kb + 1, kf[(kb + 1) & 1]);
        float acc[4];
#pragma unroll
        for (int j = 0; j < 8; j++) {
          const v16f pr = mfma_products(kf[kb & 1][j], qf[j]);
#pragma unroll
          for (int blk = 0; blk < 4; blk++)
#pragma unroll
            for (int i = 0; i < 4; i++)  // starts from the first product (a zero sum's sign cannot matter)
              acc[i] = (j == 0 && blk == 0) ? pr[i] : acc[i] + pr[4 * blk + i];
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
          s[kb][i] = acc[i] * kInvSqrtD;
          if (16 * kb + lg + 4 * i < L) mx = fmaxf(mx, s[kb][i]);
        }
      }
    }
  }
  mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
  mx = fmaxf(mx, __shfl_xor(mx, 32, 64));

  float sum = 0.0f;
#pragma unroll
  for (int kb = 0; kb < NKB; kb++) {
    if (kb < nkb) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float e = expf_libm(s[kb][i] - mx, tb);
        s[kb][i] = (16 * kb + lg + 4 * i < L) ? e : 0.0f;
      }
      float v[16];
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int g = 0; g < 4; g++) v[g + 4 * i] = __shfl(s[kb][i], lr + 16 * g, 64);
#pragma unroll
      for (int t = 0; t < 16; t++) sum += v[t];
    }
  }
  const float inv = 1.0f / sum;

  float acc[2][4] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
  auto load_vf = [&](int kb, float (&vf)[2][4]) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float* src = sV + min(16 * kb + 4 * i + lg, L - 1) * kP + lr;
      vf[0][i] = src[0];
      vf[1][i] = src[16];
    }
  };
  {
    float vf[2][2][4];
    load_vf(0, vf[0]);
#pragma unroll
    for (int kb = 0; kb < NKB; kb++) {
      if (kb < nkb) {
        if (kb + 1 < nkb) load_vf(kb + 1, vf[(kb + 1) & 1]);
        if (kb + 1 == nkb) {  // keys past the segment: exact zeros
#pragma unroll
          for (int i = 0; i < 4; i++)
            if (16 * kb + 4 * i + lg >= L) vf[kb & 1][0][i] = vf[kb & 1][1][i] = 0.0f;
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
          const float pi = s[kb][i] * inv;
          add_blocks(acc[0], mfma_products(pi, vf[kb & 1][0][i]));
          add_blocks(acc[1], mfma_products(pi, vf[kb & 1][1][i]));
        }
      }
    }
  }
  const float sm0 = p.rowmax ? p.smooth[h * 32 + lr] : 0.0f;
  const float sm1 = p.rowmax ? p.smooth[h * 32 + 16 + lr] : 0.0f;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int q = q0 + 4 * lg + r;
    if (q < L) {
      float* o = p.ctx + (size_t)(s0 + q) * H + h * 32 + lr;
      o[0] = acc[0][r];
      o[16] = acc[1][r];
    }
    if (p.rowmax) {
      float a = nanless_max(0.0f, fabsf(acc[0][r] * sm0));
      a = nanless_max(a, fabsf(acc[1][r] * sm1));
#pragma unroll
      for (int off = 1; off < 16; off <<= 1) a = nanless_max(a, __shfl_xor(a, off, 64));
      if (q < L && lr == 0) atomicMax(&p.rowmax[s0 + q], __float_as_uint(a));
    }
  }
}

// test hook: for each set of 64 operand pairs, the 16 results per lane of
// mfma_products (out[set][lane][r]), the multiplier attention_kernel relies on
__global__ __launch_bounds__(64) void mfma_products_kernel(const float* a, const float* b, float* out, int n_sets) {
  const int set = blockIdx.x, l = threadIdx.x;
  const v16f d = mfma_products(a[set * 64 + l], b[set * 64 + l]);
#pragma unroll
  for (int r = 0; r < 16; r++) out[((size_t)set * 64 + l) * 16 + r] = d[r];
}
void launch_mfma_products(const float* a, const float* b, float* out, int n_sets, hipStream_t st) {
  if (n_sets > 0) hipLaunchKernelGGL(mfma_products_kernel, dim3(n_sets), dim3(64), 0, st, a, b, out, n_sets);
}

size_t attention_lds_bytes(int s_pitch) { return sizeof(float) * (size_t)kAttnQ * s_pitch; }

int attention_pitch(int max_len) {
  const int L = max(1, min(max_len, 512));
  return ((L + 15) / 16) * 16 + 4;
}

__global__ __launch_bounds__(256) void cls_attention_kernel(ClsArgs p);

// allow > 64 KiB of dynamic LDS for the tiled kernel on the current device; called
// at engine open and by the stand-alone operator, never inside a stream capture
void init_attention_kernels() {
  const int lds = (int)attention_lds_bytes(attention_pitch(512));
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(attention_kernel<true, 0, 4>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  (void)hipFuncSetAttribute(reinterpret_cast<const void*>(attention_kernel<false, 0, 4>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds);
}

// The wide variant (3 workgroups per CU by registers) is faster from rows of
// about 64 keys up; batches of mostly shorter rows, whose workgroups are short
// and latency-bound, run faster with the narrow one's 6.  The choice is by the
// batch's mean length (both variants give the same bits).
constexpr int kWideMinMeanLen = 48;
// mean length up to which the rows over kAttnLongL keys get a launch of their
// own (above it, nearly every row is long and the short rows' launch would be
// empty: its workgroups still cost C4 0.4 %)
constexpr int kSplitMaxMean = 448;

void launch_attention_plan(const AttnArgs& p, hipStream_t st, int split, int max_tiles) {
  hipLaunchKernelGGL(attention_plan_kernel, dim3(1), dim3(256), 0, st, p.cu, p.B, p.s_pitch - 4, max_tiles, split,
                     reinterpret_cast<int4*>(p.plan));
}

// Batches whose 32-query tiles leave CUs idle or end on a long critical path take
// the latency form's 16-query tiles; a full chip runs them 7 to 13 % slower than
// 32-query tiles.  Kernel times in us, 16-query against 32-query tiles (these need
// the plan kernel's 12 to 19 us first, once per pass): one row of 256 keys 11.0 /
// 14.2, 512: 22.6 / 24.8; 2 x 512: 29.3 / 31.1, 8 x 128: 12.0 / 12.2, 12 x 128: 16.4 /
// 14.9, 3 x 384: 26.9 / 25.9, 16 x 96: 14.7 / 12.7, so up to kHalfMaxT tokens.
//
// Beyond, up to kHalfMaxMixedT tokens, only batches whose longest row is over 1.5
// times the mean.  Up to kHalfMaxSegs segments they need no plan, and the bound of
// the lengths stands for the longest row: 1,782 tokens of 16 to 512 keys 31.5 / 45.7,
// 2,843: 44 / 60.6, 8 rows of 260 behind a bound of 512 39 / 55 per operator call.
// With more (times per operator call, plan included; the 32-query tiles run rows
// over kAttnLongL keys in a second launch, the 16-query tiles all rows in one):
//  * a row of more than kAttnLongL keys among others: 4,353 tokens of 16 to 512 0.88
//    of the time, 5,138: 0.87, 6,166: 0.91, 7,486: 120.0 / 120.2, 8,126: 127.6 / 126.3,
//    a pass of 8,985 2,665 / 2,705.  Where only a bound of the lengths is known,
//    it may be far above them: with rows of up to 300 keys behind a bound of 512,
//    3,400 tokens 56.7 / 52.9, 8,320: 125 / 112, so up to kHalfMaxBoundT tokens then;
//  * mostly rows too short for the wide variant: 130 of 8 to 40 and one of 512 0.76
//    of the time, 130 of 16 to 64 behind a bound of 512 0.84; without a row over
//    kAttnLongL less far: rows of 8 to 40 and one of 100, 2,553 tokens 29.4 / 30.7,
//    4,804: 44.1 / 43.5, 7,101: 61.6 / 58.6 (in a pass, whose plan serves all layers,
//    2,215 tokens 785 / 767);
//  * else never: 24 rows of 16 to 128 (1,669 tokens) 28.2 / 27.0, 40 of 60 to 260
//    (6,265) 79 / 71, 32 of 100 to 400 (7,963) 119 / 105.
constexpr int kHalfMaxT = 1024, kHalfMaxMixedT = 9000, kHalfMaxBoundT = 2500, kHalfMaxShortT = 4000;
// 16-query tiles (counting the longest row's for every row) whose workgroups, 12
// per tile, are resident at once at 4 per CU
constexpr int kHalfResidentTiles = 80;
// and at 2 per CU with 8 waves each: eight waves against four, 2 x 80 keys 6.2 /
// 6.7, one row of 320: 12.8 / 13.6, 512 (32 tiles): 22.6 / 23.1; 3 x 256 (48 tiles): 20.4 / 16.8
constexpr int kHalfWaves8Tiles = 42;
static int g_attention_form = 0;  // 0 by the batch, 1 tiled (32 queries) / register rows only, 2 latency form only
void set_attention_form(int form) { g_attention_form = form; }
int attention_form() { return g_attention_form; }

// attention_lat_kernel's workgroups run one to a compute unit: a batch of at most
// this many 32-query tiles (the longest row's for every row, which bounds the
// surplus workgroups) takes it while those with a query, at most 12 per (T + 7 B)
// / 8, fit in one round.  Kernel times in us against attention_kernel's 16-query
// tiles: one row of 128 keys 6.6 / 7.4, two of 128 (two rounds) 11 / 7.6.  Passes:
// one row of 129 427 / 444, 168: 445 / 461; 2 x 66: 414 / 431; 140 + 16: 432 / 448;
// 80 + 3 x 20: 414 / 429.
constexpr int kLatMaxTiles = 16, kLatMaxT = 256;

int attention_choice(int B, int T, int max_len, int longest, int cus) {
  if (max_len <= 64) return kAttnTiles32;
  if (B * (long)((max_len + 31) / 32) <= kLatMaxTiles && 12 * ((T + 7 * B) / 8) <= cus && T <= kLatMaxT) return kAttnLat;
  if (T <= kHalfMaxT) return kAttnTiles16;
  const long top = longest > 0 && B > kHalfMaxSegs ? longest : max_len;
  const bool is_short = T <= kWideMinMeanLen * (long)B;
  int most = kHalfMaxMixedT;
  if (2 * top * B <= 3L * T) most = 0;
  else if (B > kHalfMaxSegs && top <= kAttnLongL) most = is_short ? kHalfMaxShortT : 0;
  else if (B > kHalfMaxSegs && longest <= 0 && !is_short) most = kHalfMaxBoundT;
  return T <= most ? kAttnTiles16 : kAttnTiles32;
}

void launch_attention(const AttnArgs& p, int T, hipStream_t st, bool plan) {
  if (T <= 0 || p.B <= 0) return;
  const int max_len = p.s_pitch - 4;  // round16 of the bound of the lengths
  const int cus = max_len > 64 && T <= kLatMaxT ? device_cu_count() : 0;  // (asked for only where it counts)
  const int choice = attention_choice(p.B, T, max_len, p.longest, cus);
  const bool lat = g_attention_form != 1 && choice == kAttnLat;
  const bool half = g_attention_form == 2 || (g_attention_form == 0 && choice == kAttnTiles16);
  const int max_tiles = attention_max_tiles(p.B, T);
  const int records = (int)attention_plan_list_records(p.B, T);
  if (lat) {
    const int tps = (min(max_len, T) + kLatQ - 1) / kLatQ;  // (no segment exceeds the batch's tokens)
    const dim3 grid(p.B * tps * 12);
    if (min(max_len, T) <= 128) hipLaunchKernelGGL(attention_lat_kernel<1>, grid, dim3(512), 0, st, p, tps);
    else hipLaunchKernelGGL(attention_lat_kernel<2>, grid, dim3(512), 0, st, p, tps);
    return;
  }
  if (half) {
    const size_t lds = attention_lds_bytes(p.s_pitch) / 2;
    if (p.B <= kHalfMaxSegs) {
      const int tps = (max_len + 15) / 16, tiles = p.B * tps;
      if (tiles <= kHalfWaves8Tiles) {
        hipLaunchKernelGGL((attention_kernel<true, 2, 8>), dim3(12 * tiles), dim3(512), lds, st, p, tps, 0);
      } else if (tiles <= kHalfResidentTiles) {
        hipLaunchKernelGGL((attention_kernel<true, 2, 4>), dim3(12 * tiles), dim3(256), lds, st, p, tps, 0);
      } else {  // the most tiles an XCD gets: half as many again as the batch has, plus half a segment's
        const int slots = (3 * ((T + 15 * p.B) / 16) + tps) / 2 + 1;
        hipLaunchKernelGGL((attention_kernel<true, 2, 4>), dim3(8 * slots), dim3(256), lds, st, p, 0, 0);
      }
      return;
    }
    if (plan) launch_attention_plan(p, st, 0, max_tiles);
    hipLaunchKernelGGL((attention_kernel<true, 1, 4>), dim3(2 * 8 * attention_plan_cap(max_tiles)), dim3(256), lds, st, p,
                       records, 0);
    return;
  }
  if (max_len <= 32) {
    hipLaunchKernelGGL(attention_rows_kernel<2>, dim3(p.B * 12), dim3(256), 0, st, p);
    return;
  }
  if (max_len <= 64) {
    hipLaunchKernelGGL(attention_rows_kernel<4>, dim3(p.B * 12), dim3(256), 0, st, p);
    return;
  }
  // In batches of mostly shorter rows (by the mean length; the plan, built once
  // per pass, and every launch of the pass make the same choice), the rows over
  // kAttnLongL keys get a launch of their own, so that the short rows' tiles run
  // three workgroups per CU.  The grids are sized for the worst case; the
  // surplus workgroups leave after one scalar load (plan_item).
  const bool split = max_len > kAttnLongL && T <= kSplitMaxMean * p.B;
  if (plan) launch_attention_plan(p, st, split ? 1 : 0, max_tiles);
  const bool wide = T > kWideMinMeanLen * p.B;
  const dim3 grid(8 * attention_plan_cap(max_tiles));
  auto launch = [&](int list, size_t lds) {
    if (wide)
      hipLaunchKernelGGL((attention_kernel<true, 0, 4>), grid, dim3(256), lds, st, p, records, list);
    else
      hipLaunchKernelGGL((attention_kernel<false, 0, 4>), grid, dim3(256), lds, st, p, records, list);
  };
  if (split) {
    launch(0, attention_lds_bytes(kAttnLongL + 4));
    launch(1, attention_lds_bytes(p.s_pitch));
  } else {
    launch(0, attention_lds_bytes(p.s_pitch));
  }
}

// ---------------------------------------------------------------------------
// The attention operator's only scratch, the tile plan, in a file-scope device
// array for callers that cannot allocate (ae_attention_varlen_noalloc).  Each
// GPU holds its own copy until the process ends; host code reaches it only
// through the per-device address that hipGetSymbolAddress returns (the array's
// name is a host-side stand-in, not a device address).  Every call on a GPU
// shares that GPU's array: calls that overlap on one GPU race.  The plan kernel
// rewrites every record a launch reads, so nothing needs clearing between calls.
// ---------------------------------------------------------------------------
static __device__ __align__(256) int4 scratch[kNoAllocPlanRecords];

namespace {
constexpr int kNoAllocMaxDevices = 64;
std::mutex g_noalloc_mu;
int* g_noalloc_plan[kNoAllocMaxDevices] = {};
}  // namespace

hipError_t noalloc_plan_scratch(int** plan) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kNoAllocMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_noalloc_mu);
  if (!g_noalloc_plan[dev]) {  // first call on this device (current): resolve its copy once
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    init_attention_kernels();
    g_noalloc_plan[dev] = static_cast<int*>(ptr);
  }
  *plan = g_noalloc_plan[dev];
  return hipSuccess;
}

void launch_attention_short(const AttnArgs& p, hipStream_t st) {
  if (p.B <= 0) return;
  AttnArgs q = p;
  q.skip_from = 16;
  hipLaunchKernelGGL(attention_rows_kernel<1>, dim3(p.B * 12), dim3(64), 0, st, q);
}

// ---------------------------------------------------------------------------
// Layer-11 [CLS] pruning (reference src/model.rs:770-913)
// ---------------------------------------------------------------------------
// one workgroup (4 waves) per (sequence, head): the [CLS] query attends to its
// segment with the same exact scalar order as attention_kernel
// (src/model.rs:814-843).  The global loads of the [CLS] row's int8
// activations, the head's q_only weight fragments and the K rows of the
// thread's keys (tid, tid + 256) are issued at the start.  Wave 0 forms the
// head's 32 q values as the q_only GEMM does for that row (int8 MFMA with the
// [CLS] row as row 0 of the A tile, then fma(f32(acc), sa * ws, bias)).  The PV
// lanes read V from global memory through a register ring 16 keys ahead, its
// first loads issued before the softmax phases, so the workgroup needs no large
// LDS tile and many fit on a CU.  Keys past p.max_len (<= 512) are not attended
// (the embedding kernel reports such sequences through the workspace's error
// word).
// float4 i of the [CLS] row (token s0) of hidden: as stored, or (hidden_stats)
// the LayerNorm output of that row, recomputed as the LayerNorm forms it
__device__ __forceinline__ float4 cls_hidden_row(const ClsArgs& p, int s0, int i) {
  float4 v = reinterpret_cast<const float4*>(p.hidden + (size_t)s0 * H)[i];
  if (p.hidden_stats) {
    const float2 st = p.hidden_stats[s0];
    const float4 g = reinterpret_cast<const float4*>(p.ln_gamma)[i];
    const float4 bt = reinterpret_cast<const float4*>(p.ln_beta)[i];
    v.x = (v.x - st.x) * st.y * g.x + bt.x;
    v.y = (v.y - st.x) * st.y * g.y + bt.y;
    v.z = (v.z - st.x) * st.y * g.z + bt.z;
    v.w = (v.w - st.x) * st.y * g.w + bt.w;
  }
  return v;
}

__global__ __launch_bounds__(256) void cls_attention_kernel(ClsArgs p) {
  __shared__ __attribute__((aligned(16))) float S[512];
  __shared__ __attribute__((aligned(16))) float sQ[32];
  __shared__ float s_m[4];
  __shared__ float s_inv;
  __shared__ uint64_t s_tab[32];
  const int b = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int s0 = p.cu[b], L = min(p.cu[b + 1] - s0, p.max_len);
  exp_tab_fill(s_tab, tid);  // ordered before the exp phase by the barriers of the scores and max
  const ExpTabLds tb{s_tab};
  // q_only for the [CLS] row and this head's 32 columns: A fragment (row 0 only,
  // K steps 0..5) and the two 16-column weight blocks (fragment order of
  // swizzle_weights: [K/64][N/16][64 lanes][16 bytes])
  v4i qa[6], qb[6][2];
  if (wave == 0) {
#pragma unroll
    for (int kt = 0; kt < 6; kt++) {
      qa[kt] = (lane & 15) == 0 ? *reinterpret_cast<const v4i*>(p.act_q + (size_t)s0 * H + kt * 64 + (lane >> 4) * 16)
                                : v4i{0, 0, 0, 0};
#pragma unroll
      for (int j = 0; j < 2; j++)
        qb[kt][j] = *reinterpret_cast<const v4i*>(p.wq + (((size_t)kt * (H / 16) + 2 * h + j) * 64 + lane) * 16);
    }
  }
  if (h == 0 && tid < 96)  // gather the [CLS] row of hidden (the tail's residual)
    reinterpret_cast<float4*>(p.hidden_c + (size_t)b * H)[tid] = cls_hidden_row(p, s0, tid);
  float4 kr[2][8];
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int j = tid + 256 * u;
    if (j < L) {
#pragma unroll
      for (int e = 0; e < 8; e++) kr[u][e] = *reinterpret_cast<const float4*>(p.kv + (size_t)(s0 + j) * 2 * H + h * 32 + 4 * e);
    }
  }
  if (wave == 0) {
    v4i acc[2] = {v4i{0, 0, 0, 0}, v4i{0, 0, 0, 0}};
#pragma unroll
    for (int kt = 0; kt < 6; kt++)
#pragma unroll
      for (int j = 0; j < 2; j++) acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(qa[kt], qb[kt][j], acc[j], 0, 0, 0);
    if (lane < 16) {  // row 0 of the result: lane l holds columns 16 j + l, register 0
      const float sa = p.act_scale[s0];
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int col = h * 32 + 16 * j + lane;
        sQ[16 * j + lane] = fmaf((float)acc[j][0], sa * p.wq_scale[col], p.wq_bias[col]);
      }
    }
  }
  __syncthreads();
  float q[32];
#pragma unroll
  for (int d = 0; d < 32; d += 4) {
    const float4 v = *reinterpret_cast<const float4*>(&sQ[d]);
    q[d] = v.x; q[d + 1] = v.y; q[d + 2] = v.z; q[d + 3] = v.w;
  }
  // scores (dot32_f32 order) and their max
  float m = -INFINITY;
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int j = tid + 256 * u;
    if (j < L) {
      float sum = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; e++) {
        sum += q[4 * e] * kr[u][e].x;
        sum += q[4 * e + 1] * kr[u][e].y;
        sum += q[4 * e + 2] * kr[u][e].z;
        sum += q[4 * e + 3] * kr[u][e].w;
      }
      const float sc = sum * kInvSqrtD;
      S[j] = sc;
      m = nanless_max(m, sc);
    }
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) m = nanless_max(m, __shfl_xor(m, off, 64));
  if (lane == 0) s_m[wave] = m;
  // the PV lanes' first V values (keys 0-15, dim `lane`; rows past the segment
  // clamped), issued now so that their latency hides behind the softmax
  const float* vcol = p.kv + (size_t)s0 * 2 * H + H + h * 32 + (lane & 31);
  const int nvb = L >> 3;  // full batches of 8 keys
  float va[8], vb[8];
  auto ldv = [&](int bi, float (&v)[8]) {
    const int t0 = 8 * min(bi, max(nvb - 1, 0));
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = vcol[(size_t)min(t0 + k, L - 1) * 2 * H];
  };
  if (wave == 0 && L > 0) {
    ldv(0, va);
    ldv(1, vb);
  }
  __syncthreads();
  m = nanless_max(nanless_max(s_m[0], s_m[1]), nanless_max(s_m[2], s_m[3]));
#pragma unroll
  for (int u = 0; u < 2; u++) {  // uniform trip count (expf_libm needs all lanes)
    const int j = tid + 256 * u;
    const float e = expf_libm((j < L ? S[j] : 0.0f) - m, tb);
    if (j < L) S[j] = e;
  }
  __syncthreads();
  if (tid == 0) {  // in-order denominator; batches of 16 keys, each read while the previous one is added
    float sum = 0.0f;
    const int nb = L >> 4;
    float4 ea[4], eb[4];
    auto ld = [&](int bi, float4 (&v)[4]) {
      const float4* src = reinterpret_cast<const float4*>(&S[16 * min(bi, nb - 1)]);
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] = src[i];
    };
    auto add = [&](const float4 (&v)[4]) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        sum += v[i].x; sum += v[i].y; sum += v[i].z; sum += v[i].w;
      }
    };
    if (nb > 0) {
      ld(0, ea);
      int bi = 0;
      for (; bi + 2 <= nb; bi += 2) {
        ld(bi + 1, eb);
        __builtin_amdgcn_sched_barrier(0);
        add(ea);
        __builtin_amdgcn_sched_barrier(0);
        ld(bi + 2, ea);
        __builtin_amdgcn_sched_barrier(0);
        add(eb);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (bi < nb) add(ea);
    }
    for (int j = 16 * nb; j < L; j++) sum += S[j];
    s_inv = 1.0f / sum;
  }
  __syncthreads();
  const float inv = s_inv;
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int j = tid + 256 * u;
    if (j < L) S[j] = S[j] * inv;
  }
  __syncthreads();
  if (wave == 0) {
    float o = 0.0f;
    if (lane < 32) {  // ctx_d = sum_t p_t * v_t,d in order; V two batches of 8 keys ahead
      auto add = [&](int bi, const float (&v)[8]) {
        const float4 p0 = *reinterpret_cast<const float4*>(&S[8 * bi]);
        const float4 p1 = *reinterpret_cast<const float4*>(&S[8 * bi + 4]);
        o = o + p0.x * v[0];
        o = o + p0.y * v[1];
        o = o + p0.z * v[2];
        o = o + p0.w * v[3];
        o = o + p1.x * v[4];
        o = o + p1.y * v[5];
        o = o + p1.z * v[6];
        o = o + p1.w * v[7];
      };
      int bi = 0;
      for (; bi + 2 <= nvb; bi += 2) {  // va holds batch bi, vb batch bi + 1
        add(bi, va);
        ldv(bi + 2, va);
        add(bi + 1, vb);
        ldv(bi + 3, vb);
      }
      if (bi < nvb) add(bi, va);
      for (int t = 8 * nvb; t < L; t++) o = o + S[t] * vcol[(size_t)t * 2 * H];
      p.ctx_c[(size_t)b * H + h * 32 + lane] = o;
    }
    float a = lane < 32 ? fabsf(o * p.smooth[h * 32 + lane]) : 0.0f;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) a = nanless_max(a, __shfl_xor(a, off, 64));
    if (lane == 0) atomicMax(&p.rowmax_ctx_c[b], __float_as_uint(a));
  }
}

// The same for batches whose segments are at most 64 tokens long: one wave per
// (sequence, head), lane t holding key t, four heads per workgroup (grid B x 3),
// the same arithmetic in the same order as cls_attention_kernel.  With a
// workgroup per (sequence, head), three of its four waves had no key in most
// phases, and the launch was bound by the latency of its ~100 k workgroups.
__global__ __launch_bounds__(256, 6) void cls_attention_short_kernel(ClsArgs p) {
  __shared__ __attribute__((aligned(16))) float S[4][64];
  __shared__ __attribute__((aligned(16))) float sQ[4][32];
  const int b = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h = 4 * blockIdx.y + wave;
  const int s0 = p.cu[b], L = min(p.cu[b + 1] - s0, min(p.max_len, 64));
  const ExpTab tb = exp_tab_regs();
  // q_only for the [CLS] row and this head's 32 columns (as cls_attention_kernel)
  v4i qa[6], qb[6][2];
#pragma unroll
  for (int kt = 0; kt < 6; kt++) {
    qa[kt] = (lane & 15) == 0 ? *reinterpret_cast<const v4i*>(p.act_q + (size_t)s0 * H + kt * 64 + (lane >> 4) * 16)
                              : v4i{0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 2; j++)
      qb[kt][j] = *reinterpret_cast<const v4i*>(p.wq + (((size_t)kt * (H / 16) + 2 * h + j) * 64 + lane) * 16);
  }
  float4 kr[8];
  {
    v4i acc[2] = {v4i{0, 0, 0, 0}, v4i{0, 0, 0, 0}};
#pragma unroll
    for (int kt = 0; kt < 6; kt++)
#pragma unroll
      for (int j = 0; j < 2; j++) acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(qa[kt], qb[kt][j], acc[j], 0, 0, 0);
    // the K row of key `lane`, loaded once the MFMA operands' registers are free
    // (loaded with them, the three sets held 104 registers: 4 waves per SIMD)
    if (lane < L) {
#pragma unroll
      for (int e = 0; e < 8; e++) kr[e] = *reinterpret_cast<const float4*>(p.kv + (size_t)(s0 + lane) * 2 * H + h * 32 + 4 * e);
    }
    if (lane < 16) {  // row 0 of the result: lane l holds columns 16 j + l, register 0
      const float sa = p.act_scale[s0];
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int col = h * 32 + 16 * j + lane;
        sQ[wave][16 * j + lane] = fmaf((float)acc[j][0], sa * p.wq_scale[col], p.wq_bias[col]);
      }
    }
  }
  wave_lds_sync();
  // the PV lanes' first V values (keys 0-15, dim `lane`; rows past the segment
  // clamped), issued now so that their latency hides behind the softmax
  const float* vcol = p.kv + (size_t)s0 * 2 * H + H + h * 32 + (lane & 31);
  const int nvb = L >> 3;  // full batches of 8 keys
  float va[8], vb[8];
  auto ldv = [&](int bi, float (&v)[8]) {
    const int t0 = 8 * min(bi, max(nvb - 1, 0));
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = vcol[(size_t)min(t0 + k, L - 1) * 2 * H];
  };
  if (L > 0) {
    ldv(0, va);
    ldv(1, vb);
  }
  // score of key `lane` (dot32_f32 order) and the max over the keys
  float sc = 0.0f, m = -INFINITY;
  if (lane < L) {
    float sum = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; e++) {  // q read as needed (an LDS broadcast), not held in 32 registers
      const float4 q = *reinterpret_cast<const float4*>(&sQ[wave][4 * e]);
      sum += q.x * kr[e].x;
      sum += q.y * kr[e].y;
      sum += q.z * kr[e].z;
      sum += q.w * kr[e].w;
    }
    sc = sum * kInvSqrtD;
    m = nanless_max(m, sc);  // a NaN score is never the max (the reference's `if s > max`)
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) m = nanless_max(m, __shfl_xor(m, off, 64));
  const float e = expf_libm(sc - m, tb);  // all lanes (expf_libm); keys past L unused
  if (lane < L) S[wave][lane] = e;
  wave_lds_sync();
  float inv = 0.0f;
  if (lane == 0) {  // in-order denominator, 16-key batches read ahead of their adds
    float sum = 0.0f;
    const int nb = L >> 4;
    float4 ea[4], eb[4];
    auto ld = [&](int bi, float4 (&v)[4]) {
      const float4* src = reinterpret_cast<const float4*>(&S[wave][16 * min(bi, nb - 1)]);
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] = src[i];
    };
    auto add = [&](const float4 (&v)[4]) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        sum += v[i].x; sum += v[i].y; sum += v[i].z; sum += v[i].w;
      }
    };
    if (nb > 0) {
      ld(0, ea);
      int bi = 0;
      for (; bi + 2 <= nb; bi += 2) {
        ld(bi + 1, eb);
        __builtin_amdgcn_sched_barrier(0);
        add(ea);
        __builtin_amdgcn_sched_barrier(0);
        ld(bi + 2, ea);
        __builtin_amdgcn_sched_barrier(0);
        add(eb);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (bi < nb) add(ea);
    }
    for (int j = 16 * nb; j < L; j++) sum += S[wave][j];
    inv = 1.0f / sum;
  }
  inv = __shfl(inv, 0, 64);
  if (lane < L) S[wave][lane] = e * inv;
  wave_lds_sync();
  float o = 0.0f;
  if (lane < 32) {  // ctx_d = sum_t p_t * v_t,d in order; V two batches of 8 keys ahead
    auto add = [&](int bi, const float (&v)[8]) {
      const float4 p0 = *reinterpret_cast<const float4*>(&S[wave][8 * bi]);
      const float4 p1 = *reinterpret_cast<const float4*>(&S[wave][8 * bi + 4]);
      o = o + p0.x * v[0];
      o = o + p0.y * v[1];
      o = o + p0.z * v[2];
      o = o + p0.w * v[3];
      o = o + p1.x * v[4];
      o = o + p1.y * v[5];
      o = o + p1.z * v[6];
      o = o + p1.w * v[7];
    };
    int bi = 0;
    for (; bi + 2 <= nvb; bi += 2) {  // va holds batch bi, vb batch bi + 1
      add(bi, va);
      ldv(bi + 2, va);
      add(bi + 1, vb);
      ldv(bi + 3, vb);
    }
    if (bi < nvb) add(bi, va);
    for (int t = 8 * nvb; t < L; t++) o = o + S[wave][t] * vcol[(size_t)t * 2 * H];
    p.ctx_c[(size_t)b * H + h * 32 + lane] = o;
  }
  float a = lane < 32 ? fabsf(o * p.smooth[h * 32 + lane]) : 0.0f;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) a = nanless_max(a, __shfl_xor(a, off, 64));
  if (lane == 0) atomicMax(&p.rowmax_ctx_c[b], __float_as_uint(a));
  if (h == 0)  // gather the [CLS] row of hidden (the tail's residual), last: no registers held meanwhile
    for (int i = lane; i < 96; i += 64) reinterpret_cast<float4*>(p.hidden_c + (size_t)b * H)[i] = cls_hidden_row(p, s0, i);
}

void launch_cls(const ClsArgs& p, hipStream_t st) {
  if (p.max_len <= 64)
    hipLaunchKernelGGL(cls_attention_short_kernel, dim3(p.B, 3), dim3(256), 0, st, p);
  else
    hipLaunchKernelGGL(cls_attention_kernel, dim3(p.B, 12), dim3(256), 0, st, p);
}

}  // namespace aek
