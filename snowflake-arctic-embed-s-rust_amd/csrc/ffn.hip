// ffn.hip -- the FFN block of one encoder layer as one gfx950 kernel:
//
//   g   = GELU(fma(f32(A . W1^T), sa*ws1, b1)) * inv_smooth2      FFN-up + GELU
//   q,s = per-row absmax int8 quantization of g                    gelu_smooth_quantize
//   out = fma(f32(q . W2^T), s*ws2, b2 + res)                       FFN-down + residual
//
// (reference src/model.rs:725-755: gemm_int8_fused(ffn_inter) -> inter_buf,
// gelu_smooth_quantize_batch -> inter_q/act_scale, gemm_int8_fused(ffn_out,
// residual hidden); the arithmetic of each step is the one of gemm.hip's
// kEpiGelu epilogue, the row quantizer and the kAF32Q epilogue.)
//
// A workgroup of 8 waves owns 16 NR kP complete token rows, in kP passes of
// 16 NR rows, so the [rows, 1536] intermediate never leaves the CU.  What its
// registers hold of it is the pre-activation v: the row maximum of |g| needs v
// only at a few candidates, and a value whose quantization the fast GELU leaves
// undecided is recomputed from v on the spot.  Per pass:
//
//  1. FFN-up.  Wave w takes the 16-column blocks w, w + 8, .. (12 of them).
//     The weights are the MFMA's A operand and the tokens its B operand, so a
//     lane ends with four consecutive columns of one token: the row maxima, the
//     row scales and the quantizer's factors are one register per 16 rows, and
//     four quantized values are one dword of the int8 row.
//  2. Row maxima, exactly, from a few candidates (below).
//  3. GELU and quantization into the int8 row tile in LDS.
//
// FFN-down then streams W2 once for all rows of the workgroup; wave w computes
// columns [48 w, 48 w + 48).
//
// What bounds it (s_memtime stamps of one 32-row pass, cycles at 2.4 GHz): FFN-up
// 13 K (590 KB of W1 through the CU's 64 B/clk vector memory path; its 8 K of MFMA
// and VALU work hide behind it), row maxima 7 K (two barriers and the scan), GELU
// and quantization 16 K (VALU issue: 27 instructions per value, 83 cycles per
// wave64 value), FFN-down 8 K per 32 rows (at 16 and 32 rows per workgroup the W2
// stream).  MFMA and VALU work of different waves do not overlap on this part.
// The code is kept to 27-48 KB: every workgroup runs most of it once, and at 72
// or 98 KB (all loops unrolled) it fell out of the instruction cache between
// workgroups (first round of 64-row workgroups 67 us instead of 54).
// Measured against the kernel before it (32- and 64-row workgroups holding g in
// place of v, the tokens as the A operand: row state in four registers per 16
// rows, a byte transpose per dword, 22 cycles per value of top-element tracking,
// 40 of quantization, and an undecided value recomputed from W1): 2,048 rows 26.9
// -> 19.2 us (16-row workgroups), 8,192 rows 32.4 -> 29.2, 32,768 rows 112 -> 107,
// 68,270 rows 247 -> 233, 294,912 rows 987 -> 900 us (same box).
// Tried: 12 or 16 waves in one workgroup with FFN-down interleaved by chunks of
// 192 or 256 columns (8 or 6 more barriers per tile: 20-25 % slower), FFN-up
// computed twice instead of holding v (152 us at 32,768 rows), the FFN-up and
// GELU loops rolled too (indexed register moves; 12 % slower at 2,048 rows).
//
// Weights are the pre-swizzled fragment order of gemm.hip ([K/64][N/16][64
// lanes][16 B]), streamed per wave from L2.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_common.hpp"
#include "kernels.hpp"

namespace aek {

namespace {
constexpr int kH = 384, kF = 1536;
constexpr int kWaves = 8, kThreads = 64 * kWaves;
constexpr int kAPitch = kH + 16;          // LDS row pitch of the input tile (bytes)
constexpr int kQPitch = kF + 16;          // LDS row pitch of the quantized intermediate (bytes)
constexpr int kUpCB = kF / 16 / kWaves;   // FFN-up 16-column blocks per wave (12)
constexpr int kDnCB = kH / 16 / kWaves;   // FFN-down 16-column blocks per wave (3)
constexpr int kRing = 8;                  // FFN-down K steps of weight fragments in flight
constexpr int kUpSteps = kH / 64, kDnSteps = kF / 64;

typedef float v12f __attribute__((ext_vector_type(12)));
typedef float v4f __attribute__((ext_vector_type(4)));

// a raw buffer resource over `bytes` bytes of weights (gfx9 descriptor word 3:
// 32-bit data format) and a 16-byte load at a vector plus scalar byte offset
__device__ __forceinline__ __amdgpu_buffer_rsrc_t weight_rsrc(const int8_t* base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(base), 0, bytes, 0x00020000);
}
__device__ __forceinline__ v4i weight_load(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff) {
  return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}
// lanes of a wave mask below this one
__device__ __forceinline__ int lanes_below(uint64_t mask) {
  return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0));
}
}  // namespace

// Bounds of the fast path (kFast), from gelu_fast's certified bound
// |G - G'| <= kGeluFastRel |G'| + kGeluFastAbs (device_common.hpp), u = 2^-24 the
// unit roundoff.  The reference quantizes x = RN(RN(G gs) inv), the kernel
// x' = RN(G' RN(gs inv)); two roundings on either side give
//   |x - x'| <= (kGeluFastRel + 4u)(1 + 2^-20) |x'| + kGeluFastAbs gs_max inv (1 + 2^-20) + tiny,
// gs_max = max |gs| over all columns.  x' and x round to the same int8 value when
// x' is farther than that from every half-integer, i.e. when
//   |x' - round(x')| + kQRel |x'| < 0.5 - (kGeluFastAbs gs_max inv (1 + 2^-20) + 2^-24)
// (the distance is exact; 2^-24 covers the rounding of the sums).
constexpr float kQRel = 0x1.ep-21f;    // >= (2^-21 + 2^-22)(1 + 2^-20)
constexpr float kQAbs = 0x1.65p-24f;   // >= kGeluFastAbs (1 + 2^-20)
// |GELU(v)| <= max(kCapMul v - kCapSub, kCapMin) for every v: a line just above
// the tangent at v = 2, and a constant above |GELU| to its left.  Below 0.25,
// |GELU(v)| <= max(v, 0.17) < kCapMin; from 8 on, GELU(v) <= v is below the line;
// the floats in between are enumerated by test_ffn_gelu_cap_on_every_float.  The
// row maxima use the bound times |gs| (rounding is monotonic, so |g| <= it).
constexpr float kCapMul = 1.0854f, kCapSub = 0.2158f, kCapMin = 0.44f;
// the share of a row's largest bound from which an element is a candidate for
// its maximum: GELU(v) exceeds that share of the bound for every v from 0.57 on
// (it falls to 1 / kCapMul = 0.9213 for large v)
constexpr float kCandShare = 0.92f;

// repair counters (test hook ae_debug_ffn_repairs): [0] 16-row x 16-column tiles
// recomputed exactly because a quantized value was undecided, [1] the NR 16-row
// groups of each pass whose first scan had more candidates than the pass has rows
__device__ unsigned long long g_ffn_repairs[2];

// kFast: the GELU is gelu_fast with exact repair (the same bits as the exact
// kernel, kFast = false, whose registers hold g = GELU(v) gs in place of v).
//
// Row maxima (kFast): FFN-up keeps, per lane, row and column block, the largest
// bound B = max(kCapMul v - kCapSub, kCapMin) |gs| of its four columns, and from
// those U, the row's largest.  Every element whose bound reaches kCandShare U,
// the top one among them, is evaluated exactly; the largest, M1, is the row
// maximum if M1 >= kCandShare U, because no other element can exceed that.
// Otherwise (rows whose largest v is below 0.57) a second scan evaluates every
// element whose bound reaches M1.  The candidates of a wave (a few) go to a list
// in LDS first, so that one gelu_exact serves them all.
//
// kLn (16-row workgroups): the LayerNorm + SmoothQuant of the output rows (`ln`,
// with ln_quant_kernel's arithmetic in its order) follows in the same kernel,
// its 32 threads per row and in-order sums working on the rows in sQ's space.
// As a launch of its own it took 7.1 us at 1,280 rows and 7.9 at 3,769, most of
// it the launch and the rows' way through memory: passes of 1,280 rows 651 -> 616
// us, 2,844 rows 1,031 -> 993, 4,096 rows 1,622 -> 1,579.
template <int NR, int kP, bool kFast, bool kLn = false>
__global__ __launch_bounds__(kThreads, 2) void ffn_kernel(FfnArgs p, LnArgs ln) {
  static_assert(!kLn || NR * kP == 1, "LayerNorm of 16 rows by 512 threads");
  constexpr int RP = 16 * NR, R = RP * kP;  // token rows per pass and per workgroup
  __shared__ __attribute__((aligned(16))) int8_t sA[R * kAPitch];
  // the quantized intermediate; before a pass's quantization its rows hold the waves' candidate lists
  __shared__ __attribute__((aligned(16))) int8_t sQ[R * kQPitch];
  constexpr int kListCap = RP * kQPitch / kWaves / 8;  // (v, column | row << 16) per wave
  __shared__ __attribute__((aligned(16))) float sWs[kF], sB[kF], sGs[kF];
  __shared__ __attribute__((aligned(16))) float sU[R][kWaves];  // per-wave row maxima of the bound (exact kernel: of |g|)
  __shared__ float sSa[R], sMax[R];
  __shared__ uint32_t sM[2][R];  // row maxima of |g| over the first scan's elements and the second's (f32 bits)
  __shared__ int sCnt[kP], s_full[kP];  // candidates of a pass's first scan; a wave's exceeded its list
  __shared__ uint32_t s_gmax;
  __shared__ uint64_t s_tab[32];
  // (wave via readfirstlane: known uniform, so the weight fragments' offsets are scalars)
  int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int lane = tid & 63, fr = lane & 15, fq = lane >> 4;  // fr: token of the 16-row block, fq: k group and column quad
  const int m0 = blockIdx.x * R;

  // weight fragments through buffer resources: the fragment's offset is a scalar
  // and the lane's 16 bytes one VGPR shared by every load.  Opaque copies of the
  // bases: the offsets are formed next to their loads, not hoisted and held
  const __amdgpu_buffer_rsrc_t w1r = weight_rsrc(p.w1, kF * kH), w2r = weight_rsrc(p.w2, kF * kH);
  const uint32_t lane16 = (uint32_t)lane * 16u;

  // input rows (rows past M repeat row M-1; never stored)
  constexpr int kLd = (R * (kH / 16) + kThreads - 1) / kThreads;
  v4i an[kLd];
#pragma unroll
  for (int i = 0; i < kLd; i++) {
    const int c = min(tid + kThreads * i, R * (kH / 16) - 1), row = c / (kH / 16), c16 = c - row * (kH / 16);
    an[i] = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(p.A + (size_t)min(m0 + row, p.M - 1) * kH + c16 * 16));
  }
  v4i w1[2][kUpSteps];  // column blocks j and j + 1
  auto load_w1 = [&](int j, v4i (&dst)[kUpSteps]) {
    int base = (j * kWaves + wave) * 1024;
    asm volatile("" : "+s"(base));
#pragma unroll
    for (int kt = 0; kt < kUpSteps; kt++) dst[kt] = weight_load(w1r, lane16, base + kt * (kF / 16) * 1024);
  };
  load_w1(0, w1[0]);
  load_w1(1, w1[1]);
  // the column operands
  float gmx = 0.0f;
  for (int c = tid; c < kF / 4; c += kThreads) {
    reinterpret_cast<float4*>(sWs)[c] = reinterpret_cast<const float4*>(p.w1_scale)[c];
    reinterpret_cast<float4*>(sB)[c] = reinterpret_cast<const float4*>(p.b1)[c];
    const float4 g = reinterpret_cast<const float4*>(p.g_smooth)[c];
    reinterpret_cast<float4*>(sGs)[c] = g;
    gmx = fmaxf(fmaxf(fmaxf(gmx, fabsf(g.x)), fmaxf(fabsf(g.y), fabsf(g.z))), fabsf(g.w));
  }
  if (tid < R) {
    sSa[tid] = p.a_scale[min(m0 + tid, p.M - 1)];
    sM[0][tid] = __float_as_uint(1e-8f);
    sM[1][tid] = 0u;
  }
  if (tid < kP) sCnt[tid] = 0, s_full[tid] = 0;
  if (tid == 0) s_gmax = 0u;
  exp_tab_fill(s_tab, tid);
#pragma unroll
  for (int i = 0; i < kLd; i++) {
    const int c = tid + kThreads * i, row = c / (kH / 16), c16 = c - row * (kH / 16);
    if (R * (kH / 16) % kThreads == 0 || c < R * (kH / 16)) *reinterpret_cast<v4i*>(&sA[row * kAPitch + c16 * 16]) = an[i];
  }
  __syncthreads();
  if constexpr (kFast) {
    gmx = row16_max(gmx);
    if (fr == 0) atomicMax(&s_gmax, __float_as_uint(gmx));  // read after the first row-maximum barrier
  }
  const ExpTabLds tb{s_tab};
  // (constants that an f32 instruction would otherwise read from an SGPR, at half its rate)
  float kc = kGeluFastK, kcap = kCapMul, kq = kQRel;
  asm volatile("" : "+v"(kc), "+v"(kcap), "+v"(kq));
  // opaque per phase: addresses formed from them are not kept from one phase to the next (spills)
  auto opaque_ids = [&]() { asm volatile("" : "+v"(tid), "+v"(lane), "+v"(fr), "+v"(fq)); };

#pragma unroll 1
  for (int pp = 0; pp < kP; pp++) {
    const int r0 = RP * pp;  // this pass's first row in the tile
    opaque_ids();
    float sa[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) sa[i] = sSa[r0 + i * 16 + fr];

    // ---- FFN-up: v = fma(f32(acc), sa * ws, b) and its bound ----
    // (vectors over the column blocks: the scans index them in rolled loops)
    v12f v[NR][4], bm[NR];
    float mx[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) mx[i] = 0.0f;
#pragma unroll
    for (int j = 0; j < kUpCB; j++) {
      const int col = (j * kWaves + wave) * 16 + fq * 4;  // this lane's four columns
      v4i acc[NR];
#pragma unroll
      for (int i = 0; i < NR; i++) acc[i] = v4i{0, 0, 0, 0};
#pragma unroll
      for (int kt = 0; kt < kUpSteps; kt++)
#pragma unroll
        for (int i = 0; i < NR; i++) {
          const v4i t = *reinterpret_cast<const v4i*>(&sA[(r0 + i * 16 + fr) * kAPitch + kt * 64 + fq * 16]);
          acc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w1[j & 1][kt], t, acc[i], 0, 0, 0);
        }
      if (j + 2 < kUpCB) load_w1(j + 2, w1[j & 1]);
      const v4f ws = *reinterpret_cast<const v4f*>(&sWs[col]);
      const v4f bb = *reinterpret_cast<const v4f*>(&sB[col]);
      const v4f gs = *reinterpret_cast<const v4f*>(&sGs[col]);
      const float cap0 = kCapMin * fmaxf(fmaxf(fabsf(gs[0]), fabsf(gs[1])), fmaxf(fabsf(gs[2]), fabsf(gs[3])));
#pragma unroll
      for (int i = 0; i < NR; i++) {
        float u[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          float x = fmaf((float)acc[i][r], sa[i] * ws[r], bb[r]);
          if constexpr (kFast) {
            // in program order: else the int32 sums of later blocks are held beside their operands
            asm volatile("" : "+v"(x));
            v[i][r][j] = x;
            u[r] = fmaf(x, kcap, -kCapSub) * fabsf(gs[r]);
          } else {
            x = gelu_exact(x, tb) * gs[r];
            asm volatile("" : "+v"(x));
            v[i][r][j] = x;
            u[r] = fabsf(x);
          }
        }
        // (ignores a NaN, as `if a > max_abs`)
        float m = fmaxf(fmaxf(fmaxf(kFast ? cap0 : 0.0f, u[0]), fmaxf(u[1], u[2])), u[3]);
        asm volatile("" : "+v"(m));
        bm[i][j] = m;
        mx[i] = fmaxf(mx[i], m);
      }
    }
    opaque_ids();
    // ---- row maxima: over this wave's columns, then over the waves through LDS ----
#pragma unroll
    for (int i = 0; i < NR; i++) {
      mx[i] = fmaxf(mx[i], __shfl_xor(mx[i], 16, 64));
      mx[i] = fmaxf(mx[i], __shfl_xor(mx[i], 32, 64));
      if (fq == 0) sU[r0 + i * 16 + fr][wave] = mx[i];
    }
    __syncthreads();
    float M[NR], thr[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) {
      const float4* u4 = reinterpret_cast<const float4*>(&sU[r0 + i * 16 + fr][0]);
      const float4 a = u4[0], b = u4[1];
      const float U = fmaxf(fmaxf(fmaxf(a.x, a.y), fmaxf(a.z, a.w)), fmaxf(fmaxf(b.x, b.y), fmaxf(b.z, b.w)));
      M[i] = fmaxf(U, 1e-8f);  // max_abs starts at 1e-8 (src/simd_math.rs:1295-1312)
      thr[i] = kCandShare * U;
    }
    float gs_max = 0.0f;
    if constexpr (kFast) {
      gs_max = __uint_as_float(s_gmax);
      {  // first scan: candidates to the wave's list, then one gelu_exact for up to 64 of them
        // (two arrays: as pairs, every v would sit in a register pair of its own)
        float* lv = reinterpret_cast<float*>(sQ + r0 * kQPitch) + wave * 2 * kListCap;
        uint32_t* lid = reinterpret_cast<uint32_t*>(lv) + kListCap;
        int n = 0;  // (wave-uniform)
        bool full = false;
#pragma unroll 1
        for (int j = 0; j < kUpCB; j++) {
          const int col = (j * kWaves + wave) * 16 + fq * 4;
#pragma unroll
          for (int i = 0; i < NR; i++) {
            if (__builtin_amdgcn_ballot_w64(bm[i][j] >= thr[i]) == 0) continue;  // wave-uniform
            const v4f gs = *reinterpret_cast<const v4f*>(&sGs[col]);
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const float x = v[i][r][j];
              const bool c = fmaxf(fmaf(x, kcap, -kCapSub), kCapMin) * fabsf(gs[r]) >= thr[i];
              const uint64_t m = __builtin_amdgcn_ballot_w64(c);
              if (m == 0) continue;
              if (n + __builtin_popcountll(m) <= kListCap) {
                if (c) {
                  const int k = n + lanes_below(m);
                  lv[k] = x;
                  lid[k] = (uint32_t)(col + r) | (uint32_t)(r0 + i * 16 + fr) << 16;
                }
                n += __builtin_popcountll(m);
              } else {
                full = true;
              }
            }
          }
        }
        wave_lds_sync();
        for (int k = 0; k < n; k += 64) {
          const int e = min(k + lane, n - 1);
          const uint32_t id = lid[e];
          const float g = fabsf(gelu_exact(lv[e], tb) * sGs[id & 0xffffu]);
          if (k + lane < n && g > 0.0f) atomicMax(&sM[0][id >> 16], __float_as_uint(g));  // a NaN is ignored
        }
        if (lane == 0) {
          if (n > 0) atomicAdd(&sCnt[pp], n);
          if (full) s_full[pp] = 1;
        }
      }
      __syncthreads();
      bool open = s_full[pp] != 0;  // the same in every wave: each reads all rows' U and M1, which no longer change
#pragma unroll
      for (int i = 0; i < NR; i++) {
        M[i] = __uint_as_float(sM[0][r0 + i * 16 + fr]);
        open = open || !(M[i] >= thr[i] * (1.0f + 0x1p-20f));
      }
      if (__builtin_amdgcn_ballot_w64(open) != 0) {  // second scan
#pragma unroll 1
        for (int j = 0; j < kUpCB; j++) {
          const int col = (j * kWaves + wave) * 16 + fq * 4;
#pragma unroll
          for (int i = 0; i < NR; i++) {
            if (__builtin_amdgcn_ballot_w64(bm[i][j] >= M[i]) == 0) continue;
            v4f x = v4f{v[i][0][j], v[i][1][j], v[i][2][j], v[i][3][j]}, g = *reinterpret_cast<const v4f*>(&sGs[col]);
            float top = 0.0f;
#pragma unroll 1
            for (int r = 0; r < 4; r++) {  // element 0 evaluated, then the four rotated
              top = nanless_max(top, fabsf(gelu_exact(x[0], tb) * g[0]));
              x = v4f{x[1], x[2], x[3], x[0]};
              g = v4f{g[1], g[2], g[3], g[0]};
            }
            atomicMax(&sM[1][r0 + i * 16 + fr], __float_as_uint(top));
          }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NR; i++) M[i] = fmaxf(M[i], __uint_as_float(sM[1][r0 + i * 16 + fr]));
      }
      if (tid == 0 && sCnt[pp] > RP) atomicAdd(&g_ffn_repairs[1], (unsigned long long)NR);
    }
    // the next pass's first weight blocks, behind the GELUs
    if (kP > 1 && pp + 1 < kP) {
      load_w1(0, w1[0]);
      load_w1(1, w1[1]);
    }

    // ---- GELU and quantization into the LDS tile ----
    opaque_ids();
    if (wave == 0 && fq == 0) {
#pragma unroll
      for (int i = 0; i < NR; i++) sMax[r0 + i * 16 + fr] = M[i];  // for the epilogue
    }
    float inv[NR], lim[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) {
      inv[i] = 127.0f / M[i];
      lim[i] = fmaxf(0.5f - fmaf(gs_max * kQAbs, inv[i], 0x1p-24f), 0.0f);
    }
#pragma unroll
    for (int j = 0; j < kUpCB; j++) {
      // waves w and w + 4 share a SIMD; alternating their priority per column block
      // keeps them level, so neither waits long at the barrier after the loop
      if ((j ^ (wave >> 2)) & 1) __builtin_amdgcn_s_setprio(1);
      else __builtin_amdgcn_s_setprio(0);
      const int col = (j * kWaves + wave) * 16;
      uint32_t pk[NR];
      if constexpr (kFast) {
        const v4f gs = *reinterpret_cast<const v4f*>(&sGs[col + fq * 4]);
        bool bad[NR], any = false;
        constexpr int N = 4 * NR;
        float vv[N], x[N], t[N], d[N], gi[N];
#pragma unroll
        for (int k = 0; k < N; k++) vv[k] = v[k >> 2][k & 3][j];
        gelu_fast<N>(vv, kc, x);
        auto each = [&](auto f) {
#pragma unroll
          for (int k = 0; k < N; k++) f(k);
          __builtin_amdgcn_sched_barrier(0);
        };
        each([&](int k) { gi[k] = gs[k & 3] * inv[k >> 2]; });
        each([&](int k) { x[k] = x[k] * gi[k]; });
        each([&](int k) { t[k] = x[k] + 0x1.8p23f; });  // round to nearest: the low byte of t is q
        each([&](int k) { d[k] = t[k] - 0x1.8p23f; });
        each([&](int k) { d[k] = x[k] - d[k]; });
        each([&](int k) { d[k] = fmaf(fabsf(x[k]), kq, fabsf(d[k])); });
#pragma unroll
        for (int i = 0; i < NR; i++) {
          uint32_t worst = 0;
#pragma unroll
          for (int r = 0; r < 4; r++) worst = max(worst, __float_as_uint(d[4 * i + r]));  // (as u32: a NaN is the largest)
          auto tb4 = [&](int r) { return __float_as_uint(t[4 * i + r]); };
          pk[i] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(tb4(3), tb4(2), 0x0c0c0400u),
                                        __builtin_amdgcn_perm(tb4(1), tb4(0), 0x0c0c0400u), 0x05040100u);
          bad[i] = worst >= __float_as_uint(lim[i]);
          any = any || bad[i];
        }
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(any) != 0, 0)) {  // rare: the tiles' exact values
#pragma unroll
          for (int i = 0; i < NR; i++) {
            if (__builtin_amdgcn_ballot_w64(bad[i]) == 0) continue;
            if (lane == 0) atomicAdd(&g_ffn_repairs[0], 1ull);
            v4f x = v4f{v[i][0][j], v[i][1][j], v[i][2][j], v[i][3][j]}, g = gs;
            uint32_t w = 0;
#pragma unroll 1
            for (int r = 0; r < 4; r++) {  // element 0 evaluated, then the four rotated
              const int q = qround_bounded(gelu_exact(x[0], tb) * g[0] * inv[i]);
              w = (w >> 8) | ((uint32_t)q << 24);
              x = v4f{x[1], x[2], x[3], x[0]};
              g = v4f{g[1], g[2], g[3], g[0]};
            }
            pk[i] = w;
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < NR; i++)
          pk[i] = pack4(qround_bounded(v[i][0][j] * inv[i]), qround_bounded(v[i][1][j] * inv[i]),
                        qround_bounded(v[i][2][j] * inv[i]), qround_bounded(v[i][3][j] * inv[i]));
      }
#pragma unroll
      for (int i = 0; i < NR; i++)
        *reinterpret_cast<uint32_t*>(&sQ[(r0 + i * 16 + fr) * kQPitch + col + fq * 4]) = pk[i];
    }
    __builtin_amdgcn_s_setprio(0);
  }

  // ---- FFN-down: acc2[i][n] = rows 16i.., columns 48 w + 16 n.., K = 1536 ----
  opaque_ids();
  constexpr int kRB = NR * kP;  // 16-row blocks
  const int dcol = wave * kDnCB * 16;
  auto load_w2 = [&](int kt, v4i (&dst)[kDnCB]) {
    int base = (kt * (kH / 16)) * 1024 + dcol * 64;
    asm volatile("" : "+s"(base));
#pragma unroll
    for (int n = 0; n < kDnCB; n++) dst[n] = weight_load(w2r, lane16, base + n * 1024);
  };
  v4i ring[kRing][kDnCB];
#pragma unroll
  for (int s = 0; s < kRing; s++) load_w2(s, ring[s]);
  // the epilogue's operands, loaded now so that the residual's HBM latency hides behind FFN-down
  v4f res[kRB][kDnCB];
#pragma unroll
  for (int i = 0; i < kRB; i++)
#pragma unroll
    for (int n = 0; n < kDnCB; n++)
      res[i][n] = __builtin_nontemporal_load(
          reinterpret_cast<const v4f*>(p.res + (size_t)min(m0 + i * 16 + fr, p.M - 1) * kH + dcol + n * 16 + fq * 4));
  // kLn: thread t takes float4 columns t % 32 + 32 i of row t / 32
  constexpr int kLnPitch = 388;  // floats
  static_assert(16 * kLnPitch * 4 <= 16 * kQPitch, "the LayerNorm's rows fit in sQ");
  v4f lg[3], lb[3], lsm[3];
  if constexpr (kLn) {
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int c = ((tid & 31) + 32 * i) * 4;
      lg[i] = *reinterpret_cast<const v4f*>(ln.gamma + c);
      lb[i] = *reinterpret_cast<const v4f*>(ln.beta + c);
      lsm[i] = *reinterpret_cast<const v4f*>(ln.smooth + c);
    }
  }
  __syncthreads();  // sQ complete
  v4i acc2[kRB][kDnCB];
#pragma unroll
  for (int i = 0; i < kRB; i++)
#pragma unroll
    for (int n = 0; n < kDnCB; n++) acc2[i][n] = v4i{0, 0, 0, 0};
#pragma unroll
  for (int kt = 0; kt < kDnSteps; kt++) {  // fully unrolled ring of kRing steps
    v4i q[kRB];
#pragma unroll
    for (int i = 0; i < kRB; i++) q[i] = *reinterpret_cast<const v4i*>(&sQ[(i * 16 + fr) * kQPitch + kt * 64 + fq * 16]);
#pragma unroll
    for (int n = 0; n < kDnCB; n++)
#pragma unroll
      for (int i = 0; i < kRB; i++)
        acc2[i][n] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ring[kt % kRing][n], q[i], acc2[i][n], 0, 0, 0);
    if (kt + kRing < kDnSteps) load_w2(kt + kRing, ring[kt % kRing]);
  }

  // ---- epilogue: out = fma(f32(acc), s * ws2, b2 + res), whole float4s per lane ----
  v4f ws2[kDnCB], b2[kDnCB];
#pragma unroll
  for (int n = 0; n < kDnCB; n++) {
    ws2[n] = *reinterpret_cast<const v4f*>(p.w2_scale + dcol + n * 16 + fq * 4);
    b2[n] = *reinterpret_cast<const v4f*>(p.b2 + dcol + n * 16 + fq * 4);
  }
  float* T = reinterpret_cast<float*>(sQ);  // kLn: the output rows [16][kLnPitch]
  if constexpr (kLn) __syncthreads();       // every wave's FFN-down is done with sQ
#pragma unroll
  for (int i = 0; i < kRB; i++) {
    const float s = sMax[i * 16 + fr] / 127.0f;  // scale = max_abs / 127.0
    const int row = m0 + i * 16 + fr;
#pragma unroll
    for (int n = 0; n < kDnCB; n++) {
      v4f o;
#pragma unroll
      for (int r = 0; r < 4; r++) o[r] = fmaf((float)acc2[i][n][r], s * ws2[n][r], b2[n][r] + res[i][n][r]);
      if (row < p.M)  // streaming store: keeps the weights resident in L2
        __builtin_nontemporal_store(o, reinterpret_cast<v4f*>(p.out + (size_t)row * kH + dcol + n * 16 + fq * 4));
      if constexpr (kLn) *reinterpret_cast<v4f*>(&T[fr * kLnPitch + dcol + n * 16 + fq * 4]) = o;
    }
  }
  if constexpr (kLn) {
    __shared__ float s_stat[2][16];
    const int rr = tid >> 5, sub = tid & 31, row = m0 + rr;
    __syncthreads();
    v4f x[3];
#pragma unroll
    for (int i = 0; i < 3; i++) x[i] = *reinterpret_cast<const v4f*>(&T[rr * kLnPitch + (sub + 32 * i) * 4]);
    if (tid < 16) s_stat[0][tid] = lds_row_sum(&T[tid * kLnPitch], [](float v) { return v; }) / 384.0f;
    __syncthreads();  // (and every read of the rows is done)
    const float mean = s_stat[0][rr];
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const v4f d = x[i] - mean;
      *reinterpret_cast<v4f*>(&T[rr * kLnPitch + (sub + 32 * i) * 4]) = d * d;
    }
    __syncthreads();
    if (tid < 16)
      s_stat[1][tid] = 1.0f / sqrtf(lds_row_sum(&T[tid * kLnPitch], [](float v) { return v; }) / 384.0f + 1e-12f);
    __syncthreads();
    const float rstd = s_stat[1][rr];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const v4f y = (x[i] - mean) * rstd * lg[i] + lb[i];
      if (ln.dst && row < p.M) *reinterpret_cast<v4f*>(ln.dst + (size_t)row * kH + (sub + 32 * i) * 4) = y;
      x[i] = y * lsm[i];
#pragma unroll
      for (int r = 0; r < 4; r++) amax = nanless_max(amax, fabsf(x[i][r]));
    }
    amax = lanes32_max(amax);  // amax is never NaN: fmaxf is nanless_max here
    const float max_abs = nanless_max(1e-8f, amax), inv_scale = 127.0f / max_abs;
    if (row < p.M) {
#pragma unroll
      for (int i = 0; i < 3; i++)
        *reinterpret_cast<uint32_t*>(ln.q + (size_t)row * kH + (sub + 32 * i) * 4) =
            pack4(qround(x[i][0] * inv_scale), qround(x[i][1] * inv_scale), qround(x[i][2] * inv_scale),
                  qround(x[i][3] * inv_scale));
      if (sub == 0) {
        ln.scale[row] = max_abs / 127.0f;
        if (ln.stats) ln.stats[row] = make_float2(mean, rstd);
        if (ln.rowmax_init) ln.rowmax_init[row] = __float_as_uint(1e-8f);
      }
    }
  }
}

static int g_ffn_rows = 0;  // 0 by the batch, 16, 32, 64, or -m: the mixed plan with m rows first (test hook)
void set_ffn_rows(int rows) { g_ffn_rows = rows; }
int ffn_rows() { return g_ffn_rows; }
static bool g_ffn_exact_gelu = false;  // test hook: the exact-GELU kernel for every launch
void set_ffn_exact_gelu(bool exact) { g_ffn_exact_gelu = exact; }
bool ffn_exact_gelu() { return g_ffn_exact_gelu; }

// The certification of gelu_fast (device_common.hpp) over all 2^32 f32 inputs
// against gelu_exact, both as ffn_kernel evaluates them (gelu_fast on 8 values at
// once, its 32- and 64-row workgroups, and on 4, its 16-row ones).  Counters: [0]
// inputs breaking the certified bound (G' NaN only for NaN / +-inf v, else
// gelu_exact finite and |G - G'| <= kGeluFastRel |G'| + kGeluFastAbs, in f64) or
// whose two G' differ in a bit, [1] NaN G'
// for another v, [2] v >= kGeluSatPos with gelu_exact(v) != v, [3] finite
// v <= kGeluSatNeg with gelu_exact(v) != 0, [4] inputs breaking the bound with
// half its absolute term (a too-tight bound must fail: the check is not
// vacuous), [5] inputs checked.
__global__ __launch_bounds__(256) void gelu_fast_certify_kernel(unsigned long long* out, uint32_t base) {
  const ExpTab tb = exp_tab_regs();
  const uint32_t i0 = base + (blockIdx.x * 256u + threadIdx.x) * 16u;
  unsigned c[6] = {0, 0, 0, 0, 0, 0};
  float kc = kGeluFastK;
  asm volatile("" : "+v"(kc));
  float v8[8], g8[8], v4[4], g4[4];
#pragma unroll
  for (int u = 0; u < 16; u++) {
    if (u % 8 == 0) {
#pragma unroll
      for (int k = 0; k < 8; k++) v8[k] = __uint_as_float(i0 + (uint32_t)(u + k));
      gelu_fast<8>(v8, kc, g8);
    }
    if (u % 4 == 0) {
#pragma unroll
      for (int k = 0; k < 4; k++) v4[k] = __uint_as_float(i0 + (uint32_t)(u + k));
      gelu_fast<4>(v4, kc, g4);
    }
    const float v = v8[u % 8], G = gelu_exact(v, tb), Gp = g8[u % 8];
    if (__float_as_uint(g4[u % 4]) != __float_as_uint(Gp)) c[0]++;
    const bool special = __builtin_isnan(v) || __builtin_isinf(v);
    if (__builtin_isnan(Gp)) {
      if (!special) c[1]++;
    } else {
      const double d = fabs((double)G - (double)Gp), a = fabs((double)Gp);
      const bool finite = !__builtin_isnan(G) && !__builtin_isinf(G);
      if (special || !finite || !(d <= (double)kGeluFastRel * a + (double)kGeluFastAbs)) c[0]++;
      if (finite && !(d <= (double)kGeluFastRel * a + 0.5 * (double)kGeluFastAbs)) c[4]++;
    }
    if (v >= kGeluSatPos && G != v) c[2]++;
    if (v <= kGeluSatNeg && v >= -3.40282347e38f && G != 0.0f) c[3]++;
    c[5]++;
  }
#pragma unroll
  for (int k = 0; k < 6; k++) {  // wave sums, one atomic per wave and counter
    unsigned long long t = c[k];
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    if ((threadIdx.x & 63) == 0 && t) atomicAdd(&out[k], t);
  }
}

hipError_t gelu_fast_certify(unsigned long long* out_dev, hipStream_t st) {
  hipError_t e = hipMemsetAsync(out_dev, 0, 6 * sizeof(unsigned long long), st);
  for (uint32_t c = 0; c < 16 && e == hipSuccess; c++) {  // 2^28 inputs per launch: 65536 x 256 threads x 16
    hipLaunchKernelGGL(gelu_fast_certify_kernel, dim3(65536), dim3(256), 0, st, out_dev, c << 28);
    e = hipGetLastError();
  }
  return e;
}

hipError_t ffn_repair_counts(unsigned long long counts[2], bool reset) {
  hipError_t e = hipMemcpyFromSymbol(counts, HIP_SYMBOL(g_ffn_repairs), sizeof(unsigned long long) * 2, 0,
                                     hipMemcpyDeviceToHost);
  if (e == hipSuccess && reset) {
    const unsigned long long zero[2] = {0, 0};
    e = hipMemcpyToSymbol(HIP_SYMBOL(g_ffn_repairs), zero, sizeof(zero), 0, hipMemcpyHostToDevice);
  }
  return e;
}

template <int NR, int kP, bool kLn = false>
static void launch_ffn_rows(const FfnArgs& p, hipStream_t st, const LnArgs& ln = LnArgs{}) {
  constexpr int R = 16 * NR * kP;
  const dim3 grid((unsigned)((p.M + R - 1) / R));
  if (p.fast_gelu && !g_ffn_exact_gelu)
    hipLaunchKernelGGL((ffn_kernel<NR, kP, true, kLn>), grid, dim3(kThreads), 0, st, p, ln);
  else
    hipLaunchKernelGGL((ffn_kernel<NR, kP, false, kLn>), grid, dim3(kThreads), 0, st, p, ln);
}
static void launch_ffn_tile(const FfnArgs& p, int rows, hipStream_t st) {
  if (rows == 16) launch_ffn_rows<1, 1>(p, st);
  else if (rows == 32) launch_ffn_rows<2, 1>(p, st);
  else launch_ffn_rows<2, 2>(p, st);
}

// With one workgroup per CU a launch takes about as many workgroup times as it
// has rounds of workgroups over the CUs.  Times in hundredths of a 16-row
// workgroup's (18 to 21 us): a 32-row one 140 (25 to 29 us), a 64-row one 255 (54
// us for one round, 107 for two, 900 for 18).  The plan is the cheapest of: all
// rows in 16-, 32- or 64-row workgroups, or k full rounds of 64-row ones and then
// a second launch for the remaining rows, whose last, partial round then holds
// short workgroups (68,270 rows: 233 us, against 245 in 64-row and 251 in 32-row
// workgroups).
struct FfnPlan {
  int tile;   // rows per workgroup, all rows (m64 = 0)
  long m64;   // the mixed plan: rows in 64-row workgroups,
  int tail;   // rows per workgroup of the others
};
static FfnPlan ffn_plan(const FfnArgs& p) {
  const long cus = device_cu_count();
  auto rounds = [&](long rows, long tile) { return ((rows + tile - 1) / tile + cus - 1) / cus; };
  constexpr long kT16 = 100, kT32 = 140, kT64 = 255, kFirst64 = 15, kLaunch = 10;
  auto short_tile = [&](long rows) { return kT16 * rounds(rows, 16) <= kT32 * rounds(rows, 32) ? 16 : 32; };
  auto short_time = [&](long rows) { return std::min(kT16 * rounds(rows, 16), kT32 * rounds(rows, 32)); };
  int tile = short_tile(p.M), tail = 0;
  long best = short_time(p.M), m64 = 0;
  if (kT64 * rounds(p.M, 64) + kFirst64 < best) best = kT64 * rounds(p.M, 64) + kFirst64, tile = 64;
  for (long k = 1; 64 * cus * k < p.M; k++) {
    const long rem = p.M - 64 * cus * k, t = kT64 * k + kFirst64 + short_time(rem) + kLaunch;
    if (t < best) best = t, m64 = 64 * cus * k, tail = short_tile(rem);
  }
  if (g_ffn_rows > 0) tile = g_ffn_rows, m64 = 0;
  if (g_ffn_rows < 0) {  // forced mixed plan (m64 rows in 64-row workgroups, when there are more)
    m64 = -g_ffn_rows < p.M ? -g_ffn_rows : 0;
    tile = 64, tail = 32;
  }
  return {tile, m64, tail};
}

bool launch_ffn(const FfnArgs& p, hipStream_t st, hipStream_t side, hipEvent_t fork, hipEvent_t join, const LnArgs* ln) {
  if (p.M <= 0) return false;
  const FfnPlan plan = ffn_plan(p);
  const long m64 = plan.m64;
  const int tail = plan.tail;
  if (m64 == 0) {
    // 16-row workgroups run in one round (ffn_plan), so all end on the LayerNorm's in-order sums together
    const bool fused = ln && plan.tile == 16;
    if (fused) launch_ffn_rows<1, 1, true>(p, st, *ln);
    else launch_ffn_tile(p, plan.tile, st);
    return fused;
  }
  FfnArgs a = p, b = p;
  a.M = (int)m64;
  b.M = (int)(p.M - m64);
  b.A = p.A + m64 * kH;
  b.a_scale = p.a_scale + m64;
  b.res = p.res + m64 * kH;
  b.out = p.out + m64 * kH;
  if (side && fork && join) {
    (void)hipEventRecord(fork, st);
    (void)hipStreamWaitEvent(side, fork, 0);
    launch_ffn_tile(b, tail, side);
    (void)hipEventRecord(join, side);
    launch_ffn_tile(a, 64, st);
    (void)hipStreamWaitEvent(st, join, 0);
  } else {
    launch_ffn_tile(a, 64, st);
    launch_ffn_tile(b, tail, st);
  }
  return false;
}

}  // namespace aek
