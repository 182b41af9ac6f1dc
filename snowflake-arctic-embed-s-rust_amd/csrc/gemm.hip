// gemm.hip -- W8A8 int8 MFMA GEMM for gfx950 with the reference's fused epilogue.
//
//   out[m,n] = fma(f32(sum_k a[m,k]*w[n,k]), sa[m]*ws[n], bias[n] (+ res[m,n]))
//
// (gemm_scalar_fused, reference src/gemm.rs:2000-2029: integer accumulation,
// then one f32 conversion, one product sa*ws, one sum bias+res and one fma.)
//
// Tiling: one workgroup = 4 waves = 64 rows x 384 columns; wave w owns columns
// [w*96, w*96+96) as 4 x 6 tiles of v_mfma_i32_16x16x64_i8 (96 accumulator
// VGPRs), K step 64.
//  * A (64 x 64 int8 per step) is staged through LDS and shared by the 4 waves.
//    Its global loads run two K steps ahead in registers; f32 A (the
//    quantize-on-load variants) is converted to int8 only when it is written
//    to LDS, so the load latency overlaps two steps of MFMA work.
//  * Each wave streams its B fragments straight from global memory: W is
//    pre-swizzled at load time into MFMA fragment order [K/64][N/16][64][16],
//    so every fragment load is one coalesced 1 KiB transaction (one step ahead).
//  * The epilogue stages each 16-row block of int32 accumulators through LDS
//    and then walks whole rows with float4 accesses, so outputs and residuals
//    move as full 128-byte lines.
// For the N = 384 GEMMs (attn_out, FFN-down) one workgroup spans the whole row,
// so f32 A rows are read and quantized exactly once.
//
// MFMA operand layout (16x16x64 i8): lane l supplies row (l%16) of A and column
// (l%16) of B, 16 k-values from k-group (l/16); A and B share that k order, so the
// integer sum is exact.  Output: lane l, register r holds D[4*(l/16)+r][l%16].
#include <hip/hip_runtime.h>

#include <atomic>

#include <algorithm>
#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"

namespace aek {

constexpr int kBM = 64;      // rows per workgroup
constexpr int kAPitch = 80;  // LDS row pitch of the A tile (bytes): conflict-free fragment reads
constexpr int kEPitch = 100; // LDS row pitch of the epilogue staging tile (words)

template <int AM>
struct ARegs;
template <>
struct ARegs<kAI8> {
  v4i v;
};
template <int AM>
struct ARegs {
  float4 v[4];
};

// NW = columns per wave: 96 (workgroup = 384 columns, 2 waves/SIMD) or 48
// (192 columns, 48 accumulator VGPRs: 4 waves/SIMD for int8 A, 3 for f32 A,
// whose two-step register prefetch of A is four times larger).
template <int AM, int EM, int NW>
__global__ __launch_bounds__(256, NW == 96 ? 2 : (AM == kAI8 ? 4 : 3)) void gemm_w8a8_kernel(GemmArgs p) {
  constexpr int kWaveN = NW, kBN = 4 * NW, kCB = NW / 16;
  constexpr int kF4 = NW / 4;  // float4 columns of one wave row
  __shared__ __attribute__((aligned(16))) int8_t sA[2][kBM * kAPitch];
  __shared__ __attribute__((aligned(16))) int sE[4][16 * kEPitch];  // per-wave epilogue staging
  __shared__ uint32_t sRowMax[4][16];
  __shared__ __attribute__((aligned(16))) float sEpSa[kBM], sEpWs[kBN], sEpB[kBN];  // epilogue operands
  __shared__ uint64_t s_tab[EM == kEpiGelu ? 32 : 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // 1-D grid of (row tile, column tile) items.  p.col_fast: column tile fastest,
  // numbered XCD-contiguously, so the column tiles of one row tile run back to
  // back on one XCD and their A rows come from HBM once (f32 A always; int8 A
  // when A is too large to stay in the Infinity Cache between column tiles).
  // Otherwise row tile fastest: neighbouring workgroups share W columns.
  const int nt = p.N / kBN, mt = (p.M + kBM - 1) / kBM, nbase = mt * nt;
  const int bid = blockIdx.x;
  int m0, n0;
  if (!p.col_fast) {
    m0 = (bid % mt) * kBM;
    n0 = (bid / mt) * kBN;
  } else {
    const int item = xcd_contiguous(bid, nbase);
    m0 = (item / nt) * kBM;
    n0 = (item % nt) * kBN;
  }
  const int KB = 0, KT = p.K >> 6;  // K steps
  const int NB = p.N >> 4;  // 16-column fragments per K step in the swizzled W
  if constexpr (EM == kEpiGelu) exp_tab_fill(s_tab, tid);  // ordered before the epilogue by the K loop's barriers
  const ExpTabLds tb{s_tab};  // the epilogue loop below is wave-uniform

  // A loader: 4 threads per row, 16 k-values each
  const int lrow = tid >> 2, lpart = tid & 3;
  const int arow = min(m0 + lrow, p.M - 1);
  float a_inv = 0.0f;
  if (AM != kAI8) a_inv = 127.0f / __uint_as_float(p.a_rowmax[arow]);  // inv_scale = 127.0 / max_abs
  // epilogue operands, loaded now and put in LDS after the K loop: thread t < kBM
  // the scale of row m0 + t, then the w_scale and the bias float4s of the
  // workgroup's kBN columns
  float4 ep_reg = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (tid < kBM) {
    const int r = min(m0 + tid, p.M - 1);
    ep_reg.x = AM == kAI8 ? p.a_scale[r] : __uint_as_float(p.a_rowmax[r]) / 127.0f;  // scale = max_abs / 127.0
  } else if (tid < kBM + kBN / 4) {
    ep_reg = reinterpret_cast<const float4*>(p.w_scale + n0)[tid - kBM];
  } else if (tid < kBM + kBN / 2) {
    ep_reg = reinterpret_cast<const float4*>(p.bias + n0)[tid - kBM - kBN / 4];
  }
  auto aload = [&](int kt, ARegs<AM>& r) {
    const int kb = (KB + kt) * 64 + lpart * 16;
    if constexpr (AM == kAI8) {
      r.v = *reinterpret_cast<const v4i*>(reinterpret_cast<const int8_t*>(p.A) + (size_t)arow * p.K + kb);
    } else {
      const float4* src = reinterpret_cast<const float4*>(reinterpret_cast<const float*>(p.A) + (size_t)arow * p.K + kb);
#pragma unroll
      for (int i = 0; i < 4; i++) r.v[i] = src[i];
    }
  };
  auto astore = [&](int kt, int buf, const ARegs<AM>& r) {
    v4i q;
    if constexpr (AM == kAI8) {
      q = r.v;
    } else {
      const int kb = (KB + kt) * 64 + lpart * 16;
      uint32_t w[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float4 x = r.v[i];
        if (AM == kAF32QSmooth) {  // (x * inv_smooth[j]) * inv_scale
          const float4 s = reinterpret_cast<const float4*>(p.a_smooth + kb)[i];
          x.x = x.x * s.x; x.y = x.y * s.y; x.z = x.z * s.z; x.w = x.w * s.w;
        }
        w[i] = pack4(qround(x.x * a_inv), qround(x.y * a_inv), qround(x.z * a_inv), qround(x.w * a_inv));
      }
      q = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
    }
    *reinterpret_cast<v4i*>(&sA[buf][lrow * kAPitch + lpart * 16]) = q;
  };
  // B fragments of this wave for one K step
  const int cb0 = (n0 + wave * kWaveN) >> 4;
  const int8_t* wbase = p.w + (size_t)lane * 16;
  v4i bcur[kCB], bnext[kCB];
  auto bload = [&](int kt, v4i* dst) {
#pragma unroll
    for (int j = 0; j < kCB; j++)
      dst[j] = *reinterpret_cast<const v4i*>(wbase + ((size_t)(KB + kt) * NB + cb0 + j) * 1024);
  };

  v4i acc[4][kCB];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < kCB; j++) acc[i][j] = v4i{0, 0, 0, 0};

  ARegs<AM> r1, r2;  // A for steps kt+1 and kt+2
  {
    ARegs<AM> r0;
    aload(0, r0);
    if (KT > 1) aload(1, r1);
    bload(0, bcur);
    astore(0, 0, r0);
  }
  __syncthreads();
  const int fr = lane & 15, fk = (lane >> 4) * 16;
  for (int kt = 0; kt < KT; kt++) {
    const int buf = kt & 1;
    if (kt + 2 < KT) aload(kt + 2, r2);
    if (kt + 1 < KT) bload(kt + 1, bnext);
    v4i af[4];
#pragma unroll
    for (int i = 0; i < 4; i++) af[i] = *reinterpret_cast<const v4i*>(&sA[buf][(i * 16 + fr) * kAPitch + fk]);
#pragma unroll
    for (int j = 0; j < kCB; j++)
#pragma unroll
      for (int i = 0; i < 4; i++) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[i], bcur[j], acc[i][j], 0, 0, 0);
    if (kt + 1 < KT) astore(kt + 1, buf ^ 1, r1);
    __syncthreads();
    if (kt + 1 < KT) {
#pragma unroll
      for (int j = 0; j < kCB; j++) bcur[j] = bnext[j];
      r1 = r2;
    }
  }

  // epilogue, one 16-row block at a time through this wave's LDS tile:
  // accumulators -> sE[16][96] (int32), then lanes walk rows with float4s
  int* E = sE[wave];
  const int col0 = n0 + wave * kWaveN;  // first column of this wave
  // Epilogue operands.  The row scales and the w_scale / bias columns of this
  // workgroup, loaded at the start (ep_reg), are in LDS (sEp*) by now.  Lane
  // (k, idx = lane + 64k) covers block row idx / kF4 and float4 column idx % kF4
  // of every 16-row block; with f32 A (registers to spare once the K loop is
  // done) the residual float4s of block i + 1 are loaded while block i is
  // processed, otherwise each block loads its own.
  constexpr bool kPre = AM != kAI8;
  constexpr int kEk = kF4 / 4;  // float4s per lane and block
  float4 resv[2][kPre ? kEk : 1];
  auto load_res = [&](int i, int k) {
    const int row = min(m0 + i * 16 + (lane + 64 * k) / kF4, p.M - 1);
    const int col = col0 + ((lane + 64 * k) % kF4) * 4;
    const v4i r4i = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(p.res + (size_t)row * p.N + col));
    return make_float4(__int_as_float(r4i.x), __int_as_float(r4i.y), __int_as_float(r4i.z), __int_as_float(r4i.w));
  };
  if constexpr (kPre) {
    if (p.res) {
#pragma unroll
      for (int k = 0; k < kEk; k++) resv[0][k] = load_res(0, k);
    }
  }
  if (tid < kBM) sEpSa[tid] = ep_reg.x;
  else if (tid < kBM + kBN / 4) reinterpret_cast<float4*>(sEpWs)[tid - kBM] = ep_reg;
  else if (tid < kBM + kBN / 2) reinterpret_cast<float4*>(sEpB)[tid - kBM - kBN / 4] = ep_reg;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; i++) {
#pragma unroll
    for (int j = 0; j < kCB; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) E[((lane >> 4) * 4 + r) * kEPitch + j * 16 + fr] = acc[i][j][r];
    if (EM == kEpiGelu && lane < 16) sRowMax[wave][lane] = 0u;
    wave_lds_sync();  // E and sRowMax are private to this wave
    if constexpr (kPre) {
      if (p.res && i + 1 < 4) {
#pragma unroll
        for (int k = 0; k < kEk; k++) resv[(i + 1) & 1][k] = load_res(i + 1, k);
      }
    }
#pragma unroll
    for (int k = 0; k < kEk; k++) {  // 16 rows x kF4 float4 over 64 lanes
      const int idx = lane + 64 * k, rr = idx / kF4, c4 = idx % kF4;
      const int row = m0 + i * 16 + rr;
      const bool ok = row < p.M;
      const int col = col0 + c4 * 4;
      const int4 a4 = *reinterpret_cast<const int4*>(&E[rr * kEPitch + c4 * 4]);
      const float sa = sEpSa[i * 16 + rr];
      const float4 ws4 = *reinterpret_cast<const float4*>(&sEpWs[wave * kWaveN + c4 * 4]);
      float4 b4 = *reinterpret_cast<const float4*>(&sEpB[wave * kWaveN + c4 * 4]);
      if (p.res) {
        const float4 r4 = kPre ? resv[i & 1][kPre ? k : 0] : load_res(i, k);
        b4.x = b4.x + r4.x; b4.y = b4.y + r4.y; b4.z = b4.z + r4.z; b4.w = b4.w + r4.w;
      }
      float4 v;
      v.x = fmaf((float)a4.x, sa * ws4.x, b4.x);
      v.y = fmaf((float)a4.y, sa * ws4.y, b4.y);
      v.z = fmaf((float)a4.z, sa * ws4.z, b4.z);
      v.w = fmaf((float)a4.w, sa * ws4.w, b4.w);
      if (EM == kEpiGelu) {
        const float4 g4 = *reinterpret_cast<const float4*>(p.g_smooth + col);
        v.x = gelu_exact(v.x, tb) * g4.x;
        v.y = gelu_exact(v.y, tb) * g4.y;
        v.z = gelu_exact(v.z, tb) * g4.z;
        v.w = gelu_exact(v.w, tb) * g4.w;
        float gm = nanless_max(nanless_max(fabsf(v.x), fabsf(v.y)), nanless_max(fabsf(v.z), fabsf(v.w)));
        atomicMax(&sRowMax[wave][rr], __float_as_uint(gm));  // non-negative f32 bits order like u32
      }
      if (ok) *reinterpret_cast<float4*>(p.out + (size_t)row * p.N + col) = v;
    }
    wave_lds_sync();
    if (EM == kEpiGelu && lane < 16) {
      const int row = m0 + i * 16 + lane;
      if (row < p.M) atomicMax(&p.g_rowmax[row], sRowMax[wave][lane]);
    }
  }
}

// ---------------------------------------------------------------------------
// int8 A, K = 384, f32 epilogue without residual, many rows (the QKV GEMM):
// A-stationary.  A workgroup of 4 waves stages its A tile (16 RB rows x 384
// int8) in LDS once and walks every 192-column tile of N with it, so A leaves
// HBM once instead of once per column tile.  Each column tile's W fragments (6 K steps x
// 3 per wave) stream from L2 into registers; the next tile's are issued into the
// same registers once this tile's MFMAs are done, before its epilogue.  The
// arithmetic is gemm_w8a8_kernel's.
// ---------------------------------------------------------------------------
constexpr int kAsPitch = 384 + 16;  // LDS bytes per A row: conflict-free fragment reads

template <int RB>
__global__ __launch_bounds__(256, 2) void gemm_astat_kernel(GemmArgs p) {
  constexpr int kCB = 3, kF4 = 12, kEk = 3;  // 48 columns per wave
  constexpr int kRows = 16 * RB, kChunks = kRows * 24, kLd = (kChunks + 255) / 256;  // A tile: 16-byte chunks
  __shared__ __attribute__((aligned(16))) int8_t sA[kRows * kAsPitch];
  __shared__ __attribute__((aligned(16))) int sE[4][16 * kEPitch];
  __shared__ float sEpSa[kRows];
  __shared__ __attribute__((aligned(16))) float sWs[2][192], sB[2][192];  // w_scale / bias of column tiles c, c + 1
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int fr = lane & 15, fk = (lane >> 4) * 16;
  // row tiles last to first: the rows written last (still in the Infinity Cache
  // when the next kernel starts) are the batch's first, which attention reads first
  const int m0 = (gridDim.x - 1 - blockIdx.x) * kRows, nt = p.N / 192, NB = p.N >> 4;
  const int8_t* A = reinterpret_cast<const int8_t*>(p.A);
  // the A tile: chunk c = tid + 256 i of 16 bytes is row c / 24, k 16 (c % 24)
  v4i ach[kLd];
#pragma unroll
  for (int i = 0; i < kLd; i++) {
    const int c = min(tid + 256 * i, kChunks - 1);
    ach[i] = *reinterpret_cast<const v4i*>(A + (size_t)min(m0 + c / 24, p.M - 1) * 384 + (c % 24) * 16);
  }
  const float sa_t = tid < kRows ? p.a_scale[min(m0 + tid, p.M - 1)] : 0.0f;
  // W fragments of column tile c for this wave; the tile's w_scale / bias go to
  // LDS (threads 0-47: w_scale float4s, 48-95: bias float4s)
  const int8_t* wbase = p.w + (size_t)lane * 16;
  v4i bf[6][kCB];
  auto wload = [&](int c) {
    const int cb0 = (c * 192 + wave * 48) >> 4;
#pragma unroll
    for (int kt = 0; kt < 6; kt++)
#pragma unroll
      for (int j = 0; j < kCB; j++)
        bf[kt][j] = *reinterpret_cast<const v4i*>(wbase + ((size_t)kt * NB + cb0 + j) * 1024);
  };
  auto eload = [&](int c) {  // returns this thread's float4 (threads < 96)
    if (tid < 48) return reinterpret_cast<const float4*>(p.w_scale + c * 192)[tid];
    if (tid < 96) return reinterpret_cast<const float4*>(p.bias + c * 192)[tid - 48];
    return make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  };
  auto estore = [&](int buf, const float4& v) {
    if (tid < 48) reinterpret_cast<float4*>(sWs[buf])[tid] = v;
    else if (tid < 96) reinterpret_cast<float4*>(sB[buf])[tid - 48] = v;
  };
  wload(0);
  estore(0, eload(0));
#pragma unroll
  for (int i = 0; i < kLd; i++) {
    const int c = tid + 256 * i;
    if (kChunks % 256 == 0 || c < kChunks) *reinterpret_cast<v4i*>(&sA[(c / 24) * kAsPitch + (c % 24) * 16]) = ach[i];
  }
  if (tid < kRows) sEpSa[tid] = sa_t;
  __syncthreads();

  int* E = sE[wave];
  for (int c = 0; c < nt; c++) {  // workgroup-uniform
    v4i acc[RB][kCB];
#pragma unroll
    for (int i = 0; i < RB; i++)
#pragma unroll
      for (int j = 0; j < kCB; j++) acc[i][j] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int kt = 0; kt < 6; kt++) {
      v4i af[RB];
#pragma unroll
      for (int i = 0; i < RB; i++) af[i] = *reinterpret_cast<const v4i*>(&sA[(i * 16 + fr) * kAsPitch + kt * 64 + fk]);
#pragma unroll
      for (int j = 0; j < kCB; j++)
#pragma unroll
        for (int i = 0; i < RB; i++) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[i], bf[kt][j], acc[i][j], 0, 0, 0);
    }
    float4 en = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (c + 1 < nt) {  // the next tile's operands, into the registers just released
      wload(c + 1);
      en = eload(c + 1);
    }
    const float* ws = sWs[c & 1];
    const float* bs = sB[c & 1];
    // epilogue, one 16-row block at a time through this wave's LDS tile
    const int col0 = c * 192 + wave * 48;
#pragma unroll
    for (int i = 0; i < RB; i++) {
#pragma unroll
      for (int j = 0; j < kCB; j++)
#pragma unroll
        for (int r = 0; r < 4; r++) E[((lane >> 4) * 4 + r) * kEPitch + j * 16 + fr] = acc[i][j][r];
      wave_lds_sync();
#pragma unroll
      for (int k = 0; k < kEk; k++) {
        const int idx = lane + 64 * k, rr = idx / kF4, c4 = idx % kF4;
        const int row = m0 + i * 16 + rr;
        const int4 a4 = *reinterpret_cast<const int4*>(&E[rr * kEPitch + c4 * 4]);
        const float sa = sEpSa[i * 16 + rr];
        const float4 w4 = *reinterpret_cast<const float4*>(&ws[wave * 48 + c4 * 4]);
        const float4 b4 = *reinterpret_cast<const float4*>(&bs[wave * 48 + c4 * 4]);
        float4 v;
        v.x = fmaf((float)a4.x, sa * w4.x, b4.x);
        v.y = fmaf((float)a4.y, sa * w4.y, b4.y);
        v.z = fmaf((float)a4.z, sa * w4.z, b4.z);
        v.w = fmaf((float)a4.w, sa * w4.w, b4.w);
        if (row < p.M) {
          float4* dst = reinterpret_cast<float4*>(p.out + (size_t)row * p.N + col0 + c4 * 4);
          if (col0 < p.stream_cols)  // wave-uniform
            __builtin_nontemporal_store(v4i{__float_as_int(v.x), __float_as_int(v.y), __float_as_int(v.z),
                                            __float_as_int(v.w)},
                                        reinterpret_cast<v4i*>(dst));
          else
            *dst = v;
        }
      }
      wave_lds_sync();
    }
    if (c + 1 < nt) estore((c + 1) & 1, en);
    __syncthreads();  // tile c + 1's w_scale / bias are in LDS; tile c's are no longer read
  }
}

// ---------------------------------------------------------------------------
// Many rows, N = K = 384, f32 A quantized on load with smoothing, residual, and
// the LayerNorm + SmoothQuant of the output rows: the attention output GEMM and
// LN1 (reference src/model.rs:695-724: smooth_quantize_row of ctx,
// gemm_int8_fused(attn_out, residual hidden), then layernorm_smooth_quantize_row,
// src/simd_math.rs:208-247).
// A workgroup of 4 or 8 waves owns 32 complete rows (wave w: its 96 or 48 columns),
// so the GEMM's output rows stay in LDS for the LayerNorm instead of going to
// HBM and back.  The arithmetic is gemm_w8a8_kernel's kAF32QSmooth / kEpiF32
// and ln_quant_kernel's, in the same order.  ln.dst may alias p.res: a
// workgroup reads its rows' residuals before it writes their LayerNorm.
// ---------------------------------------------------------------------------
constexpr int kLrRows = 32;
constexpr int kLrPitch = 388;  // LDS floats per row of the output tile

template <int kWaves>
__global__ __launch_bounds__(64 * kWaves, kWaves == 4 ? 3 : 4) void gemm_ln_rows_kernel(GemmArgs p, LnArgs ln) {
  constexpr int kCB = 24 / kWaves, kRing = 3, kSteps = 6, NB = 384 / 16;
  constexpr int kLpr = 64 * kWaves / kLrRows, kF4 = 96 / kLpr;  // lanes and float4s per lane of a row
  static_assert(kLrRows * kAsPitch <= kLrRows * kLrPitch * 4, "the A tile lives in the row tile's space");
  // the int8 A tile during the K loop; then the int32 accumulators, the f32
  // output rows and their squared deviations (3 workgroups fit a CU's LDS)
  __shared__ __attribute__((aligned(16))) float sT[kLrRows * kLrPitch];
  int8_t* sA = reinterpret_cast<int8_t*>(sT);
  __shared__ __attribute__((aligned(16))) float sWs[384], sB[384];
  __shared__ float s_mean[kLrRows], s_rstd[kLrRows];
  // res_stats: res_gamma / res_beta in the row tile's space past the A tile,
  // free until the accumulators are written (after the residual is formed)
  constexpr int kRgOff = 4096;  // floats (the A tile takes 32 x 400 bytes)
  static_assert(kLrRows * kAsPitch <= 4 * kRgOff && kRgOff + 768 <= kLrRows * kLrPitch, "residual LN parameters fit");
  float* sRg = sT + kRgOff;
  float* sRb = sRg + 384;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int fr = lane & 15, fq = lane >> 4;
  const int m0 = blockIdx.x * kLrRows;
  // row rl of the tile, float4 columns sub + kLpr i (i < kF4): the A quantization,
  // the epilogue and the LayerNorm all use this mapping
  const int rl = tid / kLpr, sub = tid % kLpr, row = m0 + rl;
  const bool valid = row < p.M;
  const int rrow = valid ? row : p.M - 1;

  // loads in the order of use (memory operations retire in order): the A row,
  // its max, the first kRing K steps of W, w_scale and bias; the residual row
  // after the K loop
  const float* xr = reinterpret_cast<const float*>(p.A) + (size_t)rrow * 384;
  float4 xa[kF4];
#pragma unroll
  for (int i = 0; i < kF4; i++) xa[i] = *reinterpret_cast<const float4*>(xr + (sub + kLpr * i) * 4);
  const float amax_a = __uint_as_float(p.a_rowmax[rrow]);
  const int8_t* wbase = p.w + (size_t)lane * 16;
  v4i ring[kRing][kCB];
  auto wload = [&](int kt, v4i (&dst)[kCB]) {
#pragma unroll
    for (int j = 0; j < kCB; j++)
      dst[j] = *reinterpret_cast<const v4i*>(wbase + ((size_t)kt * NB + wave * kCB + j) * 1024);
  };
#pragma unroll
  for (int u = 0; u < kRing; u++) wload(u, ring[u]);
  if (tid < 96) reinterpret_cast<float4*>(sWs)[tid] = reinterpret_cast<const float4*>(p.w_scale)[tid];
  else if (tid < 192) reinterpret_cast<float4*>(sB)[tid - 96] = reinterpret_cast<const float4*>(p.bias)[tid - 96];
  if (p.res_stats) {
    if (tid < 96) reinterpret_cast<float4*>(sRg)[tid] = reinterpret_cast<const float4*>(p.res_gamma)[tid];
    else if (tid < 192) reinterpret_cast<float4*>(sRb)[tid - 96] = reinterpret_cast<const float4*>(p.res_beta)[tid - 96];
  }

  {  // A quantized as kAF32QSmooth: q = round((x * inv_smooth[j]) * (127 / max_abs))
    const float inv = 127.0f / amax_a;  // inv_scale = 127.0 / max_abs
#pragma unroll
    for (int i = 0; i < kF4; i++) {
      const int c = (sub + kLpr * i) * 4;
      const float4 sm = *reinterpret_cast<const float4*>(p.a_smooth + c);
      const float4 v = make_float4(xa[i].x * sm.x, xa[i].y * sm.y, xa[i].z * sm.z, xa[i].w * sm.w);
      *reinterpret_cast<uint32_t*>(&sA[rl * kAsPitch + c]) =
          pack4(qround(v.x * inv), qround(v.y * inv), qround(v.z * inv), qround(v.w * inv));
    }
  }
  __syncthreads();

  v4i acc[2][kCB];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < kCB; j++) acc[i][j] = v4i{0, 0, 0, 0};
#pragma unroll
  for (int kt = 0; kt < kSteps; kt++) {
    v4i af[2];
#pragma unroll
    for (int i = 0; i < 2; i++) af[i] = *reinterpret_cast<const v4i*>(&sA[(i * 16 + fr) * kAsPitch + kt * 64 + fq * 16]);
#pragma unroll
    for (int j = 0; j < kCB; j++)
#pragma unroll
      for (int i = 0; i < 2; i++)
        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[i], ring[kt % kRing][j], acc[i][j], 0, 0, 0);
    if (kt + kRing < kSteps) wload(kt + kRing, ring[kt % kRing]);
  }
  float4 res[kF4];
  const float* rr = p.res + (size_t)rrow * 384;
#pragma unroll
  for (int i = 0; i < kF4; i++) {
    const v4i r = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(rr + (sub + kLpr * i) * 4));
    res[i] = make_float4(__int_as_float(r.x), __int_as_float(r.y), __int_as_float(r.z), __int_as_float(r.w));
  }
  if (p.res_stats) {  // the residual is the LayerNorm of these rows, recomputed as that LayerNorm forms it
    const float2 st = p.res_stats[rrow];
#pragma unroll
    for (int i = 0; i < kF4; i++) {
      const int c = (sub + kLpr * i) * 4;
      const float4 g = *reinterpret_cast<const float4*>(&sRg[c]);
      const float4 bt = *reinterpret_cast<const float4*>(&sRb[c]);
      res[i].x = (res[i].x - st.x) * st.y * g.x + bt.x;
      res[i].y = (res[i].y - st.x) * st.y * g.y + bt.y;
      res[i].z = (res[i].z - st.x) * st.y * g.z + bt.z;
      res[i].w = (res[i].w - st.x) * st.y * g.w + bt.w;
    }
  }
  __syncthreads();  // every wave's K loop is done with the A tile
  // accumulators into the row tile (lane: rows 16 i + 4 fq + r of column 16 kCB w + 16 j + fr)
  int* T32 = reinterpret_cast<int*>(sT);
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < kCB; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) T32[(i * 16 + fq * 4 + r) * kLrPitch + wave * 16 * kCB + j * 16 + fr] = acc[i][j][r];
  __syncthreads();

  // epilogue: out = fma(f32(acc), sa * ws, bias + res), kept in registers and in the tile
  const float sa = amax_a / 127.0f;  // scale = max_abs / 127.0
  float4 xv[kF4];
#pragma unroll
  for (int i = 0; i < kF4; i++) {
    const int c = (sub + kLpr * i) * 4;
    const int4 a4 = *reinterpret_cast<const int4*>(&T32[rl * kLrPitch + c]);
    const float4 ws4 = *reinterpret_cast<const float4*>(&sWs[c]);
    float4 b4 = *reinterpret_cast<const float4*>(&sB[c]);
    b4.x = b4.x + res[i].x; b4.y = b4.y + res[i].y; b4.z = b4.z + res[i].z; b4.w = b4.w + res[i].w;
    float4 v;
    v.x = fmaf((float)a4.x, sa * ws4.x, b4.x);
    v.y = fmaf((float)a4.y, sa * ws4.y, b4.y);
    v.z = fmaf((float)a4.z, sa * ws4.z, b4.z);
    v.w = fmaf((float)a4.w, sa * ws4.w, b4.w);
    xv[i] = v;
    *reinterpret_cast<float4*>(&sT[rl * kLrPitch + c]) = v;
  }
  __syncthreads();

  // LayerNorm + SmoothQuant of the 32 rows (as ln_quant_kernel): one lane per
  // row takes the in-order sums, kLpr threads per row the rest
  if (tid < kLrRows) s_mean[tid] = lds_row_sum(&sT[tid * kLrPitch], [](float v) { return v; }) / 384.0f;
  __syncthreads();
  const float mean = s_mean[rl];
#pragma unroll
  for (int i = 0; i < kF4; i++) {
    float4 d = xv[i];
    d.x = d.x - mean; d.y = d.y - mean; d.z = d.z - mean; d.w = d.w - mean;
    *reinterpret_cast<float4*>(&sT[rl * kLrPitch + (sub + kLpr * i) * 4]) = make_float4(d.x * d.x, d.y * d.y, d.z * d.z, d.w * d.w);
  }
  __syncthreads();
  if (tid < kLrRows) {
    const float var_sum = lds_row_sum(&sT[tid * kLrPitch], [](float v) { return v; });
    s_rstd[tid] = 1.0f / sqrtf(var_sum / 384.0f + 1e-12f);
  }
  __syncthreads();
  const float rstd = s_rstd[rl];
  float amax = 0.0f;
  float4 ys[kF4];
#pragma unroll
  for (int i = 0; i < kF4; i++) {
    const int c = (sub + kLpr * i) * 4;
    const float4 g = *reinterpret_cast<const float4*>(ln.gamma + c);
    const float4 b = *reinterpret_cast<const float4*>(ln.beta + c);
    const float4 sm = *reinterpret_cast<const float4*>(ln.smooth + c);
    float4 y;
    y.x = (xv[i].x - mean) * rstd * g.x + b.x;
    y.y = (xv[i].y - mean) * rstd * g.y + b.y;
    y.z = (xv[i].z - mean) * rstd * g.z + b.z;
    y.w = (xv[i].w - mean) * rstd * g.w + b.w;
    if (valid) *reinterpret_cast<float4*>(ln.dst + (size_t)row * 384 + c) = y;
    ys[i] = make_float4(y.x * sm.x, y.y * sm.y, y.z * sm.z, y.w * sm.w);
    amax = nanless_max(amax, fabsf(ys[i].x));
    amax = nanless_max(amax, fabsf(ys[i].y));
    amax = nanless_max(amax, fabsf(ys[i].z));
    amax = nanless_max(amax, fabsf(ys[i].w));
  }
  amax = kLpr == 16 ? row16_max(amax) : lanes8_max(amax);  // amax is never NaN: fmaxf is nanless_max here
  const float max_abs = nanless_max(1e-8f, amax);
  const float inv_scale = 127.0f / max_abs;
  if (valid) {
#pragma unroll
    for (int i = 0; i < kF4; i++) {
      const int c = (sub + kLpr * i) * 4;
      *reinterpret_cast<uint32_t*>(ln.q + (size_t)row * 384 + c) =
          pack4(qround(ys[i].x * inv_scale), qround(ys[i].y * inv_scale), qround(ys[i].z * inv_scale),
                qround(ys[i].w * inv_scale));
    }
    if (sub == 0) {
      ln.scale[row] = max_abs / 127.0f;
      if (ln.rowmax_init) ln.rowmax_init[row] = __float_as_uint(1e-8f);
      if (ln.rowmax_init2) ln.rowmax_init2[row] = __float_as_uint(1e-8f);
    }
  }
}

// ---------------------------------------------------------------------------
// Small M (latency-bound launches: single sequences, short batches, the
// layer-11 tail): 16 rows per workgroup of 8 waves.  The workgroup
// stages its whole A tile (16 x K int8; f32 A is quantized on the way, as astore
// does above; kALn: through a LayerNorm; kAPreLn: a LayerNorm of the rows of a
// first GEMM) into LDS once, so the K loop has no barrier; each wave streams its
// B fragments through a register ring kRing K steps deep.
//
// The 8 waves form CG = 8 / KS column groups of 48 columns, and the KS waves
// of a group split K: wave w takes column group w % CG and K steps
// [(w / CG) KT / KS, (w / CG + 1) KT / KS).  Their int32 partial sums (exact in
// any order) meet in LDS, and each of them applies the epilogue to 16 / KS of
// the 16 rows.  KS = 1: the workgroup spans 384 columns (with LN it applies the
// LayerNorm + SmoothQuant of `ln` to its 16 output rows, reference
// src/simd_math.rs:208-247, and p.out is not written); KS = 2: 192 columns;
// KS = 8: 48 columns (a workgroup streams an eighth of the weights of the
// KS = 1 form), for long K.  A LayerNorm prologue takes the KS that fills the
// compute units in one round (launch_gemm_ln_prologue).
// ---------------------------------------------------------------------------
constexpr int kSmallMaxK = 1536;
constexpr int kSmallPitch = kSmallMaxK + 16;  // LDS bytes per A row: conflict-free fragment reads
constexpr int kLnPitchS = 388;                // LDS floats per row of the fused LayerNorm
constexpr int kEPitchS = 52;                  // LDS words per row of a wave's epilogue staging tile

template <int AM, int EM, bool LN, int KS, int RT = 16>
__global__ __launch_bounds__(512) void gemm_small_kernel(GemmArgs p, LnArgs ln, PreArgs pre) {
  constexpr int WAVES = 8, NW = 48, kThreads = 512;
  constexpr int CG = WAVES / KS, kBN = CG * NW, kCB = NW / 16, kF4 = NW / 4;
  constexpr int RPW = 16 / KS, kPos = RPW * kF4, kEk = (kPos + 63) / 64;  // epilogue rows / float4s per wave
  constexpr int kRing = KS == 1 ? 6 : 3;  // B ring depth (K steps in flight per wave)
  constexpr bool kLnIn = AM == kALn || AM == kAPreLn;  // a LayerNorm in front of the GEMM
  static_assert(KS == 1 || KS == 2 || KS == 4 || KS == 8, "K splits");
  static_assert(RT == 16 || (RT == 8 && KS == 8 && !LN && AM != kALn && AM != kAPreLn), "8-row tiles: KS = 8 only");
  static_assert(!LN || (KS == 1 && EM == kEpiF32), "fused LayerNorm: 16 rows x 384 columns");
  static_assert(!kLnIn || !LN, "LayerNorm prologue or epilogue");
  constexpr bool kLnTile = LN || kLnIn;  // an f32 row tile for a LayerNorm
  __shared__ __attribute__((aligned(16))) int8_t sA[16 * kSmallPitch];
  __shared__ __attribute__((aligned(16))) int sE[WAVES][16 * kEPitchS];
  static_assert(!kLnTile || sizeof(sE) >= 16 * kLnPitchS * sizeof(float), "LN squares reuse the staging tile");
  __shared__ uint32_t sRowMax[WAVES][16];
  __shared__ __attribute__((aligned(16))) float sEpSa[16], sEpWs[kBN], sEpB[kBN];
  __shared__ __attribute__((aligned(16))) float sLn[kLnTile ? 16 * kLnPitchS : 4];
  __shared__ float s_stat[2][16];
  __shared__ float s_pre_sa[16];  // kAPreLn: the first GEMM's row scales
  __shared__ uint64_t s_tab[EM == kEpiGelu ? 32 : 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int fr = lane & 15, fk = (lane >> 4) * 16;
  // RT rows per tile (RT = 8: the MFMA's rows 8-15 read zeros and are not stored)
  const int mt = (p.M + RT - 1) / RT;
  const int m0 = (blockIdx.x % mt) * RT, n0 = (blockIdx.x / mt) * kBN;
  const int NB = p.N >> 4;
  const int cg = wave % CG, ks = wave / CG;
  const int col0 = n0 + cg * NW;
  // this wave's K steps [kb0, kb0 + KT)
  // (KS need not divide the K steps: wave ks takes [ks KTT / KS, (ks + 1) KTT / KS))
  const int KTT = p.K >> 6, kb0 = ks * KTT / KS, KT = (ks + 1) * KTT / KS - kb0;
  if constexpr (EM == kEpiGelu) exp_tab_fill(s_tab, tid);  // ordered before the epilogue by the K loop's barrier
  const ExpTabLds tb{s_tab};  // the epilogue below is wave-uniform

  // The A tile's global loads go out first, then the B ring and the epilogue
  // operands: memory operations retire in order, so the wait for A does not wait
  // for the weights.  The A tile is 16 rows x K as 16-byte chunks (16 k-values);
  // thread t takes chunks t + 512 i (kALn: f32 columns 4 (sub + 32 i) .. +3 of
  // row tid / 32).
  constexpr int kChunks = (16 * kSmallMaxK / 16 + kThreads - 1) / kThreads;  // per thread at the largest K
  const int cpr = p.K >> 4, nch = RT * cpr;                // chunks per row, in the tile
  const int rr = tid >> 5, sub = tid & 31, lrow = m0 + rr;  // kALn: row and column group
  float4 xv[3], lg[3], lb[3], lsm[3];                       // kALn: x, gamma, beta, inv_smooth
  v4i qa[kChunks];                                          // kAI8
  float4 xa[kChunks][4];                                    // f32 A
  float a_inv[kChunks];
  // kAPreLn: the first GEMM's A chunk (thread t < 384: row t / 24, columns
  // 16 (t % 24) .. +15) and row max, all six K steps of its weight fragments for
  // this wave's 48 columns, and the epilogue operands of its 3 float4 positions
  float4 pa[4], pres[3], pws[3], pbias[3];
  float pa_max = 1.0f;
  v4i pring[6][kCB];
  if constexpr (AM == kAPreLn) {
    if (tid < 384) {
      const int row = min(m0 + tid / 24, p.M - 1);
#pragma unroll
      for (int k = 0; k < 4; k++) pa[k] = reinterpret_cast<const float4*>(pre.A + (size_t)row * 384 + (tid % 24) * 16)[k];
      pa_max = __uint_as_float(pre.a_rowmax[row]);
    }
    const int8_t* pw = pre.w + (size_t)lane * 16;
#pragma unroll
    for (int kt = 0; kt < 6; kt++)
#pragma unroll
      for (int j = 0; j < kCB; j++)
        pring[kt][j] = *reinterpret_cast<const v4i*>(pw + ((size_t)kt * 24 + wave * kCB + j) * 1024);
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const int e = lane + 64 * k, er = e / kF4, col = wave * NW + (e % kF4) * 4;
      pres[k] = *reinterpret_cast<const float4*>(pre.res + (size_t)min(m0 + er, p.M - 1) * 384 + col);
      pws[k] = *reinterpret_cast<const float4*>(pre.w_scale + col);
      pbias[k] = *reinterpret_cast<const float4*>(pre.bias + col);
    }
  }
  if constexpr (kLnIn) {
    if constexpr (AM == kALn) {
      const float* xr = reinterpret_cast<const float*>(p.A) + (size_t)min(lrow, p.M - 1) * 384;
#pragma unroll
      for (int i = 0; i < 3; i++) xv[i] = *reinterpret_cast<const float4*>(xr + (sub + 32 * i) * 4);
    }
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int c = (sub + 32 * i) * 4;
      lg[i] = *reinterpret_cast<const float4*>(ln.gamma + c);
      lb[i] = *reinterpret_cast<const float4*>(ln.beta + c);
      lsm[i] = *reinterpret_cast<const float4*>(ln.smooth + c);
    }
  } else if constexpr (AM == kAI8) {
#pragma unroll
    for (int i = 0; i < kChunks; i++) {
      const int c = tid + kThreads * i, r = c / cpr;
      if (c < nch)
        qa[i] = *reinterpret_cast<const v4i*>(reinterpret_cast<const int8_t*>(p.A) +
                                              (size_t)min(m0 + r, p.M - 1) * p.K + (c - r * cpr) * 16);
    }
  } else {
#pragma unroll
    for (int i = 0; i < kChunks; i++) {
      const int c = tid + kThreads * i, r = c / cpr;
      if (c < nch) {
        const int row = min(m0 + r, p.M - 1);
        const float4* src =
            reinterpret_cast<const float4*>(reinterpret_cast<const float*>(p.A) + (size_t)row * p.K + (c - r * cpr) * 16);
#pragma unroll
        for (int k = 0; k < 4; k++) xa[i][k] = src[k];
        a_inv[i] = __uint_as_float(p.a_rowmax[row]);
      }
    }
  }

  // B ring: the first kRing K steps
  const int cb0 = col0 >> 4;
  const int8_t* wbase = p.w + (size_t)lane * 16;
  v4i bring[kRing][kCB];
  auto bload = [&](int kt, v4i (&dst)[kCB]) {
#pragma unroll
    for (int j = 0; j < kCB; j++)
      dst[j] = *reinterpret_cast<const v4i*>(wbase + ((size_t)(kb0 + kt) * NB + cb0 + j) * 1024);
  };
  if constexpr (AM != kAPreLn) {  // (kAPreLn: after the first GEMM)
#pragma unroll
    for (int u = 0; u < kRing; u++)
      if (u < KT) bload(u, bring[u]);
  }
  // epilogue operands: row scales, w_scale and bias of the workgroup's columns
  float4 ep_reg = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  if (tid < 16) {
    const int r = min(m0 + tid, p.M - 1);
    if (AM == kAI8) ep_reg.x = p.a_scale[r];
    else if (!kLnIn) ep_reg.x = __uint_as_float(p.a_rowmax[r]) / 127.0f;  // scale = max_abs / 127.0
  } else if (tid < 16 + kBN / 4) {
    ep_reg = reinterpret_cast<const float4*>(p.w_scale + n0)[tid - 16];
  } else if (tid < 16 + kBN / 2) {
    ep_reg = reinterpret_cast<const float4*>(p.bias + n0)[tid - 16 - kBN / 4];
  }
  // Epilogue position k of this lane: float4 e = lane + 64 k of the wave's
  // RPW x kF4 block (clamped to the last one, so that every lane runs the
  // wave-uniform GELU), row ks * RPW + e / kF4, columns col0 + 4 (e % kF4).
  auto epos = [&](int k, int& er, int& ec4) {
    const int e = min(lane + 64 * k, kPos - 1);
    er = ks * RPW + e / kF4;
    ec4 = e % kF4;
  };
  float4 resv[kEk];
  if (p.res) {
#pragma unroll
    for (int k = 0; k < kEk; k++) {
      int er, ec4;
      epos(k, er, ec4);
      resv[k] = *reinterpret_cast<const float4*>(p.res + (size_t)min(m0 + er, p.M - 1) * p.N + col0 + ec4 * 4);
    }
    if constexpr (LN) {
      if (p.res_stats) {  // the residual is the LayerNorm of these rows, recomputed as that LayerNorm forms it
#pragma unroll
        for (int k = 0; k < kEk; k++) {
          int er, ec4;
          epos(k, er, ec4);
          const float2 st = p.res_stats[min(m0 + er, p.M - 1)];
          const float4 g = *reinterpret_cast<const float4*>(p.res_gamma + col0 + ec4 * 4);
          const float4 b = *reinterpret_cast<const float4*>(p.res_beta + col0 + ec4 * 4);
          resv[k].x = (resv[k].x - st.x) * st.y * g.x + b.x;
          resv[k].y = (resv[k].y - st.x) * st.y * g.y + b.y;
          resv[k].z = (resv[k].z - st.x) * st.y * g.z + b.z;
          resv[k].w = (resv[k].w - st.x) * st.y * g.w + b.w;
        }
      }
    }
  }

  // the A tile into LDS: int8 A as loaded, f32 A quantized as astore does above,
  // kALn through the LayerNorm; kAPreLn: the first GEMM's rows, then the LayerNorm
  if constexpr (RT < 16) {  // the tile's unused rows: zeros
    for (int c = tid; c < (16 - RT) * cpr; c += kThreads) {
      const int r = RT + c / cpr;
      *reinterpret_cast<v4i*>(&sA[r * kSmallPitch + (c % cpr) * 16]) = v4i{0, 0, 0, 0};
    }
  }
  if constexpr (AM == kAPreLn) {
    // its A tile (quantized as kAF32QSmooth) and row scales
    if (tid < 384) {
      const int r = tid / 24, kc = (tid % 24) * 16;
      const float inv = 127.0f / pa_max;  // inv_scale = 127.0 / max_abs
      uint32_t w[4];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const float4 sm = reinterpret_cast<const float4*>(pre.a_smooth + kc)[k];
        const float4 v = make_float4(pa[k].x * sm.x, pa[k].y * sm.y, pa[k].z * sm.z, pa[k].w * sm.w);
        w[k] = pack4(qround(v.x * inv), qround(v.y * inv), qround(v.z * inv), qround(v.w * inv));
      }
      *reinterpret_cast<v4i*>(&sA[r * kSmallPitch + kc]) = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
      if (tid % 24 == 0) s_pre_sa[r] = pa_max / 127.0f;  // scale = max_abs / 127.0
    }
    __syncthreads();
    // its K loop: this wave's 48 columns, all six K steps
    v4i acc1[kCB];
#pragma unroll
    for (int j = 0; j < kCB; j++) acc1[j] = v4i{0, 0, 0, 0};
#pragma unroll
    for (int kt = 0; kt < 6; kt++) {
      const v4i af = *reinterpret_cast<const v4i*>(&sA[fr * kSmallPitch + kt * 64 + fk]);
#pragma unroll
      for (int j = 0; j < kCB; j++) acc1[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af, pring[kt][j], acc1[j], 0, 0, 0);
    }
    // the second GEMM's B ring, whose latency hides behind the LayerNorm
#pragma unroll
    for (int u = 0; u < kRing; u++)
      if (u < KT) bload(u, bring[u]);
    // its epilogue, through this wave's staging tile, into the LayerNorm's row tile
    int* E1 = sE[wave];
#pragma unroll
    for (int j = 0; j < kCB; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) E1[((lane >> 4) * 4 + r) * kEPitchS + j * 16 + fr] = acc1[j][r];
    wave_lds_sync();
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const int e = lane + 64 * k, er = e / kF4, c4 = e % kF4;
      const int4 a4 = *reinterpret_cast<const int4*>(&E1[er * kEPitchS + c4 * 4]);
      const float sa = s_pre_sa[er];
      float4 b4 = pbias[k];
      b4.x = b4.x + pres[k].x; b4.y = b4.y + pres[k].y; b4.z = b4.z + pres[k].z; b4.w = b4.w + pres[k].w;
      float4 v;
      v.x = fmaf((float)a4.x, sa * pws[k].x, b4.x);
      v.y = fmaf((float)a4.y, sa * pws[k].y, b4.y);
      v.z = fmaf((float)a4.z, sa * pws[k].z, b4.z);
      v.w = fmaf((float)a4.w, sa * pws[k].w, b4.w);
      *reinterpret_cast<float4*>(&sLn[er * kLnPitchS + wave * NW + c4 * 4]) = v;
    }
    __syncthreads();  // sA is free again; the rows are in sLn
#pragma unroll
    for (int i = 0; i < 3; i++) xv[i] = *reinterpret_cast<const float4*>(&sLn[rr * kLnPitchS + (sub + 32 * i) * 4]);
  }
  if constexpr (kLnIn) {
    // LayerNorm + SmoothQuant of the 16 rows (layernorm_smooth_quantize_row_scalar,
    // reference src/simd_math.rs:208-247, as ln_quant_kernel computes it): one
    // lane per row takes the in-order sums, 32 threads per row the rest; the
    // int8 result is the A tile and its scale the epilogue's row scale.
    const bool writer = n0 == 0 && lrow < p.M;
    if constexpr (AM == kALn) {
#pragma unroll
      for (int i = 0; i < 3; i++) *reinterpret_cast<float4*>(&sLn[rr * kLnPitchS + (sub + 32 * i) * 4]) = xv[i];
      __syncthreads();
    }
    if (tid < 16) s_stat[0][tid] = lds_row_sum(&sLn[tid * kLnPitchS], [](float x) { return x; }) / 384.0f;
    __syncthreads();
    const float mean = s_stat[0][rr];
    float* sSq = reinterpret_cast<float*>(&sE[0][0]);  // (x - mean)^2 rows; the staging tile is free until the epilogue
#pragma unroll
    for (int i = 0; i < 3; i++) {
      float4 d = xv[i];
      d.x = d.x - mean; d.y = d.y - mean; d.z = d.z - mean; d.w = d.w - mean;
      *reinterpret_cast<float4*>(&sSq[rr * kLnPitchS + (sub + 32 * i) * 4]) =
          make_float4(d.x * d.x, d.y * d.y, d.z * d.z, d.w * d.w);
    }
    __syncthreads();
    if (tid < 16)
      s_stat[1][tid] = 1.0f / sqrtf(lds_row_sum(&sSq[tid * kLnPitchS], [](float x) { return x; }) / 384.0f + 1e-12f);
    __syncthreads();
    const float rstd = s_stat[1][rr];
    float4 ys[3];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int c = (sub + 32 * i) * 4;
      float4 y;
      y.x = (xv[i].x - mean) * rstd * lg[i].x + lb[i].x;
      y.y = (xv[i].y - mean) * rstd * lg[i].y + lb[i].y;
      y.z = (xv[i].z - mean) * rstd * lg[i].z + lb[i].z;
      y.w = (xv[i].w - mean) * rstd * lg[i].w + lb[i].w;
      if (writer) *reinterpret_cast<float4*>(ln.dst + (size_t)lrow * 384 + c) = y;
      ys[i] = make_float4(y.x * lsm[i].x, y.y * lsm[i].y, y.z * lsm[i].z, y.w * lsm[i].w);
      amax = nanless_max(amax, fabsf(ys[i].x));
      amax = nanless_max(amax, fabsf(ys[i].y));
      amax = nanless_max(amax, fabsf(ys[i].z));
      amax = nanless_max(amax, fabsf(ys[i].w));
    }
    amax = lanes32_max(amax);  // amax is never NaN: fmaxf is nanless_max here
    const float max_abs = nanless_max(1e-8f, amax);
    const float inv_scale = 127.0f / max_abs;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int c = (sub + 32 * i) * 4;
      const uint32_t q4 = pack4(qround(ys[i].x * inv_scale), qround(ys[i].y * inv_scale),
                                qround(ys[i].z * inv_scale), qround(ys[i].w * inv_scale));
      *reinterpret_cast<uint32_t*>(&sA[rr * kSmallPitch + c]) = q4;
      if (writer && ln.q) *reinterpret_cast<uint32_t*>(ln.q + (size_t)lrow * 384 + c) = q4;
    }
    if (sub == 0) {
      sEpSa[rr] = max_abs / 127.0f;
      if (writer) {
        if (ln.scale) ln.scale[lrow] = max_abs / 127.0f;
        if (ln.rowmax_init) ln.rowmax_init[lrow] = __float_as_uint(1e-8f);
        if (ln.rowmax_init2) ln.rowmax_init2[lrow] = __float_as_uint(1e-8f);
      }
    }
  } else if constexpr (AM == kAI8) {
#pragma unroll
    for (int i = 0; i < kChunks; i++) {
      const int c = tid + kThreads * i, r = c / cpr;
      if (c < nch) *reinterpret_cast<v4i*>(&sA[r * kSmallPitch + (c - r * cpr) * 16]) = qa[i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < kChunks; i++) {
      const int c = tid + kThreads * i, r = c / cpr, kc = (c - r * cpr) * 16;
      if (c < nch) {
        const float inv = 127.0f / a_inv[i];  // inv_scale = 127.0 / max_abs
        uint32_t w[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
          float4 v = xa[i][k];
          if (AM == kAF32QSmooth) {  // (x * inv_smooth[j]) * inv_scale
            const float4 sm = reinterpret_cast<const float4*>(p.a_smooth + kc)[k];
            v.x = v.x * sm.x; v.y = v.y * sm.y; v.z = v.z * sm.z; v.w = v.w * sm.w;
          }
          w[k] = pack4(qround(v.x * inv), qround(v.y * inv), qround(v.z * inv), qround(v.w * inv));
        }
        *reinterpret_cast<v4i*>(&sA[r * kSmallPitch + kc]) = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
      }
    }
  }
  if (tid < 16) {
    if (!kLnIn) sEpSa[tid] = ep_reg.x;
  } else if (tid < 16 + kBN / 4) {
    reinterpret_cast<float4*>(sEpWs)[tid - 16] = ep_reg;
  } else if (tid < 16 + kBN / 2) {
    reinterpret_cast<float4*>(sEpB)[tid - 16 - kBN / 4] = ep_reg;
  }
  __syncthreads();

  v4i acc[kCB];
#pragma unroll
  for (int j = 0; j < kCB; j++) acc[j] = v4i{0, 0, 0, 0};
  for (int k0 = 0; k0 < KT; k0 += kRing) {
#pragma unroll
    for (int u = 0; u < kRing; u++) {
      const int kt = k0 + u;
      if (kt < KT) {  // wave-uniform
        const v4i af = *reinterpret_cast<const v4i*>(&sA[fr * kSmallPitch + (kb0 + kt) * 64 + fk]);
#pragma unroll
        for (int j = 0; j < kCB; j++) acc[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af, bring[u][j], acc[j], 0, 0, 0);
        if (kt + kRing < KT) bload(kt + kRing, bring[u]);
      }
    }
  }

  // epilogue: every wave's accumulators through its LDS tile; each wave then
  // adds its column group's KS partial tiles for its rows and writes whole
  // float4s
  {
    int* E = sE[wave];
#pragma unroll
    for (int j = 0; j < kCB; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) E[((lane >> 4) * 4 + r) * kEPitchS + j * 16 + fr] = acc[j][r];
  }
  if (EM == kEpiGelu && lane < 16) sRowMax[wave][lane] = 0u;
  if constexpr (KS > 1) __syncthreads();  // the partial tiles of the other waves
  else wave_lds_sync();                   // E and sRowMax are private to this wave
#pragma unroll
  for (int k = 0; k < kEk; k++) {
    int er, c4;
    epos(k, er, c4);
    const bool valid = lane + 64 * k < kPos && er < RT;  // uniform in k but the last; rows < RT
    const int row = m0 + er, col = col0 + c4 * 4;
    int4 a4 = *reinterpret_cast<const int4*>(&sE[cg][er * kEPitchS + c4 * 4]);
#pragma unroll
    for (int s2 = 1; s2 < KS; s2++) {
      const int4 b = *reinterpret_cast<const int4*>(&sE[cg + CG * s2][er * kEPitchS + c4 * 4]);
      a4.x += b.x; a4.y += b.y; a4.z += b.z; a4.w += b.w;
    }
    const float sa = sEpSa[er];
    const float4 ws4 = *reinterpret_cast<const float4*>(&sEpWs[cg * NW + c4 * 4]);
    float4 b4 = *reinterpret_cast<const float4*>(&sEpB[cg * NW + c4 * 4]);
    if (p.res) {
      b4.x = b4.x + resv[k].x; b4.y = b4.y + resv[k].y; b4.z = b4.z + resv[k].z; b4.w = b4.w + resv[k].w;
    }
    float4 v;
    v.x = fmaf((float)a4.x, sa * ws4.x, b4.x);
    v.y = fmaf((float)a4.y, sa * ws4.y, b4.y);
    v.z = fmaf((float)a4.z, sa * ws4.z, b4.z);
    v.w = fmaf((float)a4.w, sa * ws4.w, b4.w);
    if (EM == kEpiGelu) {
      const float4 g4 = *reinterpret_cast<const float4*>(p.g_smooth + col);
      v.x = gelu_exact(v.x, tb) * g4.x;
      v.y = gelu_exact(v.y, tb) * g4.y;
      v.z = gelu_exact(v.z, tb) * g4.z;
      v.w = gelu_exact(v.w, tb) * g4.w;
      float gm = nanless_max(nanless_max(fabsf(v.x), fabsf(v.y)), nanless_max(fabsf(v.z), fabsf(v.w)));
      if (valid) atomicMax(&sRowMax[wave][er - ks * RPW], __float_as_uint(gm));  // non-negative f32 bits order like u32
    }
    if constexpr (LN) *reinterpret_cast<float4*>(&sLn[er * kLnPitchS + col]) = v;
    else if (valid && row < p.M) *reinterpret_cast<float4*>(p.out + (size_t)row * p.N + col) = v;
  }
  wave_lds_sync();
  if (EM == kEpiGelu && lane < RPW && ks * RPW + lane < RT && m0 + ks * RPW + lane < p.M)
    atomicMax(&p.g_rowmax[m0 + ks * RPW + lane], sRowMax[wave][lane]);
  if constexpr (LN) {
    // sequential sums per row (one lane each), then 32 lanes per row normalize
    // and quantize; ln.dst may equal p.res (its rows were loaded above)
    const int rr = tid >> 5, sub = tid & 31, row = m0 + rr;
    float4 g[3], b[3], sm[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int c = (sub + 32 * i) * 4;
      g[i] = *reinterpret_cast<const float4*>(ln.gamma + c);
      b[i] = *reinterpret_cast<const float4*>(ln.beta + c);
      sm[i] = *reinterpret_cast<const float4*>(ln.smooth + c);
    }
    // The in-order sums are the only serial part: one lane per row adds, every
    // other step (the squares (x - mean)^2 included) runs on all 512 threads.
    // A lone wave issues about one VALU instruction per 5 cycles, so a chain that
    // also formed the squares would take three instructions per element.
    __syncthreads();
    if (tid < 16) s_stat[0][tid] = lds_row_sum(&sLn[tid * kLnPitchS], [](float x) { return x; }) / 384.0f;
    __syncthreads();
    const float mean = s_stat[0][rr];
    float* sSq = reinterpret_cast<float*>(&sE[0][0]);  // the epilogue staging is free now: (x - mean)^2 rows
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int c = (sub + 32 * i) * 4;
      float4 d = *reinterpret_cast<const float4*>(&sLn[rr * kLnPitchS + c]);
      d.x = d.x - mean; d.y = d.y - mean; d.z = d.z - mean; d.w = d.w - mean;
      *reinterpret_cast<float4*>(&sSq[rr * kLnPitchS + c]) = make_float4(d.x * d.x, d.y * d.y, d.z * d.z, d.w * d.w);
    }
    __syncthreads();
    if (tid < 16) {
      const float var_sum = lds_row_sum(&sSq[tid * kLnPitchS], [](float x) { return x; });
      s_stat[1][tid] = 1.0f / sqrtf(var_sum / 384.0f + 1e-12f);
    }
    __syncthreads();
    const float rstd = s_stat[1][rr];
    float4 ys[3];
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < 3; i++) {
      const int c = (sub + 32 * i) * 4;
      const float4 x = *reinterpret_cast<const float4*>(&sLn[rr * kLnPitchS + c]);
      float4 y;
      y.x = (x.x - mean) * rstd * g[i].x + b[i].x;
      y.y = (x.y - mean) * rstd * g[i].y + b[i].y;
      y.z = (x.z - mean) * rstd * g[i].z + b[i].z;
      y.w = (x.w - mean) * rstd * g[i].w + b[i].w;
      if (row < p.M) *reinterpret_cast<float4*>(ln.dst + (size_t)row * 384 + c) = y;
      ys[i] = make_float4(y.x * sm[i].x, y.y * sm[i].y, y.z * sm[i].z, y.w * sm[i].w);
      amax = nanless_max(amax, fabsf(ys[i].x));
      amax = nanless_max(amax, fabsf(ys[i].y));
      amax = nanless_max(amax, fabsf(ys[i].z));
      amax = nanless_max(amax, fabsf(ys[i].w));
    }
    amax = lanes32_max(amax);  // amax is never NaN: fmaxf is nanless_max here
    const float max_abs = nanless_max(1e-8f, amax);
    const float inv_scale = 127.0f / max_abs;
    if (row < p.M) {
#pragma unroll
      for (int i = 0; i < 3; i++) {
        const int c = (sub + 32 * i) * 4;
        *reinterpret_cast<uint32_t*>(ln.q + (size_t)row * 384 + c) =
            pack4(qround(ys[i].x * inv_scale), qround(ys[i].y * inv_scale), qround(ys[i].z * inv_scale),
                  qround(ys[i].w * inv_scale));
      }
      if (sub == 0) {
        ln.scale[row] = max_abs / 127.0f;
        if (ln.rowmax_init) ln.rowmax_init[row] = __float_as_uint(1e-8f);
        if (ln.rowmax_init2) ln.rowmax_init2[row] = __float_as_uint(1e-8f);
      }
    }
  }
}

// Up to this many rows (and K <= kSmallMaxK) the GEMMs take gemm_small_kernel.

// compute units of the current device (cached per device; 256 on MI355X)
int device_cu_count() {
  static std::atomic<int> cache[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cache[dev].load(std::memory_order_relaxed);
  if (n <= 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cache[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}
// int8 A of more bytes than this is re-read from HBM if each column tile walks
// all row tiles (measured: 113 MB of A at M = 294,912 runs 8-12 % faster column
// tile fastest, 25 MB at M = 65,536 up to 13 % slower)
constexpr size_t kColFastABytes = size_t(96) << 20;

// (the K-split forms need an even number of 64-deep K steps)
static bool small_gemm(const GemmArgs& p) { return p.M <= kSmallM && p.K <= kSmallMaxK && p.K % 128 == 0; }
// From this K on (a multiple of 512), a small-M f32-epilogue GEMM splits K over
// the 8 waves of 16 x 48 workgroups (gemm_small_kernel KS = 8)
constexpr int kSplitMinK = 1024;

// int8 A with more rows than kSmallM (kEpiF32) keeps the 16-row workgroups while
// these are the faster: their whole A tile is in flight at once, where
// gemm_w8a8_kernel's K loop is a chain of 6 or 24 steps of 64 behind a barrier
// each on a few 64 x 192 tiles.  K = 384: one round of them, three per compute
// unit (N = 1152: 1,280 rows 6.6 -> 5.2 us, 2,048 rows 7.1 -> 6.4, but 2,843 rows
// 8.2 -> 8.9; N = 1536: 1,536 rows 7.0 -> 6.4, 2,048 rows 7.5 -> 8.1).  K of 1,024
// and 1,536, by the workgroups per compute unit (three run at once; medians over 10
// to 16 placements of the buffers in us, 64 x 192 tiles / 16-row workgroups):
//  * no residual: up to 7 (K = 1024) or 8 (K = 1536).  N = 384: K = 1024, 3,584 rows
//    10.4 / 9.9, 3,840 rows 10.5 / 10.8; K = 1536, 4,096 rows 13.6 / 13.1, 4,352 rows
//    13.9 / 14.2.  N = 1152: K = 1024, 1,184 rows 10.5 / 9.7, 1,280 rows 10.5 / 10.8;
//  * a residual, which costs the 64 x 192 tiles 2.5 to 9 us (by where the buffers
//    lie): up to 12.  N = 384: K = 1024, 6,144 rows 17.3 / 15.4; K = 1536, 1,280 rows
//    17.7 / 6.8, 6,144 rows 19.7 / 18.7, 8,192 rows 22.3 / 26.0.  N = 1152: K = 1024,
//    1,536 rows 14.8 / 12.2, 2,048 rows 16.6 / 15.6.
bool gemm_int8_rows16(int m, int n, int k, bool res, int cus) {
  const long mt = (m + 15) / 16;
  if (k == 384) return mt * (n / 192) <= 3L * cus;
  if (k < kSplitMinK || k > kSmallMaxK || k % 512 != 0) return false;
  return mt * (n / 48) <= (res ? 12L : k == 1024 ? 7L : 8L) * cus;
}

// The attention output GEMM with LN1 (kAF32QSmooth, N = K = 384) takes
// gemm_small_kernel's 16-row workgroups of 8 waves while one per compute unit
// covers the rows.  Both forms are latency chains there (quantize, six K steps,
// two in-order sums of 384), and gemm_ln_rows_kernel's 32-row workgroups of 4
// waves take twice as long for theirs on half the compute units: in passes of
// 1,280, 2,844 and 4,096 rows it took 7.5, 7.2 and 6.7 us more per layer (771 ->
// 689, 1,111 -> 1,032, 1,701 -> 1,627 us per pass).  With more rows a second
// workgroup per CU waits for registers: 5,200 rows 1,029 us against 1,023 in
// 32-row workgroups of 4 waves, which take 8 there now.
static bool ln_rows16(const GemmArgs& p) { return small_gemm(p) || (p.M + 15) / 16 <= device_cu_count(); }

template <int AM, int EM>
static void launch_variant(GemmArgs p, hipStream_t st) {
  const int mt16 = (p.M + 15) / 16;
  if (small_gemm(p) ||
      (AM == kAI8 && EM == kEpiF32 && gemm_int8_rows16(p.M, p.N, p.K, p.res != nullptr, device_cu_count()))) {
    if (EM == kEpiF32 && p.K >= kSplitMinK && p.K % 512 == 0) {
      if (AM != kAI8 && mt16 * (p.N / 48) < 256)  // 8-row tiles: half the f32 A per workgroup, twice the workgroups
        hipLaunchKernelGGL((gemm_small_kernel<AM, kEpiF32, false, 8, 8>), dim3(((p.M + 7) / 8) * (p.N / 48)),
                           dim3(512), 0, st, p, LnArgs{}, PreArgs{});
      else
        hipLaunchKernelGGL((gemm_small_kernel<AM, kEpiF32, false, 8>), dim3(mt16 * (p.N / 48)), dim3(512), 0, st, p,
                           LnArgs{}, PreArgs{});
    } else {
      hipLaunchKernelGGL((gemm_small_kernel<AM, EM, false, 2>), dim3(mt16 * (p.N / 192)), dim3(512), 0, st, p,
                         LnArgs{}, PreArgs{});
    }
    return;
  }
  const int slots = 2 * device_cu_count();
  // at least one full round of 48-row tiles: below that the A-stationary form
  // leaves CUs idle, and the column-tiled kernel's 6x more workgroups are faster
  // (M = 4,096: 18.3 against 9.9 us)
  if (AM == kAI8 && EM == kEpiF32 && p.K == 384 && !p.res && p.N % 192 == 0 && (p.M + 47) / 48 >= slots) {
    // row tiles of 48 or 64 rows, whichever leaves fewer rows' worth of time in
    // a last, partly filled round of workgroups (2 per CU)
    const long t4 = 4L * (((p.M + 63) / 64 + slots - 1) / slots), t3 = 3L * (((p.M + 47) / 48 + slots - 1) / slots);
    if (t3 < t4)
      hipLaunchKernelGGL(gemm_astat_kernel<3>, dim3((p.M + 47) / 48), dim3(256), 0, st, p);
    else
      hipLaunchKernelGGL(gemm_astat_kernel<4>, dim3((p.M + 63) / 64), dim3(256), 0, st, p);
    return;
  }
  p.col_fast = AM != kAI8 || (size_t)p.M * p.K > kColFastABytes;
  const int nbase = ((p.M + 63) / 64) * (p.N / 192);
  hipLaunchKernelGGL((gemm_w8a8_kernel<AM, EM, 48>), dim3(nbase), dim3(256), 0, st, p);
}

// A workgroup with a LayerNorm in front (174 to 182 VGPRs, with 384 columns 224;
// FFN-up behind attn_out 216 and 242; 8 waves) has a compute unit to itself, and most of its time is that LayerNorm, whatever its columns.
// So the K split is the largest whose workgroups still run in one round: 48
// columns each up to 160 rows (N = 1152), 96 up to 336, 192 up to 672, then 384.
// Passes with 48 / 96 / 192 / 384 columns: 128 rows 411 / 412 / 416 / 427 us,
// 256 rows 523 / 472 / 476 / 485, 512 rows 737 / 673 / 625 / 635, 1,024 rows
// 1,132 / 962 / 907 / 861 (48 columns throughout before: the QKV kernel of a
// 509-token document took 19.3 us in three rounds).
void launch_gemm_ln_prologue(const GemmArgs& p, const LnArgs& ln, hipStream_t st) {
  if (p.M <= 0 || p.M > kSmallM || p.K != 384) return;
  const int mt = (p.M + 15) / 16, cus = device_cu_count();
  auto run = [&](auto ks) {
    hipLaunchKernelGGL((gemm_small_kernel<kALn, kEpiF32, false, ks>), dim3(mt * (p.N / (384 / ks))), dim3(512), 0, st,
                       p, ln, PreArgs{});
  };
  if (mt * (p.N / 48) <= cus) run(std::integral_constant<int, 8>{});
  else if (mt * (p.N / 96) <= cus) run(std::integral_constant<int, 4>{});
  else if (mt * (p.N / 192) <= cus) run(std::integral_constant<int, 2>{});
  else run(std::integral_constant<int, 1>{});
}

void launch_gemm_pre_ln(const GemmArgs& p, const PreArgs& pre, const LnArgs& ln, hipStream_t st) {
  if (p.M <= 0 || p.M > kSmallM || p.K != 384) return;
  // 192 columns per workgroup while these run in one round (512 rows at N =
  // 1536), 384 beyond
  const int mt = (p.M + 15) / 16;
  if (mt * (p.N / 192) <= device_cu_count())
    hipLaunchKernelGGL((gemm_small_kernel<kAPreLn, kEpiGelu, false, 2>), dim3(mt * (p.N / 192)), dim3(512), 0, st, p,
                       ln, pre);
  else
    hipLaunchKernelGGL((gemm_small_kernel<kAPreLn, kEpiGelu, false, 1>), dim3(mt * (p.N / 384)), dim3(512), 0, st, p,
                       ln, pre);
}

void launch_gemm_ln(const GemmArgs& p, const LnArgs& ln, hipStream_t st) {
  if (p.M <= 0 || p.N != 384 || p.K != 384 || !p.res) return;
  if (ln_rows16(p)) {
    hipLaunchKernelGGL((gemm_small_kernel<kAF32QSmooth, kEpiF32, true, 1>), dim3((p.M + 15) / 16), dim3(512), 0, st, p,
                       ln, PreArgs{});
    return;
  }
  // 8 waves (114 VGPRs, two workgroups per CU) halve every phase but the in-order
  // sums, 4 waves (165, three per CU) hide one another's latency in several
  // rounds: 8 while they run in one round, 16,384 rows.  Passes with 4 / 8 waves:
  // 4,500 rows 942 / 891 us, 8,190 rows 1,094 / 1,041, 16,380 rows 1,629 / 1,586,
  // 24,000 rows 2,294 / 2,351, 33,000 rows 3,572 / 3,534, 66,000 rows 6,163 / 6,168.
  const int wgs = (p.M + kLrRows - 1) / kLrRows;
  if (wgs <= 2 * device_cu_count())
    hipLaunchKernelGGL(gemm_ln_rows_kernel<8>, dim3(wgs), dim3(512), 0, st, p, ln);
  else
    hipLaunchKernelGGL(gemm_ln_rows_kernel<4>, dim3(wgs), dim3(256), 0, st, p, ln);
}

void launch_gemm(const GemmArgs& p, int amode, int emode, hipStream_t st) {
  if (p.M <= 0) return;
  if (amode == kAI8 && emode == kEpiF32) launch_variant<kAI8, kEpiF32>(p, st);
  else if (amode == kAI8 && emode == kEpiGelu) launch_variant<kAI8, kEpiGelu>(p, st);
  else if (amode == kAF32Q && emode == kEpiF32) launch_variant<kAF32Q, kEpiF32>(p, st);
  else if (amode == kAF32QSmooth && emode == kEpiF32) launch_variant<kAF32QSmooth, kEpiF32>(p, st);
}

// [N,K] row-major int8 -> [K/64][N/16][64 lanes][16 bytes]: lane l of fragment
// (kt, cb) holds w[cb*16 + l%16][kt*64 + (l/16)*16 .. +16]
void swizzle_weights(int n, int k, const int8_t* w, int8_t* out) {
  const int nb = n / 16;
  for (int kt = 0; kt < k / 64; kt++)
    for (int cb = 0; cb < nb; cb++)
      for (int l = 0; l < 64; l++) {
        const int8_t* src = w + (size_t)(cb * 16 + (l & 15)) * k + kt * 64 + (l >> 4) * 16;
        int8_t* dst = out + (((size_t)kt * nb + cb) * 64 + l) * 16;
        for (int b = 0; b < 16; b++) dst[b] = src[b];
      }
}

}  // namespace aek
