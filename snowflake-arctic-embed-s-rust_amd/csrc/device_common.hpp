// device_common.hpp -- exact scalar building blocks shared by the gfx950 kernels.
//
// Build flags that carry semantics: -ffp-contract=off (no a*b+c fusion: the
// reference is Rust, which never contracts), correctly rounded f32 divide and
// sqrt (HIP's default), no fast-math.  Every kernel evaluates exactly the
// reference's scalar expression order (sequential sums, separately rounded
// products, glibc's expf), so its outputs are bit-identical to the reference's
// scalar backend on the same inputs, and so is the whole forward pass.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.hpp"  // kPlanHdr

namespace aek {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int H = 384;
constexpr int HQKV = 3 * 384;
constexpr float kInvSqrtD = 0.17677669529663687f;  // 1.0f / sqrtf(32.0f), src/model.rs:222

// ---------------------------------------------------------------------------
// exact scalar building blocks
// ---------------------------------------------------------------------------

// `(v).round().clamp(-127.0, 127.0) as i8` (f32::round = half away from zero;
// `as i8` maps NaN to 0), as the truncating, saturating v_cvt_i32_f32 (NaN -> 0)
// of v + (0.5 - 2^-25) with v's sign, then the clamp: |v| + (0.5 - 2^-25) rounds
// up to the next integer exactly when |v| has a fraction >= 0.5, and a
// round-to-nearest-even sum is odd under negation, so adding the signed
// constant and truncating equals trunc(|v| + 0.5 - 2^-25) with v's sign.  Equal
// to the roundf / NaN test / clamp form on all 2^32 inputs (exhaustive CPU check
// with the conversion's saturation), in four instructions.
__device__ __forceinline__ int qround(float v) {
  const float r = v + copysignf(0x1.fffffep-2f, v);
  int q;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(q) : "v"(r));
  return max(-127, min(q, 127));
}

// qround for |x| <= 127.5 or NaN, which holds wherever x = v * (127 / max_abs)
// with max_abs >= |v| (|x| <= 127 * (1 + 2^-24)^2 after the two roundings):
// round half away from zero as the truncating convert of x + (0.5 - 2^-25) with
// x's sign (as qround; equal to roundf on all 2.26 G such floats, exhaustive CPU
// check).  The clamp to [-127, 127] cannot bind in that range; v_cvt_i32_f32
// maps NaN to 0, as the reference's `as i8` does (inline asm: a C++
// float-to-int cast of NaN would be undefined).
__device__ __forceinline__ int qround_bounded(float x) {
  const float r = x + copysignf(0x1.fffffep-2f, x);
  int q;
  asm("v_cvt_i32_f32 %0, %1" : "=v"(q) : "v"(r));
  return q;
}

__device__ __forceinline__ uint32_t pack4(int a, int b, int c, int d) {
  return (uint32_t)(a & 0xff) | ((uint32_t)(b & 0xff) << 8) | ((uint32_t)(c & 0xff) << 16) |
         ((uint32_t)(d & 0xff) << 24);
}

// max(m, a) that ignores a NaN `a`, like `if a > max_abs { max_abs = a }`.
__device__ __forceinline__ float nanless_max(float m, float a) { return a > m ? a : m; }

// DPP lane permutations within rows of 16 lanes
constexpr int kDppXor1 = 0xB1;        // quad_perm [1,0,3,2]
constexpr int kDppXor2 = 0x4E;        // quad_perm [2,3,0,1]
constexpr int kDppHalfMirror = 0x141; // lane i <-> 7-i within 8 lanes
constexpr int kDppMirror = 0x140;     // lane i <-> 15-i within 16 lanes
template <int kCtrl>
__device__ __forceinline__ uint32_t dpp(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, kCtrl, 0xF, 0xF, true);  // every lane has a source
}

// max over the 16 lanes of this lane's DPP row (every lane gets it)
__device__ __forceinline__ float row16_max(float m) {
  m = fmaxf(m, __uint_as_float(dpp<kDppXor1>(__float_as_uint(m))));
  m = fmaxf(m, __uint_as_float(dpp<kDppXor2>(__float_as_uint(m))));
  m = fmaxf(m, __uint_as_float(dpp<kDppHalfMirror>(__float_as_uint(m))));
  return fmaxf(m, __uint_as_float(dpp<kDppMirror>(__float_as_uint(m))));
}

// unsigned max over the 16 lanes of this lane's DPP row (every lane gets it)
__device__ __forceinline__ uint32_t row16_max_u32(uint32_t m) {
  m = max(m, dpp<kDppXor1>(m));
  m = max(m, dpp<kDppXor2>(m));
  m = max(m, dpp<kDppHalfMirror>(m));
  return max(m, dpp<kDppMirror>(m));
}

// max over this lane's group of 8 lanes (DPP; every lane gets it)
__device__ __forceinline__ float lanes8_max(float m) {
  m = fmaxf(m, __uint_as_float(dpp<kDppXor1>(__float_as_uint(m))));
  m = fmaxf(m, __uint_as_float(dpp<kDppXor2>(__float_as_uint(m))));
  return fmaxf(m, __uint_as_float(dpp<kDppHalfMirror>(__float_as_uint(m))));
}

// max over this lane's half-wave of 32 lanes (every lane gets it): DPP within
// each 16-lane row, then one cross-row exchange
__device__ __forceinline__ float lanes32_max(float m) {
  m = row16_max(m);
  return fmaxf(m, __shfl_xor(m, 16, 64));
}

// Orders this wave's LDS accesses before and after it (LDS data private to one
// wave needs no workgroup barrier: a wave's LDS operations complete in order once
// the counter is drained).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// bits(2^(i/32) rounded to double) - (i << 47), i = 0..31: the exp2 table of
// expf_libm below (computed from 2^(i/32) in quad precision).
static __constant__ uint64_t kExp2Tab[32] = {
    0x3ff0000000000000ull, 0x3fefd9b0d3158574ull, 0x3fefb5586cf9890full, 0x3fef9301d0125b51ull,
    0x3fef72b83c7d517bull, 0x3fef54873168b9aaull, 0x3fef387a6e756238ull, 0x3fef1e9df51fdee1ull,
    0x3fef06fe0a31b715ull, 0x3feef1a7373aa9cbull, 0x3feedea64c123422ull, 0x3feece086061892dull,
    0x3feebfdad5362a27ull, 0x3feeb42b569d4f82ull, 0x3feeab07dd485429ull, 0x3feea47eb03a5585ull,
    0x3feea09e667f3bcdull, 0x3fee9f75e8ec5f74ull, 0x3feea11473eb0187ull, 0x3feea589994cce13ull,
    0x3feeace5422aa0dbull, 0x3feeb737b0cdc5e5ull, 0x3feec49182a3f090ull, 0x3feed503b23e255dull,
    0x3feee89f995ad3adull, 0x3feeff76f2fb5e47ull, 0x3fef199bdd85529cull, 0x3fef3720dcef9069ull,
    0x3fef5818dcfba487ull, 0x3fef7c97337b9b5full, 0x3fefa4afa2a490daull, 0x3fefd0765b6e4540ull,
};

// The table lives in registers across the wave: lane l keeps entry l % 32 as two
// 32-bit halves, and a lookup is a pair of ds_bpermute (a crossbar read of
// another lane's register: no LDS bank conflicts, unlike a data-dependent
// ds_read of a shared table).  ds_bpermute picks lane (address / 4) mod 64
// (checked on gfx950), and both halves of the wave hold the table, so the
// lookup of index k reads lane k mod 64 without masking k to 5 bits.  A lookup
// may read any lane, so EVERY lane of the wave must be active at every
// expf_libm / gelu_exact call: call them only from wave-uniform control flow.
struct ExpTab {
  uint32_t lo, hi;
};

__device__ __forceinline__ ExpTab exp_tab_regs() {
  const uint64_t t = kExp2Tab[threadIdx.x & 31];
  return ExpTab{(uint32_t)t, (uint32_t)(t >> 32)};
}

// entry k % 32 (k: any 32-bit value)
__device__ __forceinline__ uint64_t exp_tab_lookup(const ExpTab& tb, uint32_t k) {
  const int addr = (int)(k << 2);  // byte address of lane k mod 64, which holds entry k % 32
  const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(addr, (int)tb.lo);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute(addr, (int)tb.hi);
  return ((uint64_t)hi << 32) | lo;
}

// The same table in LDS (kernels that have 256 spare bytes): its 32 entries of
// 8 bytes fill the 64 banks once, so a ds_read_b64 of data-dependent entries is
// free of bank conflicts (lanes that read one entry share the read).  One LDS
// read per lookup instead of two crossbar reads.  The kernel fills it with
// exp_tab_fill before a barrier.
struct ExpTabLds {
  const uint64_t* t;  // LDS
};
__device__ __forceinline__ void exp_tab_fill(uint64_t* lds_tab, int tid) {
  if (tid < 32) lds_tab[tid] = kExp2Tab[tid];
}
__device__ __forceinline__ uint64_t exp_tab_lookup(const ExpTabLds& tb, uint32_t k) { return tb.t[k & 31]; }

// expf as glibc computes it on x86_64 (sysdeps/ieee754/flt-32/e_expf.c, the
// ARM optimized-routines design with a 32-entry 2^(i/32) table and a cubic
// polynomial, evaluated in double with the FMA contractions of glibc's -mfma
// build).  The reference's scalar GELU and softmax call f32::exp, i.e. this
// function.  Verified equal to glibc expf on every float in [-104, -0]; valid
// for x <= 0 and NaN.  Branch-free (see ExpTab): the underflow case of glibc,
// x < log(2^-150), is applied as a final select.
template <typename Tab>
__device__ __forceinline__ float expf_libm(float x, const Tab& tb) {
  const double kInvLn2N = 0x1.71547652b82fep+0 * 32.0;
  const double kShift = 0x1.8p+52;
  const double c0 = 0x1.c6af84b912394p-5 / 32.0 / 32.0 / 32.0;
  const double c1 = 0x1.ebfce50fac4f3p-3 / 32.0 / 32.0;
  const double c2 = 0x1.62e42ff0c52d6p-1 / 32.0;
  const double xd = (double)x;
  double kd = __builtin_fma(kInvLn2N, xd, kShift);
  const uint64_t ki = (uint64_t)__double_as_longlong(kd);
  kd -= kShift;
  const double r = __builtin_fma(kInvLn2N, xd, -kd);
  const uint64_t t = exp_tab_lookup(tb, (uint32_t)ki) + (ki << 47);
  const double s = __longlong_as_double((long long)t);
  const double z = __builtin_fma(c0, r, c1);
  const double r2 = r * r;
  double y = __builtin_fma(c2, r, 1.0);
  y = __builtin_fma(z, r2, y);
  y = y * s;
  const float res = (float)y;
  return x < -0x1.9fe368p6f ? 0.0f : res;  // glibc's underflow branch
}

// exp2f as glibc computes it (sysdeps/ieee754/flt-32/e_exp2f.c: the same
// 32-entry table and cubic as expf_libm, unscaled coefficients, r = x - k/32 in
// double, the -mfma build's contractions), for x <= 0 and NaN; x <= -150 gives
// +0 as glibc's underflow branch does.  Wave-uniform control flow required
// (see ExpTab).
template <typename Tab>
__device__ __forceinline__ float exp2f_libm(float x, const Tab& tb) {
  const double kShift = 0x1.8p+52 / 32.0;
  const double c0 = 0x1.c6af84b912394p-5, c1 = 0x1.ebfce50fac4f3p-3, c2 = 0x1.62e42ff0c52d6p-1;
  const double xd = (double)x;
  double kd = xd + kShift;
  const uint64_t ki = (uint64_t)__double_as_longlong(kd);
  kd -= kShift;
  const double r = xd - kd;
  const uint64_t t = exp_tab_lookup(tb, (uint32_t)ki) + (ki << 47);
  const double s = __longlong_as_double((long long)t);
  const double z = __builtin_fma(c0, r, c1);
  const double r2 = r * r;
  double y = __builtin_fma(c2, r, 1.0);
  y = __builtin_fma(z, r2, y);
  y = y * s;
  const float res = (float)y;
  return x <= -150.0f ? 0.0f : res;
}

// scalar_gelu (reference src/simd_math.rs:15-23), same operation order.
// Wave-uniform control flow required (see ExpTab).
//
// t = 1 / (1 + p z) is v_rcp_f32 plus one Newton step instead of the IEEE
// divide sequence: on every float y in [1, 8) the two are bit-identical
// (all 25.2 M values compared on gfx950).  y is clamped at 8 first: there
// z >= 21.3, exp(-z^2) is +0, and erf is +-1 whatever finite t is, so the clamp
// changes nothing and keeps t finite for x = +-inf.  The whole function equals
// the IEEE-divide form on all 2^32 inputs (NaN for NaN), at ~10 % fewer cycles.
template <typename Tab>
__device__ __forceinline__ float gelu_exact(float x, const Tab& tb) {
  const float z = fabsf(x) * 0.70710677f;
  const float y = fminf(1.0f + 0.3275911f * z, 8.0f);
  const float r0 = __builtin_amdgcn_rcpf(y);
  const float t = __builtin_fmaf(__builtin_fmaf(-y, r0, 1.0f), r0, r0);
  const float poly =
      t * (0.254829592f + t * (-0.284496736f + t * (1.421413741f + t * (-1.453152027f + t * 1.061405429f))));
  const float erf_val = copysignf(1.0f - poly * expf_libm(-z * z, tb), x);
  return 0.5f * x * (1.0f + erf_val);
}

// A fast GELU with a certified distance from gelu_exact, for the fused FFN's
// decide-or-repair quantization (ffn.hip).  The same terms as scalar_gelu,
// reassociated: G'(v) = max(v, 0) - |v| * ((poly/2) * 2^(-v^2 log2(e) / 2)), with
// t = v_rcp_f32(1 + (p/sqrt 2)|v|) and v_exp_f32 (hardware reciprocal and exp2,
// about 1 ulp each).  11 VALU operations and 2 transcendental ones against
// gelu_exact's ~45 (10 of them f64): 47 against 133 SIMD cycles per wave64 GELU
// at the FFN's 2 waves per SIMD (microbenchmark).
//
// Certified on all 2^32 inputs against gelu_exact (GPU enumeration; the
// enumeration is a committed test): G'(v) is NaN exactly for NaN and +-inf v,
// and for every other v, gelu_exact(v) is finite and
//     |gelu_exact(v) - G'(v)| <= 2^-21 |G'(v)| + 0x1.62c111p-24.
// kGeluFastRel / kGeluFastAbs round that up.  Also from the enumeration:
// gelu_exact(v) == v for every v >= kGeluSatPos and gelu_exact(v) == +-0 for
// every finite v <= kGeluSatNeg.
constexpr float kGeluFastRel = 0x1p-21f;
constexpr float kGeluFastAbs = 0x1.64p-24f;
constexpr float kGeluSatPos = 0x1.563c42p+2f;   // the float after 5.34742737 (0x1.563c4p+2)
constexpr float kGeluSatNeg = -0x1.62c12ep+2f;  // the float below -5.54304028 (-0x1.62c12cp+2)
constexpr float kGeluFastK = 0.3275911f * 0.70710677f;  // p / sqrt 2
// N values at once: a dependent VALU instruction issues about 10 cycles after its
// source, so a wave beside one other on its SIMD needs several independent chains
// in flight; the scheduling barriers keep the compiler from serializing them again
// (it orders the values one after the other to save registers).
// kc: kGeluFastK in a VGPR (its instruction takes |v|, so it cannot hold the
// constant itself, and an f32 instruction that reads an SGPR issues at half the
// rate).  The maximum by hand: fmaxf would canonicalize v first.
template <int N>
__device__ __forceinline__ void gelu_fast(const float (&v)[N], float kc, float (&out)[N]) {
  constexpr float kA1 = 0.5f * 0.254829592f, kA2 = 0.5f * -0.284496736f, kA3 = 0.5f * 1.421413741f,
                  kA4 = 0.5f * -1.453152027f, kA5 = 0.5f * 1.061405429f;
  float t[N], a[N], ph[N], m[N];
  auto each = [&](auto f) {
#pragma unroll
    for (int k = 0; k < N; k++) f(k);
    __builtin_amdgcn_sched_barrier(0);
  };
  each([&](int k) { t[k] = __builtin_fmaf(fabsf(v[k]), kc, 1.0f); });
  each([&](int k) { a[k] = v[k] * (-0.5f * 1.44269504088896340736f); });
  each([&](int k) { t[k] = __builtin_amdgcn_rcpf(t[k]); });
  each([&](int k) { a[k] = v[k] * a[k]; });
  each([&](int k) { a[k] = __builtin_amdgcn_exp2f(a[k]); });
  each([&](int k) { ph[k] = __builtin_fmaf(kA5, t[k], kA4); });
  each([&](int k) { ph[k] = __builtin_fmaf(ph[k], t[k], kA3); });
  each([&](int k) { ph[k] = __builtin_fmaf(ph[k], t[k], kA2); });
  each([&](int k) { ph[k] = __builtin_fmaf(ph[k], t[k], kA1); });
  each([&](int k) { ph[k] = t[k] * ph[k]; });
  each([&](int k) { asm("v_max_f32 %0, 0, %1" : "=v"(m[k]) : "v"(v[k])); });
  each([&](int k) { ph[k] = ph[k] * a[k]; });
  each([&](int k) { out[k] = __builtin_fmaf(-fabsf(v[k]), ph[k], m[k]); });
}

// Sequential sum of f(row[j]) over one 384-float LDS row (float4-aligned), in
// index order: 12 batches of 8 float4, each read while the previous one is added.
template <typename F>
__device__ __forceinline__ float lds_row_sum(const float* row, F f) {
  const float4* r4 = reinterpret_cast<const float4*>(row);
  float4 va[8], vb[8];
  auto ld = [&](int bi, float4 (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = r4[8 * min(bi, 11) + i];
  };
  float acc = 0.0f;
  auto add = [&](const float4 (&v)[8]) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      acc += f(v[i].x); acc += f(v[i].y); acc += f(v[i].z); acc += f(v[i].w);
    }
  };
  // sched_barrier: keep each batch's reads issued before the previous batch's
  // adds (the scheduler would otherwise gather both batches' reads at the top of
  // the loop and expose the LDS latency once per iteration)
  ld(0, va);
  for (int bi = 0; bi < 12; bi += 2) {
    ld(bi + 1, vb);
    __builtin_amdgcn_sched_barrier(0);
    add(va);
    __builtin_amdgcn_sched_barrier(0);
    ld(bi + 2, va);
    __builtin_amdgcn_sched_barrier(0);
    add(vb);
    __builtin_amdgcn_sched_barrier(0);
  }
  return acc;
}

// Workgroups are dispatched round-robin over the 8 XCDs (WG p -> XCD p % 8),
// each with its own L2.  xcd_contiguous(p, n) renumbers the n workgroups of a
// launch so that XCD x runs one contiguous range of logical items: neighbouring
// items, which share input data, then run on one XCD and hit in its L2.
__device__ __forceinline__ int xcd_contiguous(int p, int n) {
  const int q = n >> 3, r = n & 7, x = p & 7, i = p >> 3;
  return (x < r ? x * (q + 1) : r * (q + 1) + (x - r) * q) + i;
}

// The attention kernels' workgroup -> item map over one list of a tile plan
// (attention_plan_kernel): workgroup p runs on XCD x = p mod 8 (the hardware's
// round-robin dispatch) and takes item i (p / 8, or what the kernel makes of it)
// of XCD x's list, whose count and first item are int2 x of the list's header.  The surplus workgroups of the
// worst-case grid come last on every XCD and leave after the header load:
// false for those.  rec = {s0, L, q0, nq}.
__device__ __forceinline__ bool plan_item(const int4* list, int i, int& h, int& seg, int4& rec) {
  const int2 hx = reinterpret_cast<const int2*>(list)[blockIdx.x & 7];
  if (i >= hx.x) return false;
  rec = list[kPlanHdr + hx.y + i];
  h = rec.z >> 16;
  rec.z &= 0xffff;
  seg = (int)((uint32_t)rec.w >> 8);
  rec.w &= 0xff;
  return true;
}
__device__ __forceinline__ bool plan_item(const int4* list, int i, int& h, int4& rec) {
  int seg;
  return plan_item(list, i, h, seg, rec);
}

// index of the segment containing token t: largest b with cu[b] <= t (cu has B+1 entries)
__device__ __forceinline__ int find_segment(const int* cu, int B, int t) {
  int lo = 0, hi = B - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (cu[mid] <= t) lo = mid; else hi = mid - 1;
  }
  return lo;
}

}  // namespace aek
