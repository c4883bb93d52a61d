// Shared device helpers for the gfx950 kernels of libaeris_hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace aeris {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;

// bf16 <-> f32 on raw bits (round to nearest even; NaN kept quiet)
__device__ __forceinline__ float bf16_bits_to_f32(uint32_t b) { return __uint_as_float(b << 16); }
__device__ __forceinline__ float bf16_lo(uint32_t packed) { return __uint_as_float(packed << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t packed) { return __uint_as_float(packed & 0xffff0000u); }

typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

// round-to-nearest-even conversions; on gfx950 a pair is one v_cvt_pk_bf16_f32
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  bf16x2 v = {(__bf16)lo, (__bf16)hi};
  return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) { return pack_bf16x2(f, 0.f) & 0xffffu; }
// acc + lo + hi of a packed bf16 pair, in fp32 (v_dot2c_f32_bf16 with a pair of ones)
__device__ __forceinline__ float dot2_ones(uint32_t packed, float acc) {
  const bf16x2 ones = {(__bf16)1.0f, (__bf16)1.0f};
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, packed), ones, acc, false);
}

// 64-lane wavefront sum, the same value in every lane.  Data-parallel-primitive adds inside the 16-lane rows (quad
// permutes, half mirror, mirror), two row broadcasts across the rows, total read from lane 63: six VALU operations
// instead of six round trips through the LDS crossbar (ds_bpermute), which a row-per-wave kernel feels twice per row.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ float dpp_add(float v) {  // v + v[lane selected by CTRL]; rows outside ROW_MASK add 0
  return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xF, true));
}
__device__ __forceinline__ float wave_sum(float v) {
  v = dpp_add<0xB1, 0xF>(v);   // quad_perm [1,0,3,2]
  v = dpp_add<0x4E, 0xF>(v);   // quad_perm [2,3,0,1]
  v = dpp_add<0x141, 0xF>(v);  // row_half_mirror
  v = dpp_add<0x140, 0xF>(v);  // row_mirror: every lane holds the sum of its row
  v = dpp_add<0x142, 0xA>(v);  // row_bcast15: rows 1 and 3 add the row before them
  v = dpp_add<0x143, 0xC>(v);  // row_bcast31: rows 2 and 3 add rows 0 + 1
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// sum over the 64 / SUB lanes of a row, the same value in each of them, in wave_sum's order (lanes without elements add zeros)
template <int SUB>
__device__ __forceinline__ float lanes_sum(float v) {
  if (SUB == 1) return wave_sum(v);
  v = dpp_add<0xB1, 0xF>(v);   // quad_perm [1,0,3,2]
  v = dpp_add<0x4E, 0xF>(v);   // quad_perm [2,3,0,1]
  v = dpp_add<0x141, 0xF>(v);  // row_half_mirror
  v = dpp_add<0x140, 0xF>(v);  // row_mirror: every lane holds the sum of its 16
  if (SUB == 2) {              // + that of the other 16 of the 32
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  return v;
}

// ---- buffer_load_dwordx4 ... lds (16 bytes per lane from global memory straight into LDS, lane l at LDS byte
// m0 + 16 l) as inline assembly.  The compiler's builtin form makes every later LDS access a possible alias of the load
// in the compiler's eyes: it then guards LDS reads with s_waitcnt vmcnt(0) wherever it cannot count the operations in
// between, e.g. inside a loop that is entered with stores still in flight.  Issued from assembly the load is invisible
// to that bookkeeping; what orders it against the LDS reads is the kernels' own counted s_waitcnt + barrier, as
// before.  (Vector memory operations complete in order, so operations the compiler does not know of only make its own
// counted waits stricter.)  The descriptor is built by hand: base, stride 0, size in bytes, raw 32-bit format.
typedef u32x4 lds_dma_rsrc;
__device__ __forceinline__ lds_dma_rsrc make_lds_dma_rsrc(const void* base, uint32_t bytes) {
  const uint64_t a = reinterpret_cast<uint64_t>(base);
  lds_dma_rsrc r;
  r.x = __builtin_amdgcn_readfirstlane((uint32_t)a);
  r.y = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu);
  r.z = __builtin_amdgcn_readfirstlane(bytes);
  r.w = 0x00020000u;
  return r;
}
// lds_address, soffset: wave-uniform; voffset: per lane.  Out-of-range lanes arrive as zeros: a raw buffer's check covers both
// offsets (the ISA guides: out of range if voffset + instruction offset >= size - soffset; seen on gfx950 for the load into LDS
// and the ordinary load alike, with soffset below, at and far beyond the size).
__device__ __forceinline__ void lds_dma_load16(const lds_dma_rsrc& rsrc, uint32_t lds_address, uint32_t voffset, uint32_t soffset) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(lds_address), "v"(voffset), "s"(rsrc), "s"(soffset)
               : "memory");
}

// ---- ds_read_b64_tr_b16 (the LDS read that transposes 4 x 4 blocks of 16-bit elements on the way out) as inline assembly.
// The compiler's builtin form may not be used while a buffer_load ... lds is in flight: the compiler cannot tell that
// the read does not alias the load's destination and puts an s_waitcnt vmcnt(0) in front of it, which makes a wave
// wait for the next unit's (or chunk's) loads in the middle of the arithmetic that they are meant to run under.
// The assembly form is invisible to that analysis - and to the compiler's count of outstanding LDS operations: the
// result registers must pass through lds_tr_wait() (s_waitcnt lgkmcnt(0)) before anything reads them.  ("memory"
// keeps the compiler from moving LDS accesses of its own across the read; its own lgkmcnt waits stay correct, LDS
// operations return in order and extra outstanding ones only make a counted wait stricter.)
// Nor does the compiler keep such a read away from registers that a running MFMA is still writing (see the sweep in
// attention_sweep.h).  Both rules are checked on the emitted assembly by every build (asm_check.py, run by build.py).
__device__ __forceinline__ uint32_t lds_byte_address(const void* p) {
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)p;
}
template <int OFFSET>
__device__ __forceinline__ u32x2 lds_read_tr16_b64(uint32_t lds_address) {
  u32x2 r;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(lds_address), "n"(OFFSET) : "memory");
  return r;
}
struct TrFrag { u32x2 lo, hi; };  // two transposing reads = the 8 k slots of one MFMA operand
__device__ __forceinline__ void lds_tr_wait(TrFrag& a, TrFrag& b) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a.lo), "+v"(a.hi), "+v"(b.lo), "+v"(b.hi));
}
__device__ __forceinline__ void lds_tr_wait(TrFrag& a, TrFrag& b, TrFrag& c, TrFrag& d) {
  asm volatile("s_waitcnt lgkmcnt(0)"
               : "+v"(a.lo), "+v"(a.hi), "+v"(b.lo), "+v"(b.hi), "+v"(c.lo), "+v"(c.hi), "+v"(d.lo), "+v"(d.hi));
}
__device__ __forceinline__ bf16x8 tr_frag_value(const TrFrag& f) {
  return __builtin_bit_cast(bf16x8, u32x4{f.lo.x, f.lo.y, f.hi.x, f.hi.y});
}

__device__ __forceinline__ float silu_f(float x) { return x * __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }
__device__ __forceinline__ float erf_poly(float x) {
  // Abramowitz-Stegun 7.1.26, abs error <= 1.5e-7 (below bf16 and fp32-accumulation noise)
  const float ax = fabsf(x);
  const float t = __frcp_rn(fmaf(0.3275911f, ax, 1.0f));
  float pol = fmaf(1.061405429f, t, -1.453152027f);
  pol = fmaf(pol, t, 1.421413741f);
  pol = fmaf(pol, t, -0.284496736f);
  pol = fmaf(pol, t, 0.254829592f);
  const float r = 1.0f - pol * t * __expf(-ax * ax);
  return copysignf(r, x);
}
__device__ __forceinline__ float gelu_erf_f(float x) { return 0.5f * x * (1.0f + erf_poly(x * 0.70710678118654752440f)); }

// The same for results that are rounded to bf16: the same erf formula (Abramowitz-Stegun 7.1.26) as
// GELU(x) = max(x, 0) - |x| q(|x| / sqrt 2) / 2, q = 1 - erf, with the hardware's reciprocal and exp2 (1 ulp each) instead of
// correctly rounded ones, and no subtraction of nearly equal numbers for negative x.  Evaluated in fp32 against erfc in fp64 on
// [-12, 12]: at most 3.3e-7 absolute (the form with correctly rounded operations: 4.7e-7) and 4.1e-7 |x|.  The formula's error
// is absolute, GELU's tail goes to zero: in bf16 ulps of the result 7e-4 at most from -2 up, 7e-3 from -3, 0.09 from -4, 0.4
// from -5, 1.6 from -7, where the result is -9e-12.  12 VALU operations and two transcendentals: as the epilogue of a
// 4096 x 3072 x 768 product 35.1 -> 29.7 us.  |x| is limited to 30 (q = 0 from 5.6 on) so that an infinite x has no infinity
// times zero in it.
__device__ __forceinline__ float gelu_erf_bf16_f(float x) {
  const float ax = fminf(fabsf(x), 30.0f);
  const float t = __builtin_amdgcn_rcpf(fmaf(0.23164189f, ax, 1.0f));  // 0.3275911 / sqrt 2
  float pol = fmaf(0.5307027145f, t, -0.7265760135f);  // the coefficients halved
  pol = fmaf(pol, t, 0.7107068705f);
  pol = fmaf(pol, t, -0.142248368f);
  pol = fmaf(pol, t, 0.127414796f);
  const float e = __builtin_amdgcn_exp2f(x * x * -0.72134752044f);  // log2(e) / 2
  return fmaf(-ax, pol * t * e, fmaxf(x, 0.0f));
}

// erf-GELU for results that are rounded to bf16, for the problems whose epilogue is a sizeable part of a tile:
// GELU(x) = max(x, 0) - a * 2^P(a), a = |x|, P the degree-4 polynomial for which 2^P is the minimax approximation of
// 1 - Phi(a): log2 of the normal tail is nearly a parabola, so four coefficients do for it what a polynomial for Phi itself
// needs seven for.  In fp32 against erfc in fp64 on [-12, 12]: at most 6.9e-6 |x| and 2.2e-5 absolute, 7.4e-6 of the 2-norm on
// normal inputs (the degree-6 polynomial in x^2 with clamps that stood here: 2.0e-4 |x| down to
// -3.5, 8e-4 absolute below, 3.3e-5).  From 12 on a is held at 12, where 2^P = 9e-21: -inf goes to -1e-19, +inf stays; both
// min and max hand NaN on.
// Seven VALU operations and one transcendental against eleven: the epilogue of a 256 x 256 tile is bound by the VALU, 12.2 K
// cycles of 32 K (K = 512): 64 800 x 2048 x 512 163 -> 157 us, 51 840 x 1280 x 320 63 -> 59.5 us, 259 200 x 6144 x 1536
// 3.80 -> 3.72 ms.  (Degree 3, six operations and one: another 1 %, but 8.2e-5 of the 2-norm.)
__device__ __forceinline__ float gelu_bf16_f(float x) {
  const float a = __builtin_elementwise_minimum(fabsf(x), 12.0f);
  float p = fmaf(0.004708853117f, a, -0.0479899716f);
  p = fmaf(p, a, -0.4622178112f);
  p = fmaf(p, a, -1.150467664f);
  p = fmaf(p, a, -1.00001968f);
  return fmaf(-a, __builtin_amdgcn_exp2f(p), __builtin_elementwise_maximum(x, 0.0f));
}

}  // namespace aeris
