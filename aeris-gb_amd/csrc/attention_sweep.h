// The arithmetic of one 32-query group against the keys of one window, shared by every one-window attention kernel:
// logits' start values (relative-position bias) and shift mask, the sweep over the key blocks, the two-pass form for
// rows whose logits leave the range of the sweep, and the normalised store of the output rows.
//
// Operand layout (v_mfma_f32_32x32x16_bf16, lane = l31 + 32 hi):
//   S^T block kb = K[32 kb ..][:] Q^T: a[4g + i] is the logit (times log2 e) of key 32 kb + 8 g + 4 hi + i and the lane's
//   query l31.  P^T = exp2(S^T) packed to bf16 pairs is, register for register, the B operand of O^T = V^T P^T: k slots
//   0-3 of PV step 2 kb + t2 are the keys 32 kb + 16 t2 + 4 hi + (0..3), slots 4-7 the keys 32 kb + 16 t2 + 8 + 4 hi + (0..3).
//   o[db][4g + i] = O[query][32 db + 8 g + 4 hi + i].
// A kernel supplies how its K and V^T fragments are read from LDS: `load_k(kb, f)`, and for V^T one of the two
// loaders below (`load_v(step, raw)` issues the reads of one 16-key step, `load_v.ready(...)` turns what was read into
// MFMA operands once it is needed).
#pragma once
#include "common.h"

namespace aeris {

// V^T fragments from a row-major V tile by the transposing LDS read.  Within every 16 lanes, source lane 4 e + a reads 4
// consecutive elements and result lane 4 a + b receives element b of the source lanes a, 4 + a, 8 + a, 12 + a: with
// source lane 4 e + a at V[key0 + e][d0 + 4 a ..] the result lane owns column d0 + (lane & 15) of the keys
// key0 .. key0 + 3, half of an MFMA operand's 8 k slots.  V rows are 128 B with 16-byte chunks XOR-swizzled by
// 2 (key & 3).  `step_base(step)` is the LDS byte address of V row 16 step.  The reads are issued as inline assembly
// (see lds_read_tr16_b64): ready() is the s_waitcnt that makes their results usable.
template <int DB, class StepBase>
struct LoadVTransposed {
  using Raw = TrFrag;
  uint32_t v_lane[DB];
  StepBase step_base;
  __device__ __forceinline__ LoadVTransposed(int lane, StepBase sb) : step_base(sb) {
    const int jb = lane >> 4, e = (lane >> 2) & 3, a = lane & 3;  // 16-lane block (column half jb & 1, key half jb >> 1), source lane 4 e + a
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int chunk = (4 * db + 2 * (jb & 1) + (a >> 1)) ^ (2 * e);
      v_lane[db] = (uint32_t)((4 * (jb >> 1) + e) * 128 + (chunk << 4) + (a & 1) * 8);
    }
  }
  __device__ __forceinline__ void operator()(int step, Raw (&f)[DB]) const {
    const uint32_t b = step_base(step);
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      f[db].lo = lds_read_tr16_b64<0>(b + v_lane[db]);
      f[db].hi = lds_read_tr16_b64<1024>(b + v_lane[db]);
    }
  }
  __device__ __forceinline__ void ready(Raw (&a)[DB], Raw (&b)[DB], bf16x8 (&va)[DB], bf16x8 (&vb)[DB]) const {
    static_assert(DB == 2, "head_dim 64");
    lds_tr_wait(a[0], a[1], b[0], b[1]);
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      va[db] = tr_frag_value(a[db]);
      vb[db] = tr_frag_value(b[db]);
    }
  }
  __device__ __forceinline__ void ready(Raw (&a)[DB], bf16x8 (&va)[DB]) const {
    static_assert(DB == 2, "head_dim 64");
    lds_tr_wait(a[0], a[1]);
#pragma unroll
    for (int db = 0; db < DB; ++db) va[db] = tr_frag_value(a[db]);
  }
};

// V^T fragments by ordinary reads (`read(step, f)`: a tile that was transposed when it was written): nothing to wait for.
template <int DB, class Read>
struct LoadVPlain {
  using Raw = bf16x8;
  Read read;
  __device__ __forceinline__ explicit LoadVPlain(Read r) : read(r) {}
  __device__ __forceinline__ void operator()(int step, Raw (&f)[DB]) const { read(step, f); }
  __device__ __forceinline__ void ready(Raw (&a)[DB], Raw (&b)[DB], bf16x8 (&va)[DB], bf16x8 (&vb)[DB]) const {
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      va[db] = a[db];
      vb[db] = b[db];
    }
  }
  __device__ __forceinline__ void ready(Raw (&a)[DB], bf16x8 (&va)[DB]) const {
#pragma unroll
    for (int db = 0; db < DB; ++db) va[db] = a[db];
  }
};

// Start values and mask of the logits of one query group.  The bias table lies in LDS as fp32 4-vectors
// R4[s] = (R[s..s+3]), R reversed and multiplied by log2 e, so that the biases of 4 consecutive keys are one
// ds_read_b128 at index sp(query) + qt(first key), read straight into the accumulators of K Q^T before its MFMAs:
// the bias costs neither an add nor a zero-fill.  The index is a part of the lane's own plus a part that is a constant once kb
// is one (the unrolled sweep): a per-lane base address and an immediate offset, no arithmetic per key group.  (Per-lane key
// divisions instead, and whole padded key blocks below: 12x12 windows, 64800 tokens x 8 heads of 64 64.9 us, shifted 72.0; so
// 62.5 and 65.1.  8 heads of 32 49.7 -> 42.5 us, 51840 tokens x 5 heads of 64 37.5 -> 35.0 us.)
// The cyclic-shift mask is computed from the window position (only windows on the wrapped border of a shifted grid carry
// more than one region; -100 across regions); keys past the window (windows whose token count is not a multiple of 32)
// get -inf.
template <int WS_Y, int WS_X, bool HAS_BIAS, int PITCH = 2 * WS_X - 1>
struct WindowLogits {
  static constexpr int L = WS_Y * WS_X, LPAD = (L + 31) / 32 * 32, TBL = (2 * WS_Y - 1) * (2 * WS_X - 1);
  static constexpr float MASK_NEG = -100.0f * 1.4426950408889634f;  // the additive -100, in the exp2 domain
  static_assert(WS_X % 4 == 0 && L % 16 == 0, "4 consecutive keys lie in one window row, 8 and 16 inside or outside the window");
  // the lane's part of a bias vector's address: its upper half's keys are 4 further on, in the same window row or at the
  // start of the next one (table rows are 2 WS_X - 1 entries: WS_X + 3 further)
  const unsigned char *sB_same, *sB_next;
  int hi;
  bool my, mx;
  int ry_q, rx_q, sy, sx;

  // qpos: the lane's query position in the window (already clamped to L - 1); my / mx: the window lies on the wrapped
  // border in y / x and the mask is on
  __device__ __forceinline__ WindowLogits(const unsigned char* bias_lds, int qpos, int hi_, bool my_, bool mx_, int sy_, int sx_)
      : hi(hi_), my(my_), mx(mx_), sy(sy_), sx(sx_) {
    const int qiy = qpos / WS_X, qix = qpos % WS_X;
    const int sp = (2 * WS_Y - 2) * PITCH + 2 * WS_X - 2 - (qiy + WS_Y - 1) * PITCH - qix - (WS_X - 1);
    sB_same = bias_lds + (sp + 4 * hi) * 16;
    sB_next = bias_lds + (sp + (PITCH - WS_X + 4) * hi) * 16;
    ry_q = my ? (qiy < WS_Y - sy ? 1 : 2) : 0;
    rx_q = mx ? (qix < WS_X - sx ? 1 : 2) : 0;
  }
  __device__ __forceinline__ void init_acc(int kb, f32x16& a) const {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 bv = {0.f, 0.f, 0.f, 0.f};
      const int base = kb * 32 + g * 8;
      if (HAS_BIAS && (LPAD == L || base < L)) {
        const int qt0 = (base / WS_X) * PITCH + (base % WS_X);
        bv = *reinterpret_cast<const f32x4*>((base % WS_X + 4 < WS_X ? sB_same : sB_next) + qt0 * 16);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) a[g * 4 + i] = bv[i];
    }
  }
  __device__ __forceinline__ void mask_block(int kb, f32x16& a) const {
    if (my || mx) {
      // as in init_acc: the lane's 4 keys of a group lie in one window row; where and in which row its upper half's lie is
      // known once kb is.  What depends on the lane is whether column (first key's) + i has wrapped around.
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int base = kb * 32 + g * 8, cx0 = base % WS_X;
        if (LPAD != L && base >= L) break;
        const bool next = cx0 + 4 >= WS_X;
        const int kiy = base / WS_X + (next ? hi : 0), dx = next ? -cx0 * hi : 4 * hi;
        const bool ydiff = my && ((kiy < WS_Y - sy) != (ry_q == 1));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const bool xdiff = mx && ((dx < WS_X - sx - i - cx0) != (rx_q == 1));
          if (ydiff || xdiff) a[g * 4 + i] += MASK_NEG;
        }
      }
    }
    if (LPAD != L) {
#pragma unroll
      for (int g = 0; g < 4; ++g)
        if (kb * 32 + g * 8 >= L) {
#pragma unroll
          for (int i = 0; i < 4; ++i) a[g * 4 + i] = -INFINITY;
        }
    }
  }
};

// Build the head's bias column in LDS (see WindowLogits): R4[j - e][e] = R[j] = table[TBL - 1 - j][head] * log2 e.
// Tail components R4[s][e] with s + e >= TBL are never read by a valid key group.
template <int TBL>
__device__ __forceinline__ void build_bias_lds(unsigned char* sB, const uint16_t* table, int heads, int head, int tid, int nt) {
  float* sBf = reinterpret_cast<float*>(sB);
  for (int j = tid; j < TBL; j += nt) {
    const float r = bf16_bits_to_f32(table[(int64_t)(TBL - 1 - j) * heads + head]) * 1.4426950408889634f;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (j - e >= 0) sBf[(j - e) * 4 + e] = r;
  }
}

// The same with rows of PITCH = 2 WS_X - 4 vectors: those that start in a row's first 2 WS_X - 4 columns are all that a key
// group (whose first column is a multiple of 4) reads.
template <int WS_Y, int WS_X>
__device__ __forceinline__ void build_bias_rows_lds(unsigned char* sB, const uint16_t* table, int heads, int head, int tid, int nt) {
  constexpr int ROW = 2 * WS_X - 1, PITCH = 2 * WS_X - 4, TBL = (2 * WS_Y - 1) * ROW;
  float* sBf = reinterpret_cast<float*>(sB);
  for (int j = tid; j < TBL; j += nt) {
    const int y = j / ROW, x = j - y * ROW;
    const float r = bf16_bits_to_f32(table[(int64_t)(TBL - 1 - j) * heads + head]) * 1.4426950408889634f;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (x - e >= 0 && x - e < PITCH) sBf[(y * PITCH + x - e) * 4 + e] = r;
  }
}

// o = sum over the window's keys of P V and `sum` = the row sum of P, for the lane's query, P = softmax numerator.
// Fast path: ONE sweep over the key blocks with P = exp2(logit) and no row maximum (q carries scale * log2 e, the bias
// table log2 e, so the accumulators of K Q^T are the logits in the exp2 domain).  softmax does not depend on the
// subtracted constant; it only guards the range, and the range is checked afterwards: a row sum outside
// [2^-40, 2^100] (or not finite) in any lane sends the wave through the two-pass form with the row maximum (S^T
// recomputed block by block).  Per key block the MFMAs of S^T for block kb + 1 are issued ahead of the exp2 of block
// kb and those of P V for block kb after it, so that the matrix pipe runs while the VALU forms P; K fragments are read
// from LDS two blocks ahead, V^T fragments one block ahead.  Without a bias the first MFMA of an S^T block takes a
// literal zero as its C operand, and so does the first one of O^T: no accumulator is zero-filled by the VALU.
// `mid(kb)` is called at the start of key block kb (a hook for work a kernel wants issued inside the sweep).
// Of a last key block that is half outside the window only the half inside is exponentiated and multiplied by V (whose tile
// then needs no rows past the window; K rows past it may hold anything).
template <int NQ, int KS, int DB, bool HAS_BIAS, class Logits, class LoadK, class LoadV, class Mid>
__device__ __forceinline__ void attention_sweep(const Logits& lg, const LoadK& load_k, const LoadV& load_v, const Mid& mid,
                                                const bf16x8 (&qf)[KS], f32x16 (&o)[DB], float& sum) {
  constexpr int L = Logits::L;
  {
    const f32x16 zero16 = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    f32x16 acc2[2];
    bf16x8 kf[2][KS], vf[2][DB];
    typename LoadV::Raw vraw[2][DB];
    uint32_t pk[8];
    sum = 0.f;
    auto qk_block = [&](f32x16& acc, const bf16x8 (&kfr)[KS]) {
#pragma unroll
      for (int s2 = 0; s2 < KS; ++s2)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kfr[s2], qf[s2], (!HAS_BIAS && s2 == 0) ? zero16 : acc, 0, 0, 0);
    };
    load_k(0, kf[0]);
    if (HAS_BIAS) lg.init_acc(0, acc2[0]);
    if (NQ > 1) {
      load_k(1, kf[1]);
      if (HAS_BIAS) lg.init_acc(1, acc2[1]);
    }
    __builtin_amdgcn_sched_barrier(0);
    qk_block(acc2[0], kf[0]);
#pragma unroll
    for (int kb = 0; kb < NQ; ++kb) {
      f32x16& a = acc2[kb & 1];
      __builtin_amdgcn_sched_barrier(0);
      mid(kb);
      // S^T of the next block first, the V^T reads of this block behind it: the compiler's wait for the bias vectors
      // and K fragments that those MFMAs consume (it does not know of the assembly reads and waits for "all") then
      // falls where only reads issued a block ago are outstanding, not on top of the V^T reads just issued
      if (kb + 1 < NQ) qk_block(acc2[(kb + 1) & 1], kf[(kb + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
      const bool both = kb * 32 + 16 < L;  // whether the block's upper 16 keys are inside the window
      load_v(2 * kb, vraw[0]);
      if (both) load_v(2 * kb + 1, vraw[1]);
      // Keep every accumulator of the S^T block just issued live across these reads.  Where the compiler can prove part
      // of it unused (keys past the window become -inf whatever the MFMA wrote) it would hand those registers to the
      // V^T reads, and it places no wait between an MFMA still writing a register and an assembly read returning into
      // it: the MFMA's late write would replace the V^T fragment.
      if (kb + 1 < NQ) asm volatile("" : "+v"(acc2[(kb + 1) & 1]));
      __builtin_amdgcn_sched_barrier(0);
      if (kb + 2 < NQ) load_k(kb + 2, kf[kb & 1]);
      lg.mask_block(kb, a);
#pragma unroll
      for (int h = 0; h < (both ? 8 : 4); ++h) {
        const float e0 = __builtin_amdgcn_exp2f(a[2 * h]);
        const float e1 = __builtin_amdgcn_exp2f(a[2 * h + 1]);
        pk[h] = pack_bf16x2(e0, e1);
        sum = dot2_ones(pk[h], sum);  // the row sum of what PV multiplies: the rounded values
      }
      __builtin_amdgcn_sched_barrier(0);
      if (both) load_v.ready(vraw[0], vraw[1], vf[0], vf[1]);
      else load_v.ready(vraw[0], vf[0]);
      // the accumulators of block kb are consumed: the bias of block kb + 2 goes straight into them
      if (HAS_BIAS && kb + 2 < NQ) lg.init_acc(kb + 2, a);
#pragma unroll
      for (int t2 = 0; t2 < (both ? 2 : 1); ++t2) {
        const u32x4 pw = {pk[4 * t2], pk[4 * t2 + 1], pk[4 * t2 + 2], pk[4 * t2 + 3]};
        const bf16x8 pf = __builtin_bit_cast(bf16x8, pw);
#pragma unroll
        for (int db = 0; db < DB; ++db)
          o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[t2][db], pf, (kb == 0 && t2 == 0) ? zero16 : o[db], 0, 0, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    sum += __shfl_xor(sum, 32, 64);
  }
  const bool in_range = sum >= 0x1p-40f && sum <= 0x1p100f;  // false for NaN as well
  if (__builtin_amdgcn_ballot_w64(!in_range) != 0) {
    float mrow = -INFINITY;
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
      if (pass == 1) {
        mrow = fmaxf(mrow, __shfl_xor(mrow, 32, 64));
        sum = 0.f;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int e = 0; e < 16; ++e) o[db][e] = 0.f;
      }
#pragma unroll 1
      for (int kb = 0; kb < NQ; ++kb) {
        f32x16 a;
        bf16x8 kf[KS];
        load_k(kb, kf);
        lg.init_acc(kb, a);
#pragma unroll
        for (int s2 = 0; s2 < KS; ++s2) a = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s2], qf[s2], a, 0, 0, 0);
        lg.mask_block(kb, a);
        if (pass == 0) {
#pragma unroll
          for (int e = 0; e < 16; e += 2) mrow = fmaxf(fmaxf(mrow, a[e]), a[e + 1]);
        } else {
#pragma unroll
          for (int t2 = 0; t2 < 2; ++t2) {
            if (L % 32 != 0 && kb * 32 + 16 * t2 >= L) break;
            bf16x8 vf[DB];
            typename LoadV::Raw vraw[DB];
            load_v(2 * kb + t2, vraw);
            load_v.ready(vraw, vf);
            uint32_t pk[4];
#pragma unroll
            for (int h = 0; h < 4; ++h) {
              const int h2 = 4 * t2 + h;
              pk[h] = pack_bf16x2(__builtin_amdgcn_exp2f(a[2 * h2] - mrow), __builtin_amdgcn_exp2f(a[2 * h2 + 1] - mrow));
              sum = dot2_ones(pk[h], sum);
            }
            const u32x4 pw = {pk[0], pk[1], pk[2], pk[3]};
            const bf16x8 pf = __builtin_bit_cast(bf16x8, pw);
#pragma unroll
            for (int db = 0; db < DB; ++db) o[db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[db], pf, o[db], 0, 0, 0);
          }
        }
      }
    }
    sum += __shfl_xor(sum, 32, 64);
  }
}

// Normalise and store the lane's output row: o[db][4g + i] = O[query][32 db + 8 g + 4 hi + i].  The two lanes of a
// query (l31 and l31 + 32) each hold half of every 16-byte piece of the row; v_permlane32_swap on the pieces 2m and
// 2m + 1 gives the lower lane all of piece 2m and the upper lane all of piece 2m + 1: 32 contiguous bytes per row and
// instruction.  `op` points at element hi * 8 of the row's head slice.  attention_rows_stores(DB) store
// instructions, issued by every lane for which `valid` holds.
constexpr int attention_rows_stores(int db) { return db * 2; }
template <int DB>
__device__ __forceinline__ void store_attention_rows(uint16_t* op, const f32x16 (&o)[DB], float sum, bool valid) {
  const float inv = __builtin_amdgcn_rcpf(sum);
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int m = 0; m < attention_rows_stores(1); ++m) {
      const int g0 = 2 * m, g1 = 2 * m + 1;
      const uint32_t x0 = pack_bf16x2(o[db][g0 * 4] * inv, o[db][g0 * 4 + 1] * inv);
      const uint32_t x1 = pack_bf16x2(o[db][g0 * 4 + 2] * inv, o[db][g0 * 4 + 3] * inv);
      const uint32_t y0 = pack_bf16x2(o[db][g1 * 4] * inv, o[db][g1 * 4 + 1] * inv);
      const uint32_t y1 = pack_bf16x2(o[db][g1 * 4 + 2] * inv, o[db][g1 * 4 + 3] * inv);
      const auto rx = __builtin_amdgcn_permlane32_swap(x0, y0, false, false);
      const auto ry = __builtin_amdgcn_permlane32_swap(x1, y1, false, false);
      if (valid) *reinterpret_cast<u32x4*>(op + db * 32 + m * 16) = u32x4{rx[0], ry[0], rx[1], ry[1]};
    }
}

// ---------------------------------------------------------------------------------------------
// The same arithmetic in blocks of 16 queries and 16 keys (v_mfma_f32_16x16x32_bf16, lane = l15 + 16 q4): QN query blocks of a wave
// against the window's keys, 32 a step.  Same work per cycle and LDS byte as the 32x32x16 shape at a higher clock, and a window
// whose token count is an odd multiple of 16 (12x12) has no padded keys and a last wave of one query block instead of two.
//   S^T block: acc[n][kb][i] is the logit (times log2 e) of key 16 kb + 4 q4 + i and query 16 n + l15.  The two key blocks of a
//   step, packed, are the 8 k slots of P^T for O^T = V^T P^T: keys 32 p + 4 q4 + (0..3) and 32 p + 16 + 4 q4 + (0..3); a last
//   single block is the 4 k slots of v_mfma_f32_16x16x16_bf16.
//   o[n][db][i] = O[query 16 n + l15][16 db + 4 q4 + i].
template <int WS_Y, int WS_X, bool HAS_BIAS, int PITCH = 2 * WS_X - 1>
struct WindowLogits16 {
  static constexpr int L = WS_Y * WS_X, KB = L / 16;
  static constexpr float MASK_NEG = -100.0f * 1.4426950408889634f;  // the additive -100, in the exp2 domain
  static_assert(WS_X % 4 == 0 && L % 16 == 0 && (WS_X == 8 || WS_X == 12 || WS_X == 16), "4 consecutive keys lie in one window row");
  // Where a lane's 4 keys of a block stand relative to the block's first key: one way for windows of 8 and 16 columns, for 12 one
  // per column (0, 4, 8) that a block can begin at.
  static constexpr int WAYS = WS_X == 12 ? 3 : 1;
  const unsigned char* bias_at[WAYS];
  int q4;
  bool my, mx;
  int qiy, qix, sy, sx;

  __device__ __forceinline__ WindowLogits16(const unsigned char* bias_lds, int qpos, int q4_, bool my_, bool mx_, int sy_, int sx_)
      : q4(q4_), my(my_), mx(mx_), qiy(qpos / WS_X), qix(qpos % WS_X), sy(sy_), sx(sx_) {
    const int sp = (2 * WS_Y - 2) * PITCH + 2 * WS_X - 2 - (qiy + WS_Y - 1) * PITCH - qix - (WS_X - 1);
#pragma unroll
    for (int w = 0; w < WAYS; ++w) bias_at[w] = bias_lds + (sp + rows_on(4 * w) * PITCH + column(4 * w) - 4 * w) * 16;
  }
  // of the lane's keys, the block beginning in column c0: window rows below the block's first, column
  __device__ __forceinline__ int rows_on(int c0) const { return (c0 + 4 * q4) / WS_X; }
  __device__ __forceinline__ int column(int c0) const { return (c0 + 4 * q4) % WS_X; }
  __device__ __forceinline__ f32x4 start(int kb) const {
    if (!HAS_BIAS) return f32x4{0.f, 0.f, 0.f, 0.f};
    const int r0 = kb * 16 / WS_X, c0 = kb * 16 % WS_X;
    const unsigned char* at = bias_at[0];
    if (WAYS == 3) at = c0 == 0 ? bias_at[0] : c0 == 4 ? bias_at[1 % WAYS] : bias_at[2 % WAYS];
    return *reinterpret_cast<const f32x4*>(at + (r0 * PITCH + c0) * 16);
  }
  __device__ __forceinline__ bool masked() const { return my || mx; }  // wave-uniform
  __device__ __forceinline__ void mask(int kb, f32x4& a) const {
    const int r0 = kb * 16 / WS_X, c0 = kb * 16 % WS_X;
    const int kiy = r0 + rows_on(c0), kix = column(c0);
    const bool ydiff = my && ((kiy < WS_Y - sy) != (qiy < WS_Y - sy));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool xdiff = mx && ((kix + i < WS_X - sx) != (qix < WS_X - sx));
      if (ydiff || xdiff) a[i] += MASK_NEG;
    }
  }
};

// V^T fragments of head_dim 64 from a row-major V tile whose rows (128 B) have their 16-byte chunks XOR-swizzled by 2 ((key >> 1) & 3):
// the 8 keys x 2 chunks that a 32-lane pass of the transposing read gathers lie on distinct banks.
template <class Base>
struct LoadVTransposed16 {
  static constexpr int DB = 4;
  uint32_t v_lane[DB];
  __device__ __forceinline__ LoadVTransposed16(int lane, Base base) {
    const int q4 = lane >> 4, e = (lane >> 2) & 3, a = lane & 3, row = 4 * q4 + e;
#pragma unroll
    for (int db = 0; db < DB; ++db)
      v_lane[db] = base + (uint32_t)(row * 128 + (((2 * db + (a >> 1)) ^ (2 * ((row >> 1) & 3))) << 4) + (a & 1) * 8);
  }
  // keys 16 kb .. (low half) and, of a whole step, 16 kb + 16 .. (high half)
  __device__ __forceinline__ void operator()(int kb, bool whole, TrFrag (&f)[DB]) const {
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      f[db].lo = lds_read_tr16_b64<0>(v_lane[db] + (uint32_t)kb * 2048u);
      if (whole) f[db].hi = lds_read_tr16_b64<2048>(v_lane[db] + (uint32_t)kb * 2048u);
    }
  }
};

// `load_k(kb, s)` returns K's fragment: row 16 kb + l15, 8 elements from 32 s + 8 q4; `lg[n]` are the logits' start values and mask.
// Otherwise as attention_sweep: one sweep without a row maximum, sums checked, the two-pass form for what leaves the range.
template <int QN, class Logits, class LoadK, class LoadV, class Mid>
__device__ __forceinline__ void attention_sweep16(const Logits (&lg)[QN], const LoadK& load_k, const LoadV& load_v, const Mid& mid,
                                                  const bf16x8 (&qf)[QN][2], f32x4 (&o)[QN][4], float (&sum)[QN]) {
  constexpr int KB = Logits::KB, NP = (KB + 1) / 2, DB = 4, KS = 2;
  typedef __attribute__((ext_vector_type(4))) short s16x4;
  const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
  auto blocks = [](int p) { return 2 * p + 2 <= KB ? 2 : 1; };  // key blocks of a step
  auto pv_half = [](const u32x2& v, uint32_t p0, uint32_t p1, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, v), __builtin_bit_cast(s16x4, u32x2{p0, p1}), c, 0, 0, 0);
  };
  {
    f32x4 acc[2][QN][2];
    bf16x8 kf[2][2][KS];
    auto read_k = [&](int p) {
#pragma unroll
      for (int b = 0; b < blocks(p); ++b)
#pragma unroll
        for (int s = 0; s < KS; ++s) kf[p & 1][b][s] = load_k(2 * p + b, s);
    };
    auto start = [&](int p) {
#pragma unroll
      for (int b = 0; b < blocks(p); ++b)
#pragma unroll
        for (int n = 0; n < QN; ++n) acc[p & 1][n][b] = lg[n].start(2 * p + b);
    };
    auto qk = [&](int p) {
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int b = 0; b < blocks(p); ++b)
#pragma unroll
          for (int n = 0; n < QN; ++n)
            acc[p & 1][n][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[p & 1][b][s], qf[n][s], acc[p & 1][n][b], 0, 0, 0);
    };
#pragma unroll
    for (int n = 0; n < QN; ++n) sum[n] = 0.f;
    read_k(0);
    start(0);
    if (NP > 1) {
      read_k(1);
      start(1);
    }
    TrFrag vraw[DB];
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), see below
    __builtin_amdgcn_sched_barrier(0);
    load_v(0, KB > 1, vraw);
    __builtin_amdgcn_sched_barrier(0);
    qk(0);
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const bool whole = blocks(p) == 2;
      __builtin_amdgcn_sched_barrier(0);
      mid(p);
      // This step's V^T reads, then the next step's S^T.  The K fragments and bias vectors of the latter, requested a step ago, are waited
      // for ahead of the reads: the compiler's own wait would count the assembly reads in.  (Behind the MFMAs the reads could return into
      // registers that the first of two MFMAs on an accumulator is still writing: the shape's chains need not stay in one register.)
      if (p > 0) {
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __builtin_amdgcn_sched_barrier(0);
        load_v(2 * p, whole, vraw);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (p + 1 < NP) qk(p + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (p + 2 < NP) read_k(p + 2);
      if (lg[0].masked()) {
#pragma unroll
        for (int n = 0; n < QN; ++n)
#pragma unroll
          for (int b = 0; b < (whole ? 2 : 1); ++b) lg[n].mask(2 * p + b, acc[p & 1][n][b]);
      }
      uint32_t pk[QN][4];
#pragma unroll
      for (int n = 0; n < QN; ++n)
#pragma unroll
        for (int b = 0; b < (whole ? 2 : 1); ++b) {
          const f32x4& a = acc[p & 1][n][b];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            pk[n][2 * b + h] = pack_bf16x2(__builtin_amdgcn_exp2f(a[2 * h]), __builtin_amdgcn_exp2f(a[2 * h + 1]));
            sum[n] = dot2_ones(pk[n][2 * b + h], sum[n]);  // the row sum of what PV multiplies: the rounded values
          }
        }
      __builtin_amdgcn_sched_barrier(0);
      if (whole) lds_tr_wait(vraw[0], vraw[1], vraw[2], vraw[3]);
      else asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(vraw[0].lo), "+v"(vraw[1].lo), "+v"(vraw[2].lo), "+v"(vraw[3].lo));
      if (p + 2 < NP) start(p + 2);
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int n = 0; n < QN; ++n) {
          const f32x4 c = p == 0 ? zero4 : o[n][db];
          if (whole)
            o[n][db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(tr_frag_value(vraw[db]), __builtin_bit_cast(bf16x8, u32x4{pk[n][0], pk[n][1], pk[n][2], pk[n][3]}), c, 0, 0, 0);
          else
            o[n][db] = pv_half(vraw[db].lo, pk[n][0], pk[n][1], c);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  bool out_of_range = false;
#pragma unroll
  for (int n = 0; n < QN; ++n) {
    sum[n] += __shfl_xor(sum[n], 16, 64);
    sum[n] += __shfl_xor(sum[n], 32, 64);
    out_of_range = out_of_range || !(sum[n] >= 0x1p-40f && sum[n] <= 0x1p100f);  // true for NaN as well
  }
  if (__builtin_amdgcn_ballot_w64(out_of_range) != 0) {
    float m[QN];
#pragma unroll
    for (int n = 0; n < QN; ++n) m[n] = -INFINITY;
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass) {
      if (pass == 1) {
#pragma unroll
        for (int n = 0; n < QN; ++n) {
          m[n] = fmaxf(m[n], __shfl_xor(m[n], 16, 64));
          m[n] = fmaxf(m[n], __shfl_xor(m[n], 32, 64));
          sum[n] = 0.f;
#pragma unroll
          for (int db = 0; db < DB; ++db) o[n][db] = zero4;
        }
      }
#pragma unroll 1
      for (int kb = 0; kb < KB; ++kb) {
        f32x4 a[QN];
#pragma unroll
        for (int n = 0; n < QN; ++n) a[n] = lg[n].start(kb);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          const bf16x8 f = load_k(kb, s);
#pragma unroll
          for (int n = 0; n < QN; ++n) a[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f, qf[n][s], a[n], 0, 0, 0);
        }
        if (lg[0].masked()) {
#pragma unroll
          for (int n = 0; n < QN; ++n) lg[n].mask(kb, a[n]);
        }
        if (pass == 0) {
#pragma unroll
          for (int n = 0; n < QN; ++n) m[n] = fmaxf(fmaxf(fmaxf(m[n], a[n][0]), fmaxf(a[n][1], a[n][2])), a[n][3]);
        } else {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int n = 0; n < QN; ++n) asm volatile("s_nop 15\n\ts_nop 15" : "+v"(a[n]));  // (no MFMA is writing a register when the reads below are issued)
          TrFrag vraw[DB];
          load_v(kb, false, vraw);
          asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(vraw[0].lo), "+v"(vraw[1].lo), "+v"(vraw[2].lo), "+v"(vraw[3].lo));
#pragma unroll
          for (int n = 0; n < QN; ++n) {
            uint32_t pk[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
              pk[h] = pack_bf16x2(__builtin_amdgcn_exp2f(a[n][2 * h] - m[n]), __builtin_amdgcn_exp2f(a[n][2 * h + 1] - m[n]));
              sum[n] = dot2_ones(pk[h], sum[n]);
            }
#pragma unroll
            for (int db = 0; db < DB; ++db) o[n][db] = pv_half(vraw[db].lo, pk[0], pk[1], o[n][db]);
          }
        }
      }
    }
#pragma unroll
    for (int n = 0; n < QN; ++n) {
      sum[n] += __shfl_xor(sum[n], 16, 64);
      sum[n] += __shfl_xor(sum[n], 32, 64);
    }
  }
}

// Normalise and store a query block's rows: v_permlane16_swap on the pieces of row blocks 2m and 2m + 1 leaves lane (l15, q4) with 8
// consecutive elements, 32 m + 16 (q4 & 1) + 8 (q4 >> 1) .., of row l15: 64 contiguous bytes per row and instruction.  `op` points at the
// row's head slice.  ATTENTION_ROWS16_STORES store instructions, issued by every lane for which `valid` holds.
constexpr int ATTENTION_ROWS16_STORES = 2;
__device__ __forceinline__ void store_attention_rows16(uint16_t* op, const f32x4 (&o)[4], float sum, int q4, bool valid) {
  const float inv = __builtin_amdgcn_rcpf(sum);
  static_assert(ATTENTION_ROWS16_STORES * 32 == 64, "head_dim 64 in pieces of 32 elements");
#pragma unroll
  for (int m = 0; m < ATTENTION_ROWS16_STORES; ++m) {
    const f32x4 a = o[2 * m] * inv, b = o[2 * m + 1] * inv;
    const auto rx = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[0], a[1]), pack_bf16x2(b[0], b[1]), false, false);
    const auto ry = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[2], a[3]), pack_bf16x2(b[2], b[3]), false, false);
    if (valid) *reinterpret_cast<u32x4*>(op + 32 * m + 16 * (q4 & 1) + 8 * (q4 >> 1)) = u32x4{rx[0], ry[0], rx[1], ry[1]};
  }
}

}  // namespace aeris
