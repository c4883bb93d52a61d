// bf16 MFMA GEMM for gfx950:  C[M,N] = epilogue(A[M,K] * W[N,K]^T), one output tile per workgroup
//
// For the problems that do not give the 256 x 256 persistent kernel (gemm_persistent.hip) enough tiles to fill the chip.
// What bounds those is latency: a handful of k-tiles per workgroup, each a round trip to L2, and the first loads and the
// epilogue on top of them.  Hence 64 x 64 tiles (four waves of 32 x 32, 48 KB of LDS: three workgroups per CU, free of each
// other, so one's first loads and epilogue fall under another's main loop; 32 x 64 where there are not enough of those, and two
// k-tiles where that lets a fourth run: launch_kind), three k-tiles in flight, every epilogue
// operand requested ahead of the main loop, and little code (fetched cold: the kernel before this one, 128 x 128
// register-staged with every epilogue option in one body, took 18-24 us for what takes 4-5 us here).  Measured before -> after:
// 2048 x 128 x 128 17.9 -> 3.4 us, 2048 x 128 x 512 22.1 -> 4.2 us, 2048 x 256 x 1024 32.1 -> 5.8 us, 8192 x 256 x 256 25.0 ->
// 6.8 us.  128 x 128 tiles of the same kernel take what neither this size nor the persistent kernel can (odd N, unaligned
// rows, W of 2 GiB and more, SiLU).
//   - global loads go straight into LDS (buffer_load ... lds, 16 bytes per lane); a load instruction of a wave fetches
//     8 rows x 128 B and the lane -> chunk map is the inverse of the LDS swizzle (swz_off), so fragment reads are
//     conflict-free ds_read_b128 and nothing is staged through registers
//   - STAGES k-tiles of 64 in LDS, one barrier per k-tile: the loads of k-tile j + STAGES - 1 are issued right behind the
//     barrier that ends the reading of k-tile j - 1 (tiles of 64: and the fragment reads of k-tile j), and waited for with a
//     counted vmcnt
//   - v_mfma_f32_16x16x32_bf16 with the weight fragment first and accumulators that start at the bias: the same
//     arithmetic in the same order as the persistent kernel, bit for bit
//   - the epilogue works on the accumulators where they are: a lane holds 4 consecutive n of one row; for bf16 C two column
//     fragments are swapped between lane rows (v_permlane16_swap) into 8 consecutive n, 16 bytes.  No LDS staging: the
//     64-byte row pieces cost store bandwidth, which the other workgroup's main loop hides, and a short epilogue
//     matters more here - the kernels this file is for run a few microseconds, and code that is fetched cold counts
//   - blockIdx is remapped so that each XCD (blockIdx % 8) works on a contiguous range of tiles, groups of GM row panels
//     x all column tiles, which keeps the panels in use in that XCD's L2
// Epilogue (all optional, fused): + bias[n], GELU / SiLU / SwiGLU, * gate[b, n], + residual[m, n].
#include "common.h"
#include "gemm_common.h"
#include "kernels.h"

namespace aeris {

namespace {
constexpr int BK = 64;
constexpr int NT = 256;
constexpr int GM = 8;  // row panels per L2 group

// a b + c with both results rounded
__device__ __forceinline__ float mul_add_rounded(float a, float b, float c) {
#pragma clang fp contract(off)
  const float ab = a * b;
  return ab + c;
}

// ends a wave's use of a k-tile: its LDS reads have returned, all but its n newest loads have arrived, then the barrier
// (one asm statement: nothing the compiler schedules may come between, and no LDS access may cross it)
template <int N>
__device__ __forceinline__ void wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
}  // namespace

// VEC: C and the residual are accessed 4 / 8 columns at a time (N % 4 == 0, rows 4-element aligned); else one by one
// BM 32, 64 or 128: of 32 rows a wave computes 16 x 32 of the tile and loads one block of A
template <int BM, int BN, int STAGES, int ACT, bool OUT_F32, bool VEC>
__global__ void __launch_bounds__(NT, 2) gemm_bf16_nt_tile_kernel(GemmParams p) {
  constexpr bool SWIGLU = ACT == AERIS_ACT_SWIGLU;
  constexpr int FM = BM / 32, FN = BN / 32;  // 16 x 16 fragments per wave (2 x 2 waves)
  constexpr int A_BYTES = BM * BK * 2, B_BYTES = BN * BK * 2, STAGE = A_BYTES + B_BYTES;
  constexpr int A_LD = BM / 32, B_LD = BN / 32;  // load instructions of a wave per k-tile (8 rows each)
  constexpr int LPT = A_LD + B_LD;
  constexpr int BN_OUT = SWIGLU ? BN / 2 : BN;
  constexpr int NJ = SWIGLU ? FN / 2 : FN;  // column fragments of the output
  static_assert(BM % 32 == 0 && BN % 64 == 0 && STAGES >= 2 && (STAGES - 2) * LPT < 64, "tile shape");
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];

  // ---- tile of this workgroup: XCD-contiguous remap, then groups of GM row panels x all column tiles
  int pid = blockIdx.x;
  {
    const int np = gridDim.x;
    const int per = (np + 7) >> 3;
    int tall = np & 7;
    if (tall == 0) tall = 8;
    const int xcd = pid & 7, loc = pid >> 3;
    pid = (xcd < tall) ? xcd * per + loc : tall * per + (xcd - tall) * (per - 1) + loc;
  }
  int tile_m, tile_n;
  {
    const int gsz = GM * p.tiles_n;
    const int grp = pid / gsz, within = pid - grp * gsz;
    int gm = p.tiles_m - grp * GM;
    if (gm > GM) gm = GM;
    tile_n = within / gm;
    tile_m = grp * GM + (within - tile_n * gm);
  }
  const int64_t m0 = (int64_t)tile_m * BM;
  const int n0 = tile_n * BN_OUT;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int l15 = lane & 15, q = lane >> 4;
  const int K = p.K, N = p.N;
  const int KT = K / BK;

  // ---- loads: a wave brings in BM / 4 rows of A and BN / 4 rows of W per k-tile.  Rows past the end of A or W are
  // outside the descriptors (size in bytes: whole rows) and arrive as zeros; they feed only what is never stored.
  constexpr int AR = BM / 4, BR = BN / 4;
  // (The range check covers both parts of an offset, the per-lane one and the k-tile's: a byte k < 2 K of row r is at 2 K r + k, past
  // the end exactly for the rows past the end.)
  constexpr int LD_MAX = A_LD > B_LD ? A_LD : B_LD;
  uint32_t ld_voff[LD_MAX];  // lane part of the source offset, per 8-row block
  uint32_t a_voff0;          // of A's first block: tiles of 32 rows have one a wave, odd in the odd waves
  {
    const int dr = lane >> 4, pos = lane & 15;
    auto voff = [&](int i, int odd) {
      const int logical = pos ^ (odd * 4 + dr);
      return (uint32_t)((i * 8 + dr * 2 + (logical >> 3)) * K * 2 + (logical & 7) * 16);
    };
#pragma unroll
    for (int i = 0; i < LD_MAX; ++i) ld_voff[i] = voff(i, i & 1);
    a_voff0 = A_LD == 1 ? voff(0, wave & 1) : ld_voff[0];
  }
  auto rows_rsrc = [&](const uint16_t* base, int64_t row, int64_t limit, int count) {
    int64_t have = limit - row;
    if (have > count) have = count;
    if (have < 0) { have = 0; row = 0; }
    return make_lds_dma_rsrc(base + row * K, (uint32_t)(have * K * 2));
  };
  const lds_dma_rsrc rs_a = rows_rsrc(p.A, m0 + wave * AR, p.M, AR);
  // SwiGLU: a wave column's BN / 2 tile rows are the gate rows, then the up rows, of BN / 4 output columns
  const int w_out = n0 + (SWIGLU ? (wave >> 1) : wave) * BR;
  const int64_t w_first = (SWIGLU ? (int64_t)(wave & 1) * N : 0) + w_out;
  const lds_dma_rsrc rs_w = rows_rsrc(p.W, w_first, w_out < N ? w_first + (N - w_out) : w_first, BR);
  const uint32_t lds0 = lds_byte_address(smem);
  auto issue = [&](int kt, int stage) {
    const uint32_t sa = lds0 + stage * STAGE + wave * (AR * 128), sw = lds0 + stage * STAGE + A_BYTES + wave * (BR * 128);
    const uint32_t k_off = (uint32_t)kt * (BK * 2);
#pragma unroll
    for (int i = 0; i < A_LD; ++i) lds_dma_load16(rs_a, sa + i * 1024, i == 0 ? a_voff0 : ld_voff[i], k_off);
#pragma unroll
    for (int i = 0; i < B_LD; ++i) lds_dma_load16(rs_w, sw + i * 1024, ld_voff[i], k_off);
  };

  // ---- per-column and (small tiles) per-element operands are requested ahead of the first k-tile: their latency is
  // that of the first loads instead of a second one at the end
  const int n_w = n0 + wn * (BN_OUT / 2);  // first output column of this wave
  f32x4 acc[FM][FN];
  u32x2 bq[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    bq[j] = u32x2{0u, 0u};
    if (p.bias) {
      const uint16_t* b = p.bias + (SWIGLU && j >= NJ ? N : 0);
      const int n = n_w + (SWIGLU ? j % NJ : j) * 16 + q * 4;
      if (VEC) {
        bq[j] = *reinterpret_cast<const u32x2*>(b + (n < N ? n : N - 4));
      } else {
        uint32_t h[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) h[e] = b[n + e < N ? n + e : N - 1];
        bq[j] = u32x2{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
      }
    }
  }
  const int m_w = wm * (BM / 2);  // first row of this wave in the tile
  const int rows = (int)(p.M - m0 < BM ? p.M - m0 : BM);
  const int64_t rs = c_row_stride(p);
  // residual of fragment (i, j), f32 or bf16, at this lane's 4 columns
  auto load_res = [&](int i, int j) -> u32x4 {
    int r = m_w + i * 16 + l15, n = n_w + j * 16 + q * 4;
    if (r > rows - 1) r = rows - 1;  // rows and columns outside the matrix: any valid address, the values are not stored
    if (n > N - 4) n = N - 4;
    const int64_t off = (m0 + r) * p.ldc + n;
    if (p.res_dtype == AERIS_F32) return *reinterpret_cast<const u32x4*>(reinterpret_cast<const float*>(p.residual) + off);
    const u32x2 h = *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint16_t*>(p.residual) + off);
    return u32x4{h.x << 16, h.x & 0xffff0000u, h.y << 16, h.y & 0xffff0000u};
  };
  u32x4 res[VEC ? FM : 1][VEC ? NJ : 1];
  auto load_all_res = [&]() {
    if (p.res_dtype < 0) return;
    if (p.res_dtype == AERIS_F32) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) res[VEC ? i : 0][VEC ? j : 0] = load_res(i, j);
    } else {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) res[VEC ? i : 0][VEC ? j : 0] = load_res(i, j);
    }
  };
  constexpr bool RES_EARLY = VEC && FM * NJ <= 4;
  if (RES_EARLY) load_all_res();
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < KT) issue(s, s);
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const f32x4 b = {bf16_lo(bq[j].x), bf16_hi(bq[j].x), bf16_lo(bq[j].y), bf16_hi(bq[j].y)};
#pragma unroll
    for (int i = 0; i < FM; ++i) acc[i][j] = b;
  }

  // ---- main loop
  uint32_t a_roff[2], b_roff[2];  // fragment read offsets per k-step of 32
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    a_roff[ks] = swz_off(m_w + l15, ks * 4 + q);
    b_roff[ks] = A_BYTES + swz_off(wn * (BN / 2) + l15, ks * 4 + q);
  }
  int rd = 0, wr = STAGES - 1;
  for (int kt = 0; kt < KT; ++kt) {
    // k-tile kt has arrived when at most the loads of the min(STAGES - 2, KT - 1 - kt) k-tiles behind it are outstanding
    const int behind = KT - 1 - kt;
    static_assert(STAGES <= 4, "one more wait per further stage");
    if (STAGES > 2 && behind >= STAGES - 2) wait_barrier<(STAGES - 2) * LPT>();
    else if (STAGES > 3 && behind == 1) wait_barrier<LPT>();
    else wait_barrier<0>();
    const unsigned char* st = smem + rd * STAGE;
    // Tiles of 64: the loads come behind the fragment reads: each holds the wave for 70-95 cycles, in which the fragments arrive.  (The
    // serial chain of a k-tile, not the latency of its loads, is what a small problem waits for: four, six or nine k-tiles in flight
    // instead of three measured the same or slower.  Loads first -> reads first: 2048 x 256 x 1024 8.0 -> 7.1 us, 2048 x 512 x 2048
    // 13.0 -> 10.9; 2048 x 128 x 128 the same.)  With two stages, tiles of 128, the one k-tile ahead is requested at once: reads
    // first, 2048 x 1538 x 1536 25.2 -> 26.6 us, 4096 x 4098 x 4096 167 -> 174, SiLU 3000 x 3072 x 1024 31.4 -> 33.4 (but
    // 1000 x 1002 x 1024, 64 tiles in all, 17.1 -> 16.4).
    constexpr bool READS_FIRST = STAGES > 2;
    constexpr int STEPS = READS_FIRST ? 2 : 1;  // k-steps of 32 whose fragments are held at once
    if (!READS_FIRST && behind >= STAGES - 1) issue(kt + STAGES - 1, wr);
#pragma unroll
    for (int k0 = 0; k0 < 2; k0 += STEPS) {
      bf16x8 af[STEPS][FM], bf[STEPS][FN];
#pragma unroll
      for (int ks = 0; ks < STEPS; ++ks) {
#pragma unroll
        for (int i = 0; i < FM; ++i) af[ks][i] = *reinterpret_cast<const bf16x8*>(st + a_roff[k0 + ks] + i * 16 * 128);
#pragma unroll
        for (int j = 0; j < FN; ++j) bf[ks][j] = *reinterpret_cast<const bf16x8*>(st + b_roff[k0 + ks] + j * 16 * 128);
      }
      if (READS_FIRST && behind >= STAGES - 1) issue(kt + STAGES - 1, wr);
#pragma unroll
      for (int ks = 0; ks < STEPS; ++ks)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[ks][j], af[ks][i], acc[i][j], 0, 0, 0);
    }
    if (++rd == STAGES) rd = 0;
    if (++wr == STAGES) wr = 0;
  }

  // ---- epilogue
  if (VEC && !RES_EARLY) load_all_res();
  if (p.q_cols > n_w) {  // query part of a qkv projection: scaled in fp32 ahead of its only rounding
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float s = n_w + j * 16 + q * 4 + e < p.q_cols ? p.q_scale : 1.0f;
#pragma unroll
        for (int i = 0; i < FM; ++i) acc[i][j][e] *= s;
      }
  }
  // gate row of tile row r: the tile's first row is in batch entry b0, row `g_off` of it
  const float* gate0 = p.gate;
  int64_t g_off = 0;
  if (p.gate && p.gate_batch_stride) {
    const int64_t b0 = (p.row0 + m0) / p.rows_per_batch;
    g_off = p.row0 + m0 - b0 * p.rows_per_batch;
    gate0 += b0 * p.gate_batch_stride;
  }
  auto gate_row = [&](int r) -> const float* {
    if (!p.gate_batch_stride) return gate0;
    const int64_t in = g_off + r;
    if (in < p.rows_per_batch) return gate0;
    // (a tile spans further entries only when an entry has fewer rows than a tile: small numbers then)
    return gate0 + (in < 2 * p.rows_per_batch ? 1 : (int64_t)((uint32_t)in / (uint32_t)p.rows_per_batch)) * p.gate_batch_stride;
  };
  auto activated = [&](int i, int j, float (&v)[4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float x = acc[i][j][e];
      if (SWIGLU) x = silu_f(x) * acc[i][j + NJ][e];
      else if (ACT == GEMM_ACT_GELU_ERF) x = gelu_erf_bf16_f(x);
      else if (ACT == AERIS_ACT_GELU) x = OUT_F32 ? gelu_erf_f(x) : gelu_bf16_f(x);
      else if (ACT == AERIS_ACT_SILU) x = silu_f(x);
      v[e] = x;
    }
  };
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int r = m_w + i * 16 + l15;
    const bool row_ok = r < rows;
    const float* gr = p.gate ? gate_row(row_ok ? r : rows - 1) : nullptr;
    float v[NJ][4];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      activated(i, j, v[j]);
      const int n = n_w + j * 16 + q * 4;
      if (VEC) {
        f32x4 g = {1.f, 1.f, 1.f, 1.f};
        if (p.gate) g = *reinterpret_cast<const f32x4*>(gr + (n < N ? n : N - 4));
        if (p.res_dtype >= 0) {
          const u32x4 x = res[VEC ? i : 0][VEC ? j : 0];
          if (p.row0) {  // the last rows of a call whose others have the persistent kernel: rounded once, as there
#pragma unroll
            for (int e = 0; e < 4; ++e) v[j][e] = fmaf(v[j][e], g[e], __uint_as_float(x[e]));
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[j][e] = mul_add_rounded(v[j][e], g[e], __uint_as_float(x[e]));
          }
        } else if (p.gate) {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[j][e] *= g[e];
        }
      } else {
        const int64_t off = (m0 + r) * rs + c_col_off(p, n);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (row_ok && n + e < N) {
            float x = v[j][e];
            if (p.gate) x *= gr[n + e];
            if (p.res_dtype == AERIS_BF16) x += bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p.residual)[off + e]);
            else if (p.res_dtype == AERIS_F32) x += reinterpret_cast<const float*>(p.residual)[off + e];
            if (OUT_F32) reinterpret_cast<float*>(p.C)[off + e] = x;
            else reinterpret_cast<uint16_t*>(p.C)[off + e] = (uint16_t)f32_to_bf16_bits(x);
          }
        }
      }
    }
    if (!VEC) continue;
    if (OUT_F32) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const int n = n_w + j * 16 + q * 4;
        if (row_ok && n < N)
          *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.C) + (m0 + r) * rs + c_col_off(p, n)) =
              f32x4{v[j][0], v[j][1], v[j][2], v[j][3]};
      }
    } else if (NJ == 1) {
      const int n = n_w + q * 4;
      if (row_ok && n < N)
        *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(p.C) + (m0 + r) * rs + c_col_off(p, n)) =
            u32x2{pack_bf16x2(v[0][0], v[0][1]), pack_bf16x2(v[0][2], v[0][3])};
    } else {
      // lane (l15, q) of the swapped pair of column fragments 2 m, 2 m + 1 holds the columns 32 m + 16 (q & 1) + 8 (q >> 1) ..
#pragma unroll
      for (int m = 0; m < NJ / 2; ++m) {
        const auto x = __builtin_amdgcn_permlane16_swap(pack_bf16x2(v[2 * m][0], v[2 * m][1]), pack_bf16x2(v[2 * m + 1][0], v[2 * m + 1][1]), false, false);
        const auto y = __builtin_amdgcn_permlane16_swap(pack_bf16x2(v[2 * m][2], v[2 * m][3]), pack_bf16x2(v[2 * m + 1][2], v[2 * m + 1][3]), false, false);
        const int n = n_w + 32 * m + 16 * (q & 1) + 8 * (q >> 1);
        if (row_ok && n < N) {
          // N % 4 == 0: 8 columns are whole or exactly their first half is inside
          uint16_t* c = reinterpret_cast<uint16_t*>(p.C) + (m0 + r) * rs + c_col_off(p, n);
          if (n + 8 <= N) *reinterpret_cast<u32x4*>(c) = u32x4{x[0], y[0], x[1], y[1]};
          else *reinterpret_cast<u32x2*>(c) = u32x2{x[0], y[0]};
        }
      }
    }
  }
}

namespace {

template <int BM, int BN, int STAGES, int ACT, bool OUT_F32, bool VEC>
hipError_t launch_tile(const GemmParams& p0, hipStream_t stream) {
  GemmParams p = p0;
  constexpr int BN_OUT = ACT == AERIS_ACT_SWIGLU ? BN / 2 : BN;
  const int64_t tiles_m = (p.M + BM - 1) / BM;
  p.tiles_n = (p.N + BN_OUT - 1) / BN_OUT;
  p.tiles_m = (int)tiles_m;
  constexpr int smem = STAGES * (BM + BN) * BK * 2;
  hipLaunchKernelGGL((gemm_bf16_nt_tile_kernel<BM, BN, STAGES, ACT, OUT_F32, VEC>), dim3((unsigned)(tiles_m * p.tiles_n)), dim3(NT), smem, stream, p);
  return hipGetLastError();
}

// SiLU has tiles of 64 x 64 below 128 of 128 x 128 only, fewer than 512: never the two-stage ones (launch_kind)
constexpr bool takes_silu(int bm, int stages) { return !(bm == 64 && stages == 2); }

template <int BM, int BN, int STAGES, bool VEC>
hipError_t launch_tile_act(const GemmParams& p, hipStream_t stream) {
#define GO(A)                                                                              \
  return p.c_dtype == AERIS_F32 ? launch_tile<BM, BN, STAGES, A, true, VEC>(p, stream) \
                                : launch_tile<BM, BN, STAGES, A, false, VEC>(p, stream)
  switch (p.act) {
    case AERIS_ACT_GELU:
      if (p.c_dtype == AERIS_F32) return launch_tile<BM, BN, STAGES, AERIS_ACT_GELU, true, VEC>(p, stream);
      // the polynomial: only as the last rows of a problem whose other rows take it, which are given to 64 x 64 tiles
      return launch_tile<BM, BN, STAGES, BM <= 64 ? AERIS_ACT_GELU : GEMM_ACT_GELU_ERF, false, VEC>(p, stream);
    case GEMM_ACT_GELU_ERF: return launch_tile<BM, BN, STAGES, GEMM_ACT_GELU_ERF, false, VEC>(p, stream);
    case AERIS_ACT_SWIGLU: GO(AERIS_ACT_SWIGLU);
    case AERIS_ACT_SILU:
      if constexpr (takes_silu(BM, STAGES)) GO(AERIS_ACT_SILU);
      return hipErrorInvalidValue;
    default: GO(AERIS_ACT_NONE);
  }
#undef GO
}

template <int BM, int BN, int STAGES, bool VEC, int ACT, bool OUT_F32>
hipError_t configure_tile_kernel() {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_bf16_nt_tile_kernel<BM, BN, STAGES, ACT, OUT_F32, VEC>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, STAGES * (BM + BN) * BK * 2);
}
template <int BM, int BN, int STAGES, bool VEC, int ACT>
hipError_t configure_tile_act() {
  const hipError_t e = configure_tile_kernel<BM, BN, STAGES, VEC, ACT, false>();
  return e != hipSuccess ? e : configure_tile_kernel<BM, BN, STAGES, VEC, ACT, true>();
}
template <int BM, int BN, int STAGES, bool VEC>
hipError_t configure_tile() {
  hipError_t e = configure_tile_act<BM, BN, STAGES, VEC, AERIS_ACT_NONE>();
  if (e == hipSuccess) e = configure_tile_kernel<BM, BN, STAGES, VEC, AERIS_ACT_GELU, true>();
  if (e == hipSuccess) e = configure_tile_kernel<BM, BN, STAGES, VEC, BM <= 64 ? AERIS_ACT_GELU : GEMM_ACT_GELU_ERF, false>();
  if (e == hipSuccess) e = configure_tile_kernel<BM, BN, STAGES, VEC, GEMM_ACT_GELU_ERF, false>();
  if (e == hipSuccess) e = configure_tile_act<BM, BN, STAGES, VEC, AERIS_ACT_SWIGLU>();
  if constexpr (takes_silu(BM, STAGES)) {
    if (e == hipSuccess) e = configure_tile_act<BM, BN, STAGES, VEC, AERIS_ACT_SILU>();
  }
  return e;
}
}  // namespace

// touch every instantiation so that attribute set-up never happens inside a captured region
hipError_t gemm_configure_all() {
  hipError_t e = configure_tile<64, 64, 3, true>();
  if (e == hipSuccess) e = configure_tile<64, 64, 2, true>();
  if (e == hipSuccess) e = configure_tile<32, 64, 3, true>();
  if (e == hipSuccess) e = configure_tile<128, 128, 2, true>();
  if (e == hipSuccess) e = configure_tile<128, 128, 2, false>();
  if (e == hipSuccess) e = gemm_persistent_configure();
  return e;
}

namespace {

// ---- which kernel: the one whose estimated time is the smallest.
// The estimates are fits, in microseconds, to 50 shapes measured on one GPU (M 2048 .. 1 036 800, N 128 .. 6144, K 128 ..
// 6144, every epilogue; calls replayed from a HIP graph) of the quantities that decide: how many rounds of tiles the
// busiest CU works through, the k-tiles of a tile, an epilogue term per tile.  They need to order the kernels, not to be
// exact.  Measured (estimated) us, f32 C with gate and residual:
//        M,    N,    K   256-row tiles  128-row tiles  64 x 64 tiles
//     2048,  256, 1024      22.8 (32)      16.3 (21)      7.7  (9)    32 small tiles on an empty chip: the shortest k-tile
//     8192,  256, 1024      24.3 (32)      17.7 (21)     11.0 (13)    two small workgroups per CU
//     8192, 1024, 1024      29.2 (32)      26.0 (22)     34.5 (41)    256 tiles of 128 rows: one round
//     8192, 1536, 1536      43.7 (42)      50.1 (53)     64.6 (79)    192 tiles of 256 rows: one round
//    14400, 1536, 6144     259  (269)     264  (264)    497  (570)    342 tiles of 256 rows: two rounds
// (Over 740 shapes, M 1024 .. 54 000, N 192 .. 6144, K 192 .. 6144, every epilogue, all forms timed: the choice takes 1.0 % longer than the
// fastest form on average, more than 5 % at 56 of them, 22 % at most: 2500 x 2048 x 256 with bf16 residual 11.9 us in small tiles, 9.8 in
// tiles of 128 rows; GELU the other way, 4096 x 1152 x 1024 20.8 against 18.2 in small tiles, whose estimate is from before they had 32 rows
// or two stages.)
//
// Tiles of 192 columns take 0.85-0.95 of the time of those of 256 for three quarters of the work, so they pay only where they need
// no more rounds: N just over a multiple of 256, or a last round that is mostly empty.  256 -> 192 columns of the same height, us:
//   256 rows   8192 x 1536 x 1536 (f32 C and residual) 42.4 -> 41.3, x 6144 117.3 -> 114.8; 9000 x 1152 x 1152 33.5 -> 31.4; 14400 x 1536 x 1536
//              82.0 -> 70.7; 10000 x 2304 x 768 (bf16) 38.1 -> 32.1; 51840 x 320 x 1280 (bf16 residual) 53.0 -> 49.4; 32768 x 576 x 192 (bf16)
//              16.8 -> 15.2
//   128 rows   12480 x 384 x 384 (f32) 13.3 -> 12.6, x 1088 21.4 -> 20.1, 30000 x 576 x 576 38.5 -> 36.5 (256 rows: 43.1 -> 37.6)
//   more rounds: 64800 x 1536 x 512 87.6 -> 101, 64800 x 512 x 2048 (bf16 residual) 113 -> 135
// A bf16 residual is read in 64-byte pieces there, which short products wait for (51840 x 320 x 320 24.2 -> 25.0).
enum Kind { TILE64, PERSISTENT128, PERSISTENT256, PERSISTENT128_192, PERSISTENT256_192 };

struct Shape {
  int64_t M;
  int N, KT, act;
  bool f32, res, w192[2];  // w192: tiles of 128 / 256 rows x 192 columns take the problem
};

float epilogue_us(const Shape& s) {  // of a 256 x 256 tile
  return s.f32 ? 8.0f : s.act == GEMM_ACT_GELU_ERF ? 9.0f : s.act == AERIS_ACT_GELU ? 6.5f : s.res || s.act == AERIS_ACT_SWIGLU ? 6.0f : 4.5f;
}

int64_t tiles_of(const Shape& s, int bm, int bn) {
  const int bn_out = s.act == AERIS_ACT_SWIGLU ? bn / 2 : bn;
  return ((s.M + bm - 1) / bm) * ((s.N + bn_out - 1) / bn_out);
}

float estimate_us(Kind kind, const Shape& s) {
  if (kind == TILE64) {
    // n workgroups per CU, up to three of them resident: a k-tile takes 0.31 us with one resident, 0.49 with two, 0.66 with three
    const float n = (float)((tiles_of(s, 64, 64) + 255) / 256);
    const float per_k = n <= 3.f ? 0.15f + 0.17f * n : 0.22f * n;
    return 3.0f + s.KT * per_k + n * (s.f32 ? 1.0f : 0.5f);
  }
  if (kind == PERSISTENT128_192 || kind == PERSISTENT256_192) {
    const bool tall = kind == PERSISTENT256_192;
    const int bm = tall ? 256 : 128;
    auto rounds = [&](int bn) { return ((tiles_of(s, bm, bn) + 7) / 8 + 31) / 32; };
    if (!s.w192[tall] || rounds(192) > rounds(256) || (s.res && !s.f32 && s.KT < 16)) return 1e30f;
    return (s.f32 ? (tall ? 0.93f : 0.88f) : 0.95f) * estimate_us(tall ? PERSISTENT256 : PERSISTENT128, s);
  }
  const int bm = kind == PERSISTENT256 ? 256 : 128;
  const int64_t per_xcd = (tiles_of(s, bm, 256) + 7) / 8;
  const float rounds = (float)((per_xcd + 31) / 32);
  return bm == 256 ? 3.0f + rounds * (1.30f * s.KT + epilogue_us(s))
                   : 3.0f + rounds * (0.86f * s.KT + 0.5f * epilogue_us(s) + 0.5f);
}

Kind best_kind(const Shape& s, float* us) {
  Kind best = TILE64;
  *us = estimate_us(TILE64, s);
  for (Kind k : {PERSISTENT128, PERSISTENT256, PERSISTENT128_192, PERSISTENT256_192}) {
    const float t = estimate_us(k, s);
    if (t < *us) { *us = t; best = k; }
  }
  return best;
}

Shape shape_of(const GemmParams& p, int act) {
  return {p.M, p.N, p.K / BK, act, p.c_dtype == AERIS_F32, p.residual != nullptr, {gemm_persistent_takes_192(p, 128), gemm_persistent_takes_192(p, 256)}};
}

hipError_t launch_kind(Kind kind, const GemmParams& p, hipStream_t stream) {
  if (kind == TILE64) {
    // Three stages are 48 KB: three workgroups per CU.  Of four per CU the last would have the chip nearly to itself: with two stages
    // (32 KB) all four run at once.  Three stages -> two, us, plain bf16: 3000 x 1152 x 384 (846 tiles) 10.3 -> 9.0, 6144 x 576 x 192
    // (864) 8.7 -> 7.1, 4096 x 960 x 320 (960) 9.7 -> 8.5, 8192 x 512 x 2048 (1024) 28.4 -> 27.0; SwiGLU 2048 x 1024 x 256 (1024) 7.2 -> 6.4.
    // With up to three per CU the third stage is worth 0 to 20 % (4096 x 512 x 2048, two per CU, 15.7 against 18.8), from five on there
    // are further rounds either way (4096 x 1152 x 384, 1152 tiles, 11.3 against 11.9).
    const int64_t tiles = tiles_of(shape_of(p, p.act), 64, 64);
    // Up to one tile per CU, the rate at which a CU brings in its k-tiles (16 KB each, about 37 bytes a clock) bounds the call: tiles of
    // half the rows move 3 / 4 of the bytes per workgroup and twice as many of them share the CUs' loads.  64 -> 32 rows, us:
    // 2048 x 256 x 256 (128 tiles of 64) 4.6 -> 3.8, x 1024 7.0 -> 5.8, 2048 x 384 x 1536 (192) 8.9 -> 8.4, 2500 x 384 x 1536 (240)
    // 10.0 -> 8.9, 4096 x 256 x 256 (256) 4.9 -> 4.5.  Beyond, where some CU has two tiles of 64 anyway, that holds while first loads and
    // epilogue weigh more than the loop: K = 512 and less, 6144 x 192 x 192 (288) 5.7 -> 4.9, 2500 x 512 x 512 (320) 6.8 -> 6.5,
    // 4096 x 384 x 384 (384) 6.4 -> 6.2, but 2048 x 768 x 768 (384) 8.0 -> 8.2, 5000 x 320 x 320 (395) 6.3 -> 6.4; SwiGLU, whose tiles
    // of 32 rows have half the result of the others, 2048 x 384 x 192 (384) 4.10 -> 4.14.
    if (tiles <= 256 || (tiles <= 384 && p.K <= 512 && p.act != AERIS_ACT_SWIGLU)) return launch_tile_act<32, 64, 3, true>(p, stream);
    if (tiles > 3 * 256 && tiles <= 4 * 256) return launch_tile_act<64, 64, 2, true>(p, stream);
    return launch_tile_act<64, 64, 3, true>(p, stream);
  }
  return gemm_persistent_launch(p, kind == PERSISTENT256 || kind == PERSISTENT256_192 ? 256 : 128,
                                kind == PERSISTENT128_192 || kind == PERSISTENT256_192 ? 192 : 256, stream);
}


// vector epilogue: 8 / 16-byte accesses to C and the residual (4-element alignment of every row), to bias and gate rows
bool vector_epilogue(const GemmParams& p) {
  return (p.split || (p.ldc & 3) == 0) && (p.N & 3) == 0 && (reinterpret_cast<uintptr_t>(p.gate) & 15) == 0 &&
         (p.gate_batch_stride & 3) == 0 && (reinterpret_cast<uintptr_t>(p.bias) & 7) == 0;
}

// what the persistent kernel cannot take: it addresses W through one buffer descriptor (31-bit size), forms row offsets
// with 24-bit multiplies, row numbers, gate row offsets and batch numbers in 32 bits, numbers its tiles in 24 bits and
// scales whole 64-column wave blocks of the query part
bool persistent_takes(const GemmParams& p) {
  return p.act != AERIS_ACT_SILU && (int64_t)(p.act == AERIS_ACT_SWIGLU ? 2 : 1) * p.N * p.K * 2 < (int64_t(1) << 31) &&
         p.ldc < (1 << 23) && p.split < (1 << 23) && p.gate_batch_stride < (int64_t(1) << 31) &&
         (p.rows_per_batch <= 0 || p.M / p.rows_per_batch < (int64_t(1) << 31)) && p.M + 512 < (int64_t(1) << 31) &&
         tiles_of(shape_of(p, p.act), 128, 256) < (int64_t(1) << 24) && p.q_cols % 64 == 0 && p.N >= 64;
}

// the same problem from row `first` on, `rows` of them
GemmParams rows_of(const GemmParams& p0, int64_t first, int64_t rows) {
  GemmParams p = p0;
  p.M = rows;
  p.row0 = p0.row0 + first;
  p.A += first * p.K;
  p.C = reinterpret_cast<unsigned char*>(p.C) + first * (p.split ? p.split : p.ldc) * (p.c_dtype == AERIS_F32 ? 4 : 2);
  if (p.residual)
    p.residual = reinterpret_cast<const unsigned char*>(p.residual) + first * p.ldc * (p.res_dtype == AERIS_F32 ? 4 : 2);
  return p;
}

}  // namespace

bool gemm_gelu_by_polynomial(const GemmParams& p) {
  return vector_epilogue(p) && persistent_takes(p) && p.M >= 256 && (p.N % 256 == 0 || p.N >= 1024) &&
         tiles_of(shape_of(p, AERIS_ACT_GELU), 256, 256) >= 256;
}

hipError_t gemm_launch(const void* A, const void* W, void* C, const void* bias, const float* gate,
                       const void* residual, int64_t M, int N, int K, int64_t ldc, int act, int res_dtype,
                       int c_dtype, int64_t gate_batch_stride, int64_t rows_per_batch, int split, int64_t plane_stride,
                       float q_scale, int q_cols, hipStream_t stream) {
  GemmParams p;
  p.q_scale = q_scale;
  p.q_cols = q_cols;
  p.split = split;
  p.plane_stride = plane_stride;
  p.A = reinterpret_cast<const uint16_t*>(A);
  p.W = reinterpret_cast<const uint16_t*>(W);
  p.C = C;
  p.bias = reinterpret_cast<const uint16_t*>(bias);
  p.gate = gate;
  p.residual = residual;
  p.M = M; p.N = N; p.K = K; p.ldc = ldc;
  p.row0 = 0;
  p.gate_batch_stride = gate_batch_stride;
  p.rows_per_batch = rows_per_batch > 0 ? rows_per_batch : M;
  p.tiles_n = 0;
  // GELU of bf16 results: by erf, but for the problems below that have a chip's worth of large tiles
  p.act = act == AERIS_ACT_GELU && c_dtype == AERIS_BF16 ? GEMM_ACT_GELU_ERF : act;
  p.res_dtype = residual ? res_dtype : -1;
  p.c_dtype = c_dtype;
  if (!vector_epilogue(p)) return launch_tile_act<128, 128, 2, false>(p, stream);
  Shape s = shape_of(p, p.act);
  bool persistent_ok = persistent_takes(p);
  // The polynomial where there is a chip's worth of 256 x 256 tiles, erf otherwise: one of them for all rows of a call, whatever
  // tiles they are given to (equal rows, the members of a batch say, have equal results wherever they stand)
  if (p.act == GEMM_ACT_GELU_ERF) {
    if (gemm_gelu_by_polynomial(p))
      p.act = s.act = AERIS_ACT_GELU;
    else
      persistent_ok = persistent_ok && !gate && !residual;
  }
  if (!persistent_ok)
    return tiles_of(s, 128, 128) < 128 ? launch_kind(TILE64, p, stream) : launch_tile_act<128, 128, 2, true>(p, stream);
  float one = 0.f;
  const Kind kind = best_kind(s, &one);
  // Whole rounds of 256-row tiles first, the rows of the last, partly filled round by smaller tiles in a launch of its own:
  // the rows are split, nothing else.  (14400 x 4608 x 1536: 1026 tiles, two more than four rounds of 256: 164 -> 147 us;
  // 14400 x 1536 x 6144: 342 tiles: 264 -> 239 us.)
  const int bn_out = act == AERIS_ACT_SWIGLU ? 128 : 256;
  const int64_t tiles_n = (N + bn_out - 1) / bn_out, tiles = tiles_of(s, 256, 256);
  const int64_t panels = (tiles - 1) / 256 * 256 / tiles_n;  // row panels of the rounds before the last
  if (panels > 0 && panels * 256 < M) {
    Shape head = s, rest = s;
    head.M = panels * 256;
    rest.M = M - head.M;
    float t_rest = 0.f;
    const Kind rest_kind = best_kind(rest, &t_rest);
    // Against one launch of 192-column tiles the sum of two estimates is too low, by 6 to 11 us at K = 1536 and 14 to 24 at K = 6144, while
    // the one launch, whose CUs are never all busy to the end, takes 0.87 to 0.99 of its own.  With 3 us and 0.88 the choice takes 0.2 %
    // longer than the faster of the two over 255 shapes, 7 % at most (with 0.90 of the plain sum 1.9 and 14).  f32 C and residual, N = 1536,
    // us, one launch of 192 / two: K = 1536, M = 12544 65.7 / 70.2, 13312 67.1 / 74.1, 14400 70.7 / 78.2, 14848 71.4 / 78.5; K = 6144, M =
    // 12544 233.7 / 226.1, 13312 232.8 / 233.5, 14400 244.6 / 239.4, 14848 247.7 / 239.1.  bf16, plain: 8192 x 2304 x 1024 38.4 / 39.7,
    // 14400 x 1536 x 3072 100.6 / 109.0.
    const float two = estimate_us(PERSISTENT256, head) + t_rest;
    if (kind == PERSISTENT256_192 ? two + 3.0f < 0.88f * one : two < 0.97f * one) {
      const hipError_t e = launch_kind(PERSISTENT256, rows_of(p, 0, head.M), stream);
      return e != hipSuccess ? e : launch_kind(rest_kind, rows_of(p, head.M, rest.M), stream);
    }
  }
  return launch_kind(kind, p, stream);
}

}  // namespace aeris
