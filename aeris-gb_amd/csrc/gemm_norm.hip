// Row norm, modulation and the projection behind them in one kernel for gfx950, for rows of 64 or 128 elements:
//   C[M,N] = act(y W^T + bias),  y = bf16(norm and modulation of x)   (the norm ahead of to_qkv and of the MLP's first Linear)
//
// What bounds such a call is latency while it is small (the norm of 2048 rows of 128 is a launch of 2.8 us for 0.2 us of traffic,
// and what it writes comes back from memory into the next launch) and memory when it is large (y written and read again: a third
// of the bytes of to_qkv).  Here a workgroup normalises the 64 rows of x that it multiplies, keeps them in LDS for the whole
// kernel (64 x K bf16: 16 KB at K = 128) and walks over its share of the columns in tiles of 64, W streaming through a ring of
// k-tiles whose loads run ahead across the tiles and were started before the rows were read.  The columns are shared out so that
// there are about two workgroups per CU: each share repeats the norm of its rows (0.5 us of VALU work at K = 128), which is also
// why wider rows stay with two kernels (norm_gemm_takes).  Same arithmetic in the same order as norm_modulate_block_kernel and
// gemm_bf16_nt_tile_kernel: the same bits.
#include "common.h"
#include "gemm_common.h"
#include "kernels.h"

namespace aeris {

namespace {
constexpr int BM = 64, BN = 64, BK = 64, NT = 256;
constexpr int STAGES = 4, STAGE = BN * BK * 2;  // 8 KB per k-tile of W
constexpr int FM = 2, FN = 2;                   // 16 x 16 fragments of a wave (2 x 2 waves)
constexpr int LPT = 2;                          // load instructions of a wave per k-tile (8 rows each)
constexpr int SUB = 4;                          // rows of x side by side in a wave
constexpr int MAX_K = 512 / SUB;

struct NormGemmParams {
  GemmParams g;  // of it M, N, K, W, C, bias, ldc, split, plane_stride, q_scale, q_cols, tiles_n
  const void* x;
  const void* gamma;
  const void* beta;
  const float* shift;
  const float* scale;
  int64_t mod_batch_stride, rows_per_batch;  // a tile's rows are all of one batch entry where the stride is not 0
  int x_f32, param_f32, kind;
  float eps;
  int col_tiles;  // column tiles of a workgroup
  int shares;     // workgroups per row tile
};

template <int N>
__device__ __forceinline__ void wait_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}
// ... with the loads of min(MOST, behind) k-tiles left outstanding
template <int MOST>
__device__ __forceinline__ void wait_k_tile(int behind) {
  if constexpr (MOST > 0) {
    if (behind < MOST) {
      wait_k_tile<MOST - 1>(behind);
      return;
    }
  }
  wait_barrier<MOST * LPT>();
}

}  // namespace

template <int ACT, bool PRE>
__global__ void __launch_bounds__(NT, 2) norm_gemm_kernel(NormGemmParams p) {
  constexpr bool SWIGLU = ACT == AERIS_ACT_SWIGLU;
  constexpr int BN_OUT = SWIGLU ? BN / 2 : BN, NJ = SWIGLU ? FN / 2 : FN;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const GemmParams& g = p.g;
  const int K = g.K, N = g.N, KT = K / BK;
  unsigned char* const sW = smem + (size_t)KT * STAGE;  // behind the rows of y: k-tiles of 64 rows x 64, as the W tiles are
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // ---- workgroups of one row tile are neighbours on one XCD (blockIdx % 8): they read the same rows of x
  int pid = blockIdx.x;
  {
    const int np = gridDim.x, per = (np + 7) >> 3;
    int tall = np & 7;
    if (tall == 0) tall = 8;
    const int xcd = pid & 7, loc = pid >> 3;
    pid = xcd < tall ? xcd * per + loc : tall * per + (xcd - tall) * (per - 1) + loc;
  }
  const int tile_m = pid / p.shares, share = pid - tile_m * p.shares;
  const int64_t m0 = (int64_t)tile_m * BM;
  const int tn0 = share * p.col_tiles;
  const int n_tiles = (g.tiles_n - tn0 < p.col_tiles ? g.tiles_n - tn0 : p.col_tiles);
  const int total = n_tiles * KT;  // k-tiles of W, in order

  // ---- W: a wave brings in 16 rows of a k-tile
  uint32_t ld_voff[2];
  {
    const int dr = lane >> 4, pos = lane & 15;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int logical = pos ^ (i * 4 + dr);
      ld_voff[i] = (uint32_t)((i * 8 + dr * 2 + (logical >> 3)) * K * 2 + (logical & 7) * 16);
    }
  }
  const lds_dma_rsrc rs_w = make_lds_dma_rsrc(g.W, (uint32_t)((SWIGLU ? 2 : 1) * (int64_t)N * K * 2));
  const uint32_t lds_w = lds_byte_address(sW) + (uint32_t)wave * 2048;
  int ld_tile = 0, ld_kt = 0, ld_stage = 0;
  auto issue = [&]() {
    const int n0 = (tn0 + ld_tile) * BN_OUT;
    // SwiGLU: a wave column's 32 tile rows are the gate rows, then the up rows, of 16 output columns
    const uint32_t row = SWIGLU ? (uint32_t)((wave & 1) * N + n0 + (wave >> 1) * 16) : (uint32_t)(n0 + wave * 16);
    const uint32_t off = row * (uint32_t)(K * 2) + (uint32_t)ld_kt * (BK * 2);
#pragma unroll
    for (int i = 0; i < 2; ++i) lds_dma_load16(rs_w, lds_w + ld_stage * STAGE + i * 1024, ld_voff[i], off);
    if (++ld_stage == STAGES) ld_stage = 0;
    if (++ld_kt == KT) {
      ld_kt = 0;
      ++ld_tile;
    }
  };
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < total) issue();

  // ---- norm and modulation: 16 rows a wave, SUB side by side in its lanes; a lane has the same 8 columns of all of them
  {
    constexpr int LPR = 64 / SUB, IT = 16 / SUB;
    const int c = lane & (LPR - 1), sub = lane / LPR;
    const bool act = c * 8 < K;
    const int col = act ? c * 8 : 0;
    u32x4 xa[IT], xb[IT];
    int64_t row_last = g.M - 1;
#pragma unroll
    for (int j = 0; j < IT; ++j) {
      int64_t row = m0 + wave * 16 + j * SUB + sub;
      if (row > row_last) row = row_last;  // past the end: the last row again, never stored
      if (p.x_f32) {
        const u32x4* xp = reinterpret_cast<const u32x4*>(reinterpret_cast<const float*>(p.x) + row * K + col);
        xa[j] = xp[0];
        xb[j] = xp[1];
      } else {
        const u32x4 h = *reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(p.x) + row * K + col);
        xa[j] = h;
        xb[j] = u32x4{0u, 0u, 0u, 0u};
      }
    }
    // parameters of the lane's columns, folded: pre  u = x * P1 + P0,  post  y = n(u) * G + Bc
    float G[8], Bc[8], P1[PRE ? 8 : 1], P0[PRE ? 8 : 1];
    {
      const int64_t mo = p.mod_batch_stride ? m0 / p.rows_per_batch * p.mod_batch_stride : 0;
      const float *sh = p.shift ? p.shift + mo : nullptr, *sc = p.scale ? p.scale + mo : nullptr;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        f32x4 ga, be = {0.f, 0.f, 0.f, 0.f}, s1 = {1.f, 1.f, 1.f, 1.f}, s0 = {0.f, 0.f, 0.f, 0.f};
        if (p.param_f32) {
          ga = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(p.gamma) + col + 4 * h);
          if (p.beta) be = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(p.beta) + col + 4 * h);
        } else {
          const u32x2 w = *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint16_t*>(p.gamma) + col + 4 * h);
          ga = f32x4{bf16_lo(w.x), bf16_hi(w.x), bf16_lo(w.y), bf16_hi(w.y)};
          if (p.beta) {
            const u32x2 v = *reinterpret_cast<const u32x2*>(reinterpret_cast<const uint16_t*>(p.beta) + col + 4 * h);
            be = f32x4{bf16_lo(v.x), bf16_hi(v.x), bf16_lo(v.y), bf16_hi(v.y)};
          }
        }
        if (sc) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(sc + col + 4 * h);
#pragma unroll
          for (int e = 0; e < 4; ++e) s1[e] = 1.f + v[e];
        }
        if (sh) s0 = *reinterpret_cast<const f32x4*>(sh + col + 4 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int k = 4 * h + e;
          if (PRE) { P1[k] = s1[e]; P0[k] = s0[e]; G[k] = ga[e]; Bc[k] = be[e]; }
          else { G[k] = ga[e] * s1[e]; Bc[k] = be[e] * s1[e] + s0[e]; }
        }
      }
    }
    const float inv_d = 1.0f / (float)K;
    unsigned char* const y_lane = smem + (c >> 3) * STAGE;
#pragma unroll
    for (int j = 0; j < IT; ++j) {
      float u[8];
      if (p.x_f32) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          u[e] = __uint_as_float(xa[j][e]);
          u[4 + e] = __uint_as_float(xb[j][e]);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          u[2 * e] = bf16_lo(xa[j][e]);
          u[2 * e + 1] = bf16_hi(xa[j][e]);
        }
      }
      float s = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (PRE) u[e] = fmaf(u[e], P1[e], P0[e]);
        if (!act) u[e] = 0.f;
        s += p.kind == AERIS_NORM_RMS ? u[e] * u[e] : u[e];
      }
      s = lanes_sum<SUB>(s);
      float mean = 0.f, rstd;
      if (p.kind == AERIS_NORM_RMS) {
        rstd = rsqrtf(s * inv_d + p.eps);
      } else {
        mean = s * inv_d;
        float qs = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float d = act ? u[e] - mean : 0.f;
          qs += d * d;
        }
        qs = lanes_sum<SUB>(qs);
        rstd = rsqrtf(qs * inv_d + p.eps);
      }
      float o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = fmaf((u[e] - mean) * rstd, G[e], Bc[e]);
      if (act)
        *reinterpret_cast<u32x4*>(y_lane + swz_off(wave * 16 + j * SUB + sub, c & 7)) =
            u32x4{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]), pack_bf16x2(o[4], o[5]), pack_bf16x2(o[6], o[7])};
    }
  }

  // ---- main loop over the column tiles
  const int wm = wave >> 1, wn = wave & 1;
  const int l15 = lane & 15, q = lane >> 4;
  const int m_w = wm * (BM / 2);
  uint32_t a_roff[2], b_roff[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    a_roff[ks] = swz_off(m_w + l15, ks * 4 + q);
    b_roff[ks] = swz_off(wn * (BN / 2) + l15, ks * 4 + q);
  }
  const int rows = (int)(g.M - m0 < BM ? g.M - m0 : BM);
  const int64_t rs = c_row_stride(g);
  const __amdgpu_buffer_rsrc_t rs_bias =
      __builtin_amdgcn_make_buffer_rsrc((void*)g.bias, 0, g.bias ? (SWIGLU ? 4 : 2) * N : 0, 0x00020000);  // without a bias everything reads 0
  typedef uint32_t __attribute__((__vector_size__(2 * sizeof(uint32_t)))) raw2;
  int done = 0, rd = 0;
  for (int t = 0; t < n_tiles; ++t) {
    const int n_w = (tn0 + t) * BN_OUT + wn * (BN_OUT / 2);  // first output column of this wave
    f32x4 acc[FM][FN];
    {
      raw2 bq[FN];
#pragma unroll
      for (int j = 0; j < FN; ++j)
        bq[j] = __builtin_bit_cast(raw2, __builtin_amdgcn_raw_buffer_load_b64(
                    rs_bias, ((SWIGLU && j >= NJ ? N : 0) + n_w + (SWIGLU ? j % NJ : j) * 16 + q * 4) * 2, 0, 0));
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const f32x4 b = {bf16_lo(bq[j][0]), bf16_hi(bq[j][0]), bf16_lo(bq[j][1]), bf16_hi(bq[j][1])};
#pragma unroll
        for (int i = 0; i < FM; ++i) acc[i][j] = b;
      }
    }
    for (int kt = 0; kt < KT; ++kt, ++done) {
      // (the first wait also ends the writing of y)
      wait_k_tile<STAGES - 2>(total - 1 - done);
      const unsigned char *sa = smem + kt * STAGE, *sb = sW + rd * STAGE;
      bf16x8 af[2][FM], bf[2][FN];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int i = 0; i < FM; ++i) af[ks][i] = *reinterpret_cast<const bf16x8*>(sa + a_roff[ks] + i * 16 * 128);
#pragma unroll
        for (int j = 0; j < FN; ++j) bf[ks][j] = *reinterpret_cast<const bf16x8*>(sb + b_roff[ks] + j * 16 * 128);
      }
      if (done + STAGES - 1 < total) issue();  // behind the fragment reads, as in gemm_bf16_nt_tile_kernel
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[ks][j], af[ks][i], acc[i][j], 0, 0, 0);
      if (++rd == STAGES) rd = 0;
    }
    // ---- epilogue: a lane holds 4 consecutive n of one row
    if (ACT == AERIS_ACT_NONE && g.q_cols > n_w) {  // query part of a qkv projection: scaled in fp32 ahead of its only rounding
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float s = n_w + j * 16 + q * 4 + e < g.q_cols ? g.q_scale : 1.0f;
#pragma unroll
          for (int i = 0; i < FM; ++i) acc[i][j][e] *= s;
        }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int r = m_w + i * 16 + l15;
      const bool row_ok = r < rows;
      float v[NJ][4];
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float x = acc[i][j][e];
          if (SWIGLU) x = silu_f(x) * acc[i][j + NJ][e];
          else if (ACT == GEMM_ACT_GELU_ERF) x = gelu_erf_bf16_f(x);
          else if (ACT == AERIS_ACT_GELU) x = gelu_bf16_f(x);
          v[j][e] = x;
        }
      uint16_t* const c_row = reinterpret_cast<uint16_t*>(g.C) + (m0 + r) * rs;
      if (NJ == 1) {
        const int n = n_w + q * 4;
        if (row_ok) *reinterpret_cast<u32x2*>(c_row + c_col_off(g, n)) = u32x2{pack_bf16x2(v[0][0], v[0][1]), pack_bf16x2(v[0][2], v[0][3])};
      } else {
        // lane (l15, q) of the swapped pair of column fragments holds the columns 16 (q & 1) + 8 (q >> 1) ..
        const auto x = __builtin_amdgcn_permlane16_swap(pack_bf16x2(v[0][0], v[0][1]), pack_bf16x2(v[NJ - 1][0], v[NJ - 1][1]), false, false);
        const auto y = __builtin_amdgcn_permlane16_swap(pack_bf16x2(v[0][2], v[0][3]), pack_bf16x2(v[NJ - 1][2], v[NJ - 1][3]), false, false);
        const int n = n_w + 16 * (q & 1) + 8 * (q >> 1);
        if (row_ok) *reinterpret_cast<u32x4*>(c_row + c_col_off(g, n)) = u32x4{x[0], y[0], x[1], y[1]};
      }
    }
  }
}

namespace {
template <int ACT, bool PRE>
void launch_one(const NormGemmParams& p, dim3 grid, hipStream_t stream) {
  hipLaunchKernelGGL((norm_gemm_kernel<ACT, PRE>), grid, dim3(NT), p.g.K / BK * STAGE + STAGES * STAGE, stream, p);
}
template <int ACT>
void launch_pre(const NormGemmParams& p, bool pre, dim3 grid, hipStream_t stream) {
  if (pre) launch_one<ACT, true>(p, grid, stream);
  else launch_one<ACT, false>(p, grid, stream);
}
}  // namespace

// Rows of 64 and 128 elements.  Two kernels -> this one, us (f32 rows, layer norm; calls replayed from a HIP graph):
//        rows      128 -> 384     128 -> 512 GELU    64 -> 192     192 -> 576     256 -> 768     256 -> 1024 GELU
//         256     6.2 ->  4.7     6.4 ->  5.2      5.9 ->  4.5     6.9 ->  7.5    7.1 ->  7.7     7.4 ->  8.2
//        2048     6.6 ->  5.1     7.1 ->  5.8      6.2 ->  4.7     8.0 ->  9.0    8.6 ->  9.7     9.3 -> 10.5
//        8192     8.6 ->  8.1    11.2 ->  9.2      7.2 ->  5.8    13.0 -> 13.2   14.5 -> 14.8    20.2 -> 19.1
//       32768    20.0 -> 16.9    27.2 -> 22.8     13.4 ->  9.4    31.8 -> 26.7
//      131072    61.2 -> 47.0    74.3 -> 63.1     31.1 -> 24.0
// From 192 on the norm that every share of the columns repeats costs more than the launch and the traffic that go, until there are
// many rows (not built for those).
// The rest is whole column tiles (N is 3 * heads * head_dim or the hidden width, both multiples of 64 wherever the projection behind
// them is taken), what the vector epilogue and one descriptor over W need, and one modulation row per row tile.
//
// A ceiling on the rows (rows_taken).  Once x and C are larger than the last-level cache (256 MB) the plain product with its tiles of
// 256 waits for memory less than tiles of 64 do, more than the norm's pass costs, except where
//   - x is f32 and not much smaller than C (N <= 4 K): the norm's pass is much of the traffic
//   - the plain product's column tiles are partly empty: GELU with N % 256 != 0 and N < 1024 (and by erf), SwiGLU of 64 columns
// SwiGLU reads two rows of W per output column; from 320 columns of 128 or 512 of 64 on its products lose sooner.  Time of the two
// kernels over this one's, mean of both orders of the two results in memory:
//            rows      8192  12288  16384  24576  32768  45056  65536  92160 131072 196608 259200 345600 524288 1036800
//   none  K=128 N=384 f32   1.08   1.18   1.29   1.35   1.21   1.37   1.08   1.16   1.21   1.15   1.01   1.03   1.04   1.02
//                    bf16   1.05   1.13   1.21   1.32   1.24   1.42   1.11   1.06   1.16   1.07   1.08   0.91   0.89   0.85
//         K=64  N=192 bf16  1.19   1.14   1.19   1.34   1.42   1.46   1.35   1.38   1.39   1.15   1.21   1.23   1.15   0.83
//         K=64  N=768 f32   1.13   1.07   1.05   1.17   1.04   1.22   1.13   1.06   1.10   0.84   0.85   0.87   0.83   0.82
//   GELU  K=128 N=512 f32   1.26   1.03   1.22   1.37   1.15   1.29   1.07   1.13   1.13   0.96   1.01   1.01   1.01   0.99
//                    bf16   1.21   1.00   1.21   1.35   1.20   1.26   1.16   1.06   1.09   1.03   0.93   0.94   0.88   0.88
//         K=64  N=320 bf16  1.01   1.07   1.14   1.18   1.27   1.32   1.43   1.40   1.49   1.50   1.50   1.43   1.32   1.33
//   SwiGLU K=64 N=64  bf16  1.27   1.29   1.35   1.32   1.71   1.54   1.79   1.57   1.80   1.61   1.56   1.53   1.59   1.49
//         K=64  N=256 f32   1.26   1.12   1.14   1.16   1.12   1.17   1.17   1.08   1.10   1.10   1.12   1.09   0.88   0.89
//         K=128 N=256 bf16  1.23   1.03   1.11   1.28   1.18   1.23   1.00   0.91   0.98   0.93   0.91   0.87   0.77   0.78
//         K=128 N=384 f32   1.11   1.18   1.11   1.29   1.12   1.13   0.87   1.04   0.97   0.94   0.83   0.86   0.86   0.84
//         K=128 N=512 f32   1.00   0.93   0.99   1.13   0.93   0.93   0.82   0.94   0.93   0.82   0.88   0.89   0.92   0.88
//         K=64  N=1024 f32  0.93   0.85   0.87   0.85   0.80   0.86   0.93   0.92   0.84   0.90   0.86   0.84   0.87   0.85
// (A block of dim 128, hidden 512, bf16, on 720 x 1440: SwiGLU 1885 -> 1703 us with two kernels again.)
static bool rows_taken(int64_t M, int N, int K, bool x_f32, int act) {
  const int64_t nk = (int64_t)N * K;
  const bool cached = M * (K * (x_f32 ? 4 : 2) + N * (int64_t)2) <= 280000000;
  if (act == AERIS_ACT_SWIGLU) {
    if (N <= 64) return true;
    if (N >= 1024) return M <= 4096;
    if (N > 512 || nk > 49152) return M <= 10240;
    if (nk > 40960) return M <= 49152;
    return cached && (x_f32 || K < 128 || N < 256 || M <= 65536);
  }
  if (act == AERIS_ACT_GELU && N % 256 && N < 1024) return true;
  return cached || (x_f32 && N <= 4 * K);
}

bool norm_gemm_takes(int64_t M, int N, int K, bool x_f32, int act, const void* bias, bool modulated, int64_t mod_batch_stride, int64_t B,
                     int64_t rows_per_batch) {
  return K % BK == 0 && K <= MAX_K && N % BN == 0 && (reinterpret_cast<uintptr_t>(bias) & 7) == 0 && M < (int64_t(1) << 31) &&
         (int64_t)(act == AERIS_ACT_SWIGLU ? 2 : 1) * N * K * 2 < (int64_t(1) << 31) && rows_taken(M, N, K, x_f32, act) &&
         (!modulated || mod_batch_stride == 0 || B == 1 || rows_per_batch % BM == 0) &&
         (M + BM - 1) / BM * (N / 32) < (int64_t(1) << 31);
}

hipError_t norm_gemm_launch(const void* x, int x_dtype, const void* gamma, const void* beta, int param_dtype, const float* shift,
                            const float* scale, int64_t mod_batch_stride, int64_t rows_per_batch, int kind, int order, float eps,
                            const void* W, void* C, const void* bias, int64_t M, int N, int K, int64_t ldc, int act, int split,
                            int64_t plane_stride, float q_scale, int q_cols, hipStream_t stream) {
  NormGemmParams p = {};
  GemmParams& g = p.g;
  g.W = reinterpret_cast<const uint16_t*>(W);
  g.C = C;
  g.bias = reinterpret_cast<const uint16_t*>(bias);
  g.M = M; g.N = N; g.K = K; g.ldc = ldc;
  g.rows_per_batch = M;
  g.act = act; g.res_dtype = -1; g.c_dtype = AERIS_BF16;
  g.split = split; g.plane_stride = plane_stride;
  g.q_scale = q_scale; g.q_cols = q_cols;
  p.x = x; p.x_f32 = x_dtype == AERIS_F32;
  p.gamma = gamma; p.beta = beta; p.param_f32 = param_dtype == AERIS_F32;
  p.shift = shift; p.scale = scale;
  p.mod_batch_stride = (shift || scale) && M > rows_per_batch ? mod_batch_stride : 0;
  p.rows_per_batch = rows_per_batch;
  p.kind = kind; p.eps = eps;
  const int bn_out = act == AERIS_ACT_SWIGLU ? BN / 2 : BN;
  const int64_t tiles_m = (M + BM - 1) / BM;
  g.tiles_n = N / bn_out;
  // two workgroups per CU (three fit): one hides the other's norm (8192 x 128 -> 512: 11.5 us with one, 9.55 with two, 12.8 with
  // four, 2048 rows 6.4 with any)
  const int64_t want = (512 + tiles_m - 1) / tiles_m;
  p.col_tiles = (int)((g.tiles_n + want - 1) / want);
  p.shares = (g.tiles_n + p.col_tiles - 1) / p.col_tiles;
  const dim3 grid((unsigned)(tiles_m * p.shares));
  const bool pre = order == AERIS_MOD_THEN_NORM && (shift || scale);
  if (act == AERIS_ACT_SWIGLU) launch_pre<AERIS_ACT_SWIGLU>(p, pre, grid, stream);
  else if (act == AERIS_ACT_GELU && gemm_gelu_by_polynomial(g)) launch_pre<AERIS_ACT_GELU>(p, pre, grid, stream);
  else if (act == AERIS_ACT_GELU) launch_pre<GEMM_ACT_GELU_ERF>(p, pre, grid, stream);
  else launch_pre<AERIS_ACT_NONE>(p, pre, grid, stream);
  return hipGetLastError();
}

}  // namespace aeris
