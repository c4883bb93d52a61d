// Row norm (LayerNorm / RMSNorm) fused with the noise-level scale/shift modulation.  HBM-bound:
// every row of x is read once and every row of y written once, 16 bytes per lane per access, both
// marked non-temporal (streamed once: 4 % faster than with the default cache policy; either one alone is not).
//
// One wavefront owns a row and keeps it in registers (NV vectors of 8 elements per lane).  Statistics are
// fp32: mean, then the centred second moment (LayerNorm), or the plain second moment (RMSNorm).  The
// per-column parameters are folded into
//     pre :  u = x * P1 + P0          (P1 = 1 + scale, P0 = shift;  only for "modulate then norm")
//     post:  y = n(u) * G + Bc        (G = gamma, Bc = beta, or for "norm then modulate"
//                                      G = gamma*(1+scale), Bc = beta*(1+scale) + shift)
// Two kernels: rows of up to 2048 elements go to norm_modulate_block_kernel (no loop: a block of four
// waves takes sixteen rows and folds the parameters once into LDS); longer rows to norm_modulate_kernel
// (persistent waves walk down the rows with the folded parameters in registers, the next row's loads
// issued before the current row is reduced).
#include "common.h"
#include "kernels.h"

namespace aeris {

struct NormParams {
  const void* x;
  void* y;
  const void* gamma;
  const void* beta;
  int param_f32;
  const float* shift;
  const float* scale;
  int64_t mod_batch_stride;
  int64_t rows;
  int64_t rows_per_batch;
  int d;
  int kind;
  int y_dtype;
  float eps;
};

// FULL: d == NV * 512, every lane holds NV full 16-byte pieces of the row (no per-piece predicates in the loop)
template <int NV, bool X_F32, bool PRE, bool FULL>
__global__ void __launch_bounds__(256) norm_modulate_kernel(NormParams p) {
  const int lane = threadIdx.x & 63;
  const int64_t wave_id = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int64_t n_waves = (int64_t)gridDim.x * 4;
  const int d = p.d;
  const float inv_d = 1.0f / (float)d;

  bool act[NV];
  int col[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    col[v] = (v * 64 + lane) * 8;
    act[v] = FULL || col[v] < d;
  }

  float G[NV][8], Bc[NV][8], P1[PRE ? NV : 1][8], P0[PRE ? NV : 1][8];
  auto fold = [&](int64_t b) {
    const float* sh = p.shift ? p.shift + b * p.mod_batch_stride : nullptr;
    const float* sc = p.scale ? p.scale + b * p.mod_batch_stride : nullptr;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float g = 1.f, be = 0.f, s1 = 1.f, s0 = 0.f;
        if (act[v]) {
          const int c = col[v] + e;
          if (p.param_f32) {
            g = reinterpret_cast<const float*>(p.gamma)[c];
            if (p.beta) be = reinterpret_cast<const float*>(p.beta)[c];
          } else {
            g = bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p.gamma)[c]);
            if (p.beta) be = bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(p.beta)[c]);
          }
          if (sc) s1 = 1.f + sc[c];
          if (sh) s0 = sh[c];
        }
        if (PRE) {
          P1[v][e] = s1; P0[v][e] = s0; G[v][e] = g; Bc[v][e] = be;
        } else {
          G[v][e] = g * s1; Bc[v][e] = be * s1 + s0;
        }
      }
    }
  };

  struct Raw { u32x4 a, b; };
  auto load_row = [&](int64_t row, Raw (&raw)[NV]) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      raw[v].a = u32x4{0u, 0u, 0u, 0u};
      raw[v].b = u32x4{0u, 0u, 0u, 0u};
      if (act[v]) {
        if (X_F32) {
          const float* xp = reinterpret_cast<const float*>(p.x) + row * d + col[v];
          raw[v].a = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(xp));
          raw[v].b = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(xp + 4));
        } else {
          raw[v].a = __builtin_nontemporal_load(
              reinterpret_cast<const u32x4*>(reinterpret_cast<const uint16_t*>(p.x) + row * d + col[v]));
        }
      }
    }
  };

  int64_t row = wave_id;
  if (row >= p.rows) return;
  int64_t cur_b = row / p.rows_per_batch;
  fold(p.mod_batch_stride ? cur_b : 0);

  Raw cur[NV], nxt[NV];
  load_row(row, cur);
  for (; row < p.rows; row += n_waves) {
    const int64_t next = row + n_waves;
    if (next < p.rows) load_row(next, nxt);

    if (p.mod_batch_stride) {
      const int64_t b = row / p.rows_per_batch;
      if (b != cur_b) { cur_b = b; fold(b); }
    }

    float u[NV][8];
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (X_F32) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          u[v][e] = __uint_as_float(cur[v].a[e]);
          u[v][4 + e] = __uint_as_float(cur[v].b[e]);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          u[v][2 * e] = bf16_lo(cur[v].a[e]);
          u[v][2 * e + 1] = bf16_hi(cur[v].a[e]);
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (PRE) u[v][e] = act[v] ? fmaf(u[v][e], P1[v][e], P0[v][e]) : 0.f;
        s += (p.kind == AERIS_NORM_RMS) ? u[v][e] * u[v][e] : u[v][e];
      }
    }
    s = wave_sum(s);
    float mean = 0.f, rstd;
    if (p.kind == AERIS_NORM_RMS) {
      rstd = rsqrtf(s * inv_d + p.eps);
    } else {
      mean = s * inv_d;
      float q = 0.f;
#pragma unroll
      for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float c = act[v] ? u[v][e] - mean : 0.f;
          q += c * c;
        }
      q = wave_sum(q);
      rstd = rsqrtf(q * inv_d + p.eps);
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (!act[v]) continue;
      float o[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = fmaf((u[v][e] - mean) * rstd, G[v][e], Bc[v][e]);
      if (p.y_dtype == AERIS_BF16) {
        u32x4 w = {pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]), pack_bf16x2(o[4], o[5]), pack_bf16x2(o[6], o[7])};
        __builtin_nontemporal_store(w, reinterpret_cast<u32x4*>(reinterpret_cast<uint16_t*>(p.y) + row * d + col[v]));
      } else {
        float* yp = reinterpret_cast<float*>(p.y) + row * d + col[v];
        __builtin_nontemporal_store(f32x4{o[0], o[1], o[2], o[3]}, reinterpret_cast<f32x4*>(yp));
        __builtin_nontemporal_store(f32x4{o[4], o[5], o[6], o[7]}, reinterpret_cast<f32x4*>(yp + 4));
      }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) cur[v] = nxt[v];
  }
}

// Rows of up to 2048 elements: a kernel without a loop.  A block of four waves takes 4 * ROWS consecutive rows of one
// batch entry (wave w the rows w, w + 4, ...; SUB rows side by side in a wave's lanes count as so many waves), requests all of them first, folds the per-column parameters once into
// LDS while the rows are in flight (as fp32, the first and second four columns of a lane's eight in separate arrays so
// that the 16-byte reads of neighbouring lanes do not share banks), and then normalises row by row.  Short-lived waves
// with few registers (eight waves per SIMD) keep more bytes in flight and mix loads and stores more evenly than waves
// that walk down the matrix: a plain copy reaches 5.85 TB/s this way against 5.3 TB/s with the persistent structure.
template <int NV, bool X_F32, bool PRE, bool FULL, int ROWS, int SUB>
__global__ void __launch_bounds__(256) norm_modulate_block_kernel(NormParams p, int64_t blocks_per_batch) {
  static_assert(SUB == 1 || NV == 1, "several rows in a wave's lanes: rows of one column group per lane");
  constexpr int LPR = 64 / SUB;  // lanes of a row
  constexpr int GROUPS = NV * LPR;  // column groups of 8 that the LDS arrays hold
  __shared__ f32x4 sG[2][GROUPS], sB[2][GROUPS];
  __shared__ f32x4 sP1[PRE ? 2 : 1][PRE ? GROUPS : 1], sP0[PRE ? 2 : 1][PRE ? GROUPS : 1];
  typedef __attribute__((address_space(1))) const unsigned char* gc_ptr;
  typedef __attribute__((address_space(1))) unsigned char* g_ptr;
  const gc_ptr xg = (gc_ptr)p.x;
  const g_ptr yg = (g_ptr)p.y;
  const int lane = threadIdx.x & (LPR - 1), w = threadIdx.x / LPR;  // lane within the row's lanes; row slot of the block
  const int d = p.d;
  const float inv_d = 1.0f / (float)d;
  const int64_t b = (int64_t)blockIdx.x / blocks_per_batch;
  const int64_t first = b * p.rows_per_batch + ((int64_t)blockIdx.x - b * blocks_per_batch) * (4 * SUB * ROWS);
  int64_t end = (b + 1) * p.rows_per_batch;  // rows of this batch entry end here
  if (end > p.rows) end = p.rows;

  struct Raw { u32x4 a, b; };
  Raw raw[ROWS][NV];
#pragma unroll
  for (int j = 0; j < ROWS; ++j) {
    int64_t row = first + j * (4 * SUB) + w;
    if (row > end - 1) row = end - 1;  // past the end: the last row again, never stored
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int col = (v * LPR + lane) * 8;
      raw[j][v].a = u32x4{0u, 0u, 0u, 0u};
      raw[j][v].b = u32x4{0u, 0u, 0u, 0u};
      if (FULL || col < d) {
        if (X_F32) {
          const gc_ptr xp = xg + (row * d + col) * 4;
          raw[j][v].a = __builtin_nontemporal_load((const __attribute__((address_space(1))) u32x4*)xp);
          raw[j][v].b = __builtin_nontemporal_load((const __attribute__((address_space(1))) u32x4*)(xp + 16));
        } else {
          raw[j][v].a = __builtin_nontemporal_load((const __attribute__((address_space(1))) u32x4*)(xg + (row * d + col) * 2));
        }
      }
    }
  }

  // ---- fold the parameters of this batch entry: pre  u = x * P1 + P0,  post  y = n(u) * G + Bc.
  // All loads of a column group are issued before the first of them is used (vector memory returns in order: a
  // wait inside a chain of dependent loads would also wait for the rows requested above, once per link).  A
  // pointer that is absent is replaced by one that is present and its values are discarded.
  {
    const float* sh = p.shift ? p.shift + (p.mod_batch_stride ? b * p.mod_batch_stride : 0) : nullptr;
    const float* sc = p.scale ? p.scale + (p.mod_batch_stride ? b * p.mod_batch_stride : 0) : nullptr;
    const bool has_mod = sh || sc, has_beta = p.beta != nullptr;
    const float* shp = sh ? sh : sc;
    const float* scp = sc ? sc : sh;
    const void* betap = has_beta ? p.beta : p.gamma;
    for (int g = threadIdx.x; g < GROUPS; g += 256) {
      if (!(FULL || g * 8 < d)) continue;
      f32x4 gv[2], bv[2], shv[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}}, scv[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      u32x4 gq = {0u, 0u, 0u, 0u}, bq = {0u, 0u, 0u, 0u};
      if (p.param_f32) {
        gv[0] = reinterpret_cast<const f32x4*>(p.gamma)[2 * g];
        gv[1] = reinterpret_cast<const f32x4*>(p.gamma)[2 * g + 1];
        bv[0] = reinterpret_cast<const f32x4*>(betap)[2 * g];
        bv[1] = reinterpret_cast<const f32x4*>(betap)[2 * g + 1];
      } else {
        gq = reinterpret_cast<const u32x4*>(p.gamma)[g];
        bq = reinterpret_cast<const u32x4*>(betap)[g];
      }
      if (has_mod) {
        shv[0] = reinterpret_cast<const f32x4*>(shp)[2 * g];
        shv[1] = reinterpret_cast<const f32x4*>(shp)[2 * g + 1];
        scv[0] = reinterpret_cast<const f32x4*>(scp)[2 * g];
        scv[1] = reinterpret_cast<const f32x4*>(scp)[2 * g + 1];
      }
      float G[8], Bc[8], P1[8], P0[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float ga, be;
        if (p.param_f32) {
          ga = gv[e >> 2][e & 3];
          be = bv[e >> 2][e & 3];
        } else {
          ga = (e & 1) ? bf16_hi(gq[e >> 1]) : bf16_lo(gq[e >> 1]);
          be = (e & 1) ? bf16_hi(bq[e >> 1]) : bf16_lo(bq[e >> 1]);
        }
        if (!has_beta) be = 0.f;
        const float s1 = sc ? 1.f + scv[e >> 2][e & 3] : 1.f;
        const float s0 = sh ? shv[e >> 2][e & 3] : 0.f;
        if (PRE) { P1[e] = s1; P0[e] = s0; G[e] = ga; Bc[e] = be; }
        else { G[e] = ga * s1; Bc[e] = be * s1 + s0; }
      }
      sG[0][g] = f32x4{G[0], G[1], G[2], G[3]};  sG[1][g] = f32x4{G[4], G[5], G[6], G[7]};
      sB[0][g] = f32x4{Bc[0], Bc[1], Bc[2], Bc[3]};  sB[1][g] = f32x4{Bc[4], Bc[5], Bc[6], Bc[7]};
      if (PRE) {
        sP1[0][g] = f32x4{P1[0], P1[1], P1[2], P1[3]};  sP1[1][g] = f32x4{P1[4], P1[5], P1[6], P1[7]};
        sP0[0][g] = f32x4{P0[0], P0[1], P0[2], P0[3]};  sP0[1][g] = f32x4{P0[4], P0[5], P0[6], P0[7]};
      }
    }
  }
  __syncthreads();

#pragma unroll
  for (int j = 0; j < ROWS; ++j) {
    const int64_t row = first + j * (4 * SUB) + w;
    float u[NV][8];
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int g = v * LPR + lane;
      const bool act = FULL || g * 8 < d;
      if (X_F32) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          u[v][e] = __uint_as_float(raw[j][v].a[e]);
          u[v][4 + e] = __uint_as_float(raw[j][v].b[e]);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          u[v][2 * e] = bf16_lo(raw[j][v].a[e]);
          u[v][2 * e + 1] = bf16_hi(raw[j][v].a[e]);
        }
      }
      if (PRE) {
        const f32x4 p1a = sP1[0][g], p1b = sP1[1][g], p0a = sP0[0][g], p0b = sP0[1][g];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          u[v][e] = act ? fmaf(u[v][e], p1a[e], p0a[e]) : 0.f;
          u[v][4 + e] = act ? fmaf(u[v][4 + e], p1b[e], p0b[e]) : 0.f;
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) s += (p.kind == AERIS_NORM_RMS) ? u[v][e] * u[v][e] : u[v][e];
    }
    s = lanes_sum<SUB>(s);
    float mean = 0.f, rstd;
    if (p.kind == AERIS_NORM_RMS) {
      rstd = rsqrtf(s * inv_d + p.eps);
    } else {
      mean = s * inv_d;
      float qs = 0.f;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const bool act = FULL || (v * LPR + lane) * 8 < d;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float c = act ? u[v][e] - mean : 0.f;
          qs += c * c;
        }
      }
      qs = lanes_sum<SUB>(qs);
      rstd = rsqrtf(qs * inv_d + p.eps);
    }
    if (row < end) {
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const int g = v * LPR + lane;
        if (!(FULL || g * 8 < d)) continue;
        const f32x4 ga = sG[0][g], gb = sG[1][g], ba = sB[0][g], bb = sB[1][g];
        float o[8];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          o[e] = fmaf((u[v][e] - mean) * rstd, ga[e], ba[e]);
          o[4 + e] = fmaf((u[v][4 + e] - mean) * rstd, gb[e], bb[e]);
        }
        if (p.y_dtype == AERIS_BF16) {
          const u32x4 wv = {pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]), pack_bf16x2(o[4], o[5]), pack_bf16x2(o[6], o[7])};
          __builtin_nontemporal_store(wv, (__attribute__((address_space(1))) u32x4*)(yg + (row * d + g * 8) * 2));
        } else {
          const g_ptr yp = yg + (row * d + g * 8) * 4;
          __builtin_nontemporal_store(f32x4{o[0], o[1], o[2], o[3]}, (__attribute__((address_space(1))) f32x4*)yp);
          __builtin_nontemporal_store(f32x4{o[4], o[5], o[6], o[7]}, (__attribute__((address_space(1))) f32x4*)(yp + 16));
        }
      }
    }
  }
}

bool norm_supported(int d) { return d > 0 && d % 8 == 0 && d <= 12 * 512; }

template <int NV, int ROWS, int SUB>
static hipError_t launch_rows(NormParams p, bool x_f32, bool pre, hipStream_t stream) {
  constexpr int BLOCK = 4 * SUB * ROWS;  // rows of a block, all of one batch entry
  if (!p.mod_batch_stride) p.rows_per_batch = p.rows;
  const int64_t batches = (p.rows + p.rows_per_batch - 1) / p.rows_per_batch, bpb = (p.rows_per_batch + BLOCK - 1) / BLOCK;
  if (batches * bpb >= (int64_t(1) << 31)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(batches * bpb)), block(256);
#define AERIS_NORM_BLK(XF, PR)                                                                                            \
  do {                                                                                                                    \
    if (p.d == NV * 512 / SUB)                                                                                            \
      hipLaunchKernelGGL((norm_modulate_block_kernel<NV, XF, PR, true, ROWS, SUB>), grid, block, 0, stream, p, bpb);      \
    else                                                                                                                  \
      hipLaunchKernelGGL((norm_modulate_block_kernel<NV, XF, PR, false, ROWS, SUB>), grid, block, 0, stream, p, bpb);     \
  } while (0)
  if (x_f32) {
    if (pre) AERIS_NORM_BLK(true, true);
    else AERIS_NORM_BLK(true, false);
  } else {
    if (pre) AERIS_NORM_BLK(false, true);
    else AERIS_NORM_BLK(false, false);
  }
#undef AERIS_NORM_BLK
  return hipGetLastError();
}

// Four rows per wave and lane group (1, 2, 3: 2-4 % slower on 1 036 800 rows of 1536), one where that leaves a CU with no more than
// two blocks (SUB > 1: 2048 x 128 bf16 3.8 -> 2.8 us; at 728 blocks, 23296 x 192, 6.7 against 7.3) and the parameters, which every
// block of four rows then reads again, do not outweigh the waves that it adds.  Time with four over time with one row per wave, each
// the mean of both orders of the two outputs in memory (which alone move it by up to a tenth):
//   rows               3000   3400   4096   5000   6000   7000   8192
//   f32   d =  448            1.18   1.16   1.34   1.21   1.11   1.00
//              512     1.26   1.26   1.24   1.32   1.18   1.17   0.96
//              768     1.35   1.26   1.21   1.31   1.19   0.98   0.86
//             1024     1.28   1.11   1.07   1.17   1.13   1.08   1.02
//             1280     1.37   1.06   1.01   1.28   1.15   1.05   0.96
//             1536     1.07   0.93   0.91   1.31   1.14   1.07   1.00
//             2048     1.10   0.94   0.90   1.28   1.10   1.00   0.98
//   bf16  d =  448            1.18   1.15   1.18   1.12   1.09   0.93
//              768     1.34   1.25   1.26   1.37   1.27   1.10   1.02
//             1024     1.34   1.31   1.22   1.21   1.02   0.89   0.98
//             1280     1.36   1.26   1.23   1.33   1.23   0.98   0.88
//             1536     1.33   1.24   1.00   1.06   0.87   0.82   0.73
//             1792     1.40   1.26   1.23   1.31   1.04   0.83   0.81
//             2048     1.26   0.98   0.97   1.04   0.89   0.88   0.80
// (4096 rows are one round of one block of sixteen per CU: wide f32 rows just short of that keep it.)
static bool one_row_per_wave(int64_t rows, int d, bool x_f32, int sub) {
  if (sub > 1) return rows <= (int64_t)512 * 16 * sub;
  if (x_f32) {
    if (d > 1408 && rows > 3072 && rows <= 4096) return false;
    return rows <= (d < 512 || d >= 1536 ? 8192 : d == 512 || d > 896 ? 7680 : d <= 704 ? 7168 : 6656);
  }
  if (d < 1024) return rows <= (d > 416 && d < 512 ? 7168 : 8192);
  if (d % 512 == 0) return rows <= (d == 1024 ? 6144 : d == 1536 ? 5120 : 3072);  // rows that fill the lanes
  return rows <= (d <= 1280 ? 6656 : d < 1536 ? 6144 : 5632);
}
template <int NV, int SUB>
static hipError_t launch_few_or_many(const NormParams& p, bool x_f32, bool pre, hipStream_t stream) {
  return one_row_per_wave(p.rows, p.d, x_f32, SUB) ? launch_rows<NV, 1, SUB>(p, x_f32, pre, stream) : launch_rows<NV, 4, SUB>(p, x_f32, pre, stream);
}

template <int NV>
static hipError_t launch_norm(const NormParams& p, bool x_f32, bool pre, hipStream_t stream) {
  if constexpr (NV <= 4) {
    // Rows of up to 2048 elements: blocks of four waves that never straddle a batch entry.  Rows of up to 256 (128) elements lie in
    // half (a quarter) of a wave's lanes, two (four) beside each other: 500 000 x 128 f32 104.7 -> 65.9 us, 500 000 x 256 bf16
    // 109.8 -> 83.7, 23296 x 192 f32 9.3 -> 6.7.
    if constexpr (NV == 1) {
      if (p.d <= 128) return launch_few_or_many<NV, 4>(p, x_f32, pre, stream);
      if (p.d <= 256) return launch_few_or_many<NV, 2>(p, x_f32, pre, stream);
    }
    return launch_few_or_many<NV, 1>(p, x_f32, pre, stream);
  } else {
  // enough waves to cover HBM latency, few enough that parameter folding is amortised over many rows
  int64_t blocks = (p.rows + 3) / 4;
  const int64_t cap = 256 * 8;
  if (blocks > cap) blocks = cap;
  dim3 grid((unsigned)blocks), block(256);
#define AERIS_NORM_GO(XF, PR)                                                                                   \
  do {                                                                                                          \
    if (p.d == NV * 512) hipLaunchKernelGGL((norm_modulate_kernel<NV, XF, PR, true>), grid, block, 0, stream, p);  \
    else hipLaunchKernelGGL((norm_modulate_kernel<NV, XF, PR, false>), grid, block, 0, stream, p);                 \
  } while (0)
  if (x_f32) {
    if (pre) AERIS_NORM_GO(true, true);
    else AERIS_NORM_GO(true, false);
  } else {
    if (pre) AERIS_NORM_GO(false, true);
    else AERIS_NORM_GO(false, false);
  }
#undef AERIS_NORM_GO
  return hipGetLastError();
  }
}

hipError_t norm_modulate_launch(const void* x, int x_dtype, void* y, int y_dtype, const void* gamma, const void* beta,
                                int param_dtype, const float* shift, const float* scale, int64_t mod_batch_stride, int64_t B,
                                int64_t rows_per_batch, int d, int kind, int order, float eps, hipStream_t stream) {
  NormParams p;
  p.x = x; p.y = y;
  p.gamma = gamma;
  p.beta = beta;
  p.param_f32 = param_dtype == AERIS_F32;
  p.shift = shift; p.scale = scale;
  p.mod_batch_stride = (shift || scale) ? mod_batch_stride : 0;
  p.rows = B * rows_per_batch;
  p.rows_per_batch = rows_per_batch;
  p.d = d; p.kind = kind; p.y_dtype = y_dtype; p.eps = eps;
  const bool pre = (order == AERIS_MOD_THEN_NORM) && (shift || scale);
  const bool xf = x_dtype == AERIS_F32;
  const int nv = (d + 511) / 512;
  switch (nv) {
    case 1: return launch_norm<1>(p, xf, pre, stream);
    case 2: return launch_norm<2>(p, xf, pre, stream);
    case 3: return launch_norm<3>(p, xf, pre, stream);
    case 4: return launch_norm<4>(p, xf, pre, stream);
    case 5: case 6: return launch_norm<6>(p, xf, pre, stream);
    case 7: case 8: return launch_norm<8>(p, xf, pre, stream);
    default: return launch_norm<12>(p, xf, pre, stream);
  }
}

}  // namespace aeris
