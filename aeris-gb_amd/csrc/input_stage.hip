// Input embedding in one pass:  tokens = ([x0 / div0 | x1] + ape) W^T + b
// (src/aeris_wp_inference/model.py:346-356: cast to fp32, add the positional encoding, Linear(C -> d) in fp32;
// inference.py:160 for the [x / sigma_d | cond] form).  HBM-bound on its output: the C <= 159 input channels are
// read once, the d-wide token rows are written once, and no [M, K] operand matrix goes through memory in between.
//
// Arithmetic: bf16 MFMA at fp32 accuracy.  Inputs and weights are each split into a bf16 head and a bf16 remainder
// (hi = bf16(v), lo = bf16(v - hi)); hi*hi + lo*hi + hi*lo are accumulated in fp32, only lo*lo (2^-16 relative) is
// dropped.  The bias rides in a spare k column: the input operand holds 1 at k = C and the weight holds b[n] there.
//
// A workgroup of four waves owns 128 (small problems: 64) token rows; a wave builds the split operand of its 32 (16) rows
// once, keeps it in registers, and then walks over the output columns in chunks of 64.  (With 64 rows per wave the operand
// fills the register file: spills, and an eighth of the workgroups when the problem is small.)  The split weight is packed once (when the
// parameter changes) in the order the MFMA operand wants it - 16 bytes per lane, lanes consecutive, 1 KB per
// fragment - so a chunk is one contiguous piece of memory that goes to LDS by DMA (buffer_load ... lds), double
// buffered, and every fragment read is one conflict-free ds_read_b128.  With the weight fragment as first MFMA
// operand a lane ends up with 4 consecutive output columns of one row; pieces are exchanged between lanes so that every
// store instruction writes whole 128-byte lines (in 64-byte pieces the stores alone took longer than everything else).
// What bounds it now is those stores: without them the kernel takes 1.12 ms where it takes 1.83 ms with them, without
// two thirds of its MFMAs 1.55 ms.
// Measured before (64 rows per wave, operand built row by row through an LDS tile, 64-byte stores) -> now: 1 036 800 rows,
// 138 -> 1536: 2.84 -> 1.83 ms (3.8 TB/s); 259 200 rows, 144 -> 512: 382 -> 170 us (4.0 TB/s); 51 840, 138 -> 320 (bf16): 85 -> 26 us;
// 14 400, 144 -> 1536: 167 -> 42 us; 8192, 138 -> 1536: 163 -> 23 us; 2048, 138 -> 256: 52 -> 6.7 us.
#include "common.h"
#include "kernels.h"

namespace aeris {

namespace {
constexpr int IS_THREADS = 256;
constexpr int IS_NBC = 4;   // 16-column blocks per chunk
constexpr int IS_MAX_KB = 5;

struct InStageParams {
  const float* x0;
  const float* x1;
  const float* ape;
  const unsigned char* wp;  // [d / 16][NKB][hi, lo][64 lanes][8] bf16
  void* out;
  int64_t M, M_ape;
  int C0, C1, d;
  int splits;     // workgroups that share the columns of one row tile
  float div0;
};

struct PackParams {
  const float* W;     // [d, C]
  const float* bias;  // [d] or null
  unsigned char* wp;
  int d, C, NKB;
};

// one thread per 16-byte piece of the packed weight
__global__ void __launch_bounds__(256) input_pack_weight_kernel(PackParams p) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int per_nb = p.NKB * 2 * 64;
  if (t >= (int64_t)(p.d / 16) * per_nb) return;
  const int nb = (int)(t / per_nb);
  int r = (int)(t - (int64_t)nb * per_nb);
  const int kb = r / 128;
  r -= kb * 128;
  const int part = r >> 6, lane = r & 63;
  const int n = 16 * nb + (lane & 15), k0 = 32 * kb + 8 * (lane >> 4);
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int k = k0 + e;
    float w = 0.f;
    if (k < p.C) w = p.W[(int64_t)n * p.C + k];
    else if (k == p.C && p.bias) w = p.bias[n];
    const float hi = bf16_bits_to_f32(f32_to_bf16_bits(w));
    v[e] = part ? w - hi : hi;
  }
  const u32x4 o = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
  *reinterpret_cast<u32x4*>(p.wp + t * 16) = o;
}

// a: rows 0-7 of the 16 lanes' pair (x | y), b: rows 8-15; the lower 8 lanes take the x part, the upper 8 the y part
__device__ __forceinline__ void exchange8(bool upper, u32x4 x, u32x4 y, u32x4& a, u32x4& b) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t give = upper ? x[e] : y[e];
    const uint32_t got = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)give, 0x128, 0xF, 0xF, true);  // row_ror:8
    a[e] = upper ? got : x[e];
    b[e] = upper ? y[e] : got;
  }
}

// IS_RB: 16-row blocks per wave, i.e. 64 IS_RB rows per workgroup
// STREAM: non-temporal stores, for token matrices that do not fit the last-level cache
template <int NKB, int IS_RB, bool OUT_F32, bool STREAM>
__global__ void __launch_bounds__(IS_THREADS, 2) input_stage_kernel(InStageParams p) {
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  typedef __attribute__((address_space(3))) void* lds_ptr;
  constexpr int NB_BYTES = NKB * 2 * 1024;        // one 16-column block: NKB k-steps x (hi, lo) fragments of 1 KB
  constexpr int CHUNK_BYTES = IS_NBC * NB_BYTES;  // 64 columns
  constexpr int DMA_PER_WAVE = CHUNK_BYTES / 1024 / 4;
  constexpr int ESZ = OUT_F32 ? 4 : 2;

  const int tid = threadIdx.x, lane = tid & 63, l15 = lane & 15, q = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile_m = blockIdx.x / p.splits, part = blockIdx.x - tile_m * p.splits;
  const int64_t m0 = (int64_t)tile_m * (64 * IS_RB) + wave * (16 * IS_RB);
  const int d = p.d;
  // this workgroup's chunks of 64 columns: c_lo .. c_hi
  const int chunks = d / (16 * IS_NBC), c_lo = part * chunks / p.splits, c_hi = (part + 1) * chunks / p.splits;
  const int C0 = p.C0, C = p.C0 + p.C1;

  const __amdgpu_buffer_rsrc_t rs_w =
      __builtin_amdgcn_make_buffer_rsrc((void*)p.wp, 0, (int)((int64_t)(d / 16) * NB_BYTES), 0x00020000);
  auto issue_dma = [&](int c, int stage) {
    unsigned char* const dst = smem + stage * CHUNK_BYTES + wave * (DMA_PER_WAVE * 1024);
    const uint32_t src = (uint32_t)c * CHUNK_BYTES + (uint32_t)wave * (DMA_PER_WAVE * 1024);
#pragma unroll
    for (int i = 0; i < DMA_PER_WAVE; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_w, (lds_ptr)(dst + i * 1024), 16, (uint32_t)lane * 16, src + i * 1024, 0, 0);
  };
  issue_dma(c_lo, 0);

  // ---- the wave's operand: IS_RB row blocks x NKB k-steps, split into head and remainder, kept in registers.
  // A lane loads its fragment where it lies: 8 consecutive channels of one row, two 16-byte loads (4-byte aligned, rows
  // have any length) per k-step, for the input and for the positional encoding.  Only the k-steps that hold the boundary
  // between x0 and x1 or the end of the row pick their 8 channels one by one.
  bf16x8 a_hi[IS_RB][NKB], a_lo[IS_RB][NKB];
  unsigned char* orow[IS_RB];
  const int64_t last_row = p.M - 1;
  const int64_t m0c = m0 < last_row ? m0 : last_row;
  const int nvalid = (int)(p.M - m0c < 16 * IS_RB ? p.M - m0c : 16 * IS_RB);  // >= 1
  // the wave's rows wrap around the positional encoding at most once: 64 <= M_ape < 2^31 (checked by the host)
  const int ape_row0 = (int)(m0c % p.M_ape), ape_rows = (int)p.M_ape;
  const float inv_div = 1.0f / p.div0;
  typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_u;  // 16 bytes at any float
#pragma unroll
  for (int rb = 0; rb < IS_RB; ++rb) {
    // Rows below the matrix recompute its last row and store it again (same bits to the same address): every
    // wave then issues the same number of stores per chunk, which the wait at the end of a chunk counts on.
    const int roff = min(rb * 16 + l15, nvalid - 1);
    orow[rb] = reinterpret_cast<unsigned char*>(p.out) + (m0c + min(rb * 16 + (l15 & 7), nvalid - 1)) * d * ESZ;
    int arow = ape_row0 + roff;
    arow -= arow >= ape_rows ? ape_rows : 0;
    const float* const r0 = p.x0 + (m0c + roff) * C0;
    const float* const r1 = p.x1 ? p.x1 + (m0c + roff) * p.C1 - C0 : r0;  // indexed by channel
    const float* const ra = p.ape ? p.ape + (int64_t)arow * C : nullptr;
    float v[NKB][8], pe[NKB][8];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      const int k0 = 32 * kb + 8 * q;
      // wave-uniform: all 32 channels of this k-step from one array, none past the end
      const bool one_part = 32 * kb + 32 <= C && (32 * kb + 32 <= C0 || 32 * kb >= C0);
      if (one_part) {
        const float* const src = (32 * kb < C0 ? r0 : r1) + k0;
        const f32x4_u x = *reinterpret_cast<const f32x4_u*>(src), y = *reinterpret_cast<const f32x4_u*>(src + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) { v[kb][e] = x[e]; v[kb][4 + e] = y[e]; }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int k = min(k0 + e, C - 1);
          v[kb][e] = (k < C0 ? r0 : r1)[k];
        }
      }
      if (ra) {
        if (32 * kb + 32 <= C) {
          const f32x4_u x = *reinterpret_cast<const f32x4_u*>(ra + k0), y = *reinterpret_cast<const f32x4_u*>(ra + k0 + 4);
#pragma unroll
          for (int e = 0; e < 4; ++e) { pe[kb][e] = x[e]; pe[kb][4 + e] = y[e]; }
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) pe[kb][e] = ra[min(k0 + e, C - 1)];
        }
      }
    }
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb) {
      const int k0 = 32 * kb + 8 * q;
      uint32_t hi[4], lo[4];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float x = v[kb][e];
        if (p.div0 != 1.0f) {
          // x / div0 for the state channels: quotient by reciprocal with one correction step
          float quo = x * inv_div;
          quo = fmaf(fmaf(-quo, p.div0, x), inv_div, quo);
          x = k0 + e < C0 ? quo : x;
        }
        if (ra) x += pe[kb][e];
        if (32 * kb + 32 > C) x = k0 + e < C ? x : (k0 + e == C ? 1.0f : 0.0f);
        v[kb][e] = x;
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        hi[e] = pack_bf16x2(v[kb][2 * e], v[kb][2 * e + 1]);
        lo[e] = pack_bf16x2(v[kb][2 * e] - bf16_lo(hi[e]), v[kb][2 * e + 1] - bf16_hi(hi[e]));
      }
      a_hi[rb][kb] = __builtin_bit_cast(bf16x8, u32x4{hi[0], hi[1], hi[2], hi[3]});
      a_lo[rb][kb] = __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], lo[2], lo[3]});
    }
  }
  // second rows of a pair of stores (see below): 8 rows further down, where there are that many
  int64_t row_step[IS_RB];
#pragma unroll
  for (int rb = 0; rb < IS_RB; ++rb)
    row_step[rb] = (int64_t)(min(rb * 16 + 8 + (l15 & 7), nvalid - 1) - min(rb * 16 + (l15 & 7), nvalid - 1)) * d * ESZ;
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0): chunk 0 has landed
  __syncthreads();

  for (int c = c_lo; c < c_hi; ++c) {
    const int stage = (c - c_lo) & 1;
    __builtin_amdgcn_sched_barrier(0);
    if (c + 1 < c_hi) issue_dma(c + 1, stage ^ 1);
    __builtin_amdgcn_sched_barrier(0);
    u32x4 half_line[IS_RB][2];
    const unsigned char* const ws = smem + stage * CHUNK_BYTES + lane * 16;
    constexpr int NBG = IS_RB == 1 ? 4 : 2;  // column blocks at a time: four or more independent accumulator chains
    const bool upper = l15 >= 8;
#pragma unroll
    for (int nb0 = 0; nb0 < IS_NBC; nb0 += NBG) {
      f32x4 acc[NBG][IS_RB];
#pragma unroll
      for (int nb = 0; nb < NBG; ++nb)
#pragma unroll
        for (int rb = 0; rb < IS_RB; ++rb) acc[nb][rb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) {
        bf16x8 w_hi[NBG], w_lo[NBG];
#pragma unroll
        for (int nb = 0; nb < NBG; ++nb) {
          w_hi[nb] = *reinterpret_cast<const bf16x8*>(ws + (nb0 + nb) * NB_BYTES + (kb * 2 + 0) * 1024);
          w_lo[nb] = *reinterpret_cast<const bf16x8*>(ws + (nb0 + nb) * NB_BYTES + (kb * 2 + 1) * 1024);
        }
        // weight fragment first: a lane ends up with 4 consecutive output columns of one row
#pragma unroll
        for (int nb = 0; nb < NBG; ++nb)
#pragma unroll
          for (int rb = 0; rb < IS_RB; ++rb) acc[nb][rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w_hi[nb], a_hi[rb][kb], acc[nb][rb], 0, 0, 0);
#pragma unroll
        for (int nb = 0; nb < NBG; ++nb)
#pragma unroll
          for (int rb = 0; rb < IS_RB; ++rb) acc[nb][rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w_hi[nb], a_lo[rb][kb], acc[nb][rb], 0, 0, 0);
#pragma unroll
        for (int nb = 0; nb < NBG; ++nb)
#pragma unroll
          for (int rb = 0; rb < IS_RB; ++rb) acc[nb][rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w_lo[nb], a_hi[rb][kb], acc[nb][rb], 0, 0, 0);
      }
      // Stores as full 128-byte lines: a lane holds 4 columns of row l15 for each column block; the lanes of rows 0-7 give
      // their second block's piece for the first block's piece of rows 8-15 (a rotation by 8 within 16 lanes), after which
      // one store covers 8 rows x 128 B (f32: two column blocks; bf16: four, two of them joined per lane first).
#pragma unroll
      for (int rb = 0; rb < IS_RB; ++rb) {
        if (OUT_F32) {
#pragma unroll
          for (int nb = 0; nb < NBG; nb += 2) {
            u32x4 a, b;
            exchange8(upper, __builtin_bit_cast(u32x4, acc[nb][rb]), __builtin_bit_cast(u32x4, acc[nb + 1][rb]), a, b);
            unsigned char* const o = orow[rb] + ((c * IS_NBC + nb0 + nb + (upper ? 1 : 0)) * 16 + 4 * q) * 4;
            if (STREAM) {
              __builtin_nontemporal_store(a, reinterpret_cast<u32x4*>(o));
              __builtin_nontemporal_store(b, reinterpret_cast<u32x4*>(o + row_step[rb]));
            } else {
              *reinterpret_cast<u32x4*>(o) = a;
              *reinterpret_cast<u32x4*>(o + row_step[rb]) = b;
            }
          }
        } else {
#pragma unroll
          for (int nb = 0; nb < NBG; nb += 2) {
            // (v_permlane16_swap: 8 consecutive columns of the pair of blocks per lane, 16 (q & 1) + 8 (q >> 1) ..)
            const f32x4 v = acc[nb][rb], w = acc[nb + 1][rb];
            const auto x = __builtin_amdgcn_permlane16_swap(pack_bf16x2(v[0], v[1]), pack_bf16x2(w[0], w[1]), false, false);
            const auto y = __builtin_amdgcn_permlane16_swap(pack_bf16x2(v[2], v[3]), pack_bf16x2(w[2], w[3]), false, false);
            half_line[rb][(nb0 + nb) / 2] = u32x4{x[0], y[0], x[1], y[1]};
          }
        }
      }
    }
    if (!OUT_F32) {
#pragma unroll
      for (int rb = 0; rb < IS_RB; ++rb) {
        u32x4 a, b;
        exchange8(upper, half_line[rb][0], half_line[rb][1], a, b);
        unsigned char* const o = orow[rb] + (c * 64 + (upper ? 32 : 0) + 16 * (q & 1) + 8 * (q >> 1)) * 2;
        *reinterpret_cast<u32x4*>(o) = a;
        *reinterpret_cast<u32x4*>(o + row_step[rb]) = b;
      }
    }
    // The DMA loads of the next chunk were issued ahead of this chunk's stores and vector memory operations complete
    // in order: "all but the newest STORES" is exactly those loads, without waiting for any of those stores.
    constexpr int STORES = (OUT_F32 ? IS_NBC : 2) * IS_RB;
    static_assert(STORES <= 63, "vmcnt");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0F70 | (STORES & 15) | ((STORES >> 4) << 14));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  }
}

constexpr int lds_bytes(int nkb) { return 2 * IS_NBC * nkb * 2 * 1024; }

template <int NKB, int RB>
hipError_t launch_rb(InStageParams p, bool out_f32, int splits, hipStream_t stream) {
  p.splits = splits;
  const int64_t tiles = (p.M + 64 * RB - 1) / (64 * RB);
  const dim3 grid((unsigned)(tiles * splits)), block(IS_THREADS);
  // (530 MB of tokens: 198 us with the default cache policy, 170 us non-temporal; 50-90 MB: the same, and the next kernel
  // finds them in the cache)
  const bool big = RB == 2 && out_f32 && p.M * p.d * 4 > (int64_t(256) << 20);
  if (big) hipLaunchKernelGGL((input_stage_kernel<NKB, RB, true, RB == 2>), grid, block, lds_bytes(NKB), stream, p);
  else if (out_f32) hipLaunchKernelGGL((input_stage_kernel<NKB, RB, true, false>), grid, block, lds_bytes(NKB), stream, p);
  else hipLaunchKernelGGL((input_stage_kernel<NKB, RB, false, false>), grid, block, lds_bytes(NKB), stream, p);
  return hipGetLastError();
}

template <int NKB>
hipError_t launch_main(const InStageParams& p, bool out_f32, hipStream_t stream) {
  // 128 rows per workgroup where that gives most of two workgroups per CU, else 64 rows and the columns of a row tile
  // shared by up to four workgroups, each of which builds the row operand for itself.  Measured, us for (RB, splits):
  //   M = 1 036 800, d 1536:  (2, 1) 1830  (1, 1) 2000  (1, 2) 2125      51 840, d 320:  (2, 1) 25.6  (1, 1) 28.0
  //   M = 14 400, d 1536:     (2, 1) 60.8  (1, 1) 41.0  (1, 2) 37-42     8192, d 1536:  (1, 1) 36.0  (1, 2) 22.9  (1, 4) 22.7
  //   M = 2048, d 256:        (2, 1) 14.7  (1, 1) 9.6   (1, 4) 6.7  (1, 8) 6.6
  if (p.M >= 128 * 320) return launch_rb<NKB, 2>(p, out_f32, 1, stream);
  int64_t splits = 512 / ((p.M + 63) / 64);
  if (splits > 4) splits = 4;
  if (splits > p.d / 64) splits = p.d / 64;
  if (splits < 1) splits = 1;
  return launch_rb<NKB, 1>(p, out_f32, (int)splits, stream);
}

template <int NKB, int RB, bool OUT_F32, bool STREAM>
hipError_t configure_kernel() {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(&input_stage_kernel<NKB, RB, OUT_F32, STREAM>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes(NKB));
}
template <int NKB>
hipError_t configure_one() {
  hipError_t e = configure_kernel<NKB, 2, true, true>();
  if (e == hipSuccess) e = configure_kernel<NKB, 2, true, false>();
  if (e == hipSuccess) e = configure_kernel<NKB, 2, false, false>();
  if (e == hipSuccess) e = configure_kernel<NKB, 1, true, false>();
  if (e == hipSuccess) e = configure_kernel<NKB, 1, false, false>();
  return e;
}
}  // namespace

// k-steps of 32 that hold C input channels plus the bias column
static int input_stage_ksteps(int C) { return (C + 1 + 31) / 32; }

bool input_stage_supported(int C, int d) { return C >= 1 && input_stage_ksteps(C) <= IS_MAX_KB && d >= 64 && d % 64 == 0; }

int64_t input_stage_weight_bytes(int C, int d) { return (int64_t)(d / 16) * input_stage_ksteps(C) * 2 * 1024; }

hipError_t input_stage_configure() {
  hipError_t e = configure_one<1>();
  if (e == hipSuccess) e = configure_one<2>();
  if (e == hipSuccess) e = configure_one<3>();
  if (e == hipSuccess) e = configure_one<4>();
  if (e == hipSuccess) e = configure_one<5>();
  return e;
}

hipError_t input_stage_pack_weight_launch(const float* W, const float* bias, void* packed, int C, int d, hipStream_t stream) {
  PackParams p;
  p.W = W; p.bias = bias; p.wp = reinterpret_cast<unsigned char*>(packed); p.d = d; p.C = C; p.NKB = input_stage_ksteps(C);
  const int64_t pieces = (int64_t)(d / 16) * p.NKB * 2 * 64;
  hipLaunchKernelGGL(input_pack_weight_kernel, dim3((unsigned)((pieces + 255) / 256)), dim3(256), 0, stream, p);
  return hipGetLastError();
}

hipError_t input_stage_launch(const float* x0, int C0, float div0, const float* x1, int C1, const float* ape, int64_t M_ape,
                              const void* packed, void* out, int out_dtype, int64_t M, int d, hipStream_t stream) {
  InStageParams p;
  p.x0 = x0; p.x1 = x1; p.ape = ape; p.wp = reinterpret_cast<const unsigned char*>(packed); p.out = out;
  p.M = M; p.M_ape = M_ape > 0 ? M_ape : 1; p.C0 = C0; p.C1 = x1 ? C1 : 0; p.d = d; p.div0 = div0;
  const bool f32 = out_dtype == AERIS_F32;
  switch (input_stage_ksteps(p.C0 + p.C1)) {
    case 1: return launch_main<1>(p, f32, stream);
    case 2: return launch_main<2>(p, f32, stream);
    case 3: return launch_main<3>(p, f32, stream);
    case 4: return launch_main<4>(p, f32, stream);
    default: return launch_main<5>(p, f32, stream);
  }
}

}  // namespace aeris
