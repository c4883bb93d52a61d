// Windowed multi-head self-attention for gfx950, streaming variant: windows of any size up to 4096 tokens
// (the reference's 60 x 60) and head_dim 64 or 128, no relative-position bias, no shift mask (model.py:289-293).
//
// One workgroup = a block of queries of one (window, head), 32 per wave; the keys of the window are streamed through LDS in
// chunks of 64 with an online softmax.  How many waves and chunk buffers a workgroup has follows the window (the rule
// stands at the launch):
//   8 waves, 4 buffers   windows of more than 2048 tokens with head_dim 128, and few windows: one workgroup per CU, a barrier per
//                        two chunks
//   4 waves, 2 buffers   the others: two workgroups per CU (head_dim 64: three), so that one's start - token table, Q, the first
//                        chunk - and its output stores run beside another's sweep, and windows whose size is no multiple of
//                        256 leave fewer waves without queries
//   2 waves, 1 buffer    windows of up to 64 tokens: a single chunk, nothing to prefetch
// (8 waves for all windows, before -> now: 280 x 570 tokens in 10 x 38 windows with 4 heads x 64 156 -> 97 us,
// 6 x 6 windows on 360 x 720 with 6 x 64 535 -> 193 us, two members of 60 x 104 with 12 x 8 windows and 3 x 128 16.1 -> 11.8 us.)
// The global loads of the next chunks are in flight while a chunk is consumed; with a running row max m and row sum l the
// output is rescaled only when a max moves).  Window partition, window reverse and the cyclic shift are address arithmetic exactly as in the
// one-window-per-workgroup kernel (window_attention.hip); the token row of every window position is computed once
// per workgroup into an LDS table, so the streaming loop needs no integer division.
//
//   K chunk [64][HD]   global -> registers -> LDS, 16-byte chunks XOR-swizzled (conflict-free ds_read_b128)
//   V chunk [64][HD]   global -> registers (4 keys x 8 d per thread) -> 4x8 register transpose -> LDS as
//                      V^T [HD][64], key groups permuted so that a PV fragment is one ds_read_b128
//   Q                  global -> registers (MFMA B operand), once
//   S^T = K Q^T        v_mfma_f32_16x16x32_bf16; lane = one query, registers = keys
//   O^T += V^T P^T     P^T straight from the S^T accumulator registers
// What bounds it is the stream of MFMAs at the clock that the power budget leaves: with 32x32x16 MFMAs the loop without any exp2
// and row sum was 4 % faster than with them, and two query groups a wave, which halve the LDS reads, 6 % slower.  The 16x16x32 shape
// does the same FLOP per cycle and LDS bytes per FLOP at a higher clock.  32x32x16 -> 16x16x32, us: 360 x 720 tokens in 60 x 60 windows
// with 8 x 128 3800 -> 3510, 120 x 120 with 12 x 128 333 -> 319; 20 x 20 windows, 3 x 128 320 -> 301; 8 x 16 182 -> 172; head_dim 64, 60 x 60
// with 8 heads 2060 -> 1983, 6 x 6 with 6 202 -> 181 (before the wider output stores).  (PV with the two query blocks of a V^T fragment back to back: 1.3 % of that; K Q^T
// over four key blocks in turn, two or two pairs: 0.5 %; reading K fragments 3 or 4 ahead, raised wave priority: nothing.)
// The query blocks of one (window, head) are placed on the same XCD (blockIdx % 8), so its K / V rows are fetched
// into that XCD's L2 once and re-read from there by the other query blocks.
#include "common.h"
#include "kernels.h"
#include <type_traits>

namespace aeris {

namespace {

struct StreamParams {
  const uint16_t* qkv;
  uint16_t* out;
  int64_t tok_stride, head_stride, part_stride;  // q / k / v addressing, as in the one-window kernel
  int B, H, W, heads;
  int nWy, nWx, ws_y, ws_x;
  int sy, sx;
  int n_units, qblks;
  float scale;
  int q_prescaled;  // q already holds q * scale * log2(e)
  uint32_t span_bytes;  // DMA form: bytes of one image's k (or v) plane that a token offset can reach, < 2^32
};

constexpr int KC = 64;    // keys per chunk
constexpr int MAX_L = 4096;

// byte offset of 16-byte chunk `chunk` of row `row` in a tile with 128-byte rows (8 chunks), swizzled over double rows
__device__ __forceinline__ uint32_t off128(int row, int chunk) {
  return (uint32_t)((row >> 1) * 256 + (((((row & 1) << 3) | chunk) ^ ((row >> 1) & 7)) << 4));
}
// V^T tile (rows = d, 128 bytes = 64 keys each): the chunk XOR also takes bits 4-6 of the row.  With the thread -> (key
// group, d piece) map of the V staging below, both the transposing 8-byte writes (16 lanes = 8 pieces 8 rows apart x 2
// key groups in the two halves of a chunk) and the fragment reads (16 lanes = 16 consecutive rows) are free of bank
// conflicts (LDS counters: 3.9 cycles per instruction each); with off128() and consecutive threads on the pieces of
// one key group the writes were 8-way conflicts, 31 cycles per instruction, and took most of the kernel's LDS time.
// (head_dim 64, where half of the threads stage V and the writes are 4-way conflicts, is faster with the plain
// layout and thread order: measured, -8 % with this one.)
template <int HD>
__device__ __forceinline__ uint32_t vt_off(int d, int chunk) {
  return (uint32_t)((d >> 1) * 256 + ((((d & 1) << 3) | (chunk ^ ((d >> 1) & 7) ^ (HD == 128 ? (d >> 4) & 7 : 0))) << 4));
}
// the same for 256-byte rows (16 chunks)
__device__ __forceinline__ uint32_t off256(int row, int chunk) { return (uint32_t)(row * 256 + ((chunk ^ (row & 15)) << 4)); }

template <int HD, int NBUF>
struct StreamCfg {
  static constexpr int K_BYTES = KC * HD * 2;
  static constexpr int V_BYTES = HD * KC * 2;
  static constexpr int BUF = K_BYTES + V_BYTES;
  // the K chunks of all buffers first, then the V^T chunks: with head_dim 128 every K fragment of every buffer is
  // then within the 64 KB that the offset field of an LDS read reaches from one per-lane base
  static constexpr int V_BASE = NBUF * K_BYTES;
  static constexpr int TBL_OFF = NBUF * BUF;
};

}  // namespace

// DMA: K and V chunks go into LDS by the load unit itself (buffer_load ... lds: no staging registers, no ds_write, no
// transposing VALU work) and V stays row-major; the V^T fragments of P V then come from ds_read_b64_tr_b16, the LDS read that
// transposes on the way out (within 16 lanes, source lane 4e + a reads 4 consecutive elements and result lane 4a + b
// receives element b of source lanes a, 4 + a, 8 + a, 12 + a).  The 16-byte chunks of a row are XOR-swizzled.  head_dim 128,
// rows of 256 B: K by row & 15 (conflict-free ds_read_b128 fragments), V by 2 (row & 7) (the 8 keys x 2 chunks that the
// two 16-lane halves of a transposing read's 32-lane pass gather - 16 pieces of 16 bytes - land on the 16 distinct slots of a
// 256-byte bank period).  head_dim 64, rows of 128 B: K over double rows (off128()), V by 2 ((row >> 1) & 3), which with the two rows
// of a bank period are 16 slots again.  Needs every byte offset inside an image's k / v plane to fit 32
// bits (span_bytes; checked by the launcher); the register form, eight waves, takes what does not (head_dim 64, 360 x 720 tokens in
// 60 x 60 windows with 8 heads: 2160 us against 1983).
template <int HD, bool DMA, int NWAVE, int NBUF>
__global__ void __launch_bounds__(64 * NWAVE) __attribute__((amdgpu_waves_per_eu(2)))
window_attention_stream_kernel(StreamParams p) {
  static_assert(DMA ? (NWAVE == 8 && NBUF == 4) || (NWAVE == 4 && NBUF == 2) || (NWAVE == 2 && NBUF == 1) : NWAVE == 8 && NBUF == 4, "forms that exist");
  using Cfg = StreamCfg<HD, NBUF>;
  constexpr int QB = 32 * NWAVE;  // queries per workgroup
  constexpr int CH = HD / 8;   // 16-byte chunks per head row
  constexpr int QN = 2;        // blocks of 16 queries per wave
  constexpr int KS = HD / 32;  // k32 steps of QK^T
  constexpr int KB = KC / 16;  // blocks of 16 keys per chunk
  constexpr int DB = HD / 16;  // 16-row blocks of O^T
  constexpr int NT = 64 * NWAVE;
  constexpr int KIT = KC * CH / NT;                     // 16-byte K pieces per thread and chunk (1 or 2)
  constexpr int V_ITEMS = (KC / 4) * CH;                // (4 keys x 8 d) V pieces per chunk: 128 or 256
  constexpr float LOG2E = 1.4426950408889634f;

  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const uint32_t smem_addr = lds_byte_address(smem);
  int* tok = reinterpret_cast<int*>(smem + Cfg::TBL_OFF);  // token row (inside the image) of every window position
  int* const redo = tok + ((p.ws_y * p.ws_x + 3) & ~3);    // set by a wave whose sums left the range of the fast sweep

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l15 = lane & 15, q4 = lane >> 4;

  // all query blocks of one (window, head) on one XCD
  const int xcd = blockIdx.x & 7, s_idx = blockIdx.x >> 3;
  const int unit = xcd + 8 * (s_idx / p.qblks);
  const int qb = s_idx % p.qblks;
  if (unit >= p.n_units) return;
  const int head = unit % p.heads;
  const int win = unit / p.heads;
  const int wpi = p.nWy * p.nWx;
  const int b = win / wpi;
  const int wrem = win - b * wpi;
  const int wy = wrem / p.nWx, wx = wrem - wy * p.nWx;
  const int H = p.H, W = p.W;
  const int L = p.ws_y * p.ws_x;
  const int inner = p.heads * HD;
  const uint32_t ld_qkv = (uint32_t)p.tok_stride;  // token rows and their stride fit 32 bits: one 32 x 32 -> 64-bit multiply-add per address
  const int64_t img_base = (int64_t)b * H * W;
  const int y0 = wy * p.ws_y + p.sy, x0 = wx * p.ws_x + p.sx;

  for (int pos = tid; pos < L; pos += NT) {
    int Y = y0 + pos / p.ws_x;
    int X = x0 + pos % p.ws_x;
    if (Y >= H) Y -= H;
    if (X >= W) X -= W;
    tok[pos] = Y * W + X;
  }
  if (tid == 0) *redo = 0;
  __syncthreads();

  // ---- Q fragments (B operand): lane = query, 8 consecutive d per k32 step
  bool q_valid[QN];
  int64_t q_row[QN];
  bf16x8 qf[QN][KS];
#pragma unroll
  for (int n = 0; n < QN; ++n) {
    int qpos = qb * QB + wave * 32 + n * 16 + l15;
    q_valid[n] = qpos < L;
    if (!q_valid[n]) qpos = L - 1;
    q_row[n] = img_base + tok[qpos];
    const uint16_t* qp = p.qkv + head * p.head_stride + (uint64_t)(uint32_t)q_row[n] * ld_qkv + q4 * 8;
#pragma unroll
    for (int s = 0; s < KS; ++s) qf[n][s] = *reinterpret_cast<const bf16x8*>(qp + s * 32);
  }
  {
    // q is multiplied by scale * log2(e) once, here (the reference scales q in bf16 too, model.py:290): the
    // accumulators of K Q^T are then the logits in the exp2 domain and no score needs a multiply.  q_prescaled: the
    // producer of q has applied the factor in fp32 before its only rounding, and this is a multiplication by one
    const float c = p.q_prescaled ? 1.0f : p.scale * LOG2E;
#pragma unroll
    for (int n = 0; n < QN; ++n)
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const u32x4 w = __builtin_bit_cast(u32x4, qf[n][s]);
        u32x4 r;
#pragma unroll
        for (int e = 0; e < 4; ++e) r[e] = pack_bf16x2(bf16_lo(w[e]) * c, bf16_hi(w[e]) * c);
        qf[n][s] = __builtin_bit_cast(bf16x8, r);
      }
  }

  const uint16_t* kbase = p.qkv + img_base * (int64_t)ld_qkv + p.part_stride + head * p.head_stride;
  const uint16_t* vbase = p.qkv + img_base * (int64_t)ld_qkv + 2 * p.part_stride + head * p.head_stride;
  const int nch = (L + KC - 1) / KC;

  u32x4 kreg[KIT], vreg[4];
  const bool v_item = (V_ITEMS >= NT) || tid < V_ITEMS;  // waves 0-3 (head_dim 64: waves 0-1) carry a V piece
  // V piece of this thread: 4 keys (key group v_kg of the chunk) x 8 d (piece v_c).  Lane bits 0-2 (and 4 for head_dim
  // 128) select the piece - the lanes of a key group still cover whole rows of V - bit 3 the key group within a pair
  // that shares a 16-byte chunk of V^T: see vt_off().
  const int v_b3 = (tid >> 3) & 1, v_b4 = (tid >> 4) & 1, v_b5 = (tid >> 5) & 1;
  const int v_c = HD == 128 ? 8 * v_b4 + (tid & 7) : tid % CH;
  const int v_kg = HD == 128 ? 4 * (tid >> 6) + 2 * v_b3 + v_b5 : tid / CH;
  auto load_chunk = [&](int j) {
    const int key0 = j * KC;
#pragma unroll
    for (int it = 0; it < KIT; ++it) {
      const int idx = tid + it * NT, key = idx / CH, c = idx % CH;
      int kp = key0 + key;
      if (kp > L - 1) kp = L - 1;  // rows past the window: any valid row, their scores are masked
      kreg[it] = *reinterpret_cast<const u32x4*>(kbase + (uint64_t)(uint32_t)tok[kp] * ld_qkv + c * 8);
    }
    if (v_item) {
      const int kg = v_kg, c = v_c;
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        int kp = key0 + kg * 4 + jj;
        if (kp > L - 1) kp = L - 1;
        vreg[jj] = *reinterpret_cast<const u32x4*>(vbase + (uint64_t)(uint32_t)tok[kp] * ld_qkv + c * 8);
      }
    }
  };
  auto store_chunk = [&](int buf) {
    unsigned char* sK = smem + buf * Cfg::K_BYTES;
    unsigned char* sV = smem + Cfg::V_BASE + buf * Cfg::V_BYTES;
#pragma unroll
    for (int it = 0; it < KIT; ++it) {
      const int idx = tid + it * NT, key = idx / CH, c = idx % CH;
      *reinterpret_cast<u32x4*>(sK + (HD == 64 ? off128(key, c) : off256(key, c))) = kreg[it];
    }
    // V: 4 keys x 8 d register transpose -> V^T[d][key].  Inside every block of 32 keys the eight key groups are
    // stored in the order 0, 4, 1, 5, 2, 6, 3, 7: the 8 keys one lane needs for a k32 step of PV (4 q4 .. 4 q4 + 3 and
    // 16 + 4 q4 .., the accumulator layout of S^T) are then one aligned 16-byte chunk.
    if (v_item) {
      const int kg = v_kg, c = v_c;
      const int pos = (kg & ~7) | ((kg & 3) << 1) | ((kg >> 2) & 1);
#pragma unroll
      for (int w = 0; w < 4; ++w) {  // word w holds d = 8c + 2w (low half) and 8c + 2w + 1 (high half)
        u32x2 lo, hi2;
        lo.x = (vreg[0][w] & 0xffffu) | (vreg[1][w] << 16);
        lo.y = (vreg[2][w] & 0xffffu) | (vreg[3][w] << 16);
        hi2.x = (vreg[0][w] >> 16) | (vreg[1][w] & 0xffff0000u);
        hi2.y = (vreg[2][w] >> 16) | (vreg[3][w] & 0xffff0000u);
        const int d0 = c * 8 + 2 * w, d1 = d0 + 1;
        *reinterpret_cast<u32x2*>(sV + vt_off<HD>(d0, pos >> 1) + (pos & 1) * 8) = lo;
        *reinterpret_cast<u32x2*>(sV + vt_off<HD>(d1, pos >> 1) + (pos & 1) * 8) = hi2;
      }
    }
  };

  // DMA form: one instruction of a wave fills 1 KB = RPI rows of a chunk; wave w issues the pieces w, w + NWAVE, ... of K and of V.
  // Lane = (row within the piece, LDS chunk slot); it fetches the global chunk that the swizzle keeps there.
  // Keys past the window get an offset outside the descriptor and arrive as zeros (their scores are masked).
  typedef __attribute__((address_space(3))) void* lds_vptr;
  const __amdgpu_buffer_rsrc_t rs_k = __builtin_amdgcn_make_buffer_rsrc((void*)kbase, 0, (int)p.span_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_v = __builtin_amdgcn_make_buffer_rsrc((void*)vbase, 0, (int)p.span_bytes, 0x00020000);
  constexpr int RPI = 1024 / (HD * 2);  // rows per instruction: 4 (head_dim 128) or 8
  auto issue_chunk = [&](int j, int buf) {
#pragma unroll
    for (int i = 0; i < KC / (RPI * NWAVE); ++i) {
      const int ii = wave + NWAVE * i;
      auto row_offset = [&](int row) {
        const int key = j * KC + row;
        return key < L ? (uint32_t)tok[key < L ? key : 0] * (ld_qkv * 2u) : 0xFFFFF000u;
      };
      uint32_t ok, ov;
      if constexpr (HD == 128) {
        const int rsub = lane >> 4, pc = lane & 15, row = 4 * ii + rsub;
        const uint32_t rowoff = row_offset(row);
        ok = rowoff + (uint32_t)((pc ^ (row & 15)) << 4);
        ov = rowoff + (uint32_t)((pc ^ (2 * (row & 7))) << 4);
      } else {
        const int pair = 4 * ii + (lane >> 4), logical = (lane & 15) ^ (pair & 7);  // K: off128(), double rows
        const int row_v = 8 * ii + (lane >> 3);
        ok = row_offset(2 * pair + (logical >> 3)) + (uint32_t)((logical & 7) << 4);
        ov = row_offset(row_v) + (uint32_t)(((lane & 7) ^ (2 * ((row_v >> 1) & 3))) << 4);
      }
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_k, (lds_vptr)(smem + buf * Cfg::K_BYTES + ii * 1024), 16, ok, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs_v, (lds_vptr)(smem + Cfg::V_BASE + buf * Cfg::V_BYTES + ii * 1024), 16, ov, 0, 0, 0);
    }
  };
  // per-lane part of the transposing V reads: of the 16 lanes q4, lane 4e + a reads V[key0 + 4 q4 + e][16 db + 4a ..]
  uint32_t v_tr[DB];
  if (DMA) {
    const int e = (lane >> 2) & 3, a = lane & 3, row = 4 * q4 + e;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const int chunk = (2 * db + (a >> 1)) ^ (2 * (HD == 128 ? row & 7 : (row >> 1) & 3));
      v_tr[db] = smem_addr + (uint32_t)(Cfg::V_BASE + row * (HD * 2) + (chunk << 4) + (a & 1) * 8);
      asm volatile("" : "+v"(v_tr[db]));
    }
  }

  // Fragment addresses = per-lane part (below, loop-invariant) + compile-time part (buffer, key block / row block):
  //   K fragment of k32 step s, key block kb:  k_lane[s] + buf * K_BYTES + kb * 16 rows
  //   V^T fragment of step, row block db:      v_lane[head_dim 128: 4 step ^ db, else step] + V_BASE + buf * V_BYTES + db * 2048
  // (the swizzles depend on the row only through bits that the block offsets leave alone)
  // (kept as opaque 32-bit LDS addresses: left to itself the compiler splits them again into a common and a per-step
  // part and adds the two in front of every read)
  typedef __attribute__((address_space(3))) const unsigned char* lds_cptr;
  constexpr int VL = DMA ? 1 : HD == 128 ? 8 : 2;
  lds_cptr k_lane[KS], v_lane[VL];
#pragma unroll
  for (int sq = 0; sq < KS; ++sq) {
    k_lane[sq] = (lds_cptr)(smem + (HD == 64 ? off128(l15, 4 * sq + q4) : off256(l15, 4 * sq + q4)));
    asm volatile("" : "+v"(k_lane[sq]));
  }
#pragma unroll
  for (int x = 0; x < VL; ++x) {
    // vt_off(l15, chunk) with chunk = q4 ^ x (head_dim 128) or 4 x + q4; bits 4 to 6 of the row come in through x
    v_lane[x] = (lds_cptr)(smem + Cfg::V_BASE + vt_off<HD>(l15, HD == 128 ? q4 ^ x : 4 * x + q4));
    asm volatile("" : "+v"(v_lane[x]));
  }
  float m[QN], l[QN];
  f32x4 o[QN][DB];
  // A wave whose 32 queries all lie past the window (last query block of a window whose size is not a multiple of 256)
  // only stages K / V and keeps the barriers; its MFMA and softmax work would be thrown away.
  const bool wave_active = qb * QB + wave * 32 < L;  // wave-uniform

  // One pass over the window's keys.  FAST: P = exp2(logit) without a row maximum - softmax does not depend on the
  // subtracted constant, the maximum only guards the range, and the range is checked afterwards.  Otherwise the
  // online form: running maximum m, accumulated output and sum rescaled whenever a maximum moves.
  auto sweep = [&](auto fast_tag) {
  constexpr bool FAST = decltype(fast_tag)::value;
#pragma unroll
  for (int n = 0; n < QN; ++n) {
    m[n] = -INFINITY;
    l[n] = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db) o[n][db] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  if (DMA) {
    issue_chunk(0, 0);
    if (NBUF > 1 && nch > 1) issue_chunk(1, 1);
    // vmcnt(0) lgkmcnt(0): this wave's loads into LDS have landed.  (With two buffers chunk 1 need not have: a wait for chunk 0 alone,
    // counted, and a barrier without the compiler's fence, which waits for everything.  Units of 128 and 256 tokens, head_dim 128:
    // 3200 x 128 99 -> 89 us, 1600 x 256 74 -> 54 - 60; but 416 x 256, one round of workgroups, 16.9 -> 17.9.  Not taken here.)
    __builtin_amdgcn_s_waitcnt(0x0070);
  } else {
    load_chunk(0);
    store_chunk(0);
    if (NBUF == 4 && nch > 1) {
      load_chunk(1);
      store_chunk(1);
    }
  }
  __syncthreads();

  // the chunk loop is unrolled over the buffers, so that the buffer a chunk sits in is a compile-time constant
  for (int j0 = 0; j0 < nch; j0 += NBUF) {
#pragma unroll
  for (int u = 0; u < NBUF; ++u) {
    const int j = j0 + u;
    if (j >= nch) break;
    constexpr int LEAD = NBUF / 2;  // chunk j + LEAD is loaded and written to LDS while chunk j is consumed
    if (DMA) {
      // Two buffers: the next chunk is requested at the start of this one and awaited at the barrier that ends this one.  Four: both
      // chunks of the next pair at the start of this pair, awaited at the barrier that ends it.  (The buffers were last read before
      // the barrier ahead of the request.)
      if (NBUF == 2) {
        if (j > 0 && j + 1 < nch) issue_chunk(j + 1, (u + 1) & 1);  // (chunk 1 was requested with chunk 0)
      } else if (NBUF == 4 && (u & 1) == 0) {
        if (j + LEAD < nch) issue_chunk(j + LEAD, (u + LEAD) & (NBUF - 1));
        if (j + LEAD + 1 < nch) issue_chunk(j + LEAD + 1, (u + LEAD + 1) & (NBUF - 1));
      }
    } else if (j + LEAD < nch) {
      load_chunk(j + LEAD);
    }
    f32x4 acc[QN][KB];
    if (wave_active) {

    // ---- S^T = K Q^T for the 64 keys of the chunk: acc[n][kb][i] = <k[key], q>, key = 64j + 16kb + 4 q4 + i, query 16n + l15
    // The K fragments are read PF fragments ahead of their use (left to itself the compiler reads each one right before
    // its MFMAs and exposes the LDS latency every time).
    {
      constexpr int PF = 2, NS = KB * KS;
      const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
      bf16x8 kfr[PF + 1];
      // fragment t: the key blocks in turn, so that an accumulator is not needed again at once
      auto step_of = [](int t) { return t / KB; };
      auto block_of = [](int t) { return t % KB; };
      auto read_k = [&](int t) {  // rows 16 kb + l15, 16-byte chunk 4 s + q4
        typedef __attribute__((address_space(3))) const bf16x8* frag_ptr;
        return *(frag_ptr)(k_lane[step_of(t)] + u * Cfg::K_BYTES + block_of(t) * 16 * (HD * 2));
      };
#pragma unroll
      for (int t = 0; t < PF; ++t) kfr[t] = read_k(t);
#pragma unroll
      for (int t = 0; t < NS; ++t) {
        if (t + PF < NS) kfr[(t + PF) % (PF + 1)] = read_k(t + PF);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < QN; ++n)
          acc[n][block_of(t)] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kfr[t % (PF + 1)], qf[n][step_of(t)], step_of(t) == 0 ? zero4 : acc[n][block_of(t)], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (j * KC + KC > L) {  // last, partial chunk (uniform): keys past the window do not take part
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int key = j * KC + kb * 16 + q4 * 4 + i;
          if (key >= L) {
#pragma unroll
            for (int n = 0; n < QN; ++n) acc[n][kb][i] = -INFINITY;
          }
        }
    }

    // PV step p (32 keys): k slots 0-3 <-> keys 32p + 4 q4 + (0..3); slots 4-7 <-> keys 32p + 16 + 4 q4 + (0..3): one V^T
    // chunk per 16-row block of O^T.  The fragments of half of the row blocks are read ahead of the MFMAs of the half before.
    // DMA form: the transposing reads are inline assembly (the builtin form would make the compiler wait for the load
    // unit's pending loads of the next chunks in front of every one of them, see lds_read_tr16_b64); what they return
    // becomes usable in v_ready().
    constexpr int DH = DB / 2, PARTS = KC / 32 * 2;  // row blocks of a half; halves of a chunk
    bf16x8 vfb[2][DH];
    TrFrag vtr[2][DMA ? DH : 1];
    auto load_v = [&](int part, int slot) {
      const int step = part >> 1;
#pragma unroll
      for (int d = 0; d < DH; ++d) {
        const int db = (part & 1) * DH + d;
        if (DMA) {  // keys 32 step + 4 q4 + (0..3) and 32 step + 16 + 4 q4 + (0..3) of row-major V, transposed by the read
          const uint32_t a0 = v_tr[db] + u * Cfg::V_BYTES + step * 32 * (HD * 2);
          vtr[slot][DMA ? d : 0].lo = lds_read_tr16_b64<0>(a0);
          vtr[slot][DMA ? d : 0].hi = lds_read_tr16_b64<16 * (HD * 2)>(a0);
        } else {
          vfb[slot][d] = *(__attribute__((address_space(3))) const bf16x8*)(v_lane[HD == 128 ? ((4 * step) ^ db) % VL : step % VL] + u * Cfg::V_BYTES + db * 2048);
        }
      }
    };
    auto v_ready = [&](int slot) {
      if (DMA) {
        if constexpr (DH == 4) lds_tr_wait(vtr[slot][0], vtr[slot][DMA ? 1 : 0], vtr[slot][DMA ? 2 : 0], vtr[slot][DMA ? 3 : 0]);
        else lds_tr_wait(vtr[slot][0], vtr[slot][DMA ? 1 : 0]);
#pragma unroll
        for (int d = 0; d < DH; ++d) vfb[slot][d] = tr_frag_value(vtr[slot][DMA ? d : 0]);
      }
    };
    load_v(0, 0);  // in flight during the softmax arithmetic below

    // ---- online softmax (exp2 domain): new row max, rescale what has been accumulated if any max moved
    if (!FAST) {
#pragma unroll
      for (int n = 0; n < QN; ++n) {
        float cm = acc[n][0][0];
#pragma unroll
        for (int kb = 0; kb < KB; ++kb)
#pragma unroll
          for (int i = 0; i < 4; i += 2) cm = fmaxf(fmaxf(cm, acc[n][kb][i]), acc[n][kb][i + 1]);
        cm = fmaxf(cm, __shfl_xor(cm, 16, 64));
        cm = fmaxf(cm, __shfl_xor(cm, 32, 64));
        const float m_new = fmaxf(m[n], cm);
        if (__builtin_amdgcn_ballot_w64(m_new > m[n]) != 0) {
          const float alpha = __builtin_amdgcn_exp2f(m[n] - m_new);  // 0 for the first chunk (m = -inf)
          l[n] *= alpha;
#pragma unroll
          for (int db = 0; db < DB; ++db) o[n][db] *= alpha;
          m[n] = m_new;
        }
      }
    }

    // ---- P = exp2(s) or exp2(s - m) for 32 keys at a time and O^T += V^T P^T: while the MFMAs of a step run, the P of the next
    // step is formed (the VALU work hides the MFMAs) and the V^T fragments of the next half are read
    uint32_t pkb[2][QN][4];
    auto exp_step = [&](int step, int n) {
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const float a0 = acc[n][2 * step + (h >> 1)][2 * (h & 1)], a1 = acc[n][2 * step + (h >> 1)][2 * (h & 1) + 1];
        const float e0 = __builtin_amdgcn_exp2f(FAST ? a0 : a0 - m[n]);
        const float e1 = __builtin_amdgcn_exp2f(FAST ? a1 : a1 - m[n]);
        pkb[step & 1][n][h] = pack_bf16x2(e0, e1);
        l[n] = dot2_ones(pkb[step & 1][n][h], l[n]);  // the row sum of what PV multiplies: the rounded values, one instruction per pair
      }
    };
#pragma unroll
    for (int n = 0; n < QN; ++n) exp_step(0, n);
#pragma unroll
    for (int part = 0; part < PARTS; ++part) {
      const int step = part >> 1;
      __builtin_amdgcn_sched_barrier(0);
      v_ready(part & 1);  // ahead of the next half's reads: the wait then covers reads issued a whole half ago only
      if (part + 1 < PARTS) load_v(part + 1, (part + 1) & 1);
      if (step + 1 < KC / 32) exp_step(step + 1, part & 1);
#pragma unroll
      for (int d = 0; d < DH; ++d) {
#pragma unroll
        for (int n = 0; n < QN; ++n) {
          const u32x4 pw = {pkb[step & 1][n][0], pkb[step & 1][n][1], pkb[step & 1][n][2], pkb[step & 1][n][3]};
          const bf16x8 pf = __builtin_bit_cast(bf16x8, pw);
          f32x4& od = o[n][(part & 1) * DH + d];
          od = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vfb[part & 1][d], pf, od, 0, 0, 0);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    }  // wave_active

    if (!DMA && j + LEAD < nch) store_chunk((u + LEAD) & (NBUF - 1));
    if (NBUF == 2 || (NBUF == 4 && (u & 1))) {
      if (DMA) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the next chunk or pair of chunks, requested at the start of this one
      __syncthreads();
    }
  }
  }
  };  // sweep

  sweep(std::true_type{});
  // Range check of the sweep without maximum: a row sum that left [2^-40, 2^100] (or is not a number) means logits
  // beyond what exp2 holds without the maximum; the workgroup then repeats the window's keys in the online form.
  {
    bool bad = false;
#pragma unroll
    for (int n = 0; n < QN; ++n) {
      float lt = l[n] + __shfl_xor(l[n], 16, 64);
      lt += __shfl_xor(lt, 32, 64);
      bad = bad || (wave_active && !(lt >= 0x1p-40f && lt <= 0x1p100f));
    }
    if (__builtin_amdgcn_ballot_w64(bad) != 0 && lane == 0) *redo = 1;
    __syncthreads();
    if (*redo != 0) sweep(std::false_type{});
  }

  // ---- normalise and store: o[n][db][i] = O[query 16n + l15][16db + 4 q4 + i]
#pragma unroll
  for (int n = 0; n < QN; ++n) {
    l[n] += __shfl_xor(l[n], 16, 64);
    l[n] += __shfl_xor(l[n], 32, 64);
    const float inv = __builtin_amdgcn_rcpf(l[n]);
    uint16_t* op = p.out + q_row[n] * inner + head * HD + 16 * (q4 & 1) + 8 * (q4 >> 1);
    // 8 consecutive elements a lane: v_permlane16_swap on the pieces of two row blocks.  The address unit takes one lane's piece a cycle
    // here (neighbouring lanes are different rows), 8 or 16 bytes alike: 4 elements a lane -> 8, us: 360 x 720 tokens, 3 heads x 128 in 8 x 8
    // windows 156 -> 145, 20 x 20 300 -> 283; 6 x 64, 8 x 16 164 -> 152; two of 60 x 104 in 12 x 8 windows, 3 x 128 11.5 -> 10.8.
#pragma unroll
    for (int m2 = 0; m2 < DB / 2; ++m2) {
      const f32x4 a = o[n][2 * m2] * inv, c = o[n][2 * m2 + 1] * inv;
      const auto rx = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[0], a[1]), pack_bf16x2(c[0], c[1]), false, false);
      const auto ry = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[2], a[3]), pack_bf16x2(c[2], c[3]), false, false);
      if (q_valid[n]) *reinterpret_cast<u32x4*>(op + m2 * 32) = u32x4{rx[0], ry[0], rx[1], ry[1]};
    }
  }
}

// ---------------------------------------------------------------------------------------------

static int stream_smem(int head_dim, int L, int nbuf) { return nbuf * (KC * head_dim * 2 + head_dim * KC * 2) + ((L * 4 + 15) / 16) * 16 + 16; }

bool attention_stream_supported(int ws_y, int ws_x, int head_dim, bool has_bias, bool use_mask) {
  const int64_t L = (int64_t)ws_y * ws_x;
  return (head_dim == 64 || head_dim == 128) && L >= 1 && L <= MAX_L && !has_bias && !use_mask;
}

namespace {
template <int HD, bool DMA, int NWAVE, int NBUF>
hipError_t configure_one() {
  return hipFuncSetAttribute(reinterpret_cast<const void*>(window_attention_stream_kernel<HD, DMA, NWAVE, NBUF>),
                             hipFuncAttributeMaxDynamicSharedMemorySize, stream_smem(HD, MAX_L, NBUF));
}
template <int HD, bool DMA, int NWAVE, int NBUF>
hipError_t launch_one(StreamParams p, int L, hipStream_t stream) {
  p.qblks = (L + 32 * NWAVE - 1) / (32 * NWAVE);
  const int64_t grid = (int64_t)((p.n_units + 7) / 8) * 8 * p.qblks;
  hipLaunchKernelGGL((window_attention_stream_kernel<HD, DMA, NWAVE, NBUF>), dim3((unsigned)grid), dim3(64 * NWAVE),
                     stream_smem(HD, L, NBUF), stream, p);
  return hipGetLastError();
}
}  // namespace

hipError_t attention_stream_configure_all() {
  hipError_t e = configure_one<64, false, 8, 4>();
  if (e == hipSuccess) e = configure_one<128, false, 8, 4>();
  if (e == hipSuccess) e = configure_one<64, true, 8, 4>();
  if (e == hipSuccess) e = configure_one<64, true, 2, 1>();
  if (e == hipSuccess) e = configure_one<128, true, 2, 1>();
  if (e == hipSuccess) e = configure_one<64, true, 4, 2>();
  if (e == hipSuccess) e = configure_one<128, true, 8, 4>();
  if (e == hipSuccess) e = configure_one<128, true, 4, 2>();
  return e;
}

hipError_t attention_stream_launch(const void* qkv, void* out, int B, int H, int W, int heads, int head_dim, int ws_y,
                                   int ws_x, int shift_y, int shift_x, float scale, int q_prescaled, int64_t tok_stride,
                                   int64_t head_stride, int64_t part_stride, hipStream_t stream) {
  StreamParams p;
  p.q_prescaled = q_prescaled;
  p.tok_stride = tok_stride; p.head_stride = head_stride; p.part_stride = part_stride;
  p.qkv = reinterpret_cast<const uint16_t*>(qkv);
  p.out = reinterpret_cast<uint16_t*>(out);
  p.B = B; p.H = H; p.W = W; p.heads = heads;
  p.nWy = H / ws_y; p.nWx = W / ws_x; p.ws_y = ws_y; p.ws_x = ws_x;
  p.sy = shift_y; p.sx = shift_x;
  p.scale = scale;
  const int L = ws_y * ws_x;
  p.n_units = B * p.nWy * p.nWx * heads;
  // bytes of an image's k (or v) plane that a token offset can reach; the DMA form addresses them with 32 bits
  const int64_t span = ((int64_t)H * W - 1) * tok_stride * 2 + (int64_t)head_dim * 2;
  p.span_bytes = span < ((int64_t)1 << 32) - 4096 ? (uint32_t)span : 0u;
  const bool dma = p.span_bytes != 0 && tok_stride > 0;
  // Windows above 2048 tokens with head_dim 128: 8 waves (4 windows of 3600 with 12 heads: 320 us against 325; 360 x 720 with 8 heads
  // 3530, 3615).  Below, 4 waves (250 000 tokens x 3 heads, 8 -> 4 waves: L = 1364 581 -> 550 us, 960 471 -> 460, 400 343 -> 304, 192 226 -> 206,
  // 128 222 -> 174), head_dim 64 for any L (250 000 x 6: L = 1364 693 -> 600), except where 8 waves are one workgroup per CU and 4 waves would
  // be up to two: the chip is as full either way, and the two load every K / V chunk twice (`lone`, per XCD of 32 CUs; 8 -> 4 waves):
  //   head_dim 128, units of 130 tokens  144: 11.8 -> 12.8 us   240: 12.6 -> 13.9   (the second workgroup has two queries)   192 tokens  144: 13.4 -> 13.3
  //     400 tokens  72: 21.6 -> 21.6   120: 23.6 -> 23.7      900 tokens  48: 36.9 -> 38.5      1395  32: 48.1 -> 49.9      2048  24: 66.9 -> 69.2
  //   head_dim 64   130 tokens  144: 7.9 -> 8.5   192 tokens  144: 8.6 -> 8.5   400 tokens  72: 13.8 -> 13.9   120: 14.8 -> 15.0
  //     900 tokens  40: 23.2 -> 23.8   64: 24.8 -> 25.8   1395  24: 30.7 -> 31.4   2048  24: 43.0 -> 44.7   3600  16: 71.5 -> 75.6
  const int64_t per_xcd = (p.n_units + 7) / 8, wgs4 = per_xcd * ((L + 127) / 128), wgs8 = per_xcd * ((L + 255) / 256);
  const bool lone = wgs8 <= 32 && wgs4 > 32;
  if (head_dim == 64) {
    if (!dma) return launch_one<64, false, 8, 4>(p, L, stream);
    if (lone && (L <= 160 || L > 256)) return launch_one<64, true, 8, 4>(p, L, stream);
    return L <= KC ? launch_one<64, true, 2, 1>(p, L, stream) : launch_one<64, true, 4, 2>(p, L, stream);
  }
  if (!dma) return launch_one<128, false, 8, 4>(p, L, stream);
  if (L > 2048 || (lone && (L <= 160 || L > 512 || (L > 384 && wgs4 <= 48)))) return launch_one<128, true, 8, 4>(p, L, stream);
  return L <= KC ? launch_one<128, true, 2, 1>(p, L, stream) : launch_one<128, true, 4, 2>(p, L, stream);
}

}  // namespace aeris
