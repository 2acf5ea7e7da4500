// G1 on bf6 operands for gfx950: the INT4 x INT4 projection of
// kernels/gemm_integer.loom:394-433 with both operands re-encoded, once, as
// 6-bit floats and multiplied by v_mfma_scale_f32_32x32x64_f8f6f4.
//
// Exactness. bf6 is e3m2 (sign, 3 exponent bits with bias 3, 2 mantissa
// bits); every integer -8..7 is an e3m2 value (0, 1, 2, 3 = 1.5*2, 4, 5 =
// 1.25*4, 6 = 1.5*4, 7 = 1.75*4, 8 = 2^3), so each product of two codes is
// exact and the MFMA's f32 sum of them is the exact integer dot product as
// long as it stays below 2^24 (|dot| <= 64 K: K < 2^18). With the unit block
// scale (e8m0 127) the instruction computes exactly sum a * w. The G1
// epilogue then runs on f32(dot) itself, bit-identical to the INT4 path.
//
// Why: on gfx950 this MFMA takes 64 k per 32x32 tile in about the time the
// int8 MFMA takes 32 k (measured 35 against 32 cycles), and the operands
// need no unpacking: LDS holds them in the form the MFMA reads.
//
// Formats (this library's own; produced from the reference's packed
// activation and tiled weight by clef_i4_f6_activation / clef_i4_f6_weight):
//  * bf6 row: value k at bits 6k .. 6k+5 of the row, little-endian; K * 3/4
//    bytes per row (K % 128 == 0).
//  * bf6 activation: blocks of 128 rows x 128 k (96 bytes per row, 12 KiB)
//    at ((m / 128) * (K / 128) + k / 128) * 12288, row r of a block at
//    r * 96 (f6_offset); rows past M in the last block are padding. A
//    k-step's 256 rows are then two contiguous 12 KiB blocks: each 1 KiB DMA
//    instruction reads 8 whole 128-byte lines, where 96-byte pieces of
//    3072-byte rows would touch 1.5 lines each (3.7 % faster at M4096 K4096
//    N12288).
//  * bf6 tiled weight: the same blocks over n, with the 16-byte chunk c of
//    block row r stored at chunk c ^ ((r >> 3) & 1) (the LDS swizzle,
//    applied on the global side; the activation's is applied by the DMA's
//    per-lane offsets).
//
// Kernels: gemm_ring_kernel (gemm_ring.hpp), a persistent grid of 8-wave workgroups walking
// tiles of 256 x 256, 128 x 256 or 128 x 128 outputs on their XCD, and
// gemm_f6_ksplit_kernel for the shapes with fewer tiles than CUs
// (launch_gemm_f6_impl chooses). Lane half h of a 32-row fragment reads bytes
// 48h .. 48h+47 of the row's 96 (k = 64h .. 64h+63): the first 24 are the
// operand of the k-step's first MFMA, the last 24 of its second; A and B use
// the same map, so the two MFMAs of a k-step together cover its 128 k exactly
// once.

#include "gemm_ring.hpp"

namespace clef {

namespace {

typedef int v8i __attribute__((ext_vector_type(8)));

// e3m2 values of the codes in the low nibbles of n's four bytes, one per byte:
// two 8-entry table lookups (codes 0..7 and -8..-1 by their low three bits)
// and a select by the sign nibble bit.
__device__ __forceinline__ uint32_t f6_bytes(uint32_t n) {
  constexpr auto four = [](uint32_t a) {
    uint32_t t = 0;
    for (uint32_t i = 0; i < 4; ++i) t |= e3m2_of_nibble(a + i) << (8 * i);
    return t;
  };
  constexpr uint32_t p0 = four(0), p1 = four(4), n0 = four(8), n1 = four(12);
  const uint32_t sel = n & 0x07070707u;
  const uint32_t pos = __builtin_amdgcn_perm(p1, p0, sel), neg = __builtin_amdgcn_perm(n1, n0, sel);
  const uint32_t mask = ((n >> 3) & 0x01010101u) * 0xFFu;
  return (neg & mask) | (pos & ~mask);
}

// 32 codes (four packed words, code j in nibble j % 8 of word j / 8) -> 32
// e3m2 values, value j at bits 6j of out[0..5].
__device__ __forceinline__ void f6_pack32(const uint32_t (&w)[4], uint32_t (&out)[6]) {
  uint32_t q[8];  // 24 bits each: values 4i .. 4i + 3
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t ev = f6_bytes(w[i] & 0x0F0F0F0Fu), od = f6_bytes((w[i] >> 4) & 0x0F0F0F0Fu);
    const uint32_t p02 = (ev & 0x00FF00FFu) | ((od & 0x00FF00FFu) << 6);                // pairs 0 and 2 of the word
    const uint32_t p13 = ((ev >> 8) & 0x00FF00FFu) | ((od >> 2) & 0x3FC03FC0u);         // pairs 1 and 3
    q[2 * i] = (p02 & 0xFFFFu) | ((p13 & 0xFFFFu) << 12);
    q[2 * i + 1] = (p02 >> 16) | ((p13 >> 16) << 12);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    out[3 * i] = q[4 * i] | (q[4 * i + 1] << 24);
    out[3 * i + 1] = (q[4 * i + 1] >> 8) | (q[4 * i + 2] << 16);
    out[3 * i + 2] = (q[4 * i + 2] >> 16) | (q[4 * i + 3] << 8);
  }
}

// 32 codes (four packed words) -> bytes 24 (g % 4) .. + 23 of the 96-byte row at
// `row`, chunks stored at chunk ^ s.
__device__ __forceinline__ void f6_store32(uint4 in, uint8_t* row, int g, int s) {
  const uint32_t wv[4] = {in.x, in.y, in.z, in.w};
  uint32_t o[6];
  f6_pack32(wv, o);
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    const int off = 24 * (g % 4) + 8 * p;  // logical byte offset in the row
    *reinterpret_cast<v2u*>(row + (((off >> 4) ^ s) << 4) + (off & 15)) = v2u{o[2 * p], o[2 * p + 1]};
  }
}

// Operands re-encoded as bf6, one thread per 32 codes, a wave per 8 rows x 256
// k (so it reads eight 128-byte row pieces, one contiguous KiB of a weight, and
// writes two runs of 768 bytes, 8 rows of each 128-k block). The first
// `wtotal` threads take the tiled INT4 weight (the reference layout: 128-row x
// 256-k blocks of 32 words per row) to the bf6 tiled weight, the others the
// packed activation (a_words per row) to the bf6 activation layout; either may
// be absent. Codes through byte-permute tables: weight 12288 x 4096 23.5 ->
// 13.4 us, activation 8192 x 17408 54.4 -> 43.3.
__global__ __launch_bounds__(256) void f6_convert_kernel(const uint32_t* __restrict__ w, int64_t wtotal,
                                                         uint8_t* __restrict__ w_out, const uint32_t* __restrict__ a,
                                                         int a_words, int64_t rows, int kb4, int64_t total,
                                                         uint8_t* __restrict__ a_out) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
    if (t < wtotal) {  // whole waves: wtotal is a multiple of 1024
      const int g = (int)(t & 7), r = (int)(t >> 3) & 127;
      const int64_t block = t >> 10;  // panel * kb4 + 256-k block: its two 128-k blocks are 2 block, 2 block + 1
      f6_store32(reinterpret_cast<const uint4*>(w)[t], w_out + (2 * block + (g >> 2)) * 12288 + r * 96, g,
                 (r >> 3) & 1);
    } else {
      const int64_t u = t - wtotal;
      const int g = (int)(u & 7), r8 = (int)(u >> 3) & 7;
      const int64_t unit = u >> 6, rg = unit / kb4;
      const int kt = (int)(unit - rg * kb4);
      const int64_t row = rg * 8 + r8;
      if (row >= rows) continue;
      const uint4 in = *reinterpret_cast<const uint4*>(a + row * a_words + kt * 32 + 4 * g);
      f6_store32(in, a_out + ((row >> 7) * (2 * kb4) + 2 * kt + (g >> 2)) * 12288 + (row & 127) * 96, g, 0);
    }
  }
}

// bf6 operands of the ring kernel: k-steps of 128 k, 96 bytes per row.
struct F6Op {
  typedef v16f Acc;
  typedef v8i Frag;
  static constexpr int kStep = 128;
  [[maybe_unused]] static constexpr float kDotPerStep = 64.0f * kStep;  // |dot| per k-step, codes of magnitude 8

  // One k-step's operand of fragment rows `base` (+ lane row) for MFMA `mf`:
  // 24 bytes = a 16-byte and an 8-byte read (mf 0) or an 8-byte and a 16-byte
  // read (mf 1) at the lane's swizzled chunk offsets.
  struct Reader {
    int c0, c1, c2;  // byte offsets of logical chunks 3h, 3h+1, 3h+2 in the row
    __device__ __forceinline__ explicit Reader(int = 0) {
      const int lane = threadIdx.x & 63;
      const int h = lane >> 5, s = ((lane & 31) >> 3) & 1;
      c0 = ((3 * h) ^ s) << 4;
      c1 = ((3 * h + 1) ^ s) << 4;
      c2 = ((3 * h + 2) ^ s) << 4;
    }
    __device__ __forceinline__ v8i operand(const char* row, int mf) const {
      if (mf == 0) {
        const v4u x = *reinterpret_cast<const v4u*>(row + c0);
        const v2u y = *reinterpret_cast<const v2u*>(row + c1);
        return v8i{(int)x[0], (int)x[1], (int)x[2], (int)x[3], (int)y[0], (int)y[1], 0, 0};
      }
      const v2u y = *reinterpret_cast<const v2u*>(row + c1 + 8);
      const v4u x = *reinterpret_cast<const v4u*>(row + c2);
      return v8i{(int)y[0], (int)y[1], (int)x[0], (int)x[1], (int)x[2], (int)x[3], 0, 0};
    }
  };

  __device__ __forceinline__ static v16f mfma(v8i w, v8i a, v16f c) {
    // cbsz = blgp = 3: both operands e3m2; scale 127 (e8m0) = 1.0
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w, a, c, 3, 3, 0, 127, 0, 127);
  }

  // DMA of a stage: instruction q = wave + NW * slot moves KiB q of the stage,
  // A rows first. voff[slot]: the lane's source offset. A: flat chunk
  // f = 64 q + lane of the KG x BM x 6 stage chunks is row f / 6, stored chunk
  // f % 6, which holds logical chunk (f % 6) ^ ((row >> 3) & 1), read from the
  // row's 96 bytes in block row / 128: of the tile's one or two row blocks (kb
  // k-steps of 12 KiB each) or, for KG 2, of the stage's two k-steps. B: the
  // blocks as stored. Either way the 64 lanes of an instruction read one
  // contiguous KiB; the k-step's block is in the scalar offset.
  template <class T>
  __device__ __forceinline__ static void offsets(int kb, int, int (&voff)[T::SLOTS]) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int block = T::KG == 1 ? kb * 12288 : 12288;
#pragma unroll
    for (int slot = 0; slot < T::SLOTS; ++slot) {
      const int q = wave + T::NW * slot;
      const int f = 64 * q + lane;
      const int row = f / 6, p = f % 6;
      voff[slot] = q < T::A_QS ? (row >> 7) * block + (row & 127) * T::ROW + ((p ^ ((row >> 3) & 1)) << 4) : lane * 16;
    }
  }

  // DMA instruction `slot` of this wave's share of stage kt (k-steps KG kt ..)
  // of tile `x` into `stage`. GU: the second half of a k-step's B rows comes
  // from b_rsrc2.
  template <class T, bool GU>
  __device__ __forceinline__ static void issue_slot(char* stage, const RingTiles& x, const int (&voff)[T::SLOTS],
                                                    int kb, int kt, int slot) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = wave + T::NW * slot;
    if (T::QS % T::NW != 0 && slot == T::SLOTS - 1 && q >= T::QS) return;
    const lds_ptr_t dst = (lds_ptr_t)(stage + q * 1024);
    // A / B is static except in a slot that holds both
    const bool is_a = T::NW * (slot + 1) <= T::A_QS || (T::NW * slot < T::A_QS && q < T::A_QS);
    if (is_a) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x.a_rsrc, dst, 16, voff[slot], kt * (T::KG * 12288), 0, 0);
      return;
    }
    const int qb = q - T::A_QS;
    if constexpr (GU && T::KG == 2) {
      // per k-step 6 KiB of gate rows, then 6 KiB of up rows
      const int part = qb / 6;
      __builtin_amdgcn_raw_ptr_buffer_load_lds((part & 1) == 0 ? x.b_rsrc : x.b_rsrc2, dst, 16, voff[slot],
                                               (2 * kt + (part >> 1)) * 12288 + (qb % 6) * 1024 + x.b_off, 0, 0);
    } else if constexpr (T::KG == 2) {
      // the stage's k-steps are consecutive 12 KiB blocks of the panel
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x.b_rsrc, dst, 16, voff[slot], kt * (2 * 12288) + qb * 1024, 0, 0);
    } else {
      const int panel = qb / 12, in_blk = (qb % 12) * 1024;
      if constexpr (GU)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(panel == 0 ? x.b_rsrc : x.b_rsrc2, dst, 16, voff[slot],
                                                 kt * 12288 + in_blk, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(x.b_rsrc, dst, 16, voff[slot], (panel * kb + kt) * 12288 + in_blk, 0,
                                                 0);
    }
  }

  // DMA addressing of tile b of the grid (XCD-aware order, tile_of_block).
  template <class T, bool GU>
  __device__ __forceinline__ static RingTiles tile(int b, int tiles_m, int tiles_n, const uint8_t* a, int,
                                                   const uint8_t* w, const uint8_t* w2, int64_t M, int kb) {
    constexpr int TILE_N = GU ? T::BN / 2 : T::BN;  // output columns per tile
    int tm, tn;
    tile_of_block(b, tiles_m * tiles_n, tiles_m, tiles_n, tm, tn);
    RingTiles x;
    x.m0 = (int64_t)tm * T::BM;
    x.n0 = tn * TILE_N;
    // the tile's one or two 128-row blocks of activation codes (a second
    // block past M does not exist: its loads fall outside the resource)
    const int blocks_here = T::BM > 128 && M - x.m0 > 128 ? 2 : 1;
    x.a_rsrc = make_rsrc(a + (x.m0 >> 7) * kb * 12288, (uint32_t)(blocks_here * kb * 12288));
    x.b_off = x.n0 % 128 * T::ROW;
    x.b_rsrc = make_rsrc(w + (int64_t)(x.n0 / 128) * kb * 12288, (uint32_t)((TILE_N + 127) / 128 * kb * 12288));
    x.b_rsrc2 = GU ? make_rsrc(w2 + (int64_t)(x.n0 / 128) * kb * 12288, (uint32_t)(kb * 12288)) : x.b_rsrc;
    return x;
  }
};
using F6Tile256 = RingTile<96, 128, 64, 2, 4, 1, 3>;   // 256 x 256, 48 KiB stages
using F6Tile128W = RingTile<96, 64, 64, 2, 4, 1, 4>;   // 128 x 256, 36 KiB stages
using F6Tile128 = RingTile<96, 64, 64, 2, 2, 2, 3>;    // 128 x 128, stages of two k-steps (48 KiB)

// Small-M form: the tile's k-steps shared among the eight waves of a
// workgroup, each of which loads its own (k-steps wave, wave + 8, ..) into its
// own ring of NB LDS stages and multiplies the whole tile of 32 MT rows x
// 32 NT weight rows (GU: NT / 2 fragments of gate rows, then the same up
// rows), so it only waits for its own loads and no barrier runs in the loop.
// The weight stream sets the time of these shapes: the tiles are small enough
// that the grid covers the CUs, and every stage of every wave is in flight.
// The partial accumulators (exact integers) meet in LDS, and each thread runs
// the epilogue of 8 consecutive columns of a row. 37 x 4096 x 4096 28.9 ->
// 5.4 us, 1 x 12288 x 4096 28.6 -> 9.6, 64 x 5120 x 17408 100.0 -> 16.1; GU
// 16 x 4096 x 2048 20.9 -> 6.3 (256 x 256 tiles before; same box).
template <int MT, int NT, int NB, bool RESID, bool GU>
__global__ __launch_bounds__(512) void gemm_f6_ksplit_kernel(const uint8_t* __restrict__ a,
                                                             const float* __restrict__ as,
                                                             const uint8_t* __restrict__ w,
                                                             const float* __restrict__ ws, int64_t M, int N, int kb,
                                                             const uint16_t* __restrict__ residual,
                                                             uint16_t* __restrict__ out,
                                                             const uint8_t* __restrict__ w2,
                                                             const float* __restrict__ ws2) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NW = 8, ROW = 96, FRAG = 32 * ROW;
  constexpr int BM = 32 * MT, BN = 32 * NT;     // activation and weight rows of the tile
  constexpr int COLS = GU ? BN / 2 : BN;        // output columns of the tile
  constexpr int STAGE = (MT + NT) * FRAG;
  constexpr int PART = MT * NT * 4096;          // a wave's accumulators
  constexpr int WAVE = NB * STAGE > PART ? NB * STAGE : PART;
  constexpr int CHUNKS = BM * COLS / 8;         // 8-column row chunks of the tile
  constexpr int IPT = (CHUNKS + NW * 64 - 1) / (NW * 64);
  constexpr int INST = 3 * (MT + NT);           // DMA instructions per stage
  static_assert(!GU || NT % 2 == 0, "gate and up fragments");
  static_assert(NW * WAVE <= 160 * 1024 && NB * INST < 64, "LDS per workgroup, vmcnt range");
  // Every argument into SGPRs at once (one scalar round trip).
  asm volatile("" ::"s"(a), "s"(as), "s"(w), "s"(ws), "s"(residual), "s"(out), "s"(M), "s"(N), "s"(kb), "s"(w2),
               "s"(ws2));
  extern __shared__ __align__(16) char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 31;
  const int n0 = blockIdx.x * COLS;
  const int64_t m0 = (int64_t)blockIdx.y * BM;
  const __amdgpu_buffer_rsrc_t a_rsrc = make_rsrc(a + (m0 >> 7) * kb * 12288, (uint32_t)(kb * 12288));
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(w + (int64_t)(n0 / 128) * kb * 12288, (uint32_t)(kb * 12288));
  const __amdgpu_buffer_rsrc_t w_rsrc2 =
      GU ? make_rsrc(w2 + (int64_t)(n0 / 128) * kb * 12288, (uint32_t)(kb * 12288)) : w_rsrc;
  // DMA instruction q of a fragment moves KiB q of its 32 rows' 3 KiB: flat
  // chunk f = 64 q + lane -> row f / 6, stored chunk f % 6, which holds logical
  // chunk (f % 6) ^ ((row >> 3) & 1); weight blocks are stored that way.
  int a_voff[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    const int f = 64 * q + lane, row = f / 6;
    a_voff[q] = (int)(m0 & 127) * ROW + row * ROW + (((f % 6) ^ ((row >> 3) & 1)) << 4);
  }
  const int w_voff = (n0 & 127) * ROW + lane * 16;

  char* my = lds + wave * WAVE;
  auto issue = [&](char* stage, int kt) {
#pragma unroll
    for (int f = 0; f < MT; ++f)
#pragma unroll
      for (int q = 0; q < 3; ++q)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_ptr_t)(stage + f * FRAG + q * 1024), 16, a_voff[q],
                                                 kt * 12288 + f * FRAG, 0, 0);
#pragma unroll
    for (int f = 0; f < NT; ++f) {
      const bool up = GU && f >= NT / 2;
#pragma unroll
      for (int q = 0; q < 3; ++q)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(up ? w_rsrc2 : w_rsrc,
                                                 (lds_ptr_t)(stage + (MT + f) * FRAG + q * 1024), 16, w_voff,
                                                 kt * 12288 + (up ? f - NT / 2 : f) * FRAG + q * 1024, 0, 0);
    }
  };
  const int steps = wave < kb ? (kb - 1 - wave) / NW + 1 : 0;
#pragma unroll
  for (int b = 0; b < NB; ++b)
    if (b < steps) issue(my + b * STAGE, wave + NW * b);

  const F6Op::Reader o;
  v16f acc[NT][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) acc[i][j] = v16f{};
  // The stage's operands into registers, then the DMA of k-step `next` into
  // it (if any), then the MFMAs.
  auto compute = [&](char* stage, int next) {
    v8i fa[2][MT], fw[2][NT];
#pragma unroll
    for (int mf = 0; mf < 2; ++mf) {
#pragma unroll
      for (int f = 0; f < MT; ++f) fa[mf][f] = o.operand(stage + f * FRAG + lr * ROW, mf);
#pragma unroll
      for (int f = 0; f < NT; ++f) fw[mf][f] = o.operand(stage + (MT + f) * FRAG + lr * ROW, mf);
    }
    if (next < kb) {
      // the reads above have returned before the DMA overwrites their stage
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      issue(stage, next);
    }
#pragma unroll
    for (int mf = 0; mf < 2; ++mf)
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = F6Op::mfma(fw[mf][i], fa[mf][j], acc[i][j]);
  };
  // k-step s of the wave has landed once at most the DMA of the (up to
  // NB - 1) k-steps after it is outstanding.
  int s = 0;
  for (; s + NB <= steps; s += NB) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (s + NB + b <= steps)
        wait_vmcnt<(NB - 1) * INST>();
      else
        wait_vmcnt<0>();
      compute(my + b * STAGE, wave + NW * (s + b + NB));
    }
  }
  if (s < steps) {
    wait_vmcnt<0>();
#pragma unroll
    for (int b = 0; b < NB - 1; ++b)
      if (s + b < steps) compute(my + b * STAGE, kb);
  }
  __syncthreads();  // every wave is done with its stages
  // Partial sums: block b = i * MT + j, register quad rq, lane -> 16 bytes.
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq)
        *reinterpret_cast<float4*>(my + (((i * MT + j) * 4 + rq) * 64 + lane) * 16) =
            make_float4(acc[i][j][4 * rq], acc[i][j][4 * rq + 1], acc[i][j][4 * rq + 2], acc[i][j][4 * rq + 3]);
  __syncthreads();
  // The sum of 8 columns (8 cc ..) of row rr of weight fragments base ..:
  // register quad cc % 4 of fragment cc / 4, lane halves 0 and 1.
  auto sum8 = [&](int rr, int cc, int base, float (&y)[8]) {
    const int qd = (((base + (cc >> 2)) * MT + (rr >> 5)) * 4 + (cc & 3)) * 64 + (rr & 31);
    float4 lo = *reinterpret_cast<const float4*>(lds + qd * 16);
    float4 hi = *reinterpret_cast<const float4*>(lds + (qd + 32) * 16);
#pragma unroll
    for (int q = 1; q < NW; ++q) {
      const float4 l2 = *reinterpret_cast<const float4*>(lds + q * WAVE + qd * 16);
      const float4 h2 = *reinterpret_cast<const float4*>(lds + q * WAVE + (qd + 32) * 16);
      lo.x += l2.x, lo.y += l2.y, lo.z += l2.z, lo.w += l2.w;
      hi.x += h2.x, hi.y += h2.y, hi.z += h2.z, hi.w += h2.w;
    }
    y[0] = lo.x, y[1] = lo.y, y[2] = lo.z, y[3] = lo.w;
    y[4] = hi.x, y[5] = hi.y, y[6] = hi.z, y[7] = hi.w;
  };
#pragma unroll
  for (int i = 0; i < IPT; ++i) {
    const int c = threadIdx.x + i * NW * 64;
    const int rr = c % BM, cc = c / BM;
    const int64_t m = m0 + rr;
    if (c >= CHUNKS || m >= M) continue;
    const int n = n0 + 8 * cc;
    const float av = as[m];
    float y[8], sw[8];
    uint32_t p[4];
    *reinterpret_cast<float4*>(sw) = *reinterpret_cast<const float4*>(ws + n);
    *reinterpret_cast<float4*>(sw + 4) = *reinterpret_cast<const float4*>(ws + n + 4);
    uint4 rv = make_uint4(0, 0, 0, 0);
    if constexpr (RESID) rv = *reinterpret_cast<const uint4*>(residual + m * N + n);
    sum8(rr, cc, 0, y);
    if constexpr (GU) {
      float su[8], u[8];
      *reinterpret_cast<float4*>(su) = *reinterpret_cast<const float4*>(ws2 + n);
      *reinterpret_cast<float4*>(su + 4) = *reinterpret_cast<const float4*>(ws2 + n + 4);
      sum8(rr, cc, NT / 2, u);
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        float hv[2];
#pragma unroll
        for (int b = 0; b < 2; ++b)
          hv[b] = swiglu1(bf16_to_f32(g1_f6(y[2 * t + b], sw[2 * t + b], av)),
                          bf16_to_f32(g1_f6(u[2 * t + b], su[2 * t + b], av)));
        p[t] = pack_bf16x2(hv[0], hv[1]);
      }
    } else {
#pragma unroll
      for (int t = 0; t < 4; ++t)
        p[t] = g1_f6(y[2 * t], sw[2 * t], av) | (g1_f6(y[2 * t + 1], sw[2 * t + 1], av) << 16);
    }
    if constexpr (RESID) {
      const uint32_t r4[4] = {rv.x, rv.y, rv.z, rv.w};
#pragma unroll
      for (int t = 0; t < 4; ++t) p[t] = pack_bf16x2(bf16_lo(r4[t]) + bf16_lo(p[t]), bf16_hi(r4[t]) + bf16_hi(p[t]));
    }
    *reinterpret_cast<uint4*>(out + m * N + n) = make_uint4(p[0], p[1], p[2], p[3]);
  }
#endif
}

template <int MT, int NT, int NB, bool RESID, bool GU>
hipError_t launch_f6_ksplit(const RingArgs& x, hipStream_t stream) {
  constexpr int stages = NB * (MT + NT) * 3072, part = MT * NT * 4096;
  constexpr int lds = 8 * (stages > part ? stages : part);
  constexpr int cols = GU ? 16 * NT : 32 * NT;
  static LaunchCache cache;
  const void* kern = reinterpret_cast<const void*>(&gemm_f6_ksplit_kernel<MT, NT, NB, RESID, GU>);
  if (hipError_t e = ensure_dynamic_lds(cache, kern, lds)) return e;
  const int64_t groups = (x.m + 32 * MT - 1) / (32 * MT);
  if (groups > 65535 || x.n % cols != 0) return hipErrorInvalidValue;
  const dim3 grid((unsigned)(x.n / cols), (unsigned)groups);
  gemm_f6_ksplit_kernel<MT, NT, NB, RESID, GU><<<grid, 512, lds, stream>>>(
      x.a, x.as, x.w, x.ws, x.m, x.n, x.k / 128, x.residual, x.out, x.w2, x.ws2);
  return hipGetLastError();
}

// Which kernel. Times are of one launch (graph replay, three weights in turn,
// M x N x K, us); 256 stands for the CUs.
//  * Split-K tiles while they number at most one per CU, the smallest such
//    tile (32 x 32, 32 x 64, 64 x 64 weight rows; GU 32 and 64 rows x 32
//    columns of h): 37 x 4096 x 4096 5.4 (32 x 64 6.4, 64 x 64 7.7, 128 x 128
//    tiles 13.4), 64 x 5120 x 17408 16.1 (32 x 32, two rounds, 22.3), 192 x
//    4096 x 4096 8.4 (32 x 64 11.1, 128 x 128 13.8), 400 x 4096 x 4096 14.6
//    in two rounds of 64 x 64 against 14.3 for 128 x 128. GU 64 x 4096 x 2048
//    6.5 (64 rows 7.3, 128 x 128 11.9), 64 x 12288 x 4096 20.0 in two rounds
//    against 18.4.
//  * Else the persistent tile with the least rounds x its cost. A round of
//    128 x 256 tiles takes about 0.9 of one of 256 x 256, a round of 128 x
//    128 tiles about 0.55 (620 x 5120 x 17408 44.3 against 87.0 and 81.1 for
//    one round each; 1500 x 4096 x 4096 29.0 for two rounds against 29.0 and
//    28.0 for one; GU 620 x 12288 x 4096 57.6 for two rounds of 128 x 256
//    against 67.0 for two of 256 x 256 and 63.1 for four of 128 x 128).
template <bool RESID, bool GU>
hipError_t launch_gemm_f6_impl(const RingArgs& x, hipStream_t stream) {
  auto tiles = [&](int bm, int bn) { return (x.m + bm - 1) / bm * (x.n / bn); };
  auto rounds = [&](int bm, int bn) { return (tiles(bm, bn) + 255) / 256; };
  if constexpr (GU) {
    if (tiles(32, 32) <= 256) return launch_f6_ksplit<1, 2, 2, RESID, GU>(x, stream);
    if (tiles(64, 32) <= 256) return launch_f6_ksplit<2, 2, 1, RESID, GU>(x, stream);
  } else {
    if (tiles(32, 32) <= 256) return launch_f6_ksplit<1, 1, 3, RESID, GU>(x, stream);
    if (tiles(32, 64) <= 256) return launch_f6_ksplit<1, 2, 2, RESID, GU>(x, stream);
    if (tiles(64, 64) <= 256) return launch_f6_ksplit<2, 2, 1, RESID, GU>(x, stream);
  }
  constexpr int half = GU ? 2 : 1;  // output columns per weight row of a tile
  const int64_t c256 = 100 * rounds(256, 256 / half), c128w = 90 * rounds(128, 256 / half),
                c128 = 55 * rounds(128, 128 / half);
  if (c128 <= c128w && c128 <= c256) return launch_ring<F6Op, F6Tile128, RESID, GU>(x, stream);
  if (c128w < c256) return launch_ring<F6Op, F6Tile128W, RESID, GU>(x, stream);
  return launch_ring<F6Op, F6Tile256, RESID, GU>(x, stream);
}

}  // namespace

// Packed activation rows (k % 128 == 0) -> bf6 activation, for widths that are
// not whole 256-k blocks.
__global__ __launch_bounds__(256) void f6_rows_kernel(const uint32_t* __restrict__ a, int a_words, int64_t rows,
                                                      int k, uint8_t* __restrict__ out) {
  const int groups = k / 32;
  const int64_t total = rows * groups;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = t / groups;
    const int g = (int)(t - r * groups);
    f6_store32(*reinterpret_cast<const uint4*>(a + r * a_words + 4 * g),
               out + ((r >> 7) * (k / 128) + (g >> 2)) * 12288 + (r & 127) * 96, g, 0);
  }
}

hipError_t launch_f6_convert(const uint32_t* w_tiled, int64_t n, uint8_t* w_out, const uint32_t* a, int a_words,
                             int64_t rows, uint8_t* a_out, int k, hipStream_t stream) {
  const int64_t wtotal = n * (k / 32);
  const int64_t total = wtotal + (rows + 7) / 8 * 64 * (k / 256);
  const int64_t blocks = (total + 255) / 256;
  f6_convert_kernel<<<(unsigned)(blocks < 8192 ? blocks : 8192), 256, 0, stream>>>(w_tiled, wtotal, w_out, a, a_words,
                                                                                  rows, k / 256, total, a_out);
  return hipGetLastError();
}

hipError_t launch_f6_rows(const uint32_t* a, int a_words, int64_t rows, int k, uint8_t* out, hipStream_t stream) {
  if (k % 256 == 0) return launch_f6_convert(nullptr, 0, nullptr, a, a_words, rows, out, k, stream);
  const int64_t total = rows * (k / 32);
  const int64_t blocks = (total + 255) / 256;
  f6_rows_kernel<<<(unsigned)(blocks < 8192 ? blocks : 8192), 256, 0, stream>>>(a, a_words, rows, k, out);
  return hipGetLastError();
}

hipError_t launch_f6_tiled(const uint32_t* w_tiled, int64_t n, int k, uint8_t* out, hipStream_t stream) {
  return launch_f6_convert(w_tiled, n, out, nullptr, 0, 0, nullptr, k, stream);
}

// The bf6 GEMM is a quarter faster than the INT4 one on the same tiles (twice
// the MFMA rate, no unpacking), and re-encoding both operands costs one pass
// over them. Per 1024 k a round of 256 x 256 tiles (one per CU) saves about
// 3 us, and the pass takes about 0.32 us per 1024 rows of either operand: it
// pays while the rounds exceed (m + n) / 9500, at K below 4096, where a round's
// start and stores weigh more, (m + n) / 7500. Whole calls (graph replay, three
// weights in turn, m x n x k, us, INT4 / via bf6): 1024 x 17408 x 5120 105 /
// 94, 2729: 171 / 158; 33024 x 4096 at 1280 rows 137 / 140, at 1400 172 / 169;
// 65536 x 6144 at 1536 433 / 456, at 2729 762 / 711; 98304 x 2048 at 2048 330 /
// 344, at 2729 456 / 443; 128256 x 4096 at 1536 574 / 599, at one row 46 / 256.
// One round: 1500 x 6144 x 5120 53.1 / 47.0; fewer tiles leave CUs idle either
// way (1500 x 4096 x 4096, 96 tiles, 31.2 / 38.0). Below 1024 rows the INT4
// GEMM runs smaller tiles, whose last round is fuller (769 x 17408 x 5120 71 /
// 86). Below K 2048 a call is stores and launches (2729 x 12288 x 1024 45.2 /
// 50.4).
bool gemm_i4_via_f6(int64_t m, int n, int k) {
  // clef_i4_gemm_f6's limits
  if (n % 256 != 0 || k > 32768 || n >= (1 << 22) || m > ((int64_t)1 << 29)) return false;
  const int64_t tiles = (m + 255) / 256 * (n / 256);
  if (tiles > kMaxTiles / 4) return false;  // tiles of 128 x 128 are indexed in 32 bits
  if (m < 1024 || k < 2048) return false;
  const int64_t rounds = (tiles + 255) / 256;
  if (k < 4096) return tiles > 320 && 7500 * rounds > m + n;
  return (rounds > 1 || (m >= 1500 && tiles >= 144)) && 9500 * rounds > m + n;
}

hipError_t launch_gemm_f6(const uint8_t* a, const float* as, const uint8_t* w, const float* ws, int64_t m, int n,
                          int k, const uint16_t* residual, uint16_t* out, hipStream_t stream) {
  const RingArgs x{a, 0, as, w, ws, m, n, k, residual, out, nullptr, nullptr};
  return residual ? launch_gemm_f6_impl<true, false>(x, stream) : launch_gemm_f6_impl<false, false>(x, stream);
}

hipError_t launch_gemm_f6_gate_up(const uint8_t* a, const float* as, const uint8_t* gate_w, const float* gate_s,
                                  const uint8_t* up_w, const float* up_s, int64_t m, int n, int k, uint16_t* h,
                                  hipStream_t stream) {
  return launch_gemm_f6_impl<false, true>(RingArgs{a, 0, as, gate_w, gate_s, m, n, k, nullptr, h, up_w, up_s}, stream);
}

}  // namespace clef
