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
// Kernels: gemm_f6_kernel, a persistent grid of 8-wave workgroups walking
// tiles of 256 x 256, 128 x 256 or 128 x 128 outputs on their XCD, and
// gemm_f6_ksplit_kernel for the shapes with fewer tiles than CUs
// (launch_gemm_f6_impl chooses). Lane half h of a 32-row fragment reads bytes
// 48h .. 48h+47 of the row's 96 (k = 64h .. 64h+63): the first 24 are the
// operand of the k-step's first MFMA, the last 24 of its second; A and B use
// the same map, so the two MFMAs of a k-step together cover its 128 k exactly
// once.

#include <type_traits>

#include "common.hpp"
#include "gemm_dma.hpp"
#include "kernels.hpp"
#include "launch.hpp"
#include "silu_table.hpp"

namespace clef {

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef unsigned f6_v2u __attribute__((ext_vector_type(2)));
typedef unsigned f6_v4u __attribute__((ext_vector_type(4)));

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

// Packed activation (k_stride words per row) -> the bf6 activation layout
// (f6_offset); one thread per 32 codes.
__global__ __launch_bounds__(256) void f6_rows_kernel(const uint32_t* __restrict__ a, int a_words, int64_t rows,
                                                      int k, uint8_t* __restrict__ out) {
  const int groups = k / 32;
  const int64_t total = rows * groups;
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = t / groups;
    const int g = (int)(t - r * groups);
    const uint4 in = *reinterpret_cast<const uint4*>(a + r * a_words + 4 * g);
    const uint32_t w[4] = {in.x, in.y, in.z, in.w};
    uint32_t o[6];
    f6_pack32(w, o);
    f6_v2u* dst = reinterpret_cast<f6_v2u*>(out + f6_offset(r, 32 * g, k));
    dst[0] = f6_v2u{o[0], o[1]};
    dst[1] = f6_v2u{o[2], o[3]};
    dst[2] = f6_v2u{o[4], o[5]};
  }
}

// Tiled INT4 weight (the reference layout: 128-row x 256-k blocks of 32 words
// per row) -> bf6 tiled weight (header comment); one thread per 32 codes, in
// the order of the INT4 weight, so that a wave reads one KiB and writes two
// runs of 768 bytes (8 rows of each 128-k block). Codes through byte-permute
// tables: 12288 x 4096 23.5 -> 13.9 us.
__global__ __launch_bounds__(256) void f6_tiled_kernel(const uint32_t* __restrict__ w, int64_t total,
                                                       uint8_t* __restrict__ out) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total; t += (int64_t)gridDim.x * blockDim.x) {
    const uint4 in = reinterpret_cast<const uint4*>(w)[t];
    const int g = (int)(t & 7), r = (int)(t >> 3) & 127;
    const int64_t block = t >> 10;  // panel * kb4 + 256-k block: its two 128-k blocks are 2 block, 2 block + 1
    const uint32_t wv[4] = {in.x, in.y, in.z, in.w};
    uint32_t o[6];
    f6_pack32(wv, o);
    uint8_t* blk = out + (2 * block + (g >> 2)) * 12288 + r * 96;
    const int s = (r >> 3) & 1;
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const int off = 24 * (g % 4) + 8 * p;  // logical byte offset in the 96-byte row
      *reinterpret_cast<f6_v2u*>(blk + ((((off >> 4) ^ s)) << 4) + (off & 15)) = f6_v2u{o[2 * p], o[2 * p + 1]};
    }
  }
}

// Tile shape of the bf6 GEMM: KG groups of WAVES_M x WAVES_N waves, each wave
// WM rows x WN weight rows; a stage holds KG k-steps and group g contracts
// the g-th of them.
template <int WM_, int WN_, int WAVES_M_, int WAVES_N_, int KG_, int NST_>
struct F6TileShape {
  static constexpr int WM = WM_, WN = WN_, WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, KG = KG_;
  static constexpr int NST = NST_;                              // LDS stages
  static constexpr int GROUP = WAVES_M * WAVES_N;               // waves per k-group
  static constexpr int NW = GROUP * KG, THREADS = 64 * NW;
  static constexpr int BM = WM * WAVES_M, BN = WN * WAVES_N;
  static constexpr int TM = WM / 32, TN = WN / 32;              // fragments per wave
  static constexpr int EM = TM / KG;                            // row fragments a wave takes through the epilogue
  static constexpr int ROW = 96;                                // bytes per row per k-step (128 k)
  static constexpr int A_STEP = BM * ROW, B_STEP = BN * ROW;    // bytes of one k-step
  static constexpr int A_BYTES = KG * A_STEP, B_BYTES = KG * B_STEP;
  static constexpr int STAGE_BYTES = A_BYTES + B_BYTES;
  static constexpr int A_QS = A_BYTES / 1024, QS = STAGE_BYTES / 1024;  // DMA instructions per stage
  static constexpr int SLOTS = (QS + NW - 1) / NW;              // and per wave, at most
  static constexpr int EPI_WAVE = 32 * WN * 2;                  // staging bytes per wave (32 rows of WN bf16)
  static constexpr int SCALE_WAVE = 1024;                       // per-wave epilogue scales (768 bytes used)
  static constexpr int LDS = NST * STAGE_BYTES + NW * SCALE_WAVE;  // 152 KiB
  // fused gate/up: the SiLU window after the scales (exactly 160 KiB)
  static constexpr int LUT_OFF = LDS;
  static constexpr int LDS_GU = LUT_OFF + kSiluWinBytes;
  static_assert(NW == 8 && LDS == 152 * 1024, "workgroup shape");
  static_assert(NW * EPI_WAVE <= STAGE_BYTES, "the epilogue stages its output in one free stage");
};
using F6Tile256 = F6TileShape<128, 64, 2, 4, 1, 3>;   // 256 x 256, 48 KiB stages
using F6Tile128W = F6TileShape<64, 64, 2, 4, 1, 4>;   // 128 x 256, 36 KiB stages
using F6Tile128 = F6TileShape<64, 64, 2, 2, 2, 3>;    // 128 x 128, stages of two k-steps (48 KiB)

// One k-step's operand of fragment rows `base` (+ lane row) for MFMA `mf`:
// 24 bytes = a 16-byte and an 8-byte read (mf 0) or an 8-byte and a 16-byte
// read (mf 1) at the lane's swizzled chunk offsets.
struct F6Offsets {
  int c0, c1, c2;  // byte offsets of logical chunks 3h, 3h+1, 3h+2 in the row
  __device__ __forceinline__ F6Offsets() {
    const int lane = threadIdx.x & 63;
    const int h = lane >> 5, s = ((lane & 31) >> 3) & 1;
    c0 = ((3 * h) ^ s) << 4;
    c1 = ((3 * h + 1) ^ s) << 4;
    c2 = ((3 * h + 2) ^ s) << 4;
  }
  __device__ __forceinline__ v8i operand(const char* row, int mf) const {
    if (mf == 0) {
      const f6_v4u x = *reinterpret_cast<const f6_v4u*>(row + c0);
      const f6_v2u y = *reinterpret_cast<const f6_v2u*>(row + c1);
      return v8i{(int)x[0], (int)x[1], (int)x[2], (int)x[3], (int)y[0], (int)y[1], 0, 0};
    }
    const f6_v2u y = *reinterpret_cast<const f6_v2u*>(row + c1 + 8);
    const f6_v4u x = *reinterpret_cast<const f6_v4u*>(row + c2);
    return v8i{(int)y[0], (int)y[1], (int)x[0], (int)x[1], (int)x[2], (int)x[3], 0, 0};
  }
};

__device__ __forceinline__ v16f mfma_f6(v8i w, v8i a, v16f c) {
  // cbsz = blgp = 3: both operands e3m2; scale 127 (e8m0) = 1.0
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(w, a, c, 3, 3, 0, 127, 0, 127);
}

// DMA addressing of one workgroup tile (fused gate/up: B rows 0..127 from
// the gate panel b_rsrc, 128..255 from the up panel b_rsrc2).
struct F6Tiles {
  __amdgpu_buffer_rsrc_t a_rsrc, b_rsrc, b_rsrc2;
  int64_t m0;
  int n0;
  int b_off;  // byte offset of the tile's first weight row in a 128-row block
};

// DMA of a stage: instruction q = wave + NW * slot moves KiB q of the stage,
// A rows first. voff[slot]: the lane's source offset. A: flat chunk
// f = 64 q + lane of the KG x BM x 6 stage chunks is row f / 6, stored chunk
// f % 6, which holds logical chunk (f % 6) ^ ((row >> 3) & 1), read from the
// row's 96 bytes in block row / 128: of the tile's one or two row blocks (kb
// k-steps of 12 KiB each) or, for KG 2, of the stage's two k-steps. B: the
// blocks as stored. Either way the 64 lanes of an instruction read one
// contiguous KiB; the k-step's block is in the scalar offset.
template <class T>
__device__ __forceinline__ void f6_offsets(int kb, int (&voff)[T::SLOTS]) {
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

// Scales of a tile's epilogue into the wave's LDS block `sc` by 4-byte LDS
// DMA (64 per instruction): the wave's WM row scales at byte 0 (rows past M
// read as zero) and its WN column scales at byte 512.
struct F6Scales {
  __amdgpu_buffer_rsrc_t as_rsrc;  // the whole row-scale vector
  const float* ws;
  int64_t row0;  // first row of the wave's rows
  int col0;      // first column of the wave's columns
};
// Fused gate/up (GU): the wave's WN / 2 gate column scales at byte 512 and
// its WN / 2 up column scales at byte 768 (ws2), from column col0.
template <class T, bool GU>
__device__ __forceinline__ void f6_issue_scales(char* __restrict__ sc, const F6Scales& s, const float* ws2 = nullptr) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int r = 0; r < T::WM / 64; ++r)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(s.as_rsrc, (lds_ptr_t)(sc + 256 * r), 4, lane * 4,
                                             (int)((s.row0 + 64 * r) * 4), 0, 0);
  if constexpr (GU) {
    const __amdgpu_buffer_rsrc_t g_rsrc = make_rsrc(s.ws + s.col0, T::WN / 2 * 4);
    const __amdgpu_buffer_rsrc_t u_rsrc = make_rsrc(ws2 + s.col0, T::WN / 2 * 4);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(g_rsrc, (lds_ptr_t)(sc + 512), 4, lane * 4, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(u_rsrc, (lds_ptr_t)(sc + 768), 4, lane * 4, 0, 0, 0);
  } else {
    const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(s.ws + s.col0, T::WN * 4);
#pragma unroll
    for (int c = 0; c < T::WN / 64; ++c)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(w_rsrc, (lds_ptr_t)(sc + 512 + 256 * c), 4, lane * 4, 256 * c, 0, 0);
  }
}

// DMA instruction `slot` of this wave's share of stage kt (k-steps KG kt ..)
// of tile `x` into `stage`. GU: the second half of a k-step's B rows comes
// from b_rsrc2.
template <class T, bool GU>
__device__ __forceinline__ void f6_issue_slot(char* stage, const F6Tiles& x, const int (&voff)[T::SLOTS], int kb,
                                              int kt, int slot) {
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

// DMA of stage kt of tile `x` into `stage` (all of this wave's slots).
template <class T, bool GU>
__device__ __forceinline__ void f6_issue(char* stage, const F6Tiles& x, const int (&voff)[T::SLOTS], int kb, int kt) {
#pragma unroll
  for (int slot = 0; slot < T::SLOTS; ++slot) f6_issue_slot<T, GU>(stage, x, voff, kb, kt, slot);
}

// Workgroup barrier that waits for this wave's LDS operations only (a
// __syncthreads() would also drain the DMA in flight for later k-steps).
__device__ __forceinline__ void f6_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The accumulators of the wave's EM row fragments over all of K. With two
// k-groups the waves w and w + GROUP hold the same fragments over their own
// k-steps: wave group g keeps row fragment g, takes the other group's part of
// it and gives its own part of the other, one weight fragment at a time
// through 4 KiB of LDS per wave at `ex` (integers below 2^24: the f32 sums are
// exact in any order). On entry every wave is done reading the stage `ex`
// lies in; on return every part has been read.
template <class T>
__device__ __forceinline__ void f6_reduce(const v16f (&acc)[T::TM][T::TN], v16f (&out)[T::EM][T::TN],
                                          char* __restrict__ ex) {
  static_assert(T::KG == 2 && T::TM == 2 && T::EM == 1, "one row fragment per k-group");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool hi = wave >= T::GROUP;
  char* mine = ex + wave * 4096 + lane * 16;
  const char* theirs = ex + (wave ^ T::GROUP) * 4096 + lane * 16;
#pragma unroll
  for (int j = 0; j < T::TN; ++j) {
    if (j > 0) f6_lds_barrier();  // the previous part has been read
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float4 v;
      v.x = hi ? acc[0][j][4 * q] : acc[1][j][4 * q];
      v.y = hi ? acc[0][j][4 * q + 1] : acc[1][j][4 * q + 1];
      v.z = hi ? acc[0][j][4 * q + 2] : acc[1][j][4 * q + 2];
      v.w = hi ? acc[0][j][4 * q + 3] : acc[1][j][4 * q + 3];
      *reinterpret_cast<float4*>(mine + q * 1024) = v;
    }
    f6_lds_barrier();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4 v = *reinterpret_cast<const float4*>(theirs + q * 1024);
      out[0][j][4 * q] = (hi ? acc[1][j][4 * q] : acc[0][j][4 * q]) + v.x;
      out[0][j][4 * q + 1] = (hi ? acc[1][j][4 * q + 1] : acc[0][j][4 * q + 1]) + v.y;
      out[0][j][4 * q + 2] = (hi ? acc[1][j][4 * q + 2] : acc[0][j][4 * q + 2]) + v.z;
      out[0][j][4 * q + 3] = (hi ? acc[1][j][4 * q + 3] : acc[0][j][4 * q + 3]) + v.w;
    }
  }
  f6_lds_barrier();
}

// First tile row of the rows that wave `wave` takes through the epilogue.
template <class T>
__device__ __forceinline__ int f6_wave_row(int wave) {
  const int g = wave / T::GROUP, wm = wave % T::GROUP / T::WAVES_N;
  return wm * T::WM + g * T::EM * 32;
}

// G1 value of f32(dot) (kernels/gemm_integer.loom:394-433): RN(RN(dot * ws)
// * as) + 0, finite values clamped to the bf16 finite range, then bf16.
__device__ __forceinline__ uint32_t g1_f6(float dot, float ws, float as) {
  float y = dot * ws;
  y = y * as;
  y = y + 0.0f;
  const float sat = __builtin_fmaxf(__builtin_fminf(y, kBf16Max), -kBf16Max);
  const float checked = __builtin_fabsf(y) < __builtin_huge_valf() ? sat : y;
  return f32_to_bf16(checked);
}

// Epilogue of one tile: G1 values staged per wave (32 rows at a time) and
// stored as 16-byte row pieces, the residual added on that pass. `asr` and
// `wsr` are the lane's row scales and column scales (loaded during the last
// k-step). Fast path when, over the wave's rows below M and its columns,
// every scale is finite and positive and 64 K max|ws| max|as| < bf16 max:
// the clamp cannot fire and the value is RN(RN(dot * ws) * as) + 0.
template <class T, bool RESID>
__device__ __forceinline__ void f6_epilogue(const v16f (&acc)[T::EM][T::TN], int K, int64_t M, int N,
                                            int64_t m0, int n0, const uint16_t* __restrict__ residual,
                                            uint16_t* __restrict__ out, char* __restrict__ wlds,
                                            const char* __restrict__ sc) {
  constexpr int kRowBytes = T::WN * 2, kLanesPerRow = T::WN / 8, kRowsPerRead = 64 / kLanesPerRow;
  constexpr int kReads = T::EPI_WAVE / 1024;
  int lane = threadIdx.x & 63;
  // opaque: the addresses below are computed here, not kept in registers (and
  // spilled) through the main loop
  asm volatile("" : "+v"(lane));
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wrow = f6_wave_row<T>(wave), wn = wave % T::WAVES_N;
  const int h = lane >> 5, lr = lane & 31;
  const float inf = __builtin_huge_valf();
  // the scales placed by f6_issue_scales
  float asr[T::EM];
  float4 wsr[T::TN][4];
#pragma unroll
  for (int i = 0; i < T::EM; ++i) asr[i] = *reinterpret_cast<const float*>(sc + (32 * i + lr) * 4);
#pragma unroll
  for (int j = 0; j < T::TN; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) wsr[j][q] = *reinterpret_cast<const float4*>(sc + 512 + (32 * j + 8 * q + 4 * h) * 4);
  bool ok = true;
  float amax = 0.0f, wmax = 0.0f;
#pragma unroll
  for (int i = 0; i < T::EM; ++i) {
    if (m0 + wrow + 32 * i + lr < M) {
      ok = ok & (asr[i] > 0.0f) & (asr[i] < inf);
      amax = __builtin_fmaxf(amax, asr[i]);
    }
  }
#pragma unroll
  for (int j = 0; j < T::TN; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float w4[4] = {wsr[j][q].x, wsr[j][q].y, wsr[j][q].z, wsr[j][q].w};
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        ok = ok & (w4[t] > 0.0f) & (w4[t] < inf);
        wmax = __builtin_fmaxf(wmax, w4[t]);
      }
    }
  ok = ok & (wmax * amax * (64.0f * (float)K) < kBf16Max);
  const bool fast = __all(ok);
  const int64_t rows_here = M - m0 < T::BM ? M - m0 : T::BM;
  const __amdgpu_buffer_rsrc_t out_rsrc = make_rsrc(out + m0 * N, (uint32_t)(rows_here * N * 2));
  const __amdgpu_buffer_rsrc_t res_rsrc =
      make_rsrc(RESID ? residual + m0 * N : out, RESID ? (uint32_t)(rows_here * N * 2) : 0u);
  // one copy of the loop per path (a flag tested inside would branch per value)
  auto values = [&](auto fast_tag) {
    constexpr bool FAST = decltype(fast_tag)::value;
#pragma unroll
    for (int i = 0; i < T::EM; ++i) {
      const float asv = asr[i];
#pragma unroll
      for (int j = 0; j < T::TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float w4[4] = {wsr[j][q].x, wsr[j][q].y, wsr[j][q].z, wsr[j][q].w};
          uint32_t p0, p1;
          if constexpr (FAST) {
            float y[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) y[t] = acc[i][j][4 * q + t] * w4[t] * asv + 0.0f;
            p0 = pack_bf16x2(y[0], y[1]);
            p1 = pack_bf16x2(y[2], y[3]);
          } else {
            p0 = g1_f6(acc[i][j][4 * q + 0], w4[0], asv) | (g1_f6(acc[i][j][4 * q + 1], w4[1], asv) << 16);
            p1 = g1_f6(acc[i][j][4 * q + 2], w4[2], asv) | (g1_f6(acc[i][j][4 * q + 3], w4[3], asv) << 16);
          }
          const int chunk = 4 * j + q;  // 16-byte chunk of the wave row: columns 8 * chunk .. + 7
          *reinterpret_cast<f6_v2u*>(wlds + lr * kRowBytes + ((chunk ^ (lr & 7)) << 4) + 8 * h) = f6_v2u{p0, p1};
        }
#pragma unroll
      for (int r = 0; r < kReads; ++r) {
        const int lrow = lane / kLanesPerRow, row = kRowsPerRead * r + lrow, chunk = lane % kLanesPerRow;
        f6_v4u v = *reinterpret_cast<const f6_v4u*>(wlds + row * kRowBytes + ((chunk ^ (row & 7)) << 4));
        const int voff = ((wrow + lrow) * N + n0 + wn * T::WN + 8 * chunk) * 2;
        const int soff = (32 * i + kRowsPerRead * r) * N * 2;
        if (RESID) {
          const v4i rv = __builtin_amdgcn_raw_buffer_load_b128(res_rsrc, voff, soff, 0);
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const uint32_t p = v[t], rr = (uint32_t)rv[t];
            v[t] = pack_bf16x2(bf16_lo(rr) + bf16_lo(p), bf16_hi(rr) + bf16_hi(p));
          }
        }
        store_b128(out_rsrc, voff + soff, v4i{(int)v[0], (int)v[1], (int)v[2], (int)v[3]});
      }
    }
  };
  if (fast)
    values(std::true_type{});
  else
    values(std::false_type{});
}

// Epilogue of the fused gate/up projection: h = S1(G1(gate), G1(up)) =
// bf16(silu_bf16(g) * u) for the wave's WN / 2 output columns, where the
// wave's weight fragment 0 holds gate rows and fragment 1 the up rows of the
// same columns (kernels/swiglu.loom:43-51 on the two G1 outputs, each rounded
// to bf16 first, as the separate gate, up and SwiGLU steps do). Staged per
// wave 32 rows at a time (64-byte rows, chunk q of row r at q ^ (r & 3)) and
// stored as 16-byte row pieces. The SiLU comes from the table window in LDS
// (silu_window_pair); values outside it take silu_bf16 on a wave-uniform
// branch.
template <class T>
__device__ __forceinline__ void f6_epilogue_gu(const v16f (&acc)[T::EM][T::TN], int K, int64_t M, int N,
                                               int64_t m0, int n0, uint16_t* __restrict__ out,
                                               char* __restrict__ wlds, const char* __restrict__ sc,
                                               const char* __restrict__ lut) {
  constexpr int WC = T::WN / 2;  // output columns per wave
  constexpr int kRowBytes = WC * 2, kLanesPerRow = WC / 8, kRowsPerRead = 64 / kLanesPerRow;
  constexpr int kReads = 32 / kRowsPerRead;
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));  // as in f6_epilogue
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wrow = f6_wave_row<T>(wave), wn = wave % T::WAVES_N;
  const int h = lane >> 5, lr = lane & 31;
  const float inf = __builtin_huge_valf();
  float asr[T::EM];
#pragma unroll
  for (int i = 0; i < T::EM; ++i) asr[i] = *reinterpret_cast<const float*>(sc + (32 * i + lr) * 4);
  // fast path as in f6_epilogue, over the wave's rows and both column sets
  // (the clamp cannot fire: every G1 value is RN(RN(dot * ws) * as) + 0)
  bool ok = true;
  float amax = 0.0f, wmax = 0.0f;
#pragma unroll
  for (int i = 0; i < T::EM; ++i) {
    if (m0 + wrow + 32 * i + lr < M) {
      ok = ok & (asr[i] > 0.0f) & (asr[i] < inf);
      amax = __builtin_fmaxf(amax, asr[i]);
    }
  }
  {
    // lane lr holds gate and up scale lr of the wave's 32 columns; the bound
    // takes the wave's largest column and row scales (a lane's values mix
    // rows and columns that other lanes checked)
    const float wgl = *reinterpret_cast<const float*>(sc + 512 + lr * 4);
    const float wul = *reinterpret_cast<const float*>(sc + 768 + lr * 4);
    ok = ok & (wgl > 0.0f) & (wgl < inf) & (wul > 0.0f) & (wul < inf);
    wmax = __builtin_fmaxf(wgl, wul);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      wmax = __builtin_fmaxf(wmax, __shfl_xor(wmax, off));
      amax = __builtin_fmaxf(amax, __shfl_xor(amax, off));
    }
  }
  ok = ok & (wmax * amax * (64.0f * (float)K) < kBf16Max);
  const bool fast = __all(ok);
  const int64_t rows_here = M - m0 < T::BM ? M - m0 : T::BM;
  const __amdgpu_buffer_rsrc_t out_rsrc = make_rsrc(out + m0 * N, (uint32_t)(rows_here * N * 2));
  // this lane's 16 gate and 16 up column scales (columns 8q + 4h .. + 3)
  float4 wg[4], wu[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    wg[q] = *reinterpret_cast<const float4*>(sc + 512 + (8 * q + 4 * h) * 4);
    wu[q] = *reinterpret_cast<const float4*>(sc + 768 + (8 * q + 4 * h) * 4);
  }
  // one copy of the loop per path (a wave-uniform flag tested inside would be
  // re-tested per value, a scheduling barrier between the table reads)
  auto values = [&](auto fast_tag) {
    constexpr bool FAST = decltype(fast_tag)::value;
#pragma unroll
    for (int i = 0; i < T::EM; ++i) {
      const float asv = asr[i];
      // the fragment's 16 gate and up pairs first, their 32 table reads in
      // flight together, then one wave-uniform check for values the window
      // does not cover
      uint32_t gp[4][2], upv[4][2], act[4][2];
      uint32_t outside = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float g4[4] = {wg[q].x, wg[q].y, wg[q].z, wg[q].w};
        const float u4[4] = {wu[q].x, wu[q].y, wu[q].z, wu[q].w};
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          if constexpr (FAST) {
            gp[q][p] = pack_bf16x2(acc[i][0][4 * q + 2 * p] * g4[2 * p] * asv + 0.0f,
                                   acc[i][0][4 * q + 2 * p + 1] * g4[2 * p + 1] * asv + 0.0f);
            upv[q][p] = pack_bf16x2(acc[i][1][4 * q + 2 * p] * u4[2 * p] * asv + 0.0f,
                                    acc[i][1][4 * q + 2 * p + 1] * u4[2 * p + 1] * asv + 0.0f);
          } else {
            gp[q][p] = g1_f6(acc[i][0][4 * q + 2 * p], g4[2 * p], asv) |
                       (g1_f6(acc[i][0][4 * q + 2 * p + 1], g4[2 * p + 1], asv) << 16);
            upv[q][p] = g1_f6(acc[i][1][4 * q + 2 * p], u4[2 * p], asv) |
                        (g1_f6(acc[i][1][4 * q + 2 * p + 1], u4[2 * p + 1], asv) << 16);
          }
          act[q][p] = silu_window_pair<true>(gp[q][p], lut, outside);
        }
      }
      if (__any(outside != 0)) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            uint32_t fix = 0;
            silu_window_pair<true>(gp[q][p], lut, fix);
#pragma unroll
            for (int t = 0; t < 2; ++t)
              if ((fix >> (16 * t)) & 0x8000u) {
                const uint32_t gb = (gp[q][p] >> (16 * t)) & 0xFFFFu;
                const uint32_t sb = f32_to_bf16(silu_bf16(bf16_to_f32(gb)));
                act[q][p] = (act[q][p] & (0xFFFF0000u >> (16 * t))) | (sb << (16 * t));
              }
          }
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t h0 =
            pack_bf16x2(bf16_lo(act[q][0]) * bf16_lo(upv[q][0]), bf16_hi(act[q][0]) * bf16_hi(upv[q][0]));
        const uint32_t h1 =
            pack_bf16x2(bf16_lo(act[q][1]) * bf16_lo(upv[q][1]), bf16_hi(act[q][1]) * bf16_hi(upv[q][1]));
        *reinterpret_cast<f6_v2u*>(wlds + lr * kRowBytes + ((q ^ (lr & 3)) << 4) + 8 * h) = f6_v2u{h0, h1};
      }
#pragma unroll
      for (int r = 0; r < kReads; ++r) {
        const int lrow = lane / kLanesPerRow, row = kRowsPerRead * r + lrow, chunk = lane % kLanesPerRow;
        const f6_v4u v = *reinterpret_cast<const f6_v4u*>(wlds + row * kRowBytes + ((chunk ^ (row & 3)) << 4));
        const int voff = ((wrow + 32 * i + row) * N + n0 + wn * WC + 8 * chunk) * 2;
        store_b128(out_rsrc, voff, v4i{(int)v[0], (int)v[1], (int)v[2], (int)v[3]});
      }
    }
  };
  if (fast)
    values(std::true_type{});
  else
    values(std::false_type{});
}

// DMA addressing of tile b of the grid (XCD-aware order, tile_of_block).
template <class T, bool GU>
__device__ __forceinline__ F6Tiles f6_tile(int b, int tiles_m, int tiles_n, const uint8_t* a, const uint8_t* w,
                                           const uint8_t* w2, int64_t M, int kb) {
  constexpr int TILE_N = GU ? T::BN / 2 : T::BN;  // output columns per tile
  int tm, tn;
  tile_of_block(b, tiles_m * tiles_n, tiles_m, tiles_n, tm, tn);
  F6Tiles x;
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

// DMA of the SiLU window: one KiB per wave (sign half wave / 4, KiB wave % 4).
template <class T>
__device__ __forceinline__ void f6_issue_lut(char* lds) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const __amdgpu_buffer_rsrc_t lut_rsrc = make_rsrc(g_silu_lut, kSiluLutSize * 2);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(lut_rsrc, (lds_ptr_t)(lds + T::LUT_OFF + wave * 1024), 16, lane * 16,
                                           (wave >> 2) * (kSiluLutSize / 2) * 2 + kSiluWinSrc + (wave & 3) * 1024, 0,
                                           0);
}

// Persistent bf6 G1: workgroup b walks tiles b, b + grid, ... (grid a
// multiple of 8: all on its XCD, in the XCD-aware order of tile_of_block).
// NST LDS stages in a ring, stage kt % NST holding k-step (KG k-steps) kt.
//
// What bounds it: with the operands of a k-step read and then multiplied, the
// LDS reads (144 KiB per 256 x 256 k-step, 96 KiB for the 128-row tiles) and
// the MFMAs took turns on every wave. So each MFMA round runs on operands
// that were read during the round before: while round 0 of k-step kt runs,
// round 1's operands are read; then one barrier (kt + 1 has landed for every
// wave, kt is read by every wave), and while round 1 runs, kt + 1's round-0
// operands are read and the DMA of kt + NST goes into kt's stage, one
// instruction per MFMA. M4096 K4096 N12288 123.6 -> 119.4 us, 128 x 5120 x
// 17408 99.1 -> 86.1, GU M4096 K5120 N17408 441.5 -> 422.2 (same box).
// What is left (timing-only copies, 256 x 256 tiles at M4096 K4096 N12288,
// 125.7 us on that box): without the DMA 105.7, without the LDS reads 113.2,
// without the MFMAs 91.0; at 128 x 128 tiles (37 x 5120 x 17408, 36.2 us) the
// DMA and the reads alone take 35.7.
//
// The k-steps before a tile's last load the next tile's first. The last k-step's stage stays free: the epilogue stages its output there, and
// the next tile's k-step NST - 1 goes into it afterwards. The epilogue's
// stores drain under the next tile's first k-steps.
//
// GU (fused gate/up, benches/kernels/omni_gate_up_i4.loom's dense form): a
// tile is BM rows x BN / 2 output columns of h; its B stage holds the gate
// rows (w) and the same up rows (w2) of those columns, wave (wm, wn)
// multiplies gate rows 32 wn .. and the same up rows, and the epilogue
// writes h = S1(G1(gate), G1(up)) (f6_epilogue_gu); N is the width of h.
template <class T, bool RESID, bool GU>
__global__ __launch_bounds__(T::THREADS) void gemm_f6_kernel(
    const uint8_t* __restrict__ a, const float* __restrict__ as, const uint8_t* __restrict__ w,
    const float* __restrict__ ws, int64_t M, int N, int kb, const uint16_t* __restrict__ residual,
    uint16_t* __restrict__ out, int tiles_m, int tiles_n, const uint8_t* __restrict__ w2,
    const float* __restrict__ ws2) {
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __align__(16) char lds[];
  constexpr int NST = T::NST, NF = T::TM + T::TN, MF = T::TM * T::TN;
  constexpr int STORES = T::EM * (GU ? 2 : 4);  // output stores per wave and tile
  static_assert(NST == 3 || NST == 4, "ring of three or four stages");
  const int total = tiles_m * tiles_n;  // below 2^31 (launch_f6_tile)
  int t = blockIdx.x;
  if (t >= total) return;
  auto tile = [&](int b) { return f6_tile<T, GU>(b, tiles_m, tiles_n, a, w, w2, M, kb); };
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave / T::GROUP, wm = wave % T::GROUP / T::WAVES_N, wn = wave % T::WAVES_N;
  const int lr = lane & 31;
  const int ksteps = kb / T::KG;  // k-steps (of KG) per tile
  int voff[T::SLOTS];
  f6_offsets<T>(kb, voff);
  const F6Offsets o;
  const int a_base = kg * T::A_STEP + (wm * T::WM + lr) * T::ROW;
  const int b_base = T::A_BYTES + kg * T::B_STEP + ((GU ? wn * (T::WN / 2) : wn * T::WN) + lr) * T::ROW;
  const int b_step = (GU ? T::BN / 2 : 32) * T::ROW;  // weight fragment 1: the up rows (GU)
  auto st = [&](int i) { return lds + i * T::STAGE_BYTES; };
  char* sc = lds + NST * T::STAGE_BYTES + wave * T::SCALE_WAVE;
  F6Scales scales;
  scales.as_rsrc = make_rsrc(as, (uint32_t)(M * 4));
  scales.ws = ws;
  // Waits until at most the DMA of R stages and S more operations are
  // outstanding (vector memory operations complete in issue order). Where the
  // waves' shares differ, the first QS % NW waves issue one instruction more.
  const bool full = T::QS % T::NW == 0 || wave < T::QS % T::NW;
  auto wait_stages = [&](auto r_tag, auto s_tag) {
    constexpr int R = decltype(r_tag)::value, S = decltype(s_tag)::value;
    if (full)
      wait_vmcnt<R * T::SLOTS + S>();
    else
      wait_vmcnt<R * (T::SLOTS - 1) + S>();
  };
  using I0 = std::integral_constant<int, 0>;
  using INext = std::integral_constant<int, NST - 2>;

  F6Tiles cur = tile(t);
  if constexpr (GU) f6_issue_lut<T>(lds);
  int rot = 0;         // ring position of the tile's k-step 0
  bool fresh = true;   // no k-step of this tile has been loaded by the one before
  v16f acc[T::TM][T::TN];
  v8i fr[2][NF];       // operands of the two rounds: activation fragments, weight fragments
  while (true) {
    const int t_next = t + (int)gridDim.x;
    const bool has_next = t_next < total;
    const bool chain = has_next && ksteps >= NST;  // this tile loads the next one's first k-steps
    const F6Tiles nxt = tile(has_next ? t_next : t);
    // What the DMA behind this tile's k-steps loads: the next tile's first
    // k-steps, or nothing (an empty resource: the stages get zeros that
    // nothing reads), so that every k-step issues and waits alike.
    F6Tiles ahead = nxt;
    if (!chain) ahead.a_rsrc = ahead.b_rsrc = ahead.b_rsrc2 = make_rsrc(a, 0);
    scales.row0 = cur.m0 + f6_wave_row<T>(wave);
    scales.col0 = cur.n0 + wn * (GU ? T::WN / 2 : T::WN);
#pragma unroll
    for (int i = 0; i < T::TM; ++i)
#pragma unroll
      for (int j = 0; j < T::TN; ++j) acc[i][j] = v16f{};
    // the ring as distinct restrict pointers of one body (the compiler then
    // keeps the other stages' DMA in flight across a stage's reads)
    auto tile_body = [&](char* __restrict__ r0, char* __restrict__ r1, char* __restrict__ r2, char* __restrict__ r3,
                         const char* rl, char* __restrict__ scl) {
      auto read = [&](const char* stage, int mf, int f) {
        fr[mf][f] = o.operand(f < T::TM ? stage + a_base + f * 32 * T::ROW : stage + b_base + (f - T::TM) * b_step, mf);
      };
      f6_issue_scales<T, GU>(scl, scales, ws2);
      if (fresh) {
        f6_issue<T, GU>(r0, cur, voff, kb, 0);
        if (ksteps > 1) f6_issue<T, GU>(r1, cur, voff, kb, 1);
        if (ksteps > 2) f6_issue<T, GU>(r2, cur, voff, kb, 2);
        if (NST == 4 && ksteps > 3) f6_issue<T, GU>(r3, cur, voff, kb, 3);
        if (ksteps >= NST)
          wait_stages(std::integral_constant<int, NST - 1>{}, I0{});
        else
          wait_vmcnt<0>();
        f6_lds_barrier();
      } else {
        // k-step 0 landed before the barrier that ended the last tile
        f6_issue<T, GU>(NST == 4 ? r3 : r2, cur, voff, kb, NST - 1);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int f = 0; f < NF; ++f) read(r0, 0, f);
      auto round0 = [&](const char* stage) {
#pragma unroll
        for (int x = 0; x < MF; ++x) {
          const int i = x / T::TN, j = x % T::TN;
          acc[i][j] = mfma_f6(fr[0][T::TM + j], fr[0][i], acc[i][j]);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int f = x * NF / MF; f < (x + 1) * NF / MF; ++f) read(stage, 1, f);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      auto step = [&](char* stage, const char* next, int kt) {
        round0(stage);
        // k-step kt + 1 has landed: behind it NST - 2 stages (operations in
        // between only tighten the wait)
        wait_stages(INext{}, I0{});
        f6_lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const bool own = kt + NST < ksteps;
        F6Tiles src;  // selected field by field: scalar selects
        src.a_rsrc = own ? cur.a_rsrc : ahead.a_rsrc;
        src.b_rsrc = own ? cur.b_rsrc : ahead.b_rsrc;
        src.b_rsrc2 = own ? cur.b_rsrc2 : ahead.b_rsrc2;
        src.b_off = own ? cur.b_off : ahead.b_off;
        const int ks = own ? kt + NST : kt + NST - ksteps;
#pragma unroll
        for (int x = 0; x < MF; ++x) {
          const int i = x / T::TN, j = x % T::TN;
          acc[i][j] = mfma_f6(fr[1][T::TM + j], fr[1][i], acc[i][j]);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int f = x * NF / MF; f < (x + 1) * NF / MF; ++f) read(next, 0, f);
#pragma unroll
          for (int slot = x * T::SLOTS / MF; slot < (x + 1) * T::SLOTS / MF; ++slot)
            f6_issue_slot<T, GU>(stage, src, voff, kb, ks, slot);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      const int steps = ksteps - 1;
      for (int kt = 0; kt < steps; kt += NST) {
        step(r0, r1, kt);
        if (kt + 1 < steps) step(r1, r2, kt + 1);
        if (kt + 2 < steps) step(r2, NST == 4 ? r3 : r0, kt + 2);
        if constexpr (NST == 4)
          if (kt + 3 < steps) step(r3, r0, kt + 3);
      }
      // the last k-step, whose stage takes no DMA
      round0(rl);
      f6_lds_barrier();  // read by every wave
#pragma unroll
      for (int x = 0; x < MF; ++x) {
        const int i = x / T::TN, j = x % T::TN;
        acc[i][j] = mfma_f6(fr[1][T::TM + j], fr[1][i], acc[i][j]);
      }
    };
    char* last = st((rot + ksteps - 1) % NST);
    tile_body(st(rot), st((rot + 1) % NST), st((rot + 2) % NST), st((rot + 3) % NST), last, sc);
    // this tile's scales have landed: issued before k-step NST - 1, which the
    // loop waited for
    if (ksteps < NST || !chain) wait_vmcnt<0>();
    auto epilogue = [&](const v16f (&sum)[T::EM][T::TN]) {
      if constexpr (GU)
        f6_epilogue_gu<T>(sum, kb * 128, M, N, cur.m0, cur.n0, out, last + wave * T::EPI_WAVE, sc, lds + T::LUT_OFF);
      else
        f6_epilogue<T, RESID>(sum, kb * 128, M, N, cur.m0, cur.n0, residual, out, last + wave * T::EPI_WAVE, sc);
    };
    if constexpr (T::KG == 1) {
      epilogue(acc);
    } else {
      v16f sum[T::EM][T::TN];
      f6_reduce<T>(acc, sum, last);
      epilogue(sum);
    }
    if (!has_next) break;
    // the next tile's k-step 0 has landed: behind it k-steps 1 .. NST - 2 and
    // this tile's stores
    if (chain) wait_stages(INext{}, std::integral_constant<int, STORES>{});
    f6_lds_barrier();  // for every wave, and every wave is done with the staging stage
    fresh = !chain;
    rot = (rot + ksteps) % NST;
    t = t_next;
    cur = nxt;
  }
#endif
}

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

  const F6Offsets o;
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
        for (int j = 0; j < MT; ++j) acc[i][j] = mfma_f6(fw[mf][i], fa[mf][j], acc[i][j]);
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

// Operands of one launch. GU: w / ws the gate weight, w2 / ws2 the up weight,
// n the width of h (n % 128 == 0), out = h.
struct F6Args {
  const uint8_t* a;
  const float* as;
  const uint8_t* w;
  const float* ws;
  int64_t m;
  int n, k;
  const uint16_t* residual;
  uint16_t* out;
  const uint8_t* w2;
  const float* ws2;
};

template <class T, bool RESID, bool GU>
hipError_t launch_f6_tile(const F6Args& x, hipStream_t stream) {
  constexpr int lds = GU ? T::LDS_GU : T::LDS;
  static_assert(lds <= 160 * 1024, "LDS per workgroup");
  static LaunchCache cache;
  auto* kernel = &gemm_f6_kernel<T, RESID, GU>;
  const void* kern = reinterpret_cast<const void*>(kernel);
  if (hipError_t e = ensure_dynamic_lds(cache, kern, lds)) return e;
  int per_cu = 0, cus = 0;
  if (hipError_t e = resident_per_cu(cache, kern, T::THREADS, lds, per_cu, cus)) return e;
  const int tiles_n = x.n / (GU ? T::BN / 2 : T::BN);
  const int64_t tiles_m = (x.m + T::BM - 1) / T::BM;
  const int64_t total = tiles_m * tiles_n;
  if (total > kMaxTiles) return hipErrorInvalidValue;  // the kernel's 32-bit tile indices
  int64_t grid = (int64_t)cus * per_cu / 8 * 8;
  if (grid < 8) grid = 8;
  if (grid > total) grid = total;
  kernel<<<(unsigned)grid, T::THREADS, lds, stream>>>(
      x.a, x.as, x.w, x.ws, x.m, x.n, x.k / 128, x.residual, x.out, (int)tiles_m, tiles_n, x.w2, x.ws2);
  return hipGetLastError();
}

template <int MT, int NT, int NB, bool RESID, bool GU>
hipError_t launch_f6_ksplit(const F6Args& x, hipStream_t stream) {
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
hipError_t launch_gemm_f6_impl(const F6Args& x, hipStream_t stream) {
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
  if (c128 <= c128w && c128 <= c256) return launch_f6_tile<F6Tile128, RESID, GU>(x, stream);
  if (c128w < c256) return launch_f6_tile<F6Tile128W, RESID, GU>(x, stream);
  return launch_f6_tile<F6Tile256, RESID, GU>(x, stream);
}

}  // namespace

hipError_t launch_f6_rows(const uint32_t* a, int a_words, int64_t rows, int k, uint8_t* out, hipStream_t stream) {
  const int64_t total = rows * (k / 32);
  const int64_t blocks = (total + 255) / 256;
  f6_rows_kernel<<<(unsigned)(blocks < 8192 ? blocks : 8192), 256, 0, stream>>>(a, a_words, rows, k, out);
  return hipGetLastError();
}

hipError_t launch_f6_tiled(const uint32_t* w_tiled, int64_t n, int k, uint8_t* out, hipStream_t stream) {
  const int64_t total = n * (k / 32);
  const int64_t blocks = (total + 255) / 256;
  f6_tiled_kernel<<<(unsigned)(blocks < 8192 ? blocks : 8192), 256, 0, stream>>>(w_tiled, total, out);
  return hipGetLastError();
}

hipError_t launch_gemm_f6(const uint8_t* a, const float* as, const uint8_t* w, const float* ws, int64_t m, int n,
                          int k, const uint16_t* residual, uint16_t* out, hipStream_t stream) {
  const F6Args x{a, as, w, ws, m, n, k, residual, out, nullptr, nullptr};
  return residual ? launch_gemm_f6_impl<true, false>(x, stream) : launch_gemm_f6_impl<false, false>(x, stream);
}

hipError_t launch_gemm_f6_gate_up(const uint8_t* a, const float* as, const uint8_t* gate_w, const float* gate_s,
                                  const uint8_t* up_w, const float* up_s, int64_t m, int n, int k, uint16_t* h,
                                  hipStream_t stream) {
  return launch_gemm_f6_impl<false, true>(F6Args{a, as, gate_w, gate_s, m, n, k, nullptr, h, up_w, up_s}, stream);
}

}  // namespace clef
