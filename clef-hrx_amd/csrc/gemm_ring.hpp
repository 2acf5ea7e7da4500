// Persistent G1 on operands that are multiplied as LDS holds them (bf6 codes,
// gemm_f6.hip; INT8 codes, gemm_i8.hip): the tile shapes, the ring of LDS
// stages, the epilogues and the kernel. An operand form `Op` gives the bytes of
// a row per k-step, the DMA addressing, a fragment's LDS read and the MFMA.
#pragma once

#include <type_traits>

#include "common.hpp"
#include "gemm_dma.hpp"
#include "kernels.hpp"
#include "launch.hpp"
#include "silu_table.hpp"

namespace clef {

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef unsigned v2u __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// Tile shape: KG groups of WAVES_M x WAVES_N waves, each wave
// WM rows x WN weight rows; a stage holds KG k-steps and group g contracts
// the g-th of them.
// SPLIT: a row of a stage holds the groups' k-steps side by side (ROW bytes in
// all); otherwise each group has its own rows.
template <int ROW_, int WM_, int WN_, int WAVES_M_, int WAVES_N_, int KG_, int NST_, bool SPLIT_ = false>
struct RingTile {
  static constexpr int WM = WM_, WN = WN_, WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, KG = KG_;
  static constexpr int NST = NST_;                              // LDS stages
  static constexpr int GROUP = WAVES_M * WAVES_N;               // waves per k-group
  static constexpr int NW = GROUP * KG, THREADS = 64 * NW;
  static constexpr int BM = WM * WAVES_M, BN = WN * WAVES_N;
  static constexpr int TM = WM / 32, TN = WN / 32;              // fragments per wave
  static constexpr int EM = TM / KG;                            // row fragments a wave takes through the epilogue
  static constexpr int ROW = ROW_;                              // bytes per row per k-step
  static constexpr int A_STEP = BM * ROW, B_STEP = BN * ROW;    // bytes of one k-step
  static constexpr bool SPLIT = SPLIT_;
  static constexpr int A_BYTES = (SPLIT ? 1 : KG) * A_STEP, B_BYTES = (SPLIT ? 1 : KG) * B_STEP;
  static constexpr int STAGE_BYTES = A_BYTES + B_BYTES;
  static constexpr int A_QS = A_BYTES / 1024, QS = STAGE_BYTES / 1024;  // DMA instructions per stage
  static constexpr int SLOTS = (QS + NW - 1) / NW;              // and per wave, at most
  static constexpr int EPI_WAVE = 32 * WN * 2;                  // staging bytes per wave (32 rows of WN bf16)
  static constexpr int SCALE_WAVE = 1024;                       // per-wave epilogue scales (768 bytes used)
  static constexpr int LDS = NST * STAGE_BYTES + NW * SCALE_WAVE;
  // fused gate/up: the SiLU window after the scales
  static constexpr int LUT_OFF = LDS;
  static constexpr int LDS_GU = LUT_OFF + kSiluWinBytes;
  static_assert(NW == 8 && LDS_GU <= 160 * 1024, "workgroup shape");
  static_assert(NW * EPI_WAVE <= STAGE_BYTES, "the epilogue stages its output in one free stage");
};
// DMA addressing of one workgroup tile (fused gate/up: the first
// half of a k-step's B rows from the gate panel b_rsrc, the second from the up
// panel b_rsrc2).
struct RingTiles {
  __amdgpu_buffer_rsrc_t a_rsrc, b_rsrc, b_rsrc2;
  int64_t m0;
  int n0;
  int b_off;  // byte offset of the tile's first weight row in a 128-row block
};

// Scales of a tile's epilogue into the wave's LDS block `sc` by 4-byte LDS
// DMA (64 per instruction): the wave's WM row scales at byte 0 (rows past M
// read as zero) and its WN column scales at byte 512.
struct RingScales {
  __amdgpu_buffer_rsrc_t as_rsrc;  // the whole row-scale vector
  const float* ws;
  int64_t row0;  // first row of the wave's rows
  int col0;      // first column of the wave's columns
};
// Fused gate/up (GU): the wave's WN / 2 gate column scales at byte 512 and
// its WN / 2 up column scales at byte 768 (ws2), from column col0.
template <class T, bool GU>
__device__ __forceinline__ void ring_issue_scales(char* __restrict__ sc, const RingScales& s, const float* ws2 = nullptr) {
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

// DMA of stage kt of tile `x` into `stage` (all of this wave's slots).
template <class Op, class T, bool GU>
__device__ __forceinline__ void ring_issue(char* stage, const RingTiles& x, const int (&voff)[T::SLOTS], int kb, int kt) {
#pragma unroll
  for (int slot = 0; slot < T::SLOTS; ++slot) Op::template issue_slot<T, GU>(stage, x, voff, kb, kt, slot);
}

// Workgroup barrier that waits for this wave's LDS operations only (a
// __syncthreads() would also drain the DMA in flight for later k-steps).
__device__ __forceinline__ void ring_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The accumulators of the wave's EM row fragments over all of K. With two
// k-groups the waves w and w + GROUP hold the same fragments over their own
// k-steps: wave group g keeps row fragment g, takes the other group's part of
// it and gives its own part of the other, one weight fragment at a time
// through 4 KiB of LDS per wave at `ex` (integers: exact in any order). On entry every wave is done reading the stage `ex`
// lies in; on return every part has been read.
template <class T, class Acc>
__device__ __forceinline__ void ring_reduce(const Acc (&acc)[T::TM][T::TN], Acc (&out)[T::EM][T::TN],
                                          char* __restrict__ ex) {
  static_assert(T::KG == 2 && T::TM == 2 && T::EM == 1, "one row fragment per k-group");
  typedef std::remove_reference_t<decltype(out[0][0][0])> elem;
  typedef elem v4e __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool hi = wave >= T::GROUP;
  char* mine = ex + wave * 4096 + lane * 16;
  const char* theirs = ex + (wave ^ T::GROUP) * 4096 + lane * 16;
#pragma unroll
  for (int j = 0; j < T::TN; ++j) {
    if (j > 0) ring_lds_barrier();  // the previous part has been read
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v4e v;
      v[0] = hi ? acc[0][j][4 * q] : acc[1][j][4 * q];
      v[1] = hi ? acc[0][j][4 * q + 1] : acc[1][j][4 * q + 1];
      v[2] = hi ? acc[0][j][4 * q + 2] : acc[1][j][4 * q + 2];
      v[3] = hi ? acc[0][j][4 * q + 3] : acc[1][j][4 * q + 3];
      *reinterpret_cast<v4e*>(mine + q * 1024) = v;
    }
    ring_lds_barrier();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const v4e v = *reinterpret_cast<const v4e*>(theirs + q * 1024);
      out[0][j][4 * q] = (hi ? acc[1][j][4 * q] : acc[0][j][4 * q]) + v[0];
      out[0][j][4 * q + 1] = (hi ? acc[1][j][4 * q + 1] : acc[0][j][4 * q + 1]) + v[1];
      out[0][j][4 * q + 2] = (hi ? acc[1][j][4 * q + 2] : acc[0][j][4 * q + 2]) + v[2];
      out[0][j][4 * q + 3] = (hi ? acc[1][j][4 * q + 3] : acc[0][j][4 * q + 3]) + v[3];
    }
  }
  ring_lds_barrier();
}

// First tile row of the rows that wave `wave` takes through the epilogue.
template <class T>
__device__ __forceinline__ int ring_wave_row(int wave) {
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
// every scale is finite and positive and dot_max max|ws| max|as| < bf16 max
// (dot_max: the largest |dot| codes can give):
// the clamp cannot fire and the value is RN(RN(dot * ws) * as) + 0.
template <class T, bool RESID, class Acc>
__device__ __forceinline__ void ring_epilogue(const Acc (&acc)[T::EM][T::TN], float dot_max, int64_t M, int N,
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
  const int wrow = ring_wave_row<T>(wave), wn = wave % T::WAVES_N;
  const int h = lane >> 5, lr = lane & 31;
  const float inf = __builtin_huge_valf();
  // the scales placed by ring_issue_scales
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
  ok = ok & (wmax * amax * dot_max < kBf16Max);
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
            for (int t = 0; t < 4; ++t) y[t] = (float)acc[i][j][4 * q + t] * w4[t] * asv + 0.0f;
            p0 = pack_bf16x2(y[0], y[1]);
            p1 = pack_bf16x2(y[2], y[3]);
          } else {
            p0 = g1_f6((float)acc[i][j][4 * q + 0], w4[0], asv) | (g1_f6((float)acc[i][j][4 * q + 1], w4[1], asv) << 16);
            p1 = g1_f6((float)acc[i][j][4 * q + 2], w4[2], asv) | (g1_f6((float)acc[i][j][4 * q + 3], w4[3], asv) << 16);
          }
          const int chunk = 4 * j + q;  // 16-byte chunk of the wave row: columns 8 * chunk .. + 7
          *reinterpret_cast<v2u*>(wlds + lr * kRowBytes + ((chunk ^ (lr & 7)) << 4) + 8 * h) = v2u{p0, p1};
        }
#pragma unroll
      for (int r = 0; r < kReads; ++r) {
        const int lrow = lane / kLanesPerRow, row = kRowsPerRead * r + lrow, chunk = lane % kLanesPerRow;
        v4u v = *reinterpret_cast<const v4u*>(wlds + row * kRowBytes + ((chunk ^ (row & 7)) << 4));
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
template <class T, class Acc>
__device__ __forceinline__ void ring_epilogue_gu(const Acc (&acc)[T::EM][T::TN], float dot_max, int64_t M, int N,
                                               int64_t m0, int n0, uint16_t* __restrict__ out,
                                               char* __restrict__ wlds, const char* __restrict__ sc,
                                               const char* __restrict__ lut) {
  constexpr int WC = T::WN / 2;  // output columns per wave
  constexpr int kRowBytes = WC * 2, kLanesPerRow = WC / 8, kRowsPerRead = 64 / kLanesPerRow;
  constexpr int kReads = 32 / kRowsPerRead;
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));  // as in ring_epilogue
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wrow = ring_wave_row<T>(wave), wn = wave % T::WAVES_N;
  const int h = lane >> 5, lr = lane & 31;
  const float inf = __builtin_huge_valf();
  float asr[T::EM];
#pragma unroll
  for (int i = 0; i < T::EM; ++i) asr[i] = *reinterpret_cast<const float*>(sc + (32 * i + lr) * 4);
  // fast path as in ring_epilogue, over the wave's rows and both column sets
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
  ok = ok & (wmax * amax * dot_max < kBf16Max);
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
            gp[q][p] = pack_bf16x2((float)acc[i][0][4 * q + 2 * p] * g4[2 * p] * asv + 0.0f,
                                   (float)acc[i][0][4 * q + 2 * p + 1] * g4[2 * p + 1] * asv + 0.0f);
            upv[q][p] = pack_bf16x2((float)acc[i][1][4 * q + 2 * p] * u4[2 * p] * asv + 0.0f,
                                    (float)acc[i][1][4 * q + 2 * p + 1] * u4[2 * p + 1] * asv + 0.0f);
          } else {
            gp[q][p] = g1_f6((float)acc[i][0][4 * q + 2 * p], g4[2 * p], asv) |
                       (g1_f6((float)acc[i][0][4 * q + 2 * p + 1], g4[2 * p + 1], asv) << 16);
            upv[q][p] = g1_f6((float)acc[i][1][4 * q + 2 * p], u4[2 * p], asv) |
                        (g1_f6((float)acc[i][1][4 * q + 2 * p + 1], u4[2 * p + 1], asv) << 16);
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
        *reinterpret_cast<v2u*>(wlds + lr * kRowBytes + ((q ^ (lr & 3)) << 4) + 8 * h) = v2u{h0, h1};
      }
#pragma unroll
      for (int r = 0; r < kReads; ++r) {
        const int lrow = lane / kLanesPerRow, row = kRowsPerRead * r + lrow, chunk = lane % kLanesPerRow;
        const v4u v = *reinterpret_cast<const v4u*>(wlds + row * kRowBytes + ((chunk ^ (row & 3)) << 4));
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

// DMA of the SiLU window: one KiB per wave (sign half wave / 4, KiB wave % 4).
template <class T>
__device__ __forceinline__ void ring_issue_lut(char* lds) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const __amdgpu_buffer_rsrc_t lut_rsrc = make_rsrc(g_silu_lut, kSiluLutSize * 2);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(lut_rsrc, (lds_ptr_t)(lds + T::LUT_OFF + wave * 1024), 16, lane * 16,
                                           (wave >> 2) * (kSiluLutSize / 2) * 2 + kSiluWinSrc + (wave & 3) * 1024, 0,
                                           0);
}

// Persistent G1: workgroup b walks tiles b, b + grid, ... (grid a
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
// The k-steps before a tile's last load the next tile's first. The last k-step's
// stage stays free: the epilogue stages its output there, and the next tile's
// k-step NST - 1 goes into it afterwards. The epilogue's stores drain under the
// next tile's first k-steps. A tile of NST - 1 k-steps leaves one stage of the
// ring free from its start, which takes the next tile's k-step 0. Tiles of fewer
// load, contract and store in turn.
//
// GU (fused gate/up, benches/kernels/omni_gate_up_i4.loom's dense form): a
// tile is BM rows x BN / 2 output columns of h; its B stage holds the gate
// rows (w) and the same up rows (w2) of those columns, wave (wm, wn)
// multiplies gate rows 32 wn .. and the same up rows, and the epilogue
// writes h = S1(G1(gate), G1(up)) (ring_epilogue_gu); N is the width of h.
template <class Op, class T, bool RESID, bool GU>
__global__ __launch_bounds__(T::THREADS) void gemm_ring_kernel(
    const uint8_t* __restrict__ a, int a_row_bytes, const float* __restrict__ as, const uint8_t* __restrict__ w,
    const float* __restrict__ ws, int64_t M, int N, int kb, const uint16_t* __restrict__ residual,
    uint16_t* __restrict__ out, int tiles_m, int tiles_n, const uint8_t* __restrict__ w2,
    const float* __restrict__ ws2) {
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __align__(16) char lds[];
  constexpr int NST = T::NST, NF = T::TM + T::TN, MF = T::TM * T::TN;
  constexpr int STORES = T::EM * (GU ? 2 : 4);  // output stores per wave and tile
  static_assert(NST == 3 || NST == 4, "ring of three or four stages");
  const int total = tiles_m * tiles_n;  // below 2^31 (launch_ring)
  int t = blockIdx.x;
  if (t >= total) return;
  auto tile = [&](int b) { return Op::template tile<T, GU>(b, tiles_m, tiles_n, a, a_row_bytes, w, w2, M, kb); };
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kg = wave / T::GROUP, wm = wave % T::GROUP / T::WAVES_N, wn = wave % T::WAVES_N;
  const int lr = lane & 31;
  const int ksteps = kb / T::KG;  // k-steps (of KG) per tile
  int voff[T::SLOTS];
  Op::template offsets<T>(kb, a_row_bytes, voff);
  const typename Op::Reader o(kg);
  const int a_base = (T::SPLIT ? 0 : kg * T::A_STEP) + (wm * T::WM + lr) * T::ROW;
  const int b_base = T::A_BYTES + (T::SPLIT ? 0 : kg * T::B_STEP) + ((GU ? wn * (T::WN / 2) : wn * T::WN) + lr) * T::ROW;
  const int b_step = (GU ? T::BN / 2 : 32) * T::ROW;  // weight fragment 1: the up rows (GU)
  auto st = [&](int i) { return lds + i * T::STAGE_BYTES; };
  char* sc = lds + NST * T::STAGE_BYTES + wave * T::SCALE_WAVE;
  RingScales scales;
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

  RingTiles cur = tile(t);
  if constexpr (GU) ring_issue_lut<T>(lds);
  int rot = 0;         // ring position of the tile's k-step 0
  bool fresh = true;   // no k-step of this tile has been loaded by the one before
  typename Op::Acc acc[T::TM][T::TN];
  typename Op::Frag fr[2][NF];       // operands of the two rounds: activation fragments, weight fragments
  while (true) {
    const int t_next = t + (int)gridDim.x;
    const bool has_next = t_next < total;
    const bool chain = has_next && ksteps >= NST - 1;  // this tile loads the next one's first k-steps
    const RingTiles nxt = tile(has_next ? t_next : t);
    // What the DMA behind this tile's k-steps loads: the next tile's first
    // k-steps, or nothing (an empty resource: the stages get zeros that
    // nothing reads), so that every k-step issues and waits alike.
    RingTiles ahead = nxt;
    if (!chain) ahead.a_rsrc = ahead.b_rsrc = ahead.b_rsrc2 = make_rsrc(a, 0);
    scales.row0 = cur.m0 + ring_wave_row<T>(wave);
    scales.col0 = cur.n0 + wn * (GU ? T::WN / 2 : T::WN);
#pragma unroll
    for (int i = 0; i < T::TM; ++i)
#pragma unroll
      for (int j = 0; j < T::TN; ++j) acc[i][j] = typename Op::Acc{};
    // the ring as distinct restrict pointers of one body (the compiler then
    // keeps the other stages' DMA in flight across a stage's reads)
    auto tile_body = [&](char* __restrict__ r0, char* __restrict__ r1, char* __restrict__ r2, char* __restrict__ r3,
                         const char* rl, char* __restrict__ scl) {
      auto read = [&](const char* stage, int mf, int f) {
        fr[mf][f] = o.operand(f < T::TM ? stage + a_base + f * 32 * T::ROW : stage + b_base + (f - T::TM) * b_step, mf);
      };
      ring_issue_scales<T, GU>(scl, scales, ws2);
      if (fresh) {
        ring_issue<Op, T, GU>(r0, cur, voff, kb, 0);
        if (ksteps > 1) ring_issue<Op, T, GU>(r1, cur, voff, kb, 1);
        if (NST == 4 && ksteps > 2) ring_issue<Op, T, GU>(r2, cur, voff, kb, 2);
      }  // else k-step 0 landed before the barrier that ended the last tile
      if (ksteps >= NST)
        ring_issue<Op, T, GU>(NST == 4 ? r3 : r2, cur, voff, kb, NST - 1);
      else if (ksteps == NST - 1)
        ring_issue<Op, T, GU>(NST == 4 ? r3 : r2, ahead, voff, kb, 0);
      if (fresh) {
        if (ksteps >= NST - 1)
          wait_stages(std::integral_constant<int, NST - 1>{}, I0{});
        else
          wait_vmcnt<0>();
        ring_lds_barrier();
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int f = 0; f < NF; ++f) read(r0, 0, f);
      auto round0 = [&](const char* stage) {
#pragma unroll
        for (int x = 0; x < MF; ++x) {
          const int i = x / T::TN, j = x % T::TN;
          acc[i][j] = Op::mfma(fr[0][T::TM + j], fr[0][i], acc[i][j]);
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
        ring_lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const bool own = kt + NST < ksteps;
        RingTiles src;  // selected field by field: scalar selects
        src.a_rsrc = own ? cur.a_rsrc : ahead.a_rsrc;
        src.b_rsrc = own ? cur.b_rsrc : ahead.b_rsrc;
        src.b_rsrc2 = own ? cur.b_rsrc2 : ahead.b_rsrc2;
        src.b_off = own ? cur.b_off : ahead.b_off;
        const int ks = own ? kt + NST : kt + NST - ksteps;
#pragma unroll
        for (int x = 0; x < MF; ++x) {
          const int i = x / T::TN, j = x % T::TN;
          acc[i][j] = Op::mfma(fr[1][T::TM + j], fr[1][i], acc[i][j]);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int f = x * NF / MF; f < (x + 1) * NF / MF; ++f) read(next, 0, f);
#pragma unroll
          for (int slot = x * T::SLOTS / MF; slot < (x + 1) * T::SLOTS / MF; ++slot)
            Op::template issue_slot<T, GU>(stage, src, voff, kb, ks, slot);
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
      ring_lds_barrier();  // read by every wave
#pragma unroll
      for (int x = 0; x < MF; ++x) {
        const int i = x / T::TN, j = x % T::TN;
        acc[i][j] = Op::mfma(fr[1][T::TM + j], fr[1][i], acc[i][j]);
      }
    };
    char* last = st((rot + ksteps - 1) % NST);
    tile_body(st(rot), st((rot + 1) % NST), st((rot + 2) % NST), st((rot + 3) % NST), last, sc);
    // this tile's scales have landed: issued before k-step NST - 1, which the
    // loop waited for
    if (!chain) wait_vmcnt<0>();
    auto epilogue = [&](const typename Op::Acc (&sum)[T::EM][T::TN]) {
      if constexpr (GU)
        ring_epilogue_gu<T>(sum, Op::kDotPerStep * (float)kb, M, N, cur.m0, cur.n0, out, last + wave * T::EPI_WAVE, sc, lds + T::LUT_OFF);
      else
        ring_epilogue<T, RESID>(sum, Op::kDotPerStep * (float)kb, M, N, cur.m0, cur.n0, residual, out, last + wave * T::EPI_WAVE, sc);
    };
    if constexpr (T::KG == 1) {
      epilogue(acc);
    } else {
      typename Op::Acc sum[T::EM][T::TN];
      ring_reduce<T>(acc, sum, last);
      epilogue(sum);
    }
    if (!has_next) break;
    // the next tile's k-step 0 has landed: behind it k-steps 1 .. NST - 2 and
    // this tile's stores
    if (chain) wait_stages(INext{}, std::integral_constant<int, STORES>{});
    ring_lds_barrier();  // for every wave, and every wave is done with the staging stage
    fresh = !chain;
    rot = (rot + ksteps) % NST;
    t = t_next;
    cur = nxt;
  }
#endif
}

// Operands of one launch. GU: w / ws the gate weight, w2 / ws2 the up weight,
// n the width of h, out = h.
struct RingArgs {
  const uint8_t* a;
  int a_row_bytes;  // row pitch of row-major activation codes
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

template <class Op, class T, bool RESID, bool GU>
hipError_t launch_ring(const RingArgs& x, hipStream_t stream) {
  constexpr int lds = GU ? T::LDS_GU : T::LDS;
  static LaunchCache cache;
  auto* kernel = &gemm_ring_kernel<Op, T, RESID, GU>;
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
  kernel<<<(unsigned)grid, T::THREADS, lds, stream>>>(x.a, x.a_row_bytes, x.as, x.w, x.ws, x.m, x.n,
                                                      x.k / Op::kStep, x.residual, x.out, (int)tiles_m, tiles_n,
                                                      x.w2, x.ws2);
  return hipGetLastError();
}

}  // namespace

}  // namespace clef
