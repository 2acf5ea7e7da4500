// G1 on INT8 codes (h3_gemm_i8_256, kernels/gemm_integer.loom:454-485): the
// ring kernel of gemm_ring.hpp on v_mfma_i32_32x32x32_i8. A 16-byte read of
// LDS is an operand as it stands (16 codes; lane half h takes the odd chunk of
// a pair), so a k-step is 64 k: 64 bytes per row, two MFMA rounds.
#include "gemm_ring.hpp"

namespace clef {

namespace {

struct I8Op {
  typedef v16i Acc;
  typedef v4i Frag;
  static constexpr int kStep = 64;
  [[maybe_unused]] static constexpr float kDotPerStep = 16384.0f * kStep;  // |dot| per k-step, codes of magnitude 128

  // A stage row is 128 bytes, both groups' k-steps (one row of a weight block);
  // row r's logical 16-byte chunk c is stored at c ^ ((r >> 1) & 7): 16
  // consecutive rows of one chunk cover the 64 banks once. Round s of group kg
  // takes chunk 4 kg + 2 s + h.
  struct Reader {
    int c[2];
    __device__ __forceinline__ explicit Reader(int kg) {
      const int lane = threadIdx.x & 63;
      const int h = lane >> 5, g = ((lane & 31) >> 1) & 7;
      c[0] = ((4 * kg + h) ^ g) << 4;
      c[1] = ((4 * kg + 2 + h) ^ g) << 4;
    }
    __device__ __forceinline__ v4i operand(const char* row, int s) const {
      return *reinterpret_cast<const v4i*>(row + c[s]);
    }
  };

  __device__ __forceinline__ static v16i mfma(v4i w, v4i a, v16i c) { return mfma32_i8(w, a, c); }

  // DMA instruction q moves 8 whole 128-byte rows, lane -> row 8 q + lane / 8,
  // stored chunk lane % 8. Activation rows are a_row_bytes apart, weight rows
  // those of a tiled block. Whole lines per instruction: with each group's 64
  // bytes in rows of their own, 16 half lines an instruction, every line was
  // requested twice (m x n x k, graph replay, three runs of each in turn:
  // 235 x 12288 x 4096 21.8 -> 20.5 us, 620 x 4096 x 12288 49.5 -> 46.5,
  // 620 x 5120 x 6144 29.8 -> 27.8, 1000 x 12288 x 4096 69.2 -> 67.5).
  template <class T>
  __device__ __forceinline__ static void offsets(int, int a_row_bytes, int (&voff)[T::SLOTS]) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int slot = 0; slot < T::SLOTS; ++slot) {
      const int q = wave + T::NW * slot;
      const bool is_a = T::NW * slot < T::A_QS;
      const int row = 8 * (is_a ? q : q - T::A_QS) + (lane >> 3);
      voff[slot] = (is_a ? row * a_row_bytes : row * 128) + (((lane & 7) ^ ((row >> 1) & 7)) << 4);
    }
  }

  template <class T, bool GU>
  __device__ __forceinline__ static void issue_slot(char* stage, const RingTiles& x, const int (&voff)[T::SLOTS],
                                                    int, int kt, int slot) {
    static_assert(!GU && T::A_QS % T::NW == 0 && T::QS % T::NW == 0 && T::KG == 2 && T::SPLIT && T::BN == 128, "whole slots");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = wave + T::NW * slot;
    const lds_ptr_t dst = (lds_ptr_t)(stage + q * 1024);
    if (T::NW * slot < T::A_QS) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x.a_rsrc, dst, 16, voff[slot], kt * 128, 0, 0);
    } else {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(x.b_rsrc, dst, 16, voff[slot], kt * 16384, 0, 0);
    }
  }

  template <class T, bool GU>
  __device__ __forceinline__ static RingTiles tile(int b, int tiles_m, int tiles_n, const uint8_t* a, int a_row_bytes,
                                                   const uint8_t* w, const uint8_t*, int64_t M, int kb) {
    int tm, tn;
    tile_of_block(b, tiles_m * tiles_n, tiles_m, tiles_n, tm, tn);
    RingTiles x;
    x.m0 = (int64_t)tm * T::BM;
    x.n0 = tn * T::BN;
    x.b_off = 0;
    // rows past M are outside the resource and read as zero
    const int64_t rows = M - x.m0 < T::BM ? M - x.m0 : T::BM;
    x.a_rsrc = make_rsrc(a + x.m0 * a_row_bytes, (uint32_t)(rows * a_row_bytes));
    const int block_bytes = kb / 2 * 16384;
    x.b_rsrc = make_rsrc(w + (int64_t)(x.n0 / 128) * block_bytes, (uint32_t)(T::BN / 128 * block_bytes));
    x.b_rsrc2 = x.b_rsrc;
    return x;
  }
};

// 128 x 128 tiles, 32 KiB stages of 128-byte rows (the two groups split each row)
using I8Tile128 = RingTile<128, 64, 64, 2, 2, 2, 4, true>;

}  // namespace

hipError_t launch_gemm_i8_ring(const uint32_t* a, int a_words, const float* as, const uint32_t* w, const float* ws,
                               int64_t m, int n, int k, const uint16_t* residual, uint16_t* out, hipStream_t stream) {
  const RingArgs x{reinterpret_cast<const uint8_t*>(a), 4 * a_words, as, reinterpret_cast<const uint8_t*>(w), ws, m, n, k,
                   residual, out, nullptr, nullptr};
  return residual ? launch_ring<I8Op, I8Tile128, true, false>(x, stream)
                  : launch_ring<I8Op, I8Tile128, false, false>(x, stream);
}

}  // namespace clef
