// Grouped expert GEMM for few routed rows per expert (more than the dot-product
// kernel takes, on the schedule's 32-slot tiles): the experts' weights stream
// once through LDS, and that stream is the whole cost.
//
// A workgroup of four waves owns one tile and 128 SPW output columns of its
// expert. The tile's 32 gathered activation rows stay in LDS for all of K
// (kb x 4 KiB, one copy for the four waves). Each wave walks its own SPW
// slices of 32 columns (GU: 32 gate rows, then the same 32 up rows of a
// k-step) through a private ring of NB 4 KiB stages, 32 weight rows x 256 k
// each, in whole 128-byte rows by LDS DMA: a stage is read into registers and
// takes the DMA of the step NB ahead before its MFMAs run, across k-steps,
// slices and epilogues, so the stream never drains inside a workgroup and no
// barrier or partial sum meets in the loop. About 80 KiB of LDS per workgroup:
// two per CU, 96 KiB in flight.
//
// expert_skinny_kernel before it (one workgroup per 32 columns, the k-steps
// split over its waves, loads in the MFMA layout) drained the stream once per
// workgroup; figures at the launcher.
//
// LDS rows are 128 bytes, physical 16-byte chunk c of row r holding logical
// chunk c ^ ((r >> 1) & 7), as in the dense DMA cores; the MFMA roles and the
// epilogue (E1, and S1 for GU) are expert_skinny_kernel's on the same integers.
#pragma once

#include "common.hpp"
#include "gemm_dma.hpp"
#include "kernels.hpp"

namespace clef {

namespace {

constexpr int kStreamWaves = 4, kStreamStage = 4096;

// Dynamic LDS: activation rows, rings, column scales (ONE: none).
template <bool GU, int NB, bool ONE>
constexpr int expert_stream_lds(int kb, int spw) {
  return kb * kStreamStage + kStreamWaves * NB * kStreamStage + (ONE ? 0 : (GU ? 2 : 1) * spw * 512);
}

// ONE: spw is 1 and the column scales are kept in registers (the activation
// rows of K 2048 and three stages per wave take exactly half of the CU's LDS).
template <bool GU, int NB, bool ONE>
__global__ __launch_bounds__(64 * kStreamWaves) void expert_stream_kernel(
    const uint32_t* __restrict__ a, int a_words, uint32_t a_bytes, const float* __restrict__ as,
    const uint32_t* __restrict__ w, const float* __restrict__ ws, const uint32_t* __restrict__ w2,
    const float* __restrict__ ws2, const float* __restrict__ groups, const int32_t* __restrict__ schedule,
    int64_t list_stride, int topk, int kb, int n, int input_routed, uint16_t* __restrict__ out, uint32_t out_bytes,
    int colgroups, int spw) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int NA = GU ? 2 : 1;
  constexpr int kDma = kStreamStage / 1024;  // DMA instructions per stage
  constexpr int kStores = 4;                 // output stores per slice
  static_assert((NB - 1) * kDma + kStores < 64, "vmcnt range");
  extern __shared__ __align__(16) char lds[];
  const int tile = (int)(blockIdx.x / colgroups);
  const int cbase = (int)(blockIdx.x - (int64_t)tile * colgroups) * (128 * spw);  // first column within the expert
  // the entry is read together with the tile count (every launched tile
  // indexes inside the schedule buffer)
  const int tiles = schedule[0];
  const int e = schedule[kSchedEntries + 2 * tile];
  const int row0 = schedule[kSchedEntries + 1 + 2 * tile];
  if (tile >= tiles || e < 0) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 31, h = lane >> 5;
  char* const arows = lds;
  char* const ring = lds + kb * kStreamStage + wave * (NB * kStreamStage);
  char* const wscale = lds + kb * kStreamStage + kStreamWaves * NB * kStreamStage;

  // Weight rows of slice i: 32 wave .. of 128-row block (e n + cbase) / 128 + i.
  const int64_t nrow = (int64_t)e * n + cbase;
  const uint32_t w_bytes = (uint32_t)(spw * kb) * 16384u;
  const __amdgpu_buffer_rsrc_t w_rsrc = make_rsrc(w + (nrow / 128) * kb * 4096, w_bytes);
  const __amdgpu_buffer_rsrc_t w2_rsrc = make_rsrc((GU ? w2 : w) + (nrow / 128) * kb * 4096, w_bytes);
  const int c_even = ((lane & 7) ^ (lane >> 4)) * 16, c_odd = ((lane & 7) ^ (4 | (lane >> 4))) * 16;
  const int w_voff = (32 * wave + (lane >> 3)) * 128;
  // step s of the wave: s = (slice * kb + k-step) * NA + (gate / up); steps
  // past the last load nothing (outside the resource: zeros never read)
  auto issue = [&](char* stage, int block, int which) {
#pragma unroll
    for (int q = 0; q < kDma; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(GU && which ? w2_rsrc : w_rsrc, (lds_ptr_t)(stage + q * 1024), 16,
                                               block < spw * kb ? w_voff + ((q & 1) ? c_odd : c_even)
                                                                : (int)0x80000000u,
                                               block * 16384 + q * 1024, 0, 0);
  };
#pragma unroll
  for (int b = 0; b < NB; ++b) issue(ring + b * kStreamStage, b / NA, b % NA);

  // The tile's slots: routes, row scales, activation rows. Slots past the
  // group's end read zeros.
  const float* list = groups + (int64_t)e * list_stride;
  const int64_t cap = list_stride - 1 - row0;
  const __amdgpu_buffer_rsrc_t l_rsrc =
      make_rsrc(list + 1 + row0, (uint32_t)((cap < 32 ? (cap > 0 ? cap : 0) : 32) * 4));
  const float route_f = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(l_rsrc, lr * 4, 0, 0));
  const int count = (int)list[0];
  const int route = row0 + lr < count ? (int)route_f : -1;
  const int xr = route < 0 ? -1 : input_routed ? route : route / topk;
  {
    const int row_x = __shfl(xr, 8 * wave + (lane >> 3));
    const __amdgpu_buffer_rsrc_t a_rsrc = make_rsrc(a, a_bytes);
    const int a_voff = row_x >= 0 ? row_x * a_words * 4 + ((wave & 1) ? c_odd : c_even) : (int)0x80000000u;
    for (int kt = 0; kt < kb; ++kt)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rsrc, (lds_ptr_t)(arows + kt * kStreamStage + wave * 1024), 16,
                                               a_voff, kt * 128, 0, 0);
  }
  // column scales: 128 spw floats (gate, then up)
  for (int i = wave; !ONE && i < 2 * NA * spw; i += kStreamWaves) {
    const bool up = GU && i >= 2 * spw;
    const __amdgpu_buffer_rsrc_t s_rsrc = make_rsrc((up ? ws2 : ws) + nrow, (uint32_t)(spw * 512));
    __builtin_amdgcn_raw_ptr_buffer_load_lds(s_rsrc, (lds_ptr_t)(wscale + i * 256), 4, lane * 4,
                                             (up ? i - 2 * spw : i) * 256, 0, 0);
  }
  float asv = route >= 0 ? as[xr] : 0.0f;
  float4 wsr[NA][4];
  if constexpr (ONE) {
#pragma unroll
    for (int rq = 0; rq < 4; ++rq) {
      const int col = 32 * wave + 8 * rq + 4 * h;
      wsr[0][rq] = *reinterpret_cast<const float4*>(ws + nrow + col);
      if constexpr (GU) wsr[NA - 1][rq] = *reinterpret_cast<const float4*>(ws2 + nrow + col);
    }
  }
  wait_vmcnt<0>();
  pin_vgpr(asv);
  __syncthreads();

  const __amdgpu_buffer_rsrc_t o_rsrc = make_rsrc(out, out_bytes);
  int pos = 0;         // ring stage of the current step
  int ahead = NB;      // the step to load next
  int off[4];
#pragma unroll
  for (int p = 0; p < 4; ++p) off[p] = lr * 128 + (((4 * h + p) ^ ((lr >> 1) & 7)) << 4);
  // the ring, the activation rows and the scales as distinct restrict pointers
  // of one body: the compiler then keeps the ring's DMA in flight across reads
  // of the others
  auto slices = [&](char* __restrict__ rg, const char* __restrict__ ar_lds, const char* __restrict__ sc) {
    for (int i = 0; i < (ONE ? 1 : spw); ++i) {
      v16i acc[NA];
#pragma unroll
      for (int s = 0; s < NA; ++s) acc[s] = v16i{};
      for (int kt = 0; kt < kb; ++kt) {
#pragma unroll
        for (int s = 0; s < NA; ++s) {
          // The step's DMA has landed once at most the NB - 1 steps behind it
          // are outstanding, and the last slice's stores where they were issued
          // after it (its first NB steps; vector memory completes in issue order).
          if (i > 0 && kt * NA + s < NB)
            wait_vmcnt<(NB - 1) * kDma + kStores>();
          else
            wait_vmcnt<(NB - 1) * kDma>();
          char* stage = rg + pos * kStreamStage;
          u4 wr[4], ar[4];
#pragma unroll
          for (int p = 0; p < 4; ++p) wr[p] = *reinterpret_cast<const u4*>(stage + off[p]);
#pragma unroll
          for (int p = 0; p < 4; ++p) ar[p] = *reinterpret_cast<const u4*>(ar_lds + kt * kStreamStage + off[p]);
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the DMA overwrites it
          issue(stage, ahead / NA, ahead % NA);
          ++ahead;
          pos = pos + 1 == NB ? 0 : pos + 1;
#pragma unroll
          for (int p = 0; p < 4; ++p) {
            acc[s] = mfma32_i8(unpack_pair(wr[p][0], wr[p][1]), unpack_pair(ar[p][0], ar[p][1]), acc[s]);
            acc[s] = mfma32_i8(unpack_pair(wr[p][2], wr[p][3]), unpack_pair(ar[p][2], ar[p][3]), acc[s]);
          }
        }
      }
      // lane: slot lr, columns c0 + 8 rq + 4 h + 0..3
      const int c0 = (4 * i + wave) * 32;
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        const int col = c0 + 8 * rq + 4 * h;
        const float4 wg4 = ONE ? wsr[0][rq] : *reinterpret_cast<const float4*>(sc + col * 4);
        const float wg[4] = {wg4.x, wg4.y, wg4.z, wg4.w};
        float y[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) y[t] = (float)(acc[0][4 * rq + t] >> 8) * (asv * wg[t]);
        if constexpr (GU) {
          const float4 wu4 = ONE ? wsr[NA - 1][rq] : *reinterpret_cast<const float4*>(sc + spw * 512 + col * 4);
          const float wu[4] = {wu4.x, wu4.y, wu4.z, wu4.w};
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const float g = as_float(pack_bf16x2(0.0f, y[t]));  // bf16(gate)
            const float u = (float)(acc[NA - 1][4 * rq + t] >> 8) * (asv * wu[t]);
            y[t] = silu_bf16(g) * bf16_round(u);
          }
        }
        // slots past the group's end store outside the resource: every wave
        // issues kStores stores per slice
        const int o_voff = route >= 0 ? (route * n + cbase + col) * 2 : (int)0x80000000u;
        __builtin_amdgcn_raw_buffer_store_b64(
            v2i{(int)pack_bf16x2(y[0], y[1]), (int)pack_bf16x2(y[2], y[3])}, o_rsrc, o_voff, 0, 0);
      }
    }
  };
  slices(ring, arows, wscale);
  wait_vmcnt<0>();  // no DMA into this workgroup's LDS is left
#endif
}

}  // namespace

}  // namespace clef
