// C ABI of the gfx950 INT4 path (include/clef_i4.h): argument checks with the
// reference's predicates and messages, then stream-ordered launches. The
// composite entry points (pack_weight, project, moe_layer) are the host side
// of the reference's operators: Engine::load_quantized_weight
// (src/quantized.rs:147-234), Engine::project_quantized (:235-303) and the
// MoE block of omni::forward_layers_cached (src/omni.rs:760-857).
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>
#include <mutex>

#include "../../include/clef_i4.h"
#include "build_id.inc"  // CLEF_BUILD_ID, generated by the Makefile
#include "kernels.hpp"

namespace {

thread_local char g_error[1024] = "";

int fail(const char* msg) {
  std::snprintf(g_error, sizeof g_error, "%s", msg);
  return CLEF_EINVAL;
}

int hip_status(hipError_t e) {
  if (e == hipSuccess) return CLEF_OK;
  std::snprintf(g_error, sizeof g_error, "HIP error %d: %s", (int)e, hipGetErrorString(e));
  return (int)e;
}

bool aligned(const void* p, size_t a) { return p && (reinterpret_cast<uintptr_t>(p) % a) == 0; }

bool overlap(const void* a, size_t a_bytes, const void* b, size_t b_bytes) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(a), y = reinterpret_cast<uintptr_t>(b);
  return x < y + b_bytes && y < x + a_bytes;
}

hipStream_t hs(clef_stream_t s) { return reinterpret_cast<hipStream_t>(s); }

constexpr const char* kAlign = "device pointer is NULL or not 16-byte aligned";
constexpr const char* kWorkspace = "workspace too small";

size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

// Route ordinals t * topk + r travel as f32 (the reference's table layout),
// exact only below 2^24.
bool routes_in_range(int64_t tokens, int32_t topk) {
  return tokens >= 1 && topk >= 1 && tokens <= 1048576 && topk <= 128 && tokens * topk <= 16777216;
}

// The grouped expert kernels address gathered activation rows with 32-bit
// buffer offsets: the packed codes of the operand must stay below 2 GiB.
constexpr const char* kOperand =
    "expert activation operand of 2 GiB or more (split the tokens into chunks, as the reference does)";
bool operand_below_2gib(int64_t rows, int32_t stride) {
  return rows * (int64_t)(stride / 8) * 4 < ((int64_t)1 << 31);
}

// Quantizer preconditions, src/quantized.rs:640-649.
int check_prepare(int64_t rows, int32_t width, int32_t stride, int32_t bits) {
  if (!((bits == 4 || bits == 8) && width >= 256 && width <= 32768 && width % 256 == 0 && rows >= 1 &&
        rows <= 1048576 && stride >= width && stride <= 65536 && stride % (512 / bits) == 0))
    return fail("unsupported rotated integer operand");
  return CLEF_OK;
}

int check_norm(int64_t rows, int32_t width, int32_t stride, int32_t bits) {
  if (!(width == 5120 && (bits == 4 || bits == 8) && rows >= 1 && rows <= 1048576 && stride >= width &&
        stride <= 65536 && stride % (512 / bits) == 0))
    return fail("unsupported normalized packing shape");
  return CLEF_OK;
}

int check_gemm(int64_t m, int32_t n, int32_t k, int32_t k_stride) {
  if (!(m >= 1 && n >= 128 && n % 128 == 0 && k >= 256 && k % 256 == 0 && k_stride >= k &&
        k_stride % 32 == 0))
    return fail("unsupported integer projection shape");
  return CLEF_OK;
}

int64_t prepared_words(int64_t rows, int32_t stride, int32_t bits) {
  return rows * (stride / (32 / bits) + 1);
}

int32_t stride_for(int32_t width, int32_t bits) {
  return width + (width % 1024 == 0 ? 512 / bits : 0);
}

}  // namespace

namespace clef {
int set_last_error(const char* msg) { return fail(msg); }
}  // namespace clef

extern "C" {

const char* clef_last_error(void) { return g_error; }

int clef_abi_version(void) { return 100; }

// Kept as one string in the library's read-only data so that the identity can
// also be read from the file without loading it.
static const char kBuildTag[] __attribute__((used)) = "clef-build-id:" CLEF_BUILD_ID;

const char* clef_build_id(void) { return kBuildTag + sizeof("clef-build-id:") - 1; }

int32_t clef_i4_activation_stride(int32_t width, int32_t bits) { return stride_for(width, bits); }

int64_t clef_i4_prepared_words(int64_t rows, int32_t stride, int32_t bits) {
  if (bits != 4 && bits != 8) return -1;
  return prepared_words(rows, stride, bits);
}

int clef_i4_prepare(const uint16_t* x, int64_t rows, int32_t width, int32_t stride, int32_t bits,
                    uint32_t* out, clef_stream_t stream) {
  if (int rc = check_prepare(rows, width, stride, bits)) return rc;
  if (!aligned(x, 16) || !aligned(out, 16)) return fail(kAlign);
  return hip_status(clef::launch_prepare(x, rows, width, stride, bits, out, hs(stream)));
}

int clef_i4_prepare_swiglu(const uint16_t* gate, const uint16_t* up, int64_t rows, int32_t width,
                           int32_t stride, int32_t bits, uint32_t* out, clef_stream_t stream) {
  if (int rc = check_prepare(rows, width, stride, bits)) return rc;
  if (!aligned(gate, 16) || !aligned(up, 16) || !aligned(out, 16)) return fail(kAlign);
  return hip_status(clef::launch_prepare_swiglu(gate, up, rows, width, stride, bits, out, hs(stream)));
}

int clef_i4_prepare_attention_gate(const uint16_t* attention, const uint16_t* q_gate, int64_t rows,
                                   int32_t width, int32_t stride, int32_t bits, uint32_t* out,
                                   clef_stream_t stream) {
  if (int rc = check_prepare(rows, width, stride, bits)) return rc;
  if (!aligned(attention, 16) || !aligned(q_gate, 16) || !aligned(out, 16)) return fail(kAlign);
  return hip_status(
      clef::launch_prepare_attention_gate(attention, q_gate, rows, width, stride, bits, out, hs(stream)));
}

namespace {
// Byte offset of the stored normalized rows: the packed words rounded up to
// 128 bytes (src/quantized.rs:733-734).
int64_t norm_offset_bytes(int64_t rows, int32_t stride, int32_t bits) {
  return (prepared_words(rows, stride, bits) * 4 + 127) / 128 * 128;
}
}  // namespace

int64_t clef_i4_prepare_norm_words(int64_t rows, int32_t width, int32_t stride, int32_t bits,
                                   int32_t store) {
  if ((bits != 4 && bits != 8) || rows < 0 || width < 0) return -1;
  if (!store) return prepared_words(rows, stride, bits);
  return norm_offset_bytes(rows, stride, bits) / 4 + rows * width / 2;
}

int clef_i4_prepare_norm(const uint16_t* x, const uint16_t* weight, int64_t rows, int32_t width,
                         int32_t stride, int32_t bits, int32_t store, uint32_t* out,
                         clef_stream_t stream) {
  if (int rc = check_norm(rows, width, stride, bits)) return rc;
  if (!aligned(x, 16) || !aligned(weight, 16) || !aligned(out, 16)) return fail(kAlign);
  uint16_t* normalized =
      store ? reinterpret_cast<uint16_t*>(reinterpret_cast<char*>(out) + norm_offset_bytes(rows, stride, bits))
            : nullptr;
  return hip_status(
      clef::launch_prepare_norm(x, weight, rows, width, stride, bits, out, normalized, hs(stream)));
}

int clef_i4_prepare_filled(const uint16_t* x, const uint16_t* second, int32_t producer, int64_t rows, int32_t width,
                           int32_t stride, int32_t bits, uint32_t* out, clef_stream_t stream) {
  if (producer == CLEF_PRODUCER_NORM) {
    if (int rc = check_norm(rows, width, stride, bits)) return rc;
  } else if (producer == CLEF_PRODUCER_PLAIN || producer == CLEF_PRODUCER_SWIGLU ||
             producer == CLEF_PRODUCER_ATTENTION_GATE) {
    if (int rc = check_prepare(rows, width, stride, bits)) return rc;
  } else {
    return fail("unknown packing producer");
  }
  if (!aligned(x, 16) || (producer != CLEF_PRODUCER_PLAIN && !aligned(second, 16)) || !aligned(out, 16))
    return fail(kAlign);
  hipError_t e;
  switch (producer) {
    case CLEF_PRODUCER_SWIGLU:
      e = clef::launch_prepare_swiglu(x, second, rows, width, stride, bits, out, hs(stream), true);
      break;
    case CLEF_PRODUCER_ATTENTION_GATE:
      e = clef::launch_prepare_attention_gate(x, second, rows, width, stride, bits, out, hs(stream), true);
      break;
    case CLEF_PRODUCER_NORM:
      e = clef::launch_prepare_norm(x, second, rows, width, stride, bits, out, nullptr, hs(stream), true);
      break;
    default:
      e = clef::launch_prepare(x, rows, width, stride, bits, out, hs(stream), true);
  }
  return hip_status(e);
}

int clef_i4_retile(const uint32_t* codes, int64_t rows, int32_t in_words, int32_t cols, int32_t bits,
                   uint32_t* tiled, clef_stream_t stream) {
  if (bits != 4 && bits != 8) return fail("unsupported packed weight shape for tiling");
  const int32_t words = cols / (32 / bits);
  // src/quantized.rs:550-558.
  if (!(rows > 0 && rows % 128 == 0 && cols > 0 && cols % (32 / bits) == 0 && words % 32 == 0 &&
        in_words >= words))
    return fail("unsupported packed weight shape for tiling");
  if (!aligned(codes, 16) || !aligned(tiled, 16)) return fail(kAlign);
  return hip_status(clef::launch_retile(codes, rows, in_words, words, tiled, hs(stream)));
}

size_t clef_i4_pack_weight_workspace_bytes(int64_t rows, int32_t cols, int32_t bits) {
  if ((bits != 4 && bits != 8) || rows < 0 || cols < 0) return 0;
  return align256((size_t)prepared_words(rows, stride_for(cols, bits), bits) * 4);
}

int clef_i4_pack_weight(const uint16_t* w, int64_t rows, int32_t cols, int32_t bits, uint32_t* tiled,
                        float* scales, void* workspace, size_t workspace_bytes,
                        clef_stream_t stream) {
  if (!(rows > 0 && cols > 0 && rows % 256 == 0 && cols % 256 == 0))
    return fail("unsupported quantized weight shape");
  const int32_t stride = stride_for(cols, bits);
  if (int rc = check_prepare(rows, cols, stride, bits)) return rc;
  if (!aligned(w, 16) || !aligned(tiled, 16) || !aligned(scales, 4) || !aligned(workspace, 16))
    return fail(kAlign);
  if (workspace_bytes < clef_i4_pack_weight_workspace_bytes(rows, cols, bits)) return fail(kWorkspace);
  const size_t in_bytes = (size_t)rows * cols * 2, out_bytes = (size_t)rows * cols * bits / 8;
  if (!overlap(w, in_bytes, tiled, out_bytes) && !overlap(w, in_bytes, scales, (size_t)rows * 4))
    return hip_status(clef::launch_pack_weight(w, rows, cols, bits, false, tiled, scales, hs(stream)));
  // packing over the weight itself: through the row-major codes in the workspace
  uint32_t* staging = static_cast<uint32_t*>(workspace);
  const int32_t words = stride / (32 / bits);
  if (int rc = hip_status(clef::launch_prepare(w, rows, cols, stride, bits, staging, hs(stream))))
    return rc;
  if (int rc = hip_status(clef::launch_retile(staging, rows, words, cols / (32 / bits), tiled, hs(stream))))
    return rc;
  return hip_status(hipMemcpyAsync(scales, staging + rows * words, (size_t)rows * 4,
                                   hipMemcpyDeviceToDevice, hs(stream)));
}

int clef_i4_pack_checkpoint(const uint16_t* w, int64_t rows, int32_t cols, int32_t bits,
                            int32_t checkpoint_tiled, uint32_t* tiled, float* scales, clef_stream_t stream) {
  if (checkpoint_tiled && !(rows > 0 && cols > 0 && rows % 256 == 0 && cols % 64 == 0))
    return fail("tiled layout requires 256-row and 64-column multiples");
  if (checkpoint_tiled && !aligned(w, 16)) return fail(kAlign);
  if (!(rows > 0 && cols > 0 && rows % 256 == 0 && cols % 256 == 0))
    return fail("unsupported quantized weight shape");
  if (int rc = check_prepare(rows, cols, stride_for(cols, bits), bits)) return rc;
  if (!aligned(w, 16) || !aligned(tiled, 16) || !aligned(scales, 4)) return fail(kAlign);
  return hip_status(
      clef::launch_pack_weight(w, rows, cols, bits, checkpoint_tiled != 0, tiled, scales, hs(stream)));
}

int clef_untile_rows(const uint16_t* tiled, int64_t rows, int32_t cols, uint16_t* out,
                     clef_stream_t stream) {
  if (!(rows > 0 && cols > 0 && rows % 256 == 0 && cols % 64 == 0))
    return fail("tiled layout requires 256-row and 64-column multiples");
  if (!aligned(tiled, 16) || !aligned(out, 16)) return fail(kAlign);
  return hip_status(clef::launch_tile_permute(tiled, rows, cols, out, false, hs(stream)));
}

int clef_tile_rows(const uint16_t* dense, int64_t rows, int32_t cols, uint16_t* out,
                   clef_stream_t stream) {
  if (!(rows > 0 && cols > 0 && rows % 256 == 0 && cols % 64 == 0))
    return fail("tiled layout requires 256-row and 64-column multiples");
  if (!aligned(dense, 16) || !aligned(out, 16)) return fail(kAlign);
  return hip_status(clef::launch_tile_permute(dense, rows, cols, out, true, hs(stream)));
}

int clef_i4_gemm_configs(void) { return clef::gemm_config_count(); }

int clef_i4_gemm_config(const uint32_t* a, int32_t k_stride, const float* a_scales,
                        const uint32_t* w_tiled, const float* w_scales, int64_t m, int32_t n,
                        int32_t k, const uint16_t* residual, uint16_t* out, int32_t config,
                        clef_stream_t stream) {
  if (int rc = check_gemm(m, n, k, k_stride)) return rc;
  if (config < -1 || config >= clef::gemm_config_count()) return fail("unknown GEMM tile configuration");
  if (!aligned(a, 16) || !aligned(a_scales, 4) || !aligned(w_tiled, 16) || !aligned(w_scales, 16) ||
      !aligned(out, 16) || (residual && !aligned(residual, 16)))
    return fail(kAlign);
  return hip_status(clef::launch_gemm_i4(a, k_stride / 8, a_scales, w_tiled, w_scales, m, n, k,
                                         residual, out, config, hs(stream)));
}

int clef_i4_gemm(const uint32_t* a, int32_t k_stride, const float* a_scales, const uint32_t* w_tiled,
                 const float* w_scales, int64_t m, int32_t n, int32_t k, const uint16_t* residual,
                 uint16_t* out, clef_stream_t stream) {
  return clef_i4_gemm_config(a, k_stride, a_scales, w_tiled, w_scales, m, n, k, residual, out, -1,
                             stream);
}

size_t clef_i4_gemm_workspace_bytes(int64_t m, int32_t n, int32_t k) {
  if (check_gemm(m, n, k, k) != CLEF_OK || !clef::gemm_i4_via_f6(m, n, k)) return 0;
  return align256((size_t)clef::f6_codes_bytes(m, k)) + (size_t)n * k * 3 / 4;
}

int clef_i4_gemm_ws(const uint32_t* a, int32_t k_stride, const float* a_scales, const uint32_t* w_tiled,
                    const float* w_scales, int64_t m, int32_t n, int32_t k, const uint16_t* residual, uint16_t* out,
                    void* workspace, size_t workspace_bytes, clef_stream_t stream) {
  if (int rc = check_gemm(m, n, k, k_stride)) return rc;
  const size_t need = clef_i4_gemm_workspace_bytes(m, n, k);
  if (need == 0 || workspace == nullptr || workspace_bytes < need)
    return clef_i4_gemm(a, k_stride, a_scales, w_tiled, w_scales, m, n, k, residual, out, stream);
  if (!aligned(a, 16) || !aligned(a_scales, 4) || !aligned(w_tiled, 16) || !aligned(w_scales, 16) ||
      !aligned(out, 16) || (residual && !aligned(residual, 16)) || !aligned(workspace, 16))
    return fail(kAlign);
  uint8_t* a6 = static_cast<uint8_t*>(workspace);
  uint8_t* w6 = a6 + align256((size_t)clef::f6_codes_bytes(m, k));
  if (int rc = hip_status(clef::launch_f6_convert(w_tiled, n, w6, a, k_stride / 8, m, a6, k, hs(stream)))) return rc;
  return hip_status(clef::launch_gemm_f6(a6, a_scales, w6, w_scales, m, n, k, residual, out, hs(stream)));
}

int clef_i8_gemm(const uint32_t* a, int32_t k_stride, const float* a_scales, const uint32_t* w_tiled,
                 const float* w_scales, int64_t m, int32_t n, int32_t k, const uint16_t* residual,
                 uint16_t* out, clef_stream_t stream) {
  if (int rc = check_gemm(m, n, k, k_stride)) return rc;
  if (k_stride % 64 != 0) return fail("unsupported integer projection shape");
  if (!aligned(a, 16) || !aligned(w_tiled, 16) || !aligned(w_scales, 16) || !aligned(out, 16) ||
      (residual && !aligned(residual, 16)))
    return fail(kAlign);
  return hip_status(
      clef::launch_gemm_i8(a, k_stride / 4, a_scales, w_tiled, w_scales, m, n, k, residual, out, hs(stream)));
}

int clef_i4_f6_activation(const uint32_t* a, int32_t k_stride, int64_t rows, int32_t k, uint8_t* out,
                          clef_stream_t stream) {
  if (rows < 1 || k < 128 || k % 128 != 0 || k_stride < k || k_stride % 32 != 0 || rows > ((int64_t)1 << 40))
    return fail("unsupported integer projection shape");
  if (!aligned(a, 16) || !aligned(out, 16)) return fail(kAlign);
  return hip_status(clef::launch_f6_rows(a, k_stride / 8, rows, k, out, hs(stream)));
}

int clef_i4_f6_weight(const uint32_t* w_tiled, int64_t n, int32_t k, uint8_t* out, clef_stream_t stream) {
  if (n < 128 || n % 128 != 0 || k < 256 || k % 256 != 0 || n > ((int64_t)1 << 31))
    return fail("unsupported integer projection shape");
  if (!aligned(w_tiled, 16) || !aligned(out, 16)) return fail(kAlign);
  return hip_status(clef::launch_f6_tiled(w_tiled, n, k, out, hs(stream)));
}

int64_t clef_i4_f6_prepared_bytes(int64_t rows, int32_t width) {
  if (rows < 0 || width < 0) return -1;
  return clef::f6_codes_bytes(rows, width) + rows * 4;
}

int clef_i4_prepare_f6(const uint16_t* x, int64_t rows, int32_t width, uint8_t* out, clef_stream_t stream) {
  if (int rc = check_prepare(rows, width, width, 4)) return rc;
  if (!aligned(x, 16) || !aligned(out, 16)) return fail(kAlign);
  return hip_status(clef::launch_prepare(x, rows, width, width, 6, reinterpret_cast<uint32_t*>(out), hs(stream)));
}

int clef_i4_prepare_swiglu_f6(const uint16_t* gate, const uint16_t* up, int64_t rows, int32_t width,
                              uint8_t* out, clef_stream_t stream) {
  if (int rc = check_prepare(rows, width, width, 4)) return rc;
  if (!aligned(gate, 16) || !aligned(up, 16) || !aligned(out, 16)) return fail(kAlign);
  return hip_status(clef::launch_prepare_swiglu(gate, up, rows, width, width, 6, reinterpret_cast<uint32_t*>(out),
                                                hs(stream)));
}

int clef_i4_gemm_f6(const uint8_t* a_f6, const float* a_scales, const uint8_t* w_f6, const float* w_scales,
                    int64_t m, int32_t n, int32_t k, const uint16_t* residual, uint16_t* out,
                    clef_stream_t stream) {
  // The kernel's buffer resources take 32-bit byte extents: a 256-row block of
  // activation rows and of outputs, the row scales, a 256-column weight panel.
  // k is at most 32768, the quantizer's widest row: every f32 partial sum of
  // the bf6 products is then an integer below 2^22, so the sums are exact and
  // the result equals clef_i4_gemm's (exactness alone would allow k < 2^18).
  if (m < 1 || n < 256 || n % 256 != 0 || k < 256 || k % 256 != 0 || k > 32768 || m > ((int64_t)1 << 29) ||
      (int64_t)k * 3 / 4 * 256 >= ((int64_t)1 << 31) || (int64_t)n * 2 * 256 >= ((int64_t)1 << 31) ||
      (int64_t)k / 128 * 12288 * 2 >= ((int64_t)1 << 31))
    return fail("unsupported integer projection shape");
  if (!aligned(a_f6, 16) || !aligned(w_f6, 16) || !aligned(w_scales, 16) || !aligned(out, 16) ||
      (residual && !aligned(residual, 16)))
    return fail(kAlign);
  return hip_status(clef::launch_gemm_f6(a_f6, a_scales, w_f6, w_scales, m, n, k, residual, out, hs(stream)));
}

int clef_i4_gemm_f6_gate_up(const uint8_t* a_f6, const float* a_scales, const uint8_t* gate_f6,
                            const float* gate_scales, const uint8_t* up_f6, const float* up_scales, int64_t m,
                            int32_t n, int32_t k, uint16_t* h, clef_stream_t stream) {
  // clef_i4_gemm_f6's limits with 128-column panels (n % 128 == 0)
  if (m < 1 || n < 128 || n % 128 != 0 || k < 256 || k % 256 != 0 || k > 32768 || m > ((int64_t)1 << 29) ||
      (int64_t)k * 3 / 4 * 256 >= ((int64_t)1 << 31) || (int64_t)n * 2 * 256 >= ((int64_t)1 << 31) ||
      (int64_t)k / 128 * 12288 >= ((int64_t)1 << 31))
    return fail("unsupported integer projection shape");
  if (!aligned(a_f6, 16) || !aligned(gate_f6, 16) || !aligned(gate_scales, 16) || !aligned(up_f6, 16) ||
      !aligned(up_scales, 16) || !aligned(h, 16))
    return fail(kAlign);
  return hip_status(clef::launch_gemm_f6_gate_up(a_f6, a_scales, gate_f6, gate_scales, up_f6, up_scales, m, n, k, h,
                                                 hs(stream)));
}

size_t clef_i4_project_f6_workspace_bytes(int64_t m, int32_t k) {
  if (m < 0 || k < 0) return 0;
  return align256((size_t)clef_i4_f6_prepared_bytes(m, k));
}

int clef_i4_project_f6(const uint16_t* x, int64_t m, int32_t k, const uint8_t* w_f6, const float* w_scales,
                       int32_t n, const uint16_t* residual, uint16_t* out, void* workspace,
                       size_t workspace_bytes, clef_stream_t stream) {
  if (!workspace || workspace_bytes < clef_i4_project_f6_workspace_bytes(m, k)) return fail(kWorkspace);
  uint8_t* a = static_cast<uint8_t*>(workspace);
  if (int rc = clef_i4_prepare_f6(x, m, k, a, stream)) return rc;
  const float* a_scales = reinterpret_cast<const float*>(a + clef::f6_codes_bytes(m, k));
  return clef_i4_gemm_f6(a, a_scales, w_f6, w_scales, m, n, k, residual, out, stream);
}

size_t clef_i4_project_workspace_bytes(int64_t m, int32_t k) {
  if (m < 0 || k < 0) return 0;
  return align256((size_t)prepared_words(m, stride_for(k, 4), 4) * 4);
}

int clef_i4_project(const uint16_t* x, int64_t m, int32_t k, const uint32_t* w_tiled,
                    const float* w_scales, int32_t n, const uint16_t* residual, uint16_t* out,
                    void* workspace, size_t workspace_bytes, clef_stream_t stream) {
  const int32_t stride = stride_for(k, 4);
  if (int rc = check_prepare(m, k, stride, 4)) return rc;
  if (int rc = check_gemm(m, n, k, stride)) return rc;
  if (!aligned(x, 16) || !aligned(workspace, 16) || !aligned(w_tiled, 16) || !aligned(w_scales, 16) ||
      !aligned(out, 16) || (residual && !aligned(residual, 16)))
    return fail(kAlign);
  if (workspace_bytes < clef_i4_project_workspace_bytes(m, k)) return fail(kWorkspace);
  // a few rows in one launch, unless the output overlaps the input that every
  // workgroup of that launch reads
  if (clef::project_fusable(m, n, k) && !overlap(x, (size_t)m * k * 2, out, (size_t)m * n * 2))
    return hip_status(clef::launch_project_i4(x, w_tiled, w_scales, m, n, k, residual, out, hs(stream)));
  uint32_t* packed = static_cast<uint32_t*>(workspace);
  if (int rc = hip_status(clef::launch_prepare(x, m, k, stride, 4, packed, hs(stream)))) return rc;
  const float* a_scales = reinterpret_cast<const float*>(packed + m * (stride / 8));
  const size_t used = clef_i4_project_workspace_bytes(m, k);
  return clef_i4_gemm_ws(packed, stride, a_scales, w_tiled, w_scales, m, n, k, residual, out,
                         static_cast<char*>(workspace) + used, workspace_bytes - used, stream);
}

int clef_moe_route(const void* logits, int32_t logits_dtype, int64_t tokens, int32_t experts,
                   int32_t topk, float* routes, clef_stream_t stream) {
  // src/omni.rs:171-174.
  if (!(topk > 0 && topk <= experts && experts <= 128)) return fail("invalid expert router shape");
  if (logits_dtype != 0 && logits_dtype != 1) return fail("invalid router logits dtype");
  if (tokens < 1 || tokens > 16777216) return fail("invalid expert router shape");
  // The router reads a token's logits as 16-byte pieces when the row length
  // allows it, so the logits start on a 16-byte boundary.
  if (!aligned(logits, 16) || !aligned(routes, 4)) return fail(kAlign);
  return hip_status(clef::launch_route(logits, logits_dtype, tokens, experts, topk, routes, hs(stream)));
}

int clef_moe_router_logits(const uint16_t* x, const uint16_t* gate_w, int64_t tokens, int32_t hidden,
                           int32_t experts, uint16_t* logits, clef_stream_t stream) {
  if (!(tokens >= 1 && hidden >= 64 && hidden % 64 == 0 && experts >= 32 && experts <= 128 && experts % 32 == 0))
    return fail("linear shape/dtype mismatch");
  if (!aligned(x, 16) || !aligned(gate_w, 16) || !aligned(logits, 2)) return fail(kAlign);
  return hip_status(clef::launch_router_gate(x, gate_w, tokens, hidden, experts, logits, hs(stream)));
}

size_t clef_moe_group_workspace_bytes(int64_t tokens) {
  if (tokens < 1) return 0;
  return align256(clef::group_workspace_bytes(tokens));
}

int clef_moe_group_routes(const float* routes, int64_t tokens, int32_t topk, float* groups,
                          float* order, void* workspace, size_t workspace_bytes,
                          clef_stream_t stream) {
  // src/omni.rs:194-197, with the chunk cap raised.
  if (!routes_in_range(tokens, topk)) return fail("unsupported Omni route grouping shape");
  if (!aligned(routes, 4) || !aligned(groups, 4) || (order && !aligned(order, 4)) ||
      !aligned(workspace, 16))
    return fail(kAlign);
  if (workspace_bytes < clef_moe_group_workspace_bytes(tokens)) return fail(kWorkspace);
  return hip_status(clef::launch_group_routes(routes, tokens, topk, groups, order, workspace, hs(stream)));
}

int clef_moe_expert_tasks(const float* groups, int64_t tokens, float* tasks, clef_stream_t stream) {
  if (!(tokens >= 1 && tokens <= 1048576)) return fail("unsupported compact Omni routes");
  if (!aligned(groups, 4) || !aligned(tasks, 4)) return fail(kAlign);
  return hip_status(clef::launch_expert_tasks(groups, tokens, tasks, hs(stream)));
}

size_t clef_moe_expert_workspace_bytes(int64_t tokens, int32_t topk) {
  if (tokens < 1 || topk < 1) return 0;
  return align256(clef::expert_schedule_bound(tokens * topk));
}

int clef_moe_expert_i4(const uint32_t* a, int32_t stride, const float* a_scales,
                       const uint32_t* w_tiled, const float* w_scales, const float* groups,
                       int64_t tokens, int32_t topk, int32_t k, int32_t n, int32_t input_routed,
                       uint16_t* out, void* workspace, size_t workspace_bytes,
                       clef_stream_t stream) {
  if (!(tokens >= 1 && tokens <= 1048576 && topk >= 1 && topk <= 128))
    return fail("invalid grouped expert routes");
  if (!routes_in_range(tokens, topk)) return fail("unsupported Omni route grouping shape");
  // src/omni.rs:461-466.
  if (!(k % 256 == 0 && n % 256 == 0 && k >= 256 && n >= 256 && stride >= k && stride % 32 == 0))
    return fail("unsupported Omni expert tile shape");
  if (!operand_below_2gib(input_routed ? tokens * topk : tokens, stride)) return fail(kOperand);
  if (!aligned(a, 16) || !aligned(a_scales, 4) || !aligned(w_tiled, 16) || !aligned(w_scales, 16) ||
      !aligned(groups, 4) || !aligned(out, 16) || !aligned(workspace, 16))
    return fail(kAlign);
  const int bm = clef::expert_tile_rows(tokens * topk, k, workspace_bytes);
  if (workspace_bytes < align256(clef::expert_schedule_bytes(tokens * topk, bm))) return fail(kWorkspace);
  int32_t* schedule = static_cast<int32_t*>(workspace);
  if (int rc = hip_status(clef::launch_expert_schedule(groups, tokens, bm, schedule, hs(stream)))) return rc;
  return hip_status(clef::launch_expert_i4(a, stride / 8, a_scales, w_tiled, w_scales, groups, schedule, bm,
                                           tokens, topk, k, n, input_routed ? 1 : 0, out, hs(stream)));
}

namespace {
// Workspace of the ungrouped expert GEMM: the route slots as one-slot tokens,
// their per-expert lists [128][routes + 1], the grouping scratch and the tile
// schedule.
struct UngroupedLayout {
  size_t slots, groups, group_ws, schedule;  // the schedule lies last
};
UngroupedLayout ungrouped_layout(int64_t tokens, int32_t topk) {
  const int64_t routes = tokens * topk;
  UngroupedLayout l{};
  size_t at = 0;
  auto take = [&](size_t bytes) {
    size_t here = at;
    at += align256(bytes);
    return here;
  };
  l.slots = take((size_t)routes * 2 * 4);
  l.groups = take((size_t)128 * (routes + 1) * 4);
  l.group_ws = take(clef::group_workspace_bytes(routes));
  l.schedule = at;
  return l;
}
}  // namespace

size_t clef_moe_expert_ungrouped_workspace_bytes(int64_t tokens, int32_t topk) {
  if (!routes_in_range(tokens, topk)) return 0;
  return ungrouped_layout(tokens, topk).schedule + align256(clef::expert_schedule_bound(tokens * topk));
}

int clef_moe_expert_i4_ungrouped(const uint32_t* a, int32_t stride, const float* a_scales,
                                 const uint32_t* w_tiled, const float* w_scales, const float* routes,
                                 int64_t tokens, int32_t topk, int32_t k, int32_t n, int32_t input_routed,
                                 uint16_t* out, void* workspace, size_t workspace_bytes, clef_stream_t stream) {
  if (!(tokens >= 1 && tokens <= 1048576 && topk >= 1 && topk <= 128))
    return fail("invalid grouped expert routes");
  if (!routes_in_range(tokens, topk)) return fail("unsupported Omni route grouping shape");
  if (!(k % 256 == 0 && n % 256 == 0 && k >= 256 && n >= 256 && stride >= k && stride % 32 == 0))
    return fail("unsupported Omni expert tile shape");
  if (!operand_below_2gib(input_routed ? tokens * topk : tokens, stride)) return fail(kOperand);
  if (!aligned(a, 16) || !aligned(a_scales, 4) || !aligned(w_tiled, 16) || !aligned(w_scales, 16) ||
      !aligned(routes, 4) || !aligned(out, 16) || !aligned(workspace, 256))
    return fail(kAlign);
  const UngroupedLayout l = ungrouped_layout(tokens, topk);
  if (workspace_bytes < l.schedule) return fail(kWorkspace);
  const int bm = clef::expert_tile_rows(tokens * topk, k, workspace_bytes - l.schedule);
  if (workspace_bytes - l.schedule < align256(clef::expert_schedule_bytes(tokens * topk, bm))) return fail(kWorkspace);
  char* ws = static_cast<char*>(workspace);
  float* slots = reinterpret_cast<float*>(ws + l.slots);
  float* groups = reinterpret_cast<float*>(ws + l.groups);
  int32_t* schedule = reinterpret_cast<int32_t*>(ws + l.schedule);
  const int64_t routed = tokens * topk;
  hipStream_t s = hs(stream);
  // Each route slot is grouped as a token of its own (topk 1), so every slot
  // naming an expert is listed, duplicates included, under its ordinal
  // t * topk + r; E1 then reads the lists with that row pitch.
  if (int rc = hip_status(clef::launch_route_slots(routes, tokens, topk, slots, s))) return rc;
  if (int rc = hip_status(clef::launch_group_routes(slots, routed, 1, groups, nullptr, ws + l.group_ws, s, schedule,
                                                    bm)))
    return rc;
  return hip_status(clef::launch_expert_i4(a, stride / 8, a_scales, w_tiled, w_scales, groups, schedule, bm, tokens,
                                           topk, k, n, input_routed ? 1 : 0, out, s, routed + 1));
}

int clef_moe_expert_gate_up_i4(const uint32_t* a, int32_t stride, const float* a_scales, const uint32_t* gate_w,
                               const float* gate_s, const uint32_t* up_w, const float* up_s,
                               const float* groups, int64_t tokens, int32_t topk, int32_t k, int32_t n,
                               uint16_t* h, void* workspace, size_t workspace_bytes, clef_stream_t stream) {
  // src/omni.rs:309-320, 333-344.
  if (!(tokens >= 1 && tokens <= 1048576 && topk >= 1 && topk <= 128))
    return fail("fused gate/up requires regular grouped routes");
  if (!routes_in_range(tokens, topk)) return fail("unsupported Omni route grouping shape");
  if (!(k % 256 == 0 && k >= 256 && n % 128 == 0 && n >= 128 && stride >= k && stride % 32 == 0))
    return fail("incompatible fused expert weights");
  if (!operand_below_2gib(tokens, stride)) return fail(kOperand);
  if (!aligned(a, 16) || !aligned(a_scales, 4) || !aligned(gate_w, 16) || !aligned(gate_s, 16) ||
      !aligned(up_w, 16) || !aligned(up_s, 16) || !aligned(groups, 4) || !aligned(h, 16) ||
      !aligned(workspace, 16))
    return fail(kAlign);
  const int bm = clef::expert_tile_rows(tokens * topk, k, workspace_bytes);
  if (workspace_bytes < align256(clef::expert_schedule_bytes(tokens * topk, bm))) return fail(kWorkspace);
  int32_t* schedule = static_cast<int32_t*>(workspace);
  if (int rc = hip_status(clef::launch_expert_schedule(groups, tokens, bm, schedule, hs(stream)))) return rc;
  return hip_status(clef::launch_expert_gate_up(a, stride / 8, a_scales, gate_w, gate_s, up_w, up_s, groups,
                                                schedule, bm, tokens, topk, k, n, h, hs(stream)));
}

int clef_swiglu(const uint16_t* gate, const uint16_t* up, int64_t n, uint16_t* h, clef_stream_t stream) {
  if (n < 0) return fail("SwiGLU shape/dtype mismatch");
  if (n == 0) return CLEF_OK;
  if (!aligned(gate, 16) || !aligned(up, 16) || !aligned(h, 16)) return fail(kAlign);
  return hip_status(clef::launch_swiglu(gate, up, n, h, hs(stream)));
}

int clef_moe_combine(const uint16_t* values, const float* routes, const float* order,
                     int64_t tokens, int32_t width, int32_t topk, uint16_t* out,
                     clef_stream_t stream) {
  // src/omni.rs:253-262.
  if (!(tokens >= 1 && width >= 8 && width % 8 == 0 && topk >= 1 && topk <= 128))
    return fail("unsupported ordered Omni accumulation");
  if (!aligned(values, 16) || !aligned(routes, 4) || (order && !aligned(order, 4)) || !aligned(out, 16))
    return fail(kAlign);
  return hip_status(clef::launch_combine(values, routes, order, tokens, width, topk, out, hs(stream)));
}

}  // extern "C"

namespace {

// Workspace carve-up of the MoE block; offsets are 256-byte aligned. `bytes`:
// what the workspace holds; the schedule, last, takes expert tiles that fit.
struct MoeLayout {
  int bm;  // slots per expert tile
  size_t routes, groups, order, group_ws, ax, h, ah, values, schedule, total;
};

MoeLayout moe_layout(int64_t tokens, int32_t hidden, int32_t inter, int32_t topk, size_t bytes = SIZE_MAX) {
  MoeLayout l{};
  const int64_t routed = tokens * topk;
  size_t at = 0;
  auto take = [&](size_t bytes) {
    size_t here = at;
    at += align256(bytes);
    return here;
  };
  l.routes = take((size_t)tokens * 2 * topk * 4);
  l.groups = take((size_t)128 * (tokens + 1) * 4);
  l.order = take((size_t)routed * 4);
  const size_t grouping = clef::group_workspace_bytes(tokens);
  const size_t counted = clef::group_counted_fusable(tokens, topk) ? clef::group_counted_bytes(tokens) : 0;
  l.group_ws = take(grouping > counted ? grouping : counted);  // the three-pass grouping's or the router's counts
  l.ax = take((size_t)prepared_words(tokens, stride_for(hidden, 4), 4) * 4);
  l.h = take((size_t)routed * inter * 2);
  l.ah = take((size_t)prepared_words(routed, stride_for(inter, 4), 4) * 4);
  l.values = take((size_t)routed * hidden * 2);
  l.bm = clef::expert_tile_rows(routed, hidden > inter ? hidden : inter, bytes > at ? bytes - at : 0);
  l.schedule = take(clef::expert_schedule_bytes(routed, l.bm));
  l.total = at;
  return l;
}

}  // namespace

extern "C" {

size_t clef_moe_layer_workspace_bytes(int64_t tokens, int32_t hidden, int32_t inter, int32_t topk) {
  if (tokens < 1 || hidden < 1 || inter < 1 || topk < 1) return 0;
  return moe_layout(tokens, hidden, inter, topk).total;
}

}  // extern "C"

namespace {

// Shape checks of the MoE block (shared by clef_moe_layer and
// clef_moe_layer_static); no pointer is dereferenced.
int check_moe_layer(int64_t tokens, int32_t hidden, int32_t inter, int32_t experts, int32_t topk) {
  if (experts != 128) return fail("Omni MoE requires 128 experts");
  if (!(topk >= 1 && topk <= experts)) return fail("invalid expert router shape");
  if (!routes_in_range(tokens, topk)) return fail("unsupported Omni route grouping shape");
  if (!(hidden % 256 == 0 && inter % 256 == 0 && hidden >= 256 && inter >= 256))
    return fail("unsupported Omni expert tile shape");
  const int32_t sx = stride_for(hidden, 4), sh = stride_for(inter, 4);
  if (int rc = check_prepare(tokens, hidden, sx, 4)) return rc;
  if (int rc = check_prepare(tokens * topk, inter, sh, 4)) return rc;
  if (!operand_below_2gib(tokens, sx) || !operand_below_2gib(tokens * topk, sh)) return fail(kOperand);
  return CLEF_OK;
}

int check_moe_pointers(const uint16_t* x, const void* logits, const uint32_t* gate_w, const float* gate_s,
                       const uint32_t* up_w, const float* up_s, const uint32_t* down_w, const float* down_s,
                       const float* routes_out, const uint16_t* out) {
  if (!aligned(x, 16) || !aligned(logits, 16) || !aligned(gate_w, 16) || !aligned(gate_s, 16) ||
      !aligned(up_w, 16) || !aligned(up_s, 16) || !aligned(down_w, 16) || !aligned(down_s, 16) ||
      !aligned(out, 16) || (routes_out && !aligned(routes_out, 4)))
    return fail(kAlign);
  return CLEF_OK;
}

// The MoE block's launches on a checked shape, intermediates carved from `ws`
// (moe_layout). Every intermediate is written before it is read, so `ws`
// needs no clearing.
int moe_layer_run(const uint16_t* x, const void* logits, int32_t logits_dtype, int64_t tokens, int32_t hidden,
                  int32_t inter, int32_t experts, int32_t topk, const uint32_t* gate_w, const float* gate_s,
                  const uint32_t* up_w, const float* up_s, const uint32_t* down_w, const float* down_s,
                  float* routes_out, uint16_t* out, char* ws, const MoeLayout& l, hipStream_t s) {
  const int32_t sx = stride_for(hidden, 4), sh = stride_for(inter, 4);
  float* routes = routes_out ? routes_out : reinterpret_cast<float*>(ws + l.routes);
  float* groups = reinterpret_cast<float*>(ws + l.groups);
  float* order = reinterpret_cast<float*>(ws + l.order);
  int32_t* schedule = reinterpret_cast<int32_t*>(ws + l.schedule);
  uint32_t* ax = reinterpret_cast<uint32_t*>(ws + l.ax);
  uint16_t* h = reinterpret_cast<uint16_t*>(ws + l.h);
  uint32_t* ah = reinterpret_cast<uint32_t*>(ws + l.ah);
  uint16_t* values = reinterpret_cast<uint16_t*>(ws + l.values);
  const int64_t routed = tokens * topk;
  const float* axs = reinterpret_cast<const float*>(ax + tokens * (sx / 8));
  const float* ahs = reinterpret_cast<const float*>(ah + routed * (sh / 8));

#define CLEF_STEP(call) \
  if (int rc = hip_status(call)) return rc
  if (clef::route_gate_up_fusable(tokens, topk, experts, hidden, inter)) {
    // a few tokens: routing, Q1(x) and gate/up + SwiGLU in one launch, then
    // the down projection (with its quantizer) and combine in another
    CLEF_STEP(clef::launch_route_gate_up(logits, logits_dtype, tokens, x, gate_w, gate_s, up_w, up_s, hidden, inter,
                                         routes, order, h, s));
    CLEF_STEP(clef::launch_down_combine(h, down_w, down_s, routes, order, tokens, topk, inter, hidden, out, s));
    return CLEF_OK;
  }
  if (clef::route_prepare_fusable(hidden) && clef::route_group_fusable(tokens, topk)) {
    // at most 16 tokens: the routing workgroup also groups them
    CLEF_STEP(clef::launch_route_prepare(logits, logits_dtype, tokens, experts, topk, routes, x, hidden, sx, ax, s,
                                         groups, order, schedule, l.bm));
  } else if (clef::route_prepare_fusable(hidden) && clef::group_counted_fusable(tokens, topk)) {
    // the router also counts each 16-token block's routes per expert; one
    // launch then scans the counts and lists the routes
    int* counts16 = reinterpret_cast<int*>(ws + l.group_ws);
    CLEF_STEP(clef::launch_route_prepare(logits, logits_dtype, tokens, experts, topk, routes, x, hidden, sx, ax, s,
                                         nullptr, nullptr, nullptr, 0, counts16));
    CLEF_STEP(clef::launch_group_counted(routes, tokens, counts16, groups, order, schedule,
                                         l.bm, s));
  } else if (clef::route_prepare_fusable(hidden)) {  // router and the quantizer of x side by side
    CLEF_STEP(clef::launch_route_prepare(logits, logits_dtype, tokens, experts, topk, routes, x, hidden, sx, ax, s));
    CLEF_STEP(clef::launch_group_routes(routes, tokens, topk, groups, order, ws + l.group_ws, s, schedule,
                                        l.bm));
  } else {
    CLEF_STEP(clef::launch_route(logits, logits_dtype, tokens, experts, topk, routes, s));
    CLEF_STEP(clef::launch_group_routes(routes, tokens, topk, groups, order, ws + l.group_ws, s, schedule,
                                        l.bm));
    CLEF_STEP(clef::launch_prepare(x, tokens, hidden, sx, 4, ax, s));
  }
  // Gate and up share one pass over the gathered x rows and SwiGLU runs in
  // their epilogue; h is then quantized per routed row. Bit-equal to the
  // separate gate, up, swiglu and prepare (each lane applies the same E1
  // rounding and S1 to the same bf16 values).
  CLEF_STEP(clef::launch_expert_gate_up(ax, sx / 8, axs, gate_w, gate_s, up_w, up_s, groups, schedule, l.bm, tokens,
                                        topk, hidden, inter, h, s));
  if (clef::down_combine_fusable(tokens, topk, inter, hidden)) {
    // a few tokens: down projection, its quantizer and combine in one launch
    CLEF_STEP(clef::launch_down_combine(h, down_w, down_s, routes, order, tokens, topk, inter, hidden, out, s));
    return CLEF_OK;
  }
  if (clef::expert_down_h_fusable(routed, inter, hidden)) {
    // few routed rows: the down projection quantizes its h rows itself
    CLEF_STEP(clef::launch_expert_down_h(h, down_w, down_s, groups, schedule, tokens, topk, inter, hidden, values, s));
  } else {
    CLEF_STEP(clef::launch_prepare(h, routed, inter, sh, 4, ah, s));
    CLEF_STEP(clef::launch_expert_i4(ah, sh / 8, ahs, down_w, down_s, groups, schedule, l.bm, tokens, topk,
                                     inter, hidden, 1, values, s));
  }
  CLEF_STEP(clef::launch_combine(values, routes, order, tokens, hidden, topk, out, s));
#undef CLEF_STEP
  return CLEF_OK;
}

// ---------------------------------------------------------------- static scratch

// Scratch of clef_moe_layer_static: one array per device that loads the
// library, held until the process ends. The host-side name `scratch` is not a
// device address; its device address comes from hipGetSymbolAddress, once
// per device, and only that pointer is handed to kernels.
constexpr size_t kStaticScratchBytes = CLEF_MOE_STATIC_SCRATCH_BYTES;
__device__ __align__(256) char scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
char* g_scratch_ptr[kMaxDevices] = {};

// The current device's scratch address, looked up on the first call on that
// device (with the device current).
int static_scratch(char** ptr) {
  int dev = 0;
  if (int rc = hip_status(hipGetDevice(&dev))) return rc;
  if (dev < 0 || dev >= kMaxDevices) return fail("device index beyond the static scratch table");
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    if (int rc = hip_status(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)))) return rc;
    g_scratch_ptr[dev] = static_cast<char*>(p);
  }
  *ptr = g_scratch_ptr[dev];
  return CLEF_OK;
}

}  // namespace

extern "C" {

int clef_moe_layer(const uint16_t* x, const void* logits, int32_t logits_dtype, int64_t tokens,
                   int32_t hidden, int32_t inter, int32_t experts, int32_t topk,
                   const uint32_t* gate_w, const float* gate_s, const uint32_t* up_w,
                   const float* up_s, const uint32_t* down_w, const float* down_s,
                   float* routes_out, uint16_t* out, void* workspace, size_t workspace_bytes,
                   clef_stream_t stream) {
  if (int rc = check_moe_layer(tokens, hidden, inter, experts, topk)) return rc;
  if (int rc = check_moe_pointers(x, logits, gate_w, gate_s, up_w, up_s, down_w, down_s, routes_out, out)) return rc;
  if (!aligned(workspace, 256)) return fail(kAlign);
  const MoeLayout l = moe_layout(tokens, hidden, inter, topk, workspace_bytes);
  if (workspace_bytes < l.total) return fail(kWorkspace);
  return moe_layer_run(x, logits, logits_dtype, tokens, hidden, inter, experts, topk, gate_w, gate_s, up_w, up_s,
                       down_w, down_s, routes_out, out, static_cast<char*>(workspace), l, hs(stream));
}

int clef_moe_layer_static(const uint16_t* x, const void* logits, int32_t logits_dtype, int64_t tokens,
                          int32_t hidden, int32_t inter, int32_t experts, int32_t topk,
                          const uint32_t* gate_w, const float* gate_s, const uint32_t* up_w,
                          const float* up_s, const uint32_t* down_w, const float* down_s,
                          float* routes_out, uint16_t* out, clef_stream_t stream) {
  if (int rc = check_moe_layer(tokens, hidden, inter, experts, topk)) return rc;
  if (int rc = check_moe_pointers(x, logits, gate_w, gate_s, up_w, up_s, down_w, down_s, routes_out, out)) return rc;
  const MoeLayout l = moe_layout(tokens, hidden, inter, topk, kStaticScratchBytes);
  const size_t need = l.total;
  if (need > kStaticScratchBytes) {
    std::snprintf(g_error, sizeof g_error,
                  "MoE layer needs %zu bytes of scratch; the static scratch holds %zu (use clef_moe_layer "
                  "with a workspace, or fewer tokens)",
                  need, kStaticScratchBytes);
    return CLEF_EINVAL;
  }
  char* ws = nullptr;
  if (int rc = static_scratch(&ws)) return rc;
  return moe_layer_run(x, logits, logits_dtype, tokens, hidden, inter, experts, topk, gate_w, gate_s, up_w, up_s,
                       down_w, down_s, routes_out, out, ws, l, hs(stream));
}

}  // extern "C"
