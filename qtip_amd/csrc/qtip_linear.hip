// A quantized projection as one library call (qtip_linear): the launches of the transforms and the product, with
// the scratch between them.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/qtip_hip.h"
#include "qtip_setup.h"

namespace {

// Scratch of a call: the transformed input (unless the matvec makes it), the product, the GEMM's partial sums.
struct LinearPlan {
  bool in_matvec;
  int S;
  size_t y_off, ws_off, ws_bytes, total;
};

LinearPlan linear_plan(int m, int k, int bits, int rows, int order_in, int x_dtype, bool fine) {
  auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
  LinearPlan p{};
  p.S = rows == 1 ? qtip_matvec_split(m, k, bits) : 1;
  p.in_matvec = rows == 1 && order_in == 1 && x_dtype == QTIP_F16 && (k == 2048 || k == 4096 || k == 8192);
  p.y_off = p.in_matvec ? 0 : up((size_t)rows * k * 2);
  p.ws_off = p.y_off + up(rows == 1 ? (size_t)p.S * m * sizeof(float) : (size_t)rows * m * 2);
  p.ws_bytes = rows == 1 ? 0 : qtip_gemm_scratch(m, k, bits, rows, fine);
  p.total = p.ws_off + p.ws_bytes;
  return p;
}

bool linear_shape_ok(int m, int k, int bits, int rows) {
  return m > 0 && k > 0 && !((m | k) & 31) && bits >= 2 && bits <= 4 && rows >= 1 && rows <= 65535 &&
         (long)m * k * bits / 8 < (1L << 31);
}

int run_linear(void* out, const void* x, int x_dtype, const void* packed, const void* tlut, const void* su_f16, const float* sv,
               const uint32_t* had_in, int order_in, const uint32_t* had_out, int order_out, int m, int k, int bits, int rows,
               float scale_in, float scale_out, void* workspace, size_t workspace_bytes, bool fine, void* stream,
               int pre_mode = 0, const void* norm_w = nullptr, float eps = 0.f, const void* residual = nullptr) {
  if (!out || !x || !packed || !tlut || !su_f16 || !sv || !workspace) return QTIP_E_NULL;
  if (!linear_shape_ok(m, k, bits, rows)) return QTIP_E_SHAPE;
  if (x_dtype != QTIP_F16 && x_dtype != QTIP_F32) return QTIP_E_DTYPE;
  if (!aligned16(workspace)) return QTIP_E_ALIGN;
  const LinearPlan p = linear_plan(m, k, bits, rows, order_in, x_dtype, fine);
  if (rows == 1 && p.S < 1) return QTIP_E_SHAPE;
  if (workspace_bytes < p.total) return QTIP_E_WORKSPACE;
  uint8_t* ws = (uint8_t*)workspace;
  void* y = ws + p.y_off;
  int rc;
  if (p.in_matvec) {
    rc = qtip_decompress_matvec_parts_rht((float*)y, packed, x, su_f16, scale_in, tlut, m, k, bits, p.S, stream);
  } else {
    rc = qtip_rht_fused(ws, QTIP_F16, x, x_dtype, 1, rows, k, order_in, had_in, su_f16, nullptr, scale_in, pre_mode, norm_w,
                        eps, nullptr, stream);
    if (rc) return rc;
    // A product cut along k: the output transform adds the ranges on load where it is a form of many rows that takes them; a
    // launch for the sums and a pass over them less, the same bits.  us per call in a graph, fp16, m x k, rows (ranges), before
    // -> now: 2048 x 4096, 2 (4) 13.9 -> 12.3; 4096 x 4096, 5 (4) 15.0 -> 12.9, 9 (4) 14.8 -> 13.2, 64 (4) 20.4 -> 18.3,
    // 120 (2) 23.7 -> 21.4; 4096 x 11008, 64 (4) 33.6 -> 31.6; 8192 x 28672, 400 (4) 232.7 -> 227.9; 5120 x 2048, 64 (2)
    // 21.3 -> 19.7.
    if (rows > 1 && p.ws_bytes && aligned16(out) && aligned16(sv) && aligned16(residual)) {
      const int S = qtip_gemm_ranges(m, k, bits, rows, fine);
      if (S > 1 && qtip_rht_takes_parts(m, order_out, rows, S, residual != nullptr)) {
        auto* parts = (float*)(ws + p.ws_off);
        rc = qtip_gemm_parts(parts, S, packed, ws, tlut, m, k, bits, rows, fine, stream);
        if (rc) return rc;
        return qtip_rht_from_parts(out, x_dtype, parts, S, rows, m, order_out, had_out, sv, scale_out, residual, stream);
      }
    }
    auto* product = fine ? qtip_decompress_gemm_f16 : qtip_decompress_gemm_long_f16;
    rc = rows == 1 ? qtip_decompress_matvec_parts((float*)y, packed, ws, tlut, m, k, bits, p.S, stream)
                   : product(y, packed, ws, tlut, m, k, bits, rows, p.ws_bytes ? ws + p.ws_off : nullptr, p.ws_bytes, stream);
  }
  if (rc) return rc;
  return qtip_rht_fused(out, x_dtype, y, rows == 1 ? QTIP_F32 : QTIP_F16, p.S, rows, m, order_out, had_out, nullptr, sv,
                        scale_out, 0, nullptr, 0.f, residual, stream);
}

}  // namespace

extern "C" {

size_t qtip_linear_workspace_bytes(int m, int k, int bits, int rows, int order_in, int x_dtype) {
  return linear_shape_ok(m, k, bits, rows) ? linear_plan(m, k, bits, rows, order_in, x_dtype, true).total : 0;
}

size_t qtip_linear_long_workspace_bytes(int m, int k, int bits, int rows, int order_in, int x_dtype) {
  return linear_shape_ok(m, k, bits, rows) ? linear_plan(m, k, bits, rows, order_in, x_dtype, false).total : 0;
}

int qtip_linear(void* out, const void* x, int x_dtype, const void* packed, const void* tlut, const void* su_f16,
                const float* sv, const uint32_t* had_in, int order_in, const uint32_t* had_out, int order_out, int m,
                int k, int bits, int rows, float scale_in, float scale_out, void* workspace, size_t workspace_bytes,
                void* stream) {
  return run_linear(out, x, x_dtype, packed, tlut, su_f16, sv, had_in, order_in, had_out, order_out, m, k, bits, rows, scale_in,
                    scale_out, workspace, workspace_bytes, true, stream);
}

int qtip_linear_long(void* out, const void* x, int x_dtype, const void* packed, const void* tlut, const void* su_f16,
                     const float* sv, const uint32_t* had_in, int order_in, const uint32_t* had_out, int order_out, int m,
                     int k, int bits, int rows, float scale_in, float scale_out, void* workspace, size_t workspace_bytes,
                     void* stream) {
  return run_linear(out, x, x_dtype, packed, tlut, su_f16, sv, had_in, order_in, had_out, order_out, m, k, bits, rows, scale_in,
                    scale_out, workspace, workspace_bytes, false, stream);
}

int qtip_linear_rows(void* out_f16, const void* x_f16, const void* packed, const void* tlut, const void* su_f16,
                     const float* sv, const uint32_t* had_in, int order_in, const uint32_t* had_out, int order_out, int m,
                     int k, int bits, int rows, float scale_in, float scale_out, int pre_mode,
                     const void* norm_weight_f16, float eps, const void* residual_f16, int long_sums, void* workspace,
                     size_t workspace_bytes, void* stream) {
  if (rows < 2) return QTIP_E_SHAPE;
  return run_linear(out_f16, x_f16, QTIP_F16, packed, tlut, su_f16, sv, had_in, order_in, had_out, order_out, m, k, bits, rows,
                    scale_in, scale_out, workspace, workspace_bytes, !long_sums, stream, pre_mode, norm_weight_f16, eps,
                    residual_f16);
}

}  // extern "C"
