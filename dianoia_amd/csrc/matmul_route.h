// The product route of one matmul command: which kernels
// lab_gpu_enc_matmul_q8 / _q4 (lib/src/gpu.dart:137-190, encoded by
// GpuLinear.apply :1327-1341) run for its format, input mode, token count
// and shape. Shared by the lab_gpu_* command recorder (lab_gpu.hip) and the
// dnx_matmul_* device-pointer entry points (matmul.hip), so both always take
// the same path.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dnx_kernels.h"

namespace dnx {

// Kernel launches of a route, reported to the caller's hook after each one.
enum class MatmulStep { kGemvFloat, kGemmFloat, kGemv, kQuantize, kGemm, kQuantizeF6, kGemmF6 };

inline int64_t align256(int64_t v) { return (v + 255) & ~(int64_t)255; }

// The fp6-MFMA GEMM against quantize + int8-MFMA GEMM (us with the quantizer,
// graph-timed, six weight copies in turn). On the engine's layout (96-row
// tiles): 6144 x 2048 at 256 / 320 / 375 / 512 / 1024 tokens 25.3 / 23.0 / 23.3
// / 26.1 / 46.0 against 24.0 / 25.2 / 30.4 / 31.8 / 58.2, 4096 x 4096 at 320 /
// 512 37.6 / 38.7 against 37.7 / 51.0; 4096 x 1024 at 320 / 512 ties (15.2 /
// 15.7 against 15.0 / 15.3), and with fewer rows it loses up to 512 tokens
// (3072 x 1024 at 375 / 512 19.2 / 21.6 against 15.4 / 15.1, 2048 x 2048 at 320
// / 512 20.7 / 21.8 against 19.5 / 21.6). On prepacked weights (dnx_gemm_q4_f6p,
// 32 to 128 rows) against the chunk route below: 6144 x 2048 at 256 / 320 / 512
// 23.7 / 20.4 / 23.6 against 20.7 / 22.0 / 30.9, 2048 x 2048 at 512 19.7
// against 14.7. The line is one for both, and leaves two ranges to the int8
// GEMM where the prepacked kernel is the faster by now: above 512 tokens with
// fewer rows (2048 x 2048 at 1024 21.8 against 26.6, 3072 x 1024 at 640 13.4
// against 15.5) or K above 4096 (2048 x 6144 at 1000 43.0 against 70.9).
inline bool matmul_uses_f6(bool q4, int64_t rows, int64_t cols, int64_t n) {
  return q4 && n >= 320 && rows >= 4096 && cols <= 4096;
}

// A prefill chunk (the reference prefills in chunks of up to 64 tokens,
// lib/src/model.dart:91) or another batch of up to 512 tokens of a Q4
// matrix that the tiled fp6 route above does not take (the audio encoder's
// 375 frames, the callers' 128 and 256): with a prepacked copy of the
// weights (the lab_gpu_* command buffer keeps one per weight region) it runs
// as the f6 panel quantizer + dnx_gemm_q4_f6s, one launch over the whole K.
// Measured against quantize + int8 GEMM (skinny, chunk or tile kernel by
// shape; us, graph-timed with the quantizer): 6144 x 2048 at 8 / 16 / 32 / 64
// tokens 8.0 / 8.1 / 8.5 / 10.3 against 11.7 / 12.9 / 13.0 / 15.6, at 128 / 256
// 12.8 / 20.7 against 18.9 / 24.0; 3072 x 1024 at 64 / 512 6.5 / 14.8 against
// 8.1 / 15.1; 2048 x 2048 at 33 / 64 / 128 7.9 / 8.0 / 8.6 against 10.6 / 11.8 /
// 12.1; 512 x 2048, 2048 x 512, 4096 x 1024 and 1024 x 4096 at 375 9.7 / 8.7 /
// 14.4 / 17.0 against 12.7 / 13.4 / 15.0 / 20.5.
inline bool matmul_uses_f6_chunk(bool q4, int64_t rows, int64_t cols, int64_t n) {
  return q4 && n >= 5 && n <= 512 && !matmul_uses_f6(q4, rows, cols, n);
}

// Q8 batches (the vision encoder's attention projections, fc1 / fc2 and
// projector at its 1024 patches, lib/src/vision_encoder.dart:252-316) with
// a prepacked copy of the weights (the lab_gpu_* command buffer keeps one
// per weight region): the int8 panel quantizer + dnx_gemm_q8_i8p.
// Measured against quantize + int8 GEMM (us with the quantizer, graph-timed,
// six weight copies in turn): 1152 x 4320 and 4320 x 1152 at 1024 tokens 33.6 /
// 27.3 against 43.8 / 31.1, 4096 x 4096 at 1024 54.6 against 78.9, 1152 x 1152
// at 1024 15.0 against 17.5, 1024 x 1024 at 1024 13.6 against 14.7, 6144 x 2048
// at 256 18.2 against 24.3, 4096 x 1024 at 256 / 512 13.3 / 14.9 against 13.3 /
// 15.6. Below 256 tokens the int8 GEMM wins (2048 x 2048 and 1024 x 1024 at 128
// 10.9 / 7.4 against 13.9 / 10.1). Inside the bounds it has become the faster
// where its chunk kernel takes the shape (1024 x 1024 at 256 / 512 7.7 / 10.0
// against 12.1 / 14.3, 768 x 768 at 512 9.2 against 12.4, 2048 x 1024 at 256 9.4
// against 12.6) and on 2048 x 2048 at 256 (14.5 against 15.7); the bounds are
// older than that kernel and do not leave those shapes to it.
inline bool matmul_uses_i8p(bool q4, int64_t rows, int64_t cols, int64_t n) {
  return !q4 && n >= 256 && rows * cols * n >= (1ll << 28);
}

// Device bytes a route needs for its quantized activations: int8 xq and fp32
// block scales (each 256-byte aligned), or the fp6 activation panel.
inline int64_t matmul_workspace_bytes(int64_t cols, int64_t n) {
  if (cols <= 0 || n <= 0 || cols % 32 != 0) return -1;
  const int64_t q8 = align256(n * cols) + align256(n * (cols / 32) * 4);
  const int64_t f6 = dnx_f6_panel_bytes(n, cols);
  return q8 > f6 ? q8 : f6;
}

// int8_inputs (mode 1, lab_native.c:553-579, :1059-1080): n <= 4 runs the
// exact GEMV (its prologue quantizes x); wider n, or an x too wide for the
// GEMV's LDS, quantizes x into the workspace and runs a GEMM. Float inputs
// (mode 0): n <= 4 the exact float-input GEMV; wider n, or an x too wide for
// the GEMV's LDS, the bf16-MFMA float GEMM (fp32 rounding of the CPU's).
// after(step) follows every successful launch. Returns the first error.
template <class After>
int matmul_route(bool q4, const void* qs, const void* scales, const float* x, float* y,
                 int64_t rows, int64_t cols, int64_t n, bool int8_inputs, void* workspace,
                 int64_t workspace_bytes, hipStream_t stream, After&& after) {
  auto s = (dnx_stream_t)stream;
  int rc;
  if (!int8_inputs) {
    if (n <= 4) {
      rc = q4 ? dnx_gemv_q4_float((const uint8_t*)qs, (const uint16_t*)scales, x, y, rows, cols,
                                  n, s)
              : dnx_gemv_q8_float((const int8_t*)qs, (const float*)scales, x, y, rows, cols, n, s);
      if (rc == DNX_OK) after(MatmulStep::kGemvFloat);
      if (rc != DNX_EINVAL) return rc;  // EINVAL: x too wide for the GEMV, nothing launched
    }
    rc = q4 ? dnx_gemm_q4_float((const uint8_t*)qs, (const uint16_t*)scales, x, y, rows, cols, n, s)
            : dnx_gemm_q8_float((const int8_t*)qs, (const float*)scales, x, y, rows, cols, n, s);
    if (rc == DNX_OK) after(MatmulStep::kGemmFloat);
    return rc;
  }
  if (n <= 4) {
    rc = q4 ? dnx_gemv_q4((const uint8_t*)qs, (const uint16_t*)scales, x, y, rows, cols, n, s)
            : dnx_gemv_q8((const int8_t*)qs, (const float*)scales, x, y, rows, cols, n, s);
    if (rc == DNX_OK) after(MatmulStep::kGemv);
    if (rc != DNX_EINVAL) return rc;  // EINVAL: x too wide for the GEMV, nothing launched
  }
  const int64_t need = matmul_workspace_bytes(cols, n);
  if (need < 0 || workspace == nullptr || workspace_bytes < need) return DNX_EINVAL;
  // The fp6 panel quantizer reads x 16 bytes at a time; an x that is only
  // 4-byte aligned (a float offset into a caller's buffer) takes the int8
  // route below, which reads it a float at a time where it must.
  if (matmul_uses_f6(q4, rows, cols, n) && ((uintptr_t)x & 15) == 0) {
    rc = dnx_quantize_q8_f6panel(x, workspace, n, cols, s);
    if (rc != DNX_OK) return rc;
    after(MatmulStep::kQuantizeF6);
    rc = dnx_gemm_q4_f6((const uint8_t*)qs, (const uint16_t*)scales, workspace, y, rows, cols, n,
                        s);
    if (rc == DNX_OK) after(MatmulStep::kGemmF6);
    return rc;
  }
  int8_t* xq = (int8_t*)workspace;
  float* xs = (float*)((char*)workspace + align256(n * cols));
  rc = dnx_quantize_q8(x, xq, xs, n, cols, cols, s);
  if (rc != DNX_OK) return rc;
  after(MatmulStep::kQuantize);
  rc = q4 ? dnx_gemm_q4((const uint8_t*)qs, (const uint16_t*)scales, xq, xs, y, rows, cols, n, s)
          : dnx_gemm_q8((const int8_t*)qs, (const float*)scales, xq, xs, y, rows, cols, n, s);
  if (rc == DNX_OK) after(MatmulStep::kGemm);
  return rc;
}

}  // namespace dnx
