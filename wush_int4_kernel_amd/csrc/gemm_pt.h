// gemm_pt.h -- launcher of the per-tensor int8-MFMA tiles (gemm_pt.hip), called
// by the planner in gemm_s4.hip.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace wush {

// y = alpha * (xq @ wq^T), M x N fp16, exact int32 dots; K % 256 == 0, code
// tensors 16-byte aligned.  Output tiles of 256 x 256, 256 x 128 or 128 x 128;
// hipErrorInvalidValue for others.  alpha_dev overrides alpha when not NULL.
int launch_gemm_pt(const uint8_t* xq, const uint8_t* wq, uint16_t* y, int M, int N, int K, float alpha,
                   const float* alpha_dev, int tile_rows, int tile_cols, hipStream_t stream);

}  // namespace wush
