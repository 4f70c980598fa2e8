// Host entry of the rowwise matrix-core product (rowwise_mm.hpp), one
// translation unit per bit width (lb_rowwise_mm.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace lb {
namespace rwmm {

struct Params {
  const uint8_t* q[2];
  const uint16_t* s[2];
  uint16_t* y[2];
  const uint16_t* x;
  int64_t x_stride;  // halves between activation rows
  int64_t y_stride;  // halves between output rows
  int64_t packed_cols, scale_cols;
  int rows, cols, batch;
  uint32_t span_mul;  // group of scale span t (of 128 / sps columns): t where 0, else mulhi(t, span_mul)
};

// Launches the product of `mats` matrices (1, or 2 sharing x) for a layout of
// `sps` scale spans per 128 columns (1, 2 or 4); returns an lb_status code.
template <int BITS>
int launch(const Params& p, int sps, int mats, hipStream_t st);

}  // namespace rwmm
}  // namespace lb
