// The product of a few activation rows (skinny.hip).
#pragma once
#include <algorithm>

#include "common.h"

namespace oco {

constexpr uint32_t SKINNY_ROWS = 31;  // activation rows it takes: fewer than the dequantize pass pays for

// Whether it covers this format and geometry.
bool skinny_fits(uint32_t format, uint32_t m, uint32_t n, uint32_t k);

// Y = X W^T (times inv[row]) + bf16(bias); X f16 or bf16 rows, Y f32 or bf16.
int skinny_launch(uint32_t format, const void *w, const void *x, bool x_f16, void *y, bool y_bf16, const float *bias,
                  const float *inv, uint32_t m, uint32_t n, uint32_t k, hipStream_t stream);

}  // namespace oco
