// The prompt-chunk GEMM that decodes weights in registers (panel.hip).
#pragma once
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace oco {

// Tile and K parts chosen for a geometry; mt == 0: the dequantize pass and
// the GEMM are the better choice, or the geometry is not covered.
struct PanelPlan {
    int mt, nt;
    uint32_t splits;
};
// direct: the GEMM's f32 product would be the output (no bias, no row gain).
PanelPlan panel_plan(uint32_t format, uint32_t m, uint32_t n, uint32_t k, bool direct);
// Whether a tile and K parts can run: a tile built for the format, offsets
// within 32 bits, and the f32 parts within the f16 weights' place.
bool panel_fits(uint32_t format, const PanelPlan &pl, uint32_t m, uint32_t n, uint32_t k);

// x: f16 rows, 16-byte aligned.  With pl.splits > 1 the f32 parts go to
// part[splits][m][n] and the caller sums them; else y = X W^T (times
// inv[row]) + bf16(bias), f32 or bf16.
int panel_launch(uint32_t format, const PanelPlan &pl, const void *w, const uint16_t *x, void *y, bool y_bf16,
                 const float *bias, const float *inv, float *part, uint32_t m, uint32_t n, uint32_t k, hipStream_t stream);

}  // namespace oco
