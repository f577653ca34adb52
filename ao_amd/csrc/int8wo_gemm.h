// The tiled int8 product (int8wo_gemm.hip) as the dispatch of int8wo_linear.hip sees it.
#pragma once
#include "tile_gemm.h"

namespace ao {
TilePlan int8wo_gemm_plan(int64_t M, int64_t N, int64_t K, int max_parts);
void int8wo_gemm_describe(const TilePlan& p, char* out, size_t cap);
// Adds `parts` fp32 products [parts][M][N] at a.parts and finishes as the tiles do
void int8wo_finish_parts(const TileGemmArgs& a, int parts, hipStream_t st);
void launch_int8wo_gemm(TileGemmArgs a, const TilePlan& p, hipStream_t st);
}  // namespace ao
