// Host side of the grouped GEMM's dual tiles (grouped_gemm_dual.hip).
#pragma once

#include "grouped_gemm.hpp"

namespace fluxmi {

// Whether the dual tiles take a launch that is the macro tiles' otherwise.
bool dual_takes(const GemmParams &p, int dtype);
// few: row counts in the arguments (count > 0) and a second factor per row, as the forms for few rows take them.
int launch_grouped_gemm_dual(const GemmParams &p, const FewRowsArgs &few, int dtype, int grid, hipStream_t s);

}  // namespace fluxmi
