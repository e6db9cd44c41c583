// Host side of the grouped GEMM's dual tiles (grouped_gemm_dual.hip).
#pragma once

#include "grouped_gemm.hpp"

namespace fluxmi {

// Whether the dual tiles take a launch that is the macro tiles' otherwise.
bool dual_takes(const GemmParams &p, int dtype);
int launch_grouped_gemm_dual(const GemmParams &p, int dtype, int grid, hipStream_t s);

}  // namespace fluxmi
