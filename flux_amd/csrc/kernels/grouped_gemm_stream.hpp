// Launcher of the weight-streaming form of the grouped GEMM (grouped_gemm_stream.hip).
#pragma once

#include "grouped_gemm.hpp"

namespace fluxmi {

// Whether a launch that the MFMA kernels can take goes to this form: few rows per expert on average.
bool grouped_gemm_stream_takes(const GemmParams &p, int dtype);
// cus: compute units it may use, 0 for all of them.
void launch_grouped_gemm_stream(const GemmParams &p, int dtype, int cus, hipStream_t s);

}  // namespace fluxmi
