// Launcher of the weight-streaming form of the grouped GEMM (grouped_gemm_stream.hip).
#pragma once

#include "grouped_gemm.hpp"

namespace fluxmi {

struct StreamPlan {
  int cols, waves;      // columns per workgroup; waves that split K
  int blocks;           // items the launch is numbered for
  unsigned workgroups;  // workgroups launched; fewer than `blocks`: each walks several items
  bool walk;
  int lds_bytes;        // per workgroup
};

// Whether a launch that the MFMA kernels can take may go to this form: few rows per expert on average.  With more than
// kStreamRows rows in the launch an expert can have several chunks; which form runs is then decided on the device
// (GemmParams::by_splits).
bool grouped_gemm_stream_takes(const GemmParams &p, int dtype);
// Waves that split K.  Of one weight group: a launch of several has the bits of one launch each.
int stream_waves(const GemmParams &p, int dtype);
// cus: compute units the launch may use; leave_cus: the others are to be left to other work.
StreamPlan plan_grouped_gemm_stream(const GemmParams &p, int dtype, int cus, bool leave_cus);
void launch_grouped_gemm_stream(const GemmParams &p, const FewRowsArgs &few, int dtype, const StreamPlan &plan, hipStream_t s);

}  // namespace fluxmi
