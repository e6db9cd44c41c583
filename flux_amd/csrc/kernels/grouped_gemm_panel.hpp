// Launcher of the panel forms of the grouped GEMM (grouped_gemm_panel.hip).
#pragma once

#include "grouped_gemm.hpp"

namespace fluxmi {

// cols == 0: the launch is not for these forms.
struct PanelPlan {
  int cols;             // columns per workgroup: 64 or 128 (weights through LDS), 256 (weights through registers)
  int chunk_rows;       // most rows of a work item: 32, 64 or 128
  int sums;             // partial sums of a result over K: 4 or 8 (few rows per expert, the streaming form's bits), 1
  bool deep;            // 64 columns, 64 rows: a ring of six stages in pairs, one workgroup to a unit
  bool pairs;           // 64 columns, 32 rows: lines of K are asked for in pairs
  int blocks;           // items the launch is numbered for
  unsigned workgroups;  // workgroups launched; fewer than `blocks`: each walks several items
  bool walk;
  int chunk_items;      // items of a chunk of rows,
  int round_items;      // items that run at once: where a round more is not worth it (stream_chunks_limit), otherwise 0
  bool any_splits;      // computes every distribution of the rows; otherwise only those with few chunks (stream_chunks_limit)
  int lds_bytes;        // per workgroup
};

// few_rows: the launch has few enough rows for the streaming form.
PanelPlan plan_panel(const GemmParams &p, int dtype, bool few_rows, int cus, bool leave_cus);
// The plan for a launch of `chunks` chunks of rows, known on the host: no workgroups without an item.
void set_chunks(const GemmParams &p, int64_t chunks, int cus, PanelPlan &plan);
int launch_grouped_gemm_panel(const GemmParams &p, const FewRowsArgs &few, int dtype, const PanelPlan &plan, hipStream_t s);

}  // namespace fluxmi
