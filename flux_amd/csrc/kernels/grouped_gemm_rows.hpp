// Device code shared by the forms of the grouped GEMM for few rows per expert (grouped_gemm_stream.hip, grouped_gemm_panel.hip).
#pragma once

#include "grouped_gemm_stream.hpp"

namespace fluxmi {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

enum class Elem { BF16, F16, FP8, FP8_BLOCKSCALED };
constexpr bool is_fp8(Elem t) { return t == Elem::FP8 || t == Elem::FP8_BLOCKSCALED; }

#if defined(__HIP_DEVICE_COMPILE__)

constexpr uint32_t kOutOfRange = 0xfffffff0u;  // a byte offset past every buffer: the load returns zeros

// Clamped like the macro-tile kernel's: negative counts are 0, rows past max_rows do not exist.
struct WorkItem {
  int e, expert_base, expert_rows;  // the expert, its first row, its row count
  int row_base, rows;               // the item's rows (0: there is no such item)
  int nt;                           // column tile, over all weight groups
};

typedef const __attribute__((address_space(4))) FewRowsArgs *ArgSegment;

// Scale of output row `row`, the tile's included.
__device__ __forceinline__ float row_factor(const GemmParams &p, const FewRowsArgs &f, float tile_scale, int row) {
  float s = p.row_scale ? p.row_scale[row] : 1.f;
  if (f.row_scale2) s *= f.row_scale2[row];
  return tile_scale * s;
}

// Work item -> (expert, chunk of its rows, column tile); a chunk is at most chunk_rows rows (a power of two, 16 or more), and the chunks of
// an expert are about equally long.  One wave-wide pass over the splits counts the chunks, a second finds the item's; with up to
// 64 experts both work on the same registers.
template <Elem T>
__device__ __forceinline__ WorkItem locate(const GemmParams &p, int tiles_n, int chunk_rows, int block) {
  const int lane = threadIdx.x & 63;
  int begin, rows, chunks_end;  // this lane's expert of the 64 looked at
  const ArgSegment args = (ArgSegment)__builtin_amdgcn_kernarg_segment_ptr();
  auto load = [&](int e0, int &row_carry, int &chunk_carry) {
    const int ee = e0 + lane;
    int r = 0;
    if (ee < p.nexperts) r = args->count > 0 ? args->splits[ee] : p.splits[ee];
    if (r < 0) r = 0;
    const int incl = wave_inclusive_scan(r);
    begin = row_carry + incl - r;
    int end = row_carry + incl;
    if (begin > p.max_rows) begin = p.max_rows;
    if (end > p.max_rows) end = p.max_rows;
    rows = end - begin;
    row_carry += __builtin_amdgcn_readlane(incl, 63);
    chunks_end = chunk_carry + wave_inclusive_scan((rows + chunk_rows - 1) / chunk_rows);
    chunk_carry = __builtin_amdgcn_readlane(chunks_end, 63);
    return __popcll(__ballot(rows > 0));
  };
  int row_carry = 0, total = 0, active = 0;
  for (int e0 = 0; e0 < p.nexperts; e0 += 64) active += load(e0, row_carry, total);
  WorkItem w = {0, 0, 0, 0, 0, 0};
  if (p.by_splits && total > stream_chunks_limit(active, chunk_rows, is_fp8(T), p.chunk_items, p.round_items)) return w;  // the macro tiles run this launch
  // Workgroups are dealt to the eight XCDs round-robin.
  const int items = total * tiles_n, per_xcd = (items + 7) / 8, i = block >> 3, item = (block & 7) * per_xcd + i;
  if (i >= per_xcd || item >= items) return w;
  int row_carry2 = 0, chunk_carry2 = 0;
  for (int e0 = 0; e0 < p.nexperts; e0 += 64) {
    if (p.nexperts > 64) load(e0, row_carry2, chunk_carry2);
    const uint64_t hit = __ballot(item < chunks_end * tiles_n);
    if (hit != 0) {
      const int src = __ffsll(static_cast<unsigned long long>(hit)) - 1;
      w.e = e0 + src;
      w.expert_base = __builtin_amdgcn_readlane(begin, src);
      w.expert_rows = __builtin_amdgcn_readlane(rows, src);
      const int chunks = (w.expert_rows + chunk_rows - 1) / chunk_rows;
      const int local = item - (__builtin_amdgcn_readlane(chunks_end, src) - chunks) * tiles_n;
      w.nt = local;
      w.row_base = w.expert_base;
      w.rows = w.expert_rows;
      if (chunks == 1) return w;
      // (readfirstlane: quotients of scalars, which the compiler leaves in vector registers)
      const int per = (__builtin_amdgcn_readfirstlane((w.expert_rows + chunks - 1) / chunks) + 15) & ~15;
      w.nt = __builtin_amdgcn_readfirstlane(local / chunks);
      const int first = (local - w.nt * chunks) * per;
      w.row_base += first;
      w.rows = w.expert_rows - first < per ? w.expert_rows - first : per;
      return w;
    }
  }
  return w;
}

// Two loads of eight rows each (lane: row l & 7, chunk 2 * (l >> 4) + bit 3 of l) -> two MFMA fragments of the sixteen rows
// (lane: row l & 15, chunks 2 * (l >> 4) and 2 * (l >> 4) + 1): the lanes with bit 3 set of the first change places with
// the lanes with bit 3 clear of the second.
__device__ __forceinline__ void to_fragments(i32x4 (&v)[2]) {
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int a = v[0][c], b = v[1][c];
    v[0][c] = __builtin_amdgcn_update_dpp(a, b, 0x128, 0xf, 0xc, false);  // row_ror:8 into lanes 8..15 of every 16
    v[1][c] = __builtin_amdgcn_update_dpp(b, a, 0x128, 0xf, 0x3, false);  // ... into lanes 0..7
  }
}

template <Elem T>
__device__ __forceinline__ f32x4 mfma_line(const i32x4 (&w)[2], const i32x4 (&x)[2], f32x4 acc) {
  if constexpr (is_fp8(T)) {
    const i32x8 wa = {w[0][0], w[0][1], w[0][2], w[0][3], w[1][0], w[1][1], w[1][2], w[1][3]};
    const i32x8 xa = {x[0][0], x[0][1], x[0][2], x[0][3], x[1][0], x[1][1], x[1][2], x[1][3]};
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wa, xa, acc, 0, 0, 0, 0, 0, 0);
  } else {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if constexpr (T == Elem::F16)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w[h]), __builtin_bit_cast(f16x8, x[h]), acc, 0, 0, 0);
      else
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[h]), __builtin_bit_cast(bf16x8, x[h]), acc, 0, 0, 0);
    }
    return acc;
  }
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void *base, int64_t bytes) {
  const uint32_t n = bytes > 0xffffffffll ? 0xffffffffu : static_cast<uint32_t>(bytes < 0 ? 0 : bytes);
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, static_cast<int>(n), 0x00020000);
}

template <int AUX>
__device__ __forceinline__ i32x4 load16(__amdgpu_buffer_rsrc_t r, uint32_t voff, int soff) {
  return __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(voff), soff, AUX));
}

#endif  // __HIP_DEVICE_COMPILE__

}  // namespace
}  // namespace fluxmi
