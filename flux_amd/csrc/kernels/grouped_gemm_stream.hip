// Grouped GEMM for few rows per expert (decoding, small batches): D[r,:] = scale(r,:) * A[gather(r),:] @ B[e(r)]^T.
//
// Bound by HBM: every weight is read once and used for a handful of rows.  What that needs is bytes in flight on every
// compute unit all the time (about 50 KB each to cover the memory latency at the card's read rate), not operand reuse,
// so the shape of this kernel is the opposite of the macro-tile kernel's (grouped_gemm_kernel.hpp):
//
//  * A workgroup computes 16 * NB columns of up to 32 rows of one expert over the whole of K; its waves split K
//    between them by 128-byte lines (wave w takes lines w, w + WAVES, ...), so that the workgroup reads each row of
//    weights front to back.  The partial sums meet in LDS at the end and are added in wave order (same bits every run).
//  * Operands go from memory straight into registers, eight whole 128-byte lines per load instruction, non-temporally for the
//    weights.  A read-only probe of this access (0.94 GB, rows of 2 to 28 KiB): whole lines 6.7-7.1 TB/s non-temporally and
//    6.1-6.6 with ordinary loads; the MFMA fragment layout itself (16 rows x 64 bytes per instruction, the two halves of a
//    line in two instructions) 4.9-5.5 and 5.9-6.5; 1 KiB of one row per instruction 3.3-6.7.  Two loads become two
//    fragments by exchanging lanes 8..15 of every 16 with lanes 0..7 (three register moves per four bytes and lane).
//  * No barriers and no waits between waves in the loop; a ring of two lines per wave is in flight (128 KiB of weights per
//    compute unit), several workgroups share a compute unit.
//  * Rows beyond the expert's last repeat it (their lanes hit the same lines) and are not stored; bytes past the end of K
//    are out-of-range buffer loads, which return zeros.
//  * The items (expert, column tile, chunk of 32 rows) are numbered with the chunks of one column tile next to each other, and
//    each XCD takes a contiguous eighth of them: weights that several chunks share and the rows of an expert are fetched into
//    few L2s.
//
// Which launches.  Where (nearly) every expert's rows are one chunk, every weight is read once, the items take about the same
// time and the XCDs' shares are even.  The form once took any splits with few rows on average, in chunks of up to 64 rows: under
// a skewed routing one XCD had the long items and a busy expert's weights were read once per chunk.  So launches in which an
// expert can have more than one chunk are launched in both forms and the splits decide (stream_chunks_limit): this form up to a
// quarter more chunks than experts with rows, and none more with under 16 experts, where one more can be a whole round of the
// card (8 experts 4096 x 14336, 10 chunks 241 us, macro tiles 219).  The launch that returns at once costs 2 to 4 us when it is
// the macro tiles' and 3 to 10 when it is this form's.  us per launch, any splits / now / macro tiles: Zipf (exponent 1.2), fp8 32
// experts 7168 x 2048, 512 and 768 rows 154 / 124 / 125 and 165 / 124 / 115; block-scaled, 256 and 512 rows 175 / 117 / 156 and
// 214 / 129 / 159; bf16 64 experts 1408 x 2048, 512 rows 90 / 87 / 123; all 768 rows on eight of the 32 72 / 42 / 33, on
// one 62 / 34 / 24.
//
// The panel tiles (grouped_gemm_panel.hip) take most launches that this form could compute as well, with the same sums; plan_panel says
// which stay here: up to four rows per expert, few columns at long K, and up to 16 rows per expert in many columns of rows a multiple of
// 4 KiB apart, and fewer than 64 columns.
//
// Measured (us per launch, the macro tiles -> this form; weights at 6.5 TB/s in brackets; with more rows than that by runs without the
// panel tiles), even splits, bf16 8 experts 14336 x
// 4096: 64 rows 216 -> 138 [145], 128 rows 216 -> 141, 256 rows 218 -> 165; 4096 x 14336: 64 rows 212 -> 145 [145], 256 rows
// 218 -> 165; 64 experts 1408 x 2048, 256 rows: 113 -> 57 [57], 2048 rows 116 -> 78; fp8 32 experts 2048 x 7168, 256 rows:
// 94 -> 72 [72], 768 rows 96 -> 82; 7168 x 2048: 115 -> 80 [72] and 118 -> 98; block-scaled, the same four: 123 -> 74,
// 125 -> 83, 148 -> 85 and 152 -> 104.
#include "grouped_gemm_rows.hpp"

namespace fluxmi {
namespace {

#if defined(__HIP_DEVICE_COMPILE__)

template <Elem T, int MB, int NB>
struct Line {  // one 128-byte line of every row of the wave's operand blocks, as loaded
  i32x4 w[NB][2], x[MB][2];
  float as[MB], bs;
};

// 16 * MB rows x 16 * NB columns of one expert: partial sums of this wave's lines of K into acc.
template <Elem T, int MB, int NB, int WAVES>
__device__ __forceinline__ void accumulate_tile(const GemmParams &p, const WorkItem &t, int g, int n0, int wave, f32x4 (&acc)[MB][NB]) {
  const int lane = threadIdx.x & 63;
  const int64_t kbytes = static_cast<int64_t>(p.k) * (is_fp8(T) ? 1 : 2);
  const int kb32 = static_cast<int>(kbytes);
  // Lane l of a load fetches 16 bytes of row l & 7 of an eight-row block, chunk 2 * (l >> 4) + ((l >> 3) & 1) of the line.
  const int cbyte = (lane >> 4) * 32 + ((lane >> 3) & 1) * 16;
  const auto wr = buffer_of(p.b[g] + (static_cast<int64_t>(t.e) * p.n + n0) * kbytes, static_cast<int64_t>(p.n - n0) * kbytes);
  const bool gathered = p.gather_a != nullptr;
  const auto xr = gathered ? buffer_of(p.a, static_cast<int64_t>(p.a_rows) * kbytes)
                           : buffer_of(p.a + static_cast<int64_t>(t.row_base) * kbytes, static_cast<int64_t>(t.rows) * kbytes);
  uint32_t woff[NB][2], xoff[MB][2];
#pragma unroll
  for (int j = 0; j < NB; ++j)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      int r = j * 16 + h * 8 + (lane & 7);
      if (r > p.n - n0 - 1) r = p.n - n0 - 1;
      woff[j][h] = static_cast<uint32_t>(r * kbytes) + cbyte;
    }
  auto source_row = [&](int r) {  // row of A that row r of the chunk reads (the last one again past the end)
    if (r > t.rows - 1) r = t.rows - 1;
    if (!gathered) return static_cast<int64_t>(r);
    const int64_t arow = p.gather_a[t.row_base + r];
    return arow < 0 ? 0 : (arow >= p.a_rows ? p.a_rows - 1 : arow);
  };
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h) xoff[i][h] = static_cast<uint32_t>(source_row(i * 16 + h * 8 + (lane & 7)) * kbytes) + cbyte;
  __amdgpu_buffer_rsrc_t sr = xr;
  uint32_t soff[MB];
  int a_kstep = 0, b_base = 0, b_kstep = 0;
  const int kblocks = p.k >> 7;
  if constexpr (T == Elem::FP8_BLOCKSCALED) {
    sr = buffer_of(p.a_scale, 0xffffffffll);
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int r = i * 16 + (lane & 15);
      const int64_t srow = source_row(r) + (gathered ? 0 : t.row_base);
      soff[i] = p.a_scale_layout == FLUXMI_ASCALE_BLOCK128
                    ? static_cast<uint32_t>(((srow >> 7) * kblocks * 128 + (srow & 127)) * 4)
                    : static_cast<uint32_t>((static_cast<int64_t>(t.expert_base) * (kblocks - 1) + srow) * 4);
    }
    a_kstep = p.a_scale_layout == FLUXMI_ASCALE_BLOCK128 ? 512 : t.expert_rows * 4;
    const int nb = n0 >> 7, nblocks = (p.n + 127) >> 7;
    b_base = p.b_scale_layout == FLUXMI_BSCALE_N_K ? (t.e * nblocks + nb) * kblocks : t.e * kblocks * nblocks + nb;
    b_kstep = p.b_scale_layout == FLUXMI_BSCALE_N_K ? 1 : nblocks;
  }

  constexpr int DEPTH = 2;
  Line<T, MB, NB> ring[DEPTH];
  auto load_line = [&](Line<T, MB, NB> &l, int line) {
    const int kb = line * 128;
    const bool ok = kb + cbyte < kb32;
    const int ks = kb < kb32 ? kb : 0;
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) l.w[j][h] = load16<2>(wr, ok ? woff[j][h] : kOutOfRange, ks);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) l.x[i][h] = load16<0>(xr, ok ? xoff[i][h] : kOutOfRange, ks);
    if constexpr (T == Elem::FP8_BLOCKSCALED) {
      const int kblk = line < kblocks ? line : 0;
#pragma unroll
      for (int i = 0; i < MB; ++i)
        l.as[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(sr, static_cast<int>(soff[i]), kblk * a_kstep, 0));
      l.bs = p.b_scale[b_base + kblk * b_kstep];
    }
  };
  auto use_line = [&](Line<T, MB, NB> &l, int line) {
#pragma unroll
    for (int j = 0; j < NB; ++j) to_fragments(l.w[j]);
#pragma unroll
    for (int i = 0; i < MB; ++i) to_fragments(l.x[i]);
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      if constexpr (T == Elem::FP8_BLOCKSCALED) {
        // A line past K has zero operands and the scales of block 0, whose product may be infinite: 0 * inf is not 0.
        const float s = line < kblocks ? l.as[i] * l.bs : 0.f;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const f32x4 b = mfma_line<T>(l.w[j], l.x[i], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
          for (int v = 0; v < 4; ++v) acc[i][j][v] = fmaf(b[v], s, acc[i][j][v]);
        }
      } else {
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = mfma_line<T>(l.w[j], l.x[i], acc[i][j]);
      }
    }
  };
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int lines = static_cast<int>((kbytes + 127) >> 7);
  const int steps = (lines + WAVES - 1) / WAVES;
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    load_line(ring[d], d * WAVES + wave);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int s = 0; s < steps; s += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      use_line(ring[d], (s + d) * WAVES + wave);
      __builtin_amdgcn_sched_barrier(0);
      load_line(ring[d], (s + d + DEPTH) * WAVES + wave);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// Partial sums of one wave's lines of K to LDS.
template <Elem T, int MB, int NB, int WAVES>
__device__ __forceinline__ void partial_sums(const GemmParams &p, f32x4 *red, const WorkItem &t, int g, int n0, int wave) {
  f32x4 acc[MB][NB];
  accumulate_tile<T, MB, NB, WAVES>(p, t, g, n0, wave, acc);
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) red[(wave * MB * NB + i * NB + j) * 64 + lane] = acc[i][j];
}

// Sum of the waves' partial sums, scaled, cast and stored.  A unit is one lane's four consecutive columns of one row.
template <Elem T, int MB, int NB, int WAVES>
__device__ __forceinline__ void finish_tile(const GemmParams &p, const FewRowsArgs &few, const f32x4 *red, const WorkItem &t, int g, int n0, int wave) {
  const int lane = threadIdx.x & 63;
  const float tile_scale = p.scalar * (p.scalar_dev ? p.scalar_dev[0] : 1.f) * (p.alpha[g] ? p.alpha[g][t.e] : 1.f);
  for (int u = wave * 64 + lane; u < MB * NB * 64; u += WAVES * 64) {
    f32x4 v = red[u];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) v += red[w * MB * NB * 64 + u];
    const int l = u & 63, b = u >> 6;
    const int r = (b / NB) * 16 + (l & 15), col = n0 + (b % NB) * 16 + (l >> 4) * 4;
    if (r >= t.rows || col >= p.n) continue;  // n % 4 == 0: the four columns are all in or all out
    const int row = t.row_base + r;
    const float rs = row_factor(p, few, tile_scale, row);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      v[c] *= rs;
      if (p.col_scale) v[c] *= p.col_scale[static_cast<int64_t>(t.e) * p.n + col + c];
    }
    int64_t drow = row;
    if (p.scatter_d) {
      drow = p.scatter_d[row];
      if (drow < 0 || drow >= p.d_rows) continue;
    }
    const int64_t at = drow * p.n + col;
    if (p.accumulate) {
#pragma unroll
      for (int c = 0; c < 4; ++c) unsafeAtomicAdd(static_cast<float *>(p.d[g]) + at + c, v[c]);
    } else if (p.d_fp32) {
      *reinterpret_cast<f32x4 *>(static_cast<float *>(p.d[g]) + at) = v;
    } else {
      u32x2 o;
#pragma unroll
      for (int c = 0; c < 2; ++c)
        o[c] = T == Elem::F16 ? static_cast<uint32_t>(float_to_f16_bits(v[2 * c])) | (static_cast<uint32_t>(float_to_f16_bits(v[2 * c + 1])) << 16)
                              : static_cast<uint32_t>(float_to_bf16_bits(v[2 * c])) | (static_cast<uint32_t>(float_to_bf16_bits(v[2 * c + 1])) << 16);
      *reinterpret_cast<u32x2 *>(static_cast<uint16_t *>(p.d[g]) + at) = o;
    }
  }
}

#endif  // __HIP_DEVICE_COMPILE__


// WALK: a workgroup per compute unit that walks the `blocks` items with the grid's stride, as many at a time as the unit holds
// workgroups of the other form (its teams of WAVES waves); otherwise one workgroup per item.  Two forms because the loop costs
// registers (the 32-column fp8 and block-scaled ones spill 4 to 9 with it).
constexpr int unit_waves(int nb) { return nb <= 2 ? 16 : 8; }  // what the registers of a compute unit hold
template <Elem T, int NB, int WAVES, bool WALK>
__global__ __launch_bounds__(WALK ? unit_waves(NB) * 64 : WAVES * 64) __attribute__((amdgpu_waves_per_eu(unit_waves(NB) / 4)))
void grouped_gemm_stream_kernel(const FewRowsArgs few, const GemmParams p, const int blocks) {
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int TEAMS = WALK ? unit_waves(NB) / WAVES : 1;
  constexpr int TEAM_SUMS = WAVES * 2 * NB * 64;
  __shared__ f32x4 red_all[TEAMS * TEAM_SUMS];
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int team = TEAMS > 1 ? wave_all / WAVES : 0, wave = TEAMS > 1 ? wave_all % WAVES : wave_all;
  f32x4 *const red = red_all + team * TEAM_SUMS;
  const int tiles_n1 = (p.n + 16 * NB - 1) / (16 * NB);
  const int stride = static_cast<int>(gridDim.x);
  int block = blockIdx.x;
  do {
    const WorkItem t = locate<T>(p, tiles_n1 * p.ngroups, kStreamRows, block + team * stride);
    const int g = p.ngroups > 1 ? t.nt / tiles_n1 : 0;
    const int n0 = (t.nt - g * tiles_n1) * (16 * NB);
    if constexpr (!WALK) {
      if (t.rows == 0) return;
    }
    if (t.rows > 16) partial_sums<T, 2, NB, WAVES>(p, red, t, g, n0, wave);
    else if (t.rows > 0) partial_sums<T, 1, NB, WAVES>(p, red, t, g, n0, wave);
    __syncthreads();
    if (t.rows > 16) finish_tile<T, 2, NB, WAVES>(p, few, red, t, g, n0, wave);
    else if (t.rows > 0) finish_tile<T, 1, NB, WAVES>(p, few, red, t, g, n0, wave);
    if constexpr (WALK) __syncthreads();  // the sums have been read before the next items' go there
    block += TEAMS * stride;
  } while (WALK && block < blocks);
#endif
}

// Items of a launch in which every expert that can get rows is one per column tile of 16 * nb, and the most items a launch of
// this form can have.
int64_t one_chunk_items(const GemmParams &p, int ngroups, int nb) {
  const int64_t active = p.nexperts < p.max_rows ? p.nexperts : p.max_rows;
  return active * ((p.n + 16 * nb - 1) / (16 * nb)) * ngroups;
}
int64_t most_items(const GemmParams &p, int ngroups, int nb) {
  const int active = p.nexperts < p.max_rows ? p.nexperts : p.max_rows;
  const int chunks = active + (p.max_rows - active) / kStreamRows, limit = stream_chunks_limit(active, kStreamRows, false, 0, 0);
  return static_cast<int64_t>(chunks < limit ? chunks : limit) * ((p.n + 16 * nb - 1) / (16 * nb)) * ngroups;
}

// A walking workgroup's sums take 64 KiB of LDS; with what it asks for on top that is more than half of a compute unit's
// 160 KiB, so no unit takes two of them and N workgroups occupy N units.
constexpr int kWalkSums = 64 * 1024, kWalkExtra = 32 * 1024;

template <Elem T, int NB, int WAVES>
void launch(const GemmParams &p, const FewRowsArgs &few, const StreamPlan &plan, hipStream_t s) {
  if (!plan.walk) {
    hipLaunchKernelGGL((grouped_gemm_stream_kernel<T, NB, WAVES, false>), dim3(plan.workgroups), dim3(WAVES * 64), 0, s, few, p, plan.blocks);
    return;
  }
  static_assert(unit_waves(NB) * 2 * NB * 1024 == kWalkSums, "LDS of the walking form");
  hipLaunchKernelGGL((grouped_gemm_stream_kernel<T, NB, WAVES, true>), dim3(plan.workgroups), dim3(unit_waves(NB) * 64), kWalkExtra, s, few, p, plan.blocks);
}

template <Elem T>
void launch_by_plan(const GemmParams &p, const FewRowsArgs &few, const StreamPlan &plan, hipStream_t s) {
  if (plan.waves == 8 && plan.cols == 32) launch<T, 2, 8>(p, few, plan, s);
  else if (plan.waves == 8) launch<T, 4, 8>(p, few, plan, s);
  else if (plan.cols == 32) launch<T, 2, 4>(p, few, plan, s);
  else launch<T, 4, 4>(p, few, plan, s);
}

}  // namespace

// Up to how many rows per expert on average this form is faster than the macro tiles on even splits (plan_panel has the line between it and
// the panel tiles, which up to here sum K as this form does; the macro tiles' time hardly depends on
// the rows while they are few; this one's grows with them): 16-bit at 32 rows 165 / 218 us on the two 8-expert shapes above,
// 78 / 116 and 80 / 92 on 64 experts of 1408 x 2048 and 2048 x 1408, 12 / 19 on 8 of 2048 x 1024; fp8 at 24 rows 82 / 96 and 98 /
// 118, at 32 an earlier build 95 / 97 and 128 / 118; block-scaled at 24 rows 83 / 125 and 104 / 152.  Items are numbered with ints
// (for the most weight groups a launch can have, so that their number does not choose the form).
bool grouped_gemm_stream_takes(const GemmParams &p, int dtype) {
  const int64_t rows = dtype == FLUXMI_FP8_E4M3 ? 24 : kStreamRows;
  return p.max_rows <= rows * p.nexperts && most_items(p, kMaxWeightGroups, 2) < (int64_t{1} << 31) - (1 << 20);
}

int stream_waves(const GemmParams &p, int dtype) {
  const int64_t lines = (static_cast<int64_t>(p.k) * (dtype == FLUXMI_FP8_E4M3 ? 1 : 2) + 127) / 128;
  return one_chunk_items(p, 1, 4) < 512 && lines >= 64 ? 8 : 4;
}

// Columns per workgroup: 64 reads the rows' own operand least often (its loads share the queue behind the weights' with them), but
// takes two waves per SIMD; 32 columns with four waves per SIMD is as fast or faster on most shapes while there is hardly a row (us at
// 2 rows per expert, 32 / 64 columns: bf16 4096 x 14336 140 / 143, 64 experts of 1408 x 2048 59 / 66, fp8 7168 x 2048
// 77 / 80; not on 8 experts of 14336 x 4096, 158 / 136).  Block-scaled launches differ by 1 to 4 us either way and take 64.  Where
// 64-column tiles would leave compute units without work (512 of them fill the card) it is 32 columns, and eight waves per
// workgroup if K is long enough to share (two experts, 4096 x 14336: 42 us, four waves 47, 64 columns 61; at K = 2048 bytes per row
// eight waves lose, 17 against 14 us).
// With compute units to be left to other work there is one workgroup for each of the others, which walks several items; the results
// do not change, which is why a margin does not choose the macro tiles either where those are faster.  us at a margin of 8 / 64 / 128
// / 224 of 256 units, this form and the macro tiles: bf16 8 experts 14336 x 4096, 74 rows 162 / 185 / 255 / 995 and 215 / 238 / 268 /
// 773; fp8 32 experts 7168 x 2048, 400 rows 97 / 118 / 168 / 642 and 111 / 120 / 147 / 500 (a unit alone streams 30 GB/s here; a
// ring of three or four lines in place of two changed nothing).
StreamPlan plan_grouped_gemm_stream(const GemmParams &p, int dtype, int cus, bool leave_cus) {
  StreamPlan plan;
  const bool few = one_chunk_items(p, p.ngroups, 4) < 512;
  plan.waves = stream_waves(p, dtype);
  plan.cols = few || (p.a_scale == nullptr && p.max_rows <= 4 * p.nexperts) ? 32 : 64;
  const int64_t blocks = (most_items(p, p.ngroups, plan.cols / 16) + 7) / 8 * 8;
  plan.blocks = static_cast<int>(blocks);
  plan.walk = leave_cus || blocks * plan.waves * 64 > 0xffffffffll;  // a launch has less than 2^32 threads
  const int64_t most = cus >= 8 ? cus / 8 * 8 : cus;  // whole rounds over the XCDs where there are enough units
  plan.workgroups = static_cast<unsigned>(plan.walk && blocks > most ? most : blocks);
  plan.lds_bytes = plan.walk ? kWalkSums + kWalkExtra : plan.waves * 2 * (plan.cols / 16) * 1024;
  return plan;
}

void launch_grouped_gemm_stream(const GemmParams &p, const FewRowsArgs &few, int dtype, const StreamPlan &plan, hipStream_t s) {
  if (p.a_scale != nullptr) launch_by_plan<Elem::FP8_BLOCKSCALED>(p, few, plan, s);
  else if (dtype == FLUXMI_FP8_E4M3) launch_by_plan<Elem::FP8>(p, few, plan, s);
  else if (dtype == FLUXMI_FP16) launch_by_plan<Elem::F16>(p, few, plan, s);
  else launch_by_plan<Elem::BF16>(p, few, plan, s);
}

}  // namespace fluxmi
