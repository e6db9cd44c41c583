// Grouped GEMM entry point: argument checks, choice between the MFMA kernels and the generic kernel, and
// the generic kernel itself.  The MFMA kernels are the macro tiles (grouped_gemm_kernel.hpp), the dual tiles of the same size
// (grouped_gemm_dual.hip) and, for few rows per expert, the panel tiles (grouped_gemm_panel.hip) and the streaming form
// (grouped_gemm_stream.hip).
#include "grouped_gemm_dual.hpp"
#include "grouped_gemm_panel.hpp"
#include "grouped_gemm_stream.hpp"

namespace fluxmi {
namespace {

// ---- generic kernel: any K / N, no alignment demands beyond element size -------------------------
// One thread per output element, a wave covers 64 consecutive columns of one row.  Only used when the
// MFMA kernel's shape requirements do not hold.
__device__ __forceinline__ float e4m3_to_float(uint8_t b) {
  const uint32_t sign = (b & 0x80u) << 24;
  const uint32_t em = b & 0x7fu;
  if (em == 0x7fu) return __uint_as_float(sign | 0x7fc00000u);
  if (em < 8u) return __uint_as_float(sign) + (sign ? -1.f : 1.f) * static_cast<float>(em) * 0x1p-9f;
  return __uint_as_float(sign | ((em + (120u << 3)) << 20));
}

template <int ELT>
__global__ __launch_bounds__(256) void grouped_gemm_generic_kernel(const GemmParams p, const int g) {
  __shared__ int32_t s_row_off[kMaxExperts + 1];
  if (threadIdx.x == 0) {
    int acc = 0;
    for (int e = 0; e < p.nexperts; ++e) {
      s_row_off[e] = acc;
      const int v = p.splits[e];
      acc += v > 0 ? v : 0;
    }
    s_row_off[p.nexperts] = acc;
  }
  __syncthreads();
  const int total_rows = s_row_off[p.nexperts] < p.max_rows ? s_row_off[p.nexperts] : p.max_rows;
  float scalar = p.scalar;
  if (p.scalar_dev) scalar *= p.scalar_dev[0];
  const int ncol_blocks = (p.n + 255) / 256;
  for (int64_t item = blockIdx.x; item < static_cast<int64_t>(total_rows) * ncol_blocks;
       item += gridDim.x) {
    const int r = static_cast<int>(item / ncol_blocks);
    const int n = static_cast<int>(item % ncol_blocks) * 256 + threadIdx.x;
    int e = 0;
    while (r >= s_row_off[e + 1]) ++e;
    if (n >= p.n) continue;
    int64_t arow = r;
    if (p.gather_a) {
      arow = p.gather_a[r];
      if (p.a_rows > 0) arow = arow < 0 ? 0 : (arow >= p.a_rows ? p.a_rows - 1 : arow);
    }
    const uint8_t *ap = p.a + arow * p.k * ELT;
    const uint8_t *bp = p.b[g] + (static_cast<int64_t>(e) * p.n + n) * p.k * ELT;
    float acc = 0.f, total = 0.f;
    const int kblocks = p.k / 128;
    for (int kk = 0; kk < p.k; ++kk) {
      float av, bv;
      if (ELT == 2) {
        const uint16_t ab = reinterpret_cast<const uint16_t *>(ap)[kk], bb = reinterpret_cast<const uint16_t *>(bp)[kk];
        av = p.half_is_f16 ? f16_bits_to_float(ab) : bf16_bits_to_float(ab);
        bv = p.half_is_f16 ? f16_bits_to_float(bb) : bf16_bits_to_float(bb);
      } else {
        av = e4m3_to_float(ap[kk]);
        bv = e4m3_to_float(bp[kk]);
      }
      acc = fmaf(av, bv, acc);
      if (p.a_scale != nullptr && (kk & 127) == 127) {  // end of a scale block of K: promote
        const int kb = kk >> 7, nb = n >> 7, nblocks = (p.n + 127) >> 7;
        const float as = p.a_scale_layout == FLUXMI_ASCALE_BLOCK128
                             ? p.a_scale[((arow >> 7) * kblocks + kb) * 128 + (arow & 127)]
                             : p.a_scale[static_cast<int64_t>(s_row_off[e]) * kblocks +
                                         static_cast<int64_t>(kb) * (s_row_off[e + 1] - s_row_off[e]) + (r - s_row_off[e])];
        const float bs = p.b_scale_layout == FLUXMI_BSCALE_N_K
                             ? p.b_scale[(static_cast<int64_t>(e) * nblocks + nb) * kblocks + kb]
                             : p.b_scale_layout == FLUXMI_BSCALE_K_N
                                   ? p.b_scale[(static_cast<int64_t>(e) * kblocks + kb) * nblocks + nb]
                                   : p.b_scale[((static_cast<int64_t>(e) * nblocks + nb) * kblocks + kb) * 128 + (n & 127)];
        total = fmaf(acc, as * bs, total);
        acc = 0.f;
      }
    }
    if (p.a_scale != nullptr) acc = total;
    float v = acc * scalar * (p.alpha[g] ? p.alpha[g][e] : 1.f) * (p.row_scale ? p.row_scale[r] : 1.f);
    if (p.col_scale) v *= p.col_scale[static_cast<int64_t>(e) * p.n + n];
    int64_t drow = r;
    if (p.scatter_d) {
      drow = p.scatter_d[r];
      if (drow < 0 || drow >= p.d_rows) continue;
    }
    if (p.accumulate) unsafeAtomicAdd(static_cast<float *>(p.d[g]) + drow * p.n + n, v);
    else if (p.d_fp32) static_cast<float *>(p.d[g])[drow * p.n + n] = v;
    else static_cast<uint16_t *>(p.d[g])[drow * p.n + n] = p.half_is_f16 ? float_to_f16_bits(v) : float_to_bf16_bits(v);
  }
}

// Shapes the MFMA kernel takes: rows of K a multiple of 16 bytes (K % 8 == 0 for bf16, K % 16 == 0 for fp8),
// N a multiple of 4, aligned pointers, and operands its 32-bit buffer offsets can span (a gathered A as a
// whole, which needs its extent a_rows; 256 rows of an ungathered A; one expert's weights).  Everything else
// runs the generic kernel.
bool mfma_path_ok(const fluxmi_grouped_gemm_args *a, const void *b, const void *d, bool d_is_fp32) {
  const int elt = a->dtype == FLUXMI_FP8_E4M3 ? 1 : 2;
  const int64_t kbytes = static_cast<int64_t>(a->k) * elt;
  const int64_t span = 0xffffffffll;
  const bool a_fits = a->gather_a ? (a->a_rows > 0 && a->a_rows * kbytes <= span) : BM * kbytes <= span;
  return kbytes % 16 == 0 && kbytes >= 16 && a->n % 4 == 0 && aligned16(a->a) &&
         aligned16(b) && (reinterpret_cast<uintptr_t>(d) & (d_is_fp32 ? 15u : 7u)) == 0 &&
         (a->col_scale == nullptr || aligned16(a->col_scale)) && a_fits && a->n * kbytes <= span;
}

}  // namespace
}  // namespace fluxmi

extern "C" size_t fluxmi_grouped_gemm_workspace_bytes(const fluxmi_grouped_gemm_args *) { return 0; }

namespace fluxmi {
namespace {

struct BlockScales {
  const float *a_scale = nullptr, *b_scale = nullptr;
  int32_t a_layout = 0, b_layout = 0;
};

// What a launch would be, without launching it; cus: the compute units of the device it is asked for.
struct DryRun {
  int cus = 0;
  bool stream = false, macro = false, dual = false;
  StreamPlan plan = {};
  PanelPlan panel = {};
};

// Chunks of up to chunk_rows rows of a launch with these splits, and the experts that have rows.
int count_chunks(const fluxmi_grouped_gemm_args *args, const int32_t *splits_host, int chunk_rows, int &active) {
  int left = args->max_rows, chunks = 0;
  active = 0;
  for (int e = 0; e < args->nexperts; ++e) {
    const int rows = splits_host[e] < 0 ? 0 : (splits_host[e] < left ? splits_host[e] : left);
    left -= rows;
    active += rows > 0 ? 1 : 0;
    chunks += (rows + chunk_rows - 1) / chunk_rows;
  }
  return chunks;
}

// Whether a form for few rows per expert, with chunks of chunk_rows rows, computes a launch with these splits.
bool few_chunks(const fluxmi_grouped_gemm_args *args, const int32_t *splits_host, int chunk_rows, const PanelPlan &panel) {
  int active;
  const int chunks = count_chunks(args, splits_host, chunk_rows, active);
  return chunks <= stream_chunks_limit(active, chunk_rows, args->dtype == FLUXMI_FP8_E4M3, panel.chunk_items, panel.round_items);
}

// Launches that leave most of the dual tiles' waves or phases without work; tiles: the most that a launch can have.  Dual tiles against macro
// tiles, both with up to four workgroups to a tile, in the mean, and launches slower by more than 3 %; where macro tiles had one workgroup to
// a tile, before the dual tiles were there, is the third figure:
//   up to 128 columns, up to 128 tiles, rows of K of 1 KiB and more   0.73, 88 %; 0.94  (5 experts 32 x 12672, 104 rows each: fp8 90 us, 42, 36)
//     the same with shorter K                                         1.16,  9 %; 1.27, taken
//     129 to 256 tiles, K of 4 KiB and more                           1.02,  9 %; 1.06  (bf16 107 experts 32 x 5888, 118 rows each 86 us, 58, 59)
//     the same with shorter K                                         1.27,  1 %; 1.29, taken
//     block-scaled, up to 128 tiles, any K                            0.99, 16 %; 1.29  (3 experts 88 x 896, 64 rows each: 16.2 us; before 11.5)
//     block-scaled, 129 to 256 tiles, rows of K of 1 KiB and more     0.97, 58 %; 1.29
//   block-scaled, few rows that no form for few rows takes (columns not in 64s):
//     R up to 64, up to 128 tiles                                     0.65, 99 %; 1.01  (one expert 1904 x 13696, 51 rows: 112 us, 46, 86)
//                 129 to 256 tiles                                    1.02, 26 %; 1.09, taken
//                 257 to 448 tiles                                    1.00, 43 %; 0.99
//     R up to 96, more than 256 tiles, K of 4 KiB and more            1.00, 38 %; 1.00  (shorter K 1.12,  5 %; 1.12, taken)
bool dual_tiles_idle(const fluxmi_grouped_gemm_args *args, bool block_scaled, int64_t kbytes, int64_t tiles) {
  auto at_most = [&](int64_t rows) { return args->max_rows <= rows * args->nexperts; };
  if (args->n <= 128 && tiles <= 128 && (block_scaled || kbytes >= 1024)) return true;
  if (args->n <= 128 && tiles <= 256 && kbytes >= (block_scaled ? 1024 : 4096)) return true;
  if (!block_scaled) return false;
  return (at_most(64) && (tiles <= 128 || (tiles > 256 && tiles <= 448))) || (at_most(96) && tiles > 256 && kbytes >= 4096);
}

// Whether the dual tiles are the faster ones for a launch that the macro tiles would compute.  Speed against the macro tiles in the mean, and how
// many launches are slower by more than 3 %: 19125 launches of 1 to 128 experts with more than 128 tiles, R = 97 to 4000 rows each on average,
// rows of K of 0.5 to 28 KiB, even, random and Zipf row counts, plain and scaled, gathered and not, weights not in the cache.  fp32 results have
// lines of their own: a tile's stores drain ahead of the next tile's fills, and these are twice as many.
//                                         16-bit results                      fp32 results
//   16 bits  R up to 320                  1.20,  2 %                          1.16,  3 %
//            R up to 512, K < 6 KiB       1.17,  1 %                          1.09,  5 %
//            more rows, K < 1 KiB         1.42,  none                         1.27,  none
//                       K < 2 KiB         1.20,  none                         R up to 1500 1.15,  3 %; more 1.09, 14 %: not taken
//                       K < 3 KiB         1.12,  none                         R up to 1024 1.06, 10 %; more 1.02, 25 %: not taken
//                       K < 4 KiB         R up to 768 1.09, 2 %; 1.06, 5 %    1.02, 21 %: not taken
//            the rest                     1.00, 34 %: not taken               0.99, 44 %: not taken
//   fp8      R up to 512                  1.20,  2 %                          1.16,  4 %
//            more rows, K < 1 KiB         1.30,  none                         1.19,  6 %
//                       K < 2 KiB         1.15,  none                         R up to 1500 1.09,  6 %; more 1.05, 19 %: not taken
//                       K < 3 KiB         1.07,  4 %                          R up to 1024 1.05, 11 %; more 1.03, 15 %: not taken
//                       K < 4 KiB         R up to 1024 1.05, 9 %; 1.03, 13 %  1.02, 20 %: not taken
//            the rest                     1.00, 30 %: not taken               0.99, 38 %: not taken
//   block-scaled                          1.21,  2 %                          1.12,  5 %; of these with K < 1 KiB, more than 1024 columns and 256
//                                                                             rows, up to 512 tiles 1.02, 31 %, taken: the macro tiles are no safer
// Launches of fewer tiles, which both forms cut into pieces, are not told apart here: up to 192 rows 0.92 to 1.06, more rows 0.74 to 1.14, so the
// macro tiles would be the faster ones for many.  None of them loses against macro tiles with one workgroup to a tile (1.28 to 1.49 in the mean).
// The flags of the fill forms name forms of the macro tiles.
bool dual_is_faster(const fluxmi_grouped_gemm_args *args, bool block_scaled, bool by_splits, int64_t tiles) {
  const bool fp8 = args->dtype == FLUXMI_FP8_E4M3;
  const int64_t kbytes = static_cast<int64_t>(args->k) * (fp8 ? 1 : 2);
  if (!by_splits && dual_tiles_idle(args, block_scaled, kbytes, tiles)) return false;
  if (block_scaled) return true;
  if ((args->sched_flags & (FLUXMI_SCHED_HALF_LINE_FILLS | FLUXMI_SCHED_WHOLE_LINE_FILLS)) != 0) return false;
  auto at_most = [&](int64_t rows) { return args->max_rows <= rows * args->nexperts; };
  if (at_most(fp8 ? 512 : 320) || (kbytes < 6144 && at_most(512))) return true;
  if (args->d_fp32 != 0) return kbytes < 1024 || (kbytes < 2048 && at_most(1500)) || (kbytes < 3072 && at_most(1024));
  return kbytes < 3072 || (kbytes < 4096 && at_most(fp8 ? 1024 : 768));
}

// Row counts that are known on the host, and a second factor per row.
struct HostSplits {
  const int32_t *splits;
  const float *row_scale2;
  bool dual;  // the dual tiles take them as well
};

// dry_run: check the arguments and report which kernel would run (1 MFMA, 0 generic) without launching.
// accumulate_rows > 0: D is fp32 with that many rows and results are added to it atomically.
// host: the launch is made for these row counts, one kernel.  Without args->splits that takes a form for few rows per expert that
// computes them; returns 1 if it was launched, otherwise 0.
int run_grouped_gemm(const fluxmi_grouped_gemm_args *args, int ngroups, const void *const *b, void *const *d,
                     const float *const *alpha, void *stream, DryRun *dry_run = nullptr, int32_t accumulate_rows = 0,
                     const BlockScales *bs = nullptr, const HostSplits *host = nullptr) {
  FLUXMI_REQUIRE(args != nullptr, FLUXMI_ERR_INVALID_ARG, "grouped_gemm: null args");
  FLUXMI_REQUIRE(args->dtype == FLUXMI_BF16 || args->dtype == FLUXMI_FP8_E4M3 || args->dtype == FLUXMI_FP16, FLUXMI_ERR_INVALID_ARG,
                 "grouped_gemm: unknown dtype %d", args->dtype);
  FLUXMI_REQUIRE(args->d_fp32 == 0 || args->d_fp32 == 1, FLUXMI_ERR_INVALID_ARG,
                 "grouped_gemm: d_fp32 must be 0 or 1");
  FLUXMI_REQUIRE(args->a_rows >= 0, FLUXMI_ERR_INVALID_ARG, "grouped_gemm: negative a_rows");
  FLUXMI_REQUIRE(args->reserved == 0, FLUXMI_ERR_INVALID_ARG, "grouped_gemm: reserved must be 0, got %d",
                 args->reserved);
  FLUXMI_REQUIRE(args->nexperts >= 1 && args->nexperts <= kMaxExperts, FLUXMI_ERR_UNSUPPORTED,
                 "grouped_gemm: nexperts=%d outside [1,%d]", args->nexperts, kMaxExperts);
  FLUXMI_REQUIRE(args->max_rows >= 0 && args->n >= 0 && args->k >= 0, FLUXMI_ERR_INVALID_ARG,
                 "grouped_gemm: negative size (max_rows=%d, n=%d, k=%d)", args->max_rows, args->n,
                 args->k);
  FLUXMI_REQUIRE(ngroups >= 1 && ngroups <= kMaxWeightGroups, FLUXMI_ERR_UNSUPPORTED,
                 "grouped_gemm: ngroups=%d outside [1,%d]", ngroups, kMaxWeightGroups);
  if (args->max_rows == 0 || args->n == 0) return dry_run || host ? 1 : FLUXMI_OK;
  FLUXMI_REQUIRE(args->k >= 1, FLUXMI_ERR_UNSUPPORTED, "grouped_gemm: k must be positive");
  FLUXMI_REQUIRE(args->a && (args->splits || host) && b && d, FLUXMI_ERR_INVALID_ARG, "grouped_gemm: null a / b / d / splits");

  GemmParams p;
  bool mfma = true;
  for (int g = 0; g < kMaxWeightGroups; ++g) {
    const int src = g < ngroups ? g : 0;
    FLUXMI_REQUIRE(b[src] && d[src], FLUXMI_ERR_INVALID_ARG, "grouped_gemm: null b / d of weight group %d", src);
    p.b[g] = static_cast<const uint8_t *>(b[src]);
    p.d[g] = d[src];
    p.alpha[g] = alpha ? alpha[src] : nullptr;
    mfma = mfma && mfma_path_ok(args, b[src], d[src], accumulate_rows > 0 || args->d_fp32 != 0);
  }
  // The tile schedule numbers the column tiles of all groups with one int.
  mfma = mfma && (static_cast<int64_t>(args->n) + BN) * ngroups < (1ll << 30);
  p.a = static_cast<const uint8_t *>(args->a);
  p.splits = args->splits;
  p.gather_a = args->gather_a;
  p.scatter_d = args->scatter_d;
  p.row_scale = args->row_scale;
  p.col_scale = args->col_scale;
  p.scalar_dev = args->scalar_scale_dev;
  p.scalar = args->scalar_scale;
  p.nexperts = args->nexperts;
  p.max_rows = args->max_rows;
  p.a_rows = args->a_rows;
  p.n = args->n;
  p.k = args->k;
  p.d_fp32 = accumulate_rows > 0 ? 1 : args->d_fp32;
  p.accumulate = accumulate_rows > 0 ? 1 : 0;
  p.d_rows = accumulate_rows > 0 ? accumulate_rows : args->max_rows;
  p.ngroups = ngroups;
  p.half_is_f16 = args->dtype == FLUXMI_FP16 ? 1 : 0;
  p.a_scale = bs ? bs->a_scale : nullptr;
  p.b_scale = bs ? bs->b_scale : nullptr;
  p.a_scale_layout = bs ? bs->a_layout : 0;
  p.b_scale_layout = bs ? bs->b_layout : 0;
  if (bs != nullptr) {
    FLUXMI_REQUIRE(args->dtype == FLUXMI_FP8_E4M3, FLUXMI_ERR_UNSUPPORTED, "grouped_gemm_blockscale: dtype must be fp8 e4m3");
    FLUXMI_REQUIRE(args->k % 128 == 0, FLUXMI_ERR_UNSUPPORTED, "grouped_gemm_blockscale: K=%d is not a multiple of 128", args->k);
    FLUXMI_REQUIRE(bs->a_scale != nullptr && bs->b_scale != nullptr, FLUXMI_ERR_INVALID_ARG,
                   "grouped_gemm_blockscale: null a_scale / b_scale");
    FLUXMI_REQUIRE((bs->a_layout == FLUXMI_ASCALE_BLOCK128 || bs->a_layout == FLUXMI_ASCALE_EXPERT_K_M) &&
                       (bs->b_layout == FLUXMI_BSCALE_N_K || bs->b_layout == FLUXMI_BSCALE_K_N ||
                        bs->b_layout == FLUXMI_BSCALE_COL_N_K),
                   FLUXMI_ERR_INVALID_ARG, "grouped_gemm_blockscale: unknown scale layout (%d, %d)", bs->a_layout, bs->b_layout);
    FLUXMI_REQUIRE(!(bs->a_layout == FLUXMI_ASCALE_EXPERT_K_M && args->gather_a != nullptr), FLUXMI_ERR_INVALID_ARG,
                   "grouped_gemm_blockscale: per-expert a_scale segments cannot be combined with gather_a");
    FLUXMI_REQUIRE(ngroups == 1, FLUXMI_ERR_UNSUPPORTED, "grouped_gemm_blockscale: one weight tensor per launch");
    if (bs->b_layout == FLUXMI_BSCALE_COL_N_K) mfma = false;  // per-column weight scales: the generic kernel only
    // a_scale is addressed with 32-bit byte offsets
    const int64_t srows = args->gather_a ? args->a_rows : args->max_rows;
    mfma = mfma && ((srows + 127) / 128 * 128) * (args->k / 128) * 4 < (int64_t{1} << 32) &&
           (reinterpret_cast<uintptr_t>(bs->a_scale) & 3u) == 0;
  }
  FLUXMI_REQUIRE(args->raster_rows >= 0 && args->raster_rows <= 1024, FLUXMI_ERR_INVALID_ARG,
                 "grouped_gemm: raster_rows=%d outside [0,1024]", args->raster_rows);
  FLUXMI_REQUIRE(args->cu_margin >= 0, FLUXMI_ERR_INVALID_ARG, "grouped_gemm: negative cu_margin");
  FLUXMI_REQUIRE((args->sched_flags & ~(FLUXMI_SCHED_WHOLE_TAIL_TILES | FLUXMI_SCHED_NO_HALF_TILES |
                                        FLUXMI_SCHED_NO_SKINNY_TAIL | FLUXMI_SCHED_FORCE_SKINNY_TAIL | FLUXMI_SCHED_HALF_LINE_FILLS |
                                        FLUXMI_SCHED_WHOLE_LINE_FILLS)) == 0,
                 FLUXMI_ERR_INVALID_ARG, "grouped_gemm: unknown sched_flags 0x%x", args->sched_flags);
  FLUXMI_REQUIRE((args->sched_flags & FLUXMI_SCHED_HALF_LINE_FILLS) == 0 || (args->sched_flags & FLUXMI_SCHED_WHOLE_LINE_FILLS) == 0,
                 FLUXMI_ERR_INVALID_ARG, "grouped_gemm: sched_flags ask for half-line and whole-line fills at once");
  // fp32 outputs beyond half a GB go out non-temporally (measured on a 805 MB intermediate: the GEMM 5 % faster,
  // the reduce that reads it unchanged; at 268 MB the GEMM is unchanged and the reduce 10 % slower).
  p.nt_stores = (args->d_fp32 != 0 && accumulate_rows == 0 && static_cast<int64_t>(args->max_rows) * args->n * 4 > (int64_t{512} << 20)) ? 1 : 0;
  p.raster_rows = args->raster_rows > 0 ? args->raster_rows : 8;
  p.sched_flags = args->sched_flags;

  const bool stream_form = mfma && grouped_gemm_stream_takes(p, args->dtype);
  hipStream_t s = static_cast<hipStream_t>(stream);
  p.by_splits = 0;
  int cus = dry_run ? dry_run->cus : fluxmi_device_cu_count();
  FLUXMI_REQUIRE(cus > 0 || dry_run, FLUXMI_ERR_HIP, "grouped_gemm: cannot query the device");
  // CUs left to other work of the caller (Flux's sm_margin): every MFMA form launches fewer workgroups.
  cus = cus - args->cu_margin > 1 ? cus - args->cu_margin : 1;
  const bool leave_cus = args->cu_margin > 0;
  PanelPlan panel = {};
  if (mfma) panel = plan_panel(p, args->dtype, stream_form, cus, leave_cus);
  const StreamPlan plan = stream_form && panel.cols == 0 ? plan_grouped_gemm_stream(p, args->dtype, cus, leave_cus) : StreamPlan{};
  const bool macro = mfma && !panel.any_splits && (!stream_form || args->max_rows > kStreamRows);
  if (macro) p.by_splits = panel.cols != 0 ? panel.chunk_rows : (stream_form ? kStreamRows : 0);
  p.chunk_items = panel.chunk_items;
  p.round_items = panel.round_items;
  const int64_t tiles_n = (args->n + BN - 1) / BN * ngroups;
  const int64_t max_tiles = (static_cast<int64_t>(args->max_rows) / BM + args->nexperts) * tiles_n;  // whatever the splits
  const bool dual = macro && dual_is_faster(args, bs != nullptr, p.by_splits != 0, max_tiles) && dual_takes(p, args->dtype);
  if (dry_run) {
    dry_run->stream = stream_form;
    dry_run->macro = macro;
    dry_run->dual = dual;
    dry_run->plan = plan;
    dry_run->panel = panel;
    return mfma ? 1 : 0;
  }

  FewRowsArgs few;
  few.count = 0;
  few.row_scale2 = nullptr;
  bool run_few = panel.cols != 0 || stream_form, run_macro = macro;
  if (host != nullptr) {
    const bool computes = run_few && (!macro || few_chunks(args, host->splits, p.by_splits, panel));
    p.by_splits = 0;
    // In the dual tiles' arguments they save a copy to the device ahead of the launch and, with row_scale2, a product of the factors, each a
    // launch of its own of 4 to 5 us (a layer of 8 fp16 experts 4096 x 14336 with 1554 rows: 550 -> 535 us; block-scaled prefill at 780
    // us and fp8 at 1165, where the card's power is what runs out, did not change).
    const bool in_dual = host->dual && !computes && dual;
    if ((computes || in_dual) && args->nexperts <= kArgSplits) {
      run_few = computes;
      run_macro = in_dual;
      few.row_scale2 = host->row_scale2;
      few.count = args->nexperts;
      for (int e = 0; e < args->nexperts; ++e) few.splits[e] = host->splits[e];
      if (computes && panel.cols != 0) {
        int active;
        set_chunks(p, count_chunks(args, host->splits, panel.chunk_rows, active), cus, panel);
      }
    } else {
      if (args->splits == nullptr) return 0;
      FLUXMI_REQUIRE(host->row_scale2 == nullptr, FLUXMI_ERR_UNSUPPORTED, "grouped_gemm_host_splits: row_scale2 with splits on the device");
      run_few = computes;
      run_macro = macro && !computes;
    }
  }
  if (run_few && panel.cols != 0) {
    const int rc = launch_grouped_gemm_panel(p, few, args->dtype, panel, s);
    if (rc != FLUXMI_OK) return rc;
  } else if (run_few) {
    launch_grouped_gemm_stream(p, few, args->dtype, plan, s);
  }
  if (run_macro) {
    // Workgroups: the upper bound of the tile count, or up to four for each of those where there are too few tiles for the card: the kernels cut the
    // tiles of a round that is not full into two or four pieces when these still fit the grid.  us, one workgroup to a tile -> up to four: dual
    // tiles fp16 8 experts 4096 x 14336, 194 rows each 299 -> 267; bf16 2 experts 4096 x 8192, 200 rows 154 -> 117; block-scaled 4 experts 1024 x 4096, 500
    // rows 61 -> 44; macro tiles bf16 4 experts 2048 x 4096, 500 rows 105 -> 70; fp8 one expert 2048 x 4096, 2000 rows 48 -> 29.  Both deal a round
    // that is not full to all XCDs (bf16 8 experts 2048 x 4096, 600 rows, 192 whole tiles: 88, in 256 workgroups without that 96, with it 87; 360 rows 77 -> 71).
    const int64_t most = max_tiles * 4;
    const int grid = static_cast<int>(most < cus ? most : cus);
    // Form of the ring fills.  Whole 128-byte lines cost the memory pipeline less per byte and need one barrier per
    // pair of k-steps, but a pair's 64 KiB stay in LDS for both of its steps, so fewer fills are in flight: faster
    // (2-5 %) where the compute units that share operand panels run in step (uniform row counts) or K is long, slower
    // (up to 7 %) on ragged row counts at short K, where single units run ahead of the others and every one of their
    // fills misses L2.  Default: whole lines for rows that are not gathered and hold at least 16 KiB of K (measured on
    // 8 ragged experts at K = 14336 bf16: -1.2 ... -2.5 %), half lines otherwise (a single-expert rule was tried: the
    // dense bf16 GEMM 4096 x 12288 x 6144 gains under 1 %, the dense fp8 GEMMs 32768 x 7168 x 2048 lose 3-6 %); the flags force either, and `profiling()`
    // of the layer ops times both on the caller's own row counts.
    const int64_t kbytes = static_cast<int64_t>(args->k) * (args->dtype == FLUXMI_FP8_E4M3 ? 1 : 2);
    const bool lines = (args->sched_flags & FLUXMI_SCHED_WHOLE_LINE_FILLS) != 0 ||
                       ((args->sched_flags & FLUXMI_SCHED_HALF_LINE_FILLS) == 0 && args->gather_a == nullptr && kbytes >= 16384);
    const int rc = dual ? launch_grouped_gemm_dual(p, few, args->dtype, grid, s)
                   : bs != nullptr ? launch_grouped_gemm_fp8_blockscale(p, grid, s)
                   : args->dtype == FLUXMI_BF16 ? (lines ? launch_grouped_gemm_bf16_lines(p, grid, s) : launch_grouped_gemm_bf16(p, grid, s))
                   : args->dtype == FLUXMI_FP16 ? launch_grouped_gemm_f16(p, grid, s)  // the half-line form only
                                                : (lines ? launch_grouped_gemm_fp8_lines(p, grid, s) : launch_grouped_gemm_fp8(p, grid, s));
    if (rc != FLUXMI_OK) return rc;
  }
  if (!mfma) {
    const int grid = cus * 8;
    for (int g = 0; g < ngroups; ++g) {
      if (args->dtype != FLUXMI_FP8_E4M3)
        hipLaunchKernelGGL(grouped_gemm_generic_kernel<2>, dim3(grid), dim3(256), 0, s, p, g);
      else
        hipLaunchKernelGGL(grouped_gemm_generic_kernel<1>, dim3(grid), dim3(256), 0, s, p, g);
    }
  }
  FLUXMI_HIP_CHECK(hipGetLastError());
  return host != nullptr ? 1 : FLUXMI_OK;
}

}  // namespace
}  // namespace fluxmi

extern "C" int fluxmi_grouped_gemm(const fluxmi_grouped_gemm_args *args, void *, size_t, void *stream) {
  FLUXMI_REQUIRE(args != nullptr, FLUXMI_ERR_INVALID_ARG, "grouped_gemm: null args");
  const void *b = args->b;
  void *d = args->d;
  const float *alpha = args->alpha;
  return fluxmi::run_grouped_gemm(args, 1, &b, &d, &alpha, stream);
}

namespace fluxmi {
namespace {

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// 16-byte units of fp32 accumulators: cleared before the accumulating GEMM (a fill kernel, not a memset node,
// so that the sequence can be captured in a HIP graph) and rounded to bf16 after it.
__global__ __launch_bounds__(256) void zero_f32x4_kernel(float4 *__restrict__ dst, int64_t nvec) {
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < nvec; i += static_cast<int64_t>(gridDim.x) * 256)
    dst[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

template <bool F16>
__global__ __launch_bounds__(256) void cast_f32x4_half_kernel(const float4 *__restrict__ src, u32x2_t *__restrict__ dst,
                                                              int64_t nvec) {
  auto cvt = [](float f) { return static_cast<uint32_t>(F16 ? float_to_f16_bits(f) : float_to_bf16_bits(f)); };
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; i < nvec; i += static_cast<int64_t>(gridDim.x) * 256) {
    const float4 v = src[i];
    u32x2_t o;
    o[0] = cvt(v.x) | (cvt(v.y) << 16);
    o[1] = cvt(v.z) | (cvt(v.w) << 16);
    __builtin_nontemporal_store(o, dst + i);
  }
}

}  // namespace
}  // namespace fluxmi

extern "C" size_t fluxmi_grouped_gemm_topk_reduce_workspace_bytes(int32_t ntokens, int32_t n) {
  if (ntokens < 0 || n < 0) return 0;
  return static_cast<size_t>(ntokens) * static_cast<size_t>(n) * sizeof(float);
}

extern "C" int fluxmi_grouped_gemm_topk_reduce(const fluxmi_grouped_gemm_args *args, const int32_t *token_of_row,
                                               int32_t ntokens, void *out, void *workspace, size_t workspace_bytes,
                                               void *stream) {
  using namespace fluxmi;
  FLUXMI_REQUIRE(args != nullptr, FLUXMI_ERR_INVALID_ARG, "grouped_gemm_topk_reduce: null args");
  FLUXMI_REQUIRE(ntokens >= 0 && args->n >= 0, FLUXMI_ERR_INVALID_ARG, "grouped_gemm_topk_reduce: negative size");
  FLUXMI_REQUIRE(args->scatter_d == nullptr, FLUXMI_ERR_INVALID_ARG,
                 "grouped_gemm_topk_reduce: scatter_d must be NULL (token_of_row takes its place)");
  if (ntokens == 0 || args->n == 0) return FLUXMI_OK;
  FLUXMI_REQUIRE(token_of_row != nullptr && out != nullptr, FLUXMI_ERR_INVALID_ARG,
                 "grouped_gemm_topk_reduce: null token_of_row / out");
  FLUXMI_REQUIRE(args->n % 4 == 0 && (reinterpret_cast<uintptr_t>(out) & 7u) == 0, FLUXMI_ERR_UNSUPPORTED,
                 "grouped_gemm_topk_reduce: n must be a multiple of 4 and out 8-byte aligned");
  const size_t need = fluxmi_grouped_gemm_topk_reduce_workspace_bytes(ntokens, args->n);
  FLUXMI_REQUIRE(workspace != nullptr && workspace_bytes >= need && aligned16(workspace), FLUXMI_ERR_WORKSPACE,
                 "grouped_gemm_topk_reduce: a 16-byte aligned workspace of %zu bytes is needed, %zu given", need,
                 workspace_bytes);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t nvec = static_cast<int64_t>(ntokens) * args->n / 4;
  int cus = fluxmi_device_cu_count();
  FLUXMI_REQUIRE(cus > 0, FLUXMI_ERR_HIP, "grouped_gemm_topk_reduce: cannot query the device");
  const int64_t want = (nvec + 255) / 256;
  const unsigned grid = static_cast<unsigned>(want < static_cast<int64_t>(cus) * 16 ? want : static_cast<int64_t>(cus) * 16);
  hipLaunchKernelGGL(zero_f32x4_kernel, dim3(grid), dim3(256), 0, s, static_cast<float4 *>(workspace), nvec);
  fluxmi_grouped_gemm_args a = *args;
  a.scatter_d = token_of_row;
  const void *b = a.b;
  void *d = workspace;
  const float *alpha = a.alpha;
  const int rc = run_grouped_gemm(&a, 1, &b, &d, &alpha, stream, nullptr, ntokens);
  if (rc != FLUXMI_OK) return rc;
  if (args->dtype == FLUXMI_FP16)
    hipLaunchKernelGGL(cast_f32x4_half_kernel<true>, dim3(grid), dim3(256), 0, s, static_cast<const float4 *>(workspace),
                       static_cast<u32x2_t *>(out), nvec);
  else
    hipLaunchKernelGGL(cast_f32x4_half_kernel<false>, dim3(grid), dim3(256), 0, s, static_cast<const float4 *>(workspace),
                       static_cast<u32x2_t *>(out), nvec);
  FLUXMI_HIP_CHECK(hipGetLastError());
  return FLUXMI_OK;
}

extern "C" int fluxmi_grouped_gemm_blockscale(const fluxmi_grouped_gemm_args *args, const float *a_scale,
                                              int32_t a_scale_layout, const float *b_scale, int32_t b_scale_layout,
                                              void *stream) {
  FLUXMI_REQUIRE(args != nullptr, FLUXMI_ERR_INVALID_ARG, "grouped_gemm_blockscale: null args");
  fluxmi::BlockScales bs;
  bs.a_scale = a_scale;
  bs.b_scale = b_scale;
  bs.a_layout = a_scale_layout;
  bs.b_layout = b_scale_layout;
  const void *b = args->b;
  void *d = args->d;
  const float *alpha = args->alpha;
  return fluxmi::run_grouped_gemm(args, 1, &b, &d, &alpha, stream, nullptr, 0, &bs);
}

namespace fluxmi {
namespace {
int run_host_counts(const fluxmi_grouped_gemm_args *args, const int32_t *splits_host, const float *row_scale2, bool dual, const float *a_scale,
                    int32_t a_scale_layout, const float *b_scale, int32_t b_scale_layout, void *stream) {
  FLUXMI_REQUIRE(args != nullptr && splits_host != nullptr, FLUXMI_ERR_INVALID_ARG, "grouped_gemm_host_splits: null args / splits");
  BlockScales bs;
  bs.a_scale = a_scale;
  bs.b_scale = b_scale;
  bs.a_layout = a_scale_layout;
  bs.b_layout = b_scale_layout;
  const HostSplits host = {splits_host, row_scale2, dual};
  const void *b = args->b;
  void *d = args->d;
  const float *alpha = args->alpha;
  return run_grouped_gemm(args, 1, &b, &d, &alpha, stream, nullptr, 0, a_scale != nullptr || b_scale != nullptr ? &bs : nullptr, &host);
}
}  // namespace
}  // namespace fluxmi

extern "C" int fluxmi_grouped_gemm_host_splits(const fluxmi_grouped_gemm_args *args, const int32_t *splits_host, const float *row_scale2,
                                               const float *a_scale, int32_t a_scale_layout, const float *b_scale,
                                               int32_t b_scale_layout, void *stream) {
  return fluxmi::run_host_counts(args, splits_host, row_scale2, false, a_scale, a_scale_layout, b_scale, b_scale_layout, stream);
}

extern "C" int fluxmi_grouped_gemm_host_counts(const fluxmi_grouped_gemm_args *args, const int32_t *splits_host, const float *row_scale2,
                                               const float *a_scale, int32_t a_scale_layout, const float *b_scale,
                                               int32_t b_scale_layout, void *stream) {
  return fluxmi::run_host_counts(args, splits_host, row_scale2, true, a_scale, a_scale_layout, b_scale, b_scale_layout, stream);
}

extern "C" int fluxmi_grouped_gemm_kernel_kind(const fluxmi_grouped_gemm_args *args) {
  FLUXMI_REQUIRE(args != nullptr, FLUXMI_ERR_INVALID_ARG, "grouped_gemm: null args");
  const void *b = args->b;
  void *d = args->d;
  const float *alpha = args->alpha;
  fluxmi::DryRun dry;
  return fluxmi::run_grouped_gemm(args, 1, &b, &d, &alpha, nullptr, &dry);
}

namespace fluxmi {
namespace {

// The dry run of a launch of ngroups weight groups that all look like args->b / d / alpha.
int describe_launch(const fluxmi_grouped_gemm_args *args, int32_t ngroups, const float *a_scale, int32_t cu_count, DryRun &dry) {
  FLUXMI_REQUIRE(cu_count >= 1, FLUXMI_ERR_INVALID_ARG, "grouped_gemm_launch_info: cu_count must be positive");
  FLUXMI_REQUIRE(ngroups >= 1 && ngroups <= kMaxWeightGroups, FLUXMI_ERR_UNSUPPORTED, "grouped_gemm_launch_info: ngroups=%d outside [1,%d]",
                 ngroups, kMaxWeightGroups);
  const void *b[kMaxWeightGroups];
  void *d[kMaxWeightGroups];
  const float *alpha[kMaxWeightGroups];
  for (int g = 0; g < kMaxWeightGroups; ++g) b[g] = args->b, d[g] = args->d, alpha[g] = args->alpha;
  BlockScales bs;
  bs.a_scale = bs.b_scale = a_scale;
  dry.cus = cu_count;
  return run_grouped_gemm(args, ngroups, b, d, alpha, nullptr, &dry, 0, a_scale != nullptr ? &bs : nullptr);
}

}  // namespace
}  // namespace fluxmi

extern "C" int fluxmi_grouped_gemm_launch_info(const fluxmi_grouped_gemm_args *args, int32_t ngroups, const float *a_scale,
                                               const int32_t *splits_host, int32_t cu_count, fluxmi_gemm_launch_info *info) {
  using namespace fluxmi;
  FLUXMI_REQUIRE(args != nullptr && info != nullptr, FLUXMI_ERR_INVALID_ARG, "grouped_gemm_launch_info: null args / info");
  *info = fluxmi_gemm_launch_info{};
  DryRun dry;
  const int kind = describe_launch(args, ngroups, a_scale, cu_count, dry);
  if (kind < 0) return kind;
  const bool panel = dry.panel.cols != 0;
  const int32_t few_rows_form = panel ? FLUXMI_GEMM_PANEL : FLUXMI_GEMM_STREAM;
  if (kind == 0) info->form = FLUXMI_GEMM_GENERIC;
  else if (!panel && !dry.stream) info->form = FLUXMI_GEMM_MACRO_TILES;
  else if (!dry.macro) info->form = few_rows_form;
  else if (splits_host == nullptr) info->form = FLUXMI_GEMM_BY_SPLITS;
  else info->form = few_chunks(args, splits_host, panel ? dry.panel.chunk_rows : kStreamRows, dry.panel) ? few_rows_form : FLUXMI_GEMM_MACRO_TILES;
  if (dry.stream && !panel) {
    info->stream_cols = dry.plan.cols;
    info->stream_waves = dry.plan.waves;
    info->stream_workgroups = static_cast<int32_t>(dry.plan.workgroups);
    info->stream_lds_bytes = dry.plan.lds_bytes;
  }
  return FLUXMI_OK;
}

extern "C" int fluxmi_grouped_gemm_panel_info(const fluxmi_grouped_gemm_args *args, int32_t ngroups, const float *a_scale,
                                              const int32_t *splits_host, int32_t cu_count, fluxmi_gemm_panel_info *info) {
  using namespace fluxmi;
  FLUXMI_REQUIRE(args != nullptr && info != nullptr, FLUXMI_ERR_INVALID_ARG, "grouped_gemm_panel_info: null args / info");
  *info = fluxmi_gemm_panel_info{};
  DryRun dry;
  const int kind = describe_launch(args, ngroups, a_scale, cu_count, dry);
  if (kind < 0) return kind;
  if (kind == 0 || dry.panel.cols == 0) return FLUXMI_OK;
  info->cols = dry.panel.cols;
  info->chunk_rows = dry.panel.chunk_rows;
  info->workgroups = static_cast<int32_t>(dry.panel.workgroups);
  info->lds_bytes = dry.panel.lds_bytes;
  info->macro_tiles_too = dry.macro ? 1 : 0;
  info->computes = !dry.macro || (splits_host != nullptr && few_chunks(args, splits_host, dry.panel.chunk_rows, dry.panel)) ? 1 : 0;
  info->sums = dry.panel.sums;
  return FLUXMI_OK;
}

extern "C" int fluxmi_grouped_gemm_dual_tiles(const fluxmi_grouped_gemm_args *args, int32_t ngroups, const float *a_scale, int32_t cu_count) {
  FLUXMI_REQUIRE(args != nullptr, FLUXMI_ERR_INVALID_ARG, "grouped_gemm_dual_tiles: null args");
  fluxmi::DryRun dry;
  const int kind = fluxmi::describe_launch(args, ngroups, a_scale, cu_count, dry);
  return kind < 0 ? kind : (dry.dual ? 1 : 0);
}

extern "C" int fluxmi_grouped_gemm_multi(const fluxmi_grouped_gemm_args *args, int32_t ngroups, const void *const *b,
                                         void *const *d, const float *const *alpha, void *, size_t, void *stream) {
  return fluxmi::run_grouped_gemm(args, ngroups, b, d, alpha, stream);
}
