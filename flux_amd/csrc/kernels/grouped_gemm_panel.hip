// Grouped GEMM for up to about a hundred rows per expert: D[r,:] = scale(r,:) * A[gather(r),:] @ B[e(r)]^T.
//
// Bound by HBM: every weight is read once, for a chunk of up to 128 rows of its expert.  A workgroup of four waves computes 64,
// 128 or 256 columns of one chunk over the whole of K; each wave has a quarter of the columns and all of the rows.
//
//  * K goes by lines of 128 bytes per row.  Every load instruction covers eight whole lines, weights non-temporally (a stream of such
//    lines from HBM: 50 to 53 GB/s per compute unit alone and 26 with all of them, ordinary loads 45 and 20).  Where rows do not
//    start on lines (WHOLE false), each load covers parts of two lines and the next one wants the second again, which a
//    non-temporal load has given up: ordinary loads there (whole passes, non-temporal -> ordinary, us: bf16 40 experts 3760 x 1456,
//    80 rows each 311 -> 282, macro tiles 293; fp8 44 experts 5792 x 1680, 36 rows each 302 -> 269, macro tiles 299).
//  * The rows' operand goes through LDS: the four waves fill one ring of lines for all (direct-to-LDS loads), one wait and one
//    barrier per line.
//  * The weights are used by one wave only.  64- and 128-column workgroups pass them through LDS too, each wave through a ring of its
//    own, without a barrier; the row and its 16-byte chunk c lie at slot c ^ ((row >> 1) & 7), so that the fragment reads of one chain in
//    16 bits hit all banks (in fp8 and with several sums, where a lane reads neighbouring chunks, 0.45 to 0.5 of the access cycles are
//    conflicts, behind the memory's time).
//    256-column workgroups load them into registers and turn two loads into two fragments by exchanging lanes (to_fragments): LDS
//    then holds the rows' ring alone, and two workgroups with 128 rows share a compute unit.  What both do is keep about 64 KiB
//    of weights in flight per unit; more does not help (16 KiB 26 GB/s, 32 KiB 44, 64 KiB 52, 128 KiB 52 through LDS, but 30 with 32
//    register loads outstanding per wave).
//  * A result is summed over K in one wave.  In launches of few rows per expert, which the streaming form takes as well, it is the sum
//    of as many partial sums as that form has waves, line l of K in sum l % SUMS, added in ascending order: the bits of the streaming
//    form, so the choice between the two is free to follow the time.  One chain over K loses precision there (fp32 results
//    against float64, one chain / four sums: bf16 K = 4096 4.0e-7 / 1.9e-7, K = 14336 7.7e-7 / 3.7e-7; the sums are registers that were
//    free).  With more rows it is one chain in ascending lines, the macro tiles' order and for 16-bit operands their bits (the same
//    MFMAs over the same 32 elements).  Columns per workgroup, chunks, weight groups and cu_margin do not change a bit.
//  * A wave whose columns would end past N takes the last ones instead and stores only those that are its own; rows past the
//    chunk's last repeat it and are not stored; bytes past the end of K are zeros (of a page of zeros, or buffer loads out of range).
#include "grouped_gemm_panel.hpp"
#include "grouped_gemm_rows.hpp"

namespace fluxmi {
namespace {

#if defined(__HIP_DEVICE_COMPILE__)

// s_waitcnt vmcnt(vm) alone
#define FLUXMI_VMCNT(vm) __builtin_amdgcn_s_waitcnt(((vm)&15) | (((vm) >> 4) << 14) | (7 << 4) | (15 << 8))

typedef __attribute__((address_space(3))) void *lds_ptr_t;
typedef const __attribute__((address_space(1))) void *gbl_ptr_t;

__device__ __attribute__((aligned(1024))) const uint8_t g_zero_line[1024] = {};

// What a wave needs to know of its part of the item.
struct Columns {
  int w0;     // first column it computes
  int first;  // first column it stores, >= w0
};
template <int NB>
__device__ __forceinline__ Columns columns_of(int n, int n0, int wave) {
  const int first = n0 + wave * (16 * NB);
  return {first < n - 16 * NB ? first : n - 16 * NB, first};
}

// The rows' side of a line: fills of the ring and fragment reads.  A stage holds 16 * MB rows of 128 bytes and, block-scaled, a
// scale for each of up to 128 rows.
template <Elem T, int MB>
struct Rows {
  static constexpr bool BS = T == Elem::FP8_BLOCKSCALED;
  static constexpr int XF = MB > 1 ? MB / 2 : 1;    // per wave and line, of eight rows each (MB == 1: of four, by half of the lanes)
  static constexpr int FILLS = XF + (BS ? 1 : 0);
  static constexpr int BYTES = 16 * MB * 128, SCALES = BS ? 512 : 0;
  static_assert(MB == 1 || (MB % 2 == 0 && MB <= 8), "every wave has the same number of fills");
  const uint8_t *base, *sbase;
  uint32_t off[XF], soff;
  int byte[2], kb32, sstep, lane, wave;

  __device__ __forceinline__ void init(const GemmParams &p, const WorkItem &t, int wave_, int64_t kbytes) {
    lane = threadIdx.x & 63;
    wave = wave_;
    kb32 = static_cast<int>(kbytes);
    const bool gathered = p.gather_a != nullptr;
    base = gathered ? p.a : p.a + static_cast<int64_t>(t.row_base) * kbytes;
    auto source_row = [&](int r) {  // row of A that row r of the chunk reads, counted from `base`
      if (r > t.rows - 1) r = t.rows - 1;
      if (!gathered) return static_cast<int64_t>(r);
      const int64_t arow = p.gather_a[t.row_base + r];
      return arow < 0 ? 0 : (arow >= p.a_rows ? p.a_rows - 1 : arow);
    };
    // Fill j of a wave: lane l fetches row l >> 3 of its rows, the chunk that belongs into slot l & 7.
    auto fill_row = [&](int j) { return MB > 1 ? (wave * XF + j) * 8 + (lane >> 3) : wave * 4 + ((lane >> 3) & 3); };
#pragma unroll
    for (int j = 0; j < 2; ++j) byte[j] = ((lane & 7) ^ ((fill_row(j) >> 1) & 7)) * 16;
#pragma unroll
    for (int j = 0; j < XF; ++j) off[j] = static_cast<uint32_t>(source_row(fill_row(j)) * kbytes) + byte[j & 1];
    if constexpr (BS) {
      const int kblocks = kb32 >> 7;
      const int64_t srow = source_row((MB > 4 ? (wave & 1) * 64 : 0) + lane) + (gathered ? 0 : t.row_base);
      sbase = reinterpret_cast<const uint8_t *>(p.a_scale);
      soff = p.a_scale_layout == FLUXMI_ASCALE_BLOCK128 ? static_cast<uint32_t>(((srow >> 7) * kblocks * 128 + (srow & 127)) * 4)
                                                       : static_cast<uint32_t>((static_cast<int64_t>(t.expert_base) * (kblocks - 1) + srow) * 4);
      sstep = p.a_scale_layout == FLUXMI_ASCALE_BLOCK128 ? 512 : t.expert_rows * 4;
    }
  }
  __device__ __forceinline__ void fill(uint8_t *stage, int line) const {
    const int kb = line * 128;
    const uint8_t *const b = base + (kb < kb32 ? kb : 0);
    if constexpr (MB == 1) {
      const uint8_t *src = kb + byte[0] < kb32 ? b + off[0] : g_zero_line + lane * 16;
      if (lane < 32) __builtin_amdgcn_global_load_lds((gbl_ptr_t)src, (lds_ptr_t)(stage + wave * 512), 16, 0, 0);
    } else {
#pragma unroll
      for (int j = 0; j < XF; ++j) {
        const uint8_t *src = kb + byte[j & 1] < kb32 ? b + off[j] : g_zero_line + lane * 16;
        __builtin_amdgcn_global_load_lds((gbl_ptr_t)src, (lds_ptr_t)(stage + (wave * XF + j) * 1024), 16, 0, 0);
      }
    }
    if constexpr (BS) {  // 64 scales per wave, two or all four waves the same ones
      const uint8_t *src = kb < kb32 ? sbase + static_cast<int64_t>(line) * sstep + soff : g_zero_line + lane * 4;
      __builtin_amdgcn_global_load_lds((gbl_ptr_t)src, (lds_ptr_t)(stage + BYTES + (MB > 4 ? (wave & 1) * 256 : 0)), 4, 0, 0);
    }
  }
};

// Byte offset of this lane's fragment half h inside a block of sixteen rows of a line.  fp8: one MFMA takes all eight chunks, a lane two
// neighbours.  16-bit: MFMA h takes four of them, 4h .. 4h + 3 as the macro tiles do (one chain over K) or every second one as the
// streaming form does (several sums).
template <Elem T, int SUMS>
__device__ __forceinline__ int fragment_offset(int lane, int h) {
  const int r = lane & 15, c = is_fp8(T) || SUMS > 1 ? 2 * (lane >> 4) + h : (lane >> 4) + 4 * h;
  return r * 128 + ((c ^ ((r >> 1) & 7)) << 4);
}

// The MFMAs of one line on GB row blocks x NB column blocks.  s: scales of this lane's row in each block (block-scaled).
template <Elem T, int GB, int NB>
__device__ __forceinline__ void multiply(const i32x4 (&w)[NB][2], const i32x4 (&x)[GB][2], const float (&s)[GB], f32x4 (*acc)[NB]) {
#pragma unroll
  for (int i = 0; i < GB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if constexpr (T == Elem::FP8_BLOCKSCALED) {
        const f32x4 b = mfma_line<T>(w[j], x[i], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[i][j][v] = fmaf(b[v], s[i], acc[i][j][v]);
      } else {
        acc[i][j] = mfma_line<T>(w[j], x[i], acc[i][j]);
      }
    }
}

// What a lane multiplies its sums with and where it puts them: everything that is read, before the first store.  A load behind
// stores waits until those have drained, once per row block (fp8 32 experts 7168 x 2048, 32 rows each, all factors: 104 us -> 96; bf16 8 experts 1024 x 2048, 64 rows each 18.3 -> 16.3); asked for
// ahead of the loop over K they are there at its end.
template <int MB, int NB>
struct Factors {
  float row[MB], row2[MB], tile;
  f32x4 col[NB];
  int drow[MB];  // -1: not stored
  __device__ __forceinline__ void load(const GemmParams &p, const FewRowsArgs &few, const WorkItem &t, int g, const Columns &c) {
    const int lane = threadIdx.x & 63;
    tile = p.scalar * (p.scalar_dev ? p.scalar_dev[0] : 1.f) * (p.alpha[g] ? p.alpha[g][t.e] : 1.f);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int at = c.w0 + j * 16 + (lane >> 4) * 4;
      col[j] = f32x4{1.f, 1.f, 1.f, 1.f};
      if (p.col_scale) col[j] = *reinterpret_cast<const f32x4 *>(p.col_scale + static_cast<int64_t>(t.e) * p.n + at);
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int r = i * 16 + (lane & 15), at = t.row_base + (r < t.rows ? r : 0);
      row[i] = p.row_scale ? p.row_scale[at] : 1.f;
      row2[i] = few.row_scale2 ? few.row_scale2[at] : 1.f;
      drow[i] = p.scatter_d ? p.scatter_d[at] : at;
      if (r >= t.rows || (p.scatter_d && drow[i] >= p.d_rows)) drow[i] = -1;
    }
  }
};

// Scale, cast and store: a lane holds four consecutive columns of one row per block.
template <Elem T, int MB, int NB>
__device__ __forceinline__ void store(const GemmParams &p, int g, const Columns &c, const Factors<MB, NB> &f, const f32x4 (&acc)[MB][NB]) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    if (f.drow[i] < 0) continue;
    const float scale = f.tile * (f.row[i] * f.row2[i]);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int col = c.w0 + j * 16 + (lane >> 4) * 4;
      if (col < c.first) continue;
      f32x4 v = acc[i][j];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        v[q] *= scale;
        if (p.col_scale) v[q] *= f.col[j][q];
      }
      const int64_t at = static_cast<int64_t>(f.drow[i]) * p.n + col;
      if (p.accumulate) {
#pragma unroll
        for (int q = 0; q < 4; ++q) unsafeAtomicAdd(static_cast<float *>(p.d[g]) + at + q, v[q]);
      } else if (p.d_fp32) {
        *reinterpret_cast<f32x4 *>(static_cast<float *>(p.d[g]) + at) = v;
      } else {
        u32x2 o;
#pragma unroll
        for (int q = 0; q < 2; ++q)
          o[q] = T == Elem::F16 ? static_cast<uint32_t>(float_to_f16_bits(v[2 * q])) | (static_cast<uint32_t>(float_to_f16_bits(v[2 * q + 1])) << 16)
                                : static_cast<uint32_t>(float_to_bf16_bits(v[2 * q])) | (static_cast<uint32_t>(float_to_bf16_bits(v[2 * q + 1])) << 16);
        *reinterpret_cast<u32x2 *>(static_cast<uint16_t *>(p.d[g]) + at) = o;
      }
    }
  }
}

// Scale of a 128 x 128 block of the weights, for line `line` of the columns from w0 on.
struct WeightScale {
  const __attribute__((address_space(4))) float *b_scale;
  int base, step, kblocks;
  __device__ __forceinline__ void init(const GemmParams &p, const WorkItem &t, int w0) {
    kblocks = p.k >> 7;
    const int nb = w0 >> 7, nblocks = (p.n + 127) >> 7;
    base = p.b_scale_layout == FLUXMI_BSCALE_N_K ? (t.e * nblocks + nb) * kblocks : t.e * kblocks * nblocks + nb;
    step = p.b_scale_layout == FLUXMI_BSCALE_N_K ? 1 : nblocks;
    b_scale = (const __attribute__((address_space(4))) float *)p.b_scale;
  }
  // A scalar load (asked for a line ahead): a vector load would wait for every fill asked for before it.
  __device__ __forceinline__ float operator()(int line) const {
    return b_scale[__builtin_amdgcn_readfirstlane(base + (line < kblocks ? line : 0) * step)];
  }
};

template <int N>
__device__ __forceinline__ void zero(f32x4 *acc) {
#pragma unroll
  for (int i = 0; i < N; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
}

// 16 * MB rows x 64 * NB columns, weights through LDS.  Ring of DEPTH stages: the rows' line, then a line of each wave's weights.
// WHOLE: rows start on lines.  STEP: lines that are asked for together, waited for and computed.  Two halve the waits, and neighbouring lines of a row are
// fetched one after the other (64 columns, bf16 8 experts 14336 x 4096, 8 rows each: 142 us line by line, 136 in pairs).
// SUMS: partial sums of a result, line l belongs to sum l % SUMS.
template <Elem T, int MB, int NB, int DEPTH, int STEP, int SUMS, bool WHOLE>
__device__ __forceinline__ void lds_tile(const GemmParams &p, const FewRowsArgs &few, uint8_t *smem, const WorkItem &t, int g, int n0, int wave) {
  typedef Rows<T, MB> X;
  constexpr bool BS = X::BS;
  constexpr int WF = 2 * NB, PER_STEP = (X::FILLS + WF) * STEP, STEPS = DEPTH / STEP;  // vector-memory instructions per wave and step
  constexpr int WBYTES = 16 * NB * 128, STAGE = X::BYTES + X::SCALES + 4 * WBYTES;
  constexpr int UNROLL = SUMS > STEP ? SUMS / STEP : 1;  // steps until a line's sum is that of the first one again
  static_assert(SUMS == 1 || SUMS % STEP == 0, "a step starts at the same sum in every round");
  static_assert(DEPTH % STEP == 0 && STEPS >= 3, "a step computed, a step waited for, a step under way");
  const int lane = threadIdx.x & 63;
  const int64_t kbytes = static_cast<int64_t>(p.k) * (is_fp8(T) ? 1 : 2);
  const int kb32 = static_cast<int>(kbytes);
  const Columns c = columns_of<NB>(p.n, n0, wave);
  X x;
  x.init(p, t, wave, kbytes);
  WeightScale ws;
  float bs_next[STEP] = {};
  if constexpr (BS) {
    ws.init(p, t, c.w0);
#pragma unroll
    for (int u = 0; u < STEP; ++u) bs_next[u] = ws(u);
  }
  const uint8_t *const wbase = p.b[g] + (static_cast<int64_t>(t.e) * p.n + c.w0) * kbytes;
  int wbyte[2];
  uint32_t woff[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    wbyte[j] = ((lane & 7) ^ ((j * 4 + (lane >> 4)) & 7)) * 16;
    woff[j] = static_cast<uint32_t>(lane >> 3) * kb32 + wbyte[j];
  }
  auto fill = [&](int step, int line) {
    uint8_t *const at = smem + step * (STEP * STAGE);
#pragma unroll
    for (int u = 0; u < STEP; ++u) x.fill(at + u * STAGE, line + u);
    const int kb = line * 128;
    const uint8_t *const b = wbase + (kb < kb32 ? kb : 0);
#pragma unroll
    for (int j = 0; j < WF; ++j)
#pragma unroll
      for (int u = 0; u < STEP; ++u) {
        const uint8_t *src = kb + u * 128 + wbyte[j & 1] < kb32 ? b + u * 128 + j * 8 * kbytes + woff[j & 1] : g_zero_line + lane * 16;
        __builtin_amdgcn_global_load_lds((gbl_ptr_t)src, (lds_ptr_t)(at + u * STAGE + X::BYTES + X::SCALES + wave * WBYTES + j * 1024), 16, 0, WHOLE ? 2 : 0);
      }
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4 acc[SUMS][MB][NB];
  zero<SUMS * MB * NB>(&acc[0][0][0]);
  const int foff[2] = {fragment_offset<T, SUMS>(lane, 0), fragment_offset<T, SUMS>(lane, 1)};
  auto compute = [&](const uint8_t *sx, float bs, f32x4 (&sum)[MB][NB]) {
    const uint8_t *const sw = sx + X::BYTES + X::SCALES + wave * WBYTES;
    i32x4 w[NB][2], xf[2][1][2];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) w[j][h] = *reinterpret_cast<const i32x4 *>(sw + j * 2048 + foff[h]);
    float as[MB];
    if constexpr (BS) {
#pragma unroll
      for (int i = 0; i < MB; ++i) as[i] = reinterpret_cast<const float *>(sx + X::BYTES)[i * 16 + (lane & 15)] * bs;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) xf[0][0][h] = *reinterpret_cast<const i32x4 *>(sx + foff[h]);
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      if (i + 1 < MB) {
#pragma unroll
        for (int h = 0; h < 2; ++h) xf[(i + 1) & 1][0][h] = *reinterpret_cast<const i32x4 *>(sx + (i + 1) * 2048 + foff[h]);
      }
      __builtin_amdgcn_sched_barrier(0);
      const float s[1] = {BS ? as[i] : 1.f};
      multiply<T, 1, NB>(w, xf[i & 1], s, &sum[i]);
      if constexpr (BS) {  // added here: sunk towards the next use of this sum, they keep products alive (308 spilled registers)
#pragma unroll
        for (int j = 0; j < NB; ++j) asm volatile("" : "+v"(sum[i][j]));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  const int lines = (kb32 + 127) >> 7;
#pragma unroll
  for (int d = 0; d < STEPS - 1; ++d) fill(d, d * STEP);
  // (Ahead of the loop also where the registers do not suffice: block-scaled tiles of 128 rows x 64 columns have 20 bytes of scratch per lane,
  // and none with these loads behind the loop, but are 3.6 % faster so, 21925 launches in the mean and 3 of them slower.)
  Factors<MB, NB> f;
  f.load(p, few, t, g, c);
  int step = 0;
  for (int line = 0; line < lines;) {
#pragma unroll
    for (int q = 0; q < UNROLL; ++q) {
      if (q > 0 && line >= lines) break;
      FLUXMI_VMCNT((STEPS - 2) * PER_STEP);  // these lines have landed for this wave's share
      __builtin_amdgcn_s_barrier();          // ... and for everybody's; nobody reads the lines before them any more
      __builtin_amdgcn_sched_barrier(0);
      fill(step == 0 ? STEPS - 1 : step - 1, line + (STEPS - 1) * STEP);
#pragma unroll
      for (int u = 0; u < STEP; ++u) {
        float bs = 1.f;
        if constexpr (BS) {
          bs = line + u < lines ? bs_next[u] : 0.f;  // past K the rows' scales are zeros, and 0 * inf is not 0
          bs_next[u] = ws(line + STEP + u);
        }
        compute(smem + (step * STEP + u) * STAGE, bs, acc[(q * STEP + u) % SUMS]);
      }
      line += STEP;
      step = step == STEPS - 1 ? 0 : step + 1;
    }
  }
  FLUXMI_VMCNT(0);  // no fill may reach LDS after the workgroup has ended (or its next item has begun)
#pragma unroll
  for (int u = 1; u < SUMS; ++u)
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[0][i][j] += acc[u][i][j];
  store<T, MB, NB>(p, g, c, f, acc[0]);
}

// 16 * MB rows x 64 * NB columns, weights through registers, two lines ahead; the rows' ring has a stage more.  Not block-scaled.
template <Elem T, int MB, int NB, bool WHOLE>
__device__ __forceinline__ void register_tile(const GemmParams &p, const FewRowsArgs &few, uint8_t *smem, const WorkItem &t, int g, int n0, int wave) {
  typedef Rows<T, MB> X;
  static_assert(!X::BS, "no registers left for block scales");
  constexpr int DEPTH = 2, GB = 2, GROUPS = MB / GB, STAGE = X::BYTES, PER_LINE = X::FILLS + 2 * NB;
  const int lane = threadIdx.x & 63;
  const int64_t kbytes = static_cast<int64_t>(p.k) * (is_fp8(T) ? 1 : 2);
  const int kb32 = static_cast<int>(kbytes);
  const Columns c = columns_of<NB>(p.n, n0, wave);
  X x;
  x.init(p, t, wave, kbytes);
  // Lane l of a load fetches row l & 7 of eight; which 16 bytes: what to_fragments makes the chunks of fragment_offset of.
  const int wbyte = is_fp8(T) ? (lane >> 4) * 32 + ((lane >> 3) & 1) * 16 : (lane >> 4) * 16 + ((lane >> 3) & 1) * 64;
  const auto wr = buffer_of(p.b[g] + (static_cast<int64_t>(t.e) * p.n + c.w0) * kbytes, 16 * NB * kbytes);
  const uint32_t woff = static_cast<uint32_t>(lane & 7) * kb32 + wbyte;
  i32x4 w[DEPTH][NB][2];
  auto load_w = [&](i32x4 (&v)[NB][2], int line) {
    const int kb = line * 128;
    const uint32_t off = kb + wbyte < kb32 ? woff : kOutOfRange;
    const uint32_t ks = kb < kb32 ? kb : 0;
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int h = 0; h < 2; ++h) v[j][h] = load16<WHOLE ? 2 : 0>(wr, off, static_cast<int>(ks + (2 * j + h) * 8u * static_cast<uint32_t>(kb32)));
  };
  f32x4 acc[MB][NB];
  zero<MB * NB>(&acc[0][0]);
  const int foff[2] = {fragment_offset<T, 1>(lane, 0), fragment_offset<T, 1>(lane, 1)};
  i32x4 xf[2][GB][2];
  auto read_x = [&](i32x4 (&v)[GB][2], const uint8_t *sx, int grp) {
#pragma unroll
    for (int i = 0; i < GB; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) v[i][h] = *reinterpret_cast<const i32x4 *>(sx + (grp * GB + i) * 2048 + foff[h]);
  };
  const int lines = (kb32 + 127) >> 7;
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) {
    x.fill(smem + d * STAGE, d);
    load_w(w[d], d);
    __builtin_amdgcn_sched_barrier(0);
  }
  int stage = 0;
  for (int s = 0; s < lines; s += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      FLUXMI_VMCNT((DEPTH - 1) * PER_LINE);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      const uint8_t *const sx = smem + stage * STAGE;
      read_x(xf[0], sx, 0);
      x.fill(smem + (stage == 0 ? DEPTH : stage - 1) * STAGE, s + d + DEPTH);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NB; ++j) to_fragments(w[d][j]);
#pragma unroll
      for (int grp = 0; grp < GROUPS; ++grp) {
        if (grp + 1 < GROUPS) read_x(xf[(grp + 1) & 1], sx, grp + 1);
        __builtin_amdgcn_sched_barrier(0);
        const float unscaled[GB] = {};
        multiply<T, GB, NB>(w[d], xf[grp & 1], unscaled, &acc[grp * GB]);
        __builtin_amdgcn_sched_barrier(0);
      }
      load_w(w[d], s + d + DEPTH);
      __builtin_amdgcn_sched_barrier(0);
      stage = stage == DEPTH ? 0 : stage + 1;
    }
  }
  FLUXMI_VMCNT(0);
  Factors<MB, NB> f;
  f.load(p, few, t, g, c);
  store<T, MB, NB>(p, g, c, f, acc);
}

#endif  // __HIP_DEVICE_COMPILE__

constexpr int kUnits = 256;  // compute units
constexpr int kCuLds = 160 * 1024, kWalkLds = 96 * 1024;

// CH: most 16-row blocks of a chunk; DEPTH: stages of the ring, 0: weights through registers.
template <Elem T, int CH, int NB, int DEPTH>
constexpr int lds_bytes() {
  constexpr int scales = T == Elem::FP8_BLOCKSCALED ? 512 : 0;
  return DEPTH > 0 ? DEPTH * (CH * 2048 + scales + NB * 8192) : 3 * CH * 2048;
}

template <Elem T, int CH, int NB, int DEPTH, int SUMS, bool WHOLE>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
void grouped_gemm_panel_kernel(const FewRowsArgs few, const GemmParams p, const int blocks) {
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tiles_n1 = (p.n + 64 * NB - 1) / (64 * NB);
  int block = blockIdx.x;
  while (true) {
    const WorkItem t = locate<T>(p, tiles_n1 * p.ngroups, 16 * CH, block);
    if (t.rows > 0) {
      const int g = p.ngroups > 1 ? __builtin_amdgcn_readfirstlane(t.nt / tiles_n1) : 0;
      const int n0 = (t.nt - g * tiles_n1) * (64 * NB);
      auto tile = [&](auto BLOCKS) {
        constexpr int mb = decltype(BLOCKS)::value;
        if constexpr (mb <= CH) {
          if constexpr (DEPTH > 0) lds_tile<T, mb, NB, DEPTH, DEPTH == 6 ? 2 : 1, SUMS, WHOLE>(p, few, smem, t, g, n0, wave);
          else register_tile<T, mb, NB, WHOLE>(p, few, smem, t, g, n0, wave);
        }
      };
      if (CH == 2 && t.rows <= 16) tile(std::integral_constant<int, CH == 2 ? 1 : 2>{});
      else if (t.rows <= 32) tile(std::integral_constant<int, 2>{});
      else if (t.rows <= 64) tile(std::integral_constant<int, 4>{});
      else if (t.rows <= 96) tile(std::integral_constant<int, 6>{});
      else tile(std::integral_constant<int, 8>{});
    }
    if constexpr (DEPTH == 0) return;  // a loop costs this form the registers that it does not have (20 of them would be spilled)
    block += gridDim.x;
    if (block >= blocks) return;
    __syncthreads();  // nobody reads the ring of this item any more
  }
#endif
}

template <Elem T, int CH, int NB, int DEPTH, int SUMS, bool WHOLE>
int launch_tiles(const GemmParams &p, const FewRowsArgs &few, const PanelPlan &plan, hipStream_t s) {
  static std::atomic<uint64_t> done{0};
  const void *kernel = reinterpret_cast<const void *>(grouped_gemm_panel_kernel<T, CH, NB, DEPTH, SUMS, WHOLE>);
  const int rc = ensure_dynamic_lds(kernel, kCuLds, done);
  if (rc != FLUXMI_OK) return rc;
  hipLaunchKernelGGL((grouped_gemm_panel_kernel<T, CH, NB, DEPTH, SUMS, WHOLE>), dim3(plan.workgroups), dim3(256), plan.lds_bytes, s, few, p, plan.blocks);
  return FLUXMI_OK;
}

// Whether every row of the weights starts on a line of 128 bytes.
bool whole_lines(const GemmParams &p, int elt) {
  uint64_t bits = static_cast<uint64_t>(p.k) * elt;
  for (int g = 0; g < p.ngroups; ++g) bits |= reinterpret_cast<uintptr_t>(p.b[g]);
  return bits % 128 == 0;
}

template <Elem T, int CH, int NB, int DEPTH, int SUMS>
int launch(const GemmParams &p, const FewRowsArgs &few, const PanelPlan &plan, hipStream_t s) {
  if (whole_lines(p, is_fp8(T) ? 1 : 2)) return launch_tiles<T, CH, NB, DEPTH, SUMS, true>(p, few, plan, s);
  return launch_tiles<T, CH, NB, DEPTH, SUMS, false>(p, few, plan, s);
}

// Stages of the ring for 128 columns and 32 rows: four fill half of a compute unit's LDS exactly; with scales three do.
template <Elem T>
constexpr int kDepth32 = T == Elem::FP8_BLOCKSCALED ? 3 : 4;

template <Elem T>
int launch_by_plan(const GemmParams &p, const FewRowsArgs &few, const PanelPlan &plan, hipStream_t s) {
  if constexpr (T != Elem::FP8_BLOCKSCALED)
    if (plan.cols == 256) return launch<T, 8, 4, 0, 1>(p, few, plan, s);
  const bool wide = plan.cols == 128;
  if (plan.chunk_rows == 128) return wide ? launch<T, 8, 2, 3, 1>(p, few, plan, s) : launch<T, 8, 1, 3, 1>(p, few, plan, s);
  if (plan.chunk_rows == 32) {  // always few rows, and four sums
    if (wide) return launch<T, 2, 2, kDepth32<T>, 4>(p, few, plan, s);
    return plan.pairs ? launch<T, 2, 1, 6, 4>(p, few, plan, s) : launch<T, 2, 1, 4, 4>(p, few, plan, s);
  }
  if (wide) return plan.sums == 4 ? launch<T, 4, 2, 3, 4>(p, few, plan, s) : launch<T, 4, 2, 3, 1>(p, few, plan, s);
  if constexpr (T != Elem::FP8_BLOCKSCALED)
    if (plan.deep)
      return plan.sums == 8 ? launch<T, 4, 1, 6, 8>(p, few, plan, s)
                            : (plan.sums == 4 ? launch<T, 4, 1, 6, 4>(p, few, plan, s) : launch<T, 4, 1, 6, 1>(p, few, plan, s));
  return plan.sums == 8 ? launch<T, 4, 1, 4, 8>(p, few, plan, s)
                        : (plan.sums == 4 ? launch<T, 4, 1, 4, 4>(p, few, plan, s) : launch<T, 4, 1, 4, 1>(p, few, plan, s));
}

template <Elem T>
int lds_of(const PanelPlan &plan) {
  const int blocks16 = plan.chunk_rows / 16;
  if (plan.cols == 256) return lds_bytes<T, 8, 4, 0>();
  if (plan.cols == 128) return blocks16 <= 2 ? lds_bytes<T, 2, 2, kDepth32<T>>() : (blocks16 <= 4 ? lds_bytes<T, 4, 2, 3>() : lds_bytes<T, 8, 2, 3>());
  if (blocks16 <= 2 && plan.pairs) return lds_bytes<T, 2, 1, 6>();
  if (plan.deep) return lds_bytes<T, 4, 1, 6>();
  return blocks16 <= 2 ? lds_bytes<T, 2, 1, 4>() : (blocks16 <= 4 ? lds_bytes<T, 4, 1, 4>() : lds_bytes<T, 8, 1, 3>());
}

int64_t row_bytes(const GemmParams &p, int dtype) { return static_cast<int64_t>(p.k) * (dtype == FLUXMI_FP8_E4M3 ? 1 : 2); }

// A wave has up to 64 columns, inside one 128 x 128 block of scales; offsets along K and over a wave's columns fit 32 bits.
bool shape_ok(const GemmParams &p, int dtype) {
  return p.n >= 64 && (p.a_scale == nullptr || p.n % 64 == 0) && row_bytes(p, dtype) < (1 << 24);
}

// Items of `cols` columns if every expert that can get rows is one chunk.
int64_t even_items(const GemmParams &p, int cols, int ngroups) {
  const int64_t active = p.nexperts < p.max_rows ? p.nexperts : p.max_rows;
  return active * ((p.n + cols - 1) / cols) * ngroups;
}

int64_t most_items(const GemmParams &p, int dtype, int cols, int chunk_rows, bool any_splits, int ngroups) {
  const int active = p.nexperts < p.max_rows ? p.nexperts : p.max_rows;
  int64_t chunks = active + (p.max_rows - active) / chunk_rows;
  const int limit = stream_chunks_limit(active, chunk_rows, dtype == FLUXMI_FP8_E4M3, 0, 0);  // (rounds make it no larger)
  if (!any_splits && chunks > limit) chunks = limit;
  return chunks * ((p.n + cols - 1) / cols) * ngroups;
}

constexpr int64_t kMostItems = (int64_t{1} << 31) - (1 << 20);  // items are numbered with ints

int64_t block_count(const GemmParams &p, int dtype, const PanelPlan &plan) {
  return (most_items(p, dtype, plan.cols, plan.chunk_rows, plan.any_splits, p.ngroups) + 7) / 8 * 8;
}

// Whether the workgroups of a launch walk several items: compute units are to be left free, or it would have 2^31 threads and more.
bool walks(int64_t blocks, bool leave_cus) { return leave_cus || blocks * 256 > 0x7fffffffll; }

// A ring of six stages, lines in pairs: 96 KiB, so one workgroup to a unit, which is all there is where no unit gets two.  A line then costs its wait, barrier
// and chain of reads and MFMAs (0.2 us), and pairs halve the waits.  us per launch, weights not in the cache, four stages line by line / six in
// pairs / eight in pairs: bf16 8 experts 1024 x 2048, R 16 13.6 / 12.3 / 12.0, R 64 16.0 / 15.1 / 15.7; 4 experts 2048 x 1024, R 48 10.2 / 9.7 / 10.1; fp8 8
// experts 1024 x 2048, R 64 11.0 / 10.4 / 11.1; fp16 4 experts 1024 x 4096, R 80 24.9 / 22.3 / 22.6.  Eight stages line by line 17.5, 11.6, 12.1, 26.2: more to
// ask for before the first line.  Block-scaled 13.4 / 13.4 / 14.1: four stages.
bool is_deep(const PanelPlan &plan, int64_t blocks, bool block_scaled, int cus) {
  return plan.cols == 64 && plan.chunk_rows == 64 && !plan.walk && !block_scaled && blocks <= cus;
}

// Sizes of the launch of a plan whose columns and chunks are decided.
void finish(const GemmParams &p, int dtype, int cus, bool leave_cus, PanelPlan &plan) {
  const int64_t blocks = block_count(p, dtype, plan);
  plan.blocks = static_cast<int>(blocks);
  plan.chunk_items = (p.n + plan.cols - 1) / plan.cols * p.ngroups;
  plan.round_items = plan.chunk_rows == 128 && plan.cols == 128 && p.a_scale != nullptr ? kUnits : 0;
  plan.walk = walks(blocks, leave_cus);
  plan.deep = is_deep(plan, blocks, p.a_scale != nullptr, cus);
  const int64_t most = cus >= 8 ? cus / 8 * 8 : cus;  // whole rounds over the XCDs where there are enough units
  plan.workgroups = static_cast<unsigned>(plan.walk && blocks > most ? most : blocks);
  plan.lds_bytes = p.a_scale != nullptr ? lds_of<Elem::FP8_BLOCKSCALED>(plan) : lds_of<Elem::FP8>(plan);
  // More than half of a compute unit's LDS: no unit takes two of the walking workgroups, and N of them occupy N units.
  if (plan.walk && plan.lds_bytes < kWalkLds) plan.lds_bytes = kWalkLds;
}

}  // namespace

void set_chunks(const GemmParams &p, int64_t chunks, int cus, PanelPlan &plan) {
  if (plan.walk) return;
  const int64_t blocks = (chunks > 0 ? chunks * plan.chunk_items + 7 : 8) / 8 * 8;
  if (blocks >= plan.blocks) return;
  plan.blocks = static_cast<int>(blocks);
  plan.workgroups = static_cast<unsigned>(blocks);
  plan.deep = is_deep(plan, blocks, p.a_scale != nullptr, cus);
  plan.lds_bytes = p.a_scale != nullptr ? lds_of<Elem::FP8_BLOCKSCALED>(plan) : lds_of<Elem::FP8>(plan);
}

// Rules by rows per expert on average (R), items and bytes of the weights; us are bf16 unless they say otherwise, before (streaming
// form or macro tiles) -> these tiles.  The sums of a result follow from the launch of one weight group, whatever its margin.
PanelPlan plan_panel(const GemmParams &p, int dtype, bool few_rows, int cus, bool leave_cus) {
  PanelPlan plan = {};
  const int64_t line_count = (row_bytes(p, dtype) + 127) / 128, items64 = even_items(p, 64, 1);
  auto at_most = [&](int64_t rows) { return p.max_rows <= rows * p.nexperts; };
  // Weight groups are items and weights as well (two groups of fp8 16 experts 2048 x 2048, R 64 / 80, random: macro tiles 37 and 38, as
  // small launches 45 and 56).  Not where the streaming form is the other one: whether the macro tiles, with another order of sums, can
  // compute a launch must not follow from the groups there, and it does not lose (the same at R 23: 34 -> 32).
  const int groups = few_rows ? 1 : p.ngroups;
  const bool small = items64 * groups <= 512 && static_cast<int64_t>(groups) * p.nexperts * p.n * row_bytes(p, dtype) <= (64 << 20);
  const bool long_k = line_count >= 48, many_items = even_items(p, 128, p.ngroups) >= 1024;
  if (!shape_ok(p, dtype)) return plan;
  plan.sums = few_rows ? stream_waves(p, dtype) : 1;
  // Hardly a row: the streaming form (64 experts 2816 x 2048, R 1: 78 against 86; fp8 32 experts 2048 x 7168 46 against 50).
  if (few_rows && at_most(4)) return PanelPlan{};
  // Few columns and long K: the streaming form splits K over eight waves (8 rows on 8 experts 4096 x 14336: 77 against 82).
  if (few_rows && at_most(16) && items64 < 512 && line_count >= 64) return PanelPlan{};
  // 128 columns of rows that lie a multiple of 4 KiB apart, all of them read at the same line: few memory channels at a time.  The
  // streaming form's waves are at different lines (64 experts 2816 x 2048, R 8: 115 against 118, fp8 4096 117 against 126; K = 2112
  // 126 against 119, K = 1984 114 against 113).
  if (few_rows && at_most(16) && many_items && !long_k && row_bytes(p, dtype) % 4096 == 0) return PanelPlan{};
  const int64_t items_one = (p.max_rows + 127) / 128 * ((p.n + 63) / 64) * groups;  // all rows on one expert
  if (small && (at_most(96) || (at_most(192) && items_one <= 512))) {
    // Weights that fit the Infinity Cache in few items: latency counts, so many workgroups, and no second launch whatever the splits
    // (the macro tiles that return at once cost 5).  8 experts of 2048 x 1024, R 16 / 64 / 128: 14.4 -> 11.9, 23 -> 13, 34 -> 20; of
    // 1024 x 2048: 14.4 -> 12.7, 31 -> 15.6, 47 -> 23; all rows on one expert, R 16 / 128: 19 -> 10 and 22 -> 16.  With more than 96
    // rows while even that is one round, two workgroups to a unit (weights that are not in the cache, R 128 and 150, all rows on one
    // expert: 64 experts 512 x 1024 30 -> 27 and 30 -> 37, fp8 16 experts 2048 x 2048 26 -> 22 and 27 -> 36; 48 experts 512 x 1024, R 170
    // and 192: 30 -> 27 and 29 -> 37).
    plan.cols = 64;
    plan.chunk_rows = at_most(96) ? 64 : 128;
    plan.any_splits = true;
  } else if (few_rows) {
    // R 8 and 16: 8 experts 14336 x 4096 145 -> 140 and 157 -> 142, 64 experts 2048 x 1408 64 -> 60 and 71 -> 62, 1408 x 2048 65 -> 61 and
    // 71 -> 63; fp8 32 experts 7168 x 2048 87 -> 75 and 95 -> 79, block-scaled 88 -> 81 and 100 -> 85.  64 columns where K is long,
    // lines in pairs (8 experts 14336 x 4096, R 8: 136; one by one 142; 128 columns 146); at short K 128 where they give items enough,
    // which read the rows half as often (64 experts 2048 x 1408 59, 64 columns one by one 63, pairs 62).  Ordinary random routing at
    // R 20 has experts with more than 32 rows, so chunks of 64 from 16 on (8 experts 14336 x 4096, R 32: 222 -> 154).
    plan.pairs = long_k;
    plan.cols = many_items && !long_k ? 128 : 64;
    plan.chunk_rows = at_most(16) ? 32 : 64;
  } else if (at_most(40)) {
    // R 32: fp8 32 experts 7168 x 2048 120 -> 94, 2048 x 7168 97 -> 77, block-scaled 155 -> 95 and 130 -> 79.
    plan.cols = even_items(p, 128, p.ngroups) >= 192 ? 128 : 64;
    plan.chunk_rows = 64;
  } else if (at_most(96)) {
    // R 64: 8 experts 14336 x 4096 228 -> 176 (256 columns; 128: 198), 4096 x 14336 390 -> 165 (128 columns; 256: 315), 64 experts 2048
    // x 1408 100 -> 76, fp8 32 experts 7168 x 2048 125 -> 108, block-scaled 161 -> 143; R 88: 239 -> 185, 241 -> 172, 104 -> 85, 133 ->
    // 117, 164 -> 162.  R 128, where half of the experts have two chunks: 243 -> 268.  The 256-column form has no registers left for a
    // loop over items, so it takes no launch that walks, nor for block scales.
    plan.chunk_rows = 128;
    plan.cols = 256;
    if (even_items(p, 256, p.ngroups) < 384 || p.a_scale != nullptr || walks(block_count(p, dtype, plan), leave_cus))
      plan.cols = even_items(p, 128, p.ngroups) >= 192 ? 128 : 64;
    // fp8 with more than 64 rows and short K, two rounds of 128 columns and more: half of a macro tile's columns is no gain any more (770
    // launches of random, log-normal and square-root-skewed rows, K below 6 KiB, macro tiles / these tiles in the mean: two rounds R 65 to 80
    // 0.98, R 81 to 96 0.95, more rounds 1.00 and 0.98; at least 0.82; two groups of 16 experts 2048 x 2048, R 80: 38 against 44).  R 41 to 64
    // 1.04 and 1.11, longer K 1.05, block-scaled 1.00 to 1.17, 16 bits 1.01 to 1.2, one round 1.05 to 1.6.
    if (dtype == FLUXMI_FP8_E4M3 && p.a_scale == nullptr && !at_most(64) && plan.cols == 128 && even_items(p, 128, p.ngroups) > kUnits &&
        row_bytes(p, dtype) < 6144)
      return PanelPlan{};
  } else {
    return PanelPlan{};
  }
  // Counted in the streaming form's narrowest columns and the most weight groups: where that form gives up the macro tiles run.
  if (most_items(p, dtype, 32, plan.chunk_rows, plan.any_splits, kMaxWeightGroups) > kMostItems) return PanelPlan{};
  finish(p, dtype, cus, leave_cus, plan);
  return plan;
}

int launch_grouped_gemm_panel(const GemmParams &p, const FewRowsArgs &few, int dtype, const PanelPlan &plan, hipStream_t s) {
  if (p.a_scale != nullptr) return launch_by_plan<Elem::FP8_BLOCKSCALED>(p, few, plan, s);
  if (dtype == FLUXMI_FP8_E4M3) return launch_by_plan<Elem::FP8>(p, few, plan, s);
  if (dtype == FLUXMI_FP16) return launch_by_plan<Elem::F16>(p, few, plan, s);
  return launch_by_plan<Elem::BF16>(p, few, plan, s);
}

}  // namespace fluxmi
