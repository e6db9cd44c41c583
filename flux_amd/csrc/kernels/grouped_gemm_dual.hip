// Grouped GEMM, tiles of 256 x 256 on eight waves, two to a SIMD ("dual tiles"): D[r,:] = scale(r,:) * A[gather(r),:] @ B[e(r)]^T.
//
// Bound by the MFMAs and by what brings operands to them.  The macro tiles (grouped_gemm_kernel.hpp) have one wave on a SIMD: what is not
// an MFMA (LDS reads, fills, the promotion of block-scaled sums) takes its time beside the MFMAs.  Here the waves of a SIMD take turns:
// while one group of four waves computes, one wave to a SIMD, the other reads its next fragments from LDS and requests fills, and a
// barrier ends the phase for both.  With both groups in step instead, each with reads, fills and MFMAs interleaved, fills that wait for the
// memory pipeline stop both waves of a SIMD, and everything takes 1.2 to 1.4 times as long.
//
//  * A wave's 128 x 64 quarter columns of a tile are rows wm * 64 .. + 63 of both of the tile's halves of 128 rows and columns wn * 64 ..
//    + 63.  A step is 128 bytes of K and four phases for each group: read (the first half's rows, all columns), compute 64 x 64, read (the
//    second half's rows), compute; the second group is one phase behind.  Phases of 64 rows that an expert does not have are left out, and
//    an expert's rows are dealt to its tiles in units of 64 as evenly as they go.
//  * LDS is a ring of units of 128 rows (of A or of B) x 128 bytes, four units to a step, filled seven phases ahead by whichever group is
//    reading.  Units are requested across tile ends: a tile starts with its first steps in LDS.
//  * Block-scaled sums are promoted out of the MFMA's result three MFMAs later, one multiply-add per sum, beside the MFMAs of the same
//    wave; 128 running sums and 64 fragment registers per lane leave room for them, which one wave with 256 x 256 / 4 sums does not have.
//  * A lane's four sums of a block are neighbouring columns of one row.  16-bit results: which column an LDS row of B holds is chosen so
//    that two blocks' sums are eight neighbours, and a store instruction writes 64 bytes of 16 rows straight from registers.
//
// us, macro tiles -> these.  Block-scaled fp8 (there pieces of 256 x 128): 32 experts 2048 x 7168 and 7168 x 2048, 16384 rows in all at
// random 309 -> 272 and 330 -> 279; 1024 rows each 523 -> 434 and 593 -> 484 (2.22 and 1.99 PFLOP/s); 188 rows each 146 -> 120 and 166 ->
// 134.  fp16, 8 experts, 194 rows each: 14336 x 4096 270 -> 247, 4096 x 14336 334 -> 301.  fp8 32 experts 7168 x 2048, 1024 rows each
// 516 -> 505.  Without block scales long K with many rows stays on the macro tiles: both are at the board's power limit there, and
// these read half as much again from LDS per MFMA (dense fp8 8192 x 8192 x 8192: 736 k cycles against 771 k, at 1.73 GHz against 1.95;
// bf16 8 experts 4096 x 14336, 2048 rows each 1361 -> 1540).
#include "grouped_gemm_dual.hpp"
#include "grouped_gemm_rows.hpp"

namespace fluxmi {
namespace {

constexpr int kDualThreads = 512;
constexpr int kTile = 256;            // rows and columns of a tile
constexpr int kUnit = 16384;          // 128 rows of one operand x 128 bytes of K
constexpr int kRing = 9;              // units
constexpr int kAhead = 7;             // phases from a unit's request on until the first group may read it
constexpr int kScaleSlot = 1024;      // a tile's row scales of one step, three steps of them behind the ring
constexpr int kDualExperts = 128;     // two to a lane
// Behind the scales: the experts' rows and tiles, and what a wave knows of its next tile's rows.
constexpr int kTables = kUnit * kRing + 3 * kScaleSlot, kStash = kTables + 2 * kDualExperts * 4;
constexpr int kDualLds = kStash + 5 * 4 * kDualThreads;
constexpr uint32_t kNoRow = 0x80000000u;  // a byte offset past every operand, with offsets along K still below 2^32

struct DualArgs {
  GemmParams p;
  FewRowsArgs few;
};

#if defined(__HIP_DEVICE_COMPILE__)

#define FLUXMI_VMCNT(vm) __builtin_amdgcn_s_waitcnt(((vm)&15) | (((vm) >> 4) << 14) | (7 << 4) | (15 << 8))
#define FLUXMI_LGKM0() __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4) | (0 << 8))

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(3))) i32x4 *LdsFrag;

// Where a work item lies: rows row0 .. row0 + rows of the sorted rows (rows <= 256; 0: there is no such item), columns n0 .. of weight
// group g.  wide: columns beyond the tile's first 128 exist and belong to the item.
struct DualTile {
  int e, row0, rows, g, n0;
  bool wide, alone;    // alone: its expert has no other row tile
  int e_row0, e_rows;  // the expert's rows
};

template <int FIRST, class F, int... I>
__device__ __forceinline__ void static_for_seq(F &f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, FIRST + I>{}), ...);
}
template <int FIRST, int END, class F>
__device__ __forceinline__ void static_for(F &&f) {
  if constexpr (FIRST < END) static_for_seq<FIRST>(f, std::make_integer_sequence<int, END - FIRST>{});
}

// One block of 16 x 16 over 64 (16-bit elements, half h of a step) or 128 bytes of K, added to c.
template <Elem T>
__device__ __forceinline__ f32x4 mfma_block(const i32x4 (&w)[2], const i32x4 (&x)[2], int h, f32x4 c) {
  if constexpr (is_fp8(T)) {
    const i32x8 wa = {w[0][0], w[0][1], w[0][2], w[0][3], w[1][0], w[1][1], w[1][2], w[1][3]};
    const i32x8 xa = {x[0][0], x[0][1], x[0][2], x[0][3], x[1][0], x[1][1], x[1][2], x[1][3]};
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wa, xa, c, 0, 0, 0, 0, 0, 0);
  } else if constexpr (T == Elem::F16) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w[h]), __builtin_bit_cast(f16x8, x[h]), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[h]), __builtin_bit_cast(bf16x8, x[h]), c, 0, 0, 0);
  }
}

// 64 rows (four blocks, from I0 on) x 32 columns (two blocks, from J0 on) over 128 bytes of K.
template <Elem T, bool FIRST, int I0, int J0>
__device__ __forceinline__ void quadrant(f32x4 (&acc)[8][4], const i32x4 (&x)[4][2], const i32x4 (&w)[4][2], const float (&scale)[4]) {
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  if constexpr (T == Elem::FP8_BLOCKSCALED) {
    constexpr int DIST = 3;  // MFMAs between a block's and its promotion (2: the compiler's wait states in between are exposed)
    f32x4 part[8];
    auto promote = [&](auto M) {
      constexpr int m = decltype(M)::value, i = m / 2, j = m % 2;
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[I0 + i][J0 + j][v] = fmaf(part[m][v], scale[i], FIRST ? 0.f : acc[I0 + i][J0 + j][v]);
      asm volatile("" : "+v"(acc[I0 + i][J0 + j]));  // here, not where the sums are next used: the block's registers are needed again
    };
    static_for<0, 8>([&](auto M) {
      constexpr int m = decltype(M)::value;
      part[m] = mfma_block<T>(w[J0 + m % 2], x[m / 2], 0, zero);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (m >= DIST) promote(std::integral_constant<int, (m >= DIST ? m - DIST : 0)>{});
      __builtin_amdgcn_sched_barrier(0);
    });
    static_for<8 - DIST, 8>(promote);
  } else {
    // (16-bit: the halves of a step in ascending order, which are the macro tiles' sums.)
#pragma unroll
    for (int h = 0; h < (is_fp8(T) ? 1 : 2); ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[I0 + i][J0 + j] = mfma_block<T>(w[J0 + j], x[i], h, FIRST && h == 0 ? zero : acc[I0 + i][J0 + j]);
  }
}

template <Elem T>
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  if constexpr (T == Elem::F16) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    const f16x2 h = {static_cast<_Float16>(lo), static_cast<_Float16>(hi)};
    return __builtin_bit_cast(uint32_t, h);
  } else {
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
  }
}

// The kernel's argument, read again where it is used; the empty asm keeps the compiler from keeping copies in registers through the loop.
typedef const __attribute__((address_space(4))) DualArgs *DualArgSegment;
typedef const __attribute__((address_space(4))) GemmParams *KernArgs;
typedef const __attribute__((address_space(4))) FewRowsArgs *FewArgs;
__device__ __forceinline__ DualArgSegment all_args() {
  DualArgSegment k = (DualArgSegment)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(k));
  return k;
}
__device__ __forceinline__ KernArgs kernel_args() { return &all_args()->p; }
__device__ __forceinline__ FewArgs few_args() { return &all_args()->few; }

// The lane, opaque to the compiler: what is computed from it is not moved out of the tile loop, where it would occupy registers.
__device__ __forceinline__ int fresh_lane() {
  int l = lane_id();
  asm volatile("" : "+v"(l));
  return l;
}

#endif  // __HIP_DEVICE_COMPILE__

template <Elem T>
__global__ __launch_bounds__(kDualThreads, 2) void grouped_gemm_dual_kernel(const DualArgs args) {
#if defined(__HIP_DEVICE_COMPILE__)
  const GemmParams &p = args.p;
  extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
  constexpr bool BS = T == Elem::FP8_BLOCKSCALED;
  constexpr int ELT = is_fp8(T) ? 1 : 2;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int kbytes = p.k * ELT, steps = kbytes >> 7;
  const int tiles_n1 = (p.n + kTile - 1) / kTile, tiles_n = tiles_n1 * p.ngroups;
  const int grid = gridDim.x, bid = blockIdx.x;
  const int virt = (grid & 7) == 0 ? (bid & 7) * (grid >> 3) + (bid >> 3) : bid;

  // ---- the experts: rows and tiles up to each of them, in LDS (registers are short) --------------------------
  typedef __attribute__((address_space(3))) int *LdsInt;
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) uint8_t *)smem));
  const LdsInt row_ends = reinterpret_cast<LdsInt>(lds0 + kTables), tile_ends = row_ends + kDualExperts;
  int total_tiles;
  {
    int row_carry = 0, tile_carry = 0, chunks = 0, active = 0;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int ee = c * 64 + lane;
      int r = 0;
      if (ee < p.nexperts) r = few_args()->count > 0 ? few_args()->splits[ee] : p.splits[ee];
      if (r < 0) r = 0;
      const int incl = wave_inclusive_scan(r);
      int begin = row_carry + incl - r, end = row_carry + incl;
      if (begin > p.max_rows) begin = p.max_rows;
      if (end > p.max_rows) end = p.max_rows;
      row_ends[ee] = end;  // (the same from every wave)
      row_carry += __builtin_amdgcn_readlane(incl, 63);
      if (p.by_splits) {
        active += __popcll(__ballot(end > begin));
        chunks += __builtin_amdgcn_readlane(wave_inclusive_scan((end - begin + p.by_splits - 1) >> (31 - __builtin_clz(p.by_splits))), 63);
      }
      const int tile_end = tile_carry + wave_inclusive_scan(((end - begin + kTile - 1) / kTile) * tiles_n);
      tile_ends[ee] = tile_end;
      tile_carry = __builtin_amdgcn_readlane(tile_end, 63);
    }
    // (another form runs this launch)
    if (p.by_splits && chunks <= stream_chunks_limit(active, p.by_splits, is_fp8(T), p.chunk_items, p.round_items)) return;
    total_tiles = tile_carry;
  }
  // Full rounds run whole tiles; the tiles of the last, partly filled round are cut into two or four pieces when they still fit it.
  const int full_items = total_tiles / grid * grid, rem = total_tiles - full_items;
  const int pieces = (p.sched_flags & FLUXMI_SCHED_WHOLE_TAIL_TILES) != 0 ? 1 : (rem * 4 <= grid ? 4 : (rem * 2 <= grid ? 2 : 1));
  const int total_items = full_items + rem * pieces;

  auto locate = [&](int item) {
    const KernArgs a = kernel_args();
    const int n = a->n, raster = a->raster_rows;
    DualTile t = {0, 0, 0, 0, 0, false, false, 0, 0};
    // A launch of one round that is not full deals its items to the eight XCDs evenly.
    if (full_items == 0 && (grid & 7) == 0) {
      const int per_xcd = (total_items + 7) >> 3, xcd = item / (grid >> 3), i = item - xcd * (grid >> 3);
      if (xcd > 7 || i >= per_xcd) return t;
      item = __builtin_amdgcn_readfirstlane(xcd * per_xcd + i);
    }
    if (item >= total_items) return t;
    int tile = item, piece = 0;
    if (item >= full_items) {
      const int i = item - full_items;
      tile = full_items + (pieces == 4 ? i >> 2 : (pieces == 2 ? i >> 1 : i));
      piece = i & (pieces - 1);
    }
    const int l = fresh_lane();
    int c = 0, end_of_lane = tile_ends[l];
    uint64_t hit = __ballot(tile < end_of_lane);
    if (hit == 0) {
      c = 64;
      end_of_lane = tile_ends[64 + l];
      hit = __ballot(tile < end_of_lane);
    }
    const int src = __ffsll(static_cast<unsigned long long>(hit)) - 1;
    t.e = c + src;
    const int end_tile = __builtin_amdgcn_readlane(end_of_lane, src);
    const int end_row = __builtin_amdgcn_readfirstlane(row_ends[t.e]);
    const int begin_row = t.e > 0 ? __builtin_amdgcn_readfirstlane(row_ends[t.e - 1]) : 0;
    const int tiles_n1 = (n + kTile - 1) / kTile, tiles_n = tiles_n1 * a->ngroups;
    const int rows_e = end_row - begin_row, m_tiles = (rows_e + kTile - 1) / kTile;
    const int local = tile - (end_tile - m_tiles * tiles_n);
    // Groups of at most `raster` row tiles, each walked column by column, as the macro tiles do.
    const int ngroups_m = (m_tiles + raster - 1) / raster;
    const int gm = (m_tiles + ngroups_m - 1) / ngroups_m;
    const int group = local / (gm * tiles_n), group_first = group * gm;
    const int group_rows = m_tiles - group_first < gm ? m_tiles - group_first : gm;
    const int in_group = local - group * gm * tiles_n;
    const int nt = __builtin_amdgcn_readfirstlane(in_group / group_rows);
    const int mt = __builtin_amdgcn_readfirstlane(group_first + (in_group - nt * group_rows));
    t.g = a->ngroups > 1 ? __builtin_amdgcn_readfirstlane(nt / tiles_n1) : 0;
    t.n0 = (nt - t.g * tiles_n1) * kTile;
    // An expert's rows are dealt to its tiles in units of 64, what a wave has of a phase, as evenly as they go.
    const int units = (rows_e + 63) / 64, per = __builtin_amdgcn_readfirstlane(units / m_tiles), longer = units - per * m_tiles;
    int m0 = 64 * (mt * per + (mt < longer ? mt : longer));
    const int height = 64 * (per + (mt < longer ? 1 : 0));
    t.rows = rows_e - m0 < height ? rows_e - m0 : height;
    if (pieces > 1 && item >= full_items) {
      t.n0 += (piece & 1) * 128;
      if (pieces == 4) {
        m0 += (piece >> 1) * 128;
        t.rows = (piece >> 1) != 0 ? t.rows - 128 : (t.rows < 128 ? t.rows : 128);
      }
    } else {
      t.wide = n - t.n0 > 128;
    }
    t.row0 = begin_row + m0;
    t.e_row0 = begin_row;
    t.e_rows = rows_e;
    t.alone = m_tiles == 1;
    if (t.n0 >= n) t.rows = -1;  // (a piece without columns, or rows)
    if (t.rows <= 0) t.rows = -1;
    return t;
  };
  // Pieces without work are passed over.
  int next_item = virt;
  auto next_tile = [&]() {
    DualTile t;
    do {
      t = locate(next_item);
      next_item += grid;
    } while (t.rows < 0);
    return t;
  };

  // ---- ring fills ------------------------------------------------------------------------------------------
  // LDS row R of a unit lies at R * 128, its 16-byte chunk c at slot c ^ ((R >> 1) & 7).  A fill covers eight rows, lane l row l >> 3
  // and slot l & 7; the four waves of a group fill a unit, wave wn rows 32 * wn + 8 * j + (l >> 3), j = 0 .. 3.
  // The units of a step are X's first half, W's first half, W's second half and X's second half (X: rows of A).  Phase f, four to a step,
  // fills unit f + 7: the first group, which reads in even phases, X's second half one step ahead and W's first two steps, the second
  // group X's first and W's second half two steps ahead.  Unit u lies in slot u mod 9: of a step's units the first three are read in
  // phases 0 (first group) and 1, the fourth in 2 and 3, so unit f + 7 - 9 has been read when phase f starts.
  const int xhalf = 1 - wm, whalf = wm;
  uint32_t xoff0, xoff1, xoff2, xoff3;  // of the producer's tile
  uint32_t nxt0, nxt1, nxt2, nxt3;      // rows of A, then offsets, of the tile after it
  // 16-bit results: a lane has columns 8 g .. 8 g + 7 in the two blocks of a group of 32 (g = lane / 16), fp32: 4 g .. in each block
  const bool f32_out = p.d_fp32 != 0;
  const uint32_t wstep1 = (f32_out ? 8u : 16u) * kbytes, wstep2 = (f32_out ? 16u : 4u) * kbytes;
  auto chunk_of = [&](int l) { return static_cast<uint32_t>(((l & 7) ^ (l >> 4)) * 16); };  // of even fills; odd ones: ^ 64
  const int row_first = xhalf * 128 + wn * 32;                 // first row of the tile that this wave fills
  uint32_t nxts = 0;  // the same for the row whose scale this lane fetches
  auto load_rows = [&](const DualTile &t) {  // requests the rows of A that X fills of tile t read
    const KernArgs a = kernel_args();
    if (a->gather_a != nullptr) {
      const int r = row_first + (fresh_lane() >> 3);
      const int32_t *src = a->gather_a + t.row0 + r;
      nxt0 = nxt1 = nxt2 = nxt3 = 0;
      if (r < t.rows) nxt0 = src[0];
      if (r + 8 < t.rows) nxt1 = src[8];
      if (r + 16 < t.rows) nxt2 = src[16];
      if (r + 24 < t.rows) nxt3 = src[24];
      if constexpr (BS) {
        const int rs = wn * 64 + fresh_lane();
        nxts = 0;
        if (rs < t.rows) nxts = a->gather_a[t.row0 + rs];
      }
    }
  };
  auto rows_to_offsets = [&](const DualTile &t) {
    const KernArgs a = kernel_args();
    const bool gathered = a->gather_a != nullptr;
    const int a_rows = a->a_rows, l = fresh_lane(), r = row_first + (l >> 3);
    const uint32_t chunk0 = chunk_of(l);
    auto offset = [&](uint32_t v, int j) {
      uint32_t row = r + 8 * j;
      if (gathered) {
        const int x = static_cast<int>(v);
        row = x < 0 ? 0 : (x >= a_rows ? a_rows - 1 : x);
      }
      return r + 8 * j < t.rows ? row * static_cast<uint32_t>(kbytes) + (chunk0 ^ ((j & 1) * 64)) : kNoRow;
    };
    nxt0 = offset(nxt0, 0);
    nxt1 = offset(nxt1, 1);
    nxt2 = offset(nxt2, 2);
    nxt3 = offset(nxt3, 3);
    if constexpr (BS) {
      const int rs = wn * 64 + l;
      int64_t row = t.row0 + rs;
      if (gathered) row = static_cast<int>(nxts) < 0 ? 0 : (static_cast<int>(nxts) >= a_rows ? a_rows - 1 : static_cast<int>(nxts));
      const uint32_t off = a->a_scale_layout == FLUXMI_ASCALE_BLOCK128
                               ? static_cast<uint32_t>(((row >> 7) * steps * 128 + (row & 127)) * 4)
                               : static_cast<uint32_t>((static_cast<int64_t>(t.e_row0) * (steps - 1) + row) * 4);
      nxts = rs < t.rows ? off : kNoRow;
    }
  };
  __amdgpu_buffer_rsrc_t xrsrc, wrsrc;
  uint32_t woff0, woff1, woff2, woff3;
  auto start_x = [&](const DualTile &t) {  // with the offsets in nxt
    const KernArgs a = kernel_args();
    const bool any = t.rows > 0, gathered = a->gather_a != nullptr;
    const int64_t xrows = !any ? 0 : (gathered ? a->a_rows : t.rows);
    xrsrc = buffer_of(gathered ? a->a : a->a + static_cast<int64_t>(t.row0) * kbytes, xrows * kbytes);
    xoff0 = nxt0, xoff1 = nxt1, xoff2 = nxt2, xoff3 = nxt3;
  };
  bool w_once = false;
  auto start_w = [&](const DualTile &t) {
    const KernArgs a = kernel_args();
    w_once = !BS && t.alone && (reinterpret_cast<uintptr_t>(a->b[t.g]) & 127) == 0;
    wrsrc = buffer_of(a->b[t.g] + (static_cast<int64_t>(t.e) * a->n + t.n0) * kbytes, t.rows > 0 ? static_cast<int64_t>(a->n - t.n0) * kbytes : 0);
    // Fill 0's first column; the others' lie 8, 16, 24 further on, or in the order of 16-bit results.
    const uint32_t cols = t.wide ? wn * 64 + whalf * 32 : wn * 32, wbase = !t.wide && whalf != 0 ? kNoRow : cols * kbytes;
    const int l = fresh_lane(), r = l >> 3, col = f32_out ? r : (r >> 2) * 8 + (r & 3);
    const uint32_t w0 = static_cast<uint32_t>(col) * kbytes + wbase, chunk0 = chunk_of(l);
    woff0 = w0 + chunk0;
    woff1 = w0 + wstep1 + (chunk0 ^ 64);
    woff2 = w0 + wstep2 + chunk0;
    woff3 = w0 + wstep1 + wstep2 + (chunk0 ^ 64);
  };
  const LdsInt stash = reinterpret_cast<LdsInt>(lds0 + kStash);
  auto put_next = [&]() {
    const int t = wave * 64 + fresh_lane();
    stash[t] = nxt0, stash[512 + t] = nxt1, stash[1024 + t] = nxt2, stash[1536 + t] = nxt3;
    if constexpr (BS) stash[2048 + t] = nxts;
  };
  auto get_next = [&]() {
    const int t = wave * 64 + fresh_lane();
    nxt0 = stash[t], nxt1 = stash[512 + t], nxt2 = stash[1024 + t], nxt3 = stash[1536 + t];
    if constexpr (BS) nxts = stash[2048 + t];
  };
  uint32_t soff = 0;   // block scales: of the scale that this lane of the first group fetches
  int sstep = 0;       // ... and their distance between steps
  auto start_scales = [&](const DualTile &t) {
    const KernArgs a = kernel_args();
    soff = nxts;
    sstep = a->a_scale_layout == FLUXMI_ASCALE_BLOCK128 ? 512 : t.e_rows * 4;
  };
  const uint32_t fill0 = lds0 + wn * 4096;
  // Four fills of one unit, 1 KiB of LDS apart.  The first load comes five wait states after the statement's start: what a scalar register needs
  // that a vector instruction wrote (v_readlane, with which the compiler brings back spilled ones), and it does not look into asm for that.
  // (Costs 0.6 % of launches of up to 64 tiles, 0.3 % of a layer's pass.)
#define FLUXMI_FILL_UNIT(MOD)                                                                                    \
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %5, %6 offen " MOD "lds\n\t"             \
               "s_add_u32 m0, %0, 0x400\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %5, %6 offen " MOD "lds\n\t"      \
               "s_add_u32 m0, %0, 0x800\n\ts_nop 0\n\tbuffer_load_dwordx4 %3, %5, %6 offen " MOD "lds\n\t"      \
               "s_add_u32 m0, %0, 0xc00\n\ts_nop 0\n\tbuffer_load_dwordx4 %4, %5, %6 offen " MOD "lds"          \
               : : "s"(dst), "v"(o0), "v"(o1), "v"(o2), "v"(o3), "s"(r), "s"(kb) : "memory", "scc")
  auto fill_unit = [&](bool once, __amdgpu_buffer_rsrc_t r, uint32_t dst, uint32_t o0, uint32_t o1, uint32_t o2, uint32_t o3, int kb) {
    if (once) FLUXMI_FILL_UNIT("nt ");
    else FLUXMI_FILL_UNIT("");
  };
#undef FLUXMI_FILL_UNIT
  auto fill_x = [&](uint32_t slot, int kb) { fill_unit(false, xrsrc, fill0 + slot, xoff0, xoff1, xoff2, xoff3, kb); };
  // Weights of an expert that is one row tile come non-temporally, where rows start on lines (a load that covers parts of two lines needs the
  // second again): 3 to 5 % up to 256 rows per expert (fp16 32 experts 2048 x 4096, 194 rows each 145 -> 127 us, 8 experts 14336 x 4096 250 ->
  // 237, 4096 x 14336 312 -> 297; fp8 32 experts 2048 x 7168 110 -> 91).  Block-scaled launches gain nothing and lose 1 % by the branch.
  // Where the tile of such an expert is cut in four, two workgroups read each weight, and still do so non-temporally: ordinary loads there are 0.4 %
  // slower (8003 launches of up to 64 tiles, 120 to 260 rows per expert; 199 slower by more than 3 %, 47 as much faster).
  auto fill_w = [&](uint32_t slot, int kb) { fill_unit(!BS && w_once, wrsrc, fill0 + slot, woff0, woff1, woff2, woff3, kb); };

  // ---- fragments -------------------------------------------------------------------------------------------
  i32x4 x[4][2], w[4][2];
  uint32_t xread[2], wread[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const uint32_t chunk = ((c * 4 + (lane >> 4)) ^ ((lane >> 1) & 7)) * 16;
    xread[c] = lds0 + (wm * 64 + (lane & 15)) * 128 + chunk;
    wread[c] = lds0 + (wn * 32 + (lane & 15)) * 128 + chunk;
  }
  const uint32_t sread = lds0 + kRing * kUnit + (wm * 64 + (lane & 15)) * 4;  // row scales of this lane
  // (An opaque address: the distance of the blocks goes into the instructions.)
  auto address = [&](uint32_t at, uint32_t slot) {
    uint32_t a = at + slot;
    asm volatile("" : "+v"(a));
    return reinterpret_cast<__attribute__((address_space(3))) uint8_t *>(a);
  };
  auto read_x = [&](uint32_t slot) {
    const auto a = address(xread[0], slot), b = address(xread[1], slot);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x[i][0] = *reinterpret_cast<LdsFrag>(a + i * 2048);
      x[i][1] = *reinterpret_cast<LdsFrag>(b + i * 2048);
    }
  };
  auto read_w = [&](uint32_t slot, int j0) {
    const auto a = address(wread[0], slot), b = address(wread[1], slot);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      w[j0 + j][0] = *reinterpret_cast<LdsFrag>(a + j * 2048);
      w[j0 + j][1] = *reinterpret_cast<LdsFrag>(b + j * 2048);
    }
  };
  // Unit U lies in slot U mod 9.  base: unit number of the current step's first unit, mod 9.
  auto slot_of = [&](int u) { return static_cast<uint32_t>(u >= kRing ? u - kRing : u) * kUnit; };
  auto sync = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // ---- first tile ------------------------------------------------------------------------------------------
  DualTile cur = next_tile();
  if (cur.rows == 0) return;
  load_rows(cur);
  rows_to_offsets(cur);
  start_x(cur);
  start_w(cur);
  if constexpr (BS) start_scales(cur);
  DualTile nx = next_tile();
  // Row scales of step st into slot st mod 3 (of the launch's steps).
  auto fill_scales = [&](uint32_t slot, int st) {
    const uint8_t *const src = reinterpret_cast<const uint8_t *>(kernel_args()->a_scale) + static_cast<int64_t>(st) * sstep;
    const __amdgpu_buffer_rsrc_t r = buffer_of(src, kNoRow);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dword %1, %2, 0 offen lds"
                 : : "s"(lds0 + kRing * kUnit + slot * kScaleSlot + wn * 256), "v"(soff), "s"(r) : "memory");
  };
  for (int s = 0; s < 2; ++s) {  // units 0 to 6
    if (wm == 0) {
      fill_w(slot_of(4 * s + 1), s * 128);
      if (s == 0) fill_x(slot_of(3), 0);
      if constexpr (BS) fill_scales(s, s);
    } else {
      fill_x(slot_of(4 * s), s * 128);
      fill_w(slot_of(4 * s + 2), s * 128);
    }
  }
  load_rows(nx);
  float scalar = p.scalar;
  if (p.scalar_dev) scalar *= p.scalar_dev[0];
  DualTile nx2 = next_tile();
  FLUXMI_VMCNT(0);
  rows_to_offsets(nx);
  put_next();
  sync();
  if (wm != 0) sync();  // the second group runs one phase behind the first
  int base = 0, scale_slot = 0;

  while (true) {
    f32x4 acc[8][4];
    const bool wide = cur.wide;
    const int rows0 = cur.rows - wm * 64;  // rows of the tile from this wave's first on; 128 further on lies its second half
    // B's scales of this wave's columns.
    int bs_index = 0, bs_step = 0;
    if constexpr (BS) {
      const KernArgs a = kernel_args();
      const int nblocks = (a->n + 127) >> 7, first = (cur.n0 + (wide ? wn * 64 : 0)) >> 7, nb = first < nblocks ? first : nblocks - 1;
      if (a->b_scale_layout == FLUXMI_BSCALE_N_K) {
        bs_index = (cur.e * nblocks + nb) * steps;
        bs_step = 1;
      } else {
        bs_index = cur.e * steps * nblocks + nb;
        bs_step = nblocks;
      }
    }
    auto step = [&](auto FIRSTSTEP, int s) {
      constexpr bool FS = decltype(FIRSTSTEP)::value;
      // The steps of K whose X and W this wave requests.
      int fw = s + 2, fx = s + 1 + wm;
      if (fw >= steps) {
        fw -= steps;
        if (fw == 0) {
          start_w(nx);
          if (BS && wm == 0) {
            get_next();
            start_scales(nx);
          }
        }
      }
      if (fx >= steps) {
        fx -= steps;
        if (fx == 0) {
          get_next();
          start_x(nx);
        }
      }
      float scale[4], bscale = 1.f;
      if constexpr (BS) {
        typedef const __attribute__((address_space(4))) float *ConstF32;
        bscale = ((ConstF32)(kernel_args()->b_scale))[bs_index];
        bs_index += bs_step;
      }
      auto read_scales = [&](int half) {
        if constexpr (BS) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            scale[i] = *reinterpret_cast<const __attribute__((address_space(3))) float *>(sread + scale_slot * kScaleSlot + half * 512 + i * 64);
        }
      };
      auto scale_rows = [&]() {
        if constexpr (BS) {
#pragma unroll
          for (int i = 0; i < 4; ++i) scale[i] *= bscale;
        }
      };
      // What the waits count: a unit's fills are four instructions of a wave, and with block scales the first group's fills of a step's row
      // scales, one each, follow those of X.  The first steps of a tile were waited for at its start.
      // Read: the first half's rows, all columns.  Reads before fills: the phase ends when the last of them is issued.
      read_x(slot_of(base));
      read_w(slot_of(base + 1), 0);
      read_w(slot_of(base + 2), 2);
      read_scales(0);
      fill_x(slot_of(base + 7 + wm), fx * 128);
      if (BS && wm == 0) fill_scales(scale_slot == 0 ? 2 : scale_slot - 1, fw);
      FLUXMI_LGKM0();
      scale_rows();
      sync();
      __builtin_amdgcn_s_setprio(1);
      if (rows0 > 0) {
        quadrant<T, FS, 0, 0>(acc, x, w, scale);
        if (wide) quadrant<T, FS, 0, 2>(acc, x, w, scale);
      }
      __builtin_amdgcn_s_setprio(0);
      if (wm == 0 && s > 0) FLUXMI_VMCNT(BS ? 10 : 8);  // X's second half, requested in the step before: two units, and scales, since
      sync();
      // Read: the second half's rows.
      read_x(slot_of(base + 3));
      read_scales(1);
      fill_w(slot_of(base + wm), fw * 128);
      if (wm != 0 && s > 0) FLUXMI_VMCNT(8);  // the next step's X and W, requested two units ago and before
      FLUXMI_LGKM0();
      scale_rows();
      sync();
      __builtin_amdgcn_s_setprio(1);
      if (rows0 > 128) {
        quadrant<T, FS, 4, 0>(acc, x, w, scale);
        if (wide) quadrant<T, FS, 4, 2>(acc, x, w, scale);
      }
      __builtin_amdgcn_s_setprio(0);
      if (wm == 0 && s > 0) FLUXMI_VMCNT(BS ? 9 : 8);  // the next step's W, requested in the step before: the same
      base = base + 4 >= kRing ? base + 4 - kRing : base + 4;
      scale_slot = scale_slot == 2 ? 0 : scale_slot + 1;
      if (wm == 0 || s + 1 < steps) sync();
    };
    step(std::true_type{}, 0);
    for (int s = 1; s < steps; ++s) step(std::false_type{}, s);

    // ---- epilogue ------------------------------------------------------------------------------------------
    FLUXMI_VMCNT(0);  // the next tile's first units; this wave's, the others' by the barriers
    load_rows(nx2);
    rows_to_offsets(nx2);
    put_next();
    {
      const KernArgs a = kernel_args();
      const int lane = fresh_lane(), n = a->n;
      const float *alpha = a->alpha[cur.g], *row_scale = a->row_scale, *row_scale2 = few_args()->row_scale2, *col_scale = a->col_scale;
      const int32_t *scatter = a->scatter_d;
      const float tile_scale = scalar * (alpha ? alpha[cur.e] : 1.f);
      const bool f32 = a->d_fp32 != 0, nt = a->nt_stores != 0;
      const int cgrp = lane >> 4, rows = cur.rows - wm * 64 - (lane & 15);  // block i has a row of this lane if its first row is below that
      const int col0 = cur.n0 + (wide ? wn * 64 : wn * 32);                 // first column of group 0; group 1: 32 further
      const int first_row = cur.row0 + wm * 64 + (lane & 15);
      // Everything that is read, before the first store: a load behind stores waits until those have drained.
      int cols[4];  // first column of this lane in block j
      float4 cs[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        cols[j] = col0 + (j >> 1) * 32 + (f32 ? (j & 1) * 16 + cgrp * 4 : cgrp * 8 + (j & 1) * 4);
        cs[j] = make_float4(1.f, 1.f, 1.f, 1.f);
        if (col_scale != nullptr && cols[j] < n && (j < 2 || wide))
          cs[j] = *reinterpret_cast<const float4 *>(col_scale + static_cast<int64_t>(cur.e) * n + cols[j]);
      }
      float rs[8];
      int out_row[8];  // -1: not stored
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int m = (i >> 2) * 128 + (i & 3) * 16;
        rs[i] = 1.f;
        out_row[i] = m < rows ? first_row + m : -1;
        if (row_scale != nullptr && m < rows) rs[i] = row_scale[first_row + m];
        if (row_scale2 != nullptr && m < rows) rs[i] *= row_scale2[first_row + m];
        if (scatter != nullptr && m < rows) {
          const int to = scatter[first_row + m];
          out_row[i] = to < a->d_rows ? to : -1;
        }
      }
      uint8_t *const d = static_cast<uint8_t *>(a->d[cur.g]);
      const int64_t row_bytes = static_cast<int64_t>(n) * (f32 ? 4 : 2);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if (i >= 4 && rows0 <= 128) break;
        const float scale = tile_scale * rs[i];
        uint8_t *const drow = d + out_row[i] * row_bytes;
#pragma unroll
        for (int jg = 0; jg < 2; ++jg) {
          if (jg == 1 && !wide) break;
          f32x4 v[2];
#pragma unroll
          for (int j2 = 0; j2 < 2; ++j2) {
            const int j = jg * 2 + j2;
            v[j2] = acc[i][j] * scale;
            if (col_scale != nullptr) v[j2] = f32x4{v[j2][0] * cs[j].x, v[j2][1] * cs[j].y, v[j2][2] * cs[j].z, v[j2][3] * cs[j].w};
          }
          if (out_row[i] < 0) continue;
          if (f32) {
#pragma unroll
            for (int j2 = 0; j2 < 2; ++j2) {
              const int j = jg * 2 + j2;
              if (cols[j] >= n) continue;
              f32x4 *const dst = reinterpret_cast<f32x4 *>(drow + static_cast<int64_t>(cols[j]) * 4);
              if (nt) __builtin_nontemporal_store(v[j2], dst);
              else *dst = v[j2];
            }
          } else if (cols[jg * 2] < n) {
            const u32x4 o = {pack2<T>(v[0][0], v[0][1]), pack2<T>(v[0][2], v[0][3]), pack2<T>(v[1][0], v[1][1]), pack2<T>(v[1][2], v[1][3])};
            *reinterpret_cast<u32x4 *>(drow + static_cast<int64_t>(cols[jg * 2]) * 2) = o;
          }
        }
      }
    }
    // The second group ends its last phase with its results stored: the groups' stores are one pause, not two (2 to 4 %).
    if (nx.rows == 0) {
      sync();
      break;
    }
    cur = nx;
    nx = nx2;
    nx2 = next_tile();
    if (wm != 0) sync();
  }
  FLUXMI_VMCNT(0);
#endif  // __HIP_DEVICE_COMPILE__
}

template <Elem T>
int launch(const GemmParams &p, const FewRowsArgs &few, int grid, hipStream_t s) {
  static std::atomic<uint64_t> lds_done{0};
  const int rc = ensure_dynamic_lds(reinterpret_cast<const void *>(grouped_gemm_dual_kernel<T>), kDualLds, lds_done);
  if (rc != FLUXMI_OK) return rc;
  hipLaunchKernelGGL(grouped_gemm_dual_kernel<T>, dim3(grid), dim3(kDualThreads), kDualLds, s, DualArgs{p, few});
  return FLUXMI_OK;
}

}  // namespace

// Whole steps of K, at least two; offsets below kNoRow; 16-bit results in stores of 16 bytes.
bool dual_takes(const GemmParams &p, int dtype) {
  const int64_t kbytes = static_cast<int64_t>(p.k) * (dtype == FLUXMI_FP8_E4M3 ? 1 : 2), span = 0x70000000ll;
  if (p.accumulate || p.nexperts > kDualExperts || kbytes % 128 != 0 || kbytes < 256) return false;
  if (kTile * kbytes > span || p.n * kbytes > span || (p.gather_a != nullptr && p.a_rows * kbytes > span)) return false;
  const int64_t scale_rows = p.gather_a != nullptr ? p.a_rows : p.max_rows;
  if (p.a_scale != nullptr && (scale_rows + 127) / 128 * 128 * (kbytes / 128) * 4 > span) return false;
  if (p.d_fp32) return true;
  bool aligned = p.n % 8 == 0;
  for (int g = 0; g < p.ngroups; ++g) aligned = aligned && aligned16(p.d[g]);
  return aligned;
}

int launch_grouped_gemm_dual(const GemmParams &p, const FewRowsArgs &few, int dtype, int grid, hipStream_t s) {
  if (p.a_scale != nullptr) return launch<Elem::FP8_BLOCKSCALED>(p, few, grid, s);
  if (dtype == FLUXMI_FP8_E4M3) return launch<Elem::FP8>(p, few, grid, s);
  if (dtype == FLUXMI_FP16) return launch<Elem::F16>(p, few, grid, s);
  return launch<Elem::BF16>(p, few, grid, s);
}

}  // namespace fluxmi
