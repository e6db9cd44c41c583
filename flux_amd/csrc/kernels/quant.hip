// bf16 -> fp8-e4m3 absmax quantisation with one scale per row, per (row, 128-column block) or per
// 128 x 128 block (with an optional transposed copy of the bytes).
//
// HBM-streaming kernel: one read of x (2 B/elt), one write of q (1 B/elt).  A row (or row block) is
// held in registers between the amax pass and the cast pass, so x is fetched exactly once.
#include "common.hpp"

namespace fluxmi {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr float kE4M3Max = 448.f;

// scale = 448 / max(amax, eps) with the special cases of the reference's ComputeScale
// (src/quantization/quantization.cu:306-367, bf16 input type, no power-of-two rounding).
__device__ __forceinline__ float compute_scale(float amax, float eps) {
  const float a = fmaxf(amax, eps);
  if (a == 0.f) return 1.f;
  const float s = kE4M3Max / a;  // IEEE fp32 division
  if (__builtin_isinf(s)) return 0x1.FEp127f;
  return s;  // includes s == 0 when amax is +inf
}

// fp8 codes of two values times their scale, in the low (HIGH: the high) half of `old`: v_cvt_pk_fp8_f32 (OCP e4m3 on
// gfx950, round to nearest even).  No clamp is needed: every value is at most the amax that its scale was made from, so
// the product is at most 448 * (1 + 2^-22), which rounds to 448, or (an infinity times the scale 0, a NaN) a NaN.
template <bool HIGH>
__device__ __forceinline__ uint32_t pack2_e4m3(float lo, float hi, uint32_t old) {
  return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(lo, hi, static_cast<int>(old), HIGH));
}
__device__ __forceinline__ uint32_t pack4_e4m3(float a, float b, float c, float d) {
  return pack2_e4m3<true>(c, d, pack2_e4m3<false>(a, b, 0u));
}

// Maxima of |x| are taken on packed pairs of keys, one per bf16 value: its bits without the sign, plus 0x7f, compared as
// signed 16-bit numbers.  For finite values and infinity (0x7f80 -> 0x7fff) that is the numeric order; every NaN,
// signalling ones included, wraps to a negative key and loses against the key of zero that each maximum starts from, so it
// is skipped exactly as CUDA's fmaxf skips it.  Three instructions for two values (two conversions, two
// NaN tests and two maxima took nine).
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef int16_t i16x2 __attribute__((ext_vector_type(2)));
constexpr uint32_t kZeroKeys = 0x007f007fu;
__device__ __forceinline__ uint32_t abs_keys(uint32_t pair) {
  const u16x2 a = __builtin_bit_cast(u16x2, pair & 0x7fff7fffu);
  const u16x2 k = a + __builtin_bit_cast(u16x2, kZeroKeys);
  return __builtin_bit_cast(uint32_t, k);
}
__device__ __forceinline__ uint32_t max_keys(uint32_t a, uint32_t b) {
  const i16x2 m = __builtin_elementwise_max(__builtin_bit_cast(i16x2, a), __builtin_bit_cast(i16x2, b));
  return __builtin_bit_cast(uint32_t, m);
}
__device__ __forceinline__ uint32_t max_keys8(const u32x4 v) {
  return max_keys(max_keys(abs_keys(v[0]), abs_keys(v[1])), max_keys(abs_keys(v[2]), abs_keys(v[3])));
}
// The larger key of a pair (never below zero's), as an fp32 value.
__device__ __forceinline__ float key_to_float(uint32_t key) { return __uint_as_float((key - 0x7fu) << 16); }
__device__ __forceinline__ uint32_t larger_of_pair(uint32_t keys) { return max_keys(keys, keys >> 16) & 0xffffu; }

// Maxima over the 16 lanes of a row, and over the four rows of a wave on top (every lane gets the result).
template <int CTRL>
__device__ __forceinline__ uint32_t max_dpp(uint32_t v) {
  return max_keys(v, static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xf, 0xf, true)));
}
__device__ __forceinline__ uint32_t row16_max(uint32_t v) {
  v = max_dpp<0xb1>(v);     // quad_perm [1, 0, 3, 2]
  v = max_dpp<0x4e>(v);     // quad_perm [2, 3, 0, 1]
  v = max_dpp<0x141>(v);    // row_half_mirror: the other quad of eight lanes
  return max_dpp<0x140>(v);  // row_mirror: the other eight lanes of sixteen
}
__device__ __forceinline__ uint32_t across_rows_max(uint32_t v) {
  const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  v = max_keys(a[0], a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return max_keys(b[0], b[1]);
}
__device__ __forceinline__ uint32_t wave_max(uint32_t v) { return across_rows_max(row16_max(v)); }

__device__ __forceinline__ float bf16_lo(uint32_t pair) { return __uint_as_float(pair << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t pair) { return __uint_as_float(pair & 0xffff0000u); }

__device__ __forceinline__ u32x2 cast8(const u32x4 v, const float scale) {
  u32x2 o;
#pragma unroll
  for (int h = 0; h < 2; ++h)
    o[h] = pack4_e4m3(bf16_lo(v[2 * h]) * scale, bf16_hi(v[2 * h]) * scale, bf16_lo(v[2 * h + 1]) * scale,
                      bf16_hi(v[2 * h + 1]) * scale);
  return o;
}

// ---- one scale per row -------------------------------------------------------------------------
// THREADS_PER_ROW lanes (64, 128 or 256) cooperate on one row; a 256-thread workgroup therefore
// handles 256/THREADS_PER_ROW rows.  Each lane keeps up to VPT 16-byte vectors in registers.
template <int THREADS_PER_ROW, int VPT>
__global__ __launch_bounds__(256) void quant_row_kernel(const uint16_t *__restrict__ x, int64_t rows,
                                                        int32_t nvec, float eps,
                                                        uint8_t *__restrict__ q,
                                                        float *__restrict__ scale_inv) {
  constexpr int kRowsPerBlock = 256 / THREADS_PER_ROW;
  constexpr int kWavesPerRow = THREADS_PER_ROW / 64;
  __shared__ uint32_t s_amax[4];
  const int sub = threadIdx.x / THREADS_PER_ROW;
  const int tid = threadIdx.x % THREADS_PER_ROW;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kRowsPerBlock + sub;
  const bool row_ok = row < rows;
  const u32x4 *src = reinterpret_cast<const u32x4 *>(x) + (row_ok ? row : 0) * nvec;

  u32x4 v[VPT];
  uint32_t m = kZeroKeys;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int c = tid + i * THREADS_PER_ROW;
    v[i] = u32x4{0u, 0u, 0u, 0u};
    if (row_ok && c < nvec) v[i] = __builtin_nontemporal_load(src + c);
    m = max_keys(m, max_keys8(v[i]));
  }
  m = wave_max(m);
  if constexpr (kWavesPerRow > 1) {
    const int wave = threadIdx.x / 64;
    if ((threadIdx.x & 63) == 0) s_amax[wave] = m;
    __syncthreads();
    const int w0 = sub * kWavesPerRow;
#pragma unroll
    for (int w = 0; w < kWavesPerRow; ++w) m = max_keys(m, s_amax[w0 + w]);
  }
  const float scale = compute_scale(key_to_float(larger_of_pair(m)), eps);
  if (!row_ok) return;
  if (tid == 0) scale_inv[row] = 1.0f / scale;
  u32x2 *dst = reinterpret_cast<u32x2 *>(q) + row * nvec;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int c = tid + i * THREADS_PER_ROW;
    if (c < nvec) __builtin_nontemporal_store(cast8(v[i], scale), dst + c);
  }
}

// Rows too long for the register-resident kernel: two passes over the row (the second hits L2).
__global__ __launch_bounds__(256) void quant_row_long_kernel(const uint16_t *__restrict__ x,
                                                             int64_t rows, int32_t nvec, float eps,
                                                             uint8_t *__restrict__ q,
                                                             float *__restrict__ scale_inv) {
  __shared__ uint32_t s_amax[4];
  const int64_t row = blockIdx.x;
  const u32x4 *src = reinterpret_cast<const u32x4 *>(x) + row * nvec;
  uint32_t m = kZeroKeys;
  for (int c = threadIdx.x; c < nvec; c += 256) m = max_keys(m, max_keys8(src[c]));
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) s_amax[threadIdx.x / 64] = m;
  __syncthreads();
  m = max_keys(max_keys(s_amax[0], s_amax[1]), max_keys(s_amax[2], s_amax[3]));
  const float scale = compute_scale(key_to_float(larger_of_pair(m)), eps);
  if (threadIdx.x == 0) scale_inv[row] = 1.0f / scale;
  u32x2 *dst = reinterpret_cast<u32x2 *>(q) + row * nvec;
  for (int c = threadIdx.x; c < nvec; c += 256) dst[c] = cast8(src[c], scale);
}

// ---- one scale per (row, 128-column block) -----------------------------------------------------
// 16 consecutive lanes own one block (16 vectors of 8 elements); the amax reduction is four DPP moves
// inside that lane group.
template <int THREADS_PER_ROW>
__global__ __launch_bounds__(256) void quant_block128_kernel(const uint16_t *__restrict__ x,
                                                             int64_t rows, int32_t nvec,
                                                             int32_t nblocks, float eps,
                                                             uint8_t *__restrict__ q,
                                                             float *__restrict__ scale_inv,
                                                             int32_t permute) {
  // THREADS_PER_ROW lanes walk one row in steps of THREADS_PER_ROW vectors; blocks start at multiples
  // of 16 vectors, so the 16 lanes of a block always step together.
  constexpr int kRowsPerBlock = 256 / THREADS_PER_ROW;
  const int tid = threadIdx.x % THREADS_PER_ROW;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * kRowsPerBlock + threadIdx.x / THREADS_PER_ROW;
  if (row >= rows) return;
  const u32x4 *src = reinterpret_cast<const u32x4 *>(x) + row * nvec;
  u32x2 *dst = reinterpret_cast<u32x2 *>(q) + row * nvec;
  for (int c = tid; c < nblocks * 16; c += THREADS_PER_ROW) {
    const bool ok = c < nvec;  // a partial last block: missing vectors count as zeros
    u32x4 v = u32x4{0u, 0u, 0u, 0u};
    if (ok) v = __builtin_nontemporal_load(src + c);
    const uint32_t m = row16_max(max_keys(kZeroKeys, max_keys8(v)));
    const float scale = compute_scale(key_to_float(larger_of_pair(m)), eps);
    if ((c & 15) == 0) {
      const int blk = c >> 4;
      const float inv = 1.0f / scale;
      if (permute)
        scale_inv[(row >> 7) * (static_cast<int64_t>(nblocks) * 128) + static_cast<int64_t>(blk) * 128 +
                  (row & 127)] = inv;
      else
        scale_inv[row * nblocks + blk] = inv;
    }
    if (ok) __builtin_nontemporal_store(cast8(v, scale), dst + c);
  }
}

// ---- 128 x 128 tiles: what the two kernels below share -------------------------------------------
// One workgroup per tile.  Lane (rg, cg) = (tid / 16, tid % 16) holds the 8 x 8 patch at rows rg*8.., columns cg*8.. of
// the tile in registers: a load instruction of a wave covers 4 x 256 contiguous bytes.  A transposed copy goes through
// LDS: each lane writes the eight columns of its patch as 8-byte pieces (piece p of transposed row c at slot
// p ^ (c / 8): spreads the 16 lanes that share p over the banks), and the workgroup reads the 128 transposed rows back 16
// bytes per lane, 8 lanes per row.
struct Tile {
  int bx, by;
  int64_t batch;
};

// Tile of a workgroup: along the rows of tiles, or DOWN the columns (which the transposed output is stored along).  PER_XCD:
// workgroups are dealt to the eight XCDs round-robin, and each XCD takes a contiguous run of tiles, so that the 128-byte
// pieces of a transposed row that meet inside a cache line are put together in one L2.  Measured, 11000 x 7168
// transposed: 56 us; in plain order 58 (across) and 62 (down), per XCD across 62.  Where no line is shared the plain order is
// faster: 8192 x 7168 transposed 45.9 us (down) against 46.4, 16384 x 2048 alone 19.0 (across) against 21.1.
template <bool DOWN, bool PER_XCD>
__device__ __forceinline__ Tile tile_of_block(int32_t nbx, int32_t nby) {
  uint32_t id = blockIdx.x;
  if constexpr (PER_XCD) {
    const uint32_t per = gridDim.x >> 3, extra = gridDim.x & 7u, xcd = blockIdx.x & 7u;
    id = xcd * per + (xcd < extra ? xcd : extra) + (blockIdx.x >> 3);
  }
  const uint32_t tiles = static_cast<uint32_t>(nbx) * static_cast<uint32_t>(nby);
  Tile t;
  t.batch = id / tiles;
  const uint32_t i = id % tiles;
  t.bx = DOWN ? i / nby : i % nbx;
  t.by = DOWN ? i % nby : i / nbx;
  return t;
}

// The patch at (r0, c0); what lies outside the matrix counts as zero.  VEC: cols % 8 == 0 and an aligned x (16-byte
// loads), else element accesses.
template <bool VEC>
__device__ __forceinline__ void load_patch(const uint16_t *__restrict__ x, int64_t rows, int64_t cols, int64_t r0, int64_t c0,
                                           u32x4 (&v)[8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    v[i] = u32x4{0u, 0u, 0u, 0u};
    const int64_t r = r0 + i;
    if (r < rows) {
      if constexpr (VEC) {
        if (c0 < cols) v[i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(x + r * cols + c0));
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (c0 + e < cols) v[i][e >> 1] |= static_cast<uint32_t>(x[r * cols + c0 + e]) << ((e & 1) * 16);
      }
    }
  }
}

// Row r of the patch's codes.  VEC: 8-byte stores, else bytes.
template <bool VEC>
__device__ __forceinline__ void store_codes(uint8_t *__restrict__ q, int64_t rows, int64_t cols, int64_t r, int64_t c0, const u32x2 o) {
  if (r >= rows) return;
  if constexpr (VEC) {
    if (c0 < cols) __builtin_nontemporal_store(o, reinterpret_cast<u32x2 *>(q + r * cols + c0));
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (c0 + e < cols) q[r * cols + c0 + e] = static_cast<uint8_t>(o[e >> 2] >> ((e & 3) * 8));
  }
}

// Column j of the patch's codes into the LDS tile.
__device__ __forceinline__ void put_column(uint8_t *s_t, int rg, int cg, int j, const u32x2 t) {
  *reinterpret_cast<u32x2 *>(s_t + (cg * 8 + j) * 128 + ((rg ^ cg) * 8)) = t;
}

// The LDS tile to the transposed output, 16 bytes per lane.  WHOLE: rows % 128 == 0 and q_t aligned, so that every
// transposed row of the tile is one whole cache line, stored non-temporally.  Otherwise the address of a store may be any
// byte: global stores need no alignment on this target (the type says so to the compiler), only the matrix's last rows are
// stored as bytes, and the stores are ordinary ones, for the L2 to put neighbouring tiles' pieces of a line together
// (11000 x 7168: 56 us, non-temporal 92, byte stores 186).
typedef u32x4 u32x4_any __attribute__((aligned(1)));
template <bool WHOLE>
__device__ __forceinline__ void store_transposed(const uint8_t *s_t, uint8_t *__restrict__ q_t, int64_t rows, int64_t cols, int bx, int by) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int vid = threadIdx.x + 256 * k;
    const int trow = vid >> 3, pp = vid & 7;  // transposed row (a column of x), 16-byte unit in it
    const int tcg = trow >> 3;
    // Pieces 2pp and 2pp+1 sit in slots (2pp ^ tcg) and (2pp ^ tcg) ^ 1: one aligned 16-byte unit,
    // its halves swapped when tcg is odd.
    u32x4 d = *reinterpret_cast<const u32x4 *>(s_t + trow * 128 + (((2 * pp) ^ tcg) & ~1) * 8);
    if (tcg & 1) d = u32x4{d[2], d[3], d[0], d[1]};
    const int64_t c = static_cast<int64_t>(bx) * 128 + trow;
    const int64_t r = static_cast<int64_t>(by) * 128 + pp * 16;
    if (c >= cols || r >= rows) continue;
    uint8_t *dst = q_t + c * rows + r;
    if constexpr (WHOLE) {
      __builtin_nontemporal_store(d, reinterpret_cast<u32x4 *>(dst));
    } else if (r + 16 <= rows) {
      *reinterpret_cast<u32x4_any *>(dst) = d;
    } else {
#pragma unroll
      for (int e = 0; e < 16; ++e)
        if (r + e < rows) dst[e] = static_cast<uint8_t>(d[e >> 2] >> ((e & 3) * 8));
    }
  }
}

// 4 x 4 bytes: byte j of the four words becomes word j.
__device__ __forceinline__ void transpose4x4(uint32_t &a, uint32_t &b, uint32_t &c, uint32_t &d) {
  const uint32_t ab_lo = __builtin_amdgcn_perm(b, a, 0x05010400u), ab_hi = __builtin_amdgcn_perm(b, a, 0x07030602u);
  const uint32_t cd_lo = __builtin_amdgcn_perm(d, c, 0x05010400u), cd_hi = __builtin_amdgcn_perm(d, c, 0x07030602u);
  a = __builtin_amdgcn_perm(cd_lo, ab_lo, 0x05040100u);
  b = __builtin_amdgcn_perm(cd_lo, ab_lo, 0x07060302u);
  c = __builtin_amdgcn_perm(cd_hi, ab_hi, 0x05040100u);
  d = __builtin_amdgcn_perm(cd_hi, ab_hi, 0x07060302u);
}

// ---- one scale per 128 x 128 block, optional transposed copy -----------------------------------
// Measured with the transposed copy: 11000 x 7168 164 -> 56 us, 8192 x 7168 47.5 -> 45.9.
template <bool VEC, bool TRANSPOSE, bool WHOLE_T>
__global__ __launch_bounds__(256) void quant_square_kernel(const uint16_t *__restrict__ x, int64_t rows,
                                                           int64_t cols, int32_t nbx, int32_t nby,
                                                           float eps, uint8_t *__restrict__ q,
                                                           float *__restrict__ scale_inv,
                                                           uint8_t *__restrict__ q_t,
                                                           float *__restrict__ scale_inv_t) {
  __shared__ uint32_t s_amax[4];
  __shared__ __attribute__((aligned(16))) uint8_t s_t[TRANSPOSE ? 128 * 128 : 16];
  const Tile tile = tile_of_block<TRANSPOSE, TRANSPOSE && !WHOLE_T>(nbx, nby);
  const int cg = threadIdx.x & 15, rg = threadIdx.x >> 4;
  const int64_t r0 = static_cast<int64_t>(tile.by) * 128 + rg * 8;
  const int64_t c0 = static_cast<int64_t>(tile.bx) * 128 + cg * 8;
  const int64_t base = tile.batch * rows * cols;

  u32x4 v[8];
  load_patch<VEC>(x + base, rows, cols, r0, c0, v);
  uint32_t m = kZeroKeys;
#pragma unroll
  for (int i = 0; i < 8; ++i) m = max_keys(m, max_keys8(v[i]));
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) s_amax[threadIdx.x >> 6] = m;
  __syncthreads();
  m = max_keys(max_keys(s_amax[0], s_amax[1]), max_keys(s_amax[2], s_amax[3]));
  const float scale = compute_scale(key_to_float(larger_of_pair(m)), eps);
  if (threadIdx.x == 0) {
    const float inv = 1.0f / scale;  // fp32 division (src/quantization/quantization.cu:1117)
    scale_inv[(tile.batch * nby + tile.by) * nbx + tile.bx] = inv;
    if constexpr (TRANSPOSE) scale_inv_t[(tile.batch * nbx + tile.bx) * nby + tile.by] = inv;
  }

  u32x2 o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    o[i] = cast8(v[i], scale);
    store_codes<VEC>(q + base, rows, cols, r0 + i, c0, o[i]);
  }
  if constexpr (TRANSPOSE) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // columns 4h .. 4h+3: two 4 x 4 squares of codes
      uint32_t a[4] = {o[0][h], o[1][h], o[2][h], o[3][h]}, b[4] = {o[4][h], o[5][h], o[6][h], o[7][h]};
      transpose4x4(a[0], a[1], a[2], a[3]);
      transpose4x4(b[0], b[1], b[2], b[3]);
#pragma unroll
      for (int j = 0; j < 4; ++j) put_column(s_t, rg, cg, 4 * h + j, u32x2{a[j], b[j]});
    }
    __syncthreads();
    store_transposed<WHOLE_T>(s_t, q_t + base, rows, cols, tile.bx, tile.by);
  }
}

// ---- one scale per (row, 128-column block), optional transposed copy with its own scales --------
// Both outputs come from one read of x.  The |x| keys are made once and reduced in both directions: along a row over the
// 16 lanes of a row segment with DPP, down a column over the lane's eight rows, the four row groups of a wave (lane
// swaps) and the four waves (LDS).  Each scale and its reciprocal are divided once per tile: lane cg < 8 of a row group does
// row cg and passes the scale to the 16 lanes with a DPP broadcast, the first two waves do the columns and pass theirs through
// LDS.  (Every lane used to divide for all its eight rows and eight columns: 32 divisions a lane instead of
// four were a third of the kernel.)
// Measured, both outputs: 11000 x 7168 186 -> 56 us (5.6 TB/s; a copy of as many bytes takes 53 to 61 us), 4096 x 7168 36.8 -> 24.4, 1000 x 2048 15 -> 7;
// without the transposed output 16384 x 7168 64.5 -> 60.3, 16384 x 2048 22.6 -> 19.0.  104 registers, four waves per SIMD: held to
// 96 or 80 the compiler spills (70 and 109 us).
// `fill` writes 0 to the scales of rows (columns) past the end, which the last tiles hold anyway: a caller that wants
// them 0 had a fill launch before this one (11000 x 7168 with
// both outputs as a torch call: 57.3 us with the fill launch, 55.2 without; small matrices 33.0 -> 29.5).
// Scales are stored as [ceil(rows/128)][ceil(cols/128)][128] (row inside its block fastest), the
// transposed ones as [ceil(cols/128)][ceil(rows/128)][128].  scale_inv is the fp32 quotient 1.0f / scale:
// equal to the reference's float(1.0 / double(scale)), since a quotient rounded to 53 bits and then to 24
// (or fewer, for a denormal result) is the correctly rounded quotient.
template <int ROW>
__device__ __forceinline__ float row16_broadcast(float v) {
  return __uint_as_float(__builtin_amdgcn_update_dpp(0, static_cast<int>(__float_as_uint(v)), 0x150 + ROW, 0xf, 0xf, true));
}

template <bool VEC, bool TRANSPOSE, bool WHOLE_T>
__global__ __launch_bounds__(256) void quant_block128_tile_kernel(const uint16_t *__restrict__ x, int64_t rows,
                                                                  int64_t cols, int32_t nbx, int32_t nby,
                                                                  float eps, uint8_t *__restrict__ q,
                                                                  float *__restrict__ scale_inv,
                                                                  uint8_t *__restrict__ q_t,
                                                                  float *__restrict__ scale_inv_t, bool fill) {
  __shared__ __attribute__((aligned(16))) uint32_t s_col[TRANSPOSE ? 4 * 64 : 4];  // a pair of columns per word
  __shared__ __attribute__((aligned(16))) float s_scale[TRANSPOSE ? 128 : 4];
  __shared__ __attribute__((aligned(16))) uint8_t s_t[TRANSPOSE ? 128 * 128 : 16];
  const Tile tile = tile_of_block<TRANSPOSE, TRANSPOSE && !WHOLE_T>(nbx, nby);
  const int cg = threadIdx.x & 15, rg = threadIdx.x >> 4;
  const int64_t r0 = static_cast<int64_t>(tile.by) * 128 + rg * 8;
  const int64_t c0 = static_cast<int64_t>(tile.bx) * 128 + cg * 8;

  u32x4 v[8];
  load_patch<VEC>(x, rows, cols, r0, c0, v);

  uint32_t rmax[8];
  u32x4 cmax = u32x4{kZeroKeys, kZeroKeys, kZeroKeys, kZeroKeys};
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    rmax[i] = kZeroKeys;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const uint32_t k = abs_keys(v[i][d]);
      rmax[i] = max_keys(rmax[i], k);
      if constexpr (TRANSPOSE) cmax[d] = max_keys(cmax[d], k);
    }
  }
  if constexpr (TRANSPOSE) {
#pragma unroll
    for (int d = 0; d < 4; ++d) cmax[d] = across_rows_max(cmax[d]);
    if ((threadIdx.x & 48) == 0) *reinterpret_cast<u32x4 *>(s_col + (threadIdx.x >> 6) * 64 + cg * 4) = cmax;
  }

  // Rows 2i and 2i + 1 share a word from here on; lane cg picks out row cg & 7.
  uint32_t key = 0u;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t lo = __builtin_amdgcn_perm(rmax[2 * i + 1], rmax[2 * i], 0x05040100u);
    const uint32_t hi = __builtin_amdgcn_perm(rmax[2 * i + 1], rmax[2 * i], 0x07060302u);
    const uint32_t pair = row16_max(max_keys(lo, hi));
    if (((cg >> 1) & 3) == i) key = pair;
  }
  const float row_scale = compute_scale(key_to_float((cg & 1) ? key >> 16 : key & 0xffffu), eps);
  if (cg < 8 && (fill || r0 + cg < rows))
    scale_inv[static_cast<int64_t>(tile.by) * (static_cast<int64_t>(nbx) * 128) + static_cast<int64_t>(tile.bx) * 128 + rg * 8 + cg] =
        r0 + cg < rows ? 1.0f / row_scale : 0.0f;
  const float sc[8] = {row16_broadcast<0>(row_scale), row16_broadcast<1>(row_scale), row16_broadcast<2>(row_scale),
                       row16_broadcast<3>(row_scale), row16_broadcast<4>(row_scale), row16_broadcast<5>(row_scale),
                       row16_broadcast<6>(row_scale), row16_broadcast<7>(row_scale)};
  if constexpr (TRANSPOSE) {
    __syncthreads();
    if (threadIdx.x < 128) {
      const uint16_t *col = reinterpret_cast<const uint16_t *>(s_col) + threadIdx.x;
      const uint32_t m = max(max(col[0], col[128]), max(col[256], col[384]));  // non-negative keys: unsigned order
      const float scale = compute_scale(key_to_float(m), eps);
      s_scale[threadIdx.x] = scale;
      const bool inside = static_cast<int64_t>(tile.bx) * 128 + threadIdx.x < cols;
      if (fill || inside)
        scale_inv_t[static_cast<int64_t>(tile.bx) * (static_cast<int64_t>(nby) * 128) + static_cast<int64_t>(tile.by) * 128 +
                    threadIdx.x] = inside ? 1.0f / scale : 0.0f;
    }
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) store_codes<VEC>(q, rows, cols, r0 + i, c0, cast8(v[i], sc[i]));

  if constexpr (TRANSPOSE) {
    __syncthreads();
    float cs[8];
    *reinterpret_cast<float4 *>(cs) = *reinterpret_cast<const float4 *>(s_scale + cg * 8);
    *reinterpret_cast<float4 *>(cs + 4) = *reinterpret_cast<const float4 *>(s_scale + cg * 8 + 4);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      u32x2 t;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float f[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = ((j & 1) ? bf16_hi(v[4 * h + i][j >> 1]) : bf16_lo(v[4 * h + i][j >> 1])) * cs[j];
        t[h] = pack4_e4m3(f[0], f[1], f[2], f[3]);
      }
      put_column(s_t, rg, cg, j, t);
    }
    __syncthreads();
    store_transposed<WHOLE_T>(s_t, q_t, rows, cols, tile.bx, tile.by);
  }
}

template <int TPR>
void launch_block128(hipStream_t s, const uint16_t *x, int64_t rows, int32_t nvec, int32_t nblocks, float eps,
                     uint8_t *q, float *si, int32_t permute) {
  constexpr int kRowsPerBlock = 256 / TPR;
  const unsigned grid = static_cast<unsigned>((rows + kRowsPerBlock - 1) / kRowsPerBlock);
  hipLaunchKernelGGL((quant_block128_kernel<TPR>), dim3(grid), dim3(256), 0, s, x, rows, nvec, nblocks, eps, q, si,
                     permute);
}

template <int TPR, int VPT>
void launch_row(hipStream_t s, const uint16_t *x, int64_t rows, int32_t nvec, float eps, uint8_t *q,
                float *si) {
  constexpr int kRowsPerBlock = 256 / TPR;
  const unsigned grid = static_cast<unsigned>((rows + kRowsPerBlock - 1) / kRowsPerBlock);
  hipLaunchKernelGGL((quant_row_kernel<TPR, VPT>), dim3(grid), dim3(256), 0, s, x, rows, nvec, eps, q,
                     si);
}

}  // namespace
}  // namespace fluxmi

extern "C" int fluxmi_quant_e4m3_rowwise(const void *x_bf16, int64_t rows, int64_t cols,
                                         int32_t block_cols, float eps, void *q_out,
                                         float *scale_inv_out, int32_t permute_scale, void *stream) {
  using namespace fluxmi;
  FLUXMI_REQUIRE(x_bf16 != nullptr && q_out != nullptr && scale_inv_out != nullptr,
                 FLUXMI_ERR_INVALID_ARG, "quant_e4m3_rowwise: null pointer argument");
  FLUXMI_REQUIRE(rows >= 0 && cols >= 0, FLUXMI_ERR_INVALID_ARG,
                 "quant_e4m3_rowwise: negative size (rows=%lld, cols=%lld)",
                 static_cast<long long>(rows), static_cast<long long>(cols));
  FLUXMI_REQUIRE(block_cols == 0 || block_cols == 128, FLUXMI_ERR_UNSUPPORTED,
                 "quant_e4m3_rowwise: block_cols=%d (0 = whole row, or 128)", block_cols);
  FLUXMI_REQUIRE(cols % 8 == 0, FLUXMI_ERR_UNSUPPORTED,
                 "quant_e4m3_rowwise: cols=%lld is not a multiple of 8", static_cast<long long>(cols));
  FLUXMI_REQUIRE(cols / 8 <= INT32_MAX && rows <= (int64_t{1} << 40), FLUXMI_ERR_UNSUPPORTED,
                 "quant_e4m3_rowwise: matrix too large");
  FLUXMI_REQUIRE(aligned16(x_bf16) && (reinterpret_cast<uintptr_t>(q_out) & 7u) == 0,
                 FLUXMI_ERR_INVALID_ARG, "quant_e4m3_rowwise: x must be 16-byte and q 8-byte aligned");
  if (rows == 0 || cols == 0) return FLUXMI_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const uint16_t *x = static_cast<const uint16_t *>(x_bf16);
  uint8_t *q = static_cast<uint8_t *>(q_out);
  const int32_t nvec = static_cast<int32_t>(cols / 8);

  if (block_cols == 128 && permute_scale) {
    // The reference's layout: the tile kernel (faster than walking rows: eight loads in flight per lane).
    return fluxmi_quant_e4m3_block128(x_bf16, rows, cols, eps, q_out, scale_inv_out, nullptr, nullptr, stream);
  }
  if (block_cols == 128) {
    const int32_t nblocks = static_cast<int32_t>((cols + 127) / 128);
    FLUXMI_REQUIRE(rows <= INT32_MAX, FLUXMI_ERR_UNSUPPORTED, "quant_e4m3_rowwise: too many rows");
    const int32_t lanes = nblocks * 16;
    if (lanes <= 64) launch_block128<64>(s, x, rows, nvec, nblocks, eps, q, scale_inv_out, permute_scale);
    else if (lanes <= 128) launch_block128<128>(s, x, rows, nvec, nblocks, eps, q, scale_inv_out, permute_scale);
    else launch_block128<256>(s, x, rows, nvec, nblocks, eps, q, scale_inv_out, permute_scale);
  } else {
    FLUXMI_REQUIRE(rows <= INT32_MAX, FLUXMI_ERR_UNSUPPORTED, "quant_e4m3_rowwise: too many rows");
    if (nvec <= 64) launch_row<64, 1>(s, x, rows, nvec, eps, q, scale_inv_out);
    else if (nvec <= 128) launch_row<64, 2>(s, x, rows, nvec, eps, q, scale_inv_out);
    else if (nvec <= 256) launch_row<64, 4>(s, x, rows, nvec, eps, q, scale_inv_out);
    else if (nvec <= 512) launch_row<128, 4>(s, x, rows, nvec, eps, q, scale_inv_out);
    else if (nvec <= 1024) launch_row<256, 4>(s, x, rows, nvec, eps, q, scale_inv_out);
    else if (nvec <= 2048) launch_row<256, 8>(s, x, rows, nvec, eps, q, scale_inv_out);
    else
      hipLaunchKernelGGL(quant_row_long_kernel, dim3(static_cast<unsigned>(rows)), dim3(256), 0, s, x,
                         rows, nvec, eps, q, scale_inv_out);
  }
  FLUXMI_HIP_CHECK(hipGetLastError());
  return FLUXMI_OK;
}

extern "C" int fluxmi_quant_e4m3_square(const void *x_bf16, int64_t batch, int64_t rows, int64_t cols,
                                        float eps, void *q_out, float *scale_inv_out, void *q_t_out,
                                        float *scale_inv_t_out, void *stream) {
  using namespace fluxmi;
  FLUXMI_REQUIRE(x_bf16 != nullptr && q_out != nullptr && scale_inv_out != nullptr,
                 FLUXMI_ERR_INVALID_ARG, "quant_e4m3_square: null pointer argument");
  FLUXMI_REQUIRE((q_t_out == nullptr) == (scale_inv_t_out == nullptr), FLUXMI_ERR_INVALID_ARG,
                 "quant_e4m3_square: q_t_out and scale_inv_t_out go together");
  FLUXMI_REQUIRE(batch >= 0 && rows >= 0 && cols >= 0, FLUXMI_ERR_INVALID_ARG,
                 "quant_e4m3_square: negative size (batch=%lld, rows=%lld, cols=%lld)",
                 static_cast<long long>(batch), static_cast<long long>(rows), static_cast<long long>(cols));
  FLUXMI_REQUIRE((reinterpret_cast<uintptr_t>(x_bf16) & 1u) == 0, FLUXMI_ERR_INVALID_ARG,
                 "quant_e4m3_square: x must be 2-byte aligned");
  if (batch == 0 || rows == 0 || cols == 0) return FLUXMI_OK;
  const int64_t nbx = (cols + 127) / 128, nby = (rows + 127) / 128;
  FLUXMI_REQUIRE(nbx <= INT32_MAX && nby <= INT32_MAX && batch <= INT32_MAX &&
                     nbx * nby <= INT32_MAX / batch,
                 FLUXMI_ERR_UNSUPPORTED, "quant_e4m3_square: more than 2^31 blocks");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const uint16_t *x = static_cast<const uint16_t *>(x_bf16);
  uint8_t *q = static_cast<uint8_t *>(q_out);
  uint8_t *qt = static_cast<uint8_t *>(q_t_out);
  const dim3 grid(static_cast<unsigned>(batch * nbx * nby)), block(256);
  const bool vec = cols % 8 == 0 && aligned16(x_bf16) && (reinterpret_cast<uintptr_t>(q_out) & 7u) == 0;
  const bool whole_t = rows % 128 == 0 && aligned16(q_t_out);
#define FLUXMI_SQ(V, T, VT)                                                                            \
  hipLaunchKernelGGL((quant_square_kernel<V, T, VT>), grid, block, 0, s, x, rows, cols,                \
                     static_cast<int32_t>(nbx), static_cast<int32_t>(nby), eps, q, scale_inv_out, qt,  \
                     scale_inv_t_out)
  if (qt == nullptr) {
    if (vec) FLUXMI_SQ(true, false, false);
    else FLUXMI_SQ(false, false, false);
  } else if (vec) {
    if (whole_t) FLUXMI_SQ(true, true, true);
    else FLUXMI_SQ(true, true, false);
  } else {
    if (whole_t) FLUXMI_SQ(false, true, true);
    else FLUXMI_SQ(false, true, false);
  }
#undef FLUXMI_SQ
  FLUXMI_HIP_CHECK(hipGetLastError());
  return FLUXMI_OK;
}

namespace fluxmi {
namespace {
int quant_block128(const void *x_bf16, int64_t rows, int64_t cols, float eps, void *q_out, float *scale_inv_out,
                   void *q_t_out, float *scale_inv_t_out, bool fill, void *stream) {
  FLUXMI_REQUIRE(x_bf16 != nullptr && q_out != nullptr && scale_inv_out != nullptr,
                 FLUXMI_ERR_INVALID_ARG, "quant_e4m3_block128: null pointer argument");
  FLUXMI_REQUIRE((q_t_out == nullptr) == (scale_inv_t_out == nullptr), FLUXMI_ERR_INVALID_ARG,
                 "quant_e4m3_block128: q_t_out and scale_inv_t_out go together");
  FLUXMI_REQUIRE(rows >= 0 && cols >= 0, FLUXMI_ERR_INVALID_ARG,
                 "quant_e4m3_block128: negative size (rows=%lld, cols=%lld)", static_cast<long long>(rows),
                 static_cast<long long>(cols));
  FLUXMI_REQUIRE((reinterpret_cast<uintptr_t>(x_bf16) & 1u) == 0, FLUXMI_ERR_INVALID_ARG,
                 "quant_e4m3_block128: x must be 2-byte aligned");
  if (rows == 0 || cols == 0) return FLUXMI_OK;
  const int64_t nbx = (cols + 127) / 128, nby = (rows + 127) / 128;
  FLUXMI_REQUIRE(nbx <= INT32_MAX && nby <= INT32_MAX && nbx * nby <= INT32_MAX, FLUXMI_ERR_UNSUPPORTED,
                 "quant_e4m3_block128: more than 2^31 blocks");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const uint16_t *x = static_cast<const uint16_t *>(x_bf16);
  uint8_t *q = static_cast<uint8_t *>(q_out);
  uint8_t *qt = static_cast<uint8_t *>(q_t_out);
  const dim3 grid(static_cast<unsigned>(nbx * nby)), block(256);
  const bool vec = cols % 8 == 0 && aligned16(x_bf16) && (reinterpret_cast<uintptr_t>(q_out) & 7u) == 0;
  const bool whole_t = rows % 128 == 0 && aligned16(q_t_out);
#define FLUXMI_B128(V, T, VT)                                                                          \
  hipLaunchKernelGGL((quant_block128_tile_kernel<V, T, VT>), grid, block, 0, s, x, rows, cols,         \
                     static_cast<int32_t>(nbx), static_cast<int32_t>(nby), eps, q, scale_inv_out, qt,  \
                     scale_inv_t_out, fill)
  if (qt == nullptr) {
    if (vec) FLUXMI_B128(true, false, false);
    else FLUXMI_B128(false, false, false);
  } else if (vec) {
    if (whole_t) FLUXMI_B128(true, true, true);
    else FLUXMI_B128(true, true, false);
  } else {
    if (whole_t) FLUXMI_B128(false, true, true);
    else FLUXMI_B128(false, true, false);
  }
#undef FLUXMI_B128
  FLUXMI_HIP_CHECK(hipGetLastError());
  return FLUXMI_OK;
}
}  // namespace
}  // namespace fluxmi

extern "C" int fluxmi_quant_e4m3_block128(const void *x_bf16, int64_t rows, int64_t cols, float eps,
                                          void *q_out, float *scale_inv_out, void *q_t_out,
                                          float *scale_inv_t_out, void *stream) {
  return fluxmi::quant_block128(x_bf16, rows, cols, eps, q_out, scale_inv_out, q_t_out, scale_inv_t_out, false, stream);
}

extern "C" int fluxmi_quant_e4m3_block128_filled(const void *x_bf16, int64_t rows, int64_t cols, float eps,
                                                 void *q_out, float *scale_inv_out, void *q_t_out,
                                                 float *scale_inv_t_out, void *stream) {
  return fluxmi::quant_block128(x_bf16, rows, cols, eps, q_out, scale_inv_out, q_t_out, scale_inv_t_out, true, stream);
}
