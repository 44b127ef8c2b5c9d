// Many tokens through one compressed matrix on the matrix cores.
//
// Sub1Linear.forward on a sequence (reference sub1.py:132-143 launches one
// product per token and calls that "naive") is a skinny GEMM Y += X W^T, and
// the matrix cores do it (v_mfma_f32_32x32x16_bf16) once the ternary weights
// are bf16 values again.  Nothing is walked per token and nothing is scattered:
// the work no longer grows with tokens x non-zeros.
//
// The tile form of a matrix (sub1_tiles_*) is made for that, once, from the
// packed codes: 2 bits per weight, whatever the density, cut into units of
// 32 rows x 128 columns of 64 x 16 bytes.  In unit (u, w) lane l = 32 h + r
// holds the weights of row 32 u + r that it feeds the matrix core as its share
// of the B operand: in step s (0..7) of the window the eight columns
// 128 w + 16 s + 8 h + q.  Word s / 2 of its 16 bytes holds steps s and s + 1;
// the weight of step s = 2 m + e and q = 4 f + b sits in bits
// 8 b + 4 e + 2 f (+1) of word m, as 0 (the row's min), 1 (its max) or 2
// (zero).  A wavefront fetches a unit with one coalesced 16-byte load per
// lane.  Rows are padded to a multiple of 64 and columns to a multiple of 128
// with zeros; (min, max) per row are copied.
//
// From the codes to bf16 pairs without a table in memory: (word >> (4 e + 2 f))
// & 0x03030303 is the codes of four weights a byte each, which is a byte
// selector (v_perm_b32) into (min, max, 0, 0) of the row's upper and of its
// lower bytes; two more permutes put the four upper and lower bytes together as
// two pairs.  Twelve plain instructions for the eight weights of an operand.
// (With a pair's codes 16 bits apart, widened to a selector into the row's
// (min, max) word by a multiply-add, it is sixteen: behind an operand that
// serves 64 tokens that is eight instructions per MFMA instead of six, and six
// are what an MFMA hides.)
//
// Kernels: a workgroup owns 64 rows x 64 tokens, or up to 128 of either.  It
// walks windows of 128 columns; the tokens' activations of a window lie in LDS
// as tiles of 64 x 128 (16 KB; 16-byte pieces, four tokens an instruction; the
// pieces of a token are XOR-swizzled with the token's number so that neither
// the arrivals nor the operand reads meet in a bank), and per step of 16
// columns a wavefront reads its A operands from there, builds its B operands
// from the codes and adds into 64 x 64 fp32 accumulators (2 x 2 MFMA blocks).
// Short launches give each wavefront windows and tiles of its own
// (matvec_tiles_kernel: wavefront v takes windows v, v + n, ...); elsewhere the
// wavefronts share the tiles (matvec_tiles_shared_kernel).  Where x rows are
// 16-byte aligned the loads go straight into LDS, into a second buffer, a whole
// window ahead of the arithmetic; otherwise the shared kernel takes them
// through registers, in the widest loads that every row's address allows.
// Either way what lies past the last token, past the width or past the last
// window is given an offset outside the buffer (or an empty buffer) and reads
// nothing, without a branch or a mask.  The columns are cut into parts, each
// summed in order, and the parts are added in order, rounded to bf16 and added
// onto y in bf16 (reference sub1_cuda_kernel.cu:199-200).  The number of parts
// depends on the matrix alone, so a token's result does not depend on the
// launch it is part of.
//
// Bound: a wavefront alone on its SIMD issues an MFMA of this shape every
// 18 ns (the matrix core needs 13.4); with the four plain instructions per
// pair of weights that build the B operands behind it, and the LDS reads of
// the A operands, 22 to 24 ns where an operand serves 128 tokens (four
// instructions per MFMA) and 27 to 30 ns where it serves 64 (eight), measured
// on loops of just these instructions; the kernels here take 28 and 35 ns.
// A second wavefront on the SIMD fills part of the gap, and then the issue of
// the decoding instructions is what the SIMD runs out of.
//
// Results: each product x * w is exact in fp32 and the sums are fp32, but in
// the matrix cores' own order; they agree with the row-walking kernels and the
// oracle to rounding (the tests hold them to 1e-2 and to the fp32 error bound),
// not to the bit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <type_traits>

#include "sub1_common.h"

namespace {

using sub1::bf16_to_f32;
using sub1::f32_to_bf16;
using sub1::fail;
using sub1::misaligned;

constexpr int kUnitRows = 32;             // rows per unit
constexpr int kRows = 64;                 // rows per workgroup: two units
constexpr int kCols = 128;                // columns per window
constexpr int kTokens = 64;               // tokens per workgroup
constexpr int kSteps = kCols / 16;        // MFMA steps per window
constexpr int kMaxWaves = 4;              // wavefronts per workgroup, at most
constexpr uint32_t kAllZero = 0xaaaaaaaau; // a word of codes of zero weights

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

int64_t align256(int64_t v) { return (v + 255) / 256 * 256; }

// The meta block: arrays back to back, each 256-byte aligned.
struct TileLayout {
  int units_down;     // units of 32 rows per matrix, even
  int windows;
  int64_t units;      // of all matrices
  int64_t minmax;     // u32 [count * height]
  int64_t status;     // i32 [4]: [0] rows whose codes do not cover the width
  int64_t bytes;
};

TileLayout tile_layout(int count, int height, int width) {
  TileLayout t;
  t.units_down = (height + kRows - 1) / kRows * (kRows / kUnitRows);
  t.windows = (width + kCols - 1) / kCols;
  t.units = static_cast<int64_t>(count) * t.units_down * t.windows;
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    int64_t o = off;
    off += align256(bytes);
    return o;
  };
  t.minmax = take(static_cast<int64_t>(count) * height * 4);
  t.status = take(16);
  t.bytes = off;
  return t;
}

// Calls nz(column, symbol) for every non-zero weight of a row, in column order,
// and returns the columns the row's codes cover (dictionary layout: reference
// sub1.py:60-72, sub1_cuda_kernel.cu:186-192).
template <class F>
__device__ __forceinline__ int each_nonzero(const uint16_t *codes, int n,
                                            const int32_t *__restrict__ dec, int width, F &&nz) {
  int col = 0;
  for (int i = 0; i < n; i++) {
    const int e = codes[i];
    const uint32_t w0 = static_cast<uint32_t>(dec[2 * e]);
    const uint32_t w1 = static_cast<uint32_t>(dec[2 * e + 1]);
    unsigned long long digits = static_cast<unsigned long long>(w0 >> 4) |
                                (static_cast<unsigned long long>(w1 >> 4) << 28);
    while (digits) {
      const int d = (__ffsll(digits) - 1) >> 1;
      const int sym = static_cast<int>(digits >> (2 * d)) & 3;
      digits &= ~(3ull << (2 * d));
      if (col + d < width && sym != 3) nz(col + d, sym);   // digits past the width are dropped
    }
    col += 2 * static_cast<int>(w0 & 15u);
  }
  return col;
}

struct RowSource {
  const int32_t *dec;
  const uint16_t *w_comp;
  const int64_t *code_base;   // NULL: one matrix, base 0
  const int32_t *row_off;     // [count, height + 1]
  int count, height, width;
};

__device__ __forceinline__ const uint16_t *codes_of(const RowSource &s, int m, int r, int &n) {
  const int32_t *ro = s.row_off + static_cast<int64_t>(m) * (s.height + 1);
  n = ro[r + 1] - ro[r];
  if (n < 1 || n > (s.width + 1) / 2) n = 0;   // counted as a bad row
  return s.w_comp + (s.code_base ? s.code_base[m] : 0) + ro[r];
}

// Where the weight of column c of a window sits in its lane's 16 bytes.
__device__ __forceinline__ void code_place(int c, int &half, int &word, int &shift) {
  const int step = c >> 4, q = c & 7;
  half = (c >> 3) & 1;
  word = step >> 1;
  shift = 8 * (q & 3) + 4 * (step & 1) + 2 * (q >> 2);
}

// One thread per row of every matrix: its codes into the units (all zero
// weights before).
__global__ __launch_bounds__(256) void code_emit_kernel(RowSource s, int units_down, int windows,
                                                        u32x4 *__restrict__ units,
                                                        int32_t *__restrict__ status,
                                                        int64_t rows_total) {
  const int64_t gl = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (gl >= rows_total) return;
  const int m = static_cast<int>(gl / s.height);
  const int r = static_cast<int>(gl % s.height);
  u32x4 *mine = units + (static_cast<int64_t>(m) * units_down + r / kUnitRows) * windows * 64 +
                r % kUnitRows;
  uint32_t held[2][4];   // [half][word] of the window at hand
  int w_cur = 0;
  bool dirty = false;
  auto clear = [&]() {
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int d = 0; d < 4; d++) held[h][d] = kAllZero;
    dirty = false;
  };
  auto flush = [&]() {
    if (dirty) {
#pragma unroll
      for (int h = 0; h < 2; h++) {
        u32x4 v = {held[h][0], held[h][1], held[h][2], held[h][3]};
        mine[static_cast<int64_t>(w_cur) * 64 + h * kUnitRows] = v;
      }
    }
    clear();
  };
  clear();
  int n;
  const uint16_t *codes = codes_of(s, m, r, n);
  const int covered = each_nonzero(codes, n, s.dec, s.width, [&](int col, int sym) {
    const int w = col / kCols;
    if (w != w_cur) {
      flush();
      w_cur = w;
    }
    int half, word, shift;
    code_place(col % kCols, half, word, shift);
    // symbol 1 (min) is code 0, symbol 2 (max) code 1; the place holds 2 (zero)
    const uint32_t flip = (sym == 2 ? 3u : 2u) << shift;
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int d = 0; d < 4; d++)
        if (h == half && d == word) held[h][d] ^= flip;
    dirty = true;
  });
  flush();
  if (covered != ((s.width + 1) & ~1)) atomicAdd(&status[0], 1);
}

// The symbols of one matrix back out of its units, a thread per weight.
__global__ __launch_bounds__(256) void code_decode_kernel(const u32x4 *__restrict__ units,
                                                          uint8_t *__restrict__ out, int matrix,
                                                          int units_down, int windows, int height,
                                                          int width) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= static_cast<int64_t>(height) * width) return;
  const int r = static_cast<int>(i / width), col = static_cast<int>(i % width);
  int half, word, shift;
  code_place(col % kCols, half, word, shift);
  const u32x4 v = units[((static_cast<int64_t>(matrix) * units_down + r / kUnitRows) * windows +
                         col / kCols) * 64 + half * kUnitRows + r % kUnitRows];
  const uint32_t code = (v[word] >> shift) & 3u;
  out[i] = static_cast<uint8_t>(code == 2 ? 0 : code + 1);
}

__global__ void tile_fill_kernel(uint32_t *p, int64_t n, uint32_t v) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void tile_copy_words_kernel(const uint32_t *src, uint32_t *dst, int64_t n) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

// --------------------------------------------------------------- product ---

struct TileArgs {
  const u32x4 *units;
  const uint32_t *minmax;
  const uint16_t *x;
  uint16_t *y;
  int64_t ldx, ldy;
  int height, width, tokens;
  int units_down, windows, matrix;
  int fresh;   // y holds nothing yet: it counts as zeros and is not read
  int column_blocks, larger_columns;   // shared kernel: blocks of 32 tokens a column; one more in the first ones
};

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// A buffer over `bytes` bytes from base on: loads at offsets from `bytes` on
// return zeros and touch no memory.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_over(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, static_cast<int>(bytes),
                                           0x00020000);
}
constexpr uint32_t kOutside = 0x80000000u;   // an offset past every buffer here

// (min, max, 0, 0) of a row's lower bytes and of its upper ones, from its
// (min, max) word: what the codes select from.
struct RowTables {
  uint32_t lo[2], hi[2];   // of a lane's two rows
};
__device__ __forceinline__ void set_tables(RowTables &t, int j, uint32_t min_max) {
  t.lo[j] = __builtin_amdgcn_perm(0u, min_max, 0x0c0c0200u);
  t.hi[j] = __builtin_amdgcn_perm(0u, min_max, 0x0c0c0301u);
}

// The B operands of a step in the making: the weights of a lane's two rows from
// half kE of a word of codes each, as 24 instructions of which none needs the
// one just before it.  They are issued in equal shares behind the MFMAs of the
// step before.
struct WeightsInTheMaking {
  uint32_t at[4], lo[4], hi[4];   // [2 row + f]: codes, lower and upper bytes of four weights
};
constexpr int kDecodeOps = 24;
template <int kOp, int kE>
__device__ __forceinline__ void decode_op(WeightsInTheMaking &m, uint32_t word0, uint32_t word1,
                                          const RowTables &rows, u32x4 (&wv)[2]) {
  // (each is pinned to its place: the scheduler would gather them elsewhere)
  if constexpr (kOp < 4) {
    constexpr int shift = 4 * kE + 2 * (kOp & 1);
    m.at[kOp] = (kOp >> 1 ? word1 : word0) >> shift;
    if (shift) asm volatile("" : "+v"(m.at[kOp]));
  } else if constexpr (kOp < 8) {
    m.at[kOp - 4] &= 0x03030303u;
    asm volatile("" : "+v"(m.at[kOp - 4]));
  } else if constexpr (kOp < 16) {
    constexpr int i = (kOp - 8) >> 1;
    uint32_t &out = kOp & 1 ? m.hi[i] : m.lo[i];
    out = __builtin_amdgcn_perm(0u, kOp & 1 ? rows.hi[i >> 1] : rows.lo[i >> 1], m.at[i]);
    asm volatile("" : "+v"(out));
  } else {
    constexpr int i = (kOp - 16) >> 1;
    uint32_t pair = __builtin_amdgcn_perm(m.hi[i], m.lo[i], kOp & 1 ? 0x07030602u : 0x05010400u);
    asm volatile("" : "+v"(pair));
    wv[i >> 1][2 * (i & 1) + (kOp & 1)] = pair;
  }
}
// Share kSlot of kSlots of them.
template <int kSlot, int kSlots, int kE, int kAt = kSlot * kDecodeOps / kSlots>
__device__ __forceinline__ void decode_share(WeightsInTheMaking &m, uint32_t word0, uint32_t word1,
                                             const RowTables &rows, u32x4 (&wv)[2]) {
  if constexpr (kAt < (kSlot + 1) * kDecodeOps / kSlots) {
    decode_op<kAt, kE>(m, word0, word1, rows, wv);
    decode_share<kSlot, kSlots, kE, kAt + 1>(m, word0, word1, rows, wv);
  }
}

// What the kernels share.  A workgroup owns rows 64 block .. +64 and tokens
// t0 .. +64; as the B operand (and as an output column) a lane has the rows
// 32 j + lane % 32, as the A operand the tokens 32 i + lane % 32 and in step s
// their piece 2 s + half.  In LDS piece p of token t of a window sits at
// 256 t + 16 (p ^ (t % 16)) of the wavefront's 16 KB.
struct TileLane {
  int lane, half, block, t0, rows_here;
  RowTables rows;
  uint32_t unit_at[2];   // byte offset of the lane's codes in window 0, per unit
  uint32_t get_at;       // of its A operand of step 0 in the wavefront's tile
};

__device__ __forceinline__ TileLane tile_lane(const TileArgs &a) {
  TileLane l;
  l.lane = threadIdx.x & 63;
  l.half = l.lane >> 5;
  l.block = blockIdx.x;
  l.t0 = blockIdx.y * kTokens;
  l.rows_here = min(kTokens, a.tokens - l.t0);
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int row = l.block * kRows + j * kUnitRows + (l.lane & 31);
    set_tables(l.rows, j,
               row < a.height ? a.minmax[static_cast<int64_t>(a.matrix) * a.height + row] : 0u);
    l.unit_at[j] = static_cast<uint32_t>(j * a.windows * 1024 + l.lane * 16);
  }
  l.get_at = static_cast<uint32_t>((l.lane & 31) * 256 + ((l.half ^ (l.lane & 15)) << 4));
  return l;
}

// The codes of this workgroup's two units, window after window.
// (`any` false: an empty buffer, every load from it returns zeros.)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t units_of(const TileArgs &a, int block,
                                                           bool any = true) {
  return buffer_over(
      a.units + (static_cast<int64_t>(a.matrix) * a.units_down + block * 2) * a.windows * 64,
      any ? static_cast<uint32_t>(2 * a.windows * 1024) : 0u);
}

// The activations of this workgroup's tokens.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tokens_of(const TileArgs &a, const TileLane &l,
                                                            bool any = true) {
  return buffer_over(
      a.x + static_cast<int64_t>(l.t0) * a.ldx,
      any ? static_cast<uint32_t>((static_cast<int64_t>(l.rows_here - 1) * a.ldx + a.width) * 2)
          : 0u);
}

// What the neighbour (lane ^ 1) has.
__device__ __forceinline__ float neighbour(float v) {
  constexpr int kDppQuadXor1 = 0xb1;   // quad_perm [1, 0, 3, 2]
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kDppQuadXor1, 0xf, 0xf, true));
}

// The end of a workgroup of kKP parts times kRG groups of rows.  The parts of a group each
// finish a share of its tiles of 32 tokens x 32 rows: what the others have of them goes through
// `lds`, which no wavefront reads any more, whole registers at a time, and is added in the parts' order;
// the sum is rounded to bf16 and added onto y in bf16 (reference sub1_cuda_kernel.cu:199-200), tokens
// past the last and rows past the height dropped.  kPairs: y takes two rows in a 4-byte store.
// (Through LDS a token's rows at a time, with y read back where it counts as zeros, as it was done
// first, the end took 10 of 40 us of c-2048 wi on 1136 tokens, against 2 to 3 now.)
template <bool kPairs, int kRG, int kKP, int kNB>
__device__ __forceinline__ void finish_tiles(const TileArgs &a, const TileLane &l, int g, int k, bool rows, int live,
                                             unsigned char *lds, const f32x16 (&acc)[kNB][2]) {
  constexpr int kTiles = 2 * kNB, kFinish = (kTiles + kKP - 1) / kKP;
  static_assert(kTiles % kFinish == 0, "equal shares (where there are fewer tiles than parts the last ones have none)");
  float4 *sums = reinterpret_cast<float4 *>(lds);
  // of tile `n` of what part `of` finishes, from part `from`
  auto place = [&](int of, int from, int n) {
    return sums + ((((g * kKP + of) * (kKP - 1) + (from < of ? from : from - 1)) * kFinish + n) * 4) * 64 + l.lane;
  };
  if constexpr (kKP > 1) {
    __syncthreads();
#pragma unroll
    for (int n = 0; n < kTiles; n++)
      if (n / kFinish != k && n / 2 < live)
#pragma unroll
        for (int v = 0; v < 4; v++)
          place(n / kFinish, k, n % kFinish)[v * 64] =
              make_float4(acc[n >> 1][n & 1][4 * v], acc[n >> 1][n & 1][4 * v + 1], acc[n >> 1][n & 1][4 * v + 2],
                          acc[n >> 1][n & 1][4 * v + 3]);
    __syncthreads();
  }
  const uint32_t y_bytes =
      static_cast<uint32_t>((static_cast<int64_t>(l.rows_here - 1) * a.ldy + a.height) * 2);
  const __amdgpu_buffer_rsrc_t yb = buffer_over(a.y + static_cast<int64_t>(l.t0) * a.ldy, y_bytes);
  const uint32_t y_step = static_cast<uint32_t>(a.ldy * 2);
  const bool odd = l.lane & 1;
#pragma unroll
  for (int n = 0; n < kTiles; n++) {
    if (n / kFinish != k || n / 2 >= live || !rows) continue;
    // Value v of a lane is row lane % 32 and token 8 (v / 4) + 4 half + v % 4: added in the parts'
    // order, then exchanged with the neighbour, so that a lane has two rows of a token
    float t[16];
#pragma unroll
    for (int v = 0; v < 16; v++) t[v] = acc[n >> 1][n & 1][v];
    if constexpr (kKP > 1) {
#pragma unroll
      for (int v = 0; v < 4; v++) {
        float s[4] = {t[4 * v], t[4 * v + 1], t[4 * v + 2], t[4 * v + 3]};
#pragma unroll
        for (int part = 0; part < kKP; part++) {
          if (part == k) {
#pragma unroll
            for (int m = 0; m < 4; m++) s[m] = part ? s[m] + t[4 * v + m] : t[4 * v + m];
          } else {
            const float4 q = place(k, part, n % kFinish)[v * 64];
            s[0] = part ? s[0] + q.x : q.x;
            s[1] = part ? s[1] + q.y : q.y;
            s[2] = part ? s[2] + q.z : q.z;
            s[3] = part ? s[3] + q.w : q.w;
          }
        }
#pragma unroll
        for (int m = 0; m < 4; m++) t[4 * v + m] = s[m];
      }
    }
    const int row = l.block * kRows + 32 * (n & 1) + (l.lane & 30);
    const int token = 32 * (n >> 1) + 4 * l.half + (l.lane & 1);
    const uint32_t y_at = row < a.height ? static_cast<uint32_t>(row * 2) + token * y_step : kOutside;
    const uint32_t y_at1 = row + 1 < a.height ? y_at + 2 : kOutside;   // !kPairs
    uint32_t before[8];
#pragma unroll
    for (int m = 0; m < 8; m++) before[m] = 0u;   // a y that holds nothing yet
    if (!a.fresh)
#pragma unroll
      for (int m = 0; m < 8; m++) {
        const uint32_t at = (8 * (m >> 1) + 2 * (m & 1)) * y_step;
        before[m] = kPairs ? __builtin_amdgcn_raw_buffer_load_b32(yb, y_at + at, 0, 0)
                            : static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b16(yb, y_at + at, 0, 0)) |
                                  static_cast<uint32_t>(__builtin_amdgcn_raw_buffer_load_b16(yb, y_at1 + at, 0, 0)) << 16;
      }
#pragma unroll
    for (int m = 0; m < 8; m++) {
      const float mine = odd ? t[2 * m + 1] : t[2 * m], other = odd ? t[2 * m] : t[2 * m + 1];
      const float theirs = neighbour(other);
      const bf16x2 sum = {static_cast<__bf16>(odd ? theirs : mine), static_cast<__bf16>(odd ? mine : theirs)};
      const uint32_t bits = __builtin_bit_cast(uint32_t, sum);
      // y += bf16(sum) in bf16
      const bf16x2 out = {static_cast<__bf16>(__uint_as_float(before[m] << 16) + __uint_as_float(bits << 16)),
                          static_cast<__bf16>(__uint_as_float(before[m] & 0xffff0000u) + __uint_as_float(bits & 0xffff0000u))};
      const uint32_t now = __builtin_bit_cast(uint32_t, out);
      const uint32_t at = (8 * (m >> 1) + 2 * (m & 1)) * y_step;
      if (kPairs) {
        __builtin_amdgcn_raw_buffer_store_b32(now, yb, y_at + at, 0, 0);
      } else {
        __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(now), yb, y_at + at, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b16(static_cast<uint16_t>(now >> 16), yb, y_at1 + at, 0, 0);
      }
    }
  }
}

// ---- x rows 16-byte aligned, the width a multiple of 8 ----------------------
//
// Activations and codes go from global memory straight into LDS (buffer loads
// with the lds bit, 16 bytes a lane: four tokens of activations, or one unit
// of codes, an instruction).  A wavefront has two buffers (a tile of
// activations of 16 KB and a block of codes of 2 KB each) and asks for the next
// window before it starts on the current one.
//
// Waiting is done by hand.  Left to the compiler, an LDS read behind such
// loads waits for all of them (it cannot tell the two buffers apart), which
// puts the memory latency of every window back in front of its arithmetic.  So
// the loop reads LDS through ds_read_b128 written as inline assembly, which
// the compiler does not see as LDS reads, and counts the loads itself: every
// turn issues exactly kLoadsPerWindow of them (after a wavefront's last window
// from empty buffers: nothing is read, nothing lands), loads complete in the
// order issued, and "all but the newest kLoadsPerWindow have landed" is the
// wait before a window is read.  The LDS reads are waited for with lgkmcnt(0)
// in statements that take the read registers as operands, so nothing uses them
// earlier.

constexpr int kActivationLoads = 16;   // of a window: four tokens each
constexpr int kCodeLoads = 2;          // one per unit of 32 rows
constexpr int kLoadsPerWindow = kActivationLoads + kCodeLoads;   // what fetch_window issues, every time
constexpr int kTileBytes = 16384;     // a tile of activations
constexpr int kBlockBytes = 2048;     // a window's codes (two units)

// Load u (0..15) of a window brings tokens 4 u + lane / 16, the lane its piece
// (lane % 16) ^ (token % 16): the one that belongs at its place in LDS.  `at`
// holds the lane's byte offsets for u = 0..3 (token % 16 takes four values per
// lane), `col` the first column of each.
struct Fetch {
  uint32_t at[4];
  int col[4];
  uint32_t step;   // sixteen tokens on
};

__device__ __forceinline__ Fetch fetch_of(const TileArgs &a, int lane) {
  Fetch f;
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int token = 4 * u + (lane >> 4);
    f.col[u] = 8 * ((lane & 15) ^ token);
    f.at[u] = static_cast<uint32_t>((token * a.ldx + f.col[u]) * 2);
  }
  f.step = static_cast<uint32_t>(16 * a.ldx * 2);
  return f;
}

typedef __attribute__((address_space(3))) unsigned char *lds_bytes;

// 16 bytes a lane straight into LDS.  (No template: on the host's side the size would not pass in one.)
__device__ __forceinline__ void load_to_lds(__amdgpu_buffer_rsrc_t from, lds_bytes to, uint32_t at, uint32_t more) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(from, to, 16, at, more, 0, 0);
}

// Window w on its way: the activations into the tile at `tile`, the codes into
// the block at `block`.  Pieces from the width on are not fetched (`edge`: this
// window reaches past the width; their places hold zeros or older activations,
// and the weights there are zeros).
__device__ __forceinline__ void fetch_window(__amdgpu_buffer_rsrc_t xb, __amdgpu_buffer_rsrc_t ub,
                                             const Fetch &f, const TileArgs &a, const TileLane &l,
                                             int w, bool edge, lds_bytes tile, lds_bytes block) {
  if (edge) {
    const int inside = a.width - w * kCols;
#pragma unroll
    for (int u = 0; u < kActivationLoads; u++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          xb, tile + u * 1024, 16,
          f.col[u & 3] < inside ? f.at[u & 3] + (u >> 2) * f.step : kOutside, w * (kCols * 2), 0, 0);
  } else {
#pragma unroll
    for (int u = 0; u < kActivationLoads; u++)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xb, tile + u * 1024, 16,
                                               f.at[u & 3] + (u >> 2) * f.step, w * (kCols * 2), 0, 0);
  }
#pragma unroll
  for (int j = 0; j < kCodeLoads; j++)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(ub, block + j * 1024, 16, l.unit_at[j], w * 1024, 0, 0);
}

// 16 bytes from LDS address `at` and from `at` + kFar, requested only.
template <int kFar>
__device__ __forceinline__ void lds_request(uint32_t at, u32x4 &near, u32x4 &far) {
  asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %2 offset:%3"
               : "=&v"(near), "=&v"(far)
               : "v"(at), "n"(kFar)
               : "memory");
}
// What was requested has arrived.
__device__ __forceinline__ void lds_arrived(u32x4 &p, u32x4 &q) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(p), "+v"(q)::"memory");
}

// window_steps with the operands read by hand: the tile at LDS address `tile`,
// the codes at `block`.
__device__ __forceinline__ void window_steps_counted(uint32_t tile, uint32_t block,
                                                     const TileLane &l, f32x16 (&acc)[2][2]) {
  const uint32_t get = tile + l.get_at;
  u32x4 xa[2], codes[2], wv[2];
  lds_request<1024>(block + l.lane * 16, codes[0], codes[1]);
  lds_request<32 * 256>(get, xa[0], xa[1]);
  lds_arrived(codes[0], codes[1]);
  lds_arrived(xa[0], xa[1]);
  WeightsInTheMaking m;
  decode_share<0, 1, 0>(m, codes[0][0], codes[1][0], l.rows, wv);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = 0; s < kSteps; s++) {
    u32x4 xa_next[2], wv_next[2];
    const int sn = s + 1 < kSteps ? s + 1 : s;   // after the last step nothing new
    const uint32_t word0 = codes[0][sn >> 1], word1 = codes[1][sn >> 1];
    if (s + 1 < kSteps) lds_request<32 * 256>(get ^ static_cast<uint32_t>(32 * sn), xa_next[0], xa_next[1]);
    const bf16x8 wb0 = __builtin_bit_cast(bf16x8, wv[0]), wb1 = __builtin_bit_cast(bf16x8, wv[1]);
    const bf16x8 xa0 = __builtin_bit_cast(bf16x8, xa[0]), xa1 = __builtin_bit_cast(bf16x8, xa[1]);
    auto next_weights = [&](auto slot) {
      constexpr int kSlot = decltype(slot)::value;
      if (s + 1 < kSteps) {
        if (sn & 1) decode_share<kSlot, 4, 1>(m, word0, word1, l.rows, wv_next);
        else decode_share<kSlot, 4, 0>(m, word0, word1, l.rows, wv_next);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa0, wb0, acc[0][0], 0, 0, 0);
    next_weights(std::integral_constant<int, 0>{});
    acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa0, wb1, acc[0][1], 0, 0, 0);
    next_weights(std::integral_constant<int, 1>{});
    acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa1, wb0, acc[1][0], 0, 0, 0);
    next_weights(std::integral_constant<int, 2>{});
    acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xa1, wb1, acc[1][1], 0, 0, 0);
    next_weights(std::integral_constant<int, 3>{});
    if (s + 1 < kSteps) {
      lds_arrived(xa_next[0], xa_next[1]);
      xa[0] = xa_next[0];
      xa[1] = xa_next[1];
      wv[0] = wv_next[0];
      wv[1] = wv_next[1];
    }
  }
}

template <int kWaves>
__global__ __launch_bounds__(64 * kWaves) __attribute__((amdgpu_waves_per_eu(1, 2)))
void matvec_tiles_kernel(TileArgs a) {
  __shared__ __align__(16384) unsigned char tiles[2 * kWaves * kTileBytes];   // [buffer][wavefront]
  __shared__ __align__(1024) unsigned char blocks[2 * kWaves * kBlockBytes];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const TileLane l = tile_lane(a);
  const Fetch f = fetch_of(a, l.lane);
  // (the rows' min and max are waited for here, while nothing else is on its way)
  asm volatile("" ::"v"(l.rows.lo[0]), "v"(l.rows.lo[1]));
  const lds_bytes my_tiles = (lds_bytes)tiles + wave * kTileBytes;
  const lds_bytes my_blocks = (lds_bytes)blocks + wave * kBlockBytes;
  const int last = a.windows - 1;
  const bool ragged_edge = (a.width & (kCols - 1)) != 0;
  if (ragged_edge) {
    // places that no fetch writes must not hold what LDS happened to hold
    const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int u = 0; u < 16; u++)
        *reinterpret_cast<u32x4 *>(tiles + (b * kWaves + wave) * kTileBytes + (u * 64 + l.lane) * 16) =
            zero;
    // these stores and the fetches below go to LDS by different ways: the
    // zeros must have arrived before the first fetch is asked for
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }

  f32x16 acc[2][2];   // [32 tokens][32 rows] blocks
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

  if (wave < a.windows) {
    int w = wave;
    int cur = 0;   // the buffer that holds, or is about to hold, window w
    fetch_window(tokens_of(a, l), units_of(a, l.block), f, a, l, w, ragged_edge && w == last,
                 my_tiles, my_blocks);
    for (;;) {
      const int wn = __builtin_amdgcn_readfirstlane(w + kWaves);
      const bool more = wn < a.windows;
      const int next = __builtin_amdgcn_readfirstlane(cur ^ 1);
      // that buffer was read a turn ago, and those reads have been waited for
      fetch_window(tokens_of(a, l, more), units_of(a, l.block, more), f, a, l, wn,
                   ragged_edge && wn == last, my_tiles + next * (kWaves * kTileBytes),
                   my_blocks + next * (kWaves * kBlockBytes));
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kLoadsPerWindow) : "memory");
      window_steps_counted(
          static_cast<uint32_t>(reinterpret_cast<uintptr_t>(my_tiles + cur * (kWaves * kTileBytes))),
          static_cast<uint32_t>(reinterpret_cast<uintptr_t>(my_blocks + cur * (kWaves * kBlockBytes))),
          l, acc);
      if (!more) break;
      w = wn;
      cur = next;
    }
  }
  // nothing is on its way into LDS any more
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  finish_tiles<true, 1, kWaves, 2>(a, l, 0, wave, true, (l.rows_here + 31) / 32, tiles, acc);
}

// ---- wavefronts that share what they fetch ------------------------------------
//
// The four or eight wavefronts of a workgroup form kKP parts of the windows
// (part k takes windows k, k + kKP, ...: the sums and their order are those of
// matvec_tiles_kernel<kKP>) times kRG groups of 64 rows; a workgroup owns
// 64 kRG rows and 32 kNB tokens.  The kRG wavefronts of a part bring each
// window of activations into LDS together, once, and every one of them
// multiplies its own rows with it: a window's activations cross the L1 once per
// 64 kRG rows instead of once per 64, and with kNB = 4 a B operand serves 128
// tokens.  The codes go straight into registers.  Eight wavefronts put two on
// a SIMD at the LDS of four: c-2048 wo on 64 tokens 22.5 us instead of 26,
// large wi on 568 11.1 instead of 13.6, both with the end below.
//
// The steps of 16 columns form one pipeline across the windows: while the
// MFMAs of a step run, the B operands of the next step are built and its A
// operands read, also from the last step of a window to the first of the
// next.  A part has two tiles and a wavefront two sets of code registers.
// Before the last step of a window a wavefront waits for all it has asked for
// (its share of the next window, asked for a window ago) and meets the others
// at a barrier: then the next window is there whole, and everyone has read
// the last operands of this one, so during that step the window after the
// next is asked for into this window's tile and registers.  Nothing is counted
// by hand: at the barrier nothing of this wavefront is on its way.  Blocks of
// 32 tokens past the last token are neither multiplied nor stored.

template <int kOff>
__device__ __forceinline__ void lds_request_at(uint32_t at, u32x4 &v) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(v) : "v"(at), "n"(kOff) : "memory");
}
// The operands of kN blocks of 32 tokens (kStride bytes apart), requested only.
template <int kN, int kStride = 8192>
__device__ __forceinline__ void lds_request_blocks(uint32_t at, u32x4 (&v)[kN]) {
  lds_request_at<0>(at, v[0]);
  if constexpr (kN > 1) lds_request_at<kStride>(at, v[1]);
  if constexpr (kN > 2) lds_request_at<2 * kStride>(at, v[2]);
  if constexpr (kN > 3) lds_request_at<3 * kStride>(at, v[3]);
}
template <int kN>
__device__ __forceinline__ void lds_arrived_blocks(u32x4 (&v)[kN]) {
  static_assert(kN >= 1 && kN <= 4, "one to four blocks");
  if constexpr (kN == 1) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v[0])::"memory");
  if constexpr (kN == 2) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v[0]), "+v"(v[1])::"memory");
  if constexpr (kN == 3) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2])::"memory");
  if constexpr (kN == 4)
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3])::"memory");
}

// What a wavefront carries from one step of 16 columns to the next: the A
// operands of kLive blocks of 32 tokens and the B operands of its two units of
// rows.
template <int kLive>
struct StepOperands {
  u32x4 xa[kLive];
  u32x4 wv[2];
};

// One step: 2 kLive MFMAs on `now`.  Each MFMA is followed by an equal share
// of the work for the step after it, which the matrix core's time covers: the
// B operands from half kE of `word0` and `word1` (the codes of the two units),
// and whatever `extra(m)` issues.  The A operands of that step are requested
// from `next_get` before the first MFMA and waited for after the last.  The
// fences keep every MFMA ahead of the work that hides behind it.
template <int kLive, int kNB, int kE, int kStride = 8192, class Extra>
__device__ __forceinline__ void tile_step(StepOperands<kLive> &now, uint32_t next_get,
                                          uint32_t word0, uint32_t word1, const RowTables &rows,
                                          f32x16 (&acc)[kNB][2], Extra &&extra) {
  StepOperands<kLive> next;
  WeightsInTheMaking making;
  // (nothing that derives from the words is to be computed before this step)
  asm volatile("" : "+v"(word0), "+v"(word1));
  lds_request_blocks<kLive, kStride>(next_get, next.xa);
  const bf16x8 wb0 = __builtin_bit_cast(bf16x8, now.wv[0]), wb1 = __builtin_bit_cast(bf16x8, now.wv[1]);
  __builtin_amdgcn_sched_barrier(0);
  auto slot = [&](auto m_c) {
    constexpr int m = decltype(m_c)::value;
    if constexpr (m < 2 * kLive) {
      acc[m >> 1][m & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
          __builtin_bit_cast(bf16x8, now.xa[m >> 1]), m & 1 ? wb1 : wb0, acc[m >> 1][m & 1], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      decode_share<m, 2 * kLive, kE>(making, word0, word1, rows, next.wv);
      extra(m);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  slot(std::integral_constant<int, 0>{});
  slot(std::integral_constant<int, 1>{});
  slot(std::integral_constant<int, 2>{});
  slot(std::integral_constant<int, 3>{});
  slot(std::integral_constant<int, 4>{});
  slot(std::integral_constant<int, 5>{});
  slot(std::integral_constant<int, 6>{});
  slot(std::integral_constant<int, 7>{});
  lds_arrived_blocks<kLive>(next.xa);
  now = next;
}

// A wavefront's share of a window of activations on its way through registers: kLoads pieces
// of eight columns a lane.  `left`: columns of the rows from the window on.  A piece that would reach
// past them (in the last window) is taken from eight columns before the end, and shifted; rows of
// fewer than eight columns, whose matrix is in one part (kNarrow), are read one by one.
template <int kLoads>
struct Pieces {
  u32x4 v[kLoads];
  static __device__ __forceinline__ int past(int col, int left) { return max(col - (left - 8), 0); }
  template <bool kNarrow>
  __device__ __forceinline__ void load(const uint16_t *x, const uint32_t (&at)[kLoads], const int (&col)[4], int left,
                                       bool wide) {
    if (kNarrow && !wide) {
#pragma unroll
      for (int u = 0; u < kLoads; u++) {
        uint32_t e[8];
#pragma unroll
        for (int q = 0; q < 8; q++) e[q] = col[u & 3] + q < left ? x[at[u] + q] : 0u;
        v[u] = u32x4{e[0] | e[1] << 16, e[2] | e[3] << 16, e[4] | e[5] << 16, e[6] | e[7] << 16};
      }
    } else if (left < kCols) {
#pragma unroll
      for (int u = 0; u < kLoads; u++)
        __builtin_memcpy(&v[u], x + static_cast<int>(at[u]) - past(col[u & 3], left), 16);
    } else {
#pragma unroll
      for (int u = 0; u < kLoads; u++) __builtin_memcpy(&v[u], x + at[u], 16);
    }
  }
  __device__ __forceinline__ void store(unsigned char *to, const int (&col)[4], int left, bool wide) {
#pragma unroll
    for (int u = 0; u < kLoads; u++) {
      u32x4 w = v[u];
      if (left < kCols && wide) {
        const int d = past(col[u & 3], left);
        if (d & 4) w = u32x4{w[2], w[3], 0u, 0u};
        if (d & 2) w = u32x4{w[1], w[2], w[3], 0u};
        if (d & 1) w = u32x4{w[0] >> 16 | w[1] << 16, w[1] >> 16 | w[2] << 16, w[2] >> 16 | w[3] << 16, w[3] >> 16};
        if (d >= 8) w = u32x4{0u, 0u, 0u, 0u};
      }
      *reinterpret_cast<u32x4 *>(to + u * 1024) = w;
    }
  }
};

// kDirect (x rows 16-byte aligned, the width a multiple of 8, y in pairs of rows): the activations
// go straight into LDS.  Others come through registers, 16 bytes of any alignment a lane: the loads of
// the window after the next are issued as a window begins, and written to LDS behind the barrier
// that frees its tile.
template <bool kDirect, int kRG, int kKP, int kNB>
__global__ __launch_bounds__(64 * kRG * kKP)
__attribute__((amdgpu_waves_per_eu(kRG * kKP == 8 || kNB <= 2 || kRG == 4 ? 2 : 1, 4)))
void matvec_tiles_shared_kernel(TileArgs a) {
  static_assert(kNB == 1 ? kRG == 1 : (kRG * kKP == 4 || kRG * kKP == 8) && (kNB == 2 || kNB == 4),
                "four or eight wavefronts; blocks of 32 tokens: a wavefront a part");
  constexpr int kTile = kNB * 32 * 256;        // a window of activations
  constexpr int kLoads = 8 * kNB / kRG;        // of them this wavefront's loads
  static_assert(kLoads >= 2, "a load is four tokens");
  extern __shared__ __align__(16384) unsigned char shared_tiles[];   // [part][2][kTile]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = wave % kRG, k = wave / kRG;
  const int blocks = a.units_down / 2;
  TileLane l;
  l.lane = threadIdx.x & 63;
  l.half = l.lane >> 5;
  l.block = blockIdx.x * kRG + g;
  const bool has_rows = l.block < blocks;
  const int live = a.column_blocks + (static_cast<int>(blockIdx.y) < a.larger_columns ? 1 : 0);
  l.t0 = 32 * (blockIdx.y * a.column_blocks + min(static_cast<int>(blockIdx.y), a.larger_columns));
  l.rows_here = min(32 * live, a.tokens - l.t0);
#pragma unroll
  for (int j = 0; j < 2; j++) {
    const int row = l.block * kRows + j * kUnitRows + (l.lane & 31);
    set_tables(l.rows, j,
               row < a.height ? a.minmax[static_cast<int64_t>(a.matrix) * a.height + row] : 0u);
    l.unit_at[j] = static_cast<uint32_t>(j * a.windows * 1024 + l.lane * 16);
  }
  l.get_at = static_cast<uint32_t>((l.lane & 31) * 256 + ((l.half ^ (l.lane & 15)) << 4));
  // Load u of this wavefront brings tokens 4 (g kLoads + u) + lane / 16 of the block, the lane the
  // eight columns from piece_col[u % 4] on: those that belong at its place in LDS.
  int piece_col[4];
  uint32_t piece_at[kLoads];   // kDirect: in bytes; else in elements, of the last token at most
#pragma unroll
  for (int u = 0; u < 4; u++) piece_col[u] = 8 * ((l.lane & 15) ^ ((4 * (g * kLoads + u) + (l.lane >> 4)) & 15));
#pragma unroll
  for (int u = 0; u < kLoads; u++) {
    const int token = 4 * (g * kLoads + u) + (l.lane >> 4);
    piece_at[u] = kDirect ? static_cast<uint32_t>((token * a.ldx + piece_col[u & 3]) * 2)
                          : static_cast<uint32_t>(min(token, l.rows_here - 1) * a.ldx + piece_col[u & 3]);
  }
  const lds_bytes part_tiles = (lds_bytes)shared_tiles + k * (2 * kTile);
  const int last = a.windows - 1;
  const bool ragged_edge = (a.width & (kCols - 1)) != 0;
  if (kDirect && ragged_edge) {
    // places that no fetch writes must not hold what LDS happened to hold
    const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int u = 0; u < 2 * kLoads; u++)
      *reinterpret_cast<u32x4 *>(shared_tiles + k * (2 * kTile) + ((g * 2 * kLoads + u) * 64 + l.lane) * 16) =
          zero;
    __syncthreads();
  }

  f32x16 acc[kNB][2];   // [32 tokens][32 rows] blocks
#pragma unroll
  for (int i = 0; i < kNB; i++)
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0.f;

  // Load u (0 .. kLoads - 1) of this wavefront's share of window w of the
  // activations, into tile `buffer` of its part; and its own codes of window w.
  auto issue_x = [&](const __amdgpu_buffer_rsrc_t &xb, int w, int buffer, int u) {
    const bool edge = ragged_edge && w == last;
    load_to_lds(xb, part_tiles + buffer * kTile + g * (kLoads * 1024) + u * 1024,
                edge && piece_col[u & 3] >= a.width - w * kCols ? kOutside : piece_at[u], w * (kCols * 2));
  };
  Pieces<kDirect ? 1 : kLoads> pieces;
  auto load_pieces = [&](int w, auto may_be_narrow) {   // (narrow rows are one window)
    if constexpr (!kDirect)
      if (w < a.windows)
        pieces.template load<decltype(may_be_narrow)::value>(a.x + static_cast<int64_t>(l.t0) * a.ldx + w * kCols, piece_at, piece_col,
                                       a.width - w * kCols, a.width >= 8);
  };
  auto store_pieces = [&](int w, int buffer) {
    if constexpr (!kDirect)
      if (w < a.windows)
        pieces.store(shared_tiles + k * (2 * kTile) + buffer * kTile + g * (kLoads * 1024) + l.lane * 16, piece_col,
                     a.width - w * kCols, a.width >= 8);
  };
  auto issue_codes = [&](int w, u32x4 (&codes)[2]) {
    const __amdgpu_buffer_rsrc_t ub =
        units_of(a, has_rows ? l.block : 0, has_rows && w < a.windows);
#pragma unroll
    for (int j = 0; j < 2; j++)
      codes[j] = __builtin_bit_cast(
          u32x4, __builtin_amdgcn_raw_buffer_load_b128(ub, l.unit_at[j], w * 1024, 0));
  };

  // The first two windows of this part are asked for at once; from then on
  // the window after the next is asked for during the last step of a window,
  // into the tile and the registers that this window has just finished with.
  const int turns = (a.windows + kKP - 1) / kKP;
  u32x4 codes_a[2], codes_b[2];
  {
    const __amdgpu_buffer_rsrc_t x0 = tokens_of(a, l, k < a.windows);
    const __amdgpu_buffer_rsrc_t x1 = tokens_of(a, l, k + kKP < a.windows);
    if constexpr (kDirect) {
#pragma unroll
      for (int u = 0; u < kLoads; u++) issue_x(x0, k, 0, u);
    }
    load_pieces(k, std::bool_constant<kKP == 1>{});
    issue_codes(k, codes_a);
    store_pieces(k, 0);
    if constexpr (kDirect) {
#pragma unroll
      for (int u = 0; u < kLoads; u++) issue_x(x1, k + kKP, 1, u);
    }
    load_pieces(k + kKP, std::false_type{});
    issue_codes(k + kKP, codes_b);
    store_pieces(k + kKP, 1);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  const uint32_t tile_at[2] = {
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>(part_tiles)) + l.get_at,
      static_cast<uint32_t>(reinterpret_cast<uintptr_t>(part_tiles + kTile)) + l.get_at};

  auto run = [&](auto live_c) {
    constexpr int kLive = decltype(live_c)::value;
    constexpr int kSlots = 2 * kLive;                          // MFMAs of a step
    constexpr int kPerSlot = (kLoads + kSlots - 1) / kSlots;   // loads issued behind each
    StepOperands<kLive> now;
    lds_request_blocks<kLive>(tile_at[0], now.xa);
    WeightsInTheMaking first;
    decode_share<0, 1, 0>(first, codes_a[0][0], codes_a[1][0], l.rows, now.wv);
    lds_arrived_blocks<kLive>(now.xa);
    auto nothing = [](int) {};
    // one window: the tile and codes `cur`, then on to `nxt`
    auto turn_of = [&](int turn, int cur, u32x4 (&codes_cur)[2], u32x4 (&codes_nxt)[2]) {
      const int w = __builtin_amdgcn_readfirstlane(k + turn * kKP);
      const int w2 = w + 2 * kKP;
      const __amdgpu_buffer_rsrc_t x2 = tokens_of(a, l, w2 < a.windows);
      load_pieces(w2, std::false_type{});
      if (has_rows && w < a.windows) {
        const uint32_t get = tile_at[cur];
        tile_step<kLive, kNB, 1>(now, get ^ 32u, codes_cur[0][0], codes_cur[1][0], l.rows, acc, nothing);
        tile_step<kLive, kNB, 0>(now, get ^ 64u, codes_cur[0][1], codes_cur[1][1], l.rows, acc, nothing);
        tile_step<kLive, kNB, 1>(now, get ^ 96u, codes_cur[0][1], codes_cur[1][1], l.rows, acc, nothing);
        tile_step<kLive, kNB, 0>(now, get ^ 128u, codes_cur[0][2], codes_cur[1][2], l.rows, acc, nothing);
        tile_step<kLive, kNB, 1>(now, get ^ 160u, codes_cur[0][2], codes_cur[1][2], l.rows, acc, nothing);
        tile_step<kLive, kNB, 0>(now, get ^ 192u, codes_cur[0][3], codes_cur[1][3], l.rows, acc, nothing);
        tile_step<kLive, kNB, 1>(now, get ^ 224u, codes_cur[0][3], codes_cur[1][3], l.rows, acc, nothing);
        // the next window is there (this wavefront's share of it, and after
        // the barrier everyone's), and everyone has read the last of this one
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const uint32_t word0 = codes_nxt[0][0], word1 = codes_nxt[1][0];
        tile_step<kLive, kNB, 0>(now, tile_at[cur ^ 1], word0, word1, l.rows, acc, [&](int m) {
          if constexpr (kDirect) {
#pragma unroll
            for (int u = m * kPerSlot; u < (m + 1) * kPerSlot && u < kLoads; u++) issue_x(x2, w2, cur, u);
          }
          if (m == kSlots - 1) issue_codes(w2, codes_cur);
        });
        store_pieces(w2, cur);
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if constexpr (kDirect) {
#pragma unroll
          for (int u = 0; u < kLoads; u++) issue_x(x2, w2, cur, u);
        }
        store_pieces(w2, cur);
        issue_codes(w2, codes_cur);
      }
    };
    for (int turn = 0; turn < turns; turn += 2) {
      turn_of(turn, 0, codes_a, codes_b);
      if (turn + 1 < turns) turn_of(turn + 1, 1, codes_b, codes_a);
    }
  };
  if (kNB == 1 || live == kNB)
    run(std::integral_constant<int, kNB>{});
  else if (kNB == 4 && live == 3)
    run(std::integral_constant<int, kNB == 4 ? 3 : kNB>{});
  else
    run(std::integral_constant<int, (kNB + 1) / 2>{});
  // nothing is on its way into LDS any more
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  finish_tiles<kDirect, kRG, kKP, kNB>(a, l, g, k, has_rows, live, shared_tiles, acc);
}

// Parts that the windows of a matrix are cut into: 1, 2 or 4.  The choice depends on
// the matrix alone, never on the tokens of a launch, and the parts are added in
// the same order by all kernels: a token's result is the same whatever launch
// it is part of.  By estimates at nine blocks of 64 tokens (568, the longest sequence of the
// Switch encoders) for matvec_tiles_kernel<n>, in rounds of workgroups, and for workgroups
// of four wavefronts that share their activations.  (They price the kernels as those were first built.
// The estimates below would cut a seventh of all matrices finer: faster on short sequences, slower
// on long ones.  c-2048 wo in four parts: 14.5 us instead of 22.6 on 64 tokens, 43.4 and 41.7
// on 1136, 55.7 and 47.3 on 1900.)
int parts_of(int blocks, int windows) {
  int best = 1;
  double best_cost = 0;
  for (int n = 1; n <= kMaxWaves; n *= 2) {
    const int turns = (windows + n - 1) / n;
    const int64_t slots = 256 * (kMaxWaves / n), tiles = 9;
    double cost = static_cast<double>((blocks * tiles + slots - 1) / slots) * (4.0 + 1.25 * turns);
    if (n <= 2) {
      const int groups = kMaxWaves / n, cap = n == 1 ? 3 : 2;
      const int64_t workgroups = (blocks + groups - 1) / groups * tiles;
      const int64_t per_unit = std::min<int64_t>(cap, (workgroups + 255) / 256);
      const double fill = static_cast<double>(workgroups) / (256.0 * cap);
      const double rounds = fill <= 1.0 ? 1.0 : 0.5 * (std::ceil(fill) + fill);
      cost = std::min(cost, rounds * (4.0 + 1.35 * turns * (1.0 + 0.6 * (per_unit - 1))));
    }
    if (n == 1 || cost < best_cost - 1e-9) {
      best = n;
      best_cost = cost;
    }
  }
  return best;
}

// The forms a launch of a matrix in `parts` parts may take: workgroups of `groups` groups of
// 64 rows (0: one wavefront's own tiles, matvec_tiles_kernel) and 32 `blocks` tokens, `held` of
// which a compute unit holds at once.  One of them takes start + turn us a window of its part; each
// further one on the unit makes `beside` of the windows' time more.  Fitted to 14 shapes, the
// six of Switch among them, on 64 to 2272 tokens (rms 4 to 15 %, the larger ones where 10 us of host
// calls hide the kernel), before columns of 128 tokens were evened out (columns_of), which made those
// faster than the estimate knows.  Of 168 launches now (12 shapes, the six among them, 64 to 2272
// tokens) the form picked is 3.7 % off the fastest on average; 49 are off by more than 5 %: 26 on blocks of
// 64 tokens where 128 would do, by up to 21 % (c-2048 wi on 720 tokens 28.5 us, 23.6 in blocks of 128; large
// wi on 1136 16.3 and 13.9), the others by up to 10 %.
struct TileForm {
  int parts, groups, blocks, held;
  double start, turn, beside;
};
constexpr TileForm kTileForms[] = {
    {1, 0, 2, 4, 4.4, 0.77, 0.09}, {1, 4, 2, 3, 4.2, 0.92, 0.80}, {1, 4, 4, 2, 5.9, 1.37, 1.00},
    {2, 0, 2, 2, 3.2, 0.86, 0.25}, {2, 2, 2, 2, 3.2, 1.16, 0.57}, {2, 4, 2, 2, 5.3, 1.40, 1.60},
    {2, 4, 4, 1, 7.3, 2.20, 0.0},  {4, 0, 2, 1, 2.8, 1.17, 0.0},  {4, 2, 2, 1, 3.7, 1.92, 0.0}};
double cost_of(const TileForm &f, int row_blocks, int windows, int tokens) {
  const int groups = std::max(f.groups, 1), turns = (windows + f.parts - 1) / f.parts;
  const int64_t workgroups = static_cast<int64_t>((row_blocks + groups - 1) / groups) *
                             ((tokens + 32 * f.blocks - 1) / (32 * f.blocks));
  auto with = [&](int64_t on_a_unit) { return f.start + f.turn * turns * (1.0 + f.beside * (on_a_unit - 1)); };
  const int64_t rounds = workgroups / (256 * f.held), rest = workgroups % (256 * f.held);
  return rounds * with(f.held) + (rest ? with((rest + 255) / 256) : 0.0);
}
// `direct`: x and y as the forms on the activations' straight way into LDS need them (`wide`: x).  Blocks of
// 128 tokens have to promise a fifth where there are two parts, and are taken where there is
// one if blocks of 64 would make more workgroups than the chip holds at once: the fit is coarse
// there (c-2048 wi on 1136 tokens 33.0 us, in blocks of 64 38.0; large wi 16.8 and 17.8).
//
// Activations that come through registers, in two or four parts: a workgroup of 64 rows and 32 tokens
// with a wavefront a part, where there are at most two of them for each compute unit (one, where rows of x
// are aligned after all: 1999 x 4000 on 250 tokens 23.5 / 20.4, on 400, 416 workgroups, 24.4 / 26.4).  The forms above
// are then few workgroups, whose loads and decoding nothing hides (us, blocks of 64 tokens / so:
// 1293 x 5497 on 64, 336, 568 tokens 28.4 / 19.1, 33.2 / 23.4, 31.6 / 28.4, on 900, 609 workgroups, 35.4 / 47.1;
// 1675 x 4874 on 336 25.2 / 20.6, on 900, 783, 27.5 / 37.6; in two parts 5003 x 1501 on 128, 316
// workgroups, 13.2 / 12.1, on 200, 553, 14.3 / 14.7, 2081 x 6143 on 400, 429, 48.2 / 41.0).  Where they go straight into LDS it gained 7 % on
// two shapes of thirteen and lost elsewhere.
constexpr TileForm kNarrowForms[] = {{2, 1, 1, 2, 0.0, 0.0, 0.0}, {4, 1, 1, 2, 0.0, 0.0, 0.0}};
const TileForm &pick_form(int parts, int row_blocks, int windows, int tokens, bool direct, bool wide) {
  if (!direct && parts > 1 && static_cast<int64_t>(row_blocks) * ((tokens + 31) / 32) <= (wide ? 1 : 2) * 256)
    return kNarrowForms[parts == 2 ? 0 : 1];
  const TileForm *best = nullptr;
  double best_cost = 0;
  const bool wide_of_one = (row_blocks + 3) / 4 * static_cast<int64_t>((tokens + 63) / 64) > 3 * 256;
  for (const TileForm &f : kTileForms) {
    if (f.parts != parts || (!direct && (f.groups == 0 || f.blocks == 4))) continue;
    if (direct && parts == 1 && f.groups && (f.blocks == 4) != wide_of_one) continue;
    const double cost = cost_of(f, row_blocks, windows, tokens) / (parts == 2 && f.blocks == 4 ? 0.8 : 1.0);
    if (!best || cost < best_cost) {
      best = &f;
      best_cost = cost;
    }
  }
  return *best;
}

std::atomic<int> g_forced_kernel{0};   // sub1_test_tiles_kernel

// The columns of workgroups that a launch's blocks of 32 tokens are shared among, `most` blocks to
// a column or fewer, the larger ones first.  Columns of four blocks that make 1.1 or 1.7
// workgroups a compute unit cost the time of two on every unit; as many columns as make
// whole rounds, if some unit then has fewer blocks to do, even them out (c-2048 wi on 2272 tokens:
// 21 columns of three and four blocks for 18 of four, seven blocks a unit instead of eight:
// 59.4 -> 55.5 us; c-2048 wo 69.4 -> 58.7).
// Launches of many rounds have little to gain.
int columns_of(int tokens, int most, int row_groups) {
  const int token_blocks = (tokens + 31) / 32, least = (token_blocks + most - 1) / most;
  const int64_t rounds = (static_cast<int64_t>(least) * row_groups + 255) / 256;
  if (most < 4 || rounds > 4) return least;
  auto longest = [&](int64_t columns) {   // blocks of the unit that has most
    return token_blocks / columns * rounds + (token_blocks % columns * row_groups + 255) / 256;
  };
  int best = least;
  for (int64_t n = least + 1; n <= std::min<int64_t>(rounds * 256 / row_groups, token_blocks / 2); n++)
    if (longest(n) < longest(best)) best = static_cast<int>(n);
  return best;
}

template <bool kDirect, int kRG, int kKP, int kNB>
int launch_shared_as(TileArgs a, int blocks, hipStream_t stream) {
  constexpr int waves = kRG * kKP;
  constexpr int lds = kKP * 2 * kNB * 32 * 256;
  static_assert(lds >= waves * (kKP - 1) * ((2 * kNB + kKP - 1) / kKP) * 4096 && lds <= 160 * 1024, "tiles, then sums");
  HIP_TRY(sub1::allow_lds<lds>(matvec_tiles_shared_kernel<kDirect, kRG, kKP, kNB>));
  const int row_groups = (blocks + kRG - 1) / kRG, token_blocks = (a.tokens + 31) / 32;
  const int columns = columns_of(a.tokens, kNB, row_groups);
  a.column_blocks = token_blocks / columns;
  a.larger_columns = token_blocks % columns;
  const dim3 grid(row_groups, columns);
  matvec_tiles_shared_kernel<kDirect, kRG, kKP, kNB><<<grid, 64 * waves, lds, stream>>>(a);
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}

template <int kWaves>
int launch_own(const TileArgs &a, int blocks, hipStream_t stream) {
  matvec_tiles_kernel<kWaves><<<dim3(blocks, (a.tokens + kTokens - 1) / kTokens), 64 * kWaves, 0, stream>>>(a);
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}

int launch_form(const TileArgs &a, const TileForm &f, bool direct, int blocks, hipStream_t s) {
  sub1::note_kernel(f.groups == 0   ? "matvec_tiles_kernel"
                    : f.blocks == 4 ? "matvec_tiles_shared_kernel<128>"
                    : f.blocks == 1 ? "matvec_tiles_shared_kernel<32>"
                                    : "matvec_tiles_shared_kernel<64>");
  if (f.groups == 0) {
    if (f.parts == 1) return launch_own<1>(a, blocks, s);
    if (f.parts == 2) return launch_own<2>(a, blocks, s);
    return launch_own<4>(a, blocks, s);
  }
  if (f.blocks == 1) return f.parts == 2 ? launch_shared_as<false, 1, 2, 1>(a, blocks, s) : launch_shared_as<false, 1, 4, 1>(a, blocks, s);
  if (f.parts == 1) {
    if (!direct) return launch_shared_as<false, 4, 1, 2>(a, blocks, s);
    return f.blocks == 4 ? launch_shared_as<true, 4, 1, 4>(a, blocks, s) : launch_shared_as<true, 4, 1, 2>(a, blocks, s);
  }
  if (f.parts == 2 && f.groups == 2)
    return direct ? launch_shared_as<true, 2, 2, 2>(a, blocks, s) : launch_shared_as<false, 2, 2, 2>(a, blocks, s);
  if (f.parts == 2) {
    if (!direct) return launch_shared_as<false, 4, 2, 2>(a, blocks, s);
    return f.blocks == 4 ? launch_shared_as<true, 4, 2, 4>(a, blocks, s) : launch_shared_as<true, 4, 2, 2>(a, blocks, s);
  }
  return direct ? launch_shared_as<true, 2, 4, 2>(a, blocks, s) : launch_shared_as<false, 2, 4, 2>(a, blocks, s);
}

int check_set(const sub1_matrix_set *ms, const char *who) {
  if (!ms) return fail(SUB1_ERR_NULL, "%s: NULL matrix set", who);
  if (!ms->dec || !ms->w_comp || !ms->row_off || !ms->ter_minmax ||
      (ms->count > 1 && !ms->code_base))
    return fail(SUB1_ERR_NULL, "%s: NULL pointer", who);
  if (ms->count < 1 || ms->height < 1 || ms->width < 1 ||
      static_cast<int64_t>(ms->count) * ((ms->height + kRows - 1) / kRows) *
              ((ms->width + kCols - 1) / kCols) > (1 << 28))
    return fail(SUB1_ERR_SHAPE, "%s: %d matrices of %d x %d", who, ms->count, ms->height,
                ms->width);
  if (misaligned(ms->dec, 4) || misaligned(ms->w_comp, 2) || misaligned(ms->row_off, 4) ||
      misaligned(ms->ter_minmax, 4) || misaligned(ms->code_base, 8))
    return fail(SUB1_ERR_ALIGN, "%s: misaligned pointer", who);
  return SUB1_OK;
}

RowSource source_of(const sub1_matrix_set *ms) {
  RowSource s;
  s.dec = ms->dec;
  s.w_comp = reinterpret_cast<const uint16_t *>(ms->w_comp);
  s.code_base = ms->code_base;
  s.row_off = ms->row_off;
  s.count = ms->count;
  s.height = ms->height;
  s.width = ms->width;
  return s;
}

int check_tiles(const sub1_tiles *t, const char *who) {
  if (!t || !t->meta || !t->entries) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (t->count < 1 || t->height < 1 || t->width < 1)
    return fail(SUB1_ERR_SHAPE, "%s: %d matrices of %d x %d", who, t->count, t->height, t->width);
  if (misaligned(t->meta, 256) || misaligned(t->entries, 256))
    return fail(SUB1_ERR_ALIGN, "%s: buffers must be 256-byte aligned", who);
  const TileLayout l = tile_layout(t->count, t->height, t->width);
  if (t->meta_bytes < l.bytes) return fail(SUB1_ERR_SHAPE, "%s: meta smaller than its layout", who);
  if (t->total_chunks != l.units || t->entry_bytes < l.units * 1024)
    return fail(SUB1_ERR_SHAPE, "%s: entries buffer smaller than the layout needs", who);
  return SUB1_OK;
}

}  // namespace

// ================================================================ C ABI =====

extern "C" int64_t sub1_tiles_meta_bytes(int count, int height, int width) {
  if (count < 1 || height < 1 || width < 1) return 0;
  return tile_layout(count, height, width).bytes;
}

extern "C" int sub1_tiles_layout(const sub1_matrix_set *ms, void *meta, int64_t meta_bytes,
                                 sub1_tiles *out, void *stream) {
  const char *who = "sub1_tiles_layout";
  (void)stream;
  int rc = check_set(ms, who);
  if (rc) return rc;
  if (!meta || !out) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (misaligned(meta, 256)) return fail(SUB1_ERR_ALIGN, "%s: meta must be 256-byte aligned", who);
  const TileLayout t = tile_layout(ms->count, ms->height, ms->width);
  if (meta_bytes < t.bytes)
    return fail(SUB1_ERR_SHAPE, "%s: meta needs %lld bytes", who, static_cast<long long>(t.bytes));
  out->meta = meta;
  out->entries = nullptr;
  out->meta_bytes = t.bytes;
  out->total_chunks = t.units;
  out->entry_bytes = t.units * 1024;
  out->count = ms->count;
  out->height = ms->height;
  out->width = ms->width;
  return SUB1_OK;
}

extern "C" int sub1_tiles_entries(const sub1_matrix_set *ms, const sub1_tiles *t, void *stream) {
  const char *who = "sub1_tiles_entries";
  int rc = check_set(ms, who);
  if (rc) return rc;
  rc = check_tiles(t, who);
  if (rc) return rc;
  if (t->count != ms->count || t->height != ms->height || t->width != ms->width)
    return fail(SUB1_ERR_SHAPE, "%s: the layout belongs to other matrices", who);
  const TileLayout l = tile_layout(t->count, t->height, t->width);
  hipStream_t s = static_cast<hipStream_t>(stream);
  char *base = static_cast<char *>(const_cast<void *>(t->meta));
  int32_t *status = reinterpret_cast<int32_t *>(base + l.status);
  u32x4 *units = static_cast<u32x4 *>(const_cast<void *>(t->entries));
  tile_fill_kernel<<<1, 64, 0, s>>>(reinterpret_cast<uint32_t *>(status), 4, 0u);
  const int64_t unit_words = l.units * 256;
  tile_fill_kernel<<<static_cast<unsigned>((unit_words + 255) / 256), 256, 0, s>>>(
      reinterpret_cast<uint32_t *>(units), unit_words, kAllZero);
  const int64_t rows = static_cast<int64_t>(ms->count) * ms->height;
  code_emit_kernel<<<static_cast<unsigned>((rows + 255) / 256), 256, 0, s>>>(
      source_of(ms), l.units_down, l.windows, units, status, rows);
  tile_copy_words_kernel<<<static_cast<unsigned>((rows + 255) / 256), 256, 0, s>>>(
      static_cast<const uint32_t *>(ms->ter_minmax), reinterpret_cast<uint32_t *>(base + l.minmax),
      rows);
  HIP_TRY(hipGetLastError());
  int32_t bad = 0;
  HIP_TRY(hipMemcpyAsync(&bad, status, 4, hipMemcpyDeviceToHost, s));
  HIP_TRY(hipStreamSynchronize(s));
  if (bad) return fail(SUB1_ERR_SHAPE, "%s: the codes of %d rows do not cover the width", who, bad);
  return SUB1_OK;
}

namespace {

int launch_product(const sub1_tiles *t, int matrix, const void *x, int64_t ldx, void *y, int64_t ldy,
                   int tokens, bool fresh, void *stream, const char *who) {
  if (tokens == 0) return SUB1_OK;
  int rc = check_tiles(t, who);
  if (rc) return rc;
  if (!x || !y) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (matrix < 0 || matrix >= t->count) return fail(SUB1_ERR_SHAPE, "%s: no matrix %d", who, matrix);
  if (tokens < 0 || tokens > 65535 * kTokens)   // (a grid's second dimension)
    return fail(SUB1_ERR_SHAPE, "%s: tokens %d outside 0..%d", who, tokens, 65535 * kTokens);
  if (ldx < t->width || ldy < t->height)
    return fail(SUB1_ERR_SHAPE, "%s: token strides smaller than the rows", who);
  if (misaligned(x, 2) || misaligned(y, 2)) return fail(SUB1_ERR_ALIGN, "%s: misaligned pointer", who);
  const TileLayout l = tile_layout(t->count, t->height, t->width);
  const char *base = static_cast<const char *>(t->meta);
  TileArgs a;
  a.units = static_cast<const u32x4 *>(t->entries);
  a.minmax = reinterpret_cast<const uint32_t *>(base + l.minmax);
  a.x = static_cast<const uint16_t *>(x);
  a.y = static_cast<uint16_t *>(y);
  a.ldx = ldx;
  a.ldy = ldy;
  a.height = t->height;
  a.width = t->width;
  a.tokens = tokens;
  a.units_down = l.units_down;
  a.windows = l.windows;
  a.matrix = matrix;
  a.fresh = fresh;
  const bool wide = !misaligned(x, 16) && ldx % 8 == 0 && t->width % 8 == 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (ldx >= (1 << 24) || ldy >= (1 << 24))
    return fail(SUB1_ERR_SHAPE, "%s: token strides of 2^24 elements or more", who);
  // Rows of x that are 16-byte aligned and y in pairs of rows: straight into LDS, or through
  // registers (5003 x 1501 on 64, 568 and 2272 tokens 13.5, 17.7 and 50 us; element by element,
  // a wavefront with tiles of its own, 31, 72 and 263).
  const bool direct = wide && !misaligned(y, 4) && ldy % 2 == 0 && t->height % 2 == 0;
  const int blocks = l.units_down / 2, parts = parts_of(blocks, l.windows);
  const TileForm *form = &pick_form(parts, blocks, l.windows, tokens, direct, wide);
  const int forced = g_forced_kernel.load(std::memory_order_relaxed);
  // (a block's rows of x and y are addressed in 32 bits: 128 of them up to these strides)
  const bool far = ldx >= (1 << 22) || ldy >= (1 << 22);
  if ((forced && direct) || (far && form->blocks == 4))
    for (const TileForm &f : kTileForms)
      if (f.parts == parts && (forced == 1) == (f.groups == 0) &&
          (f.blocks == 4) == (forced == 3 && parts < 4 && !far)) {
        form = &f;
        break;
      }
  return launch_form(a, *form, direct, blocks, s);
}

}  // namespace

extern "C" int sub1_matvec_tiles(const sub1_tiles *t, int matrix, const void *x, int64_t ldx,
                                 void *y, int64_t ldy, int tokens, void *stream) {
  return launch_product(t, matrix, x, ldx, y, ldy, tokens, false, stream, "sub1_matvec_tiles");
}

extern "C" int sub1_product_tiles(const sub1_tiles *t, int matrix, const void *x, int64_t ldx,
                                  void *y, int64_t ldy, int tokens, void *stream) {
  return launch_product(t, matrix, x, ldx, y, ldy, tokens, true, stream, "sub1_product_tiles");
}

extern "C" int sub1_test_tiles_kernel(int which) {
  if (which < 0 || which > 3) return fail(SUB1_ERR_SHAPE, "sub1_test_tiles_kernel: no kernel %d", which);
  g_forced_kernel.store(which, std::memory_order_relaxed);
  return SUB1_OK;
}

extern "C" int sub1_tiles_decode(const sub1_tiles *t, int matrix, void *tern_out, void *stream) {
  const char *who = "sub1_tiles_decode";
  int rc = check_tiles(t, who);
  if (rc) return rc;
  if (!tern_out) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (matrix < 0 || matrix >= t->count) return fail(SUB1_ERR_SHAPE, "%s: no matrix %d", who, matrix);
  const TileLayout l = tile_layout(t->count, t->height, t->width);
  const int64_t n = static_cast<int64_t>(t->height) * t->width;
  code_decode_kernel<<<static_cast<unsigned>((n + 255) / 256), 256, 0,
                        static_cast<hipStream_t>(stream)>>>(
      static_cast<const u32x4 *>(t->entries), static_cast<uint8_t *>(tern_out), matrix,
      l.units_down, l.windows, t->height, t->width);
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}
