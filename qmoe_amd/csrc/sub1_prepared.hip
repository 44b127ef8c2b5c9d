// Prepared expert stack: the fast form of the grouped expert launch.
//
// sub1_moe_prepare_* turn an expert stack in the reference's packed layout
// (reference sub1.py:114-130: one row-major code stream per matrix plus
// row_off) into a form the GPU can stream at full width:
//
//   * every row's dictionary codes are decoded once and its non-zero weights
//     written as a gap-coded stream: 7-bit entries, each the distance to the
//     next non-zero in units of the LDS activation array (2 dwords per column:
//     the activation for a row-min weight and for a row-max weight; every 17th
//     column is a zero column), so an entry names the column and the symbol at
//     once; gaps beyond 127 units step over zero columns.  At 10% non-zeros
//     this is 0.72 bit per weight against 0.69 for the dictionary codes, and
//     the kernel needs no decode table;
//   * rows of every matrix are ordered by entry count and cut into slices of
//     64 rows (one wavefront lane each);
//   * a slice's entries are interleaved in chunks of 9 (8 bytes) per lane:
//     chunk c of lane l sits at slice_base*512 + (c*64 + l)*8 bytes, so one
//     wavefront load fetches 512 contiguous bytes and every byte of a cache
//     line is used; lanes are padded to the slice's longest row with entries
//     that stay on a zero dword.
//
// The kernels then walk 64 rows per wavefront: per entry one address add, one
// LDS read of a bf16 pair (x, 0) or (0, x), and one v_dot2c_f32_bf16 with the
// row's (min, max) pair, which adds x * min or x * max onto the row's fp32 sum;
// no cross-lane traffic at all.  They compute what reference
// sub1_cuda_kernel.cu:163-201 computes per row.
// Four kernels share that loop and give the same bits:
// moe_prepared_fused_kernel streams whole tokens (wi, ReLU, wo in one
// workgroup, h kept in LDS) when there is at least a token per compute unit;
// moe_prepared_shared_kernel lets several workgroups share a token, each in
// both projections, when there are fewer tokens than half the compute units;
// moe_prepared_kernel streams tiles of one matrix (persistent grid, a wavefront
// per slice, the next slice's loads in flight) for the batches in between and
// for single matrices; moe_prepared_small_kernel is the latency form for a
// handful of tokens through single matrices (wavefronts share a slice from
// position checkpoints).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

#include "sub1_common.h"

namespace {

using sub1::bf16_to_f32;
using sub1::f32_to_bf16;
using sub1::fail;
using sub1::misaligned;

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kMaxThreads = 1024;    // 16 wavefronts per workgroup
constexpr int kFields = 9;           // entries per lane per chunk (7 bits each in 8 bytes)
constexpr int kFieldBits = 7;
constexpr int kMaxStep = 127;        // the largest entry
constexpr int kRing = 4;             // chunks in flight per lane (2 KB per wavefront)
constexpr int kGroupChunks = 8;      // chunks (72 entries) per partial sum, a multiple of kRing
constexpr int kSplitRing = 8;        // chunks in flight per lane where wavefronts share a slice
constexpr int kMaxRowEntries = 16383; // entries per row the row ordering can count (widths to 12288)
using sub1::kCtrlBadIds;
using sub1::kCtrlGaveUp;
using sub1::kCtrlHeader;
using sub1::kCtrlTicket;
using sub1::kCtrlTiles;

// ------------------------------------------------------------- meta layout --
//
// One block of device memory, arrays back to back, each 256-byte aligned.
// Kind 0 = wi (rows d_ff, width d_model), kind 1 = wo.
struct KindMeta {
  int64_t slice_base;   // u32 [E*S] (+1): this kind's part of the scanned counts
  int64_t slice_len;    // u16 [E*S]: entries of the slice's longest row
  int64_t row_len;      // u16 [E*H]: entries of every row, in the matrix's own row order
  int64_t row_idx;      // u16 [E*S*64]
  int64_t minmax;       // u32 [E*S*64]
  int slices;           // S
  int height, width;
};

constexpr int kStatusWords = 64, kStatusLong = 4, kLongBits = 32 * (kStatusWords - kStatusLong);
struct MetaLayout {
  KindMeta k[2];
  int kinds;
  int64_t counts;       // i32 [all slices + 1] chunk counts, scanned in place
  int64_t status;       // i32 [kStatusWords]: [0] rows whose codes do not cover the width, [1], [2]
                        // longest slice of kind 0 / 1 in chunks, [3] what check_on_device
                        // found; from [4] on a bit for every slice, mod kLongBits, that has long
                        // rows (emitting)
  int64_t bytes;
};

int64_t align256(int64_t v) { return (v + 255) / 256 * 256; }

// kinds = 2: an expert stack (kind 0 = wi, rows d_ff; kind 1 = wo);
// kinds = 1: `experts` matrices of one shape.
MetaLayout meta_layout(int experts, int kinds, const int height[2], const int width[2]) {
  MetaLayout m;
  m.kinds = kinds;
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    int64_t o = off;
    off += align256(bytes);
    return o;
  };
  int64_t nslices = 0;
  int64_t first[2] = {0, 0};
  for (int i = 0; i < kinds; i++) {
    KindMeta &k = m.k[i];
    k.height = height[i];
    k.width = width[i];
    k.slices = (height[i] + 63) / 64;
    int64_t es = static_cast<int64_t>(experts) * k.slices;
    first[i] = nslices;
    nslices += es;
    k.slice_len = take(es * 2);
    k.row_len = take(static_cast<int64_t>(experts) * height[i] * 2);
    k.row_idx = take(es * 64 * 2);
    k.minmax = take(es * 64 * 4);
  }
  m.counts = take((nslices + 1) * 4);
  for (int i = 0; i < kinds; i++) m.k[i].slice_base = m.counts + first[i] * 4;
  m.status = take(kStatusWords * 4);
  m.bytes = off;
  return m;
}

MetaLayout moe_layout(int experts, int d_model, int d_ff) {
  const int h[2] = {d_ff, d_model}, w[2] = {d_model, d_ff};
  return meta_layout(experts, 2, h, w);
}

MetaLayout matrix_layout(int count, int height, int width) {
  const int h[2] = {height, 0}, w[2] = {width, 0};
  return meta_layout(count, 1, h, w);
}

// ---------------------------------------------------------- prepare kernels --

// A slice is as long as its longest row, counted in ENTRIES; its chunks, and how
// many entries of the last one are walked (1..9; the rest of that chunk is
// padding nobody reads).
__host__ __device__ constexpr int chunks_of(int len) { return (len + kFields - 1) / kFields; }
__host__ __device__ constexpr int last_entries_of(int len) { return len - kFields * (chunks_of(len) - 1); }

// Positions.  The kernels keep the activations in LDS by physical column: real
// column c is physical column q = c + c/16 + 1, so that every 17th physical
// column (0, 17, 34, ...) is a zero column; a physical column is two dwords,
// and position p = 2q + (symbol - 1) is the dword a weight with that symbol
// reads: (x, 0) for a row-min weight, (0, x) for a row-max weight, zero in a
// zero column.  The low bit of a position is the symbol, the rest the column.
constexpr int kZeroPeriod = 17;                  // physical columns from one zero column to the next
__host__ __device__ constexpr int physical_column(int c) { return c + (c >> 4) + 1; }
__host__ __device__ constexpr int position_of(int c, int sym) {
  return 2 * physical_column(c) + (sym - 1);
}
// Physical columns an array for `width` real columns needs: up to and including
// the zero column that follows the last real one.
__host__ __device__ constexpr int physical_columns(int width) {
  return (physical_column(width - 1) / kZeroPeriod + 1) * kZeroPeriod + 1;
}

// Where the matrices of one kind come from: one buffer of codes with a base
// offset per matrix and [count, height + 1] / [count, height] arrays of row
// offsets and (min, max) - an expert stack - or, with the *_of tables set, a
// device array of device pointers per buffer, one entry per matrix - the
// layers' own tensors, wherever they lie.
struct KindSource {
  const uint16_t *w_comp;
  const int64_t *code_base;      // NULL with one matrix: its codes start at w_comp
  const int32_t *row_off;
  const uint32_t *minmax;
  const uint16_t *const *w_comp_of;
  const int32_t *const *row_off_of;
  const uint32_t *const *minmax_of;
};

// A row of more than `average` times its matrix's average of codes (and a few) is a LONG one.  Twice
// where there is at most one group of 64 rows or two to a compute unit: a group waits for its longest row, and
// hardly anything else is there to do.  More of them hide that, and the words of the dictionary that long rows take
// from memory count: as many times as a unit has groups, up to 4.2.  (Preparing, rows with 90 % zeros, us, a lane to every
// row / to eight codes of the rows without zeros, of which there are a tenth, a fifth, two fifths.  One 6144 x 2080
// 325 / 171, 331 / 181, 323 / 195; eight, 3 groups a unit, 372 / 253, 361 / 331, 346 / 500; 64 base
// experts, 15 a unit, 523 / 509, 509 / 740, 501 / 1300; 30 of c-2048 936 / 1000, 959 / 1630, 1055 / 2770.)
constexpr float kLongFromFew = 2.f, kLongFromMany = 4.2f;
constexpr int kLongRowsFrom = 16;
__device__ __forceinline__ const uint16_t *row_codes(const KindSource &ks, int e, int r, int height, int width,
                                                     float average, int &n, bool &is_long) {
  const int32_t *ro = ks.row_off_of ? ks.row_off_of[e]
                                    : ks.row_off + static_cast<int64_t>(e) * (height + 1);
  n = ro[r + 1] - ro[r];
  if (n < 1 || n > (width + 1) / 2) n = 0;   // counted as a bad row by walk_rows_kernel
  // (the sixteen: short rows stay with the lanes; in floating point, which a division costs less in)
  is_long = n > kLongRowsFrom && static_cast<float>(n - kLongRowsFrom) * height > average * static_cast<float>(ro[height]);
  const uint16_t *codes = ks.w_comp_of ? ks.w_comp_of[e]
                                       : ks.w_comp + (ks.code_base ? ks.code_base[e] : 0);
  return codes + ro[r];
}

// Both prepare passes walk all rows' codes, a lane to a row.  What bounds them is the
// instructions for a code and, before those, fetching its dictionary entry: a wavefront's
// gather from a table in global memory costs a compute unit 54 ns, one from LDS 3 ns.
// So a compute unit takes one workgroup, persistent, that keeps a table in LDS, and a
// lane asks for eight codes and their eight entries at once.
//
// A wavefront of rows takes as long as the longest of them, and a row without zeros has
// seven times the codes of others.  Long rows are therefore left aside, for a lane to take eight of
// their codes: counting notes them in LDS and does them last, emit_long_rows_kernel emits them.
//
// Counting needs little of an entry, 16 bits, so that all 65 536 are held, and beside
// them two more bits of each for the rare gap that takes several steps:
//   bits 0-3 pairs, 4-5 non-zeros, 6-10 column of the first, 11-15 columns from the
//   last to the entry's end (0 where there is none); symbols - 1 of the first and the
//   last non-zero.
// Emitting needs all of it, a word: pairs in bits 0-3, non-zeros in 4-5, then a byte for
// each of three: 2 column + symbol - 1, the last one's again where there are fewer.  The
// first 40 000 words are held (the low codes are the frequent ones: three quarters of
// the codes of weights with 90% zeros and more).
constexpr int kWalkThreads = 1024;
constexpr int kHeldWords = 40000;
constexpr int kCountWords = SUB1_DICT_ENTRIES / 2 + SUB1_DICT_ENTRIES / 16;   // 16-bit entries, then symbols
constexpr size_t kWalkLds = kHeldWords * sizeof(uint32_t);
constexpr int kLongList = 2048;   // long rows of a workgroup that counting leaves aside (a lane walks what there are more)
constexpr size_t kCountLds = (kCountWords + kLongList) * sizeof(uint32_t);

struct HeldTable {
  const uint32_t *all;    // global memory
  const uint32_t *head;   // LDS
  __device__ __forceinline__ uint32_t operator[](uint32_t code) const {
    // lanes whose code is held read the table's first word, one line for all of them
    const uint32_t far = all[code < kHeldWords ? 0u : code];
    const uint32_t near = head[min(code, kHeldWords - 1u)];
    return code < kHeldWords ? near : far;
  }
};

struct CountTable {
  const uint32_t *words;   // global memory: the emitting pass's words
  const uint32_t *lds;
  __device__ __forceinline__ uint32_t operator[](uint32_t code) const {
    return reinterpret_cast<const uint16_t *>(lds)[code];
  }
  __device__ __forceinline__ uint32_t symbols(uint32_t code) const {   // bit 0 of the first, bit 1 of the last
    return lds[SUB1_DICT_ENTRIES / 2 + (code >> 4)] >> (2 * (code & 15u));
  }
};

__device__ __forceinline__ void hold_table(const uint32_t *table, uint32_t *lds, int words) {
  for (int i = 4 * threadIdx.x; i < words; i += 4 * kWalkThreads)
    *reinterpret_cast<uint4 *>(lds + i) = *reinterpret_cast<const uint4 *>(table + i);
  __syncthreads();
}

// The rows' codes are followed through pointers read from memory; as a global
// address, a load of them need not wait for the LDS too.
typedef const __attribute__((address_space(1))) uint16_t global_u16;
typedef uint32_t unaligned_u32x4 __attribute__((ext_vector_type(4), aligned(2)));   // eight codes
__device__ __forceinline__ unaligned_u32x4 eight_codes(global_u16 *codes) {
  return *(const __attribute__((address_space(1))) unaligned_u32x4 *)codes;
}

// A row's codes in turn to each(entry, code), eight entries fetched at a time, and the
// last one to eight of them to last_ones(entry, code), where entries of no pairs and no
// non-zeros stand in for what is missing to eight.
template <class Table, class Each, class Last>
__device__ __forceinline__ void walk_codes(const Table &table, const uint16_t *row, int n, Each &&each,
                                           Last &&last_ones) {
  global_u16 *codes = (global_u16 *)row;
  if (n < 8) {
#pragma unroll 1
    for (int i = 0; i < n; i++) last_ones(table[codes[i]], static_cast<uint32_t>(codes[i]));
    return;
  }
  unaligned_u32x4 next = eight_codes(codes);
  uint32_t code[8], w[8];
  auto look_up = [&]() {
#pragma unroll
    for (int j = 0; j < 8; j++) {
      code[j] = (j & 1) ? next[j / 2] >> 16 : next[j / 2] & 0xffffu;
      w[j] = table[code[j]];
    }
  };
  int i = 0;
#pragma unroll 1
  for (; i + 8 < n; i += 8) {
    look_up();
    next = eight_codes(codes + min(i + 8, n - 8));   // the last, partial eight: from eight before the end
#pragma unroll
    for (int j = 0; j < 8; j++) each(w[j], code[j]);
  }
  look_up();
#pragma unroll
  for (int j = 0; j < 8; j++) last_ones(j < i + 8 - n ? 0u : w[j], code[j]);
}

// A row's non-zeros as entries.  An entry is the step from the row's position (0 at
// the start) to the next, 0..127; a longer gap goes over zero columns, as far as each
// step reaches: the place that such a step ends at.
constexpr int kZeroStep = kMaxStep / (2 * kZeroPeriod) * (2 * kZeroPeriod);   // from one zero column as far as a step goes
__host__ __device__ constexpr int farthest_zero(int at) {
  return (at + kMaxStep) / (2 * kZeroPeriod) * (2 * kZeroPeriod);
}
// Entries before the last one of a gap: while the target is too far, to the farthest zero
// column; from the second such step on they are of one length.
__host__ __device__ constexpr int steps_between(int at, int target) {
  if (target - at <= kMaxStep) return 0;
  const int rest = target - farthest_zero(at) - kMaxStep;
  return 1 + (rest > 0 ? (rest + kZeroStep - 1) / kZeroStep : 0);
}
// The position of 2 column + symbol - 1.  (Written out: the compiler takes one more.)
__device__ __forceinline__ int position_at(int a) {
  int p;
  asm("v_lshl_add_u32 %0, %1, 1, %2" : "=v"(p) : "v"(a >> 5), "v"(a + 2));
  return p;
}
// n ? a : b, without a branch around what may differ from lane to lane.
__device__ __forceinline__ int pick(int n, int a, int b) {
  asm volatile("" : "+v"(a), "+v"(b));
  return n ? a : b;
}

// A prepare pass over all rows of one kind of matrices, 64 at a time; kinds with
// longer rows first, so that the launch does not end on them.
struct WalkKind {
  KindSource source;
  int height, width, slices;
  float long_from;              // from how many times a matrix's average of codes on a row is a long one
  int64_t tasks;                // of 64 rows (counting: in the matrices' own order; emitting: slices)
  int64_t first_slice;          // emitting: among all kinds' slices
  uint16_t *row_len;            // counting
  const uint32_t *slice_base;   // emitting
  const uint16_t *slice_len, *row_idx;
};
struct WalkArgs {
  WalkKind k[2];
  int kinds, count;
  const uint32_t *table;         // the emitting pass's words, all of them
  const uint32_t *count_table;   // what the counting pass holds in LDS
  const int32_t *found;          // what check_source_kernel has found: nothing is followed unless zero
  uint32_t *long_bits;           // emitting: long rows are another launch's, and these slices have some (NULL: they are not)
  sub1::Answer answer;           // emitting: the first word says what that is
  int32_t *status;
  uint2 *stream;
  uint16_t *ckpt;
};

// Columns from a row's last non-zero to the next from which on one step may not do:
// 60 columns are 63 or 64 physical ones, 126 to 129 positions.
constexpr int kLongGap = 60;

// How many entries the non-zeros of every row take (the step onto a zero column
// that a padded row makes after them is not counted: it fits the padding).  An entry's
// non-zeros are 27 columns apart at most, so only the gap before the first of them can
// take more than one.
__device__ __forceinline__ const uint16_t *task_row(const WalkKind &k, int64_t task, int lane, int &n, bool &is_long) {
  // rows of a task: from row `first` of a matrix on, and of the next ones
  const int first_e = static_cast<int>(task * 64 / k.height);
  const uint32_t past = static_cast<uint32_t>(task * 64 + lane - static_cast<int64_t>(first_e) * k.height);
  const int e = first_e + static_cast<int>(past / static_cast<uint32_t>(k.height));
  const int r = static_cast<int>(past % static_cast<uint32_t>(k.height));
  return row_codes(k.source, e, r, k.height, k.width, k.long_from, n, is_long);
}
__device__ __forceinline__ void count_rows(const CountTable &table, const WalkKind &k, int count,
                                           int64_t task, int turn, int32_t *status, uint32_t *longs, int *n_longs) {
  const int lane = threadIdx.x & 63;
  const int64_t g = task * 64 + lane;
  if (g >= static_cast<int64_t>(count) * k.height) return;
  int n;
  bool is_long;
  const uint16_t *codes = task_row(k, task, lane, n, is_long);
  if (is_long) {
    const int i = atomicAdd(n_longs, 1);
    if (i < kLongList) {
      longs[i] = static_cast<uint32_t>(turn) << 6 | static_cast<uint32_t>(lane);
      return;
    }
  }
  int col = 0, entries = 0;
  int since = 0;       // columns from the last non-zero's to col (from column 0 where there is none)
  int holder = -1;     // the code that holds the last non-zero
  auto step = [&](uint32_t w, uint32_t code, bool over) {
    const int nonzeros = (w >> 4) & 3u, first = (w >> 6) & 31u, tail = w >> 11;
    const int pairs = w & 15u;
    if (__builtin_expect(since + first >= kLongGap || over, 0)) {
      // digits past the width are dropped: which those are, the whole entry says
      int inside = nonzeros;
      if (over) {
        const uint32_t all = table.words[code];
        inside = 0;
        for (int j = 0; j < nonzeros; j++)
          if (2 * col + static_cast<int>((all >> (8 + 8 * j)) & 255u) < 2 * k.width) inside++;
      }
      if (inside) {
        int at = holder < 0 ? 0 : position_at(2 * (col - since)) + static_cast<int>((table.symbols(holder) >> 1) & 1u);
        const int target = position_at(2 * (col + first)) + static_cast<int>(table.symbols(code) & 1u);
        while (target - at > kMaxStep) {
          at = farthest_zero(at);
          entries++;
        }
      }
      entries -= nonzeros - inside;   // what is added below; nothing follows a dropped digit
    }
    entries += nonzeros;
    col += 2 * pairs;
    since = pick(nonzeros, tail, since + 2 * pairs);
    holder = pick(nonzeros, static_cast<int>(code), holder);
  };
  // (only a row's last code can reach past its width, if its codes cover it exactly)
  walk_codes(table, codes, n, [&](uint32_t w, uint32_t code) { step(w, code, false); },
             [&](uint32_t w, uint32_t code) {
               step(w, code, (w & 0x30u) && col + 2 * static_cast<int>(w & 15u) > k.width);
             });
  // a row's codes cover its width rounded up to a whole pair, exactly
  if (col != ((k.width + 1) & ~1)) atomicAdd(&status[0], 1);
  k.row_len[g] = static_cast<uint16_t>(min(entries, kMaxRowEntries));
}

// Position checkpoints.  For every slice and every group of kGroupChunks chunks,
// the position at which each lane's row stands when the group begins: 64 x u16
// per group, groups of slice g stored from entry slice_base[g]/kGroupChunks + g
// on.  With them a wavefront can start in the middle of a slice, which is how a
// small batch is spread over the GPU.
__device__ __forceinline__ int64_t checkpoint_entry(uint32_t slice_base, int64_t slice) {
  return static_cast<int64_t>(slice_base / kGroupChunks) + slice;
}

// A row's entries, nine to a chunk, a codeword's (up to three) at a time.  The lanes of a
// wavefront fill their chunks at different times, so that nearly every place that may
// store one is taken by a few of them: there is one such place to a codeword.
// kShared: a chunk may hold entries of other lanes', before these or behind, and is zero before
// all of them.
template <bool kShared>
struct ChunkSink {
  char *chunks, *ckpt;          // the slice's; the same in all lanes (kShared: a row of the slice each)
  uint32_t end;                 // bytes of its chunks
  uint32_t at;                  // of this lane's next one: 512 c + 8 (the row's place)
  int bits = 0;                 // that it holds, seven an entry
  uint32_t lo = 0, hi = 0;
  __device__ __forceinline__ void put() {
    if (at >= end) return;
    if (kShared)
      __hip_atomic_fetch_or(reinterpret_cast<unsigned long long *>(chunks + at),
                            static_cast<unsigned long long>(hi & 0x7fffffffu) << 32 | lo, __ATOMIC_RELAXED,
                            __HIP_MEMORY_SCOPE_WORKGROUP);
    else
      *reinterpret_cast<uint2 *>(chunks + at) = make_uint2(lo, hi & 0x7fffffffu);
  }
  // The chunk is stored and the next one begins with the entries in `rest` (two at most);
  // `position`: what the row has reached with them.
  __device__ __forceinline__ void store(uint32_t rest, int position) {
    put();
    at += 512;
    if ((at & (kGroupChunks - 1) << 9) == 0 && at < end)
      *reinterpret_cast<uint16_t *>(ckpt + ((at >> 12) * 128 + (at & 511u) / 4)) =
          static_cast<uint16_t>(position - static_cast<int>((rest & 127u) + (rest >> kFieldBits)));
    lo = rest;
    hi = 0;
    bits -= kFields * kFieldBits;
  }
  // `n` entries (0 to 3), the first in the lowest bits of `packed`.
  __device__ __forceinline__ void add(uint32_t packed, int n, int position) {
    const unsigned long long shifted = static_cast<unsigned long long>(packed) << bits;
    lo |= static_cast<uint32_t>(shifted);
    hi |= static_cast<uint32_t>(shifted >> 32);
    const int room = kFields * kFieldBits - bits;
    bits += kFieldBits * n;
    if (bits >= kFields * kFieldBits) store(packed >> room, position);
  }
};
static_assert(kGroupChunks == 8, "a group's chunks are 4096 bytes");

// The zero column from which on a row stays where it is.
__device__ __forceinline__ int next_zero(int at) { return (at + 2 * kZeroPeriod - 1) / (2 * kZeroPeriod) * (2 * kZeroPeriod); }
// Non-zeros of a codeword (places a0, a1, a2: 2 column + symbol - 1) that are within the width; the
// others' positions become the last one's.
__device__ __forceinline__ int inside_width(int nonzeros, int a0, int a1, int a2, int width, int p0, int &p1, int &p2) {
  if (a2 >= 2 * width) {   // digits past the width are dropped
    nonzeros = min(nonzeros, 2);
    p2 = p1;
  }
  if (a1 >= 2 * width) {
    nonzeros = min(nonzeros, 1);
    p1 = p2 = p0;
  }
  return a0 >= 2 * width ? 0 : nonzeros;
}

// Where a slice goes.
struct SliceOut {
  char *chunks, *ckpt;
  int len;
  uint32_t end;   // bytes of its chunks
};
__device__ __forceinline__ SliceOut slice_out(const WalkKind &k, int64_t slice, uint2 *stream, uint16_t *ckpt) {
  const uint32_t base = __builtin_amdgcn_readfirstlane(k.slice_base[slice]);
  const int len = __builtin_amdgcn_readfirstlane(k.slice_len[slice]);
  return {reinterpret_cast<char *>(stream + static_cast<int64_t>(base) * 64),
          reinterpret_cast<char *>(ckpt + checkpoint_entry(base, k.first_slice + slice) * 64), len, 512u * chunks_of(len)};
}

// A slice's rows, a lane each, into the interleaved stream, nine entries to a chunk;
// a row shorter than its slice then steps onto the next zero column and stays there
// (steps of 0) to the end of the slice's last chunk; and the row's position at the
// start of every group of chunks into the checkpoints.
__device__ __forceinline__ void emit_rows(const HeldTable &table, const WalkKind &k, int64_t slice,
                                          uint2 *__restrict__ stream, uint16_t *__restrict__ ckpt,
                                          uint32_t *long_bits) {
  const int lane = threadIdx.x & 63;
  const int e = static_cast<int>(slice / k.slices);
  const int ridx = k.row_idx[slice * 64 + lane];
  const SliceOut s = slice_out(k, slice, stream, ckpt);
  ChunkSink<false> sink{s.chunks, s.ckpt, s.end, 8u * lane};
  *reinterpret_cast<uint16_t *>(sink.ckpt + 2 * lane) = 0;
  int at = 0;
  if (ridx != 0xffff) {
    int n;
    bool is_long;
    const uint16_t *codes = row_codes(k.source, e, ridx, k.height, k.width, k.long_from, n, is_long);
    if (is_long && long_bits) {
      const uint32_t bit = static_cast<uint32_t>(k.first_slice + slice) % kLongBits;
      atomicOr(&long_bits[bit / 32], 1u << (bit % 32));
      return;
    }
    int from = 0;   // twice the column at which the codeword starts
    auto step = [&](uint32_t w, uint32_t) {
      int nonzeros = (w >> 4) & 3u;
      const int a0 = from + static_cast<int>((w >> 8) & 255u), a1 = from + static_cast<int>((w >> 16) & 255u);
      const int a2 = from + static_cast<int>(w >> 24);
      const int p0 = position_at(a0);
      int p1 = position_at(a1), p2 = position_at(a2);
      const int end = from + 4 * static_cast<int>(w & 15u);
      if (__builtin_expect(p0 - at > kMaxStep || end > 2 * k.width, 0)) {
        if (end > 2 * k.width) nonzeros = inside_width(nonzeros, a0, a1, a2, k.width, p0, p1, p2);
        if (nonzeros)
#pragma unroll 1
          while (p0 - at > kMaxStep) {
            const int zero = farthest_zero(at);
            sink.add(zero - at, 1, zero);
            at = zero;
          }
      }
      const int packed = (p0 - at) | (p1 - p0) << kFieldBits | (p2 - p1) << (2 * kFieldBits);
      at = pick(nonzeros, p2, at);
      sink.add(static_cast<uint32_t>(pick(nonzeros, packed, 0)), nonzeros, at);
      from = end;
    };
    walk_codes(table, codes, n, step, step);
    if (static_cast<int>(sink.at >> 9) * (kFields * kFieldBits) + sink.bits < s.len * kFieldBits && (at >> 1) % kZeroPeriod != 0) {
      // padding follows: it must read zeros
      const int zero = next_zero(at);
      sink.add(zero - at, 1, zero);
      at = zero;
    }
  }
#pragma unroll 1
  while (sink.at < sink.end) sink.store(0u, at);
}

// ------------------------------------------------------------- long rows --
//
// A wavefront takes a long row, a lane a GROUP of eight of its codes.  What a group has to know
// of the codes before it (the column, the last non-zero, the entries so far) comes from prefix
// sums over the lanes and, from one turn of 64 groups to the next, from the last lane: twice the
// instructions a code, but a row of 1024 codes is two turns and not 1024 steps.  The dictionary's words
// come from global memory: these are few codes.
//
// 63 base experts whose rows have 75 to 98 % zeros, one in a hundred none: counting 177 us before,
// 54 with that (ordering them 15), emitting 303, 104 and 75 in a launch of its own.  (Taken by groups where they are met
// they make the walks of even rows slower, by 2 of 33 and 4 of 85 us, with none there; counted by the
// workgroup that orders their matrix, one 6144 x 2080 with two fifths of them takes 1400 us to prepare, 320 with a
// lane to each, 195 now.)
constexpr int kGroupOfCodes = 8;

// Eight of a row's codes, from code `at` on, and which of them there are.  (Loads stay within
// the row: its last, partial eight is read from eight before its end.)
struct EightCodes {
  unaligned_u32x4 v;
  uint32_t present;
  __device__ __forceinline__ EightCodes(const uint16_t *codes, int n, int at) {   // n > kLongRowsFrom
    const int here = min(max(n - at, 0), kGroupOfCodes);
    present = (0xffu << (kGroupOfCodes - here)) & 0xffu;
    v = here ? eight_codes((global_u16 *)codes + min(at, n - kGroupOfCodes)) : unaligned_u32x4{0, 0, 0, 0};
  }
  __device__ __forceinline__ uint32_t word(const uint32_t *table, int j) const {
    const uint32_t code = (j & 1) ? v[j / 2] >> 16 : v[j / 2] & 0xffffu;
    return table[code] & static_cast<uint32_t>(static_cast<int32_t>(present << (31 - j)) >> 31);
  }
};

// A codeword's entries: long steps, then a step to each non-zero.
struct CodeSteps {
  int more, nonzeros;
  uint32_t packed;
  // from (twice the column) and at (the position): where the row stands before it, and then behind it
  __device__ __forceinline__ CodeSteps(uint32_t w, int width, int &from, int &at) {
    nonzeros = (w >> 4) & 3u;
    const int a0 = from + static_cast<int>((w >> 8) & 255u), a1 = from + static_cast<int>((w >> 16) & 255u);
    const int a2 = from + static_cast<int>(w >> 24);
    const int p0 = position_at(a0);
    int p1 = position_at(a1), p2 = position_at(a2), here = at;
    more = 0;
    from += 4 * static_cast<int>(w & 15u);
    if (__builtin_expect(p0 - at > kMaxStep || from > 2 * width, 0)) {
      if (from > 2 * width) nonzeros = inside_width(nonzeros, a0, a1, a2, width, p0, p1, p2);
      if (nonzeros) {
        more = steps_between(at, p0);
        if (more) here = farthest_zero(at) + (more - 1) * kZeroStep;
      }
    }
    packed = static_cast<uint32_t>(
        pick(nonzeros, (p0 - here) | (p1 - p0) << kFieldBits | (p2 - p1) << (2 * kFieldBits), 0));
    at = pick(nonzeros, p2, at);
  }
};

// A long row's turns of 64 groups to turn(words, from, at), which moves from and at (twice the
// column and the position, before the group) on to behind it; all lanes together.
template <class Turn>
__device__ __forceinline__ void walk_long_row(const uint32_t *table, const uint16_t *codes, int n, Turn &&turn) {
  const int lane = threadIdx.x & 63;
  int carry_from = 0, carry_at = 0;
  EightCodes next(codes, n, kGroupOfCodes * lane);
#pragma unroll 1
  for (int first = 0; first < n; first += 64 * kGroupOfCodes) {
    const EightCodes now = next;
    next = EightCodes(codes, n, first + (64 + lane) * kGroupOfCodes);
    uint32_t w[kGroupOfCodes];
#pragma unroll
    for (int j = 0; j < kGroupOfCodes; j++) w[j] = now.word(table, j);
    int span = 0, key = 0;   // twice the group's columns; one more than its last non-zero's 2 column + symbol - 1
#pragma unroll
    for (int j = 0; j < kGroupOfCodes; j++) {
      key = pick(w[j] & 0x30u, span + static_cast<int>(w[j] >> 24) + 1, key);
      span += 4 * static_cast<int>(w[j] & 15u);
    }
    const int before = sub1::wave_prefix_sum(span) - span;
    const int below = sub1::wave_max_below(key ? before + key : 0);
    int from = carry_from + before;
    int at = below ? position_at(carry_from + below - 1) : carry_at;
    turn(w, from, at, first + kGroupOfCodes * lane < n, first + kGroupOfCodes * (lane + 1) >= n);
    carry_from = __builtin_amdgcn_readlane(from, 63);
    carry_at = __builtin_amdgcn_readlane(at, 63);
  }
}

__device__ __forceinline__ const uint16_t *codes_of_lane(const uint16_t *codes, int lane) {
  const uint64_t address = reinterpret_cast<uint64_t>(codes);
  const uint32_t low = __builtin_amdgcn_readlane(static_cast<int>(address), lane);
  const uint32_t high = __builtin_amdgcn_readlane(static_cast<int>(address >> 32), lane);
  return reinterpret_cast<const uint16_t *>(static_cast<uint64_t>(high) << 32 | low);
}

// The entries of the long rows that a workgroup has left aside (as `turn` << 6 | lane), its
// wavefronts in turn.
__device__ __forceinline__ void count_long_rows(const WalkArgs &a, const uint32_t *longs, int n_longs) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr int kWaves = kWalkThreads / 64;
  for (int first = wave; first < n_longs; first += 64 * kWaves) {
    // a lane asks for where one of them is
    const int i = first + kWaves * lane;
    const int here = min((n_longs - first + kWaves - 1) / kWaves, 64);
    int n = 0;
    int64_t g = 0;
    bool second = false;
    const uint16_t *codes = nullptr;
    if (lane < here) {
      const uint32_t what = longs[i];
      int64_t task = blockIdx.x + static_cast<int64_t>(gridDim.x) * (what >> 6);
      second = task >= a.k[0].tasks;
      if (second) task -= a.k[0].tasks;
      bool is_long;
      codes = task_row(a.k[second ? 1 : 0], task, what & 63u, n, is_long);
      g = task * 64 + (what & 63u);
    }
    uint16_t entries_of = 0;
    for (int who = 0; who < here; who++) {
      const int width = a.k[__builtin_amdgcn_readlane(second, who)].width;
      int entries = 0;
      walk_long_row(a.table, codes_of_lane(codes, who), __builtin_amdgcn_readlane(n, who),
                    [&](const uint32_t (&w)[kGroupOfCodes], int &from, int &at, bool live, bool ends) {
#pragma unroll
                      for (int j = 0; j < kGroupOfCodes; j++) {
                        const CodeSteps c(w[j], width, from, at);
                        entries += c.nonzeros + c.more;
                      }
                      // a row's codes cover its width rounded up to a whole pair, exactly
                      if (live && ends && from != 2 * ((width + 1) & ~1)) atomicAdd(&a.status[0], 1);
                    });
      entries = __builtin_amdgcn_readlane(sub1::wave_prefix_sum(entries), 63);
      if (lane == who) entries_of = static_cast<uint16_t>(min(entries, kMaxRowEntries));
    }
    if (lane < here) a.k[second ? 1 : 0].row_len[g] = entries_of;
  }
}

// Task t goes to workgroup t mod grid: a matrix of a few slices is spread over as many
// compute units.  Within it the wavefronts take the next one when they are done: a row of
// wo has four times the codes of one of wi, and dealt out beforehand the busiest wavefront
// has 1.7 times the average (counting 40 us, emitting 96).
// 128 base experts (26 million codes): counting takes 32 us, 22 vector instructions a code
// (64 with entry by entry of a whole word, 60 instructions); emitting 84 and about 65 (113
// with a place that may store behind every entry, 99 instructions).  Both are bound by
// issuing those, beside 6 us of filling LDS.  (32 codes asked for together instead of 8,
// a cache line's worth: 37 and 81 us.)
template <bool kEmit>
__global__ __launch_bounds__(kWalkThreads) void walk_rows_kernel(WalkArgs a) {
  extern __shared__ __align__(16) uint32_t held[];
  __shared__ int s_turn, s_longs;
  const int found = *a.found;
  if (kEmit && blockIdx.x == 0 && threadIdx.x == 0) sub1::tell(a.answer, 0, found);
  if (found) return;
  if (threadIdx.x == 0) {
    s_turn = 0;
    s_longs = 0;
  }
  hold_table(kEmit ? a.table : a.count_table, held, kEmit ? kHeldWords : kCountWords);
  const int64_t all = a.k[0].tasks + (a.kinds == 2 ? a.k[1].tasks : 0);
  for (;;) {
    int turn = 0;
    if ((threadIdx.x & 63) == 0) turn = atomicAdd(&s_turn, 1);
    turn = __builtin_amdgcn_readfirstlane(turn);
    int64_t task = blockIdx.x + static_cast<int64_t>(gridDim.x) * turn;
    if (task >= all) break;
    const bool second = task >= a.k[0].tasks;
    if (second) task -= a.k[0].tasks;
    const WalkKind &k = a.k[second ? 1 : 0];
    if (kEmit)
      emit_rows(HeldTable{a.table, held}, k, task, a.stream, a.ckpt, a.long_bits);
    else
      count_rows(CountTable{a.table, held}, k, a.count, task, turn, a.status, held + kCountWords, &s_longs);
  }
  if (!kEmit) {
    __syncthreads();
    count_long_rows(a, held + kCountWords, min(s_longs, kLongList));
  }
}

// The long rows into the stream.  They are the first ones of a matrix's first slices: four small
// workgroups share a slice's, on different dies (on one the rows' entries, which share cache
// lines, wait for each other in its L2: 127 us instead of 79).
constexpr int kLongThreads = 256, kLongShares = 4;
constexpr int kLongWaves = kLongShares * kLongThreads / 64;   // of a slice
__global__ __launch_bounds__(kLongThreads) void emit_long_rows_kernel(WalkArgs a) {
  if (*a.found) return;
  const int lane = threadIdx.x & 63;
  const int64_t all = a.k[0].tasks + (a.kinds == 2 ? a.k[1].tasks : 0);
  for (int64_t t = blockIdx.x; t < kLongShares * all; t += gridDim.x) {
    const int64_t task = t / kLongShares;
    const int wave = static_cast<int>(t % kLongShares) * (kLongThreads / 64) + static_cast<int>(threadIdx.x >> 6);
    const bool second = task >= a.k[0].tasks;
    const WalkKind &k = a.k[second ? 1 : 0];
    const int64_t slice = second ? task - a.k[0].tasks : task;
    const uint32_t bit = static_cast<uint32_t>(k.first_slice + slice) % kLongBits;
    if (!((a.long_bits[bit / 32] >> (bit % 32)) & 1u)) continue;
    const int ridx = k.row_idx[slice * 64 + lane];
    int n = 0;
    bool is_long = false;
    const uint16_t *codes = nullptr;
    if (ridx != 0xffff)
      codes = row_codes(k.source, static_cast<int>(slice / k.slices), ridx, k.height, k.width, k.long_from, n, is_long);
    const SliceOut s = slice_out(k, slice, a.stream, a.ckpt);
    int turn_of = 0;   // the wavefronts take the long rows in turn
    for (unsigned long long longs = __ballot(is_long); longs; longs &= longs - 1) {
      if (turn_of++ % kLongWaves != wave) continue;
      const int who = __ffsll(longs) - 1;
      // its chunks are put together in memory: zeros first, which the padding is too
      for (uint32_t c = 512u * lane; c < s.end; c += 512u * 64)
        *reinterpret_cast<uint2 *>(s.chunks + 8 * who + c) = make_uint2(0u, 0u);
      sub1::drain_stores();
      int carry_entries = 0;
      walk_long_row(a.table, codes_of_lane(codes, who), __builtin_amdgcn_readlane(n, who),
                    [&](const uint32_t (&w)[kGroupOfCodes], int &from, int &at, bool live, bool ends) {
        // the steps of every codeword (7 bits each), how many (2 bits), and over them how many long
        // ones come first (up to 256)
        uint32_t steps[kGroupOfCodes];
        int entries = 0, reached = at;
#pragma unroll
        for (int j = 0; j < kGroupOfCodes; j++) {
          const CodeSteps c(w[j], k.width, from, at);
          steps[j] = c.packed | static_cast<uint32_t>(c.nonzeros) << (3 * kFieldBits) |
                     static_cast<uint32_t>(c.more) << (3 * kFieldBits + 2);
          entries += c.nonzeros + c.more;
        }
        const int behind = carry_entries + sub1::wave_prefix_sum(entries), first = behind - entries;
        ChunkSink<true> sink{s.chunks, s.ckpt, s.end, 512u * (first / kFields) + 8u * who, kFieldBits * (first % kFields)};
#pragma unroll
        for (int j = 0; j < kGroupOfCodes; j++) {
          int more = steps[j] >> (3 * kFieldBits + 2);
          if (__builtin_expect(more != 0, 0)) {
            int zero = farthest_zero(reached);
#pragma unroll 1
            for (; more > 0; more--) {
              sink.add(zero - reached, 1, zero);
              reached = zero;
              zero += kZeroStep;
            }
          }
          const uint32_t three = steps[j] & ((1u << (3 * kFieldBits)) - 1);
          reached += static_cast<int>((three & 127u) + ((three >> kFieldBits) & 127u) + (three >> (2 * kFieldBits)));
          sink.add(three, (steps[j] >> (3 * kFieldBits)) & 3u, reached);
        }
        if (live && ends && behind < s.len && (at >> 1) % kZeroPeriod != 0) {
          const int zero = next_zero(at);
          sink.add(zero - at, 1, zero);
          at = zero;
        }
        if (sink.lo | sink.hi) sink.put();
        if (live && ends) {   // where the groups of chunks that hold nothing but padding begin
          const uint32_t filled = (sink.at & ~511u) + (sink.bits ? 512u : 0u);
          for (uint32_t c = (filled + 4095u) >> 12; c << 12 < s.end; c++)
            *reinterpret_cast<uint16_t *>(s.ckpt + c * 128 + 2 * who) = static_cast<uint16_t>(at);
        }
        carry_entries = __builtin_amdgcn_readlane(behind, 63);
      });
    }
  }
}

// One workgroup per matrix: order the rows by entry count, longest first, rows
// of equal count by row number, and describe the 64-row slices.  A counting sort,
// the same order on every run: the rows are cut into parts, one per wavefront, each
// with a histogram of its own over the counts between the smallest and the largest;
// prefix sums over the bins, and within a bin over the parts, say where each
// part's rows of a count begin; then every wavefront places its rows 64 at a time,
// each after the places that the ones before it have taken.  A row's rank among
// the equal counts of its 64 is found with the histogram (a ballot per bit of the
// count).  Where the counts spread so far that a histogram for every wavefront does not
// fit, there are fewer parts, down to one.
// 128 base experts, wi and wo (3072 and 768 rows): 13 us.  One wavefront that placed
// all rows, two dependent LDS accesses per 64, took 23; one thread that walked the
// histogram and took the rows one by one 750 for wi alone.
// Dynamic LDS: the bins, the entry count of the first row of up to 1024 slices
// (65534 rows), a few words per wavefront, and a byte per row.
constexpr int kOrderThreads = 1024;
constexpr int kOrderWaves = kOrderThreads / 64;
constexpr int kOrderBins = kMaxRowEntries + 1;
constexpr int kOrderAhead = 8;   // runs of 64 rows whose counts are asked for together
constexpr size_t order_rows_lds(int height) {
  return (kOrderBins + 1024 + 2 * kOrderWaves) * sizeof(int) + static_cast<size_t>(height + 63) / 64 * 64;
}
// Both kinds of a layer in one launch, a matrix of either to a workgroup: 128 base
// experts then take as long as wi alone (24 us, 34 one kind after the other).
struct OrderKind {
  KindSource source;
  const uint16_t *row_len;
  uint16_t *row_idx;
  uint32_t *minmax;
  uint16_t *slice_len;
  int32_t *counts;
  int height, slices;
};
struct OrderArgs {
  OrderKind k[2];
  const int32_t *found;
  int32_t *status;
};

__global__ __launch_bounds__(kOrderThreads) void order_rows_kernel(OrderArgs a) {
  if (*a.found) return;
  const int kind = blockIdx.y;
  const OrderKind &k = a.k[kind];
  const KindSource &ks = k.source;
  const uint16_t *__restrict__ row_len_all = k.row_len;
  uint16_t *__restrict__ row_idx = k.row_idx;
  uint32_t *__restrict__ minmax_sorted = k.minmax;
  uint16_t *__restrict__ slice_len = k.slice_len;
  int32_t *__restrict__ counts = k.counts;
  int32_t *__restrict__ status = a.status;
  const int height = k.height, slices = k.slices;
  extern __shared__ int order_lds[];
  int *bins = order_lds;
  int *first_len = bins + kOrderBins;
  int *wave_a = first_len + 1024, *wave_b = wave_a + kOrderWaves;
  uint8_t *rank = reinterpret_cast<uint8_t *>(wave_b + kOrderWaves);
  const int e = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint16_t *rl = row_len_all + static_cast<int64_t>(e) * height;
  const uint32_t *mm = ks.minmax_of ? ks.minmax_of[e] : ks.minmax + static_cast<int64_t>(e) * height;
  const int64_t lane0 = static_cast<int64_t>(e) * slices * 64;

  int low = kMaxRowEntries, high = 0;
  for (int r = tid; r < height; r += kOrderThreads) {
    low = min(low, static_cast<int>(rl[r]));
    high = max(high, static_cast<int>(rl[r]));
  }
  for (int m = 1; m < 64; m <<= 1) {
    low = min(low, __shfl_xor(low, m, 64));
    high = max(high, __shfl_xor(high, m, 64));
  }
  if (lane == 0) {
    wave_a[wave] = low;
    wave_b[wave] = high;
  }
  __syncthreads();
  for (int w = 0; w < kOrderWaves; w++) {
    low = min(low, wave_a[w]);
    high = max(high, wave_b[w]);
  }
  const int range = high - low + 1;   // bin b: the rows of high - b entries
  int parts = kOrderWaves;            // bins[range * part + b]: part's rows in bin b, then where the next one goes
  while (parts > 1 && parts * range > kOrderBins) parts >>= 1;
  const int groups = (height + 63) / 64, part_groups = (groups + parts - 1) / parts;
  const int from = 64 * part_groups * wave, to = min(from + 64 * part_groups, height);   // this wavefront's rows
  for (int i = tid; i < parts * range; i += kOrderThreads) bins[i] = 0;
  __syncthreads();
  int *mine = bins + range * wave;
  if (wave < parts)
    for (int r0 = from; r0 < to; r0 += 64 * kOrderAhead) {
      int len[kOrderAhead];
#pragma unroll
      for (int u = 0; u < kOrderAhead; u++) {
        const int r = r0 + 64 * u + lane;
        len[u] = r < to ? rl[r] : 0;
      }
#pragma unroll
      for (int u = 0; u < kOrderAhead; u++) {
        if (r0 + 64 * u >= to) break;
        const int r = r0 + 64 * u + lane;
        const int bin = r < to ? high - len[u] : 0;
        unsigned long long same = __ballot(r < to);
        for (int bit = 1; bit < range; bit <<= 1) {
          const unsigned long long with = __ballot((bin & bit) != 0);
          same &= (bin & bit) ? with : ~with;
        }
        if (r < to) {
          const int before = __popcll(same & ((1ull << lane) - 1));
          const bool last = lane == 63 - __clzll(same);
          rank[r] = static_cast<uint8_t>(before | (last ? 64 : 0));
          if (last) atomicAdd(&mine[bin], before + 1);
        }
      }
    }
  __syncthreads();
  int carry = 0;
  for (int b0 = 0; b0 < range; b0 += kOrderThreads) {   // every bin's first place, and every part's in it
    const int b = b0 + tid;
    int n = 0;
    if (b < range)
      for (int q = 0; q < parts; q++) n += bins[range * q + b];
    int upto = n;
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(upto, d, 64);
      if (lane >= d) upto += v;
    }
    if (lane == 63) wave_a[wave] = upto;
    __syncthreads();
    int before = carry;
    for (int w = 0; w < kOrderWaves; w++) {
      if (w < wave) before += wave_a[w];
      carry += wave_a[w];
    }
    int place = before + upto - n;
    if (b < range)
      for (int q = 0; q < parts; q++) {
        const int rows = bins[range * q + b];
        bins[range * q + b] = place;
        place += rows;
      }
    __syncthreads();
  }
  if (wave < parts) {
    volatile int *place = mine;   // read and written by this wavefront alone, in program order
    for (int r0 = from; r0 < to; r0 += 64 * kOrderAhead) {
      int len[kOrderAhead];
      uint32_t values[kOrderAhead];
#pragma unroll
      for (int u = 0; u < kOrderAhead; u++) {
        const int r = r0 + 64 * u + lane;
        len[u] = r < to ? rl[r] : 0;
        values[u] = r < to ? mm[r] : 0u;
      }
#pragma unroll
      for (int u = 0; u < kOrderAhead; u++) {
        const int r = r0 + 64 * u + lane;
        if (r < to) {
          const int before = rank[r];
          const int p = place[high - len[u]] + (before & 63);
          if (before & 64) place[high - len[u]] = p + 1;
          row_idx[lane0 + p] = static_cast<uint16_t>(r);
          minmax_sorted[lane0 + p] = values[u];
          if ((p & 63) == 0) first_len[p >> 6] = len[u];
        }
      }
    }
  }
  for (int p = height + tid; p < slices * 64; p += kOrderThreads) {
    row_idx[lane0 + p] = 0xffffu;
    minmax_sorted[lane0 + p] = 0u;
  }
  __syncthreads();
  for (int s = tid; s < slices; s += kOrderThreads) {
    const int len = max(first_len[s], 1);   // a slice is as long as its first row, and at least one entry
    const int64_t g = static_cast<int64_t>(e) * slices + s;
    slice_len[g] = static_cast<uint16_t>(len);
    counts[g + 1] = chunks_of(len);
    atomicMax(&status[1 + kind], chunks_of(len));
  }
}

// What the prepare passes take on trust is looked at on the GPU first: whether
// dec is the fixed dictionary's table, and the tables of device pointers entry by
// entry.  A workgroup of 256 compares 4 KB of dec; the workgroups then share the
// pointers.  *found: bit 0 = dec differs, bit 1 = a pointer is NULL or misaligned.
struct PointerTables {
  const void *const *table[6];
  uint32_t align[6];
  int n, count;
};
constexpr int kCheckBlocks = SUB1_DEC_WORDS / 4 / 256;
__global__ __launch_bounds__(256) void check_source_kernel(const int32_t *__restrict__ dec,
                                                           const int32_t *__restrict__ fixed,
                                                           PointerTables pt, int32_t *found) {
  const int at = blockIdx.x * 256 + threadIdx.x;
  int32_t a[4], b[4];
  __builtin_memcpy(a, dec + 4 * at, 16);
  __builtin_memcpy(b, fixed + 4 * at, 16);
  int bad = ((a[0] ^ b[0]) | (a[1] ^ b[1]) | (a[2] ^ b[2]) | (a[3] ^ b[3])) ? 1 : 0;
  for (int t = 0; t < pt.n; t++)
    for (int i = at; i < pt.count; i += kCheckBlocks * 256) {
      const uintptr_t v = reinterpret_cast<uintptr_t>(pt.table[t][i]);
      if (v == 0 || (v & (pt.align[t] - 1)) != 0) bad |= 2;
    }
  if (bad) atomicOr(found, bad);
}

// ... and what the host waits for: the total, then the four status words.
__global__ __launch_bounds__(sub1::kScanThreads) void scan_counts_kernel(int32_t *v, int n, const int32_t *status,
                                                                        sub1::Answer answer) {
  const bool found = status[3] != 0;
  if (!found) sub1::scan_in_place(v, n);
  __syncthreads();
  if (threadIdx.x == 0) sub1::tell(answer, 0, found ? 0 : v[n]);
  if (threadIdx.x < 4) sub1::tell(answer, 1 + threadIdx.x, status[threadIdx.x]);
}

// The symbols of one prepared matrix back out of the stream: out[row, column]
// = 1 or 2 at every entry that stands on an activation; out is zero before.
__global__ __launch_bounds__(256) void decode_entries_kernel(
    const uint2 *__restrict__ stream, const uint32_t *__restrict__ slice_base,
    const uint16_t *__restrict__ slice_len, const uint16_t *__restrict__ row_idx,
    uint8_t *__restrict__ out, int64_t first, int slices, int width) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= slices * 64) return;
  const int64_t sl = first + (t >> 6);
  const int ridx = row_idx[sl * 64 + (t & 63)];
  if (ridx == 0xffff) return;
  const uint2 *p = stream + static_cast<int64_t>(slice_base[sl]) * 64 + (t & 63);
  const int len = slice_len[sl];
  const int nch = chunks_of(len);
  int j = 0;
  for (int c = 0; c < nch; c++) {
    const uint2 cw = p[c * 64];
    const unsigned long long w = (static_cast<unsigned long long>(cw.y) << 32) | cw.x;
    for (int q = 0; q < kFields && c * kFields + q < len; q++) {
      j += static_cast<int>(w >> (kFieldBits * q)) & kMaxStep;
      const int pc = j >> 1;   // physical column
      const int col = pc - 1 - pc / kZeroPeriod;
      if (pc % kZeroPeriod != 0 && col < width)
        out[static_cast<int64_t>(ridx) * width + col] = static_cast<uint8_t>((j & 1) + 1);
    }
  }
}

__global__ void fill_bytes_kernel(uint8_t *p, int64_t n, uint8_t v) {
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

__global__ void zero_words_kernel(int32_t *p, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ------------------------------------------------------------- main kernel --

struct KindArgs {
  const uint32_t *slice_base;
  const uint16_t *slice_len;
  const uint16_t *row_idx;
  const uint32_t *minmax;
  int slices, height, width, parts;
  int split;            // wavefronts that share one slice (1 = a slice per wavefront)
  int groups_max;       // most groups of chunks in a slice of this kind
  int64_t first_slice;  // global index of the kind's first slice (checkpoint addressing)
  int tail_split;       // fused kernel: wavefronts per slice of a short last pass (0: none)
};

struct PreparedArgs {
  const uint2 *stream;        // the interleaved entries
  const uint16_t *ckpt;       // position checkpoints, behind the stream
  KindArgs k[2];
  const int32_t *token_expert;   // NULL: every token uses matrix 0
  const int32_t *order;          // fused kernel, tokens grouped by expert: token ids by expert,
  const int2 *groups;            // and tiles (expert or -1, first index into order * 8 + tokens)
  const uint16_t *x;
  uint16_t *y;
  uint16_t *h;                   // kinds == 2 only
  int32_t *ctrl;                 // NULL: no dependencies between tiles, static tile order
  int64_t ldx, ldy;              // element strides between tokens of x and y
  int kinds;                     // 2: y = wo(relu(wi x));  1: y += W x
  int fresh;                     // kinds == 1: y counts as zeros and is not read
  int tokens, experts;
  int xdwords;                   // LDS dwords reserved for the activations
  int hdwords;                   // fused kernel: LDS dwords of h (wo's activations)
  int tail_room;                 // persistent kernel: partial sums (groups x 64 lanes) LDS has room for
  int wi_expect;                 // workgroups of a token's wi a wait expects (k[0].parts outside tests)
  int by_ticket;                 // shared-token kernel: a workgroup's place comes from the ticket
  unsigned long long *tagged;    // shared-token kernel: h is handed over by tag (NULL: by count)
  int lane_parts;                // one-token kernel with wo in workgroups of its own: these share a slice by lanes
  int64_t wait_ticks;            // longest wait between workgroups, ticks of wall_clock64
  int32_t *sticky;               // fault flags in pinned host memory
};

// Activations in LDS: two dwords per physical column, A = (x, 0) and B = (0, x)
// as bf16 pairs, zeros in the zero columns (see "Positions" above).  Rounded up
// to whole 16 bytes (what follows in LDS stays aligned).
__host__ __device__ constexpr int activation_dwords(int width) {
  return (2 * physical_columns(width) + 3) / 4 * 4;
}

// Every load of a thread is in flight before its first LDS store, so a tile
// pays one memory round trip for its activations, not one per pass.  In two
// steps, so that a kernel can ask for the activations long before it needs
// them: stage_request issues a thread's first four loads (all of them up to a
// width of eight times the workgroup), stage_finish stores them and does the
// rest.
struct StagedPairs {
  uint32_t v[4];
};

__device__ __forceinline__ uint32_t load_pair(const uint16_t *x, int m, int width, bool aligned) {
  uint32_t v = 0u;
  if (aligned && 2 * m + 1 < width) {
    v = *reinterpret_cast<const uint32_t *>(x + 2 * m);
  } else {
    if (2 * m < width) v = x[2 * m];
    if (2 * m + 1 < width) v |= static_cast<uint32_t>(x[2 * m + 1]) << 16;
  }
  return v;
}

__device__ __forceinline__ void store_pair(uint32_t *xa, int m, int width, uint32_t v) {
  if (2 * m >= width) return;
  // columns 2m and 2m+1 are neighbours among the physical columns too
  uint32_t *p = xa + 2 * physical_column(2 * m);
  p[0] = v & 0xffffu;
  p[1] = v << 16;
  if (2 * m + 1 < width) {
    p[2] = v >> 16;
    p[3] = v & 0xffff0000u;
  }
}

__device__ __forceinline__ StagedPairs stage_request(const uint16_t *x, int width) {
  const bool aligned = (reinterpret_cast<uintptr_t>(x) & 3u) == 0;
  StagedPairs s;
#pragma unroll
  for (int u = 0; u < 4; u++)
    s.v[u] = load_pair(x, threadIdx.x + u * blockDim.x, width, aligned);
  return s;
}

__device__ __forceinline__ void stage_finish(uint32_t *xa, const uint16_t *x, int width,
                                             const StagedPairs &s) {
  const int npairs = (width + 1) / 2;
  const int step = blockDim.x;
  const bool aligned = (reinterpret_cast<uintptr_t>(x) & 3u) == 0;
  for (int z = threadIdx.x * kZeroPeriod; z < physical_columns(width); z += step * kZeroPeriod) {
    xa[2 * z] = 0u;
    xa[2 * z + 1] = 0u;
  }
#pragma unroll
  for (int u = 0; u < 4; u++) store_pair(xa, threadIdx.x + u * step, width, s.v[u]);
  for (int m0 = threadIdx.x + 4 * step; m0 < npairs; m0 += 4 * step) {
    uint32_t v[4];
#pragma unroll
    for (int u = 0; u < 4; u++) v[u] = load_pair(x, m0 + u * step, width, aligned);
#pragma unroll
    for (int u = 0; u < 4; u++) store_pair(xa, m0 + u * step, width, v[u]);
  }
}

__device__ __forceinline__ void stage_activations(uint32_t *xa, const uint16_t *x, int width) {
  const StagedPairs s = stage_request(x, width);
  stage_finish(xa, x, width, s);
}

typedef __attribute__((address_space(3))) const uint32_t lds_word;

// The LDS byte address of a dword of the activation array.
__device__ __forceinline__ uint32_t lds_address(const uint32_t *xa) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_word *)xa));
}

// The nine entries of a chunk: each moves the row's LDS address `at` (bytes)
// and adds the bf16 pair found there, times the row's (min, max), onto acc.
// v_bfe_u32 and v_lshl_add_u32 are written out because the compiler expands the
// same arithmetic into three instructions per entry instead of two.
__device__ __forceinline__ void add_chunk(uint2 cw, uint32_t &at, float &acc, bf16x2 minmax) {
  const uint32_t mid = __builtin_amdgcn_alignbit(cw.y, cw.x, 28);   // bits 28..59: entries 4..7
  uint32_t f[kFields];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    asm("v_bfe_u32 %0, %1, %2, 7" : "=v"(f[q]) : "v"(cw.x), "n"(kFieldBits * q));
    asm("v_bfe_u32 %0, %1, %2, 7" : "=v"(f[4 + q]) : "v"(mid), "n"(kFieldBits * q));
  }
  asm("v_bfe_u32 %0, %1, 24, 7" : "=v"(f[8]) : "v"(cw.y));           // bits 56..62
#pragma unroll
  for (int q = 0; q < kFields; q++) {
    asm("v_lshl_add_u32 %0, %1, 2, %0" : "+v"(at) : "v"(f[q]));
    const bf16x2 v = __builtin_bit_cast(bf16x2, *(lds_word *)static_cast<uintptr_t>(at));
    acc = __builtin_amdgcn_fdot2_f32_bf16(v, minmax, acc, false);
  }
}

// The same sums in the same order with all nine LDS reads of the chunk asked
// for before the first is used: where a compute unit has few wavefronts at work
// (a handful of tokens), a walk is a chain of LDS round trips, and this makes it
// one per chunk instead of one per entry.  (With sixteen wavefronts at it the
// LDS is busy either way, and the registers are better spent elsewhere.)
__device__ __forceinline__ void add_chunk_ahead(uint2 cw, uint32_t &at, float &acc,
                                                bf16x2 minmax) {
  const uint32_t mid = __builtin_amdgcn_alignbit(cw.y, cw.x, 28);
  uint32_t f[kFields], where[kFields];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    asm("v_bfe_u32 %0, %1, %2, 7" : "=v"(f[q]) : "v"(cw.x), "n"(kFieldBits * q));
    asm("v_bfe_u32 %0, %1, %2, 7" : "=v"(f[4 + q]) : "v"(mid), "n"(kFieldBits * q));
  }
  asm("v_bfe_u32 %0, %1, 24, 7" : "=v"(f[8]) : "v"(cw.y));
#pragma unroll
  for (int q = 0; q < kFields; q++) {
    asm("v_lshl_add_u32 %0, %1, 2, %2" : "=v"(where[q]) : "v"(f[q]), "v"(q ? where[q - 1] : at));
  }
  at = where[kFields - 1];
  bf16x2 v[kFields];
#pragma unroll
  for (int q = 0; q < kFields; q++)
    v[q] = __builtin_bit_cast(bf16x2, *(lds_word *)static_cast<uintptr_t>(where[q]));
#pragma unroll
  for (int q = 0; q < kFields; q++) acc = __builtin_amdgcn_fdot2_f32_bf16(v[q], minmax, acc, false);
}

// A chunk of the stream.  kOnce: the launch reads more of the stream than the
// caches hold and every chunk exactly once, and the load says so (a
// non-temporal load; measured 2% faster on the Switch-c-2048 sweep, 2% slower
// where the same few matrices are read over and over from the caches).
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
template <bool kOnce>
__device__ __forceinline__ uint2 load_chunk(const uint2 *p) {
  if (kOnce) {
    const u32x2 v = __builtin_nontemporal_load(reinterpret_cast<const u32x2 *>(p));
    return make_uint2(v.x, v.y);
  }
  return *p;
}

// The first n entries of a chunk, n the same in every lane: the last chunk of a
// slice, which is walked only as far as the slice's longest row goes.
__device__ __forceinline__ void add_entries(uint2 cw, int n, uint32_t &at, float &acc,
                                            bf16x2 minmax) {
  if (n == kFields) {
    add_chunk(cw, at, acc, minmax);
    return;
  }
  unsigned long long w = (static_cast<unsigned long long>(cw.y) << 32) | cw.x;
  for (int q = 0; q < n; q++) {
    at += (static_cast<uint32_t>(w) & static_cast<uint32_t>(kMaxStep)) << 2;
    w >>= kFieldBits;
    const bf16x2 v = __builtin_bit_cast(bf16x2, *(lds_word *)static_cast<uintptr_t>(at));
    acc = __builtin_amdgcn_fdot2_f32_bf16(v, minmax, acc, false);
  }
}

// The same with the reads asked for together (see add_chunk_ahead).
__device__ __forceinline__ void add_entries_ahead(uint2 cw, int n, uint32_t &at, float &acc,
                                                  bf16x2 minmax) {
  if (n == kFields) {
    add_chunk_ahead(cw, at, acc, minmax);
    return;
  }
  unsigned long long w = (static_cast<unsigned long long>(cw.y) << 32) | cw.x;
  uint32_t where[kFields - 1];
  bf16x2 v[kFields - 1];
#pragma unroll
  for (int q = 0; q < kFields - 1; q++) {
    where[q] = (q ? where[q - 1] : at) + ((static_cast<uint32_t>(w) & static_cast<uint32_t>(kMaxStep)) << 2);
    w >>= kFieldBits;
  }
#pragma unroll
  for (int q = 0; q < kFields - 1; q++)
    if (q < n) v[q] = __builtin_bit_cast(bf16x2, *(lds_word *)static_cast<uintptr_t>(where[q]));
#pragma unroll
  for (int q = 0; q < kFields - 1; q++)
    if (q < n) acc = __builtin_amdgcn_fdot2_f32_bf16(v[q], minmax, acc, false);
  if (n > 0) {
    uint32_t last = where[0];
#pragma unroll
    for (int q = 1; q < kFields - 1; q++)
      if (q < n) last = where[q];
    at = last;
  }
}

// This lane's chunk 0 of the slice that starts at chunk `base` of the stream.
__device__ __forceinline__ const uint2 *chunk_pointer(const uint2 *stream, uint32_t base) {
  return stream + static_cast<int64_t>(base) * 64 + (threadIdx.x & 63);
}

// What a lane needs to walk its row of one slice; load_slice issues the loads
// of the first chunks, so calling it for the NEXT slice before walking the
// current one hides their latency.
template <int R, bool kOnce = false>
struct Walk {
  uint32_t base;     // the slice's first chunk, in chunks; the same in every lane,
  int nch;           // like the chunk count (where this wavefront stops),
  int last;          // the entries of chunk nch - 1 that are walked (9 unless it ends the slice)
  int c0;            // and the chunk this wavefront starts at (0 unless it shares the slice)
  int j0;            // this lane's position at chunk c0
  int ridx;
  uint32_t minmax;
  uint2 ring[R];
};
typedef Walk<kRing> SliceWalk;

// g_lo, g_hi: the run of chunk groups to walk, for a wavefront that shares the
// slice with others (it then starts from the position checkpoint of group g_lo).
constexpr int kAllGroups = 1 << 20;
// (len, base: the slice's description, where the caller has read it already.)
template <int R = kRing, bool kOnce = false>
__device__ __forceinline__ Walk<R, kOnce> load_slice_described(const PreparedArgs &a,
                                                               const KindArgs &k, int64_t sl,
                                                               int len, uint32_t base, int g_lo,
                                                               int g_hi) {
  const int lane = threadIdx.x & 63;
  Walk<R, kOnce> w;
  const int nch_all = chunks_of(len);
  w.nch = min(g_hi * kGroupChunks, nch_all);
  w.last = w.nch == nch_all ? last_entries_of(len) : kFields;
  w.c0 = g_lo * kGroupChunks;
  w.ridx = k.row_idx[sl * 64 + lane];
  w.minmax = k.minmax[sl * 64 + lane];
  w.base = base;
  w.j0 = 0;
  if (g_lo)
    w.j0 = a.ckpt[(checkpoint_entry(w.base, k.first_slice + sl) + g_lo) * 64 + lane];
  const uint2 *p = chunk_pointer(a.stream, w.base);
#pragma unroll
  for (int i = 0; i < R; i++) w.ring[i] = load_chunk<kOnce>(p + min(w.c0 + i, w.nch - 1) * 64);
  return w;
}

template <int R = kRing, bool kOnce = false>
__device__ __forceinline__ Walk<R, kOnce> load_slice(const PreparedArgs &a, const KindArgs &k,
                                                     int64_t sl, int g_lo = 0,
                                                     int g_hi = kAllGroups) {
  const int len_word = k.slice_len[sl];
  const uint32_t base_word = k.slice_base[sl];
  return load_slice_described<R, kOnce>(a, k, sl, __builtin_amdgcn_readfirstlane(len_word),
                                        __builtin_amdgcn_readfirstlane(base_word), g_lo, g_hi);
}

// R chunks (the depth of the walk's ring) starting at chunk c added onto the
// partial sum; all of them whole (c + R <= nch - 1), each replaced in the ring
// by the chunk R further on.
// kChecked: the walk's last chunks, fewer than R whole ones and then chunk
// nch - 1 with its `last` entries; nothing is requested any more.
// kEarly: the next R chunks are asked for before these are begun.  (Left to the compiler the last of them may be
// asked for just before the loop waits for them all, which shows where a wavefront walks alone at the end.)
constexpr int kAllButLoads = 0x38f;   // what may be moved over a sched_barrier: ALU and LDS instructions
template <bool kChecked, bool kEarly = false, int R, bool kOnce>
__device__ __forceinline__ void run_chunks(Walk<R, kOnce> &w, const uint2 *p, int c, uint32_t &at,
                                           float &part, bf16x2 minmax) {
  const int nch = w.nch;
  // the deep ring is the one of the walks built for latency
  constexpr bool kAhead = R == kSplitRing;
  if (kEarly && !kChecked) {
    uint2 cw[R];
#pragma unroll
    for (int i = 0; i < R; i++) cw[i] = w.ring[i];
#pragma unroll
    for (int i = 0; i < R; i++) w.ring[i] = load_chunk<kOnce>(p + min(c + i + R, nch - 1) * 64);
    __builtin_amdgcn_sched_barrier(kAllButLoads);
#pragma unroll
    for (int i = 0; i < R; i++) {
      if (kAhead) add_chunk_ahead(cw[i], at, part, minmax);
      else add_chunk(cw[i], at, part, minmax);
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < R; i++) {
    if (!kChecked) {
      const uint2 cw = w.ring[i];
      // unconditional, clamped to the last chunk: the load can target the ring
      // register itself and the loop needs no wait for it
      w.ring[i] = load_chunk<kOnce>(p + min(c + i + R, nch - 1) * 64);
      if (kAhead) add_chunk_ahead(cw, at, part, minmax);
      else add_chunk(cw, at, part, minmax);
    } else if (c + i < nch - 1) {
      if (kAhead) add_chunk_ahead(w.ring[i], at, part, minmax);
      else add_chunk(w.ring[i], at, part, minmax);
    } else if (c + i == nch - 1) {
      if (kAhead) add_entries_ahead(w.ring[i], w.last, at, part, minmax);
      else add_entries(w.ring[i], w.last, at, part, minmax);
    }
  }
}

// The hardware serves the oldest wavefront of a SIMD first; left alone, the
// wavefronts of a workgroup drift apart and the last ones finish a phase on an
// idle compute unit.  A wavefront therefore lowers its priority as it gets
// through its share of the phase, in steps that get finer towards the end
// (`done` of `total`: below 5/8 priority 3, below 13/16 2, below 15/16 1, then
// 0), so that the laggards catch up and all finish together.
__device__ __forceinline__ void progress_priority(int done, int total) {
  const int p = done * 16 / total;
  if (p < 10) {
    __builtin_amdgcn_s_setprio(3);
  } else if (p < 13) {
    __builtin_amdgcn_s_setprio(2);
  } else if (p < 15) {
    __builtin_amdgcn_s_setprio(1);
  } else {
    __builtin_amdgcn_s_setprio(0);
  }
}

// The sum of this lane's row, in the library's canonical order: groups of 72
// entries (kGroupChunks chunks), a partial sum per group from zero, the partial
// sums added first group first.
// With `part` the wavefront shares its slice: it leaves each group's partial
// sum at part[group * 64 + lane] for the wavefront that adds them up.
// pass / passes (passes != 0): this slice is the wavefront's pass-th of `passes`
// about equal ones in the current phase; sets the priority by progress.
template <bool kEarly = false, int R, bool kOnce>
__device__ __forceinline__ float run_slice(Walk<R, kOnce> &w, const uint2 *stream,
                                           const uint32_t *xa, float *part = nullptr,
                                           int pass = 0, int passes = 0) {
  static_assert(kGroupChunks % R == 0, "a group of chunks is a whole number of ring turns");
  // a walk that went through `cur = nxt` may sit in vector registers: put what
  // is the same in all lanes back into scalar ones, for scalar loop control
  // and scalar address arithmetic
  w.nch = __builtin_amdgcn_readfirstlane(w.nch);
  w.last = __builtin_amdgcn_readfirstlane(w.last);
  const uint2 *p = chunk_pointer(stream, __builtin_amdgcn_readfirstlane(w.base));
  const int lane = threadIdx.x & 63;
  const bf16x2 minmax = __builtin_bit_cast(bf16x2, w.minmax);
  float sum = 0.f, partial = 0.f;
  uint32_t at = lds_address(xa) + 4u * static_cast<uint32_t>(w.j0);
  int c = __builtin_amdgcn_readfirstlane(w.c0);
  if (passes) progress_priority(pass, passes);
  auto group_done = [&]() {
    if (passes) progress_priority(pass * w.nch + c + R, passes * w.nch);
    if (part) {
      part[((c + R) / kGroupChunks - 1) * 64 + lane] = partial;
    } else {
      sum += partial;
    }
    partial = 0.f;
  };
  for (; c + R <= w.nch - 1; c += R) {
    run_chunks<false, kEarly>(w, p, c, at, partial, minmax);
    if ((c + R) % kGroupChunks == 0) group_done();
  }
  // fewer than R whole chunks are left, and the last chunk
  run_chunks<true>(w, p, c, at, partial, minmax);
  if ((c + R) % kGroupChunks == 0) group_done();
  c += R;
  if (part) {
    // the slice's last group, unless the loop has just closed it
    if (c % kGroupChunks) part[(c / kGroupChunks) * 64 + lane] = partial;
  } else {
    sum += partial;   // the last, partial group (+0 if it was just folded)
  }
  return sum;
}

// The slice a wavefront takes in its pass-th turn through `count` slices that
// are ordered longest first: back and forth, so that every wavefront gets
// about the same number of chunks.  >= count: no slice left in this pass.
__device__ __forceinline__ int slice_of_pass(int pass, int wave, int waves, int count) {
  const int s = pass * waves + ((pass & 1) ? waves - 1 - wave : wave);
  return s < count ? s : count;
}

// How a row's result leaves the kernel.
// kFresh: kAccumulate onto a y that counts as zeros and is not read.
enum OutMode { kStoreRelu = 0, kStore = 1, kAccumulate = 2, kFresh = 3 };

__device__ __forceinline__ void write_row(uint16_t *dst, int ridx, float res, int mode) {
  if (ridx == 0xffff) return;   // padding lane
  uint16_t out = f32_to_bf16(res);
  if (mode == kStoreRelu) {
    if (out & 0x8000u) out = 0;   // relu between the projections, on the bf16 value
    // h in the workspace, read by other workgroups: written through to where
    // every compute unit sees it (see publish_h)
    __hip_atomic_store(&dst[ridx], out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  } else if (mode == kAccumulate) {
    // reference sub1_cuda_kernel.cu:200: y[row] += bf16(res), the sum in bf16
    out = f32_to_bf16(bf16_to_f32(dst[ridx]) + bf16_to_f32(out));
  } else if (mode == kFresh) {
    out = f32_to_bf16(0.f + bf16_to_f32(out));   // (0 + -0 is 0)
  }
  dst[ridx] = out;
}

// ----------------------------------------------------- four tokens per walk --
//
// Where several tokens go through the same matrix, the stream is walked once
// for four of them.  The activation array then holds, per physical column, the
// two dwords (x0, x1) and (x2, x3) of tokens 0..3 as bf16 pairs (zeros in the
// zero columns), and an entry costs one address, one 8-byte LDS read and four
// v_dot2c_f32_bf16: the weight, picked by the position's low bit, sits in one
// half of the second operand so that each instruction adds one token's term.
// (Two 4-byte reads from separate arrays measured 10% slower in this kernel.)
// Every token's sum is taken in the same order as when it is walked alone, so
// the results are the same to the bit (for finite activations: a token's
// infinity or NaN also spoils the sum of the token it shares a dword with).
constexpr int kGroupTokens = 4;

struct GroupSums {
  float v[kGroupTokens];
};

struct GroupRows {
  const uint16_t *row[kGroupTokens];   // NULL: no token in this place
};

__device__ __forceinline__ void stage_group(uint32_t *xa, const GroupRows &rows, int width) {
  const int npairs = (width + 1) / 2;
  const int step = blockDim.x;
  for (int z = threadIdx.x * kZeroPeriod; z < physical_columns(width); z += step * kZeroPeriod) {
    xa[2 * z] = 0u;
    xa[2 * z + 1] = 0u;
  }
  for (int m = threadIdx.x; m < npairs; m += step) {
    uint32_t v[kGroupTokens];
#pragma unroll
    for (int t = 0; t < kGroupTokens; t++) {
      v[t] = 0u;
      const uint16_t *row = rows.row[t];
      if (row) {
        if ((reinterpret_cast<uintptr_t>(row) & 3u) == 0 && 2 * m + 1 < width) {
          v[t] = *reinterpret_cast<const uint32_t *>(row + 2 * m);
        } else {
          v[t] = row[2 * m];
          if (2 * m + 1 < width) v[t] |= static_cast<uint32_t>(row[2 * m + 1]) << 16;
        }
      }
    }
    uint32_t *p = xa + 2 * physical_column(2 * m);
    p[0] = (v[0] & 0xffffu) | (v[1] << 16);
    p[1] = (v[2] & 0xffffu) | (v[3] << 16);
    if (2 * m + 1 < width) {
      p[2] = (v[0] >> 16) | (v[1] & 0xffff0000u);
      p[3] = (v[2] >> 16) | (v[3] & 0xffff0000u);
    }
  }
}

// The nine entries of a chunk for four tokens.  `at` is the position's LDS byte
// address as in add_chunk (the array starts on an 8-byte boundary): bit 2 is
// the symbol, the rest the physical column's two dwords.
__device__ __forceinline__ void add_chunk_group(uint2 cw, uint32_t &at, GroupSums &acc,
                                                uint32_t w_min, uint32_t w_max) {
  const uint32_t mid = __builtin_amdgcn_alignbit(cw.y, cw.x, 28);
  uint32_t f[kFields];
#pragma unroll
  for (int q = 0; q < 4; q++) {
    asm("v_bfe_u32 %0, %1, %2, 7" : "=v"(f[q]) : "v"(cw.x), "n"(kFieldBits * q));
    asm("v_bfe_u32 %0, %1, %2, 7" : "=v"(f[4 + q]) : "v"(mid), "n"(kFieldBits * q));
  }
  asm("v_bfe_u32 %0, %1, 24, 7" : "=v"(f[8]) : "v"(cw.y));
#pragma unroll
  for (int q = 0; q < kFields; q++) {
    asm("v_lshl_add_u32 %0, %1, 2, %0" : "+v"(at) : "v"(f[q]));
    const uint32_t is_max = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(at), 2, 1));
    const uint32_t k_lo = (w_max & is_max) | (w_min & ~is_max);   // (w, 0): one v_bfi_b32
    const uint32_t k_hi = k_lo << 16;                             // (0, w)
    lds_word *col = (lds_word *)static_cast<uintptr_t>(at & ~7u);
    const bf16x2 v01 = __builtin_bit_cast(bf16x2, col[0]);
    const bf16x2 v23 = __builtin_bit_cast(bf16x2, col[1]);
    acc.v[0] = __builtin_amdgcn_fdot2_f32_bf16(v01, __builtin_bit_cast(bf16x2, k_lo), acc.v[0], false);
    acc.v[1] = __builtin_amdgcn_fdot2_f32_bf16(v01, __builtin_bit_cast(bf16x2, k_hi), acc.v[1], false);
    acc.v[2] = __builtin_amdgcn_fdot2_f32_bf16(v23, __builtin_bit_cast(bf16x2, k_lo), acc.v[2], false);
    acc.v[3] = __builtin_amdgcn_fdot2_f32_bf16(v23, __builtin_bit_cast(bf16x2, k_hi), acc.v[3], false);
  }
}

// The first n entries of a chunk for four tokens (see add_entries).
__device__ __forceinline__ void add_entries_group(uint2 cw, int n, uint32_t &at, GroupSums &acc,
                                                  uint32_t w_min, uint32_t w_max) {
  if (n == kFields) {
    add_chunk_group(cw, at, acc, w_min, w_max);
    return;
  }
  unsigned long long w = (static_cast<unsigned long long>(cw.y) << 32) | cw.x;
  for (int q = 0; q < n; q++) {
    at += (static_cast<uint32_t>(w) & static_cast<uint32_t>(kMaxStep)) << 2;
    w >>= kFieldBits;
    const uint32_t is_max = static_cast<uint32_t>(__builtin_amdgcn_sbfe(static_cast<int>(at), 2, 1));
    const uint32_t k_lo = (w_max & is_max) | (w_min & ~is_max);
    const uint32_t k_hi = k_lo << 16;
    lds_word *col = (lds_word *)static_cast<uintptr_t>(at & ~7u);
    const bf16x2 v01 = __builtin_bit_cast(bf16x2, col[0]);
    const bf16x2 v23 = __builtin_bit_cast(bf16x2, col[1]);
    acc.v[0] = __builtin_amdgcn_fdot2_f32_bf16(v01, __builtin_bit_cast(bf16x2, k_lo), acc.v[0], false);
    acc.v[1] = __builtin_amdgcn_fdot2_f32_bf16(v01, __builtin_bit_cast(bf16x2, k_hi), acc.v[1], false);
    acc.v[2] = __builtin_amdgcn_fdot2_f32_bf16(v23, __builtin_bit_cast(bf16x2, k_lo), acc.v[2], false);
    acc.v[3] = __builtin_amdgcn_fdot2_f32_bf16(v23, __builtin_bit_cast(bf16x2, k_hi), acc.v[3], false);
  }
}

// run_slice for four tokens: the same groups of 72 entries per token.  With
// `part` the wavefront shares its slice and leaves each group's four partial
// sums at part[group * 64 + lane].
__device__ __forceinline__ GroupSums run_slice_group(SliceWalk &w, const uint2 *stream,
                                                     const uint32_t *xa, GroupSums *part,
                                                     int pass, int passes) {
  w.nch = __builtin_amdgcn_readfirstlane(w.nch);
  w.last = __builtin_amdgcn_readfirstlane(w.last);
  const uint2 *p = chunk_pointer(stream, __builtin_amdgcn_readfirstlane(w.base));
  const int lane = threadIdx.x & 63;
  const uint32_t w_min = w.minmax & 0xffffu, w_max = w.minmax >> 16;
  GroupSums sum = {{0.f, 0.f, 0.f, 0.f}}, partial = {{0.f, 0.f, 0.f, 0.f}};
  uint32_t at = lds_address(xa) + 4u * static_cast<uint32_t>(w.j0);
  int c = __builtin_amdgcn_readfirstlane(w.c0);
  if (passes) progress_priority(pass, passes);
  auto group_done = [&](int g) {
    if (part) {
      part[g * 64 + lane] = partial;
    } else {
#pragma unroll
      for (int t = 0; t < kGroupTokens; t++) sum.v[t] += partial.v[t];
    }
#pragma unroll
    for (int t = 0; t < kGroupTokens; t++) partial.v[t] = 0.f;
  };
  for (; c < w.nch; c += kRing) {
#pragma unroll
    for (int i = 0; i < kRing; i++) {
      if (c + i < w.nch - 1) {
        const uint2 cw = w.ring[i];
        w.ring[i] = p[min(c + i + kRing, w.nch - 1) * 64];
        add_chunk_group(cw, at, partial, w_min, w_max);
      } else if (c + i == w.nch - 1) {
        add_entries_group(w.ring[i], w.last, at, partial, w_min, w_max);   // the walk's last chunk
      }
    }
    if ((c + kRing) % kGroupChunks == 0) {
      if (passes) progress_priority(pass * w.nch + c + kRing, passes * w.nch);
      group_done((c + kRing) / kGroupChunks - 1);
    }
  }
  // the last, partial group, unless the loop has just closed it
  if (c % kGroupChunks) group_done(c / kGroupChunks);
  return sum;
}

// Small-batch form of a tile: `split` wavefronts share each slice, every one
// taking a run of the slice's chunk groups (it starts from the position
// checkpoint of its first group) and leaving one partial sum per group in LDS;
// after a barrier the slice's first wavefront adds the groups in order, which
// is the canonical order, so the result is the same to the bit as with a
// wavefront per slice.  Built for latency: split_begin puts the loads of a
// whole group in flight, and the kernel calls it before it waits for and
// stages the activations.
struct SplitWalk {
  Walk<kSplitRing> w;   // w.nch: this wavefront's last chunk + 1
  int g_lo, g_hi, ngroups;
  int64_t sl;
  bool mine;
};

// Everything but the position and the ring is the same in all lanes and is kept
// in scalar registers (the wavefront index goes through readfirstlane).  The
// ring loads are unconditional, with the chunk index clamped to the wavefront's
// last chunk, so that they all leave at once.
__device__ __forceinline__ SplitWalk split_begin(const PreparedArgs &a, const KindArgs &k, int e,
                                                 int s0, int s_hi) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int sub = wave % k.split;
  const int s = s0 + wave / k.split;
  SplitWalk r;
  r.mine = s < s_hi;
  r.ngroups = 0;
  r.g_lo = 0;
  r.g_hi = 0;
  r.sl = static_cast<int64_t>(e) * k.slices + s;
  r.w.base = 0;
  r.w.j0 = 0;
  r.w.nch = 0;
  r.w.last = kFields;
  r.w.minmax = 0u;
  r.w.ridx = 0xffff;
  // both words of the slice's description in one round trip (a slice that
  // exists is read also where this wavefront has none)
  const int64_t described = r.mine ? r.sl : static_cast<int64_t>(e) * k.slices + s0;
  const int len_word = k.slice_len[described];
  const uint32_t base_word = k.slice_base[described];
  if (r.mine) {
    const int len = __builtin_amdgcn_readfirstlane(len_word);
    const int nch_all = chunks_of(len);
    r.ngroups = (nch_all + kGroupChunks - 1) / kGroupChunks;
    r.g_lo = sub * r.ngroups / k.split;
    r.g_hi = (sub + 1) * r.ngroups / k.split;
    r.w.minmax = k.minmax[r.sl * 64 + lane];
    if (sub == 0) r.w.ridx = k.row_idx[r.sl * 64 + lane];   // it will write the slice's rows
    if (r.g_lo < r.g_hi) {
      const uint32_t base = __builtin_amdgcn_readfirstlane(base_word);
      r.w.base = base;
      const uint2 *p = chunk_pointer(a.stream, base);
      const int c_lo = r.g_lo * kGroupChunks;
      r.w.nch = min(r.g_hi * kGroupChunks, nch_all);
      r.w.last = r.w.nch == nch_all ? last_entries_of(len) : kFields;
      if (r.g_lo)
        r.w.j0 = a.ckpt[(checkpoint_entry(base, k.first_slice + r.sl) + r.g_lo) * 64 + lane];
#pragma unroll
      for (int i = 0; i < kSplitRing; i++)
        r.w.ring[i] = p[min(c_lo + i, r.w.nch - 1) * 64];
    }
  }
  return r;
}

// The groups of a tile; contains a workgroup barrier.  A wavefront that
// has its slice to itself (split 1) adds the groups in registers, in the same
// order, and leaves the partial-sum area alone.
__device__ __forceinline__ void split_run(const PreparedArgs &a, const KindArgs &k, SplitWalk &r,
                                          const uint32_t *xa, uint16_t *dst, int mode) {
  float *part = reinterpret_cast<float *>(const_cast<uint32_t *>(xa) + a.xdwords);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int local = wave / k.split;
  const bool alone = k.split == 1;
  const bf16x2 minmax = __builtin_bit_cast(bf16x2, r.w.minmax);
  uint32_t at = lds_address(xa) + 4u * static_cast<uint32_t>(r.w.j0);
  float sum = 0.f;
  const uint2 *p = chunk_pointer(a.stream, r.w.base);
  for (int g = r.g_lo; g < r.g_hi; g++) {
    float partial = 0.f;
    const int c_end = min((g + 1) * kGroupChunks, r.w.nch);
    for (int c = g * kGroupChunks; c < c_end; c += kSplitRing) {
      if (c + kSplitRing <= r.w.nch - 1)      // whole chunks only, and more to come
        run_chunks<false>(r.w, p, c, at, partial, minmax);
      else                                    // the run that ends with this wavefront's last chunk
        run_chunks<true>(r.w, p, c, at, partial, minmax);
    }
    if (alone) {
      sum += partial;
    } else {
      part[(local * k.groups_max + g) * 64 + lane] = partial;
    }
  }
  __syncthreads();
  if (r.mine && wave % k.split == 0) {
    if (!alone)
      for (int g = 0; g < r.ngroups; g++) sum += part[(local * k.groups_max + g) * 64 + lane];
    write_row(dst, r.w.ridx, sum, mode);
  }
}

// A wo tile waits until its token's wi tiles have published h (bounded spin of
// one lane, then a barrier that extends its acquire to the workgroup); then the
// tile's activations go into LDS.  Ends with a barrier.  The tile says that it
// has waited (done_waiting) once its work is done: that takes a round trip to
// memory, which does not belong between the wait and the walk.
__device__ __forceinline__ void await_activations(const PreparedArgs &a, const KindArgs &k,
                                                  int kind, int t, uint32_t *xa) {
  if (kind == 1) {
    if (threadIdx.x == 0)
      sub1::bounded_wait(&a.ctrl[sub1::token_word(t)], a.wi_expect, a.wait_ticks, a.sticky,
                         &a.ctrl[kCtrlGaveUp]);
    __syncthreads();
  }
  const uint16_t *src = kind ? a.h + static_cast<int64_t>(t) * k.width
                             : a.x + static_cast<int64_t>(t) * a.ldx;
  stage_activations(xa, src, k.width);
  __syncthreads();
}

__device__ __forceinline__ void done_waiting(const PreparedArgs &a, int t) {
  if (threadIdx.x == 0) sub1::waited_on(&a.ctrl[sub1::token_word(t)], a.k[1].parts);
}

// What a ticket stands for.  Every field is the same in all lanes.
struct Tile {
  int kind, t, s_lo, s_hi, e;   // e < 0: no matrix (token dropped or index out of range)
};

__device__ __forceinline__ Tile decode_tile(const PreparedArgs &a, int ticket, bool count_faults) {
  const int n_wi = a.tokens * a.k[0].parts;
  Tile tile;
  tile.kind = ticket < n_wi ? 0 : 1;
  const KindArgs &k = a.k[tile.kind];
  const int rel = tile.kind ? ticket - n_wi : ticket;
  tile.t = rel / k.parts;
  const int part = rel - tile.t * k.parts;
  // slices [s_lo, s_hi) of the matrix
  tile.s_lo = static_cast<int>(static_cast<int64_t>(k.slices) * part / k.parts);
  tile.s_hi = static_cast<int>(static_cast<int64_t>(k.slices) * (part + 1) / k.parts);
  tile.e = a.token_expert ? __builtin_amdgcn_readfirstlane(a.token_expert[tile.t]) : 0;
  if (tile.e >= a.experts) {
    if (count_faults && tile.kind == a.kinds - 1 && part == 0 && threadIdx.x == 0)
      __hip_atomic_fetch_add(&a.ctrl[kCtrlBadIds], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    tile.e = -1;
  }
  return tile;
}

// A dropped token keeps its input (reference sub1.py:312).
__device__ __forceinline__ void pass_through(const PreparedArgs &a, const KindArgs &k, int t,
                                             int s_lo, int s_hi) {
  const int r_lo = min(64 * s_lo, k.height), r_hi = min(64 * s_hi, k.height);
  for (int i = r_lo + threadIdx.x; i < r_hi; i += blockDim.x)
    a.y[static_cast<int64_t>(t) * a.ldy + i] = a.x[static_cast<int64_t>(t) * a.ldx + i];
}

__device__ __forceinline__ uint16_t *tile_output(const PreparedArgs &a, const KindArgs &k,
                                                 int kind, int t, int &mode) {
  if (a.kinds == 2 && kind == 0) {
    mode = kStoreRelu;
    return a.h + static_cast<int64_t>(t) * k.height;
  }
  mode = a.kinds == 2 ? kStore : a.fresh ? kFresh : kAccumulate;
  return a.y + static_cast<int64_t>(t) * a.ldy;
}

// h of a token's wi tile becomes visible to the wo tiles.  The rows of h are
// stored at agent scope (write_row), i.e. written through the L2 of this
// wavefront's die; every wavefront waits until its own stores are acknowledged,
// the barrier collects the wavefronts, and one lane counts the tile as done.
// A release fence instead of the write-through stores would write back the
// whole L2 (measured 8 us per tile with all compute units at it).
__device__ __forceinline__ void publish_h(const PreparedArgs &a, int t) {
  sub1::drain_stores();
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_fetch_add(&a.ctrl[sub1::token_word(t)], 1, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
}

// The wavefronts of a workgroup walk `all` slices of one matrix: slice `first`
// of the stream's slices and every `stride`-th after it.  `before()` runs once
// the first loads of the stream are out (it stages the activations `act` and
// ends with a barrier); `out(row, sum, slice)` takes every row's result.  A short last
// pass (at most half the wavefronts busy) is shared out: `split` wavefronts per
// slice, each a run of its chunk groups, partial sums in `partials`
// (a.tail_room groups of 64 lanes).
template <class Before, class Out>
__device__ __forceinline__ void walk_alike(const PreparedArgs &a, const KindArgs &k, int64_t first,
                                           int stride, int all, const uint32_t *act,
                                           float *partials, Before &&before, Out &&out,
                                           bool active = true) {
  const int waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int split = 1;
  const int rest = all % waves;
  if (rest > 0 && rest * 2 <= waves && rest * k.groups_max <= a.tail_room)
    split = min(waves / rest, k.groups_max);
  const int count = split > 1 ? all - rest : all;
  const int passes = (count + waves - 1) / waves + (split > 1);
  // the shared last pass: slice `tail_sl` of the tile, this wavefront its
  // groups g_lo .. g_hi - 1 of `groups`
  const int tail_sl = count + wave / split;
  const int sub = wave % split;
  const int64_t tail_slice = first + static_cast<int64_t>(tail_sl) * stride;
  // With a few tokens that pass is the whole walk, and the walk a chain of
  // memory round trips: its loads (the slice's description, then a whole group
  // of chunks) go out before the wait and the staging like the first loads of
  // any other walk.
  const bool tail_only = split > 1 && count == 0;
  int groups = 0, g_lo = 0, g_hi = 0, tail_len = 0;
  uint32_t tail_base = 0;
  auto tail_groups = [&]() {
    if (tail_sl < all) {
      // both words of the slice's description in one round trip
      const int len_word = k.slice_len[tail_slice];
      const uint32_t base_word = k.slice_base[tail_slice];
      tail_len = __builtin_amdgcn_readfirstlane(len_word);
      tail_base = __builtin_amdgcn_readfirstlane(base_word);
      groups = (chunks_of(tail_len) + kGroupChunks - 1) / kGroupChunks;
      g_lo = sub * groups / split;
      g_hi = (sub + 1) * groups / split;
    }
  };
  Walk<kSplitRing> tail_ahead;
  int tail_ridx = 0xffff;   // the rows of the shared slice, in the wavefront that adds them up
  if (tail_only) {
    if (sub == 0 && tail_sl < all && active) tail_ridx = k.row_idx[tail_slice * 64 + (threadIdx.x & 63)];
    tail_groups();
    if (g_lo < g_hi && active)
      tail_ahead = load_slice_described<kSplitRing>(a, k, tail_slice, tail_len, tail_base, g_lo, g_hi);
  }
  int s = slice_of_pass(0, wave, waves, count);
  SliceWalk cur;
  // the first loads of the stream go out before the wait and the staging
  if (s < count && active) cur = load_slice(a, k, first + static_cast<int64_t>(s) * stride);
  before();
  for (int pass = 0; s < count; pass++) {
    const int s_next = slice_of_pass(pass + 1, wave, waves, count);
    SliceWalk nxt;
    if (active) {
      if (s_next < count) nxt = load_slice(a, k, first + static_cast<int64_t>(s_next) * stride);
      const float res = run_slice(cur, a.stream, act, nullptr, pass, passes);
      out(cur.ridx, res, first + static_cast<int64_t>(s) * stride);
      if (s_next < count) cur = nxt;
    }
    s = s_next;
  }
  if (split > 1) {
    __builtin_amdgcn_s_setprio(0);
    const int lane = threadIdx.x & 63;
    float *mine = partials + (wave / split) * k.groups_max * 64;
    if (tail_only) {
      if (g_lo < g_hi && active) run_slice(tail_ahead, a.stream, act, mine);
    } else {
      if (sub == 0 && tail_sl < all && active) tail_ridx = k.row_idx[tail_slice * 64 + lane];
      tail_groups();
      if (g_lo < g_hi && active) {
        SliceWalk tail = load_slice_described(a, k, tail_slice, tail_len, tail_base, g_lo, g_hi);
        run_slice(tail, a.stream, act, mine);
      }
    }
    __syncthreads();
    if (sub == 0 && tail_sl < all && active) {
      float sum = 0.f;
      for (int g = 0; g < groups; g++) sum += mine[g * 64 + lane];
      out(tail_ridx, sum, tail_slice);
    }
  }
}

// The slices that all of a workgroup's wavefronts share, where lengths differ: the
// longest ones, each by as many wavefronts as make their shares alike.
struct SharedSlices {
  int slice;            // this wavefront's, among the shared ones; -1: none
  int split, sub;       // the wavefronts that share it, and which of them this is
  int groups, first_group;   // its groups; where their partial sums begin
  int len;
  uint32_t base;
};

// What is known of a tile's first 64 slices (from `first` on, every `stride`-th, longest first) before
// they are walked: those of slice `lane`.
struct SliceLengths {
  int len;
  uint32_t base;
  int chunks, groups;   // zero: there is no such slice
};
__device__ __forceinline__ SliceLengths slice_lengths(const KindArgs &k, int64_t first, int stride, int all) {
  const int lane = threadIdx.x & 63;
  SliceLengths s = {};
  if (all == 0) return s;
  const int64_t sl = first + static_cast<int64_t>(min(lane, all - 1)) * stride;
  s.len = k.slice_len[sl];
  s.base = k.slice_base[sl];
  s.chunks = lane < all ? chunks_of(s.len) : 0;
  s.groups = (s.chunks + kGroupChunks - 1) / kGroupChunks;
  return s;
}

// How many of the longest slices the wavefronts share: at most half as many as there are of those, and
// as many as have room for their partial sums.  All of a few slices; of more those that leave whole passes, or half
// as many as wavefronts, if what is left is short.  Else as many as give the least for what a wavefront has of them
// and the first wavefront of the others, or none where long ones would be left all the same (a wavefront that
// walks one has its share of the others' behind it).
__host__ __device__ constexpr bool all_shared(int all, int waves, int groups_max, int room) {
  return all <= waves / 2 && all * groups_max <= room;
}
__device__ __forceinline__ int slices_to_share(const SliceLengths &s, int all, int waves, int groups_max, int room) {
  if (all_shared(all, waves, groups_max, room)) return all;   // (known before the lengths are here)
  const int lane = threadIdx.x & 63;
  const int groups_upto = sub1::wave_prefix_sum(s.groups);
  const int rest = all % waves, usual = rest && 2 * rest <= waves ? rest : min(all, waves / 2);
  const int longest = __builtin_amdgcn_readfirstlane(s.chunks);
  // (nothing is left of a few slices: chunks of none are zero)
  if (__builtin_expect(__builtin_amdgcn_readlane(groups_upto, max(usual, 1) - 1) <= room &&
                           2 * __builtin_amdgcn_readlane(s.chunks, usual) <= longest, 1))
    return usual;
  // lane c: with c of them (0.4 us).  Slices beyond the 64 weigh about the same whatever c.
  int others = 0;
#pragma unroll 1
  for (int at = 0; at < 64 && at < all; at += waves) others += __shfl(s.chunks, at + lane, 64);
  // (the barrier and adding up: another group's time)
  const int cost = sub1::wave_prefix_sum(s.chunks) - s.chunks + waves * (others + (lane ? kGroupChunks : 0));
  const bool may = lane <= min(all, waves / 2) && groups_upto - s.groups <= room && (lane == 0 || 2 * s.chunks <= longest);
  constexpr int kMost = (1 << 26) - 1;
  const int gain = may ? max(kMost - cost, 1) : 0;
  // the largest of lanes 0 to 15
  int best = gain;
  best = max(best, sub1::dpp_or_zero<sub1::kDppRowShr1, 0xf>(best));
  best = max(best, sub1::dpp_or_zero<sub1::kDppRowShr2, 0xf>(best));
  best = max(best, sub1::dpp_or_zero<sub1::kDppRowShr4, 0xf>(best));
  best = max(best, sub1::dpp_or_zero<sub1::kDppRowShr8, 0xf>(best));
  return __ffsll(__ballot(gain == __builtin_amdgcn_readlane(best, 15))) - 1;
}

// The `count` longest slices (at most half of `waves`).  A row without zeros has ten times the
// entries of the others, and a slice of 64 such rows kept one or two wavefronts walking long after the rest.
__device__ __forceinline__ SharedSlices share_slices(const SliceLengths &lengths, int count, int waves, int wave) {
  const int lane = threadIdx.x & 63;
  const bool mine = lane < count;
  const int groups = mine ? lengths.groups : 0;
  const int groups_upto = sub1::wave_prefix_sum(groups);
  const int total = __builtin_amdgcn_readlane(groups_upto, 63);
  // the fewest groups a wavefront may have at most with which there are wavefronts enough
  // (at the latest with twice as many as they have on average)
  int split, split_upto;
  for (int most = max((total + waves - 1) / waves, 1);; most++) {
    split = mine ? max((groups + most - 1) / most, 1) : 0;
    split_upto = sub1::wave_prefix_sum(split);
    if (__builtin_amdgcn_readlane(split_upto, 63) <= waves) break;
  }
  const int which = __popcll(__ballot(mine && split_upto - split <= wave)) - 1;
  SharedSlices s;
  s.split = __builtin_amdgcn_readlane(split, which);
  s.sub = wave - (__builtin_amdgcn_readlane(split_upto, which) - s.split);
  s.slice = s.sub < s.split ? which : -1;
  s.groups = __builtin_amdgcn_readlane(groups, which);
  s.first_group = __builtin_amdgcn_readlane(groups_upto, which) - s.groups;
  s.len = __builtin_amdgcn_readlane(lengths.len, which);
  s.base = __builtin_amdgcn_readlane(lengths.base, which);
  return s;
}

// Slices of a tile: of about one length; of differing lengths, so few that the wavefronts share all
// of them (all_shared); of differing lengths, of which they share those that slices_to_share says.
enum Lengths { kAlike, kFew, kDiffer };

// As walk_alike, where lengths differ: the last pass has the longest slices instead, and the
// wavefronts by length.
//
// Bound by the longest slice's chain of groups: a wavefront walked it alone, or a few did where eight
// slices' partial sums, at the longest one's size, fit LDS (beyond rows of some 4400 columns without zeros they
// did not, and the launch fell back on tiles of one projection).  Rows of 75 to 98 % zeros, one in a
// hundred without, us, alike / so: 587 x 4467 one token 22.5 / 17.9, 60 tokens 106 / 30, 200 108 / 54;
// c-2048 13 tokens 48.6 / 33.0, 60 104 / 64, 120 197 / 101, 512 418 / 361; large 60 47 / 32, 200 120 / 72; base 60
// 36 / 25, 400 110 / 79.  (With sixteen slices in that pass, a wavefront each at least, large 200 took 136.)
// More long rows than that pass takes, as slices_to_share counts / with half as many slices as
// wavefronts or those that leave whole passes: c-2048, a tenth of the rows, 128 tokens 109 / 173, 200 196 / 330, 600
// 490 / 757; 1100 x 9000, a fifth, 200 273 / 391; 2048 x 12000, a tenth, 200 459 / 631 (alike 185, 234, 672, 265, 448).
//
// kAhead: where that pass is the whole walk its loads go out before the wait and the staging.  (Whole tokens have
// others to walk, and the code for both costs their loop: base 400 tokens 87 / 81, with kEarly 79.)
template <Lengths kLengths, bool kAhead, class Before, class Out>
__device__ __forceinline__ void walk_by_length(const PreparedArgs &a, const KindArgs &k, int64_t first,
                                               int stride, int all, const uint32_t *act,
                                               float *partials, Before &&before, Out &&out,
                                               bool active = true) {
  const int waves = blockDim.x >> 6, lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const SliceLengths lengths = slice_lengths(k, first, stride, all);
  const int longest = kLengths == kFew ? all : slices_to_share(lengths, all, waves, k.groups_max, a.tail_room);
  const int count = all - longest, passes = (count + waves - 1) / waves + 1;
  const int64_t other = first + static_cast<int64_t>(longest) * stride;   // the first of the others
  int s = slice_of_pass(0, wave, waves, count);
  SliceWalk cur;
  if (s < count && active) {
    // (its description is here already)
    const int at = longest + s;
    cur = load_slice_described(a, k, other + static_cast<int64_t>(s) * stride, __builtin_amdgcn_readlane(lengths.len, at),
                               __builtin_amdgcn_readlane(lengths.base, at), 0, kAllGroups);
  }
  SharedSlices mine;
  mine.slice = -1;
  if (longest == 1) {
    mine.len = __builtin_amdgcn_readfirstlane(lengths.len);
    mine.base = __builtin_amdgcn_readfirstlane(lengths.base);
    mine.groups = __builtin_amdgcn_readfirstlane(lengths.groups);
    mine.split = waves;
    mine.sub = wave;
    mine.slice = 0;
    mine.first_group = 0;
  } else if (longest) {
    mine = share_slices(lengths, longest, waves, wave);
  }
  const int64_t slice = first + static_cast<int64_t>(max(mine.slice, 0)) * stride;
  const bool shares = mine.slice >= 0 && active;
  int g_lo = 0, g_hi = 0;
  if (shares) {
    g_lo = mine.sub * mine.groups / mine.split;
    g_hi = (mine.sub + 1) * mine.groups / mine.split;
  }
  float *sums = shares && mine.split > 1 ? partials + mine.first_group * 64 : nullptr;
  Walk<kSplitRing> ahead;
  int ridx = 0xffff;   // the rows of the slice, in the wavefront that adds them up
  if (shares && mine.sub == 0) ridx = k.row_idx[slice * 64 + lane];
  if (kAhead && count == 0 && g_lo < g_hi) ahead = load_slice_described<kSplitRing>(a, k, slice, mine.len, mine.base, g_lo, g_hi);
  before();
  for (int pass = 0; s < count; pass++) {
    const int s_next = slice_of_pass(pass + 1, wave, waves, count);
    SliceWalk nxt;
    if (active) {
      if (s_next < count) nxt = load_slice(a, k, other + static_cast<int64_t>(s_next) * stride);
      const float res = run_slice<!kAhead>(cur, a.stream, act, nullptr, pass, passes);
      out(cur.ridx, res, other + static_cast<int64_t>(s) * stride);
      if (s_next < count) cur = nxt;
    }
    s = s_next;
  }
  __builtin_amdgcn_s_setprio(0);
  float sum = 0.f;
  if (g_lo < g_hi) {
    if (kAhead && count == 0) {
      sum = run_slice(ahead, a.stream, act, sums);
    } else {
      SliceWalk walk = load_slice_described(a, k, slice, mine.len, mine.base, g_lo, g_hi);
      sum = run_slice<!kAhead>(walk, a.stream, act, sums);
    }
  }
  __syncthreads();
  if (shares && mine.sub == 0) {
    if (sums) {
      sum = 0.f;
#pragma unroll 8
      for (int g = 0; g < mine.groups; g++) sum += sums[g * 64 + lane];
    }
    out(ridx, sum, slice);
  }
}

// (A form of its own of each kernel: the choice within one cost even rows 0.2 us of 12.)
template <Lengths kLengths, class... Args>
__device__ __forceinline__ void walk_tile(const PreparedArgs &a, const KindArgs &k, Args &&...args) {
  if constexpr (kLengths != kAlike) walk_by_length<kLengths, true>(a, k, static_cast<Args &&>(args)...);
  else walk_alike(a, k, static_cast<Args &&>(args)...);
}

// Persistent grid.  A tile is (token, projection, part): the slices of one
// matrix, or of one of `parts` equal ranges of them when there are too few
// tokens to occupy the GPU otherwise; a workgroup stages the token's
// activations once per tile and its wavefronts take the tile's slices in turn.
// All wi tiles are numbered before all wo tiles and handed out by an atomic
// ticket.  A wo tile waits for the wi tiles of its token, which hold smaller
// tickets and so are running or done: the wait always ends.  h is published by
// ONE agent-scope release per tile (thread 0, after every wavefront drained its
// stores and the workgroup barrier) and picked up by one acquire; an agent-scope
// fence costs an L2 write-back on this part, which is why the lanes do not fence
// individually.
template <Lengths kLengths>
__global__ __launch_bounds__(kMaxThreads) void moe_prepared_kernel(PreparedArgs a) {
  extern __shared__ __align__(16) uint32_t lds[];
  __shared__ int s_ticket;
  uint32_t *xa = lds;
  const int n_wi = a.tokens * a.k[0].parts;
  const int n_all = n_wi + (a.kinds == 2 ? a.tokens * a.k[1].parts : 0);
  const bool dynamic = a.ctrl != nullptr;
  // dynamic order: thread 0 asks for the next ticket when its own part of the
  // tile is done, so that the atomic's round trip overlaps the tile's tail (any
  // earlier and the workgroups that start first take tiles away from the last
  // ones); static order: tile = workgroup index + k * grid
  int static_ticket = blockIdx.x;   // the same in every lane, unlike thread 0's next_ticket
  int next_ticket = 0;
  auto fetch_next = [&]() {
    if (dynamic && threadIdx.x == 0)
      next_ticket = __hip_atomic_fetch_add(&a.ctrl[0], 1, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
  };
  fetch_next();
  for (;;) {
    __syncthreads();
    int ticket;
    if (dynamic) {
      if (threadIdx.x == 0) s_ticket = next_ticket;
      __syncthreads();
      ticket = __builtin_amdgcn_readfirstlane(s_ticket);   // the same in every lane: scalar
    } else {
      ticket = static_ticket;
      static_ticket += gridDim.x;
    }
    if (ticket >= n_all) break;
    const Tile tile = decode_tile(a, ticket, dynamic);
    const int kind = tile.kind, t = tile.t, s_lo = tile.s_lo, s_hi = tile.s_hi, e = tile.e;
    const KindArgs &k = a.k[kind];
    if (a.kinds == 2 && kind == 1 && e < 0) {
      pass_through(a, k, t, s_lo, s_hi);
      fetch_next();
      continue;
    }
    if (e >= 0) {
      int mode;
      uint16_t *dst = tile_output(a, k, kind, t, mode);
      walk_tile<kLengths>(a, k, static_cast<int64_t>(e) * k.slices + s_lo, 1, s_hi - s_lo, xa,
                reinterpret_cast<float *>(xa + a.xdwords),
                [&]() { await_activations(a, k, kind, t, xa); },
                [&](int ridx, float res, int64_t) { write_row(dst, ridx, res, mode); });
    }
    fetch_next();
    if (a.kinds == 2 && kind == 0 && e >= 0) publish_h(a, t);   // a dropped token's word stays untouched
    if (a.kinds == 2 && kind == 1 && e >= 0) done_waiting(a, t);
  }
  if (dynamic && threadIdx.x == 0) sub1::leave_launch(a.ctrl, gridDim.x);
}

// Tokens by expert, for the fused kernel when experts receive several tokens
// each.  One workgroup: counts per expert (tokens that name no expert in a
// bucket of their own), prefix sums, then every token takes a place among its
// expert's tokens and, if its place starts one, writes a tile: four tokens of
// an expert walk the stream together, three too; one or two left over go one
// by one (a walk for four costs about as much as 2.3 single ones).
//   tab: int32 [4, experts + 1]: counts, first place, first tile, next place
// ctrl[3] receives the number of tiles, ctrl[2] the tokens whose expert id is
// too large.  Which tokens share a walk depends on the order in which they
// take their places (atomics) and may differ from run to run; each token's
// result does not depend on it.
__device__ __forceinline__ int32_t load_l2(const int32_t *p) {   // past the L1: atomics update L2 only
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__host__ __device__ constexpr int tiles_of(int n) {
  return n / kGroupTokens + (n % kGroupTokens == 3 ? 1 : n % kGroupTokens);
}

__global__ __launch_bounds__(1024) void group_tokens_kernel(
    const int32_t *__restrict__ token_expert, int tokens, int experts, int32_t *__restrict__ tab,
    int32_t *__restrict__ order, int2 *__restrict__ groups, int32_t *__restrict__ ctrl) {
  __shared__ int32_t seg_tokens[1024], seg_tiles[1024];
  const int tid = threadIdx.x;
  const int buckets = experts + 1;
  int32_t *count = tab, *first = tab + buckets, *tile0 = tab + 2 * buckets,
          *next = tab + 3 * buckets;
  for (int b = tid; b < buckets; b += 1024) count[b] = 0;
  __syncthreads();
  int faults = 0;
  for (int t = tid; t < tokens; t += 1024) {
    const int e = token_expert[t];
    if (e >= experts) faults++;
    atomicAdd(&count[e < 0 || e >= experts ? experts : e], 1);
  }
  if (faults) atomicAdd(&ctrl[2], faults);
  __syncthreads();
  // prefix sums over the buckets: a run of buckets per thread, then the runs
  const int seg = (buckets + 1023) / 1024;
  const int lo = min(tid * seg, buckets), hi = min(lo + seg, buckets);
  int32_t n_tok = 0, n_tile = 0;
  for (int b = lo; b < hi; b++) {
    const int n = load_l2(&count[b]);
    n_tok += n;
    n_tile += b == experts ? n : tiles_of(n);
  }
  seg_tokens[tid] = n_tok;
  seg_tiles[tid] = n_tile;
  __syncthreads();
  for (int d = 1; d < 1024; d *= 2) {
    const int32_t a0 = tid >= d ? seg_tokens[tid - d] : 0, a1 = tid >= d ? seg_tiles[tid - d] : 0;
    __syncthreads();
    seg_tokens[tid] += a0;
    seg_tiles[tid] += a1;
    __syncthreads();
  }
  int32_t run_tok = tid ? seg_tokens[tid - 1] : 0, run_tile = tid ? seg_tiles[tid - 1] : 0;
  for (int b = lo; b < hi; b++) {
    const int n = load_l2(&count[b]);
    first[b] = run_tok;
    next[b] = run_tok;
    tile0[b] = run_tile;
    run_tok += n;
    run_tile += b == experts ? n : tiles_of(n);
  }
  if (tid == 1023) ctrl[3] = seg_tiles[1023];
  __syncthreads();
  for (int t = tid; t < tokens; t += 1024) {
    const int e = token_expert[t];
    const int b = e < 0 || e >= experts ? experts : e;
    const int place = atomicAdd(&next[b], 1);
    order[place] = t;
    const int i = place - load_l2(&first[b]), n = load_l2(&count[b]);
    const int t0 = load_l2(&tile0[b]);
    const int whole = b == experts ? 0 : n / kGroupTokens * kGroupTokens;   // tokens in tiles of four
    const int rest = n - whole;
    if (i < whole) {
      if (i % kGroupTokens == 0) groups[t0 + i / kGroupTokens] = make_int2(e, place * 8 + kGroupTokens);
    } else if (b != experts && rest == 3) {
      if (i == whole) groups[t0 + whole / kGroupTokens] = make_int2(e, place * 8 + 3);
    } else {
      groups[t0 + whole / kGroupTokens + (i - whole)] = make_int2(b == experts ? -1 : e, place * 8 + 1);
    }
  }
}

// A tile of the fused kernel with three or four tokens of one expert: the
// same two phases, both walked once for all of them (see "four tokens per
// walk").  order[place ..] are the tokens; h sits in LDS as (h0, h1), (h2, h3)
// per physical column.  Ends before the loop's barrier.
template <class FetchNext>
__device__ __forceinline__ void fused_group_tile(const PreparedArgs &a, uint32_t *xa, uint32_t *ha,
                                                 int e, int place, int n, FetchNext &&fetch_next) {
  const KindArgs &ki = a.k[0];
  const KindArgs &ko = a.k[1];
  const int waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  int tok[kGroupTokens];
  GroupRows rows;
#pragma unroll
  for (int k = 0; k < kGroupTokens; k++) {
    tok[k] = k < n ? __builtin_amdgcn_readfirstlane(a.order[place + k]) : -1;
    rows.row[k] = k < n ? a.x + static_cast<int64_t>(tok[k]) * a.ldx : nullptr;
  }
  // wi: x -> relu(h) into LDS
  const int64_t first_i = static_cast<int64_t>(e) * ki.slices;
  int s = slice_of_pass(0, wave, waves, ki.slices);
  SliceWalk cur;
  if (s < ki.slices) cur = load_slice(a, ki, first_i + s);
  stage_group(xa, rows, ki.width);
  __syncthreads();
  for (int pass = 0; s < ki.slices; pass++) {
    const int s_next = slice_of_pass(pass + 1, wave, waves, ki.slices);
    SliceWalk nxt;
    if (s_next < ki.slices) nxt = load_slice(a, ki, first_i + s_next);
    const GroupSums res = run_slice_group(cur, a.stream, xa, nullptr, pass,
                                          (ki.slices + waves - 1) / waves);
    if (cur.ridx != 0xffff) {
      uint32_t out[kGroupTokens];
#pragma unroll
      for (int k = 0; k < kGroupTokens; k++) {
        out[k] = f32_to_bf16(res.v[k]);
        if (out[k] & 0x8000u) out[k] = 0;   // relu between the projections, on the bf16 value
      }
      uint32_t *p = ha + 2 * physical_column(cur.ridx);
      p[0] = out[0] | (out[1] << 16);
      p[1] = out[2] | (out[3] << 16);
    }
    if (s_next < ki.slices) cur = nxt;
    s = s_next;
  }
  fetch_next();
  // wo: h -> y, the short last pass shared out as for a single token
  const int whole = ko.tail_split ? ko.slices - ko.slices % waves : ko.slices;
  const int64_t first = static_cast<int64_t>(e) * ko.slices;
  s = slice_of_pass(0, wave, waves, whole);
  if (s < whole) cur = load_slice(a, ko, first + s);
  __syncthreads();
  auto write_rows = [&](int ridx, const GroupSums &res) {
#pragma unroll
    for (int k = 0; k < kGroupTokens; k++)
      if (k < n) write_row(a.y + static_cast<int64_t>(tok[k]) * a.ldy, ridx, res.v[k], kStore);
  };
  for (int pass = 0; s < whole; pass++) {
    const int s_next = slice_of_pass(pass + 1, wave, waves, whole);
    SliceWalk nxt;
    if (s_next < whole) nxt = load_slice(a, ko, first + s_next);
    const GroupSums res = run_slice_group(cur, a.stream, ha, nullptr, pass, (whole + waves - 1) / waves);
    write_rows(cur.ridx, res);
    if (s_next < whole) cur = nxt;
    s = s_next;
  }
  __builtin_amdgcn_s_setprio(0);
  if (ko.tail_split) {
    const int sl = whole + wave / ko.tail_split;
    const int sub = wave % ko.tail_split;
    GroupSums *mine = reinterpret_cast<GroupSums *>(xa) + (wave / ko.tail_split) * ko.groups_max * 64;
    int groups = 0;
    if (sl < ko.slices) {
      groups = (chunks_of(__builtin_amdgcn_readfirstlane(ko.slice_len[first + sl])) +
                kGroupChunks - 1) / kGroupChunks;
      const int g_lo = sub * groups / ko.tail_split, g_hi = (sub + 1) * groups / ko.tail_split;
      if (g_lo < g_hi) {
        SliceWalk tail = load_slice(a, ko, first + sl, g_lo, g_hi);
        run_slice_group(tail, a.stream, ha, mine, 0, 0);
      }
    }
    __syncthreads();
    if (sub == 0 && sl < ko.slices) {
      GroupSums sum = {{0.f, 0.f, 0.f, 0.f}};
      for (int g = 0; g < groups; g++) {
        const GroupSums v = mine[g * 64 + lane];
#pragma unroll
        for (int k = 0; k < kGroupTokens; k++) sum.v[k] += v.v[k];
      }
      write_rows(ko.row_idx[(first + sl) * 64 + lane], sum);
    }
  }
}

// Streaming form for batches of at least one token per compute unit: a tile is
// a token, and the workgroup runs wi, ReLU and wo back to back with h kept in
// LDS, already in the layout wo reads its activations from.  No workspace
// traffic for h, no waiting between workgroups; tickets only balance the load.
// LDS: x (wi's activations) | h (wo's activations).
// kOnce: see load_chunk.  kUneven: the longest slices are shared (walk_tile; LDS: x | h | partial sums).
template <bool kGrouped, bool kOnce, bool kUneven = false>
__global__ __launch_bounds__(kMaxThreads) void moe_prepared_fused_kernel(PreparedArgs a) {
  typedef Walk<kRing, kOnce> TokenWalk;
  extern __shared__ __align__(16) uint32_t lds[];
  __shared__ int s_ticket;
  uint32_t *xa = lds;
  uint32_t *ha = xa + a.xdwords;
  const int threads = blockDim.x;
  const int waves = threads >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const KindArgs &ki = a.k[0];
  const KindArgs &ko = a.k[1];
  // h: the lanes overwrite the two value dwords of their rows; the zeros between
  // them stay for the whole launch
  for (int i = threadIdx.x; i < a.hdwords; i += threads) ha[i] = 0u;
  // tokens grouped by expert: the tiles are in a.groups, ctrl[3] of them
  const int n_tiles = kGrouped ? __builtin_amdgcn_readfirstlane(a.ctrl[3]) : a.tokens;
  int next_ticket = 0;
  auto fetch_next = [&]() {
    if (threadIdx.x == 0)
      next_ticket = __hip_atomic_fetch_add(&a.ctrl[0], 1, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
  };
  fetch_next();
  for (;;) {
    __syncthreads();   // the previous token's wo has read h; s_ticket is free
    if (threadIdx.x == 0) s_ticket = next_ticket;
    __syncthreads();
    const int tile = __builtin_amdgcn_readfirstlane(s_ticket);
    if (tile >= n_tiles) break;
    int t = tile, e, n = 1, place = 0;
    if (kGrouped) {
      const int2 rec = a.groups[tile];
      e = __builtin_amdgcn_readfirstlane(rec.x);
      place = __builtin_amdgcn_readfirstlane(rec.y >> 3);
      n = __builtin_amdgcn_readfirstlane(rec.y & 7);
      t = __builtin_amdgcn_readfirstlane(a.order[place]);
    } else {
      e = __builtin_amdgcn_readfirstlane(a.token_expert[t]);
      if (e >= a.experts) {
        if (threadIdx.x == 0)
          __hip_atomic_fetch_add(&a.ctrl[2], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        e = -1;
      }
    }
    if (e < 0) {
      pass_through(a, ko, t, 0, ko.slices);
      fetch_next();
      continue;
    }
    if (kGrouped && n > 2) {
      fused_group_tile(a, xa, ha, e, place, n, fetch_next);
      continue;
    }
    // wi: x -> relu(h) into LDS
    const int64_t first_i = static_cast<int64_t>(e) * ki.slices;
    if constexpr (kUneven) {
      float *partials = reinterpret_cast<float *>(ha + a.hdwords);
      walk_by_length<kDiffer, false>(a, ki, first_i, 1, ki.slices, xa, partials,
                      [&]() {
                        stage_activations(xa, a.x + static_cast<int64_t>(t) * a.ldx, ki.width);
                        __syncthreads();
                      },
                      [&](int ridx, float res, int64_t) {
                        if (ridx == 0xffff) return;
                        uint32_t out = f32_to_bf16(res);
                        if (out & 0x8000u) out = 0;
                        uint32_t *p = ha + 2 * physical_column(ridx);
                        p[0] = out;
                        p[1] = out << 16;
                      });
      fetch_next();
      uint16_t *dst = a.y + static_cast<int64_t>(t) * a.ldy;
      walk_by_length<kDiffer, false>(a, ko, static_cast<int64_t>(e) * ko.slices, 1, ko.slices, ha, partials,
                      [&]() { __syncthreads(); },
                      [&](int ridx, float res, int64_t) { write_row(dst, ridx, res, kStore); });
      __builtin_amdgcn_s_setprio(0);
      continue;
    }
    int s = slice_of_pass(0, wave, waves, ki.slices);
    TokenWalk cur;
    if (s < ki.slices) cur = load_slice<kRing, kOnce>(a, ki, first_i + s);
    stage_activations(xa, a.x + static_cast<int64_t>(t) * a.ldx, ki.width);
    __syncthreads();
    for (int pass = 0; s < ki.slices; pass++) {
      const int s_next = slice_of_pass(pass + 1, wave, waves, ki.slices);
      TokenWalk nxt;
      if (s_next < ki.slices) nxt = load_slice<kRing, kOnce>(a, ki, first_i + s_next);
      const float res = run_slice(cur, a.stream, xa, nullptr, pass,
                                  (ki.slices + waves - 1) / waves);
      if (cur.ridx != 0xffff) {
        uint32_t out = f32_to_bf16(res);
        if (out & 0x8000u) out = 0;   // relu between the projections, on the bf16 value
        uint32_t *p = ha + 2 * physical_column(cur.ridx);
        p[0] = out;
        p[1] = out << 16;
      }
      if (s_next < ki.slices) cur = nxt;
      s = s_next;
    }
    // the next token is asked for halfway through this one: early enough to
    // hide the round trip, late enough that the workgroups that started first
    // do not take the last tokens away from the others
    fetch_next();
    // wo: h -> y; its first loads go out before the barrier.  A short last pass
    // (tail_split != 0) is shared out: tail_split wavefronts per slice, each a
    // run of its chunk groups, partial sums into the LDS that held x.
    const int whole = ko.tail_split ? ko.slices - ko.slices % waves : ko.slices;
    const int64_t first = static_cast<int64_t>(e) * ko.slices;
    s = slice_of_pass(0, wave, waves, whole);
    if (s < whole) cur = load_slice<kRing, kOnce>(a, ko, first + s);
    __syncthreads();
    uint16_t *dst = a.y + static_cast<int64_t>(t) * a.ldy;
    for (int pass = 0; s < whole; pass++) {
      const int s_next = slice_of_pass(pass + 1, wave, waves, whole);
      TokenWalk nxt;
      if (s_next < whole) nxt = load_slice<kRing, kOnce>(a, ko, first + s_next);
      const float res = run_slice(cur, a.stream, ha, nullptr, pass, (whole + waves - 1) / waves);
      write_row(dst, cur.ridx, res, kStore);
      if (s_next < whole) cur = nxt;
      s = s_next;
    }
    __builtin_amdgcn_s_setprio(0);
    if (ko.tail_split) {
      const int lane = threadIdx.x & 63;
      const int sl = whole + wave / ko.tail_split;
      const int sub = wave % ko.tail_split;
      float *mine = reinterpret_cast<float *>(xa) + (wave / ko.tail_split) * ko.groups_max * 64;
      int groups = 0;
      if (sl < ko.slices) {
        groups = (chunks_of(__builtin_amdgcn_readfirstlane(ko.slice_len[first + sl])) +
                  kGroupChunks - 1) / kGroupChunks;
        const int g_lo = sub * groups / ko.tail_split, g_hi = (sub + 1) * groups / ko.tail_split;
        if (g_lo < g_hi) {
          TokenWalk tail = load_slice<kRing, kOnce>(a, ko, first + sl, g_lo, g_hi);
          run_slice(tail, a.stream, ha, mine);
        }
      }
      __syncthreads();
      if (sub == 0 && sl < ko.slices) {
        // the slice's first wavefront adds the groups in order and writes the rows
        float sum = 0.f;
        for (int g = 0; g < groups; g++) sum += mine[g * 64 + lane];
        write_row(dst, ko.row_idx[(first + sl) * 64 + lane], sum, kStore);
      }
    }
  }
  if (threadIdx.x == 0) sub1::leave_launch(a.ctrl, gridDim.x);
}

// ---- h by tag ----------------------------------------------------------------
//
// A row of relu(h) into the tagged copy: value and tag in one 64-bit store,
// written through like the plain rows of h.
__device__ __forceinline__ void write_tagged(unsigned long long *dst, int ridx, float res,
                                             unsigned long long tag) {
  if (ridx == 0xffff) return;   // padding lane
  uint16_t out = f32_to_bf16(res);
  if (out & 0x8000u) out = 0;   // relu between the projections, on the bf16 value
  __hip_atomic_store(&dst[ridx], (tag << 16) | out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The same into a copy kept in wi's row order: `where` is the row's place in
// that order, so that a wavefront's 64 results are 512 consecutive bytes.
__device__ __forceinline__ void write_tagged_placed(unsigned long long *dst, int ridx, int where,
                                                    float res, unsigned long long tag) {
  if (ridx == 0xffff) return;   // padding lane
  uint16_t out = f32_to_bf16(res);
  if (out & 0x8000u) out = 0;   // relu between the projections, on the bf16 value
  __hip_atomic_store(&dst[where], (tag << 16) | out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The activations of wo from the tagged copy into LDS: a thread reads its
// entries, all in flight at once, until each carries `want` (the value then
// belongs to this launch: no count, no fence).  Bounded in time like the other
// waits; a thread that gives up raises the flag, counts itself and stages what
// it has.  Ends with a barrier.  The launch runs 1024 threads a workgroup.
constexpr int kTaggedWidthPerThread = sub1::kTaggedWidth / kMaxThreads;
__device__ __forceinline__ void await_tagged(const PreparedArgs &a, const KindArgs &k,
                                             const unsigned long long *src,
                                             unsigned long long want, uint32_t *xa) {
  constexpr int kMine = kTaggedWidthPerThread;   // entries a thread may have (width / 1024)
  const int width = k.width;
  const int step = blockDim.x;
  for (int z = threadIdx.x * kZeroPeriod; z < physical_columns(width); z += step * kZeroPeriod) {
    xa[2 * z] = 0u;
    xa[2 * z + 1] = 0u;
  }
  unsigned long long v[kMine];
#pragma unroll
  for (int u = 0; u < kMine; u++) v[u] = 0;
  int looks = 0;
  int64_t t0 = 0;
  for (;;) {
    bool all = true;
#pragma unroll
    for (int u = 0; u < kMine; u++) {
      const int i = threadIdx.x + u * step;
      if (i < width && (v[u] >> 16) != want) {
        v[u] = __hip_atomic_load(&src[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        all = all && (v[u] >> 16) == want;
      }
    }
    if (all) break;
    if ((++looks & 15) == 1) {
      const int64_t now = static_cast<int64_t>(wall_clock64());
      if (looks == 1) t0 = now;
      if (now - t0 > a.wait_ticks) {
        sub1::raise_fault(a.sticky, sub1::kFaultWait);
        __hip_atomic_fetch_add(&a.ctrl[kCtrlGaveUp], 1, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
    }
    __builtin_amdgcn_s_sleep(1);
  }
#pragma unroll
  for (int u = 0; u < kMine; u++) {
    const int i = threadIdx.x + u * step;
    if (i < width) {
      uint32_t *p = xa + 2 * physical_column(i);
      const uint32_t value = static_cast<uint32_t>(v[u]) & 0xffffu;
      p[0] = value;
      p[1] = value << 16;
    }
  }
  __syncthreads();
}

// The same from a copy kept in wi's row order (write_tagged_placed): entry p
// belongs to row `order[p]` of h (0xffff: a padding lane, never written).  A
// thread asks for its part of `order` first - the workgroups that call this
// have nothing else to do until h is there - and then reads its entries, all
// in flight at once, until each
// carries `want` (the value then belongs to this launch: no count, no fence).
// Bounded in time like the other waits; a thread that gives up raises the flag,
// counts itself and stages what it has.  Ends with a barrier.  The launch runs
// 1024 threads a workgroup.
__device__ __forceinline__ void await_tagged_placed(const PreparedArgs &a, const KindArgs &k,
                                             const unsigned long long *src,
                                             const uint16_t *order, int places,
                                             unsigned long long want, uint32_t *xa) {
  constexpr int kMine = kTaggedWidthPerThread;   // entries a thread may have (places / 1024)
  static_assert(kMine % 2 == 0, "rows and values are kept two to a register");
  const int width = k.width;
  const int step = blockDim.x;
  // two 16-bit row indices, and later two bf16 values, to a register: the
  // wavefronts of this workgroup hold their chunks of wo in registers meanwhile
  uint32_t rows[kMine / 2], vals[kMine / 2];
  uint32_t pending = 0;   // bit u: entry u is a row of h and has not been seen with the tag yet
#pragma unroll
  for (int u = 0; u < kMine; u++) {
    const int i = threadIdx.x + u * step;
    const uint32_t r = i < places ? static_cast<uint32_t>(order[i]) : 0xffffu;
    if (u & 1) rows[u / 2] |= r << 16;
    else rows[u / 2] = r;
    if (r != 0xffffu) pending |= 1u << u;
  }
#pragma unroll
  for (int u = 0; u < kMine / 2; u++) vals[u] = 0u;
  for (int z = threadIdx.x * kZeroPeriod; z < physical_columns(width); z += step * kZeroPeriod) {
    xa[2 * z] = 0u;
    xa[2 * z + 1] = 0u;
  }
  int looks = 0;
  int64_t t0 = 0;
  while (pending) {
#pragma unroll
    for (int u = 0; u < kMine; u++) {
      if (pending & (1u << u)) {
        const unsigned long long v = __hip_atomic_load(&src[threadIdx.x + u * step], __ATOMIC_RELAXED,
                                                       __HIP_MEMORY_SCOPE_AGENT);
        if ((v >> 16) == want) {
          pending &= ~(1u << u);
          vals[u / 2] |= (static_cast<uint32_t>(v) & 0xffffu) << (16 * (u & 1));
        }
      }
    }
    if (!pending) break;
    if ((++looks & 15) == 1) {
      const int64_t now = static_cast<int64_t>(wall_clock64());
      if (looks == 1) t0 = now;
      if (now - t0 > a.wait_ticks) {
        sub1::raise_fault(a.sticky, sub1::kFaultWait);
        __hip_atomic_fetch_add(&a.ctrl[kCtrlGaveUp], 1, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
    }
    __builtin_amdgcn_s_sleep(1);
  }
#pragma unroll
  for (int u = 0; u < kMine; u++) {
    const uint32_t r = (rows[u / 2] >> (16 * (u & 1))) & 0xffffu;
    if (r != 0xffffu) {
      uint32_t *p = xa + 2 * physical_column(static_cast<int>(r));
      const uint32_t value = (vals[u / 2] >> (16 * (u & 1))) & 0xffffu;
      p[0] = value;
      p[1] = value << 16;
    }
  }
  __syncthreads();
}

// Thread 0 of a workgroup that leaves a launch of the tagged kind: the last one
// out makes the next launch's tag.
__device__ __forceinline__ void leave_tagged(int32_t *ctrl, int workgroups) {
  const int32_t before = __hip_atomic_fetch_add(&ctrl[sub1::kCtrlExits], 1, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
  if (before + 1 == workgroups) {
    __hip_atomic_store(&ctrl[sub1::kCtrlExits], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_fetch_add(reinterpret_cast<unsigned long long *>(ctrl + sub1::kCtrlLaunch), 1ull,
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Between the latency form and a token per workgroup: with fewer tokens than
// half the compute units, `parts` workgroups share a token.  Each takes every
// parts-th slice of wi (the slices are ordered longest first, so the shares are
// even), writes its rows of relu(h) to the workspace, counts itself done, waits
// for the others of its token, stages the whole of h and takes every parts-th
// slice of wo.  Unlike tiles of one projection handed out by ticket, every
// workgroup works in both phases, the token's activations are staged once per
// phase and workgroup, and h crosses memory once.
// The workgroups of a token wait for each other.  A grid (tokens x parts) of at
// most one workgroup per compute unit runs all at once on a GPU that does
// nothing else, whatever order the hardware starts them in, and a workgroup's
// place in it is its index: no round trip before the work starts, which
// measured 1.5 to 2.0 us per launch against places by ticket (c-2048 shapes: 4
// tokens 15.9 against 17.4 us, 16 tokens 22.5 against 24.6, 64 tokens 43.0
// against 45.0, 128 tokens 75.9 against 77.9).  Where other work holds compute
// units, the missing workgroups start when that work ends, and the waits are
// bounded in any case.
// A larger grid cannot be on the GPU at once, and there a workgroup takes its
// place by ticket when it starts (by_ticket): the workgroups that are running
// then hold the lowest places, the places of a token are consecutive, so at
// most one token is partly on the GPU whatever order the hardware starts
// workgroups in; all others run to completion and make room.
template <Lengths kOfWi, Lengths kOfWo>
__global__ __launch_bounds__(kMaxThreads) void moe_prepared_shared_kernel(PreparedArgs a) {
  extern __shared__ __align__(16) uint32_t lds[];
  __shared__ int s_place;
  uint32_t *xa = lds;
  float *partials = reinterpret_cast<float *>(xa + a.xdwords);
  const KindArgs &ki = a.k[0];
  const KindArgs &ko = a.k[1];
  const int parts = ki.parts;
  int place = blockIdx.x;
  if (a.by_ticket) {
    if (threadIdx.x == 0)
      s_place = __hip_atomic_fetch_add(&a.ctrl[kCtrlTicket], 1, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    place = __builtin_amdgcn_readfirstlane(s_place);
  }
  const int t = place / parts;
  const int part = place - t * parts;
  // the token's activations are asked for before anything else is known
  const uint16_t *x = a.x + static_cast<int64_t>(t) * a.ldx;
  const StagedPairs x_ahead = stage_request(x, ki.width);
  int e = __builtin_amdgcn_readfirstlane(a.token_expert[t]);
  if (e >= a.experts) {
    if (part == 0 && threadIdx.x == 0)
      __hip_atomic_fetch_add(&a.ctrl[2], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    e = -1;
  }
  if (e < 0) {
    if (part == 0) pass_through(a, ko, t, 0, ko.slices);
    if (a.by_ticket && threadIdx.x == 0) sub1::leave_launch(a.ctrl, gridDim.x);
    return;
  }
  uint16_t *h = a.h + static_cast<int64_t>(t) * ki.height;
  walk_tile<kOfWi>(a, ki, static_cast<int64_t>(e) * ki.slices + part, parts,
            (ki.slices - part + parts - 1) / parts, xa, partials,
            [&]() {
              stage_finish(xa, x, ki.width, x_ahead);
              __syncthreads();
            },
            [&](int ridx, float res, int64_t) { write_row(h, ridx, res, kStoreRelu); });
  publish_h(a, t);
  uint16_t *y = a.y + static_cast<int64_t>(t) * a.ldy;
  walk_tile<kOfWo>(a, ko, static_cast<int64_t>(e) * ko.slices + part, parts,
            (ko.slices - part + parts - 1) / parts, xa, partials,
            [&]() { await_activations(a, ko, 1, t, xa); },
            [&](int ridx, float res, int64_t) { write_row(y, ridx, res, kStore); });
  done_waiting(a, t);
  if (a.by_ticket && threadIdx.x == 0) sub1::leave_launch(a.ctrl, gridDim.x);
}

// The shared-token kernel for a token or two, h handed over by tag (see
// await_tagged): no drain, no barrier, no count between the projections, and no
// word to give back at the end.  A workgroup's place is its index: the grid is
// at most 64 workgroups.
template <Lengths kLengths>
__global__ __launch_bounds__(kMaxThreads) void moe_prepared_tagged_kernel(PreparedArgs a) {
  extern __shared__ __align__(16) uint32_t lds[];
  uint32_t *xa = lds;
  float *partials = reinterpret_cast<float *>(xa + a.xdwords);
  const KindArgs &ki = a.k[0];
  const KindArgs &ko = a.k[1];
  const int parts = ki.parts;
  const int t = blockIdx.x / parts;
  const int part = blockIdx.x - t * parts;
  // the token's activations and this launch's tag (one more than the launches
  // so far) are asked for before anything else is known
  const uint16_t *x = a.x + static_cast<int64_t>(t) * a.ldx;
  const StagedPairs x_ahead = stage_request(x, ki.width);
  const unsigned long long tag =
      __hip_atomic_load(reinterpret_cast<unsigned long long *>(a.ctrl + sub1::kCtrlLaunch),
                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
  int e = __builtin_amdgcn_readfirstlane(a.token_expert[t]);
  if (e >= a.experts) {
    if (part == 0 && threadIdx.x == 0)
      __hip_atomic_fetch_add(&a.ctrl[2], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    e = -1;
  }
  if (e < 0) {
    if (part == 0) pass_through(a, ko, t, 0, ko.slices);
    if (threadIdx.x == 0) leave_tagged(a.ctrl, gridDim.x);
    return;
  }
  unsigned long long *ht = a.tagged + static_cast<int64_t>(t) * sub1::kTaggedWidth;
  walk_tile<kLengths>(a, ki, static_cast<int64_t>(e) * ki.slices + part, parts,
            (ki.slices - part + parts - 1) / parts, xa, partials,
            [&]() {
              stage_finish(xa, x, ki.width, x_ahead);
              __syncthreads();
            },
            [&](int ridx, float res, int64_t) { write_tagged(ht, ridx, res, tag); });
  __syncthreads();   // every wavefront is done with x before h takes its place
  uint16_t *y = a.y + static_cast<int64_t>(t) * a.ldy;
  // (a test that overstates the wait looks for a tag that nobody writes)
  const unsigned long long want = a.wi_expect == parts ? tag : tag + 1;
  walk_tile<kLengths>(a, ko, static_cast<int64_t>(e) * ko.slices + part, parts,
            (ko.slices - part + parts - 1) / parts, xa, partials,
            [&]() { await_tagged(a, ko, ht, want, xa); },
            [&](int ridx, float res, int64_t) { write_row(y, ridx, res, kStore); });
  if (threadIdx.x == 0) leave_tagged(a.ctrl, gridDim.x);
}

// The same with workgroups of its own for wo (one token; two through shapes
// whose wo rows are long).  The first k[0].parts of a token's workgroups walk wi
// (every k[0].parts-th slice from their own; they wait for nobody, so there is
// one per slice where the chip has room) and leave; the others belong to wo and
// ask for all they need of the stream - the descriptions of their slices, the
// row indices and every chunk they will walk (a wavefront's share is one group
// of chunks, which its ring holds) - while wi is still being walked elsewhere.
// Between the last row of h and the first row of y then lie the hand-over and
// a walk whose chunks are in registers already.  For one token a.lane_parts = 2
// workgroups share each slice of wo, 32 lanes (rows) each: the 9 to 14
// wavefronts of a slice gather from one LDS, which takes 32 lanes a pass.
// One token through a c-2048 expert: 13.4 -> 11.9 us (a different expert every
// launch 14.8 -> 12.2), two tokens 15.4 -> 12.8; one token through a base
// expert 11.5 -> 10.7, a large one 11.7 -> 11.5.
// 62 KB of code, each instruction of it run about once: where it lies makes 0.15 us
// (the same instructions behind kernels of another size 11.83 and 11.97), so it has a place of its own.
template <Lengths kLengths>
__device__ __forceinline__ void tagged_split(const PreparedArgs &a) {
  extern __shared__ __align__(16) uint32_t lds[];
  uint32_t *xa = lds;
  float *partials = reinterpret_cast<float *>(xa + a.xdwords);
  const KindArgs &ki = a.k[0];
  const KindArgs &ko = a.k[1];
  const int per_token = ki.parts + ko.parts * a.lane_parts;
  const int t = blockIdx.x / per_token;
  const int place = blockIdx.x - t * per_token;
  const bool for_wo = place >= ki.parts;
  // this launch's tag (one more than the launches so far), and for wi the
  // token's activations, are asked for before anything else is known
  const uint16_t *x = a.x + static_cast<int64_t>(t) * a.ldx;
  StagedPairs x_ahead;
  if (!for_wo) x_ahead = stage_request(x, ki.width);
  const unsigned long long tag =
      __hip_atomic_load(reinterpret_cast<unsigned long long *>(a.ctrl + sub1::kCtrlLaunch),
                        __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
  int e = __builtin_amdgcn_readfirstlane(a.token_expert[t]);
  if (e >= a.experts) {
    if (place == 0 && threadIdx.x == 0)
      __hip_atomic_fetch_add(&a.ctrl[2], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    e = -1;
  }
  if (e < 0) {
    if (place == 0) pass_through(a, ko, t, 0, ko.slices);
    if (threadIdx.x == 0) leave_tagged(a.ctrl, gridDim.x);
    return;
  }
  unsigned long long *ht = a.tagged + static_cast<int64_t>(t) * sub1::kTaggedWidth;
  if (!for_wo) {
    walk_tile<kLengths>(a, ki, static_cast<int64_t>(e) * ki.slices + place, ki.parts,
              (ki.slices - place + ki.parts - 1) / ki.parts, xa, partials,
              [&]() {
                stage_finish(xa, x, ki.width, x_ahead);
                __syncthreads();
              },
              [&](int ridx, float res, int64_t slice) {
                const int where = static_cast<int>(slice - static_cast<int64_t>(e) * ki.slices) * 64 +
                                  (threadIdx.x & 63);
                write_tagged_placed(ht, ridx, where, res, tag);
              });
  } else {
    // a.lane_parts workgroups share a slice of wo, each with its part of the
    // lanes (rows): the others do nothing in its walk
    const int part = (place - ki.parts) / a.lane_parts;
    const int lanes_of = (place - ki.parts) % a.lane_parts;
    const bool active = static_cast<int>((threadIdx.x & 63) * a.lane_parts) >> 6 == lanes_of;
    uint16_t *y = a.y + static_cast<int64_t>(t) * a.ldy;
    // (a test that overstates the wait looks for a tag that nobody writes)
    const unsigned long long want = a.wi_expect == ki.parts ? tag : tag + 1;
    walk_tile<kLengths>(a, ko, static_cast<int64_t>(e) * ko.slices + part, ko.parts,
              (ko.slices - part + ko.parts - 1) / ko.parts, xa, partials,
              [&]() {
                await_tagged_placed(a, ko, ht,
                                    ki.row_idx + static_cast<int64_t>(e) * ki.slices * 64,
                                    ki.slices * 64, want, xa);
              },
              [&](int ridx, float res, int64_t) { write_row(y, ridx, res, kStore); }, active);
  }
  if (threadIdx.x == 0) leave_tagged(a.ctrl, gridDim.x);
}
__global__ __launch_bounds__(kMaxThreads) __attribute__((aligned(65536)))
void moe_prepared_tagged_split_kernel(PreparedArgs a) { tagged_split<kAlike>(a); }
template <Lengths kLengths>
__global__ __launch_bounds__(kMaxThreads) void moe_prepared_uneven_split_kernel(PreparedArgs a) { tagged_split<kLengths>(a); }

// For the batches too small to occupy the GPU with a wavefront per slice: built
// for latency.  `split` wavefronts share a slice (split_begin / split_run) and
// all of a wavefront's loads leave before anything waits.  With no more tiles
// than compute units every workgroup runs one tile; beyond that the grid is
// persistent.  Tiles are taken by ticket like in the streaming kernel, so a wo
// tile's wait for its token's wi tiles ends for the same reason.
__global__ __launch_bounds__(kMaxThreads) void moe_prepared_small_kernel(PreparedArgs a) {
  extern __shared__ __align__(16) uint32_t lds[];
  __shared__ int s_ticket;
  uint32_t *xa = lds;
  const bool dynamic = a.ctrl != nullptr;
  const int n_all = a.tokens * (a.k[0].parts + (a.kinds == 2 ? a.k[1].parts : 0));
  int static_ticket = blockIdx.x;
  int next_ticket = 0;
  if (dynamic && threadIdx.x == 0)
    next_ticket = __hip_atomic_fetch_add(&a.ctrl[0], 1, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT);
  for (;;) {
    int ticket;
    if (dynamic) {
      __syncthreads();   // the previous tile is done with s_ticket, x and the partial sums
      if (threadIdx.x == 0) s_ticket = next_ticket;
      __syncthreads();
      ticket = __builtin_amdgcn_readfirstlane(s_ticket);
    } else {
      __syncthreads();
      ticket = static_ticket;
      static_ticket += gridDim.x;
    }
    if (ticket >= n_all) break;
    const Tile tile = decode_tile(a, ticket, dynamic);
    const int kind = tile.kind, t = tile.t, e = tile.e;
    const KindArgs &k = a.k[kind];
    // the next ticket is asked for late (see the streaming kernel), and not at
    // all when every workgroup has exactly one tile
    auto fetch_next = [&]() {
      if (dynamic && threadIdx.x == 0)
        next_ticket = n_all > static_cast<int>(gridDim.x)
                          ? __hip_atomic_fetch_add(&a.ctrl[0], 1, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT)
                          : n_all;
    };
    if (a.kinds == 2 && kind == 1 && e < 0) {
      pass_through(a, k, t, tile.s_lo, tile.s_hi);
      fetch_next();
      continue;
    }
    if (e >= 0) {
      int mode;
      uint16_t *dst = tile_output(a, k, kind, t, mode);
      // the launch cuts the matrices so that a tile has at most waves / split slices
      SplitWalk walk = split_begin(a, k, e, tile.s_lo, tile.s_hi);
      await_activations(a, k, kind, t, xa);
      split_run(a, k, walk, xa, dst, mode);
    }
    fetch_next();
    if (a.kinds == 2 && kind == 0 && e >= 0) publish_h(a, t);
    if (a.kinds == 2 && kind == 1 && e >= 0) done_waiting(a, t);
  }
  if (dynamic && threadIdx.x == 0) sub1::leave_launch(a.ctrl, gridDim.x);
}

// y[t] += W x[t] for many tokens through ONE matrix (matrix 0 of the prepared
// set): a tile is (four tokens, part of the matrix), static order, persistent
// grid; the stream of a tile's slices is walked once for its four tokens.
__global__ __launch_bounds__(kMaxThreads) void matvec_group_kernel(PreparedArgs a) {
  extern __shared__ __align__(16) uint32_t lds[];
  uint32_t *xa = lds;
  const KindArgs &k = a.k[0];
  const int waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int groups = (a.tokens + kGroupTokens - 1) / kGroupTokens;
  const int n_all = groups * k.parts;
  for (int tile = blockIdx.x; tile < n_all; tile += gridDim.x) {
    const int g = tile / k.parts;
    const int part = tile - g * k.parts;
    const int s_lo = static_cast<int>(static_cast<int64_t>(k.slices) * part / k.parts);
    const int s_hi = static_cast<int>(static_cast<int64_t>(k.slices) * (part + 1) / k.parts);
    const int count = s_hi - s_lo;
    const int passes = (count + waves - 1) / waves;
    const int t0 = g * kGroupTokens;
    const int left = min(a.tokens - t0, kGroupTokens);
    int s = slice_of_pass(0, wave, waves, count);
    SliceWalk cur;
    if (s < count) cur = load_slice(a, k, s_lo + s);
    __syncthreads();   // the previous tile has read its activations
    GroupRows rows;
#pragma unroll
    for (int t = 0; t < kGroupTokens; t++)
      rows.row[t] = t < left ? a.x + static_cast<int64_t>(t0 + t) * a.ldx : nullptr;
    stage_group(xa, rows, k.width);
    __syncthreads();
    for (int pass = 0; s < count; pass++) {
      const int s_next = slice_of_pass(pass + 1, wave, waves, count);
      SliceWalk nxt;
      if (s_next < count) nxt = load_slice(a, k, s_lo + s_next);
      const GroupSums res = run_slice_group(cur, a.stream, xa, nullptr, pass, passes);
#pragma unroll
      for (int t = 0; t < kGroupTokens; t++)
        if (t < left)
          write_row(a.y + static_cast<int64_t>(t0 + t) * a.ldy, cur.ridx, res.v[t],
                    a.fresh ? kFresh : kAccumulate);
      if (s_next < count) cur = nxt;
      s = s_next;
    }
  }
}

#include "sub1_batch.h"

// ------------------------------------------------------------ host side --

// The prepare kernels read dec as the fixed dictionary's table (symbols 0..2,
// unused digits zero) and refuse any other; dec is compared in full on every
// call, with this copy of the table (512 KB a GPU, filled on its first prepare
// and held until the process ends).  Building the table on the host and fetching
// dec to compare it there, as it was done first, took 9 ms a call, two calls to
// a layer; the kernel and reading its answer back take about 20 us.
static __device__ __align__(16) int32_t fixed_dec[SUB1_DEC_WORDS];
// ... and as the walks read it: whole words, and what counting holds in LDS.
static __device__ __align__(16) uint32_t fixed_words[SUB1_DICT_ENTRIES];
static __device__ __align__(16) uint32_t fixed_counts[kCountWords];
std::mutex g_fixed_mutex;
std::vector<int> g_fixed_devices;   // where fixed_dec is filled

struct FixedTables {
  const int32_t *dec;
  const uint32_t *words, *counts;
};
int fixed_tables_of_current_device(FixedTables *out) {
  int device = 0;
  void *at_dec = nullptr, *at_words = nullptr, *at_counts = nullptr;
  HIP_TRY(hipGetDevice(&device));
  HIP_TRY(hipGetSymbolAddress(&at_dec, HIP_SYMBOL(fixed_dec)));
  HIP_TRY(hipGetSymbolAddress(&at_words, HIP_SYMBOL(fixed_words)));
  HIP_TRY(hipGetSymbolAddress(&at_counts, HIP_SYMBOL(fixed_counts)));
  std::lock_guard<std::mutex> lock(g_fixed_mutex);
  if (std::find(g_fixed_devices.begin(), g_fixed_devices.end(), device) == g_fixed_devices.end()) {
    std::vector<int32_t> table(SUB1_DEC_WORDS);
    const int rc = sub1_build_tables(table.data(), nullptr);
    if (rc) return fail(rc, "sub1_build_tables failed");
    std::vector<uint32_t> words(SUB1_DICT_ENTRIES), counts(kCountWords);
    for (int e = 0; e < SUB1_DICT_ENTRIES; e++) {
      // digit d of entry e is (dec[2e + d/14] >> (4 + 2 (d % 14))) & 3, the low nibble of
      // dec[2e] its pair count (reference sub1.py:60-72, sub1_cuda_kernel.cu:186-192)
      const uint32_t pairs = static_cast<uint32_t>(table[2 * e]) & 15u;
      uint32_t place[3] = {0, 0, 0};   // 2 digit + symbol - 1
      int n = 0;
      for (int d = 0; d < 28; d++) {
        const uint32_t t = (static_cast<uint32_t>(table[2 * e + d / 14]) >> (4 + 2 * (d % 14))) & 3u;
        if (t == 0) continue;
        if (t == 3 || n == 3 || d >= 2 * static_cast<int>(pairs))
          return fail(SUB1_ERR_INTERNAL, "dictionary entry %d is outside the form of the walks", e);
        for (int j = n; j < 3; j++) place[j] = 2u * d + t - 1;
        n++;
      }
      words[e] = pairs | static_cast<uint32_t>(n) << 4 | place[0] << 8 | place[1] << 16 | place[2] << 24;
      const uint32_t tail = n ? 2 * pairs - place[2] / 2 : 0u;
      counts[e / 2] |= (pairs | static_cast<uint32_t>(n) << 4 | place[0] / 2 << 6 | tail << 11) << (16 * (e & 1));
      counts[SUB1_DICT_ENTRIES / 2 + e / 16] |= ((place[0] & 1u) | (place[2] & 1u) << 1) << (2 * (e & 15));
    }
    HIP_TRY(hipMemcpy(at_dec, table.data(), table.size() * sizeof(int32_t), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(at_words, words.data(), words.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(at_counts, counts.data(), counts.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
    g_fixed_devices.push_back(device);
  }
  *out = {static_cast<const int32_t *>(at_dec), static_cast<const uint32_t *>(at_words),
          static_cast<const uint32_t *>(at_counts)};
  return SUB1_OK;
}

// What the prepare passes read: `kinds` groups of `count` matrices each.
struct Source {
  const int32_t *dec;
  KindSource k[2];
  int kinds, count;
  int height[2], width[2];
};

// Names the first NULL or misaligned entry of a pointer table (its contents are
// fetched for that: check_source_kernel has found that there is one).
int name_bad_pointer(const void *const *table, int count, size_t align, const char *what,
                     const char *who, hipStream_t s) {
  std::vector<const void *> host(count);
  HIP_TRY(hipMemcpyAsync(host.data(), table, sizeof(void *) * count, hipMemcpyDeviceToHost, s));
  HIP_TRY(hipStreamSynchronize(s));
  for (int i = 0; i < count; i++) {
    if (!host[i]) return fail(SUB1_ERR_NULL, "%s: %s of matrix %d is NULL", who, what, i);
    if (misaligned(host[i], align))
      return fail(SUB1_ERR_ALIGN, "%s: %s of matrix %d is not %zu-byte aligned", who, what, i, align);
  }
  return SUB1_OK;
}

// dec and the pointer tables, looked at on the GPU, which leaves what it finds in `found`
// (a device word, zero before): the launches that follow go by it.  The walk's tables
// receive the dictionary as it reads it.
int check_on_device(const Source &src, int32_t *found, WalkArgs &w, hipStream_t s) {
  FixedTables fixed;
  int rc = fixed_tables_of_current_device(&fixed);
  if (rc) return rc;
  w.table = fixed.words;
  w.count_table = fixed.counts;
  w.found = found;
  PointerTables pt{};
  pt.count = src.count;
  for (int i = 0; i < src.kinds; i++) {
    const KindSource &k = src.k[i];
    if (!k.w_comp_of) continue;
    const void *const *of[3] = {reinterpret_cast<const void *const *>(k.w_comp_of),
                                reinterpret_cast<const void *const *>(k.row_off_of),
                                reinterpret_cast<const void *const *>(k.minmax_of)};
    for (int j = 0; j < 3; j++) {
      pt.table[pt.n] = of[j];
      pt.align[pt.n++] = j == 0 ? 2 : 4;
    }
  }
  check_source_kernel<<<kCheckBlocks, 256, 0, s>>>(src.dec, fixed.dec, pt, found);
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}

// The error for what it has found.
int refuse_source(const Source &src, int found, hipStream_t s, const char *who) {
  const char *const names[3] = {"w_comp", "row_off", "ter_minmax"};
  if (found & 2)
    for (int i = 0; i < src.kinds; i++) {
      const KindSource &k = src.k[i];
      if (!k.w_comp_of) continue;
      const void *const *of[3] = {reinterpret_cast<const void *const *>(k.w_comp_of),
                                  reinterpret_cast<const void *const *>(k.row_off_of),
                                  reinterpret_cast<const void *const *>(k.minmax_of)};
      for (int j = 0; j < 3; j++) {
        const int rc = name_bad_pointer(of[j], src.count, j == 0 ? 2 : 4, names[j], who, s);
        if (rc) return rc;
      }
    }
  return fail(SUB1_ERR_SHAPE,
              "sub1_moe_prepare: dec is not the fixed dictionary; use sub1_moe_grouped");
}

int check_source(const Source &src, const char *who) {
  if (!src.dec) return fail(SUB1_ERR_NULL, "%s: NULL pointer", who);
  if (src.count < 1) return fail(SUB1_ERR_SHAPE, "%s: %d matrices", who, src.count);
  int64_t slices = 0;
  for (int i = 0; i < src.kinds; i++) {
    const KindSource &k = src.k[i];
    if (src.height[i] < 1 || src.height[i] > 65534 || src.width[i] < 1 ||
        src.width[i] > SUB1_PREPARED_MAX_WIDTH)
      return fail(SUB1_ERR_SHAPE, "%s: matrix %d x %d (height 1..65534, width 1..%d)", who,
                  src.height[i], src.width[i], SUB1_PREPARED_MAX_WIDTH);
    if (k.w_comp_of || k.row_off_of || k.minmax_of) {
      const void *const tables[3] = {k.w_comp_of, k.row_off_of, k.minmax_of};
      const char *const names[3] = {"w_comp", "row_off", "ter_minmax"};
      for (int j = 0; j < 3; j++) {
        if (!tables[j])
          return fail(SUB1_ERR_NULL, "%s: NULL table of %s pointers", who, names[j]);
        if (misaligned(tables[j], 8))
          return fail(SUB1_ERR_ALIGN, "%s: misaligned table of %s pointers", who, names[j]);
      }
    } else {
      if (!k.w_comp || !k.row_off || !k.minmax || (src.count > 1 && !k.code_base))
        return fail(SUB1_ERR_NULL, "%s: NULL pointer", who);
      if (misaligned(k.row_off, 4) || misaligned(k.minmax, 4) || misaligned(k.code_base, 8) ||
          misaligned(k.w_comp, 2))
        return fail(SUB1_ERR_ALIGN, "%s: misaligned pointer", who);
    }
    slices += static_cast<int64_t>(src.count) * ((src.height[i] + 63) / 64);
  }
  if (slices > (1 << 24)) return fail(SUB1_ERR_SHAPE, "%s: too many 64-row slices", who);
  if (misaligned(src.dec, 4)) return fail(SUB1_ERR_ALIGN, "%s: misaligned pointer", who);
  return SUB1_OK;
}

KindSource stacked(const void *w_comp, const int64_t *code_base, const int32_t *row_off,
                   const void *minmax) {
  return KindSource{static_cast<const uint16_t *>(w_comp), code_base, row_off,
                    static_cast<const uint32_t *>(minmax), nullptr, nullptr, nullptr};
}

KindSource scattered(const void *const *w_comp, const void *const *row_off,
                     const void *const *minmax) {
  return KindSource{nullptr, nullptr, nullptr, nullptr,
                    reinterpret_cast<const uint16_t *const *>(w_comp),
                    reinterpret_cast<const int32_t *const *>(row_off),
                    reinterpret_cast<const uint32_t *const *>(minmax)};
}

Source moe_source(const sub1_moe_stack *st) {
  Source src;
  src.dec = st->dec;
  src.k[0] = stacked(st->w_comp, st->wi_code_base, st->wi_row_off, st->wi_minmax);
  src.k[1] = stacked(st->w_comp, st->wo_code_base, st->wo_row_off, st->wo_minmax);
  src.kinds = 2;
  src.count = st->experts;
  src.height[0] = st->d_ff;
  src.width[0] = st->d_model;
  src.height[1] = st->d_model;
  src.width[1] = st->d_ff;
  return src;
}

Source layers_source(const sub1_moe_layers *l) {
  Source src;
  src.dec = l->dec;
  src.k[0] = scattered(l->wi_w_comp, l->wi_row_off, l->wi_minmax);
  src.k[1] = scattered(l->wo_w_comp, l->wo_row_off, l->wo_minmax);
  src.kinds = 2;
  src.count = l->experts;
  src.height[0] = l->d_ff;
  src.width[0] = l->d_model;
  src.height[1] = l->d_model;
  src.width[1] = l->d_ff;
  return src;
}

Source matrix_source(const sub1_matrix_set *ms) {
  Source src;
  src.dec = ms->dec;
  src.k[0] = stacked(ms->w_comp, ms->code_base, ms->row_off, ms->ter_minmax);
  src.k[1] = KindSource{};
  src.kinds = 1;
  src.count = ms->count;
  src.height[0] = ms->height;
  src.width[0] = ms->width;
  src.height[1] = 0;
  src.width[1] = 0;
  return src;
}

// What a prepared buffer pair holds, in the terms of the kernels.
struct Prepared {
  const void *meta;
  const void *codes;
  int64_t meta_bytes, code_bytes, total_chunks;
  int kinds, count;
  int height[2], width[2];
  int max_chunks[2];
};

// Chunks of an average slice of a kind, by what its width is of the stream.
double average_chunks(const Prepared &p, int kind) {
  double weight = 0.0;
  for (int i = 0; i < p.kinds; i++) weight += static_cast<double>((p.height[i] + 63) / 64) * p.width[i];
  return static_cast<double>(p.total_chunks) / p.count * p.width[kind] / weight;
}

// The longest slice of rows of one share of zeros has 1.2 to 1.4 times an average one's chunks (1.7 of 500
// columns with 95 %, hence the two chunks), of rows of which one in a hundred has no zeros 5 to 10 times.
// In between, rows of 90 % zeros and one in a hundred of fewer, the forms for differing lengths begin to pay at
// 2 (few tokens) to 2.8 times (whole tokens).  us, alike / differing, the longest slice 1.9 times an average one: base, 4, 60 and
// 200 tokens 12.6 / 12.4, 17.6 / 19.2, 35.6 / 38.1, c-2048 17.9 / 17.7, 51.6 / 53.3, 128 / 137; 2.4 times: 12.9 / 12.7, 19.6 / 19.9,
// 37.8 / 38.4, 18.9 / 18.7, 55.8 / 51.3, 129 / 135; 2.9 times: 13.8 / 13.2, 20.3 / 20.5, 41.5 / 39.0, 19.6 / 19.3, 63.9 / 53.0, 135 / 135.
bool is_uneven(const Prepared &p, int kind) {
  return p.max_chunks[kind] > 2.0 * average_chunks(p, kind) + 2.0;
}

struct LayoutResult {
  int64_t meta_bytes, code_bytes, total_chunks;
  int max_chunks[2];
};

// Where kind i stands in a walk's order: longer rows first.
int walk_place(const Source &src, int i) {
  return src.kinds == 2 && src.width[1] > src.width[0] ? 1 - i : i;
}

template <bool kEmit>
int launch_walk(const Source &src, const MetaLayout &m, WalkArgs &w, hipStream_t s) {
  w.kinds = src.kinds;
  w.count = src.count;
  int device = 0, cus = 0;
  HIP_TRY(hipGetDevice(&device));
  HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
  int64_t tasks = 0, groups = 0;
  for (int i = 0; i < src.kinds; i++) groups += static_cast<int64_t>(src.count) * m.k[i].slices;
  for (int i = 0; i < src.kinds; i++) {
    WalkKind &k = w.k[walk_place(src, i)];
    k.long_from = std::min(std::max(static_cast<float>(groups) / cus, kLongFromFew), kLongFromMany);
    k.source = src.k[i];
    k.height = m.k[i].height;
    k.width = m.k[i].width;
    k.slices = m.k[i].slices;
    tasks += k.tasks;
  }
  constexpr size_t lds = kEmit ? kWalkLds : kCountLds;
  HIP_TRY(sub1::allow_lds<lds>(walk_rows_kernel<kEmit>));
  walk_rows_kernel<kEmit><<<static_cast<unsigned>(std::min<int64_t>(tasks, cus)), kWalkThreads, lds, s>>>(w);
  HIP_TRY(hipGetLastError());
  if (w.long_bits) emit_long_rows_kernel<<<static_cast<unsigned>(std::min<int64_t>(tasks * kLongShares, 8 * cus)), kLongThreads, 0, s>>>(w);
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}

int prepare_layout(const Source &src, void *meta, int64_t meta_bytes, LayoutResult *out,
                   hipStream_t s, const char *who) {
  if (!meta || !out) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (misaligned(meta, 256)) return fail(SUB1_ERR_ALIGN, "%s: meta must be 256-byte aligned", who);
  const MetaLayout m = meta_layout(src.count, src.kinds, src.height, src.width);
  if (meta_bytes < m.bytes)
    return fail(SUB1_ERR_SHAPE, "%s: meta needs %lld bytes", who, static_cast<long long>(m.bytes));
  char *base = static_cast<char *>(meta);
  int32_t *status = reinterpret_cast<int32_t *>(base + m.status);
  sub1::AnswerSlot slot;
  int rc = slot.take(s, who);
  if (rc) return rc;
  zero_words_kernel<<<1, 64, 0, s>>>(status, 4);
  WalkArgs w{};
  rc = check_on_device(src, status + 3, w, s);
  if (!rc) rc = slot.launched(who);
  if (rc) return rc;
  int32_t *counts = reinterpret_cast<int32_t *>(base + m.counts);
  w.status = status;
  for (int i = 0; i < src.kinds; i++) {
    const KindMeta &k = m.k[i];
    WalkKind &wk = w.k[walk_place(src, i)];
    wk.row_len = reinterpret_cast<uint16_t *>(base + k.row_len);
    wk.tasks = (static_cast<int64_t>(src.count) * k.height + 63) / 64;
  }
  rc = launch_walk<false>(src, m, w, s);
  if (rc) return rc;
  HIP_TRY(sub1::allow_lds<order_rows_lds(65534)>(order_rows_kernel));
  int64_t slice0 = 0;
  OrderArgs o{};
  o.status = status;
  o.found = status + 3;
  size_t lds = 0;
  for (int i = 0; i < src.kinds; i++) {
    const KindMeta &k = m.k[i];
    o.k[i] = {src.k[i],
              reinterpret_cast<const uint16_t *>(base + k.row_len),
              reinterpret_cast<uint16_t *>(base + k.row_idx),
              reinterpret_cast<uint32_t *>(base + k.minmax),
              reinterpret_cast<uint16_t *>(base + k.slice_len),
              counts + slice0,
              k.height,
              k.slices};
    lds = std::max(lds, order_rows_lds(k.height));
    slice0 += static_cast<int64_t>(src.count) * k.slices;
  }
  order_rows_kernel<<<dim3(static_cast<unsigned>(src.count), static_cast<unsigned>(src.kinds)), kOrderThreads,
                      lds, s>>>(o);
  scan_counts_kernel<<<1, sub1::kScanThreads, 0, s>>>(counts, static_cast<int>(slice0), status, slot.answer());
  HIP_TRY(hipGetLastError());
  int32_t host[5] = {0, 0, 0, 0, 0};   // the total, bad rows, the longest slices, what was found
  rc = slot.wait(s, 5, host, who);
  if (rc) return rc;
  if (host[4]) return refuse_source(src, host[4], s, who);
  const int32_t total = host[0];
  if (host[1])
    return fail(SUB1_ERR_SHAPE, "%s: the codes of %d rows do not cover the width", who, host[1]);
  if (total < 0) return fail(SUB1_ERR_SHAPE, "%s: stream too large", who);
  out->meta_bytes = m.bytes;
  out->total_chunks = total;
  // the entry stream, then one 128-byte checkpoint entry per group of chunks
  out->code_bytes = static_cast<int64_t>(total) * 512 +
                    (static_cast<int64_t>(total) / kGroupChunks + slice0 + 1) * 128;
  out->max_chunks[0] = host[2];
  out->max_chunks[1] = host[3];
  return SUB1_OK;
}

int prepare_codes(const Source &src, const Prepared &p, hipStream_t s, const char *who) {
  if (!p.meta || !p.codes) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (misaligned(p.meta, 256) || misaligned(p.codes, 256))
    return fail(SUB1_ERR_ALIGN, "%s: buffers must be 256-byte aligned", who);
  const MetaLayout m = meta_layout(src.count, src.kinds, src.height, src.width);
  char *base = static_cast<char *>(const_cast<void *>(p.meta));
  int64_t nslices = 0;
  for (int i = 0; i < src.kinds; i++) nslices += static_cast<int64_t>(src.count) * m.k[i].slices;
  if (p.total_chunks < 0 || p.meta_bytes < m.bytes ||
      p.code_bytes < p.total_chunks * 512 + (p.total_chunks / kGroupChunks + nslices + 1) * 128)
    return fail(SUB1_ERR_SHAPE, "%s: buffers smaller than the layout needs", who);
  sub1::AnswerSlot slot;
  int rc = slot.take(s, who);
  if (rc) return rc;
  int32_t *found = reinterpret_cast<int32_t *>(base + m.status) + 3;
  zero_words_kernel<<<1, 64, 0, s>>>(found, kStatusWords - 3);
  WalkArgs w{};
  rc = check_on_device(src, found, w, s);
  if (!rc) rc = slot.launched(who);
  if (rc) return rc;
  uint2 *stream = static_cast<uint2 *>(const_cast<void *>(p.codes));
  uint16_t *ckpt = reinterpret_cast<uint16_t *>(stream + p.total_chunks * 64);
  // Some rows are long ones, if any are (or a few are, of a narrow matrix: the launch for them then finds none, 4 us).
  for (int i = 0; i < src.kinds; i++)
    if (is_uneven(p, i))
      w.long_bits = reinterpret_cast<uint32_t *>(base + m.status) + kStatusLong;
  w.stream = stream;
  w.ckpt = ckpt;
  int64_t first_slice = 0;
  for (int i = 0; i < src.kinds; i++) {
    const KindMeta &k = m.k[i];
    WalkKind &wk = w.k[walk_place(src, i)];
    wk.slice_base = reinterpret_cast<const uint32_t *>(base + k.slice_base);
    wk.slice_len = reinterpret_cast<const uint16_t *>(base + k.slice_len);
    wk.row_idx = reinterpret_cast<const uint16_t *>(base + k.row_idx);
    wk.first_slice = first_slice;
    wk.tasks = static_cast<int64_t>(src.count) * k.slices;
    first_slice += wk.tasks;
  }
  w.answer = slot.answer();
  rc = launch_walk<true>(src, m, w, s);
  if (rc) return rc;
  // the walk says what was found as it begins, and does its work behind the host's back
  int32_t bad = 0;
  rc = slot.wait(s, 1, &bad, who);
  return rc ? rc : bad ? refuse_source(src, bad, s, who) : SUB1_OK;
}

// Cut of the matrices for a batch that cannot occupy the GPU with a wavefront
// per slice.  Per projection: a workgroup takes per_wg slices (16 = no sharing)
// and waves / per_wg wavefronts share each slice, at most one per chunk group.
// The choice minimises an estimate of the kernel time in microseconds: a round
// of workgroups costs a fixed part (activations, first loads: they do not
// overlap with the previous round) plus the groups that the busiest SIMD walks
// one after the other.  Sets split and parts of every projection; returns the
// LDS bytes for partial sums, 0 if sharing nothing is estimated best (then
// nothing is changed), and the estimate in *estimate_us.
// The constants come from timing every cut of the Switch base, large and
// c-2048 layers at 1 to 64 tokens on an MI355X; the estimate ranks the cuts and
// is about 13 us below the measured time of a launch.
constexpr double kRoundFixedUs = 6.0;      // a round of workgroups before its first entry
constexpr double kGroupUs = 0.75;          // one group of 72 entries on a SIMD
constexpr double kResidentBonusUs = 8.0;   // wo workgroups already waiting when h arrives
constexpr double kLaunchUs = 13.0;         // measured launch minus estimate
size_t plan_small(PreparedArgs &a, int kinds, int tokens, int cus, int waves, size_t lds_room,
                  double *estimate_us) {
  struct Option {
    int split, parts;
    int64_t tiles;
    double round_us;
    size_t partials;
  };
  Option opt[2][5];
  int nopt[2] = {0, 0};
  for (int i = 0; i < kinds; i++) {
    const KindArgs &k = a.k[i];
    int groups_pow2 = 1;
    while (groups_pow2 < k.groups_max) groups_pow2 *= 2;
    for (int per_wg = 1; per_wg <= waves; per_wg *= 2) {
      Option o;
      o.split = waves / per_wg < groups_pow2 ? waves / per_wg : groups_pow2;
      o.partials = o.split > 1 ? static_cast<size_t>(per_wg) * k.groups_max * 256 : 0;
      if (o.partials > lds_room) continue;
      if (o.split == 1 && per_wg != waves) continue;
      o.parts = (k.slices + per_wg - 1) / per_wg;
      o.tiles = static_cast<int64_t>(tokens) * o.parts;
      const int busy = per_wg * (o.split < k.groups_max ? o.split : k.groups_max);
      const int serial = ((busy + 3) / 4) * ((k.groups_max + o.split - 1) / o.split);
      o.round_us = kRoundFixedUs + kGroupUs * serial;
      opt[i][nopt[i]++] = o;
    }
  }
  double best = 1e30;
  int pick[2] = {-1, -1};
  for (int i0 = 0; i0 < nopt[0]; i0++)
    for (int i1 = 0; i1 < (kinds == 2 ? nopt[1] : 1); i1++) {
      const Option &o0 = opt[0][i0];
      double us = std::max(1.0, static_cast<double>(o0.tiles) / cus) * o0.round_us;
      if (kinds == 2) {
        const Option &o1 = opt[1][i1];
        // wo workgroups that found a free compute unit at the start have their
        // fixed part behind them when h arrives
        const bool resident = o0.tiles + o1.tiles <= cus;
        us += std::max(1.0, static_cast<double>(o1.tiles) / cus) * o1.round_us -
              (resident ? kResidentBonusUs : 0.0);
      }
      if (us < best) {
        best = us;
        pick[0] = i0;
        pick[1] = i1;
      }
    }
  size_t partials = 0;
  for (int i = 0; i < kinds; i++)
    if (opt[i][pick[i]].partials > partials) partials = opt[i][pick[i]].partials;
  *estimate_us = best;
  if (partials == 0) return 0;
  for (int i = 0; i < kinds; i++) {
    a.k[i].split = opt[i][pick[i]].split;
    a.k[i].parts = opt[i][pick[i]].parts;
  }
  return partials;
}

// Passes a workgroup needs for a tile of `slices` slices (a pass = one slice per
// wavefront); a last pass of at most half the wavefronts is shared out between
// all of them by chunk groups and costs a fraction of one.
double tile_passes(int slices, int waves, int groups_max) {
  const int rest = slices % waves;
  double passes = slices / waves;
  if (rest > 0) {
    int split = 1;
    if (rest * 2 <= waves)
      while (split * 2 * rest <= waves && split * 2 <= groups_max) split *= 2;
    passes += split > 1 ? 1.0 / split + 0.1 : 1.0;
  }
  return passes;
}

// The time, in units of a full pass (16 wavefronts, a slice each), that a
// workgroup of `waves` wavefronts needs for `slices` slices: whole passes, then
// the rest either as a pass of its own or, if it is at most half the
// wavefronts, shared out `split` ways.  A pass with few wavefronts in it is
// faster than a full one (less contention for LDS), down to about 0.3 of it.
double part_passes(int slices, int waves, int groups_max) {
  const int rest = slices % waves;
  double passes = slices / waves;
  if (rest > 0) {
    int split = 1;
    if (rest * 2 <= waves) split = std::max(1, std::min(waves / rest, groups_max));
    passes += std::max(static_cast<double>(rest * split) / waves, 0.3) / split;
  }
  return passes;
}

// Launch of the prepared kernels.  kinds == 2: y = wo(relu(wi x)) per token,
// workspace required; kinds == 1: y += W x per token, no workspace.
// `piece`: 0 for a caller's launch; 1 and 2 for the two pieces when a launch is
// split in two (a piece is not split again).
int launch_prepared(const Prepared &p, const int32_t *token_matrix, const void *x, int64_t ldx,
                    void *y, int64_t ldy, int tokens, void *workspace, int64_t workspace_bytes,
                    hipStream_t s, const char *who, int piece = 0, bool may_allocate = true, bool fresh = false) {
  if (!p.meta || !p.codes || !x || !y) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (p.kinds == 2 && !token_matrix) return fail(SUB1_ERR_NULL, "%s: NULL token_expert", who);
  if (tokens < 0 || tokens > (1 << 20))
    return fail(SUB1_ERR_SHAPE, "%s: tokens %d outside 0..2^20", who, tokens);
  if (ldx < p.width[0] || ldy < (p.kinds == 2 ? p.height[1] : p.height[0]))
    return fail(SUB1_ERR_SHAPE, "%s: token strides smaller than the rows", who);
  if (misaligned(p.meta, 256) || misaligned(p.codes, 256) || misaligned(token_matrix, 4) ||
      misaligned(x, 2) || misaligned(y, 2))
    return fail(SUB1_ERR_ALIGN, "%s: misaligned pointer", who);
  const int d_ff = p.kinds == 2 ? p.height[0] : 0;
  if (p.kinds == 2) {
    if (!workspace || workspace_bytes < sub1_moe_workspace_bytes(tokens, d_ff))
      return fail(SUB1_ERR_SHAPE, "%s: workspace of %lld bytes needed", who,
                  static_cast<long long>(sub1_moe_workspace_bytes(tokens, d_ff)));
    if (misaligned(workspace, 256)) return fail(SUB1_ERR_ALIGN, "%s: misaligned workspace", who);
  }
  const MetaLayout m = meta_layout(p.count, p.kinds, p.height, p.width);
  if (p.meta_bytes < m.bytes) return fail(SUB1_ERR_SHAPE, "%s: meta smaller than its layout", who);
  const char *base = static_cast<const char *>(p.meta);

  PreparedArgs a;
  a.by_ticket = 0;
  a.fresh = fresh;
  a.tagged = nullptr;
  a.lane_parts = 1;
  a.stream = static_cast<const uint2 *>(p.codes);
  a.ckpt = reinterpret_cast<const uint16_t *>(a.stream + p.total_chunks * 64);
  a.kinds = p.kinds;
  int wmax = 0;
  for (int i = 0; i < 2; i++) {
    KindArgs &ka = a.k[i];
    if (i >= p.kinds) {
      ka = a.k[0];
      ka.parts = 0;
      continue;
    }
    const KindMeta &k = m.k[i];
    ka.slice_base = reinterpret_cast<const uint32_t *>(base + k.slice_base);
    ka.slice_len = reinterpret_cast<const uint16_t *>(base + k.slice_len);
    ka.row_idx = reinterpret_cast<const uint16_t *>(base + k.row_idx);
    ka.minmax = reinterpret_cast<const uint32_t *>(base + k.minmax);
    ka.slices = k.slices;
    ka.height = k.height;
    ka.width = k.width;
    if (k.width > wmax) wmax = k.width;
  }
  // 16 wavefronts per workgroup.  A count that divides the slice counts better
  // (11 for the c-2048 shapes) leaves fewer idle wavefront slots but measured
  // 10% slower: the kernel needs the wavefronts to hide LDS latency.
  const int waves = 16;
  int device = 0, cus = 0;
  HIP_TRY(hipGetDevice(&device));
  HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
  a.token_expert = token_matrix;
  a.x = static_cast<const uint16_t *>(x);
  a.y = static_cast<uint16_t *>(y);
  a.ldx = ldx;
  a.ldy = ldy;
  a.ctrl = nullptr;
  a.h = nullptr;
  a.order = nullptr;
  a.groups = nullptr;
  if (p.kinds == 2) {
    a.ctrl = static_cast<int32_t *>(workspace);
    a.h = reinterpret_cast<uint16_t *>(sub1::h_base(workspace, workspace_bytes, tokens, d_ff));
  }
  a.tokens = tokens;
  a.experts = p.count;
  a.xdwords = activation_dwords(wmax);
  a.hdwords = 0;
  a.tail_room = 0;
  a.wait_ticks = sub1::wait_limit_ticks();
  {
    const int rc = sub1::fault_words(&a.sticky, may_allocate);
    if (rc) return rc;
  }
  constexpr size_t lds_limit = sub1::kMostLds;
  const size_t lds_base = static_cast<size_t>(a.xdwords) * 4;
  if (lds_base > lds_limit) return fail(SUB1_ERR_SHAPE, "%s: width %d does not fit LDS", who, wmax);
  // Tiles.  Whole matrices when the tokens alone keep every compute unit busy;
  // otherwise each matrix is cut into parts, down to one slice per wavefront
  // (the persistent kernel).  When even that leaves compute units idle (a
  // handful of tokens), the other kernel runs: a workgroup takes fewer slices
  // (8, 4, 2 or 1) and the wavefronts this frees share the slices, each
  // starting from a position checkpoint.  plan_small picks the cut by estimate.
  const int want = (cus + tokens - 1) / tokens;   // tiles per token and projection
  int64_t first_slice = 0;
  bool idle_units = false, uneven = false;
  for (int i = 0; i < p.kinds; i++) {
    KindArgs &k = a.k[i];
    k.first_slice = first_slice;
    first_slice += static_cast<int64_t>(p.count) * k.slices;
    k.groups_max = (p.max_chunks[i] + kGroupChunks - 1) / kGroupChunks;
    k.split = 1;
    k.tail_split = 0;
    uneven = uneven || is_uneven(p, i);
    const int max_parts = (k.slices + waves - 1) / waves;
    if (want > max_parts) idle_units = true;
    // Parts per matrix for the streaming kernel: the count that needs the fewest
    // passes of a workgroup per compute unit (a pass = one slice per wavefront;
    // a last pass of at most 8 slices is shared out between the wavefronts and
    // costs a fraction of one).
    double best = 1e30;
    for (int parts = 1; parts <= max_parts; parts++) {
      const int per_tile = (k.slices + parts - 1) / parts;
      const int64_t rounds = (static_cast<int64_t>(tokens) * parts + cus - 1) / cus;
      // a quarter of a pass per tile for staging its activations
      const double cost = rounds * (tile_passes(per_tile, waves, k.groups_max) + 0.25);
      if (cost < best - 1e-9) {
        best = cost;
        k.parts = parts;
      }
    }
  }
  // Many tokens through one matrix: four tokens per walk of the stream, once
  // such tiles (four tokens x 16 slices at least) can occupy half the compute
  // units; below that the per-token kernels, which can cut a matrix finer, are
  // faster (measured on the Switch shapes: 1.9x faster at 568 tokens, 2.3x at
  // 2048, break-even between 50 and 400 tokens depending on the shape).
  const int groups = (tokens + kGroupTokens - 1) / kGroupTokens;
  const int group_parts = (a.k[0].slices + waves - 1) / waves;
  const bool by_groups = p.kinds == 1 && !token_matrix &&
                   static_cast<int64_t>(groups) * group_parts * 2 >= cus;
  if (by_groups) {
    KindArgs &k = a.k[0];
    const int max_parts = group_parts;
    double best = 1e30;
    for (int parts = 1; parts <= max_parts; parts++) {
      const int per_tile = (k.slices + parts - 1) / parts;
      const int64_t rounds = (static_cast<int64_t>(groups) * parts + cus - 1) / cus;
      const double cost = rounds * ((per_tile + waves - 1) / waves + 0.25);
      if (cost < best - 1e-9) {
        best = cost;
        k.parts = parts;
      }
    }
    const int64_t tiles = static_cast<int64_t>(groups) * k.parts;
    HIP_TRY(sub1::allow_lds<lds_limit>(matvec_group_kernel));
    sub1::note_kernel("matvec_group_kernel");
    matvec_group_kernel<<<static_cast<unsigned>(tiles < cus ? tiles : cus), 64 * waves, lds_base,
                          s>>>(a);
    HIP_TRY(hipGetLastError());
    return SUB1_OK;
  }
  const int stream_parts[2] = {a.k[0].parts, a.k[1].parts};   // plan_small may change them
  size_t lds_partials = 0;
  double small_us = 0.0;
  if (idle_units)
    lds_partials = plan_small(a, p.kinds, tokens, cus, waves, lds_limit - lds_base, &small_us);
  const bool small = lds_partials != 0;
  int64_t tiles = 0;
  for (int i = 0; i < p.kinds; i++) tiles += static_cast<int64_t>(tokens) * a.k[i].parts;
  if (tiles > INT32_MAX - (1 << 20)) return fail(SUB1_ERR_SHAPE, "%s: too many tiles", who);
  // Whole tokens per workgroup with h in LDS (the fused kernel), or the matrices
  // cut into tiles?  By estimate, in microseconds, from measurements on the
  // Switch shapes.  One token on one compute unit takes about 8 us + entries /
  // 23400 per us; the fused kernel takes that per round of workgroups (1.94
  // times that with two workgroups of 8 wavefronts per compute unit).  The cut
  // versions pay about 8 us per launch and, per round of tiles of a projection,
  // 3 us for staging plus the tile's passes, a pass of 16 slices weighing in the
  // token's time by its share of the chunks; where wavefronts share slices
  // (plan_small) their own estimate + 13 us if that is less.
  const size_t lds_fused = (static_cast<size_t>(activation_dwords(a.k[0].width)) +
                            activation_dwords(a.k[1].width)) * 4;
  bool fused = false;
  int fused_per_cu = 1;
  int shared_parts = 0, shared_room = 0;
  // Partial sums of a shared pass (walk_tile), in groups of 64 lanes: those of half the wavefronts'
  // slices; of slices whose lengths differ what LDS has room for, the longest one's at least.
  const auto tail_groups = [&](size_t room_bytes) {
    const int room = static_cast<int>(room_bytes / 256);
    int longest = 0;
    for (int i = 0; i < p.kinds; i++) longest = std::max(longest, a.k[i].groups_max);
    const int most = (uneven ? waves : waves / 2) * longest;
    return most <= room ? most : uneven && longest <= room ? room : 0;
  };
  if (p.kinds == 2 && lds_fused <= lds_limit) {
    const double token_us = 8.0 + static_cast<double>(p.total_chunks) * (64.0 * kFields) /
                                      p.count / 23400.0;
    auto fused_estimate = [&](int64_t n, int *per_cu) {
      const int64_t rounds16 = (n + cus - 1) / cus, rounds8 = (n + 2 * cus - 1) / (2 * cus);
      *per_cu = 1;
      if (2 * lds_fused <= lds_limit && 1.94 * rounds8 < rounds16) {
        *per_cu = 2;
        return 1.94 * rounds8 * token_us;
      }
      return rounds16 * token_us;
    };
    const double fused_us = fused_estimate(tokens, &fused_per_cu);
    double weight = 0.0;
    for (int i = 0; i < 2; i++) weight += static_cast<double>(a.k[i].slices) * p.max_chunks[i];
    double cut_us = 8.0;
    for (int i = 0; i < 2; i++) {
      const KindArgs &k = a.k[i];
      const int per_tile = (k.slices + stream_parts[i] - 1) / stream_parts[i];
      const int64_t rounds = (static_cast<int64_t>(tokens) * stream_parts[i] + cus - 1) / cus;
      const double pass_us = (token_us - 8.0) * waves * p.max_chunks[i] / weight;
      cut_us += rounds * (tile_passes(per_tile, waves, k.groups_max) * pass_us + 3.0);
    }
    cut_us *= 1.05;   // the estimate ran 5 to 8% low where tiles take several rounds
    if (small) cut_us = std::min(cut_us, small_us + kLaunchUs);
    // Up to a token per compute unit: several workgroups per token, each in
    // both projections (moe_prepared_shared_kernel), one workgroup per compute
    // unit at a time.  Up to half a token per unit that is all of them at once;
    // up to one, two rounds can still beat whole tokens on half the units (they
    // do for the c-2048 shapes at 129 to 170 tokens).  Fixed costs of 8 us plus
    // staging (by the widths), the walk of the largest share, and what more
    // workgroups cost in dispatch and in waiting for each other; measured on
    // the Switch shapes it is the fastest form from 2 tokens (1 for the smaller
    // shapes) to half the compute units: 1.1 to 1.5 times faster than cutting
    // by projection.
    shared_room = tail_groups(lds_limit - lds_base);
    auto shared_estimate = [&](int64_t n, int *best_parts) {
      double best_us = 1e30;
      *best_parts = 0;
      if (n > cus || !shared_room) return best_us;
      for (int parts = 2; parts <= 64 && n * parts <= 2 * cus; parts++) {
        // beyond one workgroup per compute unit the rest of the grid starts as
        // the first tokens finish: two rounds, measured 7% above twice one
        const int rounds = n * parts > cus ? 2 : 1;
        double task = (a.k[0].width + a.k[1].width) / 2700.0 + 0.03 * parts;
        for (int i = 0; i < 2; i++) {
          const KindArgs &k = a.k[i];
          const double pass_us = (token_us - 8.0) * waves * p.max_chunks[i] / weight;
          double passes = part_passes((k.slices + parts - 1) / parts, waves, k.groups_max);
          // the slices of the longest one's length, if the others have a seventh: a wavefront walks each of a
          // workgroup's if there is no room for the partial sums of all of them
          const double longest = std::max((k.slices * average_chunks(p, i) / p.max_chunks[i] - k.slices / 7.0) * 7 / 6, 1.0);
          if (uneven && std::ceil(longest / parts) * k.groups_max > shared_room) passes = std::max(passes, 1.0);
          task += passes * pass_us + 0.5;
        }
        const double us = 8.0 + (rounds == 2 ? 2.24 : 1.0) * task + 0.008 * n * parts;
        if (us < best_us) {
          best_us = us;
          *best_parts = parts;
        }
      }
      return best_us;
    };
    int best_parts = 0;
    const double shared_us = shared_estimate(tokens, &best_parts);
    if (best_parts && shared_us < cut_us && shared_us < fused_us) shared_parts = best_parts;
    // More than a token per compute unit, and a last round of whole tokens that
    // would be mostly empty: whole rounds as they are, the rest as shared
    // tokens in a launch of its own (300 tokens on 256 units: 256 whole and 44
    // shared instead of cut tiles or two rounds; measured 5 to 25% faster just
    // above a whole number of rounds).  The second launch is taken as 6 us, and
    // the split must promise 7%: the estimates are no better than that.  Not
    // where tokens are grouped by expert, which wants them all in one launch.
    if (piece == 0 && tokens > cus && tokens % cus != 0 &&
        !(tokens >= 4 * static_cast<int64_t>(p.count) && tokens >= 4 * cus)) {
      const int whole = tokens / cus * cus;
      int unused = 0, rest_parts = 0;
      const double split_us = fused_estimate(whole, &unused) +
                              shared_estimate(tokens - whole, &rest_parts) + 6.0;
      if (rest_parts && split_us < 0.93 * std::min(cut_us, fused_us)) {
        const uint16_t *xs = static_cast<const uint16_t *>(x);
        uint16_t *ys = static_cast<uint16_t *>(y);
        const int rc = launch_prepared(p, token_matrix, xs, ldx, ys, ldy, whole, workspace,
                                       workspace_bytes, s, who, 1, may_allocate);
        if (rc) return rc;
        return launch_prepared(p, token_matrix + whole, xs + static_cast<int64_t>(whole) * ldx, ldx,
                               ys + static_cast<int64_t>(whole) * ldy, ldy, tokens - whole,
                               workspace, workspace_bytes, s, who, 2, may_allocate);
      }
    }
    if (!shared_parts && fused_us < cut_us) {
      fused = true;
      for (int i = 0; i < 2; i++) {
        a.k[i].parts = 1;
        a.k[i].split = 1;
      }
    }
  }
  if (shared_parts) {
    for (int i = 0; i < 2; i++) {
      a.k[i].parts = shared_parts;
      a.k[i].split = 1;
    }
    a.tail_room = shared_room;
    a.wi_expect = a.k[0].parts + sub1::expect_extra();
    a.by_ticket = static_cast<int64_t>(tokens) * shared_parts > cus;
    const size_t lds_shared = lds_base + static_cast<size_t>(a.tail_room) * 256;
    // (sharing all of a few slices needs no choice, which is 0.4 us, nor code for others)
    const auto lengths = [&](int i) {
      const int most = (a.k[i].slices + a.k[i].parts - 1) / a.k[i].parts;
      return !uneven ? kAlike : all_shared(most, waves, a.k[i].groups_max, a.tail_room) ? kFew : kDiffer;
    };
    const auto lengths_of_both = [&]() { return std::max(lengths(0), lengths(1)); };
    // A token or two: h goes from wi to wo by tag (every workgroup of wo reads
    // all of it, eight bytes an entry: for small grids only).  One token, and
    // two where wo's rows are long (eight groups of chunks and more: the c-2048
    // shapes), give wo workgroups of its own, as many as give every wavefront at
    // most one group of chunks, so that all of wo's stream is in registers before
    // h is there (two tokens through the shorter rows of the base and large
    // shapes measured 11.4 and 12.4 us that way against 11.5 and 11.8).
    if (tokens <= sub1::kTaggedTokens && 64 * waves == kMaxThreads) {
      const KindArgs &ko = a.k[1];
      const int per_wg = std::max(1, waves / std::max(1, ko.groups_max));
      const int wo_parts = (ko.slices + per_wg - 1) / per_wg;
      // One token: two workgroups share each slice of wo by lanes, 32 rows each.
      // The walk of a slice's 9 to 14 wavefronts is bound by the one LDS they
      // gather from, and a gather of 32 lanes takes the LDS one pass instead of
      // two (c-2048: 12.3 -> 11.9 us; in four parts, and for two tokens, the
      // larger grid costs more than the walk gains: 12.6, and 12.9 -> 13.4).
      const int lane_parts = tokens == 1 ? 2 : 1;
      const bool own_wo = (tokens == 1 || ko.groups_max >= 8) &&
                          static_cast<int64_t>(tokens) * (shared_parts + wo_parts * lane_parts) <= cus;
      if (own_wo || static_cast<int64_t>(tokens) * shared_parts <= 64) {
        a.tagged = reinterpret_cast<unsigned long long *>(a.ctrl + sub1::kCtrlTagged);
        if (own_wo) {
          a.k[1].parts = wo_parts;
          // wi's workgroups wait for nobody, so the more of them the shorter their
          // walks: up to a slice each, within two thirds of the compute units
          // that wo leaves a token (one token through a c-2048 expert: 96 instead
          // of 48 workgroups 12.7 -> 12.4 us; two tokens, 63 each instead of 24:
          // 13.8 -> 12.8; with all units taken two tokens measured 13.4)
          a.lane_parts = lane_parts;
          shared_parts = std::max(shared_parts,
                                  std::min(a.k[0].slices, (cus / tokens - wo_parts * lane_parts) * 2 / 3));
          a.k[0].parts = shared_parts;
          a.wi_expect = a.k[0].parts + sub1::expect_extra();
          const Lengths both = lengths_of_both();
          void (*const split)(PreparedArgs) = both == kAlike ? moe_prepared_tagged_split_kernel
                                              : both == kFew ? moe_prepared_uneven_split_kernel<kFew>
                                                             : moe_prepared_uneven_split_kernel<kDiffer>;
          HIP_TRY(sub1::allow_lds<lds_limit>(split));
          sub1::note_kernel(both == kAlike ? "moe_prepared_tagged_split_kernel"
                            : both == kFew ? "moe_prepared_uneven_split_kernel<kFew>"
                                           : "moe_prepared_uneven_split_kernel<kDiffer>");
          split<<<tokens * (shared_parts + wo_parts * lane_parts), 64 * waves, lds_shared, s>>>(a);
        } else {
          const Lengths both = lengths_of_both();
          void (*const tagged)(PreparedArgs) = both == kAlike ? moe_prepared_tagged_kernel<kAlike>
                                               : both == kFew ? moe_prepared_tagged_kernel<kFew>
                                                              : moe_prepared_tagged_kernel<kDiffer>;
          HIP_TRY(sub1::allow_lds<lds_limit>(tagged));
          sub1::note_kernel(both == kAlike ? "moe_prepared_tagged_kernel"
                            : both == kFew ? "moe_prepared_tagged_kernel<kFew>"
                                           : "moe_prepared_tagged_kernel<kDiffer>");
          tagged<<<tokens * shared_parts, 64 * waves, lds_shared, s>>>(a);
        }
        HIP_TRY(hipGetLastError());
        return SUB1_OK;
      }
    }
    void (*const shared)(PreparedArgs) = !uneven                    ? moe_prepared_shared_kernel<kAlike, kAlike>
                                         : lengths_of_both() == kFew ? moe_prepared_shared_kernel<kFew, kFew>
                                         : lengths(1) == kFew        ? moe_prepared_shared_kernel<kDiffer, kFew>
                                                                     : moe_prepared_shared_kernel<kDiffer, kDiffer>;
    HIP_TRY(sub1::allow_lds<lds_limit>(shared));
    sub1::note_kernel(!uneven                     ? "moe_prepared_shared_kernel"
                      : lengths_of_both() == kFew ? "moe_prepared_shared_kernel<kFew, kFew>"
                      : lengths(1) == kFew        ? "moe_prepared_shared_kernel<kDiffer, kFew>"
                                                  : "moe_prepared_shared_kernel<kDiffer, kDiffer>");
    shared<<<tokens * shared_parts, 64 * waves, lds_shared, s>>>(a);
    HIP_TRY(hipGetLastError());
    return SUB1_OK;
  }
  if (fused) {
    a.xdwords = activation_dwords(a.k[0].width);
    a.hdwords = activation_dwords(a.k[1].width);
    // Several tokens per expert: three or four tokens of one expert walk its
    // streams together (measured on the Switch shapes: nothing to gain below
    // four tokens per expert and four per compute unit, 1.1 to 1.3 times faster
    // at 8 to 16 per expert, 1.7 to 1.95 at 32 to 64).  The tables of the
    // grouping go where the other kernels keep h (this one keeps it in LDS).
    const int64_t table_ints = 4 * (static_cast<int64_t>(p.count) + 1);
    const int64_t order_ints = (tokens + 1) / 2 * 2;
    const int64_t group_bytes = (table_ints + order_ints) * 4 + static_cast<int64_t>(tokens) * 8;
    const bool grouped = tokens >= 4 * static_cast<int64_t>(p.count) && tokens >= 4 * cus &&
                         group_bytes <= static_cast<int64_t>(tokens) * d_ff * 2;
    // wo's last pass: with at most half the wavefronts busy, the idle ones take
    // groups of those slices (partial sums go where x was)
    KindArgs &ko = a.k[1];
    // Two workgroups of 8 wavefronts per compute unit, where two fit LDS and it
    // costs no round of workgroups more (568 tokens are three rounds of
    // workgroups of 16 but two, each twice as long, of workgroups of 8): one's
    // barriers between the phases of a token fall into the other's work
    // (measured 3% faster than one of 16 on 2048 tokens).
    // (Where lengths differ, one if two leave no room for the partial sums of a long slice.)
    const bool by_length = uneven && !grouped && tail_groups(lds_limit - lds_fused) > 0;
    const int per_cu = by_length && tail_groups(lds_limit / fused_per_cu - lds_fused) == 0 ? 1 : fused_per_cu;
    const int fw = waves / per_cu;   // wavefronts per workgroup
    const int rest = ko.slices % fw;
    if (rest > 0 && rest * 2 <= fw && ko.groups_max > 1) {
      int split = 1;
      while (split * 2 * rest <= fw && split * 2 <= ko.groups_max) split *= 2;
      // a partial sum per group of chunks and lane, four with grouped tokens
      const size_t partials = static_cast<size_t>(rest) * ko.groups_max * (grouped ? 1024 : 256);
      if (split > 1 && partials <= static_cast<size_t>(a.xdwords) * 4) ko.tail_split = split;
    }
    // a stream larger than the last-level cache (256 MB), swept by at least a
    // token per compute unit: the chunks are loaded as read-once data
    const bool once = !grouped && p.total_chunks * 512 > (256ll << 20);
    // where lengths differ the longest slices are shared by length, with partial sums behind h
    if (by_length) {
      a.tail_room = tail_groups(lds_limit / per_cu - lds_fused);
      const size_t lds_uneven = lds_fused + static_cast<size_t>(a.tail_room) * 256;
      HIP_TRY(sub1::allow_lds<lds_limit>(moe_prepared_fused_kernel<false, false, true>));
      sub1::note_kernel("moe_prepared_fused_kernel<false, false, true>");
      moe_prepared_fused_kernel<false, false, true>
          <<<tokens < cus * per_cu ? tokens : cus * per_cu, 64 * fw, lds_uneven, s>>>(a);
      HIP_TRY(hipGetLastError());
      return SUB1_OK;
    }
    HIP_TRY(sub1::allow_lds<lds_limit>(grouped ? moe_prepared_fused_kernel<true, false>
                                       : once  ? moe_prepared_fused_kernel<false, true>
                                               : moe_prepared_fused_kernel<false, false>));
    if (grouped) {
      int32_t *tab = reinterpret_cast<int32_t *>(a.h);
      int32_t *order = tab + table_ints;
      int2 *groups = reinterpret_cast<int2 *>(order + order_ints);
      group_tokens_kernel<<<1, 1024, 0, s>>>(token_matrix, tokens, p.count, tab, order, groups,
                                              a.ctrl);
      a.order = order;
      a.groups = groups;
    }
    const int grid = tokens < cus * per_cu ? tokens : cus * per_cu;
    sub1::note_kernel(grouped ? "moe_prepared_fused_kernel<true, false>"
                      : once  ? "moe_prepared_fused_kernel<false, true>"
                              : "moe_prepared_fused_kernel<false, false>");
    if (grouped)
      moe_prepared_fused_kernel<true, false><<<grid, 64 * fw, lds_fused, s>>>(a);
    else if (once)
      moe_prepared_fused_kernel<false, true><<<grid, 64 * fw, lds_fused, s>>>(a);
    else
      moe_prepared_fused_kernel<false, false><<<grid, 64 * fw, lds_fused, s>>>(a);
    HIP_TRY(hipGetLastError());
    return SUB1_OK;
  }
  // the persistent kernel shares out a tile's short last pass: room for the
  // partial sums of up to half the wavefronts' slices
  size_t lds_tail = 0;
  a.tail_room = 0;
  if (!small) {
    a.tail_room = tail_groups(lds_limit - lds_base);
    lds_tail = static_cast<size_t>(a.tail_room) * 256;
  }
  uneven = uneven && a.tail_room;
  const size_t lds = lds_base + lds_partials + lds_tail;
  a.wi_expect = a.k[0].parts + sub1::expect_extra();
  // Batches too small to occupy the GPU with a wavefront per slice go to the
  // latency kernel, everything else to the persistent one; either way at most
  // a workgroup per compute unit (16 wavefronts of 72 to 80 registers each).
  HIP_TRY(sub1::allow_lds<lds_limit>(small ? moe_prepared_small_kernel
                                     : uneven ? moe_prepared_kernel<kDiffer>
                                              : moe_prepared_kernel<kAlike>));
  if (small) {
    const int64_t grid = tiles < cus ? tiles : cus;
    sub1::note_kernel("moe_prepared_small_kernel");
    moe_prepared_small_kernel<<<static_cast<unsigned>(grid), 64 * waves, lds, s>>>(a);
  } else {
    const int64_t grid = tiles < cus ? tiles : cus;
    sub1::note_kernel(uneven ? "moe_prepared_kernel<kDiffer>" : "moe_prepared_kernel");
    if (uneven)
      moe_prepared_kernel<kDiffer><<<static_cast<unsigned>(grid), 64 * waves, lds, s>>>(a);
    else
      moe_prepared_kernel<kAlike><<<static_cast<unsigned>(grid), 64 * waves, lds, s>>>(a);
  }
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}

// ---- batches on the matrix cores (sub1_batch.h) ----

int batch_piece(int tokens) {
  const int pieces = (tokens + kBatchPiece - 1) / kBatchPiece;
  return (tokens + pieces - 1) / pieces;
}

// Steps of a product: x has its columns in their own order, h in the order of wi's slices.
int product_steps(const Prepared &p, int kind) {
  return kind ? steps_of_slices((p.height[0] + 63) / 64) : steps_of(p.width[0]);
}

// How a product's slices are given to workgroups.
struct BatchPlan {
  int per_group, parts;
  bool table_in_lds;
  size_t lds;
};

constexpr size_t kBatchLds = sub1::kMostLds;

// LDS holds the codes of `fit` slices beside a table: with room for three and more, workgroups
// of up to four wavefronts, one to a SIMD; for two, of up to eight; for one, of twelve.  (128 base
// experts on 4096 tokens: wi 52 us with four wavefronts of a slice each, 60 with two to each
// of two slices, 62 with eight slices; 40 c-2048 experts on 700, wo, whose codes take 98 KB, with 4, 8, 12 and 16
// wavefronts: 205, 166, 162 and 165 for the call.)  Wavefronts share a slice as long as
// each gets a group of chunks, the least that one can expand, and take slices of their
// own beyond that (c-2048 wi by 1, 2 and 4 to a slice: 208, 181, 166 us) - but not where a
// compute unit would then hold fewer than twelve wavefronts, as it does of rows with few entries,
// whose slices are short but whose codes take LDS as any: more of them share a slice then, the
// ones without a group of chunks for its multiplying alone (95 % zeros, sharing by chunks alone:
// 128 base experts on 4096 tokens 166 us against 128) - nor where small workgroups with a table each
// leave room for too few: then one holds all the slices that fit (base wo by one slice of four
// wavefronts, two of those to a unit, 82 us, by one of eight 67, by three of four 65) - if that divides
// the slices and four wavefronts are enough for one; else two workgroups of one slice and eight wavefronts
// share the unit (28 layers of 9 to 33 slices, rows of 3072 to 3152 columns, 9 to 64 tokens an expert: by
// three of four 1.02 to 1.17 times the time where 3 does not divide the slices, so that the last
// workgroup of an expert has places empty, 0.98 to 1.12 where it does; 50 experts of 2000 x 3100, 88 %
// zeros 200 us and 182).
//
// Where two slices fit beside one table and two workgroups with a table each do not (wo of about
// 4500 to 4730 columns), one workgroup of 16 wavefronts takes both (58 experts of 1000 x 4600, 92 % zeros,
// 9 and 64 tokens an expert: by one slice of twelve 104 and 177 us, by two of eight 87 and 158) - unless
// one slice is much longer than the others, which the other one's wavefronts then wait for, and the layer
// has not two for every compute unit (12 experts of 1500 x 4650, shares of zeros that differ from row
// to row, 72 and 79 us; 58 of 1000 x 4600 155 and 142).  Where two slices fit only without a table (up to
// about 5050), the table stays in global memory for two workgroups of a slice, if the layer has two for
// every compute unit, no slice is much longer, one long chain of looks into it, and the entries are few
// (55 experts of 1000 x 4800, 92 % zeros 172 and 150 us, 80 % 206 and 195, 70 % 210 and 227, differing
// shares 226 and 232; 20 experts of 1000 x 5030, 85 % 63 and 67).  A table that does not fit beside a single slice, of rows of more than
// 9000 columns, stays there too.
bool plan_batch(const Prepared &p, int kind, size_t lds_limit, BatchPlan *out) {
  const int slices[2] = {(p.height[0] + 63) / 64, (p.height[1] + 63) / 64};
  const double chunks = average_chunks(p, kind);
  const size_t code_bytes = slice_code_bytes(product_steps(p, kind));
  // (wi needs no table)
  const size_t wanted = kind ? table_bytes(p.width[kind]) : 0;
  const bool even = p.max_chunks[kind] <= 2.0 * chunks, few = chunks * kFields <= 0.25 * p.width[kind];
  const bool many = static_cast<int64_t>(p.count) * slices[kind] >= 2 * 256;
  const bool pair = 2 * code_bytes <= lds_limit;
  out->table_in_lds = code_bytes + wanted <= lds_limit &&
                      !(pair && 2 * code_bytes + wanted > lds_limit && even && few && many);
  const size_t table = out->table_in_lds ? wanted : 0;
  if (code_bytes + table > lds_limit) return false;
  const int fit = static_cast<int>((lds_limit - table) / code_bytes);
  if (fit == 2 && 2 * (code_bytes + table) > lds_limit && slices[kind] > 1 && (even || many)) {
    out->per_group = 2;
    out->parts = 8;
    out->lds = 2 * code_bytes + table;
    return true;
  }
  int waves = fit >= 3 ? 4 : fit == 2 ? 8 : 12;
  for (int parts = 1;; parts *= 2) {
    if (parts > waves) parts = waves;
    if (parts < waves && parts * kGroupChunks < 0.75 * chunks) continue;
    int per_group = std::min(waves / parts, slices[kind]);
    for (; per_group > 0; per_group--) {
      const size_t sums = parts > 1 ? static_cast<size_t>(2 * per_group * parts) * 4096 : 0;
      out->lds = std::max(per_group * code_bytes + table, sums);
      if (out->lds <= lds_limit) break;
    }
    if (per_group == 0) return false;
    out->per_group = per_group;
    out->parts = parts;
    if (static_cast<int>(lds_limit / out->lds) * per_group * parts >= 12) return true;
    if (parts == waves) {
      if (waves == 12) return true;
      if (waves == 4 && (slices[kind] % fit || waves * kGroupChunks < 0.75 * chunks) && 2 * (code_bytes + table) <= lds_limit) {
        out->per_group = 1;
        out->parts = 8;
        out->lds = std::max(code_bytes + table, static_cast<size_t>(2 * 8) * 4096);
        return true;
      }
      waves = 12;   // and look on from as many parts
      parts /= 2;
    }
  }
}

bool batch_takes(const Prepared &p) {
  BatchPlan plan;
  const size_t lds_fused = (static_cast<size_t>(activation_dwords(p.width[0])) + activation_dwords(p.width[1])) * 4;
  return p.count <= kBatchMaxExperts && lds_fused <= kBatchLds && plan_batch(p, 0, kBatchLds, &plan) &&
         plan_batch(p, 1, kBatchLds, &plan);
}

// The scratch memory of a piece, arrays back to back, 256-byte aligned.
struct BatchLayout {
  int64_t totals, slots, spoiled, block_expert, chunks;
  int64_t x, h;        // operands
  int64_t tables;      // where LDS has no room for them
  int64_t bytes;
  int max_blocks, max_chunks;
};

BatchLayout batch_layout(const Prepared &p, int tokens) {
  BatchLayout b;
  const int64_t hit = std::min(tokens, p.count);
  // every bucket's tokens (the experts hit, and one of tokens without an expert) fill
  // all of their blocks but the last
  b.max_blocks = static_cast<int>((tokens + (kBlockTokens - 1) * (hit + 1)) / kBlockTokens);
  b.max_chunks = static_cast<int>((b.max_blocks + (kChunkBlocks - 1) * hit) / kChunkBlocks);
  int64_t off = 0;
  auto take = [&](int64_t bytes) {
    const int64_t o = off;
    off += align256(bytes);
    return o;
  };
  const int64_t blocks = b.max_blocks, slots = blocks * kBlockTokens;
  b.totals = take(kTotalWords * 4);
  b.slots = take(slots * 4);
  b.spoiled = take(slots * 4);
  b.block_expert = take(blocks * 4);
  b.chunks = take((static_cast<int64_t>(b.max_chunks) + 7) / 8 * 8 * 16);
  b.x = take(blocks * product_steps(p, 0) * 1024);
  b.h = take(blocks * product_steps(p, 1) * 1024);
  BatchPlan plan;
  b.tables = off;
  if (plan_batch(p, 1, kBatchLds, &plan) && !plan.table_in_lds)
    take(static_cast<int64_t>(p.count) * physical_columns(p.width[1]) * 2);
  b.bytes = off;
  return b;
}

// Blocks of `per` that an expert's tokens fill, on average, where their number is spread
// about `each` as independent tokens spread it (the k-th block is begun by more than k * per).
double blocks_on_average(double each, int per) {
  double blocks = 0.0;
  for (int k = 0;; k++) {
    const double begun = 0.5 * std::erfc((per * k + 0.5 - each) / std::sqrt(2.0 * each));
    blocks += begun;
    if (per * k > each && begun < 1e-3) return blocks;
  }
}

// Whether the matrix cores are the faster way for `tokens` tokens, by estimates in microseconds
// fitted to both at 8 to 128 tokens an expert through 8 to 128 experts of the three Switch shapes
// and of three odd ones, with 80 to 95 % zeros (168 launches).  Here, for every piece of a batch,
// which expands every expert that it hits: 35 and, per million weights, 0.29 times the entries
// of a weight for every 64 of an expert's tokens, 0.08 for every 32 (within 11 %, root mean
// square; on the 1300 below 11 % low on average, within 13 %).  Walking: a compute unit takes
// token_us = 8 + entries / 23400 for a token and, where launch_prepared groups tokens by expert,
// 7 + 1.85 (token_us - 8) for up to four, in whole rounds.  The matrix cores must promise 5 %: of those
// launches that leaves none on the slower way, and 18 where they would have been faster, by up to 44 %.
// Of 1300 others (130 layers of 4 to 300 experts, Switch shapes and odd ones, 80 to 95 % zeros or shares that
// differ from row to row, 8 to 48 tokens an expert) 3 go the slower way, by 3 % at most, and 137 walk that
// would be faster here, 90 of them by more than 10 % and one by 98 %: few experts or uneven rows, whose walking
// is estimated low (a quarter on average; 38 us for 140 tokens through 7 uneven large experts, which take
// 125, and 68 here).  A piece with less than 8 tokens an expert never goes there.  (Pricing one pass over
// the experts for a batch that runs in pieces, as it was done first, sent 32 768 tokens through 2048 base
// experts this way: 5862 us, walking takes 1735.)
bool batch_pays(const Prepared &p, int tokens, int cus) {
  const int piece = batch_piece(tokens), pieces = (tokens + piece - 1) / piece;
  if (piece < 8 * static_cast<int64_t>(p.count) || !batch_takes(p)) return false;
  const double each = static_cast<double>(piece) / p.count;
  const double weights = 2e-6 * p.count * p.height[0] * p.width[0];
  const double entries = 1e-6 * p.total_chunks * (64.0 * kFields);
  const double by_chunks = blocks_on_average(each, kChunkBlocks * kBlockTokens) * 0.29 * entries;
  const double by_blocks = blocks_on_average(each, kBlockTokens) * 0.08 * weights;
  const double batch_us = pieces * (35.0 + 256.0 / cus * (by_chunks + by_blocks));
  const double walk_us = 1e6 * entries / p.count / 23400.0;   // of a token, besides its 8 us
  const bool grouped = tokens >= 4 * static_cast<int64_t>(p.count) && tokens >= 4 * cus;
  const double rounds = (0.25 * tokens + 0.375 * p.count) / cus;
  const double other_us = grouped ? 14.0 + std::ceil(rounds) * (7.0 + 1.85 * walk_us)
                                  : static_cast<double>(tokens) / cus * (8.0 + walk_us);
  return 1.05 * batch_us < other_us;
}

int launch_batch(const Prepared &p, const int32_t *token_expert, const uint16_t *x, uint16_t *y, int tokens,
                 int32_t *ctrl, char *scratch, hipStream_t s, const char *who) {
  const BatchLayout b = batch_layout(p, tokens);
  const MetaLayout m = meta_layout(p.count, p.kinds, p.height, p.width);
  const char *meta = static_cast<const char *>(p.meta);
  int32_t *totals = reinterpret_cast<int32_t *>(scratch + b.totals);
  int32_t *slots = reinterpret_cast<int32_t *>(scratch + b.slots);
  int32_t *spoiled = reinterpret_cast<int32_t *>(scratch + b.spoiled);
  int32_t *block_expert = reinterpret_cast<int32_t *>(scratch + b.block_expert);
  int4 *chunks = reinterpret_cast<int4 *>(scratch + b.chunks);
  u32x4 *xs = reinterpret_cast<u32x4 *>(scratch + b.x), *hs = reinterpret_cast<u32x4 *>(scratch + b.h);
  const int d_model = p.width[0], d_ff = p.height[0];
  const bool aligned = d_model % 8 == 0 && !misaligned(x, 16);

  // workgroups that share a block's tokens: as many as leave each thread a step, within two to a unit
  unsigned shares = 1;
  while (shares < 4 && steps_of(d_model) > 32 * static_cast<int>(shares) && 2 * shares * b.max_blocks <= 2 * 256) shares *= 2;
  pack_blocks_kernel<<<dim3(b.max_blocks, shares), kMaxThreads, static_cast<size_t>(p.count + 1) * 4, s>>>(
      token_expert, x, y, d_model, d_model, d_model, aligned, tokens, p.count, slots, spoiled, block_expert, chunks,
      totals, ctrl, xs);
  PreparedArgs a = {};
  a.stream = static_cast<const uint2 *>(p.codes);
  a.ckpt = reinterpret_cast<const uint16_t *>(a.stream + p.total_chunks * 64);
  int64_t first_slice = 0;
  for (int i = 0; i < 2; i++) {
    const KindMeta &k = m.k[i];
    KindArgs &ka = a.k[i];
    ka.slice_base = reinterpret_cast<const uint32_t *>(meta + k.slice_base);
    ka.slice_len = reinterpret_cast<const uint16_t *>(meta + k.slice_len);
    ka.row_idx = reinterpret_cast<const uint16_t *>(meta + k.row_idx);
    ka.minmax = reinterpret_cast<const uint32_t *>(meta + k.minmax);
    ka.slices = k.slices;
    ka.height = k.height;
    ka.width = k.width;
    ka.first_slice = first_slice;
    first_slice += static_cast<int64_t>(p.count) * k.slices;
  }
  for (int i = 0; i < 2; i++) {
    BatchPlan plan;
    if (!plan_batch(p, i, kBatchLds, &plan)) return fail(SUB1_ERR_SHAPE, "%s: widths too large", who);
    BatchArgs b_args = {};
    b_args.stream = a.stream;
    b_args.ckpt = a.ckpt;
    b_args.k = a.k[i];
    b_args.in = i ? hs : xs;
    if (i == 0) {
      b_args.h = hs;
      b_args.h_steps = product_steps(p, 1);
      b_args.wo_minmax = a.k[1].minmax;
      b_args.wo_rows = a.k[1].slices * 64;
    } else {
      b_args.order = a.k[0].row_idx;
      b_args.order_rows = a.k[0].slices * 64;
      b_args.y = y;
      b_args.ldy = d_model;
    }
    b_args.slots = slots;
    b_args.chunks = chunks;
    b_args.totals = totals;
    b_args.spoiled = spoiled;
    b_args.steps = product_steps(p, i);
    b_args.parts = plan.parts;
    b_args.per_group = plan.per_group;
    b_args.slice_groups = (a.k[i].slices + plan.per_group - 1) / plan.per_group;
    if (i == 1 && !plan.table_in_lds) {
      uint16_t *tables = reinterpret_cast<uint16_t *>(scratch + b.tables);
      b_args.tables = tables;
      fill_tables_kernel<<<p.count, kMaxThreads, 0, s>>>(b_args, tables);
    }
    void (*const product)(BatchArgs) = i == 0               ? batch_product_kernel<true, false>
                                       : plan.table_in_lds ? batch_product_kernel<false, true>
                                                           : batch_product_kernel<false, false>;
    HIP_TRY(sub1::allow_lds<kBatchLds>(product));
    product<<<static_cast<unsigned>((b.max_chunks + 7) / 8 * 8 * b_args.slice_groups),
              64 * plan.per_group * plan.parts, plan.lds, s>>>(b_args);
  }
  // what they leave to the walking kernels
  a.x = x;
  a.y = y;
  a.ldx = a.ldy = d_model;
  a.xdwords = activation_dwords(d_model);
  a.hdwords = activation_dwords(d_ff);
  HIP_TRY(sub1::allow_lds<kBatchLds>(walk_spoiled_kernel));
  const size_t lds = static_cast<size_t>(a.xdwords + a.hdwords) * 4;
  walk_spoiled_kernel<<<std::min(tokens, 256), kMaxThreads, lds, s>>>(a, slots, spoiled, block_expert, totals);
  HIP_TRY(hipGetLastError());
  sub1::note_kernel("batch_product_kernel");
  return SUB1_OK;
}

// The symbols of matrix `index` of kind `kind`, read back from the stream.
int decode_prepared(const Prepared &p, int kind, int index, void *tern_out, hipStream_t s,
                    const char *who) {
  if (!p.meta || !p.codes || !tern_out) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (kind < 0 || kind >= p.kinds || index < 0 || index >= p.count)
    return fail(SUB1_ERR_SHAPE, "%s: no matrix %d of kind %d", who, index, kind);
  if (misaligned(p.meta, 256) || misaligned(p.codes, 256))
    return fail(SUB1_ERR_ALIGN, "%s: misaligned pointer", who);
  const MetaLayout m = meta_layout(p.count, p.kinds, p.height, p.width);
  if (p.meta_bytes < m.bytes) return fail(SUB1_ERR_SHAPE, "%s: meta smaller than its layout", who);
  const char *base = static_cast<const char *>(p.meta);
  const KindMeta &k = m.k[kind];
  const int64_t n = static_cast<int64_t>(k.height) * k.width;
  uint8_t *out = static_cast<uint8_t *>(tern_out);
  fill_bytes_kernel<<<static_cast<unsigned>((n + 255) / 256), 256, 0, s>>>(out, n, 0);
  decode_entries_kernel<<<(k.slices * 64 + 255) / 256, 256, 0, s>>>(
      static_cast<const uint2 *>(p.codes), reinterpret_cast<const uint32_t *>(base + k.slice_base),
      reinterpret_cast<const uint16_t *>(base + k.slice_len),
      reinterpret_cast<const uint16_t *>(base + k.row_idx), out,
      static_cast<int64_t>(index) * k.slices, k.slices, k.width);
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}

int check_moe_stack(const sub1_moe_stack *st, const char *who) {
  if (!st) return fail(SUB1_ERR_NULL, "%s: NULL stack", who);
  if (st->experts < 1 || st->d_model < 1 || st->d_ff < 1)
    return fail(SUB1_ERR_SHAPE, "%s: experts %d d_model %d d_ff %d", who, st->experts,
                st->d_model, st->d_ff);
  return check_source(moe_source(st), who);
}

int check_moe_layers(const sub1_moe_layers *l, const char *who) {
  if (!l) return fail(SUB1_ERR_NULL, "%s: NULL layers", who);
  if (l->experts < 1 || l->d_model < 1 || l->d_ff < 1)
    return fail(SUB1_ERR_SHAPE, "%s: experts %d d_model %d d_ff %d", who, l->experts, l->d_model,
                l->d_ff);
  return check_source(layers_source(l), who);
}

void fill_moe_prepared(sub1_moe_prepared *out, void *meta, const LayoutResult &r, int experts,
                       int d_model, int d_ff) {
  out->meta = meta;
  out->codes = nullptr;
  out->meta_bytes = r.meta_bytes;
  out->code_bytes = r.code_bytes;
  out->total_chunks = r.total_chunks;
  out->experts = experts;
  out->d_model = d_model;
  out->d_ff = d_ff;
  out->max_chunks[0] = r.max_chunks[0];
  out->max_chunks[1] = r.max_chunks[1];
}

int check_matrix_set(const sub1_matrix_set *ms, const char *who) {
  if (!ms) return fail(SUB1_ERR_NULL, "%s: NULL matrix set", who);
  return check_source(matrix_source(ms), who);
}

}  // namespace

// ================================================================ C ABI =====


extern "C" int64_t sub1_moe_prepared_meta_bytes(int experts, int d_model, int d_ff) {
  if (experts < 1 || d_model < 1 || d_ff < 1) return 0;
  return moe_layout(experts, d_model, d_ff).bytes;
}

extern "C" int sub1_moe_prepare_layout(const sub1_moe_stack *st, void *meta, int64_t meta_bytes,
                                       sub1_moe_prepared *out, void *stream) {
  int rc = check_moe_stack(st, "sub1_moe_prepare_layout");
  if (rc) return rc;
  if (!out) return fail(SUB1_ERR_NULL, "sub1_moe_prepare_layout: NULL argument");
  LayoutResult r;
  rc = prepare_layout(moe_source(st), meta, meta_bytes, &r, static_cast<hipStream_t>(stream),
                      "sub1_moe_prepare_layout");
  if (rc) return rc;
  fill_moe_prepared(out, meta, r, st->experts, st->d_model, st->d_ff);
  return SUB1_OK;
}

extern "C" int sub1_moe_prepare_layout_from_layers(const sub1_moe_layers *layers, void *meta,
                                                   int64_t meta_bytes, sub1_moe_prepared *out,
                                                   void *stream) {
  const char *who = "sub1_moe_prepare_layout_from_layers";
  hipStream_t s = static_cast<hipStream_t>(stream);
  int rc = check_moe_layers(layers, who);
  if (rc) return rc;
  if (!out) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  LayoutResult r;
  rc = prepare_layout(layers_source(layers), meta, meta_bytes, &r, s, who);
  if (rc) return rc;
  fill_moe_prepared(out, meta, r, layers->experts, layers->d_model, layers->d_ff);
  return SUB1_OK;
}

extern "C" int sub1_moe_prepared_entry_counts(const sub1_moe_prepared *p, int64_t *walked,
                                              int64_t *in_rows, void *stream) {
  const char *who = "sub1_moe_prepared_entry_counts";
  if (!p || !walked || !in_rows) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (!p->meta) return fail(SUB1_ERR_NULL, "%s: NULL meta", who);
  const MetaLayout m = moe_layout(p->experts, p->d_model, p->d_ff);
  if (p->meta_bytes < m.bytes) return fail(SUB1_ERR_SHAPE, "%s: meta smaller than its layout", who);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const char *base = static_cast<const char *>(p->meta);
  *walked = *in_rows = 0;
  for (int i = 0; i < 2; i++) {
    const KindMeta &k = m.k[i];
    const int64_t nslices = static_cast<int64_t>(p->experts) * k.slices;
    const int64_t nrows = static_cast<int64_t>(p->experts) * k.height;
    std::vector<uint16_t> slice_len(nslices), row_len(nrows);
    HIP_TRY(hipMemcpyAsync(slice_len.data(), base + k.slice_len, nslices * 2, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipMemcpyAsync(row_len.data(), base + k.row_len, nrows * 2, hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    // the rows that pad a matrix's last slice are walked like any other lane
    for (int64_t g = 0; g < nslices; g++) *walked += 64ll * slice_len[g];
    for (int64_t g = 0; g < nrows; g++) *in_rows += row_len[g];
  }
  return SUB1_OK;
}

namespace {
Prepared from_moe(const sub1_moe_prepared *p) {
  Prepared q;
  q.meta = p->meta;
  q.codes = p->codes;
  q.meta_bytes = p->meta_bytes;
  q.code_bytes = p->code_bytes;
  q.total_chunks = p->total_chunks;
  q.kinds = 2;
  q.count = p->experts;
  q.height[0] = p->d_ff;
  q.width[0] = p->d_model;
  q.height[1] = p->d_model;
  q.width[1] = p->d_ff;
  q.max_chunks[0] = p->max_chunks[0];
  q.max_chunks[1] = p->max_chunks[1];
  return q;
}

Prepared from_matrix(const sub1_matrix_prepared *p) {
  Prepared q;
  q.meta = p->meta;
  q.codes = p->codes;
  q.meta_bytes = p->meta_bytes;
  q.code_bytes = p->code_bytes;
  q.total_chunks = p->total_chunks;
  q.kinds = 1;
  q.count = p->count;
  q.height[0] = p->height;
  q.width[0] = p->width;
  q.height[1] = 0;
  q.width[1] = 0;
  q.max_chunks[0] = p->max_chunks;
  q.max_chunks[1] = 0;
  return q;
}

bool bad_dims(int count, int h, int w) {
  return count < 1 || h < 1 || w < 1 || h > 65534 || w > SUB1_PREPARED_MAX_WIDTH;
}
}  // namespace

// ------------------------------------------------ launch without allocating --
//
// Scratch memory of sub1_moe_grouped_prepared_static: what the workspace
// argument of sub1_moe_grouped_prepared brings in (control words, then h), held
// by every GPU the library runs on until the process ends.  The name is a
// host-side stand-in, not a device address: host code uses the per-device
// address that hipGetSymbolAddress returns, never the name.
static __device__ __align__(256) unsigned char scratch[SUB1_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices] = {};   // each GPU's own copy of `scratch`

// The current device's address of the scratch array (resolved once per device,
// with that device current; no allocation).
int scratch_of_current_device(void **out) {
  int device = 0;
  HIP_TRY(hipGetDevice(&device));
  if (device < 0 || device >= kMaxDevices)
    return fail(SUB1_ERR_SHAPE, "device %d: the static scratch serves devices 0..%d", device,
                kMaxDevices - 1);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[device]) {
    void *ptr = nullptr;
    HIP_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) return fail(SUB1_ERR_HIP, "hipGetSymbolAddress returned no address for the scratch");
    g_scratch_ptr[device] = ptr;
  }
  *out = g_scratch_ptr[device];
  return SUB1_OK;
}
}  // namespace

extern "C" int sub1_init(void) {
  int32_t *sticky = nullptr;
  int rc = sub1::fault_words(&sticky, true);
  if (rc) return rc;
  void *ws = nullptr;
  return scratch_of_current_device(&ws);
}

extern "C" int sub1_moe_grouped_prepared_static(const sub1_moe_prepared *p,
                                                const int32_t *token_expert, const void *x,
                                                void *y, int tokens, void *stream) {
  const char *who = "sub1_moe_grouped_prepared_static";
  if (!p) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (tokens == 0) return SUB1_OK;
  if (bad_dims(p->experts, p->d_ff, p->d_model) || bad_dims(p->experts, p->d_model, p->d_ff))
    return fail(SUB1_ERR_SHAPE, "%s: experts %d d_model %d d_ff %d", who, p->experts, p->d_model,
                p->d_ff);
  if (tokens < 0) return fail(SUB1_ERR_SHAPE, "%s: tokens %d", who, tokens);
  // The array is split for good: control words for SUB1_STATIC_MAX_TOKENS at its
  // head, h in what follows.  Stacks of different d_ff share the array, and h of
  // one launch must never lie on words that another, larger launch counts with.
  const int64_t h_room = SUB1_STATIC_SCRATCH_BYTES - sub1::control_bytes(SUB1_STATIC_MAX_TOKENS);
  const int64_t h_bytes = static_cast<int64_t>(tokens) * p->d_ff * 2;
  if (tokens > SUB1_STATIC_MAX_TOKENS || h_bytes > h_room)
    return fail(SUB1_ERR_SHAPE,
                "%s: %d tokens of d_ff %d need %lld bytes for h, the static buffer serves up to "
                "%d tokens and %lld bytes of h; use sub1_moe_grouped_prepared with a workspace",
                who, tokens, p->d_ff, static_cast<long long>(h_bytes), SUB1_STATIC_MAX_TOKENS,
                static_cast<long long>(h_room));
  void *ws = nullptr;
  const int rc = scratch_of_current_device(&ws);
  if (rc) return rc;
  return launch_prepared(from_moe(p), token_expert, x, p->d_model, y, p->d_model, tokens, ws,
                         SUB1_STATIC_SCRATCH_BYTES, static_cast<hipStream_t>(stream), who, 0,
                         /*may_allocate=*/false);
}

extern "C" int sub1_static_scratch_pointer(void **out) {
  if (!out) return fail(SUB1_ERR_NULL, "sub1_static_scratch_pointer: NULL argument");
  return scratch_of_current_device(out);
}

extern "C" int sub1_static_scratch_reset(void *stream) {
  void *ws = nullptr;
  const int rc = scratch_of_current_device(&ws);
  if (rc) return rc;
  const int words = static_cast<int>(sub1::control_bytes(SUB1_STATIC_MAX_TOKENS) / 4);
  zero_words_kernel<<<(words + 255) / 256, 256, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<int32_t *>(ws), words);
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}

extern "C" int sub1_moe_prepare_codes(const sub1_moe_stack *st, const sub1_moe_prepared *p,
                                      void *stream) {
  int rc = check_moe_stack(st, "sub1_moe_prepare_codes");
  if (rc) return rc;
  if (!p) return fail(SUB1_ERR_NULL, "sub1_moe_prepare_codes: NULL argument");
  if (p->experts != st->experts || p->d_model != st->d_model || p->d_ff != st->d_ff)
    return fail(SUB1_ERR_SHAPE, "sub1_moe_prepare_codes: the layout belongs to another stack");
  return prepare_codes(moe_source(st), from_moe(p), static_cast<hipStream_t>(stream),
                       "sub1_moe_prepare_codes");
}

extern "C" int sub1_moe_prepare_codes_from_layers(const sub1_moe_layers *layers,
                                                  const sub1_moe_prepared *p, void *stream) {
  const char *who = "sub1_moe_prepare_codes_from_layers";
  hipStream_t s = static_cast<hipStream_t>(stream);
  int rc = check_moe_layers(layers, who);
  if (rc) return rc;
  if (!p) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (p->experts != layers->experts || p->d_model != layers->d_model || p->d_ff != layers->d_ff)
    return fail(SUB1_ERR_SHAPE, "%s: the layout belongs to other layers", who);
  return prepare_codes(layers_source(layers), from_moe(p), s, who);
}

extern "C" int sub1_moe_grouped_prepared(const sub1_moe_prepared *p, const int32_t *token_expert,
                                         const void *x, void *y, int tokens, void *workspace,
                                         int64_t workspace_bytes, void *stream) {
  if (!p) return fail(SUB1_ERR_NULL, "sub1_moe_grouped_prepared: NULL argument");
  if (tokens == 0) return SUB1_OK;
  if (bad_dims(p->experts, p->d_ff, p->d_model) || bad_dims(p->experts, p->d_model, p->d_ff))
    return fail(SUB1_ERR_SHAPE, "sub1_moe_grouped_prepared: experts %d d_model %d d_ff %d",
                p->experts, p->d_model, p->d_ff);
  return launch_prepared(from_moe(p), token_expert, x, p->d_model, y, p->d_model, tokens,
                         workspace, workspace_bytes, static_cast<hipStream_t>(stream),
                         "sub1_moe_grouped_prepared");
}

extern "C" int64_t sub1_moe_batch_scratch_bytes(const sub1_moe_prepared *p, int tokens) {
  if (!p || tokens < 1 || tokens > (1 << 20) || bad_dims(p->experts, p->d_ff, p->d_model) ||
      bad_dims(p->experts, p->d_model, p->d_ff))
    return 0;
  const Prepared q = from_moe(p);
  return batch_takes(q) ? batch_layout(q, batch_piece(tokens)).bytes : 0;
}

extern "C" int sub1_moe_batch_pays(const sub1_moe_prepared *p, int tokens) {
  if (sub1_moe_batch_scratch_bytes(p, tokens) <= 0) return 0;
  int device = 0, cus = 0;
  if (hipGetDevice(&device) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < 1)
    return 0;
  return batch_pays(from_moe(p), tokens, cus);
}

extern "C" int sub1_test_batch_plan(const sub1_moe_prepared *p, int projection, int32_t *plan) {
  const char *who = "sub1_test_batch_plan";
  if (!p || !plan) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (projection < 0 || projection > 1 || sub1_moe_batch_scratch_bytes(p, 1) <= 0)
    return fail(SUB1_ERR_SHAPE, "%s: no such form", who);
  BatchPlan b;
  if (!plan_batch(from_moe(p), projection, kBatchLds, &b)) return fail(SUB1_ERR_INTERNAL, "%s: no plan", who);
  plan[0] = b.per_group;
  plan[1] = b.parts;
  plan[2] = static_cast<int32_t>(b.lds);
  return SUB1_OK;
}

extern "C" int sub1_moe_batch_prepared(const sub1_moe_prepared *p, const int32_t *token_expert, const void *x,
                                       void *y, int tokens, void *workspace, int64_t workspace_bytes,
                                       void *scratch, int64_t scratch_bytes, void *stream) {
  const char *who = "sub1_moe_batch_prepared";
  if (!p) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (tokens == 0) return SUB1_OK;
  if (bad_dims(p->experts, p->d_ff, p->d_model) || bad_dims(p->experts, p->d_model, p->d_ff))
    return fail(SUB1_ERR_SHAPE, "%s: experts %d d_model %d d_ff %d", who, p->experts, p->d_model, p->d_ff);
  if (!p->meta || !p->codes || !token_expert || !x || !y || !workspace || !scratch)
    return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (tokens < 0 || tokens > (1 << 20)) return fail(SUB1_ERR_SHAPE, "%s: tokens %d outside 0..2^20", who, tokens);
  const Prepared q = from_moe(p);
  if (!batch_takes(q)) return fail(SUB1_ERR_SHAPE, "%s: shapes that have no such form", who);
  const int piece = batch_piece(tokens);
  if (scratch_bytes < batch_layout(q, piece).bytes || workspace_bytes < sub1_moe_workspace_bytes(piece, p->d_ff))
    return fail(SUB1_ERR_SHAPE, "%s: scratch or workspace too small", who);
  if (p->meta_bytes < moe_layout(p->experts, p->d_model, p->d_ff).bytes)
    return fail(SUB1_ERR_SHAPE, "%s: meta smaller than its layout", who);
  if (misaligned(p->meta, 256) || misaligned(p->codes, 256) || misaligned(token_expert, 4) || misaligned(x, 2) ||
      misaligned(y, 2) || misaligned(workspace, 256) || misaligned(scratch, 256))
    return fail(SUB1_ERR_ALIGN, "%s: misaligned pointer", who);
  for (int first = 0; first < tokens; first += piece) {
    const int64_t at = static_cast<int64_t>(first) * p->d_model;
    const int rc = launch_batch(q, token_expert + first, static_cast<const uint16_t *>(x) + at,
                                static_cast<uint16_t *>(y) + at, std::min(piece, tokens - first),
                                static_cast<int32_t *>(workspace), static_cast<char *>(scratch), static_cast<hipStream_t>(stream), who);
    if (rc) return rc;
  }
  return SUB1_OK;
}

extern "C" int sub1_moe_prepared_decode(const sub1_moe_prepared *p, int expert, int projection,
                                        void *tern_out, void *stream) {
  if (!p) return fail(SUB1_ERR_NULL, "sub1_moe_prepared_decode: NULL argument");
  if (bad_dims(p->experts, p->d_ff, p->d_model) || bad_dims(p->experts, p->d_model, p->d_ff))
    return fail(SUB1_ERR_SHAPE, "sub1_moe_prepared_decode: experts %d d_model %d d_ff %d",
                p->experts, p->d_model, p->d_ff);
  return decode_prepared(from_moe(p), projection, expert, tern_out,
                         static_cast<hipStream_t>(stream), "sub1_moe_prepared_decode");
}

extern "C" int64_t sub1_matrix_prepared_meta_bytes(int count, int height, int width) {
  if (count < 1 || height < 1 || width < 1) return 0;
  return matrix_layout(count, height, width).bytes;
}

extern "C" int sub1_matrix_prepare_layout(const sub1_matrix_set *ms, void *meta,
                                          int64_t meta_bytes, sub1_matrix_prepared *out,
                                          void *stream) {
  int rc = check_matrix_set(ms, "sub1_matrix_prepare_layout");
  if (rc) return rc;
  if (!out) return fail(SUB1_ERR_NULL, "sub1_matrix_prepare_layout: NULL argument");
  LayoutResult r;
  rc = prepare_layout(matrix_source(ms), meta, meta_bytes, &r, static_cast<hipStream_t>(stream),
                      "sub1_matrix_prepare_layout");
  if (rc) return rc;
  out->meta = meta;
  out->codes = nullptr;
  out->meta_bytes = r.meta_bytes;
  out->code_bytes = r.code_bytes;
  out->total_chunks = r.total_chunks;
  out->count = ms->count;
  out->height = ms->height;
  out->width = ms->width;
  out->max_chunks = r.max_chunks[0];
  return SUB1_OK;
}

extern "C" int sub1_matrix_prepare_codes(const sub1_matrix_set *ms,
                                         const sub1_matrix_prepared *p, void *stream) {
  int rc = check_matrix_set(ms, "sub1_matrix_prepare_codes");
  if (rc) return rc;
  if (!p) return fail(SUB1_ERR_NULL, "sub1_matrix_prepare_codes: NULL argument");
  if (p->count != ms->count || p->height != ms->height || p->width != ms->width)
    return fail(SUB1_ERR_SHAPE, "sub1_matrix_prepare_codes: the layout belongs to other matrices");
  return prepare_codes(matrix_source(ms), from_matrix(p), static_cast<hipStream_t>(stream),
                       "sub1_matrix_prepare_codes");
}

extern "C" int sub1_matvec_prepared(const sub1_matrix_prepared *p, const int32_t *token_matrix,
                                    const void *x, int64_t ldx, void *y, int64_t ldy,
                                    int tokens, void *stream) {
  if (!p) return fail(SUB1_ERR_NULL, "sub1_matvec_prepared: NULL argument");
  if (tokens == 0) return SUB1_OK;
  if (bad_dims(p->count, p->height, p->width))
    return fail(SUB1_ERR_SHAPE, "sub1_matvec_prepared: %d matrices of %d x %d", p->count,
                p->height, p->width);
  return launch_prepared(from_matrix(p), token_matrix, x, ldx, y, ldy, tokens, nullptr, 0,
                         static_cast<hipStream_t>(stream), "sub1_matvec_prepared");
}

extern "C" int sub1_product_prepared(const sub1_matrix_prepared *p, const void *x, int64_t ldx,
                                     void *y, int64_t ldy, int tokens, void *stream) {
  if (!p) return fail(SUB1_ERR_NULL, "sub1_product_prepared: NULL argument");
  if (tokens == 0) return SUB1_OK;
  if (bad_dims(p->count, p->height, p->width))
    return fail(SUB1_ERR_SHAPE, "sub1_product_prepared: %d matrices of %d x %d", p->count,
                p->height, p->width);
  return launch_prepared(from_matrix(p), nullptr, x, ldx, y, ldy, tokens, nullptr, 0,
                         static_cast<hipStream_t>(stream), "sub1_product_prepared", 0, true, true);
}

extern "C" int sub1_matrix_prepared_decode(const sub1_matrix_prepared *p, int matrix,
                                           void *tern_out, void *stream) {
  if (!p) return fail(SUB1_ERR_NULL, "sub1_matrix_prepared_decode: NULL argument");
  if (bad_dims(p->count, p->height, p->width))
    return fail(SUB1_ERR_SHAPE, "sub1_matrix_prepared_decode: %d matrices of %d x %d", p->count,
                p->height, p->width);
  return decode_prepared(from_matrix(p), 0, matrix, tern_out, static_cast<hipStream_t>(stream),
                         "sub1_matrix_prepared_decode");
}
