// The encoder: rows of ternary weights to dictionary codes, the longest entry at
// every place (reference sub1_cuda_kernel.cu:90-126, 211-250 and sub1.py:145-166).
//
// The reference walks the trie pair by pair, one row a thread.  The walk is a
// chain of dependent reads of a 2.4 MB table, 1040 of them for a row of 2080
// weights, and it cannot be cut: a parse that starts elsewhere in the row hardly
// ever falls in step with the true one.  For the fixed dictionary the walk is not
// needed.  Its entries are all strings of pairs with
//   * at most two non-zero symbols, up to 14 pairs,
//   * three, up to 12 pairs, and some of 13 pairs,
// so that the longest entry at a place follows from where the third and the
// fourth non-zero symbol after it stand, for all places of the row at once, and
// the entry's number from one look into a table by string.  Both tables are
// derived from the dictionary on the host, which refuses a dictionary that is not
// of this form.
//
// pack_rows_kernel (a wavefront per row) does this; pack_count_kernel walks a
// caller's trie where that is not the fixed one.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <vector>

#include "sub1_common.h"

namespace {

using sub1::fail;
using sub1::misaligned;
using sub1::wave_lds_fence;

// ------------------------------------------------ the dictionary by string --

constexpr int kMaxPairs = 14;                     // pairs of an entry
constexpr int kFreeNonzeros = 2;                  // up to so many non-zeros, every string is an entry
constexpr int kBorderPairs = 13;                  // with one more: every string shorter than this,
constexpr int kBorderStrings = 2600 * 8;          // and some of this length, C(26, 3) places x 2^3 symbols

// A string of `pairs` pairs: bit d of nz set where symbol d is not zero, of mx
// where it is 2.  Strings with k non-zeros, shorter ones first, by the places of
// the non-zeros (colexicographic), then by their symbols.
__host__ __device__ inline int combinations2(int n) { return n * (n - 1) / 2; }
__host__ __device__ inline int combinations3(int n) { return n * (n - 1) * (n - 2) / 6; }

__host__ __device__ inline int string_places(uint32_t nz, uint32_t mx, int k) {
  int places = 0, symbols = 0;
  for (int j = 1; j <= k; j++) {
    const int d = __builtin_ctz(nz);
    nz &= nz - 1;
    places += j == 1 ? d : j == 2 ? combinations2(d) : combinations3(d);
    symbols |= static_cast<int>((mx >> d) & 1u) << (j - 1);
  }
  return (places << k) + symbols;
}

constexpr int kFirst1 = kMaxPairs;                               // one string of zeros per length
constexpr int kFirst2 = kFirst1 + 2 * kMaxPairs * (kMaxPairs + 1);
constexpr int kFirst3 = kFirst2 + 4 * (kMaxPairs * (kMaxPairs + 1) * (4 * kMaxPairs - 1) / 6);
constexpr int kStrings = kFirst3 + 8 * (kBorderPairs * kBorderPairs * (kBorderPairs * kBorderPairs - 1) / 3);
__host__ __device__ inline int string_index(uint32_t nz, uint32_t mx, int pairs) {
  const int k = __builtin_popcount(nz), m = pairs - 1;
  if (k == 0) return m;
  // strings of fewer pairs: sums over l of 2 C(2l, 1), 4 C(2l, 2), 8 C(2l, 3)
  const int first = k == 1   ? kFirst1 + 2 * m * (m + 1)
                    : k == 2 ? kFirst2 + 4 * (m * (m + 1) * (4 * m - 1) / 6)
                             : kFirst3 + 8 * (m * m * (m * m - 1) / 3);
  return first + string_places(nz, mx, k);
}

static __device__ uint16_t string_code[kStrings];
static __device__ uint32_t border_entry[kBorderStrings / 32];    // which 13-pair strings are entries
static __device__ int32_t fixed_trie[SUB1_TRIE_WORDS];

struct PackTables {
  const uint16_t *code;
  const uint32_t *border;
  const int32_t *trie;
};

std::mutex g_tables_mutex;
std::vector<int> g_tables_devices;   // where the three arrays are filled

int fill_tables(const PackTables &t, hipStream_t stream) {
  std::vector<int32_t> dec(SUB1_DEC_WORDS), trie(SUB1_TRIE_WORDS);
  int rc = sub1_build_tables(dec.data(), trie.data());
  if (rc) return fail(rc, "sub1_build_tables failed");
  std::vector<uint16_t> code(kStrings, 0);
  std::vector<uint32_t> border(kBorderStrings / 32, 0);
  int64_t short_strings = 0;   // entries below the border
  for (int e = 0; e < SUB1_DICT_ENTRIES; e++) {
    const uint32_t w[2] = {static_cast<uint32_t>(dec[2 * e]), static_cast<uint32_t>(dec[2 * e + 1])};
    const int pairs = static_cast<int>(w[0] & 15u);
    uint32_t nz = 0, mx = 0;
    for (int d = 0; d < 2 * kMaxPairs; d++) {
      const uint32_t sym = (w[d / 14] >> (4 + 2 * (d % 14))) & 3u;
      if (sym) nz |= 1u << d;
      if (sym == 2) mx |= 1u << d;
    }
    const int k = __builtin_popcount(nz);
    const bool at_border = k == kFreeNonzeros + 1 && pairs == kBorderPairs;
    if (k > kFreeNonzeros + 1 || pairs < 1 || pairs > kMaxPairs ||
        (k == kFreeNonzeros + 1 && pairs > kBorderPairs) || (nz >> 1) >> (2 * pairs - 1))
      return fail(SUB1_ERR_INTERNAL, "dictionary entry %d is outside the form of the encoder", e);
    if (at_border) {
      const int i = string_places(nz, mx, k);
      border[i / 32] |= 1u << (i % 32);
    } else {
      short_strings++;
    }
    code[string_index(nz, mx, pairs)] = static_cast<uint16_t>(e);
  }
  // every string below the border has to be an entry (they are distinct)
  if (short_strings != kStrings - kBorderStrings)
    return fail(SUB1_ERR_INTERNAL, "the dictionary lacks strings below the border");
  // A copy on a stream in a capture, or on the default one beside it, fails and spoils the
  // capture: the copies then take a stream of their own, this thread's calls checked against no
  // capture.  Only then, because that stream's hardware queue stays with the process, in which
  // the calls that wait for a word from the GPU take 1 to 3 % longer from then on.
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  HIP_TRY(hipThreadExchangeStreamCaptureMode(&mode));
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  const bool unknown = hipStreamIsCapturing(stream, &capture) != hipSuccess;   // the default stream beside a capture
  if (unknown) (void)hipGetLastError();
  const bool aside = unknown || capture != hipStreamCaptureStatusNone;
  hipStream_t s = stream;
  hipError_t e = aside ? hipStreamCreateWithFlags(&s, hipStreamNonBlocking) : hipSuccess;
  const bool own = aside && e == hipSuccess;
  const auto copy = [&](const void *to, const void *from, size_t bytes) {
    if (e == hipSuccess) e = hipMemcpyAsync(const_cast<void *>(to), from, bytes, hipMemcpyHostToDevice, s);
  };
  copy(t.code, code.data(), code.size() * 2);
  copy(t.border, border.data(), border.size() * 4);
  copy(t.trie, trie.data(), trie.size() * 4);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (own) (void)hipStreamDestroy(s);
  (void)hipThreadExchangeStreamCaptureMode(&mode);   // as it was
  return e == hipSuccess ? SUB1_OK : fail(SUB1_ERR_HIP, "filling the encoder's tables: %s", hipGetErrorString(e));
}

// The three arrays on the current device (2.7 MB a GPU, filled on the first call
// there and held until the process ends).
int tables_of_current_device(PackTables *t, hipStream_t stream) {
  int device = 0;
  void *code = nullptr, *border = nullptr, *trie = nullptr;
  HIP_TRY(hipGetDevice(&device));
  HIP_TRY(hipGetSymbolAddress(&code, HIP_SYMBOL(string_code)));
  HIP_TRY(hipGetSymbolAddress(&border, HIP_SYMBOL(border_entry)));
  HIP_TRY(hipGetSymbolAddress(&trie, HIP_SYMBOL(fixed_trie)));
  *t = {static_cast<const uint16_t *>(code), static_cast<const uint32_t *>(border),
        static_cast<const int32_t *>(trie)};
  std::lock_guard<std::mutex> lock(g_tables_mutex);
  if (std::find(g_tables_devices.begin(), g_tables_devices.end(), device) == g_tables_devices.end()) {
    const int rc = fill_tables(*t, stream);
    if (rc) return rc;
    g_tables_devices.push_back(device);
  }
  return SUB1_OK;
}

// --------------------------------------------------- rows by wavefront ------

struct PackArgs {
  int32_t *symbols;          // int32 [height, width], overwritten with the rows' codes; or
  const uint16_t *weights;   // bf16 [height, width] and
  uint16_t *codes;           // u16 [height, (width + 1) / 2], where the rows' codes go
  uint32_t *minmax;          // with weights: (min, max) of every row, as two bf16
  int32_t *row_cnt;          // [height + 1]: entry row + 1 receives the row's number of codes
  const int32_t *foreign;    // a word that is not zero where the caller's trie is not the fixed one (NULL: it is)
  PackTables tables;
  int height, width;
  int window;                // pairs of a row taken at a time
};

constexpr int kPackWaves = 4;           // of a workgroup: a row each, or one row together
constexpr int kSharedRows = 10, kSharedWidth = 2048;   // up to so many rows a compute unit, and from this width on, wavefronts share a row
constexpr int kJumpRounds = 4;          // sixteen entries at a time
constexpr int kPackWindow = 4096;       // pairs of a row in LDS at most
constexpr int kBorderLdsWords = (kBorderStrings / 32 + 3) / 4 * 4;
constexpr int kAhead = 4;               // loads of a lane that are asked for together
constexpr int kLookahead = 2 * kMaxPairs;   // symbols past a place that decide its entry

// LDS of a row: two bit planes over the window's symbols (which are not
// zero, which are 2), the pairs at which the parse has an entry and, where wavefronts share
// a row, what they tell each other, the longest entry at every pair and, twice, where
// several of them in turn lead to.
__host__ __device__ constexpr int plane_words(int window) { return (2 * window + kLookahead + 31) / 32 + 1; }
__host__ __device__ constexpr size_t pack_lds_per_row(int window, bool shared) {
  return static_cast<size_t>(2 * plane_words(window)) * 4 + (static_cast<size_t>(window) * 2 + 15) / 16 * 16 +
         (shared ? 2 * kPackWaves * sizeof(int) + (static_cast<size_t>(window) + 15) / 16 * 16 * 5 : 0);
}

__device__ __forceinline__ uint32_t plane_bits(const uint32_t *plane, int at) {
  const uint32_t lo = plane[at >> 5], hi = plane[(at >> 5) + 1];
  return __builtin_amdgcn_alignbit(hi, lo, at & 31) & ((1u << kLookahead) - 1);
}

// Eight values of a row from `at` on, as they lie in memory.  Where that would go
// past the row's end the last eight of it are read instead, so that a lane's
// loads take no branch; what was asked for is then `at - from_of(at)` places
// further up.  (Rows of fewer than eight values: those, the last one repeated.)
__device__ __forceinline__ int from_of(int at, int width) { return max(min(at, width - 8), 0); }
struct EightWeights {
  uint32_t v[4];
  EightWeights() = default;
  __device__ __forceinline__ EightWeights(const uint16_t *row, int at, int width) {
    if (width >= 8) {
      __builtin_memcpy(v, row + from_of(at, width), sizeof v);
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++)
        v[j] = row[min(2 * j, width - 1)] | static_cast<uint32_t>(row[min(2 * j + 1, width - 1)]) << 16;
    }
  }
};
struct EightSymbols {
  uint32_t v[8];
  EightSymbols() = default;
  __device__ __forceinline__ EightSymbols(const int32_t *row, int at, int width) {
    if (width >= 8) {
      __builtin_memcpy(v, row + from_of(at, width), sizeof v);
    } else {
#pragma unroll
      for (int j = 0; j < 8; j++) v[j] = static_cast<uint32_t>(row[min(j, width - 1)]);
    }
  }
};
// Bits of the eight values asked for at `at`, zero past the row's end.
__device__ __forceinline__ uint32_t eight_bits(uint32_t bits, int at, int width) {
  return at < width ? (bits >> (at - from_of(at, width))) & ((1u << min(width - at, 8)) - 1) : 0u;
}

// bf16 pairs as pairs of int16 in the order of their values (-0 below 0, NaNs
// outside the infinities); its own inverse.
typedef int16_t i16x2 __attribute__((ext_vector_type(2)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ i16x2 ordered(i16x2 v) { return v ^ ((v >> 15) & static_cast<int16_t>(0x7fff)); }
__device__ __forceinline__ int16_t ordered_one(int16_t v) { return v ^ ((v >> 15) & 0x7fff); }

// 1 in either half whose value is not the one sought (`mask` leaves the sign out
// where that is a zero).
__device__ __forceinline__ uint32_t not_equal(uint32_t pair, uint32_t mask, uint32_t sought) {
  const u16x2 d = __builtin_bit_cast(u16x2, (pair & mask) ^ sought);
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(d, u16x2{1, 1}));
}
// Four pairs of bits 0 and 16 to eight bits.
__device__ __forceinline__ uint32_t gather_bits(const uint32_t (&pair)[4]) {
  const uint32_t x = pair[0] | pair[1] << 2 | pair[2] << 4 | pair[3] << 6;
  return (x | x >> 15) & 0xffu;
}
// The even bits of the low half.
__device__ __forceinline__ uint32_t even_bits(uint32_t x) {
  x &= 0x5555u;
  x = (x | x >> 1) & 0x3333u;
  x = (x | x >> 2) & 0x0f0fu;
  return (x | x >> 4) & 0xffu;
}

template <bool kWeights>
__device__ __forceinline__ auto row_source(const uint16_t *w, const int32_t *t) {
  if constexpr (kWeights) return w; else return t;
}

// What bounds it: instructions.  A 6144 x 2080 matrix takes 31 us, of which 7.5
// find the rows' extremes (25 MB read, 5 us at the copy rate), 4 the planes (of the
// same registers, as far as they hold the row), 10 the lengths (75 vector instructions for 64 places,
// 7.5 million over the chip), 6 the way from entry to entry (a scalar read of a lane each, hidden behind
// the other five rows of a SIMD), 2.5 the codes.  The walk of the trie took 472 us after 60 for the
// symbols and 33 for the extremes in torch.  Looking border strings up only where the parse comes
// by them (in scalar code) measured 41, the lengths in LDS instead of registers 37.
//
// Few, wide rows leave a SIMD one or two wavefronts, whose latencies then show, above all that way
// (36 ns an entry).  There a workgroup's wavefronts share a row, and go from entry to entry by
// sixteens: where sixteen entries from a place lead to is found for all places at once, by going
// twice as far four times.  526 x 3775 with 80 % zeros: 26.4 -> 16.1 us, 1024 x 4096 with a hundredth
// of the rows without zeros 85 -> 29, 2080 x 6144 47 -> 40.  (Shared by four wavefronts with the way entry by entry:
// 21.9, 79 and 47; rows of fewer than 2048 weights or more of them are faster apart: 3500 x 2080 23.5
// against 29.1, 2500 x 1500 16.1 and 19.4.)
template <bool kWeights, bool kShared>
__global__ __launch_bounds__(64 * kPackWaves) void pack_rows_kernel(PackArgs a) {
  extern __shared__ uint32_t pack_lds[];
  if (a.foreign && *a.foreign) return;
  constexpr int kSharing = kShared ? kPackWaves : 1;   // wavefronts of a row
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int row = kShared ? blockIdx.x : blockIdx.x * kPackWaves + wave;
  const int sub = kShared ? wave : 0;
  const auto row_fence = [&]() {
    if (kShared)
      __syncthreads();
    else
      wave_lds_fence();
  };
  // (asked for first, and put into LDS behind the row's extremes)
  uint32_t *border = pack_lds;
  constexpr int kBorderTurns = (kBorderStrings / 32 + 64 * kPackWaves - 1) / (64 * kPackWaves);
  uint32_t border_part[kBorderTurns];
#pragma unroll
  for (int k = 0; k < kBorderTurns; k++)
    border_part[k] = a.tables.border[min(static_cast<int>(threadIdx.x) + 64 * kPackWaves * k, kBorderStrings / 32 - 1)];
  const bool mine = row < a.height;
  const int words = plane_words(a.window);
  uint32_t *nz_plane = pack_lds + kBorderLdsWords + (kShared ? 0 : wave) * (pack_lds_per_row(a.window, kShared) / 4);
  uint32_t *mx_plane = nz_plane + words;
  uint16_t *entry_at = reinterpret_cast<uint16_t *>(mx_plane + words);
  int *told = reinterpret_cast<int *>(entry_at + (a.window + 7) / 8 * 8);   // kShared
  uint8_t *longest_at = reinterpret_cast<uint8_t *>(told + 2 * kPackWaves);
  const int places = (a.window + 15) / 16 * 16;
  uint16_t *jump = reinterpret_cast<uint16_t *>(longest_at + places);
  const int64_t row_first = static_cast<int64_t>(row) * a.width;
  const uint16_t *w = kWeights ? a.weights + row_first : nullptr;
  int32_t *t = kWeights ? nullptr : a.symbols + row_first;

  // the row's smallest and largest weight, and what finds them: bits sought, under a mask
  uint32_t low = 0, high = 0, low_mask = 0, high_mask = 0;
  using Loaded = std::conditional_t<kWeights, EightWeights, EightSymbols>;
  Loaded kept[kAhead] = {};   // kWeights: the row's first ones
  if (kWeights && mine) {
    i16x2 least = {0x7fff, 0x7fff}, most = {-0x8000, -0x8000};
    constexpr int kStep = 512 * kSharing;
    for (int c0 = 8 * lane + 512 * sub; c0 - 8 * lane < a.width; c0 += kStep * kAhead) {
      EightWeights v[kAhead] = {{w, c0, a.width}, {w, c0 + kStep, a.width}, {w, c0 + 2 * kStep, a.width},
                                {w, c0 + 3 * kStep, a.width}};
      if constexpr (kWeights)
        if (c0 < kStep)
#pragma unroll
          for (int u = 0; u < kAhead; u++) kept[u] = v[u];
#pragma unroll
      for (int u = 0; u < kAhead; u++) {
        if (c0 - 8 * lane + kStep * u >= a.width) break;
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const i16x2 o = ordered(__builtin_bit_cast(i16x2, v[u].v[j]));
          least = __builtin_elementwise_min(least, o);
          most = __builtin_elementwise_max(most, o);
        }
      }
    }
    int l = min(least.x, least.y), h = max(most.x, most.y);
    for (int m = 1; m < 64; m <<= 1) {
      l = min(l, __shfl_xor(l, m, 64));
      h = max(h, __shfl_xor(h, m, 64));
    }
    if (kShared) {
      if (lane == 0) {
        told[2 * wave] = l;
        told[2 * wave + 1] = h;
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < kPackWaves; k++) {
        l = min(l, told[2 * k]);
        h = max(h, told[2 * k + 1]);
      }
      __syncthreads();
    }
    low = static_cast<uint16_t>(ordered_one(static_cast<int16_t>(l)));
    high = static_cast<uint16_t>(ordered_one(static_cast<int16_t>(h)));
    const bool nan = h > 0x7f80 || l < ordered_one(static_cast<int16_t>(0xff80));
    if (nan) low = high = 0x7fc0;   // a NaN makes both NaN, and nothing equals one
    if (lane == 0 && sub == 0) a.minmax[row] = low | high << 16;
    low_mask = low & 0x7fffu ? 0xffffffffu : 0x7fff7fffu;
    high_mask = high & 0x7fffu ? 0xffffffffu : 0x7fff7fffu;
    if (nan) low_mask = high_mask = 0;   // (x & 0) ^ 0x7fc0 is never zero
    low = (low | low << 16) & (nan ? ~0u : low_mask);
    high = (high | high << 16) & (nan ? ~0u : high_mask);
  }
#pragma unroll
  for (int k = 0; k < kBorderTurns; k++)
    border[min(static_cast<int>(threadIdx.x) + 64 * kPackWaves * k, kBorderStrings / 32 - 1)] = border_part[k];
  __syncthreads();
  if (!mine) return;

  const int pairs = (a.width + 1) / 2;
  int first = 0, out = 0;   // the window's first pair, the row's codes so far
  while (first < pairs) {
    const int here = min(pairs - first, a.window);   // pairs that may start an entry
    const int col0 = 2 * first;
    // eight symbols a lane to a byte of either plane, zeros past the row's end
    const int bytes = min(4 * words, (a.width - col0 + 7) / 8 + 8);   // with zeros to look ahead into
    constexpr int kStep = 64 * kSharing;   // bytes
    for (int b0 = lane + 64 * sub; b0 - lane < bytes; b0 += kStep * kAhead) {
      const auto *src = row_source<kWeights>(w, t);
      const int c0 = col0 + 8 * b0;
      Loaded v[kAhead];
      if (kWeights && c0 < 8 * kStep) {   // (of the first window)
#pragma unroll
        for (int u = 0; u < kAhead; u++) v[u] = kept[u];
      } else {
#pragma unroll
        for (int u = 0; u < kAhead; u++) v[u] = Loaded(src, c0 + 8 * kStep * u, a.width);
      }
#pragma unroll
      for (int u = 0; u < kAhead; u++) {
        if (b0 - lane + kStep * u >= bytes) break;
        uint32_t nz, mx;
        if constexpr (kWeights) {
          uint32_t not_mx[4], neither[4];
#pragma unroll
          for (int j = 0; j < 4; j++) {
            not_mx[j] = not_equal(v[u].v[j], high_mask, high);   // a row of one value: all 2
            neither[j] = not_mx[j] & not_equal(v[u].v[j], low_mask, low);
          }
          nz = gather_bits(neither) ^ 0xffu;
          mx = gather_bits(not_mx) ^ 0xffu;
        } else {
          uint32_t both = 0;
#pragma unroll
          for (int j = 0; j < 8; j++) both |= v[u].v[j] << (2 * j);
          nz = even_bits(both | both >> 1);
          mx = even_bits(both >> 1);
        }
        const int b = b0 + kStep * u;
        if (b < bytes) {
          const int at = col0 + 8 * b;
          reinterpret_cast<uint8_t *>(nz_plane)[b] = static_cast<uint8_t>(eight_bits(nz, at, a.width));
          reinterpret_cast<uint8_t *>(mx_plane)[b] = static_cast<uint8_t>(eight_bits(mx, at, a.width));
        }
      }
    }
    row_fence();
    // The longest entry at every pair, a lane each: up to the pair of the third
    // non-zero, or up to that of the fourth as far as entries with three reach.
    const auto longest_from = [&](int p) {
      const uint32_t nz = plane_bits(nz_plane, 2 * p);
      uint32_t rest = nz & (nz - 1);
      rest &= rest - 1;                                                        // from the third non-zero on
      const uint32_t end = 1u << kLookahead;
      const int upto2 = __builtin_ctz(rest | end) >> 1;
      const uint32_t rest3 = rest & (rest - 1);
      const int upto3 = min(__builtin_ctz(rest3 | end) >> 1, kBorderPairs);
      const int longest = min(max(upto2, upto3), pairs - first - p);
      // for every lane, so that several runs' LDS reads are in flight together: a
      // string of other than three non-zeros looks up something within the table
      const uint32_t three = (nz & ((1u << (2 * kBorderPairs)) - 1)) | 7u << (2 * kBorderPairs);
      const int i = min(string_places(three, plane_bits(mx_plane, 2 * p), kFreeNonzeros + 1), kBorderStrings - 1);
      const int entry = (border[i >> 5] >> (i & 31)) & 1u;
      const bool at_border = upto3 == kBorderPairs && upto2 < kBorderPairs && longest == kBorderPairs;
      return at_border ? kBorderPairs - 1 + entry : longest;
    };
    int n = 0, at = 0;   // entries found, the pair after the last of them
    if constexpr (kShared) {
      const int thread = threadIdx.x;
      for (int p0 = 0; p0 < here; p0 += 64 * kPackWaves) {
        const int p = p0 + thread, len = longest_from(min(p, here - 1));
        if (p < here) {
          longest_at[p] = static_cast<uint8_t>(len);
          jump[p] = static_cast<uint16_t>(p + len);
        }
      }
      __syncthreads();
      // Where two entries from a pair lead to, then four, eight, sixteen.
#pragma unroll
      for (int round = 0; round < kJumpRounds; round++) {
        const uint16_t *from = jump + (round & 1 ? places : 0);
        uint16_t *to = jump + (round & 1 ? 0 : places);
        for (int p = thread; p < here; p += 64 * kPackWaves) {
          const int q = from[p];
          to[p] = q < here ? from[q] : static_cast<uint16_t>(q);
        }
        __syncthreads();
      }
      // Every sixteenth entry, one after the other; then a thread goes from each to the next.
      uint16_t *every = jump + places;   // (the last round has left it)
      static_assert(kJumpRounds % 2 == 0 && 64 * kPackWaves << kJumpRounds >= kPackWindow, "a thread for each of these");
      if (sub == 0) {
        int steps = 0;
        for (; at < here; steps++) {
          if (lane == 0) every[steps] = static_cast<uint16_t>(at);
          at = __builtin_amdgcn_readfirstlane(jump[at]);
        }
        if (lane == 0) {
          told[0] = steps;
          told[1] = at;
        }
      }
      __syncthreads();
      const int steps = told[0];
      at = __builtin_amdgcn_readfirstlane(told[1]);
      if (thread < steps) {
        int p = every[thread], i = thread << kJumpRounds;
        for (const int end = i + (1 << kJumpRounds); i < end && p < here; i++) {
          entry_at[i] = static_cast<uint16_t>(p);
          p += longest_at[p];
        }
        if (thread == steps - 1) told[2] = i;
      }
      __syncthreads();
      n = __builtin_amdgcn_readfirstlane(told[2]);
    } else {
      // Two runs of 64 at a time, from entry to entry by scalar reads of the lengths.
      for (int p0 = 0; p0 < here; p0 += 128) {
        int len[2];
#pragma unroll
        for (int u = 0; u < 2; u++) len[u] = longest_from(min(p0 + 64 * u + lane, here - 1));
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const int limit = min(here - p0 - 64 * u, 64);
          unsigned long long starts = 0;
          int q = at - p0 - 64 * u;
          while (q < limit) {
            starts |= 1ull << q;
            q += __builtin_amdgcn_readlane(len[u], q);
          }
          at = p0 + 64 * u + q;
          if ((starts >> lane) & 1)
            entry_at[n + __popcll(starts & ((1ull << lane) - 1))] = static_cast<uint16_t>(p0 + 64 * u + lane);
          n += __popcll(starts);
        }
      }
    }
    if (!kShared) wave_lds_fence();
    for (int i0 = 64 * sub; i0 < n; i0 += 64 * kSharing * kAhead) {
      uint16_t code[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; u++) {
        const int i = i0 + 64 * kSharing * u + lane;
        if (i < n) {
          const int from = entry_at[i];
          const int len = (i + 1 < n ? entry_at[i + 1] : at) - from;
          const uint32_t mask = (1u << (2 * len)) - 1;
          const uint32_t nz = plane_bits(nz_plane, 2 * from) & mask;
          code[u] = a.tables.code[string_index(nz, plane_bits(mx_plane, 2 * from), len)];
        }
      }
#pragma unroll
      for (int u = 0; u < kAhead; u++) {
        const int i = i0 + 64 * kSharing * u + lane;
        if (i < n) {
          if (kWeights)
            a.codes[static_cast<int64_t>(row) * pairs + out + i] = code[u];
          else
            t[out + i] = code[u];   // at most as many as pairs taken: never ahead of what is still to be read
        }
      }
    }
    out += n;
    first += at;
    row_fence();
  }
  if (lane == 0 && sub == 0) a.row_cnt[row + 1] = out;
}

// ---------------------------------------------------- a caller's own trie ---

// *foreign, zero before, is set where trie is not the fixed dictionary's.
__global__ __launch_bounds__(256) void compare_trie_kernel(const int32_t *__restrict__ trie,
                                                           const int32_t *__restrict__ fixed,
                                                           int32_t *foreign) {
  const int i = 4 * (blockIdx.x * 256 + threadIdx.x);
  int32_t v[4] = {0, 0, 0, 0}, f[4] = {0, 0, 0, 0};
  if (i + 4 <= SUB1_TRIE_WORDS) {
    __builtin_memcpy(v, trie + i, 16);
    __builtin_memcpy(f, fixed + i, 16);
  } else {
    for (int j = 0; i + j < SUB1_TRIE_WORDS; j++) {
      v[j] = trie[i + j];
      f[j] = fixed[i + j];
    }
  }
  if ((v[0] ^ f[0]) | (v[1] ^ f[1]) | (v[2] ^ f[2]) | (v[3] ^ f[3])) *foreign = 1;
}

constexpr int kTrieRoot = SUB1_DICT_ENTRIES;

// A thread per row walks the trie, for a trie that is not the fixed one.
__global__ void pack_count_kernel(const int32_t *__restrict__ trie, int32_t *__restrict__ w_tern,
                                  int32_t *__restrict__ row_cnt, int height, int width) {
  if (!row_cnt[0]) return;   // the fixed trie: pack_rows_kernel has packed the rows
  int row = blockIdx.x * blockDim.x + threadIdx.x;
  if (row >= height) return;
  int32_t *w = w_tern + static_cast<int64_t>(row) * width;
  int node = kTrieRoot;
  int n = 0;
  for (int i = 0; i < width; i += 2) {
    int lo = w[i];
    int hi = i + 1 < width ? w[i + 1] : 0;
    int sym = 3 * hi + lo;
    int child = trie[9 * node + sym];
    if (child < 0) {
      // n <= i/2 < i: the slot written was already consumed
      w[n++] = node;
      child = trie[9 * kTrieRoot + sym];
    }
    node = child;
  }
  w[n++] = node;
  row_cnt[row + 1] = n;
}

__global__ void zero_word_kernel(int32_t *p) { *p = 0; }

// ------------------------------------------------ offsets and compaction ----

__global__ __launch_bounds__(sub1::kScanThreads) void row_offset_scan_kernel(int32_t *cnt, int height,
                                                                            sub1::Answer answer) {
  sub1::scan_in_place(cnt, height);
  if (!answer.words) return;
  // all offsets are in memory, for any stream to read, before the host hears of the last
  sub1::drain_stores();
  __syncthreads();
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    sub1::tell(answer, 0, cnt[height]);
  }
}

// A wavefront per row, lanes stride over the row's codes.
template <typename Code>
__global__ __launch_bounds__(256) void pack_emit_kernel(const Code *__restrict__ codes,
                                                        const int32_t *__restrict__ row_off,
                                                        uint16_t *__restrict__ w_comp, int height,
                                                        int stride) {
  int row = blockIdx.x * 4 + threadIdx.x / 64;
  if (row >= height) return;
  int lane = threadIdx.x % 64;
  int off = row_off[row];
  int n = row_off[row + 1] - off;
  const Code *src = codes + static_cast<int64_t>(row) * stride;
  for (int i = lane; i < n; i += 64) w_comp[off + i] = static_cast<uint16_t>(src[i]);
}

int check_pack_shape(const char *who, int height, int width) {
  if (height < 1 || width < 1) return fail(SUB1_ERR_SHAPE, "%s: height %d width %d", who, height, width);
  // the cumulative count is kept in int32 like the reference's row_off
  if (static_cast<int64_t>(height) * ((width + 1) / 2) > INT32_MAX)
    return fail(SUB1_ERR_SHAPE, "%s: more than 2^31 pairs in one call", who);
  return SUB1_OK;
}

template <bool kWeights>
int launch_pack_rows(PackArgs &a, hipStream_t s) {
  a.window = std::min((a.width + 1) / 2, kPackWindow);
  int device = 0, cus = 0;
  HIP_TRY(hipGetDevice(&device));
  HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
  if (a.width >= kSharedWidth && a.height <= kSharedRows * cus)
    pack_rows_kernel<kWeights, true><<<a.height, 64 * kPackWaves,
                                       kBorderLdsWords * 4 + pack_lds_per_row(a.window, true), s>>>(a);
  else
    pack_rows_kernel<kWeights, false><<<(a.height + kPackWaves - 1) / kPackWaves, 64 * kPackWaves,
                                        kBorderLdsWords * 4 + kPackWaves * pack_lds_per_row(a.window, false), s>>>(a);
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}

}  // namespace

extern "C" int sub1_pack_count(const int32_t *trie, int32_t *w_tern, int32_t *row_off,
                               int height, int width, void *stream) {
  if (!trie || !w_tern || !row_off) return fail(SUB1_ERR_NULL, "sub1_pack_count: NULL argument");
  int rc = check_pack_shape("sub1_pack_count", height, width);
  if (rc) return rc;
  if (misaligned(trie, 4) || misaligned(w_tern, 4) || misaligned(row_off, 4))
    return fail(SUB1_ERR_ALIGN, "sub1_pack_count: misaligned pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  PackArgs a{};
  rc = tables_of_current_device(&a.tables, s);
  if (rc) return rc;
  // row_off[0] is zero in the end; until then it says whose trie this is
  zero_word_kernel<<<1, 1, 0, s>>>(row_off);
  compare_trie_kernel<<<(SUB1_TRIE_WORDS / 4 + 256) / 256, 256, 0, s>>>(trie, a.tables.trie, row_off);
  a.symbols = w_tern;
  a.row_cnt = row_off;
  a.foreign = row_off;
  a.height = height;
  a.width = width;
  rc = launch_pack_rows<false>(a, s);
  if (rc) return rc;
  pack_count_kernel<<<(height + 63) / 64, 64, 0, s>>>(trie, w_tern, row_off, height, width);
  row_offset_scan_kernel<<<1, sub1::kScanThreads, 0, s>>>(row_off, height, sub1::Answer{});
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}

extern "C" int sub1_pack_emit(const int32_t *w_tern, const int32_t *row_off,
                              int16_t *w_comp, int height, int width, void *stream) {
  if (!w_tern || !row_off || !w_comp) return fail(SUB1_ERR_NULL, "sub1_pack_emit: NULL argument");
  if (height < 1 || width < 1)
    return fail(SUB1_ERR_SHAPE, "sub1_pack_emit: height %d width %d", height, width);
  if (misaligned(w_tern, 4) || misaligned(row_off, 4) || misaligned(w_comp, 2))
    return fail(SUB1_ERR_ALIGN, "sub1_pack_emit: misaligned pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  pack_emit_kernel<<<(height + 3) / 4, 256, 0, s>>>(
      w_tern, row_off, reinterpret_cast<uint16_t *>(w_comp), height, width);
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}

namespace {

int pack_weights(const void *w, uint16_t *codes, void *ter_minmax, int32_t *row_off, int32_t *total, int height,
                 int width, hipStream_t s, const char *who) {
  if (!w || !codes || !ter_minmax || !row_off) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  int rc = check_pack_shape(who, height, width);
  if (rc) return rc;
  if (misaligned(w, 2) || misaligned(codes, 2) || misaligned(ter_minmax, 4) || misaligned(row_off, 4))
    return fail(SUB1_ERR_ALIGN, "%s: misaligned pointer", who);
  sub1::AnswerSlot slot;
  if (total) {
    rc = slot.take(s, who);
    if (rc) return rc;
  }
  PackArgs a{};
  rc = tables_of_current_device(&a.tables, s);
  if (rc) return rc;
  a.weights = static_cast<const uint16_t *>(w);
  a.codes = codes;
  a.minmax = static_cast<uint32_t *>(ter_minmax);
  a.row_cnt = row_off;
  a.height = height;
  a.width = width;
  rc = launch_pack_rows<true>(a, s);
  if (rc) return rc;
  if (total) {
    rc = slot.launched(who);
    if (rc) return rc;
  }
  row_offset_scan_kernel<<<1, sub1::kScanThreads, 0, s>>>(row_off, height, slot.answer());
  HIP_TRY(hipGetLastError());
  return total ? slot.wait(s, 1, total, who) : SUB1_OK;
}

}  // namespace

extern "C" int sub1_pack_weights_count(const void *w, uint16_t *codes, void *ter_minmax,
                                       int32_t *row_off, int height, int width, void *stream) {
  return pack_weights(w, codes, ter_minmax, row_off, nullptr, height, width, static_cast<hipStream_t>(stream),
                      "sub1_pack_weights_count");
}

extern "C" int sub1_pack_weights_total(const void *w, uint16_t *codes, void *ter_minmax, int32_t *row_off,
                                       int32_t *total, int height, int width, void *stream) {
  const char *who = "sub1_pack_weights_total";
  if (!total) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  return pack_weights(w, codes, ter_minmax, row_off, total, height, width, static_cast<hipStream_t>(stream), who);
}

extern "C" int sub1_pack_weights_emit(const uint16_t *codes, const int32_t *row_off, int16_t *w_comp,
                                      int height, int width, void *stream) {
  const char *who = "sub1_pack_weights_emit";
  if (!codes || !row_off || !w_comp) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (height < 1 || width < 1) return fail(SUB1_ERR_SHAPE, "%s: height %d width %d", who, height, width);
  if (misaligned(codes, 2) || misaligned(row_off, 4) || misaligned(w_comp, 2))
    return fail(SUB1_ERR_ALIGN, "%s: misaligned pointer", who);
  pack_emit_kernel<<<(height + 3) / 4, 256, 0, static_cast<hipStream_t>(stream)>>>(
      codes, row_off, reinterpret_cast<uint16_t *>(w_comp), height, (width + 1) / 2);
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}
