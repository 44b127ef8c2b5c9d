// gfx950 kernels and C ABI of libsub1_hip on the reference's packed layout:
// the decode-fused matrix-vector product over dictionary-coded ternary
// weights, a plain decoder and the grouped expert-FFN launch that
// needs no preparation.  Written for 64-wide wavefronts.  The single product
// (matvec_wave_kernel) gives a wavefront to a row: lane j takes codeword j of
// each run of 64, a prefix sum across the lanes places it, a butterfly adds the
// lanes' sums.  The expert launch (moe_kernel) gives a lane to a group of 32
// codes of a row, whose start a prefix sum finds, or to a whole row where the
// rows of a wavefront are alike.
// Either way the work per codeword is proportional to the non-zero weights in
// it (at most three for the fixed dictionary).
//
// Reference behaviour being reproduced (not its implementation):
//   sub1_cuda_kernel.cu:129-202  Sub1MatVec       -> matvec_wave_kernel / moe_kernel
//   test.py:103-115              decompress       -> decode_kernel
//   sub1.py:306-321              expert loop      -> moe_kernel
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "sub1_common.h"

namespace sub1 {

thread_local std::string g_err;
thread_local const char *g_kernel = "";

void note_kernel(const char *name) { g_kernel = name; }

int fail(int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_err = buf;
  return code;
}

namespace {
std::mutex g_fault_mutex;
int32_t *g_fault_host = nullptr;     // pinned, mapped: kFaultWords words
int32_t *g_fault_device = nullptr;   // the same words as the GPUs address them
std::atomic<int64_t> g_wait_limit_us{250000};
std::atomic<int> g_expect_extra{0};
std::atomic<int> g_late_us{0};
std::atomic<int> g_clock_khz{0};     // rate of wall_clock64 on the device first asked
}  // namespace

int fault_words(int32_t **device_ptr, bool may_allocate) {
  std::lock_guard<std::mutex> lock(g_fault_mutex);
  if (!g_fault_host) {
    if (!may_allocate)
      return fail(SUB1_ERR_INTERNAL, "call sub1_init() once before an entry point that does not allocate");
    void *host = nullptr, *dev = nullptr;
    HIP_TRY(hipHostMalloc(&host, kFaultWords * sizeof(int32_t),
                          hipHostMallocPortable | hipHostMallocMapped));
    for (int i = 0; i < kFaultWords; i++) static_cast<int32_t *>(host)[i] = 0;
    HIP_TRY(hipHostGetDevicePointer(&dev, host, 0));
    g_fault_host = static_cast<int32_t *>(host);
    g_fault_device = static_cast<int32_t *>(dev);
  }
  *device_ptr = g_fault_device;
  return SUB1_OK;
}

bool fault_flag_host(int word) {
  std::lock_guard<std::mutex> lock(g_fault_mutex);
  return g_fault_host && *const_cast<volatile int32_t *>(&g_fault_host[word]) != 0;
}

int64_t ticks_of(int64_t microseconds) {
  int khz = g_clock_khz.load();
  if (khz <= 0) {
    int device = 0, rate = 0;
    if (hipGetDevice(&device) == hipSuccess &&
        hipDeviceGetAttribute(&rate, hipDeviceAttributeWallClockRate, device) == hipSuccess &&
        rate > 0)
      khz = rate;
    else
      khz = 100000;   // 100 MHz
    g_clock_khz.store(khz);
  }
  return microseconds * khz / 1000;
}

int64_t wait_limit_ticks() { return ticks_of(g_wait_limit_us.load()); }

int expect_extra() { return g_expect_extra.load(); }

namespace {
constexpr int kAnswerSlots = 64;   // calls that may wait at once
std::mutex g_answer_mutex;         // over the two below
unsigned long long *g_answer_host = nullptr, *g_answer_device = nullptr;   // 4 KB, held until the process ends
std::atomic<uint32_t> g_answer_ticket{0};
std::atomic<int> g_fail_answers{0};   // sub1_test_fail_answers
static __device__ int32_t answer_counts[kAnswerSlots * kAnswerCountStride];
__global__ void clear_count_kernel(int32_t *count) { *count = 0; }
SlotPool &answer_slots() {
  static SlotPool *pool = new SlotPool(kAnswerSlots);   // (never destroyed: threads may still wait at the process's end)
  return *pool;
}
}  // namespace

SlotPool::SlotPool(int slots) : left_(slots) {
  for (int i = 0; i < slots; i++) free_.push_back(i);
}

int SlotPool::take() {
  std::unique_lock<std::mutex> lock(mutex_);
  changed_.wait(lock, [this] { return !free_.empty() || left_ == 0; });
  if (left_ == 0) return -1;
  const int slot = free_.back();
  free_.pop_back();
  return slot;
}

void SlotPool::give_back(int slot) {
  {
    std::lock_guard<std::mutex> lock(mutex_);
    free_.push_back(slot);
  }
  changed_.notify_one();
}

void SlotPool::lose() {
  {
    std::lock_guard<std::mutex> lock(mutex_);
    left_--;
  }
  changed_.notify_all();
}

int AnswerSlot::take(hipStream_t stream, const char *who) {
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &capture) != hipSuccess) (void)hipGetLastError();   // (the launch will say)
  if (capture != hipStreamCaptureStatusNone)
    return fail(SUB1_ERR_HIP, "%s: waits for the GPU, which a stream that is being captured cannot", who);
  void *counts = nullptr;
  HIP_TRY(hipGetSymbolAddress(&counts, HIP_SYMBOL(answer_counts)));
  {
    std::lock_guard<std::mutex> lock(g_answer_mutex);
    if (!g_answer_host) {
      void *host = nullptr, *device = nullptr;
      const size_t bytes = kAnswerSlots * kAnswerWords * sizeof(unsigned long long);
      HIP_TRY(hipHostMalloc(&host, bytes, hipHostMallocPortable | hipHostMallocMapped));
      memset(host, 0, bytes);
      HIP_TRY(hipHostGetDevicePointer(&device, host, 0));
      g_answer_host = static_cast<unsigned long long *>(host);
      g_answer_device = static_cast<unsigned long long *>(device);
    }
  }
  slot_ = answer_slots().take();
  if (slot_ < 0)
    return fail(SUB1_ERR_INTERNAL, "%s: %d calls could not wait for the GPU, and none waits after them", who, kAnswerSlots);
  answer_.words = g_answer_device + slot_ * kAnswerWords;
  answer_.count = static_cast<int32_t *>(counts) + slot_ * kAnswerCountStride;
  do answer_.ticket = ++g_answer_ticket;
  while (answer_.ticket == 0);   // what the words hold at first
  stream_ = stream;
  return SUB1_OK;
}

int AnswerSlot::launched(const char *who) {
  HIP_TRY(hipGetLastError());
  open_ = true;
  int left = g_fail_answers.load();
  while (left > 0)
    if (g_fail_answers.compare_exchange_weak(left, left - 1))
      return fail(SUB1_ERR_INTERNAL, "%s: made to fail by sub1_test_fail_answers", who);
  return SUB1_OK;
}

AnswerSlot::~AnswerSlot() {
  if (slot_ < 0) return;
  if (open_) {
    // a call that ends without its answer, by an error: what it has launched still counts and stores
    clear_count_kernel<<<1, 1, 0, stream_>>>(answer_.count);
    const bool cleared = hipGetLastError() == hipSuccess;
    if (hipStreamSynchronize(stream_) != hipSuccess || !cleared) {
      (void)hipGetLastError();
      answer_slots().lose();
      return;
    }
  }
  answer_slots().give_back(slot_);
}

int AnswerSlot::wait(hipStream_t stream, int n, int32_t *values, const char *who) {
  const unsigned long long *words = g_answer_host + slot_ * kAnswerWords;
  auto arrived = [&]() {
    for (int i = 0; i < n; i++) {
      const unsigned long long v = __atomic_load_n(&words[i], __ATOMIC_RELAXED);
      if (static_cast<uint32_t>(v >> 32) != answer_.ticket) return false;
      values[i] = static_cast<int32_t>(static_cast<uint32_t>(v));
    }
    return true;
  };
  // looked for over the time that a layer's passes may take, then waited for
  const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(5);
  do {
    for (int i = 0; i < 64; i++) {
      if (arrived()) {
        open_ = false;
        return SUB1_OK;
      }
      __builtin_ia32_pause();
    }
  } while (std::chrono::steady_clock::now() < until);
  const hipError_t e = hipStreamSynchronize(stream);
  if (e == hipSuccess && arrived()) {
    open_ = false;
    return SUB1_OK;
  }
  if (e != hipSuccess) return fail(SUB1_ERR_HIP, "%s: %s", who, hipGetErrorString(e));
  return fail(SUB1_ERR_INTERNAL, "%s: the launch has ended without its answer", who);
}

}  // namespace sub1

namespace {

using sub1::bf16_to_f32;
using sub1::f32_to_bf16;
using sub1::fail;
using sub1::misaligned;
using sub1::row_result;
using sub1::wave_prefix_sum;

// ------------------------------------------------------------ slot table ---
//
// The reference table spends two 32-bit words per entry on 28 two-bit digits
// of which at most three are non-zero.  The kernels use a derived one-word
// form that lists the non-zeros:
//   bits 0-3          pair count L (the entry spans 2L weights)
//   bits 4+7j..8+7j   slot j: the non-zero's place in the entry (0..27)
//   bit 9+7j, 10+7j   set where it is the row min, the row max (neither: no slot j)
constexpr int kSlots = 3;
constexpr int kSlotBits = 7;

__global__ void derive_slot_table_kernel(const int32_t *__restrict__ dec,
                                         uint32_t *__restrict__ tab,
                                         int32_t *__restrict__ unsupported) {
  int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= SUB1_DICT_ENTRIES) return;
  uint32_t w0 = static_cast<uint32_t>(dec[2 * e]);
  uint32_t w1 = static_cast<uint32_t>(dec[2 * e + 1]);
  uint32_t out = w0 & 0xfu;
  int n = 0;
  bool bad = false;
  for (int d = 0; d < 28; d++) {
    uint32_t w = d < 14 ? w0 : w1;
    uint32_t t = (w >> (4 + 2 * (d % 14))) & 3u;
    if (t == 0) continue;
    if (t == 3 || n == kSlots) {
      bad = true;
      break;
    }
    out |= static_cast<uint32_t>(d | (t << 5)) << (4 + kSlotBits * n);
    n++;
  }
  tab[e] = out;
  if (bad) atomicOr(unsupported, 1);
}

// The cached table is found by the address of the caller's dec.  To notice an
// address that now holds something else, 64 words of dec at fixed scattered
// places are kept beside the table and compared by one wavefront of every
// launch; a difference sets the sticky kFaultDec flag (the host then drops its
// cached tables).
constexpr int kPrintWords = 64;
__host__ __device__ constexpr int print_index(int i) {
  return (i * 4099 + 7) & (SUB1_DEC_WORDS - 1);
}

__global__ void capture_print_kernel(const int32_t *__restrict__ dec, int32_t *__restrict__ print) {
  if (threadIdx.x < kPrintWords) print[threadIdx.x] = dec[print_index(threadIdx.x)];
}

__device__ __forceinline__ void compare_print(const int32_t *__restrict__ dec,
                                              const int32_t *__restrict__ print,
                                              int32_t *sticky) {
  if (threadIdx.x < kPrintWords && dec[print_index(threadIdx.x)] != print[threadIdx.x])
    sub1::raise_fault(sticky, sub1::kFaultDec);
}

// ----------------------------------------------- activations in LDS --------
//
// x is kept in LDS as fp32, with zeros behind the row for the digits of a last
// codeword that hang over its end (the reference pads the same way,
// sub1_cuda_kernel.cu:147-151) and for lanes that have no codeword left.
__host__ __device__ constexpr int lds_dwords_for_width(int width) { return (width + 32 + 3) / 4 * 4; }

template <int kThreads>
__device__ __forceinline__ void stage_activations(float *lds, const uint16_t *x, int width) {
  const int n = lds_dwords_for_width(width);
  for (int k = 4 * threadIdx.x; k < n; k += 4 * kThreads) {
    uint16_t v[4] = {0, 0, 0, 0};
    if (k + 4 <= width) {
      __builtin_memcpy(v, x + k, 8);
    } else {
      for (int j = 0; j < 4 && k + j < width; j++) v[j] = x[k + j];
    }
    *reinterpret_cast<float4 *>(lds + k) =
        make_float4(bf16_to_f32(v[0]), bf16_to_f32(v[1]), bf16_to_f32(v[2]), bf16_to_f32(v[3]));
  }
}

// The table word of a code: from the copy of the table's first `held` words in
// LDS where the code lies in it, from the table in global memory otherwise.  A
// gather from the 256 KB table costs a compute unit about 54 ns per wavefront
// instruction (every lane fetches a cache line of its own through the L1), one
// from LDS 3 ns, and the low codes are the frequent ones: the first 21 500
// entries take 64% of the codes of weights with 90% zeros.  Lanes whose code is
// held all read the table's first word, one line, so that the two reads need no
// branch and every lane's are in flight together.
template <bool kHeld>
__device__ __forceinline__ uint32_t table_word(const uint32_t *__restrict__ tab,
                                               const uint32_t *held_words, uint32_t held,
                                               uint32_t code) {
  if (!kHeld) return tab[code];
  const uint32_t far = tab[code < held ? 0u : code];
  const uint32_t near = held_words[min(code, held - 1)];
  return code < held ? near : far;
}

// ------------------------------------------------------------- matvec ------
//
// One product y += W x on the packed layout, built for the latency of a single
// call (reference sub1_cuda_kernel.cu:163-201 re-thought for 64-wide
// wavefronts): a WAVEFRONT per row.  Lane j takes codeword j of each run of 64
// consecutive codes of the row: one coalesced 128-byte load per run; its
// dictionary entry straight from the caller's dec (8 bytes per lane, from L2: no
// derived table and nothing remembered between calls); the column at which the
// codeword starts from a DPP prefix sum of the entries' lengths across the
// lanes; the activation under each of the entry's non-zero digits (at most
// three for the fixed dictionary) from x through the vector cache; products
// x * (row min | row max) added in fp32 per lane; and at the row's end a
// butterfly sum over the 64 lanes.  Every load a wavefront needs is requested
// as early as its address is known: row offsets, (min, max) and y at once, the codes of four
// runs before the first table read, the next four's entries and the codes behind them while these are
// multiplied, and the activations of all four before the first multiplication.  (Rows of 75 to 98 % zeros, a
// hundredth without: 1024 x 4096 18.5 -> 16.1 us of kernel time with that, c-2048 wo at 90 % 8.6 -> 8.2.)
//
// Order of additions (the oracle's sub1o_matvec_wave): lane j adds its
// codewords j, j + 64, ... in turn, the digits of a codeword left to right, one
// fused multiply-add each; then six butterfly steps, lane l adding lane l ^ m
// for m = 1, 2, 4, 8, 16, 32; bf16; y += in bf16.

// dpp_ctrl values (CDNA ISA, DPP)
constexpr int kDppQuadXor1 = 0xb1, kDppQuadXor2 = 0x4e;      // quad_perm [1,0,3,2], [2,3,0,1]
constexpr int kDppHalfMirror = 0x141, kDppRowMirror = 0x140;

template <int kCtrl>
__device__ __forceinline__ float dpp_float(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xf, 0xf, false));
}

// Lane l receives the sum of the butterfly over all 64 lanes: l + (l ^ 1), then
// ^ 2, ^ 4, ^ 8, ^ 16, ^ 32.  After the steps 1 and 2 the four lanes of a quad
// hold the same value, so the mirror within eight lanes pairs a lane with the
// other quad exactly as ^ 4 does, and the mirror within a row of sixteen as ^ 8.
__device__ __forceinline__ float wave_butterfly_sum(float v) {
  v += dpp_float<kDppQuadXor1>(v);
  v += dpp_float<kDppQuadXor2>(v);
  v += dpp_float<kDppHalfMirror>(v);
  v += dpp_float<kDppRowMirror>(v);
  v += __shfl_xor(v, 16);
  v += __shfl_xor(v, 32);
  return v;
}

constexpr int kWaveRuns = 4;   // runs of 64 codes whose loads are requested together

// A row's codes, kWaveRuns runs at a time, and their dictionary entries, a turn ahead: the
// entries are asked for while the turn before is worked on, the codes one turn earlier.
struct RowEntries {
  const uint2 *table;
  const uint16_t *codes;
  int len;
  int code[kWaveRuns];      // of the turn behind `entry`'s
  uint2 entry[kWaveRuns];   // no code: no digits, length 0

  __device__ __forceinline__ RowEntries(const int32_t *dec, const uint16_t *row, int n)
      : table(reinterpret_cast<const uint2 *>(dec)), codes(row), len(n) {
    ask_codes(0);
    ask_entries();
    if (len > 64 * kWaveRuns) ask_codes(64 * kWaveRuns);
  }
  __device__ __forceinline__ void ask_codes(int c0) {
#pragma unroll
    for (int u = 0; u < kWaveRuns; u++) {
      const int i = c0 + 64 * u + static_cast<int>(threadIdx.x & 63);
      code[u] = i < len ? codes[i] : -1;
    }
  }
  __device__ __forceinline__ void ask_entries() {
#pragma unroll
    for (int u = 0; u < kWaveRuns; u++) entry[u] = code[u] >= 0 ? table[code[u]] : make_uint2(0u, 0u);
  }
  // The entries of the turn from code c0 on; the next turn's are asked for.
  __device__ __forceinline__ void take(int c0, uint2 (&now)[kWaveRuns]) {
#pragma unroll
    for (int u = 0; u < kWaveRuns; u++) now[u] = entry[u];
    if (c0 + 64 * kWaveRuns < len) {
      ask_entries();
      if (c0 + 128 * kWaveRuns < len) ask_codes(c0 + 128 * kWaveRuns);
    }
  }
};

// What the row's digits are multiplied by.  An entry's first three non-zero digits (all there
// are, by the fixed dictionary) are looked up side by side, whatever more there is one by one.
constexpr int kDigitsAtOnce = 3;

template <int kWaves>
__global__ __launch_bounds__(64 * kWaves) void matvec_wave_kernel(
    const int32_t *__restrict__ dec, const uint16_t *__restrict__ w_comp,
    const int32_t *__restrict__ row_off, const uint32_t *__restrict__ minmax,
    const uint16_t *__restrict__ x, uint16_t *__restrict__ y, int height, int width,
    int64_t ldx, int64_t ldy) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * kWaves + (threadIdx.x >> 6);
  if (row >= height) return;
  x += static_cast<int64_t>(blockIdx.y) * ldx;
  y += static_cast<int64_t>(blockIdx.y) * ldy;
  const int off = __builtin_amdgcn_readfirstlane(row_off[row]);
  const int len = __builtin_amdgcn_readfirstlane(row_off[row + 1]) - off;
  const uint32_t mm = minmax[row];
  const uint16_t y_old = y[row];
  const float w_min = __uint_as_float(mm << 16), w_max = __uint_as_float(mm & 0xffff0000u);
  RowEntries entries(dec, w_comp + off, len);
  float acc = 0.f;
  int col = 0;   // the column at which the current run of codes starts
  for (int c0 = 0; c0 < len; c0 += 64 * kWaveRuns) {
    uint2 entry[kWaveRuns];
    entries.take(c0, entry);
    unsigned long long digits[kWaveRuns];   // what is left of them
    int at[kWaveRuns];                      // where this lane's codeword starts
    uint16_t xv[kWaveRuns][kDigitsAtOnce];
    uint32_t kinds = 0;                     // two bits for each: what it is multiplied by, 0: nothing
#pragma unroll
    for (int u = 0; u < kWaveRuns; u++) {
      if (c0 + 64 * u >= len) break;
      const int span = 2 * static_cast<int>(entry[u].x & 15u);     // weights the codeword covers
      const int upto = wave_prefix_sum(span);
      at[u] = col + upto - span;
      col += __builtin_amdgcn_readlane(upto, 63);
      digits[u] = static_cast<unsigned long long>(entry[u].x >> 4) |
                  (static_cast<unsigned long long>(entry[u].y >> 4) << 28);
#pragma unroll
      for (int j = 0; j < kDigitsAtOnce; j++) {
        const int d = digits[u] ? (__ffsll(digits[u]) - 1) >> 1 : 0;
        const bool inside = digits[u] && at[u] + d < width;   // digits past the width are dropped
        if (inside) kinds |= (static_cast<uint32_t>(digits[u] >> (2 * d)) & 3u) << (2 * (kDigitsAtOnce * u + j));
        digits[u] &= ~(3ull << (2 * d));
        xv[u][j] = x[inside ? at[u] + d : 0];
      }
    }
#pragma unroll
    for (int u = 0; u < kWaveRuns; u++) {
      if (c0 + 64 * u >= len) break;
#pragma unroll
      for (int j = 0; j < kDigitsAtOnce; j++) {
        const uint32_t sym = (kinds >> (2 * (kDigitsAtOnce * u + j))) & 3u;
        const float sum = __fmaf_rn(bf16_to_f32(xv[u][j]), sym == 1 ? w_min : (sym == 2 ? w_max : 0.f), acc);
        acc = sym ? sum : acc;
      }
      while (digits[u]) {
        const int d = (__ffsll(digits[u]) - 1) >> 1;
        const int sym = static_cast<int>(digits[u] >> (2 * d)) & 3;
        digits[u] &= ~(3ull << (2 * d));
        if (at[u] + d < width)
          acc = __fmaf_rn(bf16_to_f32(x[at[u] + d]), sym == 1 ? w_min : (sym == 2 ? w_max : 0.f), acc);
      }
    }
  }
  const float res = wave_butterfly_sum(acc);
  if (lane == 0) {
    // reference sub1_cuda_kernel.cu:200: y[row] += bf16(res), the sum in bf16
    y[row] = f32_to_bf16(bf16_to_f32(y_old) + bf16_to_f32(f32_to_bf16(res)));
  }
}

// ------------------------------------------------------------- decode ------

// A wavefront per row.  As in the product above, lane j takes codeword j of each run
// of 64 and a prefix sum of the entries' lengths places it; here the run's symbols
// (up to 64 x 30) are put together in LDS, shifted so that four symbols of a word are
// four that share a word of the output, and go out in whole words.  Columns behind
// the last codeword become zero.  3001 x 1023 (9.2 MB out, 2 us at the copy rate):
// 6.2 us, a chain of four trips to memory and the writing; a thread per row, walking
// its codes and writing byte by byte, took 178.
constexpr int kDecodeRun = 64 * 30 + 4;   // bytes of LDS per wavefront, a multiple of 4

// Symbols w (four bytes) at elements first .. first + 3, as far as from <= element < to.
__device__ __forceinline__ void write_four(uint32_t w, uint32_t minmax, int64_t first, int64_t from,
                                           int64_t to, uint8_t *__restrict__ out_tern,
                                           uint16_t *__restrict__ out_w) {
  uint16_t v[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    const uint32_t t = (w >> (8 * j)) & 3u;
    v[j] = static_cast<uint16_t>(t == 1 ? minmax : t == 2 ? minmax >> 16 : 0u);
  }
  if (first >= from && first + 4 <= to) {
    if (out_tern) *reinterpret_cast<uint32_t *>(out_tern + first) = w;
    if (out_w)
      *reinterpret_cast<uint2 *>(out_w + first) =
          make_uint2(v[0] | static_cast<uint32_t>(v[1]) << 16, v[2] | static_cast<uint32_t>(v[3]) << 16);
    return;
  }
#pragma unroll
  for (int j = 0; j < 4; j++)
    if (first + j >= from && first + j < to) {
      if (out_tern) out_tern[first + j] = static_cast<uint8_t>(w >> (8 * j));
      if (out_w) out_w[first + j] = v[j];
    }
}

template <int kWaves>
__global__ __launch_bounds__(64 * kWaves) void decode_kernel(
    const int32_t *__restrict__ dec, const uint16_t *__restrict__ w_comp,
    const int32_t *__restrict__ row_off, const uint32_t *__restrict__ minmax,
    uint8_t *__restrict__ out_tern, uint16_t *__restrict__ out_w, int32_t *__restrict__ bad_rows,
    int height, int width, int phase) {
  __shared__ uint32_t run_lds[kWaves][kDecodeRun / 4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = blockIdx.x * kWaves + wave;
  if (row >= height) return;
  uint32_t *words = run_lds[wave];
  uint8_t *bytes = reinterpret_cast<uint8_t *>(words);
  const int off = __builtin_amdgcn_readfirstlane(row_off[row]);
  const int len = __builtin_amdgcn_readfirstlane(row_off[row + 1]) - off;
  const uint32_t mm = minmax ? minmax[row] : 0u;
  const uint2 *table = reinterpret_cast<const uint2 *>(dec);
  // elements of the output, counted from a place where its words begin
  const int64_t row_first = static_cast<int64_t>(row) * width + phase, row_last = row_first + width;
  out_tern = out_tern ? out_tern - phase : nullptr;
  out_w = out_w ? out_w - phase : nullptr;
  int64_t at = row_first;   // the element at which the run starts
  for (int c0 = 0; c0 < len; c0 += 64) {
    const int i = c0 + lane;
    const int code = i < len ? w_comp[off + i] : -1;
    const uint2 entry = code >= 0 ? table[code] : make_uint2(0u, 0u);
#pragma unroll
    for (int k = 0; k < (kDecodeRun / 4 + 63) / 64; k++)
      if (lane + 64 * k < kDecodeRun / 4) words[lane + 64 * k] = 0u;
    const int span = 2 * static_cast<int>(entry.x & 15u);
    const int upto = wave_prefix_sum(span);
    const int shift = static_cast<int>(at & 3);
    // digit d is bits 4 + 2 (d % 14) of word d / 14 (of the second, past it)
    unsigned long long digits = static_cast<unsigned long long>(entry.x >> 4) |
                                static_cast<unsigned long long>(entry.y >> 4) << 28 |
                                static_cast<unsigned long long>(entry.y >> 4 & 15u) << 56;
    digits &= (1ull << (2 * span)) - 1;
    uint8_t *mine = bytes + shift + upto - span;
    __builtin_amdgcn_wave_barrier();
    while (digits) {
      const int d = (__ffsll(digits) - 1) >> 1;
      mine[d] = static_cast<uint8_t>((digits >> (2 * d)) & 3);
      digits &= ~(3ull << (2 * d));
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int64_t end = at + __builtin_amdgcn_readlane(upto, 63);
    const int64_t to = end < row_last ? end : row_last;
    for (int k = lane; (at - shift) + 4 * k < to; k += 64)
      write_four(words[k], mm, at - shift + 4 * k, at, to, out_tern, out_w);
    at = end;
    __builtin_amdgcn_wave_barrier();
  }
  const int shift = static_cast<int>(at & 3);
  for (int64_t first = at - shift + 4 * lane; first < row_last; first += 256)
    write_four(0u, mm, first, at, row_last, out_tern, out_w);
  if (bad_rows && lane == 0 && at - row_first != ((width + 1) & ~1)) atomicAdd(bad_rows, 1);
}

// Behind the launches that counted.  (Told by their own last workgroup, the host heard of the
// count while rows were still on their way to memory, and of two launches before the second:
// a call on 3001 x 1023 took 20.8 us so, takes 22.8 now, and 30 with the count copied to the host.)
__global__ void tell_count_kernel(sub1::Answer answer) {
  // an exchange: the zero is there before the host hears of the count and gives the slot to
  // a call on another stream
  const int32_t count = __hip_atomic_exchange(answer.count, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  sub1::tell(answer, 0, count);
}

// ------------------------------------------------------ grouped experts ----
//
// Persistent grid.  Work is cut into tiles (token, projection, part of its rows),
// numbered with all wi tiles before all wo tiles, and handed out by an atomic
// ticket.  A wo tile of token t needs all of h[t], so it waits until the wi tiles
// of t have signalled; those have smaller tickets, were therefore taken by
// workgroups that are already running, and never wait themselves, so the wait
// always ends.
//
// A few tokens have a workgroup for every tile instead, by number, so that wi's tiles lie one to a compute
// unit, and a wo tile's has its rows' codes and their words of the table by the time h is there.
// (One token of base and c-2048 shapes 17.7 us and 23.4, nine of base shapes 21.9; 28.9, 44.5 and 43.8 with
// tickets and everything fetched behind the wait; with a ticket that only says which tile, of the launch
// or of the token, 14 tokens of base shapes 22.6 -> 28.8 and 24.5, nine of c-2048 50.5 -> 62 and 68, as wi's tiles
// then share units.)  They run all at once on a GPU that does nothing else; where other launches hold
// units, workgroups that wait may keep those that they wait for from starting.  Every wi tile is therefore
// CLAIMED by the workgroup that does it, and one that has waited for some time claims what nobody has, does
// it and waits on: nobody waits for a tile that no running workgroup has, so this wait always ends too.
// (Claims take 0.5 us of the 17 to 25 of a few tokens of base and large shapes.  Asked for behind the loads, which
// wait for the answer, they come so late that others are claimed for nothing: c-2048, two tokens, 30 -> 45.)
//
// Within a tile the wavefronts take runs of rows from a counter in LDS and give a
// LANE to a GROUP of 32 codes, not to a row: a row's sum is the sum of its groups'
// sums in order (the library's canonical order on this layout), so groups are
// what can be worked on side by side.  Rows differ in length by a factor of 20 where
// their shares of zeros differ, and a wavefront of rows takes as long as the
// longest of them; a wavefront of groups takes 32 codes.  A lane reads its codes in
// four 16-byte loads, next to its neighbours', fetches all their table words at
// once, and from the words' lengths a prefix sum over the lanes gives the column at
// which each group starts.
//
// What bounds it: 48 vector instructions a codeword (20 ns a wavefront and compute
// unit: in the sweep of 2048 c-2048 experts the VALUs are 73 % busy), beside LDS gathers of
// activations (three a codeword, 8 ns) and the words outside the held head of the
// table (54 ns times the share of lanes that miss).  A wavefront's 64 codewords take 28 ns
// there.  Switch shapes with shares of zeros between 75 and 98 %,
// 64 tokens, us: base 381 -> 74, large 526 -> 105, c-2048 956 -> 230, where the lane per
// row waited for the longest of 64; with 90 % everywhere 99 -> 51, 109 -> 61, 255 -> 133.
struct MoeArgs {
  const uint32_t *tab;
  const uint16_t *w_comp;
  const int64_t *wi_code_base;
  const int64_t *wo_code_base;
  const int32_t *wi_row_off;
  const int32_t *wo_row_off;
  const uint32_t *wi_minmax;
  const uint32_t *wo_minmax;
  const int32_t *token_expert;
  const uint16_t *x;
  uint16_t *y;
  uint16_t *h;
  int32_t *ctrl;  // the control words (sub1_common.h): ticket, fault counts, a word per token
  int tokens, d_model, d_ff, experts;
  int wi_tiles, wo_tiles;  // per token
  int act_dwords;          // LDS dwords of the activations; the table's first words follow
  int held;                // words of the table kept in LDS (0: none)
  int wi_expect;           // wi tiles a wo tile waits for (wi_tiles outside tests)
  int64_t patience;        // a workgroup for every tile: ticks after which a wo tile's claims tiles of wi
  int64_t late;            // tests: ticks that every other wi tile's workgroup starts late
  int64_t wait_ticks;      // longest wait, in ticks of wall_clock64
  int32_t *sticky;         // fault flags in pinned host memory
  const int32_t *dec;      // the caller's table and the words kept of it
  const int32_t *print;
};

using sub1::kCtrlHeader;

constexpr int kGroupCodes = 32;   // codes per partial sum: part of the results' definition
constexpr int kGroupStep = 30;    // what a turn of 64 groups takes, in steps of a lane with a row of its own

// Table words of a lane's group: `count` codes from `codes` on, of a row that
// ends at codes + count at the earliest eight codes after it began (`whole`), or of
// a shorter row; zero words (nothing, no advance) make up the rest.
template <bool kHeld>
__device__ __forceinline__ void group_words(const uint32_t *__restrict__ tab, const uint32_t *held_words,
                                            uint32_t held, const uint16_t *codes, int count, bool whole,
                                            uint32_t (&e)[kGroupCodes]) {
  uint32_t w[kGroupCodes / 8][4];
  int skip[kGroupCodes / 8];   // codes of an eight that are not the group's: the first ones
#pragma unroll
  for (int k = 0; k < kGroupCodes / 8; k++) {
    // a partial eight, and one behind the group's end, is read from eight codes
    // before that end (lanes without a group: from where they stand)
    const int left = min(max(count - 8 * k, 0), 8);
    skip[k] = whole ? 8 - left : 8;
    const uint16_t *from = codes + (left > 0 ? 8 * k - (8 - left) : count > 0 ? count - 8 : 0);
    if (whole) {
      __builtin_memcpy(w[k], from, 16);   // any alignment
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++) w[k][j] = 0;
    }
  }
#pragma unroll
  for (int i = 0; i < kGroupCodes; i++) {
    const uint32_t code = (i & 1) ? w[i / 8][(i & 7) / 2] >> 16 : w[i / 8][(i & 7) / 2] & 0xffffu;
    const uint32_t word = table_word<kHeld>(tab, held_words, held, code);
    e[i] = (i & 7) < skip[i / 8] ? 0u : word;
  }
  if (!whole)   // rows of up to seven codes
#pragma unroll
    for (int i = 0; i < 7; i++)
      if (i < count) e[i] = table_word<kHeld>(tab, held_words, held, codes[i]);
}

// The activations under a codeword's weights onto the sums of either symbol, left
// to right; `at`, the column at which it starts, moves on.
__device__ __forceinline__ void add_codeword(uint32_t e, const float *X, int &at, float &p1, float &p2) {
#pragma unroll
  for (int j = 0; j < kSlots; j++) {
    const uint32_t slot = e >> (4 + kSlotBits * j);
    const uint32_t xv = __float_as_uint(X[at + static_cast<int>(slot & 31u)]);
    const uint32_t is1 = static_cast<uint32_t>(static_cast<int32_t>(slot << 26) >> 31);
    const uint32_t is2 = static_cast<uint32_t>(static_cast<int32_t>(slot << 25) >> 31);
    p1 += __uint_as_float(xv & is1);
    p2 += __uint_as_float(xv & is2);
  }
  at += 2 * static_cast<int>(e & 15u);
}

// A lane's row from its first code to its last: the sums of its groups, first
// group first.
template <bool kHeld>
__device__ __forceinline__ void row_by_lane(const uint32_t *__restrict__ tab, const uint32_t *held_words,
                                            uint32_t held, const uint16_t *codes, int len,
                                            const float *X, float &s1, float &s2) {
  s1 = s2 = 0.f;
  float p1 = 0.f, p2 = 0.f;
  int at = 0;
  uint32_t next[4];
  if (len >= 8) __builtin_memcpy(next, codes, 16);
  for (int i = 0; i < len; i += 8) {
    const uint32_t w[4] = {next[0], next[1], next[2], next[3]};
    // the row's last, partial eight is read from eight codes before its end
    const int ahead = min(i + 8, max(len - 8, 0));
    if (i + 8 < len) __builtin_memcpy(next, codes + ahead, 16);
    const int skip = len >= 8 ? max(i + 8 - len, 0) : 8;
    uint32_t e[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      const uint32_t code = (j & 1) ? w[j / 2] >> 16 : w[j / 2] & 0xffffu;
      e[j] = table_word<kHeld>(tab, held_words, held, code);
      if (j < skip) e[j] = 0u;
    }
    if (len < 8)   // a row of up to seven codes
      for (int j = 0; j < len; j++) add_codeword(table_word<kHeld>(tab, held_words, held, codes[j]), X, at, p1, p2);
#pragma unroll
    for (int j = 0; j < 8; j++) add_codeword(e[j], X, at, p1, p2);
    if (((i + 8) & (kGroupCodes - 1)) == 0) {   // a group is complete
      s1 += p1;
      s2 += p2;
      p1 = p2 = 0.f;
    }
  }
  s1 += p1;   // the last, possibly partial, group (adds +0 if it was just folded)
  s2 += p2;
}

// Rows row0 .. row0 + rows - 1 of one matrix (rows <= 64, a wavefront), 64 groups a turn.  Where
// the table is in memory, what a turn needs of the matrix is fetched ahead: the first one's before the
// activations are there.  (With the table's head in LDS the wavefronts of a compute unit are four times
// as many, and their registers do not hold it.)
template <bool kHeld>
struct RowRun {
  const uint32_t *tab, *held_words;
  uint32_t held;
  const uint16_t *codes;
  int off, len;               // a lane's row
  int first, last, total;     // its groups, among the run's; all groups
  bool by_lane;               // the rows are walked by a lane each
  int turn;
  // of a lane's group in the turn
  int r_first;                // its row's first group
  uint32_t e[kGroupCodes];

  __device__ __forceinline__ void take(const uint16_t *matrix, const int32_t *__restrict__ row_off, int row0, int rows) {
    const int lane = threadIdx.x & 63;
    const bool mine = lane < rows;
    codes = matrix;
    off = mine ? row_off[row0 + lane] : 0;
    len = mine ? row_off[row0 + lane + 1] - off : 0;
    const int groups = (max(len, 0) + kGroupCodes - 1) / kGroupCodes;
    last = wave_prefix_sum(groups);
    first = last - groups;
    total = __builtin_amdgcn_readlane(last, 63);
    // A lane to a row instead where the rows are alike and there are enough of them: it
    // then takes as many steps as the longest has codes, and no prefix sums.  (256
    // tokens, us: groups always 125 base, 163 large, 428 c-2048; rows always 103, 163,
    // 483, and 685, 960, 2176 where the shares of zeros differ from row to row; by this
    // rule 98, 149, 416, and 165, 263, 651.)
    int longest = len;
    for (int m = 1; m < 64; m <<= 1) longest = max(longest, __shfl_xor(longest, m, 64));
    by_lane = (longest + 7) / 8 * 8 <= (total + 63) / 64 * kGroupStep;
    turn = 0;
    if (!kHeld && !by_lane && total) fetch();
  }

  __device__ __forceinline__ void fetch() {
    // the row of this lane's group: the first whose groups end behind it
    const int lane = threadIdx.x & 63;
    const int g = min(turn + lane, total - 1);
    int r = 0;
#pragma unroll
    for (int step = 32; step >= 1; step >>= 1)
      if (__shfl(last, r + step - 1, 64) <= g) r += step;
    r_first = __shfl(first, r, 64);
    const int r_off = __shfl(off, r, 64), r_len = __shfl(len, r, 64);
    const bool active = turn + lane < total;
    const int in_row = active ? kGroupCodes * (g - r_first) : 0;
    const int count = active ? min(r_len - in_row, kGroupCodes) : 0;
    group_words<kHeld>(tab, held_words, held, codes + r_off + in_row, count, r_len >= 8, e);
  }

  // Lane r receives the sums of row row0 + r.  `partial` is the wavefront's own LDS, 64 pairs.
  __device__ __forceinline__ void sums(const float *X, float2 *partial, float &s1, float &s2) {
    if (by_lane) {
      row_by_lane<kHeld>(tab, held_words, held, codes + off, len, X, s1, s2);
      return;
    }
    const int lane = threadIdx.x & 63;
    s1 = 0.f;
    s2 = 0.f;
    int carry = 0;   // the column reached in a row that goes on from the turn before
    while (turn < total) {
      if (kHeld) fetch();
      int span = 0;
#pragma unroll
      for (int i = 0; i < kGroupCodes; i++) span += static_cast<int>(e[i] & 15u);
      span *= 2;
      const int before = wave_prefix_sum(span) - span;
      const int row_before = __shfl(before, max(r_first - turn, 0), 64);
      const int at = before - row_before + (r_first < turn ? carry : 0);
      carry = __builtin_amdgcn_readlane(at + span, 63);
      float2 p = {0.f, 0.f};
      int col = at;
#pragma unroll
      for (int i = 0; i < kGroupCodes; i++) add_codeword(e[i], X, col, p.x, p.y);
      partial[lane] = p;
      sub1::wave_lds_fence();
      for (int i = max(first - turn, 0); i < min(last - turn, 64); i++) {
        const float2 q = partial[i];
        s1 += q.x;
        s2 += q.y;
      }
      __builtin_amdgcn_wave_barrier();
      turn += 64;
      if (!kHeld && turn < total) fetch();
    }
  }
};

// Rows that a wavefront takes at a time: a lane each where a tile has that many
// for all its wavefronts, but at least about 64 groups of them (a row of W weights
// with 90% zeros has W / 23 codes); where there are enough workgroups for all tiles at
// once, as many as make all wavefronts work side by side.  (Rounded up: a run more than there are wavefronts
// is a turn of its own for one of them.  99 tokens, 569 x 3563, 61.2 -> 58.7 us; 130, 900 x 2500, 95.6 -> 90.8;
// 61, 1501 x 3001, 65.2 -> 63.6; sizes that divide as before.)
template <bool kHeld>
__device__ __forceinline__ int rows_at_a_time(int rows, int width, int waves) {
  if (!kHeld) return min((rows + waves - 1) / waves, 64);
  return min(max((rows + waves - 1) / waves, max(64 * 640 / (width + 640), 1)), 64);
}

// Claims of a token's wi tiles, and its word where there are some: 64 bits, with a third count beside the
// two of the others' (sub1_common.h), tiles that were done by workgroups of wo.  All of it is zero between launches.
constexpr int kClaimWord = 2;          // from the token's word on: a bit for every tile
constexpr int kMostClaims = 256;
static_assert(kClaimWord + kMostClaims / 32 <= sub1::kCtrlTokenStride && sub1::kCtrlHeader % 2 == 0, "within the token's words");
constexpr unsigned long long kTokenHelped = 1ull << 32;

// Whether the tile was free.
__device__ __forceinline__ bool claim_tile(int32_t *token, int tile) {
  const int32_t bit = static_cast<int32_t>(1u << (tile & 31));
  return !(__hip_atomic_fetch_or(&token[kClaimWord + tile / 32], bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit);
}

// Thread 0 of a wo tile's workgroup: bounded_wait, which after `patience` ticks claims a wi tile that
// nobody has started and returns it; -1 once h is there (or the time is up).
__device__ __forceinline__ int wait_or_claim(const MoeArgs &a, int32_t *token, int64_t patience) {
  int looks = 0;
  int64_t t0 = 0;
  while ((__hip_atomic_load(token, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 0xffff) < a.wi_expect) {
    if ((++looks & 15) == 1) {
      const int64_t now = static_cast<int64_t>(wall_clock64());
      if (looks == 1) t0 = now;
      if (now - t0 >= patience)
        for (int first = 0; first < a.wi_tiles; first += 32) {
          const uint32_t all = a.wi_tiles - first < 32 ? (1u << (a.wi_tiles - first)) - 1 : ~0u;
          const uint32_t free = all & ~static_cast<uint32_t>(__hip_atomic_load(&token[kClaimWord + first / 32], __ATOMIC_RELAXED,
                                                                               __HIP_MEMORY_SCOPE_AGENT));
          if (!free) continue;
          const int tile = first + __ffs(free) - 1;
          // (counted first: whose tile it was leaves once it finds the claim)
          unsigned long long *word = reinterpret_cast<unsigned long long *>(token);
          __hip_atomic_fetch_add(word, kTokenHelped, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          sub1::drain_stores();
          if (claim_tile(token, tile)) return tile;
          __hip_atomic_fetch_add(word, ~0ull << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;   // somebody was faster: look again
        }
      if (now - t0 > a.wait_ticks) {
        sub1::raise_fault(a.sticky, sub1::kFaultWait);
        __hip_atomic_fetch_add(&a.ctrl[sub1::kCtrlGaveUp], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
    }
    __builtin_amdgcn_s_sleep(2);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  return -1;
}

// Thread 0 of a workgroup of wo that is done, or of one of wi whose tile another has done.  With the last of
// them nobody looks at the token's words any more, and they go back to zero.
__device__ __forceinline__ void leave_token(const MoeArgs &a, int32_t *token) {
  unsigned long long *word = reinterpret_cast<unsigned long long *>(token);
  const unsigned long long before = __hip_atomic_fetch_add(word, static_cast<unsigned long long>(sub1::kTokenWaited),
                                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int left = static_cast<int>(before >> 16 & 0xffff) + 1;
  if (left != a.wo_tiles + static_cast<int>(before >> 32)) return;
  for (int i = 0; i < (a.wi_tiles + 31) / 32; i++)
    __hip_atomic_store(&token[kClaimWord + i], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(word, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int kThreads>
__global__ __launch_bounds__(kThreads, kThreads == 1024 ? 4 : 2) void moe_kernel(MoeArgs a) {
  constexpr bool kHeld = kThreads == 1024;   // the form with the table's head in LDS, and with tickets
  extern __shared__ __align__(16) float lds[];
  __shared__ int s_ticket, s_row, s_claimed;
  __shared__ float2 s_partial[kThreads];
  const int n_wi = a.tokens * a.wi_tiles;
  const int n_all = n_wi + a.tokens * a.wo_tiles;
  if (blockIdx.x == 0) compare_print(a.dec, a.print, a.sticky);
  // the table's first words into LDS, once per workgroup (a persistent grid)
  uint32_t *held_words = reinterpret_cast<uint32_t *>(lds + a.act_dwords);
  if (kHeld)
    for (int i = 4 * threadIdx.x; i < a.held; i += 4 * kThreads)
      *reinterpret_cast<uint4 *>(held_words + i) = *reinterpret_cast<const uint4 *>(a.tab + i);
  float2 *partial = s_partial + (threadIdx.x & ~63u);
  constexpr int kWaves = kThreads / 64;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  RowRun<kHeld> run;
  run.tab = a.tab;
  run.held_words = held_words;
  run.held = a.held;
  int help = -1;   // a workgroup for every tile, of wo: one of wi that it does first
  bool waited = false;
  for (;;) {
    int ticket = !kHeld && help >= 0 ? help : static_cast<int>(blockIdx.x);
    if (kHeld) {
      __syncthreads();  // previous tile's readers of lds and s_ticket are done
      if (threadIdx.x == 0)
        s_ticket = __hip_atomic_fetch_add(&a.ctrl[0], 1, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
      __syncthreads();
      ticket = s_ticket;
      if (ticket >= n_all) break;
    }

    const bool is_wi = ticket < n_wi;
    const int j = is_wi ? ticket : ticket - n_wi;
    const int tiles = is_wi ? a.wi_tiles : a.wo_tiles;
    const int t = j / tiles, part = j - t * tiles;
    const int height = is_wi ? a.d_ff : a.d_model, width = is_wi ? a.d_model : a.d_ff;
    const int row_begin = static_cast<int>(static_cast<int64_t>(height) * part / tiles);
    const int row_end = static_cast<int>(static_cast<int64_t>(height) * (part + 1) / tiles);
    int e = a.token_expert[t];
    if (e >= a.experts) {
      if (!is_wi && part == 0 && threadIdx.x == 0)
        __hip_atomic_fetch_add(&a.ctrl[sub1::kCtrlBadIds], 1, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
      e = -1;
    }
    if (e < 0) {
      if (!is_wi)
        for (int row = row_begin + threadIdx.x; row < row_end; row += kThreads) {
          const int64_t i = static_cast<int64_t>(t) * a.d_model + row;
          a.y[i] = a.x[i];
        }
      if (!kHeld) break;
      continue;   // a dropped token's word stays untouched
    }
    const int32_t *row_off = (is_wi ? a.wi_row_off : a.wo_row_off) + static_cast<int64_t>(e) * (height + 1);
    const uint16_t *codes = a.w_comp + (is_wi ? a.wi_code_base : a.wo_code_base)[e];
    const uint32_t *minmax = (is_wi ? a.wi_minmax : a.wo_minmax) + static_cast<int64_t>(e) * height;
    int32_t *token = &a.ctrl[sub1::token_word(t)];
    bool taken = false;   // thread 0: somebody else does this tile of wi
    if (!kHeld && is_wi && help < 0) {
      if (a.late && part % 2 == 0) {
        const int64_t t0 = static_cast<int64_t>(wall_clock64());
        while (static_cast<int64_t>(wall_clock64()) - t0 < a.late) __builtin_amdgcn_s_sleep(64);
      }
      if (threadIdx.x == 0) taken = !claim_tile(token, part);
    }
    const int at_a_time = rows_at_a_time<kHeld>(row_end - row_begin, width, kWaves);
    int row0 = row_begin + at_a_time * wave;   // the first run; further ones from s_row
    if (row0 < row_end) run.take(codes, row_off, row0, min(at_a_time, row_end - row0));
    if (threadIdx.x == 0) {
      s_row = row_begin + at_a_time * kWaves;
      if (kHeld && !is_wi) sub1::bounded_wait(token, a.wi_expect, a.wait_ticks, a.sticky, &a.ctrl[sub1::kCtrlGaveUp]);
      if (!kHeld && !is_wi) s_claimed = wait_or_claim(a, token, waited ? 0 : a.patience);
    }
    __syncthreads();  // thread 0's acquire covers the whole workgroup
    if (!kHeld && !is_wi) {
      waited = true;
      if (s_claimed >= 0) {
        help = t * a.wi_tiles + s_claimed;
        continue;
      }
    }
    stage_activations<kThreads>(lds, (is_wi ? a.x : a.h) + static_cast<int64_t>(t) * width, width);
    // (asked for above: by now its answer is here)
    if (!kHeld && is_wi && threadIdx.x == 0) s_claimed = taken;
    __syncthreads();
    if (!kHeld && is_wi && s_claimed) {
      if (threadIdx.x == 0) leave_token(a, token);
      break;
    }
    while (row0 < row_end) {
      const int rows = min(at_a_time, row_end - row0);
      const int row = row0 + lane;
      float s1, s2;
      run.sums(lds, partial, s1, s2);
      if (lane < rows) {
        uint16_t b = f32_to_bf16(row_result(minmax[row], s1, s2));
        if (is_wi) {
          if (b & 0x8000u) b = 0;  // relu
          // stored at agent scope: written through this die's L2, where the
          // workgroups on other dies will read it
          __hip_atomic_store(&a.h[static_cast<int64_t>(t) * a.d_ff + row], b, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
        } else {
          a.y[static_cast<int64_t>(t) * a.d_model + row] = b;
        }
      }
      row0 = 0;
      if (lane == 0) row0 = atomicAdd(&s_row, at_a_time);
      row0 = __builtin_amdgcn_readfirstlane(row0);
      if (row0 < row_end) run.take(codes, row_off, row0, min(at_a_time, row_end - row0));
    }
    if (is_wi) {
      // every wavefront waits for its h stores to be acknowledged, then the
      // barrier, then thread 0 counts the tile (a release fence here would write
      // back the whole L2)
      sub1::drain_stores();
      __syncthreads();
      if (threadIdx.x == 0)
        __hip_atomic_fetch_add(token, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else if (threadIdx.x == 0) {
      // said once the tile's work is done: it takes a round trip to memory
      if (kHeld)
        sub1::waited_on(token, a.wo_tiles);
      else
        leave_token(a, token);
    }
    if (!kHeld && help < 0) break;
    help = -1;   // (its own tile next)
  }
  if (kHeld && threadIdx.x == 0) sub1::leave_launch(a.ctrl, gridDim.x);
}

__global__ void zero_i32_kernel(int32_t *p, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// ------------------------------------------------- derived-table cache -----

struct TableSlot {
  int device;
  const int32_t *dec;
  uint32_t *tab;          // kDictEntries table words, a flag word, kPrintWords of dec
  const int32_t *print;
};

std::mutex g_tab_mutex;
std::vector<TableSlot> g_tabs;
bool g_purged = false;   // the tables were dropped for the kFaultDec flag now standing

void drop_tables_locked(const int32_t *dec, bool all) {
  for (size_t i = 0; i < g_tabs.size();) {
    if (all || g_tabs[i].dec == dec) {
      (void)hipFree(g_tabs[i].tab);   // synchronises: no launch is still reading it
      g_tabs.erase(g_tabs.begin() + i);
    } else {
      i++;
    }
  }
}

// The compact table for `dec` on the current device, and the fault flags.  The
// first call with an address derives the table (one allocation, two small
// kernels, one synchronisation: not for a stream that is being captured).
int slot_table_for(const int32_t *dec, hipStream_t stream, TableSlot *out, int32_t **sticky) {
  int device = 0;
  HIP_TRY(hipGetDevice(&device));
  int rc = sub1::fault_words(sticky, true);
  if (rc) return rc;
  std::lock_guard<std::mutex> lock(g_tab_mutex);
  // a launch found other contents at a cached address: every cached table is
  // suspect, derive them afresh (once per raised flag)
  const bool flagged = sub1::fault_flag_host(sub1::kFaultDec);
  if (flagged && !g_purged) {
    drop_tables_locked(nullptr, true);
    g_purged = true;
  }
  if (!flagged) g_purged = false;
  for (const TableSlot &s : g_tabs)
    if (s.device == device && s.dec == dec) {
      *out = s;
      return SUB1_OK;
    }
  uint32_t *tab = nullptr;
  HIP_TRY(hipMalloc(&tab, (SUB1_DICT_ENTRIES + 64 + kPrintWords) * sizeof(uint32_t)));
  int32_t *flag = reinterpret_cast<int32_t *>(tab + SUB1_DICT_ENTRIES);
  int32_t *print = flag + 64;
  zero_i32_kernel<<<1, 64, 0, stream>>>(flag, 1);
  derive_slot_table_kernel<<<SUB1_DICT_ENTRIES / 256, 256, 0, stream>>>(dec, tab, flag);
  capture_print_kernel<<<1, 64, 0, stream>>>(dec, print);
  int32_t bad = 0;
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(&bad, flag, sizeof bad, hipMemcpyDeviceToHost, stream);
  if (e == hipSuccess) e = hipStreamSynchronize(stream);
  if (e != hipSuccess || bad) {
    (void)hipFree(tab);
    if (e != hipSuccess) return fail(SUB1_ERR_HIP, "deriving the table: %s", hipGetErrorString(e));
    return fail(SUB1_ERR_SHAPE,
                "dec holds an entry with a digit 3 or more than %d non-zero weights",
                kSlots);
  }
  g_tabs.push_back({device, dec, tab, print});
  *out = g_tabs.back();
  return SUB1_OK;
}

constexpr int kMoeThreads = 256;
constexpr int kGroupsAtOnce = 48 * kMoeThreads / 64;   // groups that a workgroup's wavefronts take in a turn, with room
constexpr int kPatienceUs = 20;          // all workgroups of a launch have started by then on a GPU that does nothing else
constexpr int kMoeSweepThreads = 1024;   // one workgroup per compute unit, the table's head in its LDS

hipEvent_t g_ev_begin = nullptr, g_ev_end = nullptr;

}  // namespace

// ================================================================ C ABI =====

extern "C" const char *sub1_last_error(void) { return sub1::g_err.c_str(); }

extern "C" const char *sub1_last_kernel(void) { return sub1::g_kernel; }

extern "C" int sub1_abi_version(void) { return 4; }

extern "C" int sub1_matvec_tokens(const int32_t *dec, const int16_t *w_comp,
                                  const int32_t *row_off, const void *ter_minmax,
                                  const void *x, void *y, int height, int width,
                                  int tokens, int64_t ldx, int64_t ldy, void *stream) {
  if (tokens == 0) return SUB1_OK;
  if (!dec || !row_off || !ter_minmax || !x || !y)
    return fail(SUB1_ERR_NULL, "sub1_matvec: NULL argument");
  if (height < 1 || width < 1)
    return fail(SUB1_ERR_SHAPE, "sub1_matvec: height %d width %d", height, width);
  if (tokens < 0 || tokens > 65535)
    return fail(SUB1_ERR_SHAPE, "sub1_matvec: tokens %d outside 0..65535", tokens);
  if (tokens > 1 && (ldx < width || ldy < height))
    return fail(SUB1_ERR_SHAPE, "sub1_matvec: row strides smaller than the rows");
  if (!w_comp) return fail(SUB1_ERR_NULL, "sub1_matvec: NULL w_comp");
  if (misaligned(dec, 4) || misaligned(row_off, 4) || misaligned(ter_minmax, 4) ||
      misaligned(w_comp, 2) || misaligned(x, 2) || misaligned(y, 2))
    return fail(SUB1_ERR_ALIGN, "sub1_matvec: misaligned pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  constexpr int kWaves = 4;   // rows per workgroup
  dim3 grid((height + kWaves - 1) / kWaves, tokens);
  sub1::note_kernel("matvec_wave_kernel<4>");
  matvec_wave_kernel<kWaves><<<grid, 64 * kWaves, 0, s>>>(
      dec, reinterpret_cast<const uint16_t *>(w_comp), row_off,
      static_cast<const uint32_t *>(ter_minmax), static_cast<const uint16_t *>(x),
      static_cast<uint16_t *>(y), height, width, ldx, ldy);
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}

extern "C" int sub1_matvec(const int32_t *dec, const int16_t *w_comp,
                           const int32_t *row_off, const void *ter_minmax,
                           const void *x, void *y, int height, int width,
                           void *stream) {
  return sub1_matvec_tokens(dec, w_comp, row_off, ter_minmax, x, y, height, width, 1,
                            width, height, stream);
}

namespace {

int launch_decode(const int32_t *dec, const int16_t *w_comp, const int32_t *row_off, const void *ter_minmax,
                  uint8_t *out_tern, void *out_w, int32_t *bad_rows, int32_t *counted, int height, int width,
                  hipStream_t s, const char *who) {
  if (!dec || !w_comp || !row_off) return fail(SUB1_ERR_NULL, "%s: NULL argument", who);
  if (out_w && !ter_minmax) return fail(SUB1_ERR_NULL, "%s: out_w needs ter_minmax", who);
  if (height < 1 || width < 1)
    return fail(SUB1_ERR_SHAPE, "%s: height %d width %d", who, height, width);
  if (misaligned(dec, 4) || misaligned(row_off, 4) || misaligned(w_comp, 2) ||
      misaligned(ter_minmax, 4) || misaligned(out_w, 2) || misaligned(bad_rows, 4))
    return fail(SUB1_ERR_ALIGN, "%s: misaligned pointer", who);
  sub1::AnswerSlot slot;
  if (counted) {
    const int rc = slot.take(s, who);
    if (rc) return rc;
    bad_rows = slot.answer().count;
  }
  // Whole words go out where both outputs begin theirs at the same elements; else
  // (an output that begins within a word) the symbols and the weights each in a launch
  constexpr int kWaves = 4;
  auto launch = [&](uint8_t *tern, uint16_t *w, int32_t *bad, int phase) {
    decode_kernel<kWaves><<<(height + kWaves - 1) / kWaves, 64 * kWaves, 0, s>>>(
        dec, reinterpret_cast<const uint16_t *>(w_comp), row_off,
        static_cast<const uint32_t *>(ter_minmax), tern, w, bad, height, width, phase);
  };
  uint16_t *w = static_cast<uint16_t *>(out_w);
  const int tern_phase = static_cast<int>(reinterpret_cast<uintptr_t>(out_tern) & 3);
  const int w_phase = static_cast<int>((reinterpret_cast<uintptr_t>(out_w) & 7) / 2);
  const bool each = out_tern && w && tern_phase != w_phase;
  launch(out_tern, each ? nullptr : w, bad_rows, out_tern ? tern_phase : w_phase);
  HIP_TRY(hipGetLastError());
  if (counted) {
    const int rc = slot.launched(who);
    if (rc) return rc;
  }
  if (each) {
    launch(nullptr, w, nullptr, w_phase);
    HIP_TRY(hipGetLastError());
  }
  if (!counted) return SUB1_OK;
  tell_count_kernel<<<1, 1, 0, s>>>(slot.answer());
  HIP_TRY(hipGetLastError());
  return slot.wait(s, 1, counted, who);
}

}  // namespace

extern "C" int sub1_decode(const int32_t *dec, const int16_t *w_comp, const int32_t *row_off,
                           const void *ter_minmax, uint8_t *out_tern, void *out_w, int32_t *bad_rows,
                           int height, int width, void *stream) {
  return launch_decode(dec, w_comp, row_off, ter_minmax, out_tern, out_w, bad_rows, nullptr, height, width,
                       static_cast<hipStream_t>(stream), "sub1_decode");
}

extern "C" int sub1_decode_counted(const int32_t *dec, const int16_t *w_comp, const int32_t *row_off,
                                   const void *ter_minmax, uint8_t *out_tern, void *out_w, int32_t *bad_rows,
                                   int height, int width, void *stream) {
  if (!bad_rows) return fail(SUB1_ERR_NULL, "sub1_decode_counted: NULL argument");
  return launch_decode(dec, w_comp, row_off, ter_minmax, out_tern, out_w, nullptr, bad_rows, height, width,
                       static_cast<hipStream_t>(stream), "sub1_decode_counted");
}

extern "C" int64_t sub1_moe_workspace_bytes(int tokens, int d_ff) {
  if (tokens < 0 || d_ff < 0) return 0;
  return sub1::control_bytes(tokens) + static_cast<int64_t>(tokens) * d_ff * 2;
}

extern "C" int sub1_moe_grouped(const sub1_moe_stack *st, const int32_t *token_expert,
                                const void *x, void *y, int tokens, void *workspace,
                                int64_t workspace_bytes, void *stream) {
  if (!st) return fail(SUB1_ERR_NULL, "sub1_moe_grouped: NULL stack");
  if (tokens == 0) return SUB1_OK;
  if (!token_expert || !x || !y)
    return fail(SUB1_ERR_NULL, "sub1_moe_grouped: NULL argument");
  if (!st->dec || !st->w_comp || !st->wi_code_base || !st->wo_code_base ||
      !st->wi_row_off || !st->wo_row_off || !st->wi_minmax || !st->wo_minmax)
    return fail(SUB1_ERR_NULL, "sub1_moe_grouped: NULL pointer in the stack");
  if (st->experts < 1 || st->d_model < 1 || st->d_ff < 1 ||
      st->d_model > SUB1_MAX_WIDTH || st->d_ff > SUB1_MAX_WIDTH)
    return fail(SUB1_ERR_SHAPE, "sub1_moe_grouped: experts %d d_model %d d_ff %d (sizes 1..%d)",
                st->experts, st->d_model, st->d_ff, SUB1_MAX_WIDTH);
  if (tokens < 0 || tokens > (1 << 20))
    return fail(SUB1_ERR_SHAPE, "sub1_moe_grouped: tokens %d outside 0..2^20", tokens);
  if (!workspace || workspace_bytes < sub1_moe_workspace_bytes(tokens, st->d_ff))
    return fail(SUB1_ERR_SHAPE, "sub1_moe_grouped: workspace of %lld bytes needed",
                static_cast<long long>(sub1_moe_workspace_bytes(tokens, st->d_ff)));
  if (misaligned(workspace, 256) || misaligned(st->dec, 4) || misaligned(st->w_comp, 2) ||
      misaligned(st->wi_code_base, 8) || misaligned(st->wo_code_base, 8) ||
      misaligned(st->wi_row_off, 4) || misaligned(st->wo_row_off, 4) ||
      misaligned(st->wi_minmax, 4) || misaligned(st->wo_minmax, 4) ||
      misaligned(token_expert, 4) || misaligned(x, 2) || misaligned(y, 2))
    return fail(SUB1_ERR_ALIGN, "sub1_moe_grouped: misaligned pointer");

  hipStream_t s = static_cast<hipStream_t>(stream);
  TableSlot slot;
  int32_t *sticky = nullptr;
  int rc = slot_table_for(st->dec, s, &slot, &sticky);
  if (rc) return rc;

  MoeArgs a;
  a.tab = slot.tab;
  a.dec = st->dec;
  a.print = slot.print;
  a.sticky = sticky;
  a.w_comp = reinterpret_cast<const uint16_t *>(st->w_comp);
  a.wi_code_base = st->wi_code_base;
  a.wo_code_base = st->wo_code_base;
  a.wi_row_off = st->wi_row_off;
  a.wo_row_off = st->wo_row_off;
  a.wi_minmax = static_cast<const uint32_t *>(st->wi_minmax);
  a.wo_minmax = static_cast<const uint32_t *>(st->wo_minmax);
  a.token_expert = token_expert;
  a.x = static_cast<const uint16_t *>(x);
  a.y = static_cast<uint16_t *>(y);
  a.ctrl = static_cast<int32_t *>(workspace);
  a.h = reinterpret_cast<uint16_t *>(sub1::h_base(workspace, workspace_bytes, tokens, st->d_ff));
  a.tokens = tokens;
  a.d_model = st->d_model;
  a.d_ff = st->d_ff;
  a.experts = st->experts;
  a.wait_ticks = sub1::wait_limit_ticks();
  a.patience = sub1::ticks_of(kPatienceUs);
  a.late = sub1::ticks_of(sub1::g_late_us.load());
  int device = 0, cus = 0;
  HIP_TRY(hipGetDevice(&device));
  HIP_TRY(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
  const int wmax = st->d_model > st->d_ff ? st->d_model : st->d_ff;
  a.act_dwords = lds_dwords_for_width(wmax);
  // One workgroup of 16 wavefronts per compute unit with all the LDS that the
  // activations leave for the table's first words, or workgroups of 4 wavefronts
  // and the table from memory, which from some 90 million weights on takes longer:
  // base shapes, 16, 32 and 48 tokens 42, 46 and 48 us against 23, 35 and 51; large ones, 16 and 24 tokens
  // 44 and 48 against 37 and 51; c-2048, 4, 8 and 12 tokens 57, 58 and 61 against 36, 50 and 64.
  constexpr size_t lds_limit = sub1::kMostLds - kMoeSweepThreads * sizeof(float2);
  constexpr size_t most_activations = lds_dwords_for_width(SUB1_MAX_WIDTH) * sizeof(float);
  static_assert(most_activations + 16384 * sizeof(uint32_t) <= lds_limit,
                "room for a head of the table beside any activations");
  const bool sweep = tokens >= cus || (tokens >= 10 && static_cast<int64_t>(tokens) * st->d_model * st->d_ff >= 90000000);
  a.held = 0;
  int64_t grid = cus;
  if (sweep) {
    const size_t room = (lds_limit - a.act_dwords * sizeof(float)) / sizeof(uint32_t) / 4 * 4;
    a.held = static_cast<int>(room < SUB1_DICT_ENTRIES ? room : SUB1_DICT_ENTRIES);
    // Parts of a projection: the number with which its tiles take the least time in
    // rounds of the grid.  A tile costs about 8 us (ticket, activations, the wait, the
    // wavefronts that finish early) besides its share of the projection, of which a
    // compute unit takes some 80 000 weights a microsecond.
    const double tile_share = 8.0 * 80000.0 / (static_cast<double>(st->d_model) * st->d_ff);
    constexpr int least_rows = kMoeSweepThreads / 4;   // of a tile
    auto parts_of = [&](int height) {
      int best = 1;
      double best_cost = 1e30;
      for (int parts = 1; parts <= std::max(1, height / least_rows); parts++) {
        const int64_t rounds = (static_cast<int64_t>(tokens) * parts + grid - 1) / grid;
        const double cost = rounds * (1.0 / parts + tile_share);
        if (cost < best_cost - 1e-9) {
          best_cost = cost;
          best = parts;
        }
      }
      return best;
    };
    a.wi_tiles = parts_of(st->d_ff);
    a.wo_tiles = parts_of(st->d_model);
  } else {
    // A workgroup for every tile.  As many tiles as give every wavefront a turn of its
    // own (64 groups, of which a row of W weights with 90 % zeros has W / 736 and a half), more where compute
    // units would have none, and at most one of either projection for each.  (More are slower again:
    // each counts itself and asks for words of the table.  Base and c-2048 shapes, 48, 96 and 192 tiles a
    // token, us: one token 17.4, 19.7, 26.6 and 29.9, 22.9, 29.4.)
    const auto tiles_of = [&](int height, int width) {
      const int turns = static_cast<int>(height * (width / 736.0 + 0.5) / kGroupsAtOnce) + 1;
      return std::min({std::max(turns, std::min(48, cus / (2 * tokens))), cus / tokens, (height + 3) / 4, kMostClaims});
    };
    a.wi_tiles = tiles_of(st->d_ff, st->d_model);
    a.wo_tiles = tiles_of(st->d_model, st->d_ff);
  }
  const size_t lds = (static_cast<size_t>(a.act_dwords) + a.held) * sizeof(float);
  if (sweep)
    HIP_TRY(sub1::allow_lds<lds_limit>(moe_kernel<kMoeSweepThreads>));
  else
    HIP_TRY(sub1::allow_lds<most_activations>(moe_kernel<kMoeThreads>));
  a.wi_expect = a.wi_tiles + sub1::expect_extra();
  const int64_t tiles = static_cast<int64_t>(tokens) * (a.wi_tiles + a.wo_tiles);
  if (tiles > INT32_MAX - (1 << 20))
    return fail(SUB1_ERR_SHAPE, "sub1_moe_grouped: too many tiles");

  if (sweep) {
    sub1::note_kernel("moe_kernel<1024>");
    moe_kernel<kMoeSweepThreads><<<static_cast<unsigned>(std::min(grid, tiles)), kMoeSweepThreads, lds, s>>>(a);
  } else {
    sub1::note_kernel("moe_kernel<256>");
    moe_kernel<kMoeThreads><<<static_cast<unsigned>(tiles), kMoeThreads, lds, s>>>(a);
  }
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}

// ---------------------------------------------------------- routing ------
//
// A wavefront per token: the first largest element of the token's row of the
// router's mask (what torch.argmax returns, reference sub1.py:311) and whether
// the row has a non-zero element at all (a token that the router's capacity
// limit dropped has none and keeps its input, reference sub1.py:312-318).
template <typename T>
__global__ __launch_bounds__(256) void route_from_mask_kernel(const T *__restrict__ mask,
                                                              int tokens, int experts,
                                                              int32_t *__restrict__ route,
                                                              int64_t *__restrict__ index) {
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= tokens) return;
  const int lane = threadIdx.x & 63;
  const T *row = mask + static_cast<int64_t>(t) * experts;
  long long best = 0;
  int at = experts;   // no element yet
  bool any = false;
  for (int e = lane; e < experts; e += 64) {
    const long long v = static_cast<long long>(row[e]);
    any = any || v != 0;
    if (at == experts || v > best) {
      best = v;
      at = e;
    }
  }
  // the lanes' candidates, largest value first, lowest index among equals
  for (int m = 1; m < 64; m <<= 1) {
    const long long v = __shfl_xor(best, m, 64);
    const int a = __shfl_xor(at, m, 64);
    if (a < experts && (at == experts || v > best || (v == best && a < at))) {
      best = v;
      at = a;
    }
  }
  const bool some = __ballot(any) != 0ull;
  if (lane == 0) {
    route[t] = some ? at : -1;
    if (index) index[t] = at;
  }
}

extern "C" int sub1_route_from_mask(const void *mask, int element_bytes, int tokens, int experts,
                                    int32_t *route, int64_t *expert_index, void *stream) {
  if (!mask || !route) return fail(SUB1_ERR_NULL, "sub1_route_from_mask: NULL argument");
  if (tokens < 0 || experts < 1)
    return fail(SUB1_ERR_SHAPE, "sub1_route_from_mask: tokens %d experts %d", tokens, experts);
  if (element_bytes != 1 && element_bytes != 4 && element_bytes != 8)
    return fail(SUB1_ERR_SHAPE, "sub1_route_from_mask: elements of %d bytes (1, 4 or 8)",
                element_bytes);
  if (misaligned(mask, element_bytes) || misaligned(route, 4) || misaligned(expert_index, 8))
    return fail(SUB1_ERR_ALIGN, "sub1_route_from_mask: misaligned pointer");
  if (tokens == 0) return SUB1_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const unsigned grid = static_cast<unsigned>((tokens + 3) / 4);
  if (element_bytes == 8)
    route_from_mask_kernel<<<grid, 256, 0, s>>>(static_cast<const int64_t *>(mask), tokens,
                                                experts, route, expert_index);
  else if (element_bytes == 4)
    route_from_mask_kernel<<<grid, 256, 0, s>>>(static_cast<const int32_t *>(mask), tokens,
                                                experts, route, expert_index);
  else
    route_from_mask_kernel<<<grid, 256, 0, s>>>(static_cast<const uint8_t *>(mask), tokens,
                                                experts, route, expert_index);
  HIP_TRY(hipGetLastError());
  return SUB1_OK;
}

extern "C" int sub1_fault_flags(int32_t *flags) {
  if (!flags) return fail(SUB1_ERR_NULL, "sub1_fault_flags: NULL argument");
  flags[0] = sub1::fault_flag_host(sub1::kFaultWait) ? 1 : 0;
  flags[1] = sub1::fault_flag_host(sub1::kFaultDec) ? 1 : 0;
  return SUB1_OK;
}

extern "C" const int32_t *sub1_fault_words_host(void) {
  std::lock_guard<std::mutex> lock(sub1::g_fault_mutex);
  return sub1::g_fault_host;
}

// Wait faults cleared so far.  A wait that gave up may have left the control
// words of its workspace at other values than zero (a writer that reports after
// the waiters have given up and cleared the word), and nothing in a later
// launch would notice: whoever owns a workspace compares this count with the
// one it saw when it last zeroed the buffer, and zeroes it again when they
// differ (ExpertStack.workspace and PreparedStack.workspace do).
std::atomic<int64_t> g_fault_epoch{0};

extern "C" int64_t sub1_fault_epoch(void) { return g_fault_epoch.load(); }

extern "C" int sub1_clear_faults(void) {
  // a standing kFaultDec flag means a cached table is stale: drop them all, so
  // that the calls after the reset derive theirs afresh
  if (sub1::fault_flag_host(sub1::kFaultDec)) {
    std::lock_guard<std::mutex> lock(g_tab_mutex);
    drop_tables_locked(nullptr, true);
  }
  if (sub1::fault_flag_host(sub1::kFaultWait)) g_fault_epoch.fetch_add(1);
  std::lock_guard<std::mutex> lock(sub1::g_fault_mutex);
  if (sub1::g_fault_host)
    for (int i = 0; i < sub1::kFaultWords; i++)
      *const_cast<volatile int32_t *>(&sub1::g_fault_host[i]) = 0;
  return SUB1_OK;
}

extern "C" int sub1_set_wait_limit_us(int64_t microseconds) {
  if (microseconds < 1 || microseconds > 60000000)
    return fail(SUB1_ERR_SHAPE, "sub1_set_wait_limit_us: %lld outside 1..60000000",
                static_cast<long long>(microseconds));
  sub1::g_wait_limit_us.store(microseconds);
  return SUB1_OK;
}

extern "C" int sub1_test_overstate_wait(int extra) {
  if (extra < 0) return fail(SUB1_ERR_SHAPE, "sub1_test_overstate_wait: negative count");
  sub1::g_expect_extra.store(extra);
  return SUB1_OK;
}

extern "C" int sub1_test_fail_answers(int calls) {
  if (calls < 0) return fail(SUB1_ERR_SHAPE, "sub1_test_fail_answers: negative count");
  sub1::g_fail_answers.store(calls);
  return SUB1_OK;
}

extern "C" int sub1_test_late_tiles(int microseconds) {
  if (microseconds < 0 || microseconds > 10000)
    return fail(SUB1_ERR_SHAPE, "sub1_test_late_tiles: %d us outside 0..10000", microseconds);
  sub1::g_late_us.store(microseconds);
  return SUB1_OK;
}

extern "C" int sub1_test_slot_pool(int slots, int lost) {
  const char *who = "sub1_test_slot_pool";
  if (lost < 0 || slots <= lost || slots > 4096) return fail(SUB1_ERR_SHAPE, "%s: %d of %d", who, lost, slots);
  sub1::SlotPool pool(slots);
  std::vector<int> held;
  for (int i = 0; i < slots; i++) held.push_back(pool.take());
  std::sort(held.begin(), held.end());
  for (int i = 0; i < slots; i++)
    if (held[i] != i) return fail(SUB1_ERR_INTERNAL, "%s: a slot was handed out twice", who);
  for (int i = 0; i < lost; i++) pool.lose();
  int got = -2;
  std::thread waits([&]() { got = pool.take(); });
  pool.give_back(held.back());
  waits.join();
  if (got != held.back()) return fail(SUB1_ERR_INTERNAL, "%s: %d taken, %d was free", who, got, held.back());
  got = -2;
  std::thread waits_for_none([&]() { got = pool.take(); });
  for (int i = lost; i < slots; i++) pool.lose();
  waits_for_none.join();
  if (got != -1 || pool.take() != -1) return fail(SUB1_ERR_INTERNAL, "%s: a lost slot was handed out", who);
  return SUB1_OK;
}

extern "C" int sub1_unregister_dec(const int32_t *dec) {
  std::lock_guard<std::mutex> lock(g_tab_mutex);
  drop_tables_locked(dec, dec == nullptr);
  return SUB1_OK;
}

extern "C" int sub1_timing_begin(void *stream) {
  if (!g_ev_begin) {
    HIP_TRY(hipEventCreate(&g_ev_begin));
    HIP_TRY(hipEventCreate(&g_ev_end));
  }
  HIP_TRY(hipEventRecord(g_ev_begin, static_cast<hipStream_t>(stream)));
  return SUB1_OK;
}

extern "C" int sub1_timing_end(void *stream, double *elapsed_us) {
  if (!g_ev_begin) return fail(SUB1_ERR_INTERNAL, "sub1_timing_end without sub1_timing_begin");
  if (!elapsed_us) return fail(SUB1_ERR_NULL, "sub1_timing_end: NULL argument");
  HIP_TRY(hipEventRecord(g_ev_end, static_cast<hipStream_t>(stream)));
  HIP_TRY(hipEventSynchronize(g_ev_end));
  float ms = 0.f;
  HIP_TRY(hipEventElapsedTime(&ms, g_ev_begin, g_ev_end));
  *elapsed_us = 1e3 * static_cast<double>(ms);
  return SUB1_OK;
}
