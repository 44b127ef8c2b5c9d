// The expert layer on the matrix cores, for batches with many tokens per expert:
// device code that sub1_prepared.hip includes (it reads the prepared stream).
//
// Walking the stream costs an LDS read per weight and four tokens; with tens of
// tokens per expert it is cheaper to expand a slice once and multiply on the matrix
// cores.  Expanding does not make dense weights: a slice of 64 rows becomes codes of
// 2 bits in LDS, 256 bytes per 16 columns (768 columns: 12 KB, 6144: 98 KB), so a
// whole row fits whatever its length, and no form of the weights beside the stream
// is kept in memory.  Word g of row r lies at (64 g + r) * 4: a lane expands one
// row, so its writes never meet another lane's in a bank, wherever they go.  An
// entry costs nine plain instructions and an LDS `or` (walking: 3.5 and a random
// gather), then nothing per token.
//
// One launch: group_blocks_kernel gives every token a slot in a block of 32 of its
// expert's tokens; pack_tokens_kernel lays a block's activations out as MFMA
// operands; batch_product_kernel multiplies (wi, ReLU); pack_hidden_kernel lays h
// out; batch_product_kernel (wo); unpack_tokens_kernel writes y.  The products leave
// their rows as 64-byte runs of 32 tokens (rows come in the slices' order, so anything
// finer would be scattered), which the passes around them transpose.
//
// 128 base experts on 4096 tokens: 274 -> 132 us (group 7, pack 7, wi 45, h 13, wo 52, y 6,
// the listed tokens' launch 4), 40 c-2048 experts on 700 tokens 366 -> 167.  With the
// multiplying taken out the same launch takes 82, with the expanding 120: what bounds
// the products is the 24 instructions that make a step's two operands of weights, beside
// two MFMAs for every block of tokens (15 plain instructions an MFMA with up to 32 tokens, 8 with
// 64), then the start and end of workgroups that LDS holds to 12 to 16 wavefronts a compute unit.
// No unit is full (counters: VALUs 47 % busy, matrix cores 21, LDS 10): on average a launch has
// 1.9 wavefronts on a SIMD, each a chain of expanding, making operands and multiplying.
//
// A token whose activations or h hold an infinity or NaN is left to the walking
// kernel (0 x inf is NaN here, and a weight of zero adds nothing there), and so are the
// tokens of an expert with such a (min, max) (walking, every weight of its row meets it): the
// passes and the products mark them, and unpack_tokens_kernel lists them for the launch that follows.

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kBlockTokens = 32;     // tokens of an MFMA operand
constexpr int kChunkBlocks = 2;      // blocks that share an expansion
constexpr int kTurn = 2;             // steps whose operands are asked for together
constexpr int kStepColumns = 16;     // columns of an MFMA, and of a word of codes
constexpr int kBatchPiece = 8192;    // tokens of a launch sequence: bounds the scratch memory
constexpr int kBatchMaxExperts = 4096;   // group_blocks_kernel's tables in LDS

__host__ __device__ constexpr int steps_of(int width) { return (width + kStepColumns - 1) / kStepColumns; }
// A slice's codes in LDS; one row of words more, which stays zero: steps onto the last
// zero column name it, and a turn of steps may end with it.
__host__ __device__ constexpr int slice_code_bytes(int width) { return (steps_of(width) + 1) * 256; }

// Totals a launch's kernels read.
enum BatchTotals { kTotalChunks = 0, kTotalLive = 1, kTotalBlocks = 2, kTotalWords = 4 };

// Column of a step that slot k of an operand holds for a lane of half h.  Position p of
// the stream falls on bit p % 34 of word p / 34 (mod 32, bits 32 and 33 being column 15,
// 0 and 1 the zero column, which is not written): field j of a word, bits 2j and 2j + 1,
// is column j - 1 mod 16.  Byte b of a word holds fields 4b .. 4b + 3, and a lane of
// half h takes fields 2h (slots 0-3, byte by byte) and 2h + 1 (slots 4-7).
__host__ __device__ constexpr int slot_column(int h, int k) {
  return (4 * (k & 3) + 2 * h + (k >> 2) + 15) & 15;
}

struct BatchArgs {
  const uint2 *stream;
  const uint16_t *ckpt;
  KindArgs k;
  const u32x4 *in;        // [block][step][64 lanes]: 16-byte operands
  uint16_t *out;          // [block][height][32]
  const int4 *chunks;     // (expert, first block, blocks, 0)
  int32_t *spoiled;       // [slot]: left to the walking kernel
  const int32_t *totals;
  int steps, parts;       // parts: wavefronts that share a slice
  int per_group;          // slices of a workgroup
  int slice_groups;       // workgroups of a chunk
  int relu;
};

// The nine entries of a chunk onto the row's codes.  `at` is the position reached,
// `lane_codes` the row's word 0.  The stream's entries never leave the row (what pads
// a row stays on a zero column or repeats its last entry, which or's the same bit).
__device__ __forceinline__ void expand_chunk(uint2 cw, uint32_t &at, uint32_t *lane_codes) {
  const uint32_t mid = __builtin_amdgcn_alignbit(cw.y, cw.x, 28);
#pragma unroll
  for (int q = 0; q < kFields; q++) {
    const uint32_t step = q < 4 ? (cw.x >> (kFieldBits * q)) & 127u
                        : q < 8 ? (mid >> (kFieldBits * (q - 4))) & 127u
                                : (cw.y >> 24) & 127u;
    at += step;
    const uint32_t g = __umul24(at, 30841u) >> 20;   // at / 34, exact up to 50 000
    const uint32_t r = at - 34u * g;
    const uint32_t bit = r < 2u ? 0u : 1u << (r & 31u);
    __hip_atomic_fetch_or(lane_codes + g * 64u, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
}

// Two rows' weights (a lane's B operands of a step) from their words of codes.
struct RowBytes {
  uint32_t lo, hi;   // (0, min, max, 0): the values' lower bytes, and their upper ones
};
__device__ __forceinline__ RowBytes row_bytes(uint32_t min_max) {
  return RowBytes{__builtin_amdgcn_perm(0u, min_max, 0x0c02000cu),
                  __builtin_amdgcn_perm(0u, min_max, 0x0c03010cu)};
}
__device__ __forceinline__ bf16x8 weights_of(uint32_t word, int shift, const RowBytes &t) {
  u32x4 w;
#pragma unroll
  for (int f = 0; f < 2; f++) {
    const uint32_t at = (word >> (shift + 2 * f)) & 0x03030303u;
    const uint32_t lo = __builtin_amdgcn_perm(0u, t.lo, at), hi = __builtin_amdgcn_perm(0u, t.hi, at);
    w[2 * f] = __builtin_amdgcn_perm(hi, lo, 0x05010400u);
    w[2 * f + 1] = __builtin_amdgcn_perm(hi, lo, 0x07030602u);
  }
  return __builtin_bit_cast(bf16x8, w);
}

// Loads through a buffer are asked for where they stand (a loop that asks for its next
// turn's operands with plain loads is turned into one that loads them when it needs them).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void *base, int bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, bytes, 0x00020000);
}

// What a workgroup does: its slices' codes into LDS, then every wavefront's share of a
// slice's steps, then the sums of the wavefronts that share a slice, added in order and
// written.  Everything that is read from memory is asked for before the codes are expanded.
template <int kBlocks>
__device__ __forceinline__ void slices_times_tokens(const BatchArgs &a, uint32_t *lds, int e, int group,
                                                    int64_t first_block) {
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int local = wave / a.parts, sub = wave % a.parts;
  const int s = group * a.per_group + local;
  const bool mine = s < a.k.slices;
  const int64_t sl = static_cast<int64_t>(e) * a.k.slices + (mine ? s : 0);
  const int slice_words = (a.steps + 1) * 64;
  uint32_t *codes = lds + local * slice_words;

  const int len = a.k.slice_len[sl];
  const uint32_t base_word = a.k.slice_base[sl];
  uint32_t minmax[2];
  int row[2];
#pragma unroll
  for (int j = 0; j < 2; j++) {
    minmax[j] = a.k.minmax[sl * 64 + 32 * j + (lane & 31)];
    row[j] = a.k.row_idx[sl * 64 + 32 * j + (lane & 31)];
  }
  const int nch = chunks_of(__builtin_amdgcn_readfirstlane(len));
  const uint32_t base = __builtin_amdgcn_readfirstlane(base_word);
  const int groups = (nch + kGroupChunks - 1) / kGroupChunks;
  const int g_lo = mine ? sub * groups / a.parts : 0;
  const int g_hi = mine ? (sub + 1) * groups / a.parts : 0;
  const int c_end = min(g_hi * kGroupChunks, nch);
  const __amdgpu_buffer_rsrc_t stream = buffer_of(a.stream + static_cast<int64_t>(base) * 64, nch * 512);
  uint2 ring[kGroupChunks];
  auto ask_chunk = [&](int c, int i) {   // past the slice: zeros, steps that go nowhere
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(stream, lane * 8, (c + i) * 512, 0);
    ring[i] = make_uint2(v[0], v[1]);
  };
  uint32_t at = 0;
  if (g_lo < g_hi) {
    if (g_lo) at = a.ckpt[(checkpoint_entry(base, a.k.first_slice + sl) + g_lo) * 64 + lane];
#pragma unroll
    for (int i = 0; i < kGroupChunks; i++) ask_chunk(g_lo * kGroupChunks, i);
  }
  // whole turns of the steps; the last may go one step further, where the codes are zeros
  const int turns = (a.steps + kTurn - 1) / kTurn;
  const int lo = mine ? sub * turns / a.parts * kTurn : 0, hi = mine ? (sub + 1) * turns / a.parts * kTurn : 0;
  const __amdgpu_buffer_rsrc_t in = buffer_of(a.in + first_block * a.steps * 64, kBlocks * a.steps * 1024);
  u32x4 next[kTurn][kBlocks];
  auto ask = [&](int st) {
#pragma unroll
    for (int u = 0; u < kTurn; u++)
#pragma unroll
      for (int i = 0; i < kBlocks; i++)
        next[u][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
            in, lane * 16, (i * a.steps + min(st + u, a.steps - 1)) * 1024, 0));
  };
  if (lo < hi) ask(lo);

  const int all_words = a.per_group * slice_words;   // a multiple of 64
  for (int i = 4 * threadIdx.x; i < all_words; i += 4 * blockDim.x)
    *reinterpret_cast<uint4 *>(lds + i) = make_uint4(0u, 0u, 0u, 0u);
  // (an exponent of all ones in either half: the sum carries into its sign)
  const uint32_t high = ((minmax[0] & 0x7f807f80u) + 0x00800080u) | ((minmax[1] & 0x7f807f80u) + 0x00800080u);
  if ((high & 0x80008000u) && mine && sub == 0)
    for (int t = 0; t < kBlocks * kBlockTokens; t++) a.spoiled[first_block * kBlockTokens + t] = 1;
  __syncthreads();
#pragma unroll 1
  for (int c = g_lo * kGroupChunks; c < c_end; c += kGroupChunks) {
    uint2 now[kGroupChunks];
#pragma unroll
    for (int i = 0; i < kGroupChunks; i++) now[i] = ring[i];
    if (c + kGroupChunks < c_end)
#pragma unroll
      for (int i = 0; i < kGroupChunks; i++) ask_chunk(c + kGroupChunks, i);
#pragma unroll
    for (int i = 0; i < kGroupChunks; i++)
      if (c + i < c_end) expand_chunk(now[i], at, codes + lane);
  }
  __syncthreads();

  f32x16 acc[kBlocks][2];
#pragma unroll
  for (int i = 0; i < kBlocks; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = f32x16{};
  RowBytes rows[2];
#pragma unroll
  for (int j = 0; j < 2; j++) rows[j] = row_bytes(minmax[j]);
  const uint32_t *word = codes + (lane & 31);
#pragma unroll 1
  for (int st = lo; st < hi; st += kTurn) {
    u32x4 x[kTurn][kBlocks];
#pragma unroll
    for (int u = 0; u < kTurn; u++)
#pragma unroll
      for (int i = 0; i < kBlocks; i++) x[u][i] = next[u][i];
    uint32_t w[kTurn][2];
#pragma unroll
    for (int u = 0; u < kTurn; u++)
#pragma unroll
      for (int j = 0; j < 2; j++) w[u][j] = word[(st + u) * 64 + 32 * j];
    ask(st + kTurn);
#pragma unroll
    for (int u = 0; u < kTurn; u++) {
      const bf16x8 w0 = weights_of(w[u][0], 4 * half, rows[0]);
      const bf16x8 w1 = weights_of(w[u][1], 4 * half, rows[1]);
#pragma unroll
      for (int i = 0; i < kBlocks; i++) {
        const bf16x8 xv = __builtin_bit_cast(bf16x8, x[u][i]);
        acc[i][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xv, w0, acc[i][0], 0, 0, 0);
        acc[i][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(xv, w1, acc[i][1], 0, 0, 0);
      }
    }
  }

  // a lane has row 32 j + lane % 32 and tokens 8 g + 4 half + 0..3, values 4 g + 0..3
  auto write = [&](const float (&v)[4], int i, int j, int g) {
    if (!mine || row[j] == 0xffff) return;
    uint32_t w[2];
#pragma unroll
    for (int m = 0; m < 2; m++) {
      float lower = v[2 * m], upper = v[2 * m + 1];
      if (a.relu) {
        lower = __uint_as_float(max(__float_as_int(lower), 0));
        upper = __uint_as_float(max(__float_as_int(upper), 0));
      }
      const bf16x2 pair = {static_cast<__bf16>(lower), static_cast<__bf16>(upper)};
      w[m] = __builtin_bit_cast(uint32_t, pair);
    }
    *reinterpret_cast<uint2 *>(a.out + ((first_block + i) * a.k.height + row[j]) * kBlockTokens + 8 * g + 4 * half) =
        make_uint2(w[0], w[1]);
  };
  if (a.parts == 1) {
#pragma unroll
    for (int i = 0; i < kBlocks; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const float v[4] = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
          write(v, i, j, g);
        }
    return;
  }
  float4 *sums = reinterpret_cast<float4 *>(lds);
  __syncthreads();   // every wavefront is through with the codes, whose place the sums take
#pragma unroll
  for (int i = 0; i < kBlocks; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) {
      // a tile at a time, in one of two places; the parts share its groups of four values
      float4 *place = sums + ((2 * i + j) & 1) * waves * 256;
#pragma unroll
      for (int g = 0; g < 4; g++)
        place[wave * 256 + g * 64 + lane] =
            make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
      __syncthreads();
      for (int g = sub; g < 4; g += a.parts) {
        const float4 *from = place + (wave - sub) * 256 + g * 64 + lane;
        float4 sum = from[0];
        for (int p = 1; p < a.parts; p++) {
          const float4 v = from[p * 256];
          sum.x += v.x;
          sum.y += v.y;
          sum.z += v.z;
          sum.w += v.w;
        }
        const float v[4] = {sum.x, sum.y, sum.z, sum.w};
        write(v, i, j, g);
      }
    }
}

__global__ __launch_bounds__(kMaxThreads) void batch_product_kernel(BatchArgs a) {
  extern __shared__ __align__(16) uint32_t lds[];
  // the workgroups of a chunk, which read the same activations, run on one die
  const int die = blockIdx.x & 7, turn = blockIdx.x >> 3;
  const int chunk = turn / a.slice_groups * 8 + die;
  const int group = turn % a.slice_groups;
  const int total = a.totals[kTotalChunks];
  const int4 what = a.chunks[chunk];   // (there is room for a whole turn of them)
  if (chunk >= total) return;
  const int e = __builtin_amdgcn_readfirstlane(what.x);
  const int first_block = __builtin_amdgcn_readfirstlane(what.y);
  if (__builtin_amdgcn_readfirstlane(what.z) > 1)
    slices_times_tokens<2>(a, lds, e, group, first_block);
  else
    slices_times_tokens<1>(a, lds, e, group, first_block);
}

// One workgroup.  Every token gets a slot: its expert's tokens fill blocks of 32, an
// expert's blocks lie together, those of tokens without an expert come last.
__global__ __launch_bounds__(1024) void group_blocks_kernel(
    const int32_t *__restrict__ token_expert, int tokens, int experts, int32_t *__restrict__ slots,
    int32_t *__restrict__ spoiled, int32_t *__restrict__ block_expert, int4 *__restrict__ chunks,
    int32_t *__restrict__ totals, int32_t *__restrict__ ctrl) {
  extern __shared__ __align__(16) int32_t table[];
  __shared__ int32_t wave_blocks[16], wave_chunks[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int buckets = experts + 1;
  int32_t *count = table, *next = table + buckets;
  for (int b = tid; b < buckets; b += 1024) count[b] = 0;
  __syncthreads();
  int faults = 0;
  int bucket[kBatchPiece / 1024];
#pragma unroll
  for (int i = 0; i < kBatchPiece / 1024; i++) {
    const int t = i * 1024 + tid;
    const int e = t < tokens ? token_expert[t] : -1;
    if (e >= experts) faults++;
    bucket[i] = e < 0 || e >= experts ? experts : e;
  }
#pragma unroll
  for (int i = 0; i < kBatchPiece / 1024; i++)
    if (i * 1024 + tid < tokens) atomicAdd(&count[bucket[i]], 1);
  if (faults) atomicAdd(&ctrl[kCtrlBadIds], faults);
  __syncthreads();
  const int seg = (buckets + 1023) / 1024;
  const int lo = min(tid * seg, buckets), hi = min(lo + seg, buckets);
  auto blocks_of = [](int n) { return (n + kBlockTokens - 1) / kBlockTokens; };
  auto chunks_in = [](int n) { return (n + kChunkBlocks - 1) / kChunkBlocks; };
  int32_t n_blocks = 0, n_chunks = 0;
  for (int b = lo; b < hi; b++) {
    const int n = blocks_of(count[b]);
    n_blocks += n;
    if (b != experts) n_chunks += chunks_in(n);
  }
  int32_t up_blocks = n_blocks, up_chunks = n_chunks;
  for (int d = 1; d < 64; d <<= 1) {
    const int32_t u = __shfl_up(up_blocks, d, 64), v = __shfl_up(up_chunks, d, 64);
    if (lane >= d) {
      up_blocks += u;
      up_chunks += v;
    }
  }
  if (lane == 63) {
    wave_blocks[wave] = up_blocks;
    wave_chunks[wave] = up_chunks;
  }
  __syncthreads();
  int32_t block = up_blocks - n_blocks, chunk = up_chunks - n_chunks;
  for (int w = 0; w < wave; w++) {
    block += wave_blocks[w];
    chunk += wave_chunks[w];
  }
  for (int b = lo; b < hi; b++) {
    const int n = count[b], nb = blocks_of(n);
    next[b] = block * kBlockTokens;
    for (int i = n; i < nb * kBlockTokens; i++) slots[block * kBlockTokens + i] = -1;
    for (int i = 0; i < nb; i++) block_expert[block + i] = b == experts ? -1 : b;
    if (b == experts) {
      totals[kTotalChunks] = chunk;
      totals[kTotalLive] = block;
      totals[kTotalBlocks] = block + nb;
      ctrl[kCtrlTiles] = 0;
    } else {
      for (int i = 0; i < nb; i += kChunkBlocks)
        chunks[chunk++] = make_int4(b, block + i, min(kChunkBlocks, nb - i), 0);
    }
    block += nb;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kBatchPiece / 1024; i++) {
    const int t = i * 1024 + tid;
    if (t < tokens) {
      const int place = atomicAdd(&next[bucket[i]], 1);
      slots[place] = t;
      spoiled[place] = 0;
    }
  }
}

__device__ __forceinline__ bool not_finite(uint32_t bits) { return (bits & 0x7f80u) == 0x7f80u; }

// A step's 16 columns of a token (bits, zeros past the width) as its two operands.
__device__ __forceinline__ void write_operands(u32x4 *out, int64_t step, int t, const uint16_t (&v)[16]) {
#pragma unroll
  for (int h = 0; h < 2; h++) {
    u32x4 w;
#pragma unroll
    for (int k = 0; k < 4; k++)
      w[k] = v[slot_column(h, 2 * k)] | static_cast<uint32_t>(v[slot_column(h, 2 * k + 1)]) << 16;
    out[step * 64 + h * 32 + t] = w;
  }
}

// x by blocks of 32 slots into operands; tokens without an expert keep their input.
__global__ __launch_bounds__(256) void pack_tokens_kernel(
    const uint16_t *x, uint16_t *y, int64_t ldx, int64_t ldy, int width, bool aligned,
    const int32_t *__restrict__ slots, int32_t *__restrict__ spoiled, const int32_t *__restrict__ totals,
    u32x4 *__restrict__ out) {
  const int block = blockIdx.x;
  if (block >= totals[kTotalBlocks]) return;
  const int steps = steps_of(width);
  const int t = threadIdx.x & 31;
  const int token = slots[block * kBlockTokens + t];
  const bool live = block < totals[kTotalLive];
  const uint16_t *from = x + (token < 0 ? 0 : token) * ldx;
  bool bad = false;
  for (int st = blockIdx.y * 8 + (threadIdx.x >> 5); st < steps; st += gridDim.y * 8) {
    const int c = st * kStepColumns;
    uint16_t v[16];
    if (token < 0) {
#pragma unroll
      for (int i = 0; i < 16; i++) v[i] = 0;
    } else if (aligned && c + 16 <= width) {
      const uint4 a = *reinterpret_cast<const uint4 *>(from + c);
      const uint4 b = *reinterpret_cast<const uint4 *>(from + c + 8);
      __builtin_memcpy(v, &a, 16);
      __builtin_memcpy(v + 8, &b, 16);
    } else {
#pragma unroll
      for (int i = 0; i < 16; i++) v[i] = c + i < width ? from[c + i] : 0;
    }
    if (live) {
#pragma unroll
      for (int i = 0; i < 16; i++) bad |= not_finite(v[i]);
      write_operands(out + static_cast<int64_t>(block) * steps * 64, st, t, v);
    } else if (token >= 0) {
      for (int i = 0; i < 16; i++)
        if (c + i < width) y[token * ldy + c + i] = v[i];
    }
  }
  if (bad) spoiled[block * kBlockTokens + t] = 1;
}

// h, rows of 32 tokens, into operands.
__global__ __launch_bounds__(256) void pack_hidden_kernel(
    const uint16_t *__restrict__ rows, int width, int32_t *__restrict__ spoiled,
    const int32_t *__restrict__ totals, u32x4 *__restrict__ out) {
  const int block = blockIdx.x;
  if (block >= totals[kTotalLive]) return;
  const int steps = steps_of(width);
  const int pair = threadIdx.x & 15;   // tokens 2 pair and 2 pair + 1
  const uint32_t *from = reinterpret_cast<const uint32_t *>(rows + static_cast<int64_t>(block) * width * kBlockTokens) + pair;
  uint32_t bad = 0;
  for (int st = blockIdx.y * 16 + (threadIdx.x >> 4); st < steps; st += gridDim.y * 16) {
    uint16_t v[2][16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
      const int c = st * kStepColumns + i;
      const uint32_t w = c < width ? from[c * (kBlockTokens / 2)] : 0u;
      v[0][i] = static_cast<uint16_t>(w);
      v[1][i] = static_cast<uint16_t>(w >> 16);
      if (not_finite(w)) bad |= 1;
      if (not_finite(w >> 16)) bad |= 2;
    }
#pragma unroll
    for (int m = 0; m < 2; m++)
      write_operands(out + static_cast<int64_t>(block) * steps * 64, st, 2 * pair + m, v[m]);
  }
#pragma unroll
  for (int m = 0; m < 2; m++)
    if (bad >> m & 1) spoiled[block * kBlockTokens + 2 * pair + m] = 1;
}

// y from rows of 32 tokens; spoiled tokens are listed, one to a tile.
__global__ __launch_bounds__(256) void unpack_tokens_kernel(
    const uint16_t *__restrict__ rows, uint16_t *__restrict__ y, int64_t ldy, int height, bool aligned,
    const int32_t *__restrict__ slots, const int32_t *__restrict__ spoiled,
    const int32_t *__restrict__ block_expert, const int32_t *__restrict__ totals,
    int2 *__restrict__ tiles, int32_t *__restrict__ ctrl) {
  const int block = blockIdx.x;
  if (block >= totals[kTotalLive]) return;
  const int t = threadIdx.x & 31;
  const int slot = block * kBlockTokens + t;
  const int token = slots[slot];
  if (token < 0) return;
  if (spoiled[slot]) {
    if (blockIdx.y == 0 && threadIdx.x < 32)
      tiles[atomicAdd(&ctrl[kCtrlTiles], 1)] = make_int2(block_expert[block], slot);
    return;
  }
  const uint16_t *from = rows + static_cast<int64_t>(block) * height * kBlockTokens + t;
  uint16_t *to = y + token * ldy;
  for (int c = (blockIdx.y * 8 + (threadIdx.x >> 5)) * 8; c < height; c += gridDim.y * 64) {
    uint16_t v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = c + i < height ? from[(c + i) * kBlockTokens] : 0;
    if (aligned && c + 8 <= height) {
      uint4 w;
      __builtin_memcpy(&w, v, 16);
      *reinterpret_cast<uint4 *>(to + c) = w;
    } else {
      for (int i = 0; i < 8; i++)
        if (c + i < height) to[c + i] = v[i];
    }
  }
}

// The listed tokens (ctrl[kCtrlTiles] of them), a workgroup each, as
// moe_prepared_fused_kernel walks them: the same sums.  LDS: x | h.
__global__ __launch_bounds__(kMaxThreads) void walk_listed_kernel(PreparedArgs a) {
  extern __shared__ __align__(16) uint32_t lds[];
  const int listed = __builtin_amdgcn_readfirstlane(a.ctrl[kCtrlTiles]);
  if (static_cast<int>(blockIdx.x) >= listed) return;
  uint32_t *xa = lds, *ha = lds + a.xdwords;
  const int waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int i = threadIdx.x; i < a.hdwords; i += blockDim.x) ha[i] = 0u;
  for (int tile = blockIdx.x; tile < listed; tile += gridDim.x) {
    const int2 what = a.groups[tile];
    const int e = __builtin_amdgcn_readfirstlane(what.x);
    const int t = __builtin_amdgcn_readfirstlane(a.order[what.y]);
    __syncthreads();   // the previous token is through
    stage_activations(xa, a.x + static_cast<int64_t>(t) * a.ldx, a.k[0].width);
    __syncthreads();
    for (int s = wave; s < a.k[0].slices; s += waves) {
      SliceWalk w = load_slice(a, a.k[0], static_cast<int64_t>(e) * a.k[0].slices + s);
      const float res = run_slice(w, a.stream, xa);
      if (w.ridx != 0xffff) {
        uint32_t out = f32_to_bf16(res);
        if (out & 0x8000u) out = 0;
        uint32_t *p = ha + 2 * physical_column(w.ridx);
        p[0] = out;
        p[1] = out << 16;
      }
    }
    __syncthreads();
    for (int s = wave; s < a.k[1].slices; s += waves) {
      SliceWalk w = load_slice(a, a.k[1], static_cast<int64_t>(e) * a.k[1].slices + s);
      const float res = run_slice(w, a.stream, ha);
      write_row(a.y + static_cast<int64_t>(t) * a.ldy, w.ridx, res, kStore);
    }
  }
}
