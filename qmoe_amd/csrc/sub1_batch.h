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
// entry costs nine plain instructions and an LDS `or` (walking: 3.5 and a random gather), then
// nothing per token.
//
// wo takes its columns in the order in which wi's slices have their rows (seven
// instructions an entry and a look into a table that says where a column's code goes): wi's
// product, which has the weights as its first operand, then holds h just as wo's product
// wants it, eight columns of a token to a lane, and stores it so.  (With wo's columns in
// their own order h went out as rows of 32 tokens and through a pass that transposed
// it, 13 us of 133 below; y through another, 6, where its two-byte stores now go straight to
// the tokens' rows.)
//
// One launch: pack_blocks_kernel gives every token a slot in a block of 32 of its
// expert's tokens and lays a block's activations out as MFMA operands; batch_product_kernel<true> multiplies (wi, ReLU), batch_product_kernel<false>
// (wo); walk_spoiled_kernel walks what they leave.
//
// 128 base experts on 4096 tokens: walking 274 us, here 110 (133 with a pass for h and one for y);
// 40 c-2048 experts on 640 tokens 311 and 159 (167).  Under a profiler, one after the other:
// slots and x 9, wi 48, wo 60, marks 4.5.  Of the products' times multiplying is 27 each (with it taken
// out they take that less): the 24 instructions that make a step's two operands of weights, beside
// two MFMAs for every block of tokens, issued at 80 % of what the SIMDs can; expanding 8 and 12;
// starting, clearing LDS and adding up what the wavefronts of a slice have, in workgroups
// that leave no LDS for another one meanwhile, the rest.
//
// A token whose activations or h hold an infinity or NaN is left to the walking
// kernel (0 x inf is NaN here, and a weight of zero adds nothing there), and so are the
// tokens of an expert with such a (min, max) (walking, every weight of its row meets it): the
// pass over x and wi's product mark them, and walk_spoiled_kernel finds the marks.

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kBlockTokens = 32;     // tokens of an MFMA operand
constexpr int kChunkBlocks = 2;      // blocks that share an expansion
constexpr int kTurn = 4;             // steps whose operands are asked for together, and ahead
constexpr int kStepColumns = 16;     // columns of an MFMA, and of a word of codes
constexpr int kBatchPiece = 8192;    // tokens of a launch sequence: bounds the scratch memory
constexpr int kBatchMaxExperts = 4096;   // pack_blocks_kernel's counts in LDS

__host__ __device__ constexpr int steps_of(int width) { return (width + kStepColumns - 1) / kStepColumns; }
// Steps of a product over the rows of 64-row slices.
__host__ __device__ constexpr int steps_of_slices(int slices) { return slices * (64 / kStepColumns); }
// A slice's codes in LDS: whole turns of steps (zeros where the last is half a one), and a
// row of words that entries go to which stay on a zero column.
__host__ __device__ constexpr int idle_step(int steps) { return (steps + kTurn - 1) / kTurn * kTurn; }
__host__ __device__ constexpr int slice_code_bytes(int steps) { return (idle_step(steps) + 1) * 256; }
__host__ __device__ constexpr int table_bytes(int width) { return (physical_columns(width) * 2 + 15) / 16 * 16; }

// Totals a launch's kernels read.
enum BatchTotals { kTotalChunks = 0, kTotalLive = 1, kTotalBlocks = 2, kTotalWords = 4 };

// A word of codes holds a step's 16 columns: field j, bits 2j and 2j + 1, is 1 for a row
// min, 2 for a max, 0 for neither.  Byte b holds fields 4b .. 4b + 3, and a lane of half h
// takes fields 2h (places 0-3 of its operand, byte by byte) and 2h + 1 (places 4-7).  An entry of
// the table: the step in bits 5 and up, twice the field in bits 0-4.
__host__ __device__ constexpr uint32_t table_entry(int step, int half, int place) {
  return static_cast<uint32_t>(step << 5 | 2 * (4 * (place & 3) + 2 * half + (place >> 2)));
}
// x's columns keep their own order and need no table: position p of the stream falls on bit
// p % 34 of word p / 34 (mod 32, bits 32 and 33 being column 15, 0 and 1 the zero column, which
// is not written), so that field j is column j - 1 mod 16.
__host__ __device__ constexpr int column_of_place(int half, int place) {
  return (4 * (place & 3) + 2 * half + (place >> 2) + 15) & 15;
}
// Row r of a matrix's slices as the product of them leaves it in its lanes: of 32 rows a
// lane of half h has rows 8 g + 4 h + 0..3 for g = 0..3, which are two operands of eight.
__host__ __device__ constexpr uint32_t entry_of_row(int r) {
  return table_entry(r >> 4, (r >> 2) & 1, ((r >> 3) & 1) << 2 | (r & 3));
}

struct BatchArgs {
  const uint2 *stream;
  const uint16_t *ckpt;
  KindArgs k;
  const u32x4 *in;           // [block][step][64 lanes]: 16-byte operands
  const uint16_t *order;     // wo: wi's rows in the order of its slices, [expert][order_rows]
  int order_rows;
  const uint16_t *tables;    // [expert][columns]: where LDS has no room for a table beside a slice
  u32x4 *h;                  // wi: wo's operands, of h_steps steps
  int h_steps;
  const uint32_t *wo_minmax; // wi: [expert][wo_rows], looked over for tokens to be walked
  int wo_rows;
  uint16_t *y;               // wo
  int64_t ldy;
  const int32_t *slots;      // the token in every slot, or -1
  const int4 *chunks;        // (expert, first block, blocks, 0)
  int32_t *spoiled;          // [slot]: left to the walking kernel
  const int32_t *totals;
  int steps, parts;          // parts: wavefronts that share a slice
  int per_group;             // slices of a workgroup
  int slice_groups;          // workgroups of a chunk
};

// An expert's table, shared among `threads` threads.  A thread holds eight rows of wi's
// order, asked for beforehand (a row at a time, c-2048 wo took 5 us a workgroup for its
// table); longer orders are gone through in turns.
__device__ __forceinline__ u32x4 order_piece(const BatchArgs &a, int e, int piece) {
  const uint16_t *order = a.order + static_cast<int64_t>(e) * a.order_rows;   // whole slices: aligned
  return 8 * piece < a.order_rows ? *reinterpret_cast<const u32x4 *>(order + 8 * piece)
                                  : u32x4{~0u, ~0u, ~0u, ~0u};
}
__device__ __forceinline__ void fill_table(const BatchArgs &a, int e, uint16_t *table, u32x4 first, int thread,
                                           int threads) {
  const uint16_t idle = static_cast<uint16_t>(idle_step(a.steps) << 5);
  for (int q = thread * kZeroPeriod; q < physical_columns(a.k.width); q += threads * kZeroPeriod) table[q] = idle;
  const int last = physical_column(a.k.width - 1);
  for (int q = last + 1 + thread; q < physical_columns(a.k.width); q += threads) table[q] = idle;
  for (int piece = thread; 8 * piece < a.order_rows; piece += threads) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const int c = (first[i / 2] >> (16 * (i & 1))) & 0xffffu;
      if (c != 0xffff) table[physical_column(c)] = static_cast<uint16_t>(entry_of_row(8 * piece + i));
    }
    if (8 * (piece + threads) < a.order_rows) first = order_piece(a, e, piece + threads);
  }
}

// The nine entries of a chunk onto the row's codes.  `at` is the position reached,
// `lane_codes` the row's word 0.  The stream's entries never leave the row (what pads
// a row stays on a zero column or repeats its last entry, which or's the same bit).
template <bool kByTable>
__device__ __forceinline__ void expand_chunk(uint2 cw, uint32_t &at, uint32_t *lane_codes, const uint16_t *table) {
  const uint32_t mid = __builtin_amdgcn_alignbit(cw.y, cw.x, 28);
  uint32_t word[kFields], bit[kFields];
#pragma unroll
  for (int q = 0; q < kFields; q++) {
    const uint32_t step = q < 4 ? (cw.x >> (kFieldBits * q)) & 127u
                        : q < 8 ? (mid >> (kFieldBits * (q - 4))) & 127u
                                : (cw.y >> 24) & 127u;
    at += step;
    if (kByTable) {
      const uint32_t place = table[at >> 1];
      word[q] = place >> 5;
      bit[q] = 1u << ((place | (at & 1u)) & 31u);
    } else {
      word[q] = __umul24(at, 30841u) >> 20;   // at / 34, exact up to 50 000
      const uint32_t r = at - 34u * word[q];
      bit[q] = r < 2u ? 0u : 1u << (r & 31u);
    }
  }
#pragma unroll
  for (int q = 0; q < kFields; q++)
    __hip_atomic_fetch_or(lane_codes + word[q] * 64u, bit[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
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

// An exponent of all ones in either half: the sum carries into its sign.
__device__ __forceinline__ uint32_t high_exponents(uint32_t pair) {
  return ((pair & 0x7f807f80u) + 0x00800080u) & 0x80008000u;
}
__device__ __forceinline__ uint32_t bf16_pair(float lower, float upper) {
  const bf16x2 pair = {static_cast<__bf16>(lower), static_cast<__bf16>(upper)};
  return __builtin_bit_cast(uint32_t, pair);
}
__device__ __forceinline__ float relu_bits(float v) { return __uint_as_float(max(__float_as_int(v), 0)); }

// What a workgroup does: its slices' codes into LDS, then every wavefront's share of a
// slice's steps, then the sums of the wavefronts that share a slice, added in order and
// written.  Everything that is read from memory is asked for before the codes are expanded.
template <bool kHidden, bool kTableInLds, int kBlocks>
__device__ __forceinline__ void slices_times_tokens(const BatchArgs &a, uint32_t *lds, int e, int group,
                                                    int64_t first_block) {
  const int lane = threadIdx.x & 63, half = lane >> 5;
  const int waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int local = wave / a.parts;
  // (wavefronts with the same share of a slice on different SIMDs: the last has most to expand)
  const int sub = (wave + local) % a.parts;
  const int s = group * a.per_group + local;
  const bool mine = s < a.k.slices;
  const int64_t sl = static_cast<int64_t>(e) * a.k.slices + (mine ? s : 0);
  const int slice_words = slice_code_bytes(a.steps) / 4;
  uint32_t *codes = lds + local * slice_words;
  uint16_t *table_lds = reinterpret_cast<uint16_t *>(lds + a.per_group * slice_words);

  const u32x4 order = !kHidden && kTableInLds ? order_piece(a, e, threadIdx.x) : u32x4{};
  const int len = a.k.slice_len[sl];
  const uint32_t base_word = a.k.slice_base[sl];
  uint32_t minmax[2];
  int row[2];
#pragma unroll
  for (int j = 0; j < 2; j++) {
    minmax[j] = a.k.minmax[sl * 64 + 32 * j + (lane & 31)];
    if (!kHidden) row[j] = mine ? a.k.row_idx[sl * 64 + 32 * j + (lane & 31)] : 0xffff;
  }
  bool taken[kBlocks];   // the lane's slot: h of one without a token is not written, nor used
#pragma unroll
  for (int i = 0; i < kBlocks; i++)
    taken[i] = kHidden && mine && a.slots[(first_block + i) * kBlockTokens + (lane & 31)] >= 0;
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
  if (!kHidden && kTableInLds) fill_table(a, e, table_lds, order, threadIdx.x, blockDim.x);
  if (kHidden) {
    // the tokens that such weights leave to the walking kernel, of wo too (its product
    // goes by the marks as soon as it has a result)
    uint32_t high = 0;
    if (mine && sub == 0) high = high_exponents(minmax[0]) | high_exponents(minmax[1]);
    if (group == 0)
      for (int r = threadIdx.x; r < a.wo_rows; r += blockDim.x)
        high |= high_exponents(a.wo_minmax[static_cast<int64_t>(e) * a.wo_rows + r]);
    if (high)
      for (int t = 0; t < kBlocks * kBlockTokens; t++) a.spoiled[first_block * kBlockTokens + t] = 1;
  }
  __syncthreads();
  const uint16_t *table = kHidden ? nullptr
                          : kTableInLds ? table_lds
                                        : a.tables + static_cast<int64_t>(e) * physical_columns(a.k.width);
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
      if (c + i < c_end) expand_chunk<!kHidden>(now[i], at, codes + lane, table);
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
        // the first operand's 32 lie in a lane's values, the second's in the lanes
        acc[i][0] = kHidden ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(w0, xv, acc[i][0], 0, 0, 0)
                            : __builtin_amdgcn_mfma_f32_32x32x16_bf16(xv, w0, acc[i][0], 0, 0, 0);
        acc[i][1] = kHidden ? __builtin_amdgcn_mfma_f32_32x32x16_bf16(w1, xv, acc[i][1], 0, 0, 0)
                            : __builtin_amdgcn_mfma_f32_32x32x16_bf16(xv, w1, acc[i][1], 0, 0, 0);
      }
    }
  }

  // Values 4 g + 0..3 of block i and rows 32 j + 0..31.  h: a lane has token lane % 32 and rows
  // 8 g + 4 half + 0..3; y: row lane % 32 and tokens 8 g + 4 half + 0..3.
  uint32_t high[kBlocks];
#pragma unroll
  for (int i = 0; i < kBlocks; i++) high[i] = 0;
  auto tokens_of = [&](int i, int g) {   // -1: none, or one that is walked
    if (kHidden) return make_int4(0, 0, 0, 0);
    const int64_t slot = (first_block + i) * kBlockTokens + 8 * g + 4 * half;
    int4 t = *reinterpret_cast<const int4 *>(a.slots + slot);
    const int4 left = *reinterpret_cast<const int4 *>(a.spoiled + slot);
    if (left.x) t.x = -1;
    if (left.y) t.y = -1;
    if (left.z) t.z = -1;
    if (left.w) t.w = -1;
    return t;
  };
  auto write = [&](const float (&v)[4], const int4 &tokens, int i, int j, int g) {
    if (kHidden) {
      const uint2 w = make_uint2(bf16_pair(relu_bits(v[0]), relu_bits(v[1])), bf16_pair(relu_bits(v[2]), relu_bits(v[3])));
      high[i] |= high_exponents(w.x) | high_exponents(w.y);
      u32x4 *to = a.h + ((first_block + i) * a.h_steps + s * 4 + 2 * j + (g >> 1)) * 64 + lane;
      if (taken[i]) reinterpret_cast<uint2 *>(to)[g & 1] = w;
      return;
    }
    if (row[j] == 0xffff) return;
    const int t[4] = {tokens.x, tokens.y, tokens.z, tokens.w};
#pragma unroll
    for (int m = 0; m < 4; m++)
      if (t[m] >= 0) a.y[t[m] * a.ldy + row[j]] = __builtin_bit_cast(uint16_t, static_cast<__bf16>(v[m]));
  };
  if (a.parts == 1) {
    int4 tokens[kBlocks][4];
#pragma unroll
    for (int i = 0; i < kBlocks; i++)
#pragma unroll
      for (int g = 0; g < 4; g++) tokens[i][g] = tokens_of(i, g);
#pragma unroll
    for (int i = 0; i < kBlocks; i++)
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int g = 0; g < 4; g += kHidden ? 2 : 1) {
          if (kHidden) {   // an operand whole
            u32x4 w;
#pragma unroll
            for (int m = 0; m < 4; m++) {
              w[m] = bf16_pair(relu_bits(acc[i][j][4 * g + 2 * m]), relu_bits(acc[i][j][4 * g + 2 * m + 1]));
              high[i] |= high_exponents(w[m]);
            }
            if (taken[i]) a.h[((first_block + i) * a.h_steps + s * 4 + 2 * j + (g >> 1)) * 64 + lane] = w;
          } else {
            const float v[4] = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
            write(v, tokens[i][g], i, j, g);
          }
        }
  } else {
    int4 tokens[kBlocks][2];   // for the one or two groups of four values that are this wavefront's
#pragma unroll
    for (int i = 0; i < kBlocks; i++)
#pragma unroll
      for (int n = 0; n < 2; n++) tokens[i][n] = tokens_of(i, min(sub + n * a.parts, 3));
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
          place[(local * a.parts + sub) * 256 + g * 64 + lane] =
              make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
        __syncthreads();
#pragma unroll
        for (int n = 0; n < 2; n++) {
          const int g = sub + n * a.parts;
          if (g >= 4) break;
          const float4 *from = place + local * a.parts * 256 + g * 64 + lane;
          float4 sum = from[0];
          for (int p = 1; p < a.parts; p++) {
            const float4 v = from[p * 256];
            sum.x += v.x;
            sum.y += v.y;
            sum.z += v.z;
            sum.w += v.w;
          }
          const float v[4] = {sum.x, sum.y, sum.z, sum.w};
          write(v, tokens[i][n], i, j, g);
        }
      }
  }
  if (kHidden)
#pragma unroll
    for (int i = 0; i < kBlocks; i++)
      if (high[i]) a.spoiled[(first_block + i) * kBlockTokens + (lane & 31)] = 1;
}

template <bool kHidden, bool kTableInLds>
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
    slices_times_tokens<kHidden, kTableInLds, 2>(a, lds, e, group, first_block);
  else
    slices_times_tokens<kHidden, kTableInLds, 1>(a, lds, e, group, first_block);
}

// The tables of all experts, a workgroup each, for products that keep none in LDS.
__global__ __launch_bounds__(kMaxThreads) void fill_tables_kernel(BatchArgs a, uint16_t *tables) {
  fill_table(a, blockIdx.x, tables + static_cast<int64_t>(blockIdx.x) * physical_columns(a.k.width),
             order_piece(a, blockIdx.x, threadIdx.x), threadIdx.x, blockDim.x);
}

__device__ __forceinline__ bool not_finite(uint32_t bits) { return (bits & 0x7f80u) == 0x7f80u; }

// A step's 16 columns of a token (bits, zeros past the width) as its two operands.
__device__ __forceinline__ void write_operands(u32x4 *out, int64_t step, int t, const uint16_t (&v)[16]) {
#pragma unroll
  for (int h = 0; h < 2; h++) {
    u32x4 w;
#pragma unroll
    for (int k = 0; k < 4; k++)
      w[k] = v[column_of_place(h, 2 * k)] | static_cast<uint32_t>(v[column_of_place(h, 2 * k + 1)]) << 16;
    out[step * 64 + h * 32 + t] = w;
  }
}

// Prefix sum over a workgroup of 1024: what the threads below have, and the total.
__device__ __forceinline__ int below_in_workgroup(int v, int32_t *wave_sums, int *total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int upto = sub1::wave_prefix_sum(v);
  if (lane == 63) wave_sums[wave] = upto;
  __syncthreads();
  int below = upto - v, all = 0;
#pragma unroll
  for (int w = 0; w < 16; w++) {
    if (w < wave) below += wave_sums[w];
    all += wave_sums[w];
  }
  *total = all;
  return below;
}

// Every token gets a slot: its expert's tokens, in order, fill blocks of 32, an expert's blocks lie
// together, those of tokens without an expert come last.  A workgroup finds out for itself which tokens
// make its block - counts per expert, whose blocks these are, and which of that expert's tokens come
// before - and lays their activations out as operands; tokens without an expert keep their input.
// Bound by the chain of those stations.  (In a launch of one workgroup that grouped and one that laid
// out: 8.1 and 5.7 us for 4096 tokens of 128 base experts, here 8.6; the call 114 and 110.
// 30 experts of 901 x 2503 on 700 tokens 46.7 and 45.8, 51.1 with a block to a single workgroup.)
__global__ __launch_bounds__(kMaxThreads) void pack_blocks_kernel(
    const int32_t *__restrict__ token_expert, const uint16_t *x, uint16_t *y, int64_t ldx, int64_t ldy, int width,
    bool aligned, int tokens, int experts, int32_t *__restrict__ slots, int32_t *__restrict__ spoiled,
    int32_t *__restrict__ block_expert, int4 *__restrict__ chunks, int32_t *__restrict__ totals,
    int32_t *__restrict__ ctrl, u32x4 *__restrict__ out) {
  extern __shared__ __align__(16) int32_t count[];   // tokens of every expert, then of none
  __shared__ int32_t sums[3][16];
  __shared__ int s_bucket, s_nth, s_blocks, s_chunk;
  __shared__ int32_t s_token[kBlockTokens], s_bad[kBlockTokens];
  const int tid = threadIdx.x, block = blockIdx.x;
  const int buckets = experts + 1;
  // a thread's tokens are neighbours
  constexpr int kMine = kBatchPiece / kMaxThreads;
  const int each = (tokens + kMaxThreads - 1) / kMaxThreads;
  int bucket[kMine], faults = 0;
#pragma unroll
  for (int i = 0; i < kMine; i++) {
    const int t = tid * each + i;
    const bool mine = i < each && t < tokens;
    const int e = mine ? token_expert[t] : -1;
    if (e >= experts) faults++;
    bucket[i] = !mine ? -1 : e < 0 || e >= experts ? experts : e;
  }
  for (int b = tid; b < buckets; b += kMaxThreads) count[b] = 0;
  if (tid < kBlockTokens) {
    s_token[tid] = -1;
    s_bad[tid] = 0;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kMine; i++)
    if (bucket[i] >= 0) atomicAdd(&count[bucket[i]], 1);
  if (block == 0 && blockIdx.y == 0 && faults) atomicAdd(&ctrl[kCtrlBadIds], faults);
  __syncthreads();
  // whose block this is
  const int seg = (buckets + kMaxThreads - 1) / kMaxThreads;
  const int lo = min(tid * seg, buckets), hi = min(lo + seg, buckets);
  auto blocks_of = [](int n) { return (n + kBlockTokens - 1) / kBlockTokens; };
  auto chunks_in = [](int n) { return (n + kChunkBlocks - 1) / kChunkBlocks; };
  int n_blocks = 0, n_chunks = 0;
  for (int b = lo; b < hi; b++) {
    const int n = blocks_of(count[b]);
    n_blocks += n;
    if (b != experts) n_chunks += chunks_in(n);
  }
  int all_blocks, all_chunks;
  int at = below_in_workgroup(n_blocks, sums[0], &all_blocks);
  int chunk = below_in_workgroup(n_chunks, sums[1], &all_chunks);
  const int live_blocks = all_blocks - blocks_of(count[experts]);
  if (block == 0 && blockIdx.y == 0 && tid == 0) {
    totals[kTotalChunks] = all_chunks;
    totals[kTotalLive] = live_blocks;
    totals[kTotalBlocks] = all_blocks;
  }
  if (block >= all_blocks) return;
  for (int b = lo; b < hi; b++) {
    const int n = blocks_of(count[b]);
    if (block >= at && block < at + n) {
      s_bucket = b;
      s_nth = block - at;
      s_blocks = n;
      s_chunk = chunk;
    }
    at += n;
    chunk += chunks_in(n);
  }
  __syncthreads();
  const int mine = s_bucket, nth = s_nth;
  const bool live = mine != experts;
  // which of its tokens: 32 of them from number 32 nth on
  int found = 0;
#pragma unroll
  for (int i = 0; i < kMine; i++) found += bucket[i] == mine;
  int all_found;
  int number = below_in_workgroup(found, sums[2], &all_found) - kBlockTokens * nth;
#pragma unroll
  for (int i = 0; i < kMine; i++)
    if (bucket[i] == mine) {
      if (number >= 0 && number < kBlockTokens) s_token[number] = tid * each + i;
      number++;
    }
  __syncthreads();
  if (blockIdx.y == 0 && tid == 0) {
    block_expert[block] = live ? mine : -1;
    if (live && nth % kChunkBlocks == 0)
      chunks[s_chunk + nth / kChunkBlocks] = make_int4(mine, block, min(kChunkBlocks, s_blocks - nth), 0);
  }
  const int steps = steps_of(width);
  // the tokens of a block are shared by the workgroups of a column
  const int tokens_here = kBlockTokens / gridDim.y, first_here = blockIdx.y * tokens_here;
  const int t = first_here + tid % tokens_here;
  const int token = s_token[t];
  if (token >= 0) {   // (what the operands hold of an empty slot goes nowhere)
    const uint16_t *from = x + token * ldx;
    bool bad = false;
    for (int st = tid / tokens_here; st < steps; st += kMaxThreads / tokens_here) {
      const int c = st * kStepColumns;
      uint16_t v[16];
      if (aligned && c + 16 <= width) {
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
      } else {
        for (int i = 0; i < 16; i++)
          if (c + i < width) y[token * ldy + c + i] = v[i];
      }
    }
    if (bad) s_bad[t] = 1;
  }
  __syncthreads();
  if (tid < tokens_here) {
    const int slot = block * kBlockTokens + first_here + tid;
    slots[slot] = s_token[first_here + tid];
    spoiled[slot] = s_bad[first_here + tid];
  }
}

// The tokens in the slots that are marked, a workgroup each, as moe_prepared_fused_kernel
// walks them: the same sums.  LDS: x | h.  Workgroup b looks at slots b, b + grid, ...: an
// expert's tokens, which may all be marked, lie side by side.
__global__ __launch_bounds__(kMaxThreads) void walk_spoiled_kernel(PreparedArgs a, const int32_t *__restrict__ slots,
                                                                   const int32_t *__restrict__ spoiled,
                                                                   const int32_t *__restrict__ block_expert,
                                                                   const int32_t *__restrict__ totals) {
  extern __shared__ __align__(16) uint32_t lds[];
  uint32_t *xa = lds, *ha = lds + a.xdwords;
  const int waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int live = totals[kTotalLive] * kBlockTokens, grid = gridDim.x;
  bool fresh = true;
  for (int first = 0; first < live; first += 64 * grid) {
    // (every wavefront looks at the same 64 slots)
    const int mine = first + static_cast<int>(threadIdx.x & 63) * grid + static_cast<int>(blockIdx.x);
    unsigned long long found = __ballot(mine < live && slots[mine] >= 0 && spoiled[mine]);
    for (; found; found &= found - 1) {
      const int slot = first + (__ffsll(found) - 1) * grid + static_cast<int>(blockIdx.x);
      const int e = __builtin_amdgcn_readfirstlane(block_expert[slot / kBlockTokens]);
      const int t = __builtin_amdgcn_readfirstlane(slots[slot]);
      if (fresh)
        for (int i = threadIdx.x; i < a.hdwords; i += blockDim.x) ha[i] = 0u;
      fresh = false;
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
}
