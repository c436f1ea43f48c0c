// Internal launch interface between the C ABI (capi.hip) and the kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bt {

// Largest number of splits one sequence may use.
constexpr int kMaxSplitsPerSeq = 4096;

// Tokens per decode tile (the unit dealt round-robin to splits).
constexpr int kDecodeTileTokens = 16;

struct DecodeSplitParams {
  const void* q;             // (batch, heads, D) f32 or bf16; head stride = D
  int64_t q_stride_seq;      // elements between sequences in q
  int q_bf16;                // 1: q is bf16, 0: f32
  const uint16_t* k;         // bf16 cache, token-major
  const uint16_t* v;
  int64_t kv_stride_tok;     // elements between consecutive token slots
  int64_t kv_stride_head;    // elements between kv heads of one slot
  const int64_t* seq_offset; // (batch,) first slot of each sequence, or null (0)
  const int32_t* pos;        // (batch,) valid = pos + 1, or null
  const int32_t* seq_len;    // (batch,) valid lengths, or null
  int32_t seqlen;            // valid length when pos and seq_len are null; capacity when pos is set
  const int4* work;          // (num_work,) {b, s, ns_b, base_b}, or null: uniform num_split
  int32_t num_split;
  int32_t total_splits;      // row length of lse / part per head
  int32_t heads;
  int32_t kv_heads;
  int32_t group;             // heads / kv_heads
  float scale_log2;          // softmax scale * log2(e)
  float* lse;                // (heads, total_splits)
  float* part;               // (heads, total_splits, D)
  int32_t tiles_per_split;   // > 0: a sequence of n tiles uses min(num_split, ceil(n / this)) splits
  // Set where every sequence has one split: the split's rows are the results
  // and go here, (batch, heads, D) f32 or bf16, instead of to part and lse.
  void* out;
  int out_bf16;
  int64_t out_stride_seq;
};

// Waves per decode split work-group, and the tiles per split below which
// bt_gqa_decode's single-sequence and uniform-batch modes use fewer splits
// (measured on MI355X, config 2: 8 waves x 2 tiles took 7.8 / 8.8 / 17.6 us
// per call at 1k / 4k / 32k tokens, against 15.1 / 15.6 / 21.1 us for 16
// waves x 16 tiles and 9.0 / 9.7 / 17.2 us for a fixed 128 splits).
constexpr int kDecodeWaves = 8;
constexpr int kDecodeTilesPerSplit = 2;

struct CombineParams {
  const float* lse;
  const float* part;
  int32_t num_split;            // uniform split count (split_base == null)
  int32_t total_splits;
  const int32_t* split_base;    // (batch,) first split of each sequence, or null
  const int32_t* split_count;   // (batch,) splits of each sequence, or null
  void* out;                    // (batch, heads, D)
  int out_bf16;
  int64_t out_stride_seq;
};

struct PrefillParams {
  const uint16_t* q;   // (S, H, D) with strides, f32 or bf16 (q_f32)
  const uint16_t* k;   // bf16 (S, Hkv, D)
  const uint16_t* v;
  int64_t q_stride_tok, q_stride_head;
  int64_t kv_stride_tok, kv_stride_head;
  int32_t seqlen;      // new query rows S
  int32_t q_offset;    // absolute position of query row 0 (keys: q_offset + S)
  int32_t heads;
  int32_t kv_heads;
  int32_t group;       // heads / kv_heads
  // Two-waves-per-SIMD kernel: the group runs as head_subs subsets of
  // sub_group heads (sub_group in {1, 2, 4, 8}, the largest power of two
  // dividing group; grid y = kv_heads x head_subs).
  int32_t sub_group;
  int32_t head_subs;
  float scale_log2;
  void* out;
  int out_bf16;
  int64_t out_stride_tok, out_stride_head;
  uint16_t* vt;        // workspace: fp16 V^T image, prefill_vt_bytes() bytes
  int32_t* vexp;       // workspace: per (kv head, 64-key block) power-of-two scale of the image
  uint16_t* kimg;      // workspace: fp16 K image (row-major, XOR-swizzled slots), prefill_vt_bytes() bytes
  int32_t* kexp;       // workspace: per (kv head, 64-key block) power-of-two scale of the K image
  int32_t img_blocks;  // 64-key blocks per kv head in the image layout (>= those of q_offset + seqlen keys)
  int32_t img_first;   // first block the pre-pass converts (the images already hold the earlier ones)
  int32_t q_f32;       // 1: q is f32, 0: bf16 (either enters Q.K^T as fp16 scaled per row)
  int32_t keep_images; // 1: the images must hold every block afterwards (kept across chunked-prefill calls)
  // Split-key mode of the two-waves-per-SIMD kernel (kb_chunk > 0): work-group
  // (query block, kv head, chunk c) covers key blocks [c*kb_chunk, +kb_chunk);
  // a query block with more than one chunk writes one normalised partial and
  // its log2-domain LSE per (query, head) row and chunk, merged by
  // prefill_combine_kernel.  kb_chunk = 0: one work-group per query block.
  int32_t kb_chunk;
  // split_compact = 1: the uniform split's grid x lists only the (chunk, kv
  // head subset, query block) items that have keys, each chunk's query blocks
  // padded to a multiple of 8 (grid y = z = 1); 2: the items of at most two
  // chunks, longest first over all subsets (longest_ahead in gqa_prefill8.hip); 0: grid (query
  // blocks, kv heads x subsets, max_chunks), the items past a query block's
  // keys exiting.
  int32_t split_compact;
  // Paired split (pair_parts > 0, kb_chunk = 0): query blocks nqb-1-r and r
  // form pair r; the pair's key blocks (those of nqb-1-r, then those of r) are
  // cut into pair_parts equal ranges, one per work-group (grid x = pairs x
  // pair_parts), each covering at most two segments; a query block covered
  // by more than one range writes partials for prefill_combine_kernel.
  int32_t pair_parts;
  int32_t max_chunks;  // chunks of the longest query block (grid z of the uniform split)
  int32_t part_blocks; // query blocks per subset with room for partials: the last ones
  float* part;         // (subsets, part_blocks, max_chunks, 128 rows, D) f32
  float* lse;          // (subsets, part_blocks, max_chunks, 128 rows) f32
};

// Split-key plan of the two-waves-per-SIMD prefill: used when one work-group
// per query block would leave CUs idle (short prompts, long cached prefixes).
struct PrefillSplitPlan {
  int32_t kb_chunk = 0;    // 0: no uniform split
  int32_t compact = 0;     // uniform split on a compact grid (split_compact of PrefillParams)
  int32_t pair_parts = 0;  // 0: no paired split
  int32_t max_chunks = 1;
  int32_t query_blocks = 0;
  int32_t part_blocks = 0; // query blocks per subset that may have several chunks
  size_t part_rows = 0;    // subsets x part_blocks x max_chunks x rows per work-group
  size_t part_bytes = 0;   // part_rows x (head_dim f32 partials + 1 f32 LSE)
  float busiest = 0;       // estimate: key blocks of the busiest CU, its fixed costs among them
  bool idle = false;       // a work-group per query block, fewer of them than CUs
  bool active() const { return kb_chunk > 0 || pair_parts > 0; }
  bool uses_partials() const { return active() && max_chunks > 1; }
};
// `partials` false: only plans that need none.
PrefillSplitPlan prefill8_split_plan(int seqlen, int q_offset, int group, int kv_heads, int head_dim,
                                     int num_cus, bool partials);

// Per-row RMSNorm + RoPE (row mode) and the fused decode-step preparation
// (attention mode); see attn_prep.hip.
struct RowPrepParams {
  const float* x;            // row mode: (rows, D) rows; attention mode: the fused projection output
  int64_t x_stride;          // row mode: elements between rows
  int32_t rows;              // row mode
  float* out;                // row mode: (rows, D) f32
  int64_t out_stride;
  const float* w;            // RMSNorm weight (D,) (q weight in attention mode), or null: no norm
  const float* wk;           // attention mode: k RMSNorm weight (D,), or null
  float eps;
  const float* cos;          // (rope_cap, rope_dim) tables, or null: no rotation
  const float* sin;
  const int32_t* pos;        // device position (1,)
  int32_t rope_dim;
  int32_t rope_cap;
  int32_t heads;             // attention mode
  int32_t kv_heads;
  void* q_out;               // (heads, D) f32 or bf16
  int q_out_bf16;
  uint16_t* cache_k;         // bf16 cache, token-major slots
  uint16_t* cache_v;
  int64_t kv_stride_tok;
  int64_t kv_stride_head;
  int32_t cache_cap;
};

// Gated DeltaNet single-token decode step (gdn_decode.hip).
struct GdnParams {
  const float* q;      // (heads_k, D)
  const float* k;      // (heads_k, D)
  const float* v;      // (heads_v, D)
  const float* g;      // (heads_v,) log decay
  const float* beta;   // (heads_v,) logits of the write strength
  float* state;        // (heads_v, D, D), updated in place
  float* out;          // (heads_v, D)
  int32_t heads_k;
  int32_t heads_v;
  float scale;
  float eps;
};

// Decode matvec y = x . W (gemv.hip).
struct GemvParams {
  const float* x;        // (K,) f32
  const uint16_t* w;     // (K, N) bf16, row stride ldw elements
  int64_t ldw;
  int32_t K;
  int32_t N;
  int32_t splits;        // shares of K (SK); 1: no partials
  float* partial;        // (SK, N) f32 when SK > 1
  float* y;              // (N,) f32
};

// Launch shape of the matvec, for one of two kernels (gemv.hip).
//
// vec > 0: the column kernel, VEC columns per lane (tile = 64*VEC columns) and
// `splits` shares of K.  A wide matrix (>= 256 tiles of 512 columns, e.g. the
// vocabulary head) is not split: every CU already streams whole columns.
// Otherwise about 512 work-groups stream W with at least 64 rows per share.
// lanes > 0: the strip kernel, `lanes` lanes across a strip of 8 * lanes
// columns.  It takes, per the rates beside it,
//  * K of 256..1536 without a split, where strips fill the chip: strips of 32
//    columns for N of 3072 per 512 rows up to 8192 (256 work-groups: 9216 takes a
//    second round, 1024 x 9216 9.8 us against 8.2), of 64 from there to 16,384
//    (the same), of 128 from there to 65,536 (1024 x 100,000 45.3 us against
//    42.4); past K = 1024 the last two begin at 12,288 and 24,576 columns;
//  * else K > 2048, or K > 1024 and N >= 4096, up to N = 32,768, in strips of 128
//    columns and shares of one pass (256 rows), at most 1024 work-groups.  Where
//    that makes 257..512 of them, a second round that is not full, shares are 512
//    rows if then all run at once.
// Which of these the strip kernel really takes also depends on where W's rows lie
// (gemv_strips_suit).
constexpr int kGemvTargetGroups = 512;
constexpr int kGemvMinRows = 64;
struct GemvShape {
  int vec, lanes, splits, tiles;
};
inline GemvShape gemv_column_shape(int K, int N) {
  GemvShape g{};
  const int tiles8 = (N + 511) / 512;
  g.vec = tiles8 >= 8 ? 8 : 4;
  g.tiles = (N + 64 * g.vec - 1) / (64 * g.vec);
  g.splits = 1;
  if (tiles8 >= 256) return g;
  const int sk = (kGemvTargetGroups + g.tiles - 1) / g.tiles;
  const int cap = K / kGemvMinRows > 1 ? K / kGemvMinRows : 1;
  g.splits = sk < 1 ? 1 : (sk > cap ? cap : sk);
  return g;
}
// lanes = 0 outside the sizes above.
inline GemvShape gemv_strip_shape(int K, int N) {
  GemvShape g{};
  if (N > 65536) return g;
  const bool narrow = N >= 3072 * ((K + 511) / 512) && N <= 8192;
  const bool middle = N > (K <= 1024 ? 8192 : 12287) && N <= 16384;
  const bool wide = N > (K <= 1024 ? 16384 : 24575);
  if (K >= 256 && K <= 1536 && (narrow || middle || wide)) {
    g.lanes = narrow ? 4 : middle ? 8 : 16;
    g.tiles = (N + 8 * g.lanes - 1) / (8 * g.lanes);
    g.splits = 1;
  } else if ((K > 2048 || (K > 1024 && N >= 4096)) && N <= 32768) {
    g.lanes = 16;
    g.tiles = (N + 127) / 128;
    const int one = (K + 255) / 256, two = (K + 511) / 512, cap = 1024 / g.tiles;
    const int64_t groups = (int64_t)g.tiles * one;
    const int sk = groups > 256 && groups <= 512 && g.tiles * two <= 256 ? two : one;
    g.splits = sk < cap ? sk : cap;
  }
  return g;
}
// Whether the strip kernel is the faster one for a W whose rows begin at `base` and
// lie `pitch` bytes apart; us, column kernel / strips.
//  * Rows that do not begin on a line (half a line for strips of 32 columns): each
//    strip's lines are fetched by its neighbours too, so the column kernel keeps
//    most of them: 1536 x 16,392 13.1 / 16.1, 3072 x 16,392 21.7 / 25.8, 2560 x 1024
//    in a pitch of 1032 columns 6.35 / 6.53, 4096 x 4104 12.1 / 12.6, 16,384 x 2056
//    19.3 / 21.6.  Strips are still the faster ones
//    - unsplit: K up to 512 (512 x 16,392 0.79 of the column kernel's time, 50,008
//      0.96, 65,528 1.08), 768 in narrow strips (0.82 to 0.96; 1024 1.00 to 1.03),
//      1024 between 18,433 and 32,768 columns, which fill its rounds badly (1024 x
//      19,432 / 24,584 0.86 / 0.87; 32,776 1.02);
//    - in shares: where the column kernel's tiles do not fill 512 work-groups evenly
//      and a few run in a second round, up to 8192 columns (8192 x 1672 15.1 / 10.5,
//      5120 x 3000 13.5 / 11.0, 6144 x 5128 22.5 / 19.3), one of them only with K under
//      8192 / 4096 (5120 x 2056 12.1 / 9.6, 2304 x 4104 9.9 / 8.9); from K = 4608 up to 1536
//      columns always (0.63 to 0.90).
//  * A pitch of whole 4 KB and 1921 to 2048 columns, 16 strips, which past K = 8192
//    take a second round and land on few memory channels, while eight column tiles
//    fill one round: 8453 / 10,240 / 12,288 x 2048 10.9 / 12.1, 11.2 / 12.9, 12.5 / 13.8
//    (9500 and 11,500 0.92 to 0.97 of the column kernel's time).  Up to there strips
//    (7000 x 2048 10.7 / 9.3, 8192 11.8 / 9.8), but for whole rows of it in shares of
//    whole 32-row passes: 6144 x 2048 8.73 / 8.95.  A power of two of rows in 8 KB puts
//    the column kernel's shares on few channels too: 16,384 x 2048 23.7 / 18.6.
inline bool gemv_strips_suit(const GemvShape& strip, int K, int N, int64_t pitch, uint64_t base) {
  const int line = strip.lanes == 4 ? 64 : 128;
  if (((uint64_t)pitch | base) % line) {
    if (strip.splits == 1) {
      if (K <= 512) return N <= 57344;
      return strip.lanes == 4 ? K <= 768 : K <= 1024 && N > 18432 && N <= 32768;
    }
    if (K >= 4608 && N <= 1536) return true;
    const int tiles = gemv_column_shape(K, N).tiles;
    const int second_round = (kGemvTargetGroups + tiles - 1) / tiles * tiles - kGemvTargetGroups;
    return N <= 8192 && second_round > 0 && (second_round > 1 || K < (N < 4096 ? 8192 : 4096));
  }
  if (N > 1920 && N <= 2048 && pitch % 4096 == 0) {
    const bool two_power = (K & (K - 1)) == 0;
    if (K > 8192) return two_power && pitch % 8192 == 0;
    return two_power || K < 6144 || K % 2048 || N * 2 % 4096;
  }
  return true;
}
inline GemvShape gemv_shape(int K, int N, int64_t pitch, uint64_t base) {
  const GemvShape strip = gemv_strip_shape(K, N);
  return strip.lanes && gemv_strips_suit(strip, K, N, pitch, base) ? strip : gemv_column_shape(K, N);
}

// Workspace of the split-K matvec, the partial rows, for any pitch: of the kernel
// with more shares.
inline size_t gemv_workspace_bytes(int K, int N) {
  const GemvShape strip = gemv_strip_shape(K, N);
  int splits = gemv_column_shape(K, N).splits;
  if (strip.lanes && strip.splits > splits) splits = strip.splits;
  return splits == 1 ? 0 : (size_t)splits * N * 4;
}

// Keys per block of the prefill key loop, and the size of the transposed,
// block-scaled fp16 V image the prefill builds in its workspace: per kv head and 64-key block,
// 8 chunks of 8 keys x head_dim rows x 16 bytes, for kv_len keys.
constexpr int kPrefillKeyBlock = 64;
inline size_t prefill_vt_bytes(int kv_len, int kv_heads, int head_dim) {
  const size_t blocks = (size_t)(kv_len + kPrefillKeyBlock - 1) / kPrefillKeyBlock;
  return (size_t)kv_heads * blocks * kPrefillKeyBlock * (size_t)head_dim * 2;
}

// Which kernel variant serves a combination of length sources, or -1 if the
// combination is not served:
//   work table (ragged)              -> needs seq_len and seq_offset, no pos
//   pos, batch 1, no seq_offset      -> single sequence, device position
//   pos + seq_offset                 -> batch of device positions
//   seq_len + seq_offset             -> batch of device lengths
//   none of them, batch 1            -> explicit length argument
inline int decode_mode(bool work, bool pos, bool seq_len, bool seq_offset, int batch) {
  if (work) return (seq_len && seq_offset && !pos) ? 3 : -1;
  if (pos) {
    if (seq_len) return -1;
    if (!seq_offset) return batch == 1 ? 1 : -1;
    return 2;
  }
  if (seq_len) return seq_offset ? 4 : -1;
  return (batch == 1 && !seq_offset) ? 0 : -1;
}

// Whether one round of `round` work-groups serves a ragged batch evenly: its n
// splits, of at most `longest` tokens each, take ceil(n / round) rounds; even
// means that these hold at most 1.5 times the batch's tokens.
inline __host__ __device__ bool ragged_round_is_even(int64_t n, int64_t longest, int64_t tokens, int64_t round) {
  return 2 * ((n + round - 1) / round) * longest * round <= 3 * tokens;
}

// Whether more splits (n2 under a cap of `cap2` tokens, for n and `longest` of
// one round) pay: what the longest loses, over the CUs of a round, against the
// fixed cost of the further splits, split_tokens tokens each (prologue, merge,
// partials through memory).  0: always.  A split has at most cap2 tokens, or 32.
inline __host__ __device__ bool ragged_splits_pay(int64_t n, int64_t longest, int64_t n2, int64_t cap2,
                                                  int64_t round, int64_t split_tokens) {
  return split_tokens == 0 || split_tokens * (n2 - n) <= (longest - (cap2 > 32 ? cap2 : 32)) * round;
}

// Device-side ragged plan (ragged_plan.hip): the plan bt_ragged_plan_cost
// makes on the host, from device lengths, padded to work_capacity entries with
// {-1, ..}.
constexpr int kRaggedPlanMaxBatch = 4096;
struct RaggedPlanParams {
  const int32_t* seq_len;  // (batch,) device lengths
  int32_t batch;
  int32_t round_groups;    // work-groups of one round
  int32_t target_groups;   // work-groups where one round is uneven and more splits pay
  int32_t split_tokens;    // fixed cost of a split in tokens (ragged_splits_pay)
  int32_t* work;           // (work_capacity, 4) entries {b, s, ns_b, base_b}
  int32_t work_capacity;   // >= max(batch, target_groups, round_groups)
  int32_t* split_base;     // (batch,)
  int32_t* split_count;    // (batch,)
  int32_t* total;          // optional: the number of real entries
};
hipError_t launch_ragged_plan(const RaggedPlanParams& p, hipStream_t stream);

hipError_t launch_decode_split(const DecodeSplitParams& p, int head_dim, int grid_x, int batch,
                               hipStream_t stream);
hipError_t launch_decode_combine(const CombineParams& p, int head_dim, int heads, int batch,
                                 hipStream_t stream);
// Two-waves-per-SIMD prefill (gqa_prefill8.hip) for group sizes 1..8: a
// group runs as subsets of prefill8_sub_group(group) heads.
bool prefill8_serves(int group, int head_dim);
int prefill8_sub_group(int group);
// Work-groups of the longest-first grid (split_compact = 2) of at most two chunks of
// kb_chunk blocks; item >= 0: that work-group's item too, subset -1 for a padding slot.
int prefill8_longest_first(int seqlen, int q_offset, int group, int subsets, int kb_chunk, int item, int* subset,
                           int* qblk, int* chunk);
// Pair kernel (gqa_prefill_pair.hip): two query blocks per work-group, 32
// query columns per wave; group sizes 1, 2, 4, 8.
bool prefill_pair_serves(int group, int head_dim);
// Work-groups of a launch and the steps each takes.
int prefill_pair_grid(int seqlen, int q_offset, int group, int kv_heads, bool q_f32, int* steps);
hipError_t launch_prefill_pair(const PrefillParams& p, int head_dim, hipStream_t stream);
// Scaled fp16 V^T image + per-block exponents (p.vt, p.vexp) in the key order
// of the 16x16 MFMA result layout, and the scaled fp16 K image + exponents
// (p.kimg, p.kexp).
hipError_t launch_prefill_vts(const PrefillParams& p, int head_dim, hipStream_t stream);
hipError_t launch_prefill8(const PrefillParams& p, int head_dim, hipStream_t stream);
hipError_t launch_row_norm_rope(const RowPrepParams& p, int head_dim, hipStream_t stream);
hipError_t launch_attn_prep(const RowPrepParams& p, int head_dim, hipStream_t stream);
hipError_t launch_gdn_decode(const GdnParams& p, int dim, hipStream_t stream);
hipError_t launch_gemv(const GemvParams& p, const GemvShape& shape, hipStream_t stream);

}  // namespace bt
