// The C ABI of libbreezetoken_amd.so: argument validation and launches.
// Declarations and documentation live in include/breezetoken_amd.h.
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <vector>

#include "../../include/breezetoken_amd.h"
#include "bt_kernels.h"

namespace {

constexpr double kLog2e = 1.4426950408889634;

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline bool served_dim(int d) { return d == 64 || d == 128 || d == 256; }
inline int64_t align256(int64_t x) { return (x + 255) & ~int64_t(255); }

int check_decode_common(const void* q, int32_t q_dtype, int64_t q_stride_seq, const void* k,
                        const void* v, int64_t kv_stride_tok, int64_t kv_stride_head,
                        int32_t batch, int32_t heads, int32_t kv_heads, int32_t head_dim) {
  if (!q || !k || !v) return BT_EINVAL;
  if (batch < 1 || heads < 1 || kv_heads < 1 || head_dim < 1) return BT_EINVAL;
  if (heads % kv_heads != 0) return BT_EINVAL;
  if (q_dtype != BT_DTYPE_F32 && q_dtype != BT_DTYPE_BF16) return BT_EINVAL;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v)) return BT_EINVAL;
  if (kv_stride_tok <= 0 || kv_stride_head < 0 || kv_stride_tok % 8 || kv_stride_head % 8)
    return BT_EINVAL;
  if (batch > 1 && (q_stride_seq < (int64_t)heads * head_dim || q_stride_seq % 8)) return BT_EINVAL;
  if (!served_dim(head_dim)) return BT_ENOTSUP;
  if (heads / kv_heads > 8) return BT_ENOTSUP;
  if (batch > 65535 || kv_heads > 65535) return BT_ENOTSUP;
  return BT_OK;
}

int check_out(const void* out, int32_t out_dtype, int64_t out_stride_seq, int32_t batch,
              int32_t heads, int32_t head_dim) {
  if (!out) return BT_EINVAL;
  if (out_dtype != BT_DTYPE_F32 && out_dtype != BT_DTYPE_BF16) return BT_EINVAL;
  if (!aligned16(out)) return BT_EINVAL;
  if (batch > 1 && (out_stride_seq < (int64_t)heads * head_dim || out_stride_seq % 8))
    return BT_EINVAL;
  return BT_OK;
}

bt::DecodeSplitParams make_split_params(const void* q, int32_t q_dtype, int64_t q_stride_seq,
                                        const void* k, const void* v, int64_t kv_stride_tok,
                                        int64_t kv_stride_head, const int64_t* seq_offset,
                                        const int32_t* pos, const int32_t* seq_len,
                                        int32_t seqlen, int32_t heads, int32_t kv_heads,
                                        int32_t head_dim, float scale, float* lse, float* part) {
  bt::DecodeSplitParams p{};
  p.q = q;
  p.q_stride_seq = q_stride_seq > 0 ? q_stride_seq : (int64_t)heads * head_dim;
  p.q_bf16 = q_dtype == BT_DTYPE_BF16;
  p.k = static_cast<const uint16_t*>(k);
  p.v = static_cast<const uint16_t*>(v);
  p.kv_stride_tok = kv_stride_tok;
  p.kv_stride_head = kv_stride_head;
  p.seq_offset = seq_offset;
  p.pos = pos;
  p.seq_len = seq_len;
  p.seqlen = seqlen;
  p.heads = heads;
  p.kv_heads = kv_heads;
  p.group = heads / kv_heads;
  p.scale_log2 = (float)((double)scale * kLog2e);
  p.lse = lse;
  p.part = part;
  return p;
}

inline int hip_rc(hipError_t e) { return e == hipSuccess ? BT_OK : (int)e; }

}  // namespace

namespace {

// Compute units of the current device, cached per device.
int device_cus() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return 256;
  static int cache[64] = {0};
  if (dev >= 0 && dev < 64 && cache[dev] > 0) return cache[dev];
  int n = 0;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
  if (dev >= 0 && dev < 64) cache[dev] = n;
  return n;
}

// Prefill workspace, each part 256-byte aligned: the fp16 V^T image, one int32
// scale exponent per kv head and 64-key block, the fp16 K image of the same
// size, and its exponents.
struct PrefillLayout {
  int64_t vexp, kimg, kexp, bytes;
};
PrefillLayout prefill_layout(int32_t kv_len, int32_t kv_heads, int32_t head_dim) {
  const int64_t img = align256((int64_t)bt::prefill_vt_bytes(kv_len, kv_heads, head_dim));
  const int64_t nblk = ((int64_t)kv_len + bt::kPrefillKeyBlock - 1) / bt::kPrefillKeyBlock;
  const int64_t tab = align256(nblk * kv_heads * 4);
  PrefillLayout l;
  l.vexp = img;
  l.kimg = l.vexp + tab;
  l.kexp = l.kimg + img;
  l.bytes = l.kexp + tab;
  return l;
}
int64_t prefill_base_bytes(int32_t kv_len, int32_t kv_heads, int32_t head_dim) {
  return prefill_layout(kv_len, kv_heads, head_dim).bytes;
}

// The split-key plan of the two-waves-per-SIMD kernel for this shape on the
// current device (inactive: a work-group per query block), without `partials`
// one that needs none.
bt::PrefillSplitPlan prefill8_plan(int32_t seqlen, int32_t q_offset, int32_t heads, int32_t kv_heads,
                                   int32_t head_dim, bool partials = true) {
  const int group = heads / kv_heads;
  if (!bt::prefill8_serves(group, head_dim)) return bt::PrefillSplitPlan{};
  // The kernel runs the group as subsets of sub_group heads, each subset a
  // row of the grid like a kv head of its own.
  const int sub = bt::prefill8_sub_group(group);
  return bt::prefill8_split_plan(seqlen, q_offset, sub, kv_heads * (group / sub), head_dim, device_cus(),
                                 partials);
}

// Whether the pair kernel serves this call faster than the two-waves-per-SIMD
// kernel under `plan`, both estimated in microseconds.  The pair kernel's
// work-groups all take the same steps of 32 keys and run one per CU, so its
// time is a whole number of rounds, and a grid just past one costs two: at S =
// 4500 it took 257 us against 187 (H = 16, Hkv = 2, D = 256, bf16 q), 182
// against 117 (D = 128).  Within one round it is the faster one once its steps
// outweigh its start and final merge: H = 8, Hkv = 2, D = 256, bf16 q, S = 7000
// 209 against 217 us; f32 q, whose pair work-groups are half as large, S =
// 1024 41 against 51 us, 3001 82 against 120 us (no partials).  A grid that
// leaves CUs idle lasts as long as its longest work-group, whose blocks take
// less than under full load, and starts sooner: bf16 q, S = 1024 / 2048 / 3001
// 41 / 69 / 95 us against the pair kernel's 53 / 80 / 104.
// The rates (us) are fits to S = 130 .. 16,384 at four shapes for each head
// dimension and q type, medians over seven rounds in turn; over those 900 choices
// the kernel taken is the faster one or within 1% of it, but for three (4%).
struct PrefillRates {
  double pair_start, pair_step;    // pair kernel: per call, per step of 32 keys
  double two_start, two_block;     // two-wave kernel: per call, per 64-key block of the busiest CU
  double idle_start, idle_factor;  // the same where CUs stay idle: per call, of two_block
  double paired_factor;            // a block of the paired split, of two_block
};
bool prefill_pair_faster(const bt::PrefillSplitPlan& plan, int32_t seqlen, int32_t q_offset, int32_t heads,
                         int32_t kv_heads, int32_t head_dim, bool q_f32) {
  const int group = heads / kv_heads;
  if (!bt::prefill_pair_serves(group, head_dim)) return false;
  const bool wide = head_dim == 256;
  const PrefillRates r = wide ? (q_f32 ? PrefillRates{17.0, 1.36, 10.0, 2.55, 6.0, 0.88, 1.05}
                                       : PrefillRates{23.0, 1.68, 11.0, 2.0, 5.0, 0.88, 1.12})
                              : (q_f32 ? PrefillRates{12.5, 0.89, 10.0, 1.4, 5.0, 0.97, 1.1}
                                       : PrefillRates{15.0, 1.17, 10.0, 1.18, 5.0, 1.0, 1.1});
  const int64_t cus = device_cus();
  int steps = 0;
  const int64_t groups = bt::prefill_pair_grid(seqlen, q_offset, group, kv_heads, q_f32, &steps);
  double rounds = (double)((groups + cus - 1) / cus);
  // At D = 128 two f32-q work-groups fit a CU and take 1.56 times one's time;
  // half-filled rounds of two pass as such.
  if (!wide && q_f32 && groups > cus) rounds = 1.56 * std::max(1.0, 0.5 * (double)((groups + cus - 1) / cus));
  const double pair = r.pair_start + rounds * steps * r.pair_step;
  // Short prompts whose work-groups convert their own blocks have no pre-pass.
  const int64_t longest = ((int64_t)q_offset + seqlen + bt::kPrefillKeyBlock - 1) / bt::kPrefillKeyBlock;
  const double start = (plan.kb_chunk > 0 ? plan.kb_chunk : longest) <= 2 ? 4.0 : r.two_start;
  double two = start + plan.busiest * r.two_block * (plan.pair_parts > 0 ? r.paired_factor : 1.0);
  if (plan.idle) two = r.idle_start + plan.busiest * r.two_block * r.idle_factor;
  // Plans of whole query blocks, or with the longest cut, are fitted to 3%, the others to 10%.
  const bool close = plan.pair_parts == 0 && (plan.compact == 2 || plan.kb_chunk == 0);
  return pair < (close ? 0.99 : 0.95) * two;
}

// What bt_gqa_prefill and bt_gqa_prefill_cached run for a call whose partials
// may take `partials_bytes`.
struct PrefillChoice {
  bool pair;
  bt::PrefillSplitPlan plan;  // of the two-wave kernel
};
PrefillChoice prefill_choice(int32_t seqlen, int32_t q_offset, int32_t heads, int32_t kv_heads, int32_t head_dim,
                             bool q_f32, int64_t partials_bytes) {
  bt::PrefillSplitPlan plan = prefill8_plan(seqlen, q_offset, heads, kv_heads, head_dim);
  if (plan.uses_partials() && partials_bytes < (int64_t)plan.part_bytes)
    plan = prefill8_plan(seqlen, q_offset, heads, kv_heads, head_dim, false);
  return {prefill_pair_faster(plan, seqlen, q_offset, heads, kv_heads, head_dim, q_f32), plan};
}

}  // namespace

extern "C" {

int bt_version(void) { return 100; }

const char* bt_strerror(int code) {
  switch (code) {
    case BT_OK: return "success";
    case BT_EINVAL: return "invalid argument (null pointer, shape, stride or alignment)";
    case BT_ENOTSUP: return "shape not served (head_dim, group size or split count)";
    case BT_ENOSPC: return "workspace too small";
    default: return code > 0 ? hipGetErrorString((hipError_t)code) : "unknown error";
  }
}

int32_t bt_decode_tile_tokens(void) { return bt::kDecodeTileTokens; }

int64_t bt_decode_workspace_bytes(int32_t heads, int32_t head_dim, int32_t total_splits) {
  if (heads < 1 || head_dim < 1 || total_splits < 1) return 0;
  const int64_t lse = align256((int64_t)heads * total_splits * 4);
  return lse + (int64_t)heads * total_splits * head_dim * 4;
}

int32_t bt_decode_pick_splits(int32_t kv_heads, int32_t ctx_len, int32_t num_cus) {
  if (kv_heads < 1) kv_heads = 1;
  if (num_cus < 1) num_cus = 256;
  int32_t ns = (num_cus + kv_heads - 1) / kv_heads;
  const int32_t tiles = ctx_len > 0 ? (ctx_len + 31) / 32 : 1;
  if (ns > tiles) ns = tiles;
  if (ns > bt::kMaxSplitsPerSeq) ns = bt::kMaxSplitsPerSeq;
  return ns < 1 ? 1 : ns;
}

int32_t bt_decode_pick_splits_batch(int32_t batch, int32_t heads, int32_t kv_heads, int32_t max_len,
                                    int32_t num_cus) {
  if (batch < 1) batch = 1;
  if (kv_heads < 1) kv_heads = 1;
  if (heads < kv_heads) heads = kv_heads;
  if (num_cus < 1) num_cus = 256;
  if (max_len < 1) max_len = 1;
  const int64_t pairs = (int64_t)batch * kv_heads, cus = num_cus;
  // The time of ns splits in tokens of one CU's stream: a work-group streams
  // max_len / ns tokens and costs as much as kFixed + 2 * group more (prologue,
  // merge; its partials' way through memory); work-groups run in rounds of one
  // per CU, and a round that is not full is hardly faster (a CU alone reads 26
  // GB/s against 23 GB/s with all of them streaming); a quarter of a
  // work-group stands for the lengths' spread at the end; more than one split
  // costs the combine's launch.
  constexpr int64_t kFixed = 80, kCombine = 64;
  const int64_t fixed = kFixed + 2 * (heads / kv_heads);
  const int64_t tiles = (max_len + 31) / 32;
  const int64_t most = std::min<int64_t>(std::min<int64_t>(tiles, bt::kMaxSplitsPerSeq), 1 + 4 * cus / pairs);
  int64_t best = 1, best_cost = INT64_MAX;
  for (int64_t ns = 1; ns <= most; ++ns) {
    const int64_t groups = pairs * ns, share = max_len / ns, full = groups / cus;
    const int64_t cost = full * (fixed + share) + (groups % cus ? fixed + share * 9 / 10 : 0) + share / 4 +
                         (ns > 1 ? kCombine : 0);
    if (cost < best_cost) {
      best = ns;
      best_cost = cost;
    }
  }
  return (int32_t)best;
}

int32_t bt_decode_pick_splits_uniform(int32_t batch, int32_t heads, int32_t kv_heads, int32_t head_dim,
                                      int32_t max_len, int32_t num_cus) {
  if (batch < 1) batch = 1;
  if (kv_heads < 1) kv_heads = 1;
  if (heads < kv_heads) heads = kv_heads;
  if (num_cus < 1) num_cus = 256;
  if (max_len < 1) max_len = 1;
  const int64_t pairs = (int64_t)batch * kv_heads, cus = num_cus;
  const int64_t most = std::min<int64_t>(((int64_t)max_len + 31) / 32, bt::kMaxSplitsPerSeq);
  // Microseconds of a call with ns splits, lengths between 60% of max_len and all
  // of it.  Two things bound it together: the tokens the fullest CU streams, at
  // the rate of one that streams alone, and what all of them move, at 7 TB/s, with
  // each work-group's fixed time on its CU (one fits a CU at D = 256, two at 128,
  // three at 64).  More than one split costs the combine's launch and its work.
  // Fitted to 767 calls at eight shapes, 1 to 128 sequences of 30 to 20,000 tokens.
  struct Rates {
    double token, rounds, group;  // a token alone, a round's share of one where there are several, fixed
  };
  const Rates r = head_dim > 128  ? Rates{0.0158, 0.7, 1.9}
                  : head_dim > 64 ? Rates{0.009, 0.84, 0.27}
                                  : Rates{0.0056, 0.87, 0.06};
  auto time = [&](int64_t ns) {
    const double share = std::max(32.0, (double)max_len / (double)ns), n = (double)(pairs * ns);
    const double rounds = pairs * ns > cus ? r.rounds * (double)((pairs * ns + cus - 1) / cus) : 1.0;
    const double fullest = rounds * share * r.token + 0.5;
    const double all = n * (0.8 * share * 4 * head_dim / 7.0e6 + r.group / (double)cus);
    const double combine = ns > 1 ? 1.8 + 2.5e-5 * (double)batch * heads * head_dim : 0.0;
    return 3.0 + 0.06 * (heads / kv_heads) + combine + std::sqrt(fullest * fullest + all * all);
  };
  // One split, and the counts that fill one to five rounds; more than one round
  // where it is faster by over 1.5%.
  const int64_t one = std::max<int64_t>(1, std::min(most, cus / pairs));
  int64_t best = 1;
  double best_time = time(1);
  for (int64_t rounds = 1; rounds <= 5; ++rounds) {
    const int64_t ns = std::max<int64_t>(1, std::min(most, rounds * cus / pairs));
    const double t = time(ns) * (ns > one ? 1.015 : 1.0);
    if (t < best_time) {
      best = ns;
      best_time = t;
    }
  }
  return (int32_t)best;
}

int bt_gqa_decode_split(const void* q, int32_t q_dtype, int64_t q_stride_seq, const void* k,
                        const void* v, int64_t kv_stride_tok, int64_t kv_stride_head,
                        const int64_t* seq_offset, const int32_t* pos, const int32_t* seq_len,
                        int32_t seqlen, int32_t batch, int32_t heads, int32_t kv_heads,
                        int32_t head_dim, int32_t num_split, float scale, float* lse,
                        float* part, void* stream) {
  int rc = check_decode_common(q, q_dtype, q_stride_seq, k, v, kv_stride_tok, kv_stride_head,
                               batch, heads, kv_heads, head_dim);
  if (rc) return rc;
  if (!lse || !part || !aligned16(part)) return BT_EINVAL;
  if (num_split < 1) return BT_EINVAL;
  if (num_split > bt::kMaxSplitsPerSeq) return BT_ENOTSUP;
  if (!pos && !seq_len && seqlen < 0) return BT_EINVAL;
  if (pos && seqlen < 1) return BT_EINVAL;  // capacity bound for the position path
  if (bt::decode_mode(false, pos != nullptr, seq_len != nullptr, seq_offset != nullptr, batch) < 0)
    return BT_EINVAL;
  if ((int64_t)seqlen * kv_stride_tok * 2 > (int64_t)UINT32_MAX) return BT_ENOTSUP;
  if ((int64_t)batch * num_split > INT32_MAX / 2) return BT_ENOTSUP;
  bt::DecodeSplitParams p = make_split_params(q, q_dtype, q_stride_seq, k, v, kv_stride_tok,
                                              kv_stride_head, seq_offset, pos, seq_len, seqlen,
                                              heads, kv_heads, head_dim, scale, lse, part);
  p.work = nullptr;
  p.num_split = num_split;
  p.total_splits = batch * num_split;
  return hip_rc(bt::launch_decode_split(p, head_dim, num_split, batch, (hipStream_t)stream));
}

int bt_gqa_decode_combine(const float* lse, const float* part, int32_t batch, int32_t heads,
                          int32_t head_dim, int32_t num_split, const int32_t* split_base,
                          const int32_t* split_count, int32_t total_splits, void* out,
                          int32_t out_dtype, int64_t out_stride_seq, void* stream) {
  if (!lse || !part || !aligned16(part)) return BT_EINVAL;
  if (batch < 1 || heads < 1 || total_splits < 1) return BT_EINVAL;
  if ((split_base == nullptr) != (split_count == nullptr)) return BT_EINVAL;
  if (!split_base && (num_split < 1 || (int64_t)batch * num_split > total_splits)) return BT_EINVAL;
  if (!split_base && num_split > bt::kMaxSplitsPerSeq) return BT_ENOTSUP;
  if (!served_dim(head_dim)) return BT_ENOTSUP;
  if (heads > 65535 || batch > 65535) return BT_ENOTSUP;
  int rc = check_out(out, out_dtype, out_stride_seq, batch, heads, head_dim);
  if (rc) return rc;
  bt::CombineParams c{};
  c.lse = lse;
  c.part = part;
  c.num_split = num_split;
  c.total_splits = total_splits;
  c.split_base = split_base;
  c.split_count = split_count;
  c.out = out;
  c.out_bf16 = out_dtype == BT_DTYPE_BF16;
  c.out_stride_seq = out_stride_seq > 0 ? out_stride_seq : (int64_t)heads * head_dim;
  return hip_rc(bt::launch_decode_combine(c, head_dim, heads, batch, (hipStream_t)stream));
}

int bt_gqa_decode(const void* q, int32_t q_dtype, int64_t q_stride_seq, const void* k,
                  const void* v, int64_t kv_stride_tok, int64_t kv_stride_head,
                  const int64_t* seq_offset, const int32_t* pos, const int32_t* seq_len,
                  int32_t seqlen, int32_t batch, int32_t heads, int32_t kv_heads,
                  int32_t head_dim, int32_t num_split, float scale, void* workspace,
                  int64_t workspace_bytes, void* out, int32_t out_dtype,
                  int64_t out_stride_seq, void* stream) {
  int rc = check_decode_common(q, q_dtype, q_stride_seq, k, v, kv_stride_tok, kv_stride_head,
                               batch, heads, kv_heads, head_dim);
  if (rc) return rc;
  rc = check_out(out, out_dtype, out_stride_seq, batch, heads, head_dim);
  if (rc) return rc;
  if (num_split < 1) return BT_EINVAL;
  if (num_split > bt::kMaxSplitsPerSeq) return BT_ENOTSUP;
  if ((int64_t)batch * num_split > INT32_MAX / 2) return BT_ENOTSUP;
  if (!workspace || !aligned16(workspace)) return BT_EINVAL;
  const int32_t total = batch * num_split;
  if (workspace_bytes < bt_decode_workspace_bytes(heads, head_dim, total)) return BT_ENOSPC;
  float* lse = static_cast<float*>(workspace);
  float* part = reinterpret_cast<float*>(static_cast<char*>(workspace) +
                                         align256((int64_t)heads * total * 4));
  if (!pos && !seq_len && seqlen < 0) return BT_EINVAL;
  if (pos && seqlen < 1) return BT_EINVAL;  // capacity bound for the position path
  if (bt::decode_mode(false, pos != nullptr, seq_len != nullptr, seq_offset != nullptr, batch) < 0)
    return BT_EINVAL;
  if ((int64_t)seqlen * kv_stride_tok * 2 > (int64_t)UINT32_MAX) return BT_ENOTSUP;
  bt::DecodeSplitParams p = make_split_params(q, q_dtype, q_stride_seq, k, v, kv_stride_tok,
                                              kv_stride_head, seq_offset, pos, seq_len, seqlen,
                                              heads, kv_heads, head_dim, scale, lse, part);
  p.work = nullptr;
  p.num_split = num_split;
  p.total_splits = total;
  // A short context in a large grid uses fewer, fuller splits (the split count
  // follows the length on the device; the combine skips the empty splits).
  p.tiles_per_split = bt::kDecodeTilesPerSplit;
  if (num_split == 1) {
    // The only split's rows are the results (the combine would weigh them by
    // 2^0 / 1), so it writes them and no combine is launched.
    p.out = out;
    p.out_bf16 = out_dtype == BT_DTYPE_BF16;
    p.out_stride_seq = out_stride_seq > 0 ? out_stride_seq : (int64_t)heads * head_dim;
  }
  rc = hip_rc(bt::launch_decode_split(p, head_dim, num_split, batch, (hipStream_t)stream));
  if (rc || num_split == 1) return rc;
  return bt_gqa_decode_combine(lse, part, batch, heads, head_dim, num_split, nullptr, nullptr,
                               total, out, out_dtype, out_stride_seq, stream);
}

}  // extern "C"

// Split workspace of bt_gqa_decode_noalloc: one copy per GPU, held from the
// library's load on that GPU until the process ends.  Host code never names it
// as a device address: it uses the pointer hipGetSymbolAddress returns for the
// current device.
static __device__ __align__(256) unsigned char scratch[BT_NOALLOC_SCRATCH_BYTES];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device, looked up once per
// device with that device current.
int scratch_address(void** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return (int)e;
  if (dev < 0 || dev >= kMaxDevices) return BT_ENOTSUP;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch_ptr[dev] == nullptr) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return (int)e;
    if (ptr == nullptr) return (int)hipErrorInvalidSymbol;
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return BT_OK;
}

}  // namespace

extern "C" {

int bt_gqa_decode_noalloc(const void* q, int32_t q_dtype, int64_t q_stride_seq, const void* k,
                          const void* v, int64_t kv_stride_tok, int64_t kv_stride_head,
                          const int64_t* seq_offset, const int32_t* pos, const int32_t* seq_len,
                          int32_t seqlen, int32_t batch, int32_t heads, int32_t kv_heads,
                          int32_t head_dim, int32_t num_split, float scale, void* out,
                          int32_t out_dtype, int64_t out_stride_seq, void* stream) {
  int rc = check_decode_common(q, q_dtype, q_stride_seq, k, v, kv_stride_tok, kv_stride_head,
                               batch, heads, kv_heads, head_dim);
  if (rc) return rc;
  if (num_split < 1) return BT_EINVAL;
  if (num_split > bt::kMaxSplitsPerSeq || (int64_t)batch * num_split > INT32_MAX / 2) return BT_ENOTSUP;
  if (bt_decode_workspace_bytes(heads, head_dim, batch * num_split) > (int64_t)BT_NOALLOC_SCRATCH_BYTES)
    return BT_ENOSPC;
  void* ws = nullptr;
  rc = scratch_address(&ws);
  if (rc) return rc;
  // Every split writes its lse (-inf when it has no tokens) before the combine
  // reads it, and the combine reads only the partials of splits with tokens,
  // so nothing left in the scratch by an earlier call is ever used.
  return bt_gqa_decode(q, q_dtype, q_stride_seq, k, v, kv_stride_tok, kv_stride_head, seq_offset, pos,
                       seq_len, seqlen, batch, heads, kv_heads, head_dim, num_split, scale, ws,
                       (int64_t)BT_NOALLOC_SCRATCH_BYTES, out, out_dtype, out_stride_seq, stream);
}

int32_t bt_ragged_plan(const int32_t* lens, int32_t batch, int32_t target_groups, int32_t* work,
                       int32_t work_capacity, int32_t* split_base, int32_t* split_count,
                       int32_t* total_splits) {
  return bt_ragged_plan_rounds(lens, batch, target_groups, target_groups, work, work_capacity, split_base,
                               split_count, total_splits);
}

int32_t bt_ragged_plan_rounds(const int32_t* lens, int32_t batch, int32_t round_groups, int32_t target_groups,
                              int32_t* work, int32_t work_capacity, int32_t* split_base, int32_t* split_count,
                              int32_t* total_splits) {
  return bt_ragged_plan_cost(lens, batch, round_groups, target_groups, 0, work, work_capacity, split_base,
                             split_count, total_splits);
}

int32_t bt_ragged_plan_cost(const int32_t* lens, int32_t batch, int32_t round_groups, int32_t target_groups,
                            int32_t split_tokens, int32_t* work, int32_t work_capacity, int32_t* split_base,
                            int32_t* split_count, int32_t* total_splits) {
  if (!lens || !work || !split_base || !split_count || !total_splits) return BT_EINVAL;
  if (batch < 1 || round_groups < 1 || target_groups < 1 || split_tokens < 0) return BT_EINVAL;
  int32_t max_len = 1;
  int64_t tokens = 0;
  for (int32_t b = 0; b < batch; ++b) {
    if (lens[b] < 0) return BT_EINVAL;
    max_len = std::max(max_len, lens[b]);
    tokens += lens[b];
  }
  // Splits of sequence b under a cap of T tokens per split: ceil(len / T),
  // at least 1, at most one per 32 tokens and kMaxSplitsPerSeq.
  auto splits_of = [](int32_t len, int32_t cap) {
    int64_t ns = ((int64_t)len + cap - 1) / cap;
    ns = std::min<int64_t>(ns, ((int64_t)len + 31) / 32);
    ns = std::min<int64_t>(ns, bt::kMaxSplitsPerSeq);
    return (int32_t)std::max<int64_t>(ns, 1);
  };
  auto count_at = [&](int32_t cap) {
    int64_t n = 0;
    for (int32_t b = 0; b < batch; ++b) n += splits_of(lens[b], cap);
    return n;
  };
  // The smallest cap whose split total fits `target` (the count only falls as
  // the cap grows): every work-group then streams at most that many tokens and
  // the batch runs in rounds of work-groups per kv head.  A batch with more
  // sequences than `target` gets one split each.
  auto cap_for = [&](int32_t target) {
    int32_t lo = 1, hi = max_len;
    while (lo < hi) {
      const int32_t mid = lo + (hi - lo) / 2;
      if (count_at(mid) <= target) hi = mid;
      else lo = mid + 1;
    }
    return lo;
  };
  int32_t cap = cap_for(round_groups);
  if (target_groups != round_groups) {
    int64_t longest = 0;
    for (int32_t b = 0; b < batch; ++b) {
      const int64_t ns = splits_of(lens[b], cap);
      longest = std::max(longest, (lens[b] + ns - 1) / ns);
    }
    const int64_t n = count_at(cap);
    if (!bt::ragged_round_is_even(n, longest, tokens, round_groups)) {
      const int32_t more = cap_for(target_groups);
      if (bt::ragged_splits_pay(n, longest, count_at(more), more, round_groups, split_tokens)) cap = more;
    }
  }
  int32_t total = 0;
  for (int32_t b = 0; b < batch; ++b) {
    const int32_t ns = splits_of(lens[b], cap);
    if ((int64_t)total + ns > work_capacity) return BT_ENOSPC;
    split_base[b] = total;
    split_count[b] = ns;
    total += ns;
  }
  // Work entries, longest splits first (when the grid takes more than one
  // round, the long ones start early).
  std::vector<int32_t> order(batch);
  for (int32_t b = 0; b < batch; ++b) order[b] = b;
  std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t c) {
    return (int64_t)lens[a] * split_count[c] > (int64_t)lens[c] * split_count[a];
  });
  int64_t i = 0;
  for (const int32_t b : order) {
    for (int32_t s = 0; s < split_count[b]; ++s, ++i) {
      int32_t* w = work + 4 * i;
      w[0] = b;
      w[1] = s;
      w[2] = split_count[b];
      w[3] = split_base[b];
    }
  }
  *total_splits = total;
  return total;
}

int bt_ragged_plan_device(const int32_t* seq_len, int32_t batch, int32_t target_groups, int32_t* work,
                          int32_t work_capacity, int32_t* split_base, int32_t* split_count,
                          int32_t* total_splits, void* stream) {
  return bt_ragged_plan_rounds_device(seq_len, batch, target_groups, target_groups, work, work_capacity, split_base,
                                      split_count, total_splits, stream);
}

int bt_ragged_plan_rounds_device(const int32_t* seq_len, int32_t batch, int32_t round_groups, int32_t target_groups,
                                 int32_t* work, int32_t work_capacity, int32_t* split_base, int32_t* split_count,
                                 int32_t* total_splits, void* stream) {
  return bt_ragged_plan_cost_device(seq_len, batch, round_groups, target_groups, 0, work, work_capacity, split_base,
                                    split_count, total_splits, stream);
}

int bt_ragged_plan_cost_device(const int32_t* seq_len, int32_t batch, int32_t round_groups, int32_t target_groups,
                               int32_t split_tokens, int32_t* work, int32_t work_capacity, int32_t* split_base,
                               int32_t* split_count, int32_t* total_splits, void* stream) {
  if (!seq_len || !work || !split_base || !split_count) return BT_EINVAL;
  if (batch < 1 || round_groups < 1 || target_groups < 1 || split_tokens < 0 || !aligned16(work)) return BT_EINVAL;
  if (batch > bt::kRaggedPlanMaxBatch) return BT_ENOTSUP;
  if (work_capacity < std::max(batch, std::max(round_groups, target_groups))) return BT_ENOSPC;
  bt::RaggedPlanParams p{};
  p.seq_len = seq_len;
  p.batch = batch;
  p.round_groups = round_groups;
  p.split_tokens = split_tokens;
  p.target_groups = target_groups;
  p.work = work;
  p.work_capacity = work_capacity;
  p.split_base = split_base;
  p.split_count = split_count;
  p.total = total_splits;
  return hip_rc(bt::launch_ragged_plan(p, (hipStream_t)stream));
}

int bt_gqa_decode_ragged(const void* q, int32_t q_dtype, int64_t q_stride_seq, const void* k,
                         const void* v, int64_t kv_stride_tok, int64_t kv_stride_head,
                         const int64_t* seq_offset, const int32_t* seq_len, int32_t batch,
                         int32_t heads, int32_t kv_heads, int32_t head_dim, const int32_t* work,
                         int32_t num_work, const int32_t* split_base, const int32_t* split_count,
                         int32_t total_splits, float scale, void* workspace,
                         int64_t workspace_bytes, void* out, int32_t out_dtype,
                         int64_t out_stride_seq, void* stream) {
  int rc = check_decode_common(q, q_dtype, q_stride_seq, k, v, kv_stride_tok, kv_stride_head,
                               batch, heads, kv_heads, head_dim);
  if (rc) return rc;
  rc = check_out(out, out_dtype, out_stride_seq, batch, heads, head_dim);
  if (rc) return rc;
  if (!seq_offset || !seq_len || !work || !split_base || !split_count) return BT_EINVAL;
  if (num_work < 1 || total_splits < num_work) return BT_EINVAL;
  if (!workspace || !aligned16(workspace)) return BT_EINVAL;
  if (workspace_bytes < bt_decode_workspace_bytes(heads, head_dim, total_splits)) return BT_ENOSPC;
  if (!aligned16(work)) return BT_EINVAL;
  float* lse = static_cast<float*>(workspace);
  float* part = reinterpret_cast<float*>(static_cast<char*>(workspace) +
                                         align256((int64_t)heads * total_splits * 4));
  bt::DecodeSplitParams p = make_split_params(q, q_dtype, q_stride_seq, k, v, kv_stride_tok,
                                              kv_stride_head, seq_offset, nullptr, seq_len, 0,
                                              heads, kv_heads, head_dim, scale, lse, part);
  p.work = reinterpret_cast<const int4*>(work);
  p.num_split = 0;
  p.total_splits = total_splits;
  rc = hip_rc(bt::launch_decode_split(p, head_dim, num_work, 1, (hipStream_t)stream));
  if (rc) return rc;
  return bt_gqa_decode_combine(lse, part, batch, heads, head_dim, 0, split_base, split_count,
                               total_splits, out, out_dtype, out_stride_seq, stream);
}

int64_t bt_prefill_workspace_bytes(int32_t kv_len, int32_t kv_heads, int32_t head_dim) {
  if (kv_len < 1 || kv_heads < 1 || head_dim < 1) return 0;
  return prefill_base_bytes(kv_len, kv_heads, head_dim);
}

int64_t bt_prefill_split_workspace_bytes(int32_t seqlen, int32_t q_offset, int32_t heads, int32_t kv_heads,
                                         int32_t head_dim) {
  if (seqlen < 1 || q_offset < 0 || heads < 1 || kv_heads < 1 || heads % kv_heads || head_dim < 1) return 0;
  if ((int64_t)q_offset + seqlen > INT32_MAX) return 0;
  const int64_t vt = prefill_base_bytes(q_offset + seqlen, kv_heads, head_dim);
  const int64_t part = bt_prefill_partials_bytes(seqlen, q_offset, heads, kv_heads, head_dim);
  return part > 0 ? align256(vt) + part : vt;
}

// Shared by bt_gqa_prefill and bt_gqa_prefill_cached: validates the call and
// launches the pre-pass and the attention kernel.  `images` holds the K / V^T
// images and their exponents laid out for img_keys keys (prefill_layout); the
// pre-pass converts the blocks from key img_first_key on.  `partials` (may be
// null) holds the split-key partials when it is large enough.
static int prefill_run(const void* q, int32_t q_dtype, const void* k, const void* v, int64_t q_stride_tok,
                       int64_t q_stride_head, int64_t kv_stride_tok, int64_t kv_stride_head, int32_t seqlen,
                       int32_t q_offset, int32_t heads, int32_t kv_heads, int32_t head_dim, float scale,
                       void* images, int32_t img_keys, int32_t img_first_key, bool keep_images,
                       void* partials, int64_t partials_bytes, void* out, int32_t out_dtype,
                       int64_t out_stride_tok, int64_t out_stride_head, void* stream) {
  if (!q || !k || !v || !out || !images) return BT_EINVAL;
  if (seqlen < 1 || q_offset < 0 || heads < 1 || kv_heads < 1 || heads % kv_heads) return BT_EINVAL;
  if ((int64_t)q_offset + seqlen > INT32_MAX) return BT_EINVAL;
  if (out_dtype != BT_DTYPE_F32 && out_dtype != BT_DTYPE_BF16) return BT_EINVAL;
  if (q_dtype != BT_DTYPE_F32 && q_dtype != BT_DTYPE_BF16) return BT_EINVAL;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out)) return BT_EINVAL;
  if (q_stride_tok <= 0 || q_stride_head <= 0 || kv_stride_tok <= 0 || kv_stride_head < 0 ||
      out_stride_tok <= 0 || out_stride_head <= 0)
    return BT_EINVAL;
  if (q_stride_tok % 8 || q_stride_head % 8 || kv_stride_tok % 8 || kv_stride_head % 8 ||
      out_stride_tok % 8 || out_stride_head % 8)
    return BT_EINVAL;
  if (!aligned16(images) || (partials && !aligned16(partials))) return BT_EINVAL;
  if (head_dim != 256 && head_dim != 128) return BT_ENOTSUP;
  if (heads / kv_heads > 8) return BT_ENOTSUP;
  // 32-bit buffer offsets: the K rows of one kv head (plus the last block's
  // tail) and its images
  const int32_t kv_len = q_offset + seqlen;
  if (img_keys < kv_len || img_first_key < 0 || img_first_key > q_offset) return BT_EINVAL;
  const int64_t nblk = ((int64_t)kv_len + bt::kPrefillKeyBlock - 1) / bt::kPrefillKeyBlock;
  const int64_t img_blocks = ((int64_t)img_keys + bt::kPrefillKeyBlock - 1) / bt::kPrefillKeyBlock;
  if ((nblk + 1) * bt::kPrefillKeyBlock * kv_stride_tok * 2 > (int64_t)UINT32_MAX ||
      img_blocks * bt::kPrefillKeyBlock * head_dim * 2 > (int64_t)UINT32_MAX)
    return BT_ENOTSUP;
  bt::PrefillParams p{};
  p.q = static_cast<const uint16_t*>(q);
  p.k = static_cast<const uint16_t*>(k);
  p.v = static_cast<const uint16_t*>(v);
  p.q_stride_tok = q_stride_tok;
  p.q_stride_head = q_stride_head;
  p.kv_stride_tok = kv_stride_tok;
  p.kv_stride_head = kv_stride_head;
  p.seqlen = seqlen;
  p.q_offset = q_offset;
  p.heads = heads;
  p.kv_heads = kv_heads;
  p.group = heads / kv_heads;
  p.scale_log2 = (float)((double)scale * kLog2e);
  p.out = out;
  p.out_bf16 = out_dtype == BT_DTYPE_BF16;
  p.out_stride_tok = out_stride_tok;
  p.out_stride_head = out_stride_head;
  const PrefillLayout lay = prefill_layout(img_keys, kv_heads, head_dim);
  p.vt = static_cast<uint16_t*>(images);
  p.vexp = reinterpret_cast<int32_t*>(static_cast<char*>(images) + lay.vexp);
  p.kimg = reinterpret_cast<uint16_t*>(static_cast<char*>(images) + lay.kimg);
  p.kexp = reinterpret_cast<int32_t*>(static_cast<char*>(images) + lay.kexp);
  p.img_blocks = (int32_t)img_blocks;
  p.img_first = img_first_key / bt::kPrefillKeyBlock;
  p.q_f32 = q_dtype == BT_DTYPE_F32 ? 1 : 0;
  p.keep_images = keep_images ? 1 : 0;
  const PrefillChoice choice = prefill_choice(seqlen, q_offset, heads, kv_heads, head_dim, p.q_f32 != 0,
                                              partials ? partials_bytes : 0);
  const bt::PrefillSplitPlan& plan = choice.plan;
  if (choice.pair)
    return hip_rc(bt::launch_prefill_pair(p, head_dim, (hipStream_t)stream));
  // Every other shape runs two waves per SIMD (groups of 3, 5, 6, 7 as
  // subsets of 1 or 2 heads).  When one work-group per query block would
  // leave CUs idle or the causal triangle's work is uneven, the key ranges are
  // split.
  if (bt::prefill8_serves(p.group, head_dim)) {
    p.sub_group = bt::prefill8_sub_group(p.group);
    p.head_subs = p.group / p.sub_group;
    if (plan.active()) {
      p.kb_chunk = plan.kb_chunk;
      p.split_compact = plan.compact;
      p.pair_parts = plan.pair_parts;
      p.max_chunks = plan.max_chunks;
      if (plan.uses_partials()) {
        p.part_blocks = plan.part_blocks;
        p.part = static_cast<float*>(partials);
        p.lse = p.part + plan.part_rows * (size_t)head_dim;
      }
    }
    return hip_rc(bt::launch_prefill8(p, head_dim, (hipStream_t)stream));
  }
  return BT_ENOTSUP;
}

int bt_gqa_prefill(const void* q, int32_t q_dtype, const void* k, const void* v, int64_t q_stride_tok,
                   int64_t q_stride_head, int64_t kv_stride_tok, int64_t kv_stride_head,
                   int32_t seqlen, int32_t q_offset, int32_t heads, int32_t kv_heads,
                   int32_t head_dim, float scale, void* workspace, int64_t workspace_bytes,
                   void* out, int32_t out_dtype, int64_t out_stride_tok, int64_t out_stride_head,
                   void* stream) {
  if (!workspace) return BT_EINVAL;
  if (seqlen < 1 || q_offset < 0 || heads < 1 || kv_heads < 1 || heads % kv_heads) return BT_EINVAL;
  if ((int64_t)q_offset + seqlen > INT32_MAX) return BT_EINVAL;
  const int32_t kv_len = q_offset + seqlen;
  if (workspace_bytes < bt_prefill_workspace_bytes(kv_len, kv_heads, head_dim)) return BT_ENOSPC;
  // the split-key partials follow the images (256-byte aligned)
  const int64_t part_offset = align256(prefill_base_bytes(kv_len, kv_heads, head_dim));
  void* partials = workspace_bytes > part_offset ? static_cast<char*>(workspace) + part_offset : nullptr;
  return prefill_run(q, q_dtype, k, v, q_stride_tok, q_stride_head, kv_stride_tok, kv_stride_head, seqlen,
                     q_offset, heads, kv_heads, head_dim, scale, workspace, kv_len, 0, false, partials,
                     partials ? workspace_bytes - part_offset : 0, out, out_dtype, out_stride_tok,
                     out_stride_head, stream);
}

int64_t bt_prefill_partials_bytes(int32_t seqlen, int32_t q_offset, int32_t heads, int32_t kv_heads,
                                  int32_t head_dim) {
  if (seqlen < 1 || q_offset < 0 || heads < 1 || kv_heads < 1 || heads % kv_heads || head_dim < 1) return 0;
  if ((int64_t)q_offset + seqlen > INT32_MAX) return 0;
  const bt::PrefillSplitPlan plan = prefill8_plan(seqlen, q_offset, heads, kv_heads, head_dim);
  if (!plan.uses_partials()) return 0;
  // The pair kernel needs none; the query type, which decides between the
  // kernels, is not known here.
  const bool never = prefill_pair_faster(plan, seqlen, q_offset, heads, kv_heads, head_dim, false) &&
                     prefill_pair_faster(plan, seqlen, q_offset, heads, kv_heads, head_dim, true);
  return never ? 0 : (int64_t)plan.part_bytes;
}

int bt_prefill_plan(int32_t seqlen, int32_t q_offset, int32_t heads, int32_t kv_heads, int32_t head_dim,
                    int32_t q_dtype, int64_t partials_bytes, int32_t* plan) {
  if (!plan || seqlen < 1 || q_offset < 0 || heads < 1 || kv_heads < 1 || heads % kv_heads) return BT_EINVAL;
  if ((int64_t)q_offset + seqlen > INT32_MAX) return BT_EINVAL;
  if (q_dtype != BT_DTYPE_F32 && q_dtype != BT_DTYPE_BF16) return BT_EINVAL;
  if (!bt::prefill8_serves(heads / kv_heads, head_dim)) return BT_ENOTSUP;
  const PrefillChoice c =
      prefill_choice(seqlen, q_offset, heads, kv_heads, head_dim, q_dtype == BT_DTYPE_F32, partials_bytes);
  plan[0] = c.pair ? 1 : 0;
  plan[1] = c.pair ? 0 : c.plan.kb_chunk;
  plan[2] = c.pair ? 1 : c.plan.max_chunks;
  plan[3] = c.pair ? 0 : c.plan.compact;
  plan[4] = c.pair ? 0 : c.plan.pair_parts;
  return BT_OK;
}

int bt_prefill_longest_first(int32_t seqlen, int32_t q_offset, int32_t heads, int32_t kv_heads, int32_t kb_chunk,
                             int32_t item, int32_t* out) {
  if (!out || seqlen < 1 || q_offset < 0 || heads < 1 || kv_heads < 1 || heads % kv_heads) return BT_EINVAL;
  if ((int64_t)q_offset + seqlen > INT32_MAX - bt::kPrefillKeyBlock) return BT_EINVAL;
  const int group = heads / kv_heads, sub = bt::prefill8_sub_group(group);
  const int nkb = (q_offset + seqlen + bt::kPrefillKeyBlock - 1) / bt::kPrefillKeyBlock;
  if (group > 8 || kb_chunk < (nkb + 1) / 2 || kb_chunk > nkb) return BT_EINVAL;
  const int subsets = kv_heads * (group / sub);
  out[0] = out[1] = out[2] = 0;
  const int items = bt::prefill8_longest_first(seqlen, q_offset, sub, subsets, kb_chunk, -1, out, out + 1, out + 2);
  if (item < 0) return items;
  if (item >= items) return BT_EINVAL;
  return bt::prefill8_longest_first(seqlen, q_offset, sub, subsets, kb_chunk, item, out, out + 1, out + 2);
}

int bt_gqa_prefill_cached(const void* q, int32_t q_dtype, const void* k, const void* v, int64_t q_stride_tok,
                          int64_t q_stride_head, int64_t kv_stride_tok, int64_t kv_stride_head, int32_t seqlen,
                          int32_t q_offset, int32_t heads, int32_t kv_heads, int32_t head_dim, float scale,
                          void* images, int64_t images_bytes, int32_t capacity, int32_t cached_keys,
                          void* partials, int64_t partials_bytes, void* out, int32_t out_dtype,
                          int64_t out_stride_tok, int64_t out_stride_head, void* stream) {
  if (capacity < 1 || (int64_t)q_offset + seqlen > capacity) return BT_EINVAL;
  if (cached_keys < 0 || cached_keys > q_offset) return BT_EINVAL;
  if (images_bytes < bt_prefill_workspace_bytes(capacity, kv_heads, head_dim)) return BT_ENOSPC;
  return prefill_run(q, q_dtype, k, v, q_stride_tok, q_stride_head, kv_stride_tok, kv_stride_head, seqlen,
                     q_offset, heads, kv_heads, head_dim, scale, images, capacity, cached_keys, true,
                     partials, partials_bytes, out, out_dtype, out_stride_tok, out_stride_head, stream);
}

static bool prep_dim_served(int32_t d) { return d == 64 || d == 128 || d == 256 || d == 512; }

int bt_rms_norm_rope(const float* x, int64_t x_stride, int32_t rows, int32_t dim, const float* w,
                     float eps, const float* cos, const float* sin, const int32_t* pos,
                     int32_t rope_dim, int32_t rope_cap, float* out, int64_t out_stride,
                     void* stream) {
  if (!x || !out || rows < 1 || dim < 1 || x_stride < dim || out_stride < dim) return BT_EINVAL;
  if ((cos == nullptr) != (sin == nullptr)) return BT_EINVAL;
  if (cos && (!pos || rope_dim < 2 || rope_dim % 2 || rope_dim > dim || rope_cap < 1)) return BT_EINVAL;
  if (!w && !cos) return BT_EINVAL;
  if (!(eps >= 0.f)) return BT_EINVAL;
  if (!prep_dim_served(dim)) return BT_ENOTSUP;
  bt::RowPrepParams p{};
  p.x = x;
  p.x_stride = x_stride;
  p.rows = rows;
  p.out = out;
  p.out_stride = out_stride;
  p.w = w;
  p.eps = eps;
  p.cos = cos;
  p.sin = sin;
  p.pos = pos;
  p.rope_dim = cos ? rope_dim : 0;
  p.rope_cap = rope_cap;
  return hip_rc(bt::launch_row_norm_rope(p, dim, (hipStream_t)stream));
}

int bt_attn_prep(const float* qkv, int32_t heads, int32_t kv_heads, int32_t head_dim,
                 const float* q_norm, const float* k_norm, float eps, const float* cos,
                 const float* sin, const int32_t* pos, int32_t rope_dim, int32_t rope_cap,
                 void* q_out, int32_t q_dtype, void* cache_k, void* cache_v, int64_t kv_stride_tok,
                 int64_t kv_stride_head, int32_t cache_cap, void* stream) {
  if (!qkv || !pos || !q_out || !cache_k || !cache_v) return BT_EINVAL;
  if (heads < 1 || kv_heads < 1 || head_dim < 1 || cache_cap < 1) return BT_EINVAL;
  if ((q_norm == nullptr) != (k_norm == nullptr)) return BT_EINVAL;
  if ((cos == nullptr) != (sin == nullptr)) return BT_EINVAL;
  if (cos && (rope_dim < 2 || rope_dim % 2 || rope_dim > head_dim || rope_cap < 1)) return BT_EINVAL;
  if (q_dtype != BT_DTYPE_F32 && q_dtype != BT_DTYPE_BF16) return BT_EINVAL;
  if (kv_stride_tok < 1 || kv_stride_head < 1) return BT_EINVAL;
  if (!(eps >= 0.f)) return BT_EINVAL;
  if (!prep_dim_served(head_dim)) return BT_ENOTSUP;
  bt::RowPrepParams p{};
  p.x = qkv;
  p.w = q_norm;
  p.wk = k_norm;
  p.eps = eps;
  p.cos = cos;
  p.sin = sin;
  p.pos = pos;
  p.rope_dim = cos ? rope_dim : 0;
  p.rope_cap = rope_cap;
  p.heads = heads;
  p.kv_heads = kv_heads;
  p.q_out = q_out;
  p.q_out_bf16 = q_dtype == BT_DTYPE_BF16;
  p.cache_k = static_cast<uint16_t*>(cache_k);
  p.cache_v = static_cast<uint16_t*>(cache_v);
  p.kv_stride_tok = kv_stride_tok;
  p.kv_stride_head = kv_stride_head;
  p.cache_cap = cache_cap;
  return hip_rc(bt::launch_attn_prep(p, head_dim, (hipStream_t)stream));
}

int bt_gdn_decode(const float* q, const float* k, const float* v, const float* g, const float* beta,
                  float* state, int32_t heads_k, int32_t heads_v, int32_t dim, float scale, float eps,
                  float* out, void* stream) {
  if (!q || !k || !v || !g || !beta || !state || !out) return BT_EINVAL;
  if (heads_k < 1 || heads_v < 1 || heads_v % heads_k || dim < 1) return BT_EINVAL;
  if (!aligned16(v) || !aligned16(state) || !aligned16(out)) return BT_EINVAL;
  if (!(eps >= 0.f)) return BT_EINVAL;
  if (dim != 64 && dim != 128) return BT_ENOTSUP;
  bt::GdnParams p{};
  p.q = q;
  p.k = k;
  p.v = v;
  p.g = g;
  p.beta = beta;
  p.state = state;
  p.out = out;
  p.heads_k = heads_k;
  p.heads_v = heads_v;
  p.scale = scale;
  p.eps = eps;
  return hip_rc(bt::launch_gdn_decode(p, dim, (hipStream_t)stream));
}

int64_t bt_gemv_workspace_bytes(int32_t K, int32_t N) {
  if (K < 1 || N < 1) return 0;
  return (int64_t)bt::gemv_workspace_bytes(K, N);
}

int bt_gemv_plan(const void* w, int64_t ldw, int32_t K, int32_t N, int32_t* plan) {
  if (!plan || K < 1 || N < 1 || ldw < N) return BT_EINVAL;
  if (N % 8 || ldw % 8 || !aligned16(w)) return BT_EINVAL;
  const bt::GemvShape g = bt::gemv_shape(K, N, ldw * 2, reinterpret_cast<uintptr_t>(w));
  plan[0] = g.lanes > 0 ? 1 : 0;
  plan[1] = g.lanes > 0 ? 8 * g.lanes : 64 * g.vec;
  plan[2] = g.splits;
  return BT_OK;
}

int bt_gemv_bf16(const float* x, const void* w, int64_t ldw, int32_t K, int32_t N, float* y,
                 void* workspace, int64_t workspace_bytes, void* stream) {
  if (!x || !w || !y || K < 1 || N < 1 || ldw < N) return BT_EINVAL;
  if (N % 8 || ldw % 8 || !aligned16(w)) return BT_EINVAL;
  if ((int64_t)K * ldw * 2 > (int64_t)INT32_MAX) return BT_ENOTSUP;
  const bt::GemvShape shape = bt::gemv_shape(K, N, ldw * 2, reinterpret_cast<uintptr_t>(w));
  const int64_t need = (int64_t)shape.splits * N * 4;
  if (shape.splits > 1 && (!workspace || !aligned16(workspace) || workspace_bytes < need)) return BT_ENOSPC;
  bt::GemvParams p{};
  p.x = x;
  p.w = static_cast<const uint16_t*>(w);
  p.ldw = ldw;
  p.K = K;
  p.N = N;
  p.splits = shape.splits;
  p.partial = static_cast<float*>(workspace);
  p.y = y;
  return hip_rc(bt::launch_gemv(p, shape, (hipStream_t)stream));
}

}  // extern "C"
