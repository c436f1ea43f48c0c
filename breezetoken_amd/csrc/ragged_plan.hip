// Ragged-batch split plan computed on the device from device lengths, so a
// multi-sequence decode step needs no host synchronisation and can be captured
// in a hipGraph.  It makes exactly the plan bt_ragged_plan_cost (and with
// round_groups = target_groups, bt_ragged_plan) makes on the host:
//  * ns_b = ceil(len_b / T), at least 1, at most ceil(len_b / 32) and
//    kMaxSplitsPerSeq, for the smallest token cap T whose total fits
//    round_groups, or target_groups where the former leaves the batch uneven and
//    the further splits pay;
//  * split_base[b] = sum of ns over sequences before b, split_count[b] = ns_b;
//  * work entries {b, s, ns_b, base_b}, sequences ordered by tokens per split,
//    largest first (ties by index, as a stable sort);
// and pads the work table to its capacity with entries {-1, 0, 0, 0}, which the
// split kernel skips.  One work-group of 1024 threads; batch <= 4096.
//
// The kernel is one serial chain of LDS round trips and barriers, so what
// bounds it is their number.  The search for T takes up to 16 candidates per
// round (a wave or a few waves count each one's splits), i.e. 4 to 5 rounds
// where a bisection took 15 to 17 with two barriers each; scans step through
// lanes, not LDS; the order's comparisons are spread over all threads, and every
// work entry finds its sequence by a search over the scanned starts instead of
// a thread writing all splits of a sequence.  As nodes of a graph, batch 4 / 32
// / 144 / 512 / 1500 / 4096: 11.2 / 15.6 / 19.4 / 38.7 / 159 / 1060 -> 6.5 / 7.5
// / 11.7 / 25 / 42 / 89 us.
#include "bt_common.h"
#include "bt_kernels.h"

namespace bt {

namespace {

constexpr int kPlanThreads = 1024;
constexpr int kPlanWaves = kPlanThreads / 64;
constexpr int kRankMax = 256;  // sequences whose order is found by counting ranks

// A cap T on the tokens per split, with 1 / T to 2^-45 for its quotients.
struct PlanCap {
  double inv;
  __device__ explicit PlanCap(int T) {
    const double d = (double)T, r = (double)__builtin_amdgcn_rcpf((float)T);
    inv = r * fma(-d, r, 2.0);  // one Newton step on the float reciprocal
  }
  // bt_ragged_plan's split count (len >= 0).  (len - 1/2) / T lies at least
  // 1 / (2T) from an integer and its product is off by at most 2^-14 / T, so
  // it rounds down to floor((len - 1) / T); an integer division takes ten
  // times the time.
  __device__ __forceinline__ int splits(int len) const {
    const int by_cap = (int)(((double)len - 0.5) * inv) + 1;
    const int ns = min(min(by_cap, (int)((uint32_t)(len - 1) / 32u) + 1), kMaxSplitsPerSeq);
    return len > 0 ? ns : 1;
  }
};

// Whether sequence c {length, splits} comes ahead of b: more tokens per split
// (len_c / ns_c > len_b / ns_b, cross-multiplied), ties by index.  The
// products stay below 2^43, so float64 holds them exactly (its multiply runs
// at four times the rate of the 64-bit integer one).
__device__ __forceinline__ bool ahead(int2 sc, int c, int2 sb, int b) {
  const double lhs = (double)sc.x * (double)sb.y, rhs = (double)sb.x * (double)sc.y;
  return lhs > rhs || (lhs == rhs && c < b);
}

__device__ __forceinline__ int wave_add(int x) { return (int)wave_op_desc((uint32_t)x, OpIAdd{}); }
__device__ __forceinline__ int wave_imax(int x) { return (int)wave_op_desc((uint32_t)x, OpIMax{}); }

struct PlanShared {
  int2 seq[kRaggedPlanMaxBatch];     // {length, splits}
  int base[kRaggedPlanMaxBatch];
  int start[kRaggedPlanMaxBatch];    // by rank: splits, then their exclusive scan
  int order[kRaggedPlanMaxBatch];    // by rank: the sequence
  int rank[kRankMax];
  int count[2][kPlanWaves];          // splits at each candidate, two rounds' worth
  int wave_sum[kPlanWaves];
  int longest[kPlanWaves];
  long long tokens[kPlanWaves];
};

// Exclusive prefix sum of in(0) .. in(n - 1) into out; returns the total.  Up
// to 1024 values per pass: a lane scan, then the waves' totals.
template <typename In>
__device__ int block_scan(int n, int* out, int* wave_sum, In in) {
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  int carry = 0;
  for (int j0 = 0; j0 < n; j0 += kPlanThreads) {
    const int j = j0 + t;
    const int x = j < n ? in(j) : 0;
    int incl = x;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int up = __shfl_up(incl, off);
      if (lane >= off) incl += up;
    }
    __syncthreads();  // wave_sum may still be read from the previous pass
    if (lane == 63) wave_sum[wave] = incl;
    __syncthreads();
    int before = carry, all = carry;
#pragma unroll
    for (int w = 0; w < kPlanWaves; ++w) {
      const int ws = wave_sum[w];
      before += w < wave ? ws : 0;
      all += ws;
    }
    if (j < n) out[j] = before + incl - x;
    carry = all;
  }
  return carry;
}

// The smallest T in [1, max_len] whose splits total at most `target`, or
// max_len if none does (the total only falls as T grows).  Every thread
// returns it.  Each round splits [lo, hi) at NC candidates, counted by
// kPlanWaves / NC waves each, and keeps the interval in which the total first
// fits.
template <int NC>
__device__ int find_cap(PlanShared& sh, int B, int target, int max_len) {
  constexpr int kWavesEach = kPlanWaves / NC;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int cand = wave / kWavesEach;
  int lo = 1, hi = max_len;
  for (int round = 0; lo < hi; round ^= 1) {  // uniform: every thread sees the same counts
    // Candidates lo + (c + 1) * step - 1, c < NC, all in [lo, hi).
    const uint32_t step = (uint32_t)(hi - lo) / (NC + 1) + 1;
    auto at = [&](int c) { return (int)min((uint32_t)lo + (uint32_t)(c + 1) * step - 1, (uint32_t)hi - 1); };
    const PlanCap T(at(cand));
    int part = 0;
    for (int b = (wave % kWavesEach) * 64 + lane; b < B; b += kWavesEach * 64) part += T.splits(sh.seq[b].x);
    part = wave_add(part);
    if (lane == 0) sh.count[round][wave] = part;
    __syncthreads();  // the next round writes the other half: one barrier a round
    int n = 0;
#pragma unroll
    for (int w = 0; w < kWavesEach; ++w) n += sh.count[round][(lane % NC) * kWavesEach + w];
    const uint64_t fits = __builtin_amdgcn_ballot_w64(lane < NC && n <= target);
    const int first = fits ? __builtin_ctzll(fits) : NC;
    const int lo_next = first > 0 ? at(first - 1) + 1 : lo;
    if (first < NC) hi = at(first);
    lo = lo_next;
  }
  __syncthreads();  // count is free for another search
  return lo;
}

__device__ int plan_cap(PlanShared& sh, int B, int target, int max_len) {
  return B <= 512 ? find_cap<16>(sh, B, target, max_len) : find_cap<4>(sh, B, target, max_len);
}

__global__ __launch_bounds__(kPlanThreads) void ragged_plan_kernel(RaggedPlanParams p) {
  __shared__ PlanShared sh;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int B = p.batch;

  int mx = 1;
  long long tokens = 0;
  for (int b = t; b < B; b += kPlanThreads) {
    const int len = max(p.seq_len[b], 0);
    sh.seq[b] = int2{len, 1};
    if (b < kRankMax) sh.rank[b] = 0;
    mx = max(mx, len);
    tokens += len;
  }
  mx = wave_imax(mx);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) tokens += __shfl_xor(tokens, off);
  if (lane == 0) {
    sh.longest[wave] = mx;
    sh.tokens[wave] = tokens;
  }
  __syncthreads();
  int max_len = 1;
  tokens = 0;
#pragma unroll
  for (int w = 0; w < kPlanWaves; ++w) {
    max_len = max(max_len, sh.longest[w]);
    tokens += sh.tokens[w];
  }

  // Splits under `cap`, their first entries and their total.
  auto assign = [&](int cap) {
    const PlanCap T(cap);
    for (int b = t; b < B; b += kPlanThreads) sh.seq[b].y = T.splits(sh.seq[b].x);
    __syncthreads();
    return block_scan(B, sh.base, sh.wave_sum, [&](int b) { return sh.seq[b].y; });
  };
  const int cap = plan_cap(sh, B, p.round_groups, max_len);
  bool one_round = true;
  int n = 0, longest = 0;
  if (p.target_groups != p.round_groups) {
    // Is one round even enough?  (See ragged_round_is_even.)
    const PlanCap T(cap);
    for (int b = t; b < B; b += kPlanThreads) {
      const int len = sh.seq[b].x, ns = T.splits(len);
      n += ns;
      if (len > 0) longest = max(longest, (int)((uint32_t)(len - 1) / (uint32_t)ns + 1u));
    }
    n = wave_add(n);
    longest = wave_imax(longest);
    if (lane == 0) {
      sh.wave_sum[wave] = n;
      sh.longest[wave] = longest;
    }
    __syncthreads();
    n = 0;
    longest = 0;
#pragma unroll
    for (int w = 0; w < kPlanWaves; ++w) {
      n += sh.wave_sum[w];
      longest = max(longest, sh.longest[w]);
    }
    __syncthreads();
    one_round = ragged_round_is_even(n, longest, tokens, p.round_groups);
  }
  int total;
  if (one_round) {
    total = assign(cap);
  } else {
    // More splits, unless they cost more than they shorten: their number is
    // known once they are laid out, so that is done first.
    const int more = plan_cap(sh, B, p.target_groups, max_len);
    total = assign(more);
    if (!ragged_splits_pay(n, longest, total, more, p.round_groups, p.split_tokens)) total = assign(cap);
  }
  // The order of the entries.  Few sequences: each one's rank is counted, the
  // comparisons shared by all threads (B2 threads hold a sequence each, `shares`
  // of them per sequence; lanes of a wave hold one share, so c is uniform).
  // Many: a sorting network, whose steps cost a barrier each but whose
  // comparisons do not grow with the square of the batch.
  if (B <= kRankMax) {
    int B2 = 64;
    while (B2 < B) B2 <<= 1;
    const int shares = kPlanThreads / B2, share = t / B2;
    const int b = t % B2;
    if (b < B) {
      const int2 me = sh.seq[b];
      int r = 0;
#pragma unroll 4
      for (int c = share; c < B; c += shares) r += ahead(sh.seq[c], c, me, b) ? 1 : 0;
      atomicAdd(&sh.rank[b], r);
    }
    __syncthreads();
    for (int i = t; i < B; i += kPlanThreads) sh.order[sh.rank[i]] = i;
  } else {
    int n = 2 * kRankMax;
    while (n < B) n <<= 1;
    for (int i = t; i < n; i += kPlanThreads) sh.order[i] = i;
    for (int size = 2; size <= n; size <<= 1)
      for (int dist = size >> 1; dist > 0; dist >>= 1) {
        __syncthreads();
        for (int i = t; i < n / 2; i += kPlanThreads) {
          const int lo = 2 * i - (i & (dist - 1)), hi = lo + dist;
          const int x = sh.order[lo], y = sh.order[hi];
          // Indices from B on (no sequence) sort behind all others.
          const bool y_first = y < B && (x >= B || ahead(sh.seq[y], y, sh.seq[x], x));
          const bool x_first = x < B && !y_first;
          if ((lo & size) == 0 ? y_first : x_first) {
            sh.order[lo] = y;
            sh.order[hi] = x;
          }
        }
      }
  }
  __syncthreads();
  for (int i = t; i < B; i += kPlanThreads) {
    sh.start[i] = sh.seq[sh.order[i]].y;
    p.split_base[i] = sh.base[i];
    p.split_count[i] = sh.seq[i].y;
  }
  __syncthreads();
  // In place: a pass reads its values before its barriers and writes after.
  block_scan(B, sh.start, sh.wave_sum, [&](int r) { return sh.start[r]; });
  __syncthreads();
  int top = 1;  // the largest power of two below B
  while (2 * top < B) top <<= 1;
  for (int i = t; i < p.work_capacity; i += kPlanThreads) {
    int4 w = {-1, 0, 0, 0};
    if (i < total) {
      int r = 0;  // the last rank whose first entry is at or before i
      for (int step = top; step > 0; step >>= 1)
        if (r + step < B && sh.start[r + step] <= i) r += step;
      const int b = sh.order[r];
      w = int4{b, i - sh.start[r], sh.seq[b].y, sh.base[b]};
    }
    reinterpret_cast<int4*>(p.work)[i] = w;
  }
  if (t == 0 && p.total) *p.total = total;
}

}  // namespace

hipError_t launch_ragged_plan(const RaggedPlanParams& p, hipStream_t stream) {
  if (p.batch < 1 || p.batch > kRaggedPlanMaxBatch || p.target_groups < 1 || p.round_groups < 1) return hipErrorInvalidValue;
  if (p.work_capacity < max(p.batch, max(p.target_groups, p.round_groups))) return hipErrorInvalidValue;
  hipLaunchKernelGGL(ragged_plan_kernel, dim3(1), dim3(kPlanThreads), 0, stream, p);
  return hipGetLastError();
}

}  // namespace bt
