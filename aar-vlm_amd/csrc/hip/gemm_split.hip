// The plan of the split-operand products (gemm_split_kernel.hpp).
#include "gemm_split.hpp"

#include <algorithm>

#include "common.hpp"

namespace aar {

// Cost model: workgroups spread evenly over the CUs, n on the fullest one;
// each takes its matrix ops at the configuration's rate plus a fixed time (its
// first loads, its stores); split-K adds the partial products' traffic and the
// reduction launch.  A configuration whose matrix ops alone take no less
// than `limit` or the best plan so far is passed over (a plan costs 0.1 us where
// none is of use, 0.2-0.5 else, on the host).
SplitPlan plan_split_gemm(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t batch, size_t ws_bytes,
                          int chains, double limit) {
  SplitPlan best;
  constexpr int64_t kMaxSplitLd = (int64_t(1) << 32) / (4 * 256) - 1;  // 32-bit offsets: 256 rows * ld * 4 < 2^32
  if (lda > kMaxSplitLd || ldb > kMaxSplitLd) return best;
  constexpr int kSplits[] = {1, 2, 3, 4, 6, 8, 10, 12, 14, 16, 20, 24, 28, 32};
  constexpr int kNum = sizeof(kSplits) / sizeof(kSplits[0]);
  const int cus = device_cu_count();
  const double cu_rate = 329e6 / 256;  // FLOP per us and CU
  for (int c = 0; c < kNumSplitCfgs; ++c) {
    const SplitCfg& cf = kSplitCfgs[c];
    const int64_t tiles = ceil_div(M, (int64_t)cf.bm) * ceil_div(N, (int64_t)cf.bn) * batch;
    const double ops = 2.0 * cf.bm * cf.bn / (cf.eff * cu_rate);  // us per k of a workgroup on a full CU
    const double spread = ops * (double)tiles * (double)K / cus;  // over all CUs
    const double one = std::min(ops * (double)K, 3.0 + ops * 128.0);  // a workgroup's: K whole, or a split's chunk
    if (3.3 + cf.round_us + std::max(spread, one) >= limit) continue;
    const int64_t fill = std::min<int64_t>((int64_t)cus * cf.resident / std::max<int64_t>(tiles, 1), 64);
    for (int i = 0; i <= kNum; ++i) {
      const int splits = i < kNum ? kSplits[i] : (int)fill;
      if (splits < 1) break;
      if (splits > 1 && (batch > 1 || K < 128 * (int64_t)splits)) {
        i = std::max(i, kNum - 1);  // the longer lists' chunks are shorter still; `fill` may be less
        continue;
      }
      // chunks of a multiple of 64 k: whole chunks of the column sums of A
      const int64_t kps = splits > 1 ? ceil_div(ceil_div(K, (int64_t)splits), (int64_t)64) * 64 : K;
      const int64_t real = ceil_div(K, kps);
      if (real * 2 < (int64_t)chains) continue;
      if (real > 1 && (size_t)real * M * N * sizeof(float) > ws_bytes) continue;
      const int64_t n = ceil_div(tiles * real, (int64_t)cus);
      const double occ = n >= cf.resident ? 1.0 : cf.occ + (1.0 - cf.occ) * (double)(n - 1) / (cf.resident - 1);
      const double steps = (double)ceil_div(kps, (int64_t)cf.bk) * cf.bk;
      double us = 3.3 + (double)n * (ops * steps / occ + cf.round_us);
      if (real > 1) us += 3.0 + (double)(real + 1) * M * N * 4.0 / 4e6;
      if (us < limit) {
        limit = us;
        best = SplitPlan{c, (int)real, kps, us};
      }
    }
  }
  return best;
}

}  // namespace aar
