// The NN products of gemm_split_kernel.hpp.
#include "gemm_split_kernel.hpp"

namespace aar {

int launch_split_nn(const SplitPlan& p, const float* A, const float* B, float* C, int64_t M, int64_t N, int64_t K,
                    int64_t lda, int64_t ldb, int64_t ldc, int64_t split_stride, int64_t batch, int64_t sA, int64_t sB,
                    int64_t sC, const GemmEpiArgs& e, hipStream_t st) {
  return launch_split_layout<true, false>(p, A, B, C, M, N, K, lda, ldb, ldc, split_stride, batch, sA, sB, sC, e, st);
}

}  // namespace aar
