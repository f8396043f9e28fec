// Tiled GEMM on the bf16 matrix cores with operands split into three bf16
// parts (gemm_split_kernel.hpp), called by the GEMM entry points in gemm_f32.hip.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace aar {

// The epilogue (gemm_epi.hpp) and its operands.
struct GemmEpiArgs {
  int epi;
  const float* bias;
  const float* aux;
  uint32_t* bits;
  float* part;
};

// Tile configurations.  `resident`: workgroups a CU holds (LDS; it sets the
// launch bounds).  eff, round_us, occ: the cost model's rate on a CU with all
// its workgroups (fraction of 329 TFLOP/s, six bf16 products per fp32 one),
// time per workgroup beside its matrix ops, and the rate with one workgroup
// relative to a full CU.  Fitted to 3889 times (shape, layout, configuration,
// split) on MI355X over 49 shapes from 100^3 and 64 x 64 x 4096 to 4096^3 and
// 8192 x 8192 x 512, the GPT step's among them: the model's pick is 1.0 %
// slower than the best on average and 12 % at most (20000 x 200 x 100).  Its times
// are for comparing plans: products that the chip's power bounds take 15-25 %
// longer (4096^3 534 us by the model, 640-670 measured).
// Measured and not built: 256 x 128 and 128 x 256 as four waves of 128 x 64 / 64
// x 128 (one wave per SIMD: 4096^3 NN / NT / TN 650 / 642 / 675 us against
// 641 / 625 / 646 for eight waves of 64 x 64; the GPT step's shapes 4-15 %
// slower), and 256 x 256 (its two accumulator sets need the whole register
// file; with one, 4096^3 ran 584-630 us and the GPT step's products 2 %
// slower, with three times the rounding error).
struct SplitCfg {
  int bm, bn, bk, wm, wn, resident;
  float eff, round_us, occ;
  constexpr int waves() const { return (bm / wm) * (bn / wn); }
};
constexpr SplitCfg kSplitCfgs[] = {
    {256, 128, 32, 64, 64, 1, 0.798f, 3.57f, 1.f},    {128, 128, 16, 64, 64, 2, 0.656f, 2.55f, 0.875f},
    {128, 192, 32, 64, 96, 1, 0.668f, 4.21f, 1.f},    {128, 64, 32, 64, 32, 2, 0.607f, 2.06f, 0.736f},
    {64, 128, 32, 32, 64, 2, 0.585f, 1.34f, 0.71f},   {64, 64, 32, 32, 32, 3, 0.562f, 1.14f, 0.625f},
};
constexpr int kNumSplitCfgs = sizeof(kSplitCfgs) / sizeof(kSplitCfgs[0]);

struct SplitPlan {
  int cfg = -1;  // -1: no plan
  int splits = 1;
  int64_t k_per_split = 0;
  double us = 0;  // the model's time
};

// The plan of a product (`batch` of them) with `ws_bytes` of scratch for
// split-K partial products (splits * M * N floats).  chains: the number of
// separate sums over K that the fp32 plan adds up; this plan keeps at least
// half of them, so that its rounding error stays the smaller one (over the same
// K it is 0.33-0.44 of the fp32 instruction's, and errors grow with the square
// root of a chain's length).  limit: plans that take no less are of no use.
SplitPlan plan_split_gemm(int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t batch, size_t ws_bytes,
                          int chains, double limit);

// Launch the products of every split into C + split * split_stride.
// AAR_EUNSUPPORTED, launching nothing, where the configuration lacks the
// epilogue.
#define AAR_SPLIT_ARGS                                                                                            \
  const SplitPlan &p, const float *A, const float *B, float *C, int64_t M, int64_t N, int64_t K, int64_t lda,     \
      int64_t ldb, int64_t ldc, int64_t split_stride, int64_t batch, int64_t sA, int64_t sB, int64_t sC,          \
      const GemmEpiArgs &e, hipStream_t st
int launch_split_nn(AAR_SPLIT_ARGS);
int launch_split_nt(AAR_SPLIT_ARGS);
int launch_split_tn(AAR_SPLIT_ARGS);
#undef AAR_SPLIT_ARGS

}  // namespace aar
