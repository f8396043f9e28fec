// Shared parts of the tiled GEMM kernels (gemm_f32.hip and gemm_split.hip): the
// workgroup -> tile mapping and the epilogues that store a wave's 32x32
// accumulator blocks.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"

namespace aar {
namespace {

constexpr int kGroupM = 4;

__device__ __forceinline__ void map_tile(int tiles_m, int tiles_n, int& tm, int& tn) {
  int w = blockIdx.x;
  const int nb = gridDim.x;
  if ((nb & 7) == 0) w = (w & 7) * (nb >> 3) + (w >> 3);  // XCD-contiguous ranges
  const int group_size = kGroupM * tiles_n;
  const int group = w / group_size;
  const int first_m = group * kGroupM;
  const int rows = min(tiles_m - first_m, kGroupM);
  const int in_group = w - group * group_size;
  tm = first_m + in_group % rows;
  tn = in_group / rows;
}

// Epilogues (a template argument, because every one but the plain store
// needs the accumulators in VGPRs: the kernels without one store straight
// from the accumulators and keep their occupancy).  Each is the same fp32
// operation as the separate op applied to the stored product:
//   kEpiBias      C = acc + bias[col]            (linear layer: add_bias)
//   kEpiBiasRelu  C = max(0, acc + bias[col])    (linear layer, then relu)
//   kEpiMask      C = aux[row][col] > 0 ? acc : 0  (relu backward, aux = the
//                 relu's output, which is positive exactly where its input is;
//                 aux has C's layout)
//   kEpiAdd       C = acc + aux[row][col]          (a residual add after the
//                 product: x + y W^T)
//   kEpiBiasAdd   C = (acc + bias[col]) + aux[row][col]  (the same after a
//                 linear layer with a bias)
// and two that carry a relu's mask as bits from the forward product to the
// backward one (store_tile_bits), so the backward reads 1 bit per element
// where kEpiMask reads the relu's whole output:
//   kEpiBiasReluBits  C = max(0, acc + bias[col]) as kEpiBiasRelu, and bit
//                     row % 32 of word bits[(row / 32) * N + col] set where
//                     C > 0: a word holds one column of a 32-row block, the
//                     rows of one accumulator block
//   kEpiMaskBits      C = bit(row, col) ? acc : 0 (the relu backward), and
//                     part[row / 64][col] = the sum of C over the 64 rows of
//                     that chunk, in aar_colsum_f32's stage-1 order (two
//                     running sums, see colsum_stage1_kernel): its partials
//                     (a wave owns one chunk)
enum : int {
  kEpiNone = 0,
  kEpiBias = 1,
  kEpiBiasRelu = 2,
  kEpiMask = 3,
  kEpiAdd = 4,
  kEpiBiasAdd = 5,
  kEpiBiasReluBits = 6,
  kEpiMaskBits = 7,
  kEpiColsumA = 8
};
// kEpiColsumA is not an epilogue (TN only): C is stored plainly, and the kernel
// also sums A's columns: part[k / 64][m] = the sum of A[k][m] over the 64-row
// chunk of k, in aar_colsum_f32's stage-1 order.  A lane holds the k's with
// k & 4 == 4h of its column in order, i.e. one of that order's two running sums;
// the halves add them at the chunk's end.  Chunk q is summed by the workgroups
// with tn == q % tiles_n, so the work spreads over the grid.  The fp32 tiles do it
// in the main loop (the first column of waves, from the staged tile), the
// split-operand ones ahead of it.
struct GemmEpi {
  const float* bias;
  const float* aux;
  uint32_t* bits = nullptr;  // [ceil(M / 32)][N]: kEpiBiasReluBits writes, kEpiMaskBits reads
  float* part = nullptr;     // kEpiMaskBits: [M / 64][N] column partials; kEpiColsumA: [K / 64][M]
};
constexpr bool epi_bits(int epi) { return epi == kEpiBiasReluBits || epi == kEpiMaskBits; }
constexpr bool epi_dma_only(int epi) { return epi_bits(epi) || epi == kEpiColsumA; }

// Epilogue: a wave's (32*TM) x (32*TN) accumulators to C.  Accumulator
// layout of a 32x32 block: lane (lr, h), register r holds row
// 8*(r/4) + 4*h + (r%4), column lr.
// A wave tile wholly inside C (the common case) stores without bounds tests;
// element offsets from the lane's first element are a constant row count
// times ldc, which the compiler forms once in scalar registers.
// NQ < 4: only register quads q0 .. q0 + NQ - 1 of each accumulator are
// stored, their values held in quads 0 .. NQ - 1 of acc (a K group's share).
constexpr bool epi_has_bias(int epi) {
  return epi == kEpiBias || epi == kEpiBiasRelu || epi == kEpiBiasAdd || epi == kEpiBiasReluBits;
}

// The bias values a lane's accumulator columns need (column c0 + 32 j + lr),
// read before the main loop so their latency is hidden under it: read at
// the epilogue, they cost a memory round trip per workgroup round (measured
// +10 us on a 16384 x 1536 x 384 product with the bias epilogue).
template <int TN, int EPI>
__device__ __forceinline__ void load_bias(const GemmEpi& ep, int64_t N, int64_t c0, int lr, float (&bias)[TN]) {
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int64_t col = c0 + 32 * j + lr;
    bias[j] = 0.f;
    if constexpr (epi_has_bias(EPI)) bias[j] = col < N ? ep.bias[col] : 0.f;
  }
}

// Mask words the kEpiMaskBits epilogue needs, read before the main loop like
// the bias: lane (lr, h) holds, for block (i, j), the word of column
// c0 + 32 j + lr over rows r0 + 32 i .. + 31 (both halves read the same word,
// 128 contiguous bytes per half-wave).
template <int TM, int TN, int EPI>
__device__ __forceinline__ void load_bits(const GemmEpi& ep, int64_t M, int64_t N, int64_t r0, int64_t c0, int lr,
                                          uint32_t (&words)[TM][TN]) {
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      words[i][j] = 0u;
      if constexpr (EPI == kEpiMaskBits) {
        const int64_t col = c0 + 32 * j + lr;
        if (r0 + 32 * i < M && col < N) words[i][j] = ep.bits[((r0 + 32 * i) >> 5) * N + col];
      }
    }
}

// The two mask-bit epilogues (see kEpiBiasReluBits / kEpiMaskBits).  Wave
// tiles start at multiples of 32 rows, so accumulator block (i, j) covers
// whole mask words: lane (lr, h) holds the bits 8 (r / 4) + 4 h + r % 4 of the
// word of its column c0 + 32 j + lr, its half's 16 rows.
//   kEpiBiasReluBits: each lane sets its 16 bits, the two halves OR their
//   words (v_permlane32_swap) and half 0 stores the word.
//   kEpiMaskBits (WM = 64: the wave's rows are one 64-row chunk): each lane
//   tests its 16 bits of the prefetched word and sums its 32 rows of the
//   chunk in order, the row set (row & 4 == 4h) of one of colsum's two
//   running sums; half 0 adds its partner's (v_permlane32_swap) and stores
//   the chunk partial s0 + s1.
// The swap hands each lane its own value and its partner's, one in each
// result; where the two are equal either is the partner's.
__device__ __forceinline__ uint32_t partner_u32(uint32_t u) {
#if defined(__HIP_DEVICE_COMPILE__)
  const auto sw = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return sw[0] == u ? sw[1] : sw[0];
#else
  return u;
#endif
}

template <int TM, int TN, int EPI>
__device__ __forceinline__ void store_tile_bits(const f32x16 (&acc)[TM][TN], float* __restrict__ C,
                                                const GemmEpi& ep, const float (&bias)[TN],
                                                const uint32_t (&words)[TM][TN], int64_t M, int64_t N, int64_t ldc,
                                                int64_t r0, int64_t c0, int lr, int h) {
  static_assert(epi_bits(EPI), "mask-bit epilogues only");
  static_assert(EPI != kEpiMaskBits || TM == 2, "a kEpiMaskBits wave owns one 64-row chunk");
  // addressing as store_tile: a lane base and row offsets dr * ldc that the
  // compiler forms in scalar registers, bounds tests only off the interior
  const bool interior = r0 + 32 * TM <= M && c0 + 32 * TN <= N;
  float* const Cl = C + (r0 + 4 * h) * ldc + c0 + lr;
  wait_vm_lgkm0<0>();  // bias / mask words (see store_tile)
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int64_t col = c0 + 32 * j + lr;
    float vals[TM][16];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      uint32_t w = 0u;                           // this half's bits, at 8 (r / 4) + r % 4
      const uint32_t mine = words[i][j] >> (4 * h);  // kEpiMaskBits: the same positions
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int dr = 32 * i + 8 * (r >> 2) + (r & 3);  // row - r0 - 4h
        const int bit = 8 * (r >> 2) + (r & 3);
        const bool ok = interior || (r0 + 4 * h + dr < M && col < N);
        float v;
        // (the bit tests stay free of the bounds test: with it, the compiler
        // kept every element's lane mask live and spilled them to VGPR lanes)
        if constexpr (EPI == kEpiBiasReluBits) {
          v = fmaxf(0.0f, acc[i][j][r] + bias[j]);
          w |= v > 0.0f ? (1u << bit) : 0u;
        } else {
          // all ones where the bit is set: acc, else +0.0f
#if defined(__HIP_DEVICE_COMPILE__)
          const uint32_t keep = (uint32_t)__builtin_amdgcn_sbfe((int)mine, bit, 1);
#else
          const uint32_t keep = ((mine >> bit) & 1u) ? ~0u : 0u;
#endif
          v = __uint_as_float(__float_as_uint(acc[i][j][r]) & keep);
          vals[i][r] = v;
        }
        if (ok) Cl[(int64_t)dr * ldc + 32 * j] = v;
      }
      if constexpr (EPI == kEpiBiasReluBits) {
        w <<= 4 * h;
        w |= partner_u32(w);
        const int64_t rows = M - (r0 + 32 * i);  // rows of this word inside C
        if (rows < 32) w &= (1u << (rows > 0 ? rows : 0)) - 1u;
        if (h == 0 && rows > 0 && col < N) ep.bits[((r0 + 32 * i) >> 5) * N + col] = w;
      }
    }
    if constexpr (EPI == kEpiMaskBits) {
      if (!ep.part) continue;  // the mask only
      // colsum's chunk partial: half h's running sum over its rows (row & 4
      // == 4h) in row order, i.e. its registers in order, then s0 + s1
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) s += vals[i][r];
      s += __uint_as_float(partner_u32(__float_as_uint(s)));
      if (h == 0 && col < N && r0 < M) ep.part[(r0 >> 6) * N + col] = s;
    }
  }
}

template <int TM, int TN, int EPI, int NQ = 4, bool BATCH = false>
__device__ __forceinline__ void store_tile(const f32x16 (&acc)[TM][TN], float* __restrict__ C, const GemmEpi& ep,
                                           const float (&bias)[TN], int64_t M, int64_t N, int64_t ldc, int64_t r0,
                                           int64_t c0, int lr, int h, int q0 = 0) {
  const bool interior = r0 + 32 * TM <= M && c0 + 32 * TN <= N;
  const int64_t lane0 = (r0 + 4 * h) * ldc + c0 + lr;  // offset of the lane's first element
  float* const Cl = C + lane0;
  constexpr bool kAux = EPI == kEpiMask || EPI == kEpiAdd || EPI == kEpiBiasAdd;
  // The loaded operands (bias, aux) are waited for once, explicitly, before
  // the stores.  Left to the compiler, the per-element bounds branches made
  // it wait for vmcnt(0) before every store that uses one (stores count in
  // vmcnt), one memory round trip per element: measured +10 us on a
  // 16384 x 1536 x 384 product with the bias epilogue.
  if constexpr (epi_has_bias(EPI)) wait_vm_lgkm0<0>();
  const float* const Xl = kAux ? ep.aux + lane0 : nullptr;
  // The aux values are loaded before any store they feed: C and aux may
  // alias (an in-place residual), so a load placed after a store would wait
  // for it, one memory round trip per element.  (Each element is read and
  // then written by the same lane, so an aliased aux still reads the old
  // values.)  BATCH (the DMA kernels, whose staging registers are free by
  // the epilogue): when the wave tile's aux values fit in 96 registers (the
  // accumulators' count for a 64 x 96 wave tile), all rows of blocks are
  // loaded in one batch and waited for once, one memory round trip per wave
  // instead of one per row of blocks.  Otherwise a row of blocks at a time
  // (in the register path the batch cost occupancy).
  constexpr int kRowsPerBatch = BATCH && kAux && TM * TN * 4 * NQ <= 96 ? TM : 1;
  auto load_aux = [&](int i, float (&xv)[TN][4 * NQ]) {
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int64_t col = c0 + 32 * j + lr;
#pragma unroll
      for (int r = 0; r < 4 * NQ; ++r) {
        const int dr = 32 * i + 8 * (q0 + r / 4) + (r % 4);
        const int64_t off = (int64_t)dr * ldc + 32 * j;
        xv[j][r] = (interior || (r0 + 4 * h + dr < M && col < N)) ? Xl[off] : 0.0f;
      }
    }
  };
#pragma unroll
  for (int i0 = 0; i0 < TM; i0 += kRowsPerBatch) {
    float xv[kRowsPerBatch][TN][4 * NQ];
    if constexpr (kAux) {
#pragma unroll
      for (int ib = 0; ib < kRowsPerBatch; ++ib) load_aux(i0 + ib, xv[ib]);
      wait_vm_lgkm0<0>();
    }
#pragma unroll
    for (int ib = 0; ib < kRowsPerBatch; ++ib) {
      const int i = i0 + ib;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int64_t col = c0 + 32 * j + lr;
        const float b = bias[j];
#pragma unroll
        for (int r = 0; r < 4 * NQ; ++r) {
          const int dr = 32 * i + 8 * (q0 + r / 4) + (r % 4);  // row - r0 - 4h
          const int64_t off = (int64_t)dr * ldc + 32 * j;
          if (interior || (r0 + 4 * h + dr < M && col < N)) {
            float v = acc[i][j][r];
            if constexpr (EPI == kEpiBias) v = v + b;
            if constexpr (EPI == kEpiBiasRelu) v = fmaxf(0.0f, v + b);
            if constexpr (EPI == kEpiMask) v = xv[ib][j][r] > 0.0f ? v : 0.0f;
            if constexpr (EPI == kEpiAdd) v = v + xv[ib][j][r];
            if constexpr (EPI == kEpiBiasAdd) v = (v + b) + xv[ib][j][r];
            Cl[off] = v;
          }
        }
      }
    }
  }
}

}  // namespace
}  // namespace aar
