// fp32 GEMM on the bf16 matrix cores (bf16x3.hpp: each operand in three bf16
// parts, six products), the three layouts of gemm_f32.hip:
//   NN  C[M,N] = A[M,K]   . B[K,N]
//   NT  C[M,N] = A[M,K]   . B[N,K]^T
//   TN  C[M,N] = A[K,M]^T . B[K,N]
//
// Bound by the matrix cores' power on large products: at 4096^3 the chip holds
// 1.8 GHz with the unit 65 % busy, 1.24 PFLOP/s of bf16 products, where a large
// plain bf16 product reaches 1.18 PFLOP/s at 4096^3 and 1.37 at 16384^3 on this
// card.  So the work around it is kept small:
//  * Each element is split once per workgroup, not once per wave: tiles go
//    HBM -> registers -> three bf16 planes in LDS, double buffered.  A thread
//    stages units of 8 consecutive k of one row, which is one lane's operand
//    of v_mfma_f32_32x32x16_bf16, so a fragment is one ds_read_b128 whichever
//    way the operand lies in HBM: a K-contiguous row gives a unit in two
//    128-bit loads, a row-contiguous operand in eight 32-bit loads that are
//    coalesced over the rows.  Loads need 4-byte alignment only, so ragged and
//    unaligned operands take the same path.
//  * Two accumulators per output: the hi hi products, and the five smaller ones.
//    The matrix unit truncates the sum of its 16 products and the accumulator
//    toward minus infinity, some bits below the accumulator's last; with the small
//    products in the same accumulator every output came out about 2e-8 of its
//    scale low at K = 384 (8e-8 at 1536), which column sums over many rows
//    collected (2.0e-6 instead of 3.6e-7 on the sums of 16384 rows), and the
//    rounding error was 2.7 times as large (2.9e-7 against 1.1e-7 at K = 384).
//    It costs registers only (and took 2 % off the times over 147 shapes: the
//    chains of dependent matrix ops are shorter).
//  * A K tile's matrix ops are cut into slots of WM/32 instructions; the
//    conversions of the next tile (13 VALU ops per pair of elements), its LDS
//    stores, the loads of the one after and the next fragments are spread over
//    the slots, with scheduling fences between, so that each slot's VALU work
//    runs under its matrix ops (left to itself the compiler bunched them: 128x192
//    tile 16384 x 384 x 1536 NT 115 -> 100 us).
//  * LDS planes are [part][octet of k][row] in 16-byte units, with the octets of
//    a K-contiguous operand 128 / (octets) bytes apart, so that eight lanes
//    storing (row, octet) neighbours hit distinct banks (the same tile: conflicts
//    were 30 % of its LDS cycles).
//  * A ragged K end is staged first, with predicates and zeros, so the main
//    loop has no branches; loads past the last tile repeat it.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "bf16x3.hpp"
#include "common.hpp"
#include "gemm_epi.hpp"
#include "gemm_split.hpp"

namespace aar {
namespace {

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// Stages a BR x BK tile of an operand (BR of its M or N rows).
//   KC: element (r, k) at P[r * ld + k]; else P[k * ld + r].
template <int BR, int BK, int NT, bool KC>
struct SplitTile {
  static constexpr int NO = BK / 8;        // octets of k
  static constexpr int kU = BR * NO / NT;  // units of 8 k per thread
  static_assert(BR * NO % NT == 0, "whole units per thread");
  static constexpr int kOs = BR + (KC ? 8 / NO : 0);  // octet stride in 16-byte units
  static constexpr int kUnits = 3 * NO * kOs;
  static constexpr int kPairs = kU * 4;

  float f[kU][8];
  float top = 0.f;  // largest magnitude of this thread's elements
  uint32_t off[kU];
  u32x4 parts[3];

  __device__ __forceinline__ static void coords(int u, int& row, int& oct) {
    if (KC) {
      row = u / NO;
      oct = u % NO;
    } else {
      row = u % BR;
      oct = u / BR;
    }
  }
  __device__ __forceinline__ static const char* origin(const float* P, int64_t ld, int64_t r0, int64_t k0) {
    return reinterpret_cast<const char*>(KC ? P + r0 * ld + k0 : P + k0 * ld + r0);
  }

  // Rows past the operand are clamped onto its last one; they feed only
  // outputs that are not stored.  The host guarantees BR * ld * 4 < 2^32.
  __device__ __forceinline__ void init(int64_t ld, int64_t r0, int64_t R, int tid) {
    const int lim = (int)min<int64_t>(R - r0 - 1, BR - 1);
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      int row, oct;
      coords(tid + i * NT, row, oct);
      const uint32_t r = (uint32_t)min(row, lim);
      off[i] = (KC ? r * (uint32_t)ld + 8u * oct : 8u * oct * (uint32_t)ld + r) * 4u;
    }
  }

  __device__ __forceinline__ void load_unit(const float* __restrict__ P, int64_t ld, int64_t r0, int64_t k0, int i) {
    const char* base = origin(P, ld, r0, k0);
    if constexpr (KC) {
      const f32x4 a = *reinterpret_cast<const f32x4u*>(base + off[i]);
      const f32x4 b = *reinterpret_cast<const f32x4u*>(base + off[i] + 16);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f[i][e] = a[e];
        f[i][4 + e] = b[e];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) f[i][e] = *reinterpret_cast<const float*>(base + (int64_t)e * ld * 4 + off[i]);
    }
  }
  __device__ __forceinline__ void load(const float* __restrict__ P, int64_t ld, int64_t r0, int64_t k0) {
#pragma unroll
    for (int i = 0; i < kU; ++i) load_unit(P, ld, r0, k0, i);
  }
  // A ragged tile: k >= kend is zero.
  __device__ __forceinline__ void load_tail(const float* __restrict__ P, int64_t ld, int64_t r0, int64_t k0,
                                            int64_t kend, int tid) {
    const char* base = origin(P, ld, r0, k0);
    const int klim = (int)(kend - k0);
#pragma unroll
    for (int i = 0; i < kU; ++i) {
      int row, oct;
      coords(tid + i * NT, row, oct);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        f[i][e] = 8 * oct + e < klim
                      ? *reinterpret_cast<const float*>(base + (KC ? (int64_t)e * 4 : (int64_t)e * ld * 4) + off[i])
                      : 0.f;
    }
  }

  // Splits pair q of this thread's elements; a unit's last pair stores it.  rem:
  // bf16_split_pair's.
  __device__ __forceinline__ void pair(u32x4* __restrict__ s, int tid, int q, uint32_t& rem) {
    const int i = q >> 2, e = q & 3;
    const float a = f[i][2 * e], b = f[i][2 * e + 1];
    top = fmaxf(fmaxf(top, fabsf(a)), fabsf(b));
    uint32_t w[3];
    bf16_split_pair(a, b, w, rem);
#pragma unroll
    for (int p = 0; p < 3; ++p) parts[p][e] = w[p];
    if (e == 3) {
      int row, oct;
      coords(tid + i * NT, row, oct);
#pragma unroll
      for (int p = 0; p < 3; ++p) s[(p * NO + oct) * kOs + row] = parts[p];
    }
  }
  __device__ __forceinline__ void store(u32x4* __restrict__ s, int tid, uint32_t& rem) {
#pragma unroll
    for (int q = 0; q < kPairs; ++q) pair(s, tid, q, rem);
  }
  __device__ __forceinline__ static u32x4 frag(const u32x4* __restrict__ s, int part, int oct, int row) {
    return s[(part * NO + oct) * kOs + row];
  }
};

// The wave's accumulators from the fp32 instruction, straight from HBM (rare, so
// no staging): the tiles that the split does not cover.  Step s of S multiplies
// k = s and k = S + s of 2 S (lane halves), so that a lane's 16 steps read half a
// line of a K-contiguous operand; without one, 16 steps' addresses spilled.
// Measured with an infinity in every row of A (the split product and this one):
// 4096^3 NN / NT / TN 2.0 / 1.7 / 1.9 ms beside 0.74 / 0.73 / 0.75 of finite
// operands (3.3 / 4.1 / 2.8 with one step's loads at a time and no half lines),
// 16384 x 1152 x 384 NT 234 beside 96 us.
template <int S, int T, bool KC>
__device__ __forceinline__ void fp32_operand(float (&v)[S][T], const float* __restrict__ P, int64_t R, int64_t ld,
                                             int64_t r0, int64_t k0, int64_t kend, int lr, int h) {
  // (a wave past the operand reads its last row; 32-bit, so that it is a scalar)
  const int first = min((int)r0, (int)R - 1);
  const bool whole = k0 + 2 * S <= kend;
#pragma unroll
  for (int i = 0; i < T; ++i) {
    const uint32_t r = (uint32_t)min((int)R - 1 - first, 32 * i + lr);
    // 32-bit lane offsets, as SplitTile's, from a scalar row base
    const uint32_t off = (KC ? r * (uint32_t)ld + (uint32_t)(S * h) : (uint32_t)(S * h) * (uint32_t)ld + r) * 4u;
    const char* base = reinterpret_cast<const char*>(KC ? P + (int64_t)first * ld + k0 : P + k0 * ld + first);
    if (KC && whole) {
#pragma unroll
      for (int g = 0; g < S / 4; ++g) {
        const f32x4 x = *reinterpret_cast<const f32x4u*>(base + off + 16 * g);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * g + e][i] = x[e];
      }
    } else {
      const int64_t step = KC ? 4 : ld * 4;
#pragma unroll
      for (int s = 0; s < S; ++s)
        v[s][i] = whole || k0 + S * h + s < kend ? *reinterpret_cast<const float*>(base + s * step + off) : 0.f;
    }
  }
}
template <int TM, int TN, bool A_KC, bool B_KC>
__device__ __forceinline__ void fp32_tile(f32x16 (&acc)[TM][TN], const float* __restrict__ A,
                                          const float* __restrict__ B, int64_t M, int64_t N, int64_t lda, int64_t ldb,
                                          int64_t r0, int64_t c0, int64_t kbeg, int64_t kend, int lr, int h) {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  constexpr int S = A_KC || B_KC ? 16 : 8;
#pragma unroll 1
  for (int64_t k0 = kbeg; k0 < kend; k0 += 2 * S) {
    float a[S][TM], b[S][TN];
    fp32_operand<S, TM, A_KC>(a, A, M, lda, r0, k0, kend, lr, h);
    fp32_operand<S, TN, B_KC>(b, B, N, ldb, c0, k0, kend, lr, h);
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s][i], b[s][j], acc[i][j], 0, 0, 0);
  }
#endif
}

// kEpiColsumA's sums for A column m: lane half h takes the chunk's k with
// k & 4 == 4h in order, one of aar_colsum_f32's two running sums; chunk q (64
// rows of A) belongs to the workgroups with tn == q % tiles_n.  Two chunks' loads
// are in flight together.  Ahead of the K loop, where nothing else holds registers:
// among the matrix ops the sums cost 12 % (384 x 1536 x 16384 132 us, now 119, the
// plain product 116; 4096^3 712 -> 658).
__device__ __forceinline__ void colsum_a(const float* __restrict__ A, int64_t M, int64_t lda, float* __restrict__ part,
                                         int64_t m, int h, int64_t kbeg, int64_t kend, int tn, int tiles_n) {
  const int64_t first = kbeg >> 6, last = kend >> 6;
  const float* col = A + min(m, M - 1) + 4 * h * lda;
#pragma unroll 1
  for (int64_t q = first + (tn + tiles_n - first % tiles_n) % tiles_n; q < last; q += 2 * tiles_n) {
    const int64_t q2 = q + tiles_n < last ? q + tiles_n : q;  // (the same chunk twice at the end)
    float v[2][32];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const float* p = col + (c ? q2 : q) * 64 * lda;
#pragma unroll
      for (int i = 0; i < 32; ++i) v[c][i] = p[(8 * (i / 4) + i % 4) * lda];
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < 32; ++i) s += v[c][i];
      s += __uint_as_float(partner_u32(__float_as_uint(s)));
      if (h == 0 && m < M) part[(c ? q2 : q) * M + m] = s;
    }
  }
}

// WPE: waves per SIMD the register allocation must allow.
template <int BM, int BN, int BK, int WM, int WN, int WPE, bool A_KC, bool B_KC, int EPI>
__global__ void __launch_bounds__((BM / WM) * (BN / WN) * 64, WPE)
gemm_split_kernel(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C, int64_t M,
                  int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int64_t k_per_split,
                  int64_t split_stride, int tiles_m, int tiles_n, int64_t sA, int64_t sB, int64_t sC, GemmEpi ep) {
  constexpr int NWM = BM / WM;
  constexpr int NW = NWM * (BN / WN);
  constexpr int NT = NW * 64;
  constexpr int TM = WM / 32;
  constexpr int TN = WN / 32;
  constexpr int KS = BK / 16;  // matrix-op steps per K tile
  using TA = SplitTile<BM, BK, NT, A_KC>;
  using TB = SplitTile<BN, BK, NT, B_KC>;
  constexpr int kStage = TA::kUnits + TB::kUnits;
  static_assert(EPI != kEpiColsumA || BM <= 32 * NW, "a wave sums 32 columns of A");
  __shared__ u32x4 lds[2 * kStage];
  __shared__ int unplain, lossy;  // set by any thread: look closer; an element was split inexactly
  __shared__ uint32_t top[2];     // largest magnitude of A's and of B's elements, as bits

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 31;
  const int h = lane >> 5;
  const int wm0 = (wave % NWM) * WM;
  const int wn0 = (wave / NWM) * WN;

  int tm, tn;
  map_tile(tiles_m, tiles_n, tm, tn);
  const int64_t m0 = (int64_t)tm * BM;
  const int64_t n0 = (int64_t)tn * BN;
  const int64_t kbeg = (int64_t)blockIdx.y * k_per_split;
  const int64_t kend = min(K, kbeg + k_per_split);
  C += (int64_t)blockIdx.y * split_stride;
  A += (int64_t)blockIdx.z * sA;
  B += (int64_t)blockIdx.z * sB;
  C += (int64_t)blockIdx.z * sC;
  if (tid == 0) unplain = lossy = top[0] = top[1] = 0;

  f32x16 acc[TM][TN], low[TM][TN];  // the hi hi products, and the five smaller ones
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = low[i][j][r] = 0.f;

  TA ta;
  TB tb;
  uint32_t rem = 0;  // what the splits left over, of both operands
  ta.init(lda, m0, M, tid);
  tb.init(ldb, n0, N, tid);
  float bias[TN];
  load_bias<TN, EPI>(ep, N, n0 + wn0, lr, bias);
  uint32_t words[TM][TN];
  load_bits<TM, TN, EPI>(ep, M, N, m0 + wm0, n0 + wn0, lr, words);

  // K tiles: the ragged one (if any) first, then the whole ones in order
  const int nt = (int)ceil_div(kend - kbeg, (int64_t)BK);
  const bool ragged = (kend - kbeg) % BK != 0;
  const int whole = ragged ? nt - 1 : nt;
  const int64_t klast = kbeg + (int64_t)max(whole - 1, 0) * BK;  // start of the last whole tile
  int64_t kf = kbeg;                                             // start of the next whole tile to load
  if (ragged) {
    ta.load_tail(A, lda, m0, kbeg + (int64_t)whole * BK, kend, tid);
    tb.load_tail(B, ldb, n0, kbeg + (int64_t)whole * BK, kend, tid);
  } else {
    ta.load(A, lda, m0, kf);
    tb.load(B, ldb, n0, kf);
    kf = min(kf + BK, klast);
  }
  // While the first tile is on its way: the column sums of A (K and the splits
  // are multiples of 64, so every chunk is whole).
  if constexpr (EPI == kEpiColsumA) {
    if (wave < BM / 32) colsum_a(A, M, lda, ep.part, m0 + 32 * wave + lr, h, kbeg, kend, tn, tiles_n);
  }
  ta.store(lds, tid, rem);
  tb.store(lds + TA::kUnits, tid, rem);
  if (nt > 1) {
    ta.load(A, lda, m0, kf);
    tb.load(B, ldb, n0, kf);
    kf = min(kf + BK, klast);
  }
  lds_barrier();

  auto tile = [&](int t, auto more_tag) {
    constexpr bool kMore = decltype(more_tag)::value;  // another tile follows
    const u32x4* as = lds + (t & 1) * kStage;
    const u32x4* bs = as + TA::kUnits;
    u32x4* next = lds + ((t + 1) & 1) * kStage;
    // slots of TM matrix ops; the next tile's pairs start at slot kFirst, after
    // the fragments the first slots wait for
    constexpr int kSlots = KS * TN * kSplitProducts;
    constexpr int kFirst = 2;
    constexpr int kPairs = TA::kPairs + TB::kPairs;
    u32x4 af[2][TM][3], bf[2][3];
    auto read_a = [&](int ks, int p) {
#pragma unroll
      for (int i = 0; i < TM; ++i) af[ks & 1][i][p] = TA::frag(as, p, 2 * ks + h, wm0 + 32 * i + lr);
    };
    auto read_b = [&](int q, int p) {
      bf[q & 1][p] = TB::frag(bs, p, 2 * (q / TN) + h, wn0 + 32 * (q % TN) + lr);
    };
    read_b(0, 0);
    read_a(0, 2);
    read_a(0, 0);
    read_b(0, 2);
    read_a(0, 1);
    read_b(0, 1);
    sched_fence();
#pragma unroll
    for (int q = 0; q < KS * TN; ++q) {
      const int ks = q / TN, j = q % TN;
#pragma unroll
      for (int pr = 0; pr < kSplitProducts; ++pr) {
        const int s = q * kSplitProducts + pr;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          f32x16& c = pr + 1 == kSplitProducts ? acc[i][j] : low[i][j];
          c = mfma_bf16(af[ks & 1][i][kSplitA[pr]], bf[q & 1][kSplitB[pr]], c);
        }
        if (q + 1 < KS * TN) {
          if (pr == 2) read_b(q + 1, 0);
          if (pr == 3) read_b(q + 1, 2);
          if (pr == 4) read_b(q + 1, 1);
          if (j == TN - 1) {
            if (pr == 1) read_a(ks + 1, 2);
            if (pr == 2) read_a(ks + 1, 0);
            if (pr == 3) read_a(ks + 1, 1);
          }
        }
        if constexpr (kMore) {
#pragma unroll
          for (int p = 0; p < kPairs; ++p) {
            if (kFirst + p * (kSlots - kFirst) / kPairs == s) {
              if (p < TA::kPairs) {
                ta.pair(next, tid, p, rem);
                if ((p & 3) == 3) ta.load_unit(A, lda, m0, kf, p >> 2);
              } else {
                tb.pair(next + TA::kUnits, tid, p - TA::kPairs, rem);
                if ((p & 3) == 3) tb.load_unit(B, ldb, n0, kf, (p - TA::kPairs) >> 2);
              }
            }
          }
        }
        sched_fence();
      }
    }
    if constexpr (kMore) kf = min(kf + BK, klast);
  };
  for (int t = 0; t < nt - 1; ++t) {
    tile(t, std::true_type{});
    lds_barrier();
  }
  tile(nt - 1, std::false_type{});

#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] += low[i][j];

  // Operands that the split might not cover, seen by any thread: where the sums
  // might overflow, or a wave's smallest output feels a remainder left over, the
  // wave's tile is done again in fp32.
  const bool loss = (rem & kSplitRemBits) != 0;
  if (loss || !(ta.top <= kSplitPlain && tb.top <= kSplitPlain)) unplain = 1;
  if (loss) lossy = 1;
  lds_barrier();
  if (unplain) {
    atomicMax(&top[0], __float_as_uint(ta.top));  // >= 0: ordered as their bits
    atomicMax(&top[1], __float_as_uint(tb.top));
    __syncthreads();
    const float ma = __uint_as_float(top[0]), mb = __uint_as_float(top[1]), n = (float)(kend - kbeg);
    bool redo = split_overflows(ma, mb, n);
    if (!redo && lossy) {
      float least = INFINITY;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) least = fminf(least, fabsf(acc[i][j][r]));
      redo = __any(least < split_loss_floor(ma, mb, n));
    }
    if (redo) fp32_tile<TM, TN, A_KC, B_KC>(acc, A, B, M, N, lda, ldb, m0 + wm0, n0 + wn0, kbeg, kend, lr, h);
  }

  if constexpr (epi_bits(EPI)) {
    store_tile_bits<TM, TN, EPI>(acc, C, ep, bias, words, M, N, ldc, m0 + wm0, n0 + wn0, lr, h);
  } else {
    store_tile<TM, TN, EPI, 4, true>(acc, C, ep, bias, M, N, ldc, m0 + wm0, n0 + wn0, lr, h);
  }
}

template <int I, bool A_KC, bool B_KC>
int launch_split_cfg(const SplitPlan& p, const float* A, const float* B, float* C, int64_t M, int64_t N, int64_t K,
                 int64_t lda, int64_t ldb, int64_t ldc, int64_t split_stride, int64_t batch, int64_t sA, int64_t sB,
                 int64_t sC, int epi, const GemmEpi& ep, hipStream_t st) {
  constexpr SplitCfg c = kSplitCfgs[I];
  constexpr int kWaves = c.waves();
  constexpr int kWpe = (c.resident * kWaves + 3) / 4;
  const int64_t tiles_m = ceil_div(M, (int64_t)c.bm), tiles_n = ceil_div(N, (int64_t)c.bn);
  // a dispatch holds each grid extent as a 32-bit work-item count
  if (tiles_m * tiles_n * kWaves * 64 > (int64_t)UINT32_MAX) return AAR_EUNSUPPORTED;
  const dim3 grid((unsigned)(tiles_m * tiles_n), (unsigned)p.splits, (unsigned)batch);
  auto go = [&](auto epi_tag) {
    constexpr int E = decltype(epi_tag)::value;
    if constexpr (E == kEpiMaskBits && c.wm != 64) {  // a wave owns one 64-row column-sum chunk
      return AAR_EUNSUPPORTED;
    } else {
      gemm_split_kernel<c.bm, c.bn, c.bk, c.wm, c.wn, kWpe, A_KC, B_KC, E><<<grid, dim3(kWaves * 64), 0, st>>>(
          A, B, C, M, N, K, lda, ldb, ldc, p.k_per_split, split_stride, (int)tiles_m, (int)tiles_n, sA, sB, sC, ep);
      return launch_status();
    }
  };
  switch (epi) {
    case kEpiNone: return go(std::integral_constant<int, kEpiNone>{});
    case kEpiBias: return go(std::integral_constant<int, kEpiBias>{});
    case kEpiBiasRelu:
      if constexpr (A_KC && B_KC) return go(std::integral_constant<int, kEpiBiasRelu>{});
      return AAR_EUNSUPPORTED;
    case kEpiAdd:
      if constexpr (A_KC && B_KC) return go(std::integral_constant<int, kEpiAdd>{});
      return AAR_EUNSUPPORTED;
    case kEpiBiasAdd:
      if constexpr (A_KC && B_KC) return go(std::integral_constant<int, kEpiBiasAdd>{});
      return AAR_EUNSUPPORTED;
    case kEpiBiasReluBits:
      if constexpr (A_KC && B_KC) return go(std::integral_constant<int, kEpiBiasReluBits>{});
      return AAR_EUNSUPPORTED;
    case kEpiMask:
      if constexpr (A_KC && !B_KC) return go(std::integral_constant<int, kEpiMask>{});
      return AAR_EUNSUPPORTED;
    case kEpiMaskBits:
      if constexpr (A_KC && !B_KC) return go(std::integral_constant<int, kEpiMaskBits>{});
      return AAR_EUNSUPPORTED;
    case kEpiColsumA:
      if constexpr (!A_KC && !B_KC) return go(std::integral_constant<int, kEpiColsumA>{});
      return AAR_EUNSUPPORTED;
    default: return AAR_EINVAL;
  }
}

template <bool A_KC, bool B_KC, int... I>
int launch_split_any(std::integer_sequence<int, I...>, const SplitPlan& p, const float* A, const float* B, float* C,
                     int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc, int64_t split_stride,
                     int64_t batch, int64_t sA, int64_t sB, int64_t sC, int epi, const GemmEpi& ep, hipStream_t st) {
  int rc = AAR_EINVAL;
  (void)((p.cfg == I && ((rc = launch_split_cfg<I, A_KC, B_KC>(p, A, B, C, M, N, K, lda, ldb, ldc, split_stride, batch,
                                                               sA, sB, sC, epi, ep, st)),
                         true)) ||
         ...);
  return rc;
}

// Every configuration of one layout (each layout is a source file of its own,
// so that they compile side by side).
template <bool A_KC, bool B_KC>
int launch_split_layout(const SplitPlan& p, const float* A, const float* B, float* C, int64_t M, int64_t N, int64_t K,
                        int64_t lda, int64_t ldb, int64_t ldc, int64_t split_stride, int64_t batch, int64_t sA,
                        int64_t sB, int64_t sC, const GemmEpiArgs& e, hipStream_t st) {
  GemmEpi ep{e.bias, e.aux};
  ep.bits = e.bits;
  ep.part = e.part;
  return launch_split_any<A_KC, B_KC>(std::make_integer_sequence<int, kNumSplitCfgs>{}, p, A, B, C, M, N, K, lda, ldb,
                                      ldc, split_stride, batch, sA, sB, sC, e.epi, ep, st);
}

}  // namespace
}  // namespace aar
