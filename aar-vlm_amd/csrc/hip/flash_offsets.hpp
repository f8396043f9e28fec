// The 32-bit byte offsets of a [32][up to 128] operand tile, relative to its
// first row.  Plain C++, so that the arithmetic can be run on the host.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define AAR_HD __host__ __device__ __forceinline__
#else
#define AAR_HD inline
#endif

namespace aar {

// Whether every element of a tile with row stride st (in elements) lies at a
// byte offset that an unsigned 32-bit number holds: 31 rows of 2^25 - 1 floats
// do.  Offsets of a negative stride lie below the first row and would wrap.
AAR_HD constexpr bool tile_offsets_fit(int64_t st) { return st >= 0 && st < (int64_t(1) << 25); }

// Byte offset of element (row, col); meaningful where tile_offsets_fit(st).
AAR_HD constexpr uint32_t tile_offset(int row, int64_t st, int col) { return (uint32_t)(row * st + col) * 4u; }

}  // namespace aar

#undef AAR_HD
