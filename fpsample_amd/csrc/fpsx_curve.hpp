// fpsx_curve.hpp -- the 3-D Hilbert index of the spatial ordering, usable on
// the device (fpsx_spatial.hip) and on the host (the CPU test that checks it).
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#define FPSX_HD __host__ __device__ __forceinline__
#else
#define FPSX_HD inline
#endif

namespace fpsx {

// Bits 0..9 of v at every third place.
FPSX_HD uint32_t spread3(uint32_t v) {
  v = (v | (v << 16)) & 0x030000ffu;
  v = (v | (v << 8)) & 0x0300f00fu;
  v = (v | (v << 4)) & 0x030c30c3u;
  return (v | (v << 2)) & 0x09249249u;
}

// Hilbert index of (x, y, z), BITS bits each (at most 10), by Skilling's transform
// ("Programming the Hilbert curve", AIP Conf. Proc. 707, 2004): undo the excess work axis by
// axis, Gray-encode, then interleave the bits with x the most significant of every triple.
// A bijection of the 2^(3 BITS) grid on [0, 2^(3 BITS)) in which consecutive indices are unit
// steps; the index of the leading bits is the leading part of the index.  Written without
// branches (a lane's bits are a mask): the ordering spends its time here.
template <int BITS>
FPSX_HD uint32_t hilbert(uint32_t x, uint32_t y, uint32_t z) {
  const uint32_t all = (1u << BITS) - 1u;
  uint32_t X[3] = {x & all, y & all, z & all};
#if defined(__HIPCC__)
#pragma unroll
#endif
  for (int b = BITS - 1; b > 0; --b) {
    const uint32_t P = (1u << b) - 1u;
    for (int i = 0; i < 3; ++i) {
      const uint32_t set = 0u - ((X[i] >> b) & 1u);  // all ones where the bit is set
      const uint32_t t = (X[0] ^ X[i]) & P & ~set;
      X[0] ^= t | (P & set);
      X[i] ^= t;
    }
  }
  X[1] ^= X[0];
  X[2] ^= X[1];
  // Every bit takes the parity of the bits above it.
  uint32_t t = X[2] >> 1;
  t ^= t >> 1;
  t ^= t >> 2;
  t ^= t >> 4;
  t ^= t >> 8;
  return (spread3(X[0] ^ t) << 2) | (spread3(X[1] ^ t) << 1) | spread3(X[2] ^ t);
}

FPSX_HD uint32_t hilbert10(uint32_t x, uint32_t y, uint32_t z) { return hilbert<10>(x, y, z); }

}  // namespace fpsx
