// The pair form of sixteen 6-bit residuals (GRF_RAW_PAIRS): the same 96 bits as in the packed form, arranged so
// that the residuals of two neighbouring words come out of a dword by one rotation.
//
// A residual gives a BF16 word its sign (bit 15) and its five lowest bits, so a pair of words (the first in the low
// half) takes its twelve residual bits at kPairBits: in each half six places that follow one another round the
// half's sixteen, 15 0 1 2 3 4.  Turned by a multiple of 16 such a set falls on itself, so places can be counted
// modulo 16: a dword holds two pairs (places 15..4 and, turned by six, 5..10) and four places are left (11..14).  Three
// dwords hold pairs 0 to 5; pairs 6 and 7 are made of what is left, the four middle places 1..4 of each in the
// first and second dword, the places 15 and 0 of both in the third.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace grf {

constexpr uint32_t kPairBits = 0x801F801Fu;
constexpr uint32_t kPairOuter = 0x80018001u;  // places 15 and 0 of both halves
constexpr uint32_t kPairInner = 0x001E001Eu;  // places 1..4

__device__ __forceinline__ uint32_t turned_right(uint32_t v, int by) { return by ? __builtin_amdgcn_alignbit(v, v, by) : v; }
__device__ __forceinline__ uint32_t turned_left(uint32_t v, int by) { return turned_right(v, (32 - by) & 31); }

// The residual bits of words 2 i and 2 i + 1 at kPairBits, other bits anything.
__device__ __forceinline__ uint32_t residual_pair(const uint32_t (&d)[3], int i) {
  if (i < 6) return turned_right(d[i / 2], i % 2 * 6);
  const uint32_t outer = turned_right(d[2], i == 6 ? 12 : 14), inner = turned_right(d[i - 6], 10);
  return (outer & kPairOuter) | (inner & ~kPairOuter);
}

// All eight pairs (at kPairBits, other bits zero) -> the group's dwords.
__device__ __forceinline__ void residual_group(const uint32_t (&pair)[8], uint32_t (&d)[3]) {
  for (int k = 0; k < 3; ++k) d[k] = pair[2 * k] | turned_left(pair[2 * k + 1], 6);
  d[0] |= turned_left(pair[6] & kPairInner, 10);
  d[1] |= turned_left(pair[7] & kPairInner, 10);
  d[2] |= turned_left(pair[6] & kPairOuter, 12) | turned_left(pair[7] & kPairOuter, 14);
}

}  // namespace grf
