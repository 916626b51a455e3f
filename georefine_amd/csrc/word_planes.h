// Where the words of a matrix that is resident as planes lie (planes.hip).
//
// Rows go in blocks of sixteen, a block's columns in visits of 256 and one shorter visit of up to three units of 64; what
// a block lacks of sixteen rows and the last unit of 64 columns is laid out like the rest and never read as a result.
// Lane l of the wave that reads a visit has row l % 16 and, in step t of eight, columns 32 t + 8 (l / 16) .. + 7.
// Its place among the 64 is 4 (l % 16) + l / 16: every load of the wave is one run, and a row's share of a load 64 bytes of it.
//   signs and mantissas, two bytes a pair of words in four loads of 16 bytes a lane, two steps each: a
//     dword holds the fields 0x807F807F of words 0 and 1 as they are and of words 2 and 3 rotated by eight, the next one words 4 to 7;
//   exponents, numbered from the row's lowest: two words share p = n + 11 n' < 121.  A step has four p of seven bits, of
//     words 0 and 2, 1 and 3 (bits 0 and 16 on of its dword), 4 and 6, 5 and 7 (7 and 23 on).  The dwords of steps 0 to 6 are stored, in a load of 16 and one of
//     12 bytes a lane; the fourteen bits a half of step 7 are the two that each of these has left.
// A unit of the shorter visit is two steps: 16 bytes of signs and mantissas a lane, and two dwords of exponents.
#pragma once
#include <cstdint>

#if defined(__HIPCC__)
#define GRF_BOTH __host__ __device__
#else
#define GRF_BOTH
#endif

namespace grf {
constexpr uint32_t kExponents = 11;                  // of a row that the planes hold
constexpr uint32_t kSignMantissa = 0x807F807Fu, kCodeFields = 0x007F007Fu;
constexpr uint32_t kVisitBytes = 5888, kUnitBytes = 1536;  // of sixteen rows by 256 and by 64 columns

struct PlanesShape {
  uint32_t full, units;  // whole visits, units of the shorter one
  GRF_BOTH explicit PlanesShape(uint32_t cols) : full(cols / 256), units((cols % 256 + 63) / 64) {}
  GRF_BOTH uint32_t visits() const { return full + (units ? 1 : 0); }
  GRF_BOTH uint32_t block_bytes() const { return full * kVisitBytes + units * kUnitBytes; }
};
}  // namespace grf
