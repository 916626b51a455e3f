// What the kernels that read planes (word_planes.h) share: a visit's words from what a lane holds of it.
#pragma once
#include "fused_kernels.h"
#include "word_planes.h"

namespace grf {

typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint2v __attribute__((ext_vector_type(2)));
typedef uint32_t uint3v __attribute__((ext_vector_type(3)));
typedef uint16_t pair16 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t scalar(uint32_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_readfirstlane(v);
#else
  return v;
#endif
}

// LDS operations of one wave take effect in order; the compiler is kept from moving them across.
__device__ __forceinline__ void wave_order() {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#endif
}

// Eight words of a step: signs and mantissas s (two dwords), exponent numbers `codes` of four pairs: fields of seven bits
// at 0 and 16, and 7 and 23.  base: the row's lowest exponent, in place, in both halves.
__device__ __forceinline__ void join_words(uint32_t s0, uint32_t s1, uint32_t first, uint32_t second, uint32_t base, uint32_t (&o)[4]) {
#if defined(__HIP_DEVICE_COMPILE__)
  const pair16 b = __builtin_bit_cast(pair16, base);
  uint32_t place = 0x00800080u;  // (as a constant it would be a shift and an addition in place of one multiply-add)
  asm("" : "+s"(place));
  const pair16 k = __builtin_bit_cast(pair16, place);
  auto two = [&](uint32_t codes, uint32_t s, uint32_t &low, uint32_t &high) {
    const pair16 p = __builtin_bit_cast(pair16, codes);
    const pair16 q = (p * (uint16_t)187) >> (uint16_t)11;  // p / 11 for p < 121
    const pair16 r = p - q * (uint16_t)11;
    const uint32_t lo = __builtin_bit_cast(uint32_t, (pair16)(r * k + b));
    const uint32_t hi = __builtin_bit_cast(uint32_t, (pair16)(q * k + b));
    low = (s & kSignMantissa) | lo;
    high = (__builtin_amdgcn_alignbit(s, s, 8) & kSignMantissa) | hi;
  };
  two(first, s0, o[0], o[1]);
  two(second, s1, o[2], o[3]);
#else
  (void)s0, (void)s1, (void)first, (void)second, (void)base, (void)o;
#endif
}

// A row block's whole visits [0, full), beyond which a load gives zeros and reads nothing: the visit after the last one is
// asked for like the rest, and the loads under way are never waited for at a branch.
struct VisitBytes {
#if defined(__HIP_DEVICE_COMPILE__)
  __amdgpu_buffer_rsrc_t bytes;
  __device__ __forceinline__ VisitBytes(const uint8_t *block, uint32_t full)
      : bytes(__builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(block), 0, (int)(full * kVisitBytes), 0x00020000)) {}
  __device__ __forceinline__ uint4v four(uint32_t at) const { return __builtin_bit_cast(uint4v, __builtin_amdgcn_raw_buffer_load_b128(bytes, at, 0, 0)); }
  __device__ __forceinline__ uint3v three(uint32_t at) const { return __builtin_bit_cast(uint3v, __builtin_amdgcn_raw_buffer_load_b96(bytes, at, 0, 0)); }
#else
  __device__ VisitBytes(const uint8_t *, uint32_t) {}
  __device__ uint4v four(uint32_t) const { return {}; }
  __device__ uint3v three(uint32_t) const { return {}; }
#endif
};

// What a lane holds of a visit.
struct Exponents {
  uint4v e0;
  uint3v e1;
  __device__ __forceinline__ void load(const VisitBytes &from, uint32_t v, uint32_t slot) {
    e0 = from.four(v * kVisitBytes + 4096 + slot * 16);
    e1 = from.three(v * kVisitBytes + 5120 + slot * 12);
  }
};

struct Visit {
  uint4v s[4];  // steps 2 j and 2 j + 1
  Exponents e;
  __device__ __forceinline__ void load(const uint8_t *at, uint32_t slot) {
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] = *reinterpret_cast<const uint4v *>(at + j * 1024 + slot * 16);
    e.e0 = *reinterpret_cast<const uint4v *>(at + 4096 + slot * 16);
    e.e1 = *reinterpret_cast<const uint3v *>(at + 5120 + slot * 12);
  }
  __device__ __forceinline__ void load_signs(const VisitBytes &from, uint32_t v, uint32_t j, uint32_t slot) {
    s[j] = from.four(v * kVisitBytes + j * 1024 + slot * 16);
  }
  __device__ __forceinline__ void load(const VisitBytes &from, uint32_t v, uint32_t slot) {
#pragma unroll
    for (int j = 0; j < 4; ++j) load_signs(from, v, j, slot);
    e.load(from, v, slot);
  }
  template <int T>
  __device__ __forceinline__ void step(uint32_t base, uint32_t (&o)[4]) const {
    constexpr uint32_t kCodes = kCodeFields;
    const uint4v &e0 = e.e0;
    const uint3v &e1 = e.e1;
    uint32_t d;
    if constexpr (T < 4) {
      d = e0[T];
    } else if constexpr (T < 7) {
      d = e1[T - 4];
    } else {  // the two bits above the fields of each half, dword after dword
      constexpr uint32_t k = 0x00030003u;
      d = (e0[0] >> 14) & k;
      d |= (e0[1] >> 12) & (k << 2);
      d |= (e0[2] >> 10) & (k << 4);
      d |= (e0[3] >> 8) & (k << 6);
      d |= (e1[0] >> 6) & (k << 8);
      d |= (e1[1] >> 4) & (k << 10);
      d |= (e1[2] >> 2) & (k << 12);
    }
    join_words(s[T / 2][T % 2 * 2], s[T / 2][T % 2 * 2 + 1], d & kCodes, (d >> 7) & kCodes, base, o);
  }
};

// A unit of 64 columns of the last, shorter visit: two steps.
struct ShortVisit {
  uint4v s;
  uint2 e;
  __device__ __forceinline__ void load(const uint8_t *at, uint32_t slot) {
    s = *reinterpret_cast<const uint4v *>(at + slot * 16);
    e = *reinterpret_cast<const uint2 *>(at + 1024 + slot * 8);
  }
  template <int T>
  __device__ __forceinline__ void step(uint32_t base, uint32_t (&o)[4]) const {
    const uint32_t d = T ? e.y : e.x;
    join_words(s[T * 2], s[T * 2 + 1], d & kCodeFields, (d >> 7) & kCodeFields, base, o);
  }
};

}  // namespace grf
