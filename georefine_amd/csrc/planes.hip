// Products, decode and row gather of a matrix that is resident as planes, and the kernels that lay it out.
//
// A BF16 word is a sign and seven mantissa bits that do not compress (8 bits) and an exponent that does.  A
// context frame codes the exponents near their entropy (2.5 bits) as one chain of states, which costs a wave 15 vector
// instructions and two dependent LDS reads a symbol.  Here a row's exponents are numbered from the lowest of the
// eleven that hold most of it; two numbers below eleven share seven bits (3.5 a weight), and the few words outside
// (one in 400 of a normal distribution) are listed.  That is 11.5 bits a weight and the list, what the frame takes with its
// index, at fixed places: 2.6 vector instructions a weight, no chain, no LDS table.
//
// Blocks of sixteen rows are cut into visits of 256 columns (word_planes.h has the places).  A visit's
// 5888 bytes are read once by one wave, whose lane holds what v_mfma_f32_16x16x32_bf16 takes as its second
// operand: row lane % 16, in step t of eight the columns 32 t + 8 (lane / 16) .. + 7.
#include "fused_kernels.h"
#include "word_planes.h"

namespace {

using grf::bf16x8_t;
using grf::float4v;
using grf::round_bf16;

typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef uint32_t uint3v __attribute__((ext_vector_type(3)));
typedef uint16_t pair16 __attribute__((ext_vector_type(2)));

constexpr uint32_t kMaxMembers = 4;
constexpr uint32_t kMaxTileRows = 128;  // activation rows of a launch
constexpr uint32_t kInPlaceRows = 16;   // up to which x is read where it is
constexpr uint32_t kMaxSharing = 2;    // splits of a part
constexpr uint32_t kPatch = 4096;       // LDS bytes in which a wave's half visit is completed

struct PlanesMember {
  grf_planes p;
  uint16_t *y;
  const uint16_t *bias;
  float *partials;                   // [parts][activation rows][rows]
  uint32_t ldy, first, blocks_each;  // first workgroup; row blocks a workgroup
};

struct PlanesGroup {
  PlanesMember m[kMaxMembers];
  uint32_t n;
};

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
  auto two = [&](uint32_t codes, uint32_t s, uint32_t &low, uint32_t &high) {
    const pair16 p = __builtin_bit_cast(pair16, codes);
    const pair16 q = (p * (uint16_t)187) >> (uint16_t)11;  // p / 11 for p < 121
    const pair16 r = p - q * (uint16_t)11;
    const uint32_t lo = __builtin_bit_cast(uint32_t, (pair16)(r * (uint16_t)128 + b));
    const uint32_t hi = __builtin_bit_cast(uint32_t, (pair16)(q * (uint16_t)128 + b));
    low = (s & grf::kSignMantissa) | lo;
    high = (__builtin_amdgcn_alignbit(s, s, 8) & grf::kSignMantissa) | hi;
  };
  two(first, s0, o[0], o[1]);
  two(second, s1, o[2], o[3]);
#else
  (void)s0, (void)s1, (void)first, (void)second, (void)base, (void)o;
#endif
}

// What a lane holds of a visit.
struct Visit {
  uint4v s[4];  // steps 2 j and 2 j + 1
  uint4v e0;
  uint3v e1;
  __device__ __forceinline__ void load(const uint8_t *at, uint32_t slot) {
#pragma unroll
    for (int j = 0; j < 4; ++j) s[j] = *reinterpret_cast<const uint4v *>(at + j * 1024 + slot * 16);
    e0 = *reinterpret_cast<const uint4v *>(at + 4096 + slot * 16);
    e1 = *reinterpret_cast<const uint3v *>(at + 5120 + slot * 12);
  }
  template <int T>
  __device__ __forceinline__ void step(uint32_t base, uint32_t (&o)[4]) const {
    constexpr uint32_t kCodes = grf::kCodeFields;
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
    join_words(s[T * 2], s[T * 2 + 1], d & grf::kCodeFields, (d >> 7) & grf::kCodeFields, base, o);
  }
};

// Words of a visit that its planes do not hold: entries [first, first + count) of the list, the lane's first in hand.
struct Listed {
  const uint32_t *list;
  uint32_t first, count, entry;
  __device__ __forceinline__ void load(const uint32_t *all, uint32_t from, uint32_t to, uint32_t lane) {
    list = all, first = from, count = to - from;
    entry = all[from + min(lane, count ? count - 1 : 0)];  // (the list ends with an entry that nobody owns)
  }
  // Those of the N words from word FIRST of the visit on, into the words at `lds`.
  template <uint32_t FIRST, uint32_t N>
  __device__ __forceinline__ void patch(uint8_t *lds, uint32_t lane) const {
    for (uint32_t k = 0; k < count; k += 64) {  // uniform
      const uint32_t mine = k ? list[first + min(k + lane, count - 1)] : entry;
      const uint32_t place = (mine >> 16) - FIRST;
      if (k + lane < count && place < N) *reinterpret_cast<uint16_t *>(lds + place * 2) = (uint16_t)mine;
    }
  }
};

// ------------------------------------------------------------------- products

struct PlanesX {
  const uint8_t *data;
  uint32_t row_bytes, chunk_bytes, m_rows, cols;  // bytes from a row to the next, from eight columns to the next
};

// MT: tiles of sixteen activation rows.  A workgroup's waves share out the visits of `blocks_each` row blocks, `splits`
// waves a block, and add their sums in wave order: what a row of x gives depends on nothing but the matrix's
// sizes, so all row counts, single and grouped launches agree bit for bit.
template <int MT>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(6))) void planes_product_kernel(PlanesGroup g, PlanesX x) {
  extern __shared__ __align__(16) uint8_t lds[];
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t lane = threadIdx.x % 64, wave = scalar(threadIdx.x / 64);
  uint32_t i = 0;
  while (i + 1 < g.n && blockIdx.x >= g.m[i + 1].first) ++i;
  const PlanesMember &m = g.m[i];
  const uint32_t splits = m.p.splits, sub = wave / splits, split = wave % splits;
  const uint32_t blocks = (m.p.rows + 15) / 16, block = (blockIdx.x - m.first) * m.blocks_each + sub;
  const grf::PlanesShape shape(x.cols);
  const bool works = sub < m.blocks_each && block < blocks;
  float4v acc[MT] = {};
  if (works) {
    const uint32_t each = (shape.visits() + splits - 1) / splits;
    const uint32_t v0 = min(split * each, shape.visits()), v1 = min(v0 + each, shape.visits()), full = min(v1, shape.full);
    const uint32_t q = lane / 16, r = lane % 16, slot = r * 4 + q;
    uint8_t *patch = lds + wave * kPatch;
    const uint8_t *at = m.p.planes + (size_t)block * shape.block_bytes();
    const uint32_t base = m.p.bases[block * 16 + r];
    const uint32_t ends = m.p.listed_at[block * shape.visits() + min(v0 + lane, shape.visits())];  // (of up to 63 visits)
    auto end_of = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane(ends, v - v0); };
    const uint8_t *xr[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) xr[j] = x.data + (size_t)min(r + 16 * j, x.m_rows - 1) * x.row_bytes + q * x.chunk_bytes;

    auto multiply = [&](const uint32_t (&o)[4], const uint8_t *const (&from)[MT], uint32_t offset) {
      const bf16x8_t w = __builtin_bit_cast(bf16x8_t, (uint4v){o[0], o[1], o[2], o[3]});
#pragma unroll
      for (int j = 0; j < MT; ++j)
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4v *>(from[j] + offset)), w,
                                                         acc[j], 0, 0, 0);
    };

    if (v0 < full) {
      for (uint32_t v = v0; v < full; ++v) {
        Visit now;
        Listed listed;
        now.load(at + (size_t)v * grf::kVisitBytes, slot);
        listed.load(m.p.listed, end_of(v), end_of(v + 1), lane);
        const uint32_t x0 = v * 32 * x.chunk_bytes, xs = 4 * x.chunk_bytes;
        auto half = [&](auto which) {
          constexpr int H = decltype(which)::value;
          uint32_t o[4][4];
          now.step<4 * H>(base, o[0]);
          now.step<4 * H + 1>(base, o[1]);
          now.step<4 * H + 2>(base, o[2]);
          now.step<4 * H + 3>(base, o[3]);
          if (listed.count) {
            uint4v *words = reinterpret_cast<uint4v *>(patch);
#pragma unroll
            for (int t = 0; t < 4; ++t) words[t * 64 + lane] = (uint4v){o[t][0], o[t][1], o[t][2], o[t][3]};
            wave_order();
            listed.patch<H * 2048, 2048>(patch, lane);
            wave_order();
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              const uint4v w = words[t * 64 + lane];
              o[t][0] = w[0], o[t][1] = w[1], o[t][2] = w[2], o[t][3] = w[3];
            }
            wave_order();
          }
#pragma unroll
          for (int t = 0; t < 4; ++t) multiply(o[t], xr, x0 + (4 * H + t) * xs);
        };
        half(std::integral_constant<int, 0>{});
        half(std::integral_constant<int, 1>{});
      }
    }
    if (v0 < v1 && v1 > shape.full) {  // the shorter visit, a unit at a time
      Listed listed;
      listed.load(m.p.listed, end_of(shape.full), end_of(shape.full + 1), lane);
      for (uint32_t u = 0; u < shape.units; ++u) {
        ShortVisit now;
        now.load(at + shape.full * grf::kVisitBytes + u * grf::kUnitBytes, slot);
        uint32_t o[2][4];
        now.step<0>(base, o[0]);
        now.step<1>(base, o[1]);
        uint4v *words = reinterpret_cast<uint4v *>(patch);  // (the unit's steps are 2 u and 2 u + 1 of the visit)
#pragma unroll
        for (int t = 0; t < 2; ++t) words[t * 64 + lane] = (uint4v){o[t][0], o[t][1], o[t][2], o[t][3]};
        wave_order();
        for (uint32_t k = 0; k < listed.count; k += 64) {
          const uint32_t mine = k ? listed.list[listed.first + min(k + lane, listed.count - 1)] : listed.entry;
          if (k + lane < listed.count && (mine >> 16) / 1024 == u) *reinterpret_cast<uint16_t *>(patch + (mine >> 16) % 1024 * 2) = (uint16_t)mine;
        }
        wave_order();
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const uint4v w = words[t * 64 + lane];
          // columns past the last one: the planes hold numbers there, x is not read and counts as zeros
          const uint32_t chunk = (shape.full * 8 + u * 2 + t) * 4 + q;
          const bool inside = chunk * 8 < x.cols;
#pragma unroll
          for (int j = 0; j < MT; ++j) {
            uint4v a = *reinterpret_cast<const uint4v *>(xr[j] + (inside ? (chunk - q) * x.chunk_bytes : 0));
            if (!inside) a = (uint4v){0, 0, 0, 0};
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, w), acc[j], 0, 0, 0);
          }
        }
        wave_order();
      }
    }
  }
  __syncthreads();  // the words of all waves are read
  float4v *sums = reinterpret_cast<float4v *>(lds);
#pragma unroll
  for (int j = 0; j < MT; ++j) sums[(wave * MT + j) * 64 + lane] = acc[j];
  __syncthreads();
  // Four activation rows of one weight row at a time: the waves' sums in their order, the bias, one rounding.
  for (uint32_t t = threadIdx.x; t < m.blocks_each * MT * 64; t += blockDim.x) {
    const uint32_t l = t % 64, j = t / 64 % MT, s = t / (64 * MT);
    const uint32_t row = ((blockIdx.x - m.first) * m.blocks_each + s) * 16 + l % 16, m0 = j * 16 + l / 16 * 4;
    if (row >= m.p.rows || m0 >= x.m_rows) continue;
    // a part's splits one after the other, then the parts
    const uint32_t per_part = splits / m.p.parts;
    float4v sum = {};
    for (uint32_t part = 0; part < m.p.parts; ++part) {
      const float4v *from = sums + ((s * splits + part * per_part) * MT + j) * 64 + l;
      float4v one = *from;
      for (uint32_t w = 1; w < per_part; ++w) one += from[w * MT * 64];
      sum = part ? sum + one : one;
    }
    const float b = m.bias ? __uint_as_float((uint32_t)m.bias[row] << 16) : 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (m0 + k < x.m_rows) m.y[(size_t)(m0 + k) * m.ldy + row] = round_bf16(m.bias ? sum[k] + b : sum[k]);
  }
#else
  (void)g, (void)x, (void)lds;
#endif
}

// More than sixteen rows of x: a wave has a row block and one split of its visits.  The four waves of a workgroup that
// share a split share its x as well, which comes into LDS a quarter of a visit at a time in operand order, the next
// while this one is multiplied.  (In place every row block reads all of x: 64 rows of 17408 x 5120 109 us, the
// lines of a step in few cache sets.)  A workgroup has the splits of one part.
constexpr uint32_t kBatchBlocks = 4;
template <int MT>
__global__ __launch_bounds__(kBatchBlocks * kMaxSharing * 64) __attribute__((amdgpu_waves_per_eu(MT == 8 ? 4 : 5))) void planes_batch_kernel(
    PlanesGroup g, PlanesX x) {
  extern __shared__ __align__(16) uint8_t lds[];
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int kCopies = MT / 2;                   // operands that a wave brings for a quarter
  constexpr uint32_t kQuarterX = 2 * MT * 1024;     // bytes of x for a quarter
  const uint32_t lane = threadIdx.x % 64, wave = scalar(threadIdx.x / 64), own = wave % kBatchBlocks, share = wave / kBatchBlocks;
  uint32_t i = 0;
  while (i + 1 < g.n && blockIdx.x >= g.m[i + 1].first) ++i;
  const PlanesMember &m = g.m[i];
  const grf::PlanesShape shape(x.cols);
  const uint32_t blocks = (m.p.rows + 15) / 16, groups = (blocks + kBatchBlocks - 1) / kBatchBlocks;
  const uint32_t part = (blockIdx.x - m.first) / groups, wanted = (blockIdx.x - m.first) % groups * kBatchBlocks + own;
  const uint32_t sharing = m.p.splits / m.p.parts;  // (members of a group may have fewer than the launch)
  const uint32_t block = min(wanted, blocks - 1);   // (a wave without a block copies and waits like the rest)
  const uint32_t each = (shape.visits() + m.p.splits - 1) / m.p.splits, split = part * sharing + min(share, sharing - 1);
  const uint32_t v0 = split * each, v1 = min(v0 + each, shape.visits()), full = min(v1, shape.full);
  const uint32_t q = lane / 16, r = lane % 16, slot = r * 4 + q;
  uint8_t *const xlds = lds + share * 2 * kQuarterX, *const patch = lds + blockDim.x / (kBatchBlocks * 64) * 2 * kQuarterX + wave * (kPatch / 2);
  const uint8_t *at = m.p.planes + (size_t)block * shape.block_bytes();
  const uint32_t base = m.p.bases[block * 16 + r];
  const uint32_t *listed_at = m.p.listed_at + block * shape.visits();

  uint4v held[kCopies];
  const uint8_t *xr[kCopies];
#pragma unroll
  for (int j = 0; j < kCopies; ++j) xr[j] = x.data + (size_t)min(r + 16 * ((own + kBatchBlocks * j) % MT), x.m_rows - 1) * x.row_bytes;
  auto fetch_x = [&](uint32_t quarter) {
#pragma unroll
    for (int j = 0; j < kCopies; ++j) {
      const uint32_t chunk = (quarter * 2 + (own + kBatchBlocks * j) / MT) * 4 + q;
      held[j] = *reinterpret_cast<const uint4v *>(xr[j] + (size_t)(chunk * 8 < x.cols ? chunk : 0) * x.chunk_bytes);
      if (chunk * 8 >= x.cols) held[j] = (uint4v){0, 0, 0, 0};  // columns past the last one
    }
  };
  auto keep_x = [&](uint32_t quarter) {
    uint4v *to = reinterpret_cast<uint4v *>(xlds + quarter % 2 * kQuarterX);
#pragma unroll
    for (int j = 0; j < kCopies; ++j) to[(own + kBatchBlocks * j) * 64 + lane] = held[j];
  };
  // The workgroup's LDS is written; loads under way stay so.
  auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  float4v acc[MT] = {};
  Visit now;
  Listed listed;
  auto fetch = [&](uint32_t v) {
    const uint32_t there = min(v, shape.visits() - 1);
    if (v < full) now.load(at + (size_t)there * grf::kVisitBytes, slot);
    listed.load(m.p.listed, listed_at[there], listed_at[there + 1], lane);
  };
  fetch_x(4 * v0);
  fetch(v0);
  keep_x(4 * v0);
  meet();
  for (uint32_t v = v0; v < v0 + each; ++v) {  // (as many for all: they meet)
    auto quarter = [&](auto which) {
      constexpr int Q = decltype(which)::value;
      const uint32_t h = 4 * v + Q;
      fetch_x(h + 1);
      if (v < v1) {
        uint32_t o[2][4] = {};
        if (v < shape.full) {
          now.step<2 * Q>(base, o[0]);
          now.step<2 * Q + 1>(base, o[1]);
        } else if (Q < shape.units) {
          ShortVisit one;
          one.load(at + (size_t)v * grf::kVisitBytes + Q * grf::kUnitBytes, slot);
          one.step<0>(base, o[0]);
          one.step<1>(base, o[1]);
        }
        if (listed.count) {
          uint4v *words = reinterpret_cast<uint4v *>(patch);
#pragma unroll
          for (int t = 0; t < 2; ++t) words[t * 64 + lane] = (uint4v){o[t][0], o[t][1], o[t][2], o[t][3]};
          wave_order();
          listed.patch<Q * 1024, 1024>(patch, lane);
          wave_order();
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const uint4v w = words[t * 64 + lane];
            o[t][0] = w[0], o[t][1] = w[1], o[t][2] = w[2], o[t][3] = w[3];
          }
          wave_order();
        }
        if constexpr (Q == 3) fetch(v + 1);  // (into the registers that this visit no longer needs)
        const uint4v *from = reinterpret_cast<const uint4v *>(xlds + h % 2 * kQuarterX);
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const bf16x8_t w = __builtin_bit_cast(bf16x8_t, (uint4v){o[t][0], o[t][1], o[t][2], o[t][3]});
#pragma unroll
          for (int j = 0; j < MT; ++j)
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, from[(t * MT + j) * 64 + lane]), w, acc[j], 0, 0, 0);
        }
      }
      keep_x(h + 1);
      meet();
    };
    quarter(std::integral_constant<int, 0>{});
    quarter(std::integral_constant<int, 1>{});
    quarter(std::integral_constant<int, 2>{});
    quarter(std::integral_constant<int, 3>{});
  }
  // The splits' sums in their order, in the first one's wave.
  float4v *sums = reinterpret_cast<float4v *>(lds);
  for (uint32_t k = 1; k < sharing; ++k) {
    if (share == k)
#pragma unroll
      for (int j = 0; j < MT; ++j) sums[(own * MT + j) * 64 + lane] = acc[j];
    __syncthreads();
    if (!share)
#pragma unroll
      for (int j = 0; j < MT; ++j) acc[j] += sums[(own * MT + j) * 64 + lane];
    __syncthreads();
  }
  const uint32_t row = block * 16 + r;
  if (share || wanted >= blocks || row >= m.p.rows) return;
  const float b = m.bias ? __uint_as_float((uint32_t)m.bias[row] << 16) : 0.0f;
#pragma unroll
  for (int j = 0; j < MT; ++j)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t xrow = j * 16 + q * 4 + k;
      if (xrow >= x.m_rows) continue;
      if (m.p.parts > 1)
        m.partials[((size_t)part * x.m_rows + xrow) * m.p.rows + row] = acc[j][k];
      else
        m.y[(size_t)xrow * m.ldy + row] = round_bf16(m.bias ? acc[j][k] + b : acc[j][k]);
    }
#else
  (void)g, (void)x, (void)lds;
#endif
}

// The parts of a batch's members in order, the bias, one rounding.
__global__ __launch_bounds__(256) void planes_sum_kernel(PlanesGroup g, uint32_t m_rows) {
  uint32_t i = 0;
  while (i + 1 < g.n && blockIdx.x >= g.m[i + 1].first) ++i;
  const PlanesMember &m = g.m[i];
  const uint32_t columns = (m.p.rows + 255) / 256, at = blockIdx.x - m.first;
  const uint32_t row = at % columns * 256 + threadIdx.x, xrow = at / columns;
  if (row >= m.p.rows) return;
  const float *from = m.partials + (size_t)xrow * m.p.rows + row;
  const size_t pitch = (size_t)m_rows * m.p.rows;
  float sum = *from;
  for (uint32_t k = 1; k < m.p.parts; ++k) sum += from[k * pitch];
  if (m.bias) sum += __uint_as_float((uint32_t)m.bias[row] << 16);
  m.y[(size_t)xrow * m.ldy + row] = round_bf16(sum);
}

template <int MT>
int launch_batch(const PlanesGroup &g, const PlanesX &x, uint32_t sharing, uint32_t grid, hipStream_t s) {
  constexpr auto kernel = &planes_batch_kernel<MT>;
  const uint32_t bytes = sharing * (2 * 2 * MT * 1024 + kBatchBlocks * kPatch / 2);
  if (bytes > 64 * 1024)
    if (int rc = grf::allow_full_lds<kernel>()) return rc;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(sharing * kBatchBlocks * 64), bytes, s, g, x);
  return GRF_OK;
}

template <int MT>
int launch_product(const PlanesGroup &g, const PlanesX &x, uint32_t waves, uint32_t grid, hipStream_t s) {
  constexpr auto kernel = &planes_product_kernel<MT>;
  const uint32_t bytes = waves * std::max<uint32_t>(kPatch, MT * 1024);
  if (bytes > 64 * 1024)
    if (int rc = grf::allow_full_lds<kernel>()) return rc;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(waves * 64), bytes, s, g, x);
  return GRF_OK;
}

int check_planes(const char *who, const grf_planes *p) {
  if (!p || !p->planes || !p->bases || !p->listed_at || !p->listed)
    return grf::set_error(GRF_BAD_ARGUMENT, std::string(who) + ": null argument");
  const grf::PlanesShape shape(p->cols);
  if (!p->rows || !p->cols || p->cols % 8 || ((uintptr_t)p->planes & 15) || p->rows > 1u << 28 || p->cols > GRF_PLANES_MAX_COLS)
    return grf::set_error(GRF_BAD_ARGUMENT, std::string(who) + ": sizes or alignment of the planes");
  const uint32_t each = p->splits ? (shape.visits() + p->splits - 1) / p->splits : 0;
  if (!each || p->splits > 16 || each > 63 || each * (p->splits - 1) >= shape.visits() || !p->parts || p->splits % p->parts || p->splits / p->parts > kMaxSharing)
    return grf::set_error(GRF_BAD_ARGUMENT, std::string(who) + ": 1 to 16 splits of 1 to 63 visits each, in parts of one or two");
  return GRF_OK;
}

// fp32 sums of a launch of `m` rows whose members are cut in parts, in bytes.
size_t partial_bytes(const grf_planes &p, uint32_t m) {
  return m > kInPlaceRows && p.parts > 1 ? ((size_t)p.parts * m * p.rows * 4 + 255) / 256 * 256 : 0;
}

int product(const char *who, uint32_t n, const grf_planes *const *planes, const uint16_t *x, uint32_t ldx, uint32_t m_rows, bool packed,
            uint16_t *const *y, const uint32_t *ldy, const uint16_t *const *bias, void *workspace, size_t workspace_bytes, hipStream_t s) {
  if (!n || n > kMaxMembers || !planes || !x || !y || !ldy) return grf::set_error(GRF_BAD_ARGUMENT, std::string(who) + ": null argument or member count");
  PlanesGroup g{};
  g.n = n;
  uint32_t waves = 1, sharing = 1;
  size_t space = 0;
  const uint32_t cols = planes[0] ? planes[0]->cols : 0, most = std::min(m_rows, kMaxTileRows);
  for (uint32_t i = 0; i < n; ++i) {
    if (int rc = check_planes(who, planes[i])) return rc;
    if (!y[i] || ldy[i] < planes[i]->rows || planes[i]->cols != cols)
      return grf::set_error(GRF_BAD_ARGUMENT, std::string(who) + ": output rows or member widths");
    waves = std::max(waves, planes[i]->splits), sharing = std::max(sharing, planes[i]->splits / planes[i]->parts);
    g.m[i] = {*planes[i], y[i], bias ? bias[i] : nullptr, reinterpret_cast<float *>(static_cast<uint8_t *>(workspace) + space), ldy[i], 0, 0};
    space += partial_bytes(*planes[i], most);
  }
  if (((uintptr_t)x & 15) || (!packed && (ldx < cols || ldx % 8 || ldx > 1u << 24)) || (packed && m_rows > kMaxTileRows))
    return grf::set_error(GRF_BAD_ARGUMENT, std::string(who) + ": activation rows are 16-byte aligned");
  if (space && (!workspace || workspace_bytes < space || ((uintptr_t)workspace & 15)))
    return grf::set_error(GRF_BAD_ARGUMENT, std::string(who) + ": workspace too small (grf_planes_workspace_bytes)");
  for (uint32_t done = 0; done < m_rows; done += kMaxTileRows) {
    const uint32_t m = std::min(kMaxTileRows, m_rows - done), m_pad = 16 * grf::gemm_tiles(m);
    const bool batch = m > kInPlaceRows;
    const PlanesX rows{reinterpret_cast<const uint8_t *>(x) + (size_t)done * ldx * 2, packed ? 16 : ldx * 2, packed ? m_pad * 16 : 16, m, cols};
    uint32_t grid = 0;
    bool parts = false;
    for (uint32_t i = 0; i < n; ++i) {
      PlanesMember &one = g.m[i];
      const uint32_t blocks = (one.p.rows + 15) / 16;
      one.blocks_each = batch ? kBatchBlocks : waves / one.p.splits;
      one.y = y[i] + (size_t)done * ldy[i];
      one.first = grid;
      grid += (blocks + one.blocks_each - 1) / one.blocks_each * (batch ? one.p.parts : 1);
      parts |= batch && one.p.parts > 1;
    }
    if (int rc = !batch   ? launch_product<1>(g, rows, waves, grid, s)
                 : m <= 32 ? launch_batch<2>(g, rows, sharing, grid, s)
                 : m <= 64 ? launch_batch<4>(g, rows, sharing, grid, s)
                           : launch_batch<8>(g, rows, sharing, grid, s))
      return rc;
    if (parts) {
      PlanesGroup sums{};
      grid = 0;
      for (uint32_t i = 0; i < n; ++i)
        if (g.m[i].p.parts > 1) {
          sums.m[sums.n] = g.m[i];
          sums.m[sums.n++].first = grid;
          grid += (g.m[i].p.rows + 255) / 256 * m;
        }
      hipLaunchKernelGGL(planes_sum_kernel, dim3(grid), dim3(256), 0, s, sums, m);
    }
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return grf::set_error(GRF_LAUNCH_FAILED, std::string(who) + ": " + hipGetErrorString(e));
  return GRF_OK;
}

// ------------------------------------------------------------------- the dense matrix, and rows of it

// A wave a visit: its words in LDS in the lanes' order, completed there, and read back row by row, so that a store
// of the wave is two runs of whole lines.
__global__ __launch_bounds__(256) void planes_decode_kernel(grf_planes p, uint16_t *out) {
  __shared__ __align__(16) uint8_t lds[4][2 * kPatch];
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t lane = threadIdx.x % 64, wave = scalar(threadIdx.x / 64);
  const grf::PlanesShape shape(p.cols);
  const uint32_t id = blockIdx.x * 4 + wave, block = id / shape.visits(), v = id % shape.visits();
  if (block >= (p.rows + 15) / 16) return;
  const uint32_t q = lane / 16, r = lane % 16, slot = r * 4 + q;
  const uint8_t *at = p.planes + (size_t)block * shape.block_bytes() + (size_t)v * grf::kVisitBytes;
  Listed listed;
  listed.load(p.listed, p.listed_at[id], p.listed_at[id + 1], lane);
  const uint32_t base = p.bases[block * 16 + r];
  uint4v *words = reinterpret_cast<uint4v *>(lds[wave]);
  auto keep = [&](int t, const uint32_t (&o)[4]) { words[t * 64 + lane] = (uint4v){o[0], o[1], o[2], o[3]}; };
  uint32_t o[4];
  if (v < shape.full) {
    Visit now;
    now.load(at, slot);
    now.step<0>(base, o), keep(0, o);
    now.step<1>(base, o), keep(1, o);
    now.step<2>(base, o), keep(2, o);
    now.step<3>(base, o), keep(3, o);
    now.step<4>(base, o), keep(4, o);
    now.step<5>(base, o), keep(5, o);
    now.step<6>(base, o), keep(6, o);
    now.step<7>(base, o), keep(7, o);
  } else {
    for (uint32_t u = 0; u < shape.units; ++u) {
      ShortVisit now;
      now.load(at + u * grf::kUnitBytes, slot);
      now.step<0>(base, o), keep(2 * u, o);
      now.step<1>(base, o), keep(2 * u + 1, o);
    }
  }
  wave_order();
  listed.patch<0, 4096>(lds[wave], lane);
  wave_order();
  const uint32_t c = lane % 32, col = v * 256 + c * 8;  // chunk c of eight words: step c / 4, quad c % 4
#pragma unroll
  for (uint32_t i = 0; i < 8; ++i) {
    const uint32_t row = 2 * i + lane / 32;
    if (block * 16 + row < p.rows && col < p.cols)
      *reinterpret_cast<uint4v *>(out + (size_t)(block * 16 + row) * p.cols + col) = words[c / 4 * 64 + c % 4 * 16 + row];
  }
#else
  (void)p, (void)out, (void)lds;
#endif
}

// A workgroup a requested row, a quad of lanes a visit: a wave holds sixteen visits, 4096 columns.
template <bool TOLD>
__global__ __launch_bounds__(1024) void planes_gather_kernel(grf_planes p, const int64_t *ids, uint16_t *out, int32_t *flag, grf::GatherDone done) {
  extern __shared__ __align__(16) uint8_t lds[];
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t lane = threadIdx.x % 64, wave = scalar(threadIdx.x / 64);
  const int64_t id = ids[blockIdx.x];
  uint32_t row = (uint32_t)id;
  bool refused = false;
  if (id < 0 || id >= (int64_t)p.rows) {  // uniform
    if (flag) {
      if (!threadIdx.x) __hip_atomic_fetch_or(flag, GRF_ERR_INDEX, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      refused = true;
    }
    row = id < 0 ? 0 : p.rows - 1;
  }
  const grf::PlanesShape shape(p.cols);
  const uint32_t block = row / 16, r = row % 16, q = lane % 4, slot = r * 4 + q;
  const uint32_t base = p.bases[row];
  const grf::Words<grf::kSystem> dst{out + (size_t)blockIdx.x * p.cols, p.cols * 2};
  uint8_t *mine = lds + wave * 2 * kPatch + lane / 4 * 512;  // the visit's columns in order
  for (uint32_t first = wave * 16; !refused && first < shape.visits(); first += blockDim.x / 64 * 16) {
    const uint32_t v = first + lane / 4;
    const bool any = v < shape.visits();
    const uint8_t *at = p.planes + (size_t)block * shape.block_bytes() + (size_t)v * grf::kVisitBytes;
    uint32_t from = 0, to = 0, o[4];
    if (any) {
      from = p.listed_at[block * shape.visits() + v], to = p.listed_at[block * shape.visits() + v + 1];
      auto keep = [&](int t) { *reinterpret_cast<uint4v *>(mine + (t * 4 + q) * 16) = (uint4v){o[0], o[1], o[2], o[3]}; };
      if (v < shape.full) {
        Visit now;
        now.load(at, slot);
        now.step<0>(base, o), keep(0);
        now.step<1>(base, o), keep(1);
        now.step<2>(base, o), keep(2);
        now.step<3>(base, o), keep(3);
        now.step<4>(base, o), keep(4);
        now.step<5>(base, o), keep(5);
        now.step<6>(base, o), keep(6);
        now.step<7>(base, o), keep(7);
      } else {
        for (uint32_t u = 0; u < shape.units; ++u) {
          ShortVisit now;
          now.load(at + u * grf::kUnitBytes, slot);
          now.step<0>(base, o), keep(2 * u);
          now.step<1>(base, o), keep(2 * u + 1);
        }
      }
    }
    wave_order();
    for (uint32_t k = from + q; k < to; k += 16) {  // the list is of sixteen rows: four entries a lane at a time
      uint32_t entry[4];
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) entry[j] = p.listed[min(k + 4 * j, to - 1)];
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        const uint32_t place = entry[j] >> 16, its = place / 8 % 64;  // step, lane, word
        if (its % 16 == r) *reinterpret_cast<uint16_t *>(mine + (place / 512 * 32 + its / 16 * 8 + place % 8) * 2) = (uint16_t)entry[j];
      }
    }
    wave_order();
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {  // two visits, 1 KiB, a store
      const uint32_t chunk = i * 64 + lane, col = first * 256 + chunk * 8;
      if (col < p.cols)
        dst.put(col, *reinterpret_cast<const grf::words8_t *>(lds + wave * 2 * kPatch + chunk * 16));
    }
    wave_order();
  }
  if constexpr (TOLD) grf::gather_done(done);
#else
  (void)p, (void)ids, (void)out, (void)flag, (void)done, (void)lds;
#endif
}

// ------------------------------------------------------------------- laying a matrix out

// The lowest of the eleven exponents that hold most of a row (the lowest such, on a tie), a workgroup a row.
__global__ __launch_bounds__(256) void planes_bases_kernel(const uint16_t *words, uint32_t rows, uint32_t cols, uint32_t *bases) {
  __shared__ uint32_t held[256], best;
  const uint32_t row = blockIdx.x, tid = threadIdx.x;
  held[tid] = 0;
  if (!tid) best = 0;
  __syncthreads();
  if (row < rows)
    for (uint32_t c = tid; c < cols; c += 256) atomicAdd(&held[words[(size_t)row * cols + c] >> 7 & 255], 1u);
  __syncthreads();
  uint32_t sum = 0;
  for (uint32_t k = 0; k < grf::kExponents; ++k) sum += tid + k < 256 ? held[tid + k] : 0;
  const bool fits = tid + grf::kExponents <= 256;
  if (fits) atomicMax(&best, sum);
  __syncthreads();
  const uint32_t most = best;
  __syncthreads();
  if (!tid) best = 256;
  __syncthreads();
  if (fits && sum == most) atomicMin(&best, tid);
  __syncthreads();
  if (!tid) bases[row] = best << 7 | best << 23;
}

// A wave a visit: counts[id] = the words outside its rows' exponents, or with `at` the planes and the list.
template <bool WRITE>
__global__ __launch_bounds__(256) void planes_fill_kernel(const uint16_t *words, uint32_t rows, uint32_t cols, const uint32_t *bases,
                                                          uint32_t *counts, const uint32_t *at, uint8_t *planes, uint32_t *listed) {
#if defined(__HIP_DEVICE_COMPILE__)
  const uint32_t lane = threadIdx.x % 64, wave = scalar(threadIdx.x / 64);
  const grf::PlanesShape shape(cols);
  const uint32_t id = blockIdx.x * 4 + wave, block = id / shape.visits(), v = id % shape.visits();
  if (block >= (rows + 15) / 16) return;
  const uint32_t q = lane / 16, r = lane % 16, slot = r * 4 + q, row = block * 16 + r;
  const uint32_t lowest = bases[row] >> 7 & 255;
  const uint32_t steps = v < shape.full ? 8 : shape.units * 2;
  uint32_t found = WRITE ? at[id] : 0, s[2], e[7] = {}, last = 0;
  uint8_t *to = planes + (size_t)block * shape.block_bytes() + (size_t)v * grf::kVisitBytes;
#pragma unroll
  for (uint32_t t = 0; t < 8; ++t) {
    if (t >= steps) continue;  // uniform
    const uint32_t col = v * 256 + t * 32 + q * 8;
    uint4v got = {0, 0, 0, 0};
    const bool inside = row < rows && col < cols;
    if (inside) got = *reinterpret_cast<const uint4v *>(words + (size_t)row * cols + col);
    uint32_t word[8], code[8];
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
      word[i] = got[i / 2] >> (i % 2 * 16) & 0xFFFF;
      code[i] = (word[i] >> 7 & 255) - lowest;
      const bool outside = inside && code[i] >= grf::kExponents;
      const uint64_t mask = __ballot(outside);
      if (outside) {
        if constexpr (WRITE) listed[found + __popcll(mask & ((1ull << lane) - 1))] = ((t * 64 + lane) * 8 + i) << 16 | word[i];
      }
      if (outside || !inside) code[i] = 0, word[i] = 0;
      found += __popcll(mask);
    }
    if constexpr (WRITE) {
      auto sm = [&](uint32_t i) { return word[i] & 0x807F; };
      uint32_t p[2];
#pragma unroll
      for (uint32_t k = 0; k < 2; ++k) {
        const uint32_t low = sm(4 * k) | sm(4 * k + 1) << 16, high = sm(4 * k + 2) | sm(4 * k + 3) << 16;
        s[k] = low | (high << 8 | high >> 24);
        p[k] = (code[4 * k] + 11 * code[4 * k + 2]) | (code[4 * k + 1] + 11 * code[4 * k + 3]) << 16;
      }
      const uint32_t both = p[0] | p[1] << 7;
      if (v < shape.full) {
        *reinterpret_cast<uint2 *>(to + t / 2 * 1024 + slot * 16 + t % 2 * 8) = make_uint2(s[0], s[1]);
        if (t < 7) e[t] = both;
        else last = both;
      } else {
        uint8_t *unit = to + t / 2 * grf::kUnitBytes;
        *reinterpret_cast<uint2 *>(unit + slot * 16 + t % 2 * 8) = make_uint2(s[0], s[1]);
        *reinterpret_cast<uint32_t *>(unit + 1024 + slot * 8 + t % 2 * 4) = both;
      }
    }
  }
  if constexpr (WRITE) {
    if (v < shape.full) {
#pragma unroll
      for (uint32_t t = 0; t < 7; ++t) e[t] |= (last >> (2 * t) & 0x00030003u) << 14;
      *reinterpret_cast<uint4v *>(to + 4096 + slot * 16) = (uint4v){e[0], e[1], e[2], e[3]};
      *reinterpret_cast<uint3v *>(to + 5120 + slot * 12) = (uint3v){e[4], e[5], e[6]};
    }
  } else if (!lane) {
    counts[id] = found;
  }
#else
  (void)words, (void)rows, (void)cols, (void)bases, (void)counts, (void)at, (void)planes, (void)listed;
#endif
}

int launched(const char *who) {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? GRF_OK : grf::set_error(GRF_LAUNCH_FAILED, std::string(who) + ": " + hipGetErrorString(e));
}

int check_words(const char *who, const void *words, uint32_t rows, uint32_t cols, const void *a, const void *b) {
  if (!words || !a || !b || !rows || !cols || cols % 8 || ((uintptr_t)words & 15) || rows > 1u << 28 || cols > GRF_PLANES_MAX_COLS ||
      (uint64_t)((rows + 15) / 16) * grf::PlanesShape(cols).visits() > 1u << 30)
    return grf::set_error(GRF_BAD_ARGUMENT, std::string(who) + ": sizes or alignment");
  return GRF_OK;
}

uint32_t visit_groups(uint32_t rows, uint32_t cols) {
  return ((rows + 15) / 16 * grf::PlanesShape(cols).visits() + 3) / 4;
}

}  // namespace

extern "C" {

uint64_t grf_planes_bytes(uint32_t rows, uint32_t cols) { return (uint64_t)((rows + 15) / 16) * grf::PlanesShape(cols).block_bytes(); }
uint32_t grf_planes_visits(uint32_t rows, uint32_t cols) { return (rows + 15) / 16 * grf::PlanesShape(cols).visits(); }

int grf_planes_count(const uint16_t *words, uint32_t rows, uint32_t cols, uint32_t *bases, uint32_t *counts, void *hip_stream) {
  if (int rc = check_words("grf_planes_count", words, rows, cols, bases, counts)) return rc;
  hipLaunchKernelGGL(planes_bases_kernel, dim3((rows + 15) / 16 * 16), dim3(256), 0, (hipStream_t)hip_stream, words, rows, cols, bases);
  hipLaunchKernelGGL(planes_fill_kernel<false>, dim3(visit_groups(rows, cols)), dim3(256), 0, (hipStream_t)hip_stream, words, rows, cols,
                     bases, counts, nullptr, nullptr, nullptr);
  return launched("grf_planes_count");
}

int grf_planes_fill(const uint16_t *words, uint32_t rows, uint32_t cols, const uint32_t *bases, const uint32_t *listed_at, void *planes,
                    uint32_t *listed, void *hip_stream) {
  if (int rc = check_words("grf_planes_fill", words, rows, cols, bases, listed_at)) return rc;
  if (!planes || !listed || ((uintptr_t)planes & 15)) return grf::set_error(GRF_BAD_ARGUMENT, "grf_planes_fill: null argument or alignment");
  hipLaunchKernelGGL(planes_fill_kernel<true>, dim3(visit_groups(rows, cols)), dim3(256), 0, (hipStream_t)hip_stream, words, rows, cols,
                     bases, nullptr, listed_at, static_cast<uint8_t *>(planes), listed);
  return launched("grf_planes_fill");
}

size_t grf_planes_workspace_bytes(uint32_t n, const grf_planes *const *planes, uint32_t m_rows) {
  size_t bytes = 0;
  for (uint32_t i = 0; planes && i < n; ++i)
    if (planes[i]) bytes += partial_bytes(*planes[i], std::min(m_rows, kMaxTileRows));
  return bytes;
}

int grf_planes_linear(const grf_planes *planes, const uint16_t *x, uint32_t ldx, uint32_t m_rows, uint32_t packed, uint16_t *y,
                      const uint16_t *bias, void *workspace, size_t workspace_bytes, void *hip_stream) {
  const uint32_t ldy = planes ? planes->rows : 0;
  return product("grf_planes_linear", 1, &planes, x, ldx, m_rows, packed != 0, &y, &ldy, &bias, workspace, workspace_bytes,
                 (hipStream_t)hip_stream);
}

int grf_planes_group(uint32_t n, const grf_planes *const *planes, const uint16_t *x, uint32_t ldx, uint32_t m_rows, uint32_t packed,
                     uint16_t *const *y, const uint32_t *ldy, const uint16_t *const *bias, void *workspace, size_t workspace_bytes,
                     void *hip_stream) {
  return product("grf_planes_group", n, planes, x, ldx, m_rows, packed != 0, y, ldy, bias, workspace, workspace_bytes, (hipStream_t)hip_stream);
}

int grf_planes_decode(const grf_planes *planes, uint16_t *out, void *hip_stream) {
  if (int rc = check_planes("grf_planes_decode", planes)) return rc;
  if (!out || ((uintptr_t)out & 15)) return grf::set_error(GRF_BAD_ARGUMENT, "grf_planes_decode: out is 16-byte aligned");
  hipLaunchKernelGGL(planes_decode_kernel, dim3(visit_groups(planes->rows, planes->cols)), dim3(256), 0, (hipStream_t)hip_stream, *planes, out);
  return launched("grf_planes_decode");
}

int grf_planes_gather(const grf_planes *planes, const int64_t *ids, uint32_t count, uint16_t *out, int32_t *index_error, void *counters,
                      int32_t *done, void *hip_stream) {
  if (int rc = check_planes("grf_planes_gather", planes)) return rc;
  if (!ids || !out || ((uintptr_t)out & 15)) return grf::set_error(GRF_BAD_ARGUMENT, "grf_planes_gather: out is 16-byte aligned");
  if (done && (!counters || !count || (uintptr_t)counters & 127))
    return grf::set_error(GRF_BAD_ARGUMENT, "grf_planes_gather: counters (128-byte aligned) and ids are needed");
  if (!count) return GRF_OK;
  const uint32_t waves = std::min(8u, (grf::PlanesShape(planes->cols).visits() + 15) / 16);
  const grf::GatherDone told{static_cast<uint32_t *>(counters), done};
  const auto kernel = done ? &planes_gather_kernel<true> : &planes_gather_kernel<false>;
  hipLaunchKernelGGL(kernel, dim3(count), dim3(waves * 64), waves * 2 * kPatch, (hipStream_t)hip_stream, *planes, ids, out, index_error, told);
  return launched("grf_planes_gather");
}

}  // extern "C"
