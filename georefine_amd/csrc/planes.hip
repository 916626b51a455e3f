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
#include "planes_device.h"

namespace {

using grf::bf16x8_t;
using grf::Exponents;
using grf::float4v;
using grf::round_bf16;
using grf::scalar;
using grf::ShortVisit;
using grf::uint3v;
using grf::uint4v;
using grf::Visit;
using grf::VisitBytes;
using grf::wave_order;

constexpr uint32_t kMaxMembers = 4;
constexpr uint32_t kMaxTileRows = 128;  // activation rows of a launch
// Rows of x up to which every wave brings its own: it needs no other wave and no second launch, but reads x once a row block where
// four waves share it once in eight.  us of launches in a row, own and shared, 16 and 32 rows: 1024 x 5120 8.4 13.4, 10.2 14.8; 4096 x 4096
// 9.8 15.6, 11.8 17.3; 8192 x 4096 14.4 19.5, 17.8 20.9; 5120 x 5120 16.4 18.7, 21.8 20.4; 10240 x 5120 22.9 26.1, 30.1 28.4; one row of
// 17408 x 5120 twice 52 57, 16 rows 65 58.  The line by visits is coarse: 16 rows of 4608 x 14336 37.0 30.9, 32 rows of 6144 x 6144 24.9 23.5.
constexpr uint32_t kOwnAlways = 8;                    // up to which it always does
constexpr uint32_t kOwnRows = 32, kOwnVisits = 16384;  // and, in launches of fewer visits than that
// More than sixteen rows take 16 KiB of LDS a wave, so that six waves are alone on a unit; where more such workgroups come than there are
// units, and a wave has more than one visit, x is shared (32 rows, own and shared: 4112 x 3072 16.2 16.1, 4112 x 5120 21.9 19.2, 5120 x
// 6144 26.8 20.9, 5120 x 12288 46.7 29.8, 9000 x 6144 39.4 27.6, 11000 x 4096 29.7 26.4; of one visit 5120 x 1536 12.1 13.6).
constexpr uint32_t kPatch = 4096;       // LDS bytes in which a wave's half visit is completed

struct PlanesMember {
  grf_planes p;
  uint16_t *y;
  const uint16_t *bias;
  float *partials;                   // [splits][activation rows][rows]
  uint32_t ldy, first, blocks_each;  // first workgroup; row blocks a workgroup
  uint32_t parts;                    // workgroups that share a row block's splits, few rows of x
};

struct PlanesGroup {
  PlanesMember m[kMaxMembers];
  uint32_t n;
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
  uint32_t row_bytes, chunk_bytes, m_rows, cols, packed;  // bytes from a row to the next, from eight columns to the next
};

// Where a quarter of a visit, 64 columns, of x lies in LDS.  Copy i is eight rows, a line each: lane l brings sixteen bytes of row l / 8,
// and which of the eight is turned by the row, so that the operand reads meet no bank twice.  (Sixteen rows a copy, in operand
// order, are an access of its own a lane: TCP 92 accesses a KiB where lines take 16.)  Packed activations are in operand order as they are.
struct XPlaces {
  uint32_t first, second;  // the lane's operands of the two steps
  uint32_t packed, rows, lane;
  __device__ __forceinline__ XPlaces(const PlanesX &x, uint32_t l) : packed(x.packed), rows(x.m_rows), lane(l) {
    const uint32_t r = l % 16, q = l / 16;
    first = packed ? l * 16 : r * 128 + (q ^ r % 8) * 16;
    second = packed ? first + 1024 : first ^ 64;
  }
  __device__ __forceinline__ void source(uint32_t i, uint32_t &row, uint32_t &chunk) const {
    row = min(packed ? i / 2 * 16 + lane % 16 : i * 8 + lane / 8, rows - 1);
    chunk = packed ? i % 2 * 4 + lane / 16 : (lane % 8) ^ (lane / 8);
  }
};

// Sixteen bytes a lane from base + from straight to LDS, lane l's at `to` + 16 l (the compiler would let every LDS read wait
// for all copies that it knows of), when the wave's reads there are done.
__device__ __forceinline__ void copy_to_lds(const uint8_t *base, uint32_t from, uint32_t to) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(from), "s"(base), "s"(to) : "m0", "memory");
#else
  (void)base, (void)from, (void)to;
#endif
}

// All but the wave's last LEFT loads are answered; its LDS operations are done as well, and the workgroup's waves here.
template <int LEFT>
__device__ __forceinline__ void wait_for_loads() {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LEFT) : "memory");
#endif
}

template <int LEFT>
__device__ __forceinline__ void meet_after_loads() {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LEFT) : "memory");
#endif
}

constexpr uint32_t kUnits = 256;  // the chip's compute units
constexpr uint32_t kLdsBytes = 160 * 1024;  // of one of them

// LDS of a wave that has its own x.
template <int HR>
struct Product {
  static constexpr uint32_t kRing = HR == 4 ? 3 : 4;            // quarters of a visit of x
  static constexpr uint32_t kFirst = kRing * HR * 1024 + 2048;  // before it a quarter's words, there the sums of the first split of two
  static constexpr uint32_t kWaveBytes = kFirst + (HR + 1) / 2 * 1024;
};

// Few rows of x, HR eights of them.  A workgroup's waves share out the visits of
// `blocks_each` row blocks, a split or two a wave, and the splits' sums are added in their order: what a row of x gives depends on nothing
// but the matrix's sizes, so all row counts, single and grouped launches agree bit for bit.  A wave brings its own x into LDS,
// a quarter of a visit at a time and two or three ahead (a ring), and meets no other wave until its sums are there.  One row is
// bound by memory (17408 x 5120 twice 5.0 TB/s), more by the lines of x that every wave reads; us with x read where it is, in operand
// order, and now: one row of 5120 x 17408 37 and 34, 16 of 6144, 1024 and 1024 x 5120 21 and 18, of 17408 x 5120 twice 73 and 65.
template <int HR>
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(4))) void planes_product_kernel(PlanesGroup g, PlanesX x) {
  extern __shared__ __align__(16) uint8_t lds[];  // (all of the kernel's: copies go by absolute address)
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int MT = (HR + 1) / 2;
  constexpr uint32_t kQuarterX = HR * 1024, kWave = Product<HR>::kWaveBytes, kRing = Product<HR>::kRing, kAhead = kRing - 1;
  const uint32_t lane = threadIdx.x % 64, wave = scalar(threadIdx.x / 64);
  uint32_t i = 0;
  while (i + 1 < g.n && blockIdx.x >= g.m[i + 1].first) ++i;
  const PlanesMember &m = g.m[i];
  const uint32_t splits = m.p.splits, waves = blockDim.x / 64;
  const uint32_t at_once = splits > waves ? (splits + 1) / 2 : splits, sub = wave / at_once;  // (a wave has one split or two)
  const uint32_t blocks = (m.p.rows + 15) / 16, in_parts = m.parts > 1;
  const uint32_t block = in_parts ? (blockIdx.x - m.first) % blocks : (blockIdx.x - m.first) * m.blocks_each + sub;
  const grf::PlanesShape shape(x.cols);
  const uint32_t each = (shape.visits() + splits - 1) / splits;
  const bool works = in_parts || (sub < m.blocks_each && block < blocks);
  const uint32_t split0 = in_parts ? (blockIdx.x - m.first) / blocks * waves + wave : wave % at_once;
  const uint32_t next_split = in_parts ? splits : at_once;
  float4v acc[MT] = {};
  float4v *const before = reinterpret_cast<float4v *>(lds + wave * kWave + Product<HR>::kFirst) + lane;
  for (uint32_t split = split0; works && split < splits; split += next_split) {
#pragma unroll
    for (int j = 0; j < MT; ++j) before[j * 64] = acc[j], acc[j] = (float4v){};
    const uint32_t v0 = min(split * each, shape.visits()), v1 = min(v0 + each, shape.visits()), full = min(v1, shape.full);
    const uint32_t q = lane / 16, r = lane % 16, slot = r * 4 + q, at_wave = wave * kWave;
    uint8_t *const own = lds + at_wave, *const patch = own + kRing * kQuarterX;
    const uint8_t *at = m.p.planes + (size_t)block * shape.block_bytes();
    const uint32_t base = m.p.bases[block * 16 + r];
    const uint32_t ends = m.p.listed_at[block * shape.visits() + min(v0 + lane, shape.visits())];  // (of up to 63 visits)
    auto end_of = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane(ends, min(v, v1) - v0); };
    auto first_listed = [&](uint32_t v) {  // (the list ends with an entry that nobody owns)
      const uint32_t from = end_of(v), count = end_of(v + 1) - from;
      return m.p.listed[from + min(lane, count ? count - 1 : 0)];
    };
    const XPlaces places(x, lane);
    uint32_t xr[HR];  // (up to 31 rows of 2^25 bytes)
#pragma unroll
    for (int k = 0; k < HR; ++k) {
      uint32_t row, chunk;
      places.source(k, row, chunk);
      xr[k] = row * x.row_bytes + chunk * x.chunk_bytes;
    }
    auto copy_x = [&](uint32_t quarter) {  // 64 columns
      const uint8_t *from = x.data + (size_t)(quarter * 8) * x.chunk_bytes;
#pragma unroll
      for (int k = 0; k < HR; ++k) copy_to_lds(from, xr[k], at_wave + quarter % kRing * kQuarterX + k * 1024);
    };
    auto complete = [&](uint32_t(&o)[2][4], auto &&put) {
      uint4v *words = reinterpret_cast<uint4v *>(patch);
#pragma unroll
      for (int t = 0; t < 2; ++t) words[t * 64 + lane] = (uint4v){o[t][0], o[t][1], o[t][2], o[t][3]};
      wave_order();
      put();
      wave_order();
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const uint4v w = words[t * 64 + lane];
        o[t][0] = w[0], o[t][1] = w[1], o[t][2] = w[2], o[t][3] = w[3];
      }
      wave_order();
    };
    auto multiply = [&](const uint32_t(&o)[2][4], uint32_t quarter) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < MT; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4v *>(own + quarter * kQuarterX + j * 2048 + (t ? places.second : places.first))),
              __builtin_bit_cast(bf16x8_t, (uint4v){o[t][0], o[t][1], o[t][2], o[t][3]}), acc[j], 0, 0, 0);
    };

    if (v0 < full) {
      // A visit's words are asked for a visit ahead, each as soon as the register is free that they come into.
      const VisitBytes bytes(at, full);
      const uint32_t end = full * 4;  // quarters
      Visit now;
#pragma unroll
      for (uint32_t k = 0; k < kAhead; ++k) copy_x(v0 * 4 + k);
      now.load(bytes, v0, slot);
      uint32_t entry = first_listed(v0);
      for (uint32_t v = v0; v < full; ++v) {
        Exponents next;
        uint32_t next_entry;
        const uint32_t from = end_of(v), count = end_of(v + 1) - from;
        auto quarter = [&](auto which) {
          constexpr int Q = decltype(which)::value;
          const uint32_t h = 4 * v + Q;
          if (h + kAhead < end) copy_x(h + kAhead);
          if constexpr (Q == 0) next.load(bytes, v + 1, slot), next_entry = first_listed(v + 1);
          uint32_t o[2][4];
          now.step<2 * Q>(base, o[0]);
          now.step<2 * Q + 1>(base, o[1]);
          now.load_signs(bytes, v + 1, Q, slot);
          if (count) complete(o, [&] { Listed{m.p.listed, from, count, entry}.patch<Q * 1024, 1024>(patch, lane); });
          // This quarter's x was asked for kAhead quarters ago: since then as many more (at the end, none) and the words
          // of these quarters and this one, four or one load each.
          constexpr int kAfter = kAhead == 3 ? 7 : Q == 3 ? 3 : 6;
          if (h + kAhead < end) wait_for_loads<kAfter + kAhead * HR>();
          else wait_for_loads<kAfter>();
          multiply(o, h % kRing);
        };
        quarter(std::integral_constant<int, 0>{});
        quarter(std::integral_constant<int, 1>{});
        quarter(std::integral_constant<int, 2>{});
        quarter(std::integral_constant<int, 3>{});
        now.e = next, entry = next_entry;
      }
    }
    if (v0 < v1 && v1 > shape.full) {  // the shorter visit, a unit at a time; zeros in x's columns past the last one
      const uint32_t from = end_of(shape.full), count = end_of(shape.full + 1) - from;
      for (uint32_t u = 0; u < shape.units; ++u) {
#pragma unroll
        for (int k = 0; k < HR; ++k) {
          uint32_t row, chunk;
          places.source(k, row, chunk);
          chunk += shape.full * 32 + u * 8;
          uint4v one = {0, 0, 0, 0};
          if (chunk * 8 < x.cols) one = *reinterpret_cast<const uint4v *>(x.data + (size_t)row * x.row_bytes + (size_t)chunk * x.chunk_bytes);
          reinterpret_cast<uint4v *>(own)[k * 64 + lane] = one;
        }
        ShortVisit now;
        now.load(at + shape.full * grf::kVisitBytes + u * grf::kUnitBytes, slot);
        uint32_t o[2][4];
        now.step<0>(base, o[0]);
        now.step<1>(base, o[1]);
        complete(o, [&] {
          for (uint32_t k = lane; k < count; k += 64) {
            const uint32_t mine = m.p.listed[from + k];
            if ((mine >> 16) / 1024 == u) *reinterpret_cast<uint16_t *>(patch + (mine >> 16) % 1024 * 2) = (uint16_t)mine;
          }
        });
        multiply(o, 0);
        wave_order();
      }
    }
  }
  if (in_parts) {  // (uniform) the sums are added by a launch of their own
    const uint32_t row = block * 16 + lane % 16;
    if (split0 >= splits || row >= m.p.rows) return;
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t xrow = j * 16 + lane / 16 * 4 + k;
        if (xrow < x.m_rows) m.partials[((size_t)split0 * x.m_rows + xrow) * m.p.rows + row] = acc[j][k];
      }
    return;
  }
  const bool two = works && split0 + at_once < splits;
  float4v first[MT];
#pragma unroll
  for (int j = 0; j < MT; ++j) first[j] = two ? before[j * 64] : acc[j];
  __syncthreads();  // x, words and sums of all waves are read
  float4v *sums = reinterpret_cast<float4v *>(lds);
  if (works) {
#pragma unroll
    for (int j = 0; j < MT; ++j) {
      sums[((sub * splits + split0) * MT + j) * 64 + lane] = first[j];
      if (two) sums[((sub * splits + split0 + at_once) * MT + j) * 64 + lane] = acc[j];
    }
  }
  __syncthreads();
  // Four activation rows of one weight row at a time: the waves' sums in their order, the bias, one rounding.
  for (uint32_t t = threadIdx.x; t < m.blocks_each * MT * 64; t += blockDim.x) {
    const uint32_t l = t % 64, j = t / 64 % MT, s = t / (64 * MT);
    const uint32_t row = ((blockIdx.x - m.first) * m.blocks_each + s) * 16 + l % 16, m0 = j * 16 + l / 16 * 4;
    if (row >= m.p.rows || m0 >= x.m_rows) continue;
    const float4v *from = sums + (s * splits * MT + j) * 64 + l;
    float4v sum = *from;
    for (uint32_t w = 1; w < splits; ++w) sum += from[w * MT * 64];
    const float b = m.bias ? __uint_as_float((uint32_t)m.bias[row] << 16) : 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (m0 + k < x.m_rows) m.y[(size_t)(m0 + k) * m.ldy + row] = round_bf16(m.bias ? sum[k] + b : sum[k]);
  }
#else
  (void)g, (void)x, (void)lds;
#endif
}

// More rows of x: a wave has two row blocks and one split of their visits, W waves share the split's x, and an operand that
// is read meets both blocks.  What bounds it, besides memory, is how evenly the workgroups fall on the compute units (product()
// chooses W; 64 rows of 17408 x 5120 twice 84 us with four waves, 75 with three) and how far ahead the words are asked for: a
// wave's loads are answered in order, so whatever it waits for ends the waits for all before.  x therefore goes past the
// registers, straight into LDS, a quarter of a visit at a time and three ahead (a ring of four), words come a visit ahead,
// each as soon as the register is free that they come into, and between a copy of x and its use lie exactly the loads
// that kAfter counts, which stay under way.  us for 32 of 6144, 1024 and 1024 x 5120 26 (through registers, one block
// a wave) and 23; 64 of 17408 x 5120 twice 107 and 75, 128 164 and 114; 128 of 5120 x 17408 103 and 59.
constexpr uint32_t kBatchEach = 2;                   // row blocks a wave
constexpr uint32_t kBatchPatch = kBatchEach * 2048;  // LDS bytes in which a wave's quarters of a visit are completed

template <int MT, int W>
__global__ __launch_bounds__(W * 64) __attribute__((amdgpu_waves_per_eu(MT == 8 ? 2 : MT == 4 ? 3 : 4))) void planes_batch_kernel(
    PlanesGroup g, PlanesX x) {
  extern __shared__ __align__(16) uint8_t lds[];  // (all of the kernel's: copies go by absolute address)
#if defined(__HIP_DEVICE_COMPILE__)
  constexpr int kCopies = (2 * MT + W - 1) / W;  // of 1 KiB that a wave makes a quarter (some twice where W does not divide them)
  constexpr uint32_t kQuarterX = 2 * MT * 1024;
  const uint32_t lane = threadIdx.x % 64, own = scalar(threadIdx.x / 64);
  uint32_t i = 0;
  while (i + 1 < g.n && blockIdx.x >= g.m[i + 1].first) ++i;
  const PlanesMember &m = g.m[i];
  const grf::PlanesShape shape(x.cols);
  const uint32_t blocks = (m.p.rows + 15) / 16, groups = (blocks + (W * kBatchEach) - 1) / (W * kBatchEach);
  const uint32_t split = (blockIdx.x - m.first) / groups, wanted = (blockIdx.x - m.first) % groups * (W * kBatchEach) + own * kBatchEach;
  const uint32_t each = (shape.visits() + m.p.splits - 1) / m.p.splits;
  const uint32_t v0 = split * each, v1 = min(v0 + each, shape.visits()), full = min(v1, shape.full);
  const uint32_t q = lane / 16, r = lane % 16, slot = r * 4 + q;
  uint8_t *const patch = lds + 4 * kQuarterX + own * kBatchPatch;

  const XPlaces places(x, lane);
  uint32_t xr[kCopies];  // (up to 127 rows of 2^25 bytes)
#pragma unroll
  for (int k = 0; k < kCopies; ++k) {
    uint32_t row, chunk;
    places.source((own + W * k) % (2 * MT), row, chunk);
    xr[k] = row * x.row_bytes + chunk * x.chunk_bytes;
  }
  auto copy_x = [&](uint32_t quarter) {  // 64 columns
    const uint8_t *from = x.data + (size_t)(quarter * 8) * x.chunk_bytes;
#pragma unroll
    for (int k = 0; k < kCopies; ++k) copy_to_lds(from, xr[k], quarter % 4 * kQuarterX + (own + W * k) % (2 * MT) * 1024);
  };

  // (a wave without a block reads the last one's list, no planes, and waits like the rest)
  const uint8_t *at[kBatchEach];
  uint32_t base[kBatchEach], ends[kBatchEach];
#pragma unroll
  for (uint32_t b = 0; b < kBatchEach; ++b) {
    const uint32_t block = min(wanted + b, blocks - 1);
    at[b] = m.p.planes + (size_t)block * shape.block_bytes();
    base[b] = m.p.bases[block * 16 + r];
    ends[b] = m.p.listed_at[block * shape.visits() + min(v0 + lane, shape.visits())];  // (of up to 63 visits)
  }
  auto end_of = [&](uint32_t b, uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane(ends[b], min(v, v1) - v0); };
  auto first_listed = [&](uint32_t b, uint32_t v) {  // (the list ends with an entry that nobody owns)
    const uint32_t from = end_of(b, v), count = end_of(b, v + 1) - from;
    return m.p.listed[from + min(lane, count ? count - 1 : 0)];
  };
  // The words of two steps with those of the list that belong there, which `put` writes.
  auto complete = [&](uint32_t(&o)[kBatchEach][2][4], auto &&put) {
    uint4v *words = reinterpret_cast<uint4v *>(patch);
#pragma unroll
    for (uint32_t b = 0; b < kBatchEach; ++b)
#pragma unroll
      for (int t = 0; t < 2; ++t) words[(b * 2 + t) * 64 + lane] = (uint4v){o[b][t][0], o[b][t][1], o[b][t][2], o[b][t][3]};
    wave_order();
#pragma unroll
    for (uint32_t b = 0; b < kBatchEach; ++b) put(b, patch + b * 2048);
    wave_order();
#pragma unroll
    for (uint32_t b = 0; b < kBatchEach; ++b)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const uint4v w = words[(b * 2 + t) * 64 + lane];
        o[b][t][0] = w[0], o[b][t][1] = w[1], o[b][t][2] = w[2], o[b][t][3] = w[3];
      }
    wave_order();
  };

  float4v acc[kBatchEach][MT] = {};
  auto multiply = [&](const uint32_t(&o)[kBatchEach][2][4], uint32_t quarter) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        const bf16x8_t a = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const uint4v *>(lds + quarter * kQuarterX + j * 2048 + (t ? places.second : places.first)));
#pragma unroll
        for (uint32_t b = 0; b < kBatchEach; ++b)
          acc[b][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              a, __builtin_bit_cast(bf16x8_t, (uint4v){o[b][t][0], o[b][t][1], o[b][t][2], o[b][t][3]}), acc[b][j], 0, 0, 0);
      }
  };

  if (v0 < full) {
    const VisitBytes bytes[kBatchEach] = {{at[0], wanted < blocks ? full : 0}, {at[1], wanted + 1 < blocks ? full : 0}};
    const uint32_t end = full * 4;  // quarters
    Visit now[kBatchEach];
    uint32_t entry[kBatchEach];
    copy_x(v0 * 4), copy_x(v0 * 4 + 1), copy_x(v0 * 4 + 2);
#pragma unroll
    for (uint32_t b = 0; b < kBatchEach; ++b) now[b].load(bytes[b], v0, slot), entry[b] = first_listed(b, v0);
    meet_after_loads<2 * kCopies + kBatchEach * 7>();
    for (uint32_t v = v0; v < full; ++v) {
      Exponents next[kBatchEach];
      uint32_t from[kBatchEach], count[kBatchEach], next_entry[kBatchEach];
#pragma unroll
      for (uint32_t b = 0; b < kBatchEach; ++b) from[b] = end_of(b, v), count[b] = end_of(b, v + 1) - from[b];
      auto quarter = [&](auto which) {
        constexpr int Q = decltype(which)::value;
        const uint32_t h = 4 * v + Q;
        if (h + 3 < end) copy_x(h + 3);
        if constexpr (Q == 0) {
#pragma unroll
          for (uint32_t b = 0; b < kBatchEach; ++b) next[b].load(bytes[b], v + 1, slot), next_entry[b] = first_listed(b, v + 1);
        }
        uint32_t o[kBatchEach][2][4];
#pragma unroll
        for (uint32_t b = 0; b < kBatchEach; ++b) {
          now[b].template step<2 * Q>(base[b], o[b][0]);
          now[b].template step<2 * Q + 1>(base[b], o[b][1]);
          now[b].load_signs(bytes[b], v + 1, Q, slot);
        }
        if (count[0] | count[1])
          complete(o, [&](uint32_t b, uint8_t *there) { Listed{m.p.listed, from[b], count[b], entry[b]}.patch<Q * 1024, 1024>(there, lane); });
        multiply(o, Q);
        // The next quarter's x was asked for two quarters ago: since then two (here and below, at the end, none) more of x,
        // this quarter's words and the two quarters' before, four or one load a block each.
        constexpr int kAfter = kBatchEach * (Q == 3 ? 3 : 6);
        if (h + 3 < end) meet_after_loads<kAfter + 2 * kCopies>();
        else meet_after_loads<kAfter>();
      };
      quarter(std::integral_constant<int, 0>{});
      quarter(std::integral_constant<int, 1>{});
      quarter(std::integral_constant<int, 2>{});
      quarter(std::integral_constant<int, 3>{});
#pragma unroll
      for (uint32_t b = 0; b < kBatchEach; ++b) now[b].e = next[b], entry[b] = next_entry[b];
    }
  }
  if (v1 > shape.full) {  // the shorter visit: x in the ring's place, zeros in columns past the last one, then a unit at a time
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the loop's copies were waited for, but for the last barrier's)
    for (uint32_t k = own; k < 2 * shape.units * MT; k += W) {
      uint32_t row, chunk;
      places.source(k % (2 * MT), row, chunk);
      chunk += shape.full * 32 + k / (2 * MT) * 8;
      uint4v one = {0, 0, 0, 0};
      if (chunk * 8 < x.cols) one = *reinterpret_cast<const uint4v *>(x.data + (size_t)row * x.row_bytes + (size_t)chunk * x.chunk_bytes);
      reinterpret_cast<uint4v *>(lds)[k * 64 + lane] = one;
    }
    __syncthreads();
    uint32_t from[kBatchEach], count[kBatchEach];
#pragma unroll
    for (uint32_t b = 0; b < kBatchEach; ++b) from[b] = end_of(b, shape.full), count[b] = end_of(b, shape.full + 1) - from[b];
    for (uint32_t u = 0; u < shape.units; ++u) {
      uint32_t o[kBatchEach][2][4];
#pragma unroll
      for (uint32_t b = 0; b < kBatchEach; ++b) {
        ShortVisit one;
        one.load(at[b] + shape.full * grf::kVisitBytes + u * grf::kUnitBytes, slot);
        one.step<0>(base[b], o[b][0]);
        one.step<1>(base[b], o[b][1]);
      }
      complete(o, [&](uint32_t b, uint8_t *there) {
        for (uint32_t k = lane; k < count[b]; k += 64) {
          const uint32_t mine = m.p.listed[from[b] + k];
          if ((mine >> 16) / 1024 == u) *reinterpret_cast<uint16_t *>(there + (mine >> 16) % 1024 * 2) = (uint16_t)mine;
        }
      });
      multiply(o, u);
    }
  }
#pragma unroll
  for (uint32_t b = 0; b < kBatchEach; ++b) {
    const uint32_t row = (wanted + b) * 16 + r;
    if (row >= m.p.rows) continue;
    const float added = m.bias ? __uint_as_float((uint32_t)m.bias[row] << 16) : 0.0f;
#pragma unroll
    for (int j = 0; j < MT; ++j)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t xrow = j * 16 + q * 4 + k;
        if (xrow >= x.m_rows) continue;
        if (m.p.splits > 1)
          m.partials[((size_t)split * x.m_rows + xrow) * m.p.rows + row] = acc[b][j][k];
        else
          m.y[(size_t)xrow * m.ldy + row] = round_bf16(m.bias ? acc[b][j][k] + added : acc[b][j][k]);
      }
  }
#else
  (void)g, (void)x, (void)lds;
#endif
}

// The splits' sums of a batch's members in order, the bias, one rounding.  A thread has N rows of W.
template <int N>
__global__ __launch_bounds__(256) void planes_sum_kernel(PlanesGroup g, uint32_t m_rows) {
  typedef float floats __attribute__((ext_vector_type(N)));
  typedef uint16_t halves __attribute__((ext_vector_type(N)));
  uint32_t i = 0;
  while (i + 1 < g.n && blockIdx.x >= g.m[i + 1].first) ++i;
  const PlanesMember &m = g.m[i];
  const uint32_t columns = (m.p.rows + 256 * N - 1) / (256 * N), at = blockIdx.x - m.first;
  const uint32_t row = (at % columns * 256 + threadIdx.x) * N, xrow = at / columns;
  if (row >= m.p.rows) return;
  const float *from = m.partials + (size_t)xrow * m.p.rows + row;
  const size_t pitch = (size_t)m_rows * m.p.rows;
  floats sum = *reinterpret_cast<const floats *>(from);
  for (uint32_t k = 1; k < m.p.splits; ++k) sum += *reinterpret_cast<const floats *>(from + k * pitch);
  halves out;
#pragma unroll
  for (int k = 0; k < N; ++k) out[k] = round_bf16(m.bias ? sum[k] + __uint_as_float((uint32_t)m.bias[row + k] << 16) : sum[k]);
  *reinterpret_cast<halves *>(m.y + (size_t)xrow * m.ldy + row) = out;
}

template <int MT, int W>
int launch_batch_w(const PlanesGroup &g, const PlanesX &x, uint32_t grid, hipStream_t s) {
  constexpr auto kernel = &planes_batch_kernel<MT, W>;
  constexpr uint32_t kBytes = 8 * MT * 1024 + W * kBatchPatch;
  if (kBytes > 64 * 1024)
    if (int rc = grf::allow_full_lds<kernel>()) return rc;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(W * 64), kBytes, s, g, x);
  return GRF_OK;
}
template <int MT>
int launch_batch(const PlanesGroup &g, const PlanesX &x, uint32_t waves, uint32_t grid, hipStream_t s) {
  return waves == 3 ? launch_batch_w<MT, 3>(g, x, grid, s) : launch_batch_w<MT, 4>(g, x, grid, s);
}

template <int HR>
int launch_product(const PlanesGroup &g, const PlanesX &x, uint32_t waves, uint32_t grid, hipStream_t s) {
  constexpr auto kernel = &planes_product_kernel<HR>;
  const uint32_t bytes = waves * Product<HR>::kWaveBytes;
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
  if (!each || p->splits > 16 || each > 63 || each * (p->splits - 1) >= shape.visits())
    return grf::set_error(GRF_BAD_ARGUMENT, std::string(who) + ": 1 to 16 splits of 1 to 63 visits each");
  return GRF_OK;
}

// fp32 sums of all splits for `m` rows, and those that a launch of `m` rows of n members has to have room for, in bytes.
size_t sums_bytes(const grf_planes &p, uint32_t m) { return ((size_t)p.splits * m * p.rows * 4 + 255) / 256 * 256; }
size_t partial_bytes(const grf_planes &p, uint32_t m) { return m > kOwnAlways && p.splits > 1 ? sums_bytes(p, m) : 0; }

// Workgroups that share the splits of a row block where few rows of x meet a matrix alone.  Whole row blocks fall unevenly on the units:
// of 320 blocks some have two and most one, and the last of 5120 x 17408 ends after 136 visits where 85 are a unit's share (256
// blocks of these 23 us, 320 36).  Four workgroups of three splits a block leave the busiest 90 and cost a launch that adds the sums: us,
// one row and six of 5120 x 17408 35.8 37.0, in parts 33.9 33.7; of 4200 x 17408 32.9 35.2, 32.6 32.5.  Of fewer blocks than units each has
// one, and wide matrices end sooner in parts because a block's visits are shared out: 512 x 32768 24.6 27.9, 21.2 22.0.
// It pays from a number of visits saved on: 40 where blocks are more than units (5120 x 14336, 45: 30.2 31.7, 29.0 29.6; 6144 x 17408, 28: 35.3 whole,
// 36.9 in parts).  Else 50 (48: 1600 x 24576 21.4 24.2, 23.0 22.5; 50: 1024 x 17408 16.8 18.5, 17.1 17.6; 55: 512 x 17408 16.5 18.0, 16.0 16.7;
// 40: 512 x 12800 11.7 12.0, 13.0 13.6; 1600 x 17408 17.4 19.2, 19.3 19.5), and for more than eight rows, whose visits are
// longer, 44 (16 rows: 40: 512 x 12800 13.0, 14.3; 44: 400 x 14336 14.4, 14.3; 50: 1024 x 17408 23.0, 18.6), or 40 of more
// than 32 blocks (720 x 12800 17.2, 15.5; 1600 x 17408 23.5, 20.3).
uint32_t own_parts(const grf_planes &p, uint32_t m) {
  const uint64_t blocks = (p.rows + 15) / 16, visits = grf::PlanesShape(p.cols).visits(), each = (visits + p.splits - 1) / p.splits;
  const uint64_t saved = blocks > kUnits || (m > 8 && blocks > 32) ? 40 : m > 8 ? 44 : 50;
  uint32_t best = 1;
  uint64_t least = (blocks + kUnits - 1) / kUnits * each * p.splits;
  least = least > saved ? least - saved + 1 : 0;  // to be below
  for (uint32_t waves = p.splits - 1; waves >= 3; --waves) {
    const uint64_t parts = (p.splits + waves - 1) / waves, busiest = (blocks * parts + kUnits - 1) / kUnits * waves * each;
    if (busiest < least) least = busiest, best = (uint32_t)parts;
  }
  return best;
}

int product(const char *who, uint32_t n, const grf_planes *const *planes, const uint16_t *x, uint32_t ldx, uint32_t m_rows, bool packed,
            uint16_t *const *y, const uint32_t *ldy, const uint16_t *const *bias, void *workspace, size_t workspace_bytes, hipStream_t s) {
  if (!n || n > kMaxMembers || !planes || !x || !y || !ldy) return grf::set_error(GRF_BAD_ARGUMENT, std::string(who) + ": null argument or member count");
  PlanesGroup g{};
  g.n = n;
  uint32_t waves = 1, longest = 0;
  uint64_t visits = 0;
  size_t space = 0;
  const uint32_t cols = planes[0] ? planes[0]->cols : 0, most = std::min(m_rows, kMaxTileRows);
  for (uint32_t i = 0; i < n; ++i) {
    if (int rc = check_planes(who, planes[i])) return rc;
    if (!y[i] || ldy[i] < planes[i]->rows || planes[i]->cols != cols)
      return grf::set_error(GRF_BAD_ARGUMENT, std::string(who) + ": output rows or member widths");
    if (planes[i]->rows > longest) {
      longest = planes[i]->rows, waves = planes[i]->splits;
      if (waves > 8 && longest > 16 * kUnits) waves = (waves + 1) / 2;  // (some units get two workgroups: one row of 5120 x 17408 37 us, 34)
    }
    visits += (uint64_t)((planes[i]->rows + 15) / 16) * grf::PlanesShape(cols).visits();
    g.m[i] = {*planes[i], y[i], bias ? bias[i] : nullptr, reinterpret_cast<float *>(static_cast<uint8_t *>(workspace) + space), ldy[i], 0, 0};
    space += partial_bytes(*planes[i], most);
  }
  for (uint32_t i = 0; i < n; ++i) waves = std::max(waves, (planes[i]->splits + 1) / 2);  // the largest member's, and no wave more than two
  uint32_t own_groups = 0, each = 0;  // workgroups of waves with their own x, and the most visits of a split
  for (uint32_t i = 0; i < n; ++i) {
    const uint32_t blocks = (planes[i]->rows + 15) / 16, blocks_each = std::max(1u, waves / planes[i]->splits);
    own_groups += (blocks + blocks_each - 1) / blocks_each;
    each = std::max(each, (grf::PlanesShape(cols).visits() + planes[i]->splits - 1) / planes[i]->splits);
  }
  if (((uintptr_t)x & 15) || (!packed && (ldx < cols || ldx % 8 || ldx > 1u << 24)) || (packed && m_rows > kMaxTileRows))
    return grf::set_error(GRF_BAD_ARGUMENT, std::string(who) + ": activation rows are 16-byte aligned");
  if (space && (!workspace || workspace_bytes < space || ((uintptr_t)workspace & 15)))
    return grf::set_error(GRF_BAD_ARGUMENT, std::string(who) + ": workspace too small (grf_planes_workspace_bytes)");
  for (uint32_t done = 0; done < m_rows; done += kMaxTileRows) {
    const uint32_t m = std::min(kMaxTileRows, m_rows - done), m_pad = 16 * grf::gemm_tiles(m);
    const bool alone = m > 16 && waves * Product<4>::kWaveBytes > kLdsBytes / 2;  // (a workgroup on its unit)
    const bool batch = m > kOwnRows || (m > kOwnAlways && visits >= kOwnVisits) || (alone && own_groups > kUnits && each > 1) ||
                       (m > 16 && waves * Product<4>::kWaveBytes > kLdsBytes);
    // (rows that need no workspace use one that is there and aligned)
    const bool room = workspace && !((uintptr_t)workspace & 15) && workspace_bytes >= sums_bytes(*planes[0], m);
    const uint32_t parts = batch || n > 1 || !room ? 1 : own_parts(*planes[0], m);
    // (fifteen or sixteen waves with two eights of rows do not fit in a unit's LDS; eight have the splits two each)
    const uint32_t own_waves = parts > 1 ? (planes[0]->splits + parts - 1) / parts
                               : waves * Product<2>::kWaveBytes > kLdsBytes && (m > 8 || packed) ? 8 : waves;
    const PlanesX rows{reinterpret_cast<const uint8_t *>(x) + (size_t)done * ldx * 2, packed ? 16 : ldx * 2, packed ? m_pad * 16 : 16, m, cols, packed};
    uint32_t grid = 0, batch_waves = 4, busiest = ~0u;
    for (uint32_t w : {4u, 3u}) {  // the visits of a compute unit that has most of them
      uint32_t count = 0;
      for (uint32_t i = 0; i < n; ++i) count += ((g.m[i].p.rows + 15) / 16 + w * kBatchEach - 1) / (w * kBatchEach) * g.m[i].p.splits;
      const uint32_t most = (count + kUnits - 1) / kUnits * w;
      if (most < busiest) busiest = most, batch_waves = w;
    }
    bool split = false;
    for (uint32_t i = 0; i < n; ++i) {
      PlanesMember &one = g.m[i];
      const uint32_t blocks = (one.p.rows + 15) / 16;
      one.blocks_each = batch ? batch_waves * kBatchEach : std::max(1u, own_waves / one.p.splits);
      one.y = y[i] + (size_t)done * ldy[i];
      one.first = grid;
      one.parts = parts;
      grid += parts > 1 ? blocks * parts : (blocks + one.blocks_each - 1) / one.blocks_each * (batch ? one.p.splits : 1);
      split |= parts > 1 || (batch && one.p.splits > 1);
    }
    if (int rc = !batch ? (m <= 8 && !packed ? launch_product<1>(g, rows, own_waves, grid, s)
                           : m <= 16         ? launch_product<2>(g, rows, own_waves, grid, s)
                                             : launch_product<4>(g, rows, own_waves, grid, s))
                 : m <= 16 ? launch_batch<1>(g, rows, batch_waves, grid, s)
                 : m <= 32 ? launch_batch<2>(g, rows, batch_waves, grid, s)
                 : m <= 64 ? launch_batch<4>(g, rows, batch_waves, grid, s)
                           : launch_batch<8>(g, rows, batch_waves, grid, s))
      return rc;
    if (split) {
      PlanesGroup sums{};
      uint32_t each = 4;
      for (uint32_t i = 0; i < n; ++i)
        if ((g.m[i].p.rows | g.m[i].ldy) % 4 || (uintptr_t)g.m[i].y & 7) each = 1;
      grid = 0;
      for (uint32_t i = 0; i < n; ++i)
        if (g.m[i].p.splits > 1) {
          sums.m[sums.n] = g.m[i];
          sums.m[sums.n++].first = grid;
          grid += (g.m[i].p.rows + 256 * each - 1) / (256 * each) * m;
        }
      if (each == 4) hipLaunchKernelGGL(planes_sum_kernel<4>, dim3(grid), dim3(256), 0, s, sums, m);
      else hipLaunchKernelGGL(planes_sum_kernel<1>, dim3(grid), dim3(256), 0, s, sums, m);
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
    if (check_planes("grf_planes_workspace_bytes", planes[i]) == GRF_OK) {  // (what a launch refuses needs none)
      const uint32_t m = std::min(m_rows, kMaxTileRows);
      bytes += n == 1 && own_parts(*planes[i], m) > 1 ? sums_bytes(*planes[i], m) : partial_bytes(*planes[i], m);
    }
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
