// y = x W^T (+ bias) for many rows of x and a W that is resident as planes (word_planes.h), without a dense W in memory.
//
// A decode and a dense product move W three times more (5120 x 17408: 57 us for the decode, where 200 rows' product takes 61).
// Here a workgroup of eight waves makes a tile of 256 of W's rows by TM of x's, in steps of 64 columns (a quarter of a visit), of
// which LDS holds two of W and two of x.  x comes by copies straight to LDS; W's words are made by the wave that has two row blocks'
// planes in registers, asked for two steps ahead, are written to LDS a step ahead, where the listed ones are put over them, and
// are read by all.  The making of a step's words lies between the products of the step before and is done in four pieces, one a slice
// of 16 columns, which is what v_mfma_f32_32x32x16_bf16 takes: operands of 16 columns need half the registers of 32's, and 242 are
// in use (nine more and some spill).  One barrier a step, after which the buffers that all have read are filled again.
//
// Bound by two things that nearly meet: a step's products are 2048 cycles of a unit's four matrix cores, its 256 KiB through LDS as many
// (waves of 128 x 64; of 32 x 256 with W in registers, which each wave makes for itself, 2800).  A lone unit's step takes
// 1.32 us, without the products 1.1; with all units at work 1.8 to 2.0, without the products 1.2.  A sixth of that is the clock, 2.4 GHz for a
// lone unit and 1.95 to 2.02 for all; the rest is 3250 cycles a step that become 3600 to 4000.  By the counters (1000 rows of 5120 x
// 17408) matrix cores are busy 46 % of a launch's cycles, vector ALUs 30, LDS with indexed accesses 29, a fifth of these conflicts,
// and waves wait for something 44 % of theirs.  What was
// measured on the way: places turned by row % 8 rather than row / 2, 42 % of LDS cycles conflicts (thirty-two rows of one
// chunk meet where sixteen of four do not); a branch around the listed words puts a slice's words before its products, 1.45; one
// list a block rather than one a wave 1.40.
#include "dense_device.h"
#include "planes_device.h"

namespace {

using namespace grf;

typedef float float16v __attribute__((ext_vector_type(16)));

constexpr uint32_t kUnits = 256;     // compute units
constexpr uint32_t kTileRows = 256;  // of W that a workgroup takes

// What a lane holds of a block's quarter of a visit, two steps.
struct Quarter {
  uint4v s;
  uint2v e;  // (the last quarter's second is made of what all seven have left)
};

template <int TM>
struct PromptLds {
  static constexpr uint32_t kW = kTileRows * 128, kX = TM * 128;  // bytes of a buffer of 64 columns; two of W, then two of x
  static constexpr uint32_t kNowhere = 2 * kW + 2 * kX, kBytes = kNowhere + 256;
};

// A value that what is made of it is made of anew: sixteen places in LDS in registers would spill others.
__device__ __forceinline__ uint32_t fresh(uint32_t v) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(v));
#endif
  return v;
}

// Waves WN x WM, each 256 / WN of W's rows by TM / WM of x's.
template <int TM, int WM, int WN>
__global__ __launch_bounds__(64 * WM *WN) __attribute__((amdgpu_waves_per_eu(2))) void planes_prompt_kernel(grf_planes p, DenseArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __align__(16) uint8_t lds[];
  typedef __attribute__((address_space(3))) uint4v lds_uint4v;  // (by absolute address: the kernel has no other LDS)
  typedef __attribute__((address_space(3))) uint16_t lds_uint16;
  constexpr int W = WM * WN, NI = kTileRows / WN / 32, MJ = TM / WM / 32, CX = TM / 8 / W;
  constexpr uint32_t kW = PromptLds<TM>::kW, kX = PromptLds<TM>::kX, kEach = kTileRows / 16 / W;  // blocks whose words a wave makes
  static_assert(kEach == 2 && TM % (8 * W) == 0);
  const uint32_t lane = threadIdx.x % 64, wave = scalar(threadIdx.x / 64);
  // Workgroups of one XCD (every eighth) take tiles that follow one another, x's tiles first: they share planes and x in
  // their second-level cache.
  const uint32_t total = a.tiles_m * a.tiles_n * a.parts, xcd = blockIdx.x % 8;
  uint32_t at = xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;
  const uint32_t tm = at % a.tiles_m;
  at /= a.tiles_m;
  const uint32_t tn = at % a.tiles_n, part = at / a.tiles_n;
  const uint32_t m0 = tm * TM, n0 = tn * kTileRows;
  const PlanesShape shape(a.cols);
  const uint32_t v0 = part * a.steps_per_part, v1 = min(v0 + a.steps_per_part, shape.visits()), full = min(v1, shape.full);

  const uint16_t *x0 = a.x + (size_t)m0 * a.ldx;
  const uint64_t x_at = (uint64_t)x0;
  // rows past the last are beyond the buffer: nothing is read, and what comes of them is not stored
  const uint32_t row_bytes = a.ldx * 2, in_tile = min(a.m_rows - m0, (uint32_t)TM);
  const uint4v rx = {(uint32_t)x_at, (uint32_t)(x_at >> 32) & 0xffffu, (in_tile - 1) * row_bytes + a.cols * 2, 0x00020000u};
  const uint32_t chunk = ((lane % 8) ^ (wave % 2 * 4 + lane / 16)) * 16, from_x = (wave * 8 + lane / 8) * row_bytes + chunk;
  auto copy_x = [&](uint32_t buffer, uint32_t step) {
    const uint32_t from = fresh(from_x);
#pragma unroll
    for (int i = 0; i < CX; ++i) copy_to_lds(rx, from + i * W * 8 * row_bytes, step * 128, 2 * kW + buffer * kX + (i * W + wave) * 1024);
  };

  // The wave's two blocks (in place of one past the last the last one, which is not stored there).
  const uint32_t q = lane / 16, r = lane % 16, own = r * 4 + q, blocks = (p.rows + 15) / 16, wanted = n0 / 16 + wave * kEach;
  const uint8_t *bytes_at[kEach];
  uint32_t base[kEach], ends[kEach];
#pragma unroll
  for (uint32_t b = 0; b < kEach; ++b) {
    const uint32_t block = min(wanted + b, blocks - 1);
    bytes_at[b] = p.planes + (size_t)block * shape.block_bytes();
    base[b] = p.bases[block * 16 + r];
    ends[b] = p.listed_at[block * shape.visits() + min(v0 + lane, shape.visits())];  // (of up to 63 visits)
  }
  auto end_of = [&](uint32_t b, uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane(ends[b], min(v, v1) - v0); };
  // Lane l has word l % 32 of block l / 32's list of a visit (the list ends with an entry that nobody owns).
  auto listed = [&](uint32_t v) { return lane / 32 ? end_of(1, v + 1) - end_of(1, v) : end_of(0, v + 1) - end_of(0, v); };
  auto first_listed = [&](uint32_t v) {
    const uint32_t count = listed(v);
    return p.listed[(lane / 32 ? end_of(1, v) : end_of(0, v)) + min(lane % 32, count ? count - 1 : 0)];
  };
  // The quarter a listed word belongs to (7: no word), where in the wave's 32 lines of a buffer, and the word.
  auto placed = [&](uint32_t entry, uint32_t b, bool any) {
    const uint32_t place = entry >> 16, its = place / 8 % 64, row = its % 16;
    const uint32_t to = b * 2048 + row * 128 + ((place / 512 % 2 * 4 + its / 16) ^ row / 2) * 16 + place % 8 * 2;
    return (any ? place / 1024 : 7u) << 29 | to << 16 | (entry & 0xffff);
  };

  // The lane's places: of the words it makes, and of its operands in a slice of 16 columns.
  const uint32_t make = wave * kEach * 2048 + r * 128 + (q ^ r / 2) * 16;  // of the first of two steps; the second's at (that ^ 64)
  const uint32_t wm = wave % WM, wn = wave / WM, l32 = lane % 32, place = ((lane / 32) ^ (lane / 2 % 8)) * 16;
  const uint32_t at_w = (wn * (kTileRows / WN) + l32) * 128 + place, at_x = 2 * kW + (wm * (TM / WM) + l32) * 128 + place;

  float16v acc[NI][MJ] = {};
  struct Operands {
    uint4v w[NI], x[MJ];
  };
  Operands even, odd;
  auto read = [&](Operands &o, uint32_t buffer, uint32_t slice) {
    const uint32_t pw = (fresh(at_w) ^ slice * 32) + buffer * kW, px = (fresh(at_x) ^ slice * 32) + buffer * kX;
#pragma unroll
    for (int j = 0; j < MJ; ++j) o.x[j] = *reinterpret_cast<lds_uint4v *>(px + j * 4096);
#pragma unroll
    for (int i = 0; i < NI; ++i) o.w[i] = *reinterpret_cast<lds_uint4v *>(pw + i * 4096);
  };
  auto multiply = [&](const Operands &o) {
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int j = 0; j < MJ; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, o.w[i]), __builtin_bit_cast(bf16x8_t, o.x[j]), acc[i][j], 0, 0, 0);
  };
  auto keep = [&](const uint32_t(&o)[4], uint32_t b, uint32_t half, uint32_t buffer) {
    *reinterpret_cast<lds_uint4v *>((fresh(make) ^ half * 64) + buffer * kW + b * 2048) = (uint4v){o[0], o[1], o[2], o[3]};
  };

  if (v0 < full) {
    const uint32_t first = v0 * 4, last = full * 4 - 1;  // quarters of visits: 64 columns
    Quarter held[kEach][2];                              // of the next two quarters
    uint32_t left[kEach], entry, next_entry;
    // A lane's share of a quarter (past the last visit, of the last one again: it is not multiplied).
    const uint32_t by16 = own * 16, by12 = own * 12;
    __amdgpu_buffer_rsrc_t planes[kEach];
#pragma unroll
    for (uint32_t b = 0; b < kEach; ++b)
      planes[b] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(bytes_at[b]), 0, (int)(full * kVisitBytes), 0x00020000);
    auto ask = [&](auto which, uint32_t b, uint32_t v) {
      constexpr int Q = decltype(which)::value;
      const uint32_t from = min(v, full - 1) * kVisitBytes;
      Quarter &to = held[b][Q % 2];
      to.s = __builtin_bit_cast(uint4v, __builtin_amdgcn_raw_buffer_load_b128(planes[b], by16, from + Q * 1024, 0));
      if constexpr (Q < 2) to.e = __builtin_bit_cast(uint2v, __builtin_amdgcn_raw_buffer_load_b64(planes[b], by16, from + 4096 + Q * 8, 0));
      else if constexpr (Q == 2) to.e = __builtin_bit_cast(uint2v, __builtin_amdgcn_raw_buffer_load_b64(planes[b], by12, from + 5120, 0));
      else to.e[0] = __builtin_amdgcn_raw_buffer_load_b32(planes[b], by12, from + 5128, 0);
    };
    // Step HALF of a quarter's words of block b, into buffer Q % 2 of W; then what is listed there, and the quarter after next is asked for.
    auto decode = [&](auto which, auto part_of, uint32_t b, uint32_t v) {
      constexpr int Q = decltype(which)::value, HALF = decltype(part_of)::value;
      constexpr uint32_t k = 0x00030003u;
      Quarter &from = held[b][Q % 2];
      uint32_t d = from.e[HALF], o[4];
      constexpr int T = 2 * Q + HALF;
      if constexpr (T == 0) left[b] = (d >> 14) & k;
      else if constexpr (T < 7) left[b] |= (d >> (14 - 2 * T)) & (k << (2 * T));
      else d = left[b];
      join_words(from.s[2 * HALF], from.s[2 * HALF + 1], d & kCodeFields, (d >> 7) & kCodeFields, base[b], o);
      keep(o, b, HALF, Q % 2);
      if constexpr (HALF == 1) {
        if (b == 1) {  // (constant)
          const uint32_t nowhere = PromptLds<TM>::kNowhere + fresh(lane) * 4, there = (entry >> 16 & 4095) + wave * kEach * 2048 + Q % 2 * kW;
          *reinterpret_cast<lds_uint16 *>(entry >> 29 == Q ? there : nowhere) = (uint16_t)entry;
          if constexpr (Q == 3) entry = placed(next_entry, lane / 32, lane % 32 < listed(v + 1));
        }
        ask(std::integral_constant<int, (Q + 2) % 4>{}, b, v + (Q >= 2));
        if (Q == 1 && b == 1) next_entry = first_listed(v + 1);
      }
    };
    // The listed words past the 32 of a block's visit that the lanes hold.
    auto rest = [&](uint32_t quarter, uint32_t v) {
#pragma unroll
      for (uint32_t b = 0; b < kEach; ++b) {
        const uint32_t from = end_of(b, v), count = end_of(b, v + 1) - from;
        for (uint32_t k = 32 + lane; k < count; k += 64) {
          const uint32_t one = placed(p.listed[from + k], b, true);
          if (one >> 29 == quarter) *reinterpret_cast<lds_uint16 *>(wave * kEach * 2048 + quarter % 2 * kW + (one >> 16 & 4095)) = (uint16_t)one;
        }
      }
    };
    auto most = [&](uint32_t v) { return max(end_of(0, v + 1) - end_of(0, v), end_of(1, v + 1) - end_of(1, v)); };
    uint32_t in_list = most(v0);  // of the visit whose words are made
    constexpr std::integral_constant<int, 0> k0{};
    constexpr std::integral_constant<int, 1> k1{};

    copy_x(0, first), copy_x(1, min(first + 1, last));
#pragma unroll
    for (uint32_t b = 0; b < kEach; ++b) {
      ask(k0, b, v0), ask(k1, b, v0);
    }
    entry = placed(first_listed(v0), lane / 32, lane % 32 < listed(v0));
    decode(k0, k0, 0, v0), decode(k0, k1, 0, v0), decode(k0, k0, 1, v0), decode(k0, k1, 1, v0);
    if (in_list > 32) rest(0, v0);
    operands_landed();
    copies_landed_everywhere<0>();
    read(even, 0, 0);
    decode(k1, k0, 0, v0);
    for (uint32_t v = v0; v < full; ++v) {
      auto quarter = [&](auto which) {
        constexpr int Q = decltype(which)::value;
        constexpr std::integral_constant<int, (Q + 1) % 4> next{};
        constexpr std::integral_constant<int, (Q + 2) % 4> after{};
        const uint32_t h = 4 * v + Q, vn = v + (Q == 3), va = v + (Q >= 2);
        read(odd, Q % 2, 1);
        decode(next, k1, 0, vn);
        multiply(even);
        __builtin_amdgcn_sched_barrier(0);
        read(even, Q % 2, 2);
        decode(next, k0, 1, vn);
        multiply(odd);
        __builtin_amdgcn_sched_barrier(0);
        read(odd, Q % 2, 3);
        decode(next, k1, 1, vn);
        multiply(even);
        if (Q == 3) in_list = most(vn);
        if (in_list > 32) rest((Q + 1) % 4, vn);
        operands_landed();  // nothing is read from these buffers any more by this wave, and its words are there ..
        // .. nor by another, and the next quarter's x has landed: since that was asked for came two loads or more of each block's words
        copies_landed_everywhere<2 * kEach>();
        // What is decoded until the next barrier has landed as well, but the compiler, which does not count the copies of x, would
        // wait behind them for loads that were just made: it waits here, for nothing.
#pragma unroll
        for (uint32_t b = 0; b < kEach; ++b) {
          asm volatile("" : "+v"(held[b][Q % 2].s), "+v"(held[b][Q % 2].e));
        }
        if constexpr (Q == 1) asm volatile("" : "+v"(next_entry));
        copy_x(Q % 2, min(h + 2, last));
        read(even, (Q + 1) % 2, 0);
        decode(after, k0, 0, va);
        multiply(odd);
        __builtin_amdgcn_sched_barrier(0);
      };
      quarter(std::integral_constant<int, 0>{});
      quarter(std::integral_constant<int, 1>{});
      quarter(std::integral_constant<int, 2>{});
      quarter(std::integral_constant<int, 3>{});
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  }
  if (v0 < v1 && v1 > shape.full) {  // the shorter visit, a unit at a time; zeros in x's columns past the last one
    for (uint32_t u = 0; u < shape.units; ++u) {
      __syncthreads();
      const uint32_t step = shape.full * 256 + u * 64, column = step * 2 + chunk;
#pragma unroll 1
      for (int i = 0; i < CX; ++i) {
        uint4v one = {0, 0, 0, 0};
        if (column < a.cols * 2 && (uint32_t)(i * W + wave) * 8 + lane / 8 < in_tile)
          one = *reinterpret_cast<const uint4v *>(reinterpret_cast<const uint8_t *>(x0) + from_x + i * W * 8 * row_bytes + step * 2);
        *reinterpret_cast<lds_uint4v *>(2 * kW + (i * W + wave) * 1024 + lane * 16) = one;
      }
#pragma unroll
      for (uint32_t b = 0; b < kEach; ++b) {
        ShortVisit now;
        uint32_t o[4];
        now.load(bytes_at[b] + shape.full * kVisitBytes + u * kUnitBytes, own);
        now.step<0>(base[b], o), keep(o, b, 0, 0);
        now.step<1>(base[b], o), keep(o, b, 1, 0);
        const uint32_t from = end_of(b, shape.full), count = end_of(b, shape.full + 1) - from;
        for (uint32_t k = lane; k < count; k += 64) {
          const uint32_t one = placed(p.listed[from + k], b, true);
          if (one >> 29 == u) *reinterpret_cast<lds_uint16 *>(wave * kEach * 2048 + (one >> 16 & 4095)) = (uint16_t)one;
        }
      }
      __syncthreads();
#pragma unroll 1
      for (uint32_t slice = 0; slice < 4; ++slice) {
        read(even, 0, slice);
        multiply(even);
      }
    }
  }

  // a lane holds columns n .. n + 3 of row m of y, four times a tile of 32 x 32
  const bool fours = a.rows % 4 == 0 && a.ldy % 4 == 0;
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const uint32_t n = n0 + wn * (kTileRows / WN) + i * 32 + g * 8 + lane / 32 * 4;
      if (n >= a.rows) continue;
      float4v bias = {0, 0, 0, 0};
      if (a.bias && a.parts == 1)
        for (int v = 0; v < 4; ++v) bias[v] = __uint_as_float((uint32_t)a.bias[min(n + v, a.rows - 1)] << 16);
#pragma unroll
      for (int j = 0; j < MJ; ++j) {
        const uint32_t m = m0 + wm * (TM / WM) + j * 32 + l32;
        if (m >= a.m_rows) continue;
        float4v sum;
#pragma unroll
        for (int v = 0; v < 4; ++v) sum[v] = acc[i][j][g * 4 + v];
        if (a.parts > 1) {
          *reinterpret_cast<float4v *>(a.partials + ((size_t)part * a.m_rows + m) * sums_pitch(a.rows) + n) = sum;
        } else {
          uint16_t *to = a.y + (size_t)m * a.ldy + n;
          half4v out;
#pragma unroll
          for (int v = 0; v < 4; ++v) out[v] = round_bf16(a.bias ? sum[v] + bias[v] : sum[v]);
          if (fours) *reinterpret_cast<half4v *>(to) = out;
          else
            for (int v = 0; v < 4; ++v)
              if (n + v < a.rows) to[v] = out[v];
        }
      }
    }
#else
  (void)p, (void)a;
#endif
}

// The tiles, and what their launches take (us): one at the start, a step of a lone unit and what it takes more the more units
// are at work, each round of workgroups after the first, each part's sums and what they take a million bytes. Fitted to 2523 launches
// of 300 products (129 to 2048 rows by 256 to 17408 x 512 to 17408), 9 and 10 % off rms; the choice is 0.9 % slower than
// the best measured on average.
struct PromptTile {
  uint32_t m;
  double start, step, busy, round, part, sums;
};
constexpr PromptTile kTiles[] = {{128, 11.3, 0.922, 0.319, 4.15, 0.04, 0.112}, {256, 14.3, 1.341, 0.476, 5.9, 0.015, 0.111}};

struct PromptPlan {
  uint32_t tile = 0, parts = 0, each = 0;  // rows of x a workgroup takes, parts of K, visits a part
  double us = 1e30;
};

uint32_t up(uint32_t v, uint32_t by) { return v / by + (v % by != 0); }

PromptPlan plan_prompt(uint32_t rows, uint32_t cols, uint32_t m_rows) {
  const uint32_t visits = PlanesShape(cols).visits();
  PromptPlan best;
  for (const PromptTile &t : kTiles) {
    const uint64_t tiles = (uint64_t)up(m_rows, t.m) * up(rows, kTileRows);
    for (uint32_t want : {1u, 2u, 3u, (uint32_t)(kUnits / tiles), (uint32_t)(2 * kUnits / tiles), (uint32_t)(3 * kUnits / tiles)}) {
      const uint32_t each = std::min(up(visits, std::max(1u, std::min(want, visits))), 63u), parts = up(visits, each);
      const uint64_t groups = tiles * parts, rounds = (groups + kUnits - 1) / kUnits;
      const double busy = rounds > 1 ? 1.0 : (double)groups / kUnits;
      double us = t.start + (rounds - 1) * (4 * each * (t.step + t.busy) + t.round) + 4 * each * (t.step + t.busy * busy);
      if (parts > 1) us += parts * (t.part + t.sums * 8e-6 * m_rows * rows);
      if (us < best.us) best = PromptPlan{t.m, parts, each, us};
    }
  }
  return best;
}

// Whether the launch is to be preferred to a decode and a dense product: it makes every word once a tile of x's rows where the decode
// makes it once, so the fewer rows the rather (200 rows of 5120 x 17408 123 us and 66, 400 161 and 112, 1000 219 and 192, 1500 of 14355 x 4288 219 and 290).
// The decode takes 0.6 us a million words.  The models are each a tenth off, so it has to be clearly less: of the 300 products 74
// are taken, 1.24 times as fast in the mean, one of them slower (545 rows of 6835 x 3072, 4 %); with 1 and 0 here 163, of which 37 are slower,
// by up to a quarter.
constexpr double kClearly = 0.93, kAtLeast = 0.5;
// The dense model ranks tiles; where that product is what follows a decode and keeps the chip at work for long, it takes longer than the model
// says (1000 rows of 5120 x 17408 162 us for 135, six of 64 to 128 us a sixth more).
constexpr double kWorking = 0.25;

template <int TM, int WM, int WN>
int launch(const grf_planes &p, const DenseArgs &a, hipStream_t s) {
  constexpr auto kernel = &planes_prompt_kernel<TM, WM, WN>;
  if (int rc = allow_full_lds<kernel>()) return rc;
  hipLaunchKernelGGL(kernel, dim3(a.tiles_m * a.tiles_n * a.parts), dim3(64 * WM * WN), PromptLds<TM>::kBytes, s, p, a);
  if (a.parts > 1) hipLaunchKernelGGL(dense_sum_kernel, dim3((a.rows + 1023) / 1024, a.m_rows), dim3(256), 0, s, a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? GRF_OK : set_error(GRF_LAUNCH_FAILED, std::string("grf_planes_prompt: ") + hipGetErrorString(e));
}

constexpr uint32_t kWidest = 1u << 21;  // values from a row of x to the next: a tile's offsets are 31 bits

}  // namespace

extern "C" {

int64_t grf_planes_prompt_plan(uint32_t rows, uint32_t cols, uint32_t m_rows) {
  if (!rows || !cols || cols % 8 || cols > GRF_PLANES_MAX_COLS || m_rows <= 128 || (uint64_t)rows * m_rows > 1u << 30) return -1;
  const PromptPlan p = plan_prompt(rows, cols, m_rows);
  const double decode = std::max(6.5, 3.5 + 0.6e-6 * rows * cols);
  double dense = dense_product_us(rows, cols, m_rows);
  if (grf_dense_gemm_plan(rows, cols, m_rows) >= 0) dense += kWorking * std::max(0.0, dense - 40);
  return p.us < kClearly * (decode + dense) - kAtLeast ? (int64_t)p.parts << 16 | p.tile : -1;
}

size_t grf_planes_prompt_workspace_bytes(uint32_t rows, uint32_t m_rows, uint32_t plan) {
  return plan >> 16 > 1 ? (size_t)(plan >> 16) * m_rows * sums_pitch(rows) * 4 : 0;
}

int grf_planes_prompt(const grf_planes *planes, const uint16_t *x, uint32_t ldx, uint32_t m_rows, uint32_t plan, uint16_t *y,
                      uint32_t ldy, const uint16_t *bias, void *workspace, size_t workspace_bytes, void *hip_stream) {
  auto bad = [](const char *why) { return set_error(GRF_BAD_ARGUMENT, std::string("grf_planes_prompt: ") + why); };
  if (!planes || !x || !y || !planes->planes || !planes->bases || !planes->listed_at || !planes->listed) return bad("null argument");
  const uint32_t rows = planes->rows, cols = planes->cols, visits = PlanesShape(cols).visits(), tile = plan & 0xffff, parts = plan >> 16;
  if (!rows || !cols || cols % 8 || (uintptr_t)planes->planes & 15 || cols > GRF_PLANES_MAX_COLS) return bad("sizes or alignment of the planes");
  if (!m_rows || (uint64_t)m_rows * rows > 1u << 30 || rows > 1u << 28) return bad("rows * m_rows up to 2^30");
  if (ldx < cols || ldx % 8 || ldx > kWidest || ldy < rows || (uintptr_t)x & 15 || (uintptr_t)y & 7) return bad("leading dimension or alignment");
  if (tile != 128 && tile != 256) return bad("tiles are of 128 or 256 rows");
  const uint32_t each = parts ? (visits + parts - 1) / parts : 0;
  if (!each || each > 63 || (uint64_t)each * (parts - 1) >= visits) return bad("parts of 1 to 63 visits");
  if (parts > 1 && (!workspace || (uintptr_t)workspace & 15 || workspace_bytes < grf_planes_prompt_workspace_bytes(rows, m_rows, plan)))
    return bad("workspace missing, misaligned or too small");
  const DenseArgs a{x, nullptr, bias, y, static_cast<float *>(workspace), ldx, m_rows, rows, cols, ldy, (m_rows + tile - 1) / tile,
                    (rows + kTileRows - 1) / kTileRows, parts, each};
  return tile == 256 ? launch<256, 4, 2>(*planes, a, (hipStream_t)hip_stream) : launch<128, 2, 4>(*planes, a, (hipStream_t)hip_stream);
}

}  // extern "C"
