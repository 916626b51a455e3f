// y = x W^T (+ bias) for a dense BF16 W of rows x cols: what a product of more activation rows than the
// fused kernels take does after the matrix has been decoded to a transient.
//
// A workgroup makes a TN x TM tile of W's rows by x's rows, the sum over a part of K, in steps of 64 columns, which
// loads that write LDS directly copy there (a line of 128 bytes a row): BX buffers of x, whose lines the workgroups of an
// XCD share in their second-level cache, and as many or one more of W, which comes from further away.  A wave reads operands of
// v_mfma_f32_16x16x32_bf16 from LDS, the next 32 columns' while it multiplies the ones in hand, and
// keeps its tile in registers.  A row's eight 16-byte chunks lie at (chunk ^ row % 8): the copy leaves the lanes'
// places fixed, so the order is made by which chunk a lane fetches, and the reads of 16 rows then meet no bank twice.
//
// Bound by three things that nearly meet in the tile of 256 x 256: a step's 64 KiB take 0.73 us at the 38 bytes a
// cycle that a compute unit gets from its second-level cache into LDS, its products 0.87 us, its operand reads 0.4;
// together 1.43 us with every unit at work on rows that begin on lines, 1.1 where few are, up to 1.8 where rows begin
// between lines (profiles/dense_tilings.csv; with two buffers of W 1.65 for the 1.43, steps of 32 columns in five buffers 1.7,
// because half a line a row comes at 23 bytes a cycle; lines touched two steps ahead, the copy spread between the
// products, the first buffer given back earlier: no change; four waves of 128 x 128: spills).  1000 rows of
// 5120 x 17408: 159 us, 200 rows 61, where the library takes 250 and 222.
//
// A matrix whose tiles do not fill the GPU is cut along K: part p walks its share of the steps and leaves fp32
// sums in `partials` [parts][m_rows][rows in whole fours], which dense_sum_kernel adds in part order.
#include "dense_device.h"

namespace {

using namespace grf;

// Waves WN x WM, each TN / WN of W's rows by TM / WM of x's.
template <int TM, int TN, int WM, int WN, int BX, int BW>
__global__ __launch_bounds__(64 * WM *WN) void dense_gemm_kernel(DenseArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __align__(16) uint8_t lds[];
  typedef __attribute__((address_space(3))) uint4v lds_uint4v;  // (by absolute address: the kernel has no other LDS)
  constexpr int W = WM * WN, NI = TN / WN / 16, MJ = TM / WM / 16;
  constexpr int CX = TM / 8 / W, CW = TN / 8 / W;  // copies a wave makes a step, eight rows each
  constexpr uint32_t kX = TM * 128, kW = TN * 128;  // bytes of a buffer; BX of x, then BW of W
  static_assert(TM % (8 * W) == 0 && TN % (8 * W) == 0 && NI <= 32 && MJ <= 32);
  const uint32_t lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  // Workgroups of one XCD (every eighth) take tiles that follow one another, x's tiles first: they share rows of W
  // and of x in their second-level cache.
  const uint32_t total = a.tiles_m * a.tiles_n * a.parts, xcd = blockIdx.x % 8;
  uint32_t q = xcd * (total / 8) + min(xcd, total % 8) + blockIdx.x / 8;
  const uint32_t tm = q % a.tiles_m;
  q /= a.tiles_m;
  const uint32_t tn = q % a.tiles_n, part = q / a.tiles_n;
  const uint32_t m0 = tm * TM, n0 = tn * TN;
  const uint32_t steps = (a.cols + kStep - 1) / kStep, first = part * a.steps_per_part;
  const uint32_t past = min(steps, first + a.steps_per_part);
  const bool ragged = past == steps && a.cols % kStep;  // this part ends with fewer columns than a step
  const uint32_t whole = past - first - ragged;

  const uint16_t *x0 = a.x + (size_t)m0 * a.ldx, *w0 = a.w + (size_t)n0 * a.cols;
  auto buffer_at = [](const uint16_t *p) {
    const uint64_t at = (uint64_t)p;
    return (uint4v){(uint32_t)at, (uint32_t)(at >> 32) & 0xffffu, 0x7fffffffu, 0x00020000u};
  };
  const uint4v rx = buffer_at(x0), rw = buffer_at(w0);
  // where the lane copies from; rows past the last read the last one, and what comes of them is not stored
  const uint32_t chunk = ((lane % 8) ^ (lane / 8)) * 16;
  auto from_x = [&](int i) { return min((uint32_t)(i * W + wave) * 8 + lane / 8, a.m_rows - 1 - m0) * a.ldx * 2 + chunk; };
  auto from_w = [&](int i) { return min((uint32_t)(i * W + wave) * 8 + lane / 8, a.rows - 1 - n0) * a.cols * 2 + chunk; };
  uint32_t vx[CX], vw[CW];
#pragma unroll
  for (int i = 0; i < CX; ++i) vx[i] = from_x(i);
#pragma unroll
  for (int i = 0; i < CW; ++i) vw[i] = from_w(i);
  auto copy_x = [&](uint32_t buffer, uint32_t step) {
#pragma unroll
    for (int i = 0; i < CX; ++i) copy_to_lds(rx, vx[i], step * 128, buffer * kX + (i * W + wave) * 1024);
  };
  auto copy_w = [&](uint32_t buffer, uint32_t step) {
#pragma unroll
    for (int i = 0; i < CW; ++i) copy_to_lds(rw, vw[i], step * 128, BX * kX + buffer * kW + (i * W + wave) * 1024);
  };

  const uint32_t wm = wave % WM, wn = wave / WM;
  // the lane's operands of the first 32 columns in the first buffer; those of the other 32 are at (that ^ 64)
  const uint32_t place = ((lane / 16) ^ (lane % 8)) * 16;
  const uint32_t at_x = (wm * (TM / WM) + lane % 16) * 128 + place, at_w = BX * kX + (wn * (TN / WN) + lane % 16) * 128 + place;
  float4v acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j) acc[i][j] = (float4v){0.f, 0.f, 0.f, 0.f};
  uint4v w_a[NI], x_a[MJ], w_b[NI], x_b[MJ];
  auto read_one = [&](auto k, uint4v(&w)[NI], uint4v(&x)[MJ], uint32_t pw, uint32_t px) {
    constexpr int K = decltype(k)::value;
    if constexpr (K < MJ) x[K] = *reinterpret_cast<lds_uint4v *>(px + K * 2048);
    else w[K - MJ] = *reinterpret_cast<lds_uint4v *>(pw + (K - MJ) * 2048);
  };
  auto read = [&](uint4v(&w)[NI], uint4v(&x)[MJ], uint32_t in_w, uint32_t in_x, uint32_t half) {
    const uint32_t pw = (at_w + in_w * kW) ^ half, px = (at_x + in_x * kX) ^ half;
    unrolled<0, NI + MJ>([&](auto k) { read_one(k, w, x, pw, px); });
  };
  auto multiply_one = [&](auto k, const uint4v(&w)[NI], const uint4v(&x)[MJ]) {
    constexpr int i = decltype(k)::value / MJ, j = decltype(k)::value % MJ;
    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w[i]), __builtin_bit_cast(bf16x8_t, x[j]),
                                                        acc[i][j], 0, 0, 0);
  };
  auto multiply = [&](const uint4v(&w)[NI], const uint4v(&x)[MJ]) {
    unrolled<0, NI * MJ>([&](auto k) { multiply_one(k, w, x); });
  };
  // the products of one pair of operands with the reads of the next between them (all reads first: 3 % slower)
  auto multiply_and_read = [&](const uint4v(&w)[NI], const uint4v(&x)[MJ], uint4v(&w2)[NI], uint4v(&x2)[MJ], uint32_t in_w,
                               uint32_t in_x, uint32_t half) {
    const uint32_t pw = (at_w + in_w * kW) ^ half, px = (at_x + in_x * kX) ^ half;
    constexpr int kReads = NI + MJ, kEach = NI * MJ / kReads;
    unrolled<0, kReads>([&](auto k) {
      read_one(k, w2, x2, pw, px);
      __builtin_amdgcn_sched_barrier(0);
      unrolled<decltype(k)::value * kEach, (decltype(k)::value + 1) * kEach>([&](auto p) { multiply_one(p, w, x); });
      __builtin_amdgcn_sched_barrier(0);
    });
    unrolled<kReads * kEach, NI * MJ>([&](auto p) { multiply_one(p, w, x); });
  };

  if (whole) {
    const uint32_t last = first + whole - 1;  // (past it the last step again rather than a branch: it is not read)
    // Copies land in the order they are made in.  A step's are x's for BX steps on and then W's for BW on, so when the
    // next step's have landed those of BX - 2 steps may be under way, and where W is a step further ahead the last W's.
    static_assert(BX >= 2 && (BW == BX || BW == BX + 1));
    constexpr int kUnderWay = (BX - 2) * (CX + CW) + (BW - BX) * CW;
#pragma unroll
    for (uint32_t b = 0; b < BX; ++b) copy_x(b, min(first + b, last)), copy_w(b, min(first + b, last));
    if constexpr (BW > BX) copy_w(BX, min(first + BX, last));
    copies_landed_everywhere<kUnderWay + CX + CW>();
    read(w_a, x_a, 0, 0, 0);
    uint32_t in_x = 0, in_w = 0;
    for (uint32_t t = 0; t + 1 < whole; ++t) {
      multiply_and_read(w_a, x_a, w_b, x_b, in_w, in_x, 64);
      operands_landed();  // nothing is read from these buffers any more by this wave ..
      copies_landed_everywhere<kUnderWay>();  // .. nor by another, and the next step's copies have landed
      copy_x(in_x, min(first + t + BX, last));
      copy_w(in_w, min(first + t + BW, last));
      in_x = in_x == BX - 1 ? 0 : in_x + 1, in_w = in_w == BW - 1 ? 0 : in_w + 1;
      multiply_and_read(w_b, x_b, w_a, x_a, in_w, in_x, 0);
    }
    read(w_b, x_b, in_w, in_x, 64);
    multiply(w_a, x_a);
    multiply(w_b, x_b);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  if (ragged) {  // the last columns, zeros behind them
    __syncthreads();
    const uint32_t at = (past - 1) * 128;
    const bool in = at + chunk < a.cols * 2;
    auto fill = [&](uint8_t *to, const uint16_t *from, uint32_t offset) {
      uint4v v = {0, 0, 0, 0};
      if (in) v = *reinterpret_cast<const uint4v *>(reinterpret_cast<const uint8_t *>(from) + offset + at);
      *reinterpret_cast<uint4v *>(to + lane * 16) = v;
    };
#pragma unroll 1
    for (int i = 0; i < CX; ++i) fill(lds + (i * W + wave) * 1024, x0, from_x(i));
#pragma unroll 1
    for (int i = 0; i < CW; ++i) fill(lds + BX * kX + (i * W + wave) * 1024, w0, from_w(i));
    __syncthreads();
#pragma unroll 1
    for (uint32_t half = 0; half < 128; half += 64) {
      read(w_a, x_a, 0, 0, half);
      multiply(w_a, x_a);
    }
  }

  // a lane holds columns n .. n + 3 of row m of y
  const bool fours = a.rows % 4 == 0 && a.ldy % 4 == 0;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const uint32_t n = n0 + wn * (TN / WN) + i * 16 + lane / 16 * 4;
    if (n >= a.rows) continue;
    float4v bias = {0, 0, 0, 0};
    if (a.bias && a.parts == 1)
      for (int v = 0; v < 4; ++v) bias[v] = __uint_as_float((uint32_t)a.bias[min(n + v, a.rows - 1)] << 16);
#pragma unroll
    for (int j = 0; j < MJ; ++j) {
      const uint32_t m = m0 + wm * (TM / WM) + j * 16 + lane % 16;
      if (m >= a.m_rows) continue;
      if (a.parts > 1) {
        *reinterpret_cast<float4v *>(a.partials + ((size_t)part * a.m_rows + m) * sums_pitch(a.rows) + n) = acc[i][j];
      } else {
        uint16_t *to = a.y + (size_t)m * a.ldy + n;
        half4v out;
#pragma unroll
        for (int v = 0; v < 4; ++v) out[v] = round_bf16(a.bias ? acc[i][j][v] + bias[v] : acc[i][j][v]);
        if (fours) *reinterpret_cast<half4v *>(to) = out;
        else
          for (int v = 0; v < 4; ++v)
            if (n + v < a.rows) to[v] = out[v];
      }
    }
  }
#else
  (void)a;
#endif
}

// ---------------------------------------------------------------- which tile, and whether at all

struct DensePlan {
  uint32_t tile, tiles_m, tiles_n, parts, steps_per_part;
  double us;
};

// The tiles there are: x's rows and W's rows a workgroup takes, workgroups a compute unit holds, and the times (us) that
// make a launch: one at the start, a step of a unit that is part full and of a full one, what each round of workgroups
// adds, the second launch and its sums a million bytes.  They rank tiles and do not foretell times: a step has one
// figure, whatever its rows begin on and whether other units are at work, so many products take up to half as long again
// and wide outputs of short rows (4054 x 592 at 1955 rows) nearly twice as long.  Against 1482
// launches of 150 products (profiles/dense_tilings.csv, made by dense_plan.py there; 129 to 2048 rows by 256 to 17408 x 512 to
// 17408) they are 14 to 23 % off rms, and the tile they choose is 1.7 % slower than the best of them on average, more than
// 16 % in three products below 12 us.  128 x 256, and 128 x 64 in two buffers, three workgroups a unit, gained nothing.
struct DenseTile {
  uint32_t m, n, resident;
  double start, part, full, round, second, sums;
};
constexpr DenseTile kTiles[] = {{256, 256, 1, 7.7, 0.0, 1.163, 7.43, 0.0, 0.114},
                                {256, 192, 1, 7.9, 0.0, 0.937, 4.28, 1.7, 0.113},
                                {256, 128, 1, 5.5, 0.0, 0.697, 3.83, 2.1, 0.140},
                                {128, 128, 2, 3.2, 0.573, 1.007, 1.64, 6.0, 0.110},
                                {128, 64, 2, 5.5, 0.369, 0.685, 1.20, 1.9, 0.160}};
constexpr uint32_t kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr uint32_t kUnits = 256;  // compute units
// A product that is cut takes two calls, and the host 3.5 us more: beside a short decode it is never sooner than this
// (with the decode, 306 x 768 at 156 rows 20.7 us in four parts, 18.3 whole; 490 x 512 at 160, whole, 17.3).
constexpr double kCutAtLeast = 12.5;

uint32_t up(uint32_t v, uint32_t by) { return v / by + (v % by != 0); }

// The product in one of the tiles, cut along K into at most `parts`, with the time the model gives it.
DensePlan plan_tile(uint32_t t, uint32_t parts, uint32_t rows, uint32_t cols, uint32_t m_rows) {
  const DenseTile &g = kTiles[t];
  const uint32_t steps = up(cols, kStep), tiles_m = up(m_rows, g.m), tiles_n = up(rows, g.n);
  const uint64_t tiles = (uint64_t)tiles_m * tiles_n;
  parts = std::min({parts, std::max(1u, steps / 2), 64u});
  const uint32_t per = up(steps, parts);
  parts = up(steps, per);
  const uint32_t on_unit = (uint32_t)((tiles * parts + kUnits - 1) / kUnits);
  const double step = g.full * (on_unit / g.resident) + (on_unit % g.resident ? g.part : 0.0);
  double us = g.start + per * step + g.round * up(on_unit, g.resident);
  if (parts > 1) us = std::max(us + g.second + g.sums * 8e-6 * parts * m_rows * rows, kCutAtLeast);
  return DensePlan{t, tiles_m, tiles_n, parts, per, us};
}

DensePlan plan_dense(uint32_t rows, uint32_t cols, uint32_t m_rows) {
  DensePlan best{};
  best.us = 1e30;
  for (uint32_t t = 0; t < kTileCount; ++t) {
    const uint64_t tiles = (uint64_t)up(m_rows, kTiles[t].m) * up(rows, kTiles[t].n);
    for (uint32_t fill = 0; fill <= kTiles[t].resident; ++fill) {  // whole, or cut to fill that many workgroups a unit
      const uint32_t parts = fill ? (uint32_t)std::max<uint64_t>(1, kUnits * fill / tiles) : 1u;
      const DensePlan p = plan_tile(t, parts, rows, cols, m_rows);
      if (p.us < best.us) best = p;
    }
  }
  return best;
}

// The fewest rows that the times above were fitted to; the fused kernels take fewer.
constexpr uint32_t kFewest = 129;

// The widest row of x, in values: a tile's offsets in it are 32 bits.
constexpr uint32_t kWidest = 1u << 21;

bool dense_fits(uint32_t rows, uint32_t cols, uint32_t m_rows) {
  return rows && cols && m_rows && cols % 8 == 0 && cols <= kWidest && (uint64_t)rows * m_rows <= (1u << 30);
}

size_t workspace_of(const DensePlan &p, uint32_t rows, uint32_t m_rows) {
  return p.parts > 1 ? (size_t)p.parts * m_rows * sums_pitch(rows) * 4 : 0;
}

template <int TM, int TN, int WM, int WN, int BX, int BW>
int launch_dense(const DenseArgs &a, hipStream_t s) {
  constexpr uint32_t lds = (BX * TM + BW * TN) * 128;
  if (lds > 64 * 1024)
    if (int rc = grf::allow_full_lds<&dense_gemm_kernel<TM, TN, WM, WN, BX, BW>>()) return rc;
  hipLaunchKernelGGL((dense_gemm_kernel<TM, TN, WM, WN, BX, BW>), dim3(a.tiles_m * a.tiles_n * a.parts), dim3(64 * WM * WN), lds, s, a);
  return GRF_OK;
}

int launch_plan(const DensePlan &p, const DenseArgs &a, hipStream_t s) {
  const int rc = p.tile == 0   ? launch_dense<256, 256, 4, 2, 2, 3>(a, s)
                 : p.tile == 1 ? launch_dense<256, 192, 4, 2, 2, 3>(a, s)
                 : p.tile == 2 ? launch_dense<256, 128, 4, 2, 3, 3>(a, s)
                 : p.tile == 3 ? launch_dense<128, 128, 2, 4, 2, 3>(a, s)
                               : launch_dense<128, 64, 2, 2, 3, 3>(a, s);
  if (rc) return rc;
  if (p.parts > 1)
    hipLaunchKernelGGL(dense_sum_kernel, dim3((a.rows + 1023) / 1024, a.m_rows), dim3(256), 0, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return grf::set_error(GRF_LAUNCH_FAILED, std::string("dense GEMM: ") + hipGetErrorString(e));
  return GRF_OK;
}

}  // namespace

double grf::dense_product_us(uint32_t rows, uint32_t cols, uint32_t m_rows) { return plan_dense(rows, cols, m_rows).us; }

extern "C" {

int64_t grf_dense_gemm_plan(uint32_t rows, uint32_t cols, uint32_t m_rows) {
  if (!dense_fits(rows, cols, m_rows) || m_rows < kFewest) return -1;
  const DensePlan p = plan_dense(rows, cols, m_rows);
  // Where the decode and this product together are faster than the decode and the library's product:
  //   rows of 13000 and longer: the library cuts little along K, above 16384 nothing (5120 x 17408 at 192, 512, 1000 rows
  //   3.1, 1.9, 1.6 times), up to the output that fills the GPU uncut (2048 rows 0.92);
  //   few tiles of output, more of them the longer the rows (6144 x 8192 at 129 rows 2.2 times; rows of 10240 to 13000 with more
  //   than 32 tiles 0.94 to 1.09, half of them slower, 1842 x 11520 at 1460 rows 97.3 us with the library and 103.9);
  //   anything short: its call is 19 us of the host's time, and a decode that ends sooner does not hide them.  A decode adds
  //   1.5 us a million weights to its first 7 (599 x 512 at 270 rows, with the decode, 25.5 and 16.3 us; 4708 x 1600 at 273,
  //   beyond the line, 30.9 and 33.0).
  // Of 1062 drawn calls (profiles/dense_linear.csv) 623 are taken, 1.35 times as fast in the mean; 14 of them are slower, by 2 to
  // 7 % (the rule goes by tiles of 256 x 256 and knows nothing of how evenly they fill the GPU).
  const uint64_t tiles = (uint64_t)((m_rows + 255) / 256) * ((rows + 255) / 256);
  const bool pays = cols >= 5000 ? tiles <= (cols >= 13000 ? 128 : cols >= 8192 ? 32 : 24)
                                 : tiles <= 32 && p.us + 1.5e-6 * rows * cols < 17.5;
  return pays ? (int64_t)workspace_of(p, rows, m_rows) : -1;
}

size_t grf_dense_gemm_workspace_bytes(uint32_t rows, uint32_t cols, uint32_t m_rows) {
  return dense_fits(rows, cols, m_rows) ? workspace_of(plan_dense(rows, cols, m_rows), rows, m_rows) : 0;
}

int grf_dense_gemm(const uint16_t *w, uint32_t rows, uint32_t cols, const uint16_t *x, uint32_t ldx, uint32_t m_rows,
                   uint16_t *y, uint32_t ldy, const uint16_t *bias, void *workspace, size_t workspace_bytes, void *hip_stream) {
  auto bad = [](const char *why) { return grf::set_error(GRF_BAD_ARGUMENT, std::string("grf_dense_gemm: ") + why); };
  if (!w || !x || !y) return bad("null argument");
  if (!dense_fits(rows, cols, m_rows)) return bad("cols a multiple of 8 up to 2^21, rows * m_rows up to 2^30");
  if (ldx < cols || ldx % 8 || ldx > kWidest || ldy < rows) return bad("leading dimension");
  if (((uintptr_t)w | (uintptr_t)x) & 15 || (uintptr_t)y & 7) return bad("w and x are 16-byte, y 8-byte aligned");
  const DensePlan p = plan_dense(rows, cols, m_rows);
  if (workspace_of(p, rows, m_rows) > workspace_bytes || (p.parts > 1 && (!workspace || (uintptr_t)workspace & 15)))
    return bad("workspace missing, misaligned or too small");
  hipStream_t s = (hipStream_t)hip_stream;
  const DenseArgs a{x, w, bias, y, static_cast<float *>(workspace), ldx, m_rows, rows, cols, ldy, p.tiles_m, p.tiles_n,
                    p.parts, p.steps_per_part};
  return launch_plan(p, a, s);
}

}  // extern "C"
