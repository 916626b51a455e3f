// y = x W^T (+ bias) for a dense BF16 W of rows x cols: what a product of more activation rows than the
// fused kernels take does after the matrix has been decoded to a transient.
//
// A workgroup makes a TN x TM tile of W's rows by x's rows, the sum over a part of K.  Steps of 64 columns
// go through two buffers of LDS, copied by loads that write it directly (a line of 128 bytes a row); a wave reads
// operands of v_mfma_f32_16x16x32_bf16 from there, the next 32 columns' while it multiplies the ones in hand, and
// keeps its tile in registers.  A row's eight 16-byte chunks lie at (chunk ^ row % 8): the copy leaves the lanes'
// places fixed, so the order is made by which chunk a lane fetches, and the reads of 16 rows then meet no bank twice.
//
// Bound by three things that nearly meet in the tile of 256 x 256: a step's 64 KiB take 0.73 us at the 38 bytes a
// cycle that a compute unit gets from its second-level cache into LDS, its products 0.87 us, its operand reads 0.4;
// together 1.4 us, 1.65 with every unit at work (steps of 32 columns in five buffers: 1.7, because half a line a
// row comes at 23 bytes a cycle; lines touched two steps ahead, the copy spread between the products, the first
// buffer given back earlier: no change; four waves of 128 x 128: spills).  1000 rows of 5120 x 17408: 174 us,
// 200 rows 66, where the library takes 250 and 222.
//
// A matrix whose tiles do not fill the GPU is cut along K: part p walks its share of the steps and leaves fp32
// sums in `partials` [parts][m_rows][rows], which dense_sum_kernel adds in part order.
#include "fused_kernels.h"

namespace {

using grf::bf16x8_t;
using grf::float4v;
using grf::round_bf16;

typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef uint16_t half4v __attribute__((ext_vector_type(4)));

constexpr uint32_t kStep = 64;  // columns a step takes: a line of 128 bytes a row

struct DenseArgs {
  const uint16_t *x, *w, *bias;
  uint16_t *y;
  float *partials;
  uint32_t ldx, m_rows, rows, cols, ldy, tiles_m, tiles_n, parts, steps_per_part;
};

template <int I, int N, class F>
__device__ __forceinline__ void unrolled(const F &f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    unrolled<I + 1, N>(f);
  }
}

// An operand read that the compiler does not wait for: `operands_landed` does.  (Left to it, a read behind a copy into
// the other buffer would wait for that copy.)
template <int OFFSET>
__device__ __forceinline__ void read_operand(uint4v &v, uint32_t at) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(OFFSET));
#else
  (void)v, (void)at;
#endif
}
template <int N>
__device__ __forceinline__ void keep_after(uint4v (&v)[N]) {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(v[i]));
#else
  (void)v;
#endif
}
template <int A, int B>
__device__ __forceinline__ void operands_landed(uint4v (&a)[A], uint4v (&b)[B]) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#endif
  keep_after(a);
  keep_after(b);
}

__device__ __forceinline__ void copies_landed_everywhere() {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
#endif
}

// Waves WN x WM, each TN / WN of W's rows by TM / WM of x's.
template <int TM, int TN, int WM, int WN>
__global__ __launch_bounds__(64 * WM *WN) void dense_gemm_kernel(DenseArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __align__(16) uint8_t lds[];
  typedef __attribute__((address_space(3))) void lds_void;
  constexpr int W = WM * WN, NI = TN / WN / 16, MJ = TM / WM / 16;
  constexpr int CX = TM / 8 / W, CW = TN / 8 / W;  // copies a wave makes a step, eight rows each
  constexpr uint32_t kBuffer = (TM + TN) * 128;
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
  const auto rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(x0), 0, 0x7fffffff, 0x00020000);
  const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t *>(w0), 0, 0x7fffffff, 0x00020000);
  // where the lane copies from; rows past the last read the last one, and what comes of them is not stored
  const uint32_t chunk = ((lane % 8) ^ (lane / 8)) * 16;
  auto from_x = [&](int i) { return min((uint32_t)(i * W + wave) * 8 + lane / 8, a.m_rows - 1 - m0) * a.ldx * 2 + chunk; };
  auto from_w = [&](int i) { return min((uint32_t)(i * W + wave) * 8 + lane / 8, a.rows - 1 - n0) * a.cols * 2 + chunk; };
  uint32_t vx[CX], vw[CW];
#pragma unroll
  for (int i = 0; i < CX; ++i) vx[i] = from_x(i);
#pragma unroll
  for (int i = 0; i < CW; ++i) vw[i] = from_w(i);
  auto copy = [&](uint32_t buffer, uint32_t step) {
    uint8_t *to = lds + buffer * kBuffer + wave * 1024;
#pragma unroll
    for (int i = 0; i < CX; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void *)(to + i * W * 1024), 16, vx[i], step * 128, 0, 0);
#pragma unroll
    for (int i = 0; i < CW; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_void *)(to + TM * 128 + i * W * 1024), 16, vw[i], step * 128, 0, 0);
  };

  const uint32_t wm = wave % WM, wn = wave / WM;
  // the lane's operands of the first 32 columns in the first buffer; those of the other 32 are at (that ^ 64)
  const uint32_t place = ((lane / 16) ^ (lane % 8)) * 16;
  const uint32_t at_x = (wm * (TM / WM) + lane % 16) * 128 + place, at_w = TM * 128 + (wn * (TN / WN) + lane % 16) * 128 + place;
  float4v acc[NI][MJ];
#pragma unroll
  for (int i = 0; i < NI; ++i)
#pragma unroll
    for (int j = 0; j < MJ; ++j) acc[i][j] = (float4v){0.f, 0.f, 0.f, 0.f};
  uint4v w_a[NI], x_a[MJ], w_b[NI], x_b[MJ];
  auto read_one = [&](auto k, uint4v(&w)[NI], uint4v(&x)[MJ], uint32_t pw, uint32_t px) {
    constexpr int K = decltype(k)::value;
    if constexpr (K < MJ) read_operand<K * 2048>(x[K], px);
    else read_operand<(K - MJ) * 2048>(w[K - MJ], pw);
  };
  auto read = [&](uint4v(&w)[NI], uint4v(&x)[MJ], uint32_t offset, uint32_t half) {
    const uint32_t pw = (at_w + offset) ^ half, px = (at_x + offset) ^ half;
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
  auto multiply_and_read = [&](const uint4v(&w)[NI], const uint4v(&x)[MJ], uint4v(&w2)[NI], uint4v(&x2)[MJ], uint32_t offset,
                               uint32_t half) {
    const uint32_t pw = (at_w + offset) ^ half, px = (at_x + offset) ^ half;
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
    copy(0, first);
    copies_landed_everywhere();
    if (whole > 1) copy(1, first + 1);
    read(w_a, x_a, 0, 0);
    for (uint32_t t = 0; t + 1 < whole; ++t) {
      const uint32_t offset = (t & 1) * kBuffer;
      operands_landed(w_a, x_a);
      multiply_and_read(w_a, x_a, w_b, x_b, offset, 64);
      operands_landed(w_b, x_b);  // nothing is read from this buffer any more by this wave ..
      copies_landed_everywhere();  // .. nor by another, and the next step's copies have landed
      copy(t & 1, min(first + t + 2, first + whole - 1));  // (the last step again rather than a branch: it is not read)
      multiply_and_read(w_b, x_b, w_a, x_a, kBuffer - offset, 0);
    }
    operands_landed(w_a, x_a);
    read(w_b, x_b, ((whole - 1) & 1) * kBuffer, 64);
    multiply(w_a, x_a);
    operands_landed(w_b, x_b);
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
    for (int i = 0; i < CW; ++i) fill(lds + TM * 128 + (i * W + wave) * 1024, w0, from_w(i));
    __syncthreads();
#pragma unroll 1
    for (uint32_t half = 0; half < 128; half += 64) {
      read(w_a, x_a, 0, half);
      operands_landed(w_a, x_a);
      multiply(w_a, x_a);
    }
  }

  // a lane holds columns n .. n + 3 of row m of y
  const bool fours = a.rows % 4 == 0;
#pragma unroll
  for (int j = 0; j < MJ; ++j) {
    const uint32_t m = m0 + wm * (TM / WM) + j * 16 + lane % 16;
    if (m >= a.m_rows) continue;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const uint32_t n = n0 + wn * (TN / WN) + i * 16 + lane / 16 * 4;
      if (n >= a.rows) continue;
      if (a.parts > 1) {
        float *to = a.partials + ((size_t)part * a.m_rows + m) * a.rows + n;
        if (fours) *reinterpret_cast<float4v *>(to) = acc[i][j];
        else
          for (int v = 0; v < 4; ++v)
            if (n + v < a.rows) to[v] = acc[i][j][v];
      } else {
        uint16_t *to = a.y + (size_t)m * a.ldy + n;
        half4v out;
#pragma unroll
        for (int v = 0; v < 4; ++v)
          out[v] = round_bf16(a.bias && n + v < a.rows ? acc[i][j][v] + __uint_as_float((uint32_t)a.bias[n + v] << 16) : acc[i][j][v]);
        if (fours && a.ldy % 4 == 0) *reinterpret_cast<half4v *>(to) = out;
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

// y = the parts in part order, the bias, one rounding; four columns a thread where the rows allow it.
template <int COLS>
__global__ __launch_bounds__(256) void dense_sum_kernel(DenseArgs a) {
  typedef float vec __attribute__((ext_vector_type(COLS)));
  const uint32_t n = (blockIdx.x * 256 + threadIdx.x) * COLS, m = blockIdx.y;
  if (n >= a.rows) return;
  const vec *own = reinterpret_cast<const vec *>(a.partials + (size_t)m * a.rows + n);
  const size_t pitch = (size_t)a.m_rows * a.rows / COLS;
  vec sum;
  for (uint32_t p = 0; p < a.parts; p += 4) {  // four parts under way at a time
    vec v[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) v[k] = own[min(p + k, a.parts - 1) * pitch];
    sum = p ? sum + v[0] : v[0];
#pragma unroll
    for (uint32_t k = 1; k < 4; ++k) sum = p + k < a.parts ? sum + v[k] : sum;
  }
#pragma unroll
  for (int c = 0; c < COLS; ++c) {
    float s;
    if constexpr (COLS == 1) s = sum[0];
    else s = sum[c];
    if (a.bias) s += __uint_as_float((uint32_t)a.bias[n + c] << 16);
    a.y[(size_t)m * a.ldy + n + c] = round_bf16(s);
  }
}

// ---------------------------------------------------------------- which tile, and whether at all

struct DensePlan {
  uint32_t tile, tiles_m, tiles_n, parts, steps_per_part;
  double us;
};

// The tiles there are: x's rows and W's rows a workgroup takes, workgroups a compute unit holds, and the times (us) that
// make a launch: one at the start, a step of a workgroup that has its unit alone and its share of a full one, what
// each workgroup of a unit adds, the second launch and its sums a million bytes.  Fitted to 26 000 launches of 1544
// products (129 to 2048 rows by 256 to 17408 x 512 to 17408, parts as below): 13 to 17 % rms, and the tile they choose is
// 3 % slower than the best measured on average.  128 x 256, 256 x 128 and 64 x 128 besides gained less than 1 %.
struct DenseTile {
  uint32_t m, n, resident;
  double start, alone, share, each, second, sums;
};
constexpr DenseTile kTiles[] = {{256, 256, 1, 14.3, 1.351, 0.500, 8.37, 0.0, 0.095},
                                {128, 128, 2, 3.5, 0.690, 0.518, 4.26, 6.6, 0.059},
                                {128, 64, 3, 3.2, 0.567, 0.346, 2.55, 5.9, 0.043}};
constexpr uint32_t kTileCount = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr uint32_t kUnits = 256;  // compute units

DensePlan plan_dense(uint32_t rows, uint32_t cols, uint32_t m_rows) {
  auto up = [](uint32_t v, uint32_t by) { return v / by + (v % by != 0); };
  const uint32_t steps = up(cols, kStep);
  DensePlan best{};
  best.us = 1e30;
  for (uint32_t t = 0; t < kTileCount; ++t) {
    const DenseTile &g = kTiles[t];
    const uint32_t tiles_m = up(m_rows, g.m), tiles_n = up(rows, g.n);
    const uint64_t tiles = (uint64_t)tiles_m * tiles_n;
    for (uint32_t fill = 0; fill <= g.resident; ++fill) {  // whole, or cut to fill that many workgroups a unit
      uint32_t parts = fill ? (uint32_t)std::max<uint64_t>(1, kUnits * fill / tiles) : 1u;
      parts = std::min({parts, std::max(1u, steps / 2), 64u});
      const uint32_t per = up(steps, parts);
      parts = up(steps, per);
      const uint32_t on_unit = (uint32_t)((tiles * parts + kUnits - 1) / kUnits);
      double us = g.start + per * std::max(g.alone * up(on_unit, g.resident), g.share * on_unit) + g.each * on_unit;
      if (parts > 1) us += g.second + g.sums * 8e-6 * parts * m_rows * rows;
      if (us < best.us) best = DensePlan{t, tiles_m, tiles_n, parts, per, us};
    }
  }
  return best;
}

// The widest row of x, in values: a tile's offsets in it are 32 bits.
constexpr uint32_t kWidest = 1u << 21;

bool dense_fits(uint32_t rows, uint32_t cols, uint32_t m_rows) {
  return rows && cols && m_rows && cols % 8 == 0 && cols <= kWidest && (uint64_t)rows * m_rows <= (1u << 30);
}

size_t workspace_of(const DensePlan &p, uint32_t rows, uint32_t m_rows) {
  return p.parts > 1 ? (size_t)p.parts * m_rows * rows * 4 : 0;
}

template <int TM, int TN, int WM, int WN>
int launch_dense(const DenseArgs &a, hipStream_t s) {
  constexpr uint32_t lds = 2 * (TM + TN) * 128;
  if (lds > 64 * 1024)
    if (int rc = grf::allow_full_lds<&dense_gemm_kernel<TM, TN, WM, WN>>()) return rc;
  hipLaunchKernelGGL((dense_gemm_kernel<TM, TN, WM, WN>), dim3(a.tiles_m * a.tiles_n * a.parts), dim3(64 * WM * WN), lds, s, a);
  return GRF_OK;
}

}  // namespace

extern "C" {

int64_t grf_dense_gemm_plan(uint32_t rows, uint32_t cols, uint32_t m_rows) {
  if (!dense_fits(rows, cols, m_rows)) return -1;
  const DensePlan p = plan_dense(rows, cols, m_rows);
  // Where the library's product is the slower one (1544 products, above; times are both sides'):
  //   rows longer than 16384: it has nothing cut along K there (5120 x 17408 at 200 rows 222 and 66 us, at 1000
  //   250 and 175; 1024 x 16896 at 512 rows 98 and 36), up to the output that fills the GPU uncut (2048 rows 279 and 418);
  //   from 10240: few tiles (5120 x 14336 at 256 rows 1.9 times, 1024 x 12288 at 512 40 and 29), at 1000 rows even;
  //   anything short: its call alone is 19 us of the host's time (1024 x 1040 at 129 rows 20 and 11), but for a few
  //   long rows, where a second launch is most of the work (256 x 8192 at 129 rows 19 and 23).
  const uint64_t tiles = (uint64_t)((m_rows + 255) / 256) * ((rows + 255) / 256);
  const bool pays = cols > 16384   ? tiles <= 128
                    : cols >= 10240 && rows >= 1024 && tiles <= 64 ? true
                                   : p.us < 17 && (rows >= 512 || cols <= 2048);
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
  const int rc = p.tile == 0   ? launch_dense<256, 256, 4, 2>(a, s)
                 : p.tile == 1 ? launch_dense<128, 128, 2, 4>(a, s)
                               : launch_dense<128, 64, 2, 2>(a, s);
  if (rc) return rc;
  if (p.parts > 1) {
    if (rows % 4 == 0)
      hipLaunchKernelGGL(dense_sum_kernel<4>, dim3((rows / 4 + 255) / 256, m_rows), dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL(dense_sum_kernel<1>, dim3((rows + 255) / 256, m_rows), dim3(256), 0, s, a);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return grf::set_error(GRF_LAUNCH_FAILED, std::string("dense GEMM: ") + hipGetErrorString(e));
  return GRF_OK;
}

}  // extern "C"
