// What the products of many rows share (dense_gemm.hip, planes_prompt.hip): their arguments, copies straight to LDS and the waits for
// them, and the sums of products that are cut along K.
#pragma once
#include "fused_kernels.h"

namespace grf {

typedef uint32_t uint4v __attribute__((ext_vector_type(4)));
typedef uint16_t half4v __attribute__((ext_vector_type(4)));

constexpr uint32_t kStep = 64;  // columns a step takes: a line of 128 bytes a row

struct DenseArgs {
  const uint16_t *x, *w, *bias;
  uint16_t *y;
  float *partials;
  uint32_t ldx, m_rows, rows, cols, ldy, tiles_m, tiles_n, parts, steps_per_part;
};

// Floats from one row of a part's sums to the next: whole fours, so that a lane's four columns are one store and one load
// whatever W's rows (826 rows of 2121 x 13440 in five parts 83 us with four of each where the rows are odd).
__host__ __device__ constexpr uint32_t sums_pitch(uint32_t rows) { return (rows + 3) & ~3u; }

// What the product takes where W is dense, by the model of dense_gemm.hip (us).
double dense_product_us(uint32_t rows, uint32_t cols, uint32_t m_rows);

template <int I, int N, class F>
__device__ __forceinline__ void unrolled(const F &f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    unrolled<I + 1, N>(f);
  }
}

// Sixteen bytes a lane from the buffer at `from` + step_bytes straight to LDS, lane l's at `to` + 16 l.  In assembly,
// because of the copies that it knows about the compiler lets every operand read wait for all; there is no register that
// they write, and copies_landed waits for them.
__device__ __forceinline__ void copy_to_lds(uint4v buffer, uint32_t from, uint32_t step_bytes, uint32_t to) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(from), "s"(buffer), "s"(step_bytes),
               "s"(to)
               : "m0", "memory");
#else
  (void)buffer, (void)from, (void)step_bytes, (void)to;
#endif
}

// Every operand read of this wave has its value (and the reads are not put off past here).
__device__ __forceinline__ void operands_landed() {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#endif
}

// All but the last LEFT copies of every wave have landed.
template <int LEFT>
__device__ __forceinline__ void copies_landed_everywhere() {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(LEFT) : "memory");
#endif
}

// y = the parts in part order, the bias, one rounding; four columns a thread.
static __global__ __launch_bounds__(256) void dense_sum_kernel(DenseArgs a) {
  const uint32_t n = (blockIdx.x * 256 + threadIdx.x) * 4, m = blockIdx.y;
  if (n >= a.rows) return;
  const float4v *own = reinterpret_cast<const float4v *>(a.partials + (size_t)m * sums_pitch(a.rows) + n);
  const size_t pitch = (size_t)a.m_rows * (sums_pitch(a.rows) / 4);
  float4v sum;
  for (uint32_t p = 0; p < a.parts; p += 4) {  // four parts under way at a time
    float4v v[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) v[k] = own[min(p + k, a.parts - 1) * pitch];
    sum = p ? sum + v[0] : v[0];
#pragma unroll
    for (uint32_t k = 1; k < 4; ++k) sum = p + k < a.parts ? sum + v[k] : sum;
  }
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if (n + c >= a.rows) break;
    const float s = a.bias ? sum[c] + __uint_as_float((uint32_t)a.bias[n + c] << 16) : sum[c];
    a.y[(size_t)m * a.ldy + n + c] = round_bf16(s);
  }
}

}  // namespace grf
