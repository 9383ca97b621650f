// Blockwise FP8 quantisation of expert weights (gfx950).
//
// tt_fp8_quantize_blocks turns bf16 weights [E, R, C] into e4m3 codes and one
// scale per 128 x 128 block: s = amax / 448 (1 for a block of zeros, or one
// whose amax is NaN), rounded to the scale dtype, and q = e4m3(clamp(w / s)).
#include "common.h"

namespace {

constexpr int QB = 128;      // rows and columns of a scale block
constexpr int Q_THREADS = 256;
constexpr int Q_VEC = 8;     // bf16 values per 16-byte load
constexpr int Q_ITER = QB * QB / (Q_THREADS * Q_VEC);  // loads per thread (8)

// e4m3 code of v (already clamped to +-448), NaN as 0x7f with its sign.
__device__ __forceinline__ uint32_t e4m3_code(float v) {
  if (v != v) return 0x7fu | ((__float_as_uint(v) >> 24) & 0x80u);
  return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(v, v, 0, false) & 0xffu;
}

__device__ __forceinline__ float clamp448(float v) {
  return __builtin_amdgcn_fmed3f(v, -448.f, 448.f);
}

// One block of four waves per scale block. Bound by memory: 2 bytes read and
// 1 written per weight, each once; a thread's eight 16-byte loads are all in
// flight before the first is used and the values stay in registers between
// the maximum and the codes, so the weights are read once (64 experts of
// 4096 x 7168 and 7168 x 2048: the passes of abs, amax, the two expansions of
// the scales, the division, clamp, cast and copy that this replaces took
// 27.3 ms, this kernel 1.52 ms, 5.55 TB/s, byte for byte the same).
//
// The quotient is the correctly rounded fp32 w / s without a division per
// element: y = 1 / s is formed once per block (rounded from fp64), then with
// t = w y (within 1.5 ulp of the quotient) and the remainder r = w - t s, t + r y
// is Markstein's correction. It rounds to w / s for every pair of a bf16 weight's
// 128 significands and a scale's 128 (those of amax / 448 in either scale dtype),
// enumerated in exact arithmetic in tests/test_fp8_checkpoint.py; powers of two
// change nothing while nothing under- or overflows: blocks
// whose scale lies outside [2^-60, 2^60] or whose amax is not finite divide.
template <class ST>
__global__ __launch_bounds__(Q_THREADS) void fp8_quantize_kernel(
    const uint16_t* __restrict__ w, int64_t cols, int blocks_c, uint8_t* __restrict__ q,
    typename ST::storage* __restrict__ scale) {
  __shared__ uint32_t part[Q_THREADS / TT_WAVE];
  const int64_t b = blockIdx.x;
  const int64_t br = b / blocks_c;  // block row over all experts (R is a multiple of 128)
  const int64_t bc = b - br * blocks_c;
  // 16 lanes of 8 values to a row, 16 rows per load.
  const int64_t at = (br * QB + (threadIdx.x >> 4)) * cols + bc * QB + (threadIdx.x & 15) * Q_VEC;
  uint32_t v[Q_ITER][4];
#pragma unroll
  for (int i = 0; i < Q_ITER; ++i) load_stream<16>(v[i], w + at + (int64_t)i * 16 * cols);
  // amax over the bit patterns of |w|: ordered as the values are, NaN on top.
  uint32_t m = 0;
#pragma unroll
  for (int i = 0; i < Q_ITER; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t lo = v[i][j] & 0x7fffu, hi = (v[i][j] >> 16) & 0x7fffu;
      m = max(m, max(lo, hi));
    }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, off, TT_WAVE));
  if (lane_id() == 0) part[threadIdx.x / TT_WAVE] = m;
  __syncthreads();
  m = max(max(part[0], part[1]), max(part[2], part[3]));
  const float amax = bf16_to_f32((uint16_t)m);
  const float s = ST::to_f32(ST::from_f32(amax > 0.f ? amax * (1.0f / 448.0f) : 1.0f));
  if (threadIdx.x == 0) scale[b] = ST::from_f32(s);
  const bool fast = m < 0x7f80u && s >= 0x1p-60f && s <= 0x1p60f;
  const float y = (float)(1.0 / (double)s);
#pragma unroll
  for (int i = 0; i < Q_ITER; ++i) {
    uint32_t o[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float x[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t pair = v[i][2 * j + (e >> 1)];
        x[e] = __uint_as_float((e & 1) ? pair & 0xffff0000u : pair << 16);
      }
      if (fast) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float t = x[e] * y;
          const float r = __builtin_fmaf(-t, s, x[e]);
          const float f = __builtin_fmaf(r, y, t);
          x[e] = clamp448(copysignf(f, x[e]));  // the correction drops the sign of -0
        }
        int c = __builtin_amdgcn_cvt_pk_fp8_f32(x[0], x[1], 0, false);
        o[j] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(x[2], x[3], c, true);
      } else {
        o[j] = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float f = x[e] / s;
          o[j] |= e4m3_code(f != f ? f : clamp448(f)) << (8 * e);
        }
      }
    }
    store_stream<8>(q + at + (int64_t)i * 16 * cols, o);
  }
}

}  // namespace

extern "C" int tt_fp8_quantize_blocks(const void* w, int dtype, int64_t num_experts, int64_t rows,
                                      int64_t cols, uint8_t* q, void* scale, int scale_dtype,
                                      void* stream) {
  TT_REQUIRE(num_experts >= 0 && rows >= 0 && cols >= 0, "fp8_quantize: negative sizes");
  TT_REQUIRE(dtype == TT_BF16, "fp8_quantize: weights must be bf16");
  TT_REQUIRE(scale_dtype == TT_BF16 || scale_dtype == TT_F32,
             "fp8_quantize: scales must be bf16 or f32");
  TT_REQUIRE(rows % QB == 0 && cols % QB == 0,
             "fp8_quantize: rows and columns must be multiples of 128 (got %lld, %lld)",
             (long long)rows, (long long)cols);
  TT_REQUIRE((reinterpret_cast<uintptr_t>(w) & 15) == 0 && (reinterpret_cast<uintptr_t>(q) & 7) == 0,
             "fp8_quantize: weights must be 16-byte and codes 8-byte aligned");
  const int64_t blocks = num_experts * (rows / QB) * (cols / QB);
  if (blocks == 0) return TT_OK;
  TT_REQUIRE(blocks < 0x7fffffff, "fp8_quantize: grid too large");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)blocks), block(Q_THREADS);
  const int bc = (int)(cols / QB);
  const uint16_t* src = static_cast<const uint16_t*>(w);
  if (scale_dtype == TT_BF16)
    hipLaunchKernelGGL(fp8_quantize_kernel<BF16T>, grid, block, 0, s, src, cols, bc, q,
                       static_cast<uint16_t*>(scale));
  else
    hipLaunchKernelGGL(fp8_quantize_kernel<F32T>, grid, block, 0, s, src, cols, bc, q,
                       static_cast<float*>(scale));
  return tt_check_launch("fp8_quantize");
}
