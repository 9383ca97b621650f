// Per-expert LoRA residual on a grouped linear layer (gfx950):
//   y[m] = base[m] + round(round(h[m] B_e) * s),  h = x A_e
// for expert-major packed rows m, x / base / y in bf16 or f16, A [E, K, r] and
// B [E, r, N] in fp32, r at most 64. Every product and sum runs in fp32 on
// v_mfma_f32_16x16x4_f32 (16-bit activations widen exactly), and only the r-wide
// h is kept in fp32: a composition of grouped products instead writes and reads
// an fp32 copy of x and the fp32 product h B.
//
// * lora_down_kernel: h = x A_e, and dh = round(dy s) B_e^T in the backward.
// * lora_up_kernel: y from h, and dx = round(dh A_e^T).
// * lora_wgrad_kernel: dA_e = x_e^T dh_e and dB_e = h_e^T round(dy_e s).
//
// Low ranks are bound by the 16-bit activations that they stream and by the
// latency of a block's few loads, ranks above about 32 by the fp32 MFMAs.
// Layer of 128 experts, 2048 tokens, top-8, H 2048, F 768, r 16 (16384 rows),
// both linears: down 49 us forward and 68 backward, up 90 and 63, wgrad 37 (A)
// and 48 (B), 354 us in place of 1609 us of fp32 grouped products and 380 us of
// casts, scalings and sums; forward and backward 2821 -> 1204 us. At 4096
// tokens r 8 takes 4099 -> 1833 us, r 64 5018 -> 3043.
#include "gemm.h"

#include <type_traits>

namespace {

struct BF { static constexpr int code = TT_BF16; };
struct HF { static constexpr int code = TT_F16; };

constexpr int LR_NT = 256;
constexpr int LD_NT = 512;  // lora_down: eight waves share a reduction
typedef __attribute__((ext_vector_type(4))) float f32x4;

__device__ __forceinline__ f32x4 mfma16(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Two fp32 values to packed 16 bits by the hardware conversion (round to
// nearest even). Without the empty asm the compiler forms f16 products with a
// mixed-precision instruction that rounds once, where the composition's
// multiplication rounds to fp32 first (0.6 % of values times 0.37 differ).
template <class TT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
  asm("" : "+v"(a), "+v"(b));
  return pack4<TT::code>(a, b, 0.f, 0.f).x;
}
template <class TT>
__device__ __forceinline__ float lo16(uint32_t w) {
  if constexpr (TT::code == TT_BF16) return __uint_as_float(w << 16);
  else return f16_to_f32((uint16_t)(w & 0xffffu));
}
template <class TT>
__device__ __forceinline__ float hi16(uint32_t w) {
  if constexpr (TT::code == TT_BF16) return __uint_as_float(w & 0xffff0000u);
  else return f16_to_f32((uint16_t)(w >> 16));
}

// Eight packed 16-bit values widened; with SCALE times s and rounded to 16
// bits first.
template <class TT, bool SCALE>
__device__ __forceinline__ void widen8(const uint4& v, float s, float (&x)[8]) {
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t u = w[i];
    if constexpr (SCALE) u = pack2<TT>(lo16<TT>(u) * s, hi16<TT>(u) * s);
    x[2 * i] = lo16<TT>(u);
    x[2 * i + 1] = hi16<TT>(u);
  }
}

// ---------------------------------------------------------------------------
// out[m, j] (fp32 [M, r]) = sum over c of in[m, c] W_e(c, j), in [M, C] 16-bit.
// W_e: [C, r] (forward), or [r, C] (WT, the backward's B) with in scaled by s
// and rounded first (SCALE). A block takes 64 rows and every column; wave w
// takes the 32-deep steps w, w + 8, ... of the reduction and the waves' sums
// meet in LDS. Operands go straight to registers: lane (l % 16, l / 16) holds
// eight consecutive c of its row, or of its W column, and MFMA i of a step
// multiplies element i of each, so that no operand is transposed.
// ---------------------------------------------------------------------------
template <class TT, int RT, bool WT, bool SCALE>
__global__ __launch_bounds__(LD_NT) void lora_down_kernel(const uint16_t* __restrict__ in,
                                                          const float* __restrict__ W,
                                                          float* __restrict__ out, int C, int r,
                                                          float s, int E,
                                                          const int64_t* __restrict__ counts) {
  constexpr int BM = 64, MI = BM / 16, NW = LD_NT / 64;
  constexpr int RS = 16 * RT + 1;  // row stride of the partial sums
  __shared__ __align__(16) float part[NW * BM * RS];
  RowTile t;
  if (!row_tile<BM, LD_NT>(counts, E, 1, reinterpret_cast<char*>(part), t)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int64_t row0 = t.seg0 + (int64_t)t.mt * BM;
  const int rows = (int)(t.nrows - (int64_t)t.mt * BM < BM ? t.nrows - (int64_t)t.mt * BM : BM);
  const float* We = W + (int64_t)t.e * C * r;
  const uint16_t* src[MI];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    const int m = 16 * mi + l16;
    src[mi] = in + (row0 + (m < rows ? m : rows - 1)) * C;  // rows past the end: unused
  }
  int jl[RT];
#pragma unroll
  for (int jt = 0; jt < RT; ++jt) jl[jt] = 16 * jt + l16 < r ? 16 * jt + l16 : 0;
  f32x4 acc[MI][RT] = {};
  const int steps = (C + 31) / 32;
#pragma unroll 4
  for (int st = wave; st < steps; st += NW) {
    // Lanes past the end (C is a multiple of 8) or past the rank read a valid
    // element and drop it: no branch around a load.
    const int c0 = 32 * st + 8 * g;
    const bool live = c0 < C;
    const int cl = live ? c0 : 0;
    uint4 xv[MI];
    float wv[RT][8];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) xv[mi] = *reinterpret_cast<const uint4*>(src[mi] + cl);
#pragma unroll
    for (int jt = 0; jt < RT; ++jt) {
      const bool ok = live && 16 * jt + l16 < r;
      if constexpr (WT) {
        const float4* p = reinterpret_cast<const float4*>(We + (int64_t)jl[jt] * C + cl);
        const float4 a = p[0], b = p[1];
        wv[jt][0] = ok ? a.x : 0.f; wv[jt][1] = ok ? a.y : 0.f;
        wv[jt][2] = ok ? a.z : 0.f; wv[jt][3] = ok ? a.w : 0.f;
        wv[jt][4] = ok ? b.x : 0.f; wv[jt][5] = ok ? b.y : 0.f;
        wv[jt][6] = ok ? b.z : 0.f; wv[jt][7] = ok ? b.w : 0.f;
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) wv[jt][i] = We[(int64_t)(cl + i) * r + jl[jt]];
#pragma unroll
        for (int i = 0; i < 8; ++i) wv[jt][i] = ok ? wv[jt][i] : 0.f;
      }
    }
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      float x[8];
      widen8<TT, SCALE>(live ? xv[mi] : uint4{0, 0, 0, 0}, s, x);
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int jt = 0; jt < RT; ++jt) acc[mi][jt] = mfma16(x[i], wv[jt][i], acc[mi][jt]);
    }
  }
  // Lane l holds rows 16 mi + 4 (l / 16) + 0..3, column 16 jt + l % 16.
  __syncthreads();
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int jt = 0; jt < RT; ++jt)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        part[(wave * BM + 16 * mi + 4 * g + e) * RS + 16 * jt + l16] = acc[mi][jt][e];
  __syncthreads();
  for (int idx = threadIdx.x; idx < rows * r; idx += LD_NT) {
    const int m = idx / r, j = idx - m * r;
    const float* p = part + m * RS + j;
    float sum = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) sum += p[w * BM * RS];
    out[(row0 + m) * r + j] = sum;
  }
}

// ---------------------------------------------------------------------------
// d[m, n] = sum over j of h[m, j] W_e(j, n), h fp32 [M, r]. W_e: [r, N]
// (forward), or [N, r] (WT, the backward's A). y = base + round(round(d) s)
// (BASE), or y = round(d). A block takes 64 rows x 256 columns: W_e's columns
// go to LDS once, wave w multiplies columns 64 w .. + 63 for all rows, and the
// rounded products pass through LDS so that base and y move as whole 128-byte
// row segments.
// ---------------------------------------------------------------------------
template <class TT, int RT, bool WT, bool BASE>
__global__ __launch_bounds__(LR_NT) void lora_up_kernel(const float* __restrict__ h,
                                                        const float* __restrict__ W,
                                                        const uint16_t* __restrict__ base,
                                                        uint16_t* __restrict__ y, int N, int r,
                                                        float s, int E,
                                                        const int64_t* __restrict__ counts,
                                                        int tiles_n) {
  constexpr int BM = 64, BN = 256, MI = BM / 16, R = 16 * RT;
  constexpr int WS = BN + 16;  // row stride of W in LDS: four rows on distinct banks
  constexpr int LDS = R * WS * 4 > BM * BN * 2 ? R * WS * 4 : BM * BN * 2;
  __shared__ __align__(16) char lds_raw[LDS];
  RowTile t;
  if (!row_tile<BM, LR_NT>(counts, E, tiles_n, lds_raw, t)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int64_t row0 = t.seg0 + (int64_t)t.mt * BM;
  const int rows = (int)(t.nrows - (int64_t)t.mt * BM < BM ? t.nrows - (int64_t)t.mt * BM : BM);
  const int n0 = t.nt * BN;
  float* const wl = reinterpret_cast<float*>(lds_raw);
  const float* We = W + (int64_t)t.e * N * r;
  // The rows of base this lane adds to at the end, in flight from the start:
  // row 8 p + lane / 8, columns 8 (lane % 8) .. + 7 of the wave's 64.
  const int c = lane & 7, n = n0 + 64 * wave + 8 * c;  // N is a multiple of 8
  uint4 bv[BM / 8];
  if constexpr (BASE) {
#pragma unroll
    for (int p = 0; p < BM / 8; ++p) {
      const int m = 8 * p + (lane >> 3);
      bv[p] = *reinterpret_cast<const uint4*>(base + (row0 + (m < rows ? m : 0)) * N +
                                              (n < N ? n : 0));
    }
  }
  // All loads first, then the LDS writes; elements past N or the rank are zero.
  constexpr int WL = BN * R / (4 * LR_NT);
  float4 wr[WL];
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int idx = threadIdx.x + i * LR_NT;
    if constexpr (WT) {  // row n of W: its r values together, four j per load
      const int nn = idx / (R / 4), j = 4 * (idx % (R / 4));
      const float* p = We + (int64_t)(n0 + nn < N ? n0 + nn : 0) * r;
      float* const d = &wr[i].x;
#pragma unroll
      for (int k = 0; k < 4; ++k) d[k] = p[j + k < r ? j + k : 0];
    } else {  // row j of W: four columns per load (N is a multiple of 8)
      const int j = idx / (BN / 4), nn = 4 * (idx % (BN / 4));
      wr[i] = *reinterpret_cast<const float4*>(We + (int64_t)(j < r ? j : 0) * N +
                                               (n0 + nn < N ? n0 + nn : 0));
    }
  }
  // Step q of the reduction takes j = 4 q + l / 16.
  float hv[MI][4 * RT];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    const int m = 16 * mi + l16;
    const float* p = h + (row0 + (m < rows ? m : rows - 1)) * r;
#pragma unroll
    for (int q = 0; q < 4 * RT; ++q) hv[mi][q] = p[4 * q + g < r ? 4 * q + g : 0];
  }
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int q = 0; q < 4 * RT; ++q) hv[mi][q] = 4 * q + g < r ? hv[mi][q] : 0.f;
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int idx = threadIdx.x + i * LR_NT;
    if constexpr (WT) {
      const int nn = idx / (R / 4), j = 4 * (idx % (R / 4));
      const float* const d = &wr[i].x;
#pragma unroll
      for (int k = 0; k < 4; ++k) wl[(j + k) * WS + nn] = n0 + nn < N && j + k < r ? d[k] : 0.f;
    } else {
      const int j = idx / (BN / 4), nn = 4 * (idx % (BN / 4));
      *reinterpret_cast<float4*>(wl + j * WS + nn) =
          n0 + nn < N && j < r ? wr[i] : float4{0.f, 0.f, 0.f, 0.f};
    }
  }
  __syncthreads();
  f32x4 acc[4][MI] = {};
#pragma unroll
  for (int nt = 0; nt < 4; ++nt)
#pragma unroll
    for (int q = 0; q < 4 * RT; ++q) {
      const float w = wl[(4 * q + g) * WS + 64 * wave + 16 * nt + l16];
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) acc[nt][mi] = mfma16(w, hv[mi][q], acc[nt][mi]);
    }
  // Lane l holds row 16 mi + l % 16, columns 64 wave + 16 nt + 4 (l / 16) + 0..3.
  // Staging row m of wave: 128 bytes, 16-byte chunk c in slot c ^ (m % 8).
  __syncthreads();  // W is no longer needed
  char* const stg = lds_raw + wave * (BM * 128);
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const int m = 16 * mi + l16, ch = 2 * nt + (g >> 1);
      const f32x4 a = acc[nt][mi];
      uint2 v;
      v.x = pack2<TT>(a[0], a[1]);
      v.y = pack2<TT>(a[2], a[3]);
      *reinterpret_cast<uint2*>(stg + m * 128 + ((ch ^ (m & 7)) << 4) + 8 * (g & 1)) = v;
    }
  __syncthreads();
  if (n >= N) return;
#pragma unroll
  for (int p = 0; p < BM / 8; ++p) {
    const int m = 8 * p + (lane >> 3);
    if (m >= rows) continue;
    uint4 v = *reinterpret_cast<const uint4*>(stg + m * 128 + ((c ^ (m & 7)) << 4));
    const int64_t at = (row0 + m) * N + n;
    if constexpr (BASE) {
      float d[8], b[8];
      widen8<TT, true>(v, s, d);
      widen8<TT, false>(bv[p], 1.f, b);
      v = uint4{pack2<TT>(b[0] + d[0], b[1] + d[1]), pack2<TT>(b[2] + d[2], b[3] + d[3]),
                pack2<TT>(b[4] + d[4], b[5] + d[5]), pack2<TT>(b[6] + d[6], b[7] + d[7])};
    }
    *reinterpret_cast<uint4*>(y + at) = v;
  }
}

// ---------------------------------------------------------------------------
// G_e[c, j] = sum over e's rows m of in[m, c] v[m, j], in [M, C] 16-bit (scaled
// by s and rounded first with SCALE), v fp32 [M, r]; written [C, r], or [r, C]
// (GT). A block takes 128 columns of one expert; the waves split its rows four
// at a time and their sums meet in LDS. Lane (l % 16, l / 16) loads columns
// 8 (l % 16) .. + 7 of row l / 16, and MFMA i multiplies element i, column
// 8 (l % 16) + i: whole 256-byte row segments without a transpose. An expert
// without rows gets zeros.
// ---------------------------------------------------------------------------
template <class TT, int RT, bool GT, bool SCALE>
__global__ __launch_bounds__(LR_NT) void lora_wgrad_kernel(const uint16_t* __restrict__ in,
                                                           const float* __restrict__ v,
                                                           float* __restrict__ out, int C, int r,
                                                           float s,
                                                           const int64_t* __restrict__ counts) {
  __shared__ __align__(16) float red[4 * 8 * 4 * 64];  // [wave][i][reg][lane], one j tile
  __shared__ int64_t seg_part[LR_NT / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4;
  const int e = blockIdx.y;
  int64_t before = 0;  // rows of the experts before e
  for (int i = tid; i < e; i += LR_NT) before += counts[i];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off, 64);
  if (lane == 0) seg_part[wave] = before;
  __syncthreads();
  const int64_t row0 = seg_part[0] + seg_part[1] + seg_part[2] + seg_part[3];
  const int64_t rows = counts[e];
  const int c0 = blockIdx.x * 128 + 8 * l16;
  const bool live = c0 < C;  // C is a multiple of 8
  f32x4 acc[RT][8] = {};
#pragma unroll 4
  for (int64_t m0 = 4 * wave; m0 < rows; m0 += 16) {
    const int64_t m = m0 + g;
    const bool ok = m < rows;
    const int64_t at = row0 + (ok ? m : 0);
    uint4 x = *reinterpret_cast<const uint4*>(in + at * C + (live ? c0 : 0));
    float vv[RT];
#pragma unroll
    for (int jt = 0; jt < RT; ++jt) {
      const int j = 16 * jt + l16;
      vv[jt] = v[at * r + (j < r ? j : 0)];
      vv[jt] = ok && j < r ? vv[jt] : 0.f;
    }
    if (!ok || !live) x = uint4{0, 0, 0, 0};
    float a[8];
    widen8<TT, SCALE>(x, s, a);
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int jt = 0; jt < RT; ++jt)
        acc[jt][i] = GT ? mfma16(vv[jt], a[i], acc[jt][i]) : mfma16(a[i], vv[jt], acc[jt][i]);
  }
  float* const o = out + (int64_t)e * C * r;
#pragma unroll
  for (int jt = 0; jt < RT; ++jt) {
    if (jt) __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) red[((wave * 8 + i) * 4 + q) * 64 + lane] = acc[jt][i][q];
    __syncthreads();
    // Thread (lane, wave) sums registers q = wave of the eight tiles.
    float sum[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float* p = red + (i * 4 + wave) * 64 + lane;
      sum[i] = (p[0] + p[8 * 4 * 64]) + (p[2 * 8 * 4 * 64] + p[3 * 8 * 4 * 64]);
    }
    if constexpr (GT) {
      // Row j = 16 jt + 4 g + wave, columns 8 l16 + i.
      const int j = 16 * jt + 4 * g + wave;
      if (j < r && live) {
        float4* d = reinterpret_cast<float4*>(o + (int64_t)j * C + c0);
        d[0] = float4{sum[0], sum[1], sum[2], sum[3]};
        d[1] = float4{sum[4], sum[5], sum[6], sum[7]};
      }
    } else {
      // Column 8 (4 g + wave) + i, j = 16 jt + l16.
      const int j = 16 * jt + l16, c = blockIdx.x * 128 + 8 * (4 * g + wave);
      if (j < r && c < C)
#pragma unroll
        for (int i = 0; i < 8; ++i) o[(int64_t)(c + i) * r + j] = sum[i];
    }
  }
}

inline hipStream_t S(void* s) { return reinterpret_cast<hipStream_t>(s); }

struct LoraArgs {
  const uint16_t* in;
  const float* w;
  const uint16_t* base;
  void* out;
  int64_t M;
  int C, r;
  float s;
  int E;
  const int64_t* counts;
};

int64_t row_blocks(int64_t M, int E) { return M / 64 + (M < E ? M : E); }

template <class TT, int RT, bool WT, bool SCALE>
int launch_down(const LoraArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((lora_down_kernel<TT, RT, WT, SCALE>), dim3((unsigned)row_blocks(a.M, a.E)),
                     dim3(LD_NT), 0, s, a.in, a.w, static_cast<float*>(a.out), a.C, a.r, a.s, a.E,
                     a.counts);
  return tt_check_launch("lora_down");
}
template <class TT, int RT, bool WT, bool BASE>
int launch_up(const LoraArgs& a, const float* h, hipStream_t s) {
  const int tn = (a.C + 255) / 256;
  hipLaunchKernelGGL((lora_up_kernel<TT, RT, WT, BASE>),
                     dim3((unsigned)(row_blocks(a.M, a.E) * tn)), dim3(LR_NT), 0, s, h, a.w, a.base,
                     static_cast<uint16_t*>(a.out), a.C, a.r, a.s, a.E, a.counts, tn);
  return tt_check_launch("lora_up");
}
template <class TT, int RT, bool GT, bool SCALE>
int launch_wgrad(const LoraArgs& a, const float* v, hipStream_t s) {
  hipLaunchKernelGGL((lora_wgrad_kernel<TT, RT, GT, SCALE>),
                     dim3((unsigned)((a.C + 127) / 128), (unsigned)a.E), dim3(LR_NT), 0, s, a.in, v,
                     static_cast<float*>(a.out), a.C, a.r, a.s, a.counts);
  return tt_check_launch("lora_wgrad");
}

// f(type, r / 16 rounded up to 1, 2 or 4).
template <typename F>
int typed(int dtype, int r, F f) {
  auto go = [&](auto tt) {
    if (r <= 16) return f(tt, std::integral_constant<int, 1>{});
    if (r <= 32) return f(tt, std::integral_constant<int, 2>{});
    return f(tt, std::integral_constant<int, 4>{});
  };
  return dtype == TT_BF16 ? go(BF{}) : go(HF{});
}

int lora_checks(int dtype, int64_t m, int64_t c, int r, int E, const void* p0, const void* p1,
                const void* p2) {
  TT_REQUIRE(dtype == TT_BF16 || dtype == TT_F16, "lora: activations must be bf16 or f16");
  TT_REQUIRE(m >= 0 && m < (1ll << 31) && c >= 0 && c < (1ll << 24), "lora: bad sizes");
  TT_REQUIRE(c % 8 == 0, "lora: feature counts must be multiples of 8 (got %lld)", (long long)c);
  TT_REQUIRE(r >= 1 && r <= 64, "lora: the rank must be in [1, 64] (got %d)", r);
  TT_REQUIRE(E >= 1 && E <= 4096, "lora: num_experts must be in [1, 4096]");
  TT_REQUIRE(((reinterpret_cast<uintptr_t>(p0) | reinterpret_cast<uintptr_t>(p1) |
               reinterpret_cast<uintptr_t>(p2)) & 15) == 0,
             "lora: operands must be 16-byte aligned");
  TT_REQUIRE(row_blocks(m, E) * ((c + 255) / 256) < 0x7fffffff, "lora: grid too large");
  return TT_OK;
}

}  // namespace

extern "C" int tt_lora_down(const void* in, const float* w, int dtype, int64_t m, int64_t c,
                            int32_t r, int32_t transposed, float scale, int32_t num_experts,
                            const int64_t* counts, float* out, void* stream) {
  const int rc = lora_checks(dtype, m, c, r, num_experts, in, w, nullptr);
  if (rc != TT_OK) return rc;
  if (m == 0) return TT_OK;
  const LoraArgs a{static_cast<const uint16_t*>(in), w, nullptr, out, m, (int)c, r, scale,
                   num_experts, counts};
  return typed(dtype, r, [&](auto tt, auto rt) {
    typedef decltype(tt) TT;
    constexpr int RT = decltype(rt)::value;
    return transposed ? launch_down<TT, RT, true, true>(a, S(stream))
                      : launch_down<TT, RT, false, false>(a, S(stream));
  });
}

extern "C" int tt_lora_up(const float* h, const float* w, const void* base, int dtype, int64_t m,
                          int64_t c, int32_t r, int32_t transposed, float scale,
                          int32_t num_experts, const int64_t* counts, void* out, void* stream) {
  const int rc = lora_checks(dtype, m, c, r, num_experts, base, w, out);
  if (rc != TT_OK) return rc;
  TT_REQUIRE((base == nullptr) == (transposed != 0),
             "lora: the base is added in the forward form only");
  if (m == 0 || c == 0) return TT_OK;
  const LoraArgs a{nullptr, w, static_cast<const uint16_t*>(base), out, m, (int)c, r, scale,
                   num_experts, counts};
  return typed(dtype, r, [&](auto tt, auto rt) {
    typedef decltype(tt) TT;
    constexpr int RT = decltype(rt)::value;
    return transposed ? launch_up<TT, RT, true, false>(a, h, S(stream))
                      : launch_up<TT, RT, false, true>(a, h, S(stream));
  });
}

extern "C" int tt_lora_wgrad(const void* in, const float* v, int dtype, int64_t m, int64_t c,
                             int32_t r, int32_t transposed, float scale, int32_t num_experts,
                             const int64_t* counts, float* out, void* stream) {
  const int rc = lora_checks(dtype, m, c, r, num_experts, in, out, nullptr);
  if (rc != TT_OK) return rc;
  if (c == 0) return TT_OK;
  const LoraArgs a{static_cast<const uint16_t*>(in), nullptr, nullptr, out, m, (int)c, r, scale,
                   num_experts, counts};
  return typed(dtype, r, [&](auto tt, auto rt) {
    typedef decltype(tt) TT;
    constexpr int RT = decltype(rt)::value;
    return transposed ? launch_wgrad<TT, RT, true, true>(a, v, S(stream))
                      : launch_wgrad<TT, RT, false, false>(a, v, S(stream));
  });
}
