// Per-expert LoRA residual on a grouped linear layer (gfx950):
//   y[m] = base[m] + round(round(h[m] B_e) * s),  h = x A_e
// for expert-major packed rows m, x / base / y in bf16 or f16, A [E, K, r] and
// B [E, r, N] in fp32, r at most 64. Every product and sum runs in fp32 on
// v_mfma_f32_16x16x4_f32 (16-bit activations widen exactly), and only the r-wide
// h is kept in fp32: a composition of grouped products instead writes and reads
// an fp32 copy of x and the fp32 product h B. The results are the composition's
// bit for bit (chain16 below).
//
// * lora_down_kernel: h = x A_e, and dh = round(dy s) B_e^T in the backward.
// * lora_up_kernel: y from h, and dx = round(dh A_e^T).
// * lora_wgrad_kernel: dA_e = x_e^T dh_e and dB_e = h_e^T round(dy_e s).
//
// Low ranks are bound by the 16-bit activations that they stream and by the
// chain of products, ranks above about 32 by the fp32 MFMAs. Layer of 128
// experts, 2048 tokens, top-8, H 2048, F 768, r 16 (16384 rows), both linears:
// down 53 us forward and 77 backward, up 89 and 63, wgrad 38 (A) and 52 (B),
// 372 us in place of 1609 us of fp32 grouped products and 380 us of casts,
// scalings and sums; forward and backward 2821 -> 1211 us, at 4096 tokens r 8
// 4098 -> 1843 us, r 64 5017 -> 2980. (Sums split over the waves of a block
// took 354 us, but in an order of their own: other last bits.)
#include "gemm.h"

#include <type_traits>

namespace {

struct BF { static constexpr int code = TT_BF16; };
struct HF { static constexpr int code = TT_F16; };

constexpr int LR_NT = 256;
constexpr int64_t LD_BLOCKS = 400;  // see launch_down
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(3))) float lds_float;

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

// Every sum runs in the order of the fp32 grouped products (gmm_f32_kernel),
// one chain of products per result: 0, 8, 1, 9, ... 7, 15 of each 16
// reduction elements, so that the results are a composition's bit for bit.
// Lane group g = lane / 16 of product q of such a 16 takes element
// 2 q + g / 2 + 8 (g % 2), the element chain16(4 q + g) of a position in the chain.
__device__ __forceinline__ int chain16(int p) {
  return (p & ~15) + 2 * ((p & 15) >> 2) + ((p >> 1) & 1) + 8 * (p & 1);
}

// The position of element j: chain16(place16(j)) = j.
__device__ __forceinline__ int place16(int j) {
  return (j & ~15) + 4 * ((j & 7) >> 1) + 2 * (j & 1) + ((j >> 3) & 1);
}

// Element `odd` of a packed pair, widened; with SCALE times s and rounded to
// 16 bits first.
template <class TT, bool SCALE>
__device__ __forceinline__ float widen1(uint32_t w, bool odd, float s) {
  float v = odd ? hi16<TT>(w) : lo16<TT>(w);
  if constexpr (SCALE) v = lo16<TT>(pack2<TT>(v * s, 0.f));
  return v;
}

// ---------------------------------------------------------------------------
// out[m, j] (fp32 [M, r]) = sum over c of in[m, c] W_e(c, j), in [M, C] 16-bit.
// W_e: [C, r] (forward), or [r, C] (WT, the backward's B) with in scaled by s
// and rounded first (SCALE). A block takes BM rows and every column, a wave 16
// rows and the columns of 1 / WC of the 16-wide tiles over the whole reduction;
// 64-deep k-tiles of in and W_e stream into a ring of S LDS stages (about 48
// KiB, three blocks per CU), one barrier per k-tile, as in gmm_thin_kernel. LDS of a stage: in 128 bytes per row, chunk c of row r in
// slot c ^ ((r >> 1) & 7); then W_e's 64 x r elements as they lie in memory,
// or (WT) 256 bytes per row j, chunk c in slot c ^ (j % 16).
// ---------------------------------------------------------------------------
template <class TT, int RT, bool WT, bool SCALE, int WC>
__global__ __launch_bounds__(LR_NT) void lora_down_kernel(const uint16_t* __restrict__ in,
                                                          const float* __restrict__ W,
                                                          float* __restrict__ out, int C, int r,
                                                          float s, int E,
                                                          const int64_t* __restrict__ counts) {
  constexpr int BM = 64 / WC, BK = 64, S = RT == 1 ? 4 : RT == 2 ? 3 : 2;
  constexpr int T_X = BM * BK * 2, T_W = 16 * RT * BK * 4, STAGE = T_X + T_W;
  constexpr int LX = BM / 32, LD = LX + RT;  // loads per wave and k-tile
  constexpr int CT = RT / WC;                // column tiles per wave
  __shared__ __align__(16) char lds_raw[S * STAGE];
  RowTile t;
  if (!row_tile<BM, LR_NT>(counts, E, 1, lds_raw, t)) return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int64_t row0 = t.seg0 + (int64_t)t.mt * BM;
  const int rows = (int)(t.nrows - (int64_t)t.mt * BM < BM ? t.nrows - (int64_t)t.mt * BM : BM);
  const int nkt = (C + BK - 1) / BK;
  const i32x4 rx = make_rsrc(in + row0 * C, (int64_t)rows * C * 2);
  const i32x4 rw = make_rsrc(W + (int64_t)t.e * C * r, (int64_t)C * r * 4);
  uint32_t xoff[LX], woff[RT];
  int xk[LX], wk[RT];
#pragma unroll
  for (int q = 0; q < LX; ++q) {
    const int m = 8 * (LX * wave + q) + (lane >> 3), c = (lane & 7) ^ ((m >> 1) & 7);
    xk[q] = 8 * c;
    xoff[q] = (uint32_t)(((int64_t)m * C + 8 * c) * 2);
  }
#pragma unroll
  for (int q = 0; q < RT; ++q) {
    if constexpr (WT) {
      const int j = 4 * (RT * wave + q) + g, c = l16 ^ (j & 15);
      wk[q] = 4 * c;
      woff[q] = j < r ? (uint32_t)(((int64_t)j * C + 4 * c) * 4) : DM_OOB;
    } else {
      const int at = 16 * (64 * (RT * wave + q) + lane);  // of the k-tile's 256 r bytes
      wk[q] = 0;
      woff[q] = at < 256 * r ? (uint32_t)at : DM_OOB;
    }
  }
  lds_char* const lds = (lds_char*)lds_raw;
  auto issue = [&](int kt, int slot) {
    const uint32_t base = lds_addr_of(lds) + (uint32_t)slot * STAGE;
    const i32x4 ax = advance_rsrc(rx, (uint32_t)kt * (BK * 2));
    const i32x4 aw = advance_rsrc(rw, (uint32_t)kt * (uint32_t)(BK * 4 * (WT ? 1 : r)));
#pragma unroll
    for (int q = 0; q < LX; ++q)
      dma16(kt * BK + xk[q] < C ? xoff[q] : DM_OOB, ax, base + (uint32_t)(LX * wave + q) * 1024u);
#pragma unroll
    for (int q = 0; q < RT; ++q)
      dma16(WT && kt * BK + wk[q] >= C ? DM_OOB : woff[q], aw,
            base + T_X + (uint32_t)(RT * wave + q) * 1024u);
  };
  const bool odd = g >> 1;
  const int wr = wave / WC, wc = wave % WC;  // the wave's rows and columns
  const int row = 16 * wr + l16;
  f32x4 acc[CT] = {};
#pragma unroll
  for (int i = 0; i < S - 1; ++i)
    if (i < nkt) issue(i, i);
  int slot = 0;
  for (int kt = 0; kt < nkt; ++kt) {
    // k-tile kt has landed once at most the later ones are outstanding.
    const int later = nkt - 1 - kt;
    if (S >= 4 && later >= 2) TT_WAIT_VMCNT(2 * LD);
    else if (S >= 3 && later >= 1) TT_WAIT_VMCNT(LD);
    else TT_WAIT_VMCNT(0);
    TT_LDS_BARRIER();
    if (kt + S - 1 < nkt) issue(kt + S - 1, slot == 0 ? S - 1 : slot - 1);  // the stage of kt - 1
    lds_char* const stg = lds + slot * STAGE;
    const lds_float* const wl = reinterpret_cast<const lds_float*>(stg + T_X);
    // The fragments of 16 elements are read while the 16 before are multiplied.
    uint4 xv[2];
    float wv[2][4][CT];
    auto read = [&](int b) {
      xv[b & 1] = read_k(
          stg, (uint32_t)(row * 128 + (((2 * b + (g & 1)) ^ ((row >> 1) & 7)) << 4)));
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int jt = 0; jt < CT; ++jt) {
          const int c = 16 * b + 8 * (g & 1) + 2 * q + (g >> 1);
          const int j = 16 * (CT * wc + jt) + l16;  // results of j >= r are not stored
          wv[b & 1][q][jt] = WT ? wl[j * 64 + (((c >> 2) ^ (j & 15)) << 2) + (c & 3)]
                                : wl[c * r + (j < r ? j : 0)];
        }
    };
    if (16 * wr < rows) {
      read(0);
#pragma unroll
      for (int b = 0; b < BK / 16; ++b) {
        if (b + 1 < BK / 16) read(b + 1);
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t x[4] = {xv[b & 1].x, xv[b & 1].y, xv[b & 1].z, xv[b & 1].w};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float a = widen1<TT, SCALE>(x[q], odd, s);
#pragma unroll
          for (int jt = 0; jt < CT; ++jt) acc[jt] = mfma16(a, wv[b & 1][q][jt], acc[jt]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    slot = slot == S - 1 ? 0 : slot + 1;
  }
  // Lane l holds rows 16 wr + 4 (l / 16) + 0..3, column 16 (CT wc + jt) + l % 16.
#pragma unroll
  for (int jt = 0; jt < CT; ++jt)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int m = 16 * wr + 4 * g + e, j = 16 * (CT * wc + jt) + l16;
      if (m < rows && j < r) out[(row0 + m) * r + j] = acc[jt][e];
    }
}

// ---------------------------------------------------------------------------
// d[m, n] = sum over j of h[m, j] W_e(j, n), h fp32 [M, r]. W_e: [r, N]
// (forward), or [N, r] (WT, the backward's A). y = base + round(round(d) s)
// (BASE), or y = round(d). A block takes 64 rows x 256 columns: W_e's columns
// go to LDS once (row j in the order of the chain), wave w multiplies columns
// 64 w .. + 63 for all rows, and the rounded products pass through LDS so that
// base and y move as whole 128-byte row segments.
// ---------------------------------------------------------------------------
template <class TT, int RT, bool WT, bool BASE>
__global__ __launch_bounds__(LR_NT, RT == 2 && WT ? 3 : 1) void lora_up_kernel(
    const float* __restrict__ h, const float* __restrict__ W, const uint16_t* __restrict__ base,
    uint16_t* __restrict__ y, int N, int r, float s, int E, const int64_t* __restrict__ counts,
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
  // Step q of the reduction takes j = chain16(4 q + l / 16).
  float hv[MI][4 * RT];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    const int m = 16 * mi + l16;
    const float* p = h + (row0 + (m < rows ? m : rows - 1)) * r;
#pragma unroll
    for (int q = 0; q < 4 * RT; ++q) {
      const int j = chain16(4 * q + g);
      hv[mi][q] = p[j < r ? j : 0];
    }
  }
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int q = 0; q < 4 * RT; ++q) hv[mi][q] = chain16(4 * q + g) < r ? hv[mi][q] : 0.f;
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int idx = threadIdx.x + i * LR_NT;
    if constexpr (WT) {
      const int nn = idx / (R / 4), j = 4 * (idx % (R / 4));
      const float* const d = &wr[i].x;
#pragma unroll
      for (int k = 0; k < 4; ++k)
        wl[place16(j + k) * WS + nn] = n0 + nn < N && j + k < r ? d[k] : 0.f;
    } else {
      const int j = idx / (BN / 4), nn = 4 * (idx % (BN / 4));
      *reinterpret_cast<float4*>(wl + place16(j) * WS + nn) =
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
// (GT). A block takes 128 columns of one expert, wave w columns 32 w .. + 31
// over all of its rows: lane (l % 16, l / 16) loads columns 2 (l % 16) and
// + 1 of the four rows of a step, and MFMA i multiplies column 2 (l % 16) + i,
// so that no operand is transposed. An expert without rows gets zeros.
// ---------------------------------------------------------------------------
template <class TT, int RT, bool GT, bool SCALE>
__global__ __launch_bounds__(LR_NT) void lora_wgrad_kernel(const uint16_t* __restrict__ in,
                                                           const float* __restrict__ v,
                                                           float* __restrict__ out, int C, int r,
                                                           float s,
                                                           const int64_t* __restrict__ counts) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, g = lane >> 4;
  const int e = blockIdx.y;
  const int cw = blockIdx.x * 128 + 32 * wave;
  if (cw >= C) return;
  int64_t before = 0;  // rows of the experts before e
  for (int i = lane; i < e; i += 64) before += counts[i];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off, 64);
  const int64_t row0 = before, rows = counts[e];
  const int c0 = cw + 2 * l16;
  const bool live = c0 < C;  // C is a multiple of 8
  const uint16_t* const src = in + row0 * C + (live ? c0 : 0);
  const float* const vsrc = v + row0 * r;
  f32x4 acc[RT][2] = {};
  const int first = chain16(g);
  // 16 rows are loaded while the 16 before are multiplied.
  uint32_t x[2][4];
  float vv[2][4][RT];
  auto load = [&](int64_t m0, int buf) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t m = m0 + first + 2 * q;  // chain16(4 q + g)
      const int64_t at = m < rows ? m : 0;
      x[buf][q] = *reinterpret_cast<const uint32_t*>(src + at * C);
#pragma unroll
      for (int jt = 0; jt < RT; ++jt)
        vv[buf][q][jt] = vsrc[at * r + (16 * jt + l16 < r ? 16 * jt + l16 : 0)];
    }
  };
  auto multiply = [&](int64_t m0, int buf) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const bool ok = m0 + first + 2 * q < rows;
      const uint32_t xq = ok && live ? x[buf][q] : 0;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const float a = widen1<TT, SCALE>(xq, i == 1, s);
#pragma unroll
        for (int jt = 0; jt < RT; ++jt) {
          const float b = ok && 16 * jt + l16 < r ? vv[buf][q][jt] : 0.f;
          acc[jt][i] = GT ? mfma16(b, a, acc[jt][i]) : mfma16(a, b, acc[jt][i]);
        }
      }
    }
  };
  if (rows > 0) load(0, 0);
  for (int64_t m0 = 0; m0 < rows; m0 += 32) {
    if (m0 + 16 < rows) load(m0 + 16, 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(m0, 0);
    if (m0 + 16 >= rows) break;
    if (m0 + 32 < rows) load(m0 + 32, 0);
    __builtin_amdgcn_sched_barrier(0);
    multiply(m0 + 16, 1);
  }
  float* const o = out + (int64_t)e * C * r;
#pragma unroll
  for (int jt = 0; jt < RT; ++jt)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if constexpr (GT) {  // row j = 16 jt + 4 g + q, columns c0 and c0 + 1
        const int j = 16 * jt + 4 * g + q;
        if (j < r && live)
          *reinterpret_cast<float2*>(o + (int64_t)j * C + c0) = float2{acc[jt][0][q], acc[jt][1][q]};
      } else {  // columns cw + 2 (4 g + q) + i, j = 16 jt + l16
        const int j = 16 * jt + l16, c = cw + 2 * (4 * g + q);
        if (j < r && c < C) {
          o[(int64_t)c * r + j] = acc[jt][0][q];
          o[(int64_t)(c + 1) * r + j] = acc[jt][1][q];
        }
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

int64_t row_blocks(int64_t M, int E, int bm = 64) { return M / bm + (M < E ? M : E); }

template <class TT, int RT, bool WT, bool SCALE, int WC>
int launch_down_wc(const LoraArgs& a, hipStream_t s) {
  hipLaunchKernelGGL((lora_down_kernel<TT, RT, WT, SCALE, WC>),
                     dim3((unsigned)row_blocks(a.M, a.E, 64 / WC)), dim3(LR_NT), 0, s, a.in, a.w,
                     static_cast<float*>(a.out), a.C, a.r, a.s, a.E, a.counts);
  return tt_check_launch("lora_down");
}
// Ranks above 32 in blocks of 32 rows, two waves to the columns, ranks above 16
// while 64-row blocks make at most LD_BLOCKS. 64- / 32-row blocks, 2432 columns,
// forward and transposed: r 64, 32 experts of 55 rows 70.9 + 80.2 / 42.2 + 49.3 us,
// 128 of 130 108.6 + 119.5 / 85.4 + 97.9, of 256 149.4 + 162.8 / 136.9 + 155.0; r
// 32, 32 of 55 43.9 + 47.3 / 29.2 + 34.3, 128 of 130 (388 blocks) 65.4 + 70.4 /
// 52.1 + 65.1, of 200 (528) 65.6 + 71.0 / 65.7 + 80.6.
template <class TT, int RT, bool WT, bool SCALE>
int launch_down(const LoraArgs& a, hipStream_t s) {
  if constexpr (RT == 4) {
    return launch_down_wc<TT, RT, WT, SCALE, 2>(a, s);
  } else {
    if constexpr (RT == 2)
      if (row_blocks(a.M, a.E) <= LD_BLOCKS) return launch_down_wc<TT, RT, WT, SCALE, 2>(a, s);
    return launch_down_wc<TT, RT, WT, SCALE, 1>(a, s);
  }
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
