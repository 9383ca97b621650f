// Backward of the router's gating linear (gfx950): from the fp32 gradient g
// [T, E] of the logits, dx = g w [T, H] and dw = g^T x [E, H] with bf16 x, w.
//
// As fp32 products these are bound by the fp32 matrix rate (T 4096, H 7168, E
// 256: 15 GFLOP each, 139 + 136 us in a library GEMM at 110 TFLOP/s, and 62 us
// more for fp32 copies of x and w and the casts of the results). An fp32 value
// of 2^-110 or more is the exact sum of three bf16 values of eight significant
// bits each (below, the third ends at bf16's smallest subnormal and up to 2^-133
// is lost, the spacing of the smallest bf16 results), so g is split into three
// bf16 planes and both products run on bf16 matrix instructions with fp32
// accumulation: the same products, exact, in three times the operations at
// sixteen times the rate, and no larger error against float64. Both gradients,
// composition / here: T 4096, H 7168, E 256 344 / 110 us (split 6, dx 50, dw 48,
// the sum of its parts 5), 1024, 7168, 64 64 / 31, 16384, 2048, 128 277 / 85,
// 128, 1024, 64 24 / 17.
#include "gemm.h"

namespace {

constexpr int GB_NT = 256, GB_M = 128, GB_N = 128, GB_K = 32;
constexpr int GB_PLANE = GB_M * GB_K * 2;                // one plane's k-tile (8 KiB)
constexpr int GB_STAGE = 3 * GB_PLANE + GB_N * GB_K * 2;  // 32 KiB, two stages
// Tiles of dw are split along the tokens until about this many blocks run (two
// per CU).
constexpr int64_t GB_BLOCKS = 512;
constexpr int GB_RUN = 64, GB_GROUP = 8;  // tile order, as in gmm_wgrad_thin.hip

// v as three bf16 values whose sum it is (from 2^-110 up): the upper eight
// significant bits by truncation, then those of the exact remainders. Infinities
// and NaNs stay in the first.
__device__ __forceinline__ void split3(float v, uint16_t (&p)[3]) {
  const uint32_t b = __builtin_bit_cast(uint32_t, v);
  const bool finite = (b & 0x7f800000u) != 0x7f800000u;
  const uint32_t quiet = !finite && (b & 0x7fffffu) ? 0x400000u : 0u;
  const float hi = __builtin_bit_cast(float, b & 0xffff0000u);
  const float r1 = finite ? v - hi : 0.0f;
  const uint32_t b1 = __builtin_bit_cast(uint32_t, r1) & 0xffff0000u;
  const float r2 = r1 - __builtin_bit_cast(float, b1);
  p[0] = (uint16_t)((b | quiet) >> 16);
  p[1] = (uint16_t)(b1 >> 16);
  p[2] = (uint16_t)(__builtin_bit_cast(uint32_t, r2) >> 16);
}

// g = ga + gb (gb optional) as planes gp [3][T][E] and, transposed, gt
// [3][E][Tp] with zeros for tokens T .. Tp - 1; either may be null. A block
// takes 64 tokens x 32 experts.
__global__ __launch_bounds__(GB_NT) void gate_split_kernel(const float* __restrict__ ga,
                                                           const float* __restrict__ gb, int64_t T,
                                                           int E, int64_t Tp,
                                                           uint16_t* __restrict__ gp,
                                                           uint16_t* __restrict__ gt) {
  __shared__ uint16_t tile[3][32][64 + 4];
  const int64_t t0 = (int64_t)blockIdx.x * 64;
  const int e0 = blockIdx.y * 32;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = 32 * h + (threadIdx.x >> 3), c = 4 * (threadIdx.x & 7);
    const int64_t t = t0 + r;
    float4 v = {0.f, 0.f, 0.f, 0.f};
    if (t < T) {
      v = *reinterpret_cast<const float4*>(ga + t * E + e0 + c);
      if (gb != nullptr) {
        const float4 u = *reinterpret_cast<const float4*>(gb + t * E + e0 + c);
        v = float4{v.x + u.x, v.y + u.y, v.z + u.z, v.w + u.w};
      }
    }
    uint16_t q[4][3];
    split3(v.x, q[0]);
    split3(v.y, q[1]);
    split3(v.z, q[2]);
    split3(v.w, q[3]);
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      if (gp != nullptr && t < T)
        *reinterpret_cast<uint2*>(gp + ((int64_t)p * T + t) * E + e0 + c) =
            uint2{q[0][p] | (uint32_t)q[1][p] << 16, q[2][p] | (uint32_t)q[3][p] << 16};
#pragma unroll
      for (int i = 0; i < 4; ++i) tile[p][c + i][r] = q[i][p];
    }
  }
  if (gt == nullptr) return;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 6; ++k) {  // 3 planes x 32 experts x 16 pieces of 4 tokens
    const int idx = k * GB_NT + threadIdx.x, p = idx / 512, e = idx / 16 % 32, c = 4 * (idx & 15);
    if (t0 + c < Tp)
      *reinterpret_cast<uint2*>(gt + ((int64_t)p * E + e0 + e) * Tp + t0 + c) =
          *reinterpret_cast<const uint2*>(&tile[p][e][c]);
  }
}

// out[i, j] = sum over k of (a0 + a1 + a2)[k, i] b[k, j], planes a of K x lda
// elements one after the other, b [K, J]; I <= lda. One block computes a 128 x
// 128 tile over kc of the K rows (part z of them), each wave a 64 x 64
// quarter: 32-deep k-tiles of the three planes and b through two LDS stages,
// two blocks per CU; b's fragments serve the three planes' products, added
// smallest first. SPLIT stores fp32 parts [z][I][J], else bf16.
//
// A zero plane times an infinity in b would be a NaN that the fp32 product
// does not have: a tile with a NaN is computed again, element by element, from
// the planes' sums.
template <bool SPLIT>
__global__ __launch_bounds__(GB_NT, 2) void gate_bwd_kernel(const uint16_t* __restrict__ a,
                                                            const uint16_t* __restrict__ b,
                                                            void* __restrict__ out, int64_t K,
                                                            int64_t lda, int I, int J, int ti,
                                                            int tj, int64_t kc) {
  __shared__ __align__(16) char lds_raw[2 * GB_STAGE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int slot = blockIdx.x;
  if (slot < (int)gridDim.x / (8 * GB_RUN) * (8 * GB_RUN)) {
    const int p = slot / 8;
    slot = (p / GB_RUN * 8 + slot % 8) * GB_RUN + p % GB_RUN;
  }
  const int z = slot / (ti * tj), local = slot % (ti * tj);
  const int grp = local / (ti * GB_GROUP), gl = local % (ti * GB_GROUP);
  const int gw = tj - grp * GB_GROUP < GB_GROUP ? tj - grp * GB_GROUP : GB_GROUP;
  const int i0 = gl / gw * GB_M, j0 = (grp * GB_GROUP + gl % gw) * GB_N;
  const int64_t k0 = z * kc, kn = K - k0 < kc ? K - k0 : kc;  // kn may be negative: no rows
  const int nkt = kn > 0 ? (int)((kn + GB_K - 1) / GB_K) : 0;

  i32x4 ra[3];
#pragma unroll
  for (int p = 0; p < 3; ++p)
    ra[p] = make_rsrc(a + ((int64_t)p * K + k0) * lda + i0, (kn * lda - i0) * 2);
  const i32x4 rb = make_rsrc(b + k0 * J + j0, (kn * J - j0) * 2);
  // Two loads of four k-rows (256 bytes) per wave and operand, chunk slot s of
  // k-row r holding chunk s ^ (4 (r % 4)).
  uint32_t aoff[2], boff[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int r = 8 * wave + 4 * q + (lane >> 4), c = (lane & 15) ^ (4 * (r & 3));
    aoff[q] = (uint32_t)((r * lda + 8 * c) * 2);
    boff[q] = (uint32_t)((r * (int64_t)J + 8 * c) * 2);
  }
  lds_char* const lds = (lds_char*)lds_raw;
  auto issue = [&](int kt, int sl) {
    const uint32_t base = lds_addr_of(lds) + (uint32_t)(sl * GB_STAGE + 2 * wave * 1024);
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      const i32x4 r = advance_rsrc(ra[p], (uint32_t)(kt * GB_K * lda * 2));
#pragma unroll
      for (int q = 0; q < 2; ++q) dma16(aoff[q], r, base + p * GB_PLANE + q * 1024u);
    }
    const i32x4 r = advance_rsrc(rb, (uint32_t)((int64_t)kt * GB_K * J * 2));
#pragma unroll
    for (int q = 0; q < 2; ++q) dma16(boff[q], r, base + 3 * GB_PLANE + q * 1024u);
  };
  const int wm = wave >> 1, wn = wave & 1;
  auto frag_off = [&](int col) {
    const int g = lane >> 4, i = lane & 15;
    const int r = 8 * (g >> 1) + (i >> 2), c = col + 16 * (g & 1) + 4 * (i & 3);
    return (uint32_t)(r * 256 + (((c >> 3) ^ (4 * (r & 3))) << 4) + (c & 7) * 2);
  };
  auto frag = [&](lds_char* p) -> uint4 {
    const i16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)p);
    const i16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(p + 1024));
    const uint2 w0 = __builtin_bit_cast(uint2, v0), w1 = __builtin_bit_cast(uint2, v1);
    return uint4{w0.x, w0.y, w1.x, w1.y};
  };
  uint32_t fa[2], fb[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    fa[m] = frag_off(64 * wm + 32 * m);
    fb[m] = 3 * GB_PLANE + frag_off(64 * wn + 32 * m);
  }
  f32x16 acc[2][2] = {};
  if (nkt > 0) issue(0, 0);
  for (int kt = 0; kt < nkt; ++kt) {
    TT_WAIT_VMCNT(0);   // k-tile kt has landed
    TT_LDS_BARRIER();   // for every wave; the stage of kt - 1 is free
    if (kt + 1 < nkt) issue(kt + 1, (kt + 1) & 1);
    lds_char* const stg = lds + (kt & 1) * GB_STAGE;
#pragma unroll
    for (int s = 0; s < GB_K / 16; ++s) {
      uint4 bf[2];
#pragma unroll
      for (int n = 0; n < 2; ++n) bf[n] = frag(stg + fb[n] + s * 4096);
#pragma unroll
      for (int p = 2; p >= 0; --p)
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const uint4 af = frag(stg + p * GB_PLANE + fa[m] + s * 4096);
#pragma unroll
          for (int n = 0; n < 2; ++n) acc[m][n] = Mma<TT_BF16>::run(bf[n], af, acc[m][n]);
        }
    }
  }

  bool bad = false;
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int x = 0; x < 16; ++x) bad |= acc[m][n][x] != acc[m][n][x];
  float* const part = static_cast<float*>(out) + (int64_t)z * I * J;
  uint16_t* const o16 = static_cast<uint16_t*>(out);
  if (__syncthreads_or(bad)) {
    for (int idx = threadIdx.x; idx < GB_M * GB_N; idx += GB_NT) {
      const int i = i0 + idx / GB_N, j = j0 + idx % GB_N;
      if (i >= I || j >= J) continue;
      float s = 0.0f;
      for (int64_t k = k0; k < k0 + kn; ++k) {
        float g = 0.0f;
        for (int p = 2; p >= 0; --p) g += bf16_to_f32(a[((int64_t)p * K + k) * lda + i]);
        s = __builtin_fmaf(g, bf16_to_f32(b[k * J + j]), s);
      }
      if (SPLIT) part[(int64_t)i * J + j] = s;
      else o16[(int64_t)i * J + j] = (uint16_t)pack4<TT_BF16>(s, s, s, s).x;
    }
    return;
  }
  // Block (m, n), register 4 q + x of lane l: row 32 m + l % 32, column 32 n +
  // 8 q + 4 (l / 32) + x of the wave's quarter.
  if constexpr (SPLIT) {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int i = i0 + 64 * wm + 32 * m + (lane & 31);
          const int j = j0 + 64 * wn + 32 * n + 8 * q + 4 * (lane >> 5);
          if (i < I && j < J)
            *reinterpret_cast<float4*>(part + (int64_t)i * J + j) =
                float4{acc[m][n][4 * q], acc[m][n][4 * q + 1], acc[m][n][4 * q + 2],
                       acc[m][n][4 * q + 3]};
        }
  } else {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int r = 64 * wm + 32 * m + (lane & 31), c = 8 * wn + 4 * n + q;
          const uint2 v = pack4<TT_BF16>(acc[m][n][4 * q], acc[m][n][4 * q + 1],
                                         acc[m][n][4 * q + 2], acc[m][n][4 * q + 3]);
          *reinterpret_cast<lds_u32x2*>(lds + r * 256 + ((c ^ (r & 15)) << 4) + 8 * (lane >> 5)) =
              u32x2{v.x, v.y};
        }
    __syncthreads();
    const int c = threadIdx.x & 15;
    if (j0 + 8 * c >= J) return;
#pragma unroll
    for (int p = 0; p < GB_M / 16; ++p) {
      const int r = 16 * p + (threadIdx.x >> 4);
      if (i0 + r < I)
        *reinterpret_cast<uint4*>(o16 + (int64_t)(i0 + r) * J + j0 + 8 * c) =
            read_k(lds, (uint32_t)(r * 256 + ((c ^ (r & 15)) << 4)));
    }
  }
}

// out = bf16 of the parts' sum, in order; n elements, a multiple of 4.
__global__ __launch_bounds__(GB_NT) void gate_sum_kernel(const float* __restrict__ part, int parts,
                                                         int64_t n, uint16_t* __restrict__ out) {
  const int64_t i = ((int64_t)blockIdx.x * GB_NT + threadIdx.x) * 4;
  if (i >= n) return;
  float4 s = *reinterpret_cast<const float4*>(part + i);
  for (int z = 1; z < parts; ++z) {
    const float4 v = *reinterpret_cast<const float4*>(part + z * n + i);
    s = float4{s.x + v.x, s.y + v.y, s.z + v.z, s.w + v.w};
  }
  *reinterpret_cast<uint2*>(out + i) = pack4<TT_BF16>(s.x, s.y, s.z, s.w);
}

struct Plan {
  int64_t Tp, kc, gp, gt, part, bytes;  // byte offsets of the planes and parts
  int parts;
};
Plan plan(int64_t T, int H, int E) {
  Plan p;
  p.Tp = (T + 7) / 8 * 8;
  const int64_t tiles = ((int64_t)(E + GB_M - 1) / GB_M) * ((H + GB_N - 1) / GB_N);
  int64_t parts = GB_BLOCKS / tiles;
  const int64_t most = (T + 8 * GB_K - 1) / (8 * GB_K);  // eight k-tiles at least
  if (parts > most) parts = most;
  if (parts < 1) parts = 1;
  p.kc = ((T + parts - 1) / parts + GB_K - 1) / GB_K * GB_K;
  p.parts = (int)((T + p.kc - 1) / p.kc);
  p.gp = 0;
  p.gt = p.gp + (3 * T * E * 2 + 255) / 256 * 256;
  p.part = p.gt + (3 * p.Tp * E * 2 + 255) / 256 * 256;
  p.bytes = p.part + (p.parts > 1 ? (int64_t)p.parts * E * H * 4 : 0);
  return p;
}

bool takes(int64_t T, int64_t H, int64_t E) {
  // Rows of the planes and of x are addressed through 32-bit buffer offsets.
  return T >= 1 && E >= 32 && E <= 256 && E % 32 == 0 && H >= 64 && H % 64 == 0 &&
         (T + 2 * GB_K) * H * 2 < (int64_t)DM_OOB && (T + 64) * 2 * E < (int64_t)DM_OOB;
}

}  // namespace

extern "C" size_t tt_router_gate_bwd_workspace(int64_t T, int64_t H, int64_t E) {
  return takes(T, H, E) ? (size_t)plan(T, (int)H, (int)E).bytes : 0;
}

extern "C" int tt_router_gate_bwd(const float* grad, const float* grad2, const void* x,
                                  const void* w, int64_t T, int64_t H, int64_t E, void* workspace,
                                  size_t workspace_bytes, void* dx, void* dw, void* stream) {
  TT_REQUIRE(takes(T, H, E), "router_gate_bwd: unsupported size T=%lld H=%lld E=%lld",
             (long long)T, (long long)H, (long long)E);
  TT_REQUIRE(grad != nullptr && (dx == nullptr || w != nullptr) && (dw == nullptr || x != nullptr),
             "router_gate_bwd: missing operand");
  auto bits = [](const void* p) { return reinterpret_cast<uintptr_t>(p); };
  TT_REQUIRE(((bits(grad) | bits(grad2) | bits(x) | bits(w) | bits(workspace) | bits(dx) | bits(dw)) &
              15) == 0,
             "router_gate_bwd: operands must be 16-byte aligned");
  const Plan p = plan(T, (int)H, (int)E);
  TT_REQUIRE(workspace != nullptr && workspace_bytes >= (size_t)p.bytes,
             "router_gate_bwd: workspace of %lld bytes required", (long long)p.bytes);
  if (dx == nullptr && dw == nullptr) return TT_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  char* const ws = static_cast<char*>(workspace);
  uint16_t* const gp = reinterpret_cast<uint16_t*>(ws + p.gp);
  uint16_t* const gt = reinterpret_cast<uint16_t*>(ws + p.gt);
  hipLaunchKernelGGL(gate_split_kernel, dim3((unsigned)((T + 63) / 64), (unsigned)(E / 32)),
                     dim3(GB_NT), 0, s, grad, grad2, T, (int)E, p.Tp, dw ? gp : nullptr,
                     dx ? gt : nullptr);
  int rc = tt_check_launch("router_gate_bwd");
  if (rc != TT_OK) return rc;
  const int tj = (int)((H + GB_N - 1) / GB_N);
  if (dx != nullptr) {
    const int ti = (int)((T + GB_M - 1) / GB_M);
    TT_REQUIRE((int64_t)ti * tj < 0x7fffffff, "router_gate_bwd: grid too large");
    hipLaunchKernelGGL((gate_bwd_kernel<false>), dim3((unsigned)(ti * tj)), dim3(GB_NT), 0, s, gt,
                       static_cast<const uint16_t*>(w), dx, E, p.Tp, (int)T, (int)H, ti, tj, E);
    rc = tt_check_launch("router_gate_bwd");
    if (rc != TT_OK) return rc;
  }
  if (dw != nullptr) {
    const int ti = (int)((E + GB_M - 1) / GB_M);
    if (p.parts == 1) {
      hipLaunchKernelGGL((gate_bwd_kernel<false>), dim3((unsigned)(ti * tj)), dim3(GB_NT), 0, s,
                         gp, static_cast<const uint16_t*>(x), dw, T, E, (int)E, (int)H, ti, tj,
                         p.kc);
      return tt_check_launch("router_gate_bwd");
    }
    float* const part = reinterpret_cast<float*>(ws + p.part);
    hipLaunchKernelGGL((gate_bwd_kernel<true>), dim3((unsigned)(ti * tj * p.parts)), dim3(GB_NT),
                       0, s, gp, static_cast<const uint16_t*>(x), part, T, E, (int)E, (int)H, ti,
                       tj, p.kc);
    rc = tt_check_launch("router_gate_bwd");
    if (rc != TT_OK) return rc;
    const int64_t n = E * H;
    hipLaunchKernelGGL(gate_sum_kernel, dim3((unsigned)((n / 4 + GB_NT - 1) / GB_NT)), dim3(GB_NT),
                       0, s, part, p.parts, n, static_cast<uint16_t*>(dw));
    return tt_check_launch("router_gate_bwd");
  }
  return TT_OK;
}
