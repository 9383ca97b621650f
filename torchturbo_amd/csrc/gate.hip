// Logits of the router's gating linear with the experts spread over blocks
// (gfx950): x [T, H] W [E, H]^T in 16 bits with fp32 accumulation, rounded to
// the logits dtype. The top-k follows in a kernel of its own (route.hip).
#include "gemm.h"

namespace {

constexpr int GL_NT = 256;

// A block computes 32 MT tokens x 32 NE experts over the whole hidden size,
// one 32x32 tile per wave, accumulated in the order of the gate's one-kernel
// form (64-deep chunks, four MFMA steps each), so the logits are the same
// bits. The one-kernel form holds every expert's rows of a chunk in LDS, which
// leaves two chunks in flight and few blocks: it is bound by the latency of
// its chunks (H 7168, E 256: 0.65 us each, 76 us from 24 to 8192 tokens). Here
// the chunks of a few expert rows go through a ring of S stages.
template <int ET, int MT, int NE, int CH, int S>
__global__ __launch_bounds__(GL_NT) void gate_logits_kernel(const char* __restrict__ x,
                                                            const char* __restrict__ w,
                                                            int64_t T, int H, int E, int ldt,
                                                            void* __restrict__ logits) {
  constexpr int CHUNK = 32 * (MT + NE) * 128, STAGE = CH * CHUNK;
  constexpr int LD = MT + NE;  // loads (8 rows) per wave and chunk
  __shared__ __align__(16) char lds_raw[S * STAGE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t t0 = (int64_t)blockIdx.x * (32 * MT);
  const int e0 = blockIdx.y * (32 * NE);
  const int nch = H / 64;
  const int64_t rows = T - t0 < 32 * MT ? T - t0 : 32 * MT;
  const i32x4 rx = make_rsrc(x + t0 * H * 2, rows * H * 2);
  const i32x4 rw = make_rsrc(w + (int64_t)e0 * H * 2, (int64_t)(E - e0) * H * 2);
  // Load q of this wave fills rows 8 (LD wave + q) .. + 7 of a stage (tokens,
  // then experts): lane / 8 the row, slot lane % 8 holding chunk
  // slot ^ ((row >> 1) & 7).
  uint32_t off[LD];
  bool isx[LD];
#pragma unroll
  for (int q = 0; q < LD; ++q) {
    const int g = LD * wave + q;
    const int r = 8 * g + (lane >> 3);
    isx[q] = 8 * g < 32 * MT;
    off[q] = (uint32_t)(((isx[q] ? r : r - 32 * MT) * (int64_t)H +
                         8 * ((lane & 7) ^ ((r >> 1) & 7))) * 2);
  }
  lds_char* const lds = (lds_char*)lds_raw;
  const uint32_t lds0 = lds_addr_of(lds);
  // Chunks CH st .. of stage st; nothing is read past the hidden size, but the
  // loads are issued, so that the counts below stay fixed.
  auto issue = [&](int st, int slot) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int kc = CH * st + c;
      i32x4 ax = advance_rsrc(rx, (uint32_t)kc * 128u), aw = advance_rsrc(rw, (uint32_t)kc * 128u);
      if (kc >= nch) ax.z = aw.z = 0;
#pragma unroll
      for (int q = 0; q < LD; ++q)
        dma16(off[q], isx[q] ? ax : aw,
              lds0 + (uint32_t)(slot * STAGE + c * CHUNK + (LD * wave + q) * 1024));
    }
  };
  // The wave has a tile (the last block's may lie past the experts).
  const bool busy = wave < MT * NE && e0 + 32 * (wave / MT) < E;
  const int mt = wave % MT, ne = busy ? wave / MT : 0;
  uint32_t fa[4], fb[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    fa[s] = fragk64(32 * mt, s, lane);
    fb[s] = fragk64(32 * (MT + ne), s, lane);
  }
  f32x16 acc = {};
#pragma unroll
  for (int s = 0; s < S - 1; ++s) issue(s, s);
  int slot = 0;
  const int nst = (nch + CH - 1) / CH;
  for (int st = 0; st < nst; ++st) {
    TT_WAIT_VMCNT((S - 2) * LD * CH);  // stage st has landed
    TT_LDS_BARRIER();                  // for every wave; the one before it is free
    issue(st + S - 1, slot == 0 ? S - 1 : slot - 1);
    if (busy) {
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        if (CH * st + c >= nch) break;
        lds_char* const base = lds + slot * STAGE + c * CHUNK;
#pragma unroll
        for (int s = 0; s < 4; ++s)
          acc = Mma<ET>::run(read_k(base, fb[s]), read_k(base, fa[s]), acc);
      }
    }
    slot = slot == S - 1 ? 0 : slot + 1;
  }
  TT_WAIT_VMCNT(0);  // no load lands after the block has gone
  if (!busy) return;
  // Lane l holds token 32 mt + l % 32, experts 32 ne + 8 g + 4 (l / 32) + 0..3
  // in registers 4 g ...
  const int row = 32 * mt + (lane & 31);
  if (row >= rows) return;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int64_t at = (t0 + row) * E + e0 + 32 * ne + 8 * g + 4 * (lane >> 5);
    const float a = acc[4 * g], b = acc[4 * g + 1], c = acc[4 * g + 2], d = acc[4 * g + 3];
    if (ldt == TT_F32) {
      *reinterpret_cast<float4*>(static_cast<float*>(logits) + at) = float4{a, b, c, d};
    } else {
      const uint2 v = pack4<ET>(a, b, c, d);  // the logits dtype is the inputs'
      *reinterpret_cast<uint2*>(static_cast<uint16_t*>(logits) + at) = v;
    }
  }
}

// Tokens x experts per block by the number of 32x32 tiles: 32x32 (two chunks a
// stage, four stages) while they make about a block per CU, 32x64 (three
// stages) while those do, 64x64 (two stages) above, which reads x once per 64
// experts and w once per 64 tokens. Logits and top-k, one-kernel gate / 32x32 /
// 32x64 / 64x64 (tiles): H 2048, E 128, 1000 tokens (128) 23.0 / 13.9 / 15.3 /
// 16.0 us, 4000 (500) 23.9 / 23.0 / 18.3 / 20.0, 8192 (1024) 25.5 / 32.1 / 25.4
// / 24.9; H 7168, E 256, 1000 (256) 67.7 / 32.0 / 35.2 / 42.8, 2000 (504) 67.4 /
// 47.9 / 37.1 / 43.4, 4000 (1000) 69.5 / 80.9 / 51.1 / 53.3, 8192 (2048) 71.6 /
// 127 / 80.6 / 59.1; H 4096, E 224, 1000 (224) 42.2 / 22.7 / 24.4 / 26.2, 8192
// (1792) 45.3 / 104 / 72.2 / 40.0; H 4096, E 64, 8192 (512) 30.5 / 39.1 / 30.5 /
// 31.5. What is left is the chain of dependent MFMAs (H / 16 of them).
constexpr int64_t GL_TILES1 = 288, GL_TILES2 = 576;

template <int MT, int NE, int CH, int S>
int launch_gate_logits(const void* x, const void* w, int dtype, int64_t T, int H, int E, int ldt,
                       void* logits, hipStream_t s) {
  const dim3 grid((unsigned)((T + 32 * MT - 1) / (32 * MT)),
                  (unsigned)((E + 32 * NE - 1) / (32 * NE)));
  if (dtype == TT_BF16)
    hipLaunchKernelGGL((gate_logits_kernel<TT_BF16, MT, NE, CH, S>), grid, dim3(GL_NT), 0, s,
                       static_cast<const char*>(x), static_cast<const char*>(w), T, H, E, ldt,
                       logits);
  else
    hipLaunchKernelGGL((gate_logits_kernel<TT_F16, MT, NE, CH, S>), grid, dim3(GL_NT), 0, s,
                       static_cast<const char*>(x), static_cast<const char*>(w), T, H, E, ldt,
                       logits);
  return tt_check_launch("router_gate_logits");
}

}  // namespace

int tt_gate_logits(const void* x, const void* w, int dtype, int64_t T, int H, int E, int ldt,
                   void* logits, hipStream_t s) {
  const int64_t tiles = (T + 31) / 32 * (E / 32);
  if (tiles <= GL_TILES1)
    return launch_gate_logits<1, 1, 2, 4>(x, w, dtype, T, H, E, ldt, logits, s);
  if (tiles <= GL_TILES2)
    return launch_gate_logits<1, 2, 2, 3>(x, w, dtype, T, H, E, ldt, logits, s);
  return launch_gate_logits<2, 2, 2, 2>(x, w, dtype, T, H, E, ldt, logits, s);
}
