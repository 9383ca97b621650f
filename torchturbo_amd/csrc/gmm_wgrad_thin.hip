// Grouped GEMM, weight gradient, for experts of few rows (gfx950).
//
// With a few hundred rows per expert an output tile takes little time to
// compute and the launch is bound by writing every expert's gradient. The
// persistent 256x256 kernel of gmm.hip holds one block per CU, so a tile's
// stores and the next tile's products take turns, and it launches a queue
// reset first. Here a block computes one small tile and ends; two (or four)
// blocks share a CU, one storing while another multiplies.
#include "gemm.h"

namespace {

constexpr int W_NT = 256;
// 128 x 128 tiles (32-deep k-tiles, two stages, four blocks per CU) up to this
// many rows per expert on average, or for launches that 256 x 128 tiles leave
// without two blocks for each of 256 CUs; 256 x 128 tiles (16-deep, three
// stages, two blocks per CU), which read fewer operand bytes per output,
// otherwise. 128-row / 256-row tiles: 128 experts of 2048 x 1536 at 16 rows
// 134 / 144 us, 32 rows 131 / 143, 62 rows 146 / 138, 128 rows 180 / 162, 256
// rows 291 / 260; 16 of 4096 x 3072 at 25 rows 66 / 72, 100 rows 81 / 78; 8 of
// 512 x 1024 at 128 rows 8.8 / 9.5, at 500 rows 14.5 / 16.6.
constexpr int64_t W_ROWS128 = 40;
constexpr int64_t W_BLOCKS = 512;
// Consecutive tiles that go to one XCD: 8 x 8 of them share 16 operand panels
// in its L2, and a long expert spreads over all XCDs. In runs of 16 / 32 / 64
// / 128 tiles 128 experts of 2048 x 1536 at 62 rows took 155 / 151 / 144 / 146
// us, an eighth of the launch at a time 162.
constexpr int W_RUN = 64, W_GROUP = 8;

// One block computes BM x BN elements of one expert's gradient out[e] [I, J],
// the sum over its rows r of a[r, i] b[r, j]; each of the four waves takes a
// quarter of the tile. Both operands are MN-major: BK-deep k-tiles (BK rows of
// the expert) stream into a ring of S LDS stages, one barrier per k-tile,
// which publishes k-tile kt and frees the stage of kt - 1, into which kt + S -
// 1 is then loaded. Rows past the expert's end lie past the resources and read
// as zeros; columns past I or J are read from wherever they lead inside the
// resource and never stored. Products are summed in row order, 16 rows per
// step, as in the other kernels: the same bits. Stores bypass L2's retention
// (128 experts of 2048 x 1536 at 62 rows: 145 us, 219 with the default policy,
// whose lines push the operand panels out).
template <int ET, int BM, int BN, int BK, int S, int OCC>
__global__ __launch_bounds__(W_NT, OCC) void gmm_wgrad_thin_kernel(
    const char* __restrict__ a, const char* __restrict__ b, char* __restrict__ out, int I, int J,
    const int64_t* __restrict__ counts, int ti, int tj) {
  constexpr int T_A = BM * BK * 2, T_B = BN * BK * 2, STAGE = T_A + T_B;
  constexpr int FM = BM / 64, FN = BN / 64;  // 32x32 blocks of a wave
  constexpr int LA = T_A / 4096, LB = T_B / 4096, LD = LA + LB;  // loads per wave and k-tile
  // The epilogue goes through the stages in one pass, or in two of BM / 2 rows.
  constexpr int EPI = BM * BN * 2 <= S * STAGE ? 1 : 2, PR = BM / EPI;
  static_assert(PR * BN * 2 <= S * STAGE && S >= 2 && S <= 3, "tile through the stages");
  __shared__ __align__(16) char lds_raw[S * STAGE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

  // Tile: runs of W_RUN go to the XCDs in turn (the rest in order); an
  // expert's tiles in groups of W_GROUP columns, row by row.
  int slot = blockIdx.x;
  if (slot < (int)gridDim.x / (8 * W_RUN) * (8 * W_RUN)) {
    const int p = slot / 8;
    slot = (p / W_RUN * 8 + slot % 8) * W_RUN + p % W_RUN;
  }
  const int e = slot / (ti * tj), local = slot % (ti * tj);
  const int grp = local / (ti * W_GROUP), gl = local % (ti * W_GROUP);
  const int gw = tj - grp * W_GROUP < W_GROUP ? tj - grp * W_GROUP : W_GROUP;
  const int i0 = gl / gw * BM, j0 = (grp * W_GROUP + gl % gw) * BN;
  int64_t seg = 0;  // rows before the expert
  for (int x = lane; x < e; x += 64) seg += counts[x];
#pragma unroll
  for (int o = 32; o; o >>= 1) seg += __shfl_xor(seg, o, 64);
  const int64_t seg0 = rfl64(seg), rows = rfl64(counts[e]);
  const int nkt = (int)((rows + BK - 1) / BK);

  // Loads, 1 KiB per instruction: whole k-rows of the tile (256 or 512 bytes),
  // chunk slot s of k-row r holding chunk s ^ (4 (r % 4)).
  const i32x4 ra = make_rsrc(a + (seg0 * I + i0) * 2, (rows * I - i0) * 2);
  const i32x4 rb = make_rsrc(b + (seg0 * J + j0) * 2, (rows * J - j0) * 2);
  const uint32_t ks_a = (uint32_t)(BK * I * 2), ks_b = (uint32_t)(BK * J * 2);
  constexpr int CA = BM / 8, CB = BN / 8;  // chunks per k-row
  uint32_t aoff[LA], boff[LB];
#pragma unroll
  for (int q = 0; q < LA; ++q) {
    const int r = (LA * wave + q) * (64 / CA) + lane / CA, c = (lane % CA) ^ (4 * (r & 3));
    aoff[q] = (uint32_t)((r * I + 8 * c) * 2);
  }
#pragma unroll
  for (int q = 0; q < LB; ++q) {
    const int r = (LB * wave + q) * (64 / CB) + lane / CB, c = (lane % CB) ^ (4 * (r & 3));
    boff[q] = (uint32_t)((r * J + 8 * c) * 2);
  }
  lds_char* const lds = (lds_char*)lds_raw;
  auto issue = [&](int kt, int sl) {
    const uint32_t base = lds_addr_of(lds) + (uint32_t)sl * STAGE;
    const i32x4 rak = advance_rsrc(ra, (uint32_t)kt * ks_a);
    const i32x4 rbk = advance_rsrc(rb, (uint32_t)kt * ks_b);
#pragma unroll
    for (int q = 0; q < LA; ++q) dma16(aoff[q], rak, base + (uint32_t)(LA * wave + q) * 1024u);
#pragma unroll
    for (int q = 0; q < LB; ++q)
      dma16(boff[q], rbk, base + T_A + (uint32_t)(LB * wave + q) * 1024u);
  };

  // Fragments by transposing reads: k-rows 8 (g / 2) + i / 4 (and 4 further
  // on) of a step, columns col + 16 (g % 2) + 4 (i % 4) .. + 3, for lane i of
  // 16-lane group g.
  const int wm = wave >> 1, wn = wave & 1;
  auto frag_off = [&](int col, int width) {
    const int g = lane >> 4, i = lane & 15;
    const int r = 8 * (g >> 1) + (i >> 2), c = col + 16 * (g & 1) + 4 * (i & 3);
    return (uint32_t)(r * width * 2 + (((c >> 3) ^ (4 * (r & 3))) << 4) + (c & 7) * 2);
  };
  auto frag = [&](lds_char* p, int width) -> uint4 {
    const i16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)p);
    const i16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(p + 8 * width));
    const uint2 w0 = __builtin_bit_cast(uint2, v0), w1 = __builtin_bit_cast(uint2, v1);
    return uint4{w0.x, w0.y, w1.x, w1.y};
  };
  uint32_t fa[FM], fb[FN];
#pragma unroll
  for (int m = 0; m < FM; ++m) fa[m] = frag_off(wm * (BM / 2) + 32 * m, BM);
#pragma unroll
  for (int n = 0; n < FN; ++n) fb[n] = T_A + frag_off(wn * (BN / 2) + 32 * n, BN);

  f32x16 acc[FM][FN] = {};
#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    if (s < nkt) issue(s, s);
  int sl = 0;
  for (int kt = 0; kt < nkt; ++kt) {
    // k-tile kt has landed once at most the later ones are outstanding.
    if (S >= 3 && kt < nkt - 1) TT_WAIT_VMCNT(LD);
    else TT_WAIT_VMCNT(0);
    TT_LDS_BARRIER();
    if (kt + S - 1 < nkt) issue(kt + S - 1, sl == 0 ? S - 1 : sl - 1);
    lds_char* const stg = lds + sl * STAGE;
#pragma unroll
    for (int s = 0; s < BK / 16; ++s) {
      uint4 af[FM], bf[FN];
#pragma unroll
      for (int m = 0; m < FM; ++m) af[m] = frag(stg + fa[m] + s * (32 * BM), BM);
#pragma unroll
      for (int n = 0; n < FN; ++n) bf[n] = frag(stg + fb[n] + s * (32 * BN), BN);
#pragma unroll
      for (int m = 0; m < FM; ++m)
#pragma unroll
        for (int n = 0; n < FN; ++n) acc[m][n] = Mma<ET>::run(bf[n], af[m], acc[m][n]);
    }
    sl = sl == S - 1 ? 0 : sl + 1;
  }

  // Epilogue: row-major through LDS (chunk c of row r in slot c ^ (r % 16)),
  // stored as whole row segments. Block (m, n), register 4 q + x of lane l is
  // row 32 m + l % 32, column 32 n + 8 q + 4 (l / 32) + x of the wave's part.
  char* const o = out + (int64_t)e * I * J * 2;
#pragma unroll
  for (int ps = 0; ps < EPI; ++ps) {
    TT_LDS_BARRIER();  // fragment reads, or the last pass's reads, are done
    if (EPI == 1 || wm == ps) {
#pragma unroll
      for (int m = 0; m < FM; ++m)
#pragma unroll
        for (int n = 0; n < FN; ++n)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int r = (EPI == 1 ? wm * (BM / 2) : 0) + 32 * m + (lane & 31);
            const int c = wn * (BN / 16) + 4 * n + q;
            const uint2 v = pack4<ET>(acc[m][n][4 * q], acc[m][n][4 * q + 1],
                                      acc[m][n][4 * q + 2], acc[m][n][4 * q + 3]);
            *reinterpret_cast<lds_u32x2*>(lds + r * (BN * 2) + ((c ^ (r & 15)) << 4) +
                                          8 * (lane >> 5)) = u32x2{v.x, v.y};
          }
    }
    __syncthreads();
    const int c = threadIdx.x % CB;
    if (j0 + 8 * c < J) {
#pragma unroll
      for (int p = 0; p < PR * CB / W_NT; ++p) {
        const int r = p * (W_NT / CB) + threadIdx.x / CB, i = i0 + ps * PR + r;
        if (i < I)
          __builtin_nontemporal_store(
              __builtin_bit_cast(u32x4, read_k(lds, (uint32_t)(r * (BN * 2) + ((c ^ (r & 15)) << 4)))),
              reinterpret_cast<u32x4*>(o + ((int64_t)i * J + j0 + 8 * c) * 2));
      }
    }
  }
}

template <int ET, int BM, int BN, int BK, int S, int OCC>
int launch(const void* a, const void* b, void* out, int64_t I, int64_t J, int E,
           const int64_t* counts, hipStream_t s) {
  const int ti = (int)((I + BM - 1) / BM), tj = (int)((J + BN - 1) / BN);
  const int64_t nblk = (int64_t)E * ti * tj;
  if (nblk == 0) return TT_OK;
  TT_REQUIRE(nblk < 0x7fffffff, "gmm: grid too large");
  hipLaunchKernelGGL((gmm_wgrad_thin_kernel<ET, BM, BN, BK, S, OCC>), dim3((unsigned)nblk),
                     dim3(W_NT), 0, s, static_cast<const char*>(a), static_cast<const char*>(b),
                     static_cast<char*>(out), (int)I, (int)J, counts, ti, tj);
  return tt_check_launch("gmm");
}

template <int ET>
int launch_et(const void* a, const void* b, void* out, int64_t M, int64_t I, int64_t J, int E,
              const int64_t* counts, hipStream_t s) {
  if (M <= (int64_t)E * W_ROWS128 || E * ((I + 255) / 256) * ((J + 127) / 128) < W_BLOCKS)
    return launch<ET, 128, 128, 32, 2, 4>(a, b, out, I, J, E, counts, s);
  return launch<ET, 256, 128, 16, 3, 2>(a, b, out, I, J, E, counts, s);
}

}  // namespace

int tt_gmm_wgrad_thin(bool tb, int dtype, const void* x, const void* dy, void* dw, int64_t M,
                      int64_t K, int64_t N, int E, const int64_t* counts, hipStream_t s) {
  const void* const a = tb ? dy : x;
  const void* const b = tb ? x : dy;
  const int64_t I = tb ? N : K, J = tb ? K : N;
  return dtype == TT_BF16 ? launch_et<TT_BF16>(a, b, dw, M, I, J, E, counts, s)
                          : launch_et<TT_F16>(a, b, dw, M, I, J, E, counts, s);
}
