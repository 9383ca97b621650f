// Grouped GEMM, forward and data gradient, for experts of few rows (gfx950).
//
// With a few rows per expert the launch streams every used expert's weights
// once and is bound by that stream. The persistent 256x256 kernel of gmm.hip
// holds one block per CU: a tile's prologue and epilogue leave the CU's
// memory path idle, and its few tiles (48 for one token of Qwen3-30B-A3B's
// fc1) leave most CUs idle. Here a block computes BM x 128 outputs over the
// whole reduction, small enough that two blocks share a CU and one streams
// while the other starts or ends.
#include "gemm.h"

#include <type_traits>

namespace {

constexpr int T_BN = 128, T_BK = 64, T_NT = 256;
// Up to this many bytes of weights (half the memory-side cache) a launch
// reads with the default policy: they may still be cached from the last call.
// Larger streams only push each other out, and the streaming policy reads
// them faster: 119 experts of 2048 x 1536 (751 MB) 120 us, 6.3 TB/s, against
// 135 us with the default policy; 8 of them (50 MB, cached) 20 against 15 us.
constexpr int64_t T_CACHED = 128 << 20;
// Rows per expert on average up to which tiles have 64 rows. 64- / 128-row
// tiles, even loads and ones skewed by a Zipf(0.8) / Zipf(1.1) prior: 128 experts
// of 2048 x 1536 fwd at 48 rows 157 + 161 + 133 / 158 + 163 + 126 us, at 60 155 +
// 168 + 150 / 161 + 164 + 150, at 66 183 + 168 + 159 / 162 + 170 + 156, dgrad at
// 48 155 + 155 + 132 / 161 + 165 + 127, at 66 190 + 168 + 157 / 172 + 185 + 158;
// 16 of 1536 x 4096 fwd at 48 35 + 45 + 45 / 34 + 57 + 57; 64 of 1024 x 1408 fwd
// at 48 34 + 37 + 40 / 41 + 42 + 40, at 66 40 + 42 + 42 / 43 + 43 + 42.
constexpr int64_t T_ROWS64 = 60;
constexpr int T_B = T_BN * T_BK * 2;  // weight tile (16 KiB)

// Byte offset of row r of a tile (first packed row `at`, `rows` valid): from
// the tile's first row, or, with rows gathered through arow, in the source
// [src_rows, R]. Gathered rows past the expert's end, or out of the source,
// read as zeros: T_NOROW and a lane's chunk lie past any resource (sources are
// smaller than 2 GiB), as rows past the packed tile's resource do.
constexpr uint32_t T_NOROW = 0x80000000u;
__device__ __forceinline__ uint32_t thin_row_offset(const int32_t* __restrict__ arow, int64_t at,
                                                    int r, int64_t rows, int64_t src_rows,
                                                    int64_t R) {
  if (arow == nullptr) return (uint32_t)(r * R * 2);
  if (r >= rows) return T_NOROW;
  const uint32_t v = (uint32_t)arow[at + r];
  return v < (uint64_t)src_rows ? (uint32_t)(v * R * 2) : T_NOROW;
}

// Epilogue: the BM x 128 tile row-major through LDS (256-byte rows, 16-byte
// chunk c of row r in slot c ^ (r % 16)), stored as whole row segments.
// Block mi, register 4g + e of lane l is row 32 mi + l % 32, column
// 32 wave + 8 g + 4 (l / 32) + e. row0: the tile's first output row; rows: its
// valid ones.
template <int ET, int BM>
__device__ __forceinline__ void thin_store(const f32x16 (&acc)[BM / 32], char* out, lds_char* lds,
                                           int64_t row0, int64_t rows, int64_t j0, int64_t J,
                                           int lane, int wave) {
  TT_LDS_BARRIER();  // every wave is past its fragment reads
#pragma unroll
  for (int mi = 0; mi < BM / 32; ++mi)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int r = 32 * mi + (lane & 31), c = 4 * wave + g;
      const uint2 v = pack4<ET>(acc[mi][4 * g], acc[mi][4 * g + 1], acc[mi][4 * g + 2],
                                acc[mi][4 * g + 3]);
      *reinterpret_cast<lds_u32x2*>(lds + r * 256 + ((c ^ (r & 15)) << 4) + 8 * (lane >> 5)) =
          u32x2{v.x, v.y};
    }
  __syncthreads();
  const int c = threadIdx.x & 15;
  if (j0 + 8 * c >= J) return;
#pragma unroll
  for (int p = 0; p < BM / 16; ++p) {
    const int r = 16 * p + (threadIdx.x >> 4);
    if (r < rows)
      *reinterpret_cast<uint4*>(out + ((row0 + r) * J + j0 + 8 * c) * 2) =
          read_k(lds, (uint32_t)(r * 256 + ((c ^ (r & 15)) << 4)));
  }
}

// One block computes BM x 128 outputs of one expert; wave w owns columns
// 32 w .. 32 w + 31 of every row, so each weight fragment is read from LDS
// once. The 64-deep k-tiles stream into a ring of S LDS stages (weights
// 16 KiB, activations 128 bytes per row), S - 1 of them in flight or being
// waited for, with one barrier per k-tile: it publishes k-tile kt and frees
// the stage of kt - 1, into which kt + S - 1 is then loaded. Resources end at
// the expert's rows and weights, so rows past them read as zeros without
// memory traffic; a K-major reduction tail (KMASK) is masked per chunk.
template <int MODE, bool TRANS_B, int ET, bool KMASK, int BM, int S, int OCC>
__global__ __launch_bounds__(T_NT, OCC) void gmm_thin_kernel(
    const char* __restrict__ p0, const char* __restrict__ p1, char* __restrict__ out, int64_t K,
    int64_t N, int E, const int64_t* __restrict__ counts, int tiles_j, int stream,
    const int32_t* __restrict__ arow, int64_t src_rows) {
  constexpr bool B_K = Layout<MODE, TRANS_B>::B_K;
  constexpr int T_A = BM * T_BK * 2, STAGE = T_A + T_B;
  constexpr int FM = BM / 32;           // 32-row blocks
  constexpr int LA = BM / 32, LD = 4 + LA;  // loads per wave and k-tile
  __shared__ __align__(16) char lds_raw[S * STAGE];
  RowTile t;
  if (!row_tile<BM, T_NT>(counts, E, tiles_j, lds_raw, t)) return;
  const int64_t R = MODE == MODE_FWD ? K : N, J = MODE == MODE_FWD ? N : K;
  const int64_t ldb = TRANS_B ? K : N;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nkt = (int)((R + T_BK - 1) / T_BK);
  const int64_t i0 = (int64_t)t.mt * BM, j0 = (int64_t)t.nt * T_BN;
  const int64_t rows = t.nrows - i0;  // valid rows of the tile, at least one

  // Weights that only this block reads go past the caches.
  const bool once = stream && t.nrows <= BM;

  // Resources at the tile origin, advanced by a k-tile at a time.
  const i32x4 ra = arow != nullptr
                       ? make_rsrc(p0, src_rows * R * 2)
                       : make_rsrc(p0 + (t.seg0 + i0) * R * 2, (rows < BM ? rows : BM) * R * 2);
  const char* wb = p1 + (int64_t)t.e * K * N * 2;
  const int64_t boff = B_K ? j0 * ldb * 2 : j0 * 2;
  const i32x4 rb = make_rsrc(wb + boff, K * N * 2 - boff);
  const uint32_t ks_a = T_BK * 2, ks_b = B_K ? T_BK * 2 : (uint32_t)(T_BK * ldb * 2);

  // Loads, 1 KiB per instruction. A: rows (BM / 4) w + 8 q + lane / 8, chunk
  // slot lane % 8 holding chunk slot ^ ((row >> 1) & 7); K-major weights the
  // same with rows 32 w + 8 q. MN-major weights: k-rows 16 w + 4 q + lane / 16
  // of 256 bytes, slot lane % 16 holding chunk slot ^ (4 (k-row % 4)).
  uint32_t aoff[LA], boffs[4];
  int akof[LA], bkof[4];
#pragma unroll
  for (int q = 0; q < LA; ++q) {
    const int r = 8 * LA * wave + 8 * q + (lane >> 3);
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    akof[q] = 8 * c;
    aoff[q] = thin_row_offset(arow, t.seg0 + i0, r, rows, src_rows, R) + (uint32_t)(16 * c);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if constexpr (B_K) {
      const int r = 32 * wave + 8 * q + (lane >> 3);
      const int c = (lane & 7) ^ ((r >> 1) & 7);
      bkof[q] = 8 * c;
      boffs[q] = (uint32_t)((r * ldb + 8 * c) * 2);
    } else {
      const int kr = 16 * wave + 4 * q + (lane >> 4);
      const int c = (lane & 15) ^ (4 * (kr & 3));
      bkof[q] = 0;
      boffs[q] = (uint32_t)((kr * ldb + 8 * c) * 2);
    }
  }
  lds_char* const lds = (lds_char*)lds_raw;
  auto issue = [&](int kt, int slot) {
    const uint32_t base = lds_addr_of(lds) + (uint32_t)slot * STAGE;
    const i32x4 rbk = advance_rsrc(rb, (uint32_t)kt * ks_b);
    const i32x4 rak = advance_rsrc(ra, (uint32_t)kt * ks_a);
    uint32_t off[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      off[q] = KMASK && B_K && kt * T_BK + bkof[q] >= (int)R ? DM_OOB : boffs[q];
    const uint32_t wbase = base + T_A + (uint32_t)(4 * wave) * 1024u;
    if (once) {
#pragma unroll
      for (int q = 0; q < 4; ++q) dma16_stream(off[q], rbk, wbase + q * 1024u);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) dma16(off[q], rbk, wbase + q * 1024u);
    }
#pragma unroll
    for (int q = 0; q < LA; ++q) {
      dma16(KMASK && kt * T_BK + akof[q] >= (int)R ? DM_OOB : aoff[q], rak, base + (uint32_t)(LA * wave + q) * 1024u);
    }
  };

  // Fragment offsets within a stage.
  uint32_t fa[4], fb[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    fa[s] = fragk64(0, s, lane);
    if constexpr (B_K) {
      fb[s] = T_A + fragk64(32 * wave, s, lane);
    } else {
      const int g = lane >> 4, i = lane & 15;
      const int col = 32 * wave + 16 * (g & 1) + 4 * (i & 3);
      const int kr = 16 * s + 8 * (g >> 1) + (i >> 2);
      fb[s] = T_A + (uint32_t)(kr * 256 + (((col >> 3) ^ (4 * (kr & 3))) << 4) + (col & 7) * 2);
    }
  }
  f32x16 acc[FM] = {};
  const int nmi = __builtin_amdgcn_readfirstlane((int)((rows + 31) / 32));  // blocks with rows

#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    if (s < nkt) issue(s, s);
  // The k-loop for the NM 32-row blocks that hold rows.
  auto loop = [&](auto nm_c) {
    constexpr int NM = decltype(nm_c)::value;
    int slot = 0;
    for (int kt = 0; kt < nkt; ++kt) {
      // k-tile kt has landed once at most the later ones are outstanding.
      const int later = nkt - 1 - kt;
      if (S >= 4 && later >= 2) TT_WAIT_VMCNT(2 * LD);
      else if (S >= 3 && later >= 1) TT_WAIT_VMCNT(LD);
      else TT_WAIT_VMCNT(0);
      TT_LDS_BARRIER();
      const int nslot = slot == 0 ? S - 1 : slot - 1;  // the stage of kt - 1
      if (kt + S - 1 < nkt) issue(kt + S - 1, nslot);
      lds_char* const stg = lds + slot * STAGE;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        uint4 b;
        if constexpr (B_K) {
          b = read_k(stg, fb[s]);
        } else {
          const i16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(stg + fb[s]));
          const i16x4 v1 =
              __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(stg + fb[s] + 1024));
          const uint2 w0 = __builtin_bit_cast(uint2, v0), w1 = __builtin_bit_cast(uint2, v1);
          b = uint4{w0.x, w0.y, w1.x, w1.y};
        }
#pragma unroll
        for (int mi = 0; mi < NM; ++mi)
          acc[mi] = Mma<ET>::run(b, read_k(stg, fa[s] + mi * 4096), acc[mi]);
      }
      slot = slot == S - 1 ? 0 : slot + 1;
    }
  };
  if (FM == 1 || nmi == 1) loop(std::integral_constant<int, 1>{});
  else if (FM == 2 || nmi == 2) loop(std::integral_constant<int, (FM < 2 ? FM : 2)>{});
  else if (nmi == 3) loop(std::integral_constant<int, (FM < 3 ? FM : 3)>{});
  else loop(std::integral_constant<int, FM>{});

  thin_store<ET, BM>(acc, out, lds, t.seg0 + i0, rows, j0, J, lane, wave);
}

// The same for e4m3 weights [E, N, K] with 128 x 128 block scales, dequantised
// in registers to bf16(f32(q) * f32(scale)). k-tiles are 128 deep, so that a
// K-major weight row is a whole 128-byte line and a block has one scale per
// k-tile (T_BN is the scale blocks' width), kept in two registers across the
// lanes. fwd reads 16 bytes of a row per lane, two MFMA steps at once: lane
// half h reads reduction elements 32 p + 16 h .. + 15 of step pair p, and the
// halves exchange eight of them, so that each step multiplies 16 consecutive
// elements as gmm_q8_kernel does: the same bits whichever kernel a launch
// takes. dgrad reads N-major weight rows with the transposing 8-bit read (two
// lanes per row and 16 columns). LDS: weights 16 KiB, activations 256 bytes per row, as two
// 64-deep tiles. Measured on DeepSeek-V3's fc1 and fc2 (256 experts), forward,
// gmm_q8_kernel / this kernel: one token 187 + 58 / 49 + 25 us, 24 tokens (137
// experts used) 947 + 470 / 610 + 319 us (6.6 TB/s), 1024 tokens 1718 + 879 /
// 1418 + 802; data gradient at 512 tokens 1567 + 751 / 1353 + 630.
__device__ __forceinline__ void swap_halves(uint32_t& a, uint32_t& b) {
  // The upper 32 lanes of a against the lower 32 of b.
  const auto v = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = v[0];
  b = v[1];
}

constexpr int T8_BK = 128;
constexpr int T8_SMAX = TT_THIN8_SCALES;  // scale blocks along the reduction
static_assert(T8_SMAX == 128, "two registers of one scale per lane");
// Rows per expert on average up to which tiles have 32 rows (three stages, 72
// KiB of LDS) rather than 64 (two, 64 KiB): at 16 rows per expert fc1 + fc2
// forward 1213 + 689 / 1276 + 744 us, data gradient 1353 + 630 / 1414 + 645; at
// 32 rows 1614 + 887 / 1418 + 802 and 1732 + 816 / 1575 + 718.
// Even loads and ones skewed by a Zipf(0.8) / Zipf(1.1) prior, 32- / 64-row
// tiles: fc1 forward at 16 rows 1244 + 1136 + 807 / 1315 + 1110 + 715, at 20 1271 +
// 1239 + 958 / 1335 + 1202 + 849, at 24 1345 + 1398 + 1033 / 1368 + 1314 + 891,
// data gradient at 20 1402 + 1310 + 978 / 1449 + 1214 + 866.
constexpr int64_t T8_ROWS32 = 20;

template <int MODE, bool KMASK, int BM, int S, int OCC>
__global__ __launch_bounds__(T_NT, OCC) void gmm_thin8_kernel(
    const char* __restrict__ p0, const char* __restrict__ qw, const char* __restrict__ scale,
    int sdt, char* __restrict__ out, int64_t K, int64_t N, int E,
    const int64_t* __restrict__ counts, int tiles_j, int stream,
    const int32_t* __restrict__ arow, int64_t src_rows) {
  constexpr bool FW = MODE == MODE_FWD;
  constexpr int T_A = BM * T8_BK * 2, STAGE = T_A + T_B;
  constexpr int FM = BM / 32;
  constexpr int LA = BM / 16, LD = 4 + LA;  // loads per wave and k-tile
  __shared__ __align__(16) char lds_raw[S * STAGE];
  RowTile t;
  if (!row_tile<BM, T_NT>(counts, E, tiles_j, lds_raw, t)) return;
  const int64_t R = FW ? K : N, J = FW ? N : K;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nkt = (int)((R + T8_BK - 1) / T8_BK);
  const int64_t i0 = (int64_t)t.mt * BM, j0 = (int64_t)t.nt * T_BN;
  const int64_t rows = t.nrows - i0;
  const bool once = stream && t.nrows <= BM;
  const i32x4 ra = arow != nullptr
                       ? make_rsrc(p0, src_rows * R * 2)
                       : make_rsrc(p0 + (t.seg0 + i0) * R * 2, (rows < BM ? rows : BM) * R * 2);
  const int64_t boff = FW ? j0 * K : j0;
  const i32x4 rb = make_rsrc(qw + (int64_t)t.e * K * N + boff, K * N - boff);
  const uint32_t ks_b = FW ? (uint32_t)T8_BK : (uint32_t)(T8_BK * K);

  // Loads. A, 64-deep half q / (LA / 2): rows (BM / 4) w + 8 (q % (LA / 2)) +
  // lane / 8, chunk slot lane % 8 holding chunk slot ^ ((row >> 1) & 7).
  // Weights, 8 rows of 128 bytes per instruction, rows 32 w + 8 q + lane / 8:
  // fwd (columns) swizzled like A; dgrad (k-rows) slot holding chunk
  // slot ^ (2 ((row >> 1) & 3)), which keeps the 16-column chunk pairs.
  uint32_t aoff[LA], boffs[4];
  int akof[LA], bkof[4];
#pragma unroll
  for (int q = 0; q < LA; ++q) {
    const int r = (BM / 4) * wave + 8 * (q % (LA / 2)) + (lane >> 3);
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    akof[q] = 64 * (q / (LA / 2)) + 8 * c;
    aoff[q] = thin_row_offset(arow, t.seg0 + i0, r, rows, src_rows, R) + (uint32_t)(2 * akof[q]);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int r = 32 * wave + 8 * q + (lane >> 3);
    const int c = FW ? (lane & 7) ^ ((r >> 1) & 7) : (lane & 7) ^ (2 * ((r >> 1) & 3));
    bkof[q] = 16 * c;
    boffs[q] = (uint32_t)(r * K + 16 * c);
  }
  lds_char* const lds = (lds_char*)lds_raw;
  auto issue = [&](int kt, int slot) {
    const uint32_t base = lds_addr_of(lds) + (uint32_t)slot * STAGE;
    const i32x4 rbk = advance_rsrc(rb, (uint32_t)kt * ks_b);
    const i32x4 rak = advance_rsrc(ra, (uint32_t)kt * (T8_BK * 2));
    uint32_t off[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      off[q] = KMASK && FW && kt * T8_BK + bkof[q] >= (int)R ? DM_OOB : boffs[q];
    const uint32_t wbase = base + T_A + (uint32_t)(4 * wave) * 1024u;
    if (once) {
#pragma unroll
      for (int q = 0; q < 4; ++q) dma16_stream(off[q], rbk, wbase + q * 1024u);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) dma16(off[q], rbk, wbase + q * 1024u);
    }
#pragma unroll
    for (int q = 0; q < LA; ++q)
      dma16(KMASK && kt * T8_BK + akof[q] >= (int)R ? DM_OOB : aoff[q], rak,
            base + (uint32_t)(q / (LA / 2)) * (BM * 128) +
                (uint32_t)((LA / 2) * wave + q % (LA / 2)) * 1024u);
  };

#pragma unroll
  for (int s = 0; s < S - 1; ++s)
    if (s < nkt) issue(s, s);

  // Scale of k-tile i in lane i % 64 of register i / 64.
  float sv[2];
  {
    const int64_t snb = (N + 127) / 128, skb = (K + 127) / 128;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int i = lane + 64 * h;
      const int64_t at = (int64_t)t.e * snb * skb +
                         (FW ? (int64_t)t.nt * skb + i : (int64_t)i * skb + t.nt);
      sv[h] = 1.0f;
      if (i < nkt)
        sv[h] = sdt == TT_F32 ? reinterpret_cast<const float*>(scale)[at]
                              : bf16_to_f32(reinterpret_cast<const uint16_t*>(scale)[at]);
    }
    asm volatile("" : "+v"(sv[0]), "+v"(sv[1]));  // awaited here, with the first k-tiles
  }

  // Fragment offsets within a stage. A: chunk 2 s + h of the k-tile, in its
  // 64-deep half s / 4.
  uint32_t fa[8], fb[8];
#pragma unroll
  for (int s = 0; s < 8; ++s) {
    const int h = lane >> 5, r = lane & 31;
    const int c = 2 * s + h;  // of 16
    fa[s] = (uint32_t)((c >> 3) * (BM * 128) + r * 128 + (((c & 7) ^ ((r >> 1) & 7)) << 4));
    if constexpr (FW) {  // steps 2 p, 2 p + 1: chunk 2 p + h of row 32 w + lane % 32
      fb[s] = T_A + fragk64(32 * wave, s >> 1, lane);
    } else {
      const int g = lane >> 4, i = lane & 15;
      const int kr = 16 * s + 8 * (g >> 1) + (i >> 1);
      const int ch = (2 * wave + (g & 1)) ^ (2 * ((kr >> 1) & 3));
      fb[s] = T_A + (uint32_t)(kr * 128 + 16 * ch + 8 * (i & 1));
    }
  }
  f32x16 acc[FM] = {};
  const int nmi = __builtin_amdgcn_readfirstlane((int)((rows + 31) / 32));

  auto loop = [&](auto nm_c) {
    constexpr int NM = decltype(nm_c)::value;
    int slot = 0;
    for (int kt = 0; kt < nkt; ++kt) {
      const int later = nkt - 1 - kt;
      if (S >= 4 && later >= 2) TT_WAIT_VMCNT(2 * LD);
      else if (S >= 3 && later >= 1) TT_WAIT_VMCNT(LD);
      else TT_WAIT_VMCNT(0);
      TT_LDS_BARRIER();
      const int nslot = slot == 0 ? S - 1 : slot - 1;
      if (kt + S - 1 < nkt) issue(kt + S - 1, nslot);
      const float sc = __uint_as_float((uint32_t)__builtin_amdgcn_readlane(
          (int)__float_as_uint(kt < 64 ? sv[0] : sv[1]), kt & 63));
      lds_char* const stg = lds + slot * STAGE;
      uint4 pair;
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        uint2 q;
        if constexpr (FW) {
          if ((s & 1) == 0) {
            // Elements 0-7 | 16-23 and 8-15 | 24-31 of the pair's 32 (lower |
            // upper lane half) become 0-7 | 8-15 and 16-23 | 24-31.
            pair = read_k(stg, fb[s]);
            swap_halves(pair.x, pair.z);
            swap_halves(pair.y, pair.w);
          }
          q = (s & 1) ? uint2{pair.z, pair.w} : uint2{pair.x, pair.y};
        } else {
          typedef __attribute__((ext_vector_type(2))) int i32x2_t;
          typedef __attribute__((address_space(3))) i32x2_t lds_i32x2;
          q = __builtin_bit_cast(uint2,
                                 __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i32x2*)(stg + fb[s])));
        }
        const uint2 lo = deq4(q.x, sc), hi = deq4(q.y, sc);
        const uint4 b = uint4{lo.x, lo.y, hi.x, hi.y};
#pragma unroll
        for (int mi = 0; mi < NM; ++mi)
          acc[mi] = Mma<TT_BF16>::run(b, read_k(stg, fa[s] + mi * 4096), acc[mi]);
      }
      slot = slot == S - 1 ? 0 : slot + 1;
    }
  };
  if (FM == 1 || nmi == 1) loop(std::integral_constant<int, 1>{});
  else if (FM == 2 || nmi == 2) loop(std::integral_constant<int, (FM < 2 ? FM : 2)>{});
  else if (nmi == 3) loop(std::integral_constant<int, (FM < 3 ? FM : 3)>{});
  else loop(std::integral_constant<int, FM>{});
  thin_store<TT_BF16, BM>(acc, out, lds, t.seg0 + i0, rows, j0, J, lane, wave);
}

template <int MODE, bool TB, int ET, bool KMASK, int BM, int S, int OCC>
int launch_thin_k(const void* p0, const void* p1, void* out, int64_t M, int64_t K, int64_t N,
                  int E, const int64_t* counts, hipStream_t s, const int32_t* arow,
                  int64_t src_rows) {
  const int64_t J = MODE == MODE_FWD ? N : K;
  const int tj = (int)((J + T_BN - 1) / T_BN);
  // Each used expert adds at most one partial row tile.
  const int64_t nblk = (M / BM + (M < E ? M : E)) * tj;
  if (nblk == 0) return TT_OK;
  TT_REQUIRE(nblk < 0x7fffffff, "gmm: grid too large");
  const int stream = (M < E ? M : E) * K * N * 2 > T_CACHED ? 1 : 0;
  hipLaunchKernelGGL((gmm_thin_kernel<MODE, TB, ET, KMASK, BM, S, OCC>), dim3((unsigned)nblk),
                     dim3(T_NT), 0, s, static_cast<const char*>(p0),
                     static_cast<const char*>(p1), static_cast<char*>(out), K, N, E, counts, tj,
                     stream, arow, src_rows);
  return tt_check_launch("gmm");
}

// 64-row tiles (72 KiB of LDS, three stages) up to an average of T_ROWS64
// rows per expert, 128-row tiles (64 KiB, two stages) above.
template <int MODE, bool TB, int ET>
int launch_thin(const void* p0, const void* p1, void* out, int64_t M, int64_t K, int64_t N,
                int E, const int64_t* counts, hipStream_t s, const int32_t* arow,
                int64_t src_rows) {
  const int64_t R = MODE == MODE_FWD ? K : N;
  if (M <= (int64_t)E * T_ROWS64) {
    if (R % T_BK)
      return launch_thin_k<MODE, TB, ET, true, 64, 3, 2>(p0, p1, out, M, K, N, E, counts, s, arow,
                                                              src_rows);
    return launch_thin_k<MODE, TB, ET, false, 64, 3, 2>(p0, p1, out, M, K, N, E, counts, s, arow,
                                                              src_rows);
  }
  if (R % T_BK)
    return launch_thin_k<MODE, TB, ET, true, 128, 2, 2>(p0, p1, out, M, K, N, E, counts, s, arow,
                                                              src_rows);
  return launch_thin_k<MODE, TB, ET, false, 128, 2, 2>(p0, p1, out, M, K, N, E, counts, s, arow,
                                                              src_rows);
}

template <int MODE, bool KMASK, int BM, int S>
int launch_thin8_k(const void* p0, const uint8_t* qw, const void* scale, int sdt, void* out,
                   int64_t M, int64_t K, int64_t N, int E, const int64_t* counts, hipStream_t s,
                   const int32_t* arow, int64_t src_rows) {
  const int64_t J = MODE == MODE_FWD ? N : K;
  const int tj = (int)((J + T_BN - 1) / T_BN);
  const int64_t nblk = (M / BM + (M < E ? M : E)) * tj;
  if (nblk == 0) return TT_OK;
  TT_REQUIRE(nblk < 0x7fffffff, "gmm_fp8: grid too large");
  const int stream = (M < E ? M : E) * K * N > T_CACHED ? 1 : 0;
  hipLaunchKernelGGL((gmm_thin8_kernel<MODE, KMASK, BM, S, 2>), dim3((unsigned)nblk), dim3(T_NT),
                     0, s, static_cast<const char*>(p0), reinterpret_cast<const char*>(qw),
                     static_cast<const char*>(scale), sdt, static_cast<char*>(out), K, N, E,
                     counts, tj, stream, arow, src_rows);
  return tt_check_launch("gmm_fp8");
}

template <int MODE>
int launch_thin8(const void* p0, const uint8_t* qw, const void* scale, int sdt, void* out,
                 int64_t M, int64_t K, int64_t N, int E, const int64_t* counts, hipStream_t s,
                 const int32_t* arow, int64_t src_rows) {
  const int64_t R = MODE == MODE_FWD ? K : N;
  if (M <= (int64_t)E * T8_ROWS32) {
    if (R % T8_BK)
      return launch_thin8_k<MODE, true, 32, 3>(p0, qw, scale, sdt, out, M, K, N, E, counts, s, arow,
                                              src_rows);
    return launch_thin8_k<MODE, false, 32, 3>(p0, qw, scale, sdt, out, M, K, N, E, counts, s, arow,
                                              src_rows);
  }
  if (R % T8_BK)
    return launch_thin8_k<MODE, true, 64, 2>(p0, qw, scale, sdt, out, M, K, N, E, counts, s, arow,
                                              src_rows);
  return launch_thin8_k<MODE, false, 64, 2>(p0, qw, scale, sdt, out, M, K, N, E, counts, s, arow,
                                              src_rows);
}

}  // namespace

int tt_gmm_thin8(int mode, const void* p0, const uint8_t* qw, const void* scale, int sdt,
                 void* out, int64_t M, int64_t K, int64_t N, int E, const int64_t* counts,
                 hipStream_t s, const int32_t* arow, int64_t src_rows) {
  if (mode == MODE_FWD)
    return launch_thin8<MODE_FWD>(p0, qw, scale, sdt, out, M, K, N, E, counts, s, arow, src_rows);
  return launch_thin8<MODE_DGRAD>(p0, qw, scale, sdt, out, M, K, N, E, counts, s, arow, src_rows);
}

int tt_gmm_thin(int mode, bool tb, int dtype, const void* p0, const void* p1, void* out,
                int64_t M, int64_t K, int64_t N, int E, const int64_t* counts, hipStream_t s,
                const int32_t* arow, int64_t src_rows) {
  auto go = [&](auto mode_c, auto tb_c, auto et_c) {
    return launch_thin<decltype(mode_c)::value, decltype(tb_c)::value, decltype(et_c)::value>(
        p0, p1, out, M, K, N, E, counts, s, arow, src_rows);
  };
  using FW = std::integral_constant<int, MODE_FWD>;
  using DG = std::integral_constant<int, MODE_DGRAD>;
  using BF = std::integral_constant<int, TT_BF16>;
  using HF = std::integral_constant<int, TT_F16>;
  auto typed = [&](auto mode_c, auto et_c) {
    return tb ? go(mode_c, std::true_type{}, et_c) : go(mode_c, std::false_type{}, et_c);
  };
  if (mode == MODE_FWD) return dtype == TT_BF16 ? typed(FW{}, BF{}) : typed(FW{}, HF{});
  return dtype == TT_BF16 ? typed(DG{}, BF{}) : typed(DG{}, HF{});
}
