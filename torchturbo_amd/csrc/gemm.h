// Building blocks shared by the grouped-GEMM kernels: MFMA wrappers, buffer
// resources, loads straight into LDS, fragment reads and conversions.
#pragma once

#include "common.h"

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) short i16x4;
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
typedef __attribute__((address_space(3))) char lds_char;

enum { MODE_FWD = 0, MODE_DGRAD = 1, MODE_WGRAD = 2 };

template <int ET>
struct Mma;
template <>
struct Mma<TT_BF16> {
  static __device__ __forceinline__ f32x16 run(const uint4& a, const uint4& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                    __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
};
template <>
struct Mma<TT_F16> {
  static __device__ __forceinline__ f32x16 run(const uint4& a, const uint4& b, const f32x16& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                   __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
};

__device__ __forceinline__ int xcd_remap(int b, int nb) {
  const int q = nb / 8, r = nb % 8;
  const int xcd = b % 8, pos = b / 8;
  return xcd < r ? xcd * (q + 1) + pos : r * (q + 1) + (xcd - r) * q + pos;
}

// A block-uniform 64-bit value (read from LDS) into scalar registers.
__device__ __forceinline__ int64_t rfl64(int64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)hi << 32) | lo);
}

// Operand layouts per mode: A is K-major except in wgrad; B is K-major for
// fwd with trans_b and dgrad without.
template <int MODE, bool TRANS_B>
struct Layout {
  static constexpr bool A_K = MODE != MODE_WGRAD;
  static constexpr bool B_K = (MODE == MODE_FWD) ? TRANS_B : (MODE == MODE_DGRAD ? !TRANS_B : false);
};

constexpr uint32_t DM_OOB = 0xFFFFFFF0u;    // buffer offset past any resource
// Gathered A rows: the offset of a row past an expert's end, past any gathered
// source (sources are smaller than 2 GiB) with room for the chunk and k-tile
// offsets added to it.
constexpr uint32_t GA_NOROW = 0x80000000u;

typedef __attribute__((ext_vector_type(4))) int i32x4;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) u32x2 lds_u32x2;

// Buffer resource over [base, base + bytes): offsets at or past `bytes` read
// as zeros. Word 3 is the raw 32-bit data format of the gfx9 family.
__device__ __forceinline__ i32x4 make_rsrc(const void* base, int64_t bytes) {
  const uint64_t b = reinterpret_cast<uint64_t>(base);
  const uint32_t n = bytes <= 0 ? 0u : (bytes < (int64_t)DM_OOB ? (uint32_t)bytes : DM_OOB);
  i32x4 r;
  r.x = __builtin_amdgcn_readfirstlane((int)(uint32_t)b);
  r.y = __builtin_amdgcn_readfirstlane((int)((uint32_t)(b >> 32) & 0xFFFFu));
  r.z = __builtin_amdgcn_readfirstlane((int)n);
  r.w = 0x00020000;
  return r;
}

// The resource moved `adv` bytes along (scalar arithmetic): an offset from
// the new base is in range exactly when the same offset plus adv was before,
// and nothing is once adv passes the end.
__device__ __forceinline__ i32x4 advance_rsrc(i32x4 r, uint32_t adv) {
  const uint64_t b = (((uint64_t)(uint32_t)r.y << 32) | (uint32_t)r.x) + adv;  // stride 0
  i32x4 o;
  o.x = (int)(uint32_t)b;
  o.y = (int)(uint32_t)(b >> 32);
  // records - adv, or 0 on a borrow (SCC), in scalar instructions: the
  // compiler's saturating subtract is a vector one.
  uint32_t n;
  asm("s_sub_u32 %0, %1, %2\n\ts_cselect_b32 %0, 0, %0" : "=s"(n) : "s"(r.z), "s"(adv) : "scc");
  o.z = (int)n;
  o.w = r.w;
  return o;
}

// One 16-byte buffer load per lane straight into LDS at lds_addr + 16 * lane
// (lds_addr is wave-uniform and goes to M0). Inline assembly, so that the
// compiler does not drain outstanding loads before every LDS read:
// completion of a stage is awaited explicitly (TT_WAIT_VMCNT) before the
// barrier that publishes it. Nothing else in these kernels uses M0.
__device__ __forceinline__ void dma16(uint32_t voff, i32x4 rsrc, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :
               : "s"(lds_addr), "v"(voff), "s"(rsrc)
               : "memory");
}

// The same with the streaming cache policy, for data that one block reads once.
__device__ __forceinline__ void dma16_stream(uint32_t voff, i32x4 rsrc, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds"
               :
               : "s"(lds_addr), "v"(voff), "s"(rsrc)
               : "memory");
}

// One dword per lane into LDS at m0 + 4 lane (row indices of a gathered operand).
__device__ __forceinline__ void dma4(uint32_t voff, i32x4 rsrc, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds"
               :
               : "s"(lds_addr), "v"(voff), "s"(rsrc)
               : "memory");
}

__device__ __forceinline__ uint32_t lds_addr_of(lds_char* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>(p));
}

// s_waitcnt with only vmcnt = n (gfx9 encoding: vmcnt[3:0] | vmcnt[5:4] << 14,
// expcnt and lgkmcnt left at their maxima).
#define TT_WAIT_VMCNT(n) \
  __builtin_amdgcn_s_waitcnt(((n) & 0xF) | ((((n) >> 4) & 3) << 14) | (0x7 << 4) | (0xF << 8))

__device__ __forceinline__ uint4 read_k(lds_char* tile, uint32_t off) {
  return __builtin_bit_cast(uint4, *reinterpret_cast<const lds_u32x4*>(tile + off));
}
// Four fp32 values -> four 16-bit values (hardware round to nearest even).
template <int ET>
__device__ __forceinline__ uint2 pack4(float a, float b, float c, float d) {
  if constexpr (ET == TT_BF16) {
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
    const bf16x2 lo = {(__bf16)a, (__bf16)b}, hi = {(__bf16)c, (__bf16)d};
    return uint2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
  } else {
    typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
    const f16x2 lo = {(_Float16)a, (_Float16)b}, hi = {(_Float16)c, (_Float16)d};
    return uint2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
  }
}

typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
// Four e4m3 bytes -> four bf16 (two dwords), each bf16(f32(q) * s).
__device__ __forceinline__ uint2 deq4(uint32_t q, float s) {
  const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)q, false);
  const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)q, true);
  const bf16x2_t a = {(__bf16)(lo.x * s), (__bf16)(lo.y * s)};
  const bf16x2_t b = {(__bf16)(hi.x * s), (__bf16)(hi.y * s)};
  return uint2{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b)};
}

// K-major 64-deep tile: LDS row r (128 bytes) holds tile row r, its 16-byte
// chunk c in slot c ^ ((r >> 1) & 7): any 16 consecutive rows then cover the
// 16 distinct 16-byte bank groups of a 256-byte bank line, so a fragment
// read (one chunk of 32 rows per half-wave) is free of bank conflicts.
// Fragment for k-step s (0..3): rows r0 + lane % 32, chunk 2 s + lane / 32;
// further 32-row blocks add 4096.
__device__ __forceinline__ uint32_t fragk64(int r0, int s, int lane) {
  const int r = r0 + (lane & 31);
  const int c = 2 * s + (lane >> 5);
  return (uint32_t)(r * 128 + ((c ^ ((r >> 1) & 7)) << 4));
}

// Barrier that also publishes this wave's LDS stores and retires its LDS
// reads: wait for them, then s_barrier; the memory clobber keeps the
// compiler from moving LDS accesses across it. Loads in flight (vmcnt) are
// not waited for.
#define TT_LDS_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")

// Tile of a grid with one block per (expert, row tile, column tile).
struct RowTile {
  int e, mt, nt;
  int64_t seg0, nrows;
};

// The block's (expert, row tile, column tile) from the per-expert counts:
// consecutive slots, an expert's row tiles of one column tile first (they
// share its weights), on one XCD. Returns false past the last slot. `scratch`:
// at least 256 bytes of LDS, free again afterwards; NT threads.
template <int BM, int NT>
__device__ __forceinline__ bool row_tile(const int64_t* __restrict__ counts, int E, int tiles_j,
                                          char* scratch, RowTile& t) {
  int64_t* const wrow = reinterpret_cast<int64_t*>(scratch);
  int64_t* const found_seg = wrow + NT / 64;
  int* const wtile = reinterpret_cast<int*>(found_seg + 2);
  int* const found = wtile + NT / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int per = (E + NT - 1) / NT;
  int64_t r = 0;
  int tl = 0;
  for (int i = 0; i < per; ++i) {
    const int e = tid * per + i;
    const int64_t c = e < E ? counts[e] : 0;
    r += c;
    tl += (int)((c + BM - 1) / BM);
  }
  int64_t ri = r;
  int ti = tl;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int64_t o = __shfl_up(ri, off, 64);
    const int ot = __shfl_up(ti, off, 64);
    if (lane >= off) {
      ri += o;
      ti += ot;
    }
  }
  if (lane == 63) {
    wrow[wave] = ri;
    wtile[wave] = ti;
  }
  __syncthreads();
  int64_t rb = 0;
  int tb = 0, total = 0;
#pragma unroll
  for (int w = 0; w < NT / 64; ++w) {
    if (w < wave) {
      rb += wrow[w];
      tb += wtile[w];
    }
    total += wtile[w];
  }
  rb += ri - r;
  tb += ti - tl;
  total *= tiles_j;
  if ((int)blockIdx.x >= total) return false;
  const int slot = xcd_remap(blockIdx.x, total);
  if (slot >= tb * tiles_j && slot < (tb + tl) * tiles_j) {
    for (int i = 0;; ++i) {
      const int e = tid * per + i;
      const int64_t c = counts[e];
      const int m = (int)((c + BM - 1) / BM);
      if (slot < (tb + m) * tiles_j) {
        const int local = slot - tb * tiles_j;
        found[0] = e;
        found[1] = local % m;
        found[2] = local / m;
        found_seg[0] = rb;
        found_seg[1] = c;
        break;
      }
      rb += c;
      tb += m;
    }
  }
  __syncthreads();
  t.e = __builtin_amdgcn_readfirstlane(found[0]);
  t.mt = __builtin_amdgcn_readfirstlane(found[1]);
  t.nt = __builtin_amdgcn_readfirstlane(found[2]);
  t.seg0 = rfl64(found_seg[0]);
  t.nrows = rfl64(found_seg[1]);
  __syncthreads();  // the scratch is the first stage's memory
  return true;
}

}  // namespace

// fwd / dgrad for experts of few rows (gmm_thin.hip): operands as
// tt_gmm_fwd / tt_gmm_dgrad, already checked; see thin_row_limit in gmm.hip. With
// arow, activation row r is row arow[r] of p0 (src_rows rows, under 2 GiB).
int tt_gmm_thin(int mode, bool tb, int dtype, const void* p0, const void* p1, void* out,
                int64_t M, int64_t K, int64_t N, int E, const int64_t* counts, hipStream_t s,
                const int32_t* arow = nullptr, int64_t src_rows = 0);
// Weight gradient for experts of few rows (gmm_wgrad_thin.hip): operands as
// tt_gmm_wgrad, already checked; see wgrad_thin in gmm.hip.
int tt_gmm_wgrad_thin(bool tb, int dtype, const void* x, const void* dy, void* dw, int64_t M,
                      int64_t K, int64_t N, int E, const int64_t* counts, hipStream_t s);
// tt_gmm_thin with e4m3 weights and block scales, as tt_gmm_fp8_fwd / _dgrad, at
// most TT_THIN8_SCALES scale blocks along the reduction; see thin8_rows in
// gmm.hip.
#define TT_THIN8_SCALES 128
int tt_gmm_thin8(int mode, const void* p0, const uint8_t* qw, const void* scale, int sdt,
                 void* out, int64_t M, int64_t K, int64_t N, int E, const int64_t* counts,
                 hipStream_t s, const int32_t* arow = nullptr, int64_t src_rows = 0);

// fc1 of a forward over few rows with the token rows gathered (gmm.hip): 1
// when the launch was made, 0 when the shape takes another kernel (the caller
// permutes), or an error. scale (with its dtype) for e4m3 weights [E, N, K],
// else w is 16-bit [E, K, N].
int tt_gmm_rows_fwd(const void* x, int64_t src_rows, const int32_t* arow, const void* w,
                    const void* scale, int sdt, int dtype, int64_t M, int64_t K, int64_t N, int E,
                    const int64_t* counts, void* y, hipStream_t s);

// Router logits of few tokens (gate.hip): logits [T, E] = x [T, H] w [E, H]^T
// in 16 bits (dtype), E a multiple of 32, H of 64; ldt is TT_F32 or dtype.
int tt_gate_logits(const void* x, const void* w, int dtype, int64_t T, int H, int E, int ldt,
                   void* logits, hipStream_t s);
