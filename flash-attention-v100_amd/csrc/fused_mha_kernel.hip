// FlashAttention-2 forward and backward for gfx950 (CDNA4, wave64, MFMA).
//
// Takes the place of the reference's kernel/fused_mha_kernel.cu (forward
// :20-323, backward :325-735, launchers :891-916) with a different design:
//
//   * Every GEMM runs on v_mfma_f32_32x32x16_f16 or, where all CUs are busy long
//     enough to meet the power cap, v_mfma_f32_16x16x32_f16 (Geom16), with fp32
//     accumulation; either gives the same bits.
//   * A wave owns 32 "resident" sequence positions (queries in the forward and
//     in the dQ pass, keys in the dK/dV pass).  Their rows stay in registers as
//     MFMA B operands for the whole kernel.  The other sequence dimension is
//     streamed through LDS in 64-row tiles shared by the waves of a block.
//   * Tiles go global -> LDS with global_load_lds_dwordx4 (no registers in
//     between) into a ring of two to four slots, two tiles ahead of their use
//     where one work group has the CU (256-query forward, D = 128 backward), one
//     ahead where two share it (128-query forward, D = 64 backward); one barrier
//     per tile.  The LDS layout is XOR-swizzled so that both the row-wise
//     128-bit reads and the transposing ds_read_b64_tr_b16 reads are free of
//     bank conflicts without padding.
//   * The first GEMM is computed transposed, tile^T[streamed][resident], so a
//     lane holds 16 streamed positions of ONE resident position per 32x32
//     block (16 x 16 MFMAs: of two).  Row statistics (max, sum, logsumexp, delta)
//     are therefore plain per-lane scalars plus one exchange between lane groups.
//   * The accumulator registers of the first GEMM, rounded to fp16, are
//     already laid out as the B operand of the second GEMM.  P and dS therefore
//     need no shuffling; they go through LDS only in the D = 128 backward, where
//     the waves of a pair hand P over, lane for lane, and where dS comes back from
//     memory.  The matching A operand (V^T, K^T, Q^T, dO^T) is read
//     transposed out of the same row-major tile.
//   * The backward is split into a dQ pass (query-block parallel) and a dK/dV
//     pass (key-block parallel): no atomics, no fp32 dQ scratch, deterministic.
//   * Work-group ids are remapped so that each XCD (private L2) works on whole
//     (batch, head) slices.
//
// Layouts: q/k/v/o/do/dq/dk/dv are (B, N, H, D) fp16, lse/delta are (B, H, N)
// fp32 (reference: kernel/fused_mha_kernel.cu:57-67).

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <math.h>
#include <mutex>
#include <tuple>
#include <type_traits>
#include <utility>

#include "fused_mha.h"
#include "fmha_internal.h"
#include "block_map.h"


// Backward workspace of fused_mha_backward_noalloc (delta and lse*log2(e), fp32
// (batch, head, n) each): lives in the code object, one copy per GPU, so that
// entry point never allocates.  Host code must not use this name as an address;
// it asks the runtime for the device address once per device (scratch_for_device).
static __device__ __align__(256) unsigned char scratch[2 * (size_t)FUSED_MHA_NOALLOC_MAX_ROWS * sizeof(float)];

namespace {

typedef _Float16 half_t;
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));

constexpr int kResident = 32;      // resident positions per wave
constexpr int kTile = 64;          // streamed rows per LDS tile
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

template <int D>
struct TileGeom {
  static constexpr int kKSteps = D / 16;                   // MFMA k-steps over D
  static constexpr int kDBlocks = D / 32;                  // 32-row blocks over D
};

__device__ __forceinline__ f16v mfma(h8 a, h8 b, f16v c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f4v mfma16(h8 a, h8 b, f4v c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// dS for two neighbouring positions: fp16(-p.lo * x0) and fp16(-p.hi * x1), the products in fp32, as
// two mixed-precision FMAs that read the fp16 halves of p directly (the same bits as converting p to
// fp32, multiplying and converting back, in 2 instructions instead of 5).
typedef unsigned u4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ unsigned neg_mul_to_f16x2(unsigned p_pair, float x0, float x1) {
  unsigned r;
  asm("v_fma_mixlo_f16 %0, %1, -%2, 0 op_sel_hi:[1,0,0]\n\t"
      "v_fma_mixhi_f16 %0, %1, -%3, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]"
      : "=&v"(r)
      : "v"(p_pair), "v"(x0), "v"(x1));
  return r;
}
// y[.] = fp16(-p[.] * x[.]) for the 8 values of one B-operand fragment
__device__ __forceinline__ h8 neg_mul_to_f16x8(h8 p, const float* x) {
  const u4v pp = __builtin_bit_cast(u4v, p);
  u4v r;
#pragma unroll
  for (int j = 0; j < 4; ++j) r[j] = neg_mul_to_f16x2(pp[j], x[2 * j], x[2 * j + 1]);
  return __builtin_bit_cast(h8, r);
}

// Element strides of a (batch, n, head, d) tensor whose last dimension is
// contiguous.  The dense layout of reference kernel/fused_mha_kernel.cu:57-59 is
// {n*head*d, head*d, d}.
struct Strides {
  long b;
  int n, h;
};

// Combine a value with the one held by the lane 32 positions away.
__device__ __forceinline__ float other_half(float x) {
  int xi = __float_as_int(x);
  auto r = __builtin_amdgcn_permlane32_swap(xi, xi, false, false);
  // r[0]: lanes 0-31 keep own, lanes 32-63 get lane-32's; r[1] the converse.
  int mine_or_other = (threadIdx.x & 32) ? r[0] : r[1];
  return __int_as_float(mine_or_other);
}

// Streamed-row index of accumulator register r in row-block rb for half hh.
__device__ __forceinline__ int acc_row(int rb, int r, int hh) {
  return rb * 32 + 8 * (r >> 2) + 4 * hh + (r & 3);
}

// The rows of a staging tile as they leave.  All of them are asked for before the first is stored, and only a block with rows
// past the end looks at each: one after the other, as read, wait, test and store, they take 200 cycles each.
// Kernels in graphs of 20 calls, us one after the other and as it is, forward, then backward, N x slices: D = 64 77 x 8 causal
// 5.76, 5.67 and 6.86, 6.61; 128 x 4 5.15, 5.06 and 6.48, 6.31; 1024 x 64 causal 17.3, 17.2 and 43.4, 43.1; D = 128 200 x 48
// causal 9.45, 9.32 and 14.8 both; 2048 x 80 causal 95.7, 95.4 and 296, 295.
template <int D, int kPitch, typename Piece>
__device__ __forceinline__ void store_staged(half_t* __restrict__ base, int row_stride, int row0, int n, int lane,
                                             const char* __restrict__ stage, int upper_off) {
  constexpr int kLanesPerRow = D / 8, kRowsPerPass = 64 / kLanesPerRow, kPasses = kResident / kRowsPerPass;
  const int r_in = lane / kLanesPerRow, ch = lane % kLanesPerRow;
  union Row {
    Piece piece[16 / sizeof(Piece)];
    h8 v;
  } rows[kPasses];
#pragma unroll
  for (int pass = 0; pass < kPasses; ++pass) {
    const int r = pass * kRowsPerPass + r_in;
    const char* const src = stage + (r & 15) * kPitch + (r >> 4) * upper_off + ch * 16;
#pragma unroll
    for (int e = 0; e < (int)(16 / sizeof(Piece)); ++e) rows[pass].piece[e] = *reinterpret_cast<const Piece*>(src + e * sizeof(Piece));
  }
  char* const out = reinterpret_cast<char*>(base + (long)row0 * row_stride);
  const unsigned off = r_in * row_stride * 2 + ch * 16;
  auto store = [&](int pass) __attribute__((always_inline)) {
    *reinterpret_cast<h8*>(out + (long)pass * kRowsPerPass * 2 * row_stride + off) = rows[pass].v;
  };
  if (row0 + kResident <= n) {
#pragma unroll
    for (int pass = 0; pass < kPasses; ++pass) store(pass);
  } else {
#pragma unroll
    for (int pass = 0; pass < kPasses; ++pass)
      if (row0 + pass * kRowsPerPass + r_in < n) store(pass);
  }
}

// Store a [D][32 resident] fp32 accumulator, scaled, as fp16 rows of a dense
// (B, N, H, D) tensor, through a staging tile in LDS that belongs to the wave
// (32 rows of kStagePitch bytes): each lane first writes the 4-feature pieces it
// holds of its own row, then the wave reads the tile back row-wise, so that
// every row leaves as whole 16-byte pieces written by neighbouring lanes (a
// 256-byte row by 16 lanes, as the reference's epilogue does with its 128-bit
// stores, kernel/fused_mha_kernel.cu:318-322, 714-734).  Lane (i, hh) owns row
// row0 + i; per 32-feature block it holds features 8*g + 4*hh + 0..3 for g = 0..3.
// The caller makes sure (with a block barrier) that nobody still reads what the
// staging tile overwrites.
template <int D>
struct StageGeom {
  // bytes per row: a row plus 8, so that the lanes of a half wave, which write 8 bytes each to
  // 32 different rows, spread over the banks; the rows are read back as 8-byte pieces.
  // (Measured: no bank conflicts with D = 64; with D = 128 four conflict cycles per 8-byte
  // store instruction remain whatever the padding or swizzle, 64 cycles per wave and launch.)
  static constexpr int kPitch = D * 2 + 8;
  static constexpr int kBytes = kResident * kPitch;  // per wave
};
template <int D>
__device__ __forceinline__ void store_resident(half_t* __restrict__ base, int row_stride, int row0, int n,
                                               const f16v (&acc)[TileGeom<D>::kDBlocks], float mul, int lane,
                                               char* __restrict__ stage, int my_row = -1,
                                               int upper_off = 16 * StageGeom<D>::kPitch) {
  // my_row: the row (0..31, relative to row0) this lane's column of the accumulator belongs
  // to, when that is not lane & 31; upper_off: where rows 16..31 are staged, relative to `stage`,
  // when the staging tile is not contiguous (see fmha_bwd_dq_spill_kernel for both)
  constexpr int kPitch = StageGeom<D>::kPitch;
  const int i = my_row < 0 ? (lane & 31) : my_row, hh = lane >> 5;
  char* mine = stage + (i & 15) * kPitch + (i >> 4) * upper_off + hh * 8;
#pragma unroll
  for (int db = 0; db < TileGeom<D>::kDBlocks; ++db) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      h4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (half_t)(acc[db][4 * g + e] * mul);
      *reinterpret_cast<h4*>(mine + (db * 32 + 8 * g) * 2) = v;
    }
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the wave's own writes have landed
  asm volatile("" ::: "memory");
  store_staged<D, kPitch, h4>(base, row_stride, row0, n, lane, stage, upper_off);
}

// Blocks of a persistent work group (schedule: block_map.h).
struct PersistentBlocks {
  int total;
  __device__ __forceinline__ int lin(int r) const {  // >= total: this group has no block in round r
    return fmha_persistent_block(r, blockIdx.x, gridDim.x);
  }
  __device__ __forceinline__ int next_round(int r) const {  // the next round with a block for this group, or -1
    return fmha_persistent_next_round(r, blockIdx.x, gridDim.x, total);
  }
};

// ---------------------------------------------------------------------------
// 64-row tiles copied global -> LDS by global_load_lds_dwordx4 (no registers in
// between).  One wave-level instruction moves 1 KiB: 16 rows x 64 bytes, every
// 4 lanes reading one 64-byte row segment.  The tile is an array of such 1 KiB
// blocks, block (R, C) = rows 16R..16R+15, bytes 64C..64C+63 of each row.
// Inside a block the 16-byte chunk c4 of row r16 sits at
//     r16 * 64 + ((c4 ^ swz(r16 >> 2)) * 16),
// which makes all read patterns below bank-conflict free without padding:
//   rows:  16 lanes read the same chunk of 16 rows      (128-bit reads)
//   cols:  16 lanes read 4 rows x 32 bytes, transposed  (ds_read_b64_tr_b16)
// ---------------------------------------------------------------------------
__host__ __device__ constexpr int swz(int rows4) { return -rows4 & 3; }
template <int D>
struct SwzTile {
  static constexpr int kNC = D / 32;              // 64-byte column groups per row
  static constexpr int kBytes = kTile * D * 2;
  static constexpr int kInstrs = 4 * kNC;         // 1 KiB copies per tile
  __host__ __device__ static constexpr int block_off(int R, int C) { return (R * kNC + C) * 1024; }
};

// Per-lane source of copy instruction t (block R = t / kNC, C = t % kNC):
// byte offset from the tile's first row, and the row inside the tile.
template <int D>
__device__ __forceinline__ void copy_src(int t, int lane, int row_stride, int& row, int& goff) {
  const int R = t / SwzTile<D>::kNC, C = t % SwzTile<D>::kNC;
  const int r16 = lane >> 2, pos = lane & 3;
  const int c4 = pos ^ swz(r16 >> 2);
  row = 16 * R + r16;
  goff = (row * row_stride + (4 * C + c4) * 8) * 2;  // bytes
}

// One 1 KiB copy: lane l fetches 16 bytes at tile_base + voff and they land in
// LDS at lds_block + 16 * l.  Written as inline asm on purpose: the compiler's
// wait-count insertion then knows nothing of the copy, so it cannot make later
// LDS reads wait for it (it cannot tell the ring slots apart and would wait for
// every copy in flight); the waits for these copies are the explicit wait_vm<>
// calls in the kernels.  tile_base and lds_block must be wave-uniform.
// The LDS address travels in m0, which the compiler reserves for itself and
// does not accept as a clobber: the statement saves and restores it, so a value
// the compiler keeps there (indirect register indexing, its own LDS copies)
// survives.
__device__ __forceinline__ void copy16(const half_t* tile_base, int voff, char* lds_block) {
  const unsigned lds_addr = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds_block;
  unsigned saved_m0;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %3\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %2\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved_m0)
      : "v"(voff), "s"(tile_base), "s"(lds_addr)
      : "memory");
}
// The same for dS.  STREAM: with the hint that it is read once, which keeps it from displacing the tiles other work groups
// re-read out of the L2.  SHARED: other work groups of the launch have written it (sc1: not out of this XCD's L2, see store_ds).
template <bool SHARED, bool STREAM>
__device__ __forceinline__ void copy16_ds(const half_t* tile_base, int voff, char* lds_block) {
  const unsigned lds_addr = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds_block;
  unsigned saved_m0;
#define FMHA_COPY16(HINTS)                            \
  asm volatile(                                       \
      "s_mov_b32 %0, m0\n\t"                          \
      "s_mov_b32 m0, %3\n\t"                          \
      "s_nop 0\n\t"                                   \
      "global_load_lds_dwordx4 %1, %2" HINTS "\n\t"   \
      "s_mov_b32 m0, %0"                              \
      : "=&s"(saved_m0)                               \
      : "v"(voff), "s"(tile_base), "s"(lds_addr)      \
      : "memory")
  if constexpr (SHARED && STREAM) FMHA_COPY16(" sc1 nt");
  else if constexpr (SHARED) FMHA_COPY16(" sc1");
  else if constexpr (STREAM) FMHA_COPY16(" nt");
  else FMHA_COPY16("");
#undef FMHA_COPY16
}

// kCount copies of 1 KiB to consecutive blocks of LDS: lane l's 16 bytes of block u land at lds + 1024 * u + 16 * l.
// The instruction's offset counts for both addresses, so they come from base + voff + 64 * u with voff lowered by
// 960 * u.
template <int kCount>
__device__ __forceinline__ void copy16_blocks(const half_t* base, int voff, unsigned lds) {
  static_assert(kCount == 2 || kCount == 4, "");
  unsigned saved_m0;
  if constexpr (kCount == 2) {
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %2\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %3, %1\n\t"
        "global_load_lds_dwordx4 %4, %1 offset:1024\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved_m0)
        : "s"(base), "s"(lds), "v"(voff), "v"(voff - 960)
        : "memory");
  } else {
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %2\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %3, %1\n\t"
        "global_load_lds_dwordx4 %4, %1 offset:1024\n\t"
        "global_load_lds_dwordx4 %5, %1 offset:2048\n\t"
        "global_load_lds_dwordx4 %6, %1 offset:3072\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved_m0)
        : "s"(base), "s"(lds), "v"(voff), "v"(voff - 960), "v"(voff - 1920), "v"(voff - 2880)
        : "memory");
  }
}

// The same with 4 bytes per lane (256 bytes per instruction): lane l fetches the
// dword at base + voff and it lands in LDS at lds_dst + 4 * l.
__device__ __forceinline__ void copy4(const float* base, int voff, char* lds_dst) {
  const unsigned lds_addr = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds_dst;
  unsigned saved_m0;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %3\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dword %1, %2\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved_m0)
      : "v"(voff), "s"(base), "s"(lds_addr)
      : "memory");
}

// rows pattern: lane (i, hh) reads chunk 2*kk + hh of row rb*32 + i.
// Two lane offsets (kk even / odd); the rest is an immediate.
template <int D>
__device__ __forceinline__ void swz_rows_off(int lane, int (&off)[2]) {
  const int i = lane & 31, hh = lane >> 5, r16 = i & 15, g = swz(r16 >> 2);
  const int base = (i >> 4) * SwzTile<D>::kNC * 1024 + r16 * 64;
  off[0] = base + ((hh ^ g) * 16);
  off[1] = base + (((2 + hh) ^ g) * 16);
}
template <int D>
__device__ __forceinline__ h8 swz_rows(const char* tile, int rb, int kk, const int (&off)[2]) {
  return *reinterpret_cast<const h8*>(tile + off[kk & 1] + SwzTile<D>::block_off(2 * rb, kk >> 1));
}
// cols pattern: MFMA A operand, rows = features db*32 + (lane & 31), k = streamed
// rows of chunk c16 in accumulator order.  Two lane offsets (rows +0 / +8).
template <int D>
__device__ __forceinline__ void swz_cols_off(int lane, int (&off)[2]) {
  const int L = lane & 15, half = (lane >> 4) & 1, hh = lane >> 5;
  const int c4 = 2 * half + ((L & 3) >> 1);
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int r16 = 8 * e + 4 * hh + (L >> 2);
    off[e] = r16 * 64 + ((c4 ^ swz(r16 >> 2)) * 16) + (L & 1) * 8;
  }
}
template <int D>
__device__ __forceinline__ h8 swz_cols(const char* tile, int c16, int db, const int (&off)[2]) {
  typedef __attribute__((address_space(3))) s4 lds_s4;
  const char* p = tile + SwzTile<D>::block_off(c16, db);
  s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(p + off[0]));
  s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(p + off[1]));
  return __builtin_bit_cast(h8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// The same reads through LDS addresses formed by the caller (tile + off[e]) and hidden from the optimiser:
// seen whole, it may split tile + off[e] + constant into a loop-invariant part per fragment, kept in a
// register each (and spilled), and the ring slot; opaque, the constant is the instruction's immediate offset.
__device__ __forceinline__ unsigned opaque_lds_address(const char* p) {
  unsigned a = (unsigned)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
  asm volatile("" : "+v"(a));
  return a;
}
template <int D>
__device__ __forceinline__ h8 swz_rows_at(unsigned a_even, unsigned a_odd, int rb, int kk) {
  typedef __attribute__((address_space(3))) h8 lds_h8;
  return *(const lds_h8*)(uintptr_t)(((kk & 1) ? a_odd : a_even) + (unsigned)SwzTile<D>::block_off(2 * rb, kk >> 1));
}
template <int D>
__device__ __forceinline__ h8 swz_cols_at(unsigned a0, unsigned a1, int c16, int db) {
  typedef __attribute__((address_space(3))) s4 lds_s4;
  const unsigned o = SwzTile<D>::block_off(c16, db);
  s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(uintptr_t)(a0 + o));
  s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(uintptr_t)(a1 + o));
  return __builtin_bit_cast(h8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// ---------------------------------------------------------------------------
// 16 x 16 x 32 MFMAs over the same tiles.  At the power cap they do 13 % more products per second than the 32 x 32 x 16
// ones (registers only, random operands, all CUs busy: 1,766 against 1,555 TFLOP/s; with each A operand read from LDS for
// 2 x 16 columns 1,580 against 1,400), so the kernels that run there use them.  They are twice as many instructions, which
// a wave alone on its SIMD feels (B1 H2 N4000 forward: 51 -> 59 us), and where vector instructions are the bound they gain
// nothing (B1 H12 N8192 D64 forward: 218 -> 223 us): those kernels keep the others.
//
// Both give the same bits.  One 16 x 16 x 32 MFMA adds the products of its lanes 0..31 first, then those of lanes
// 32..63, each the way a 32 x 32 x 16 MFMA adds its 16; and the streamed rows are dealt out so that these are the same 16:
// of 32 streamed rows kc, row block p (0 or 1) has, in MFMA row 4 g + r (held by lanes 16 g .. in register r), the row
//     32 kc + 16 (g >> 1) + 8 p + 4 (g & 1) + r.
// The second GEMM takes rows 32 kc .. as one step, register e = 4 p + r of lane group g as its k = 8 g + e.
// ---------------------------------------------------------------------------
template <int D>
struct Geom16 {
  static constexpr int kKS = D / 32;  // steps over the features
  static constexpr int kDB = D / 16;  // blocks of 16 features
};
// first of the four streamed rows, inside 32, that lane group g holds in row block p
__device__ __forceinline__ int acc16_row(int p, int g) { return 16 * (g >> 1) + 8 * p + 4 * (g & 1); }
// rows pattern: lane (m, g) reads chunk g of the row of MFMA row m; two lane offsets (row block even / odd).
template <int D>
__device__ __forceinline__ int rows16_off(int lane, int p) {
  const int m = lane & 15, g = lane >> 4, r16 = 8 * p + (m & 7);
  return (m >> 3) * SwzTile<D>::kNC * 1024 + r16 * 64 + ((g ^ swz(r16 >> 2)) * 16);
}
template <int D>
__device__ __forceinline__ h8 rows16_at(unsigned a_even, unsigned a_odd, int rb, int kk) {
  typedef __attribute__((address_space(3))) h8 lds_h8;
  return *(const lds_h8*)(uintptr_t)(((rb & 1) ? a_odd : a_even) + (unsigned)SwzTile<D>::block_off(rb & 2, kk));
}
// cols pattern: MFMA A operand, rows = features 16 db + (lane & 15), k = 32 streamed rows kc in accumulator order.  Two
// lane offsets (rows +0 / +8) for even db; odd ones are 32 bytes away, one way or the other.
template <int D>
__device__ __forceinline__ int cols16_off(int lane, int p, int odd) {
  const int L = lane & 15, g = lane >> 4, r16 = 8 * p + 4 * (g & 1) + (L >> 2);
  return (g >> 1) * SwzTile<D>::kNC * 1024 + r16 * 64 + (((2 * odd + ((L & 3) >> 1)) ^ swz(r16 >> 2)) * 16) + (L & 1) * 8;
}
template <int D>
struct Cols16 {
  unsigned a[2][2];  // [rows +0 / +8][feature block even / odd]
  __device__ __forceinline__ Cols16(const char* tile, int lane) {
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int odd = 0; odd < 2; ++odd) a[p][odd] = opaque_lds_address(tile + cols16_off<D>(lane, p, odd));
  }
  __device__ __forceinline__ h8 at(unsigned slot, int kc, int db) const {
    typedef __attribute__((address_space(3))) s4 lds_s4;
    const unsigned o = slot + SwzTile<D>::block_off(2 * kc, db >> 1);
    s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(uintptr_t)(a[0][db & 1] + o));
    s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(uintptr_t)(a[1][db & 1] + o));
    return __builtin_bit_cast(h8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
};
// s_waitcnt vmcnt(N) with the other counters left alone.  Issued through the
// builtin (not inline asm) so that the compiler's wait-count bookkeeping sees it.
template <int N>
__device__ __forceinline__ void wait_vm() {
  static_assert(N >= 0 && N < 64, "vmcnt immediate");  // bits 3:0 and 15:14 of the immediate
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// A wave's 32 resident rows on their way to registers: copied to D / 16 KiB of LDS that are the wave's own (rows row0 .. of a
// slice, row N-1 in the place of those past the end) and, once they are there, read as MFMA B operands.  Loaded straight to
// registers, neighbouring lanes ask for 16 bytes of different rows each, and the CU's path to memory takes 64 cycles for
// what a copy takes 16 for, 64 bytes of a row from every four lanes: 2,000 to 4,000 cycles at the start of a block.
// Kernels in graphs of 20 calls, us loaded straight and this way, forward and backward, N x slices: D = 64 128 x 4 4.92, 4.70 and 6.31,
// 5.87; 300 x 80 causal 7.38, 7.21 and 13.3, 12.4; 1024 x 64 causal 16.7, 16.6 and 43.1, 42.1; D = 128 128 x 32 6.69, 6.13 and 9.86,
// 8.59; 200 x 48 causal 9.08, 8.79 and 14.9, 13.6; 700 x 24 13.9, 13.5 and 34.1, 33.2; 2048 x 80 causal 94.6, 93.3 and 296, 295.
template <int D>
__device__ __forceinline__ void copy_rows(const half_t* slice, int stride, int row0, int n, int lane, char* lds) {
  constexpr int kNC = SwzTile<D>::kNC, kBack = 960 * (kNC - 1);  // see copy16_blocks
  row0 = min(row0, n - 1);
  const half_t* const base = slice + (long)row0 * stride - kBack / 2;
  const unsigned to = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  const int r16 = lane >> 2, col = ((lane & 3) ^ swz(lane >> 4)) * 16 + kBack;
#pragma unroll
  for (int R = 0; R < 2; ++R) {
    const int row = min(16 * R + r16, n - 1 - row0);
    copy16_blocks<kNC>(base, row * stride * 2 + col, to + SwzTile<D>::block_off(R, 0));
  }
}
template <int D>
struct StagedRows {
  const char* at;
  int lane;
  __device__ __forceinline__ h8 wide(int kk) const {  // for 32 x 32 MFMAs: features 16 kk .. of row lane & 31
    int off[2];
    swz_rows_off<D>(lane, off);
    return swz_rows<D>(at, 0, kk, off);
  }
  __device__ __forceinline__ h8 narrow(int kk, int cb) const {  // for 16 x 16 ones: features 32 kk .. of row 16 cb + (lane & 15)
    const int i = lane & 15;
    return *reinterpret_cast<const h8*>(at + SwzTile<D>::block_off(cb, kk) + i * 64 + (((lane >> 4) ^ swz(i >> 2)) * 16));
  }
};
// The copies are there: read them.
__device__ __forceinline__ void staged_rows_landed() {
  wait_vm<0>();
  asm volatile("" ::: "memory");
}
// They are read: others may take their place.
__device__ __forceinline__ void staged_rows_read() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  asm volatile("" ::: "memory");
}

// Over the four lanes with the same l & 15: first the two that are 32 apart, then the others.
__device__ __forceinline__ float max_over_groups(float x) {
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(x), __float_as_int(x), false, false);
  x = fmaxf(__int_as_float(r[0]), __int_as_float(r[1]));
  r = __builtin_amdgcn_permlane16_swap(__float_as_int(x), __float_as_int(x), false, false);
  return fmaxf(__int_as_float(r[0]), __int_as_float(r[1]));
}
// store_resident for accumulators of 16 x 16 blocks: acc[db][cb] has features 16 db + 4 g + 0..3 of resident position
// 16 cb + (lane & 15), to be scaled by mul[cb].
template <int D>
struct Stage16 {
  // bytes per row: the 8-byte pieces that 32 lanes write, 16 rows x 2, fall on different banks
  static constexpr int kPitch = D * 2 + 16;
  static constexpr int kBytes = kResident * kPitch;  // per wave
};
template <int D>
__device__ __forceinline__ void store_resident16(half_t* __restrict__ base, int row_stride, int row0, int n,
                                                 const f4v (*acc)[2], const float (&mul)[2], int lane,
                                                 char* __restrict__ stage, int row_of_0 = -1, int row_of_1 = -1,
                                                 int upper_off = 16 * Stage16<D>::kPitch) {
  // row_of_cb: the row (0..31, relative to row0) of this lane's column of block cb, when that is not 16 cb + (lane & 15);
  // upper_off: where rows 16..31 are staged, relative to `stage`, when the staging tile is not contiguous
  constexpr int kPitch = Stage16<D>::kPitch;
#pragma unroll
  for (int cb = 0; cb < 2; ++cb) {
    const int row = row_of_0 < 0 ? 16 * cb + (lane & 15) : cb ? row_of_1 : row_of_0;
    char* mine = stage + (row & 15) * kPitch + (row >> 4) * upper_off + (lane >> 4) * 8;
#pragma unroll
    for (int db = 0; db < D / 16; ++db) {
      h4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (half_t)(acc[db][cb][e] * mul[cb]);
      *reinterpret_cast<h4*>(mine + db * 32) = v;
    }
  }
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the wave's own writes have landed
  asm volatile("" ::: "memory");
  store_staged<D, kPitch, h8>(base, row_stride, row0, n, lane, stage, upper_off);
}

// Arguments of a kernel, asked for here: left to the compiler they come in four or five groups, each where it is first needed and
// each waited for by itself.  128-query forward, which also tests for a negative scale now instead of negating and
// choosing, us before and after, N x slices: D = 64 77 x 8 causal 5.66, 5.45; 512 x 192 21.8, 21.1; 1024 x 64 causal 17.2, 16.7; D =
// 128 200 x 48 causal 9.33, 9.08.  The kernels of the backward gain nothing from it.
__device__ __forceinline__ void load_now(const Strides& s) { asm volatile("" ::"s"(s.b), "s"(s.n), "s"(s.h)); }
__device__ __forceinline__ void load_now(const FmhaDivisor& v) { asm volatile("" ::"s"(v.d), "s"(v.mul), "s"(v.shift)); }
template <typename T>
__device__ __forceinline__ void load_now(T v) { asm volatile("" ::"s"(v)); }
template <typename... T>
__device__ __forceinline__ void load_all_now(const T&... v) { (load_now(v), ...); }

// Wait until at most n (0 to 4) of this wave's LDS reads are on their way.
__device__ __forceinline__ void wait_lds(int n) {
  if (n == 0) __builtin_amdgcn_s_waitcnt(0xC07F);
  else if (n == 1) __builtin_amdgcn_s_waitcnt(0xC17F);
  else if (n == 2) __builtin_amdgcn_s_waitcnt(0xC27F);
  else if (n == 3) __builtin_amdgcn_s_waitcnt(0xC37F);
  else __builtin_amdgcn_s_waitcnt(0xC47F);
}
// The same at this place in the program, so that the compiler adds no wait of its own in front of it.
__device__ __forceinline__ void wait_lds_pinned(int n) {
  __builtin_amdgcn_sched_barrier(0);
  wait_lds(n);
  __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void block_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's LDS reads have landed
  asm volatile("" ::: "memory");       // keep LDS accesses on their side of the barrier
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
// Wait until at most min(later, kMax) * kPer of this wave's copies are in flight.
template <int kPer, int kMax>
__device__ __forceinline__ void wait_vm_tiles(int later) {
  if constexpr (kMax == 0) {
    wait_vm<0>();
  } else {
    if (later >= kMax) wait_vm<kMax * kPer>();
    else wait_vm_tiles<kPer, kMax - 1>(later);
  }
}
template <int V>
struct IntTag { static constexpr int value = V; };
// f(IntTag<0>{}), f(IntTag<1>{}), .. f(IntTag<kN - 1>{}): unrolled whatever the size of the body.
template <typename F, int... I>
__device__ __forceinline__ void static_for_each(std::integer_sequence<int, I...>, F&& f) {
  (f(IntTag<I>{}), ...);
}
template <int kN, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_each(std::make_integer_sequence<int, kN>{}, f);
}

// 16 bytes of dS per lane to p + kOffset bytes.  KEEP: without the non-temporal hint (data that is read once, by other work
// groups of this launch or of a later one).  SHARED: work groups of this launch read it, so it goes past the XCD's L2 (sc1) and
// those of any XCD see it once the store is done.  Not where a later launch reads it (forward and backward, 80 x 2048 x 128
// causal: 397 us, with sc1 on either side 429).  Inline asm because the compiler keeps the hint only on the first of several
// stores that share a base address; like the tile copies it is therefore invisible to the compiler's wait counts.
template <bool SHARED, bool KEEP, int kOffset>
__device__ __forceinline__ void store_ds(half_t* p, h8 v, IntTag<kOffset>) {
#define FMHA_STORE16(HINTS) \
  asm volatile("global_store_dwordx4 %0, %1, off offset:%2" HINTS : : "v"(p), "v"(v), "n"(kOffset) : "memory")
  if constexpr (SHARED && !KEEP) FMHA_STORE16(" sc1 nt");
  else if constexpr (SHARED) FMHA_STORE16(" sc1");
  else if constexpr (!KEEP) FMHA_STORE16(" nt");
  else FMHA_STORE16("");
#undef FMHA_STORE16
}

// Row statistics of 64-row tiles for a work group of 4 * D threads: D / 8 lanes to a row, two rows each, in the order of
// fmha_bwd_delta_kernel.  load asks for the rows of a tile, one tile after the other; make sums up what was asked for.
template <int D>
struct TileStats {
  static constexpr int kLanes = D / 8;
  h8 o[2], g[2];
  float l[2];
  const half_t *op, *gp;  // the next tile to ask for
  const float* lp;
  int o_stride, g_stride, row, col, o_off, g_off, l_off;
  __device__ __forceinline__ TileStats(const half_t* O, const half_t* dO, const float* LSE, int rs, int gs_n, int tile) {
    op = O + (long)tile * kTile * rs, gp = dO + (long)tile * kTile * gs_n, lp = LSE + tile * kTile;
    o_stride = rs, g_stride = gs_n;
    row = threadIdx.x / kLanes, col = threadIdx.x % kLanes * 16;
    o_off = row * rs * 2 + col, g_off = row * gs_n * 2 + col, l_off = row * 4;
  }
  __device__ __forceinline__ void load(int last_row) {  // last_row: of the tile, N - 1 if it holds that; 63 or more if not
    const auto at = [](const void* base, int off) { return reinterpret_cast<const char*>(base) + (unsigned)off; };
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const half_t *ou = op + 32 * u * (long)o_stride, *gu = gp + 32 * u * (long)g_stride;
      const float* lu = lp + 32 * u;
      if (last_row < kTile - 1) {  // rows past the end re-read row N-1
        const int r = min(32 * u + row, last_row);
        ou = op, gu = gp, lu = lp;
        o_off = r * o_stride * 2 + col, g_off = r * g_stride * 2 + col, l_off = r * 4;
      }
      o[u] = *reinterpret_cast<const h8*>(at(ou, o_off));
      g[u] = *reinterpret_cast<const h8*>(at(gu, g_off));
      l[u] = *reinterpret_cast<const float*>(at(lu, l_off));
    }
    op += kTile * (long)o_stride, gp += kTile * (long)g_stride, lp += kTile;
  }
  __device__ __forceinline__ void make(char* slot) const {  // 64 lse * log2(e), then 64 delta values
    const auto dpp = [](float x, auto ctrl) __attribute__((always_inline)) {
      return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), decltype(ctrl)::value, 15, 15, true));
    };
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      float a = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) a = fmaf((float)o[u][e], (float)g[u][e], a);
      if (kLanes == 16) a += dpp(a, IntTag<0x128>{});                                       // of the lane at ^ 8 (of 16)
      a += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(a), (4 << 10) | 31));  // ^ 4
      a += dpp(a, IntTag<0x4E>{});                                                          // ^ 2
      a += dpp(a, IntTag<0xB1>{});                                                          // ^ 1
      float* const mine = reinterpret_cast<float*>(slot) + 32 * u + row;
      mine[0] = l[u] * kLog2e;  // the same from all lanes of the row
      mine[kTile] = a;
    }
  }
};

// ---------------------------------------------------------------------------
// Forward for D = 128 where blocks of 256 queries share out well over the CUs
// (rule: fmha_persistent_forward_pays).  Block = 8 waves = 256 queries, wave = 32 queries; K/V
// tiles of 64 keys stream through a 3-slot LDS ring, copied asynchronously two
// tiles ahead.
//
// Online softmax as in reference kernel/fused_mha_kernel.cu:159-181, except that
// no tile's maximum is looked for as long as the running one serves: the
// probabilities of a tile are formed relative to the running maximum first, and
// only if the sum of half of them (32 keys of a query) exceeds kRescaleSum (so every
// single one stays far below the fp16 range) or is no number (no maximum yet) the
// maximum is raised, O and l are rescaled, and they are formed again.  That takes
// the 16 max instructions and the exchange between the half waves out of nearly
// every tile (B2 H16 N4096 D128 without mask: 254 -> 243 us).
//
// The two waves that share a SIMD (w and w+4) run the same three steps per
// tile, scores (MFMA), softmax (VALU), accumulate (MFMA), in rotated order:
// waves 0-3 do  accumulate(j-1), scores(j), softmax(j)  in iteration j, waves
// 4-7 do  softmax(j-1), accumulate(j-1), scores(j).  Both need exactly K(j)
// and V(j-1) in iteration j, so one barrier per iteration is enough, and one
// wave's MFMA stretch coincides with the other's VALU stretch.
//
// What bounds it is the power cap; 16 x 16 x 32 MFMAs take less of it (Geom16).  With them, one wait for the fragments of two
// units and half of the waves copying late (below), against the kernel without the three, in turn: B2 H32 N4096 D128 causal 267
// -> 251 us, without a mask 486 -> 450 us (1.22 PFLOP/s), B1 H16 N16384 causal 965 -> 895.
// ---------------------------------------------------------------------------
constexpr float kRescaleSum = 4096.f;
constexpr int kFwdWaves = 8;
constexpr int kFwdThreads = kFwdWaves * 64;
constexpr int kFwdBlockQ = kFwdWaves * kResident;
static_assert(kFwdBlockQ == kPersistentForwardRows, "");
constexpr int kRing = 3;

// The kernel is persistent: the launch has one work group per CU (fewer for small
// problems) and each walks its own list of blocks (PersistentBlocks).  While a block's
// last tiles are being worked on, the first K and V tiles of the group's next block are
// already copied into the ring slots that come next, and the next block's Q rows are
// loaded during the last iteration (which no longer needs Q); O leaves through staging
// tiles of its own in LDS.  So a block boundary costs one pipeline fill, not a work-group
// launch, a round trip to HBM and an epilogue during which the CU has nothing else to do.
// A block is found while others' tiles are on their way, and which divisor it takes shows in what the compiler makes of the rest: us
// with int and with FmhaDivisor, 4096 x 64 causal 254.8, 257.0; 8192 x 16 causal 234.3, 237.0; 4096 x 32 without a mask 227.5, 225.1.
template <bool CAUSAL>
using FwdDivisor = std::conditional_t<CAUSAL, int, FmhaDivisor>;
template <int D, bool CAUSAL>
__global__ void __launch_bounds__(kFwdThreads, 1)
fmha_fwd_kernel(const half_t* __restrict__ Q, const half_t* __restrict__ K, const half_t* __restrict__ V,
                Strides qs, Strides ks, Strides vs, half_t* __restrict__ O, float* __restrict__ LSE, FwdDivisor<CAUSAL> H, int N,
                FwdDivisor<CAUSAL> nmb, int slices, float c, int negate_q) {
  using G = Geom16<D>;
  using T = SwzTile<D>;
  constexpr int kIPW = T::kInstrs / kFwdWaves;  // copy instructions per wave per tile
  // K ring then V ring, kRing slots each, then per wave a staging tile for 64 features of
  // its 32 output rows.  The copies into the ring are inline asm (see copy16), so slots
  // can be addressed at run time.
  __shared__ __attribute__((aligned(1024))) char smem[2 * kRing * T::kBytes + kFwdWaves * Stage16<64>::kBytes];
  char* const k_ring = smem;
  char* const v_ring = smem + kRing * T::kBytes;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 15, g = lane >> 4;
  char* const stage = smem + 2 * kRing * T::kBytes + wave * Stage16<64>::kBytes;
  const int rs = H * D;  // O is dense
  const int nt_all = (N + kTile - 1) / kTile;
  const int total = slices * nmb;
  const PersistentBlocks pb{total};

  struct Block {
    const half_t *q, *k, *v;  // first row of the (batch, head) slice
    long o_off, stat_off;     // of the slice in O and in LSE
    int m0, nt;               // first query of the block; tiles it streams
  };
  auto decode = [&](int lin) __attribute__((always_inline)) {
    int bh, mb;
    fmha_slice_and_block(lin, slices, nmb, bh, mb);
    const int mblk = CAUSAL ? nmb - 1 - mb : mb;  // heavy blocks first
    const int b = bh / H, h = bh - b * H;
    Block B;
    B.q = Q + b * qs.b + (long)h * qs.h;
    B.k = K + b * ks.b + (long)h * ks.h;
    B.v = V + b * vs.b + (long)h * vs.h;
    B.o_off = ((long)b * N * H + h) * D;
    B.stat_off = ((long)b * H + h) * N;
    B.m0 = mblk * kFwdBlockQ;
    B.nt = CAUSAL ? min(nt_all, (min(B.m0 + kFwdBlockQ, N) - 1) / kTile + 1) : nt_all;
    return B;
  };

  // this wave's share of every tile copy
  int c_row[kIPW], c_kgoff[kIPW], c_vgoff[kIPW], c_blk[kIPW];
#pragma unroll
  for (int u = 0; u < kIPW; ++u) {
    const int t = wave * kIPW + u;
    copy_src<D>(t, lane, ks.n, c_row[u], c_kgoff[u]);
    copy_src<D>(t, lane, vs.n, c_row[u], c_vgoff[u]);
    c_blk[u] = t * 1024;
  }
  auto copy_tile = [&](const half_t* src, int src_rs, const int (&goff)[kIPW], char* dst, int tile_idx)
                       __attribute__((always_inline)) {
    const int row0 = tile_idx * kTile;
    const half_t* tp = src + (long)row0 * src_rs;  // wave-uniform
    if (row0 + kTile <= N) {
#pragma unroll
      for (int u = 0; u < kIPW; ++u) copy16(tp, goff[u], dst + c_blk[u]);
    } else {
#pragma unroll
      for (int u = 0; u < kIPW; ++u) {  // rows past the end re-read row N-1
        const int back = max(row0 + c_row[u] - (N - 1), 0);
        copy16(tp, goff[u] - back * src_rs * 2, dst + c_blk[u]);
      }
    }
  };

  h8 qf[G::kKS][2];
  auto load_q = [&](const Block& B) __attribute__((always_inline)) {
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      const half_t* qp = B.q + (long)min(B.m0 + wave * kResident + cb * 16 + i, N - 1) * qs.n + g * 8;
#pragma unroll
      for (int kk = 0; kk < G::kKS; ++kk) qf[kk][cb] = *reinterpret_cast<const h8*>(qp + kk * 32);
    }
  };
  auto negate = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < G::kKS; ++kk) {
      qf[kk][0] = -qf[kk][0];
      qf[kk][1] = -qf[kk][1];
    }
  };

  const int k_off0 = rows16_off<D>(lane, 0), k_off1 = rows16_off<D>(lane, 1);

  // state of the block being worked on; [2]: of this lane's queries q0w + i and q0w + 16 + i
  int q0w = 0, ntw = 0;
  f4v o[G::kDB][2];
  float mc[2] = {-INFINITY, -INFINITY};  // running maximum times c
  float l_run = 0.f;  // lanes 0..31: of query q0w + i, lanes 32..63: of q0w + 16 + i; over the keys of lane groups g and g ^ 2
  f4v s[4][2];   // scores of the tile in flight
  h8 pf[2][2];   // its probabilities, fp16, B-operand order

  // The fragment reads of both GEMMs run kLead units (of one fragment and two MFMAs) ahead of their use.  The order is
  // written out and pinned with scheduling barriers: left to itself the scheduler, once registers get scarce,
  // puts every read right before its MFMA, which then waits a full LDS round trip each time.  The fragments of two units
  // are waited for together (half as many s_waitcnt: 1 % at B2 H32 N4096).
  constexpr int kLead = 4;
  constexpr int kN = 4 * G::kKS;  // units of either GEMM
  static_assert(kN == 2 * G::kDB, "");
  auto scores = [&](const char* Kl, int t) __attribute__((always_inline)) {
    if (t >= ntw) return;
    const unsigned a0 = opaque_lds_address(Kl + k_off0), a1 = opaque_lds_address(Kl + k_off1);
    h8 frag[kLead];  // unit n: row block rb = n & 3, feature step kk = n >> 2
#pragma unroll
    for (int n = 0; n < kLead; ++n) frag[n] = rows16_at<D>(a0, a1, n & 3, n >> 2);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < kN; ++n) {
      const int rb = n & 3, kk = n >> 2;
      if (n % 2 == 0) wait_lds_pinned(n + 3 < kN ? 2 : n + 2 < kN ? 1 : 0);
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
        s[rb][cb] = mfma16(frag[n % kLead], qf[kk][cb], kk == 0 ? f4v{0.f, 0.f, 0.f, 0.f} : s[rb][cb]);
      if (n + kLead < kN) frag[n % kLead] = rows16_at<D>(a0, a1, (n + kLead) & 3, (n + kLead) >> 2);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  auto exponentials = [&]() __attribute__((always_inline)) {  // returns the tile's part of l_run
    float l[2] = {0.f, 0.f};
#pragma unroll
    for (int kc = 0; kc < 2; ++kc)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float p = fast_exp2(fmaf(s[2 * kc + (e >> 2)][cb][e & 3], c, -mc[cb]));
          pf[kc][cb][e] = (half_t)p;
          l[cb] += p;
        }
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_int(l[0]), __float_as_int(l[1]), false, false);
    return __int_as_float(r[0]) + __int_as_float(r[1]);
  };
  auto softmax = [&](int t) __attribute__((always_inline)) {
    if (t < 0 || t >= ntw) return;
    const int key0 = t * kTile;
    if ((CAUSAL && key0 + kTile - 1 > q0w) || (key0 + kTile > N)) {
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        const int last = (CAUSAL ? min(q0w + cb * 16 + i, N - 1) : N - 1) - key0 - acc16_row(0, g);  // last key that counts
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if ((rb >> 1) * 32 + (rb & 1) * 8 + r > last) s[rb][cb][r] = -INFINITY;
      }
    }
    // Optimistic: probabilities relative to the running maximum as it stands.  If the sum over the 32 keys of a query
    // that lane groups g and g ^ 2 have is past kRescaleSum (or not a number: no maximum yet), the maximum is brought up to date and they are formed again.
    // A wave's last tile always brings it up to date, as in fmha_fwd_pipe_kernel: both kernels give the same bits, so
    // that a slice's result does not depend on how many others the call has.
    float lt = exponentials();
    if (t == ntw - 1 || __builtin_amdgcn_ballot_w64(!(lt <= kRescaleSum)) != 0) {
      float alpha[2];
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) {
        float mx = s[0][cb][0];
#pragma unroll
        for (int rb = 0; rb < 4; ++rb)
#pragma unroll
          for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[rb][cb][r]);
        mx = max_over_groups(mx);
        const float mc_new = fmaxf(mc[cb], mx * c);
        alpha[cb] = fast_exp2(mc[cb] - mc_new);
        mc[cb] = mc_new;
#pragma unroll
        for (int db = 0; db < G::kDB; ++db)
#pragma unroll
          for (int r = 0; r < 4; ++r) o[db][cb][r] *= alpha[cb];
      }
      l_run *= lane < 32 ? alpha[0] : alpha[1];
      asm volatile("" : "+v"(l_run));  // rounded here: contracted with the sum below the loop is 4 % slower without a mask
      lt = exponentials();
    }
    l_run += lt;
  };
  auto accumulate = [&](const char* Vl, int t) __attribute__((always_inline)) {
    if (t < 0 || t >= ntw) return;
    const Cols16<D> cols(Vl, lane);
    h8 frag[kLead];  // unit n: 32 keys kc = n / kDB, feature block db = n % kDB
#pragma unroll
    for (int n = 0; n < kLead; ++n) frag[n] = cols.at(0, n / G::kDB, n % G::kDB);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < kN; ++n) {
      const int kc = n / G::kDB, db = n % G::kDB;
      if (n % 2 == 0) wait_lds_pinned(n + 3 < kN ? 4 : n + 2 < kN ? 2 : 0);
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) o[db][cb] = mfma16(frag[n % kLead], pf[kc][cb], o[db][cb]);
      if (n + kLead < kN) frag[n % kLead] = cols.at(0, (n + kLead) / G::kDB, (n + kLead) % G::kDB);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  const bool first_group = wave < kFwdWaves / 2;
  // Iteration j of a block: K(j) sits in K slot s0, V(j-1) in V slot s2; K(j+2) is copied
  // into K slot s2 and V(j+1) into V slot s1, where tiles past the block's last one are the
  // first tiles of the group's next block (at most K(0), K(1) and V(0) of it).  The slots
  // rotate after every iteration but a block's last, so the next block finds its tile 0 in s0.
  auto run = [&](auto group_tag) __attribute__((always_inline)) {
    constexpr bool kFirst = decltype(group_tag)::value == 0;
    int lin_cur = pb.lin(0), round = 0;
    {
      const Block first = decode(lin_cur);
      copy_tile(first.k, ks.n, c_kgoff, k_ring, 0);
      if (first.nt > 1) copy_tile(first.k, ks.n, c_kgoff, k_ring + T::kBytes, 1);
      copy_tile(first.v, vs.n, c_vgoff, v_ring, 0);
      load_q(first);
    }
    int s0 = 0, s1 = 1, s2 = 2;
    // Copies this wave issued in the previous iteration: all it may leave in flight at the top of
    // an iteration (the tiles needed now were issued earlier).  0 at a block's first iteration:
    // everything issued so far (Q rows, the previous block's output rows) is waited for there, so
    // that no wait for a register load is left to be placed inside the loop, where it would also
    // wait for the copies in flight.
    int in_flight = 0;
    for (;;) {
      // Only what the main loop needs is decoded here; the next block and the output addresses are
      // worked out after it, so that they do not occupy scalar registers across it.
      const half_t *cur_k, *cur_v;
      int nt;
      {
        const Block cur = decode(lin_cur);
        cur_k = cur.k;
        cur_v = cur.v;
        nt = cur.nt;
        q0w = cur.m0 + wave * kResident;
      }
      ntw = nt;
      if (CAUSAL) {
        ntw = min(nt, (min(q0w + kResident, N) - 1) / kTile + 1);
        if (q0w >= N) ntw = 0;
      }
#pragma unroll
      for (int db = 0; db < G::kDB; ++db) o[db][0] = o[db][1] = f4v{0.f, 0.f, 0.f, 0.f};
      mc[0] = mc[1] = -INFINITY;
      l_run = 0.f;
      auto wait_and_sync = [&]() __attribute__((always_inline)) {
        if (in_flight == 2 * kIPW) wait_vm<2 * kIPW>();
        else if (in_flight == kIPW) wait_vm<kIPW>();
        else wait_vm<0>();
        block_barrier();
      };
      auto compute = [&](int j, auto drain_tag, auto copies) __attribute__((always_inline)) {
        constexpr bool kDrain = decltype(drain_tag)::value != 0;
        const char* Kl = k_ring + s0 * T::kBytes;
        const char* Vl = v_ring + s2 * T::kBytes;
        // The first group issues its half of the tile copies at the end of the iteration, the second at its start: all at
        // once after the barrier they held every wave until the copy path had taken them.  This alone, 16 x 16 MFMAs and merged
        // waits in place, on one card: B2 H32 N4096 causal 254 -> 250 us, without a mask 460 -> 446, B1 H16 N32768
        // causal 3642 -> 3509; other places 0.5-1 % slower than this, both at the end 0.5 % slower than before.
        if (kFirst) {
          accumulate(Vl, j - 1);
          if (!kDrain) { scores(Kl, j); softmax(j); }
          copies();
        } else {
          copies();
          softmax(j - 1);
          accumulate(Vl, j - 1);
          if (!kDrain) scores(Kl, j);
        }
        if (!kDrain) { const int t = s0; s0 = s1; s1 = s2; s2 = t; }
      };
      // main part: both tiles to copy belong to this block
      int j = 0;
      for (; j + 2 < nt; ++j) {
        wait_and_sync();
        if (j == 0 && negate_q) negate();
        in_flight = 2 * kIPW;
        compute(j, IntTag<0>{}, [&]() __attribute__((always_inline)) {
          copy_tile(cur_k, ks.n, c_kgoff, k_ring + s2 * T::kBytes, j + 2);
          copy_tile(cur_v, vs.n, c_vgoff, v_ring + s1 * T::kBytes, j + 1);
        });
      }
      // tail: the last two tiles, during which the first tiles of the next block are copied
      const int round_next = pb.next_round(round);
      const int lin_next = round_next >= 0 ? pb.lin(round_next) : -1;
      int pre_k = 0, pre_v = 0;  // tiles of the next block already issued
      {
        Block nxt = decode(lin_next >= 0 ? lin_next : lin_cur);
        for (; j < nt; ++j) {
          wait_and_sync();
          if (j == 0 && negate_q) negate();
          in_flight = 0;
          const int ek = j + 2, ev = j + 1;
          if (ek < nt) {
            copy_tile(cur_k, ks.n, c_kgoff, k_ring + s2 * T::kBytes, ek);
            in_flight += kIPW;
          } else if (lin_next >= 0 && ek - nt == pre_k && pre_k < min(2, nxt.nt)) {
            copy_tile(nxt.k, ks.n, c_kgoff, k_ring + s2 * T::kBytes, pre_k);
            ++pre_k;
            in_flight += kIPW;
          }
          if (ev < nt) {
            copy_tile(cur_v, vs.n, c_vgoff, v_ring + s1 * T::kBytes, ev);
            in_flight += kIPW;
          } else if (lin_next >= 0 && ev - nt == pre_v && pre_v < 1) {
            copy_tile(nxt.v, vs.n, c_vgoff, v_ring + s1 * T::kBytes, 0);
            ++pre_v;
            in_flight += kIPW;
          }
          compute(j, IntTag<0>{}, []() {});
        }
        // The last iteration has no tile of its own, only the second half of tile nt - 1.  Q was last used
        // by scores(nt - 1), an iteration ago: the next block's rows are loaded over it.  This is a separate
        // copy of the code so that, in the compiler's eyes, those loads never flow into a use of Q without the
        // wait at the top of the next block between them.
        wait_and_sync();
        in_flight = 0;
        if (lin_next >= 0) load_q(nxt);
        compute(nt, IntTag<1>{}, []() {});
      }
      // the block's output: O rows through this wave's staging tile, 64 features at a time
      {
        const Block cur = decode(lin_cur);
        const auto other = __builtin_amdgcn_permlane16_swap(__float_as_int(l_run), __float_as_int(l_run), false, false);
        const int l_sum = __float_as_int(__int_as_float(other[0]) + __int_as_float(other[1]));
        const auto both = __builtin_amdgcn_permlane32_swap(l_sum, l_sum, false, false);
        const float l_tot[2] = {__int_as_float(both[0]), __int_as_float(both[1])};
        const float inv[2] = {1.f / l_tot[0], 1.f / l_tot[1]};
#pragma unroll
        for (int part = 0; part < D / 64; ++part)
          store_resident16<64>(O + cur.o_off + part * 64, rs, q0w, N, o + 4 * part, inv, lane, stage);
        if (LSE && lane < kResident && q0w + lane < N)
          LSE[cur.stat_off + q0w + lane] = ((lane < 16 ? mc[0] : mc[1]) +
                                            __builtin_amdgcn_logf(lane < 16 ? l_tot[0] : l_tot[1])) * kLn2;
      }
      if (lin_next < 0) break;
      lin_cur = lin_next;
      round = round_next;
      {
        // what a short previous block could not prefetch
        const Block cur = decode(lin_cur);
        if (pre_k < 1) copy_tile(cur.k, ks.n, c_kgoff, k_ring + s0 * T::kBytes, 0);
        if (pre_k < 2 && cur.nt > 1) copy_tile(cur.k, ks.n, c_kgoff, k_ring + s1 * T::kBytes, 1);
        if (pre_v < 1) copy_tile(cur.v, vs.n, c_vgoff, v_ring + s0 * T::kBytes, 0);
      }
      in_flight = 0;
    }
  };
  // Each group runs its own copy of the loop: no joins between the two
  // orders inside the loop, so no register shuffling at branch merges.
  if (first_group) run(IntTag<0>{});
  else run(IntTag<1>{});
}

// ---------------------------------------------------------------------------
// Forward for D = 64, and for D = 128 where blocks of 256 queries do not share out evenly (rule:
// fmha_persistent_forward_pays).  Block = 4 waves, one per SIMD, of 32 queries each; two blocks share a CU.
//
// What bounds it: a wave issues one instruction every 4-5 cycles, so one that runs scores, softmax and accumulation one
// after the other needs 1,800 cycles per 32 x 64 tile at D = 64 (MFMA 512, vector instructions 700) and a SIMD needs
// several such waves before either unit is busy, which small problems do not have.  Here the three are interleaved
// inside the wave: step j runs softmax(j) and spreads the MFMAs of accumulate(j - 1) and scores(j + 1) between its vector
// instructions, in an order that is written out and pinned.  A wave alone on its SIMD then needs 1,450 cycles (B1 H4
// N8192 D64: 168 -> 83 us against the 8-wave kernel; D128: 184 -> 134 us); with two waves per SIMD and all CUs busy
// the chip runs at its power limit (B1 H12 N8192 D64: 263 -> 220 us).
// Small blocks cost twice the K/V copies per query of 256-query blocks and are worth it for balance: B1 H32 N1500 D128
// causal 41 -> 31 us, B4 H16 N1024 D64 causal 24 -> 17 us, B16 H12 N512 D64 24 -> 20 us, B3 H20 N1031 D128 67 -> 50 us.
// Where the last block of a slice has up to 32 queries, one wave of four works: fwd_tail_rows.
// Three blocks per CU at D = 64 (168 registers) gain 2 % on the long shape and lose 2-5 % on the short ones: not taken.
//
// The maximum is handled as in fmha_fwd_kernel.  Bringing it up to date happens outside the main loop.  K and V have two
// slots each; a tile is copied one tile ahead of its use.
// ---------------------------------------------------------------------------
constexpr int kPipeWaves = 4;
constexpr int kPipeThreads = kPipeWaves * 64;
constexpr int kPipeBlockQ = kPipeWaves * kResident;
constexpr int kPipeBlockKeys = kPipeWaves * kResident;  // of the dK/dV pass
// Two fp32 values as a pair of fp16 values, at this place in the program: seen through, the optimiser moves the
// conversions of a tile past the next branch, and keeps the fp32 values in registers until then.
__device__ __forceinline__ unsigned pack_f16(float lo, float hi) {
  unsigned r = __builtin_bit_cast(unsigned, h2{(half_t)lo, (half_t)hi});
  asm volatile("" : "+v"(r));
  return r;
}

// Of two waves that share a SIMD one goes first whenever both could issue: the one in an odd wave slot (bits 0 to 3 of the
// register say which slot a wave has).  Rule and figures: half_round_left.
__device__ __forceinline__ void odd_slots_first() {
  int slot;
  asm volatile("s_getreg_b32 %0, hwreg(HW_REG_HW_ID, 0, 4)" : "=s"(slot));
  if (slot & 1) __builtin_amdgcn_s_setprio(1);
}

// The last, up to 32, queries of a slice by one wave for itself, with no other wave or barrier (rule: fmha_tails_per_block).
// As a block of their own they take a whole place of a CU for three waves that do nothing; here two or four slices share one.
// K and V of 64 keys take turns in a tile of LDS that is the wave's own: K(t + 1) comes while the scores of tile t are formed
// from registers and goes to registers, V(t) then comes while the softmax is.  Not interleaved further: at D = 128 the
// registers are used up.  At D = 128 a tile takes 2,500 cycles (kernel below: 2,000), of which the MFMAs take 1,024; all that
// counts is that the block ends before the others of its round, so its waves go first wherever they could issue (a tail that is
// still there when the others have ended: 4100 x 20 slices, D = 128, 186 us without, 170 with).  Two tiles of LDS to a wave, so
// that copies are under way longer: nothing gained.  All sums are those of the kernel below, in the same order.
template <int D, bool CAUSAL>
__device__ __forceinline__ void fwd_tail_rows(const half_t* __restrict__ Q, const half_t* __restrict__ K,
                                              const half_t* __restrict__ V, Strides qs, Strides ks, Strides vs,
                                              half_t* __restrict__ O, float* __restrict__ LSE, FmhaDivisor H, int N, int bh, float c,
                                              int negate_q, char* ring) {
  using G = TileGeom<D>;
  using T = SwzTile<D>;
  constexpr int kKS = G::kKSteps, kDB = G::kDBlocks;
  __builtin_amdgcn_s_setprio(3);
  const int lane = threadIdx.x & 63, i = lane & 31, hh = lane >> 5;
  const int b = bh / H, h = bh - b * H, nt = (N + kTile - 1) / kTile, q0 = (N - 1) / kPipeBlockQ * kPipeBlockQ;
  const unsigned lds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)ring;
  auto copy = [&](const half_t* base, int stride, int t) __attribute__((always_inline)) {
    constexpr int kBack = 960 * (T::kNC - 1);  // see copy16_blocks
    base += (long)t * kTile * stride - kBack / 2;
    const int r16 = lane >> 2, col = ((lane & 3) ^ swz(r16 >> 2)) * 16 + kBack;
#pragma unroll
    for (int R = 0; R < 4; ++R) {
      const int row = 16 * R + r16, back = max(t * kTile + row - (N - 1), 0);  // rows past the end re-read row N-1
      copy16_blocks<T::kNC>(base, (row - back) * stride * 2 + col, lds + T::block_off(R, 0));
    }
  };
  const half_t* const Kb = K + b * ks.b + (long)h * ks.h;
  const half_t* const Vb = V + b * vs.b + (long)h * vs.h;
  copy(Kb, ks.n, 0);
  h8 qf[kKS];
  {
    const half_t* const qp = Q + b * qs.b + (long)h * qs.h + (long)min(q0 + i, N - 1) * qs.n + hh * 8;
#pragma unroll
    for (int kk = 0; kk < kKS; ++kk) {
      qf[kk] = *reinterpret_cast<const h8*>(qp + kk * 16);
      if (negate_q) qf[kk] = -qf[kk];
    }
  }
  unsigned ka0, ka1, va0, va1;
  {
    int k_off[2], v_off[2];
    swz_rows_off<D>(lane, k_off);
    swz_cols_off<D>(lane, v_off);
    ka0 = opaque_lds_address(ring + k_off[0]);
    ka1 = opaque_lds_address(ring + k_off[1]);
    va0 = opaque_lds_address(ring + v_off[0]);
    va1 = opaque_lds_address(ring + v_off[1]);
  }
  f16v o[kDB], s[2], zero;
#pragma unroll
  for (int r = 0; r < 16; ++r) zero[r] = 0.f;
#pragma unroll
  for (int db = 0; db < kDB; ++db) o[db] = zero;
  float mc = -INFINITY, l_run = 0.f;
  u4v pf[4];
  auto exponentials = [&]() __attribute__((always_inline)) {
    float l0 = 0.f, l1 = 0.f;
#pragma unroll
    for (int c16 = 0; c16 < 4; ++c16) {
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float p0 = fast_exp2(fmaf(s[c16 >> 1][(c16 & 1) * 8 + e], c, -mc));
        const float p1 = fast_exp2(fmaf(s[c16 >> 1][(c16 & 1) * 8 + e + 1], c, -mc));
        pf[c16][e >> 1] = pack_f16(p0, p1);
        if (D == 64) {
          l0 += p0;
          l1 += p1;
        } else {
          float& l = c16 & 1 ? l1 : l0;
          l += p0;
          l += p1;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    return l0 + l1;
  };
  auto lds_read = []() __attribute__((always_inline)) {  // the tile is read: another may take its place
    __builtin_amdgcn_s_waitcnt(0xC07F);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  h8 kf[2][kKS];
  auto read_k = [&]() __attribute__((always_inline)) {
    wait_vm<0>();
    asm volatile("" ::: "memory");
#pragma unroll
    for (int kk = 0; kk < kKS; ++kk)
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) kf[rb][kk] = swz_rows_at<D>(ka0, ka1, rb, kk);
    lds_read();
  };
  read_k();
  if (nt > 1) copy(Kb, ks.n, 1);
  for (int t = 0; t < nt; ++t) {
#pragma unroll
    for (int kk = 0; kk < kKS; ++kk)
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) s[rb] = mfma(kf[rb][kk], qf[kk], kk == 0 ? zero : s[rb]);
    __builtin_amdgcn_sched_barrier(0);
    if (t + 1 < nt) read_k();
    copy(Vb, vs.n, t);
    __builtin_amdgcn_sched_barrier(0);
    if (t == nt - 1) {  // the only tile with keys that do not count
      const int last = (CAUSAL ? min(q0 + i, N - 1) : N - 1) - t * kTile - 4 * hh;
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (acc_row(rb, r, 0) > last) s[rb][r] = -INFINITY;
    }
    float lt = 0.f;
    bool raise = t == 0 || t == nt - 1;
    if (!raise) {
      lt = exponentials();
      raise = __builtin_amdgcn_ballot_w64(!(lt <= kRescaleSum)) != 0;
    }
    if (raise) {  // the maximum is brought up to date, as by raise_max of the kernel below
      float mx = s[0][0];
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[rb][r]);
      mx = fmaxf(mx, other_half(mx));
      const float mc_new = fmaxf(mc, mx * c);
      const float alpha = fast_exp2(mc - mc_new);
      mc = mc_new;
      l_run *= alpha;
      asm volatile("" : "+v"(l_run));
#pragma unroll
      for (int db = 0; db < kDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
      lt = exponentials();
    }
    l_run += lt;
    wait_vm<0>();
    asm volatile("" ::: "memory");
    {
      constexpr int kLead = 4, kNP = 4 * kDB;
      h8 frag[kLead];
#pragma unroll
      for (int n = 0; n < kLead; ++n) frag[n] = swz_cols_at<D>(va0, va1, n / kDB, n % kDB);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < kNP; ++n) {
        o[n % kDB] = mfma(frag[n % kLead], __builtin_bit_cast(h8, pf[n / kDB]), o[n % kDB]);
        if (n + kLead < kNP) frag[n % kLead] = swz_cols_at<D>(va0, va1, (n + kLead) / kDB, (n + kLead) % kDB);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    lds_read();
    if (t + 2 < nt) copy(Kb, ks.n, t + 2);
  }
  const float l_tot = l_run + other_half(l_run);
  store_resident<D>(O + ((long)b * N * H + h) * D, H * D, q0, N, o, 1.f / l_tot, lane, ring);
  if (LSE && lane < 32 && q0 + i < N) LSE[((long)b * H + h) * N + q0 + i] = (mc + __builtin_amdgcn_logf(l_tot)) * kLn2;
}

// The arguments of the kernel below as they lie in memory (checked behind it), and a second look at them.  A work group with the last
// rows of slices takes them from there: from the loads at the kernel's start they stay in registers across the branch for both
// ways, which spills six vector registers in the main body at D = 128, where without that way it spills three, and 22 to 25
// scalar ones at both head sizes, where it spills none.  Forward, us that way and this way, N x slices: D = 128 129 x 400 16.4, 15.9;
// causal 14.3, 13.9; 385 x 300 causal 33.0, 32.6; 1031 x 60 43.3, 43.2; D = 64 129 x 400 8.8, 8.5; 520 x 160 23.0, 22.7; 391 x 300
// causal 20.7, 20.0.  With PipeArgs as the one parameter of the kernel, variants without that way got slower: D = 64, 300 x 80
// causal 7.2, 7.4.
struct PipeArgs {
  const half_t *Q, *K, *V;
  Strides qs, ks, vs;
  half_t* O;
  float* LSE;
  FmhaDivisor H;
  int N;
  FmhaOrder order;
  int nb, tails, tails_per_block;
  float c;
  int negate_q;
};
__device__ __forceinline__ PipeArgs pipe_args_again() {
  typedef __attribute__((address_space(4))) const unsigned Word;
  Word* from = (Word*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(from));
  struct Words {
    unsigned w[sizeof(PipeArgs) / 4];
  } words;
#pragma unroll
  for (unsigned i = 0; i < sizeof(PipeArgs) / 4; ++i) words.w[i] = from[i];
  return __builtin_bit_cast(PipeArgs, words);
}
template <int D, bool CAUSAL, bool ODD_FIRST, bool TAIL>
__global__ void __launch_bounds__(kPipeThreads, 2)
fmha_fwd_pipe_kernel(const half_t* __restrict__ Q, const half_t* __restrict__ K, const half_t* __restrict__ V,
                     Strides qs, Strides ks, Strides vs, half_t* __restrict__ O, float* __restrict__ LSE, FmhaDivisor H, int N,
                     FmhaOrder order, int nb, int tails, int tails_per_block, float c, int negate_q) {
  using G = TileGeom<D>;
  using T = SwzTile<D>;
  constexpr int kDB = G::kDBlocks;
  constexpr int kIPW = T::kInstrs / kPipeWaves;
  static_assert(kIPW == T::kNC, "a wave copies the 16 rows of one block row of a tile");
  // two K tiles, then two V tiles; tile t of either sits in slot t & 1
  __shared__ __attribute__((aligned(1024))) char smem[4 * T::kBytes];
  constexpr int kVOff = 2 * T::kBytes;

  load_all_now(Q, K, V, H, N, order.run, order.last_level, order.slices, nb, qs, ks, vs, negate_q);
  if (ODD_FIRST) odd_slots_first();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // what depends on the lane is worked out again where it is needed, not kept in registers across the main loop
  auto lane_now = []() __attribute__((always_inline)) {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t & 63;
  };
  int bh, mb;
  const int lin = CAUSAL ? fmha_paired_block(blockIdx.x, gridDim.x) : blockIdx.x;
  if constexpr (TAIL) {
    if (lin < tails) {
      const PipeArgs a = pipe_args_again();
      bh = fmha_tail_slice(lin, wave, a.tails, a.tails_per_block);
      if (wave < a.tails_per_block && bh < a.order.slices)
        fwd_tail_rows<D, CAUSAL>(a.Q, a.K, a.V, a.qs, a.ks, a.vs, a.O, a.LSE, a.H, a.N, bh, a.c, a.negate_q, smem + wave * T::kBytes);
      return;
    }
  }
  fmha_ordered_block(TAIL ? lin - tails : lin, order.slices, order.run, order.last_level, CAUSAL,
                     !TAIL && order.short_last, bh, mb);
  const int mblk = CAUSAL ? nb - 1 - mb : mb;  // heavy blocks first
  const int b = bh / H, h = bh - b * H;
  const int rs = H * D;  // O is dense
  const long head_off = ((long)b * N * H + h) * D;
  const int m0 = mblk * kPipeBlockQ;
  const int q0w = m0 + wave * kResident;

  const int nt_all = (N + kTile - 1) / kTile;
  int nt = nt_all, ntw = q0w < N ? nt_all : 0;  // tiles the block streams; tiles this wave works on
  if (CAUSAL) {
    nt = min(nt, (min(m0 + kPipeBlockQ, N) - 1) / kTile + 1);
    ntw = q0w < N ? min(nt, (min(q0w + kResident, N) - 1) / kTile + 1) : 0;
  }

  // Wave w copies rows 16 w .. 16 w + 15 of every tile, 64 bytes of each per instruction; in the last tile rows past
  // the end re-read row N-1.  Offsets are relative to kBack bytes before the tile (see copy16_blocks).
  constexpr int kBack = 960 * (kIPW - 1);
  int k_goff, v_goff, c_past;  // c_past: how many rows past the end this lane's row of the last tile is
  {
    const int lane = lane_now(), row = 16 * wave + (lane >> 2), col = ((lane & 3) ^ swz(lane >> 4)) * 16;
    k_goff = row * ks.n * 2 + col + kBack;
    v_goff = row * vs.n * 2 + col + kBack;
    asm volatile("" : "+v"(k_goff), "+v"(v_goff));
    c_past = max((nt_all - 1) * kTile + row - (N - 1), 0) * 2;
  }
  const half_t* kp = K + b * ks.b + (long)h * ks.h - kBack / 2;  // the next tile to copy
  const half_t* vp = V + b * vs.b + (long)h * vs.h - kBack / 2;
  const unsigned lds0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
  const unsigned lds_w = lds0 + wave * (kIPW * 1024);
  auto copy_k = [&](int tile, int slot) __attribute__((always_inline)) {
    if (tile == nt_all - 1) k_goff -= c_past * ks.n;
    copy16_blocks<kIPW>(kp, k_goff, lds_w + slot * T::kBytes);
    kp += (long)kTile * ks.n;
  };
  auto copy_v = [&](int tile, int slot) __attribute__((always_inline)) {
    if (tile == nt_all - 1) v_goff -= c_past * vs.n;
    copy16_blocks<kIPW>(vp, v_goff, lds_w + kVOff + slot * T::kBytes);
    vp += (long)kTile * vs.n;
  };
  char* const my_rows = smem + kVOff + wave * (T::kBytes / 2);  // the block's rows of Q fill the slots of V, which comes later
  copy_rows<D>(Q + b * qs.b + (long)h * qs.h, qs.n, q0w, N, lane_now(), my_rows);
  copy_k(0, 0);
  if (nt > 1) copy_k(1, 1);
  h8 qf[G::kKSteps];
  int k_off[2], v_off[2];
  swz_rows_off<D>(lane_now(), k_off);
  swz_cols_off<D>(lane_now(), v_off);
  const unsigned ka0 = opaque_lds_address(smem + k_off[0]), ka1 = opaque_lds_address(smem + k_off[1]);
  const unsigned va0 = opaque_lds_address(smem + v_off[0]), va1 = opaque_lds_address(smem + v_off[1]);
  auto k_frag = [&](unsigned at, int n) __attribute__((always_inline)) {  // at: byte offset of the tile's slot
    return swz_rows_at<D>(ka0 + at, ka1 + at, n & 1, n >> 1);
  };
  auto v_frag = [&](unsigned at, int n) __attribute__((always_inline)) {
    return swz_cols_at<D>(va0 + kVOff + at, va1 + kVOff + at, n / kDB, n % kDB);
  };

  f16v o[kDB];
#pragma unroll
  for (int db = 0; db < kDB; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0.f;
  float mc = -INFINITY, l_run = 0.f;
  f16v sA[2], sB[2];
  u4v pf[4];  // probabilities of a tile, fp16 pairs in B-operand order
  f16v zero;
#pragma unroll
  for (int r = 0; r < 16; ++r) zero[r] = 0.f;

  constexpr int kLead = 3;  // LDS fragments are read this many MFMAs ahead (2 to 5 make no difference)
  constexpr int kNS = 2 * G::kKSteps, kNP = 4 * kDB;  // MFMAs of a tile: scores, accumulation
  static_assert(kNS == kNP, "");
  auto scores = [&](unsigned at, f16v (&s)[2]) __attribute__((always_inline)) {
    h8 frag[kLead];
#pragma unroll
    for (int n = 0; n < kLead; ++n) frag[n] = k_frag(at, n);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < kNS; ++n) {
      const int rb = n & 1, kk = n >> 1;
      s[rb] = mfma(frag[n % kLead], qf[kk], kk == 0 ? zero : s[rb]);
      if (n + kLead < kNS) frag[n % kLead] = k_frag(at, n + kLead);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // A lane's sum over a tile has two parts.  At D = 128 the even and the odd chunks of 16 keys, which are the parts that
  // two lanes of fmha_fwd_kernel have; at D = 64 the even and the odd keys, which wait less for each other.
  auto add_up = [&](float& l0, float& l1, int c16, float p0, float p1) __attribute__((always_inline)) {
    if (D == 64) {
      l0 += p0;
      l1 += p1;
    } else {
      float& l = c16 & 1 ? l1 : l0;
      l += p0;
      l += p1;
    }
  };
  auto exponentials = [&](const f16v (&s)[2]) __attribute__((always_inline)) {
    float l0 = 0.f, l1 = 0.f;
#pragma unroll
    for (int c16 = 0; c16 < 4; ++c16) {
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const float p0 = fast_exp2(fmaf(s[c16 >> 1][(c16 & 1) * 8 + e], c, -mc));
        const float p1 = fast_exp2(fmaf(s[c16 >> 1][(c16 & 1) * 8 + e + 1], c, -mc));
        pf[c16][e >> 1] = pack_f16(p0, p1);
        add_up(l0, l1, c16, p0, p1);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    return l0 + l1;
  };
  auto mask = [&](f16v (&s)[2], int t) __attribute__((always_inline)) {
    const int key0 = t * kTile;
    if ((CAUSAL && key0 + kTile - 1 > q0w) || (key0 + kTile > N)) {
      const int lane = lane_now();
      const int last = (CAUSAL ? min(q0w + (lane & 31), N - 1) : N - 1) - key0 - 4 * (lane >> 5);  // last key that counts
#pragma unroll
      for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (acc_row(rb, r, 0) > last) s[rb][r] = -INFINITY;
    }
  };
  auto too_large = [&](float lt) __attribute__((always_inline)) {
    return __builtin_amdgcn_ballot_w64(!(lt <= kRescaleSum)) != 0;
  };
  // probabilities of a tile with the running maximum brought up to date
  auto raise_max = [&](const f16v (&s)[2]) __attribute__((always_inline)) {
    float mx = s[0][0];
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[rb][r]);
    mx = fmaxf(mx, other_half(mx));
    const float mc_new = fmaxf(mc, mx * c);
    const float alpha = fast_exp2(mc - mc_new);
    mc = mc_new;
    l_run *= alpha;
    asm volatile("" : "+v"(l_run));  // rounded here, as in fmha_fwd_kernel
#pragma unroll
    for (int db = 0; db < kDB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
    l_run += exponentials(s);
  };
  auto accumulate = [&](unsigned at) __attribute__((always_inline)) {
    h8 frag[kLead];
#pragma unroll
    for (int n = 0; n < kLead; ++n) frag[n] = v_frag(at, n);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < kNP; ++n) {
      o[n % kDB] = mfma(frag[n % kLead], __builtin_bit_cast(h8, pf[n / kDB]), o[n % kDB]);
      if (n + kLead < kNP) frag[n % kLead] = v_frag(at, n + kLead);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Iteration j uses K(j+1) and V(j-1), both in slot (j+1) & 1; K(j+2) and V(j) are copied into the other one.
  auto top_wait = [&]() __attribute__((always_inline)) {
    wait_vm<0>();
    block_barrier();
  };
  auto top_copy = [&](int j, int slot) __attribute__((always_inline)) {
    if (j + 2 < nt) copy_k(j + 2, slot);
    if (j < nt) copy_v(j, slot);
  };
  // The pipelined step of tile j: softmax(j) with the MFMAs of accumulate(j-1) and scores(j+1) spread between its
  // vector instructions.  Per 16 keys: kDB MFMAs of the accumulation, then as many of the scores.
  auto step = [&](int j, auto slot_tag, const f16v (&s)[2], f16v (&sn)[2]) __attribute__((always_inline)) {
    constexpr int kSlot = decltype(slot_tag)::value;  // (j + 1) & 1
    constexpr unsigned at = kSlot * T::kBytes;
    constexpr int kM = kNS + kNP;
    h8 frag[kLead];
    float l0 = 0.f, l1 = 0.f, p0 = 0.f, p1 = 0.f;
    auto read = [&](int m) __attribute__((always_inline)) {
      const int ch = m / (2 * kDB), in = m % (2 * kDB);
      return in < kDB ? v_frag(at, ch * kDB + in) : k_frag(at, ch * kDB + in - kDB);
    };
    auto reads = [](int m) { return m >= kM ? 0 : m % (2 * kDB) < kDB ? 2 : 1; };  // LDS reads of a fragment
    auto start = [&](int x) __attribute__((always_inline)) {
      const int c16 = x >> 2, e = (x & 3) * 2;
      p0 = fast_exp2(fmaf(s[c16 >> 1][(c16 & 1) * 8 + e], c, -mc));
      p1 = fast_exp2(fmaf(s[c16 >> 1][(c16 & 1) * 8 + e + 1], c, -mc));
    };
    auto finish = [&](int x) __attribute__((always_inline)) {
      const int c16 = x >> 2, e = (x & 3) * 2;
      add_up(l0, l1, c16, p0, p1);
      asm volatile("" : "+v"(l0), "+v"(l1));  // sums now, not all at the end
      pf[c16][e >> 1] = pack_f16(p0, p1);
    };
    top_wait();
#pragma unroll
    for (int m = 0; m < kLead; ++m) frag[m] = read(m);
    // At D = 128 a step's eight copies, issued by all waves at once, hold them until the copy path has taken them (64
    // bytes per clock and CU): K follows when V is through.  B1 H2 N4000: 54.6 -> 50.8 us, B3 H20 N1031: 50.4 -> 49.6.
    // Much later (unit 28: 61.4 us) it does not arrive in time.  At D = 64 there are half as many and it changes nothing.
    constexpr int kCopyKAt = D == 128 ? 8 : 0;
    if (j < nt) copy_v(j, 1 - kSlot);
    if (kCopyKAt == 0 && j + 2 < nt) copy_k(j + 2, 1 - kSlot);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < kM + 2; ++m) {
      if (kCopyKAt != 0 && m == kCopyKAt && j + 2 < nt) copy_k(j + 2, 1 - kSlot);
      if (m < kM && m % 2 == 0) {
        // One wait for the fragments of this unit and the next instead of the compiler's one before each: a wave alone on
        // its SIMD pays for every instruction.  B1 H4 N8192 D64: 80.2 -> 79.2 us, B1 H12 N8192 D64: 217 -> 214, B1 H32
        // N1500 D128 causal: 29.6 -> 28.8, B1 H2 N4000 D128: 51.0 -> 49.1.  At D = 128 the first MFMA may move before it
        // (pinned: 50.0).
        if (D == 64) wait_lds_pinned(reads(m + 2));
        else wait_lds(reads(m + 2));
      }
      if (m < kM) {
        const int ch = m / (2 * kDB), in = m % (2 * kDB);
        if (in < kDB) {
          o[in] = mfma(frag[m % kLead], __builtin_bit_cast(h8, pf[ch]), o[in]);
        } else {
          const int n = ch * kDB + in - kDB, rb = n & 1, kk = n >> 1;
          sn[rb] = mfma(frag[m % kLead], qf[kk], kk == 0 ? zero : sn[rb]);
        }
        if (m + kLead < kM) frag[m % kLead] = read(m + kLead);
      }
      if (D == 64) {
        if (m >= 1 && m - 1 < 16) finish(m - 1);
        if (m < 16) start(m);
      } else {
        if (m & 1) {
          if (m >= 3 && m < 35) finish((m - 3) / 2);
        } else if (m >= 2 && m < 34) {
          start((m - 2) / 2);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    return l0 + l1;
  };

  if (nt > 1) wait_vm<kIPW>();  // the second tile of K may still be on its way
  else wait_vm<0>();
  asm volatile("" ::: "memory");
  {
    const StagedRows<D> rows{my_rows, lane_now()};
#pragma unroll
    for (int kk = 0; kk < G::kKSteps; ++kk) qf[kk] = rows.wide(kk);
    staged_rows_read();
  }
  if (negate_q) {
#pragma unroll
    for (int kk = 0; kk < G::kKSteps; ++kk) {
      qf[kk] = -qf[kk];
      asm volatile("" : "+v"(qf[kk]));
    }
  }
  block_barrier();
  if (ntw > 0) scores(0, sA);
  int j = 0;
  if (ntw > 1) {
    top_wait();
    top_copy(0, 0);
    scores(T::kBytes, sB);
    raise_max(sA);
    ++j;
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) sA[rb] = sB[rb];
    // Main loop, two tiles per round, the scores alternating between two sets of registers: those of odd tiles in
    // sA, of even ones in sB.  It is left where a tile's probabilities came out too large, so that what has to be
    // done then is not held twice.  At D = 128 the kernel still uses all 256 registers and spills three (16 bytes of
    // scratch per lane): two across the whole loop, one in the path that raises the maximum, where the reload waits for
    // the tile copies in flight.  Nothing is spilled or reloaded inside a step.
    // A wave alone on its SIMD is held up where instructions are fetched across a 32-byte line at the wrong place.  The nops, which run
    // once, put the loop where it was fastest in the variants without work groups for last rows, as ROCm 7.2.0's compiler lays them out:
    // it begins on a line at D = 128 and 24 bytes past one at D = 64 (tests/test_code_object.py has it by the first barrier; where
    // that moves, time 0 to 7 nops again).  us with the loop at + 8, 12, 16, 20, 24, 28, 0 and 4: D = 128 8415 x 3 causal 97.2, 96.3,
    // 96.1, 97.5, 95.8, 97.3, 95.2, 98.1; 4000 x 2 49.0, 49.0, 48.9, 49.8, 48.7, 49.0, 48.4, 48.7; causal 48.2, 48.2, 48.2, 49.0, 47.9,
    // 48.2, 47.6, 48.0; D = 64 8143 x 6 causal 79.1, 79.6, 79.9, 79.9, 79.1, 79.7, 79.2, 79.2; 8192 x 3 71.9, 72.4, 72.4, 72.6, 72.1, 72.6,
    // 72.3, 72.1.  The variants with such work groups have the loop 8 bytes further on; they run two waves to a SIMD and are within
    // 0.6 % wherever it is (1031 x 60 43.1 to 43.5, D = 64 520 x 60 12.65 to 12.77).
    asm volatile(".p2align 6\n\t.rept %0\n\ts_nop 0\n\t.endr" ::"n"(D == 128 ? 6 : 4));
    bool odd_done = false;
    for (;;) {
      int why;
      for (;;) {
        if (!odd_done) {
          if (j + 2 > ntw) { why = 0; break; }
          const float lt = step(j, IntTag<0>{}, sA, sB);
          if (too_large(lt)) { why = 1; break; }
          l_run += lt;
          ++j;
        }
        odd_done = false;
        if (j + 2 > ntw) { why = 2; break; }
        const float lt = step(j, IntTag<1>{}, sB, sA);
        if (too_large(lt)) { why = 3; break; }
        l_run += lt;
        ++j;
      }
      if (why == 0) break;
      if (why == 2) {
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) sA[rb] = sB[rb];
        break;
      }
      if (why == 1) raise_max(sA);
      else raise_max(sB);
      ++j;
      odd_done = why == 1;
    }
  }
  // the wave's last tile (the one with a mask, if any) and the accumulation after it
  for (; j <= nt; ++j) {
    const unsigned at = ((j + 1) & 1) * T::kBytes;
    top_wait();
    top_copy(j, j & 1);
    if (j > 0 && j <= ntw) accumulate(at);
    if (j < ntw) {
      mask(sA, j);
      raise_max(sA);
    }
  }

  block_barrier();  // every wave is done with the rings: they become the staging tiles
  const int lane = lane_now(), qi = q0w + (lane & 31);
  const float l_tot = l_run + other_half(l_run);
  const float inv = 1.f / l_tot;
  store_resident<D>(O + head_off, rs, q0w, N, o, inv, lane, smem + wave * StageGeom<D>::kBytes);
  if (LSE && lane < 32 && qi < N) LSE[((long)b * H + h) * N + qi] = (mc + __builtin_amdgcn_logf(l_tot)) * kLn2;
}
// A kernel's arguments lie one behind the other, each at the next multiple of its own alignment.
template <typename... Params>
constexpr bool lie_at(void (*)(Params...), const size_t (&at)[sizeof...(Params)]) {
  constexpr size_t size[] = {sizeof(Params)...}, align[] = {alignof(Params)...};
  size_t next = 0;
  for (size_t i = 0; i < sizeof...(Params); ++i) {
    next = (next + align[i] - 1) / align[i] * align[i];
    if (next != at[i]) return false;
    next += size[i];
  }
  return true;
}
#define AT(member) offsetof(PipeArgs, member)
static_assert(lie_at(fmha_fwd_pipe_kernel<64, false, false, true>,
                     {AT(Q), AT(K), AT(V), AT(qs), AT(ks), AT(vs), AT(O), AT(LSE), AT(H), AT(N), AT(order), AT(nb), AT(tails),
                      AT(tails_per_block), AT(c), AT(negate_q)}),
              "PipeArgs is not what the kernel takes");
#undef AT

// ---------------------------------------------------------------------------
// delta[b][h][n] = sum_d dO * O in fp32.  One 16-byte chunk per thread.
// Takes the place of the two PyTorch ops at reference
// flash_attn_interface.py:43-44 (which work in fp16).  Also writes the
// logsumexp scaled to the exp2 domain, lse2 = lse * log2(e), behind delta in
// the workspace, so the dK/dV pass gets both row statistics with one copy.
// Bound by its bytes (5.6-6.1 TB/s on tensors used again and again; small problems take 7 us to start and end).  Rows are
// numbered through slice by slice, which is the order of the statistics: a block writes its 16 (D = 64: 32) together, and
// none of it idles where sequences are short.  Slice and row come from divisions of the block's first row by the scalar unit;
// only threads past the end of that slice divide again.  Blocks in flight at a time are those of the same positions of
// different heads (fmha_interleaved_block), so that O and dO are read through: in the order of the rows, 256 bytes of each
// position, strides that are a power of two can meet in a few channels.  D = 128, us: rows in the order of O with three 64-bit
// divisions a thread; blocks one after the other in this order, with an end at each slice; and as it is: B1024 H32 N1 7.2,
// 11.9, 6.9; B256 H32 N17 14.8, 18.9, 14.3; B3 H20 N1031 7.1, 6.9, 6.9; B64 H16 N512 52.9, 46.1, 45.8; B2 H40 N2048 18.1, 15.2,
// 15.4; B2 H32 N4096 25.4, 28.6, 23.6; B1 H64 N8192 44.7, 45 or 68 by where the tensors lie, 44.8; B1 H16 N32768 52, 46, 43.
// ---------------------------------------------------------------------------
constexpr int delta_rows(int d) { return 256 * 8 / d; }  // of a block
template <int D>
__global__ void __launch_bounds__(256)
fmha_bwd_delta_kernel(const half_t* __restrict__ O, const half_t* __restrict__ dO, Strides gs,
                      const float* __restrict__ LSE, float* __restrict__ delta, float* __restrict__ lse2, FmhaDivisor H,
                      FmhaDivisor N, int first, int end, int chain, FmhaDivisor chains, unsigned* __restrict__ clear,
                      unsigned words) {
  constexpr int kLanesPerRow = D / 8;
  for (unsigned at = blockIdx.x * 256 + threadIdx.x; at < words; at += gridDim.x * 256) clear[at] = 0;  // for a later kernel
  const int row0 = first + fmha_interleaved_block((int)blockIdx.x, chain, chains) * delta_rows(D);  // rows first .. end - 1
  const int slice0 = row0 / N, b0 = slice0 / H;
  const int in_block = threadIdx.x / kLanesPerRow, row = row0 + in_block, c = threadIdx.x % kLanesPerRow;
  int n = row0 - slice0 * N + in_block, h = slice0 - b0 * H, b = b0;
  if (n >= N) {  // past the end of the slice that the block starts in
    const int later = n / N;
    n -= later * N;
    h += later;
    if (h >= H) {
      const int batches = h / H;
      b += batches;
      h -= batches * H;
    }
  }
  float acc = 0.f;
  if (row < end) {  // O is dense, dO has its own strides
    const h8 a = *reinterpret_cast<const h8*>(O + (((long)b * N + n) * H + h) * D + c * 8);
    const h8 g = *reinterpret_cast<const h8*>(dO + b * gs.b + (long)n * gs.n + (long)h * gs.h + c * 8);
#pragma unroll
    for (int j = 0; j < 8; ++j) acc = fmaf((float)a[j], (float)g[j], acc);
  }
#pragma unroll
  for (int off = kLanesPerRow / 2; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
  if (row < end && c == 0) {
    delta[row] = acc;
    lse2[row] = LSE[row] * kLog2e;
  }
}

// ---------------------------------------------------------------------------
// Backward, dQ pass.  Block = 128 queries = 4 pairs of waves; a pair owns 32
// queries and splits the work (two waves per SIMD fit):
//   wave A (waves 0-3), tile j: S^T = K Q^T, P^T = exp(S^T - lse) -> P^T(j) to LDS
//   wave B (waves 4-7), tile j: dS^T(j-1) = P^T(j-1) o T(j-1), dQ^T += K(j-1)^T dS^T(j-1),
//                               then dP^T = V(j) dO^T, T(j) = dP^T - delta (kept in registers,
//                               as -T: the GEMM runs on -dO with accumulators that start at delta)
// (formulas: reference kernel/fused_mha_kernel.cu:598-603, 653-656, 680-683).
// B runs one tile behind A for the part that needs P^T, so one barrier per tile
// is enough and neither wave waits for the other inside a tile.  lse and delta
// belong to the resident query, so they are per-lane scalars.  P^T travels in
// the accumulator layout, lane for lane (double-buffered).  K tiles of 64 keys
// stream through a 4-slot LDS ring (B still needs tile j-1), V tiles through a
// 3-slot ring, both copied two tiles ahead.
// ---------------------------------------------------------------------------
constexpr int kDqPairs = 4;
constexpr int kDqWaves = 2 * kDqPairs;
constexpr int kDqThreads = kDqWaves * 64;
constexpr int kDqBlockQ = kDqPairs * kResident;

// STATS: the kernel also produces the two row statistics of the backward,
// delta = rowsum(dO o O) and lse2 = lse * log2(e), for its own queries, uses
// them and stores them in the workspace; fmha_bwd_delta_kernel is not needed in
// that case.  A dK/dV pass that reads them must be launched after this one; the
// dK/dV blocks that share a launch with these (fmha_bwd_both_kernel) form their
// own.  Otherwise delta is read from the workspace.
template <int D>
constexpr int dq_lds() { return 7 * SwzTile<D>::kBytes + 2 * kDqPairs * 4096; }
template <int D, bool CAUSAL, bool STATS>
__device__ __forceinline__ void
bwd_dq_block(const half_t* __restrict__ Q, const half_t* __restrict__ K, const half_t* __restrict__ V,
             const half_t* __restrict__ O, const half_t* __restrict__ dO, Strides qs, Strides ks, Strides vs, Strides gs,
             const float* __restrict__ LSE, float* __restrict__ delta, float* __restrict__ lse2, half_t* __restrict__ dQ, FmhaDivisor H,
             int N, float c, float scale, char* smem, int bh, int mblk) {
  using G = TileGeom<D>;
  using T = SwzTile<D>;
  constexpr int kIPW = T::kInstrs / kDqWaves;  // copies per wave per tile, per tensor
  // K ring (4), V ring (3), then two buffers of per pair a 64x32 fp16 block (4 KiB) of P^T
  constexpr int kPBytes = kDqPairs * 4096;
  static_assert(dq_lds<D>() == 7 * T::kBytes + 2 * kPBytes, "");
  char* const k_ring = smem;
  char* const v_ring = smem + 4 * T::kBytes;
  char* const p_xchg = smem + 7 * T::kBytes;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pair = wave & (kDqPairs - 1);
  const bool role_b = wave >= kDqPairs;
  const int i = lane & 31, hh = lane >> 5;
  const int b = bh / H, h = bh - b * H;
  const int rs = H * D;  // O and dQ are dense
  const long head_off = ((long)b * N * H + h) * D;
  const half_t* Kb = K + b * ks.b + (long)h * ks.h;
  const half_t* Vb = V + b * vs.b + (long)h * vs.h;

  const int m0 = mblk * kDqBlockQ;
  const int q0w = m0 + pair * kResident;
  const int qi = q0w + i;
  const int qrow = min(qi, N - 1);

  int nt = (N + kTile - 1) / kTile;  // tiles the block streams
  int ntw = nt;                      // tiles this pair takes part in
  if (CAUSAL) {
    nt = min(nt, (min(m0 + kDqBlockQ, N) - 1) / kTile + 1);
    ntw = min(nt, (min(q0w + kResident, N) - 1) / kTile + 1);
    if (q0w >= N) ntw = 0;
  }

  int c_row[kIPW], c_kgoff[kIPW], c_vgoff[kIPW], c_blk[kIPW];
#pragma unroll
  for (int u = 0; u < kIPW; ++u) {
    const int t = wave * kIPW + u;
    copy_src<D>(t, lane, ks.n, c_row[u], c_kgoff[u]);
    copy_src<D>(t, lane, vs.n, c_row[u], c_vgoff[u]);
    c_blk[u] = t * 1024;
  }
  auto copy_tiles = [&](int j) __attribute__((always_inline)) {
    const int row0 = j * kTile;
    const half_t* kp = Kb + (long)row0 * ks.n;  // wave-uniform
    const half_t* vp = Vb + (long)row0 * vs.n;
    char* kdst = k_ring + (j & 3) * T::kBytes;
    char* vdst = v_ring + (j % 3) * T::kBytes;
    if (row0 + kTile <= N) {
#pragma unroll
      for (int u = 0; u < kIPW; ++u) copy16(kp, c_kgoff[u], kdst + c_blk[u]);
#pragma unroll
      for (int u = 0; u < kIPW; ++u) copy16(vp, c_vgoff[u], vdst + c_blk[u]);
    } else {
#pragma unroll
      for (int u = 0; u < kIPW; ++u) {  // rows past the end re-read row N-1
        const int back = max(row0 + c_row[u] - (N - 1), 0);
        copy16(kp, c_kgoff[u] - back * ks.n * 2, kdst + c_blk[u]);
      }
#pragma unroll
      for (int u = 0; u < kIPW; ++u) {
        const int back = max(row0 + c_row[u] - (N - 1), 0);
        copy16(vp, c_vgoff[u] - back * vs.n * 2, vdst + c_blk[u]);
      }
    }
  };

  // rows of Q: slots 2 and 3 of K; of dO: slot 2 of V and the buffers of P
  char* const my_rows = !role_b ? k_ring + 2 * T::kBytes + pair * (T::kBytes / 2)
                        : pair < 2 ? v_ring + 2 * T::kBytes + pair * (T::kBytes / 2) : p_xchg + (pair - 2) * (T::kBytes / 2);
  static_assert(2 * kPBytes >= T::kBytes, "the rows of dO of two pairs fit where P goes");
  if (role_b) copy_rows<D>(dO + b * gs.b + (long)h * gs.h, gs.n, q0w, N, lane, my_rows);
  else copy_rows<D>(Q + b * qs.b + (long)h * qs.h, qs.n, q0w, N, lane, my_rows);
  copy_tiles(0);
  if (nt > 1) copy_tiles(1);

  // resident rows of this wave: Q for role A, dO for role B; and the row statistic it needs
  h8 rf[G::kKSteps];
  const long stat_at = ((long)b * H + h) * N + qrow;
  float stat;
  {
    h8 ov[STATS ? G::kKSteps : 1];
    if (STATS && role_b) {
      const half_t* op = O + head_off + (long)qrow * rs + hh * 8;
#pragma unroll
      for (int kk = 0; kk < (STATS ? G::kKSteps : 1); ++kk) ov[kk] = *reinterpret_cast<const h8*>(op + kk * 16);
    }
    staged_rows_landed();
    const StagedRows<D> rows{my_rows, lane};
#pragma unroll
    for (int kk = 0; kk < G::kKSteps; ++kk) rf[kk] = rows.wide(kk);
    staged_rows_read();
    if (STATS) {
      if (role_b) {
        // delta of this lane's query.  The lane has every other 8-feature chunk of
        // the row; the partial sums are combined in the order of
        // fmha_bwd_delta_kernel's shuffle tree, so both give the same bits.
        float part[G::kKSteps];
#pragma unroll
        for (int kk = 0; kk < G::kKSteps; ++kk) {
          part[kk] = 0.f;
#pragma unroll
          for (int e = 0; e < 8; ++e) part[kk] = fmaf((float)ov[STATS ? kk : 0][e], (float)rf[kk][e], part[kk]);
        }
#pragma unroll
        for (int stride = G::kKSteps / 2; stride > 0; stride >>= 1)
#pragma unroll
          for (int kk = 0; kk < stride; ++kk) part[kk] += part[kk + stride];
        stat = part[0] + other_half(part[0]);
        if (hh == 0 && qi < N) delta[stat_at] = stat;
      } else {
        stat = LSE[stat_at] * kLog2e;
        if (hh == 0 && qi < N) lse2[stat_at] = stat;
      }
    } else {
      stat = role_b ? delta[stat_at] : LSE[stat_at] * kLog2e;
    }
    // Role B works with -dO: its first GEMM then gives delta - dP^T on top of
    // accumulators that start at delta, with no subtraction afterwards.
    if (role_b) {
#pragma unroll
      for (int kk = 0; kk < G::kKSteps; ++kk) rf[kk] = -rf[kk];
    }
  }

  int r_off[2], c_off[2];
  swz_rows_off<D>(lane, r_off);
  swz_cols_off<D>(lane, c_off);
  char* const p_mine = p_xchg + pair * 4096 + lane * 16;  // + buffer * kPBytes + rb * 2048 + half * 1024

  // first GEMM of a tile: rows of K (role A) or V (role B) against the resident
  // rows, on top of the value `init` in every accumulator element
  auto gemm1 = [&](const char* tile_lds, f16v (&x)[2], float init) __attribute__((always_inline)) {
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int r = 0; r < 16; ++r) x[rb][r] = init;
#pragma unroll
    for (int kk = 0; kk < G::kKSteps; ++kk) {
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) x[rb] = mfma(swz_rows<D>(tile_lds, rb, kk, r_off), rf[kk], x[rb]);
    }
    constexpr int kN = 2 * G::kKSteps, kLead = 4;
    __builtin_amdgcn_sched_group_barrier(0x100, kLead, 0);
#pragma unroll
    for (int n = 0; n < kN - kLead; ++n) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kLead, 0);
  };
  // P^T = exp2(S^T*c - lse2) -> LDS.  MASKED tiles straddle the diagonal or the
  // end of the sequence.
  auto probabilities = [&](const f16v (&x)[2], char* pw, int key0, auto masked_tag) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value != 0;
#pragma unroll
    for (int rb = 0; rb < 2; ++rb) {
      h8 y0, y1;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float p = fast_exp2(fmaf(x[rb][r], c, -stat));
        if (MASKED) {
          const int key = key0 + acc_row(rb, r, hh);
          if ((CAUSAL && key > qi) || key >= N) p = 0.f;
        }
        if (r < 8) y0[r] = (half_t)p; else y1[r - 8] = (half_t)p;
      }
      *reinterpret_cast<h8*>(pw + rb * 2048) = y0;
      *reinterpret_cast<h8*>(pw + rb * 2048 + 1024) = y1;
    }
  };
  // Per iteration: wait for tile j (issued two iterations ago; the copies of tile
  // j+1 may still be in flight), one barrier, issue the copies of tile j+2.
  auto step_sync = [&](int j) __attribute__((always_inline)) {
    if (j + 1 < nt) wait_vm<2 * kIPW>();
    else wait_vm<0>();
    block_barrier();
    if (j + 2 < nt) copy_tiles(j + 2);
  };

  wait_vm<0>();  // resident rows, statistics and the first copies
  f16v dq[G::kDBlocks];  // role B's accumulator
  if (!role_b) {
    for (int j = 0; j <= nt; ++j) {
      step_sync(j);
      if (j < ntw) {
        const int key0 = j * kTile;
        const bool masked = (CAUSAL && key0 + kTile - 1 > q0w) || (key0 + kTile > N);
        f16v x[2];
        gemm1(k_ring + (j & 3) * T::kBytes, x, 0.f);
        char* pw = p_mine + (j & 1) * kPBytes;
        if (masked) probabilities(x, pw, key0, IntTag<1>{});
        else probabilities(x, pw, key0, IntTag<0>{});
      }
    }
  } else {
#pragma unroll
    for (int db = 0; db < G::kDBlocks; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) dq[db][r] = 0.f;
    f16v x[2];  // delta - dP^T of the previous tile
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
      for (int r = 0; r < 16; ++r) x[rb][r] = 0.f;
    for (int j = 0; j <= nt; ++j) {
      step_sync(j);
      if (j >= 1 && j - 1 < ntw) {  // the part that needs P^T, one tile behind
        const char* Kl = k_ring + ((j - 1) & 3) * T::kBytes;
        const char* pr = p_mine + ((j - 1) & 1) * kPBytes;
        h8 y[4];
#pragma unroll
        for (int rb = 0; rb < 2; ++rb) {
          const h8 p0 = *reinterpret_cast<const h8*>(pr + rb * 2048);
          const h8 p1 = *reinterpret_cast<const h8*>(pr + rb * 2048 + 1024);
          float xr[16];
#pragma unroll
          for (int e = 0; e < 16; ++e) xr[e] = x[rb][e];
          y[rb * 2] = neg_mul_to_f16x8(p0, xr);
          y[rb * 2 + 1] = neg_mul_to_f16x8(p1, xr + 8);
        }
#pragma unroll
        for (int c16 = 0; c16 < 4; ++c16) {
#pragma unroll
          for (int db = 0; db < G::kDBlocks; ++db) dq[db] = mfma(swz_cols<D>(Kl, c16, db, c_off), y[c16], dq[db]);
        }
        constexpr int kN = 4 * G::kDBlocks, kLead = 4;
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * kLead, 0);
#pragma unroll
        for (int n = 0; n < kN - kLead; ++n) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, kLead, 0);
      }
      if (j < ntw) gemm1(v_ring + (j % 3) * T::kBytes, x, stat);
    }
  }
  static_assert(kDqPairs * StageGeom<D>::kBytes <= 7 * T::kBytes, "the output staging tiles fit the rings");
  block_barrier();  // every wave is done with the rings: they become the staging tiles
  if (role_b) store_resident<D>(dQ + head_off, rs, q0w, N, dq, scale, lane, smem + pair * StageGeom<D>::kBytes);
}

template <int D, bool CAUSAL, bool STATS>
__global__ void __launch_bounds__(kDqThreads, 1)
fmha_bwd_dq_kernel(const half_t* __restrict__ Q, const half_t* __restrict__ K, const half_t* __restrict__ V,
                   const half_t* __restrict__ O, const half_t* __restrict__ dO, Strides qs, Strides ks, Strides vs,
                   Strides gs, const float* __restrict__ LSE, float* __restrict__ delta, float* __restrict__ lse2,
                   half_t* __restrict__ dQ, FmhaDivisor H, int N, FmhaDivisor nmb, int slices, float c, float scale) {
  __shared__ __attribute__((aligned(1024))) char smem[dq_lds<D>()];
  int bh, mb;
  fmha_slice_and_block(blockIdx.x, slices, nmb, bh, mb);
  bwd_dq_block<D, CAUSAL, STATS>(Q, K, V, O, dO, qs, ks, vs, gs, LSE, delta, lse2, dQ, H, N, c, scale, smem, bh,
                                 CAUSAL ? nmb - 1 - mb : mb);  // heavy blocks first
}

// ---------------------------------------------------------------------------
// Backward for D = 64: a dQ pass and a dK/dV pass that both form S and dP themselves, 4 waves of 32 resident rows per
// block, two blocks per CU, everything of a wave's rows inside that wave.
//
// At D = 64 writing and reading dS costs more than forming it twice: 4 bytes of HBM traffic per element against 256
// FLOP, and the wave-pair kernels behind it (probabilities handed over through LDS, one block per CU) were bound by
// latency.  Here, as in fmha_fwd_pipe_kernel, a wave's instruction stream interleaves the MFMAs of one step with the
// vector instructions of its neighbours, in units of one MFMA whose order is pinned.  us at B16 H12 N512 / B4 H16 N1024
// causal / B16 H16 N1024 / B4 H16 N4096 causal, against the wave-pair kernels over and without dS:
//   dQ pass     30 / 24 / 148 / 240   (22 / 18 / 106 / 217 plus delta pass 7 / 5 / 17 / 17; 40 / 38 / 172 / 315)
//   dK/dV pass  34 / 28 / 178 / 300   (45 / 44 / 275 / 455;                                 45 / 45 / 205 / 385)
// What bounds them: the issue of one instruction every 4-5 cycles per wave in small problems, the power limit (clock at
// 1.9 GHz) in large ones.  64 keys per wave with one wave per SIMD halves the LDS reads per MFMA but is slower or
// equal everywhere (43 / 36 / 179 / 310): a lone wave cannot cover its own issue gaps.
//
// dQ pass.  The formulas are those of fmha_bwd_dq_kernel, and so are the results, bit for bit.
// ---------------------------------------------------------------------------
constexpr int kDqPipeLds = 2 * 3 * SwzTile<64>::kBytes + 2 * SwzTile<64>::kBytes;  // rings, rows of O
template <bool CAUSAL, bool STATS>
__device__ __forceinline__ void
bwd_dq_pipe_block(const half_t* __restrict__ Q, const half_t* __restrict__ K, const half_t* __restrict__ V,
                  const half_t* __restrict__ O, const half_t* __restrict__ dO, Strides qs, Strides ks, Strides vs,
                  Strides gs, const float* __restrict__ LSE, float* __restrict__ delta, float* __restrict__ lse2,
                  half_t* __restrict__ dQ, FmhaDivisor H, int N, float c, float scale, char* smem, int bh, int mblk) {
  constexpr int D = 64;
  using G = TileGeom<D>;
  using T = SwzTile<D>;
  constexpr int kDB = G::kDBlocks, kKS = G::kKSteps;
  constexpr int kIPW = T::kInstrs / kPipeWaves;
  static_assert(kIPW == T::kNC, "a wave copies the 16 rows of one block row of a tile");
  constexpr int kSlots = 3;  // K tiles, then V tiles: the current one, the one before it, the one being copied
  constexpr int kVOff = kSlots * T::kBytes;
  static_assert(kDqPipeLds == 2 * kSlots * T::kBytes + kPipeWaves * T::kBytes / 2, "");

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 31, hh = lane >> 5;
  const int b = bh / H, h = bh - b * H;
  const int rs = H * D;  // O and dQ are dense
  const long head_off = ((long)b * N * H + h) * D;
  const int m0 = mblk * kPipeBlockQ;
  const int q0w = m0 + wave * kResident;
  const int qi = q0w + i, qrow = min(qi, N - 1);

  const int nt_all = (N + kTile - 1) / kTile;
  int nt = nt_all, ntw = q0w < N ? nt_all : 0;  // tiles the block streams; tiles this wave works on
  if (CAUSAL) {
    nt = min(nt, (min(m0 + kPipeBlockQ, N) - 1) / kTile + 1);
    ntw = q0w < N ? min(nt, (min(q0w + kResident, N) - 1) / kTile + 1) : 0;
  }

  // tile copies as in fmha_fwd_pipe_kernel
  constexpr int kBack = 960 * (kIPW - 1);
  int k_goff, v_goff, c_past;
  {
    const int row = 16 * wave + (lane >> 2), col = ((lane & 3) ^ swz(lane >> 4)) * 16;
    k_goff = row * ks.n * 2 + col + kBack;
    v_goff = row * vs.n * 2 + col + kBack;
    c_past = max((nt_all - 1) * kTile + row - (N - 1), 0) * 2;
  }
  const half_t* kp = K + b * ks.b + (long)h * ks.h - kBack / 2;  // the next tile to copy
  const half_t* vp = V + b * vs.b + (long)h * vs.h - kBack / 2;
  const unsigned lds_w = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem + wave * (kIPW * 1024);
  auto copy_tile = [&](int tile, int slot) __attribute__((always_inline)) {
    if (tile == nt_all - 1) {
      k_goff -= c_past * ks.n;
      v_goff -= c_past * vs.n;
    }
    copy16_blocks<kIPW>(kp, k_goff, lds_w + slot * T::kBytes);
    copy16_blocks<kIPW>(vp, v_goff, lds_w + kVOff + slot * T::kBytes);
    kp += (long)kTile * ks.n;
    vp += (long)kTile * vs.n;
  };
  copy_tile(0, 0);

  // Resident rows and the row statistics.  dO is negated: its product with V on top of delta gives delta - dP.  The rows come
  // through slots 1 and 2 of the rings, those of O behind them.
  h8 qf[kKS], gf[kKS];
  float my_lse2, my_delta;
  {
    char* const q_rows = smem + T::kBytes + wave * (T::kBytes / 2);
    copy_rows<D>(Q + b * qs.b + (long)h * qs.h, qs.n, q0w, N, lane, q_rows);
    copy_rows<D>(dO + b * gs.b + (long)h * gs.h, gs.n, q0w, N, lane, q_rows + kVOff);
    char* const o_rows = smem + 2 * kVOff + wave * (T::kBytes / 2);
    if (STATS) copy_rows<D>(O + head_off, rs, q0w, N, lane, o_rows);
    const long stat_at = ((long)b * H + h) * N + qrow;
    my_lse2 = LSE[stat_at] * kLog2e;
    if (!STATS) my_delta = delta[stat_at];
    staged_rows_landed();
    const StagedRows<D> q_at{q_rows, lane}, g_at{q_rows + kVOff, lane}, o_at{o_rows, lane};
#pragma unroll
    for (int kk = 0; kk < kKS; ++kk) {
      qf[kk] = q_at.wide(kk);
      gf[kk] = g_at.wide(kk);
    }
    staged_rows_read();
    if (STATS) {
      // partial sums combined in the order of fmha_bwd_delta_kernel's shuffle tree: the same bits
      float part[kKS];
#pragma unroll
      for (int kk = 0; kk < kKS; ++kk) {
        const h8 ov = o_at.wide(kk);
        part[kk] = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) part[kk] = fmaf((float)ov[e], (float)gf[kk][e], part[kk]);
      }
#pragma unroll
      for (int stride = kKS / 2; stride > 0; stride >>= 1)
#pragma unroll
        for (int kk = 0; kk < stride; ++kk) part[kk] += part[kk + stride];
      my_delta = part[0] + other_half(part[0]);
      if (hh == 0 && qi < N) {
        delta[stat_at] = my_delta;
        lse2[stat_at] = my_lse2;
      }
    }
#pragma unroll
    for (int kk = 0; kk < kKS; ++kk) {
      gf[kk] = -gf[kk];
      asm volatile("" : "+v"(gf[kk]));  // negated here, not in the loop
    }
  }

  int r_off[2], c_off[2];
  swz_rows_off<D>(lane, r_off);
  swz_cols_off<D>(lane, c_off);
  // fragment addresses: rows in the slot of the current tile, columns in that of the tile before it
  unsigned ra0 = opaque_lds_address(smem + r_off[0]), ra1 = opaque_lds_address(smem + r_off[1]);
  unsigned ca0 = opaque_lds_address(smem + c_off[0]), ca1 = opaque_lds_address(smem + c_off[1]);

  f16v dq[kDB], s[2], x[2], dl, zero;
  u4v p[4], y[4];  // probabilities and dS of a tile, fp16 pairs in B-operand order
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    dl[r] = my_delta;
    zero[r] = 0.f;
    x[0][r] = x[1][r] = 0.f;
#pragma unroll
    for (int db = 0; db < kDB; ++db) dq[db][r] = 0.f;
  }
#pragma unroll
  for (int c16 = 0; c16 < 4; ++c16) p[c16] = y[c16] = u4v{0, 0, 0, 0};

  constexpr int kLead = 3;
  auto ds_pair = [&](int n) __attribute__((always_inline)) {  // pair n of 16: two neighbouring keys
    const int c16 = n >> 2, e = (n & 3) * 2, rb = c16 >> 1, r = (c16 & 1) * 8 + e;
    y[c16][e >> 1] = neg_mul_to_f16x2(p[c16][e >> 1], x[rb][r], x[rb][r + 1]);
  };
  // dQ^T += K^T dS^T, MFMA n of 8
  auto dq_mfma = [&](h8 frag, int n) __attribute__((always_inline)) {
    dq[n % kDB] = mfma(frag, __builtin_bit_cast(h8, y[n / kDB]), dq[n % kDB]);
  };
  // Tile j in 24 units of one MFMA and what is issued in its shadow:
  //   0.. 7  S^T(j) = K(j) Q^T                     dS(j-1) = P o (dP - delta)
  //   8..15  delta - dP^T(j) = delta - V(j) dO^T   P(j) = exp2(S c - lse2), from unit 10 (S complete) to 23
  //  16..23  dQ^T += K(j-1)^T dS(j-1)^T
  // so that no vector instruction waits for an MFMA of its own tile just issued, nor the other way round.
  auto tile = [&](int j, auto masked_tag) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value != 0;
    h8 frag[kLead];
    const int last = (CAUSAL ? min(qi, N - 1) : N - 1) - j * kTile - 4 * hh;  // last key that counts
    auto p_pair = [&](int n) __attribute__((always_inline)) {
      const int c16 = n >> 2, e = (n & 3) * 2, rb = c16 >> 1, r = (c16 & 1) * 8 + e;
      float a0 = fmaf(s[rb][r], c, -my_lse2), a1 = fmaf(s[rb][r + 1], c, -my_lse2);
      if (MASKED) {
        if (acc_row(rb, r, 0) > last) a0 = -INFINITY;
        if (acc_row(rb, r + 1, 0) > last) a1 = -INFINITY;
      }
      p[c16][e >> 1] = pack_f16(fast_exp2(a0), fast_exp2(a1));
    };
    auto read = [&](int m) __attribute__((always_inline)) {
      const int n = m % 8;
      if (m < 8) return swz_rows_at<D>(ra0, ra1, n & 1, n >> 1);
      if (m < 16) return swz_rows_at<D>(ra0 + kVOff, ra1 + kVOff, n & 1, n >> 1);
      return swz_cols_at<D>(ca0, ca1, n / kDB, n % kDB);
    };
#pragma unroll
    for (int m = 0; m < kLead; ++m) frag[m] = read(m);
    __builtin_amdgcn_sched_barrier(0);
    static_for<24>([&](auto m_tag) __attribute__((always_inline)) {
      constexpr int m = decltype(m_tag)::value, n = m % 8;
      if constexpr (m < 8) s[n & 1] = mfma(frag[m % kLead], qf[n >> 1], n < 2 ? zero : s[n & 1]);
      else if constexpr (m < 16) x[n & 1] = mfma(frag[m % kLead], gf[n >> 1], n < 2 ? dl : x[n & 1]);
      else dq_mfma(frag[m % kLead], n);
      if constexpr (m + kLead < 24) frag[m % kLead] = read(m + kLead);
      if constexpr (m < 8) {
        ds_pair(2 * m);
        ds_pair(2 * m + 1);
      }
      if constexpr (m >= 10) {
        p_pair(m - 10);
        if constexpr (m >= 22) p_pair(m - 8);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  wait_vm<0>();  // resident rows and the first tile: no wait for a register load is left to be placed in the loop
  int slot = 0, next_slot = 1;
  auto top = [&](int j) __attribute__((always_inline)) {
    wait_vm<0>();
    block_barrier();
    if (j + 1 < nt) copy_tile(j + 1, next_slot);
  };
  auto next = [&](int j) __attribute__((always_inline)) {
    const int step = (next_slot - slot) * T::kBytes;
    ra0 += step, ra1 += step;
    if (j > 0) {
      const int cstep = (slot == 0 ? -(kSlots - 1) : 1) * T::kBytes;
      ca0 += cstep, ca1 += cstep;
    }
    slot = next_slot;
    next_slot = next_slot == kSlots - 1 ? 0 : next_slot + 1;
  };
  int j = 0;
  // Only the wave's last tile can need a mask, under which it is a third longer.  The mask goes on the exponent: on the
  // probabilities it keeps the compiler from converting two at a time.  Both: B16 H12 N512 26.9 -> 26.4 us (eight tiles a
  // block, none masked now), B4 H16 N1024 causal 21.1 -> 20.8 us; in the dK/dV pass 25.2 -> 24.9 us.
  const int plain = CAUSAL || N % kTile != 0 ? ntw - 1 : ntw;
  for (; j < plain; ++j) {
    top(j);
    tile(j, IntTag<0>{});
    next(j);
  }
  if (j < ntw) {
    top(j);
    tile(j, IntTag<1>{});
    next(j);
    ++j;
  }
  if (ntw > 0) {  // what is left of the wave's last tile
#pragma unroll
    for (int n = 0; n < 16; ++n) ds_pair(n);
#pragma unroll
    for (int n = 0; n < 8; ++n) dq_mfma(swz_cols_at<D>(ca0, ca1, n / kDB, n % kDB), n);
  }
  for (; j < nt; ++j) {
    top(j);
    next(j);
  }

  block_barrier();  // every wave is done with the rings: they become the staging tiles
  store_resident<D>(dQ + head_off, rs, q0w, N, dq, scale, lane, smem + wave * StageGeom<D>::kBytes);
}

template <bool CAUSAL, bool STATS, bool ODD_FIRST>
__global__ void __launch_bounds__(kPipeThreads, 2)
fmha_bwd_dq_pipe_kernel(const half_t* __restrict__ Q, const half_t* __restrict__ K, const half_t* __restrict__ V,
                        const half_t* __restrict__ O, const half_t* __restrict__ dO, Strides qs, Strides ks, Strides vs,
                        Strides gs, const float* __restrict__ LSE, float* __restrict__ delta, float* __restrict__ lse2,
                        half_t* __restrict__ dQ, FmhaDivisor H, int N, FmhaOrder order, int nmb, float c, float scale) {
  __shared__ __attribute__((aligned(1024))) char smem[kDqPipeLds];
  if (ODD_FIRST) odd_slots_first();
  int bh, mb;
  fmha_ordered_block(CAUSAL ? fmha_paired_block(blockIdx.x, gridDim.x) : blockIdx.x, order.slices, order.run, order.last_level,
                     CAUSAL, order.short_last, bh, mb);
  bwd_dq_pipe_block<CAUSAL, STATS>(Q, K, V, O, dO, qs, ks, vs, gs, LSE, delta, lse2, dQ, H, N, c, scale, smem, bh,
                                   CAUSAL ? nmb - 1 - mb : mb);  // heavy blocks first
}

// ---------------------------------------------------------------------------
// Backward, dK/dV pass.  Block = 128 keys = 4 pairs of waves; a pair owns 32
// keys and splits the work so that each wave keeps only one accumulator and one
// of K / V in registers (two waves per SIMD fit):
//   wave A (waves 0-3), tile j:   S = Q K^T, P = exp(S - lse) -> P(j) to LDS,
//                                 dV^T += dO^T P
//   wave B (waves 4-7), tile j:   dS(j-1) = P(j-1) o T(j-1),  dK^T += Q(j-1)^T dS(j-1),
//                                 then dP = dO(j) V^T, T(j) = dP - delta (kept in registers, as -T:
//                                 the GEMM runs on -V with accumulators loaded with delta)
// (formulas: reference kernel/fused_mha_kernel.cu:598-603, 618-629, 653-656,
// 697-712; key-block-parallel launch as at :908-915).  B runs one tile behind A
// for the part that needs P, so one barrier per tile is enough and neither wave
// waits for the other inside a tile.  P travels in the accumulator layout, lane
// for lane (double-buffered).  Q tiles of 64 queries stream through a 4-slot
// LDS ring (B still needs tile j-1), dO tiles and the tile's lse2/delta rows
// through 3-slot rings, all copied two tiles ahead.
// What bounds it: the MFMAs and LDS reads that the two waves of a SIMD share, and with all CUs busy the power cap, which
// is why those launches take the 16 x 16 x 32 MFMAs.  With them and the copies as they are placed now, against 32 x 32 ones, in
// turn: B2 H40 N2048 causal 211 -> 203 us; B2 H32 N4096 causal, dS stored: 597 -> 574 us, 958 TFLOP/s of its four products; B3
// H20 N1031: 98.7 -> 94.5 us.
// ---------------------------------------------------------------------------
constexpr int kKvPairs = 4;
constexpr int kKvWaves = 2 * kKvPairs;
constexpr int kKvThreads = kKvWaves * 64;
constexpr int kKvBlockKeys = kKvPairs * kResident;

//
// SPILL: wave B also writes every dS tile it forms (fp16, without the scale factor) to
// the workspace `dS`, for fmha_bwd_dq_spill_kernel, which then needs no S and dP of
// its own.  Layout per (batch, head) slice, np = n rounded up to 128:
//   [np / 128 query blocks][np / 64 key tiles] x 16 KiB, the tile a block of 128 queries
//   streams per 64 keys, made of 16 pieces of 1 KiB:
//   [2 halves of 32 keys][2 query tiles of 64][4 fragments] x 1 KiB.
// A 1 KiB piece is what one store instruction of wave B writes: each lane puts the 16 bytes of registers it holds, an
// operand fragment of the second GEMM, at 16 * lane (consecutive lanes, consecutive addresses).  WIDE: fragment f is
// queries 16 f .. of the 64, lane 32 * hh + i holds key i and as element e query 8 * (e >> 2) + 4 * hh + (e & 3).
// Otherwise fragment f is queries 32 (f >> 1) .. and keys 16 (f & 1) .., and lane 16 * g + i holds key i and as element e
// query 16 * (g >> 1) + 8 * (e >> 2) + 4 * (g & 1) + (e & 3).  Rows of keys at or past n are written as zeros; (key tile,
// query tile) pairs above the diagonal are not written (and not read) under causal masking.
// KEEP: without the non-temporal hint on those stores (rule: fmha_ds_used_once).
// WIDE: 32 x 32 x 16 MFMAs instead of 16 x 16 x 32 ones (same bits; rule and both times: fmha_wide_mfmas).
// STATS: the row statistics of every tile are formed here, from O, dO and LSE, a tile ahead; delta and lse2 are not read.
// SHARED: work groups of this launch read dS; stored counts the waves that have stored all of theirs, kKvPairs of every block
// (fmha_bwd_both_spill_kernel).
constexpr int kKvStBytes = 1024;
template <int D>
constexpr int dkdv_lds() { return 7 * SwzTile<D>::kBytes + 3 * kKvStBytes + 2 * kKvPairs * 2 * 2048; }
template <int D, bool CAUSAL, bool SPILL, bool KEEP, bool WIDE, bool STATS, bool SHARED = false>
__device__ __forceinline__ void
bwd_dkdv_block(const half_t* __restrict__ Q, const half_t* __restrict__ K, const half_t* __restrict__ V,
               const half_t* __restrict__ O, const half_t* __restrict__ dO, Strides qs, Strides ks, Strides vs, Strides gs,
               const float* __restrict__ LSE, const float* __restrict__ delta, const float* __restrict__ lse2,
               half_t* __restrict__ dK, half_t* __restrict__ dV, half_t* __restrict__ dS, int np, FmhaDivisor H, int N, int slice0,
               float c, float scale, char* smem, int bh, int nblk, unsigned* stored = nullptr) {
  using G = TileGeom<D>;
  using G16 = Geom16<D>;
  using T = SwzTile<D>;
  constexpr int kIPW = T::kInstrs / kKvWaves;  // copies per wave per tile, per tensor
  // Q ring (4), dO ring (3), per stats slot 64 lse2 then 64 delta values (1 KiB, half
  // unused), and the P exchange: 2 buffers x per pair the four fragments of P, 16 bytes per lane each, in separate 1 KiB
  // planes so that the accesses are free of bank conflicts.
  constexpr int kStBytes = kKvStBytes;
  constexpr int kPBytes = kKvPairs * 2 * 2048;
  static_assert(dkdv_lds<D>() == 7 * T::kBytes + 3 * kStBytes + 2 * kPBytes, "");
  char* const q_ring = smem;
  char* const g_ring = smem + 4 * T::kBytes;
  char* const st_ring = smem + 7 * T::kBytes;
  char* const p_xchg = st_ring + 3 * kStBytes;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pair = wave & (kKvPairs - 1);
  const bool role_b = wave >= kKvPairs;
  const int i = WIDE ? lane & 31 : lane & 15;        // resident position of this lane's columns, and
  const int g = WIDE ? lane >> 5 : lane >> 4;        // which streamed rows it has
  const int b = (slice0 + bh) / H, h = slice0 + bh - b * H;  // bh: the slice in this launch and in dS
  const int rs = H * D;  // dK and dV are dense
  const long head_off = ((long)b * N * H + h) * D;
  const half_t* Qb = Q + b * qs.b + (long)h * qs.h;
  const half_t* dOb = dO + b * gs.b + (long)h * gs.h;
  const float* delta_b = STATS ? nullptr : delta + ((long)b * H + h) * N;
  const float* lse2_b = STATS ? nullptr : lse2 + ((long)b * H + h) * N;

  const int n0 = nblk * kKvBlockKeys;
  // In a last block of at most 32 keys all four pairs own those: each takes one half of the rows of the even or of the odd
  // tiles, and their sums are put together at the end.  One pair alone took 23 us for such a block where four take 40 for a
  // whole one (N = 1031, dS stored), its two waves on one SIMD and the others idle; now 17 us.  dK/dV pass, us, before and after:
  // 1031 x 60 100.8, 88.0; x 32 63.5, 57.3; x 64 100.9, 93; 2053 x 60 295, 290; 4097 x 30 515, 504; 140 x 640 62.6, 60.5.  Two
  // pairs each for up to 64 keys gain nothing (1080 x 60 100.3, 99.2; x 32 63.9, 66.1).  The rule is one of N and the mask alone,
  // so the bits of a slice don't depend on the size of the call.  Under causal masking such a block has one tile.
  const bool shared = !CAUSAL && nblk > 0 && N - n0 <= kResident;
  const int group = shared ? 0 : pair;  // which 32 keys of the block
  const int k0w = n0 + group * kResident;

  const int nt = (N + kTile - 1) / kTile;
  const int t_begin = CAUSAL ? n0 / kTile : 0;
  const int n_it = nt - t_begin;  // >= 1

  // this wave's share of every tile copy
  // (its two copies of a tile as one, B2 H32 N4096 causal 590 -> 581 us, B2 H40 N2048 causal 201.6 -> 198.4; in the forward,
  // which forms fewer addresses per iteration, 1 % slower)
  static_assert(kIPW == 2 && T::kNC % 2 == 0, "a wave's copies of a tile are of the same 16 rows");
  constexpr int kBack = 960;  // see copy16_blocks
  int c_row, c_qgoff, c_ggoff;
  copy_src<D>(wave * kIPW, lane, qs.n, c_row, c_qgoff);
  copy_src<D>(wave * kIPW, lane, gs.n, c_row, c_ggoff);
  c_qgoff += kBack, c_ggoff += kBack;
  const unsigned lds_w = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem + wave * (kIPW * 1024);
  auto copy_tiles = [&](int it) __attribute__((always_inline)) {  // tile t_begin + it
    const int row0 = (t_begin + it) * kTile;
    const half_t* qp = Qb + (long)row0 * qs.n - kBack / 2;   // wave-uniform
    const half_t* gp = dOb + (long)row0 * gs.n - kBack / 2;
    const unsigned qdst = lds_w + (it & 3) * T::kBytes, gdst = lds_w + (4 + it % 3) * T::kBytes;
    if (row0 + kTile <= N) {
      copy16_blocks<kIPW>(qp, c_qgoff, qdst);
      copy16_blocks<kIPW>(gp, c_ggoff, gdst);
    } else {
      const int back = max(row0 + c_row - (N - 1), 0);  // rows past the end re-read row N-1
      copy16_blocks<kIPW>(qp, c_qgoff - back * qs.n * 2, qdst);
      copy16_blocks<kIPW>(gp, c_ggoff - back * gs.n * 2, gdst);
    }
    if (!STATS && wave == 0) {  // lane l: lse2 and delta of row row0 + l (rows past the end re-read row N-1)
      const int at = min(row0 + lane, N - 1) * 4;
      copy4(lse2_b, at, st_ring + (it % 3) * kStBytes);
      copy4(delta_b, at, st_ring + (it % 3) * kStBytes + 256);
    }
  };

  // resident rows of this wave: K for role A, V for role B; [feature step] of key k0w + i, or [feature step][cb] of keys
  // k0w + 16 cb + i.  They and the first tile are all that the loops need to start; the second tile is asked for when these
  // are there, not waited for with them.  What that gives, 0.2 to 0.8 % of B3 H20 N1031, B2 H40 N2048 causal and B2 H32 N4096
  // causal, is within what runs of one side differ by.
  static_assert(2 * kKvPairs * 4096 >= T::kBytes, "the rows of V of two pairs fit where P goes");
  h8 rf[G::kKSteps];
  // rows of K: slots 2 and 3 of Q; of V: slot 2 of dO and the buffers of P
  char* const my_rows = !role_b ? q_ring + 2 * T::kBytes + pair * (T::kBytes / 2)
                        : pair < 2 ? g_ring + 2 * T::kBytes + pair * (T::kBytes / 2) : p_xchg + (pair - 2) * (T::kBytes / 2);
  if (role_b) copy_rows<D>(V + b * vs.b + (long)h * vs.h, vs.n, k0w, N, lane, my_rows);
  else copy_rows<D>(K + b * ks.b + (long)h * ks.h, ks.n, k0w, N, lane, my_rows);
  copy_tiles(0);

  // statistics: the rows are asked for two tiles ahead, into registers, and summed up one tile ahead
  TileStats<D> stats(O + head_off, dOb, LSE + ((long)b * H + h) * N, rs, gs.n, t_begin);
  auto stats_ahead = [&](int it) __attribute__((always_inline)) {  // of tile it + 1; those of tile it + 2 are asked for
    if (it + 1 < n_it) stats.make(st_ring + (it + 1) % 3 * kStBytes);
    if (it + 2 < n_it) stats.load(N - 1 - (t_begin + it + 2) * kTile);
  };
  if (STATS) stats.load(N - 1 - t_begin * kTile);

  int r_off[2], c_off[2];
  if constexpr (WIDE) {
    swz_rows_off<D>(lane, r_off);
    swz_cols_off<D>(lane, c_off);
  } else {
    r_off[0] = rows16_off<D>(lane, 0);
    r_off[1] = rows16_off<D>(lane, 1);
  }
  // this role's statistics of the four rows at + 4 * stat_row(quad)
  const int st_off = (WIDE ? 4 * g : acc16_row(0, g)) * 4 + (role_b ? 256 : 0);
  constexpr auto stat_row = [](int quad) { return WIDE ? 8 * quad : 32 * (quad >> 1) + 8 * (quad & 1); };
  char* const p_mine = p_xchg + pair * 4096 + lane * 16;  // + buffer * kPBytes + 1024 * fragment

  // Products of 64 (or, sharing, 32) streamed rows and the 32 resident ones, and the accumulator of the second GEMM: dV^T
  // (role A) or dK^T (role B).  Either way 32 (16) registers of the one, in the order of the fragments of the second GEMM,
  // and 64 of the other.
  typedef typename std::conditional<WIDE, f16v[2], f4v[4][2]>::type Product;
  typedef typename std::conditional<WIDE, f16v[1], f4v[2][2]>::type HalfProduct;
  typename std::conditional<WIDE, f16v[G::kDBlocks], f4v[G16::kDB][2]>::type acc;
  auto clear = [](auto& x) __attribute__((always_inline)) {
    if constexpr (WIDE) {
#pragma unroll
      for (auto& v : x)
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] = 0.f;
    } else {
#pragma unroll
      for (auto& row : x) row[0] = row[1] = f4v{0.f, 0.f, 0.f, 0.f};
    }
  };
  // element e of 8 of fragment f of 4: 16 streamed rows f, or 32 streamed rows f >> 1 and resident block f & 1
  auto element = [](const auto& x, int f, int e) __attribute__((always_inline)) {
    if constexpr (WIDE) return x[f >> 1][(f & 1) * 8 + e];
    else return x[2 * (f >> 1) + (e >> 2)][f & 1][e & 3];
  };
  clear(acc);

  // Two waves of a SIMD that both have MFMAs ready do not take turns: one runs, the other waits, and which one is up to the
  // priorities.  The products that an iteration begins with go first: those that would be held up meet the next ones too.
  // That gained 5 % while role B copied before its second product (B2 H40 N2048 causal: 212 us without priorities, 201 with
  // these); since it copies later, it is B3 H20 N1031 alone that gains, on three cards 94.4 -> 94.0, 96.8 -> 94.9, 98.0 -> 95.2,
  // others lose up to 1.5 % (B2 H40 N2048 201.8, 202.0; 200.2, 201.6; 196.9, 198.2; B1 H12 N8192 without a mask 765, 777).
  // Kernels of another stream do not run any slower for it: half_round_left.  32 x 32 MFMAs: no difference.
  auto priority = [&](auto b_tag, auto a_tag) __attribute__((always_inline)) {
    if constexpr (!WIDE) {
      if (role_b) __builtin_amdgcn_s_setprio(decltype(b_tag)::value);
      else __builtin_amdgcn_s_setprio(decltype(a_tag)::value);
    }
  };
  // first GEMM of a tile: rows of Q (role A) or dO (role B) against the resident
  // rows, on top of what x holds
  // Both GEMMs read their LDS fragments kLead MFMAs ahead of their use, in an order that is written out and
  // pinned (see the forward: scheduling hints alone are dropped when registers get scarce).
  constexpr int kLead = 4, kUnits = 2 * G::kKSteps;  // units of one fragment of a whole tile; both GEMMs have as many
  static_assert(kUnits == 4 * G::kDBlocks, "");
  auto gemm1 = [&](const char* tile_lds, auto& x) __attribute__((always_inline)) {
    constexpr int kN = kUnits * sizeof(x) / sizeof(Product), kRB = kN / (WIDE ? G::kKSteps : G16::kKS);  // row blocks
    const unsigned a0 = opaque_lds_address(tile_lds + r_off[0]), a1 = opaque_lds_address(tile_lds + r_off[1]);
    // unit n: row block n % kRB and feature step n / kRB
    auto read = [&](int n) __attribute__((always_inline)) {
      if constexpr (WIDE) return swz_rows_at<D>(a0, a1, n % kRB, n / kRB);
      else return rows16_at<D>(a0, a1, n % kRB, n / kRB);
    };
    h8 frag[kLead];
#pragma unroll
    for (int n = 0; n < kLead; ++n) frag[n] = read(n);
    priority(IntTag<1>{}, IntTag<2>{});
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < kN; ++n) {
      if constexpr (WIDE) {
        x[n % kRB] = mfma(frag[n % kLead], rf[n / kRB], x[n % kRB]);
      } else {
        if (n % 2 == 0) wait_lds_pinned(n + 3 < kN ? 2 : n + 2 < kN ? 1 : 0);
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
          x[n % kRB][cb] = mfma16(frag[n % kLead], rf[2 * (n / kRB) + cb], x[n % kRB][cb]);
      }
      if (n + kLead < kN) frag[n % kLead] = read(n + kLead);
      __builtin_amdgcn_sched_barrier(0);
    }
    priority(IntTag<0>{}, IntTag<0>{});
  };
  // second GEMM: columns of dO (role A) or Q (role B) against the fp16 operand y
  auto gemm2 = [&](const char* tile_lds, const auto& y) __attribute__((always_inline)) {
    constexpr int kN = kUnits * sizeof(y) / sizeof(h8[4]);
    auto run = [&](auto read) __attribute__((always_inline)) {
      h8 frag[kLead];
#pragma unroll
      for (int n = 0; n < kLead; ++n) frag[n] = read(n);
      priority(IntTag<3>{}, IntTag<2>{});
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < kN; ++n) {
        if constexpr (WIDE) {
          constexpr int kDB = G::kDBlocks;
          acc[n % kDB] = mfma(frag[n % kLead], y[n / kDB], acc[n % kDB]);
        } else {
          constexpr int kDB = G16::kDB;
          if (n % 2 == 0) wait_lds_pinned(n + 3 < kN ? 4 : n + 2 < kN ? 2 : 0);
#pragma unroll
          for (int cb = 0; cb < 2; ++cb) acc[n % kDB][cb] = mfma16(frag[n % kLead], y[2 * (n / kDB) + cb], acc[n % kDB][cb]);
        }
        if (n + kLead < kN) frag[n % kLead] = read(n + kLead);
        __builtin_amdgcn_sched_barrier(0);
      }
      priority(IntTag<0>{}, IntTag<0>{});
    };
    // unit n: 16 streamed rows n / 4 and feature block n % 4, or 32 streamed rows n / 8 and feature block n % 8
    if constexpr (WIDE) {
      const unsigned a0 = opaque_lds_address(tile_lds + c_off[0]), a1 = opaque_lds_address(tile_lds + c_off[1]);
      run([&](int n) __attribute__((always_inline)) { return swz_cols_at<D>(a0, a1, n / G::kDBlocks, n % G::kDBlocks); });
    } else {
      const Cols16<D> cols(tile_lds, lane);
      run([&](int n) __attribute__((always_inline)) { return cols.at(0, n / G16::kDB, n % G16::kDB); });
    }
  };
  // P = exp2(S*c - lse2), fp16, in B-operand order.  MASKED tiles straddle the
  // diagonal or the end of the sequence.
  auto probabilities = [&](const auto& x, auto& y, const char* Sl, int q0, auto masked_tag) __attribute__((always_inline)) {
    constexpr bool MASKED = decltype(masked_tag)::value != 0;
    constexpr int kQuads = sizeof(x) / (WIDE ? 16 : 32);
    const int at = q0 + (WIDE ? 4 * g : acc16_row(0, g)), key = k0w + i;  // this lane's first query; its key (and the one 16 on)
#pragma unroll
    for (int quad = 0; quad < kQuads; ++quad) {
      const f4v l4 = *reinterpret_cast<const f4v*>(Sl + stat_row(quad) * 4);
#pragma unroll
      for (int cb = 0; cb < (WIDE ? 1 : 2); ++cb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int f = WIDE ? quad >> 1 : 2 * (quad >> 1) + cb, e = (quad & 1) * 4 + r;
          float p = fast_exp2(fmaf(element(x, f, e), c, -l4[r]));
          if (MASKED) {  // causal: queries key .. N - 1 count, one comparison: 200 x 48 13.6, 13.1 us; 2048 x 80 295, 292
            const int row = stat_row(quad) + r;
            if (CAUSAL ? (unsigned)(row - (key + 16 * cb - at)) >= (unsigned)max(N - key - 16 * cb, 0) : row >= N - at) p = 0.f;
          }
          y[f][e] = (half_t)p;
        }
    }
  };
  // a pair without keys has nothing to do, except for the zeros of dS it owes the last 64-key tile
  const bool has_keys = k0w < (SPILL ? (N + kTile - 1) / kTile * kTile : N);
  const int first_active = !has_keys ? n_it : CAUSAL ? k0w / kTile - t_begin : 0;
  auto tile_active = [&](int it) __attribute__((always_inline)) {
    return CAUSAL ? it >= first_active : has_keys && (!shared || (it & 1) == pair >> 1);
  };

  // Per iteration: wait for tile `it` (issued two iterations ago; the copies of tile
  // it+1 may still be in flight), one barrier, issue the copies of tile it+2.  Role A issues its half of them at the end
  // of the iteration and role B after the stores of dS: all at once right after the barrier they held every wave until the
  // copy path had taken them (32 x 32 MFMAs, B2 H32 N4096 causal: 608 us, role A at the end 591, role A after its first GEMM
  // 627; 16 x 16 ones, role B's places: below).
  auto step_wait = [&](int it) __attribute__((always_inline)) {
    if (!STATS && it + 1 < n_it) {
      if (wave == 0) wait_vm<2 * kIPW + 2>();
      else wait_vm<2 * kIPW>();
    } else {
      wait_vm<0>();
    }
    block_barrier();
    if (STATS) stats_ahead(it);
  };
  auto step_copy = [&](int it) __attribute__((always_inline)) {
    if (it + 2 < n_it) copy_tiles(it + 2);
  };
  // where this lane's registers of dS go (SPILL): its 16 bytes of fragment 0 of query tile 0 of
  // query block 0; per query tile t: + (t >> 1) * np * 128 + (t & 1) * 2048, per fragment + 512 (elements)
  half_t* const ds_lane = SPILL ? dS + ((long)bh * (np >> 7)) * np * 128 + (long)(k0w >> 6) * 8192 +
                                      ((k0w >> 5) & 1) * 4096 + lane * 8
                                : nullptr;
  if (STATS) stats_ahead(-1);
  staged_rows_landed();  // resident rows and the first tile: nothing is left for the compiler to wait on in the loops
  {
    const StagedRows<D> rows{my_rows, lane};
#pragma unroll
    for (int kk = 0; kk < G::kKSteps; ++kk) rf[kk] = WIDE ? rows.wide(kk) : rows.narrow(kk >> 1, kk & 1);
    staged_rows_read();
  }
  // Role B works with -V: its first GEMM then gives delta - dP on top of accumulators loaded with delta, with no
  // subtraction afterwards.
  const unsigned sign = role_b ? 0x80008000u : 0u;
#pragma unroll
  for (h8& r : rf) {
    r = __builtin_bit_cast(h8, __builtin_bit_cast(u4v, r) ^ u4v{sign, sign, sign, sign});
    asm volatile("" : "+v"(r));  // here, not in the loop
  }
  if (n_it > 1) copy_tiles(1);
  // half_tag: the pairs share their keys, and each works on 32 rows of a tile.
  auto run = [&](auto half_tag) __attribute__((always_inline)) {
    constexpr bool HALF = decltype(half_tag)::value != 0;
    constexpr int kFrags = HALF ? 2 : 4;
    typedef typename std::conditional<HALF, HalfProduct, Product>::type Rows;
    const int half = HALF ? pair & 1 : 0, rows_at = half * (T::kBytes / 2);
    if (!role_b) {
      for (int it = 0; it <= n_it; ++it) {
        step_wait(it);
        if (it < n_it && tile_active(it)) {
          const char* Ql = q_ring + (it & 3) * T::kBytes + rows_at;
          const char* Gl = g_ring + (it % 3) * T::kBytes + rows_at;
          const char* Sl = st_ring + (it % 3) * kStBytes + st_off + half * 128;
          const int q0 = (t_begin + it) * kTile + half * 32;
          const bool masked = (CAUSAL && q0 < k0w + kResident - 1) || (q0 + (HALF ? 32 : kTile) > N);
          Rows x;
          h8 y[kFrags];
          clear(x);
          gemm1(Ql, x);
          if (masked) probabilities(x, y, Sl, q0, IntTag<1>{});
          else probabilities(x, y, Sl, q0, IntTag<0>{});
          char* pw = p_mine + (it & 1) * kPBytes;
  #pragma unroll
          for (int f = 0; f < kFrags; ++f) *reinterpret_cast<h8*>(pw + f * 1024) = y[f];
          gemm2(Gl, y);
        }
        step_copy(it);
      }
    } else {
      Rows x;  // delta - dP of the previous tile
      clear(x);
      for (int it = 0; it <= n_it; ++it) {
        // After the second GEMM this wave issues the four stores of dS (SPILL) and then its copies of tile it + 2.  The wait
        // at the top of the next iteration leaves at most as many operations in flight as those copies, the newest:
        // every earlier copy has then landed, whatever order stores and copies complete in.  (Copies before the second GEMM,
        // where the wait is for them too: B2 H40 N2048 causal 198.6 us against 195.7, B2 H32 N4096 causal 566.7 against
        // 560.6, B3 H20 N1031 94.7 against 91.9.  After the GEMM and before the stores 200.1, 569.0, 91.9; at the end of the
        // iteration 201.7, 573.6, 95.0.)
        step_wait(it);
        const bool prev_active = it >= 1 && tile_active(it - 1);
        h8 y[kFrags];
        if (prev_active) {  // the part that needs P, one tile behind
          const char* pr = p_mine + ((it - 1) & 1) * kPBytes;
  #pragma unroll
          for (int f = 0; f < kFrags; ++f) {
            const h8 p = *reinterpret_cast<const h8*>(pr + f * 1024);
            float xr[8];
  #pragma unroll
            for (int e = 0; e < 8; ++e) xr[e] = element(x, f, e);
            y[f] = neg_mul_to_f16x8(p, xr);
          }
          if (SPILL && k0w + kResident > N) {  // keys past the end contribute nothing to dQ
  #pragma unroll
            for (int f = 0; f < kFrags; ++f)
              if (k0w + (WIDE ? 0 : 16 * (f & 1)) + i >= N) y[f] = h8{};
          }
        }
        if (prev_active) gemm2(q_ring + ((it - 1) & 3) * T::kBytes + rows_at, y);
        if (SPILL && prev_active) {
          // dS(it - 1) leaves here, between the two GEMMs, before the tile copies of role A, which come at the end of the
          // iteration: the stores go through the same path and would queue.
          const int t = t_begin + it - 1;  // the query tile
          half_t* dst = ds_lane + (long)(t >> 1) * np * 128 + (t & 1) * 2048 + half * 1024;
          static_for<kFrags>([&](auto f_tag) __attribute__((always_inline)) {
            constexpr int f = decltype(f_tag)::value, at = f * 1024;
            store_ds<SHARED, KEEP>(dst, y[f], IntTag<at>{});
          });
          if (HALF) {  // the zeros that the other 32 keys of the last 64-key tile owe
            static_for<kFrags>([&](auto f_tag) __attribute__((always_inline)) {
              constexpr int at = decltype(f_tag)::value * 1024;
              store_ds<SHARED, KEEP>(dst + 4096, h8{}, IntTag<at>{});
            });
          }
        }
        step_copy(it);
        if (it < n_it && tile_active(it)) {
          const char* Gl = g_ring + (it % 3) * T::kBytes + rows_at;
          const char* Sl = st_ring + (it % 3) * kStBytes + st_off + half * 128;
  #pragma unroll
          for (int quad = 0; quad < (int)sizeof(Rows) / (WIDE ? 16 : 32); ++quad) {
            const f4v d4 = *reinterpret_cast<const f4v*>(Sl + stat_row(quad) * 4);
            if constexpr (WIDE) {
  #pragma unroll
              for (int r = 0; r < 4; ++r) x[quad >> 2][4 * (quad & 3) + r] = d4[r];
            } else {
              x[quad][0] = x[quad][1] = d4;
            }
          }
          __builtin_amdgcn_sched_barrier(0);  // keep the delta loads out of the GEMM's read/MFMA pipeline
          gemm1(Gl, x);
        }
      }
    }
  };
  if (shared) run(IntTag<1>{});
  else run(IntTag<0>{});

  static_assert(kKvWaves * Stage16<D>::kBytes <= 7 * T::kBytes && kKvWaves * StageGeom<D>::kBytes <= 7 * T::kBytes,
                "the output staging tiles fit the rings");
  block_barrier();  // every wave is done with the rings: they become the staging tiles
  if (SHARED && role_b) {  // this wave's dS is where every work group of the launch can read it
    wait_vm<0>();
    if (lane == 0) __hip_atomic_fetch_add(stored, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (shared) {  // the sums of the four pairs, added in the order of the pairs by the first one
    constexpr int kSums = sizeof(acc) / 16, kBytes = kSums * 1024;  // per wave, 16 bytes of a lane at a time
    static_assert(2 * (kKvPairs - 1) * kBytes <= 7 * T::kBytes, "the sums of three pairs fit the rings");
    f4v* const sums = reinterpret_cast<f4v*>(&acc);
    char* const first = smem + (role_b ? kKvPairs - 1 : 0) * kBytes + lane * 16;  // + (pair - 1) * kBytes
    if (pair > 0) {
#pragma unroll
      for (int u = 0; u < kSums; ++u) *reinterpret_cast<f4v*>(first + (pair - 1) * kBytes + u * 1024) = sums[u];
    }
    block_barrier();
    if (pair == 0) {
      for (int other = 0; other < kKvPairs - 1; ++other) {
#pragma unroll
        for (int u = 0; u < kSums; ++u) {
          const f4v x = *reinterpret_cast<const f4v*>(first + other * kBytes + u * 1024);
#pragma unroll
          for (int r = 0; r < 4; ++r) sums[u][r] += x[r];
        }
      }
    }
    block_barrier();
    if (pair > 0) return;
  }
  half_t* const out = (role_b ? dK : dV) + head_off;
  const float mul = role_b ? scale : 1.f;
  if constexpr (WIDE) {
    store_resident<D>(out, rs, k0w, N, acc, mul, lane, smem + wave * StageGeom<D>::kBytes);
  } else {
    const float both[2] = {mul, mul};
    store_resident16<D>(out, rs, k0w, N, acc, both, lane, smem + wave * Stage16<D>::kBytes);
  }
}

template <int D, bool CAUSAL, bool SPILL, bool KEEP, bool WIDE>
__global__ void __launch_bounds__(kKvThreads, 1)
fmha_bwd_dkdv_kernel(const half_t* __restrict__ Q, const half_t* __restrict__ K, const half_t* __restrict__ V,
                     const half_t* __restrict__ dO, Strides qs, Strides ks, Strides vs, Strides gs,
                     const float* __restrict__ delta, const float* __restrict__ lse2,
                     half_t* __restrict__ dK, half_t* __restrict__ dV, half_t* __restrict__ dS, int np, FmhaDivisor H, int N,
                     FmhaOrder order, int slice0, float c, float scale) {
  __shared__ __attribute__((aligned(1024))) char smem[dkdv_lds<D>()];
  int bh, nblk;
  // causal: low key blocks are the heavy ones and come first
  fmha_ordered_block(blockIdx.x, order.slices, order.run, order.last_level, CAUSAL, order.short_last, bh, nblk);
  bwd_dkdv_block<D, CAUSAL, SPILL, KEEP, WIDE, false>(Q, K, V, nullptr, dO, qs, ks, vs, gs, nullptr, delta, lse2, dK, dV, dS, np,
                                                      H, N, slice0, c, scale, smem, bh, nblk);
}

// The dK/dV pass and the dQ pass that recomputes S and dP in one launch, for problems of so few blocks that neither fills the
// chip: dS is not stored.  STATS as in fmha_bwd_both_pipe_kernel.  The blocks are those of the kernels for either pass, and so
// are the results, bit for bit; the dQ pass over dS adds the same dS up in the same order and gives them too.  Rules and both
// sides: fmha_passes_at_once, fmha_blocks_make_stats.
static_assert(kDqBlockQ == kKvBlockKeys && kDqThreads == kKvThreads, "as many blocks of either pass, of the same size");
template <bool CAUSAL, bool STATS>
__global__ void __launch_bounds__(kKvThreads, 1)
fmha_bwd_both_kernel(const half_t* __restrict__ Q, const half_t* __restrict__ K, const half_t* __restrict__ V,
                     const half_t* __restrict__ O, const half_t* __restrict__ dO, Strides qs, Strides ks, Strides vs, Strides gs,
                     const float* __restrict__ LSE, float* __restrict__ delta, float* __restrict__ lse2, half_t* __restrict__ dQ,
                     half_t* __restrict__ dK, half_t* __restrict__ dV, FmhaDivisor H, int N, FmhaOrder order, int nb, float c,
                     float scale) {
  constexpr int D = 128;
  constexpr int kLds = dkdv_lds<D>() > dq_lds<D>() ? dkdv_lds<D>() : dq_lds<D>();
  __shared__ __attribute__((aligned(1024))) char smem[kLds];
  int bh, blk;
  bool dq;
  fmha_two_pass_ordered_block(blockIdx.x, order.slices, order.run, order.last_level, CAUSAL, order.short_last, bh, blk, dq);
  if (dq)
    bwd_dq_block<D, CAUSAL, STATS>(Q, K, V, O, dO, qs, ks, vs, gs, LSE, delta, lse2, dQ, H, N, c, scale, smem, bh,
                                   CAUSAL ? nb - 1 - blk : blk);
  else
    bwd_dkdv_block<D, CAUSAL, false, false, true, STATS>(Q, K, V, O, dO, qs, ks, vs, gs, LSE, delta, lse2, dK, dV, nullptr, 0, H,
                                                         N, 0, c, scale, smem, bh, blk);
}

// ---------------------------------------------------------------------------
// Backward, dK/dV pass for D = 64 (see fmha_bwd_dq_pipe_kernel).  Formulas and results are those of fmha_bwd_dkdv_kernel.
// A 64-query tile is worked on in two halves of 32 queries; the accumulation into dV and dK of a half runs during the
// next one, so Q and dO have three slots: the tile before, the current one, the one being copied.
// ---------------------------------------------------------------------------
// STATS: the row statistics of every tile are formed here, from O, dO and LSE, a tile ahead; delta and lse2 are not read.
constexpr int kDkDvPipeStBytes = 512;                     // 64 lse2 then 64 delta values
constexpr int kDkDvPipeLds = 3 * (2 * SwzTile<64>::kBytes + kDkDvPipeStBytes);
template <bool CAUSAL, bool STATS>
__device__ __forceinline__ void
bwd_dkdv_pipe_block(const half_t* __restrict__ Q, const half_t* __restrict__ K, const half_t* __restrict__ V,
                    const half_t* __restrict__ O, const half_t* __restrict__ dO, Strides qs, Strides ks, Strides vs, Strides gs,
                    const float* __restrict__ LSE, const float* __restrict__ delta, const float* __restrict__ lse2,
                    half_t* __restrict__ dK, half_t* __restrict__ dV, FmhaDivisor H, int N, float c, float scale, char* smem, int bh,
                    int nblk) {
  constexpr int D = 64;
  using G = TileGeom<D>;
  using T = SwzTile<D>;
  constexpr int kDB = G::kDBlocks, kKS = G::kKSteps;
  constexpr int kIPW = T::kInstrs / kPipeWaves;
  constexpr int kSlots = 3;                               // the current tile, the one before it, the one being copied
  constexpr int kGOff = kSlots * T::kBytes, kStOff = 2 * kSlots * T::kBytes;
  constexpr int kStBytes = kDkDvPipeStBytes;
  static_assert(kDkDvPipeLds == kStOff + kSlots * kStBytes, "");
  static_assert(kPipeWaves * StageGeom<D>::kBytes <= kStOff, "the output staging tiles fit the rings");

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 31, hh = lane >> 5;
  const int b = bh / H, h = bh - b * H;
  const int rs = H * D;                                   // dK and dV are dense
  const long head_off = ((long)b * N * H + h) * D;
  const int n0 = nblk * kPipeBlockKeys;
  const int k0w = n0 + wave * kResident, ki = k0w + i;

  const int nt = (N + kTile - 1) / kTile;
  const int t_begin = CAUSAL ? n0 / kTile : 0;
  // tiles this wave works on: from the one with the first query that sees a key of it
  const int t_active = k0w < N ? (CAUSAL ? k0w / kTile : 0) : nt;

  // tile copies as in fmha_fwd_pipe_kernel
  constexpr int kBack = 960 * (kIPW - 1);
  int q_goff, g_goff, c_past;
  {
    const int row = 16 * wave + (lane >> 2), col = ((lane & 3) ^ swz(lane >> 4)) * 16;
    q_goff = row * qs.n * 2 + col + kBack;
    g_goff = row * gs.n * 2 + col + kBack;
    c_past = max((nt - 1) * kTile + row - (N - 1), 0) * 2;
  }
  const half_t* qp = Q + b * qs.b + (long)h * qs.h + (long)t_begin * kTile * qs.n - kBack / 2;  // next tile to copy
  const half_t* gp = dO + b * gs.b + (long)h * gs.h + (long)t_begin * kTile * gs.n - kBack / 2;
  const float* const stat = STATS ? nullptr : (wave == 0 ? lse2 : delta) + ((long)b * H + h) * N;
  const unsigned lds_w = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)smem + wave * (kIPW * 1024);
  auto copy_tile = [&](int t, int slot) __attribute__((always_inline)) {
    if (t == nt - 1) {
      q_goff -= c_past * qs.n;
      g_goff -= c_past * gs.n;
    }
    copy16_blocks<kIPW>(qp, q_goff, lds_w + slot * T::kBytes);
    copy16_blocks<kIPW>(gp, g_goff, lds_w + kGOff + slot * T::kBytes);
    qp += (long)kTile * qs.n;
    gp += (long)kTile * gs.n;
    if (!STATS && wave < 2) copy4(stat, min(t * kTile + lane, N - 1) * 4, smem + kStOff + slot * kStBytes + wave * 256);
  };
  char* const k_rows = smem + T::kBytes + wave * (T::kBytes / 2);  // through slots 1 and 2 of the rings; of V: + kGOff
  copy_rows<D>(K + b * ks.b + (long)h * ks.h, ks.n, k0w, N, lane, k_rows);
  copy_rows<D>(V + b * vs.b + (long)h * vs.h, vs.n, k0w, N, lane, k_rows + kGOff);
  copy_tile(t_begin, 0);

  // statistics: the rows are asked for two tiles ahead, into registers, and summed up one tile ahead
  TileStats<D> stats(O + head_off, dO + b * gs.b + (long)h * gs.h, LSE + ((long)b * H + h) * N, rs, gs.n, t_begin);
  auto load_stats = [&](int t) __attribute__((always_inline)) { stats.load(N - 1 - t * kTile); };
  auto make_stats = [&](int slot) __attribute__((always_inline)) { stats.make(smem + kStOff + slot * kStBytes); };
  if (STATS) load_stats(t_begin);

  // resident rows: K, and V negated, so that the dP product on top of delta gives delta - dP
  h8 kf[kKS], vf[kKS];
  {
    staged_rows_landed();
    const StagedRows<D> k_at{k_rows, lane}, v_at{k_rows + kGOff, lane};
#pragma unroll
    for (int kk = 0; kk < kKS; ++kk) {
      kf[kk] = k_at.wide(kk);
      vf[kk] = v_at.wide(kk);
    }
    staged_rows_read();
#pragma unroll
    for (int kk = 0; kk < kKS; ++kk) {
      vf[kk] = -vf[kk];
      asm volatile("" : "+v"(vf[kk]));  // negated here, not in the loop
    }
  }

  int r_off[2], c_off[2];
  swz_rows_off<D>(lane, r_off);
  swz_cols_off<D>(lane, c_off);
  // fragment addresses in the slot of the current tile, and of columns in that of the tile before it
  unsigned ra0 = opaque_lds_address(smem + r_off[0]), ra1 = opaque_lds_address(smem + r_off[1]);
  unsigned ca0 = opaque_lds_address(smem + c_off[0]), ca1 = opaque_lds_address(smem + c_off[1]);
  unsigned pa0 = ca0, pa1 = ca1;
  unsigned st0 = opaque_lds_address(smem + kStOff + hh * 16);

  f16v dv[kDB], dk[kDB], s, x[2], zero;
  u4v p[2], y[2];  // [16 queries]: probabilities and dS, fp16 pairs in B-operand order
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    zero[r] = x[0][r] = x[1][r] = 0.f;
#pragma unroll
    for (int db = 0; db < kDB; ++db) dv[db][r] = dk[db][r] = 0.f;
  }
#pragma unroll
  for (int cc = 0; cc < 2; ++cc) p[cc] = y[cc] = u4v{0, 0, 0, 0};

  auto ds_pair = [&](int n, const f16v& xx) __attribute__((always_inline)) {  // pair n of 8: two neighbouring queries
    const int cc = n >> 2, e = (n & 3) * 2, r = cc * 8 + e;
    y[cc][e >> 1] = neg_mul_to_f16x2(p[cc][e >> 1], xx[r], xx[r + 1]);
  };
  auto dv_mfma = [&](h8 frag, int n) __attribute__((always_inline)) {
    dv[n % kDB] = mfma(frag, __builtin_bit_cast(h8, p[n / kDB]), dv[n % kDB]);
  };
  auto dk_mfma = [&](h8 frag, int n) __attribute__((always_inline)) {
    dk[n % kDB] = mfma(frag, __builtin_bit_cast(h8, y[n / kDB]), dk[n % kDB]);
  };
  // columns of the half before the one with rows 32 hq .. of the current tile
  auto cols_before = [&](int hq, unsigned at, int n) __attribute__((always_inline)) {
    return hq == 0 ? swz_cols_at<D>(pa0 + at, pa1 + at, 2 + n / kDB, n % kDB)
                   : swz_cols_at<D>(ca0 + at, ca1 + at, n / kDB, n % kDB);
  };

  constexpr int kLead = 4;
  // Half a tile (32 queries, rows 32 hq ..) in 16 units of one MFMA and what is issued in its shadow:
  //   0.. 7  S = Q K^T and delta - dP = delta - dO V^T in turn      dS = P o (dP - delta) of the half before
  //   8..11  dV^T += dO^T P of the half before                      P = exp2(S c - lse2), from unit 10
  //  12..15  dK^T += Q^T dS of the half before
  auto half = [&](int t, auto hq_tag, auto masked_tag) __attribute__((always_inline)) {
    constexpr int hq = decltype(hq_tag)::value;
    constexpr bool MASKED = decltype(masked_tag)::value != 0;
    typedef __attribute__((address_space(3))) f4v lds_f4;
    h8 frag[kLead];
    const int first_q = ki - t * kTile - 4 * hh, end_q = N - t * kTile - 4 * hh;  // queries that count, as acc_row(hq, r, 0)
    // Causal: how many count, from the first on, so a mask is one comparison and not two and a merge, in the shadow of the
    // MFMAs, which masked tiles (the diagonal, the last) outgrow.  us before and with it: 77 x 8 6.60, 6.19; 300 x 80 12.4, 11.9;
    // 777 x 36 22.0, 21.6; 1024 x 64 42.1, 42.2
    const unsigned seen = max(N - ki, 0);
    f16v dl;
    f4v ls[4];
    auto read = [&](int m) __attribute__((always_inline)) {
      if (m < 8) return swz_rows_at<D>(ra0 + (m & 1) * kGOff, ra1 + (m & 1) * kGOff, hq, m >> 1);
      if (m < 12) return cols_before(hq, kGOff, m - 8);
      return cols_before(hq, 0, m - 12);
    };
    auto p_pair = [&](int n) __attribute__((always_inline)) {
      const int cc = n >> 2, e = (n & 3) * 2, r = cc * 8 + e;
      float a0 = fmaf(s[r], c, -ls[r >> 2][r & 3]), a1 = fmaf(s[r + 1], c, -ls[r >> 2][(r & 3) + 1]);
      if (MASKED) {
        const int q = acc_row(hq, r, 0);
        if (CAUSAL ? (unsigned)(q - first_q) >= seen : q >= end_q) a0 = -INFINITY;
        if (CAUSAL ? (unsigned)(q + 1 - first_q) >= seen : q + 1 >= end_q) a1 = -INFINITY;
      }
      p[cc][e >> 1] = pack_f16(fast_exp2(a0), fast_exp2(a1));
    };
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f4v d4 = *(const lds_f4*)(uintptr_t)(st0 + 256 + hq * 128 + 32 * g);
#pragma unroll
      for (int e = 0; e < 4; ++e) dl[4 * g + e] = d4[e];
    }
#pragma unroll
    for (int m = 0; m < kLead; ++m) frag[m] = read(m);
    __builtin_amdgcn_sched_barrier(0);
    static_for<16>([&](auto m_tag) __attribute__((always_inline)) {
      constexpr int m = decltype(m_tag)::value;
      if constexpr (m < 8) {
        if constexpr (m % 2 == 0) s = mfma(frag[m % kLead], kf[m / 2], m == 0 ? zero : s);
        else x[hq] = mfma(frag[m % kLead], vf[m / 2], m == 1 ? dl : x[hq]);
      } else if constexpr (m < 12) {
        dv_mfma(frag[m % kLead], m - 8);
      } else {
        dk_mfma(frag[m % kLead], m - 12);
      }
      if constexpr (m + kLead < 16) frag[m % kLead] = read(m + kLead);
      if constexpr (m < 8) {
        ds_pair(m, x[hq ^ 1]);
        if constexpr (m % 2 == 0) ls[m / 2] = *(const lds_f4*)(uintptr_t)(st0 + hq * 128 + 16 * m);
      }
      // P of queries 0..15 after the last reader of the half before's (unit 9), of queries 16..31 after unit 11
      if constexpr (m == 10 || m == 11) p_pair(m - 10);
      if constexpr (m == 12 || m == 13) {
        p_pair(2 * m - 22);
        p_pair(2 * m - 21);
      }
      if constexpr (m >= 14) p_pair(m - 8);
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  if (STATS) {
    make_stats(0);
    if (t_begin + 1 < nt) load_stats(t_begin + 1);
  }
  wait_vm<0>();
  int slot = 0, next_slot = 1, t = t_begin;
  auto top = [&]() __attribute__((always_inline)) {
    wait_vm<0>();
    block_barrier();
    if (t + 1 < nt) {
      copy_tile(t + 1, next_slot);
      if (STATS) {
        make_stats(next_slot);
        if (t + 2 < nt) load_stats(t + 2);
      }
    }
  };
  auto next = [&]() __attribute__((always_inline)) {
    const int step = next_slot - slot;
    if (t >= t_active) pa0 = ca0, pa1 = ca1;
    ra0 += step * T::kBytes, ra1 += step * T::kBytes, ca0 += step * T::kBytes, ca1 += step * T::kBytes;
    if (t < t_active) pa0 = ca0, pa1 = ca1;  // the first tile worked on: P and dS before it are zero, any rows will do
    st0 += step * kStBytes;
    slot = next_slot;
    next_slot = next_slot == kSlots - 1 ? 0 : next_slot + 1;
    ++t;
  };
  // The wave's tiles in order: not seen by its keys (copies only), then spans of masked tiles (on the diagonal, at the
  // end of the sequence) and of unmasked ones, each in a loop of its own so that no accumulator crosses a branch.
  const int t_diag = CAUSAL ? t_active + 1 : 0;  // first tile below the diagonal
  const int nt_full = N / kTile;                 // tiles without rows past the end
  while (t < min(t_active, nt)) {
    top();
    next();
  }
  while (t < nt) {
    while (t < nt && (t < t_diag || t >= nt_full)) {
      top();
      half(t, IntTag<0>{}, IntTag<1>{});
      half(t, IntTag<1>{}, IntTag<1>{});
      next();
    }
    while (t >= t_diag && t < nt_full) {
      top();
      half(t, IntTag<0>{}, IntTag<0>{});
      half(t, IntTag<1>{}, IntTag<0>{});
      next();
    }
  }
  if (t_active < nt) {  // what is left of the last half
#pragma unroll
    for (int n = 0; n < 8; ++n) ds_pair(n, x[1]);
#pragma unroll
    for (int n = 0; n < 4; ++n) dv_mfma(cols_before(0, kGOff, n), n);
#pragma unroll
    for (int n = 0; n < 4; ++n) dk_mfma(cols_before(0, 0, n), n);
  }

  block_barrier();  // every wave is done with the rings: they become the staging tiles
  char* const stage = smem + wave * StageGeom<D>::kBytes;
  store_resident<D>(dV + head_off, rs, k0w, N, dv, 1.f, lane, stage);
  store_resident<D>(dK + head_off, rs, k0w, N, dk, scale, lane, stage);
}

template <bool CAUSAL, bool ODD_FIRST>
__global__ void __launch_bounds__(kPipeThreads, 2)
fmha_bwd_dkdv_pipe_kernel(const half_t* __restrict__ Q, const half_t* __restrict__ K, const half_t* __restrict__ V,
                          const half_t* __restrict__ dO, Strides qs, Strides ks, Strides vs, Strides gs,
                          const float* __restrict__ delta, const float* __restrict__ lse2, half_t* __restrict__ dK,
                          half_t* __restrict__ dV, FmhaDivisor H, int N, FmhaOrder order, float c, float scale) {
  __shared__ __attribute__((aligned(1024))) char smem[kDkDvPipeLds];
  if (ODD_FIRST) odd_slots_first();
  int bh, nblk;  // causal: low key blocks are the heavy ones and come first
  fmha_ordered_block(CAUSAL ? fmha_paired_block(blockIdx.x, gridDim.x) : blockIdx.x, order.slices, order.run, order.last_level,
                     CAUSAL, order.short_last, bh, nblk);
  bwd_dkdv_pipe_block<CAUSAL, false>(Q, K, V, nullptr, dO, qs, ks, vs, gs, nullptr, delta, lse2, dK, dV, H, N, c, scale, smem,
                                     bh, nblk);
}

// Both passes in one launch: neither waits for the other, and a launch that leaves places empty (two blocks to a CU), or whose
// last round does, takes the blocks of the other pass along.  STATS: every block makes the row statistics it needs, otherwise
// they come from fmha_bwd_delta_kernel.  The blocks are those of the two kernels above, and so are the results, bit for bit.
// Rules and both sides: fmha_passes_at_once, fmha_blocks_make_stats.
static_assert(kPipeBlockQ == kPipeBlockKeys, "as many blocks of either pass");
template <bool CAUSAL, bool STATS>
__global__ void __launch_bounds__(kPipeThreads, 2)
fmha_bwd_both_pipe_kernel(const half_t* __restrict__ Q, const half_t* __restrict__ K, const half_t* __restrict__ V,
                          const half_t* __restrict__ O, const half_t* __restrict__ dO, Strides qs, Strides ks, Strides vs,
                          Strides gs, const float* __restrict__ LSE, float* __restrict__ delta, float* __restrict__ lse2,
                          half_t* __restrict__ dQ, half_t* __restrict__ dK, half_t* __restrict__ dV, FmhaDivisor H, int N,
                          FmhaOrder order, int nb, float c, float scale) {
  constexpr int kLds = kDkDvPipeLds > kDqPipeLds ? kDkDvPipeLds : kDqPipeLds;
  __shared__ __attribute__((aligned(1024))) char smem[kLds];
  int bh, blk;
  bool dq;
  fmha_two_pass_ordered_block(CAUSAL ? fmha_paired_block(blockIdx.x, gridDim.x) : blockIdx.x, order.slices, order.run,
                              order.last_level, CAUSAL, order.short_last, bh, blk, dq);
  if (dq)
    bwd_dq_pipe_block<CAUSAL, STATS>(Q, K, V, O, dO, qs, ks, vs, gs, LSE, delta, lse2, dQ, H, N, c, scale, smem, bh,
                                    CAUSAL ? nb - 1 - blk : blk);
  else
    bwd_dkdv_pipe_block<CAUSAL, STATS>(Q, K, V, O, dO, qs, ks, vs, gs, LSE, delta, lse2, dK, dV, H, N, c, scale, smem, bh, blk);
}

// ---------------------------------------------------------------------------
// Backward, dQ from spilled dS: dQ = scale * dS K, one GEMM, for callers whose
// workspace holds the dS tiles fmha_bwd_dkdv_kernel<.., SPILL> wrote (layout there).
// A block is P = 1 or 2 of the 128-query panels of the workspace; computing wave
// w of 4 P owns its 32 queries and computes per 64 keys
//     dQ^T[d][q] += K^T[d][key] dS^T[key][q]
// with both operands read transposed out of LDS (the K tile as everywhere else, the
// dS tile as its 1 KiB pieces), so the order of the keys inside a 16-key step is the
// same for both.
// What bounds the kernel is the path that copies tiles into LDS (64 bytes per clock and
// CU at best), then HBM (dS is read once):
//   * with P = 2 a K tile serves 256 queries, so per 32 KiB of dS only 16 KiB of K go through it (P = 1 is
//     for launches with too few blocks to balance otherwise);
//   * four more waves do nothing but copy, two the dS tiles (half of the pieces each) and two the
//     K tiles: issuing a tile's copy instructions holds a wave for about as long as its
//     share of the MFMAs takes; and a wave's copies complete in order, so a wave that
//     issued both kinds would wait for young dS copies whenever it needs an older K tile;
//   * the launch is persistent (PersistentBlocks) and the tiles of a work group's blocks
//     form ONE sequence that runs through the rings without regard to block boundaries;
//     an output block leaves through staging tiles of its own while the copies of the
//     next blocks' tiles are already in flight.  Both rings are filled two tiles ahead: behind the dS copies
//     that a CU has in flight, a K tile takes as long to arrive as they do, L2 hit or not;
//   * the LDS is full with that, so the epilogue stages a wave's output rows in the 4 KiB of the block's last dS
//     tile that hold the wave's own queries and that no other wave reads.
// The queries of a fragment sit in the order the dK/dV pass's registers held them; the epilogue puts the rows back in
// place.  WIDE as in that pass.  The 16 x 16 MFMAs take less of the power that the copies also need (B2 H40 N2048 causal:
// 97 -> 88 us, B2 H32 N4096 causal 242 -> 229 us); more copying waves, deeper rings or K fragments read further ahead
// change nothing.
// (formula: reference kernel/fused_mha_kernel.cu:680-683.)
// ---------------------------------------------------------------------------
constexpr int kDsCopyWaves = 4;    // waves that only copy tiles: two for dS, two for K
constexpr int kDsPanelQ = 128;     // queries per panel of the workspace
constexpr int kDsRingS = 3;   // dS tiles
constexpr int kDsRingK = 3;   // K tiles
constexpr int kDsPanelTileBytes = kTile * kDsPanelQ * 2;
constexpr int kDsStageD = 32;          // features staged at a time in the epilogue
constexpr int ds_threads(int panels) { return (4 * panels + kDsCopyWaves) * 64; }

// A pointer that is the same in all lanes, in scalar registers.
__device__ __forceinline__ const half_t* wave_uniform(const half_t* p) {
  const uint64_t a = (uint64_t)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((int)(unsigned)a), hi = __builtin_amdgcn_readfirstlane((int)(a >> 32));
  return (const half_t*)((uint64_t)hi << 32 | lo);
}

// The blocks of a launch of this pass alone.  With one block per work group the hardware shares them out, otherwise the
// persistent schedule does.
template <bool CAUSAL>
struct DsBlocks {
  static constexpr bool kShared = false;  // a launch before this one has stored dS
  const FmhaOrder& order;
  int total;
  __device__ __forceinline__ int next_round(int r) const { return PersistentBlocks{total}.next_round(r); }
  __device__ __forceinline__ void locate(int round, int& bh, int& mb) const {
    const int lin = round >= 0 ? PersistentBlocks{total}.lin(round) : 0;
    if ((int)gridDim.x == total) fmha_ordered_block(lin, order.slices, order.run, order.last_level, CAUSAL, false, bh, mb);
    else fmha_slice_and_block(lin, order.slices, order.run, bh, mb);
  }
};
// One block that is known already.
struct DsBlock {
  static constexpr bool kShared = true;
  int bh, mb;
  __device__ __forceinline__ int next_round(int) const { return -1; }
  __device__ __forceinline__ void locate(int, int& bh_, int& mb_) const { bh_ = bh, mb_ = mb; }
};

template <int D, int kDsPanels>
constexpr int ds_lds() { return kDsRingS * kDsPanels * kDsPanelTileBytes + kDsRingK * SwzTile<D>::kBytes; }
template <int D, bool CAUSAL, int kDsPanels, bool WIDE, typename Blocks>
__device__ __forceinline__ void
bwd_dq_spill_blocks(const half_t* __restrict__ K, Strides ks, const half_t* __restrict__ dS, int np,
                    half_t* __restrict__ dQ, FmhaDivisor H, int N, int nqb, int slice0, int stream_ds, float scale, char* smem,
                    const Blocks blocks) {
  using T = SwzTile<D>;             // K tile: 64 keys x D features
  constexpr int kKIPW = T::kInstrs / 2;              // K copies per K-copying wave and tile
  constexpr int kDsWaves = 4 * kDsPanels;            // computing waves
  constexpr int kDsBlockQ = kDsPanels * kDsPanelQ;
  constexpr int kDsTileBytes = kDsPanels * kDsPanelTileBytes;
  constexpr int kSIPW = kDsTileBytes / 1024 / 2;     // dS copies per dS-copying wave and tile: half of the pieces
  static_assert(16 * StageGeom<kDsStageD>::kPitch <= 2048 && 16 * Stage16<kDsStageD>::kPitch <= 2048,
                "half a staging tile must fit into two dS pieces");
  static_assert(ds_lds<D, kDsPanels>() == kDsRingS * kDsTileBytes + kDsRingK * T::kBytes, "");
  char* const s_ring = smem;
  char* const k_ring = smem + kDsRingS * kDsTileBytes;

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool computes = wave < kDsWaves;             // then two waves that copy dS and two that copy K
  const int qb = wave & (kDsWaves - 1);              // computing wave: its 32 queries of the block
  const bool copies_k = wave >= kDsWaves + 2;
  const int cw = wave & 1;                           // copying wave: which half of its tensor's copies
  const int rs = H * D;  // dQ is dense
  const int nt_all = (N + kTile - 1) / kTile;
  const int n_panels = np / kDsPanelQ;

  // A position in the work group's sequence of tiles: block (round, number), tile j of its nt.
  struct Cursor {
    int round, j, nt, mblk;
    const half_t* base;  // dS copies: this wave's pieces of the block's tile 0; K copies: the slice's K rows
    long out_off;        // consumer: element offset of the slice in dQ
  };
  auto open = [&](int round, bool for_k) __attribute__((always_inline)) {
    Cursor c;
    c.round = round;
    int bh, mb;
    blocks.locate(round, bh, mb);
    c.mblk = CAUSAL ? nqb - 1 - mb : mb;  // heavy blocks first
    const int b = (slice0 + bh) / H, h = slice0 + bh - b * H;  // bh: the slice in this launch and in dS
    c.j = 0;
    c.nt = CAUSAL ? min(nt_all, 2 * kDsPanels * (c.mblk + 1)) : nt_all;
    // the pieces of a dS-copying wave: with two panels per block one whole panel (the last block of a sequence
    // may have one panel only: the second wave then re-reads the first), else one half of the panel
    const int panel = kDsPanels == 2 ? min(2 * c.mblk + cw, n_panels - 1) : c.mblk;
    const int first_piece = kDsPanels == 2 ? 0 : cw * kSIPW;
    c.base = for_k ? K + b * ks.b + (long)h * ks.h
                   : dS + (((long)bh * n_panels + panel) * np) * kDsPanelQ + first_piece * 512;
    c.out_off = ((long)b * N * H + h) * D;
    return c;
  };
  auto advance = [&](Cursor& c, bool for_k) __attribute__((always_inline)) {  // to the next tile of the sequence
    if (++c.j == c.nt) {
      const int r = blocks.next_round(c.round);
      if (r >= 0) c = open(r, for_k);
      else c.round = -1;  // past the end
    }
  };
  int n_tiles = 0;  // tiles in this work group's sequence
  for (int r = 0; r >= 0; r = blocks.next_round(r)) {
    int bh, mb;
    blocks.locate(r, bh, mb);
    const int mblk = CAUSAL ? nqb - 1 - mb : mb;
    n_tiles += CAUSAL ? min(nt_all, 2 * kDsPanels * (mblk + 1)) : nt_all;
  }

  // K copies: this wave's half of a tile (as in the other kernels).  dS copies: this wave's kSIPW pieces of
  // 1 KiB, lane l fetching 16 bytes, in an order in which the 32 lanes of a transposing read fall on different banks.
  // WIDE: in memory a piece is [2 halves][32 keys] x 16 bytes; in LDS it becomes [32 keys][2 halves] x 16 bytes (rows of 16
  // queries), and the pieces of odd query chunks land rotated by 128 bytes (LDS offset o holds row-major byte (o - 128) mod
  // 1024).  Otherwise a piece is [4 lane groups j][16 keys] x 16 bytes, and in LDS the keys of odd j are 8 further (modulo 16).
  int c_row[kKIPW], c_kgoff[kKIPW], c_kblk[kKIPW];
#pragma unroll
  for (int u = 0; u < kKIPW; ++u) {
    const int t = cw * kKIPW + u;
    copy_src<D>(t, lane, ks.n, c_row[u], c_kgoff[u]);
    c_kblk[u] = t * 1024;
  }
  int c_sgoff[2];  // even and odd pieces; + piece * 1024
  if constexpr (WIDE) {
    const int at = (lane - 8) & 63;  // position (key, half) = (at >> 1, at & 1) in LDS of what lane l fetches of an odd piece
    c_sgoff[0] = ((lane & 1) * 32 + (lane >> 1)) * 16;
    c_sgoff[1] = ((at & 1) * 32 + (at >> 1)) * 16;
  } else {
    c_sgoff[0] = c_sgoff[1] = (lane ^ ((lane >> 4 & 1) * 8)) * 16;
  }
  auto copy_s = [&](const Cursor& c, int slot) __attribute__((always_inline)) {
    // Pieces that no query needs, above the diagonal or past the end, are copies of others of the same tile (or of the
    // last tile that has any): they then come from the L2, and the number of copies in flight stays what the waits count
    // on.  H256 N512 causal 30.9 -> 27.4 us, B2 H40 N2048 causal 87.8 -> 85.4, B2 H32 N4096 causal 228.5 -> 223.8, B3 H20
    // N1031 39.8 -> 38.8.
    const int panel = kDsPanels == 2 ? min(2 * c.mblk + cw, n_panels - 1) : c.mblk;
    const int j = CAUSAL ? min(c.j, 2 * panel + 1) : c.j;
    const int g_first = CAUSAL && j == 2 * panel + 1 ? 2 : 0, g_last = (N - 1) / kResident - 4 * panel;  // groups of 32 queries
    const half_t* sp[4];  // where the pieces of group g come from, less their place in the tile
#pragma unroll
    for (int g = 0; g < 4; ++g)
      sp[g] = wave_uniform(c.base + (long)j * (kDsPanelTileBytes / 2) + (max(min(g, g_last), g_first) - g) * 1024);
    char* dst = s_ring + slot * kDsTileBytes + cw * kSIPW * 1024;
    if (stream_ds) {
#pragma unroll
      for (int u = 0; u < kSIPW; ++u)
        copy16_ds<Blocks::kShared, true>(sp[(u >> 1) & 3], c_sgoff[u & 1] + u * 1024, dst + u * 1024);
    } else {
#pragma unroll
      for (int u = 0; u < kSIPW; ++u)
        copy16_ds<Blocks::kShared, false>(sp[(u >> 1) & 3], c_sgoff[u & 1] + u * 1024, dst + u * 1024);
    }
  };
  auto copy_k = [&](const Cursor& c, int slot) __attribute__((always_inline)) {
    const int row0 = c.j * kTile;
    const half_t* kp = c.base + (long)row0 * ks.n;  // wave-uniform
    char* dst = k_ring + slot * T::kBytes;
    if (row0 + kTile <= N) {
#pragma unroll
      for (int u = 0; u < kKIPW; ++u) copy16(kp, c_kgoff[u], dst + c_kblk[u]);
    } else {
#pragma unroll
      for (int u = 0; u < kKIPW; ++u) {  // rows past the end re-read row N-1 (their dS rows are zero)
        const int back = max(row0 + c_row[u] - (N - 1), 0);
        copy16(kp, c_kgoff[u] - back * ks.n * 2, dst + c_kblk[u]);
      }
    }
  };

  // the first of this wave's pieces of a dS tile: two adjacent ones per 32 keys
  const int own_pieces = (qb >> 2) * kDsPanelTileBytes + (((qb >> 1) & 1) * 4 + 2 * (qb & 1)) * 1024;
  // LDS offsets of this lane's transposing reads.  WIDE: key step kc, read e: key row (kc & 1) * 16 + 8 * e + 4 * g +
  // (L >> 2), with g = lane >> 5, of the piece [panel][(kc >> 1)][query tile][chunk 2 * (qb & 1) + lane bit 4], 8 bytes at
  // (L & 3) * 8 of its 32-byte row, plus the rotation of odd chunks.
  // Otherwise lane 16 g + L reads 8 bytes, 4 queries, of lane group j = L & 3 of the key 16 (g >> 1) + 8 p + 4 (g & 1) + (L >> 2), and then holds query L of 16 of the four keys.  The 16 bytes of a key
  // and j are queries 16 (j >> 1) + 4 (j & 1) + 0..3 and the same + 8; query block nb takes the first half of j = 0, 1
  // and the second of j = 2, 3, or the other way round: so its reads touch all banks.
  int s_off[2][2];  // WIDE: [kc & 1][e], otherwise [nb][p]
  {
    const int L = lane & 15;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        if constexpr (WIDE) {
          const int odd = (lane >> 4) & 1, in_piece = (u * 16 + 8 * e + 4 * (lane >> 5) + (L >> 2)) * 32 + (L & 3) * 8;
          s_off[u][e] = own_pieces + odd * 1024 + ((in_piece + odd * 128) & 1023);
        } else {
          const int g = lane >> 4, j = L & 3;
          s_off[u][e] = own_pieces + (g >> 1) * 1024 + (16 * j + ((8 * e + 4 * (g & 1) + (L >> 2)) ^ (8 * (j & 1)))) * 16 +
                        ((j >> 1) ^ u) * 8;
        }
      }
  }
  int c_off[2];
  swz_cols_off<D>(lane, c_off);
  auto s_frag = [&](const char* tile, int f) __attribute__((always_inline)) {  // 16 keys f, or 32 keys f >> 1 and nb = f & 1
    typedef __attribute__((address_space(3))) s4 lds_s4;
    const char* at = tile + (f >> 1) * 8192;
    s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(at + s_off[f & 1][0]));
    s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(at + s_off[f & 1][1]));
    return __builtin_bit_cast(h8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  typename std::conditional<WIDE, f16v[TileGeom<D>::kDBlocks], f4v[Geom16<D>::kDB][2]>::type acc;
  auto clear = [&](int part) __attribute__((always_inline)) {
    if constexpr (WIDE) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[part][r] = 0.f;
    } else {
      acc[2 * part][0] = acc[2 * part][1] = acc[2 * part + 1][0] = acc[2 * part + 1][1] = f4v{0.f, 0.f, 0.f, 0.f};
    }
  };
#pragma unroll
  for (int part = 0; part < D / kDsStageD; ++part) clear(part);
  // The query, of the wave's 32, of this lane's column.  WIDE: that at position i of the 32, bits 2 and 3 swapped;
  // otherwise that of block nb is my_row ^ (8 * nb).
  const int my_row = WIDE ? (lane & 0x13) | ((lane & 8) >> 1) | ((lane & 4) << 1)
                          : 24 * ((lane >> 3) & 1) + 4 * ((lane >> 2) & 1) + (lane & 3);

  constexpr int kAheadS = kDsRingS - 1, kAheadK = kDsRingK - 1;
  // the copying waves run ahead of the sequence: kAhead tiles are issued before the first is used
  Cursor ahead = open(0, copies_k);
  if (!computes) {
    const int n_first = min(copies_k ? kAheadK : kAheadS, n_tiles);
    for (int t = 0; t < n_first; ++t) {
      if (copies_k) copy_k(ahead, t);
      else copy_s(ahead, t);
      advance(ahead, copies_k);
    }
  }
  Cursor cur = open(0, false);
  int slot_s = 0, slot_k = 0;                                    // ring slots of tile t
  int next_s = kAheadS % kDsRingS, next_k = kAheadK % kDsRingK;  // ring slots of the tiles to copy next
  for (int t = 0; t < n_tiles; ++t) {
    // tile t must have landed; the copies of the tiles after it (at most kAhead - 1 of them) may be in flight
    const int later = n_tiles - 1 - t;
    if (!computes) {
      if (copies_k) wait_vm_tiles<kKIPW, kAheadK - 1>(later);
      else wait_vm_tiles<kSIPW, kAheadS - 1>(later);
    }
    block_barrier();  // tile t is visible to all; everybody is done with tile t - 1, whose slots are reused now
    if (!computes && ahead.round >= 0) {
      if (copies_k) copy_k(ahead, next_k);
      else copy_s(ahead, next_s);
      advance(ahead, copies_k);
    }
    const int qt = 2 * kDsPanels * cur.mblk + (qb >> 1);                          // this wave's query tile
    const int jend = qt >= nt_all ? 0 : (CAUSAL ? min(cur.nt, qt + 1) : cur.nt);  // tiles this wave takes part in
    if (computes && cur.j < jend) {
      const char* Kl = k_ring + slot_k * T::kBytes;
      const char* Sl = s_ring + slot_s * kDsTileBytes;
      // unit n: 16 keys n / 4 and feature block n % 4, or 32 keys n / 8 and feature block n % 8; the K fragments are read
      // kLead units ahead, the four dS fragments up front (order pinned, see the forward)
      constexpr int kN = D / 8, kLead = 4;
      h8 bfrag[4], afrag[kLead];
#pragma unroll
      for (int f = 0; f < 4; ++f) bfrag[f] = s_frag(Sl, f);
      auto run = [&](auto read) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < kLead; ++n) afrag[n] = read(n);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < kN; ++n) {
          if constexpr (WIDE) {
            constexpr int kDB = TileGeom<D>::kDBlocks;
            acc[n % kDB] = mfma(afrag[n % kLead], bfrag[n / kDB], acc[n % kDB]);
          } else {
            constexpr int kDB = Geom16<D>::kDB;
            if (n % 2 == 0) wait_lds_pinned(n + 3 < kN ? 4 : n + 2 < kN ? 2 : 0);
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) acc[n % kDB][nb] = mfma16(afrag[n % kLead], bfrag[2 * (n / kDB) + nb], acc[n % kDB][nb]);
          }
          if (n + kLead < kN) afrag[n % kLead] = read(n + kLead);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      if constexpr (WIDE) {
        run([&](int n) __attribute__((always_inline)) {
          return swz_cols<D>(Kl, n / TileGeom<D>::kDBlocks, n % TileGeom<D>::kDBlocks, c_off);
        });
      } else {
        const Cols16<D> cols(Kl, lane);
        run([&](int n) __attribute__((always_inline)) { return cols.at(0, n / Geom16<D>::kDB, n % Geom16<D>::kDB); });
      }
    }
    if (computes && cur.j == cur.nt - 1) {
      // the block's last tile: the wave's rows leave, staged where its own part of the tile was (rows 0..15 in
      // the pieces of keys 0..31, rows 16..31 in those of keys 32..63); the slot is not refilled before the
      // barrier of the next tile
      char* stage = s_ring + slot_s * kDsTileBytes + own_pieces;
      half_t* out = dQ + cur.out_off;
      const int row0 = cur.mblk * kDsBlockQ + qb * kResident;
#pragma unroll
      for (int part = 0; part < D / kDsStageD; ++part) {
        if constexpr (WIDE) {
          store_resident<kDsStageD>(out + part * kDsStageD, rs, row0, N, *reinterpret_cast<const f16v(*)[1]>(&acc[part]),
                                    scale, lane, stage, my_row, 8192);
        } else {
          const float mul[2] = {scale, scale};
          store_resident16<kDsStageD>(out + part * kDsStageD, rs, row0, N, acc + 2 * part, mul, lane, stage, my_row,
                                      my_row ^ 8, 8192);
        }
        clear(part);
      }
    }
    advance(cur, false);
    slot_s = slot_s + 1 == kDsRingS ? 0 : slot_s + 1;
    slot_k = slot_k + 1 == kDsRingK ? 0 : slot_k + 1;
    next_s = next_s + 1 == kDsRingS ? 0 : next_s + 1;
    next_k = next_k + 1 == kDsRingK ? 0 : next_k + 1;
  }
}

template <int D, bool CAUSAL, int kDsPanels, bool WIDE>
__global__ void __launch_bounds__(ds_threads(kDsPanels), 1)
fmha_bwd_dq_spill_kernel(const half_t* __restrict__ K, Strides ks, const half_t* __restrict__ dS, int np,
                         half_t* __restrict__ dQ, FmhaDivisor H, int N, FmhaOrder order, int slice0, int stream_ds,
                         float scale) {
  __shared__ __attribute__((aligned(1024))) char smem[ds_lds<D, kDsPanels>()];
  bwd_dq_spill_blocks<D, CAUSAL, kDsPanels, WIDE>(K, ks, dS, np, dQ, H, N, order.run, slice0, stream_ds, scale, smem,
                                                  DsBlocks<CAUSAL>{order, order.slices * order.run});
}

// ---------------------------------------------------------------------------
// The dK/dV pass that stores dS and the dQ pass over it in one launch: first all blocks of the former, then those of the
// latter, one to a work group.  One after the other, each pass leaves CUs idle in its last round and the second starts when the
// first has drained; here the dQ blocks of slices that are finished fill the places that the dK/dV blocks leave.  What that
// gives, and where the passes still go one by one: fmha_ds_in_one_launch.
//
// A dQ block waits for the dS of its slice: every wave that stores some counts itself when its stores are done, and the block
// starts when the count is whole.  dS is stored and read past the XCDs' L2s (store_ds), so that is all it takes, on whatever
// XCD the blocks are; a release of everything written (an L2 write-back per block) takes 8 % longer.  The counts of a slice
// have a cache line of their own and are asked for about once a microsecond: with those of 32 slices in one line the work
// groups that ask hold up those that work (24 x 2048 x 128 causal, 111 us; a line each 89).  The wait ends by itself: past
// fmha_ds_wait_ticks, which is longer once all dK/dV blocks of the slice have started, the block forms S and dP itself, as
// fmha_bwd_dq_kernel does, with the same bits as result.  Counting what has started costs up to 0.8 us of a launch (520 x 64),
// so only the slices that need it do.
// ---------------------------------------------------------------------------
constexpr int kReadyStride = 32;  // words from one slice's counts to the next
enum ReadyWord {
  kWavesStored,
  kBlocksStarted,  // of the dK/dV pass, where they are not all on one XCD
  kBlocksAlone     // of the dQ pass, that have not waited to the end
};
template <bool CAUSAL, bool KEEP>
__global__ void __launch_bounds__(kKvThreads, 1)
fmha_bwd_both_spill_kernel(const half_t* __restrict__ Q, const half_t* __restrict__ K, const half_t* __restrict__ V,
                           const half_t* __restrict__ dO, Strides qs, Strides ks, Strides vs, Strides gs,
                           const float* __restrict__ LSE, float* __restrict__ delta, float* __restrict__ lse2,
                           half_t* __restrict__ dQ, half_t* __restrict__ dK, half_t* __restrict__ dV, half_t* dS, unsigned* ready,
                           int np, FmhaDivisor H, int N, FmhaOrder order, unsigned ticks, float c, float scale) {
  constexpr int D = 128;
  static_assert(ds_threads(1) == kKvThreads && kDqThreads == kKvThreads && kDsPanelQ == kKvBlockKeys, "one grid for all");
  constexpr int kLds = dkdv_lds<D>() > dq_lds<D>() ? dkdv_lds<D>() : dq_lds<D>();
  static_assert(ds_lds<D, 1>() <= kLds, "");
  __shared__ __attribute__((aligned(1024))) char smem[kLds];
  int bh, blk;
  bool dq;
  const int nb = order.run;
  if (!fmha_ds_launch_ordered_block(blockIdx.x, order.slices, order.run, order.last_level, CAUSAL, bh, blk, dq)) return;
  unsigned* const counts = ready + (long)bh * kReadyStride;
  auto count = [&](int word) { __hip_atomic_fetch_add(counts + word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  const bool one_xcd = bh < (order.slices & ~7);  // all blocks of the slice: the dK/dV blocks have then started before this dQ block
  if (!dq) {
    if (!one_xcd && threadIdx.x == 0) count(kBlocksStarted);
    bwd_dkdv_block<D, CAUSAL, true, KEEP, false, false, true>(Q, K, V, nullptr, dO, qs, ks, vs, gs, nullptr, delta, lse2, dK, dV, dS,
                                                              np, H, N, 0, c, scale, smem, bh, blk, counts + kWavesStored);
    return;
  }
  if (threadIdx.x == 0) {
    const unsigned long long start = wall_clock64();
    auto read = [&](int word) { return __hip_atomic_load(counts + word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    int whole;
    for (;;) {
      whole = read(kWavesStored) == (unsigned)(kKvPairs * nb);
      if (whole) break;
      const unsigned long long most = fmha_ds_wait_ticks(N, one_xcd || read(kBlocksStarted) == (unsigned)nb);
      if (wall_clock64() - start >= (most < ticks ? most : ticks)) break;
      __builtin_amdgcn_s_sleep(32);  // 2048 cycles
    }
    if (!whole) count(kBlocksAlone);
    *reinterpret_cast<volatile int*>(smem) = whole;
  }
  block_barrier();
  const int whole = __builtin_amdgcn_readfirstlane(*reinterpret_cast<volatile int*>(smem));
  block_barrier();  // the answer is read: the tiles may go where it was
  if (whole)
    bwd_dq_spill_blocks<D, CAUSAL, 1, false>(K, ks, dS, np, dQ, H, N, nb, 0, !KEEP, scale, smem, DsBlock{bh, blk});
  else
    bwd_dq_block<D, CAUSAL, false>(Q, K, V, nullptr, dO, qs, ks, vs, gs, LSE, delta, lse2, dQ, H, N, c, scale, smem, bh,
                                   CAUSAL ? nb - 1 - blk : blk);  // blocks are numbered heaviest first
}

// ---------------------------------------------------------------------------
// Backward of a whole slice in one work group, for slices that a CU can hold: K, all dK and dV, and the dS of 32 queries
// ---------------------------------------------------------------------------
// A wave owns 32 keys (D = 64 past 256 rows: twice 32, blocks w and 15 - w, which under causal masking are together as heavy as
// any other two).  It keeps their dK and dV and their rows of V, negated, in registers.  K lies in LDS whole.  The work group
// walks the queries 32 at a time: Q, dO and O come by copies to LDS that are two tiles ahead, delta is made from them as
// fmha_bwd_delta_kernel makes it, each wave forms S, P, dP and dS of its keys (32 x 32 MFMAs, as bwd_dkdv_block), adds to dV
// and dK, and leaves dS in LDS; behind the next barrier the waves share out the 16 x 16 tiles of dQ of those 32 queries and add
// up all keys in order.  So S and dP are formed once and neither dS nor partial dQ leaves the CU, each input is read once, and
// there is one barrier for 32 queries.  All sums are in the order of the other paths, which give the same bits.
// Bound by the chain of a wave from one barrier to the next: at D = 64 with two blocks of keys a tile takes 5,300 cycles, of which
// the MFMAs of the two waves of a SIMD take 2,560; with one wave to a SIMD doing its work it still takes 4,800.  A wave reads
// 24 to 32 KiB of Q, dO and K for 32 MFMAs of 32 x 32 x 16 and 32 KiB of K and dS for 16 of 16 x 16 x 32, 120 instructions, each
// of which holds it for 15 cycles; the CU's LDS is busy half of the time.  What helps is fewer instructions between two
// barriers, and MFMAs above all vector work: the products of a tile in an order in which P and dS are formed in the shadow of
// others (work), no copies of fragments between registers (queries), what depends on the lane worked out once.  us without and
// with these, backward, N x slices: D = 64 512 x 192 52.9, 50.4; 300 x 256 33.9, 32.8; 256 x 256 22.9, 22.2; causal 384 x 256 36.5,
// 33.1; 160 x 256 15.1, 13.8; D = 128 256 x 256 36.7, 35.4; causal 32.4, 30.5; 100 x 256 17.2, 16.2.
// Not taken, 512 x 192: 16 waves of 32 keys 52.7; dQ of the tile before between the products of a tile 49.7; waves 4 to 7 with
// dQ at the end of a tile 52.7; S and dP of both blocks from the same fragments 54.2, and before, with P and dS in stretches
// without MFMAs, 54.6; priorities +-1 %.
// 512 x 192 slices, D = 64: 50.7 us, 635 TFLOP/s on the 192 CUs that have work; two passes that form S and dP twice: 61.  256 x
// 256, D = 128: 35.3 us, 610 TFLOP/s; over dS in memory: 50.7.
// At D = 128 without a mask 129 to 160 rows have four idle waves and one of up to 32 keys.  bwd_dkdv_block shares such keys
// between its four pairs of waves, tile j to pair j mod 4, and adds the four sums up at the end; to have its bits the idle
// waves do the same here.
constexpr int kSliceWaves = 8;
constexpr int kSliceThreads = kSliceWaves * 64;
template <int D, int KB>
struct SliceGeom {
  static constexpr int kRows = kSliceWaves * KB * kResident;  // the longest slice
  static constexpr int kTileBytes = kResident * D * 2;        // 32 rows of Q or dO
  static constexpr int kExchange = kRows * kResident * 2;     // dS of 32 queries
  static constexpr int kRingOff = kRows * D * 2;              // behind K
  static constexpr int kOOff = kRingOff + 3 * 2 * kTileBytes;
  static constexpr int kStOff = kOOff + kTileBytes;
  static constexpr int kExOff = kStOff + 2 * kRows * 4;
  static constexpr int kLds = kExOff + 2 * kExchange;
};
template <int D, int KB, bool CAUSAL>
__global__ void __launch_bounds__(kSliceThreads, 1)
fmha_bwd_slice_kernel(const half_t* __restrict__ Q, const half_t* __restrict__ K, const half_t* __restrict__ V,
                      const half_t* __restrict__ O, const half_t* __restrict__ dO, Strides qs, Strides ks, Strides vs, Strides gs,
                      const float* __restrict__ LSE, float* __restrict__ Delta, float* __restrict__ LSE2, half_t* __restrict__ dQ,
                      half_t* __restrict__ dK, half_t* __restrict__ dV, FmhaDivisor H, int N, float c, float scale) {
  using Geo = SliceGeom<D, KB>;
  using T = SwzTile<D>;
  constexpr int kKS = TileGeom<D>::kKSteps, kDB = TileGeom<D>::kDBlocks;
  constexpr int kC = 2 * T::kNC / 4;  // copies of a wave per 32-row tile
  __shared__ __attribute__((aligned(1024))) char smem[Geo::kLds];
  char* const ring = smem + Geo::kRingOff;
  float* const st_lse = reinterpret_cast<float*>(smem + Geo::kStOff);
  float* const st_delta = st_lse + Geo::kRows;

  // what depends on the lane is worked out again where it is needed, not kept in registers across the loop
  auto thread_now = []() __attribute__((always_inline)) {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
  };
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int bh = blockIdx.x, b = bh / H, h = bh - b * H;
  const int rs = H * D;
  const long head_off = ((long)b * N * H + h) * D;
  const int nj = (N + kResident - 1) / kResident;  // 32-query tiles, 32-key blocks
  const half_t* const Qb = Q + b * qs.b + (long)h * qs.h;
  const half_t* const Gb = dO + b * gs.b + (long)h * gs.h;
  const half_t* const Kb = K + b * ks.b + (long)h * ks.h;
  int blk[KB];  // this wave's key blocks
  blk[0] = wave;
  const bool shared = D == 128 && !CAUSAL && nj == 5;  // waves 4 to 7 own block 4, each every fourth tile
  if (shared && wave > 4) blk[0] = 4;
  if constexpr (KB == 2) blk[KB - 1] = 2 * kSliceWaves - 1 - wave;

  // Q (waves 0-3) or dO (4-7) of 32 rows
  const bool copies_q = wave < 4;
  const half_t* const c_base = copies_q ? Qb : Gb;
  const int c_stride = copies_q ? qs.n : gs.n;
  char* const c_dst = ring + (copies_q ? 0 : Geo::kTileBytes) + (wave & 3) * kC * 1024;
  // What depends on the lane is worked out once; a tile costs a few scalar additions.
  int c_off[kC];
#pragma unroll
  for (int u = 0; u < kC; ++u) {
    int row;
    copy_src<D>((wave & 3) * kC + u, threadIdx.x & 63, c_stride, row, c_off[u]);
  }
  const half_t* c_next = c_base;  // the next tile to copy
  auto copy_tile = [&](int j, int slot) __attribute__((always_inline)) {
    char* const dst = c_dst + slot * 2 * Geo::kTileBytes;
    if ((j + 1) * kResident <= N) {
#pragma unroll
      for (int u = 0; u < kC; ++u) copy16(c_next, c_off[u], dst + u * 1024);
    } else {  // the last tile: rows past the end re-read row N-1
      const int lane = thread_now() & 63;
#pragma unroll
      for (int u = 0; u < kC; ++u) {
        int row, off;
        copy_src<D>((wave & 3) * kC + u, lane, c_stride, row, off);
        copy16(c_next, off - max(j * kResident + row - (N - 1), 0) * c_stride * 2, dst + u * 1024);
      }
    }
    c_next += kResident * (long)c_stride;
  };
  {  // K, all of it
    constexpr int kPer = T::kInstrs / kSliceWaves;
    int row[kPer], off[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) copy_src<D>(wave * kPer + u, threadIdx.x & 63, ks.n, row[u], off[u]);
    for (int t = 0; t * kTile < N; ++t) {
      const half_t* const base = Kb + (long)t * kTile * ks.n;
#pragma unroll
      for (int u = 0; u < kPer; ++u) {
        const int back = max(t * kTile + row[u] - (N - 1), 0);
        copy16(base, off[u] - back * ks.n * 2, smem + t * T::kBytes + (wave * kPer + u) * 1024);
      }
    }
  }
  copy_tile(0, 0);

  // V rows, negated
  h8 vf[KB][kKS];
  constexpr bool kStaged = D == 64;  // through where dS goes, which at D = 128 holds only half of them
  if constexpr (kStaged) {
    static_assert(D != 64 || 2 * Geo::kExchange >= kSliceWaves * KB * T::kBytes / 2, "");
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
      copy_rows<D>(V + b * vs.b + (long)h * vs.h, vs.n, blk[kb] * kResident, N, thread_now() & 63,
                   smem + Geo::kExOff + (wave * KB + kb) * (T::kBytes / 2));
  } else {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const int lane = thread_now() & 63;
      const half_t* const vp = V + b * vs.b + (long)h * vs.h + (long)min(blk[kb] * kResident + (lane & 31), N - 1) * vs.n +
                               (lane >> 5) * 8;
#pragma unroll
      for (int kk = 0; kk < kKS; ++kk) vf[kb][kk] = *reinterpret_cast<const h8*>(vp + kk * 16);
    }
  }
  // Row statistics of 32 rows, in the order of fmha_bwd_delta_kernel, by the first D / 16 waves.  The rows of O that a wave
  // adds up it copies itself, 1 KiB of them, for its lanes to read back.
  constexpr int kLanes = D / 8;
  const bool makes_stats = wave < D / 16;
  char* const o_mine = smem + Geo::kOOff + (wave & (D / 16 - 1)) * 1024;
  char* const o_second = ring + 2 * 2 * Geo::kTileBytes + (wave & (D / 16 - 1)) * 1024;  // free until tile 2 is copied
  const int st_row = (threadIdx.x / kLanes) & (kResident - 1), st_col = threadIdx.x % kLanes;
  const int o_off = (st_row * rs + st_col * 8) * 2;
  const half_t* o_next = O + head_off;  // the next tile to ask for
  // of this lane's piece of O where it was copied to, and of dO (chunk st_col of row st_row of a tile, SwzTile) in slot 0
  const unsigned o_at = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)o_mine + (threadIdx.x & 63) * 16;
  const unsigned g_at = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)ring + Geo::kTileBytes +
                        T::block_off(st_row >> 4, st_col >> 2) + (st_row & 15) * 64 +
                        (((st_col & 3) ^ swz((st_row & 15) >> 2)) * 16);
  auto stats_load = [&](int j, char* to) __attribute__((always_inline)) {
    if (makes_stats) {
      const int past = max(j * kResident + st_row - (N - 1), 0);  // rows past the end re-read row N-1
      copy16(o_next, o_off - past * rs * 2, to);
      o_next += kResident * (long)rs;
    }
  };
  auto stats_make = [&](int j, int slot, unsigned from) __attribute__((always_inline)) {
    if (makes_stats) {
      typedef __attribute__((address_space(3))) h8 lds_h8;
      const h8 o8 = *(const lds_h8*)(uintptr_t)from;
      const h8 g8 = *(const lds_h8*)(uintptr_t)(g_at + slot * 2 * Geo::kTileBytes);
      float a = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) a = fmaf((float)o8[e], (float)g8[e], a);
      const auto dpp = [](float x, auto ctrl) __attribute__((always_inline)) {
        return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(x), decltype(ctrl)::value, 15, 15, true));
      };
      if (kLanes == 16) a += dpp(a, IntTag<0x128>{});                                       // of the lane at ^ 8 (of 16)
      a += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(a), (4 << 10) | 31));  // ^ 4
      a += dpp(a, IntTag<0x4E>{});                                                          // ^ 2
      a += dpp(a, IntTag<0xB1>{});                                                          // ^ 1
      const int at = j * kResident + st_row;
      if (st_col == 0) {
        st_delta[at] = a;
        if (at < N) Delta[(long)bh * N + at] = a;
      }
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the rows of O are read, others may take their place
      asm volatile("" ::: "memory");
    }
  };
  stats_load(0, o_mine);
  if (nj > 1) {
    copy_tile(1, 1);
    stats_load(1, o_second);
  }
  if ((int)threadIdx.x < Geo::kRows) {
    const int at = min((int)threadIdx.x, N - 1);
    const float l2 = LSE[(long)bh * N + at] * kLog2e;
    st_lse[threadIdx.x] = l2;
    LSE2[(long)bh * N + at] = l2;  // rows past the end write that of row N-1 again
  }

  // LDS addresses of this lane's fragments: rows and columns of Q (+ kTileBytes: of dO) in slot 0, rows of this wave's K, and for
  // dQ columns of K and dS: features 16 db .. and 16 of the 32 queries (D = 128: both halves).  Odd fragments of rows are at ^
  // kOddRows, the upper eight rows of a fragment of columns at ^ kUpper, those of dS at + 256.
  constexpr unsigned kOddRows = 32, kUpper = 512 + 32;
  constexpr int kQB = D == 128 ? 2 : 1;
  const int db = D == 128 ? wave : wave & 3, qb0 = D == 128 ? 0 : wave >> 2;
  unsigned ra, ca, kr[KB], ka, ea;
  {
    const int lane = threadIdx.x & 63, L = lane & 15, g = lane >> 4, m = L & 3;
    int r_off[2], t_off[2];
    swz_rows_off<D>(lane, r_off);
    swz_cols_off<D>(lane, t_off);
    ra = opaque_lds_address(ring + r_off[0]);
    ca = opaque_lds_address(ring + t_off[0]);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
      kr[kb] = opaque_lds_address(smem + (blk[kb] >> 1) * T::kBytes + (blk[kb] & 1) * T::block_off(2, 0) + r_off[0]);
    ka = opaque_lds_address(smem + cols16_off<D>(lane, 0, db & 1) + T::block_off(0, db >> 1));
    ea = opaque_lds_address(smem + Geo::kExOff + qb0 * 1024 + (16 * (g >> 1) + 4 * (g & 1) + (L >> 2)) * 32 + (m & 1) * 16 +
                            (m >> 1) * 8);
  }

  f16v dv[KB][kDB], dk[KB][kDB];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int d = 0; d < kDB; ++d)
#pragma unroll
      for (int r = 0; r < 16; ++r) dv[kb][d][r] = dk[kb][d][r] = 0.f;

  f16v zero;
#pragma unroll
  for (int r = 0; r < 16; ++r) zero[r] = 0.f;
  staged_rows_landed();
  if constexpr (kStaged) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      const StagedRows<D> rows{smem + Geo::kExOff + (wave * KB + kb) * (T::kBytes / 2), (int)threadIdx.x & 63};
#pragma unroll
      for (int kk = 0; kk < kKS; ++kk) vf[kb][kk] = rows.wide(kk);
    }
    staged_rows_read();
  }
#pragma unroll
  for (int kb = 0; kb < KB; ++kb)
#pragma unroll
    for (int kk = 0; kk < kKS; ++kk) {
      vf[kb][kk] = -vf[kb][kk];
      asm volatile("" : "+v"(vf[kb][kk]));  // negated here, not in the loop
    }

  // dQ of tile j
  auto queries = [&](int j) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) s4 lds_s4;
    struct Pair { h8 a, b[kQB]; };
    unsigned ex = ea + (j & 1) * Geo::kExchange;
    const int n_blocks = CAUSAL ? j + 1 : nj;
    f4v dq[kQB];
#pragma unroll
    for (int n = 0; n < kQB; ++n) dq[n] = f4v{0.f, 0.f, 0.f, 0.f};
    auto both = [](unsigned a0, unsigned a1) __attribute__((always_inline)) {
      const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(uintptr_t)a0);
      const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(uintptr_t)a1);
      return __builtin_bit_cast(h8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    // every address is one of these and a constant
    unsigned k_lo = ka, k_hi = ka ^ kUpper;
    auto read = [&](int kb) __attribute__((always_inline)) {
      Pair f;
      const unsigned kt = (kb >> 1) * T::kBytes + (kb & 1) * T::block_off(2, 0), et = kb * 2048;
      f.a = both(k_lo + kt, k_hi + kt);
#pragma unroll
      for (int n = 0; n < kQB; ++n) f.b[n] = both(ex + (et + n * 1024), ex + (et + n * 1024 + 256));
      return f;
    };
    auto use = [&](const Pair& f) __attribute__((always_inline)) {
#pragma unroll
      for (int n = 0; n < kQB; ++n) dq[n] = mfma16(f.a, f.b[n], dq[n]);
    };
    // Four blocks of keys at a time, the next four read while they are used; then the last one to four.  As a loop: unrolled, with
    // an exit after each four, the compiler copies the fragments from registers to registers at every exit, 150 instructions.
    constexpr int kGroup = CAUSAL ? 2 : 4;
    Pair frag[kGroup];
#pragma unroll
    for (int u = 0; u < kGroup; ++u) frag[u] = read(u);  // also past the last block: of no use then
    __builtin_amdgcn_sched_barrier(0);
    int left = n_blocks;
#pragma unroll 1
    for (; left > kGroup; left -= kGroup) {
      k_lo += kGroup / 2 * T::kBytes, k_hi += kGroup / 2 * T::kBytes, ex += kGroup * 2048;
#pragma unroll
      for (int u = 0; u < kGroup; ++u) {
        use(frag[u]);
        frag[u] = read(u);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int u = 0; u < kGroup; ++u)
      if (u < left) use(frag[u]);
    const int lane = thread_now() & 63;
#pragma unroll
    for (int n = 0; n < kQB; ++n) {
      const int q = j * kResident + 16 * (qb0 + n) + (lane & 15);
      h4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (half_t)(dq[n][e] * scale);
      if (q < N) *reinterpret_cast<h4*>(dQ + head_off + (long)q * rs + 16 * db + 4 * (lane >> 4)) = v;
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // Tile j, NB of this wave's key blocks, in units of an A fragment and its MFMAs, and what is formed in their shadow:
  //   NB x kKS  S of one block after the other          P of the block before
  //   NB x kKS  dP - delta                              P of the last block
  //   2 x kDB   dV += of queries 0..15, then 16..31     dS of queries 0..15, behind the products with their P
  //   2 x kDB   dK                                      dS of queries 16..31
  auto work = [&](int j, int slot, auto nb_tag, auto masked_tag) __attribute__((always_inline)) {
    constexpr int NB = decltype(nb_tag)::value;
    constexpr bool MASKED = decltype(masked_tag)::value != 0;
    constexpr int kS = NB * kKS, kP = 2 * kS, kV = kP + 2 * kDB, kUnits = kV + 2 * kDB;  // the first unit past each kind
    constexpr int kPairs = 8 / kKS;  // pairs of P formed in a unit
    constexpr int kLead = NB == 2 ? 2 : 3;
    // The first unit that forms dS.  neg_mul_to_f16x2 is inline asm: the compiler leaves no time in front of it for the results of
    // the last MFMA of dP - delta to arrive, 11 wait states after its issue.  The MFMAs of the units in between, of 8 passes
    // each and issued one after the other, do: two of them are 16.
    constexpr int kDs = kP + kDB;
    static_assert(kDs - kP >= 2, "dS would be formed from a dP that is not there yet");
    struct Frag { h8 a, k; };
    const unsigned at = slot * 2 * Geo::kTileBytes;
    const int q0 = j * kResident, lane = thread_now() & 63, i = lane & 31, hh = lane >> 5;
    const char* const st = smem + Geo::kStOff + (q0 + 4 * hh) * 4;
    const unsigned qa0 = ra + at, qa1 = qa0 ^ kOddRows, qc0 = ca + at, qc1 = qc0 ^ kUpper;
    f16v s[NB], x[NB];
    u4v y[NB][2];  // [16 queries]: P, then dS, fp16 pairs in B-operand order
    f4v l4[NB];
    Frag frag[kLead];
    auto read = [&](int m) __attribute__((always_inline)) {
      Frag f;
      if (m < kS) {
        f.a = swz_rows_at<D>(qa0, qa1, 0, m % kKS);
        f.k = swz_rows_at<D>(kr[m / kKS], kr[m / kKS] ^ kOddRows, 0, m % kKS);
      } else if (m < kP) {
        f.a = swz_rows_at<D>(qa0 + Geo::kTileBytes, qa1 + Geo::kTileBytes, 0, m % kKS);
      } else if (m < kV) {
        f.a = swz_cols_at<D>(qc0 + Geo::kTileBytes, qc1 + Geo::kTileBytes, (m - kP) / kDB, (m - kP) % kDB);
      } else {
        f.a = swz_cols_at<D>(qc0, qc1, (m - kV) / kDB, (m - kV) % kDB);
      }
      return f;
    };
    auto p_pair = [&](int n, int e) __attribute__((always_inline)) {  // of 8: two neighbouring queries
      const int r = 2 * e;
      if (e % 2 == 0) l4[n] = *reinterpret_cast<const f4v*>(st + 16 * e);
      float p0 = fast_exp2(fmaf(s[n][r], c, -l4[n][r & 3])), p1 = fast_exp2(fmaf(s[n][r + 1], c, -l4[n][(r & 3) + 1]));
      if (MASKED) {  // causal: queries key .. N - 1 count, one comparison: 384 x 256, D = 64 32.9, 32.2 us
        const int row = 8 * (r >> 2) + (r & 3), at = q0 + 4 * hh, q = q0 + row + 4 * hh, key = blk[n] * kResident + i;
        const unsigned seen = max(N - key, 0);
        if (CAUSAL ? (unsigned)(row - (key - at)) >= seen : q >= N) p0 = 0.f;
        if (CAUSAL ? (unsigned)(row + 1 - (key - at)) >= seen : q + 1 >= N) p1 = 0.f;
      }
      y[n][e >> 2][e & 3] = pack_f16(p0, p1);
    };
    auto ds_pair = [&](int n, int e) __attribute__((always_inline)) {
      y[n][e >> 2][e & 3] = neg_mul_to_f16x2(y[n][e >> 2][e & 3], x[n][2 * e], x[n][2 * e + 1]);
    };
    auto ds_out = [&](int cc) __attribute__((always_inline)) {
      const int lane2 = thread_now() & 63, i2 = lane2 & 31;
      char* const ex = smem + Geo::kExOff + (j & 1) * Geo::kExchange + (2 * i2 + (lane2 >> 5)) * 16;
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        h8 v = __builtin_bit_cast(h8, y[n][cc]);
        if (MASKED && blk[n] * kResident + i2 >= N) v = h8{};  // keys past the end: no dQ
        *reinterpret_cast<h8*>(ex + blk[n] * 2048 + cc * 1024) = v;
      }
    };
    auto delta_in = [&](int n) __attribute__((always_inline)) {
#pragma unroll
      for (int quad = 0; quad < 4; ++quad) {
        const f4v d4 = *reinterpret_cast<const f4v*>(st + Geo::kRows * 4 + 32 * quad);
#pragma unroll
        for (int r = 0; r < 4; ++r) x[n][4 * quad + r] = d4[r];
      }
    };
#pragma unroll
    for (int m = 0; m < kLead; ++m) frag[m] = read(m);
    __builtin_amdgcn_sched_barrier(0);
    static_for<kUnits>([&](auto m_tag) __attribute__((always_inline)) {
      constexpr int m = decltype(m_tag)::value;
      const Frag f = frag[m % kLead];
      if constexpr (m < kS) {
        constexpr int n = m / kKS;
        s[n] = mfma(f.a, f.k, m % kKS == 0 ? zero : s[n]);
        if constexpr (m == kS - 1) delta_in(0);
      } else if constexpr (m < kP) {
        constexpr int n = (m - kS) / kKS;
        x[n] = mfma(f.a, vf[n][m % kKS], x[n]);
        if constexpr (NB == 2 && m == kS + kKS - 1) delta_in(NB - 1);
      } else if constexpr (m < kV) {
        constexpr int u = m - kP;
#pragma unroll
        for (int n = 0; n < NB; ++n) dv[n][u % kDB] = mfma(f.a, __builtin_bit_cast(h8, y[n][u / kDB]), dv[n][u % kDB]);
      } else {
        constexpr int u = m - kV;
#pragma unroll
        for (int n = 0; n < NB; ++n) dk[n][u % kDB] = mfma(f.a, __builtin_bit_cast(h8, y[n][u / kDB]), dk[n][u % kDB]);
      }
      if constexpr (m + kLead < kUnits) frag[m % kLead] = read(m + kLead);
      static_for<NB>([&](auto n_tag) __attribute__((always_inline)) {
        constexpr int n = decltype(n_tag)::value, first = (n + 1) * kKS + 1;
        if constexpr (m >= first && m < first + kKS) {
#pragma unroll
          for (int e = 0; e < kPairs; ++e) p_pair(n, kPairs * (m - first) + e);
        }
      });
      static_for<2>([&](auto cc_tag) __attribute__((always_inline)) {
        constexpr int cc = decltype(cc_tag)::value, first = kDs + cc * kDB;
        if constexpr (m >= first && m < first + kDB) {
          constexpr int kOf = 4 / kDB;
#pragma unroll
          for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int e = 0; e < kOf; ++e) ds_pair(n, 4 * cc + kOf * (m - first) + e);
          if constexpr (m == first + kDB - 1) ds_out(cc);
        }
      });
      __builtin_amdgcn_sched_barrier(0);
    });
  };

  block_barrier();
  stats_make(0, 0, o_at);
  if (nj > 1) stats_make(1, 1, o_at + (unsigned)(o_second - o_mine));
  int slot = 0, j = 0;
  auto top = [&]() __attribute__((always_inline)) {
    wait_vm<0>();  // tile j + 1 and its rows of O, asked for an iteration ago
    block_barrier();
    if (j > 0 && j + 1 < nj) stats_make(j + 1, slot == 2 ? 0 : slot + 1, o_at);
    if (j + 2 < nj) {
      stats_load(j + 2, o_mine);
      copy_tile(j + 2, slot == 0 ? 2 : slot - 1);
    }
    if (j > 0) queries(j - 1);
  };
  auto next = [&]() __attribute__((always_inline)) {
    ++j;
    slot = slot == 2 ? 0 : slot + 1;
  };
  // Tiles in which none, one or both of this wave's key blocks count; those on the diagonal of one and at the end of the slice
  // with the mask, each in a loop of its own so that no accumulator crosses a branch.
  const int whole = N / kResident;
  // This wave has keys past the end, which the mask keeps out of dQ.  (Under causal masking only tiles from `whole` on need it, which
  // have a mask anyway; without it in the others, us: D = 64 300 x 256 26.4, 26.5; 500 x 256 45.0 both; 200 x 256 18.1, 17.9.)
  const bool past = nj > whole && (blk[0] == whole || blk[KB - 1] == whole);
  auto span = [&](int end, int diag, auto nb_tag) __attribute__((always_inline)) {  // up to `end`, with a diagonal tile `diag`
    while (j < end) {
      while (j < end && (past || j == diag || j >= whole)) {
        top();
        work(j, slot, nb_tag, IntTag<1>{});
        next();
      }
      while (j < end && !past && j != diag && j < whole) {
        top();
        work(j, slot, nb_tag, IntTag<0>{});
        next();
      }
    }
  };
  const int first = blk[0] >= nj ? nj : CAUSAL ? blk[0] : 0, second = blk[KB - 1] >= nj ? nj : CAUSAL ? blk[KB - 1] : 0;
  while (j < first) {
    top();
    next();
  }
  if constexpr (D == 128 && !CAUSAL) {
    if (shared && wave >= 4) {
      for (int mine = wave - 4; mine < nj; mine += 4) {
        while (j < mine) {
          top();
          next();
        }
        top();
        work(j, slot, IntTag<1>{}, IntTag<1>{});
        next();
      }
      while (j < nj) {
        top();
        next();
      }
    }
  }
  if constexpr (KB == 1) {
    span(nj, CAUSAL ? blk[0] : -1, IntTag<1>{});
  } else {
    span(second, CAUSAL ? blk[0] : -1, IntTag<1>{});
    span(nj, CAUSAL ? blk[1] : -1, IntTag<2>{});
  }
  top();

  static_assert(kSliceWaves * StageGeom<D>::kBytes <= Geo::kExOff, "the output staging tiles do not reach the dS of a tile");
  block_barrier();
  char* const stage = smem + wave * StageGeom<D>::kBytes;
  const int lane = thread_now() & 63;
  if constexpr (D == 128 && !CAUSAL) {
    if (shared) {  // the sums of the four waves, added in their order by the first one
      constexpr int kQuads = kDB * 4, kOff = kSliceWaves * StageGeom<D>::kBytes;  // four sums of a lane at a time
      static_assert(kOff + 3 * kQuads * 1024 <= Geo::kLds, "the sums of three waves fit, of dV and then of dK");
      auto add = [&](f16v (&acc)[KB][kDB]) __attribute__((always_inline)) {
        char* const at = smem + kOff + lane * 16;
        if (wave > 4) {
#pragma unroll
          for (int u = 0; u < kQuads; ++u) {
            f4v x;
#pragma unroll
            for (int r = 0; r < 4; ++r) x[r] = acc[0][u >> 2][4 * (u & 3) + r];
            *reinterpret_cast<f4v*>(at + ((wave - 5) * kQuads + u) * 1024) = x;
          }
        }
        block_barrier();
        if (wave == 4) {
          for (int other = 0; other < 3; ++other)
#pragma unroll
            for (int u = 0; u < kQuads; ++u) {
              const f4v x = *reinterpret_cast<const f4v*>(at + (other * kQuads + u) * 1024);
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[0][u >> 2][4 * (u & 3) + r] += x[r];
            }
        }
        block_barrier();
      };
      add(dv);
      add(dk);
      if (wave > 4) return;
    }
  }
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    store_resident<D>(dV + head_off, rs, blk[kb] * kResident, N, dv[kb], 1.f, lane, stage);
    store_resident<D>(dK + head_off, rs, blk[kb] * kResident, N, dk[kb], scale, lane, stage);
  }
}

// ---------------------------------------------------------------------------
// Host side: validation and launches.
// ---------------------------------------------------------------------------
// Limits of the 32-bit arithmetic in the kernels and of what a launch can take:
//   - a (batch, head) row of lse / delta is addressed with 32-bit byte offsets (n < 2^29);
//   - the dense row stride head * d and the per-lane byte offsets built from it are 32-bit
//     (head * d < 2^24, the bound the strided entry points put on the sequence stride);
//   - a launch holds fewer than 2^32 threads: the finest non-persistent grids are the 128-row
//     blocks of the backward at 512 threads each (fewer than 2^23 blocks) and the delta pass
//     at one thread per 8 features of a row (batch * head * n * d / 8 < 2^32).
// Checked up front, so that nothing is enqueued for a problem a later pass would refuse.
int check_shape(int batch, int head, int m, int n, int d) {
  if (batch <= 0 || head <= 0 || n <= 0 || m != n) return FUSED_MHA_ERR_BAD_SHAPE;
  if (d != 64 && d != 128) return FUSED_MHA_ERR_BAD_HEAD_DIM;
  if (n >= (1 << 29)) return FUSED_MHA_ERR_TOO_LARGE;
  if ((long)head * d >= (1L << 24)) return FUSED_MHA_ERR_TOO_LARGE;
  const long blocks = (long)((n + 127) / 128) * batch * head;
  if (blocks >= (1L << 23)) return FUSED_MHA_ERR_TOO_LARGE;
  if ((long)batch * head * n * (d / 8) >= (1L << 32)) return FUSED_MHA_ERR_TOO_LARGE;
  return FUSED_MHA_OK;
}

// Launch through the C API: the status returned belongs to this launch alone
// (the <<<>>> form plus hipGetLastError would also report, and clear, an error
// left behind by earlier, unrelated work on the thread).
template <typename... Params, typename... Args>
hipError_t launch(void (*kernel)(Params...), unsigned grid, unsigned block, hipStream_t stream, Args... args) {
  static_assert(sizeof...(Params) == sizeof...(Args), "argument count");
  auto pack = [](Params... p) { return std::tuple<Params...>(p...); };
  std::tuple<Params...> vals = pack(args...);  // converted to the kernel's parameter types
  void* ptrs[sizeof...(Params)];
  int idx = 0;
  std::apply([&](auto&... v) { ((ptrs[idx++] = (void*)&v), ...); }, vals);
  return hipLaunchKernel((const void*)kernel, dim3(grid), dim3(block), ptrs, 0, stream);
}

// Work groups of a persistent launch over `total` blocks: one per CU of the current device,
// rounded down to a multiple of 8 (the XCDs take work-group ids round-robin), or one per block
// when there are no more blocks than that.
unsigned persistent_grid(int total) {
  static std::mutex mu;
  static int cus[64] = {};
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < 64) {
    std::lock_guard<std::mutex> lock(mu);
    if (!cus[dev]) {
      int v = 0;
      if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0) cus[dev] = v;
    }
    n = cus[dev];
  }
  if (n < 8) n = 256;  // the query failed: MI355X has 256
  n &= ~7;
  return (unsigned)(total <= n ? total : n);
}

bool misaligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) != 0; }

// Strides from the C structure, or the dense layout when the caller gave none.
Strides to_strides(const fused_mha_strides* st, int head, int n, int d) {
  if (!st) return Strides{(long)n * head * d, head * d, d};
  return Strides{(long)st->batch, (int)st->seq, (int)st->head};
}

// Every row must start on a 16-byte boundary (strides in multiples of 8 halves);
// the per-lane byte offsets inside a 64-row tile are 32-bit.
bool bad_strides(const fused_mha_strides* st) {
  if (!st) return false;
  if (st->batch < 0 || st->seq < 0 || st->head < 0) return true;
  if ((st->batch | st->seq | st->head) & 7) return true;
  return st->seq >= (1 << 24) || st->head >= (1LL << 31);
}

// Whether a launch of equal blocks, two to a CU, has work for at most half of the places in its last round, the second one or
// (up to max_rounds) the third.  Two blocks that share a CU evenly end together, and the last ones then run alone, at little
// over half the rate of a pair; with one of the two going first (odd_slots_first) its place is free sooner, and the last
// blocks run beside the others.  us without and with that, D = 64, N x slices (rounds), forward, then backward: 1024 x 66
// (1.03) 31.1, 29.6; 92.1, 90.6.  1024 x 96 (1.5) 34.3, 33.1; 102.8, 102.7.  2048 x 40 (1.25) 56.2, 53.3; 174, 170.  8192 x 12
// (1.5) 218, 211; 725, 703.  2048 x 66 (2.06) 89.7, 88.7; 279, 271.  1024 x 160 (2.5) 54.7, 55.2; 166, 164.  2048 x 80 (2.5)
// 96.7, 96.8; 300, 297.  (Backwards of 1 to 1.25 rounds go in one launch, unless their passes are called one by one:
// fmha_passes_at_once.)  Forward D = 128: 1031 x 60 (1.05) 48.9, 46.8; 2048 x 40 91.8, 90.1; 4096 x 20 174, 170.
// Short blocks have nothing to gain (512 x 192: 21.6, 21.5; 61.1, 62.2.  256 x 320: 14.1, 14.3; 39.2, 39.4), nor has a fuller
// last round (1024 x 112, 1.75: 41.2, 42.2; dK/dV 69.1, 70.1.  1024 x 192, 3: 65.5, 65.6; dK/dV 110, 118), nor more rounds
// (1024 x 288, 4.5: 96.9, 98.4), nor a causal launch, where the blocks differ (1024 x 64 forward: 16.4, 18.2).
// A wave keeps its priority to its end, also before waves of another stream on the same CU.  Those take no longer for it: us of
// a 128 MiB elementwise kernel, of one of 4 MiB and of a 4096 cubed fp16 product on a second stream, without and with it:
// beside the forward 8192 x 12 59.3, 58.3; 10.7, 10.7; 234, 228; beside its backward 57.7, 55.3; 10.3, 10.3; 220, 217; beside
// the forward 1031 x 60 67.1, 65.7; 13.1, 13.1; 148, 149; beside the D = 128 backward, where the dK/dV pass has priorities of
// its own, 2048 x 80 72.6, 73.0; 11.0, 11.0; 212, 211.  (The D = 64 backward itself gives way more: 960, 1057 beside the first
// kernel; both streams' work together is done as early, 46.1, 45.4 ms.)
bool half_round_left(long blocks, int n, int max_rounds) {
  if (n < 1024) return false;
  const long places = 2 * (long)persistent_grid(1 << 30), rounds = blocks / places, left = blocks % places;
  return rounds >= 1 && rounds < max_rounds && left > 0 && 2 * left <= places;
}

template <int D, bool CAUSAL>
int launch_forward(const void* q, const void* k, const void* v, Strides qs, Strides ks, Strides vs, void* o, void* lse,
                   int batch, int head, int n, float scale, hipStream_t stream) {
  // scale == 0 would turn the masked scores (-inf) into NaN when multiplied; a
  // tiny positive factor gives the same uniform softmax and keeps -inf * c = -inf.
  const float c = fmaxf(fabsf(scale) * kLog2e, 1e-30f);
  const int negate = scale < 0.f ? 1 : 0;
  const bool short_tail = n > kPipeBlockQ && (n - 1) % kPipeBlockQ < kResident;
  // the number of CUs is a question to the runtime, which small calls feel: not asked where no rule needs it
  const int cus = D == 128 || short_tail ? (int)persistent_grid(1 << 30) : 0;
  if constexpr (D == 128) {
    const int nmb = (n + kFwdBlockQ - 1) / kFwdBlockQ, total = nmb * batch * head;
    if (fmha_persistent_forward_pays(batch * head, n, cus, CAUSAL)) {
      const hipError_t rc = launch(fmha_fwd_kernel<D, CAUSAL>, persistent_grid(total), kFwdThreads, stream,
                                   (const half_t*)q, (const half_t*)k, (const half_t*)v, qs, ks, vs, (half_t*)o,
                                   (float*)lse, head, n, nmb, batch * head, c, negate);
      return rc == hipSuccess ? FUSED_MHA_OK : FUSED_MHA_ERR_LAUNCH;
    }
  }
  const int nmb = (n + kPipeBlockQ - 1) / kPipeBlockQ, total = nmb * batch * head;
  const int slices = batch * head;
  int tails_per_block = 0, tails = 0, nb = nmb;  // nb: blocks of a slice beside the one with the tail
  auto kernel = fmha_fwd_pipe_kernel<D, CAUSAL, false, false>;
  unsigned blocks = total;
  static_assert(kPipeBlockQ == 128 && kResident == 32, "as fmha_tails_per_block has it");
  if (short_tail) tails_per_block = fmha_tails_per_block(D, n, slices, cus, CAUSAL);
  if (tails_per_block) {
    tails = fmha_tail_blocks(slices, tails_per_block);
    nb = nmb - 1;
    blocks = tails + slices * nb;
    kernel = fmha_fwd_pipe_kernel<D, CAUSAL, false, true>;
  }
  if constexpr (!CAUSAL) {
    if (half_round_left(blocks, n, 2))
      kernel = tails_per_block ? fmha_fwd_pipe_kernel<D, CAUSAL, true, true> : fmha_fwd_pipe_kernel<D, CAUSAL, true, false>;
  }
  const hipError_t rc = launch(kernel, blocks, kPipeThreads, stream, (const half_t*)q,
                               (const half_t*)k, (const half_t*)v, qs, ks, vs, (half_t*)o, (float*)lse, head, n,
                               FmhaOrder(slices, nb, CAUSAL, !tails && n % kPipeBlockQ != 0), nb, tails, tails_per_block, c,
                               negate);
  return rc == hipSuccess ? FUSED_MHA_OK : FUSED_MHA_ERR_LAUNCH;
}

int dispatch_forward(const void* q, const fused_mha_strides* q_st, const void* k, const fused_mha_strides* k_st,
                     const void* v, const fused_mha_strides* v_st, void* o, void* lse, bool need_lse, int batch, int head,
                     int m, int n, int d, float scale, int causal, void* stream) {
  if (!q || !k || !v || !o || (need_lse && !lse)) return FUSED_MHA_ERR_NULL_POINTER;
  if (int rc = check_shape(batch, head, m, n, d)) return rc;
  if (!isfinite(scale)) return FUSED_MHA_ERR_BAD_SCALE;
  if (misaligned(q) || misaligned(k) || misaligned(v) || misaligned(o) || misaligned(lse))
    return FUSED_MHA_ERR_MISALIGNED;
  if (bad_strides(q_st) || bad_strides(k_st) || bad_strides(v_st)) return FUSED_MHA_ERR_BAD_STRIDE;
  hipStream_t s = (hipStream_t)stream;
  const Strides qs = to_strides(q_st, head, n, d), ks = to_strides(k_st, head, n, d), vs = to_strides(v_st, head, n, d);
#define FMHA_FWD(DD, CC) launch_forward<DD, CC>(q, k, v, qs, ks, vs, o, lse, batch, head, n, scale, s)
  if (d == 128) return causal ? FMHA_FWD(128, true) : FMHA_FWD(128, false);
  return causal ? FMHA_FWD(64, true) : FMHA_FWD(64, false);
#undef FMHA_FWD
}

enum BwdPass { kPassDelta = 1, kPassDq = 2, kPassDkDv = 4, kPassAll = 7, kNotBySlice = 8 /* by the passes in any case */ };

// Workspace of the backward: delta and lse * log2(e), fp32 (batch, head, n) each; then, for
// the spill path, at the next multiple of 256 bytes, the fp16 dS tiles
// (batch * head slices of np * np elements, np = n rounded up to 128).
size_t stats_bytes(int batch, int head, int n) { return 2 * (size_t)batch * head * n * sizeof(float); }
size_t spill_offset(int batch, int head, int n) { return (stats_bytes(batch, head, n) + 255) & ~(size_t)255; }
int padded_n(int n) { return (n + 127) & ~127; }
size_t slice_bytes(int n) { return (size_t)padded_n(n) * padded_n(n) * sizeof(half_t); }
int key_blocks(int n) { return (n + kKvBlockKeys - 1) / kKvBlockKeys; }
// Slices whose dS tiles a workspace has room for (of at most FUSED_MHA_SPILL_MAX_BYTES).
int spill_slices(int batch, int head, int n, size_t workspace_bytes) {
  const size_t offset = spill_offset(batch, head, n);
  if (workspace_bytes <= offset) return 0;
  size_t room = workspace_bytes - offset;
  if (room > FUSED_MHA_SPILL_MAX_BYTES) room = FUSED_MHA_SPILL_MAX_BYTES;
  const size_t fit = room / slice_bytes(n), all = (size_t)batch * head;
  return (int)(fit < all ? fit : all);
}
// Behind the dS of all slices: the counts of fmha_bwd_both_spill_kernel.
size_t ready_bytes(int slices) { return (size_t)slices * kReadyStride * sizeof(unsigned); }
// Whether rounds of that many slices keep the CUs busy: two key blocks for each.
bool rounds_fill(int slices, int n, int cus) { return (long)slices * key_blocks(n) >= 2L * cus; }
// The workspace of at most `room` bytes that the backward makes the best use of.  dS of all slices where that is at most
// FUSED_MHA_SPILL_MAX_BYTES.  Otherwise rounds of eight key blocks per CU or 4 GiB, whichever is more, if there is room:
// larger ones gain next to nothing.  Backward in ms, without dS / with the dS of rounds of so many GiB:
//   N32768 H16 causal     13.9 / 4: 13.6, 8: 12.1, 16: 11.6 (2, 4, 8 blocks per CU)
//   N20000 H32            20.9 / 3: 19.5, 6: 17.8, 7.5: 17.6, 16: 17.3
//   N8192 H256 causal     14.9 / 1: 13.3, 2: 12.6, 4: 12.6, 16: 12.8 (2, 4, 8, 32 blocks per CU)
//   N2048 H2100 causal     9.8 / 0.2: 9.3, 1: 8.7, 4: 8.7, 16: 8.6
//   N512 H33000 causal    16.6 / 0.1: 17.9, 0.5: 16.7, 1: 16.6, 2: 16.1, 16: 16.1
// Rounds of less than 1 GiB are not worth it (last line).  The size is that for the 256 CUs of an MI355X, whatever device
// is current.
size_t best_workspace(int batch, int head, int n, int d, size_t room) {
  constexpr size_t kGiB = (size_t)1 << 30;
  const size_t least = stats_bytes(batch, head, n), offset = spill_offset(batch, head, n), slice = slice_bytes(n);
  if (d == 64) return least;  // see fmha_bwd_dq_pipe_kernel
  const size_t all = (size_t)batch * head;
  size_t want = all;
  if (all * slice > FUSED_MHA_SPILL_MAX_BYTES) {
    const size_t blocks = (size_t)key_blocks(n);
    want = (8 * kCus + blocks - 1) / blocks;
    if (want * slice < 4 * kGiB) want = 4 * kGiB / slice;
    if (want * slice > FUSED_MHA_SPILL_MAX_BYTES) want = FUSED_MHA_SPILL_MAX_BYTES / slice;
  }
  const size_t fit = room > offset ? (room - offset) / slice : 0;
  if (fit < want) want = fit;
  const bool use = want == all || (want * slice >= kGiB && rounds_fill((int)want, n, kCus));
  return use ? offset + want * slice : least;
}

template <int D, bool CAUSAL>
int launch_backward(int passes, int slices_at_once, size_t workspace_bytes, unsigned ticks, const void* q, const void* k,
                    const void* v, const void* o, const void* d_o, Strides qs, Strides ks, Strides vs, Strides gs, const void* lse, float* delta,
                    void* dq, void* dk, void* dv, int batch, int head, int n, float scale, hipStream_t stream) {
  // slices_at_once: how many slices' dS the workspace holds, 0 for the passes that need none; ticks: the most that a block may
  // wait for another's dS, fmha_ds_wait_ticks if that is less
  if (D == 64) slices_at_once = 0;  // see fmha_bwd_dq_pipe_kernel
  // Rounds of so few slices that they leave CUs idle cost more than the GEMMs they save.
  const int cus = (int)persistent_grid(1 << 30);
  if (slices_at_once < batch * head && !rounds_fill(slices_at_once, n, cus)) slices_at_once = 0;
  const bool spill = slices_at_once > 0;
  int slice0 = 0, slices = batch * head;  // what the passes over dS are launched for
  // Without the spill and with all three passes asked for, the dQ pass produces delta and lse2 itself.
  const bool dq_makes_stats = !spill && (passes & kPassAll) == kPassAll;
  float* lse2 = delta + (long)batch * head * n;
  half_t* ds = spill ? (half_t*)((char*)delta + spill_offset(batch, head, n)) : nullptr;
  const int np = padded_n(n);
  const size_t ds_bytes = slice_bytes(n) * (spill ? slices_at_once : 0) / (CAUSAL ? 2 : 1);
  const size_t touched = ds_bytes + 6 * (size_t)slices_at_once * n * D * sizeof(half_t);
  const int stream_ds = fmha_ds_used_once(ds_bytes, touched, n, CAUSAL);
  // Both passes over dS in one launch, where the workspace has room for the counts behind the dS of all slices.
  unsigned* ready = nullptr;
  if constexpr (D == 128) {
    const size_t at = spill_offset(batch, head, n) + (size_t)slices * slice_bytes(n);
    if (spill && slices_at_once == slices && (passes & kPassAll) == kPassAll && workspace_bytes >= at + ready_bytes(slices) &&
        fmha_ds_in_one_launch(slices, n, cus, CAUSAL))
      ready = (unsigned*)((char*)delta + at);
  }
  auto delta_pass = [&]() {
    const unsigned rows = (unsigned)slices * n;              // fewer than 2^32 / (D / 8): check_shape
    const unsigned most = (1u << 23) * delta_rows(D);        // a launch of fewer than 2^32 threads: fewer than twice the blocks
    for (unsigned first = 0; first < rows; first += most) {
      const unsigned end = rows - first < most ? rows : first + most;
      const unsigned blocks = (end - first + delta_rows(D) - 1) / delta_rows(D);
      const unsigned per_slice = (unsigned)(n + delta_rows(D) - 1) / delta_rows(D);
      const unsigned chain = per_slice < blocks ? per_slice : blocks, chains = (blocks + chain - 1) / chain;
      const hipError_t rc = launch(fmha_bwd_delta_kernel<D>, chain * chains, 256, stream, (const half_t*)o, (const half_t*)d_o,
                                   gs, (const float*)lse, delta, lse2, head, n, (int)first, (int)end, (int)chain, (int)chains,
                                   ready, ready ? (unsigned)(ready_bytes(slices) / 4) : 0u);
      if (rc != hipSuccess) return rc;
    }
    return hipSuccess;
  };
  const float c = scale * kLog2e;
  const int nb = (n + 127) / 128;
  if ((passes & kPassAll) == kPassAll && !(passes & kNotBySlice) && fmha_backward_by_slice(D, n, slices, cus, CAUSAL)) {
    auto kernel = n <= 256 ? fmha_bwd_slice_kernel<D, 1, CAUSAL> : fmha_bwd_slice_kernel<D, D == 64 ? 2 : 1, CAUSAL>;
    const hipError_t rc = launch(kernel, (unsigned)slices, kSliceThreads, stream, (const half_t*)q, (const half_t*)k, (const half_t*)v,
                                 (const half_t*)o, (const half_t*)d_o, qs, ks, vs, gs, (const float*)lse, delta, lse2, (half_t*)dq,
                                 (half_t*)dk, (half_t*)dv, head, n, c, scale);
    return rc == hipSuccess ? FUSED_MHA_OK : FUSED_MHA_ERR_LAUNCH;
  }
  if ((passes & kPassAll) == kPassAll && fmha_passes_at_once(D, (long)nb * slices, n, cus, CAUSAL, spill)) {
    const bool stats = fmha_blocks_make_stats(D, n, CAUSAL);
    if (!stats && delta_pass() != hipSuccess) return FUSED_MHA_ERR_LAUNCH;
    auto both = [&](auto kernel, int threads) {
      return launch(kernel, 2u * nb * slices, threads, stream, (const half_t*)q, (const half_t*)k, (const half_t*)v,
                    (const half_t*)o, (const half_t*)d_o, qs, ks, vs, gs, (const float*)lse, delta, lse2, (half_t*)dq, (half_t*)dk,
                    (half_t*)dv, head, n, FmhaOrder(slices, nb, CAUSAL, n % 128 != 0, 2), nb, c, scale);
    };
    hipError_t rc;
    if constexpr (D == 64) {
      static_assert(kPipeBlockQ == 128 && kPipeBlockKeys == 128, "");
      rc = both(stats ? fmha_bwd_both_pipe_kernel<CAUSAL, true> : fmha_bwd_both_pipe_kernel<CAUSAL, false>, kPipeThreads);
    } else {
      static_assert(kDqBlockQ == 128 && kKvBlockKeys == 128, "");
      rc = both(stats ? fmha_bwd_both_kernel<CAUSAL, true> : fmha_bwd_both_kernel<CAUSAL, false>, kKvThreads);
    }
    return rc == hipSuccess ? FUSED_MHA_OK : FUSED_MHA_ERR_LAUNCH;
  }
  if ((passes & kPassDelta) && !dq_makes_stats && delta_pass() != hipSuccess) return FUSED_MHA_ERR_LAUNCH;
  auto wide = [&]() { return fmha_wide_mfmas((long)key_blocks(n) * slices, cus, CAUSAL); };
  auto dq_pass = [&]() {
    if constexpr (D == 64) {
      const int nmb = (n + kPipeBlockQ - 1) / kPipeBlockQ;
      auto pick = [&](auto odd_first) {
        constexpr bool kOddFirst = decltype(odd_first)::value != 0;
        return dq_makes_stats ? fmha_bwd_dq_pipe_kernel<CAUSAL, true, kOddFirst>
                              : fmha_bwd_dq_pipe_kernel<CAUSAL, false, kOddFirst>;
      };
      auto kernel = pick(IntTag<0>{});
      if constexpr (!CAUSAL)
        if (half_round_left((long)nmb * batch * head, n, 3)) kernel = pick(IntTag<1>{});
      return launch(kernel, (unsigned)nmb * batch * head, kPipeThreads, stream, (const half_t*)q, (const half_t*)k,
                    (const half_t*)v, (const half_t*)o, (const half_t*)d_o, qs, ks, vs, gs, (const float*)lse, delta, lse2,
                    (half_t*)dq, head, n, FmhaOrder(batch * head, nmb, CAUSAL, n % kPipeBlockQ != 0), nmb, c, scale);
    } else {
      if (spill) {
        // Two panels per block when that leaves every CU at least two blocks (a heavy and a light one).  The persistent
        // schedule only where its static shares come out even, otherwise one block per work group, heaviest first (B2 H40
        // N2048 causal, 2.5 blocks per CU: 116 -> 95 us).  Under causal masking nearly full pairs of rounds are not even
        // (forward and backward, us of the hardware's and of the persistent schedule, N x slices: 3072 x 42: 488, 516;
        // 4096 x 60: 1098, 1136; 8192 x 30: 2003, 2060), but up to N = 1024, where a block is a few us, they do as well (512
        // x 120: 81, 77; 1024 x 120: 208, 204; 768 x 80: 93, 92).  Even launches are within 1 % of each other (2048 x 64:
        // 335, 331; 4096 x 64: 1144, 1156; 8192 x 32: 2087, 2097; 16384 x 16: 3976, 3964).
        auto groups = [&](int blocks_per_slice) {
          const int total = blocks_per_slice * slices;
          const bool even = CAUSAL && n <= 1024 ? fmha_even_shares(slices, blocks_per_slice, 2 * cus, false)
                                                : fmha_even_shares(slices, blocks_per_slice, cus, CAUSAL);
          return even ? persistent_grid(total) : (unsigned)total;
        };
        const int nqb2 = (n + 2 * kDsPanelQ - 1) / (2 * kDsPanelQ), total2 = nqb2 * slices;
        if (total2 >= 2 * cus)  // so many blocks are never `wide`
          return launch(fmha_bwd_dq_spill_kernel<D, CAUSAL, 2, false>, groups(nqb2), ds_threads(2), stream, (const half_t*)k, ks,
                        (const half_t*)ds, np, (half_t*)dq, head, n, FmhaOrder(slices, nqb2, CAUSAL, false), slice0, stream_ds, scale);
        const int nqb = np / kDsPanelQ;
        auto kernel = wide() ? fmha_bwd_dq_spill_kernel<D, CAUSAL, 1, true> : fmha_bwd_dq_spill_kernel<D, CAUSAL, 1, false>;
        return launch(kernel, groups(nqb), ds_threads(1), stream, (const half_t*)k, ks,
                      (const half_t*)ds, np, (half_t*)dq, head, n, FmhaOrder(slices, nqb, CAUSAL, false), slice0, stream_ds, scale);
      }
      const int nmb = (n + kDqBlockQ - 1) / kDqBlockQ;
      auto kernel = dq_makes_stats ? fmha_bwd_dq_kernel<D, CAUSAL, true> : fmha_bwd_dq_kernel<D, CAUSAL, false>;
      return launch(kernel, (unsigned)nmb * batch * head, kDqThreads, stream, (const half_t*)q, (const half_t*)k,
                    (const half_t*)v, (const half_t*)o, (const half_t*)d_o, qs, ks, vs, gs, (const float*)lse, delta, lse2,
                    (half_t*)dq, head, n, nmb, batch * head, c, scale);
    }
  };
  auto dkdv_pass = [&]() {
    if constexpr (D == 64) {
      const int nnb = (n + kPipeBlockKeys - 1) / kPipeBlockKeys;
      auto kernel = fmha_bwd_dkdv_pipe_kernel<CAUSAL, false>;
      if constexpr (!CAUSAL)
        if (half_round_left((long)nnb * batch * head, n, 3)) kernel = fmha_bwd_dkdv_pipe_kernel<CAUSAL, true>;
      return launch(kernel, (unsigned)nnb * batch * head, kPipeThreads, stream,
                    (const half_t*)q, (const half_t*)k, (const half_t*)v, (const half_t*)d_o, qs, ks, vs, gs,
                    (const float*)delta, (const float*)lse2, (half_t*)dk, (half_t*)dv, head, n,
                    FmhaOrder(batch * head, nnb, CAUSAL, n % kPipeBlockKeys != 0), c, scale);
    } else {
      const int nnb = key_blocks(n);
      auto pick = [&](auto wide_tag) {
        constexpr bool kWide = decltype(wide_tag)::value != 0;
        return !spill ? fmha_bwd_dkdv_kernel<D, CAUSAL, false, false, kWide>
               : stream_ds ? fmha_bwd_dkdv_kernel<D, CAUSAL, true, false, kWide>
                           : fmha_bwd_dkdv_kernel<D, CAUSAL, true, true, kWide>;
      };
      auto kernel = wide() ? pick(IntTag<1>{}) : pick(IntTag<0>{});
      return launch(kernel, (unsigned)nnb * slices, kKvThreads, stream, (const half_t*)q, (const half_t*)k,
                    (const half_t*)v, (const half_t*)d_o, qs, ks, vs, gs, (const float*)delta, (const float*)lse2,
                    (half_t*)dk, (half_t*)dv, ds, np, head, n, FmhaOrder(slices, nnb, CAUSAL, n % kKvBlockKeys != 0), slice0, c,
                    scale);
    }
  };
  if constexpr (D == 128) {
    if (ready) {
      auto kernel = stream_ds ? fmha_bwd_both_spill_kernel<CAUSAL, false> : fmha_bwd_both_spill_kernel<CAUSAL, true>;
      const hipError_t rc = launch(kernel, (unsigned)fmha_ds_launch_blocks(slices, nb), kKvThreads, stream, (const half_t*)q,
                                   (const half_t*)k, (const half_t*)v, (const half_t*)d_o, qs, ks, vs, gs, (const float*)lse, delta, lse2,
                                   (half_t*)dq, (half_t*)dk, (half_t*)dv, ds, ready, np, head, n, FmhaOrder(slices, nb, CAUSAL, false), ticks, c,
                                   scale);
      return rc == hipSuccess ? FUSED_MHA_OK : FUSED_MHA_ERR_LAUNCH;
    }
  }
  // The spilling dK/dV pass feeds the dQ pass; otherwise the dQ pass (which may make the statistics) goes first.
  if (spill) {
    // as many slices at a time as the workspace holds dS of, in rounds of equal size
    const int rounds = (slices + slices_at_once - 1) / slices_at_once, all = slices;
    int per = (all + rounds - 1) / rounds;
    if (((per + 7) & ~7) <= slices_at_once) per = (per + 7) & ~7;  // whole slices per XCD
    for (slice0 = 0; slice0 < all; slice0 += per) {
      slices = all - slice0 < per ? all - slice0 : per;
      if ((passes & kPassDkDv) && dkdv_pass() != hipSuccess) return FUSED_MHA_ERR_LAUNCH;
      if ((passes & kPassDq) && dq_pass() != hipSuccess) return FUSED_MHA_ERR_LAUNCH;
    }
  } else {
    if ((passes & kPassDq) && dq_pass() != hipSuccess) return FUSED_MHA_ERR_LAUNCH;
    if ((passes & kPassDkDv) && dkdv_pass() != hipSuccess) return FUSED_MHA_ERR_LAUNCH;
  }
  return FUSED_MHA_OK;
}

int dispatch_backward(int passes, const void* q, const fused_mha_strides* q_st, const void* k,
                      const fused_mha_strides* k_st, const void* v, const fused_mha_strides* v_st, const void* o,
                      const void* d_o, const fused_mha_strides* g_st, const void* lse, void* workspace,
                      size_t workspace_bytes, void* dq, void* dk, void* dv, int batch, int head, int m, int n, int d,
                      float scale, int causal, void* stream, unsigned ticks = ~0u) {
  const bool need_o = passes & kPassDelta, need_dq = passes & kPassDq, need_dkdv = passes & kPassDkDv;
  if (!d_o || !workspace || !lse || (need_o && !o) || ((need_dq || need_dkdv) && (!q || !k || !v)) ||
      (need_dq && !dq) || (need_dkdv && (!dk || !dv)))
    return FUSED_MHA_ERR_NULL_POINTER;
  if (int rc = check_shape(batch, head, m, n, d)) return rc;
  if (!isfinite(scale)) return FUSED_MHA_ERR_BAD_SCALE;
  if (workspace_bytes < stats_bytes(batch, head, n)) return FUSED_MHA_ERR_BAD_SHAPE;
  // A workspace with room for dS tiles selects the spill path (5 GEMMs executed instead of 7; D = 128 only): with room
  // for some of the slices in rounds, which takes all passes in one call.
  int slices_at_once = spill_slices(batch, head, n, workspace_bytes);
  if (slices_at_once < batch * head && (passes & kPassAll) != kPassAll) slices_at_once = 0;
  if (misaligned(q) || misaligned(k) || misaligned(v) || misaligned(o) || misaligned(d_o) || misaligned(lse) ||
      misaligned(workspace) || misaligned(dq) || misaligned(dk) || misaligned(dv))
    return FUSED_MHA_ERR_MISALIGNED;
  if (bad_strides(q_st) || bad_strides(k_st) || bad_strides(v_st) || bad_strides(g_st)) return FUSED_MHA_ERR_BAD_STRIDE;
  hipStream_t s = (hipStream_t)stream;
  float* delta = (float*)workspace;
  const Strides qs = to_strides(q_st, head, n, d), ks = to_strides(k_st, head, n, d),
                vs = to_strides(v_st, head, n, d), gs = to_strides(g_st, head, n, d);
#define FMHA_BWD(DD, CC) \
  launch_backward<DD, CC>(passes, slices_at_once, workspace_bytes, ticks, q, k, v, o, d_o, qs, ks, vs, gs, lse, delta, dq, dk, \
                          dv, batch, head, n, scale, s)
  if (d == 128) return causal ? FMHA_BWD(128, true) : FMHA_BWD(128, false);
  return causal ? FMHA_BWD(64, true) : FMHA_BWD(64, false);
#undef FMHA_BWD
}

// Device address of `scratch` on the current device, looked up on the first call
// per device (each GPU holds its own copy of the array at its own address).
constexpr int kMaxDevices = 64;
int scratch_for_device(void** out) {
  static std::mutex mu;
  static void* ptrs[kMaxDevices] = {};
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return FUSED_MHA_ERR_RUNTIME;
  std::lock_guard<std::mutex> lock(mu);
  if (!ptrs[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return FUSED_MHA_ERR_RUNTIME;
    ptrs[dev] = p;
  }
  *out = ptrs[dev];
  return FUSED_MHA_OK;
}

}  // namespace

extern "C" {

int fused_mha_forward(const void* query_ptr, const void* key_ptr, const void* value_ptr, void* output_ptr,
                      void* lse_ptr, int batch, int head, int m, int n, int d, float scale, int causal,
                      void* stream) {
  return dispatch_forward(query_ptr, nullptr, key_ptr, nullptr, value_ptr, nullptr, output_ptr, lse_ptr, true, batch,
                          head, m, n, d, scale, causal, stream);
}

int fused_mha_forward_strided(const void* query_ptr, const fused_mha_strides* query_strides, const void* key_ptr,
                              const fused_mha_strides* key_strides, const void* value_ptr,
                              const fused_mha_strides* value_strides, void* output_ptr, void* lse_ptr, int batch,
                              int head, int n, int d, float scale, int causal, void* stream) {
  return dispatch_forward(query_ptr, query_strides, key_ptr, key_strides, value_ptr, value_strides, output_ptr,
                          lse_ptr, true, batch, head, n, n, d, scale, causal, stream);
}

int fmha_forward_without_lse(const void* query_ptr, const fused_mha_strides* query_strides, const void* key_ptr,
                             const fused_mha_strides* key_strides, const void* value_ptr,
                             const fused_mha_strides* value_strides, void* output_ptr, int batch, int head, int n, int d,
                             float scale, int causal, void* stream) {
  return dispatch_forward(query_ptr, query_strides, key_ptr, key_strides, value_ptr, value_strides, output_ptr, nullptr,
                          false, batch, head, n, n, d, scale, causal, stream);
}

size_t fused_mha_backward_min_workspace_bytes(int batch, int head, int n, int d) {
  if (check_shape(batch, head, n, n, d) != FUSED_MHA_OK) return 0;
  return stats_bytes(batch, head, n);
}

size_t fused_mha_backward_workspace_bytes(int batch, int head, int n, int d) {
  if (check_shape(batch, head, n, n, d) != FUSED_MHA_OK) return 0;
  return best_workspace(batch, head, n, d, SIZE_MAX);
}

size_t fmha_backward_workspace_within(int batch, int head, int n, int d, size_t room) {
  if (check_shape(batch, head, n, n, d) != FUSED_MHA_OK) return 0;
  return best_workspace(batch, head, n, d, room);
}

size_t fmha_backward_workspace_for(int batch, int head, int n, int d, int causal) {
  if (check_shape(batch, head, n, n, d) != FUSED_MHA_OK) return 0;
  if (d == 64) return stats_bytes(batch, head, n);  // whatever the launches: the device is not asked
  const int cus = (int)persistent_grid(1 << 30);
  if (fmha_backward_by_slice(d, n, batch * head, cus, causal != 0)) return stats_bytes(batch, head, n);
  if (fmha_passes_at_once(d, (long)key_blocks(n) * batch * head, n, cus, causal != 0)) return stats_bytes(batch, head, n);
  return best_workspace(batch, head, n, d, SIZE_MAX);
}

size_t fmha_backward_count_bytes(int batch, int head, int n, int d, int causal) {
  if (check_shape(batch, head, n, n, d) != FUSED_MHA_OK || d == 64) return 0;
  const int cus = (int)persistent_grid(1 << 30), slices = batch * head;
  if (fmha_backward_by_slice(d, n, slices, cus, causal != 0) ||
      fmha_passes_at_once(d, (long)key_blocks(n) * slices, n, cus, causal != 0) ||
      slices * slice_bytes(n) > FUSED_MHA_SPILL_MAX_BYTES || !fmha_ds_in_one_launch(slices, n, cus, causal != 0))
    return 0;
  return ready_bytes(slices);
}

int fmha_backward_waiting(const void* query_ptr, const void* key_ptr, const void* value_ptr, const void* output_ptr,
                          const void* d_output_ptr, const void* lse_ptr, void* workspace, size_t workspace_bytes,
                          void* d_query_ptr, void* d_key_ptr, void* d_value_ptr, int batch, int head, int n, int d, float scale,
                          int causal, unsigned ticks, void* stream) {
  return dispatch_backward(kPassAll | kNotBySlice, query_ptr, nullptr, key_ptr, nullptr, value_ptr, nullptr, output_ptr,
                           d_output_ptr, nullptr, lse_ptr, workspace, workspace_bytes, d_query_ptr, d_key_ptr, d_value_ptr,
                           batch, head, n, n, d, scale, causal, stream, ticks);
}

int fused_mha_backward(const void* query_ptr, const void* key_ptr, const void* value_ptr, const void* output_ptr,
                       const void* d_output_ptr, const void* lse_ptr, void* workspace, size_t workspace_bytes,
                       void* d_query_ptr, void* d_key_ptr, void* d_value_ptr, int batch, int head, int m, int n,
                       int d, float scale, int causal, void* stream) {
  return dispatch_backward(kPassAll, query_ptr, nullptr, key_ptr, nullptr, value_ptr, nullptr, output_ptr,
                           d_output_ptr, nullptr, lse_ptr, workspace, workspace_bytes, d_query_ptr, d_key_ptr,
                           d_value_ptr, batch, head, m, n, d, scale, causal, stream);
}

int fused_mha_backward_noalloc(const void* query_ptr, const void* key_ptr, const void* value_ptr,
                               const void* output_ptr, const void* d_output_ptr, const void* lse_ptr,
                               void* d_query_ptr, void* d_key_ptr, void* d_value_ptr, int batch, int head, int m,
                               int n, int d, float scale, int causal, void* stream) {
  if (int rc = check_shape(batch, head, m, n, d)) return rc;
  const size_t rows = (size_t)batch * head * n;
  if (rows > (size_t)FUSED_MHA_NOALLOC_MAX_ROWS) return FUSED_MHA_ERR_SCRATCH_LIMIT;
  void* ws = nullptr;
  if (int rc = scratch_for_device(&ws)) return rc;
  // Every workspace element that a pass reads is written before it by the same
  // call, by the dQ pass or the kernel for the statistics (rows 0 ..
  // batch*head*n-1 of both halves; launches whose blocks all make their own read
  // none), so nothing from an earlier call is ever read and nothing needs clearing.
  return dispatch_backward(kPassAll, query_ptr, nullptr, key_ptr, nullptr, value_ptr, nullptr, output_ptr,
                           d_output_ptr, nullptr, lse_ptr, ws, 2 * rows * sizeof(float), d_query_ptr, d_key_ptr,
                           d_value_ptr, batch, head, m, n, d, scale, causal, stream);
}

int fused_mha_backward_strided(const void* query_ptr, const fused_mha_strides* query_strides, const void* key_ptr,
                               const fused_mha_strides* key_strides, const void* value_ptr,
                               const fused_mha_strides* value_strides, const void* output_ptr,
                               const void* d_output_ptr, const fused_mha_strides* d_output_strides,
                               const void* lse_ptr, void* workspace, size_t workspace_bytes, void* d_query_ptr,
                               void* d_key_ptr, void* d_value_ptr, int batch, int head, int n, int d, float scale,
                               int causal, void* stream) {
  return dispatch_backward(kPassAll, query_ptr, query_strides, key_ptr, key_strides, value_ptr, value_strides,
                           output_ptr, d_output_ptr, d_output_strides, lse_ptr, workspace, workspace_bytes,
                           d_query_ptr, d_key_ptr, d_value_ptr, batch, head, n, n, d, scale, causal, stream);
}

int fused_mha_backward_delta(const void* output_ptr, const void* d_output_ptr, const void* lse_ptr, void* workspace,
                             size_t workspace_bytes, int batch, int head, int n, int d, void* stream) {
  return dispatch_backward(kPassDelta, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, output_ptr, d_output_ptr,
                           nullptr, lse_ptr, workspace, workspace_bytes, nullptr, nullptr, nullptr, batch, head, n, n,
                           d, 1.f, 0, stream);
}

int fused_mha_backward_dq(const void* query_ptr, const void* key_ptr, const void* value_ptr,
                          const void* d_output_ptr, const void* lse_ptr, void* workspace, size_t workspace_bytes,
                          void* d_query_ptr, int batch, int head, int n, int d, float scale, int causal,
                          void* stream) {
  return dispatch_backward(kPassDq, query_ptr, nullptr, key_ptr, nullptr, value_ptr, nullptr, nullptr, d_output_ptr,
                           nullptr, lse_ptr, workspace, workspace_bytes, d_query_ptr, nullptr, nullptr, batch, head, n,
                           n, d, scale, causal, stream);
}

int fused_mha_backward_dkdv(const void* query_ptr, const void* key_ptr, const void* value_ptr,
                            const void* d_output_ptr, const void* lse_ptr, void* workspace, size_t workspace_bytes,
                            void* d_key_ptr, void* d_value_ptr, int batch, int head, int n, int d, float scale,
                            int causal, void* stream) {
  return dispatch_backward(kPassDkDv, query_ptr, nullptr, key_ptr, nullptr, value_ptr, nullptr, nullptr, d_output_ptr,
                           nullptr, lse_ptr, workspace, workspace_bytes, nullptr, d_key_ptr, d_value_ptr, batch, head,
                           n, n, d, scale, causal, stream);
}

const char* fused_mha_error_string(int code) {
  switch (code) {
    case FUSED_MHA_OK: return "ok";
    case FUSED_MHA_ERR_NULL_POINTER: return "a required pointer is NULL";
    case FUSED_MHA_ERR_BAD_SHAPE: return "bad shape: need batch, head, n > 0, m == n and a large enough workspace";
    case FUSED_MHA_ERR_BAD_HEAD_DIM: return "head dimension must be 64 or 128";
    case FUSED_MHA_ERR_MISALIGNED: return "a pointer is not 16-byte aligned";
    case FUSED_MHA_ERR_LAUNCH: return "the HIP runtime refused a kernel launch";
    case FUSED_MHA_ERR_BAD_SCALE: return "scale must be finite";
    case FUSED_MHA_ERR_TOO_LARGE:
      return "problem too large: need n < 2^29, head * d < 2^24, ceil(n/128) * batch * head < 2^23 and "
             "batch * head * n * d / 8 < 2^32";
    case FUSED_MHA_ERR_BAD_STRIDE:
      return "strides must be non-negative multiples of 8 elements, sequence stride below 2^24, head stride below 2^31";
    case FUSED_MHA_ERR_SCRATCH_LIMIT:
      return "batch * head * n exceeds FUSED_MHA_NOALLOC_MAX_ROWS, the size of the static scratch";
    case FUSED_MHA_ERR_RUNTIME: return "a HIP runtime query failed (current device, scratch address)";
    default: return "unknown fused_mha error code";
  }
}

}  // extern "C"
