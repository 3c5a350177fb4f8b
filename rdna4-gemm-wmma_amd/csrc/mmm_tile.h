// Block tiles of the gfx950 matrix-core kernels and what every kernel on them shares: LDS layouts
// and swizzles, fragment reads, the MFMA issue order, the cross-stage K loop on direct-to-LDS
// loads, and C stores as whole 128-byte lines.  Used by the GEMM kernels (mmm_gemm.hip) and the
// folded contraction kernels (mmm_fold.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "mmm.h"
#include "mmm_dma.h"
#include "mmm_kernels.h"
#include "mmm_tile_map.h"

namespace mmm {

// Fragment offsets a wave keeps per K-step (A) or per B fragment: at most kMaxOff of each.
constexpr int kMaxOff = 8;

// Block tile BM x BN, K step BK (32 or 64), WGM x WGN waves, STAGES-deep LDS ring, OCC
// workgroups per CU targeted by the launch bounds (OCC > 1 caps registers accordingly), MFMA
// shape MF: 32 = v_mfma_f32_32x32x16_f16, 16 = v_mfma_f32_16x16x32_f16 (same MACs per LDS byte;
// a quarter of the accumulator bytes per instruction for half the MACs).
template <int BM_, int BN_, int WGM_, int WGN_, int BK_, int STAGES_, int OCC_ = 1, int MF_ = 32>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, BK = BK_, WGM = WGM_, WGN = WGN_, STAGES = STAGES_, OCC = OCC_;
  static constexpr int MF = MF_;
  static constexpr int NT = 64 * WGM * WGN;
  static constexpr int TM = BM / WGM, TN = BN / WGN;
  static constexpr int FM = TM / MF, FN = TN / MF;
  static constexpr int KK = MF == 32 ? 16 : 32;  // K per MFMA
  static constexpr int KSTEPS = BK / KK;         // MFMA K-steps per stage
  static constexpr int CA = BK / 8;       // 16-byte chunks per A row
  static constexpr int CB = BN / 8;       // 16-byte chunks per B row
  static constexpr int A_BYTES = BM * BK * 2, B_BYTES = BK * BN * 2;
  static constexpr int STAGE = A_BYTES + B_BYTES;
  static constexpr int RA = BM * CA / NT;  // A chunks per thread per stage
  static constexpr int RB = BK * CB / NT;  // B chunks per thread per stage
  static constexpr int LPT = RA + RB;      // direct-to-LDS loads per thread per stage
  // A-row swizzle (chunk c of row m stored at c ^ swz_a(m)).  32x32 fragments, rows of 128 B
  // (BK = 64): 8 consecutive rows take 8 distinct chunk slots and 16 consecutive rows 16
  // distinct 16-byte bank groups of the 256-byte bank window.  Rows of 64 B (BK = 32): four
  // rows share a 256-byte window, so the swizzle uses row bits 1..3.  Both are conflict-free
  // for the 32x32 fragment reads (measured).
  // 16x16 fragments (BK = 64): each ds_read_b128 reads 16 consecutive rows at four logical
  // chunks; row bits 1..3 as the chunk swizzle make it conflict-free (measured with
  // SQ_LDS_BANK_CONFLICT on MI355X: the 32x32 swizzle costs this pattern a 2-way conflict).
  static __device__ __forceinline__ int swz_a(int m) {
    if constexpr (MF == 16) return (m >> 1) & 7;
    else if constexpr (BK == 64) return (m & 7) ^ ((m >> 3) & 3);
    else return ((m >> 1) & 3) ^ ((m >> 3) & 1);
  }
  static constexpr int SWZ_A_ROWS = MF == 16 ? 16 : BK == 64 ? 32 : 16;  // swz_a depends on m % SWZ_A_ROWS
  // A fragment offsets per K-step: 16-row fragments alternate between two swizzle phases when
  // the swizzle spans 32 rows; fragment mb sits (mb / APAR) * AROWS rows past phase mb % APAR.
  static constexpr int APAR = (MF == 16 && SWZ_A_ROWS == 32) ? 2 : 1;
  static constexpr int AROWS = APAR * MF;
  // B-row swizzle (chunk c of row k stored at c ^ swz_bk(k)).  32x32 fragments: {0, 6, 10, 12}
  // by k % 4 (the 4 rows x 4 chunks that 32 lanes of one ds_read_b64_tr_b16 touch land in 16
  // distinct bank groups).  16x16 fragments: those 32 lanes read rows k .. k+3 and k+8 .. k+11
  // (2 chunks each), so rows with bit 3 set also flip chunk bit 1 ({2, 4, 8, 14}).
  static __device__ __forceinline__ int swz_bk(int k) {
    if constexpr (CB == 8 || CB == 24) {
      // Rows of 128 or 384 B (BN = 64, 192): rows k and k+1 start half a 256-byte bank window
      // apart, so {0, 0, 4, 4} by k % 4 puts rows k..k+3 on the four distinct 64-byte quarters
      // of their windows; 16x16 fragments read rows k and k+8 at the same two chunks, so bit 3
      // of k flips chunk bit 1 as for wider rows.  XOR values below 8 keep every chunk inside
      // its group of 8, so a 24-chunk row stays a permutation of itself.
      const int s = (k & 2) << 1;
      if constexpr (MF == 16) return s ^ (((k >> 3) & 1) << 1);
      else return s;
    }
    const int s = (0xCA60 >> (4 * (k & 3))) & 15;
    if constexpr (MF == 16) return s ^ (((k >> 3) & 1) << 1);
    else return s;
  }
  static constexpr int SWZ_B_ROWS = MF == 16 ? 16 : 4;  // swz_bk depends on k % SWZ_B_ROWS
  static_assert(MF == 32 || (MF == 16 && BK == 64), "MFMA shape (16x16 fragments with 64-deep stages)");
  static_assert(BK == 32 || BK == 64, "K step must be 32 or 64");
  static_assert(TM % 32 == 0 && (TN % 32 == 0 || (MF == 16 && TN % 16 == 0)),
                "wave tile must be a multiple of 32x32 (32 x 16 with 16x16 fragments)");
  static_assert(FN <= kMaxOff && KSTEPS * APAR <= kMaxOff, "fragment offsets per wave");
  static_assert(CB == 8 || CB == 24 || CB >= 16, "B swizzle: rows of 8 or 24 chunks or at least 16");
  // B staging: chunk slot s = r*NT + w*64 + lane of a stage's [BK][CB] chunk grid is row s / CB.
  // When CB divides 64, a wave's slots are whole rows and rows advance by NT / CB per r; if that
  // step is also a multiple of the rows the B swizzle depends on, the logical chunk is the same
  // for every r (one base offset plus a uniform step per r).  Otherwise (BN = 192; four waves
  // over 32-chunk rows, 8 rows per round against a 16-row swizzle) each r has its own row and chunk.
  static constexpr bool B_UNIFORM = 64 % CB == 0 && (NT / CB) % SWZ_B_ROWS == 0;
  static_assert((BM * CA) % NT == 0 && (BK * CB) % NT == 0, "chunks must divide evenly over threads");
  static_assert(STAGES >= 2 && OCC * STAGES * STAGE <= 160 * 1024, "LDS rings must fit the 160 KB LDS");
};

// B-row swizzle of the 32x32 layouts (chunk c of row k stored at c ^ swz_b(k)), {0, 6, 10, 12}
// by k % 4.
__device__ __forceinline__ int swz_b(int k) { return (0xCA60 >> (4 * (k & 3))) & 15; }

__device__ __forceinline__ half8 lds_read_a(const char LDS_AS* p) { return *(const half8 LDS_AS*)p; }

__device__ __forceinline__ half8 lds_read_b_tr(const char LDS_AS* p_lo, const char LDS_AS* p_hi) {
  fp16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4f16((fp16x4 LDS_AS*)p_lo);
  fp16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4f16((fp16x4 LDS_AS*)p_hi);
  half4 l4 = __builtin_bit_cast(half4, lo);
  half4 h4 = __builtin_bit_cast(half4, hi);
  return __builtin_shufflevector(l4, h4, 0, 1, 2, 3, 4, 5, 6, 7);
}

// Wait until at most n tiles of LPT loads each are still in flight (0 <= n <= NMAX; n is
// wave-uniform, the branch is scalar).
template <int LPT, int NMAX>
__device__ __forceinline__ void wait_tiles(int n) {
  static_assert(NMAX * LPT <= 63, "vmcnt range");
  if constexpr (NMAX == 0) {
    wait_vmcnt<0>();
  } else {
    if (n >= NMAX)
      wait_vmcnt<NMAX * LPT>();
    else
      wait_tiles<LPT, NMAX - 1>(n);
  }
}

// One pass over an LDS stage: KSTEPS K-steps of FM x FN MFMAs.  `after_first_reads` runs
// once the first K-step's fragment reads are issued (the DMA of a later stage goes there,
// so the MFMA pipe is fed before the loads are queued).
// BKM = false: B stage is [BK][BN] (N contiguous), fragments by two transposing reads;
//              b_off[nb] addresses fragment nb, K-steps add whole rows.
// BKM = true : B stage is [BN][BK] (K contiguous, swizzled like A), fragments by one
//              ds_read_b128; b_off[kk] addresses K-step kk, fragments add 32 rows.
// One K-step's MFMA operands for a wave: FM A fragments and FN B fragments.
template <class T>
struct Frags {
  half8 a[T::FM], b[T::FN];
};

// Accumulator of one MF x MF output block (C^T: lane l owns row m = l % MF).
template <class T>
using AccT = typename std::conditional<T::MF == 32, f32x16, f32x4>::type;

// Fragment read unit u of K-step kk: u < FM reads A fragment u; otherwise B fragment u - FM,
// by one ds_read_b128 from a K-major B stage (BKM) or two transposing reads from an
// N-contiguous one.  a_off[kk * APAR + phase]: A fragment offsets; b_off[nb] (N-contiguous
// B) or b_off[kk * APAR + phase] (K-major B, laid out and swizzled like A).
template <class T, bool BKM>
__device__ __forceinline__ void load_frag_unit(const char LDS_AS* a_st, const char LDS_AS* b_st,
                                               const uint32_t (&a_off)[kMaxOff], const uint32_t (&b_off)[kMaxOff], int kk, int u,
                                               Frags<T>& f) {
  if (u < T::FM) {
    f.a[u] = lds_read_a(a_st + a_off[kk * T::APAR + u % T::APAR] + (u / T::APAR) * T::AROWS * T::BK * 2);
  } else {
    const int nb = u - T::FM;
    if constexpr (BKM)
      f.b[nb] = lds_read_a(b_st + b_off[kk * T::APAR + nb % T::APAR] + (nb / T::APAR) * T::AROWS * T::BK * 2);
    else
      f.b[nb] = lds_read_b_tr(b_st + b_off[nb] + (kk * T::KK) * T::BN * 2,
                              b_st + b_off[nb] + (kk * T::KK + 4) * T::BN * 2);
  }
}

// All fragment reads of K-step kk from an LDS stage.
template <class T, bool BKM>
__device__ __forceinline__ void load_frags(const char LDS_AS* a_st, const char LDS_AS* b_st, const uint32_t (&a_off)[kMaxOff],
                                           const uint32_t (&b_off)[kMaxOff], int kk, Frags<T>& f) {
#pragma unroll
  for (int u = 0; u < T::FM + T::FN; ++u) load_frag_unit<T, BKM>(a_st, b_st, a_off, b_off, kk, u, f);
}

// One MFMA of the tile's shape, operands swapped (B fragment as src A): acc holds C^T.
template <class T>
__device__ __forceinline__ void mfma_one(const half8& b, const half8& a, AccT<T>& acc) {
  if constexpr (T::MF == 32)
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(b, a, acc, 0, 0, 0);
  else
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(b, a, acc, 0, 0, 0);
}

// Issue order of a K-step's FM x FN MFMAs: MFMA i updates accumulator (ord_mb(i), ord_nb(i)),
// row by row with the column order reversed on every other row (a snake), so consecutive MFMAs
// share an operand at the turns too.  Each accumulator still sees its K-steps in order, so the
// order does not change any result.  Under sustained load the MI355X runs at its power cap, and
// fewer operand changes between consecutive MFMAs cost less power: at 8192^3 (interleaved runs,
// bit-identical results) the snake ran 1363 TFLOP/s against 1354 for plain row-major or
// column-major order and 1359 for a column snake.
template <class T>
__host__ __device__ constexpr int ord_mb(int i) {
  return i / T::FN;
}
template <class T>
__host__ __device__ constexpr int ord_nb(int i) {
  return ((i / T::FN) & 1) ? T::FN - 1 - i % T::FN : i % T::FN;
}

template <class T>
__device__ __forceinline__ void mfma_frags(const Frags<T>& f, AccT<T> (&acc)[T::FM][T::FN]) {
#pragma unroll
  for (int i = 0; i < T::FM * T::FN; ++i) {
    mfma_one<T>(f.b[ord_nb<T>(i)], f.a[ord_mb<T>(i)], acc[ord_mb<T>(i)][ord_nb<T>(i)]);
  }
}

template <class T, bool BKM, class Hook>
__device__ __forceinline__ void compute_stage(const char LDS_AS* a_st, const char LDS_AS* b_st,
                                              const uint32_t (&a_off)[kMaxOff], const uint32_t (&b_off)[kMaxOff],
                                              AccT<T> (&acc)[T::FM][T::FN], Hook&& after_first_reads) {
  using Frags = mmm::Frags<T>;
  auto load = [&](int kk, Frags& f) { load_frags<T, BKM>(a_st, b_st, a_off, b_off, kk, f); };
  auto mfma = [&](const Frags& f) { mfma_frags<T>(f, acc); };
#pragma unroll
  for (int kk = 0; kk < T::KSTEPS; ++kk) {
    Frags f;
    load(kk, f);
    if (kk == 0) after_first_reads();
    mfma(f);
  }
}

__device__ __forceinline__ void block_sync() { __syncthreads(); }

// ---- C stores as whole 128-byte lines (16x16x32 tiles).  A 16x16 accumulator block gives lane l
// row l % 16 and columns 4*(l/16) .. +3, so one float4 store of a block writes 16 rows x 64
// bytes: half lines.  Blocks nb and nb+1 of a row of blocks cover 32 columns; lanes l and l ^ 8
// (rows r and r + 8) trade their block-(nb+1) values (one DPP move per register), after which
// one store writes rows 0-7 and the next rows 8-15, each row 32 columns: one 128-byte line (the
// 192x192 tile's odd third block of a row stays half lines).  gemm_nn_kernel stores its interior
// tiles this way with every store policy; the persistent kernels with non-temporal stores only.
// Measured on MI355X (interleaved runs,
// same box, exact results), against half lines: 8192^3 +0.6-0.9%, 12288^2 x 4096 +1.4%,
// 16384^2 x 4096 +1.0%, 8192 x 2048 x 2048 +1.4%, 4096^3 +0.8%, 6144^3 +0.4%; with plain
// (L2-allocating) stores the persistent grids lost up to 2% at short K (8192^2 x 2048 -1.6%,
// 16384 x 8192 x 1024 -2.0%).
enum CStore { kStorePlain = 0, kStoreNonTemporal = 1, kStoreWriteThrough = 2 };

// System-scope write-through 16-byte store (sc0 sc1), as inline asm.  The compiler does not see
// a store in inline asm, so it does not add the wait states a VALU write of the store's data
// registers needs after a VMEM store of more than 8 bytes (2 on gfx950); the s_nop supplies them.
// Without it the next VALU write could replace the data before the store read it (seen as
// wrong C values when the epilogue reused the registers at once).
#define WT_STORE_X4 "global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1"

template <int POLICY>
__device__ __forceinline__ void store_c4(float* dst, f32x4 v) {
  if constexpr (POLICY == kStoreNonTemporal)
    __builtin_nontemporal_store(v, (f32x4*)dst);
  else if constexpr (POLICY == kStoreWriteThrough)
    asm volatile(WT_STORE_X4 ::"v"(dst), "v"(v) : "memory");
  else
    *(f32x4*)dst = v;
}

// Lane l's result is lane (l ^ 8)'s x (DPP row_ror:8 within each 16-lane row).  Called
// unconditionally: a cross-lane move inside one arm of a lane-dependent ?: runs with the other
// lanes switched off and reads nothing from them.  Written per element: a loop over a vector's
// elements here compiled to one DPP move reused for all four.
__device__ __forceinline__ float from_lane_xor8(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x128, 0xf, 0xf, false));
}
__device__ __forceinline__ f32x4 from_lane_xor8(f32x4 v) {
  return f32x4{from_lane_xor8(v.x), from_lane_xor8(v.y), from_lane_xor8(v.z), from_lane_xor8(v.w)};
}

// The lane index read afresh (v_mbcnt in asm, which the compiler cannot hoist out of a loop):
// values derived from it are rebuilt where they are used instead of being kept live.
__device__ __forceinline__ int lane_id_fresh() {
  int lane;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
  return lane;
}

template <class T>
constexpr bool c_lines_ok() {
  return T::MF == 16 && T::FN >= 2;
}
// every store of the tile a whole line (an even number of blocks per row)
template <class T>
constexpr bool c_lines_all() {
  return c_lines_ok<T>() && T::FN % 2 == 0;
}
template <class T, int POLICY>
constexpr bool use_c_lines() {
  return c_lines_ok<T>() && POLICY != kStorePlain;
}

// The wave's whole TM x TN accumulator tile to C at `c` (the wave tile's first element; rows
// ldc floats apart), every 32-column pair of blocks as 16 row lines (an odd last block as half
// lines).  The lane's row and column offsets are built here from a fresh lane index: kept from
// before a persistent kernel's tile loop they would stay live across its K loop, which runs at
// the register limit (they spilled).
// LIMIT: only the 16-row blocks that start below `rows`.
template <class T, int POLICY, bool LIMIT = false>
__device__ __forceinline__ void store_wave_tile_lines(float* c, int64_t ldc, const AccT<T> (&acc)[T::FM][T::FN],
                                                      int rows = 0) {
  static_assert(c_lines_ok<T>(), "16x16 blocks, at least two per row");
  const int lane = lane_id_fresh();
  const bool lo = (lane & 8) == 0;
  float* r0 = c + (int64_t)(lane & 7) * ldc + 4 * (lane >> 4) + (lo ? 0 : 16);        // rows 0-7
  float* r1 = c + (int64_t)((lane & 7) + 8) * ldc + 4 * (lane >> 4) + (lo ? 16 : 0);  // rows 8-15
#pragma unroll
  for (int mb = 0; mb < T::FM; ++mb) {
    if (LIMIT && 16 * mb >= rows) break;
#pragma unroll
    for (int nb = 0; nb + 1 < T::FN; nb += 2) {
      // rows 0-7: lanes 0-7 keep block nb, lanes 8-15 take block nb + 1 of lanes 0-7;
      // rows 8-15: lanes 8-15 keep block nb, lanes 0-7 take block nb + 1 of lanes 8-15
      const f32x4 traded = from_lane_xor8(acc[mb][nb + 1]);
      const f32x4 rows_lo = lo ? acc[mb][nb] : traded, rows_hi = lo ? traded : acc[mb][nb];
      store_c4<POLICY>(r0 + (int64_t)16 * mb * ldc + 16 * nb, rows_lo);
      store_c4<POLICY>(r1 + (int64_t)16 * mb * ldc + 16 * nb, rows_hi);
      __builtin_amdgcn_sched_barrier(0);  // one pair at a time: the traded values stay few
    }
    if constexpr (T::FN % 2 != 0)  // the odd last block: lane l's row l % 16, 16 rows x 64 bytes
      store_c4<POLICY>(c + (int64_t)(16 * mb + (lane & 15)) * ldc + 16 * (T::FN - 1) + 4 * (lane >> 4),
                       acc[mb][T::FN - 1]);
  }
}

// Most K ranges of any split (the planners' limit).
constexpr int kMaxSplits = 16;

// src[0] + src[stride] + ... over `splits` (uniform, 1 .. kMaxSplits) partial sums, in that order.  Every
// load is issued before the first addition, so a reduction costs one memory round trip, not one per
// K range: with a load per iteration of a run-time loop, 64 x 512 x 8192 in 16 ranges ran 14.4 us
// against 11.0, 100 x 200 x 8192 12.8 against 10.5, 256 x 1024 x 16384 25.1 against 22.7.
__device__ __forceinline__ f32x4 sum_splits(const f32x4* src, int64_t stride, int splits) {
  f32x4 v[kMaxSplits];
#pragma unroll
  for (int q = 0; q < kMaxSplits; ++q)
    if (q < splits) v[q] = src[q * stride];
  f32x4 sum = v[0];
#pragma unroll
  for (int q = 1; q < kMaxSplits; ++q)
    if (q < splits) sum += v[q];
  return sum;
}

// Measurement: thread 0 of workgroup 0 writes the shader-clock counter (s_memtime) and the 100 MHz
// real-time counter (s_memrealtime) to clk[at], clk[at + 1] when the caller asked for them.
__device__ __forceinline__ void record_clock(uint64_t* clk, int at) {
  if (clk != nullptr && blockIdx.x == 0 && threadIdx.x == 0) {
    clk[at] = __builtin_amdgcn_s_memtime();
    clk[at + 1] = __builtin_amdgcn_s_memrealtime();
  }
}

// K-steps 0 .. KSTEPS-2 of the K tile in LDS stage `st`: each step's MFMAs (fragments f[kk & 1])
// run while the next step's fragments are read into f[(kk + 1) & 1]; MFMA i carries fragment
// read i, and scheduling fences keep that order.
template <class T, bool BKM>
__device__ __forceinline__ void ktile_body(const char LDS_AS* st, const uint32_t (&a_off)[kMaxOff],
                                           const uint32_t (&b_off)[kMaxOff], Frags<T> (&f)[2],
                                           AccT<T> (&acc)[T::FM][T::FN]) {
#pragma unroll
  for (int kk = 0; kk + 1 < T::KSTEPS; ++kk) {
#pragma unroll
    for (int i = 0; i < T::FM * T::FN; ++i) {
      mfma_one<T>(f[kk & 1].b[ord_nb<T>(i)], f[kk & 1].a[ord_mb<T>(i)], acc[ord_mb<T>(i)][ord_nb<T>(i)]);
      if (i < T::FM + T::FN) load_frag_unit<T, BKM>(st, st + T::A_BYTES, a_off, b_off, kk + 1, i, f[(kk + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// The last K-step of a K tile, after the barrier that publishes the next one in stage `ns`: its
// MFMAs (fragments f[1]) carry the next stage's first fragment reads (into f[0], MFMA i carrying
// read i) and the LPT refill loads dma_one(d, 0 .. LPT-1), spread evenly over the MFMAs after the
// reads when there are enough of them (every load is a 1 KB request to the address unit, and all
// waves refill in the same K-step, so a burst of them fills its queue and stalls each wave's
// MFMAs behind its next load).  Measured on the 256x256 tile (32 MFMAs, 8 loads) at 8192^3: one
// load every MFMA 1258 TFLOP/s, every 2 within 1%, every 3 +1%, every 4 (the even spread) +4.4%.
template <class T, bool BKM, class D, class DmaOne>
__device__ __forceinline__ void ktile_last_step(const char LDS_AS* ns, const uint32_t (&a_off)[kMaxOff],
                                                const uint32_t (&b_off)[kMaxOff], Frags<T> (&f)[2],
                                                AccT<T> (&acc)[T::FM][T::FN], const D& d, DmaOne&& dma_one) {
  constexpr int NM = T::FM * T::FN, NU = T::FM + T::FN;
  constexpr int NL = T::LPT;
  constexpr int DS = NM / NL > 1 ? NM / NL : 1;  // MFMAs between loads
  constexpr int D0 = NM - DS * NL >= NU ? NU : (NM > DS * NL ? NM - DS * NL : 0);
  int issued = 0;
#pragma unroll
  for (int i = 0; i < NM; ++i) {
    const int mb = ord_mb<T>(i), nb = ord_nb<T>(i);
    mfma_one<T>(f[1].b[nb], f[1].a[mb], acc[mb][nb]);
    if (i < NU) load_frag_unit<T, BKM>(ns, ns + T::A_BYTES, a_off, b_off, 0, i, f[0]);
    if (i >= D0 && (i - D0) % DS == 0 && issued < NL) dma_one(d, issued++);
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int j = 0; j < NL; ++j)
    if (j >= issued) dma_one(d, j);
}

// Cross-stage K loop over KT K tiles (the direct-to-LDS kernels).  The caller supplies the
// loads: prep(t, slot) builds the per-tile load state of K tile t for ring slot `slot` (and
// advances any running state: tiles are prepared in order), dma_one(d, j) issues load j of
// T::LPT, and issue_tile(t, slot) fills slot `slot` with tile t by whatever means (the last
// tile of an unaligned problem is gathered through VGPRs when tail_regs is set, which leaves
// no loads in flight for it).
//
// pre = 0: the loop issues the first tiles itself.  pre = 1: the caller has issued tiles
// 0 .. S-1 already (KT >= S).  pre = 2: as 1, and NST further vector-memory operations (the
// previous tile's C stores) were issued after them; the first wait lets those stay
// outstanding (vmcnt retires in issue order).
//
// first_wait() runs once tile 0 has landed, before the barrier that publishes it;
// tail_patch(slot) runs once this wave's loads of the last tile (in ring slot `slot`) have
// landed, before the barrier that publishes it: a thread may overwrite the chunks its own
// loads put there.  tile_patch(t, slot) is the same for every tile t, called before tail_patch.
// tile_done(t) runs when the MFMAs of tile t (not the last) have been issued; half_done() before the
// last K-step of each tile of a loop of at most S + 1 tiles, and of the last S + 1 of a longer one.
struct NoHook {
  __device__ __forceinline__ void operator()() const {}
};
struct NoSlotHook {
  __device__ __forceinline__ void operator()(int) const {}
  __device__ __forceinline__ void operator()(int, int) const {}
};

template <class T, bool BKM, int NST = 0, class Prep, class DmaOne, class IssueTile, class FirstWait = NoHook,
          class TailPatch = NoSlotHook, class TilePatch = NoSlotHook, class TileDone = NoSlotHook,
          class HalfDone = NoHook>
__device__ __forceinline__ void cross_stage(char LDS_AS* lds_base, int KT, bool tail_regs, const uint32_t (&a_off)[kMaxOff],
                                            const uint32_t (&b_off)[kMaxOff], AccT<T> (&acc)[T::FM][T::FN], Prep&& prep,
                                            DmaOne&& dma_one, IssueTile&& issue_tile, int pre = 0,
                                            FirstWait&& first_wait = FirstWait{}, TailPatch&& tail_patch = TailPatch{},
                                            TilePatch&& tile_patch = TilePatch{},
                                            TileDone&& tile_done = TileDone{}, HalfDone&& half_done = HalfDone{}) {
  // Ring of S slots, tile u in slot u % S.  Cross-stage pipeline: during the last K-step of
  // tile t, this wave waits for its own loads of tile t+1, then the barrier (a) publishes
  // tile t+1 -- every wave's loads of it have landed -- and (b) retires slot t % S: every
  // wave has completed its reads of tile t, since a barrier waits for outstanding LDS reads
  // and tile t's last fragments were read before it.  After the barrier the wave reads
  // tile t+1's first fragments and refills slot t % S with tile t+S, and only then issues
  // tile t's last MFMAs, which cover the barrier and the first reads' latency.
  constexpr int S = T::STAGES;
  static_assert(T::KSTEPS % 2 == 0, "fragment double buffer alternates per K-step");
  const int first = KT < S ? KT : S;
  if (pre == 0)
    for (int s = 0; s < first; ++s) issue_tile(s, s);
  // tile 0 must land; later tiles may stay in flight (a gathered last tile has no loads)
  if (pre == 2) {
    static_assert((S - 1) * T::LPT + NST <= 63, "vmcnt range");
    wait_vmcnt<(S - 1) * T::LPT + NST>();
  } else {
    wait_tiles<T::LPT, S - 1>(first - 1 - ((tail_regs && first == KT) ? 1 : 0));
  }
  first_wait();
  tile_patch(0, 0);
  if (KT == 1) tail_patch(0);
  block_sync();
  Frags<T> f[2];
  load_frags<T, BKM>(lds_base, lds_base + T::A_BYTES, a_off, b_off, 0, f[0]);
  int cur = 0;
  // K-steps 0 .. KSTEPS-2 of the tile in slot `cur` (each step's MFMAs run while the next
  // step's fragments are read).
  auto tile_body = [&] { ktile_body<T, BKM>(lds_base + cur * T::STAGE, a_off, b_off, f, acc); };
  // Last K-step of tile t < KT-1: publish tile t+1, read its first fragments, refill the
  // retired slot (`refill` loads tile t+S into slot `cur`), then the MFMAs.
  auto tile_next = [&](int t, auto&& refill) {
    __builtin_amdgcn_sched_barrier(0);  // the body's MFMAs stay ahead of the waits
    const int issued = t + S < KT ? t + S : KT;  // tiles 0 .. issued-1 are issued
    int ahead = issued - (t + 2);                // of those, after t+1 (may stay in flight)
    if (tail_regs && issued == KT && ahead > 0) --ahead;
    wait_tiles<T::LPT, (S > 2 ? S - 2 : 0)>(ahead);
    const int nslot = cur + 1 == S ? 0 : cur + 1;
    tile_patch(t + 1, nslot);
    if (t + 1 == KT - 1) tail_patch(nslot);
    block_sync();
    const char LDS_AS* ns = lds_base + nslot * T::STAGE;
    load_frags<T, BKM>(ns, ns + T::A_BYTES, a_off, b_off, 0, f[0]);
    refill();
    mfma_frags<T>(f[1], acc);
    cur = nslot;
  };
  // Steady state: after the barrier the next tile's first fragment reads and the refill's
  // loads are interleaved with the last K-step's MFMAs (ktile_last_step), so neither a burst of
  // LDS reads nor a burst of load issue leaves the matrix pipe idle.
  auto tile_next_interleaved = [&](int t) {
    __builtin_amdgcn_sched_barrier(0);  // the body's MFMAs stay ahead of the waits
    wait_tiles<T::LPT, (S > 2 ? S - 2 : 0)>(S - 2);  // steady state: S-2 tiles after t+1 in flight
    const int nslot = cur + 1 == S ? 0 : cur + 1;
    tile_patch(t + 1, nslot);
    block_sync();
    ktile_last_step<T, BKM>(lds_base + nslot * T::STAGE, a_off, b_off, f, acc, prep(t + S, cur), dma_one);
    cur = nslot;
  };
  // steady state refills by DMA only; the refill of the last tile (possibly gathered
  // through VGPRs) is peeled so the loop carries no gather registers
  int t = 0;
  for (; t + S < KT - 1; ++t) {
    tile_body();
    tile_next_interleaved(t);
    tile_done(t);
  }
  if (t + S == KT - 1) {
    tile_body();
    half_done();
    tile_next(t, [&] { issue_tile(t + S, cur); });
    tile_done(t);
    ++t;
  }
  for (; t + 1 < KT; ++t) {
    tile_body();
    half_done();
    tile_next(t, [] {});
    tile_done(t);
  }
  tile_body();
  half_done();
  mfma_frags<T>(f[1], acc);
}

// Launch bounds: the 64x64 tile declares the three workgroups per CU its LDS ring allows.  With
// one, the compiler kept that tile's accumulators in AGPRs and copied them to and from VGPRs
// every K tile of the instantiation without the tail code (20 copies per 8 MFMAs; 1024^2 x 2048
// ran 14.7 against 14.1 us); with three it keeps them in VGPRs.
template <class T>
constexpr int nn_launch_occupancy() {
  return T::BM == 64 && T::BN == 64 ? 3 : T::OCC;
}

// Shortest K for which the multi-round kernels store C non-temporally in half lines (see their
// launches).
constexpr int kNtMinK = 4096;

// Direct-to-LDS path: K step, ring depth and wave grid (compile-time).  Measured on MI355X
// at 8192^3 (median TFLOP/s): 64 x 2 stages with 2 x 4 waves (two waves per SIMD, so one
// wave's MFMAs cover the other's barrier and LDS waits) 1126; the same with 2 x 2 waves
// 1077; 32 x 4 or 32 x 5 stages 1055-1106 -- deeper prefetch does not pay, latency of the
// operand fetch is not the limiter.  MFMA shape of the 256x256 tile: 16x16x32 (measured at
// 8192^3 under sustained load, it runs at a 16% higher power-limited clock than 32x32x16 -- a
// quarter of the accumulator traffic per instruction -- and is 2-9% faster across 4096^3 ..
// 16384^2 x 4096).
constexpr int kDmaBK = 64;
using Tile256 = Tile<256, 256, 2, 4, kDmaBK, 2, 1, 16>;
// The 128-wide tiles run eight 16x16x32 waves (two per SIMD) like the 256x256 tile.  Measured on
// MI355X against the four-wave 32x32x16 versions they replace (interleaved runs, same box):
//   128x256 (2 x 4 waves of 64x64, 3 x 48 KB ring): 2048 x 4096 x 4096 858 -> 939 TFLOP/s,
//     8192 x 1024 x 8192 1022 -> 1136, 1024 x 8192 x 8192 1030 -> 1145, 4096^3 1063 -> 1106,
//     8192^3 1120 -> 1136, 3072^3 830 -> 827;
//   256x128 (4 x 2 waves of 64x64, 3 x 48 KB ring): 2048 x 4096 x 4096 926 -> 1039,
//     8192 x 1024 x 8192 1023 -> 1160, 4096^3 1008 -> 1109, 8192^3 1034 -> 1137;
//   128x128 in multi-round grids (2 x 4 waves of 64x32, 2 x 32 KB ring, two workgroups per CU):
//     4096^3 971 -> 1007, 6144^2 x 2048 918 -> 952, 8192^3 1032 -> 1048, 3072^3 738 -> 764.
// With four waves a one-round launch holds one wave per SIMD, and nothing covers a wave's
// barrier and LDS waits.
template <int BM, int BN>
struct DmaCfg {  // 128x128
  using T = Tile<BM, BN, 2, 4, 64, 2, 2, 16>;
};
// 64x64: for grids too small to fill the chip with 128x128 tiles (1024^3 is 64 of those, 256
// of these).  Four waves of 32x32 (2 x 2 16x16x32 fragments each) on a 3-stage ring (48 KB).
// Measured on MI355X against the 128x128 tile (interleaved runs, same box): 1024^3 139 -> 200
// TFLOP/s, 512^3 23.8 -> 30.4, 768^3 67 -> 96, 1024^2 x 2048 207 -> 297; it loses where 128x128
// tiles fill a round or split well (1536^3 333 vs 365, 2048^3 515 vs 640).  8 stages (K = 512
// in flight at once) ran 3-7% slower than 3 or 4; two workgroups per CU at 2 stages, slower still.
template <>
struct DmaCfg<64, 64> {
  using T = Tile<64, 64, 2, 2, 64, 3, 1, 16>;
};
// 192x192: 16 x 16 tiles fill one round exactly at 3072 x 3072, where 256x256 tiles leave 112
// of the 256 CUs idle, and whole multiples of 256 tiles run as the persistent grid (6144^2 x
// 2048: 1024 tiles, four rounds, 1006 -> 1047 TFLOP/s over one workgroup per tile, against 926
// for 256x256 tiles' 2.25 rounds; 3072 x 6144 x 2048 996 -> 1030, against 888).  Eight waves of
// 96x48 (6 x 3 16x16x32 fragments), a 3-stage ring of 48 KB stages; rows of 24 chunks use the
// per-slot B staging map.  Measured on MI355X (interleaved runs, same box): 3072^3 763 -> 1007
// TFLOP/s against the 256x256 tile, 3072^2 x 8192 963 -> 1159, 4357 x 4095 x 4111 805 -> 885;
// 8192^3 1172 against 1380 (per-CU rate 0.85).
template <>
struct DmaCfg<192, 192> {
  using T = Tile<192, 192, 2, 4, 64, 3, 1, 16>;
};
template <>
struct DmaCfg<256, 256> {
  using T = Tile256;
};
template <>
struct DmaCfg<256, 128> {
  using T = Tile<256, 128, 4, 2, 64, 3, 1, 16>;
};
template <>
struct DmaCfg<128, 256> {
  using T = Tile<128, 256, 2, 4, 64, 3, 1, 16>;
};
template <int BM, int BN>
using DmaTile = typename DmaCfg<BM, BN>::T;
// The 128x128 tile in a launch of at most one round (one workgroup per CU): no second
// workgroup on the CU covers the load latency, so the ring is one stage deeper (3 x 32 KB).
// Measured on MI355X (interleaved runs, same box), first with four waves: 2048^3 567 -> 624
// TFLOP/s, 2048^2 x 4096 720 -> 791, 1024^2 x 8192 (K split) 508 -> 540, 4 stages no better
// than 3; then eight waves of 16x16x32 instead of four of 32x32x16: 2048^3 601 -> 645, 2048^2 x
// 4096 760 -> 822, 1024^2 x 8192 538 -> 564, 512 x 8192 x 8192 783 -> 852.
using DeepTile128 = Tile<128, 128, 2, 4, 64, 3, 1, 16>;
// Register-staged path: 64-deep stages, double-buffered.
template <int BM, int BN>
using RegTile = Tile<BM, BN, 2, 2, 64, 2>;

}  // namespace mmm
