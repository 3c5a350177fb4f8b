// MI355X (gfx950, CDNA4, wave64) FP16->FP32 GEMM kernels.
//
// Computes C[M][N] = A[M][K] * B[K][N] (fp16 in, fp32 accumulate and out, row-major), the
// operation of the reference's templated WMMA lineage (mmm.cpp:694-1374; definition at
// mmm.cpp:52-62).  The design is CDNA4's own, not a translation of the RDNA4 kernel:
//
//  * Math: v_mfma_f32_32x32x16_f16 (one wave, 32x32 outputs, K 16 per instruction).  The
//    MFMA operands are issued swapped (B fragment as src A, A fragment as src B), so the
//    accumulator holds C^T: lane l owns row m = l%32 and, for accumulator v, column
//    n = 8*(v/4) + 4*(l/32) + v%4 -- four consecutive columns per lane, stored as float4.
//  * Block tile BM x BN with K step 64, WGM x WGN waves, each wave (BM/WGM) x (BN/WGN).
//    The default 256x256 tile with 2x2 waves gives every wave 4x4 MFMA tiles (256 fp32
//    accumulators, held in AGPRs), i.e. 32 MACs per LDS byte read -- twice what the
//    MFMA rate needs from LDS.
//  * Operand staging: HBM -> LDS by buffer_load_dwordx4 ... lds (direct to LDS, no VGPR
//    round trip), double-buffered (2 x 64 KB of the 160 KB LDS).  Out-of-range rows and
//    the K tail read as zero through the buffer descriptor's range check.
//  * LDS layouts and swizzles (16-byte chunks, chosen for CDNA4's 64-bank LDS):
//      A stage [BM][64] fp16, row = 8 chunks, chunk c of row m at c ^ fA(m),
//          fA(m) = (m & 7) ^ ((m >> 3) & 3): 16 consecutive rows at one chunk hit 16
//          distinct 16-byte bank groups (ds_read_b128 conflict-free).
//      B stage [64][BN] fp16 (N contiguous, as in HBM), chunk c of row k at c ^ gB(k & 3),
//          gB = {0, 6, 10, 12}: the 4 rows x 4 chunks that 32 lanes of one
//          ds_read_b64_tr_b16 touch land in 16 distinct bank groups.
//    The A fragment is one ds_read_b128 (8 consecutive k of one row).  The B fragment needs
//    8 consecutive k of one column of an N-contiguous tile: two ds_read_b64_tr_b16, which
//    transpose 4x16 blocks across each 16-lane group (lane i receives column i of the 4
//    rows that lanes 4e + i/4 address).
//  * Workgroup -> tile: XCD-aware, L2-grouped bijection (mmm_tile_map.h).
//
// A second instantiation of the same kernel ("generic") stages through VGPRs with
// element-wise masked loads; it serves leading dimensions or pointers that are not
// 16-byte aligned (e.g. the ragged 4097 x 4095 x 4111 configuration) and arbitrary K.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "mmm.h"
#include "mmm_dma.h"
#include "mmm_kernels.h"
#include "mmm_tile.h"
#include "mmm_tile_map.h"

namespace mmm {

// GENERIC = false: direct-to-LDS buffer loads; needs 2-byte-aligned A and B and per-tile byte
//                  offsets within 32 bits (dma_ok).  Rows that are not 16-byte aligned are read
//                  by unaligned buffer loads.  The last K tile of an unaligned problem
//                  (tail_regs) is loaded like the others with its chunks across K (A) and
//                  across N in B's last row patched from a copy gathered at the start, or,
//                  for operands narrower than the tile (ldb < BN or lda < 8), gathered
//                  through VGPRs.
// GENERIC = true : element-wise masked loads through VGPRs; any shape and alignment.
// CPOL: how C's 16-byte pieces are stored (CStore): plain, non-temporal or system-scope
//       write-through (sc0 sc1); the last two for 16-byte-aligned C rows only (see launch_nn).
// TAIL: the direct-to-LDS kernel handles an unaligned last K tile (p.tail_regs); launches
//       without one run the instantiation with TAIL = false, which carries none of that code.
template <class T, bool GENERIC, int CPOL = kStorePlain, bool TAIL = true>
__global__ __launch_bounds__(T::NT, nn_launch_occupancy<T>()) void gemm_nn_kernel(GemmProblem p, int tiles_m,
                                                                                  int tiles_n) {
  __shared__ __attribute__((aligned(1024))) char lds[T::STAGES * T::STAGE];
  // The last K tile's straddling chunks, gathered at the start: A's chunk across K of each
  // tile row (entry = row in the tile), then B's chunk across N in row K-1 (entry BM).
  constexpr int kSpare = TAIL && !GENERIC ? T::BM + 1 : 1;
  __shared__ half8 tail_spare[kSpare];
  static_assert(GENERIC || T::OCC * (T::STAGES * T::STAGE + kSpare * 16) <= 160 * 1024,
                "LDS rings and the tail copy must fit the 160 KB LDS");
  record_clock(p.clk, 0);

  // K split (direct-to-LDS path only).  Blocks [0, whole) compute tiles 0 .. whole-1 of the
  // XCD-aware order over their full K range; the last split_tiles tiles of that order are split:
  // block whole + q * split_tiles + j computes K range q of tile whole + j (each split layer
  // walks those tiles in the same order).
  const int ntiles = tiles_m * tiles_n;
  const int ksplit = (!GENERIC && p.k_splits > 1) ? p.k_splits : 1;
  const int whole = ksplit > 1 ? ntiles - p.split_tiles : ntiles;
  const bool split_block = (int)blockIdx.x >= whole;
  const int nsplit = split_block ? ksplit : 1;
  int q = 0, j = -1, tm, tn;
  if (split_block) split_item((int)blockIdx.x, whole, p.split_tiles, ksplit, p.split_major, &q, &j);
  q = __builtin_amdgcn_readfirstlane(q);
  tile_of_item((int)blockIdx.x, j, whole, p.split_major, tiles_m, tiles_n, &tm, &tn);
  // The tile origin is uniform; readfirstlane keeps it (and everything derived from it, such
  // as the buffer descriptors) in SGPRs -- the integer divisions above are expanded on the VALU.
  const int m0 = __builtin_amdgcn_readfirstlane(tm * T::BM), n0 = __builtin_amdgcn_readfirstlane(tn * T::BN);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w / T::WGN, wn = w % T::WGN;
  const int M = p.M, N = p.N, K = p.K;
  const int64_t lda = p.lda, ldb = p.ldb;

  // ---- staging map.  Thread (w, lane) moves chunk slot s = r*NT + w*64 + lane of a stage
  // (r = 0..RA-1 for A, 0..RB-1 for B).  A round of NT slots covers RPA = NT/CA rows of A
  // and RPB = NT/CB rows of B, so slot rows are row0 + r*RP; RPA is a multiple of the rows
  // the A swizzle depends on and RPB of 4, so the logical chunk is the same every round.
  constexpr int RPA = T::NT / T::CA, RPB = T::NT / T::CB;
  static_assert(RPA % T::SWZ_A_ROWS == 0 && (!T::B_UNIFORM || RPB % T::SWZ_B_ROWS == 0),
                "round strides must preserve the swizzle");
  static_assert(!GENERIC || T::B_UNIFORM, "the register-staged path uses the uniform B map");
  const int a_row0 = w * (64 / T::CA) + lane / T::CA;
  const int a_kc = 8 * ((lane % T::CA) ^ T::swz_a(a_row0));
  const int b_row0 = T::B_UNIFORM ? w * (64 / T::CB) + lane / T::CB : 0;
  const int b_nc = T::B_UNIFORM ? 8 * ((lane % T::CB) ^ T::swz_bk(b_row0)) : 0;
  // B row and column of slot r (any CB)
  auto b_row_of = [&](int r) {
    if constexpr (T::B_UNIFORM) return b_row0 + r * RPB;
    else return (r * T::NT + w * 64 + lane) / T::CB;
  };
  auto b_col_of = [&](int r) {
    if constexpr (T::B_UNIFORM) return b_nc;
    else {
      const int sl = r * T::NT + w * 64 + lane;
      return 8 * ((sl % T::CB) ^ T::swz_bk(sl / T::CB));
    }
  };

  // ---- fragment read offsets (bytes within a stage).  MF = 32: lane l reads row l % 32 of
  // A, k chunk l / 32 of each 16-deep step; B rows 8*(l/32) + (l/4)%4 (+4), columns
  // 16*((l/16)%2) + 4*(l%4) of each 32-column fragment.  MF = 16: row l % 16 of A, k chunk
  // l / 16 of each 32-deep step; B rows 8*(l/16) + (l/4)%4 (+4), columns 4*(l%4) of each
  // 16-column fragment.
  uint32_t a_off[kMaxOff] = {};
#pragma unroll
  for (int kk = 0; kk < T::KSTEPS; ++kk)
#pragma unroll
    for (int ph = 0; ph < T::APAR; ++ph) {
      const int m = wm * T::TM + ph * T::MF + (lane % T::MF);
      const int chunk = (T::KK / 8) * kk + lane / T::MF;
      a_off[kk * T::APAR + ph] = m * T::BK * 2 + (chunk ^ T::swz_a(m)) * 16;
    }
  uint32_t b_off[kMaxOff] = {};
  {
    const int k = 8 * (lane / T::MF) + ((lane >> 2) & 3);
#pragma unroll
    for (int nb = 0; nb < T::FN; ++nb) {
      const int n = T::MF == 32 ? wn * T::TN + 32 * nb + 16 * ((lane >> 4) & 1) + 4 * (lane & 3)
                                : wn * T::TN + 16 * nb + 4 * (lane & 3);
      b_off[nb] = k * T::BN * 2 + (((n >> 3) ^ T::swz_bk(k)) * 16) + (n & 7) * 2;
    }
  }

  AccT<T> acc[T::FM][T::FN];
#pragma unroll
  for (int i = 0; i < T::FM; ++i)
#pragma unroll
    for (int j = 0; j < T::FN; ++j) acc[i][j] = AccT<T>{};

  const int KT_all = (K + T::BK - 1) / T::BK;
  const int t_begin = __builtin_amdgcn_readfirstlane((q * KT_all) / nsplit);
  const int t_end = __builtin_amdgcn_readfirstlane(((q + 1) * KT_all) / nsplit);
  const int KT = t_end - t_begin;  // K tiles of this block
  char LDS_AS* lds_base = (char LDS_AS*)lds;

  if constexpr (!GENERIC) {
    const uint32_t a_goff = (uint32_t)((a_row0 * lda + a_kc) * 2);
    const uint32_t b_goff = (uint32_t)((b_row0 * ldb + b_nc) * 2);
    const uint32_t a_rstep = (uint32_t)(RPA * lda * 2), b_rstep = (uint32_t)(RPB * ldb * 2);
    uint32_t b_goffr[T::B_UNIFORM ? 1 : T::RB];  // per-slot B offsets (non-uniform map)
    if constexpr (!T::B_UNIFORM) {
#pragma unroll
      for (int r = 0; r < T::RB; ++r) b_goffr[r] = (uint32_t)((b_row_of(r) * ldb + b_col_of(r)) * 2);
    }

    // The last K tile of an unaligned problem (p.tail_regs: K or N not a multiple of 8, or rows
    // not 16-byte aligned), in the block that holds it.  When B's rows are at least a tile wide
    // and A's at least a chunk (dma_tail), no chunk of any tile reaches across a descriptor's
    // range end other than two of the last tile: A's chunk across K in row M-1 and B's chunk
    // across N in row K-1.  The last tile's ranges end before those two, so they read as zero
    // like every chunk past the ends, and its chunks across K (every row of A: past K they hold
    // the next row's values) and across N in B's row K-1 are overwritten from tail_spare before
    // the tile is published (tail_fix).  Narrower operands gather the whole last tile through
    // VGPRs instead (tail_regs).
    const bool tail_block = TAIL && p.tail_regs && t_end == KT_all;
    const bool dma_tail = ldb >= T::BN && lda >= 8;
    const bool tail_regs = tail_block && !dma_tail;
    const bool tail_fix = tail_block && dma_tail;

    // DMA of K tile t into ring slot `stage`: RA + RB buffer_load_dwordx4 ... lds per thread.
    // Each range ends at the operand's last element (row M-1, column K-1 of A; row K-1,
    // column N-1 of B), so nothing past the caller's data is ever fetched; rows past the end
    // read as zero.  With N, K multiples of 8 no chunk straddles a range end.  K tiles are
    // issued in order (t = 0, 1, ...), so bases and remaining byte counts advance by a
    // constant per tile instead of being recomputed.
    const char* a_ptr = (const char*)(p.A + (int64_t)m0 * lda + (int64_t)t_begin * T::BK);
    const char* b_ptr = (const char*)(p.B + (int64_t)t_begin * T::BK * ldb + n0);
    int64_t a_left = ((int64_t)(M - 1 - m0) * lda + K - (int64_t)t_begin * T::BK) * 2;
    int64_t b_left = ((int64_t)(K - 1 - t_begin * T::BK) * ldb + N - n0) * 2;
    const int64_t b_step = (int64_t)T::BK * ldb * 2;
    // A K tile's loads: descriptors and bases (prep; advances the running state), then the
    // LPT loads, j = 0 .. RA-1 for A and RA .. LPT-1 for B (dma_one).
    struct TileDma {
      i32x4 ra, rb;
      uint32_t a_dst, b_dst, a_base;
    };
    auto prep = [&](int t, int stage) {
      const int k0 = (t_begin + t) * T::BK;
      TileDma d;
      d.ra = make_rsrc(a_ptr, clip_records(a_left));
      d.rb = make_rsrc(b_ptr, clip_records(b_left));
      a_ptr += T::BK * 2, a_left -= T::BK * 2;
      b_ptr += b_step, b_left -= b_step;
      d.a_dst = lds_addr_of(lds_base) + stage * T::STAGE + w * 64 * 16;
      d.b_dst = d.a_dst + T::A_BYTES;
      // K tail: a chunk at or past K gets kOobOffset added, which puts it beyond the
      // descriptor's range so it reads as zero (no select: keeps the loads branch-free).
      const uint32_t a_dead = (uint32_t)(K - 1 - (k0 + a_kc)) >> 31;
      d.a_base = a_goff + ((0u - a_dead) & kOobOffset);
      return d;
    };
    auto dma_one = [&](const TileDma& d, int j) {
      if (j < T::RA)
        dma_b128(d.a_dst + j * T::NT * 16, d.ra, d.a_base + j * a_rstep);
      else
        dma_b128(d.b_dst + (j - T::RA) * T::NT * 16, d.rb,
                 T::B_UNIFORM ? b_goff + (j - T::RA) * b_rstep : b_goffr[T::B_UNIFORM ? 0 : j - T::RA]);
    };
    auto issue = [&](int t, int stage) {
      const TileDma d = prep(t, stage);
#pragma unroll
      for (int j = 0; j < T::LPT; ++j) dma_one(d, j);
    };

    // tail_regs: the last K tile gathered element by element through VGPRs into the same slot
    // layout.
    const _Float16* Ah = (const _Float16*)p.A;
    const _Float16* Bh = (const _Float16*)p.B;
    auto fill_regs = [&](int t, int stage) {
      const int k0 = (t_begin + t) * T::BK;
      char LDS_AS* a_dst = lds_base + stage * T::STAGE + (w * 64 + lane) * 16;
      char LDS_AS* b_dst = a_dst + T::A_BYTES;
      // Element loads under lane conditions, one memory round trip each: this path serves
      // operands narrower than the tile only, and it runs in the refill peeled off the K loop,
      // where the registers that would keep a chunk's loads in flight together are not free
      // (the 256x256 tile spilled; on the 64x64 tile, where they fit, the extra registers cost
      // its patched-tail launches 0.2-0.3 us per call, more than the gather gained).
#pragma unroll
      for (int r = 0; r < T::RA; ++r) {
        const int m = m0 + a_row0 + r * RPA, k = k0 + a_kc;
        half8 v = {};
        if (m < M) {
          const _Float16* src = Ah + (int64_t)m * lda + k;
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (k + e < K) v[e] = src[e];
        }
        *(half8 LDS_AS*)(a_dst + r * T::NT * 16) = v;
      }
#pragma unroll
      for (int r = 0; r < T::RB; ++r) {
        const int k = k0 + b_row_of(r), n = n0 + b_col_of(r);
        half8 v = {};
        if (k < K) {
          const _Float16* src = Bh + (int64_t)k * ldb + n;
#pragma unroll
          for (int e = 0; e < 8; ++e)
            if (n + e < N) v[e] = src[e];
        }
        *(half8 LDS_AS*)(b_dst + r * T::NT * 16) = v;
      }
    };
    // tail_fix: the chunk of the last K tile across K (column k0t + a_kcs .. +7 of each row of
    // A, K % 8 of them valid) and across N in B's row K-1 (columns n0 + n_cs .. +7, N % 8
    // valid), gathered here (their loads overlap the first tiles'), kept in tail_spare from
    // the first tile's wait on, and copied over what the DMA put in their slots.  Thread
    // (w, lane) owns the same chunks in every tile: its A chunks when its chunk column is
    // a_kcs, and B slot r when that slot is row K-1, column n_cs.
    const int k0t = (KT_all - 1) * T::BK;
    const int a_kcs = (K - k0t) & ~7, n_cs = (N - n0) & ~7;
    const bool a_fix = tail_fix && (K & 7) != 0 && a_kc == a_kcs;
    // What the last tile needs, packed into one scalar that lives through the K loop: bit 0
    // tail_fix, then K % 8, N % 8, a_kcs (6 bits), K-1 as a row of the last tile (< 64) and n_cs
    // clamped to BN (no chunk of the tile when the tile does not reach N).  a_kcs is used only
    // when K % 8 != 0, where it is at most 56; with K a multiple of 64 it is 64 and is masked to
    // keep it out of the row field (whose low bit it would otherwise set: that field is then 63,
    // so the OR changed nothing, but the mask does not rely on that).
    const uint32_t tp = !TAIL ? 0u
                              : __builtin_amdgcn_readfirstlane(
                                    (uint32_t)tail_fix | (uint32_t)(K & 7) << 1 | (uint32_t)(N & 7) << 4 |
                                    (uint32_t)(a_kcs & 63) << 7 | (uint32_t)(K - 1 - k0t) << 13 |
                                    (uint32_t)(n_cs < T::BN ? n_cs : T::BN) << 19);
    // Both the gather and the store sit behind the scalar test of tp: the wait for the gathered
    // registers (a full vmcnt drain, the compiler not seeing the DMA loads) must not reach the
    // prologue of a launch without a patched tail.
    half8 a_fixv[T::RA];
    int b_fix_r = -1;
    half8 b_fixv = {};
    // Every lane loads (addresses clamped into the operands, values masked afterwards), so the
    // loads carry no branches and go out together: a load under a lane condition is merged
    // into its vector before the next one issues, one memory round trip each.
    if (tp & 1) {
      const int ka = K & 7, kb = N & 7;
      if (ka != 0) {
#pragma unroll
        for (int r = 0; r < T::RA; ++r) {
          const int m = m0 + a_row0 + r * RPA;
          const _Float16* src = Ah + (int64_t)(m < M ? m : M - 1) * lda + k0t + a_kcs;
          _Float16 x[7];
#pragma unroll
          for (int e = 0; e < 7; ++e) x[e] = src[e < ka ? e : ka - 1];  // columns below K
          half8 v = {};
#pragma unroll
          for (int e = 0; e < 7; ++e) v[e] = (e < ka && m < M) ? x[e] : (_Float16)0;
          a_fixv[r] = v;
        }
      }
      if (kb != 0) {
#pragma unroll
        for (int r = 0; r < T::RB; ++r)
          if (k0t + b_row_of(r) == K - 1 && b_col_of(r) == n_cs) b_fix_r = r;
        const _Float16* src = Bh + (int64_t)(K - 1) * ldb;
        const int c0 = n0 + n_cs;
        _Float16 x[7];
#pragma unroll
        for (int e = 0; e < 7; ++e) x[e] = src[c0 + e < N ? c0 + e : N - 1];
#pragma unroll
        for (int e = 0; e < 7; ++e) b_fixv[e] = e < kb ? x[e] : (_Float16)0;
      }
    }
    auto spare_store = [&] {
      if (tp & 1) {
        if (a_fix) {
#pragma unroll
          for (int r = 0; r < T::RA; ++r) tail_spare[a_row0 + r * RPA] = a_fixv[r];
        }
        if (b_fix_r >= 0) tail_spare[kSpare - 1] = b_fixv;  // entry BM
      }
    };
    // At the last tile the lane-derived values are rebuilt from a fresh lane index rather than
    // kept live through the K loop.
    auto tail_patch = [&](int slot) {
      if (!(tp & 1)) return;
      const int ln = lane_id_fresh();
      char LDS_AS* a_dst = lds_base + slot * T::STAGE + (w * 64 + ln) * 16;
      const int row0 = w * (64 / T::CA) + ln / T::CA;
      if ((tp >> 1 & 7) != 0 && 8 * ((ln % T::CA) ^ T::swz_a(row0)) == (int)(tp >> 7 & 63)) {
#pragma unroll
        for (int r = 0; r < T::RA; ++r) *(half8 LDS_AS*)(a_dst + r * T::NT * 16) = tail_spare[row0 + r * RPA];
      }
      if ((tp >> 4 & 7) != 0) {
#pragma unroll
        for (int r = 0; r < T::RB; ++r) {
          const int sl = r * T::NT + w * 64 + ln;
          const int row = sl / T::CB, col = 8 * ((sl % T::CB) ^ T::swz_bk(row));
          if (row == (int)(tp >> 13 & 63) && col == (int)(tp >> 19))
            *(half8 LDS_AS*)(a_dst + T::A_BYTES + r * T::NT * 16) = tail_spare[kSpare - 1];
        }
      }
    };

    // The last tile is issued by the prologue or by the refill peeled off the steady loop
    // (cross_stage), never by the steady loop's own refill.
    auto issue_tile = [&](int t, int stage) {
      if (tail_regs && t == KT - 1) {
        fill_regs(t, stage);
      } else {
        if ((tp & 1) && t == KT - 1) a_left -= (tp >> 1 & 7) * 2, b_left -= (tp >> 4 & 7) * 2;  // the cut ranges
        issue(t, stage);
      }
    };

    cross_stage<T, false>(lds_base, KT, tail_regs, a_off, b_off, acc, prep, dma_one, issue_tile, 0, spare_store,
                          tail_patch);
  } else {
    static_assert(!GENERIC || T::STAGES == 2, "the register-staged path double-buffers");
    (void)t_begin;
    u32x4 ra[T::RA], rb[T::RB];
    const _Float16* A = (const _Float16*)p.A;
    const _Float16* B = (const _Float16*)p.B;
    auto load = [&](int t) {
      const int k0 = t * T::BK;
#pragma unroll
      // Elements past the operands load from kZeroHalves: no load sits under a lane condition,
      // so a stage's loads go out together (a conditional load is merged into its vector before
      // the next one issues).
      for (int r = 0; r < T::RA; ++r) {
        const int m = m0 + a_row0 + r * RPA, k = k0 + a_kc;
        const _Float16* src = A + (int64_t)m * lda + k;
        half8 v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = *(m < M && k + e < K ? src + e : kZeroHalves);
        ra[r] = __builtin_bit_cast(u32x4, v);
      }
#pragma unroll
      for (int r = 0; r < T::RB; ++r) {
        const int k = k0 + b_row0 + r * RPB, n = n0 + b_nc;
        const _Float16* src = B + (int64_t)k * ldb + n;
        half8 v;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = *(k < K && n + e < N ? src + e : kZeroHalves);
        rb[r] = __builtin_bit_cast(u32x4, v);
      }
    };
    auto store = [&](int stage) {
      char LDS_AS* a_dst = lds_base + stage * T::STAGE + (w * 64 + lane) * 16;
      char LDS_AS* b_dst = lds_base + stage * T::STAGE + T::A_BYTES + (w * 64 + lane) * 16;
#pragma unroll
      for (int r = 0; r < T::RA; ++r) *(u32x4 LDS_AS*)(a_dst + r * T::NT * 16) = ra[r];
#pragma unroll
      for (int r = 0; r < T::RB; ++r) *(u32x4 LDS_AS*)(b_dst + r * T::NT * 16) = rb[r];
    };

    load(0);
    store(0);
    block_sync();
    for (int t = 0; t + 1 < KT; ++t) {
      const int cur = t & 1;
      load(t + 1);
      compute_stage<T, false>(lds_base + cur * T::STAGE, lds_base + cur * T::STAGE + T::A_BYTES, a_off, b_off, acc,
                              NoHook{});
      store(cur ^ 1);
      block_sync();
    }
    {
      const int cur = (KT - 1) & 1;
      compute_stage<T, false>(lds_base + cur * T::STAGE, lds_base + cur * T::STAGE + T::A_BYTES, a_off, b_off, acc,
                              NoHook{});
    }
  }

  // ---- epilogue: lane owns row m, columns n..n+3 for each (mb, nb, q).  MF = 32: m = l % 32,
  // n = 32*nb + 8*q + 4*(l/32) (q = 0..3); MF = 16: m = l % 16, n = 16*nb + 4*(l/16) (q = 0).
  constexpr int NQ = T::MF == 32 ? 4 : 1;  // float4 groups per accumulator
  static_assert(NQ * 4 == sizeof(AccT<T>) / 4, "accumulator groups");
  auto col_of = [&](int nb, int qq) {
    return T::MF == 32 ? 32 * nb + 8 * qq + 4 * (lane >> 5) : 16 * nb + 4 * (lane >> 4);
  };
  if (nsplit > 1) {  // K split: the whole tile (rows/columns past M/N included) to the partials
    float* part = p.partials + ((int64_t)j * nsplit + q) * (T::BM * T::BN);
    // Whole lines, written through (sc0 sc1): reduce_tiles_kernel, next on the stream, reads
    // them on other XCDs.  Measured on MI355X (interleaved, against L2-allocating half lines):
    // 256 x 4096 x 4096 +9.2%, 1024^2 x 8192 +5.9%, 1024 x 2048 x 4096 +4.7%, 128 x 14336 x 4096
    // +3.3%, 1536^2 x 12288 +2.6%, 2304^2 x 8192 +1.9%; non-temporal lines -4% to +6%.
    if constexpr (c_lines_ok<T>()) {
      store_wave_tile_lines<T, kStoreWriteThrough>(part + wm * T::TM * T::BN + wn * T::TN, T::BN, acc);
      record_clock(p.clk, 2);
      return;
    }
#pragma unroll
    for (int mb = 0; mb < T::FM; ++mb) {
      float* prow = part + (wm * T::TM + T::MF * mb + (lane % T::MF)) * T::BN + wn * T::TN;
#pragma unroll
      for (int nb = 0; nb < T::FN; ++nb)
#pragma unroll
        for (int qq = 0; qq < NQ; ++qq)
          *(f32x4*)(prow + col_of(nb, qq)) = f32x4{acc[mb][nb][4 * qq + 0], acc[mb][nb][4 * qq + 1],
                                                   acc[mb][nb][4 * qq + 2], acc[mb][nb][4 * qq + 3]};
    }
    record_clock(p.clk, 2);
    return;
  }
  float* C = p.C;
  const int64_t ldc = p.ldc;
  const bool vec_ok = p.c_vec4;
  // Interior tiles store whole lines with every store policy here (plain ones too: the ragged
  // configuration +0.7-1%, other plain grids +-0.5%).
  if constexpr (c_lines_ok<T>()) {
    if (vec_ok && m0 + T::BM <= M && n0 + T::BN <= N) {  // interior tile (uniform)
      store_wave_tile_lines<T, CPOL>(C + (int64_t)(m0 + wm * T::TM) * ldc + n0 + wn * T::TN, ldc, acc);
      record_clock(p.clk, 2);
      return;
    }
  }
#pragma unroll
  for (int mb = 0; mb < T::FM; ++mb) {
    const int m = m0 + wm * T::TM + T::MF * mb + (lane % T::MF);
    if (m >= M) continue;
    float* crow = C + (int64_t)m * ldc;
#pragma unroll
    for (int nb = 0; nb < T::FN; ++nb) {
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const int n = n0 + wn * T::TN + col_of(nb, q);
        f32x4 v = {acc[mb][nb][4 * q + 0], acc[mb][nb][4 * q + 1], acc[mb][nb][4 * q + 2], acc[mb][nb][4 * q + 3]};
        if (vec_ok && n + 3 < N) {
          store_c4<CPOL>(crow + n, v);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < N) crow[n + e] = v[e];
        }
      }
    }
  }
  record_clock(p.clk, 2);
}

// ------------------------------------------------------------------------------------
// Persistent direct-to-LDS tile kernel, for grids of whole interior tiles (M and N multiples
// of the tile, aligned operands and C; a K split of the last round runs as
// gemm_nn_persistent_split_kernel instead) over more than one round: grid =
// min(tiles, 256) workgroups; workgroup b computes tiles b, b + grid, b + 2*grid, ... of the
// XCD-aware order (grid % 8 == 0 keeps it on one XCD, walking that XCD's tile patches in
// order).  Between two tiles it waits for every wave to finish reading the ring, issues the
// next tile's first S K tiles, and only then stores the finished tile's C: the stores drain
// while those loads are in flight, and the next tile's first wait lets the NST stores
// (issued after the loads) stay outstanding, since vector-memory operations retire in issue
// order.
// ------------------------------------------------------------------------------------
template <class T, bool NT>
__global__ __launch_bounds__(T::NT, T::OCC) void gemm_nn_persistent_kernel(GemmProblem p, int tiles_m, int tiles_n) {
  __shared__ __attribute__((aligned(1024))) char lds[T::STAGES * T::STAGE];
  record_clock(p.clk, 0);
  constexpr int S = T::STAGES;
  constexpr int NQ = T::MF == 32 ? 4 : 1;       // float4 groups per accumulator
  constexpr int NST = T::FM * T::FN * NQ;       // C stores per thread per tile
  const int ntiles = tiles_m * tiles_n;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w / T::WGN, wn = w % T::WGN;
  const int K = p.K;
  const int64_t lda = p.lda, ldb = p.ldb;

  // staging map and fragment offsets: as gemm_nn_kernel
  constexpr int RPA = T::NT / T::CA, RPB = T::NT / T::CB;
  static_assert(RPA % T::SWZ_A_ROWS == 0 && (!T::B_UNIFORM || RPB % T::SWZ_B_ROWS == 0),
                "round strides must preserve the swizzle");
  // Fragment offsets (as gemm_nn_kernel), rebuilt at every tile from a freshly read lane index:
  // kept from the kernel's start they would be live through the epilogue, whose line stores
  // need the registers.
  uint32_t a_off[kMaxOff], b_off[kMaxOff];
  auto frag_offsets = [&]() {
    const int ln = lane_id_fresh();
#pragma unroll
    for (int q = 0; q < kMaxOff; ++q) a_off[q] = b_off[q] = 0;
#pragma unroll
    for (int kk = 0; kk < T::KSTEPS; ++kk)
#pragma unroll
      for (int ph = 0; ph < T::APAR; ++ph) {
        const int m = wm * T::TM + ph * T::MF + (ln % T::MF);
        const int chunk = (T::KK / 8) * kk + ln / T::MF;
        a_off[kk * T::APAR + ph] = m * T::BK * 2 + (chunk ^ T::swz_a(m)) * 16;
      }
    const int k = 8 * (ln / T::MF) + ((ln >> 2) & 3);
#pragma unroll
    for (int nb = 0; nb < T::FN; ++nb) {
      const int n = T::MF == 32 ? wn * T::TN + 32 * nb + 16 * ((ln >> 4) & 1) + 4 * (ln & 3)
                                : wn * T::TN + 16 * nb + 4 * (ln & 3);
      b_off[nb] = k * T::BN * 2 + (((n >> 3) ^ T::swz_bk(k)) * 16) + (n & 7) * 2;
    }
  };

  const int KT = (K + T::BK - 1) / T::BK;
  char LDS_AS* lds_base = (char LDS_AS*)lds;
  const uint32_t a_rstep = (uint32_t)(RPA * lda * 2), b_rstep = (uint32_t)(RPB * ldb * 2);
  // Per-lane load offset bases (as gemm_nn_kernel; b_goffr: per-slot B offsets of a non-uniform
  // map), rebuilt at every tile from a freshly read lane index, so that they are not live
  // through a tile's last K step and epilogue, which run at the register limit.
  int a_kc_t;  // a_kc, for the K-tail test
  uint32_t a_goff, b_goff;
  uint32_t b_goffr[T::B_UNIFORM ? 1 : T::RB];
  auto dma_bases = [&]() {
    const int ln = lane_id_fresh();
    const int ar0 = w * (64 / T::CA) + ln / T::CA;
    a_kc_t = 8 * ((ln % T::CA) ^ T::swz_a(ar0));
    a_goff = (uint32_t)((ar0 * lda + a_kc_t) * 2);
    if constexpr (T::B_UNIFORM) {
      const int br0 = w * (64 / T::CB) + ln / T::CB;
      b_goff = (uint32_t)((br0 * ldb + 8 * ((ln % T::CB) ^ T::swz_bk(br0))) * 2);
    } else {
      b_goff = 0;
#pragma unroll
      for (int r = 0; r < T::RB; ++r) {
        const int sl = r * T::NT + w * 64 + ln;
        b_goffr[r] = (uint32_t)(((sl / T::CB) * ldb + 8 * ((sl % T::CB) ^ T::swz_bk(sl / T::CB))) * 2);
      }
    }
  };
  const int64_t b_step = (int64_t)T::BK * ldb * 2;
  // per-tile running load state (K tiles are prepared in order from 0)
  const char* a_ptr;
  const char* b_ptr;
  int64_t a_left, b_left;
  auto start_tile = [&](int tm0, int tn0) {
    dma_bases();
    a_ptr = (const char*)(p.A + (int64_t)tm0 * lda);
    b_ptr = (const char*)(p.B + tn0);
    a_left = ((int64_t)(p.M - 1 - tm0) * lda + K) * 2;
    b_left = ((int64_t)(K - 1) * ldb + p.N - tn0) * 2;
  };
  struct TileDma {
    i32x4 ra, rb;
    uint32_t a_dst, b_dst, a_base;
  };
  auto prep = [&](int t, int stage) {
    const int k0 = t * T::BK;
    TileDma d;
    d.ra = make_rsrc(a_ptr, clip_records(a_left));
    d.rb = make_rsrc(b_ptr, clip_records(b_left));
    a_ptr += T::BK * 2, a_left -= T::BK * 2;
    b_ptr += b_step, b_left -= b_step;
    d.a_dst = lds_addr_of(lds_base) + stage * T::STAGE + w * 64 * 16;
    d.b_dst = d.a_dst + T::A_BYTES;
    const uint32_t a_dead = (uint32_t)(K - 1 - (k0 + a_kc_t)) >> 31;
    d.a_base = a_goff + ((0u - a_dead) & kOobOffset);
    return d;
  };
  auto dma_one = [&](const TileDma& d, int j) {
    if (j < T::RA)
      dma_b128(d.a_dst + j * T::NT * 16, d.ra, d.a_base + j * a_rstep);
    else
      dma_b128(d.b_dst + (j - T::RA) * T::NT * 16, d.rb,
               T::B_UNIFORM ? b_goff + (j - T::RA) * b_rstep : b_goffr[T::B_UNIFORM ? 0 : j - T::RA]);
  };
  auto issue = [&](int t, int stage) {
    const TileDma d = prep(t, stage);
#pragma unroll
    for (int j = 0; j < T::LPT; ++j) dma_one(d, j);
  };

  int b = blockIdx.x;
  int tm, tn;
  tile_of_block(b, tiles_m, tiles_n, 4, &tm, &tn);
  int m0 = __builtin_amdgcn_readfirstlane(tm * T::BM), n0 = __builtin_amdgcn_readfirstlane(tn * T::BN);
  start_tile(m0, n0);
#pragma unroll
  for (int s = 0; s < S; ++s) issue(s, s);
  int pre = 1;
  AccT<T> acc[T::FM][T::FN];
  while (true) {
#pragma unroll
    for (int i = 0; i < T::FM; ++i)
#pragma unroll
      for (int jj = 0; jj < T::FN; ++jj) acc[i][jj] = AccT<T>{};
    frag_offsets();
    // again after the previous tile's line-store epilogue, which they need not live through
    if constexpr (use_c_lines<T, NT ? kStoreNonTemporal : kStorePlain>()) dma_bases();
    cross_stage<T, false, NST>(lds_base, KT, false, a_off, b_off, acc, prep, dma_one, issue, pre);
    const int nb = b + (int)gridDim.x;
    int nm0 = 0, nn0 = 0;
    if (nb < ntiles) {
      block_sync();  // every wave has read its last fragments of the ring
      tile_of_block(nb, tiles_m, tiles_n, 4, &tm, &tn);
      nm0 = __builtin_amdgcn_readfirstlane(tm * T::BM), nn0 = __builtin_amdgcn_readfirstlane(tn * T::BN);
      start_tile(nm0, nn0);
#pragma unroll
      for (int s = 0; s < S; ++s) issue(s, s);
      __builtin_amdgcn_sched_barrier(0);  // the loads go out before the stores below
    }
    // epilogue: interior tile, NST 16-byte stores per thread
    if constexpr (use_c_lines<T, NT ? kStoreNonTemporal : kStorePlain>()) {
      store_wave_tile_lines<T, NT ? kStoreNonTemporal : kStorePlain>(
          p.C + (int64_t)(m0 + wm * T::TM) * p.ldc + n0 + wn * T::TN, p.ldc, acc);
    } else
#pragma unroll
    for (int mb = 0; mb < T::FM; ++mb) {
      float* crow = p.C + (int64_t)(m0 + wm * T::TM + T::MF * mb + (lane % T::MF)) * p.ldc + n0 + wn * T::TN;
#pragma unroll
      for (int nb2 = 0; nb2 < T::FN; ++nb2)
#pragma unroll
        for (int qq = 0; qq < NQ; ++qq) {
          const int n = T::MF == 32 ? 32 * nb2 + 8 * qq + 4 * (lane >> 5) : 16 * nb2 + 4 * (lane >> 4);
          const f32x4 v = {acc[mb][nb2][4 * qq + 0], acc[mb][nb2][4 * qq + 1], acc[mb][nb2][4 * qq + 2],
                           acc[mb][nb2][4 * qq + 3]};
          if constexpr (NT)
            __builtin_nontemporal_store(v, (f32x4*)(crow + n));
          else
            *(f32x4*)(crow + n) = v;
        }
    }
    if (nb >= ntiles) break;
    b = nb, m0 = nm0, n0 = nn0, pre = 2;
  }
  record_clock(p.clk, 2);
}

// ------------------------------------------------------------------------------------
// Persistent grid over whole tiles and the last round's K-split pieces (same conditions as
// gemm_nn_persistent_kernel, plus a K split of an under-filled last round): the split pieces
// are the grid's final work items, so each workgroup's whole tiles keep the next-tile overlap
// and the split pieces follow without a kernel boundary; their partial tiles go to the
// workspace for reduce_tiles_kernel.  A separate kernel: folding the item bookkeeping into
// gemm_nn_persistent_kernel changed its register allocation (it spilled).
// ------------------------------------------------------------------------------------
template <class T, bool NT>
__global__ __launch_bounds__(T::NT, T::OCC) void gemm_nn_persistent_split_kernel(GemmProblem p, int tiles_m, int tiles_n) {
  __shared__ __attribute__((aligned(1024))) char lds[T::STAGES * T::STAGE];
  record_clock(p.clk, 0);
  constexpr int S = T::STAGES;
  constexpr int NQ = T::MF == 32 ? 4 : 1;       // float4 groups per accumulator
  constexpr int NST = T::FM * T::FN * NQ;       // C stores per thread per tile
  const int ntiles = tiles_m * tiles_n;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w / T::WGN, wn = w % T::WGN;
  const int K = p.K;
  const int64_t lda = p.lda, ldb = p.ldb;

  // staging map and fragment offsets: as gemm_nn_kernel
  constexpr int RPA = T::NT / T::CA, RPB = T::NT / T::CB;
  static_assert(RPA % T::SWZ_A_ROWS == 0 && RPB % T::SWZ_B_ROWS == 0, "round strides must preserve the swizzle");
  const int a_row0 = w * (64 / T::CA) + lane / T::CA;
  const int a_kc = 8 * ((lane % T::CA) ^ T::swz_a(a_row0));
  const int b_row0 = w * (64 / T::CB) + lane / T::CB;
  const int b_nc = 8 * ((lane % T::CB) ^ T::swz_bk(b_row0));
  uint32_t a_off[kMaxOff] = {};
#pragma unroll
  for (int kk = 0; kk < T::KSTEPS; ++kk)
#pragma unroll
    for (int ph = 0; ph < T::APAR; ++ph) {
      const int m = wm * T::TM + ph * T::MF + (lane % T::MF);
      const int chunk = (T::KK / 8) * kk + lane / T::MF;
      a_off[kk * T::APAR + ph] = m * T::BK * 2 + (chunk ^ T::swz_a(m)) * 16;
    }
  uint32_t b_off[kMaxOff] = {};
  {
    const int k = 8 * (lane / T::MF) + ((lane >> 2) & 3);
#pragma unroll
    for (int nb = 0; nb < T::FN; ++nb) {
      const int n = T::MF == 32 ? wn * T::TN + 32 * nb + 16 * ((lane >> 4) & 1) + 4 * (lane & 3)
                                : wn * T::TN + 16 * nb + 4 * (lane & 3);
      b_off[nb] = k * T::BN * 2 + (((n >> 3) ^ T::swz_bk(k)) * 16) + (n & 7) * 2;
    }
  }

  const int KT_all = (K + T::BK - 1) / T::BK;
  // Work items: whole tiles 0 .. whole-1 of the XCD-aware order over all of K, then (K split)
  // item whole + q * split_tiles + j = K range q of tile whole + j, as gemm_nn_kernel numbers
  // its blocks.  Workgroup b takes items b, b + grid, ...: whole tiles first, split pieces last.
  const int ksplit = p.k_splits > 1 ? p.k_splits : 1;
  const int whole = ksplit > 1 ? ntiles - p.split_tiles : ntiles;
  const int nitems = whole + (ksplit > 1 ? p.split_tiles * ksplit : 0);
  struct Item {
    int m0, n0, kt0, kt, q, j;  // tile origin, first K tile and K tiles, split index, split tile
  };
  auto item_of = [&](int it) {
    Item r;
    int bt = it, nsplit = 1;
    r.q = 0, r.j = 0;
    if (it >= whole) {
      const int i2 = it - whole;
      r.q = i2 / p.split_tiles, r.j = i2 - r.q * p.split_tiles;
      bt = whole + r.j, nsplit = ksplit;
    }
    int tmi, tni;
    tile_of_block(bt, tiles_m, tiles_n, 4, &tmi, &tni);
    r.m0 = __builtin_amdgcn_readfirstlane(tmi * T::BM), r.n0 = __builtin_amdgcn_readfirstlane(tni * T::BN);
    r.kt0 = __builtin_amdgcn_readfirstlane((r.q * KT_all) / nsplit);
    r.kt = __builtin_amdgcn_readfirstlane(((r.q + 1) * KT_all) / nsplit) - r.kt0;
    r.q = __builtin_amdgcn_readfirstlane(r.q), r.j = __builtin_amdgcn_readfirstlane(r.j);
    return r;
  };
  char LDS_AS* lds_base = (char LDS_AS*)lds;
  int a_kc_t = a_kc;  // a_kc for the K-tail test, made opaque per tile like the offset bases
  uint32_t a_goff = (uint32_t)((a_row0 * lda + a_kc) * 2);
  uint32_t b_goff = (uint32_t)((b_row0 * ldb + b_nc) * 2);
  const uint32_t a_rstep = (uint32_t)(RPA * lda * 2), b_rstep = (uint32_t)(RPB * ldb * 2);
  const int64_t b_step = (int64_t)T::BK * ldb * 2;
  // per-item running load state (an item's K tiles are prepared in order from its first)
  const char* a_ptr;
  const char* b_ptr;
  int64_t a_left, b_left;
  int kt0 = 0;  // the item's first K tile
  auto start_tile = [&](const Item& it) {
    // The per-lane offset bases pass through an empty asm each tile, so the offsets of a tile's
    // first loads are recomputed from them rather than kept live across the K loop (which
    // runs at the register limit).
    asm volatile("" : "+v"(a_goff), "+v"(b_goff), "+v"(a_kc_t));
    kt0 = it.kt0;
    const int64_t k0 = (int64_t)kt0 * T::BK;
    a_ptr = (const char*)(p.A + (int64_t)it.m0 * lda + k0);
    b_ptr = (const char*)(p.B + k0 * ldb + it.n0);
    a_left = ((int64_t)(p.M - 1 - it.m0) * lda + K - k0) * 2;
    b_left = ((K - 1 - k0) * ldb + p.N - it.n0) * 2;
  };
  struct TileDma {
    i32x4 ra, rb;
    uint32_t a_dst, b_dst, a_base;
  };
  auto prep = [&](int t, int stage) {
    const int k0 = (kt0 + t) * T::BK;
    TileDma d;
    d.ra = make_rsrc(a_ptr, clip_records(a_left));
    d.rb = make_rsrc(b_ptr, clip_records(b_left));
    a_ptr += T::BK * 2, a_left -= T::BK * 2;
    b_ptr += b_step, b_left -= b_step;
    d.a_dst = lds_addr_of(lds_base) + stage * T::STAGE + w * 64 * 16;
    d.b_dst = d.a_dst + T::A_BYTES;
    const uint32_t a_dead = (uint32_t)(K - 1 - (k0 + a_kc_t)) >> 31;
    d.a_base = a_goff + ((0u - a_dead) & kOobOffset);
    return d;
  };
  auto dma_one = [&](const TileDma& d, int j) {
    if (j < T::RA)
      dma_b128(d.a_dst + j * T::NT * 16, d.ra, d.a_base + j * a_rstep);
    else
      dma_b128(d.b_dst + (j - T::RA) * T::NT * 16, d.rb, b_goff + (j - T::RA) * b_rstep);
  };
  auto issue = [&](int t, int stage) {
    const TileDma d = prep(t, stage);
#pragma unroll
    for (int j = 0; j < T::LPT; ++j) dma_one(d, j);
  };

  int b = blockIdx.x;
  Item cur = item_of(b);
  start_tile(cur);
#pragma unroll
  for (int s = 0; s < S; ++s) issue(s, s);
  int pre = 1;
  AccT<T> acc[T::FM][T::FN];
  while (true) {
#pragma unroll
    for (int i = 0; i < T::FM; ++i)
#pragma unroll
      for (int jj = 0; jj < T::FN; ++jj) acc[i][jj] = AccT<T>{};
    cross_stage<T, false, NST>(lds_base, cur.kt, false, a_off, b_off, acc, prep, dma_one, issue, pre);
    const int nb = b + (int)gridDim.x;
    Item nxt = cur;
    if (nb < nitems) {
      block_sync();  // every wave has read its last fragments of the ring
      nxt = item_of(nb);
      start_tile(nxt);
#pragma unroll
      for (int s = 0; s < S; ++s) issue(s, s);
      __builtin_amdgcn_sched_barrier(0);  // the loads go out before the stores below
    }
    // epilogue: NST 16-byte stores per thread -- an interior tile of C, or a split piece's whole
    // partial tile, [split tile][split][BM][BN], for reduce_tiles_kernel
    const bool split_item = b >= whole;  // uniform
    float* base = split_item ? p.partials + ((int64_t)cur.j * ksplit + cur.q) * (T::BM * T::BN)
                             : p.C + (int64_t)cur.m0 * p.ldc + cur.n0;
    const int64_t ld = split_item ? T::BN : p.ldc;
    if constexpr (use_c_lines<T, NT ? kStoreNonTemporal : kStorePlain>()) {
      store_wave_tile_lines<T, NT ? kStoreNonTemporal : kStorePlain>(base + (int64_t)wm * T::TM * ld + wn * T::TN, ld,
                                                                      acc);
    } else
#pragma unroll
    for (int mb = 0; mb < T::FM; ++mb) {
      float* crow = base + (int64_t)(wm * T::TM + T::MF * mb + (lane % T::MF)) * ld + wn * T::TN;
#pragma unroll
      for (int nb2 = 0; nb2 < T::FN; ++nb2)
#pragma unroll
        for (int qq = 0; qq < NQ; ++qq) {
          const int n = T::MF == 32 ? 32 * nb2 + 8 * qq + 4 * (lane >> 5) : 16 * nb2 + 4 * (lane >> 4);
          const f32x4 v = {acc[mb][nb2][4 * qq + 0], acc[mb][nb2][4 * qq + 1], acc[mb][nb2][4 * qq + 2],
                           acc[mb][nb2][4 * qq + 3]};
          if constexpr (NT)
            __builtin_nontemporal_store(v, (f32x4*)(crow + n));
          else
            *(f32x4*)(crow + n) = v;
        }
    }
    if (nb >= nitems) break;
    b = nb, cur = nxt, pre = 2;
  }
  record_clock(p.clk, 2);
}

// ------------------------------------------------------------------------------------
// Host-side launch
// ------------------------------------------------------------------------------------
// C tile = sum over the K splits, in split order (fixed order: deterministic), of the partial
// tiles written by gemm_nn_kernel for split tile j (tile `first + j` of the XCD-aware order);
// one thread per 4 consecutive columns.
template <int BM, int BN>
__global__ __launch_bounds__(256) void reduce_tiles_kernel(GemmProblem p, int tiles_m, int tiles_n, int first,
                                                           int splits) {
  constexpr int F4 = BM * BN / 4;  // float4s per tile
  const int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int j = (int)(g / F4), e = (int)(g % F4);
  int tm, tn;
  tile_of_item(0, j, first, p.split_major, tiles_m, tiles_n, &tm, &tn);
  const int r = e / (BN / 4), c = 4 * (e % (BN / 4));
  const int m = tm * BM + r, n = tn * BN + c;
  if (m >= p.M || n >= p.N) return;
  const f32x4* src = (const f32x4*)(p.partials + (int64_t)j * splits * (BM * BN)) + e;
  const f32x4 sum = sum_splits(src, F4, splits);
  float* crow = p.C + (int64_t)m * p.ldc;
  if (p.c_vec4 && n + 3 < p.N) {
    *(f32x4*)(crow + n) = sum;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n + i < p.N) crow[n + i] = sum[i];
  }
}


template <class T, bool GENERIC>
static hipError_t launch_nn(const GemmProblem& p0, hipStream_t stream) {
  GemmProblem p = p0;
  const int tiles_m = (p.M + T::BM - 1) / T::BM;
  const int tiles_n = (p.N + T::BN - 1) / T::BN;
  const int64_t tiles = (int64_t)tiles_m * tiles_n;
  const int splits = p.k_splits > 1 ? p.k_splits : 1;
  const int64_t split_tiles = splits > 1 ? p.split_tiles : 0;
  if (split_tiles < 0 || split_tiles > tiles) return hipErrorInvalidValue;
  const int64_t blocks = tiles - split_tiles + split_tiles * splits;
  if (blocks > 0x7fffffff) return hipErrorInvalidValue;
  p.split_major = splits > 1 && split_major((int)(tiles - split_tiles), splits, T::BM, T::BN,
                                            (p.K + 63) / 64 / splits, ((int64_t)p.M + p.N) * p.K * 2);
  const LaunchPair pair(splits > 1 ? p.partials : nullptr);
  // A one-round grid writes all of C after its last K step, with nothing left to overlap, and
  // system-scope write-through stores (sc0 sc1) drain that burst faster.  As half lines they won
  // only where C outgrew the eight XCDs' L2 (32 MB; 256x256 tile: 8192 x 2048 x 2048 +3.1%,
  // 4096^3 +1.3%, but 2048^3 -4.7%, 1024^3 -7.5%); as whole lines (store_wave_tile_lines) they win
  // at every size measured on MI355X, against L2-allocating half lines: 2048^2 x 1024 +11%,
  // 2048^3 +6.7%, 1536^3 +5%, 2048^2 x 4096 +4.4%, 8192 x 1024 x 8192 +2.8%, 1024 x 8192 x 8192
  // +2.1%, 1024^3 +1.5-2.3%, 512^3 +-0.  Not with a K split (as half lines: 3072^3 on 128x256
  // -8.8%) or for rows of an odd ldc (-9%).
  const bool c16 = ((uintptr_t)p.C & 15) == 0 && p.ldc % 4 == 0;
  const bool wt = splits == 1 && blocks <= 256 * T::OCC && c16 &&
                  (c_lines_ok<T>() || (double)p.M * p.N * 4.0 > 32.0 * (1 << 20));
  // (Multi-round grids keep plain stores: non-temporal whole lines there measured -4.6% at
  // 5000^3, -1% at 4096^3 on 256x128, +7% at 8192^2 x 2048 on 256x128, +-0 elsewhere.)
  // the direct-to-LDS kernel with or without the unaligned-tail code
  auto launch_dma = [&](auto cpol) {
    constexpr int CP = decltype(cpol)::value;
    if (p.tail_regs)
      hipLaunchKernelGGL((gemm_nn_kernel<T, false, CP, true>), dim3((unsigned)blocks), dim3(T::NT), 0, stream, p,
                         tiles_m, tiles_n);
    else
      hipLaunchKernelGGL((gemm_nn_kernel<T, false, CP, false>), dim3((unsigned)blocks), dim3(T::NT), 0, stream, p,
                         tiles_m, tiles_n);
  };
  if constexpr (GENERIC) {
    (void)wt;
    (void)launch_dma;
    hipLaunchKernelGGL((gemm_nn_kernel<T, true>), dim3((unsigned)blocks), dim3(T::NT), 0, stream, p, tiles_m, tiles_n);
  } else if constexpr (c_lines_ok<T>() || (T::BM == 256 && T::BN == 256)) {
    if (wt)
      launch_dma(std::integral_constant<int, kStoreWriteThrough>{});
    else
      launch_dma(std::integral_constant<int, kStorePlain>{});
  } else {
    (void)wt;
    launch_dma(std::integral_constant<int, kStorePlain>{});
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || splits == 1) return e;
  const int64_t per_tile = T::BM * T::BN / 4 / 256;  // blocks of 256 float4s per tile
  hipLaunchKernelGGL((reduce_tiles_kernel<T::BM, T::BN>), dim3((unsigned)(split_tiles * per_tile)), dim3(256), 0,
                     stream, p, tiles_m, tiles_n, (int)(tiles - split_tiles), splits);
  return hipGetLastError();
}


// True when the direct-to-LDS path can serve the problem: fp16 operands (2-byte aligned), and
// per-tile byte offsets that fit the 32-bit buffer offsets.  Rows that are not 16-byte aligned
// (odd lda or ldb, e.g. the 4097 x 4095 x 4111 configuration) are read by 16-byte buffer loads
// at 2-byte-aligned addresses: this relies on the unaligned buffer access the gfx9 family
// serves in ROCm's default (unaligned) memory mode, which MI355X boxes run -- the exact
// full-size ragged tests cover it.  A platform without unaligned buffer access must send
// 2-byte-aligned rows to the register-staged path (return false for them here).
static bool dma_ok(const GemmProblem& p, int bm) {
  const uintptr_t a = (uintptr_t)p.A, b = (uintptr_t)p.B;
  if ((a & 1) || (b & 1)) return false;
  if ((int64_t)bm * p.lda * 2 >= (int64_t)kOobOffset) return false;
  if ((int64_t)kDmaBK * p.ldb * 2 >= (int64_t)kOobOffset) return false;
  return true;
}

// True when every DMA chunk of the last K tile also lies wholly inside the operands (K and
// N multiples of 8, 16-byte aligned rows); otherwise gemm_nn_kernel patches that tile's
// straddling chunks or gathers it through VGPRs, and the persistent kernels do not run.
static bool tail_aligned(const GemmProblem& p) {
  const uintptr_t a = (uintptr_t)p.A, b = (uintptr_t)p.B;
  return !((a & 15) || (b & 15) || p.lda % 8 || p.ldb % 8 || p.K % 8 || p.N % 8);
}

bool gemm_nn_direct_to_lds(const GemmProblem& p, int tile_id) {
  return dma_ok(p, tile_bm(tile_id));
}

// K split for a tile launch whose last round of 256 workgroups (one per CU) is less than half
// full -- the whole grid when it is one small round: the last round's tiles each run as
// `splits` K ranges, enough to refill about one workgroup per CU (at least 8 64-deep K tiles
// each, at most 16, partial tiles within the stream workspace).  Taken only when the round
// time it saves exceeds the reduction's traffic (each split writes its partial tile; the
// reduction reads them and writes C) and launch.  Direct-to-LDS path only.
TileSplit gemm_nn_split(const GemmProblem& p, int tile_id) {
  if (!gemm_nn_direct_to_lds(p, tile_id)) return {1, 0};
  const int bm = tile_bm(tile_id), bn = tile_bn(tile_id);
  const int64_t tiles = (int64_t)((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn);
  // A round counts one workgroup per CU for every tile (counting the 128x128 tile's two per CU
  // measured 3072^3 -5.5%, 1536^2 x 12288 -5%, 2304^2 x 8192 -2%).
  const int64_t slots = 256;
  const int64_t last = tiles - (tiles - 1) / slots * slots;  // tiles in the last round (1 .. slots)
  if (last * 2 >= slots) return {1, 0};
  const int kt = (p.K + 63) / 64;  // 64-deep K tiles (the 32-deep tiles have twice as many)
  int64_t splits = slots / last;
  if (splits > kt / 8) splits = kt / 8;
  if (splits > kMaxSplits) splits = kMaxSplits;
  const int64_t cap = (int64_t)(kMaxWorkspaceBytes / ((size_t)bm * bn * 4)) / last;
  if (splits > cap) splits = cap;
  if (splits < 2) return {1, 0};
  // one tile's round at 4.8 TFLOP/s per CU (the 256x256 tile at 8192^3; smaller tiles run
  // slower, so this underestimates the saving); reduction traffic at kSplitTrafficBps plus 3 us
  const double round = 2.0 * bm * bn * (kt * 64.0) / 4.8e12;
  const double saved = round * (1.0 - 1.0 / (double)splits);
  const double cost = (double)last * bm * bn * 4.0 * (2.0 * splits + 1.0) / kSplitTrafficBps + 3e-6;
  // split only with a clear margin: near break-even the estimate's error decides (measured on
  // MI355X: 6144^2 x 1024 split in two -2%, 6150 x 6144 x 2048 +2.4%)
  if (saved <= 1.5 * cost) return {1, 0};
  return {(int)splits, (int)last};
}

int gemm_nn_splits(const GemmProblem& p, int tile_id) { return gemm_nn_split(p, tile_id).splits; }

size_t gemm_nn_workspace_bytes(const GemmProblem& p, int tile_id) {
  const TileSplit sp = gemm_nn_split(p, tile_id);
  if (sp.splits < 2) return 0;
  const size_t bm = tile_bm(tile_id), bn = tile_bn(tile_id);
  return (size_t)sp.tiles * sp.splits * bm * bn * 4;
}

// The persistent kernel's conditions: whole interior tiles (256x256, or 192x192 without a K
// split) over more than one round of 256 workgroups, aligned operands (no masked last K tile),
// 4-byte-aligned C, and at least S + 1 K tiles.  Measured against one workgroup per tile (same
// box): 8192^3 +1%, 8192^2 x 2048 +3.7%, 16384 x 8192 x 1024 +3.8%; 192x192 at 6144^2 x 2048 +4%.
template <class TP = DmaTile<256, 256>>
static bool persistent_ok(const GemmProblem& p) {
  if (!dma_ok(p, TP::BM) || p.tail_regs || !p.c_vec4) return false;
  if (p.M % TP::BM || p.N % TP::BN) return false;
  if ((int64_t)(p.M / TP::BM) * (p.N / TP::BN) <= 256) return false;
  return (p.K + TP::BK - 1) / TP::BK >= TP::STAGES + 1;
}

// Workgroups of a non-persistent tile launch (whole tiles plus the split tiles' K ranges).
static int64_t launch_blocks(const GemmProblem& p, int bm, int bn) {
  const int64_t tiles = (int64_t)((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn);
  return p.k_splits > 1 ? tiles - p.split_tiles + (int64_t)p.split_tiles * p.k_splits : tiles;
}

// ------------------------------------------------------------------------------------
// Operand-path probe (measurement only; entry point mmm_probe_lds_mfma).  The persistent 256x256
// kernel's K loop on operands that are already in LDS: each workgroup stages K tiles 0 and 1 of
// its first output tile into the two ring slots once (the kernels' staging map), then runs the
// kernel's own per-K-tile code -- ktile_body and ktile_last_step: the same MFMAs and fragment
// reads, at the same LDS addresses, in the same order -- over as many K tiles as its share of the
// M x N x K problem holds, alternating the slots as the ring does.  Left out: the refill loads (the
// last step's load hook is empty), their waits and the C stores.  With BARRIER the workgroup
// barrier stays where the kernel publishes the next K tile; without it the waves run
// unsynchronised (nothing writes the LDS after the staging, so nothing races).  Each thread
// writes the sum of its accumulators at the end.  A workgroup's accumulators see slot 0 (K 0..63
// of its first tile) and slot 1 (K 64..127) total/2 = tiles * K / 128 times each, so the sum of
// its threads' outputs is (total / 2) * (1^T A0)(B0 1), A0 = A[m0 .. m0+255][0 .. 127],
// B0 = B[0 .. 127][n0 .. n0+255] (exact for small integer inputs).
// ------------------------------------------------------------------------------------
template <class T, bool BARRIER>
__global__ __launch_bounds__(T::NT, T::OCC) void lds_mfma_probe_kernel(GemmProblem p, int tiles_m, int tiles_n,
                                                                       float* out) {
  __shared__ __attribute__((aligned(1024))) char lds[T::STAGES * T::STAGE];
  static_assert(T::STAGES == 2 && T::B_UNIFORM, "two ring slots, the uniform staging map");
  record_clock(p.clk, 0);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w / T::WGN, wn = w % T::WGN;
  const int K = p.K;
  const int64_t lda = p.lda, ldb = p.ldb;
  char LDS_AS* lds_base = (char LDS_AS*)lds;

  // staging of K tiles 0 and 1 of the first output tile, as the kernels stage them (thread
  // (w, lane) moves chunk slot r * NT + w * 64 + lane of each operand's rounds r)
  constexpr int RPA = T::NT / T::CA, RPB = T::NT / T::CB;
  int tm, tn;
  tile_of_block(blockIdx.x, tiles_m, tiles_n, 4, &tm, &tn);
  const int m0 = __builtin_amdgcn_readfirstlane(tm * T::BM), n0 = __builtin_amdgcn_readfirstlane(tn * T::BN);
  {
    const int a_row0 = w * (64 / T::CA) + lane / T::CA;
    const int a_kc = 8 * ((lane % T::CA) ^ T::swz_a(a_row0));
    const int b_row0 = w * (64 / T::CB) + lane / T::CB;
    const int b_nc = 8 * ((lane % T::CB) ^ T::swz_bk(b_row0));
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const i32x4 ra = make_rsrc(p.A + (int64_t)m0 * lda + s * T::BK,
                                 clip_records(((int64_t)(p.M - 1 - m0) * lda + K - s * T::BK) * 2));
      const i32x4 rb = make_rsrc(p.B + (int64_t)s * T::BK * ldb + n0,
                                 clip_records(((int64_t)(K - 1 - s * T::BK) * ldb + p.N - n0) * 2));
      const uint32_t a_dst = lds_addr_of(lds_base) + s * T::STAGE + w * 64 * 16, b_dst = a_dst + T::A_BYTES;
#pragma unroll
      for (int r = 0; r < T::RA; ++r)
        dma_b128(a_dst + r * T::NT * 16, ra, (uint32_t)(((a_row0 + r * RPA) * lda + a_kc) * 2));
#pragma unroll
      for (int r = 0; r < T::RB; ++r)
        dma_b128(b_dst + r * T::NT * 16, rb, (uint32_t)(((b_row0 + r * RPB) * ldb + b_nc) * 2));
    }
    wait_vmcnt<0>();
  }
  block_sync();

  // fragment read offsets (as gemm_nn_kernel)
  uint32_t a_off[kMaxOff] = {};
#pragma unroll
  for (int kk = 0; kk < T::KSTEPS; ++kk)
#pragma unroll
    for (int ph = 0; ph < T::APAR; ++ph) {
      const int m = wm * T::TM + ph * T::MF + (lane % T::MF);
      const int chunk = (T::KK / 8) * kk + lane / T::MF;
      a_off[kk * T::APAR + ph] = m * T::BK * 2 + (chunk ^ T::swz_a(m)) * 16;
    }
  uint32_t b_off[kMaxOff] = {};
  {
    const int k = 8 * (lane / T::MF) + ((lane >> 2) & 3);
#pragma unroll
    for (int nb = 0; nb < T::FN; ++nb) {
      const int n = wn * T::TN + 16 * nb + 4 * (lane & 3);
      b_off[nb] = k * T::BN * 2 + (((n >> 3) ^ T::swz_bk(k)) * 16) + (n & 7) * 2;
    }
  }
  static_assert(T::MF == 16, "the 16x16x32 tile's fragment map");

  // this workgroup's K tiles: its output tiles b, b + grid, ... times K / BK each
  const int mine = (tiles_m * tiles_n - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x;
  const int total = __builtin_amdgcn_readfirstlane(mine * (K / T::BK));
  AccT<T> acc[T::FM][T::FN];
#pragma unroll
  for (int i = 0; i < T::FM; ++i)
#pragma unroll
    for (int j = 0; j < T::FN; ++j) acc[i][j] = AccT<T>{};
  Frags<T> f[2];
  load_frags<T, false>(lds_base, lds_base + T::A_BYTES, a_off, b_off, 0, f[0]);
  int cur = 0;
  for (int t = 0; t < total; ++t) {
    ktile_body<T, false>(lds_base + cur * T::STAGE, a_off, b_off, f, acc);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (BARRIER) block_sync();
    cur ^= 1;
    ktile_last_step<T, false>(lds_base + cur * T::STAGE, a_off, b_off, f, acc, 0, [](int, int) {});
  }
  float keep = 0.0f;
#pragma unroll
  for (int i = 0; i < T::FM; ++i)
#pragma unroll
    for (int j = 0; j < T::FN; ++j) keep += acc[i][j][0] + acc[i][j][1] + acc[i][j][2] + acc[i][j][3];
  out[(int64_t)blockIdx.x * T::NT + tid] = keep;
  record_clock(p.clk, 2);
}

hipError_t launch_lds_mfma_probe(const GemmProblem& p, bool barrier, float* out, hipStream_t stream) {
  using T = Tile256;
  const int tiles_m = p.M / T::BM, tiles_n = p.N / T::BN;
  const int64_t tiles = (int64_t)tiles_m * tiles_n;
  const int grid = (int)(tiles < 256 ? tiles : 256);
  if (barrier)
    hipLaunchKernelGGL((lds_mfma_probe_kernel<T, true>), dim3(grid), dim3(T::NT), 0, stream, p, tiles_m, tiles_n, out);
  else
    hipLaunchKernelGGL((lds_mfma_probe_kernel<T, false>), dim3(grid), dim3(T::NT), 0, stream, p, tiles_m, tiles_n, out);
  return hipGetLastError();
}

bool gemm_nn_persistent(const GemmProblem& p0, int tile_id) {
  if (tile_id != kTile256x256 && tile_id != kTile192x192) return false;
  GemmProblem p = p0;
  p.c_vec4 = (uintptr_t)p.C % 4 == 0;
  p.tail_regs = !tail_aligned(p);
  p.k_splits = gemm_nn_split(p, tile_id).splits;
  if (tile_id == kTile192x192) return p.k_splits <= 1 && persistent_ok<DmaTile<192, 192>>(p);
  return persistent_ok(p);
}

hipError_t launch_gemm_nn(const GemmProblem& p0, int tile_id, hipStream_t stream) {
  GemmProblem p = p0;
  // 16-byte stores of C need only 4-byte alignment on gfx950 (rows of an odd ldc included)
  p.c_vec4 = (uintptr_t)p.C % 4 == 0;
  p.tail_regs = !tail_aligned(p);
  p.k_splits = 1;
  p.split_tiles = 0;
  p.partials = nullptr;
  const TileSplit sp = gemm_nn_split(p, tile_id);
  if (sp.splits > 1 && p.ws && p.ws_bytes >= gemm_nn_workspace_bytes(p, tile_id))
    p.k_splits = sp.splits, p.split_tiles = sp.tiles, p.partials = p.ws;  // else unsplit
  switch (tile_id) {
    case kTile256x256:
      if (persistent_ok(p)) {
        using TP = DmaTile<256, 256>;
        // Non-temporal C stores: the persistent grid stores a tile's C while its next tile's
        // operand loads run, and L2-allocating stores would evict the operand panels other
        // workgroups of the XCD are about to read.  As half-line stores that won only when each
        // tile's K loop is long (measured on MI355X: 12288^2 x 4096 +6.7%, 8192^3 +1.6-2.8%,
        // 8192^2 x 2048 -7.1%, 16384 x 8192 x 1024 -9.3%); as whole lines (store_wave_tile_lines)
        // they win at every K (against L2-allocating half lines: 8192^2 x 2048 +8%, 12288^2 x
        // 2048 +5.2%, 8192^2 x 1024 +4.2-4.8%, 16384 x 8192 x 1024 +4.2%).  16-byte-aligned C
        // rows only.
        const int tiles_m = p.M / TP::BM, tiles_n = p.N / TP::BN;
        const bool nt = ((uintptr_t)p.C & 15) == 0 && p.ldc % 4 == 0 &&
                        (c_lines_all<TP>() || p.K >= kNtMinK);
        if (p.k_splits <= 1) {
          if (nt)
            hipLaunchKernelGGL((gemm_nn_persistent_kernel<TP, true>), dim3(256), dim3(TP::NT), 0, stream, p, tiles_m,
                               tiles_n);
          else
            hipLaunchKernelGGL((gemm_nn_persistent_kernel<TP, false>), dim3(256), dim3(TP::NT), 0, stream, p, tiles_m,
                               tiles_n);
          return hipGetLastError();
        }
        const LaunchPair pair(p.partials);
        if (nt)
          hipLaunchKernelGGL((gemm_nn_persistent_split_kernel<TP, true>), dim3(256), dim3(TP::NT), 0, stream, p, tiles_m,
                             tiles_n);
        else
          hipLaunchKernelGGL((gemm_nn_persistent_split_kernel<TP, false>), dim3(256), dim3(TP::NT), 0, stream, p, tiles_m,
                             tiles_n);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        // the last round's K-split pieces ran as the grid's final items: sum their partials
        const int64_t tiles = (int64_t)tiles_m * tiles_n;
        constexpr int64_t per_tile = TP::BM * TP::BN / 4 / 256;  // blocks of 256 float4s per tile
        hipLaunchKernelGGL((reduce_tiles_kernel<TP::BM, TP::BN>), dim3((unsigned)(p.split_tiles * per_tile)), dim3(256),
                           0, stream, p, tiles_m, tiles_n, (int)(tiles - p.split_tiles), p.k_splits);
        return hipGetLastError();
      }
      return dma_ok(p, 256) ? launch_nn<DmaTile<256, 256>, false>(p, stream)
                            : launch_nn<RegTile<256, 256>, true>(p, stream);
    case kTile128x256:
      return dma_ok(p, 128) ? launch_nn<DmaTile<128, 256>, false>(p, stream)
                            : launch_nn<RegTile<128, 256>, true>(p, stream);
    case kTile256x128:
      return dma_ok(p, 256) ? launch_nn<DmaTile<256, 128>, false>(p, stream)
                            : launch_nn<RegTile<256, 128>, true>(p, stream);
    case kTile128x128:
      if (!dma_ok(p, 128)) return launch_nn<RegTile<128, 128>, true>(p, stream);
      return launch_blocks(p, 128, 128) <= 256 ? launch_nn<DeepTile128, false>(p, stream)
                                                : launch_nn<DmaTile<128, 128>, false>(p, stream);
    case kTile64x64:
      return dma_ok(p, 64) ? launch_nn<DmaTile<64, 64>, false>(p, stream) : launch_nn<RegTile<64, 64>, true>(p, stream);
    case kTile192x192:
      if (p.k_splits <= 1 && persistent_ok<DmaTile<192, 192>>(p)) {
        using TP = DmaTile<192, 192>;
        const int tiles_m = p.M / TP::BM, tiles_n = p.N / TP::BN;
        // non-temporal C as for the 256x256 tile; this tile's third block of a row is stored as
        // half lines, and at short K its non-temporal stores lose (6144^2 x 2048 -2.9%,
        // 3072 x 6144 x 2048 -3.7% with them at every K; long K: 6144^3 +1.2%)
        const bool nt = ((uintptr_t)p.C & 15) == 0 && p.ldc % 4 == 0 &&
                        (c_lines_all<TP>() || p.K >= kNtMinK);
        if (nt)
          hipLaunchKernelGGL((gemm_nn_persistent_kernel<TP, true>), dim3(256), dim3(TP::NT), 0, stream, p, tiles_m,
                             tiles_n);
        else
          hipLaunchKernelGGL((gemm_nn_persistent_kernel<TP, false>), dim3(256), dim3(TP::NT), 0, stream, p, tiles_m,
                             tiles_n);
        return hipGetLastError();
      }
      // the register-staged path has no 192x192 instantiation: 128x128 tiles compute the same C
      return dma_ok(p, 192) ? launch_nn<DmaTile<192, 192>, false>(p, stream)
                            : launch_nn<RegTile<128, 128>, true>(p, stream);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace mmm
