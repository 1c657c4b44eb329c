// Second MFMA mainloop for gfx950 (MI355X), 16-bit operands only: four waves, each owning 128 x 128 of a
// 256 x 256 workgroup tile as 8 x 8 blocks of v_mfma_f32_16x16x32.
//
// Why a second one (measured on N(0,1) x N(0,0.02) operands, 16384 x 16384 x 3584, no epilogue, same box):
// the eight-wave 32x32x16 loop of gemm_core.hpp reaches 1.34 PFLOP/s, this one 1.48.  With such data the chip is
// power-limited (a register-resident MFMA loop runs at 1.83 PFLOP/s with 32x32x16 and 1.97 with 16x16x32,
// against 2.48 on all-zero operands), so what counts is energy per FLOP: the 16x16x32 shape moves a fifth less
// register data per FLOP, and a 128 x 128 wave tile needs a third fewer LDS operand reads than 64 x 128.
//
// The accumulators (256 registers per lane) live in AGPRs, the operand fragments (two k-steps of 8 + 8
// fragments, 128 registers) in VGPRs.  The MFMAs and the LDS reads are inline assembly: the compiler moves
// accumulators between the two register classes otherwise, and it cannot interleave what it does not order.
// Consequently the s_waitcnt for the reads are placed by hand (LDS reads return in order).
//
// LDS ring: the split ring of gemm_core.hpp (five half slabs of 32 KB, the B operand early), one workgroup
// barrier per slab, placed between its two k-steps.
//
// Accumulator layout of one 16 x 16 block: lane l holds column n = l % 16 and rows m = 4 * (l / 16) + r,
// r = 0..3.  Block (i, j) of a wave covers rows 16 i .. and columns 16 j .. of its 128 x 128.
#pragma once
#include <type_traits>
#include <utility>

#include "gemm_core.hpp"

namespace lce {

template <typename T>
struct Mma16;
template <>
struct Mma16<bf16_t> {
  static LCE_DEV void run(f32x4_t& acc, const u32x4_t& a, const u32x4_t& b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
  }
  static LCE_DEV void first(f32x4_t& acc, const u32x4_t& a, const u32x4_t& b) {  // acc = a b
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc) : "v"(a), "v"(b));
  }
  static LCE_DEV void over(f32x4_t& acc, const u32x4_t& a, const u32x4_t& b) {  // the same, in the registers of what acc was
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "+a"(acc) : "v"(a), "v"(b));
  }
};
template <>
struct Mma16<f16_t> {
  static LCE_DEV void run(f32x4_t& acc, const u32x4_t& a, const u32x4_t& b) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
  }
  static LCE_DEV void first(f32x4_t& acc, const u32x4_t& a, const u32x4_t& b) {  // acc = a b
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "=a"(acc) : "v"(a), "v"(b));
  }
  static LCE_DEV void over(f32x4_t& acc, const u32x4_t& a, const u32x4_t& b) {  // the same, in the registers of what acc was
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, 0" : "+a"(acc) : "v"(a), "v"(b));
  }
};

template <int... Is, typename F>
LCE_DEV void static_for(std::integer_sequence<int, Is...>, F&& f) {
  (f(std::integral_constant<int, Is>{}), ...);
}

// TRANS_: 0 both operands K-contiguous (row-major A[m][k], B[n][k]); 1 both K-major in memory, A[k][m] and
// B[k][n], fetched with the transposing LDS read (two ds_read_b64_tr_b16 per fragment); 2 only A K-major (mixed).
// NBN_: 16-column blocks per wave along the MFMA columns (tokens): 8 for tiles 256 columns wide, 6 for 192, 5 and 7 for the last of a
// row of tiles (ragged token counts: less work for padding; the loop itself runs a few per cent below the square tile's rate).
// A_EARLY_: the ring's early operand (see main) is A instead of B.
// TERMS_: products per slab.  1: the operands are what they are.  6: fp32 operands, each held as three bfloat16 planes
// x = x1 + x2 + x3 (exact: 3 x 8 significant bits); a slab is multiplied as a1 b3 + a1 b2 + a2 b2 + a2 b1 + a1 b1 + a3 b1 into
// the same fp32 accumulators (main6).  What is left out, a2 b3 + a3 b2 + a3 b3, is below 2^-26 of |a b|, a quarter of what rounding
// ONE fp32 product or partial sum costs, and the products themselves are exact.  Six bfloat16 MFMAs take six sixteenths
// of the matrix pipe's time of the fp32 one.
// A_ONCE_: the loads of A are marked non-temporal (A is read once, or nearly, and larger than the caches).
// NBM_: 16-row blocks per wave along the MFMA rows: 8 for tiles of 256 rows, 7 for 224 (A K-major only: hidden_tile).
template <typename TIN_, int TRANS_ = 0, int NBN_ = 8, int A_EARLY_ = 0, int TERMS_ = 1, int A_ONCE_ = 0, int NBM_ = 8>
struct GemmCfg16 {
  typedef TIN_ TIN;
  static_assert(sizeof(TIN_) == 2, "16-bit operands");
  static constexpr bool CORE16 = true;
  static_assert(NBN_ == 8 || TRANS_ != 1, "both operands K-major: square tiles");
  static constexpr int BM = 32 * NBM_, BN = 32 * NBN_, BKB = 128, BK = 64, NSTAGE = 5, SPLIT = 2, TRANS = TRANS_;
  static constexpr bool A_EARLY = A_EARLY_ != 0, A_ONCE = A_ONCE_ != 0;
  static constexpr int TERMS = TERMS_;
  static_assert(TERMS_ == 1 || TERMS_ == 6, "products per slab");
  static constexpr int WAVES_M = 2, WAVES_N = 2, NW = 4, NTHREADS = 256;
  static constexpr int WM = 16 * NBM_, WN = 16 * NBN_;
  static constexpr int NB = NBM_, NBN = NBN_;        // 16-row / 16-column blocks of a wave tile
  static constexpr int STAGE_BYTES = 32768;          // one operand's slab: 256 rows x 128 bytes (or BN rows), or 64 k-rows x 512 bytes
  static constexpr int LDS_BYTES = NSTAGE * STAGE_BYTES;
  static constexpr int HL = 8, HLB = NBN_;           // wave-wide 16-byte-per-lane loads per wave and half slab of A, of B
};

// The lane number, worked out anew where it is asked for.  A kernel that walks tiles has no register to spare across its K
// loop: what follows from the lane number and is wanted at every tile would be kept in scratch memory, and a load from
// there waits for every load and store issued before it.
LCE_DEV int lane_anew() {
  uint32_t zero = 0;
  asm volatile("" : "+s"(zero));
  return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, zero));
}

template <typename Cfg>
struct GemmCore16 {
  typedef typename Cfg::TIN TIN;
  static constexpr int NB = Cfg::NB, NBN = Cfg::NBN, HL = Cfg::HL, HLB = Cfg::HLB, SLOT = Cfg::STAGE_BYTES;
  static constexpr bool TN = Cfg::TRANS == 1, AE = Cfg::A_EARLY;
  static constexpr bool TA = Cfg::TRANS != 0, TB = Cfg::TRANS == 1;  // which operand is K-major in memory

  const char* a_base;
  const char* b_base;
  uint32_t va[HL], vb[HLB];  // per-lane byte offsets of the loads inside slab 0
  uint32_t a_rd, b_rd;      // per-lane LDS read offsets inside a slot (block 0, k-step 0)
  int64_t a_slab, b_slab;   // bytes from one K slab to the next in memory
  int64_t a_plane = 0, b_plane = 0;  // TERMS == 6: bytes from plane to plane
  int wave, lane, wave_m, wave_n;
  // mixed mode: row of A inside a slab that each load fetches, A's row stride in bytes and the number of its rows that exist
  uint32_t va_tail[HL];         // mixed mode: va of the last slab of A that has rows, rows beyond them clamped
  int64_t a_ks_full, a_ks_last;  // slabs below a_ks_full have all their 64 rows; a_ks_last: the last slab with any

  LCE_DEV void set_lane() {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lane = threadIdx.x & 63;
    wave_m = wave >> 1;
    wave_n = wave & 1;
  }

  // Row-major operands.  MFMA rows come from A (rows m0 .. of an M-row matrix), MFMA columns from B (rows n0 .. of
  // an N-row matrix); rows beyond a matrix are clamped to its last row (the epilogue discards them).  With `b_rows`,
  // row n of the B operand is B[b_rows[n]] (a gather; every row's byte offset from B must then fit 32 bits).
  // LDS layout of a slab: row-major, 128 bytes per row, 16-byte chunk c of row r at position c ^ ((r / 2) % 8): the
  // 16 rows x 4 chunks that a quarter wave reads for one fragment then fall into 64 different banks.
  LCE_DEV void init(const TIN* A, int64_t lda, int64_t m0, int64_t M, const TIN* B, int64_t ldb, int64_t n0, int64_t N,
                    const int* b_rows = nullptr) {
    static_assert(Cfg::BM == 256, "row-major A: tiles of 256 rows");
    set_lane();
    a_base = reinterpret_cast<const char*>(A + m0 * lda);
    b_base = reinterpret_cast<const char*>(b_rows ? B : B + n0 * ldb);
    a_slab = b_slab = Cfg::BKB;
    const int rows_a = (int)((M - m0) < (int64_t)Cfg::BM ? (M - m0) : (int64_t)Cfg::BM);
    const int rows_b = (int)((N - n0) < (int64_t)Cfg::BN ? (N - n0) : (int64_t)Cfg::BN);
    const int lr = lane >> 3, pc = lane & 7;
#pragma unroll
    for (int j = 0; j < HL; ++j) {
      const int row = (j * Cfg::NW + wave) * 8 + lr;
      const int c = pc ^ ((row >> 1) & 7);
      const int ra = row < rows_a ? row : rows_a - 1;
      va[j] = (uint32_t)((int64_t)ra * lda * 2) + (uint32_t)(c * 16);
      if (j < HLB) {
        const int rb = row < rows_b ? row : rows_b - 1;
        const int64_t gb = b_rows ? (int64_t)b_rows[n0 + rb] : (int64_t)rb;
        vb[j < HLB ? j : 0] = (uint32_t)(gb * ldb * 2) + (uint32_t)(c * 16);
      }
    }
    const int r16 = lane & 15, g = lane >> 4;
    const uint32_t off = (uint32_t)(r16 * 128 + ((g ^ (r16 >> 1)) * 16));
    a_rd = (uint32_t)(wave_m * Cfg::WM * 128) + off;
    b_rd = (uint32_t)(wave_n * Cfg::WN * 128) + off;
  }

  // K-major operands: A[k][m0 + 0..BM), B[k][n0 + 0..256) with row strides lda / ldb (elements); both must be
  // allocated in whole tiles.  A ring slot holds 64 k-rows of 512 bytes; chunk c of row r sits at
  // position c ^ swz(r), swz(r) = 4 (r % 4) ^ 2 ((r / 8) % 2), so that the eight k-rows that half a wave touches
  // in one transposing read fall into different banks.
  // The transposing read: in each group of 16 lanes, lane 4e + q supplies the address of X[k0 + e][x0 + 4q ..] and
  // lane i receives X[k0 .. k0+3][x0 + i]; group g of the wave takes the k-octet 8g of the 32 k-values of a k-step,
  // and a second read 4 rows further completes the octet.
  // With b_pcol, B lies in panels of 64 columns, b_pcol elements apart (ldb = 64: the rows of a panel follow each other).
  LCE_DEV void init_tn(const TIN* A, int64_t lda, int64_t m0, const TIN* B, int64_t ldb, int64_t n0, int64_t b_pcol = 0) {
    set_lane();
    a_base = reinterpret_cast<const char*>(A + m0);
    b_base = reinterpret_cast<const char*>(b_pcol ? B + (n0 >> 6) * b_pcol : B + n0);
    a_slab = 64 * lda * 2;
    b_slab = 64 * ldb * 2;
#pragma unroll
    for (int j = 0; j < HL; ++j) {
      const int row = (j * Cfg::NW + wave) * 2 + (lane >> 5);
      const int c = (lane & 31) ^ tn_swz(row);
      va[j] = (uint32_t)((int64_t)row * lda * 2) + (uint32_t)(a_chunk(c) * 16);
      vb[j] = (uint32_t)((int64_t)row * ldb * 2) + (b_pcol ? (uint32_t)((c >> 3) * b_pcol * 2) + (uint32_t)((c & 7) * 16) : (uint32_t)(c * 16));
    }
    reads_tn(lane);
  }
  LCE_DEV void reads_tn(int ln) {
    const int g = ln >> 4, e = (ln & 15) >> 2, q = ln & 3;
    const int row = 8 * g + e;  // (k-step 0, first half of the octet)
    const uint32_t in_row = (uint32_t)((((q >> 1) ^ tn_swz(row)) * 16) + (q & 1) * 8);
    a_rd = (uint32_t)(row * 512 + wave_m * 256) + in_row;
    b_rd = (uint32_t)(row * 512 + wave_n * Cfg::WN * 2) + in_row;
  }
  // 16-byte chunk of a row of a K-major A that chunk c of the LDS row holds: each wave's columns begin at a multiple of 256 bytes
  // there, whatever their number (the blocks' offsets are XORed in); what is left over repeats the last chunk
  static LCE_DEV int a_chunk(int c) {
    if (NB == 8) return c;
    const int in = c & 15;
    return (c >> 4) * 2 * NB + (in < 2 * NB ? in : 2 * NB - 1);
  }
  // another tile of the same matrices after init_tn
  LCE_DEV void move_tn(const TIN* A, int64_t m0, const TIN* B, int64_t n0, int64_t b_pcol) {
    a_base = reinterpret_cast<const char*>(A + m0);
    b_base = reinterpret_cast<const char*>(b_pcol ? B + (n0 >> 6) * b_pcol : B + n0);
  }
  static LCE_DEV int tn_swz(int row) { return ((row & 3) * 4) ^ (((row >> 3) & 1) * 2); }

  // Mixed: A[k][m0 + 0..BM) K-major as in init_tn, B row-major as in init (rows n0 .. of an N-row matrix, clamped).
  // LDS row r of an A slab holds memory row perm(r) of the slab (perm: a permutation of 0..63, the order in which B's
  // K index was stored); rows at or beyond `kvalid` > 0 are replaced by rows that exist (B is zero there), and columns at
  // or beyond `mcols` (a last tile that is not full) by the row's first chunk: in bounds, and they
  // feed only results that the epilogue discards.  b_slab_bytes: from one K slab of B to the next (its rows' 128 bytes for
  // rows of ldb elements; a panel where B lies in panels of 64 columns).
  template <typename Perm>
  LCE_DEV void init_mixed(const TIN* A, int64_t lda, int64_t m0, int64_t mcols, int64_t kvalid, Perm perm, const TIN* B, int64_t ldb,
                          int64_t n0, int64_t N, int64_t b_slab_bytes) {
    static_assert(Cfg::TRANS == 2, "mixed mode");
    set_lane();
    a_base = reinterpret_cast<const char*>(A + m0);
    b_base = reinterpret_cast<const char*>(B + n0 * ldb);
    a_slab = 64 * lda * 2;
    b_slab = b_slab_bytes;
    a_ks_full = kvalid / 64;
    a_ks_last = (kvalid - 1) / 64;
    const int last_row = (int)(kvalid - 1 - a_ks_last * 64);  // of slab a_ks_last
    const int rows_b = (int)((N - n0) < (int64_t)Cfg::BN ? (N - n0) : (int64_t)Cfg::BN);
    const int lr = lane >> 3, pc = lane & 7;
#pragma unroll
    for (int j = 0; j < HL; ++j) {
      const int rowa = (j * Cfg::NW + wave) * 2 + (lane >> 5);
      const int ca = a_chunk((lane & 31) ^ tn_swz(rowa));
      const int prow = (int)perm(rowa);
      const uint32_t col = (uint32_t)(((int64_t)ca * 8 < mcols ? ca : 0) * 16);
      va[j] = (uint32_t)((int64_t)prow * lda * 2) + col;
      va_tail[j] = (uint32_t)((int64_t)(prow < last_row ? prow : last_row) * lda * 2) + col;
      if (j < HLB) {
        const int rowb = (j * Cfg::NW + wave) * 8 + lr;
        const int cb = pc ^ ((rowb >> 1) & 7);
        const int rb = rowb < rows_b ? rowb : rows_b - 1;
        vb[j < HLB ? j : 0] = (uint32_t)((int64_t)rb * ldb * 2) + (uint32_t)(cb * 16);
      }
    }
    const int g = lane >> 4, e = (lane & 15) >> 2, q = lane & 3;
    const int row = 8 * g + e;
    a_rd = (uint32_t)(row * 512 + wave_m * 256) + (uint32_t)((((q >> 1) ^ tn_swz(row)) * 16) + (q & 1) * 8);
    const int r16 = lane & 15;
    b_rd = (uint32_t)(wave_n * Cfg::WN * 128) + (uint32_t)(r16 * 128 + ((g ^ (r16 >> 1)) * 16));
  }

  // ---- instruction-level pieces ----------------------------------------------------------------------------
  // load j of one operand's half slab number `ks` into ring slot `slot`
  LCE_DEV void dma(char* lds, int slot, int64_t ks, bool is_b, int j) const {
    char* dst = lds + slot * SLOT + (j * Cfg::NW + wave) * 1024;
    const char* src;
    if (Cfg::TRANS == 2 && !is_b) {
      // slabs with rows that do not exist take the last slab that has any, with its rows clamped (branch-free: the
      // hand-placed schedule of a k-step must stay one basic block)
      const bool tail = ks >= a_ks_full;
      src = a_base + (tail ? a_ks_last : ks) * a_slab + (tail ? va_tail[j] : va[j]);
    } else {
      src = (is_b ? b_base + ks * b_slab + vb[j] : a_base + ks * a_slab + va[j]);
    }
    if (Cfg::A_ONCE && !is_b) __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)dst, 16, 0, kBufNonTemporal);  // (constants after inlining)
    else __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)dst, 16, 0, 0);
  }

  // Fragments are read in the order a0, b0 .. b(NBN-1), a1 .. a7 (F = 0 .. NF-1): the MFMAs walk the A blocks in the outer
  // loop, so the first row of NBN needs a0 and every b, the later rows one more a each.
  static constexpr int NF = NB + NBN;
  static constexpr bool frag_is_a(int f) { return f == 0 || f > NBN; }
  static constexpr int frag_blk(int f) { return f == 0 ? 0 : (f <= NBN ? f - 1 : f - NBN); }
  static constexpr int CA = TA ? 2 : 1, CB = TB ? 2 : 1;  // LDS instructions per fragment of each operand
  // ra / rb: LDS address of the slot plus a_rd / b_rd; S: k-step inside the slab
  template <int F, int S>
  LCE_DEV void read_frag(uint32_t ra, uint32_t rb, u32x4_t (&af)[NB], u32x4_t (&bf)[NBN]) const {
    read_block<frag_is_a(F), frag_blk(F), S>(ra, rb, af, bf);
  }
  template <bool is_a, int blk, int S>
  LCE_DEV void read_block(uint32_t ra, uint32_t rb, u32x4_t (&af)[NB], u32x4_t (&bf)[NBN]) const {
    u32x4_t v;
    if constexpr (is_a ? TA : TB) {
      // block: 16 columns = 32 bytes further, inside the swizzled chunk bits; k-step: 32 rows; second half: 4 rows
      const uint32_t base = (is_a ? ra : rb) ^ (uint32_t)(blk * 32);
      const u32x2_t lo = tr_read<S * 16384>(base), hi = tr_read<S * 16384 + 2048>(base);
      v = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
    } else {
      v = lds_read16<blk * 2048>((is_a ? ra : rb) ^ (uint32_t)(S * 64));
    }
    if constexpr (is_a) af[blk] = v;
    else bf[blk] = v;
  }

  // LDS instructions issued up to and including fragment f of a k-step (f = -1: none)
  static constexpr int upto(int f) { return f < 0 ? 0 : (f == 0 ? CA : (f <= NBN ? CA + CB * f : CA + NBN * CB + CA * (f - NBN))); }
  static constexpr int ALLI = NB * CA + NBN * CB;
  // fragments of the next k-step issued before MFMA m of this one: one after each even MFMA of the first half
  static constexpr int frags_before(int m) { return (m + 1) / 2 > NF ? NF : (m + 1) / 2; }

  // One k-step: NB x NBN MFMAs on (af, bf); the NF fragment reads of the next k-step (from ra_n / rb_n, k-step S_N) and the
  // global->LDS loads of a half slab are dealt between them.  WAIT: the fragments of this step were read during the previous step
  // and may still be in flight.  DMA_B: the loads fetch the B operand's half slab `dma_ks` (else A's) into `dma_slot`; with
  // FROM, the half slab at `dma_from` instead.  FIRST: the accumulators start here.
  template <bool WAIT, int S_N, bool DMA_B, bool FROM = false, bool FIRST = false>
  LCE_DEV void kstep(f32x4_t (&acc)[NB][NBN], const u32x4_t (&af)[NB], const u32x4_t (&bf)[NBN], uint32_t ra_n, uint32_t rb_n,
                     u32x4_t (&af_n)[NB], u32x4_t (&bf_n)[NBN], char* lds, int dma_slot, int64_t dma_ks,
                     const char* dma_from = nullptr) const {
    constexpr int DMAS = DMA_B ? HLB : HL, EVERY = NB * NBN / DMAS;
    static_assert(2 * NF <= NB * NBN && DMAS * EVERY <= NB * NBN && EVERY > 3, "one fragment read after every second MFMA");
    static_for(std::make_integer_sequence<int, NB * NBN>{}, [&](auto mc) {
      constexpr int m = decltype(mc)::value;
      constexpr int i = m / NBN, j = m % NBN;
      if constexpr (WAIT && (i == 0 || j == 0)) {
        constexpr int need = i == 0 ? 1 + j : NBN + i;  // the last fragment this MFMA depends on
        constexpr int allow = (ALLI - upto(need)) + upto(frags_before(m) - 1);
        wait_lgkm<(allow > 15 ? 15 : allow)>();
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (FIRST) Mma16<TIN>::first(acc[i][j], af[i], bf[j]);
      else Mma16<TIN>::run(acc[i][j], af[i], bf[j]);
      if constexpr ((m & 1) == 0 && m / 2 < NF) read_frag<m / 2, S_N>(ra_n, rb_n, af_n, bf_n);
      if constexpr (m % EVERY == 3 && m / EVERY < DMAS) {
        constexpr int j8 = m / EVERY;
        if constexpr (FROM)
          __builtin_amdgcn_global_load_lds((gptr_t)(dma_from + (DMA_B ? vb[j8] : va[j8])), (lptr_t)(lds + dma_slot * SLOT + (j8 * Cfg::NW + wave) * 1024),
                                           16, 0, 0);
        else dma(lds, dma_slot, dma_ks, DMA_B, j8);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  }

  template <int N>
  static LCE_DEV void wait_lgkm() { __builtin_amdgcn_s_waitcnt(0xC07F | (N << 8)); }
  template <int N>
  static LCE_DEV void wait_vm() {
    static_assert(N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt(((N & 0xF) | ((N >> 4) << 14)) | 0x0F70);
  }

  // Issues the loads of the first two slabs (half slabs E0 L0 E1 L1 into slots 0..3; E = the early operand).  LDS must be
  // free: every wave past its last read of the previous tile and its own loads drained (a workgroup barrier after main()).
  LCE_DEV void prologue(char* lds, int64_t K) const {
    if constexpr (Cfg::TERMS == 6) {
      fetch6<true>(lds, 0, 0, 2);
      fetch6<false>(lds, 1, 0, 0);
      fetch6<true>(lds, 2, 0, 1);
      fetch6<false>(lds, 3, 0, 1);
      fetch6<true>(lds, 4, 0, 0);
      return;
    }
    const int64_t last = K / Cfg::BK - 1;
#pragma unroll
    for (int hf = 0; hf < 4; ++hf) {
      const int64_t ks = hf / 2 < last ? hf / 2 : last;
#pragma unroll
      for (int j = 0; j < (((hf & 1) == 0) != AE ? HLB : HL); ++j) dma(lds, hf, ks, ((hf & 1) == 0) != AE, j);
    }
  }

  // The K loop (K a positive multiple of 64); prologue() must have been called for this tile, and no other vector memory
  // load may have been issued by this wave since (the waits count outstanding loads).  One operand is early (E: B, or A with
  // A_EARLY), the other late (L).  Slab i reads E from slot 2i % 5 and L from the next slot.  Its first k-step issues the
  // loads of E(i+2) into the slot that L(i-1) left; the barrier
  // between the two k-steps waits for slab i+1 (everything but those youngest loads) and for every wave's reads of slab
  // i; the second k-step then issues L(i+2) into E(i)'s slot and reads the first fragments of slab i+1.  So E has a slab and
  // a half to arrive and L one slab.  Past the end
  // of K the loader re-fetches the last slab into slots nobody reads (a branch-free body), drained at the end.
  LCE_DEV void main(char* lds, int64_t K, f32x4_t (&acc)[NB][NBN]) const {
    if constexpr (Cfg::TERMS == 6) return main6(lds, (int)(K / Cfg::BK), acc);
    const int nk = (int)(K / Cfg::BK);
    const int64_t last = nk - 1;
    wait_vm<HL + HLB>();  // slab 0 has landed
    __builtin_amdgcn_s_barrier();
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(lds);
    u32x4_t af[2][NB], bf[2][NBN];
    static_for(std::make_integer_sequence<int, NF>{}, [&](auto fc) {
      read_frag<decltype(fc)::value, 0>(lds0 + (AE ? 0 : SLOT) + a_rd, lds0 + (AE ? SLOT : 0) + b_rd, af[0], bf[0]);
    });
    int se = 0;  // slot of this slab's early half; its late half is in the next slot
    auto slab = [&](auto first, int it) {
      constexpr bool FIRST = decltype(first)::value;
      const int sl = se + 1 >= 5 ? se + 1 - 5 : se + 1;
      const int ne = se + 2 >= 5 ? se + 2 - 5 : se + 2;
      const int nl = se + 3 >= 5 ? se + 3 - 5 : se + 3;
      const int fr = se + 4 >= 5 ? se + 4 - 5 : se + 4;  // free slot: takes E(it+2)
      const int64_t ks = it + 2 < last ? it + 2 : last;
      kstep<true, 1, !AE, false, FIRST>(acc, af[0], bf[0], lds0 + (AE ? se : sl) * SLOT + a_rd, lds0 + (AE ? sl : se) * SLOT + b_rd, af[1], bf[1], lds,
                                        fr, ks);
      wait_vm<AE ? HL : HLB>();  // slab it+1 has landed; E(it+2) may still be in flight
      wait_lgkm<0>();            // this wave's reads of slab it have returned
      __builtin_amdgcn_s_barrier();
      kstep<false, 0, AE>(acc, af[1], bf[1], lds0 + (AE ? ne : nl) * SLOT + a_rd, lds0 + (AE ? nl : ne) * SLOT + b_rd, af[0], bf[0], lds, se, ks);
      se = ne;
    };
    // (the first slab starts the accumulators: zeroing them beforehand takes 512 instructions and, while they are ordinary values
    // to the compiler, the registers of everything else that lives across the loop)
    slab(std::true_type{}, 0);
    for (int it = 1; it < nk; ++it) slab(std::false_type{}, it);
    wait_vm<0>();    // drain the redundant tail fetches before LDS is reused
    wait_lgkm<0>();  // and the reads of the slab after the last
    retire(acc);
  }

  // ---- TERMS == 6: a slab's six products -----------------------------------------------------------------------
  // Consecutive products share an operand: a1 b3, a1 b2, a2 b2, a2 b1, a1 b1, a3 b1.  Its fragments stay in registers, so that a
  // slab of K is seven half slabs read from LDS (a1 twice) and six fetched, where products that each bring both operands are
  // twelve and twelve.  What that saves is energy: on such data the loop runs at the socket's power cap.  Against products that each
  // bring both, H=896: 1024 tokens, forward 1422 -> 1287 us, forward + backward 5.84 -> 5.09 ms; 400 tokens 749 and 2761 for 806 and 2995;
  // H=5120, 1000 tokens, forward 7.83 -> 7.00 ms.
  // The fragments a k-step reads for the next one, WHAT: 1 of A, 2 of B, 3 both in kstep's order.
  template <int WHAT>
  struct Reads {
    static constexpr int N = WHAT == 3 ? NF : WHAT == 1 ? NB : NBN;
    static constexpr bool is_a(int f) { return WHAT == 3 ? frag_is_a(f) : WHAT == 1; }
    static constexpr int blk(int f) { return WHAT == 3 ? frag_blk(f) : f; }
    static constexpr int upto(int f) { return f < 0 ? 0 : WHAT == 3 ? GemmCore16::upto(f) : (f + 1) * (WHAT == 1 ? CA : CB); }
    static constexpr int before(int m) { return (m + 1) / 2 > N ? N : (m + 1) / 2; }
    // the last fragment that MFMA (i, j) is the first to depend on; -1: none
    static constexpr int need(int i, int j) {
      return WHAT == 3 ? (i == 0 ? 1 + j : j == 0 ? NBN + i : -1) : WHAT == 1 ? (j == 0 ? i : -1) : (i == 0 ? j : -1);
    }
  };
  // half slab `ks` of plane `which`, its address in scalar registers (the compiler otherwise keeps the planes' addresses per lane)
  struct Half6 {
    const char* base;
    bool tail;
  };
  template <bool IS_B>
  LCE_DEV Half6 half6(int ks, int which) const {
    const bool tail = Cfg::TRANS == 2 && !IS_B && ks >= a_ks_full;
    Half6 h = {IS_B ? b_base + ks * b_slab + which * b_plane : a_base + (tail ? a_ks_last : ks) * a_slab + which * a_plane, tail};
    asm volatile("" : "+s"(h.base));
    return h;
  }
  template <bool IS_B>
  LCE_DEV void load6(char* lds, int slot, Half6 h, int j) const {
    const uint32_t at = IS_B ? vb[j < HLB ? j : 0] : Cfg::TRANS == 2 && h.tail ? va_tail[j] : va[j];
    __builtin_amdgcn_global_load_lds((gptr_t)(h.base + at), (lptr_t)(lds + slot * SLOT + (j * Cfg::NW + wave) * 1024), 16, 0, 0);
  }
  template <bool IS_B>
  LCE_DEV void fetch6(char* lds, int slot, int ks, int which) const {
    const Half6 h = half6<IS_B>(ks, which);
#pragma unroll
    for (int j = 0; j < (IS_B ? HLB : HL); ++j) load6<IS_B>(lds, slot, h, j);
  }

  // One k-step.  CUR: what was read for it during the step before and may still be in flight (0: nothing).  NEXT: what is read for
  // the next one, k-step S_N of its product.  LOAD: 1 / 2: the half slab `from` of A / B is fetched into `slot`.
  template <int CUR, int NEXT, int S_N, int LOAD, bool FIRST = false>
  LCE_DEV void kstep6(f32x4_t (&acc)[NB][NBN], const u32x4_t (&af)[NB], const u32x4_t (&bf)[NBN], uint32_t ra_n, uint32_t rb_n,
                      u32x4_t (&af_n)[NB], u32x4_t (&bf_n)[NBN], char* lds = nullptr, int slot = 0, Half6 from = {}) const {
    typedef Reads<NEXT> Nx;
    constexpr int LOADS = LOAD == 1 ? HL : HLB, EVERY = NB * NBN / LOADS;
    static_assert(2 * NF <= NB * NBN && EVERY > 3, "one fragment read after every second MFMA");
    static_for(std::make_integer_sequence<int, NB * NBN>{}, [&](auto mc) {
      constexpr int m = decltype(mc)::value;
      constexpr int i = m / NBN, j = m % NBN;
      if constexpr (CUR != 0) {
        typedef Reads<CUR> Cu;
        if constexpr (Cu::need(i, j) >= 0) {
          constexpr int allow = Cu::upto(Cu::N - 1) - Cu::upto(Cu::need(i, j)) + Nx::upto(Nx::before(m) - 1);
          wait_lgkm<(allow > 15 ? 15 : allow)>();
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (FIRST) Mma16<TIN>::first(acc[i][j], af[i], bf[j]);
      else Mma16<TIN>::run(acc[i][j], af[i], bf[j]);
      if constexpr ((m & 1) == 0 && m / 2 < Nx::N) read_block<Nx::is_a(m / 2), Nx::blk(m / 2), S_N>(ra_n, rb_n, af_n, bf_n);
      if constexpr (LOAD != 0 && m % EVERY == 3 && m / EVERY < LOADS) load6<LOAD == 2>(lds, slot, from, m / EVERY);
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  // Half slabs are fetched in the order b3 a1 b2 a2 b1 | a3 b3' a1' b2' a2' b1' | ..., each into the slot that the product before
  // has read for the last time (behind the barrier between a product's two k-steps), three to four products ahead of its own
  // first read.  The waits count the loads behind the half slab that the next product is the first to read.
  LCE_DEV void main6(char* lds, int nk, f32x4_t (&acc)[NB][NBN]) const {
    const int last = nk - 1;
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(lds);
    wait_vm<2 * HLB + HL>();
    __builtin_amdgcn_s_barrier();
    u32x4_t af[2][NB], bf[2][NBN];
    static_for(std::make_integer_sequence<int, NF>{}, [&](auto fc) {
      read_frag<decltype(fc)::value, 0>(lds0 + SLOT + a_rd, lds0 + b_rd, af[0], bf[0]);
    });
    int b3 = 0, a1 = 1, b2 = 2, a2 = 3, b1 = 4;  // slots; a3 follows b3
    auto meet = [&](auto in_flight) {  // every wave's loads but so many have landed, every wave's reads have returned
      constexpr int N = decltype(in_flight)::value;
      if constexpr (N >= 0) wait_vm<N>();
      wait_lgkm<0>();
      __builtin_amdgcn_s_barrier();
    };
    constexpr std::integral_constant<int, HL + HLB> two{};
    constexpr std::integral_constant<int, HL + 2 * HLB> three{};
    constexpr std::integral_constant<int, -1> all_here{};
    auto slab = [&](auto first, int it) {
      constexpr bool FIRST = decltype(first)::value;
      const int nx = it < last ? it + 1 : last;  // (past the end the last slab is fetched once more, into slots nobody reads)
      auto ra = [&](int slot) { return lds0 + slot * SLOT + a_rd; };
      auto rb = [&](int slot) { return lds0 + slot * SLOT + b_rd; };
      kstep6<3, 3, 1, 0, FIRST>(acc, af[0], bf[0], ra(a1), rb(b3), af[1], bf[1]);  // a1 b3
      meet(two);                                                                  // (b2)
      kstep6<0, 2, 0, 1>(acc, af[1], bf[1], 0, rb(b2), af[0], bf[0], lds, b3, half6<false>(it, 2));
      kstep6<2, 2, 1, 0>(acc, af[0], bf[0], 0, rb(b2), af[1], bf[1]);  // a1 b2
      meet(two);                                                      // (a2)
      kstep6<0, 1, 0, 2>(acc, af[1], bf[1], ra(a2), 0, af[0], bf[0], lds, b2, half6<true>(nx, 2));
      kstep6<1, 1, 1, 0>(acc, af[0], bf[0], ra(a2), 0, af[1], bf[1]);  // a2 b2
      meet(two);                                                      // (b1)
      kstep6<0, 2, 0, 1>(acc, af[1], bf[1], 0, rb(b1), af[0], bf[0], lds, a2, half6<false>(nx, 0));
      kstep6<2, 2, 1, 0>(acc, af[0], bf[0], 0, rb(b1), af[1], bf[1]);  // a2 b1
      meet(all_here);
      kstep6<0, 1, 0, 2>(acc, af[1], bf[1], ra(a1), 0, af[0], bf[0], lds, b1, half6<true>(nx, 1));
      kstep6<1, 1, 1, 0>(acc, af[0], bf[0], ra(a1), 0, af[1], bf[1]);  // a1 b1
      meet(three);                                                    // (a3)
      kstep6<0, 1, 0, 1>(acc, af[1], bf[1], ra(b3), 0, af[0], bf[0], lds, a1, half6<false>(nx, 1));
      kstep6<1, 1, 1, 0>(acc, af[0], bf[0], ra(b3), 0, af[1], bf[1]);  // a3 b1
      meet(two);                                                      // (b3', a1')
      kstep6<0, 3, 0, 2>(acc, af[1], bf[1], ra(a2), rb(b2), af[0], bf[0], lds, b3, half6<true>(nx, 0));
      const int was_b3 = b3, was_a1 = a1;
      b3 = b2;
      b2 = b1;
      b1 = was_b3;
      a1 = a2;
      a2 = was_a1;
    };
    slab(std::true_type{}, 0);
    for (int it = 1; it < nk; ++it) slab(std::false_type{}, it);
    wait_vm<0>();
    wait_lgkm<0>();
    retire(acc);
  }

  // The accumulators are read by ordinary instructions from here on: let the last MFMAs deliver.  They are inline assembly, so
  // the compiler knows nothing of their latency, and would be free to place a copy of an accumulator right behind the
  // statement that last wrote it, ahead of this wait (seen once, in a variant that zeroed the accumulators beforehand: copied
  // to scratch a few instructions behind the last MFMA, wrong statistics).  What keeps it from that is the chain of tied
  // operands from the first slab's products, which start the accumulators, through every k-step to stay(): there is no other
  // value to copy in between.  That it holds is checked on the listing of the built library
  // (tests/test_mfma_distance_on_cpu.py), not assumed.
  static LCE_DEV void retire(f32x4_t (&acc)[NB][NBN]) {
    asm volatile("s_nop 15\n\ts_nop 7" ::);
    stay(acc);
  }

  // The accumulators are in AGPRs at this point of the program (the compiler otherwise moves many of them into ordinary registers
  // as soon as a loop ends, ahead of their use, and what lived there into scratch memory).
  static LCE_DEV void stay(f32x4_t (&acc)[NB][NBN]) {
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < NBN; ++j) asm volatile("" : "+a"(acc[i][j]));
  }

  // the same for one block column, where the epilogues begin with it
  static LCE_DEV void stay_column(f32x4_t (&acc)[NB][NBN], int j) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NB; ++i) asm volatile("" : "+a"(acc[i][j]));
  }

  // ---- a workgroup that walks tiles: the K loops of successive tiles as one stream of slabs -------------------
  // The loads two slabs ahead of the end of a tile are those of the next tile's first slabs, and the fragments that the last
  // k-step reads are the next tile's first: between two tiles there is neither a drain nor a first load to wait for.
  struct Stream {
    u32x4_t af[NB], bf[NBN];  // the next slab's first fragments
    int sb;                   // slot of its B half
  };
  // prologue() of the first tile has been called, and nothing else was loaded since
  LCE_DEV void stream_begin(char* lds, Stream& s) const {
    wait_vm<HL + HLB>();
    __builtin_amdgcn_s_barrier();
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(lds);
    static_for(std::make_integer_sequence<int, NF>{}, [&](auto fc) {
      read_frag<decltype(fc)::value, 0>(lds0 + SLOT + a_rd, lds0 + b_rd, s.af, s.bf);
    });
    s.sb = 0;
  }
  // What slab `it` of nk fetches meanwhile: the slab two further on, beyond this tile's last (a_base / b_base) the first ones of
  // the next tile (a_next / b_next; this one's again when there is none).
  struct Ahead {
    const char *a, *b;
  };
  LCE_DEV Ahead stream_ahead(int it, int nk, const char* a_next, const char* b_next) const {
    const bool nx = it + 2 >= nk;
    const int ks = nx ? it + 2 - nk : it + 2;
    return {(nx ? a_next : a_base) + ks * a_slab, (nx ? b_next : b_base) + ks * b_slab};
  }
  static LCE_DEV int ring(int slot) { return slot >= 5 ? slot - 5 : slot; }

  // Slab `it` of a tile of nk >= 2 slabs.  Ring slot (s.sb + 4) % 5 is free when this returns.
  template <bool FIRST>
  LCE_DEV void stream_slab(char* lds, int it, int nk, f32x4_t (&acc)[NB][NBN], Stream& s, const char* a_next, const char* b_next) const {
    static_assert(Cfg::TRANS != 2 && NBN == 8 && !AE && Cfg::TERMS == 1 && !Cfg::A_ONCE, "whole tiles, B early");
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(lds);
    u32x4_t af1[NB], bf1[NBN];  // the fragments of the slab's second k-step
    const int sb = s.sb, sa = ring(sb + 1), nb = ring(sb + 2), na = ring(sb + 3), fr = ring(sb + 4);
    const Ahead from = stream_ahead(it, nk, a_next, b_next);
    kstep<true, 1, true, true, FIRST>(acc, s.af, s.bf, lds0 + sa * SLOT + a_rd, lds0 + sb * SLOT + b_rd, af1, bf1, lds, fr, 0, from.b);
    wait_vm<HL>();
    wait_lgkm<0>();
    __builtin_amdgcn_s_barrier();
    kstep<false, 0, false, true>(acc, af1, bf1, lds0 + na * SLOT + a_rd, lds0 + nb * SLOT + b_rd, s.af, s.bf, lds, sb, 0, from.a);
    s.sb = nb;
  }

  // the next tile's first fragments are in registers from here on, whatever the compiler does with those meanwhile
  static LCE_DEV void stream_settle(Stream& s) {
    wait_lgkm<0>();
#pragma unroll
    for (int i = 0; i < NB; ++i) asm volatile("" : "+v"(s.af[i]));
#pragma unroll
    for (int j = 0; j < NBN; ++j) asm volatile("" : "+v"(s.bf[j]));
  }

  // One tile.
  LCE_DEV void stream_tile(char* lds, int nk, f32x4_t (&acc)[NB][NBN], Stream& s, const char* a_next, const char* b_next) const {
    stream_slab<true>(lds, 0, nk, acc, s, a_next, b_next);
    for (int it = 1; it < nk; ++it) stream_slab<false>(lds, it, nk, acc, s, a_next, b_next);
    stream_settle(s);
    retire(acc);
  }

  // A tile's last slab when only its first k-step holds anything.  The next tile's first fragments are not read yet when it
  // returns (stream_fragments).
  LCE_DEV void stream_half_slab(char* lds, int nk, f32x4_t (&acc)[NB][NBN], Stream& s, const char* a_next, const char* b_next) const {
    const Ahead from = stream_ahead(nk - 1, nk, a_next, b_next);
    const int fr = ring(s.sb + 4);
    constexpr int EVERY = NB * NBN / HLB;
    wait_lgkm<0>();
    static_for(std::make_integer_sequence<int, NB * NBN>{}, [&](auto mc) {
      constexpr int m = decltype(mc)::value;
      __builtin_amdgcn_sched_barrier(0);
      Mma16<TIN>::run(acc[m / NBN][m % NBN], s.af[m / NBN], s.bf[m % NBN]);
      if constexpr (m % EVERY == 3 && m / EVERY < HLB) fetch_b(lds, fr, from.b, m / EVERY);
      __builtin_amdgcn_sched_barrier(0);
    });
    wait_vm<HLB>();
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int j = 0; j < HL; ++j) fetch_a(lds, s.sb, from.a, j);
    s.sb = ring(s.sb + 2);
  }
  LCE_DEV void stream_fragments(char* lds, Stream& s) const {
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(lds);
    static_for(std::make_integer_sequence<int, NF>{}, [&](auto fc) {
      read_frag<decltype(fc)::value, 0>(lds0 + ring(s.sb + 1) * SLOT + a_rd, lds0 + s.sb * SLOT + b_rd, s.af, s.bf);
    });
  }
  LCE_DEV void fetch_a(char* lds, int slot, const char* from, int j) const {
    __builtin_amdgcn_global_load_lds((gptr_t)(from + va[j]), (lptr_t)(lds + slot * SLOT + (j * Cfg::NW + wave) * 1024), 16, 0, 0);
  }
  LCE_DEV void fetch_b(char* lds, int slot, const char* from, int j) const {
    __builtin_amdgcn_global_load_lds((gptr_t)(from + vb[j]), (lptr_t)(lds + slot * SLOT + (j * Cfg::NW + wave) * 1024), 16, 0, 0);
  }

  // A tile's first slab, whose first k-step takes the finished tile out of the accumulators as it starts them anew: block (i, j) is
  // handed to `out` (out.block<i, j>(value)) ahead of the MFMA that overwrites it, block columns in the outer loop, and
  // out.send<j>() and out.store<j>() follow while column j + 1 goes through the matrix pipe: a column's NB LDS writes, then its
  // out.READS LDS reads, then its out.STORES stores.  The finished tile meets LDS in ring slot (s.sb + 4) % 5, so that the B half
  // that would be fetched into it comes with the A half, in the second k-step.  `last`: there is no next tile, and the accumulators
  // hold nothing afterwards (a way out of a walk that read them elsewhere would have the compiler move them about).
  template <typename Out>
  LCE_DEV void stream_slab_over(char* lds, int nk, f32x4_t (&acc)[NB][NBN], Stream& s, const char* a_next, const char* b_next, Out& out, bool last) const {
    static_assert(Cfg::TRANS != 2 && NBN == 8 && NB >= 7 && !AE && Cfg::TERMS == 1 && !Cfg::A_ONCE, "whole tiles, B early");
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(lds);
    u32x4_t af1[NB], bf1[NBN];
    const int sb = s.sb, sa = ring(sb + 1), nb = ring(sb + 2), na = ring(sb + 3), fr = ring(sb + 4);
    const Ahead from = stream_ahead(0, nk, a_next, b_next);
    const uint32_t ra = lds0 + sa * SLOT + a_rd, rb = lds0 + sb * SLOT + b_rd;
    wait_lgkm<0>();
    static_for(std::make_integer_sequence<int, NB * NBN>{}, [&](auto mc) {
      constexpr int m = decltype(mc)::value, j = m / NB, i = m % NB;
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" : "+a"(acc[i][j]));  // (read here and not ahead of the first MFMA)
      out.template block<i, j>(acc[i][j]);
      Mma16<TIN>::over(acc[i][j], s.af[i], s.bf[j]);
      if constexpr (j > 0 && i == 1) out.template send<j - 1>();  // (a wave's LDS operations are done in order)
      if constexpr (j > 0 && i == 5) {
        wait_lgkm<4>();  // (the writes of blocks 2 to 5 came behind those reads)
        out.template store<j - 1>();
      }
      if constexpr (i == NB - 1) {
        if constexpr (2 * j < NF) read_frag<2 * j, 1>(ra, rb, af1, bf1);
        if constexpr (2 * j + 1 < NF) read_frag<2 * j + 1, 1>(ra, rb, af1, bf1);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    out.template send<NBN - 1>();
    wait_lgkm<0>();
    out.template store<NBN - 1>();
    __builtin_amdgcn_sched_barrier(0);
    if (last) return;
    wait_vm<NBN * Out::STORES>();  // slab 1 has landed; the stores may be on their way
    __builtin_amdgcn_s_barrier();
    constexpr int LOADS = HLB + HL, EVERY = NB * NBN / LOADS;
    static_assert(2 * NF <= NB * NBN && LOADS * EVERY <= NB * NBN, "one fragment read after every second MFMA");
    static_for(std::make_integer_sequence<int, NB * NBN>{}, [&](auto mc) {
      constexpr int m = decltype(mc)::value, l = m / EVERY;
      __builtin_amdgcn_sched_barrier(0);
      Mma16<TIN>::run(acc[m / NBN][m % NBN], af1[m / NBN], bf1[m % NBN]);
      if constexpr ((m & 1) == 0 && m / 2 < NF) read_frag<m / 2, 0>(lds0 + na * SLOT + a_rd, lds0 + nb * SLOT + b_rd, s.af, s.bf);
      if constexpr (m % EVERY == EVERY - 1 && l < LOADS) {
        if constexpr (l < HLB) fetch_b(lds, fr, from.b, l);
        else fetch_a(lds, sb, from.a, l - HLB);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    s.sb = nb;
  }

  LCE_DEV void run(char* lds, int64_t K, f32x4_t (&acc)[NB][NBN]) const {
    prologue(lds, K);
    main(lds, K, acc);
  }
};

}  // namespace lce
