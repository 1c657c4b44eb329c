// The fused kernels on the four-wave 16x16x32 mainloop (gemm_core16.hpp): same arguments, same results layout
// and the same orientation as lce_kernels.hpp (MFMA rows = vocabulary, MFMA columns = tokens, so a lane owns
// whole tokens), with the accumulator layout of the 16 x 16 blocks: in block (i, j) of a wave tile lane l holds
// token 16 j + l % 16 and the vocabulary rows 16 i + 4 (l / 16) + r, r = 0..3.
#pragma once
#include "gemm_core16.hpp"
#include "lce_kernels.hpp"

namespace lce {

// K order of the backward's private intermediates (see KPerm in lce_kernels.hpp): inside each group of 128
// vocabulary rows (one wave tile) the entries are ordered so that what a lane holds of two neighbouring blocks is one
// 16-byte run and the four lane groups follow each other (64 contiguous bytes per token and store instruction):
// row v = 16 i + 4 g + r  ->  position 32 (i / 2) + 8 g + 4 (i % 2) + r.  Tokens keep their order.
template <typename TIN, int TR, int NBN, int AE, int TERMS, int AO, int NBM>
struct KPerm<GemmCfg16<TIN, TR, NBN, AE, TERMS, AO, NBM>> {
  static constexpr int GT = 128, GV = 128;
  static __host__ __device__ __forceinline__ int64_t token(int64_t t) { return t; }
  static __host__ __device__ __forceinline__ int64_t token_at(int64_t u) { return u; }
  static __host__ __device__ __forceinline__ int64_t vocab(int64_t v) {
    const int64_t l = v % GV, i = l / 16, w = l % 16;
    return v - l + (i / 2) * 32 + (w / 4) * 8 + (i % 2) * 4 + (w % 4);
  }
  static __host__ __device__ __forceinline__ int64_t vocab_at(int64_t u) {
    const int64_t l = u % GV, ip = l / 32, rem = l % 32, g = rem / 8, ih = (rem % 8) / 4, r = rem % 4;
    return u - l + (2 * ip + ih) * 16 + 4 * g + r;
  }
};

// ------------------------------------------------------------------------------------------------
// forward
// ------------------------------------------------------------------------------------------------
// folds one finished tile into the running per-token statistics (FULL: no padded vocabulary rows in the tile)
template <typename Cfg, bool FULL, typename F>
LCE_DEV void fwd16_fold(const FwdArgs<typename Cfg::TIN>& p, f32x4_t (&acc)[Cfg::NB][Cfg::NBN], float (&m)[Cfg::NBN],
                        float (&a)[Cfg::NBN], float (&b)[Cfg::NBN], const int (&lab)[Cfg::NBN], int vbase, int vend, int64_t tok0, int g4,
                        int l16, F&& column) {
  constexpr int NB = Cfg::NB, NBN = Cfg::NBN;
#pragma unroll
  for (int j = 0; j < NBN; ++j) {
    // One block column at a time (register pressure).  Its accumulators are in AGPRs up to here: the compiler otherwise reads
    // all 256 of a lane ahead of the first column and keeps other values in scratch memory meanwhile.
    GemmCore16<Cfg>::stay_column(acc, j);
    column(j);
    float x[NB * 4];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = acc[i][j][r];
        if (!FULL && vbase + 16 * i + 4 * g4 + r >= vend) v = -INFINITY;  // padded vocabulary rows
        x[i * 4 + r] = v;
      }
    // four independent chains each for the maximum and the two sums: one wave per SIMD has no neighbour to hide the
    // latency of a dependent chain of 32
    float t4[4] = {x[0], x[1], x[2], x[3]};
#pragma unroll
    for (int q = 4; q < NB * 4; ++q) t4[q & 3] = fmaxf(t4[q & 3], x[q]);
    const float tmax = fmaxf(fmaxf(t4[0], t4[1]), fmaxf(t4[2], t4[3]));
    const float mn = fmaxf(m[j], tmax);
    const float sc = fast_exp2((m[j] - mn) * p.c);
    const float mc = mn * p.c;
    m[j] = mn;
    float a4[4] = {a[j] * sc, 0.f, 0.f, 0.f}, b4[4] = {b[j] * sc, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NB * 4; ++q) {
      const float e = fast_exp2(__builtin_fmaf(x[q], p.c, -mc));
      a4[q & 3] += e;
      // padded rows: -inf in the log-sum-exp, 0 in the sum of x * exp
      b4[q & 3] = __builtin_fmaf(FULL ? x[q] : (x[q] == -INFINITY ? 0.f : x[q]), e, b4[q & 3]);
    }
    const float aj = (a4[0] + a4[1]) + (a4[2] + a4[3]), bj = (b4[0] + b4[1]) + (b4[2] + b4[3]);
    a[j] = aj;
    b[j] = bj;
    asm volatile("" : "+v"(m[j]), "+v"(a[j]), "+v"(b[j]));  // (this column is finished here, not after the branches below)
    // label logit: rare (a token's label falls in this wave tile with probability WM / V)
    const int rel = lab[j] - vbase;
    const bool mine = lab[j] >= 0 && lab[j] < vend && rel >= 0 && rel < Cfg::WM && (((rel >> 2) & 3) == g4);
    if (__builtin_amdgcn_ballot_w64(mine) != 0) {
      float pick = 0.f;
#pragma unroll
      for (int q = 0; q < NB * 4; ++q)
        if (mine && 16 * (q >> 2) + (q & 3) == (rel & ~12)) pick = x[q];
      // exactly one lane in the whole grid owns a token's label: plain store, no merge needed
      if (mine) p.xlabel[tok0 + j * 16 + l16] = pick;
    }
  }
}

// Which forwards run the stream of slabs: the square tile on plain operands.  (The kept logits are stores whose number the
// stream's waits would have to know; the narrow tile's early operand is the other one.)  It wants two slabs of K at least.
template <typename Cfg, bool KEEP>
struct Fwd16Stream {
  static constexpr bool value = !KEEP && Cfg::NBN == Cfg::NB && !Cfg::A_EARLY && Cfg::TERMS == 1;
};

// A last token tile with fewer tokens left is multiplied on the narrowest of 160, 192 and 224 columns that holds them, by a workgroup
// of the same launch: the matrix work of the columns beyond costs time even where it is padding, at some 1400 W of socket power as energy.
// Where the tiles are narrow already or the products six (forward in us, H=3584: 130 tokens 231 -> 214, 300: 380 -> 371, 333: 383 -> 374,
// 352: 384 -> 370; fp32 on planes 300: 3401 -> 3220, 600: 4377 -> 4225); on the square tile's stream it does not show (1100 tokens
// 1004 -> 1016, 5003: 4049 -> 4080).
template <typename Cfg>
struct Fwd16Tails {
  static constexpr bool value = (Cfg::A_EARLY || Cfg::TERMS == 6) && Cfg::NBN > 5;
  template <int NBN>
  using Narrow = GemmCfg16<typename Cfg::TIN, 0, NBN, Cfg::A_EARLY, Cfg::TERMS, Cfg::A_ONCE>;
};

// KEEP: the tiles also write their logits to p.xcache (FwdArgs), for a backward that then does not recompute them
template <typename Cfg, bool KEEP>
LCE_DEV void fwd16_body(const FwdArgs<typename Cfg::TIN>& p, int64_t n0, int s, char* lds) {
  constexpr int NB = Cfg::NB, NBN = Cfg::NBN;
  const int lane = threadIdx.x & 63, g4 = lane >> 4, l16 = lane & 15;
  GemmCore16<Cfg> g;
  g.set_lane();
  g.a_plane = p.w_plane;
  g.b_plane = p.h_plane;

  float m[NBN], a[NBN], b[NBN];
  int lab[NBN];
#pragma unroll
  for (int j = 0; j < NBN; ++j) {
    m[j] = kNegBig;
    a[j] = 0.f;
    b[j] = 0.f;
    const int64_t t = n0 + g.wave_n * Cfg::WN + j * 16 + l16;
    const int64_t y = t < p.T ? p.labels[t] - p.label_offset : -1;
    lab[j] = (y >= 0 && y < p.V) ? (int)y : -1;
  }

  f32x4_t acc[NB][NBN];
  const int64_t row0 = (int64_t)s * p.split_stride;
  const int64_t vend64 = row0 + p.split_span < p.V ? row0 + p.split_span : p.V;
  const int vend = (int)vend64;
  g.init(p.W, p.ldw, row0, vend64, p.h, p.ldh, n0, p.T);
  g.prologue(lds, p.H);
  if constexpr (Fwd16Stream<Cfg, KEEP>::value) {
    // The K loops of successive tiles are one stream of slabs (GemmCore16::stream_tile): nothing is drained between them and
    // the next tile's first slabs are in LDS while this one is folded in.  Only a last tile with fewer rows, whose loads
    // are clamped, starts anew.
    const int nk = (int)(p.H / Cfg::BK);  // (>= 2)
    typename GemmCore16<Cfg>::Stream st;
    g.stream_begin(lds, st);
    for (int64_t m0 = row0; m0 < vend64; m0 += p.tile_step) {
      const int64_t next = m0 + p.tile_step;
      const bool flows = next + Cfg::BM <= vend64;
      const char* a_next = flows ? g.a_base + p.tile_step * p.ldw * 2 : g.a_base;
      g.stream_tile(lds, nk, acc, st, a_next, g.b_base);
      g.a_base = a_next;
      const bool anew = next < vend64 && !flows;
      if (anew) {
        GemmCore16<Cfg>::template wait_vm<0>();
        __syncthreads();
        g.init(p.W, p.ldw, next, vend64, p.h, p.ldh, n0, p.T);
        g.prologue(lds, p.H);
      }
      const int vbase = (int)m0 + g.wave_m * Cfg::WM;  // vocabulary index of this wave's first row
      if (m0 + Cfg::BM <= vend64) fwd16_fold<Cfg, true>(p, acc, m, a, b, lab, vbase, vend, n0 + g.wave_n * Cfg::WN, g4, l16, [](int) {});
      else fwd16_fold<Cfg, false>(p, acc, m, a, b, lab, vbase, vend, n0 + g.wave_n * Cfg::WN, g4, l16, [](int) {});
      if (anew) g.stream_begin(lds, st);
    }
    GemmCore16<Cfg>::template wait_vm<0>();  // (the last tile's loads ahead, which nobody reads)
  } else {
    for (int64_t m0 = row0; m0 < vend64; m0 += p.tile_step) {
      g.main(lds, p.H, acc);
      const int vbase = (int)m0 + g.wave_m * Cfg::WM;  // vocabulary index of this wave's first row
      const bool full = m0 + Cfg::BM <= vend64;
      auto fold = [&](auto&& column) {
        if (full) fwd16_fold<Cfg, true>(p, acc, m, a, b, lab, vbase, vend, n0 + g.wave_n * Cfg::WN, g4, l16, column);
        else fwd16_fold<Cfg, false>(p, acc, m, a, b, lab, vbase, vend, n0 + g.wave_n * Cfg::WN, g4, l16, column);
      };
      // With kept logits a column is stored just before it is folded in, so that the stores leave during the fold, and the next
      // tile's first loads come behind both: the K loop waits on counts of outstanding vector-memory operations, and with the stores
      // older than every load it waits for, those counts mean what they say.  (With six products there are not the registers for it:
      // the stores first, then the loads, then the fold.)  Forward + backward against that order, us, nine runs a side in turn: H=896, 300
      // tokens with a frozen head 302.9 -> 296.4; H=3584, 333: 1228 -> 1216, 512: 1535 -> 1524, 1000: 2921 -> 2902 (2911 to 2925, 2897 to 2904), 1700:
      // 4817 -> 4800; 0.2 to 0.3 % and within the runs' spread for 400 of H=5120 and 1000 of H=4096.
      constexpr bool kWithFold = KEEP && Cfg::TERMS == 1;
      if constexpr (KEEP) {
        if (Cfg::TERMS == 1 || m0 < p.keep_rows) {
          // a lane holds four consecutive vocabulary rows of a token per block: one 16-byte store.
          // The count is a 6-bit field: four columns' stores, then two at a time, and behind the last column, whichever it is, so many
          // are waited for that with the prologue's loads behind them fewer than 64 operations are ever in flight (8 stores a
          // column, 12 where the compiler gives lanes without a token a store of their own; tests/test_ring_loads_on_cpu.py counts
          // them on the listing).  Non-temporal: 130 tokens, H=3584, step 812 -> 794 us, 192: 859 -> 842, level from 333 on.
          constexpr int kColumn = NB + NB / 2, kBehindLast = Cfg::TERMS == 6 ? 16 : 24, kBetween = 32;
          constexpr int kPrologue = Cfg::TERMS == 6 ? 2 * Cfg::HL + 3 * Cfg::HLB : 2 * (Cfg::HL + Cfg::HLB);
          static_assert(kBetween + 2 * kColumn < 64 && 4 * kColumn < 64 && kBehindLast + kPrologue < 64, "vmcnt range");
          const int64_t t0 = n0 + g.wave_n * Cfg::WN + l16;
          // the eight panels of this wave's rows; tokens beyond T and rows beyond the split (whole fours) are dropped
          const buf_t kept = make_buf(kept_logit(p.xcache, p.T, 0, vbase), (int64_t)NB * p.T * 64);
          const int row_at = g4 * 16, panel = (int)p.T * 64;
          auto store = [&](int j) {
            const int at = t0 + j * 16 < p.T ? (int)(t0 + j * 16) * 64 + row_at : kBufNowhere;
#pragma unroll
            for (int i = 0; i < NB; ++i) {
              const int o = at == kBufNowhere || (!full && vbase + 16 * i + 4 * g4 >= vend) ? kBufNowhere : at + i * panel;
              __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc[i][j]), kept, o, 0, kBufNonTemporal);
            }
            if (kWithFold) __builtin_amdgcn_sched_barrier(0);  // (ahead of the column's fold, all of them)
            if (j % 2 == 1 && j >= 3 && j < NBN - 1) {
              __builtin_amdgcn_sched_barrier(0);
              GemmCore16<Cfg>::template wait_vm<kBetween>();
            }
          };
          if constexpr (kWithFold) {
            fold(store);
          } else {
#pragma unroll
            for (int j = 0; j < NBN; ++j) {
              GemmCore16<Cfg>::stay_column(acc, j);
              store(j);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
          GemmCore16<Cfg>::template wait_vm<kBehindLast>();
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __syncthreads();  // every wave is past its last LDS read and has drained its own loads
      if (m0 + p.tile_step < vend64) {
        g.init(p.W, p.ldw, m0 + p.tile_step, vend64, p.h, p.ldh, n0, p.T);
        g.prologue(lds, p.H);
      }
      // the next tile's first slabs fly while this tile's statistics are folded in
      if constexpr (!kWithFold) fold([](int) {});
    }
  }
  __syncthreads();

  // merge the four lane groups (same token, different vocabulary rows), then the two waves along the vocabulary
  f32x4_t* red = reinterpret_cast<f32x4_t*>(lds);  // [WAVES_M][BN]
#pragma unroll
  for (int j = 0; j < NBN; ++j) {
#pragma unroll
    for (int off = 16; off <= 32; off <<= 1) {
      const float m2 = __shfl_xor(m[j], off), a2 = __shfl_xor(a[j], off), b2 = __shfl_xor(b[j], off);
      merge_stats(m[j], a[j], b[j], m2, a2, b2, p.c);
    }
    if (g4 == 0) {
      const f32x4_t v = {m[j], a[j], b[j], 0.f};
      red[g.wave_m * Cfg::BN + g.wave_n * Cfg::WN + j * 16 + l16] = v;
    }
  }
  __syncthreads();
  for (int t = threadIdx.x; t < Cfg::BN; t += Cfg::NTHREADS) {
    const f32x4_t v0 = red[t];
    float vm = v0[0], va = v0[1], vb = v0[2];
#pragma unroll
    for (int w = 1; w < Cfg::WAVES_M; ++w) {
      const f32x4_t u = red[w * Cfg::BN + t];
      merge_stats(vm, va, vb, u[0], u[1], u[2], p.c);
    }
    const int64_t tok = n0 + t;
    const f32x4_t v = {vm, va, vb, 0.f};
    if (tok < p.T) p.parts[(int64_t)s * p.T + tok] = v;
  }
}

// ------------------------------------------------------------------------------------------------
// backward: d_logits tiles
// ------------------------------------------------------------------------------------------------
// per-position constants of the d_logits tiles (see DsArgs::tokc)
inline __global__ void ds_token_consts_kernel(const int* rows, const int* n_rows, int64_t T, int64_t tpad, const float* g_lp, int64_t g_lp_stride,
                                       float g_lp_scale, const float* g_ent, const float* maximum, const float* accumulate,
                                       const float* entropy_b, const int64_t* labels, int64_t vocab_offset, int64_t V, float rcp_tau,
                                       f32x4_t* tokc, int* tokl) {
  const int64_t pos = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (pos >= tpad) return;
  const int64_t Tc = n_rows ? (int64_t)*n_rows : T;
  token_consts_at(tokc, tokl, pos, pos < Tc ? (rows ? (int64_t)rows[pos] : pos) : -1, g_lp, g_lp_stride, g_lp_scale, g_ent, maximum, accumulate,
                  entropy_b, labels, vocab_offset, V, rcp_tau);
}

// One finished tile: d_logits of the wave's 128 tokens x 128 vocabulary entries, written to dS straight from the
// registers: a lane holds 8 consecutive positions of the wave tile's vocabulary order per pair of blocks, the four lane
// groups 64 contiguous bytes of a token's row.  (Staging the tile through LDS for whole 256-byte runs per instruction
// was measured 9% slower on the pass: 3.64 against 3.31 ms per 38144-row chunk of config 2.)
// LABEL: some token of the wave tile has its label among the tile's rows: the one lane that holds that entry patches
// it after the common arithmetic (zero when the label's entry is kept out of the tiles, + G when everything is inside).
// EDGE: the tile reaches beyond the chunk's last row; those entries are zeros.
template <typename Cfg, bool LABEL, bool EDGE>
LCE_DEV void ds16_epilogue(const DsArgs<typename Cfg::TIN>& p, f32x4_t (&acc)[Cfg::NB][Cfg::NBN], const f32x4_t (&tc)[Cfg::NBN],
                           const int (&lab)[Cfg::NBN], int64_t tok0, int vloc0, int g4, int l16) {
  typedef typename Cfg::TIN TIN;
  constexpr int NB = Cfg::NB, NBN = Cfg::NBN;
#pragma unroll
  for (int j = 0; j < NBN; ++j) {
    GemmCore16<Cfg>::stay_column(acc, j);  // (one block column at a time, as in fwd16_fold)
    const float lse2 = tc[j][0], C0 = tc[j][1], C1 = tc[j][2], G = tc[j][3];
    // the label's entry: block pair rel / 32, lane group (rel / 4) % 4, value 4 ((rel / 16) % 2) + rel % 4 of the run
    const int rel = (LABEL && p.label_outside != 1) ? lab[j] - (int)p.lab0 - vloc0 : -1;  // (1: the tiles hold the softmax terms only)
    const int own_ip = (rel >= 0 && rel < Cfg::WM && ((rel >> 2) & 3) == g4) ? rel >> 5 : -1;
    const int own_q = ((rel >> 4) & 1) * 4 + (rel & 3);
    const int64_t tok = tok0 + j * 16 + l16;
#pragma unroll
    for (int ip = 0; ip < NB / 2; ++ip) {
      float d[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int i = 2 * ip + (q >> 2), r = q & 3;
        d[q] = dlogit<false>(acc[i][j][r], p.c, lse2, C0, C1, G, false, false, false);
        if (EDGE && vloc0 + 16 * i + 4 * g4 + r >= p.vrows) d[q] = 0.f;
      }
      if (LABEL) {
        const bool mine = own_ip == ip;
        if (__builtin_amdgcn_ballot_w64(mine) != 0) {
#pragma unroll
          for (int q = 0; q < 8; ++q)
            if (mine && q == own_q) d[q] = p.label_outside == 2 ? 0.f : d[q] + G;
        }
      }
      // rows of positions without a token are zeros (their constants make them so); they pad the d_weight GEMM's K
      TIN* dst = ds_at(p.dS, p.ldS, p.pcol, tok, vloc0 + ip * 32 + g4 * 8);
      if constexpr (Cfg::TERMS == 6) store_planes<TIN, 8>(dst, p.dS_plane, d);
      else store_run<TIN, 8>(dst, d);
    }
  }
}

// One workgroup per tile.  (Workgroups that walk strips of 2, 4 or 8 consecutive vocabulary tiles, with the first loads
// of the next tile in flight while the finished one is written out, took the same time on the pass alone and more inside
// the backward's combined launch, whose tail then is a strip long.)
template <typename Cfg>
LCE_DEV void ds16_tile(const DsArgs<typename Cfg::TIN>& p, int bid, char* lds) {
  constexpr int NB = Cfg::NB, NBN = Cfg::NBN;
  const int64_t Tc = p.n_rows ? (int64_t)*p.n_rows : p.T;  // tokens that take part
  int tt, vt;
  const TileMap map = p.n_rows ? p.map.with_rows((int)((Tc + Cfg::BN - 1) / Cfg::BN)) : p.map;
  if (!map.decode(bid, tt, vt)) return;
  const int64_t n0 = (int64_t)tt * Cfg::BN;
  const int lane = threadIdx.x & 63, g4 = lane >> 4, l16 = lane & 15;
  GemmCore16<Cfg> g;
  g.set_lane();
  const int64_t tok0 = n0 + g.wave_n * Cfg::WN;  // first position of this wave's group
  g.a_plane = p.w_plane;
  g.b_plane = p.h_plane;
  g.init(p.W, p.ldw, (int64_t)vt * Cfg::BM, p.vrows, p.h, p.ldh, n0, Tc, p.rows);
  f32x4_t acc[NB][NBN];
  g.run(lds, p.H, acc);
  if (tok0 >= p.tpad) return;  // (positions are padded to whole groups: all of this wave's exist, or none)
  // the constants of the lane's positions, all asked for at once: across the K loop there are no registers for them
  f32x4_t tc[NBN];
  int lab[NBN];
#pragma unroll
  for (int j = 0; j < NBN; ++j) {
    tc[j] = p.tokc[tok0 + j * 16 + l16];
    lab[j] = p.tokl[tok0 + j * 16 + l16];
  }
  const int vloc0 = vt * Cfg::BM + g.wave_m * Cfg::WM;  // chunk-local vocabulary index of this wave's first row
  // fast path: no padded vocabulary rows and no label in the wave tile
  bool has_label = false;
  if (p.label_outside != 1) {
#pragma unroll
    for (int j = 0; j < NBN; ++j) {
      const int rel = lab[j] - (int)p.lab0 - vloc0;
      has_label |= (rel >= 0 && rel < Cfg::WM);
    }
  }
  const bool labels_here = __builtin_amdgcn_ballot_w64(has_label) != 0;
  // Labels kept out of the tiles altogether (label_outside == 2, the default): the tile is written by the common
  // path, and the lane that stored a label's entry then overwrites it with a zero (same lane, same address, later
  // store).  Measured on a 38144-column chunk of config 2, where one wave tile in nine holds a label: 3.71 -> 3.58 ms
  // against patching inside the common arithmetic.  With the one-hot part inside the tile (0) the patch adds G there.
  const bool in_tile = labels_here && p.label_outside == 0;
  const bool edge = vloc0 + Cfg::WM > p.vrows;
  if (edge && in_tile) ds16_epilogue<Cfg, true, true>(p, acc, tc, lab, tok0, vloc0, g4, l16);
  else if (edge) ds16_epilogue<Cfg, false, true>(p, acc, tc, lab, tok0, vloc0, g4, l16);
  else if (in_tile) ds16_epilogue<Cfg, true, false>(p, acc, tc, lab, tok0, vloc0, g4, l16);
  else ds16_epilogue<Cfg, false, false>(p, acc, tc, lab, tok0, vloc0, g4, l16);
  if (labels_here && p.label_outside == 2) {
#pragma unroll
    for (int j = 0; j < NBN; ++j) {
      const int rel = lab[j] - (int)p.lab0 - vloc0;  // = 16 i + 4 g + r inside the wave tile
      const int64_t tok = tok0 + j * 16 + l16;
      if (rel >= 0 && rel < Cfg::WM && ((rel >> 2) & 3) == g4)
        *ds_at(p.dS, p.ldS, p.pcol, tok, vloc0 + (rel >> 5) * 32 + g4 * 8 + ((rel >> 4) & 1) * 4 + (rel & 3)) = (typename Cfg::TIN)0.f;
    }
  }
}

// ------------------------------------------------------------------------------------------------
// plain GEMMs.  The MFMA rows are taken from the operand that indexes the CONTIGUOUS dimension of C, so that
// the four accumulator registers of a block are four neighbours in a row of C (one 16-byte or 8-byte access):
// for C[m][n] = sum_k A[m][k] B[n][k] lane l holds m = 16 j + l % 16 and n = 16 i + 4 (l / 16) + r.
// ------------------------------------------------------------------------------------------------
// A wave tile that reaches beyond C's last row or column, in fp32, C (+)= acc (ACC: old values are read), in the accumulators'
// own lane order: 16 rows x 64 bytes per instruction.  (Whole tiles: gemm16_f32_lines.)
template <typename Cfg, bool ACC>
LCE_DEV void gemm16_edge(const GemmArgs<typename Cfg::TIN>& p, f32x4_t (&acc)[Cfg::NB][Cfg::NBN], int64_t mw, int64_t nw) {
  // mw, nw: this lane's row of block column 0 and its first column of block row 0
  // the old values of the next AHEAD block columns are on their way while a column is added and stored (the operand fragments'
  // registers are free by now)
  constexpr int AHEAD = 3;
  f32x4_t prev[AHEAD + 1][Cfg::NB];
  auto fetch = [&](int j) {
    const int64_t m = mw + j * 16;
#pragma unroll
    for (int i = 0; i < Cfg::NB; ++i) {
      const int64_t n = nw + i * 16;
      prev[j % (AHEAD + 1)][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (m < p.M && n < p.N) prev[j % (AHEAD + 1)][i] = *reinterpret_cast<const f32x4_t*>(p.Cf + m * p.ldcf + n);
    }
  };
  if (ACC) {
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) fetch(j);
  }
#pragma unroll
  for (int j = 0; j < Cfg::NBN; ++j) {
    const int64_t m = mw + j * 16;
    GemmCore16<Cfg>::stay_column(acc, j);  // (one block column at a time, as in fwd16_fold)
    if (ACC && j + AHEAD < Cfg::NBN) fetch(j + AHEAD);
    if (m >= p.M) continue;
#pragma unroll
    for (int i = 0; i < Cfg::NB; ++i) {
      const int64_t n = nw + i * 16;
      if (n >= p.N) continue;  // (N is a multiple of 4)
      f32x4_t v = acc[i][j];
      if (ACC) v += prev[j % (AHEAD + 1)][i];
      *reinterpret_cast<f32x4_t*>(p.Cf + m * p.ldcf + n) = v;
    }
  }
}

// A full wave tile in fp32, C (+)= acc (ACC: old values are read), as whole lines: one block column (16 rows x 128 or 112 columns) at a
// time goes through 8 KB of LDS that belong to this wave, 16-byte chunk c of row r at c ^ r, and meets memory two rows x 512
// bytes per instruction.  In the accumulators' own lane order, 16 rows x 64 bytes, reading and writing a tile took 38300
// cycles, a sixteenth of the d_hidden GEMM's K loop, with one block column of old values on its way or with three; this way it
// takes 20600.  Two buffers in turn; the old values of the next AHEAD columns are on their way while a column is added and stored.
template <typename Cfg, bool ACC>
LCE_DEV void gemm16_f32_lines(const GemmArgs<typename Cfg::TIN>& p, f32x4_t (&acc)[Cfg::NB][Cfg::NBN], int64_t mw, int64_t nw, uint32_t stage) {
  // mw, nw: the wave tile's first row and column of C
  constexpr int NB = Cfg::NB, NBN = Cfg::NBN, AHEAD = 2, PAIRS = 8;
  const int lane = threadIdx.x & 63, g4 = lane >> 4, l16 = lane & 15, hi = lane >> 5, cl = lane & 31;
  const uint32_t wr = stage + (uint32_t)(l16 * 512 + (g4 ^ l16) * 16);   // chunk 4 i + g4: ^ i * 64
  const uint32_t rd = stage + (uint32_t)(hi * 512 + (cl ^ hi) * 16);     // row 2 k + hi: ^ k * 32, + k * 1024
  char* base = reinterpret_cast<char*>(p.Cf + mw * p.ldcf + nw);
  const uint32_t off = (uint32_t)(hi * p.ldcf * 4 + cl * 16);
  const int64_t row_bytes = p.ldcf * 4;
  const bool has = NB == 8 || cl < 4 * NB;  // (the lane has a chunk of its row)
  f32x4_t prev[AHEAD + 1][PAIRS];
  auto fetch = [&](int j) {
    if (has) {
#pragma unroll
      for (int k = 0; k < PAIRS; ++k) prev[j % (AHEAD + 1)][k] = *reinterpret_cast<const f32x4_t*>(base + (16 * j + 2 * k) * row_bytes + off);
    }
  };
  auto write = [&](int j) {
    GemmCore16<Cfg>::stay_column(acc, j);
#pragma unroll
    for (int i = 0; i < NB; ++i)
      asm volatile("ds_write_b128 %0, %1" ::"v"((wr ^ (uint32_t)(i * 64)) + (j & 1) * 8192), "a"(acc[i][j]));
  };
  if (ACC) {
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) fetch(j);
  }
  write(0);
  static_for(std::make_integer_sequence<int, NBN>{}, [&](auto jc) {
    constexpr int j = decltype(jc)::value;
    if (ACC && j + AHEAD < NBN) fetch(j + AHEAD);
    if (j + 1 < NBN) write(j + 1);
    GemmCore16<Cfg>::template wait_lgkm<(j + 1 < NBN ? NB : 0)>();  // block column j is in LDS (j + 1's writes may be on their way)
    u32x4_t v[PAIRS];
    static_for(std::make_integer_sequence<int, PAIRS>{}, [&](auto kc) {
      constexpr int k = decltype(kc)::value;
      v[k] = lds_read16<k * 1024>((rd ^ (uint32_t)(k * 32)) + (j & 1) * 8192);
    });
    GemmCore16<Cfg>::template wait_lgkm<0>();
#pragma unroll
    for (int k = 0; k < PAIRS; ++k) asm volatile("" : "+v"(v[k]));  // (the reads are assembly, the compiler does not know when they return)
    if (has) {
#pragma unroll
      for (int k = 0; k < PAIRS; ++k) {
        f32x4_t x = __builtin_bit_cast(f32x4_t, v[k]);
        if (ACC) x += prev[j % (AHEAD + 1)][k];
        *reinterpret_cast<f32x4_t*>(base + (16 * j + 2 * k) * row_bytes + off) = x;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  });
}

// C in fp32 (out_mode 0 or 1: the callers have no other).
// CoreCfg: Cfg itself, or its mixed twin GemmCfg16<TIN, 2, ..>: then B is K-major as it lies in memory, B[k][n] with row
// stride ldb, its rows in the order KPerm<Cfg>::vocab_at of A's columns (the d_hidden GEMM reading W in place: no W^T);
// rows of B at or beyond p.b_rows_valid do not exist (A is zero in those columns).
template <typename Cfg, typename CoreCfg = Cfg>
LCE_DEV void gemm16_tile(const GemmArgs<typename Cfg::TIN>& pin, int bid, char* lds) {
  GemmArgs<typename Cfg::TIN> p = pin;
  if (p.m_dev) {
    const int64_t m = *p.m_dev;
    p.M = m < p.M ? m : p.M;
  }
  if (p.k_dev) {
    const int64_t k = ((int64_t)*p.k_dev + p.k_gran - 1) / p.k_gran * p.k_gran;
    p.K = k < p.K ? k : p.K;
  }
  int64_t k0 = 0, k1 = p.K;
  int tm, tn;
  const TileMap map = p.m_dev ? p.map.with_rows((int)((p.M + Cfg::BN - 1) / Cfg::BN)) : p.map;
  if (!map.decode(bid, tm, tn)) return;
  if (p.ksplit > 1) {  // the map's columns are N tiles x slices
    const int s = tn / p.n_tiles;
    tn -= s * p.n_tiles;
    k0 = s * p.kslice;
    k1 = k0 + p.kslice < p.K ? k0 + p.kslice : p.K;
    p.Cf += s * p.cf_split_stride;
  }
  const int64_t m0 = (int64_t)tm * Cfg::BN, n0 = (int64_t)tn * Cfg::BM;  // (MFMA rows = n, MFMA columns = m)
  GemmCore16<CoreCfg> g;
  f32x4_t acc[Cfg::NB][Cfg::NBN];
  if (k0 < k1 && (CoreCfg::TRANS != 2 || k0 < p.b_rows_valid)) {
    // MFMA rows = n, MFMA columns = m
    g.a_plane = p.b_plane;
    g.b_plane = p.a_plane;
    if constexpr (CoreCfg::TRANS == 2)
      g.init_mixed(p.B + k0 * p.ldb, p.ldb, n0, p.N - n0, p.b_rows_valid - k0, [](int r) { return KPerm<Cfg>::vocab_at(r); },
                   p.a_pcol ? p.A + (k0 >> 6) * p.a_pcol : p.A + k0, p.lda, m0, p.M, p.a_pcol ? p.a_pcol * 2 : (int64_t)Cfg::BKB);
    else
      g.init(p.B + k0, p.ldb, n0, p.N, p.A + k0, p.lda, m0, p.M);
    g.run(lds, k1 - k0, acc);
  } else {  // empty K range: contributes zero (and still initialises what it owns)
    if (p.out_mode == 1) return;
    g.set_lane();
#pragma unroll
    for (int i = 0; i < Cfg::NB; ++i)
#pragma unroll
      for (int j = 0; j < Cfg::NBN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  if (m0 + Cfg::BN > p.M || n0 + Cfg::BM > p.N) {
    const int64_t mw = m0 + g.wave_n * Cfg::WN + (g.lane & 15), nw = n0 + g.wave_m * Cfg::WM + 4 * (g.lane >> 4);
    if (p.out_mode == 1) gemm16_edge<Cfg, true>(p, acc, mw, nw);
    else gemm16_edge<Cfg, false>(p, acc, mw, nw);
    return;
  }
  __syncthreads();  // (the ring is the store tiles' now)
  const uint32_t stage = (uint32_t)reinterpret_cast<uintptr_t>(lds) + g.wave * 16384;
  const int64_t mt = m0 + g.wave_n * Cfg::WN, nt = n0 + g.wave_m * Cfg::WM;
  if (p.out_mode == 1) gemm16_f32_lines<Cfg, true>(p, acc, mt, nt, stage);
  else gemm16_f32_lines<Cfg, false>(p, acc, mt, nt, stage);
}

// LDS write of 8 bytes as inline assembly, for the same reason as the reads: through the compiler it would wait for the
// global->LDS loads in flight
template <int OFF = 0>
LCE_DEV void lds_write8(uint32_t lds_addr, const u32x2_t& v) { asm volatile("ds_write_b64 %0, %1 offset:%2" ::"v"(lds_addr), "v"(v), "i"(OFF)); }

// A finished wave tile in 16 bits, C[m][n] with rows in the operand's column order (PermCfg's vocab_at), leaves the wave as
// whole lines: 16 rows x 128 columns (one block column) at a time go through 4 KB of LDS that belong to this wave, 16-byte
// chunk c of row r at c ^ r, and are stored four rows x 256 bytes per instruction.  (A CU stores such runs three to four
// times as fast as the accumulators' own lane order, 16 rows x 64 bytes.)  Two buffers in turn: block column j is
// written while j - 1 is read back, so that neither waits for the other.
// Non-temporal: unmarked, the lines of d_weight push the dS and the hidden that other workgroups are about to read out of the
// caches (forward + backward, H=3584, V=152064: 333 tokens 1289 -> 1240 us, 512: 1624 -> 1588, 700: 2111 -> 2089, level from 1600 on).
template <typename Cfg, typename PermCfg, bool FULL>
LCE_DEV void gemm16_store_lines(const GemmArgs<typename Cfg::TIN>& p, f32x4_t (&acc)[Cfg::NB][Cfg::NBN], int64_t m0, int64_t n0,
                                int wave_m, int wave_n, uint32_t stage) {
  typedef typename Cfg::TIN TIN;
  typedef typename VecOf<TIN, 4>::type vec_t;
  constexpr int NB = Cfg::NB, NBN = Cfg::NBN;
  const int lane = lane_anew(), g4 = lane >> 4, l16 = lane & 15;
  const uint32_t wr = stage + (uint32_t)(l16 * 256 + (((g4 >> 1) ^ l16) * 16) + (g4 & 1) * 8);  // chunk 2 i + g4 / 2: ^ i * 32
  const uint32_t rd = stage + (uint32_t)(g4 * 256 + ((l16 ^ g4) * 16));                          // row 4 k + g4: ^ k * 64, + k * 1024
  // the store of row 4 k + g4 of block column j, chunk l16: a uniform row pointer and one offset per lane
  const int64_t n = n0 + wave_m * Cfg::WM;
  const uint32_t off = (uint32_t)(g4 * p.ldct + l16 * 8) * (uint32_t)sizeof(TIN);
  const bool n_ok = (NB == 8 || l16 < 2 * NB) && (FULL || n + l16 * 8 < p.N);  // (the lane has a chunk of its row)
  const int64_t mw = m0 + wave_n * Cfg::WN;
  char* base = reinterpret_cast<char*>(p.Ct + mw * p.ldct + n);
  auto write = [&](auto jc) {
    constexpr int j = decltype(jc)::value;
    GemmCore16<Cfg>::stay_column(acc, j);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      vec_t o;
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = round_to<TIN>(acc[i][j][r]);
      lds_write8((wr ^ (uint32_t)(i * 32)) + (j & 1) * 4096, __builtin_bit_cast(u32x2_t, o));
    }
  };
  auto store = [&](auto jc) {
    constexpr int j = decltype(jc)::value;
    u32x4_t v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = lds_read16<0>((rd ^ (uint32_t)(k * 64)) + (j & 1) * 4096 + k * 1024);
    GemmCore16<Cfg>::template wait_lgkm<0>();
    // (opaque until the wait: the reads are assembly, the compiler does not know when they return)
#pragma unroll
    for (int k = 0; k < 4; ++k) asm volatile("" : "+v"(v[k]));
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      constexpr int u0 = 16 * j;
      const int64_t row = KPerm<PermCfg>::vocab_at(u0 + 4 * k);  // (+ g4: four consecutive rows of C)
      if (n_ok && (FULL || mw + row + g4 < p.M)) __builtin_nontemporal_store(v[k], reinterpret_cast<u32x4_t*>(base + row * p.ldct * (int64_t)sizeof(TIN) + off));
    }
  };
  static_for(std::make_integer_sequence<int, NBN + 1>{}, [&](auto jc) {
    constexpr int j = decltype(jc)::value;
    if constexpr (j < NBN) write(jc);
    if constexpr (j > 0) {
      GemmCore16<Cfg>::template wait_lgkm<(j < NBN ? NB : 0)>();  // block column j - 1 is in LDS (j's writes may be on their way)
      store(std::integral_constant<int, j - 1>{});
    }
  });
}

// The same for a workgroup that walks tiles, block by block as the next tile's first k-step comes to them
// (GemmCore16::stream_slab_over).  Rows and columns beyond C are stores to nowhere, so that their number is always the same.
template <typename Cfg, typename PermCfg>
struct LineStores16 {
  typedef typename Cfg::TIN TIN;
  static constexpr int STORES = 4;  // of a block column
  buf_t out;
  uint32_t wr, rd;
  int at, row_bytes;
  u32x4_t v[STORES];
  LCE_DEV LineStores16(const GemmArgs<TIN>& p, int64_t m0, int64_t n0, int wave_m, int wave_n, uint32_t stage) {
    const int lane = lane_anew(), g4 = lane >> 4, l16 = lane & 15;
    wr = stage + (uint32_t)(l16 * 256 + (((g4 >> 1) ^ l16) * 16) + (g4 & 1) * 8);
    rd = stage + (uint32_t)(g4 * 256 + ((l16 ^ g4) * 16));
    const int64_t n = n0 + wave_m * Cfg::WM, mw = m0 + wave_n * Cfg::WN, left = p.M - mw;
    row_bytes = (int)(p.ldct * (int64_t)sizeof(TIN));
    out = make_buf(p.Ct + mw * p.ldct + n, (left < Cfg::WN ? left > 0 ? left : 0 : Cfg::WN) * row_bytes);
    at = (Cfg::NB == 8 || l16 < 2 * Cfg::NB) && n + l16 * 8 < p.N ? g4 * row_bytes + l16 * 16 : kBufNowhere;
  }
  template <int I, int J>
  LCE_DEV void block(const f32x4_t& acc) const {
    typename VecOf<TIN, 4>::type o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = round_to<TIN>(acc[r]);
    lds_write8<(J & 1) * 4096>(wr ^ (uint32_t)(I * 32), __builtin_bit_cast(u32x2_t, o));
  }
  template <int J>
  LCE_DEV void send() {
    static_for(std::make_integer_sequence<int, STORES>{}, [&](auto kc) {
      constexpr int k = decltype(kc)::value;
      v[k] = lds_read16<(J & 1) * 4096 + k * 1024>(rd ^ (uint32_t)(k * 64));
    });
  }
  template <int J>
  LCE_DEV void store() {
#pragma unroll
    for (int k = 0; k < STORES; ++k) asm volatile("" : "+v"(v[k]));
#pragma unroll
    for (int k = 0; k < STORES; ++k) {
      const int row = (int)KPerm<PermCfg>::vocab_at(16 * J + 4 * k);
      __builtin_amdgcn_raw_buffer_store_b128(v[k], out, at + row * row_bytes, 0, kBufNonTemporal);
    }
  }
};

// C[m][n] = sum_k A[k][m] * B[k][n], both operands K-major and allocated in whole tiles, K (or *k_dev
// rounded up to k_gran) a multiple of 64.  out_mode 0: Cf = acc; out_mode 2: Ct[PermCfg's vocab_at(m)][n] = (TIN)acc
// (the rows of C are A's columns, which the d_logits epilogue leaves in KPerm::vocab order).
template <typename Cfg, typename PermCfg>
LCE_DEV void gemm16_tn_tile(const GemmArgs<typename Cfg::TIN>& pin, int bid, char* lds) {
  typedef typename Cfg::TIN TIN;
  GemmArgs<TIN> p = pin;
  if (p.k_dev) {
    const int64_t k = ((int64_t)*p.k_dev + p.k_gran - 1) / p.k_gran * p.k_gran;
    p.K = k < p.K ? k : p.K;
  }
  int tm, tn;
  if (!p.map.decode(bid, tm, tn)) return;
  const int64_t m0 = (int64_t)tm * Cfg::BN, n0 = (int64_t)tn * Cfg::BM;  // (MFMA rows = n, MFMA columns = m)
  GemmCore16<Cfg> g;
  f32x4_t acc[Cfg::NB][Cfg::NBN];
  if (p.K > 0) {
    g.a_plane = p.b_plane;
    g.b_plane = p.a_plane;
    g.init_tn(p.B, p.ldb, n0, p.A, p.lda, m0, p.a_pcol);
    g.run(lds, p.K, acc);
  } else {
    g.set_lane();
#pragma unroll
    for (int i = 0; i < Cfg::NB; ++i)
#pragma unroll
      for (int j = 0; j < Cfg::NBN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  if (p.out_mode == 2) {
    __syncthreads();  // (the ring is the store tiles' now)
    const uint32_t stage = (uint32_t)reinterpret_cast<uintptr_t>(lds) + g.wave * 8192;
    if (m0 + Cfg::BN <= p.M && n0 + Cfg::BM <= p.N) gemm16_store_lines<Cfg, PermCfg, true>(p, acc, m0, n0, g.wave_m, g.wave_n, stage);
    else gemm16_store_lines<Cfg, PermCfg, false>(p, acc, m0, n0, g.wave_m, g.wave_n, stage);
    return;
  }
  const int64_t nw = n0 + g.wave_m * Cfg::WM + 4 * (g.lane >> 4);
#pragma unroll
  for (int j = 0; j < Cfg::NBN; ++j) {
    const int u = g.wave_n * Cfg::WN + j * 16 + (g.lane & 15);  // row inside the tile, in the operand's column order
    const int64_t m = m0 + (p.perm_rows ? (int64_t)KPerm<PermCfg>::vocab_at(u) : (int64_t)u);
    GemmCore16<Cfg>::stay_column(acc, j);
    if (m >= p.M) continue;
#pragma unroll
    for (int i = 0; i < Cfg::NB; ++i) {
      const int64_t n = nw + i * 16;
      if (n >= p.N) continue;  // (N is a multiple of 4)
      *reinterpret_cast<f32x4_t*>(p.Cf + m * p.ldcf + n) = acc[i][j];
    }
  }
}

// d_weight with tokens between the streaming kernels' range and the sizes where a tile's K loop hides everything else:
// C[vocab_at(m)][n] = (TIN) sum_k A[k][m] B[k][n] as in gemm16_tn_tile (out_mode 2), by workgroups that stay (one per CU)
// and walk the tiles, the K loops of successive tiles being one stream of slabs.  With 333 tokens a
// tile is six slabs of 1.2 to 1.5 us, and a workgroup per tile paid another 9 us for its start, its first loads, the drain of
// its last and its stores.  A finished tile leaves the accumulators during the next one's first k-step (stream_slab_over: 384
// conversions beside 64 MFMAs, some 2800 cycles for 4400 + 1024 one behind the other), and a last slab of up to 32 tokens is one k-step: kernel at 333
// tokens of H=3584 432 -> 416 us, 512: 496 -> 487, 1000: 908 -> 902.  Forward + backward with neither / the first / both: 270 tokens 1181 / 1173 / 1163,
// 333: 1234 / 1226 / 1216, 600: 2037 / 2027 / 2018; where the last slab is a whole one 384: 1279 / 1271 / 1272, 500: 1541 / 1534 / 1535, 1000: 2922 /
// 2914 / 2917 (runs of a side differ by up to 0.5 %).  Without its stores it takes 347, 443 and 811: the 1.09 GB of results cost 45 to 90 us
// wherever in the tile they are issued (workgroups set off by a quarter of a tile against each other: level).
template <typename Cfg>
__global__ __launch_bounds__(Cfg::NTHREADS) void lce_dw16_kernel(GemmArgs<typename Cfg::TIN> p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  typedef GemmCfg16<typename Cfg::TIN, 1, 8, 0, 1, 0, Cfg::NB> TnCfg;
  typedef GemmCore16<TnCfg> Core;
  constexpr int TM = TnCfg::BN, TN = TnCfg::BM;  // a tile's rows and columns of C (MFMA rows = n, MFMA columns = m)
  if (p.k_dev) {
    // whole k-steps of 32 (at least two slabs, which the stream wants: token_prep_kernel, and beyond its range gather_rows_kernel,
    // zeroes that many rows of hidden, the d_logits pass those of dS)
    const int64_t k = *p.k_dev == 0 ? 0 : (*p.k_dev <= 64 ? 128 : ((int64_t)*p.k_dev + 31) / 32 * 32);
    p.K = k < p.K ? k : p.K;
  }
  const int nk = (int)((p.K + 63) / 64);
  Core g;
  g.set_lane();
  int bid = blockIdx.x, tm = 0, tn = 0;
  auto next_tile = [&]() {  // the first tile at or behind bid (uniform over the workgroup)
    for (; bid < p.map.total; bid += gridDim.x)
      if (p.map.decode(bid, tm, tn)) return true;
    return false;
  };
  if (!next_tile()) return;
  if (nk == 0) {  // no token takes part
    for (bool more = true; more; bid += gridDim.x, more = next_tile())
      for (int q = threadIdx.x; q < TM * (TN / 8); q += Cfg::NTHREADS) {
        const int64_t m = (int64_t)tm * TM + q / (TN / 8), n = (int64_t)tn * TN + q % (TN / 8) * 8;
        if (m < p.M && n < p.N) *reinterpret_cast<u32x4_t*>(p.Ct + m * p.ldct + n) = u32x4_t{0u, 0u, 0u, 0u};
      }
    return;
  }
  // (a loop of its own for a last slab that is half a slab: with one loop for both the fragments are moved from register to register)
  auto walk = [&](auto half) {
    constexpr bool HALF = decltype(half)::value;
    f32x4_t acc[TnCfg::NB][TnCfg::NBN];
    typename Core::Stream s;
    int64_t m0, n0;  // this tile
    const char *a_next, *b_next;
    bool more;
    auto look_ahead = [&]() {
      m0 = (int64_t)tm * TM;
      n0 = (int64_t)tn * TN;
      bid += gridDim.x;
      more = next_tile();
      a_next = more ? reinterpret_cast<const char*>(p.B + (int64_t)tn * TN) : g.a_base;
      b_next = more ? reinterpret_cast<const char*>(p.a_pcol ? p.A + (int64_t)tm * (TM / 64) * p.a_pcol : p.A + (int64_t)tm * TM) : g.b_base;
    };
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>(lds) + g.wave * 8192;
    auto stage = [&]() { return lds0 + (uint32_t)(Core::ring(s.sb + 4) * TnCfg::STAGE_BYTES); };
    g.init_tn(p.B, p.ldb, (int64_t)tn * TN, p.A, p.lda, (int64_t)tm * TM, p.a_pcol);
    g.prologue(lds, (int64_t)nk * 64);
    g.stream_begin(lds, s);
    look_ahead();
    g.template stream_slab<true>(lds, 0, nk, acc, s, a_next, b_next);
    while (true) {
      for (int it = 1; it < nk - HALF; ++it) g.template stream_slab<false>(lds, it, nk, acc, s, a_next, b_next);
      if constexpr (HALF) g.stream_half_slab(lds, nk, acc, s, a_next, b_next);
      else Core::stream_settle(s);
      Core::retire(acc);
      g.a_base = a_next;
      g.b_base = b_next;
      g.reads_tn(lane_anew());
      if constexpr (HALF) {
        g.stream_fragments(lds, s);
        Core::stream_settle(s);
      }
      LineStores16<TnCfg, Cfg> done(p, m0, n0, g.wave_m, g.wave_n, stage());
      const bool last = !more;
      if (!last) look_ahead();
      g.stream_slab_over(lds, nk, acc, s, a_next, b_next, done, last);
      if (last) break;
    }
    Core::template wait_vm<0>();
  };
  if (p.K % 64 != 0) walk(std::true_type{});
  else walk(std::false_type{});
}

// fp32 rows as three bfloat16 planes, out[r] = three runs of ldo elements.  Row r is in[rows[r]] (in[r] without `rows`) for
// r < R = *n_rows (R without), zeros up to the next multiple of 64.  Eight elements per thread; C a multiple of 8.
struct SplitArgs {
  const float* in;
  int64_t ldi, R, C;
  bf16_t* out;
  int64_t ldo, rpad;
  const int *rows, *n_rows;
};

// Nearest terms: x1 = bf16(x), x2 = bf16(x - x1), x3 = bf16(x - x1 - x2); the differences are exact, so x1 + x2 + x3 = x down to
// the smallest bfloat16.  An infinity would be (inf, NaN, NaN), and its products with the small terms of the other operand,
// which are zeros or of either sign, NaN: values from kWide on are left to split_same_sign.
constexpr uint32_t kWide = 0x5d000000u;  // 2^59: products of smaller values, and any sum of them, stay far from overflow
LCE_DEV void split_nearest(const float (&x)[8], float (&p)[3][8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float rest = x[e];
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      p[t][e] = (float)(bf16_t)rest;
      rest -= p[t][e];
    }
  }
}

// Terms of x's own sign, none of them zero unless x is: cut off instead of rounded (3 x 8 bits hold all 24), a zero term
// replaced by |x| 2^-40.  Every product of an infinity is then an infinity of the right sign, with zero NaN, and so is the sum
// of the six; a finite value beyond the largest bfloat16 stays finite.  Not for ordinary values: the three products that
// are left out do not average out over the signs (4e-8 of a product of N(0,1) values on average, as much as an fp32 rounding).
LCE_DEV void split_same_sign(const float (&x)[8], float (&p)[3][8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, x[e]);
    const float least = __builtin_copysignf(fmaxf(fabsf(x[e]) * 0x1p-40f, 0x1p-126f), x[e]);
    float rest = x[e];
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const float cut = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, rest) & 0xffff0000u);
      p[t][e] = cut == 0.f ? least : cut;
      rest -= cut;
    }
    if ((bits & 0x7f800000u) == 0x7f800000u || (bits & 0x7fffffffu) == 0u) {  // infinities, NaN and zero
      const bool inf = (bits & 0x7fffffffu) == 0x7f800000u;
      p[0][e] = x[e];
      p[1][e] = p[2][e] = inf ? __builtin_copysignf(1.f, x[e]) : x[e];
    }
  }
}

template <bool SAME_SIGN>
LCE_DEV uint32_t split_rows(const SplitArgs& s) {  // returns the largest magnitude this thread has seen, as bits
  const int64_t R = s.n_rows ? (int64_t)*s.n_rows : s.R;
  const int64_t rend = (R + 63) / 64 * 64 < s.rpad ? (R + 63) / 64 * 64 : s.rpad;
  const int64_t per_row = s.C / 8, n = rend * per_row;
  uint32_t most = 0;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = q / per_row, c = (q - r * per_row) * 8;
    float x[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (r < R) {
      const f32x4_t* src = reinterpret_cast<const f32x4_t*>(s.in + (s.rows ? (int64_t)s.rows[r] : r) * s.ldi + c);
      const f32x4_t lo = src[0], hi = src[1];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = e < 4 ? lo[e & 3] : hi[e & 3];
    }
    float p[3][8];
    if (SAME_SIGN) {
      split_same_sign(x, p);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t magnitude = __builtin_bit_cast(uint32_t, x[e]) & 0x7fffffffu;
        most = magnitude > most ? magnitude : most;
      }
      split_nearest(x, p);
    }
    bf16_t* dst = s.out + r * 3 * s.ldo + c;
#pragma unroll
    for (int t = 0; t < 3; ++t) store_run<bf16_t, 8>(dst + t * s.ldo, p[t]);
  }
  return most;
}

// *wide (zero before a call's first launch): some value of the operands split so far is infinite, NaN or kWide and more
inline __global__ void split_planes_kernel(SplitArgs s, int* wide) {
  if (split_rows<false>(s) >= kWide) __hip_atomic_store(wide, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Behind every chunk's split: where such a value has been met, both operands are split again, with terms of one sign.  (It
// may be in either of them and needs the other one's terms that way too.)  Otherwise nothing: 2 us per launch, against a
// second read of both operands to know beforehand.
inline __global__ void split_again_kernel(const int* wide, SplitArgs a, SplitArgs b) {
  if (*wide == 0) return;
  (void)split_rows<true>(a);
  (void)split_rows<true>(b);
}

// ------------------------------------------------------------------------------------------------
// kernels
// ------------------------------------------------------------------------------------------------
template <typename Cfg, bool KEEP = false>
__global__ __launch_bounds__(Cfg::NTHREADS) void lce_fwd16_kernel(FwdArgs<typename Cfg::TIN> p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  int tt, s;
  if (!p.map.decode(blockIdx.x, tt, s)) return;
  const int64_t n0 = (int64_t)tt * Cfg::BN, left = p.T - n0;
  if constexpr (Fwd16Tails<Cfg>::value) {
    // (the weight read once is for a launch of one tile of tokens, and up to 192 that is the 192-wide one: forward_w_once)
    constexpr bool kMoreThan192 = Cfg::A_ONCE && Cfg::NBN > 6;
    if constexpr (!kMoreThan192)
      if (left <= 160) return fwd16_body<typename Fwd16Tails<Cfg>::template Narrow<5>, KEEP>(p, n0, s, lds);
    if constexpr (!kMoreThan192 && Cfg::NBN > 6)
      if (left <= 192) return fwd16_body<typename Fwd16Tails<Cfg>::template Narrow<6>, KEEP>(p, n0, s, lds);
    if constexpr (Cfg::NBN > 6)
      if (left <= 224) return fwd16_body<typename Fwd16Tails<Cfg>::template Narrow<7>, KEEP>(p, n0, s, lds);
  }
  fwd16_body<Cfg, KEEP>(p, n0, s, lds);
}

template <typename Cfg>
__global__ __launch_bounds__(Cfg::NTHREADS) void gemm16_nt_kernel(GemmArgs<typename Cfg::TIN> p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  gemm16_tile<Cfg>(p, blockIdx.x, lds);
}

template <typename Cfg>
__global__ __launch_bounds__(Cfg::NTHREADS) void gemm16_tn_kernel(GemmArgs<typename Cfg::TIN> p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  gemm16_tn_tile<GemmCfg16<typename Cfg::TIN, 1>, Cfg>(p, blockIdx.x, lds);
}

// d_hidden on its own: C[m][n] (+)= sum_k A[m][k] B[k][n] as in gemm16_tile's mixed mode (W read in place), on tiles of 256 or 192 tokens;
// with `by_rows` in use the width and the K slices are those of the rows that take part
template <typename Wide, typename Narrow>
__global__ __launch_bounds__(Wide::NTHREADS) void lce_dh16_kernel(GemmArgs<typename Wide::TIN> p, DhSlices by_rows, bool narrow) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  if (by_rows.n[0]) {
    const int64_t rows = *p.m_dev;
    narrow = by_rows.tile(rows) == 192;
    p.ksplit = by_rows.count(rows);
    p.kslice = ((p.K + p.ksplit - 1) / p.ksplit + Wide::BK - 1) / Wide::BK * Wide::BK;
    p.cf_split_stride = DhSlices::stride(rows, p.N);
    p.map.ncol_tiles = p.n_tiles * p.ksplit;
    p.map.br = 8;  // (what TileMap::with_rows narrows to the tiles there are)
  }
  if (narrow) gemm16_tile<Narrow, GemmCfg16<typename Wide::TIN, 2, Narrow::NBN, Narrow::A_EARLY, 1, Narrow::A_ONCE, Narrow::NB>>(p, blockIdx.x, lds);
  else gemm16_tile<Wide, GemmCfg16<typename Wide::TIN, 2, Wide::NBN, Wide::A_EARLY, 1, Wide::A_ONCE, Wide::NB>>(p, blockIdx.x, lds);
}

// a tile of d_weight (p.tn == 1) or of d_hidden, NBM blocks of hidden columns to a wave
template <typename Cfg, int NBM>
LCE_DEV void any_gemm16_tile(const GemmArgs<typename Cfg::TIN>& p, int bid, char* lds) {
  typedef typename Cfg::TIN TIN;
  if (p.tn == 1) gemm16_tn_tile<GemmCfg16<TIN, 1, 8, 0, Cfg::TERMS, 0, NBM>, Cfg>(p, bid, lds);
  // (W early: the whole step 0.2 to 0.5 % faster from 2048 to 16384 tokens)
  else gemm16_tile<GemmCfg16<TIN, 0, 8, 0, Cfg::TERMS, 0, NBM>, GemmCfg16<TIN, 2, 8, 1, Cfg::TERMS, 0, NBM>>(p, bid, lds);
}

// one launch of the backward's steady state (see lce_bwd_chunk_kernel)
template <typename Cfg, int NBM>
__global__ __launch_bounds__(Cfg::NTHREADS) void lce_bwd_chunk16_kernel(BwdChunkArgs<typename Cfg::TIN> p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int bid = blockIdx.x;
  if (bid < p.n_gw) any_gemm16_tile<Cfg, NBM>(p.gw, bid, lds);
  else if (bid < p.n_gw + p.n_gh) any_gemm16_tile<Cfg, NBM>(p.gh, bid - p.n_gw, lds);
  else ds16_tile<Cfg>(p.ds, bid - p.n_gw - p.n_gh, lds);
}

}  // namespace lce
