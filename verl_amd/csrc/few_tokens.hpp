// Few tokens (gfx950).  16-bit inputs: the forward up to 96, d_hidden up to 128, d_weight up to 256, and d_logits from kept
// logits; fp32 inputs: the forward up to 128 at a time.
//
// With T <= 128 every product is one streaming pass over a [V, H] matrix and bound by HBM, not by the matrix cores:
//   logits      W[v] . hidden[t]                        reads W once; nothing is written (or the kept logits)
//   d_hidden[t][h] = sum_v dS[t][v] * W[v][h]           reads W once; its result is small
//   d_weight[v][h] = sum_t dS[t][v] * hidden[t][h]      writes [V, H] once; its operands (dS, hidden) are small
// The 256 x 256 tiles of the general path spend such a pass waiting: a d_weight tile has a K loop of one or two slabs
// between a cold start and 128 KB of scattered 2-byte stores, and a d_hidden tile keeps two half slabs of W in flight
// per CU.  The kernels here are shaped for the stream instead: workgroups that stay, operands of the next stages on their way
// in registers, and loops without a branch around a load or a store, so that no wait is longer than it has to be.  Reading and
// writing are separate launches: this card reads 1.09 GB in 155 us and writes it in 185, and takes 340 for the two in a row
// but 400 to 500 for both at once.  Everything is plain HIP with compiler-placed waits; K-major operands (hidden[t][.],
// dS[t][.], W[v][.] in the gradients) are read through the transposing LDS read ds_read_b64_tr_b16.
#pragma once
#include <type_traits>

#include "gemm_core.hpp"
#include "lce_kernels.hpp"

namespace lce {

typedef short i16x4_lds_t __attribute__((ext_vector_type(4)));

// Transposing read.  In each group of 16 lanes, lane 4e + q passes the address of four consecutive 16-bit elements of
// row e, X[e][4q' ..]; lane i of the group receives the i-th of the group's 16 columns for rows 0..3, i.e.
// column (i % 4) of the run that lane (i / 4) pointed at in each row.
LCE_DEV u32x2_t tr_read_b64(const char* lds_addr) {
  const i16x4_lds_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (i16x4_lds_t __attribute__((address_space(3)))*)(uintptr_t)(uint32_t)(uintptr_t)lds_addr);
  u32x2_t r;
  __builtin_memcpy(&r, &v, 8);
  return r;
}

template <typename T>
LCE_DEV void mma16(f32x4_t& acc, const u32x4_t& a, const u32x4_t& b) {
  if constexpr (sizeof(T) == 2 && __is_same(T, bf16_t)) {
    bf16x8_t x, y;
    __builtin_memcpy(&x, &a, 16);
    __builtin_memcpy(&y, &b, 16);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, acc, 0, 0, 0);
  } else {
    f16x8_t x, y;
    __builtin_memcpy(&x, &a, 16);
    __builtin_memcpy(&y, &b, 16);
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, y, acc, 0, 0, 0);
  }
}

// swizzle of the 16-byte chunks of a K-major LDS row of 512 bytes (32 chunks): row r holds chunk c at position
// c ^ fw_swz(r), so that the rows one transposing read touches (r, r+1, r+2, r+3 and the same 8 and 16 rows on) fall
// into different banks (values below 16: valid for rows of 16 chunks and of 32)
LCE_DEV int fw_swz(int r) { return ((r & 3) << 2) ^ ((r >> 3) & 3); }

// ------------------------------------------------------------------------------------------------------------------
// Forward, up to 96 tokens (NT: 64 or 96).  Workgroup = 512 threads = 8 waves, one per CU; it owns a contiguous range of vocabulary rows (the
// same number for every workgroup) and goes through it in passes of 256 rows, for each of which K is streamed in stages of 64:
// 256 rows of W x 128 bytes and 64 or 128 rows of hidden x 128 bytes.  What bounds it is the read of W, and that by the bytes in
// flight: DEPTH stages are on their way in registers (128 KB of W per CU) while one is multiplied out of LDS, which holds two,
// so that a stage costs one barrier; and the stages of the next pass follow those of this one without a gap.
// The products are those of the d_logits tiles, 32x32x16 blocks with k ascending (rows: vocabulary, columns: tokens), so logits
// kept here have the bits that a backward without them recomputes.  A wave owns 32 rows x NT tokens; in a short last pass the
// waves without rows stand aside (64 tokens: 182 -> 174 us).
// Measured, kernel and merge, against the 256 x 64 tile with a ring of whole LDS stages (H, V: before -> after): 64 tokens,
// 3584, 152064: 184 -> 174 us; 4096, 128256: 175 -> 160; 896, 151936: 58 -> 50; the same access pattern without any
// arithmetic takes 170, 163 and 41.  65 / 80 / 96 tokens against the 256 x 128 tile: 3584: 198 / 202 / 204 -> 186 / 193 / 197 us, 5120:
// 283 / 288 / 293 -> 266 / 276 / 285, 4096: 172 / 172 / 173 -> 166 / 172 / 173, 896: 57 / 57 / 57.5 -> 56; forward + backward 3584: 635 /
// 651 / 667 -> 622 / 639 / 655, 4096: 575 / 578 / 584 -> 560 / 567 / 577.  (97 to 128 tokens so: 206 / 211 -> 224 / 230, the tile stays.)
// fp32 inputs run it up to 128 tokens, on the fp32 MFMA, which is the bound from some 40 tokens on (64 tokens, 1.09 G products of W's
// elements: 445 us at its peak rate): the narrowest of 32, 64, 96 and 128 tokens that holds them.  Against the 256 x 64 and 256 x 128
// tiles, H=3584: 1 to 32 tokens 750 -> 440 us, 64: 746 -> 673, 65 to 96: 1335 -> 936, 128: 1335 -> 1220; H=896: 202 -> 113, 202 -> 188,
// 360 -> 285, 354 -> 333.
// ------------------------------------------------------------------------------------------------------------------
template <typename TIN, int NT_>
struct FewFwdShape {
  static constexpr int NT = NT_, DEPTH = sizeof(TIN) == 2 || NT == 32 ? 4 : 3, BM = 256, FN = NT / 32;
  static constexpr int BK = 128 / (int)sizeof(TIN);  // K elements of a stage
  static constexpr int HROWS = (NT + 63) / 64 * 64;  // rows of a stage of hidden in LDS (64 are fetched at a time)
  static constexpr int STAGE = BM * 128 + HROWS * 128;
  static constexpr int LDS_BYTES = 2 * STAGE + 8 * 4096;  // two stages, a store tile per wave
};

// The products of W's rows [row0, vend64) with the NT hidden rows, 256 rows of W at a time; `pass(acc, m0, vbase, busy)` gets those of
// rows vbase .. vbase + 31 (this wave's; busy: some exist) in acc[0][j][.], column j * 32 + lane % 32.  h_off: byte offset of hidden row
// tid / 8 + 64 i (beyond h_bytes: reads as zero) in the h_bytes behind h.
// HALF: a pass is whole turns of the loop over the DEPTH stages in flight and half a one (16 bits: H is a multiple of 128 but not of
// 256), and every second pass starts at the second half of the ring.  Rounded up to whole turns, a seventh of the stages were zeros at
// H=896: 1 / 40 / 64 tokens, V=151936, 50.7 / 51.7 / 52.1 -> 49.2 / 49.6 / 50.0 us.  (A branch around them in the loop costs more than they
// do: 57 us; the waits behind it are for all loads.)
template <typename TIN, int NT, int AUX, bool HALF, typename F>
LCE_DEV void few_products(const TIN* W, int64_t ldw, int64_t row0, int64_t vend64, int64_t H, const TIN* h, int64_t h_bytes,
                          const uint32_t (&h_off)[FewFwdShape<TIN, NT>::HROWS / 64], char* lds, F&& pass) {
  typedef FewFwdShape<TIN, NT> S;
  constexpr int DEPTH = S::DEPTH, FN = S::FN, HL = S::HROWS / 64;
  constexpr int WL = S::BM / 64;  // 16-byte chunks of a W stage per thread: row tid / 8 + 64 i, chunk tid % 8
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, hh = lane >> 5, ln = lane & 31;
  const int vend = (int)vend64;
  const int n_k = (int)(H / S::BK), n_kp = HALF ? n_k : (n_k + DEPTH - 1) / DEPTH * DEPTH;  // stages of a pass, of whole turns of the loop

  // rows beyond the range, tokens beyond T and stages beyond K read as zero
  const uint32_t w_row = (uint32_t)(ldw * sizeof(TIN));
  const uint32_t w_at = (uint32_t)(tid >> 3) * w_row + (tid & 7) * 16;
  u32x4_t pw[DEPTH][WL], pb[DEPTH][HL];
  int64_t f_row = row0;  // the next stage to fetch: first row of its pass, k
  int f_k = 0;
  auto fetch = [&](u32x4_t (&w)[WL], u32x4_t (&x)[HL]) {
    const int64_t left = vend64 - f_row < S::BM ? vend64 - f_row : S::BM;
    const bool live = f_k < n_k && left > 0;
    const buf_t wb = make_buf(W + f_row * ldw + S::BK * (int64_t)f_k, live ? left * w_row - 128 * (int64_t)f_k : 0);
    const buf_t hb = make_buf(h + S::BK * (int64_t)f_k, live ? h_bytes - 128 * (int64_t)f_k : 0);
#pragma unroll
    for (int i = 0; i < WL; ++i) w[i] = __builtin_amdgcn_raw_buffer_load_b128(wb, (int)(w_at + 64 * i * w_row), 0, AUX);
#pragma unroll
    for (int i = 0; i < HL; ++i) x[i] = __builtin_amdgcn_raw_buffer_load_b128(hb, (int)h_off[i], 0, 0);
    __builtin_amdgcn_sched_barrier(0);  // (the loads of one stage stay in front of the next one's)
    if (++f_k == n_kp) {
      f_k = 0;
      f_row += S::BM;
    }
  };
  // chunk c of row r lies at c ^ swz(r); rows 32 apart share the pattern
  auto swz = [](int r) { return (r ^ ((r >> 3) & 1)) & 7; };
  const int put = (tid >> 3) * 128 + (((tid & 7) ^ swz(tid >> 3)) * 16);
  const int a_rd = (wave * 32 + ln) * 128, b_rd = S::BM * 128 + ln * 128, sw = swz(ln);
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) fetch(pw[d], pb[d]);
  int buf = 0;
  f32x16_t acc[1][FN];
  int64_t m0 = row0;
  auto begin = [&] {
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[0][j][r] = 0.f;
  };
  // stages [D0, D1) of a turn
  auto stages = [&](auto d0, auto d1) {
    const bool busy = m0 + wave * 32 < vend;  // (a short last pass leaves the LDS to the waves that have rows)
#pragma unroll
    for (int d = d0.value; d < d1.value; ++d) {
      char* st = lds + buf * S::STAGE;
      buf ^= 1;
#pragma unroll
      for (int i = 0; i < WL; ++i) *reinterpret_cast<u32x4_t*>(st + put + i * 8192) = pw[d][i];
#pragma unroll
      for (int i = 0; i < HL; ++i) *reinterpret_cast<u32x4_t*>(st + S::BM * 128 + put + i * 8192) = pb[d][i];
      fetch(pw[d], pb[d]);
      // (a buffer is written again two stages on: every wave has passed the barrier between, after its reads of this stage)
      __syncthreads();
      if (busy) {
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          const int c = ((2 * kk + hh) ^ sw) * 16;
          const u32x4_t af = *reinterpret_cast<const u32x4_t*>(st + a_rd + c);
          u32x4_t bf[FN];
#pragma unroll
          for (int j = 0; j < FN; ++j) bf[j] = *reinterpret_cast<const u32x4_t*>(st + b_rd + j * 4096 + c);
#pragma unroll
          for (int j = 0; j < FN; ++j) Mma<TIN>::run(acc[0][j], af, bf[j]);
        }
      }
    }
  };
  auto end = [&] {
    const int vbase = (int)m0 + wave * 32;  // this wave's first row
    pass(acc, m0, vbase, vbase < vend);
    m0 += S::BM;
  };
  constexpr std::integral_constant<int, 0> zero{};
  constexpr std::integral_constant<int, DEPTH / 2> half{};
  constexpr std::integral_constant<int, DEPTH> whole{};
  while (m0 < vend64) {
    begin();
    for (int k0 = 0; k0 < (HALF ? n_k - DEPTH / 2 : n_kp); k0 += DEPTH) stages(zero, whole);
    if constexpr (HALF) stages(zero, half);
    end();
    if constexpr (HALF) {
      if (m0 >= vend64) break;
      begin();
      stages(half, whole);
      for (int k0 = DEPTH / 2; k0 < n_k; k0 += DEPTH) stages(zero, whole);
      end();
    }
  }
}

// Forward.  AUX: cache policy of the loads of W
template <typename TIN, int NT, int AUX, bool HALF>
LCE_DEV void fwd_few_body(const FwdArgs<TIN>& p, char* lds) {
  typedef FewFwdShape<TIN, NT> S;
  constexpr int FN = S::FN, HL = S::HROWS / 64;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, hh = lane >> 5, ln = lane & 31;
  const int64_t row0 = (int64_t)blockIdx.x * p.split_stride;
  const int64_t vend64 = row0 + p.split_span < p.V ? row0 + p.split_span : p.V;
  const int vend = (int)vend64;
  float m[FN], a[FN], b[FN];
  int lab[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    m[j] = kNegBig;
    a[j] = 0.f;
    b[j] = 0.f;
    const int64_t t = j * 32 + ln;
    const int64_t y = t < p.T ? p.labels[t] - p.label_offset : -1;
    lab[j] = (y >= 0 && y < p.V) ? (int)y : -1;
  }
  const uint32_t h_row = (uint32_t)(p.ldh * sizeof(TIN));
  uint32_t h_off[HL];
#pragma unroll
  for (int i = 0; i < HL; ++i) h_off[i] = (uint32_t)((tid >> 3) + 64 * i) * h_row + (tid & 7) * 16;
  few_products<TIN, NT, AUX, HALF>(p.W, p.ldw, row0, vend64, p.H, p.h, p.T * h_row, h_off, lds,
                             [&](f32x16_t (&acc)[1][FN], int64_t m0, int vbase, bool) {
    if (p.xcache) {
      // the logits of this pass, for a backward that then has no need to recompute them.  A 32x32 block passes through 4 KB of
      // LDS of this wave's own and leaves it as whole lines, 1 KB (16 tokens x 16 rows of a panel) per store; rows in whole
      // fours, the last ones of W up to the end of the cache's panel.  Non-temporal (64 tokens, H=3584: step 632 -> 615 us,
      // 40: 611 -> 597; the stores leave while W streams in, and unmarked they wait for lines of the caches).
      char* sC = lds + 2 * S::STAGE + wave * 4096;
      const int p4 = lane & 3, pt = lane >> 2;  // as it leaves: quad of rows, token
#pragma unroll
      for (int j = 0; j < FN; ++j) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int c = 2 * (q & 1) + hh;
          *reinterpret_cast<f32x4_t*>(sC + (q >> 1) * 2048 + ln * 64 + ((c ^ ((ln >> 1) & 3)) * 16)) =
              f32x4_t{acc[0][j][4 * q], acc[0][j][4 * q + 1], acc[0][j][4 * q + 2], acc[0][j][4 * q + 3]};
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int tl = 16 * (q & 1) + pt;
          const f32x4_t x4 = *reinterpret_cast<const f32x4_t*>(sC + (q >> 1) * 2048 + tl * 64 + ((p4 ^ ((tl >> 1) & 3)) * 16));
          const int v = vbase + 16 * (q >> 1) + 4 * p4;
          const int64_t t = j * 32 + tl;
          if (t < p.T && v < vend) __builtin_nontemporal_store(x4, reinterpret_cast<f32x4_t*>(kept_logit(p.xcache, p.xtok, t, v)));
        }
      }
    }
    fold_logits<1, FN>(acc, m, a, b, lab, p.c, vbase, vend, m0 + S::BM <= vend64, hh, p.xlabel + ln);
  });

  // merge the two lane halves (same token, different vocabulary rows), then the waves
  __syncthreads();
  f32x4_t* red = reinterpret_cast<f32x4_t*>(lds);  // [8][NT]
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const float m2 = __shfl_xor(m[j], 32), a2 = __shfl_xor(a[j], 32), b2 = __shfl_xor(b[j], 32);
    merge_stats(m[j], a[j], b[j], m2, a2, b2, p.c);
    if (hh == 0) red[wave * NT + j * 32 + ln] = f32x4_t{m[j], a[j], b[j], 0.f};
  }
  __syncthreads();
  if (tid < NT) {
    const int t = tid;
    const f32x4_t v0 = red[t];
    float vm = v0[0], va = v0[1], vb = v0[2];
#pragma unroll
    for (int w = 1; w < 8; ++w) {
      const f32x4_t u = red[w * NT + t];
      merge_stats(vm, va, vb, u[0], u[1], u[2], p.c);
    }
    if (t < p.T) p.parts[(int64_t)blockIdx.x * p.T + t] = f32x4_t{vm, va, vb, 0.f};
  }
}

// (which rows are read how: read_w_once, lce_host.hpp.  A branch around the whole body: none around a load.)
template <typename TIN, int NT, bool HALF>
__global__ __launch_bounds__(512, 2) void lce_fwd_few_kernel(FwdArgs<TIN> p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  if ((int64_t)blockIdx.x * p.split_stride < p.once_rows) fwd_few_body<TIN, NT, kBufNonTemporal, HALF>(p, lds);
  else fwd_few_body<TIN, NT, 0, HALF>(p, lds);
}

template <typename TIN>
struct FewArgs {
  const TIN* dS;      // d_logits of the chunk by (compact) token position, >= kt of them, at ds_at; columns in Perm order;
  int64_t ldS, pcol;  //   zero rows beyond the tokens that take part, zero columns beyond the chunk's rows
  const TIN* Ht;      // compact copy of hidden, [>= kt rows][ldHt], ldHt >= round_up(H, 256); zero rows beyond the tokens
  int64_t ldHt;
  const TIN* W;       // first row of the chunk, row stride ldw
  int64_t ldw;
  int64_t vrows;      // rows of the chunk
  int64_t ucols;      // columns of dS that are written (vrows rounded up to the permutation group)
  int64_t H;
  int kt;             // token positions summed over by d_weight: a multiple of 32, <= 128
  int nt;             // token rows of d_hidden's result that exist (<= 128)
  const int* n_rows;  // device-side count of the token positions that take part (null: kt)
  void* dW;           // [vrows][H] rows of d_weight of this chunk (TOUT)
  float* dHp;         // fp32 partials of d_hidden: slice s at dHp + s * part_stride, [nt][H]
  int64_t part_stride;
  int ksplit;         // K slices of d_hidden
  int64_t kslice;     // columns of dS per slice, a multiple of 64
  int accumulate;     // d_hidden partials: 0 store, 1 add to what is there (second and later chunks)
  int n_su;           // d_weight: workgroups side by side along the vocabulary
  int by_xcd;         // d_hidden: each XCD takes a contiguous eighth of the workgroups
};

// ------------------------------------------------------------------------------------------------------------------
// d_weight, up to 256 tokens.  Workgroup = 512 threads = 8 waves, one per CU; it owns 512 columns of H, whose hidden values its
// waves keep in registers as MFMA operands for good (64 columns of up to KT tokens each: KT / 2 registers), and walks the 64-column
// blocks of dS id / n_ht, id / n_ht + n_su, ...; a wave multiplies its columns of H with all 64 columns of the block:
//   C[m = h][n = u] = sum_t Ht[t][h] * dS[t][u].
// What bounds it is the write of [V, H], up to some 130 tokens at the rate of a plain fill, beyond that with the matrix pipes next
// to it (two waves per SIMD: one multiplies while the other converts and stores).  The workgroups side by side write the pieces
// of the same rows at about the same time and the chip works its way through d_weight as one window of n_su x 64 rows.  The stores
// are marked non-temporal: d_weight is larger than every cache, and unmarked its lines push out the dS that all of
// the columns' workgroups are about to read (the same kernel with plain stores: 130 tokens 293 us, with these 178; 256: 305, 260).
// MFMA rows are assigned to h in pairs of blocks: block 2i'+b, row 4g+r  <->  h = 32i' + 8g + 4b + r, so a lane ends
// up with 8 consecutive h for one u.  With 16-bit output a wave's results pass through a tile of its own in LDS and
// leave it as whole 128-byte lines, eight lanes per row; fp32 output is stored from the registers, 16 rows x 128 bytes
// per instruction.
// Measured, forward + backward in us, H=3584, V=152064, against workgroups of 256 columns and a map that left dS to all XCDs (up to
// 128 tokens) and lce_dw16_kernel's tiles of 256 x 256 (beyond), both with plain stores: 64 tokens 650 -> 631, 128: 786 -> 717,
// 130: 903 -> 796, 192: 933 -> 838, 256: 1050 -> 945; H=896, 192 tokens: 353 -> 315.  At 333 tokens a wave would have to share its
// registers among fewer columns, the LDS reads of dS bind (32 columns: 1287) and the tiles are faster (1240).
// ------------------------------------------------------------------------------------------------------------------
constexpr int64_t kDwFewMaxTokens = 256;

// swizzle of the 16-byte chunks of a dS tile's rows of 128 bytes: half a wave's transposing read takes 32 bytes of the rows r .. r+3
// and r+8 .. r+11, which lie in different banks this way (two rows fill the banks once)
LCE_DEV int ds_swz(int r) { return (r & 2) ^ ((r & 8) >> 1); }

template <int KT, typename TOUT>
struct DwFewShape {
  static_assert(KT % 64 == 0 && KT <= kDwFewMaxTokens, "token positions");
  static constexpr int HW = 512;                                 // columns of H per workgroup
  static constexpr int TILE = KT * 128;                          // a block of dS
  static constexpr int STG = sizeof(TOUT) == 2 ? 8192 : 0;       // a wave's store tile
  static constexpr int WALK = 2 * TILE + 8 * STG, HID = 64 * HW * 2;  // (64 rows of hidden at a time, before the walk)
  static constexpr int LDS_BYTES = WALK > HID ? WALK : HID;
};

template <typename TIN, typename TOUT, typename Perm, int KT>
__global__ __launch_bounds__(512, 2) void lce_dw_few_kernel(FewArgs<TIN> p) {
  typedef DwFewShape<KT, TOUT> S;
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  constexpr int KS = KT / 32, HW = S::HW, RB = HW * 2, CPR = HW / 8;  // bytes and 16-byte chunks of a row of the hidden tile
  constexpr int MI = 4, NJ = 4, BL = KT * 8 / 512;
  constexpr int AHEAD = KT < 256 ? 1 : 0;  // k-steps of dS fragments read ahead (at 256 tokens there are no registers for one)
  constexpr bool STAGE = sizeof(TOUT) == 2;
  constexpr int STORES = STAGE ? 2 * NJ : MI * NJ;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int g = lane >> 4, l16 = lane & 15, e = l16 >> 2, q = l16 & 3;
  const int n_ht = (int)((p.H + HW - 1) / HW);
  // each XCD takes a contiguous eighth of the numbering (columns of H fastest): the workgroups that walk the same blocks of dS
  // sit on one or two XCDs, and dS passes into each L2 about once
  const int id = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
  if (id >= n_ht * p.n_su) return;
  const int ht = id % n_ht;
  const int64_t h0 = (int64_t)ht * HW, hw = h0 + 64 * wave;  // the workgroup's first column, this wave's
  const bool live = hw < p.H;                                // (H is a multiple of 64)
  const int64_t n_ub = p.ucols / 64;
  char* sB = lds;                           // two dS tiles: KT rows x 128 bytes, chunk c of row r at c ^ ds_swz(r)
  char* sC = lds + 2 * S::TILE + wave * S::STG;
  int n_tok = p.kt;  // token positions that take part (a device-side count may cut the host's)
  if (p.n_rows) n_tok = *p.n_rows < n_tok ? *p.n_rows : n_tok;
  u32x4_t pre[BL];
  auto fetch = [&](int64_t ub) {
    const buf_t panel = make_buf(ds_at(p.dS, p.ldS, p.pcol, 0, ub * 64), n_tok * 128);  // rows of 128 bytes; zeros beyond
#pragma unroll
    for (int i = 0; i < BL; ++i) pre[i] = __builtin_amdgcn_raw_buffer_load_b128(panel, tid * 16 + i * 8192, 0, 0);
  };
  auto stash = [&](char* to) {
#pragma unroll
    for (int i = 0; i < BL; ++i) {
      const int at = tid + i * 512, r = at >> 3, c = at & 7;
      *reinterpret_cast<u32x4_t*>(to + r * 128 + ((c ^ ds_swz(r)) * 16)) = pre[i];
    }
  };
  int64_t ub = id / n_ht;  // (< n_ub: at most that many side by side)
  const int64_t ub_last = ub + (n_ub - 1 - ub) / p.n_su * p.n_su;
  fetch(ub);
  // hidden -> LDS -> fragments, 64 tokens at a time (zeros behind the last token)
  u32x4_t af[KS][MI];
  const buf_t hid = make_buf(p.Ht, (int64_t)n_tok * p.ldHt * sizeof(TIN));
#pragma unroll
  for (int part = 0; part < KT / 64; ++part) {
    if (part) __syncthreads();
#pragma unroll
    for (int i = 0; i < 64 * CPR / 512; ++i) {
      const int at = tid + i * 512, r = at / CPR, c = at % CPR;
      const int from = h0 + c * 8 < p.H ? (int)(((64 * part + r) * p.ldHt + h0 + c * 8) * sizeof(TIN)) : kBufNowhere;
      *reinterpret_cast<u32x4_t*>(lds + r * RB + ((c ^ fw_swz(r)) * 16)) = __builtin_amdgcn_raw_buffer_load_b128(hid, from, 0, 0);
    }
    __syncthreads();
#pragma unroll
    for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        // block i = 2i' + b: the run of lane q starts at column 64 wave + 32 i' + 8 q + 4 b
        const int col = 64 * wave + 32 * (i >> 1) + 8 * q + 4 * (i & 1);
        const int r0 = 32 * k2 + 8 * g + e, r1 = r0 + 4;
        const u32x2_t lo = tr_read_b64(lds + r0 * RB + (((col >> 3) ^ fw_swz(r0)) * 16) + (col & 7) * 2);
        const u32x2_t hi = tr_read_b64(lds + r1 * RB + (((col >> 3) ^ fw_swz(r1)) * 16) + (col & 7) * 2);
        af[2 * part + k2][i] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
      }
  }
  __syncthreads();
  const int ks_n = (n_tok + 31) / 32;
  // where this lane stores, relative to the block's first row (an aligned run of 64 columns of dS is a permutation of the
  // same 64 rows of the vocabulary): through LDS 16 bytes of eight rows, else runs of 8 columns of four rows
  int at[STAGE ? 2 * NJ : NJ];
#pragma unroll
  for (int k = 0; k < (STAGE ? 2 * NJ : NJ); ++k) {
    const int row = STAGE ? 8 * k + (lane >> 3) : 16 * k + l16;
    const int64_t h = hw + (STAGE ? ((lane & 7) ^ ((row >> 1) & 7)) * 8 : 8 * g);
    at[k] = live ? (int)((Perm::vocab_at(row) * p.H + h) * sizeof(TOUT)) : kBufNowhere;
  }
  stash(sB);
  fetch(ub < ub_last ? ub + p.n_su : ub);
  // (as many dropped stores as a turn of the loop issues behind its fetch: the compiler waits for the fetch in the next turn, and
  // only with that many younger operations on either way into the loop not for the previous block's stores as well)
#pragma unroll
  for (int k = 0; k < STORES; ++k)
    __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{0u, 0u, 0u, 0u}, make_buf(p.dW, 0), kBufNowhere + 16 * k, 0, 0);
  for (int buf = 0; ub <= ub_last; ub += p.n_su, buf ^= 1) {
    // one barrier per block: this block's tile is in LDS, and every wave is done with the other buffer
    __syncthreads();
    const char* tB = sB + buf * S::TILE;
    f32x4_t acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    u32x4_t bf[1 + AHEAD][NJ];
    auto frags = [&](int ks, u32x4_t (&b)[NJ]) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        // lanes (e, q) of group g address row 32 ks + 8 g + e (+4), columns 16 j + 4 q ..
        const int r0 = 32 * ks + 8 * g + e, r1 = r0 + 4, col = 16 * j + 4 * q;
        const u32x2_t lo = tr_read_b64(tB + r0 * 128 + (((col >> 3) ^ ds_swz(r0)) * 16) + (col & 7) * 2);
        const u32x2_t hi = tr_read_b64(tB + r1 * 128 + (((col >> 3) ^ ds_swz(r1)) * 16) + (col & 7) * 2);
        b[j] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
      }
    };
    if (live) {  // (the last workgroup of a row may have waves without columns)
      if (AHEAD) frags(0, bf[0]);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        if (!AHEAD) frags(ks, bf[0]);
        else if (ks + 1 < KS) frags(ks + 1, bf[(ks + 1) & AHEAD]);  // (zeros behind the last token)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) mma16<TIN>(acc[i][j], af[ks][i], bf[ks & AHEAD][j]);
        if (ks + 1 >= ks_n) break;
      }
    }
    stash(sB + (buf ^ 1) * S::TILE);  // (behind the last block: the last one again)
    fetch(ub + 2 * p.n_su <= ub_last ? ub + 2 * p.n_su : ub_last);
    const int64_t u0 = ub * 64, left = p.vrows - u0 < 64 ? p.vrows - u0 : 64;
    const buf_t out = make_buf(static_cast<TOUT*>(p.dW) + u0 * p.H, (left > 0 ? left : 0) * p.H * sizeof(TOUT));
    if constexpr (STAGE) {
      // Whole 128-byte lines per store: the wave's 64 rows x 64 columns go through a tile of its own in LDS (16-byte
      // chunk c of row r at c ^ ((r / 2) % 8), so that the 16 rows x 4 chunks of one write fall into different banks)
      // and leave it eight rows at a time, eight lanes per row.  No barrier: LDS operations of one wave complete in order.
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int ip = 0; ip < MI / 2; ++ip) {
          float d[8];
#pragma unroll
          for (int x = 0; x < 8; ++x) d[x] = acc[2 * ip + (x >> 2)][j][x & 3];
          const int row = 16 * j + l16, c = 4 * ip + g;
          store_run<TOUT, 8>(reinterpret_cast<TOUT*>(sC + row * 128 + ((c ^ ((row >> 1) & 7)) * 16)), d);
        }
#pragma unroll
      for (int k = 0; k < 2 * NJ; ++k) {
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(sC + (k * 8 + (lane >> 3)) * 128 + (lane & 7) * 16);
        __builtin_amdgcn_raw_buffer_store_b128(v, out, at[k], 0, kBufNonTemporal);
      }
    } else {
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int i = 0; i < MI; ++i)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc[i][j]), out, at[j] == kBufNowhere ? at[j] : at[j] + (32 * (i >> 1) + 4 * (i & 1)) * 4,
                                                 0, kBufNonTemporal);
    }
  }
}

// ------------------------------------------------------------------------------------------------------------------
// d_hidden, few tokens.  Workgroup = 512 threads = 8 waves, one per CU; it owns columns [h0, h0 + 256) of the result for all
// NT token rows and one K slice of the chunk's dS columns; wave w multiplies columns h0 + 64 (w % 4) .. +63 with half of the
// token rows:  C[m = h][n = t] = sum_u W[vocab_at(u)][h] * dS[t][u].
// A stage is 64 columns of dS: 64 rows of W (512 bytes of each, fetched in the order of dS's columns) and NT x 128
// bytes of dS.  What bounds it is the read of W, and that by the bytes in flight: four stages are on their way in registers
// (128 KB of W per CU) while one is multiplied out of LDS, which holds two, so that a stage costs one barrier.  Beyond 64 tokens, where
// the tiles of dS take registers too, three stages were slower, us of a step: 100 / 128 tokens, H=3584, three 674 / 686, four 667 / 678;
// H=5120 935 / 950, 923 / 945; other H level.
// The workgroups of one slice read the same dS.  Numbered across the XCDs, the neighbours of a slice read pieces of the same rows of W at
// the same time; numbered within them (by_xcd), dS passes into each L2 about once instead of in all eight.  The second from 33 tokens
// on, where dS is a tenth of W and more: frozen head, 64 tokens, H=3584 410.8 -> 406.0 us, 4096: 377.5 -> 368.2, 5120: 569.4 -> 565.0;
// step of 1 / 16 tokens at H=3584 566 -> 573, 581 -> 583.
// ------------------------------------------------------------------------------------------------------------------
template <int KT>
struct FewShape {  // KT: token positions, 64 up to 64 tokens, else 128
  static constexpr int HW = 256;                                     // columns of H per workgroup
  static constexpr int DH_DEPTH = 4;
  static constexpr int DH_STAGE = 64 * HW * 2 + KT * 128;            // W rows, dS tile
  static constexpr int DH_LDS = 2 * DH_STAGE;
};

template <typename TIN, typename Perm, int NT>
__global__ __launch_bounds__(512, 2) void lce_dh_few_kernel(FewArgs<TIN> p) {
  static_assert(NT == 64 || NT == 128, "token rows of a tile");
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  typedef FewShape<NT> S;
  constexpr int HW = S::HW, DEPTH = S::DH_DEPTH;
  constexpr int NJ = NT / 32, MI = 4;       // 16-wide MFMA blocks of a wave: tokens, columns
  constexpr int RB = HW * 2, CPR = HW / 8;  // bytes and 16-byte chunks of a W stage's row
  constexpr int WL = 64 * CPR / 512;        // chunks of a W stage per thread: row tid / CPR + (512 / CPR) i, chunk tid % CPR
  constexpr int BL = NT * 8 / 512;          // ... of the dS stage
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wc = wave & 3, wt = wave >> 2;
  const int g = lane >> 4, l16 = lane & 15, e = l16 >> 2, q = l16 & 3;
  const int n_ht = (int)((p.H + HW - 1) / HW);
  const int id = p.by_xcd ? (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3) : (int)blockIdx.x;
  if (id >= n_ht * p.ksplit) return;
  const int ht = id % n_ht, s = id / n_ht;
  const int64_t h0 = (int64_t)ht * HW;
  const int64_t k_begin = (int64_t)s * p.kslice;
  const int64_t k_left = p.ucols - k_begin;
  const int n_st = k_left <= 0 ? 0 : (int)((k_left < p.kslice ? k_left : p.kslice) / 64);  // stages (both are multiples of 64)

  f32x4_t acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // what this lane fetches of a stage, relative to the stage's first row of W (an aligned run of 64 columns of dS is a
  // permutation of the same 64 rows) and to its panel of dS.  Rows beyond the chunk and columns beyond H read as zero.
  const int ch = tid % CPR;
  int w_at[WL];
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int r = tid / CPR + (512 / CPR) * i;
    w_at[i] = h0 + ch * 8 < p.H ? (int)((Perm::vocab_at(r) * p.ldw + h0 + ch * 8) * sizeof(TIN)) : kBufNowhere;
  }
  int n_tok = p.kt;  // token positions that take part (a device-side count may cut the host's)
  if (p.n_rows) n_tok = *p.n_rows < n_tok ? *p.n_rows : n_tok;
  u32x4_t pw[DEPTH][WL], pb[DEPTH][BL];
  auto fetch = [&](u32x4_t (&w)[WL], u32x4_t (&b)[BL], int st) {
    // (stages behind the last one: W reads as zero; the number of stages is rounded up to whole turns of the loop below)
    const int64_t k0 = k_begin + 64 * (int64_t)(st < n_st ? st : n_st - 1), left = p.vrows - k0 < 64 ? p.vrows - k0 : 64;
    const buf_t wb = make_buf(p.W + k0 * p.ldw, (left > 0 && st < n_st ? left : 0) * p.ldw * sizeof(TIN));
#pragma unroll
    for (int i = 0; i < WL; ++i) w[i] = __builtin_amdgcn_raw_buffer_load_b128(wb, w_at[i], 0, kBufNonTemporal);
    const buf_t panel = make_buf(ds_at(p.dS, p.ldS, p.pcol, 0, k0), n_tok * 128);  // rows of 128 bytes
#pragma unroll
    for (int i = 0; i < BL; ++i) b[i] = __builtin_amdgcn_raw_buffer_load_b128(panel, tid * 16 + i * 8192, 0, 0);
    __builtin_amdgcn_sched_barrier(0);  // (the loads of one stage stay in front of the next one's)
  };
  if (n_st > 0) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) fetch(pw[d], pb[d], d);
  }
  int buf = 0;
  for (int st0 = 0; st0 < n_st; st0 += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      char* sA = lds + buf * S::DH_STAGE;  // 64 rows x RB bytes, chunk c of row r at c ^ fw_swz(r)
      char* sB = sA + 64 * RB;             // NT rows x 128 bytes, chunk c of row t at c ^ ((t >> 1) & 7)
      buf ^= 1;
#pragma unroll
      for (int i = 0; i < WL; ++i) {
        const int r = tid / CPR + (512 / CPR) * i;
        *reinterpret_cast<u32x4_t*>(sA + r * RB + ((ch ^ fw_swz(r)) * 16)) = pw[d][i];
      }
#pragma unroll
      for (int i = 0; i < BL; ++i) {
        const int id = tid + i * 512, t = id >> 3, c = id & 7;
        *reinterpret_cast<u32x4_t*>(sB + t * 128 + ((c ^ ((t >> 1) & 7)) * 16)) = pb[d][i];
      }
      fetch(pw[d], pb[d], st0 + d + DEPTH);
      // (a buffer is written again two stages on: every wave has passed the barrier between, after its reads of this stage)
      __syncthreads();
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        u32x4_t af[MI], bf[NJ];
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          const int col = 64 * wc + 16 * i + 4 * q;
          const int r0 = 32 * ks + 8 * g + e, r1 = r0 + 4;
          const u32x2_t lo = tr_read_b64(sA + r0 * RB + (((col >> 3) ^ fw_swz(r0)) * 16) + (col & 7) * 2);
          const u32x2_t hi = tr_read_b64(sA + r1 * RB + (((col >> 3) ^ fw_swz(r1)) * 16) + (col & 7) * 2);
          af[i] = u32x4_t{lo[0], lo[1], hi[0], hi[1]};
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          const int t = (NT / 2) * wt + 16 * j + l16, c = 4 * ks + g;  // k = 32 ks + 8 g .. +7 of token row t
          bf[j] = *reinterpret_cast<const u32x4_t*>(sB + t * 128 + ((c ^ ((t >> 1) & 7)) * 16));
        }
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) mma16<TIN>(acc[i][j], af[i], bf[j]);
      }
    }
  }
  // lane (g, l16): h = h0 + 64 wc + 16 i + 4 g + (0..3) of token row NT/2 wt + 16 j + l16
  float* out = p.dHp + (int64_t)s * p.part_stride;
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int t = (NT / 2) * wt + 16 * j + l16;
    if (t >= p.nt) continue;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int64_t h = h0 + 64 * wc + 16 * i + 4 * g;
      if (h >= p.H) continue;  // (H is a multiple of 4)
      float* dst = out + (int64_t)t * p.H + h;
      f32x4_t v = acc[i][j];
      if (p.accumulate) v += *reinterpret_cast<const f32x4_t*>(dst);
      *reinterpret_cast<f32x4_t*>(dst) = v;
    }
  }
}

// ------------------------------------------------------------------------------------------------------------------
// d_logits of a vocabulary chunk, or of its first rows, from logits that the forward kept (FwdArgs::xcache): what the
// d_logits tiles compute from their accumulators, here from the kept x(t, v), element by element with the same
// expressions, so the same bits.  One pass over 4 bytes per logit instead of a pass over W.  Workgroup b owns the 64
// columns [64 b, 64 b + 64) of dS, which lie within one group of the vocabulary order Perm (a whole group of the
// eight-wave tiles' order, half a group of the 16x16x32 tiles'), and the first `nrows` compact token positions, of which it
// writes as many as a reader takes: up to the tokens that take part, rounded up to the d_weight product's K granule (64, and
// two slabs at least) for the tiles, and `exact`ly those for the streaming kernels, which read zeros behind them (1 / 8 / 24 tokens,
// H=3584: step 559 / 569 / 580 -> 551 / 563 / 577 us, H=4096 528 / 538 / 550 -> 523 / 534 / 548; from 40 on level).
// Positions beyond the tokens and columns beyond the chunk's rows (the grid covers whole 256-row
// tiles) are written as zeros, as the tiles write them.  Eight lanes share a position: they read the 256 bytes of its
// token's logits behind the 64 columns and write 128 bytes of dS.  Bound by HBM; the constants come from the per-position
// table (worked out per workgroup they were six dependent loads and a logarithm per position) and four positions are on
// their way at once.
// p: the chunk's DsArgs (W, h, the tile map and the range are not used); x: the kept logits from the chunk's first row
// on (a multiple of 16), of xtok tokens.  TERMS == 6: d_logits in three planes, 10 bytes moved per logit; 25344 columns of 1024
// tokens 51 us, 5.1 TB/s.
// ------------------------------------------------------------------------------------------------------------------
template <typename TIN, typename Perm, int TERMS = 1>
__global__ __launch_bounds__(256) void ds_from_logits_kernel(DsArgs<TIN> p, const float* x, int64_t xtok, int nrows, bool exact) {
  static_assert(sizeof(TIN) == 2 && Perm::GV % 64 == 0, "16-bit d_logits, groups of the vocabulary order in multiples of 64 rows");
  constexpr int U = 4;
  const int tid = threadIdx.x, c = tid & 7;
  const int64_t u0 = (int64_t)blockIdx.x * 64;   // first of this workgroup's 64 columns of dS
  const int64_t g0 = u0 - u0 % Perm::GV;         // first row (= first column) of their group of the vocabulary order
  const int Tc = (int)(p.n_rows ? (int64_t)*p.n_rows : p.T);
  const int used = exact ? Tc : Tc <= 64 ? 128 : (Tc + 63) / 64 * 64, end = used < nrows ? used : nrows;
  // columns c * 8 + (0..3) and c * 8 + (4..7) of the workgroup's 64 are two runs of four consecutive vocabulary rows
  // (both orders Perm keep what one lane of a d_logits tile holds together: four consecutive rows per register quad),
  // and the cache is padded to whole groups, so each run is one aligned 16-byte load
  int r0[2];  // vocabulary row relative to the group's first
  bool live[2];
#pragma unroll
  for (int hf = 0; hf < 2; ++hf) {
    r0[hf] = (int)(Perm::vocab_at(u0 + c * 8 + 4 * hf) - g0);
    live[hf] = g0 + r0[hf] < p.vrows;
  }
  for (int base = tid >> 3; base < end; base += 32 * U) {
    int tok[U];
    f32x4_t k[U], v[U][2];
    int rel[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int pos = base + 32 * u;
      const bool on = pos < Tc;
      tok[u] = on ? (p.rows ? p.rows[pos] : pos) : -1;
      k[u] = on ? p.tokc[pos] : f32x4_t{0.f, 0.f, 0.f, 0.f};
      const int y = on ? p.tokl[pos] : -1;
      rel[u] = (p.label_outside != 1 && y >= p.lab0 + g0 && y < p.lab0 + g0 + Perm::GV) ? (int)(y - p.lab0 - g0) : -1;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        v[u][hf] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (tok[u] >= 0 && live[hf]) v[u][hf] = load_vec<true>(reinterpret_cast<const f32x4_t*>(kept_logit(x, xtok, tok[u], g0 + r0[hf])));
      }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int pos = base + 32 * u;
      float d[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int row = r0[e >> 2] + (e & 3);
        const bool dead = tok[u] < 0 || g0 + row >= p.vrows;
        d[e] = dlogit<true>(dead ? 0.f : v[u][e >> 2][e & 3], p.c, k[u][0], k[u][1], k[u][2], k[u][3], row == rel[u], dead, p.label_outside == 2);
      }
      if (pos >= end) continue;
      TIN* dst = ds_at(p.dS, p.ldS, p.pcol, pos, u0 + c * 8);
      if constexpr (TERMS == 6) store_planes<TIN, 8>(dst, p.dS_plane, d);
      else store_run<TIN, 8>(dst, d);
    }
  }
}

}  // namespace lce
