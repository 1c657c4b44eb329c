// fp32 inputs with at most 255 tokens: the backward as three streams, as in few_tokens.hpp, on the fp32 MFMA (from 129 on the first two
// in two groups of positions):
//   d_logits    reads W once (the forward's products again), or the logits that the forward kept, and writes [T, V]
//   d_hidden    reads W once
//   d_weight    writes [V, H] once
// fp32 needs no transposing reads: v_mfma_f32_32x32x2_f32 takes one element per lane of either operand, so that a K-major operand
// is read from LDS as it lies, 32 neighbours at a time.  Everything is in natural order.
#pragma once
#include "few_tokens.hpp"

namespace lce {

// An offset beyond ONE descriptor over all rows of hidden: with 255 rows of up to 16 MiB (lce_abi.hip, check_common) that spans more than
// the 2 GiB which kBufNowhere lies beyond.  Nothing is added to it but the 16 bytes of a load.
constexpr int kFewF32Rows = 255;
constexpr int kFewF32Nowhere = (int)0xff000000u;
static_assert(kFewF32Rows * ((int64_t)16 << 20) <= (int64_t)0xff000000u, "beyond the last row of hidden");

// d_logits lie in panels of 32 columns, [panel][token position][32], `pcol` elements from panel to panel.
template <typename P>
LCE_DEV P ds32_at(P dS, int64_t pcol, int64_t t, int64_t v) { return dS + (v >> 5) * pcol + t * 32 + (v & 31); }

struct FewF32Args {
  const float* W;  // first row of the chunk, row stride ldw
  int64_t ldw, vrows, H;
  const float* h;
  int64_t ldh, T;
  const int *rows, *n_rows;  // tokens that take part (null: all T)
  float* dS;
  int64_t pcol;
  const f32x4_t* tokc;  // see DsArgs
  const int* tokl;
  int64_t lab0;
  float c;
  int64_t span;        // d_logits: rows of W per workgroup, a multiple of 32
  float* dHp;          // fp32 partials of d_hidden: slice s at dHp + s * part_stride, [position][H]
  int64_t part_stride, kslice;  // columns of dS per slice, a multiple of 32
  int ksplit, accumulate;       // accumulate: 0 store, 1 add to what is there (second and later chunks)
  float* dW;           // rows of d_weight of this chunk, [vrows][H]
  int n_su;            // d_weight: workgroups side by side along the vocabulary
  int first;           // d_logits and d_hidden: this launch's first position (dS, tokc, tokl, rows and dHp point there)
  int most;            // positions of a launch

  LCE_DEV int tokens() const {
    const int t = (int)T, all = n_rows && *n_rows < t ? *n_rows : t, n = all - first;
    return n < 0 ? 0 : n < most ? n : most;
  }
};

// d_logits: the forward's products, and each pass's 32 rows x NT positions of a wave as one panel.  Bound by the read of W, from some
// 40 tokens on by the fp32 MFMA.  Kernels alone, H=3584, V=152064 (2.18 GB), 16 / 64 / 128 tokens, us: d_logits 500 / 739 / 1232,
// d_hidden 430 / 626 / 1044, d_weight 373 (5.9 TB/s) / 654 / 1078; the fp32 MFMA's peak rate is 222 / 445 / 890 for the padded tokens.
template <int NT>
__global__ __launch_bounds__(512, 2) void lce_ds_few_f32_kernel(FewF32Args p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  typedef FewFwdShape<float, NT> S;
  constexpr int FN = S::FN, HL = S::HROWS / 64;
  const int tid = threadIdx.x, lane = tid & 63, hh = lane >> 5, ln = lane & 31;
  const int64_t row0 = (int64_t)blockIdx.x * p.span;
  const int64_t vend64 = row0 + p.span < p.vrows ? row0 + p.span : p.vrows;
  const int n = p.tokens();
  if (n == 0) return;  // (nobody reads positions beyond the tokens)
  uint32_t h_off[HL];
#pragma unroll
  for (int i = 0; i < HL; ++i) {
    const int pos = (tid >> 3) + 64 * i;
    h_off[i] = pos < n ? (uint32_t)((p.rows ? (int64_t)p.rows[pos] : pos) * p.ldh * 4) + (tid & 7) * 16 : (uint32_t)kFewF32Nowhere;
  }
  f32x4_t k[FN];
  int lab[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    k[j] = p.tokc[j * 32 + ln];
    lab[j] = p.tokl[j * 32 + ln] - (int)p.lab0;
  }
  few_products<float, NT, kBufNonTemporal, false>(p.W, p.ldw, row0, vend64, p.H, p.h, p.T * p.ldh * 4, h_off, lds,
                                           [&](f32x16_t (&acc)[1][FN], int64_t, int vbase, bool busy) {
    if (!busy) return;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if (j * 32 >= n) break;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4_t d;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int v = vbase + 8 * q + 4 * hh + r;
          d[r] = dlogit<true>(acc[0][j][4 * q + r], p.c, k[j][0], k[j][1], k[j][2], k[j][3], v == lab[j], v >= p.vrows, false);
        }
        *reinterpret_cast<f32x4_t*>(ds32_at(p.dS, p.pcol, j * 32 + ln, vbase + 8 * q + 4 * hh)) = d;
      }
    }
  });
}

// The same from logits that the forward kept (FwdArgs::xcache), x from the chunk's first row on: a workgroup per panel, eight lanes to a
// position.  The same expressions, so the same bits.  Bound by HBM: 4 bytes read and 4 written per logit instead of a read of W.
inline __global__ __launch_bounds__(256) void ds_few_f32_from_logits_kernel(FewF32Args p, const float* x) {
  const int n = p.tokens(), v = 4 * (threadIdx.x & 7);
  const int64_t u0 = (int64_t)blockIdx.x * 32;
  for (int pos = threadIdx.x >> 3; pos < n; pos += 32) {
    const f32x4_t k = p.tokc[pos];
    const int64_t lab = p.tokl[pos] - p.lab0;
    const f32x4_t z = load_vec<true>(reinterpret_cast<const f32x4_t*>(kept_logit(x, p.T, p.rows ? (int64_t)p.rows[pos] : pos, u0 + v)));
    f32x4_t d;
#pragma unroll
    for (int r = 0; r < 4; ++r) d[r] = dlogit<true>(z[r], p.c, k[0], k[1], k[2], k[3], u0 + v + r == lab, u0 + v + r >= p.vrows, false);
    *reinterpret_cast<f32x4_t*>(ds32_at(p.dS, p.pcol, pos, u0 + v)) = d;
  }
}

// d_hidden.  Workgroup = 512 threads = 8 waves, one per CU; it owns columns [h0, h0 + 256) of the result for all positions and one K
// slice of the chunk; wave w multiplies columns h0 + 32 w .. +31:  C[m = h][n = t] = sum_v W[v][h] dS[t][v].  A stage is 32 rows
// of W (1 KB of each) and one panel of dS; DEPTH stages on their way in registers, two in LDS, one barrier each.
template <int NT>
struct FewDhF32Shape {
  static constexpr int HW = 256, DEPTH = 4, ROWS = (NT + 63) / 64 * 64;
  static constexpr int STAGE = 32 * HW * 4 + ROWS * 128, LDS_BYTES = 2 * STAGE;
};

template <int NT>
__global__ __launch_bounds__(512, 2) void lce_dh_few_f32_kernel(FewF32Args p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  typedef FewDhF32Shape<NT> S;
  constexpr int HW = S::HW, DEPTH = S::DEPTH, FN = NT / 32, WL = 4, BL = S::ROWS / 64;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, hh = lane >> 5, ln = lane & 31;
  const int n_ht = (int)((p.H + HW - 1) / HW);
  const int ht = blockIdx.x % n_ht, s = blockIdx.x / n_ht;
  const int64_t h0 = (int64_t)ht * HW;
  const int64_t k_begin = (int64_t)s * p.kslice, k_left = p.vrows - k_begin;
  const int n_st = k_left <= 0 ? 0 : (int)(((k_left < p.kslice ? k_left : p.kslice) + 31) / 32);  // stages
  const int n = p.tokens();
  if (n == 0) return;  // (nobody reads partials of positions beyond the tokens)
  f32x16_t acc[FN];
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;
  // 16-byte chunk tid % 64 of row tid / 64 + 8 i; rows beyond the chunk and columns beyond H read as zero
  const int ch = tid & 63, r0 = tid >> 6;
  int w_at[WL];
#pragma unroll
  for (int i = 0; i < WL; ++i) w_at[i] = h0 + ch * 4 < p.H ? (int)(((r0 + 8 * i) * p.ldw + h0 + ch * 4) * 4) : kBufNowhere;
  u32x4_t pw[DEPTH][WL], pb[DEPTH][BL];
  auto fetch = [&](u32x4_t (&w)[WL], u32x4_t (&b)[BL], int st) {
    const bool live = st < n_st;  // (stages behind the last one read as zero)
    const int64_t k0 = k_begin + 32 * (int64_t)(live ? st : 0), left = p.vrows - k0 < 32 ? p.vrows - k0 : 32;
    const buf_t wb = make_buf(p.W + k0 * p.ldw, live ? left * p.ldw * 4 : 0);
#pragma unroll
    for (int i = 0; i < WL; ++i) w[i] = __builtin_amdgcn_raw_buffer_load_b128(wb, w_at[i], 0, kBufNonTemporal);
    const buf_t panel = make_buf(ds32_at(p.dS, p.pcol, 0, k0), live ? n * 128 : 0);
#pragma unroll
    for (int i = 0; i < BL; ++i) b[i] = __builtin_amdgcn_raw_buffer_load_b128(panel, tid * 16 + i * 8192, 0, 0);
    __builtin_amdgcn_sched_barrier(0);  // (the loads of one stage stay in front of the next one's)
  };
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) fetch(pw[d], pb[d], d);
  int buf = 0;
  for (int st0 = 0; st0 < n_st; st0 += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      char* sA = lds + buf * S::STAGE;  // 32 rows x 1 KB, chunk c of row r at c ^ 8 ((r / 4) % 2): the two halves of a wave read rows 4 apart
      char* sB = sA + 32 * HW * 4;      // positions x 128 bytes, chunk c of row t at c ^ ((t / 2) % 8)
      buf ^= 1;
#pragma unroll
      for (int i = 0; i < WL; ++i) {
        const int r = r0 + 8 * i;
        *reinterpret_cast<u32x4_t*>(sA + r * (HW * 4) + ((ch ^ (((r >> 2) & 1) << 3)) * 16)) = pw[d][i];
      }
#pragma unroll
      for (int i = 0; i < BL; ++i) {
        const int at = tid + i * 512, t = at >> 3, c = at & 7;
        *reinterpret_cast<u32x4_t*>(sB + t * 128 + ((c ^ ((t >> 1) & 7)) * 16)) = pb[d][i];
      }
      fetch(pw[d], pb[d], st0 + d + DEPTH);
      // (a buffer is written again two stages on: every wave has passed the barrier between, after its reads of this stage)
      __syncthreads();
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        // rows 8 q + 4 hh + i of this half of the wave, i = 0..3
        f32x4_t b[FN];
        float a[4];
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const int t = 32 * j + ln, c = 2 * q + hh;
          b[j] = *reinterpret_cast<const f32x4_t*>(sB + t * 128 + ((c ^ ((t >> 1) & 7)) * 16));
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 8 * q + 4 * hh + i, byte = (32 * wave + ln) * 4;
          a[i] = *reinterpret_cast<const float*>(sA + r * (HW * 4) + (byte ^ (((r >> 2) & 1) << 7)));
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j][i], acc[j], 0, 0, 0);
      }
    }
  }
  // this lane: h = h0 + 32 wave + 8 q + 4 hh + (0..3) of position 32 j + ln
  float* out = p.dHp + (int64_t)s * p.part_stride;
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int t = 32 * j + ln;
    if (t >= n) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int64_t hc = h0 + 32 * wave + 8 * q + 4 * hh;
      if (hc >= p.H) continue;  // (H is a multiple of 4)
      float* dst = out + (int64_t)t * p.H + hc;
      f32x4_t v = {acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]};
      if (p.accumulate) v += *reinterpret_cast<const f32x4_t*>(dst);
      *reinterpret_cast<f32x4_t*>(dst) = v;
    }
  }
}

// d_weight.  Workgroup = 512 threads = 8 waves, one per CU; a wave keeps hidden of its 64 columns in registers as MFMA operands and the
// workgroup walks the panels id / n_ht, id / n_ht + n_su, ... of dS:  C[m = v][n = h] = sum_t dS[t][v] hidden[t][h].  A lane holds one
// column of 16 rows, 32 lanes a whole line of a row, so the results are stored as they lie.
// (Beyond 128 positions it is 32 of its columns instead of 64: the same registers.)
template <int KT>
struct FewDwF32Shape {
  static constexpr int NB = KT > 128 ? 1 : 2, HW = 256 * NB, TILE = (KT + 63) / 64 * 64 * 128, LDS_BYTES = 2 * TILE;
};

template <int KT>
__global__ __launch_bounds__(512, 2) void lce_dw_few_f32_kernel(FewF32Args p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  typedef FewDwF32Shape<KT> S;
  constexpr int HW = S::HW, KP = KT / 2, BL = S::TILE / 8192, NB = S::NB;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, hh = lane >> 5, ln = lane & 31;
  const int n_ht = (int)((p.H + HW - 1) / HW);
  const int id = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);  // (as in lce_dw_few_kernel)
  if (id >= n_ht * p.n_su) return;
  const int64_t h0 = (int64_t)(id % n_ht) * HW, hw = h0 + 32 * NB * wave;
  const int64_t n_pan = (p.vrows + 31) / 32;
  const int n = p.tokens();
  u32x4_t pre[BL];
  auto fetch = [&](int64_t pan) {
    const buf_t panel = make_buf(p.dS + pan * p.pcol, n * 128);  // positions beyond the tokens read as zero
#pragma unroll
    for (int i = 0; i < BL; ++i) pre[i] = __builtin_amdgcn_raw_buffer_load_b128(panel, tid * 16 + i * 8192, 0, 0);
  };
  auto stash = [&](char* to) {
#pragma unroll
    for (int i = 0; i < BL; ++i) *reinterpret_cast<u32x4_t*>(to + tid * 16 + i * 8192) = pre[i];
  };
  int64_t pan = id / n_ht;
  const int64_t last = pan + (n_pan - 1 - pan) / p.n_su * p.n_su;
  fetch(pan);
  float hf[KP][NB];  // position 2 kp + hh, column hw + 32 x + ln
  const buf_t hid = make_buf(p.h, p.T * p.ldh * 4);
#pragma unroll
  for (int kp = 0; kp < KP; ++kp) {
    const int pos = 2 * kp + hh;
    const int64_t tok = pos < n ? (p.rows ? (int64_t)p.rows[pos] : pos) : -1;
#pragma unroll
    for (int x = 0; x < NB; ++x) {
      const int64_t col = hw + 32 * x + ln;
      hf[kp][x] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(hid, tok >= 0 && col < p.H ? (int)((tok * p.ldh + col) * 4) : kFewF32Nowhere, 0, 0));
    }
  }
  stash(lds);
  fetch(pan < last ? pan + p.n_su : pan);
  const bool live = hw < p.H;
  // (as many dropped stores as a turn of the loop issues behind its fetch, as in lce_dw_few_kernel)
#pragma unroll
  for (int k = 0; k < 16 * NB; ++k) __builtin_amdgcn_raw_buffer_store_b32(0u, make_buf(p.dW, 0), kBufNowhere + 4 * k, 0, 0);
  for (int buf = 0; pan <= last; pan += p.n_su, buf ^= 1) {
    __syncthreads();  // this panel is in LDS, and every wave is done with the other buffer
    const char* tA = lds + buf * S::TILE;
    f32x16_t acc[NB];
#pragma unroll
    for (int x = 0; x < NB; ++x)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[x][r] = 0.f;
    if (live) {
#pragma unroll
      for (int g = 0; g < KP / 8; ++g) {
        float a[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) a[i] = *reinterpret_cast<const float*>(tA + (2 * (8 * g + i) + hh) * 128 + ln * 4);
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int x = 0; x < NB; ++x) acc[x] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], hf[8 * g + i][x], acc[x], 0, 0, 0);
        if (16 * (g + 1) >= n) break;
      }
    }
    stash(lds + (buf ^ 1) * S::TILE);  // (behind the last panel: the last one again)
    fetch(pan + 2 * p.n_su <= last ? pan + 2 * p.n_su : last);
    const int64_t v0 = pan * 32, left = p.vrows - v0 < 32 ? p.vrows - v0 : 32;
    const buf_t out = make_buf(p.dW + v0 * p.H, left * p.H * 4);
#pragma unroll
    for (int x = 0; x < NB; ++x) {
      const int64_t col = hw + 32 * x + ln;
      const int at = live && col < p.H ? (int)((4 * hh * p.H + col) * 4) : kBufNowhere;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = 8 * (r >> 2) + (r & 3);
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, (float)acc[x][r]), out, at == kBufNowhere ? at : at + (int)(row * p.H * 4), 0, kBufNonTemporal);
      }
    }
  }
}

}  // namespace lce
