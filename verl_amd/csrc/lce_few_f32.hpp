// Host side of few_tokens_f32.hpp: the backward of fp32 inputs with at most 255 tokens, and the forward of 129 to 255.
#pragma once
#include "few_tokens_f32.hpp"
#include "lce_host.hpp"

namespace {

struct FewF32Layout {
  int64_t vchunk, pcol;
  int nchunks, ksplit, nt;  // nt: token positions of the kernels
  size_t off_dS, off_dHacc, off_rows, off_inv, off_nrows, off_acounts, off_tokc, off_tokl, total;
};

// Which calls: shapes and diagnostic settings alone.  Measured, forward + backward in ms (the forward is the same), tiles of 256 x 256
// with transposed copies of W / this way, H=3584, V=152064: 1 token 7.6 / 1.57, 32: 7.8 / 1.74, 64: 8.2 / 2.7, 100: 8.7 / 4.5, 128:
// 8.8 / 4.6; H=896: 2.7 / 0.47, 2.8 / 0.50, 3.0 / 0.80, 3.1 / 1.31, 3.1 / 1.36; without d_weight, H=3584, 16 tokens 6.4 / 1.32.
// With the forward's logits (few_f32_cache_bytes): H=3584, 12 tokens 1.59 -> 1.18, 64: 2.59 -> 1.94, 128: 4.58 -> 3.38; H=896, 1: 0.43 -> 0.33, 100:
// 1.26 -> 0.96; without d_weight, H=5120, 19: 1.82 -> 1.20.  Error
// against float64 (2-norm; H=896, V=151936, 64 tokens): d_hidden 3.8e-6 / 3.8e-6, d_weight 1.2e-7 / 4.2e-8.  From 129 tokens on the
// registers, half of which hold the products of 128 positions, ask for two groups of positions in the forward and in d_hidden, which
// read W twice; d_weight keeps 32 columns of hidden a wave instead of 64 and takes them at once.  Against the tiles (which do not keep
// logits), forward + backward, us: H=896, 129 tokens 3490 -> 1285, 160: 3499 -> 1347, 255: 3532 -> 2061; H=3584, 129: 11162 -> 4263, 192: 11242 ->
// 5221, 255: 11372 -> 6746; H=5120, 255: 16409 -> 9839; d_hidden alone, H=4096, 255: 7658 -> 4329; forward alone, H=3584, 129: 2541 -> 1598, 200:
// 2544 -> 2151, 255: 2542 -> 2433; H=896, 255: level.  Error of d_hidden against float64: 200 tokens, H=896, 1.03e-6 / 6.7e-7, H=3584 1.37e-6 /
// 1.15e-6.  From 256 on the planes run (H=3584: 6.0 ms), with large vocabularies.
constexpr int64_t kFewF32Tokens = LCE_F32_FEW_TOKENS;
static_assert(kFewF32Tokens <= kFewF32Rows, "rows of hidden behind one descriptor");
bool few_f32(const Tuning& tu, int64_t T) { return T <= kFewF32Tokens && !tu.variant_forced && tu.few_token_gemms && !tu.split_bwd; }

// bytes of the logits that a forward of so few tokens keeps where it is handed the buffer
size_t few_f32_cache_bytes(int64_t T, int64_t H, int64_t V) {
  return T >= 1 && T <= kFewF32Tokens && T <= H && V > 0 ? (size_t)T * (size_t)logits_cache_row(V) * 4 : 0;
}

FewF32Layout few_f32_layout_for(const Tuning& tu, int64_t T, int64_t H, int64_t V, int64_t vchunk) {
  FewF32Layout L;
  L.nt = (int)round_up(T, 32);
  L.vchunk = std::min(round_up(vchunk, 256), round_up(V, 256));
  L.nchunks = (int)((V + L.vchunk - 1) / L.vchunk);
  L.pcol = (int64_t)L.nt * 32 + 32;
  // K slices of d_hidden: its workgroups fill the chip once, one to a CU, and twice from 129 tokens on, where the tiles summed fewer rows
  // at a time too; at least 256 rows of W per slice
  const int64_t n_ht = (H + 255) / 256, fill = std::max<int64_t>(1, (T > 128 ? 2 : 1) * kNumCUs / n_ht);
  L.ksplit = tu.dh_ksplit > 0 ? tu.dh_ksplit : (int)std::min(fill, std::max<int64_t>(1, L.vchunk / 256));
  size_t o = 0;
  L.off_dS = o;      o += align256((size_t)(L.vchunk / 32) * L.pcol * 4);
  L.off_dHacc = o;   o += (size_t)L.ksplit * align256((size_t)T * H * 4);
  L.off_rows = o;    o += align256((size_t)L.nt * 4);
  L.off_inv = o;     o += align256((size_t)T * 4);
  L.off_nrows = o;   o += 256;
  L.off_acounts = o; o += 256;
  L.off_tokc = o;    o += align256((size_t)L.nt * 16);
  L.off_tokl = o;    o += align256((size_t)L.nt * 4);
  L.total = o;
  return L;
}

// one chunk where the bound of bwd_layout (a quarter of one [T, V] plus one fp32 [V, H]) or the budget has room for it
FewF32Layout few_f32_layout(const Tuning& tu, int64_t T, int64_t H, int64_t V, int64_t vchunk) {
  if (vchunk <= 0) {
    double gate = (double)T * V + 4.0 * (double)V * H;
    if (tu.ws_budget > 0 && (double)tu.ws_budget < gate) gate = (double)tu.ws_budget;
    vchunk = round_up(V, 256);
    while (vchunk > 2048 && (double)few_f32_layout_for(tu, T, H, V, vchunk).total + 512.0 > gate) vchunk -= 1024;
    if (vchunk < 2048) vchunk = 2048;
    const int64_t n = (V + vchunk - 1) / vchunk;
    vchunk = round_up((V + n - 1) / n, 256);
  }
  return few_f32_layout_for(tu, T, H, V, vchunk);
}

#if defined(LCE_TU_DTYPE) && LCE_TU_DTYPE == 1 && LCE_TU_PART == 1
// d_logits (unless they are there) and d_hidden of one chunk, positions q.first .. + NT
template <int NT>
int launch_few_f32_group(FewF32Args q, bool need_ds, bool need_dh, hipStream_t st) {
  int rc;
  if (need_ds) {
    typedef FewFwdShape<float, NT> S;
    ProfScope prof(PC_BWD_DS, st);
    q.span = round_up((q.vrows + kNumCUs - 1) / kNumCUs, 32);
    allow_lds(lce_ds_few_f32_kernel<NT>, S::LDS_BYTES);
    hipLaunchKernelGGL(lce_ds_few_f32_kernel<NT>, dim3((unsigned)((q.vrows + q.span - 1) / q.span)), dim3(512), S::LDS_BYTES, st, q);
    if ((rc = check_launch("lce_ds_few_f32_kernel"))) return rc;
  }
  if (need_dh) {
    typedef FewDhF32Shape<NT> S;
    ProfScope prof(PC_GEMM_DH, st);
    q.kslice = round_up((q.vrows + q.ksplit - 1) / q.ksplit, 32);
    allow_lds(lce_dh_few_f32_kernel<NT>, S::LDS_BYTES);
    hipLaunchKernelGGL(lce_dh_few_f32_kernel<NT>, dim3((unsigned)((q.H + S::HW - 1) / S::HW * q.ksplit)), dim3(512), S::LDS_BYTES, st, q);
    if ((rc = check_launch("lce_dh_few_f32_kernel"))) return rc;
  }
  return LCE_OK;
}

template <int KT>
int launch_dw_few_f32(FewF32Args q, hipStream_t st) {
  typedef FewDwF32Shape<KT> S;
  ProfScope prof(PC_GEMM_DW, st);
  const int64_t n_ht = (q.H + S::HW - 1) / S::HW;
  q.n_su = (int)std::max<int64_t>(1, std::min<int64_t>(kNumCUs / n_ht, (q.vrows + 31) / 32));
  allow_lds(lce_dw_few_f32_kernel<KT>, S::LDS_BYTES);
  hipLaunchKernelGGL(lce_dw_few_f32_kernel<KT>, dim3((unsigned)round_up(n_ht * q.n_su, 8)), dim3(512), S::LDS_BYTES, st, q);
  return check_launch("lce_dw_few_f32_kernel");
}

// d_logits, d_hidden and d_weight of one chunk, nt positions (a multiple of 32)
int launch_few_f32(FewF32Args q, int nt, bool need_dh, bool need_dw, hipStream_t st, const float* x) {
  int rc;
  if (x) {
    ProfScope prof(PC_BWD_DS, st);
    hipLaunchKernelGGL(ds_few_f32_from_logits_kernel, dim3((unsigned)((q.vrows + 31) / 32)), dim3(256), 0, st, q, x);
    if ((rc = check_launch("ds_few_f32_from_logits_kernel"))) return rc;
  }
  for (int first = 0; first < nt && (need_dh || !x); first += 128) {
    FewF32Args g = q;
    g.first = first;
    g.most = std::min(128, nt - first);
    g.dS += first * 32; g.tokc += first; g.tokl += first; g.rows += first; g.dHp += (int64_t)first * q.H;
    rc = g.most == 32 ? launch_few_f32_group<32>(g, !x, need_dh, st) : g.most == 64 ? launch_few_f32_group<64>(g, !x, need_dh, st)
       : g.most == 96 ? launch_few_f32_group<96>(g, !x, need_dh, st) : launch_few_f32_group<128>(g, !x, need_dh, st);
    if (rc) return rc;
  }
  if (!need_dw) return LCE_OK;
  return nt == 32 ? launch_dw_few_f32<32>(q, st) : nt == 64 ? launch_dw_few_f32<64>(q, st) : nt == 96 ? launch_dw_few_f32<96>(q, st)
       : nt == 128 ? launch_dw_few_f32<128>(q, st) : nt <= 192 ? launch_dw_few_f32<192>(q, st) : launch_dw_few_f32<256>(q, st);
}

int backward_few_f32(const float* h, int64_t ldh, const float* W, int64_t ldw, const int64_t* labels, int64_t T, int64_t H, int64_t V, float temperature,
                     int reduction, const float* maximum, const float* accumulate, const float* entropy_b, const float* dlogprobs, const float* dentropy,
                     float* d_hidden, float* d_weight, char* ws, int64_t vchunk, hipStream_t st, int64_t vocab_offset, const Tuning& tu,
                     const float* xcache) {
  const FewF32Layout L = few_f32_layout(tu, T, H, V, vchunk);
  int* rows = reinterpret_cast<int*>(ws + L.off_rows);
  int* inv = reinterpret_cast<int*>(ws + L.off_inv);
  int* n_rows = reinterpret_cast<int*>(ws + L.off_nrows);
  int* acounts = reinterpret_cast<int*>(ws + L.off_acounts);
  const int64_t g_stride = reduction == LCE_REDUCTION_NONE ? 1 : 0, part_stride = (int64_t)(align256((size_t)T * H * 4) / 4);
  FewF32Args q = {};
  q.ldw = ldw; q.H = H; q.h = h; q.ldh = ldh; q.T = T; q.rows = rows; q.n_rows = n_rows;
  q.dS = reinterpret_cast<float*>(ws + L.off_dS); q.pcol = L.pcol;
  f32x4_t* tokc = reinterpret_cast<f32x4_t*>(ws + L.off_tokc);
  int* tokl = reinterpret_cast<int*>(ws + L.off_tokl);
  q.tokc = tokc; q.tokl = tokl; q.c = kLog2e / temperature;
  q.dHp = reinterpret_cast<float*>(ws + L.off_dHacc); q.part_stride = part_stride; q.ksplit = L.ksplit;
  q.first = 0; q.most = (int)T;
  int rc;
  {
    ProfScope prof(PC_ACTIVE_ROWS, st);
    hipLaunchKernelGGL(active_count_kernel, dim3(1), dim3(256), 0, st, dlogprobs, g_stride, dentropy, T, acounts);
    if ((rc = check_launch("active_count_kernel"))) return rc;
    hipLaunchKernelGGL(active_rows_kernel, dim3(1), dim3(256), 0, st, dlogprobs, g_stride, dentropy, T, acounts, rows, inv, n_rows);
    if ((rc = check_launch("active_rows_kernel"))) return rc;
    hipLaunchKernelGGL(ds_token_consts_kernel, dim3(1), dim3(256), 0, st, rows, n_rows, T, (int64_t)L.nt, dlogprobs, g_stride,
                       reduction == LCE_REDUCTION_MEAN ? 1.0f / (float)T : 1.0f, dentropy, maximum, accumulate, entropy_b, labels, vocab_offset, V,
                       1.0f / temperature, tokc, tokl);
    if ((rc = check_launch("ds_token_consts_kernel"))) return rc;
  }
  for (int c = 0; c < L.nchunks; ++c) {
    const int64_t v0 = (int64_t)c * L.vchunk;
    q.W = W + v0 * ldw; q.vrows = std::min(L.vchunk, V - v0); q.lab0 = v0;
    q.accumulate = c > 0;
    q.dW = d_weight ? d_weight + v0 * H : nullptr;
    const bool dh = d_hidden != nullptr, dw = d_weight != nullptr;
    const float* x = xcache ? xcache + v0 * T : nullptr;
    rc = launch_few_f32(q, L.nt, dh, dw, st, x);
    if (rc) return rc;
  }
  if (!d_hidden) return LCE_OK;
  ProfScope prof(PC_DH_FINISH, st);
  LabelTerm lt;
  lt.labels = nullptr; lt.v0 = vocab_offset; lt.V = V; lt.g_lp = dlogprobs; lt.g_stride = g_stride; lt.scale = 0.f;
  const int64_t blocks = (T * (H / 4) + 255) / 256;
  auto finish = dh_sum_deep(L.ksplit, blocks) ? dh_finish_kernel<float, float, true> : dh_finish_kernel<float, float, false>;
  hipLaunchKernelGGL(finish, dim3((unsigned)blocks), dim3(256), 0, st, q.dHp, L.ksplit, part_stride, inv, T, H, d_hidden, lt, W, ldw);
  return check_launch("dh_finish_kernel");
}
#endif

#if defined(LCE_TU_DTYPE) && LCE_TU_DTYPE == 1 && LCE_TU_PART == 0
// 129 to 255 tokens as two groups, W read twice (a tile of 256 x 256 takes what 256 tokens take).
int forward_few_twice(const float* h, int64_t ldh, const float* W, int64_t ldw, const int64_t* labels, int64_t T, int64_t H, int64_t V, float temperature,
                      int reduction, float* logprobs, float* entropy, float* maximum, float* accumulate, float* entropy_b, char* ws, size_t ws_bytes,
                      hipStream_t st, int64_t label_offset, float* shard_out, int max_splits, float* xcache) {
  // (one workspace after the other in the same place; what is left of it sets the number of splits)
  const size_t lp_at = (ws_bytes - align256((size_t)T * 4)) / 256 * 256;
  const int64_t most = ((int64_t)lp_at - 1024) / (128 * 16);
  if (most < 1) return fail(LCE_E_WORKSPACE, "forward workspace too small: %zu", ws_bytes);
  max_splits = (int)std::min<int64_t>(max_splits, most);
  float* lp = reduction == LCE_REDUCTION_NONE ? logprobs : reinterpret_cast<float*>(ws + lp_at);
  for (int64_t t0 = 0; t0 < T; t0 += 128) {
    const int64_t n = std::min<int64_t>(128, T - t0);
    auto group = [&](auto nt) {
      return forward_few<float, decltype(nt)::value>(h + t0 * ldh, ldh, W, ldw, labels + t0, n, H, V, temperature, LCE_REDUCTION_NONE, lp + t0, entropy + t0,
                                                     maximum + t0, accumulate + t0, entropy_b + t0, ws, st, label_offset,
                                                     shard_out ? shard_out + 4 * t0 : nullptr, max_splits, xcache ? xcache + t0 * 16 : nullptr, T);
    };
    const int rc = n <= 32 ? group(std::integral_constant<int, 32>{}) : n <= 64 ? group(std::integral_constant<int, 64>{})
                 : n <= 96 ? group(std::integral_constant<int, 96>{}) : group(std::integral_constant<int, 128>{});
    if (rc) return rc;
  }
  if (shard_out || reduction == LCE_REDUCTION_NONE) return LCE_OK;
  hipLaunchKernelGGL(lce_reduce_sum_kernel, dim3(1), dim3(1024), 0, st, lp, T, reduction == LCE_REDUCTION_MEAN ? 1.0f / (float)T : 1.0f, logprobs);
  return check_launch("lce_reduce_sum_kernel");
}
#endif

}  // namespace
