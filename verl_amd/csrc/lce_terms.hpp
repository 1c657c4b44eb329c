// fp32 inputs on the bfloat16 matrix pipe: every operand is held as three bfloat16 planes whose sum it is, and a K slab is
// multiplied as six products of planes (GemmCfg16, TERMS == 6).  The fp32 MFMA runs at 157 TFLOP/s dense, the bfloat16 one
// at 2.5 PFLOP/s; six products for one leave 2.5 times the rate at the clocks both reach, against which stand the passes
// that make the planes (10 bytes per element of W, forward and backward each).  Measured, fp32 MFMA / planes: H=896,
// V=151936, 1024 tokens forward + backward 9.90 / 4.30 ms (logits kept), 2000 tokens forward 4.11 / 2.23, 400 tokens forward 1.09 / 0.75;
// H=5120, 1500 tokens, half with gradient 56.6 / 26.8.  Error against float64 (2-norm, relative; H=896, V=151936, 2000 tokens):
// log-probs 7.7e-8 / 7.2e-8, entropies 5.9e-8 / 5.6e-8, d_hidden 1.0e-6 / 5.9e-7, d_weight 7.9e-7 / 4.1e-7: the products are
// exact and a sixteenth as many partial sums are rounded.
#pragma once
#include "lce_host.hpp"

namespace {

// ---- forward ----------------------------------------------------------------------------------
// The weight is split and multiplied chunk by chunk; a chunk's splits are a block of their own in the list of partial statistics.
struct TermsFwdPlan {
  int64_t rows;     // vocabulary rows of a chunk
  int nchunks, splits;  // splits: of all chunks together
  size_t off_xlabel, off_lp, off_wide, off_h, off_w, total;
};

int terms_fwd_splits(int ntt, int64_t rows) { return forward_splits_256(ntt, (int)((rows + 255) / 256)); }

TermsFwdPlan terms_fwd_plan_for(int64_t T, int64_t H, int64_t V, int64_t tiles) {  // tiles: of 256 vocabulary rows, in a chunk
  TermsFwdPlan p;
  const int ntt = (int)((T + 255) / 256);
  p.rows = tiles * 256;
  p.nchunks = (int)((V + p.rows - 1) / p.rows);
  auto splits = [&](int64_t rows) { return std::min<int>(terms_fwd_splits(ntt, rows), (int)((rows + 255) / 256)); };
  p.splits = splits(V - (p.nchunks - 1) * p.rows);
  if (p.nchunks > 1) p.splits += (p.nchunks - 1) * splits(p.rows);
  size_t o = align256((size_t)p.splits * T * 16);
  p.off_xlabel = o; o += align256((size_t)T * 4);
  p.off_lp = o;     o += align256((size_t)T * 4);
  p.off_wide = o;   o += 256;
  p.off_h = o;      o += align256((size_t)round_up(T, 64) * 3 * H * 2);
  p.off_w = o;      o += align256((size_t)std::min<int64_t>(p.rows, round_up(V, 64)) * 3 * H * 2);
  p.total = o;
  return p;
}

// A chunk whose tiles would be half as many as the CUs or fewer is multiplied on tiles of 128 tokens instead of 256, which take 0.55 of the
// time: all chunks of 256 tokens, and with more the last one where few rows are left for it.  Forward, us, 256 tokens: H=896 604 -> 529,
// 3584: 2311 -> 2105, 4096: 2498 -> 2067, 5120: 3362 -> 3051; 1000 tokens of H=896 (eighteen tiles of rows in the last chunk) 1261 -> 1237.
bool terms_fwd_half(int64_t ntt, int64_t rows) { return ntt * ((rows + 255) / 256) <= kNumCUs / 2; }

// The widest chunks that a workspace of `room` bytes has space for, between two bounds that are of shapes alone.  The lower
// one, whose workspace is always enough: 256 MB of planes, which the memory-side cache holds from the split to the product, in
// whole rounds of tiles over the CUs.  Where they hold less than a round (few tokens, a wide weight) the upper one is a round,
// through memory, but at most two fifths of the weight's own bytes.  The same bits whatever the width: a tile is a split of
// its own there.  Forward in us by MiB of workspace, H=5120, V=152064: 300 tokens 260: 10478, 611: 5534, 905: 4391 (taken, a round); 1000 tokens 287: 10632, 489: 7728 (taken, a
// round); H=4096, V=128256: 300 tokens 262: 5869, 616: 3172, 766: 2962 (taken).
TermsFwdPlan terms_fwd_plan(int64_t T, int64_t H, int64_t V, size_t room) {
  const int64_t ntt = (T + 255) / 256, nvt = (V + 255) / 256, tile_bytes = 6 * H * 256;
  const int64_t base = std::max<int64_t>(1, ((int64_t)256 << 20) / tile_bytes);  // tiles of a chunk
  const int64_t rounds = base * ntt / kNumCUs;
  if (rounds > 0) return terms_fwd_plan_for(T, H, V, std::max<int64_t>(1, rounds * kNumCUs / ntt));
  const int64_t share = V * H * 4 * 2 / 5 / tile_bytes;
  // (one tile of tokens is multiplied as two of 128: terms_fwd_half)
  const int64_t most = ntt == 1 ? std::min<int64_t>(kNumCUs / 2, std::max(base, share)) : std::max(base, std::min<int64_t>(kNumCUs / ntt, share));
  // (chunks of one length: a shorter last one would take its round all the same)
  int64_t n = (nvt + most - 1) / most;
  const int64_t n_base = (nvt + base - 1) / base;
  for (;; ++n) {
    const TermsFwdPlan p = terms_fwd_plan_for(T, H, V, (nvt + n - 1) / n);
    if (p.total <= room || n >= n_base) return p;
  }
}

// ---- backward ---------------------------------------------------------------------------------
struct TermsBwdLayout {
  int64_t vchunk, tpad, pcol, plane, ldH;  // plane: elements from plane to plane of a d_logits panel
  size_t off_dS[2], off_W[2], off_H, off_dHacc, off_rows, off_inv, off_nrows, off_acounts, off_tokc, off_tokl, total;
  int nchunks, ksplit;
  bool wide;  // the chunks of kept rows are twice as wide, with twice the K slices and partials of d_hidden (TermsChunks)
};

// upper bound of the workspace: a quarter of one [T, V] plus one fp32 [V, H], or the budget
double terms_gate(const Tuning& tu, int64_t T, int64_t H, int64_t V) {
  const double gate = (double)T * V + 4.0 * (double)V * H;
  return tu.ws_budget > 0 && (double)tu.ws_budget < gate ? (double)tu.ws_budget : gate;
}

TermsBwdLayout terms_bwd_layout_for(const Tuning& tu, int64_t T, int64_t H, int64_t V, int64_t vchunk) {
  TermsBwdLayout L;
  L.vchunk = std::min(round_up(vchunk, 256), round_up(V, 256));
  L.nchunks = (int)((V + L.vchunk - 1) / L.vchunk);
  L.ksplit = tu.dh_ksplit > 0 ? tu.dh_ksplit : dh_ksplit(T, H, L.vchunk);
  L.tpad = round_up(T, 128);
  L.plane = L.tpad * 64;
  L.pcol = 3 * L.plane + 64;
  L.ldH = round_up(H, 256) + 64;
  size_t o = 0;
  // (the two of a kind follow each other without a gap: backward_terms has chunks that take both)
  const bool two = L.nchunks > 1;
  for (int b = 0; b < 2; ++b) { L.off_dS[b] = o; o += b == 0 || two ? (size_t)(L.vchunk / 64) * L.pcol * 2 : 0; }
  o = align256(o);
  for (int b = 0; b < 2; ++b) { L.off_W[b] = o; o += b == 0 || two ? (size_t)L.vchunk * 3 * H * 2 : 0; }
  o = align256(o);
  L.off_H = o;       o += align256((size_t)L.tpad * 3 * L.ldH * 2);
  L.off_rows = o;    o += align256((size_t)L.tpad * 4);
  L.off_inv = o;     o += align256((size_t)T * 4);
  L.off_nrows = o;   o += 256;
  L.off_acounts = o; o += align256((size_t)((T + kActiveBlock - 1) / kActiveBlock) * 4);
  L.off_tokc = o;    o += align256((size_t)L.tpad * 16);
  L.off_tokl = o;    o += align256((size_t)L.tpad * 4);
  L.off_dHacc = o;   o += (size_t)L.ksplit * align256((size_t)T * H * 4);
  // The wide chunks, where a launch is few rounds of tiles and half of the rows at least are kept: forward + backward, us, H=896: 256
  // tokens 1977 -> 1659, 300: 2177 -> 2155, 600: 3225 -> 3011, 1024: 4650 -> 4383 (d_hidden alone 3325 -> 3355), 1500: 6487 -> 6404; five
  // rounds, H=4096, 2000: 26584 -> 26260; from eight rounds on they are level or slower: H=3584, 300: 7906 -> 7976, 600: 10999 -> 11174;
  // H=5120, 1000: 21342 -> 21593; with 45 % of the rows, H=896, 2000: 8791 -> 8909.
  const int64_t h_tile = hidden_tile(H);
  const size_t more = (size_t)L.ksplit * align256((size_t)T * H * 4);
  L.wide = two && L.vchunk >= 4096 && T <= 2 * H && tu.dh_ksplit == 0 && (L.vchunk / 256) * ((H + h_tile - 1) / h_tile) < 6 * kNumCUs &&
           (double)(o + more) + 512.0 <= terms_gate(tu, T, H, V);
  L.total = o + (L.wide ? more : 0);
  return L;
}

// chunk width by the same bound as bwd_layout's (a quarter of one [T, V] plus one fp32 [V, H]); within it a chunk's d_logits
// planes stay within 256 MB
TermsBwdLayout terms_bwd_layout(const Tuning& tu, int64_t T, int64_t H, int64_t V, int64_t vchunk) {
  if (vchunk <= 0) {
    const double gate = terms_gate(tu, T, H, V);
    vchunk = std::min(round_up(V, 256), std::max<int64_t>(2048, (((int64_t)256 << 20) / (6 * T)) / 256 * 256));
    while (vchunk > 2048 && (double)terms_bwd_layout_for(tu, T, H, V, vchunk).total + 512.0 > gate) vchunk -= 1024;
    if (vchunk < 2048) vchunk = 2048;
    const int64_t n = (V + vchunk - 1) / vchunk;
    vchunk = round_up((V + n - 1) / n, 256);
  }
  return terms_bwd_layout_for(tu, T, H, V, vchunk);
}

// ---- which calls ------------------------------------------------------------------------------
// LCE_DTYPE_F32_PLANES gives leave to use them, in forward and backward alike: the backward recomputes the logits, and where a
// token's distribution is peaked the rounding errors of a logit and of the forward's statistics cancel only if both come from
// the same arithmetic.  Measured, worst error of d_hidden against float64 relative to its largest entry (512 tokens, H=1024,
// V=40960, temperature 0.6, weight std 0.1): fp32 MFMA both ways 9.3e-6, planes both ways 7.1e-6, fp32 MFMA in the forward only
// 1.8e-5, planes in the forward only 2.0e-5.  A caller without the workspace for a forward on planes (lce_forward_static) has
// only LCE_DTYPE_F32, the fp32 MFMA in both.  With the leave the rule is one of shapes alone, so that nothing set between the
// two calls can part them: the planes where the default workspace bound has room for them (not for small vocabularies).
constexpr int64_t kTermsMinTokens = 256;
bool use_terms(const Tuning& tu, int64_t T, int64_t H, int64_t V) {
  if (tu.variant_forced || T < kTermsMinTokens || H % 64 != 0) return false;  // (a forced variant: diagnostics)
  return (double)terms_bwd_layout(Tuning(), T, H, V, 0).total + 512.0 <= (double)T * V + 4.0 * (double)V * H;
}

// Kept logits (see logits_cache_max_tokens) of a call on planes: of the first rows of W, as many as are no larger than the weight,
// T * rows * 4 <= V * H * 4: all up to H tokens.  Offered up to 4 H tokens, where they are a quarter of the rows and save 2 %: a kept
// logit is 4 bytes written and read once, a recomputed one 12 H operations, whatever T is.  Forward + backward, recomputed / kept,
// us: H=896, 300 tokens 2620 / 2182, 600: 3868 / 3241, 1024: 5220 / 4674 (7/8 of the rows), 2000: 9480 / 8901, 3500: 16327 / 16031;
// H=3584, 300: 10591 / 8015; H=4096, 2000: 33872 / 27158; d_hidden alone H=5120, 1500: 30957 / 21076.
constexpr int64_t kTermsKeepTokens = 4;  // times H
int64_t terms_kept_rows(int64_t T, int64_t H, int64_t V) { return T <= H ? V : V * H / T / 256 * 256; }
size_t terms_cache_bytes(const Tuning& tu, int64_t T, int64_t H, int64_t V) {
  return T <= kTermsKeepTokens * H && use_terms(tu, T, H, V) ? (size_t)T * (size_t)logits_cache_row(terms_kept_rows(T, H, V)) * 4 : 0;
}

// The chunks of a backward: of the rows whose logits a forward of this shape keeps, then the others.  With the logits at hand the
// first ones' d_logits are a pass of their own, so that both buffers may hold one chunk twice as wide (L.wide): half as many
// launches, each with a last round of tiles.  The last of them, where others follow, is of the usual width, and its products share a
// launch with the d_logits tiles of the first of the others.  The list is one of shapes and settings, whether this call has the logits or
// not: the chunks and their K slices are the order of d_hidden's sums, and whether a forward kept its logits depends on what other
// graphs hold at that moment.  Without them a wide chunk's d_logits tiles are a launch of their own.  That costs such a backward up to 4 %
// (d_hidden alone up to 10 %) against chunks that share their launches, us: H=896, 300 tokens 1825 -> 1905, 600: 2820 -> 2790 (d_hidden alone 2018
// -> 2230), 1024: 3810 -> 3900, 1500: 5240 -> 5415; H=4096, 2000: 24580 -> 25480; with the logits it is the same.
struct TermsChunks {
  struct Chunk {
    int64_t v0, rows;
    int buf;
    bool kept, wide;
  };
  int64_t to[3], width[3];  // the kept rows but the last chunk of them, that chunk, the others: end, rows of a chunk
  int n[3], wide;           // chunks; how many of them, from the first on, are wide
  bool two;
  int count() const { return n[0] + n[1] + n[2]; }
  Chunk at(int c) const {
    const int r = c < n[0] ? 0 : c < n[0] + n[1] ? 1 : 2, first = r == 0 ? 0 : r == 1 ? n[0] : n[0] + n[1];
    const int64_t v0 = (r ? to[r - 1] : 0) + (c - first) * width[r];
    return {v0, std::min(width[r], to[r] - v0), c < wide || !two ? 0 : (c & 1), r < 2, c < wide};
  }
};
TermsChunks terms_chunks(const TermsBwdLayout& L, int64_t T, int64_t H, int64_t V) {
  TermsChunks t;
  const int64_t kept = T <= kTermsKeepTokens * H ? terms_kept_rows(T, H, V) : 0;
  t.two = L.nchunks > 1;
  t.to[1] = kept;
  t.to[0] = kept - (kept < V && t.two ? std::min(kept, L.vchunk) : 0);
  t.to[2] = V;
  for (int r = 0; r < 3; ++r) {
    const int64_t rows = t.to[r] - (r ? t.to[r - 1] : 0), most = r == 0 && L.wide ? 2 * L.vchunk : L.vchunk;
    t.n[r] = (int)((rows + most - 1) / most);
    t.width[r] = t.n[r] > 0 ? round_up((rows + t.n[r] - 1) / t.n[r], 256) : most;
    t.n[r] = (int)((rows + t.width[r] - 1) / t.width[r]);
  }
  t.wide = L.wide ? t.n[0] : 0;
  return t;
}

#if defined(LCE_TU_DTYPE) && LCE_TU_DTYPE == 1
typedef GemmCfg16<bf16_t, 0, 8, 0, 6> TermsCfg;
typedef GemmCfg16<bf16_t, 0, 4, 0, 6> TermsHalfCfg;  // tiles of 128 tokens

// The planes of one operand (`s`), and then, where that or the other one (`also`, null: not there yet) holds values that want
// it, those of both once more (split_again_kernel).
int launch_split(const SplitArgs& s, const SplitArgs* also, int* wide, hipStream_t st) {
  ProfScope prof(PC_TRANSPOSE, st);
  const int64_t blocks = (s.rpad * (s.C / 8) + 255) / 256;
  hipLaunchKernelGGL(split_planes_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096)), dim3(256), 0, st, s, wide);
  int rc = check_launch("split_planes_kernel");
  if (rc || !also) return rc;
  hipLaunchKernelGGL(split_again_kernel, dim3(kNumCUs), dim3(256), 0, st, wide, *also, s);
  return check_launch("split_again_kernel");
}

#if LCE_TU_PART == 0
int forward_terms(const float* h, int64_t ldh, const float* W, int64_t ldw, const int64_t* labels, int64_t T, int64_t H, int64_t V, float temperature,
                  int reduction, float* logprobs, float* entropy, float* maximum, float* accumulate, float* entropy_b, char* ws, size_t ws_bytes,
                  hipStream_t st, int64_t label_offset, float* shard_out, float* xcache) {
  const TermsFwdPlan pl = terms_fwd_plan(T, H, V, ws_bytes);
  bf16_t* h3 = reinterpret_cast<bf16_t*>(ws + pl.off_h);
  bf16_t* w3 = reinterpret_cast<bf16_t*>(ws + pl.off_w);
  int* wide = reinterpret_cast<int*>(ws + pl.off_wide);
  hipLaunchKernelGGL(fill_zero_kernel, dim3(1), dim3(64), 0, st, reinterpret_cast<uint32_t*>(wide), (int64_t)1);
  int rc = check_launch("fill_zero_kernel");
  if (rc) return rc;
  const SplitArgs sh = {h, ldh, T, H, h3, H, round_up(T, 64), nullptr, nullptr};
  if ((rc = launch_split(sh, nullptr, wide, st))) return rc;
  const int ntt = (int)((T + 255) / 256);
  FwdArgs<bf16_t> p;
  p.W = w3; p.ldw = 3 * H; p.h = h3; p.ldh = 3 * H; p.labels = labels; p.T = T; p.H = H;
  p.w_plane = p.h_plane = H * 2;
  p.c = kLog2e / temperature;
  p.xlabel = reinterpret_cast<float*>(ws + pl.off_xlabel);
  p.once_rows = 0;
  const int64_t kept = xcache ? terms_kept_rows(T, H, V) : 0;
  f32x4_t* parts = reinterpret_cast<f32x4_t*>(ws);
  int done = 0;
  for (int c = 0; c < pl.nchunks; ++c) {
    const int64_t v0 = c * pl.rows, rows = std::min(pl.rows, V - v0);
    if ((rc = launch_split({W + v0 * ldw, ldw, rows, H, w3, H, rows, nullptr, nullptr}, &sh, wide, st))) return rc;
    p.S = std::min<int>(terms_fwd_splits(ntt, rows), (int)((rows + 255) / 256));
    p.V = rows;
    p.label_offset = label_offset + v0;
    p.parts = parts + (int64_t)done * T;
    p.split_stride = TermsCfg::BM; p.tile_step = (int64_t)p.S * TermsCfg::BM; p.split_span = rows;
    p.keep_rows = std::min(rows, kept - v0);
    p.xcache = p.keep_rows > 0 ? xcache + v0 * T : nullptr;
    auto launch = [&](auto cfg) {
      typedef decltype(cfg) Cfg;
      const int tt = (int)((T + Cfg::BN - 1) / Cfg::BN);
      p.map = TileMap::make(tt, p.S, block_rows(tt), 1);
      auto kern = p.xcache ? lce_fwd16_kernel<Cfg, true> : lce_fwd16_kernel<Cfg, false>;
      allow_lds(kern, Cfg::LDS_BYTES);
      hipLaunchKernelGGL(kern, dim3(p.map.total), dim3(Cfg::NTHREADS), Cfg::LDS_BYTES, st, p);
    };
    ProfScope prof(PC_FWD, st);
    if (terms_fwd_half(ntt, rows)) launch(TermsHalfCfg{});
    else launch(TermsCfg{});
    if ((rc = check_launch("lce_fwd16_kernel"))) return rc;
    done += p.S;
  }
  float* lp_tok = reduction == LCE_REDUCTION_NONE ? logprobs : reinterpret_cast<float*>(ws + pl.off_lp);
  return forward_merge(parts, p.xlabel, labels, label_offset, V, done, T, p.c, temperature, reduction, lp_tok, logprobs, entropy, maximum, accumulate,
                       entropy_b, shard_out, st);
}

#else
int backward_terms(const float* h, int64_t ldh, const float* W, int64_t ldw, const int64_t* labels, int64_t T, int64_t H, int64_t V, float temperature,
                   int reduction, const float* maximum, const float* accumulate, const float* entropy_b, const float* dlogprobs, const float* dentropy,
                   float* d_hidden, float* d_weight, char* ws, int64_t vchunk, hipStream_t st, int64_t vocab_offset, const Tuning& tu,
                   const float* xcache) {
  typedef TermsCfg Cfg;
  const bool need_dh = d_hidden != nullptr, need_dw = d_weight != nullptr;
  const TermsBwdLayout L = terms_bwd_layout(tu, T, H, V, vchunk);
  bf16_t* dS[2] = {reinterpret_cast<bf16_t*>(ws + L.off_dS[0]), reinterpret_cast<bf16_t*>(ws + L.off_dS[1])};
  bf16_t* w3[2] = {reinterpret_cast<bf16_t*>(ws + L.off_W[0]), reinterpret_cast<bf16_t*>(ws + L.off_W[1])};
  bf16_t* h3 = reinterpret_cast<bf16_t*>(ws + L.off_H);
  float* dHacc = reinterpret_cast<float*>(ws + L.off_dHacc);
  int* rows = reinterpret_cast<int*>(ws + L.off_rows);
  int* inv = reinterpret_cast<int*>(ws + L.off_inv);
  int* n_rows = reinterpret_cast<int*>(ws + L.off_nrows);
  int* wide = n_rows + 1;
  f32x4_t* tokc = reinterpret_cast<f32x4_t*>(ws + L.off_tokc);
  int* tokl = reinterpret_cast<int*>(ws + L.off_tokl);
  const int64_t g_stride = reduction == LCE_REDUCTION_NONE ? 1 : 0;
  const float g_scale = reduction == LCE_REDUCTION_MEAN ? 1.0f / (float)T : 1.0f;
  int rc;
  {
    ProfScope prof(PC_ACTIVE_ROWS, st);
    int* acounts = reinterpret_cast<int*>(ws + L.off_acounts);
    const unsigned nblk = (unsigned)((T + kActiveBlock - 1) / kActiveBlock);
    hipLaunchKernelGGL(active_count_kernel, dim3(nblk), dim3(256), 0, st, dlogprobs, g_stride, dentropy, T, acounts);
    if ((rc = check_launch("active_count_kernel"))) return rc;
    hipLaunchKernelGGL(active_rows_kernel, dim3(nblk), dim3(256), 0, st, dlogprobs, g_stride, dentropy, T, acounts, rows, inv, n_rows);
    if ((rc = check_launch("active_rows_kernel"))) return rc;
    hipLaunchKernelGGL(ds_token_consts_kernel, dim3((unsigned)((L.tpad + 255) / 256)), dim3(256), 0, st, rows, n_rows, T, L.tpad, dlogprobs, g_stride,
                       g_scale, dentropy, maximum, accumulate, entropy_b, labels, vocab_offset, V, 1.0f / temperature, tokc, tokl);
    if ((rc = check_launch("ds_token_consts_kernel"))) return rc;
  }
  hipLaunchKernelGGL(fill_zero_kernel, dim3(1), dim3(64), 0, st, reinterpret_cast<uint32_t*>(wide), (int64_t)1);
  if ((rc = check_launch("fill_zero_kernel"))) return rc;
  const SplitArgs sh = {h, ldh, T, H, h3, L.ldH, L.tpad, rows, n_rows};
  if ((rc = launch_split(sh, nullptr, wide, st))) return rc;
  const int ntt = (int)((T + Cfg::BN - 1) / Cfg::BN), h_tile = hidden_tile(H);
  // K slices of a wide chunk no longer than a usual one's (the same error of d_hidden), or twice as many as that has, where d_hidden's
  // tiles then fill their rounds over the CUs better by a tenth (1024 tokens of H=896, d_hidden alone: 3447 -> 3305 us)
  const TermsChunks chunks = terms_chunks(L, T, H, V);
  int wide_slices = L.ksplit;
  if (chunks.wide > 0) {
    const int64_t tiles = ntt * ((H + h_tile - 1) / h_tile), rows = chunks.at(0).rows, slice = round_up((L.vchunk + L.ksplit - 1) / L.ksplit, Cfg::BK);
    auto time = [&](int64_t s) { return (double)((tiles * s + kNumCUs - 1) / kNumCUs) * ((double)rows / (double)(s * Cfg::BK) + 2); };
    wide_slices = (int)std::max<int64_t>(L.ksplit, (rows + slice - 1) / slice);
    if (time(2 * L.ksplit) < 0.9 * time(wide_slices)) wide_slices = 2 * L.ksplit;
  }
  const int all_slices = std::max(wide_slices, L.ksplit);
  const int nchunks = chunks.count();
  // d_logits of a kept chunk, where the caller has the logits, are a pass of their own instead of tiles
  auto from_cache = [&](int c) { return xcache && c < nchunks && chunks.at(c).kept; };
  // Does chunk c share its products' launch with the d_logits tiles of the next one?  Not where those are no tiles, or where the two are not in
  // different buffers: a wide chunk is in both, and with a single chunk's layout there is but one.
  auto shares = [&](int c) { return L.nchunks > 1 && c + 1 < nchunks && !chunks.at(c).wide && !from_cache(c + 1); };
  auto launch = [&](BwdChunkArgs<bf16_t>& p) {
    if (p.n_gw + p.n_gh + p.n_ds == 0) return (int)LCE_OK;
    ProfScope prof(PC_BWD_CHUNK, st);
    auto kern = h_tile == 224 ? lce_bwd_chunk16_kernel<Cfg, 7> : lce_bwd_chunk16_kernel<Cfg, 8>;
    allow_lds(kern, Cfg::LDS_BYTES);
    hipLaunchKernelGGL(kern, dim3(p.n_gw + p.n_gh + p.n_ds), dim3(Cfg::NTHREADS), Cfg::LDS_BYTES, st, p);
    return check_launch("lce_bwd_chunk16_kernel");
  };
  // step c: the gradient GEMMs of chunk c - 1 and d_logits of chunk c, in one launch as in backward_impl where neither is a pass or a launch of its own
  for (int c = 0; c <= nchunks; ++c) {
    BwdChunkArgs<bf16_t> p;
    p.n_gw = p.n_gh = p.n_ds = 0;
    if (c > 0) {
      const TermsChunks::Chunk k = chunks.at(c - 1);
      const int64_t v0 = k.v0, vrows = k.rows;
      const int64_t kc = round_up(vrows, KPerm<Cfg>::GV);
      if (need_dh) {
        p.gh = make_gemm_args<Cfg>(dS[k.buf], 64, w3[k.buf], 3 * H, T, H, kc, dHacc, H, nullptr, 0, c == 1 ? 0 : 1, h_tile);
        p.gh.tn = 2; p.gh.b_rows_valid = vrows; p.gh.m_dev = n_rows;
        p.gh.a_pcol = L.pcol; p.gh.a_plane = L.plane * 2; p.gh.b_plane = H * 2;
        const int slices = k.wide ? wide_slices : L.ksplit;
        if (slices > 1) {
          p.gh.ksplit = slices;
          p.gh.kslice = round_up((kc + slices - 1) / slices, Cfg::BK);
          p.gh.map = TileMap::make(p.gh.map.nrow_tiles, p.gh.n_tiles * slices, p.gh.map.br, p.gh.map.rows_fastest);
          p.gh.cf_split_stride = (int64_t)(align256((size_t)T * H * 4) / 4);
        }
        p.n_gh = p.gh.map.total;
      }
      if (need_dw) {
        p.gw = make_gemm_args<Cfg>(dS[k.buf], 64, h3, 3 * L.ldH, vrows, H, round_up(T, 64), d_weight + v0 * H, H, nullptr, 0, 0, h_tile);
        p.gw.tn = 1; p.gw.perm_rows = 1; p.gw.k_dev = n_rows; p.gw.k_gran = 64;
        p.gw.a_pcol = L.pcol; p.gw.a_plane = L.plane * 2; p.gw.b_plane = L.ldH * 2;
        p.n_gw = p.gw.map.total;
      }
      if (p.n_gh && p.n_gw && p.gh.kslice > p.gw.K) {  // longer tiles go first
        std::swap(p.gh, p.gw);
        std::swap(p.n_gh, p.n_gw);
      } else if (!p.n_gw) {
        p.gw = p.gh;
        p.n_gw = p.n_gh;
        p.n_gh = 0;
      }
      if (!shares(c - 1)) {
        if ((rc = launch(p))) return rc;
        p.n_gw = p.n_gh = 0;
      }
    }
    if (c == nchunks) break;
    const TermsChunks::Chunk k = chunks.at(c);
    const int64_t v0 = k.v0, vrows = k.rows;
    // (the last reader of this buffer ran in an earlier launch)
    if ((rc = launch_split({W + v0 * ldw, ldw, vrows, H, w3[k.buf], H, vrows, nullptr, nullptr}, &sh, wide, st))) return rc;
    DsArgs<bf16_t>& d = p.ds;
    d.W = w3[k.buf]; d.ldw = 3 * H; d.h = h3; d.ldh = 3 * L.ldH; d.labels = labels; d.T = T; d.H = H;
    d.w_plane = H * 2; d.h_plane = L.ldH * 2; d.dS_plane = L.plane;
    d.v0 = vocab_offset + v0; d.vrows = vrows; d.rcp_tau = 1.0f / temperature; d.c = kLog2e / temperature;
    d.maximum = maximum; d.accumulate = accumulate; d.entropy_b = entropy_b;
    d.g_lp = dlogprobs; d.g_lp_stride = g_stride; d.g_lp_scale = g_scale; d.g_ent = dentropy;
    d.dS = dS[k.buf]; d.ldS = 64; d.pcol = L.pcol; d.dST = nullptr; d.ldST = 0; d.tpad = L.tpad;
    d.rows = nullptr; d.n_rows = n_rows; d.label_outside = 0;
    d.tokc = tokc; d.tokl = tokl; d.lab0 = v0; d.range_rows = 0;
    if (from_cache(c)) {
      ProfScope prof(PC_BWD_DS, st);
      d.rows = rows;  // (the tiles read the compact planes of hidden and no list; the cache is indexed by token)
      hipLaunchKernelGGL((ds_from_logits_kernel<bf16_t, KPerm<Cfg>, Cfg::TERMS>), dim3((unsigned)(round_up(vrows, 256) / 64)), dim3(256), 0, st, d,
                         xcache + v0 * T, T, (int)L.tpad, false);
      if ((rc = check_launch("ds_from_logits_kernel"))) return rc;
      continue;
    }
    d.map = TileMap::make(ntt, (int)((vrows + Cfg::BM - 1) / Cfg::BM), block_rows(ntt), 0);
    p.n_ds = d.map.total;
    if ((rc = launch(p))) return rc;
  }
  if (need_dh) {
    ProfScope prof(PC_DH_FINISH, st);
    LabelTerm lt;
    lt.labels = nullptr; lt.v0 = vocab_offset; lt.V = V; lt.g_lp = dlogprobs; lt.g_stride = g_stride; lt.scale = 0.f;
    int64_t blocks = (T * (H / 4) + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL((dh_finish_kernel<float, float, false>), dim3((unsigned)blocks), dim3(256), 0, st, dHacc, all_slices,
                       (int64_t)(align256((size_t)T * H * 4) / 4), inv, T, H, d_hidden, lt, W, ldw);
    if ((rc = check_launch("dh_finish_kernel"))) return rc;
  }
  return LCE_OK;
}
#endif
#endif

}  // namespace
