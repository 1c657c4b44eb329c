"""fp32 inputs with at most 255 tokens: kept logits give the same bits as the backward that recomputes them, at the edges of the
positions (32, 64, 96, 128, 192), of panels and chunks of the vocabulary, with ignored labels and tokens without gradient; 129 to 255
tokens, in two groups, against float64."""

import pytest
import torch

from oracle import lce_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,H,V,vchunk,reduction,keep", [
    (1, 128, 5003, 0, 0, 1.0),
    (31, 896, 20011, 4096, 2, 1.0),
    (33, 384, 300, 0, 0, 0.7),       # fewer panels than workgroups
    (64, 512, 5003, 2048, 0, 0.3),
    (65, 128, 40011, 0, 1, 1.0),
    (97, 640, 9001, 0, 0, 0.0),      # no token takes part
    (128, 128, 20003, 4096, 0, 0.9),  # as large as the weight
    (129, 256, 5003, 2048, 2, 1.0),
    (160, 384, 9001, 0, 1, 0.6),     # the second group may have no token that takes part
    (193, 640, 20011, 0, 0, 1.0),
    (255, 256, 12007, 4096, 0, 0.8),
])  # fmt: skip
def test_kept_logits_of_few_fp32_tokens(T, H, V, vchunk, reduction, keep):
    from verl_amd.utils.kernel import kernels

    g = torch.Generator().manual_seed(T + V)
    h = torch.randn(T, H, generator=g).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    y[2::7] = -100
    mask = (torch.rand(T, generator=g) < keep).float().to(DEV)
    g_lp = torch.randn(T, generator=g).to(DEV) * mask if reduction == 0 else torch.tensor(0.7, device=DEV)
    g_ent = torch.randn(T, generator=g).to(DEV) * mask
    plain = kernels.efficient_entropy_forward(h, w, y, reduction, 0.8)
    *kept, cache = kernels.forward_keeping_logits(h, w, y, reduction, 0.8)
    assert all(torch.equal(a, b) for a, b in zip(plain, kept))
    assert cache.numel() == T * ((V + 63) // 64 * 64) * 4
    kernels.set_vocab_chunk(vchunk)
    try:
        run = lambda **kw: kernels.efficient_entropy_backward(g_lp, g_ent, h, w, y, *kept[2:], reduction, False, 0.8, **kw)  # noqa: E731
        dh, dw = run()
        dh1, dw1 = run(logits_cache=cache)
        assert torch.equal(dh, dh1) and torch.equal(dw, dw1)
        assert torch.equal(dh, run(logits_cache=cache, need_d_weight=False)[0]) and torch.equal(dw, run(logits_cache=cache, need_d_hidden=False)[1])
        torch.cuda.synchronize()
    finally:
        kernels.set_vocab_chunk(0)
    if T <= 128:
        return  # (against float64 in other tests)
    # (an ignored label has no entry of its own; the oracle takes labels of the vocabulary only)
    known, full = y >= 0, g_lp if reduction == 0 else (g_lp / (T if reduction == 2 else 1)).expand(T)
    lp, ent = O.lce_forward(h, w, y.clamp(min=0), 0.8, compute_dtype=torch.float64)
    rdh, rdw = O.lce_backward(full * known, g_ent, h, w, y.clamp(min=0), 0.8, compute_dtype=torch.float64)
    only, only_w = O.lce_backward(full * ~known, torch.zeros(T, device=DEV), h, w, y.clamp(min=0), 0.8, compute_dtype=torch.float64)
    share = ((full * ~known) / 0.8).double()
    rdh += only - share[:, None] * w[0].double()
    only_w[0] -= share @ h.double()
    rdw += only_w
    checks = [(ent0, want) for ent0, want in ((plain[1], ent), (dh1, rdh), (dw1, rdw))]
    checks.append((plain[0][known], lp[known]) if reduction == 0 else (torch.zeros(1, device=DEV), torch.zeros(1, device=DEV).double()))
    for got, want in checks:
        assert (got.double() - want).abs().max() <= 1e-5 * want.abs().max()
        if want.norm() > 0:  # the bar of the other fp32 tests
            assert (got.double() - want).norm() <= 6e-6 * want.norm()


def test_which_few_fp32_tokens_keep_theirs():
    from verl_amd import _abi
    from verl_amd.utils.kernel import kernels

    # (a small vocabulary: no planes from 256 tokens on)
    size = lambda T, H=256: kernels.kept_logits_size(T, H, 1000, _abi.DTYPE_F32_PLANES)  # noqa: E731
    assert size(0) == 0 and size(1) == 1024 * 4 and size(255) == 255 * 1024 * 4 and size(256) == 0
    assert size(64, 64) > 0 and size(65, 64) == 0  # (never more than the weight)
    h, w, y = torch.randn(16, 256, device=DEV), torch.randn(1000, 256, device=DEV), torch.zeros(16, dtype=torch.int64, device=DEV)
    assert kernels.forward_keeping_logits(h, w, y, 0, 1.0)[5] is not None
    try:
        kernels.set_keep_logits_tokens(15)
        assert kernels.forward_keeping_logits(h, w, y, 0, 1.0)[5] is None
    finally:
        kernels.set_keep_logits_tokens(None)
