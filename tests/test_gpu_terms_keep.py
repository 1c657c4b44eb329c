"""fp32 inputs on bfloat16 planes with kept logits: of every row of the weight up to as many tokens as the hidden size, of the
first rows beyond.  Both ways to d_logits share all of their arithmetic and the order of the sums: the gradients have the bits of
the backward that recomputes."""

import importlib

import pytest
import torch

from oracle import lce_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,H,V,vchunk,reduction,keep", [
    (256, 256, 40011, 0, 0, 0.6),      # all rows, the last tile ragged, as large as the weight
    (513, 896, 30001, 4096, 2, 1.0),   # several chunks; a narrow last tile of tokens
    (700, 256, 50003, 2048, 0, 0.5),   # part of the rows: whole chunks, one cut in two, the others
    (1024, 256, 65536, 0, 1, 0.02),    # a quarter of them, the most tokens that keep any
    (640, 640, 33000, 0, 0, 0.0),      # no token takes part
    (700, 256, 50003, 65536, 0, 1.0),  # part of the rows of one chunk
    (890, 896, 52003, 0, 0, 1.0),      # the forward's last chunk on tiles of 128 tokens
])  # fmt: skip
def test_kept_logits_of_planes(T, H, V, vchunk, reduction, keep):
    from verl_amd import _abi
    from verl_amd.utils.kernel import kernels

    lib = _abi.load()
    assert lib.lce_forward_workspace_bytes(T, H, V, _abi.DTYPE_F32_PLANES) > lib.lce_forward_workspace_bytes(T, H, V, _abi.DTYPE_BF16)
    g = torch.Generator().manual_seed(T + V)
    h = torch.randn(T, H, generator=g).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    y[::7] = -100  # ignored labels
    mask = (torch.rand(T, generator=g) < keep).float().to(DEV)
    g_lp = torch.randn(T, generator=g).to(DEV) * mask if reduction == 0 else torch.tensor(0.7 if keep else 0.0, device=DEV)
    g_ent = torch.randn(T, generator=g).to(DEV) * mask
    plain = kernels.efficient_entropy_forward(h, w, y, reduction, 0.8)
    *kept, cache = kernels.forward_keeping_logits(h, w, y, reduction, 0.8)
    assert all(torch.equal(a, b) for a, b in zip(plain, kept))
    if reduction == 0:
        known = y >= 0
        for got, want in zip(plain[:2], O.lce_forward(h, w, y.clamp(min=0), 0.8, compute_dtype=torch.float64)):
            assert (got.double() - want)[known].abs().max() <= 1e-5 * want[known].abs().max()
    rows = V if T <= H else V * H // T // 256 * 256
    assert cache.numel() == T * ((rows + 63) // 64 * 64) * 4 <= (V + 63) * H * 4
    kernels.set_vocab_chunk(vchunk)
    try:
        run = lambda **kw: kernels.efficient_entropy_backward(g_lp, g_ent, h, w, y, *kept[2:], reduction, False, 0.8, **kw)  # noqa: E731
        dh, dw = run()
        dh1, dw1 = run(logits_cache=cache)
        assert torch.equal(dw, dw1) and torch.equal(dh, dh1)
        assert torch.equal(dh1, run(logits_cache=cache, need_d_weight=False)[0]) and torch.equal(dw, run(logits_cache=cache, need_d_hidden=False)[1])
        torch.cuda.synchronize()
    finally:
        kernels.set_vocab_chunk(0)
    full = g_lp if reduction == 0 else (g_lp / (T if reduction == 2 else 1)).expand(T)
    # (an ignored label has no entry of its own; the oracle takes labels of the vocabulary only)
    want = O.lce_backward(full, g_ent, h, w, y.clamp(min=0), 0.8, compute_dtype=torch.float64)[0]
    want -= ((y < 0) * full / 0.8).double()[:, None] * w[0].double()
    if want.norm() > 0:
        off = ((dh.double() - want).norm() / want.norm()).item()
        print(f"T={T} H={H} V={V}: d_hidden against float64 {off:.2e}")
        assert off <= 3e-6  # the bar of the planes' other tests
    else:
        assert (dh == 0).all()


def test_which_fp32_calls_keep_logits():
    from verl_amd import _abi
    from verl_amd.utils.kernel import kernels

    mod = importlib.import_module("verl_amd.utils.kernel.linear_cross_entropy")
    lib = _abi.load()
    V, H = 40011, 256
    size = lambda T: lib.lce_logits_cache_bytes(T, H, V, _abi.DTYPE_F32_PLANES)  # noqa: E731
    assert size(255) == 0 and size(256) == 256 * 40064 * 4  # planes begin at 256 tokens
    assert size(257) == 257 * 39680 * 4 and size(1024) == 1024 * 9984 * 4 and size(1025) == 0
    assert lib.lce_logits_cache_bytes(256, H, V, _abi.DTYPE_F32) == 0  # (no leave to use the planes)
    try:
        kernels.set_keep_logits_tokens(300)
        assert size(300) > 0 and size(301) == 0
    finally:
        kernels.set_keep_logits_tokens(None)
    # in aggregate: a second graph's logits would pass the weight's size
    w = torch.randn(V, H, device=DEV) * 0.05
    base, outs = mod.kept_logits_bytes(DEV), []
    for _ in range(2):
        h = torch.randn(400, H, device=DEV, requires_grad=True)
        outs.append(mod.linear_cross_entropy(h, w, torch.zeros(400, dtype=torch.int64, device=DEV)))
    assert mod.kept_logits_bytes(DEV) - base == size(400)
    del outs
    assert mod.kept_logits_bytes(DEV) == base
