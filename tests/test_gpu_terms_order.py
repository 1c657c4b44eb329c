"""fp32 inputs on bfloat16 planes: the gradients are a function of inputs and settings.  Whether a forward keeps its logits depends on
what other graphs hold at that moment, so the order of d_hidden's sums must not depend on it."""

import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,H,V,vchunk", [
    (256, 256, 40011, 0),      # as large as the weight
    (600, 896, 80003, 8192),   # wide chunks, the last one narrower
    (1024, 896, 151936, 0),    # wide chunks of kept rows, one of the usual width, the others
    (700, 256, 50003, 2048),   # part of the rows, chunks of the usual width
    (700, 256, 50003, 65536),  # part of the rows, one buffer
    (1100, 256, 65536, 4096),  # more tokens than keep any
])  # fmt: skip
def test_same_bits_with_and_without_room_for_the_logits(T, H, V, vchunk):
    from verl_amd.utils.kernel import kernels

    mod = importlib.import_module("verl_amd.utils.kernel.linear_cross_entropy")
    g = torch.Generator().manual_seed(T + V)
    w = (torch.randn(V, H, generator=g) * 0.05).to(DEV).requires_grad_(True)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    h = torch.randn(T, H, generator=g).to(DEV)
    g_lp, g_ent = torch.randn(T, generator=g).to(DEV), torch.randn(T, generator=g).to(DEV)
    g_lp[::5], g_ent[::5] = 0, 0
    rows = [h.clone().requires_grad_(True) for _ in range(3)]
    base, held, outs = mod.kept_logits_bytes(DEV), [], []
    kernels.set_vocab_chunk(vchunk)
    try:
        for x in rows:  # (in one graph: the weight's share of them is kept, that of the last one at most in part)
            outs.append(mod.linear_cross_entropy(x, w, y, 0.8))
            held.append(mod.kept_logits_bytes(DEV) - base)
        assert held[0] == kernels.kept_logits_size(T, H, V, 3)
        assert held[0] == 0 or held[-1] < 3 * held[0], "all of them found room"
        grads = [torch.autograd.grad(o, (x, w), (g_lp, g_ent)) for o, x in zip(outs, rows)]
    finally:
        kernels.set_vocab_chunk(0)
    for d_hidden, d_weight in grads[1:]:
        assert torch.equal(d_weight, grads[0][1])
        assert torch.equal(d_hidden, grads[0][0])
