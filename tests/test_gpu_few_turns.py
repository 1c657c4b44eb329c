"""The forward of few tokens where a pass over 256 rows of W is not whole turns of its ring (hidden sizes that are no multiple of
256): one to three passes per workgroup, against log-probs and entropies in float64, with and without kept logits."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,V", [
    (1, 128, 300),        # half a turn and nothing else
    (40, 128, 90001),     # two passes of half a turn
    (64, 384, 65536),     # one whole pass each
    (17, 640, 65537),     # rows of a second pass in some workgroups
    (64, 896, 140001),    # three passes, the last one short
    (33, 256, 140001),    # whole turns
    (65, 384, 90001),     # three blocks of 32 tokens from here on
    (96, 512, 140001),
    (80, 896, 20011),
    (97, 384, 90001),     # the 256 x 128 tile
])
def test_passes(T, H, V, dtype):
    from verl_amd.utils.kernel import kernels

    g = torch.Generator().manual_seed(T + V)
    h = torch.randn(T, H, generator=g).to(dtype).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(dtype).to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    plain = kernels.efficient_entropy_forward(h, w, y, 0, 0.9)
    *kept, cache = kernels.forward_keeping_logits(h, w, y, 0, 0.9)
    for a, b in zip(plain, kept):
        assert torch.equal(a, b)
    x = h.double() @ w.double().t() / 0.9
    p = torch.log_softmax(x, -1)
    # logits of fp32 sums over H terms of O(0.05 sqrt(H)) in all, and a fp32 sum over the vocabulary
    assert (plain[0].double() - p.gather(1, y[:, None])[:, 0]).abs().max() < 2e-4
    assert (plain[1].double() + (p.exp() * p).sum(-1)).abs().max() < 2e-4
    if cache is not None:
        panels = (V + 15) // 16
        got = cache.view(torch.float32).reshape(-1)[: panels * T * 16].view(panels, T, 16).permute(1, 0, 2).reshape(T, panels * 16)[:, :V]
        bound = H * 2.0**-24 * (h.double().abs() @ w.double().abs().t())
        assert ((got.double() - x * 0.9).abs() <= bound).all()
