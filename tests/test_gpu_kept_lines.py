"""The kept logits of 65 to 128 tokens, which leave the tile through lane swaps in whole lines: every entry of the cache, at the
edges of the 16 tokens of a line, of the panels of 16 vocabulary rows and of the splits' ranges."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,V", [(65, 20011), (79, 300), (80, 5003), (81, 66), (96, 9001), (97, 152064), (112, 65), (113, 30001), (127, 64), (128, 100003)])
def test_every_kept_logit(T, V, dtype):
    from verl_amd.utils.kernel import kernels

    H = 384
    g = torch.Generator().manual_seed(T + V)
    h = torch.randn(T, H, generator=g).to(dtype).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(dtype).to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    plain = kernels.efficient_entropy_forward(h, w, y, 0, 0.9)
    *kept, cache = kernels.forward_keeping_logits(h, w, y, 0, 0.9)
    for a, b in zip(plain, kept):
        assert torch.equal(a, b)
    panels = (V + 15) // 16
    got = cache.view(torch.float32).reshape(-1)[: panels * T * 16].view(panels, T, 16).permute(1, 0, 2).reshape(T, panels * 16)[:, :V]
    want = h.double() @ w.double().t()
    # H rounded sums of exact products: each entry within H ulps of half, of the sum of its terms' sizes
    bound = H * 2.0**-24 * (h.double().abs() @ w.double().abs().t())
    assert ((got.double() - want).abs() <= bound).all()
