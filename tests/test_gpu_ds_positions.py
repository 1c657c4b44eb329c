"""d_logits of few tokens from kept logits: only the positions of tokens with a gradient are written, and the streaming kernels read no
others.  A workspace full of NaN must not show, whatever share of the tokens takes part."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T", [1, 8, 63, 64, 65, 127, 128])
@pytest.mark.parametrize("active", [0.0, 0.1, 0.6, 1.0])
def test_nothing_is_read_behind_the_last_position(T, active, dtype):
    from verl_amd.utils.kernel import kernels

    H, V = 384, 20011
    g = torch.Generator().manual_seed(T)
    h = torch.randn(T, H, generator=g).to(dtype).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(dtype).to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    on = (torch.arange(T) < round(active * T)).to(DEV)
    g_lp, g_ent = torch.randn(T, generator=g).to(DEV) * on, torch.randn(T, generator=g).to(DEV) * on
    *out, cache = kernels.forward_keeping_logits(h, w, y, 0, 0.9)
    mx, acc, eb = out[2:]
    run = lambda **k: kernels.efficient_entropy_backward(g_lp, g_ent, h, w, y, mx, acc, eb, 0, False, 0.9, **k)  # noqa: E731
    want = run()  # recomputes the logits
    for size in (1 << 20, 1 << 22, 1 << 24, 1 << 26):  # what the allocator hands out for the workspace
        torch.full((size,), float("nan"), device=DEV)
    got = run(logits_cache=cache)
    for a, b in zip(want, got):
        assert torch.equal(a, b)
