"""d_hidden of 129 to 512 tokens with a d_weight behind it: its loads of the weight are then marked as read once (the ONCE
variants of lce_dh16_kernel), which must not change a bit, whatever share of the tokens takes part."""

import pytest
import torch

from oracle import lce_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,V,active", [
    (129, 256, 40011, (129, 40)),            # one row tile, 192 wide
    (192, 640, 20011, (192, 191, 1)),
    (256, 1152, 20011, (256, 193, 130)),     # 256 wide
    (333, 2048, 20011, (333, 200)),
    (512, 512, 40011, (512, 257, 256, 10)),
])
def test_with_and_without_a_d_weight(T, H, V, active, dtype):
    from verl_amd.utils.kernel import kernels

    g = torch.Generator().manual_seed(T)
    h = torch.randn(T, H, generator=g).to(dtype).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(dtype).to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    base_lp, base_ent = torch.randn(T, generator=g).to(DEV), torch.randn(T, generator=g).to(DEV)
    _, _, mx, acc, eb = kernels.efficient_entropy_forward(h, w, y, 0, 1.0)
    for n in active:
        on = torch.zeros(T, dtype=torch.bool)
        on[torch.randperm(T, generator=g)[:n]] = True
        on = on.to(DEV)
        g_lp, g_ent = base_lp * on, base_ent * on
        dh, dw = kernels.efficient_entropy_backward(g_lp, g_ent, h, w, y, mx, acc, eb, 0, False, 1.0)
        alone, _ = kernels.efficient_entropy_backward(g_lp, g_ent, h, w, y, mx, acc, eb, 0, False, 1.0, need_d_weight=False)
        assert torch.equal(dh, alone), n
        want_dh, want_dw = O.lce_backward(g_lp.double(), g_ent.double(), h.double(), w.double(), y, 1.0)
        # every entry of the logits' gradient and every result is rounded to the inputs' type, half an ulp each, the rest is fp32: of
        # sums of independent terms that is at most one ulp, 2^-8 or 2^-11, in the 2-norm; twice that for fp16, whose small
        # entries (a softmax over 20000 values) are below its normal range, in steps of 2^-24
        bar = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-10
        for got, want in ((dh, want_dh), (dw, want_dw)):
            rel = ((got.double() - want).norm() / want.norm()).item()
            print(f"T={T} {n} active {dtype}: {rel:.2e}")
            assert rel <= bar, (n, rel)
