"""The sum of d_hidden's partials over the vocabulary slices (16, four and one loads at a time) at counts around those steps,
against the product in float64."""

import pytest
import torch

from oracle import lce_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("slices", [1, 2, 4, 5, 6, 16, 17, 18, 20, 21, 33, 36])
def test_counts_of_slices(slices, dtype):
    from verl_amd.utils.kernel import kernels

    T, H, V = 9, 384, 512 * slices  # a slice is 512 rows of W or more
    g = torch.Generator().manual_seed(slices)
    h = torch.randn(T, H, generator=g).to(dtype).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(dtype).to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    g_lp, g_ent = torch.randn(T, generator=g).to(DEV), torch.randn(T, generator=g).to(DEV)
    _, _, mx, acc, eb = kernels.efficient_entropy_forward(h, w, y, 0, 0.8)
    got = kernels.efficient_entropy_backward(g_lp, g_ent, h, w, y, mx, acc, eb, 0, True, 0.8)[0].double()
    want = O.lce_backward(g_lp, g_ent, h, w, y, 0.8)[0].double()
    # the 16-bit rounding of d_logits (2^-9 of terms that are O(p)): the bar of the other backward tests; fp32 sums of O(1) terms
    bound = 2e-2 + 2.0**-7 * want.abs() if dtype is torch.bfloat16 else 1e-4 + 2.0**-12 * want.abs()
    assert ((got - want).abs() <= bound).all()
