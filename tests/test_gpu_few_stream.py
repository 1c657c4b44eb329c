"""Streaming kernels for few tokens (csrc/few_tokens.hpp) at their edges: vocabularies of less than a workgroup's rows and of a
second pass with few rows, K of less than one turn of the load pipeline and with a remainder, column tiles that are partly
beyond the hidden size, tokens without gradient; forward and both gradients against the oracle, padded rows untouched."""

import pytest
import torch

from oracle import lce_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,V,keep", [
    (1, 128, 5, 1.0),
    (33, 384, 1037, 0.5),
    (64, 640, 70001, 0.1),
    (63, 896, 131072, 1.0),
    (65, 1152, 66053, 0.3),
    (128, 4224, 20002, 0.9),
])
def test_few_tokens_at_the_edges(T, H, V, keep, dtype):
    from verl_amd import linear_cross_entropy

    tau = 0.7
    g = torch.Generator().manual_seed(T + V)
    h = torch.randn(T, H, generator=g).to(dtype).to(DEV).requires_grad_(True)
    w = (torch.randn(V, H, generator=g) * 0.05).to(dtype).to(DEV).requires_grad_(True)
    y = torch.randint(0, V, (T,), generator=g)
    y[0], y[-1] = 0, V - 1
    y = y.to(DEV)
    mask = (torch.rand(T, generator=g) < keep).float().to(DEV)
    g_lp, g_ent = torch.randn(T, generator=g).to(DEV) * mask, torch.randn(T, generator=g).to(DEV) * mask
    with torch.no_grad():
        plain = linear_cross_entropy(h, w, y, tau, "none")
    lp, ent = linear_cross_entropy(h, w, y, tau, "none")
    assert torch.equal(lp, plain[0]) and torch.equal(ent, plain[1])  # keeping the logits changes nothing
    torch.autograd.backward([lp, ent], [g_lp, g_ent])
    rlp, rent = O.lce_forward(h.detach(), w.detach(), y, tau)
    rdh, rdw = O.lce_backward(g_lp, g_ent, h.detach(), w.detach(), y, tau)
    torch.testing.assert_close(lp, rlp, atol=1e-3, rtol=2e-4)
    torch.testing.assert_close(ent, rent, atol=5e-3, rtol=5e-4)
    for got, want in ((h.grad, rdh), (w.grad, rdw)):
        err = (got.double() - want.double()).abs()
        assert (err <= 2e-2 + 2.0**-7 * want.double().abs()).all(), err.max().item()


@pytest.mark.parametrize("T", [1, 40, 64, 65, 128])
@pytest.mark.parametrize("H,V,dtype", [(256, 9000, torch.bfloat16), (512, 70001, torch.float16), (1024, 160001, torch.bfloat16), (1024, 163840, torch.bfloat16),
                                       (512, 60001, torch.float32), (1024, 90001, torch.float32)])
def test_forward_whatever_the_loads_of_the_weight(T, H, V, dtype):
    """Weights below 64 MB, above, just below and at 5/4 of the memory-side cache (320 MB) and above it, with and without kept
    logits: which part is read with non-temporal loads must not show.  16-bit inputs: bit for bit the outputs of the forward
    that keeps its logits, which reads everything the other way; all of them against float64."""
    from oracle import lce_oracle as O
    from verl_amd.utils.kernel import kernels

    g = torch.Generator(device=DEV).manual_seed(T + V)
    h = torch.randn(T, H, device=DEV, generator=g).to(dtype)
    w = torch.empty(V, H, device=DEV, dtype=dtype)
    for r in range(0, V, 1 << 15):
        w[r : r + (1 << 15)] = torch.randn(min(1 << 15, V - r), H, device=DEV, generator=g) * 0.05
    y = torch.randint(0, V, (T,), device=DEV, generator=g)
    got = kernels.efficient_entropy_forward(h, w, y, 0, 0.9)
    if dtype != torch.float32:
        *kept, cache = kernels.forward_keeping_logits(h, w, y, 0, 0.9)
        assert cache is not None
        for a, b in zip(got, kept):
            torch.testing.assert_close(a, b, rtol=0, atol=0)
    lp, ent = O.lce_forward(h, w, y, 0.9, compute_dtype=torch.float64)
    torch.testing.assert_close(got[0].double(), lp, rtol=2e-5, atol=2e-5)  # (fp32 sums over H and V)
    torch.testing.assert_close(got[1].double(), ent, rtol=2e-5, atol=2e-5)
