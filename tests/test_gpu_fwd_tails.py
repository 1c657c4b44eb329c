"""The forward's last token tile on the narrowest width that holds its tokens (160, 192, 224 or the whole tile): values of every token
at the edges of the widths against the oracle, bit for bit with and without kept logits, and fp32 on planes."""

import pytest
import torch

from oracle import lce_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(T, H, V, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    h = torch.randn(T, H, generator=g).to(dtype).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(dtype).to(DEV)
    return h, w, torch.randint(0, V, (T,), generator=g).to(DEV)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T", [129, 160, 161, 192, 193, 224, 225, 256, 257, 352, 353, 384, 385, 416, 417, 448, 480, 481, 512, 513])
def test_widths(T, dtype):
    from verl_amd.utils.kernel import kernels

    H, V = 1152, 9001
    h, w, y = _case(T, H, V, dtype, seed=T)
    plain = kernels.efficient_entropy_forward(h, w, y, 0, 0.9)
    *kept, cache = kernels.forward_keeping_logits(h, w, y, 0, 0.9)
    assert cache is not None
    for a, b in zip(plain, kept):
        assert torch.equal(a, b)
    rlp, rent = O.lce_forward(h.double(), w.double(), y, 0.9)
    # 16-bit inputs are exact in fp32, so these are the errors of fp32 sums of H products and of differences of numbers around max |logit|
    torch.testing.assert_close(plain[0].double(), rlp.double(), atol=2e-5, rtol=2e-5)
    torch.testing.assert_close(plain[1].double(), rent.double(), atol=2e-5, rtol=2e-5)
    # the kept logits of every token, in panels of 16 rows
    x = cache.view(torch.float32).reshape(-1, T, 16).transpose(0, 1).reshape(T, -1)[:, :V]
    want = h.float() @ w.float().t()
    assert ((x - want).abs() <= 1e-4 * want.abs().max()).all()


@pytest.mark.parametrize("T", [257, 300, 416, 417, 448, 480, 481, 600])
def test_widths_on_planes(T):
    from verl_amd.utils.kernel import kernels

    h, w, y = _case(T, 640, 20011, torch.float32, seed=T)
    lp, ent, *_ = kernels.efficient_entropy_forward(h, w, y, 0, 0.9)
    rlp, rent = O.lce_forward(h.double(), w.double(), y, 0.9)
    torch.testing.assert_close(lp.double(), rlp.double(), atol=1e-5, rtol=1e-5)
    torch.testing.assert_close(ent.double(), rent.double(), atol=1e-5, rtol=1e-5)
