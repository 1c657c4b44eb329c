"""fp32 inputs with at most 128 tokens: the streaming kernels, at the edges of their token widths (32, 64, 96, 128), of the rows a
workgroup walks and of the K stages, against float64."""

import pytest
import torch

from oracle import lce_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(T, H, V, seed):
    g = torch.Generator().manual_seed(seed)
    h = torch.randn(T, H, generator=g).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    return h, w, y, torch.randn(T, generator=g).to(DEV), torch.randn(T, generator=g).to(DEV)


SHAPES = [
    (1, 128, 300), (31, 256, 5003), (32, 384, 40000), (33, 1024, 20011), (64, 128, 70001), (65, 640, 9001), (96, 256, 30001),
    (97, 512, 20011), (128, 896, 12007), (129, 256, 5003),
]  # fmt: skip


@pytest.mark.parametrize("T,H,V", SHAPES)
def test_forward(T, H, V):
    from verl_amd.utils.kernel import kernels

    h, w, y, _, _ = _case(T, H, V, seed=T + V)
    y[::7] = -100
    lp, ent, mx, acc, eb = kernels.efficient_entropy_forward(h, w, y, 0, 0.9)
    rlp, rent = O.lce_forward(h.double(), w.double(), y.clamp(min=0), 0.9)  # (the oracle gathers by label)
    ok = y >= 0
    # fp32 sums of H products of unit size times 0.05, then differences of numbers around max |logit|: 1e-5 relative
    torch.testing.assert_close(lp.double()[ok], rlp.double()[ok], atol=1e-5, rtol=1e-5)
    torch.testing.assert_close(ent.double(), rent.double(), atol=1e-5, rtol=1e-5)
