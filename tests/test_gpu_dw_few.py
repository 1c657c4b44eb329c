"""d_weight of 129 to 256 tokens by the streaming kernel (hidden in registers, 64-column blocks of the logits' gradient through
LDS), at the edges of its token positions, of its 512 columns of the hidden size and of its 64 rows of the vocabulary: against
the oracle, and bit for bit against the tile kernels, which take the same products in the same order."""

import pytest
import torch

from oracle import lce_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
OPT_SPLIT_LAUNCHES = 1  # the three sub-problems of a backward as launches of the tile kernels


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,V,keep", [
    (129, 512, 20011, 1.0),
    (160, 640, 5003, 1.0),     # a second workgroup of 128 columns
    (191, 384, 300, 0.9),
    (192, 1024, 9001, 1.0),    # the last count of 192 positions
    (193, 512, 20011, 1.0),    # the first of 256
    (255, 1152, 4160, 0.5),    # half of the positions without a token
    (256, 896, 30001, 1.0),
    (256, 512, 20011, 0.1),    # one k-step of eight
    (200, 512, 20011, 0.0),    # no token takes part: zeros
    (257, 512, 9001, 1.0),     # the tile kernels
])
def test_against_the_oracle_and_the_tiles(T, H, V, keep, dtype):
    from verl_amd import _abi
    from verl_amd.utils.kernel import kernels

    lib = _abi.load()
    g = torch.Generator().manual_seed(T + H)
    h = torch.randn(T, H, generator=g).to(dtype).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(dtype).to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    on = (torch.rand(T, generator=g) < keep).to(DEV)
    g_lp = torch.randn(T, generator=g).to(DEV) * on
    g_ent = torch.randn(T, generator=g).to(DEV) * on
    _, _, mx, acc, eb = kernels.efficient_entropy_forward(h, w, y, 0, 0.8)
    run = lambda fp32: kernels.efficient_entropy_backward(g_lp, g_ent, h, w, y, mx, acc, eb, 0, fp32, 0.8)[1]  # noqa: E731
    dw, dw32 = run(False), run(True)
    try:
        assert lib.lce_set_option(OPT_SPLIT_LAUNCHES, 1) == 0
        tiles, tiles32 = run(False), run(True)
    finally:
        lib.lce_set_option(OPT_SPLIT_LAUNCHES, 0)
    assert torch.equal(dw, tiles) and torch.equal(dw32, tiles32)
    want = O.lce_backward(g_lp, g_ent, h, w, y, 0.8)[1].double()
    # half an ulp of the result's own rounding, and the 16-bit rounding of d_logits (2^-9 of terms that are O(p)): the bar of the
    # other backward tests
    assert ((dw.double() - want).abs() <= 2e-2 + 2.0**-7 * want.abs()).all()
