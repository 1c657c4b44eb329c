"""d_weight of 257 to 2048 tokens by workgroups that walk tiles, a tile leaving the accumulators as the next one starts: last slabs
of half a slab and whole ones, two slabs and many, one tile to a workgroup and two, tiles cut by the last rows and columns; bit for
bit against a workgroup per tile, which takes the same products in the same order, and against the oracle."""

import pytest
import torch

from oracle import lce_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
OPT_SPLIT_LAUNCHES = 1  # the three sub-problems of a backward as launches of the tile kernels


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,V,with_gradient", [
    (257, 1024, 20011, (257, 256, 97, 96, 65, 64, 1, 0)),  # five slabs, the last a half; 2, 1.5 and 1 (as two)
    (289, 640, 20011, (289, 160)),                         # the last k-step of 32; a last tile of 128 columns
    (500, 896, 30001, (500, 333, 129)),                    # tiles of 224 columns
    (1000, 2048, 9001, (1000, 700)),                       # some workgroups walk two tiles, the others one
    (300, 1024, 1003, (300, 288)),                         # fewer tiles than workgroups, the last of 235 rows
])
def test_tiles_of_a_walk(T, H, V, with_gradient, dtype):
    from verl_amd import _abi
    from verl_amd.utils.kernel import kernels

    lib = _abi.load()
    g = torch.Generator().manual_seed(T + H)
    h = torch.randn(T, H, generator=g).to(dtype).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(dtype).to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    g_lp, g_ent = torch.randn(T, generator=g).to(DEV), torch.randn(T, generator=g).to(DEV)
    _, _, mx, acc, eb = kernels.efficient_entropy_forward(h, w, y, 0, 0.8)
    for n in with_gradient:
        on = torch.zeros(T, device=DEV)
        on[torch.randperm(T, generator=g)[:n].to(DEV)] = 1.0
        run = lambda: kernels.efficient_entropy_backward(g_lp * on, g_ent * on, h, w, y, mx, acc, eb, 0, False, 0.8)[1]  # noqa: E731
        dw = run()
        try:
            assert lib.lce_set_option(OPT_SPLIT_LAUNCHES, 1) == 0
            tiles = run()
        finally:
            lib.lce_set_option(OPT_SPLIT_LAUNCHES, 0)
        assert torch.equal(dw, tiles), n
        want = O.lce_backward(g_lp * on, g_ent * on, h, w, y, 0.8, compute_dtype=torch.float64)[1]
        # the rounding of the result, and the 16-bit rounding of d_logits (2^-8 of terms that are O(p)): the bar of the
        # other backward tests
        assert ((dw.double() - want).abs() <= 2e-2 + 2.0**-7 * want.abs()).all(), n
        # the rows without a label's entry, which is most of the result where there is one, by their own 2-norm: d_logits and the result are
        # rounded by up to 2^-8 each (independently, some 0.4 of that in the mean)
        rest = torch.ones(V, dtype=torch.bool, device=DEV)
        rest[y[on > 0]] = False
        assert n == 0 or ((dw.double() - want)[rest].norm() / want[rest].norm()).item() <= 2.0**-8, n
