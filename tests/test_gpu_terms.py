"""fp32 inputs on bfloat16 planes (csrc/lce_terms.hpp): the smallest token counts that take them, tiles with remainders on
every side, one and several vocabulary chunks, tokens without gradient, one gradient only, against float64."""

import pytest
import torch

from oracle import lce_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("T,H,V,tau,keep,reduction,vchunk", [
    (256, 128, 40011, 1.0, 1.0, 0, 0),
    (257, 384, 20003, 0.6, 0.5, 0, 4096),
    (513, 896, 30001, 1.0, 0.02, 0, 0),
    (1025, 128, 65537, 1.3, 0.7, 2, 0),
    (700, 1152, 36864, 1.0, 0.0, 0, 2048),
])  # fmt: skip
def test_planes_of_fp32_inputs(T, H, V, tau, keep, reduction, vchunk):
    from verl_amd import _abi
    from verl_amd.utils.kernel import kernels

    lib = _abi.load()
    planes = lib.lce_forward_workspace_bytes(T, H, V, _abi.DTYPE_F32) > lib.lce_forward_workspace_bytes(T, H, V, _abi.DTYPE_BF16)
    assert planes, "the shape is meant for the planes"
    g = torch.Generator().manual_seed(T + V)
    h = torch.randn(T, H, generator=g).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(DEV)
    w[3] *= 1e-6  # small and large magnitudes next to each other
    h[:, 5] *= 300.0
    w[:, 5] /= 300.0
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    mask = (torch.rand(T, generator=g) < keep).float().to(DEV)
    g_lp = torch.randn(T, generator=g).to(DEV) * mask if reduction == 0 else torch.tensor(0.7, device=DEV)
    g_ent = torch.randn(T, generator=g).to(DEV) * mask
    lp, ent, mx, ac, eb = kernels.efficient_entropy_forward(h, w, y, reduction, tau)
    rlp, rent = O.lce_forward(h, w, y, tau, compute_dtype=torch.float64)
    rlp = rlp if reduction == 0 else rlp.mean()
    full_lp = g_lp if reduction == 0 else torch.full((T,), 0.7 / T, device=DEV)
    rdh, rdw = O.lce_backward(full_lp, g_ent, h, w, y, tau, compute_dtype=torch.float64)
    kernels.set_vocab_chunk(vchunk)
    try:
        dh, dw = kernels.efficient_entropy_backward(g_lp, g_ent, h, w, y, mx, ac, eb, reduction, False, tau)
        dh1, _ = kernels.efficient_entropy_backward(g_lp, g_ent, h, w, y, mx, ac, eb, reduction, False, tau, need_d_weight=False)
        _, dw1 = kernels.efficient_entropy_backward(g_lp, g_ent, h, w, y, mx, ac, eb, reduction, False, tau, need_d_hidden=False)
    finally:
        kernels.set_vocab_chunk(0)
    assert torch.equal(dh, dh1) and torch.equal(dw, dw1)
    for got, want in ((lp, rlp), (ent, rent), (dh, rdh), (dw, rdw)):
        assert got.dtype == torch.float32
        assert (got.double() - want).abs().max().item() <= 1e-5 * want.abs().max().item()
        if want.norm() > 0:  # the fp32 matrix instruction's own error on such shapes is 1e-7 to 6e-6
            assert ((got.double() - want).norm() / want.norm()).item() <= 3e-6
    if reduction == 0:
        assert (dh[mask == 0] == 0).all()
