"""The 16x16x32 forward's stream of tiles and the line-wise epilogues of the gradient GEMMs at their edges: K of one and two
slabs, splits of one tile, of a short last tile and of several, gradients over several chunks with full and cut tiles; against
the oracle."""

import pytest
import torch

from oracle import lce_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,V,vchunk", [
    (769, 128, 300, 0),        # two slabs of K, a split of one full tile and one of a short one
    (1025, 128, 70001, 4096),  # the wavefronts walk tiles; eighteen chunks add to d_hidden
    (2561, 640, 33024, 0),     # whole tiles only along the vocabulary
    (1300, 384, 66049, 16384),
])
def test_tiles_follow_each_other(T, H, V, vchunk, dtype):
    from verl_amd import linear_cross_entropy
    from verl_amd.utils.kernel import kernels

    g = torch.Generator().manual_seed(T + V)
    h = torch.randn(T, H, generator=g).to(dtype).to(DEV).requires_grad_(True)
    w = (torch.randn(V, H, generator=g) * 0.05).to(dtype).to(DEV).requires_grad_(True)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    g_lp, g_ent = torch.randn(T, generator=g).to(DEV), torch.randn(T, generator=g).to(DEV)
    try:
        kernels.set_vocab_chunk(vchunk)
        lp, ent = linear_cross_entropy(h, w, y, 0.8, "none")
        torch.autograd.backward([lp, ent], [g_lp, g_ent])
        torch.cuda.synchronize()
    finally:
        kernels.set_vocab_chunk(0)
    rlp, rent = O.lce_forward(h.detach(), w.detach(), y, 0.8)
    rdh, rdw = O.lce_backward(g_lp, g_ent, h.detach(), w.detach(), y, 0.8)
    torch.testing.assert_close(lp, rlp, atol=1e-3, rtol=2e-4)
    torch.testing.assert_close(ent, rent, atol=5e-3, rtol=5e-4)
    for got, want in ((h.grad, rdh), (w.grad, rdw)):
        err = (got.double() - want.double()).abs()
        assert (err <= 2e-2 + 2.0**-7 * want.double().abs()).all(), err.max().item()


@pytest.mark.parametrize("T", [65, 700, 5000])
def test_one_slab_of_k(T):
    """A hidden size of 64, which the C ABI takes and the stream of slabs does not."""
    from verl_amd import _abi

    lib, H, V = _abi.load(), 64, 3001
    g = torch.Generator().manual_seed(T)
    h = torch.randn(T, H, generator=g).bfloat16().to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.1).bfloat16().to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    out = [torch.empty(T, device=DEV) for _ in range(5)]
    ws = torch.empty(lib.lce_forward_workspace_bytes(T, H, V, _abi.DTYPE_BF16), device=DEV, dtype=torch.uint8)
    rc = lib.lce_forward(
        h.data_ptr(), H, w.data_ptr(), H, y.data_ptr(), T, H, V, _abi.DTYPE_BF16, 1.0, 0, *(o.data_ptr() for o in out),
        ws.data_ptr(), ws.numel(), torch.cuda.current_stream().cuda_stream,
    )  # fmt: skip
    _abi.check(rc, "lce_forward")
    rlp, rent = O.lce_forward(h, w, y, 1.0)
    torch.testing.assert_close(out[0], rlp, atol=1e-3, rtol=2e-4)
    torch.testing.assert_close(out[1], rent, atol=5e-3, rtol=5e-4)
