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


def _close(got, want):
    # fp32 sums of up to V (d_hidden) or T (d_weight) terms whose own errors are those of a logit, 1e-6 of them: 1e-5 in the 2-norm,
    # and of the largest entry for the single ones
    want = want.double()
    err = got.double() - want
    assert err.norm() <= 1e-5 * want.norm(), (err.norm() / want.norm()).item()
    assert err.abs().max() <= 1e-5 * want.abs().max()


@pytest.mark.parametrize("T,H,V", SHAPES)
@pytest.mark.parametrize("keep,vchunk", [(1.0, 0), (0.4, 2048)])
def test_backward(T, H, V, keep, vchunk):
    """Against float64, with tokens without gradient and several chunks of the vocabulary; one gradient alone; nothing written
    beyond the workspace."""
    from verl_amd import _abi

    lib = _abi.load()
    h, w, y, g_lp, g_ent = _case(T, H, V, seed=T + H)
    on = (torch.rand(T, generator=torch.Generator().manual_seed(T)) < keep).to(DEV)
    g_lp, g_ent = g_lp * on, g_ent * on
    from verl_amd.utils.kernel import kernels

    _, _, mx, acc, eb = kernels.efficient_entropy_forward(h, w, y, 0, 0.9)
    need = lib.lce_backward_workspace_bytes(T, H, V, _abi.DTYPE_F32, vchunk)
    ws = torch.full((need + 4096,), 0x5A, device=DEV, dtype=torch.uint8)
    want = O.lce_backward(g_lp.double(), g_ent.double(), h.double(), w.double(), y, 0.9)
    for need_dh, need_dw in ((True, True), (True, False), (False, True)):
        dh, dw = torch.full_like(h, 7.0), torch.full_like(w, 7.0)
        rc = lib.lce_backward(
            h.data_ptr(), H, w.data_ptr(), H, y.data_ptr(), T, H, V, _abi.DTYPE_F32, 0.9, 0, mx.data_ptr(), acc.data_ptr(), eb.data_ptr(),
            g_lp.data_ptr(), g_ent.data_ptr(), dh.data_ptr() if need_dh else None, dw.data_ptr() if need_dw else None, ws.data_ptr(), need,
            vchunk, _abi.current_stream(h.device),
        )  # fmt: skip
        assert rc == 0 and (ws[need:] == 0x5A).all()
        if need_dh:
            _close(dh, want[0])
            assert torch.count_nonzero(dh[~on]) == 0
        if need_dw:
            _close(dw, want[1])


def test_no_token_takes_part():
    from verl_amd.utils.kernel import kernels

    h, w, y, g_lp, g_ent = _case(40, 256, 5003, seed=1)
    _, _, mx, acc, eb = kernels.efficient_entropy_forward(h, w, y, 0, 1.0)
    dh, dw = kernels.efficient_entropy_backward(g_lp * 0, None, h, w, y, mx, acc, eb, 0, False, 1.0)
    assert torch.count_nonzero(dh) == 0 and torch.count_nonzero(dw) == 0
