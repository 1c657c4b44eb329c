"""d_hidden of 129 to 2048 tokens as a launch of its own: the K slices are those of the row tiles that take part, a number that
only the device knows.  Counts of tokens with a gradient at the edges of the row tiles (192 or 256 wide), against the oracle, and
nothing written beyond the workspace that the library asks for."""

import pytest
import torch

from tiles_part import check_tiles_part

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,V,active", [
    (192, 512, 20011, (0, 1, 192)),
    (300, 640, 20011, (1, 192, 193, 300)),          # row tiles 192 wide
    (513, 1152, 9001, (100, 256, 257, 512, 513)),
    (1000, 2048, 30011, (1, 255, 256, 257, 600, 769)),
    (2048, 4096, 3001, (64, 256, 1000, 1793, 2048)),
])
def test_counts_of_tokens_with_a_gradient(T, H, V, active, dtype):
    from verl_amd import _abi
    from verl_amd.utils.kernel import kernels

    lib = _abi.load()
    g = torch.Generator().manual_seed(T)
    h = torch.randn(T, H, generator=g).to(dtype).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(dtype).to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    base_lp, base_ent = torch.randn(T, generator=g).to(DEV), torch.randn(T, generator=g).to(DEV)
    _, _, mx, acc, eb = kernels.efficient_entropy_forward(h, w, y, 0, 1.0)
    code = _abi.dtype_code(dtype)
    need = lib.lce_backward_workspace_bytes(T, H, V, code, 0)
    ws = torch.empty(need + 4096, device=DEV, dtype=torch.uint8)
    for n in active:
        on = torch.zeros(T, dtype=torch.bool)
        on[torch.randperm(T, generator=g)[:n]] = True
        on = on.to(DEV)
        g_lp, g_ent = base_lp * on, base_ent * on
        ws[need:] = 0x5A
        dh = torch.empty_like(h)
        rc = lib.lce_backward(
            h.data_ptr(), H, w.data_ptr(), H, y.data_ptr(), T, H, V, code, 1.0, 0, mx.data_ptr(), acc.data_ptr(), eb.data_ptr(),
            g_lp.data_ptr(), g_ent.data_ptr(), dh.data_ptr(), None, ws.data_ptr(), need, 0, _abi.current_stream(h.device),
        )  # fmt: skip
        assert rc == 0
        dh32 = torch.empty(T, H, device=DEV)
        rc = lib.lce_backward_f32(
            h.data_ptr(), H, w.data_ptr(), H, y.data_ptr(), T, H, V, code, 1.0, 0, mx.data_ptr(), acc.data_ptr(), eb.data_ptr(),
            g_lp.data_ptr(), g_ent.data_ptr(), dh32.data_ptr(), None, ws.data_ptr(), need, 0, _abi.current_stream(h.device),
        )  # fmt: skip
        assert rc == 0
        want = check_tiles_part(dh32, None, g_lp, g_ent, h, w, y)[0]
        assert (ws[need:] == 0x5A).all()
        assert torch.count_nonzero(dh[~on]) == 0
        # the bar of the other backward tests: half an ulp of the result, 16-bit rounding of the logits' gradient
        assert ((dh.double() - want).abs() <= 2e-2 + 2.0**-7 * want.abs()).all(), n
