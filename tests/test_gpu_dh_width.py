"""d_hidden as a launch of its own on tiles of 192 or 256 tokens, whichever fits the tokens with a gradient: counts at the edges of the
steps of 64 rows for which the width is chosen, on either side of what fits one width better; against the oracle, and nothing written
beyond the workspace."""

import pytest
import torch

from tiles_part import check_tiles_part

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,H,V,active", [
    (448, 896, 20011, (128, 129, 256, 257, 320, 384, 385, 448)),  # tiles of 224 hidden columns
    (1100, 512, 9001, (193, 300, 576, 577, 640, 960, 961, 1025, 1100)),
])
def test_counts_on_either_side_of_a_width(T, H, V, active, dtype):
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
        dh, dw = torch.empty_like(h), torch.empty_like(w)
        dh32, dw32 = (torch.empty(x.shape, device=DEV) for x in (h, w))
        for entry, a, b in ((lib.lce_backward, dh, dw), (lib.lce_backward_f32, dh32, dw32), (lib.lce_backward_f32, dh32, None)):
            ws[:need] = 0xFF  # (NaN)
            rc = entry(
                h.data_ptr(), H, w.data_ptr(), H, y.data_ptr(), T, H, V, code, 1.0, 0, mx.data_ptr(), acc.data_ptr(), eb.data_ptr(),
                g_lp.data_ptr(), g_ent.data_ptr(), a.data_ptr(), _abi.ptr(b), ws.data_ptr(), need, 0, _abi.current_stream(h.device),
            )  # fmt: skip
            assert rc == 0
            if entry is lib.lce_backward_f32:
                want, want_w = check_tiles_part(a, b, g_lp, g_ent, h, w, y)
        assert (ws[need:] == 0x5A).all()
        assert torch.count_nonzero(dh[~on]) == 0 and torch.count_nonzero(dh32[~on]) == 0
        # in 16 bits the same sums, rounded once: half an ulp, 2^-8 (2^-11) of the value, 2^-25 of fp16's smallest ones
        half = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
        assert ((dh.float() - dh32).abs() <= half * dh32.abs() + 2.0**-25).all(), n
        assert ((dw.double() - want_w).norm() / want_w.norm()).item() <= 2.0**-8, n
