"""fp32 on bfloat16 planes, forward (csrc/lce_terms.hpp): the chunks follow the workspace that is handed over.  From the least one
(what the library answers for LCE_DTYPE_F32) to the one it asks for, the values are the same and nothing is written behind it."""

import pytest
import torch

from oracle import lce_oracle as O
from verl_amd import _abi

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T,H,V", [(256, 5120, 60007), (257, 5120, 60007), (700, 5120, 60007), (300, 7168, 33000)])
def test_any_workspace_from_the_least_on(T, H, V):
    lib = _abi.load()
    g = torch.Generator(device=DEV).manual_seed(T)
    h = torch.randn(T, H, device=DEV, generator=g)
    w = torch.randn(V, H, device=DEV, generator=g).mul_(0.02)
    y = torch.randint(0, V, (T,), device=DEV, generator=g)
    least, full = (lib.lce_forward_workspace_bytes(T, H, V, code) for code in (_abi.DTYPE_F32, _abi.DTYPE_F32_PLANES))
    assert least < full
    ws = torch.empty(full + 4096, device=DEV, dtype=torch.uint8)
    outs = []
    for size in (full, (least + full) // 2, least):
        ws.fill_(0xA5)
        out = torch.full((5, T), float("nan"), device=DEV)
        rc = lib.lce_forward(h.data_ptr(), H, w.data_ptr(), H, y.data_ptr(), T, H, V, _abi.DTYPE_F32_PLANES, 1.0, 0, *(o.data_ptr() for o in out),
                             ws.data_ptr(), size, torch.cuda.current_stream().cuda_stream)  # fmt: skip
        _abi.check(rc, "lce_forward")
        assert bool((ws[size:] == 0xA5).all()), size
        outs.append(out)
    lp, ent = O.lce_forward(h, w, y, 1.0)
    torch.testing.assert_close(outs[0][0], lp, atol=1e-4, rtol=1e-5)  # (fp32 sums of some thousand products either side)
    torch.testing.assert_close(outs[0][1], ent, atol=1e-4, rtol=1e-5)
    for out in outs[1:]:
        assert torch.equal(out, outs[0])
