"""The workspace of the fp32 forward on bfloat16 planes (csrc/lce_terms.hpp): bounded by the weight, lowered by a budget, and a
call that has the least of it is served.  All checked on the host."""

import pytest
import torch

from verl_amd import _abi

MB = 1 << 20


def _planes_of_hidden(T, H):
    return (T + 63) // 64 * 64 * 6 * H


@pytest.mark.parametrize("T", [256, 257, 512, 513, 1000, 4096])
@pytest.mark.parametrize("H,V", [(896, 151936), (3584, 152064), (4096, 128256), (5120, 152064), (8192, 32000)])
def test_the_workspace_is_bounded_by_the_weight(T, H, V):
    lib = _abi.load()
    least, full = (lib.lce_forward_workspace_bytes(T, H, V, code) for code in (_abi.DTYPE_F32, _abi.DTYPE_F32_PLANES))
    rest = _planes_of_hidden(T, H) + 16 * T * ((V + 255) // 256 + 256) + MB  # + the partial statistics of every tile, and small change
    assert lib.lce_forward_workspace_bytes(T, H, V, _abi.DTYPE_BF16) < least <= full
    assert least <= 256 * MB + rest
    assert full <= max(256 * MB, V * H * 4 * 2 // 5) + rest


def test_a_budget_holds_it_and_the_least_is_enough():
    lib = _abi.load()
    T, H, V = 256, 5120, 152064
    least, full = (lib.lce_forward_workspace_bytes(T, H, V, code) for code in (_abi.DTYPE_F32, _abi.DTYPE_F32_PLANES))
    try:
        for budget in (1, 300 * MB, 600 * MB, 1 << 40):
            lib.lce_set_option(8, budget)
            assert least <= lib.lce_forward_workspace_bytes(T, H, V, _abi.DTYPE_F32_PLANES) <= min(full, max(least, budget))
            assert lib.lce_forward_workspace_bytes(T, H, V, _abi.DTYPE_F32) == least
    finally:
        lib.lce_set_option(8, 0)
    assert lib.lce_forward_workspace_bytes(T, H, V, _abi.DTYPE_F32_PLANES) == full
    room = torch.zeros(64)
    at = (room.data_ptr() + 15) // 16 * 16
    assert lib.lce_forward(at, H, at, H, at, T, H, V, _abi.DTYPE_F32_PLANES, 1.0, 0, at, at, at, at, at, at, least - 1, None) == -2
    assert f"{least - 1} < {least}".encode() in lib.lce_last_error()  # (the least is all that is asked for)
