"""fp32 inputs with at most 255 tokens, the streaming kernels (csrc/few_tokens_f32.hpp): the largest row strides there are, with which the
rows of hidden span up to 4 GiB behind one buffer descriptor.  NaN stand between the rows: what is meant to read as zero (positions
without a token, columns beyond H) must lie beyond the last row, not between them."""

import pytest
import torch

from verl_amd import _abi

from test_gpu_fp32_few_edges import _inputs, _step

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
MOST = (1 << 22) - 4  # floats: just below 16 MiB


@pytest.mark.parametrize("T,ldh,share", [
    (128, MOST, 1.0),             # just below 2 GiB
    (129, MOST, 0.6),             # just beyond it
    (200, (1 << 29) // 200 // 4 * 4 + 4, 1.0),
    (255, MOST, 1.0),
    (255, MOST, 0.3),             # one group of positions
])  # fmt: skip
def test_largest_row_strides(T, ldh, share):
    lib = _abi.load()
    H, V = 160, 2003  # (H: columns of the last workgroup, and of its waves, that do not exist)
    h, w, y, g_lp, g_ent = _inputs(T, H, V, T)
    off = torch.rand(T, generator=torch.Generator().manual_seed(T)).to(DEV) >= share
    g_lp[off], g_ent[off] = 0, 0
    room = torch.full((T, ldh), float("nan"), device=DEV)
    room[:, :H] = h
    for a, b in zip(_step(lib, room[:, :H], w, y, g_lp, g_ent), _step(lib, h, w, y, g_lp, g_ent)):
        assert torch.equal(a, b) and bool(b.isfinite().all())
