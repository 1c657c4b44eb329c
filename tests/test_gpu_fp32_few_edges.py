"""fp32 inputs with at most 128 tokens, the streaming kernels (csrc/few_tokens_f32.hpp): row strides larger than H at the edges of
their token widths, and infinities and NaN against the tiles that run at larger sizes."""

import pytest
import torch

from verl_amd import _abi

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _step(lib, h, w, y, g_lp, g_ent, tau=0.9):
    """Forward and backward through the C ABI with the tensors' own row strides."""
    (T, H), V = h.shape, w.shape[0]
    code, st = _abi.DTYPE_F32, _abi.current_stream(h.device)
    out = torch.full((5, T), float("nan"), device=DEV)
    n = lib.lce_forward_workspace_bytes(T, H, V, code)
    ws = torch.full((n,), 0xFF, device=DEV, dtype=torch.uint8)  # (NaN)
    common = (h.data_ptr(), h.stride(0), w.data_ptr(), w.stride(0), y.data_ptr(), T, H, V, code, tau, 0)
    _abi.check(lib.lce_forward(*common, *(o.data_ptr() for o in out), ws.data_ptr(), n, st), "lce_forward")
    dh, dw = torch.full((T, H), 7.0, device=DEV), torch.full((V, H), 7.0, device=DEV)
    n = lib.lce_backward_workspace_bytes(T, H, V, code, 0)
    ws = torch.full((n,), 0xFF, device=DEV, dtype=torch.uint8)
    rc = lib.lce_backward(*common, *(o.data_ptr() for o in out[2:]), g_lp.data_ptr(), g_ent.data_ptr(), dh.data_ptr(), dw.data_ptr(), ws.data_ptr(), n, 0, st)
    _abi.check(rc, "lce_backward")
    return [*out, dh, dw]


def _inputs(T, H, V, seed):
    g = torch.Generator().manual_seed(seed)
    h = torch.randn(T, H, generator=g).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    return h, w, y, torch.randn(T, generator=g).to(DEV), torch.randn(T, generator=g).to(DEV)


@pytest.mark.parametrize("T", [1, 32, 33, 65, 96, 128])
def test_row_strides(T):
    """Rows apart, with NaN between them and behind the last one: the same bits as without."""
    lib = _abi.load()
    H, V = 384, 5003
    h, w, y, g_lp, g_ent = _inputs(T, H, V, T)
    g_lp[::3], g_ent[::3] = 0, 0  # (the backward gathers rows)

    def apart(x, more):
        room = torch.full((x.shape[0], x.shape[1] + more), float("nan"), device=DEV)
        room[:, : x.shape[1]] = x
        return room[:, : x.shape[1]]

    for a, b in zip(_step(lib, apart(h, 36), apart(w, 100), y, g_lp, g_ent), _step(lib, h, w, y, g_lp, g_ent)):
        assert torch.equal(a, b) and bool(b.isfinite().all())


@pytest.mark.parametrize("T,where", [(7, "weight -inf"), (64, "weight +inf"), (90, "weight NaN"), (128, "hidden inf"), (33, "last hidden NaN"),
                                     (128, "weight beyond bfloat16")])  # fmt: skip
def test_infinities_and_nan(T, where):
    """Finite exactly where the tiles' results are, and the same there.  (A logit of -inf leaves the entropy, 0 times -inf, NaN in
    whole blocks of 256 rows and finite in the last rows of a range, here and in the tiles: row 17 is in a whole block of
    either, the last row in a last one.)"""
    lib = _abi.load()
    H, V = 128, 70001
    h, w, y, g_lp, zero = _inputs(T, H, V, 5)
    zero.zero_()
    h[:, 5] = h[:, 5].abs() + 0.25  # one sign, so that an infinite weight gives logits of one sign
    y[3] = 17
    value = {"weight -inf": -float("inf"), "weight +inf": float("inf"), "weight NaN": float("nan"), "weight beyond bfloat16": -3.4e38}.get(where)
    if value is not None:
        w[17, 5] = w[V - 1, 5] = value
    elif where == "hidden inf":
        h[2, 3] = float("inf")
    else:
        h[T - 1, H - 1] = float("nan")
    got = _step(lib, h, w, y, g_lp, zero)
    try:
        assert lib.lce_set_variant(1) == 0
        want = _step(lib, h, w, y, g_lp, zero)
    finally:
        lib.lce_set_variant(-1)
    for a, b, what in zip(got, want, ["logprobs", "entropy", "maximum", "accumulate", "entropy_b", "d_hidden", "d_weight"]):
        assert torch.equal(a.isfinite(), b.isfinite()), f"{what}: {a.isfinite().sum()} of {a.numel()} finite, {b.isfinite().sum()} by the tiles"
        assert torch.equal(a.isnan(), b.isnan()), what
        ok = b.isfinite()
        # either side's sums are of fp32 products in an order of its own: 1e-5 in the 2-norm, as against float64
        assert ok.sum() == 0 or (a[ok] - b[ok]).norm() <= 1e-5 * b[ok].norm(), what
