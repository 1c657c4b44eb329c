"""fp32 inputs with 129 to 255 tokens, two groups of positions through the streaming kernels (csrc/lce_few_f32.hpp), with what the first
group alone is tested with: row strides larger than H, workspaces of NaN, infinities and NaN, shards of the vocabulary, the forward on
the library's own scratch buffer and on the least workspace that is taken."""

import pytest
import torch

from oracle import lce_oracle as O
from verl_amd import _abi

from test_gpu_fp32_few_edges import _inputs, _step

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# two kinds of fp32 sums of H products of unit size times 0.05, in an order each of its own, and differences of numbers around max |logit|
TOL = dict(atol=1e-5, rtol=1e-5)


@pytest.mark.parametrize("T", [129, 160, 161, 192, 193, 224, 255])
@pytest.mark.parametrize("with_gradient", ["two of three", "the first 100", "none of the first 128"])
def test_row_strides(T, with_gradient):
    """Rows apart, with NaN between them and behind the last one: the same bits as without."""
    lib = _abi.load()
    H, V = 384, 5003
    h, w, y, g_lp, g_ent = _inputs(T, H, V, T)
    off = {"two of three": slice(None, None, 3), "the first 100": slice(100, None), "none of the first 128": slice(0, 128)}[with_gradient]
    g_lp[off], g_ent[off] = 0, 0

    def apart(x, more):
        room = torch.full((x.shape[0], x.shape[1] + more), float("nan"), device=DEV)
        room[:, : x.shape[1]] = x
        return room[:, : x.shape[1]]

    for a, b in zip(_step(lib, apart(h, 36), apart(w, 100), y, g_lp, g_ent), _step(lib, h, w, y, g_lp, g_ent)):
        assert torch.equal(a, b) and bool(b.isfinite().all())


@pytest.mark.parametrize("T,where", [(129, "weight -inf"), (160, "weight +inf"), (200, "weight NaN"), (255, "hidden inf"), (255, "last hidden NaN"),
                                     (140, "first hidden NaN"), (193, "weight beyond bfloat16")])  # fmt: skip
def test_infinities_and_nan(T, where):
    """Finite exactly where the tiles' results are, and the same there: a token of one group leaves the other group's alone."""
    lib = _abi.load()
    H, V = 128, 70001
    h, w, y, g_lp, zero = _inputs(T, H, V, 5)
    zero.zero_()
    h[:, 5] = h[:, 5].abs() + 0.25  # one sign, so that an infinite weight gives logits of one sign
    y[3] = y[T - 1] = 17
    value = {"weight -inf": -float("inf"), "weight +inf": float("inf"), "weight NaN": float("nan"), "weight beyond bfloat16": -3.4e38}.get(where)
    if value is not None:
        w[17, 5] = w[V - 1, 5] = value
    elif where == "hidden inf":
        h[2, 3] = h[130, 3] = float("inf")
    elif where == "last hidden NaN":
        h[T - 1, H - 1] = float("nan")
    else:
        h[0, 0] = float("nan")
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


def _forward(lib, h, w, y, reduction, size=None, static=False):
    """`size`: bytes of the workspace (None: what the query answers); behind them a guard."""
    (T, H), V = h.shape, w.shape[0]
    code, st = _abi.DTYPE_F32, _abi.current_stream(h.device)
    out = torch.full((5, T), float("nan"), device=DEV)
    args = (h.data_ptr(), H, w.data_ptr(), H, y.data_ptr(), T, H, V, code, 0.9, reduction, *(o.data_ptr() for o in out))
    if static:
        return lib.lce_forward_static(*args, st), out
    n = lib.lce_forward_workspace_bytes(T, H, V, code) if size is None else size
    ws = torch.full((n + 4096,), 0xFF, device=DEV, dtype=torch.uint8)
    rc = lib.lce_forward(*args, ws.data_ptr(), n, st)
    assert (ws[n:] == 0xFF).all()
    return rc, out


@pytest.mark.parametrize("T,H,V", [(129, 128, 300), (160, 384, 20011), (255, 256, 40003)])
@pytest.mark.parametrize("reduction", ["none", "mean"])
def test_the_least_workspace_and_the_built_in_one(T, H, V, reduction):
    """What the fp32 MFMA itself needs is what LCE_DTYPE_BF16 is answered: fewer splits of the vocabulary, the same values."""
    lib = _abi.load()
    h, w, y, _, _ = _inputs(T, H, V, T)
    mode = 0 if reduction == "none" else 2
    least, full = (lib.lce_forward_workspace_bytes(T, H, V, code) for code in (_abi.DTYPE_BF16, _abi.DTYPE_F32))
    assert least <= full
    rc, want = _forward(lib, h, w, y, mode)
    _abi.check(rc, "lce_forward")
    lp, ent = O.lce_forward(h, w, y, 0.9, reduction, compute_dtype=torch.float64)
    n = T if mode == 0 else 1
    torch.testing.assert_close(want[0, :n].double(), lp.double().reshape(-1), **TOL)
    torch.testing.assert_close(want[1].double(), ent, **TOL)
    for size, static in ((least, False), ((least + full) // 2 + 40, False), (None, True)):
        rc, got = _forward(lib, h, w, y, mode, size, static)
        _abi.check(rc, "lce_forward")
        torch.testing.assert_close(got[0, :n], want[0, :n], **TOL)
        torch.testing.assert_close(got[1:], want[1:], **TOL)
    rc, _ = _forward(lib, h, w, y, mode, least - 1)
    assert rc == -2 and b"workspace too small" in lib.lce_last_error()


@pytest.mark.parametrize("T", [129, 200, 255])
@pytest.mark.parametrize("reduction", ["none", "mean"])
def test_shards(T, reduction):
    """The vocabulary in three uneven shards against float64 and against the call on the whole of it."""
    from verl_amd.utils.kernel import kernels
    from verl_amd.utils.kernel import vocab_parallel as VP

    H, V, tau = 256, 6007, 0.8
    h, w, y, g_lp, g_ent = _inputs(T, H, V, T)
    if reduction == "mean":
        g_lp = torch.tensor(0.6, device=DEV)
    shards = [(0, 1003), (1003, 1030), (1030, V)]
    partials = torch.stack([VP.shard_forward(h, w[a:b].contiguous(), y, a, tau) for a, b in shards])
    lp, ent, mx, acc, eb = VP.merge_shards(partials, reduction)
    whole = kernels.efficient_entropy_forward(h, w, y, kernels.get_entropy_reduction_enum_number(reduction), tau)
    for a, b in zip((lp, ent, mx, acc, eb), whole):
        torch.testing.assert_close(a, b, **TOL)
    rlp, rent = O.lce_forward(h, w, y, tau, reduction, compute_dtype=torch.float64)
    torch.testing.assert_close(lp.double(), rlp, **TOL)
    torch.testing.assert_close(ent.double(), rent, **TOL)
    dh, dws = torch.zeros(T, H, device=DEV), []
    for a, b in shards:
        dh_r, dw_r = VP.shard_backward(g_lp, g_ent, h, w[a:b].contiguous(), y, a, mx, acc, eb, reduction, tau)
        dh += dh_r
        dws.append(dw_r)
    rdh, rdw = O.lce_backward(g_lp, g_ent, h, w, y, tau, reduction, compute_dtype=torch.float64)
    for got, want in ((dh, rdh), (torch.cat(dws), rdw)):
        assert ((got.double() - want).norm() / want.norm()).item() <= 6e-6  # (the bar of the other fp32 tests)
