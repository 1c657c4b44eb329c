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


def _forward(lib, code, entry, h, w, y, tau):
    """The five outputs of a forward through the C ABI, with a workspace as the code asks for, or the library's own."""
    from verl_amd import _abi

    (T, H), V = h.shape, w.shape[0]
    out = [torch.empty(T, device=DEV) for _ in range(5)]
    where = [o.data_ptr() for o in out]
    st = torch.cuda.current_stream().cuda_stream
    if entry == "static":
        rc = lib.lce_forward_static(h.data_ptr(), H, w.data_ptr(), H, y.data_ptr(), T, H, V, code, tau, 0, *where, st)
    else:
        n = lib.lce_forward_workspace_bytes(T, H, V, code)
        n = 8 << 20 if entry == "small" else n  # (what the fp32 MFMA needs: 256 splits of 512 tokens, 2.1 MB)
        ws = torch.empty(n, device=DEV, dtype=torch.uint8)
        rc = lib.lce_forward(h.data_ptr(), H, w.data_ptr(), H, y.data_ptr(), T, H, V, code, tau, 0, *where, ws.data_ptr(), n, st)
    _abi.check(rc, "forward")
    return out


def _backward(lib, code, h, w, y, tau, stats, g_lp, g_ent):
    from verl_amd import _abi

    (T, H), V = h.shape, w.shape[0]
    dh, dw = torch.empty_like(h), torch.empty_like(w)
    n = lib.lce_backward_workspace_bytes(T, H, V, code, 0)
    ws = torch.empty(n, device=DEV, dtype=torch.uint8)
    rc = lib.lce_backward(h.data_ptr(), H, w.data_ptr(), H, y.data_ptr(), T, H, V, code, tau, 0, *(s.data_ptr() for s in stats), g_lp.data_ptr(),
                          g_ent.data_ptr(), dh.data_ptr(), dw.data_ptr(), ws.data_ptr(), n, 0, torch.cuda.current_stream().cuda_stream)
    _abi.check(rc, "lce_backward")
    return dh, dw


@pytest.mark.parametrize("std", [0.1, 0.3])
def test_statistics_and_logits_come_from_the_same_arithmetic(std):
    """The backward recomputes the logits: where a distribution is peaked, their rounding errors cancel against those of the
    forward's statistics only if both were taken the same way.  The fp32 code takes the fp32 MFMA both ways, whatever
    workspace the forward had; the other one the planes both ways, whatever was set between the two calls.  The bound is
    relative: mixing the two doubles the largest error at least (printed), statistics that differ in the last bits of
    their sums, or another order of the chunks, move it by a few per cent."""
    from verl_amd import _abi
    from verl_amd.utils.kernel import kernels

    lib = _abi.load()
    T, H, V, tau = 512, 1024, 40960, 0.6
    g = torch.Generator().manual_seed(1)
    h = torch.randn(T, H, generator=g).to(DEV)
    w = (torch.randn(V, H, generator=g) * std).to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    g_lp, g_ent = (torch.randn(T, generator=g).to(DEV) for _ in range(2))
    want, _ = O.lce_backward(g_lp, g_ent, h, w, y, tau, compute_dtype=torch.float64)
    worst = {}
    stats = {"full": _forward(lib, _abi.DTYPE_F32, "full", h, w, y, tau)[2:], "static": _forward(lib, _abi.DTYPE_F32, "static", h, w, y, tau)[2:],
             "small": _forward(lib, _abi.DTYPE_F32, "small", h, w, y, tau)[2:], "planes": _forward(lib, _abi.DTYPE_F32_PLANES, "full", h, w, y, tau)[2:]}
    for name, code in (("full", _abi.DTYPE_F32), ("static", _abi.DTYPE_F32), ("small", _abi.DTYPE_F32), ("planes", _abi.DTYPE_F32_PLANES)):
        dh, _ = _backward(lib, code, h, w, y, tau, stats[name], g_lp, g_ent)
        worst[name] = ((dh.double() - want).abs().max() / want.abs().max()).item()
    _, _, *kept = kernels.efficient_entropy_forward(h, w, y, 0, tau)
    kernels.set_workspace_budget(64 << 20)  # (less than the smallest workspace of the planes here, 71 MB)
    try:
        dh, _ = kernels.efficient_entropy_backward(g_lp, g_ent, h, w, y, *kept, 0, False, tau)
    finally:
        kernels.set_workspace_budget(0)
    worst["budget"] = ((dh.double() - want).abs().max() / want.abs().max()).item()
    for a, b in (("static", "planes"), ("planes", "full")):  # (for the record: the two mixtures)
        dh, _ = _backward(lib, _abi.DTYPE_F32_PLANES if a == "static" else _abi.DTYPE_F32, h, w, y, tau, stats[a], g_lp, g_ent)
        print(f"std {std}: statistics of {a}, logits of {b}: {((dh.double() - want).abs().max() / want.abs().max()).item():.2e}")
    print(f"std {std}:", {k: f"{v:.2e}" for k, v in worst.items()})
    assert max(worst["static"], worst["small"]) < 1.2 * worst["full"] and worst["budget"] < 1.2 * worst["planes"], worst
    assert worst["planes"] < 1.2 * worst["full"], worst


@pytest.mark.parametrize("where", ["weight -inf", "weight +inf", "weight NaN", "weight beyond bfloat16", "hidden inf", "last hidden -inf"])
def test_infinities_and_values_beyond_bfloat16(where):
    """An infinity, and a finite value beyond the largest bfloat16, in either operand: what the planes make of it is finite
    exactly where the fp32 MFMA's result is, and the same there.  (A weight of -inf whose logit comes out as -inf leaves the
    other rows' log-probs alone; a token with an infinity spoils its own values only.)"""
    from verl_amd import _abi

    lib = _abi.load()
    T, H, V, tau = 300, 128, 40011, 0.8
    assert lib.lce_forward_workspace_bytes(T, H, V, _abi.DTYPE_F32_PLANES) > lib.lce_forward_workspace_bytes(T, H, V, _abi.DTYPE_BF16)
    g = torch.Generator().manual_seed(2)
    h = torch.randn(T, H, generator=g).to(DEV)
    w = (torch.randn(V, H, generator=g) * 0.05).to(DEV)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    h[:, 5] = h[:, 5].abs() + 0.25  # one sign, so that an infinite weight gives logits of one sign
    h[:7, 5] = torch.tensor([1.0, 0.5, 2.0, 1.5, 3.0, 300.0, 299.7])  # (without small terms; large ones)
    y[3] = 17
    value = {"weight -inf": -float("inf"), "weight +inf": float("inf"), "weight NaN": float("nan"), "weight beyond bfloat16": -3.4e38}.get(where)
    if value is not None:
        w[17, 5] = w[V - 1, 5] = value
    elif where == "hidden inf":
        h[7, 3] = float("inf")
    else:
        h[T - 1, H - 1] = -float("inf")
    g_lp, zero = torch.randn(T, generator=g).to(DEV), torch.zeros(T, device=DEV)

    def same(a, b, what, rel):
        assert torch.equal(a.isfinite(), b.isfinite()), f"{what}: {a.isfinite().sum()} of {a.numel()} values are finite, {b.isfinite().sum()} on the fp32 MFMA"
        ok = b.isfinite()
        if ok.any():
            assert (a[ok] - b[ok]).norm() <= rel * b[ok].norm(), what
        return int(ok.sum())

    both = []
    for code in (_abi.DTYPE_F32_PLANES, _abi.DTYPE_F32):
        out = _forward(lib, code, "full", h, w, y, tau)
        both.append(out + list(_backward(lib, code, h, w, y, tau, out[2:], g_lp, zero)))
    # 2-norm, relative: the two ways round a logit differently, by some 2^-24 of its size, and the gradients of a token follow its
    # logits' absolute error; the largest logits here are about 300 x 0.05 x 4 / 0.8
    rel = 8 * 75 * 2.0**-24
    finite = [same(a, b, what, rel) for a, b, what in zip(*both, ["logprobs", "entropy", "maximum", "accumulate", "entropy_b", "d_hidden", "d_weight"])]
    if where in ("weight -inf", "weight beyond bfloat16"):
        assert finite[0] >= T - 1
    elif where.endswith("inf") and "hidden" in where:
        assert finite[0] == T - 1
