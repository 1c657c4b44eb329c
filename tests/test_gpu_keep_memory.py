"""Kept logits are a saving, not a need: where there is no memory for them in the forward, or none for gradients and workspace beside
them in the backward, the step recomputes its logits, with the same bits."""

import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


class _Full:
    """torch.empty that fails, as the allocator would, for the calls that `fails` says."""

    def __init__(self, monkeypatch, fails):
        self.empty, self.fails, self.failed = torch.empty, fails, 0
        monkeypatch.setattr(torch, "empty", self)

    def __call__(self, *args, **kwargs):
        if self.fails(args, kwargs):
            self.failed += 1
            raise torch.cuda.OutOfMemoryError("out of memory (planted)")
        return self.empty(*args, **kwargs)


@pytest.mark.parametrize("T,H,V,dtype", [
    (100, 384, 20011, torch.bfloat16),
    (40, 384, 20011, torch.float32),    # streaming kernels
    (300, 512, 40011, torch.float32),   # planes
    (1024, 896, 60000, torch.float32),  # planes, part of the rows
])  # fmt: skip
def test_without_memory_for_the_logits(monkeypatch, T, H, V, dtype):
    mod = importlib.import_module("verl_amd.utils.kernel.linear_cross_entropy")
    g = torch.Generator().manual_seed(T)
    h = torch.randn(T, H, generator=g).to(dtype).to(DEV).requires_grad_(True)
    w = (torch.randn(V, H, generator=g) * 0.05).to(dtype).to(DEV).requires_grad_(True)
    y = torch.randint(0, V, (T,), generator=g).to(DEV)
    g_lp, g_ent = torch.randn(T, generator=g).to(DEV), torch.randn(T, generator=g).to(DEV)

    def grads(outs):
        return torch.autograd.grad(outs, (h, w), (g_lp, g_ent), retain_graph=True)

    before = mod.kept_logits_bytes(DEV)
    outs = mod.linear_cross_entropy(h, w, y, 0.9)
    size = mod.kept_logits_bytes(DEV) - before
    assert size > 0
    values, want = [o.detach() for o in outs], grads(outs)
    del outs
    assert mod.kept_logits_bytes(DEV) == before

    # the forward: the one allocation of that size
    with monkeypatch.context() as m:
        full = _Full(m, lambda args, kw: args == ((size,),) and kw.get("dtype") == torch.uint8)
        outs = mod.linear_cross_entropy(h, w, y, 0.9)
    assert full.failed == 1 and mod.kept_logits_bytes(DEV) == before
    assert all(torch.equal(a, b) for a, b in zip(outs, values))
    assert all(torch.equal(a, b) for a, b in zip(grads(outs), want))

    # the backward: gradients and workspace, while the logits are there
    outs = mod.linear_cross_entropy(h, w, y, 0.9)
    assert mod.kept_logits_bytes(DEV) - before == size
    torch.cuda.synchronize()
    held = torch.cuda.memory_allocated(DEV)
    with monkeypatch.context() as m:
        full = _Full(m, lambda args, kw: kw.get("dtype") == torch.uint8 and mod.kept_logits_bytes(DEV) > before)
        got = grads(outs)
    assert full.failed == 1
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    del got
    assert held - torch.cuda.memory_allocated(DEV) >= size and mod.kept_logits_bytes(DEV) == before
    assert all(torch.equal(a, b) for a, b in zip(grads(outs), want))  # (the graph is still whole)

    # without logits to give back it is the caller's error, as ever
    with monkeypatch.context() as m:
        _Full(m, lambda args, kw: kw.get("dtype") == torch.uint8)
        with pytest.raises(torch.cuda.OutOfMemoryError):
            grads(outs)
    del outs
    assert mod.kept_logits_bytes(DEV) == before
