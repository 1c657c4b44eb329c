"""Fused PPO actor loss on the fused head's outputs.

One HIP pass computes what the reference assembles from ``compute_policy_loss_vanilla`` + ``agg_loss``, ``kl_penalty``
and the entropy and KL terms of ``ppo_loss`` (``verl/trainer/ppo/core_algos.py:1140-1206,1286-1376,2188-2251``,
``verl/workers/utils/losses.py:57-155``) for the vanilla loss under any of ``agg_loss``'s aggregation modes, together
with the gradients w.r.t. ``log_prob`` and ``entropy``, so the backward of ``linear_cross_entropy`` starts from two
ready vectors instead of an elementwise autograd graph.  Metric names are the reference's.
"""

from __future__ import annotations

import ctypes
from typing import Optional

import torch

from ... import _abi


AGG_MODES = {
    "token-mean": 0,
    "token-sum": 1,
    "seq-mean-token-sum": 2,
    "seq-mean-token-sum-norm": 3,
    "seq-mean-token-mean": 4,
}

# kl_penalty's estimators (core_algos.py:2228-2245); a trailing "+" selects the straight-through variant (:2201-2213)
KL_TYPES = {"kl": 1, "k1": 1, "abs": 2, "mse": 3, "k2": 3, "low_var_kl": 4, "k3": 4}
KL_STRAIGHT_THROUGH = 16


def kl_type_number(kl_penalty: str) -> int:
    base = kl_penalty[:-1] if kl_penalty.endswith("+") else kl_penalty
    if base not in KL_TYPES:
        raise NotImplementedError(f"kl_penalty {kl_penalty!r}")  # core_algos.py:2247-2251 ("full" included)
    return KL_TYPES[base] | (KL_STRAIGHT_THROUGH if kl_penalty.endswith("+") else 0)


def agg_numbers(loss_agg_mode, dp_size, batch_num_tokens, global_batch_size, loss_scale_factor):
    """agg_loss's arguments as the C ABI takes them; raises what the reference raises (core_algos.py:1172-1204)."""
    if loss_agg_mode not in AGG_MODES:
        raise ValueError(f"Invalid loss_agg_mode: {loss_agg_mode}")
    if dp_size > 1:
        if loss_agg_mode == "token-mean" and batch_num_tokens is None:
            raise ValueError("(global) batch_num_tokens is required when dp_size > 1")
        if loss_agg_mode.startswith("seq-mean") and global_batch_size is None:
            raise ValueError("global_batch_size is required when dp_size > 1")
    return (
        AGG_MODES[loss_agg_mode],
        float(dp_size),
        -1.0 if batch_num_tokens is None else float(batch_num_tokens),
        -1.0 if global_batch_size is None else float(global_batch_size),
        -1.0 if loss_scale_factor is None else float(loss_scale_factor),
    )


MASK_F32, MASK_U8, MASK_I32, MASK_I64, MASK_F32_NONZERO = range(5)
_INT_MASKS = {torch.bool: MASK_U8, torch.uint8: MASK_U8, torch.int32: MASK_I32, torch.int64: MASK_I64}


def _f32(t, numel):
    """``t`` as a contiguous fp32 vector of ``numel`` elements (itself where it is one)."""
    if t is None:
        return None
    if t.dtype != torch.float32:
        t = t.to(torch.float32)
    assert t.numel() == numel, "all inputs have the shape of log_prob"
    return t if t.is_contiguous() else t.contiguous()


class _Packed:
    """Packed model outputs: where the lengths of prompts and responses come from.  Either both vectors, or the attention
    mask of a padded batch (its first ``prompt_width`` columns are the prompts'), from which the kernel counts them."""

    __slots__ = ("prompt_lens", "response_lens", "attention_mask", "prompt_width", "_pending")

    def __init__(self, prompt_lens=None, response_lens=None, attention_mask=None, prompt_width=0):
        self.prompt_lens, self.response_lens = prompt_lens, response_lens
        self.attention_mask, self.prompt_width = attention_mask, prompt_width
        self._pending = None  # (call, stream, ticket) of the forward

    def launched(self, call, stream, ticket):
        self._pending = (call, stream, ticket)

    def checks(self):
        """(sum of all lengths, prompts of length 0, longest response) of the forward that has been launched: waits for the
        kernel that adds them up.  Once per forward, whatever happens in between."""
        (call, stream, ticket), self._pending = self._pending, None
        _abi.check(_abi.load().lce_ppo_forward_end(ctypes.addressof(call), stream, ticket), "lce_ppo_forward_end")
        return tuple(call.checks)

    def __del__(self):
        if self._pending is not None:  # (an exception kept the caller from asking)
            self.checks()


_POINTERS = _abi.PpoCall.total_nnz.offset  # bytes of the call that are addresses

# a tensor that stands for a batch of them: what autograd hands a backward under is_grads_batched, and what vmap does
_is_legacy_batched = torch._C._functorch.is_legacy_batchedtensor
_is_wrapped = torch._C._functorch.is_functorch_wrapped_tensor


class _FusedPPOLoss(torch.autograd.Function):
    """``log_prob`` may be None: then the call is ``agg_loss`` of ``entropy`` (the C ABI's aggregation-only form).
    ``packed`` (a ``_Packed``): ``log_prob`` / ``entropy`` are ``[total_nnz]`` over the packed sequences, everything else is
    ``[batch, max_response_len]``.  ``nonzero_mask``: every non-zero element of the mask counts 1."""

    @staticmethod
    def forward(ctx, log_prob, entropy, old_log_prob, advantages, response_mask, is_weights, ref_log_prob, agg, kl,
                clip_low, clip_high, clip_c, entropy_coeff, packed=None, nonzero_mask=False):
        lead = log_prob if log_prob is not None else entropy
        assert lead.is_cuda, "fused_ppo_loss runs on the GPU only"
        dev = lead.device
        total = lead.numel()
        if packed is None:
            # rows are the sequences the seq-mean modes average over: the last dimension is the response
            row_len = lead.shape[-1] if lead.dim() >= 1 else 1
            rows = total // row_len if row_len else 0
            n = total
        else:
            rows, row_len = response_mask.shape
            n = rows * row_len
        lp, ent = _f32(log_prob, total), _f32(entropy, total)
        old, adv = _f32(old_log_prob, n), _f32(advantages, n)
        isw, ref = _f32(is_weights, n), _f32(ref_log_prob, n)
        mask_kind = _INT_MASKS.get(response_mask.dtype) if nonzero_mask or response_mask.dtype == torch.bool else None
        if mask_kind is not None:
            assert response_mask.numel() == n, "all inputs have the shape of log_prob"
            mask = response_mask.contiguous()
        elif nonzero_mask and response_mask.dtype != torch.float32:
            mask, mask_kind = response_mask.to(torch.bool).contiguous(), MASK_U8
        else:
            mask, mask_kind = _f32(response_mask, n), MASK_F32_NONZERO if nonzero_mask else MASK_F32
        call = _abi.PpoCall()
        call.mask_kind = mask_kind
        call.agg_mode, call.dp_size, call.batch_num_tokens, call.global_batch_size, call.loss_scale_factor = agg
        call.kl_type, call.kl_coef = kl
        call.clip_low, call.clip_high, call.clip_c, call.entropy_coeff = clip_low, clip_high, clip_c, entropy_coeff
        call.rows, call.row_len, call.total_nnz = rows, row_len, -1 if packed is None else total
        lib = _abi.load()
        call.workspace_bytes = lib.lce_ppo_loss_workspace_bytes(rows, row_len)
        # one allocation: workspace, the unscaled gradients, and the lengths of a packed batch
        grad_bytes = (total * 4 + 255) // 256 * 256
        count_lens = packed is not None and packed.attention_mask is not None
        keep = torch.empty(call.workspace_bytes + 2 * grad_bytes + (16 * rows if count_lens else 0), device=dev, dtype=torch.uint8)
        out = torch.empty(16, device=dev, dtype=torch.float32)
        at = keep.data_ptr()
        call.workspace, call.out = at, out.data_ptr()
        at += call.workspace_bytes
        call.g_log_prob = at if lp is not None else None
        call.g_entropy = at + grad_bytes if ent is not None else None
        at += 2 * grad_bytes
        ptr = _abi.ptr
        call.log_prob, call.entropy, call.old_log_prob, call.advantages = ptr(lp), ptr(ent), ptr(old), ptr(adv)
        call.mask, call.is_weights, call.ref_log_prob = mask.data_ptr(), ptr(isw), ptr(ref)
        lens = ()
        if count_lens:
            am = packed.attention_mask
            call.attention_mask, call.attention_kind = am.data_ptr(), _INT_MASKS[am.dtype]
            call.attention_stride = am.stride(0) if rows > 1 else am.shape[1]  # (a single row's stride means nothing)
            call.prompt_width, call.attention_width = packed.prompt_width, am.shape[1]
            call.prompt_lens, call.response_lens = at, at + 8 * rows
        elif packed is not None:
            lens = (packed.prompt_lens, packed.response_lens)
            call.prompt_lens, call.response_lens = lens[0].data_ptr(), lens[1].data_ptr()
        with _abi.on_device(dev):
            stream = _abi.current_stream(dev)
            if packed is None:
                _abi.check(lib.lce_ppo_forward(ctypes.addressof(call), stream), "lce_ppo_forward")
            else:
                ticket = ctypes.c_void_p()
                _abi.check(lib.lce_ppo_forward_begin(ctypes.addressof(call), stream, ctypes.addressof(ticket)), "lce_ppo_forward_begin")
                packed.launched(call, stream, ticket)
        ctx.save_for_backward(keep, *lens)
        ctx.set_materialize_grads(False)  # (the vector of statistics takes no gradient: no zeros are made for it)
        # for the backward: the numbers of the call, and where in the buffer things are (which may be elsewhere by then); no address
        ctx.numbers = _abi.PpoCall.from_buffer_copy(call)
        ctypes.memset(ctypes.addressof(ctx.numbers), 0, _POINTERS)
        ctx.parts = (call.workspace_bytes, grad_bytes, count_lens)
        ctx.like = tuple(None if t is None else (t.shape, t.dtype) for t in (log_prob, entropy))
        ctx.mark_non_differentiable(out)
        return out[0], out

    @staticmethod
    def backward(ctx, g_loss, _g_out):
        if g_loss is None:
            return (None,) * 15
        keep, *lens = ctx.saved_tensors
        dev = keep.device
        assert keep.is_cuda and g_loss.device == dev, "the loss's saved tensors are on another device"
        at = keep.data_ptr()
        if at % 16:  # (a saved-tensor hook may bring it back anywhere)
            keep = keep.clone()
            at = keep.data_ptr()
        # An upstream gradient that is itself differentiated (create_graph) or stands for a batch of them (is_grads_batched)
        # is multiplied on by torch; otherwise the kernel reads it where it is.
        traced = (g_loss.requires_grad and torch.is_grad_enabled()) or _is_legacy_batched(g_loss) or _is_wrapped(g_loss)
        if traced:
            up = torch.ones((), device=dev, dtype=torch.float32)
        else:
            up = g_loss if g_loss.dtype == torch.float32 else g_loss.to(torch.float32)
        call = _abi.PpoCall.from_buffer_copy(ctx.numbers)
        ws_bytes, grad_bytes, count_lens = ctx.parts
        call.workspace, call.g_log_prob, call.g_entropy = at, at + ws_bytes, at + ws_bytes + grad_bytes
        if count_lens:
            at += ws_bytes + 2 * grad_bytes
            call.prompt_lens, call.response_lens = at, at + 8 * call.rows
        elif lens:
            assert lens[0].device == lens[1].device == dev, "the loss's saved tensors are on another device"
            call.prompt_lens, call.response_lens = lens[0].data_ptr(), lens[1].data_ptr()
        grads = [
            torch.empty(like[0], device=dev, dtype=torch.float32) if like is not None and ctx.needs_input_grad[k] else None
            for k, like in enumerate(ctx.like)
        ]
        call.g_loss, call.d_log_prob, call.d_entropy = up.data_ptr(), _abi.ptr(grads[0]), _abi.ptr(grads[1])
        with _abi.on_device(dev):
            _abi.check(_abi.load().lce_ppo_backward(ctypes.addressof(call), _abi.current_stream(dev)), "lce_ppo_backward")
        if traced:
            grads = [g if g is None else g * g_loss for g in grads]
        d = [g if g is None or g.dtype == like[1] else g.to(like[1]) for g, like in zip(grads, ctx.like)]
        return (*d,) + (None,) * 13


def fused_ppo_loss(
    log_prob: torch.Tensor,
    entropy: Optional[torch.Tensor],
    old_log_prob: torch.Tensor,
    advantages: torch.Tensor,
    response_mask: torch.Tensor,
    clip_ratio: float = 0.2,
    clip_ratio_low: Optional[float] = None,
    clip_ratio_high: Optional[float] = None,
    clip_ratio_c: float = 3.0,
    entropy_coeff: float = 0.0,
    loss_agg_mode: str = "token-mean",
    dp_size: int = 1,
    batch_num_tokens: Optional[int] = None,
    global_batch_size: Optional[int] = None,
    loss_scale_factor: Optional[int] = None,
    rollout_is_weights: Optional[torch.Tensor] = None,
    ref_log_prob: Optional[torch.Tensor] = None,
    kl_loss_coef: float = 0.001,
    kl_loss_type: str = "low_var_kl",
    _packed=None,
    _nonzero_mask=False,
):
    """Returns ``(policy_loss, metrics)``: ``policy_loss = pg_loss - entropy_coeff * entropy_loss
    [+ kl_loss_coef * kl_loss]`` (a 0-dim tensor with autograd), ``metrics`` a dict of 0-dim tensors under the
    reference's keys (no host sync is forced).
    ``dp_size``, ``batch_num_tokens``, ``global_batch_size`` and ``loss_scale_factor`` are ``agg_loss``'s
    (``core_algos.py:1140-1206``); the sequences of the ``seq-mean-*`` modes are the rows of the last dimension.
    ``rollout_is_weights`` multiplies the per-token policy loss (``core_algos.py:1362-1363``) and takes no gradient.
    With ``ref_log_prob`` the KL penalty of ``ppo_loss`` (``use_kl_loss``, ``losses.py:142-153``) is added:
    ``kl_loss_type`` is ``kl_penalty``'s estimator name, ``kl_loss_coef`` its weight."""
    agg = agg_numbers(loss_agg_mode, dp_size, batch_num_tokens, global_batch_size, loss_scale_factor)
    assert clip_ratio_c > 1.0, f"clip_ratio_c must be greater than 1.0, got {clip_ratio_c}"
    lo = clip_ratio if clip_ratio_low is None else clip_ratio_low
    hi = clip_ratio if clip_ratio_high is None else clip_ratio_high
    kl = (0, 0.0) if ref_log_prob is None else (kl_type_number(kl_loss_type), float(kl_loss_coef))
    loss, out = _FusedPPOLoss.apply(
        log_prob, entropy, old_log_prob, advantages, response_mask, rollout_is_weights, ref_log_prob, agg, kl,
        float(lo), float(hi), float(clip_ratio_c), float(entropy_coeff), _packed, _nonzero_mask,
    )  # fmt: skip
    _, pg_loss, entropy_loss, clipfrac, ppo_kl, clipfrac_lower, _, _, kl_loss, *_ = out.unbind()
    metrics = {
        "actor/pg_loss": pg_loss,
        "actor/pg_clipfrac": clipfrac,
        "actor/ppo_kl": ppo_kl,
        "actor/pg_clipfrac_lower": clipfrac_lower,
    }
    if entropy is not None:
        metrics["actor/entropy_loss"] = entropy_loss
    if ref_log_prob is not None:
        metrics["kl_loss"] = kl_loss
        metrics["kl_coef"] = kl_loss_coef
    return loss, metrics


def response_slices(prompt_lens: torch.Tensor, response_lens: torch.Tensor, total_nnz: int):
    """``(start, length)`` per sequence of the response slice that ``no_padding_2_padding`` takes out of a packed model
    output (``verl/workers/utils/padding.py:97-141``), what ``lce_ppo_loss_packed`` takes: ``start`` = end of the sequence -
    response length - 1 (the left shift by one token), with the reference's two assertions.  ``ppo_loss`` and
    ``fused_ppo_loss_packed`` have their kernels add the lengths up instead."""
    prompt_lens, response_lens = prompt_lens.to(torch.int64), response_lens.to(torch.int64)
    ends = (prompt_lens + response_lens).cumsum(dim=0)
    assert ends[-1].item() == total_nnz
    assert not prompt_lens.eq(0).any(), f"seq_offset - resp_len - 1 assumes prompt_len > 0. Got {prompt_lens}"
    return (ends - response_lens - 1).contiguous(), response_lens.contiguous()


def _check_lengths(checks, total_nnz, width):
    """The reference's two assertions on a packed batch (``verl/workers/utils/padding.py:126-128``) and the padded width's,
    on the sums that the kernel reports."""
    total, empty_prompts, longest = checks
    assert total == total_nnz, f"prompt and response lengths add up to {total}, the packed outputs hold {total_nnz} tokens"
    assert empty_prompts == 0, f"seq_offset - resp_len - 1 assumes prompt_len > 0. Got {empty_prompts} empty prompts"
    assert longest <= width, "a response is longer than max_response_len"


def fused_ppo_loss_packed(
    log_prob: torch.Tensor,
    entropy: Optional[torch.Tensor],
    prompt_lens: torch.Tensor,
    response_lens: torch.Tensor,
    old_log_prob: torch.Tensor,
    advantages: torch.Tensor,
    response_mask: torch.Tensor,
    **kwargs,
):
    """``fused_ppo_loss`` for the no-padding engines: ``log_prob`` / ``entropy`` are the fused head's outputs over the
    PACKED sequences, ``[total_nnz]``; ``prompt_lens`` / ``response_lens`` ``[batch]`` (integer tensors on the device);
    ``old_log_prob``, ``advantages``, ``response_mask`` (and ``rollout_is_weights``, ``ref_log_prob``) stay
    ``[batch, max_response_len]`` as the data batch holds them.  The kernel applies the response slice of
    ``no_padding_2_padding`` (``verl/workers/utils/padding.py:97-141``) while it reads, and the gradients flow back in
    packed order, so the backward of ``linear_cross_entropy`` starts from them without a gather or a scatter.
    Same keyword arguments, return values and metrics as ``fused_ppo_loss``."""
    assert log_prob.dim() == 1 and (entropy is None or entropy.shape == log_prob.shape), "packed outputs are [total_nnz]"
    assert response_mask.dim() == 2 and old_log_prob.shape == response_mask.shape == advantages.shape
    assert prompt_lens.shape == response_lens.shape == (response_mask.shape[0],)
    dev = log_prob.device
    packed = _Packed(prompt_lens.to(dev, torch.int64).contiguous(), response_lens.to(dev, torch.int64).contiguous())
    result = fused_ppo_loss(log_prob, entropy, old_log_prob, advantages, response_mask, _packed=packed, **kwargs)
    # (the lengths are checked while the loss is on its way: the launches stay inside their buffers whatever they say)
    _check_lengths(packed.checks(), log_prob.numel(), response_mask.shape[1])
    return result


def _cfg(config, name, default=None):
    """``config.name`` or ``config[name]``: the reference's configs are dataclasses that also answer ``.get``."""
    if isinstance(config, dict):
        return config.get(name, default)
    if hasattr(config, name):
        return getattr(config, name)
    return config.get(name, default) if hasattr(config, "get") else default


def _get(data, key, default=None):
    try:
        return data[key]
    except KeyError:
        return default


def _has(data, key) -> bool:
    try:
        return key in data
    except TypeError:
        return _get(data, key) is not None


def batch_lens(data):
    """``(prompt_lens, response_lens)`` of a data batch the way ``no_padding_2_padding`` reads them
    (``verl/workers/utils/padding.py:110-124``): from the offsets of nested ``prompts`` / ``responses``, or from the
    two halves of ``attention_mask`` when the batch is padded."""
    prompts, responses = data["prompts"], data["responses"]
    if prompts.is_nested:
        return prompts.offsets().diff(), responses.offsets().diff()
    attention_mask = data["attention_mask"]
    assert not attention_mask.is_nested
    P = prompts.shape[1]
    return attention_mask[:, :P].sum(dim=1), attention_mask[:, P:].sum(dim=1)


def _packed_lengths(data, dev) -> _Packed:
    """``batch_lens`` for the kernel, one pair of lengths per response: a padded batch's mask of integers on ``dev`` is
    counted by the loss's own launches."""
    rows = data["responses"].shape[0]
    if not data["prompts"].is_nested:
        mask, P = data["attention_mask"], data["prompts"].shape[1]
        if not mask.is_nested and mask.dtype in _INT_MASKS and mask.device == dev and mask.dim() == 2 and mask.shape[1] >= P:
            assert mask.shape[0] == rows, f"{mask.shape[0]} rows of the attention mask for {rows} responses"
            # (the kernel takes rows of neighbouring elements that do not overlap; expanded rows and sliding windows are copied)
            if mask.stride(1) != 1 or (rows > 1 and mask.stride(0) < mask.shape[1]):
                mask = mask.contiguous()
            return _Packed(attention_mask=mask, prompt_width=P)
    lens = [t.to(dev, torch.int64).contiguous() for t in batch_lens(data)]
    assert all(t.shape == (rows,) for t in lens), f"{[tuple(t.shape) for t in lens]} prompt and response lengths for {rows} responses"
    return _Packed(*lens)


def _padded(t: torch.Tensor, width: int) -> torch.Tensor:
    """A batch field as exactly ``[batch, width]``: nested (jagged) fields are padded with zeros like
    ``to_padded_tensor``, then cut or zero-padded to ``width`` (a jagged tensor without a cached longest row can come
    back wider than its longest row; columns beyond every row's length hold padding only)."""
    if t.is_nested:
        t = torch.nested.to_padded_tensor(t, 0.0)
    if t.shape[1] > width:
        t = t[:, :width]
    elif t.shape[1] < width:
        t = torch.nn.functional.pad(t, (0, width - t.shape[1]))
    return t if t.is_contiguous() else t.contiguous()


def response_width(data, response_lens) -> int:
    """Padded width of the response slice as ``no_padding_2_padding`` picks it (``verl/workers/utils/padding.py:112-124``):
    for nested batches the non-tensor entry ``max_response_len`` when it is there and not negative, else the longest
    response; for padded batches the width of ``responses``."""
    responses = data["responses"]
    if not responses.is_nested:
        return int(responses.shape[1])
    given = _get(data, "max_response_len")
    given = getattr(given, "data", given)  # (a tensordict NonTensorData wraps its payload)
    if given is not None and int(given) >= 0:
        return int(given)
    return int(response_lens.max().item())


def metric_aggregation_for(dp_size, batch_num_tokens, global_batch_size, loss_scale_factor):
    """``losses.py:71-84``: once any global normaliser is set the loss of a micro-batch is already a share of the
    global mean, so its metric adds up over micro-batches (SUM); otherwise each is a local mean (MEAN)."""
    from ...utils.metric import AggregationType

    if dp_size > 1 or batch_num_tokens is not None or global_batch_size is not None or loss_scale_factor is not None:
        return AggregationType.SUM
    return AggregationType.MEAN


def ppo_loss(config, model_output, data, dp_group=None):
    """The reference's actor loss entry (``verl/workers/utils/losses.py:57-155``) on the fused kernels: same arguments,
    same ``(policy_loss, metrics)`` with ``Metric`` values under the reference's keys and aggregation kinds.

    ``model_output["log_probs"]`` / ``["entropy"]``: the head's outputs over the packed sequences (``[total_nnz]`` or
    nested); ``data``: a mapping with ``prompts``, ``responses`` (nested, or padded together with
    ``attention_mask``), ``response_mask``, ``old_log_probs``, ``advantages``, optionally ``rollout_is_weights`` and
    ``ref_log_prob``, and the entries ``dp_size``, ``batch_num_tokens``, ``global_batch_size``.  ``config``: an
    ``ActorConfig``-like object (``clip_ratio*``, ``entropy_coeff``, ``loss_agg_mode``, ``loss_scale_factor``,
    ``use_kl_loss``, ``kl_loss_coef``, ``kl_loss_type``, ``policy_loss.loss_mode``, dict ``global_batch_info``).
    The response slice, the policy loss, the entropy and KL terms and all metrics are ONE ``lce_ppo_forward``
    call; gradients come back in packed order.  Only ``loss_mode == "vanilla"`` has a fused kernel; other modes and
    the sampler-correction outputs (``sc_*``) raise ``NotImplementedError`` instead of taking a slower path."""
    from ...utils.metric import AggregationType, Metric

    for key in ("sc_correction", "sc_sampler_head_mass", "sc_train_head_mass"):
        if _has(model_output, key):
            raise NotImplementedError(f"model output {key!r}: the fused PPO loss has no sampler-correction term")
    loss_mode = _cfg(_cfg(config, "policy_loss", {}) or {}, "loss_mode", "vanilla")
    if loss_mode != "vanilla":
        raise NotImplementedError(f"policy loss mode {loss_mode!r}: only 'vanilla' has a fused kernel")

    log_prob = model_output["log_probs"]
    log_prob = log_prob.values() if log_prob.is_nested else log_prob
    entropy = _get(model_output, "entropy")
    if entropy is not None and entropy.is_nested:
        entropy = entropy.values()

    info = {
        "dp_size": data["dp_size"],
        "batch_num_tokens": data["batch_num_tokens"],
        "global_batch_size": data["global_batch_size"],
        "loss_scale_factor": _cfg(config, "loss_scale_factor"),
    }
    shared = _cfg(config, "global_batch_info")
    if isinstance(shared, dict):  # the reference leaves them on the config for the policy-loss function
        shared.update(info)
    metric_aggregation = metric_aggregation_for(**info)

    packed = _packed_lengths(data, log_prob.device)
    width = response_width(data, packed.response_lens)
    rows = data["responses"].shape[0]
    response_mask = _padded(data["response_mask"], width)
    old_log_prob, advantages = _padded(data["old_log_probs"], width), _padded(data["advantages"], width)
    assert log_prob.dim() == 1 and (entropy is None or entropy.shape == log_prob.shape), "packed outputs are [total_nnz]"
    assert response_mask.shape == (rows, width) == old_log_prob.shape == advantages.shape
    use_kl = bool(_cfg(config, "use_kl_loss", False))
    is_weights = _get(data, "rollout_is_weights")
    policy_loss, m = fused_ppo_loss(
        log_prob, entropy, old_log_prob, advantages, response_mask, _packed=packed, _nonzero_mask=True,
        clip_ratio=_cfg(config, "clip_ratio"),
        clip_ratio_low=_cfg(config, "clip_ratio_low"),
        clip_ratio_high=_cfg(config, "clip_ratio_high"),
        clip_ratio_c=_cfg(config, "clip_ratio_c", 3.0),
        entropy_coeff=_cfg(config, "entropy_coeff", 0.0) if entropy is not None else 0.0,
        loss_agg_mode=_cfg(config, "loss_agg_mode", "token-mean"),
        rollout_is_weights=None if is_weights is None else _padded(is_weights, width),
        ref_log_prob=_padded(data["ref_log_prob"], width) if use_kl else None,
        kl_loss_coef=_cfg(config, "kl_loss_coef", 0.001),
        kl_loss_type=_cfg(config, "kl_loss_type", "low_var_kl"),
        **info,
    )  # fmt: skip
    metrics = Metric.from_dict(
        {k: m[k] for k in ("actor/pg_clipfrac", "actor/ppo_kl", "actor/pg_clipfrac_lower")}, AggregationType.MEAN
    )
    metrics["actor/pg_loss"] = Metric(metric_aggregation, m["actor/pg_loss"])
    if entropy is not None:
        metrics["actor/entropy_loss"] = Metric(metric_aggregation, m["actor/entropy_loss"])
    if use_kl:
        metrics["kl_loss"] = Metric(metric_aggregation, m["kl_loss"])
        metrics["kl_coef"] = _cfg(config, "kl_loss_coef", 0.001)
    # (last, with everything on the host done: the loss is on its way meanwhile)
    checks = packed.checks()
    longest = checks[2]
    if longest > width:
        raise ValueError(f"max_response_len = {width} is shorter than the longest response ({longest})")
    _check_lengths(checks, log_prob.numel(), width)
    return policy_loss, metrics
