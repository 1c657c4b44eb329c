"""The calls a trainer makes of this package, at the sizes it makes them: what is timed when the package is tuned.

Four kinds of work, each through the public entry points:

* ``head``: ``linear_cross_entropy`` on one micro-batch, forward only (the no-grad passes that compute old and reference
  log-probs), forward + backward, or forward + backward of ``hidden`` alone (a frozen lm-head under LoRA);
* ``actor``: the whole post-head actor step, ``linear_cross_entropy`` -> ``ppo_loss`` -> backward;
* ``logits``: the twins on logits that exist already, forward or forward + backward;
* ``ppo``: ``ppo_loss`` alone with its backward and its metrics (the outputs of the head are given).

``listed()`` names the cases, ``draw()`` gives more of the same ranges.
"""

import math
import random

import torch

from verl_amd import linear_cross_entropy
from verl_amd.utils import torch_functional as F
from verl_amd.utils.metric import reduce_metrics
from verl_amd.workers.utils.losses import ppo_loss

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}

# (hidden size, vocabulary, weight std) of the lm-heads of the benchmark's configurations: Qwen2.5-0.5B, Qwen2.5-7B,
# Llama-3-8B, Qwen2.5-32B
HEADS = [(896, 151936, 0.02), (3584, 152064, 0.02), (4096, 128256, 0.02), (5120, 152064, 0.015)]

# no drawn case costs more than the largest listed one: 65536 tokens through the largest head, forward + backward
LARGEST = 65536 * 5120 * 152064 * 6


def _head(name, head, tokens, mode, dtype="bf16", temperature=1.0, valid=1.0, entropy=True):
    """``valid``: share of the tokens that carry a gradient (a response mask zeroes the rest)."""
    H, V, std = HEADS[head]
    case = {"kind": "head", "T": tokens, "H": H, "V": V, "std": std, "mode": mode, "dtype": dtype,
            "temperature": temperature, "valid": valid, "entropy": entropy}  # fmt: skip
    return dict(case, name=name) if name else case


def _actor(name, head, sequences, prompt, response, kl, agg="token-mean"):
    H, V, std = HEADS[head]
    case = {"kind": "actor", "B": sequences, "P": prompt, "R": response, "H": H, "V": V, "std": std, "dtype": "bf16",
            "kl": kl, "agg": agg}  # fmt: skip
    return dict(case, name=name) if name else case


def _logits(name, rows, vocab, call, backward, dtype="bf16"):
    case = {"kind": "logits", "rows": rows, "V": vocab, "call": call, "backward": backward, "dtype": dtype}
    return dict(case, name=name) if name else case


def _ppo(name, sequences, prompt, response, kl, agg="token-mean"):
    case = {"kind": "ppo", "B": sequences, "P": prompt, "R": response, "kl": kl, "agg": agg}
    return dict(case, name=name) if name else case


def listed():
    return [
        # log-probs of one short answer under a small model, no gradient: latency, one read of the weight
        _head("logprob-0.5b-T40", 0, 40, "forward"),
        # a training micro-batch of one short sequence: every pass streams the weight
        _head("train-7b-T64", 1, 64, "train"),
        # a micro-batch of one ordinary sequence of odd length, between the streaming and the matrix-bound regime
        _head("train-7b-T333", 1, 333, "train"),
        # the same in float16, most of a thousand tokens, prompt and padding positions without gradient
        _head("train-8b-T1000-fp16", 2, 1000, "train", dtype="fp16", temperature=0.6, valid=0.6),
        # float32 inputs (tests and small models trained without mixed precision)
        _head("train-0.5b-T1024-fp32", 0, 1024, "train", dtype="fp32"),
        # old / reference log-prob pass over a packed micro-batch whose length is no multiple of anything
        _head("logprob-7b-T5003", 1, 5003, "forward"),
        # LoRA: the lm-head is frozen, only the gradient of the hidden states is asked for
        _head("lora-8b-T4096", 2, 4096, "frozen", valid=0.6),
        # the headline: 16 sequences of 1024 tokens, all with gradient
        _head("train-7b-T16384", 1, 16384, "train"),
        # the largest: 32 sequences of 2048 tokens through the largest head
        _head("train-32b-T65536", 3, 65536, "train"),
        # a whole actor micro-step, packed sequences of random length, entropy bonus and KL penalty
        _actor("actor-8b-8x2048", 2, 8, 1024, 1024, True),
        # the engine that has materialised logits: both values from one pass, one gradient
        _logits("logits-1000x152064", 1000, 152064, "both", True),
        # the loss on its own: small vectors, launches and host time
        _ppo("ppo-16x512", 16, 512, 512, True),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["head", "head", "head", "head", "head", "actor", "logits", "logits", "ppo"])
    if kind == "head":
        head = rng.randrange(len(HEADS))
        mode = rng.choice(["forward", "train", "train", "frozen"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "bf16", "fp16", "fp32"])
        H, V, _ = HEADS[head]
        high = min(65536, LARGEST // (H * V * 6))
        if dtype == "fp32":  # matrix rate of float32 is a sixteenth of bfloat16's
            high = min(2048, high)
        tokens = _log(rng, 1, high)
        if rng.random() < 0.3 and tokens >= 64:  # padded to a round number, as trainers often do
            tokens = tokens // 64 * 64
        return _head(None, head, tokens, mode, dtype, rng.choice([1.0, 1.0, 0.6]), rng.choice([1.0, 0.75, 0.5]), rng.random() < 0.75)
    if kind == "actor":
        prompt, response = _log(rng, 64, 1024), _log(rng, 64, 2048)
        most = min(32, 24576 // (prompt + response))
        return _actor(None, rng.randrange(3), rng.randint(1, max(1, most)), prompt, response, rng.random() < 0.5,
                      rng.choice(["token-mean", "token-mean", "seq-mean-token-sum", "seq-mean-token-mean"]))  # fmt: skip
    if kind == "logits":
        vocab = rng.choice([32000, 128256, 151936, 152064, _log(rng, 1000, 160000)])
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        return _logits(None, _log(rng, 8, 8192), vocab, rng.choice(["logprobs", "entropy", "both"]), rng.random() < 0.6, dtype)
    return _ppo(None, _log(rng, 1, 256), _log(rng, 16, 1024), _log(rng, 16, 4096), rng.random() < 0.5,
                rng.choice(["token-mean", "token-mean", "seq-mean-token-sum", "seq-mean-token-mean"]))  # fmt: skip


# ---- inputs ----------------------------------------------------------------------------------------


def _normal(g, rows, cols, std, dtype):
    """N(0, std) rounded to `dtype`, made in pieces so that the float32 values are never all there at once."""
    out = torch.empty(rows, cols, device="cuda", dtype=dtype)
    step = max(1, (1 << 27) // cols)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        out[r : r + n] = torch.randn(n, cols, device="cuda", generator=g).mul_(std)
    return out


class _Config:
    """The fields of an actor configuration that the loss reads."""

    clip_ratio = 0.2
    clip_ratio_low = 0.2
    clip_ratio_high = 0.28
    clip_ratio_c = 3.0
    entropy_coeff = 1e-3
    loss_scale_factor = None
    kl_loss_coef = 0.001
    kl_loss_type = "low_var_kl"
    policy_loss = {"loss_mode": "vanilla"}

    def __init__(self, kl, agg):
        self.use_kl_loss = kl
        self.loss_agg_mode = agg


def _lengths(case):
    """Prompt and response lengths of a batch, from a quarter of the longest on.  They are the case's, not the seed's: the
    packed outputs are as long as their sum."""
    rng = random.Random(case["B"] * 1_000_003 + case["P"] * 1009 + case["R"])
    pick = lambda n: [rng.randint(max(1, n // 4), n) for _ in range(case["B"])]  # noqa: E731
    return pick(case["P"]), pick(case["R"])


def _batch(case, g):
    """A padded data batch: prompts on the right of their half, responses on the left of theirs."""
    B, P, R = case["B"], case["P"], case["R"]
    prompt_lens, response_lens = (torch.tensor(n, device="cuda") for n in _lengths(case))
    at_p, at_r = torch.arange(P, device="cuda"), torch.arange(R, device="cuda")
    in_prompt = at_p[None, :] >= P - prompt_lens[:, None]
    in_response = at_r[None, :] < response_lens[:, None]
    start = (prompt_lens + response_lens).cumsum(0) - response_lens - 1
    where = (start[:, None] + at_r)[in_response]  # packed positions the response is read from
    data = {
        "prompts": torch.zeros(B, P, device="cuda", dtype=torch.int64),
        "responses": torch.zeros(B, R, device="cuda", dtype=torch.int64),
        "attention_mask": torch.cat([in_prompt, in_response], 1).to(torch.int64),
        "response_mask": in_response.to(torch.int64),
        "advantages": torch.randn(B, 1, device="cuda", generator=g) * in_response,
        "dp_size": 1,
        "batch_num_tokens": None,
        "global_batch_size": None,
    }
    return data, in_response, where, int((prompt_lens + response_lens).sum())


def _old_log_probs(data, case, in_response, values, g):
    """What the rollout policy and the reference policy said about the same tokens: close to the policy's own."""
    for key, spread in (("old_log_probs", 0.05), ("ref_log_prob", 0.1)):
        if key == "ref_log_prob" and not case["kl"]:
            continue
        full = torch.zeros(in_response.shape, device="cuda")
        full[in_response] = values + torch.randn(values.shape, device="cuda", generator=g) * spread
        data[key] = full


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    state = {"case": case}
    if kind == "head":
        T, H, V, dtype = case["T"], case["H"], case["V"], DTYPES[case["dtype"]]
        grad = case["mode"] != "forward"
        state["hidden"] = _normal(g, T, H, 1.0, dtype).requires_grad_(grad)
        state["weight"] = _normal(g, V, H, case["std"], dtype).requires_grad_(case["mode"] == "train")
        state["labels"] = torch.randint(0, V, (T,), device="cuda", generator=g)
        if grad:
            # rows of equal length, each with a valid prefix; a dozen tokens are one row
            rows = max(1, T // 1024)
            length = -(-T // rows)
            keep = torch.randint(int(length * (2 * case["valid"] - 1)), length + 1, (rows,), device="cuda", generator=g)
            keep = keep.clamp_(min=1)
            mask = (torch.arange(length, device="cuda")[None, :] < keep[:, None]).reshape(-1)[:T] if case["valid"] < 1 else 1.0
            state["g_logprobs"] = torch.randn(T, device="cuda", generator=g) * mask
            state["g_entropy"] = torch.randn(T, device="cuda", generator=g) * mask
    elif kind == "actor":
        data, in_response, where, total = _batch(case, g)
        H, V, dtype = case["H"], case["V"], DTYPES[case["dtype"]]
        state["hidden"] = _normal(g, total, H, 1.0, dtype).requires_grad_(True)
        state["weight"] = _normal(g, V, H, case["std"], dtype).requires_grad_(True)
        state["labels"] = torch.randint(0, V, (total,), device="cuda", generator=g)
        with torch.no_grad():
            now = linear_cross_entropy(state["hidden"], state["weight"], state["labels"], 1.0, "none")[0]
        _old_log_probs(data, case, in_response, now[where], g)
        state["data"], state["config"] = data, _Config(case["kl"], case["agg"])
    elif kind == "logits":
        R, V, dtype = case["rows"], case["V"], DTYPES[case["dtype"]]
        state["logits"] = _normal(g, R, V, 3.0, dtype).requires_grad_(case["backward"])
        state["labels"] = torch.randint(0, V, (R,), device="cuda", generator=g)
        state["g_logprobs"] = torch.randn(R, device="cuda", generator=g).to(dtype)
        state["g_entropy"] = torch.randn(R, device="cuda", generator=g).to(dtype)
    else:
        data, in_response, where, total = _batch(case, g)
        log_probs = -torch.rand(total, device="cuda", generator=g).add_(1e-3).log_().abs_()
        _old_log_probs(data, case, in_response, log_probs[where], g)
        state["log_probs"] = log_probs.requires_grad_(True)
        state["entropy"] = (torch.rand(total, device="cuda", generator=g) * 3).requires_grad_(True)
        state["data"], state["config"] = data, _Config(case["kl"], case["agg"])
    return state


# ---- one pass --------------------------------------------------------------------------------------


def _run_head(state):
    case = state["case"]
    hidden, weight, labels = state["hidden"], state["weight"], state["labels"]
    if case["mode"] == "forward":
        with torch.no_grad():
            return linear_cross_entropy(hidden, weight, labels, case["temperature"], "none")
    logprobs, entropy = linear_cross_entropy(hidden, weight, labels, case["temperature"], "none")
    wanted = (hidden, weight) if case["mode"] == "train" else (hidden,)
    if case["entropy"]:
        grads = torch.autograd.grad((logprobs, entropy), wanted, (state["g_logprobs"], state["g_entropy"]))
    else:  # entropy_coeff = 0: the entropy is looked at, not trained on
        grads = torch.autograd.grad((logprobs,), wanted, (state["g_logprobs"],))
    return logprobs.detach(), entropy.detach(), *grads


def _run_actor(state):
    hidden, weight = state["hidden"], state["weight"]
    logprobs, entropy = linear_cross_entropy(hidden, weight, state["labels"], 1.0, "none")
    # (one of several micro-batches: its metrics are looked at when the step ends, not here)
    loss, _ = ppo_loss(state["config"], {"log_probs": logprobs, "entropy": entropy}, state["data"])
    grads = torch.autograd.grad(loss, (hidden, weight))
    return loss.detach(), logprobs.detach(), entropy.detach(), *grads


def _run_logits(state):
    case, logits, labels = state["case"], state["logits"], state["labels"]
    call = case["call"]
    if call == "logprobs":
        out, upstream = (F.logprobs_from_logits(logits, labels),), (state["g_logprobs"],)
    elif call == "entropy":
        out, upstream = (F.entropy_from_logits(logits),), (state["g_entropy"],)
    else:
        out, upstream = F.logprobs_and_entropy_from_logits(logits, labels), (state["g_logprobs"], state["g_entropy"])
    if not case["backward"]:
        return out
    (d_logits,) = torch.autograd.grad(out, (logits,), upstream)
    return *(x.detach() for x in out), d_logits


def _run_ppo(state):
    log_probs, entropy = state["log_probs"], state["entropy"]
    loss, metrics = ppo_loss(state["config"], {"log_probs": log_probs, "entropy": entropy}, state["data"])
    grads = torch.autograd.grad(loss, (log_probs, entropy))
    return loss.detach(), *grads, reduce_metrics(metrics)  # a step of one micro-batch: what it logs


def run(state):
    return {"head": _run_head, "actor": _run_actor, "logits": _run_logits, "ppo": _run_ppo}[state["case"]["kind"]](state)


# ---- what a pass cannot do without -----------------------------------------------------------------


def _head_work(T, trained, H, V, size, d_hidden, d_weight):
    """The three products of forward and backward; the hidden states, the weight and their gradients once each."""
    products = 2.0 * T + 2.0 * trained * (d_hidden + d_weight)
    return {"flops": products * H * V, "bytes": size * H * (T * (1 + d_hidden) + V * (1 + d_weight)) + 24.0 * T}


def _loss_bytes(case):
    """Two model outputs and their gradients over the packed tokens; the batch's vectors over the padded responses."""
    total = sum(map(sum, _lengths(case)))
    vectors = 4 * 2 + 8 + (4 if case["kl"] else 0)  # old log-probs, advantages, mask, reference log-probs
    return 16.0 * total + case["B"] * case["R"] * vectors + 8.0 * case["B"] * (case["P"] + case["R"])


def work(case):
    kind = case["kind"]
    size = 4 if case.get("dtype") == "fp32" else 2
    if kind == "head":
        grad = case["mode"] != "forward"
        return _head_work(case["T"], case["T"] * case["valid"], case["H"], case["V"], size, int(grad), int(case["mode"] == "train"))
    if kind == "actor":
        prompts, responses = _lengths(case)
        w = _head_work(sum(prompts) + sum(responses), sum(responses), case["H"], case["V"], size, 1, 1)
        return dict(w, bytes=w["bytes"] + _loss_bytes(case))
    if kind == "logits":
        values = float(case["rows"]) * case["V"]
        # read for the values; read again for the gradient only because a row may be larger than what a core can hold
        return {"bytes": values * size * (2 if case["backward"] else 1), "flops": values * (12 if case["backward"] else 6)}
    return {"bytes": _loss_bytes(case), "flops": 60.0 * case["B"] * case["R"]}


def tolerance(case):
    kind = case["kind"]
    if kind == "ppo":
        # float32 sums of terms of either sign: the loss is a few hundredths of the mean size of its terms
        return {"rel": 1e-4, "max": 1e-3}
    if kind == "logits":
        return {"rel": 1e-5, "max": 1e-4} if case["dtype"] == "fp32" else {"rel": 1e-2, "max": 5e-2}
    if kind == "head" and case["mode"] == "forward":
        return {"rel": 1e-5, "max": 1e-4}  # float32 sums whatever the inputs' type
    if case["dtype"] == "fp32":
        return {"rel": 2e-5, "max": 1e-3}
    # gradients rounded to 16 bits, from logits' gradients that are rounded to 16 bits too
    return {"rel": 1e-2, "max": 5e-2}
