"""ctypes binding of the C ABI declared in ``include/lce_abi.h``."""

from __future__ import annotations

import contextlib
import ctypes
import os
import threading

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.environ.get("LCE_LIBRARY_PATH") or os.path.join(_HERE, "lib", "liblce_gfx950.so")

DTYPE_BF16, DTYPE_F32, DTYPE_F16 = 0, 1, 2
DTYPE_F32_PLANES = 3  # fp32 with leave to use the bfloat16 matrix pipe: the fused head, forward and backward alike
ABI_VERSION = 11

# every symbol include/lce_abi.h declares: name -> (restype, argtypes)
_c = ctypes
_p, _i64, _i, _f, _sz = _c.c_void_p, _c.c_int64, _c.c_int, _c.c_float, _c.c_size_t
SYMBOLS = {
    "lce_abi_version": (_i, []),
    "lce_last_error": (_c.c_char_p, []),
    "lce_forward_workspace_bytes": (_sz, [_i64, _i64, _i64, _i]),
    "lce_forward": (_i, [_p, _i64, _p, _i64, _p, _i64, _i64, _i64, _i, _f, _i, _p, _p, _p, _p, _p, _p, _sz, _p]),
    "lce_forward_static": (_i, [_p, _i64, _p, _i64, _p, _i64, _i64, _i64, _i, _f, _i, _p, _p, _p, _p, _p, _p]),
    "lce_backward_workspace_bytes": (_sz, [_i64, _i64, _i64, _i, _i64]),
    "lce_backward": (
        _i,
        [_p, _i64, _p, _i64, _p, _i64, _i64, _i64, _i, _f, _i, _p, _p, _p, _p, _p, _p, _p, _p, _sz, _i64, _p],
    ),
    "lce_backward_f32": (
        _i,
        [_p, _i64, _p, _i64, _p, _i64, _i64, _i64, _i, _f, _i, _p, _p, _p, _p, _p, _p, _p, _p, _sz, _i64, _p],
    ),
    "lce_logits_cache_max_tokens": (_i64, [_i64, _i]),
    "lce_logits_cache_bytes": (_sz, [_i64, _i64, _i64, _i]),
    "lce_kept_logits_bytes": (_sz, [_i64, _i64, _i64, _i]),
    "lce_forward_keep_logits": (
        _i,
        [_p, _i64, _p, _i64, _p, _i64, _i64, _i64, _i, _f, _i, _p, _p, _p, _p, _p, _p, _sz, _p, _sz, _p],
    ),
    "lce_backward_from_logits": (
        _i,
        [_p, _i64, _p, _i64, _p, _i64, _i64, _i64, _i, _f, _i, _p, _p, _p, _p, _p, _p, _p, _i, _p, _sz, _i64, _p, _sz, _p],
    ),
    "lce_forward_shard": (_i, [_p, _i64, _p, _i64, _p, _i64, _i64, _i64, _i64, _i, _f, _p, _p, _sz, _p]),
    "lce_merge_shards": (_i, [_p, _i, _i64, _i, _p, _p, _p, _p, _p, _p, _sz, _p]),
    "lce_backward_shard": (
        _i,
        [_p, _i64, _p, _i64, _p, _i64, _i64, _i64, _i64, _i, _f, _i, _p, _p, _p, _p, _p, _p, _p, _p, _sz, _i64, _p],
    ),
    "lce_logits_forward": (_i, [_p, _i64, _p, _i64, _i64, _i, _p, _p, _p, _p]),
    "lce_logits_backward": (_i, [_p, _i64, _p, _i64, _i64, _i, _p, _p, _p, _p, _i64, _p]),
    "lce_logits_forward_as": (_i, [_p, _i64, _p, _i64, _i64, _i, _p, _i, _p, _i, _p, _p]),
    "lce_logits_backward_as": (_i, [_p, _i64, _p, _i64, _i64, _i, _p, _p, _i, _p, _i, _p, _i64, _p]),
    "lce_logits_sum_pi_squared": (_i, [_p, _i64, _i64, _i64, _i, _p, _p, _p]),
    "lce_logits_sum_pi_squared_backward": (_i, [_p, _i64, _i64, _i64, _i, _p, _p, _p, _p, _i64, _p]),
    "lce_ppo_loss_workspace_bytes": (_sz, [_i64, _i64]),
    "lce_ppo_loss": (_i, [_p, _p, _p, _p, _p, _p, _p, _i, _f, _i64, _i64, _i, _f, _f, _f, _f, _f, _f, _f, _f, _p, _p, _p, _p, _sz, _p]),
    "lce_ppo_loss_packed": (_i, [_p, _p, _i64, _p, _p, _p, _p, _p, _p, _p, _i, _f, _i64, _i64, _i, _f, _f, _f, _f, _f, _f, _f, _f, _p, _p, _p, _p, _sz, _p]),
    "lce_ppo_forward": (_i, [_p, _p]),
    "lce_ppo_forward_begin": (_i, [_p, _p, _p]),
    "lce_ppo_forward_end": (_i, [_p, _p, _p]),
    "lce_ppo_backward": (_i, [_p, _p]),
    "lce_gemm_nt": (_i, [_p, _i64, _p, _i64, _p, _i64, _i64, _i64, _i64, _i, _i, _p]),
    "lce_gemm_tn": (_i, [_p, _i64, _p, _i64, _p, _i64, _i64, _i64, _i64, _i, _p]),
    "lce_set_variant": (_i, [_i]),
    "lce_num_variants": (_i, []),
    "lce_set_option": (_i, [_i, _i64]),
    "lce_profile_enable": (_i, [_i]),
    "lce_profile_num_classes": (_i, []),
    "lce_profile_class_name": (_c.c_char_p, [_i]),
    "lce_profile_read": (_i, [_p, _p, _i]),
}

# lce_ppo_call_t
class PpoCall(_c.Structure):
    _fields_ = (
        [(n, _p) for n in ("log_prob", "entropy", "old_log_prob", "advantages", "mask", "is_weights", "ref_log_prob", "attention_mask",
                           "prompt_lens", "response_lens", "out", "g_log_prob", "g_entropy", "workspace", "g_loss", "d_log_prob", "d_entropy")]
        + [(n, _i64) for n in ("total_nnz", "rows", "row_len", "attention_stride", "prompt_width", "attention_width", "workspace_bytes")]
        + [("checks", _i64 * 3)]
        + [(n, _i) for n in ("mask_kind", "attention_kind", "kl_type", "agg_mode")]
        + [(n, _f) for n in ("kl_coef", "clip_low", "clip_high", "clip_c", "entropy_coeff", "dp_size", "batch_num_tokens",
                             "global_batch_size", "loss_scale_factor")]
    )  # fmt: skip


_lib = None
_lock = threading.Lock()


class LceError(RuntimeError):
    pass


def load() -> ctypes.CDLL:
    """Loads the HIP library; raises if it has not been built (there is no fallback path)."""
    global _lib
    if _lib is not None:
        return _lib
    with _lock:
        if _lib is not None:
            return _lib
        if not os.path.exists(LIB_PATH):
            raise LceError(
                f"{LIB_PATH} is missing: build it with `python -m verl_amd.build` (needs hipcc, targets gfx950). "
                "verl_amd has no CPU or eager fallback."
            )
        lib = ctypes.CDLL(LIB_PATH)
        # (first, and before another version's library is asked for symbols that it may not have)
        if lib.lce_abi_version() != ABI_VERSION:
            raise LceError(f"ABI version mismatch: library {lib.lce_abi_version()}, binding {ABI_VERSION}")
        for name, (res, args) in SYMBOLS.items():
            fn = getattr(lib, name, None)
            if fn is None:
                raise LceError(f"{LIB_PATH} has no {name}: it was built from older sources, build it again")
            fn.restype = res
            fn.argtypes = args
        _lib = lib
    return _lib


def check(rc: int, what: str) -> None:
    if rc != 0:
        msg = load().lce_last_error().decode(errors="replace")
        if "Invalid reduction" in msg:
            raise ValueError(msg)
        raise LceError(f"{what} failed ({rc}): {msg}")


_DTYPE_CODES = {torch.bfloat16: DTYPE_BF16, torch.float32: DTYPE_F32, torch.float16: DTYPE_F16}


def dtype_code(dtype) -> int:
    code = _DTYPE_CODES.get(dtype)
    if code is not None:
        return code
    raise NotImplementedError(f"verl_amd supports bfloat16, float16 and float32 inputs, got {dtype}")


def ptr(t) -> int | None:
    return None if t is None else t.data_ptr()


def current_stream(device) -> int:
    return torch._C._cuda_getCurrentRawStream(device.index)


_here = contextlib.nullcontext()


def on_device(device):
    """``torch.cuda.device(device)`` where that is not the current device already (the context manager costs a small call
    more than the call itself does)."""
    return _here if torch._C._cuda_getDevice() == device.index else torch.cuda.device(device)


def profile_read(reset: bool = True) -> dict[str, tuple[float, int]]:
    """{kernel class: (total ms, launches)} since profiling was enabled / last reset."""
    lib = load()
    n = lib.lce_profile_num_classes()
    ms = (ctypes.c_double * n)()
    cnt = (ctypes.c_int64 * n)()
    check(lib.lce_profile_read(ctypes.addressof(ms), ctypes.addressof(cnt), 1 if reset else 0), "lce_profile_read")
    return {lib.lce_profile_class_name(i).decode(): (ms[i], cnt[i]) for i in range(n) if cnt[i] > 0}
