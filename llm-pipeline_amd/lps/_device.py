"""Device-tensor plumbing shared by the sampler entry points: dtype codes,
pointers, the current HIP stream and per-row parameter tensors."""

from __future__ import annotations

import contextlib

import torch

from . import _lib

_DTYPES = {
    torch.float32: _lib.LPS_DTYPE_F32,
    torch.bfloat16: _lib.LPS_DTYPE_BF16,
    torch.float16: _lib.LPS_DTYPE_F16,
}


def require_device(t: torch.Tensor, name: str) -> None:
    """The sampler runs only on the GPU; there is no CPU path."""
    if not isinstance(t, torch.Tensor):
        raise TypeError(f"{name} must be a torch.Tensor")
    if t.device.type != "cuda":
        raise RuntimeError(f"lps samples on a ROCm device; {name} is on {t.device}")


def dtype_code(t: torch.Tensor) -> int:
    try:
        return _DTYPES[t.dtype]
    except KeyError:
        raise TypeError(f"unsupported logits dtype {t.dtype}; expected float32, bfloat16 or float16") from None


def ptr(t) -> int:
    return 0 if t is None else int(t.data_ptr())


def stream_of(device: torch.device) -> int:
    """The device's current stream as an integer handle (the raw accessor: a
    ``torch.cuda.Stream`` object costs 2.5 us a call, this 0.2)."""
    return torch._C._cuda_getCurrentRawStream(torch.cuda.current_device() if device.index is None else device.index)


_NO_GUARD = contextlib.nullcontext()


def guard(device: torch.device):
    """Makes ``device`` current for a launch; nothing to do (and to undo) when it is."""
    return _NO_GUARD if torch._C._cuda_getDevice() == device.index else torch.cuda.device(device)


def on(t: torch.Tensor, device: torch.device, dtype: torch.dtype) -> torch.Tensor:
    """``t`` on ``device`` as ``dtype`` (``t`` itself when it is)."""
    return t if t.dtype is dtype and t.device == device else t.to(device=device, dtype=dtype)


def flat(t: torch.Tensor, device: torch.device, dtype: torch.dtype) -> torch.Tensor:
    """``t`` on ``device`` as a contiguous vector of ``dtype``."""
    t = on(t, device, dtype)
    return t if t.dim() == 1 and t.is_contiguous() else t.reshape(-1).contiguous()


def as_f32(v, B: int, device) -> torch.Tensor:
    if isinstance(v, torch.Tensor):
        t = v.to(device=device, dtype=torch.float32).reshape(-1)
        if t.numel() == 1 and B != 1:
            t = t.expand(B)
        return t.contiguous()
    return torch.full((B,), float(v), dtype=torch.float32, device=device)


def as_i32(v, B: int, device) -> torch.Tensor:
    if isinstance(v, torch.Tensor):
        t = v.to(device=device, dtype=torch.int32).reshape(-1)
        if t.numel() == 1 and B != 1:
            t = t.expand(B)
        return t.contiguous()
    return torch.full((B,), int(v), dtype=torch.int32, device=device)
