"""Drop-in ``Sampler`` / ``SamplingConfig`` for the llm-pipeline inference engine.

Interface of ``src/llm_pipeline/inference/sampling.py`` kept verbatim:
``Sampler(config)``, ``.config``, ``sample_token(logits, config_override,
generated_tokens)`` (``:51-85``), ``_merge_config`` (``:87-106``, unknown keys
raise ``TypeError``), ``sample_mirostat_v2`` (``:240-279``) and
``get_sampling_info`` (``:281-293``).  Every call runs the HIP kernels of
``liblps.so`` on the logits' device; there is no CPU path.

Additive, default-neutral extensions: ``presence_penalty``,
``frequency_penalty``, ``logprobs`` and ``top_logprobs`` config fields, and
keyword-only ``uniforms`` / ``params`` / ``histories`` / ``history_lengths``
arguments to ``sample_token``.
"""

from __future__ import annotations

import math
from array import array
from dataclasses import dataclass
from typing import Any, Dict, Iterable, List, Optional

import torch

from . import _device as D
from .batch import SamplingParams, pad_histories, raise_on_status, row_kind_flags, sample_rows


@dataclass
class SamplingConfig:
    """Reference fields (``sampling.py:10-37``) plus the build's extensions."""

    temperature: float = 1.0
    top_k: int = 50
    top_p: float = 0.9
    repetition_penalty: float = 1.0
    typical_p: float = 1.0
    min_p: float = 0.0
    mirostat_tau: float = 5.0
    mirostat_eta: float = 0.1
    do_sample: bool = True
    pad_token_id: Optional[int] = None
    eos_token_id: Optional[int] = None
    presence_penalty: float = 0.0
    frequency_penalty: float = 0.0
    logprobs: bool = False
    top_logprobs: int = 0


_CONFIG_KEYS = (
    "temperature", "top_k", "top_p", "repetition_penalty", "typical_p", "min_p", "mirostat_tau",
    "mirostat_eta", "do_sample", "pad_token_id", "eos_token_id", "presence_penalty", "frequency_penalty",
    "logprobs", "top_logprobs",
)


def _history_ids(tokens) -> torch.Tensor:
    """A request's generated ids (any iterable, read once) as ``int32 [n]`` on the host."""
    ids = list(tokens)
    if not ids:
        return torch.empty((0,), dtype=torch.int32)
    try:
        # (an array of bytes would take their memory, not their values)
        return torch.frombuffer(array("i", ids), dtype=torch.int32)
    except (TypeError, OverflowError):   # (what torch converts or rejects)
        return torch.tensor(ids, dtype=torch.int32).reshape(-1)


def _upload_history(tokens: Iterable[int], B: int, dev: torch.device) -> tuple:
    """One history for every row: ``int32 [B, n]`` and lengths ``int32 [B]`` on
    the device, in one copy (from pinned memory, which does not wait for the
    stream, unless a graph is being captured); ``(None, None)`` without ids."""
    h = _history_ids(tokens)
    n = h.numel()
    if n == 0:
        return None, None
    pin = not torch.cuda.is_current_stream_capturing()
    buf = torch.empty((n + B,), dtype=torch.int32, pin_memory=pin)
    buf[:n] = h
    buf[n:] = n
    buf = buf.to(dev, non_blocking=pin)
    return buf[:n].unsqueeze(0).expand(B, n).contiguous(), buf[n:]


class _KeptParams(dict):
    """Parameter sets kept by a sampler.  A deep copy or a pickle of the sampler
    starts with none: copied tensors would be filled on the stream of the copy,
    not on the one that their key names."""

    def __reduce__(self):
        return _KeptParams, ()


class Sampler:
    """Centralised logits -> token sampler on MI355X."""

    _PARAM_SETS = 8   # shared parameter tensors kept per sampler

    def __init__(self, config: Optional[SamplingConfig] = None):
        self.config = config or SamplingConfig()
        self.last_output = None

    def _shared_params(self, B: int, dev: torch.device, config: "SamplingConfig") -> SamplingParams:
        """The config's values for every row as device tensors: 8 fills a call
        when built each time, so the last few sets are kept, by the values they
        hold, the rows and the stream that filled them.  A call under graph
        capture builds its own (a graph's tensors are the graph's, and a kept
        set may be dropped while the graph lives)."""
        values = (config.temperature, config.top_k, config.top_p, config.min_p, config.typical_p,
                  config.repetition_penalty, config.presence_penalty, config.frequency_penalty)
        if not all(isinstance(v, (int, float)) and v == v for v in values) or \
                torch.cuda.is_current_stream_capturing():
            return SamplingParams.build(B, dev, *values)
        key = (B, dev.index, D.stream_of(dev), values)
        # (a subclass with its own __init__, or an older pickle, has none yet)
        kept = self.__dict__.setdefault("_params", _KeptParams())
        p = kept.get(key)
        if p is None:
            if len(kept) >= self._PARAM_SETS:
                kept.clear()
            p = kept[key] = SamplingParams.build(B, dev, *values)
        return p

    def sample_token(self, logits: torch.Tensor, config_override: Optional[Dict[str, Any]] = None,
                     generated_tokens: Optional[List[int]] = None, *, uniforms: Optional[torch.Tensor] = None,
                     params: Optional[SamplingParams] = None, histories: Optional[torch.Tensor] = None,
                     history_lengths: Optional[torch.Tensor] = None, generator: Optional[torch.Generator] = None,
                     allowed: Optional[torch.Tensor] = None, strict: Optional[bool] = None) -> torch.Tensor:
        """Sample next token ids ``int64 [B]`` from ``logits [B, V]``.

        As in the reference, ``generated_tokens`` is one history applied to
        every row and the repetition penalty fires only when it is non-empty
        and the penalty differs from 1.  ``params`` (per-row
        ``SamplingParams``) and ``histories`` (padded ``int32 [B, H]``)
        replace the shared values row by row.  ``uniforms`` (``[B]`` in
        [0, 1)) drive the inverse-CDF draw; when omitted they come from
        ``torch.rand`` on the logits' device.  ``allowed`` (bool ``[B, V]`` or
        packed ``int32`` bits) masks illegal ids to -inf, as a reference
        ``LogitConstraint`` applied to the logits first would.

        ``strict`` raises the reference's ``RuntimeError`` for rows
        ``torch.multinomial`` would reject (NaN / +inf / all -inf); reading the
        row status synchronises the stream once, as the engine's ``.item()``
        after every call does anyway (``qwen3_engine.py:412-420``).  The
        default (``None``) checks unless the stream is being captured into a
        graph, where the call stays stream-ordered; ``False`` never checks
        (tokens of rejected rows are -1 and ``last_output.status`` holds the
        reason)."""
        config = self._merge_config(config_override)
        D.require_device(logits, "logits")
        if logits.dim() != 2:
            raise ValueError(f"logits must be [batch_size, vocab_size]; got {tuple(logits.shape)}")
        B = logits.shape[0]
        dev = logits.device
        hint = 0
        if params is None:
            hint = row_kind_flags(config.temperature, config.top_k, config.min_p, config.typical_p)
            params = self._shared_params(B, dev, config)
        if histories is None and generated_tokens:
            histories, history_lengths = _upload_history(generated_tokens, B, dev)
        out = sample_rows(logits, params, uniforms, histories=histories, history_lengths=history_lengths,
                          logprobs=bool(config.logprobs), top_logprobs=int(config.top_logprobs),
                          generator=generator, allowed=allowed, row_kind_hint=hint)
        self.last_output = out
        if strict is None:
            strict = not torch.cuda.is_current_stream_capturing()
        if strict:
            raise_on_status(out.status)
        return out.tokens

    def _merge_config(self, config_override: Optional[Dict[str, Any]]) -> SamplingConfig:
        """``sampling.py:87-106``: copy, ``update``, rebuild; unknown keys raise
        ``TypeError`` from the dataclass constructor."""
        if not config_override:
            return self.config
        d = {k: getattr(self.config, k) for k in _CONFIG_KEYS}
        d.update(config_override)
        return SamplingConfig(**d)

    def sample_mirostat_v2(self, logits: torch.Tensor, config_override: Optional[Dict[str, Any]] = None,
                           previous_entropy: Optional[float] = None, *,
                           uniforms: Optional[torch.Tensor] = None) -> tuple:
        """``sampling.py:240-279``: entropy of ``softmax(logits / T)`` (logits
        unscaled when ``T <= 0``), ``prev -= eta * (H - tau)``, top-k with
        ``k = max(1, int(exp(prev)))`` when ``prev > 0``, then a draw.  Like the
        reference (``.item()`` on the entropy) it takes a single row."""
        config = self._merge_config(config_override)
        D.require_device(logits, "logits")
        B = logits.shape[0]
        dev = logits.device
        T = config.temperature if config.temperature > 0 else 1.0
        stats = sample_rows(logits, SamplingParams.build(B, dev, temperature=T), None, entropy=True,
                            skip_draw=True)
        current = float(stats.entropy.reshape(-1)[0].item())
        if previous_entropy is None:
            previous_entropy = current
        previous_entropy -= config.mirostat_eta * (current - config.mirostat_tau)
        k = max(1, int(math.exp(previous_entropy))) if previous_entropy > 0 else 0
        # the reference's _apply_top_k clamps k to the vocabulary (sampling.py:151)
        k = min(k, logits.shape[-1])
        out = sample_rows(logits, SamplingParams.build(B, dev, temperature=T, top_k=k), uniforms,
                          row_kind_hint=row_kind_flags(T, k, 0.0, 1.0))
        raise_on_status(out.status)
        return out.tokens, previous_entropy

    def get_sampling_info(self) -> Dict[str, Any]:
        """``sampling.py:281-293``."""
        return {
            "temperature": self.config.temperature,
            "top_k": self.config.top_k,
            "top_p": self.config.top_p,
            "repetition_penalty": self.config.repetition_penalty,
            "typical_p": self.config.typical_p,
            "min_p": self.config.min_p,
            "mirostat_tau": self.config.mirostat_tau,
            "mirostat_eta": self.config.mirostat_eta,
            "do_sample": self.config.do_sample,
        }


__all__ = ["Sampler", "SamplingConfig", "pad_histories"]
