"""The host side of a single-request call (CPU, no GPU)."""

import copy
import pickle

import numpy as np
import pytest
import torch

from lps import Sampler, SamplingConfig
from lps.sampling import _history_ids, _upload_history


class _Tokens(list):
    """A list whose iteration is its own."""

    def __iter__(self):
        return iter([7, 8])


@pytest.mark.parametrize("make,want", [
    (lambda: [3, 5, 5], [3, 5, 5]),
    (lambda: (3, 5), [3, 5]),
    (lambda: iter([3, 5]), [3, 5]),
    (lambda: (t for t in [3, 5]), [3, 5]),
    (lambda: (t for t in [3.0, 5.9]), [3, 5]),                 # floats: what torch converts
    (lambda: iter(torch.tensor([3, 5])), [3, 5]),
    (lambda: iter([[3, 5], [6, 7]]), [3, 5, 6, 7]),
    (lambda: np.array([3, 5], dtype=np.int64), [3, 5]),
    (lambda: b"\x03\x05", [3, 5]),
    (lambda: _Tokens([1]), [7, 8]),
    (lambda: iter([]), []),
    (lambda: [[]], []),
])
def test_generated_tokens_are_read_once(make, want):
    """Any iterable of ids is one history, also one that can be read only once
    and whose elements torch, not an int array, converts."""
    h = _history_ids(make())
    assert h.dtype == torch.int32 and h.tolist() == want


@pytest.mark.parametrize("bad", [["a"], [2 ** 31], [None], [torch.tensor(3.0), torch.tensor(5.0)]])
def test_generated_tokens_rejected(bad):
    with pytest.raises((TypeError, ValueError, RuntimeError)):
        _history_ids(iter(bad))


def test_empty_iterators_are_no_history():
    assert _upload_history(iter([]), 2, torch.device("cpu")) == (None, None)


@pytest.mark.parametrize("duplicate", [copy.deepcopy, lambda s: pickle.loads(pickle.dumps(s))])
def test_copies_of_a_sampler_keep_no_parameter_tensors(monkeypatch, duplicate):
    """The kept parameter sets belong to the stream that filled them: a copy,
    whose tensors another stream would have filled, makes its own."""
    import lps.sampling as S
    monkeypatch.setattr(S.D, "stream_of", lambda dev: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    s = Sampler(SamplingConfig(temperature=0.7))
    dev = torch.device("cpu")
    kept = s._shared_params(2, dev, s.config)
    assert s._shared_params(2, dev, s.config) is kept
    d = duplicate(s)
    assert d.config == s.config and not d._params
    assert d._shared_params(2, dev, d.config) is not kept
    assert s._shared_params(2, dev, s.config) is kept
