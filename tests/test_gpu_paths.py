"""The multi-workgroup fast kernel against the oracle and against the general
kernel, on the BASELINE.json configurations: both paths must meet the parity
bar, and the fast path must finish the rows of the benchmark configurations
itself (rows it defers are finished by the general kernel)."""

import pytest
import torch

from tests import parity as PY
from tests import workloads as W

pytestmark = pytest.mark.gpu


def _paths(w, dev, rows=None, lp=False):
    fast = PY.run_workload(w, dev, path="auto")
    gen = PY.run_workload(w, dev, path="generic")
    rf = PY.check_rows(w, fast, rows=rows, lp=lp)
    rg = PY.check_rows(w, gen, rows=rows, lp=lp)
    nfast = int((fast.row_path.cpu() == 0).sum())
    same = int((fast.tokens == gen.tokens).sum())
    print(f"{w.name}: fast-path rows {nfast}/{w.B}; tokens equal to the general kernel {same}/{w.B}; "
          f"fast {rf}; general {rg}", flush=True)
    return fast, gen, nfast


def test_paths_c2(dev):
    w = W.c2()
    fast, gen, nfast = _paths(w, dev)
    assert nfast == w.B


def test_paths_c1(dev):
    for g in (False, True):
        w = W.c1(greedy=g)
        fast, gen, nfast = _paths(w, dev)
        assert nfast == 1


@pytest.mark.parametrize("B", [16, 256])
@pytest.mark.parametrize("flat", [False, True])
def test_paths_c3(dev, flat, B):
    """c3 stays on the fast path (at B=256 the launch shape the benchmark
    times).  In its flat variant the cut and draw bins hold thousands of
    logits, which the row-group kernel's second histogram level resolves: at
    most 8 of 256 rows (3 %) may be left to the general kernel."""
    w = W.c3(B=B, flat=flat)
    fast, gen, nfast = _paths(w, dev)
    if not flat:
        assert nfast == w.B
    else:
        assert w.B - nfast <= max(1, (8 * w.B) // 256), f"{w.B - nfast} rows deferred"


def test_hardware_exp2_is_monotone(dev):
    """The row-group kernel finds a histogram region's logits by a search over
    x, which needs exp2(fma(x, c, -ref)) non-decreasing in x: the device's
    hardware exp2 must not decrease anywhere over the fp32 inputs."""
    import ctypes
    from lps import _lib
    v = ctypes.c_ulonglong(12345)
    assert _lib.load().lps_selftest_exp2_monotone(ctypes.byref(v)) == 0
    assert v.value == 0, f"{v.value} decreasing steps"


def test_paths_c5(dev):
    w = W.c5(B=32)
    fast, gen, nfast = _paths(w, dev, lp=True)
    assert nfast == w.B


def test_fast_small_and_ragged(dev):
    """Vocabularies below one chunk, exactly one chunk, ragged last chunk, scalar loads."""
    from tests.test_gpu_parity import _small
    for V in (5, 777, 8192, 8193, 20011):
        for dt in (torch.float32, torch.bfloat16):
            w = _small(V, 16, dt, seed=V)
            out = PY.run_workload(w, dev)
            PY.check_rows(w, out)


@pytest.mark.parametrize("B,V,dtype", [(3, 151936, torch.bfloat16), (64, 151936, torch.bfloat16), (20, 100001, torch.float16),
                                       (5, 32001, torch.float32), (96, 40000, torch.float32)])
@pytest.mark.parametrize("n_top", [1, 20, 64])
def test_top_logprobs_of_nucleus_rows(dev, B, V, dtype, n_top):
    """Top-N logprobs of rows without top-k (nucleus, min-p, typical-p, pure, and
    a few greedy and top-k rows between them) on the row-group kernel, from one
    chunk per row to 13 and on rows read element by element: every row on the
    fast kernel, outputs against the oracle, ids exactly."""
    w = W.c2(B=B, V=V, H=64)
    i = torch.arange(B)
    w.logits = w.logits.to(dtype)
    w.temperature = torch.where(i % 7 == 6, torch.tensor(0.0), w.temperature.clamp(min=0.3))
    w.top_k = torch.where(i % 5 == 4, torch.tensor(40), torch.tensor(0)).to(torch.int32)
    w.top_p = torch.tensor([0.9, 1.0, 0.95, 0.5])[i % 4]
    w.min_p = torch.where(i % 6 == 2, torch.tensor(0.05), torch.tensor(0.0))
    w.logprobs, w.n_top = True, n_top
    out = PY.run_workload(w, dev, row_kind_hint=0)
    assert int(out.row_path.sum()) == 0
    PY.check_rows(w, out, rows=range(0, B, 1 if B < 32 else 7), lp=True)


def test_top_logprobs_left_to_the_general_kernel(dev):
    """Rows with fewer legal ids than top_logprobs, and rows that cannot be
    sampled, keep the general kernel's outputs."""
    from lps import SamplingParams, sample_rows
    g = torch.Generator().manual_seed(3)
    x = torch.randn((4, 5000), generator=g)
    x[1, 10:] = float("-inf")
    x[2, 7] = float("nan")
    p = SamplingParams.build(4, dev, top_p=0.9)
    u = torch.rand((4,), generator=g).to(dev)
    a = sample_rows(x.to(dev), p, u, logprobs=True, top_logprobs=20)
    b = sample_rows(x.to(dev), p, u, logprobs=True, top_logprobs=20, path="generic")
    assert a.row_path.tolist() == [0, 1, 1, 0]
    assert torch.equal(a.tokens, b.tokens) and torch.equal(a.status, b.status) and torch.equal(a.top_ids[:2], b.top_ids[:2])
    torch.testing.assert_close(a.top_logprobs[[0, 1, 3]], b.top_logprobs[[0, 1, 3]], rtol=1e-5, atol=2e-6)


@pytest.mark.parametrize("B", [3, 40])
def test_one_history_shared_by_every_row(dev, B):
    """A history of stride 0 (one row expanded to the batch) gives what its copies give."""
    from lps import SamplingParams, sample_rows
    g = torch.Generator().manual_seed(B)
    x = torch.randn((B, 40000), generator=g).to(dev)
    h = x[0].topk(300).indices.to(torch.int32).reshape(1, -1)         # the ids most likely to be drawn
    p = SamplingParams.build(B, dev, top_k=50, repetition_penalty=1.5, frequency_penalty=2.0)
    u = torch.rand((B,), generator=g).to(dev)
    a = sample_rows(x, p, u, histories=h.expand(B, -1), logprobs=True)
    b = sample_rows(x, p, u, histories=h.repeat(B, 1), logprobs=True)
    assert torch.equal(a.tokens, b.tokens) and torch.equal(a.chosen_logprob, b.chosen_logprob)


@pytest.mark.parametrize("V,dtype", [(151936, torch.bfloat16), (100001, torch.float32), (50257, torch.float16)])
def test_flat_threshold_rows_stay_on_the_row_group_kernel(dev, V, dtype):
    """Almost uniform rows with min-p under every logit's ratio (alone, and after
    a top-p that cuts first): the draw's bin, and the top-p cut's, hold
    thousands of logits and take the second level.  At most one row in 16 off
    the fast kernel; kept sets and draws against the oracle."""
    B = 32
    w = W.c2(B=B, V=V, H=16)
    g = torch.Generator().manual_seed(V)
    i = torch.arange(B)
    w.logits = (torch.randn((B, V), generator=g) * 0.1).to(dtype)
    w.top_k = torch.zeros(B, dtype=torch.int32)
    w.temperature = 0.5 + 0.7 * torch.rand(B, generator=g)
    w.min_p = torch.tensor([0.02, 0.05, 0.1, 0.0])[i % 4]
    w.top_p = torch.tensor([1.0, 0.95])[(i // 4) % 2]
    out = PY.run_workload(w, dev)
    assert int(out.row_path.sum()) <= B // 16
    min_p, w.min_p = w.min_p, torch.zeros(B)      # (min-p removes nothing here: the oracle's top-p band applies)
    assert float(min_p.max()) < float(torch.exp(-(w.logits.float().amax(1) - w.logits.float().amin(1)) / w.temperature).min())
    PY.check_rows(w, out)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,V", [(5, 9), (3, 1001), (3, 12289), (24, 50257), (2, 151935), (40, 100001), (70, 40963)])
def test_rows_off_the_16_byte_lines(dev, dtype, B, V):
    """Odd vocabularies (every row starts elsewhere in its 16-byte line, ids shift
    by that much in the vectors) in every row mode, with histories and legality
    masks, from a row of one partial vector to several chunks; the logits also
    as rows of a wider buffer.  Rows against the oracle, none deferred for V
    past the smallest."""
    w = W.c2(B=B, V=V, H=64)
    i = torch.arange(B)
    g = torch.Generator().manual_seed(V)
    legal = torch.rand((B, V), generator=g) < 0.7
    legal[:, V // 2] = True
    w.logits = w.logits.to(dtype).masked_fill(~legal, float("-inf"))   # (the oracle's rows)
    raw = w.logits.masked_fill(~legal, 3.0).to(dev)
    w.temperature = torch.where(i % 5 == 3, torch.tensor(0.0), w.temperature.clamp(min=0.3))
    w.top_k = torch.where(i % 3 == 0, torch.tensor(0), w.top_k.clamp(max=V)).to(torch.int32)
    w.min_p = torch.where(i % 6 == 3, torch.tensor(0.05), torch.tensor(0.0))
    w.logprobs = True
    out = PY.run_workload(w, dev, row_kind_hint=0)
    PY.check_rows(w, out, rows=range(0, B, 1 if B < 30 else 7), lp=True)
    assert int(out.row_path.sum()) == 0 or V < 2000
    ref = out
    w.logits = raw.cpu()
    out = PY.run_workload(w, dev, row_kind_hint=0, allowed=legal.to(dev))
    assert torch.equal(out.tokens, ref.tokens) and torch.equal(out.kept_count, ref.kept_count)
    wide = torch.full((B, V + 5), 50.0, dtype=dtype, device=dev)       # rows from the fourth element on
    wide[:, 3:3 + V] = raw
    from lps import SamplingParams, sample_rows
    p = SamplingParams(*[t.to(dev) for t in (w.temperature, w.top_k, w.top_p, w.min_p, w.typical_p, w.rep, w.pres, w.freq)])
    o = sample_rows(wide[:, 3:3 + V], p, w.uniforms.to(dev), histories=w.histories.to(dev),
                    history_lengths=w.hist_len.to(dev), allowed=legal.to(dev))
    assert torch.equal(o.tokens, ref.tokens)


def test_single_request_call_takes_every_form_of_history(dev):
    """A history as a list, a tuple, bytes, nested lists or whole floats is the
    same history, also for a sampler whose class has an ``__init__`` of its own."""
    from lps import Sampler, SamplingConfig

    class Own(Sampler):
        def __init__(self, config):
            self.config = config

    logits = torch.randn((1, 4099), generator=torch.Generator().manual_seed(7)).to(dev)
    ids = [3, 250, 17, 3]
    config = SamplingConfig(temperature=0.9, top_p=0.95, repetition_penalty=3.0, frequency_penalty=0.5, logprobs=True)
    seen = []
    for s in (Sampler(config), Own(config)):
        for h in (ids, tuple(ids), bytes(ids), [ids], [float(i) for i in ids]):
            t = s.sample_token(logits, generated_tokens=h, uniforms=torch.tensor([0.4], device=dev))
            seen.append((torch.as_tensor(t).reshape(-1).tolist(), s.last_output.chosen_logprob.tolist()))
    assert all(x == seen[0] for x in seen)


def test_single_request_call_reads_iterators_once(dev):
    """A history that can be read only once, of ids or of floats, is the
    list's history; an empty iterator is no history."""
    from lps import Sampler, SamplingConfig
    logits = torch.randn((2, 4099), generator=torch.Generator().manual_seed(8)).to(dev)
    u = torch.tensor([0.4, 0.7], device=dev)
    s = Sampler(SamplingConfig(temperature=0.9, top_p=0.95, repetition_penalty=3.0, frequency_penalty=0.5, logprobs=True))

    def call(h):
        t = s.sample_token(logits, generated_tokens=h, uniforms=u)
        return t.tolist(), s.last_output.chosen_logprob.tolist()

    ids = logits[0].topk(40).indices.tolist()
    want = call(ids)
    assert want != call(None)
    assert call(iter(ids)) == want and call(float(i) for i in ids) == want
    assert call(iter([])) == call(None)
