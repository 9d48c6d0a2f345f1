"""The calls a decode loop makes of this framework, as measurable cases.

One step of an inference engine turns hidden states into logits (``lm_head``),
logits into probabilities where a caller wants them (``fused_softmax``), logits
into tokens (``Sampler.sample_token`` for one request, ``sample_rows`` for a
batch) and, with a draft model, draft and target logits into accepted tokens
(``spec_verify``).  The listed cases are those calls at the sizes of the
benchmark's configurations, from one row to 512, with odd vocabularies and key
counts among them; ``draw`` gives others of the same ranges.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "llm-pipeline_amd"))

from lps import (Sampler, SamplingConfig, SamplingParams, fused_softmax, lm_head, row_kind_flags,  # noqa: E402
                 sample_rows, spec_verify)

DEVICE = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
BYTES = {"f32": 4, "bf16": 2, "f16": 2}


def listed():
    return [
        # an interactive request decoding alone: the engine's one call per token
        {"name": "token_b1_f32", "kind": "token", "vocab": 151936, "dtype": "f32", "history": 64},
        # a continuous batch whose requests each bring their own parameters
        {"name": "mixed_b64_bf16", "kind": "sample", "rows": 64, "vocab": 151936, "dtype": "bf16", "logits": "spiked",
         "mix": "mixed", "history": 512, "logprobs": False, "top": 0, "masked": False},
        # a large batch of nucleus rows (evaluation or rollout generation)
        {"name": "nucleus_b256_f32", "kind": "sample", "rows": 256, "vocab": 151936, "dtype": "f32",
         "logits": "student", "mix": "nucleus", "history": 0, "logprobs": True, "top": 0, "masked": False},
        # the largest decode batch: greedy and top-k rows with logprobs for the API's response
        {"name": "logprobs_b512_f16", "kind": "sample", "rows": 512, "vocab": 151936, "dtype": "f16",
         "logits": "normal", "mix": "greedy_topk", "history": 1024, "logprobs": True, "top": 20, "masked": False},
        # constrained decoding on an odd vocabulary (rows that do not start on a 16-byte line)
        {"name": "masked_b24_odd_bf16", "kind": "sample", "rows": 24, "vocab": 50257, "dtype": "bf16",
         "logits": "normal", "mix": "minp", "history": 256, "logprobs": True, "top": 0, "masked": True},
        # speculative decoding, the reference's rule: 32 requests, four drafted tokens each
        {"name": "verify_b32_k4_f32", "kind": "verify", "rows": 32, "k": 4, "vocab": 151936, "dtype": "f32",
         "temperature": 0.8, "top_p": 0.95, "residual": "target"},
        # the same step with the textbook residual on a small batch
        {"name": "verify_b8_k3_residual", "kind": "verify", "rows": 8, "k": 3, "vocab": 151936, "dtype": "bf16",
         "temperature": 0.8, "top_p": 1.0, "residual": "leviathan"},
        # probabilities of a decode batch's logits
        {"name": "softmax_logits_b64", "kind": "softmax", "lead": 1, "queries": 64, "cols": 151936, "dtype": "bf16",
         "causal": False, "offset": 0},
        # attention probabilities of a prompt: 32 heads, 2048 queries and keys
        {"name": "softmax_prefill", "kind": "softmax", "lead": 32, "queries": 2048, "cols": 2048, "dtype": "bf16",
         "causal": True, "offset": 0},
        # a chunk of a prompt against the keys cached so far: odd sizes, unaligned rows
        {"name": "softmax_chunk_odd", "kind": "softmax", "lead": 128, "queries": 129, "cols": 1601, "dtype": "bf16",
         "causal": True, "offset": 1472},
        # a decode batch's hidden states to logits and probabilities
        {"name": "head_b64", "kind": "head", "rows": 64, "hidden": 4096, "vocab": 151936, "dtype": "bf16",
         "out": "bf16", "probs": True},
        # a prompt's hidden states to logits (the reference projects every position)
        {"name": "head_prefill_2048", "kind": "head", "rows": 2048, "hidden": 4096, "vocab": 151936, "dtype": "bf16",
         "out": "bf16", "probs": False},
    ]


def _spread(rng, lo, hi):
    """A whole number spread over [lo, hi] by its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _vocab(rng):
    """A vocabulary of 32,000 to 151,936 ids: whole vectors, or any number."""
    v = _spread(rng, 32000, 151936)
    return v - v % 128 if rng.random() < 0.6 else v


def draw(rng):
    kind = rng.choice(["token", "sample", "sample", "sample", "verify", "softmax", "softmax", "head", "head"])
    dtype = rng.choice(["f32", "bf16", "f16"])
    if kind == "token":
        return {"kind": kind, "vocab": _vocab(rng), "dtype": dtype, "history": _spread(rng, 1, 2048)}
    if kind == "sample":
        return {"kind": kind, "rows": _spread(rng, 1, 512), "vocab": _vocab(rng), "dtype": dtype,
                "logits": rng.choice(["spiked", "normal", "student", "flat"]),
                "mix": rng.choice(["mixed", "nucleus", "greedy_topk", "topk", "minp"]),
                "history": rng.choice([0, _spread(rng, 16, 2048)]), "logprobs": rng.random() < 0.5,
                "top": rng.choice([0, 0, 5, 20]), "masked": rng.random() < 0.2}
    if kind == "verify":
        return {"kind": kind, "rows": _spread(rng, 1, 48), "k": rng.randint(1, 5), "vocab": _vocab(rng), "dtype": dtype,
                "temperature": round(rng.uniform(0.5, 1.2), 2), "top_p": rng.choice([1.0, 0.9, 0.95]),
                "residual": rng.choice(["target", "target", "leviathan"])}
    if kind == "softmax":
        if rng.random() < 0.3:   # logits
            return {"kind": kind, "lead": 1, "queries": _spread(rng, 1, 256), "cols": _vocab(rng), "dtype": dtype,
                    "causal": False, "offset": 0}
        queries, cached = _spread(rng, 1, 2048), rng.choice([0, _spread(rng, 1, 6000)])
        cols = queries + cached
        lead = max(1, min(256, (1 << 27) // (queries * cols)))
        return {"kind": kind, "lead": _spread(rng, 1, lead), "queries": queries, "cols": cols, "dtype": dtype,
                "causal": rng.random() < 0.8, "offset": cached}
    return {"kind": "head", "rows": _spread(rng, 1, 2048), "hidden": 16 * _spread(rng, 56, 256), "vocab": _vocab(rng),
            "dtype": rng.choice(["bf16", "bf16", "f16"]), "out": rng.choice(["same", "same", "f32"]),
            "probs": rng.random() < 0.3}


# --------------------------------------------------------------------------- #
# Inputs
# --------------------------------------------------------------------------- #


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(seed)


def _logits(kind, rows, vocab, dtype, g):
    x = torch.randn((rows, vocab), generator=g, device=DEVICE)
    if kind == "spiked":        # a trained model's row: a few ids stand out
        x *= 3.0
        at = torch.randint(0, vocab, (rows, 3), generator=g, device=DEVICE)
        x.scatter_(1, at, 12.0)
    elif kind == "normal":
        x *= 2.5
    elif kind == "student":     # heavy tails: 2 t(3)
        c = torch.zeros_like(x)
        for _ in range(3):
            c += torch.randn((rows, vocab), generator=g, device=DEVICE).square_()
        x = 2.0 * x / (c / 3.0).sqrt_()
    else:                       # an undecided model: almost uniform
        x *= 0.1
    return x.to(dtype)


def _params(mix, rows, history, g):
    """The batch's parameters as a batcher holds them: host values per request."""
    h = torch.Generator().manual_seed(int(torch.randint(0, 1 << 30, (1,), generator=g, device=DEVICE)))
    u = torch.rand((3, rows), generator=h)
    pick = torch.randint(0, 4, (rows,), generator=h)
    p = {"temperature": torch.ones(rows), "top_k": torch.zeros(rows, dtype=torch.int32), "top_p": torch.ones(rows),
         "min_p": torch.zeros(rows), "typical_p": torch.ones(rows), "repetition_penalty": torch.ones(rows),
         "presence_penalty": torch.zeros(rows), "frequency_penalty": torch.zeros(rows)}
    if mix == "mixed":
        p["temperature"] = 0.3 + 0.9 * u[0]
        p["top_k"] = torch.tensor([0, 20, 50, 100], dtype=torch.int32)[pick]
        p["top_p"] = 0.8 + 0.2 * u[1]
        p["presence_penalty"].fill_(0.5 if history else 0.0)
        p["frequency_penalty"].fill_(0.3 if history else 0.0)
    elif mix == "nucleus":
        p["top_p"].fill_(0.95)
    elif mix == "greedy_topk":
        greedy = torch.arange(rows) % 2 == 0
        p["temperature"] = torch.where(greedy, 0.0, 0.9)
        p["top_k"] = torch.where(greedy, 0, 40).to(torch.int32)
        p["top_p"] = torch.where(greedy, 1.0, 0.92)
        p["repetition_penalty"].fill_(1.05)
    elif mix == "topk":
        p["temperature"].fill_(0.7)
        p["top_k"].fill_(50)
        p["top_p"].fill_(0.9)
        p["repetition_penalty"].fill_(1.1)
    else:
        p["temperature"] = 0.5 + 0.7 * u[0]
        p["min_p"] = torch.tensor([0.02, 0.05, 0.1, 0.2])[pick]
        p["top_p"] = torch.where(u[1] < 0.5, 1.0, 0.95)
        p["repetition_penalty"].fill_(1.1)
    return p


def prepare(case, seed):
    g = _generator(seed)
    s = {"case": case}
    kind, dt = case["kind"], DTYPES[case["dtype"]]
    if kind == "token":
        s["logits"] = _logits("normal", 1, case["vocab"], dt, g)
        s["sampler"] = Sampler(SamplingConfig(temperature=0.7, top_k=50, top_p=0.9, repetition_penalty=1.1,
                                              logprobs=True))
        s["generated"] = torch.randint(0, case["vocab"], (case["history"],), generator=g, device=DEVICE).tolist()
        s["uniforms"] = torch.rand((1,), generator=g, device=DEVICE)
    elif kind == "sample":
        rows, vocab, n = case["rows"], case["vocab"], case["history"]
        s["logits"] = _logits(case["logits"], rows, vocab, dt, g)
        p = _params(case["mix"], rows, n, g)
        s["hint"] = row_kind_flags(p["temperature"], p["top_k"], p["min_p"], p["typical_p"])
        s["params"] = SamplingParams.build(rows, DEVICE, **p)
        s["uniforms"] = torch.rand((rows,), generator=g, device=DEVICE)
        s["history"] = s["lengths"] = s["allowed"] = None
        if n:                   # log-uniform ids: the few frequent ones repeat, as a text's do
            ids = torch.rand((rows, n), generator=g, device=DEVICE).mul_(math.log(vocab)).exp_() - 1.0
            s["history"] = ids.clamp_(0, vocab - 1).to(torch.int32)
            s["lengths"] = torch.full((rows,), n, dtype=torch.int32, device=DEVICE)
        if case["masked"]:      # packed legality bits, half of the ids legal
            s["allowed"] = torch.randint(-2 ** 31, 2 ** 31, (rows, (vocab + 31) // 32), generator=g, device=DEVICE,
                                         dtype=torch.int64).to(torch.int32)
    elif kind == "verify":
        rows, k, vocab = case["rows"], case["k"], case["vocab"]
        target = torch.randn((rows, k + 1, vocab), generator=g, device=DEVICE).mul_(2.0)
        draft = target[:, :k] + 0.5 * torch.randn((rows, k, vocab), generator=g, device=DEVICE)
        probs = torch.softmax(draft / case["temperature"], dim=-1).reshape(rows * k, vocab)
        s["drafted"] = torch.multinomial(probs, 1, generator=g).reshape(rows, k)
        s["target"], s["draft"] = target.to(dt), draft.to(dt)
        s["u_accept"] = torch.rand((rows, k), generator=g, device=DEVICE)
        s["u_resample"] = torch.rand((rows, k + 1), generator=g, device=DEVICE)
    elif kind == "softmax":
        s["x"] = torch.randn((case["lead"], case["queries"], case["cols"]), generator=g, device=DEVICE).mul_(3.0).to(dt)
    else:
        s["hidden"] = torch.randn((case["rows"], case["hidden"]), generator=g, device=DEVICE, dtype=dt)
        s["weight"] = torch.randn((case["vocab"], case["hidden"]), generator=g, device=DEVICE, dtype=dt)
        s["weight"].mul_(2.5 / math.sqrt(case["hidden"]))
        s["out"] = dt if case["out"] == "same" else DTYPES[case["out"]]
    return s


def run(state):
    c = state["case"]
    if c["kind"] == "token":
        token = state["sampler"].sample_token(state["logits"], generated_tokens=state["generated"],
                                              uniforms=state["uniforms"])
        return {"tokens": token, "logprob": state["sampler"].last_output.chosen_logprob}
    if c["kind"] == "sample":
        o = sample_rows(state["logits"], state["params"], state["uniforms"], histories=state["history"],
                        history_lengths=state["lengths"], logprobs=c["logprobs"], top_logprobs=c["top"],
                        allowed=state["allowed"], row_kind_hint=state["hint"])
        return {"tokens": o.tokens, "status": o.status, "logprob": o.chosen_logprob, "top_logprobs": o.top_logprobs,
                "top_ids": o.top_ids}
    if c["kind"] == "verify":
        o = spec_verify(state["target"], state["draft"], state["drafted"], state["u_accept"], state["u_resample"],
                        c["temperature"], c["top_p"], residual=c["residual"])
        return {"accepted": o.n_accepted, "tokens": o.tokens, "accept": o.accept, "p_target": o.p_target,
                "q_draft": o.q_draft, "status": o.status}
    if c["kind"] == "softmax":
        return fused_softmax(state["x"], causal=c["causal"], row_offset=c["offset"])
    if c["probs"]:
        logits, stats = lm_head(state["hidden"], state["weight"], out_dtype=state["out"], return_stats=True)
        return {"logits": logits, "stats": stats, "probs": fused_softmax(logits, row_stats=stats)}
    return lm_head(state["hidden"], state["weight"], out_dtype=state["out"])


def work(case):
    kind, es = case["kind"], BYTES[case["dtype"]]
    if kind == "token":
        return {"bytes": case["vocab"] * es + 4 * case["history"] + 48, "flops": 0}
    if kind == "sample":
        row = case["vocab"] * es + 4 * case["history"] + 48 + 4 * case["logprobs"] + 12 * case["top"]
        if case["masked"]:
            row += (case["vocab"] + 31) // 32 * 4
        return {"bytes": case["rows"] * row, "flops": 0}
    if kind == "verify":
        return {"bytes": case["rows"] * ((2 * case["k"] + 1) * case["vocab"] * es + 48 * case["k"]), "flops": 0}
    if kind == "softmax":
        rows, cols = case["lead"] * case["queries"], case["cols"]
        seen = rows * cols
        if case["causal"]:
            seen = case["lead"] * sum(min(cols, q + case["offset"] + 1) for q in range(case["queries"]))
        return {"bytes": (seen + rows * cols) * es, "flops": 0}
    m, n, h = case["rows"], case["vocab"], case["hidden"]
    eo = es if case["out"] == "same" else BYTES[case["out"]]
    read = (m + n) * h * es
    if case["probs"]:           # logits and probabilities out, the block statistics, the logits read once more
        return {"bytes": read + 3 * m * n * eo + 8 * m * ((n + 127) // 128), "flops": 2 * m * n * h}
    return {"bytes": read + m * n * eo, "flops": 2 * m * n * h}


def tolerance(case):
    kind = case["kind"]
    if kind in ("token", "sample", "verify"):
        # fp32 masses and log-sum-exps over whole rows; a draw may fall on a boundary
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.01}
    out = case["dtype"] if kind == "softmax" or case["out"] == "same" else case["out"]
    if kind == "head" and case["probs"]:
        # a rounded maximum that falls the other way moves its block's statistics by a unit of the output type
        return {"rel": {"f32": 1e-5, "bf16": 7e-3, "f16": 9e-4}[out], "max": {"f32": 1e-4, "bf16": 0.1, "f16": 0.02}[out]}
    return {"rel": {"f32": 2e-6, "bf16": 7e-3, "f16": 9e-4}[out], "max": {"f32": 2e-5, "bf16": 2e-2, "f16": 2e-3}[out]}


# --------------------------------------------------------------------------- #
# The same values in 64 bits
# --------------------------------------------------------------------------- #


def _penalised(x, history, p):
    """x after the penalties: repetition once per distinct id, then frequency by count, then presence."""
    if history is None:
        return x
    n = torch.zeros_like(x).scatter_add_(1, history.long(), torch.ones_like(history, dtype=torch.float64))
    rep, pres, freq = (p[m].double().unsqueeze(1)
                       for m in ("repetition_penalty", "presence_penalty", "frequency_penalty"))
    y = torch.where(x > 0, x / rep, x * rep) - n * freq - pres
    return torch.where(n > 0, y, x)


def _draw(z, p, u):
    """The drawn id of every row: the inverse CDF over the kept ids, the largest first; the argmax of greedy rows."""
    v, at = torch.sort(z, dim=1, descending=True, stable=True)
    k = p["top_k"].long().clamp(max=z.shape[1])
    kth = v.gather(1, (k - 1).clamp(min=0).unsqueeze(1))
    keep = (v >= kth) | (k <= 0).unsqueeze(1)
    e = torch.where(keep, (v - v[:, :1]).exp_(), 0.0)
    cum = e.cumsum(1)
    top_p = p["top_p"].double().unsqueeze(1)
    keep &= (cum - e <= top_p * cum[:, -1:]) | (top_p >= 1.0)
    keep &= e >= p["min_p"].double().unsqueeze(1) * e[:, :1]
    cum = torch.where(keep, e, 0.0).cumsum_(1)
    j = torch.searchsorted(cum, u.double().unsqueeze(1) * cum[:, -1:], right=True)
    j = torch.where((p["temperature"] > 0).unsqueeze(1), j.clamp(max=z.shape[1] - 1), 0)
    return at.gather(1, j)


def _sampled(logits, history, allowed, p, u, top):
    """(chosen logprob, top logprobs) of a batch in 64 bits, in blocks of rows."""
    chosen, best = [], []
    for i in range(0, logits.shape[0], 64):
        q = {m: v[i:i + 64].to(DEVICE) for m, v in p.items()}
        x = _penalised(logits[i:i + 64].double(), None if history is None else history[i:i + 64], q)
        if allowed is not None:
            bits = (allowed[i:i + 64].unsqueeze(2) >> torch.arange(32, device=DEVICE, dtype=torch.int32)) & 1
            x = x.masked_fill(bits.reshape(bits.shape[0], -1)[:, :x.shape[1]] == 0, -math.inf)
        t = q["temperature"].double().unsqueeze(1)
        z = torch.where(t > 0, x / torch.where(t > 0, t, 1.0), x)
        lse = torch.logsumexp(z, dim=1, keepdim=True)
        chosen.append(z.gather(1, _draw(z, q, u[i:i + 64])) - lse)
        best.append(torch.topk(z, top, dim=1).values - lse if top else None)
    return torch.cat(chosen).reshape(-1), torch.cat(best) if top else None


def _kept_prob(logits, tokens, temperature, top_p):
    """Probability of each row's token under softmax(top_p(logits / T))."""
    z = logits.double() / temperature
    v, at = torch.sort(z, dim=-1, descending=True, stable=True)
    e = (v - v[..., :1]).exp_()
    cum = e.cumsum(-1)
    if top_p < 1.0:
        e = torch.where(cum - e <= top_p * cum[..., -1:], e, 0.0)
    place = (at == tokens.unsqueeze(-1)).to(torch.float64)
    return (e * place).sum(-1) / e.sum(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample" and not case["logprobs"] and not case["top"]:
        return None             # tokens and status only
    s = prepare(case, seed)
    if kind == "token":
        row = {"temperature": 0.7, "top_p": 0.9, "min_p": 0.0, "repetition_penalty": 1.1, "presence_penalty": 0.0,
               "frequency_penalty": 0.0}
        p = {m: torch.tensor([v], dtype=torch.float32) for m, v in row.items()}
        p["top_k"] = torch.tensor([50], dtype=torch.int32)
        history = torch.tensor([s["generated"]], device=DEVICE)
        return {"tokens": None, "logprob": _sampled(s["logits"], history, None, p, s["uniforms"], 0)[0]}
    if kind == "sample":
        p = {m: getattr(s["params"], m) for m in ("temperature", "top_k", "top_p", "min_p", "repetition_penalty",
                                                  "presence_penalty", "frequency_penalty")}
        chosen, best = _sampled(s["logits"], s["history"], s["allowed"], p, s["uniforms"], case["top"])
        return {"tokens": None, "status": None, "logprob": chosen if case["logprobs"] else None,
                "top_logprobs": best, "top_ids": None}
    if kind == "verify":
        # the parameters as 32-bit values, as the entry point takes them
        t, top_p = (float(torch.tensor(case[m], dtype=torch.float32)) for m in ("temperature", "top_p"))
        return {"accepted": None, "tokens": None, "accept": None, "status": None,
                "p_target": _kept_prob(s["target"][:, :-1], s["drafted"], t, top_p),
                "q_draft": _kept_prob(s["draft"], s["drafted"], t, top_p)}
    if kind == "softmax":
        x = s["x"].double()
        if case["causal"]:
            q = torch.arange(case["queries"], device=DEVICE).unsqueeze(1) + case["offset"]
            x.masked_fill_(torch.arange(case["cols"], device=DEVICE).unsqueeze(0) > q, -math.inf)
        return torch.softmax(x, dim=-1)
    logits = s["hidden"].double() @ s["weight"].double().T
    if not case["probs"]:
        return logits
    # (the probabilities are those of the stored, rounded logits)
    return {"logits": logits, "stats": None, "probs": torch.softmax(logits.to(s["out"]).double(), dim=-1)}
